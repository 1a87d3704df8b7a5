// Block-form weights for few rows (m 5..64), on the matrix unit.
//
// Replaces the reference's lanes rule reading a block form through its load (engine/rules/
// linear/src/lanes.rs:17-143, every form of engine/plan/codegen/src/form.rs:10-93 and
// block.rs:251-291): the decode product of a batch. Same arithmetic as the many-row kernel
// (blockmat.hip): codes exact in bf16, one matrix-unit sum per block from zero, times the
// block's scale, added in f32.
//
// gfx950 design. At these row counts the packed bytes are the work: each is read once and
// should arrive at the rate of HBM.
//  * A group of 8 waves; a wave owns 32 weight rows (SiLU pairs: 16 gate rows and the 16 up
//    rows of the same columns) and streams them in units of 128 codes through its own LDS
//    ring, filled with 4-byte global_load_lds (blocks are 9 to 66 bytes; a unit is always
//    whole words), two units ahead of their use where LDS allows. No barrier waits on
//    weights: a wave waits for its own loads only.
//  * The rows of x are shared: a step of S units (S 2 up to 32 rows, else 1) is staged in LDS
//    as ready matrix operands, double-buffered, its loads a step ahead of the store, one
//    barrier a step. With S = 2 half the waves take the even units and half the odd ones,
//    which halves the operand reads of a step; the two halves' sums meet in LDS at the end.
//  * Lane (c, g) decodes its 8 codes of weight row c straight from LDS words into the second
//    operand, so the sums leave the matrix unit with column c = the lane's own row and the
//    block scale is a register of the lane. The 8 codes of 32 are g's quarter of the block's
//    bytes (q4_0: the low nibbles of four bytes, then the high ones; x is staged in the same
//    order). Nibbles convert as signed bytes 16 (code - 8), the 16 taken out of the scale
//    (both exact); e2m1 and e4m3 on gfx950's bf16 conversions; nvfp4 folds its e4m3 scale
//    into the codes (exact in bf16).
//  * Where the columns alone do not give every CU a group, k is split across groups: raw sums
//    to the workspace, added in split order by split_finish.
// Against the 64 x 64 tiles of blockmat.hip, which these sizes went to (64 groups, each a
// serial chain over all of k): 16 f32 rows by int4_g32 2 x 14336 x 4096 156 -> 28 us, 4096 x
// 14336 343 -> 18 us; 8 bf16 rows by q8_0 79 -> 37 and 175 -> 20 us; 64 f32 rows by int4_g32
// 157 -> 52 and 346 -> 31 us. At 16 rows what bounds it now is the decode (14 vector
// operations per 8 nibbles, then the scaling of the block sums); at 64 the matrix unit.
#include <algorithm>
#include <type_traits>

#include "blockform.h"

namespace ts {

namespace {

constexpr int kWaves = 8, kThreads = kWaves * 64;
constexpr int kUnit = 128;  // codes of a row per unit: 4 matrix steps of 32
constexpr uint32_t kCus = 256;
constexpr int kRawBuffer = 0x00020000;  // buffer descriptor word 3: a raw buffer of 32-bit data
constexpr int kMaxLds = 160 * 1024;

struct StreamParams {
    const void *x;
    const uint8_t *w;  // the packed tensor (head included)
    const float *a0;
    void *out;
    float *part;  // split sums, or NULL
    uint32_t m, n, k;
    uint32_t stages;
    int out_bf16;
    uint32_t splits;
    ts_after after;  // stage chain (count 0: none)
};

template <int F, int MT, bool XF32, bool SILU>
struct Shape {
    using BF = BlockForm<F>;
    static constexpr int S = MT <= 2 ? 2 : 1, C = kWaves / S;
    static constexpr int PARTS = XF32 ? 2 : 1;
    static constexpr int QS = 4 * S;  // matrix steps of one step
    static constexpr int XBUF = QS * MT * PARTS * 1024;
    // A unit of a row: whole blocks of 32 or 16 codes, or one block of 128 (66 bytes: the
    // odd units start on a half word, so a unit is loaded from the word it starts in).
    static constexpr int BYTES = kUnit / BF::B * BF::BB, WORDS = (BYTES + 3) / 4;
    static constexpr int LOADS = (32 * WORDS + 63) / 64, SLOT = LOADS * 256;
    static constexpr int RING = 2 * XBUF + 3 * kWaves * SLOT <= kMaxLds ? 3 : 2;
    static constexpr int LDS = 2 * XBUF + RING * kWaves * SLOT;
    static constexpr int OC = C * (SILU ? 16 : 32);  // output columns of a group
    static constexpr int PIECES = 16 * MT * QS * 4, PER = (PIECES + kThreads - 1) / kThreads;
    static_assert(LDS <= kMaxLds, "LDS");
};

// Four codes' bytes at byte `at` (a lane's) of a row's words.
TS_DEV uint32_t word_at(const uint32_t *row, uint32_t at) {
    const uint32_t w = at >> 2;
    return __builtin_amdgcn_alignbyte(row[w + 1], row[w], at & 3u);
}

template <int SH>
TS_DEV uint32_t word_static(const uint32_t *row) {
    return SH == 0 ? row[0] : __builtin_amdgcn_alignbyte(row[1], row[0], SH);
}

TS_DEV uint32_t pk_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(ts_f32x2{a, b}, ts_bf16x2));
}

// The signed byte I of w as f32.
template <int I>
TS_DEV float byte_float(uint32_t w) {
    return (float)(int8_t)(w >> (8 * I));
}

// The packed bytes of matrix step Q of a unit for lane group g: its 8 codes' words and the
// word that holds the block's scale. row: the unit's words of this lane's weight row; par:
// 1 when the unit starts on a half word (128-code blocks).
struct Packed {
    uint32_t w0, w1, s;
};

template <int F, int Q>
TS_DEV Packed packed(const uint32_t *row, uint32_t g, uint32_t par) {
    using BF = BlockForm<F>;
    Packed b = {0, 0, 0};
    if constexpr (BF::B == 128) {
        const uint32_t *p = row + 4 * Q + g;  // bytes 2 par + 2 + 16 Q + 4 g
        b.w0 = par ? p[1] : __builtin_amdgcn_alignbyte(p[1], p[0], 2);
        if (Q == 0) b.s = par ? row[0] >> 16 : row[0];
    } else if constexpr (BF::B == 16) {
        b.w0 = word_at(row, 18 * Q + 9 * (g >> 1) + 1 + 4 * (g & 1));
        const uint32_t at = 18 * Q + 9 * (g >> 1);
        b.s = row[at >> 2] >> (8 * (at & 3u));
    } else {
        constexpr uint32_t off = Q * BF::BB + BF::SB, so = Q * BF::BB;
        const uint32_t *p = row + off / 4 + g * (BF::BITS / 4);
        b.w0 = word_static<off % 4>(p);
        if (BF::BITS == 8) b.w1 = word_static<off % 4>(p + 1);
        b.s = row[so / 4] >> (8 * (so % 4));  // a 2-byte scale starts on an even byte: within the word
    }
    return b;
}

// Those 8 codes as bf16, and the scale of their block (untouched where the codes hold it).
template <int F, int Q>
TS_DEV bf16x8 decode(const Packed &b, float &scale) {
    using BF = BlockForm<F>;
    uint32_t d[4];
    const uint32_t w = b.w0;
    if constexpr (BF::BITS == 8) {
        const uint32_t w0 = b.w0, w1 = b.w1;
        if constexpr (BF::CODE == kCodeE4M3) {
            const u32x2 a = e4m3x4_to_bf16x4(w0), b = e4m3x4_to_bf16x4(w1);
            d[0] = a.x; d[1] = a.y; d[2] = b.x; d[3] = b.y;
        } else {
            d[0] = pk_bf16(byte_float<0>(w0), byte_float<1>(w0));
            d[1] = pk_bf16(byte_float<2>(w0), byte_float<3>(w0));
            d[2] = pk_bf16(byte_float<0>(w1), byte_float<1>(w1));
            d[3] = pk_bf16(byte_float<2>(w1), byte_float<3>(w1));
        }
    } else {
        if constexpr (BF::CODE == kCodeE2M1) {
            if constexpr (BF::B == 16) {
                const float s = e4m3_float(b.s & 255u);
                const ts_f32x2 c0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 0);
                const ts_f32x2 c1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 1);
                const ts_f32x2 c2 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 2);
                const ts_f32x2 c3 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(w, 1.0f, 3);
                d[0] = pk_bf16(c0[0] * s, c0[1] * s); d[1] = pk_bf16(c1[0] * s, c1[1] * s);
                d[2] = pk_bf16(c2[0] * s, c2[1] * s); d[3] = pk_bf16(c3[0] * s, c3[1] * s);
            } else {
                d[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 0));
                d[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 1));
                d[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 2));
                d[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, 1.0f, 3));
            }
        } else {
            // Nibble n as the signed byte 16 (n - 8): high nibbles in place, low ones shifted up.
            const uint32_t t = w ^ 0x88888888u, hi = t & 0xf0f0f0f0u, lo = (t << 4) & 0xf0f0f0f0u;
            if constexpr (BF::HALVES) {
                d[0] = pk_bf16(byte_float<0>(lo), byte_float<1>(lo)); d[1] = pk_bf16(byte_float<2>(lo), byte_float<3>(lo));
                d[2] = pk_bf16(byte_float<0>(hi), byte_float<1>(hi)); d[3] = pk_bf16(byte_float<2>(hi), byte_float<3>(hi));
            } else {
                d[0] = pk_bf16(byte_float<0>(lo), byte_float<0>(hi)); d[1] = pk_bf16(byte_float<1>(lo), byte_float<1>(hi));
                d[2] = pk_bf16(byte_float<2>(lo), byte_float<2>(hi)); d[3] = pk_bf16(byte_float<3>(lo), byte_float<3>(hi));
            }
        }
    }
    if constexpr (BF::SCALE == kScaleF16) {
        if (BF::B == 32 || Q == 0)
            scale = f16_value(b.s & 255u, (b.s >> 8) & 255u) * (BF::CODE == kCodeNibble ? 0.0625f : 1.0f);
    } else if constexpr (BF::SCALE == kScaleE8M0) {
        scale = e8m0_value(b.s & 255u);
    }
    return as_bf16x8(u32x4{d[0], d[1], d[2], d[3]});
}

template <int F, int MT, bool XF32, bool SILU>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void block_lanes_kernel(StreamParams p) {
    using BF = BlockForm<F>;
    using P = Shape<F, MT, XF32, SILU>;
    constexpr int S = P::S, C = P::C, PARTS = P::PARTS;
    constexpr bool FOLD = BF::B == 16;  // the codes hold their scale: one sum over all of k
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const uint32_t t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t col = lane & 15, grp = lane >> 4;
    const uint32_t slice = wave / C, wc = wave % C;
    const uint32_t N = p.n, M = p.m;
    const uint32_t n0 = blockIdx.x * P::OC + wc * (SILU ? 16 : 32);  // the wave's first output column
    char *ring = lds + wave * (P::RING * P::SLOT), *xbuf = lds + kWaves * P::RING * P::SLOT;

    const uint32_t units = p.k / kUnit, steps = (units + S - 1) / S;
    const uint32_t sb = (uint32_t)((uint64_t)steps * blockIdx.y / p.splits);
    const uint32_t se = (uint32_t)((uint64_t)steps * (blockIdx.y + 1) / p.splits);

    // Byte offsets (at unit 0, from the first row) of the words this lane's loads bring: word
    // 64 i + lane of the unit's 32 rows. Rows past the end read the last one (never stored).
    const uint32_t row_bytes = p.k / BF::B * BF::BB;
    uint32_t woff[P::LOADS];
#pragma unroll
    for (int i = 0; i < P::LOADS; i++) {
        const uint32_t f = min(64 * (uint32_t)i + lane, 32u * P::WORDS - 1), r = f / P::WORDS, w = f % P::WORDS;
        const uint32_t row = SILU ? (r < 16 ? 0 : N) + min(n0 + (r & 15), N - 1) : min(n0 + r, N - 1);
        woff[i] = row * row_bytes + 4 * w;
    }
    // Buffer loads, not global ones: the compiler counts them with the loads of x to registers
    // in order (a global_load_lds in flight makes it wait for every load before it uses x).
    const __amdgpu_buffer_rsrc_t rows =
        __builtin_amdgcn_make_buffer_rsrc((void *)(p.w + BF::HEAD), 0, (SILU ? 2 : 1) * N * row_bytes, kRawBuffer);
    // A last step of fewer units loads its last unit again.
    auto fetch = [&](uint32_t step) {
        const uint32_t u = min(step * S + slice, units - 1);
        const uint32_t at = __builtin_amdgcn_readfirstlane(u * P::BYTES / 4 * 4);
        char *slot = ring + (step % P::RING) * P::SLOT;
#pragma unroll
        for (int i = 0; i < P::LOADS; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (ts_lds *)(slot + i * 256), 4, woff[i], at, 0, 0);
    };

    // x pieces of a step: piece = t + 512 j: row piece / (4 QS), eighth c of the step's k:
    // matrix step q = c / 4, lane group c % 4.
    u32x4 xr[P::PER * PARTS];
    auto load_x = [&](uint32_t step) {
#pragma unroll
        for (int j = 0; j < P::PER; j++) {
            const uint32_t i = t + kThreads * j, c = i % (4 * P::QS), q = c >> 2, g = c & 3;
            const uint32_t row = min(i / (4 * P::QS), M - 1);
            const uint32_t k32 = min(step * (P::QS * 32) + q * 32, p.k - 32);
            const uint32_t lo = k32 + (BF::HALVES ? 4 * g : 8 * g), hi = BF::HALVES ? k32 + 16 + 4 * g : lo + 4;
            const size_t at = (size_t)row * p.k;
            if (XF32) {
                xr[PARTS * j] = *(const u32x4 *)((const float *)p.x + at + lo);
                xr[PARTS * j + PARTS - 1] = *(const u32x4 *)((const float *)p.x + at + hi);
            } else {
                const u32x2 a = *(const u32x2 *)((const uint16_t *)p.x + at + lo);
                const u32x2 b = *(const u32x2 *)((const uint16_t *)p.x + at + hi);
                xr[PARTS * j] = u32x4{a.x, a.y, b.x, b.y};
            }
        }
    };
    // Operand q of row tile mt: 1 KiB a part, lane (row, g)'s 16 bytes at 256 g + 16 (row ^ c)
    // (the stores of a row's pieces and the reads of a tile both spread over the banks).
    auto store_x = [&](uint32_t step) {
        char *buf = xbuf + (step & 1) * P::XBUF;
#pragma unroll
        for (int j = 0; j < P::PER; j++) {
            const uint32_t i = t + kThreads * j, c = i % (4 * P::QS), q = c >> 2, g = c & 3, row = i / (4 * P::QS);
            if (P::PIECES % kThreads && i >= (uint32_t)P::PIECES) continue;
            char *at = buf + (q * MT + (row >> 4)) * (PARTS * 1024) + g * 256 + (((row & 15) ^ (c & 15)) << 4);
            if (XF32) {
                uint32_t h[4], l[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const u32x4 v = xr[PARTS * j + (e >> 1) * (PARTS - 1)];
                    const float a = __uint_as_float(v[2 * (e & 1)]), b = __uint_as_float(v[2 * (e & 1) + 1]);
                    h[e] = pk_bf16(a, b);
                    l[e] = pk_bf16(a - lo_bf16(h[e]), b - hi_bf16(h[e]));
                }
                *(u32x4 *)at = u32x4{h[0], h[1], h[2], h[3]};
                *(u32x4 *)(at + 1024) = u32x4{l[0], l[1], l[2], l[3]};
            } else {
                *(u32x4 *)at = xr[PARTS * j];
            }
        }
    };

    f32x4 acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i][0] = acc[i][1] = f32x4{0, 0, 0, 0};

    auto multiply = [&](uint32_t s) {
        const uint32_t u = s * S + slice;
        if (u >= units) return;  // wave-uniform: a last step's missing unit
        const char *xs = xbuf + (s & 1) * P::XBUF;
        const uint32_t *slot = (const uint32_t *)(ring + (s % P::RING) * P::SLOT);
        const uint32_t par = BF::B == 128 ? u & 1 : 0;
        Packed raw[2][4];
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const uint32_t *row = slot + (r * 16 + col) * P::WORDS;
            raw[r][0] = packed<F, 0>(row, grp, par);
            raw[r][1] = packed<F, 1>(row, grp, par);
            raw[r][2] = packed<F, 2>(row, grp, par);
            raw[r][3] = packed<F, 3>(row, grp, par);
        }
        f32x4 d[MT][2];
        float sc[2] = {1.0f, 1.0f};
        auto part = [&](auto qc) {
            constexpr int Q = decltype(qc)::value;
            const uint32_t q = slice * 4 + Q, c = 4 * q + grp;
            bf16x8 w[2];
#pragma unroll
            for (int r = 0; r < 2; r++) w[r] = decode<F, Q>(raw[r][Q], sc[r]);
            constexpr bool first = BF::B == 128 ? Q == 0 : true, last = BF::B == 128 ? Q == 3 : true;
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const char *at = xs + (q * MT + i) * (PARTS * 1024) + grp * 256 + ((col ^ (c & 15)) << 4);
                const bf16x8 hi = as_bf16x8(*(const u32x4 *)at);
                bf16x8 lo = hi;
                if (XF32) lo = as_bf16x8(*(const u32x4 *)(at + 1024));
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    if (FOLD) {
                        acc[i][r] = mfma16(hi, w[r], acc[i][r]);
                        if (XF32) acc[i][r] = mfma16(lo, w[r], acc[i][r]);
                        continue;
                    }
                    d[i][r] = mfma16(hi, w[r], first ? f32x4{0, 0, 0, 0} : d[i][r]);
                    if (XF32) d[i][r] = mfma16(lo, w[r], d[i][r]);
                    if (last)
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[i][r][e] += sc[r] * d[i][r][e];
                }
            }
        };
        part(std::integral_constant<int, 0>());
        part(std::integral_constant<int, 1>());
        part(std::integral_constant<int, 2>());
        part(std::integral_constant<int, 3>());
    };

    load_x(sb);
    fetch(sb);
    store_x(sb);
    if (sb + 1 < se) {
        load_x(sb + 1);
        if (P::RING == 3) fetch(sb + 1);
    }
    // The barrier of a step ends the reads of the step before (its x buffer and ring slot are
    // refilled now) and publishes this step's x. A wave's loads return in the order it issued
    // them: x a step ahead, then the unit of RING - 1 steps ahead, so once at most the last
    // unit's loads are outstanding this step's unit and the next step's x are here.
    uint32_t s = sb;
    for (; s + 2 < se; s++) {
        if (P::RING == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P::LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        store_x(s + 1);
        load_x(s + 2);
        fetch(s + P::RING - 1);
        multiply(s);
    }
    for (; s < se; s++) {  // the last two steps: nothing further to load but RING 2's last unit
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        if (s + 1 < se) {
            store_x(s + 1);
            if (P::RING == 2) fetch(s + 1);
        }
        multiply(s);
    }

    if (S == 2) {  // the odd units' sums join the even units'
        __syncthreads();
        f32x4 *sums = (f32x4 *)lds + wc * (2 * MT * 64) + lane;
        if (slice == 1)
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int r = 0; r < 2; r++) sums[(i * 2 + r) * 64] = acc[i][r];
        __syncthreads();
        if (slice == 1) return;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int r = 0; r < 2; r++) acc[i][r] += sums[(i * 2 + r) * 64];
    }

    // Lane (col, grp) holds x rows 16 i + 4 grp + e of weight row col of each tile.
    const float head = BF::HEAD ? *(const float *)p.w : 1.0f;  // Block::dot: head * sum
#pragma unroll
    for (int r = 0; r < (SILU ? 1 : 2); r++) {
        const uint32_t n = n0 + (SILU ? 0 : r * 16) + col;
        if (n >= N) continue;
        if (p.part) {
            const size_t mn = (size_t)M * N;
            float *dst = p.part + (size_t)blockIdx.y * (SILU ? 2 : 1) * mn;
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t m = 16 * i + 4 * grp + e;
                    if (m >= M) continue;
                    put_part(dst + (size_t)m * N + n, acc[i][r][e]);
                    if (SILU) put_part(dst + mn + (size_t)m * N + n, acc[i][1][e]);
                }
            continue;
        }
        float val[MT * 4];
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float g = head * acc[i][r][e], u = head * acc[i][1][e];
                val[4 * i + e] = SILU ? g / (1.0f + expf(-g)) * u : g;
            }
        auto row_of = [&](int e) { return 16 * (uint32_t)(e / 4) + 4 * grp + (uint32_t)(e % 4); };
        if (p.after.count)
            after_values<MT * 4, false>(p.after, val, [&](int e) { return (size_t)row_of(e) * N + n; },
                                        [&](int e) { return row_of(e) < M; });
#pragma unroll
        for (int e = 0; e < MT * 4; e++) {
            const uint32_t m = row_of(e);
            if (m >= M) continue;
            const size_t at = (size_t)m * N + n;
            float v = val[e];
            if (p.stages & TS_AFTER_ADD) v += p.a0[at];
            if (p.out_bf16) ((uint16_t *)p.out)[at] = bf16_bits(v);
            else ((float *)p.out)[at] = v;
        }
    }
}

struct Choice {
    const void *kernel;
    hipError_t (*ready)();  // raises the kernel's dynamic LDS size, once
    int lds, cols, step;    // dynamic LDS, output columns of a group, units of a step
};

template <int F, int MT, bool XF32, bool SILU>
hipError_t ready() {
    static const hipError_t attr =
        hipFuncSetAttribute((const void *)block_lanes_kernel<F, MT, XF32, SILU>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, Shape<F, MT, XF32, SILU>::LDS);
    return attr;
}

template <int F, int MT, bool XF32, bool SILU>
Choice choice() {
    using P = Shape<F, MT, XF32, SILU>;
    return Choice{(const void *)block_lanes_kernel<F, MT, XF32, SILU>, ready<F, MT, XF32, SILU>, P::LDS, P::OC, P::S};
}

template <int F, int MT>
Choice pick2(bool xf, bool silu) {
    return xf ? (silu ? choice<F, MT, true, true>() : choice<F, MT, true, false>())
              : (silu ? choice<F, MT, false, true>() : choice<F, MT, false, false>());
}

template <int F>
Choice pick1(uint32_t mt, bool xf, bool silu) {
    return mt == 1 ? pick2<F, 1>(xf, silu) : mt == 2 ? pick2<F, 2>(xf, silu)
         : mt == 3 ? pick2<F, 3>(xf, silu) : pick2<F, 4>(xf, silu);
}

Choice pick(const ts_linear_args *a) {
    const uint32_t mt = (a->m + 15) / 16;
    const bool xf = a->x_dtype == TS_F32, silu = a->stages & TS_AFTER_SILU_MUL;
    switch (a->w_dtype) {
    case TS_Q8_0: return pick1<0>(mt, xf, silu);
    case TS_MXFP8: return pick1<1>(mt, xf, silu);
    case TS_INT4_G32: return pick1<2>(mt, xf, silu);
    case TS_Q4_0: return pick1<3>(mt, xf, silu);
    case TS_NVFP4: return pick1<4>(mt, xf, silu);
    case TS_MXFP4: return pick1<5>(mt, xf, silu);
    default: return pick1<6>(mt, xf, silu);
    }
}

// The k split: what takes the fewest steps, counting rounds of resident groups, three
// steps to fill a group's pipeline and six for the second kernel.
uint32_t plan_splits(const ts_linear_args *a, const Choice &c) {
    const uint32_t groups = (a->n + c.cols - 1) / c.cols, units = a->k / kUnit;
    const uint32_t steps = (units + c.step - 1) / c.step;
    const uint32_t resident = kCus * std::max(1, kMaxLds / c.lds);
    uint32_t best = 1, cost = ~0u;
    for (uint32_t s = 1; s <= 16 && 2 * s <= std::max(steps, 2u); s++) {
        const uint32_t rounds = (groups * s + resident - 1) / resident;
        const uint32_t took = rounds * ((steps + s - 1) / s + 3) + (s > 1 ? 6 : 0);
        if (took < cost) {
            cost = took;
            best = s;
        }
    }
    return best;
}

// Lanes address the tensor with 32-bit offsets.
bool fits(const ts_linear_args *a) {
    const BlockShape bs = block_shape(a->w_dtype);
    const uint64_t rows = (uint64_t)a->n * ((a->stages & TS_AFTER_SILU_MUL) ? 2 : 1);
    return a->m > 4 && a->m <= 64 && a->k % kUnit == 0 && rows * (a->k / bs.block) * bs.bytes < (1ull << 32);
}

}  // namespace

size_t block_lanes_workspace(const ts_linear_args *a) {
    const BlockShape bs = block_shape(a->w_dtype);
    if (a->n < 1 || a->k < 128 || a->k % (4 * bs.block) || !fits(a)) return 0;
    const uint32_t s = plan_splits(a, pick(a));
    if (s <= 1) return 0;
    return (size_t)s * a->m * a->n * ((a->stages & TS_AFTER_SILU_MUL) ? 2 : 1) * sizeof(float);
}

// m 5..64; 1 when the product is not for this kernel. Without the workspace that
// block_lanes_workspace names, k is not split.
int block_lanes_launch(const ts_linear_args *a, void *stream) {
    const int bad = block_check(a, "tiled");
    if (bad) return bad;
    if (!fits(a) || (a->stages & ~(TS_AFTER_ADD | TS_AFTER_SILU_MUL))) return 1;
    StreamParams p;
    p.x = a->x; p.w = (const uint8_t *)a->w; p.a0 = a->a0; p.out = a->out;
    p.m = a->m; p.n = a->n; p.k = a->k; p.stages = a->stages; p.out_bf16 = a->out_dtype == TS_BF16;
    int rc = linear_after(a, "tiled (block form)", &p.after);
    if (rc) return rc;
    const Choice c = pick(a);
    const size_t need = block_lanes_workspace(a);
    const bool split = need && a->workspace && a->workspace_bytes >= need && aligned(a->workspace, 16);
    p.splits = split ? plan_splits(a, c) : 1;
    p.part = split ? (float *)a->workspace : nullptr;
    hipError_t e = c.ready();
    if (e != hipSuccess) return hip_status(e, "lanes (block form): LDS attribute");
    void *args[] = {(void *)&p};
    e = hipLaunchKernel(c.kernel, dim3((a->n + c.cols - 1) / c.cols, p.splits), dim3(kThreads), args, c.lds,
                        (hipStream_t)stream);
    if (e != hipSuccess) return hip_status(e, "lanes (block form): launch");
    if (!split) return TS_OK;
    SplitSum f = {};
    f.part = p.part; f.splits = p.splits; f.out = a->out; f.a0 = a->a0;
    f.head = a->w_dtype == TS_NVFP4 ? (const float *)a->w : nullptr;
    f.m = a->m; f.n = a->n; f.stages = a->stages; f.out_bf16 = p.out_bf16; f.after = p.after;
    return split_finish(f, stream);
}

}  // namespace ts
