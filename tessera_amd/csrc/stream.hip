// Few rows (m 5..64) on the matrix unit, weights streamed: bf16, e4m3 and every block form.
//
// Replaces the reference's lanes rule (engine/rules/linear/src/lanes.rs:17-143), also where
// it reads a block form through its load (every form of engine/plan/codegen/src/form.rs:10-93
// and block.rs:251-291): the decode product of a batch. Block forms with the arithmetic of the
// many-row kernel (blockmat.hip): codes exact in bf16, one matrix-unit sum per block from
// zero, times the block's scale, added in f32.
//
// gfx950 design. At these row counts the weights are the work: each byte is read once and
// should arrive at the rate of HBM.
//  * A wave owns 32 weight rows (pairs: 16 rows and the 16 rows of the same columns in the
//    second half) and streams them in units through its own LDS ring, filled with buffer loads
//    straight to LDS, two units ahead of their use where LDS allows. No barrier waits on
//    weights: a wave waits for its own loads only. A unit of a row is 128 codes of a block
//    form (4-byte loads: blocks are 9 to 66 bytes, a unit is always whole words), or 128
//    bytes of bf16 or e4m3 (16-byte loads, chunks XOR-swizzled by row).
//  * The rows of x are shared: a step of S units is staged in LDS as ready matrix operands,
//    double-buffered, its loads issued a step ahead of the store and before the weights' own,
//    one barrier a step. (A wave's loads return in order: x issued behind the weights that
//    follow it, one chunk ahead, as the kernel in lanes.hip does, waits out the whole weight
//    ring every chunk.) With S > 1 the waves take the units of a step in S slices, which
//    gives narrower groups and fewer operand reads; the slices' sums meet in LDS at the end.
//  * Block forms: lane (c, g) decodes its 8 codes of weight row c straight from LDS words into
//    the second operand, so the sums leave the matrix unit with column c = the lane's own row
//    and the block scale is a register of the lane. The 8 codes of 32 are g's quarter of the
//    block's bytes (q4_0: the low nibbles of four bytes, then the high ones; x is staged in
//    the same order). Nibbles convert as signed bytes 16 (code - 8), the 16 taken out of the
//    scale (both exact); e2m1 and e4m3 on gfx950's bf16 conversions; nvfp4 folds its e4m3
//    scale into the codes (exact in bf16).
//  * RmsNorm before the product (m <= 16): x enters times the gain, each row's sum of squares
//    is taken from the pieces as they are staged, and its inverse root scales the finished
//    sums. (lanes.hip normalizes in every group: 16 rows by the 151936 x 1024 lm_head read x
//    twice in each of 2374 groups, 166 us; here 69.)
//  * Where the columns alone do not give every CU its groups, k is split across groups: raw
//    sums to the workspace, added in split order by split_finish.
// bf16 and e4m3 against lanes.hip: 8 bf16 rows by e4m3 2 x 14336 x 4096 36 -> 30.5 us, 4096 x
// 14336 21 -> 16.5; 64 f32 rows by e4m3 2 x 14336 x 4096 96 -> 66 us; 40 f32 rows by e4m3 2 x
// 9728 x 2560 44 -> 22 us; 16 f32 rows with the norm by bf16 4096 x 1024 19.3 -> 8.2 us.
// Block forms against the 64 x 64 tiles of blockmat.hip, which these sizes went to (64 groups,
// each a serial chain over all of k): 16 f32 rows by int4_g32 2 x 14336 x 4096 156 -> 28 us,
// 4096 x 14336 343 -> 18 us; 8 bf16 rows by q8_0 79 -> 37 and 175 -> 20 us; 64 f32 rows by
// int4_g32 157 -> 52 and 346 -> 31 us. At 16 rows what bounds it now is the decode (14 vector
// operations per 8 nibbles, then the scaling of the block sums); at 64 the matrix unit.
#include <algorithm>
#include <type_traits>

#include "blockform.h"

namespace ts {

namespace {

constexpr uint32_t kCus = 256;
constexpr int kMaxLds = 160 * 1024;
constexpr int kRawBuffer = 0x00020000;  // buffer descriptor word 3: a raw buffer of 32-bit data
constexpr int kBf16 = 7, kE4M3 = 8;     // forms past the seven block forms

struct StreamParams {
    const void *x;
    const uint8_t *w;  // block forms: the packed tensor (head included)
    const uint16_t *w_scale;
    const float *gain;
    const float *a0;
    void *out;
    float *part;   // split sums, or NULL
    float *sumsq;  // NORM: each split's sums of squares [split][m], behind the split sums
    uint32_t m, n, k;
    uint32_t stages;
    float eps;
    int out_bf16, pair_sum;
    uint32_t splits;
    ts_after after;  // stage chain (count 0: none)
};

// A unit of a weight row: UNIT values in BYTES bytes.
template <int F>
struct Unit {
    using BF = BlockForm<F < 7 ? F : 0>;
    static constexpr bool BLOCK = F < 7;
    static constexpr int UNIT = F == kBf16 ? 64 : 128, STEPS = UNIT / 32;  // matrix steps of 32
    // Block forms: whole blocks of 32 or 16 codes, or one block of 128 (66 bytes: the odd
    // units start on a half word, so a unit is loaded from the word it starts in).
    static constexpr int BYTES = BLOCK ? UNIT / BF::B * BF::BB : 128, WORDS = (BYTES + 3) / 4;
    static constexpr int LANE = BLOCK ? 4 : 16;  // bytes a lane loads at once
    static constexpr int LOADS = (32 * WORDS * 4 + 64 * LANE - 1) / (64 * LANE), SLOT = LOADS * 64 * LANE;
    // Groups of 4 waves, two a CU, where a unit is 4 KiB; block units are smaller and their
    // lanes' arithmetic is more, so 8 waves share one staging of x.
    static constexpr int WAVES = BLOCK ? 8 : 4;
};

template <int F, int MT, bool XF32, bool PAIR, int S>
struct Shape {
    using U = Unit<F>;
    static constexpr int WAVES = U::WAVES, C = WAVES / S, THREADS = 64 * WAVES;
    static constexpr int PARTS = XF32 ? 2 : 1;
    static constexpr int QS = U::STEPS * S;  // matrix steps of one step
    static constexpr int XBUF = QS * MT * PARTS * 1024;
    // Two slots instead of three where that lets two groups of 4 waves share a CU.
    static constexpr int RING = 2 * XBUF + 3 * WAVES * U::SLOT <= (WAVES == 4 ? kMaxLds / 2 : kMaxLds) ? 3
                              : 2 * XBUF + 2 * WAVES * U::SLOT <= kMaxLds / 2 || WAVES == 8 ? 2 : 3;
    static constexpr int LDS = 2 * XBUF + RING * WAVES * U::SLOT;
    static constexpr int OC = C * (PAIR ? 16 : 32);  // output columns of a group
    static constexpr int PIECES = 16 * MT * QS * 4, PER = (PIECES + THREADS - 1) / THREADS;
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

template <int F, int MT, bool XF32, bool PAIR, int S, bool NORM>
__global__ __launch_bounds__(Unit<F>::WAVES * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void stream_kernel(
    StreamParams p) {
    using U = Unit<F>;
    using BF = typename U::BF;
    using P = Shape<F, MT, XF32, PAIR, S>;
    constexpr int C = P::C, PARTS = P::PARTS, THREADS = P::THREADS;
    static_assert(P::LDS <= kMaxLds && THREADS % (4 * P::QS) == 0, "LDS and a step's pieces of x");
    constexpr bool HALVES = U::BLOCK && BF::HALVES;
    constexpr bool FOLD = !U::BLOCK || BF::B == 16;  // no block scales: one sum over all of k
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const uint32_t t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t col = lane & 15, grp = lane >> 4;
    const uint32_t slice = wave / C, wc = wave % C;
    const uint32_t N = p.n, M = p.m;
    const uint32_t n0 = blockIdx.x * P::OC + wc * (PAIR ? 16 : 32);  // the wave's first output column
    char *ring = lds + wave * (P::RING * U::SLOT), *xbuf = lds + P::WAVES * P::RING * U::SLOT;

    const uint32_t units = p.k / U::UNIT, steps = (units + S - 1) / S;
    const uint32_t sb = (uint32_t)((uint64_t)steps * blockIdx.y / p.splits);
    const uint32_t se = (uint32_t)((uint64_t)steps * (blockIdx.y + 1) / p.splits);

    // Byte offsets (at unit 0, from the first row) of what this lane's loads bring: bytes
    // LANE (64 i + lane) of the unit's 32 rows. Rows past the end read the last one (never
    // stored). bf16 and e4m3: chunk c of row r lies at c ^ (r & 7).
    const uint32_t row_bytes = U::BLOCK ? p.k / BF::B * BF::BB : p.k * (F == kBf16 ? 2 : 1);
    uint32_t woff[U::LOADS];
#pragma unroll
    for (int i = 0; i < U::LOADS; i++) {
        uint32_t r, at;
        if (U::BLOCK) {
            const uint32_t f = min(64 * (uint32_t)i + lane, 32u * U::WORDS - 1);
            r = f / U::WORDS;
            at = 4 * (f % U::WORDS);
        } else {
            r = 8 * (uint32_t)i + (lane >> 3);
            at = 16 * ((lane & 7) ^ (lane >> 3));
        }
        const uint32_t row = PAIR ? (r < 16 ? 0 : N) + min(n0 + (r & 15), N - 1) : min(n0 + r, N - 1);
        woff[i] = row * row_bytes + at;
    }
    // Buffer loads, not global ones: the compiler counts them with the loads of x to registers
    // in order (a global_load_lds in flight makes it wait for every load before it uses x).
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(p.w + (U::BLOCK ? BF::HEAD : 0)), 0, (PAIR ? 2 : 1) * N * row_bytes, kRawBuffer);
    // A last step of fewer units loads its last unit again.
    auto fetch = [&](uint32_t step) {
        const uint32_t u = min(step * S + slice, units - 1);
        const uint32_t at = __builtin_amdgcn_readfirstlane(u * U::BYTES / 4 * 4);
        char *slot = ring + (step % P::RING) * U::SLOT;
#pragma unroll
        for (int i = 0; i < U::LOADS; i++) {
            if (U::BLOCK) __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (ts_lds *)(slot + i * 256), 4, woff[i], at, 0, 0);
            else buffer_to_lds16(rows, slot + i * 1024, woff[i], at);
        }
    };

    // x pieces of a step: piece = t + THREADS j: row piece / (4 QS), eighth c of the step's k:
    // matrix step q = c / 4, lane group g = c % 4 (the same c for every j). e4m3: the 16 codes
    // a lane reads at once serve two matrix steps.
    const uint32_t pc = t % (4 * P::QS), pq = pc >> 2, pg = pc & 3;
    const uint32_t klo = F == kE4M3 ? 64 * (pq >> 1) + 16 * pg + 8 * (pq & 1) : 32 * pq + (HALVES ? 4 : 8) * pg;
    const uint32_t khi = HALVES ? klo + 16 : klo + 4;
    u32x4 xr[P::PER * PARTS], gr[NORM ? 2 : 1];
    bool counted = false;  // NORM: the pieces in xr are new ones
    float sq[NORM ? P::PER : 1] = {};
    auto load_x = [&](uint32_t step) {
        const uint32_t k0 = step * (P::QS * 32);
        // Units missing from a last step load the units before them again.
        const uint32_t back = S == 1 || k0 + klo < p.k ? 0 : U::UNIT * ((k0 + klo - p.k) / U::UNIT + 1);
        const uint32_t lo = k0 + klo - back, hi = k0 + khi - back;
        if (NORM) {
            counted = back == 0;
            gr[0] = *(const u32x4 *)(p.gain + lo);
            gr[NORM ? 1 : 0] = *(const u32x4 *)(p.gain + hi);
        }
#pragma unroll
        for (int j = 0; j < P::PER; j++) {
            const size_t at = (size_t)min((t + THREADS * j) / (4 * P::QS), M - 1) * p.k;
            if (XF32) {
                xr[PARTS * j] = *(const u32x4 *)((const float *)p.x + at + lo);
                xr[PARTS * j + PARTS - 1] = *(const u32x4 *)((const float *)p.x + at + hi);
            } else if (HALVES) {
                const u32x2 a = *(const u32x2 *)((const uint16_t *)p.x + at + lo);
                const u32x2 b = *(const u32x2 *)((const uint16_t *)p.x + at + hi);
                xr[PARTS * j] = u32x4{a.x, a.y, b.x, b.y};
            } else {
                xr[PARTS * j] = *(const u32x4 *)((const uint16_t *)p.x + at + lo);
            }
        }
    };
    // Operand q of row tile mt: 1 KiB a part, lane (row, g)'s 16 bytes at 256 g + 16 (row ^ c)
    // (the stores of a row's pieces and the reads of a tile both spread over the banks).
    auto store_x = [&](uint32_t step) {
        char *buf = xbuf + (step & 1) * P::XBUF;
#pragma unroll
        for (int j = 0; j < P::PER; j++) {
            const uint32_t i = t + THREADS * j, row = i / (4 * P::QS);
            if (P::PIECES % THREADS && i >= (uint32_t)P::PIECES) continue;
            char *at = buf + (pq * MT + (row >> 4)) * (PARTS * 1024) + pg * 256 + (((row & 15) ^ (pc & 15)) << 4);
            if (XF32) {
                uint32_t h[4], l[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const u32x4 v = xr[PARTS * j + (e >> 1) * (PARTS - 1)];
                    float a = __uint_as_float(v[2 * (e & 1)]), b = __uint_as_float(v[2 * (e & 1) + 1]);
                    if (NORM) {
                        if (counted) sq[j] += a * a + b * b;
                        const u32x4 g = gr[NORM ? e >> 1 : 0];
                        a *= __uint_as_float(g[2 * (e & 1)]);
                        b *= __uint_as_float(g[2 * (e & 1) + 1]);
                    }
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
        if (S > 1 && u >= units) return;  // wave-uniform: a last step's missing unit
        const char *xs = xbuf + (s & 1) * P::XBUF, *slot = ring + (s % P::RING) * U::SLOT;
        const uint32_t par = U::BLOCK && BF::B == 128 ? u & 1 : 0;
        Packed raw[2][4];
        u32x4 vals[2][4];  // bf16: a matrix step's operand each; e4m3: 16 codes for two steps each
#pragma unroll
        for (int r = 0; r < 2; r++) {
            if constexpr (U::BLOCK) {
                const uint32_t *row = (const uint32_t *)slot + (r * 16 + col) * U::WORDS;
                raw[r][0] = packed<F, 0>(row, grp, par);
                raw[r][1] = packed<F, 1>(row, grp, par);
                raw[r][2] = packed<F, 2>(row, grp, par);
                raw[r][3] = packed<F, 3>(row, grp, par);
            } else {
#pragma unroll
                for (int h = 0; h < 2; h++)
                    vals[r][h] = *(const u32x4 *)(slot + (r * 16 + col) * 128 + (((4 * h + grp) ^ (col & 7)) << 4));
            }
        }
        f32x4 d[MT][2];
        float sc[2] = {1.0f, 1.0f};
        auto part = [&](auto qc) {
            constexpr int Q = decltype(qc)::value;
            const uint32_t q = slice * U::STEPS + Q, c = 4 * q + grp;
            bf16x8 w[2];
#pragma unroll
            for (int r = 0; r < 2; r++) {
                if constexpr (F == kBf16) {
                    w[r] = as_bf16x8(vals[r][Q]);
                } else if constexpr (F == kE4M3) {
                    const u32x4 v = vals[r][Q / 2];
                    const u32x2 a = e4m3x4_to_bf16x4(Q % 2 ? v.z : v.x), b = e4m3x4_to_bf16x4(Q % 2 ? v.w : v.y);
                    w[r] = as_bf16x8(u32x4{a.x, a.y, b.x, b.y});
                } else {
                    w[r] = decode<F, Q>(raw[r][Q], sc[r]);
                }
            }
            constexpr bool first = U::BLOCK && BF::B == 128 ? Q == 0 : true, last = U::BLOCK && BF::B == 128 ? Q == 3 : true;
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
        if constexpr (U::STEPS == 4) {
            part(std::integral_constant<int, 2>());
            part(std::integral_constant<int, 3>());
        }
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
        if (P::RING == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(U::LOADS) : "memory");
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

    // The slices' sums join slice 0's in slice order, and the rows' sums of squares the
    // first 16 threads'.
    constexpr int kSums = 2 * MT * 64;  // f32x4 of one wave column
    float *squares = (float *)(lds + (S - 1) * C * kSums * 16);
    if (S > 1 || NORM) {
        __syncthreads();
        f32x4 *sums = (f32x4 *)lds + wc * kSums + lane;
        if (S > 1 && slice > 0)
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int r = 0; r < 2; r++) sums[(slice - 1) * (C * kSums) + (i * 2 + r) * 64] = acc[i][r];
        if (NORM)
#pragma unroll
            for (int j = 0; j < P::PER; j++)
                if (t + THREADS * j < (uint32_t)P::PIECES) squares[t + THREADS * j] = sq[j];
        __syncthreads();
        if (NORM && t < 16) {
            float ss = 0.0f;
#pragma unroll
            for (int c = 0; c < 4 * P::QS; c++) ss += squares[t * (4 * P::QS) + c];
            squares[P::PIECES + t] = ss;
            if (p.part && blockIdx.x == 0 && t < M) put_part(p.sumsq + blockIdx.y * M + t, ss);
        }
        if (NORM) __syncthreads();
        if (slice > 0) return;
#pragma unroll
        for (int o = 1; o < S; o++)
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int r = 0; r < 2; r++) acc[i][r] += sums[(o - 1) * (C * kSums) + (i * 2 + r) * 64];
    }

    // Lane (col, grp) holds x rows 16 i + 4 grp + e of weight row col of each tile.
    const float head = U::BLOCK && BF::HEAD ? *(const float *)p.w : 1.0f;  // Block::dot: head * sum
#pragma unroll
    for (int r = 0; r < (PAIR ? 1 : 2); r++) {
        const uint32_t n = n0 + (PAIR ? 0 : r * 16) + col;
        if (n >= N) continue;
        if (p.part) {
            const size_t mn = (size_t)M * N;
            float *dst = p.part + (size_t)blockIdx.y * (PAIR ? 2 : 1) * mn;
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t m = 16 * i + 4 * grp + e;
                    if (m >= M) continue;
                    put_part(dst + (size_t)m * N + n, acc[i][r][e]);
                    if (PAIR) put_part(dst + mn + (size_t)m * N + n, acc[i][1][e]);
                }
            continue;
        }
        const float sg = F == kE4M3 ? bf16_float(p.w_scale[n]) : head;
        const float su = F == kE4M3 && PAIR ? bf16_float(p.w_scale[N + n]) : head;
        float val[MT * 4];
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float g = acc[i][r][e], u = acc[i][1][e];
                if (NORM) {
                    const float inv = 1.0f / sqrtf(squares[P::PIECES + 16 * i + 4 * grp + e] / (float)p.k + p.eps);
                    g *= inv;
                    u *= inv;
                }
                g *= sg;
                u *= su;
                val[4 * i + e] = !PAIR ? g : p.pair_sum ? g + u : g / (1.0f + expf(-g)) * u;
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
    int lds, cols, span, threads;  // dynamic LDS, output columns of a group, k of a step
    int work;                      // operands of x a wave multiplies in a step
    int slices, tiles, parts;      // S, row tiles of 16, bf16 parts of x
};

template <int F, int MT, bool XF32, bool PAIR, int S, bool NORM>
hipError_t ready() {
    static const hipError_t attr =
        hipFuncSetAttribute((const void *)stream_kernel<F, MT, XF32, PAIR, S, NORM>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, Shape<F, MT, XF32, PAIR, S>::LDS);
    return attr;
}

template <int F, int MT, bool XF32, bool PAIR, int S, bool NORM = false>
Choice choice() {
    using P = Shape<F, MT, XF32, PAIR, S>;
    return Choice{(const void *)stream_kernel<F, MT, XF32, PAIR, S, NORM>, ready<F, MT, XF32, PAIR, S, NORM>, P::LDS,
                  P::OC, S * Unit<F>::UNIT, P::THREADS, Unit<F>::STEPS * MT * P::PARTS, S, MT, P::PARTS};
}

struct Plan {
    Choice c;
    uint32_t splits;
    float cost;
};

constexpr uint32_t kMostSplits = 32;

bool pair_of(const ts_linear_args *a) { return (a->stages & TS_AFTER_SILU_MUL) || a->w_dtype == TS_F32_PARTS; }

// Plain weights of up to this many bytes are small: what counts is latency, and lanes.hip may be
// the shorter way.
constexpr uint64_t kSmall = 8u << 20;

uint64_t plain_bytes(const ts_linear_args *a) {
    return (uint64_t)a->n * a->k * (pair_of(a) ? 2 : 1) * (a->w_dtype == TS_E4M3 ? 1 : 2);
}

bool small(const ts_linear_args *a) { return !block_form(a->w_dtype) && plain_bytes(a) <= kSmall; }

// What a choice takes with k split s ways, us: its start, the steps of each round of resident
// groups, and for a split the second kernel and its sums. For block forms and small plain
// weights, fits to products timed at every S and 1 to 16 splits (128 to 14336 weight rows of
// 1024 to 8192, 8 to 64 rows, both row types, pairs, weights from HBM and from the caches; mean
// error 2% for block forms, 8% for plain ones). What these choose takes 0.3% (block forms) and 1%
// (plain) more than the best choice, where the rule of the large plain weights took 8% and
// 7%: 48 bf16 rows by int4_g32 14336 x 2048 unsplit 30.7 us, in 4 splits 18.5; by bf16 1024 x
// 2048 unsplit 12.0, in 8 splits 7.7.
float took_us(const ts_linear_args *a, const Choice &c, uint32_t s, uint32_t resident) {
    const bool block = block_form(a->w_dtype), pair = pair_of(a);
    const uint32_t groups = (a->n + c.cols - 1) / c.cols * s, steps = (a->k + c.span - 1) / c.span, each = (steps + s - 1) / s;
    const uint32_t rounds = (groups + resident - 1) / resident;
    const float mt = (float)c.tiles, x = (float)(c.slices * c.tiles * c.parts), u = a->w_dtype == TS_E4M3 ? 2.0f : 1.0f;
    const float step = block ? (c.slices == 2 ? 0.85f + 0.13f * x : 1.3f + 0.12f * x)
                             : 0.4f + u * (0.027f * x + 0.025f * mt * c.parts + 0.031f * mt * (c.parts - 1));
    float t = (block ? 2.5f + 0.55f * mt : 3.18f + 0.33f * mt + (c.tiles == 4 ? 0.16f : 0.0f)) + rounds * each * step +
              (rounds - 1) * (block ? 1.0f : 0.92f);
    if (s > 1) {
        const float sums = 4e-6f * s * std::max(a->m, 16u) * a->n * (pair ? 2 : 1);
        t += block ? 2.9f - 0.38f * mt + 0.55f * sums : 2.94f - 0.38f * mt + (pair ? 0.81f : 0.0f) + 0.62f * sums;
    }
    return t;
}

// The k split of a choice: what takes the least time. Large plain weights: in steps of a group
// (~0.6 us, more where a step's matrix work outlasts its loads), rounds of resident groups,
// three steps to fill each one's pipeline, and for a split the time of six for the second
// kernel and its sums' way to memory and back (1.3 MB a step). Measured over S and splits: 16
// rows by bf16 4096 x 1536 7.7 us at S 4 unsplit, 8.8 at S 2 in 6 and S 1 in 8; 64 f32 rows by
// 2 x 3072 x 1024 14.1 us in 4 splits, 15.9 in 8; 16 by 2 x 1536 x 4096 11.7 at S 4 in 4, 13.1
// at S 1 in 16; 8 by e4m3 2 x 14336 x 4096 29.3 to 30.6 whichever.
Plan plan_splits(const ts_linear_args *a, const Choice &c, uint32_t most) {
    const uint32_t groups = (a->n + c.cols - 1) / c.cols, steps = (a->k + c.span - 1) / c.span;
    // Two waves a SIMD: one group of 8 a CU, two of 4 where their LDS allows. (Counted by LDS
    // alone, 8 bf16 rows by int4_g32 2 x 14336 x 4096 were split in two, 28.6 us against 23.4
    // unsplit, and 4096 x 14336 in 14, 18.6 against 14.6 in 8.)
    const uint32_t resident = kCus * std::min(8 * 64 / c.threads, kMaxLds / c.lds);
    const float sums = (float)a->m * a->n * (pair_of(a) ? 2 : 1) * sizeof(float);
    const float step = std::max(1.0f, c.work / 12.0f);
    const bool block = block_form(a->w_dtype), us = block || small(a);
    Plan best = {c, 1, 1e30f};
    for (uint32_t s = 1; s <= std::min({steps, most, us && !block ? 16u : kMostSplits}); s++) {  // 16: the fit's range
        // One step of little matrix work fills no pipeline.
        if (us && !block && s > 1 && 2 * s > steps && c.tiles * c.parts < 4) break;
        const uint32_t rounds = (groups * s + resident - 1) / resident;
        const float took = us ? took_us(a, c, s, resident)
                              : (float)(rounds * ((steps + s - 1) / s + 3)) * step + (s > 1 ? 6.0f + s * sums / 1.3e6f : 0.0f);
        if (took < best.cost) {
            best.splits = s;
            best.cost = took;
        }
    }
    return best;
}

// Block forms: S 2 up to 32 rows, else 1 (the operands of x outgrow LDS).
template <int F, int MT>
Plan plan_block(const ts_linear_args *a, uint32_t most) {
    constexpr int S = MT <= 2 ? 2 : 1;
    const bool pair = pair_of(a);
    return plan_splits(a,
                       a->x_dtype == TS_F32 ? (pair ? choice<F, MT, true, true, S>() : choice<F, MT, true, false, S>())
                                            : (pair ? choice<F, MT, false, true, S>() : choice<F, MT, false, false, S>()),
                       most);
}

// bf16 and e4m3: groups of 32 (S 4), 64 or 128 columns, by the plan; S 4 only where two groups
// still share a CU, S 2 where the operands of x fit.
template <int F, int MT, bool XF32, bool PAIR, bool NORM>
Plan plan_plain(const ts_linear_args *a, uint32_t most) {
    Plan best = plan_splits(a, choice<F, MT, XF32, PAIR, 1, NORM>(), most);
    if constexpr (Shape<F, MT, XF32, PAIR, 2>::LDS <= kMaxLds) {
        const Plan p = plan_splits(a, choice<F, MT, XF32, PAIR, 2, NORM>(), most);
        if (p.cost <= best.cost) best = p;
    }
    if constexpr (Shape<F, MT, XF32, PAIR, 4>::LDS <= kMaxLds / 2) {
        const Plan p = plan_splits(a, choice<F, MT, XF32, PAIR, 4, NORM>(), most);
        if (p.cost <= best.cost) best = p;
    }
    return best;
}

template <int F, int MT>
Plan plan_of(const ts_linear_args *a, uint32_t most) {
    if constexpr (Unit<F>::BLOCK) {
        return plan_block<F, MT>(a, most);
    } else {
        const bool pair = pair_of(a);
        if constexpr (MT == 1)
            if (a->stages & TS_BEFORE_RMS_NORM)
                return pair ? plan_plain<F, 1, true, true, true>(a, most) : plan_plain<F, 1, true, false, true>(a, most);
        if (a->x_dtype == TS_F32)
            return pair ? plan_plain<F, MT, true, true, false>(a, most) : plan_plain<F, MT, true, false, false>(a, most);
        return pair ? plan_plain<F, MT, false, true, false>(a, most) : plan_plain<F, MT, false, false, false>(a, most);
    }
}

template <int F>
Plan plan_rows(const ts_linear_args *a, uint32_t most) {
    const uint32_t mt = (a->m + 15) / 16;
    return mt == 1 ? plan_of<F, 1>(a, most) : mt == 2 ? plan_of<F, 2>(a, most)
         : mt == 3 ? plan_of<F, 3>(a, most) : plan_of<F, 4>(a, most);
}

// most: the splits that the workspace holds.
Plan plan(const ts_linear_args *a, uint32_t most = kMostSplits) {
    switch (a->w_dtype) {
    case TS_Q8_0: return plan_rows<0>(a, most);
    case TS_MXFP8: return plan_rows<1>(a, most);
    case TS_INT4_G32: return plan_rows<2>(a, most);
    case TS_Q4_0: return plan_rows<3>(a, most);
    case TS_NVFP4: return plan_rows<4>(a, most);
    case TS_MXFP4: return plan_rows<5>(a, most);
    case TS_INT4_G128: return plan_rows<6>(a, most);
    case TS_E4M3: return plan_rows<kE4M3>(a, most);
    default: return plan_rows<kBf16>(a, most);
    }
}

// Whole units of k, and lanes that address the weights with 32-bit offsets.
bool fits(const ts_linear_args *a) {
    const bool block = block_form(a->w_dtype), e4m3 = a->w_dtype == TS_E4M3;
    if (!block && !e4m3 && a->w_dtype != TS_BF16 && a->w_dtype != TS_F32_PARTS) return false;
    const uint64_t rows = (uint64_t)a->n * (pair_of(a) ? 2 : 1);
    const BlockShape bs = block ? block_shape(a->w_dtype) : BlockShape{1, e4m3 ? 1u : 2u, 0};
    return a->m > 4 && a->m <= 64 && a->n >= 1 && a->k >= 128 && a->k % (block || e4m3 ? 128 : 64) == 0 &&
           a->k % bs.block == 0 && rows * (a->k / bs.block) * bs.bytes < (1ull << 32);
}

// The sums of one split.
size_t split_bytes(const ts_linear_args *a) {
    return ((size_t)a->m * a->n * (pair_of(a) ? 2 : 1) + ((a->stages & TS_BEFORE_RMS_NORM) ? a->m : 0)) * sizeof(float);
}

}  // namespace

bool stream_fits(const ts_linear_args *a) { return fits(a); }

// Small products go where the times say (a norm is cheaper here at any size, and lanes.hip takes
// 1.7 times as long for a k that is no multiple of its 128): lanes.hip starts sooner and splits
// finer, here a step takes less. lanes.hip's time is a fit to the same
// products (mean error 4%). With weights from HBM, 64 bf16 rows by bf16 1024 x 1024 7.3 us
// there, 11.4 here; 8 rows by 4096 x 1024 6.5 and 6.0, the pair 7.7 and 6.1; 8 by e4m3 2 x 1024
// x 4096 7.8 and 9.5.
bool stream_better(const ts_linear_args *a) {
    if (block_form(a->w_dtype) || (a->stages & TS_BEFORE_RMS_NORM) || a->k % 128) return true;
    // Up to twice that, up to 16 bf16 rows by pairs of bf16 weights that are split here: from HBM,
    // where a model's weights are, 8 rows by 2 x 1024 x 4096 take 8.8 us there and 10.1 here (from
    // the caches 7.9 both), by 2 x 512 x 8192 10.0 and 11.4 (9.0 and 8.4). Single weights are
    // faster here from the caches by more than they lose from HBM (2048 x 4096 6.4 against 7.6, 9.4
    // against 8.6), f32 rows, e4m3 and more rows either way.
    if (!small(a))
        return a->m > 16 || a->x_dtype == TS_F32 || a->w_dtype == TS_E4M3 || !pair_of(a) || plain_bytes(a) > 2 * kSmall ||
               plan(a).splits == 1;
    const float mt = (float)((a->m + 15) / 16), parts = a->x_dtype == TS_F32 ? 2.0f : 1.0f;
    const float values = (float)a->n * a->k * (pair_of(a) ? 2 : 1) / 1048576.0f;
    const float lanes = 4.7f + 0.54f * mt + 0.8f * mt * (parts - 1.0f) + (0.2f + 0.08f * mt * parts) * values +
                        (pair_of(a) ? 1.23f : 0.0f) + (a->w_dtype == TS_E4M3 ? 0.0f : 0.52f);
    return plan(a).cost < 0.97f * lanes;
}

size_t stream_workspace(const ts_linear_args *a) {
    const Plan pl = plan(a);
    return pl.splits > 1 ? pl.splits * split_bytes(a) : 0;
}

int stream_launch(const ts_linear_args *a, void *stream) {
    StreamParams p;
    p.x = a->x; p.w = (const uint8_t *)a->w; p.w_scale = (const uint16_t *)a->w_scale; p.gain = a->gain;
    p.a0 = a->a0; p.out = a->out; p.eps = a->eps; p.pair_sum = a->w_dtype == TS_F32_PARTS;
    p.m = a->m; p.n = a->n; p.k = a->k; p.stages = a->stages; p.out_bf16 = a->out_dtype == TS_BF16;
    int rc = linear_after(a, "lanes", &p.after);
    if (rc) return rc;
    // A workspace of fewer splits than the query names (sized for other row counts) gives the
    // best plan of those, none the best unsplit one.
    const size_t holds = a->workspace && aligned(a->workspace, 16) ? a->workspace_bytes / split_bytes(a) : 0;
    const Plan pl = plan(a, (uint32_t)std::max<size_t>(1, std::min<size_t>(holds, kMostSplits)));
    const bool split = pl.splits > 1;
    p.splits = pl.splits;
    p.part = split ? (float *)a->workspace : nullptr;
    p.sumsq = split ? p.part + (size_t)pl.splits * a->m * a->n * (pair_of(a) ? 2 : 1) : nullptr;
    hipError_t e = pl.c.ready();
    if (e != hipSuccess) return hip_status(e, "lanes: LDS attribute");
    void *args[] = {(void *)&p};
    e = hipLaunchKernel(pl.c.kernel, dim3((a->n + pl.c.cols - 1) / pl.c.cols, p.splits), dim3(pl.c.threads), args, pl.c.lds,
                        (hipStream_t)stream);
    if (e != hipSuccess) return hip_status(e, "lanes: launch");
    if (!split) return TS_OK;
    SplitSum f = {};
    f.part = p.part; f.splits = p.splits; f.out = a->out; f.a0 = a->a0;
    f.head = a->w_dtype == TS_NVFP4 ? (const float *)a->w : nullptr;
    f.w_scale = a->w_dtype == TS_E4M3 ? p.w_scale : nullptr;
    if (a->stages & TS_BEFORE_RMS_NORM) f.sumsq = p.sumsq;
    f.eps = a->eps; f.pair_sum = p.pair_sum;
    f.m = a->m; f.n = a->n; f.k = a->k; f.stages = a->stages; f.out_bf16 = p.out_bf16; f.after = p.after;
    return split_finish(f, stream);
}

}  // namespace ts
