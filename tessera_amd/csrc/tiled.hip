// "tiled": out[m, n] = after(sum_k x[m, k] w[n, k]) for many rows.
//
// Replaces the reference's matrix-unit matmul rule (engine/rules/linear/src/
// tiled.rs:281-345 tiled, :186-278 tiled_parts, :441-453, :611-672 propose),
// which on gfx950 is refused today (no tile row for gfx9_5). Same product and
// fused stages (engine/plan/lower/src/kernels/map.rs:155-185).
//
// gfx950 design (depths that are a multiple of 64 take the pipelined kernel further down,
// which shares the tile, swizzle and epilogue described here):
//  * 128x128 output tile per 256-thread group (4 waves in 2x2, each 64x64 =
//    4x4 v_mfma_f32_16x16x32_bf16 tiles), k in 64-deep steps; 64x64 tiles (waves of
//    32x32) when 128x128 would give fewer than 2 groups per CU, since each group is a
//    latency chain (load, LDS, barrier, store) rather than MFMA-bound.
//  * The MFMA computes the transposed tile (weights as the first operand), so a lane
//    holds 4 consecutive output columns of one row: one 8-byte (bf16) or 16-byte (f32)
//    store per 4 outputs instead of four 2- or 4-byte ones.
//  * Both operands are k-contiguous ([m,k] and [n,k]), which is the matrix
//    unit's native operand order: a lane's 8 k values are one 16-byte LDS read.
//  * LDS holds two stages (A and B, 16 KiB each per stage, plus a second A
//    stage for the low part of f32 rows); the next k-step is fetched from HBM
//    into registers while the current one multiplies, then stored to the other
//    stage: one barrier per k-step.
//  * LDS rows are 128 bytes (8 chunks of 16B); chunk c of row r sits at chunk
//    c ^ (r & 7), so the 16 rows one MFMA operand read touches spread over all
//    banks instead of hitting one.
//  * f32 rows are split into two exact bf16 parts (as tiled_parts does with
//    three), e4m3 weights decode to bf16 on the way into LDS with the per-row
//    scale applied to the finished sum; SiLU-gate pairs are laid out so a lane
//    holds gate and up of the same column.
#include <algorithm>

#include "after.h"

namespace {

constexpr int BM = 128, BN = 128, BK = 64;  // the default tile; BT = 64 for products with few tiles
constexpr int kThreads = 256;

struct TiledParams {
    const void *x;
    const void *w;
    const uint16_t *w_scale;
    const float *a0;
    void *out;
    uint32_t m, n, k;
    uint32_t stages;
    int out_bf16;
    // Picked products (PICK): rows sorted by matrix. perm[pos] is the row at sorted
    // position pos; matrix e owns positions [row_start[e], row_start[e + 1]) and
    // row tiles [tile_start[e], tile_start[e + 1]). Row r reads x row r / repeat;
    // matrix e's rows start at w + (e * stride + offset) * k (scales likewise).
    const uint32_t *perm, *row_start, *tile_start;
    uint32_t matrices, repeat, stride, offset;
    ts_after after;  // stage chain (count 0: none)
    int pair_sum;    // TS_F32_PARTS: the second row block is the low parts; the output sums the pair
    uint32_t splits;     // pipelined tiles: groups along k; more than 1: raw sums to part
    float *part;         // [split][gate, up or one][m][n]
    uint32_t pick_cols;  // PICK on the pipelined tiles: column tiles (0: a 2-D grid of them)
    uint32_t few_most;   // PICK: matrices of up to this many rows run as 32-row tiles
};

// Byte offset of (row, chunk) in a swizzled [rows][8 chunks of 16B] tile.
TS_DEV uint32_t swz(uint32_t row, uint32_t chunk) { return row * 128 + ((chunk ^ (row & 7)) << 4); }

template <int BT, bool XF32, bool W8, bool SILU>
struct Loader {
    static constexpr int RPT = BT / 32;  // rows per thread per operand
    static constexpr int WT = BT / 2;    // a wave's share of the tile's columns
    // Per thread per stage: A: RPT chunks (rows t/8 + 32i, chunk t%8), B: RPT chunks.
    u32x4 a_hi[RPT], a_lo[RPT], b[RPT];
    // x row of each of this thread's A rows, or -1 for a zero row.
    int64_t src[RPT];
    // The weights of this tile's matrix (the whole w outside picked products).
    const void *w;
    const uint16_t *w_scale;

    // Weight row of B-tile row `br` for this output tile. SILU: each wave's WT rows are
    // WT/2 gate rows then the WT/2 up rows of the same output columns.
    TS_DEV static uint32_t wrow(uint32_t br, uint32_t n0, uint32_t N) {
        if (!SILU) return n0 + br;
        const uint32_t half = br / WT, within = br % WT;
        return within < WT / 2 ? n0 + half * (WT / 2) + within : N + n0 + half * (WT / 2) + (within - WT / 2);
    }

    TS_DEV void fetch(const TiledParams &p, uint32_t m0, uint32_t n0, uint32_t k0) {
        const uint32_t t = threadIdx.x, chunk = t & 7;
        const uint32_t kk = k0 + chunk * 8;
        const bool kin = kk < p.k;
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            const uint32_t r = (t >> 3) + 32 * i;
            const bool ain = src[i] >= 0 && kin;
            if (XF32) {
                float v[8];
                if (ain) {
                    const float4 *src4 = (const float4 *)((const float *)p.x + (size_t)src[i] * p.k + kk);
                    float4 u0 = src4[0], u1 = src4[1];
                    v[0] = u0.x; v[1] = u0.y; v[2] = u0.z; v[3] = u0.w;
                    v[4] = u1.x; v[5] = u1.y; v[6] = u1.z; v[7] = u1.w;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] = 0.0f;
                }
                uint32_t h[4], l[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float x0 = v[2 * e], x1 = v[2 * e + 1];
                    float h0 = bf16_round(x0), h1 = bf16_round(x1);
                    h[e] = pack_bf16x2(h0, h1);
                    l[e] = pack_bf16x2(x0 - h0, x1 - h1);
                }
                a_hi[i] = u32x4{h[0], h[1], h[2], h[3]};
                a_lo[i] = u32x4{l[0], l[1], l[2], l[3]};
            } else {
                a_hi[i] = ain ? *(const u32x4 *)((const uint16_t *)p.x + (size_t)src[i] * p.k + kk) : u32x4{0, 0, 0, 0};
            }
            const uint32_t nr = wrow(r, n0, p.n);
            const uint32_t nrows = SILU ? 2 * p.n : p.n;
            const bool nin = (SILU ? (n0 + (r / WT) * (WT / 2) + (r % (WT / 2))) < p.n : nr < nrows) && kin;
            if (W8) {
                if (nin) {
                    const u32x2 c = *(const u32x2 *)((const uint8_t *)w + (size_t)nr * p.k + kk);
                    u32x2 lo = e4m3x4_to_bf16x4(c.x), hi = e4m3x4_to_bf16x4(c.y);
                    b[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
                } else {
                    b[i] = u32x4{0, 0, 0, 0};
                }
            } else {
                b[i] = nin ? *(const u32x4 *)((const uint16_t *)w + (size_t)nr * p.k + kk) : u32x4{0, 0, 0, 0};
            }
        }
    }

    TS_DEV void store(char *sa, char *sa_lo, char *sb) {
        const uint32_t t = threadIdx.x, chunk = t & 7;
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            const uint32_t r = (t >> 3) + 32 * i;
            *(u32x4 *)(sa + swz(r, chunk)) = a_hi[i];
            if (XF32) *(u32x4 *)(sa_lo + swz(r, chunk)) = a_lo[i];
            *(u32x4 *)(sb + swz(r, chunk)) = b[i];
        }
    }
};

template <int BT, bool XF32, bool W8, bool SILU, bool PICK, bool CHAIN>
__global__ __launch_bounds__(kThreads) void tiled_kernel(TiledParams p) {
    constexpr int TILE = BT * BK * 2;         // bytes of one operand stage
    constexpr int WT = BT / 2, FT = WT / 16;  // wave tile, 16x16 fragments per wave side
    constexpr int RPT = BT / 32;
    __shared__ __attribute__((aligned(16))) char lds[2][XF32 ? 3 : 2][TILE];
    __shared__ uint32_t rows_out[PICK ? BT : 1];  // output row of each tile row (PICK)

    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t wm = wave >> 1, wn = wave & 1;
    const uint32_t col = lane & 15, grp = lane >> 4;
    const uint32_t n0 = blockIdx.x * (SILU ? BT / 2 : BT);  // SILU: BT / 2 output columns per tile

    Loader<BT, XF32, W8, SILU> ld;
    uint32_t m0 = blockIdx.y * BT, mend = p.m;  // tile rows [m0, min(m0 + BT, mend))
    ld.w = p.w;
    ld.w_scale = p.w_scale;
    if (PICK) {
        // Row tile blockIdx.y belongs to the matrix e with tile_start[e] <= y < tile_start[e + 1].
        const uint32_t y = blockIdx.y;
        if (y >= p.tile_start[p.matrices]) return;
        uint32_t lo = 0, hi = p.matrices;  // invariant: tile_start[lo] <= y < tile_start[hi]
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (p.tile_start[mid] <= y) lo = mid;
            else hi = mid;
        }
        const uint32_t e = lo;
        m0 = p.row_start[e] + (y - p.tile_start[e]) * BT;
        mend = p.row_start[e + 1];
        const size_t first_row = (size_t)e * p.stride + p.offset;
        ld.w = (const char *)p.w + first_row * p.k * (W8 ? 1 : 2);
        if (W8) ld.w_scale = p.w_scale + first_row;
        for (uint32_t r = threadIdx.x; r < BT; r += kThreads)
            rows_out[r] = m0 + r < mend ? p.perm[m0 + r] : 0xffffffffu;
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        const uint32_t r = (threadIdx.x >> 3) + 32 * i;
        if (PICK) ld.src[i] = rows_out[r] != 0xffffffffu ? (int64_t)(rows_out[r] / p.repeat) : -1;
        else ld.src[i] = m0 + r < p.m ? (int64_t)(m0 + r) : -1;
    }

    f32x4 acc[FT][FT];
#pragma unroll
    for (int i = 0; i < FT; i++)
#pragma unroll
        for (int j = 0; j < FT; j++) acc[i][j] = f32x4{0, 0, 0, 0};

    const uint32_t steps = (p.k + BK - 1) / BK;
    ld.fetch(p, m0, n0, 0);
    ld.store(lds[0][0], lds[0][XF32 ? 2 : 0], lds[0][1]);
    __syncthreads();

    for (uint32_t s = 0; s < steps; s++) {
        const int cur = s & 1;
        if (s + 1 < steps) ld.fetch(p, m0, n0, (s + 1) * BK);
        const char *sa = lds[cur][0], *sb = lds[cur][1], *sl = lds[cur][XF32 ? 2 : 0];
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            const uint32_t chunk = ks * 4 + grp;
            bf16x8 af[FT], al[FT], bfr[FT];
#pragma unroll
            for (int i = 0; i < FT; i++) {
                const uint32_t ra = wm * WT + i * 16 + col;
                af[i] = as_bf16x8(*(const u32x4 *)(sa + swz(ra, chunk)));
                if (XF32) al[i] = as_bf16x8(*(const u32x4 *)(sl + swz(ra, chunk)));
                const uint32_t rb = wn * WT + i * 16 + col;
                bfr[i] = as_bf16x8(*(const u32x4 *)(sb + swz(rb, chunk)));
            }
#pragma unroll
            for (int i = 0; i < FT; i++)
#pragma unroll
                for (int j = 0; j < FT; j++) {
                    acc[i][j] = mfma16(bfr[j], af[i], acc[i][j]);
                    if (XF32) acc[i][j] = mfma16(bfr[j], al[i], acc[i][j]);
                }
        }
        if (s + 1 < steps) {
            const int nxt = cur ^ 1;
            ld.store(lds[nxt][0], lds[nxt][XF32 ? 2 : 0], lds[nxt][1]);
        }
        __syncthreads();
    }

    // Epilogue. acc[i][j] is the transposed 16x16 tile: lane (col, grp) holds row
    // m = wm WT + 16 i + col and columns n = wn WT + 16 j + 4 grp + 0..3 (SILU: gate in
    // j < FT/2, up in j + FT/2, columns wn WT/2 + 16 j + 4 grp + 0..3).
    const uint32_t N = p.n;
    const uint16_t *scale = ld.w_scale;
    const bool vec = (N & 3) == 0;
    constexpr int JO = SILU ? FT / 2 : FT;
    float val[FT][JO][4];
#pragma unroll
    for (int i = 0; i < FT; i++)
#pragma unroll
        for (int j = 0; j < JO; j++) {
            const uint32_t n = n0 + (SILU ? wn * (WT / 2) : wn * WT) + j * 16 + 4 * grp;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float g = acc[i][j][r];
                if (SILU) {
                    float u = acc[i][j + FT / 2][r];
                    if (W8) {
                        g *= bf16_float(scale[min(n + r, N - 1)]);
                        u *= bf16_float(scale[N + min(n + r, N - 1)]);
                    }
                    val[i][j][r] = p.pair_sum ? g + u : g / (1.0f + expf(-g)) * u;
                } else {
                    if (W8) g *= bf16_float(scale[min(n + r, N - 1)]);
                    val[i][j][r] = g;
                }
            }
        }
    if (CHAIN) {  // the chain's variant: its values and sums need more registers
        // Value e = (i JO + j) 4 + r: row tile i, column tile j, column 4 grp + r.
        auto row_of = [&](int e) {
            const uint32_t tr = wm * WT + (e / (4 * JO)) * 16 + col;
            return m0 + tr < mend ? (PICK ? rows_out[tr] : m0 + tr) : ~0u;
        };
        auto col_of = [&](int e) {
            return n0 + (SILU ? wn * (WT / 2) : wn * WT) + (e / 4 % JO) * 16 + 4 * grp + e % 4;
        };
        ts::after_values<FT * JO * 4, false>(
            p.after, *(float(*)[FT * JO * 4])val, [&](int e) { return (size_t)row_of(e) * N + col_of(e); },
            [&](int e) { return row_of(e) != ~0u && col_of(e) < N; });
    }
#pragma unroll
    for (int i = 0; i < FT; i++) {
        const uint32_t tr = wm * WT + i * 16 + col;
        if (m0 + tr >= mend) continue;
        const uint32_t m = PICK ? rows_out[tr] : m0 + tr;
#pragma unroll
        for (int j = 0; j < JO; j++) {
            const uint32_t n = n0 + (SILU ? wn * (WT / 2) : wn * WT) + j * 16 + 4 * grp;
            if (n >= N) continue;
            float *v = val[i][j];
            const size_t at = (size_t)m * N + n;
            if (vec && n + 3 < N) {
                if (p.stages & TS_AFTER_ADD) {
                    const float4 a = *(const float4 *)(p.a0 + at);
                    v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
                }
                if (p.out_bf16) *(u32x2 *)((uint16_t *)p.out + at) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                else *(float4 *)((float *)p.out + at) = float4{v[0], v[1], v[2], v[3]};
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (n + r >= N) break;
                    float u = v[r];
                    if (p.stages & TS_AFTER_ADD) u += p.a0[at + r];
                    if (p.out_bf16) ((uint16_t *)p.out)[at + r] = bf16_bits(u);
                    else ((float *)p.out)[at + r] = u;
                }
            }
        }
    }
}


// ---------------------------------------------------------------------------
// The pipelined form (k a multiple of 64): TM x TN tiles, 4 waves, and NS LDS stages KD
// deep filled straight from memory by 16-byte buffer loads to LDS (no staging registers,
// no LDS stores), NS - 1 of them in flight ahead of the MFMAs, groups in an XCD-aware
// order, and each configuration sized so two groups (one form: three) share a CU: one group's loads,
// barriers and epilogue overlap the other's matrix work. bf16 results leave through LDS
// as whole rows.
//  * bf16 rows and weights: waves in 2 x 2, each (TM/2) x (TN/2).
//  * f32 rows (XF32) lie in LDS as f32, as many bytes as the two bf16 parts would take;
//    a lane splits the 8 values of a fragment into hi = bf16(x), lo = bf16(x - hi) right
//    after reading them (24 vector instructions a fragment). The waves are stacked along
//    the rows, so each fragment is split by one wave only, at the same LDS bytes read per
//    MFMA as 2 x 2 (a row fragment is two reads here, a weight fragment one).
//  * e4m3 weights (W8) lie in LDS as codes, half the bytes; a lane reads 16 codes of its
//    weight row and decodes them to the two fragments of a 64-deep step (8 conversions).
//    The matrix unit sums k in any order, so the rows' fragments are read at the same k.
//  * The stages come by buffer loads (buffer_to_lds16): with global loads to LDS in flight
//    the compiler waited for all LDS reads of a step before its first MFMA. With them, and
//    the steps that refill a stage in a loop without tests: e4m3 4096 x 14336 159 -> 117 us.
// Register-staged against this form: 1000 f32 rows by bf16 weights 4096 x 1024 64.2 -> 24.7
// us, 1024 x 3072 92.6 -> 24.9 us; 1000 bf16 rows by e4m3 gate/up 2 x 14336 x 4096 560 -> 223
// us (1052 TFLOP/s), down 4096 x 14336 249 -> 117 us. What the register-staged form spent
// was the load latency of every k step, with no stage in flight behind its barrier. It
// still serves depths that are no multiple of 64 and the stage chains of picked products.
// ---------------------------------------------------------------------------
// A stage's operand rows in LDS: RB bytes a row in 16-byte chunks.
template <int RB>
struct Rows {
    static constexpr int CPR = RB / 16;    // chunks per row
    static constexpr int RPI = 1024 / RB;  // rows one load instruction fills
    static_assert(RB == 64 || RB == 128 || RB == 256, "row bytes");

    // Byte offset of chunk c of row r. 256- and 128-byte rows: chunk c ^ (r & (CPR - 1)).
    // 64-byte rows: rows pair up in 128-byte lines L = r / 2, and 16-byte unit u = 4 (r &
    // 1) + c of a line sits at u ^ (L & 7). Either way the 16 rows one fragment read
    // touches (one chunk each) spread over all banks (measured: no conflicts; a per-row
    // XOR of 64-byte rows conflicts).
    TS_DEV static uint32_t at(uint32_t r, uint32_t c) {
        if (RB >= 128) return r * RB + ((c ^ (r & (CPR - 1))) << 4);
        const uint32_t L = r >> 1, u = (r & 1) * 4 + c;
        return L * 128 + ((u ^ (L & 7)) << 4);
    }
    // The row and chunk that lane l of load instruction b brings (the lane lands at byte
    // 16 l of the instruction's KiB, whose first row is RPI b).
    TS_DEV static void source(uint32_t b, uint32_t l, uint32_t &row, uint32_t &chunk) {
        if (RB >= 128) {
            row = RPI * b + l / CPR;
            chunk = (l % CPR) ^ (row & (CPR - 1));
        } else {
            const uint32_t line = l >> 3, u = (l & 7) ^ line;  // 8 lines per KiB: line is L & 7
            row = RPI * b + 2 * line + (u >> 2);
            chunk = u & 3;
        }
    }
};

template <int TM, int TN, int KD, int NS, bool XF32, bool W8>
struct Pipe {
    using A = Rows<KD * (XF32 ? 4 : 2)>;
    using B = Rows<KD * (W8 ? 1 : 2)>;
    static constexpr int AE = XF32 ? 4 : 8, BE = W8 ? 16 : 8;  // elements per chunk
    static constexpr int NA = TM / A::RPI / 4;  // A load instructions per wave per stage
    static constexpr int NB = TN / B::RPI / 4;  // B load instructions per wave per stage
    static constexpr int A_BYTES = TM * A::CPR * 16, STAGE = A_BYTES + TN * B::CPR * 16, LDS = NS * STAGE;
    static constexpr int GM = TM == 32 ? 1 : XF32 ? 4 : 2, GN = 4 / GM;  // waves along the rows and the columns
    static constexpr int WM = TM / GM, WN = TN / GN, FI = WM / 16, FJ = WN / 16;
    static_assert(NA >= 1 && NB >= 1 && FI >= 1 && (KD == 64 || (KD == 32 && !W8)), "pipe shape");
};

// Eight f32 values (two chunks) as the two bf16 parts hi = bf16(x), lo = bf16(x - hi).
TS_DEV void split_f32(f32x4 a, f32x4 b, bf16x8 &hi, bf16x8 &lo) {
    const float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    uint32_t h[4], l[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        h[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(ts_f32x2{v[2 * e], v[2 * e + 1]}, ts_bf16x2));
        const ts_f32x2 rest = {v[2 * e] - lo_bf16(h[e]), v[2 * e + 1] - hi_bf16(h[e])};
        l[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, ts_bf16x2));
    }
    hi = as_bf16x8(u32x4{h[0], h[1], h[2], h[3]});
    lo = as_bf16x8(u32x4{l[0], l[1], l[2], l[3]});
}

constexpr uint32_t kBand = 8;  // tile rows per band of the XCD-aware order

// Waits until at most N of this wave's loads are outstanding and its LDS reads of the
// previous k-step are back, then meets the group's other waves (the loads waited for here
// wrote LDS directly).
template <int N>
TS_DEV void pipe_wait() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// The wait for a stage with `ahead` later stages (L loads each) still allowed in flight.
template <int L, int A>
TS_DEV void pipe_wait_ahead(uint32_t ahead) {
    if constexpr (A == 0) {
        pipe_wait<0>();
    } else {
        if (ahead >= A) pipe_wait<L * A>();
        else pipe_wait_ahead<L, A - 1>(ahead);
    }
}

// What a pipelined kernel does with its sums: its epilogue, the epilogue with a stage chain (64
// x 64 tiles only: larger ones would spill), or raw sums of a split of k to memory.
enum Ends { kPlain, kChain, kSplit };

// Stages of the 32-row tiles (16 to 24 KiB each).
template <bool XF32>
constexpr int kFewStages = XF32 ? 3 : 4;

template <int TM, int TN, int KD, int NS, bool XF32, bool W8, bool SILU, bool PICK, Ends END, bool ROLL>
TS_DEV void pipe_tile(const TiledParams &p, char *lds, uint32_t n0, uint32_t m0, uint32_t mend, const char *w,
                      const uint16_t *scale, uint32_t split);

// Groups that share a CU, a wave of each a SIMD: two, three of the form whose stages leave LDS
// for them (bf16 rows by e4m3 on 64 x 64, 48 KiB: 700 rows by 4096 x 1024 11.7 -> 10.7 us, 704
// tiles in one round; up to 512 tiles the same).
template <int TM, int TN, int KD, int NS, bool XF32, bool W8, Ends END>
constexpr int kShare = 3 * Pipe<TM, TN, KD, NS, XF32, W8>::LDS <= 160 * 1024 && TM * TN == 64 * 64 && END != kChain ? 3 : 2;

// FEW (picked products): the matrices of at most p.few_most rows run as 32-row tiles. ROLL: the
// steps are unrolled (not in a FEW kernel, whose two forms share the instruction cache, nor in
// 32-row tiles, where f32 rows by e4m3 got slower: 64 rows on 64 matrices of 2 x 1024 x 2048 57 -> 60
// us).
template <int TM, int TN, int KD, int NS, bool XF32, bool W8, bool SILU, bool PICK, Ends END, bool FEW>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(
    kShare<TM, TN, KD, NS, XF32, W8, END>, kShare<TM, TN, KD, NS, XF32, W8, END>))) void tiled_pipe_kernel(TiledParams p) {
    extern __shared__ __attribute__((aligned(16))) char lds[];  // the only LDS: groups share a CU
    constexpr uint32_t OC = SILU ? TN / 2 : TN;  // output columns per tile
    uint32_t tx = blockIdx.x, ty = blockIdx.y, split = 0;
    if (!PICK) {
        // XCD-aware order (one-dimensional grid): group b runs on XCD b % 8, and XCD x
        // takes the x-th eighth of the tiles, walked in bands of kBand tile rows column
        // by column, so the groups an XCD runs at once share rows and weight columns
        // in its L2.
        // A split of k is a grid of tiles of its own, behind the one before it.
        const uint32_t gx = p.stride, gy = p.offset, tiles = gx * gy, all = END == kSplit ? tiles * p.splits : tiles,
                       per = (all + 7) / 8;
        uint32_t t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
        if (t >= all) return;
        if (END == kSplit) {
            split = t / tiles;
            t -= split * tiles;
        }
        const uint32_t band = t / (kBand * gx), rows = min(kBand, gy - band * kBand);
        const uint32_t within = t - band * kBand * gx;
        ty = band * kBand + within % rows;
        tx = within / rows;
    }
    uint32_t n0 = tx * OC;
    uint32_t m0 = ty * TM, mend = p.m;
    const char *w = (const char *)p.w;
    const uint16_t *scale = p.w_scale;
    if (PICK) {
        uint32_t y = blockIdx.y;
        if (p.pick_cols) {
            // XCD-aware order (one-dimensional grid, group b on XCD b % 8): XCD x takes
            // the sorted row tiles [x Y / 8, (x + 1) Y / 8) and walks them matrix by
            // matrix, each matrix's column tiles in turn over its row tiles, so the
            // gathered rows and the weight tile both stay in that XCD's L2.
            const uint32_t Y = p.tile_start[p.matrices], gx = p.pick_cols;
            const uint32_t xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
            const uint32_t y0 = (uint32_t)((uint64_t)xcd * Y / 8), y1 = (uint32_t)((uint64_t)(xcd + 1) * Y / 8);
            if (j >= gx * (y1 - y0)) return;
            uint32_t lo = 0, hi = p.matrices;  // the matrix holding row tile y0
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) / 2;
                if (p.tile_start[mid] <= y0) lo = mid;
                else hi = mid;
            }
            uint32_t e = lo, ys = y0, rem = j;
            for (;;) {  // ends: j < gx (y1 - y0), and every row tile in range belongs to a matrix
                const uint32_t ye = min(p.tile_start[e + 1], y1), ne = ye - ys;
                if (rem < gx * ne) {
                    tx = rem / ne;
                    n0 = tx * OC;
                    y = ys + rem % ne;
                    break;
                }
                rem -= gx * ne;
                ys = ye;
                e++;
            }
        }
        if (y >= p.tile_start[p.matrices]) return;
        uint32_t lo = 0, hi = p.matrices;  // invariant: tile_start[lo] <= y < tile_start[hi]
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (p.tile_start[mid] <= y) lo = mid;
            else hi = mid;
        }
        const uint32_t e = lo;
        const size_t first_row = (size_t)e * p.stride + p.offset;
        w += first_row * p.k * (W8 ? 1 : 2);
        if (W8) scale += first_row;
        mend = p.row_start[e + 1];
        if constexpr (FEW)
            if (mend - p.row_start[e] <= p.few_most)
                return pipe_tile<32, TN, 64, kFewStages<XF32>, XF32, W8, SILU, PICK, END, false>(
                    p, lds, n0, p.row_start[e] + (y - p.tile_start[e]) * 32, mend, w, scale, split);
        m0 = p.row_start[e] + (y - p.tile_start[e]) * TM;
    }
    pipe_tile<TM, TN, KD, NS, XF32, W8, SILU, PICK, END, !FEW && TM != 32>(p, lds, n0, m0, mend, w, scale, split);
}

// The tile of rows [m0, min(m0 + TM, mend)) and of the columns from n0 on.
template <int TM, int TN, int KD, int NS, bool XF32, bool W8, bool SILU, bool PICK, Ends END, bool ROLL>
TS_DEV void pipe_tile(const TiledParams &p, char *lds, uint32_t n0, uint32_t m0, uint32_t mend, const char *w,
                      const uint16_t *scale, uint32_t split) {
    using P = Pipe<TM, TN, KD, NS, XF32, W8>;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wm = wave / P::GN, wn = wave % P::GN;
    const uint32_t col = lane & 15, grp = lane >> 4;
    constexpr uint32_t OC = SILU ? TN / 2 : TN;  // output columns per tile
    // PICK: the output row of tile row tr (~0u past the matrix's rows), read where needed
    // (no LDS copy, so two groups' stages fill a CU's LDS).
    auto row_out = [&](uint32_t tr) { return m0 + tr < mend ? p.perm[m0 + tr] : 0xffffffffu; };
    // Byte offsets (at k = 0) of the chunk each of this lane's loads reads: instruction NA
    // wave + i (A) or NB wave + i (B) of the stage, from the tile's first row (A of picked
    // products: from the first row of x; B of the up rows: from the tile's first up row).
    // Rows past the end read a row that exists (never stored).
    constexpr uint32_t XB = XF32 ? 4 : 2, WB = W8 ? 1 : 2;
    uint32_t aoff[P::NA], boff[P::NB];
    bool up[P::NB];  // wave-uniform: an instruction's rows are all gate or all up rows
#pragma unroll
    for (int i = 0; i < P::NA; i++) {
        uint32_t r, c, xr;
        P::A::source(wave * P::NA + i, lane, r, c);
        if (PICK) {
            const uint32_t o = row_out(r);
            xr = (o != 0xffffffffu ? o : p.perm[m0]) / p.repeat;
        } else {
            xr = min(r, p.m - 1 - m0);
        }
        aoff[i] = (xr * p.k + c * P::AE) * XB;
    }
#pragma unroll
    for (int i = 0; i < P::NB; i++) {
        uint32_t r, c, nr;
        P::B::source(wave * P::NB + i, lane, r, c);
        up[i] = false;
        if (SILU) {
            // Each wave's WN weight rows: WN/2 gate rows, then the up rows of the same columns.
            static_assert(!SILU || P::WN / 2 % P::B::RPI == 0, "a load's rows are of one kind");
            const uint32_t half = r / P::WN, within = r % P::WN;
            nr = min(half * (P::WN / 2) + within % (P::WN / 2), p.n - 1 - n0);
            up[i] = (wave * P::NB + i) * P::B::RPI % P::WN >= P::WN / 2;
        } else {
            nr = min(r, p.n - 1 - n0);
        }
        boff[i] = (nr * p.k + c * P::BE) * WB;
    }

    const char *xbase = (const char *)p.x + (PICK ? 0 : (size_t)m0 * p.k * XB);
    const char *wbase = w + (size_t)n0 * p.k * WB;
    const __amdgpu_buffer_rsrc_t xbuf = raw_buffer(xbase), wbuf = raw_buffer(wbase),
                                 ubuf = raw_buffer(wbase + (SILU ? (size_t)p.n * p.k * WB : 0));
    auto fetch = [&](uint32_t slot, uint32_t k0) {
        char *stage = lds + slot * P::STAGE;
#pragma unroll
        for (int i = 0; i < P::NA; i++)
            buffer_to_lds16(xbuf, stage + (wave * P::NA + i) * 1024, aoff[i], k0 * XB);
#pragma unroll
        for (int i = 0; i < P::NB; i++)
            buffer_to_lds16(up[i] ? ubuf : wbuf, stage + P::A_BYTES + (wave * P::NB + i) * 1024, boff[i], k0 * WB);
    };

    f32x4 acc[P::FI][P::FJ];
#pragma unroll
    for (int i = 0; i < P::FI; i++)
#pragma unroll
        for (int j = 0; j < P::FJ; j++) acc[i][j] = f32x4{0, 0, 0, 0};

    uint32_t s0 = 0, steps = p.k / KD;
    if (END == kSplit) {
        const uint32_t each = steps / p.splits, more = steps - each * p.splits;  // the first `more` take one more
        s0 = split * each + min(split, more);
        steps = each + (split < more ? 1 : 0);
    }
    // 16-row fragments of this wave that hold a row of the tile (wave-uniform).
    const uint32_t wrow0 = m0 + wm * P::WM;
    const uint32_t live_frags = mend > wrow0 ? min((mend - wrow0 + 15) / 16, (uint32_t)P::FI) : 0u;
#pragma unroll
    for (int s = 0; s < NS - 1; s++)
        if ((uint32_t)s < steps) fetch(s, (s0 + s) * KD);
    // The matrix work of the stage in slot `at`.
    auto multiply = [&](uint32_t at) {
        const char *sa = lds + at * P::STAGE, *sb = sa + P::A_BYTES;
        // PICK mode: row fragments wholly past the matrix's last row (its partial last
        // tile) skip their MFMAs; their loads and the barriers stay, so every wave keeps
        // the same pipeline.
        auto step = [&](const bool all) {
            u32x4 codes[W8 ? P::FJ : 1];  // e4m3: the 16 codes of a 64-deep step, k 16 grp .. + 15
            if (W8)
#pragma unroll
                for (int j = 0; j < P::FJ; j++)
                    codes[j] = *(const u32x4 *)(sb + P::B::at(wn * P::WN + j * 16 + col, grp));
#pragma unroll
            for (int ks = 0; ks < KD / 32; ks++) {
                // The 8 k values of this lane: eighth `chunk` of the step (e4m3: the half of its codes).
                const uint32_t chunk = W8 ? 2 * grp + ks : ks * 4 + grp;
                bf16x8 af[P::FI], al[XF32 ? P::FI : 1], bfr[P::FJ];
#pragma unroll
                for (int i = 0; i < P::FI; i++)
                    if (all || (uint32_t)i < live_frags) {
                        const uint32_t r = wm * P::WM + i * 16 + col;
                        if (XF32)
                            split_f32(*(const f32x4 *)(sa + P::A::at(r, 2 * chunk)),
                                      *(const f32x4 *)(sa + P::A::at(r, 2 * chunk + 1)), af[i], al[XF32 ? i : 0]);
                        else
                            af[i] = as_bf16x8(*(const u32x4 *)(sa + P::A::at(r, chunk)));
                    }
#pragma unroll
                for (int j = 0; j < P::FJ; j++) {
                    if (W8) {
                        const u32x4 q = codes[W8 ? j : 0];
                        const u32x2 lo = e4m3x4_to_bf16x4(ks ? q.z : q.x), hi = e4m3x4_to_bf16x4(ks ? q.w : q.y);
                        bfr[j] = as_bf16x8(u32x4{lo.x, lo.y, hi.x, hi.y});
                    } else {
                        bfr[j] = as_bf16x8(*(const u32x4 *)(sb + P::B::at(wn * P::WN + j * 16 + col, chunk)));
                    }
                }
#pragma unroll
                for (int i = 0; i < P::FI; i++)
                    if (all || (uint32_t)i < live_frags) {
#pragma unroll
                        for (int j = 0; j < P::FJ; j++) acc[i][j] = mfma16(bfr[j], af[i], acc[i][j]);
                        if (XF32)
#pragma unroll
                            for (int j = 0; j < P::FJ; j++) acc[i][j] = mfma16(bfr[j], al[XF32 ? i : 0], acc[i][j]);
                    }
            }
        };
        if (!PICK || live_frags >= (uint32_t)P::FI) step(true);
        else step(false);
    };
    // Stage s has landed once no more than the later stages' loads are outstanding; the
    // barrier also ends every wave's reads of the stage refilled next. The steps that refill
    // run without a test of what is left, a ring's worth of them unrolled: a step's slot is a
    // constant. With stages to spare (NS > 2) the refill is issued behind the matrix work,
    // where its writes to LDS do not meet the step's reads; with two stages it has only this
    // step to land in. 2048 bf16 rows by 1024 x 3072 22.0 -> 20.4 us (64 x 64 tiles; unrolled
    // alone 21.2, the form before buffer loads 21.5), by 2 x 3072 x 1024 32.9 -> 32.1 (128 x 192); two stages refilled late: 1000
    // by 4096 x 4096 41 -> 55. Not where a step's own registers are many, which unrolled got
    // slower: f32 rows by e4m3 on 128 x 128 (1000 by 4096 x 14336 231 -> 246), f32 rows
    // by bf16 picked (4096 rows by 32 matrices of 2 x 1024 x 2048 133 -> 135).
    constexpr bool UNROLL = ROLL && (!XF32 || (PICK ? W8 : NS > 2)), LATE = UNROLL && NS > 2;
    auto refilling = [&](uint32_t s, uint32_t at, uint32_t fill) {
        pipe_wait<(P::NA + P::NB) * (NS - 2)>();
        if (!LATE) fetch(fill, (s0 + s + NS - 1) * KD);
        multiply(at);
        if (LATE) fetch(fill, (s0 + s + NS - 1) * KD);
    };
    uint32_t s = 0;
    if (UNROLL)
        for (; s + 2 * NS - 2 < steps; s += NS)
#pragma unroll
            for (int u = 0; u < NS; u++) refilling(s + u, u, (u + NS - 1) % NS);
    uint32_t at = 0, fill = NS - 1;  // the slots of this step and of the stage loaded in it
    for (; s + NS - 1 < steps; s++) {
        refilling(s, at, fill);
        at = at == NS - 1 ? 0 : at + 1;
        fill = fill == NS - 1 ? 0 : fill + 1;
    }
    for (; s < steps; s++) {
        pipe_wait_ahead<P::NA + P::NB, NS - 2>(steps - 1 - s);
        multiply(at);
        at = at == NS - 1 ? 0 : at + 1;
    }

    // Epilogue. acc[i][j] is the transposed 16x16 tile: lane (col, grp) holds tile row
    // wm WM + 16 i + col and columns wn WN + 16 j + 4 grp .. + 3 (SILU: gate in j < FJ/2,
    // up in j + FJ/2, output columns wn WN/2 + 16 j + 4 grp .. + 3).
    const uint32_t N = p.n;
    constexpr int JO = SILU ? P::FJ / 2 : P::FJ;
    constexpr uint32_t WO = SILU ? P::WN / 2 : P::WN;
    if (END == kSplit) {  // raw sums; split_finish adds the splits and runs the epilogue
        const size_t mn = (size_t)p.m * N;
        float *dst = p.part + (size_t)split * (SILU ? 2 : 1) * mn;
#pragma unroll
        for (int i = 0; i < P::FI; i++) {
            const uint32_t m = m0 + wm * P::WM + i * 16 + col;
            if (m >= p.m) continue;
#pragma unroll
            for (int j = 0; j < P::FJ; j++) {
                const uint32_t n = n0 + wn * WO + j % JO * 16 + 4 * grp;
                float *o = dst + (j < JO ? 0 : mn) + (size_t)m * N + n;
                if ((N & 3) == 0 && n < N) __builtin_nontemporal_store(acc[i][j], (f32x4 *)o);
                else
                    for (uint32_t r = 0; r < 4 && n + r < N; r++) o[r] = acc[i][j][r];
            }
        }
        return;
    }
    // e4m3: each weight row's scale on its finished sums.
    if (W8) {
#pragma unroll
        for (int j = 0; j < JO; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t n = min(n0 + wn * WO + j * 16 + 4 * grp + r, N - 1);
                const float sg = bf16_float(scale[n]), su = SILU ? bf16_float(scale[N + n]) : 0.0f;
#pragma unroll
                for (int i = 0; i < P::FI; i++) {
                    acc[i][j][r] *= sg;
                    if (SILU) acc[i][j + JO][r] *= su;
                }
            }
    }
    auto value = [&](int i, int j, int r) {
        const float g = acc[i][j][r];
        const float u = SILU ? acc[i][j + (SILU ? P::FJ / 2 : 0)][r] : 0.0f;
        return SILU ? (p.pair_sum ? g + u : g / (1.0f + expf(-g)) * u) : g;
    };
    if (!PICK && p.out_bf16 && !(p.stages & TS_AFTER_ADD) && !p.after.count) {
        // bf16 rows through LDS: the tile as TM rows of OC bf16 (16-byte chunks
        // XOR-swizzled by row), then whole 16-byte chunks of rows to memory.
        constexpr uint32_t CH = OC / 8;  // chunks per output row
        static_assert(TM * OC * 2 <= P::LDS, "pipe epilogue fits the stages");
        // Chunk c of row r: XOR by the row when CH is a power of two, else rotated by
        // the row (an XOR could leave the row).
        auto slot = [](uint32_t r, uint32_t c) {
            return (CH & (CH - 1)) == 0 ? c ^ (r % CH) : (c + r) % CH;
        };
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int i = 0; i < P::FI; i++) {
            const uint32_t r = wm * P::WM + i * 16 + col;
#pragma unroll
            for (int j = 0; j < JO; j++) {
                const uint32_t c = wn * WO + j * 16 + 4 * grp;
                *(u32x2 *)(lds + r * OC * 2 + (slot(r, c >> 3) << 4) + (c & 7) * 2) =
                    u32x2{pack_bf16x2(value(i, j, 0), value(i, j, 1)), pack_bf16x2(value(i, j, 2), value(i, j, 3))};
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const bool rows16 = (N & 7) == 0;
#pragma unroll 4
        for (uint32_t f = threadIdx.x; f < TM * CH; f += kThreads) {
            const uint32_t r = f / CH, c = f % CH;
            const uint32_t m = m0 + r, n = n0 + c * 8;
            if (m >= p.m || n >= N) continue;
            const u32x4 v = *(const u32x4 *)(lds + r * OC * 2 + (slot(r, c) << 4));
            uint16_t *o = (uint16_t *)p.out + (size_t)m * N + n;
            if (rows16 && n + 8 <= N) {
                *(u32x4 *)o = v;
            } else {
                for (uint32_t e = 0; e < 8 && n + e < N; e++) o[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
            }
        }
        return;
    }
    const bool vec = (N & 3) == 0;
    float val[P::FI][JO][4];
#pragma unroll
    for (int i = 0; i < P::FI; i++)
#pragma unroll
        for (int j = 0; j < JO; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) val[i][j][r] = value(i, j, r);
    if (END == kChain) {  // the chain's variant: its values and sums need more registers
        // Value e = (i JO + j) 4 + r: row fragment i, column fragment j, column 4 grp + r.
        auto row_of = [&](int e) {
            const uint32_t tr = wm * P::WM + (e / (4 * JO)) * 16 + col;
            return m0 + tr < mend ? (PICK ? row_out(tr) : m0 + tr) : ~0u;
        };
        auto col_of = [&](int e) { return n0 + wn * WO + (e / 4 % JO) * 16 + 4 * grp + e % 4; };
        ts::after_values<P::FI * JO * 4, false>(
            p.after, *(float(*)[P::FI * JO * 4])val, [&](int e) { return (size_t)row_of(e) * N + col_of(e); },
            [&](int e) { return row_of(e) != ~0u && col_of(e) < N; });
    }
#pragma unroll
    for (int i = 0; i < P::FI; i++) {
        const uint32_t tr = wm * P::WM + i * 16 + col;
        if (m0 + tr >= mend) continue;
        const uint32_t m = PICK ? row_out(tr) : m0 + tr;
#pragma unroll
        for (int j = 0; j < JO; j++) {
            const uint32_t n = n0 + wn * WO + j * 16 + 4 * grp;
            if (n >= N) continue;
            float *v = val[i][j];
            const size_t at = (size_t)m * N + n;
            if (vec && n + 3 < N) {
                if (p.stages & TS_AFTER_ADD) {
                    const float4 a = *(const float4 *)(p.a0 + at);
                    v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
                }
                if (p.out_bf16) *(u32x2 *)((uint16_t *)p.out + at) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                else *(float4 *)((float *)p.out + at) = float4{v[0], v[1], v[2], v[3]};
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (n + r >= N) break;
                    float u = v[r];
                    if (p.stages & TS_AFTER_ADD) u += p.a0[at + r];
                    if (p.out_bf16) ((uint16_t *)p.out)[at + r] = bf16_bits(u);
                    else ((float *)p.out)[at + r] = u;
                }
            }
        }
    }
}

template <int TM, int TN, int KD, int NS, bool XF32, bool W8, bool PICK, Ends END = kPlain, bool FEW = false>
int pipe_launch(TiledParams p, bool silu, void *stream) {
    constexpr int lds = [] {
        constexpr int own = Pipe<TM, TN, KD, NS, XF32, W8>::LDS;
        if constexpr (FEW) return std::max(own, Pipe<32, TN, 64, kFewStages<XF32>, XF32, W8>::LDS);
        return own;
    }();
    const void *k = silu ? (const void *)tiled_pipe_kernel<TM, TN, KD, NS, XF32, W8, true, PICK, END, FEW>
                         : (const void *)tiled_pipe_kernel<TM, TN, KD, NS, XF32, W8, false, PICK, END, FEW>;
    // The dynamic LDS size is raised once per kernel (thread-safe static initialisation).
    static const hipError_t attr[2] = {
        hipFuncSetAttribute((const void *)tiled_pipe_kernel<TM, TN, KD, NS, XF32, W8, false, PICK, END, FEW>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds),
        hipFuncSetAttribute((const void *)tiled_pipe_kernel<TM, TN, KD, NS, XF32, W8, true, PICK, END, FEW>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds)};
    if (attr[silu]) return ts::hip_status(attr[silu], "tiled (pipelined): LDS attribute");
    const uint32_t oc = silu ? TN / 2 : TN;
    const uint32_t gx = (p.n + oc - 1) / oc;
    dim3 grid;
    if (PICK) {
        // Row tiles: at most one partial tile per matrix beyond rows / TM full ones.
        constexpr uint32_t RT = FEW ? 32 : TM;
        const uint32_t gy = (p.m + RT - 1) / RT + p.matrices;
        // XCD-aware (C5 gate/up 1214 -> 1189 us, layer 2.48-2.53 -> 2.44 ms) where the
        // one-dimensional grid fits.
        if ((uint64_t)8 * gx * ((gy + 7) / 8) < (1ull << 31)) {
            p.pick_cols = gx;
            grid = dim3(8 * gx * ((gy + 7) / 8));
        } else {
            grid = dim3(gx, gy);
        }
    } else {
        // A one-dimensional grid of 8 x ceil(tiles / 8) groups; stride and offset,
        // unused outside picked products, carry the tile grid's width and height.
        const uint32_t gy = (p.m + TM - 1) / TM;
        p.stride = gx;
        p.offset = gy;
        grid = dim3(8 * (uint32_t)(((uint64_t)gx * gy * p.splits + 7) / 8));
    }
    void *args[] = {(void *)&p};
    const hipError_t e = hipLaunchKernel(k, grid, dim3(kThreads), args, lds, (hipStream_t)stream);
    if (e != hipSuccess) return ts::hip_status(e, "tiled (pipelined): launch");
    return TS_OK;
}

// The pipelined kernels take whole 64-deep k steps and byte offsets within the rows a tile
// may read (256 of x and of w; all of x in picked products) that fit 32 bits.
bool pipe_fits(uint32_t x_rows, uint32_t k, uint32_t x_bytes) {
    return k % 64 == 0 && (uint64_t)std::max(x_rows, 256u) * k * x_bytes < (1ull << 32);
}

// 64 x 64 tiles, four stages of 16 KiB or three of 20 to 24.
template <Ends END>
int pipe_small(const TiledParams &p, bool xf, bool w8, bool silu, void *stream) {
    if (xf) return w8 ? pipe_launch<64, 64, 64, 3, true, true, false, END>(p, silu, stream)
                      : pipe_launch<64, 64, 64, 3, true, false, false, END>(p, silu, stream);
    return w8 ? pipe_launch<64, 64, 64, 4, false, true, false, END>(p, silu, stream)
              : pipe_launch<64, 64, 64, 4, false, false, false, END>(p, silu, stream);
}

// 128 x 128 tiles. FEW: 32 x 128 for the matrices of few rows.
template <bool PICK, Ends END = kPlain, bool FEW = false>
int pipe_wide(const TiledParams &p, bool xf, bool w8, bool silu, void *stream) {
    if (xf) return w8 ? pipe_launch<128, 128, 64, 2, true, true, PICK, END, FEW>(p, silu, stream)
                      : pipe_launch<128, 128, 32, 3, true, false, PICK, END, FEW>(p, silu, stream);
    return w8 ? pipe_launch<128, 128, 64, 3, false, true, PICK, END, FEW>(p, silu, stream)
              : pipe_launch<128, 128, 64, 2, false, false, PICK, END, FEW>(p, silu, stream);
}

// 32 x 128 tiles alone: the four waves side by side along the columns.
int pipe_few(const TiledParams &p, bool xf, bool w8, bool silu, void *stream) {
    if (xf) return w8 ? pipe_launch<32, 128, 64, kFewStages<true>, true, true, true>(p, silu, stream)
                      : pipe_launch<32, 128, 64, kFewStages<true>, true, false, true>(p, silu, stream);
    return w8 ? pipe_launch<32, 128, 64, kFewStages<false>, false, true, true>(p, silu, stream)
              : pipe_launch<32, 128, 64, kFewStages<false>, false, false, true>(p, silu, stream);
}

using Kern = void (*)(TiledParams);

template <int BT, bool XF32, bool W8, bool PICK>
Kern pick_silu(bool silu, bool chain) {
    if (chain) return silu ? tiled_kernel<BT, XF32, W8, true, PICK, true> : tiled_kernel<BT, XF32, W8, false, PICK, true>;
    return silu ? tiled_kernel<BT, XF32, W8, true, PICK, false> : tiled_kernel<BT, XF32, W8, false, PICK, false>;
}

template <int BT, bool PICK>
Kern pick_kernel(bool xf, bool w8, bool silu, bool chain) {
    return xf ? (w8 ? pick_silu<BT, true, true, PICK>(silu, chain) : pick_silu<BT, true, false, PICK>(silu, chain))
              : (w8 ? pick_silu<BT, false, true, PICK>(silu, chain) : pick_silu<BT, false, false, PICK>(silu, chain));
}

}  // namespace

namespace {

// The k split of a product of more than 64 rows whose tiles alone leave CUs idle: times in us,
// from what the pipelined tiles take a 64-deep step with one group a CU and with two (64 x 64
// 0.21 and 0.33, e4m3 0.2, f32 rows 0.4 and 0.62; 128 x 128 0.65 and 0.82, e4m3 0.49, f32 rows
// 0.99 and 1.7; past two in proportion) and what the second kernel takes (3.2, 0.1 a split and
// 0.37 a MB of sums). Fitted to every split of 980 products of 65 to 2048 rows by 128 to 8192 x
// 1024 to 14336 with weights in the caches and from HBM, between which the prices stand: what this
// chooses takes 0.5% more than the best split in the mean, 18% at most (128 bf16 rows by 2048 x
// 2048 from HBM). 128 f32 rows by 1024 x 3072 23.8 -> 11.6 us, 1200 by 2048 x 8192 129 -> 91; 300
// bf16 rows by e4m3 2560 x 9728 32.0 -> 28.0, from HBM 36.1 -> 31.0; 200 by bf16 4096 x 4096 15.8
// unsplit, 21.1 in four splits.
struct Split {
    uint32_t splits;
    bool wide;  // 128 x 128 tiles
};

constexpr uint64_t kCus = 256;

Split plan_split(const ts_linear_args *a) {
    const bool pair = (a->stages & TS_AFTER_SILU_MUL) || a->w_dtype == TS_F32_PARTS;
    const bool xf = a->x_dtype == TS_F32, w8 = a->w_dtype == TS_E4M3;
    const uint32_t steps = a->k / 64;
    Split best = {1, false};
    auto tiles = [&](uint32_t t) { return (uint64_t)((a->n + (pair ? t / 2 : t) - 1) / (pair ? t / 2 : t)) * ((a->m + t - 1) / t); };
    const float sums = 4e-6f * (float)a->m * (float)a->n * (pair ? 2 : 1);  // MB
    auto step_us = [&](bool wide, uint64_t groups) {
        if (groups <= kCus) return wide ? (xf ? 0.99f : w8 ? 0.49f : 0.65f) : xf ? 0.4f : w8 ? 0.2f : 0.21f;
        const float two = wide ? (xf ? 1.7f : 0.82f) : xf ? 0.62f : 0.33f;
        return two / 2 * (float)((groups + kCus - 1) / kCus);
    };
    auto cost = [&](bool wide, uint32_t s) {
        return (float)((steps + s - 1) / s) * step_us(wide, tiles(wide ? 128 : 64) * s) + (s > 1 ? 3.2f + s * (0.1f + 0.37f * sums) : 0.0f);
    };
    if (tiles(64) > 1024) return best;  // enough tiles of some size
    float least = cost(tiles(128) >= 256, 1);
    for (int wide = 0; wide < 2; wide++)
        for (uint32_t s = 2; s <= 16 && 4 * s <= steps; s++)
            if (cost(wide, s) < least) {
                least = cost(wide, s);
                best = {s, wide != 0};
            }
    return best;
}

int tiled(const ts_linear_args *a, bool may_split, void *stream) {
    if (a && ts::block_form(a->w_dtype)) return ts::block_tiled_launch(a, stream);
    TS_REQUIRE(a && a->x && a->w && a->out, "tiled: null pointer");
    TS_REQUIRE(a->m >= 1 && a->n >= 1 && a->k >= 1, "tiled: empty product m=%u n=%u k=%u", a->m, a->n, a->k);
    TS_REQUIRE(a->k % 8 == 0, "tiled: k=%u must be a multiple of 8", a->k);
    TS_REQUIRE(a->x_dtype == TS_F32 || a->x_dtype == TS_BF16, "tiled: x dtype %d", a->x_dtype);
    TS_REQUIRE(a->w_dtype == TS_BF16 || a->w_dtype == TS_E4M3 || a->w_dtype == TS_F32_PARTS,
               "tiled: w dtype %d (f32 weights: pack them with tessera_hip_pack_f32, TS_F32_PARTS)", a->w_dtype);
    TS_REQUIRE(a->w_dtype != TS_F32_PARTS || !(a->stages & TS_AFTER_SILU_MUL),
               "tiled: TS_F32_PARTS weights with TS_AFTER_SILU_MUL");
    TS_REQUIRE(a->out_dtype == TS_F32 || a->out_dtype == TS_BF16, "tiled: out dtype %d", a->out_dtype);
    TS_REQUIRE(a->w_dtype != TS_E4M3 || a->w_scale, "tiled: e4m3 weights need w_scale");
    TS_REQUIRE(!(a->stages & TS_AFTER_ADD) || a->a0, "tiled: TS_AFTER_ADD needs a0");
    TS_REQUIRE(!(a->stages & TS_BEFORE_RMS_NORM), "tiled: RmsNorm prologue is fused only for m <= 16");
    TS_REQUIRE((a->stages & ~(TS_AFTER_ADD | TS_AFTER_SILU_MUL)) == 0, "tiled: unknown stage bits %#x",
               a->stages);
    TS_REQUIRE(ts::aligned(a->x, 16) && ts::aligned(a->w, 16), "tiled: x and w must be 16-byte aligned");
    TiledParams p;
    p.pick_cols = p.few_most = 0;
    int rc = ts::linear_after(a, "tiled", &p.after);
    if (rc) return rc;
    const int big = ts::tiled_big_launch(a, stream);
    if (big != 1) return big;
    // f32 weights as two bf16 parts run as a pair of row blocks, summed at the store.
    const bool parts = a->w_dtype == TS_F32_PARTS;
    const bool silu = (a->stages & TS_AFTER_SILU_MUL) || parts;
    const int32_t w_dtype = parts ? TS_BF16 : a->w_dtype;
    p.pair_sum = parts;
    p.x = a->x; p.w = a->w; p.w_scale = (const uint16_t *)a->w_scale; p.a0 = a->a0; p.out = a->out;
    p.m = a->m; p.n = a->n; p.k = a->k; p.stages = a->stages; p.out_bf16 = a->out_dtype == TS_BF16;
    // 64x64 tiles when 128x128 would give fewer than 2 groups per CU: more groups to
    // hide each one's load/store latency chain (measured: MFMA time is not the limit).
    const uint64_t big_tiles = (uint64_t)((a->n + (silu ? BN / 2 : BN) - 1) / (silu ? BN / 2 : BN)) *
                               ((a->m + BM - 1) / BM);
    const int bt = big_tiles < 512 ? 64 : 128;
    const uint32_t cols = silu ? bt / 2 : bt;
    const uint32_t gx = (a->n + cols - 1) / cols, gy = (a->m + bt - 1) / bt;
    TS_REQUIRE(gy <= 65535, "tiled: m=%u too large for one launch", a->m);
    p.perm = p.row_start = p.tile_start = nullptr;
    p.matrices = 0; p.repeat = 1; p.stride = 0; p.offset = 0;
    const bool xf = a->x_dtype == TS_F32, w8 = w_dtype == TS_E4M3;
    p.splits = 1;
    p.part = nullptr;
    if (pipe_fits(0, a->k, 4)) {
        const Split sp = may_split ? plan_split(a) : Split{1, false};
        const size_t need = sp.splits <= 1 ? 0 : (size_t)sp.splits * a->m * a->n * (silu ? 2 : 1) * sizeof(float);
        if (need && a->workspace && a->workspace_bytes >= need && ts::aligned(a->workspace, 16)) {
            p.splits = sp.splits;
            p.part = (float *)a->workspace;
            const ts_after after = p.after;
            p.after.count = 0;  // the second kernel's
            rc = sp.wide ? pipe_wide<false, kSplit>(p, xf, w8, silu, stream) : pipe_small<kSplit>(p, xf, w8, silu, stream);
            if (rc) return rc;
            ts::SplitSum f = {};
            f.part = p.part; f.splits = p.splits; f.out = a->out; f.a0 = a->a0;
            f.w_scale = w8 ? p.w_scale : nullptr; f.pair_sum = parts;
            f.m = a->m; f.n = a->n; f.k = a->k; f.stages = a->stages; f.out_bf16 = p.out_bf16; f.after = after;
            return ts::split_finish(f, stream);
        }
        // 128 x 128 tiles from one tile per CU up (fewer, larger tiles read less per
        // flop), 64 x 64 below that (measured on the 2048-row projections: q with 256
        // tiles of 128 runs 1.15x faster than with 1024 of 64; o, kv and down with 128
        // tiles of 128 run 1.4-1.5x slower than with 512 of 64).
        const uint64_t oc = silu ? 64 : 128;
        const uint64_t tiles = (a->n + oc - 1) / oc * ((a->m + 127) / 128);
        // 128 x 192 when that fills the 512 group slots (two groups a CU) in fewer
        // rounds of equal work than 128 x 128 does (the C2 gate_up: 768 tiles of 128,
        // a round and a half, against 512 of 192).
        const uint64_t tiles192 = (a->n + oc * 3 / 2 - 1) / (oc * 3 / 2) * ((a->m + 127) / 128);
        const bool wide = ((tiles192 + 511) / 512) * 3 < ((tiles + 511) / 512) * 2;
        // A stage chain takes 64 x 64 tiles: at 128 x 128 its values and sums spill.
        if (p.after.count) return pipe_small<kChain>(p, xf, w8, silu, stream);
        if (tiles < 256) return pipe_small<kPlain>(p, xf, w8, silu, stream);
        if (wide && !xf && !w8) return pipe_launch<128, 192, 64, 2, false, false, false>(p, silu, stream);
        return pipe_wide<false>(p, xf, w8, silu, stream);
    }
    const bool chain = p.after.count;
    Kern k = bt == 64 ? pick_kernel<64, false>(xf, w8, silu, chain) : pick_kernel<128, false>(xf, w8, silu, chain);
    hipLaunchKernelGGL(k, dim3(gx, gy), dim3(kThreads), 0, (hipStream_t)stream, p);
    TS_CHECK_LAUNCH("tiled launch");
    return TS_OK;
}

}  // namespace

extern "C" int tessera_hip_tiled(const ts_linear_args *a, void *stream) { return tiled(a, false, stream); }

static int picked_check(const ts_picked_args *a) {
    TS_REQUIRE(a && a->x && a->w && a->ids && a->out, "picked: null pointer");
    TS_REQUIRE(a->n >= 1 && a->k >= 1, "picked: empty product n=%u k=%u", a->n, a->k);
    TS_REQUIRE(a->k % 8 == 0, "picked: k=%u must be a multiple of 8", a->k);
    TS_REQUIRE(a->count >= 1 && a->count <= 16384, "picked: count=%u (1..16384 matrices)", a->count);
    TS_REQUIRE(a->repeat >= 1, "picked: repeat 0");
    const uint32_t used = (a->stages & TS_AFTER_SILU_MUL) ? 2 * a->n : a->n;
    TS_REQUIRE((uint64_t)a->offset + used <= a->stride, "picked: rows %u..%u outside a matrix of %u rows", a->offset,
               a->offset + used, a->stride);
    TS_REQUIRE(a->x_dtype == TS_F32 || a->x_dtype == TS_BF16, "picked: x dtype %d", a->x_dtype);
    TS_REQUIRE(a->w_dtype == TS_BF16 || a->w_dtype == TS_E4M3, "picked: w dtype %d", a->w_dtype);
    TS_REQUIRE(a->out_dtype == TS_F32 || a->out_dtype == TS_BF16, "picked: out dtype %d", a->out_dtype);
    TS_REQUIRE(a->w_dtype != TS_E4M3 || a->w_scale, "picked: e4m3 weights need w_scale");
    TS_REQUIRE((a->stages & ~TS_AFTER_SILU_MUL) == 0, "picked: stage bits %#x (only TS_AFTER_SILU_MUL)", a->stages);
    TS_REQUIRE(ts::aligned(a->x, 16) && ts::aligned(a->w, 16), "picked: x and w must be 16-byte aligned");
    TS_REQUIRE((uint64_t)a->rows / BM + a->count <= 65535, "picked: %u rows and %u matrices in one launch", a->rows,
               a->count);
    ts_after c;
    return ts::after_check(a->after, true, "picked", &c);
}

extern "C" size_t tessera_hip_picked_workspace(const ts_picked_args *a) {
    if (!a) return 0;
    return ts::route_words(a->rows, a->count) * sizeof(uint32_t);
}

extern "C" int tessera_hip_picked(const ts_picked_args *a, void *stream) {
    const int bad = picked_check(a);
    if (bad) return bad;
    if (a->rows == 0) return TS_OK;
    const size_t need = tessera_hip_picked_workspace(a);
    if (!a->workspace || a->workspace_bytes < need)
        return ts::fail(TS_ERR_WORKSPACE, "picked: workspace %zu bytes, need %zu", a->workspace_bytes, need);
    TS_REQUIRE(ts::aligned(a->workspace, 4), "picked: workspace must be 4-byte aligned");
    const bool xf = a->x_dtype == TS_F32, w8 = a->w_dtype == TS_E4M3;
    const bool pipe = pipe_fits((a->rows - 1) / a->repeat + 1, a->k, xf ? 4 : 2) && !(a->after && a->after->count);
    // Up to 16 rows a matrix on average 32-row tiles: most matrices have one tile either way,
    // and a 128-row one loads its few rows 128 / rows times over beside the weights. 128
    // matrices of 4096 x 1536 at 1 / 16 rows each 213 -> 186 / 324 -> 319 us (2 x 1536 x 4096
    // 374 -> 373 / 575 -> 570: HBM), at 32 rows 350 -> 369; one token's 8 matrices 62 -> 41.
    // A routing may still give most rows to few matrices. Where even that fits two rounds of
    // groups, smaller tiles win (512 rows on 4 of the 128: 39 -> 33 us); past it the matrices
    // of more than 64 rows take 128-row tiles, their weights read once for 128 rows (2048 rows
    // on 4 matrices 67 -> 46 us, 2 x 1536 x 4096 102 -> 74; on Zipf-distributed matrices within 2%
    // of 32-row tiles alone).
    const uint32_t pick_gx = a->stages & TS_AFTER_SILU_MUL ? (a->n + 63) / 64 : (a->n + 127) / 128;
    const bool few = pipe && a->rows <= 16ull * a->count, mixed = few && (uint64_t)a->rows * pick_gx > 32 * 1024;
    const uint32_t few_most = mixed ? 64 : 0;
    ts::Route route;
    int rc = ts::route_launch(a->ids, a->rows, a->first, a->count, few && !mixed ? 32 : BM, few_most, a->workspace, &route,
                              stream);
    if (rc) return rc;
    const bool silu = a->stages & TS_AFTER_SILU_MUL;
    TiledParams p;
    p.pick_cols = 0;
    p.few_most = few_most;
    p.splits = 1;
    p.part = nullptr;
    p.pair_sum = 0;
    ts::after_check(a->after, true, "picked", &p.after);
    rc = ts::zero_absent_launch(route, a->count, a->out, a->n, a->out_dtype == TS_BF16, p.after, stream);
    if (rc) return rc;
    p.x = a->x; p.w = a->w; p.w_scale = (const uint16_t *)a->w_scale; p.a0 = nullptr; p.out = a->out;
    p.m = a->rows; p.n = a->n; p.k = a->k; p.stages = a->stages; p.out_bf16 = a->out_dtype == TS_BF16;
    p.perm = route.perm; p.row_start = route.row_start; p.tile_start = route.tile_start;
    p.matrices = a->count; p.repeat = a->repeat; p.stride = a->stride; p.offset = a->offset;
    const uint32_t cols = silu ? BN / 2 : BN;
    // Row tiles: at most one partial tile per matrix beyond rows / BM full ones.
    const uint32_t gx = (a->n + cols - 1) / cols, gy = (a->rows + BM - 1) / BM + a->count;
    // A stage chain takes the register-staged kernel (the pipelined one's chain variant spills).
    // 128 x 192 tiles where the columns divide evenly (fewer re-reads of the gathered
    // rows per weight byte: C5 gate/up 1249 -> 1202 us), else 128 x 128.
    if (few) return mixed ? pipe_wide<true, kPlain, true>(p, xf, w8, silu, stream) : pipe_few(p, xf, w8, silu, stream);
    if (pipe) {
        if (!xf && !w8 && (silu ? a->n % 96 : a->n % 192) == 0)
            return pipe_launch<128, 192, 64, 2, false, false, true>(p, silu, stream);
        return pipe_wide<true>(p, xf, w8, silu, stream);
    }
    Kern k = pick_kernel<BM, true>(xf, w8, silu, p.after.count != 0);
    hipLaunchKernelGGL(k, dim3(gx, gy), dim3(kThreads), 0, (hipStream_t)stream, p);
    TS_CHECK_LAUNCH("picked launch");
    return TS_OK;
}

extern "C" size_t tessera_hip_linear_workspace(const ts_linear_args *a) {
    if (!a) return 0;
    if (a->m <= 64) return tessera_hip_lanes_workspace(a);
    if (ts::block_form(a->w_dtype) || a->n < 1 || a->k < 64 || !pipe_fits(0, a->k, 4)) return 0;
    const uint32_t splits = plan_split(a).splits;
    const bool pair = (a->stages & TS_AFTER_SILU_MUL) || a->w_dtype == TS_F32_PARTS;
    return splits <= 1 ? 0 : (size_t)splits * a->m * a->n * (pair ? 2 : 1) * sizeof(float);
}

extern "C" int tessera_hip_linear(const ts_linear_args *a, void *stream) {
    TS_REQUIRE(a, "linear: null args");
    return a->m <= 64 ? tessera_hip_lanes(a, stream) : tiled(a, true, stream);
}
