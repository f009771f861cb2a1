// Linear projection to heads with the feature map in the epilogue (gfx950).
//
// The attention modules project their input with torch.nn.Linear layers, view the result
// as heads and push the q and k projections through the feature map
// (random_feature_attention/causal_attention.py:228-247, cross_attention.py:66-76,:279-283,
// utils.py:100-120).  Here one launch computes up to three projections of the same input
//     y_p[r, h, :] = x[r, :] . W_p[h*DH .. h*DH+DH, :]^T + b_p[h*DH ..]        (fp16, fp32 accumulate)
// and, for the projections that ask for it, phi(y_p) = scale * [sin(W' y^), cos(W' y^)] with
// y^ = y / (||y|| + 1e-3), from the tile while it is still in registers.  y is rounded to
// fp16 first, exactly as the unfused chain sees it, and is written out as well (the backward
// of the feature map needs it).
//
// Layouts:  x  [R, E] fp16 row-major          W_p [H*DH, E] fp16 row-major (nn.Linear.weight)
//           b_p [H*DH] fp16 or NULL           y_p [R, H, DH] fp16
//           w' [H, D, DH] fp16                phi_p [R, H, 2D] fp16 (sin block first)
#pragma once
#include "rfa_common.h"
#include "rfa_featuremap.h"

namespace rfa {

constexpr int kMaxProjections = 3;

struct ProjectArgs {
    const half_t* w[kMaxProjections];
    const half_t* b[kMaxProjections];
    half_t* y[kMaxProjections];
    half_t* phi[kMaxProjections];     // NULL: no feature map for this projection
};

// element p of a kernel-argument array without indexing it dynamically (which would copy the
// struct to private memory)
template <typename T>
__device__ __forceinline__ T pick3(T const (&a)[kMaxProjections], int p) {
    return p == 0 ? a[0] : (p == 1 ? a[1] : a[2]);
}

// A stage array whose rows are 32 KG halves of the contraction (KG groups of waves side by side), stored without
// padding (a direct load writes 1 KiB in lane order): the 16-byte pieces of row r are stored rotated, piece c at slot
// c ^ (r's number within 256 bytes' worth of rows), which spreads a wave's operand read (16 rows x 16 bytes per 16 lanes)
// over all banks.  slot() is its own inverse.
template <int KG>
struct StageRows {
    static constexpr int kSlots = 4 * KG;
    static __device__ __forceinline__ int slot(int r, int c) { return c ^ ((r / (4 / KG)) % kSlots); }
};

// Sums of one tile over KG groups of four waves, each of which walked its own share of the contraction: wave w of every
// group holds the same tiles acc[NR][NC].  Group g < kFin leaves with own[l] = the sum of acc[kFin l + g] over all groups
// (its own first, then the others in order); the rest have nothing left to do.  One workgroup barrier, all groups call.
template <int NR, int NC, int KG>
struct GroupSum {
    static constexpr int kFin = KG > 1 && NR % 2 == 0 ? 2 : 1;
    static constexpr int kOwn = NR / kFin;
    static constexpr size_t kLds = (size_t)(KG - 1) * NR * NC * kThreads * 16;
    static __device__ __forceinline__ void run(const f4 (&acc)[NR][NC], f4 (&own)[kOwn][NC], unsigned char* lds, int kg, int tid) {
        if constexpr (KG == 1) {
#pragma unroll
            for (int a = 0; a < NR; ++a)
#pragma unroll
                for (int c = 0; c < NC; ++c) own[a][c] = acc[a][c];
        } else {
            // [finishing group][other group, in order][tile][thread]
            f4* const red = reinterpret_cast<f4*>(lds) + tid;
            auto slot = [&](int fin, int g) { return red + (fin * (KG - 1) + (g < fin ? g : g - 1)) * (kOwn * NC * kThreads); };
#pragma unroll
            for (int o = 0; o < kFin; ++o) {
                if (kg == o) continue;
                f4* const to = slot(o, kg);
#pragma unroll
                for (int l = 0; l < kOwn; ++l)
#pragma unroll
                    for (int c = 0; c < NC; ++c) to[(l * NC + c) * kThreads] = acc[kFin * l + o][c];
            }
            __syncthreads();
#pragma unroll
            for (int l = 0; l < kOwn; ++l)
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const f4 first = acc[kFin * l][c], second = acc[kFin * l + kFin - 1][c];     // values: no indexed registers
                    own[l][c] = kg == 1 ? second : first;
                }
            if (kg < kFin) {
                const f4* const from = red + kg * (KG - 1) * (kOwn * NC * kThreads);
#pragma unroll
                for (int j = 0; j < KG - 1; ++j)
#pragma unroll
                    for (int l = 0; l < kOwn; ++l)
#pragma unroll
                        for (int c = 0; c < NC; ++c) own[l][c] += from[(j * kOwn * NC + l * NC + c) * kThreads];
            }
        }
    }
};

template <int D, int DH, int BM_, int KG_ = 1>
struct ProjectCfg {
    static_assert(D % 32 == 0 && (DH == 64 || DH == 128), "D multiple of 32, DH 64 or 128");
    static constexpr int BM = BM_;                 // rows of x per workgroup
    static constexpr int BN = 128;                 // output columns: one head of 128 or two of 64
    static constexpr int BK = 32;                  // contraction step: one MFMA deep
    static constexpr int kStages = 3;              // 4 to 6 measured no faster at any size, with any number of groups
    static constexpr int PPT = BN / DH;            // heads per tile
    static constexpr int WR = 4 / PPT;             // waves along the rows; a wave owns whole heads
    static constexpr int RW = BM / WR;             // rows of a wave
    static constexpr int NR = RW / 16, NC = DH / 16;
    static constexpr int XI = BM / 64, WI = BN / 64;    // 1 KiB pieces of a stage per wave: x, W
    static constexpr int KG = KG_;                 // groups of four waves that share a tile's contraction
    static constexpr int kStageHalves = (BM + BN) * BK;
    static constexpr int LDW = DH + lds_pad(DH);   // rows of w'
    using Sum = GroupSum<NR, NC, KG>;
    static constexpr size_t kLoopLds = (size_t)kStages * KG * kStageHalves * 2;
    static constexpr size_t kEpiLds = Sum::kLds + (size_t)PPT * D * LDW * 2;
    static constexpr size_t kLds = kLoopLds > kEpiLds ? kLoopLds : kEpiLds;
    static_assert(kLds <= (KG == 1 ? 80 : 160) * 1024, "two workgroups per CU, one of several groups");
};

// 64 lanes x 16 bytes, global -> LDS without registers: lane l's bytes land at lds + 16 l
__device__ __forceinline__ void dma16(const char* g, half_t* lds) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                     (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// The same through a wave-uniform base and a 32-bit lane offset, hidden from the compiler: it makes every
// transposing LDS read wait for all direct loads it knows of (which a ring of stages must not)
__device__ __forceinline__ void dma16_opaque(const half_t* base, unsigned off_bytes, const half_t* lds) {
    const unsigned at = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) half_t*)lds;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 ::"s"(__builtin_amdgcn_readfirstlane(at)), "v"(off_bytes), "s"(base) : "memory", "m0");
}

// All but the last N direct loads of this wave have landed and its LDS reads are done; then the
// workgroup barrier: everyone's share of the stage is in place, the stage before it is free.
template <int N>
__device__ __forceinline__ void stage_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// One 128-column tile (one head of 128 or two of 64) of BM rows per workgroup of four waves.
//
// What bounds it: at large sizes the matrix pipes and the operand path L2 -> LDS behind them; where
// a tile has few contraction steps (E = 512: 16), its start and the stores of y and phi.  So:
// operands go to LDS directly (no registers, no store instructions), three stages of 32 deep in a
// ring, one barrier per step; two (256 rows) or three (128) workgroups share a CU, so that one's
// epilogue runs under another's products.  A wave owns BM / 2 rows x 64 columns (or BM / 4 x 128):
// with 256 rows 12 operand reads for 32 MFMAs, 48 KB of LDS traffic per 512 clocks of the matrix pipes.
// Where there is at most one tile to a CU nothing hides a step (0.3 us at 64 rows: barrier, direct loads of 18 bytes a
// clock, operand reads, products, one after the other), so KG = 2 groups of four waves take 32 columns each of a stage of
// 64: whole 128-byte lines, half the steps, 26 bytes a clock; the groups' sums meet in LDS.
//
// Measured (us; q, k, v projections with phi(q), phi(k); before: rows of x in registers for E <= 512,
// a register-staged two-buffer loop otherwise):
//   8192 rows, E 512, 8 heads of 64, D 64       42.1 -> 28.2      8192, 1024, 8 of 128, D 128   112 -> 83
//   32768, 1024, 16 of 64, D 64                  964 -> 304 (678 TFLOP/s)      512, 512   12.4 -> 9.6 -> 7.5 (two groups)
//   one projection without phi: 4096, 512 7.4 -> 6.6; 2048, 1024 11.3 -> 9.1 (two groups)
//
// LDS stage: x tile [BM][32 KG], then W tile [128][32 KG] halves (StageRows).  The rows of
// W sit in pair order (pair_pos), so that accumulator tiles 2p, 2p + 1 give lane (i, G) the 8
// consecutive columns 32 p + 8 G of row i: y goes out in 16-byte pieces, is the operand of the
// feature product as it stands, and phi goes out the same way; nothing passes through LDS again.
//
// Tiles are numbered row tile by row tile; each XCD gets a contiguous range of numbers, so that
// the tiles that share rows of x meet in its L2.   grid = 8 * ceil(tiles / 8).
template <int D, int DH, int BM_, int KG>
__global__ __launch_bounds__(kThreads * KG, 2) void k_project_phi(
    const half_t* __restrict__ x, ProjectArgs pa, const half_t* __restrict__ wf, int R, int E, int H, int np,
    int tiles_c, int tiles, float scale) {
    using Cfg = ProjectCfg<D, DH, BM_, KG>;
    using Sum = typename Cfg::Sum;
    constexpr int BM = Cfg::BM, BK = Cfg::BK, STAGES = Cfg::kStages, NR = Cfg::NR, NC = Cfg::NC, LDW = Cfg::LDW;
    extern __shared__ __align__(16) unsigned char smem_raw[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
    const int wv = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);      // wave inside its group
    half_t* const smem = reinterpret_cast<half_t*>(smem_raw);
    const int i = lane & 15, G = lane >> 4;

    const int per_xcd = (tiles + kXcds - 1) / kXcds;
    const int tile = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (tile >= tiles) return;                         // whole workgroup: padding of the grid
    const int row0 = (tile / tiles_c) * BM;
    const int hp0 = (tile % tiles_c) * Cfg::PPT;       // (projection, head) pairs: hp -> hp / H, hp % H
    const int pairs = H * np;

    // ---- direct-load addresses: wave-uniform base + 32-bit lane offset, set up once.  A load covers 64 / kSlots rows.
    using Rows = StageRows<KG>;
    constexpr int SK = BK * KG, RPL = 64 / Rows::kSlots;      // columns of a stage; rows of one load
    const int wave = kg * 4 + wv;
    const char* xbase = reinterpret_cast<const char*>(x + (int64_t)row0 * E);
    unsigned xoff[Cfg::XI], woff[Cfg::WI];
#pragma unroll
    for (int it = 0; it < Cfg::XI; ++it) {
        const int r = (wave * Cfg::XI + it) * RPL + lane / Rows::kSlots;
        xoff[it] = (unsigned)min(r, R - 1 - row0) * (unsigned)(E * 2) + Rows::slot(r, lane % Rows::kSlots) * 16;
    }
    // W rows of this wave: 32 / KG of them, never across a 32-row group or a head
    constexpr int WRW = 32 / KG;
    const int wrow0 = WRW * wave / 32 * 32;            // first row of the 32-row group
    const int hp_ld = min(hp0 + wrow0 / DH, pairs - 1);
    const char* wbase = reinterpret_cast<const char*>(
        pick3(pa.w, hp_ld / H) + ((int64_t)(hp_ld % H) * DH + wrow0 % DH) * E);
#pragma unroll
    for (int it = 0; it < Cfg::WI; ++it) {
        const int r = WRW * wave - wrow0 + it * RPL + lane / Rows::kSlots;      // LDS row within the group; it holds column pair_inv
        const int c = (r & 3) | ((r & 16) >> 2) | ((r & 12) << 1);
        woff[it] = (unsigned)c * (unsigned)(E * 2) + Rows::slot(wrow0 + r, lane % Rows::kSlots) * 16;
    }
    half_t* const xdst = smem + wave * Cfg::XI * 512;
    half_t* const wdst = smem + BM * SK + wave * Cfg::WI * 512;
    constexpr int kRing = KG * Cfg::kStageHalves;      // halves from one stage to the next
    auto load_stage = [&](int step, int buf) {
        const char* xb = xbase + (int64_t)step * (SK * 2);
        const char* wb = wbase + (int64_t)step * (SK * 2);
#pragma unroll
        for (int it = 0; it < Cfg::XI; ++it) dma16(xb + xoff[it], xdst + buf * kRing + it * 512);
#pragma unroll
        for (int it = 0; it < Cfg::WI; ++it) dma16(wb + woff[it], wdst + buf * kRing + it * 512);
    };
    constexpr int kPerStage = Cfg::XI + Cfg::WI;

    // y^T tiles (m = output column in pair order, n = row) of this wave's rows and head
    const int wr = wv / Cfg::PPT, wc = wv % Cfg::PPT;
    f4 acc[NR][NC];
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[a][c] = f4_zero();

    // operand rows of this lane inside a stage: row (16 t + i), piece G of its group's columns
    const int piece = Rows::slot(i, 4 * kg + G) * 8;
    const half_t* const xop = smem + (wr * Cfg::RW + i) * SK + piece;
    const half_t* const wop = smem + BM * SK + (wc * DH + i) * SK + piece;

    const int nk = E / (BK * KG);       // KG divides the steps
#pragma unroll
    for (int k = 0; k < STAGES - 1; ++k) load_stage(min(k, nk - 1), k);
    int buf = 0;
    for (int kk = 0; kk < nk; ++kk) {
        // stage kk has landed (the STAGES - 2 after it may still be on their way), stage kk - 1 is free
        stage_barrier<(STAGES - 2) * kPerStage>();
        // the last steps re-request the last stage's columns into buffers nobody reads again
        load_stage(min(kk + STAGES - 1, nk - 1), buf == 0 ? STAGES - 1 : buf - 1);
        const half_t* xs = xop + buf * kRing;
        const half_t* wsm = wop + buf * kRing;
        h8 wa[NC], xb[NR];
#pragma unroll
        for (int c = 0; c < NC; ++c) wa[c] = *reinterpret_cast<const h8*>(wsm + c * 16 * SK);
#pragma unroll
        for (int a = 0; a < NR; ++a) xb[a] = *reinterpret_cast<const h8*>(xs + a * 16 * SK);
        __builtin_amdgcn_s_setprio(1);      // the other workgroup's loads and epilogue give way: 2 % at full size
#pragma unroll
        for (int a = 0; a < NR; ++a)
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[a][c] = mfma32(wa[c], xb[a], acc[a][c]);
        __builtin_amdgcn_s_setprio(0);
        buf = buf == STAGES - 1 ? 0 : buf + 1;
    }

    // ---- epilogue: the ring becomes the place of the groups' sums and of w' (rows in pair order)
    stage_barrier<0>();
    half_t* const wfs = reinterpret_cast<half_t*>(smem_raw + Sum::kLds);
    const int hp = hp0 + wc;
    const bool live = hp < pairs;                      // an odd number of 64-wide heads leaves half a tile
    const int hpc = live ? hp : pairs - 1;
    const int p = hpc / H, h = hpc % H;
    half_t* const y = pick3(pa.y, p);
    half_t* const phi = pick3(pa.phi, p);
    const half_t* const bias = pick3(pa.b, p);
    if (wf) {
#pragma unroll
        for (int u = 0; u < Cfg::PPT; ++u) {
            const int hu = min(hp0 + u, pairs - 1);
            if (pick3(pa.phi, hu / H))
                load_w_pair_order<D, DH, kThreads * KG>(wfs + u * D * LDW, wf + (int64_t)(hu % H) * D * DH, tid);
        }
    }
    h8 bv[NC / 2];
#pragma unroll
    for (int c = 0; c < NC / 2; ++c) {
#pragma unroll
        for (int e = 0; e < 8; ++e) bv[c][e] = (half_t)0.f;
        if (bias) {
            const h4* b4 = reinterpret_cast<const h4*>(bias + h * DH + 32 * c + 8 * G);    // 8-byte aligned
            bv[c] = __builtin_shufflevector(b4[0], b4[1], 0, 1, 2, 3, 4, 5, 6, 7);
        }
    }
    f4 own[Sum::kOwn][NC];
    Sum::run(acc, own, smem_raw, kg, tid & (kThreads - 1));
    if (KG == 1) __syncthreads();
    if (!live || kg >= Sum::kFin) return;
    const half_t* const Wfs = wfs + wc * D * LDW;
#pragma unroll
    for (int a = 0; a < Sum::kOwn; ++a) {
        const int r = row0 + wr * Cfg::RW + 16 * (Sum::kFin * a + kg) + i;
        const int64_t at = (int64_t)r * H + h;
        h8 op[NC / 2];       // the rounded row pieces: y as stored, and the operand of the feature product
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < NC / 2; ++c) {
#pragma unroll
            for (int e = 0; e < 8; ++e) op[c][e] = (half_t)(own[a][2 * c + e / 4][e % 4] + (float)bv[c][e]);
            ss += dot_h8(__builtin_bit_cast(uint4, op[c]), __builtin_bit_cast(uint4, op[c]));
        }
        if (y && r < R) {    // NULL: the caller keeps only phi(y) (no backward pass will ask for y)
#pragma unroll
            for (int c = 0; c < NC / 2; ++c) *reinterpret_cast<h8*>(y + at * DH + 32 * c + 8 * G) = op[c];
        }
        if (phi) {
            ss = sum_over_groups(ss);
            const float inv_turns = rcp_nr(__builtin_amdgcn_sqrtf(ss) + 1e-3f) * 0.15915494309189535f;
#pragma unroll
            for (int t = 0; t < D / 32; ++t) {
                f4 u[2] = {f4_zero(), f4_zero()};      // u^T tiles 2t, 2t + 1 (m = feature, n = row)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int c = 0; c < NC / 2; ++c)
                        u[q] = mfma32(row8(Wfs, LDW, 32 * t + 16 * q + i, 32 * c, G), op[c], u[q]);
                h8 sv, cv;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float s_, c_;
                    sincos_turns(u[e / 4][e % 4] * inv_turns, s_, c_);
                    sv[e] = (half_t)(scale * s_);
                    cv[e] = (half_t)(scale * c_);
                }
                if (r < R) {
                    *reinterpret_cast<h8*>(phi + at * (2 * D) + 32 * t + 8 * G) = sv;
                    *reinterpret_cast<h8*>(phi + at * (2 * D) + D + 32 * t + 8 * G) = cv;
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// y[r][o] = x[r] . W[o] + b[o] for few rows: the projections of a decoding step.
//
// What bounds it is the trips to memory and the launch around them: a workgroup of four waves owns 16 or 32 columns (rows of
// W) of 16 to 64 rows of x, the waves share the contraction, each with four 32-deep steps in flight together (the
// loads of a batch before its first product, no branch between them), operands straight from memory in the
// lanes' own order; the four partial sums meet in LDS.  A lane's 16 bytes lie a whole row from its neighbour's, so
// a load asks for 16 lines: what a CU asks for decides, so the tile is the smallest that one round of workgroups allows.
// Every tile adds in the same order: y of a row is the same whatever rows it comes with.
// Measured, device us with 64 x 16 from 33 rows on and 64 x 32 past a workgroup per CU / now / the library's product (which
// costs 19 us of host time, this 4): 4 rows 512 -> 1536 2.6 / 2.6 / 3.9, 1024 -> 3072 3.6 / 3.6 / 5.7; 64 rows 512 -> 512 4.2 /
// 2.8 / 5.6, 768 -> 768 5.9 / 3.5 / 5.7, 1024 -> 1024 6.4 / 3.7, 1024 -> 3072 6.9 / 6.3 / 8.3; 160 rows 512 -> 512 4.3 / 3.3; 320 rows
// 1024 -> 1024 7.7 / 7.7 / 6.5.  Eight waves with two steps each: 64 rows 1024 -> 3072 6.1, 768 -> 768 4.0, else the same.
// Up to three layers over the same rows side by side, y [R][np Eo]: their weights stay where they are, as a stack of them
// would have to be formed again whenever one changes, and at every replay of a captured step.
// grid = (ceil(np Eo / (16 CT)), ceil(R / (16 RT)));  E % 32 == 0, Eo % 16 == 0
// ---------------------------------------------------------------------------
struct RowLayers {
    const half_t* w[kMaxProjections];
    const half_t* bias[kMaxProjections];      // NULL: none
};

template <int RT, int CT, bool SEVERAL>
__global__ __launch_bounds__(kThreads) void k_linear_rows(const half_t* __restrict__ x, RowLayers layers, half_t* __restrict__ y,
                                                          int R, int E, int Eo, int np) {
    __shared__ f4 red[4][RT * CT][64];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // the wave's bounds are scalar: no lane masks
    const int i = lane & 15, G = lane >> 4;
    const int c0 = 16 * CT * blockIdx.x, r0 = 16 * RT * blockIdx.y;
    const int nk = E / 32, per_wave = (nk + 3) / 4;
    const int k_begin = min(wv * per_wave, nk), k_end = min(k_begin + per_wave, nk);
    const int cols = SEVERAL ? np * Eo : Eo;
    // 16 columns lie within one layer (past the last one: its last 16 again)
    auto layer = [&](int c16) { return !SEVERAL || c16 < Eo ? 0 : (c16 - Eo < Eo ? 1 : 2); };
    const half_t* wp[CT];
    const half_t* xp[RT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int c16 = min(c0 + 16 * c, cols - 16), p = layer(c16);
        wp[c] = (SEVERAL ? pick3(layers.w, p) : layers.w[0]) + (int64_t)(c16 - p * Eo + i) * E + 8 * G;
    }
#pragma unroll
    for (int a = 0; a < RT; ++a) xp[a] = x + (int64_t)min(r0 + 16 * a + i, R - 1) * E + 8 * G;
    f4 acc[RT][CT];      // y^T tiles: lane (i, G) holds columns 4G .. of row i
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[a][c] = f4_zero();
    constexpr int U = 4;      // steps in flight; 8 only repeat the last step's loads where E = 512
    // steps k .. k + U - 1, no branch between the loads; steps from `end` on (none unless `ragged`) count as zeros
    auto batch = [&](int k, int end, auto ragged) __attribute__((always_inline)) {
        h8 wa[U][CT], xb[U][RT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kk = 32 * (ragged ? min(k + u, end - 1) : k + u);
#pragma unroll
            for (int c = 0; c < CT; ++c) wa[u][c] = *reinterpret_cast<const h8*>(wp[c] + kk);
#pragma unroll
            for (int a = 0; a < RT; ++a) xb[u][a] = *reinterpret_cast<const h8*>(xp[a] + kk);
        }
        __builtin_amdgcn_sched_barrier(0);      // all loads of the batch before its first product
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (ragged) {
                const bool live = k + u < end;
#pragma unroll
                for (int c = 0; c < CT; ++c) wa[u][c] = live ? wa[u][c] : h8_zero();
#pragma unroll
                for (int a = 0; a < RT; ++a) xb[u][a] = live ? xb[u][a] : h8_zero();
            }
#pragma unroll
            for (int a = 0; a < RT; ++a)
#pragma unroll
                for (int c = 0; c < CT; ++c) acc[a][c] = mfma32(wa[u][c], xb[u][a], acc[a][c]);
        }
    };
    int k = k_begin;
    for (; k + U <= k_end; k += U) batch(k, k_end, std::false_type{});
    if (k < k_end) batch(k, k_end, std::true_type{});
#pragma unroll
    for (int a = 0; a < RT; ++a)
#pragma unroll
        for (int c = 0; c < CT; ++c) red[wv][a * CT + c][lane] = acc[a][c];
    __syncthreads();
    for (int t = wv; t < RT * CT; t += 4) {
        const int r = r0 + 16 * (t / CT) + i, col = c0 + 16 * (t % CT) + 4 * G;
        const f4 s = (red[0][t][lane] + red[1][t][lane]) + (red[2][t][lane] + red[3][t][lane]);
        if (r < R && col < cols) {
            const int p = layer(c0 + 16 * (t % CT));
            const half_t* const bias = SEVERAL ? pick3(layers.bias, p) : layers.bias[0];
            h4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (half_t)(s[e] + (bias ? (float)bias[col - p * Eo + e] : 0.f));
            *reinterpret_cast<h4*>(y + (int64_t)r * cols + col) = o;
        }
    }
}

// ---------------------------------------------------------------------------
// Weight and bias gradients of those Linear layers:
//     dW_p[o][c] = sum_r dy_p[r][o] * x[r][c],      db_p[o] = sum_r dy_p[r][o]
// (what autograd computes for torch.nn.Linear).  The contraction runs over the R rows, far
// longer than either output side, so it is split: workgroup (split s, projection p, tile)
// sums a 128 x 128 tile of dW_p over the rows of split s into an fp32 partial, and
// k_weight_grad_reduce adds the partials.  Both operands are contracted over their row index,
// i.e. read from their row-major LDS tiles with the transposing read.
// Layouts: x [R, Ei], dy_p [R, Eo] fp16 row-major; part [nsplit][np][Eo][Ei], bpart
// [nsplit][np][Eo] fp32; dW_p [Eo, Ei], db_p [Eo] fp16.
// ---------------------------------------------------------------------------
struct WeightGradArgs {
    const half_t* dy[kMaxProjections];
    half_t* dw[kMaxProjections];
    half_t* db[kMaxProjections];      // NULL: no bias gradient for this projection
};

struct WeightGradCfg {
    static constexpr int TO = 128, TI = 128, C = 32;       // tile of dW, rows per step: one MFMA deep
    static constexpr int kStages = 3;                      // 4 and 5 measured the same
    static constexpr int NO = TO / 32, NI = TI / 32;       // 16-wide tiles of a wave: 64 x 64
    static constexpr int kStageHalves = C * (TO + TI);
    template <int KG> using Sum = GroupSum<NO, NI + 1, KG>;
    template <int KG> static constexpr size_t kLds =
        (size_t)kStages * KG * kStageHalves * 2 > Sum<KG>::kLds ? (size_t)kStages * KG * kStageHalves * 2 : Sum<KG>::kLds;
    static constexpr int YI = C * TO / 2048, XI = C * TI / 2048;   // 1 KiB pieces of a stage per wave
};

// Column fragment X[8G + e][c0 + i], e = 0..7, of a stage array [32][LD] (LD halves per row, no
// padding): like col8, with the 32-byte segments of row r stored at segment ^ (r % 4 + 4 (r / 8 % 2)),
// which spreads the 16 row pieces of a transposing read over all banks.  The rotation depends on
// the lane's first row only (4 rows further it is the same).
template <int LD>
__device__ __forceinline__ h8 col8_rot(const half_t* X, int seg, int lane) {
    const int s = lane & 15, G = lane >> 4;
    const int r = 8 * G + (s >> 2);
    const half_t* p = X + r * LD + (seg ^ ((s >> 2) | ((G & 1) << 2))) * 16 + 4 * (s & 3);
    const h4 a = tr_read4(p);
    const h4 b = tr_read4(p + 4 * LD);
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Workgroup (split s, projection p, tile): a 128 x 128 tile of dW_p over the rows of split s, four waves of
// 64 x 64, steps of 32 rows through a three-stage ring of direct loads with one barrier per step (the
// layout and the waits of k_project_phi).  What bounds it is the step itself -- barrier, transposing
// reads, 16 products -- which two to three workgroups per CU hide in each other; tiles of 256 x 128 spill.
// Measured with k_weight_grad_reduce, us (before: register-staged loads, two buffers, at least 8 splits):
// 8192 rows, 512 -> 3 x 512 36.4 -> 25.8; 1024 -> 3 x 1024 94 -> 67 (770 TFLOP/s); 1024 -> 1024 35.3 -> 29.9;
// 512 -> 512 26.0 -> 23.2; 1000 rows, 384 -> 3 x 384 22.8 -> 14.4.
// grid = 8 * ceil(work / 8), work = nsplit * np * tiles; each XCD gets a contiguous range of the numbers
// (split first), so that the workgroups that share rows of x and dy meet in its L2.  rows_per_split is a
// multiple of 32.  WIDE: rows of more than 2^26 halves, 32 of which lie beyond a 32-bit byte offset.
template <bool WIDE, int KG>
__device__ __forceinline__ void weight_grad_tile(unsigned char* smem_raw, int idx, const half_t* __restrict__ x,
                                                 const WeightGradArgs& wa, int64_t ld, float* __restrict__ part,
                                                 float* __restrict__ bpart, int R, int Eo, int Ei, int np, int rows_per_split) {
    using Cfg = WeightGradCfg;
    using Sum = typename Cfg::template Sum<KG>;
    constexpr int TO = Cfg::TO, TI = Cfg::TI, C = Cfg::C, NO = Cfg::NO, NI = Cfg::NI, STAGES = Cfg::kStages;
    constexpr int kRing = KG * Cfg::kStageHalves;

    const int tid = threadIdx.x, lane = tid & 63;
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
    const int wv = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);      // wave inside its group
    half_t* const smem = reinterpret_cast<half_t*>(smem_raw) + kg * Cfg::kStageHalves;      // the group's part of a stage
    const int i = lane & 15, G = lane >> 4;
    const int wo = wv >> 1, wi = wv & 1;                  // wave -> quadrant of the tile

    const int tiles_i = Ei / TI, tiles_o = Eo / TO;
    const int ti = idx % tiles_i; idx /= tiles_i;
    const int to = idx % tiles_o; idx /= tiles_o;
    const int p = idx % np, s = idx / np;
    const int r_begin = s * rows_per_split, r_end = min(r_begin + rows_per_split, R);
    const int o0 = to * TO, c0 = ti * TI;
    const bool with_bias = ti == 0 && wi == 0 && pick3(wa.db, p) != nullptr;   // wave-uniform

    // (m = o, n = c) tiles of this wave's quadrant; the last of a row: column sums of dy, the same in every column n
    f4 acc[NO][NI + 1];
#pragma unroll
    for (int a = 0; a < NO; ++a)
#pragma unroll
        for (int b = 0; b <= NI; ++b) acc[a][b] = f4_zero();
    const h8 ones = h8_ones();

    if (r_begin < r_end) {
        // 1 KiB of a stage array per instruction: 512 / LD rows, lane -> (row, 16-byte piece)
        const half_t* const dyb = pick3(wa.dy, p) + (int64_t)r_begin * ld + o0;
        const half_t* const xb = x + (int64_t)r_begin * Ei + c0;
        const int nrows = r_end - r_begin, nk = (nrows + C - 1) / C;
        auto rot = [](int r) { return ((r & 3) | ((r >> 1) & 4)) * 2; };
        // byte offsets inside a step; the rows of the last step past the end read the last row (both operands
        // drop them: that row may hold an infinity, and 0 times it is not a number)
        using Offset = std::conditional_t<WIDE, int64_t, unsigned>;
        Offset yoff[2][Cfg::YI], xoff[2][Cfg::XI];
#pragma unroll
        for (int last = 0; last < 2; ++last) {
            const int rmax = last ? nrows - 1 - (nk - 1) * C : C - 1;
#pragma unroll
            for (int it = 0; it < Cfg::YI; ++it) {
                const int r = (wv * Cfg::YI + it) * (512 / TO) + lane / (TO / 8);
                yoff[last][it] = (Offset)min(r, rmax) * ((Offset)ld * 2) + ((lane % (TO / 8)) ^ rot(r)) * 16;
            }
#pragma unroll
            for (int it = 0; it < Cfg::XI; ++it) {
                const int r = (wv * Cfg::XI + it) * (512 / TI) + lane / (TI / 8);
                xoff[last][it] = (Offset)min(r, rmax) * ((Offset)Ei * 2) + ((lane % (TI / 8)) ^ rot(r)) * 16;
            }
        }
        auto dma = [](const half_t* base, Offset off, half_t* lds) __attribute__((always_inline)) {
            if constexpr (WIDE) dma16(reinterpret_cast<const char*>(base) + off, lds);
            else dma16_opaque(base, off, lds);
        };
        auto load_stage = [&](int step, int buf) {
            const int kk = min(step * KG + kg, nk - 1);
            half_t* st = smem + buf * kRing;
            const half_t* yb = dyb + (int64_t)kk * C * ld;
            const half_t* xk = xb + (int64_t)kk * C * Ei;
            const bool last = kk == nk - 1;
#pragma unroll
            for (int it = 0; it < Cfg::YI; ++it)
                dma(yb, last ? yoff[1][it] : yoff[0][it], st + (wv * Cfg::YI + it) * 512);
#pragma unroll
            for (int it = 0; it < Cfg::XI; ++it)
                dma(xk, last ? xoff[1][it] : xoff[0][it], st + C * TO + (wv * Cfg::XI + it) * 512);
        };
        const int nsteps = (nk + KG - 1) / KG;
#pragma unroll
        for (int k = 0; k < STAGES - 1; ++k) load_stage(k, k);
        int buf = 0;
        for (int step = 0; step < nsteps; ++step) {
            const int kk = step * KG + kg;      // past nk in the last step: nothing is kept
            stage_barrier<(STAGES - 2) * (Cfg::YI + Cfg::XI)>();
            load_stage(step + STAGES - 1, buf == 0 ? STAGES - 1 : buf - 1);
            const half_t* Ys = smem + buf * kRing;
            const half_t* Xs = Ys + C * TO;
            h8 xa[NI], ya[NO];
#pragma unroll
            for (int b = 0; b < NI; ++b) xa[b] = col8_rot<TI>(Xs, 4 * wi + b, lane);
#pragma unroll
            for (int a = 0; a < NO; ++a) ya[a] = col8_rot<TO>(Ys, NO * wo + a, lane);
            if (kk * C + C > nrows) {                     // the ragged end of the rows
                const int keep = nrows - kk * C - 8 * G;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
#pragma unroll
                    for (int a = 0; a < NO; ++a) ya[a][e] = e < keep ? ya[a][e] : (half_t)0.f;
#pragma unroll
                    for (int b = 0; b < NI; ++b) xa[b][e] = e < keep ? xa[b][e] : (half_t)0.f;
                }
            }
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int a = 0; a < NO; ++a) {
#pragma unroll
                for (int b = 0; b < NI; ++b) acc[a][b] = mfma32(ya[a], xa[b], acc[a][b]);
            }
            if (with_bias) {
#pragma unroll
                for (int a = 0; a < NO; ++a) acc[a][NI] = mfma32(ya[a], ones, acc[a][NI]);
            }
            __builtin_amdgcn_s_setprio(0);
            buf = buf == STAGES - 1 ? 0 : buf + 1;
        }
        // the last re-requested stages are still on their way into this workgroup's LDS: they land before it ends
        stage_barrier<0>();
    }
    f4 own[Sum::kOwn][NI + 1];
    Sum::run(acc, own, smem_raw, kg, tid & (kThreads - 1));
    if (kg >= Sum::kFin) return;
    float* po = part + ((int64_t)(s * np + p) * Eo + o0 + TO / 2 * wo) * Ei + c0 + 64 * wi;
#pragma unroll
    for (int l = 0; l < Sum::kOwn; ++l) {
        const int o = 16 * (Sum::kFin * l + kg) + 4 * G;
#pragma unroll
        for (int b = 0; b < NI; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) po[(int64_t)(o + e) * Ei + 16 * b + i] = own[l][b][e];
    }
    if (with_bias && i == 0) {
        float* pb = bpart + (int64_t)(s * np + p) * Eo + o0 + TO / 2 * wo;
#pragma unroll
        for (int l = 0; l < Sum::kOwn; ++l) *reinterpret_cast<f4*>(pb + 16 * (Sum::kFin * l + kg) + 4 * G) = own[l][NI];
    }
}

// work number of this workgroup: each XCD gets a contiguous range (grid = 8 * ceil(work / 8)); >= work: none
__device__ __forceinline__ int xcd_range(int block, int work) {
    return (block % kXcds) * ((work + kXcds - 1) / kXcds) + block / kXcds;
}

template <bool WIDE>
__global__ __launch_bounds__(kThreads, 2) void k_weight_grad_partial(
    const half_t* __restrict__ x, WeightGradArgs wa, int64_t ld, float* __restrict__ part, float* __restrict__ bpart, int R,
    int Eo, int Ei, int np, int nsplit, int rows_per_split) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int work = nsplit * np * (Eo / WeightGradCfg::TO) * (Ei / WeightGradCfg::TI), idx = xcd_range(blockIdx.x, work);
    if (idx < work) weight_grad_tile<WIDE, 1>(smem_raw, idx, x, wa, ld, part, bpart, R, Eo, Ei, np, rows_per_split);
}

// ---------------------------------------------------------------------------
// Input gradient of those Linear layers: dx[r][c] = sum_p sum_o dy_p[r][o] W_p[o][c], one contraction over the
// output columns of all of them (fp32 accumulate, one rounding; autograd adds rounded products).
// Layouts: dy_p [R, Eo] with rows ld halves apart (the thirds of a packed gradient: 3 Eo), W_p [Eo, Ei], dx [R, Ei].
// ---------------------------------------------------------------------------
struct InputGradArgs {
    const half_t* dy[kMaxProjections];
    const half_t* w[kMaxProjections];
};

template <int BM_, int KG_ = 1>
struct InputGradCfg {
    static constexpr int BM = BM_, BN = 128, BK = 32, kStages = 3;
    static constexpr int RW = BM / 2, NR = RW / 16, NC = 4;       // a wave: BM / 2 rows x 64 columns
    static constexpr int YI = BM / 64, WI = 2;                    // 1 KiB pieces of a stage per wave: dy, W
    static constexpr int KG = KG_;
    static constexpr int kStageHalves = (BM + BN) * BK;
    using Sum = GroupSum<NR, NC, KG>;
    static constexpr size_t kLoopLds = (size_t)kStages * KG * kStageHalves * 2;
    static constexpr size_t kLds = kLoopLds > Sum::kLds ? kLoopLds : Sum::kLds;
};

// A tile of BM rows x 128 columns per workgroup of four waves; stages of 32 output columns through the three-stage
// ring of k_project_phi (dy rows as its x) with W's rows as k_weight_grad_partial stages them: contracted over
// their row index, read by the transposing read.  The weights are read where they are, no stack of them is
// formed.  Bound like k_project_phi, by the step (barrier, operand reads, 16 to 32 products) where a tile has few, by the
// direct loads (12 TB/s over the chip with 128 x 128 tiles) where 256 of them fill it; KG groups as there.
// Measured, us, one group -> as chosen (the library's products over a stacked weight, another 4.6 to 7.8 to form):
// 8192 rows, 512 -> 512 11.8 -> 10.6 (12.3), three of them 25.1 -> 19.9 (21.4); 2048 rows, three of 768 25.3 -> 16.8; 512
// rows, three of 1024 31.3 -> 19.4 (16.5); 16384 rows, two of 512 28.1 (24.2; 38 as two products); 1024 -> 1024, three 69.3 (57.3).
// grid = 8 * ceil(tiles / 8), tiles numbered row tile by row tile; each XCD gets a contiguous range.
template <int BM_, int KG>
__device__ __forceinline__ void input_grad_tile(unsigned char* smem_raw, int tile, const InputGradArgs& ga,
                                                half_t* __restrict__ dx, int R, int Eo, int Ei, int np, int64_t ld) {
    using Cfg = InputGradCfg<BM_, KG>;
    using Sum = typename Cfg::Sum;
    constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, STAGES = Cfg::kStages, NR = Cfg::NR, NC = Cfg::NC;
    const int tid = threadIdx.x, lane = tid & 63;
    const int kg = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
    const int wv = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);      // wave inside its group
    half_t* const smem = reinterpret_cast<half_t*>(smem_raw);
    constexpr int kRing = KG * Cfg::kStageHalves, SK = BK * KG;      // halves of a stage, its columns of dy
    using Rows = StageRows<KG>;
    const int i = lane & 15, G = lane >> 4;
    const int wr = wv >> 1, wc = wv & 1;

    const int tiles_c = Ei / BN;
    const int row0 = (tile / tiles_c) * BM, c0 = (tile % tiles_c) * BN;

    unsigned yoff[Cfg::YI], woff[Cfg::WI];
#pragma unroll
    for (int it = 0; it < Cfg::YI; ++it) {
        const int r = ((kg * 4 + wv) * Cfg::YI + it) * (64 / Rows::kSlots) + lane / Rows::kSlots;
        yoff[it] = (unsigned)min(r, R - 1 - row0) * (unsigned)(ld * 2) + Rows::slot(r, lane % Rows::kSlots) * 16;
    }
#pragma unroll
    for (int it = 0; it < Cfg::WI; ++it) {
        const int r = (wv * Cfg::WI + it) * 4 + (lane >> 4);
        woff[it] = (unsigned)r * (unsigned)(Ei * 2) + (((lane & 15) ^ (((r & 3) | ((r >> 1) & 4)) * 2)) * 16);
    }
    const int per_p = Eo / SK, nk = np * per_p;      // SK divides Eo
    auto load_stage = [&](int kk, int buf) {
        const int p = kk >= 2 * per_p ? 2 : (kk >= per_p ? 1 : 0), ko = (kk - p * per_p) * SK;
        const half_t* yb = pick3(ga.dy, p) + (int64_t)row0 * ld + ko;
        const half_t* wb = pick3(ga.w, p) + (int64_t)(ko + BK * kg) * Ei + c0;
        half_t* st = smem + buf * kRing;
#pragma unroll
        for (int it = 0; it < Cfg::YI; ++it) dma16_opaque(yb, yoff[it], st + ((kg * 4 + wv) * Cfg::YI + it) * 512);
#pragma unroll
        for (int it = 0; it < Cfg::WI; ++it) dma16_opaque(wb, woff[it], st + BM * SK + ((kg * 4 + wv) * Cfg::WI + it) * 512);
    };

    f4 acc[NR][NC];      // dx^T tiles (m = column, n = row)
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[a][c] = f4_zero();
    const half_t* const yop = smem + (wr * Cfg::RW + i) * SK + Rows::slot(i, 4 * kg + G) * 8;

#pragma unroll
    for (int k = 0; k < STAGES - 1; ++k) load_stage(min(k, nk - 1), k);
    int buf = 0;
    for (int kk = 0; kk < nk; ++kk) {
        stage_barrier<(STAGES - 2) * (Cfg::YI + Cfg::WI)>();
        load_stage(min(kk + STAGES - 1, nk - 1), buf == 0 ? STAGES - 1 : buf - 1);
        const half_t* ys = yop + buf * kRing;
        const half_t* Ws = smem + buf * kRing + BM * SK + kg * BK * BN;
        h8 wa[NC], yb[NR];
#pragma unroll
        for (int c = 0; c < NC; ++c) wa[c] = col8_rot<BN>(Ws, NC * wc + c, lane);
#pragma unroll
        for (int a = 0; a < NR; ++a) yb[a] = *reinterpret_cast<const h8*>(ys + a * 16 * SK);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int a = 0; a < NR; ++a)
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[a][c] = mfma32(wa[c], yb[a], acc[a][c]);
        __builtin_amdgcn_s_setprio(0);
        buf = buf == STAGES - 1 ? 0 : buf + 1;
    }
    // the last re-requested stages are still on their way into this workgroup's LDS: they land before it ends
    stage_barrier<0>();
    f4 own[Sum::kOwn][NC];
    Sum::run(acc, own, smem_raw, kg, tid & (kThreads - 1));
    if (kg >= Sum::kFin) return;
#pragma unroll
    for (int a = 0; a < Sum::kOwn; ++a) {
        const int r = row0 + wr * Cfg::RW + 16 * (Sum::kFin * a + kg) + i;
        if (r < R) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
                *reinterpret_cast<h4*>(dx + (int64_t)r * Ei + c0 + 64 * wc + 16 * c + 4 * G) = to_h4(own[a][c]);
        }
    }
}

template <int BM_, int KG>
__global__ __launch_bounds__(kThreads * KG, 2) void k_input_grad(InputGradArgs ga, half_t* __restrict__ dx, int R, int Eo,
                                                                 int Ei, int np, int64_t ld, int tiles) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int tile = xcd_range(blockIdx.x, tiles);
    if (tile < tiles) input_grad_tile<BM_, KG>(smem_raw, tile, ga, dx, R, Eo, Ei, np, ld);
}

// Input gradient and weight-gradient partials of the same layers in one launch.  Either alone leaves the CUs half empty at
// its start and its end, and both read dy: an XCD's workgroups take the same range of rows, a tile of dx and one of dW in
// turn.  Bound by the operands' way from L2 to LDS, as both are.  Measured with the reduction: 8192 rows, 512 -> 512
// 33.5 us as two launches, 24.0 here; three of 512 47.2 and 40.0; 512 rows, 512 -> 512 16.4 and 10.1.
// grid = 8 * (ceil(tiles / 8) + ceil(work / 8))
template <int BM_, int KG>
__global__ __launch_bounds__(kThreads * KG, 2) void k_linear_grads(
    InputGradArgs ga, half_t* __restrict__ dx, const half_t* __restrict__ x, WeightGradArgs wa, float* __restrict__ part,
    float* __restrict__ bpart, int R, int Eo, int Ei, int np, int64_t ld, int tiles, int work, int rows_per_split) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int xcd = blockIdx.x % kXcds, l = blockIdx.x / kXcds;
    const int nt = (tiles + kXcds - 1) / kXcds, nw = (work + kXcds - 1) / kXcds;      // per XCD
    const int both = 2 * min(nt, nw);
    const bool is_dx = l < both ? (l & 1) == 0 : nt > nw;
    const int at = l < both ? l >> 1 : l - both / 2;
    if (is_dx) {
        const int tile = xcd * nt + at;
        if (at < nt && tile < tiles) input_grad_tile<BM_, KG>(smem_raw, tile, ga, dx, R, Eo, Ei, np, ld);
    } else {
        const int idx = xcd * nw + at;
        if (at < nw && idx < work) weight_grad_tile<false, KG>(smem_raw, idx, x, wa, ld, part, bpart, R, Eo, Ei, np, rows_per_split);
    }
}

// The feature map's dW' where its shares are summed beside those of the layers: `blocks` workgroups come first, one per
// 256 elements (0: none).
struct FeatureSum {
    const float* part;
    half_t* dw;
    int blocks, shares;
};

// dW_p = sum of the partials (4 elements per thread), then db_p; grid = fs.blocks + ceil(np * (Eo * Ei + Eo) / 4 / 256).
// What bounds it is one round trip to memory behind a launch, so the feature map's shares are summed beside the layers': the
// reductions of a layer in training (8192 rows, three layers and one of 512, 64 features) 13.8 us in three launches, 10.4 in
// two; those of an encoder-decoder layer 27.5 in five, 17.5 in three.
__global__ __launch_bounds__(kThreads) void k_weight_grad_reduce(
    const float* __restrict__ part, const float* __restrict__ bpart, WeightGradArgs wa, int Eo, int Ei, int np,
    int nsplit, FeatureSum fs) {
    if ((int)blockIdx.x < fs.blocks) {
        feature_map_dw_sum(blockIdx.x, fs.part, nullptr, fs.dw, fs.shares, (int64_t)fs.blocks * 256);
        return;
    }
    const int64_t per_w = (int64_t)Eo * Ei / 4, per_b = Eo / 4;
    const int64_t t = (int64_t)((int)blockIdx.x - fs.blocks) * kThreads + threadIdx.x;
    if (t < per_w * np) {
        const int p = (int)(t / per_w);
        const int64_t q = t % per_w;
        f4 sum = f4_zero();
        for (int s = 0; s < nsplit; ++s) {
            const f4 v = *reinterpret_cast<const f4*>(part + ((int64_t)(s * np + p) * per_w + q) * 4);
            sum[0] += v[0]; sum[1] += v[1]; sum[2] += v[2]; sum[3] += v[3];
        }
        *reinterpret_cast<h4*>(pick3(wa.dw, p) + q * 4) = to_h4(sum);
    } else if (t < (per_w + per_b) * np) {
        const int64_t u = t - per_w * np;
        const int p = (int)(u / per_b);
        const int64_t q = u % per_b;
        half_t* db = pick3(wa.db, p);
        if (!db) return;
        f4 sum = f4_zero();
        for (int s = 0; s < nsplit; ++s) {
            const f4 v = *reinterpret_cast<const f4*>(bpart + ((int64_t)(s * np + p) * per_b + q) * 4);
            sum[0] += v[0]; sum[1] += v[1]; sum[2] += v[2]; sum[3] += v[3];
        }
        *reinterpret_cast<h4*>(db + q * 4) = to_h4(sum);
    }
}

}  // namespace rfa
