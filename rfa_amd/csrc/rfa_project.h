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

template <int D, int DH, int BM_>
struct ProjectCfg {
    static_assert(D % 32 == 0 && (DH == 64 || DH == 128), "D multiple of 32, DH 64 or 128");
    static constexpr int BM = BM_;                 // rows of x per workgroup
    static constexpr int BN = 128;                 // output columns: one head of 128 or two of 64
    static constexpr int BK = 32;                  // contraction step: one MFMA deep
    static constexpr int kStages = 3;              // 4 to 6 measured no faster at any size
    static constexpr int PPT = BN / DH;            // heads per tile
    static constexpr int WR = 4 / PPT;             // waves along the rows; a wave owns whole heads
    static constexpr int RW = BM / WR;             // rows of a wave
    static constexpr int NR = RW / 16, NC = DH / 16;
    static constexpr int XI = BM / 64, WI = BN / 64;    // 1 KiB pieces of a stage per wave: x, W
    static constexpr int kStageHalves = (BM + BN) * BK;
    static constexpr int LDW = DH + lds_pad(DH);   // rows of w'
    static constexpr size_t kLoopLds = (size_t)kStages * kStageHalves * 2;
    static constexpr size_t kEpiLds = (size_t)PPT * D * LDW * 2;
    static constexpr size_t kLds = kLoopLds > kEpiLds ? kLoopLds : kEpiLds;
    static_assert(kLds <= 80 * 1024, "two workgroups per CU");
};

// 64 lanes x 16 bytes, global -> LDS without registers: lane l's bytes land at lds + 16 l
__device__ __forceinline__ void dma16(const char* g, half_t* lds) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                     (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
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
//
// Measured (us; q, k, v projections with phi(q), phi(k); before: rows of x in registers for E <= 512,
// a register-staged two-buffer loop otherwise):
//   8192 rows, E 512, 8 heads of 64, D 64       42.1 -> 28.2      8192, 1024, 8 of 128, D 128   112 -> 83
//   32768, 1024, 16 of 64, D 64                  964 -> 304 (678 TFLOP/s)      512, 512   12.4 -> 9.6
//
// LDS stage: x tile [BM][32], then W tile [128][32] halves, no padding (a direct load writes 1 KiB
// in lane order); the four 16-byte pieces of row r are stored rotated, piece c at c ^ ((r >> 2) & 3),
// which spreads a wave's operand read (16 rows x 16 bytes per 16 lanes) over all banks.  The rows of
// W sit in pair order (pair_pos), so that accumulator tiles 2p, 2p + 1 give lane (i, G) the 8
// consecutive columns 32 p + 8 G of row i: y goes out in 16-byte pieces, is the operand of the
// feature product as it stands, and phi goes out the same way; nothing passes through LDS again.
//
// Tiles are numbered row tile by row tile; each XCD gets a contiguous range of numbers, so that
// the tiles that share rows of x meet in its L2.   grid = 8 * ceil(tiles / 8).
template <int D, int DH, int BM_>
__global__ __launch_bounds__(kThreads, 2) void k_project_phi(
    const half_t* __restrict__ x, ProjectArgs pa, const half_t* __restrict__ wf, int R, int E, int H, int np,
    int tiles_c, int tiles, float scale) {
    using Cfg = ProjectCfg<D, DH, BM_>;
    constexpr int BM = Cfg::BM, BK = Cfg::BK, STAGES = Cfg::kStages, NR = Cfg::NR, NC = Cfg::NC, LDW = Cfg::LDW;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    half_t* smem = reinterpret_cast<half_t*>(smem_raw);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, G = lane >> 4;

    const int per_xcd = (tiles + kXcds - 1) / kXcds;
    const int tile = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (tile >= tiles) return;                         // whole workgroup: padding of the grid
    const int row0 = (tile / tiles_c) * BM;
    const int hp0 = (tile % tiles_c) * Cfg::PPT;       // (projection, head) pairs: hp -> hp / H, hp % H
    const int pairs = H * np;

    // ---- direct-load addresses: wave-uniform base + 32-bit lane offset, set up once
    const char* xbase = reinterpret_cast<const char*>(x + (int64_t)row0 * E);
    unsigned xoff[Cfg::XI], woff[Cfg::WI];
#pragma unroll
    for (int it = 0; it < Cfg::XI; ++it) {
        const int r = (wv * Cfg::XI + it) * 16 + (lane >> 2);
        xoff[it] = (unsigned)min(r, R - 1 - row0) * (unsigned)(E * 2) + (((lane & 3) ^ ((r >> 2) & 3)) * 16);
    }
    // W rows 32 wv .. of the tile: 32-row groups never straddle a head
    const int hp_ld = min(hp0 + 32 * wv / DH, pairs - 1);
    const char* wbase = reinterpret_cast<const char*>(
        pick3(pa.w, hp_ld / H) + ((int64_t)(hp_ld % H) * DH + (32 * wv) % DH) * E);
#pragma unroll
    for (int it = 0; it < Cfg::WI; ++it) {
        const int r = it * 16 + (lane >> 2);           // LDS row within the group; it holds column pair_inv
        const int c = (r & 3) | ((r & 16) >> 2) | ((r & 12) << 1);
        woff[it] = (unsigned)c * (unsigned)(E * 2) + (((lane & 3) ^ ((r >> 2) & 3)) * 16);
    }
    half_t* const xdst = smem + wv * Cfg::XI * 512;
    half_t* const wdst = smem + BM * BK + wv * Cfg::WI * 512;
    auto load_stage = [&](int kk, int buf) {
        const char* xb = xbase + (int64_t)kk * (BK * 2);
        const char* wb = wbase + (int64_t)kk * (BK * 2);
#pragma unroll
        for (int it = 0; it < Cfg::XI; ++it) dma16(xb + xoff[it], xdst + buf * Cfg::kStageHalves + it * 512);
#pragma unroll
        for (int it = 0; it < Cfg::WI; ++it) dma16(wb + woff[it], wdst + buf * Cfg::kStageHalves + it * 512);
    };
    constexpr int kPerStage = Cfg::XI + Cfg::WI;

    // y^T tiles (m = output column in pair order, n = row) of this wave's rows and head
    const int wr = wv / Cfg::PPT, wc = wv % Cfg::PPT;
    f4 acc[NR][NC];
#pragma unroll
    for (int a = 0; a < NR; ++a)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[a][c] = f4_zero();

    // operand rows of this lane inside a stage: row (16 t + i), piece G
    const int piece = (G ^ ((i >> 2) & 3)) * 8;
    const half_t* const xop = smem + (wr * Cfg::RW + i) * BK + piece;
    const half_t* const wop = smem + BM * BK + (wc * DH + i) * BK + piece;

    const int nk = E / BK;
#pragma unroll
    for (int k = 0; k < STAGES - 1; ++k) load_stage(min(k, nk - 1), k);
    int buf = 0;
    for (int kk = 0; kk < nk; ++kk) {
        // stage kk has landed (the STAGES - 2 after it may still be on their way), stage kk - 1 is free
        stage_barrier<(STAGES - 2) * kPerStage>();
        // the last steps re-request the last stage's columns into buffers nobody reads again
        load_stage(min(kk + STAGES - 1, nk - 1), buf == 0 ? STAGES - 1 : buf - 1);
        const half_t* xs = xop + buf * Cfg::kStageHalves;
        const half_t* wsm = wop + buf * Cfg::kStageHalves;
        h8 wa[NC], xb[NR];
#pragma unroll
        for (int c = 0; c < NC; ++c) wa[c] = *reinterpret_cast<const h8*>(wsm + c * 16 * BK);
#pragma unroll
        for (int a = 0; a < NR; ++a) xb[a] = *reinterpret_cast<const h8*>(xs + a * 16 * BK);
        __builtin_amdgcn_s_setprio(1);      // the other workgroup's loads and epilogue give way: 2 % at full size
#pragma unroll
        for (int a = 0; a < NR; ++a)
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[a][c] = mfma32(wa[c], xb[a], acc[a][c]);
        __builtin_amdgcn_s_setprio(0);
        buf = buf == STAGES - 1 ? 0 : buf + 1;
    }

    // ---- epilogue: the ring becomes the place of w' (rows in pair order)
    stage_barrier<0>();
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
                load_w_pair_order<D, DH, kThreads>(smem + u * D * LDW, wf + (int64_t)(hu % H) * D * DH, tid);
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
    __syncthreads();
    if (!live) return;
    const half_t* const Wfs = smem + wc * D * LDW;
#pragma unroll
    for (int a = 0; a < NR; ++a) {
        const int r = row0 + wr * Cfg::RW + 16 * a + i;
        const int64_t at = (int64_t)r * H + h;
        h8 op[NC / 2];       // the rounded row pieces: y as stored, and the operand of the feature product
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < NC / 2; ++c) {
#pragma unroll
            for (int e = 0; e < 8; ++e) op[c][e] = (half_t)(acc[a][2 * c + e / 4][e % 4] + (float)bv[c][e]);
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
    static constexpr int TO = 128, TI = 128, C = 64;       // tile of dW, rows per step
    static constexpr int LD = 128 + lds_pad(128);
    static constexpr int kTile = C * LD;                   // halves
    static constexpr size_t kLds = (size_t)2 * 2 * kTile * 2;
    static constexpr int kPieces = C * 128 / 8 / kThreads; // 16-byte pieces per thread and tile
};

// rows [r0, r0 + 64) x columns [c0, c0 + 128) of a [R, E] matrix -> registers; rows at or past
// r_end are read from row r_end - 1 (always a valid row) and zeroed on the way to LDS
__device__ __forceinline__ void wgrad_g2r(uint4 (&v)[WeightGradCfg::kPieces], const half_t* __restrict__ src, int E,
                                          int r0, int r_end, int c0, int tid) {
#pragma unroll
    for (int it = 0; it < WeightGradCfg::kPieces; ++it) {
        const int pc = tid + kThreads * it;
        const int r = min(r0 + pc / 16, r_end - 1);
        v[it] = *reinterpret_cast<const uint4*>(src + (int64_t)r * E + c0 + (pc % 16) * 8);
    }
}

__device__ __forceinline__ void wgrad_r2s(const uint4 (&v)[WeightGradCfg::kPieces], half_t* Xs, int r0, int r_end,
                                          int tid) {
#pragma unroll
    for (int it = 0; it < WeightGradCfg::kPieces; ++it) {
        const int pc = tid + kThreads * it;
        const bool keep = r0 + pc / 16 < r_end;
        uint4 x = v[it];
        x.x = keep ? x.x : 0u; x.y = keep ? x.y : 0u; x.z = keep ? x.z : 0u; x.w = keep ? x.w : 0u;
        *reinterpret_cast<uint4*>(Xs + (pc / 16) * WeightGradCfg::LD + (pc % 16) * 8) = x;
    }
}

// grid = 8 * ceil(nsplit / 8) * np * (Eo / 128) * (Ei / 128): the workgroups of one split (which
// share its rows of x and dy) are dealt to one XCD.  rows_per_split is a multiple of 64.
__global__ __launch_bounds__(kThreads) void k_weight_grad_partial(
    const half_t* __restrict__ x, WeightGradArgs wa, float* __restrict__ part, float* __restrict__ bpart, int R,
    int Eo, int Ei, int np, int nsplit, int rows_per_split) {
    using Cfg = WeightGradCfg;
    constexpr int LD = Cfg::LD, C = Cfg::C;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    half_t* smem = reinterpret_cast<half_t*>(smem_raw);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, G = lane >> 4;
    const int wo = wv >> 1, wi = wv & 1;                  // wave -> 64 x 64 quadrant of the tile

    const int tiles_i = Ei / Cfg::TI, tiles_o = Eo / Cfg::TO;
    const int per_split = np * tiles_o * tiles_i;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int s = xcd + 8 * (slot / per_split);
    if (s >= nsplit) return;
    int idx = slot % per_split;
    const int ti = idx % tiles_i; idx /= tiles_i;
    const int to = idx % tiles_o;
    const int p = idx / tiles_o;
    const int r_begin = s * rows_per_split, r_end = min(r_begin + rows_per_split, R);
    const int o0 = to * Cfg::TO, c0 = ti * Cfg::TI;
    const half_t* __restrict__ dy = pick3(wa.dy, p);
    const bool with_bias = ti == 0 && wi == 0 && pick3(wa.db, p) != nullptr;   // wave-uniform

    f4 acc[4][4];        // (m = o, n = c) tiles of this wave's quadrant
    f4 accb[4];          // column sums of dy: every column n holds the same sum
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        accb[a] = f4_zero();
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = f4_zero();
    }
    h8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (half_t)1.0f;

    if (r_begin < r_end) {
        uint4 yr[Cfg::kPieces], xr[Cfg::kPieces];
        wgrad_g2r(yr, dy, Eo, r_begin, r_end, o0, tid);
        wgrad_g2r(xr, x, Ei, r_begin, r_end, c0, tid);
        wgrad_r2s(yr, smem, r_begin, r_end, tid);
        wgrad_r2s(xr, smem + Cfg::kTile, r_begin, r_end, tid);
        __syncthreads();
        int buf = 0;
        for (int r0 = r_begin; r0 < r_end; r0 += C) {
            // branch-free prefetch of the next step (the last one re-reads valid rows and zeroes them)
            wgrad_g2r(yr, dy, Eo, r0 + C, r_end, o0, tid);
            wgrad_g2r(xr, x, Ei, r0 + C, r_end, c0, tid);
            const half_t* Ys = smem + buf * 2 * Cfg::kTile;
            const half_t* Xs = Ys + Cfg::kTile;
#pragma unroll
            for (int rs = 0; rs < C / 32; ++rs) {
                h8 xa[4];
#pragma unroll
                for (int b = 0; b < 4; ++b) xa[b] = col8(Xs, LD, 32 * rs, 64 * wi + 16 * b, lane);
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const h8 ya = col8(Ys, LD, 32 * rs, 64 * wo + 16 * a, lane);
#pragma unroll
                    for (int b = 0; b < 4; ++b) acc[a][b] = mfma32(ya, xa[b], acc[a][b]);
                    if (with_bias) accb[a] = mfma32(ya, ones, accb[a]);
                }
            }
            buf ^= 1;
            wgrad_r2s(yr, smem + buf * 2 * Cfg::kTile, r0 + C, r_end, tid);
            wgrad_r2s(xr, smem + buf * 2 * Cfg::kTile + Cfg::kTile, r0 + C, r_end, tid);
            __syncthreads();
        }
    }
    float* po = part + ((int64_t)(s * np + p) * Eo + o0 + 64 * wo) * Ei + c0 + 64 * wi;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) po[(int64_t)(16 * a + 4 * G + e) * Ei + 16 * b + i] = acc[a][b][e];
    if (with_bias && i == 0) {
        float* pb = bpart + (int64_t)(s * np + p) * Eo + o0 + 64 * wo;
#pragma unroll
        for (int a = 0; a < 4; ++a) *reinterpret_cast<f4*>(pb + 16 * a + 4 * G) = accb[a];
    }
}

// dW_p = sum of the partials (4 elements per thread), then db_p; grid = ceil(np * (Eo * Ei + Eo) / 4 / 256)
__global__ __launch_bounds__(kThreads) void k_weight_grad_reduce(
    const float* __restrict__ part, const float* __restrict__ bpart, WeightGradArgs wa, int Eo, int Ei, int np,
    int nsplit) {
    const int64_t per_w = (int64_t)Eo * Ei / 4, per_b = Eo / 4;
    const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x;
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
