// Fused random-feature map  phi(x) = scale * [sin(W x^), cos(W x^)],  x^ = x / (||x|| + 1e-3)
// and its backward, for gfx950.
//
// Replaces the chain of ATen kernels in random_project / _normalize
// (random_feature_attention/utils.py:100-120: norm, add, div, einsum, sin, cos,
// cat, mul) by one kernel per direction.  The projection W' of one head stays
// resident in LDS while a workgroup streams rows of x through the MFMA.
//
// Every wave walks its own groups of 16 rows; rows move between registers and global memory in the lanes'
// own operand positions.  The forward, and the backward where dW'[D][DH] of a head fits a wave's accumulators
// (D * DH <= 4096), have no workgroup barrier in the row loop; else the backward's eight waves share dW'
// between them and meet twice per 128 rows.
//
// Layouts:  x   [R, H, DH] fp16   (R = seq_len * bsz rows, row-major)
//           w   [H, D, DH] fp16   (already sigma * W / tau, utils.py:90-97)
//           phi [R, H, 2D] fp16   (sin block in columns [0, D), cos block in [D, 2D))
#pragma once
#include "rfa_common.h"

namespace rfa {

template <int D, int DH>
struct FeatureCfg {
    static_assert(D % 32 == 0 && DH % 64 == 0, "D multiple of 32, DH multiple of 64");
    static constexpr int LDW = DH + lds_pad(DH);
    static constexpr size_t kFwdLds = (size_t)(D * LDW) * 2;                                     // W' only
};

// Orders this wave's earlier LDS writes before its later LDS reads of other lanes' data.  One
// wave executes its LDS instructions in order, so only the compiler has to be stopped from
// moving them; a memory fence here would also wait for every global load and store in flight
// (the next block's prefetch, the previous rows' stores).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

// ---- streaming kernels: waves that never wait for each other ---------------------------------
// A wave owns groups of 16 rows of one head and walks them with a stride; W' sits in LDS, read
// only.  Nothing a wave writes is read by another wave, so the row loop has no workgroup barrier.
//
// "Pair order": MFMA tile t of 16 features (or of 16 input columns) is made of the indices
//     32 (t / 2) + 8 G + 4 (t % 2) + e        at accumulator position m = 4 G + e,
// so that the accumulators of tiles 2p and 2p+1 together give lane (i, G) the 8 consecutive
// indices 32 p + 8 G .. + 7 of row i: 16 bytes that go to (and come from) global memory
// directly, without a pass through LDS to re-form rows.  pair_pos(f) (rfa_common.h) is the row of
// the operand matrix that holds index f.
constexpr int kFeatureWaves = 8;
constexpr int kFeatureThreads = 64 * kFeatureWaves;


// W' of one head -> LDS with its rows (features) in pair order
template <int D, int DH, int NT = kFeatureThreads>
__device__ __forceinline__ void load_w_pair_order(half_t* Ws, const half_t* __restrict__ wh, int tid) {
    constexpr int LDW = FeatureCfg<D, DH>::LDW;
    constexpr int PPR = DH / 8;
    for (int p = tid; p < D * PPR; p += NT) {
        const int r = p / PPR, c8 = p % PPR;
        *reinterpret_cast<uint4*>(Ws + pair_pos(r) * LDW + c8 * 8) = *reinterpret_cast<const uint4*>(wh + r * DH + c8 * 8);
    }
}

// Operand of y = du W' from that copy of W': features f0 + 8 G + e, e = 0..7 (rows 4 G + e % 4 and 16 further, as
// pair order has them), input columns of tile t in pair order.  By transposing reads whose lanes take every second
// piece of 4 columns: W' needs no transposed copy.
template <int LDW>
__device__ __forceinline__ h8 w_col_pair8(const half_t* Ws, int f0, int t, int lane) {
    const int s = lane & 15, G = lane >> 4;
    const half_t* p = Ws + (f0 + 4 * G + (s >> 2)) * LDW + 32 * (t / 2) + 4 * (t % 2) + 8 * (s & 3);
    const h4 a = tr_read4(p), b = tr_read4(p + 16 * LDW);
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// grid = (nblk, H, 1 or 2); wave w of workgroup b takes the row groups 8 b + w, + 8 nblk, ...
// gridDim.z = 2 maps two tensors through the same W' in one launch (q and k of a module):
// workgroups with blockIdx.z = 1 take x1 / phi1.
template <int D, int DH>
__global__ __launch_bounds__(kFeatureThreads) void k_feature_map_fwd(
    const half_t* __restrict__ x0, const half_t* __restrict__ w, half_t* __restrict__ phi0,
    const half_t* __restrict__ x1, half_t* __restrict__ phi1, int R, int H, float scale) {
    const bool second = blockIdx.z != 0;
    const half_t* __restrict__ x = second ? x1 : x0;
    half_t* __restrict__ phi = second ? phi1 : phi0;
    constexpr int LDW = FeatureCfg<D, DH>::LDW;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    half_t* Ws = reinterpret_cast<half_t*>(smem_raw);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, G = lane >> 4;
    const int h = blockIdx.y;

    load_w_pair_order<D, DH>(Ws, w + (int64_t)h * D * DH, tid);

    const int ngrp = (R + 15) / 16, gstride = gridDim.x * kFeatureWaves;
    int grp = blockIdx.x * kFeatureWaves + wv;
    // Two sets of row registers: the loads of the next group are issued into the set the
    // current group does not use, so no set is ever copied (a third set, two groups in flight,
    // measured no faster).  Rows past R read the last row (no branch around the loads) and are
    // not stored.
    struct Rows { h8 x[DH / 32]; };
    auto issue_loads = [&](Rows& t, int g) {
        const half_t* px = x + ((int64_t)min(g * 16 + i, R - 1) * H + h) * DH + 8 * G;
#pragma unroll
        for (int cs = 0; cs < DH / 32; ++cs) t.x[cs] = *reinterpret_cast<const h8*>(px + cs * 32);
    };
    auto process = [&](const Rows& t, int g) {
        const int r = g * 16 + i;
        float ss = 0.f;
#pragma unroll
        for (int cs = 0; cs < DH / 32; ++cs) ss += dot_h8(__builtin_bit_cast(uint4, t.x[cs]), __builtin_bit_cast(uint4, t.x[cs]));
        ss = sum_over_groups(ss);
        const float inv_turns = rcp_nr(__builtin_amdgcn_sqrtf(ss) + 1e-3f) * 0.15915494309189535f;
        half_t* po = phi + ((int64_t)r * H + h) * (2 * D) + 8 * G;
#pragma unroll
        for (int p = 0; p < D / 32; ++p) {
            f4 acc[2] = {f4_zero(), f4_zero()};   // u^T tiles 2p, 2p+1 (m = feature, n = row)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int cs = 0; cs < DH / 32; ++cs)
                    acc[q] = mfma32(row8(Ws, LDW, 32 * p + 16 * q + i, cs * 32, G), t.x[cs], acc[q]);
            h8 sv, cv;
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float s_, c_;
                    sincos_turns(acc[q][e] * inv_turns, s_, c_);
                    sv[4 * q + e] = (half_t)(scale * s_);
                    cv[4 * q + e] = (half_t)(scale * c_);
                }
            if (r < R) {
                *reinterpret_cast<h8*>(po + 32 * p) = sv;
                *reinterpret_cast<h8*>(po + D + 32 * p) = cv;
            }
        }
    };
    Rows ra, rb;
    if (grp < ngrp) issue_loads(ra, grp);
    __syncthreads();   // W' in place
    while (grp < ngrp) {
        if (grp + gstride < ngrp) issue_loads(rb, grp + gstride);
        process(ra, grp);
        if ((grp += gstride) >= ngrp) break;
        if (grp + gstride < ngrp) issue_loads(ra, grp + gstride);
        process(rb, grp);
        grp += gstride;
    }
}

// LDS of the backward: W' (rows in pair order), 16 rows of x and of du of every wave for the
// transposing reads of the dW product, and, where each wave has a dW' of its own, after the row loop the same
// bytes again as the area through which the eight waves exchange them (one copy of dW'[D][DH] per wave).
#ifndef RFA_FEATURE_BWD_WAVES
#define RFA_FEATURE_BWD_WAVES 8
#endif
constexpr int kFeatureBwdWaves = RFA_FEATURE_BWD_WAVES;
constexpr int kFeatureBwdThreads = 64 * kFeatureBwdWaves;

template <int D, int DH>
struct FeatureBwdCfg {
    static constexpr int LDW = DH + lds_pad(DH);
    static constexpr bool kFits = D * DH <= 4096;     // the whole dW' of a head in the accumulators of every wave: 4 registers per tile
    // a row stride of 32 bytes mod 256 spreads the 8-byte pieces of a transposing read of 16 rows over all banks, lds_pad
    // those of one of 32
    static constexpr int LDX = DH + (kFits ? 16 : lds_pad(DH)), LDU = D + (kFits ? 16 : lds_pad(D));
    static constexpr int kTiles = (DH / 16) * (D / 16);
    static constexpr size_t kLoop = (size_t)(D * LDW + kFeatureBwdWaves * 16 * (LDX + LDU)) * 2;
    static constexpr size_t kReduce = kFits ? (size_t)kFeatureBwdWaves * D * DH * 4 : 0;
    static constexpr size_t kLds = kLoop > kReduce ? kLoop : kReduce;
    // else the waves deal its tiles out: kWA of them along the input columns (one 16-wide tile each), the rest along the features
    static constexpr int kWA = DH / 16 < kFeatureBwdWaves ? DH / 16 : kFeatureBwdWaves, kWB = kFeatureBwdWaves / kWA;
    static constexpr int kTA = kFits ? DH / 16 : 1, kTB = kFits ? D / 16 : D / 16 / kWB;      // accumulator tiles of a wave
    static_assert(kFits || (DH / 16 == kWA && (D / 16) % kWB == 0), "tiles of dW' over the waves");
};

__device__ __forceinline__ f4 mfma16(h4 a, h4 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0); }

// Backward of the feature map.  grid = (nblk, H, 1 or 2) like the forward; wave w of
// workgroup b takes the row groups 8 b + w, + 8 nblk, ...
// gridDim.z = 2 differentiates two tensors that went through the same W' in one launch (phi(q) and
// phi(k) of a module): workgroups with blockIdx.z = 1 take x1 / gphi1 / dx1 and the partial
// sums nblk .. 2 nblk - 1, so that the reduction over 2 nblk shares yields the sum of both dW'.
// The rows of dx lie dx_rs halves apart (H * DH for a tensor of its own).
// Per group of 16 rows, with n = ||x||, inv = 1 / (n + 1e-3), u = W' x inv:
//     du  = scale (cos u * g_sin - sin u * g_cos) inv          accumulators of u, in registers
//     y   = du W'                                               du is the MFMA operand as it stands
//     dx  = y - x (x . y) / (n (n + 1e-3))   (0 where n = 0)    16 bytes per lane, stored directly
//     dW' += du^T x
// x and grad_phi arrive in the lane's own operand / accumulator positions (pair order), so no
// row is re-formed in LDS.  dW' where D * DH <= 4096: over the wave's own 16 rows (k = 16 MFMA, operands by transposing
// LDS reads), no wave reads what another wrote, no workgroup barrier in the row loop; at the end the eight waves add
// their dW' through LDS (one exchange, every wave sums and stores an eighth of the tiles).  Else (kFits false): the eight
// waves' 128 rows of x and du meet in LDS, each wave contracts them for its own eighth of the tiles (k = 32), behind
// one barrier and before another, with y and dx of its rows between them.  Either way the workgroup leaves one partial sum,
// dw_part[(z nblk + b)][h]; k_feature_map_dw_reduce sums the shares.
// Measured where the waves share dW' (before: four waves, blocks of 64 rows staged through LDS both ways, three
// barriers each, one workgroup to a CU), us, pairs of 8192 rows, 8 heads: D 128, d 128 53.5 -> 35.5 (with a third block to
// copy, then a launch of its own, 59.0 -> 42.0); 128, 64 28.1 -> 23.5; 64, 128 25.2 -> 23.6.  A transposed copy of W' in
// LDS for y: 36.2, and 1.5 more at a few hundred rows; D 64, d 64 17.1 with such a copy, 16.0 without.
template <int D, int DH>
__global__ __launch_bounds__(kFeatureBwdThreads) void k_feature_map_bwd(
    const half_t* __restrict__ x0, const half_t* __restrict__ w, const half_t* __restrict__ gphi0,
    half_t* __restrict__ dx0, const half_t* __restrict__ x1, const half_t* __restrict__ gphi1,
    half_t* __restrict__ dx1, float* __restrict__ dw_part, int R, int H, float scale, int64_t dx_rs,
    const half_t* __restrict__ copy_src, half_t* __restrict__ copy_dst) {
    const bool second = blockIdx.z != 0;
    const half_t* __restrict__ x = second ? x1 : x0;
    const half_t* __restrict__ gphi = second ? gphi1 : gphi0;
    half_t* __restrict__ dx = second ? dx1 : dx0;
    using Cfg = FeatureBwdCfg<D, DH>;
    constexpr bool kShared = !Cfg::kFits;
    constexpr int LDW = Cfg::LDW, LDX = Cfg::LDX, LDU = Cfg::LDU;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    half_t* Ws = reinterpret_cast<half_t*>(smem_raw);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    // this wave's 16 rows of x and of du: all rows of x, then all rows of du
    half_t* const Xall = Ws + D * LDW;
    half_t* const Uall = Xall + 16 * kFeatureBwdWaves * LDX;
    half_t* const Xs = Xall + 16 * wv * LDX;
    half_t* const Us = Uall + 16 * wv * LDU;
    const int i = lane & 15, G = lane >> 4;
    const int h = blockIdx.y;
    const half_t* wh = w + (int64_t)h * D * DH;

    load_w_pair_order<D, DH, kFeatureBwdThreads>(Ws, wh, tid);
    if (copy_src) {
        // rows of copy_src [R, H, DH] -> rows of copy_dst, dx_rs halves apart: the third block of a packed gradient, this
        // head's row groups of this workgroup, every second one (the other tensor's workgroup takes the rest)
        constexpr int PPR = DH / 8, RPI = 64 / PPR;
        for (int g = blockIdx.x * kFeatureBwdWaves + wv; g * 16 < R; g += gridDim.x * kFeatureBwdWaves) {
            if ((g & 1) != (int)blockIdx.z) continue;
            uint4 row[16 / RPI];
#pragma unroll
            for (int k = 0; k < 16 / RPI; ++k)
                row[k] = *reinterpret_cast<const uint4*>(copy_src + ((int64_t)min(g * 16 + k * RPI + lane / PPR, R - 1) * H + h) * DH +
                                                         lane % PPR * 8);
#pragma unroll
            for (int k = 0; k < 16 / RPI; ++k) {
                const int r = g * 16 + k * RPI + lane / PPR;
                if (r < R) *reinterpret_cast<uint4*>(copy_dst + (int64_t)r * dx_rs + h * DH + lane % PPR * 8) = row[k];
            }
        }
    }
    constexpr int TA = Cfg::kTA, TB = Cfg::kTB;
    f4 dwacc[TA][TB];   // (m = c, n = j); shared: tile column wv % kWA, tile rows TB (wv / kWA) ..
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b) dwacc[a][b] = f4_zero();

    const int ngrp = (R + 15) / 16, gstride = gridDim.x * kFeatureBwdWaves;
    int grp = blockIdx.x * kFeatureBwdWaves + wv;
    // Two sets of row registers: the loads of the next group are issued into the set the
    // current group does not use, so no set is ever copied.  Rows past R read the last row (no
    // branch around the loads); their du is replaced by 0 (a factor of 0 would leave NaN where that row's gradient is
    // infinite), which keeps them out of dW', and their dx is not stored.
    struct Rows { h8 x[DH / 32], gs[D / 32], gc[D / 32]; };
    auto issue_loads = [&](Rows& t, int g) {
        const int64_t row = (int64_t)min(g * 16 + i, R - 1) * H + h;
        const half_t* px = x + row * DH + 8 * G;
        const half_t* pg = gphi + row * (2 * D) + 8 * G;
#pragma unroll
        for (int cs = 0; cs < DH / 32; ++cs) t.x[cs] = *reinterpret_cast<const h8*>(px + cs * 32);
#pragma unroll
        for (int p = 0; p < D / 32; ++p) {
            t.gs[p] = *reinterpret_cast<const h8*>(pg + 32 * p);
            t.gc[p] = *reinterpret_cast<const h8*>(pg + D + 32 * p);
        }
    };
    const int trow = 4 * G + (i >> 2), tcol = 4 * (i & 3);    // this lane's address in a transposing read
    const bool want_dw = dw_part != nullptr;                  // no partial sums asked for: dx only
    auto process = [&](const Rows& t, int g) {
        const int r = g * 16 + i;
        float ss = 0.f;
#pragma unroll
        for (int cs = 0; cs < DH / 32; ++cs) {
            if (want_dw) *reinterpret_cast<h8*>(Xs + i * LDX + cs * 32 + 8 * G) = t.x[cs];
            ss += dot_h8(__builtin_bit_cast(uint4, t.x[cs]), __builtin_bit_cast(uint4, t.x[cs]));
        }
        ss = sum_over_groups(ss);
        const float nrm = __builtin_amdgcn_sqrtf(ss);
        const float inv = rcp_nr(nrm + 1e-3f);
        const float coef = nrm > 0.f ? inv * rcp_nr(nrm) : 0.f;
        const float inv_turns = inv * 0.15915494309189535f;
        const float sinv = scale * inv;

        h8 du[D / 32];
#pragma unroll
        for (int p = 0; p < D / 32; ++p) {
            f4 acc[2] = {f4_zero(), f4_zero()};   // u^T tiles 2p, 2p+1 (m = feature, n = row)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int cs = 0; cs < DH / 32; ++cs)
                    acc[q] = mfma32(row8(Ws, LDW, 32 * p + 16 * q + i, cs * 32, G), t.x[cs], acc[q]);
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float s_, c_;
                    sincos_turns(acc[q][e] * inv_turns, s_, c_);
                    du[p][4 * q + e] = (half_t)(sinv * (c_ * (float)t.gs[p][4 * q + e] - s_ * (float)t.gc[p][4 * q + e]));
                }
            if (r >= R) du[p] = h8_zero();
            if (want_dw) *reinterpret_cast<h8*>(Us + i * LDU + 32 * p + 8 * G) = du[p];
        }
        if (kShared && want_dw) __syncthreads();      // the rows of all waves are in place

        // y^T tiles (m = input column in pair order, n = row)
        f4 y[DH / 16];
        float xdot = 0.f;
#pragma unroll
        for (int ct = 0; ct < DH / 16; ++ct) {
            f4 acc = f4_zero();
#pragma unroll
            for (int p = 0; p < D / 32; ++p) acc = mfma32(w_col_pair8<LDW>(Ws, 32 * p, ct, lane), du[p], acc);
            y[ct] = acc;
#pragma unroll
            for (int e = 0; e < 4; ++e) xdot += acc[e] * (float)t.x[ct / 2][4 * (ct % 2) + e];
        }
        xdot = sum_over_groups(xdot) * coef;
        half_t* po = dx + (int64_t)r * dx_rs + h * DH + 8 * G;
#pragma unroll
        for (int u = 0; u < DH / 32; ++u) {
            h8 o;
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[4 * q + e] = (half_t)(y[2 * u + q][e] - (float)t.x[u][4 * q + e] * xdot);
            if (r < R) *reinterpret_cast<h8*>(po + 32 * u) = o;
        }

        // dW' (m = c, n = j) += x^T du over the 16 rows of the group, or the 128 of all waves
        if (!want_dw) return;
        if constexpr (kShared) {
#pragma unroll
            for (int ks = 0; ks < 16 * kFeatureBwdWaves / 32; ++ks) {
                const h8 xa = col8(Xall, LDX, 32 * ks, 16 * (wv % Cfg::kWA), lane);
#pragma unroll
                for (int b = 0; b < TB; ++b)
                    dwacc[0][b] = mfma32(xa, col8(Uall, LDU, 32 * ks, 16 * (TB * (wv / Cfg::kWA) + b), lane), dwacc[0][b]);
            }
            __syncthreads();      // before the next rows overwrite them
        } else {
            wave_lds_order();
            h4 xa[DH / 16];
#pragma unroll
            for (int a = 0; a < DH / 16; ++a) xa[a] = tr_read4(Xs + trow * LDX + 16 * a + tcol);
#pragma unroll
            for (int b = 0; b < D / 16; ++b) {
                const h4 ub = tr_read4(Us + trow * LDU + 16 * b + tcol);
#pragma unroll
                for (int a = 0; a < DH / 16; ++a) dwacc[a][b] = mfma16(xa[a], ub, dwacc[a][b]);
            }
            wave_lds_order();   // before the next group's rows overwrite Xs / Us
        }
    };
    Rows ra, rb;
    // where the waves meet, the group of wave 0 decides for all (the others' may lie past the end: nothing of it counts)
    const int ahead = kShared ? wv : 0;
    if (grp - ahead < ngrp) issue_loads(ra, grp);
    __syncthreads();   // W' in place
    while (grp - ahead < ngrp) {
        if (grp - ahead + gstride < ngrp) issue_loads(rb, grp + gstride);
        process(ra, grp);
        if ((grp += gstride) - ahead >= ngrp) break;
        if (grp - ahead + gstride < ngrp) issue_loads(ra, grp + gstride);
        process(rb, grp);
        grp += gstride;
    }
    if constexpr (kShared) {
        if (!want_dw) return;
        float* out = dw_part + ((int64_t)(blockIdx.z * gridDim.x + blockIdx.x) * H + h) * D * DH;
#pragma unroll
        for (int b = 0; b < TB; ++b)
            *reinterpret_cast<f4*>(out + (16 * (TB * (wv / Cfg::kWA) + b) + i) * DH + 16 * (wv % Cfg::kWA) + 4 * G) = dwacc[0][b];
        return;
    }

    if constexpr (!kShared) {
    // The waves' sums, one round: every wave leaves its dW' in LDS, then wave w adds up tiles
    // w, w + 8, ... of all the waves, in wave order, and stores them.
    if (!want_dw) return;
    f4* red = reinterpret_cast<f4*>(smem_raw);
    __syncthreads();   // every wave is out of the row loop: its LDS becomes the exchange area
#pragma unroll
    for (int a = 0; a < DH / 16; ++a)
#pragma unroll
        for (int b = 0; b < D / 16; ++b) red[(wv * Cfg::kTiles + a * (D / 16) + b) * 64 + lane] = dwacc[a][b];
    __syncthreads();
    float* out = dw_part + ((int64_t)(blockIdx.z * gridDim.x + blockIdx.x) * H + h) * D * DH;
    for (int t = wv; t < Cfg::kTiles; t += kFeatureBwdWaves) {
        f4 sum = red[t * 64 + lane];
#pragma unroll
        for (int o = 1; o < kFeatureBwdWaves; ++o) sum += red[(o * Cfg::kTiles + t) * 64 + lane];
        const int a = t / (D / 16), b = t % (D / 16);
        *reinterpret_cast<f4*>(out + (16 * b + i) * DH + 16 * a + 4 * G) = sum;
    }
    }
}

// dw[e] = sum_b dw_part[b][e], to fp32 or (dw16 given) rounded once to fp16, the gradient autograd wants: no
// conversion launch behind it (2.1 to 4.7 us, and 5 of host time).  One workgroup of 4 waves per 256 consecutive elements
// (64 lanes x 16 bytes); wave p sums the shares b = p, p+4, ... with all its loads in
// flight at once, then the 4 waves are added through LDS.  elems % 256 == 0.
__device__ __forceinline__ void feature_map_dw_sum(int block, const float* __restrict__ part, float* __restrict__ dw,
                                                   half_t* __restrict__ dw16, int nblk, int64_t elems) {
    __shared__ f4 red[3][64];
    const int lane = threadIdx.x & 63, p = threadIdx.x >> 6;
    const int64_t e = ((int64_t)block * 64 + lane) * 4;
    f4 acc = f4_zero();
    int b = p;
    for (; b + 28 < nblk; b += 32) {
        f4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const f4*>(part + (int64_t)(b + 4 * u) * elems + e);
#pragma unroll
        for (int u = 0; u < 8; ++u) acc += v[u];
    }
    for (; b < nblk; b += 4) acc += *reinterpret_cast<const f4*>(part + (int64_t)b * elems + e);
    if (p > 0) red[p - 1][lane] = acc;
    __syncthreads();
    if (p == 0) {
        acc += red[0][lane];
        acc += red[1][lane];
        acc += red[2][lane];
        if (dw16) *reinterpret_cast<h4*>(dw16 + e) = to_h4(acc);
        else *reinterpret_cast<f4*>(dw + e) = acc;
    }
}

__global__ __launch_bounds__(kThreads) void k_feature_map_dw_reduce(const float* __restrict__ part,
                                                                    float* __restrict__ dw,
                                                                    half_t* __restrict__ dw16, int nblk,
                                                                    int64_t elems) {
    feature_map_dw_sum(blockIdx.x, part, dw, dw16, nblk, elems);
}

// W' = (sigma * W if sigma) / tau, one element per thread, in the reference's own arithmetic
// (utils.py:90-97 on fp16 tensors: the product is rounded to fp16, then divided by tau in
// fp32 and rounded again).  w, out: [H, D, d]; sigma: [H, d] (broadcast over D) or NULL.
__global__ __launch_bounds__(kThreads) void k_build_random_matrices(const half_t* __restrict__ w,
                                                                    const half_t* __restrict__ sigma,
                                                                    half_t* __restrict__ out, float tau, int D,
                                                                    int d, int64_t total) {
    const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (e >= total) return;
    half_t t = w[e];
    if (sigma) t = (half_t)((float)sigma[(e / ((int64_t)D * d)) * d + e % d] * (float)t);
    out[e] = (half_t)((float)t / tau);
}

// Gradient of k_build_random_matrices as autograd forms it from the same fp16 operations, with
// t = fp16(g / tau):  dw = fp16(t * sigma) (t itself without sigma), one element per thread.
__global__ __launch_bounds__(kThreads) void k_build_random_matrices_dw(const half_t* __restrict__ sigma,
                                                                       const half_t* __restrict__ g,
                                                                       half_t* __restrict__ dw, float tau, int D,
                                                                       int d, int64_t total) {
    const int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x;
    if (e >= total) return;
    const half_t t = (half_t)((float)g[e] / tau);
    dw[e] = sigma ? (half_t)((float)t * (float)sigma[(e / ((int64_t)D * d)) * d + e % d]) : t;
}

// dsigma[h][c] = fp16(sum_j fp16(t[h][j][c] * w[h][j][c])), fp32 sum.  grid = H * nb, nb at most ceil(d / 64): a workgroup
// takes 64 columns of a head (then those 64 nb further), the D rows dealt to its 16 waves, the 16 partial sums added in wave order.  One round trip to memory behind a launch:
// every thread asks for all its rows of g and w (4 at D = 64) before it uses the first.  us (four waves and all columns in one
// workgroup before): 8 heads of 64 x 64 3.9 -> 3.5, 8 of 128 x 128 9.9 -> 3.9.
constexpr int kDsigmaWaves = 16;
__global__ __launch_bounds__(64 * kDsigmaWaves) void k_build_random_matrices_dsigma(const half_t* __restrict__ w,
                                                                                    const half_t* __restrict__ g,
                                                                                    half_t* __restrict__ dsigma, float tau,
                                                                                    int D, int d, int nb) {
    constexpr int NW = kDsigmaWaves, U = 8;
    __shared__ float red[NW][64];
    const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
    const int h = blockIdx.x / nb;
    const half_t* wh = w + (int64_t)h * D * d;
    const half_t* gh = g + (int64_t)h * D * d;
    for (int c0 = (int)(blockIdx.x % nb) * 64; c0 < d; c0 += 64 * nb) {
        const int c = c0 + lane;
        float acc = 0.f;
        if (c < d) {
            for (int j0 = slice; j0 < D; j0 += U * NW) {
                half_t gv[U], wv[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int j = min(j0 + NW * u, D - 1);
                    gv[u] = gh[j * d + c];
                    wv[u] = wh[j * d + c];
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (j0 + NW * u < D) {
                        const half_t t = (half_t)((float)gv[u] / tau);
                        acc += (float)(half_t)((float)t * (float)wv[u]);
                    }
                }
            }
        }
        red[slice][lane] = acc;
        __syncthreads();
        if (slice == 0 && c < d) {
            float sum = red[0][lane];
#pragma unroll
            for (int s = 1; s < NW; ++s) sum += red[s][lane];
            dsigma[(int64_t)h * d + c] = (half_t)sum;
        }
        __syncthreads();
    }
}

}  // namespace rfa
