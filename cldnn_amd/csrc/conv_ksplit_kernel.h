// Dense quantized convolution with few output tiles: the waves of a workgroup split K.
//
// A network at batch 1, the late layers of any network, a fully_connected: the tile kernels give such a layer 8 to 100
// workgroups whose four waves walk all of K one step at a time, 0.2-0.25 us a step, while most of the chip idles (7x7
// 512 -> 512 3x3 at batch 1: 8 workgroups, 72 steps, 10.3 us of kernel time; here 4.5).  What bounds the layer is the length of that
// walk, so here a workgroup owns a small tile (16 .. 64 pixels x 16 .. 64 features) and its 4, 8 or 16 waves take a share
// of the K-steps each: both operands go straight from global memory into the registers the matrix instruction reads, D
// steps ahead, no LDS and no barrier in the loop.  With K shared out a wave has 1 to 5 steps and usually requests all its
// operands before it waits for any: the layer costs about one memory round trip.  The partial sums meet in LDS (integer
// sums: any order gives the same bits) and every thread finishes four consecutive features of one pixel.
//
// The tile is the smallest one that still fills the chip (mfma_choose): bytes per workgroup are (features + pixels) * K,
// and a CU takes them at about 40 bytes per clock.
//
// Weights are the tile kernels' packed stream for 64-feature spans; a workgroup takes FT of the four 16-row fragments of a
// span.  Fragment q's row kq * 4 + i is feature 16 * kq + 4 * q + i of the span, so a lane ends up with four consecutive
// features.
//
// How the offset of an activation fragment is found (ADDR):
//   UNIFORM  the four k-chunks of a step are one tap and four slices of the bordered input: one scalar offset per step,
//            walked with scalar counters.  A feature count that is not a multiple of 64 ends in a step that starts at the
//            last four slices; the slices it repeats have zero weights.
//   LANES    anything else (fewer than four slices, no border): every lane computes tap and slice of its own chunk and
//            checks the tap against the image where there is no border.
//   GATHERED a fully_connected over a plane: the activations were put into fragment order by gemv_gather_kernel.
#pragma once
#include "conv_mfma_kernel.h"

namespace chip {

enum { ADDR_UNIFORM = 0, ADDR_LANES = 1, ADDR_GATHERED = 2 };
enum { GEMV_SLACK = 32 };  // K-steps of slack behind every gathered pixel fragment

// look-ahead in K-steps: what 128 registers hold (16 waves of a workgroup = four per SIMD)
template <int FT, int PT>
constexpr int ksplit_depth()
{
    return FT * PT == 1 ? 8 : (FT * PT == 2 ? 6 : (FT * PT == 8 ? 3 : 4));
}

template <int FT, int PT, int ADDR, int EPI>
__global__ void __launch_bounds__(FT * PT == 8 ? 512 : 1024) conv_ksplit_kernel(MfmaArgs a)
{
    fetch_arguments(a);
    constexpr int D = ksplit_depth<FT, PT>();
    constexpr int SUB = 4 / FT;  // feature tiles per span of 64
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kq = lane >> 4;
    const int l16 = lane & 15;

    // The dies share out the tiles of the larger operand (see conv_mfma_kernel); with fewer than eight tiles of either
    // kind that would leave dies idle, so then the tiles are simply counted off.
    int ptile, ntile;
    if (a.by_features == 2) {
        ntile = (int)a.div_mtiles.div(blockIdx.x);
        ptile = (int)blockIdx.x - ntile * a.mtiles;
    } else {
        const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
        const int j_by_m = (int)a.div_mtiles.div((uint32_t)j), j_by_f = (int)a.div_ofm_tiles.div((uint32_t)j);
        ptile = a.by_features ? j - j_by_m * a.mtiles : j_by_f * 8 + xcd;
        ntile = a.by_features ? j_by_m * 8 + xcd : j - j_by_f * a.ofm_tiles;
    }
    if (ptile >= a.mtiles || ntile >= a.ofm_tiles) return;
    const int span = ntile / SUB, q0 = (ntile & (SUB - 1)) * FT;

    const int s0 = wave * a.kper;
    const int n = min(a.kper, a.ksteps - s0);  // K-steps of this wave; none or fewer for the last waves
    const v4i xm = {(int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask};
    const v4i* wsrc = a.wpk + ((size_t)span * a.ksteps + s0) * 256 + kq * 64 + q0 * 16 + l16;
    const v4i* bsrc = a.bpk + ((size_t)ptile * PT * (a.ksteps + GEMV_SLACK) + s0) * 64 + lane;

    uint32_t boff[PT];
    int iy0[PT], ix0[PT];
    const int origin = a.in_off + span_origin(a, span);
#pragma unroll
    for (int pt = 0; pt < PT; ++pt) {
        bool ok;
        const PixelPos pp = pixel_at<EPI, PT>(a, (uint32_t)ptile * PT * 16, pt, l16, ok);  // pixels past the end read pixel 0
        iy0[pt] = (int)pp.oy * a.sy - a.py, ix0[pt] = (int)pp.ox * a.sx - a.px;
        boff[pt] = (uint32_t)(origin + (int)pp.b * a.in_pb + iy0[pt] * a.in_py + ix0[pt] * 16 + (ADDR == ADDR_UNIFORM ? kq * a.in_pf : 0));
    }

    // (group of four slices, filter row, filter column) of the next step to request; taps innermost
    int sg = 0, fy = 0, fx = 0;
    if constexpr (ADDR == ADDR_UNIFORM) {
        const int taps = a.FX * a.FY;
        sg = (int)a.div_taps.div((uint32_t)s0);
        const int tap = s0 - sg * taps;
        fy = (int)a.div_fx.div((uint32_t)tap);
        fx = tap - fy * a.FX;
    }
    v4i acc[FT][PT];
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int p = 0; p < PT; ++p) acc[f][p] = v4i{0, 0, 0, 0};
    v4i ra[D][FT], rb[D][PT];
    auto load = [&](int k, v4i (&xa)[FT], v4i (&xb)[PT]) {
#pragma unroll
        for (int f = 0; f < FT; ++f) xa[f] = wsrc[(size_t)k * 256 + f * 16];
        if constexpr (ADDR == ADDR_GATHERED) {
#pragma unroll
            for (int p = 0; p < PT; ++p) xb[p] = bsrc[((size_t)p * (a.ksteps + GEMV_SLACK) + k) * 64];
        } else if constexpr (ADDR == ADDR_UNIFORM) {
            const int8_t* base = a.in + (min(sg * 4, a.CB - 4) * a.in_pf + fy * a.tap_dy + fx * a.tap_dx);
#pragma unroll
            for (int p = 0; p < PT; ++p) xb[p] = *reinterpret_cast<const v4i*>(base + boff[p]);
            fx += 1;
            if (fx == a.FX) fx = 0, fy += 1;
            if (fy == a.FY) fy = 0, sg += 1;
        } else {
            // chunk -> (tap, slice), slices innermost
            const uint32_t kc = (uint32_t)(s0 + k) * 4 + kq;
            const uint32_t tap = a.div_cb.div(kc);
            const int cb = (int)(kc - tap * a.CB);
            const int ty = (int)a.div_fx.div(tap), tx = (int)tap - ty * a.FX;
            const bool real = kc < (uint32_t)a.kchunks;  // padding chunks have zero weights and read the image's first bytes
            const int off = cb * a.in_pf + ty * a.tap_dy + tx * a.tap_dx;
#pragma unroll
            for (int p = 0; p < PT; ++p) {
                bool ok = real;
                if (a.checked) {
                    const int iy = iy0[p] + ty * a.dil_y, ix = ix0[p] + tx * a.dil_x;
                    ok = real && iy >= 0 && iy < a.IH && ix >= 0 && ix < a.IW;
                }
                const int8_t* src = ok ? a.in + (boff[p] + (uint32_t)off) : a.in + a.in_off;
                v4i v = *reinterpret_cast<const v4i*>(src);
                if (a.checked && !ok) v = v4i{0, 0, 0, 0};
                xb[p] = v;
            }
        }
    };
    auto mma = [&](const v4i (&xa)[FT], const v4i (&xb)[PT]) {
#pragma unroll
        for (int p = 0; p < PT; ++p) {
            const v4i b = ADDR == ADDR_GATHERED ? xb[p] : xb[p] ^ xm;  // gathered activations are flipped already
#pragma unroll
            for (int f = 0; f < FT; ++f) acc[f][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[f], b, acc[f][p], 0, 0, 0);
        }
    };

    // Two paths.  A wave with at most D steps requests them all, then multiplies.  A longer share runs a loop that is free
    // of branches (a branch around a request makes the compiler drain the queue at the join) over the steps whose
    // successor D steps on exists, and finishes like the short one.
    if (n <= D) {
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (d < n) load(d, ra[d], rb[d]);
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (d < n) mma(ra[d], rb[d]);
    } else {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load(d, ra[d], rb[d]);
            step_fence();
        }
        int k = 0;
        for (; k + 2 * D <= n; k += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                mma(ra[d], rb[d]);
                load(k + d + D, ra[d], rb[d]);
                step_fence();
            }
        }
        const int rest = n - k - D;  // 0 .. D - 1 steps not requested yet
#pragma unroll
        for (int d = 0; d < D; ++d) {
            mma(ra[d], rb[d]);
            if (d < rest) load(k + d + D, ra[d], rb[d]);
        }
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (d < rest) mma(ra[d], rb[d]);
    }

    mfma_settle(acc);

    // ---- partial sums; wave w < FT * PT finishes fragment (w % FT, w / FT)
    constexpr int TILE = FT * PT * 64;
    extern __shared__ __align__(16) unsigned char smem[];
    v4i* part = reinterpret_cast<v4i*>(smem);
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
        for (int f = 0; f < FT; ++f) part[wave * TILE + (p * FT + f) * 64 + lane] = acc[f][p];

    const int ff = wave % FT, fp = wave / FT;
    const int fb = span * 64 + kq * 16, f0 = fb + (q0 + ff) * 4;
    constexpr bool PAIR = EPI == EPI_KIND_POOL && PT > 1;  // fragments 2k and 2k + 1 are two rows of the same windows
    const bool finisher = wave < FT * PT && !(PAIR && (fp & 1));
    bool inside;
    PixelPos pp = pixel_at<EPI, PT>(a, (uint32_t)ptile * PT * 16, finisher ? fp : 0, l16, inside);
    const bool live = finisher && inside && f0 < a.OFM;
    if constexpr (EPI == EPI_KIND_POOL) pp.oy >>= 1, pp.ox >>= 1;
    const int obase = a.out_off + (int)pp.b * a.out_pb + (fb >> 4) * a.out_pf + (int)pp.oy * a.out_py + (int)pp.ox * 16 + (f0 & 15) * a.out_f;
    const int ebase = a.el_off + (int)pp.b * a.el_pb + (fb >> 4) * a.el_pf + (int)(pp.oy * a.esy) * a.el_py + (int)(pp.ox * a.esx) * 16 + (f0 & 15);
    // what the epilogue reads, requested in front of the barrier
    v4i init = {0, 0, 0, 0};
    LaneScales sc;
    v4i ev4 = {0, 0, 0, 0};
    if constexpr (EPI != EPI_KIND_GENERIC) {
#pragma unroll
        for (int c = 0; c < 16; ++c) sc.cal[c] = sc.wq[c] = sc.ecal[c] = 0.f;
    }
    if (live) {
        init = *reinterpret_cast<const v4i*>(a.acc_init + f0);
        load_scales4<EPI == EPI_KIND_POOL ? EPI_KIND_RELU : EPI>(a, f0, sc);
        bool residual = EPI == EPI_KIND_FUSED;
        if constexpr (EPI == EPI_KIND_FAST) residual = a.fe.fused != 0;
        if (residual) ev4[0] = *reinterpret_cast<const int*>((const int8_t*)a.eltw + ebase);
    }
    __syncthreads();
    if (!live) return;
    v4i sum = init;
    const v4i* src = part + wave * 64 + lane;  // fragment (ff, fp) is number fp * FT + ff = wave
    for (int w = 0; w < a.kwaves; ++w) {
        const v4i o = src[w * TILE];
        sum[0] += o[0], sum[1] += o[1], sum[2] += o[2], sum[3] += o[3];
    }
    const int valid = a.OFM - f0;
    if constexpr (PAIR) {
        v4i low = init;
        for (int w = 0; w < a.kwaves; ++w) {
            const v4i o = src[w * TILE + FT * 64];
            low[0] += o[0], low[1] += o[1], low[2] += o[2], low[3] += o[3];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] = max_dpp<0xb1>(max(sum[i], low[i]));
        if (l16 & 1) return;  // the first of the window's lanes stores its four features
    } else if constexpr (EPI == EPI_KIND_POOL) {
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] = max_of_window(sum[i]);
        if (l16 & 3) return;
    }
    if constexpr (EPI == EPI_KIND_GENERIC) {
        const Epilogue& e = a.epi;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i >= valid) break;
            if (a.raw) {
                a.raw[(((size_t)pp.b * a.OFM + f0 + i) * a.OH + pp.oy) * a.OW + pp.ox] = sum[i];
                continue;
            }
            float ev = 0.f;
            if (e.fused) ev = load_as_float(a.eltw, e.eltw_dt, ebase + i);
            store_out(a.out, e.out_dt, obase + i * a.out_f, epilogue_generic(e, sum[i], f0 + i, ev));
        }
    } else if constexpr (EPI == EPI_KIND_F32) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = epilogue_f32(a, (float)sum[i], sc.wq[i], sc.cal[i]);
        float* dst = (float*)a.out + obase;
        if (valid >= 4) *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        else
            for (int i = 0; i < valid; ++i) dst[i] = v[i];
    } else {
        v4i acc4[4][1] = {{sum}, {v4i{0, 0, 0, 0}}, {v4i{0, 0, 0, 0}}, {v4i{0, 0, 0, 0}}};
        const v4i packed = epilogue_fast16<1, EPI == EPI_KIND_POOL ? EPI_KIND_RELU : EPI, 4>(a, acc4, 0, sc.wq, sc.cal, sc.ecal, ev4, valid);
        int8_t* dst = (int8_t*)a.out + obase;
        if (a.out_f == 1) *reinterpret_cast<int*>(dst) = packed[0];
        else  // images innermost: the lanes next to this one write the bytes beside these
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[i * a.out_f] = (int8_t)(packed[0] >> (8 * i));
    }
}

template <int FT, int PT, int ADDR>
void launch_ksplit_instance(hipStream_t s, const MfmaArgs& a, int grid, int epi)
{
    const dim3 g(grid), b(64 * a.kwaves);
    const int lds = a.kwaves * FT * PT * 1024;
    switch (epi) {
    case EPI_KIND_RELU: hipLaunchKernelGGL((conv_ksplit_kernel<FT, PT, ADDR, EPI_KIND_RELU>), g, b, lds, s, a); break;
    case EPI_KIND_FUSED: hipLaunchKernelGGL((conv_ksplit_kernel<FT, PT, ADDR, EPI_KIND_FUSED>), g, b, lds, s, a); break;
    case EPI_KIND_LINEAR: hipLaunchKernelGGL((conv_ksplit_kernel<FT, PT, ADDR, EPI_KIND_LINEAR>), g, b, lds, s, a); break;
    case EPI_KIND_FAST: hipLaunchKernelGGL((conv_ksplit_kernel<FT, PT, ADDR, EPI_KIND_FAST>), g, b, lds, s, a); break;
    case EPI_KIND_F32: hipLaunchKernelGGL((conv_ksplit_kernel<FT, PT, ADDR, EPI_KIND_F32>), g, b, lds, s, a); break;
    case EPI_KIND_POOL: hipLaunchKernelGGL((conv_ksplit_kernel<FT, PT, ADDR, EPI_KIND_POOL>), g, b, lds, s, a); break;
    default: hipLaunchKernelGGL((conv_ksplit_kernel<FT, PT, ADDR, EPI_KIND_GENERIC>), g, b, lds, s, a); break;
    }
}

template <int ADDR>
void launch_ksplit_tile(hipStream_t s, const MfmaArgs& a, int ft, int pt, int grid, int epi)
{
    switch (ft * 8 + pt) {
    case 8 + 1: launch_ksplit_instance<1, 1, ADDR>(s, a, grid, epi); break;
    case 8 + 2: launch_ksplit_instance<1, 2, ADDR>(s, a, grid, epi); break;
    case 8 + 4: launch_ksplit_instance<1, 4, ADDR>(s, a, grid, epi); break;
    case 16 + 2: launch_ksplit_instance<2, 2, ADDR>(s, a, grid, epi); break;
    case 32 + 2: launch_ksplit_instance<4, 2, ADDR>(s, a, grid, epi); break;
    default: throw error(CLDNN_HIP_INVALID_ARG, "split-K kernel: no such tile");
    }
}

}  // namespace chip
