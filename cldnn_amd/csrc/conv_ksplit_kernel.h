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
//            found by a lane each for 64 steps at once.  A feature count that is not a multiple of 64 ends in a step that starts
//            at the last four slices; the slices it repeats have zero weights.
//   LANES    anything else (fewer than four slices, no border): every lane computes tap and slice of its own chunk and
//            checks the tap against the image where there is no border.
//   GATHERED a fully_connected over a plane: the activations were put into fragment order by gemv_gather_kernel.
//
// With so few bytes a wave what is left is latency, so nothing on the way is waited for twice: all arguments come behind one wait
// (a block of their own, KsplitArgs), the lanes find the offsets of 64 K-steps at once, and what the epilogue reads is requested with
// the operands.  From the first workgroup's start to the last one's end, batch 1 (before: arguments in two waits, offsets walked by
// scalar counters, the epilogue's reads and a drain of the queue in front of the meeting): 3x3 256 -> 256 at 14x14 2.30 -> 1.99 us, 1x1
// 1024 -> 256 2.09 -> 1.83, 3x3 512 -> 512 at 7x7 3.05 -> 2.75, 1x1 512 -> 128 at 28x28 1.96 -> 1.67; of these 0.45 pass until
// the last workgroup has started and 0.6 to 0.8 until the operands are there; 4 or 8 waves instead of 16 change less than 0.1.
// The price are 10 to 20 registers: with more than 96 a workgroup of sixteen waves does not start beside the finishing waves of the one
// before.  With many workgroups to a CU that costs a tile of one to four fragments 3 to 10 %, 30 % under the run-time epilogue (256 -> 256,
// 3x3 at 14x14, batch 48, 32 x 32 tiles: 25.9 -> 27.5 us).  Such sizes go to the 32 x 64 tile or to other kernels; only a tile
// override brings them here.
#pragma once
#include "conv_mfma_kernel.h"

namespace chip {

enum { ADDR_UNIFORM = 0, ADDR_LANES = 1, ADDR_GATHERED = 2 };
enum { GEMV_SLACK = 32 };  // K-steps of slack behind every gathered pixel fragment

struct KsplitArgs {
    const int8_t* in;                    // of tap (0, 0) of output pixel (0, 0)
    const v4i *wpk, *bpk;                // weights; activations in fragment order (GATHERED)
    const int32_t* acc_init;
    void* out;
    const int8_t* eltw;
    const int32_t* origin;
    FastDiv div_inner, div_ohw, div_ow, div_taps, div_fx;
    // workgroup id -> (outer tile, inner tile): dies take every eighth outer one (die_bits 3) or tiles are counted off (0)
    int32_t inner, die_bits, features_outer, mtiles, ftiles;
    uint32_t M;
    int32_t OFM, OHW, OW;
    int32_t ksteps, kper, kwaves;
    int32_t in_pb, in_row, in_col, in_pf;  // bytes; row and column of an output pixel
    int32_t last_group, taps, FX, tap_dy, tap_dx;
    int32_t out_off, out_pb, out_pf, out_py, out_f;
    int32_t el_off, el_pb, el_pf, el_row, el_col;
    uint32_t xor_mask;
    // LANES, and the accumulators alone
    FastDiv div_cb;
    int32_t CB, kchunks, checked, sy, sx, py, px, dil_y, dil_x, IH, IW, OH;
    uint32_t inside;                     // of a byte that exists, behind `in`
    int32_t* raw;
    FastEpi fe;
    Epilogue epi;
};

// look-ahead in K-steps: what 128 registers hold (16 waves of a workgroup = four per SIMD).  32 x 64 tiles have eight waves, and above
// 128 registers a CU holds one workgroup instead of two: with lanes' addresses, or two rows of a pooling window, three steps take 130 to
// 135, two take 104 to 112.  256 -> 256, 3x3 at 14x14 without a border, three steps and two: batch 8 (224 workgroups) 5.34 and 5.26 us,
// batch 16 9.05 and 7.12, batch 64 30.3 and 22.3; with its pooling, batch 8 4.60 and 4.48, batch 64 21.4 and 17.5.  Only a walk of many
// steps on a CU of its own likes three better: 788 -> 142 at 9x9, batch 8 (15 steps a wave), 9.3 and 9.8.  The run-time form of the epilogue
// keeps three: batch 1 6.03 and 6.60, batch 8 6.28 and 6.87.
template <int FT, int PT, int ADDR, int EPI>
constexpr int ksplit_depth()
{
    constexpr bool TWO = FT * PT == 8 && (EPI == EPI_KIND_POOL || (ADDR == ADDR_LANES && EPI != EPI_KIND_FAST));
    return FT * PT == 1 ? 8 : (FT * PT == 2 ? 6 : (TWO ? 2 : FT * PT == 8 || ADDR == ADDR_LANES ? 3 : 4));
}

// Everything on the way to the stores, behind one wait.  (Fetched where it is first used it was two waits in front of the first
// request and one in front of the epilogue.)
__device__ __forceinline__ void fetch_arguments(const KsplitArgs& a)
{
    asm volatile("" ::"s"(a.in), "s"(a.wpk), "s"(a.bpk), "s"(a.acc_init), "s"(a.out), "s"(a.eltw), "s"(a.origin), "s"(a.div_inner.mul), "s"(a.div_inner.shift),
                 "s"(a.div_ohw.mul), "s"(a.div_ohw.shift), "s"(a.div_ow.mul), "s"(a.div_ow.shift), "s"(a.div_taps.mul), "s"(a.div_taps.shift), "s"(a.div_fx.mul),
                 "s"(a.div_fx.shift), "s"(a.inner), "s"(a.die_bits), "s"(a.features_outer), "s"(a.mtiles), "s"(a.ftiles), "s"(a.M), "s"(a.OFM));
    asm volatile("" ::"s"(a.OHW), "s"(a.OW), "s"(a.ksteps), "s"(a.kper), "s"(a.kwaves), "s"(a.in_pb), "s"(a.in_row), "s"(a.in_col), "s"(a.in_pf), "s"(a.last_group),
                 "s"(a.taps), "s"(a.FX), "s"(a.tap_dy), "s"(a.tap_dx), "s"(a.out_off), "s"(a.out_pb), "s"(a.out_pf), "s"(a.out_py), "s"(a.out_f), "s"(a.el_off),
                 "s"(a.el_pb), "s"(a.el_pf), "s"(a.el_row), "s"(a.el_col), "s"(a.xor_mask));
    asm volatile("" ::"s"(a.epi.calib), "s"(a.epi.eltw_calib), "s"(a.epi.wqf), "s"(a.fe.hi), "s"(a.fe.lo), "s"(a.fe.lo2), "s"(a.fe.split_valid), "s"(a.fe.eltw_u8));
}

template <int FT, int PT, int ADDR, int EPI>
__global__ void __launch_bounds__(FT * PT == 8 ? 512 : 1024) conv_ksplit_kernel(KsplitArgs a)
{
    fetch_arguments(a);
    constexpr int D = ksplit_depth<FT, PT, ADDR, EPI>();
    constexpr int SUB = 4 / FT;  // feature tiles per span of 64
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kq = lane >> 4;
    const int l16 = lane & 15;

    // The dies share out the tiles of the larger operand (see conv_mfma_kernel); with fewer than eight tiles of either
    // kind that would leave dies idle, so then the tiles are simply counted off.
    const uint32_t j = blockIdx.x >> a.die_bits, die = blockIdx.x & ((1u << a.die_bits) - 1u);
    const uint32_t turn = a.div_inner.div(j);
    const int inner = (int)(j - turn * (uint32_t)a.inner), outer = (int)((turn << a.die_bits) + die);
    const int ptile = a.features_outer ? inner : outer, ntile = a.features_outer ? outer : inner;
    if (ptile >= a.mtiles || ntile >= a.ftiles) return;
    const int span = ntile / SUB, q0 = (ntile & (SUB - 1)) * FT;

    const int s0 = wave * a.kper;
    const int n = min(a.kper, a.ksteps - s0);  // K-steps of this wave; none or fewer for the last waves
    const v4i xm = {(int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask};
    const int8_t* wsrc = (const int8_t*)(a.wpk + ((size_t)span * a.ksteps + s0) * 256 + q0 * 16);
    const uint32_t wlane = (uint32_t)(kq * 64 + l16) * 16u;
    const v4i* bsrc = a.bpk + ((size_t)ptile * PT * (a.ksteps + GEMV_SLACK) + s0) * 64 + lane;

    uint32_t boff[PT];
    int iy0[PT], ix0[PT];
    if constexpr (ADDR != ADDR_GATHERED) {
        const uint32_t origin = (uint32_t)span_origin(a, span);
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) {
            bool ok;
            const PixelPos pp = pixel_at<EPI, PT>(a, (uint32_t)ptile * PT * 16, pt, l16, ok);  // pixels past the end read pixel 0
            if constexpr (ADDR == ADDR_LANES) iy0[pt] = (int)pp.oy * a.sy - a.py, ix0[pt] = (int)pp.ox * a.sx - a.px;
            boff[pt] = origin + pp.b * (uint32_t)a.in_pb + pp.oy * (uint32_t)a.in_row + pp.ox * (uint32_t)a.in_col + (ADDR == ADDR_UNIFORM ? (uint32_t)(kq * a.in_pf) : 0u);
        }
    }
    // UNIFORM: where the slices of the wave's steps from + 0 .. 63 lie (taps innermost), a lane each.  (A walk with scalar
    // counters is twenty dependent instructions in front of every request.)
    int offsets = 0, from = 0;
    auto find_offsets = [&](int first) {
        const uint32_t step = (uint32_t)(s0 + first + lane);
        const uint32_t sg = a.div_taps.div(step), tap = step - sg * (uint32_t)a.taps;
        const uint32_t fy = a.div_fx.div(tap), fx = tap - fy * (uint32_t)a.FX;
        offsets = min((int)sg * 4, a.last_group) * a.in_pf + (int)fy * a.tap_dy + (int)fx * a.tap_dx;
        from = first;
    };
    if constexpr (ADDR == ADDR_UNIFORM) find_offsets(0);

    v4i acc[FT][PT];
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int p = 0; p < PT; ++p) acc[f][p] = v4i{0, 0, 0, 0};
    auto load = [&](int k, v4i (&xa)[FT], v4i (&xb)[PT]) {
#pragma unroll
        for (int f = 0; f < FT; ++f) xa[f] = *reinterpret_cast<const v4i*>(wsrc + (size_t)k * 4096 + f * 256 + wlane);
        if constexpr (ADDR == ADDR_GATHERED) {
#pragma unroll
            for (int p = 0; p < PT; ++p) xb[p] = bsrc[((size_t)p * (a.ksteps + GEMV_SLACK) + k) * 64];
        } else if constexpr (ADDR == ADDR_UNIFORM) {
            const uint32_t off = (uint32_t)__builtin_amdgcn_readlane(offsets, k - from);
#pragma unroll
            for (int p = 0; p < PT; ++p) xb[p] = *reinterpret_cast<const v4i*>(a.in + (boff[p] + off));
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
                v4i v = *reinterpret_cast<const v4i*>(a.in + (ok ? boff[p] + (uint32_t)off : a.inside));
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

    // What the epilogue reads, for the waves that will finish a fragment (wave w < FT * PT: fragment (w % FT, w / FT)).  Requested
    // behind the first operands: in front of the meeting of the sums it was a second trip to memory.
    const int ff = wave % FT, fp = wave / FT;
    const int fb = span * 64 + kq * 16, f0 = fb + (q0 + ff) * 4;
    constexpr bool PAIR = EPI == EPI_KIND_POOL && PT > 1;  // fragments 2k and 2k + 1 are two rows of the same windows
    const bool finisher = wave < FT * PT && !(PAIR && (fp & 1));
    bool live = false;
    int obase = 0;
    [[maybe_unused]] int ebase = 0;
    PixelPos pp{0, 0, 0};
    v4i init = {0, 0, 0, 0};
    LaneScales sc;
    v4i ev4 = {0, 0, 0, 0};
    if constexpr (EPI != EPI_KIND_GENERIC) {
#pragma unroll
        for (int c = 0; c < 16; ++c) sc.cal[c] = sc.wq[c] = sc.ecal[c] = 0.f;
    }
    auto request_rest = [&] {
        step_fence();
        if (!finisher) return;
        bool inside;
        pp = pixel_at<EPI, PT>(a, (uint32_t)ptile * PT * 16, fp, l16, inside);
        live = inside && f0 < a.OFM;
        if constexpr (EPI == EPI_KIND_POOL) pp.oy >>= 1, pp.ox >>= 1;
        obase = a.out_off + (int)pp.b * a.out_pb + (fb >> 4) * a.out_pf + (int)pp.oy * a.out_py + (int)pp.ox * 16 + (f0 & 15) * a.out_f;
        ebase = a.el_off + (int)pp.b * a.el_pb + (fb >> 4) * a.el_pf + (int)pp.oy * a.el_row + (int)pp.ox * a.el_col + (f0 & 15);
        if (live) {
            init = *reinterpret_cast<const v4i*>(a.acc_init + f0);
            load_scales4<EPI == EPI_KIND_POOL ? EPI_KIND_RELU : EPI>(a, f0, sc);
            bool residual = EPI == EPI_KIND_FUSED;
            if constexpr (EPI == EPI_KIND_FAST) residual = a.fe.fused != 0;
            if (residual) ev4[0] = *reinterpret_cast<const int*>(a.eltw + ebase);
        }
    };

    // Two paths.  A wave with at most D steps requests them all, then multiplies.  A longer share runs a loop that is free
    // of branches (a branch around a request makes the compiler drain the queue at the join) over the steps whose
    // successor D steps on exists, and finishes like the short one.
    constexpr bool EARLY = FT * PT < 8 && !(PT == 4 && (EPI == EPI_KIND_FUSED || EPI == EPI_KIND_FAST));  // (the others have no registers for it)
    if (n <= D) {
        v4i ra[D][FT], rb[D][PT];
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (d < n) load(d, ra[d], rb[d]);
        if constexpr (EARLY) request_rest();
        step_fence();
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (d < n) mma(ra[d], rb[d]);
    } else {
        v4i ra[D][FT], rb[D][PT];
#pragma unroll
        for (int d = 0; d < D; ++d) {
            load(d, ra[d], rb[d]);
            step_fence();
        }
        if constexpr (EARLY) request_rest();
        step_fence();
        int k = 0;
        for (; k + 2 * D <= n; k += D) {
            if constexpr (ADDR == ADDR_UNIFORM)
                if (k + 2 * D - from > 64) find_offsets(k + D);
#pragma unroll
            for (int d = 0; d < D; ++d) {
                mma(ra[d], rb[d]);
                load(k + d + D, ra[d], rb[d]);
                step_fence();
            }
        }
        const int rest = n - k - D;  // 0 .. D - 1 steps not requested yet
        if constexpr (ADDR == ADDR_UNIFORM)
            if (n - from > 64) find_offsets(k + D);
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

    // ---- partial sums
    constexpr int TILE = FT * PT * 64;
    extern __shared__ __align__(16) unsigned char smem[];
    v4i* part = reinterpret_cast<v4i*>(smem);
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
        for (int f = 0; f < FT; ++f) part[wave * TILE + (p * FT + f) * 64 + lane] = acc[f][p];
    if constexpr (!EARLY) request_rest();
    lds_barrier();
    if (!live) return;
    // the waves' sums of one fragment on top of `sum`, of 4, 8 or 16 waves (mfma_plan): all reads on their way before the first is added
    auto add_up = [&](const v4i* src, v4i sum) {
        auto add = [&](auto wc) {
            constexpr int W = decltype(wc)::value;
            v4i o[W];
#pragma unroll
            for (int w = 0; w < W; ++w) o[w] = src[w * TILE];
#pragma unroll
            for (int w = 0; w < W; ++w) sum[0] += o[w][0], sum[1] += o[w][1], sum[2] += o[w][2], sum[3] += o[w][3];
            src += W * TILE;
        };
        if (a.kwaves & 4) add(std::integral_constant<int, 4>{});
        if (a.kwaves & 8) add(std::integral_constant<int, 8>{});
        if (a.kwaves & 16) add(std::integral_constant<int, 16>{});
        return sum;
    };
    const v4i* src = part + wave * 64 + lane;  // fragment (ff, fp) is number fp * FT + ff = wave
    v4i sum = add_up(src, init);
    const int valid = a.OFM - f0;
    if constexpr (PAIR) {
        const v4i low = add_up(src + FT * 64, init);
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
void launch_ksplit_instance(hipStream_t s, const KsplitArgs& a, int grid, int epi)
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
void launch_ksplit_tile(hipStream_t s, const KsplitArgs& a, int ft, int pt, int grid, int epi)
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
