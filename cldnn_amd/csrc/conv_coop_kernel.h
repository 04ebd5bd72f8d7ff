// The bottleneck chain (3x3 -> expansion [+ residual] -> next reduction) with its weights in REGISTERS: the eight waves of a
// workgroup work on one granule of 16 pixels and keep their shares of all three weight tensors for as long as they live.
//
// conv_chain_kernel.h gives every wave granules of its own and keeps the weights in LDS, which takes a copy of 70 KB first;
// on a small plane (ResNet-50 at batch 1: 196 granules at 56x56) that is one long walk of dependent steps on a few CUs.  Here
//   - stage 0 is split over its K-steps: wave w takes tap w of all features, waves 0 to 3 a fragment of the ninth tap each, and the
//     partial sums meet in LDS;
//   - the rounded result (1 KB) goes back through LDS and every wave computes an eighth of the expansion's features, adds its
//     part of the residual and stores it;
//   - stage 2 is split over its K again, which is where each wave's own expansion features are: they never leave its
//     registers, only the partial sums do.
// All weights (56 registers), the residual and the input of the next granule are requested long before they are needed, so
// a granule costs three barriers and its instructions.  Kernel time, 56x56, 64 mid features, batch 1: 10.7 -> 6.2 us with three
// stages, 28x28 with two 9.5 -> 4.0.  Inside a network, where the input comes from memory, two stages are faster at every
// size (ResNet-50 at batch 32 12.7 -> 10.8, at batch 128 33.1 -> 29.0; repeated on warm caches 24.8 and 25.5); three stages
// with many granules are not, splitting costs more instructions per pixel: 10.2 -> 9.4 us at 980 granules, 11.6 -> 14.1 at 1568.
// (The ninth tap's weights in the registers of one wave were four more fragments for every wave: with three stages 128 registers were not
// enough, and a request waited for one that was spilled behind it.)
// 128 mid features (weights in 160 registers) gained 2 us of 12 at batch 1 and lost 8 of 28 at batch 32.
#pragma once
#include "conv_chain_kernel.h"

namespace chip {

struct CoopConvStage {
    int8_t* out;             // nullptr: the result is not written
    int32_t off, pb, pf, py; // of the output, elements
    uint32_t xor_mask;
    int32_t unit0, kstride, vec0;
    float hi;
    int32_t eltw_u8;
};

struct CoopConvArgs {
    const int8_t* in;
    const int8_t* img;       // weight units, vectors
    const int8_t* eltw;
    int32_t vec_bytes, vec_quads;
    int32_t el_off, el_pb, el_pf, el_py, el_px;
    uint32_t M;
    int32_t OHW, OW;
    FastDiv div_ohw, div_ow;
    int32_t in_off, in_pb, in_pf, row, col, tap_dy;
    int32_t gpw, grem;
    FastDiv div_parts;
    CoopConvStage st[CHAIN_MAX_STAGES];
};

struct CoopConvEpi {
    FastEpi fe;
};

// all arguments behind one wait
__device__ __forceinline__ void fetch_arguments(const CoopConvArgs& a)
{
    asm volatile("" ::"s"(a.in), "s"(a.img), "s"(a.eltw), "s"(a.vec_bytes), "s"(a.vec_quads), "s"(a.el_off), "s"(a.el_pb), "s"(a.el_pf), "s"(a.el_py), "s"(a.el_px), "s"(a.M), "s"(a.OHW),
                 "s"(a.OW), "s"(a.div_ohw.mul), "s"(a.div_ohw.shift), "s"(a.div_ow.mul), "s"(a.div_ow.shift), "s"(a.in_off), "s"(a.in_pb), "s"(a.in_pf), "s"(a.row), "s"(a.col),
                 "s"(a.tap_dy), "s"(a.gpw), "s"(a.grem), "s"(a.div_parts.mul), "s"(a.div_parts.shift), "s"(gridDim.x));
#pragma unroll
    for (int k = 0; k < CHAIN_MAX_STAGES; ++k)
        asm volatile("" ::"s"(a.st[k].out), "s"(a.st[k].off), "s"(a.st[k].pb), "s"(a.st[k].pf), "s"(a.st[k].py), "s"(a.st[k].xor_mask), "s"(a.st[k].unit0), "s"(a.st[k].kstride),
                     "s"(a.st[k].vec0), "s"(a.st[k].hi));
    asm volatile("" ::"s"(a.st[1].eltw_u8));
}

// 64 features in the first stage and the reduction, 256 in the expansion
template <bool HAS2, bool SUM>
__global__ void __launch_bounds__(512, 4) conv_coop_kernel(CoopConvArgs a)
{
    constexpr int W = 8, LAST_TAP = 8;
    constexpr int N0 = 4;  // fragments of stages 0 and 2
    constexpr int F1 = 2;  // fragments of the expansion per wave: half a span
    constexpr int RELU = EPI_KIND_RELU, EPI1 = SUM ? EPI_KIND_FUSED : EPI_KIND_RELU;
    fetch_arguments(a);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kq = lane >> 4;
    const int l16 = lane & 15;
    const CoopConvStage &s0 = a.st[0], &s1 = a.st[1], &s2 = a.st[2];
    CoopConvEpi e0{}, e1{}, e2{};
    e0.fe.hi = s0.hi, e1.fe.hi = s1.hi, e2.fe.hi = s2.hi;
    e1.fe.eltw_u8 = s1.eltw_u8;

    extern __shared__ __align__(16) unsigned char smem[];
    v4i* part = reinterpret_cast<v4i*>(smem);     // [W][N0][64], stage 0
    v4i* part2 = part + W * N0 * 64;              // the same, stage 2
    v4i* mid = part2 + (HAS2 ? W * N0 * 64 : 0);  // [64]: stage 0's result as the expansion's B fragments
    v4i* vecs = mid + 64;
    const int32_t* V = reinterpret_cast<const int32_t*>(vecs);

    const uint32_t wg = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);  // the grid is a multiple of 8
    const int g_begin = (int)(wg * (uint32_t)a.gpw + a.div_parts.div(wg * (uint32_t)a.grem));
    const int g_end = (int)((wg + 1) * (uint32_t)a.gpw + a.div_parts.div((wg + 1) * (uint32_t)a.grem));
    if (g_begin >= g_end) return;  // the whole workgroup

    const uint32_t row16 = (uint32_t)(kq * 64 + l16) * 16;
    auto unit = [&](int u, int mt) { return *reinterpret_cast<const v4i*>(a.img + (size_t)(u * 4096 + mt * 256) + row16); };
    const int span1 = wave >> 1, half = wave & 1;  // this wave's part of the expansion

    struct Pos {
        uint32_t b, oy, ox;
        bool ok;
    };
    v4i xb, xb8;  // the wave's tap, the ninth
    int ev[F1];
    Pos cur, nxt;
    auto request = [&](int g, Pos& p) {
        const uint32_t m = (uint32_t)g * 16 + l16;
        p.ok = m < a.M;
        const uint32_t mm = p.ok ? m : 0;  // pixels past the end read pixel 0
        p.b = a.div_ohw.div(mm);
        const uint32_t r = mm - p.b * a.OHW;
        p.oy = a.div_ow.div(r);
        p.ox = r - p.oy * a.OW;
        const uint32_t off = (uint32_t)(a.in_off + (int)p.b * a.in_pb + (int)p.oy * a.row + (int)p.ox * a.col + kq * a.in_pf);
        auto of_tap = [&](int tap) {
            const int ty = (tap * 11) >> 5;
            return *reinterpret_cast<const v4i*>(a.in + (off + (uint32_t)(ty * a.tap_dy + (tap - ty * 3) * 16)));
        };
        xb = of_tap(wave);
        if (wave < N0) xb8 = of_tap(LAST_TAP);
        else asm volatile("" : "=v"(xb8));
    };
    auto residual = [&](const Pos& p) {
        if constexpr (SUM) {
            const int8_t* src = a.eltw + (uint32_t)(a.el_off + (int)p.b * a.el_pb + (int)p.oy * a.el_py + (int)p.ox * a.el_px + (span1 * 4 + kq) * a.el_pf + half * 8);
            const int2 v = *reinterpret_cast<const int2*>(src);
            ev[0] = v.x, ev[1] = v.y;
        }
    };
    auto at = [&](const CoopConvStage& st, const Pos& p, int slice) { return (uint32_t)(st.off + (int)p.b * st.pb + slice * st.pf + (int)p.oy * st.py + (int)p.ox * 16); };

    // ---------------- everything that is needed first, in the order of its use
    v4i w0[N0], w8, w1[F1], w2[HAS2 ? N0 : 1];  // w8: the wave's fragment of the ninth tap
    {
        v4i r[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) r[u] = *reinterpret_cast<const v4i*>(a.img + a.vec_bytes + (uint32_t)min((int)threadIdx.x + u * 512, a.vec_quads - 1) * 16u);
        step_fence();
        request(g_begin, cur);
#pragma unroll
        for (int i = 0; i < N0; ++i) w0[i] = unit(s0.unit0 + wave, i);
        if (wave < N0) w8 = unit(s0.unit0 + LAST_TAP, wave);
        else asm volatile("" : "=v"(w8));
        step_fence();
        residual(cur);
#pragma unroll
        for (int i = 0; i < F1; ++i) w1[i] = unit(s1.unit0 + span1 * s1.kstride, half * 2 + i);
        if constexpr (HAS2) {
#pragma unroll
            for (int i = 0; i < N0; ++i) w2[i] = unit(s2.unit0 + span1, i);
        }
        step_fence();
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if ((int)threadIdx.x + u * 512 < a.vec_quads) vecs[threadIdx.x + u * 512] = r[u];
        for (int i = threadIdx.x + 1024; i < a.vec_quads; i += 512) vecs[i] = *reinterpret_cast<const v4i*>(a.img + a.vec_bytes + (uint32_t)i * 16u);
    }

    const v4i none = {0, 0, 0, 0};
    auto flip = [](int v, uint32_t mask) { return v ^ (int)mask; };
    auto vec4 = [&](int v_at, float(&dst)[16], int d) {
        const v4i q = *reinterpret_cast<const v4i*>(V + v_at);
        dst[d * 4 + 0] = __int_as_float(q[0]), dst[d * 4 + 1] = __int_as_float(q[1]), dst[d * 4 + 2] = __int_as_float(q[2]), dst[d * 4 + 3] = __int_as_float(q[3]);
    };
    // finishes fragment i = wave of a stage whose partial sums are in `p`: four features of the lane's pixel
    auto finish = [&](const v4i* p, const CoopConvStage& st, const CoopConvEpi& e) {
        const int f0 = kq * 16 + wave * 4;
        float cal[16] = {};
        vec4(st.vec0 + 64 + f0, cal, 0);
        v4i sum = *reinterpret_cast<const v4i*>(V + st.vec0 + f0), o[W];
#pragma unroll
        for (int w = 0; w < W; ++w) o[w] = p[(w * N0 + wave) * 64 + lane];
#pragma unroll
        for (int w = 0; w < W; ++w) sum[0] += o[w][0], sum[1] += o[w][1], sum[2] += o[w][2], sum[3] += o[w][3];
        const v4i acc4[4][1] = {{sum}, {none}, {none}, {none}};
        return epilogue_fast16<1, RELU, 4>(e, acc4, 0, cal, cal, cal, none, 16)[0];
    };

    for (int g = g_begin; g < g_end; ++g) {
        // ---------------- stage 0: this wave's tap of all features
        v4i acc0[1][N0];
        const v4i xm = {(int)s0.xor_mask, (int)s0.xor_mask, (int)s0.xor_mask, (int)s0.xor_mask};
        const v4i x = xb ^ xm;
#pragma unroll
        for (int i = 0; i < N0; ++i) acc0[0][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0[i], x, none, 0, 0, 0);
        if (wave < N0) {
            const v4i x8 = xb8 ^ xm;
#pragma unroll
            for (int i = 0; i < N0; ++i)
                if (i == wave) acc0[0][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w8, x8, acc0[0][i], 0, 0, 0);
        }
        mfma_settle(acc0);
#pragma unroll
        for (int i = 0; i < N0; ++i) part[(wave * N0 + i) * 64 + lane] = acc0[0][i];
        const bool more = g + 1 < g_end;
        if (more) request(g + 1, nxt);
        lds_barrier();
        if (wave < N0) {
            const int packed = finish(part, s0, e0);
            if (s0.out && cur.ok) *reinterpret_cast<int*>(s0.out + at(s0, cur, kq) + wave * 4) = packed;
            reinterpret_cast<int*>(mid)[lane * 4 + wave] = flip(packed, s1.xor_mask);
        }
        lds_barrier();

        // ---------------- stage 1: this wave's features
        const int f0 = span1 * 64 + kq * 16 + half * 8;
        v4i acc1[4][1];
        float cal[16] = {}, ecal[16] = {};
#pragma unroll
        for (int d = 0; d < 4; ++d) acc1[d][0] = none;
#pragma unroll
        for (int d = 0; d < F1; ++d) {
            acc1[d][0] = *reinterpret_cast<const v4i*>(V + s1.vec0 + f0 + d * 4);
            vec4(s1.vec0 + 256 + f0 + d * 4, cal, d);
            if constexpr (SUM) vec4(s1.vec0 + 512 + f0 + d * 4, ecal, d);
        }
        const v4i bf1 = mid[lane];
#pragma unroll
        for (int d = 0; d < F1; ++d) acc1[d][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1[d], bf1, acc1[d][0], 0, 0, 0);
        v4i ev4 = none;
        if constexpr (SUM) {
#pragma unroll
            for (int d = 0; d < F1; ++d) ev4[d] = ev[d];
        }
        const v4i packed1 = epilogue_fast16<1, EPI1, 8>(e1, acc1, 0, cal, cal, ecal, ev4, 16);
        if (s1.out && cur.ok)
            *reinterpret_cast<int2*>(s1.out + at(s1, cur, span1 * 4 + kq) + half * 8) = make_int2(packed1[0], packed1[1]);
        if (more) residual(nxt);

        // ---------------- stage 2: the same features as its K
        if constexpr (HAS2) {
            // the other half of the K-step is another wave's: zeros here
            const int lo = flip(packed1[0], s2.xor_mask), hi = flip(packed1[1], s2.xor_mask);
            const v4i bf = half ? v4i{0, 0, lo, hi} : v4i{lo, hi, 0, 0};
            v4i acc2[N0];
#pragma unroll
            for (int i = 0; i < N0; ++i) acc2[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w2[i], bf, none, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < N0; ++i) part2[(wave * N0 + i) * 64 + lane] = acc2[i];
            lds_barrier();
            if (wave < N0) {
                const int packed = finish(part2, s2, e2);
                if (cur.ok) *reinterpret_cast<int*>(s2.out + at(s2, cur, kq) + wave * 4) = packed;
            }
        }
        cur = nxt;
    }
}

template <bool HAS2, bool SUM>
void launch_coop_instance(hipStream_t s, const CoopConvArgs& a, int grid, int lds)
{
    static std::once_flag allowed;
    std::call_once(allowed, [] {
        CHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_coop_kernel<HAS2, SUM>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    });
    hipLaunchKernelGGL((conv_coop_kernel<HAS2, SUM>), dim3(grid), dim3(512), lds, s, a);
}

}  // namespace chip
