// The depthwise chain (conv_dwchain_kernel.h) for small planes: the waves of a workgroup work on ONE granule of 16 pixels.
//
// With one granule per wave a 14x14 layer of batch 32 occupies 104 of 256 CUs, and the granule's whole chain -- six K-steps
// of nine taps, their requantisation, the projection, six spans of the expansion -- is one serial walk of one wave, behind
// a copy of 100 KB of weights into LDS: 12.4 us at batch 1, 13.2 at batch 32, about what three separate launches take.  What
// bounds it is the number of memory round trips in a row, so here
//   - a wave takes the K-steps wave, wave + W, ... of the depthwise stage and multiplies each result with its share of the
//     projection's K at once; the partial sums of the projection (all there is to exchange: 4 KB per wave and 64 features)
//     meet in LDS, every wave finishes a fragment, the packed projection goes back through LDS (1 KB), and every wave
//     computes the spans wave, wave + W, ... of the expansion;
//   - weights are not staged: a wave needs only its own K-steps (5 to 13 KB each) and requests them with its taps, straight into
//     the registers the matrix instructions read; the per-feature vectors (up to 30 KB) go to LDS meanwhile;
//   - the arguments are what the two forms of a MobileNet block need and fit into the scalar registers: the general
//     structures took eight loads in a row, 2.4 us, before the first request went out.
// Kernel time, 14x14, 384 mid features: 12.4 -> 5.9 us at batch 1, 13.2 -> 10.3 at batch 32; and it takes the blocks whose weights
// do not fit into LDS: 14x14, 576 mid features 10.8 -> 7.9 us at batch 1 (the sum of three launches before, without their
// gaps), 7x7, 960 at batch 32 14.2 -> 10.7.
//
// Projection weights are requested when the taps have been multiplied and nothing is fetched for the next granule ahead of
// time: 164 registers (64-feature projection) let a CU hold twelve waves, which is worth more than the look-ahead (221
// registers: 20 us instead of 15 for 28x28 at batch 32).
//
// The depthwise weights are a dword per tap and lane here, the four features of the lane's rows of the diagonal, [K-step][lane
// % 16][12 taps]; a byte permute moves each into its fragment.  Spread out over the lanes they would be 9 KB a
// K-step instead of 768 bytes, and with a granule or two on the chip what one CU fetches is the time (touching the 1x1
// weights' lines early, to have them nearer, made 7x7 blocks slower: 12.4 -> 15.4 us).
#pragma once
#include "conv_dwchain_kernel.h"

namespace chip {

enum { DWCOOP_KS_BYTES = 16 * 12 * 4 };

struct CoopStage {
    int8_t* out;                          // nullptr: the result stays in registers
    int32_t off, pb, pf, py;              // of the output, elements
    int32_t ofm;
    uint32_t xor_mask;
    int32_t unit0, kstride, vec0;         // as ChainStage
};

struct DwCoopArgs {
    const int8_t* in;
    const int8_t* img;                    // diagonal weights, weight units, vectors
    const int8_t* eltw;
    int32_t unit_bytes, vec_bytes;        // where the units and the vectors start
    int32_t vec_quads;
    int32_t el_off, el_pb, el_pf, el_py, el_px;
    uint32_t M;
    int32_t OHW, OW;
    FastDiv div_ohw, div_ow;
    int32_t in_off, in_pb, in_pf, row, col, tap_dy;  // in_off: of tap (0, 0) of output pixel (0, 0); row / col: of one output row / pixel
    int32_t CB, KS, SP2, waves;
    int32_t gpw, grem;                    // granules / workgroups and the remainder
    FastDiv div_parts;
    float clamp_m0, clamp_n0, clamp_m2, clamp_n2, lo1, hi1, conv_lo, conv_hi;
    int32_t eltw_u8;
    CoopStage st[CHAIN_MAX_STAGES];
};

// what the epilogues read of an argument block
struct CoopEpi {
    FastEpi fe;
};

template <int SP1, bool HAS2, bool SUM>
__global__ void __launch_bounds__(512) conv_dwcoop_kernel(DwCoopArgs a)
{
    constexpr int CQ = EPI_KIND_CLAMPQ, EPI1 = SUM ? EPI_KIND_SUMLIN : EPI_KIND_LINEAR;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int W = a.waves;
    const int kq = lane >> 4;
    const int l16 = lane & 15;
    const CoopStage &s0 = a.st[0], &s1 = a.st[1], &s2 = a.st[2];
    CoopEpi e0{}, e1{}, e2{};
    e0.fe.act_m = a.clamp_m0, e0.fe.act_n = a.clamp_n0;
    e2.fe.act_m = a.clamp_m2, e2.fe.act_n = a.clamp_n2;
    e1.fe.lo = e1.fe.lo2 = a.lo1, e1.fe.hi = a.hi1;
    e1.fe.conv_sat = 1, e1.fe.conv_lo = a.conv_lo, e1.fe.conv_hi = a.conv_hi, e1.fe.eltw_u8 = a.eltw_u8;

    extern __shared__ __align__(16) unsigned char smem[];
    v4i* part = reinterpret_cast<v4i*>(smem);          // [wave][SP1 * 4][64]
    v4i* mid = part + W * SP1 * 256;                   // [SP1][64]: the projection as the expansion's B fragments
    v4i* vecs = mid + SP1 * 64;
    const int32_t* V = reinterpret_cast<const int32_t*>(vecs);

    const int per_xcd = gridDim.x >> 3;  // the grid is a multiple of 8
    const uint32_t wg = (blockIdx.x & 7u) * (uint32_t)per_xcd + (blockIdx.x >> 3);
    const int g_begin = (int)(wg * (uint32_t)a.gpw + a.div_parts.div(wg * (uint32_t)a.grem));
    const int g_end = (int)((wg + 1) * (uint32_t)a.gpw + a.div_parts.div((wg + 1) * (uint32_t)a.grem));
    if (g_begin >= g_end) return;  // the whole workgroup

    // everything is addressed as a uniform pointer and a 32-bit lane offset (a pointer per lane costs two registers a load)
    const uint32_t row16 = (uint32_t)(kq * 64 + l16) * 16;
    auto unit = [&](int u, int mt) { return *reinterpret_cast<const v4i*>(a.img + (size_t)(a.unit_bytes + u * 4096 + mt * 256) + row16); };
    v4i xb[9], dw[3], u1[SP1 * 4], u2[SP1 * 4];
    // fragment mt of the diagonal: byte mt of a tap's dword moves to byte l16 % 4 in the lanes of the diagonal, zeros elsewhere
    unsigned sel[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        const int sh = 8 * (l16 & 3);
        sel[mt] = kq == (l16 >> 2) ? (0x0c0c0c0cu & ~(0xffu << sh)) | ((unsigned)mt << sh) : 0x0c0c0c0cu;
    }
    uint32_t boff = 0, b = 0, oy = 0, ox = 0;
    bool ok = false;
    auto locate = [&](int g) {
        const uint32_t m = (uint32_t)g * 16 + l16;
        ok = m < a.M;
        const uint32_t mm = ok ? m : 0;  // pixels past the end read pixel 0
        b = a.div_ohw.div(mm);
        const uint32_t r = mm - b * a.OHW;
        oy = a.div_ow.div(r);
        ox = r - oy * a.OW;
        boff = (uint32_t)(a.in_off + (int)b * a.in_pb + (int)oy * a.row + (int)ox * a.col);
    };
    // The requests stand under conditions; on the other side the registers are declared free, or the compiler keeps the old
    // operands alive to the end of the loop (100 registers spilled with three spans).
    auto forget = [](auto& regs) {
        for (auto& r : regs) asm volatile("" : "=v"(r));
    };
    auto request = [&](int ks, bool real) {
        if (!real) {
            forget(xb), forget(dw);
            return;
        }
        const int slice = ks * 4 + kq;  // a slice past the end reads slice 0, its diagonal weights are zero
        const uint32_t off = boff + (uint32_t)((slice < a.CB ? slice : 0) * a.in_pf);
#pragma unroll
        for (int t = 0; t < 9; ++t) xb[t] = *reinterpret_cast<const v4i*>(a.in + ((t / 3) * a.tap_dy + (t % 3) * 16) + off);
#pragma unroll
        for (int q = 0; q < 3; ++q) dw[q] = *reinterpret_cast<const v4i*>(a.img + ((size_t)ks * DWCOOP_KS_BYTES + q * 16) + (uint32_t)(l16 * 48));
    };
    auto request1 = [&](int ks) {
#pragma unroll
        for (int i = 0; i < SP1 * 4; ++i) u1[i] = unit(s1.unit0 + (i >> 2) * s1.kstride + ks, i & 3);
    };
    auto request2 = [&](int sp, bool real) {
        if (!real) {
            forget(u2);
            return;
        }
#pragma unroll
        for (int i = 0; i < SP1 * 4; ++i) u2[i] = unit(s2.unit0 + sp * s2.kstride + (i >> 2), i & 3);
    };
    auto at = [&](const CoopStage& st) { return (uint32_t)(st.off + (int)b * st.pb + kq * st.pf + (int)oy * st.py + (int)ox * 16); };

    // the vectors are asked for first (their stores to LDS then wait for nothing else), the first K-step behind them
    {
        constexpr int BATCH = 4;
        const int step = W * 64;
        v4i r[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
            r[u] = *reinterpret_cast<const v4i*>(a.img + a.vec_bytes + (uint32_t)min((int)threadIdx.x + u * step, a.vec_quads - 1) * 16u);
        step_fence();
        locate(g_begin);
        request(wave, wave < a.KS);
        step_fence();
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
            if ((int)threadIdx.x + u * step < a.vec_quads) vecs[threadIdx.x + u * step] = r[u];
        for (int i = threadIdx.x + BATCH * step; i < a.vec_quads; i += step)
            vecs[i] = *reinterpret_cast<const v4i*>(a.img + a.vec_bytes + (uint32_t)i * 16u);
    }
    lds_barrier();

    for (int g = g_begin; g < g_end; ++g) {
        int ev_early[SP1];  // the residual of the fragments this wave will finish
        if constexpr (SUM) {
#pragma unroll
            for (int u = 0; u < SP1; ++u) {
                const int i = wave + u * W, sp = i >> 2, mt = i & 3;
                ev_early[u] = 0;
                if (i < SP1 * 4 && sp * 64 + kq * 16 < s1.ofm)
                    ev_early[u] = *reinterpret_cast<const int*>(a.eltw + (uint32_t)(a.el_off + (int)b * a.el_pb + kq * a.el_pf + (int)oy * a.el_py + (int)ox * a.el_px
                                                                                     + sp * 4 * a.el_pf + mt * 4));
            }
        }
        v4i acc1[1][SP1 * 4];
#pragma unroll
        for (int i = 0; i < SP1 * 4; ++i) acc1[0][i] = v4i{0, 0, 0, 0};
        const v4i none = {0, 0, 0, 0};
        for (int ks = wave; ks < a.KS; ks += W) {
            // ---------------- depthwise: 64 features of the granule's pixels
            const int f0 = ks * 64 + kq * 16;
            v4i acc0[4][1];
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) acc0[mt][0] = *reinterpret_cast<const v4i*>(V + s0.vec0 + f0 + mt * 4);
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                const v4i x = xb[t] ^ v4i{(int)s0.xor_mask, (int)s0.xor_mask, (int)s0.xor_mask, (int)s0.xor_mask};
#pragma unroll
                for (int mt = 0; mt < 4; ++mt) {
                    v4i fa = {0, 0, 0, 0};
                    fa[mt] = (int)__builtin_amdgcn_perm(0u, (unsigned)dw[t >> 2][t & 3], sel[mt]);
                    acc0[mt][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa, x, acc0[mt][0], 0, 0, 0);
                }
                step_fence();  // a diagonal fragment is four registers: without it all 36 are made at once
            }
            request1(ks);  // the registers of the taps are free
            step_fence();
            LaneScales sc;
            chain_vec16(V, s0.vec0 + a.KS * 64 + f0, sc.cal);
            chain_vec16(V, s0.vec0 + 3 * a.KS * 64 + f0, sc.wq);
            v4i packed = epilogue_fast16<1, CQ>(e0, acc0, 0, sc.wq, sc.cal, sc.cal, none, 16);
            if (f0 >= s0.ofm) packed = none;
            else if (s0.out && ok) *reinterpret_cast<v4i*>(s0.out + (at(s0) + (uint32_t)(ks * 4 * s0.pf))) = packed;
            // ---------------- its share of the projection
            const v4i bf = packed ^ v4i{(int)s1.xor_mask, (int)s1.xor_mask, (int)s1.xor_mask, (int)s1.xor_mask};
#pragma unroll
            for (int i = 0; i < SP1 * 4; ++i) acc1[0][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(u1[i], bf, acc1[0][i], 0, 0, 0);
            request(ks + W, ks + W < a.KS);
        }
        if constexpr (HAS2)
            request2(wave, wave < a.SP2);  // on its way while the waves exchange
        mfma_settle(acc1);
#pragma unroll
        for (int i = 0; i < SP1 * 4; ++i) part[(wave * SP1 * 4 + i) * 64 + lane] = acc1[0][i];
        lds_barrier();

        // ---------------- projection: fragment i = (span, mt) of the sum, four features of a lane
#pragma unroll
        for (int u = 0; u < SP1; ++u) {  // (at least four waves)
            const int i = wave + u * W;
            if (i >= SP1 * 4) break;
            const int sp = i >> 2, mt = i & 3;
            const int fb = sp * 64 + kq * 16, f0 = fb + mt * 4;
            const uint32_t lane_at = (uint32_t)(sp * 4 * s1.pf + mt * 4);
            v4i ev = {0, 0, 0, 0};
            if constexpr (SUM) ev[0] = ev_early[u];
            float cal[16] = {}, ecal[16] = {};
            auto vec4 = [&](int at, float(&dst)[16]) {
                const v4i q = *reinterpret_cast<const v4i*>(V + at);
                dst[0] = __int_as_float(q[0]), dst[1] = __int_as_float(q[1]), dst[2] = __int_as_float(q[2]), dst[3] = __int_as_float(q[3]);
            };
            vec4(s1.vec0 + SP1 * 64 + f0, cal);
            if constexpr (SUM) vec4(s1.vec0 + 2 * SP1 * 64 + f0, ecal);
            v4i sum = *reinterpret_cast<const v4i*>(V + s1.vec0 + f0);
            for (int w = 0; w < W; ++w) {
                const v4i o = part[(w * SP1 * 4 + i) * 64 + lane];
                sum[0] += o[0], sum[1] += o[1], sum[2] += o[2], sum[3] += o[3];
            }
            const v4i acc4[4][1] = {{sum}, {none}, {none}, {none}};
            int packed = epilogue_fast16<1, EPI1>(e1, acc4, 0, cal, cal, ecal, ev, s1.ofm - f0)[0];
            if (fb >= s1.ofm) packed = 0;
            else if (s1.out && ok) *reinterpret_cast<int*>(s1.out + (at(s1) + lane_at)) = packed;
            if constexpr (HAS2) reinterpret_cast<int*>(mid)[(sp * 64 + lane) * 4 + mt] = packed;
        }
        lds_barrier();

        // ---------------- expansion, span by span
        if constexpr (HAS2) {
            v4i bf[SP1];
#pragma unroll
            for (int sp = 0; sp < SP1; ++sp) bf[sp] = mid[sp * 64 + lane] ^ v4i{(int)s2.xor_mask, (int)s2.xor_mask, (int)s2.xor_mask, (int)s2.xor_mask};
            for (int sp = wave; sp < a.SP2; sp += W) {
                const int f0 = sp * 64 + kq * 16;
                v4i acc2[4][1];
#pragma unroll
                for (int mt = 0; mt < 4; ++mt) acc2[mt][0] = *reinterpret_cast<const v4i*>(V + s2.vec0 + f0 + mt * 4);
#pragma unroll
                for (int i = 0; i < SP1 * 4; ++i) acc2[i & 3][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(u2[i], bf[i >> 2], acc2[i & 3][0], 0, 0, 0);
                request2(sp + W, sp + W < a.SP2);
                LaneScales sc;
                chain_vec16(V, s2.vec0 + a.SP2 * 64 + f0, sc.cal);
                chain_vec16(V, s2.vec0 + 3 * a.SP2 * 64 + f0, sc.wq);
                const v4i packed = epilogue_fast16<1, CQ>(e2, acc2, 0, sc.wq, sc.cal, sc.cal, none, s2.ofm - f0);
                if (f0 < s2.ofm && ok) *reinterpret_cast<v4i*>(s2.out + (at(s2) + (uint32_t)(sp * 4 * s2.pf))) = packed;
            }
        }
        const bool more = g + 1 < g_end;
        if (more) locate(g + 1);
        request(wave, more && wave < a.KS);
    }
}

template <int SP1, bool HAS2, bool SUM>
void launch_dwcoop_instance(hipStream_t s, const DwCoopArgs& a, int grid, int lds)
{
    static std::once_flag allowed;
    std::call_once(allowed, [] {
        CHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_dwcoop_kernel<SP1, HAS2, SUM>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    });
    hipLaunchKernelGGL((conv_dwcoop_kernel<SP1, HAS2, SUM>), dim3(grid), dim3(64 * a.waves), lds, s, a);
}

}  // namespace chip
