// The depthwise chain (conv_dwchain_kernel.h) for small planes: the waves of a workgroup work on ONE granule of 16 pixels.
//
// With one granule per wave a 14x14 layer of batch 32 occupies 104 of 256 CUs, and the granule's whole chain is one serial
// walk of one wave behind a copy of 100 KB of weights into LDS.  What bounds a small plane is the number of memory round
// trips in a row and the bytes one CU has to pull, so here a granule costs three of them whatever its features:
//   - depthwise: a wave takes one K-step of the projection, i.e. 64 mid features in two units of 32 (two taps to a
//     product, conv_dwchain_kernel.h), and leaves the packed result (1 KB, a B fragment) in LDS;
//   - projection: a wave takes one fragment of 16 features over ALL K-steps, so no partial sums are exchanged (they
//     would be W x 32 bytes a feature and pixel; the packed depthwise results are 64 bytes a pixel and K-step);
//   - expansion: a wave takes the spans wave, wave + W, ... of 64 features.
// Weights are not staged: a wave requests its own, straight into the registers the matrix instructions read, as soon as the
// registers of the operands before them are free.  Its per-feature vectors lie side by side in memory (the host's image),
// come in with two loads, and are spread to the lanes through a corner of LDS that no other wave touches: the
// first barrier of a granule is the one in front of the projection.
// Where granules are so few that CUs idle, `parts` workgroups repeat the depthwise stage and the projection of a granule and
// share the spans of its expansion: at 7x7, batch 1 (four granules, 960-160-960) a CU pulls 240 KB instead of 340.  Where they
// are more than the workgroups a device holds, a workgroup takes two and fetches the weights once.
// The bound is the launch (2.5 us) and the round trips; at two granules a CU also the bytes through its L1 (64 a clock).
// Kernel time in a network, before (a wave walked over two K-steps of 64 with one tap a product, partial sums of the projection
// went through LDS) and now: 14x14, 384-64-384 6.5 -> 5.6 us at batch 1, 11.1 -> 6.9 at batch 32; 576-96-576 9.2 -> 6.4 and 15.5 ->
// 10.6; 7x7, 960-160-960 11.8 -> 8.4 and 11.8 -> 8.6.
// A wave is alone on its SIMD at batch 1, and an instruction of its is 3 to 4 ns: of 3.9 us (384-64-384) 0.2 are the arguments, 0.5 the
// way to the last request, 0.4 the taps on their way, 0.4 the depthwise products, 0.55 their requantisation, 0.5 projection and barriers,
// 0.9 its requantisation and the expansion.  Words of the later weights asked for ahead, so that they come from L2, cost as much
// of L1's time as the weights themselves (960-160-960 7.7 -> 9.4).
#pragma once
#include "conv_dwchain_kernel.h"

namespace chip {

enum { DWCOOP_UNIT_BYTES = 512,    // depthwise weights of 32 features: [tap half][16 rows][16 bytes]
       DWCOOP_VEC0_BYTES = 768,    // vectors of a K-step / a span: start values, calibration, dequantisation factors, 64 each
       DWCOOP_VEC1_BYTES = 192,    // of a projection fragment: start values, calibration, factors of the sum, 16 each
       DWCOOP_OWN = 48 + 12 + 48,  // 16-byte pieces of a wave's corner of LDS
       DWCOOP_MAX_WAVES = 16 };

struct CoopStage {
    int8_t* out;                          // nullptr: the result stays in registers
    int32_t off, pb, pf, py;              // of the output, elements
    int32_t ofm;
    uint32_t xor_mask;
};

struct DwCoopArgs {
    const int8_t* in;
    const int8_t* img;                    // depthwise weights [unit], fragments of the projection [K-step][fragment], of the expansion [K-step][unit][2], vectors
    const int8_t* eltw;
    int32_t w1, w2, v0, v1, v2;           // where the parts of the image start, bytes
    int32_t el_off, el_pb, el_pf, el_py, el_px;
    uint32_t M;
    int32_t OHW, OW;
    FastDiv div_ohw, div_ow;
    int32_t in_off, in_pb, in_pf, row, col, tap_dy;  // in_off: of tap (0, 0) of output pixel (0, 0); row / col: of one output row / pixel
    int32_t CB, KS, F1, SP2, waves, parts;           // input slices, K-steps, fragments of the projection, spans of the expansion
    FastDiv div_parts;
    float clamp_m0, clamp_n0, clamp_m2, clamp_n2, lo1, hi1, conv_lo, conv_hi;
    int32_t eltw_u8;
    CoopStage st[CHAIN_MAX_STAGES];
};

// what the epilogues read of an argument block
struct CoopEpi {
    FastEpi fe;
};

// All arguments behind one wait: fetched where they are first used they were four trips to memory in a row.
__device__ __forceinline__ void fetch_arguments(const DwCoopArgs& a)
{
    asm volatile("" ::"s"(a.in), "s"(a.img), "s"(a.eltw), "s"(a.w1), "s"(a.w2), "s"(a.v0), "s"(a.v1), "s"(a.v2), "s"(a.el_off), "s"(a.el_pb), "s"(a.el_pf), "s"(a.el_py), "s"(a.el_px),
                 "s"(a.M), "s"(a.OHW), "s"(a.OW), "s"(a.div_ohw.mul), "s"(a.div_ohw.shift), "s"(a.div_ow.mul), "s"(a.div_ow.shift), "s"(a.in_off), "s"(a.in_pb), "s"(a.in_pf), "s"(a.row),
                 "s"(a.col), "s"(a.tap_dy));
    asm volatile("" ::"s"(a.CB), "s"(a.KS), "s"(a.F1), "s"(a.SP2), "s"(a.waves), "s"(a.parts), "s"(a.div_parts.mul), "s"(a.div_parts.shift), "s"(a.clamp_m0), "s"(a.clamp_n0),
                 "s"(a.clamp_m2), "s"(a.clamp_n2), "s"(a.lo1), "s"(a.hi1), "s"(a.conv_lo), "s"(a.conv_hi), "s"(a.eltw_u8), "s"(gridDim.x));
#pragma unroll
    for (int k = 0; k < CHAIN_MAX_STAGES; ++k)
        asm volatile("" ::"s"(a.st[k].out), "s"(a.st[k].off), "s"(a.st[k].pb), "s"(a.st[k].pf), "s"(a.st[k].py), "s"(a.st[k].ofm), "s"(a.st[k].xor_mask));
}

// K1: K-steps of the expansion.  KM: K-steps of the projection that a wave has registers for.  DEEP: there are more of them, or more
// than waves: both are walked in rounds.  NG: granules of a workgroup (at most ten waves with two).
template <int K1, int KM, bool DEEP, int NG, bool HAS2, bool SUM>
__global__ void __launch_bounds__(NG > 1 ? 640 : 64 * DWCOOP_MAX_WAVES, NG > 1 ? 3 : 4) conv_dwcoop_kernel(DwCoopArgs a)
{
    constexpr int CQ = EPI_KIND_CLAMPQ, EPI1 = SUM ? EPI_KIND_SUMLIN : EPI_KIND_LINEAR, S = DWCHAIN_STEPS;
    // the expansion's weights fit into the registers of the taps beside the projection's: both are requested together
    constexpr bool BOTH = HAS2 && !DEEP && NG == 1 && KM + 4 * K1 <= 17;
    fetch_arguments(a);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int W = a.waves;
    const int kq = lane >> 4;
    const int l16 = lane & 15;
    const int lf = 16 * (kq & 1) + 8 * (kq >> 1);  // the lane's first feature in a unit
    const CoopStage &s0 = a.st[0], &s1 = a.st[1], &s2 = a.st[2];
    CoopEpi e0{}, e1{}, e2{};
    e0.fe.act_m = a.clamp_m0, e0.fe.act_n = a.clamp_n0;
    e2.fe.act_m = a.clamp_m2, e2.fe.act_n = a.clamp_n2;
    e1.fe.lo = e1.fe.lo2 = a.lo1, e1.fe.hi = a.hi1;
    e1.fe.conv_sat = 1, e1.fe.conv_lo = a.conv_lo, e1.fe.conv_hi = a.conv_hi, e1.fe.eltw_u8 = a.eltw_u8;

    extern __shared__ __align__(16) unsigned char smem[];
    v4i* mid0 = reinterpret_cast<v4i*>(smem);  // [granule][KS][64]: the depthwise result as the projection's B fragments
    v4i* mid1 = mid0 + NG * a.KS * 64;         // [granule][K1][64]: the projection as the expansion's
    v4i* own = mid1 + NG * K1 * 64 + wave * DWCOOP_OWN;
    const int32_t* V0 = reinterpret_cast<const int32_t*>(own);
    const int32_t* V1 = V0 + 48 * 4;
    const int32_t* V2 = V1 + 12 * 4;

    // workgroups of one granule have neighbouring numbers, i.e. sit on one die (the grid is a multiple of 8)
    const uint32_t wg = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const uint32_t group = a.div_parts.div(wg);
    const int part = (int)(wg - group * (uint32_t)a.parts);
    if (group * (16 * NG) >= a.M) return;  // the whole workgroup

    // the lane's pixels; pixels past the end read pixel 0
    struct Pos {
        uint32_t b, oy, ox;
        bool ok;
    } pos[NG];
#pragma unroll
    for (int n = 0; n < NG; ++n) {
        const uint32_t m = (group * NG + n) * 16 + l16;
        pos[n].ok = m < a.M;
        const uint32_t mm = pos[n].ok ? m : 0;
        pos[n].b = a.div_ohw.div(mm);
        const uint32_t r = mm - pos[n].b * a.OHW;
        pos[n].oy = a.div_ow.div(r), pos[n].ox = r - pos[n].oy * a.OW;
    }
    auto at = [&](const CoopStage& st, const Pos& p, int slice) {
        return (uint32_t)(st.off + (int)p.b * st.pb + slice * st.pf + (int)p.oy * st.py + (int)p.ox * 16 + 8 * (kq >> 1));
    };

    // everything is addressed as a uniform pointer and a 32-bit lane offset (a pointer per lane costs two registers a load)
    v4i xb[NG][2][S], dw[2], u1[KM], u2[HAS2 ? 4 * K1 : 1];
    auto request0 = [&](int ks) {
#pragma unroll
        for (int h = 0; h < 2; ++h) dw[h] = *reinterpret_cast<const v4i*>(a.img + (size_t)(ks * 2 + h) * DWCOOP_UNIT_BYTES + (uint32_t)(((lane >> 5) * 16 + l16) * 16));
#pragma unroll
        for (int n = 0; n < NG; ++n) {
            const uint32_t boff = (uint32_t)(a.in_off + (int)pos[n].b * a.in_pb + (int)pos[n].oy * a.row + (int)pos[n].ox * a.col);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // a slice past the end reads the last one, its weights are zero
                const uint32_t off = boff + (uint32_t)(min(2 * (2 * ks + h) + (kq & 1), a.CB - 1) * a.in_pf);
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    // the lane's tap in step s; the tenth tap has no weight and reads the ninth
                    const int tap = min(2 * s + (kq >> 1), 8), ty = (tap * 11) >> 5;
                    xb[n][h][s] = *reinterpret_cast<const v4i*>(a.in + (off + (uint32_t)(ty * a.tap_dy + (tap - ty * 3) * 16)));
                }
            }
        }
    };
    auto request1 = [&](int k0, int f) {
#pragma unroll
        for (int k = 0; k < KM; ++k) u1[k] = *reinterpret_cast<const v4i*>(a.img + (size_t)(a.w1 + (min(k0 + k, a.KS - 1) * a.F1 + f) * 1024) + (uint32_t)(lane * 16));
    };
    auto request2 = [&](int sp) {
        if constexpr (HAS2) {
#pragma unroll
            for (int k = 0; k < K1; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i) u2[k * 4 + i] = *reinterpret_cast<const v4i*>(a.img + (size_t)(a.w2 + ((k * a.SP2 + sp) * 4 + i) * 1024) + (uint32_t)(lane * 16));
        }
    };
    // The requests stand under conditions; on the other side the registers are declared free, or the compiler keeps the old
    // operands alive.
    auto forget = [](auto& regs) {
        for (auto& r : regs) asm volatile("" : "=v"(r));
    };
    const int sp_first = part + a.parts * wave, sp_step = a.parts * W;
    auto load_vec0 = [&](int ks, int f) {  // a K-step's vectors and a fragment's behind them
        const int off = lane < 48 ? a.v0 + ks * DWCOOP_VEC0_BYTES + lane * 16 : a.v1 + f * DWCOOP_VEC1_BYTES + (min(lane, 59) - 48) * 16;
        return *reinterpret_cast<const v4i*>(a.img + (uint32_t)off);
    };
    auto load_vec2 = [&](int sp) { return *reinterpret_cast<const v4i*>(a.img + (uint32_t)(a.v2 + sp * DWCOOP_VEC0_BYTES + min(lane, 47) * 16)); };
    auto vec4 = [](const int32_t* v, float(&dst)[16], int d) {
        const v4i q = *reinterpret_cast<const v4i*>(v);
        dst[d * 4 + 0] = __int_as_float(q[0]), dst[d * 4 + 1] = __int_as_float(q[1]), dst[d * 4 + 2] = __int_as_float(q[2]), dst[d * 4 + 3] = __int_as_float(q[3]);
    };
    const v4i none = {0, 0, 0, 0};
    // the lane's eight features of unit h of a K-step or span, requantised
    auto finish8 = [&](const CoopEpi& e, const int32_t* V, const v4i& lo, const v4i& hi, int h) {
        float cal[16] = {}, wq[16] = {};
        vec4(V + 64 + h * 32 + lf, cal, 0), vec4(V + 64 + h * 32 + lf + 4, cal, 1);
        vec4(V + 128 + h * 32 + lf, wq, 0), vec4(V + 128 + h * 32 + lf + 4, wq, 1);
        const v4i acc4[4][1] = {{lo}, {hi}, {none}, {none}};
        const v4i p = epilogue_fast16<1, CQ, 8>(e, acc4, 0, wq, cal, cal, none, 16);
        return make_int2(p[0], p[1]);
    };
    const bool works0 = wave < a.KS, works1 = wave < a.F1;

    // the vectors are asked for first: their way through LDS is over when the taps arrive
    v4i vec = load_vec0(min(wave, a.KS - 1), min(wave, a.F1 - 1));
    step_fence();
    if (works0) {
        request0(wave);
    } else {
        forget(dw);
#pragma unroll
        for (int n = 0; n < NG; ++n) forget(xb[n][0]), forget(xb[n][1]);
    }
    int ev[NG] = {};
    if constexpr (SUM) {
        const int slice = 2 * (wave >> 1) + (kq & 1);
        if (slice * 16 < s1.ofm)
#pragma unroll
            for (int n = 0; n < NG; ++n)
                ev[n] = *reinterpret_cast<const int*>(a.eltw + (uint32_t)(a.el_off + (int)pos[n].b * a.el_pb + slice * a.el_pf + (int)pos[n].oy * a.el_py
                                                                         + (int)pos[n].ox * a.el_px + 8 * (kq >> 1) + 4 * (wave & 1)));
    }
    step_fence();
    if (lane < 60) own[lane] = vec;
    if constexpr (HAS2) vec = load_vec2(min(sp_first, a.SP2 - 1));

    // ---------------- depthwise: 64 features of the granule's pixels
    // byte 2 (s % 2) + mt of the row's weights goes to byte l16 % 4 of dword 2 h + mt, h = l16 / 8, in the lanes of the row's slice
    unsigned sel[2][2][2];  // [s % 2][mt][h]
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int sh = 8 * (l16 & 3);
                const bool mine = (kq & 1) == ((l16 >> 2) & 1) && h == (l16 >> 3);
                sel[e][mt][h] = mine ? (0x0c0c0c0cu & ~(0xffu << sh)) | ((unsigned)(2 * e + mt) << sh) : 0x0c0c0c0cu;
            }
    v4i acc0[NG * 4][1];
    auto depthwise = [&] {
        // (the last word of a unit's weights is not read below: were it free to be overwritten, whatever does so would wait for
        // the weights, in front of the requests for the taps)
        asm volatile("" ::"v"(dw[0]), "v"(dw[1]));
#pragma unroll
        for (int n = 0; n < NG; ++n)
#pragma unroll
            for (int d = 0; d < 4; ++d) acc0[n * 4 + d][0] = *reinterpret_cast<const v4i*>(V0 + (d >> 1) * 32 + lf + (d & 1) * 4);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int s = 0; s < S; ++s) {
                v4i x[NG];
#pragma unroll
                for (int n = 0; n < NG; ++n) x[n] = xb[n][h][s] ^ v4i{(int)s0.xor_mask, (int)s0.xor_mask, (int)s0.xor_mask, (int)s0.xor_mask};
#pragma unroll
                for (int mt = 0; mt < 2; ++mt) {
                    v4i fa = {0, 0, 0, 0};
#pragma unroll
                    for (int hh = 0; hh < 2; ++hh) fa[2 * hh + mt] = (int)__builtin_amdgcn_perm(0u, (unsigned)dw[h][s >> 1], sel[s & 1][mt][hh]);
#pragma unroll
                    for (int n = 0; n < NG; ++n) {
                        v4i& acc = acc0[n * 4 + 2 * h + mt][0];
                        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa, x[n], acc, 0, 0, 0);
                    }
                }
                step_fence();
            }
        mfma_settle(acc0);
    };
    auto finish0 = [&](int ks) {
#pragma unroll
        for (int n = 0; n < NG; ++n) {
            int2 q[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                q[h] = finish8(e0, V0, acc0[n * 4 + 2 * h][0], acc0[n * 4 + 2 * h + 1][0], h);
                const int slice = 2 * (2 * ks + h) + (kq & 1);
                if (s0.out && pos[n].ok && part == 0 && slice < a.CB) *reinterpret_cast<int2*>(s0.out + at(s0, pos[n], slice)) = q[h];
            }
            // (features that do not exist meet weights that are zero)
            const int x = (int)s1.xor_mask;
            mid0[(n * a.KS + ks) * 64 + lane] = v4i{q[0].x ^ x, q[0].y ^ x, q[1].x ^ x, q[1].y ^ x};
        }
    };
    if constexpr (DEEP) {
        for (int ks = wave; ks < a.KS; ks += W) {
            if (ks != wave) {
                request0(ks);
                const v4i v = load_vec0(ks, 0);
                if (lane < 48) own[lane] = v;
            }
            depthwise();
            finish0(ks);
        }
        request1(0, min(wave, a.F1 - 1));
    } else {
        if (works0) depthwise();
        else forget(reinterpret_cast<v4i(&)[NG * 4]>(acc0));
        if constexpr (BOTH)
            if (lane < 48) own[60 + lane] = vec;
        if (works1) request1(0, wave);  // the registers of the taps are free
        else forget(u1);
        if constexpr (BOTH) {
            if (sp_first < a.SP2) request2(sp_first);
            else forget(u2);
        }
        step_fence();
        if (works0) finish0(wave);
    }
    lds_barrier();

    // ---------------- projection: the wave's fragment, four features of a lane
    v4i acc1[2 * NG][1];  // two chains of dependent products to a granule
#pragma unroll
    for (int i = 0; i < 2 * NG; ++i) acc1[i][0] = none;
    if (works1) {
#pragma unroll
        for (int n = 0; n < NG; ++n) acc1[2 * n][0] = *reinterpret_cast<const v4i*>(V1 + kq * 4);
        for (int k0 = 0; k0 < a.KS; k0 += KM) {
            if (DEEP && k0) request1(k0, wave);
#pragma unroll
            for (int k = 0; k < KM; ++k)
                if (k0 + k < a.KS)
#pragma unroll
                    for (int n = 0; n < NG; ++n) {
                        v4i& acc = acc1[2 * n + (k & 1)][0];
                        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(u1[k], mid0[(n * a.KS + k0 + k) * 64 + lane], acc, 0, 0, 0);
                    }
            if (!DEEP) break;
        }
        mfma_settle(acc1);
    }
    if constexpr (HAS2 && !BOTH) {
        if (sp_first < a.SP2) request2(sp_first);
        else forget(u2);
        if (lane < 48) own[60 + lane] = vec;
        step_fence();
    }
    if (works1) {
        float cal[16] = {}, ecal[16] = {};
        vec4(V1 + 16 + kq * 4, cal, 0);
        if constexpr (SUM) vec4(V1 + 32 + kq * 4, ecal, 0);
        const int unit = wave >> 1, slice = 2 * unit + (kq & 1), f0 = unit * 32 + lf + 4 * (wave & 1);
#pragma unroll
        for (int n = 0; n < NG; ++n) {
            const v4i ev4 = {ev[n], 0, 0, 0}, acc4[4][1] = {{acc1[2 * n][0] + acc1[2 * n + 1][0]}, {none}, {none}, {none}};
            int packed = epilogue_fast16<1, EPI1>(e1, acc4, 0, cal, cal, ecal, ev4, s1.ofm - f0)[0];
            if (slice * 16 >= s1.ofm) packed = 0;
            else if (s1.out && pos[n].ok && part == 0) *reinterpret_cast<int*>(s1.out + at(s1, pos[n], slice) + 4 * (wave & 1)) = packed;
            if constexpr (HAS2) reinterpret_cast<int*>(mid1)[((n * K1 + (unit >> 1)) * 64 + lane) * 4 + 2 * (unit & 1) + (wave & 1)] = packed ^ (int)s2.xor_mask;
        }
    }

    // ---------------- expansion, span by span
    if constexpr (HAS2) {
        lds_barrier();
        for (int sp = sp_first; sp < a.SP2; sp += sp_step) {
            if (sp != sp_first) {
                request2(sp);
                const v4i v = load_vec2(sp);
                if (lane < 48) own[60 + lane] = v;
            }
#pragma unroll
            for (int n = 0; n < NG; ++n) {
                v4i acc2[4][1];
#pragma unroll
                for (int d = 0; d < 4; ++d) acc2[d][0] = *reinterpret_cast<const v4i*>(V2 + (d >> 1) * 32 + lf + (d & 1) * 4);
#pragma unroll
                for (int k = 0; k < K1; ++k) {
                    const v4i bf = mid1[(n * K1 + k) * 64 + lane];
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc2[i][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(u2[k * 4 + i], bf, acc2[i][0], 0, 0, 0);
                }
                mfma_settle(acc2);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    int2 q = finish8(e2, V2, acc2[2 * h][0], acc2[2 * h + 1][0], h);
                    const int slice = 2 * (2 * sp + h) + (kq & 1);
                    if (s2.ofm & 15) {  // a partly filled last slice: its padding features stay zero
                        keep_branch();
                        v4i half = {q.x, q.y, 0, 0};
                        zero_padding_features(half, s2.ofm - (sp * 64 + h * 32 + lf));
                        q = make_int2(half[0], half[1]);
                    }
                    if (pos[n].ok && slice * 16 < s2.ofm) *reinterpret_cast<int2*>(s2.out + at(s2, pos[n], slice)) = q;
                }
            }
        }
    }
}

template <int K1, int KM, bool DEEP, int NG, bool HAS2, bool SUM>
void launch_dwcoop_instance(hipStream_t s, const DwCoopArgs& a, int grid, int lds)
{
    static std::once_flag allowed;
    std::call_once(allowed, [] {
        CHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_dwcoop_kernel<K1, KM, DEEP, NG, HAS2, SUM>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    });
    hipLaunchKernelGGL((conv_dwcoop_kernel<K1, KM, DEEP, NG, HAS2, SUM>), dim3(grid), dim3(64 * a.waves), lds, s, a);
}

}  // namespace chip
