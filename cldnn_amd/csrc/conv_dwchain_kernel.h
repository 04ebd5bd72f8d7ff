// A depthwise 3x3 convolution and the one or two 1x1 convolutions behind it in ONE launch: the tail of a MobileNet
// block and the head of the next one,
//     depthwise 3x3 (mid -> mid)  ->  1x1 projection (mid -> few)  ->  1x1 expansion of the next block (few -> 6 few).
// The depthwise result (as large as the expanded tensor it reads) and the projection's input never touch memory.
//
// What bounds these layers is the vector ALU: the requantisation of three tensors.  So the depthwise stage runs on the
// matrix cores, and everything is laid out in units of 32 features, not the dense kernels' spans of 64: a unit costs a lane
// eight values, and 16, 24, 32, 96 or 144 features fill 1, 1, 1, 3 and 5 of them (in spans of 64 they are 64, 64, 64, 128
// and 192 features' work).
//
// A unit is two slices of 16 features and two fragments of a v_mfma_i32_16x16x64_i8.  Row (q, i) of fragment mt stands for
// feature 16 (q % 2) + 8 (q / 2) + 4 mt + i of the unit, so lane (q, l16) ends with eight consecutive features of its pixel:
// half q / 2 of slice q % 2.  Two units side by side are the 64 values of a K-step of the next stage (lane q: eight bytes of
// the first, eight of the second; the host lays its weights out for that order; an absent second unit is zeros).
//
// Depthwise: the 64 values a product sums over are the unit's two slices at TWO taps (lane q: slice q % 2, tap 2 s + q / 2),
// so nine taps are five products per fragment.  The weight operand has one byte per row and tap that is not zero; a lane
// reads the ten bytes of its row (a 16-byte piece, 1 KB per unit in LDS) and a byte permute puts each in its place.
//
// Work split as in the dense chain: persistent workgroups of four independent waves, granules of 16 pixels, the
// activations of the next unit (also across granules) requested while the present one is multiplied, all weights and
// per-feature vectors in LDS.  On large planes the vector ALU is the bound: it issues in 80 to 92 % of the time (112x112 and 56x56, batch 32;
// 46 to 50 % at 28x28, where a wave has one granule).
// MobileNet v2 at batch 32, kernel time before (spans of 64, one tap per product) and now: 112x112 32-16-96 47.1 -> 30.0 us,
// 112x112 96-24-144 25.1 -> 18.1, 56x56 144-24-144 31.4 -> 22.1, 28x28 192-32-192 13.0 -> 9.8; with the first granule's requests out
// while the image is on its way to LDS 27.3, 16.9, 19.7 and 9.1.  The waves of a workgroup take its granules in turn, so that rows that
// share filter taps are read at about the same time: nothing at batch 32, at batch 100 48.8 -> 44.5, 47.7 -> 45.4, 22.0 -> 20.4 us.
#pragma once
#include <type_traits>

#include "conv_chain_kernel.h"

namespace chip {

enum { DWCHAIN_STEPS = 5 };  // pairs of taps

struct DwChainArgs {
    const int8_t* in;
    const v4i* img;            // LDS image: depthwise weights [U0][64], fragments of stage 1 [KS][P1][2], of stage 2 [U2][2], vectors
    int32_t quads;             // its 16-byte pieces
    int32_t w1, w2, vec;       // where the fragments and the vectors start, in pieces
    int32_t gpw, grem;         // granules / workgroups and the remainder
    FastDiv div_wgs;           // workgroup w starts at granule w * gpw + (w * grem) / workgroups = floor(w * granules / workgroups)
    uint32_t M;
    int32_t OHW, OW;
    FastDiv div_ohw, div_ow;
    int32_t in_off, in_pb, in_pf, row, col, tap_dy;  // bytes; in_off: of tap (0, 0) of output pixel (0, 0); row / col: of one output row / pixel
    int32_t CB, U0, KS, U2;    // slices and units of the depthwise stage, K-steps of stage 1, units of stage 2 (0: two stages)
    int32_t n0, n1, n2;        // entries of the stages' vectors
    ChainStage st[CHAIN_MAX_STAGES];
};

// P1: units of the projection.  FLIP: some stage reads u8 (see the dense kernels' xor).  EPI0 / EPI1 / EPI2: epilogue kinds of
// the three stages, fixed at compile time where the stages have one of the branch-free forms (a MobileNet block: CLAMPQ,
// LINEAR, CLAMPQ), else the run-time form FAST for all of them
template <int P1, bool HAS2, bool FLIP, int EPI0, int EPI1, int EPI2>
__global__ void __launch_bounds__(256, EPI0 == EPI_KIND_FAST ? 2 : (P1 == 1 ? 4 : 3)) conv_dwchain_kernel(DwChainArgs a)
{
    constexpr int S = DWCHAIN_STEPS;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int kq = lane >> 4;
    const int l16 = lane & 15;
    const ChainStage& s0 = a.st[0];
    const ChainStage& s1 = a.st[1];
    const ChainStage& s2 = a.st[2];

    extern __shared__ __align__(16) unsigned char smem[];
    v4i* lds = reinterpret_cast<v4i*>(smem);
    const int32_t* V = reinterpret_cast<const int32_t*>(lds + a.vec);
    // the image's way into LDS; the last pieces wait in registers until the first granule's requests have gone out
    constexpr int BATCH = 8;
    v4i copy[BATCH];
    auto request_image = [&](int i) {
#pragma unroll
        for (int u = 0; u < BATCH; ++u) copy[u] = a.img[min(i + u * 256, a.quads - 1)];
    };
    auto store_image = [&](int i) {
#pragma unroll
        for (int u = 0; u < BATCH; ++u)
            if (i + u * 256 < a.quads) lds[i + u * 256] = copy[u];
    };
    int copied = t;
    for (; copied + BATCH * 256 < a.quads; copied += BATCH * 256) {
        request_image(copied);
        store_image(copied);
    }
    request_image(copied);
    step_fence();

    const int per_xcd = gridDim.x >> 3;  // the grid is a multiple of 8
    const uint32_t vb = (blockIdx.x & 7u) * (uint32_t)per_xcd + (blockIdx.x >> 3);
    // the workgroup's range, which its waves take in turn: rows that share filter taps are read at about the same time
    const int g_begin = (int)(vb * (uint32_t)a.gpw + a.div_wgs.div(vb * (uint32_t)a.grem)) + wave;
    const int g_end = (int)((vb + 1) * (uint32_t)a.gpw + a.div_wgs.div((vb + 1) * (uint32_t)a.grem));
    if (g_begin >= g_end) {
        store_image(copied);
        __syncthreads();
        return;
    }

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
    uint32_t tap_off[S];  // of the lane's tap in step s; the tenth tap has no weight and reads the ninth
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int tap = min(2 * s + (kq >> 1), 8), ty = (tap * 11) >> 5;
        tap_off[s] = (uint32_t)(ty * a.tap_dy + (tap - ty * 3) * 16);
    }

    struct Refs {
        uint32_t boff;  // byte offset of the lane's pixel at tap (0, 0), slice 0
        int o0, o1, e1, o2;
    };
    auto setup = [&](int g, Refs& r) {
        const uint32_t m = (uint32_t)g * 16 + l16;
        const bool ok = g < g_end && m < a.M;
        const uint32_t mm = ok ? m : 0;
        const uint32_t b = a.div_ohw.div(mm);
        const uint32_t rr = mm - b * a.OHW;
        const uint32_t oy = a.div_ow.div(rr), ox = rr - oy * a.OW;
        r.boff = (uint32_t)(a.in_off + (int)b * a.in_pb + (int)oy * a.row + (int)ox * a.col);
        auto at = [&](const ChainStage& st) {
            return st.out_off + (int)b * st.out_pb + (kq & 1) * st.out_pf + (int)oy * st.out_py + (int)ox * 16 + (kq >> 1) * 8;
        };
        r.o0 = ok && s0.out ? at(s0) : -1;
        r.o1 = ok && s1.out ? at(s1) : -1;
        r.o2 = HAS2 && ok && s2.out ? at(s2) : -1;
        r.e1 = s1.el_off + (int)b * s1.el_pb + (kq & 1) * s1.el_pf + (int)oy * s1.el_py + (int)ox * s1.el_px + (kq >> 1) * 8;
    };
    v4i rb[S];
    auto load_step = [&](const Refs& r, uint32_t slice_off, int s) { rb[s] = *reinterpret_cast<const v4i*>(a.in + (r.boff + (slice_off + tap_off[s]))); };
    // a slice past the end (an odd number of them) reads the last one, its weights are zero
    auto slice_of = [&](int u) { return (uint32_t)(min(2 * u + (kq & 1), a.CB - 1) * a.in_pf); };
    auto flip = [](const v4i& v, uint32_t mask) {
        if constexpr (!FLIP) return v;
        else return v ^ v4i{(int)mask, (int)mask, (int)mask, (int)mask};
    };
    auto flip2 = [](const int2& v, uint32_t mask) {
        if constexpr (!FLIP) return v;
        else return make_int2(v.x ^ (int)mask, v.y ^ (int)mask);
    };
    auto fragment = [&](int i) { return lds[i * 64 + lane]; };
    // the lane's eight values of a vector
    auto vec8 = [&](int at, float(&dst)[16]) {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const v4i q = *reinterpret_cast<const v4i*>(V + at + d * 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[d * 4 + i] = __int_as_float(q[i]);
        }
    };
    // eight features of the lane's pixel: f0 is the first, `valid` of them exist
    auto finish = [&](auto kind, const ChainStage& st, int n, int f0, const v4i(&acc)[2], const int2& ev, int valid) {
        constexpr int EPI = decltype(kind)::value;
        float cal[16], ecal[16] = {}, wq[16] = {};
        vec8(st.vec0 + n + f0, cal);
        if constexpr (EPI == EPI_KIND_FUSED || EPI == EPI_KIND_SUMLIN || EPI == EPI_KIND_FAST) vec8(st.vec0 + 2 * n + f0, ecal);
        if constexpr (EPI == EPI_KIND_CLAMPQ || EPI == EPI_KIND_FAST) vec8(st.vec0 + 3 * n + f0, wq);
        const v4i none = {0, 0, 0, 0}, acc4[4][1] = {{acc[0]}, {acc[1]}, {none}, {none}}, ev4 = {ev.x, ev.y, 0, 0};
        const v4i p = epilogue_fast16<1, EPI, EPI == EPI_KIND_CLAMPQ ? 8 : 16>(st, acc4, 0, wq, cal, ecal, ev4, valid);
        return make_int2(p[0], p[1]);
    };
    const std::integral_constant<int, EPI0> kind0{};
    const std::integral_constant<int, EPI1> kind1{};
    const std::integral_constant<int, EPI2> kind2{};
    const int lf = 16 * (kq & 1) + 8 * (kq >> 1);  // the lane's first feature in a unit
    auto exists = [&](int u, const ChainStage& st) { return u * 32 + 16 * (kq & 1) < st.OFM; };  // its slice
    auto store = [&](const ChainStage& st, int at, int u, const int2& v) { *reinterpret_cast<int2*>((int8_t*)st.out + at + u * 2 * st.out_pf) = v; };
    const int2 zero2 = make_int2(0, 0);

    Refs cur, nxt;
    setup(g_begin, cur);
    {
        const uint32_t so = slice_of(0);
#pragma unroll
        for (int s = 0; s < S; ++s) load_step(cur, so, s);
    }
    step_fence();
    store_image(copied);
    __syncthreads();  // weights and vectors are in LDS; no barrier after this point

    for (int g = g_begin; g < g_end; g += 4) {
        setup(g + 4, nxt);
        // residual of the projection (a fused sum): requested now, used after the whole depthwise stage
        int2 ev1[P1];
        v4i acc1[P1][2];
#pragma unroll
        for (int p = 0; p < P1; ++p) {
            ev1[p] = zero2;
            if constexpr (chain_reads_residual<EPI1>())
                if (s1.fe.fused && exists(p, s1)) ev1[p] = *reinterpret_cast<const int2*>((const int8_t*)s1.eltw + cur.e1 + p * 2 * s1.el_pf);
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) acc1[p][mt] = *reinterpret_cast<const v4i*>(V + s1.vec0 + p * 32 + lf + mt * 4);
        }

        for (int k = 0; k < a.KS; ++k) {
            v4i bf0 = {0, 0, 0, 0};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int u = 2 * k + h;
                if (u >= a.U0) break;
                // ---------------- stage 0: a unit of the granule's pixels
                v4i acc0[2];
#pragma unroll
                for (int mt = 0; mt < 2; ++mt) acc0[mt] = *reinterpret_cast<const v4i*>(V + s0.vec0 + u * 32 + lf + mt * 4);
                const v4i w = fragment(u);
                const bool last = u + 1 == a.U0;
                const uint32_t so = slice_of(last ? 0 : u + 1);
#pragma unroll
                for (int s = 0; s < S; ++s) {
#pragma unroll
                    for (int mt = 0; mt < 2; ++mt) {
                        v4i fa = {0, 0, 0, 0};
#pragma unroll
                        for (int hh = 0; hh < 2; ++hh) fa[2 * hh + mt] = (int)__builtin_amdgcn_perm(0u, (unsigned)w[s >> 1], sel[s & 1][mt][hh]);
                        acc0[mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa, flip(rb[s], s0.xor_mask), acc0[mt], 0, 0, 0);
                    }
                    load_step(last ? nxt : cur, so, s);
                    step_fence();
                }
                // requantise: the packed results are half of the B fragment of stage 1's K-step k
                int2 p = finish(kind0, s0, a.n0, u * 32 + lf, acc0, zero2, 16);
                if (!exists(u, s0)) p = zero2;
                else if (cur.o0 >= 0) store(s0, cur.o0, u, p);
                p = flip2(p, s1.xor_mask);
                bf0[2 * h] = p.x, bf0[2 * h + 1] = p.y;
            }
            // ---------------- stage 1 accumulates this K-step
#pragma unroll
            for (int p = 0; p < P1; ++p)
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
                    acc1[p][mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(lds[a.w1 + ((k * P1 + p) * 2 + mt) * 64 + lane], bf0, acc1[p][mt], 0, 0, 0);
        }

        // ---------------- stage 1 epilogue: the packed results are the B fragment of stage 2
        v4i bf1 = {0, 0, 0, 0};
#pragma unroll
        for (int p = 0; p < P1; ++p) {
            int2 r = finish(kind1, s1, a.n1, p * 32 + lf, acc1[p], ev1[p], s1.OFM - p * 32 - lf);
            if (!exists(p, s1)) r = zero2;
            else if (cur.o1 >= 0) store(s1, cur.o1, p, r);
            r = flip2(r, s2.xor_mask);
            bf1[2 * p] = r.x, bf1[2 * p + 1] = r.y;
        }

        // ---------------- stage 2, unit by unit
        if constexpr (HAS2) {
            for (int u = 0; u < a.U2; ++u) {
                const int f0 = u * 32 + lf;
                v4i acc2[2];
#pragma unroll
                for (int mt = 0; mt < 2; ++mt)
                    acc2[mt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(lds[a.w2 + (u * 2 + mt) * 64 + lane], bf1, *reinterpret_cast<const v4i*>(V + s2.vec0 + f0 + mt * 4), 0, 0, 0);
                const int2 r = finish(kind2, s2, a.n2, f0, acc2, zero2, s2.OFM - f0);
                if (cur.o2 >= 0 && exists(u, s2)) store(s2, cur.o2, u, r);
            }
        }
        cur = nxt;
    }
}

template <int P1, bool HAS2, bool FLIP, int EPI0, int EPI1, int EPI2>
void launch_dwchain_instance(hipStream_t s, const DwChainArgs& a, int grid, int lds)
{
    static std::once_flag allowed;
    std::call_once(allowed, [] {
        CHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_dwchain_kernel<P1, HAS2, FLIP, EPI0, EPI1, EPI2>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    });
    hipLaunchKernelGGL((conv_dwchain_kernel<P1, HAS2, FLIP, EPI0, EPI1, EPI2>), dim3(grid), dim3(256), lds, s, a);
}

}  // namespace chip
