// 1x1 convolutions of many input features: 64 pixels x 256 output features to a workgroup of four waves.
//
// The rows of the tile table work on 64 x 64 or 128 x 128 tiles: an activation passes L1 once for every 64 or 128 output features,
// and in the LDS-staged rows the weights pass LDS too.  Here a wave takes 64 output features and all pixels of the tile; its
// weights go from L2 straight into registers, the activations are copied into LDS once (direct global -> LDS loads, 128
// input features at a time, three buffers) and every LDS read (32 pixels x 32 K, 1 KB) serves two matrix instructions of 32 clocks.
// A barrier per 128 input features is all that the waves have in common; a block's successor is requested during it, into the
// buffer that was read two blocks ago.  LDS reads are issued by hand and waited for by count, as in conv_halo_kernel.h.
//
// Measured against the tile table's row for the layer, batch 32: 512 -> 256 + 1024 features in one launch, every second pixel of 28x28,
// 12.6 -> 8.9 us; 1024 -> 512 + 2048 at 14x14 12.1 -> 8.5; 256 -> 1024 with a sum at 14x14 8.0 -> 7.3; 512 -> 2048 with a sum at 7x7
// 7.2 -> 6.5; batch 128 35.3 -> 27.2, 30.3 -> 22.8, 20.8 -> 19.6, 17.7 -> 16.1; 1024 -> 256 at 14x14 12.9 -> 11.0.  With 128 pixels to a
// workgroup the large ones of these gain another 5 %, and what has fewer workgroups than CUs loses 20 to 40.  What is left is the
// requantisation (sums: 14 instructions a value) and, at batch 128, memory.
#pragma once
#include "conv_halo_kernel.h"

namespace chip {

enum { POINT_FEATURES = 256, POINT_PIXELS = 64 };

struct PointArgs {
    const int8_t* in;
    const v4i* wpk;            // [32 features][32 input features][64 lanes]
    const int32_t* acc_init;
    const float *calib, *ecal;
    const int8_t* eltw;
    int8_t* out;
    int32_t* raw;              // the accumulators instead
    FastEpi fe;
    int32_t in_off, in_pb, in_pf, in_row, in_col;     // bytes; row and column of an output pixel
    int32_t out_off, out_pb, out_pf, out_py;
    int32_t el_off, el_pb, el_pf, el_row, el_col;
    int32_t OFM, OHW, OW;
    uint32_t M;                // pixels of the batch
    FastDiv div_ohw, div_ow;
    int32_t ftiles, total, spans, jobs;  // tiles of features; workgroups; spans of 32 features; blocks of 128 input features
    FastDiv div_ftiles;
    uint32_t xor_mask;
};

// EPI: RELU, LINEAR (two convolutions in one included) or FUSED.  FLIP: u8 activations.
template <int EPI, bool FLIP>
__global__ void __launch_bounds__(256, 2) conv_point_kernel(PointArgs a)
{
    constexpr int NP = POINT_PIXELS / 32;                       // fragments of 32 pixels
    constexpr int RG = 4, READS = 4 * NP, AT_ONCE = 2;
    constexpr int LOADS = 2, REQUESTS = LOADS + 8;              // slices of a block that a wave copies; its weights
    constexpr int SLICE = POINT_PIXELS, BUF = 8 * SLICE;        // 16-byte units
    static_assert(READS % RG == 0 && REQUESTS <= AT_ONCE * (READS - RG + 2), "the ring goes round; all requests are out before the next block is read");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = lane >> 5;
    const int l32 = lane & 31;
    asm volatile("" ::"s"(a.in), "s"(a.wpk), "s"(a.acc_init), "s"(a.calib), "s"(a.in_off), "s"(a.in_pb), "s"(a.in_pf), "s"(a.in_row), "s"(a.in_col), "s"(a.M), "s"(a.OHW), "s"(a.OW),
                 "s"(a.total), "s"(a.ftiles), "s"(a.spans), "s"(a.jobs), "s"(a.xor_mask), "s"(a.div_ohw.mul), "s"(a.div_ow.mul), "s"(a.div_ftiles.mul), "s"(a.div_ftiles.shift),
                 "s"(gridDim.x));
    // (values of their own, or the compiler fetches the arguments again where they are used)
    global_bytes in = in_global(a.in + a.in_off), eltw = in_global(a.eltw);
    global<int8_t>* out = in_global(a.out);
    int in_pf = a.in_pf, out_off = a.out_off, out_pb = a.out_pb, out_pf = a.out_pf, out_py = a.out_py, OFM = a.OFM;
    int el_off = a.el_off, el_pb = a.el_pb, el_pf = a.el_pf, el_row = a.el_row, el_col = a.el_col;
    asm volatile("" : "+s"(in), "+s"(eltw), "+s"(out), "+s"(in_pf), "+s"(out_off), "+s"(out_pb), "+s"(out_pf), "+s"(out_py), "+s"(OFM), "+s"(el_off), "+s"(el_pb), "+s"(el_pf),
                 "+s"(el_row), "+s"(el_col));

    const uint32_t wg = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);  // the grid is a multiple of 8
    if (wg >= (uint32_t)a.total) return;
    // workgroups of one tile of pixels on one die: they share the input
    const uint32_t ptile = a.div_ftiles.div(wg), ftile = wg - ptile * (uint32_t)a.ftiles;
    const uint32_t m0 = ptile * POINT_PIXELS;

    extern __shared__ __align__(16) unsigned char smem[];
    v4i* lds = reinterpret_cast<v4i*>(smem);
    v4i* vectors = lds + 3 * BUF;  // start values, factors, factors of the sum: 256 of each
    {
        const void* from = wave == 1 ? (const void*)a.calib : wave == 2 && EPI == EPI_KIND_FUSED ? (const void*)a.ecal : (const void*)a.acc_init;
        const int which = wave == 1 ? 1 : wave == 2 && EPI == EPI_KIND_FUSED ? 2 : 0;  // (the other waves: the start values again)
        __builtin_amdgcn_global_load_lds((halo_gptr)((const v4i*)from + (size_t)ftile * 64 + lane), (halo_lptr)(vectors + which * 64), 16, 0, 0);
    }
    step_fence();
    auto pixel = [&](uint32_t m, uint32_t& b, uint32_t& oy, uint32_t& ox) {
        m = min(m, a.M - 1);  // (pixels past the last one are not stored)
        b = a.div_ohw.div(m);
        const uint32_t r = m - b * (uint32_t)a.OHW;
        oy = a.div_ow.div(r), ox = r - oy * (uint32_t)a.OW;
    };
    uint32_t src;
    {
        uint32_t b, oy, ox;
        pixel(m0 + lane, b, oy, ox);
        src = b * (uint32_t)a.in_pb + oy * (uint32_t)a.in_row + ox * (uint32_t)a.in_col;
    }
    const int span0 = (int)ftile * 8 + wave * 2;
    global_bytes weights[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        weights[s] = (global_bytes)(a.wpk + (size_t)min(span0 + s, a.spans - 1) * a.jobs * 4 * 64);  // past the last span: not stored
        asm volatile("" : "+s"(weights[s]));
    }
    const uint32_t lane_bytes = (uint32_t)lane * 16u;
    v4i w[2][8];
    auto request = [&](int j, int buffer, auto pc, auto rc) {
        constexpr int P = decltype(pc)::value, R = decltype(rc)::value;
        if constexpr (R < LOADS) {
            __builtin_amdgcn_global_load_lds((halo_gptr)(in + (int64_t)(j * 8 + wave * 2 + R) * in_pf + src), (halo_lptr)(lds + buffer + (wave * 2 + R) * SLICE), 16, 0, 0);
        } else if constexpr (R < REQUESTS) {
            constexpr int T = R - LOADS;
            w[P][T] = *(const global<v4i>*)(weights[T / 4] + (uint32_t)(j * 4 + T % 4) * 1024u + lane_bytes);
        }
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    static_for<0, REQUESTS>([&](auto rc) {
        request(0, 0, B0{}, rc);
        step_fence();
    });

    const uint32_t here = lds_offset(lds) + (uint32_t)(half * SLICE + l32) * 16u;
    v16i acc[2][NP] = {};
    const v4i xm = {(int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask};
    uint32_t ob[NP];
    v4i residual[2][NP] = {};
    v4i ring[RG];
    uint32_t at;
    auto block_arrived = [] { asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory"); };  // younger: the weights
    auto read = [&](int buffer, auto ic) {
        constexpr int R = decltype(ic)::value;
        if constexpr (R == 0) at = here + (uint32_t)(buffer * 16);
        lds_read<R / NP * 2 * SLICE * 16 + R % NP * 512>(ring[R % RG], at);
    };
    int buffer = 0;
    auto job = [&](int j, auto pc, auto last) {
        constexpr int P = decltype(pc)::value;
        constexpr bool LAST = decltype(last)::value;
        using Next = std::integral_constant<int, 1 - P>;
        const int next = buffer == 2 * BUF ? 0 : buffer + BUF;
        static_for<0, READS>([&](auto ic) {
            constexpr int R = decltype(ic)::value, K = R / NP, I = R % NP;
            constexpr int AHEAD = R + RG - 2;  // the latest read
            lds_wait<(LAST && AHEAD >= READS ? READS - 1 : AHEAD) - R>(ring[R % RG]);
            v4i x = ring[R % RG];
            if constexpr (FLIP) x ^= xm;
            acc[0][I] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[P][K], x, acc[0][I], 0, 0, 0);
            acc[1][I] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[P][4 + K], x, acc[1][I], 0, 0, 0);
            step_fence();
            if constexpr (!LAST) static_for<0, AT_ONCE>([&](auto rc) { request(j + 1, next, Next{}, std::integral_constant<int, R * AT_ONCE + decltype(rc)::value>{}); });
            if constexpr (AHEAD + 1 < READS) {
                read(buffer, std::integral_constant<int, AHEAD + 1>{});
            } else if constexpr (!LAST) {
                if constexpr (AHEAD + 1 == READS) block_arrived();
                read(next, std::integral_constant<int, AHEAD + 1 - READS>{});
            }
            // for the end, in the shadow of the products: where the lane's pixels go, and what is added to them
            if constexpr (LAST && R < NP) {
                uint32_t b, oy, ox;
                pixel(m0 + R * 32 + l32, b, oy, ox);
                ob[R] = (uint32_t)out_off + b * (uint32_t)out_pb + oy * (uint32_t)out_py + ox * 16u;
                if constexpr (EPI == EPI_KIND_FUSED) {
                    const uint32_t eb = (uint32_t)el_off + b * (uint32_t)el_pb + oy * (uint32_t)el_row + ox * (uint32_t)el_col;
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        const int slice = min((span0 + s) * 2 + half, (OFM - 1) >> 4);
                        if (!a.raw) residual[s][R] = *(const global<v4i>*)(eltw + (eb + (uint32_t)slice * (uint32_t)el_pf));
                    }
                }
            }
            step_fence();
        });
        buffer = next;
    };
    block_arrived();
    static_for<0, RG - 1>([&](auto ic) { read(0, ic); });
    for (int j = 0; j + 2 < a.jobs; j += 2) {
        job(j, B0{}, std::false_type{});
        job(j + 1, B1{}, std::false_type{});
    }
    job(a.jobs - 2, B0{}, std::false_type{});
    job(a.jobs - 1, B1{}, std::true_type{});

    v4i part[2 * NP][4];
#pragma unroll
    for (int i = 0; i < 2 * NP; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d) part[i][d] = v4i{acc[i / NP][i % NP][d * 4], acc[i / NP][i % NP][d * 4 + 1], acc[i / NP][i % NP][d * 4 + 2], acc[i / NP][i % NP][d * 4 + 3]};
    asm volatile("s_nop 7\n\ts_nop 7");  // a result of sixteen registers settles later than one of four
    step_fence();
    mfma_settle(part);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int slice = (span0 + s) * 2 + half, f0 = slice * 16, v = (wave * 64 + s * 32 + half * 16) / 4;
        float cal[16], ecal[16] = {}, wq[16] = {};
        v4i init[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            init[d] = vectors[v + d];
            const float4 c = reinterpret_cast<const float4*>(vectors)[64 + v + d];
            cal[d * 4] = c.x, cal[d * 4 + 1] = c.y, cal[d * 4 + 2] = c.z, cal[d * 4 + 3] = c.w;
            if constexpr (EPI == EPI_KIND_FUSED) {
                const float4 k = reinterpret_cast<const float4*>(vectors)[128 + v + d];
                ecal[d * 4] = k.x, ecal[d * 4 + 1] = k.y, ecal[d * 4 + 2] = k.z, ecal[d * 4 + 3] = k.w;
            }
        }
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            v4i sum[4][1];
#pragma unroll
            for (int d = 0; d < 4; ++d) sum[d][0] = part[s * NP + i][d] + init[d];
            const uint32_t m = m0 + i * 32 + l32;
            const bool ok = m < a.M && f0 < OFM;
            if (a.raw) {
                keep_branch();
                if (ok) {
                    uint32_t b, oy, ox;
                    pixel(m, b, oy, ox);
#pragma unroll
                    for (int c = 0; c < 16; ++c)
                        if (f0 + c < OFM) a.raw[((size_t)b * OFM + f0 + c) * a.OHW + oy * a.OW + ox] = sum[c >> 2][0][c & 3];
                }
                continue;
            }
            const v4i q = epilogue_fast16<1, EPI>(a, sum, 0, wq, cal, ecal, residual[s][i], OFM - f0);
            if (ok) *(global<v4i>*)(out + (ob[i] + (uint32_t)slice * (uint32_t)out_pf)) = q;
        }
    }
}

}  // namespace chip
