// Pooling for the layers between the convolutions of an int8 network (max / average over a sliding window).
// Arithmetic after the reference's kernels: kernel_selector/core/cl_kernels/pooling_gpu_int8_ref.cl:15-140 (int8:
// int accumulator, average = round(sum / count) half away from zero) and pooling_gpu_ref.cl (float: accumulator in
// the unit type, no rounding).  Window taps outside the input are skipped; a window that lies outside the input
// altogether leaves its output untouched (the buffer's zero).
#include "common.h"
#include "epilogue.h"
#include "kernels.h"
#include "conv_mfma_kernel.h"  // FastDiv

namespace chip {

struct PoolArgs {
    Pitch in, out;
    int B, F, IH, IW, OH, OW;
    int ky, kx, sy, sx, py, px;
    int mode;     // CLDNN_HIP_POOL_*
    int divider;  // CLDNN_HIP_POOL_DIV_*
    int dt;
};

__device__ __forceinline__ int window_count(const PoolArgs& a, int oy0, int ox0, int valid)
{
    if (a.divider == CLDNN_HIP_POOL_DIV_FIXED) return a.ky * a.kx;
    if (a.divider == CLDNN_HIP_POOL_DIV_VALID) return valid > 0 ? valid : 1;
    // window clipped to the input plus its padding (pooling_gpu_int8_ref.cl:104-108)
    const int hend = min(oy0 + a.ky, a.IH + a.py), wend = min(ox0 + a.kx, a.IW + a.px);
    const int n = (hend - oy0) * (wend - ox0);
    return n > 0 ? n : 1;
}

// one work-item per output element, any layout
__global__ void __launch_bounds__(256) pooling_kernel(PoolArgs a, const void* __restrict__ in, void* __restrict__ out)
{
    const int64_t total = (int64_t)a.B * a.F * a.OH * a.OW;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    int b, f, y, x;
    if (a.out.fsv > 1 || a.out.pf == 1) {  // features innermost in memory
        f = (int)(idx % a.F);
        int64_t r = idx / a.F;
        x = (int)(r % a.OW);
        r /= a.OW;
        y = (int)(r % a.OH);
        b = (int)(r / a.OH);
    } else {
        x = (int)(idx % a.OW);
        int64_t r = idx / a.OW;
        y = (int)(r % a.OH);
        r /= a.OH;
        f = (int)(r % a.F);
        b = (int)(r / a.F);
    }
    const int oy0 = y * a.sy - a.py, ox0 = x * a.sx - a.px;
    if (oy0 + a.ky < 0 || oy0 >= a.IH || ox0 + a.kx < 0 || ox0 >= a.IW) {
        // A window that lies wholly outside the input: the reference's kernel leaves such an output untouched, i.e. at
        // the zero its buffers are created with (pooling_gpu_int8_ref.cl:62-68).  A buffer handed over by the memory
        // pool is not zero, so the zero is written.
        EpiOut z;
        z.f = 0.0f, z.i = 0;
        store_out(out, a.dt, a.out.at(b, f, y, x), z);
        return;
    }
    const bool is_max = a.mode == CLDNN_HIP_POOL_MAX;
    int valid = 0;
    EpiOut o;
    if (a.dt == CLDNN_HIP_F32) {
        float r = is_max ? -3.402823466e+38f : 0.0f;  // UNIT_VAL_MIN of float
        for (int j = 0; j < a.ky; ++j) {
            const int iy = oy0 + j;
            if (iy < 0 || iy >= a.IH) continue;
            for (int i = 0; i < a.kx; ++i) {
                const int ix = ox0 + i;
                if (ix < 0 || ix >= a.IW) continue;
                const float v = ((const float*)in)[a.in.at(b, f, iy, ix)];
                r = is_max ? fmaxf(r, v) : r + v;
                ++valid;
            }
        }
        if (!is_max) r = r / (float)window_count(a, oy0, ox0, valid);
        o.f = r, o.i = 0;
    } else {
        int r = is_max ? -128 : 0;  // CHAR_MIN also for unsigned data, as in the reference
        for (int j = 0; j < a.ky; ++j) {
            const int iy = oy0 + j;
            if (iy < 0 || iy >= a.IH) continue;
            for (int i = 0; i < a.kx; ++i) {
                const int ix = ox0 + i;
                if (ix < 0 || ix >= a.IW) continue;
                const int64_t at = a.in.at(b, f, iy, ix);
                const int v = a.dt == CLDNN_HIP_U8 ? (int)((const uint8_t*)in)[at] : (int)((const int8_t*)in)[at];
                r = is_max ? max(r, v) : r + v;
                ++valid;
            }
        }
        if (!is_max) r = (int)round_half_away((float)r / (float)window_count(a, oy0, ox0, valid));
        o.i = r, o.f = (float)r;
    }
    store_out(out, a.dt, a.out.at(b, f, y, x), o);
}

// int8 in the blocked layout: one work-item per (pixel, slice of 16 features), 16-byte loads and one 16-byte store.
// 32-bit index arithmetic with precomputed reciprocals; windows that lie inside the input skip the per-tap tests.
struct PoolFastArgs {
    PoolArgs a;
    FastDiv div_ow, div_oh, div_b, div_kx;
    uint32_t total;
    int32_t in_off, in_pb, in_pf, in_py, out_off, out_pb, out_pf, out_py;
};

typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// element-wise max of four bytes at a time: a byte in the upper half of a 16-bit lane orders the lane whatever lies below it,
// so the odd bytes compare where they are and the even ones after one shift
template <bool UNSIGNED>
struct ByteMax {
    unsigned odd[4], even[4];
    __device__ __forceinline__ static unsigned pick(unsigned a, unsigned b)
    {
        if constexpr (UNSIGNED) return __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
        else return __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(s16x2, a), __builtin_bit_cast(s16x2, b)));
    }
    __device__ __forceinline__ void start(const uint4& v)
    {
        const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int d = 0; d < 4; ++d) odd[d] = w[d], even[d] = w[d] << 8;
    }
    __device__ __forceinline__ void add(const uint4& v)
    {
        const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int d = 0; d < 4; ++d) odd[d] = pick(odd[d], w[d]), even[d] = pick(even[d], w[d] << 8);
    }
    __device__ __forceinline__ unsigned result(int d) const { return (odd[d] & 0xff00ff00u) | ((even[d] >> 8) & 0x00ff00ffu); }
};

// bytes of features past the end of the tensor stay zero
__device__ __forceinline__ unsigned live_bytes(unsigned w, int live)
{
    return live >= 4 ? w : (live <= 0 ? 0u : w & ((1u << (8 * live)) - 1u));
}

struct PoolPos {
    int b, fs, y, x;
};
__device__ __forceinline__ PoolPos pool_pos(const PoolFastArgs& p, uint32_t idx)
{
    const uint32_t r = p.div_ow.div(idx), r2 = p.div_oh.div(r), fs = p.div_b.div(r2);
    return PoolPos{(int)(r2 - fs * (uint32_t)p.a.B), (int)fs, (int)(r - r2 * (uint32_t)p.a.OH), (int)(idx - r * (uint32_t)p.a.OW)};
}

// Max over KxK windows, K = 2 or 3, every window with a tap inside the input.  Taps outside repeat one inside, so there is no
// test per tap, all K * K requests go out before the first is waited for, and the maximum takes three instructions per four
// features and tap.  What is left is memory.
// 3x3 of 64 x 112x112: 6.8 -> 3.2 us at batch 1, 12.3 -> 7.8 at batch 32 (6.2 at the rate of a large copy); 2x2 of 64 x 224x224
// at batch 16: 13.2 -> 11.0 (12.3 if the input came from memory).
template <bool UNSIGNED, int K>
__global__ void __launch_bounds__(256) pooling_max_kernel(PoolFastArgs p, const uint8_t* __restrict__ in, uint8_t* __restrict__ out)
{
    const PoolArgs& a = p.a;
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= p.total) return;
    const PoolPos o = pool_pos(p, idx);
    const int oy0 = o.y * a.sy - a.py, ox0 = o.x * a.sx - a.px;
    const uint8_t* src = in + (p.in_off + o.b * p.in_pb + o.fs * p.in_pf);
    int row[K], col[K];
#pragma unroll
    for (int k = 0; k < K; ++k) row[k] = min(max(oy0 + k, 0), a.IH - 1) * p.in_py, col[k] = min(max(ox0 + k, 0), a.IW - 1) * 16;
    uint4 v[K * K];
#pragma unroll
    for (int t = 0; t < K * K; ++t) v[t] = *reinterpret_cast<const uint4*>(src + (row[t / K] + col[t % K]));
    ByteMax<UNSIGNED> m;
    m.start(v[0]);
#pragma unroll
    for (int t = 1; t < K * K; ++t) m.add(v[t]);
    const int live = a.F - o.fs * 16;
    *reinterpret_cast<uint4*>(out + (p.out_off + o.b * p.out_pb + o.fs * p.out_pf + o.y * p.out_py + o.x * 16)) =
        make_uint4(live_bytes(m.result(0), live), live_bytes(m.result(1), live - 4), live_bytes(m.result(2), live - 8), live_bytes(m.result(3), live - 12));
}

template <int CTRL>
__device__ __forceinline__ unsigned dpp(unsigned v)
{
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}

// Windows of 16 to 256 taps over few outputs (the global average in front of a classifier: 49 taps, 4096 windows x slices at
// batch 32), every window with a tap inside the input.  Sixteen lanes share a window; four taps each are requested at once
// (a loop of one request and one wait per tap was most of the time before), added up, combined across the
// lanes by lane permutes inside the vector unit, and every lane finishes one feature: one division instead of sixteen.
// 2048 x 7x7: 7.7 -> 3.2 us at batch 1, 8.0 -> 3.1 at batch 32 (3.5 with sums in packed 16-bit halves).
template <bool UNSIGNED, bool MAX>
__global__ void __launch_bounds__(256) pooling_window_kernel(PoolFastArgs p, const uint8_t* __restrict__ in, uint8_t* __restrict__ out)
{
    const PoolArgs& a = p.a;
    const uint32_t gid = blockIdx.x * 256u + threadIdx.x;
    const uint32_t idx = gid / 16;
    const int part = (int)(gid % 16);
    if (idx >= p.total) return;  // whole groups of 16 lanes leave together
    const PoolPos o = pool_pos(p, idx);
    const int oy0 = o.y * a.sy - a.py, ox0 = o.x * a.sx - a.px;
    const uint8_t* src = in + (p.in_off + o.b * p.in_pb + o.fs * p.in_pf);
    const int taps = a.ky * a.kx;
    const int live = a.F - o.fs * 16;

    ByteMax<UNSIGNED> m;
    int sum[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) sum[c] = 0;
    if constexpr (MAX) m.start(make_uint4(UNSIGNED ? 0 : 0x80808080u, UNSIGNED ? 0 : 0x80808080u, UNSIGNED ? 0 : 0x80808080u, UNSIGNED ? 0 : 0x80808080u));
    for (int t0 = 0; t0 < taps; t0 += 64) {
        uint4 v[4];
        bool inside[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = min(t0 + u * 16 + part, taps - 1);
            const int j = (int)p.div_kx.div((uint32_t)t), i = t - j * a.kx;
            const int iy = oy0 + j, ix = ox0 + i;
            inside[u] = t0 + u * 16 + part < taps && iy >= 0 && iy < a.IH && ix >= 0 && ix < a.IW;
            v[u] = *reinterpret_cast<const uint4*>(src + (min(max(iy, 0), a.IH - 1) * p.in_py + min(max(ix, 0), a.IW - 1) * 16));
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if constexpr (MAX) {
                m.add(v[u]);  // a tap outside has been replaced by one inside, a tap past the last by the last
            } else {
                const unsigned w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    // a dot product with a one in the feature's byte: unpacks and adds
                    const int e = inside[u] ? (int)w[c >> 2] : 0, one = 1 << (8 * (c & 3));
                    sum[c] = UNSIGNED ? (int)__builtin_amdgcn_udot4((unsigned)e, (unsigned)one, (unsigned)sum[c], false) : __builtin_amdgcn_sdot4(e, one, sum[c], false);
                }
            }
        }
    }
    auto across = [&](unsigned x, auto combine) {
        x = combine(x, dpp<0xb1>(x));   // lanes 1 apart
        x = combine(x, dpp<0x4e>(x));   // 2 apart
        x = combine(x, dpp<0x141>(x));  // the other four of eight
        return combine(x, dpp<0x140>(x));  // the other eight of sixteen
    };
    int value;
    if constexpr (MAX) {
        unsigned w = 0;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            m.odd[d] = across(m.odd[d], ByteMax<UNSIGNED>::pick), m.even[d] = across(m.even[d], ByteMax<UNSIGNED>::pick);
            if (part / 4 == d) w = m.result(d);
        }
        value = (int)(w >> (8 * (part & 3)));
    } else {
        int total = 0;
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const int all = (int)across((unsigned)sum[c], [](unsigned x, unsigned y) { return x + y; });
            if (part == c) total = all;
        }
        const int valid = (min(oy0 + a.ky, a.IH) - max(oy0, 0)) * (min(ox0 + a.kx, a.IW) - max(ox0, 0));
        value = (int)round_half_away((float)total / (float)window_count(a, oy0, ox0, valid));
    }
    out[p.out_off + o.b * p.out_pb + o.fs * p.out_pf + o.y * p.out_py + o.x * 16 + part] = part < live ? (uint8_t)value : (uint8_t)0;
}

template <bool UNSIGNED, bool MAX>
__global__ void __launch_bounds__(256) pooling_fsv16_kernel(PoolFastArgs p, const uint8_t* __restrict__ in, uint8_t* __restrict__ out)
{
    const PoolArgs& a = p.a;
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= p.total) return;
    const PoolPos pos = pool_pos(p, idx);
    const int b = pos.b, fs = pos.fs, y = pos.y, x = pos.x;
    const int oy0 = y * a.sy - a.py, ox0 = x * a.sx - a.px;
    if (oy0 + a.ky < 0 || oy0 >= a.IH || ox0 + a.kx < 0 || ox0 >= a.IW) {
        // a window wholly outside the input: zero, as a freshly created buffer of the reference holds (see pooling_kernel)
        *reinterpret_cast<uint4*>(out + (p.out_off + b * p.out_pb + fs * p.out_pf + y * p.out_py + x * 16)) = make_uint4(0, 0, 0, 0);
        return;
    }
    int acc[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) acc[c] = MAX ? -128 : 0;
    const uint8_t* src = in + (p.in_off + b * p.in_pb + fs * p.in_pf);
    auto tap = [&](int iy, int ix) {
        const uint4 v = *reinterpret_cast<const uint4*>(src + (iy * p.in_py + ix * 16));
        const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const unsigned byte = (w[c >> 2] >> (8 * (c & 3))) & 255u;
            const int e = UNSIGNED ? (int)byte : (int)(int8_t)byte;
            acc[c] = MAX ? max(acc[c], e) : acc[c] + e;
        }
    };
    int valid = 0;
    if (oy0 >= 0 && ox0 >= 0 && oy0 + a.ky <= a.IH && ox0 + a.kx <= a.IW) {
        for (int j = 0; j < a.ky; ++j)
            for (int i = 0; i < a.kx; ++i) tap(oy0 + j, ox0 + i);
        valid = a.ky * a.kx;
    } else {
        for (int j = 0; j < a.ky; ++j) {
            const int iy = oy0 + j;
            if (iy < 0 || iy >= a.IH) continue;
            for (int i = 0; i < a.kx; ++i) {
                const int ix = ox0 + i;
                if (ix < 0 || ix >= a.IW) continue;
                tap(iy, ix);
                ++valid;
            }
        }
    }
    if (!MAX) {
        const float n = (float)window_count(a, oy0, ox0, valid);
#pragma unroll
        for (int c = 0; c < 16; ++c) acc[c] = (int)round_half_away((float)acc[c] / n);
    }
    unsigned w[4] = {0, 0, 0, 0};
    const int live = a.F - fs * 16;  // features past the end of the tensor stay zero
#pragma unroll
    for (int c = 0; c < 16; ++c)
        if (c < live) w[c >> 2] |= ((unsigned)acc[c] & 255u) << (8 * (c & 3));
    *reinterpret_cast<uint4*>(out + (p.out_off + b * p.out_pb + fs * p.out_pf + y * p.out_py + x * 16)) = make_uint4(w[0], w[1], w[2], w[3]);
}

void launch_pooling(hipStream_t s, const cldnn_hip_pooling_desc& d, const void* in, void* out)
{
    const cldnn_hip_tensor &it = d.input, &ot = d.output;
    CHIP_REQUIRE(d.mode == CLDNN_HIP_POOL_MAX || d.mode == CLDNN_HIP_POOL_AVERAGE, CLDNN_HIP_INVALID_ARG, "pooling: unknown mode");
    CHIP_REQUIRE(d.divider >= CLDNN_HIP_POOL_DIV_FIXED && d.divider <= CLDNN_HIP_POOL_DIV_PADDED, CLDNN_HIP_INVALID_ARG,
                 "pooling: unknown divider mode");
    CHIP_REQUIRE(d.size_y > 0 && d.size_x > 0 && d.stride_y > 0 && d.stride_x > 0 && d.pad_y >= 0 && d.pad_x >= 0,
                 CLDNN_HIP_INVALID_ARG, "pooling: window and stride must be positive, padding non-negative");
    CHIP_REQUIRE(it.dtype == ot.dtype, CLDNN_HIP_INVALID_ARG, "pooling keeps the data type");
    CHIP_REQUIRE(it.dtype == CLDNN_HIP_S8 || it.dtype == CLDNN_HIP_U8 || it.dtype == CLDNN_HIP_F32, CLDNN_HIP_INVALID_ARG,
                 "pooling: data must be s8, u8 or f32");
    CHIP_REQUIRE(it.b == ot.b && it.f == ot.f, CLDNN_HIP_DIMENSION_MISMATCH, "pooling keeps batch and feature counts");
    CHIP_REQUIRE(ot.y > 0 && ot.x > 0, CLDNN_HIP_DIMENSION_MISMATCH, "pooling: empty output");
    PoolArgs a{};
    a.in = make_pitch(it), a.out = make_pitch(ot);
    a.B = it.b, a.F = it.f, a.IH = it.y, a.IW = it.x, a.OH = ot.y, a.OW = ot.x;
    a.ky = d.size_y, a.kx = d.size_x, a.sy = d.stride_y, a.sx = d.stride_x, a.py = d.pad_y, a.px = d.pad_x;
    a.mode = d.mode, a.divider = d.divider, a.dt = it.dtype;
    const bool blocked = it.format == CLDNN_HIP_FMT_FS_B_YX_FSV16 && ot.format == CLDNN_HIP_FMT_FS_B_YX_FSV16 && it.dtype != CLDNN_HIP_F32;
    const int64_t total = blocked ? (int64_t)((a.F + 15) / 16) * a.B * a.OH * a.OW : (int64_t)a.B * a.F * a.OH * a.OW;
    const int64_t blocks = (total + 255) / 256;
    CHIP_REQUIRE(blocks < (1ll << 31), CLDNN_HIP_UNSUPPORTED_SIZE, "tensor too large for the pooling grid");
    if (blocked) {
        CHIP_REQUIRE(tensor_elems(it) < (1ull << 31) && tensor_elems(ot) < (1ull << 31), CLDNN_HIP_UNSUPPORTED_SIZE, "tensor of 2 GiB or more");
        PoolFastArgs p{};
        p.a = a;
        p.div_ow = make_fast_div((uint32_t)a.OW), p.div_oh = make_fast_div((uint32_t)a.OH), p.div_b = make_fast_div((uint32_t)a.B);
        p.total = (uint32_t)total;
        p.in_off = (int32_t)a.in.off, p.in_pb = (int32_t)a.in.pb, p.in_pf = (int32_t)a.in.pf, p.in_py = (int32_t)a.in.py;
        p.out_off = (int32_t)a.out.off, p.out_pb = (int32_t)a.out.pb, p.out_pf = (int32_t)a.out.pf, p.out_py = (int32_t)a.out.py;
        const bool u = it.dtype == CLDNN_HIP_U8, mx = d.mode == CLDNN_HIP_POOL_MAX;
        p.div_kx = make_fast_div((uint32_t)a.kx);
        // the fast forms: every window has a tap inside the input
        const bool inside = a.py < a.ky && a.px < a.kx && (a.OH - 1) * a.sy - a.py < a.IH && (a.OW - 1) * a.sx - a.px < a.IW;
        const int taps = a.ky * a.kx;
        const bool window = inside && taps >= 16 && taps <= 256 && total < 256 * 1024;
        const dim3 grid((unsigned)(window ? (total * 16 + 255) / 256 : blocks)), block(256);
        const uint8_t* src = (const uint8_t*)in;
        uint8_t* dst = (uint8_t*)out;
#define POOL_LAUNCH(...) hipLaunchKernelGGL((__VA_ARGS__), grid, block, 0, s, p, src, dst)
        if (window) {
            if (u && mx) POOL_LAUNCH(pooling_window_kernel<true, true>);
            else if (u) POOL_LAUNCH(pooling_window_kernel<true, false>);
            else if (mx) POOL_LAUNCH(pooling_window_kernel<false, true>);
            else POOL_LAUNCH(pooling_window_kernel<false, false>);
        } else if (inside && mx && a.ky == a.kx && (a.ky == 2 || a.ky == 3)) {
            if (u && a.ky == 2) POOL_LAUNCH(pooling_max_kernel<true, 2>);
            else if (u) POOL_LAUNCH(pooling_max_kernel<true, 3>);
            else if (a.ky == 2) POOL_LAUNCH(pooling_max_kernel<false, 2>);
            else POOL_LAUNCH(pooling_max_kernel<false, 3>);
        } else if (u && mx) POOL_LAUNCH(pooling_fsv16_kernel<true, true>);
        else if (u) POOL_LAUNCH(pooling_fsv16_kernel<true, false>);
        else if (mx) POOL_LAUNCH(pooling_fsv16_kernel<false, true>);
        else POOL_LAUNCH(pooling_fsv16_kernel<false, false>);
#undef POOL_LAUNCH
    } else {
        hipLaunchKernelGGL(pooling_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a, in, out);
    }
    CHIP_CHECK(hipGetLastError());
}

}  // namespace chip
