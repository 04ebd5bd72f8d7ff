// First layers: a convolution over at most four features of a plain bfyx image, read where it lies, with the 3x3 / stride-2 max
// pooling behind it finished on the way out where there is one.
//
// A first layer has too few features for the blocked layout: as launches of its own, the change of the layout costs a
// launch and the image once more, and the pooling reads back what the convolution has just written, four times the pooled
// tensor.  Here a workgroup of four waves turns the rows its outputs need into LDS, a dword per pixel (four features, the sign
// of u8 flipped, zeros around the image); sixteen bytes of a row are then four horizontal taps and one chunk of a K-step
// of v_mfma_i32_16x16x64_i8, at the pixel's own offset (the b_fs_yx_fsv4 layout, in LDS only).  All weights stay in registers.
//
// F: fragments of 16 features, 4 (up to 64 features; a lane ends with the sixteen of its slice) or 2 (up to 32; eight of slice
// q % 2, as in conv_dwchain_kernel.h: with four fragments half of the lanes would requantise features that do not exist).
// POOL: a wave walks down a strip of up to 15 pooled columns.  The even and the odd columns of a row are two fragments, so the
// maximum over a window's three columns is one instruction between them and one with the next lane (DPP); the third
// row of a window is the first of the next and is kept.  The maximum is taken over accumulators, without the bias: with
// factors that are not negative the ReLU requantisation is monotonic, and a pooled value costs one requantisation
// instead of four.  The even column past the edge starts from a number no sum reaches.
//
// Bound by the vector ALU (unpacking, maxima, requantisation; 56 % of the cycles) and the matrix cores (38 %) together; the image
// and the output at a copy's rate (5.16 TB/s) are 8.7 of the 36.7 us at batch 128, a quarter.  Kernel time, three or two launches before and
// now: ResNet-50 (7x7, pooled) batch 1 15.6 -> 10.4 us, 32 34 -> 15.1, 128 94 -> 36.7; MobileNet-v2 (3x3, 32 features) batch 1
// 10.7 -> 8.1, 32 21 -> 10.9; VGG-16 (3x3, 64 features) batch 1 10.8 -> 9.1, 16 23.8 -> 17.6.  (At batch 1 the image is read over the
// host link.)
#pragma once
#include "conv_mfma_kernel.h"

namespace chip {

constexpr int STEM_FAR_BELOW = -(1 << 30);  // start value of a column outside: a sum of at most 256 products of bytes stays below zero

struct StemArgs {
    const uint8_t* in;
    const v4i* wpk;            // [K-step][fragment][64 lanes]
    const int32_t* acc_init;
    int8_t* out;
    FastEpi fe;
    struct {
        const float *wqf, *calib, *eltw_calib, *bias;
        float oqf;
        int32_t oqf_on;
    } epi;
    int32_t in_off, in_pb, in_pf, in_py;       // bytes
    int32_t IFM, IH, IW;
    int32_t out_off, out_pb, out_pf, out_py;   // elements
    int32_t OFM, OH, OW, PH, PW;               // convolution and (pooled) output extents
    int32_t sy, sx, py, px, FY, nch;           // nch: chunks of four taps to a filter row
    int32_t B, row_groups, col_groups, total;  // workgroups: [image][group of rows][group of columns]
    FastDiv div_rows, div_cols;
    int32_t wg_rows, wg_cols;                  // output rows and columns of a workgroup
    int32_t wave_rows, tiles, tile_cols;       // pooling: rows of a wave, column strips of a workgroup (1, 2, 4) and their width
    int32_t lds_rows, pitch;                   // of the image part in LDS; pitch in pixels, a multiple of 4
    FastDiv div_frags;                         // 16-column fragments of a workgroup's row
    int32_t frags;
    uint32_t xor_mask;
};

// EVEN: the stride in x is 2.
template <int F, int KS, int EPI, bool POOL, bool EVEN>
__global__ void __launch_bounds__(256, POOL && F * KS > 8 ? 3 : 4) conv_stem_kernel(StemArgs a)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kq = lane >> 4;
    const int l16 = lane & 15;
    extern __shared__ __align__(16) unsigned char smem[];
    uint32_t* tile = reinterpret_cast<uint32_t*>(smem);

    // what the weights and the image rows need, behind one wait (three otherwise; 3x3 with 32 features, batch 32, 10.4 -> 10.0 us, batch 1
    // 8.4 -> 8.0; the 7x7 one at batch 5, from host memory, 19.5 -> 19.0)
    asm volatile("" ::"s"(a.in), "s"(a.wpk), "s"(a.in_off), "s"(a.in_pb), "s"(a.in_pf), "s"(a.in_py), "s"(a.IFM), "s"(a.IH), "s"(a.IW), "s"(a.sy), "s"(a.sx), "s"(a.py), "s"(a.px),
                 "s"(a.row_groups), "s"(a.col_groups), "s"(a.total), "s"(a.div_rows.mul), "s"(a.div_rows.shift), "s"(a.div_cols.mul), "s"(a.div_cols.shift), "s"(a.wg_rows),
                 "s"(a.wg_cols), "s"(a.lds_rows), "s"(a.pitch), "s"(a.xor_mask), "s"(gridDim.x));
    // neighbouring row groups on one die: they share image rows (the grid is a multiple of 8)
    const uint32_t wg = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (wg >= (uint32_t)a.total) return;
    const uint32_t t1 = a.div_cols.div(wg), b = a.div_rows.div(t1);
    const int row0 = (int)(t1 - b * (uint32_t)a.row_groups) * a.wg_rows, col0 = (int)(wg - t1 * (uint32_t)a.col_groups) * a.wg_cols;
    const int scale = POOL ? 2 : 1;  // convolution rows and columns to an output's
    const int y0 = row0 * scale * a.sy - a.py, x0 = col0 * scale * a.sx - a.px;

    v4i w[KS][F];
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int f = 0; f < F; ++f) w[k][f] = a.wpk[(k * F + f) * 64 + lane];

    // ---------------- the image rows into LDS: a wave takes every fourth row, a lane four pixels of it
    // Stride 2: a pixel's taps start at an even pixel.  The pairs of pixels lie in two halves of a row, even pairs and odd
    // pairs, so that sixteen neighbouring outputs read neighbouring pairs in either half, whichever they start with.
    const int quads = a.pitch >> 2;
    {
        const uint8_t* img = a.in + (a.in_off + (int64_t)b * a.in_pb);
        constexpr int BATCH = 4;
        for (int q0 = 0; q0 < quads; q0 += 64) {
            const int q = min(q0 + lane, quads - 1), x = x0 + q * 4;
            // the four bytes are read inside the row and moved to their place (a row has at least four pixels); a plane that does not
            // exist reads another one, its weights are zero
            const int xl = min(max(x, 0), a.IW - 4);
            const uint32_t shift = (uint32_t)(8 * (x - xl));
            const uint32_t left = x < 0 && x > -4 ? ~0u : 0u, right = x >= 0 && x < a.IW ? ~0u : 0u;
            for (int row0 = wave; row0 < a.lds_rows; row0 += 4 * BATCH) {
                uint32_t p[BATCH][4];
#pragma unroll
                for (int u = 0; u < BATCH; ++u) {
                    const uint8_t* src = img + (size_t)(uint32_t)(min(max(y0 + row0 + u * 4, 0), a.IH - 1) * a.in_py);
#pragma unroll
                    for (int c = 0; c < 3; ++c) __builtin_memcpy(&p[u][c], src + (size_t)(uint32_t)(min(c, a.IFM - 1) * a.in_pf) + (uint32_t)xl, 4);
                    p[u][3] = 0;
                    if (a.IFM == 4) __builtin_memcpy(&p[u][3], src + (size_t)(uint32_t)(3 * a.in_pf) + (uint32_t)xl, 4);
                }
#pragma unroll
                for (int u = 0; u < BATCH; ++u) {
                    const int row = row0 + u * 4;
                    if (row >= a.lds_rows) break;
                    const bool inside = (unsigned)(y0 + row) < (unsigned)a.IH;
                    const uint32_t l = inside ? left : 0u, r = inside ? right : 0u;
#pragma unroll
                    for (int c = 0; c < 4; ++c) p[u][c] = __builtin_amdgcn_alignbit(p[u][c] & l, p[u][c] & r, shift);
                    // bytes of four planes -> pixels
                    const uint32_t lo01 = __builtin_amdgcn_perm(p[u][1], p[u][0], 0x05010400u), hi01 = __builtin_amdgcn_perm(p[u][1], p[u][0], 0x07030602u);
                    const uint32_t lo23 = __builtin_amdgcn_perm(p[u][3], p[u][2], 0x05010400u), hi23 = __builtin_amdgcn_perm(p[u][3], p[u][2], 0x07030602u);
                    const uint32_t w0 = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u) ^ a.xor_mask, w1 = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u) ^ a.xor_mask;
                    const uint32_t w2 = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u) ^ a.xor_mask, w3 = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u) ^ a.xor_mask;
                    uint32_t* dst = tile + row * a.pitch;
                    if constexpr (EVEN) {
                        *reinterpret_cast<uint2*>(dst + q * 2) = make_uint2(w0, w1);
                        *reinterpret_cast<uint2*>(dst + (quads + q) * 2) = make_uint2(w2, w3);
                    } else {
                        *reinterpret_cast<uint4*>(dst + q * 4) = make_uint4(w0, w1, w2, w3);
                    }
                }
            }
        }
    }

    // where the lane's chunk of each K-step lies from its pixel on (dwords); chunks past the filter have zero weights
    int koff[KS];
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const int c = k * 4 + kq, fy = c / a.nch;
        koff[k] = fy < a.FY ? fy * a.pitch + (c - fy * a.nch) * (EVEN ? 2 : 4) : 0;
    }
    // the lane's features: sixteen of slice kq, or eight of slice kq % 2
    const int slice = F == 4 ? kq : kq & 1, f0 = F == 4 ? kq * 16 : 16 * (kq & 1) + 8 * (kq >> 1);
    // start values and factors: in registers, or (pooling, whose weights and row maxima fill those) in LDS
    v4i init[F];
    LaneScales sc;
    int32_t* vecs = reinterpret_cast<int32_t*>(tile + a.lds_rows * a.pitch);
    if constexpr (POOL) {
        if (threadIdx.x < F * 8) {
            const int f = (threadIdx.x & (F * 4 - 1)) * 4;
            *reinterpret_cast<v4i*>(vecs + threadIdx.x * 4) = *reinterpret_cast<const v4i*>(threadIdx.x < F * 4 ? (const void*)(a.acc_init + f) : (const void*)(a.epi.calib + f));
        }
    } else {
#pragma unroll
        for (int f = 0; f < F; ++f) init[f] = *reinterpret_cast<const v4i*>(a.acc_init + f0 + f * 4);
#pragma unroll
        for (int f = 0; f < F; ++f) load_scales4<EPI>(a, f0 + f * 4, sc, f);
    }
    const v4i none = {0, 0, 0, 0};
    const bool exists = slice * 16 < a.OFM;
    int8_t* const out0 = a.out + ((int64_t)a.out_off + (int64_t)b * a.out_pb + slice * a.out_pf + (F == 4 ? 0 : 8 * (kq >> 1)));
    __syncthreads();

    const int half = quads * 2;  // even: from an even pair to the odd pair behind it
    auto pair = [&](int at) { return *reinterpret_cast<const int2*>(tile + at); };
    auto join = [](const int2& lo, const int2& hi) { return v4i{lo.x, lo.y, hi.x, hi.y}; };

    auto finish = [&](const v4i(&acc)[F], int oy, int ox, bool ok) {
        v4i acc4[4][1];
#pragma unroll
        for (int f = 0; f < 4; ++f) acc4[f][0] = f < F ? acc[f < F ? f : 0] : none;
        const v4i q = epilogue_fast16<1, EPI, F * 4>(a, acc4, 0, sc.wq, sc.cal, sc.cal, none, a.OFM - f0);
        int8_t* dst = out0 + (uint32_t)(oy * a.out_py + ox * 16);
        if (ok && exists) {
            if constexpr (F == 4) *reinterpret_cast<v4i*>(dst) = q;
            else *reinterpret_cast<int2*>(dst) = make_int2(q[0], q[1]);
        }
    };

    if constexpr (POOL) {
        const int strip = wave & (a.tiles - 1), group = a.tiles == 4 ? 0 : a.tiles == 2 ? wave >> 1 : wave;
        const int c0 = col0 + strip * a.tile_cols;             // the strip's first pooled column, the lane's is c0 + l16
        const int p0 = row0 + group * a.wave_rows, p1 = min(min(p0 + a.wave_rows, row0 + a.wg_rows), a.PH);
        const int even = 2 * (c0 + l16);
        // Sixteen neighbouring even columns and the odd ones behind them, from the lane's even pixel on.  (A window's even and odd
        // column exist where the window does; the even column behind them may be past the edge.)
        const int x = 2 * (strip * a.tile_cols + l16) * a.sx;
        const int start = even < a.OW ? 0 : STEM_FAR_BELOW;
        const v4i se = {start, start, start, start};
#pragma unroll
        for (int k = 0; k < KS; ++k) koff[k] += EVEN ? x >> 1 : x;
        const bool ok = l16 < a.tile_cols && c0 + l16 < min(a.PW, col0 + a.wg_cols);
        auto row_max = [&](int r, v4i(&m)[F]) {  // over the three columns of the lane's window in convolution row r
            const int row = (r - 2 * row0) * a.sy * a.pitch;
            v4i e[F], o[F];
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                v4i ve, vo;
                const int at = row + koff[k];
                if constexpr (EVEN) {  // stride 2: the odd column starts a pair later
                    ve = join(pair(at), pair(at + half));
                    int again = at;  // (read twice: kept, the pair they share is copied in front of every second product)
                    asm("" : "+v"(again));
                    vo = join(pair(again + half), pair(again + 2));
                } else {
                    __builtin_memcpy(&ve, tile + at, 16);
                    __builtin_memcpy(&vo, tile + at + a.sx, 16);
                }
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    e[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[k][f], ve, k ? e[f] : se, 0, 0, 0);
                    o[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[k][f], vo, k ? o[f] : none, 0, 0, 0);
                }
            }
#pragma unroll
            for (int f = 0; f < F; ++f)
#pragma unroll
                for (int i = 0; i < 4; ++i)  // the next lane's even column; the last lane of sixteen has no window of its own
                    m[f][i] = max(max(e[f][i], o[f][i]), __builtin_amdgcn_update_dpp(0, e[f][i], 0x101, 0xf, 0xf, true));
        };
        v4i top[F];  // of the windows' rows so far
        if (p0 < p1) row_max(2 * p0, top);
        for (int p = p0; p < p1; ++p) {
            v4i m[F], done[F];
            if (2 * p + 1 < a.OH) {
                row_max(2 * p + 1, m);
#pragma unroll
                for (int f = 0; f < F; ++f)
#pragma unroll
                    for (int i = 0; i < 4; ++i) top[f][i] = max(top[f][i], m[f][i]);
            }
            if (2 * p + 2 < a.OH) {
                row_max(2 * p + 2, m);
#pragma unroll
                for (int f = 0; f < F; ++f)
#pragma unroll
                    for (int i = 0; i < 4; ++i) done[f][i] = max(top[f][i], m[f][i]);
            } else {
#pragma unroll
                for (int f = 0; f < F; ++f) done[f] = top[f];
            }
#pragma unroll
            for (int f = 0; f < F; ++f) {
                top[f] = m[f], done[f] += *reinterpret_cast<const v4i*>(vecs + f0 + f * 4);
                const v4i c = *reinterpret_cast<const v4i*>(vecs + F * 16 + f0 + f * 4);
#pragma unroll
                for (int i = 0; i < 4; ++i) sc.cal[f * 4 + i] = __int_as_float(c[i]);
            }
            finish(done, p, c0 + l16, ok);
        }
    } else {
        const int rows = min(a.wg_rows, a.OH - row0), work = rows * a.frags;
        for (int i = wave; i < work; i += 4) {
            const int row = (int)a.div_frags.div((uint32_t)i), col = (i - row * a.frags) * 16 + l16;
            v4i acc[F];
            // even: the pixel's pair is entry `col / 2` of the half of its parity
            const int at = row * a.sy * a.pitch + (EVEN ? (col & 1 ? half : 0) + (col >> 1) * 2 : col * a.sx);
            const int behind = EVEN ? at + (col & 1 ? 2 - half : half) : 0;
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                v4i v;
                if constexpr (EVEN) v = join(pair(at + koff[k]), pair(behind + koff[k]));
                else __builtin_memcpy(&v, tile + at + koff[k], 16);
#pragma unroll
                for (int f = 0; f < F; ++f) acc[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[k][f], v, k ? acc[f] : init[f], 0, 0, 0);
            }
            finish(acc, row0 + row, col0 + col, col0 + col < min(a.OW, col0 + a.wg_cols));
        }
    }
}

}  // namespace chip
