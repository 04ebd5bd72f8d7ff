// Depthwise quantized convolution (groups == input features == output features) on fs_b_yx_fsv16.
//
// Three kernels.  conv_dw_rows_kernel runs 3x3 (stride 1) and 5x5 filters on the matrix cores; conv_dw3x3_kernel takes the
// other 3x3 layers with dot-product instructions; both need an input with a zero border and
// the short requantisation epilogue.  conv_dw_kernel is everything else: one lane owns the 16 features of one output pixel,
// every tap is one coalesced 128-bit load and the per-slice weights [tap][16] sit in LDS.
#include "conv_mfma_kernel.h"

#include <cstring>

namespace chip {

struct DwArgs {
    const int8_t* in;
    const int8_t* wpk;        // [fs][tap][16]
    const int32_t* wmask;     // [fs][tap][16] dwords: weight of feature c alone in byte c % 4 (3x3 kernel)
    const v4i* wrows;         // [fs][row of the filter][block of 4 positions][lane] (rows kernel)
    const int32_t* acc_init;  // [fs*16]
    void* out;
    const void* eltw;
    int32_t* raw;
    Pitch in_p, out_p, eltw_p;
    int B, IH, IW, OH, OW, C, OHW;
    int FY, FX, sy, sx, dy, dx, py, px, esy, esx;
    int64_t M;
    int in_u8;
    uint32_t xor_mask;
    FastDiv div_ohw, div_ow;
    // rows kernel: OW4 groups of four output pixels in a row, OH * OW4 in an image, `chunks` workgroups to a feature slice
    uint32_t OW4, OHW4, groups, chunks, works;
    int rounds;
    uint32_t in_last;  // offset of the last 16 bytes of the input
    FastDiv div_ohw4, div_ow4, div_chunks;
    FastEpi fe;
    Epilogue epi;
};

template <bool IN_U8>
__device__ __forceinline__ void mac16(int* acc, const v4i& x, const v4i& w)
{
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const unsigned xv = (unsigned)x[d], wv = (unsigned)w[d];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int xi = IN_U8 ? (int)((xv >> (8 * i)) & 255u) : (int)(int8_t)(xv >> (8 * i));
            const int wi = (int)(int8_t)(wv >> (8 * i));
            acc[d * 4 + i] += xi * wi;
        }
    }
}

template <bool IN_U8>
__global__ void __launch_bounds__(256) conv_dw_kernel(DwArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    v4i* wl = reinterpret_cast<v4i*>(smem);  // [taps]
    const int fs = blockIdx.y;
    const int taps = a.FY * a.FX;
    for (int i = threadIdx.x; i < taps; i += blockDim.x)
        wl[i] = reinterpret_cast<const v4i*>(a.wpk)[(int64_t)fs * taps + i];
    __syncthreads();

    const int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= a.M) return;
    const int b = (int)(m / a.OHW);
    const int r = (int)(m % a.OHW);
    const int oy = r / a.OW, ox = r % a.OW;
    const int iy0 = oy * a.sy - a.py, ix0 = ox * a.sx - a.px;
    const int64_t ibase = a.in_p.off + (int64_t)b * a.in_p.pb + (int64_t)fs * a.in_p.pf;

    int acc[16];
    {
        const v4i* ai = reinterpret_cast<const v4i*>(a.acc_init + fs * 16);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const v4i v = ai[d];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[d * 4 + i] = v[i];
        }
    }
    for (int j = 0; j < a.FY; ++j) {
        const int iy = iy0 + j * a.dy;
        if (iy < 0 || iy >= a.IH) continue;
        for (int i = 0; i < a.FX; ++i) {
            const int ix = ix0 + i * a.dx;
            if (ix < 0 || ix >= a.IW) continue;
            const v4i x = *reinterpret_cast<const v4i*>(a.in + ibase + (int64_t)iy * a.in_p.py + (int64_t)ix * 16);
            mac16<IN_U8>(acc, x, wl[j * a.FX + i]);
        }
    }

    const Epilogue& e = a.epi;
    const int f0 = fs * 16;
    if (a.raw) {
#pragma unroll
        for (int c = 0; c < 16; ++c)
            if (f0 + c < a.C) a.raw[(((int64_t)b * a.C + f0 + c) * a.OH + oy) * a.OW + ox] = acc[c];
        return;
    }
    const int64_t obase = a.out_p.off + (int64_t)b * a.out_p.pb + (int64_t)fs * a.out_p.pf + (int64_t)oy * a.out_p.py
                          + (int64_t)ox * a.out_p.px;
    int64_t ebase = 0;
    if (e.fused)
        ebase = a.eltw_p.off + (int64_t)b * a.eltw_p.pb + (int64_t)fs * a.eltw_p.pf
                + (int64_t)(oy * a.esy) * a.eltw_p.py + (int64_t)(ox * a.esx) * a.eltw_p.px;
    const bool out8 = e.out_dt == CLDNN_HIP_S8 || e.out_dt == CLDNN_HIP_U8;
    v4i packed = {0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < 16; ++c) {
        const int f = f0 + c;
        EpiOut o;
        o.f = 0.f, o.i = 0;
        if (f < a.C) {
            float ev = 0.f;
            if (e.fused) ev = load_as_float(a.eltw, e.eltw_dt, ebase + c);
            o = epilogue_generic(e, acc[c], f, ev);
        }
        if (out8) packed[c >> 2] |= (int)(((unsigned)o.i & 255u) << (8 * (c & 3)));
        else store_out(a.out, e.out_dt, obase + c, o);
    }
    if (out8) *reinterpret_cast<v4i*>((int8_t*)a.out + obase) = packed;
}

// 3x3 depthwise, constant tap offsets (zero border), short epilogue.  A lane owns the 16 features of one output
// pixel.  The multiply uses the packed dot-product instruction with one weight byte unmasked per call:
// sdot4(x_dword, {0,..,w_c,..,0}, acc_c) adds x_c * w_c to the accumulator of feature c without unpacking a single
// byte; the masked weights of a feature slice are the same for every lane and come through the scalar data path.
// u8 activations are fed as x ^ 0x80 = x - 128, the accumulators start from 128 * sum(w) (+ bias).
template <int EPI>
__global__ void __launch_bounds__(256) conv_dw3x3_kernel(DwArgs a)
{
    // What the requests need, behind one wait.  Left to itself the compiler fetches it in four turns, each behind the one before (an
    // asm volatile would turn the scalar loads below into vector ones).  Relu and no activation, stride 2: 32 x 192 x 28x28 4.17 and 4.47 us in
    // four turns, 3.90 and 4.00 in one; 32 x 96 x 112x112 13.7 and 13.8, 13.4 and 13.6; batch 1 3.10 and 3.18, 3.00 and 3.06.
    uint32_t M = (uint32_t)a.M;
    FastDiv div_ohw = a.div_ohw, div_ow = a.div_ow;
    int32_t OHW = a.OHW, OW = a.OW, in_pb = (int32_t)a.in_p.pb, in_py = (int32_t)a.in_p.py, sy = a.sy, sx = a.sx, py = a.py, px = a.px, dy = a.dy, dx = a.dx;
    int64_t in_off = a.in_p.off, in_pf = a.in_p.pf;
    uintptr_t in = (uintptr_t)a.in, masked = (uintptr_t)a.wmask;
    asm("" : "+s"(M), "+s"(div_ohw.mul), "+s"(div_ohw.shift), "+s"(div_ow.mul), "+s"(div_ow.shift), "+s"(OHW), "+s"(OW), "+s"(in_pb), "+s"(in_py), "+s"(sy), "+s"(sx), "+s"(py),
        "+s"(px), "+s"(dy), "+s"(dx), "+s"(in_off), "+s"(in_pf), "+s"(in), "+s"(masked));
    const int fs = blockIdx.y;
    const uint32_t m = blockIdx.x * 256u + threadIdx.x;
    const bool ok = m < M;
    const uint32_t mm = ok ? m : 0;
    const uint32_t b = div_ohw.div(mm);
    const uint32_t r = mm - b * (uint32_t)OHW;
    const uint32_t oy = div_ow.div(r);
    const uint32_t ox = r - oy * (uint32_t)OW;
    typedef const __attribute__((address_space(1))) int8_t* global_bytes;
    const global_bytes src = (global_bytes)(in + (uintptr_t)(in_off + (int64_t)fs * in_pf)) + ((int32_t)b * in_pb + ((int32_t)oy * sy - py) * in_py + ((int32_t)ox * sx - px) * 16);
    v4i x[9];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) x[j * 3 + i] = *(const __attribute__((address_space(1))) v4i*)(src + (j * dy * in_py + i * dx * 16));

    v4i ev4 = {0, 0, 0, 0};
    const int f0 = fs * 16;
    const int obase = (int)(a.out_p.off + (int64_t)fs * a.out_p.pf) + (int)b * (int)a.out_p.pb + (int)oy * (int)a.out_p.py + (int)ox * 16;
    const int ebase = (int)(a.eltw_p.off + (int64_t)fs * a.eltw_p.pf) + (int)b * (int)a.eltw_p.pb
                      + (int)(oy * a.esy) * (int)a.eltw_p.py + (int)(ox * a.esx) * 16;
    if (a.fe.fused) ev4 = *reinterpret_cast<const v4i*>((const int8_t*)a.eltw + ebase);
    LaneScales sc;
    load_scales<EPI>(a, f0, sc);

    v4i acc[4][1];
#pragma unroll
    for (int d = 0; d < 4; ++d) acc[d][0] = *reinterpret_cast<const v4i*>(a.acc_init + f0 + d * 4);
    const const_i32_ptr wm = (const_i32_ptr)(masked + (uintptr_t)fs * 9 * 16 * 4);
#pragma unroll
    for (int t = 0; t < 9; ++t) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const int xd = x[t][d] ^ (int)a.xor_mask;
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[d][0][i] = __builtin_amdgcn_sdot4(xd, wm[t * 16 + d * 4 + i], acc[d][0][i], false);
        }
    }
    if (!ok) return;
    const int valid = a.C - f0;
    const v4i packed = epilogue_fast16<1, EPI>(a, acc, 0, sc.wq, sc.cal, sc.ecal, ev4, valid);
    *reinterpret_cast<v4i*>((int8_t*)a.out + obase) = packed;
}

// Depthwise on the matrix cores: FY rows of the filter, NB blocks of four input positions to a row.
//
// The sixteen columns of a v_mfma_i32_16x16x64_i8 are sixteen groups of four neighbouring output pixels of a row.  The 64
// values of its contraction are four input positions (lane / 16) of the slice's 16 features, one 128-bit load per lane.  Its
// rows are chosen so that four products (p = 0..3) leave in lane (group, q) the features 4p..4p+3 of output pixel q of its
// group: row (q, i) of product p holds the taps of feature 4p + i that pixel q sees in these four positions.  So every
// input byte is loaded once for four outputs (the dot-product kernel loads nine or twenty-five), a lane ends with all 16
// features of its pixel, and the row operands have one dword each that is not zero: the table holds those alone.
//
// 3x3, stride 1: 6 loads and 24 products for 64 pixels of a slice, against 9 loads and 144 dot products; 5x5: 10 and 40
// against 25 and 400.  At that rate memory is the bound of large planes; a wave keeps its table in registers for `rounds`
// sets of 64 pixels and requests the next set before it finishes the present one.  Small planes are bound by the launch and
// the latency of one set: the prologue has no branch, or the compiler fetches the arguments in four turns, each behind the one before,
// and the weights are asked for behind two of them, before the addresses of the activations are known (recorded, one behind the
// other, with a branch in front of the requests and now: 32 x 576 x 14x14, 3x3, 5.0 and 4.8 us a layer, batch 1 2.74 and 2.49; 7 x 67 x
// 93x93, 5x5 at stride 2, 7.1 and 6.4; 10 x 488 x 59x59, 5x5, 18.1 and 17.9).  A workgroup too many leaves behind its requests.  Without
// that end the 5x5 forms were a wave a SIMD short: 64 x 256 x 56x56 49.3 us, 46.8 with it, 128 x 96 x 112x112 135.8 and 130.7.
// Kernel time, 32 x 576 x 14x14, 3x3: 6.3 -> 5.3 us (1.4 us at the rate of a large copy and about 3 of launch); 8 x 512 x 28x28,
// 5x5: 32.4 -> 6.5; 32 x 64 x 112x112, 5x5: 143 -> 26 (10.3 at the rate of a large copy), 3x3: 22.7 -> 18.4.
template <int FY, int NB, int EPI>
__global__ void __launch_bounds__(256, 2) conv_dw_rows_kernel(DwArgs a)
{
    constexpr int S = FY * NB;
    // neighbouring chunks of a plane on one XCD (the grid is a multiple of 8): the rows they share are in its L2
    const uint32_t turn = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const bool spare = turn >= a.works;  // (leaves behind its requests: what is behind a branch would be fetched behind it)
    const uint32_t work = spare ? 0u : turn;
    const uint32_t fs = a.div_chunks.div(work), chunk = work - fs * a.chunks;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4, f0 = (int)fs * 16;

    v4i w[S];
    const v4i* wt = a.wrows + (size_t)fs * S * 64 + lane;
#pragma unroll
    for (int s = 0; s < S; ++s) w[s] = wt[s * 64];
    step_fence();

    const uint32_t in_py = (uint32_t)a.in_p.py, tap_py = in_py * (uint32_t)a.dy;
    int8_t* out = (int8_t*)a.out + (a.out_p.off + (int64_t)fs * a.out_p.pf);
    const int8_t* el = (const int8_t*)a.eltw + (a.eltw_p.off + (int64_t)fs * a.eltw_p.pf);
    const uint32_t in_slice = (uint32_t)(a.in_p.off + (int64_t)fs * a.in_p.pf);
    LaneScales sc;
    load_scales<EPI>(a, f0, sc);
    v4i init[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) init[p] = *reinterpret_cast<const v4i*>(a.acc_init + f0 + p * 4);

    v4i x[S], ev4 = {0, 0, 0, 0};
    uint32_t opos = 0;
    bool ok = false;
    auto request = [&](int r) {
        const uint32_t g = ((chunk * (uint32_t)a.rounds + (uint32_t)r) * 4u + (uint32_t)wave) * 16u + (uint32_t)(lane & 15);
        const bool real = g < a.groups;
        const uint32_t gg = real ? g : 0;
        const uint32_t b = a.div_ohw4.div(gg), t = gg - b * a.OHW4, oy = a.div_ow4.div(t), ox0 = (t - oy * a.OW4) * 4u;
        const uint32_t src = in_slice + b * (uint32_t)a.in_p.pb + (uint32_t)((int)oy * a.sy - a.py) * in_py
                             + (uint32_t)(((int)ox0 * a.sx - a.px) * 16) + (uint32_t)q * 16u;
#pragma unroll
        for (int j = 0; j < FY; ++j)
#pragma unroll
            for (int n = 0; n < NB; ++n)  // (positions past the row belong to pixels that do not exist, or to no tap)
                x[j * NB + n] = *reinterpret_cast<const v4i*>(a.in + min(src + (uint32_t)j * tap_py + (uint32_t)n * 64u, a.in_last));
        const uint32_t ox = ox0 + (uint32_t)q;
        ok = real && ox < (uint32_t)a.OW;
        opos = b * (uint32_t)a.out_p.pb + oy * (uint32_t)a.out_p.py + ox * 16u;
        if constexpr (EPI == EPI_KIND_FAST)
            if (a.fe.fused && ok)
                ev4 = *reinterpret_cast<const v4i*>(el + (b * (uint32_t)a.eltw_p.pb + oy * (uint32_t)(a.esy * (int)a.eltw_p.py) + ox * (uint32_t)(a.esx * 16)));
    };
    request(0);
    step_fence();
    if (spare) return;  // (with an end on the way the compiler keeps 16 registers less)
    int r = 0;
    do {
        v4i acc[4][1];
#pragma unroll
        for (int p = 0; p < 4; ++p) acc[p][0] = init[p];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            v4i xs = x[s];
            asm volatile("" : "+v"(w[s]));  // the row operands are made here: made once for all rounds they take four times the registers
#pragma unroll
            for (int d = 0; d < 4; ++d) xs[d] ^= (int)a.xor_mask;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                v4i row = {0, 0, 0, 0};
                row[p] = w[s][p];
                acc[p][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(row, xs, acc[p][0], 0, 0, 0);
            }
        }
        const v4i e = ev4;
        const uint32_t at = opos;
        const bool store = ok;
        if (r + 1 < a.rounds) request(r + 1);
        const v4i packed = epilogue_fast16<1, EPI>(a, acc, 0, sc.wq, sc.cal, sc.ecal, e, a.C - f0);
        if (store) *reinterpret_cast<v4i*>(out + at) = packed;
    } while (++r < a.rounds);
}

// blocks of four positions that four neighbouring outputs see in a row
static int dw_row_blocks(const ConvProblem& p)
{
    return (3 * p.sx + (p.FX - 1) * p.dx + 1 + 3) / 4;
}

DwPlan dw_plan(const ConvProblem& p, bool fast_epilogue, int cus)
{
    DwPlan pl{};
    pl.block = 256;
    const int nb = dw_row_blocks(p);
    // 5x5 at strides 1 and 2, 3x3 at stride 1.  At stride 2 four outputs of a 3x3 row see nine positions, three blocks: that is
    // as many loads as the dot products have taps (16 x 256 x 56x56: 7.0 us against 5.2), so those layers keep them.
    if (dw_fast_applies(p, fast_epilogue) && ((p.FY == 3 && nb == 2) || (p.FY == 5 && (nb == 2 || nb == 3)))) {
        pl.rows = 1;
        pl.row_bytes = (size_t)((p.OFM + 15) / 16) * p.FY * nb * 1024;
        const int64_t groups = (int64_t)p.B * p.OH * ((p.OW + 3) / 4), slices = (p.OFM + 15) / 16;
        // sets of 64 pixels to a wave: one or two, so that the chip holds many waves (16 x 256 x 56x56, 5x5 at stride 2: 11.2 us
        // with one, 10.4 with two, 12.5 with four), four 3x3 sets where there are 48 waves to a CU all the same
        const int64_t sets = (groups + 15) / 16, per_cu = sets * slices / cus;
        pl.rounds = p.FY == 5 ? (per_cu >= 8 ? 2 : 1) : per_cu >= 192 ? 4 : per_cu >= 96 ? 2 : 1;
        pl.chunks = (int)((sets + 4 * pl.rounds - 1) / (4 * pl.rounds));
        pl.works = (int)(pl.chunks * slices);
        pl.grid_rows = (pl.works + 7) / 8 * 8;
    }
    const int64_t m = (int64_t)p.B * p.OH * p.OW;
    const int64_t gx = (m + pl.block - 1) / pl.block;
    CHIP_REQUIRE(gx < (1ll << 31), CLDNN_HIP_UNSUPPORTED_SIZE, "convolution too large for one launch");
    pl.grid = (int)gx;  // of the accumulator probe as well
    pl.one_round = gx * ((p.OFM + 15) / 16) <= 8ll * cus ? 1 : 0;
    pl.packed_bytes = (size_t)((p.OFM + 15) / 16) * p.FY * p.FX * 16;
    pl.mask_bytes = pl.packed_bytes * 4;
    return pl;
}

// weights [C][1][FY][FX] -> [fs][tap][16]
void dw_pack_weights(const ConvProblem& p, const int8_t* w, int8_t* packed)
{
    const int taps = p.FY * p.FX;
    std::memset(packed, 0, (size_t)((p.OFM + 15) / 16) * taps * 16);
    for (int c = 0; c < p.OFM; ++c)
        for (int t = 0; t < taps; ++t) packed[((size_t)(c / 16) * taps + t) * 16 + (c % 16)] = w[(size_t)c * taps + t];
}

// masked weights for the 3x3 kernel: dword (fs, tap, c) holds weight c of the slice in byte c % 4, zeros elsewhere
void dw_mask_weights(const ConvProblem& p, const int8_t* w, int32_t* masked)
{
    const int taps = p.FY * p.FX;
    std::memset(masked, 0, (size_t)((p.OFM + 15) / 16) * taps * 16 * 4);
    for (int c = 0; c < p.OFM; ++c)
        for (int t = 0; t < taps; ++t)
            masked[((size_t)(c / 16) * taps + t) * 16 + (c % 16)] =
                (int32_t)((uint32_t)(uint8_t)w[(size_t)c * taps + t] << (8 * (c % 4)));
}

// rows [fs][filter row][block][lane] of four dwords: lane (row (q, i), position k) holds in dword p the weight with which
// feature 4p + i of output pixel q takes position 4 * block + k, in byte i
void dw_row_weights(const ConvProblem& p, const int8_t* w, int32_t* rows)
{
    const int nb = dw_row_blocks(p);
    size_t at = 0;
    for (int s = 0; s < (p.OFM + 15) / 16; ++s)
        for (int j = 0; j < p.FY; ++j)
            for (int n = 0; n < nb; ++n)
                for (int lane = 0; lane < 64; ++lane)
                    for (int d = 0; d < 4; ++d, ++at) {
                        const int q = (lane % 16) / 4, i = lane % 4, c = s * 16 + d * 4 + i, t = 4 * n + lane / 16 - q * p.sx;
                        rows[at] = 0;
                        if (c < p.OFM && t >= 0 && t % p.dx == 0 && t / p.dx < p.FX)
                            rows[at] = (int32_t)((uint32_t)(uint8_t)w[((size_t)c * p.FY + j) * p.FX + t / p.dx] << (8 * i));
                    }
}

// what the two fast kernels ask for: zero border covering the padding, short epilogue, 32-bit offsets
bool dw_fast_applies(const ConvProblem& p, bool fast_epilogue)
{
    return fast_epilogue && conv_border_covers(p) && tensor_elems(p.in_t) < (1ull << 31) && tensor_elems(p.out_t) < (1ull << 31)
           && (p.eltw_t.b <= 0 || tensor_elems(p.eltw_t) < (1ull << 31)) && (int64_t)p.B * p.OH * (p.OW + 3) < (1ll << 31);
}

template <int FY, int NB>
static void launch_rows(hipStream_t s, const DwPlan& pl, const DwArgs& a)
{
    const dim3 g(pl.grid_rows), b(256);
    const FastEpi& f = a.fe;
    const bool plain = a.epi.calib && !f.fused;
    if (plain && f.has_wqf && f.iqf_one && f.clamp_folded) hipLaunchKernelGGL((conv_dw_rows_kernel<FY, NB, EPI_KIND_CLAMPQ>), g, b, 0, s, a);
    else if (plain && !f.has_wqf && f.relu_folded) hipLaunchKernelGGL((conv_dw_rows_kernel<FY, NB, EPI_KIND_RELU>), g, b, 0, s, a);
    else if (plain && !f.has_wqf && f.act == CLDNN_HIP_ACT_NONE) hipLaunchKernelGGL((conv_dw_rows_kernel<FY, NB, EPI_KIND_LINEAR>), g, b, 0, s, a);
    else hipLaunchKernelGGL((conv_dw_rows_kernel<FY, NB, EPI_KIND_FAST>), g, b, 0, s, a);
}

void launch_conv_dw(hipStream_t s, const ConvProblem& p, const DwPlan& pl, const int8_t* packed, const int32_t* masked, const int32_t* rows,
                    const int32_t* acc_init, const Epilogue& epi, const FastEpi* fast, const void* in, const void* eltw,
                    void* out, int32_t* raw)
{
    DwArgs a{};
    a.wmask = masked;
    a.in = (const int8_t*)in, a.wpk = packed, a.acc_init = acc_init, a.out = out, a.eltw = eltw, a.raw = raw;
    a.in_p = p.in_p, a.out_p = p.out_p, a.eltw_p = p.eltw_p;
    a.B = p.B, a.IH = p.IH, a.IW = p.IW, a.OH = p.OH, a.OW = p.OW, a.C = p.OFM, a.OHW = p.OH * p.OW;
    a.FY = p.FY, a.FX = p.FX, a.sy = p.sy, a.sx = p.sx, a.dy = p.dy, a.dx = p.dx, a.py = p.py, a.px = p.px;
    a.esy = p.esy, a.esx = p.esx;
    a.M = (int64_t)p.B * p.OH * p.OW;
    a.epi = epi;
    const dim3 grid(pl.grid, (p.OFM + 15) / 16);
    if (fast) a.fe = *fast;
    a.xor_mask = p.in_dt == CLDNN_HIP_U8 ? 0x80808080u : 0u;
    if (pl.rows && !raw) {
        a.wrows = (const v4i*)rows, a.OW4 = (uint32_t)(p.OW + 3) / 4, a.OHW4 = (uint32_t)p.OH * a.OW4, a.groups = (uint32_t)p.B * a.OHW4;
        a.chunks = (uint32_t)pl.chunks, a.works = (uint32_t)pl.works, a.rounds = pl.rounds;
        a.in_last = (uint32_t)tensor_elems(p.in_t) - 16u;
        a.div_ohw4 = make_fast_div(a.OHW4), a.div_ow4 = make_fast_div(a.OW4), a.div_chunks = make_fast_div(a.chunks);
        const int nb = dw_row_blocks(p);
        if (p.FY == 3) launch_rows<3, 2>(s, pl, a);
        else if (nb == 2) launch_rows<5, 2>(s, pl, a);
        else launch_rows<5, 3>(s, pl, a);
        CHIP_CHECK(hipGetLastError());
        return;
    }
    if (fast && masked && !raw) {
        a.div_ohw = make_fast_div((uint32_t)a.OHW), a.div_ow = make_fast_div((uint32_t)a.OW);
        const bool plain = epi.calib && !fast->fused;
        // A clamp on the dequantised value has its branch-free form where the chip holds all workgroups at once.  (The run-time form was
        // 1 to 10 % slower than before, with the division's branch.)  Stride 2, with the branch, without it, branch-free: 32 x 192 x 28x28 4.86,
        // 4.90 and 3.92 us, 16 x 96 x 112x112 (1176 workgroups) 8.14, 8.78 and 7.44, 64 x 576 x 28x28 (1764) 11.1, 11.8 and 9.7.  With more
        // the waves of the slower form run into each other less, and memory is the bound: 40 x 96 x 112x112 (2940) 15.6, 15.8 and 16.3, 128
        // images 38.8, 39.3 and 43.6 (37.4 at the rate of a large copy).
        if (plain && pl.one_round && fast->has_wqf && fast->iqf_one && fast->clamp_folded) hipLaunchKernelGGL(conv_dw3x3_kernel<EPI_KIND_CLAMPQ>, grid, dim3(256), 0, s, a);
        else if (plain && !fast->has_wqf && fast->relu_folded) hipLaunchKernelGGL(conv_dw3x3_kernel<EPI_KIND_RELU>, grid, dim3(256), 0, s, a);
        else if (plain && !fast->has_wqf && fast->act == CLDNN_HIP_ACT_NONE) hipLaunchKernelGGL(conv_dw3x3_kernel<EPI_KIND_LINEAR>, grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL(conv_dw3x3_kernel<EPI_KIND_FAST>, grid, dim3(256), 0, s, a);
        CHIP_CHECK(hipGetLastError());
        return;
    }
    const int lds = p.FY * p.FX * 16;
    if (p.in_dt == CLDNN_HIP_U8) hipLaunchKernelGGL(conv_dw_kernel<true>, grid, dim3(pl.block), lds, s, a);
    else hipLaunchKernelGGL(conv_dw_kernel<false>, grid, dim3(pl.block), lds, s, a);
    CHIP_CHECK(hipGetLastError());
}

}  // namespace chip
