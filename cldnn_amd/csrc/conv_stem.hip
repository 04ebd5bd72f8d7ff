// Host side of the first-layer kernel: which layers it takes, the split into workgroups, weights, launch.
#include <algorithm>
#include <cstring>

#include "conv_stem_kernel.h"

namespace chip {

namespace {

int ceil_div(int a, int b) { return (a + b - 1) / b; }

int epilogue_of(const FastEpi& f, const Epilogue& e)
{
    if (f.f32 || f.fc || f.fused || f.split_valid || !e.calib) return EPI_KIND_GENERIC;
    if (f.has_wqf) return f.iqf_one && f.clamp_folded ? EPI_KIND_CLAMPQ : EPI_KIND_GENERIC;
    return f.relu_folded ? EPI_KIND_RELU : f.act == CLDNN_HIP_ACT_NONE ? EPI_KIND_LINEAR : EPI_KIND_GENERIC;
}

// Output rows of a wave (pooling) or workgroup: more of them read less of the image twice, fewer make more workgroups.  Four, as long
// as there is a workgroup for every CU; us by rows 1 / 2 / 4 / 8: ResNet-50's pooled layer at batch 1 (image in host memory) 10.4 /
// 11.5 / 15.4 / 21.7, batch 32 18.0 / 16.4 / 15.1 / 19.4, batch 128 52.7 / 40.3 / 36.7 / 44.2; VGG-16's at batch 1 9.1 / 10.7 / 13.1 /
// 18.2, batch 16 22.3 / 19.3 / 17.6 / 20.3.
int rows_of(int64_t groups_of_four, int cus)
{
    int r = 4;
    while (r > 1 && groups_of_four * 4 / r < cus) r /= 2;
    return r;
}

}  // namespace

StemPlan stem_plan(const ConvProblem& p, const FastEpi& f, const Epilogue& e, int cus)
{
    StemPlan s{};
    const int nch = ceil_div(p.FX, 4), kind = epilogue_of(f, e);
    const cldnn_hip_tensor& i = p.in_t;
    if (i.format != CLDNN_HIP_FMT_BFYX || p.out_t.format != CLDNN_HIP_FMT_FS_B_YX_FSV16 || p.IFM > 4 || p.OFM > 64 || p.groups != 1) return s;
    if (p.dy != 1 || p.dx != 1 || p.FY * nch > 16 || p.IW < 4 || kind == EPI_KIND_GENERIC) return s;
    if (tensor_elems(p.in_t) >= (1ull << 31) || tensor_elems(p.out_t) >= (1ull << 31)) return s;
    if (p.pooled && kind != EPI_KIND_RELU) return s;
    s.epi = kind, s.nch = nch, s.ksteps = ceil_div(p.FY * nch, 4), s.frags_f = p.OFM <= 32 ? 2 : 4;
    const int OH = p.pooled ? p.out_t.y : p.OH, OW = p.pooled ? p.out_t.x : p.OW;
    if (p.pooled) {
        const int strips = ceil_div(OW, 15);
        s.tiles = strips > 2 ? 4 : strips;
        s.col_groups = ceil_div(strips, 4), s.wg_cols = ceil_div(OW, s.col_groups), s.tile_cols = ceil_div(s.wg_cols, s.tiles);
        s.wave_rows = rows_of((int64_t)p.B * s.col_groups * ceil_div(OH * s.tiles, 16), cus);
        s.wg_rows = s.wave_rows * (4 / s.tiles);
        s.lds_rows = 2 * s.wg_rows * p.sy + p.FY;
        s.pitch = (2 * ((s.tiles - 1) * s.tile_cols + 15) + 1) * p.sx + nch * 4;
    } else {
        s.col_groups = ceil_div(p.OW, 256), s.frags = ceil_div(ceil_div(p.OW, s.col_groups), 16), s.wg_cols = s.frags * 16;
        s.col_groups = ceil_div(p.OW, s.wg_cols);
        s.wg_rows = rows_of((int64_t)p.B * s.col_groups * ceil_div(OH, 4), cus);
        s.lds_rows = (s.wg_rows - 1) * p.sy + p.FY;
        s.pitch = (s.wg_cols - 1) * p.sx + nch * 4;
    }
    s.pitch = ceil_div(s.pitch, 4) * 4;
    s.row_groups = ceil_div(OH, s.wg_rows);
    s.lds_bytes = s.lds_rows * s.pitch * 4 + (p.pooled ? s.frags_f * 128 : 0);
    if (s.lds_bytes > 64 * 1024) return s;  // strides and filters beyond those of a first layer
    s.total = p.B * s.row_groups * s.col_groups, s.grid = ceil_div(s.total, 8) * 8;
    s.packed_bytes = (size_t)s.ksteps * s.frags_f * 1024;
    s.ok = 1;
    return s;
}

void stem_pack_weights(const ConvProblem& p, const StemPlan& s, const int8_t* w, int8_t* packed)
{
    for (int k = 0; k < s.ksteps; ++k)
        for (int f = 0; f < s.frags_f; ++f)
            for (int lane = 0; lane < 64; ++lane)
                for (int j = 0; j < 16; ++j, ++packed) {
                    const int r = lane & 15, c = k * 4 + (lane >> 4), fy = c / s.nch, fx = (c - fy * s.nch) * 4 + (j >> 2), ch = j & 3;
                    const int o = s.frags_f == 4 ? 16 * (r >> 2) + 4 * f + (r & 3) : 16 * ((r >> 2) & 1) + 8 * (r >> 3) + 4 * f + (r & 3);
                    *packed = o < p.OFM && fy < p.FY && fx < p.FX && ch < p.IFM ? w[(((size_t)o * p.IFM + ch) * p.FY + fy) * p.FX + fx] : 0;
                }
}

void launch_conv_stem(hipStream_t st, const ConvProblem& p, const StemPlan& s, const void* packed, const int32_t* acc_init, const Epilogue& epi,
                      const FastEpi& fe, const void* in, void* out)
{
    StemArgs a{};
    a.in = (const uint8_t*)in, a.wpk = (const v4i*)packed, a.acc_init = acc_init, a.out = (int8_t*)out;
    a.fe = fe;
    a.epi = {epi.wqf, epi.calib, epi.eltw_calib, (const float*)epi.bias, epi.oqf, epi.oqf_on};
    a.in_off = (int32_t)p.in_p.off, a.in_pb = (int32_t)p.in_p.pb, a.in_pf = (int32_t)p.in_p.pf, a.in_py = (int32_t)p.in_p.py;
    a.IFM = p.IFM, a.IH = p.IH, a.IW = p.IW;
    a.out_off = (int32_t)p.out_p.off, a.out_pb = (int32_t)p.out_p.pb, a.out_pf = (int32_t)p.out_p.pf, a.out_py = (int32_t)p.out_p.py;
    a.OFM = p.OFM, a.OH = p.OH, a.OW = p.OW, a.PH = p.out_t.y, a.PW = p.out_t.x;
    a.sy = p.sy, a.sx = p.sx, a.py = p.py, a.px = p.px, a.FY = p.FY, a.nch = s.nch;
    a.B = p.B, a.row_groups = s.row_groups, a.col_groups = s.col_groups, a.total = s.total;
    a.div_rows = make_fast_div((uint32_t)s.row_groups), a.div_cols = make_fast_div((uint32_t)s.col_groups);
    a.wg_rows = s.wg_rows, a.wg_cols = s.wg_cols, a.wave_rows = s.wave_rows, a.tiles = s.tiles, a.tile_cols = s.tile_cols;
    a.lds_rows = s.lds_rows, a.pitch = s.pitch, a.frags = s.frags;
    a.div_frags = make_fast_div((uint32_t)std::max(1, s.frags));
    a.xor_mask = p.in_dt == CLDNN_HIP_U8 ? 0x80808080u : 0u;
#define STEM_LAUNCH(F, KS, EPI, POOL)                                                                                                             \
    {                                                                                                                                             \
        if (p.sx == 2) hipLaunchKernelGGL((conv_stem_kernel<F, KS, EPI, POOL, true>), dim3(s.grid), dim3(256), s.lds_bytes, st, a);               \
        else hipLaunchKernelGGL((conv_stem_kernel<F, KS, EPI, POOL, false>), dim3(s.grid), dim3(256), s.lds_bytes, st, a);                             \
    }
#define STEM_EPI(F, KS)                                                               \
    {                                                                                 \
        if (p.pooled) STEM_LAUNCH(F, KS, EPI_KIND_RELU, true)                         \
        else if (s.epi == EPI_KIND_RELU) STEM_LAUNCH(F, KS, EPI_KIND_RELU, false)     \
        else if (s.epi == EPI_KIND_LINEAR) STEM_LAUNCH(F, KS, EPI_KIND_LINEAR, false) \
        else STEM_LAUNCH(F, KS, EPI_KIND_CLAMPQ, false)                               \
    }
#define STEM_STEPS(F)                       \
    {                                       \
        if (s.ksteps == 1) STEM_EPI(F, 1)   \
        else if (s.ksteps == 2) STEM_EPI(F, 2) \
        else if (s.ksteps == 3) STEM_EPI(F, 3) \
        else STEM_EPI(F, 4)                 \
    }
    if (s.frags_f == 2) STEM_STEPS(2)
    else STEM_STEPS(4)
#undef STEM_STEPS
#undef STEM_EPI
#undef STEM_LAUNCH
    CHIP_CHECK(hipGetLastError());
}

}  // namespace chip
