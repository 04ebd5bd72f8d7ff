// Host side of the wide 1x1 kernel: which layers it takes, weights, launch.
#include <algorithm>

#include "conv_point_kernel.h"

namespace chip {

static int ceil_div(int a, int b) { return (a + b - 1) / b; }

// From a workgroup for every second CU on, with sums for every CU, and with nine tenths of the features of the tiles in use.  Us by
// workgroups, row of the table / this kernel: 512 -> 256 + 1024 from 28x28 128 6.5 / 5.4, 248 8.5 / 6.1; 1024 -> 256 at 14x14 104 6.3 / 6.7,
// 200 8.6 / 6.9; 512 -> 256 at 28x28 56 4.0 / 5.1, 152 6.8 / 5.3, 1232 20.6 / 17.2; with a sum 256 -> 1024 at 14x14 104 4.8 / 5.5, 200 6.0 /
// 5.7, 392 8.0 / 7.3, and 512 -> 2048 at 7x7 200 7.2 / 6.5 alone, but 8.5 / 9.0 between other layers.  640 output features, five sixths in
// use: 13.2 / 12.7, 39.0 / 39.2; 128, a half: 15.9 / 21.1.
// Up to 1024 input features: a block's successor is requested 600 clocks ahead, enough where the weights lie in L2, and a workgroup reads
// all of its 256 features' (2048 -> 512 at batch 128 alone 13.7 / 12.2, between other layers, its weights in memory, 14.3 / 18.4).
bool point_pays(const ConvProblem& p, const PointPlan& s, int cus)
{
    return p.IFM <= 1024 && s.total * (s.kind == EPI_KIND_FUSED ? 1 : 2) > cus && p.OFM * 10 >= s.ftiles * POINT_FEATURES * 9;
}

PointPlan point_plan(const ConvProblem& p, const FastEpi& f, const Epilogue& e)
{
    PointPlan s{};
    if (p.FY != 1 || p.FX != 1 || p.py != 0 || p.px != 0 || p.groups != 1 || p.by_span || p.plain_out || p.IFM % 256) return s;
    if (p.in_t.format != CLDNN_HIP_FMT_FS_B_YX_FSV16 || p.out_t.format != CLDNN_HIP_FMT_FS_B_YX_FSV16 || !conv_border_covers(p)) return s;
    if (f.f32 || f.fc || f.has_wqf || !e.calib || p.pooled) return s;
    if (f.fused) {
        if (f.act != CLDNN_HIP_ACT_NONE || !f.eltw_relu_folded || !e.eltw_calib || f.conv_sat || f.split_valid) return s;
        if (p.eltw_t.format != CLDNN_HIP_FMT_FS_B_YX_FSV16 || tensor_elems(p.eltw_t) >= (1ull << 31)) return s;
        s.kind = EPI_KIND_FUSED;
    } else {
        if (!f.relu_folded && f.act != CLDNN_HIP_ACT_NONE) return s;
        s.kind = f.relu_folded && !f.split_valid ? EPI_KIND_RELU : EPI_KIND_LINEAR;
        if (f.split_valid && f.act != CLDNN_HIP_ACT_NONE && !f.relu_folded) return s;
    }
    if (tensor_elems(p.in_t) >= (1ull << 31) || tensor_elems(p.out_t) >= (1ull << 31)) return s;
    const int64_t m = (int64_t)p.B * p.OH * p.OW;
    if (m >= (1 << 30)) return s;
    s.jobs = p.IFM / 128, s.spans = ceil_div(p.OFM, 32), s.ftiles = ceil_div(p.OFM, POINT_FEATURES);
    if ((m + 63) / 64 * s.ftiles >= (1 << 30)) return s;
    s.total = (int)((m + POINT_PIXELS - 1) / POINT_PIXELS) * s.ftiles;
    s.grid = ceil_div(s.total, 8) * 8;
    s.lds_bytes = 3 * 8 * POINT_PIXELS * 16 + 3 * 1024;
    s.packed_bytes = (size_t)s.spans * (p.IFM / 32) * 1024;
    s.ok = 1;
    return s;
}

void point_pack_weights(const ConvProblem& p, const PointPlan& s, const int8_t* w, int8_t* packed)
{
    for (int span = 0; span < s.spans; ++span)
        for (int block = 0; block < p.IFM / 32; ++block)
            for (int lane = 0; lane < 64; ++lane)
                for (int k = 0; k < 16; ++k, ++packed) {
                    // the order of the rows gives a lane 16 consecutive features
                    const int r = lane & 31, o = span * 32 + 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
                    *packed = o < p.OFM ? w[(size_t)o * p.IFM + block * 32 + (lane >> 5) * 16 + k] : 0;
                }
}

void launch_conv_point(hipStream_t st, const ConvProblem& p, const PointPlan& s, const void* packed, const int32_t* acc_init, const Epilogue& epi,
                       const FastEpi& fe, const void* in, const void* eltw, void* out, int32_t* raw)
{
    PointArgs a{};
    a.in = (const int8_t*)in, a.wpk = (const v4i*)packed, a.acc_init = acc_init, a.calib = epi.calib, a.ecal = epi.eltw_calib;
    a.eltw = (const int8_t*)eltw, a.out = (int8_t*)out, a.raw = raw, a.fe = fe;
    a.in_off = (int32_t)p.in_p.off, a.in_pb = (int32_t)p.in_p.pb, a.in_pf = (int32_t)p.in_p.pf;
    a.in_row = p.sy * (int32_t)p.in_p.py, a.in_col = p.sx * 16;
    a.out_off = (int32_t)p.out_p.off, a.out_pb = (int32_t)p.out_p.pb, a.out_pf = (int32_t)p.out_p.pf, a.out_py = (int32_t)p.out_p.py;
    if (s.kind == EPI_KIND_FUSED) {
        a.el_off = (int32_t)p.eltw_p.off, a.el_pb = (int32_t)p.eltw_p.pb, a.el_pf = (int32_t)p.eltw_p.pf;
        a.el_row = p.esy * (int32_t)p.eltw_p.py, a.el_col = 16 * p.esx;
    }
    a.OFM = p.OFM, a.OHW = p.OH * p.OW, a.OW = p.OW, a.M = (uint32_t)(p.B * a.OHW);
    a.div_ohw = make_fast_div((uint32_t)a.OHW), a.div_ow = make_fast_div((uint32_t)a.OW);
    a.ftiles = s.ftiles, a.total = s.total, a.spans = s.spans, a.jobs = s.jobs, a.div_ftiles = make_fast_div((uint32_t)s.ftiles);
    a.xor_mask = p.in_dt == CLDNN_HIP_U8 ? 0x80808080u : 0u;
#define POINT_LAUNCH(EPI)                                                                                                   \
    {                                                                                                                       \
        if (a.xor_mask) hipLaunchKernelGGL((conv_point_kernel<EPI, true>), dim3(s.grid), dim3(256), s.lds_bytes, st, a);       \
        else hipLaunchKernelGGL((conv_point_kernel<EPI, false>), dim3(s.grid), dim3(256), s.lds_bytes, st, a);                 \
    }
    if (s.kind == EPI_KIND_FUSED) POINT_LAUNCH(EPI_KIND_FUSED)
    else if (s.kind == EPI_KIND_RELU) POINT_LAUNCH(EPI_KIND_RELU)
    else POINT_LAUNCH(EPI_KIND_LINEAR)
#undef POINT_LAUNCH
    CHIP_CHECK(hipGetLastError());
}

}  // namespace chip
