// Host side of the kernel whose waves split K over a patch in LDS: which layers it takes, the tile of pixels, weights, launch.
#include <algorithm>
#include <mutex>

#include "conv_plane_kernel.h"

namespace chip {

namespace {

int ceil_div(int a, int b) { return (a + b - 1) / b; }

struct Form {
    int wide, np, nl;  // 1: 128 features, 2: 64 features and two tiles of pixels, all of K to a wave; fragments (rows of a group), loads of 64 positions
};
constexpr Form FORMS[] = {{0, 4, 4}, {0, 7, 5}, {0, 7, 6}, {1, 7, 5}, {1, 7, 6}, {1, 8, 6}, {2, 7, 6}, {2, 8, 6}};

}  // namespace

static PlanePlan form_plan(const ConvProblem& p, const FastEpi& f, const Epilogue& e, int cus, int wide)
{
    PlanePlan best{};
    if (p.FY != 3 || p.FX != 3 || p.sy != 1 || p.sx != 1 || p.dy != 1 || p.dx != 1 || p.groups != 1 || p.by_span || p.plain_out) return best;
    if (p.in_t.format != CLDNN_HIP_FMT_FS_B_YX_FSV16 || p.out_t.format != CLDNN_HIP_FMT_FS_B_YX_FSV16) return best;
    if (!conv_border_covers(p)) return best;
    if (f.f32 || f.fc || f.fused || f.split_valid || f.has_wqf || !e.calib) return best;
    if (!f.relu_folded && f.act != CLDNN_HIP_ACT_NONE) return best;
    if (p.pooled && (!f.relu_folded || p.OH % 2 || p.OW % 2)) return best;
    if (tensor_elems(p.in_t) >= (1ull << 31) || tensor_elems(p.out_t) >= (1ull << 31)) return best;
    if (p.in_p.py >= (1 << 24) || p.out_p.py >= (1 << 24)) return best;  // 24-bit products
    const int spans = ceil_div(p.OFM, PLANE_FEATURES);
    if (p.IFM % 64) return best;
    double least = 0;
    for (const Form& form : FORMS) {
        if (form.wide != wide || (form.np == 8 ? !p.pooled : p.pooled && form.np % 2)) continue;
        PlanePlan s{};
        s.wide = form.wide, s.jobs = p.IFM / (form.wide ? 32 : 128), s.ftiles = form.wide ? ceil_div(spans, 4 / form.wide) : spans;
        if (!form.wide && (p.IFM % 128 || (s.jobs != 1 && s.jobs % 2))) continue;
        s.strips = ceil_div(p.OW, 32), s.cols = ceil_div(p.OW, s.strips);
        if (p.pooled) s.cols += s.cols % 2;
        s.strips = ceil_div(p.OW, s.cols);
        s.shift = s.cols <= 8 ? 3 : s.cols <= 16 ? 4 : 5;
        const int groups = 32 >> s.shift;
        s.pitch = s.cols + 2, s.positions = groups * (form.np + 2) * s.pitch;
        if (s.positions > form.nl * 64) continue;
        s.image_units = ceil_div(p.OH, form.np) * s.strips;
        if ((int64_t)p.B * s.image_units * spans >= (1 << 30)) continue;
        s.units = p.B * s.image_units;
        s.total = ceil_div(ceil_div(s.units, groups), form.wide == 2 ? 2 : 1) * s.ftiles;
        // (512 bytes: what idle lanes read past the end)
        s.lds_bytes = form.wide ? form.wide * 3 * 2 * s.positions * 16 + 512 : std::max((s.jobs == 1 ? 1 : 2) * 4 * 2 * s.positions * 16 + 512, PLANE_MEET * 4 * 4096);
        // clocks: what a workgroup's matrix instructions take, and what it waits for at its start and its end
        const int resident = s.lds_bytes <= 80 * 1024 ? 2 : 1;
        const int64_t full = s.total / (cus * resident), left = s.total % (cus * resident);
        const double work = form.np * 9 * s.jobs * 32.0, idle = 5000.0;
        const double cost = full * (resident * work + idle) + (left > cus ? 2 * work + idle : left ? work + idle : 0);
        if (best.ok && cost >= least) continue;
        least = cost;
        s.ok = 1, s.np = form.np, s.nl = form.nl, s.spans = spans;
        s.grid = ceil_div(s.total, 8) * 8;
        s.kind = f.relu_folded ? EPI_KIND_RELU : EPI_KIND_LINEAR;
        s.packed_bytes = (size_t)spans * (p.IFM / 32) * 9 * 1024;
        best = s;
    }
    return best;
}

// Narrow form.  Up to a workgroup per CU the launch is one prologue, one loop and one meeting of the sums, and more than half of the CUs
// have to be in it: below that the split-K row is as fast (us by workgroups, row of the table / this kernel: 64 4.2 / 4.9, 128 4.9 /
// 4.9, 192 7.1 / 4.9 for 256 features at 14x14; 64 5.2 / 6.5, 128 6.5 / 6.6, 256 10.5 / 6.6 for 512 at 7x7).  Beyond that workgroups
// take turns: 512 11.8 / 10.1, 768 18.0 / 14.0, 1024 18.9 / 17.4, 2048 30.7 / 32.7 for 256 features, 1024 34.3 / 30.5, 2048 55.3 / 59.5
// for 512.  One block of 32 features to a wave is the least work beside the same fixed cost: 768 12.3 / 10.6, 1024 12.7 / 12.5.
// Wide forms, for which more than five eighths of the CUs have to have a workgroup: 128 features at 28x28, 128 workgroups 8.4 / 8.8,
// 192 12.3 / 9.0, 256 12.7 / 9.4, 384 18.5 / 14.6, 512 18.7 / 16.3; 512 at 28x28, 256 34.3 / 26.6, 512 55.3 / 51.1, 1024 110 / 99.4.
// 64 features at 56x56 128 6.5 / 6.8, 256 9.0 / 7.6, 512 14.1 / 12.0, 1024 21.6 / 21.5, pooled 224 8.0 / 6.3, 448 12.2 / 10.0, 896 19.3 / 17.6;
// at 224x224, pooled, 1568 34.3 / 30.2.  Where a narrow and a wide form would do, the wide one is the faster (192 workgroups: 9.0 against
// 10.6, 13.4 against 14.0, 22.6 against 23.0).
// All compute for lanes, rows and features that do not exist.  Row of the table / this kernel by the share in use, planes of other images
// than those of 224 pixels among them:
//   narrow, more than a workgroup per CU: 0.75 (26 and 13 columns) 8.3 / 7.5, 11.6 / 10.9, 18.7 / 17.5; 0.70 (25) 8.2 / 7.5; 0.64 (24, 12 and 6)
//     8.2 / 7.4, 11.5 / 10.7, 18.3 / 16.9; 0.60 (20) 6.5 / 7.1, 9.0 / 10.3, 12.0 / 14.9; 0.48 (18) 8.9 / 10.2; 0.45 (10 and 5) 9.0 / 10.5, 13.3 / 16.3
//   narrow, up to one: 0.75 (26, 13 and 12) 6.4 / 5.4, 13.8 / 10.0, 7.1 / 4.9; 0.70 6.4 / 5.4; 0.64 to 0.66 6.4 / 5.4, 7.1 / 4.9, 8.8 / 6.7, 13.6 / 9.8; 0.60
//     5.0 / 5.4, 7.1 / 6.4; 0.56 (6) 10.4 / 6.7; 0.52 (10) 4.9 / 4.9; 0.45 7.2 / 6.6, 10.5 / 9.6; 0.39 (5) 6.6 / 6.6; 0.36 (9) 7.2 / 6.5, 10.5 / 9.6
//   wide: 0.75 12.9 / 9.7, 18.7 / 15.0, 33.0 / 26.4; 64 features, 52 columns 8.9 / 7.2; 0.70 12.7 / 9.5, 8.9 / 7.2; 0.64 12.7 / 9.7, 18.2 / 14.7; 0.60
//     8.5 / 8.9, 19.6 / 25.3; 0.45 20.0 / 25.0; 64 output features on the form for 128 14.0 / 20.1 at 56x56, 64 images.
// The lines at 0.76 and 0.70 keep to one side of that: whatever passes them is faster here, and what lies between 0.64 and them would be too.
// Planes of images of 224 pixels have 0.766 and more.
static double used(const ConvProblem& p, const PlanePlan& s)
{
    return (double)p.B * p.OH * p.OW * p.OFM / ((double)s.total * s.np * 32 * PLANE_FEATURES * (s.wide ? 4 : 1));
}

bool plane_pays(const ConvProblem& p, const PlanePlan& s, int cus)
{
    if (s.wide) return s.total * 8 > 5 * cus && used(p, s) > 0.76;
    if (s.total <= cus) return s.total * 2 > cus && used(p, s) > 0.7;
    return s.total <= (s.jobs == 1 ? 3 : 4) * cus && used(p, s) > 0.76;
}

PlanePlan plane_plan(const ConvProblem& p, const FastEpi& f, const Epilogue& e, int cus, int only)
{
    if (only >= 0) return form_plan(p, f, e, cus, only);
    const PlanePlan wide = form_plan(p, f, e, cus, p.OFM <= 64 ? 2 : 1);
    return wide.ok && plane_pays(p, wide, cus) ? wide : form_plan(p, f, e, cus, 0);
}

void plane_pack_weights(const ConvProblem& p, const PlanePlan& s, const int8_t* w, int8_t* packed)
{
    for (int span = 0; span < s.spans; ++span)
        for (int block = 0; block < p.IFM / 32; ++block)
            for (int tap = 0; tap < 9; ++tap)
                for (int lane = 0; lane < 64; ++lane)
                    for (int k = 0; k < 16; ++k, ++packed) {
                        // the order of the rows gives a lane 16 consecutive features
                        const int r = lane & 31, o = span * PLANE_FEATURES + 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
                        const int c = block * 32 + (lane >> 5) * 16 + k;
                        *packed = o < p.OFM ? w[((size_t)o * p.IFM + c) * 9 + tap] : 0;
                    }
}

using PlaneKernel = void (*)(PlaneArgs);
template <PlaneKernel K>
struct Instance {
    static constexpr PlaneKernel kernel = K;
};

template <PlaneKernel K>
static void launch_instance(hipStream_t st, const PlaneArgs& a, const PlanePlan& s)
{
    static std::once_flag once;  // more than 64 KB of LDS has to be allowed
    std::call_once(once, [] { CHIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(K), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024)); });
    hipLaunchKernelGGL(K, dim3(s.grid), dim3(256), s.lds_bytes, st, a);
}

void launch_conv_plane(hipStream_t st, const ConvProblem& p, const PlanePlan& s, const void* packed, const int32_t* acc_init, const Epilogue& epi,
                       const FastEpi& fe, const void* in, void* out, int32_t* raw)
{
    PlaneArgs a{};
    a.in = (const int8_t*)in, a.wpk = (const v4i*)packed, a.acc_init = acc_init, a.calib = epi.calib, a.out = (int8_t*)out, a.raw = raw;
    a.hi = fe.hi, a.lo = fe.lo;
    a.in_pb = (int32_t)p.in_p.pb, a.in_pf = (int32_t)p.in_p.pf, a.in_py = (int32_t)p.in_p.py;
    a.in_off = (int32_t)p.in_p.off - p.py * a.in_py - p.px * 16;
    a.out_off = (int32_t)p.out_p.off, a.out_pb = (int32_t)p.out_p.pb, a.out_pf = (int32_t)p.out_p.pf, a.out_py = (int32_t)p.out_p.py;
    a.OFM = p.OFM, a.OH = p.OH, a.OW = p.OW, a.B = p.B;
    a.spans = s.spans, a.ftiles = s.ftiles, a.total = s.total, a.div_ftiles = make_fast_div((uint32_t)s.ftiles);
    a.units = s.units, a.image_units = s.image_units, a.strips = s.strips, a.cols = s.cols, a.shift = s.shift;
    a.div_image = make_fast_div((uint32_t)s.image_units), a.div_strips = make_fast_div((uint32_t)s.strips);
    a.pitch = s.pitch, a.positions = s.positions;
    a.div_patch = make_small_div((s.np + 2) * s.pitch), a.div_pitch = make_small_div(s.pitch);
    a.jobs = s.jobs, a.kind = s.kind;
    a.xor_mask = p.in_dt == CLDNN_HIP_U8 ? 0x80808080u : 0u;
    auto go = [&](auto flipped, auto plain) {
        if (a.xor_mask) launch_instance<decltype(flipped)::kernel>(st, a, s);
        else launch_instance<decltype(plain)::kernel>(st, a, s);
    };
#define PLANE_NARROW(NP, NL, JOBS, POOL) go(Instance<&conv_plane_kernel<NP, NL, JOBS, POOL, true>>{}, Instance<&conv_plane_kernel<NP, NL, JOBS, POOL, false>>{})
#define PLANE_WIDE(NP, NL, SPANS, POOL) go(Instance<&conv_plane_wide_kernel<NP, NL, SPANS, POOL, true>>{}, Instance<&conv_plane_wide_kernel<NP, NL, SPANS, POOL, false>>{});
#define PLANE_FORM(NP, NL, POOL)                          \
    {                                                     \
        if (s.jobs == 1) PLANE_NARROW(NP, NL, 1, POOL);   \
        else if (s.jobs == 2) PLANE_NARROW(NP, NL, 2, POOL); \
        else PLANE_NARROW(NP, NL, 0, POOL);               \
    }
    if (s.wide == 2 && p.pooled && !raw) PLANE_WIDE(8, 6, 2, true)
    else if (s.wide == 2 && s.np == 8) PLANE_WIDE(8, 6, 2, false)
    else if (s.wide == 2) PLANE_WIDE(7, 6, 2, false)
    else if (s.wide && p.pooled && !raw) PLANE_WIDE(8, 6, 4, true)
    else if (s.wide && s.np == 8) PLANE_WIDE(8, 6, 4, false)
    else if (s.wide && s.nl == 5) PLANE_WIDE(7, 5, 4, false)
    else if (s.wide) PLANE_WIDE(7, 6, 4, false)
    else if (p.pooled && !raw) PLANE_FORM(4, 4, true)
    else if (s.np == 4) PLANE_FORM(4, 4, false)
    else if (s.nl == 5) PLANE_FORM(7, 5, false)
    else PLANE_FORM(7, 6, false)
#undef PLANE_WIDE
#undef PLANE_FORM
#undef PLANE_NARROW
    CHIP_CHECK(hipGetLastError());
}

}  // namespace chip
