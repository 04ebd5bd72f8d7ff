// Instances of the split-K kernel with one scalar activation offset per K-step, the form for gathered activations, and the
// gather itself.
//
// A fully_connected over a plane (7x7 in VGG-16): a lane's 16 activation bytes of a K-step lie in 64 different cache lines,
// and every workgroup would pull all of them through its L1 again.  A small kernel first puts the activations into fragment
// order (1 KB per K-step and pixel fragment, sign flip applied), which the main kernel then reads as it reads the weights.
#include <mutex>

#include "conv_ksplit_kernel.h"

namespace chip {

// size of the gather scratch that lives in the code object (for callers that may not allocate)
enum { GEMV_STATIC_SCRATCH_BYTES = 4 << 20 };

// activations in fragment order: bpk[(ptile * (ksteps + GEMV_SLACK) + ks) * 64 + lane]
__global__ void __launch_bounds__(256) gemv_gather_kernel(MfmaArgs a)
{
    const int lane = threadIdx.x & 63;
    const int ks = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int ptile = blockIdx.y;
    if (ks >= a.ksteps) return;
    const int kq = lane >> 4;
    const int l16 = lane & 15;
    const uint32_t m = (uint32_t)ptile * 16 + l16;
    const PixelPos pp = pixel_pos(a, m < a.M ? m : 0);
    const uint32_t boff = (uint32_t)(a.in_off + (int)pp.b * a.in_pb + ((int)pp.oy * a.sy - a.py) * a.in_py
                                     + ((int)pp.ox * a.sx - a.px) * 16 + kq * a.in_pf);
    const v4i xm = {(int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask};
    const v4i v = *reinterpret_cast<const v4i*>(a.in + a.ktab[ks * 4] + boff);
    const_cast<v4i*>(a.bpk)[((size_t)ptile * (a.ksteps + GEMV_SLACK) + ks) * 64 + lane] = v ^ xm;
}

void launch_ksplit_lanes(hipStream_t s, const KsplitArgs& a, int ft, int pt, int grid, int epi);

static KsplitArgs ksplit_args(const MfmaArgs& m)
{
    KsplitArgs a{};
    a.in = m.in + (m.in_off - m.py * m.in_py - m.px * 16);
    a.inside = (uint32_t)(m.py * m.in_py + m.px * 16);
    a.wpk = m.wpk, a.bpk = m.bpk, a.acc_init = m.acc_init, a.out = m.out, a.eltw = (const int8_t*)m.eltw, a.raw = m.raw, a.origin = m.origin;
    a.mtiles = m.mtiles, a.ftiles = m.ofm_tiles;
    a.features_outer = m.by_features != 0, a.die_bits = m.by_features == 2 ? 0 : 3;
    a.inner = a.features_outer ? a.mtiles : a.ftiles;
    a.div_inner = make_fast_div((uint32_t)a.inner);
    a.M = m.M, a.OFM = m.OFM, a.OHW = m.OHW, a.OW = m.OW, a.OH = m.OH, a.IH = m.IH, a.IW = m.IW;
    a.div_ohw = make_fast_div((uint32_t)m.OHW), a.div_ow = make_fast_div((uint32_t)m.OW);
    a.ksteps = m.ksteps, a.kper = m.kper, a.kwaves = m.kwaves;
    a.in_pb = m.in_pb, a.in_row = m.sy * m.in_py, a.in_col = m.sx * 16, a.in_pf = m.in_pf;
    a.taps = m.FX * m.FY, a.FX = m.FX, a.tap_dy = m.tap_dy, a.tap_dx = m.tap_dx, a.last_group = m.CB - 4;
    a.div_taps = make_fast_div((uint32_t)a.taps), a.div_fx = make_fast_div((uint32_t)m.FX), a.div_cb = make_fast_div((uint32_t)m.CB);
    a.out_off = m.out_off, a.out_pb = m.out_pb, a.out_pf = m.out_pf, a.out_py = m.out_py, a.out_f = m.out_f;
    a.el_off = m.el_off, a.el_pb = m.el_pb, a.el_pf = m.el_pf, a.el_row = m.esy * m.el_py, a.el_col = m.esx * 16;
    a.xor_mask = m.xor_mask;
    a.CB = m.CB, a.kchunks = m.kchunks, a.checked = m.checked, a.sy = m.sy, a.sx = m.sx, a.py = m.py, a.px = m.px, a.dil_y = m.dil_y, a.dil_x = m.dil_x;
    a.fe = m.fe, a.epi = m.epi;
    return a;
}

void launch_ksplit(hipStream_t s, const MfmaArgs& m, int ft, int pt, int grid, bool lanes, int epi)
{
    const KsplitArgs a = ksplit_args(m);
    if (m.bpk) {
        hipLaunchKernelGGL(gemv_gather_kernel, dim3((m.ksteps + 3) / 4, m.mtiles * pt), dim3(256), 0, s, m);
        if (pt == 1) launch_ksplit_instance<1, 1, ADDR_GATHERED>(s, a, grid, epi);
        else launch_ksplit_instance<1, 2, ADDR_GATHERED>(s, a, grid, epi);
    } else if (lanes) {
        launch_ksplit_lanes(s, a, ft, pt, grid, epi);
    } else {
        launch_ksplit_tile<ADDR_UNIFORM>(s, a, ft, pt, grid, epi);
    }
}

size_t gemv_gather_bytes(int mtiles, int ksteps) { return ((size_t)mtiles * (ksteps + GEMV_SLACK)) * 1024; }

// ---- gather scratch that nobody allocates: one array per device, part of the loaded code object.
// Every device the library runs on holds its own copy at its own address until the process ends.  In host code the
// array's name is only a handle for hipGetSymbolAddress; kernels and copies take the address that call returns.
static __device__ __align__(256) unsigned char scratch[GEMV_STATIC_SCRATCH_BYTES];

size_t gemv_static_scratch_bytes() { return GEMV_STATIC_SCRATCH_BYTES; }

// Device address of `scratch` on `device`, which the caller has made current.  Looked up once per device.
void* gemv_static_scratch(int device)
{
    enum { MAX_DEVICES = 64 };
    static std::mutex guard;
    static void* address[MAX_DEVICES] = {};
    CHIP_REQUIRE(device >= 0 && device < MAX_DEVICES, CLDNN_HIP_INVALID_ARG, "device index beyond the static scratch table");
    std::lock_guard<std::mutex> lock(guard);
    if (!address[device]) {
        int current = -1;
        CHIP_CHECK(hipGetDevice(&current));
        CHIP_REQUIRE(current == device, CLDNN_HIP_ERROR, "the static scratch is looked up with its device current");
        void* ptr = nullptr;
        CHIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        CHIP_REQUIRE(ptr, CLDNN_HIP_DEVICE_ERROR, "hipGetSymbolAddress returned no address for the static scratch");
        address[device] = ptr;
    }
    return address[device];
}

}  // namespace chip
