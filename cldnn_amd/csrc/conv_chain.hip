// Host side of the convolution chain kernel: eligibility, LDS image of the weights, launch.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "conv_coop_kernel.h"
#include "conv_dwcoop_kernel.h"

namespace chip {

namespace {

enum { ROW_P64_F64_FOR_DWCHAIN = 4 };  // the 64x64 LDS-staged row: same 64-row unit order, any feature count (K padded with zeros)
enum { ROW_WSL_P64_FOR_CHAIN = 14 };  // the 64-feature weights-stationary row: its packed stream is the LDS image's unit order
enum { CHAIN_MAX_LDS = 160 * 1024 };

int epilogue_kind(const ChainStageIn& s)
{
    const FastEpi& f = *s.fe;
    int kind = EPI_KIND_FAST;
    if (f.has_wqf && f.iqf_one && f.clamp_folded && !f.fused && !f.fc && s.epi->calib) kind = EPI_KIND_CLAMPQ;
    if (!f.has_wqf && s.epi->calib && !f.fc) {
        if (!f.fused && f.relu_folded) kind = EPI_KIND_RELU;
        if (!f.fused && f.act == CLDNN_HIP_ACT_NONE) kind = EPI_KIND_LINEAR;
        if (f.fused && f.act == CLDNN_HIP_ACT_NONE && f.eltw_relu_folded && s.epi->eltw_calib && !f.conv_sat) kind = EPI_KIND_FUSED;
        if (f.fused && f.act == CLDNN_HIP_ACT_NONE && f.eltw_act == CLDNN_HIP_ACT_NONE && !f.eltw_relu_folded) kind = EPI_KIND_SUMLIN;
    }
    return kind;
}

struct Instance {
    int nt, d, sp0, sp1, sp2, e0, e1, e2;
    bool u8;  // of the residual
    void (*launch)(hipStream_t, const ChainArgs&, int, int);
};
#define CHAIN_INSTANCE(NT, D, SP0, SP1, SP2, E0, E1, E2, U8) \
    {NT, D, SP0, SP1, SP2, E0, E1, E2, U8, &launch_chain_instance<NT, D, SP0, SP1, SP2, E0, E1, E2, U8>}
// What is compiled: the tails of ResNet bottlenecks with 64 mid features (3x3 -> expansion [+ residual] -> next
// reduction), residual fused or not; and pairs of an expansion to 256 features and a first stage with 3 or 9 K-steps, such as
// a 1x1 from 192 or 576 features (the 3x3 over 64, also 9, runs on conv_coop_kernel.h): 56x56 at batch 32 13.7 and 18.2 us
// against 18.9 and 23.8 in two launches, equal at batch 1.
const Instance g_instances[] = {
    CHAIN_INSTANCE(1, 3, 1, 4, 1, EPI_KIND_RELU, EPI_KIND_FUSED, EPI_KIND_RELU, true),
    CHAIN_INSTANCE(2, 3, 1, 4, 0, EPI_KIND_RELU, EPI_KIND_FUSED, EPI_KIND_RELU, true),
    CHAIN_INSTANCE(1, 3, 1, 4, 1, EPI_KIND_RELU, EPI_KIND_FUSED, EPI_KIND_RELU, false),
    CHAIN_INSTANCE(2, 3, 1, 4, 0, EPI_KIND_RELU, EPI_KIND_FUSED, EPI_KIND_RELU, false),
    CHAIN_INSTANCE(1, 3, 1, 4, 1, EPI_KIND_RELU, EPI_KIND_RELU, EPI_KIND_RELU, false),
    CHAIN_INSTANCE(2, 3, 1, 4, 0, EPI_KIND_RELU, EPI_KIND_RELU, EPI_KIND_RELU, false),
};

const Instance* find_instance(const ChainPlan& pl)
{
    for (const Instance& i : g_instances)
        if (i.nt == pl.nt && i.d == pl.depth && i.sp0 == pl.sp[0] && i.sp1 == pl.sp[1] && i.sp2 == pl.sp[2] && i.e0 == pl.epi[0]
            && i.e1 == pl.epi[1] && (pl.stages < 3 || i.e2 == pl.epi[2]) && i.u8 == (pl.eltw_u8 != 0))
            return &i;
    return nullptr;
}

}  // namespace

std::string chain_plan(const ChainStageIn* st, int n, int cus, ChainPlan* out)
{
    ChainPlan pl{};
    if (n < 2 || n > CHAIN_MAX_STAGES) return "a chain has two or three stages";
    pl.stages = n;
    const ConvProblem& p0 = *st[0].p;
    for (int k = 0; k < n; ++k) {
        const ConvProblem& p = *st[k].p;
        const std::string at = "stage " + std::to_string(k) + ": ";
        if (!st[k].fast) return at + "needs the short int8 epilogue";
        if (st[k].fe->f32) return at + "float output is not chained";
        if (st[k].fe->fc) return at + "the fully_connected form is not chained";
        const bool dw0 = k == 0 && st[0].dw_wmask != nullptr;
        if (p.groups != 1 && !dw0) return at + "grouped convolution";
        if (p.in_t.format != CLDNN_HIP_FMT_FS_B_YX_FSV16 || p.out_t.format != CLDNN_HIP_FMT_FS_B_YX_FSV16) return at + "needs fs_b_yx_fsv16";
        if (st[0].dw_wmask == nullptr && (p.IFM % 64 != 0 || p.OFM % 64 != 0)) return at + "feature counts must be multiples of 64";
        if (st[0].dw_wmask != nullptr && k < 2 && p.IFM % 16 != 0) return at + "a depthwise chain needs feature counts in multiples of 16 up to the projection";
        if (st[k].fe->fused && p.eltw_t.format != CLDNN_HIP_FMT_FS_B_YX_FSV16) return at + "unblocked residual";
        if (tensor_elems(p.out_t) >= (1ull << 31) || tensor_elems(p.in_t) >= (1ull << 31)) return at + "tensor of 2 GiB or more";
        if (k > 0) {
            const ConvProblem& q = *st[k - 1].p;
            if (p.FY != 1 || p.FX != 1 || p.sy != 1 || p.sx != 1 || p.py != 0 || p.px != 0) return at + "only the first stage may be wider than 1x1";
            if (p.IFM != q.OFM || p.B != q.B || p.IH != q.OH || p.IW != q.OW) return at + "does not read the previous stage's result";
            if (p.in_dt != q.out_dt) return at + "input type differs from the previous stage's output type";
        }
        pl.sp[k] = (p.OFM + 63) / 64;
        pl.epi[k] = epilogue_kind(st[k]);
    }
    if (!conv_border_covers(p0)) return "stage 0: the input needs a zero border as wide as the padding";
    if (p0.dy != 1 || p0.dx != 1) return "stage 0: dilation";
    pl.m_total = (int64_t)p0.B * p0.OH * p0.OW;
    if (st[0].dw_wmask) {
        // ---- depthwise first stage: granules of 16 pixels
        if (p0.FY != 3 || p0.FX != 3) return "stage 0: the depthwise stage of a chain is 3x3";
        if (st[0].fe->fused) return "stage 0: a fused depthwise stage is not chained";
        if (pl.sp[1] > 3) return "stage 1: the projection behind a depthwise stage has at most 192 features";
        pl.dw = 1;
        pl.waves = 4, pl.nt = 1;
        pl.granules = (int)((pl.m_total + 15) / 16);
        pl.units = 0;
        int vec = 0;
        for (int k = 0; k < n; ++k) {
            if (k > 0) {
                MfmaPlan mp{};
                try {
                    mp = mfma_plan(*st[k].p, ROW_P64_F64_FOR_DWCHAIN, cus, true);
                } catch (const error& e) {
                    return "stage " + std::to_string(k) + ": " + e.what();
                }
                pl.unit0[k] = pl.units, pl.kstride[k] = mp.ksteps;
                pl.units += pl.sp[k] * mp.ksteps;
            }
            pl.vec0[k] = vec;
            vec += 4 * pl.sp[k] * 64;
        }
        pl.ksteps0 = pl.sp[0];  // K-steps the depthwise stage delivers to stage 1
        // The waves of a workgroup share a granule where granules are few, from two K-steps on (a single one occupies one wave
        // of four).  Against one granule per wave with the weights in LDS, and separate launches where that form does not apply:
        // 14x14, 384-64-384 11.1 -> 6.9 us at 392 granules, 16.2 -> 14.6 at 784, but 19.2 -> 26.7 at 1568; 576-96-576 (only
        // separate launches otherwise) 27.3 -> 19.3 us at 784 granules and 40 -> 34.6 at 1568.  Fewer K-steps: two granules a CU.
        // Wide projections are taken up to the K-steps and spans whose partial sums and vectors would fit into LDS: beyond, a
        // wave walks over two K-steps and more.
        const bool block = pl.epi[0] == EPI_KIND_CLAMPQ && (pl.epi[1] == EPI_KIND_LINEAR || pl.epi[1] == EPI_KIND_SUMLIN)
                           && (n < 3 || pl.epi[2] == EPI_KIND_CLAMPQ) && !st[1].fe->split_valid;
        const bool small = (pl.m_total + 15) / 16 <= (int64_t)cus * (pl.ksteps0 < 6 ? 2 : (pl.sp[1] == 1 ? 4 : 8));
        const int deep = pl.ksteps0 <= 8 ? std::max(4, pl.ksteps0) : std::min(8, (pl.ksteps0 + 1) / 2);
        const bool shared = block && small && pl.ksteps0 >= 2 && (deep * 4 + 1) * pl.sp[1] * 1024 + vec * 4 <= CHAIN_MAX_LDS;
        // (the other form has two units of 32 features of projection at most)
        if (pl.sp[1] > 1 && !shared)
            return "stage 1: a projection of more than 64 features is chained in the forms of a MobileNet block, on small planes and from 65 mid "
                   "features on only, where partial sums and vectors fit into LDS";
        for (int k = 0; k < n; ++k) pl.u32[k] = (st[k].p->OFM + 31) / 32;
        if (shared) {
            pl.coop = 1, pl.nt = 1;
            const int frags = 2 * pl.u32[1], k1 = pl.sp[1], sp2 = n > 2 ? pl.sp[2] : 0;
            pl.dwc_w1 = 2 * pl.ksteps0 * DWCOOP_UNIT_BYTES, pl.dwc_w2 = pl.dwc_w1 + pl.ksteps0 * frags * 1024;
            pl.dwc_v0 = pl.dwc_w2 + k1 * sp2 * 4096, pl.dwc_v1 = pl.dwc_v0 + pl.ksteps0 * DWCOOP_VEC0_BYTES;
            pl.dwc_v2 = pl.dwc_v1 + frags * DWCOOP_VEC1_BYTES;
            pl.img_bytes = pl.dwc_v2 + sp2 * DWCOOP_VEC0_BYTES;
            // a wave for every K-step and every fragment of the projection
            pl.waves = std::min((int)DWCOOP_MAX_WAVES, std::max(4, std::max(pl.ksteps0, frags)));
            // two granules to a workgroup cost 1.3 us more than one (the weights are fetched once), which pays where the
            // workgroups of one would not all be resident: 576-96-576 at 392 granules 12.3 -> 10.3 us, 384-64-384 6.8 -> 8.1
            pl.nt = pl.granules > cus * (DWCOOP_MAX_WAVES / pl.waves) && pl.ksteps0 <= 9 && pl.waves <= 10 ? 2 : 1;
            pl.granules = (int)((pl.m_total + 16 * pl.nt - 1) / (16 * pl.nt));
            pl.lds_bytes = pl.nt * (pl.ksteps0 + k1) * 1024 + pl.waves * DWCOOP_OWN * 16;
            // up to four (more change nothing): 576-160-960 at four granules 8.4 -> 6.7 us, 960-160-960 8.9 -> 8.4
            pl.dwc_parts = std::max(1, std::min(std::min(sp2, 4), cus / pl.granules));
            pl.grid = (pl.granules * pl.dwc_parts + 7) / 8 * 8;
            pl.dwc_rounds = pl.ksteps0 > (k1 < 3 ? 9 : 15);
            std::snprintf(pl.name, sizeof(pl.name), "conv_dwchain<%d stages,p%d shared by %d waves,mid %d%s,spans %d-%d,parts %d>", n, 16 * pl.nt, pl.waves, p0.OFM,
                          pl.dwc_rounds ? " in rounds" : "", pl.sp[1], sp2, pl.dwc_parts);
            *out = pl;
            return std::string();
        }
        // units of 32 features (conv_dwchain_kernel.h)
        pl.units = pl.u32[0] + 2 * ((pl.u32[0] + 1) / 2 * pl.u32[1] + (n > 2 ? pl.u32[2] : 0));  // kilobytes of weights
        pl.lds_bytes = pl.img_bytes = pl.units * 1024 + vec * 4;
        if (pl.lds_bytes > CHAIN_MAX_LDS) return "the weights of the chain (" + std::to_string(pl.lds_bytes / 1024) + " KiB) do not fit into LDS";
        // workgroups a CU holds at once: by LDS, and by registers (128 with a projection of 32 features, 142 with 64, 256 in
        // the run-time form).  The grid is what is resident, so that no workgroup waits for a slot.
        const int per_cu = std::min(!block ? 2 : (pl.u32[1] == 1 ? 4 : 3), CHAIN_MAX_LDS / pl.lds_bytes);
        int grid = cus * per_cu / 8 * 8;
        const int wanted = ((pl.granules + 3) / 4 + 7) / 8 * 8;  // at least one granule per wave
        if (grid > wanted) grid = wanted;
        if (grid < 8) grid = 8;
        pl.grid = grid;
        std::snprintf(pl.name, sizeof(pl.name), "conv_dwchain<%d stages,p%d,mid %d,spans %d-%d>", n, 16 * pl.nt, p0.OFM, pl.sp[1], n > 2 ? pl.sp[2] : 0);
        *out = pl;
        return std::string();
    }
    pl.nt = n > 2 ? 1 : 2, pl.waves = chain_waves(pl.nt);
    pl.granules = (int)((pl.m_total + 16 * pl.nt - 1) / (16 * pl.nt));
    // K-steps of every stage as the weights-stationary row packs them
    MfmaPlan mp[3]{};
    for (int k = 0; k < n; ++k) {
        ConvProblem q = *st[k].p;
        try {
            mp[k] = mfma_plan(q, ROW_WSL_P64_FOR_CHAIN, cus, true);
        } catch (const error&) {
            // K beyond what that row keeps in LDS: only the K-step count is wanted here
            mp[k] = MfmaPlan{};
            mp[k].ksteps = (q.FY * q.FX * ((q.IFM + 15) / 16) + 3) / 4;
            mp[k].wsl_depth = 0;
        }
        if (k > 0 && mp[k].ksteps < pl.sp[k - 1]) return "stage " + std::to_string(k) + ": fewer K-steps than the previous stage has spans";
    }
    // everything in LDS, independent waves
    {
        pl.units = 0;
        int vec = 0;
        for (int k = 0; k < n; ++k) {
            pl.unit0[k] = pl.units, pl.kstride[k] = mp[k].ksteps;
            pl.units += pl.sp[k] * mp[k].ksteps;
            pl.vec0[k] = vec;
            vec += 4 * pl.sp[k] * 64;
        }
        // The weights in the registers of eight waves that share a granule: chains of two stages, and of three up to four
        // granules per CU (with more, one granule per wave needs fewer instructions a pixel; conv_coop_kernel.h).  Inside ResNet-50,
        // one granule per wave / shared: 588 granules 9.6 / 7.9 us, 784 9.9 / 9.0, 980 10.2 / 9.4, 1568 11.6 / 14.1, 1960 12.4 / 14.6.
        const bool block = p0.FY == 3 && p0.FX == 3 && pl.sp[0] == 1 && p0.IFM == 64 && pl.sp[1] == 4 && (n < 3 || pl.sp[2] == 1)
                           && pl.epi[0] == EPI_KIND_RELU && (pl.epi[1] == EPI_KIND_RELU || pl.epi[1] == EPI_KIND_FUSED)
                           && (n < 3 || pl.epi[2] == EPI_KIND_RELU);
        const int granules = (int)((pl.m_total + 15) / 16);
        if (block && (n == 2 || granules <= 4 * cus)) {
            pl.coop = 1, pl.nt = 1, pl.waves = 8;
            pl.granules = granules;
            pl.img_bytes = pl.units * 4096 + vec * 4;
            pl.lds_bytes = (n > 2 ? 2 : 1) * 32 * 1024 + 1024 + vec * 4;
            pl.grid = std::min(cus * 2 / 8 * 8, (granules + 7) / 8 * 8);
            std::snprintf(pl.name, sizeof(pl.name), "conv_chain<%d stages,p16 shared by 8 waves,spans %d-%d-%d,epi %d-%d-%d>", n, pl.sp[0], pl.sp[1], n > 2 ? pl.sp[2] : 0,
                          pl.epi[0], pl.epi[1], n > 2 ? pl.epi[2] : -1);
            *out = pl;
            return std::string();
        }
        pl.depth = mp[0].wsl_depth, pl.ksteps0 = mp[0].ksteps;
        pl.eltw_u8 = pl.epi[1] == EPI_KIND_FUSED && st[1].fe->eltw_u8;
        pl.lds_bytes = pl.img_bytes = pl.units * 4096 + vec * 4;
        if (mp[0].wsl_depth > 0 && pl.lds_bytes <= CHAIN_MAX_LDS && find_instance(pl)) {
            const int per_cu = pl.lds_bytes * 2 <= CHAIN_MAX_LDS ? 2 : 1;
            int grid = cus * per_cu / 8 * 8;
            const int wanted = ((pl.granules + pl.waves - 1) / pl.waves + 7) / 8 * 8;  // at least one granule per wave
            if (grid > wanted) grid = wanted;
            if (grid < 8) grid = 8;
            pl.grid = grid;
            std::snprintf(pl.name, sizeof(pl.name), "conv_chain<%d stages,p%d,d%d,spans %d-%d-%d,epi %d-%d-%d>", n, 16 * pl.nt, pl.depth,
                          pl.sp[0], pl.sp[1], pl.sp[2], pl.epi[0], pl.epi[1], n > 2 ? pl.epi[2] : -1);
            *out = pl;
            return std::string();
        }
    }
    if (mp[0].wsl_depth <= 0 || pl.lds_bytes > CHAIN_MAX_LDS)
        return "the weights of the chain (" + std::to_string(pl.units * 4) + " KiB) do not fit into LDS";
    return "no compiled instance for this chain shape";
}

size_t chain_packed_bytes(const ChainPlan& pl) { return (size_t)pl.img_bytes + 4096; }

static void fill_stage(ChainStage& c, const ChainStageIn& in, const ChainPlan& pl, int k, void* out, const void* eltw)
{
    const ConvProblem& p = *in.p;
    c.out = out;
    c.eltw = eltw;
    CHIP_REQUIRE(!in.fe->fused || c.eltw, CLDNN_HIP_INVALID_ARG, "fused stage of a chain without its second input");
    c.OFM = p.OFM;
    c.out_off = (int32_t)p.out_p.off, c.out_pb = (int32_t)p.out_p.pb, c.out_pf = (int32_t)p.out_p.pf, c.out_py = (int32_t)p.out_p.py;
    c.el_off = (int32_t)p.eltw_p.off, c.el_pb = (int32_t)p.eltw_p.pb, c.el_pf = (int32_t)p.eltw_p.pf;
    c.el_py = (int32_t)p.eltw_p.py * p.esy, c.el_px = 16 * p.esx;  // a strided residual: the shortcut sub-sampled in place
    c.xor_mask = p.in_dt == CLDNN_HIP_U8 ? 0x80808080u : 0u;
    c.unit0 = pl.unit0[k], c.kstride = pl.kstride[k], c.vec0 = pl.vec0[k];
    c.fe = *in.fe;
    c.epi = *in.epi;
}

static void launch_dwcoop(hipStream_t s, const ChainStageIn* st, const ChainPlan& pl, const void* packed_dev, const void* in,
                          void* const* outs, const void* const* eltws)
{
    const ConvProblem& p0 = *st[0].p;
    const ConvProblem& p1 = *st[1].p;
    DwCoopArgs a{};
    a.in = (const int8_t*)in, a.img = (const int8_t*)packed_dev, a.eltw = eltws ? (const int8_t*)eltws[1] : nullptr;
    a.w1 = pl.dwc_w1, a.w2 = pl.dwc_w2, a.v0 = pl.dwc_v0, a.v1 = pl.dwc_v1, a.v2 = pl.dwc_v2;
    a.el_off = (int32_t)p1.eltw_p.off, a.el_pb = (int32_t)p1.eltw_p.pb, a.el_pf = (int32_t)p1.eltw_p.pf;
    a.el_py = (int32_t)p1.eltw_p.py * p1.esy, a.el_px = 16 * p1.esx;
    a.M = (uint32_t)pl.m_total;
    a.OHW = p0.OH * p0.OW, a.OW = p0.OW;
    a.div_ohw = make_fast_div((uint32_t)a.OHW), a.div_ow = make_fast_div((uint32_t)a.OW);
    a.in_off = (int32_t)p0.in_p.off - p0.py * (int32_t)p0.in_p.py - p0.px * 16;
    a.in_pb = (int32_t)p0.in_p.pb, a.in_pf = (int32_t)p0.in_p.pf;
    a.row = p0.sy * (int32_t)p0.in_p.py, a.col = p0.sx * 16, a.tap_dy = (int32_t)p0.in_p.py;
    a.CB = (p0.OFM + 15) / 16, a.KS = pl.ksteps0, a.F1 = 2 * pl.u32[1], a.SP2 = pl.stages > 2 ? pl.sp[2] : 0;
    a.waves = pl.waves, a.parts = pl.dwc_parts;
    a.div_parts = make_fast_div((uint32_t)pl.dwc_parts);
    const FastEpi &f0 = *st[0].fe, &f1 = *st[1].fe;
    const bool sum = pl.epi[1] == EPI_KIND_SUMLIN;
    CHIP_REQUIRE(!sum || a.eltw, CLDNN_HIP_INVALID_ARG, "fused stage of a chain without its second input");
    a.clamp_m0 = f0.act_m, a.clamp_n0 = f0.act_n;
    a.lo1 = f1.lo, a.hi1 = f1.hi, a.eltw_u8 = f1.eltw_u8;
    a.conv_lo = f1.conv_sat ? f1.conv_lo : -INFINITY, a.conv_hi = f1.conv_sat ? f1.conv_hi : INFINITY;
    if (pl.stages > 2) a.clamp_m2 = st[2].fe->act_m, a.clamp_n2 = st[2].fe->act_n;
    for (int k = 0; k < pl.stages; ++k) {
        const ConvProblem& p = *st[k].p;
        CoopStage& c = a.st[k];
        c.out = (int8_t*)outs[k];
        c.off = (int32_t)p.out_p.off, c.pb = (int32_t)p.out_p.pb, c.pf = (int32_t)p.out_p.pf, c.py = (int32_t)p.out_p.py;
        c.ofm = p.OFM, c.xor_mask = p.in_dt == CLDNN_HIP_U8 ? 0x80808080u : 0u;
    }
#define DWCOOP_LAUNCH(K1, KM, DEEP, NG)                                                                               \
    {                                                                                                                 \
        if (pl.stages > 2 && sum) launch_dwcoop_instance<K1, KM, DEEP, NG, true, true>(s, a, pl.grid, pl.lds_bytes);  \
        else if (pl.stages > 2) launch_dwcoop_instance<K1, KM, DEEP, NG, true, false>(s, a, pl.grid, pl.lds_bytes);   \
        else if (sum) launch_dwcoop_instance<K1, KM, DEEP, NG, false, true>(s, a, pl.grid, pl.lds_bytes);             \
        else launch_dwcoop_instance<K1, KM, DEEP, NG, false, false>(s, a, pl.grid, pl.lds_bytes);                     \
    }
    // registers for the K-steps of a projection fragment: the next larger number compiled, or rounds
    const int k1 = pl.sp[1];
    if (pl.nt == 2) {
        if (k1 == 1) DWCOOP_LAUNCH(1, 9, false, 2)
        else if (k1 == 2) DWCOOP_LAUNCH(2, 9, false, 2) else DWCOOP_LAUNCH(3, 9, false, 2)
    } else if (pl.dwc_rounds) {
        if (k1 == 1) DWCOOP_LAUNCH(1, 9, true, 1)
        else if (k1 == 2) DWCOOP_LAUNCH(2, 9, true, 1) else DWCOOP_LAUNCH(3, 8, true, 1)
    } else if (k1 == 1 && a.KS <= 3) DWCOOP_LAUNCH(1, 3, false, 1) else if (k1 == 1 && a.KS <= 6) DWCOOP_LAUNCH(1, 6, false, 1)
    else if (k1 == 1) DWCOOP_LAUNCH(1, 9, false, 1) else if (k1 == 2 && a.KS <= 6) DWCOOP_LAUNCH(2, 6, false, 1) else if (k1 == 2) DWCOOP_LAUNCH(2, 9, false, 1)
    else if (a.KS <= 9) DWCOOP_LAUNCH(3, 9, false, 1) else DWCOOP_LAUNCH(3, 15, false, 1)
#undef DWCOOP_LAUNCH
    CHIP_CHECK(hipGetLastError());
}

static void launch_coop(hipStream_t s, const ChainStageIn* st, const ChainPlan& pl, const void* packed_dev, const void* in,
                        void* const* outs, const void* const* eltws)
{
    const ConvProblem& p0 = *st[0].p;
    const ConvProblem& p1 = *st[1].p;
    CoopConvArgs a{};
    a.in = (const int8_t*)in, a.img = (const int8_t*)packed_dev, a.eltw = eltws ? (const int8_t*)eltws[1] : nullptr;
    a.vec_bytes = pl.units * 4096;
    a.vec_quads = (pl.img_bytes - a.vec_bytes) / 16;
    a.el_off = (int32_t)p1.eltw_p.off, a.el_pb = (int32_t)p1.eltw_p.pb, a.el_pf = (int32_t)p1.eltw_p.pf;
    a.el_py = (int32_t)p1.eltw_p.py * p1.esy, a.el_px = 16 * p1.esx;
    a.M = (uint32_t)pl.m_total;
    a.OHW = p0.OH * p0.OW, a.OW = p0.OW;
    a.div_ohw = make_fast_div((uint32_t)a.OHW), a.div_ow = make_fast_div((uint32_t)a.OW);
    a.in_off = (int32_t)p0.in_p.off - p0.py * (int32_t)p0.in_p.py - p0.px * 16;
    a.in_pb = (int32_t)p0.in_p.pb, a.in_pf = (int32_t)p0.in_p.pf;
    a.row = p0.sy * (int32_t)p0.in_p.py, a.col = p0.sx * 16, a.tap_dy = (int32_t)p0.in_p.py;
    a.gpw = pl.granules / pl.grid, a.grem = pl.granules % pl.grid;
    a.div_parts = make_fast_div((uint32_t)pl.grid);
    const bool sum = pl.epi[1] == EPI_KIND_FUSED;
    CHIP_REQUIRE(!sum || a.eltw, CLDNN_HIP_INVALID_ARG, "fused stage of a chain without its second input");
    for (int k = 0; k < pl.stages; ++k) {
        const ConvProblem& p = *st[k].p;
        CoopConvStage& c = a.st[k];
        c.out = (int8_t*)outs[k];
        c.off = (int32_t)p.out_p.off, c.pb = (int32_t)p.out_p.pb, c.pf = (int32_t)p.out_p.pf, c.py = (int32_t)p.out_p.py;
        c.xor_mask = p.in_dt == CLDNN_HIP_U8 ? 0x80808080u : 0u;
        c.unit0 = pl.unit0[k], c.kstride = pl.kstride[k], c.vec0 = pl.vec0[k];
        c.hi = st[k].fe->hi, c.eltw_u8 = st[k].fe->eltw_u8;
    }
    if (pl.stages > 2 && sum) launch_coop_instance<true, true>(s, a, pl.grid, pl.lds_bytes);
    else if (pl.stages > 2) launch_coop_instance<true, false>(s, a, pl.grid, pl.lds_bytes);
    else if (sum) launch_coop_instance<false, true>(s, a, pl.grid, pl.lds_bytes);
    else launch_coop_instance<false, false>(s, a, pl.grid, pl.lds_bytes);
    CHIP_CHECK(hipGetLastError());
}

static void launch_dwchain(hipStream_t s, const ChainStageIn* st, const ChainPlan& pl, const void* packed_dev, const void* in,
                           void* const* outs, const void* const* eltws)
{
    const ConvProblem& p0 = *st[0].p;
    DwChainArgs a{};
    a.in = (const int8_t*)in;
    a.img = (const v4i*)packed_dev;
    a.quads = pl.img_bytes / 16;
    a.U0 = pl.u32[0], a.KS = (a.U0 + 1) / 2, a.U2 = pl.stages > 2 ? pl.u32[2] : 0;
    a.w1 = a.U0 * 64, a.w2 = a.w1 + a.KS * pl.u32[1] * 128, a.vec = a.w2 + a.U2 * 128;
    a.n0 = pl.sp[0] * 64, a.n1 = pl.sp[1] * 64, a.n2 = pl.stages > 2 ? pl.sp[2] * 64 : 0;
    a.gpw = pl.granules / pl.grid, a.grem = pl.granules % pl.grid;
    a.div_wgs = make_fast_div((uint32_t)pl.grid);
    a.M = (uint32_t)pl.m_total;
    a.OHW = p0.OH * p0.OW, a.OW = p0.OW;
    a.div_ohw = make_fast_div((uint32_t)a.OHW), a.div_ow = make_fast_div((uint32_t)a.OW);
    a.in_off = (int32_t)p0.in_p.off - p0.py * (int32_t)p0.in_p.py - p0.px * 16;
    a.in_pb = (int32_t)p0.in_p.pb, a.in_pf = (int32_t)p0.in_p.pf;
    a.row = p0.sy * (int32_t)p0.in_p.py, a.col = p0.sx * 16, a.tap_dy = (int32_t)p0.in_p.py;
    a.CB = (p0.OFM + 15) / 16;
    for (int k = 0; k < pl.stages; ++k) fill_stage(a.st[k], st[k], pl, k, outs[k], eltws ? eltws[k] : nullptr);
    // the branch-free epilogue forms of a MobileNet block (clamp on the dequantised value, linear projection, clamp), else
    // the run-time form for every stage
    constexpr int CQ = EPI_KIND_CLAMPQ, LIN = EPI_KIND_LINEAR, SUM = EPI_KIND_SUMLIN, ANY = EPI_KIND_FAST;
    const bool ends = pl.epi[0] == CQ && (pl.stages < 3 || pl.epi[2] == CQ);
    const bool block = ends && pl.epi[1] == LIN, block_sum = ends && pl.epi[1] == SUM;  // projection without / with the block's sum
    bool flip = false;
    for (int k = 0; k < pl.stages; ++k) flip = flip || st[k].p->in_dt == CLDNN_HIP_U8;
#define DWCHAIN_LAUNCH(P1, HAS2, FLIP)                                                                          \
    {                                                                                                           \
        if (block) launch_dwchain_instance<P1, HAS2, FLIP, CQ, LIN, CQ>(s, a, pl.grid, pl.lds_bytes);           \
        else if (block_sum) launch_dwchain_instance<P1, HAS2, FLIP, CQ, SUM, CQ>(s, a, pl.grid, pl.lds_bytes);  \
        else launch_dwchain_instance<P1, HAS2, true, ANY, ANY, ANY>(s, a, pl.grid, pl.lds_bytes);               \
    }
#define DWCHAIN_STAGES(P1, FLIP)                          \
    {                                                     \
        if (pl.stages > 2) DWCHAIN_LAUNCH(P1, true, FLIP) \
        else DWCHAIN_LAUNCH(P1, false, FLIP)              \
    }
    if (pl.u32[1] == 1 && flip) DWCHAIN_STAGES(1, true)
    else if (pl.u32[1] == 1) DWCHAIN_STAGES(1, false)
    else if (flip) DWCHAIN_STAGES(2, true)
    else DWCHAIN_STAGES(2, false)
#undef DWCHAIN_STAGES
#undef DWCHAIN_LAUNCH
    CHIP_CHECK(hipGetLastError());
}

void chain_pack_weights(const ChainStageIn* st, const ChainPlan& pl, int cus, const int8_t* const* w, const ChainVectors* vec,
                        int8_t* packed)
{
    std::memset(packed, 0, chain_packed_bytes(pl));
    // feature of row r of fragment mt in a unit of 32, and of byte b of lane kq in (half h of) a K-step
    auto row = [](int r, int mt) { return 16 * ((r >> 2) & 1) + 8 * (r >> 3) + 4 * mt + (r & 3); };
    auto col = [](int kq, int b) { return 32 * (b >> 3) + 16 * (kq & 1) + 8 * (kq >> 1) + (b & 7); };
    // fragments of a 1x1 stage behind a depthwise one: [K-step][unit][mt]
    auto fragments = [&](int k, int ksteps, int units, int8_t* at) {
        const int ofm = st[k].p->OFM, ifm = st[k].p->IFM;
        for (int ks = 0; ks < ksteps; ++ks)
            for (int u = 0; u < units; ++u)
                for (int mt = 0; mt < 2; ++mt)
                    for (int lane = 0; lane < 64; ++lane)
                        for (int b = 0; b < 16; ++b, ++at) {
                            const int f = u * 32 + row(lane & 15, mt), c = ks * 64 + col(lane >> 4, b);
                            if (f < ofm && c < ifm) *at = w[k][(size_t)f * ifm + c];
                        }
        return at;
    };
    if (pl.coop && pl.dw) {
        const int mid = st[0].p->OFM, sp2 = pl.stages > 2 ? pl.sp[2] : 0;
        // byte (s / 2) * 4 + 2 (s % 2) + mt of (unit, tap half, row)
        for (int u = 0; u < 2 * pl.ksteps0; ++u)
            for (int half = 0; half < 2; ++half)
                for (int r = 0; r < 16; ++r)
                    for (int s5 = 0; s5 < DWCHAIN_STEPS; ++s5)
                        for (int mt = 0; mt < 2; ++mt) {
                            const int ch = u * 32 + row(r, mt), tap = 2 * s5 + half;
                            if (ch < mid && tap < 9) packed[((size_t)(u * 2 + half) * 16 + r) * 16 + (s5 >> 1) * 4 + 2 * (s5 & 1) + mt] = w[0][(size_t)ch * 9 + tap];
                        }
        fragments(1, pl.ksteps0, pl.u32[1], packed + pl.dwc_w1);
        if (sp2) fragments(2, pl.sp[1], 2 * sp2, packed + pl.dwc_w2);
        // factors that are absent are one, or the output quantization factor
        auto value = [&](int k, int kind, int f) {
            const void* src[3] = {vec[k].acc_init, vec[k].calib, k == 1 ? vec[k].eltw_calib : vec[k].wqf};
            const float fill = kind == 1 && st[k].epi->oqf_on ? st[k].epi->oqf : 1.0f;
            int32_t bits = 0;
            if (kind > 0) std::memcpy(&bits, &fill, 4);
            if (src[kind] && f < st[k].p->OFM) std::memcpy(&bits, (const int32_t*)src[kind] + f, 4);
            return bits;
        };
        for (int k = 0; k < pl.stages; k += 2) {
            int32_t* v = reinterpret_cast<int32_t*>(packed + (k ? pl.dwc_v2 : pl.dwc_v0));
            for (int sp = 0; sp < pl.sp[k]; ++sp)
                for (int kind = 0; kind < 3; ++kind)
                    for (int f = 0; f < 64; ++f) *v++ = value(k, kind, sp * 64 + f);
        }
        int32_t* v = reinterpret_cast<int32_t*>(packed + pl.dwc_v1);
        for (int i = 0; i < 2 * pl.u32[1]; ++i)
            for (int kind = 0; kind < 3; ++kind)
                for (int kq = 0; kq < 4; ++kq)
                    for (int j = 0; j < 4; ++j) *v++ = value(1, kind, (i >> 1) * 32 + row(kq * 4 + j, i & 1));
        return;
    } else if (pl.dw) {
        const int mid = st[0].p->OFM;
        for (int u = 0; u < pl.u32[0]; ++u)
            for (int lane = 0; lane < 64; ++lane)
                for (int s5 = 0; s5 < DWCHAIN_STEPS; ++s5)
                    for (int mt = 0; mt < 2; ++mt) {
                        const int ch = u * 32 + row(lane & 15, mt), tap = 2 * s5 + (lane >> 5);
                        if (ch < mid && tap < 9) packed[((size_t)u * 64 + lane) * 16 + (s5 >> 1) * 4 + 2 * (s5 & 1) + mt] = w[0][(size_t)ch * 9 + tap];
                    }
        int8_t* at = packed + (size_t)pl.u32[0] * 1024;
        for (int k = 1; k < pl.stages; ++k) at = fragments(k, (pl.u32[k - 1] + 1) / 2, pl.u32[k], at);
    }
    const size_t unit_bytes = (size_t)pl.units * (pl.dw ? 1024 : 4096);
    // per-feature vectors behind the weight units: per stage init, calib, eltw_calib, wqf, spans * 64 entries each
    int32_t* v = reinterpret_cast<int32_t*>(packed + unit_bytes);
    const float one = 1.0f;
    int32_t one_bits;
    std::memcpy(&one_bits, &one, 4);
    for (int k = 0; k < pl.stages; ++k) {
        const int n = pl.sp[k] * 64, ofm = st[k].p->OFM;
        const void* src[4] = {vec[k].acc_init, vec[k].calib, vec[k].eltw_calib, vec[k].wqf};
        for (int kind = 0; kind < 4; ++kind) {
            int32_t* dst = v + pl.vec0[k] + kind * n;
            // without calibration factors the epilogue multiplies by the output quantization factor (or by one)
            int32_t fill = kind == 0 ? 0 : one_bits;
            if (kind == 1 && !src[kind] && st[k].epi->oqf_on) std::memcpy(&fill, &st[k].epi->oqf, 4);
            for (int f = 0; f < n; ++f) dst[f] = fill;
            if (src[kind]) std::memcpy(dst, src[kind], (size_t)ofm * 4);
        }
    }
    if (pl.dw) return;
    for (int k = 0; k < pl.stages; ++k) {
        const MfmaPlan mp = mfma_plan(*st[k].p, ROW_WSL_P64_FOR_CHAIN, cus, true);
        std::vector<int8_t> buf(mp.packed_bytes);
        std::vector<int32_t> ktab(mp.ktab_bytes / sizeof(int32_t));
        mfma_pack_weights(*st[k].p, mp, w[k], buf.data(), ktab.data());
        std::memcpy(packed + (size_t)pl.unit0[k] * 4096, buf.data(), (size_t)pl.sp[k] * mp.ksteps * 4096);
    }
}

void launch_conv_chain(hipStream_t s, const ChainStageIn* st, const ChainPlan& pl, const void* packed_dev, const void* in,
                       void* const* outs, const void* const* eltws)
{
    if (pl.coop && !pl.dw) return launch_coop(s, st, pl, packed_dev, in, outs, eltws);
    if (pl.coop) return launch_dwcoop(s, st, pl, packed_dev, in, outs, eltws);
    if (pl.dw) return launch_dwchain(s, st, pl, packed_dev, in, outs, eltws);
    const ConvProblem& p0 = *st[0].p;
    ChainArgs a{};
    a.in = (const int8_t*)in;
    a.wpk = (const v4i*)packed_dev;
    a.units = pl.units;
    a.vec_quads = (pl.lds_bytes - pl.units * 4096) / 16;
    a.granules = pl.granules;
    a.gpw = pl.granules / pl.grid, a.grem = pl.granules % pl.grid;
    a.div_wgs = make_fast_div((uint32_t)pl.grid);
    a.M = (uint32_t)pl.m_total;
    a.OHW = p0.OH * p0.OW, a.OW = p0.OW;
    a.div_ohw = make_fast_div((uint32_t)a.OHW), a.div_ow = make_fast_div((uint32_t)a.OW);
    a.sy = p0.sy, a.sx = p0.sx, a.py = p0.py, a.px = p0.px;
    a.in_off = (int32_t)p0.in_p.off, a.in_pb = (int32_t)p0.in_p.pb, a.in_pf = (int32_t)p0.in_p.pf, a.in_py = (int32_t)p0.in_p.py;
    a.ksteps0 = pl.ksteps0, a.CB = (p0.IFM + 15) / 16, a.FX = p0.FX, a.FY = p0.FY;
    a.tap_dy = p0.dy * (int32_t)p0.in_p.py, a.tap_dx = p0.dx * 16;
    for (int k = 0; k < pl.stages; ++k) fill_stage(a.st[k], st[k], pl, k, outs[k], eltws ? eltws[k] : nullptr);
    const Instance* inst = find_instance(pl);
    CHIP_REQUIRE(inst, CLDNN_HIP_ERROR, "chain without a compiled instance");
    inst->launch(s, a, pl.grid, pl.lds_bytes);
    CHIP_CHECK(hipGetLastError());
}

}  // namespace chip
