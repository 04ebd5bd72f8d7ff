// Nine-tap stride-1 convolutions with the K dimension split over the waves of a workgroup and the input staged once.
//
// The direct-activation kernels fetch an activation fragment for every tap: a tile of 64 pixels x 64 features pulls
// (64 + 64) x K bytes through a CU's L1 (64 bytes a clock), which at 14x14 or 7x7 is most of the launch.  Here a workgroup of
// four waves owns up to 224 output pixels of 32 features, and each wave
//   - takes a quarter of the blocks of 32 input features, for ALL pixels and features of the tile;
//   - copies the pixels its taps reach, of its own block, into its own part of LDS with direct global -> LDS loads, once;
//   - keeps the block's weights in registers (each is used by this wave alone, so they never pass through LDS);
//   - reads a row of pixels from LDS once for the three taps above each other (see below).
// No wave waits for another until the partial sums meet in LDS at the end, where a wave finishes every fourth fragment.
//
// Fragments.  The 32 pixels of a matrix instruction are one row of 1, 2 or 4 groups of 32, 16 or 8 columns; a group is a run of
// NP rows of an image, and fragment i holds row i of every group.  So what tap row fy of fragment i multiplies is what tap row 0
// of fragment i + fy does: one LDS read (1 KB) serves three matrix instructions of 32 clocks.  With pixels numbered through
// the plane instead, every instruction had its own read, four waves of a CU wanted 128 bytes a clock, which is what LDS
// gives, and the loop ran at 42 to 54 clocks an instruction (14x14 x 256 features, batch 32: 7.2 us).  (The 16x16x64 form, two
// instructions to a read, took 48 clocks for the same work with a wave alone on its SIMD.)
//
// Measured, against the tile table's row for the layer: 256 features at 14x14, batch 16 7.1 -> 4.8 us, batch 32 8.9 -> 6.6, batch 128
// 18.6 -> 17.1; 512 at 7x7, batch 32 10.5 -> 6.4; 512 at 14x14, batch 16 13.1 -> 9.2; 512 at 28x28, batch 16 33.6 -> 29.8.  At batch 32
// of the first, 12200 clocks: 2100 until all requests are out, 600 until they have arrived, 5200 in the loop (126 matrix
// instructions: 4030), 4200 in the two meetings of partial sums.
// Since then the arguments come behind one wait (three: the size of the grid and a divisor came in turns of their own) and the first
// job's weights are requested before the addresses of its patch are computed: 256 at 14x14, batch 32, 7.7 -> 7.2 us inside ResNet-50;
// 512 at 28x28, batch 1, 5.2 -> 4.7; the wide form, 256 at 14x14, batch 128, 15.6 -> 15.0.
//
// LDS reads are issued by hand and waited for by count (conv_halo_kernel.h).  A fetch through the scalar unit between them
// only makes a wait longer.
#pragma once
#include "conv_halo_kernel.h"

namespace chip {

enum { PLANE_FEATURES = 32, PLANE_MEET = 4 };

// q / d for q < 512, d < 2048: a 24-bit product and a shift instead of the high half of a 32-bit product
struct SmallDiv {
    uint32_t mul;
    __device__ uint32_t div(uint32_t q) const { return __umul24(q, mul) >> 20; }
};
inline SmallDiv make_small_div(int d) { return {(1u << 20) / (uint32_t)d + 1}; }

struct PlaneArgs {
    const int8_t* in;
    const v4i* wpk;            // [32 features][block of 32 input features][tap][64 lanes]
    const int32_t* acc_init;
    const float* calib;
    int8_t* out;
    int32_t* raw;              // the accumulators instead
    float hi, lo;
    int32_t in_off, in_pb, in_pf, in_py;      // bytes; in_off: of tap (0, 0) of output pixel (0, 0)
    int32_t out_off, out_pb, out_pf, out_py;  // elements; of the pooled tensor where the result is pooled
    int32_t OFM, OH, OW, B;
    int32_t ftiles, total;                    // tiles of features; workgroups
    FastDiv div_ftiles;
    int32_t spans;                            // of 32 features
    int32_t units;                            // groups of the whole batch: [image][NP rows][cols columns]
    FastDiv div_image, div_strips;            // units of an image, of NP rows
    int32_t image_units, strips, cols, shift; // units of an image, strips of columns, their width, log2 of the lanes of a group
    int32_t pitch, positions;                 // of a group's patch: a row; all groups
    SmallDiv div_patch, div_pitch;
    int32_t jobs;                             // blocks of 32 input features of a wave
    int32_t kind;                             // epilogue
    uint32_t xor_mask;
};

// The reads of a job: rows 0 and NP + 1, which serve one instruction each, in turn (two chains of dependent products), then the
// others.  A wave alone on its SIMD takes 41 clocks an instruction, two 35 each; neither more distance between dependent products, nor
// requests between the instructions, nor a fixed place for every read, nor more reads ahead changes that.
template <int NP>
struct PlaneRead {
    static constexpr int count = (NP + 2) * 3;
    static constexpr int row(int r) { return r < 6 ? (r & 1) * (NP + 1) : r / 3 - 1; }
    static constexpr int column(int r) { return r < 6 ? r / 2 : r % 3; }
    static constexpr int place(int r) { return r < 6 ? r & 1 : 0; }  // of its row's address
};

// Which groups a tile of pixels holds, and where their pixels lie.
template <int NP>
struct PlaneTile {
    int unit0, x0, image[4], y0[4];
    __device__ __forceinline__ PlaneTile(const PlaneArgs& a, uint32_t tile)
    {
        unit0 = (int)tile * (32 >> a.shift);
        const uint32_t u = (uint32_t)unit0, b = a.div_image.div(u), r = u - b * (uint32_t)a.image_units, yb = a.div_strips.div(r);
        x0 = (int)(r - yb * (uint32_t)a.strips) * a.cols;
        image[0] = min((int)b, a.B - 1), y0[0] = (int)yb * NP;  // (a tile past the batch's end: the last image)
#pragma unroll
        for (int g = 1; g < 4; ++g) {  // more than one group: one strip.  Past the batch's end the last image again
            const bool next = y0[g - 1] + NP >= a.OH;
            image[g] = min(image[g - 1] + (next ? 1 : 0), a.B - 1), y0[g] = next ? 0 : y0[g - 1] + NP;
        }
    }
    // (values: a choice between places would be one in memory)
    static __device__ __forceinline__ int pick(int v0, int v1, int v2, int v3, uint32_t g)
    {
        const int low = g & 1u ? v1 : v0, high = g & 1u ? v3 : v2;
        return g & 2u ? high : low;
    }
    __device__ __forceinline__ int image_of(uint32_t g) const { return pick(image[0], image[1], image[2], image[3], g); }
    __device__ __forceinline__ int row_of(uint32_t g) const { return pick(y0[0], y0[1], y0[2], y0[3], g); }
    // byte offset of position q of the patch in its slice
    __device__ __forceinline__ uint32_t source(const PlaneArgs& a, uint32_t q) const
    {
        const uint32_t g = a.div_patch.div(q), r = q - __umul24(g, (uint32_t)a.pitch * (NP + 2));
        const uint32_t row = a.div_pitch.div(r), c = r - __umul24(row, a.pitch);
        int base[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) base[i] = image[i] * a.in_pb + y0[i] * a.in_py + x0 * 16;
        // rows and columns past the plane (only pixels that are not stored reach there) read the last ones
        return (uint32_t)pick(base[0], base[1], base[2], base[3], g) + __umul24(min((int)row, a.OH + 1 - row_of(g)), a.in_py) + (uint32_t)min((int)c, a.OW + 1 - x0) * 16u;
    }
};

// NP: fragments.  NL: loads of 64 positions that a slice of the patch takes.  JOBS: 1, 2, or 0 for a larger even number.
// POOL: the maxima over 2x2 windows.  FLIP: u8 activations.
template <int NP, int NL, int JOBS, bool POOL, bool FLIP>
__global__ void __launch_bounds__(256, 2) conv_plane_kernel(PlaneArgs a)
{
    constexpr int RG = NP == 4 ? 6 : 9, MEET = PLANE_MEET;  // few steps to a job: the next patch is read as late as can be
    constexpr int AT_ONCE = NP == 4 ? 4 : 2;                // and requested as early
    constexpr int BUFFERS = JOBS == 1 ? 1 : 2;
    using Read = PlaneRead<NP>;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = lane >> 5;
    const int l32 = lane & 31;
    // everything the loop needs, behind one wait
    asm volatile("" ::"s"(a.in), "s"(a.wpk), "s"(a.in_off), "s"(a.in_pb), "s"(a.in_pf), "s"(a.in_py), "s"(a.total), "s"(a.units), "s"(a.strips), "s"(a.cols), "s"(a.shift),
                 "s"(a.pitch), "s"(a.positions), "s"(a.jobs), "s"(a.xor_mask), "s"(a.acc_init), "s"(a.calib), "s"(a.OH), "s"(a.OW), "s"(a.div_patch.mul), "s"(a.div_pitch.mul), "s"(a.ftiles), "s"(a.div_ftiles.mul), "s"(a.div_ftiles.shift), "s"(gridDim.x));
    // (values of their own, or the compiler fetches the arguments again where they are used)
    const global<int32_t>* first = in_global(a.acc_init);
    const global<float>* factors = in_global(a.calib);
    global_bytes in = in_global(a.in + a.in_off);
    int in_pf = a.in_pf, row_bytes = a.pitch * 16;
    global<int8_t>* out = in_global(a.out);
    global<int32_t>* raw = in_global(a.raw);
    int out_off = a.out_off, out_pb = a.out_pb, out_pf = a.out_pf, out_py = a.out_py, kind = a.kind, OFM = a.OFM, OH = a.OH, units = a.units;
    float hi = a.hi, lo = a.lo;
    asm volatile("" : "+s"(first), "+s"(factors), "+s"(in), "+s"(in_pf), "+s"(row_bytes), "+s"(out), "+s"(raw), "+s"(out_off), "+s"(out_pb), "+s"(out_pf), "+s"(out_py),
                 "+s"(kind), "+s"(OFM), "+s"(OH), "+s"(units), "+s"(hi), "+s"(lo));

    const uint32_t wg = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);  // the grid is a multiple of 8
    if (wg >= (uint32_t)a.total) return;
    // workgroups of one pixel tile on one die: they share the input
    const uint32_t ptile = a.div_ftiles.div(wg), ftile = wg - ptile * (uint32_t)a.ftiles;
    const PlaneTile<NP> tile(a, ptile);

    extern __shared__ __align__(16) unsigned char smem[];
    v4i* lds = reinterpret_cast<v4i*>(smem);

    const int buffer_units = 2 * a.positions, wave_units = wave * BUFFERS * buffer_units;  // of 16 bytes
    global_bytes weights = (global_bytes)(a.wpk + (size_t)(ftile * 4 + (uint32_t)wave) * a.jobs * 9 * 64);
    asm volatile("" : "+s"(weights));
    const uint32_t lane_bytes = (uint32_t)lane * 16u;
    uint32_t src[NL];
    v4i w[BUFFERS][9];
    // request R of a job: the wave's patch, into LDS, then its weights
    constexpr int REQUESTS = 2 * NL + 9;
    auto request = [&](int j, auto buffer, auto rc) {
        constexpr int P = decltype(buffer)::value, R = decltype(rc)::value;
        if constexpr (R < 2 * NL) {
            constexpr int S = R / NL, I = R % NL;
            global_bytes base = in + (int64_t)((wave * a.jobs + j) * 2 + S) * in_pf;
            __builtin_amdgcn_global_load_lds((halo_gptr)(base + src[I]), (halo_lptr)(lds + wave_units + P * buffer_units + S * a.positions + min(I * 64, a.positions - 64)), 16, 0, 0);
        } else if constexpr (R < REQUESTS) {
            w[P][R - 2 * NL] = *(const global<v4i>*)(weights + (uint32_t)(j * 9 + R - 2 * NL) * 1024u + lane_bytes);
        }
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, BUFFERS - 1>;
    // of the first job the weights go out first (in front of the patch, so its arrival is everybody's): the addresses of the patch
    // take a hundred and fifty instructions
    static_for<2 * NL, REQUESTS>([&](auto rc) {
        request(0, B0{}, rc);
        step_fence();
    });
#pragma unroll
    for (int i = 0; i < NL; ++i) src[i] = tile.source(a, (uint32_t)(min(i * 64, a.positions - 64) + lane));  // the last load ends where the patch does
    static_for<0, 2 * NL>([&](auto rc) {
        request(0, B0{}, rc);
        step_fence();
    });

    const uint32_t lane_group = (uint32_t)l32 >> a.shift, column = (uint32_t)l32 & ((1u << a.shift) - 1u);
    const uint32_t here = lds_offset(lds) + ((uint32_t)(wave_units + half * a.positions) + __umul24(lane_group, (uint32_t)a.pitch * (NP + 2)) + column) * 16u;
    v16i acc[NP] = {};
    const v4i xm = {(int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask};
    const int slice = (int)ftile * 2 + half, f0 = slice * 16;
    constexpr int N = POOL ? 8 : 16;  // features a lane finishes
    const int fl = f0 + (POOL ? (wave & 1) * 8 : 0);
    float cal[16] = {}, wq[16] = {};
    v4i init[4] = {};

    // A job, its patch in LDS and its first reads on their way.  Its steps request the next job's operands, and its last ones read
    // the next patch already.
    v4i ring[RG];
    static_assert(Read::count % RG == 0 && REQUESTS <= AT_ONCE * (Read::count - RG + 2), "the ring goes round; all requests are out before the next patch is read");
    uint32_t row[2];
    auto patch_arrived = [] { asm volatile("s_waitcnt vmcnt(9)" ::: "memory"); };  // younger: the weights
    auto read = [&](auto buffer, auto ic) {
        constexpr int P = decltype(buffer)::value, R = decltype(ic)::value, Y = Read::row(R), C = Read::column(R);
        uint32_t& at = row[Read::place(R)];
        if constexpr (C == 0) at = here + (uint32_t)(Y * row_bytes + P * buffer_units * 16);
        lds_read<C * 16>(ring[R % RG], at);
    };
    auto job = [&](int j, auto buffer, auto last) {
        constexpr int P = decltype(buffer)::value;
        constexpr bool LAST = decltype(last)::value;
        using Next = std::integral_constant<int, BUFFERS - 1 - P>;
        static_for<0, Read::count>([&](auto ic) {
            constexpr int R = decltype(ic)::value, Y = Read::row(R), C = Read::column(R);
            constexpr int AHEAD = R + RG - 2;  // the latest read
            lds_wait<(LAST && AHEAD >= Read::count ? Read::count - 1 : AHEAD) - R>(ring[R % RG]);
            v4i x = ring[R % RG];
            if constexpr (FLIP) x ^= xm;
            static_for<0, 3>([&](auto fc) {
                constexpr int F = decltype(fc)::value, I = Y - F;
                if constexpr (I >= 0 && I < NP) acc[I] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[P][F * 3 + C], x, acc[I], 0, 0, 0);
            });
            step_fence();
            if constexpr (!LAST) static_for<0, AT_ONCE>([&](auto rc) { request(j + 1, Next{}, std::integral_constant<int, R * AT_ONCE + decltype(rc)::value>{}); });
            // into the place of the read before: the instructions just issued still read this one
            if constexpr (AHEAD + 1 < Read::count) {
                read(buffer, std::integral_constant<int, AHEAD + 1>{});
            } else if constexpr (!LAST) {
                if constexpr (AHEAD + 1 == Read::count) patch_arrived();
                read(Next{}, std::integral_constant<int, AHEAD + 1 - Read::count>{});
            }
            if constexpr (LAST && R == Read::count / 2) {  // for the end
#pragma unroll
                for (int d = 0; d < N / 4; ++d) {
                    init[d] = *(const global<v4i>*)(first + fl + d * 4);
                    const v4f c = *(const global<v4f>*)(factors + fl + d * 4);
                    cal[d * 4] = c.x, cal[d * 4 + 1] = c.y, cal[d * 4 + 2] = c.z, cal[d * 4 + 3] = c.w;
                }
            }
            step_fence();
        });
    };
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    static_for<0, RG - 1>([&](auto ic) { read(B0{}, ic); });
    if constexpr (JOBS == 0)
        for (int j = 0; j + 2 < a.jobs; j += 2) {
            job(j, B0{}, std::false_type{});
            job(j + 1, B1{}, std::false_type{});
        }
    if constexpr (JOBS != 1) job(a.jobs - 2, B0{}, std::false_type{});
    job(a.jobs - 1, B1{}, std::true_type{});

    // ---------------- the partial sums meet in LDS, four fragments at a time; a wave finishes one of them
    struct {
        FastEpi fe;
    } e;
    e.fe.hi = hi, e.fe.lo = e.fe.lo2 = lo, e.fe.split_valid = 0;
    v4i part[NP][4];
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d) part[i][d] = v4i{acc[i][d * 4], acc[i][d * 4 + 1], acc[i][d * 4 + 2], acc[i][d * 4 + 3]};
    asm volatile("s_nop 7\n\ts_nop 7");  // a result of sixteen registers settles later than one of four
    step_fence();
    mfma_settle(part);
    const int b = tile.image_of(lane_group), yl = tile.row_of(lane_group), x = tile.x0 + (int)column;
    const bool mine = tile.unit0 + (int)lane_group < units && (int)column < a.cols && x < a.OW && f0 < OFM;
    const v4i none = {0, 0, 0, 0};
#pragma unroll
    for (int r0 = 0; r0 < NP; r0 += MEET) {
        __syncthreads();
#pragma unroll
        for (int i = r0; i < (r0 + MEET < NP ? r0 + MEET : NP); ++i)
            if (POOL || i - r0 != wave)
#pragma unroll
                for (int d = 0; d < 4; ++d) lds[((POOL ? i * 4 + wave : (i - r0) * 3 + ((wave - i + r0) & 3) - 1) * 4 + d) * 64 + lane] = part[i][d];
        __syncthreads();
        if constexpr (POOL) {  // a wave takes half the features of two fragments
            static_assert(!POOL || NP == MEET, "two rows of windows");
            const int k = wave >> 1, d0 = (wave & 1) * 2;
            v4i best[4][1] = {{none}, {none}, {none}, {none}};
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                v4i sum[2] = {init[d], init[d]};
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int p = 0; p < 4; ++p) sum[u] += lds[(((2 * k + u) * 4 + p) * 4 + d0 + d) * 64 + lane];
#pragma unroll
                for (int c = 0; c < 4; ++c) best[d][0][c] = max_dpp<0xb1>(max(sum[0][c], sum[1][c]));
            }
            const v4i q = epilogue_fast16<1, EPI_KIND_RELU, 8>(e, best, 0, wq, cal, cal, none, OFM - fl);
            const int y = yl + 2 * k;
            if (mine && y < OH && !(lane & 1))
                *(global<v2i>*)(out + ((uint32_t)(out_off + b * out_pb + slice * out_pf + (x >> 1) * 16 + d0 * 4) + __umul24(y >> 1, out_py))) = v2i{q[0], q[1]};
        } else {
            if (r0 + wave >= NP) continue;
            v4i sum[4][1], others[4][3];
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int p = 0; p < 3; ++p) others[d][p] = lds[((wave * 3 + p) * 4 + d) * 64 + lane];
#pragma unroll
            for (int i = r0; i < (r0 + MEET < NP ? r0 + MEET : NP); ++i)
                if (i - r0 == wave) {
                    keep_branch();
#pragma unroll
                    for (int d = 0; d < 4; ++d) sum[d][0] = part[i][d] + init[d];
                }
#pragma unroll
            for (int d = 0; d < 4; ++d) sum[d][0] += others[d][0] + others[d][1] + others[d][2];
            const int y = yl + r0 + wave;
            const bool ok = mine && y < OH;
            if (raw) {
                keep_branch();
                if (ok)
#pragma unroll
                    for (int c = 0; c < 16; ++c)
                        if (f0 + c < OFM) raw[(((size_t)b * OFM + f0 + c) * OH + y) * a.OW + x] = sum[c >> 2][0][c & 3];
                continue;
            }
            v4i q;
            if (kind == EPI_KIND_RELU) {
                keep_branch();
                q = epilogue_fast16<1, EPI_KIND_RELU>(e, sum, 0, wq, cal, cal, none, OFM - f0);
            } else {
                keep_branch();
                q = epilogue_fast16<1, EPI_KIND_LINEAR>(e, sum, 0, wq, cal, cal, none, OFM - f0);
            }
            if (ok) *(global<v4i>*)(out + ((uint32_t)(out_off + b * out_pb + slice * out_pf + x * 16) + __umul24(y, out_py))) = q;
        }
    }
}

// The same tile of pixels for 128 features, a wave for every 32 of them and all of K: the waves share one patch, a block of 32
// input features after the other through three buffers, and meet at a barrier per block (126 matrix instructions or so for a
// CU's two workgroups), but neither add sums nor copy pixels four times.  A quarter of the workgroups of the form above, so it is for
// layers that have enough of them.  A block's successor is requested during it, into the buffer that was read two blocks ago:
// every wave has left that one when any wave passes the barrier between.  With POOL a wave has both rows of a window.
// SPANS: 4, or 2 for layers of up to 64 features, whose workgroups take two tiles of pixels instead, two waves to each (64 -> 64 at
// 224x224 with pooling, batch 16: 34.3 -> 30.2 us, with half of 128 features idle 52).
template <int NP, int NL, int SPANS, bool POOL, bool FLIP>
__global__ void __launch_bounds__(256, 2) conv_plane_wide_kernel(PlaneArgs a)
{
    using Read = PlaneRead<NP>;
    constexpr int RG = NP == 7 ? 9 : 6, AT_ONCE = 2;
    constexpr int LOADS = (2 * NL + SPANS - 1) / SPANS;  // of a wave: its share of a patch
    constexpr int REQUESTS = LOADS + 9;
    static_assert(Read::count % RG == 0 && REQUESTS <= AT_ONCE * (Read::count - RG + 2), "the ring goes round; all requests are out before the next patch is read");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = lane >> 5;
    const int l32 = lane & 31;
    const int member = wave % SPANS, pair = wave / SPANS;  // of the waves of a tile; which tile
    asm volatile("" ::"s"(a.in), "s"(a.wpk), "s"(a.in_off), "s"(a.in_pb), "s"(a.in_pf), "s"(a.in_py), "s"(a.total), "s"(a.units), "s"(a.strips), "s"(a.cols), "s"(a.shift),
                 "s"(a.pitch), "s"(a.positions), "s"(a.jobs), "s"(a.spans), "s"(a.xor_mask), "s"(a.acc_init), "s"(a.calib), "s"(a.OH), "s"(a.OW), "s"(a.div_patch.mul),
                 "s"(a.div_pitch.mul), "s"(a.ftiles), "s"(a.div_ftiles.mul), "s"(a.div_ftiles.shift), "s"(gridDim.x));
    const global<int32_t>* first = in_global(a.acc_init);
    const global<float>* factors = in_global(a.calib);
    global_bytes in = in_global(a.in + a.in_off);
    int in_pf = a.in_pf, row_bytes = a.pitch * 16;
    global<int8_t>* out = in_global(a.out);
    global<int32_t>* raw = in_global(a.raw);
    int out_off = a.out_off, out_pb = a.out_pb, out_pf = a.out_pf, out_py = a.out_py, kind = a.kind, OFM = a.OFM, OH = a.OH, units = a.units;
    float hi = a.hi, lo = a.lo;
    asm volatile("" : "+s"(first), "+s"(factors), "+s"(in), "+s"(in_pf), "+s"(row_bytes), "+s"(out), "+s"(raw), "+s"(out_off), "+s"(out_pb), "+s"(out_pf), "+s"(out_py),
                 "+s"(kind), "+s"(OFM), "+s"(OH), "+s"(units), "+s"(hi), "+s"(lo));

    const uint32_t wg = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (wg >= (uint32_t)a.total) return;
    const uint32_t ptile = a.div_ftiles.div(wg), ftile = wg - ptile * (uint32_t)a.ftiles;
    const PlaneTile<NP> tile(a, ptile * (4 / SPANS) + (uint32_t)pair);

    extern __shared__ __align__(16) unsigned char smem[];
    v4i* lds = reinterpret_cast<v4i*>(smem);
    const int span = (int)ftile * SPANS + member;  // (spans past the last one: its weights, nothing is stored)
    global_bytes weights = (global_bytes)(a.wpk + (size_t)min(span, a.spans - 1) * a.jobs * 9 * 64);
    asm volatile("" : "+s"(weights));
    const uint32_t lane_bytes = (uint32_t)lane * 16u;
    uint32_t src[LOADS];
    int dst[LOADS];
    v4i w[2][9];
    auto request = [&](int j, int buffer, auto pc, auto rc) {
        constexpr int P = decltype(pc)::value, R = decltype(rc)::value;
        if constexpr (R < LOADS)
            __builtin_amdgcn_global_load_lds((halo_gptr)(in + (int64_t)(2 * j) * in_pf + src[R]), (halo_lptr)(lds + buffer + dst[R]), 16, 0, 0);
        else if constexpr (R < REQUESTS)
            w[P][R - LOADS] = *(const global<v4i>*)(weights + (uint32_t)(j * 9 + R - LOADS) * 1024u + lane_bytes);
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    static_for<LOADS, REQUESTS>([&](auto rc) {
        request(0, 0, B0{}, rc);
        step_fence();
    });
    const int buffer_units = 2 * a.positions, pair_units = pair * 3 * buffer_units;
    // the wave's loads of a patch; those that are left over repeat the last one
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int c = min(i * SPANS + member, 2 * NL - 1), s = c >= NL ? 1 : 0, q = min((c - s * NL) * 64, a.positions - 64);
        src[i] = tile.source(a, (uint32_t)(q + lane)) + (uint32_t)(s * in_pf), dst[i] = pair_units + s * a.positions + q;
    }
    static_for<0, LOADS>([&](auto rc) {
        request(0, 0, B0{}, rc);
        step_fence();
    });

    const uint32_t lane_group = (uint32_t)l32 >> a.shift, column = (uint32_t)l32 & ((1u << a.shift) - 1u);
    const uint32_t here = lds_offset(lds) + ((uint32_t)(pair_units + half * a.positions) + __umul24(lane_group, (uint32_t)a.pitch * (NP + 2)) + column) * 16u;
    v16i acc[NP] = {};
    const v4i xm = {(int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask, (int)a.xor_mask};
    const int slice = span * 2 + half, f0 = slice * 16;
    constexpr int N = POOL ? 8 : 16;  // features a lane finishes: with POOL the lanes of two neighbouring columns take half each
    const int fl = min(f0, (a.spans - 1) * 32 + 16) + (POOL ? (lane & 1) * 8 : 0);
    float cal[16] = {}, wq[16] = {};
    v4i init[4] = {};

    v4i ring[RG];
    uint32_t row[2];
    auto patch_arrived = [] { asm volatile("s_waitcnt vmcnt(9)\n\ts_barrier" ::: "memory"); };  // younger: the weights
    auto read = [&](int buffer, auto ic) {
        constexpr int R = decltype(ic)::value, Y = Read::row(R), C = Read::column(R);
        uint32_t& at = row[Read::place(R)];
        if constexpr (C == 0) at = here + (uint32_t)(Y * row_bytes + buffer * 16);
        lds_read<C * 16>(ring[R % RG], at);
    };
    int buffer = 0;
    auto job = [&](int j, auto pc, auto last) {
        constexpr int P = decltype(pc)::value;
        constexpr bool LAST = decltype(last)::value;
        using Next = std::integral_constant<int, 1 - P>;
        const int next = buffer == 2 * buffer_units ? 0 : buffer + buffer_units;
        static_for<0, Read::count>([&](auto ic) {
            constexpr int R = decltype(ic)::value, Y = Read::row(R), C = Read::column(R);
            constexpr int AHEAD = R + RG - 2;  // the latest read
            lds_wait<(LAST && AHEAD >= Read::count ? Read::count - 1 : AHEAD) - R>(ring[R % RG]);
            v4i x = ring[R % RG];
            if constexpr (FLIP) x ^= xm;
            static_for<0, 3>([&](auto fc) {
                constexpr int F = decltype(fc)::value, I = Y - F;
                if constexpr (I >= 0 && I < NP) acc[I] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[P][F * 3 + C], x, acc[I], 0, 0, 0);
            });
            step_fence();
            if constexpr (!LAST) static_for<0, AT_ONCE>([&](auto rc) { request(j + 1, next, Next{}, std::integral_constant<int, R * AT_ONCE + decltype(rc)::value>{}); });
            if constexpr (AHEAD + 1 < Read::count) {
                read(buffer, std::integral_constant<int, AHEAD + 1>{});
            } else if constexpr (!LAST) {
                if constexpr (AHEAD + 1 == Read::count) patch_arrived();
                read(next, std::integral_constant<int, AHEAD + 1 - Read::count>{});
            }
            if constexpr (LAST && R == Read::count / 2) {
#pragma unroll
                for (int d = 0; d < N / 4; ++d) {
                    init[d] = *(const global<v4i>*)(first + fl + d * 4);
                    const v4f c = *(const global<v4f>*)(factors + fl + d * 4);
                    cal[d * 4] = c.x, cal[d * 4 + 1] = c.y, cal[d * 4 + 2] = c.z, cal[d * 4 + 3] = c.w;
                }
            }
            step_fence();
        });
        buffer = next;
    };
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    static_for<0, RG - 1>([&](auto ic) { read(0, ic); });
    for (int j = 0; j + 2 < a.jobs; j += 2) {
        job(j, B0{}, std::false_type{});
        job(j + 1, B1{}, std::false_type{});
    }
    job(a.jobs - 2, B0{}, std::false_type{});
    job(a.jobs - 1, B1{}, std::true_type{});

    struct {
        FastEpi fe;
    } e;
    e.fe.hi = hi, e.fe.lo = e.fe.lo2 = lo, e.fe.split_valid = 0;
    v4i part[NP][4];
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d) part[i][d] = v4i{acc[i][d * 4], acc[i][d * 4 + 1], acc[i][d * 4 + 2], acc[i][d * 4 + 3]};
    asm volatile("s_nop 7\n\ts_nop 7");
    step_fence();
    mfma_settle(part);
    const int yl = tile.row_of(lane_group), x = tile.x0 + (int)column, b = tile.image_of(lane_group);
    const bool mine = tile.unit0 + (int)lane_group < units && (int)column < a.cols && x < a.OW && f0 < OFM;
    const v4i none = {0, 0, 0, 0};
    uint32_t at = (uint32_t)(out_off + b * out_pb + slice * out_pf);
    if constexpr (POOL) {
        static_assert(!POOL || NP % 2 == 0, "rows of windows");
        at += (uint32_t)((x >> 1) * 16 + (lane & 1) * 8) + __umul24(yl >> 1, out_py);
#pragma unroll
        for (int k = 0; k < NP / 2; ++k) {
            v4i best[4][1] = {{none}, {none}, {none}, {none}};
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int v = max_dpp<0xb1>(max(part[2 * k][d][c], part[2 * k + 1][d][c]));
                    best[d & 1][0][c] = d < 2 || (lane & 1) ? v : best[d & 1][0][c];
                }
            best[0][0] += init[0], best[1][0] += init[1];
            const v4i q = epilogue_fast16<1, EPI_KIND_RELU, 8>(e, best, 0, wq, cal, cal, none, OFM - f0 - (lane & 1) * 8);
            if (mine && yl + 2 * k < OH) *(global<v2i>*)(out + at) = v2i{q[0], q[1]};
            at += (uint32_t)out_py;
        }
    } else {
        at += (uint32_t)(x * 16) + __umul24(yl, out_py);
        auto each = [&](auto finish) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                v4i sum[4][1];
#pragma unroll
                for (int d = 0; d < 4; ++d) sum[d][0] = part[i][d] + init[d];
                finish(i, sum);
            }
        };
        if (raw) {
            keep_branch();
            each([&](int i, const v4i (&sum)[4][1]) {
                if (mine && yl + i < OH)
#pragma unroll
                    for (int c = 0; c < 16; ++c)
                        if (f0 + c < OFM) raw[(((size_t)b * OFM + f0 + c) * OH + yl + i) * a.OW + x] = sum[c >> 2][0][c & 3];
            });
        } else if (kind == EPI_KIND_RELU) {
            keep_branch();
            each([&](int i, const v4i (&sum)[4][1]) {
                const v4i q = epilogue_fast16<1, EPI_KIND_RELU>(e, sum, 0, wq, cal, cal, none, OFM - f0);
                if (mine && yl + i < OH) *(global<v4i>*)(out + at) = q;
                at += (uint32_t)out_py;
            });
        } else {
            keep_branch();
            each([&](int i, const v4i (&sum)[4][1]) {
                const v4i q = epilogue_fast16<1, EPI_KIND_LINEAR>(e, sum, 0, wq, cal, cal, none, OFM - f0);
                if (mine && yl + i < OH) *(global<v4i>*)(out + at) = q;
                at += (uint32_t)out_py;
            });
        }
    }
}

}  // namespace chip
