// Mixed-precision gridder and degridder for gfx950, a phasor per (pixel, visibility) pair: FP64 phase-argument reduction,
// FP32 phasors, and the phasor x data contraction on v_mfma_f32_16x16x32_{bf16,f16} with FP32 accumulation.  The
// 3-product forms run the separable kernels (separable.hip) for subgrids up to 64^2 and fields up to 0.13 to 0.16 rad, and
// these for the subgrids whose w spreads too far; larger subgrids, wider fields and the single-product forms run these.
//
// Phase reduction.  With l = (x' + 1/2) delta, x' = x - S/2 (an integer), delta = image_size / S, and
//     du = k_c u_t / 2pi - u_off,  dv = ...,  dw = k_c w_t / 2pi - w_off      (wavelengths, formed in FP64,
// u_off = (x0 + S/2 - G/2) / image_size the subgrid's phase centre), the phase in revolutions is
//     du l + dv m + dw n = qu x' + qv y' + dw n + (qu + qv) / 2,     qu = du delta, qv = dv delta.
// Because x', y' are integers, qu and qv can be reduced mod 1 in FP64 without changing the phasor, and the
// constant (qu + qv)/2 mod 1 becomes one rotation per visibility (folded into the gridder's B operand, or
// applied to the degridder's output).  The per-pair phase is then bounded by ~S/2 + |dw n| revolutions for any
// input, so three FP32 operations evaluate it to ~1e-6 revolutions and v_sin_f32/v_cos_f32 (domain +-256
// revolutions) take it directly.  This replaces the reference's FP32 phase_offset - k (u l + v m + w n)
// (gridding/src/gridding_benchmark.cpp:112-121), whose two large terms cancel.
//
// Contraction as a real GEMM.  pixel[p][corr] = sum_v phasor[p][v] * vis[v][corr] (gridder) is
//     D[p][n] = sum_k A[p][k] B[k][n],   A[p][2v] = cos, A[p][2v+1] = sin,
//     B[2v][re] = a, B[2v+1][re] = -b, B[2v][im] = b, B[2v+1][im] = a   (vis = a + ib, 4 correlations x re/im)
// which fills 8 of the 16 MFMA columns; the other 8 carry the low half of B, so one MFMA with A_hi gives
// A_hi*B_hi + A_hi*B_lo and one with A_lo gives A_lo*B_hi (+ A_lo*B_lo): the three-product split in two
// instructions.  Columns n and n+8 are summed at the end.  The degridder is the same with pixels and
// visibilities exchanging roles (vis[v][corr] = sum_p phasor[v][p] * pixel[p][corr]).
//
// Operand layout of v_mfma_f32_16x16x32 (one wave): lane l holds A[l%16][8*(l/16) .. +7], B[8*(l/16) .. +7][l%16]
// and D[4*(l/16) .. +3][l%16].  So a lane evaluates phasors of one row (pixel, or visibility) against four
// k-pairs, packs (cos, sin) pairs straight into A registers, and reads its 16-byte B fragment from LDS.
//
// Phases.  By default the VALU forms phi = qu x' + qv y' + dw n with two FMAs per pair: the gridder's pixel
// mapping keeps a lane's column x' fixed across its tiles (strips of 16 / 8 / 4 / 2 columns), and the
// degridder's pixel slots run in rows padded to a multiple of 4 so the four pixels of a lane group share y', so
// one of the three terms is formed once per visibility.  The PM shapes take the phases from the matrix core
// instead (phi is a rank-3 product: one v_mfma_f32_16x16x4_f32 per 16 x 16 tile, whose D layout, lane l holding
// D[4*(l/16)+j][l%16], is exactly the A layout above); that frees two VALU ops per pair but measured slower, so
// the autotuner rarely picks it.
//
// hi/lo split (FP16): hi = v_cvt_pk_f16_f32 of (cos, sin); lo = the exact residual from v_fma_mix_f32 (reading
// the half straight from the packed register), packed again: 4 VALU ops per pair.  FP16 B operands are scaled
// by a power of two so that their largest value is ~2^14 (per LDS batch, or per subgrid for prepared degridder
// pixels), which keeps any data range in range; the accumulators are rescaled exactly when the scale grows.
//
// Workgroup numbering spreads the workgroups of one subgrid over the XCDs (block b = sub_block * n + s): subgrid
// costs are uneven, and grouping a subgrid's workgroups on one XCD (for L2 reuse) measured 1.2-2x slower because
// the round-robin dispatch then waits on the most loaded XCD.
#include "mixed_device.hpp"

namespace idgx
{
namespace
{
// ---------------------------------------------------------------------------------------------------------------
// Kernels: one-shot grids (workgroup b = item (b % n, b / n), so a subgrid's workgroups spread over the XCDs)
// and persistent workgroups fed from the device work queue.
// ---------------------------------------------------------------------------------------------------------------
// Resident workgroups per CU the kernels ask for: 4 (gridder) and 5 (degridder), which leaves 128 / 96 VGPRs (a
// few bytes spill outside the inner loops; measured 2 % faster than 3 / 4), fewer where the shape's LDS or its
// accumulators do not allow it.
constexpr int kLdsBytes = 160 * 1024;
template <int PT, int VB> constexpr int gridder_min_blocks()
{
    constexpr int fit = kLdsBytes / static_cast<int>(sizeof(GridderShared<PT, VB>));
    return fit < 4 ? fit : 4;
}
template <int VT, int PB> constexpr int degridder_min_blocks()
{
    constexpr int fit = kLdsBytes / static_cast<int>(sizeof(DegridderShared<VT, PB>));
    constexpr int regs = VT >= 8 ? 3 : VT >= 6 ? 4 : 5;
    return fit < regs ? fit : regs;
}

template <int DT, bool SPLIT, int PT, int VB, bool PM>
__global__ __launch_bounds__(kThreads, (gridder_min_blocks<PT, VB>())) void gridder_mfma(KernelArgs a)
{
    __shared__ GridderShared<PT, VB> sm;
    const int pblk = blockIdx.x / a.p.nr_subgrids;
    gridder_item<DT, SPLIT, PT, VB, PM>(a, blockIdx.x - pblk * a.p.nr_subgrids, pblk, sm);
}

// Behind a separable launch: the items of the subgrids that it left, over their workgroups.  (A kernel of its own: the
// check costs the one above, a workgroup per item of which many have nothing to do, up to 1.7 times its time.)
template <int DT, int PT, int VB>
__global__ __launch_bounds__(kThreads, (gridder_min_blocks<PT, VB>())) void gridder_left(KernelArgs a, int items)
{
    __shared__ GridderShared<PT, VB> sm;
    __shared__ float slots[kWaves][5];
    const int part = blockIdx.x / a.p.nr_subgrids, s = blockIdx.x - part * a.p.nr_subgrids;
    if (separable_done(a, s, 0, slots))
        return; // uniform
    for (int i = part; i < items; i += gridDim.x / a.p.nr_subgrids)
    {
        gridder_item<DT, true, PT, VB, false>(a, s, i, sm);
        __syncthreads();
    }
}

template <int DT, bool SPLIT, int VT, int PB, bool PM>
__global__ __launch_bounds__(kThreads, (degridder_min_blocks<VT, PB>())) void degridder_mfma(KernelArgs a)
{
    __shared__ DegridderShared<VT, PB> sm;
    const int vblk = blockIdx.x / a.p.nr_subgrids;
    degridder_item<DT, SPLIT, VT, PB, PM, false>(a, blockIdx.x - vblk * a.p.nr_subgrids, vblk, sm);
}

template <int DT, int VT, int PB>
__global__ __launch_bounds__(kThreads, (degridder_min_blocks<VT, PB>())) void degridder_left(KernelArgs a, int items)
{
    __shared__ DegridderShared<VT, PB> sm;
    __shared__ float slots[kWaves][5];
    const int part = blockIdx.x / a.p.nr_subgrids, s = blockIdx.x - part * a.p.nr_subgrids;
    if (separable_done(a, s, static_cast<long long>(part) * kWaves * VT * 16, slots))
        return; // uniform
    for (int i = part; i < items; i += gridDim.x / a.p.nr_subgrids)
        degridder_item<DT, true, VT, PB, false, false>(a, s, i, sm);
}

template <int DT, bool SPLIT, int PT, int VB, bool PM>
__global__ __launch_bounds__(kThreads, (gridder_min_blocks<PT, VB>())) void gridder_mfma_queue(QueueArgs q)
{
    __shared__ GridderShared<PT, VB> sm;
    if (!queue_has_work(q))
        return;
    int cls, s, blk;
    while (next_queue_item(q, cls, s, blk))
    {
        if (subgrid_done(q.cls[cls], s))
            continue;
        gridder_item<DT, SPLIT, PT, VB, PM>(q.cls[cls], s, blk, sm);
        __syncthreads();
    }
}

// One launch over items of several subgrid classes, each item with its class's tiles per wave (q.tiles[class]),
// LDS batch kDefaultVB, phases on the VALU.  The LDS holds the largest tile count's staging; every variant's
// registers fit the same occupancy (4 waves per SIMD), so a class loses nothing to sharing the launch.
template <int DT, bool SPLIT>
__global__ __launch_bounds__(kThreads, (gridder_min_blocks<8, kDefaultVB>())) void gridder_mfma_queue_tiles(QueueArgs q)
{
    __shared__ GridderShared<8, kDefaultVB> sm;
    if (!queue_has_work(q))
        return;
    int cls, s, blk;
    while (next_queue_item(q, cls, s, blk))
    {
        if (subgrid_done(q.cls[cls], s))
            continue;
        switch (q.tiles[cls]) // workgroup-uniform
        {
        case 2:
            gridder_item<DT, SPLIT, 2, kDefaultVB, false>(q.cls[cls], s, blk, sm);
            break;
        case 3:
            gridder_item<DT, SPLIT, 3, kDefaultVB, false>(q.cls[cls], s, blk, sm);
            break;
        case 4:
            gridder_item<DT, SPLIT, 4, kDefaultVB, false>(q.cls[cls], s, blk, sm);
            break;
        case 6:
            gridder_item<DT, SPLIT, 6, kDefaultVB, false>(q.cls[cls], s, blk, sm);
            break;
        default:
            gridder_item<DT, SPLIT, 8, kDefaultVB, false>(q.cls[cls], s, blk, sm);
            break;
        }
        __syncthreads();
    }
}

template <int DT, bool SPLIT, int VT, int PB, bool PM>
__global__ __launch_bounds__(kThreads, (degridder_min_blocks<VT, PB>())) void degridder_mfma_queue(QueueArgs q)
{
    __shared__ DegridderShared<VT, PB> sm;
    if (!queue_has_work(q))
        return;
    int cls, s, blk;
    while (next_queue_item(q, cls, s, blk))
        if (!subgrid_done(q.cls[cls], s))
            degridder_item<DT, SPLIT, VT, PB, PM, true>(q.cls[cls], s, blk, sm);
}

__global__ void reset_counters_kernel(int *counters, int n)
{
    if (static_cast<int>(threadIdx.x) < n)
        counters[threadIdx.x] = 0;
}

// One workgroup per subgrid: the taper x A-term-applied pixels of every slot, split into the packed words the
// degridder stages (FP16: scaled by 2^-scale so that the largest value is about 2^14).  The workgroup of subgrid 0
// also writes the slot table (x', y', n), so that the degridder's staging reads a slot's coordinates instead of
// dividing by the row stride.  Subgrids outside the arrays are skipped (the degridder skips them too).  Each XCD
// takes a contiguous run of subgrids (plan order: baseline by baseline), so the stations' A-terms it reads stay in
// its own L2 instead of every XCD streaming the whole table.
template <int DT, bool SPLIT, int CACHED>
__global__ __launch_bounds__(kThreads) void degrid_prepare_kernel(KernelArgs a)
{
    __shared__ unsigned maxbits;
    if (a.leftover_any && !*a.leftover_any)
        return; // uniform: the separable kernel has done every subgrid
    const int s = xcd_contiguous(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const int S = a.p.S, P = S * S, Sp = degrid_row_stride(S), nslots = S * Sp;
    float4 *slot_coord = const_cast<float4 *>(a.slot_coord);
    if (s == 0)
    {
        for (int q = tid; q < nslots; q += kThreads)
        {
            const int sy = q / Sp, sx = q - sy * Sp;
            const float n = sx < S ? pixel_n_f(pixel_lm_f(sx, S, a.p.image_size), pixel_lm_f(sy, S, a.p.image_size))
                                   : 0.F;
            slot_coord[q] = make_float4(pixel_offset(sx, S), pixel_offset(sy, S), n, 0.F);
        }
    }
    if (subgrid_done(a, s))
        return; // uniform
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    if (!subgrid_in_bounds(a.p, m, row0, c0, nc) || nc == 0)
        return; // uniform
    const float2 *sub = reinterpret_cast<const float2 *>(a.subgrids) + static_cast<size_t>(s) * kCorr * P;
    uint4 *dst = const_cast<uint4 *>(a.prepared) + static_cast<size_t>(s) * nslots * 2;
    // Slots per thread held in registers between the FP16 scale and the split, so that the subgrid is read once:
    // 4 covers S <= 32, 9 covers S <= 48, 16 covers S <= 64; larger subgrids read it twice.
    constexpr int kCached = CACHED;
    if (nslots <= kCached * kThreads)
    {
        // One pass over the subgrid: pixels stay in registers while the workgroup finds the FP16 scale.
        cfloat px[kCached][4];
        float vmax = 0.F;
#pragma unroll
        for (int k = 0; k < kCached; ++k)
        {
            const int q = tid + k * kThreads;
            const int sy = q / Sp, sx = q - sy * Sp;
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
                px[k][pol] = {0.F, 0.F};
            if (q < nslots && sx < S)
            {
                degrid_pixel(a, m, sub, sy * S + sx, px[k]);
#pragma unroll
                for (int pol = 0; pol < 4; ++pol)
                    vmax = fmaxf(vmax, fmaxf(fabsf(px[k][pol].re), fabsf(px[k][pol].im)));
            }
        }
        float inv1 = 1.F;
        if constexpr (DT == kFP16)
        {
            const int e = scale_exponent(block_max(vmax, maxbits));
            if (tid == 0)
                const_cast<int *>(a.prepared_scale)[s] = e;
            inv1 = ldexpf(1.F, -e);
        }
#pragma unroll
        for (int k = 0; k < kCached; ++k)
        {
            const int q = tid + k * kThreads;
            if (q >= nslots)
                break;
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
                px[k][pol] = {px[k][pol].re * inv1, px[k][pol].im * inv1};
            split_item<DT, SPLIT>(px[k], hi, lo);
            dst[2 * q] = make_uint4(hi[0], lo[0], hi[1], lo[1]);
            dst[2 * q + 1] = make_uint4(hi[2], lo[2], hi[3], lo[3]);
        }
        return;
    }
    float inv = 1.F;
    if constexpr (DT == kFP16)
    {
        float vmax = 0.F;
        for (int q = tid; q < nslots; q += kThreads)
        {
            const int sy = q / Sp, sx = q - sy * Sp;
            if (sx < S)
            {
                cfloat px[4];
                degrid_pixel(a, m, sub, sy * S + sx, px);
#pragma unroll
                for (int pol = 0; pol < 4; ++pol)
                    vmax = fmaxf(vmax, fmaxf(fabsf(px[pol].re), fabsf(px[pol].im)));
            }
        }
        const int e = scale_exponent(block_max(vmax, maxbits));
        if (tid == 0)
            const_cast<int *>(a.prepared_scale)[s] = e;
        inv = ldexpf(1.F, -e);
    }
    for (int q = tid; q < nslots; q += kThreads)
    {
        const int sy = q / Sp, sx = q - sy * Sp;
        uint32_t hi[4] = {0u, 0u, 0u, 0u}, lo[4] = {0u, 0u, 0u, 0u};
        if (sx < S)
        {
            cfloat px[4];
            degrid_pixel(a, m, sub, sy * S + sx, px);
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
                px[pol] = {px[pol].re * inv, px[pol].im * inv};
            split_item<DT, SPLIT>(px, hi, lo);
        }
        dst[2 * q] = make_uint4(hi[0], lo[0], hi[1], lo[1]);
        dst[2 * q + 1] = make_uint4(hi[2], lo[2], hi[3], lo[3]);
    }
}

// ---- launchers ------------------------------------------------------------------------------------------------


// Gridder tiles per wave for subgrid size S.  A wave with more tiles spreads each visibility's staged work over
// more pixels (issue efficiency relative to 8 tiles, measured on sizes the tiles cover exactly: 6 -> 0.965,
// 4 -> 0.89, 3 -> 0.845, 2 -> 0.78), but the last row block and the last item of a subgrid can leave tiles and
// waves idle (coverage = S^2 / pixels of the items).  The choice maximises coverage x efficiency: S = 32 and 64
// take 8, S = 48 takes 6, S = 24 takes 3, S = 16 takes 4.
constexpr int kGridTileChoices[] = {8, 6, 4, 3, 2};
constexpr double kGridTileEfficiency[] = {1.0, 0.965, 0.89, 0.845, 0.78};

double grid_coverage(int S, int tiles)
{
    const GridUnits gu = grid_units(S, tiles);
    const long long items = (gu.units + kWaves - 1) / kWaves;
    return static_cast<double>(S) * S / static_cast<double>(items * kWaves * tiles * 16);
}

int grid_tiles_for(int S)
{
    int best = kGridTileChoices[0];
    double best_score = -1.0;
    for (int i = 0; i < static_cast<int>(sizeof(kGridTileChoices) / sizeof(int)); ++i)
    {
        const double score = grid_coverage(S, kGridTileChoices[i]) * kGridTileEfficiency[i];
        if (score > best_score + 1e-9) // ties keep the larger tile count
        {
            best_score = score;
            best = kGridTileChoices[i];
        }
    }
    return best;
}

// Whether a one-shot launch runs behind a separable one.
bool behind_separable(const KernelArgs &a)
{
    return a.limits.eps_most != 0.F;
}

// Workgroups per subgrid of a one-shot launch: one per item, but behind a separable launch, where most of them only find
// that the subgrid is done, no more than fill the chip four times (8166 subgrids of 40^2, none left, both directions:
// 80 us with one per item).
long long oneshot_parts(const KernelArgs &a, long long items)
{
    constexpr long long kWorkgroups = 4096;
    return behind_separable(a) ? std::min(items, std::max(1LL, kWorkgroups / a.p.nr_subgrids)) : items;
}

template <int DT, bool SPLIT, int PT, bool PM> hipError_t grid_mfma_tiles(const KernelArgs &a, hipStream_t st)
{
    const GridUnits gu = grid_units(a.p.S, PT);
    const int items = (gu.units + kWaves - 1) / kWaves;
    const long long blocks = a.p.nr_subgrids * oneshot_parts(a, items);
    if (blocks > 0x7fffffffLL)
        return hipErrorInvalidConfiguration;
    const unsigned n = static_cast<unsigned>(blocks);
    if constexpr (SPLIT && !PM)
    {
        if (behind_separable(a))
        {
            gridder_left<DT, PT, kDefaultVB><<<n, kThreads, 0, st>>>(a, items);
            return hipGetLastError();
        }
    }
    gridder_mfma<DT, SPLIT, PT, kDefaultVB, PM><<<n, kThreads, 0, st>>>(a);
    return hipGetLastError();
}

template <int DT, bool SPLIT> hipError_t grid_mfma(const KernelArgs &a, bool pm, hipStream_t st)
{
    if (pm)
        return grid_mfma_tiles<DT, SPLIT, kDefaultPT, true>(a, st);
    switch (grid_tiles_for(a.p.S))
    {
    case 8:
        return grid_mfma_tiles<DT, SPLIT, 8, false>(a, st);
    case 6:
        return grid_mfma_tiles<DT, SPLIT, 6, false>(a, st);
    case 4:
        return grid_mfma_tiles<DT, SPLIT, 4, false>(a, st);
    case 3:
        return grid_mfma_tiles<DT, SPLIT, 3, false>(a, st);
    default:
        return grid_mfma_tiles<DT, SPLIT, 2, false>(a, st);
    }
}

template <int DT, bool SPLIT> hipError_t degrid_mfma(const KernelArgs &a, bool pm, hipStream_t st)
{
    constexpr int chunk = kWaves * kDefaultVT * 16;
    const long long vmax = static_cast<long long>(a.p.max_nr_timesteps) * a.p.nr_channels;
    const long long per = vmax > 0 ? (vmax + chunk - 1) / chunk : 1;
    const long long blocks = a.p.nr_subgrids * oneshot_parts(a, per);
    if (blocks > 0x7fffffffLL)
        return hipErrorInvalidConfiguration;
    const unsigned n = static_cast<unsigned>(blocks);
    if constexpr (SPLIT)
    {
        if (behind_separable(a))
        {
            degridder_left<DT, kDefaultVT, kDefaultPB><<<n, kThreads, 0, st>>>(a, static_cast<int>(per));
            return hipGetLastError();
        }
    }
    if (pm)
        degridder_mfma<DT, SPLIT, kDefaultVT, kDefaultPB, true><<<n, kThreads, 0, st>>>(a);
    else
        degridder_mfma<DT, SPLIT, kDefaultVT, kDefaultPB, false><<<n, kThreads, 0, st>>>(a);
    return hipGetLastError();
}

// Tile shapes the persistent kernels are built for (the autotuner picks among them): {tiles per wave, LDS batch,
// phases on the matrix core}.
constexpr MixedShape kShapes[] = {{4, 256, 0}, {2, 256, 0}, {8, 256, 0}, {4, 128, 0}, {4, 512, 0},
                                  {4, 256, 1}, {8, 256, 1}, {2, 256, 1}, {3, 256, 0}, {6, 256, 0}};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);

template <int DT, bool SPLIT, int I> void *queue_fn(bool gridder)
{
    constexpr MixedShape sh = kShapes[I];
    if (gridder)
        return reinterpret_cast<void *>(&gridder_mfma_queue<DT, SPLIT, sh.tiles, sh.batch, sh.phase_mfma != 0>);
    return reinterpret_cast<void *>(&degridder_mfma_queue<DT, SPLIT, sh.tiles, sh.batch, sh.phase_mfma != 0>);
}

template <int DT, bool SPLIT> void *queue_kernel(bool gridder, int shape)
{
    switch (shape)
    {
    case 0:
        return queue_fn<DT, SPLIT, 0>(gridder);
    case 1:
        return queue_fn<DT, SPLIT, 1>(gridder);
    case 2:
        return queue_fn<DT, SPLIT, 2>(gridder);
    case 3:
        return queue_fn<DT, SPLIT, 3>(gridder);
    case 4:
        return queue_fn<DT, SPLIT, 4>(gridder);
    case 5:
        return queue_fn<DT, SPLIT, 5>(gridder);
    case 6:
        return queue_fn<DT, SPLIT, 6>(gridder);
    case 7:
        return queue_fn<DT, SPLIT, 7>(gridder);
    case 8:
        return queue_fn<DT, SPLIT, 8>(gridder);
    case 9:
        return queue_fn<DT, SPLIT, 9>(gridder);
    default:
        return nullptr;
    }
}

void *queue_kernel_for(int precision, bool gridder, int shape)
{
    if (shape == kShapeTilesPerClass)
    {
        if (!gridder)
            return nullptr;
        switch (precision)
        {
        case IDGX_MIXED_BF16X3:
            return reinterpret_cast<void *>(&gridder_mfma_queue_tiles<kBF16, true>);
        case IDGX_MIXED_FP16X3:
            return reinterpret_cast<void *>(&gridder_mfma_queue_tiles<kFP16, true>);
        case IDGX_MIXED_BF16:
            return reinterpret_cast<void *>(&gridder_mfma_queue_tiles<kBF16, false>);
        case IDGX_MIXED_FP16:
            return reinterpret_cast<void *>(&gridder_mfma_queue_tiles<kFP16, false>);
        default:
            return nullptr;
        }
    }
    switch (precision)
    {
    case IDGX_MIXED_BF16X3:
        return queue_kernel<kBF16, true>(gridder, shape);
    case IDGX_MIXED_FP16X3:
        return queue_kernel<kFP16, true>(gridder, shape);
    case IDGX_MIXED_BF16:
        return queue_kernel<kBF16, false>(gridder, shape);
    case IDGX_MIXED_FP16:
        return queue_kernel<kFP16, false>(gridder, shape);
    default:
        return nullptr;
    }
}

hipError_t launch_queue(const QueueArgs &q, int precision, bool gridder, int shape, int workgroups, hipStream_t st)
{
    void *fn = queue_kernel_for(precision, gridder, shape);
    if (!fn || workgroups <= 0)
        return hipErrorInvalidValue;
    // The persistent degridder reads prepared pixels only (launch_degrid_prepare fills them first).
    for (int k = 0; k < kMaxClasses && !gridder; ++k)
        if (q.cls[k].p.nr_subgrids > 0 && (!q.cls[k].prepared || !q.cls[k].prepared_scale || !q.cls[k].slot_coord))
            return hipErrorInvalidValue;
    QueueArgs arg = q;
    void *args[] = {&arg};
    return hipLaunchKernel(fn, dim3(workgroups), dim3(kThreads), args, 0, st);
}
} // namespace

// One-shot plans of the separable kernels: where the plan lets expect subgrids that they leave, a launch of the per-pair
// kernels behind them, whose workgroups end at once for the others.  All subgrids of 256 visibilities left, per-pair
// kernels alone / with their items inside the separable launch / behind it: gridder 40 of 64^2 33 / 151 / 39 us, 6000 of
// 32^2 577 / 658 / 627 us; degridder 6000 of 64^2 2164 / 3786 / 2443 us.
hipError_t launch_grid_mixed(const KernelArgs &args, int precision, bool pm, hipStream_t st)
{
    KernelArgs a = args;
    SeparableArgs sp{};
    if (!pm && separable_tables(a.p, precision, sp.tables))
    {
        sp.limits = separable_limits(sp.tables, true);
        sp.leave = separable_may_leave(a.p, sp.limits);
        const hipError_t e = launch_grid_separable(
            a, sp, precision, {static_cast<long long>(a.p.max_nr_timesteps) * a.p.nr_channels, 0}, st);
        if (e != hipSuccess || !sp.leave)
            return e;
        a.limits = sp.limits;
    }
    switch (precision)
    {
    case IDGX_MIXED_BF16X3:
        return grid_mfma<kBF16, true>(a, pm, st);
    case IDGX_MIXED_FP16X3:
        return grid_mfma<kFP16, true>(a, pm, st);
    case IDGX_MIXED_BF16:
        return grid_mfma<kBF16, false>(a, pm, st);
    case IDGX_MIXED_FP16:
        return grid_mfma<kFP16, false>(a, pm, st);
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t launch_degrid_mixed(const KernelArgs &args, int precision, bool pm, hipStream_t st)
{
    KernelArgs a = args;
    SeparableArgs sp{};
    if (!pm && separable_tables(a.p, precision, sp.tables))
    {
        const long long vmax = static_cast<long long>(a.p.max_nr_timesteps) * a.p.nr_channels;
        sp.limits = separable_limits(sp.tables, false);
        sp.leave = separable_may_leave(a.p, sp.limits);
        sp.per = separable_chunk(vmax, a.p.nr_subgrids);
        const hipError_t e = launch_degrid_separable(a, sp, precision, vmax, st);
        if (e != hipSuccess || !sp.leave)
            return e;
        a.limits = sp.limits;
    }
    switch (precision)
    {
    case IDGX_MIXED_BF16X3:
        return degrid_mfma<kBF16, true>(a, pm, st);
    case IDGX_MIXED_FP16X3:
        return degrid_mfma<kFP16, true>(a, pm, st);
    case IDGX_MIXED_BF16:
        return degrid_mfma<kBF16, false>(a, pm, st);
    case IDGX_MIXED_FP16:
        return degrid_mfma<kFP16, false>(a, pm, st);
    default:
        return hipErrorInvalidValue;
    }
}

int mixed_shape_count()
{
    return kNumShapes;
}

// The one-shot kernels' tile shapes for S = 32, as persistent-kernel shapes.
constexpr int kDefaultGridShape = 2, kDefaultDegridShape = 0;
static_assert(kShapes[kDefaultGridShape].tiles == kDefaultPT && kShapes[kDefaultGridShape].batch == kDefaultVB &&
                  kShapes[kDefaultGridShape].phase_mfma == 0,
              "default gridder shape");
static_assert(kShapes[kDefaultDegridShape].tiles == kDefaultVT && kShapes[kDefaultDegridShape].batch == kDefaultPB &&
                  kShapes[kDefaultDegridShape].phase_mfma == 0,
              "default degridder shape");

int mixed_default_shape(bool gridder, int S)
{
    if (!gridder)
        return kDefaultDegridShape;
    const int tiles = grid_tiles_for(S);
    for (int i = 0; i < kNumShapes; ++i)
        if (kShapes[i].tiles == tiles && kShapes[i].batch == kDefaultVB && !kShapes[i].phase_mfma)
            return i;
    return kDefaultGridShape;
}

MixedShape mixed_shape(int i)
{
    return kShapes[i];
}

int grid_items_per_subgrid(int shape, int S)
{
    return (grid_units(S, kShapes[shape].tiles).units + kWaves - 1) / kWaves;
}

long long grid_item_pixels(int shape, int S, int item)
{
    const GridUnits gu = grid_units(S, kShapes[shape].tiles);
    long long n = 0;
    for (int u = kWaves * item; u < min(kWaves * (item + 1), gu.units); ++u)
        n += static_cast<long long>(gu.wd) * min(gu.rows, S - (u / gu.ns) * gu.rows);
    return n;
}

int degrid_visibilities_per_item(int shape)
{
    return kWaves * kShapes[shape].tiles * 16;
}

hipError_t launch_grid_mixed_queue(const QueueArgs &q, int precision, int shape, int workgroups, hipStream_t st)
{
    return launch_queue(q, precision, true, shape, workgroups, st);
}

hipError_t launch_degrid_mixed_queue(const QueueArgs &q, int precision, int shape, int workgroups, hipStream_t st)
{
    return launch_queue(q, precision, false, shape, workgroups, st);
}

size_t degrid_prepared_bytes(int S, long long nr_subgrids)
{
    return static_cast<size_t>(nr_subgrids) * S * degrid_row_stride(S) * 2 * sizeof(uint4);
}

hipError_t launch_degrid_prepare(const KernelArgs &a, int precision, hipStream_t st)
{
    if (a.p.nr_subgrids <= 0)
        return hipSuccess;
    if (!a.prepared || !a.prepared_scale || !a.slot_coord)
        return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(a.p.nr_subgrids));
    // FP16 needs the subgrid's maximum before the split: hold up to 4, 9 or 16 slots per thread, so that subgrids
    // up to S = 32, 48 or 64 and their A-terms are read once (BF16 has no scale and streams the slots in one pass
    // either way).
    const int nslots = a.p.S * degrid_row_stride(a.p.S);
    const int cached = nslots <= 4 * kThreads ? 4 : nslots <= 9 * kThreads ? 9 : 16;
    switch (precision)
    {
    case IDGX_MIXED_BF16X3:
        degrid_prepare_kernel<kBF16, true, 4><<<grid, kThreads, 0, st>>>(a);
        break;
    case IDGX_MIXED_FP16X3:
        if (cached == 16)
            degrid_prepare_kernel<kFP16, true, 16><<<grid, kThreads, 0, st>>>(a);
        else if (cached == 9)
            degrid_prepare_kernel<kFP16, true, 9><<<grid, kThreads, 0, st>>>(a);
        else
            degrid_prepare_kernel<kFP16, true, 4><<<grid, kThreads, 0, st>>>(a);
        break;
    case IDGX_MIXED_BF16:
        degrid_prepare_kernel<kBF16, false, 4><<<grid, kThreads, 0, st>>>(a);
        break;
    case IDGX_MIXED_FP16:
        if (cached == 16)
            degrid_prepare_kernel<kFP16, false, 16><<<grid, kThreads, 0, st>>>(a);
        else if (cached == 9)
            degrid_prepare_kernel<kFP16, false, 9><<<grid, kThreads, 0, st>>>(a);
        else
            degrid_prepare_kernel<kFP16, false, 4><<<grid, kThreads, 0, st>>>(a);
        break;
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_reset_counters(int *counters, int n, hipStream_t st)
{
    if (n < 1 || n > 64)
        return hipErrorInvalidValue;
    reset_counters_kernel<<<1, 64, 0, st>>>(counters, n);
    return hipGetLastError();
}

int queue_workgroups(int precision, bool gridder, int shape)
{
    void *fn = queue_kernel_for(precision, gridder, shape);
    if (!fn)
        return 0;
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, kThreads, 0) != hipSuccess || per_cu <= 0)
        per_cu = 1;
    return cus * per_cu;
}
} // namespace idgx
