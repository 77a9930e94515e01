// Plain FP32 gridder and degridder for gfx950.
//
// Phases are rounded exactly as in the reference CPU path (gridding/src/gridding_benchmark.cpp:99-121,
// gridding/src/degridding_benchmark.cpp:157-166): the whole file is compiled with contraction off, so
// `a * b + c` rounds twice; the complex multiply-accumulates are written as explicit fused multiply-adds.
//
// Gridder: one workgroup of 256 threads owns 256 pixels of one subgrid (one per thread, its 4 correlations held in
//   VGPRs).  Visibilities and uvw of the subgrid stream through LDS in batches of 256 visibilities; every lane reads the
//   same LDS address per visibility (broadcast, conflict-free).  Taper and A-term are applied in the epilogue, which
//   overwrites the subgrid.
// Degridder: one workgroup owns 256 (timestep, channel-chunk) items of one subgrid, each thread one timestep x
//   up to 2 or 4 channels.  Tapered, A-term-corrected pixels plus (l, m, n, phase offset) are staged through LDS in
//   batches of 512 pixels; each thread sums its visibilities over all pixels in registers, so no cross-lane
//   reduction is needed.
// Tile forms, for plans whose waves of 64 pixels or visibilities leave SIMDs idle: a wave sums for 16 of them, on the
//   matrix cores, with the same bits.
#include <algorithm>
#include <type_traits>

#include "idgx_device.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)

namespace idgx
{
namespace
{
constexpr int kThreads = 256;
constexpr int kGridBatchVis = 256; // visibilities per LDS stage
constexpr int kGridChunk = 64;     // channels per chunk (bounds the per-stage uvw count at 256 timesteps)
constexpr int kDegridPixBatch = 512;
constexpr int kTilePixBatch = 256; // pixels per LDS stage of the tile form, one per thread

// Visibility x phasor accumulated into acc[0..7] = {XX.re, XX.im, XY.re, ..., YY.im}, the cosine's terms first.
__device__ __forceinline__ void cmac4(float *acc, float4 va, float4 vb, float cs, float sn)
{
    acc[0] = __builtin_fmaf(va.x, cs, acc[0]);
    acc[1] = __builtin_fmaf(va.y, cs, acc[1]);
    acc[2] = __builtin_fmaf(va.z, cs, acc[2]);
    acc[3] = __builtin_fmaf(va.w, cs, acc[3]);
    acc[4] = __builtin_fmaf(vb.x, cs, acc[4]);
    acc[5] = __builtin_fmaf(vb.y, cs, acc[5]);
    acc[6] = __builtin_fmaf(vb.z, cs, acc[6]);
    acc[7] = __builtin_fmaf(vb.w, cs, acc[7]);
    acc[0] = __builtin_fmaf(-va.y, sn, acc[0]);
    acc[1] = __builtin_fmaf(va.x, sn, acc[1]);
    acc[2] = __builtin_fmaf(-va.w, sn, acc[2]);
    acc[3] = __builtin_fmaf(va.z, sn, acc[3]);
    acc[4] = __builtin_fmaf(-vb.y, sn, acc[4]);
    acc[5] = __builtin_fmaf(vb.x, sn, acc[5]);
    acc[6] = __builtin_fmaf(-vb.w, sn, acc[6]);
    acc[7] = __builtin_fmaf(vb.z, sn, acc[7]);
}

// The same sums, each one's two terms next to each other: faster where several pixels of a thread take turns (3000
// subgrids of 48^2 with 1024 visibilities, three pixels per thread: cmac4_group 3656 us, this 3534; four, 32^2, 256
// visibilities, 12,000 subgrids: 1726 and 1676).
__device__ __forceinline__ void cmac4_pairs(float *acc, float4 va, float4 vb, float cs, float sn)
{
    const float x[4] = {va.x, va.z, vb.x, vb.z}, y[4] = {va.y, va.w, vb.y, vb.w};
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
        acc[2 * j] = __builtin_fmaf(x[j], cs, acc[2 * j]);
        acc[2 * j] = __builtin_fmaf(-y[j], sn, acc[2 * j]);
        acc[2 * j + 1] = __builtin_fmaf(y[j], cs, acc[2 * j + 1]);
        acc[2 * j + 1] = __builtin_fmaf(x[j], sn, acc[2 * j + 1]);
    }
}

// The same sums of one value on N pixels (visibilities) side by side, acc(i) the i-th one's: the degridder's two or four
// visibilities per thread (3000 subgrids of 48^2 with 1024 visibilities: N calls of cmac4 3960 us, this 3835).
template <int N, class Acc>
__device__ __forceinline__ void cmac4_group(Acc acc, float4 va, float4 vb, const float (&cs)[N], const float (&sn)[N])
{
    if constexpr (N == 1)
    {
        cmac4(acc(0), va, vb, cs[0], sn[0]);
        return;
    }
    const float x[4] = {va.x, va.z, vb.x, vb.z}, y[4] = {va.y, va.w, vb.y, vb.w};
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
#pragma unroll
        for (int i = 0; i < N; ++i)
            acc(i)[2 * j] = __builtin_fmaf(x[j], cs[i], acc(i)[2 * j]);
#pragma unroll
        for (int i = 0; i < N; ++i)
            acc(i)[2 * j + 1] = __builtin_fmaf(y[j], cs[i], acc(i)[2 * j + 1]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
    {
#pragma unroll
        for (int i = 0; i < N; ++i)
            acc(i)[2 * j + 1] = __builtin_fmaf(x[j], sn[i], acc(i)[2 * j + 1]);
#pragma unroll
        for (int i = 0; i < N; ++i)
            acc(i)[2 * j] = __builtin_fmaf(-y[j], sn[i], acc(i)[2 * j]);
    }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Sums of value x phasor on v_mfma_f32_16x16x4_f32: D[16 rows][8 columns in use] += A[16][4] B[4][8], rows = the 16
// pixels (visibilities) whose sums these are, columns = (re, im) x 4 correlations, k = (cos, sin) of two of the
// visibilities (pixels) that are summed.  Lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and, in element i of the sums,
// D[4 (l / 16) + i][l % 16].  The instruction adds its four products one after the other, each as a fused multiply-add
// with one rounding, so a sum has the bits of cmac4's in the order of the values, whatever their grouping.
//
// Factors of one value in LDS, 16 floats: its columns for the cosine, then for the sine.
__device__ __forceinline__ void store_factors(float4 *f, float4 va, float4 vb)
{
    f[0] = va;
    f[1] = vb;
    f[2] = make_float4(-va.y, va.x, -va.w, va.z);
    f[3] = make_float4(-vb.y, vb.x, -vb.w, vb.z);
}

// Which of a step's four values lane group l / 16 forms the phasors of: after the swap of step_products the groups hold
// (cos, sin) of values 0 and 1, and of values 2 and 3.
__device__ __forceinline__ int step_value()
{
    const int g = (threadIdx.x & 63) >> 4;
    return ((g & 1) << 1) | (g >> 1);
}

// This lane's factors of the step's values 0 and 1, and 2 and 3; f: the factors of value 0.
__device__ __forceinline__ float2 step_factors(const float *f)
{
    const int at = ((threadIdx.x & 63) >> 4) * 8 + (threadIdx.x & 7);
    return make_float2(f[at], f[at + 32]);
}

// Four values onto one tile; cs, sn: the phasor of this lane's row and value.  Every lane of the wave takes part.
__device__ __forceinline__ void step_products(f32x4 &sums, float2 f, float cs, float sn)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(cs), __float_as_uint(sn), false, false);
    sums = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(r[0]), f.x, sums, 0, 0, 0);
    sums = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(r[1]), f.y, sums, 0, 0, 0);
}

__device__ __forceinline__ void channel_window(const KernelArgs &a, int s, int &c0, int &nc)
{
    if (a.channels)
    {
        const idgx_channels w = a.channels[s];
        c0 = w.channel_begin;
        nc = w.nr_channels;
    }
    else
    {
        c0 = 0;
        nc = a.p.nr_channels;
    }
}

// One pixel of a thread: its coordinates, the phase of the subgrid's offset, and its sums.
struct PlainPixel
{
    float l, m, n, offset;
    float acc[8];
};

__device__ __forceinline__ PlainPixel plain_pixel(const KernelArgs &a, const Offsets &off, int p)
{
    const int S = a.p.S, x = p % S, y = p / S;
    PlainPixel px;
    px.l = pixel_lm(x, S, a.p.image_size);
    px.m = pixel_lm(y, S, a.p.image_size);
    px.n = pixel_n(px.l, px.m);
    px.offset = (off.u * px.l + off.v * px.m) + off.w * px.n;
#pragma unroll
    for (int k = 0; k < 8; ++k)
        px.acc[k] = 0.F;
    return px;
}

// P <- taper * A1^H P A2 of pixel p, overwriting the subgrid's (zeros for a subgrid rejected by its bounds).
__device__ __forceinline__ void store_plain_pixel(const KernelArgs &a, const idgx_metadata &m, int s, int p, bool ok,
                                                  const float *acc)
{
    const int P = a.p.S * a.p.S;
    float2 *out = reinterpret_cast<float2 *>(a.subgrids_out) + static_cast<size_t>(s) * kCorr * P;
    cfloat px[4] = {{acc[0], acc[1]}, {acc[2], acc[3]}, {acc[4], acc[5]}, {acc[6], acc[7]}};
    if (ok)
    {
        const float4 *aterms = reinterpret_cast<const float4 *>(a.aterms);
        const size_t base = static_cast<size_t>(m.aterm_index) * a.p.nr_stations;
        cfloat a1[4], a2[4];
        load_jones(aterms, (base + m.station1) * P + p, a1);
        load_jones(aterms, (base + m.station2) * P + p, a2);
        apply_a1h_p_a2(px, a1, a2);
        const float taper = a.spheroidal[p];
#pragma unroll
        for (int pol = 0; pol < 4; ++pol)
            out[pol * P + p] = make_float2(px[pol].re * taper, px[pol].im * taper);
    }
    else
    {
#pragma unroll
        for (int pol = 0; pol < 4; ++pol)
            out[pol * P + p] = make_float2(0.F, 0.F);
    }
}

// Visibilities whose phasors a gridder of one pixel per thread forms side by side: its independent work in flight (the
// terms are still added in order), and the registers of one pixel leave room for eight waves per SIMD.
constexpr int kGridUnroll = 4;

// A workgroup grids 256 pixels of a subgrid; waves past the last pixel only stage.  VALU issue bound.  Against 4 (S = 32)
// or 3 (S = 24, 48) pixels per thread side by side at five waves per SIMD, 780 baselines x 256 timesteps x 64 channels:
// S = 32 7956 -> 7278 us, S = 48 16333 -> 15777 us, S = 24 (where a third of the lanes' third pixels were idle) 5541 ->
// 4300 us; 45 subgrids of 32^2 with 2048 visibilities each, which leave CUs idle either way, 478 -> 143 us.
// NPIX 3 and 4: large plans whose blocks of 768 or 1024 pixels are whole, where they are faster (launch_grid_plain).
template <int NPIX, int SC>
__global__ __launch_bounds__(kThreads, SC == kSincosHw ? (NPIX == 1 ? 8 : 5) : 1) void gridder_plain(KernelArgs a)
{
    __shared__ float4 s_vis[2 * kGridBatchVis];
    __shared__ float4 s_uvw[kGridBatchVis];
    __shared__ float s_wn[kGridChunk];

    const int s = blockIdx.x;
    const int tid = threadIdx.x;
    const int P = a.p.S * a.p.S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    const bool ok = subgrid_in_bounds(a.p, m, row0, c0, nc);
    const long long C = a.p.nr_channels;
    const Offsets off = gridder_offsets(m, a.p.S, a.p.G, a.p.image_size, a.p.w_step);
    const float4 *vis = reinterpret_cast<const float4 *>(a.visibilities);
    const int pbase = blockIdx.y * (kThreads * NPIX), p = pbase + tid;
    const bool wave_live = pbase + (tid & ~63) < P; // wave-uniform
    PlainPixel px[NPIX];
#pragma unroll
    for (int i = 0; i < NPIX; ++i)
        px[i] = plain_pixel(a, off, min(p + i * kThreads, P - 1));
    for (int cb = 0; ok && cb < nc; cb += kGridChunk)
    {
        const int cc = min(kGridChunk, nc - cb);
        const int tb_max = kGridBatchVis / cc;
        for (int t0 = 0; t0 < m.nr_timesteps; t0 += tb_max)
        {
            const int tb = min(tb_max, m.nr_timesteps - t0);
            __syncthreads(); // previous stage fully consumed
            if (tid < cc)
                s_wn[tid] = a.wavenumbers[c0 + cb + tid];
            for (int q = tid; q < tb; q += kThreads)
            {
                const float *uv = a.uvw + 3 * (row0 + t0 + q);
                s_uvw[q] = make_float4(uv[0], uv[1], uv[2], 0.F);
            }
            for (int q = tid; q < 2 * tb * cc; q += kThreads)
            {
                const int item = q >> 1;
                const int t = item / cc, c = item - t * cc;
                s_vis[q] = vis[((row0 + t0 + t) * C + c0 + cb + c) * 2 + (q & 1)];
            }
            __syncthreads();
            for (int t = 0; wave_live && t < tb; ++t)
            {
                const float4 uv = s_uvw[t];
                float pidx[NPIX];
#pragma unroll
                for (int i = 0; i < NPIX; ++i)
                    pidx[i] = (uv.x * px[i].l + uv.y * px[i].m) + uv.z * px[i].n;
                if constexpr (NPIX == 1)
                {
#pragma unroll kGridUnroll
                    for (int c = 0; c < cc; ++c)
                    {
                        const float phase = px[0].offset - pidx[0] * s_wn[c];
                        float sn, cs;
                        sincos_rad<SC>(phase, sn, cs);
                        cmac4(px[0].acc, s_vis[2 * (t * cc + c)], s_vis[2 * (t * cc + c) + 1], cs, sn);
                    }
                }
                else
                {
                    for (int c = 0; c < cc; ++c)
                    {
                        const float4 va = s_vis[2 * (t * cc + c)], vb = s_vis[2 * (t * cc + c) + 1];
#pragma unroll
                        for (int i = 0; i < NPIX; ++i)
                        {
                            float sn, cs;
                            sincos_rad<SC>(px[i].offset - pidx[i] * s_wn[c], sn, cs);
                            cmac4_pairs(px[i].acc, va, vb, cs, sn);
                        }
                    }
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NPIX; ++i)
        if (p + i * kThreads < P)
            store_plain_pixel(a, m, s, p + i * kThreads, ok, px[i].acc);
}

// Plans that leave SIMDs without a wave of 64 pixels: a wave per 16 pixels, on the matrix cores (a workgroup 64 pixels).
// Bound by latency there (a step of four visibilities is a chain of about ten VALU instructions and two MFMAs), so two
// steps go side by side and the next stage's loads are in flight during the sums.  45 subgrids of 32^2 with 2048
// visibilities each: 156 -> 105 us; on plans that fill the chip the 16-column tile, half of it unused, is slower than the VALU
// (6409 subgrids 6281 -> 9707 us).
template <int SC> __global__ __launch_bounds__(kThreads, 8) void gridder_plain_tiles(KernelArgs a)
{
    constexpr int kPixels = 64;
    __shared__ float4 s_fac[4 * kGridBatchVis];
    __shared__ float s_uvw[3 * kGridBatchVis];
    __shared__ float s_wn[kGridChunk];

    const int s = blockIdx.x;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int P = a.p.S * a.p.S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    const bool ok = subgrid_in_bounds(a.p, m, row0, c0, nc);
    const long long C = a.p.nr_channels;
    const Offsets off = gridder_offsets(m, a.p.S, a.p.G, a.p.image_size, a.p.w_step);
    const float4 *vis = reinterpret_cast<const float4 *>(a.visibilities);
    const int pbase = blockIdx.y * kPixels, pwave = pbase + wave * 16;
    const bool wave_live = pwave < P; // wave-uniform
    const PlainPixel px = plain_pixel(a, off, min(pwave + (lane & 15), P - 1));
    f32x4 sums = {0.F, 0.F, 0.F, 0.F};
    const int mine = step_value();
    for (int cb = 0; ok && cb < nc; cb += kGridChunk)
    {
        const int cc = min(kGridChunk, nc - cb), steps = (cc + 3) >> 2, padded = 4 * steps;
        const int tb_max = kGridBatchVis / padded;
        // This thread's visibility of a stage; channels past the last are zeros, which add nothing.
        const int te = tid / padded, ce = tid - te * padded;
        const float4 zero = make_float4(0.F, 0.F, 0.F, 0.F);
        float4 va = zero, vb = zero;
        const auto load = [&](int t0) {
            if (te < min(tb_max, m.nr_timesteps - t0) && ce < cc)
            {
                const size_t o = static_cast<size_t>((row0 + t0 + te) * C + c0 + cb + ce) * 2;
                va = vis[o];
                vb = vis[o + 1];
            }
            else
                va = vb = zero;
        };
        load(0);
        for (int t0 = 0; t0 < m.nr_timesteps; t0 += tb_max)
        {
            const int tb = min(tb_max, m.nr_timesteps - t0);
            __syncthreads(); // previous stage fully consumed
            if (tid < padded)
                s_wn[tid] = tid < cc ? a.wavenumbers[c0 + cb + tid] : 0.F;
            for (int q = tid; q < 3 * tb; q += kThreads)
                s_uvw[q] = a.uvw[3 * (row0 + t0) + q];
            store_factors(s_fac + 4 * tid, va, vb);
            __syncthreads();
            if (t0 + tb_max < m.nr_timesteps)
                load(t0 + tb_max);
            for (int t = 0; wave_live && t < tb; ++t)
            {
                const float pidx = (s_uvw[3 * t] * px.l + s_uvw[3 * t + 1] * px.m) + s_uvw[3 * t + 2] * px.n;
                const float *fac = reinterpret_cast<const float *>(s_fac + 4 * padded * t);
                const auto step = [&](auto count, int k) {
                    constexpr int N = count.value;
                    float2 f[N];
                    float sn[N], cs[N];
#pragma unroll
                    for (int i = 0; i < N; ++i)
                    {
                        f[i] = step_factors(fac + 64 * (k + i));
                        sincos_rad<SC>(px.offset - pidx * s_wn[4 * (k + i) + mine], sn[i], cs[i]);
                    }
#pragma unroll
                    for (int i = 0; i < N; ++i)
                        step_products(sums, f[i], cs[i], sn[i]);
                };
                int k = 0;
                for (; k + 2 <= steps; k += 2)
                    step(std::integral_constant<int, 2>{}, k);
                for (; k < steps; ++k)
                    step(std::integral_constant<int, 1>{}, k);
            }
        }
    }
    // The sums, per pixel, through LDS (the staging is done with).
    __syncthreads();
    float *out = reinterpret_cast<float *>(s_fac);
    if ((lane & 15) < 8)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            out[(wave * 16 + 4 * (lane >> 4) + j) * 8 + (lane & 7)] = sums[j];
    __syncthreads();
    if (tid < kPixels && pbase + tid < P)
    {
        float acc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            acc[j] = out[tid * 8 + j];
        store_plain_pixel(a, m, s, pbase + tid, ok, acc);
    }
}

// Workgroups per CU with the hardware sin/cos: two channels per thread fit six (the most the 24 KB of LDS allows)
// in 79 VGPRs without spills, four channels per thread fit five in 96 VGPRs.
template <int NCH, int SC> constexpr int degrid_plain_min_blocks()
{
    return SC == kSincosHw ? (NCH <= 2 ? 6 : 5) : 1;
}

template <int NCH, int SC>
__global__ __launch_bounds__(kThreads, (degrid_plain_min_blocks<NCH, SC>())) void degridder_plain(KernelArgs a,
                                                                                                  int per)
{
    constexpr int kUnroll = NCH <= 2 ? 4 : 1; // pixels whose phasors are in flight together (added in order)
    // Per staged pixel: (l, m, n, phase offset), then the four correlations, side by side (one address register
    // serves the pixel loop's three reads).
    __shared__ float4 s_px[3 * kDegridPixBatch];

    // Workgroup b = vblock * n + s: a subgrid's workgroups are spread over the XCDs (balances uneven subgrids).
    const int vblock = blockIdx.x / a.p.nr_subgrids;
    const int s = blockIdx.x - vblock * a.p.nr_subgrids;
    if (vblock >= per)
        return; // uniform
    const int tid = threadIdx.x;
    const int S = a.p.S;
    const int P = S * S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    if (!subgrid_in_bounds(a.p, m, row0, c0, nc) || nc == 0)
        return; // uniform: nothing of this subgrid is written
    const int nchunks = (nc + NCH - 1) / NCH;
    if (static_cast<long long>(vblock) * kThreads >= static_cast<long long>(m.nr_timesteps) * nchunks)
        return; // uniform: no item of this block exists

    const int item = vblock * kThreads + tid;
    const int t = item / nchunks;
    const int cj = (item - t * nchunks) * NCH;
    const bool active = t < m.nr_timesteps;
    const long long C = a.p.nr_channels;

    float u = 0.F, v = 0.F, w = 0.F;
    float k[NCH];
#pragma unroll
    for (int j = 0; j < NCH; ++j)
        k[j] = 0.F;
    if (active)
    {
        const float *uv = a.uvw + 3 * (row0 + t);
        u = uv[0];
        v = uv[1];
        w = uv[2];
#pragma unroll
        for (int j = 0; j < NCH; ++j)
            if (cj + j < nc)
                k[j] = a.wavenumbers[c0 + cj + j];
    }
    float acc[NCH][8];
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
        for (int q = 0; q < 8; ++q)
            acc[j][q] = 0.F;

    const Offsets off = degridder_offsets(m, S, a.p.G, a.p.image_size, a.p.w_step);
    const float2 *sub = reinterpret_cast<const float2 *>(a.subgrids) + static_cast<size_t>(s) * kCorr * P;
    const float4 *aterms = reinterpret_cast<const float4 *>(a.aterms);
    const size_t abase = static_cast<size_t>(m.aterm_index) * a.p.nr_stations;

    for (int pb = 0; pb < P; pb += kDegridPixBatch)
    {
        const int np = min(kDegridPixBatch, P - pb);
        __syncthreads();
        for (int q = tid; q < np; q += kThreads)
        {
            const int p = pb + q;
            const int x = p % S, y = p / S;
            const float taper = a.spheroidal[p];
            cfloat px[4];
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
            {
                const float2 g = sub[pol * P + p];
                px[pol] = {taper * g.x, taper * g.y};
            }
            cfloat a1[4], a2[4];
            load_jones(aterms, (abase + m.station1) * P + p, a1);
            load_jones(aterms, (abase + m.station2) * P + p, a2);
            if (a.p.convention == IDGX_ATERM_REFERENCE)
                apply_a1h_p_a2(px, a1, a2);
            else
                apply_a1_p_a2h(px, a1, a2);
            s_px[3 * q + 1] = make_float4(px[0].re, px[0].im, px[1].re, px[1].im);
            s_px[3 * q + 2] = make_float4(px[2].re, px[2].im, px[3].re, px[3].im);
            const float l = pixel_lm(x, S, a.p.image_size);
            const float mm = pixel_lm(y, S, a.p.image_size);
            const float n = pixel_n(l, mm);
            s_px[3 * q] = make_float4(l, mm, n, (off.u * l + off.v * mm) + off.w * n);
        }
        __syncthreads();
        if (active)
        {
#pragma unroll kUnroll
            for (int q = 0; q < np; ++q)
            {
                const float4 g = s_px[3 * q];
                const float4 pa = s_px[3 * q + 1];
                const float4 pbv = s_px[3 * q + 2];
                const float pidx = (u * g.x + v * g.y) + w * g.z;
#pragma unroll
                for (int j = 0; j < NCH; ++j)
                {
                    if (cj + j < nc)
                    {
                        const float phase = pidx * k[j] - g.w;
                        float sn, cs;
                        sincos_rad<SC>(phase, sn, cs);
                        cmac4(acc[j], pa, pbv, cs, sn);
                    }
                }
            }
        }
    }
    if (active)
    {
        float4 *out = reinterpret_cast<float4 *>(a.visibilities_out);
#pragma unroll
        for (int j = 0; j < NCH; ++j)
            if (cj + j < nc)
            {
                const size_t o = ((row0 + t) * C + c0 + cj + j) * 2;
                out[o] = make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
                out[o + 1] = make_float4(acc[j][4], acc[j][5], acc[j][6], acc[j][7]);
            }
    }
}

// As gridder_plain_tiles, for plans that leave SIMDs with fewer than two waves of 64 visibilities: a wave per 16 items
// (timestep, NCH channels), one tile per channel.  45 subgrids of 32^2 with 2048 visibilities each: 143 -> 94 us (6409
// subgrids 6470 -> 9157 us).
template <int NCH, int SC> __global__ __launch_bounds__(kThreads, 6) void degridder_plain_tiles(KernelArgs a, int per)
{
    constexpr int kItems = kThreads / 4;
    __shared__ float4 s_px[kTilePixBatch];       // (l, m, n, phase offset)
    __shared__ float4 s_fac[4 * kTilePixBatch];  // the corrected pixel's factors

    // Workgroup b = vblock * n + s: a subgrid's workgroups are spread over the XCDs (balances uneven subgrids).
    const int vblock = blockIdx.x / a.p.nr_subgrids;
    const int s = blockIdx.x - vblock * a.p.nr_subgrids;
    if (vblock >= per)
        return; // uniform
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int S = a.p.S;
    const int P = S * S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    if (!subgrid_in_bounds(a.p, m, row0, c0, nc) || nc == 0)
        return; // uniform: nothing of this subgrid is written
    const int nchunks = (nc + NCH - 1) / NCH;
    if (static_cast<long long>(vblock) * kItems >= static_cast<long long>(m.nr_timesteps) * nchunks)
        return; // uniform: no item of this block exists

    const int item = vblock * kItems + 16 * wave + (lane & 15);
    const int t = item / nchunks;
    const int cj = (item - t * nchunks) * NCH;
    const bool active = t < m.nr_timesteps;
    const bool wave_live = __ballot(active) != 0ULL; // wave-uniform; idle rows of a live wave sum phasors of k = 0
    const long long C = a.p.nr_channels;

    float u = 0.F, v = 0.F, w = 0.F;
    float k[NCH];
    f32x4 sums[NCH];
#pragma unroll
    for (int j = 0; j < NCH; ++j)
    {
        k[j] = 0.F;
        sums[j] = f32x4{0.F, 0.F, 0.F, 0.F};
    }
    if (active)
    {
        const float *uv = a.uvw + 3 * (row0 + t);
        u = uv[0];
        v = uv[1];
        w = uv[2];
#pragma unroll
        for (int j = 0; j < NCH; ++j)
            if (cj + j < nc)
                k[j] = a.wavenumbers[c0 + cj + j];
    }

    const Offsets off = degridder_offsets(m, S, a.p.G, a.p.image_size, a.p.w_step);
    const float2 *sub = reinterpret_cast<const float2 *>(a.subgrids) + static_cast<size_t>(s) * kCorr * P;
    const float4 *aterms = reinterpret_cast<const float4 *>(a.aterms);
    const size_t abase = static_cast<size_t>(m.aterm_index) * a.p.nr_stations;
    const int mine = step_value();

    for (int pb = 0; pb < P; pb += kTilePixBatch)
    {
        const int np = min(kTilePixBatch, P - pb); // a multiple of 4: S is even
        __syncthreads();
        for (int q = tid; q < np; q += kThreads)
        {
            const int p = pb + q;
            const int x = p % S, y = p / S;
            const float taper = a.spheroidal[p];
            cfloat px[4];
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
            {
                const float2 g = sub[pol * P + p];
                px[pol] = {taper * g.x, taper * g.y};
            }
            cfloat a1[4], a2[4];
            load_jones(aterms, (abase + m.station1) * P + p, a1);
            load_jones(aterms, (abase + m.station2) * P + p, a2);
            if (a.p.convention == IDGX_ATERM_REFERENCE)
                apply_a1h_p_a2(px, a1, a2);
            else
                apply_a1_p_a2h(px, a1, a2);
            store_factors(s_fac + 4 * q, make_float4(px[0].re, px[0].im, px[1].re, px[1].im),
                          make_float4(px[2].re, px[2].im, px[3].re, px[3].im));
            const float l = pixel_lm(x, S, a.p.image_size);
            const float mm = pixel_lm(y, S, a.p.image_size);
            const float n = pixel_n(l, mm);
            s_px[q] = make_float4(l, mm, n, (off.u * l + off.v * mm) + off.w * n);
        }
        __syncthreads();
        if (!wave_live)
            continue;
        const auto step = [&](auto count, int q) {
            constexpr int N = count.value;
            float2 f[N];
            float sn[N][NCH], cs[N][NCH];
#pragma unroll
            for (int i = 0; i < N; ++i)
            {
                const float4 g = s_px[q + 4 * i + mine];
                f[i] = step_factors(reinterpret_cast<const float *>(s_fac + 4 * (q + 4 * i)));
                const float pidx = (u * g.x + v * g.y) + w * g.z;
#pragma unroll
                for (int j = 0; j < NCH; ++j)
                    sincos_rad<SC>(pidx * k[j] - g.w, sn[i][j], cs[i][j]);
            }
#pragma unroll
            for (int i = 0; i < N; ++i)
#pragma unroll
                for (int j = 0; j < NCH; ++j)
                    step_products(sums[j], f[i], cs[i][j], sn[i][j]);
        };
        int q = 0;
        for (; q + 8 <= np; q += 8)
            step(std::integral_constant<int, 2>{}, q);
        for (; q < np; q += 4)
            step(std::integral_constant<int, 1>{}, q);
    }
    // Row 4 (lane / 16) + i of a tile is the visibility of that lane of the wave.
    float *out = reinterpret_cast<float *>(a.visibilities_out);
    const long long first = active ? (row0 + t) * C + c0 + cj : -1;
    const int count = active ? min(NCH, nc - cj) : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        const int row = 4 * (lane >> 4) + i;
        const long long o = __shfl(first, row);
        const int n = __shfl(count, row);
#pragma unroll
        for (int j = 0; j < NCH; ++j)
            if (j < n && (lane & 15) < 8)
                out[(o + j) * 8 + (lane & 7)] = sums[j][i];
    }
}

// ---- persistent work-queue forms (batches) ---------------------------------------------------------------------
//
// The same arithmetic as the kernels above, item by item from a device queue, over each subgrid's selected
// visibilities: a selection list (vis_index, flagged samples left out) or every (t, c) of its channel window.
// Flagged samples are skipped rather than multiplied by zero.  A skipped zero term leaves a running sum unchanged,
// so a gridder item equals the dense kernel on zeroed visibilities wherever both sum in (t, c) order (windows of at
// most 64 channels; wider windows are summed in 64-channel chunks by the dense kernel).

constexpr int kQueueVis = 256; // gridder entries per LDS stage (one per thread)

struct PlainGridShared
{
    // Per staged entry: its four correlations (two float4), then (k, 0, 0, 0), side by side, so that the entry loop
    // reads all three from one address register with constant offsets.
    float4 ent[3 * kQueueVis];
    float4 run_uvw[kQueueVis]; // uvw of each run of entries that share a timestep
    int run_start[kQueueVis + 1];
    int wave_runs[kThreads / 64];
};

// Per staged pixel: (l, m, n, phase offset), then the four correlations (two float4), side by side, so that the
// pixel loop reads all three from one address register with constant offsets.
struct PlainDegridShared
{
    float4 px[3 * kDegridPixBatch];
};

// Selected visibilities of subgrid s: the list entries (null = dense, every (t, c) of the window) and their count.
__device__ __forceinline__ int plain_selection(const KernelArgs &a, int s, int nr_timesteps, int nc,
                                               const uint32_t *&index)
{
    if (a.vis_index)
    {
        const long long o0 = a.vis_offset[s], o1 = a.vis_offset[s + 1];
        index = a.vis_index + o0;
        return static_cast<int>(o1 - o0);
    }
    index = nullptr;
    return nr_timesteps * nc;
}

// Entry v of a selection as (t, c) relative to the subgrid's first row and channel window; false for a list entry
// outside the window, which the kernels skip.
__device__ __forceinline__ bool plain_entry(const uint32_t *index, int v, int nr_timesteps, int nc, int &t, int &c)
{
    if (index)
    {
        const uint32_t e = index[v];
        t = static_cast<int>(e >> 16);
        c = static_cast<int>(e & 0xffffu);
        return t < nr_timesteps && c < nc;
    }
    t = v / nc;
    c = v - t * nc;
    return true;
}

// The staged runs of visibilities onto N pixels of every thread.
template <int N, int UNROLL, int SC>
__device__ __forceinline__ void grid_runs(const PlainGridShared &sm, int nruns, PlainPixel *px)
{
    for (int r = 0; r < nruns; ++r)
    {
        const float4 uv = sm.run_uvw[r];
        const int e0 = __builtin_amdgcn_readfirstlane(sm.run_start[r]);
        const int e1 = __builtin_amdgcn_readfirstlane(sm.run_start[r + 1]);
        float pidx[N];
#pragma unroll
        for (int i = 0; i < N; ++i)
            pidx[i] = (uv.x * px[i].l + uv.y * px[i].m) + uv.z * px[i].n;
        const auto entry = [&](int e) {
            const float4 va = sm.ent[3 * e];
            const float4 vb = sm.ent[3 * e + 1];
            const float k = sm.ent[3 * e + 2].x;
#pragma unroll
            for (int i = 0; i < N; ++i)
            {
                float sn, cs;
                sincos_rad<SC>(px[i].offset - pidx[i] * k, sn, cs);
                if constexpr (N == 1)
                    cmac4(px[i].acc, va, vb, cs, sn);
                else
                    cmac4_pairs(px[i].acc, va, vb, cs, sn);
            }
        };
        if constexpr (UNROLL > 1)
        {
#pragma unroll UNROLL
            for (int e = e0; e < e1; ++e)
                entry(e);
        }
        else
        {
            for (int e = e0; e < e1; ++e)
                entry(e);
        }
    }
}

// Gridder item: pixels [pblk * 256 * NPIX, ...) of subgrid s.  A wave with fewer than NPIX pixels per thread takes them one
// by one, two visibilities at a time (four spill, and S = 32 runs 2 % slower): S = 24, where three waves of four have two,
// 4982 -> 3964 us (780 baselines x 256 timesteps x 64 channels).
// Entries are staged 256 at a time; the entries of a stage that share a timestep form a run (a workgroup scan over
// "timestep differs from the previous entry"), and each run forms the per-pixel index term (u l + v m) + w n once, as
// the dense kernel does per timestep.
// WHOLE: every item of the launch has all its pixels (the plan's sizes decide), which leaves the kernel without the other
// loop and its registers (three pixels per thread: 94 -> 75 VGPRs, six workgroups per CU for five).
template <int NPIX, int SC, bool WHOLE>
__device__ __forceinline__ void gridder_plain_item(const KernelArgs &a, int s, int pblk, PlainGridShared &sm)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int P = a.p.S * a.p.S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    const bool ok = subgrid_in_bounds(a.p, m, row0, c0, nc);
    const long long C = a.p.nr_channels;
    const int T = m.nr_timesteps;
    const int pbase = pblk * (kThreads * NPIX);
    const Offsets off = gridder_offsets(m, a.p.S, a.p.G, a.p.image_size, a.p.w_step);
    PlainPixel px[NPIX];
    int live = 0; // pixels per thread of this wave (the last may end inside it)
#pragma unroll
    for (int i = 0; i < NPIX; ++i)
    {
        px[i] = plain_pixel(a, off, min(pbase + i * kThreads + tid, P - 1));
        live += pbase + i * kThreads + wave * 64 < P;
    }
    live = __builtin_amdgcn_readfirstlane(live);

    const uint32_t *index = nullptr;
    const int V = ok && T > 0 && nc > 0 ? plain_selection(a, s, T, nc, index) : 0;
    const float4 *vis = reinterpret_cast<const float4 *>(a.visibilities);
    for (int v0 = 0; v0 < V; v0 += kQueueVis)
    {
        const int nb = min(kQueueVis, V - v0);
        __syncthreads(); // the previous stage is consumed
        bool start = false;
        int t = 0;
        if (tid < nb)
        {
            int c = 0;
            float4 va = make_float4(0.F, 0.F, 0.F, 0.F), vb = va;
            float k = 0.F;
            if (plain_entry(index, v0 + tid, T, nc, t, c))
            {
                const size_t o = static_cast<size_t>((row0 + t) * C + c0 + c) * 2;
                va = vis[o];
                vb = vis[o + 1];
                k = a.wavenumbers[c0 + c];
            }
            t = min(t, T - 1); // a skipped entry still names a row inside the subgrid
            sm.ent[3 * tid] = va;
            sm.ent[3 * tid + 1] = vb;
            sm.ent[3 * tid + 2] = make_float4(k, 0.F, 0.F, 0.F);
            start = tid == 0;
            if (!start)
            {
                int tp, cp;
                (void)plain_entry(index, v0 + tid - 1, T, nc, tp, cp);
                start = min(tp, T - 1) != t;
            }
        }
        const unsigned long long mask = __ballot(start);
        const int below = static_cast<int>(__builtin_amdgcn_mbcnt_hi(
            static_cast<unsigned>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(mask), 0u)));
        if (lane == 0)
            sm.wave_runs[wave] = __popcll(mask);
        __syncthreads();
        int before = 0, nruns = 0;
#pragma unroll
        for (int w = 0; w < kThreads / 64; ++w)
        {
            const int r = sm.wave_runs[w];
            before += w < wave ? r : 0;
            nruns += r;
        }
        if (start)
        {
            const int r = before + below;
            const float *uv = a.uvw + 3 * (row0 + t);
            sm.run_start[r] = tid;
            sm.run_uvw[r] = make_float4(uv[0], uv[1], uv[2], 0.F);
        }
        if (tid == 0)
            sm.run_start[nruns] = nb;
        __syncthreads();
        nruns = __builtin_amdgcn_readfirstlane(nruns);
        if (WHOLE || live == NPIX)
        {
            grid_runs<NPIX, NPIX == 1 ? kGridUnroll : 1, SC>(sm, nruns, px);
        }
        else
        {
#pragma unroll
            for (int i = 0; i < NPIX - 1; ++i)
                if (i < live)
                    grid_runs<1, 2, SC>(sm, nruns, px + i);
        }
    }
#pragma unroll
    for (int i = 0; i < NPIX; ++i)
    {
        const int p = pbase + i * kThreads + tid;
        if (p < P)
            store_plain_pixel(a, m, s, p, ok, px[i].acc);
    }
}

// Degridder item: selected visibilities [vblk * 256 * NCH, ...) of subgrid s, NCH consecutive ones per thread.  When
// every thread of a wave holds visibilities of a single timestep (dense windows whose width NCH divides), the index
// term is formed once per pixel for all of them; otherwise once per visibility.
template <int NCH, int SC>
__device__ __forceinline__ void degridder_plain_item(const KernelArgs &a, int s, int vblk, PlainDegridShared &sm)
{
    const int tid = threadIdx.x;
    const int S = a.p.S;
    const int P = S * S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    const int T = m.nr_timesteps;
    if (!subgrid_in_bounds(a.p, m, row0, c0, nc) || nc == 0 || T == 0)
        return; // uniform: nothing of this subgrid is written
    const uint32_t *index = nullptr;
    const int V = plain_selection(a, s, T, nc, index);
    const int ebase = vblk * kThreads * NCH;
    if (ebase >= V)
        return; // uniform: no visibility of this item exists
    const long long C = a.p.nr_channels;

    float u[NCH], v[NCH], w[NCH], k[NCH];
    unsigned valid = 0u;
    int tfirst = -1;
    bool same = true;
#pragma unroll
    for (int j = 0; j < NCH; ++j)
    {
        u[j] = v[j] = w[j] = k[j] = 0.F;
        const int e = ebase + tid * NCH + j;
        int t, c;
        if (e < V && plain_entry(index, e, T, nc, t, c))
        {
            valid |= 1u << j;
            const float *uv = a.uvw + 3 * (row0 + t);
            u[j] = uv[0];
            v[j] = uv[1];
            w[j] = uv[2];
            k[j] = a.wavenumbers[c0 + c];
            same = same && (tfirst < 0 || t == tfirst);
            tfirst = tfirst < 0 ? t : tfirst;
        }
    }
    // The shared index term uses the thread's first visibility with data.
    float us = 0.F, vs = 0.F, ws = 0.F;
#pragma unroll
    for (int j = NCH - 1; j >= 0; --j)
        if (valid & (1u << j))
        {
            us = u[j];
            vs = v[j];
            ws = w[j];
        }
    const bool wave_live = __ballot(valid != 0u) != 0ull;   // wave-uniform
    const bool wave_shared = __ballot(!same) == 0ull;       // wave-uniform
    float acc[NCH][8];
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
        for (int q = 0; q < 8; ++q)
            acc[j][q] = 0.F;

    const Offsets off = degridder_offsets(m, S, a.p.G, a.p.image_size, a.p.w_step);
    const float2 *sub = reinterpret_cast<const float2 *>(a.subgrids) + static_cast<size_t>(s) * kCorr * P;
    const float4 *aterms = reinterpret_cast<const float4 *>(a.aterms);
    const size_t abase = static_cast<size_t>(m.aterm_index) * a.p.nr_stations;
    for (int pb = 0; pb < P; pb += kDegridPixBatch)
    {
        const int np = min(kDegridPixBatch, P - pb);
        __syncthreads();
        for (int q = tid; q < np; q += kThreads)
        {
            const int p = pb + q;
            const int x = p % S, y = p / S;
            const float taper = a.spheroidal[p];
            cfloat px[4];
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
            {
                const float2 g = sub[pol * P + p];
                px[pol] = {taper * g.x, taper * g.y};
            }
            cfloat a1[4], a2[4];
            load_jones(aterms, (abase + m.station1) * P + p, a1);
            load_jones(aterms, (abase + m.station2) * P + p, a2);
            if (a.p.convention == IDGX_ATERM_REFERENCE)
                apply_a1h_p_a2(px, a1, a2);
            else
                apply_a1_p_a2h(px, a1, a2);
            sm.px[3 * q + 1] = make_float4(px[0].re, px[0].im, px[1].re, px[1].im);
            sm.px[3 * q + 2] = make_float4(px[2].re, px[2].im, px[3].re, px[3].im);
            const float l = pixel_lm(x, S, a.p.image_size);
            const float mm = pixel_lm(y, S, a.p.image_size);
            const float n = pixel_n(l, mm);
            sm.px[3 * q] = make_float4(l, mm, n, (off.u * l + off.v * mm) + off.w * n);
        }
        __syncthreads();
        if (!wave_live)
            continue;
        if (NCH > 1 && wave_shared)
        {
            for (int q = 0; q < np; ++q)
            {
                const float4 g = sm.px[3 * q];
                const float4 pa = sm.px[3 * q + 1];
                const float4 pbv = sm.px[3 * q + 2];
                const float pidx = (us * g.x + vs * g.y) + ws * g.z;
                float sn[NCH], cs[NCH];
#pragma unroll
                for (int j = 0; j < NCH; ++j)
                    sincos_rad<SC>(pidx * k[j] - g.w, sn[j], cs[j]);
                cmac4_group<NCH>([&](int j) { return acc[j]; }, pa, pbv, cs, sn);
            }
        }
        else
        {
            for (int q = 0; q < np; ++q)
            {
                const float4 g = sm.px[3 * q];
                const float4 pa = sm.px[3 * q + 1];
                const float4 pbv = sm.px[3 * q + 2];
                float sn[NCH], cs[NCH];
#pragma unroll
                for (int j = 0; j < NCH; ++j)
                {
                    const float pidx = (u[j] * g.x + v[j] * g.y) + w[j] * g.z;
                    sincos_rad<SC>(pidx * k[j] - g.w, sn[j], cs[j]);
                }
                cmac4_group<NCH>([&](int j) { return acc[j]; }, pa, pbv, cs, sn);
            }
        }
    }
    float4 *out = reinterpret_cast<float4 *>(a.visibilities_out);
#pragma unroll
    for (int j = 0; j < NCH; ++j)
    {
        if (!(valid & (1u << j)))
            continue;
        int t, c;
        (void)plain_entry(index, ebase + tid * NCH + j, T, nc, t, c);
        const size_t o = static_cast<size_t>((row0 + t) * C + c0 + c) * 2;
        out[o] = make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
        out[o + 1] = make_float4(acc[j][4], acc[j][5], acc[j][6], acc[j][7]);
    }
}

template <int NPIX, int SC, bool WHOLE>
__global__ __launch_bounds__(kThreads, SC == kSincosHw ? (NPIX == 1 ? 8 : 5) : 4) void gridder_plain_queue(QueueArgs q)
{
    __shared__ PlainGridShared sm;
    int cls, s, blk;
    while (next_queue_item(q, cls, s, blk))
        gridder_plain_item<NPIX, SC, WHOLE>(q.cls[cls], s, blk, sm);
}

// One launch over items of several subgrid classes, each with its class's pixels per thread (q.tiles[class]).
template <int SC>
__global__ __launch_bounds__(kThreads, SC == kSincosHw ? 5 : 4) void gridder_plain_queue_tiles(QueueArgs q)
{
    __shared__ PlainGridShared sm;
    int cls, s, blk;
    while (next_queue_item(q, cls, s, blk))
    {
        switch (q.tiles[cls]) // workgroup-uniform
        {
        case 1:
            gridder_plain_item<1, SC, false>(q.cls[cls], s, blk, sm);
            break;
        case 2:
            gridder_plain_item<2, SC, false>(q.cls[cls], s, blk, sm);
            break;
        case 3:
            gridder_plain_item<3, SC, false>(q.cls[cls], s, blk, sm);
            break;
        default:
            gridder_plain_item<4, SC, false>(q.cls[cls], s, blk, sm);
            break;
        }
    }
}

// Workgroups per CU of the queue degridder with the hardware sin/cos: it also holds every visibility's uvw and, for
// several visibilities per thread, runs one of two inner loops, so it keeps fewer workgroups than the dense kernel:
// the most that leave no spills (96, 128 and 168 VGPRs for 1, 2 and 4 visibilities per thread).
template <int NCH, int SC> constexpr int degrid_plain_queue_min_blocks()
{
    return SC == kSincosHw ? (NCH == 1 ? 5 : NCH == 2 ? 4 : 3) : 1;
}

template <int NCH, int SC>
__global__ __launch_bounds__(kThreads, (degrid_plain_queue_min_blocks<NCH, SC>())) void degridder_plain_queue(
    QueueArgs q)
{
    __shared__ PlainDegridShared sm;
    int cls, s, blk;
    while (next_queue_item(q, cls, s, blk))
        degridder_plain_item<NCH, SC>(q.cls[cls], s, blk, sm);
}

// Shapes of the persistent plain kernels: {gridder pixels per thread, degridder visibilities per thread}.
constexpr PlainShape kPlainShapes[] = {{4, 2}, {3, 4}, {2, 1}};
constexpr int kNumPlainShapes = sizeof(kPlainShapes) / sizeof(kPlainShapes[0]);

template <int PIXELS, int SC> void *plain_grid_queue_fn(bool whole)
{
    return whole ? reinterpret_cast<void *>(&gridder_plain_queue<PIXELS, SC, true>)
                 : reinterpret_cast<void *>(&gridder_plain_queue<PIXELS, SC, false>);
}

template <int SC> void *plain_grid_queue_fn(int pixels, bool whole)
{
    switch (pixels)
    {
    case kShapeTilesPerClass:
        return reinterpret_cast<void *>(&gridder_plain_queue_tiles<SC>);
    case 1:
        return reinterpret_cast<void *>(&gridder_plain_queue<1, SC, false>);
    case 2:
        return plain_grid_queue_fn<2, SC>(whole);
    case 3:
        return plain_grid_queue_fn<3, SC>(whole);
    case 4:
        return plain_grid_queue_fn<4, SC>(whole);
    default:
        return nullptr;
    }
}

template <int SC> void *plain_degrid_queue_fn(int entries)
{
    switch (entries)
    {
    case 1:
        return reinterpret_cast<void *>(&degridder_plain_queue<1, SC>);
    case 2:
        return reinterpret_cast<void *>(&degridder_plain_queue<2, SC>);
    case 4:
        return reinterpret_cast<void *>(&degridder_plain_queue<4, SC>);
    default:
        return nullptr;
    }
}

void *plain_queue_fn(const PlainKernel &k)
{
    if (k.gridder)
        return k.accurate_sincos ? plain_grid_queue_fn<kSincosOcml>(k.work, k.whole)
                                 : plain_grid_queue_fn<kSincosHw>(k.work, k.whole);
    return k.accurate_sincos ? plain_degrid_queue_fn<kSincosOcml>(k.work) : plain_degrid_queue_fn<kSincosHw>(k.work);
}
} // namespace

hipError_t launch_plain_queue(const QueueArgs &q, const PlainKernel &k, int workgroups, hipStream_t st)
{
    void *fn = plain_queue_fn(k);
    if (!fn || workgroups <= 0)
        return hipErrorInvalidValue;
    QueueArgs arg = q;
    void *args[] = {&arg};
    return hipLaunchKernel(fn, dim3(workgroups), dim3(kThreads), args, 0, st);
}

// Waves of 64 pixels (visibilities) up to which a one-shot plan takes the tile forms: one per SIMD for the gridder, whose
// time does not fall below one wave's (45 subgrids of 32^2, 720 waves: 156 -> 105 us; 66, 1056 waves: 185 -> 159; 91, 1456
// waves: 189 -> 187; 120 of 24^2, 1080 waves: 67 -> 69), two for the degridder (1440 waves: 143 -> 94 us; 120 subgrids of
// 48^2, 1920 waves: 306 -> 268; 91 of 32^2, 2912 waves: 168 -> 179).
constexpr long long kTileGridWaves = 1024, kTileDegridWaves = 2048;

template <int NPIX> hipError_t launch_grid_plain_pixels(const KernelArgs &a, bool accurate_sincos, hipStream_t stream)
{
    const dim3 grid(a.p.nr_subgrids, (a.p.S * a.p.S + kThreads * NPIX - 1) / (kThreads * NPIX));
    if (accurate_sincos)
        gridder_plain<NPIX, kSincosOcml><<<grid, kThreads, 0, stream>>>(a);
    else
        gridder_plain<NPIX, kSincosHw><<<grid, kThreads, 0, stream>>>(a);
    return hipGetLastError();
}

// Pixels per thread of the one-shot gridder: the tile kernel's for the smallest plans, else one, but four (or three,
// plain_grid_pixels_for) in large plans whose blocks of that many are nearly whole, for large subgrids and with the
// accurate sine and cosine.  2100 subgrids, one pixel / four or three: 96^2 with 16 and 128 visibilities 318 / 315 and
// 1413 / 1389 us, 128^2 with 16 555 / 553, but 64^2 with 1024 4353 / 4331; accurate, 64^2 with 16 and 128 211 / 196 and
// 1000 / 973, 128^2 with 128 3895 / 3560.
int oneshot_grid_pixels(const PlanDev &p, bool accurate_sincos)
{
    constexpr long long kBlocks = 2048;
    const long long P = static_cast<long long>(p.S) * p.S;
    if (p.nr_subgrids * ((P + 63) / 64) <= kTileGridWaves)
        return 0;
    const int n = plain_grid_pixels_for(p.S);
    const long long blocks = (P + kThreads * n - 1) / (kThreads * n);
    const bool whole = 100 * P >= 88 * blocks * kThreads * n;
    return whole && blocks * p.nr_subgrids >= kBlocks && p.S >= (accurate_sincos ? 32 : 72) ? n : 1;
}

hipError_t launch_grid_plain(const KernelArgs &a, bool accurate_sincos, hipStream_t stream)
{
    switch (oneshot_grid_pixels(a.p, accurate_sincos))
    {
    case 4:
        return launch_grid_plain_pixels<4>(a, accurate_sincos, stream);
    case 3:
        return launch_grid_plain_pixels<3>(a, accurate_sincos, stream);
    case 1:
        return launch_grid_plain_pixels<1>(a, accurate_sincos, stream);
    default:
        break;
    }
    const dim3 grid(a.p.nr_subgrids, static_cast<unsigned>((static_cast<long long>(a.p.S) * a.p.S + 63) / 64));
    if (accurate_sincos)
        gridder_plain_tiles<kSincosOcml><<<grid, kThreads, 0, stream>>>(a);
    else
        gridder_plain_tiles<kSincosHw><<<grid, kThreads, 0, stream>>>(a);
    return hipGetLastError();
}

// Items of the default shapes, or one-shot degridder workgroups, that fill the chip.  Smaller plans run one pixel or
// visibility per thread.  Batches of 45 subgrids of 32^2 with 2048 visibilities each: gridder 586 -> 360 us, degridder
// 291 -> 246 us; 276 of them 753 -> 577 us, where the degridder gains at S = 32 and 48 (436 -> 411 us) and loses at S = 24
// (262 -> 286 us), so its line lies below (1104 items).
constexpr long long kGridFill = 2048, kDegridItems = 1024, kDegridFill = 1280;
constexpr long long kGridFewItems = 1024, kFineVisibilities = 512, kFinePairs = 110000; // plain_fine_items

template <int NCH> hipError_t launch_degrid_plain_chunks(const KernelArgs &a, bool accurate_sincos, hipStream_t stream)
{
    const long long items = static_cast<long long>(a.p.max_nr_timesteps) * ((a.p.nr_channels + NCH - 1) / NCH);
    const long long per = items > 0 ? (items + kThreads - 1) / kThreads : 1;
    const long long blocks = static_cast<long long>(a.p.nr_subgrids) * per;
    if (blocks > 0x7fffffffLL)
        return hipErrorInvalidConfiguration;
    const dim3 grid(static_cast<unsigned>(blocks));
    if (accurate_sincos)
        degridder_plain<NCH, kSincosOcml><<<grid, kThreads, 0, stream>>>(a, static_cast<int>(per));
    else
        degridder_plain<NCH, kSincosHw><<<grid, kThreads, 0, stream>>>(a, static_cast<int>(per));
    return hipGetLastError();
}

// Channels per degridder thread.  Four make each pixel's LDS reads and index term serve more visibilities, but a
// chunk that runs past the end of a subgrid's channel window idles its lanes: four channels when every subgrid
// takes all channels (no windows) and their count is a multiple of 4, two otherwise.  Measured: the reference
// generator's workload (16 channels, no windows) 17.1 ms with four, 18.3 ms with two; the SKA-Low-like workload
// (windows of 13.5 channels on average: 90 % of the lanes busy with four, 96.7 % with two) 82.3 and 79.6 ms.
// Plans too small to fill the chip take one: 45 subgrids of 32^2 with 2048 visibilities each 202 -> 143 us, 276 of them
// 428 -> 385 us (496: 628 -> 640 us).
int oneshot_degrid_channels(const PlanDev &p, bool channel_windows)
{
    const long long pairs = static_cast<long long>(p.max_nr_timesteps) * ((p.nr_channels + 1) / 2);
    if ((2 * pairs + 63) / 64 * p.nr_subgrids <= kTileDegridWaves)
        return 0;
    if ((pairs + kThreads - 1) / kThreads * p.nr_subgrids < kDegridFill)
        return 1;
    return plain_degrid_channels_for(channel_windows, p.nr_channels);
}

hipError_t launch_degrid_plain(const KernelArgs &a, bool accurate_sincos, hipStream_t stream)
{
    switch (oneshot_degrid_channels(a.p, a.channels != nullptr))
    {
    case 4:
        return launch_degrid_plain_chunks<4>(a, accurate_sincos, stream);
    case 2:
        return launch_degrid_plain_chunks<2>(a, accurate_sincos, stream);
    case 1:
        return launch_degrid_plain_chunks<1>(a, accurate_sincos, stream);
    default:
        break;
    }
    const long long pairs = static_cast<long long>(a.p.max_nr_timesteps) * ((a.p.nr_channels + 1) / 2);
    const long long per = std::max(1LL, (pairs + kThreads / 4 - 1) / (kThreads / 4));
    const unsigned blocks = static_cast<unsigned>(per * a.p.nr_subgrids);
    if (accurate_sincos)
        degridder_plain_tiles<2, kSincosOcml><<<blocks, kThreads, 0, stream>>>(a, static_cast<int>(per));
    else
        degridder_plain_tiles<2, kSincosHw><<<blocks, kThreads, 0, stream>>>(a, static_cast<int>(per));
    return hipGetLastError();
}

// Pixels per thread of a batch's gridder items for subgrid size S: 4 (1024 per item) unless 3 (768) fits the subgrid
// better, as for S = 24 (576 pixels) and S = 48 (2304).
int plain_grid_pixels_for(int S)
{
    const long long P = static_cast<long long>(S) * S;
    const long long slots4 = (P + 1023) / 1024 * 1024, slots3 = (P + 767) / 768 * 768;
    return slots3 < slots4 ? 3 : 4;
}

// Channels per degridder thread (see launch_degrid_plain).
int plain_degrid_channels_for(bool channel_windows, int nr_channels)
{
    return !channel_windows && nr_channels % 4 == 0 ? 4 : 2;
}

int plain_shape_count()
{
    return kNumPlainShapes;
}

PlainShape plain_shape(int i)
{
    return kPlainShapes[i];
}

int plain_default_shape(bool gridder, int S)
{
    if (!gridder)
        return 0; // two visibilities per thread
    const int px = plain_grid_pixels_for(S);
    for (int i = 0; i < kNumPlainShapes; ++i)
        if (kPlainShapes[i].pixels == px)
            return i;
    return 0;
}

// One pixel per thread makes three to nine items of one: each costs the queue 0.1 us, and of 256 pixels saves 0.15 us per
// visibility of the subgrid as long as the chip is not full.  Gridder time over that of the default shapes, by
// visibilities a subgrid: 512 of 32^2 (2048 items for 512) 16 1.68, 256 1.27, 512 0.85; 1000 of them 256 1.35, 512 0.97,
// 1024 0.86; 2000 512 1.11, 1024 0.99; 276 of 24^2 (828 for 276) 0.6 to 0.7 at any count.
// Degridder: subgrids of up to 256 visibilities leave half the waves of an item of 512 without any (3000 of 48^2 with 128
// 0.73, 256 0.95); beyond, small plans where an item of 256 has kFinePairs pixels x visibilities (1000 of 24^2 with 288
// 1.09, of 32^2 0.97).
bool plain_fine_items(bool gridder, const PlainWork &w)
{
    if (!gridder)
        return w.visibilities <= w.subgrids * kThreads ||
               (w.items < kDegridItems &&
                (w.fine_degrid_items <= kDegridFill || w.pairs >= w.fine_degrid_items * kFinePairs));
    return w.fine_grid_items <= kGridFewItems ||
           (w.items < kGridFill && w.visibilities >= w.subgrids * kFineVisibilities &&
            (w.items < kGridFill / 2 || w.visibilities >= w.subgrids * 2 * kFineVisibilities));
}

int plain_grid_items_per_subgrid(int pixels, int S)
{
    const long long per = static_cast<long long>(kThreads) * pixels;
    return static_cast<int>((static_cast<long long>(S) * S + per - 1) / per);
}

long long plain_grid_item_pixels(int pixels, int S, int item)
{
    const long long per = static_cast<long long>(kThreads) * pixels;
    const long long P = static_cast<long long>(S) * S;
    return std::max(0LL, std::min(per, P - item * per));
}

int plain_degrid_visibilities_per_item(int entries)
{
    return kThreads * entries;
}

int plain_queue_workgroups(const PlainKernel &k)
{
    void *fn = plain_queue_fn(k);
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
