// Device code of the mixed-precision kernels: operand packing and hi/lo splits, the FP64 phase reduction, visibility
// selections, and the items (a block of pixels, a chunk of visibilities) of the kernels that evaluate a phasor per
// (pixel, visibility) pair.  Shared by the translation units of the per-pair and the separable kernels.
#pragma once

#include "idgx_device.hpp"
#include "kernels.hpp"

namespace idgx
{
namespace
{
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

enum DType
{
    kBF16 = 0,
    kFP16 = 1
};

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr float kTurnsMost = 4.F; // separable kernels, |d a|: keeps the phases' FP32 rounding at the level of qu xh
// Default tile shape: gridder 8 tiles of 16 pixels per wave with 256 visibilities per LDS batch, degridder 4 tiles
// of 16 visibilities per wave with 256 pixels per LDS batch.
constexpr int kDefaultPT = 8, kDefaultVB = 256, kDefaultVT = 4, kDefaultPB = 256;

// Round a pair of floats to two 16-bit values (RNE), x0 in the low half.
template <int DT> __device__ __forceinline__ uint32_t pack2(float x0, float x1)
{
    if constexpr (DT == kBF16)
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x0, x1}, bf16x2));
    else
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x0, x1}, f16x2));
}

template <int DT> __device__ __forceinline__ void unpack2(uint32_t p, float &y0, float &y1)
{
    if constexpr (DT == kBF16)
    {
        y0 = __builtin_bit_cast(float, p << 16);
        y1 = __builtin_bit_cast(float, p & 0xffff0000u);
    }
    else
    {
        const f16x2 h = __builtin_bit_cast(f16x2, p);
        y0 = static_cast<float>(h[0]);
        y1 = static_cast<float>(h[1]);
    }
}

// x - float(half of h) in one v_fma_mix_f32 (the half is read straight from the packed register).  The result
// is exact: x and its RNE fp16 rounding are close enough for the difference to be a float.  (Writing the rounded
// residual straight into a register half with v_fma_mixlo/mixhi_f16 saves the pack but measured slower.)
__device__ __forceinline__ float sub_f16_lo(float x, uint32_t h)
{
    float r;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
    return r;
}
__device__ __forceinline__ float sub_f16_hi(float x, uint32_t h)
{
    float r;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(x));
    return r;
}

// hi = round(x), lo = round(x - hi), both packed as pairs.
template <int DT> __device__ __forceinline__ void split2(float x0, float x1, uint32_t &hi, uint32_t &lo)
{
    hi = pack2<DT>(x0, x1);
    if constexpr (DT == kFP16)
    {
        lo = pack2<DT>(sub_f16_lo(x0, hi), sub_f16_hi(x1, hi));
    }
    else
    {
        float h0, h1;
        unpack2<DT>(hi, h0, h1);
        lo = pack2<DT>(x0 - h0, x1 - h1);
    }
}

// FP16 B operands are scaled by a power of two per LDS batch so that the largest staged value is about 2^14:
// no overflow (65504) for any data, and the hi/lo split keeps its relative precision.  The accumulators are
// rescaled exactly when a later batch needs a larger scale, and the final result is multiplied back.
constexpr int kF16TargetExp = 14;

// Never below -126, whose inverse is still finite: fainter values (below 2^-112) stay that much smaller instead.
__device__ __forceinline__ int scale_exponent(float maxabs)
{
    if (!(maxabs > 0.F))
        return -126;
    int e;
    (void)frexpf(maxabs, &e); // maxabs in [2^(e-1), 2^e)
    return max(e - kF16TargetExp, -126);
}

// Phases of a 16 x 16 tile: D[i][j] = sum_k A[i][k] B[k][j], K = 4 (fourth component zero).
__device__ __forceinline__ f32x4 phase_mfma(float a, float b)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, (f32x4){0.F, 0.F, 0.F, 0.F}, 0, 0, 0);
}


__device__ __forceinline__ f32x4 mfma(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3, u32x4 b, f32x4 c,
                                      std::integral_constant<int, kBF16>)
{
    const u32x4 a = {a0, a1, a2, a3};
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3, u32x4 b, f32x4 c,
                                      std::integral_constant<int, kFP16>)
{
    const u32x4 a = {a0, a1, a2, a3};
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                  0, 0);
}

// Writes the B-operand words of one k-pair item (a visibility for the gridder, a pixel for the degridder) with
// complex values v[0..3] into a 1 KiB LDS block laid out as [lane][4 words]: item q of the block occupies word
// (q % 4) of lanes (q / 4) * 16 + n, n = column.  Columns 0-7 carry the high parts, 8-15 the low parts.
// Packed (re, im) high and low parts of the four correlations (low parts zero without the split).
template <int DT, bool SPLIT>
__device__ __forceinline__ void split_item(const cfloat *v, uint32_t *hi, uint32_t *lo)
{
#pragma unroll
    for (int pol = 0; pol < 4; ++pol)
    {
        split2<DT>(v[pol].re, v[pol].im, hi[pol], lo[pol]);
        if (!SPLIT)
            lo[pol] = 0;
    }
}

__device__ __forceinline__ void write_b_words(uint32_t *blk, int q, const uint32_t *hip, const uint32_t *lop)
{
    const int kg = q >> 2, slot = q & 3;
    uint32_t *base = blk + kg * 64 + slot;
#pragma unroll
    for (int pol = 0; pol < 4; ++pol)
    {
        const uint32_t hi = hip[pol], lo = lop[pol];
        // hi = (re | im << 16).  Column re: (cos row re, sin row -im); column im: (cos row im, sin row re).
        const uint32_t re_col_hi = (hi & 0xffffu) | ((hi ^ 0x80000000u) & 0xffff0000u);
        const uint32_t im_col_hi = (hi >> 16) | (hi << 16);
        const uint32_t re_col_lo = (lo & 0xffffu) | ((lo ^ 0x80000000u) & 0xffff0000u);
        const uint32_t im_col_lo = (lo >> 16) | (lo << 16);
        base[(2 * pol) * 4] = re_col_hi;
        base[(2 * pol + 1) * 4] = im_col_hi;
        base[(8 + 2 * pol) * 4] = re_col_lo;
        base[(8 + 2 * pol + 1) * 4] = im_col_lo;
    }
}

template <int DT, bool SPLIT> __device__ __forceinline__ void write_b_item(uint32_t *blk, int q, const cfloat *v)
{
    uint32_t hi[4], lo[4];
    split_item<DT, SPLIT>(v, hi, lo);
    write_b_words(blk, q, hi, lo);
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

struct CentreOffsets
{
    double u, v, w; // wavelengths
};

__device__ __forceinline__ CentreOffsets centre_offsets(const PlanDev &p, const idgx_metadata &m)
{
    const double inv_image = 1.0 / static_cast<double>(p.image_size);
    CentreOffsets o;
    o.u = (m.x + p.S * 0.5 - p.G * 0.5) * inv_image;
    o.v = (m.y + p.S * 0.5 - p.G * 0.5) * inv_image;
    o.w = static_cast<double>(p.w_step) * (m.z + 0.5);
    return o;
}

constexpr double kInv2Pi = 0.15915494309189533577;

// Reduced phase coordinates of one visibility (revolutions), signed by sgn: per-pixel-step slopes qu, qv in
// [-1/2, 1/2], the w slope dw per unit n, and the constant rot = (qu + qv)/2 mod 1.
struct Reduced
{
    float qu, qv, dw, rot;
};

__device__ __forceinline__ Reduced reduce_visibility(const float *uvw, float k, const CentreOffsets &o, double delta,
                                                     float sgn)
{
    const double kk = static_cast<double>(k) * kInv2Pi;
    const double qu = __builtin_fma(kk, static_cast<double>(uvw[0]), -o.u) * delta;
    const double qv = __builtin_fma(kk, static_cast<double>(uvw[1]), -o.v) * delta;
    const double dw = __builtin_fma(kk, static_cast<double>(uvw[2]), -o.w);
    double rot = 0.5 * (qu + qv);
    rot -= __builtin_rint(rot);
    Reduced r;
    r.qu = sgn * static_cast<float>(qu - __builtin_rint(qu));
    r.qv = sgn * static_cast<float>(qv - __builtin_rint(qv));
    r.dw = sgn * static_cast<float>(dw);
    r.rot = sgn * static_cast<float>(rot);
    return r;
}

// c * e^{2 pi i rot} for the four correlations.
__device__ __forceinline__ void rotate4(cfloat *v, float rot)
{
    const float sn = __builtin_amdgcn_sinf(rot), cs = __builtin_amdgcn_cosf(rot);
#pragma unroll
    for (int pol = 0; pol < 4; ++pol)
        v[pol] = {v[pol].re * cs - v[pol].im * sn, v[pol].re * sn + v[pol].im * cs};
}

__device__ __forceinline__ float pixel_lm_f(int x, int S, float image_size)
{
    return (static_cast<float>(x) + 0.5F - 0.5F * static_cast<float>(S)) * (image_size / static_cast<float>(S));
}

// x' = x - S/2, exact in float.
__device__ __forceinline__ float pixel_offset(int x, int S)
{
    return static_cast<float>(x - S / 2);
}

__device__ __forceinline__ float pixel_n_f(float l, float m)
{
    const float r2 = l * l + m * m;
    return r2 > 1.F ? 1.F : r2 / (1.F + __builtin_sqrtf(1.F - r2));
}

// The visibility v of subgrid s: (t, c) relative to its first row / channel window, and the subgrid's count.
struct Selection
{
    const uint32_t *index; // null: dense (t, c) = (v / nc, v % nc)
    int nc;
    __device__ __forceinline__ void at(int v, int &t, int &c) const
    {
        if (index)
        {
            const uint32_t e = index[v];
            t = static_cast<int>(e >> 16);
            c = static_cast<int>(e & 0xffffu);
        }
        else
        {
            t = v / nc;
            c = v - t * nc;
        }
    }
};

__device__ __forceinline__ int selection_of(const KernelArgs &a, int s, int nr_timesteps, int nc, Selection &sel)
{
    sel.nc = nc;
    if (a.vis_index)
    {
        const long long o0 = a.vis_offset[s], o1 = a.vis_offset[s + 1];
        sel.index = a.vis_index + o0;
        return static_cast<int>(o1 - o0);
    }
    sel.index = nullptr;
    return nr_timesteps * nc;
}

// Selected entries must lie inside the subgrid's window (entries outside are treated as empty visibilities).
__device__ __forceinline__ bool entry_ok(int t, int c, int nr_timesteps, int nc)
{
    return t >= 0 && t < nr_timesteps && c >= 0 && c < nc;
}

// Largest value over the workgroup (non-negative floats order like their bit patterns).
__device__ __forceinline__ float block_max(float v, unsigned &slot)
{
    if (threadIdx.x == 0)
        slot = 0u;
    __syncthreads();
    atomicMax(&slot, __float_as_uint(v));
    __syncthreads();
    const float m = __uint_as_float(slot);
    __syncthreads();
    return m;
}

// Degridder input pixel p: taper x (A1 P A2^H, or A1^H P A2 in the reference convention) of the subgrid values.
__device__ __forceinline__ void degrid_pixel(const KernelArgs &a, const idgx_metadata &m, const float2 *sub, int p,
                                             cfloat *px)
{
    const int P = a.p.S * a.p.S;
    const float taper = a.spheroidal[p];
#pragma unroll
    for (int pol = 0; pol < 4; ++pol)
    {
        const float2 g = sub[pol * P + p];
        px[pol] = {taper * g.x, taper * g.y};
    }
    const float4 *aterms = reinterpret_cast<const float4 *>(a.aterms);
    const size_t abase = static_cast<size_t>(m.aterm_index) * a.p.nr_stations;
    cfloat a1[4], a2[4];
    load_jones(aterms, (abase + m.station1) * P + p, a1);
    load_jones(aterms, (abase + m.station2) * P + p, a2);
    if (a.p.convention == IDGX_ATERM_REFERENCE)
        apply_a1h_p_a2(px, a1, a2);
    else
        apply_a1_p_a2h(px, a1, a2);
}

struct WRange
{
    double centre; // middle of k w / 2 pi over the subgrid's rows and channels
    float half;    // half its width
};

// Range of w (wavelengths) over a subgrid's rows and channel window, and the largest vmax: every thread of the workgroup
// gets the same.  One LDS-only barrier, which also covers what the caller has written (loads stay in flight across it).
template <int WAVES, bool MAX>
__device__ __forceinline__ WRange w_range(const KernelArgs &a, long long row0, int T, int c0, int nc,
                                          float (&slots)[WAVES][5], float &vmax)
{
    float wlo = __builtin_inff(), whi = -__builtin_inff(), klo = __builtin_inff(), khi = -__builtin_inff();
    for (int t = threadIdx.x; t < T; t += 64 * WAVES)
    {
        const float w = a.uvw[3 * (row0 + t) + 2];
        wlo = fminf(wlo, w);
        whi = fmaxf(whi, w);
    }
    for (int c = threadIdx.x; c < nc; c += 64 * WAVES)
    {
        const float k = a.wavenumbers[c0 + c];
        klo = fminf(klo, k);
        khi = fmaxf(khi, k);
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
    {
        wlo = fminf(wlo, __shfl_xor(wlo, d));
        whi = fmaxf(whi, __shfl_xor(whi, d));
        klo = fminf(klo, __shfl_xor(klo, d));
        khi = fmaxf(khi, __shfl_xor(khi, d));
        if constexpr (MAX)
            vmax = fmaxf(vmax, __shfl_xor(vmax, d));
    }
    if ((threadIdx.x & 63) == 0)
    {
        float *s = slots[threadIdx.x >> 6];
        s[0] = wlo, s[1] = whi, s[2] = klo, s[3] = khi, s[4] = vmax;
    }
    lds_barrier();
#pragma unroll
    for (int w = 0; w < WAVES; ++w)
    {
        wlo = fminf(wlo, slots[w][0]);
        whi = fmaxf(whi, slots[w][1]);
        klo = fminf(klo, slots[w][2]);
        khi = fmaxf(khi, slots[w][3]);
        if constexpr (MAX)
            vmax = fmaxf(vmax, slots[w][4]);
    }
    const double p0 = static_cast<double>(wlo) * klo, p1 = static_cast<double>(wlo) * khi;
    const double p2 = static_cast<double>(whi) * klo, p3 = static_cast<double>(whi) * khi;
    const double lo = fmin(fmin(p0, p1), fmin(p2, p3)) * kInv2Pi, hi = fmax(fmax(p0, p1), fmax(p2, p3)) * kInv2Pi;
    return {0.5 * (lo + hi), static_cast<float>(0.5 * (hi - lo))};
}

// Whether the separable kernels take a subgrid whose w spreads by `half` to both sides (false for NaN).
__device__ __forceinline__ bool separable_fits(const SeparableLimits &l, float half)
{
    return half * l.eps <= l.eps_most && half * l.a_max <= kTurnsMost;
}

// Whether a one-shot workgroup has nothing to do: a separable launch before this one has done subgrid s, by the range of w
// that it decides by, or the subgrid has no visibility `first`.  Uniform.
__device__ __forceinline__ bool separable_done(const KernelArgs &a, int s, long long first, float (&slots)[kWaves][5])
{
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    Selection sel;
    if (!subgrid_in_bounds(a.p, m, row0, c0, nc) || selection_of(a, s, m.nr_timesteps, nc, sel) <= first)
        return true;
    float none = 0.F;
    return separable_fits(a.limits, w_range<kWaves, false>(a, row0, m.nr_timesteps, c0, nc, slots, none).half);
}

template <int PT, int VB> struct GridderShared
{
    unsigned maxbits;
    u32x4 b[(VB / 16) * 64];
    float coef[(VB / 16) * 64];
    float pix[kWaves * PT * 16 * 8];
};

template <int VT, int PB> struct DegridderShared
{
    unsigned maxbits;
    u32x4 b[(PB / 16) * 64];
    float coord[(PB / 16) * 64];
    float vis[kWaves * VT * 16 * 8];
};

// ---------------------------------------------------------------------------------------------------------------
// Gridder item: 4 waves x PT tiles x 16 pixels (block pblk) of subgrid s; visibilities staged VB at a time.
// ---------------------------------------------------------------------------------------------------------------
template <int DT, bool SPLIT, int PT, int VB, bool PM, class Shared>
__device__ __forceinline__ void gridder_item(const KernelArgs &a, int s, int pblk, Shared &sm)
{
    constexpr int kBlocks = VB / 16;
    constexpr int kPix = kWaves * PT * 16;
    static_assert(sizeof(sm.b) == sizeof(u32x4) * kBlocks * 64 && sizeof(sm.pix) >= sizeof(float) * kPix * 8,
                  "LDS staging of the item's shape");
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int S = a.p.S, P = S * S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    const bool ok = subgrid_in_bounds(a.p, m, row0, c0, nc);
    const long long C = a.p.nr_channels;

    // This wave's unit: a strip of gu.wd columns by gu.rows rows; lane row r of tile t is pixel (px, y0 + t*rt).
    const GridUnits gu = grid_units(S, PT);
    const int unit = kWaves * pblk + wave;
    const bool active = unit < gu.units; // wave-uniform
    const int px = (unit % gu.ns) * gu.wd + (lane & 15) % gu.wd;
    const int py0 = (unit / gu.ns) * gu.rows + (lane & 15) / gu.wd;

    // Pixel coordinates of row lane%16 of each tile: x' (the same in every tile), y', n; for PM only component
    // lane/16 of them (the B operand of the phase MFMA).  Rows past the subgrid repeat the last row.
    const float xp = pixel_offset(px, S);
    const float lx = pixel_lm_f(px, S, a.p.image_size);
    float coord[PT], yp[PT], nn[PT];
#pragma unroll
    for (int t = 0; t < PT; ++t)
    {
        const int y = min(py0 + t * gu.rt, S - 1);
        const int kk = lane >> 4;
        yp[t] = pixel_offset(y, S);
        nn[t] = pixel_n_f(lx, pixel_lm_f(y, S, a.p.image_size));
        coord[t] = kk == 0 ? xp : kk == 1 ? yp[t] : kk == 2 ? nn[t] : 0.F;
    }
    f32x4 acc[PT];
#pragma unroll
    for (int t = 0; t < PT; ++t)
        acc[t] = (f32x4){0.F, 0.F, 0.F, 0.F};
    int scale_exp = -126; // FP16: current power-of-two scale of the staged B operand

    Selection sel;
    const int V = ok ? selection_of(a, s, m.nr_timesteps, nc, sel) : 0;
    const CentreOffsets off = centre_offsets(a.p, m);
    const double delta = static_cast<double>(a.p.image_size) / S;
    const float4 *vis = reinterpret_cast<const float4 *>(a.visibilities);
    uint32_t *s_bw = reinterpret_cast<uint32_t *>(sm.b);

    for (int v0 = 0; v0 < V; v0 += VB)
    {
        __syncthreads();
        // Stage visibilities: reduced phase coefficients and B-operand words (scaled for FP16).
        constexpr int kPer = (VB + kThreads - 1) / kThreads;
        cfloat val[kPer][4];
        Reduced rd[kPer];
        float vmax = 0.F;
#pragma unroll
        for (int i = 0; i < kPer; ++i)
        {
            const int q = tid + i * kThreads;
            const int v = v0 + q;
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
                val[i][pol] = {0.F, 0.F};
            rd[i] = {0.F, 0.F, 0.F, 0.F};
            int t = 0, c = 0;
            if (q < VB && v < V)
                sel.at(v, t, c);
            if (q < VB && v < V && entry_ok(t, c, m.nr_timesteps, nc))
            {
                const long long r = row0 + t;
                rd[i] = reduce_visibility(a.uvw + 3 * r, a.wavenumbers[c0 + c], off, delta, -1.F);
                const float4 x0 = vis[(r * C + c0 + c) * 2], x1 = vis[(r * C + c0 + c) * 2 + 1];
                val[i][0] = {x0.x, x0.y};
                val[i][1] = {x0.z, x0.w};
                val[i][2] = {x1.x, x1.y};
                val[i][3] = {x1.z, x1.w};
                rotate4(val[i], rd[i].rot);
#pragma unroll
                for (int pol = 0; pol < 4; ++pol)
                    vmax = fmaxf(vmax, fmaxf(fabsf(val[i][pol].re), fabsf(val[i][pol].im)));
            }
        }
        if constexpr (DT == kFP16)
        {
            const int e_new = max(scale_exp, scale_exponent(block_max(vmax, sm.maxbits)));
            if (e_new > scale_exp)
            {
                const float f = ldexpf(1.F, scale_exp - e_new);
#pragma unroll
                for (int t = 0; t < PT; ++t)
                    acc[t] *= f;
                scale_exp = e_new;
            }
            const float inv = ldexpf(1.F, -scale_exp);
#pragma unroll
            for (int i = 0; i < kPer; ++i)
#pragma unroll
                for (int pol = 0; pol < 4; ++pol)
                    val[i][pol] = {val[i][pol].re * inv, val[i][pol].im * inv};
        }
#pragma unroll
        for (int i = 0; i < kPer; ++i)
        {
            const int q = tid + i * kThreads;
            if (q >= VB)
                break;
            const int blk = q >> 4, qq = q & 15;
            write_b_item<DT, SPLIT>(s_bw + blk * 256, qq, val[i]);
            if constexpr (PM)
            {
                float *cf = sm.coef + blk * 64 + qq;
                cf[0] = rd[i].qu;
                cf[16] = rd[i].qv;
                cf[32] = rd[i].dw;
                cf[48] = 0.F;
            }
            else
            {
                float *cf = sm.coef + blk * 64 + (qq >> 2) * 16 + (qq & 3);
                cf[0] = rd[i].qu;
                cf[4] = rd[i].qv;
                cf[8] = rd[i].dw;
            }
        }
        __syncthreads();
        const int nblk = active ? min(kBlocks, (V - v0 + 15) >> 4) : 0;
        for (int b = 0; b < nblk; ++b)
        {
            const u32x4 bf = sm.b[b * 64 + lane];
            f32x4 phs[PT];
            if constexpr (PM)
            {
                const float coef = sm.coef[b * 64 + lane];
#pragma unroll
                for (int t = 0; t < PT; ++t)
                    phs[t] = phase_mfma(coef, coord[t]); // phi(visibility 4*(lane/16)+j, pixel lane%16)
            }
            else
            {
                // phi = qu x' + qv y' + dw n with the x' term formed once per visibility: 2 FMAs per phase.
                const f32x4 *cf = reinterpret_cast<const f32x4 *>(sm.coef + b * 64 + (lane >> 4) * 16);
                const f32x4 du = cf[0], dv = cf[1], dw = cf[2];
                f32x4 ux;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    ux[j] = du[j] * xp;
#pragma unroll
                for (int t = 0; t < PT; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        phs[t][j] = __builtin_fmaf(dv[j], yp[t], __builtin_fmaf(dw[j], nn[t], ux[j]));
            }
#pragma unroll
            for (int t = 0; t < PT; ++t)
            {
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    const float sn = __builtin_amdgcn_sinf(phs[t][j]);
                    const float cs = __builtin_amdgcn_cosf(phs[t][j]);
                    if constexpr (SPLIT)
                        split2<DT>(cs, sn, hi[j], lo[j]);
                    else
                        hi[j] = pack2<DT>(cs, sn);
                }
                acc[t] = mfma(hi[0], hi[1], hi[2], hi[3], bf, acc[t], std::integral_constant<int, DT>());
                if constexpr (SPLIT)
                    acc[t] = mfma(lo[0], lo[1], lo[2], lo[3], bf, acc[t], std::integral_constant<int, DT>());
            }
        }
    }

    // Sum the high and low column halves, gather each pixel's 8 values in LDS, apply A-term and taper.
    __syncthreads();
    const float unscale = DT == kFP16 ? ldexpf(1.F, scale_exp) : 1.F;
#pragma unroll
    for (int t = 0; t < PT; ++t)
    {
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const float v = (acc[t][j] + __shfl_xor(acc[t][j], 8)) * unscale;
            const int col = lane & 15;
            if (col < 8)
                sm.pix[((wave * PT + t) * 16 + (lane >> 4) * 4 + j) * 8 + col] = v;
        }
    }
    __syncthreads();
    float2 *out = reinterpret_cast<float2 *>(a.subgrids_out) + static_cast<size_t>(s) * kCorr * P;
    const float4 *aterms = reinterpret_cast<const float4 *>(a.aterms);
    for (int q = tid; q < kPix; q += kThreads)
    {
        // Slot q = (wave w, tile t, row r) of the accumulator gather above.
        const int w = q / (PT * 16), t = (q >> 4) % PT, r = q & 15;
        const int u = kWaves * pblk + w;
        const int y = (u / gu.ns) * gu.rows + t * gu.rt + r / gu.wd;
        if (u >= gu.units || y >= S)
            continue;
        const int p = y * S + (u % gu.ns) * gu.wd + r % gu.wd;
        const float *v = sm.pix + q * 8;
        cfloat px[4] = {{v[0], v[1]}, {v[2], v[3]}, {v[4], v[5]}, {v[6], v[7]}};
        if (ok)
        {
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
}

// ---------------------------------------------------------------------------------------------------------------
// Degridder item: chunk vblk of 4 waves x VT tiles x 16 visibilities of subgrid s.  The subgrid's pixels stream
// through LDS PB at a time (taper and A-term applied, split into B fragments); the accumulators stay in
// registers across batches, so each visibility is written once.
// ---------------------------------------------------------------------------------------------------------------
// PREP: the pixels come prepared (a.prepared, a.prepared_scale, a.slot_coord: the persistent kernels, whose batch
// prepares them before every pass); otherwise the item applies taper and A-terms as it stages them (the one-shot
// kernel).  A compile-time choice, so the persistent kernel carries no registers for the staging it never runs.
template <int DT, bool SPLIT, int VT, int PB, bool PM, bool PREP>
__device__ __forceinline__ void degridder_item(const KernelArgs &a, int s, int vblk, DegridderShared<VT, PB> &sm)
{
    constexpr int kChunk = kWaves * VT * 16;
    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int S = a.p.S, P = S * S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    if (!subgrid_in_bounds(a.p, m, row0, c0, nc) || nc == 0)
        return; // uniform: nothing of this subgrid is written
    Selection sel;
    const int V = selection_of(a, s, m.nr_timesteps, nc, sel);
    const int v0 = vblk * kChunk;
    if (v0 >= V)
        return; // uniform
    const long long C = a.p.nr_channels;
    const CentreOffsets off = centre_offsets(a.p, m);
    const double delta = static_cast<double>(a.p.image_size) / S;
    const float2 *sub = reinterpret_cast<const float2 *>(a.subgrids) + static_cast<size_t>(s) * kCorr * P;
    uint32_t *s_bw = reinterpret_cast<uint32_t *>(sm.b);

    // The FP64 reduction of each of the chunk's visibilities, once: thread tid takes visibilities tid, tid + 256, ...
    // (the ones it writes in the epilogue, so their output rotations stay in registers) and shares qu, qv, dw
    // through sm.vis, which the epilogue alone writes.  Each lane then reads visibility lane%16 of each of its tiles;
    // for PM only component lane/16 of them (the B operand of the phase MFMA).
    constexpr int kPerThread = (kChunk + kThreads - 1) / kThreads;
    float rot[kPerThread];
#pragma unroll
    for (int i = 0; i < kPerThread; ++i)
    {
        const int q = tid + i * kThreads;
        rot[i] = 0.F;
        if (q >= kChunk)
            break;
        const int v = v0 + q;
        float ru = 0.F, rv = 0.F, rw = 0.F;
        int tt = 0, c = 0;
        if (v < V)
            sel.at(v, tt, c);
        if (v < V && entry_ok(tt, c, m.nr_timesteps, nc))
        {
            const Reduced rd = reduce_visibility(a.uvw + 3 * (row0 + tt), a.wavenumbers[c0 + c], off, delta, 1.F);
            ru = rd.qu;
            rv = rd.qv;
            rw = rd.dw;
            rot[i] = rd.rot;
        }
        sm.vis[3 * q] = ru;
        sm.vis[3 * q + 1] = rv;
        sm.vis[3 * q + 2] = rw;
    }
    __syncthreads();
    float coef[VT], qu[VT], qv[VT], qw[VT];
#pragma unroll
    for (int t = 0; t < VT; ++t)
    {
        const int q = (wave * VT + t) * 16 + (lane & 15);
        qu[t] = sm.vis[3 * q];
        qv[t] = sm.vis[3 * q + 1];
        qw[t] = sm.vis[3 * q + 2];
        const int kk = lane >> 4;
        coef[t] = kk == 0 ? qu[t] : kk == 1 ? qv[t] : kk == 2 ? qw[t] : 0.F;
    }
    f32x4 acc[VT];
#pragma unroll
    for (int t = 0; t < VT; ++t)
        acc[t] = (f32x4){0.F, 0.F, 0.F, 0.F};
    const bool wave_live = v0 + wave * VT * 16 < V; // wave-uniform
    int scale_exp = -126; // FP16: current power-of-two scale of the staged B operand
    if constexpr (DT == kFP16 && PREP)
        scale_exp = a.prepared_scale[s];

    // Pixel slots: rows of Sp = S rounded up to a multiple of 4, so each lane group's 4 slots share a row.
    const int Sp = degrid_row_stride(S), nslots = S * Sp;
    for (int pb = 0; pb < nslots; pb += PB)
    {
        const int np = min(PB, nslots - pb);
        __syncthreads();
        constexpr int kPer = (PB + kThreads - 1) / kThreads;
        if constexpr (PREP)
        {
            // Prepared pixels: copy the split words and the slot coordinates into LDS.
            const uint4 *src = a.prepared + (static_cast<size_t>(s) * nslots + pb) * 2;
#pragma unroll
            for (int i = 0; i < kPer; ++i)
            {
                const int q = tid + i * kThreads;
                if (q >= PB)
                    break;
                uint32_t hi[4] = {0u, 0u, 0u, 0u}, lo[4] = {0u, 0u, 0u, 0u};
                float cx = 0.F, cy = 0.F, cn = 0.F;
                if (q < np)
                {
                    const uint4 w0 = src[2 * q], w1 = src[2 * q + 1];
                    hi[0] = w0.x, lo[0] = w0.y, hi[1] = w0.z, lo[1] = w0.w;
                    hi[2] = w1.x, lo[2] = w1.y, hi[3] = w1.z, lo[3] = w1.w;
                    const float4 c = a.slot_coord[pb + q];
                    cx = c.x;
                    cy = c.y;
                    cn = c.z;
                }
                const int blk = q >> 4, qq = q & 15;
                write_b_words(s_bw + blk * 256, qq, hi, lo);
                if constexpr (PM)
                {
                    float *r = sm.coord + blk * 64 + qq;
                    r[0] = cx;
                    r[16] = cy;
                    r[32] = cn;
                    r[48] = 0.F;
                }
                else
                {
                    float *r = sm.coord + blk * 64 + (qq >> 2) * 16 + (qq & 3);
                    r[0] = cx;
                    r[4] = cy;
                    r[8] = cn;
                }
            }
        }
        else
        {
            cfloat px[kPer][4];
            float cx[kPer], cy[kPer], cn[kPer];
            float vmax = 0.F;
#pragma unroll
            for (int i = 0; i < kPer; ++i)
            {
                const int q = tid + i * kThreads;
#pragma unroll
                for (int pol = 0; pol < 4; ++pol)
                    px[i][pol] = {0.F, 0.F};
                cx[i] = cy[i] = cn[i] = 0.F;
                const int sy = (pb + q) / Sp, sx = pb + q - sy * Sp;
                if (q < np)
                {
                    cx[i] = pixel_offset(sx, S);
                    cy[i] = pixel_offset(sy, S);
                }
                if (q < np && sx < S)
                {
                    degrid_pixel(a, m, sub, sy * S + sx, px[i]);
                    cn[i] = pixel_n_f(pixel_lm_f(sx, S, a.p.image_size), pixel_lm_f(sy, S, a.p.image_size));
#pragma unroll
                    for (int pol = 0; pol < 4; ++pol)
                        vmax = fmaxf(vmax, fmaxf(fabsf(px[i][pol].re), fabsf(px[i][pol].im)));
                }
            }
            if constexpr (DT == kFP16)
            {
                const int e_new = max(scale_exp, scale_exponent(block_max(vmax, sm.maxbits)));
                if (e_new > scale_exp)
                {
                    const float f = ldexpf(1.F, scale_exp - e_new);
#pragma unroll
                    for (int t = 0; t < VT; ++t)
                        acc[t] *= f;
                    scale_exp = e_new;
                }
                const float inv = ldexpf(1.F, -scale_exp);
#pragma unroll
                for (int i = 0; i < kPer; ++i)
#pragma unroll
                    for (int pol = 0; pol < 4; ++pol)
                        px[i][pol] = {px[i][pol].re * inv, px[i][pol].im * inv};
            }
#pragma unroll
            for (int i = 0; i < kPer; ++i)
            {
                const int q = tid + i * kThreads;
                if (q >= PB)
                    break;
                const int blk = q >> 4, qq = q & 15;
                write_b_item<DT, SPLIT>(s_bw + blk * 256, qq, px[i]);
                if constexpr (PM)
                {
                    float *r = sm.coord + blk * 64 + qq;
                    r[0] = cx[i];
                    r[16] = cy[i];
                    r[32] = cn[i];
                    r[48] = 0.F;
                }
                else
                {
                    float *r = sm.coord + blk * 64 + (qq >> 2) * 16 + (qq & 3);
                    r[0] = cx[i];
                    r[4] = cy[i];
                    r[8] = cn[i];
                }
            }
        }
        __syncthreads();
        // A wave whose visibilities all lie past V (the subgrid's last chunk) only stages and waits.
        const int nblk = wave_live ? (np + 15) >> 4 : 0;
        for (int b = 0; b < nblk; ++b)
        {
            const u32x4 bf = sm.b[b * 64 + lane];
            f32x4 phs[VT];
            if constexpr (PM)
            {
                const float cd = sm.coord[b * 64 + lane];
#pragma unroll
                for (int t = 0; t < VT; ++t)
                    phs[t] = phase_mfma(cd, coef[t]); // phi(pixel 4*(lane/16)+j, visibility lane%16)
            }
            else
            {
                // The lane group's 4 pixels share y': its term is formed once per visibility, 2 FMAs per phase.
                const float *g = sm.coord + b * 64 + (lane >> 4) * 16;
                const f32x4 x4 = *reinterpret_cast<const f32x4 *>(g), n4 = *reinterpret_cast<const f32x4 *>(g + 8);
                const float y = g[4];
#pragma unroll
                for (int t = 0; t < VT; ++t)
                {
                    const float vy = qv[t] * y;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        phs[t][j] = __builtin_fmaf(qu[t], x4[j], __builtin_fmaf(qw[t], n4[j], vy));
                }
            }
#pragma unroll
            for (int t = 0; t < VT; ++t)
            {
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                {
                    const float sn = __builtin_amdgcn_sinf(phs[t][j]);
                    const float cs = __builtin_amdgcn_cosf(phs[t][j]);
                    if constexpr (SPLIT)
                        split2<DT>(cs, sn, hi[j], lo[j]);
                    else
                        hi[j] = pack2<DT>(cs, sn);
                }
                acc[t] = mfma(hi[0], hi[1], hi[2], hi[3], bf, acc[t], std::integral_constant<int, DT>());
                if constexpr (SPLIT)
                    acc[t] = mfma(lo[0], lo[1], lo[2], lo[3], bf, acc[t], std::integral_constant<int, DT>());
            }
        }
    }

    // Combine column halves, gather 8 values per visibility in LDS, write 32 B per visibility.
    const float unscale = DT == kFP16 ? ldexpf(1.F, scale_exp) : 1.F;
#pragma unroll
    for (int t = 0; t < VT; ++t)
    {
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const float v = (acc[t][j] + __shfl_xor(acc[t][j], 8)) * unscale;
            const int col = lane & 15;
            if (col < 8)
                sm.vis[((wave * VT + t) * 16 + (lane >> 4) * 4 + j) * 8 + col] = v;
        }
    }
    __syncthreads();
    float4 *vout = reinterpret_cast<float4 *>(a.visibilities_out);
#pragma unroll
    for (int i = 0; i < kPerThread; ++i)
    {
        const int q = tid + i * kThreads, v = v0 + q;
        if (q >= kChunk || v >= V)
            break;
        int tt, c;
        sel.at(v, tt, c);
        if (!entry_ok(tt, c, m.nr_timesteps, nc))
            continue;
        const size_t o = ((row0 + tt) * C + c0 + c) * 2;
        const float *x = sm.vis + q * 8;
        cfloat val[4] = {{x[0], x[1]}, {x[2], x[3]}, {x[4], x[5]}, {x[6], x[7]}};
        rotate4(val, rot[i]);
        vout[o] = make_float4(val[0].re, val[0].im, val[1].re, val[1].im);
        vout[o + 1] = make_float4(val[2].re, val[2].im, val[3].re, val[3].im);
    }
    __syncthreads(); // LDS is reused by the next item of a persistent workgroup
}
} // namespace
} // namespace idgx
