// Separable mixed-precision gridder and degridder for gfx950: phasors per (row, visibility) and per (column,
// visibility) instead of per (pixel, visibility), contracted on v_mfma_f32_32x32x16_{f16,bf16}.
//
// Phase.  With half-integer pixel coordinates xh = x + 1/2 - S/2 (l = xh delta, delta = image_size / S) the phase of a
// visibility at a pixel is, in revolutions,
//     qu xh + qv yh + dw n(l, m),    qu = du delta, qv = dv delta  (du, dv, dw relative to the subgrid's centre).
// The w-term is taken apart in two steps.  Per subgrid, w0 = the middle of the range of w over its visibilities:
// e^{2 pi i w0 n} is one exact rotation per pixel, applied to the gridder's result and to the degridder's pixels.
// For the rest, d = dw - w0, n splits into an additive part and a remainder that is a product but for 2e-6 of its corner
// value at a field of 0.1 rad (2e-5 at 0.17):
//     n(l, m) = a(l) + a(m) + c g(l) g(m),   a(l) = n(l, l0) - n(l0, l0) / 2,  l0 = l_max / sqrt(2),
// where c = n's remainder at the corner and g, |g| <= 1, its profile along the edge (n = (l^2 + m^2) / 2 + (l^2 + m^2)^2
// / 8 + ..., so the remainder is (l^2 - l0^2)(m^2 - l0^2) / 4 to first order: 3.5e-7 at a field of 0.1 rad).  So
//     e^{2 pi i phase} = X(x) Y(y) (1 + i eps g(x) g(y)),   eps = 2 pi c d,
//     X = e^{2 pi i (qu xh + d a(x))},  Y = e^{2 pi i (qv yh + d a(y))}
// up to eps^2 / 2.  Subgrids with |eps| <= kEpsNone run without the product term (FP16 gridders of few visibilities always
// with it), up to a limit (kEpsGrid, kEpsDegrid) with it; the others (fields wider than 0.1 rad, or w far from constant over
// a subgrid) are left to the per-pair kernels: a launch of theirs behind this one, or where a one-shot plan lets expect
// none, their items inside it.
//
// Contraction, on v_mfma_f32_32x32x16.  Gridder: pixel[y][x, corr] = sum_v Y[y][v] (V[v][corr] X[v][x]), one real GEMM
// with the rows (y, re/im), the columns (x, corr) and k = (v, re/im): the rows hold Y's two real embeddings, the B operand
// the product V X, which a lane forms in FP32 for one (x, corr) and four visibilities and splits into hi/lo halves: per
// (pixel, visibility) pair 1/S of that work.  Three MFMAs per tile (hi hi, lo hi, hi lo; BF16 also lo lo) and one for the
// product term, whose factor i eps g(y) goes into a second set of rows and g(x) into the columns, as single halves (eps
// scales their rounding).  A wave owns all rows of NT column tiles (8 columns x 4 correlations each) and its own
// chunks of visibilities; no operand passes through LDS, and the waves only meet when their sums are added.
// Degridder: H[x, corr][v] = sum_y P[y][x, corr] Y[y][v], the pixels split once per workgroup and read from LDS in the A
// operand's order, then vis[v][corr] = sum_x X[x][v] H[x, corr][v] on the VALU: 16 FMAs per (column, visibility).
//
// What bounds it: the matrix cores, at the power limit.  A pair costs 128 flop there (4 products of 32).  On 128 stations,
// 64 channels, 76,865 subgrids of 32^2 (136.3 G pairs) a pass is 17.4 PFLOP, 14.7 ms at the rate a large FP16 product
// reaches on the card (1186 TFLOP/s, clocks at 1.7 to 2.0 GHz).  Measured: gridder 41.2 -> 16.1 ms, degridder 41.3 ->
// 15.2 ms (cards differ by 3 %); the per-pair kernels, 8.25 VALU instructions per pair (two of them transcendental), were
// VALU-issue bound at 97 %; these issue 2.2 and 1.7.  The interleaving of MFMA and VALU instructions (scheduling groups,
// wave priorities) and the tile (16 x 16 x 32: more cycles at a higher clock) moved the time by less than 3 %.
#include "mixed_device.hpp"

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <type_traits>

namespace idgx
{
namespace
{
// Below this the term is worth 0.27 of it at most in the root mean square, 2.7e-8 (at 3e-7 it was 8e-8, seen in subgrids
// of 8 visibilities: 1.44e-7 from 64 bits against 1.60e-7; no case got slower by more than its runs differ).
constexpr float kEpsNone = 1e-7F;
// Largest eps, per pixel of the subgrid's side.  The term's operands are single halves, in the gridder an error of 4e-4 eps
// for FP16 (2.8e-4 for kFewVisibilities), beside eps^2 / 2; the error of the per-pair kernels grows with the side, the
// degridder's most (it rounds 24 bits of phase per pixel).  Distance from 64 bits over theirs at these limits, 48
// subgrids with random uv: gridder 0.85 to 1.00, degridder 0.75 to 1.00; gridder on the subgrids with the largest eps of
// 76,865 of 32^2 (1.8e-4) 0.70, of 20,780 of 48^2 (3.9e-4) 0.77, of 13,747 of 64^2 (2e-4) 0.83.  At 1e-3 for every size
// it was 2.7 (16^2) to 1.1 (64^2).  BF16, whose 16 bits of each factor are 3.2e-6 off for every size, has one limit, where
// the term's 8 bits add 1 % to that (at 1e-3 20 %).
constexpr double kEpsGrid = 1e-5, kEpsDegrid = 2.5e-5;
constexpr double kEpsMost = 1e-3, kEpsBF16 = 4e-4;
constexpr float kTermScale = 1024.F; // moves the product term's factors into FP16's normal range
// Plans take these kernels where a half spread of w of S / image_size wavelengths (the subgrid's own extent in u and v)
// is worth at most so many times S kEpsGrid: fields up to 0.166 and 0.131 rad.  Observations spread w by 0.1 to 0.4 of that.
// Times over those of the per-pair kernels, gridder and degridder (2016 baselines, 32^2 and 64^2 subgrids; 780, 16^2), with
// the share of subgrids left to them: 32^2 at 0.13 rad 0.47 (5 %) and 0.37, at 0.16 0.68 (59 %) and 0.42; 64^2 at 0.16 0.48
// (19 %) and 0.39 (4 %); 24^2 at 0.16 0.81 (70 %) and 0.53 (5 %); 16^2 at 0.13 0.74 (48 %) and 0.40, but in batches at
// 0.14 0.89 (68 %) and 1.07 (3 %: the queue's walk over all items outweighs the small subgrids).
constexpr double kFieldMost = 10.0, kFieldMostSmall = 5.0;
constexpr int kFieldSmall = 24; // the latter below this subgrid size
// FP16 gridding of a subgrid of so few visibilities forms its phasors by their series and always takes the product term:
// over few visibilities the errors of v_sin and v_cos, here of two phasors a pair instead of one, do not average out.
// Distance from 64 bits over that of the per-pair kernels, worst of S = 16 .. 48, with v_sin and v_cos / by the series:
// 8 visibilities 1.08 / 0.94, 16 1.09 / 0.94, 32 1.03 / 0.92, 48 0.99.
constexpr int kFewVisibilities = 72;
constexpr int kFewSubgrids = 256;  // the CUs: a workgroup per subgrid would leave some of them idle
constexpr int kChunk = 64;        // visibilities a wave stages at a time, one per lane
constexpr int kValStride = 80;    // staged values of one correlation (64, padded: fewer LDS bank conflicts)

// One wave's staged visibilities.
struct alignas(16) GridStage
{
    float qu[kChunk], qv[kChunk], de[kChunk];
    float2 val[4][kValStride];
};
struct alignas(16) DegridStage
{
    float qu[kChunk], qv[kChunk], de[kChunk], scale[kChunk];
    long long out[kChunk];
};

// LDS of a workgroup: a column's (a, g) at its index, and one of the phases' working sets.
template <int COLS, int SPLITS, int ROWS, int WAVES> struct alignas(16) GridLds
{
    float2 tab[kSeparableMax];
    float slots[WAVES][5];
    union
    {
        GridStage stage[WAVES];
        float2 sum[SPLITS][ROWS * COLS * 4]; // the splits' partial sums of a pass of rows
        GridderShared<kDefaultPT, kDefaultVB> direct;
    };
};
template <int WAVES> struct alignas(16) DegridLds
{
    float2 tab[kSeparableMax];
    float slots[WAVES][5];
    DegridStage stage[WAVES];
    uint4 pixels[1]; // as many as the subgrid needs
};

// Bytes of LDS a degridder workgroup takes: the pixels in the A operand's order (hi and lo words of 4 correlations), and
// never less than the per-pair item's staging.
template <int WAVES> size_t degrid_lds_bytes(int S, int rows)
{
    const size_t cols = static_cast<size_t>((S + 7) / 8) * 8;
    return std::max(offsetof(DegridLds<WAVES>, pixels) + rows * cols * 4 * 2 * sizeof(uint32_t),
                    sizeof(DegridderShared<kDefaultVT, kDefaultPB>));
}

// q / cols for q < 4096 and cols <= 64 (q (cols - 1) < 2^20): two instructions instead of a division.
struct SmallDivisor
{
    unsigned magic;
    __device__ __forceinline__ explicit SmallDivisor(int cols)
        : magic(((1U << 20) + static_cast<unsigned>(cols) - 1U) / static_cast<unsigned>(cols))
    {
    }
    __device__ __forceinline__ int quotient(int q) const
    {
        return static_cast<int>(__umul24(static_cast<unsigned>(q), magic) >> 20);
    }
};

// Reduced phase coordinates of one visibility, signed by sgn: slopes per pixel in [-1/2, 1/2], w relative to the
// subgrid's middle, and the parity of the whole turns taken off the slopes (half-integer coordinates turn each of
// them into half a turn: a factor -1).
struct Slopes
{
    float qu, qv, de;
    bool odd;
};

__device__ __forceinline__ Slopes reduce_slopes(float u, float v, float w, float k, const CentreOffsets &o, double wc,
                                                double delta, float sgn)
{
    const double kk = static_cast<double>(k) * kInv2Pi;
    const double qu = __builtin_fma(kk, static_cast<double>(u), -o.u) * delta;
    const double qv = __builtin_fma(kk, static_cast<double>(v), -o.v) * delta;
    const double ru = __builtin_rint(qu), rv = __builtin_rint(qv);
    const double turns = 0.5 * (ru + rv);
    Slopes s;
    s.qu = sgn * static_cast<float>(qu - ru);
    s.qv = sgn * static_cast<float>(qv - rv);
    s.de = sgn * static_cast<float>(__builtin_fma(kk, static_cast<double>(w), -wc));
    s.odd = turns != __builtin_rint(turns);
    return s;
}

// e^{2 pi i (f + q / 4)} for |f| <= 1/8 of a turn, to about an FP32 rounding: the Taylor series, cut off below 2e-9.
__device__ __forceinline__ cfloat phasor_series(float f, int q)
{
    const float f2 = f * f;
    // In turns: powers of 2 pi over the factorials, and 2 pi itself in two parts.
    float ps = __builtin_fmaf(f2, 42.0586939F, -76.7058598F), pc = __builtin_fmaf(f2, -26.4262568F, 60.2446414F);
    ps = __builtin_fmaf(ps, f2, 81.6052493F);
    pc = __builtin_fmaf(pc, f2, -85.4568172F);
    ps = __builtin_fmaf(ps, f2, -41.3417022F);
    pc = __builtin_fmaf(pc, f2, 64.9393940F);
    ps = __builtin_fmaf(ps, f2, -1.74845553e-7F);
    pc = __builtin_fmaf(pc, f2, -19.7392088F);
    const float sn = __builtin_fmaf(f, 6.28318548F, f * ps), cs = __builtin_fmaf(pc, f2, 1.F);
    const float re = q & 1 ? sn : cs, im = q & 1 ? cs : sn;
    // Quarter turns 0, 1, 2, 3: (c, s), (-s, c), (-c, -s), (s, -c).
    return {(q + 1) & 2 ? -re : re, q & 2 ? -im : im};
}

// e^{2 pi i ph}: v_sin and v_cos, or (SERIES) the series, about three times their instructions.
template <bool SERIES> __device__ __forceinline__ void phasor(float ph, float &sn, float &cs)
{
    if constexpr (SERIES)
    {
        const float quarters = __builtin_rintf(4.F * ph);
        const cfloat r = phasor_series(__builtin_fmaf(-0.25F, quarters, ph), static_cast<int>(quarters));
        cs = r.re;
        sn = r.im;
    }
    else
    {
        sn = __builtin_amdgcn_sinf(ph);
        cs = __builtin_amdgcn_cosf(ph);
    }
}

// e^{2 pi i w n} of pixel (x, y): every visibility of the subgrid shares its error, so the quarter turns come off in FP64
// and what is left takes the series.  It costs 1.5 % of the gridder on 24^2 subgrids of 129 visibilities.
__device__ __forceinline__ cfloat pixel_rotation(int x, int y, int S, double delta, double w)
{
    const double n = n_series((x + 0.5 - 0.5 * S) * delta, (y + 0.5 - 0.5 * S) * delta);
    const double t = __builtin_amdgcn_fract(w * n);
    const float quarters = __builtin_rintf(4.F * static_cast<float>(t)); // 0 to 4
    return phasor_series(static_cast<float>(__builtin_fma(-0.25, static_cast<double>(quarters), t)),
                         static_cast<int>(quarters));
}

// (vr + i vi) (cs + i sn) with the phasor of lane J of the quad: four FMA-class instructions that read the phasor
// through DPP (the compiler would copy it first).  The leading s_nop covers the two wait states between a VALU write
// and a DPP read of the same register.
template <int J> __device__ __forceinline__ cfloat quad_product(float cs, float sn, float vr, float vi)
{
    cfloat r;
    if constexpr (J == 0)
        asm("s_nop 1\n\t"
            "v_mul_f32_dpp %0, %2, %4 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %1, %2, %5 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %0, -%3, %5 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %1, %3, %4 quad_perm:[0,0,0,0] row_mask:0xf bank_mask:0xf"
            : "=&v"(r.re), "=&v"(r.im)
            : "v"(cs), "v"(sn), "v"(vr), "v"(vi));
    else if constexpr (J == 1)
        asm("s_nop 1\n\t"
            "v_mul_f32_dpp %0, %2, %4 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %1, %2, %5 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %0, -%3, %5 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %1, %3, %4 quad_perm:[1,1,1,1] row_mask:0xf bank_mask:0xf"
            : "=&v"(r.re), "=&v"(r.im)
            : "v"(cs), "v"(sn), "v"(vr), "v"(vi));
    else if constexpr (J == 2)
        asm("s_nop 1\n\t"
            "v_mul_f32_dpp %0, %2, %4 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %1, %2, %5 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %0, -%3, %5 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %1, %3, %4 quad_perm:[2,2,2,2] row_mask:0xf bank_mask:0xf"
            : "=&v"(r.re), "=&v"(r.im)
            : "v"(cs), "v"(sn), "v"(vr), "v"(vi));
    else
        asm("s_nop 1\n\t"
            "v_mul_f32_dpp %0, %2, %4 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf\n\t"
            "v_mul_f32_dpp %1, %2, %5 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %0, -%3, %5 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf\n\t"
            "v_fmac_f32_dpp %1, %3, %4 quad_perm:[3,3,3,3] row_mask:0xf bank_mask:0xf"
            : "=&v"(r.re), "=&v"(r.im)
            : "v"(cs), "v"(sn), "v"(vr), "v"(vi));
    return r;
}

// Element-wise products of packed halves: a * b for FP16 (v_pk_mul_f16).
__device__ __forceinline__ uint32_t mul_f16x2(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, a) * __builtin_bit_cast(f16x2, b));
}

// The two rows of a phasor c + i s (packed pairs along k): re = (c, -s), im = (s, c), hi and lo halves.
template <int DT>
__device__ __forceinline__ void split_rows(float c, float s, uint32_t &re_hi, uint32_t &re_lo, uint32_t &im_hi,
                                           uint32_t &im_lo)
{
    re_hi = pack2<DT>(c, -s);
    im_hi = pack2<DT>(s, c);
    float rc, rs;
    if constexpr (DT == kFP16)
    {
        rs = sub_f16_lo(s, im_hi);
        rc = sub_f16_hi(c, im_hi);
    }
    else
    {
        float h0, h1;
        unpack2<DT>(im_hi, h0, h1);
        rs = s - h0;
        rc = c - h1;
    }
    re_lo = pack2<DT>(rc, -rs);
    im_lo = pack2<DT>(rs, rc);
}

// The rows of i f (c + i s) in single halves: re = -f (s, c), im = f (c, -s).  FP16: from the split rows, with three
// roundings to halves; BF16, and FP16 with ONCE: from the phasor, with one.
template <int DT, bool ONCE = false>
__device__ __forceinline__ void term_rows(float c, float s, float f, uint32_t re_hi, uint32_t im_hi, uint32_t &re,
                                          uint32_t &im)
{
    if constexpr (DT == kFP16 && !ONCE)
    {
        const f16x2 ff = __builtin_bit_cast(f16x2, pack2<DT>(f, f));
        re = __builtin_bit_cast(uint32_t, -ff * __builtin_bit_cast(f16x2, im_hi));
        im = __builtin_bit_cast(uint32_t, ff * __builtin_bit_cast(f16x2, re_hi));
    }
    else
    {
        re = pack2<DT>(-f * s, -f * c);
        im = pack2<DT>(f * c, -f * s);
    }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

// D[32][32] += A[32][16] B[16][32]: lane l holds A[l % 32][8 (l / 32) + 0..7], B[8 (l / 32) + 0..7][l % 32] and
// D[8 (i / 4) + 4 (l / 32) + i % 4][l % 32] in element i.  Twice the tile of the 16 x 16 form per instruction: with two
// waves per SIMD and 6 to 8 VALU instructions beside each, 15 to 19 ns per instruction against 2 x (11 to 15) ns.
template <int DT> __device__ __forceinline__ f32x16 mfma32(const uint32_t *a, const uint32_t *b, f32x16 c)
{
    const u32x4 av = {a[0], a[1], a[2], a[3]}, bv = {b[0], b[1], b[2], b[3]};
    if constexpr (DT == kFP16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, av), __builtin_bit_cast(f16x8, bv), c, 0,
                                                      0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, bv), c,
                                                       0, 0, 0);
}

// Swaps a's odd 16-lane rows with b's even ones.
__device__ __forceinline__ void swap_rows16(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// The order of a wave's own LDS writes and reads (no other wave touches its staging).
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- gridder ----------------------------------------------------------------------------------------------------

// Rows of the gridder's GEMM in tiles of 32: pairs of tiles hold re and im of 32 subgrid rows; with an odd number of
// 16-row blocks the last tile holds both of 16.
template <int YT> struct RowCoords
{
    static constexpr int kPairs = YT / 2, kBlocks = kPairs + YT % 2;
    float yh[kBlocks], ya[kBlocks], yg[kBlocks]; // this lane's row of each block: coordinate, a, term factor
};

// 8 staged visibilities onto the wave's pixels: all rows, NT tiles of 8 columns x 4 correlations.
template <int DT, int YT, int NT, bool TERM, bool SERIES>
__device__ __forceinline__ void grid_step(const GridStage &st, const float2 *tab, int base, int x0, float half_s,
                                          const RowCoords<YT> &rc, f32x16 (&acc)[NT][YT])
{
    const int lane = threadIdx.x & 63, corr = lane & 3;
    const int v = base + 4 * (lane >> 5);
    uint32_t ah[YT][4], al[YT][4], at[YT][4];
    if constexpr (YT >= 2)
    {
        const f32x4 qv = *reinterpret_cast<const f32x4 *>(&st.qv[v]);
        const f32x4 de = *reinterpret_cast<const f32x4 *>(&st.de[v]);
#pragma unroll
        for (int t = 0; t < YT / 2; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const float ph = __builtin_fmaf(qv[j], rc.yh[t], de[j] * rc.ya[t]);
                float sn, cs;
                phasor<SERIES>(ph, sn, cs);
                split_rows<DT>(cs, sn, ah[2 * t][j], al[2 * t][j], ah[2 * t + 1][j], al[2 * t + 1][j]);
                if constexpr (TERM)
                    term_rows<DT, SERIES>(cs, sn, de[j] * rc.yg[t], ah[2 * t][j], ah[2 * t + 1][j], at[2 * t][j],
                                  at[2 * t + 1][j]);
            }
    }
    if constexpr (YT % 2 == 1)
    {
        // Lanes l and l + 16 share a row: each forms the phasors of two of the four visibilities, then they swap, so
        // that the first holds all four real rows and the second all four imaginary ones.
        const int w = v + 2 * ((lane >> 4) & 1);
        const float2 qv = *reinterpret_cast<const float2 *>(&st.qv[w]);
        const float2 de = *reinterpret_cast<const float2 *>(&st.de[w]);
        constexpr int t = YT - 1, k = YT / 2;
#pragma unroll
        for (int j = 0; j < 2; ++j)
        {
            const float d = j ? de.y : de.x;
            const float ph = __builtin_fmaf(j ? qv.y : qv.x, rc.yh[k], d * rc.ya[k]);
            float sn, cs;
            phasor<SERIES>(ph, sn, cs);
            split_rows<DT>(cs, sn, ah[t][j], al[t][j], ah[t][j + 2], al[t][j + 2]);
            if constexpr (TERM)
            {
                term_rows<DT, SERIES>(cs, sn, d * rc.yg[k], ah[t][j], ah[t][j + 2], at[t][j], at[t][j + 2]);
                swap_rows16(at[t][j], at[t][j + 2]);
            }
            swap_rows16(ah[t][j], ah[t][j + 2]);
            swap_rows16(al[t][j], al[t][j + 2]);
        }
    }
    // This lane's column phasor is that of visibility v + corr; the quad shares its four.
    const float qux = st.qu[v + corr], dex = st.de[v + corr];
    const f32x4 v01 = *reinterpret_cast<const f32x4 *>(&st.val[corr][v]);
    const f32x4 v23 = *reinterpret_cast<const f32x4 *>(&st.val[corr][v + 2]);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
    {
        const int x = x0 + 8 * nt + ((lane & 31) >> 2);
        const float2 tb = tab[x];
        const float ph = __builtin_fmaf(qux, static_cast<float>(x) - half_s, dex * tb.x);
        float sn, cs;
        phasor<SERIES>(ph, sn, cs);
        const cfloat vx[4] = {quad_product<0>(cs, sn, v01[0], v01[1]), quad_product<1>(cs, sn, v01[2], v01[3]),
                              quad_product<2>(cs, sn, v23[0], v23[1]), quad_product<3>(cs, sn, v23[2], v23[3])};
        uint32_t bh[4], bl[4], bt[4];
        const uint32_t gg = pack2<DT>(tb.y, tb.y);
#pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            split2<DT>(vx[j].re, vx[j].im, bh[j], bl[j]);
            if constexpr (TERM)
                bt[j] = DT == kFP16 && !SERIES ? mul_f16x2(bh[j], gg) : pack2<DT>(vx[j].re * tb.y, vx[j].im * tb.y);
        }
#pragma unroll
        for (int t = 0; t < YT; ++t)
            acc[nt][t] = mfma32<DT>(ah[t], bh, acc[nt][t]);
#pragma unroll
        for (int t = 0; t < YT; ++t)
            acc[nt][t] = mfma32<DT>(al[t], bh, acc[nt][t]);
#pragma unroll
        for (int t = 0; t < YT; ++t)
            acc[nt][t] = mfma32<DT>(ah[t], bl, acc[nt][t]);
        if constexpr (DT == kBF16) // its lo x lo is 2^-18 of the product: above the other errors
        {
#pragma unroll
            for (int t = 0; t < YT; ++t)
                acc[nt][t] = mfma32<DT>(al[t], bl, acc[nt][t]);
        }
        if constexpr (TERM)
        {
#pragma unroll
            for (int t = 0; t < YT; ++t)
                acc[nt][t] = mfma32<DT>(at[t], bt, acc[nt][t]);
        }
    }
}

struct RawVisibility
{
    float4 x0, x1;
    float u, v, w, k;
    bool valid;
};

__device__ __forceinline__ RawVisibility load_visibility(const KernelArgs &a, const Selection &sel, int v, int V,
                                                         int T, int nc, long long row0, int c0)
{
    RawVisibility r;
    r.x0 = r.x1 = make_float4(0.F, 0.F, 0.F, 0.F);
    r.u = r.v = r.w = r.k = 0.F;
    r.valid = false;
    if (v < V)
    {
        int t, c;
        sel.at(v, t, c);
        if (entry_ok(t, c, T, nc))
        {
            const long long row = row0 + t;
            const float4 *vis = reinterpret_cast<const float4 *>(a.visibilities) + (row * a.p.nr_channels + c0 + c) * 2;
            r.x0 = vis[0];
            r.x1 = vis[1];
            r.u = a.uvw[3 * row];
            r.v = a.uvw[3 * row + 1];
            r.w = a.uvw[3 * row + 2];
            r.k = a.wavenumbers[c0 + c];
            r.valid = true;
        }
    }
    return r;
}

// One wave's chunks of V visibilities: chunk `first` (whose visibilities are in raw), then every step-th.  n
// visibilities per chunk, a multiple of 8, at most kChunk.
template <int DT, int YT, int NT, bool TERM, bool SERIES>
__device__ __forceinline__ int grid_sum(const KernelArgs &a, const SeparableArgs &sp, const Selection &sel, int V, int T,
                                        int nc, long long row0, int c0, const CentreOffsets &off, double wc,
                                        int first, int step, int n, RawVisibility raw, int x0, GridStage &st,
                                        const float2 *tab, f32x16 (&acc)[NT][YT])
{
    const int lane = threadIdx.x & 63;
    const double delta = static_cast<double>(a.p.image_size) / a.p.S;
    const float half_s = 0.5F * static_cast<float>(a.p.S) - 0.5F;
    RowCoords<YT> rc;
#pragma unroll
    for (int t = 0; t < RowCoords<YT>::kBlocks; ++t)
    {
        const int y = 32 * t + (t < YT / 2 ? lane & 31 : lane & 15);
        rc.yh[t] = static_cast<float>(y) - half_s;
        rc.ya[t] = tab[y].x;
        rc.yg[t] = tab[y].y * (sp.tables.eps * kTermScale * kTermScale); // tab holds g / kTermScale
    }
    int scale_exp = -126; // FP16: power-of-two scale of the staged visibilities
    for (int v0 = first * n; v0 < V; v0 += step * n)
    {
        cfloat val[4] = {{raw.x0.x, raw.x0.y}, {raw.x0.z, raw.x0.w}, {raw.x1.x, raw.x1.y}, {raw.x1.z, raw.x1.w}};
        Slopes s = {0.F, 0.F, 0.F, false};
        if (raw.valid)
            s = reduce_slopes(raw.u, raw.v, raw.w, raw.k, off, wc, delta, -1.F);
        float f = s.odd ? -1.F : 1.F;
        if constexpr (DT == kFP16)
        {
            float m = 0.F;
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
                m = fmaxf(m, fmaxf(fabsf(val[pol].re), fabsf(val[pol].im)));
#pragma unroll
            for (int d = 1; d < 64; d <<= 1)
                m = fmaxf(m, __shfl_xor(m, d));
            const int e_new = max(scale_exp, __builtin_amdgcn_readfirstlane(scale_exponent(m)));
            if (e_new > scale_exp)
            {
                const float r = ldexpf(1.F, scale_exp - e_new);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int t = 0; t < YT; ++t)
                        acc[nt][t] *= r;
                scale_exp = e_new;
            }
            f *= ldexpf(1.F, -scale_exp);
        }
        wave_lds_fence();
        st.qu[lane] = s.qu;
        st.qv[lane] = s.qv;
        st.de[lane] = s.de;
#pragma unroll
        for (int pol = 0; pol < 4; ++pol)
            st.val[pol][lane] = make_float2(val[pol].re * f, val[pol].im * f);
        wave_lds_fence();
        // The next chunk's visibilities, in flight during the sums.
        raw = load_visibility(a, sel, lane < n ? v0 + step * n + lane : V, V, T, nc, row0, c0);
        const int nsteps = min(n, V - v0 + 7) >> 3;
        for (int k = 0; k < nsteps; ++k)
            grid_step<DT, YT, NT, TERM, SERIES>(st, tab, 8 * k, x0, half_s, rc, acc);
    }
    return scale_exp;
}

// Columns (x, a(x) and g(x)) of the subgrid in LDS; g is scaled for the product term's columns.
__device__ __forceinline__ void fill_table(float2 *tab, const SeparableArgs &sp, int S)
{
    const int x = threadIdx.x;
    if (x < kSeparableMax)
    {
        const int j = x >= S / 2 ? min(x - S / 2, kSeparableMax / 2 - 1) : S / 2 - 1 - x;
        tab[x] = make_float2(sp.tables.a[j], sp.tables.g[j] * (1.F / kTermScale));
    }
}

// Waves per SIMD that the gridder's registers are held to.  YT = 2, NT = 3 (S = 24) spills 42 of them in its prologue
// and epilogue at three, and is 1 to 4 % faster than at two.
template <int YT, int NT> constexpr int grid_waves()
{
    return YT * NT <= 2 ? 4 : YT * NT <= 3 || (YT == 2 && NT == 3) ? 3 : 2;
}

// Which subgrids of a launch a kernel grids, by their visibilities (kFewVisibilities).  Kernels with wide column tiles
// have one form for each: a kernel with both would spill in its main loop (24^2 subgrids of 129 visibilities: 7 % slower).
enum GridSubgrids : int
{
    kEvery,
    kMany,
    kFew
};

// Workgroup (part, subgrid) grids columns [part, part + 1) x 8 NT NX of a subgrid: its waves take NX column ranges and
// WAVES / NX interleaved chunks of visibilities; the partial sums meet in LDS 16 or 32 rows at a time, in a fixed order.
template <int DT, int YT, int NT, int NX, int WAVES, int WHICH>
__global__ __launch_bounds__(64 * WAVES, (grid_waves<YT, NT>())) void grid_separable(KernelArgs a, SeparableArgs sp)
{
    constexpr int kCols = NX * NT * 8, kSplits = WAVES / NX, kCount = 64 * WAVES;
    constexpr int kPass = NT == 1 ? 32 : 16; // rows of the subgrid whose sums meet at a time
    __shared__ GridLds<kCols, kSplits, kPass, WAVES> sm;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int part = blockIdx.x / sp.count, b = blockIdx.x - part * sp.count;
    const int s = sp.order ? sp.order[b] : b;
    const int S = a.p.S, P = S * S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    const bool ok = subgrid_in_bounds(a.p, m, row0, c0, nc);
    Selection sel;
    const int T = m.nr_timesteps, V = ok ? selection_of(a, s, T, nc, sel) : 0;
    // Without an order, which the host has split at the count, both launches go over all subgrids.
    if (WHICH != kEvery && !sp.order && (V <= kFewVisibilities) != (WHICH == kFew))
        return; // uniform
    // Chunks short enough for every split to have one.
    const int split = wave / NX, n = min(kChunk, ((V + kSplits - 1) / kSplits + 7) & ~7);
    RawVisibility raw = load_visibility(a, sel, lane < n ? split * n + lane : V, V, T, nc, row0, c0);
    fill_table(sm.tab, sp, S);
    WRange wr = {0.0, 0.F};
    float none = 0.F;
    if (V > 0) // (without visibilities nothing reads the table)
        wr = w_range<WAVES, false>(a, row0, T, c0, nc, sm.slots, none);
    const float eps = wr.half * sp.tables.eps;
    const bool fits = separable_fits(sp.limits, wr.half);
    if (sp.leftover && tid == 0 && part == 0)
    {
        sp.leftover[s] = fits ? 0 : 1;
        if (!fits)
            *sp.leftover_any = 1;
    }
    if (!fits)
    {
        if (!sp.leftover && !sp.leave && tid < kThreads) // waves that have ended are not waited for at barriers
        {
            // The subgrid's per-pair items over its workgroups.
            const int items = (grid_units(S, kDefaultPT).units + kWaves - 1) / kWaves;
            for (int i = part; i < items; i += gridDim.x / sp.count)
            {
                gridder_item<DT, true, kDefaultPT, kDefaultVB, false>(a, s, i, sm.direct);
                __syncthreads();
            }
        }
        return; // uniform
    }
    const CentreOffsets off = centre_offsets(a.p, m);
    const double delta = static_cast<double>(a.p.image_size) / S;
    f32x16 acc[NT][YT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int t = 0; t < YT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                acc[nt][t][i] = 0.F;
    const int xb = part * kCols, x0 = xb + (wave % NX) * NT * 8;
    const auto sum = [&](auto term, auto series) {
        return grid_sum<DT, YT, NT, term.value, series.value>(a, sp, sel, V, T, nc, row0, c0, off, wr.centre, split,
                                                              kSplits, n, raw, x0, sm.stage[wave], sm.tab, acc);
    };
    int scale_exp;
    if constexpr (DT == kFP16 && WHICH == kFew)
        scale_exp = sum(std::true_type{}, std::true_type{});
    else if (DT == kFP16 && WHICH == kEvery && V <= kFewVisibilities)
        scale_exp = sum(std::true_type{}, std::bool_constant<DT == kFP16 && WHICH == kEvery>{});
    else if (eps <= kEpsNone)
        scale_exp = sum(std::false_type{}, std::false_type{});
    else
        scale_exp = sum(std::true_type{}, std::false_type{});
    const float unscale = DT == kFP16 ? ldexpf(1.F, scale_exp) : 1.F;
    float2 *out = reinterpret_cast<float2 *>(a.subgrids_out) + static_cast<size_t>(s) * kCorr * P;
    const float4 *aterms = reinterpret_cast<const float4 *>(a.aterms);
    const size_t abase = ok ? static_cast<size_t>(m.aterm_index) * a.p.nr_stations : 0;
    const double w0 = V > 0 ? off.w - wr.centre : 0.0; // minus the gridder's sign
    const int h = lane >> 5, xi = (lane & 31) >> 2, corr = lane & 3;
    const int cols = min(kCols, S - xb);
    const SmallDivisor by_cols(cols);
#pragma unroll
    for (int t0 = 0; t0 < YT; t0 += kPass / 16) // kPass rows of the subgrid at a time
    {
        const int y0 = 16 * t0;
        if (y0 >= S)
            break; // uniform
        // This thread's pixels' A-terms, in flight while the sums meet in LDS.
        constexpr int kPer = (kPass * kCols + kCount - 1) / kCount;
        cfloat a1[kPer][4], a2[kPer][4];
        float taper[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i)
        {
            const int q = tid + i * kCount, row = by_cols.quotient(q), x = xb + q - row * cols, y = y0 + row;
            if (row < kPass && y < S && ok)
            {
                const int p = y * S + x;
                load_jones(aterms, (abase + m.station1) * P + p, a1[i]);
                load_jones(aterms, (abase + m.station2) * P + p, a2[i]);
                taper[i] = a.spheroidal[p];
            }
        }
        lds_barrier(); // the staging, or the previous rows, are done with
#pragma unroll
        for (int t = t0; t < t0 + kPass / 16 && t < YT; ++t) // 16 rows each
        {
            constexpr int kPairs = YT / 2;
            const bool paired = t < 2 * kPairs;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
            {
                const int x = x0 - xb + 8 * nt + xi;
                if (x >= cols)
                    continue;
#pragma unroll
                for (int i = 0; i < 8; ++i)
                {
                    // Row 8 (i / 4) + 4 h + i % 4 of the block.
                    const float re = paired ? acc[nt][t / 2 * 2][t % 2 * 8 + i] : acc[nt][YT - 1][i];
                    const float im = paired ? acc[nt][t / 2 * 2 + (YT > 1)][t % 2 * 8 + i] : acc[nt][YT - 1][8 + i];
                    sm.sum[split][((16 * t - y0 + i / 4 * 8 + 4 * h + i % 4) * cols + x) * 4 + corr] =
                        make_float2(re * unscale, im * unscale);
                }
            }
        }
        lds_barrier();
#pragma unroll
        for (int i = 0; i < kPer; ++i)
        {
            const int q = tid + i * kCount, row = by_cols.quotient(q), x = xb + q - row * cols, y = y0 + row;
            if (row >= kPass || y >= S)
                continue;
            const int p = y * S + x;
            cfloat px[4] = {{0.F, 0.F}, {0.F, 0.F}, {0.F, 0.F}, {0.F, 0.F}};
            if (ok)
            {
                const cfloat r = pixel_rotation(x, y, S, delta, w0);
#pragma unroll
                for (int pol = 0; pol < 4; ++pol)
                {
                    float2 v = sm.sum[0][q * 4 + pol];
#pragma unroll
                    for (int k = 1; k < kSplits; ++k)
                    {
                        const float2 u = sm.sum[k][q * 4 + pol];
                        v = make_float2(v.x + u.x, v.y + u.y);
                    }
                    px[pol] = cmul({v.x, v.y}, r);
                }
                apply_a1h_p_a2(px, a1[i], a2[i]);
#pragma unroll
                for (int pol = 0; pol < 4; ++pol)
                    px[pol] = {px[pol].re * taper[i], px[pol].im * taper[i]};
            }
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
                out[pol * P + p] = make_float2(px[pol].re, px[pol].im);
        }
    }
}

// ---- degridder --------------------------------------------------------------------------------------------------

// Row blocks of the degridder: its k runs over 8 rows per MFMA, at most 4 of those (32 rows) with their phasors in
// registers at once.  KS of them per pass and YB passes cover the subgrid's rows.
//
// 32 staged visibilities from the subgrid's pixels: element p of `sum` is re / im (p % 2) of correlation p / 2 of
// visibility base + lane % 32, over this lane half's columns (x % 2 = lane / 32).
template <int DT, int KS, int YB, bool TERM>
__device__ __forceinline__ void degrid_tile(const DegridStage &st, const float2 *tab, const uint4 *pixels, int mts,
                                            int base, float half_s, float eps, float (&sum)[8])
{
    const int lane = threadIdx.x & 63, h = lane >> 5, v = base + (lane & 31);
    const float qu = st.qu[v], qv = st.qv[v], de = st.de[v];
    const float term = de * eps;
#pragma unroll
    for (int i = 0; i < 8; ++i)
        sum[i] = 0.F;
#pragma unroll
    for (int yb = 0; yb < YB; ++yb)
    {
        uint32_t reh[KS][4], rel[KS][4], imh[KS][4], iml[KS][4], ret[KS][4], imt[KS][4];
#pragma unroll
        for (int k = 0; k < KS; ++k)
        {
#pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const int y = 8 * (yb * KS + k) + 4 * h + j;
                const float2 tb = tab[y];
                const float p = __builtin_fmaf(qv, static_cast<float>(y) - half_s, de * tb.x);
                const float sn = __builtin_amdgcn_sinf(p), cs = __builtin_amdgcn_cosf(p);
                split_rows<DT>(cs, sn, reh[k][j], rel[k][j], imh[k][j], iml[k][j]);
                if constexpr (TERM)
                    term_rows<DT>(cs, sn, term * tb.y, reh[k][j], imh[k][j], ret[k][j], imt[k][j]);
            }
        }
        for (int mt = 0; mt < mts; ++mt)
        {
            f32x16 hr, hi;
#pragma unroll
            for (int i = 0; i < 16; ++i)
                hr[i] = hi[i] = 0.F;
            const float gx = tab[8 * mt + ((lane & 31) >> 2)].y;
            const uint32_t gg = pack2<DT>(gx, gx);
#pragma unroll
            for (int k = 0; k < KS; ++k)
            {
                const uint4 *px = pixels + (((yb * KS + k) * 2 + h) * mts + mt) * 64 + (lane & 31);
                const uint4 wh = px[0], wl = px[32];
                const uint32_t ph[4] = {wh.x, wh.y, wh.z, wh.w}, pl[4] = {wl.x, wl.y, wl.z, wl.w};
                hr = mfma32<DT>(ph, reh[k], hr);
                hi = mfma32<DT>(ph, imh[k], hi);
                hr = mfma32<DT>(pl, reh[k], hr);
                hi = mfma32<DT>(pl, imh[k], hi);
                hr = mfma32<DT>(ph, rel[k], hr);
                hi = mfma32<DT>(ph, iml[k], hi);
                if constexpr (DT == kBF16)
                {
                    hr = mfma32<DT>(pl, rel[k], hr);
                    hi = mfma32<DT>(pl, iml[k], hi);
                }
                if constexpr (TERM)
                {
                    uint32_t pt[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                    {
                        if constexpr (DT == kFP16)
                        {
                            pt[j] = mul_f16x2(ph[j], gg);
                        }
                        else
                        {
                            float re, im;
                            unpack2<DT>(ph[j], re, im);
                            pt[j] = pack2<DT>(re * gx, im * gx);
                        }
                    }
                    hr = mfma32<DT>(pt, ret[k], hr);
                    hi = mfma32<DT>(pt, imt[k], hi);
                }
            }
            // Element 4 c + pol is column 8 mt + 2 c + h, correlation pol.
#pragma unroll
            for (int c = 0; c < 4; ++c)
            {
                const int x = 8 * mt + 2 * c + h;
                const float p = __builtin_fmaf(qu, static_cast<float>(x) - half_s, de * tab[x].x);
                const float sn = __builtin_amdgcn_sinf(p), cs = __builtin_amdgcn_cosf(p);
#pragma unroll
                for (int pol = 0; pol < 4; ++pol)
                {
                    const float re = hr[4 * c + pol], im = hi[4 * c + pol];
                    sum[2 * pol] = __builtin_fmaf(cs, re, sum[2 * pol]);
                    sum[2 * pol] = __builtin_fmaf(-sn, im, sum[2 * pol]);
                    sum[2 * pol + 1] = __builtin_fmaf(cs, im, sum[2 * pol + 1]);
                    sum[2 * pol + 1] = __builtin_fmaf(sn, re, sum[2 * pol + 1]);
                }
            }
        }
    }
}

struct RawCoords
{
    float u, v, w, k;
    long long out; // -1: no visibility
};

__device__ __forceinline__ RawCoords load_coords(const KernelArgs &a, const Selection &sel, int v, int v_end, int T,
                                                 int nc, long long row0, int c0)
{
    RawCoords r = {0.F, 0.F, 0.F, 0.F, -1};
    if (v < v_end)
    {
        int t, c;
        sel.at(v, t, c);
        if (entry_ok(t, c, T, nc))
        {
            const long long row = row0 + t;
            r.u = a.uvw[3 * row];
            r.v = a.uvw[3 * row + 1];
            r.w = a.uvw[3 * row + 2];
            r.k = a.wavenumbers[c0 + c];
            r.out = (row * a.p.nr_channels + c0 + c) * 2;
        }
    }
    return r;
}

// Visibilities [v_begin, v_end) of one subgrid, in chunks interleaved over the waves.
template <int DT, int KS, int YB, bool TERM>
__device__ __forceinline__ void degrid_range(const KernelArgs &a, const SeparableArgs &sp, const Selection &sel,
                                             int v_begin, int v_end, int T, int nc, long long row0, int c0,
                                             const CentreOffsets &off, double wc, float unscale, const uint4 *pixels,
                                             int mts, DegridStage &st, const float2 *tab)
{
    const int wave = threadIdx.x >> 6, waves = blockDim.x >> 6, lane = threadIdx.x & 63;
    const double delta = static_cast<double>(a.p.image_size) / a.p.S;
    const float half_s = 0.5F * static_cast<float>(a.p.S) - 0.5F;
    float4 *vout = reinterpret_cast<float4 *>(a.visibilities_out);
    // Chunks of one or two tiles: one where that gives every wave work.
    const int n = v_end - v_begin <= waves * 32 ? 32 : kChunk;
    RawCoords raw = load_coords(a, sel, lane < n ? v_begin + wave * n + lane : v_end, v_end, T, nc, row0, c0);
    for (int v0 = v_begin + wave * n; v0 < v_end; v0 += waves * n)
    {
        Slopes s = {0.F, 0.F, 0.F, false};
        if (raw.out >= 0)
            s = reduce_slopes(raw.u, raw.v, raw.w, raw.k, off, wc, delta, 1.F);
        wave_lds_fence();
        st.qu[lane] = s.qu;
        st.qv[lane] = s.qv;
        st.de[lane] = s.de;
        st.scale[lane] = s.odd ? -unscale : unscale;
        st.out[lane] = raw.out;
        wave_lds_fence();
        // The next chunk's coordinates, in flight during the tiles.
        raw = load_coords(a, sel, lane < n ? v0 + waves * n + lane : v_end, v_end, T, nc, row0, c0);
        const int ntiles = min(n, v_end - v0 + 31) >> 5;
        for (int k = 0; k < ntiles; ++k)
        {
            float sum[8];
            degrid_tile<DT, KS, YB, TERM>(st, tab, pixels, mts, 32 * k, half_s,
                                          sp.tables.eps * kTermScale * kTermScale, sum);
            // Both lane halves' columns: the first half keeps correlations 0 and 1, the second 2 and 3.
            float x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum[i]), __float_as_uint(sum[i + 4]),
                                                                false, false);
                x[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
            }
            const int q = 32 * k + (lane & 31);
            const long long at = st.out[q];
            const float f = st.scale[q];
            if (at >= 0)
                vout[at + (lane >> 5)] = make_float4(x[0] * f, x[1] * f, x[2] * f, x[3] * f);
        }
    }
}

// Workgroup (chunk, subgrid): degrids visibilities [chunk * per, (chunk + 1) * per) of a subgrid (per a multiple of
// 256).  The subgrid's pixels (taper, A-terms and the rotation to the middle of its w range applied, FP16: scaled by a
// power of two) are split once into LDS in the A operand's order; the waves take visibilities and never meet again.
// WAVES: 4 (two workgroups per CU), or 8 where the pixels take more than half of LDS.
template <int DT, int KS, int YB, int WAVES>
__global__ __launch_bounds__(64 * WAVES, KS <= 3 && YB == 1 ? 3 : 2) void degrid_separable(KernelArgs a, SeparableArgs sp)
{
    constexpr int kCount = 64 * WAVES;
    extern __shared__ __align__(16) unsigned char lds[];
    auto &sm = *reinterpret_cast<DegridLds<WAVES> *>(lds);
    const int tid = threadIdx.x, wave = tid >> 6;
    const int chunk = blockIdx.x / a.p.nr_subgrids, b = blockIdx.x - chunk * a.p.nr_subgrids;
    const int s = sp.order ? sp.order[b] : b;
    const int S = a.p.S, P = S * S;
    const idgx_metadata m = a.metadata[s];
    int c0, nc;
    channel_window(a, s, c0, nc);
    const long long row0 = first_row(a.metadata, m);
    if (!subgrid_in_bounds(a.p, m, row0, c0, nc) || nc == 0)
    {
        if (sp.leftover && tid == 0)
            sp.leftover[s] = 0;
        return; // uniform: nothing of this subgrid is written
    }
    Selection sel;
    const int T = m.nr_timesteps, V = selection_of(a, s, T, nc, sel);
    const long long v_first = static_cast<long long>(chunk) * sp.per;
    if (v_first >= V)
    {
        if (sp.leftover && tid == 0 && chunk == 0)
            sp.leftover[s] = 0;
        return; // uniform
    }
    const int v_begin = static_cast<int>(v_first);
    const int v_end = static_cast<int>(v_first + sp.per < V ? v_first + sp.per : V);
    // The table, then the pixels q, q + kCount, ... of the padded KS YB 8 x mts 8 (zero past the subgrid) with taper and
    // A-terms applied.  FP16: their largest value, for the scale, meets with the range of w, so their loads do not wait
    // for it (21,768 subgrids of 24^2 with 129 visibilities: 531 -> 478 us, and one barrier instead of six; 45 of 32^2
    // 22.3 -> 20.4).  BF16 needs no scale and is 4 % faster with the range first.
    fill_table(sm.tab, sp, S);
    WRange wr;
    if constexpr (DT == kBF16)
    {
        float none = 0.F;
        wr = w_range<WAVES, false>(a, row0, T, c0, nc, sm.slots, none);
    }
    constexpr int kRows = 8 * KS * YB, kPer = (kRows * kRows + kCount - 1) / kCount;
    const int mts = (S + 7) / 8, cols = 8 * mts;
    const SmallDivisor by_cols(cols);
    const float2 *sub = reinterpret_cast<const float2 *>(a.subgrids) + static_cast<size_t>(s) * kCorr * P;
    cfloat px[kPer][4];
    float vmax = 0.F;
#pragma unroll
    for (int i = 0; i < kPer; ++i)
    {
        const int q = tid + i * kCount, y = by_cols.quotient(q), x = q - y * cols;
#pragma unroll
        for (int pol = 0; pol < 4; ++pol)
            px[i][pol] = {0.F, 0.F};
        if (y < S && x < S)
        {
            degrid_pixel(a, m, sub, y * S + x, px[i]);
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
                vmax = fmaxf(vmax, fmaxf(fabsf(px[i][pol].re), fabsf(px[i][pol].im)));
        }
    }
    if constexpr (DT == kFP16)
        wr = w_range<WAVES, true>(a, row0, T, c0, nc, sm.slots, vmax);
    const float eps = wr.half * sp.tables.eps;
    const bool fits = separable_fits(sp.limits, wr.half);
    if (sp.leftover && tid == 0 && chunk == 0)
    {
        sp.leftover[s] = fits ? 0 : 1;
        if (!fits)
            *sp.leftover_any = 1;
    }
    if (!fits)
    {
        if (sp.leftover || sp.leave)
            return;
        __syncthreads(); // the item's staging overlies the table and the slots, which other waves may still read
        if (tid >= kThreads) // waves that have ended are not waited for at barriers
            return;
        constexpr int per = kWaves * kDefaultVT * 16;
        auto &direct = *reinterpret_cast<DegridderShared<kDefaultVT, kDefaultPB> *>(lds);
        for (int v = v_begin; v < v_end; v += per)
            degridder_item<DT, true, kDefaultVT, kDefaultPB, false, false>(a, s, v / per, direct);
        return; // uniform
    }
    const CentreOffsets off = centre_offsets(a.p, m);
    const double delta = static_cast<double>(a.p.image_size) / S;
    const double w0 = wr.centre - off.w;
    uint32_t *words = reinterpret_cast<uint32_t *>(sm.pixels);
    float unscale = 1.F, inv = 1.F;
    if constexpr (DT == kFP16)
    {
        const int e = scale_exponent(fminf(vmax * 1.4142136F, 3.4028235e38F)); // room for the rotation
        unscale = ldexpf(1.F, e);
        inv = ldexpf(1.F, -e);
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i)
    {
        const int q = tid + i * kCount, y = by_cols.quotient(q), x = q - y * cols;
        if (y >= kRows)
            continue;
        if (y < S && x < S)
        {
            const cfloat r = pixel_rotation(x, y, S, delta, w0);
#pragma unroll
            for (int pol = 0; pol < 4; ++pol)
                px[i][pol] = cmul(px[i][pol], r);
        }
        // Word y % 4 of lane (y / 4 % 2, x % 8, correlation) of tile (y / 8, x / 8); the low halves 32 lanes on.
        uint32_t *w = words + ((((y >> 3) * 2 + ((y >> 2) & 1)) * mts + (x >> 3)) * 64 + (x & 7) * 4) * 4 + (y & 3);
#pragma unroll
        for (int pol = 0; pol < 4; ++pol)
        {
            uint32_t hi, lo;
            split2<DT>(px[i][pol].re * inv, px[i][pol].im * inv, hi, lo);
            w[pol * 4] = hi;
            w[128 + pol * 4] = lo;
        }
    }
    __syncthreads();
    DegridStage &st = sm.stage[wave];
    if (eps <= kEpsNone)
        degrid_range<DT, KS, YB, false>(a, sp, sel, v_begin, v_end, T, nc, row0, c0, off, wr.centre, unscale, sm.pixels,
                                        mts, st, sm.tab);
    else
        degrid_range<DT, KS, YB, true>(a, sp, sel, v_begin, v_end, T, nc, row0, c0, off, wr.centre, unscale, sm.pixels,
                                       mts, st, sm.tab);
}

// ---- launchers --------------------------------------------------------------------------------------------------

template <int DT, int YT, int NT, int NX, int WAVES, int WHICH>
hipError_t launch_grid(const KernelArgs &a, const SeparableArgs &sp, hipStream_t st)
{
    const long long parts = (a.p.S + 8 * NT * NX - 1) / (8 * NT * NX), blocks = parts * sp.count;
    if (blocks > 0x7fffffffLL)
        return hipErrorInvalidConfiguration;
    if (blocks > 0)
        grid_separable<DT, YT, NT, NX, WAVES, WHICH><<<static_cast<unsigned>(blocks), 64 * WAVES, 0, st>>>(a, sp);
    return hipGetLastError();
}

// Subgrids of many visibilities, then those of few (the last `few` of an order; without one, any may be).
template <int DT, int YT, int NT, int NX>
hipError_t launch_grid_wide(const KernelArgs &a, SeparableArgs sp, const GridCounts &n, hipStream_t st)
{
    if constexpr (DT != kFP16)
    {
        return launch_grid<DT, YT, NT, NX, kWaves, kEvery>(a, sp, st);
    }
    else
    {
        hipError_t e = hipSuccess;
        sp.count = sp.order ? a.p.nr_subgrids - n.few : a.p.nr_subgrids;
        if (n.most_vis > kFewVisibilities)
            e = launch_grid<DT, YT, NT, NX, kWaves, kMany>(a, sp, st);
        if (e != hipSuccess)
            return e;
        if (sp.order)
        {
            sp.order += sp.count;
            sp.count = n.few;
        }
        return launch_grid<DT, YT, NT, NX, kWaves, kFew>(a, sp, st);
    }
}

// A gridder kernel's row tiles and column tiles per wave, column ranges and waves; `wide`: one form per kind of subgrid.
template <int YT, int NT, int NX, int WAVES = kWaves, bool WIDE = (WAVES == kWaves && NT > 1)> struct GridShape
{
    static constexpr int yt = YT, nt = NT, nx = NX, waves = WAVES;
    static constexpr bool wide = WIDE;
};

// f(the shape) for n subgrids of size S.  One wave holds all columns up to S = 32 (128 accumulators); larger subgrids
// spread them over two or four waves.  A plan that would leave CUs without work takes a workgroup per 8 columns, which
// forms the row phasors once per 8 columns; where even those leave CUs idle, one of 8 waves (45 subgrids of 32^2 with
// 2048 visibilities: 30.4 -> 25.8 us; of 16^2: 24.2 -> 19.5), which would cost larger plans up to a quarter (231 subgrids
// of 32^2 with 256: 16.9 -> 20.9) and subgrids above 32^2 a tenth.
template <typename F> auto grid_shape(int S, int n, const F &f)
{
    const bool few = n <= kFewSubgrids;
    const bool fewer = static_cast<long long>(n) * ((S + 7) / 8) <= kFewSubgrids;
    if (S <= 16)
        return fewer ? f(GridShape<1, 1, 1, 8>{}) : few ? f(GridShape<1, 1, 1>{}) : f(GridShape<1, 2, 1>{});
    if (S <= 32 && fewer)
        return f(GridShape<2, 1, 1, 8>{});
    if (S <= 32 && few)
        return f(GridShape<2, 1, 1>{});
    if (S <= 24)
        return f(GridShape<2, 3, 1>{});
    if (S <= 32)
        return f(GridShape<2, 4, 1>{});
    if (S <= 48)
        return few ? f(GridShape<3, 1, 1>{}) : f(GridShape<3, 3, 2>{});
    return few ? f(GridShape<4, 1, 1>{}) : f(GridShape<4, 2, 4>{});
}

template <int DT>
hipError_t grid_size(const KernelArgs &a, const SeparableArgs &sp, const GridCounts &n, hipStream_t st)
{
    return grid_shape(a.p.S, a.p.nr_subgrids, [&](auto k) {
        using K = decltype(k);
        if constexpr (K::wide)
            return launch_grid_wide<DT, K::yt, K::nt, K::nx>(a, sp, n, st);
        else
            return launch_grid<DT, K::yt, K::nt, K::nx, K::waves, kEvery>(a, sp, st);
    });
}

template <int DT, int KS, int YB, int WAVES>
hipError_t launch_degrid(const KernelArgs &a, const SeparableArgs &sp, long long blocks, hipStream_t st)
{
    const size_t lds = degrid_lds_bytes<WAVES>(a.p.S, 8 * KS * YB);
    if (lds > 64 * 1024)
    {
        const void *fn = reinterpret_cast<const void *>(&degrid_separable<DT, KS, YB, WAVES>);
        const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess)
            return e;
    }
    degrid_separable<DT, KS, YB, WAVES><<<static_cast<unsigned>(blocks), 64 * WAVES, lds, st>>>(a, sp);
    return hipGetLastError();
}

// A degridder kernel's 8-row steps held at once, passes and waves.
template <int KS, int YB, int WAVES> struct DegridShape
{
    static constexpr int ks = KS, yb = YB, waves = WAVES;
};

template <typename F> auto degrid_shape(int S, const F &f)
{
    if (S <= 16)
        return f(DegridShape<2, 1, 4>{});
    if (S <= 24)
        return f(DegridShape<3, 1, 4>{});
    if (S <= 32)
        return f(DegridShape<4, 1, 4>{});
    if (S <= 48)
        return f(DegridShape<3, 2, 4>{});
    return f(DegridShape<4, 2, 8>{});
}

template <int DT> hipError_t degrid_size(const KernelArgs &a, const SeparableArgs &sp, long long blocks, hipStream_t st)
{
    return degrid_shape(a.p.S, [&](auto k) {
        using K = decltype(k);
        return launch_degrid<DT, K::ks, K::yb, K::waves>(a, sp, blocks, st);
    });
}

double host_n(double l, double m)
{
    const double r2 = l * l + m * m;
    return r2 / (1.0 + std::sqrt(1.0 - r2));
}
} // namespace

bool separable_tables(const PlanDev &p, int precision, SeparableTables &t)
{
    const int S = p.S;
    const double image = p.image_size;
    if ((precision != IDGX_MIXED_FP16X3 && precision != IDGX_MIXED_BF16X3) || S > kSeparableMax || !(image <= 0.2))
        return false;
    const int half = S / 2;
    const double delta = image / S, l_max = (half - 0.5) * delta, l0 = l_max * std::sqrt(0.5);
    const double a0 = 0.5 * host_n(l0, l0);
    const auto add = [&](double l) { return host_n(l, l0) - a0; };
    const double a_edge = add(l_max), c = host_n(l_max, l_max) - 2.0 * a_edge;
    t = SeparableTables{};
    double a_max = 0.0;
    for (int j = 0; j < half; ++j)
    {
        const double l = (j + 0.5) * delta, al = add(l);
        t.a[j] = static_cast<float>(al);
        t.g[j] = c > 0.0 ? static_cast<float>((host_n(l, l_max) - al - a_edge) / c) : 0.F;
        a_max = std::max(a_max, std::fabs(al));
    }
    t.a_max = static_cast<float>(a_max);
    t.eps = static_cast<float>(2.0 * M_PI * c);
    const bool fp16 = precision == IDGX_MIXED_FP16X3;
    t.eps_grid = static_cast<float>(fp16 ? std::min(S * kEpsGrid, kEpsMost) : kEpsBF16);
    t.eps_degrid = static_cast<float>(fp16 ? std::min(S * kEpsDegrid, kEpsMost) : kEpsBF16);
    return t.eps * (S / image) <= (S < kFieldSmall ? kFieldMostSmall : kFieldMost) * (S * kEpsGrid);
}

// A whole subgrid per workgroup (its pixels are prepared once) unless that leaves CUs without work: then as many
// chunks as make 4 workgroups per CU.
long long separable_chunk(long long max_vis, int n)
{
    constexpr long long kWorkgroups = 1024, kStep = kWaves * kChunk;
    const long long most = std::max(1LL, (max_vis + kStep - 1) / kStep);
    const long long chunks = std::min(most, std::max(1LL, kWorkgroups / std::max(1, n)));
    return (most + chunks - 1) / chunks * kStep;
}

SeparableLimits separable_limits(const SeparableTables &t, bool gridder)
{
    return {t.eps, gridder ? t.eps_grid : t.eps_degrid, t.a_max};
}

// Where a half spread of S / image_size wavelengths lies beyond the limit.  Below that the call has one launch, and a
// subgrid that is left all the same runs its items there, several times slower where it has the chip to itself.
bool separable_may_leave(const PlanDev &p, const SeparableLimits &l)
{
    return l.eps * p.S / p.image_size > l.eps_most;
}

long long separable_few_visibilities()
{
    return kFewVisibilities;
}

hipError_t launch_grid_separable(const KernelArgs &a, const SeparableArgs &args, int precision, const GridCounts &n,
                                 hipStream_t st)
{
    SeparableArgs sp = args;
    sp.count = a.p.nr_subgrids;
    return precision == IDGX_MIXED_FP16X3 ? grid_size<kFP16>(a, sp, n, st) : grid_size<kBF16>(a, sp, n, st);
}

hipError_t launch_degrid_separable(const KernelArgs &a, const SeparableArgs &sp, int precision, long long max_vis,
                                   hipStream_t st)
{
    const long long blocks = (max_vis + sp.per - 1) / sp.per * a.p.nr_subgrids;
    if (blocks <= 0)
        return hipSuccess;
    if (blocks > 0x7fffffffLL)
        return hipErrorInvalidConfiguration;
    return precision == IDGX_MIXED_FP16X3 ? degrid_size<kFP16>(a, sp, blocks, st)
                                          : degrid_size<kBF16>(a, sp, blocks, st);
}

int separable_kernel_shape(const PlanDev &p, int precision, bool gridder, long long most_vis, int shape[6])
{
    SeparableTables t;
    if (!separable_tables(p, precision, t))
        return 0;
    shape[0] = precision == IDGX_MIXED_FP16X3 ? kFP16 : kBF16;
    if (!gridder)
        return degrid_shape(p.S, [&](auto k) {
            using K = decltype(k);
            shape[1] = K::ks, shape[2] = K::yb, shape[3] = K::waves;
            return 4;
        });
    return grid_shape(p.S, p.nr_subgrids, [&](auto k) {
        using K = decltype(k);
        shape[1] = K::yt, shape[2] = K::nt, shape[3] = K::nx, shape[4] = K::waves;
        shape[5] = !K::wide || shape[0] != kFP16 ? kEvery : most_vis > kFewVisibilities ? kMany : kFew;
        return 6;
    });
}
} // namespace idgx
