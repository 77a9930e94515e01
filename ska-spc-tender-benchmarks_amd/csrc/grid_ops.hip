// Adder (uv subgrids onto the master grid) and splitter (master grid into uv subgrids) for gfx950.
//
// Grid layout: complex64 [4][G][G] (one plane per correlation), or [nr_layers][4][G][G] for w-stacking, where
// subgrid s belongs to layer metadata[s].z - z_min.  Subgrid s covers grid cells
// [y0, y0 + S) x [x0, x0 + S) with (x0, y0) = metadata[s].coordinate; cells outside the grid are skipped by the
// adder and read as zero by the splitter.
//
// Conflict-free adder.  The grid is cut into tiles of T >= S cells; a subgrid belongs to the tile holding its
// corner and can only touch that tile's 2T x 2T region (the tile and its right/lower neighbours).  Tiles are
// coloured by the parity of their tile coordinates: two different tiles of one colour are at least two tiles
// apart in x or y, so their regions are disjoint.  One launch per colour.  A thread owns the four cells of the region
// that agree modulo T, of which a subgrid covers exactly one when T = S (at most one otherwise): it walks the tile's
// subgrids in plan order, reads its cell of each and adds it to one of four sums, and at the end adds each sum to the
// grid once.  Every cell therefore sees a fixed summation order (deterministic, no atomics).  The tile lists are built
// on the host from the plan (idgx_adder_plan_build).
//
// What bounds them: HBM.  76,865 subgrids of 32^2 (2.52 GB) and a 4096^2 grid: the adder reads each subgrid row whole,
// once, past the caches (nontemporal), 3.7 GB with the grid in 0.76 ms (4.9 TB/s, as a large copy); with a thread per
// cell of the region, three of four idle for each subgrid and lines fetched by several workgroups, it took 1.15 ms, and
// 0.93 ms with cached reads.  The splitter writes 2.52 GB past the caches, which keeps the grid's cells there: 0.63 ms,
// against 0.88 ms with cached stores, a division per cell and neighbouring subgrids on different XCDs.
#include "idgx_device.hpp"
#include "kernels.hpp"

namespace idgx
{
namespace
{
constexpr int kThreads = 256;
constexpr int kAdderUnroll = 8; // subgrids whose loads the adder keeps in flight together (4: 202 us, 16: 202, 8: 189)
constexpr int kAdderPols = 2;   // correlations per workgroup (4: 8 % slower where a tile holds hundreds of subgrids)
constexpr int kLoadOnce = 2;    // cache policy of a buffer load: nontemporal
constexpr int kRun = 64;        // consecutive subgrids that the splitter keeps on one XCD

typedef float f32x4 __attribute__((ext_vector_type(4), aligned(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int floordiv_dev(int a, int b)
{
    return a >= 0 ? a / b : -((-a + b - 1) / b);
}

// Workgroups per tile of the adder: one residue (x mod T, y mod T) and kAdderPols correlations per thread.
__host__ __device__ inline int adder_blocks(int T)
{
    return (T * T + kThreads - 1) / kThreads * (kCorr / kAdderPols);
}

// A thread's residue of one tile.
struct AdderCells
{
    const float2 *subgrids;
    int S, T, p0, rx, ry;
    bool live;
};

// The next U subgrids of a tile's list (n left) onto the thread's cells, their loads in flight together.  Offset -1 is
// past the buffer's end: such a lane reads nothing (and the value is not used).
template <int U>
__device__ __forceinline__ void adder_step(const AdderCells &c, const int4 *list, int n, float2 (&acc)[4][kAdderPols],
                                           bool (&touched)[4])
{
    const int P = c.S * c.S;
    u32x2 val[U][kAdderPols];
    bool on[U], right[U], below[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
    {
        const int4 m = list[min(u, n - 1)];
        const int s = __builtin_amdgcn_readfirstlane(m.x);
        const int ox = __builtin_amdgcn_readfirstlane(m.y), oy = __builtin_amdgcn_readfirstlane(m.z);
        const bool in_tile = u < n && ox >= 0 && ox < c.T && oy >= 0 && oy < c.T; // uniform
        right[u] = c.rx < ox;
        below[u] = c.ry < oy;
        const int dx = c.rx - ox + (right[u] ? c.T : 0), dy = c.ry - oy + (below[u] ? c.T : 0);
        on[u] = c.live && in_tile && dx < c.S && dy < c.S;
        const int off = on[u] ? (dy * c.S + dx) * 8 : -1;
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float2 *>(c.subgrids) + static_cast<size_t>(s) * kCorr * P, 0, kCorr * P * 8, 0x00020000);
#pragma unroll
        for (int p = 0; p < kAdderPols; ++p)
            val[u][p] = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, (c.p0 + p) * P * 8, kLoadOnce);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (on[u] && right[u] == (q & 1) && below[u] == (q >> 1))
            {
                touched[q] = true;
#pragma unroll
                for (int p = 0; p < kAdderPols; ++p)
                {
                    acc[q][p].x += __uint_as_float(val[u][p].x);
                    acc[q][p].y += __uint_as_float(val[u][p].y);
                }
            }
}

__global__ __launch_bounds__(kThreads) void adder_kernel(const idgx_metadata *md, const int32_t *order,
                                                         const int32_t *tile_start, int tile_begin, int ntiles, int S,
                                                         int T, int G, int z_min, int nr_layers,
                                                         const float2 *subgrids, float2 *grid)
{
    __shared__ int4 list[kThreads];
    const int per_tile = adder_blocks(T);
    // Workgroup b -> (tile, residues): workgroups reach the 8 XCDs in turn (b % 8), so XCD x takes tiles x, x + 8,
    // x + 16, ... of the colour (heaviest first), each with all its residues.  The grid is padded to a multiple of 8
    // tiles; the padding exits.
    const int b = static_cast<int>(blockIdx.x), k = b >> 3;
    const int tl = (k / per_tile) * 8 + (b & 7);
    if (tl >= ntiles)
        return; // uniform
    const int tile = tile_begin + tl;
    const int first = tile_start[tile], last = tile_start[tile + 1];
    const idgx_metadata m0 = md[order[first]];
    // All subgrids of a tile share one w-layer (the plan keys tiles by layer); single-layer plans ignore z.
    const int layer = nr_layers > 1 ? m0.z - z_min : 0;
    if (layer < 0 || layer >= nr_layers)
        return; // uniform; the layered plan builder rejects such subgrids
    // The tile's origin, from its index as the plan keys it (clamped to -1 .. G / T + 1: subgrids beyond those tiles
    // meet no cell of the grid).
    const int ntiles_axis = floordiv_dev(G, T) + 3;
    const int bx = (min(max(floordiv_dev(m0.x, T) + 1, 0), ntiles_axis - 1) - 1) * T;
    const int by = (min(max(floordiv_dev(m0.y, T) + 1, 0), ntiles_axis - 1) - 1) * T;
    const int tid = threadIdx.x, sub_b = k % per_tile, p0 = sub_b % (kCorr / kAdderPols) * kAdderPols;
    const int e = sub_b / (kCorr / kAdderPols) * kThreads + tid;
    const int ry = e / T, rx = e - ry * T;
    float2 acc[4][kAdderPols];
    bool touched[4] = {false, false, false, false};
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int p = 0; p < kAdderPols; ++p)
            acc[q][p] = make_float2(0.F, 0.F);
    const AdderCells c = {subgrids, S, T, p0, rx, ry, ry < T};
    for (int i0 = first; i0 < last; i0 += kThreads)
    {
        const int n = min(last - i0, kThreads);
        __syncthreads(); // the previous list is done with
        if (tid < n)
        {
            const int s = order[i0 + tid];
            list[tid] = make_int4(s, md[s].x - bx, md[s].y - by, 0);
        }
        __syncthreads();
        int u0 = 0;
        for (; n - u0 > kAdderUnroll / 2; u0 += kAdderUnroll)
            adder_step<kAdderUnroll>(c, list + u0, n - u0, acc, touched);
        if (n - u0 > kAdderUnroll / 4)
            adder_step<kAdderUnroll / 2>(c, list + u0, n - u0, acc, touched);
        else if (n > u0)
            adder_step<kAdderUnroll / 4>(c, list + u0, n - u0, acc, touched);
    }
    const size_t GG = static_cast<size_t>(G) * G;
    grid += (static_cast<size_t>(layer) * kCorr + p0) * GG;
#pragma unroll
    for (int q = 0; q < 4; ++q)
    {
        const int cx = bx + rx + (q & 1) * T, cy = by + ry + (q >> 1) * T;
        if (!touched[q] || cx < 0 || cx >= G || cy < 0 || cy >= G)
            continue;
        float2 *g = grid + static_cast<size_t>(cy) * G + cx;
        float2 o[kAdderPols];
#pragma unroll
        for (int p = 0; p < kAdderPols; ++p)
            o[p] = g[p * GG];
#pragma unroll
        for (int p = 0; p < kAdderPols; ++p)
            g[p * GG] = make_float2(o[p].x + acc[q][p].x, o[p].y + acc[q][p].y);
    }
}

__global__ __launch_bounds__(kThreads) void splitter_kernel(const idgx_metadata *md, int S, int G, int z_min,
                                                            int nr_layers, const float2 *grid, float2 *subgrids)
{
    // Workgroups reach the 8 XCDs in turn: runs of kRun subgrids, near each other in uv, on one XCD read most of the
    // grid from its L2 (76,865 subgrids of 32^2: 740 us in launch order, 742 in runs of 4, 662 of 16, 639 of 64 and of
    // 256; XCD-contiguous 719, but 10 % slower than launch order for 13,747 of 64^2).
    const int whole = static_cast<int>(gridDim.x) / (8 * kRun) * (8 * kRun), b = static_cast<int>(blockIdx.x);
    const long long s = b < whole ? (b / (8 * kRun) * 8 + (b & 7)) * kRun + (b >> 3) % kRun : b;
    const int x0 = md[s].x, y0 = md[s].y;
    const int P = S * S, H = S / 2;
    const size_t GG = static_cast<size_t>(G) * G;
    const int layer = nr_layers > 1 ? md[s].z - z_min : 0;
    const bool on = layer >= 0 && layer < nr_layers; // uniform: a subgrid of no layer reads zeros
    grid += static_cast<size_t>(on ? layer : 0) * kCorr * GG;
    float2 *sub = subgrids + static_cast<size_t>(s) * kCorr * P;
    if (on && x0 >= 0 && y0 >= 0 && x0 <= G - S && y0 <= G - S) // uniform: every cell is in the grid
    {
        const float2 *g = grid + static_cast<size_t>(y0) * G + x0;
#pragma unroll 2
        for (int i = threadIdx.x; i < P / 2; i += kThreads)
        {
            const int y = i / H, x = 2 * (i - y * H);
            f32x4 v[kCorr]; // two cells (S is even), 8-byte aligned in the grid
#pragma unroll
            for (int p = 0; p < kCorr; ++p)
                v[p] = *reinterpret_cast<const f32x4 *>(g + p * GG + static_cast<size_t>(y) * G + x);
#pragma unroll
            for (int p = 0; p < kCorr; ++p)
                __builtin_nontemporal_store(v[p], reinterpret_cast<f32x4 *>(sub + p * P + 2 * i));
        }
        return;
    }
    for (int q = threadIdx.x; q < kCorr * P; q += kThreads)
    {
        const int pol = q / P, rem = q - pol * P;
        const int y = rem / S, x = rem - y * S;
        const int gy = y0 + y, gx = x0 + x;
        float2 v = make_float2(0.F, 0.F);
        if (on && gy >= 0 && gy < G && gx >= 0 && gx < G)
            v = grid[pol * GG + static_cast<size_t>(gy) * G + gx];
        sub[q] = v;
    }
}
} // namespace

hipError_t launch_adder(const idgx_metadata *md, const int32_t *order, const int32_t *tile_start,
                        const int32_t *color_begin, int S, int T, int G, int z_min, int nr_layers,
                        const void *subgrids, void *grid, hipStream_t st)
{
    if (T < S || T <= 0 || T > 32768)
        return hipErrorInvalidValue;
    const long long per_tile = adder_blocks(T);
    for (int c = 0; c < 4; ++c)
    {
        const long long n = color_begin[c + 1] - color_begin[c];
        if (n <= 0)
            continue;
        const long long padded = (n + 7) / 8 * 8; // whole groups of 8 tiles, one per XCD
        if (padded * per_tile > 0x7fffffffLL)
            return hipErrorInvalidConfiguration;
        adder_kernel<<<static_cast<unsigned>(padded * per_tile), kThreads, 0, st>>>(
            md, order, tile_start, color_begin[c], static_cast<int>(n), S, T, G, z_min, nr_layers,
            static_cast<const float2 *>(subgrids), static_cast<float2 *>(grid));
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

hipError_t launch_splitter(const idgx_metadata *md, long long nr_subgrids, int S, int G, int z_min, int nr_layers,
                           const void *grid, void *subgrids, hipStream_t st)
{
    if (nr_subgrids > 0x7fffffffLL)
        return hipErrorInvalidConfiguration;
    splitter_kernel<<<static_cast<unsigned>(nr_subgrids), kThreads, 0, st>>>(
        md, S, G, z_min, nr_layers, static_cast<const float2 *>(grid), static_cast<float2 *>(subgrids));
    return hipGetLastError();
}
} // namespace idgx
