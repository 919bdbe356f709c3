// sphe_kernels.hip -- CDNA4 (gfx950) kernels of the SPH-Erosion step.
//
// One step (all scenes of a context at once), reference Erosion/fluid_system.h
// FluidSystemSPH::Run (:104-183) + advance (:306-353):
//   scan      counts -> cell starts (one to three kernels; tiles no particle
//             counted into are not read)
//   scatter   each particle to its cell segment (arrival order); resets
//             its cell's count for the next step
//   reorder   rank inside the cell by (x slab, particle id) -> canonical
//             (cell, slab, id) order; gathers the state into sorted SoA
//             buffers and writes the cell's slab offsets
//   density   poly6 density + pressure terms over the stencil rows clipped
//             to the smoothing sphere (fluid_system.h:109-124; cells are
//             h (1 + 2^-8) along x and half that along y and z, 25 rows),
//             and the neighbour lists for the force pass
//   force     pressure, viscosity, colour normal/Laplacian (:129-178),
//             symplectic Euler + box response (:318-350, :355-407),
//             heightfield collision and erosion exchange (library-defined),
//             and the cell count of the new position for the next step
//   heights   terrain heights from the fixed-point volumes
// The neighbour predicate is the reference's FP32 one, glm::length(r) <= h,
// evaluated exactly as d2 = (dx*dx + dy*dy) + dz*dz <= T(h) with T(h) the
// largest float whose square root is <= h.  Build with -ffp-contract=off.

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>

#include "sphe_device.h"
#include "sphe_launch.h"

namespace {

template <typename T> struct V4s;
template <> struct V4s<float> { typedef float4 t; };
template <> struct V4s<double> { typedef double4 t; };
template <typename T> using V4 = typename V4s<T>::t;
template <typename T> struct V2s;
template <> struct V2s<float> { typedef float2 t; };
template <> struct V2s<double> { typedef double2 t; };
template <typename T> using V2 = typename V2s<T>::t;

__device__ __forceinline__ float d_floor(float x) { return __builtin_floorf(x); }
__device__ __forceinline__ double d_floor(double x) { return __builtin_floor(x); }
__device__ __forceinline__ float d_sqrt(float x) { return __builtin_sqrtf(x); }
__device__ __forceinline__ double d_sqrt(double x) { return __builtin_sqrt(x); }
__device__ __forceinline__ float d_fabs(float x) { return __builtin_fabsf(x); }
__device__ __forceinline__ double d_fabs(double x) { return __builtin_fabs(x); }
__device__ __forceinline__ float d_rint(float x) { return __builtin_rintf(x); }
__device__ __forceinline__ double d_rint(double x) { return __builtin_rint(x); }
__device__ __forceinline__ bool d_finite(float x) { return __builtin_isfinite(x); }
__device__ __forceinline__ bool d_finite(double x) { return __builtin_isfinite(x); }

// Blocks are dispatched round-robin over the 8 XCDs (block b on XCD b % 8).
// Chunked remap: XCD x takes runs of `chunk` consecutive tiles (run c of
// XCD x is tiles [(8c + x) chunk, (8c + x + 1) chunk)), so neighbouring
// cells share that XCD's L2 while the runs of the 8 XCDs stay interleaved
// over the domain (balanced when the work per particle varies).  chunk <= 1
// is the plain order; blocks past the last complete set of 8 runs keep
// their order.  Bijective for any count.
__device__ __forceinline__ int xcd_block(int bid, int nblk, int chunk)
{
    if (chunk <= 1) return bid;
    const int span = 8 * chunk;
    if (bid >= nblk / span * span) return bid;
    const int x = bid & 7, i = bid >> 3;
    return ((i / chunk) * 8 + x) * chunk + i % chunk;
}

// Index of this wave in block b of a one-dimensional grid of whole waves.
__device__ __forceinline__ uint32_t wave_index(int b)
{
    return (uint32_t)b * (blockDim.x / SPHE_WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x / SPHE_WAVE);
}

// A table that no kernel writes, in the constant address space: what a wave
// reads there at a uniform address it reads with scalar loads.  From a plain
// pointer the compiler takes vector loads instead wherever a store or an atomic
// may have come before, one latency after the other, each wait including the
// stores (20 in a row at the end of the force pass: 104 -> 84 us for 96 small
// scenes, 62 -> 56 for 262,144 particles, 1,280 -> 1,232 for 4.2M).
template <typename V>
__device__ __forceinline__ const V* constant_table(const V* p)
{
    return (const V*)(const __attribute__((address_space(4))) V*)(uint64_t)p;
}

// The scene of the wave's slots (each of them lies in the same 64).
__device__ __forceinline__ int wave_scene(const int32_t* chunk_scene, int64_t slot)
{
    return constant_table(chunk_scene)[__builtin_amdgcn_readfirstlane((int32_t)(slot >> 6))];
}

__device__ __forceinline__ const SceneDev& scene_ref(const DevState& D, int scene)
{
    return constant_table(D.scenes)[scene];
}

// Element j of a per-slot array, addressed by a 32-bit byte offset from the
// (wave-uniform) base: the layout keeps every such array under 4 GiB.
template <typename V>
__device__ __forceinline__ V at(const V* __restrict__ base, uint32_t j)
{
    return *(const V*)((const char*)base + j * (uint32_t)sizeof(V));
}

// The same at a byte offset (j * sizeof(V), precomputed).
template <typename V>
__device__ __forceinline__ V at_byte(const V* __restrict__ base, uint32_t off)
{
    return *(const V*)((const char*)base + off);
}

__device__ __forceinline__ float d_fmax(float a, float b) { return __builtin_fmaxf(a, b); }
__device__ __forceinline__ double d_fmax(double a, double b) { return __builtin_fmax(a, b); }
__device__ __forceinline__ float d_fmin(float a, float b) { return __builtin_fminf(a, b); }
__device__ __forceinline__ double d_fmin(double a, double b) { return __builtin_fmin(a, b); }

// A floored cell coordinate clamped to [0, nmax]; negative and NaN give 0
// (max(NaN, 0) = 0), branch-free.  nmax is exact in T: the layout keeps grid
// and sub-cell extents below 2^24.
template <typename T>
__device__ __forceinline__ int cidx(T f, int nmax)
{
    return (int)d_fmin(d_fmax(f, T(0)), T(nmax));
}

template <typename T>
__device__ __forceinline__ void cell_of(const SceneConsts<T>& K, const int32_t* dims, T x, T y, T z,
                                        int& kx, int& ky, int& kz)
{
    kx = cidx<T>(d_floor((x - K.org[0]) * K.inv_cell), dims[0] - 1);
    ky = cidx<T>(d_floor((y - K.org[1]) * K.inv_yz), dims[1] - 1);
    kz = cidx<T>(d_floor((z - K.org[2]) * K.inv_yz), dims[2] - 1);
}

// Value of lane l ^ M.  Within a quad (M = 1, 2) a DPP quad permute (ALU
// only); otherwise a wave shuffle.
template <int M>
__device__ __forceinline__ float lane_xor(float v)
{
    if constexpr (M == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false));
    else if constexpr (M == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, false));
    else return __shfl_xor(v, M, SPHE_WAVE);
}
template <int M>
__device__ __forceinline__ double lane_xor(double v)
{
    if constexpr (M <= 2) {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
        constexpr int ctrl = M == 1 ? 0xB1 : 0x4E;  // quad_perm [1,0,3,2] / [2,3,0,1]
        const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, ctrl, 0xF, 0xF, false);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), ctrl, 0xF, 0xF, false);
        return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
    } else {
        return __shfl_xor(v, M, SPHE_WAVE);
    }
}

// Neighbour-sum accumulators.  A particle's sum is split over the G lanes of
// its group (density: lane l takes positions l, l+G, ... of the candidate
// stream; forces: list entries l, l+G, ...); merge_xor<M>() combines the
// partials of lanes l and l^M, so a xor tree over M = 1, 2, .. G/2 leaves
// the whole sum in every lane.
template <typename T, bool COMP> struct Acc;
template <typename T> struct Acc<T, true> {
    // Kahan: the represented sum is s - c
    T s = T(0), c = T(0);
    __device__ __forceinline__ void add(T v)
    {
        T y = v - c;
        T t = s + y;
        c = (t - s) - y;
        s = t;
    }
    // TwoSum of the heads (exact error e), compensations added: the result
    // is the same in both lanes of the pair.
    template <int M>
    __device__ __forceinline__ void merge_xor()
    {
        const T os = lane_xor<M>(s);
        const T oc = lane_xor<M>(c);
        const bool low = (threadIdx.x & M) == 0;
        const T a = low ? s : os, b = low ? os : s;
        const T ca = low ? c : oc, cb = low ? oc : c;
        const T sum = a + b;
        const T bb = sum - a;
        const T e = (a - (sum - bb)) + (b - bb);
        s = sum;
        c = (ca + cb) - e;
    }
    __device__ __forceinline__ T value() const { return s - c; }
};
template <typename T> struct Acc<T, false> {
    T s = T(0);
    __device__ __forceinline__ void add(T v) { s = s + v; }
    template <int M>
    __device__ __forceinline__ void merge_xor()
    {
        const T os = lane_xor<M>(s);
        const bool low = (threadIdx.x & M) == 0;
        s = low ? s + os : os + s;
    }
    __device__ __forceinline__ T value() const { return s; }
};

// Summation modes of the neighbour sums (the precision argument of
// sphe_create picks one): plain; Kahan-compensated density and force sums;
// compensated density sums with the force sums accumulated in FP64.
#define SUM_PLAIN 0
#define SUM_KAHAN 1
#define SUM_F64ACC 2

// FP64 sum of FP32 terms (plain adds; the lanes of a pair merge with the
// same commutative add, so both hold identical bits), rounded to FP32 once.
struct AccF64 {
    double s = 0.0;
    __device__ __forceinline__ void add(float v) { s = s + (double)v; }
    template <int M>
    __device__ __forceinline__ void merge_xor()
    {
        const double os = lane_xor<M>(s);
        s = s + os;
    }
    __device__ __forceinline__ float value() const { return (float)s; }
};

template <int G, typename A>
__device__ __forceinline__ void group_merge(A& a)
{
    if constexpr (G > 1) a.template merge_xor<1>();
    if constexpr (G > 2) a.template merge_xor<2>();
    if constexpr (G > 4) a.template merge_xor<4>();
}

// x sub-cell of a position inside its cell: the cell is split into
// 2^sub_log2 slabs along x, and a cell's particles are sorted by (slab, id).
// gx * 2^s is exact, so the slab index lies in [0, 2^s) for every position
// (clamped and non-finite ones included).
template <typename T>
__device__ __forceinline__ int sub_cell(T gx, int kx, int nx, int sl)
{
    return cidx<T>(d_floor(gx * T(1 << sl)), (nx << sl) - 1) - (kx << sl);
}

// A row gap g (a lower bound of the distance to a row, in x-cell units)
// less the rounding margin, floored at 0.
#define SPHE_ROW_MARGIN 0.015625
template <typename T>
__device__ __forceinline__ T row_gap(T f)
{
    const T a = f - T(SPHE_ROW_MARGIN);
    return a > T(0) ? a : T(0);
}

// The stencil rows of a particle, clipped to what the smoothing sphere can
// reach.  Cells are h (1 + 2^-8) along x and 1/yz of that along y and z
// (yz = 1, 2 or 3), so the rows are the (2 yz + 1)^2 (y, z) columns around the
// particle, numbered r = W (dz + yz) + (dy + yz), W = 2 yz + 1 (dz outer, dy
// inner).  In x-cell units the radius is h / cell < 1; a row whose y and z
// gaps g satisfy gy^2 + gz^2 > 1 is skipped, and the others keep the x
// sub-cells that meet [gx - w, gx + w], w = sqrt(1 - gy^2 - gz^2) + margin.
// Every neighbour is inside the range: the bounds are monotone in the
// position and include a margin far above the rounding of the cell
// coordinates.  Cells with more than 1023 particles carry no slab offsets
// and are taken whole.
// Half-width of a clipped row, in x-cell units, before the margin: at least
// sqrt(x) - 2e-3 for x in [0, 1].  FP64: sqrt.  FP32: x / sqrt(x) with one
// Newton step y <- y (1.5 - (x/2) y^2) for 1/sqrt(x) from the integer
// estimate 0x5f375a86 - bits(x)/2 (relative error at most 1.75e-3); the row
// margin (2^-6) covers the difference, and the sequence is IEEE operations
// only, so a CPU replays the same rows.
template <typename T> struct RowWidth {
    static __device__ __forceinline__ T of(T x) { return d_sqrt(x); }
};
template <> struct RowWidth<float> {
    static __device__ __forceinline__ float of(float x)
    {
        float y = __int_as_float(0x5f375a86 - (__float_as_int(x) >> 1));
        const float t = (0.5f * x) * y;
        y = y * __builtin_fmaf(-t, y, 1.5f);
        return x * y;
    }
};

template <typename T>
struct RowProbe {
    T gx, scale;
    // gaps, in x-cell units, to the rows one, two and three cells below (l1,
    // l2, l3) and above (h1, h2, h3) along y and z (the third with yz = 3)
    T yl1, yl2, yh1, yh2, zl1, zl2, zh1, zh2, yl3, yh3, zl3, zh3;
    int kx, ky, kz, sl, smax, fmax, flo_min, fhi_max;
    uint32_t rbase;  // global index of the first cell of the particle's own row
};

// r / W for 0 <= r < W^2 and W = 3, 5 or 7 (multiply and shift)
__host__ __device__ constexpr int row_div(int r, int W)
{
    return W == 3 ? (r * 11) >> 5 : (W == 5 ? (r * 13) >> 6 : (r * 37) >> 8);
}
constexpr bool row_div_exact()
{
    for (int W = 3; W <= 7; W += 2)
        for (int r = 0; r < W * W; ++r)
            if (row_div(r, W) != r / W) return false;
    return true;
}
static_assert(row_div_exact(), "row_div");

template <typename T>
__device__ __forceinline__ RowProbe<T> row_probe(const DevState& D, const SceneDev& S, const SceneConsts<T>& K,
                                                 T xi, T yi, T zi)
{
    RowProbe<T> P;
    const int nx = S.dims[0], ny = S.dims[1], nz = S.dims[2];
    P.gx = (xi - K.org[0]) * K.inv_cell;
    const T gy = (yi - K.org[1]) * K.inv_yz;
    const T gz = (zi - K.org[2]) * K.inv_yz;
    P.kx = cidx<T>(d_floor(P.gx), nx - 1);
    P.ky = cidx<T>(d_floor(gy), ny - 1);
    P.kz = cidx<T>(d_floor(gz), nz - 1);
    P.rbase = (uint32_t)S.cell_off + (uint32_t)((P.kz * ny + P.ky) * nx);
    const T fy = gy - T(P.ky), fz = gz - T(P.kz);
    const T q = K.yz_scale;  // 1 / yz, exact
    P.yl1 = row_gap<T>(fy * q);
    P.yh1 = row_gap<T>((T(1) - fy) * q);
    P.yl2 = row_gap<T>((T(1) + fy) * q);
    P.yh2 = row_gap<T>((T(1) + (T(1) - fy)) * q);
    P.zl1 = row_gap<T>(fz * q);
    P.zh1 = row_gap<T>((T(1) - fz) * q);
    P.zl2 = row_gap<T>((T(1) + fz) * q);
    P.zh2 = row_gap<T>((T(1) + (T(1) - fz)) * q);
    P.yl3 = P.yh3 = P.zl3 = P.zh3 = T(0);
    if (D.yz > 2) {  // uniform
        P.yl3 = row_gap<T>((T(2) + fy) * q);
        P.yh3 = row_gap<T>((T(2) + (T(1) - fy)) * q);
        P.zl3 = row_gap<T>((T(2) + fz) * q);
        P.zh3 = row_gap<T>((T(2) + (T(1) - fz)) * q);
    }
    P.sl = D.sub_log2;
    P.smax = (1 << P.sl) - 1;
    P.scale = T(1 << P.sl);
    P.fmax = (nx << P.sl) - 1;
    P.flo_min = (P.kx > 0 ? P.kx - 1 : 0) << P.sl;
    P.fhi_max = ((P.kx < nx - 1 ? P.kx + 1 : nx - 1) << P.sl) + P.smax;
    return P;
}

template <typename T>
__device__ __forceinline__ T gap_of(int d, int yz, T l1, T l2, T l3, T h1, T h2, T h3)
{
    // selects of values at hand: -1 l1, 1 h1, -2 l2, 2 h2, 0, and with
    // yz = 3 (a uniform branch) -3 l3, 3 h3
    const T one = d < 0 ? l1 : h1;
    const T two = d < 0 ? l2 : h2;
    T g = (d == 2 || d == -2) ? two : one;
    if (yz > 2) {
        const T three = d < 0 ? l3 : h3;
        g = (d == 3 || d == -3) ? three : g;
    }
    return d == 0 ? T(0) : g;
}

// Slot range [j0, j1) of the row at (dy, dz); false when the row is outside
// the grid or out of the sphere's reach.  roff = (dz ny + dy) nx, the row's
// cell offset from the particle's own row (mod 2^32), kept by the callers.
// The cell records a row may need are loaded unconditionally (a skipped row
// reads the particle's own row), so a row costs one memory round trip.
template <typename T>
__device__ __forceinline__ bool row_range(const DevState& D, const SceneDev& S, const RowProbe<T>& P, int dyc,
                                          int dzc, uint32_t roff, uint32_t& j0, uint32_t& j1)
{
    const int ny = S.dims[1], nz = S.dims[2];
    const int z = P.kz + dzc, y = P.ky + dyc;
    const T mz = gap_of<T>(dzc, D.yz, P.zl1, P.zl2, P.zl3, P.zh1, P.zh2, P.zh3);
    const T my = gap_of<T>(dyc, D.yz, P.yl1, P.yl2, P.yl3, P.yh1, P.yh2, P.yh3);
    const T r2 = my * my + mz * mz;
    const bool on = (z >= 0) & (z < nz) & (y >= 0) & (y < ny) & (r2 <= T(1));
    const T w = RowWidth<T>::of(T(1) - (on ? r2 : T(0))) + T(SPHE_ROW_MARGIN);
    int flo = cidx<T>(d_floor((P.gx - w) * P.scale), P.fmax);
    int fhi = cidx<T>(d_floor((P.gx + w) * P.scale), P.fmax);
    flo = max(flo, P.flo_min);
    fhi = min(fhi, P.fhi_max);
    const uint32_t rk = on ? P.rbase + roff : P.rbase;
    const int sl = P.sl, smax = P.smax;
    const uint32_t clo = rk + (uint32_t)(flo >> sl), chi = rk + (uint32_t)(fhi >> sl);
    const uint2 rlo = D.cells[clo], rhi = D.cells[chi];
    const uint32_t s_hi1 = D.cells[(size_t)chi + 1].x;
    // slab offsets (none with one slab: slo = 0, shi = smax); an empty cell's
    // word is 0
    const int slo = flo & smax, shi = fhi & smax;
    // field shifts from byte tables: 10 (slo - 1) for slo = 1..3, 10 shi
    const uint32_t sh0 = (0x140A0000u >> ((uint32_t)slo << 3)) & 0xFFu;
    const uint32_t sh1 = (0x1E140A00u >> ((uint32_t)shi << 3)) & 0xFFu;
    const uint32_t f0 = (slo != 0 && !(rlo.y >> 31)) ? (rlo.y >> sh0) & 1023u : 0u;
    const bool use1 = shi != smax && !(rhi.y >> 31);
    const uint32_t a = rlo.x + f0;
    const uint32_t b = use1 ? rhi.x + ((rhi.y >> sh1) & 1023u) : s_hi1;
    // rows of real cells lie inside [p_begin, p_begin + n); the clamp only
    // matters if the counts were inconsistent
    const uint32_t lo = (uint32_t)S.p_begin, hi = (uint32_t)(S.p_begin + S.n);
    j0 = max(a, lo);
    j1 = min(b, hi);
    return on;
}

// Calls row(j0, j1) for each row that may hold a neighbour, in row order.
template <typename T, typename F>
__device__ __forceinline__ void for_each_row(const DevState& D, const SceneDev& S, const SceneConsts<T>& K,
                                             T xi, T yi, T zi, F&& row)
{
    const RowProbe<T> P = row_probe<T>(D, S, K, xi, yi, zi);
    const int yz = D.yz;
    const int nx = S.dims[0], nyx = S.dims[1] * nx;
    for (int dz = -yz; dz <= yz; ++dz) {
        uint32_t roff = (uint32_t)(dz * nyx - yz * nx);
        for (int dy = -yz; dy <= yz; ++dy, roff += (uint32_t)nx) {
            uint32_t j0, j1;
            if (row_range<T>(D, S, P, dy, dz, roff, j0, j1)) row(j0, j1);
        }
    }
}

// Visits the candidates of the clipped stencil rows in ascending slot order
// and calls f(j, dx, dy, dz, d2) for those inside the smoothing radius.
template <typename T, typename F>
__device__ __forceinline__ void visit_neighbours(const DevState& D, const SceneDev& S, const SceneConsts<T>& K,
                                                 const V4<T>* __restrict__ pos, T xi, T yi, T zi, F&& f)
{
    for_each_row<T>(D, S, K, xi, yi, zi, [&](uint32_t j0, uint32_t j1) {
            uint32_t j = j0;
            for (; j + 1 < j1; j += 2) {  // two loads in flight
                const V4<T> pa = pos[j];
                const V4<T> pb = pos[j + 1];
                const T ax = xi - pa.x, ay = yi - pa.y, az = zi - pa.z;
                const T a2 = (ax * ax + ay * ay) + az * az;
                if (a2 <= K.thr) f(j, ax, ay, az, a2);
                const T bx = xi - pb.x, by = yi - pb.y, bz = zi - pb.z;
                const T b2 = (bx * bx + by * by) + bz * bz;
                if (b2 <= K.thr) f(j + 1, bx, by, bz, b2);
            }
            if (j < j1) {
                const V4<T> pj = pos[j];
                const T dx = xi - pj.x, dy = yi - pj.y, dz = zi - pj.z;
                const T d2 = (dx * dx + dy * dy) + dz * dz;
                if (d2 <= K.thr) f(j, dx, dy, dz, d2);
            }
    });
}

// Counting-sort key of a position: the cell key shifted left by sub_log2,
// or-ed with the x slab.
template <typename T>
__device__ __forceinline__ int32_t position_key(const DevState& D, const SceneDev& S, const SceneConsts<T>& K, T x, T y,
                                                T z)
{
    const T gx = (x - K.org[0]) * K.inv_cell;
    const int kx = cidx<T>(d_floor(gx), S.dims[0] - 1);
    const int ky = cidx<T>(d_floor((y - K.org[1]) * K.inv_yz), S.dims[1] - 1);
    const int kz = cidx<T>(d_floor((z - K.org[2]) * K.inv_yz), S.dims[2] - 1);
    const int64_t key = S.cell_off + ((int64_t)kz * S.dims[1] + ky) * S.dims[0] + kx;
    const int sub = sub_cell<T>(gx, kx, S.dims[0], D.sub_log2);
    return (int32_t)((key << D.sub_log2) | sub);
}

// Word of scan tile t's total, and the tile of word w.
__device__ __forceinline__ uint32_t tile_word(int tlog, uint32_t t) { return ((t & ((1u << tlog) - 1u)) << 5) | (t >> tlog); }
__device__ __forceinline__ uint32_t word_tile(int tlog, uint32_t w) { return ((w & 31u) << tlog) | (w >> 5); }

// Counts a particle of that key into its scan tile and its cell: its rank of
// arrival in the cell.  In the largest contexts and those of many particles a
// tile (D.totals 0) the tile is only marked.  The lanes that count here together
// are mostly neighbours of one tile, which takes one atomic of the wave then
// (with the totals in tile order, and so on a few lines, the force pass took 77
// us instead of 57 for 262,144 particles, and 289 instead of 155 for 48 uneven
// scenes).
__device__ __forceinline__ uint32_t count_key(const DevState& D, int32_t key)
{
    const int32_t cell = key >> D.sub_log2, tile = cell >> D.scan_log2;
    const uint32_t rank = atomicAdd(&D.cnt[cell], 1u);
    if (!D.totals) {
        D.total[tile_word(D.tlog, (uint32_t)tile)] = 1u;
        return rank;
    }
    const int32_t t0 = __builtin_amdgcn_readfirstlane(tile);
    const uint64_t same = __builtin_amdgcn_ballot_w64(tile == t0);
    const bool leads =
        __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u)) == 0u;
    if (tile != t0 || leads)
        atomicAdd(&D.total[tile_word(D.tlog, (uint32_t)tile)], tile != t0 ? 1u : (uint32_t)__popcll(same));
    return rank;
}

template <typename T>
__device__ __forceinline__ void count_position(const DevState& D, const SceneDev& S, const SceneConsts<T>& K,
                                               int64_t slot, T x, T y, T z)
{
    const int32_t key = position_key<T>(D, S, K, x, y, z);
    D.key[slot] = key;
    D.arank[slot] = count_key(D, key);
}

__device__ __forceinline__ void count_pad(const DevState& D, const SceneDev& S, int64_t slot)
{
    const int64_t key = S.cell_off + S.ncell;
    D.key[slot] = (int32_t)(key << D.sub_log2);
    D.arank[slot] = count_key(D, (int32_t)(key << D.sub_log2));
}

// ------------------------------------------------------------------ sort

template <typename T>
__global__ __launch_bounds__(256) void k_hash_count(DevState D)
{
    const int64_t slot = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= D.P) return;
    const SceneDev& S = scene_ref(D, wave_scene(D.chunk_scene, slot));
    if (slot < S.p_begin + S.n) {
        const SceneConsts<T>& K = SceneSel<T>::get(S);
        const V4<T> p = ((const V4<T>*)D.u_pos)[slot];
        count_position<T>(D, S, K, slot, p.x, p.y, p.z);
    } else {
        count_pad(D, S, slot);
    }
}

// A scan tile is 256 threads x ITEMS counts (ITEMS = 8, 16 or 32: tiles of
// 2^11, 2^12 or 2^13 cells, DevState::scan_log2).  A wave takes a run of
// 64 ITEMS consecutive cells, four cells a lane at a time (chunks of 256
// cells), so that its loads and stores are runs of consecutive lines.

// Inclusive sums of x over the wave's lanes, in six DPP adds.
__device__ __forceinline__ uint32_t wave_sums(uint32_t x)
{
#define SPHE_DPP_ADD(ctrl, rows) x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ctrl, rows, 0xF, false)
    SPHE_DPP_ADD(0x111, 0xF);  // row_shr 1, 2, 4, 8: within rows of 16 lanes
    SPHE_DPP_ADD(0x112, 0xF);
    SPHE_DPP_ADD(0x114, 0xF);
    SPHE_DPP_ADD(0x118, 0xF);
    SPHE_DPP_ADD(0x142, 0xA);  // row_bcast 15 into rows 1 and 3
    SPHE_DPP_ADD(0x143, 0xC);  // row_bcast 31 into rows 2 and 3
#undef SPHE_DPP_ADD
    return x;
}
__device__ __forceinline__ uint32_t wave_total(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)wave_sums(x), 63);
}

// First cell of chunk c of this lane's wave in the tile.
template <int ITEMS>
__device__ __forceinline__ int64_t tile_cell(int64_t tile, int c)
{
    return tile * (256 * ITEMS) + (int64_t)(threadIdx.x >> 6) * (64 * ITEMS) + c * 256 + (threadIdx.x & 63) * 4;
}

template <int ITEMS>
__device__ __forceinline__ void load_tile(const uint32_t* __restrict__ p, int64_t tile, int64_t n, uint4* v)
{
#pragma unroll
    for (int c = 0; c < ITEMS / 4; ++c) {
        const int64_t i = tile_cell<ITEMS>(tile, c);
        if (i + 4 <= n) v[c] = *(const uint4*)(p + i);
        else v[c] = make_uint4(i < n ? p[i] : 0u, i + 1 < n ? p[i + 1] : 0u, i + 2 < n ? p[i + 2] : 0u, 0u);
    }
}

// Four consecutive cell records (value, 0).
__device__ __forceinline__ void store4(uint2* __restrict__ p, int64_t i, int64_t n, uint4 v)
{
    if (i + 4 <= n) {
        ((uint4*)(p + i))[0] = make_uint4(v.x, 0u, v.y, 0u);
        ((uint4*)(p + i))[1] = make_uint4(v.z, 0u, v.w, 0u);
    } else {
        if (i < n) p[i] = make_uint2(v.x, 0u);
        if (i + 1 < n) p[i + 1] = make_uint2(v.y, 0u);
        if (i + 2 < n) p[i + 2] = make_uint2(v.z, 0u);
    }
}

// Exclusive prefix, in tile order, of the 32 2^tlog words of the tiles' totals,
// word by word (tile_word's order), by one block of 1,024 threads.  A line has
// one tile of each of 32 runs of 2^tlog tiles: thread (q, g) adds up the words
// 4 q .. 4 q + 3 of its 2^tlog / 128 consecutive lines, a scan over the 32 runs'
// 128 sums each gives where it starts, and a second pass over its lines leaves
// the prefixes.  So lines are read and written whole (scan of 1,000 particles in
// 360M cells, 88,000 tiles: 63 us; 129 with 16 consecutive tiles to a thread,
// each from a line of its own).  tlog >= 8.
__global__ __launch_bounds__(1024) void k_scan_tiles(const uint32_t* __restrict__ total, int tlog,
                                                     uint32_t* __restrict__ pre)
{
    __shared__ __attribute__((aligned(16))) uint32_t sums[32 * 128];
    __shared__ uint32_t waves[16];
    const int q = threadIdx.x & 7, g = threadIdx.x >> 3, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lines = 1 << (tlog - 7);  // at least 2
    const uint4* src = (const uint4*)total + ((int64_t)g * lines * 8 + q);
    uint4* dst = (uint4*)pre + ((int64_t)g * lines * 8 + q);
    // calls f(line, words) for the thread's lines, eight or two loads in flight
    auto each = [&](auto&& f) {
        auto run = [&](auto count) {
            constexpr int U = decltype(count)::value;
            for (int i = 0; i < lines; i += U) {
                uint4 v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) v[u] = src[(i + u) * 8];
#pragma unroll
                for (int u = 0; u < U; ++u) f(i + u, v[u]);
            }
        };
        if (lines >= 8) run(std::integral_constant<int, 8>());
        else run(std::integral_constant<int, 2>());
    };
    uint4 s = make_uint4(0u, 0u, 0u, 0u);
    each([&](int, const uint4& v) { s = make_uint4(s.x + v.x, s.y + v.y, s.z + v.z, s.w + v.w); });
    uint32_t* const mine = sums + 4 * q * 128 + g;
    mine[0] = s.x;
    mine[128] = s.y;
    mine[256] = s.z;
    mine[384] = s.w;
    __syncthreads();
    uint4 t = ((const uint4*)sums)[threadIdx.x];
    const uint32_t all = (t.x + t.y) + (t.z + t.w);
    const uint32_t x = wave_sums(all);  // over the wave, then the 16 wave totals
    if (lane == 63) waves[wave] = x;
    __syncthreads();
    uint32_t at = x - all;
#pragma unroll
    for (int k = 0; k < 16; ++k) at += k < wave ? waves[k] : 0u;
    t = make_uint4(at, at + t.x, at + t.x + t.y, at + t.x + t.y + t.z);
    ((uint4*)sums)[threadIdx.x] = t;
    __syncthreads();
    uint4 r = make_uint4(mine[0], mine[128], mine[256], mine[384]);
    each([&](int i, const uint4& v) {
        dst[i * 8] = r;
        r = make_uint4(r.x + v.x, r.y + v.y, r.z + v.z, r.w + v.w);
    });
}

// Where a tile's prefix (the total of the tiles before it) comes from: a word
// that k_scan_tiles left, or the tiles' totals, added here by every block: up
// to SCAN_SUM_TILES tiles, at most four loads a thread, while a launch costs 4
// us.  The totals themselves are counted with the particles (count_key; a pass
// over the counts for them took a launch: 13.2 -> 7.3 us on 6.7M cells, 19.6 ->
// 13.8 for 96 scenes with their terrain heights; for few tiles every block added
// the counts before its tile: 5.6 -> 4.2 us on 39,000 cells), except where the
// atomics cost more (count_totals).
enum { SCAN_PREFIX, SCAN_SUMS };
#define SPHE_SCAN_SUM_TILES 4096
__host__ __device__ inline int64_t scan_tiles(const DevState& D)
{
    return (D.C + 1 + (1ll << D.scan_log2) - 1) >> D.scan_log2;
}
__host__ __device__ inline bool scan_sums(const DevState& D) { return scan_tiles(D) <= SPHE_SCAN_SUM_TILES; }

// start = exclusive prefix of the counts of one tile (each cell's first scatter
// resets its count for the next arrivals; the tile's total is reset here where
// no other block reads it, else by the scatter: scan_sums).
// A tile whose total is 0 holds only zero counts, which are not read.  fill:
// per tile, the value all of an empty tile's starts hold since the tile was
// last written empty (~0: not known); an empty tile whose prefix equals it is
// not written again.
template <int ITEMS, int FROM>
__device__ __forceinline__ void scan_down_tile(const uint32_t* __restrict__ cnt, uint2* __restrict__ start, int64_t n,
                                               uint32_t* __restrict__ total, int tlog,
                                               const uint32_t* __restrict__ tpre,
                                               uint32_t* __restrict__ fill, int tile, uint32_t* lds)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool empty = total[tile_word(tlog, (uint32_t)tile)] == 0u;  // block-uniform
    const uint32_t filled = fill[tile];
    uint4 v[ITEMS / 4];
    if (empty) {
#pragma unroll
        for (int c = 0; c < ITEMS / 4; ++c) v[c] = make_uint4(0u, 0u, 0u, 0u);
    } else {
        load_tile<ITEMS>(cnt, tile, n, v);
    }
    uint32_t pre = 0;  // this thread's share of the prefix
    if constexpr (FROM == SCAN_PREFIX) {
        pre = threadIdx.x == 0 ? tpre[tile_word(tlog, (uint32_t)tile)] : 0u;
    } else {
        // in the order of the words, so that they are read as lines
#pragma unroll 2
        for (uint32_t w = threadIdx.x * 4u; w < (32u << tlog); w += 1024u) {
            const uint4 q = *(const uint4*)(total + w);
            pre += word_tile(tlog, w) < (uint32_t)tile ? q.x : 0u;
            pre += word_tile(tlog, w + 1u) < (uint32_t)tile ? q.y : 0u;
            pre += word_tile(tlog, w + 2u) < (uint32_t)tile ? q.z : 0u;
            pre += word_tile(tlog, w + 3u) < (uint32_t)tile ? q.w : 0u;
        }
    }
    // sums over the wave of each chunk, then of the waves before
    uint32_t run[ITEMS / 4], sum = 0;
#pragma unroll
    for (int c = 0; c < ITEMS / 4; ++c) {
        const uint32_t q = (v[c].x + v[c].y) + (v[c].z + v[c].w);
        const uint32_t x = wave_sums(q);
        run[c] = sum + x - q;
        sum += (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
    }
    const uint32_t wpre = wave_total(pre);
    if (lane == 0) {
        lds[wave] = sum;
        lds[4 + wave] = wpre;
    }
    __syncthreads();
    const uint32_t ptot = (lds[4] + lds[5]) + (lds[6] + lds[7]);
    uint32_t base = ptot;
#pragma unroll
    for (int k = 0; k < 3; ++k) base += k < wave ? lds[k] : 0u;
    // an empty tile's starts all equal ptot: unwritten when they already do
    if (!(empty && filled == ptot)) {
#pragma unroll
        for (int c = 0; c < ITEMS / 4; ++c) {
            uint4 o;
            o.x = base + run[c];
            o.y = o.x + v[c].x;
            o.z = o.y + v[c].y;
            o.w = o.z + v[c].z;
            store4(start, tile_cell<ITEMS>(tile, c), n, o);
        }
    }
    // every thread read the total and the fill word before the barrier
    if (threadIdx.x == 0) {
        const uint32_t nf = empty ? ptot : ~0u;
        if (nf != filled) fill[tile] = nf;
        if (FROM == SCAN_PREFIX && !empty) total[tile_word(tlog, (uint32_t)tile)] = 0u;
    }
}

__global__ __launch_bounds__(256) void k_scatter(DevState D)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    // the tiles' totals are used up
    if (scan_sums(D))
        for (int64_t w = p; w < (32ll << D.tlog); w += (int64_t)gridDim.x * blockDim.x) D.total[w] = 0u;
    if (p >= D.P) return;
    const int32_t key = D.key[p];  // cell key << sub_log2 | slab
    const int32_t c = key >> D.sub_log2;
    if (key < 0 || (int64_t)c >= D.C) {
        atomicOr(D.status, 2u);
        return;
    }
    const uint32_t r = D.arank[p];
    const uint32_t d = D.cells[c].x + r;
    // the cell's count is used up: its first arrival (one per counted cell)
    // resets it for the next step's arrivals
    if (r == 0u) D.cnt[c] = 0u;
    if ((int64_t)d >= D.P) {  // counts inconsistent with the slots: report, never write out of range
        atomicOr(D.status, 2u);
        return;
    }
    // (key, id) as one word that compares as the pair: id's sign bit flipped
    D.tmp_kid[d] = ((uint64_t)(uint32_t)key << 32) | (uint32_t)(D.u_id[p] ^ (int32_t)0x80000000);
    D.tmp_src[d] = (int32_t)p;
}

// Canonical order inside a cell: ascending x slab, then ascending id (ties,
// which only duplicate ids produce, by previous slot).  The particle ranked
// first also writes the cell's slab offsets: for s = 1 .. 2^sub_log2 - 1 the
// number of the cell's particles in slabs below s, 10 bits each from bit
// 10 (s - 1); a cell of more than 1023 particles gets bit 31 instead.
// A particle's rank is counted over its cell's (key, id) words, staged in LDS by
// the block: at once, without waiting for the cells' ranges, the words of its
// own 256 slots and of SPHE_REORDER_SIDE on either side; where a cell reaches
// further (a pile-up), the words of the cells its slots lie in (a window of at
// most SPHE_REORDER_WINDOW slots); a block whose cells are larger still ranks
// from memory.  The pass is a chain of latencies up to some 100,000 particles:
// words, then cell ranges and the particle's state together, then the stores
// (262,144 particles: 9.9 us with the window read after the ranges and the
// state after the window, 8.0 now); bound by HBM beyond (100 bytes a particle:
// 4.2M 99 us, now 79, 5.3 TB/s).
#define SPHE_REORDER_WINDOW 2048
#define SPHE_REORDER_SIDE 256
template <typename T>
__global__ __launch_bounds__(256) void k_reorder(DevState D)
{
    __shared__ uint64_t wkid[SPHE_REORDER_WINDOW];
    __shared__ uint32_t wlo, whi;
    constexpr int SIDE = SPHE_REORDER_SIDE;
    const int64_t base = (int64_t)blockIdx.x * 256;
    const int64_t d = base + threadIdx.x;
    const bool live = d < D.P;
    const int sl = D.sub_log2;
    // slots before and after the block's, clamped to the array's (P > 0)
    const int64_t before = base - SIDE + (int64_t)threadIdx.x, after = base + 256 + (int64_t)threadIdx.x;
    const uint64_t kb = D.tmp_kid[before < 0 ? 0 : before], ka = D.tmp_kid[after < D.P ? after : D.P - 1];
    const uint64_t kid = D.tmp_kid[live ? d : D.P - 1];
    const int32_t src = D.tmp_src[live ? d : D.P - 1];
    wkid[threadIdx.x] = kb;
    wkid[SIDE + threadIdx.x] = kid;
    wkid[SIDE + 256 + threadIdx.x] = ka;
    const int32_t fk = (int32_t)(kid >> 32);
    const int32_t c = fk >> sl;
    const bool ok = live && fk >= 0 && (int64_t)c < D.C;
    const uint32_t cc = ok ? (uint32_t)c : 0u;
    // the particle's state, gathered while its rank is found (from a slot
    // clamped into range: a bad src is reported below and never stored)
    const uint32_t sc = (uint32_t)min(max(src, 0), (int32_t)(D.P - 1));
    uint32_t s0 = D.cells[cc].x, s1 = D.cells[cc + 1u].x;
    const V4<T> pv = at((const V4<T>*)D.u_pos, sc);
    const V4<T> vv = at((const V4<T>*)D.u_vel, sc);
    const int64_t sed = D.u_sed[sc];
    if (!ok) s0 = s1 = 0u;
    if ((int64_t)s1 > D.P) s1 = (uint32_t)D.P;
    uint32_t w0 = (uint32_t)(base > SIDE ? base - SIDE : 0);
    int shift = (int)(base - SIDE);  // slot of wkid[0]; negative in the first block
    bool staged = true;
    if (__syncthreads_or(s0 < s1 && (s0 < w0 || (int64_t)s1 > base + 256 + SIDE))) {
        if (threadIdx.x == 0) {
            wlo = ~0u;
            whi = 0u;
        }
        __syncthreads();
        {
            // the block's window of cell slots: reduced over each wave, then
            // one LDS atomic pair per wave
            uint32_t lo = s0 < s1 ? s0 : ~0u, hi = s0 < s1 ? s1 : 0u;
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) {
                const uint32_t a = __shfl_xor(lo, o, 64), b = __shfl_xor(hi, o, 64);
                lo = a < lo ? a : lo;
                hi = b > hi ? b : hi;
            }
            if ((threadIdx.x & 63) == 0 && lo < hi) {
                atomicMin(&wlo, lo);
                atomicMax(&whi, hi);
            }
        }
        __syncthreads();
        w0 = wlo;
        const uint32_t w1 = whi;
        staged = w0 < w1 && w1 - w0 <= (uint32_t)SPHE_REORDER_WINDOW;  // block-uniform
        if (staged)
            for (uint32_t j = w0 + threadIdx.x; j < w1; j += blockDim.x) wkid[j - w0] = D.tmp_kid[j];
        __syncthreads();
        shift = (int)w0;
    }
    if (!live) return;
    if (!ok) {
        atomicOr(D.status, 2u);
        return;
    }
    const int32_t my = (int32_t)((uint32_t)kid ^ 0x80000000u);
    // one count field per slab boundary: a particle in slab k adds 1 to the
    // fields of the boundaries s > k
    const uint32_t fields = sl == 2 ? 0x100401u : (sl == 1 ? 1u : 0u);
    const uint32_t smask = (1u << sl) - 1u;
    uint32_t rank = 0, below = 0;
    auto take = [&](uint32_t j, uint64_t o) {
        rank += o < kid ? 1u : 0u;
        if (__builtin_expect(o == kid && j != (uint32_t)d, 0)) rank += D.tmp_src[j] < src ? 1u : 0u;
        below += fields & (~0u << (10u * ((uint32_t)(o >> 32) & smask)));
    };
    uint32_t j = s0;
    if (staged) {
        for (; j + 3 < s1; j += 4) {
            const uint64_t* w = wkid + ((int)j - shift);
            const uint64_t o0 = w[0], o1 = w[1], o2 = w[2], o3 = w[3];
            take(j, o0);
            take(j + 1, o1);
            take(j + 2, o2);
            take(j + 3, o3);
        }
        for (; j < s1; ++j) take(j, wkid[(int)j - shift]);
    } else {
        for (; j + 1 < s1; j += 2) {  // two loads in flight
            const uint64_t o0 = D.tmp_kid[j], o1 = D.tmp_kid[j + 1];
            take(j, o0);
            take(j + 1, o1);
        }
        if (j < s1) take(j, D.tmp_kid[j]);
    }
    const uint32_t f = s0 + rank;
    if ((int64_t)f >= D.P || src < 0 || (int64_t)src >= D.P) {
        atomicOr(D.status, 2u);
        return;
    }
    if (rank == 0) D.cells[c].y = s1 - s0 > 1023u ? 0x80000000u : below;
    ((V4<T>*)D.s_pos)[f] = pv;
    ((V4<T>*)D.s_vel)[f] = vv;
    D.s_sed[f] = sed;
    D.s_id[f] = my;
}

// --------------------------------------------------------------- density

// Candidates per lane per iteration of the density pass (at most 4: one
// byte each in the placement word).
#define SPHE_DENSITY_UNROLL 4

// Inclusive prefix sum of x over the G lanes of a group (lane l gets
// x_0 + ... + x_l); *tot = the group's total.  The G lanes are consecutive
// lanes of the wave, starting at a multiple of G.
template <int G>
__device__ __forceinline__ uint32_t group_prefix(uint32_t x, int l, uint32_t* tot)
{
    uint32_t y = x;
#pragma unroll
    for (int d = 1; d < G; d <<= 1) {
        const uint32_t o = __shfl_up(y, d, G);
        if (l >= d) y += o;
    }
    *tot = __shfl(y, G - 1, G);
    return y;
}

// Running sums of v's bytes 0..2 in bytes 0..2 of the result (b0, b0+b1,
// b0+b1+b2; no carries while they stay below 256): the 24-bit product with
// 0x010101, one full-rate v_mul_u32_u24.  Written as that instruction: the
// compiler otherwise folds a following shift and add into a 64-bit
// multiply-add, a quarter-rate instruction.
__device__ __forceinline__ uint32_t byte_runs(uint32_t v)
{
    uint32_t r;
    asm("v_mul_u32_u24_e32 %0, 0x10101, %1" : "=v"(r) : "v"(v));
    return r;
}

// G = 4: the groups are the wave's quads; three DPP quad permutes.
template <>
__device__ __forceinline__ uint32_t group_prefix<4>(uint32_t x, int l, uint32_t* tot)
{
    // quad_perm [0,0,1,2]: lane l reads lane l-1
    const uint32_t s1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x90, 0xF, 0xF, false);
    uint32_t y = x + (l >= 1 ? s1 : 0u);
    // quad_perm [0,0,0,1]: lane l reads lane l-2
    const uint32_t s2 = (uint32_t)__builtin_amdgcn_mov_dpp((int)y, 0x40, 0xF, 0xF, false);
    y = y + (l >= 2 ? s2 : 0u);
    // quad_perm [3,3,3,3]: the total, from lane 3
    *tot = (uint32_t)__builtin_amdgcn_mov_dpp((int)y, 0xFF, 0xF, 0xF, false);
    return y;
}


// An LDS word addressed by its 32-bit LDS byte address (address space 3).
typedef __attribute__((address_space(3))) uint32_t lds_u32;

// Dynamic LDS of the density pass for ngroups lane groups: their row tables
// (W^2 + 1 entries of 8 bytes each), then their list staging rings (ring
// entries of 4 bytes each) from an offset aligned to a ring's size, so a
// ring slot's address is the ring's base or-ed with the slot's byte offset.
__host__ __device__ constexpr int density_ring_offset(int W, int ngroups, int ring)
{
    return (ngroups * (W * W + 1) * 8 + ring * 4 - 1) / (ring * 4) * (ring * 4);
}
__host__ __device__ constexpr int density_lds_bytes(int W, int ngroups, int ring)
{
    return density_ring_offset(W, ngroups, ring) + ngroups * ring * 4;
}

// Where list positions c0 .. c0+15 (c0 a multiple of 16) of a particle go: its
// list of cap entries, then the group's pool chunk of ocap entries, claimed by
// the first call past cap (one 64-bit atomic; none left: null, the claim
// failure is counted and the force pass walks the stencil).  Called by all G
// lanes of the group; lane l == 0 is lane gfirst of the wave.
struct ListOut {
    uint32_t* nbl;
    uint32_t cap, pb = ~0u;  // pb: the group's chunk in the pool (none yet)
    bool claimed = false;    // the group asked for a chunk (at most once)
    __device__ __forceinline__ uint32_t* chunk(const DevState& D, uint32_t c0, int l, int gfirst)
    {
        if (c0 < cap) return nbl + c0;
        const uint32_t ocap = (uint32_t)D.ocap;
        if (!claimed) {
            claimed = true;
            uint32_t b0 = ~0u;
            if (l == 0) {
                const unsigned long long t = atomicAdd(D.ptop, (unsigned long long)ocap);
                b0 = t + ocap <= (unsigned long long)D.pool_cap ? (uint32_t)(t / SPHE_POOL_UNIT) : ~0u;
                if (b0 == ~0u) atomicAdd(&D.ovf[1], 1u);
            }
            pb = __shfl(b0, gfirst, SPHE_WAVE);
        }
        return pb != ~0u && c0 - cap < ocap ? D.pool + (size_t)pb * SPHE_POOL_UNIT + (c0 - cap) : nullptr;
    }
};

// The end of the density pass: the largest count past the lists (one atomic
// per wave: the lanes still here; the loop over the overflowing groups is
// wave-uniform), then lane 0 of the group writes the particle's outputs.
template <typename T>
__device__ __forceinline__ void density_out(const DevState& D, const SceneConsts<T>& K, int64_t slot, int l,
                                            const V4<T>& pi, T sum, uint32_t cnt, uint32_t cap, uint32_t pb)
{
    uint64_t over = __ballot(cnt > cap);
    if (over) {
        uint32_t mx = 0;
        for (; over; over &= over - 1) {
            const uint32_t c = (uint32_t)__shfl(cnt, __ffsll((unsigned long long)over) - 1, SPHE_WAVE);
            mx = c > mx ? c : mx;
        }
        const uint64_t here = __ballot(1);
        if ((int)(threadIdx.x & (SPHE_WAVE - 1)) == __ffsll((unsigned long long)here) - 1) atomicMax(D.ovf, mx);
    }
    if (l != 0) return;
    D.nbc[slot] = cnt;
    D.pbase[slot] = pb;
    const T rho = sum * K.mc6;
    const T p = K.k * (rho - K.rho0);
    ((T*)D.rho)[slot] = rho;
    // (x, y, z, p / rho^2) and vel.w = m / rho: what the force pass gathers
    // per neighbour, in two 16-byte loads
    V4<T> pa = pi;
    pa.w = p / (rho * rho);
    ((V4<T>*)D.posa)[slot] = pa;
    ((T*)D.s_vel)[4 * slot + 3] = K.mass / rho;
}

// One G-lane group per particle (lane l = thread index mod G).  The clipped
// stencil rows form one stream of candidates; lane l takes stream positions
// l, l+G, ... (U = SPHE_DENSITY_UNROLL per iteration) for its share of the
// density sum.
// The group writes one neighbour list per particle (self left out) in
// canonical order, in chunks of 16 entries from nbl[slot * maxn] on, count in
// nbc[slot]; a byte-wise prefix sum over the group places each lane's entries
// in a ring in LDS, and every completed chunk goes out with one 16-byte store
// per lane (64-byte aligned: one cache line per group).  A chunk is stored by
// the lane that will read it: its entry e = l + G u lies at word l (16 / G)
// + u, so a force lane takes its four neighbours of an iteration
// with one 16-byte load.  List
// entries are byte offsets of the neighbours' slots in the per-slot vectors
// of V4<T> (slot * sizeof(V4<T>), below 2^32 by the layout's limits).  The
// group then merges the partial sums and lane 0 writes rho and
// (p / rho^2, m / rho).
template <typename T, int SM, int G>
__device__ __forceinline__ void density_body(const DevState& D, int b)
{
    const int64_t gt = (int64_t)b * blockDim.x + threadIdx.x;
    const int64_t slot = gt / G;
    const int l = (int)(gt & (G - 1));
    if (slot >= D.P) return;
    const SceneDev& S = scene_ref(D, wave_scene(D.chunk_scene, slot));
    if (slot >= S.p_begin + S.n) return;  // whole groups leave together
    const SceneConsts<T>& K = SceneSel<T>::get(S);
    const V4<T>* __restrict__ pos = (const V4<T>*)D.s_pos;
    const V4<T> pi = pos[slot];
    Acc<T, SM != SUM_PLAIN> sum;
    const T h2 = K.h2, thr = K.thr;
    const uint32_t cap = (uint32_t)D.maxn;
    ListOut out{D.nbl + slot * (int64_t)D.maxn, cap};
    constexpr uint32_t VB = (uint32_t)sizeof(V4<T>);  // bytes per slot of a V4<T> vector
    const uint32_t self = (uint32_t)slot * VB;          // as a byte offset
    const int gfirst = (int)(threadIdx.x & (SPHE_WAVE - 1)) & ~(G - 1);  // the group's first lane in the wave
    uint32_t cnt = 0;      // the same in every lane of the group
    uint32_t stream_total = 0;
    // The particle's clipped rows as one stream of candidates, t = 0 ..
    // total-1 in canonical order.  Lane l computes rows l, l+G, ... (the
    // group takes G rows per round) and writes (stream end, slot offset),
    // both in bytes (times VB), to the group's row table in LDS (dynamic:
    // blockDim / G tables of W^2 + 1 entries, then the groups' rings, laid
    // out by density_ring_offset): positions t of row r lie below
    // its end and hold slot t + offset.  A group prefix sum per round gives
    // the stream ends.  Entry W^2 is a sentinel row that ends at 2^32 - 1,
    // so a walk along the table stops by itself.
    const int yz = D.yz, W = 2 * yz + 1, nrows = W * W;
    extern __shared__ __attribute__((aligned(256))) uint2 rowtab[];
    constexpr int RING = SPHE_DENSITY_UNROLL * G > 16 ? 64 : 32;  // list staging ring (entries)
    constexpr uint32_t RMASK = RING * 4 - 1;                       // byte offset in a ring
    const int grp = (int)(threadIdx.x / G);
    uint2* __restrict__ tab = rowtab + grp * (nrows + 1);
    // the group's ring, size-aligned: slot offset ring_rel | (4 * position
    // mod RING) in the array; the hot stores use the LDS byte address
    // ring_abs | ..., the same with the array's own (256-byte aligned) address
    const uint32_t ring_rel = (uint32_t)(density_ring_offset(W, (int)(blockDim.x / G), RING) + grp * RING * 4);
    const uint32_t ring_abs = (uint32_t)(uintptr_t)rowtab + ring_rel;
    {
        const RowProbe<T> P = row_probe<T>(D, S, K, pi.x, pi.y, pi.z);
        uint32_t ends = 0;  // stream end of the rounds so far (all lanes)
        // row r = W dz + dy (dz, dy from 0): lane l starts at row l and steps
        // by G, carrying dz, dy and the row's cell offset (no multiplies)
        const int nx = S.dims[0], nyx = S.dims[1] * nx;
        int dz = row_div(l, W), dy = l - dz * W;
        uint32_t roff = (uint32_t)((dz - yz) * nyx + (dy - yz) * nx);
        const int rounds = (nrows + G - 1) / G;
        for (int k = 0, r = l; k < rounds; ++k, r += G) {
            uint32_t j0 = 0, len = 0;
            if (r < nrows) {
                uint32_t j1 = 0;
                const bool on = row_range<T>(D, S, P, dy - yz, dz - yz, roff, j0, j1);
                len = on && j1 > j0 ? j1 - j0 : 0u;
            }
            uint32_t rtot;
            const uint32_t end = ends + group_prefix<G>(len, l, &rtot);
            if (r < nrows) tab[r] = make_uint2(end * VB, (j0 - (end - len)) * VB);
            ends += rtot;
            dy += G;
            roff += (uint32_t)(G * nx);
            while (dy >= W) {
                dy -= W;
                ++dz;
                roff += (uint32_t)(nyx - W * nx);
            }
        }
        if (l == 0) tab[nrows] = make_uint2(~0u, 0u);
        // the group's lanes are one wave's: order its LDS writes before the reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        stream_total = ends;
    }
    // Lane l takes stream positions l, l+G, ... (U = SPHE_DENSITY_UNROLL
    // per iteration, blocks of U*G positions); its row pointer cur advances
    // through the table as its position passes each row's end (the sentinel
    // row ends every walk).  Positions, row ends and slots are in bytes
    // (times VB).  Blocks wholly inside the stream need no position checks;
    // in the last, partial block the positions past the stream load the
    // particle itself and take nothing.
    {
        constexpr int U = SPHE_DENSITY_UNROLL;
        const uint32_t total = stream_total;
        const uint2* cur = tab - 1;         // the current row's entry (none yet)
        uint32_t cur_end = 0, cur_off = 0;  // its stream end and slot offset
        const uint32_t lane_b = (uint32_t)l * VB;
        // Writes the chunk of 16 list positions from c0 (a multiple of 16) on
        // from the ring: lane l copies positions c0 + l, c0 + l + G, ... to
        // words l PER .. of the chunk, with 16-byte (G = 8: 8-byte) stores.  Of
        // the last, partial chunk the words past the count are written with
        // whatever the ring holds and never read.  The list rows and pool
        // chunks are 64-byte aligned.  Called by all lanes of the group.
        auto flush = [&](uint32_t c0) {
            constexpr int PER = 16 / G;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            uint32_t* dst = out.chunk(D, c0, l, gfirst);
            if (dst) {
                const uint32_t* src = (const uint32_t*)((char*)rowtab + (ring_rel | ((c0 * 4u) & RMASK))) + l;
                dst += l * PER;
                if constexpr (PER >= 4) {
#pragma unroll
                    for (int k = 0; k < PER; k += 4)
                        *(uint4*)(dst + k) =
                            make_uint4(src[k * G], src[(k + 1) * G], src[(k + 2) * G], src[(k + 3) * G]);
                } else {
                    *(uint2*)dst = make_uint2(src[0], src[G]);
                }
            }
            // the ring slots read here are written again only by later blocks
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        };
        auto block = [&](uint32_t base, auto tail) {
            constexpr bool TAIL = decltype(tail)::value;
            uint32_t jj[U];
            bool ok[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t t = base + (uint32_t)(u * G + l);
                const uint32_t tb = base * VB + (uint32_t)(u * G) * VB + lane_b;
                while (tb >= cur_end) {
                    const uint2 e = *++cur;
                    cur_end = e.x;
                    cur_off = e.y;
                }
                ok[u] = TAIL ? t < total : true;
                jj[u] = ok[u] ? tb + cur_off : self;
            }
            T d2[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const V4<T> p = at_byte(pos, jj[u]);
                const T dx = pi.x - p.x, dy = pi.y - p.y, dz = pi.z - p.z;
                d2[u] = (dx * dx + dy * dy) + dz * dz;
            }
            // The lane's U terms (0 for a candidate outside the radius or
            // past the stream) are added in plain arithmetic, u = 0 first,
            // and the block's partial enters the lane's sum.  Outside the
            // radius the term is 0 without a test: d2 > thr >= h2 gives
            // q = 0 (h2 = fl(h h) <= thr since fl(sqrt(fl(h h))) = h).
            // byte u of x: 1 if this lane lists its u-th candidate
            uint32_t x = 0;
            T part = T(0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const bool in = ok[u] & (d2[u] <= thr);
                T q = h2 - d2[u];
                q = q > T(0) ? q : T(0);
                const T w = ok[u] ? (q * q) * q : T(0);
                part = u ? part + w : w;
                // the force pass adds the particle's own term first: self is not listed
                x |= (uint32_t)(in & (jj[u] != self)) << (8 * u);
            }
            sum.add(part);
            // canonical place of the lane's u-th candidate (position u*G + l
            // of the block): the block's listed candidates at u' < u (all
            // lanes), then those of lanes below l at u.  Byte-wise sums over
            // the group (each byte stays <= 4 G, no carries): excl = lanes
            // below l, tot = all lanes; byte u of place is the sum of tot's
            // bytes below u plus excl's byte u.  sad_u8 adds tot's four bytes.
            uint32_t tot;
            const uint32_t excl = group_prefix<G>(x, l, &tot) - x;
            const uint32_t place = excl + (byte_runs(tot) << 8);
            const uint32_t ncnt = __builtin_amdgcn_sad_u8(tot, 0u, cnt);
            // the entries go to the group's ring in LDS (list position mod
            // RING, as byte offsets: place's bytes stay below 64, so times 4
            // they do not carry); each completed chunk of 16 is written out
            // at once
            const uint32_t place4 = place << 2, cnt4 = cnt << 2;
#pragma unroll
            for (int u = 0; u < U; ++u)
                if ((x >> (8 * u)) & 1u)
                    *(lds_u32*)(uintptr_t)(ring_abs | ((cnt4 + ((place4 >> (8 * u)) & 0xFFu)) & RMASK)) = jj[u];
            // chunks completed by this block: from the one holding position
            // cnt (one at most when a block holds 16 positions or fewer)
            if constexpr (U * G <= 16) {
                const uint32_t c0 = cnt & ~15u;
                if (c0 + 16u <= ncnt) flush(c0);
            } else {
                for (uint32_t c0 = cnt & ~15u; c0 + 16u <= ncnt; c0 += 16u) flush(c0);
            }
            cnt = ncnt;
        };
        uint32_t base = 0;
        for (; base + U * G <= total; base += U * G) block(base, std::false_type());
        if (base < total) block(base, std::true_type());
        if (cnt & 15u) flush(cnt & ~15u);  // the last, partial chunk
    }
    group_merge<G>(sum);
    density_out<T>(D, K, slot, l, pi, sum.value(), cnt, cap, out.pb);
}

template <typename T, int SM, int G>
__global__ __launch_bounds__(512) void k_density(DevState D, int nblk, int remap)
{
    density_body<T, SM, G>(D, xcd_block(blockIdx.x, nblk, remap));
}

// The density pass for four lanes a particle and cubic or halved cells (YZ =
// 1 or 2): the same streams, sums and lists as density_body, bit for bit, in
// two thirds to nine tenths of its time: 18.0 -> 10.5 us on a dam break of
// 4,096 particles, 88.5 -> 66 us on a settled column of 262,144, 162 -> 143 us
// on 48 settled scenes of 879,000 in all (cubic cells), 1,443 -> 1,273 us on a
// settled layer of 4,194,304.  density_body serves the other lane counts,
// thirds of cells and the persistent launch.
//
// Measured rates here (cycles a wave64 instruction a SIMD): plain FP32 and
// integer adds, multiplies, logic and right shifts on VGPRs or literals 2.4;
// min / max, compares, selects, bit counts, DPP, conversions, anything with
// an SGPR operand 4.4.  The pass is bound by issue, so:
// * Rows are set up plane by plane: lane l takes the rows dy = l - YZ of each
//   plane, whose y gap is the lane's own constant and whose z gap the plane's,
//   with the fifth row of each plane (YZ = 2) in the lanes of two more rounds.
//   A row or plane outside the grid has gap 2 (out of reach).  Two loads of
//   cell records a row.
// * The table of the rows that hold candidates has the offset from stream
//   position to slot and the first position of each; a bit per stream position
//   marks where a row starts.  A block's row of position p is then a bit count
//   of the block's marks up to p, with no walk along the table and no chain
//   of LDS reads.  The marks cover a segment of SPHE_SEG positions and are
//   set again from the table for each further segment.
// * A candidate's place in the list is a bit count of the block's accepted
//   positions up to it (the quad's 16 bits or-ed together with two DPP ors).
//   The entries are staged in a 32-word buffer that is moved down by 16 words
//   when its first chunk is written out, so a place is one shift and add.
// * The particle's own slot is looked for only in blocks where a group of the
//   wave has its own.
// * The accept masks stay in scalar registers (ballots): as booleans over the
//   branch around the own-slot test they became a byte per lane, 16 more
//   instructions a block.
// * Six waves a SIMD (80 registers): with 72 or 64 the loop spills (1,449 and
//   1,886 us on the layer).
// UNIT: every smoothing length is at most 1, so h^2 - d2 can be clamped to
// [0, 1] by the subtraction's own modifier instead of a max.
#define SPHE_SEG 256  // 6.4 KB of LDS a wave with 5x5 rows: no limit to six waves a SIMD
constexpr int QUAD_STAGE = 128;                 // bytes of a group's staging buffer
constexpr int QUAD_MARKS = SPHE_SEG / 8 + 16;   // marks (and the prefetch past them)
__host__ __device__ constexpr int quad_group_bytes(int yz)
{
    // 16 bytes more than needed: a stride of 100 or 68 words puts the same
    // word of a wave's 16 groups in different banks
    return QUAD_STAGE + QUAD_MARKS + ((2 * yz + 1) * (2 * yz + 1) * 8 + 15) / 16 * 16 + 16;
}

typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
template <typename P>
__device__ __forceinline__ P* lds_at(uint32_t addr) { return (P*)(uintptr_t)addr; }

// A uniform value in a VGPR: an operand that costs the full-rate form.
__device__ __forceinline__ float in_vgpr(float x) { asm volatile("" : "+v"(x)); return x; }
__device__ __forceinline__ double in_vgpr(double x) { asm volatile("" : "+v"(x)); return x; }

template <int CTRL>
__device__ __forceinline__ uint32_t quad_dpp(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, true);
}
// sum of x over the lanes of the quad up to this one (m1, m2: all ones in
// lanes 1.. and 2..), and the quad's total
__device__ __forceinline__ uint32_t quad_prefix(uint32_t x, uint32_t m1, uint32_t m2, uint32_t* tot)
{
    uint32_t y = x + (quad_dpp<0x90>(x) & m1);  // quad_perm [0,0,1,2]
    y += quad_dpp<0x40>(y) & m2;                // quad_perm [0,0,0,1]
    *tot = quad_dpp<0xFF>(y);                   // quad_perm [3,3,3,3]
    return y;
}

// max(x, 0); UNIT: x <= 1, as the clamp of the instruction that makes x
template <bool UNIT>
__device__ __forceinline__ float pos_part(float x)
{
    return UNIT ? __builtin_amdgcn_fmed3f(x, 0.f, 1.f) : (x > 0.f ? x : 0.f);
}
template <bool UNIT>
__device__ __forceinline__ double pos_part(double x) { return x > 0.0 ? x : 0.0; }

// floor(x) clamped to [lo, hi] (exact integers below 2^24), NaN giving lo
__device__ __forceinline__ int floor_clamp(float x, float lo, float hi)
{
    return (int)__builtin_amdgcn_fmed3f(__builtin_floorf(x), lo, hi);
}
__device__ __forceinline__ int floor_clamp(double x, double lo, double hi)
{
    return (int)d_fmin(d_fmax(d_floor(x), lo), hi);
}

// The half-width of a row plus its margin, times the slab count s (a power of
// two, so every step is RowWidth's scaled exactly): s (width(x) + margin).
__device__ __forceinline__ float row_width(float x, float s, float s15, float sm)
{
    float y = __int_as_float(0x5f375a86 - (__float_as_int(x) >> 1));
    const float t = ((0.5f * x) * s) * y;
    y = y * __builtin_fmaf(-t, y, s15);
    return x * y + sm;
}
__device__ __forceinline__ double row_width(double x, double s, double, double sm) { return d_sqrt(x) * s + sm; }

// Orders the wave's LDS accesses before against those after (the lanes of a
// group are one wave's, and a wave's LDS accesses are done in order).
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T, int SM, int YZ, bool UNIT>
__device__ __forceinline__ void density_quad(const DevState& D, int b)
{
    constexpr int W = 2 * YZ + 1;
    constexpr uint32_t VB = (uint32_t)sizeof(V4<T>);
    const int l = (int)(threadIdx.x & 3);
    const int lane = (int)(threadIdx.x & (SPHE_WAVE - 1));
    // the wave's first slot (slots are below 2^30; P is a multiple of 64, so
    // waves are whole)
    const uint32_t wslot = wave_index(b) * 16u;
    if (wslot >= (uint64_t)D.P) return;
    const uint32_t slot = wslot + (uint32_t)(lane >> 2);
    const SceneDev& S = scene_ref(D, wave_scene(D.chunk_scene, wslot));
    const uint32_t lo = (uint32_t)S.p_begin, hi = (uint32_t)(S.p_begin + S.n);
    if (wslot >= hi) return;  // only padding
    const SceneConsts<T>& K = SceneSel<T>::get(S);
    const V4<T>* __restrict__ pos = (const V4<T>*)D.s_pos;
    const uint32_t self = slot * VB;
    const uint32_t cap = (uint32_t)D.maxn;
    ListOut out{D.nbl + slot * (int64_t)D.maxn, cap};
    const int gfirst = lane & ~3;
    const uint32_t m1 = l >= 1 ? ~0u : 0u, m2 = l >= 2 ? ~0u : 0u;

    // the group's LDS: staging buffer, marks, row table
    extern __shared__ __attribute__((aligned(256))) uint2 rowtab[];
    constexpr uint32_t GB = (uint32_t)quad_group_bytes(YZ);
    const uint32_t stage = (uint32_t)(uintptr_t)rowtab + (threadIdx.x >> 2) * GB;
    const uint32_t marks = stage + QUAD_STAGE;
    const uint32_t tab = marks + QUAD_MARKS;

    // positions p = 4 u + l of a block, u = 0..3: the bits up to p
    uint32_t upto[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) upto[u] = (2u << (4 * u + l)) - 1u;

    Acc<T, SM != SUM_PLAIN> sum;
    const T h2 = in_vgpr(K.h2);
    const T thr = K.thr;
    uint32_t rows = 0;     // marks before the current block: rows started
    uint32_t placed = ~0u; // entries in the staging buffer, less 1
    uint32_t done = 0;     // entries written out
    uint32_t total = 0;    // candidates of the stream
    uint32_t selfpos = 0;  // this lane's stream position of the particle itself (~0: another lane's)

    // Sets the mark of stream position p of the segment.
    auto mark = [&](uint32_t p) {
        if (p < SPHE_SEG)
            (void)__hip_atomic_fetch_or(lds_at<lds_u32>(marks + (p >> 5) * 4u), 1u << (p & 31u), __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_WAVEFRONT);
    };
    auto clear_marks = [&]() {
        *lds_at<lds_u32x2>(marks + 8u * (uint32_t)l) = u32x2{0u, 0u};
        static_assert(SPHE_SEG / 8 == 32, "one 8-byte store a lane");
        wave_order();
    };
    // The clipped rows: a table of those that hold candidates, and the marks of
    // the first segment.
    // The rows' slot ranges are found with the lanes laid out by quarters of
    // the wave: lane 16 qr + g does rows of particle g, so that 16 lanes in a
    // row read cell records of neighbouring cells (a load of a wave touches a
    // few lines instead of 64; the L1 does one line access a cycle, and the
    // pass is close to that limit).  They go through the table's memory to the
    // quads.
    uint32_t nrows;
    {
        const int qr = lane >> 4;
        const int nx = S.dims[0], ny = S.dims[1], nz = S.dims[2], nyx = ny * nx;
        const int sl = D.sub_log2, smax = (1 << sl) - 1;
        const T s = T(1 << sl), q = K.yz_scale;
        const V4<T> pr = pos[wslot + (lane & 15)];
        const T gx = (pr.x - K.org[0]) * K.inv_cell;
        const T gy = (pr.y - K.org[1]) * K.inv_yz, gz = (pr.z - K.org[2]) * K.inv_yz;
        const int kx = cidx<T>(d_floor(gx), nx - 1);
        const int ky = cidx<T>(d_floor(gy), ny - 1);
        const int kz = cidx<T>(d_floor(gz), nz - 1);
        const uint32_t rbase = (uint32_t)S.cell_off + (uint32_t)((kz * ny + ky) * nx);
        const T fy = gy - T(ky), fz = gz - T(kz);
        // squared gap to the rows or planes d cells away; out of the grid: 4
        auto gap2 = [&](T f, int k, int n, int d) {
            if (d == 0) return T(0);
            const T g = row_gap<T>((d == -1 ? f : d == 1 ? T(1) - f : d == -2 ? T(1) + f : T(1) + (T(1) - f)) * q);
            return (d < 0 ? k >= -d : k + d < n) ? g * g : T(4);
        };
        T mz[W];
#pragma unroll
        for (int k = 0; k < W; ++k) mz[k] = gap2(fz, kz, nz, k - YZ);
        // the lane's rows dy = qr - YZ (YZ = 1: quarter 3 has none)
        T my = gap2(fy, ky, ny, -YZ);
        if (qr == 1) my = gap2(fy, ky, ny, 1 - YZ);
        if (qr == 2) my = gap2(fy, ky, ny, 2 - YZ);
        if (qr == 3) my = YZ == 1 ? T(4) : gap2(fy, ky, ny, 1);
        const uint32_t rlane = rbase + (uint32_t)((qr - YZ) * nx);
        const T gs = gx * s, s15 = T(1.5) * s, sm = T(SPHE_ROW_MARGIN) * s;
        // slabs of the cells kx - 1 .. kx + 1 inside the grid
        const T flo_min = T((kx > 0 ? kx - 1 : 0) << sl), fmax = T((nx << sl) - 1);
        const T fhi_max = T(((kx < nx - 1 ? kx + 1 : nx - 1) << sl) + smax);
        // offset shifts by the low two bits of a slab index, from byte tables:
        // 10 (slab - 1) for the first slab taken (30, an empty field, for slab
        // 0), 10 slab for the last
        const uint32_t tlo = sl == 2 ? 0x140A001Eu : (sl == 1 ? 0x001E001Eu : 0x1E1E1E1Eu);
        const uint32_t thi = sl == 2 ? 0x1E140A00u : (sl == 1 ? 0x1E001E00u : 0x1E1E1E1Eu);
        const uint32_t raw = (uint32_t)(uintptr_t)rowtab + ((threadIdx.x >> 2 & ~15u) + (uint32_t)(lane & 15)) * GB +
                             QUAD_STAGE + QUAD_MARKS;  // the table of the lane's particle here
        auto row = [&](int at, T r2, uint32_t cell) {
            const bool on = r2 <= T(1);
            const T w = row_width(T(1) - r2, s, s15, sm);
            const int flo = floor_clamp(gs - w, flo_min, fmax), fhi = floor_clamp(gs + w, T(0), fhi_max);
            const uint32_t rk = on ? cell : rbase;
            const uint2* clo = D.cells + (rk + (uint32_t)(flo >> sl));
            const uint2* chi = D.cells + (rk + (uint32_t)(fhi >> sl));
            const uint2 a = clo[0], c = chi[0];
            const uint32_t c1 = chi[1].x;
            const uint32_t slo = tlo >> (((uint32_t)flo << 3) & 31u), shi = thi >> (((uint32_t)fhi << 3) & 31u);
            const uint32_t first = a.x + __builtin_amdgcn_ubfe(a.y & 0x3FFFFFFFu, slo, 10);
            const bool whole = (fhi & smax) == smax || (int32_t)c.y < 0;
            const uint32_t last = c.x + __builtin_amdgcn_ubfe(c.y, shi, 10);
            const uint32_t e = min(whole ? c1 : last, hi);
            const uint32_t j = max(first, lo);
            *lds_at<lds_u32x2>(raw + 8u * (uint32_t)at) = u32x2{j, on && e > j ? e - j : 0u};
        };
#pragma unroll
        for (int k = 0; k < W; ++k) {
            if (qr < W) row(k * W + qr, my + mz[k], rlane + (uint32_t)((k - YZ) * nyx));
            if (k == 3) __builtin_amdgcn_sched_barrier(0);  // four rows' loads in flight: fewer registers
        }
        if constexpr (YZ == 2) {
            const T m5 = gap2(fy, ky, ny, 2);
            row(qr * W + 4, m5 + (qr == 0 ? mz[0] : qr == 1 ? mz[1] : qr == 2 ? mz[2] : mz[3]),
                rbase + (uint32_t)((qr - 2) * nyx + 2 * nx));
            if (qr == 0) row(4 * W + 4, m5 + mz[4], rbase + (uint32_t)(2 * nyx + 2 * nx));
        }
    }
    if (slot >= hi) return;  // padding: whole groups leave together
    const V4<T> pi = pos[slot];
    {
        // A stream that ends with a segment is looked up once more, past its end
        // and past the marks: none there, so that look-up stays at the last row.
        *lds_at<lds_u32>(marks + SPHE_SEG / 8 + 4u * (uint32_t)l) = 0u;
        static_assert(QUAD_MARKS == SPHE_SEG / 8 + 16, "one 4-byte store a lane");
        clear_marks();
        constexpr int NR = YZ == 1 ? 3 : 7;  // the planes' rows l, then the fifth rows
        uint32_t j0[NR], len[NR];
        auto take = [&](int k, bool have, int at) {
            const u32x2 e = *lds_at<lds_u32x2>(tab + 8u * (uint32_t)at);
            j0[k] = e.x;
            len[k] = have ? e.y : 0u;
        };
#pragma unroll
        for (int k = 0; k < W; ++k) take(k, l < W, k * W + (l < W ? l : 0));
        if constexpr (YZ == 2) {
            take(5, true, l * W + 4);
            take(6, l == 0, 4 * W + 4);
        }
        wave_order();
        // place of each row that holds candidates among them: 6-bit fields, one
        // a plane, of the lane's own rows; prefixes over the quad, then planes
        uint32_t has = 0, fifth = 0;
#pragma unroll
        for (int k = 0; k < W; ++k) has |= (len[k] != 0u ? 1u : 0u) << (6 * k);
        uint32_t htot;
        uint32_t place = quad_prefix(has, m1, m2, &htot) - has;
        if constexpr (YZ == 2) {
            const uint32_t f5 = len[5] != 0u ? 1u : 0u, f6 = len[6] != 0u ? 1u : 0u;
            fifth = quad_dpp<0x00>(f5) | quad_dpp<0x55>(f5) << 6 | quad_dpp<0xAA>(f5) << 12 |
                    quad_dpp<0xFF>(f5) << 18 | quad_dpp<0x00>(f6) << 24;
        }
        // rows of the planes before: running sums of the planes' totals
        const uint32_t before = ((htot + fifth) * 0x01041041u) << 6;
        place += before;
        nrows = ((before + htot + fifth) >> (6 * (W - 1))) & 63u;
        // stream starts, the table and the marks
        uint32_t ends = 0, s5 = 0, p5 = 0;
        auto put = [&](uint32_t at, uint32_t start, int k) {
            if (len[k] == 0u) return;
            *lds_at<lds_u32x2>(tab + 8u * at) = u32x2{start, (j0[k] - start) * VB};
            mark(start);
        };
#pragma unroll
        for (int k = 0; k < W; ++k) {
            uint32_t tot;
            const uint32_t st = ends + quad_prefix(len[k], m1, m2, &tot) - len[k];
            if (k == YZ)  // the particle's own row: dy = 0 is lane YZ's
                selfpos = quad_dpp<YZ * 0x55>(slot - j0[k] + st);
            put((place >> (6 * k)) & 63u, st, k);
            ends += tot;
            if constexpr (YZ == 2) {
                const uint32_t at5 = ((before + htot) >> (6 * k)) & 63u;
                const uint32_t l5 = k == 0   ? quad_dpp<0x00>(len[5])
                                    : k == 1 ? quad_dpp<0x55>(len[5])
                                    : k == 2 ? quad_dpp<0xAA>(len[5])
                                    : k == 3 ? quad_dpp<0xFF>(len[5])
                                             : quad_dpp<0x00>(len[6]);
                if (k < 4) {
                    if (l == k) {
                        s5 = ends;
                        p5 = at5;
                    }
                } else if (l == 0) {
                    put(at5, ends, 6);
                }
                ends += l5;
            }
        }
        if constexpr (YZ == 2) put(p5, s5, 5);
        selfpos = (selfpos & 3u) == (uint32_t)l ? selfpos : ~0u;
        total = ends;
        wave_order();
    }

    // Writes the first 16 staged entries out, lane l its entries l, l + 4, ...
    // with one 16-byte store, and moves the rest down.
    auto flush = [&]() {
        wave_order();
        const uint32_t at = stage + 4u * (uint32_t)l;
        const u32x4 e = {*lds_at<lds_u32>(at), *lds_at<lds_u32>(at + 16u), *lds_at<lds_u32>(at + 32u),
                         *lds_at<lds_u32>(at + 48u)};
        const u32x4 rest = *lds_at<lds_u32x4>(stage + 64u + 16u * (uint32_t)l);
        wave_order();
        *lds_at<lds_u32x4>(stage + 16u * (uint32_t)l) = rest;
        uint32_t* dst = out.chunk(D, done, l, gfirst);
        if (dst) *(u32x4*)(dst + 4 * l) = e;
        done += 16u;
        placed -= 16u;
        wave_order();
    };

    // The slots of the block at t (positions t + 4 u + l), looked up while the
    // block before is computed; a new segment's marks are set from the table
    // first.  Past the stream's end they are slots of its last row or beyond.
    uint32_t t = 0, jn[4];
    uint32_t mk = *lds_at<lds_u16>(marks), mnext = marks + 2u;
    auto lookup = [&](uint32_t at) {
        if (at != 0u && at % SPHE_SEG == 0u && at < total) {
            wave_order();
            clear_marks();
            for (uint32_t r = (uint32_t)l; r < nrows; r += 4u) mark(*lds_at<lds_u32>(tab + 8u * r) - at);
            wave_order();
            mk = *lds_at<lds_u16>(marks);
            mnext = marks + 2u;
        }
        const uint32_t m = mk;
        mk = *lds_at<lds_u16>(mnext);
        mnext += 2u;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t r = (uint32_t)__popc(m & upto[u]) + rows;      // rows started up to the position
            const uint32_t off = *lds_at<lds_u32>((r << 3) + (tab - 4u));  // row r - 1's
            jn[u] = off + (at * VB + (uint32_t)l * VB) + (uint32_t)(4 * u) * VB;
        }
        rows += (uint32_t)__popc(m);
    };
    auto block = [&](auto tail) {
        constexpr bool TAIL = decltype(tail)::value;
        uint32_t jj[4];
        V4<T> p[4];
        uint64_t ok[4];  // lanes with a candidate
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            jj[u] = jn[u];
            if constexpr (TAIL) {
                ok[u] = __builtin_amdgcn_ballot_w64(t + (uint32_t)(4 * u + l) < total);
                jj[u] = __builtin_amdgcn_inverse_ballot_w64(ok[u]) ? jj[u] : self;
            }
            p[u] = at_byte(pos, jj[u]);
        }
        if constexpr (!TAIL) lookup(t + 16u);
        T part = T(0);
        uint64_t in[4];  // lanes whose candidate is inside the radius
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const T dx = pi.x - p[u].x, dy = pi.y - p[u].y, dz = pi.z - p[u].z;
            const T d2 = (dx * dx + dy * dy) + dz * dz;
            in[u] = __builtin_amdgcn_ballot_w64(d2 <= thr);
            const T q = pos_part<UNIT>(h2 - d2);
            T w = (q * q) * q;
            if constexpr (TAIL) {
                in[u] &= ok[u];
                w = __builtin_amdgcn_inverse_ballot_w64(ok[u]) ? w : T(0);
            }
            part = u ? part + w : w;
        }
        sum.add(part);
        // the particle itself is not listed
        const uint32_t ds = selfpos - t;  // 4 u + l where it is this lane's
        if (__builtin_amdgcn_ballot_w64(ds < 16u)) {
#pragma unroll
            for (int u = 0; u < 4; ++u) in[u] &= __builtin_amdgcn_ballot_w64(ds != (uint32_t)(4 * u + l));
        }
        uint32_t acc = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) acc |= __builtin_amdgcn_inverse_ballot_w64(in[u]) ? 1u << (4 * u) : 0u;
        acc <<= l;
        acc |= quad_dpp<0xB1>(acc);  // quad_perm [1,0,3,2]
        acc |= quad_dpp<0x4E>(acc);  // quad_perm [2,3,0,1]
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t at = (uint32_t)__popc(acc & upto[u]) + placed;
            if (__builtin_amdgcn_inverse_ballot_w64(in[u])) *lds_at<lds_u32>(stage + (at << 2)) = jj[u];
        }
        placed += (uint32_t)__popc(acc);
        if ((int32_t)placed >= 15) flush();
    };
    if (total != 0u) lookup(0u);
    for (; t + 16u <= total; t += 16u) block(std::false_type());
    if (t < total) block(std::true_type());
    if ((int32_t)placed >= 0) {
        const uint32_t left = placed + 1u;
        flush();
        done = done - 16u + left;
    }
    group_merge<4>(sum);
    density_out<T>(D, K, slot, l, pi, sum.value(), done, cap, out.pb);
}

template <typename T, int SM, int YZ, bool UNIT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 6 : 4, 8))) void k_density_quad(
    DevState D, int nblk, int remap)
{
    density_quad<T, SM, YZ, UNIT>(D, xcd_block(blockIdx.x, nblk, remap));
}

// ----------------------------------------------------------------- force

template <typename T>
struct ForceOut {
    T pf[3], vf[3], nr[3], sf[3], gf[3], acc[3];
    int32_t nbmax;
    int32_t count;
};

// The terms one neighbour j != i adds to the ten force sums: pressure,
// viscosity, colour normal and colour Laplacian (fluid_system.h:136-150,
// 165-172) with the constants factored out.
// r = |d| and 1/r from d2 = |d|^2 (fluid_system.h:118, 438-441: length and
// normalize).  FP64: correctly rounded sqrt and division.  FP32: 1/sqrt by
// three Newton steps y <- y (1.5 - (d2/2) y^2) from the integer estimate
// 0x5f375a86 - bits(d2)/2 (relative error 3.4e-2 -> 1.8e-3 -> 4.6e-6 ->
// FP32 rounding), each step one multiply, one fused multiply-add and one
// multiply; r = d2 / sqrt(d2) = d2 y.  Within a few ulp of the correctly
// rounded values and made only of IEEE operations, so a CPU replays it bit
// for bit; it replaces two correctly rounded sequences of about ten
// instructions each.  d2 = 0 gives r = 0 (the coincident-pair branch).
template <typename T> struct Root {
    static __device__ __forceinline__ void of(T d2, T& r, T& inv)
    {
        r = d_sqrt(d2);
        inv = T(1) / r;
    }
};
template <> struct Root<float> {
    static __device__ __forceinline__ void of(float d2, float& r, float& inv)
    {
        float y = __int_as_float(0x5f375a86 - (__float_as_int(d2) >> 1));
        const float hx = 0.5f * d2;
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const float t = hx * y;
            y = y * __builtin_fmaf(-t, y, 1.5f);
        }
        inv = y;
        r = d2 * y;
    }
};

template <typename T> struct Terms {
    T lap, fp0, fp1, fp2, fv0, fv1, fv2, nn0, nn1, nn2;
};

// a + b, term by term (plain arithmetic)
template <typename T>
__device__ __forceinline__ Terms<T> terms_sum(const Terms<T>& a, const Terms<T>& b)
{
    Terms<T> t;
    t.lap = a.lap + b.lap;
    t.fp0 = a.fp0 + b.fp0; t.fp1 = a.fp1 + b.fp1; t.fp2 = a.fp2 + b.fp2;
    t.fv0 = a.fv0 + b.fv0; t.fv1 = a.fv1 + b.fv1; t.fv2 = a.fv2 + b.fv2;
    t.nn0 = a.nn0 + b.nn0; t.nn1 = a.nn1 + b.nn1; t.nn2 = a.nn2 + b.nn2;
    return t;
}

// The constants of the pair terms.
template <typename T>
struct PairConsts {
    T h, h2, t3h2, eps_r, inv_sqrt3;
};

template <bool UNIT, typename T>
__device__ __forceinline__ Terms<T> pair_terms(const PairConsts<T>& K, T dx, T dy, T dz, T d2, T a_i, T a_j,
                                               T b_j, const V4<T>& vi, const V4<T>& vj)
{
    Terms<T> t;
    const T q = pos_part<UNIT>(K.h2 - d2);
    t.lap = b_j * (q * (K.t3h2 - T(7) * d2));
    T r, inv;
    Root<T>::of(d2, r, inv);
    const T hr = K.h - r;
    T ux = dx * inv, uy = dy * inv, uz = dz * inv;
    // coincident pair: the reference points along normalize(1,1,1)
    // (fluid_system.h:438-440); the reciprocal is discarded then.  Rare: the
    // selects run only where a lane of the wave has one (the empty asm keeps
    // the compiler from making them unconditional).
    const bool near = r < K.eps_r;
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(near) != 0ull, 0)) {
        asm volatile("");
        ux = near ? K.inv_sqrt3 : ux;
        uy = near ? K.inv_sqrt3 : uy;
        uz = near ? K.inv_sqrt3 : uz;
    }
    const T sp = (a_i + a_j) * (hr * hr);
    t.fp0 = sp * ux;
    t.fp1 = sp * uy;
    t.fp2 = sp * uz;
    const T wv = b_j * hr;
    t.fv0 = (vj.x - vi.x) * wv;
    t.fv1 = (vj.y - vi.y) * wv;
    t.fv2 = (vj.z - vi.z) * wv;
    const T wn = b_j * (q * q);
    t.nn0 = dx * wn;
    t.nn1 = dy * wn;
    t.nn2 = dz * wn;
    return t;
}

// Force sums of one lane.  A lane's neighbours enter in consecutive groups
// of four, added in plain arithmetic as (a + b) + (c + d) before the group
// enters the lane's sum; the last one to three enter as a pair (a + b) and
// then a single.
// finish() applies the constants and forms the acceleration
// (fluid_system.h:151-154, 163, 177, 318-321).
// The force sums' accumulator: plain, Kahan-compensated, or (FP32 terms)
// FP64 sums (two instructions per term instead of the four of a
// compensated add) rounded to FP32 once.
template <typename T, int SM> struct ForceAccSel { typedef Acc<T, SM != SUM_PLAIN> type; };
template <> struct ForceAccSel<float, SUM_F64ACC> { typedef AccF64 type; };

template <typename T, int SM>
struct ForceAcc {
    typename ForceAccSel<T, SM>::type fp0, fp1, fp2, fv0, fv1, fv2, nn0, nn1, nn2, lap;

    // The particle's own colour-Laplacian term (d = 0): added first, by lane 0.
    __device__ __forceinline__ void self_term(const SceneConsts<T>& K, T b_i)
    {
        lap.add(b_i * (K.h2 * K.t3h2));
    }

    __device__ __forceinline__ void add(const Terms<T>& t)
    {
        lap.add(t.lap);
        fp0.add(t.fp0); fp1.add(t.fp1); fp2.add(t.fp2);
        fv0.add(t.fv0); fv1.add(t.fv1); fv2.add(t.fv2);
        nn0.add(t.nn0); nn1.add(t.nn1); nn2.add(t.nn2);
    }

    // four consecutive terms as two plain pair sums ab = a + b, cd = c + d:
    // ab + cd enters the sums
    __device__ __forceinline__ void add4(const Terms<T>& ab, const Terms<T>& cd)
    {
        lap.add(ab.lap + cd.lap);
        fp0.add(ab.fp0 + cd.fp0); fp1.add(ab.fp1 + cd.fp1); fp2.add(ab.fp2 + cd.fp2);
        fv0.add(ab.fv0 + cd.fv0); fv1.add(ab.fv1 + cd.fv1); fv2.add(ab.fv2 + cd.fv2);
        nn0.add(ab.nn0 + cd.nn0); nn1.add(ab.nn1 + cd.nn1); nn2.add(ab.nn2 + cd.nn2);
    }

    template <int G>
    __device__ __forceinline__ void merge()
    {
        group_merge<G>(fp0); group_merge<G>(fp1); group_merge<G>(fp2);
        group_merge<G>(fv0); group_merge<G>(fv1); group_merge<G>(fv2);
        group_merge<G>(nn0); group_merge<G>(nn1); group_merge<G>(nn2);
        group_merge<G>(lap);
    }

    __device__ __forceinline__ void finish(const SceneConsts<T>& K, T rho_i, ForceOut<T>& o) const
    {
        const T sPF = K.pf_scale * rho_i;
        o.pf[0] = fp0.value() * sPF; o.pf[1] = fp1.value() * sPF; o.pf[2] = fp2.value() * sPF;
        o.vf[0] = fv0.value() * K.vf_scale; o.vf[1] = fv1.value() * K.vf_scale; o.vf[2] = fv2.value() * K.vf_scale;
        o.nr[0] = nn0.value() * K.ng; o.nr[1] = nn1.value() * K.ng; o.nr[2] = nn2.value() * K.ng;
        const T lapv = lap.value() * K.ng;
        const T ss = (-K.surf_tens) * lapv;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            o.sf[a] = o.nr[a] * ss;
            o.gf[a] = rho_i * K.g[a];
            const T F = (o.pf[a] + o.vf[a]) + (o.gf[a] + o.sf[a]);
            o.acc[a] = F / rho_i;
        }
    }
};

// Lane l's share of the force sums of one particle by walking its clipped
// stencil rows (inspection, and particles whose list overflowed): every lane
// visits all candidates in canonical order and takes the accepted
// neighbours m = l, l+G, l+2G, ... (self excluded), as it would from the
// list.  count and nbmax cover the lane's share (self counted by lane 0).
template <typename T, int SM, int G>
__device__ __forceinline__ void force_share_walk(const DevState& D, const SceneDev& S, const SceneConsts<T>& K,
                                                 int64_t slot, int l, const V4<T>& pi, const V4<T>& vi, T a_i,
                                                 ForceAcc<T, SM>& acc, int32_t& nbmax, int32_t& count)
{
    const V4<T>* __restrict__ pos = (const V4<T>*)D.s_pos;
    const V4<T>* __restrict__ posa = (const V4<T>*)D.posa;
    const V4<T>* __restrict__ vel = (const V4<T>*)D.s_vel;
    // the start of a group of four a, b, c, d: ab = a (+ b), c
    Terms<T> ab, c;
    int np = 0;  // terms of the group so far
    uint32_t m = 0;    // canonical index of the next accepted neighbour
    const PairConsts<T> C{K.h, K.h2, K.t3h2, K.eps_r, K.inv_sqrt3};
    if (l == 0) ++count;  // the particle itself
    visit_neighbours<T>(D, S, K, pos, pi.x, pi.y, pi.z, [&](uint32_t j, T dx, T dy, T dz, T d2) {
        if ((int64_t)j == slot) return;  // own term: ForceAcc::self_term
        const bool mine = (m & (G - 1)) == (uint32_t)l;
        ++m;
        if (!mine) return;
        ++count;
        const int32_t idj = D.s_id[j];
        nbmax = idj > nbmax ? idj : nbmax;
        const V4<T> vj = at(vel, j);
        const Terms<T> t = pair_terms<false, T>(C, dx, dy, dz, d2, a_i, at(posa, j).w, vj.w, vi, vj);
        if (np == 0) ab = t;
        else if (np == 1) ab = terms_sum(ab, t);
        else if (np == 2) c = t;
        else acc.add4(ab, terms_sum(c, t));
        np = (np + 1) & 3;
    });
    // the lane's last one to three terms: a, or the pair a + b (then c)
    if (np != 0) acc.add(ab);
    if (np == 3) acc.add(c);
}

// Dominant-axis box response (fluid_system.h:342-347 with collisionS
// :355-407), generalised to a cube of centre c and half extent e.
template <typename T>
__device__ __forceinline__ void box_response(const SceneConsts<T>& K, T* p, T* v)
{
    if ((K.box_lo[0] < p[0] && p[0] < K.box_hi[0]) && (K.box_lo[1] < p[1] && p[1] < K.box_hi[1]) &&
        (K.box_lo[2] < p[2] && p[2] < K.box_hi[2]))
        return;
    int ax = 0;
    T maxP = d_fabs(p[0] - K.box_c[0]);
    const T u1 = d_fabs(p[1] - K.box_c[1]);
    if (maxP < u1) { ax = 1; maxP = u1; }
    const T u2 = d_fabs(p[2] - K.box_c[2]);
    if (maxP < u2) { ax = 2; maxP = u2; }
    T cp[3] = {p[0], p[1], p[2]};
    T nr[3] = {T(0), T(0), T(0)};
    if (p[ax] < K.box_lo[ax]) { cp[ax] = K.box_lo[ax]; nr[ax] = T(1); }
    else { cp[ax] = K.box_hi[ax]; nr[ax] = T(-1); }
    const T d0 = p[0] - cp[0], d1 = p[1] - cp[1], d2 = p[2] - cp[2];
    const T d = d_sqrt((d0 * d0 + d1 * d1) + d2 * d2);
    const T vl = d_sqrt((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]);
    const T s = T(1) + (T(0.5) * d) / (K.dt * vl);
    const T vn = (v[0] * nr[0] + v[1] * nr[1]) + v[2] * nr[2];
#pragma unroll
    for (int a = 0; a < 3; ++a) v[a] = v[a] - (nr[a] * s) * vn;
    p[0] = cp[0]; p[1] = cp[1]; p[2] = cp[2];
}

// Bilinear height of the cell-centred terrain at (x, z) and the unit normal
// of that patch (library-defined).
template <typename T>
__device__ __forceinline__ T terrain_sample(const SceneDev& S, const SceneConsts<T>& K, const float* __restrict__ H,
                                            T x, T z, T* nrm)
{
    const int tnx = S.tnx, tnz = S.tnz;
    const T u = (x - K.t_org[0]) * K.t_inv - T(0.5);
    const T w = (z - K.t_org[2]) * K.t_inv - T(0.5);
    const int i0 = cidx<T>(d_floor(u), tnx > 1 ? tnx - 2 : 0);
    const int k0 = cidx<T>(d_floor(w), tnz > 1 ? tnz - 2 : 0);
    const int i1 = tnx > 1 ? i0 + 1 : i0;
    const int k1 = tnz > 1 ? k0 + 1 : k0;
    T fu = u - T(i0), fw = w - T(k0);
    fu = fu > T(0) ? fu : T(0);
    fu = fu < T(1) ? fu : T(1);
    fw = fw > T(0) ? fw : T(0);
    fw = fw < T(1) ? fw : T(1);
    if (tnx == 1) fu = T(0);
    if (tnz == 1) fw = T(0);
    const float* Hs = H + S.t_off;
    const T h00 = (T)Hs[k0 * tnx + i0], h10 = (T)Hs[k0 * tnx + i1];
    const T h01 = (T)Hs[k1 * tnx + i0], h11 = (T)Hs[k1 * tnx + i1];
    const T gu = T(1) - fu, gw = T(1) - fw;
    const T a0 = gu * h00 + fu * h10;
    const T a1 = gu * h01 + fu * h11;
    const T hs = gw * a0 + fw * a1;
    const T dhu = gw * (h10 - h00) + fw * (h11 - h01);
    const T dhw = gu * (h01 - h00) + fu * (h11 - h10);
    const T gx = dhu * K.t_inv, gz = dhw * K.t_inv;
    const T nn = (gx * gx + T(1)) + gz * gz;
    const T inv = T(1) / d_sqrt(nn);
    nrm[0] = -gx * inv;
    nrm[1] = inv;
    nrm[2] = -gz * inv;
    return hs;
}

// Heightfield collision: projection onto the surface with the reference's
// response term (fluid_system.h:344-346) while moving into the terrain.
template <typename T>
__device__ __forceinline__ void terrain_collide(const SceneConsts<T>& K, T hs, const T* nr, T* p, T* v)
{
    if (!(p[1] < hs)) return;
    const T d = hs - p[1];
    const T vn = (v[0] * nr[0] + v[1] * nr[1]) + v[2] * nr[2];
    if (vn < T(0)) {
        const T vl = d_sqrt((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]);
        const T s = T(1) + (T(0.5) * d) / (K.dt * vl);
#pragma unroll
        for (int a = 0; a < 3; ++a) v[a] = v[a] - (nr[a] * s) * vn;
    }
    p[1] = hs;
}

// Erosion / deposition exchange of one particle (library-defined).  Returns
// the fixed-point amount taken from terrain cell *tc (negative: deposited),
// or 0 with *tc = -1 outside the contact band.
template <typename T>
__device__ __forceinline__ int64_t erode_exchange(const SceneDev& S, const SceneConsts<T>& K, const T* p, T hs,
                                                  const T* v, int64_t sed, int32_t* tc)
{
    *tc = -1;
    const T gap = p[1] - hs;
    if (!(gap <= K.band)) return 0;
    const int ti = cidx<T>(d_floor((p[0] - K.t_org[0]) * K.t_inv), S.tnx - 1);
    const int tk = cidx<T>(d_floor((p[2] - K.t_org[2]) * K.t_inv), S.tnz - 1);
    *tc = tk * S.tnx + ti;
    const T sp = d_sqrt((v[0] * v[0] + v[1] * v[1]) + v[2] * v[2]);
    const T cap = K.kcv * sp;
    const T s = (T)sed * K.dn;
    T d;
    if (cap > s) d = K.ke * (cap - s);
    else d = -(K.kd * (s - cap));
    // one exchange saturates at 2^52 units (NaN: none), far inside int64
    if (!(d_fabs(d) <= K.dmax)) d = d > T(0) ? K.dmax : (d < T(0) ? -K.dmax : T(0));
    int64_t dq = (int64_t)d_rint(d * K.up);
    if (dq < -sed) dq = -sed;
    return dq;
}

// Lane l's share of the force sums from list entries l, l+G, l+2G, ... of
// a particle's neighbour sequence: the lanes of a particle differ by one
// neighbour at most.  An entry is the byte offset of the neighbour's slot in
// the V4<T> vectors; fetch(more) gives the lane's next four (mine in all).
// Four neighbours per iteration (eight gathers in flight), summed
// (a + b) + (c + d) before they enter the lane's sums; then one pair, then a
// single.
//
// No unit is saturated: on a settled 4.2M-particle layer (1,437 us with the list
// laid out entry by entry, 1,230 now) the gathers' line accesses take 55% of the L1's cycles, the VALU is
// busy for half the time, the lists come from HBM, and 20 waves a CU wait for
// each other.  So waves in flight count most: five a SIMD, 96 registers, with
// nothing spilled on the way through the loop.  What lies behind that:
// * a wave's list read touches 16 lines, one per group, however few bytes a lane
//   takes: the four entries of an iteration come with one 16-byte load;
// * one loop for lists with and without an overflow chunk (a wave with one
//   overflowing particle ran both loops: 90 -> 70 us on a column of 262,144
//   with lists of 256 entries);
// * values that the epilogue or the rare paths make from the thread index are
//   made again there (opaque_tid): kept over the loop they were spilled by
//   every wave, 0.6 GB a launch;
// * coincident pairs' selects behind a branch that is hardly ever taken.
// Eight gathers in flight with five waves beat four gathers with six or
// seven, a pair ahead with four waves, and lists two iterations ahead.
template <bool UNIT, typename T, int SM, int G, typename F>
__device__ __forceinline__ void force_list(const DevState& D, const SceneConsts<T>& K, uint32_t mine, const V4<T>& pi,
                                           const V4<T>& vi, T a_i, ForceAcc<T, SM>& acc, uint4 n, F&& fetch)
{
    if (mine == 0u) return;
    const V4<T>* __restrict__ posa = (const V4<T>*)D.posa;
    const V4<T>* __restrict__ vel = (const V4<T>*)D.s_vel;
    const PairConsts<T> C{K.h, K.h2, K.t3h2, K.eps_r, K.inv_sqrt3};
    struct Nb { V4<T> p, v; };
    auto load = [&](uint32_t j) { return Nb{at_byte(posa, j), at_byte(vel, j)}; };
    auto terms = [&](const Nb& b) {
        const T dx = pi.x - b.p.x, dy = pi.y - b.p.y, dz = pi.z - b.p.z;
        const T d2 = (dx * dx + dy * dy) + dz * dz;
        return pair_terms<UNIT, T>(C, dx, dy, dz, d2, a_i, b.p.w, b.v.w, vi, b.v);
    };
    // The list entries of the next iteration load while the current one
    // computes: always, and after the gathers, whose waits then leave that load
    // in flight (memory operations complete in order; a load that may or may
    // not have been issued would have to be waited for).
    for (; mine >= 4u; mine -= 4u) {
        const Nb a = load(n.x), b = load(n.y), c = load(n.z), d = load(n.w);
        __builtin_amdgcn_sched_barrier(0);
        n = fetch(mine > 8u);
        __builtin_amdgcn_sched_barrier(0);
        const Terms<T> ab = terms_sum(terms(a), terms(b));
        acc.add4(ab, terms_sum(terms(c), terms(d)));
    }
    // the lane's last one to three neighbours: a pair, then a single
    if (mine >= 2u) {
        const Nb a = load(n.x), b = load(n.y);
        acc.add(terms_sum(terms(a), terms(b)));
        n.x = n.z;
    }
    if (mine & 1u) acc.add(terms(load(n.x)));
}

// The thread index as a value the compiler knows nothing of: what is made of
// it is not kept in registers from an earlier use of the index (over the list
// loop, a register more is a spill).
__device__ __forceinline__ uint32_t opaque_tid()
{
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// The start of a particle's list, loaded ahead of what it depends on: the
// number of entries and (four lanes a particle) the lane's first four, which
// may be anything where there are fewer.
struct ListHead {
    uint32_t cnt;
    uint4 first;
};
template <int G>
__device__ __forceinline__ ListHead list_head(const DevState& D, uint32_t slot, uint32_t l)
{
    ListHead h;
    h.cnt = D.nbc[slot];
    h.first = make_uint4(0u, 0u, 0u, 0u);
    if constexpr (G == 4) h.first = *(const uint4*)(D.nbl + (size_t)slot * (uint32_t)D.maxn + l * (16 / G));
    return h;
}

// Lane l's share of the force sums of one particle: from its list, the
// list continued in its overflow chunk, or (no room for all neighbours)
// by walking the stencil.  wslot: the wave's first slot.
template <bool UNIT, typename T, int SM, int G>
__device__ __forceinline__ void force_share(const DevState& D, const SceneDev& S, const SceneConsts<T>& K,
                                           const ListHead& head, uint32_t slot, uint32_t wslot, int l,
                                           const V4<T>& pi, const V4<T>& vi, T a_i, ForceAcc<T, SM>& acc,
                                           bool report_walk)
{
    constexpr uint32_t PER = 16 / G;
    const uint32_t cnt = head.cnt;
    const uint32_t cap = (uint32_t)D.maxn;
    if (cnt <= cap || (cnt - cap <= (uint32_t)D.ocap && D.pbase[slot] != ~0u)) {
        // the lane's entries l, l + G, ... are words l PER .. of each chunk of
        // 16; e: the first entry of the next iteration's 4G (uniform, since the
        // lanes go through their lists in step).  fetch(more) gives the entries
        // of this iteration, again if it was told there are no more.
        const uint32_t mine = (cnt + (uint32_t)(G - 1 - l)) / G;
        const uint32_t* list = D.nbl + (size_t)slot * cap + (uint32_t)l * PER;
        auto pool = [&]() {
            const uint32_t t = opaque_tid();
            return D.pool + (size_t)D.pbase[wslot + (t & (SPHE_WAVE - 1)) / G] * SPHE_POOL_UNIT + (t & (G - 1)) * PER;
        };
        uint32_t e = 0;
        if constexpr (G == 4) {
            auto advance = [&](bool more) {
                e += 16u;
                if (__builtin_expect(e == cap, 0)) {
                    if (more) list = pool();
                } else {
                    list += more ? 16 : 0;
                }
            };
            advance(mine > 4u);
            force_list<UNIT, T, SM, G>(D, K, mine, pi, vi, a_i, acc, head.first, [&](bool more) {
                const uint4 n = *(const uint4*)list;
                advance(more);
                return n;
            });
        } else {
            auto chunk = [&](uint32_t c) { return c < cap ? list + c : pool() + (c - cap); };
            auto fetch = [&](bool more) {
                uint4 n;
                if constexpr (G < 4) {
                    n = *(const uint4*)(chunk(e & ~15u) + (e & 15u) / G);
                } else {
                    const uint2 a = *(const uint2*)chunk(e);
                    uint2 b = a;
                    if (e + 16u < cnt) b = *(const uint2*)chunk(e + 16u);
                    n = make_uint4(a.x, a.y, b.x, b.y);
                }
                if (more) e += 4 * G;
                return n;
            };
            if (mine != 0u) force_list<UNIT, T, SM, G>(D, K, mine, pi, vi, a_i, acc, fetch(mine > 4u), fetch);
        }
        return;
    }
    // no room in list and pool: the stencil again (same order, same result)
    const uint32_t t = opaque_tid();
    l = (int)(t & (G - 1));
    if (report_walk && l == 0) atomicOr(D.status, 4u);
    int32_t nbmax = -1, count = 0;
    force_share_walk<T, SM, G>(D, S, K, wslot + (t & (SPHE_WAVE - 1)) / G, l, pi, vi, a_i, acc, nbmax, count);
}

// Copies the list-overflow words (largest overflowing count, failed pool
// claims) and the pool entries the density pass claimed, all final once it is
// done, into host memory mapped for the device (vector stores), where the host
// reads them between step sequences without waiting for the stream.
__device__ __forceinline__ void publish(const DevState& D)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const unsigned long long t = *D.ptop;
    volatile uint32_t* d = D.pub;
    d[0] = D.ovf[0];
    d[1] = D.ovf[1];
    d[2] = (uint32_t)t;
    d[3] = (uint32_t)(t >> 32);
}

// One G-lane group per particle: the lanes sum their shares, merge them
// (xor shuffles), and lane 0 integrates, collides, erodes, stores the new
// state and counts the particle's next cell.
// Outside the list loop a wave does little but wait, so what can be loaded
// together is: all that the slot alone addresses before the scene is looked up
// (the scene's padding goes through as particles without neighbours: a branch
// there would hold the loads back), the epilogue's inputs before the merge, and
// the cell count, whose answer the wave's last store waits for, before the
// other stores (batches of 48 uneven scenes: 203 -> 150 us in all, 262,144
// particles 65.5 -> 56.5, 4.2M 1,337 -> 1,230, with constant_table and one-wave
// blocks).
template <bool UNIT, typename T, int SM, int G>
__device__ __forceinline__ void force_body(const DevState& D, int b)
{
    const int l = (int)(threadIdx.x & (G - 1));
    // the wave's first slot (slots are below 2^30; P is a multiple of 64, so
    // waves are whole)
    const uint32_t wslot = wave_index(b) * (uint32_t)(SPHE_WAVE / G);
    if (wslot >= (uint64_t)D.P) return;
    const uint32_t slot0 = wslot + (uint32_t)(threadIdx.x & (SPHE_WAVE - 1)) / G;
    V4<T>* __restrict__ upos = (V4<T>*)D.u_pos;
    V4<T>* __restrict__ uvel = (V4<T>*)D.u_vel;
    const V4<T>* __restrict__ spos = (const V4<T>*)D.s_pos;
    const V4<T>* __restrict__ svel = (const V4<T>*)D.s_vel;
    // all that is loaded by the slot, before the scene is known
    ListHead head = list_head<G>(D, slot0, (uint32_t)l);
    const V4<T> pi = spos[slot0];
    const V4<T> vi = svel[slot0];
    const T a_i = ((const V4<T>*)D.posa)[slot0].w;
    const SceneDev& S = scene_ref(D, wave_scene(D.chunk_scene, wslot));
    const uint32_t end = (uint32_t)(S.p_begin + S.n);
    if (slot0 >= end) head.cnt = 0u;  // padding: no neighbours
    const SceneConsts<T>& K = SceneSel<T>::get(S);
    ForceAcc<T, SM> acc;
    if (l == 0) acc.self_term(K, vi.w);
    force_share<UNIT, T, SM, G>(D, S, K, head, slot0, wslot, l, pi, vi, a_i, acc, true);
    // what the epilogue needs, while the lanes' sums are merged
    const uint32_t tid = opaque_tid();
    const uint32_t slot = wslot + (tid & (SPHE_WAVE - 1)) / G;
    const T rho_i = ((const T*)D.rho)[slot];
    int64_t sed = D.s_sed[slot];
    const int32_t id = D.s_id[slot];
    acc.template merge<G>();
    if ((tid & (G - 1)) != 0) return;
    if (slot >= end) {
        // padding: carried through, counted into the scene's pad cell
        upos[slot] = spos[slot];
        uvel[slot] = svel[slot];
        D.u_sed[slot] = sed;
        D.u_id[slot] = id;
        count_pad(D, S, slot);
        // kept apart from the end of the function, where the rank's wait would
        // otherwise become one for every store
        asm volatile("");
        return;
    }
    ForceOut<T> o;
    acc.finish(K, rho_i, o);

    // symplectic Euler (fluid_system.h:330-331)
    T p[3], v[3];
    const T xin[3] = {pi.x, pi.y, pi.z}, vin[3] = {vi.x, vi.y, vi.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        v[a] = vin[a] + o.acc[a] * K.dt;
        p[a] = xin[a] + v[a] * K.dt;
    }
    const bool moving = K.dt != T(0);
    if (moving) box_response<T>(K, p, v);
    int32_t tc = -1;
    int64_t dq = 0;
    if (S.tnx > 0) {
        T nr[3];
        const T hs = terrain_sample<T>(S, K, D.height, p[0], p[2], nr);
        if (moving) {
            terrain_collide<T>(K, hs, nr, p, v);
            if (S.erosion) dq = erode_exchange<T>(S, K, p, hs, v, sed, &tc);
        }
    }
    // the cell count of the new position for the next step's sort: its answer
    // comes while the state is stored
    const int32_t key = position_key<T>(D, S, K, p[0], p[1], p[2]);
    const uint32_t rank = count_key(D, key);
    if (dq != 0) {  // atomic erosion: into the volume; two-phase: into the cell's sum of this step
        sed += dq;
        atomicAdd((unsigned long long*)(S.erosion == 2 ? D.tsum : D.vol) + (S.t_off + tc), (unsigned long long)(-dq));
    }
    V4<T> np, nv;
    np.x = p[0]; np.y = p[1]; np.z = p[2]; np.w = T(0);
    nv.x = v[0]; nv.y = v[1]; nv.z = v[2]; nv.w = T(0);
    upos[slot] = np;
    uvel[slot] = nv;
    D.u_sed[slot] = sed;
    D.u_id[slot] = id;
    if (!(d_finite(p[0]) && d_finite(p[1]) && d_finite(p[2]) && d_finite(v[0]) && d_finite(v[1]) &&
          d_finite(v[2])))
        atomicOr(D.status, 1u);
    D.key[slot] = key;
    D.arank[slot] = rank;
}

// FP32: at most 96 registers (5 waves per SIMD): the list loop fits, and
// only the rarely taken stencil walk of overflowing particles spills.
// Unbounded, the walk raises the count and the occupancy of the whole
// kernel drops to 4.
template <int SM, int G, bool UNIT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_force_f32(DevState D)
{
    force_body<UNIT, float, SM, G>(D, (int)blockIdx.x);
    publish(D);
}

// FP64: at most 168 registers (3 waves per SIMD instead of 2 unbounded).
template <int G>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_force_f64(DevState D)
{
    force_body<false, double, SUM_PLAIN, G>(D, (int)blockIdx.x);
    publish(D);
}

// ------------------------------------------------------ persistent passes

// Persistent form of the density and force passes: a grid of resident
// blocks takes the passes' blocks (work items, in the flattened slot order
// of all scenes) from eight queues, one per XCD: block p starts on queue
// p mod 8 (the XCD the hardware gives it), whose k-th item is the one the
// ordinary grid runs as block 8 k + x, remapped in runs of `chunk` as
// xcd_block does; a block whose queue is empty takes items from the other
// queues.  A block takes SPHE_GRAB consecutive items of a queue with one
// atomic and asks for the next ones while it works on them.  Every item is
// taken exactly once, and a block leaves when all eight queues are empty,
// so every wave exits.  The queues (work[0..7], in items) are cleared by
// k_work_reset before each launch.  The items of one block share no LDS
// between waves (each lane group has its own region), so one barrier per
// grab suffices.
#define SPHE_GRAB 4
__device__ __forceinline__ int64_t next_grab(uint32_t* work, int x, int nblk)
{
    for (int t = 0; t < 8; ++t) {
        const int q = (x + t) & 7;
        if ((int64_t)__hip_atomic_load(&work[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) * 8 + q >= nblk)
            continue;  // drained
        const int64_t bid = (int64_t)atomicAdd(&work[q], (uint32_t)SPHE_GRAB) * 8 + q;
        if (bid < nblk) return bid;
    }
    return -1;
}

__global__ void k_work_reset(uint32_t* work)
{
    if (threadIdx.x < 8) work[threadIdx.x] = 0u;
}

// g: the first item of a grab as an ordinary block index 8 k + q
#define SPHE_PERSISTENT_LOOP(BODY)                                                   \
    __shared__ int64_t s_grab[2];                                                    \
    const int x = (int)(blockIdx.x & 7u);                                            \
    if (threadIdx.x == 0) s_grab[0] = next_grab(work, x, nblk);                      \
    __syncthreads();                                                                 \
    int64_t g = s_grab[0];                                                           \
    for (int k = 0; g >= 0; ++k) {                                                   \
        const int64_t nxt = threadIdx.x == 0 ? next_grab(work, x, nblk) : -1;        \
        for (int i = 0; i < SPHE_GRAB; ++i) {                                        \
            const int64_t bid = g + 8 * i;                                           \
            if (bid >= nblk) break;                                                  \
            const int b = xcd_block((int)bid, nblk, chunk);                          \
            BODY;                                                                    \
        }                                                                            \
        if (threadIdx.x == 0) s_grab[(k + 1) & 1] = nxt;                             \
        __syncthreads();                                                             \
        g = s_grab[(k + 1) & 1];                                                     \
    }

template <typename T, int SM, int G>
__global__ __launch_bounds__(512) void k_density_pers(DevState D, int nblk, int chunk, uint32_t* work)
{
    SPHE_PERSISTENT_LOOP((density_body<T, SM, G>(D, b)))
}

template <int SM, int G>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_force_f32_pers(
    DevState D, int nblk, int chunk, uint32_t* work)
{
    SPHE_PERSISTENT_LOOP((force_body<false, float, SM, G>(D, b)))
    publish(D);
}

template <int G>
__global__ __launch_bounds__(512) void k_force_f64_pers(DevState D, int nblk, int chunk, uint32_t* work)
{
    SPHE_PERSISTENT_LOOP((force_body<false, double, SUM_PLAIN, G>(D, b)))
    publish(D);
}

// --------------------------------------------------------------- terrain

// Terrain heights from the fixed-point volumes, four consecutive cells per
// thread (16-byte loads and store).  A scene's range is padded to 64 cells,
// so the four cells share a scene; cells past the scene's nx * nz are
// padding and keep their value.
__device__ __forceinline__ void heights_quad(const DevState& D, int64_t t0)
{
    const SceneDev& S = D.scenes[D.tchunk_scene[t0 >> 6]];  // a wave's cells may belong to four scenes
    const int64_t end = S.t_off + (int64_t)S.tnx * S.tnz;
    const float y0 = S.t_y0, hq = S.hq;
    if (t0 + 4 <= end) {
        const longlong2 a = *(const longlong2*)(D.vol + t0);
        const longlong2 b = *(const longlong2*)(D.vol + t0 + 2);
        *(float4*)(D.height + t0) = make_float4(y0 + (float)a.x * hq, y0 + (float)a.y * hq,
                                                y0 + (float)b.x * hq, y0 + (float)b.y * hq);
    } else {
        for (int64_t t = t0; t < end; ++t) D.height[t] = y0 + (float)D.vol[t] * hq;
    }
}

__global__ __launch_bounds__(256) void k_heights(DevState D)
{
    const int64_t t0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (t0 < D.TC) heights_quad(D, t0);
}

// The particle scan's kernels.  Blocks past the nscan tiles of the last one
// launched (k_scan_cells) compute terrain heights: from the volumes the last
// force pass eroded, before this step's samples them.  first: the first step of
// a call, whose status word starts from 0 there (the scan's earlier launches set
// no bits; later kernels of the step do).
__device__ __forceinline__ bool heights_block(const DevState& D, int nscan)
{
    if ((int)blockIdx.x < nscan) return false;
    const int64_t t0 = ((int64_t)((int)blockIdx.x - nscan) * blockDim.x + threadIdx.x) * 4;
    if (t0 < D.TC) heights_quad(D, t0);
    return true;
}

// The totals of the marked tiles, where they were not counted with the
// particles.
template <int ITEMS>
__global__ __launch_bounds__(256) void k_scan_reduce_cells(DevState D)
{
    __shared__ uint32_t lds[4];
    uint32_t* const total = D.total + tile_word(D.tlog, blockIdx.x);
    if (*total == 0u) return;  // block-uniform; its writer is this block alone, after the barrier
    uint4 v[ITEMS / 4];
    load_tile<ITEMS>(D.cnt, (int64_t)blockIdx.x, D.C + 1, v);
    uint32_t s = 0;
#pragma unroll
    for (int c = 0; c < ITEMS / 4; ++c) s += (v[c].x + v[c].y) + (v[c].z + v[c].w);
    s = wave_total(s);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) *total = (lds[0] + lds[1]) + (lds[2] + lds[3]);
}

template <int ITEMS, int FROM>
__global__ __launch_bounds__(256) void k_scan_cells(DevState D, int nscan, int first)
{
    __shared__ uint32_t lds[8];
    if (first && blockIdx.x == 0 && threadIdx.x == 0) *D.status = 0u;
    if (heights_block(D, nscan)) return;  // block-uniform: no barrier is skipped by part of a block
    if (blockIdx.x == 0 && threadIdx.x == 0) *D.ptop = (unsigned long long)D.pool_origin;  // the pool's claims
    scan_down_tile<ITEMS, FROM>(D.cnt, D.cells, D.C + 1, D.total, D.tlog, D.tpre, D.tfill, (int)blockIdx.x, lds);
}

// Two-phase erosion, second phase: what the force pass summed up for each
// terrain cell (64-bit integers: any order gives the same sum) enters its
// volume, one read-modify-write a touched cell, and the sums are cleared.  Two
// cells a thread; bound by its launch up to some 10^6 cells.  (Sorting the
// particles' exchanges by cell, counted, scanned and scattered, and adding them
// cell by cell took five launches, 24 us of 165 for 185,193 particles over 512 x
// 512 cells; this takes 4.2.)
__global__ __launch_bounds__(256) void k_tapply(DevState D)
{
    const int64_t t = 2 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    if (t >= D.TC) return;  // TC is a multiple of 64
    const longlong2 q = *(const longlong2*)(D.tsum + t);
    if ((q.x | q.y) == 0) return;
    longlong2 v = *(const longlong2*)(D.vol + t);
    v.x += q.x;
    v.y += q.y;
    *(longlong2*)(D.vol + t) = v;
    *(longlong2*)(D.tsum + t) = make_longlong2(0, 0);
}

// ----------------------------------------------------------- inspection

// The record of one particle after a step: its group recomputes the force
// sums of that step (same lane split and merge as k_force) from the retained
// sorted state, and reads the state the step left in the same slot.  The
// slot comes from device memory (the id map or the id search; INT32_MAX or
// out of range: no such particle, out[22] = -1).  lists: the neighbour lists
// still hold the step's (else the stencil is walked: 22 us against 5.5 for 30
// neighbours, a chain of dependent loads either way).  One wave; out may be
// mapped host memory.
template <typename T, int SM, int G>
__global__ __launch_bounds__(64) void k_inspect(DevState D, const int32_t* __restrict__ slotp, int lists, double* out)
{
    if (blockIdx.x != 0) return;
    const int32_t s32 = *slotp;
    if (s32 < 0 || (int64_t)s32 >= D.P) {  // the same in every lane
        if (threadIdx.x == 0) out[22] = -1.0;
        return;
    }
    const int64_t slot = s32;
    const int l = (int)threadIdx.x;
    const SceneDev& S = scene_ref(D, wave_scene(D.chunk_scene, slot));
    const SceneConsts<T>& K = SceneSel<T>::get(S);
    const V4<T> pi = ((const V4<T>*)D.s_pos)[slot];
    const V4<T> vi = ((const V4<T>*)D.s_vel)[slot];
    const T rho_i = ((const T*)D.rho)[slot];
    const T a_i = ((const V4<T>*)D.posa)[slot].w;
    ForceAcc<T, SM> acc;
    int32_t nbmax = -1, count = 0;
    const uint32_t cnt = D.nbc[slot], cap = (uint32_t)D.maxn;
    const bool listed =
        lists && (cnt <= cap || (cnt - cap <= (uint32_t)D.ocap && D.pbase[slot] != ~0u));  // the same in every lane
    if (listed) {
        // the largest neighbour id by the whole wave
        const uint32_t* more = cnt > cap ? D.pool + (size_t)D.pbase[slot] * SPHE_POOL_UNIT : nullptr;
        for (uint32_t e = (uint32_t)l; e < cnt; e += SPHE_WAVE) {
            const uint32_t c = e & ~15u, word = (e % G) * (16 / G) + (e & 15u) / G;
            const uint32_t* q = c < cap ? D.nbl + (size_t)slot * cap + c : more + (c - cap);
            nbmax = max(nbmax, D.s_id[q[word] / (uint32_t)sizeof(V4<T>)]);
        }
#pragma unroll
        for (int m = 1; m < SPHE_WAVE; m <<= 1) nbmax = max(nbmax, __shfl_xor(nbmax, m, SPHE_WAVE));
        count = (int32_t)cnt + 1;
    }
    if (l >= G) return;
    if (l == 0) acc.self_term(K, vi.w);
    if (listed) {
        force_share<false, T, SM, G>(D, S, K, list_head<G>(D, (uint32_t)slot, (uint32_t)l), (uint32_t)slot,
                                     (uint32_t)slot, l, pi, vi, a_i, acc, false);
    } else {
        force_share_walk<T, SM, G>(D, S, K, slot, l, pi, vi, a_i, acc, nbmax, count);
#pragma unroll
        for (int m = 1; m < G; m <<= 1) {
            nbmax = max(nbmax, __shfl_xor(nbmax, m, SPHE_WAVE));
            count += __shfl_xor(count, m, SPHE_WAVE);
        }
    }
    acc.template merge<G>();
    if (l != 0) return;
    ForceOut<T> o;
    acc.finish(K, rho_i, o);
    o.nbmax = nbmax;
    o.count = count;
    out[0] = (double)rho_i;
    out[1] = (double)(K.k * (rho_i - K.rho0));
    for (int a = 0; a < 3; ++a) {
        out[2 + a] = (double)o.acc[a];
        out[5 + a] = (double)o.pf[a];
        out[8 + a] = (double)o.vf[a];
        out[11 + a] = (double)o.gf[a];
        out[14 + a] = (double)o.sf[a];
        out[17 + a] = (double)o.nr[a];
    }
    out[20] = (double)o.nbmax;
    out[21] = (double)o.count;
    out[22] = (double)slot;
    const V4<T> np = ((const V4<T>*)D.u_pos)[slot];
    const V4<T> nv = ((const V4<T>*)D.u_vel)[slot];
    out[23] = (double)np.x; out[24] = (double)np.y; out[25] = (double)np.z;
    out[26] = (double)nv.x; out[27] = (double)nv.y; out[28] = (double)nv.z;
}

__global__ __launch_bounds__(256) void k_fill_i32(int32_t* __restrict__ p, int64_t n, int32_t v)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// id -> slot of the current state, for the scenes with a map among those at
// slots p0 .. p1-1 (p0 a multiple of 64).  UNIQUE: every entry of the map
// belongs to one particle; otherwise the map was cleared to INT32_MAX first,
// and duplicate ids keep their lowest slot.
template <bool UNIQUE>
__global__ __launch_bounds__(256) void k_idmap(DevState D, int64_t p0, int64_t p1, int32_t* __restrict__ map)
{
    const int64_t slot = p0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= p1) return;
    const SceneDev& S = scene_ref(D, wave_scene(D.chunk_scene, slot));
    if (slot >= S.p_begin + S.n || S.idmap_off < 0) return;
    const int32_t id = D.u_id[slot];
    if (id < 0 || id >= S.idmap_len) return;
    if constexpr (UNIQUE) map[S.idmap_off + id] = (int32_t)slot;
    else atomicMin(&map[S.idmap_off + id], (int32_t)slot);
}

// Positions (what 0), velocities (1) or the last step's densities (2) of the
// n particles at slots p0 .. p0+n-1 in id order (the ids are 0 .. n-1): the
// current state lies at the last step's sorted slots with its ids in u_id.
// Each value is rounded to FP32 once, as the host copy rounds it.
template <typename T>
__global__ __launch_bounds__(256) void k_feed(DevState D, int64_t p0, int64_t n, int what, float* __restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t slot = p0 + i;
    const int32_t id = D.u_id[slot];
    if (id < 0 || (int64_t)id >= n) return;
    if (what == 2) {
        out[id] = (float)((const T*)D.rho)[slot];
        return;
    }
    const V4<T> v = ((const V4<T>*)(what ? D.u_vel : D.u_pos))[slot];
    float* o = out + 3 * (int64_t)id;
    o[0] = (float)v.x;
    o[1] = (float)v.y;
    o[2] = (float)v.z;
}

// The same values by the id map, for out in mapped host memory: one thread per
// value, so that every wave writes 256 consecutive bytes over the link (k_feed
// would send each value by itself).  1,000 positions 3.7 us, 13,824 5.1; with
// the map built by the first reader after a step (2.4 and 3.1), k_feed and the
// runtime's copy to pageable memory took some 17 us more for each read.
template <typename T>
__global__ __launch_bounds__(256) void k_gather(DevState D, const int32_t* __restrict__ map, int64_t n, int what,
                                                float* __restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = what == 2 ? (uint32_t)i : (uint32_t)i / 3u;
    const int32_t slot = map[p];
    if (slot < 0 || (int64_t)slot >= D.P) return;
    out[i] = (float)(what == 2 ? ((const T*)D.rho)[slot]
                               : ((const T*)(what ? D.u_vel : D.u_pos))[4 * (int64_t)slot + ((uint32_t)i - 3u * p)]);
}

// The sorted slot of particle `id` of one scene without a map (lowest slot
// for a duplicate id), into *slot_out (cleared to INT32_MAX first).
__global__ __launch_bounds__(256) void k_find_id(DevState D, int scene, int32_t id, int32_t* __restrict__ slot_out)
{
    const int64_t slot = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= D.P) return;
    const int si = wave_scene(D.chunk_scene, slot);
    if (si != scene) return;
    const SceneDev& S = D.scenes[si];
    if (slot < S.p_begin + S.n && D.s_id[slot] == id) atomicMin(slot_out, (int32_t)slot);
}

// Acceleration of every particle of one scene in the current sorted state
// (density pass done): the force pass's sums (list, pool or walk, the same
// order and lane split) and finish(), without integration.
// out[3 (slot - p_begin) + a], sorted order.
template <typename T, int SM, int G>
__global__ __launch_bounds__(256) void k_accel(DevState D, int scene, double* __restrict__ out)
{
    const int64_t gt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t slot = gt / G;
    const int l = (int)(gt & (G - 1));
    if (slot >= D.P) return;
    const int si = wave_scene(D.chunk_scene, slot);
    if (si != scene) return;
    const SceneDev& S = D.scenes[si];
    if (slot >= S.p_begin + S.n) return;  // whole groups leave together
    const SceneConsts<T>& K = SceneSel<T>::get(S);
    const V4<T> pi = ((const V4<T>*)D.s_pos)[slot];
    const V4<T> vi = ((const V4<T>*)D.s_vel)[slot];
    const T rho_i = ((const T*)D.rho)[slot];
    const T a_i = ((const V4<T>*)D.posa)[slot].w;
    ForceAcc<T, SM> acc;
    if (l == 0) acc.self_term(K, vi.w);
    force_share<false, T, SM, G>(D, S, K, list_head<G>(D, (uint32_t)slot, (uint32_t)l), (uint32_t)slot,
                                 wave_index((int)blockIdx.x) * (uint32_t)(SPHE_WAVE / G), l, pi,
                                  vi, a_i, acc, false);
    acc.template merge<G>();
    if (l != 0) return;
    ForceOut<T> o;
    acc.finish(K, rho_i, o);
#pragma unroll
    for (int a = 0; a < 3; ++a) out[3 * (slot - S.p_begin) + a] = (double)o.acc[a];
}

template <typename T>
__global__ __launch_bounds__(256) void k_neighbours(DevState D, int scene, const int64_t* __restrict__ off,
                                                    int32_t* __restrict__ counts, int32_t* __restrict__ idx)
{
    const int64_t slot = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= D.P) return;
    const int si = D.chunk_scene[slot >> 6];
    if (si != scene) return;
    const SceneDev& S = D.scenes[si];
    if (slot >= S.p_begin + S.n) return;
    const SceneConsts<T>& K = SceneSel<T>::get(S);
    const V4<T>* pos = (const V4<T>*)D.s_pos;
    const V4<T> pi = pos[slot];
    const int64_t local = slot - S.p_begin;
    int32_t c = 0;
    const int64_t o = idx ? off[local] : 0;
    visit_neighbours<T>(D, S, K, pos, pi.x, pi.y, pi.z,
                        [&](uint32_t j, T, T, T, T) {
                            if (idx) idx[o + c] = D.s_id[j];
                            ++c;
                        });
    counts[local] = c;
}

template <typename T>
__global__ __launch_bounds__(256) void k_keys(DevState D, int scene, int32_t* __restrict__ keys)
{
    const int64_t slot = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= D.P) return;
    const int si = D.chunk_scene[slot >> 6];
    if (si != scene) return;
    const SceneDev& S = D.scenes[si];
    if (slot >= S.p_begin + S.n) return;
    const SceneConsts<T>& K = SceneSel<T>::get(S);
    const V4<T> p = ((const V4<T>*)D.u_pos)[slot];
    int kx, ky, kz;
    cell_of<T>(K, S.dims, p.x, p.y, p.z, kx, ky, kz);
    keys[slot - S.p_begin] = (kz * S.dims[1] + ky) * S.dims[0] + kx;
}

// Grid::UpdateGrid's vertex stream (grid.h:138-176) of one scene's terrain,
// one thread per cell: the cell centre (org + (i + 0.5) cell), the height,
// and normalize(cross(u,l) + cross(u,r) + cross(d,l) + cross(d,r)) over the
// vectors to the edge neighbours present (normalize = v * (1 / |v|), as
// glm's; a zero sum gives a zero normal).
__global__ __launch_bounds__(256) void k_terrain_mesh(const float* __restrict__ H, int nx, int nz, float cell,
                                                      float ox, float oz, float* __restrict__ out)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)nx * nz) return;
    const int x = (int)(t % nx), z = (int)(t / nx);
    const float y = H[t];
    float u[3] = {0.f, 0.f, 0.f}, d[3] = {0.f, 0.f, 0.f}, r[3] = {0.f, 0.f, 0.f}, l[3] = {0.f, 0.f, 0.f};
    if (x - 1 >= 0) { l[0] = cell; l[1] = y - H[t - 1]; }
    if (x + 1 < nx) { r[0] = cell; r[1] = H[t + 1] - y; }
    if (z - 1 >= 0) { u[1] = y - H[t - nx]; u[2] = cell; }
    if (z + 1 < nz) { d[1] = H[t + nx] - y; d[2] = cell; }
    const float* A[4] = {u, u, d, d};
    const float* B[4] = {l, r, l, r};
    float n[3];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float* a = A[k];
        const float* b = B[k];
        const float c0 = a[1] * b[2] - a[2] * b[1];
        const float c1 = a[2] * b[0] - a[0] * b[2];
        const float c2 = a[0] * b[1] - a[1] * b[0];
        if (k == 0) { n[0] = c0; n[1] = c1; n[2] = c2; }
        else { n[0] = n[0] + c0; n[1] = n[1] + c1; n[2] = n[2] + c2; }
    }
    const float len = d_sqrt((n[0] * n[0] + n[1] * n[1]) + n[2] * n[2]);
    const float inv = len > 0.f ? 1.f / len : 0.f;
    float* o = out + 6 * t;
    o[0] = ox + ((float)x + 0.5f) * cell;
    o[1] = y;
    o[2] = oz + ((float)z + 0.5f) * cell;
    o[3] = n[0] * inv;
    o[4] = n[1] * inv;
    o[5] = n[2] * inv;
}

__global__ void k_clear_status(uint32_t* status)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *status = 0u;
}

// Mass bookkeeping of one scene: FP64 sums of terrain volume and carried
// sediment, and the exact mod-2^64 sum of their fixed-point units.  Each
// block writes its partial; k_mass_final adds them in block order.
__global__ __launch_bounds__(256) void k_mass_partial(DevState D, int scene, double* __restrict__ part)
{
    __shared__ double s_t[256];
    __shared__ double s_s[256];
    __shared__ unsigned long long s_u[256];
    const SceneDev& S = D.scenes[scene];
    const int64_t ncells = (int64_t)S.tnx * S.tnz;
    const double unit = ldexp(1.0, -S.fx_exp);
    double st = 0.0, ss = 0.0;
    unsigned long long su = 0ull;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < ncells; t += stride) {
        const int64_t v = D.vol[S.t_off + t];
        st += (double)v * unit;
        su += (unsigned long long)v;
    }
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < S.n; p += stride) {
        const int64_t v = D.u_sed[S.p_begin + p];
        ss += (double)v * unit;
        su += (unsigned long long)v;
    }
    s_t[threadIdx.x] = st;
    s_s[threadIdx.x] = ss;
    s_u[threadIdx.x] = su;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            s_t[threadIdx.x] += s_t[threadIdx.x + o];
            s_s[threadIdx.x] += s_s[threadIdx.x + o];
            s_u[threadIdx.x] += s_u[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[3 * blockIdx.x] = s_t[0];
        part[3 * blockIdx.x + 1] = s_s[0];
        part[3 * blockIdx.x + 2] = __longlong_as_double((long long)s_u[0]);
    }
}

// The same bookkeeping for every scene in one launch: block (b, s) takes
// cells and particles b, b + SPHE_MASS_BLOCKS_PER_SCENE blocks ... of scene
// s and writes its partial to part[3 (s B + b) ..]; k_mass_scenes_final adds
// a scene's B partials in block order.  Deterministic for a given layout.
// Every partial and result is written by each launch: the buffers need no
// clearing between calls.
__global__ __launch_bounds__(256) void k_mass_scenes(DevState D, double* __restrict__ part)
{
    __shared__ double s_t[256];
    __shared__ double s_s[256];
    __shared__ unsigned long long s_u[256];
    const int scene = (int)blockIdx.y;
    const SceneDev& S = D.scenes[scene];
    const int64_t ncells = (int64_t)S.tnx * S.tnz;
    const double unit = ldexp(1.0, -S.fx_exp);
    double st = 0.0, ss = 0.0;
    unsigned long long su = 0ull;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (int64_t t = first; t < ncells; t += stride) {
        const int64_t v = D.vol[S.t_off + t];
        st += (double)v * unit;
        su += (unsigned long long)v;
    }
    for (int64_t p = first; p < S.n; p += stride) {
        const int64_t v = D.u_sed[S.p_begin + p];
        ss += (double)v * unit;
        su += (unsigned long long)v;
    }
    s_t[threadIdx.x] = st;
    s_s[threadIdx.x] = ss;
    s_u[threadIdx.x] = su;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            s_t[threadIdx.x] += s_t[threadIdx.x + o];
            s_s[threadIdx.x] += s_s[threadIdx.x + o];
            s_u[threadIdx.x] += s_u[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        double* q = part + 3 * ((int64_t)scene * gridDim.x + blockIdx.x);
        q[0] = s_t[0];
        q[1] = s_s[0];
        q[2] = __longlong_as_double((long long)s_u[0]);
    }
}

__global__ __launch_bounds__(256) void k_mass_scenes_final(const double* __restrict__ part, int nscenes, int nblocks,
                                                           double* __restrict__ out)
{
    const int s = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (s >= nscenes) return;
    double st = 0.0, ss = 0.0;
    unsigned long long su = 0ull;
    const double* q = part + 3 * (int64_t)s * nblocks;
    for (int b = 0; b < nblocks; ++b) {
        st += q[3 * b];
        ss += q[3 * b + 1];
        su += (unsigned long long)__double_as_longlong(q[3 * b + 2]);
    }
    // planar: terrain[nscenes], sediment[nscenes], units[nscenes]
    out[s] = st;
    out[nscenes + s] = ss;
    out[2 * nscenes + s] = __longlong_as_double((long long)su);
}

__global__ void k_mass_final(const double* __restrict__ part, int nblocks, double* __restrict__ out)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double st = 0.0, ss = 0.0;
    unsigned long long su = 0ull;
    for (int b = 0; b < nblocks; ++b) {
        st += part[3 * b];
        ss += part[3 * b + 1];
        su += (unsigned long long)__double_as_longlong(part[3 * b + 2]);
    }
    out[0] = st;
    out[1] = ss;
    out[2] = __longlong_as_double((long long)su);
}

inline unsigned grid_of(int64_t n, int block) { return (unsigned)((n + block - 1) / block); }

}  // namespace

// ------------------------------------------------------------- launchers

// The precision modes of sphe_create: 0 FP32 with Kahan-compensated sums,
// 1 FP32 plain, 2 FP64, 3 FP32 with compensated density sums and
// FP64-accumulated force sums.  KERN(T, SM) names the kernel instantiation.
#define SPHE_PREC_SWITCH(prec, CALL)                                      \
    do {                                                                  \
        if ((prec) == 0) { CALL(float, SUM_KAHAN); }                      \
        else if ((prec) == 1) { CALL(float, SUM_PLAIN); }                 \
        else if ((prec) == 3) { CALL(float, SUM_F64ACC); }                \
        else { CALL(double, SUM_PLAIN); }                                 \
    } while (0)

// Launches kern.  With profiling events, through hipExtLaunchKernel: e0 and
// e1 then take the kernel's own start and end times, with no marker packets
// between kernels.
template <typename... P, typename... A>
static void klaunch(void (*kern)(P...), dim3 grid, dim3 block, hipStream_t st, hipEvent_t e0, hipEvent_t e1,
                    A... args)
{
    if (e0 || e1) hipExtLaunchKernelGGL(kern, grid, block, 0, st, e0, e1, 0, args...);
    else hipLaunchKernelGGL(kern, grid, block, 0, st, args...);
}

// The same with lds bytes of dynamic LDS per block.
template <typename... P, typename... A>
static void klaunch_lds(void (*kern)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t st, hipEvent_t e0,
                        hipEvent_t e1, A... args)
{
    if (e0 || e1) hipExtLaunchKernelGGL(kern, grid, block, lds, st, e0, e1, 0, args...);
    else hipLaunchKernelGGL(kern, grid, block, lds, st, args...);
}

// Blocks of `kern` (block threads, lds bytes of dynamic LDS) resident on
// the current device at once: the grid of a persistent launch (a multiple
// of the XCD count).
template <typename... P>
static int resident_grid(void (*kern)(P...), int block, size_t lds)
{
    static std::mutex mu;
    static std::map<std::tuple<const void*, int, size_t, int>, int> cache;
    int dev = 0;
    (void)hipGetDevice(&dev);
    const auto key = std::make_tuple((const void*)kern, block, lds, dev);
    std::lock_guard<std::mutex> g(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)kern, block, lds) != hipSuccess) per = 0;
    (void)hipGetLastError();
    const int n = std::max(8, (std::max(cus, 1) * std::max(per, 1)) / 8 * 8);
    cache[key] = n;
    return n;
}

// A pass as a persistent launch: the queues cleared, then a resident grid
// (at most one block per item).
template <typename... P, typename... A>
static void klaunch_pers(void (*kern)(P...), int nblk, int block, size_t lds, const DevState& D, hipStream_t st,
                         hipEvent_t e0, hipEvent_t e1, A... args)
{
    const int grid = std::min(resident_grid(kern, block, lds), nblk);
    klaunch(k_work_reset, 1, 64, st, e0, nullptr, D.work);
    klaunch_lds(kern, grid, block, lds, st, nullptr, e1, args...);
}

void sphe_launch_hash(const DevState& D, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    if (D.P == 0) return;
    if (D.precision == 2) klaunch(k_hash_count<double>, grid_of(D.P, 256), 256, st, e0, e1, D);
    else klaunch(k_hash_count<float>, grid_of(D.P, 256), 256, st, e0, e1, D);
}

template <int ITEMS>
static void launch_scan_cells_t(const DevState& D, bool heights, int first, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    const int nb = (int)scan_tiles(D);
    const int nh = heights ? (int)grid_of(D.TC / 4, 256) : 0;  // TC: a multiple of 64
    if (!D.totals) klaunch(k_scan_reduce_cells<ITEMS>, nb, 256, st, e0, nullptr, D);
    if (scan_sums(D)) {
        klaunch(k_scan_cells<ITEMS, SCAN_SUMS>, nb + nh, 256, st, D.totals ? e0 : nullptr, e1, D, nb, first);
        return;
    }
    klaunch(k_scan_tiles, 1, 1024, st, D.totals ? e0 : nullptr, nullptr, (const uint32_t*)D.total, D.tlog,
            D.tpre);
    klaunch(k_scan_cells<ITEMS, SCAN_PREFIX>, nb + nh, 256, st, nullptr, e1, D, nb, first);
}

void sphe_launch_scan_cells(const DevState& D, bool heights, bool first, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    if (D.scan_log2 == 11) launch_scan_cells_t<8>(D, heights, first, st, e0, e1);
    else if (D.scan_log2 == 13) launch_scan_cells_t<32>(D, heights, first, st, e0, e1);
    else launch_scan_cells_t<16>(D, heights, first, st, e0, e1);
}

int64_t sphe_scan_partials(int64_t n) { return (n + (1 << SPHE_SCAN_LOG2_MIN) - 1) >> SPHE_SCAN_LOG2_MIN; }

void sphe_launch_scatter(const DevState& D, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    if (D.P == 0) return;
    klaunch(k_scatter, grid_of(D.P, 256), 256, st, e0, e1, D);
}

void sphe_launch_reorder(const DevState& D, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    if (D.P == 0) return;
    if (D.precision == 2) klaunch(k_reorder<double>, grid_of(D.P, 256), 256, st, e0, e1, D);
    else klaunch(k_reorder<float>, grid_of(D.P, 256), 256, st, e0, e1, D);
}

template <int G>
static void launch_density_g(const DevState& D, int block, int remap, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    if constexpr (G == 4) {
        if (!D.persistent && D.yz <= 2) {
            const size_t lds = (size_t)quad_group_bytes(D.yz) * (size_t)(block / 4);
            const int nblk = (int)grid_of(D.P * G, block);
#define CALL(T, SM)                                                                                       \
    do {                                                                                                  \
        void (*k)(DevState, int, int) =                                                                   \
            D.yz == 1 ? (D.h_unit ? k_density_quad<T, SM, 1, true> : k_density_quad<T, SM, 1, false>)     \
                      : (D.h_unit ? k_density_quad<T, SM, 2, true> : k_density_quad<T, SM, 2, false>);    \
        klaunch_lds(k, nblk, block, lds, st, e0, e1, D, nblk, remap);                                     \
    } while (0)
            SPHE_PREC_SWITCH(D.precision, CALL);
#undef CALL
            return;
        }
    }
    // one row table and one list staging ring per group, at most 64 KiB per
    // block with the persistent form's static word (halve the block until
    // it fits)
    const int W = 2 * D.yz + 1, ring = 4 * G > 16 ? 64 : 32;
    while (block > 64 && density_lds_bytes(W, block / G, ring) > 65536 - 256) block /= 2;
    const size_t lds = (size_t)density_lds_bytes(W, block / G, ring);
    const int nblk = (int)grid_of(D.P * G, block);
    if (D.persistent) {
#define CALL(T, SM) \
    klaunch_pers(k_density_pers<T, SM, G>, nblk, block, lds, D, st, e0, e1, D, nblk, remap, D.work)
        SPHE_PREC_SWITCH(D.precision, CALL);
#undef CALL
        return;
    }
#define CALL(T, SM) klaunch_lds(k_density<T, SM, G>, nblk, block, lds, st, e0, e1, D, nblk, remap)
    SPHE_PREC_SWITCH(D.precision, CALL);
#undef CALL
}

template <int G>
static void launch_force_g(const DevState& D, int block, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    const int nblk = (int)grid_of(D.P * G, block);
    if (D.persistent) {
        if (D.precision == 2) {
            klaunch_pers(k_force_f64_pers<G>, nblk, block, 0, D, st, e0, e1, D, nblk, 1, D.work);
            return;
        }
#define CALL(T, SM) klaunch_pers(k_force_f32_pers<SM, G>, nblk, block, 0, D, st, e0, e1, D, nblk, 1, D.work)
        SPHE_PREC_SWITCH(D.precision, CALL);
#undef CALL
        return;
    }
    if (D.precision == 2) {
        klaunch(k_force_f64<G>, nblk, block, st, e0, e1, D);
        return;
    }
    const bool unit = D.h_unit != 0;
#define CALL(T, SM) klaunch(unit ? k_force_f32<SM, G, G == 4> : k_force_f32<SM, G, false>, nblk, block, st, e0, e1, D)
    SPHE_PREC_SWITCH(D.precision, CALL);
#undef CALL
}

void sphe_launch_density(const DevState& D, int block, int remap, int lanes, hipStream_t st, hipEvent_t e0,
                         hipEvent_t e1)
{
    if (D.P == 0) return;
    switch (lanes) {
    case 1: launch_density_g<1>(D, block, remap, st, e0, e1); break;
    case 2: launch_density_g<2>(D, block, remap, st, e0, e1); break;
    case 8: launch_density_g<8>(D, block, remap, st, e0, e1); break;
    default: launch_density_g<4>(D, block, remap, st, e0, e1); break;
    }
}

void sphe_launch_force(const DevState& D, int block, int lanes, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    if (D.P == 0) return;
    switch (lanes) {
    case 1: launch_force_g<1>(D, block, st, e0, e1); break;
    case 2: launch_force_g<2>(D, block, st, e0, e1); break;
    case 8: launch_force_g<8>(D, block, st, e0, e1); break;
    default: launch_force_g<4>(D, block, st, e0, e1); break;
    }
}

void sphe_launch_heights(const DevState& D, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    if (D.TC == 0) return;
    klaunch(k_heights, grid_of(D.TC / 4, 256), 256, st, e0, e1, D);  // TC: a multiple of 64
}

void sphe_launch_two_phase(const DevState& D, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    if (D.TC == 0 || D.P == 0) return;
    klaunch(k_tapply, grid_of(D.TC / 2, 256), 256, st, e0, e1, D);
}

void sphe_launch_clear_status(const DevState& D, hipStream_t st) { k_clear_status<<<1, 64, 0, st>>>(D.status); }

void sphe_launch_terrain_mesh(const float* H, int nx, int nz, float cell, float ox, float oz, float* out,
                              hipStream_t st)
{
    const int64_t n = (int64_t)nx * nz;
    if (n == 0) return;
    k_terrain_mesh<<<grid_of(n, 256), 256, 0, st>>>(H, nx, nz, cell, ox, oz, out);
}

template <int G>
static void launch_inspect_g(const DevState& D, const int32_t* slotp, bool lists, double* out, hipStream_t st)
{
#define CALL(T, SM) k_inspect<T, SM, G><<<1, 64, 0, st>>>(D, slotp, lists, out)
    SPHE_PREC_SWITCH(D.precision, CALL);
#undef CALL
}

void sphe_launch_inspect(const DevState& D, const int32_t* slotp, int lanes, bool lists, double* out, hipStream_t st)
{
    switch (lanes) {
    case 1: launch_inspect_g<1>(D, slotp, lists, out, st); break;
    case 2: launch_inspect_g<2>(D, slotp, lists, out, st); break;
    case 8: launch_inspect_g<8>(D, slotp, lists, out, st); break;
    default: launch_inspect_g<4>(D, slotp, lists, out, st); break;
    }
}

void sphe_launch_idmap(const DevState& D, int64_t p0, int64_t p1, int32_t* map, int64_t m0, int64_t m1, bool unique,
                       hipStream_t st)
{
    if (p1 <= p0 || m1 <= m0) return;
    if (unique) {
        k_idmap<true><<<grid_of(p1 - p0, 256), 256, 0, st>>>(D, p0, p1, map);
    } else {
        k_fill_i32<<<grid_of(m1 - m0, 256), 256, 0, st>>>(map + m0, m1 - m0, INT32_MAX);
        k_idmap<false><<<grid_of(p1 - p0, 256), 256, 0, st>>>(D, p0, p1, map);
    }
}

void sphe_launch_feed(const DevState& D, int64_t p0, int64_t n, int what, float* out, hipStream_t st)
{
    if (n <= 0) return;
    if (D.precision == 2) k_feed<double><<<grid_of(n, 256), 256, 0, st>>>(D, p0, n, what, out);
    else k_feed<float><<<grid_of(n, 256), 256, 0, st>>>(D, p0, n, what, out);
}

void sphe_launch_gather(const DevState& D, const int32_t* map, int64_t n, int what, float* out, hipStream_t st)
{
    if (n <= 0) return;
    if (D.precision == 2) k_gather<double><<<grid_of(n, 256), 256, 0, st>>>(D, map, n, what, out);
    else k_gather<float><<<grid_of(n, 256), 256, 0, st>>>(D, map, n, what, out);
}

void sphe_launch_find_id(const DevState& D, int scene, int32_t id, int32_t* slot_out, hipStream_t st)
{
    k_fill_i32<<<1, 64, 0, st>>>(slot_out, 1, INT32_MAX);
    if (D.P > 0) k_find_id<<<grid_of(D.P, 256), 256, 0, st>>>(D, scene, id, slot_out);
}

template <int G>
static void launch_accel_g(const DevState& D, int scene, double* out, hipStream_t st)
{
    const unsigned nb = grid_of(D.P * G, 256);
#define CALL(T, SM) k_accel<T, SM, G><<<nb, 256, 0, st>>>(D, scene, out)
    SPHE_PREC_SWITCH(D.precision, CALL);
#undef CALL
}

void sphe_launch_accel(const DevState& D, int scene, int lanes, double* out, hipStream_t st)
{
    if (D.P == 0) return;
    switch (lanes) {
    case 1: launch_accel_g<1>(D, scene, out, st); break;
    case 2: launch_accel_g<2>(D, scene, out, st); break;
    case 8: launch_accel_g<8>(D, scene, out, st); break;
    default: launch_accel_g<4>(D, scene, out, st); break;
    }
}

void sphe_launch_neighbours(const DevState& D, int scene, const int64_t* off, int32_t* counts, int32_t* idx,
                            hipStream_t st)
{
    if (D.P == 0) return;
    if (D.precision == 2) k_neighbours<double><<<grid_of(D.P, 256), 256, 0, st>>>(D, scene, off, counts, idx);
    else k_neighbours<float><<<grid_of(D.P, 256), 256, 0, st>>>(D, scene, off, counts, idx);
}

void sphe_launch_keys(const DevState& D, int scene, int32_t* keys, hipStream_t st)
{
    if (D.P == 0) return;
    if (D.precision == 2) k_keys<double><<<grid_of(D.P, 256), 256, 0, st>>>(D, scene, keys);
    else k_keys<float><<<grid_of(D.P, 256), 256, 0, st>>>(D, scene, keys);
}

int sphe_mass_blocks() { return 256; }

// Scratch of sphe_mass_all_noalloc, for callers that cannot allocate device
// memory: the per-scene block partials and the per-scene results of the
// all-scene bookkeeping for up to SPHE_NOALLOC_MAX_SCENES scenes.  Every GPU
// the library runs on holds its own copy until the process ends.  Host code
// uses the address sphe_noalloc_scratch returns, never this name.
static __device__ __align__(256) double scratch[(size_t)3 * (SPHE_MASS_BLOCKS_PER_SCENE + 1) *
                                                SPHE_NOALLOC_MAX_SCENES];

int sphe_noalloc_scratch(int device, double** ptr, size_t* doubles)
{
    static std::mutex mu;
    static std::map<int, double*> addr;  // device -> address of its scratch
    std::lock_guard<std::mutex> g(mu);
    auto it = addr.find(device);
    if (it == addr.end()) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            (void)hipGetLastError();
            *ptr = nullptr;
            *doubles = 0;
            return -1;
        }
        it = addr.emplace(device, (double*)p).first;
    }
    *ptr = it->second;
    *doubles = sizeof(scratch) / sizeof(double);
    return 0;
}

void sphe_launch_mass(const DevState& D, int scene, double* part, double* out, hipStream_t st)
{
    k_mass_partial<<<sphe_mass_blocks(), 256, 0, st>>>(D, scene, part);
    k_mass_final<<<1, 64, 0, st>>>(part, sphe_mass_blocks(), out);
}

void sphe_launch_mass_scenes(const DevState& D, double* part, double* out, hipStream_t st)
{
    if (D.nscenes == 0) return;
    k_mass_scenes<<<dim3(SPHE_MASS_BLOCKS_PER_SCENE, (unsigned)D.nscenes), 256, 0, st>>>(D, part);
    k_mass_scenes_final<<<grid_of(D.nscenes, 256), 256, 0, st>>>(part, D.nscenes, SPHE_MASS_BLOCKS_PER_SCENE, out);
}

// ------------------------------------------------------------ calibration

namespace {
// Plain streaming copy (16 bytes per thread per iteration): the reference
// point for HBM bandwidth and for scaling the FETCH_SIZE / WRITE_SIZE
// counters of the step's kernels.
__global__ __launch_bounds__(256) void k_copy(const float4* __restrict__ a, float4* __restrict__ b, int64_t n)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) b[i] = a[i];
}
}  // namespace

void sphe_launch_copy(const void* a, void* b, int64_t n16, hipStream_t st)
{
    k_copy<<<2048, 256, 0, st>>>((const float4*)a, (float4*)b, n16);
}
