// Many independent systems of uneven size in one set of launches: energy, forces and virial of
// every system, with no per-system launch and no host round trip between systems.
//
// All systems share one global bin space (each owns a contiguous range of it), so one counting
// sort bins every atom of the batch, one scan covers every bin, and one force launch covers every
// atom. The force launch builds no list: each atom's candidates come from the culled stencil of
// its own system's sub-bins, and the pair terms are summed as they are found. Two schedules:
//   - wave per sub-bin: its atoms' candidates 64 at a time across the lanes, read once for two
//     atoms, reduced over the wave;
//   - thread per atom: a lane per atom walking its own stencil.
// and two sub-bin sizes (at least the cutoff, or half of it). A host-side autotuner times the
// four on the batch and keeps the fastest.
//
// Every sum is per atom and then per system in a fixed order, so a system's results do not
// depend on the other systems of the batch: alone or in the mix, the same schedule gives the
// same bits. Geometry and mask follow the reference (space.py:11-19,
// _lennard_jones/_potential.py:218-234, _tabulated/_potential.py:146-162).

#include <algorithm>
#include <climits>

#include "common.hpp"
#include "neighbors.hpp"
#include "pair_forces.hpp"
#include "potentials.hpp"
#include "scan.hpp"

namespace ndn {

template <typename T>
struct BatchArgs
{
    const T* positions;       // [N, 3] input, anywhere
    index_t num_atoms;
    std::int64_t num_systems;
    const index_t* system_of;      // [N]
    const std::int64_t* atom_start;  // [S + 1]
    const index_t* bin_start;      // [S + 1] first global bin of each system
    const index_t* dims;           // [S, 3]
    const T* widths;               // [S, 3]
    const T* cells;                // [S, 3]
    const T* cutoffs;              // [S]
    const T* cutoffs_squared;      // [S]
    const index_t* kinds;          // [S]
    const LJRow<T>* lj;            // [S]
    const index_t* table_of;       // [S] row of the padded tables, or -1
    const T* tables;               // [R, K + 2]
    const T* table_start;          // [R]
    const T* table_spacing;  // [R]
    int knots;
    std::int64_t total_bins;
    int span;                      // sub-bins a stencil reaches on each side: 1 or 2
    // scratch
    index_t* bin_of;
    index_t* bin_counts;
    index_t* bin_offsets;
    index_t* unordered;
    index_t* order;                // slot -> atom
    T* wrapped4;                   // [N, 4] wrapped positions in atom order
    T* sorted4;                    // [N, 4] the same in slot order
    std::uint8_t* scan_temp;
    // outputs
    T* forces;                     // [N, 3]
    T* atom_terms;                 // [N, 7]: half the pair energy and virial of each atom
    T* energy;                     // [S]
    T* virial;                     // [S, 9]
};

template <typename T>
__device__ __forceinline__ index_t batch_bin(T x, T width, index_t count)
{
    const index_t bin = static_cast<index_t>(floor(x / width));
    return bin < 0 ? 0 : (bin >= count ? count - 1 : bin);
}

// Wraps each atom into its system's cell (the reference's arithmetic) and counts it in its bin.
template <typename T>
__global__ void __launch_bounds__(kBlock) batch_assign_kernel(BatchArgs<T> a)
{
#pragma clang fp contract(off)
    using V4 = typename std::conditional<sizeof(T) == 4, float4, double4>::type;
    const std::int64_t atom = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (atom >= a.num_atoms) return;
    const index_t s = a.system_of[atom];
    T w[3];
    index_t b[3];
    for (int axis = 0; axis < 3; ++axis)
    {
        const T length = a.cells[3 * s + axis];
        const T v = a.positions[3 * atom + axis];
        const T k = floor(v / length);
        T x = v - k * length;
        if (x < T(0)) x = x + length;
        if (x >= length) x = x - length;
        w[axis] = x;
        b[axis] = batch_bin(x, a.widths[3 * s + axis], a.dims[3 * s + axis]);
    }
    V4 p;
    p.x = w[0];
    p.y = w[1];
    p.z = w[2];
    p.w = T(0);
    reinterpret_cast<V4*>(a.wrapped4)[atom] = p;
    const index_t nx = a.dims[3 * s], ny = a.dims[3 * s + 1];
    const index_t bin = a.bin_start[s] + b[0] + nx * (b[1] + ny * b[2]);
    a.bin_of[atom] = bin;
    // one atomic per run of a bin's atoms in neighbouring lanes
    const LaneRun run = equal_runs(bin);
    if (run.head) atomicAdd(a.bin_counts + bin, run.length);
}

template <typename T>
__global__ void __launch_bounds__(kBlock) batch_scatter_kernel(BatchArgs<T> a)
{
    const std::int64_t atom = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (atom >= a.num_atoms) return;
    const index_t bin = a.bin_of[atom];
    // one atomic per run: the run's lanes take the places below the count it returns, one each
    // (batch_order_kernel orders a bin's atoms by index after)
    const LaneRun run = equal_runs(bin);
    index_t count = 0;
    if (run.head) count = atomicSub(a.bin_counts + bin, run.length);
    count = __shfl(count, run.first, kWave);
    a.unordered[a.bin_offsets[bin] + count - 1 - (lane_id() - run.first)] =
        static_cast<index_t>(atom);
}

// Thread per entry of the unordered array: ranks its atom by index among its bin's (deterministic),
// writes slot -> atom and the sorted position there.
template <typename T>
__global__ void __launch_bounds__(kBlock) batch_order_kernel(BatchArgs<T> a)
{
    using V4 = typename std::conditional<sizeof(T) == 4, float4, double4>::type;
    const std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= a.num_atoms) return;
    const index_t atom = a.unordered[i];
    const V4 position = reinterpret_cast<const V4*>(a.wrapped4)[atom];
    const index_t bin = a.bin_of[atom];
    const index_t begin = a.bin_offsets[bin];
    const index_t end = a.bin_offsets[bin + 1];
    index_t rank = 0;
    for (index_t k = begin; k < end; ++k) rank += a.unordered[k] < atom;
    a.order[begin + rank] = atom;
    reinterpret_cast<V4*>(a.sorted4)[begin + rank] = position;
}

template <typename T>
__device__ __forceinline__ T batch_slab(T c, T lo, T w)
{
    const T below = lo - c;
    const T above = c - (lo + w);
    return below > T(0) ? below : (above > T(0) ? above : T(0));
}

template <typename T>
struct SystemView
{
    index_t nx, ny, nz;
    T wx, wy, wz;
    T lx, ly, lz;
    T cutoff, cutoff_squared;
    index_t bin_start;
    int kind;
    LJRow<T> lj;
    const T* table;
    T table_start, table_spacing;
};

template <typename T>
__device__ __forceinline__ SystemView<T> system_view(const BatchArgs<T>& a, index_t s)
{
    SystemView<T> v;
    v.nx = a.dims[3 * s];
    v.ny = a.dims[3 * s + 1];
    v.nz = a.dims[3 * s + 2];
    v.wx = a.widths[3 * s];
    v.wy = a.widths[3 * s + 1];
    v.wz = a.widths[3 * s + 2];
    v.lx = a.cells[3 * s];
    v.ly = a.cells[3 * s + 1];
    v.lz = a.cells[3 * s + 2];
    v.cutoff = a.cutoffs[s];
    v.cutoff_squared = a.cutoffs_squared[s];
    v.bin_start = a.bin_start[s];
    v.kind = a.kinds[s];
    v.lj = a.lj[s];
    const index_t row = a.table_of[s];
    v.table = row >= 0 ? a.tables + static_cast<std::int64_t>(row) * (a.knots + 2) : nullptr;
    v.table_start = row >= 0 ? a.table_start[row] : T(0);
    v.table_spacing = row >= 0 ? a.table_spacing[row] : T(1);
    return v;
}

// u and -(du/dr)/r of a pair of the system, r^2 below its cutoff.
template <typename T>
__device__ __forceinline__ void pair_terms(const SystemView<T>& v, int knots, T r2, T& u, T& fs)
{
    if (v.kind == NDN_LJ)
    {
        const T inverse = T(1) / r2;
        const T s = v.lj.sigma_squared * inverse;
        const T p6 = s * s * s;
        u = v.lj.four_eps * (p6 * p6 - p6) - v.lj.shift;
        fs = v.lj.twentyfour_eps * (T(2) * p6 * p6 - p6) * inverse;
        return;
    }
    // r and the knot coordinate with the reference's operations, each correctly rounded
    const T r = sqrt(r2);
    const T x = (r - v.table_start) / v.table_spacing;
    T segment = floor(x);
    segment = segment < T(0) ? T(0) : (segment > T(knots - 2) ? T(knots - 2) : segment);
    const T t = x - segment;
    const T* k = v.table + static_cast<int>(segment);
    const T u0 = k[0], u1 = k[1], u2 = k[2], u3 = k[3];
    const T a1 = u2 - u0;
    const T b1 = T(2) * u0 - T(5) * u1 + T(4) * u2 - u3;
    const T c1 = T(3) * (u1 - u2) + u3 - u0;
    const T s = t > T(0) ? t : T(0);
    const bool below = t < T(0);
    u = u1 + T(0.5) * s * (a1 + s * (b1 + s * c1)) + (below ? T(0.5) * a1 * t : T(0));
    const T du_dt = below ? T(0.5) * a1 : T(0.5) * (a1 + s * (T(2) * b1 + T(3) * s * c1));
    fs = -(du_dt / v.table_spacing) / r;
}

// The stencil of a center: one lane (of 64) per candidate run of x-consecutive sub-bins in a
// (y, z) row, culled by distance. Returns this lane's [lo, lo + length) of slots.
template <typename T>
__device__ __forceinline__ void stencil_run(const BatchArgs<T>& a, const SystemView<T>& v, T cx,
                                            T cy, T cz, int lane, T cull_squared, index_t& lo,
                                            index_t& length, bool& wraps)
{
    const int reach = 2 * a.span + 1;
    const index_t hx = batch_bin(cx, v.wx, v.nx), hy = batch_bin(cy, v.wy, v.ny),
                  hz = batch_bin(cz, v.wz, v.nz);
    const bool full_x = v.nx < reach, full_y = v.ny < reach, full_z = v.nz < reach;
    const int span_x = full_x ? v.nx : reach;
    const int span_y = full_y ? v.ny : reach;
    const int span_z = full_z ? v.nz : reach;
    wraps = full_x || full_y || full_z || hx < a.span || hx + a.span >= v.nx || hy < a.span ||
            hy + a.span >= v.ny || hz < a.span || hz + a.span >= v.nz;
    lo = 0;
    length = 0;
    const int row = lane / 2, part = lane % 2;
    if (row >= span_y * span_z) return;
    const int oy = row % span_y, oz = row / span_y;
    const index_t by = full_y ? oy : hy + oy - a.span;
    const index_t bz = full_z ? oz : hz + oz - a.span;
    const T dy = full_y ? T(0) : batch_slab(cy, by * v.wy, v.wy);
    const T dz = full_z ? T(0) : batch_slab(cz, bz * v.wz, v.wz);
    const T dyz = dy * dy + dz * dz;
    if (!(dyz < cull_squared)) return;
    int first = span_x, last = -1;
    for (int ox = 0; ox < span_x; ++ox)
    {
        const index_t bx = full_x ? ox : hx + ox - a.span;
        const T dx = full_x ? T(0) : batch_slab(cx, bx * v.wx, v.wx);
        if (dx * dx + dyz < cull_squared)
        {
            first = ox < first ? ox : first;
            last = ox;
        }
    }
    if (last < first) return;
    const index_t wy = by < 0 ? by + v.ny : (by >= v.ny ? by - v.ny : by);
    const index_t wz = bz < 0 ? bz + v.nz : (bz >= v.nz ? bz - v.nz : bz);
    const std::int64_t base = v.bin_start + static_cast<std::int64_t>(v.nx) *
                                                (wy + static_cast<std::int64_t>(v.ny) * wz);
    const index_t x0 = full_x ? first : hx + first - a.span;
    const index_t x1 = full_x ? last : hx + last - a.span;
    index_t run_lo = 0, run_hi = -1;
    if (x0 < 0)
    {
        run_lo = part == 0 ? x0 + v.nx : 0;
        run_hi = part == 0 ? v.nx - 1 : x1;
    }
    else if (x1 >= v.nx)
    {
        run_lo = part == 0 ? x0 : 0;
        run_hi = part == 0 ? v.nx - 1 : x1 - v.nx;
    }
    else if (part == 0)
    {
        run_lo = x0;
        run_hi = x1;
    }
    if (run_hi < run_lo) return;
    lo = a.bin_offsets[base + run_lo];
    length = a.bin_offsets[base + run_hi + 1] - lo;
}

template <typename T>
__device__ __forceinline__ void pair_vector(bool wraps, T cx, T cy, T cz, T qx, T qy, T qz,
                                            const SystemView<T>& v, T& dx, T& dy, T& dz)
{
    if (wraps)
    {
        dx = displacement(cx, qx, v.lx);
        dy = displacement(cy, qy, v.ly);
        dz = displacement(cz, qz, v.lz);
    }
    else
    {
        dx = cx - qx;
        dy = cy - qy;
        dz = cz - qz;
    }
}

// What the wave schedule evaluates a pair with: the system's potential, its divisions by
// constants as products. x / h with y = 1 / h correctly rounded is q = x y corrected once by its
// remainder: the correctly rounded quotient (Markstein, as above), so the knot coordinate is the
// reference's.
template <typename T>
struct WavePotential
{
    int kind, knots;
    LJRow<T> lj;
    const T* table;
    T start, spacing, inverse_spacing;

    __device__ __forceinline__ void eval(T r2, T& u, T& fs) const
    {
        if (kind == NDN_LJ)
        {
            const T inverse = refined_reciprocal(r2);
            const T s = lj.sigma_squared * inverse;
            const T p6 = s * s * s;
            u = lj.four_eps * (p6 * p6 - p6) - lj.shift;
            fs = lj.twentyfour_eps * (T(2) * p6 * p6 - p6) * inverse;
            return;
        }
        const T r = pair_distance(r2);
        const T offset = r - start;
        const T q = offset * inverse_spacing;
        const T x = fma(fma(-q, spacing, offset), inverse_spacing, q);
        T segment = floor(x);
        segment = segment < T(0) ? T(0) : (segment > T(knots - 2) ? T(knots - 2) : segment);
        const T t = x - segment;
        const T* k = table + static_cast<int>(segment);
        const T u0 = k[0], u1 = k[1], u2 = k[2], u3 = k[3];
        const T a1 = u2 - u0;
        const T b1 = T(2) * u0 - T(5) * u1 + T(4) * u2 - u3;
        const T c1 = T(3) * (u1 - u2) + u3 - u0;
        const T s = t > T(0) ? t : T(0);
        const bool below = t < T(0);
        u = u1 + T(0.5) * s * (a1 + s * (b1 + s * c1)) + (below ? T(0.5) * a1 * t : T(0));
        const T du_dt = below ? T(0.5) * a1 : T(0.5) * (a1 + s * (T(2) * b1 + T(3) * s * c1));
        fs = -(du_dt * inverse_spacing) * refined_reciprocal(r);
    }
};

// Centers of a bin that a wave takes together. Each keeps ten sums of its own (F, E and W, which
// go out per atom), so more centers cost the waves that hide the gathers: the 256 systems of 64
// to 32,768 atoms in fp32 take 1.46 ms with two centers at 7 waves per SIMD (1.53 at 6), 1.57 with
// three at 6, 1.52 with four at 5; 40 systems to 10,000 atoms in fp64 237 us with two at 4, 246
// with two unbounded, 294 with three.
constexpr int kWaveCenters = 2;
template <typename T>
constexpr int kWaveOccupancy = sizeof(T) == 4 ? 7 : 4;

// How a candidate's vector is formed, uniform over a bin's centers.
constexpr int kWavePlain = 0;    // the stencil lies inside the box
constexpr int kWaveShifted = 1;  // part of it across a face: the near-face coordinate shifted
constexpr int kWaveImage = 2;    // an axis shorter than the stencil: minimum image per pair

// This lane's candidate range of a bin: row lane / 2 of the stencil's (y, z) rows of sub-bins, the
// part lane % 2 of its run along x that a face splits, cut to the sub-bins within `reach` of the
// box [low, high] of the centers. `shift` holds two bits per axis as in the list's search: 1 for
// a candidate below the box (it moves down by L), 2 above it (the center does).
template <typename T>
__device__ __forceinline__ void wave_range(const BatchArgs<T>& a, const SystemView<T>& v,
                                           const index_t home[3], const T low[3], const T high[3],
                                           T reach, int lane, index_t& lo, index_t& length,
                                           int& shift)
{
    const int span = a.span;
    const int full = 2 * span + 1;
    lo = 0;
    length = 0;
    shift = 0;
    const bool full_x = v.nx < full, full_y = v.ny < full, full_z = v.nz < full;
    const int span_y = full_y ? v.ny : full, span_z = full_z ? v.nz : full;
    const int row = lane / 2, part = lane % 2;
    if (row >= span_y * span_z) return;
    const int oy = row % span_y, oz = row / span_y;
    const index_t ry = full_y ? oy : home[1] + oy - span;
    const index_t rz = full_z ? oz : home[2] + oz - span;
    auto gap = [](T low_face, T high_face, T from, T to) {
        const T below = low_face - to, above = from - high_face;
        return fmax(fmax(below, above), T(0));
    };
    const T gy = full_y ? T(0) : gap(ry * v.wy, (ry + 1) * v.wy, low[1], high[1]);
    const T gz = full_z ? T(0) : gap(rz * v.wz, (rz + 1) * v.wz, low[2], high[2]);
    const T left = reach * reach - (gy * gy + gz * gz);
    if (!(left > T(0))) return;
    index_t x0 = 0, x1 = v.nx - 1;
    if (!full_x)
    {
        // the run along x: what the reach leaves past the centers' box, within the stencil
        const T across = sqrt(left);
        const index_t from = static_cast<index_t>(floor((low[0] - across) / v.wx));
        const index_t to = static_cast<index_t>(floor((high[0] + across) / v.wx));
        x0 = from > home[0] - span ? from : home[0] - span;
        x1 = to < home[0] + span ? to : home[0] + span;
    }
    const index_t by = ry < 0 ? ry + v.ny : (ry >= v.ny ? ry - v.ny : ry);
    const index_t bz = rz < 0 ? rz + v.nz : (rz >= v.nz ? rz - v.nz : rz);
    shift = (ry < 0 ? 4 : (ry >= v.ny ? 8 : 0)) | (rz < 0 ? 16 : (rz >= v.nz ? 32 : 0));
    index_t first = 0, last = -1;
    if (x0 < 0)
    {
        // below the box, then the rest
        first = part == 0 ? x0 + v.nx : 0;
        last = part == 0 ? v.nx - 1 : x1;
        if (part == 0) shift |= 1;
    }
    else if (x1 >= v.nx)
    {
        first = part == 0 ? x0 : 0;
        last = part == 0 ? v.nx - 1 : x1 - v.nx;
        if (part == 1) shift |= 2;
    }
    else if (part == 0)
    {
        first = x0;
        last = x1;
    }
    if (last < first) return;
    const std::int64_t base =
        v.bin_start + static_cast<std::int64_t>(v.nx) * (by + static_cast<std::int64_t>(v.ny) * bz);
    lo = a.bin_offsets[base + first];
    length = a.bin_offsets[base + last + 1] - lo;
}

// A data-parallel move into kRows of the wave's rows of 16 lanes, zeros into the others.
template <int kControl, int kRows>
__device__ __forceinline__ float moved(float value)
{
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(value), kControl, kRows, 0xF, true));
}

template <int kControl, int kRows>
__device__ __forceinline__ double moved(double value)
{
    const int lo =
        __builtin_amdgcn_update_dpp(0, __double2loint(value), kControl, kRows, 0xF, true);
    const int hi =
        __builtin_amdgcn_update_dpp(0, __double2hiint(value), kControl, kRows, 0xF, true);
    return __hiloint2double(hi, lo);
}

// a's halves added in the wave's lower half, b's in its upper: the upper half of a's lanes and
// the lower half of b's change places, then one addition.
__device__ __forceinline__ float folded(float a, float b)
{
    const auto both =
        __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(both[0]) + __uint_as_float(both[1]);
}

__device__ __forceinline__ double folded(double a, double b)
{
    const auto lo =
        __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi =
        __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}

// Two sums over the wave at once, a's in lane 31 and b's in lane 63, without LDS.
template <typename T>
__device__ __forceinline__ T two_sums(T a, T b)
{
    T sum = folded(a, b);
    sum += moved<0x111, 0xF>(sum);  // row_shr:1
    sum += moved<0x112, 0xF>(sum);  // row_shr:2
    sum += moved<0x114, 0xF>(sum);  // row_shr:4
    sum += moved<0x118, 0xF>(sum);  // row_shr:8
    sum += moved<0x142, 0xA>(sum);  // row_bcast:15 into rows 1 and 3
    return sum;
}

// A group of a bin's centers (slots first .. first + live - 1) against their candidates, 64 a
// turn, each read once for all of them.
template <typename T, int kMode>
__device__ __forceinline__ void wave_centers(const BatchArgs<T>& a, const SystemView<T>& v,
                                             const WavePotential<T>& pot, const index_t home[3],
                                             index_t first, int live, T reach)
{
    using V4 = typename std::conditional<sizeof(T) == 4, float4, double4>::type;
    constexpr int kCenters = kWaveCenters;
    const int lane = lane_id();
    const V4* sorted = reinterpret_cast<const V4*>(a.sorted4);
    const V4 own = sorted[first + (lane < live ? lane : 0)];
    T cx[kCenters], cy[kCenters], cz[kCenters];
    T low[3], high[3];
#pragma unroll
    for (int g = 0; g < kCenters; ++g)
    {
        cx[g] = read_lane(own.x, g);
        cy[g] = read_lane(own.y, g);
        cz[g] = read_lane(own.z, g);
        low[0] = g == 0 ? cx[g] : fmin(low[0], cx[g]);
        low[1] = g == 0 ? cy[g] : fmin(low[1], cy[g]);
        low[2] = g == 0 ? cz[g] : fmin(low[2], cz[g]);
        high[0] = g == 0 ? cx[g] : fmax(high[0], cx[g]);
        high[1] = g == 0 ? cy[g] : fmax(high[1], cy[g]);
        high[2] = g == 0 ? cz[g] : fmax(high[2], cz[g]);
    }
    index_t lo, length;
    int range_shift;
    wave_range(a, v, home, low, high, reach, lane, lo, length, range_shift);
    const index_t inclusive = wave_inclusive_sum(length);
    const index_t start = inclusive - length;
    const index_t to_slot = lo - start;
    const index_t total = read_lane(inclusive, kWave - 1);
    // each center's F, E and W
    constexpr int kSums = 10;
    T sums[kSums][kCenters];
#pragma unroll
    for (int k = 0; k < kSums; ++k)
#pragma unroll
        for (int g = 0; g < kCenters; ++g) sums[k][g] = T(0);
    for (index_t chunk = 0; chunk < total; chunk += kWave)
    {
        const index_t t = chunk + lane;
        int r = 0;
#pragma unroll
        for (int step = 32; step > 0; step >>= 1)
        {
            const index_t s = __shfl(start, r + step, kWave);
            if (s <= t) r += step;
        }
        const bool valid = t < total;
        const index_t other = __shfl(to_slot, r, kWave) + t;
        V4 q = sorted[valid ? other : first];
        int shift = 0;
        if (kMode == kWaveShifted)
        {
            shift = __shfl(range_shift, r, kWave);
            q.x = (shift & 1) != 0 ? q.x - v.lx : q.x;
            q.y = (shift & 4) != 0 ? q.y - v.ly : q.y;
            q.z = (shift & 16) != 0 ? q.z - v.lz : q.z;
        }
#pragma unroll
        for (int g = 0; g < kCenters; ++g)
        {
            if (g >= live) break;
            T dx, dy, dz;
            if (kMode == kWaveImage)
            {
                dx = displacement(cx[g], q.x, v.lx);
                dy = displacement(cy[g], q.y, v.ly);
                dz = displacement(cz[g], q.z, v.lz);
            }
            else if (kMode == kWaveShifted)
            {
                dx = ((shift & 2) != 0 ? cx[g] - v.lx : cx[g]) - q.x;
                dy = ((shift & 8) != 0 ? cy[g] - v.ly : cy[g]) - q.y;
                dz = ((shift & 32) != 0 ? cz[g] - v.lz : cz[g]) - q.z;
            }
            else
            {
                dx = cx[g] - q.x;
                dy = cy[g] - q.y;
                dz = cz[g] - q.z;
            }
            const T r2 = exact_squared(dx, dy, dz);
            if (valid && other != first + g && r2 < v.cutoff_squared)
            {
                T u, fs;
                pot.eval(r2, u, fs);
                const T gx = fs * dx, gy = fs * dy, gz = fs * dz;
                sums[0][g] += gx;
                sums[1][g] += gy;
                sums[2][g] += gz;
                sums[3][g] += u;
                sums[4][g] += dx * gx;
                sums[5][g] += dy * gy;
                sums[6][g] += dz * gz;
                sums[7][g] += dx * gy;
                sums[8][g] += dx * gz;
                sums[9][g] += dy * gz;
            }
        }
    }
    T out[kSums];
#pragma unroll
    for (int k = 0; k < kSums; ++k) out[k] = two_sums(sums[k][0], sums[k][1]);
    // lane 31 holds the first center's, lane 63 the second's
    const int g = lane / 32;
    if (lane % 32 == 31 && g < live)
    {
        const index_t atom = a.order[first + g];
        T* f = a.forces + 3LL * atom;
        T* terms = a.atom_terms + 7LL * atom;
        for (int k = 0; k < 3; ++k) f[k] = out[k];
        for (int k = 0; k < 7; ++k) terms[k] = T(0.5) * out[3 + k];
    }
}

// Wave per sub-bin. Its atoms share their stencil: the ranges, their prefix sums and each
// candidate's place and image are found once for two of them, where a wave per atom spent most of
// its instructions on these. The 256 systems (0.9 million atoms, half LJ, half tables): 1.97 ->
// 1.46 ms an evaluation at sub-bins of half the cutoff, 3.68 -> 2.36 at sub-bins of the cutoff.
//
// A bin's atoms are taken in groups from its first, whatever else the batch holds, so that a system
// gets the same bits alone and beside others. The groups that begin within a bin's first `share`
// slots are its own wave's; those past them go to waves by slot, after the bins': wave `bins` + x
// takes the groups beginning in [share x, share x + share) that lie as far into their bin, so that
// a clump of atoms is spread over the chip. With `bins` 0 there is no wave per sub-bin: wave s
// takes the group that begins at slot s, if one does.
template <typename T>
__global__ void __launch_bounds__(kBlock, kWaveOccupancy<T>)
batch_wave_kernel(BatchArgs<T> a, T cull_factor, std::int64_t bins, index_t share)
{
    constexpr int kCenters = kWaveCenters;
    const std::int64_t wave = static_cast<std::int64_t>(blockIdx.x) * (kBlock / kWave) +
                              __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const bool by_slot = wave >= bins;
    std::int64_t bin = wave;
    index_t slot = 0, s = 0;
    if (by_slot)
    {
        const std::int64_t at = (wave - bins) * share;
        if (at >= a.num_atoms) return;
        slot = static_cast<index_t>(at);
        const index_t atom = __builtin_amdgcn_readfirstlane(a.order[slot]);
        bin = __builtin_amdgcn_readfirstlane(a.bin_of[atom]);
        s = __builtin_amdgcn_readfirstlane(a.system_of[atom]);
    }
    const index_t begin = __builtin_amdgcn_readfirstlane(a.bin_offsets[bin]);
    const index_t end = __builtin_amdgcn_readfirstlane(a.bin_offsets[bin + 1]);
    if (begin == end) return;
    if (!by_slot) s = __builtin_amdgcn_readfirstlane(a.system_of[a.order[begin]]);
    // before the groups are known, so that its reads wait beside theirs
    const SystemView<T> v = system_view(a, s);
    // the groups that begin in [from, past); differences, as a sum past the last slot could leave
    // 32 bits
    const index_t own = bins == 0 ? begin : (end - begin < share ? end : begin + share);
    index_t from = begin, past = own;
    if (by_slot)
    {
        from = slot > own ? slot : own;
        past = end - slot < share ? end : slot + share;
        from += (from - begin) % kCenters;
        static_assert(kCenters == 2, "the next group's begin");
    }
    if (from >= past) return;
    WavePotential<T> pot;
    pot.kind = __builtin_amdgcn_readfirstlane(v.kind);
    pot.knots = a.knots;
    pot.lj = v.lj;
    pot.table = v.table;
    pot.start = v.table_start;
    pot.spacing = v.table_spacing;
    pot.inverse_spacing = T(1) / v.table_spacing;
    const index_t local = static_cast<index_t>(bin) - v.bin_start;
    const index_t home[3] = {local % v.nx, (local / v.nx) % v.ny, local / (v.nx * v.ny)};
    const index_t full = 2 * a.span + 1;
    const bool image = v.nx < full || v.ny < full || v.nz < full;
    const bool inside = home[0] >= a.span && home[0] + a.span < v.nx && home[1] >= a.span &&
                        home[1] + a.span < v.ny && home[2] >= a.span && home[2] + a.span < v.nz;
    const T reach = v.cutoff * cull_factor;
    for (index_t first = from; first < past; first += kCenters)
    {
        const int live = end - first < kCenters ? end - first : kCenters;
        if (image)
            wave_centers<T, kWaveImage>(a, v, pot, home, first, live, reach);
        else if (inside)
            wave_centers<T, kWavePlain>(a, v, pot, home, first, live, reach);
        else
            wave_centers<T, kWaveShifted>(a, v, pot, home, first, live, reach);
    }
}

// Thread per atom: each lane walks its own stencil runs, one candidate at a time.
template <typename T>
__global__ void __launch_bounds__(kBlock) batch_thread_kernel(BatchArgs<T> a, T cull_factor)
{
    using V4 = typename std::conditional<sizeof(T) == 4, float4, double4>::type;
    const std::int64_t slot = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (slot >= a.num_atoms) return;
    const V4* sorted = reinterpret_cast<const V4*>(a.sorted4);
    const index_t atom = a.order[slot];
    const index_t s = a.system_of[atom];
    const SystemView<T> v = system_view(a, s);
    const V4 c = sorted[slot];
    const T cull = v.cutoff * cull_factor;
    T fx = 0, fy = 0, fz = 0, e = 0;
    T w[6] = {0, 0, 0, 0, 0, 0};
    const int reach = 2 * a.span + 1;
    const int rows = (v.ny < reach ? v.ny : reach) * (v.nz < reach ? v.nz : reach);
    for (int range = 0; range < 2 * rows; ++range)
    {
        index_t lo, length;
        bool wraps;
        stencil_run(a, v, c.x, c.y, c.z, range, cull * cull, lo, length, wraps);
        for (index_t other = lo; other < lo + length; ++other)
        {
            if (other == slot) continue;
            const V4 q = sorted[other];
            T dx, dy, dz;
            pair_vector(wraps, c.x, c.y, c.z, q.x, q.y, q.z, v, dx, dy, dz);
            const T r2 = exact_squared(dx, dy, dz);
            if (!(r2 < v.cutoff_squared)) continue;
            T u, fs;
            pair_terms(v, a.knots, r2, u, fs);
            e += u;
            fx += fs * dx;
            fy += fs * dy;
            fz += fs * dz;
            w[0] += dx * (fs * dx);
            w[1] += dy * (fs * dy);
            w[2] += dz * (fs * dz);
            w[3] += dx * (fs * dy);
            w[4] += dx * (fs * dz);
            w[5] += dy * (fs * dz);
        }
    }
    T* f = a.forces + 3LL * atom;
    f[0] = fx;
    f[1] = fy;
    f[2] = fz;
    T* terms = a.atom_terms + 7LL * atom;
    terms[0] = T(0.5) * e;
    for (int k = 0; k < 6; ++k) terms[1 + k] = T(0.5) * w[k];
}

// The table's gradient (the vector-Jacobian product of E, F and W with upstream gE [S],
// gF [N, 3], gW [S, 9]): wave per atom over the same stencil; each hit pair adds, to the four
// padded knots of its segment, gE du/dk - ((gF_i - gF_j) . r_ij + r_ij' gW r_ij) / r d(du/dr)/dk,
// halved because every pair is met from both of its atoms. E, F and W are linear in the knots,
// so these weights are the exact derivatives. Per-block sums in LDS (fp64), written per block.
template <typename T>
__global__ void __launch_bounds__(kBlock) batch_table_vjp_kernel(BatchArgs<T> a, T cull_factor,
                                                                 const T* __restrict__ grad_energy,
                                                                 const T* __restrict__ grad_forces,
                                                                 const T* __restrict__ grad_virial,
                                                                 double* __restrict__ partials)
{
    using V4 = typename std::conditional<sizeof(T) == 4, float4, double4>::type;
    extern __shared__ double knot_sums[];
    const int width = a.knots + 2;
    for (int k = threadIdx.x; k < width; k += blockDim.x) knot_sums[k] = 0.0;
    __syncthreads();
    const std::int64_t slot =
        static_cast<std::int64_t>(blockIdx.x) * (kBlock / kWave) + threadIdx.x / kWave;
    if (slot < a.num_atoms)
    {
        const int lane = lane_id();
        const V4* sorted = reinterpret_cast<const V4*>(a.sorted4);
        const index_t atom = a.order[slot];
        const index_t s = a.system_of[atom];
        const SystemView<T> v = system_view(a, s);
        if (v.kind == NDN_TABLE)
        {
            const V4 c = sorted[slot];
            const T cull = v.cutoff * cull_factor;
            index_t lo, length;
            bool wraps;
            stencil_run(a, v, c.x, c.y, c.z, lane, cull * cull, lo, length, wraps);
            const index_t inclusive = wave_inclusive_sum(length);
            const index_t start = inclusive - length;
            const index_t total = __shfl(inclusive, kWave - 1, kWave);
            const T ge = grad_energy[s];
            const T* gw = grad_virial + 9LL * s;
            const T gix = grad_forces[3LL * atom], giy = grad_forces[3LL * atom + 1],
                    giz = grad_forces[3LL * atom + 2];
            const std::int64_t row_base = static_cast<std::int64_t>(a.table_of[s]) * width;
            (void)row_base;
            for (index_t chunk = 0; chunk < total; chunk += kWave)
            {
                const index_t t = chunk + lane;
                int r = 0;
#pragma unroll
                for (int step = 32; step > 0; step >>= 1)
                {
                    const index_t st = __shfl(start, r + step, kWave);
                    if (st <= t) r += step;
                }
                const index_t other = __shfl(lo, r, kWave) + (t - __shfl(start, r, kWave));
                if (t < total && other != slot)
                {
                    const V4 q = sorted[other];
                    T dx, dy, dz;
                    pair_vector(wraps, c.x, c.y, c.z, q.x, q.y, q.z, v, dx, dy, dz);
                    const T r2 = exact_squared(dx, dy, dz);
                    if (r2 < v.cutoff_squared)
                    {
                        const index_t j = a.order[other];
                        const T dist = sqrt(r2);
                        const T x = (dist - v.table_start) / v.table_spacing;
                        T segment = floor(x);
                        segment = segment < T(0) ? T(0)
                                : (segment > T(a.knots - 2) ? T(a.knots - 2) : segment);
                        const T tt = x - segment;
                        const bool below = tt < T(0);
                        const T sv = below ? T(0) : tt;
                        T du[4], dslope[4];
                        if (below)
                        {
                            du[0] = T(-0.5) * tt;
                            du[1] = T(1);
                            du[2] = T(0.5) * tt;
                            du[3] = T(0);
                            dslope[0] = T(-0.5);
                            dslope[1] = T(0);
                            dslope[2] = T(0.5);
                            dslope[3] = T(0);
                        }
                        else
                        {
                            const T s2 = sv * sv, s3 = s2 * sv;
                            du[0] = T(-0.5) * sv + s2 - T(0.5) * s3;
                            du[1] = T(1) - T(2.5) * s2 + T(1.5) * s3;
                            du[2] = T(0.5) * sv + T(2) * s2 - T(1.5) * s3;
                            du[3] = T(-0.5) * s2 + T(0.5) * s3;
                            dslope[0] = T(-0.5) + T(2) * sv - T(1.5) * s2;
                            dslope[1] = T(-5) * sv + T(4.5) * s2;
                            dslope[2] = T(0.5) + T(4) * sv - T(4.5) * s2;
                            dslope[3] = -sv + T(1.5) * s2;
                        }
                        const T gjx = grad_forces[3LL * j], gjy = grad_forces[3LL * j + 1],
                                gjz = grad_forces[3LL * j + 2];
                        const T projection = (gix - gjx) * dx + (giy - gjy) * dy + (giz - gjz) * dz;
                        const T quadratic =
                            dx * (gw[0] * dx + gw[1] * dy + gw[2] * dz) +
                            dy * (gw[3] * dx + gw[4] * dy + gw[5] * dz) +
                            dz * (gw[6] * dx + gw[7] * dy + gw[8] * dz);
                        // dF and dW weights: d(-(du/dr)/r) = -(d(du/dt) / h) / r
                        const T slope_weight =
                            -((projection + quadratic) / v.table_spacing) / dist;
                        const int base = static_cast<int>(segment);
                        for (int m = 0; m < 4; ++m)
                        {
                            const double g = 0.5 * (static_cast<double>(ge) * du[m] +
                                                    static_cast<double>(slope_weight) * dslope[m]);
                            atomicAdd(knot_sums + base + m, g);
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < width; k += blockDim.x)
        partials[static_cast<std::int64_t>(blockIdx.x) * width + k] = knot_sums[k];
}

// Folds the block partials [blocks, K + 2] onto their first `folds` rows: fold f sums rows f,
// f + folds, f + 2 folds, ... in that order (coalesced rows, a thread per padded knot) and writes
// the sum over row f, which only fold f reads.
__global__ void __launch_bounds__(kBlock) table_vjp_fold_kernel(double* __restrict__ partials,
                                                                int blocks, int width)
{
    const int folds = gridDim.x;
    const int f = blockIdx.x;
    for (int k = threadIdx.x; k < width; k += blockDim.x)
    {
        double sum = 0.0;
        for (int b = f; b < blocks; b += folds) sum += partials[static_cast<std::int64_t>(b) * width + k];
        partials[static_cast<std::int64_t>(f) * width + k] = sum;
    }
}

// Sums the block partials per padded knot in a fixed order, then maps the padded knots back to
// the table: the virtual first knot is 3 v0 - 3 v1 + v2, the virtual last 3 v_{K-1} - 3 v_{K-2}
// + v_{K-3} with v_{K-1} held at 0, so the last knot's gradient is 0.
template <typename T>
__global__ void __launch_bounds__(kBlock) table_vjp_finish_kernel(const double* __restrict__ partials,
                                                                  int blocks, int knots,
                                                                  T* __restrict__ grad_table)
{
    __shared__ double padded[4096];
    const int width = knots + 2;
    for (int k = threadIdx.x; k < width; k += blockDim.x)
    {
        double sum = 0.0;
        for (int b = 0; b < blocks; ++b) sum += partials[static_cast<std::int64_t>(b) * width + k];
        padded[k] = sum;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < knots; k += blockDim.x)
    {
        double g = padded[k + 1];
        if (k == 0) g += 3.0 * padded[0];
        if (k == 1) g -= 3.0 * padded[0];
        if (k == 2) g += padded[0];
        if (k == knots - 2) g -= 3.0 * padded[width - 1];
        if (k == knots - 3) g += padded[width - 1];
        if (k == knots - 1) g = 0.0;
        grad_table[k] = static_cast<T>(g);
    }
}

// Block per system: E and W from the atoms' terms, in a fixed order.
// The largest system's block is the launch's length: 1,024 threads, each reading the terms of
// four slots before it adds any.
constexpr int kReduceThreads = 1024;

template <typename T>
__global__ void __launch_bounds__(kReduceThreads) batch_reduce_kernel(BatchArgs<T> a)
{
    __shared__ double shared[16];
    constexpr int kInFlight = 4;
    const std::int64_t s = blockIdx.x;
    if (s >= a.num_systems) return;
    const std::int64_t end = a.atom_start[s + 1];
    double sums[7] = {0, 0, 0, 0, 0, 0, 0};
    for (std::int64_t base = a.atom_start[s] + threadIdx.x; base < end;
         base += kInFlight * kReduceThreads)
    {
        T terms[kInFlight][7];
#pragma unroll
        for (int u = 0; u < kInFlight; ++u)
        {
            const std::int64_t slot = base + u * kReduceThreads;
            for (int k = 0; k < 7; ++k) terms[u][k] = slot < end ? a.atom_terms[7 * slot + k] : T(0);
        }
#pragma unroll
        for (int u = 0; u < kInFlight; ++u)
            for (int k = 0; k < 7; ++k) sums[k] += static_cast<double>(terms[u][k]);
    }
    for (int k = 0; k < 7; ++k) sums[k] = block_sum(sums[k], shared);
    if (threadIdx.x == 0)
    {
        a.energy[s] = static_cast<T>(sums[0]);
        const double xx = sums[1], yy = sums[2], zz = sums[3], xy = sums[4], xz = sums[5],
                     yz = sums[6];
        const double out[9] = {xx, xy, xz, xy, yy, yz, xz, yz, zz};
        for (int k = 0; k < 9; ++k) a.virial[9 * s + k] = static_cast<T>(out[k]);
    }
}

// How the wave schedule splits a batch.
struct WaveShares
{
    std::int64_t waves, bins;
    index_t share;
};

// Batches with fewer atoms than sub-bins go by slot: a wave per sub-bin finds most of them empty (40
// systems of 500 atoms in boxes of 20 nm, sub-bins of half the cutoff: LJ 257 -> 65 us an
// evaluation, tables 180 -> 61). With fewer sub-bins than waves fill the chip twice over (256
// units of 4 SIMDs of 7), every group is a wave's own (20 systems of 4,000 atoms at 100 a nm3: LJ
// 310 -> 233, tables 957 -> 459). Above, a wave takes four groups, which costs the uniform frames
// nothing (the 256 systems 1,468 us with four or 32) and spreads a clump (100 systems of 9,000
// atoms beside one whose half lies in a clump: LJ 6,125 us with a wave per sub-bin, 2,386 with 32
// groups a wave, 1,093 with four).
inline WaveShares wave_shares(std::int64_t atoms, std::int64_t bins)
{
    if (atoms < bins) return {atoms, 0, 1};
    const index_t share = bins < 16384 ? kWaveCenters : 4 * kWaveCenters;
    return {bins + (atoms + share - 1) / share, bins, share};
}

template <typename T>
BatchArgs<T> batch_args(const ndn_batch& b);

template <typename T>
int batch_impl(const ndn_batch& b, int schedule, hipStream_t stream)
{
    const BatchArgs<T> a = batch_args<T>(b);
    const std::int64_t n = b.num_atoms;
    batch_assign_kernel<T><<<blocks_for(n), kBlock, 0, stream>>>(a);
    NDN_LAUNCHED("batch_assign");
    const int scanned = exclusive_scan(a.bin_counts, a.bin_offsets, a.total_bins + 1, a.scan_temp,
                                       nullptr, b.status, stream);
    if (scanned != NDN_OK) return scanned;
    batch_scatter_kernel<T><<<blocks_for(n), kBlock, 0, stream>>>(a);
    NDN_LAUNCHED("batch_scatter");
    batch_order_kernel<T><<<blocks_for(n), kBlock, 0, stream>>>(a);
    NDN_LAUNCHED("batch_order");
    // sub-bins of the cutoff / span: culling keeps every one a pair within it could sit in
    const T cull_factor = static_cast<T>(1.0 + 1e-4);
    if (schedule == 0)
        batch_thread_kernel<T><<<blocks_for(n), kBlock, 0, stream>>>(a, cull_factor);
    else
    {
        const WaveShares w = wave_shares(n, a.total_bins);
        batch_wave_kernel<T><<<blocks_for(w.waves, kBlock / kWave), kBlock, 0, stream>>>(
            a, cull_factor, w.bins, w.share);
    }
    NDN_LAUNCHED("batch_forces");
    batch_reduce_kernel<T><<<static_cast<unsigned>(b.num_systems), kReduceThreads, 0, stream>>>(a);
    NDN_LAUNCHED("batch_reduce");
    return NDN_OK;
}

template <typename T>
BatchArgs<T> batch_args(const ndn_batch& b)
{
    BatchArgs<T> a{};
    a.positions = static_cast<const T*>(b.positions);
    a.num_atoms = static_cast<index_t>(b.num_atoms);
    a.num_systems = b.num_systems;
    a.system_of = b.system_of;
    a.atom_start = b.atom_start;
    a.bin_start = b.bin_start;
    a.dims = b.dims;
    a.widths = static_cast<const T*>(b.widths);
    a.cells = static_cast<const T*>(b.cells);
    a.cutoffs = static_cast<const T*>(b.cutoffs);
    a.cutoffs_squared = static_cast<const T*>(b.cutoffs_squared);
    a.kinds = b.kinds;
    a.lj = static_cast<const LJRow<T>*>(b.lj_rows);
    a.table_of = b.table_of;
    a.tables = static_cast<const T*>(b.tables);
    a.table_start = static_cast<const T*>(b.table_start);
    a.table_spacing = static_cast<const T*>(b.table_spacing);
    a.knots = static_cast<int>(b.knots);
    a.total_bins = b.total_bins;
    a.span = b.span;
    a.bin_of = b.bin_of;
    a.bin_counts = b.bin_counts;
    a.bin_offsets = b.bin_offsets;
    a.unordered = b.unordered;
    a.order = b.order;
    a.wrapped4 = static_cast<T*>(b.wrapped4);
    a.sorted4 = static_cast<T*>(b.sorted4);
    a.scan_temp = b.scan_temp;
    a.forces = static_cast<T*>(b.forces);
    a.atom_terms = static_cast<T*>(b.atom_terms);
    a.energy = static_cast<T*>(b.energy);
    a.virial = static_cast<T*>(b.virial);
    return a;
}

template <typename T>
int table_vjp_impl(const ndn_batch& b, const void* grad_energy, const void* grad_forces,
                   const void* grad_virial, double* partials, void* grad_table, hipStream_t stream)
{
    const BatchArgs<T> a = batch_args<T>(b);
    const std::int64_t n = b.num_atoms;
    const unsigned blocks = blocks_for(n, kBlock / kWave);
    const T cull_factor = static_cast<T>(1.0 + 1e-4);
    const std::size_t lds = static_cast<std::size_t>(b.knots + 2) * sizeof(double);
    batch_table_vjp_kernel<T><<<blocks, kBlock, lds, stream>>>(
        a, cull_factor, static_cast<const T*>(grad_energy), static_cast<const T*>(grad_forces),
        static_cast<const T*>(grad_virial), partials);
    NDN_LAUNCHED("batch_table_vjp");
    // two fixed-order passes: the block rows folded onto at most 512 rows, then summed
    const int width = static_cast<int>(b.knots) + 2;
    const int folds = static_cast<int>(std::min<std::int64_t>(blocks, 512));
    table_vjp_fold_kernel<<<folds, kBlock, 0, stream>>>(partials, static_cast<int>(blocks), width);
    NDN_LAUNCHED("table_vjp_fold");
    table_vjp_finish_kernel<T><<<1, kBlock, 0, stream>>>(partials, folds,
                                                         static_cast<int>(b.knots),
                                                         static_cast<T*>(grad_table));
    NDN_LAUNCHED("table_vjp_finish");
    return NDN_OK;
}

}  // namespace ndn

using namespace ndn;

extern "C" {

int64_t ndn_batch_scan_bytes(int64_t total_bins)
{
    return scan_bytes(total_bins + 2);
}

int64_t ndn_batch_vjp_bytes(int64_t num_atoms, int64_t knots)
{
    return ((num_atoms + (kBlock / kWave) - 1) / (kBlock / kWave)) * (knots + 2) *
           static_cast<int64_t>(sizeof(double));
}

int ndn_batch_table_vjp(int dtype, const ndn_batch* batch, const void* grad_energy,
                        const void* grad_forces, const void* grad_virial, void* workspace,
                        int64_t workspace_bytes, void* grad_table, ndn_stream_t stream)
{
    NDN_REQUIRE(batch != nullptr && grad_energy && grad_forces && grad_virial && workspace &&
                    grad_table,
                "a buffer is null");
    NDN_REQUIRE(batch->tables != nullptr && batch->knots >= 4 && batch->knots + 2 <= 4096,
                "the table gradient needs tables of 4 to 4094 knots");
    NDN_REQUIRE(workspace_bytes >= ndn_batch_vjp_bytes(batch->num_atoms, batch->knots),
                "the workspace is too small");
    NDN_REQUIRE(batch->span == 1 || batch->span == 2, "span must be 1 or 2");
    if (dtype == NDN_F32)
        return table_vjp_impl<float>(*batch, grad_energy, grad_forces, grad_virial,
                                     static_cast<double*>(workspace), grad_table, stream);
    NDN_REQUIRE(dtype == NDN_F64, "dtype must be NDN_F32 or NDN_F64");
    return table_vjp_impl<double>(*batch, grad_energy, grad_forces, grad_virial,
                                  static_cast<double*>(workspace), grad_table, stream);
}

int ndn_batch_efw(int dtype, const ndn_batch* batch, int schedule, ndn_stream_t stream)
{
    NDN_REQUIRE(batch != nullptr, "the batch must not be null");
    const ndn_batch& b = *batch;
    NDN_REQUIRE(b.num_systems >= 1 && b.num_atoms >= 1 && b.num_atoms <= INT32_MAX,
                "a batch needs systems and at most 2**31 - 1 atoms");
    NDN_REQUIRE(b.positions && b.system_of && b.atom_start && b.bin_start && b.dims && b.widths &&
                    b.cells && b.cutoffs && b.cutoffs_squared && b.kinds && b.lj_rows && b.table_of && b.bin_of &&
                    b.bin_counts && b.bin_offsets && b.unordered && b.order && b.wrapped4 &&
                    b.sorted4 && b.scan_temp && b.forces && b.atom_terms && b.energy &&
                    b.virial && b.status,
                "a batch buffer is null");
    NDN_REQUIRE(b.total_bins >= 1 && b.total_bins < INT32_MAX, "bad bin count");
    NDN_REQUIRE(b.scan_temp_bytes >= scan_bytes(b.total_bins + 2), "scan_temp is too small");
    NDN_REQUIRE(b.span == 1 || b.span == 2, "span must be 1 or 2");
    NDN_REQUIRE(schedule == 0 || schedule == 1, "schedule must be 0 (thread) or 1 (wave)");
    NDN_REQUIRE(b.tables == nullptr || b.knots >= 4, "tables need at least 4 knots");
    if (dtype == NDN_F32) return batch_impl<float>(b, schedule, stream);
    NDN_REQUIRE(dtype == NDN_F64, "dtype must be NDN_F32 or NDN_F64");
    return batch_impl<double>(b, schedule, stream);
}

}  // extern "C"
