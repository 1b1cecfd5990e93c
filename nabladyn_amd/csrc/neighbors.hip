// The neighbor list on gfx950: reuse check, cell binning, pair count and fill (the reference's
// half list, in its column order, plus an optional full list for the fused force kernels),
// total, padding and commit. Built with -ffp-contract=off: every distance is the source-text
// IEEE expression (dx dx + dy dy) + dz dz, rounded step by step, so the pair set is bit-exact
// with a scalar CPU evaluation of the same expression.
//
// Reference semantics followed (paths under src/nabladyn/neighbors/csrc/):
//   update/update.cuh:27-75 prepare, :79-116 reuse check, :119-145 commit;
//   grid/grid.cuh:10-118 binning and (bin, atom id) order; pairs/pairs.cuh:43-157 count, fill,
//   total, pad; pairs/all_pairs.cuh:29-114 all-pairs path; common/traversal.cuh:12-147 visit
//   order and periodic images; runtime/entry_points.cu:127-508 launch order and gating.

#include <algorithm>
#include <climits>
#include <limits>
#include <mutex>
#include <string>

#include "common.hpp"
#include "neighbors.hpp"
#include "scan.hpp"

namespace ndn {

namespace {
thread_local std::string g_last_error;
}

void set_error(const std::string& message)
{
    g_last_error = message;
}

const char* last_error()
{
    return g_last_error.c_str();
}

// ---- geometry -------------------------------------------------------------------------------

__device__ __forceinline__ index_t wrap_bin(index_t home, int step, index_t count)
{
    const index_t bin = home + step;
    return bin < 0 ? bin + count : (bin >= count ? bin - count : bin);
}

template <typename T>
__device__ __forceinline__ T bin_shift(index_t home, int step, index_t count, T length)
{
    const index_t bin = home + step;
    return bin < 0 ? -length : (bin >= count ? length : T(0));
}

template <typename T>
__device__ __forceinline__ index_t axis_bin(T x, T width, index_t count)
{
    const index_t bin = static_cast<index_t>(floor(x / width));
    return bin < 0 ? 0 : (bin >= count ? count - 1 : bin);
}

template <typename T>
__device__ __forceinline__ T squared(T dx, T dy, T dz)
{
    return dx * dx + dy * dy + dz * dz;
}

// ---- prepare and reuse ----------------------------------------------------------------------

template <typename T>
__global__ void prepare_update_kernel(const T* __restrict__ cell,
                                      const T* __restrict__ reference_cell, T cutoff, T radius,
                                      const index_t* __restrict__ limits, index_t* dims, T* widths,
                                      T* reuse, index_t* rebuild, index_t* status,
                                      const index_t* pair_total, ListHeader* header)
{
    prepare_update(cell, reference_cell, cutoff, radius, limits, dims, widths, reuse, rebuild,
                   status, pair_total, header);
}

// One atom per lane: flags a non-finite coordinate, and reduces the squared displacement since
// the last rebuild over the wave. Its maximum decides the rebuild: max >= threshold is the
// reference's "any atom moved at least the threshold", bit for bit.
template <typename T>
__global__ void __launch_bounds__(kBlock) check_reuse_kernel(
    const T* __restrict__ positions, const T* __restrict__ reference_positions,
    const T* __restrict__ cell, const T* __restrict__ reuse, index_t num_atoms, index_t* rebuild,
    index_t* status, ListHeader* header)
{
    __shared__ T block_max[kBlock / kWave];
    // every thread reaches the barrier below, whatever status a wave reads
    const bool active = status[0] == 0;
    const std::int64_t atom = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    bool finite = true;
    T moved = 0;
    if (active && atom < num_atoms)
    {
        const T x = positions[3 * atom], y = positions[3 * atom + 1], z = positions[3 * atom + 2];
        finite = isfinite(x) && isfinite(y) && isfinite(z);
        if (finite) moved = moved_squared(x, y, z, reference_positions + 3 * atom, reuse, cell);
    }
    if (!finite) atomicOr(status, kStatusNonFinite);
    const T wave_moved = wave_max(finite ? moved : T(0));
    if (lane_id() == 0)
    {
        block_max[threadIdx.x / kWave] = wave_moved;
        if (active && wave_moved >= reuse[0] && rebuild[0] == 0) rebuild[0] = 1;
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        T m = block_max[0];
        for (int w = 1; w < kBlock / kWave; ++w) m = block_max[w] > m ? block_max[w] : m;
        if (m > T(0)) atomicMax(moved_slot(header, blockIdx.x), order_bits(m));
    }
}

// ---- grid: bins, counting sort, deterministic in-bin order ----------------------------------

template <typename T>
__global__ void __launch_bounds__(kBlock) assign_bins_kernel(
    const T* __restrict__ positions, const index_t* __restrict__ dims,
    const T* __restrict__ widths, index_t num_atoms, index_t* __restrict__ atom_bin,
    index_t* __restrict__ bin_counts, index_t* __restrict__ full_slices, const index_t* rebuild,
    const index_t* status)
{
    const std::int64_t atom = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (atom >= num_atoms || !rebuilding(rebuild, status)) return;
    // the full rows' slice widths start at 0: the count raises each to its widest row
    if (full_slices != nullptr && atom % kWave == 0) full_slices[atom / kWave] = 0;
    const T* p = positions + 3 * atom;
    const index_t nx = dims[0], ny = dims[1];
    const index_t bin = axis_bin(p[0], widths[0], nx) +
                        nx * (axis_bin(p[1], widths[1], ny) + ny * axis_bin(p[2], widths[2], dims[2]));
    atom_bin[atom] = bin;
    // one atomic per run of a bin's atoms in neighbouring lanes
    const LaneRun run = equal_runs(bin);
    if (run.head) atomicAdd(bin_counts + bin, run.length);
}

// Places each atom in its bin's slice in the order of the atomics; the counts return to zero.
__global__ void __launch_bounds__(kBlock) scatter_atoms_kernel(
    const index_t* __restrict__ atom_bin, const index_t* __restrict__ bin_offsets,
    index_t num_atoms, index_t* __restrict__ bin_counts, index_t* __restrict__ unordered_ids,
    const index_t* rebuild, const index_t* status)
{
    const std::int64_t atom = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (atom >= num_atoms || !rebuilding(rebuild, status)) return;
    const index_t bin = atom_bin[atom];
    // one atomic per run of a bin's atoms: the run's lanes take the places below the count it
    // returns, one each (order_bins_kernel ranks a bin's atoms by id after)
    const LaneRun run = equal_runs(bin);
    index_t count = 0;
    if (run.head) count = atomicSub(bin_counts + bin, run.length);
    count = __shfl(count, run.first, kWave);
    unordered_ids[bin_offsets[bin] + count - 1 - (lane_id() - run.first)] =
        static_cast<index_t>(atom);
}

// One wave per bin: ranks each atom among its bin's ids (readlane broadcasts, no atomics), so the
// order inside a bin is by atom id whatever the atomics did, then writes the sorted ids and
// gathers the sorted positions.
template <typename T>
__global__ void __launch_bounds__(kBlock) order_bins_kernel(
    const T* __restrict__ positions, const index_t* __restrict__ unordered_ids,
    const index_t* __restrict__ bin_offsets, const index_t* __restrict__ dims,
    std::int64_t bin_slots, index_t* __restrict__ sorted_ids, T* __restrict__ sorted_positions,
    const index_t* rebuild, const index_t* status)
{
    if (!rebuilding(rebuild, status)) return;
    const std::int64_t bin =
        static_cast<std::int64_t>(blockIdx.x) * (kBlock / kWave) + threadIdx.x / kWave;
    const std::int64_t bins = static_cast<std::int64_t>(dims[0]) * dims[1] * dims[2];
    if (bin >= bins || bin >= bin_slots - 1) return;
    const int lane = lane_id();
    const index_t begin = bin_offsets[bin];
    const index_t end = bin_offsets[bin + 1];
    for (index_t chunk = begin; chunk < end; chunk += kWave)
    {
        const bool mine = chunk + lane < end;
        const index_t id = mine ? unordered_ids[chunk + lane] : INT_MAX;
        index_t rank = 0;
        for (index_t other = begin; other < end; other += kWave)
        {
            const index_t theirs = other + lane < end ? unordered_ids[other + lane] : INT_MAX;
            const int live = end - other < kWave ? end - other : kWave;
            for (int m = 0; m < live; ++m)
            {
                rank += __shfl(theirs, m, kWave) < id;
            }
        }
        if (mine)
        {
            const index_t slot = begin + rank;
            sorted_ids[slot] = id;
            const T* p = positions + 3LL * id;
            T* q = sorted_positions + 3LL * slot;
            q[0] = p[0];
            q[1] = p[1];
            q[2] = p[2];
        }
    }
}

// ---- pair visit: a lane per center, for sparse grids ----------------------------------------

// Visits, for sorted center `center`, every candidate in the reference's order (neighbor bins
// z, y, x from -1 to +1; candidates ascending) and calls visit(neighbor, after) for each one
// closer than the list radius, after = neighbor > center. Half lists visit only candidates
// after the center, as the reference does; full lists visit all other candidates.
template <typename T, bool kFull, typename Visit>
__device__ __forceinline__ void visit_grid(const T* __restrict__ sp,
                                           const index_t* __restrict__ bin_offsets, index_t home,
                                           index_t nx, index_t ny, index_t nz, T lx, T ly, T lz,
                                           T radius_squared, index_t center, Visit& visit)
{
    const T cx = sp[3LL * center], cy = sp[3LL * center + 1], cz = sp[3LL * center + 2];
    const index_t hx = home % nx, hy = (home / nx) % ny, hz = home / (nx * ny);
    if (nx >= 3 && ny >= 3 && nz >= 3)
    {
        for (int sz = -1; sz <= 1; ++sz)
        {
            const T shz = bin_shift(hz, sz, nz, lz);
            const T az = shz > T(0) ? cz - shz : cz;
            const T bz_shift = shz < T(0) ? shz : T(0);
            const index_t bz = wrap_bin(hz, sz, nz);
            for (int sy = -1; sy <= 1; ++sy)
            {
                const T shy = bin_shift(hy, sy, ny, ly);
                const T ay = shy > T(0) ? cy - shy : cy;
                const T by_shift = shy < T(0) ? shy : T(0);
                const index_t by = wrap_bin(hy, sy, ny);
                for (int sx = -1; sx <= 1; ++sx)
                {
                    const T shx = bin_shift(hx, sx, nx, lx);
                    const T ax = shx > T(0) ? cx - shx : cx;
                    const T bx_shift = shx < T(0) ? shx : T(0);
                    const index_t bin = wrap_bin(hx, sx, nx) + nx * (by + ny * bz);
                    const index_t first = bin_offsets[bin];
                    const index_t end = bin_offsets[bin + 1];
                    const index_t start = kFull ? first : (first > center ? first : center + 1);
                    for (index_t nb = start; nb < end; ++nb)
                    {
                        const T* p = sp + 3LL * nb;
                        const T dx = ax - (p[0] + bx_shift);
                        const T dy = ay - (p[1] + by_shift);
                        const T dz = az - (p[2] + bz_shift);
                        if (squared(dx, dy, dz) < radius_squared && nb != center)
                        {
                            visit(nb, nb > center);
                        }
                    }
                }
            }
        }
        return;
    }
    // A short axis (fewer than three bins): every bin along it, minimum image per candidate.
    const int span_x = nx >= 3 ? 3 : nx, span_y = ny >= 3 ? 3 : ny, span_z = nz >= 3 ? 3 : nz;
    for (int iz = 0; iz < span_z; ++iz)
    {
        const index_t bz = nz >= 3 ? wrap_bin(hz, iz - 1, nz) : iz;
        for (int iy = 0; iy < span_y; ++iy)
        {
            const index_t by = ny >= 3 ? wrap_bin(hy, iy - 1, ny) : iy;
            for (int ix = 0; ix < span_x; ++ix)
            {
                const index_t bin = (nx >= 3 ? wrap_bin(hx, ix - 1, nx) : ix) + nx * (by + ny * bz);
                const index_t first = bin_offsets[bin];
                const index_t end = bin_offsets[bin + 1];
                const index_t start = kFull ? first : (first > center ? first : center + 1);
                for (index_t nb = start; nb < end; ++nb)
                {
                    const T* p = sp + 3LL * nb;
                    const T dx = minimum_image(cx, p[0], lx);
                    const T dy = minimum_image(cy, p[1], ly);
                    const T dz = minimum_image(cz, p[2], lz);
                    if (squared(dx, dy, dz) < radius_squared && nb != center)
                    {
                        visit(nb, nb > center);
                    }
                }
            }
        }
    }
}

struct CountVisit
{
    index_t half = 0;
    index_t full = 0;
    __device__ __forceinline__ void operator()(index_t, bool after)
    {
        half += after;
        ++full;
    }
};

struct FillVisit
{
    const index_t* __restrict__ sorted_ids;
    index_t center_id;
    std::int64_t column;
    std::int64_t capacity;
    index_t* __restrict__ pairs;
    // full list
    index_t* __restrict__ full_index;
    std::int64_t full_slot;     // slice base + lane within slice
    std::int64_t full_capacity;
    __device__ __forceinline__ void operator()(index_t nb, bool after)
    {
        const index_t id = sorted_ids[nb];
        if (after)
        {
            if (column < capacity)
            {
                pairs[column] = center_id;
                pairs[capacity + column] = id;
            }
            ++column;
        }
        if (full_index != nullptr)
        {
            if (full_slot < full_capacity) full_index[full_slot] = id;
            full_slot += kWave;
        }
    }
};

// Thread per sorted center. Writes the half count (and with a full list the full count, and
// the slice widths: 64 * the largest full count of each 64 rows) for the scans that follow.
template <typename T, bool kFull>
__global__ void __launch_bounds__(kBlock) count_pairs_kernel(
    const T* __restrict__ sp, const index_t* __restrict__ sorted_ids,
    const index_t* __restrict__ atom_bin, const index_t* __restrict__ bin_offsets,
    const index_t* __restrict__ dims, const T* __restrict__ cell, T radius_squared,
    index_t num_atoms, index_t* __restrict__ pair_counts, index_t* __restrict__ full_counts,
    index_t* __restrict__ full_slices, const index_t* rebuild, const index_t* status)
{
    if (!rebuilding(rebuild, status)) return;
    const std::int64_t center = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    CountVisit visit;
    if (center < num_atoms)
    {
        visit_grid<T, kFull>(sp, bin_offsets, atom_bin[sorted_ids[center]], dims[0], dims[1],
                             dims[2], cell[0], cell[1], cell[2], radius_squared,
                             static_cast<index_t>(center), visit);
        pair_counts[center] = visit.half;
        if (kFull) full_counts[center] = visit.full;
    }
    if (kFull)
    {
        const index_t width = wave_max(center < num_atoms ? visit.full : 0);
        const std::int64_t slice = center / kWave;
        if (lane_id() == 0 && slice * kWave < num_atoms) full_slices[slice] = width * kWave;
    }
}

template <typename T, bool kFull>
__global__ void __launch_bounds__(kBlock) fill_pairs_kernel(
    const T* __restrict__ sp, const index_t* __restrict__ sorted_ids,
    const index_t* __restrict__ atom_bin, const index_t* __restrict__ bin_offsets,
    const index_t* __restrict__ dims, const T* __restrict__ cell,
    const index_t* __restrict__ pair_offsets, T radius_squared, index_t num_atoms,
    std::int64_t capacity, index_t* __restrict__ pairs, const index_t* __restrict__ full_slices,
    index_t* __restrict__ full_index, std::int64_t full_capacity, const index_t* rebuild,
    const index_t* status)
{
    const std::int64_t center = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (center >= num_atoms || !rebuilding(rebuild, status)) return;
    FillVisit visit{sorted_ids, sorted_ids[center], pair_offsets[center], capacity, pairs,
                    kFull ? full_index : nullptr,
                    kFull ? full_slices[center / kWave] + center % kWave : 0, full_capacity};
    visit_grid<T, kFull>(sp, bin_offsets, atom_bin[sorted_ids[center]], dims[0], dims[1], dims[2],
                         cell[0], cell[1], cell[2], radius_squared, static_cast<index_t>(center),
                         visit);
}

// ---- pair search ----------------------------------------------------------------------------

// Centers a wave tests against each chunk of 64 candidates: with 8 in fp32 the scalar registers
// no longer hold the centers and their masks (2.24 ms a rebuild at 2,097,152 atoms, radius 1.1
// nm, against 2.17).
constexpr int kSearchCenters = 4;
constexpr int kSearchRanges = 32;  // lanes that may hold a range of candidates (18 are used)

// How a candidate's vector is formed, uniform over a wave's centers (one bin).
constexpr int kSearchPlain = 0;    // every candidate bin inside the box: center - candidate
constexpr int kSearchShifted = 1;  // some bins across a face: the near-face coordinate shifted
constexpr int kSearchImage = 2;    // an axis of fewer than three bins: minimum image per pair

template <typename T>
struct SearchArgs
{
    const T* sp;                  // [N, 3] positions in slot order
    const index_t* sorted_ids;    // slot -> atom
    const index_t* bin_offsets;
    const index_t* dims;
    const T* cell;
    T radius_squared;
    const index_t* atom_bin;
    index_t num_atoms;
    index_t share;                // slots of a bin to a block
    std::int64_t bin_slots;
    // count
    index_t* pair_counts;
    index_t* full_counts;
    index_t* full_slices;         // zero before the count; the fill reads their prefix sums
    // fill
    const index_t* pair_offsets;
    index_t* pairs;
    std::int64_t capacity;
    index_t* full_index;
    std::int64_t full_capacity;
    const index_t* rebuild;
    const index_t* status;
};

// The candidate ranges of a bin, one per lane, in the reference's visit order (bins z, y, x from
// -1 to +1): consecutive bins along x are consecutive slots, so a (z, y) row is one range, or two
// where it crosses an x face. `shift` holds two bits per axis: 1 below the box (the candidate
// moves down by L), 2 above it (the center does).
struct SearchRange
{
    index_t lo, length;
    int shift;
};

template <typename T>
__device__ __forceinline__ SearchRange search_range(const SearchArgs<T>& a, index_t hx, index_t hy,
                                                    index_t hz, index_t nx, index_t ny, index_t nz,
                                                    int lane)
{
    SearchRange r{0, 0, 0};
    const int span_y = ny >= 3 ? 3 : ny, span_z = nz >= 3 ? 3 : nz;
    const int row = lane / 2, part = lane % 2;
    if (row >= span_y * span_z) return r;
    const int oy = row % span_y, oz = row / span_y;
    const index_t ry = ny >= 3 ? hy + oy - 1 : oy, rz = nz >= 3 ? hz + oz - 1 : oz;
    const index_t by = ry < 0 ? ry + ny : (ry >= ny ? ry - ny : ry);
    const index_t bz = rz < 0 ? rz + nz : (rz >= nz ? rz - nz : rz);
    r.shift = (ry < 0 ? 4 : (ry >= ny ? 8 : 0)) | (rz < 0 ? 16 : (rz >= nz ? 32 : 0));
    index_t first = 0, last = -1;
    if (nx < 3)
    {
        if (part == 0) last = nx - 1;
    }
    else if (hx == 0)
    {
        first = part == 0 ? nx - 1 : 0;
        last = part == 0 ? nx - 1 : 1;
        if (part == 0) r.shift |= 1;
    }
    else if (hx == nx - 1)
    {
        first = part == 0 ? nx - 2 : 0;
        last = part == 0 ? nx - 1 : 0;
        if (part == 1) r.shift |= 2;
    }
    else if (part == 0)
    {
        first = hx - 1;
        last = hx + 1;
    }
    if (last < first) return r;
    const index_t base = nx * (by + ny * bz);
    r.lo = a.bin_offsets[base + first];
    r.length = a.bin_offsets[base + last + 1] - r.lo;
    return r;
}

// A tile of a bin's candidates in LDS, in visit order, without those too far from the bin's atoms
// to pair with any of them.
constexpr int kSearchWaves = 4;
constexpr int kSearchPerLane = 4;

// Slots of a bin that one block takes as centers, at most: 64 up to 524,288 atoms, and 128 above,
// as most of the blocks by slot (search_pairs_kernel) have nothing to do in most frames (2,097,152
// atoms: an idle update 70 us without them, 82 with 64 slots, 76 with 128). At 100 atoms a bin
// (100,000 atoms, full list) a rebuild takes 668 us with 64, 688 with 128; at 125 (8,000 atoms)
// 325 and 535.
constexpr int kSearchShare = 128;
constexpr std::int64_t kSmallShares = 524288;
inline index_t search_share(std::int64_t atoms)
{
    return atoms <= kSmallShares ? kSearchShare / 2 : kSearchShare;
}

template <typename T>
struct SearchTile
{
    static constexpr int kRaw = kSearchWaves * kWave * kSearchPerLane;  // candidates read per tile
    T x[kRaw], y[kRaw], z[kRaw];
    index_t slot[kRaw], id[kRaw];
    std::uint8_t shift[kRaw];
    index_t start[kSearchRanges], to_slot[kSearchRanges], range_shift[kSearchRanges];
    index_t kept[kSearchWaves * kSearchPerLane];
    // the centers' running places between one tile and the next
    index_t half[kSearchShare], row[kSearchShare];
    T box[6];
};

// Candidates [base, base + kRaw) of the bin's ranges into the tile; returns how many it holds.
// `reach` bounds the distance from the box of the bin's atoms at which a candidate can still be
// a neighbor (image mode keeps every one).
template <typename T, bool kFill, int kMode>
__device__ __forceinline__ index_t stage_candidates(const SearchArgs<T>& a,
                                                    SearchTile<T>& tile, index_t base,
                                                    index_t total, T lx, T ly, T lz, T reach_squared)
{
    using Tile = SearchTile<T>;
    constexpr int kThreads = kSearchWaves * kWave;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    T px[kSearchPerLane], py[kSearchPerLane], pz[kSearchPerLane];
    index_t slot[kSearchPerLane], id[kSearchPerLane], shift[kSearchPerLane];
    std::uint64_t keep[kSearchPerLane];
    // every read of the tile before any use: a turn waits for memory once
#pragma unroll
    for (int u = 0; u < kSearchPerLane; ++u)
    {
        const index_t t = base + u * kThreads + static_cast<index_t>(threadIdx.x);
        int r = 0;
#pragma unroll
        for (int step = kSearchRanges / 2; step > 0; step >>= 1)
            if (tile.start[r + step] <= t) r += step;
        slot[u] = t < total ? tile.to_slot[r] + t : -1;
        shift[u] = kMode == kSearchShifted ? tile.range_shift[r] : 0;
    }
#pragma unroll
    for (int u = 0; u < kSearchPerLane; ++u)
    {
        const index_t from = slot[u] < 0 ? 0 : slot[u];
        px[u] = a.sp[3LL * from];
        py[u] = a.sp[3LL * from + 1];
        pz[u] = a.sp[3LL * from + 2];
        id[u] = kFill ? a.sorted_ids[from] : 0;
    }
#pragma unroll
    for (int u = 0; u < kSearchPerLane; ++u)
    {
        bool take = slot[u] >= 0;
        if (kMode != kSearchImage)
        {
            T qx = px[u], qy = py[u], qz = pz[u];
            if (kMode == kSearchShifted)
            {
                const int code = shift[u];
                px[u] = px[u] + ((code & 1) != 0 ? -lx : T(0));
                py[u] = py[u] + ((code & 4) != 0 ? -ly : T(0));
                pz[u] = pz[u] + ((code & 16) != 0 ? -lz : T(0));
                qx = px[u] + ((code & 2) != 0 ? lx : T(0));
                qy = py[u] + ((code & 8) != 0 ? ly : T(0));
                qz = pz[u] + ((code & 32) != 0 ? lz : T(0));
            }
            const T gx = fmax(fmax(tile.box[0] - qx, qx - tile.box[3]), T(0));
            const T gy = fmax(fmax(tile.box[1] - qy, qy - tile.box[4]), T(0));
            const T gz = fmax(fmax(tile.box[2] - qz, qz - tile.box[5]), T(0));
            take = take && squared(gx, gy, gz) < reach_squared;
        }
        keep[u] = ballot(take);
        if (lane == 0) tile.kept[u * kSearchWaves + wave] = __popcll(keep[u]);
    }
    __syncthreads();
    index_t count = 0;
    index_t before[kSearchPerLane];
#pragma unroll
    for (int u = 0; u < kSearchPerLane; ++u)
#pragma unroll
        for (int w = 0; w < kSearchWaves; ++w)
        {
            if (w == wave) before[u] = count;
            count += tile.kept[u * kSearchWaves + w];
        }
#pragma unroll
    for (int u = 0; u < kSearchPerLane; ++u)
        if ((keep[u] >> lane) & 1ull)
        {
            const int at = before[u] + bits_below(keep[u]);
            tile.x[at] = px[u];
            tile.y[at] = py[u];
            tile.z[at] = pz[u];
            tile.slot[at] = slot[u];
            if (kFill) tile.id[at] = id[u];
            if (kMode == kSearchShifted) tile.shift[at] = static_cast<std::uint8_t>(shift[u]);
        }
    __syncthreads();
    static_assert(Tile::kRaw == kThreads * kSearchPerLane, "one candidate per lane and turn");
    return __builtin_amdgcn_readfirstlane(count);
}

// The centers of one wave: kSearchCenters consecutive slots, their coordinates and running
// places scalar.
template <typename T>
struct SearchGroup
{
    T x[kSearchCenters], y[kSearchCenters], z[kSearchCenters];
    index_t id[kSearchCenters];
    index_t half[kSearchCenters];  // count: pairs so far; fill: the next column
    index_t row[kSearchCenters];   // count: neighbors so far; fill: the next full entry
};

// The group against the tile's candidates, 64 a turn. A turn's hits of a center are a ballot: its
// bits count them, and rank each hit in the center's columns (half list: candidates after the
// center) and in its full row, so a turn's hits go out as one run from a scalar address.
template <typename T, bool kFull, bool kFill, int kMode>
__device__ __forceinline__ void search_tile(const SearchArgs<T>& a,
                                            const SearchTile<T>& tile, index_t count,
                                            index_t first, int live, T lx, T ly, T lz,
                                            SearchGroup<T>& c)
{
    const int lane = lane_id();
    for (index_t chunk = 0; chunk < count; chunk += kWave)
    {
        const index_t at = chunk + lane < count ? chunk + lane : count - 1;
        const T px = tile.x[at], py = tile.y[at], pz = tile.z[at];
        const index_t slot = tile.slot[at];
        const index_t id = kFill ? tile.id[at] : 0;
        const int shift = kMode == kSearchShifted ? tile.shift[at] : 0;
        const std::uint64_t valid =
            count - chunk >= kWave ? ~0ull : (1ull << (count - chunk)) - 1ull;
        // candidates after every center, and those that are centers of this group themselves
        const std::uint64_t beyond = valid & ballot(slot >= first + live);
        const std::uint64_t own = valid & ballot(slot >= first && slot < first + live);
#pragma unroll
        for (int g = 0; g < kSearchCenters; ++g)
        {
            if (g >= live) break;
            T dx, dy, dz;
            if (kMode == kSearchImage)
            {
                dx = minimum_image(c.x[g], px, lx);
                dy = minimum_image(c.y[g], py, ly);
                dz = minimum_image(c.z[g], pz, lz);
            }
            else if (kMode == kSearchShifted)
            {
                dx = ((shift & 2) != 0 ? c.x[g] - lx : c.x[g]) - px;
                dy = ((shift & 8) != 0 ? c.y[g] - ly : c.y[g]) - py;
                dz = ((shift & 32) != 0 ? c.z[g] - lz : c.z[g]) - pz;
            }
            else
            {
                dx = c.x[g] - px;
                dy = c.y[g] - py;
                dz = c.z[g] - pz;
            }
            std::uint64_t hits = valid & ballot(squared(dx, dy, dz) < a.radius_squared);
            std::uint64_t after = hits & beyond;
            if (own != 0)
            {
                hits &= ~ballot(slot == first + g);
                after = hits & ballot(slot > first + g);
            }
            if (kFill)
            {
                // an overflowing build (which the status reports) writes up to the capacity
                if (after != 0)
                {
                    const std::uint32_t rank = bits_below(after);
                    const std::int64_t room = a.capacity - c.half[g];
                    if (((after >> lane) & 1ull) && static_cast<std::int64_t>(rank) < room &&
                        c.half[g] >= 0)
                    {
                        index_t* column = a.pairs + c.half[g];
                        column[rank] = c.id[g];
                        column[a.capacity + rank] = id;
                    }
                    c.half[g] += __popcll(after);
                }
                if (kFull && hits != 0)
                {
                    const std::uint32_t step = bits_below(hits) * kWave;
                    const std::int64_t room = a.full_capacity - c.row[g];
                    if (((hits >> lane) & 1ull) && static_cast<std::int64_t>(step) < room &&
                        c.row[g] >= 0)
                    {
                        index_t* entry = a.full_index + c.row[g];
                        entry[step] = id;
                    }
                    c.row[g] += __popcll(hits) * kWave;
                }
            }
            else
            {
                c.half[g] += __popcll(after);
                if (kFull) c.row[g] += __popcll(hits);
            }
        }
    }
}

// The centers [begin, end), at most kSearchShare slots of a bin, against its candidates: a tile at a
// time, and for each tile kSearchWaves groups of centers a turn. Most bins' candidates are one
// tile; past it the centers' places wait in LDS for the next, so that every tile is read once.
template <typename T, bool kFull, bool kFill, int kMode>
__device__ __forceinline__ void search_bin(const SearchArgs<T>& a, SearchTile<T>& tile,
                                           index_t begin, index_t end, index_t total)
{
    constexpr int kCenters = kSearchCenters;
    using Tile = SearchTile<T>;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const T lx = a.cell[0], ly = a.cell[1], lz = a.cell[2];
    // a candidate this far from the box of the centers pairs with none of them, whatever the
    // rounding of its image
    const T radius = sqrt(a.radius_squared);
    const T longest = fmax(lx, fmax(ly, lz));
    const T reach = radius * T(1.001) + T(16) * std::numeric_limits<T>::epsilon() * longest;
    const T reach_squared = reach * reach;
    for (index_t base = 0; base == 0 || base < total; base += Tile::kRaw)
    {
        if (base > 0) __syncthreads();
        const index_t count =
            stage_candidates<T, kFill, kMode>(a, tile, base, total, lx, ly, lz, reach_squared);
        const bool last = total - base <= Tile::kRaw;
        for (index_t round = begin; round < end; round += kSearchWaves * kCenters)
        {
            const index_t first = round + wave * kCenters;
            const int live = first >= end ? 0 : (end - first < kCenters ? end - first : kCenters);
            if (live == 0) continue;
            const index_t mine = first + (lane < live ? lane : 0);
            const T mx = a.sp[3LL * mine], my = a.sp[3LL * mine + 1], mz = a.sp[3LL * mine + 2];
            const index_t id = kFill ? a.sorted_ids[mine] : 0;
            index_t half, row;
            if (base > 0)
            {
                half = tile.half[mine - begin];
                row = tile.row[mine - begin];
            }
            else
            {
                half = kFill ? a.pair_offsets[mine] : 0;
                row = kFill && kFull ? a.full_slices[mine / kWave] + mine % kWave : 0;
            }
            SearchGroup<T> c;
#pragma unroll
            for (int g = 0; g < kCenters; ++g)
            {
                c.x[g] = read_lane(mx, g);
                c.y[g] = read_lane(my, g);
                c.z[g] = read_lane(mz, g);
                c.id[g] = read_lane(id, g);
                c.half[g] = read_lane(half, g);
                c.row[g] = read_lane(row, g);
            }
            search_tile<T, kFull, kFill, kMode>(a, tile, count, first, live, lx, ly, lz, c);
            if (kFill && last) continue;
#pragma unroll
            for (int g = 0; g < kCenters; ++g)
            {
                half = lane == g ? c.half[g] : half;
                row = lane == g ? c.row[g] : row;
            }
            if (lane < live)
            {
                if (last)
                {
                    a.pair_counts[mine] = half;
                    if (kFull)
                    {
                        a.full_counts[mine] = row;
                        atomicMax(a.full_slices + mine / kWave, row * kWave);
                    }
                }
                else
                {
                    // read by the same lane
                    tile.half[mine - begin] = half;
                    tile.row[mine - begin] = row;
                }
            }
        }
    }
}

// A block per bin, or per share of a crowded one. The candidates of a bin are the same for all its
// atoms: the block reads them into LDS, leaving out those out of reach of the box of its centers
// (a quarter of the 27 bins' atoms at 28 atoms a bin), and each wave tests its centers against
// them. Bound by the issue of vector and scalar instructions (about 11 of each per center and 64
// candidates). A lane per center, each writing columns of its own, wrote the lists 4 bytes to a
// line. A rebuild at 2,097,152 atoms, radius 1.1 nm, full list: 6.9 -> 2.1 ms (the fill 5.8 ->
// 1.36, the count 1.05 -> 0.72); a fill of 4,096 atoms, whose 64 waves left the chip idle, 140 ->
// 13 us.
//
// A bin of more atoms than a share leaves the rest to blocks by slot, past those of the bins:
// block `bins` + x takes those of the slots [share x, share x + share) that lie as far into their
// bin. 100,000 atoms, half of them in a clump of 1 nm: 27 ms a rebuild with a lane per center, 125
// with a block per bin whatever it holds, 13 so; at 291 atoms a bin 5.2, 3.5 and 2.2.
template <typename T, bool kFull, bool kFill>
__global__ void __launch_bounds__(kSearchWaves * kWave) search_pairs_kernel(SearchArgs<T> a)
{
    __shared__ SearchTile<T> tile;
    if (!rebuilding(a.rebuild, a.status)) return;
    const index_t nx = a.dims[0], ny = a.dims[1], nz = a.dims[2];
    const std::int64_t bins = a.bin_slots - 1;
    std::int64_t bin = blockIdx.x;
    index_t slot = 0;
    if (bin >= bins)
    {
        // a block by slot
        const std::int64_t at = (bin - bins) * a.share;
        if (at >= a.num_atoms) return;
        slot = static_cast<index_t>(at);
        bin = __builtin_amdgcn_readfirstlane(a.atom_bin[a.sorted_ids[slot]]);
    }
    if (bin >= static_cast<std::int64_t>(nx) * ny * nz || bin >= bins) return;
    index_t begin = __builtin_amdgcn_readfirstlane(a.bin_offsets[bin]);
    index_t end = __builtin_amdgcn_readfirstlane(a.bin_offsets[bin + 1]);
    // the bin's own block ends here (differences: a sum past the last slot could leave 32 bits)
    const index_t own = end - begin < a.share ? end : begin + a.share;
    if (blockIdx.x < bins)
        end = own;
    else
    {
        begin = slot > own ? slot : own;
        end = end - slot < a.share ? end : slot + a.share;
    }
    if (begin >= end) return;
    const index_t home = static_cast<index_t>(bin);
    const index_t hx = home % nx, hy = (home / nx) % ny, hz = home / (nx * ny);
    const int lane = lane_id();
    // every wave finds the ranges for itself; the first writes them for the staging
    SearchRange range = search_range(a, hx, hy, hz, nx, ny, nz, lane);
    if (!kFull && range.lo <= begin)
    {
        // a half list alone needs no candidate up to the block's first atom
        const index_t cut =
            range.lo + range.length <= begin + 1 ? range.length : begin + 1 - range.lo;
        range.lo += cut;
        range.length -= cut;
    }
    const index_t inclusive = wave_inclusive_sum(range.length);
    const index_t total = read_lane(inclusive, kWave - 1);
    if (threadIdx.x < kSearchRanges)
    {
        tile.start[lane] = inclusive - range.length;
        tile.to_slot[lane] = range.lo - (inclusive - range.length);
        tile.range_shift[lane] = range.shift;
    }
    // the box of the block's atoms, found by the first wave
    if (threadIdx.x < kWave)
    {
        T low[3], high[3];
        for (int axis = 0; axis < 3; ++axis)
        {
            low[axis] = std::numeric_limits<T>::max();
            high[axis] = -std::numeric_limits<T>::max();
        }
        for (index_t k = begin + lane; k < end; k += kWave)
            for (int axis = 0; axis < 3; ++axis)
            {
                const T v = a.sp[3LL * k + axis];
                low[axis] = fmin(low[axis], v);
                high[axis] = fmax(high[axis], v);
            }
        for (int axis = 0; axis < 3; ++axis)
        {
            const T l = -wave_max(-low[axis]), h = wave_max(high[axis]);
            if (lane == 0)
            {
                tile.box[axis] = l;
                tile.box[3 + axis] = h;
            }
        }
    }
    __syncthreads();
    const bool image = nx < 3 || ny < 3 || nz < 3;
    const bool inside = hx > 0 && hx < nx - 1 && hy > 0 && hy < ny - 1 && hz > 0 && hz < nz - 1;
    if (image)
        search_bin<T, kFull, kFill, kSearchImage>(a, tile, begin, end, total);
    else if (inside)
        search_bin<T, kFull, kFill, kSearchPlain>(a, tile, begin, end, total);
    else
        search_bin<T, kFull, kFill, kSearchShifted>(a, tile, begin, end, total);
}

// ---- all-pairs path -------------------------------------------------------------------------

// One wave per atom i: 64 candidates per ballot, each 64-bit hit mask stored as two words of
// i's bit row. A half list tests j > i only; a full list tests every j != i.
template <typename T, bool kFull>
__global__ void __launch_bounds__(kBlock) test_all_pairs_kernel(
    const T* __restrict__ positions, const T* __restrict__ cell, T radius_squared,
    index_t num_atoms, std::uint32_t* __restrict__ bits, std::int64_t row_words,
    index_t* __restrict__ pair_counts, index_t* __restrict__ full_counts,
    index_t* __restrict__ full_slices, const index_t* rebuild, const index_t* status)
{
    if (!rebuilding(rebuild, status)) return;
    const std::int64_t center =
        static_cast<std::int64_t>(blockIdx.x) * (kBlock / kWave) + threadIdx.x / kWave;
    if (center >= num_atoms) return;
    const int lane = lane_id();
    const T lx = cell[0], ly = cell[1], lz = cell[2];
    const T cx = positions[3 * center], cy = positions[3 * center + 1],
            cz = positions[3 * center + 2];
    const std::int64_t chunks = (num_atoms + kWave - 1) / kWave;
    index_t half = 0, full = 0;
    for (std::int64_t chunk = kFull ? 0 : (center + 1) / kWave; chunk < chunks; ++chunk)
    {
        const std::int64_t j = chunk * kWave + lane;
        bool hit = false;
        if (j < num_atoms && j != center && (kFull || j > center))
        {
            const T dx = minimum_image(cx, positions[3 * j], lx);
            const T dy = minimum_image(cy, positions[3 * j + 1], ly);
            const T dz = minimum_image(cz, positions[3 * j + 2], lz);
            hit = squared(dx, dy, dz) < radius_squared;
        }
        const std::uint64_t mask = ballot(hit);
        const std::uint64_t after = ballot(hit && j > center);
        half += __popcll(after);
        full += __popcll(mask);
        if (lane == 0)
        {
            bits[center * row_words + 2 * chunk] = static_cast<std::uint32_t>(mask);
            if (2 * chunk + 1 < row_words)
                bits[center * row_words + 2 * chunk + 1] = static_cast<std::uint32_t>(mask >> 32);
        }
    }
    if (lane == 0)
    {
        pair_counts[center] = half;
        if (kFull) full_counts[center] = full;
    }
}

// Slice widths of the full list on the all-pairs path, from the full counts.
__global__ void __launch_bounds__(kBlock) slice_widths_kernel(
    const index_t* __restrict__ full_counts, index_t num_atoms, index_t* __restrict__ full_slices,
    const index_t* rebuild, const index_t* status)
{
    if (!rebuilding(rebuild, status)) return;
    const std::int64_t row = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const index_t width = wave_max(row < num_atoms ? full_counts[row] : 0);
    if (lane_id() == 0 && row < num_atoms) full_slices[row / kWave] = width * kWave;
}

template <bool kFull>
__global__ void __launch_bounds__(kBlock) fill_all_pairs_kernel(
    const std::uint32_t* __restrict__ bits, std::int64_t row_words,
    const index_t* __restrict__ pair_offsets, index_t num_atoms, std::int64_t capacity,
    index_t* __restrict__ pairs, const index_t* __restrict__ full_slices,
    index_t* __restrict__ full_index, std::int64_t full_capacity, const index_t* rebuild,
    const index_t* status)
{
    if (!rebuilding(rebuild, status)) return;
    const std::int64_t center =
        static_cast<std::int64_t>(blockIdx.x) * (kBlock / kWave) + threadIdx.x / kWave;
    if (center >= num_atoms) return;
    const int lane = lane_id();
    const std::int64_t chunks = (num_atoms + kWave - 1) / kWave;
    std::int64_t column = pair_offsets[center];
    std::int64_t full_column = 0;
    const std::int64_t slice_base = kFull ? full_slices[center / kWave] + center % kWave : 0;
    for (std::int64_t chunk = kFull ? 0 : (center + 1) / kWave; chunk < chunks; ++chunk)
    {
        const std::uint32_t low = bits[center * row_words + 2 * chunk];
        const std::uint32_t high =
            2 * chunk + 1 < row_words ? bits[center * row_words + 2 * chunk + 1] : 0u;
        const std::uint64_t mask = (static_cast<std::uint64_t>(high) << 32) | low;
        const std::int64_t j = chunk * kWave + lane;
        const bool hit = (mask >> lane) & 1ull;
        const std::uint64_t after = ballot(hit && j > center);
        if (hit && j > center)
        {
            const std::int64_t slot = column + bits_below(after);
            if (slot < capacity)
            {
                pairs[slot] = static_cast<index_t>(center);
                pairs[capacity + slot] = static_cast<index_t>(j);
            }
        }
        column += __popcll(after);
        if (kFull)
        {
            if (hit)
            {
                const std::int64_t slot = slice_base + (full_column + bits_below(mask)) * kWave;
                if (slot < full_capacity) full_index[slot] = static_cast<index_t>(j);
            }
            full_column += __popcll(mask);
        }
    }
}

// ---- total, pad, commit ---------------------------------------------------------------------

// The pair total and, above the capacity, the overflow bit with the pairs needed; then the
// padding. Column k past the pairs holds (k mod N, k mod N) whatever the build, so after the
// first frame only the columns between this total and the previous one need writing. A rebuild
// that fits is committed in the same launch (reference_positions null for a first frame, whose
// caller keeps the frame itself): its frame and cell become the reuse rule's reference. Every
// block decides from the totals, which no block writes, so a status bit set meanwhile changes
// nothing.
template <typename T>
__global__ void __launch_bounds__(kBlock) total_pad_commit_kernel(
    const index_t* __restrict__ pair_counts, const index_t* __restrict__ pair_offsets,
    index_t num_atoms, std::int64_t capacity, index_t* __restrict__ pair_total, index_t* status,
    index_t* __restrict__ pairs, const ListHeader* __restrict__ header, int first_frame,
    const index_t* __restrict__ full_slices, std::int64_t num_slices, std::int64_t full_capacity,
    const T* __restrict__ positions, const T* __restrict__ cell,
    T* __restrict__ reference_positions, T* __restrict__ reference_cell,
    index_t* __restrict__ rebuild_count, const index_t* rebuild)
{
    if (!rebuilding(rebuild, status)) return;
    const index_t total = pair_offsets[num_atoms - 1] + pair_counts[num_atoms - 1];
    const std::int64_t gid = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const bool full_over = full_slices != nullptr && full_slices[num_slices] > full_capacity;
    if (gid == 0)
    {
        pair_total[0] = total;
        index_t flags = 0;
        if (total > capacity)
        {
            flags |= kStatusOverflow;
            status[1] = total > status[1] ? total : status[1];
        }
        if (full_over) flags |= kStatusFullOverflow;
        if (flags) status[0] |= flags;
    }
    if (total > capacity || full_over) return;
    const std::int64_t end =
        first_frame ? capacity : (header->old_total < capacity ? header->old_total : capacity);
    const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    for (std::int64_t column = total + gid; column < end; column += stride)
    {
        const index_t atom = static_cast<index_t>(column % num_atoms);
        pairs[column] = atom;
        pairs[capacity + column] = atom;
    }
    if (reference_positions == nullptr) return;
    for (std::int64_t k = gid; k < 3LL * num_atoms; k += stride)
        reference_positions[k] = positions[k];
    if (gid < 3) reference_cell[gid] = cell[gid];
    if (gid == 0) ++rebuild_count[0];
}

// What a first frame's host code reads: the cell's edges in found [0..2] and how many coordinates
// are not finite in found [3] (found zero before the launch).
template <typename T>
__global__ void __launch_bounds__(kBlock) inspect_frame_kernel(const T* __restrict__ positions,
                                                               const T* __restrict__ cell,
                                                               std::int64_t count,
                                                               double* __restrict__ found)
{
    const std::int64_t first = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    int bad = 0;
    for (std::int64_t k = first; k < count; k += stride) bad += !isfinite(positions[k]);
    if (bad != 0) unsafeAtomicAdd(found + 3, static_cast<double>(bad));
    if (first < 3) found[first] = static_cast<double>(cell[first]);
}

// The pairs of a count in totals [0], as 64-bit sums, and the entries of its full list in
// totals [1] (totals zero before the launch).
__global__ void __launch_bounds__(kBlock) count_totals_kernel(
    const index_t* __restrict__ pair_counts, std::int64_t num_atoms,
    const index_t* __restrict__ full_slices, std::int64_t num_slices,
    unsigned long long* __restrict__ totals)
{
    __shared__ unsigned long long shared[16];
    const std::int64_t first = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
    unsigned long long sum = 0;
    for (std::int64_t k = first; k < num_atoms; k += stride)
        sum += static_cast<unsigned long long>(pair_counts[k]);
    sum = block_sum(sum, shared);
    if (threadIdx.x == 0 && sum != 0) atomicAdd(totals, sum);
    if (first == 0 && full_slices != nullptr)
        totals[1] = static_cast<unsigned long long>(full_slices[num_slices]);
}

// Coordinates [frames, N, 3] into the frames' cells [frames, 3], `per_frame` = 3N coordinates to a
// frame.
template <typename T>
__global__ void __launch_bounds__(kBlock) wrap_kernel(const T* positions, const T* __restrict__ cell,
                                                      std::int64_t count, std::int64_t per_frame,
                                                      T* out, std::int64_t* __restrict__ images)
{
    const std::int64_t index = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (index >= count) return;
    const std::int64_t frame = count == per_frame ? 0 : index / per_frame;
    const T length = cell[3 * frame + index % 3];
    const T v = positions[index];
    T k = floor(v / length);
    T w = v - k * length;
    if (w < T(0))
    {
        w = w + length;
        k = k - T(1);
    }
    if (w >= length)
    {
        w = w - length;
        k = k + T(1);
    }
    out[index] = w;
    if (images != nullptr) images[index] += static_cast<std::int64_t>(k);
}

// ---- launch sequences -----------------------------------------------------------------------

constexpr unsigned kPadBlocks = 1024;

template <typename T>
int launch_grid(const T* positions, const ndn_neighbor_buffers& b, const index_t* rebuild,
                hipStream_t stream)
{
    const index_t n = static_cast<index_t>(b.num_atoms);
    assign_bins_kernel<T><<<blocks_for(n), kBlock, 0, stream>>>(
        positions, b.dims, static_cast<const T*>(b.widths), n, b.atom_bin, b.bin_counts,
        b.full_index != nullptr ? b.full_slices : nullptr, rebuild, b.status);
    NDN_LAUNCHED("assign_bins");
    const int scanned = exclusive_scan(b.bin_counts, b.bin_offsets, b.bin_slots, b.scan_temp,
                                       rebuild, b.status, stream);
    if (scanned != NDN_OK) return scanned;
    scatter_atoms_kernel<<<blocks_for(n), kBlock, 0, stream>>>(
        b.atom_bin, b.bin_offsets, n, b.bin_counts, b.unordered_ids, rebuild, b.status);
    NDN_LAUNCHED("scatter_atoms");
    const std::int64_t bins = b.bin_slots - 1;
    order_bins_kernel<T><<<blocks_for(bins, kBlock / kWave), kBlock, 0, stream>>>(
        positions, b.unordered_ids, b.bin_offsets, b.dims, b.bin_slots, b.sorted_ids,
        static_cast<T*>(b.sorted_positions), rebuild, b.status);
    NDN_LAUNCHED("order_bins");
    return NDN_OK;
}

// Whether a block per bin searches the grid, or a lane per center. A block stages 27 bins for the
// centers of one, which pays from about seven atoms a bin (a rebuild of 100,000 atoms, radius
// 1.0 nm, full list: 283 us against a lane per center's 179 at 4.1 atoms a bin, 229 against 204
// at 6.4, 213 against 285 at 9.4, 204 against 398 at 14.6); up to 8,192 atoms, whose lanes fill
// a small part of the chip, from two (3,000 atoms: 85 us against 110 at 2.3).
bool block_per_bin(std::int64_t atoms, std::int64_t bins)
{
    return atoms >= bins * (atoms <= 8192 ? 2 : 7);
}

// The search over the grid: the count (kFill false) or the fill.
template <typename T, bool kFill>
void launch_search(const T* cell, T radius_squared, const ndn_neighbor_buffers& b,
                   const index_t* rebuild, hipStream_t stream)
{
    const std::int64_t bins = b.bin_slots - 1;
    const index_t n = static_cast<index_t>(b.num_atoms);
    const T* sp = static_cast<const T*>(b.sorted_positions);
    const bool full = b.full_index != nullptr;
    if (!block_per_bin(b.num_atoms, bins))
    {
        const unsigned blocks = blocks_for(n);
        if (kFill && full)
            fill_pairs_kernel<T, true><<<blocks, kBlock, 0, stream>>>(
                sp, b.sorted_ids, b.atom_bin, b.bin_offsets, b.dims, cell, b.pair_offsets,
                radius_squared, n, b.capacity, b.pairs, b.full_slices, b.full_index,
                b.full_capacity, rebuild, b.status);
        else if (kFill)
            fill_pairs_kernel<T, false><<<blocks, kBlock, 0, stream>>>(
                sp, b.sorted_ids, b.atom_bin, b.bin_offsets, b.dims, cell, b.pair_offsets,
                radius_squared, n, b.capacity, b.pairs, nullptr, nullptr, 0, rebuild, b.status);
        else if (full)
            count_pairs_kernel<T, true><<<blocks, kBlock, 0, stream>>>(
                sp, b.sorted_ids, b.atom_bin, b.bin_offsets, b.dims, cell, radius_squared, n,
                b.pair_counts, b.full_counts, b.full_slices, rebuild, b.status);
        else
            count_pairs_kernel<T, false><<<blocks, kBlock, 0, stream>>>(
                sp, b.sorted_ids, b.atom_bin, b.bin_offsets, b.dims, cell, radius_squared, n,
                b.pair_counts, nullptr, nullptr, rebuild, b.status);
        return;
    }
    SearchArgs<T> a{};
    a.sp = sp;
    a.sorted_ids = b.sorted_ids;
    a.bin_offsets = b.bin_offsets;
    a.dims = b.dims;
    a.cell = cell;
    a.radius_squared = radius_squared;
    a.atom_bin = b.atom_bin;
    a.num_atoms = n;
    a.share = search_share(n);
    a.bin_slots = b.bin_slots;
    a.pair_counts = b.pair_counts;
    a.full_counts = b.full_counts;
    a.full_slices = b.full_slices;
    a.pair_offsets = b.pair_offsets;
    a.pairs = b.pairs;
    a.capacity = b.capacity;
    a.full_index = b.full_index;
    a.full_capacity = b.full_capacity;
    a.rebuild = rebuild;
    a.status = b.status;
    const unsigned blocks = static_cast<unsigned>(bins + (b.num_atoms + a.share - 1) / a.share);
    if (full)
        search_pairs_kernel<T, true, kFill><<<blocks, kSearchWaves * kWave, 0, stream>>>(a);
    else
        search_pairs_kernel<T, false, kFill><<<blocks, kSearchWaves * kWave, 0, stream>>>(a);
}

template <typename T>
int launch_count(const T* positions, const T* cell, double radius, const ndn_neighbor_buffers& b,
                 const index_t* rebuild, hipStream_t stream)
{
    const index_t n = static_cast<index_t>(b.num_atoms);
    const T r = static_cast<T>(radius);
    const T r2 = r * r;
    const bool full = b.full_index != nullptr;
    const std::int64_t slices = (b.num_atoms + kWave - 1) / kWave;
    if (b.bits_words > 0)
    {
        const std::int64_t row_words = (b.num_atoms + 31) / 32;
        auto* bits = reinterpret_cast<std::uint32_t*>(b.bits);
        const unsigned blocks = blocks_for(n, kBlock / kWave);
        if (full)
        {
            test_all_pairs_kernel<T, true><<<blocks, kBlock, 0, stream>>>(
                positions, cell, r2, n, bits, row_words, b.pair_counts, b.full_counts,
                b.full_slices, rebuild, b.status);
            NDN_LAUNCHED("test_all_pairs");
            slice_widths_kernel<<<blocks_for(n), kBlock, 0, stream>>>(b.full_counts, n,
                                                                      b.full_slices, rebuild,
                                                                      b.status);
            NDN_LAUNCHED("slice_widths");
        }
        else
        {
            test_all_pairs_kernel<T, false><<<blocks, kBlock, 0, stream>>>(
                positions, cell, r2, n, bits, row_words, b.pair_counts, nullptr, nullptr, rebuild,
                b.status);
            NDN_LAUNCHED("test_all_pairs");
        }
    }
    else
    {
        launch_search<T, false>(cell, r2, b, rebuild, stream);
        NDN_LAUNCHED("count_pairs");
    }
    // the columns' offsets, and with a full list the slices' (slices + 1 entries: the last, an
    // output only, becomes the total), in the same launches; the slices' tile sums go where the
    // build's unordered ids were
    const ScanArray columns{b.pair_counts, b.pair_offsets, b.num_atoms,
                            reinterpret_cast<index_t*>(b.scan_temp + kHeaderBytes)};
    ScanArray widths{};
    if (full) widths = ScanArray{b.full_slices, b.full_slices, slices + 1, b.unordered_ids};
    return exclusive_scans(columns, widths, rebuild, b.status, stream);
}

// A first frame's (reference_positions null) or an update's fill, padding and commit.
template <typename T>
int launch_fill(const T* positions, const T* cell, double radius, const ndn_neighbor_buffers& b,
                T* reference_positions, T* reference_cell, index_t* rebuild_count,
                const index_t* rebuild, hipStream_t stream)
{
    const index_t n = static_cast<index_t>(b.num_atoms);
    const T r = static_cast<T>(radius);
    const T r2 = r * r;
    const bool full = b.full_index != nullptr;
    const std::int64_t slices = (b.num_atoms + kWave - 1) / kWave;
    if (b.bits_words > 0)
    {
        const std::int64_t row_words = (b.num_atoms + 31) / 32;
        const auto* bits = reinterpret_cast<const std::uint32_t*>(b.bits);
        const unsigned blocks = blocks_for(n, kBlock / kWave);
        if (full)
            fill_all_pairs_kernel<true><<<blocks, kBlock, 0, stream>>>(
                bits, row_words, b.pair_offsets, n, b.capacity, b.pairs, b.full_slices,
                b.full_index, b.full_capacity, rebuild, b.status);
        else
            fill_all_pairs_kernel<false><<<blocks, kBlock, 0, stream>>>(
                bits, row_words, b.pair_offsets, n, b.capacity, b.pairs, nullptr, nullptr, 0,
                rebuild, b.status);
        NDN_LAUNCHED("fill_all_pairs");
    }
    else
    {
        launch_search<T, true>(cell, r2, b, rebuild, stream);
        NDN_LAUNCHED("fill_pairs");
    }
    total_pad_commit_kernel<T><<<kPadBlocks, kBlock, 0, stream>>>(
        b.pair_counts, b.pair_offsets, n, b.capacity, b.pair_total, b.status, b.pairs,
        reinterpret_cast<const ListHeader*>(b.scan_temp), reference_positions == nullptr ? 1 : 0,
        full ? b.full_slices : nullptr, slices, b.full_capacity, positions, cell,
        reference_positions, reference_cell, rebuild_count, rebuild);
    NDN_LAUNCHED("total_pad_commit");
    return NDN_OK;
}

template <typename T>
int launch_rebuild(const T* positions, const T* cell, double radius, const ndn_neighbor_buffers& b,
                   T* reference_positions, T* reference_cell, index_t* rebuild_count,
                   const index_t* rebuild, hipStream_t stream)
{
    if (b.bits_words == 0)
    {
        const int grid = launch_grid<T>(positions, b, rebuild, stream);
        if (grid != NDN_OK) return grid;
    }
    const int counted = launch_count<T>(positions, cell, radius, b, rebuild, stream);
    if (counted != NDN_OK) return counted;
    return launch_fill<T>(positions, cell, radius, b, reference_positions, reference_cell,
                          rebuild_count, rebuild, stream);
}

template int launch_rebuild<float>(const float*, const float*, double, const ndn_neighbor_buffers&,
                                   float*, float*, index_t*, const index_t*, hipStream_t);
template int launch_rebuild<double>(const double*, const double*, double,
                                    const ndn_neighbor_buffers&, double*, double*, index_t*,
                                    const index_t*, hipStream_t);

int check_buffers(const ndn_neighbor_buffers* b)
{
    NDN_REQUIRE(b != nullptr, "buffers must not be null");
    NDN_REQUIRE(b->num_atoms >= 1 && b->num_atoms <= INT32_MAX, "N must satisfy 1 <= N < 2**31");
    NDN_REQUIRE(b->dims && b->widths && b->atom_bin && b->bin_counts && b->bin_offsets &&
                    b->unordered_ids && b->sorted_ids && b->sorted_positions && b->scan_temp &&
                    b->pair_counts && b->pair_offsets && b->pair_total && b->status && b->pairs,
                "a list buffer is null");
    NDN_REQUIRE(b->bin_slots >= 2, "bin_counts must hold at least 2 entries");
    NDN_REQUIRE(b->capacity >= 1 && b->capacity <= INT32_MAX, "pairs must be [2, C] with int32 C");
    const std::int64_t words = b->num_atoms * ((b->num_atoms + 31) / 32);
    NDN_REQUIRE(b->bits_words == 0 || (b->bits_words == words && b->bits != nullptr),
                "bits must be empty or hold N rows of ceil(N / 32) words");
    const std::int64_t slices = (b->num_atoms + kWave - 1) / kWave;
    const std::int64_t items = std::max(std::max(b->bin_slots, b->num_atoms), slices + 1);
    NDN_REQUIRE(b->scan_temp_bytes >= scan_bytes(items), "scan_temp is too small");
    if (b->full_index != nullptr || b->full_counts != nullptr || b->full_slices != nullptr)
    {
        NDN_REQUIRE(b->full_index && b->full_counts && b->full_slices && b->full_capacity >= 1 &&
                        b->full_capacity <= INT32_MAX,
                    "a full list needs counts, slices and an int32-sized index");
    }
    return NDN_OK;
}

template <typename T>
int count_first_frame_impl(const void* positions, const void* cell, double radius,
                           const ndn_neighbor_buffers& b, hipStream_t stream)
{
    const T* x = static_cast<const T*>(positions);
    if (b.bits_words == 0)
    {
        const int grid = launch_grid<T>(x, b, nullptr, stream);
        if (grid != NDN_OK) return grid;
    }
    return launch_count<T>(x, static_cast<const T*>(cell), radius, b, nullptr, stream);
}

template <typename T>
int fill_first_frame_impl(const void* cell, double radius, const ndn_neighbor_buffers& b,
                          hipStream_t stream)
{
    return launch_fill<T>(nullptr, static_cast<const T*>(cell), radius, b, nullptr, nullptr,
                          nullptr, nullptr, stream);
}

template <typename T>
int update_impl(const void* positions, const void* cell, double cutoff, double radius,
                void* reference_positions, void* reference_cell, const index_t* limits,
                void* reuse, index_t* rebuild, index_t* rebuild_count,
                const ndn_neighbor_buffers& b, hipStream_t stream)
{
    const T* x = static_cast<const T*>(positions);
    const T* L = static_cast<const T*>(cell);
    const index_t n = static_cast<index_t>(b.num_atoms);
    auto* header = reinterpret_cast<ListHeader*>(b.scan_temp);
    prepare_update_kernel<T><<<1, 1, 0, stream>>>(
        L, static_cast<const T*>(reference_cell), static_cast<T>(cutoff), static_cast<T>(radius),
        limits, b.dims, static_cast<T*>(b.widths), static_cast<T*>(reuse), rebuild, b.status,
        b.pair_total, header);
    NDN_LAUNCHED("prepare_update");
    check_reuse_kernel<T><<<blocks_for(n), kBlock, 0, stream>>>(
        x, static_cast<const T*>(reference_positions), L, static_cast<const T*>(reuse), n, rebuild,
        b.status, header);
    NDN_LAUNCHED("check_reuse");
    return launch_rebuild<T>(x, L, radius, b, static_cast<T*>(reference_positions),
                             static_cast<T*>(reference_cell), rebuild_count, rebuild, stream);
}

}  // namespace ndn

using namespace ndn;

extern "C" {

const char* ndn_last_error(void)
{
    return ndn::last_error();
}

int ndn_scan_temp_bytes(int64_t items, int64_t* bytes)
{
    NDN_REQUIRE(items > 0 && items <= INT32_MAX, "the scan length must fit int32");
    NDN_REQUIRE(bytes != nullptr, "bytes must not be null");
    // Room for the largest scan a list runs: max(bins + 1, N) and, with a full list, the
    // ceil(N / 64) + 1 slice widths, which never exceed N + 1.
    *bytes = scan_bytes(items + 1);
    return NDN_OK;
}

int ndn_count_first_frame(int dtype, const void* positions, const void* cell, double radius,
                          const ndn_neighbor_buffers* buffers, ndn_stream_t stream)
{
    const int checked = check_buffers(buffers);
    if (checked != NDN_OK) return checked;
    NDN_REQUIRE(positions && cell, "positions and cell must not be null");
    NDN_REQUIRE(radius > 0, "the radius must be positive");
    if (dtype == NDN_F32)
        return count_first_frame_impl<float>(positions, cell, radius, *buffers, stream);
    NDN_REQUIRE(dtype == NDN_F64, "dtype must be NDN_F32 or NDN_F64");
    return count_first_frame_impl<double>(positions, cell, radius, *buffers, stream);
}

int ndn_fill_first_frame(int dtype, const void* positions, const void* cell, double radius,
                         const ndn_neighbor_buffers* buffers, ndn_stream_t stream)
{
    const int checked = check_buffers(buffers);
    if (checked != NDN_OK) return checked;
    NDN_REQUIRE(positions && cell, "positions and cell must not be null");
    NDN_REQUIRE(radius > 0, "the radius must be positive");
    if (dtype == NDN_F32) return fill_first_frame_impl<float>(cell, radius, *buffers, stream);
    NDN_REQUIRE(dtype == NDN_F64, "dtype must be NDN_F32 or NDN_F64");
    return fill_first_frame_impl<double>(cell, radius, *buffers, stream);
}

int ndn_update(int dtype, const void* positions, const void* cell, double cutoff, double radius,
               void* reference_positions, void* reference_cell, const int32_t* limits,
               void* reuse, int32_t* rebuild, int32_t* rebuild_count,
               const ndn_neighbor_buffers* buffers, ndn_stream_t stream)
{
    const int checked = check_buffers(buffers);
    if (checked != NDN_OK) return checked;
    NDN_REQUIRE(positions && cell && reference_positions && reference_cell && limits && reuse &&
                    rebuild && rebuild_count,
                "an update buffer is null");
    NDN_REQUIRE(cutoff > 0 && radius >= cutoff, "need 0 < cutoff <= radius");
    if (dtype == NDN_F32)
        return update_impl<float>(positions, cell, cutoff, radius, reference_positions,
                                  reference_cell, limits, reuse, rebuild, rebuild_count,
                                  *buffers, stream);
    NDN_REQUIRE(dtype == NDN_F64, "dtype must be NDN_F32 or NDN_F64");
    return update_impl<double>(positions, cell, cutoff, radius, reference_positions,
                               reference_cell, limits, reuse, rebuild, rebuild_count, *buffers,
                               stream);
}

int ndn_inspect_frame(int dtype, const void* positions, const void* cell, int64_t num_atoms,
                      double* found, ndn_stream_t stream)
{
    NDN_REQUIRE(positions && cell && found, "a buffer is null");
    NDN_REQUIRE(num_atoms >= 1 && num_atoms <= INT32_MAX, "N must satisfy 1 <= N < 2**31");
    const std::int64_t count = 3 * num_atoms;
    const unsigned blocks = std::min(blocks_for(count), kPadBlocks);
    if (dtype == NDN_F32)
        inspect_frame_kernel<float><<<blocks, kBlock, 0, stream>>>(
            static_cast<const float*>(positions), static_cast<const float*>(cell), count, found);
    else
    {
        NDN_REQUIRE(dtype == NDN_F64, "dtype must be NDN_F32 or NDN_F64");
        inspect_frame_kernel<double><<<blocks, kBlock, 0, stream>>>(
            static_cast<const double*>(positions), static_cast<const double*>(cell), count, found);
    }
    NDN_LAUNCHED("inspect_frame");
    return NDN_OK;
}

int ndn_count_totals(const ndn_neighbor_buffers* buffers, int64_t* totals, ndn_stream_t stream)
{
    const int checked = check_buffers(buffers);
    if (checked != NDN_OK) return checked;
    NDN_REQUIRE(totals != nullptr, "totals must not be null");
    const std::int64_t n = buffers->num_atoms;
    const bool full = buffers->full_index != nullptr;
    count_totals_kernel<<<std::min(blocks_for(n), kPadBlocks), kBlock, 0, stream>>>(
        buffers->pair_counts, n, full ? buffers->full_slices : nullptr, (n + kWave - 1) / kWave,
        reinterpret_cast<unsigned long long*>(totals));
    NDN_LAUNCHED("count_totals");
    return NDN_OK;
}

int ndn_wrap_frames(int dtype, const void* positions, const void* cells, int64_t frames,
                    int64_t num_atoms, void* out, int64_t* images, ndn_stream_t stream)
{
    NDN_REQUIRE(positions && cells && out, "positions, cell and out must not be null");
    NDN_REQUIRE(frames >= 0 && num_atoms >= 0, "N must be nonnegative");
    const std::int64_t each = 3 * num_atoms;
    const std::int64_t count = frames * each;
    if (count == 0) return NDN_OK;
    if (dtype == NDN_F32)
        wrap_kernel<float><<<blocks_for(count), kBlock, 0, stream>>>(
            static_cast<const float*>(positions), static_cast<const float*>(cells), count, each,
            static_cast<float*>(out), images);
    else
    {
        NDN_REQUIRE(dtype == NDN_F64, "dtype must be NDN_F32 or NDN_F64");
        wrap_kernel<double><<<blocks_for(count), kBlock, 0, stream>>>(
            static_cast<const double*>(positions), static_cast<const double*>(cells), count, each,
            static_cast<double*>(out), images);
    }
    NDN_LAUNCHED("wrap");
    return NDN_OK;
}

int ndn_wrap(int dtype, const void* positions, const void* cell, int64_t num_atoms, void* out,
             int64_t* images, ndn_stream_t stream)
{
    return ndn_wrap_frames(dtype, positions, cell, 1, num_atoms, out, images, stream);
}

}  // extern "C"
