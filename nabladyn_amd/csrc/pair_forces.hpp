// Device helpers shared by the pair-force kernels: exact geometry, the potential view, and the
// per-block partial sums of energy and virial.
#pragma once

#include "common.hpp"
#include "potentials.hpp"

namespace ndn {

// Partial slots every workspace reserves at least: enough for any fixed-grid launch here.
constexpr int kPartialSlots = 4096;

// center - other by minimum image with the near-face coordinate shifted first
// (space.py:11-19): (left - L) - right when raw > L/2, left - (right - L) when raw < -L/2.
template <typename T>
__device__ __forceinline__ T displacement(T left, T right, T length)
{
#pragma clang fp contract(off)
    const T raw = left - right;
    const T half = T(0.5) * length;
    const T left_shift = raw > half ? length : T(0);
    const T right_shift = raw < -half ? length : T(0);
    return (left - left_shift) - (right - right_shift);
}

// (dx dx + dy dy) + dz dz, each product and sum rounded on its own.
template <typename T>
__device__ __forceinline__ T exact_squared(T dx, T dy, T dz)
{
#pragma clang fp contract(off)
    const T xx = dx * dx;
    const T yy = dy * dy;
    const T zz = dz * dz;
    return (xx + yy) + zz;
}

// Which of the stored frames a launch over frames reads: frame f of the launch is stored frame
// at[f], or f itself without a choice. An entry outside the stored frames gives -1, and its block
// does nothing.
struct FrameChoice
{
    const std::int64_t* at = nullptr;
    std::int64_t stored = 0;

    __device__ __forceinline__ std::int64_t frame(unsigned f) const
    {
        if (at == nullptr) return f;
        const std::int64_t chosen = at[f];
        return chosen >= 0 && chosen < stored ? chosen : -1;
    }
};

template <typename T>
struct PotentialView
{
    int kind;
    T cutoff_squared;
    LJ<T> lj;
    Table<T> table;
};

// The sum of `value` over each run of lanes with the same key (a run starts where the key
// changes), left in the run's last lane; `start` is the run's first lane. Equal keys apart are
// separate runs.
template <typename T>
__device__ __forceinline__ T run_sum(T value, int lane, int start)
{
#pragma unroll
    for (int offset = 1; offset < kWave; offset <<= 1)
    {
        const T other = __shfl_up(value, offset, kWave);
        if (lane - offset >= start) value += other;
    }
    return value;
}

// Adds a wave's pair forces to both atoms, f to `i` and -f to `j` (a negative id takes nothing),
// for lanes that walk consecutive columns of a half list; every lane of the wave takes part.
//
// What bounds it is the atomics, which meet in memory past the XCDs' own L2s, each a request of
// its own. So the forces of the first atom are summed over its run of columns before they go out,
// and those of the second go out as its three components in neighboring lanes, which a request
// takes together: 100,000 shuffled LJ atoms 670 us with a component an instruction, 278 so; a
// table in fp64 725 and 346. The strained kernel, with both atoms' forces a pair at a time, took
// 1,488 and 2,582, and now 278 and 343.
template <typename T>
__device__ __forceinline__ void add_pair_forces(T* __restrict__ forces, index_t i, index_t j, T fx,
                                                T fy, T fz, int lane)
{
#pragma unroll
    for (int turn = 0; turn < 3; ++turn)
    {
        const int component = kWave * turn + lane;
        const int from = component / 3, axis = component - 3 * from;
        const index_t atom = __shfl(j, from, kWave);
        const T x = __shfl(fx, from, kWave), y = __shfl(fy, from, kWave),
                z = __shfl(fz, from, kWave);
        const T value = axis == 0 ? x : (axis == 1 ? y : z);
        if (atom >= 0) unsafeAtomicAdd(forces + 3LL * atom + axis, -value);
    }
    const index_t before = __shfl_up(i, 1, kWave);
    const bool head = lane == 0 || before != i;
    int start = head ? lane : 0;
#pragma unroll
    for (int offset = 1; offset < kWave; offset <<= 1)
    {
        const int other = __shfl_up(start, offset, kWave);
        if (lane >= offset && other > start) start = other;
    }
    const T sx = run_sum(fx, lane, start);
    const T sy = run_sum(fy, lane, start);
    const T sz = run_sum(fz, lane, start);
    const int next_start = __shfl_down(start, 1, kWave);
    const bool tail = lane == kWave - 1 || next_start != start;
    if (tail && i >= 0)
    {
        unsafeAtomicAdd(forces + 3LL * i, sx);
        unsafeAtomicAdd(forces + 3LL * i + 1, sy);
        unsafeAtomicAdd(forces + 3LL * i + 2, sz);
    }
}

// Writes this block's energy and virial sums to partials[8 * blockIdx.x ...].
template <bool kVirial, typename T>
__device__ __forceinline__ void store_partials(double energy, const T* w, double* shared,
                                               double* partials)
{
    const double e = block_sum(energy, shared);
    double v[6] = {0, 0, 0, 0, 0, 0};
    if (kVirial)
        for (int k = 0; k < 6; ++k) v[k] = block_sum(static_cast<double>(w[k]), shared);
    if (threadIdx.x == 0)
    {
        double* out = partials + 8LL * blockIdx.x;
        out[0] = e;
        for (int k = 0; k < 6; ++k) out[1 + k] = v[k];
        out[7] = 0.0;
    }
}

// Bytes of a potential's coefficients; without the reciprocals of a table's spacings on request.
std::int64_t coefficient_bytes(const ndn_potential* pot, int element, bool reciprocals = true);
int check_potential(const ndn_potential* pot, std::int64_t num_atoms);

template <typename T>
int prepare_potential(const ndn_potential* pot, void* workspace, hipStream_t stream,
                      PotentialView<T>* view);

template <typename T>
int finish(const double* partials, int blocks, void* energy, void* virial, double scale,
           hipStream_t stream);

}  // namespace ndn
