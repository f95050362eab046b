// Fused DGTD Maxwell stage kernels for gfx950 (the "hesthaven" operator of
// OpenSEMBA/dgtd, HesthavenEvolution.cpp:450-542, with the RK stage update).
//
// One launch = one Runge-Kutta stage over all elements:
//   1. stage the block's fields (6 x Np per element), geometry and
//      connectivity records in LDS (coalesced: component-major state, one
//      contiguous chunk per component per element block);
//   2. per face node: gather the neighbour trace through (neighbour id,
//      permutation code), apply PEC/PMC/SMA, form the upwind/centred flux and
//      scale it by fscale/2 -- into LDS, never to HBM;
//   3. per volume node: reference derivatives [Dr;Ds;Dt] of the 6 fields and
//      LIFT * flux from LDS-resident reference matrices, metric combine into
//      the curl, 1/eps and 1/mu, then the stage update, writing each state
//      buffer once.
// Blocks are persistent (grid = resident capacity) and loop over element
// blocks, so the reference matrices are staged once per block.
//
// The Global operator (GLOBAL kernels, StageArgs::global) is the same
// semi-discrete operator with fully upwinded SMA faces and conductivity, so it
// runs here and no matrix is read: 24 Np values per element and stage instead
// of the matrix's 190 entries per row at order 3 (10,368 tetrahedra with no two
// alike, FP32 order 3: 659 us per stage from the assembled matrix, 13.2 us
// here).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.hpp"
#include "stage_body.hpp"

namespace dgtd {

namespace {

using namespace valu;

// The element blocks of one thread block.  The first one's fields and records,
// the tables and the matrices travel together, one memory latency instead of
// three on a mesh of a block or two per CU (order 3 FP64, 48 / 3,072
// tetrahedra: 8.7 -> 8.2 and 10.2 -> 9.8 us per stage; order 1 FP32, 1,296:
// 5.4 -> 5.2 us; order 3 FP32, 24,576: 23.3 -> 22.1 us).
template <int P, typename T, int MODE, bool GLOBAL, bool KEEP, bool SMALL>
__device__ __forceinline__ void stage_blocks(const StageArgs<T>& a, unsigned char* smem_raw)
{
    int blk = blockIdx.x;
    if (blk >= a.nblk) return;
    Fetched<P, T, SMALL> f;
    stage_fetch<P, T, SMALL>(a, blk, f);
    stage_load_ref<P, T, SMALL>(a.mats, a.tabs, smem_raw);
    for (;;) {
        stage_block<P, T, MODE, GLOBAL, KEEP, SMALL>(a, smem_raw, blk, f);
        blk += gridDim.x;
        if (blk >= a.nblk) break;
        __syncthreads();  // LDS tiles free for the next block
        stage_fetch<P, T, SMALL>(a, blk, f);
    }
}

template <int P, typename T, int MODE, bool GLOBAL, bool SMALL>
__global__ __launch_bounds__(256) void dg_stage_kernel(StageArgs<T> a)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    if (!SMALL && a.keep_out) stage_blocks<P, T, MODE, GLOBAL, true, SMALL>(a, smem_raw);
    else stage_blocks<P, T, MODE, GLOBAL, false, SMALL>(a, smem_raw);
}

// A mesh of small blocks is far below the state size from which the shortened
// LSERK4 stages are used, so those have no SMALL form.
template <int MODE>
constexpr bool has_small() { return MODE != kModeLserkFirst && MODE != kModeLserkLast; }

template <int P, typename T, int MODE, bool SMALL>
hipError_t launch_one(const StageArgs<T>& a, int grid, hipStream_t s)
{
    if constexpr (SMALL && !has_small<MODE>()) {
        return hipErrorInvalidValue;
    } else {
        constexpr size_t bytes = Smem<P, T, SMALL>::bytes;
        auto kern = a.global ? dg_stage_kernel<P, T, MODE, true, SMALL> : dg_stage_kernel<P, T, MODE, false, SMALL>;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(256), bytes, s, a);
        return hipGetLastError();
    }
}

template <int P, typename T, int MODE>
hipError_t launch_size(const StageArgs<T>& a, int grid, hipStream_t s)
{
    return a.small_blocks ? launch_one<P, T, MODE, true>(a, grid, s) : launch_one<P, T, MODE, false>(a, grid, s);
}

template <int P, typename T>
hipError_t launch_mode(const StageArgs<T>& a, int mode, int grid, hipStream_t s)
{
    switch (lserk_mode(a, mode)) {
        case kModeMult: return launch_size<P, T, kModeMult>(a, grid, s);
        case kModeLserk: return launch_size<P, T, kModeLserk>(a, grid, s);
        case kModeLserkFirst: return launch_size<P, T, kModeLserkFirst>(a, grid, s);
        case kModeLserkLast: return launch_size<P, T, kModeLserkLast>(a, grid, s);
        case kModeRk1: return launch_size<P, T, kModeRk1>(a, grid, s);
        case kModeRk2: return launch_size<P, T, kModeRk2>(a, grid, s);
        case kModeRk3: return launch_size<P, T, kModeRk3>(a, grid, s);
        case kModeRk4: return launch_size<P, T, kModeRk4>(a, grid, s);
        default: return hipErrorInvalidValue;
    }
}

template <int P, typename T, int MODE>
void set_smem_attr()
{
    for (const void* kern : {reinterpret_cast<const void*>(dg_stage_kernel<P, T, MODE, false, false>),
                             reinterpret_cast<const void*>(dg_stage_kernel<P, T, MODE, true, false>)})
        (void)hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Smem<P, T>::bytes);
    if constexpr (has_small<MODE>())
        for (const void* kern : {reinterpret_cast<const void*>(dg_stage_kernel<P, T, MODE, false, true>),
                                 reinterpret_cast<const void*>(dg_stage_kernel<P, T, MODE, true, true>)})
            (void)hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Smem<P, T, true>::bytes);
}

// Raises the dynamic-LDS limit of every stage variant of this order (needed
// above 64 KiB) and returns resident blocks per CU.
template <int P, typename T>
int occupancy_one()
{
    int nb = 0;
    constexpr size_t bytes = Smem<P, T>::bytes;
    set_smem_attr<P, T, kModeMult>();
    set_smem_attr<P, T, kModeLserk>();
    set_smem_attr<P, T, kModeLserkFirst>();
    set_smem_attr<P, T, kModeLserkLast>();
    set_smem_attr<P, T, kModeRk1>();
    set_smem_attr<P, T, kModeRk2>();
    set_smem_attr<P, T, kModeRk3>();
    set_smem_attr<P, T, kModeRk4>();
    auto kern = dg_stage_kernel<P, T, kModeLserk, false, false>;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, 256, bytes) != hipSuccess) return 1;
    return nb > 0 ? nb : 1;
}

}  // namespace

template <typename T>
hipError_t launch_stage(int order, const StageArgs<T>& a, int mode, int grid, hipStream_t s)
{
    switch (order) {
        case 1: return launch_mode<1, T>(a, mode, grid, s);
        case 2: return launch_mode<2, T>(a, mode, grid, s);
        case 3: return launch_mode<3, T>(a, mode, grid, s);
        case 4: return launch_mode<4, T>(a, mode, grid, s);
        case 5: return launch_mode<5, T>(a, mode, grid, s);
        default: return hipErrorInvalidValue;
    }
}

template <typename T>
int stage_blocks_per_cu(int order)
{
    switch (order) {
        case 1: return occupancy_one<1, T>();
        case 2: return occupancy_one<2, T>();
        case 3: return occupancy_one<3, T>();
        case 4: return occupancy_one<4, T>();
        case 5: return occupancy_one<5, T>();
        default: return 1;
    }
}

int elements_per_block(int order, bool small)
{
    switch (order) {
        case 1: return small ? Shape<1, true>::EB : Shape<1>::EB;
        case 2: return small ? Shape<2, true>::EB : Shape<2>::EB;
        case 3: return small ? Shape<3, true>::EB : Shape<3>::EB;
        case 4: return small ? Shape<4, true>::EB : Shape<4>::EB;
        case 5: return small ? Shape<5, true>::EB : Shape<5>::EB;
        default: return 1;
    }
}

template hipError_t launch_stage<double>(int, const StageArgs<double>&, int, int, hipStream_t);
template hipError_t launch_stage<float>(int, const StageArgs<float>&, int, int, hipStream_t);
template int stage_blocks_per_cu<double>(int);
template int stage_blocks_per_cu<float>(int);

}  // namespace dgtd
