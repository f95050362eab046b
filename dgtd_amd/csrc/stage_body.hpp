// Device body of the per-node (VALU) fused DGTD stage, shared by the
// single-mesh kernel (dg_kernels.hip) and the multi-instance batch kernel
// (dg_batch.hip).  See dg_kernels.hip for the algorithm.
#pragma once

#include <hip/hip_runtime.h>

#include "bc_coeffs.hpp"
#include "kernels.hpp"
#include "lds_copy.hpp"
#include "stability.hpp"

namespace dgtd {
namespace valu {

// SMALL: element blocks half as large, for meshes that leave CUs idle
// (StageArgs::small_blocks).  A block's LDS reads in the products go through
// its CU's one LDS, so half the elements finish sooner: order 3 FP64, 48
// tetrahedra: 8.3 -> 7.8 us per stage; order 1 FP32, 1,296: 5.2 -> 4.8; order 2
// FP32, 3,072: 6.6 -> 6.0.  A quarter of the elements gains no more, and two
// half blocks on a CU instead of one block lose (order 3 FP64, 3,072: 9.8 ->
// 10.3 us).
template <int P, bool SMALL = false>
struct Shape {
    static constexpr int NP = (P + 1) * (P + 2) * (P + 3) / 6;
    static constexpr int NFP = (P + 1) * (P + 2) / 2;
    static constexpr int NF = 4 * NFP;
    static constexpr int EB = (SMALL ? 128 : 256) / NP;  // elements per block
};

template <int P, typename T, bool SMALL = false>
struct Smem {
    using S = Shape<P, SMALL>;
    static constexpr int nD = 3 * S::NP * S::NP;
    static constexpr int nL = S::NF * S::NP;
    static constexpr int nQ = 6 * S::EB * S::NP;
    static constexpr int nF = 6 * S::EB * S::NF;
    static constexpr int nG = S::EB * kGeoStrideDev;
    static constexpr int nReal = nD + nL + nQ + nF + nG;
    static constexpr int nInt = S::EB * kConnStrideDev + 4 * S::NFP + 96 * S::NFP;
    static constexpr size_t bytes = sizeof(T) * (size_t)nReal + sizeof(int) * (size_t)nInt;
};

// Threads per block of the per-node kernels (single-mesh and batch).
constexpr int kThreads = 256;

// A block's fields and records on their way from memory into LDS.
template <int P, typename T, bool SMALL = false>
struct Fetched {
    using S = Shape<P, SMALL>;
    static constexpr int NG = (S::EB * kGeoStrideDev + kThreads - 1) / kThreads;
    static constexpr int NC = (S::EB * kConnStrideDev + kThreads - 1) / kThreads;
    T q[6], g[NG];
    int c[NC];
};

// Issues every load of element block blk's fields and records (threads past
// the end load a clamped, valid address).
template <int P, typename T, bool SMALL = false>
__device__ __forceinline__ void stage_fetch(const StageArgs<T>& a, int blk, Fetched<P, T, SMALL>& f)
{
    using S = Shape<P, SMALL>;
    constexpr int NP = S::NP, EB = S::EB;
    const int tid = threadIdx.x;
    const size_t N = (size_t)NP * a.K;
    const int e0 = blk * EB;
    const int ne = min(EB, a.K - e0);
    const size_t base = (size_t)e0 * NP;
    const int cnt = ne * NP, ng = ne * kGeoStrideDev, nc = ne * kConnStrideDev;
    const int iq = tid < cnt ? tid : cnt - 1;
#pragma unroll
    for (int c = 0; c < 6; ++c) f.q[c] = a.qin[c * N + base + iq];
#pragma unroll
    for (int k = 0; k < Fetched<P, T, SMALL>::NG; ++k) {
        const int i = tid + k * kThreads;
        f.g[k] = a.geo[(size_t)e0 * kGeoStrideDev + (i < ng ? i : ng - 1)];
    }
#pragma unroll
    for (int k = 0; k < Fetched<P, T, SMALL>::NC; ++k) {
        const int i = tid + k * kThreads;
        f.c[k] = a.conn[(size_t)e0 * kConnStrideDev + (i < nc ? i : nc - 1)];
    }
}

// Loads the order-P reference matrices and tables into LDS (block-wide;
// stage_block's first barrier follows).  The tables' loads are issued before
// the matrices', of which several are in flight per thread (up to 55 values
// per thread at order 5), so one memory latency covers both.
template <int P, typename T, bool SMALL = false>
__device__ __forceinline__ void stage_load_ref(const T* __restrict__ mats, const int* __restrict__ tabs,
                                               unsigned char* smem_raw)
{
    using S = Shape<P, SMALL>;
    using L = Smem<P, T, SMALL>;
    constexpr int NT = 4 * S::NFP + 96 * S::NFP, NTT = (NT + kThreads - 1) / kThreads;
    T* sD = reinterpret_cast<T*>(smem_raw);
    int* sFm = reinterpret_cast<int*>(sD + L::nReal) + S::EB * kConnStrideDev;
    const int tid = threadIdx.x;
    int tv[NTT];
#pragma unroll
    for (int k = 0; k < NTT; ++k) {
        const int i = tid + k * kThreads;
        tv[k] = tabs[i < NT ? i : NT - 1];
    }
    lds_copy<8>(sD, mats, L::nD + L::nL, tid, kThreads);
#pragma unroll
    for (int k = 0; k < NTT; ++k)
        if (tid + k * kThreads < NT) sFm[tid + k * kThreads] = tv[k];
}

// One element block (EB elements from e0 = blk*EB, fetched in f) of one stage:
// gather, flux, curl, LIFT and the stage update.  The reference matrices are in
// LDS or on their way there (its first barrier waits for them); the caller puts
// a block-wide barrier between two element blocks.
// GLOBAL: the Global operator's form of the same stage (GlobalEvolution.cpp:
// 628-1088): SMA faces weighted as at alpha = 1 (DGOperatorFactory.h:485-495,
// 587-591) and -sigma/eps E on the E rows (:1351-1361).
template <int P, typename T, int MODE, bool GLOBAL = false, bool KEEP = false, bool SMALL = false>
__device__ __forceinline__ void stage_block(const StageArgs<T>& a, unsigned char* smem_raw, int blk,
                                            const Fetched<P, T, SMALL>& fetched)
{
    using S = Shape<P, SMALL>;
    using L = Smem<P, T, SMALL>;
    constexpr int NP = S::NP, NFP = S::NFP, NF = S::NF, EB = S::EB;
    T* sD = reinterpret_cast<T*>(smem_raw);  // [3][j][i]
    T* sL = sD + L::nD;                      // [m][i]
    T* sQ = sL + L::nL;                      // [c][el*NP + j]
    T* sF = sQ + L::nQ;                      // [c][el*NF + m]
    T* sG = sF + L::nF;                      // [el][kGeoStride]
    int* sC = reinterpret_cast<int*>(sG + L::nG);  // [el][kConnStride]
    int* sFm = sC + EB * kConnStrideDev;            // [4*NFP]
    int* sPt = sFm + 4 * NFP;                       // [96*NFP]

    const int tid = threadIdx.x;
    const int K = a.K;
    const size_t N = (size_t)NP * K;
    static_assert(EB * NP <= kThreads, "one volume node per thread");
    {
        const int e0 = blk * EB;
        const int ne = min(EB, K - e0);
        {
            const int cnt = ne * NP, ng = ne * kGeoStrideDev, nc = ne * kConnStrideDev;
            if (tid < cnt) {
#pragma unroll
                for (int c = 0; c < 6; ++c) sQ[c * EB * NP + tid] = fetched.q[c];
            }
#pragma unroll
            for (int k = 0; k < Fetched<P, T, SMALL>::NG; ++k)
                if (tid + k * kThreads < ng) sG[tid + k * kThreads] = fetched.g[k];
#pragma unroll
            for (int k = 0; k < Fetched<P, T, SMALL>::NC; ++k)
                if (tid + k * kThreads < nc) sC[tid + k * kThreads] = fetched.c[k];
        }
        __syncthreads();

        // ---- surface: jumps, boundary conditions, flux, fscale/2 ----
        // A thread's face nodes (at most NS): first every exterior trace is
        // gathered, then the fluxes are formed.
        constexpr int NS = (EB * NF + kThreads - 1) / kThreads;
        const int nsf = ne * NF;
        T uM[NS][6], d[NS][6];
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const int s = tid + k * kThreads < nsf ? tid + k * kThreads : nsf - 1;
            const int el = s / NF;
            const int m = s - el * NF;
            const int f = m / NFP;
            const int b = m - f * NFP;
            const int nb = sC[el * kConnStrideDev + f];
            const int iM = sFm[f * NFP + b];
#pragma unroll
            for (int c = 0; c < 6; ++c) uM[k][c] = sQ[c * EB * NP + el * NP + iM];
            // a boundary face reads the element's own node (its value is
            // replaced below)
            const int code = sC[el * kConnStrideDev + 4 + f];
            const size_t gP = nb >= 0 ? (size_t)nb * NP + sPt[code * NFP + b] : (size_t)(e0 + el) * NP + iM;
#pragma unroll
            for (int c = 0; c < 6; ++c) d[k][c] = a.qin[c * N + gP];
        }
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const int s = tid + k * kThreads;
            if (s >= nsf) break;
            const int el = s / NF;
            const int m = s - el * NF;
            const int f = m / NFP;
            const T* g = sG + el * kGeoStrideDev;
            const int nb = sC[el * kConnStrideDev + f];
            T* dk = d[k];
            T alpha = a.alpha;
            if (nb >= 0) {
#pragma unroll
                for (int c = 0; c < 6; ++c) dk[c] -= uM[k][c];
            } else {
                if constexpr (GLOBAL)
                    if (-nb - 1 == 3 || -nb - 1 == 6) alpha = T(1);
                T ce, ch;
                bc_coeffs<T>(-nb - 1, alpha, ce, ch);
#pragma unroll
                for (int c = 0; c < 3; ++c) { dk[c] = ce * uM[k][c]; dk[3 + c] = ch * uM[k][3 + c]; }
            }
            const T nx = g[9 + 4 * f], ny = g[10 + 4 * f], nz = g[11 + 4 * f], fs = g[12 + 4 * f];
            const T n3[3] = {nx, ny, nz};
            const T ndH = nx * dk[3] + ny * dk[4] + nz * dk[5];
            const T ndE = nx * dk[0] + ny * dk[1] + nz * dk[2];
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                const int y = (x + 1) % 3, z = (x + 2) % 3;
                const T fH = -n3[y] * dk[z] + n3[z] * dk[y] + alpha * (dk[3 + x] - ndH * n3[x]);
                const T fE = n3[y] * dk[3 + z] - n3[z] * dk[3 + y] + alpha * (dk[x] - ndE * n3[x]);
                sF[(3 + x) * EB * NF + el * NF + m] = fH * fs;
                sF[x * EB * NF + el * NF + m] = fE * fs;
            }
        }
        __syncthreads();

        // ---- volume: curl + LIFT, stage update ----
        bool bad = false;  // an unstable state entry stored by this thread (a.unstable set)
        if (tid < ne * NP) {
            const int t = tid;
            const int el = t / NP;
            const int i = t - el * NP;
            const size_t idx = (size_t)(e0 + el) * NP + i;
            // the stage's reads of the residual / base state, issued before
            // the products (all reads before the first store, see the MFMA variant)
            T rv[6], xv[6];
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                if constexpr (MODE == kModeLserk || MODE == kModeLserkLast || MODE == kModeRk2 || MODE == kModeRk3 ||
                              MODE == kModeRk4)
                    rv[c] = __builtin_nontemporal_load(a.res + c * N + idx);
                if constexpr (MODE == kModeRk2 || MODE == kModeRk3) xv[c] = a.x[c * N + idx];
            }
            T sg = T(0);
            if constexpr (GLOBAL)
                if (a.sig != nullptr) sg = a.sig[e0 + el];
            T ar[6], as[6], at[6], lf[6];
#pragma unroll
            for (int c = 0; c < 6; ++c) { ar[c] = T(0); as[c] = T(0); at[c] = T(0); lf[c] = T(0); }
#pragma unroll 5
            for (int j = 0; j < NP; ++j) {
                const T dr = sD[j * NP + i], ds = sD[NP * NP + j * NP + i], dt = sD[2 * NP * NP + j * NP + i];
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    const T u = sQ[c * EB * NP + el * NP + j];
                    ar[c] += dr * u;
                    as[c] += ds * u;
                    at[c] += dt * u;
                }
            }
#pragma unroll 4
            for (int m = 0; m < NF; ++m) {
                const T l = sL[m * NP + i];
#pragma unroll
                for (int c = 0; c < 6; ++c) lf[c] += l * sF[c * EB * NF + el * NF + m];
            }
            const T* g = sG + el * kGeoStrideDev;
            // D_d u = r_d ur + s_d us + t_d ut
            auto Dd = [&](int dd, int c) { return g[dd] * ar[c] + g[3 + dd] * as[c] + g[6 + dd] * at[c]; };
            T rhs[6];
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                const int y = (x + 1) % 3, z = (x + 2) % 3;
                rhs[3 + x] = (-Dd(y, z) + Dd(z, y) + lf[3 + x]) * g[26];
                rhs[x] = (Dd(y, 3 + z) - Dd(z, 3 + y) + lf[x]) * g[25];
                if constexpr (GLOBAL) rhs[x] -= sg * sQ[x * EB * NP + el * NP + i];
            }
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                const size_t o = c * N + idx;
                const T qv = sQ[c * EB * NP + el * NP + i];
                auto store_out = [&](T v) {
                    if constexpr (KEEP) a.out[o] = v;
                    else __builtin_nontemporal_store(v, a.out + o);
                };
                if constexpr (MODE == kModeMult) {
                    store_out(rhs[c]);
                } else if constexpr (is_lserk(MODE)) {
                    T r = a.dt * rhs[c];
                    if constexpr (MODE != kModeLserkFirst) r = a.ca * rv[c] + r;
                    const T qn = qv + a.cb * r;
                    if constexpr (MODE != kModeLserkLast) __builtin_nontemporal_store(r, a.res + o);
                    store_out(qn);
                    bad = bad || unstable_entry(qn);
                } else if constexpr (MODE == kModeRk1) {
                    store_out(qv + a.ca * rhs[c]);
                    __builtin_nontemporal_store(qv + a.cb * rhs[c], a.res + o);
                } else if constexpr (MODE == kModeRk2 || MODE == kModeRk3) {
                    store_out(xv[c] + a.ca * rhs[c]);
                    __builtin_nontemporal_store(rv[c] + a.cb * rhs[c], a.res + o);
                } else {  // kModeRk4
                    const T qn = rv[c] + a.ca * rhs[c];
                    store_out(qn);
                    bad = bad || unstable_entry(qn);
                }
            }
        }
        if constexpr (is_lserk(MODE) || MODE == kModeRk4) report_unstable(a.unstable, bad);
    }
}

}  // namespace valu
}  // namespace dgtd
