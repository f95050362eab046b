// Matrix-free stage kernel for quadrilaterals (parallelograms) and hexahedra
// (parallelepipeds) under the Global operator's flux (GlobalEvolution::Mult,
// GlobalEvolution.cpp:628-1088): the same semi-discrete operator the
// assembled matrix holds, applied without the matrix.  On the Gauss-Lobatto
// tensor element a reference derivative touches the p + 1 nodes of one grid
// line, and the lift of a face node reaches only the normal line through it
// (weight M1^-1[i, b], b = 0 or p the face's index on that line), so a node
// costs 6 DIM (p+1) multiply-adds and the HBM traffic per DOF is the state
// vectors and a share of the element's record.
//
// A block of six waves takes EB = 256 / Np elements:
//   1. state (four values per access, whole lines) and records into LDS; the
//      threads that form fluxes start their chain neighbour id -> neighbour
//      node -> exterior trace at the same time;
//   2. per face node: jump (or the boundary / interior-condition weights of
//      the own trace), flux fluxE = a (dE - n (n . dE)) + n x dH, fluxH = a
//      (dH - n (n . dH)) - n x dE, scaled by fscale/2 and 1/eps or 1/mu, into
//      LDS; a = 1 on SMA faces whatever alpha, as the Global operator
//      assembles them;
//   3. per node: metric-weighted tensor derivatives of the six components,
//      the curl, the lifted face fluxes, -sigma/eps E;
//   4. the right-hand sides through LDS, then the stage update, four values
//      per access.
// What bounds it is the vector-memory address path, not HBM: a 4-byte access
// of a wave occupies it as long as a 16-byte one, so state, records and update
// move in wide accesses and only the traces are gathered value by value.
// Measured per LSERK stage, order 3: 256^2 quadrilaterals FP64 46 us, FP32
// 25 us (assembled matrix: 375 and 290 us on a mesh with no two elements
// alike); 32^3 hexahedra FP64 141 us, FP32 55 us (164 and 57 us with 4-byte
// accesses, records read from memory and component-last flux tiles, whose
// stride of six words made the LDS banks collide).
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "stability.hpp"
#include "tensor_dev.hpp"

namespace dgtd {

namespace {

// Six waves: one component's part of the block is at most 64 vectors of four
// values, so each wave moves one component.
constexpr int kThreads = 384;

template <int P, int DIM>
struct Tensor {
    static constexpr int N1 = P + 1;
    static constexpr int NFP = DIM == 3 ? N1 * N1 : N1;
    static constexpr int NP = NFP * N1;
    static constexpr int NFACE = 2 * DIM;
    static constexpr int NF = NFACE * NFP;
    static constexpr int EB = 256 / NP;
    static constexpr int GEO = DIM == 3 ? kHexGeoDev : kQuadGeoDev;
    static constexpr int CONN = DIM == 3 ? kHexConnDev : kQuadConnDev;
    static constexpr int METRIC = DIM * DIM;      // record: metric, faces (normal, fscale/2), 1/eps, 1/mu, sigma/eps
    static constexpr int FREC = DIM + 1;
    static constexpr int NE = EB * NP;            // values per component and block
    static constexpr int FN = NF > NP ? NF : NP;  // LDS values per element and component: fluxes, then right-hand sides
};

// Four consecutive values, aligned to one value (the component stride is
// arbitrary), which global accesses allow.
template <typename T>
struct Wide {
    typedef T type __attribute__((ext_vector_type(4), aligned(sizeof(T))));
};

template <typename T, int P, int DIM, int MODE>
__global__ __launch_bounds__(kThreads) void tensor_stage(StageArgs<T> a)
{
    using S = Tensor<P, DIM>;
    constexpr int N1 = S::N1, NP = S::NP, NFP = S::NFP, NF = S::NF, EB = S::EB, NE = S::NE, FN = S::FN;
    using v4 = typename Wide<T>::type;
    __shared__ T sq[6 * NE];       // [c][el*NP + i]
    __shared__ T sf[6 * EB * FN];  // fluxes [el][c][f*NFP + b], then right-hand sides [c][el*NP + i]
    __shared__ T sg[EB * S::GEO];
    __shared__ T sD[N1 * N1];
    __shared__ T sMi[N1 * 2];
    const int t = threadIdx.x;
    const int K = a.K;
    const size_t N = (size_t)NP * K;
    // consecutive element blocks on one XCD (block b runs on XCD b % 8; the
    // grid is a multiple of 8), so neighbours' traces are in its L2
    const int blk = (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8);
    const int e0 = blk * EB;
    if (e0 >= K) return;
    const int ne = min(EB, K - e0);
    const bool full = ne == EB;
    const int cnt = ne * NP;

    // ---- every load that depends on nothing ----
    // lane l of wave c: values 4 l .. 4 l + 3 of component c's part of the
    // block (lanes past the end repeat the last vector, which overlaps its
    // predecessor when NE is no multiple of 4: the same values twice)
    const int c0 = __builtin_amdgcn_readfirstlane(t / 64);
    const int first = min(4 * (t % 64), NE - 4);
    const size_t off = (size_t)c0 * N + (size_t)e0 * NP;
    auto load = [&](const T* p) -> v4 {
        v4 v;
        if (full) {
            v = *reinterpret_cast<const v4*>(p + off + first);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = p[off + min(first + r, cnt - 1)];
        }
        return v;
    };
    const v4 q = load(a.qin);
    constexpr int NGL = (EB * S::GEO + kThreads - 1) / kThreads;
    T gv[NGL];
#pragma unroll
    for (int k = 0; k < NGL; ++k) gv[k] = a.geo[(size_t)e0 * S::GEO + min(t + kThreads * k, ne * S::GEO - 1)];
    // the thread's face nodes: neighbour, own and neighbour volume node
    constexpr int NS = (EB * NF + kThreads - 1) / kThreads;
    const int* fmask = a.tabs;      // [NFACE][NFP]
    const int* perm = a.tabs + NF;  // neighbour-node table rows of NFP
    int nb[NS], own[NS];
    T d[NS][6];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int s = min(t + kThreads * k, ne * NF - 1);
        const int el = s / NF, m = s - el * NF, f = m / NFP;
        const size_t rec = (size_t)(e0 + el) * S::CONN;
        nb[k] = a.conn[rec + f];
        const int row = a.conn[rec + S::NFACE + f];
        own[k] = fmask[m];
        // a boundary face reads the element's own trace (replaced below)
        const int pn = perm[(nb[k] >= 0 ? row : 0) * NFP + (m - f * NFP)];
        const size_t g = nb[k] >= 0 ? (size_t)nb[k] * NP + pn : (size_t)(e0 + el) * NP + own[k];
#pragma unroll
        for (int c = 0; c < 6; ++c) d[k][c] = a.qin[c * N + g];
    }
    // D1 row-major, then M1^-1 columns 0 and p
    if (t < N1 * N1) sD[t] = a.mats[t];
    if (t < N1 * 2) sMi[t] = a.mats[N1 * N1 + t];
    // the update's operands, in flight until the end
    constexpr bool kNeedRes = MODE != kModeMult && MODE != kModeRk1;
    constexpr bool kNeedX = MODE == kModeRk2 || MODE == kModeRk3;
    v4 rv = {T(0), T(0), T(0), T(0)}, xv;
    if constexpr (kNeedRes)
        if (MODE != kModeLserk || a.res_in) rv = load(a.res);
    if constexpr (kNeedX) xv = load(a.x);
#pragma unroll
    for (int r = 0; r < 4; ++r) sq[c0 * NE + first + r] = q[r];
#pragma unroll
    for (int k = 0; k < NGL; ++k)
        if (t + kThreads * k < EB * S::GEO) sg[t + kThreads * k] = gv[k];
    __syncthreads();

    // ---- fluxes ----
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int s = t + kThreads * k;
        if (s >= ne * NF) break;
        const int el = s / NF, m = s - el * NF, f = m / NFP;
        const T* g = sg + el * S::GEO;
        const T* fr = g + S::METRIC + S::FREC * f;
        const T* u = sq + el * NP + own[k];
        T al = a.alpha;
        T* dk = d[k];
        if (nb[k] >= 0) {
#pragma unroll
            for (int c = 0; c < 6; ++c) dk[c] -= u[c * NE];
        } else {
            const int bc = -nb[k] - 1;
            if (bc == 3 || bc == 6) al = T(1);
            const T sma = al != T(0) ? T(-1) / al : T(0);
            const T ce = bc == 1 ? T(-2) : bc == 3 ? sma : bc == 4 ? T(-1) : bc == 6 ? T(-0.5) : T(0);
            const T ch = bc == 2 ? T(-2) : bc == 3 ? sma : bc == 5 ? T(-1) : bc == 6 ? T(-0.5) : T(0);
#pragma unroll
            for (int c = 0; c < 6; ++c) dk[c] = (c < 3 ? ce : ch) * u[c * NE];
        }
        T n[3] = {fr[0], fr[1], T(0)};
        if constexpr (DIM == 3) n[2] = fr[2];
        const T fs = fr[DIM];
        const T nE = n[0] * dk[0] + n[1] * dk[1] + n[2] * dk[2], nH = n[0] * dk[3] + n[1] * dk[4] + n[2] * dk[5];
        const T se = fs * g[S::GEO - 3], sh = fs * g[S::GEO - 2];
        T* o = sf + el * 6 * FN + m;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            const int y = (x + 1) % 3, z = (x + 2) % 3;
            o[x * FN] = se * (al * (dk[x] - n[x] * nE) + (n[y] * dk[3 + z] - n[z] * dk[3 + y]));
            o[(3 + x) * FN] = sh * (al * (dk[3 + x] - n[x] * nH) - (n[y] * dk[z] - n[z] * dk[y]));
        }
    }
    __syncthreads();

    // ---- right-hand sides, a node per thread (the first NE threads) ----
    const bool node = t < cnt;
    const int el = t / NP, i = t - el * NP;
    const int ix = i % N1, iy = i / N1 % N1, iz = DIM == 3 ? i / NFP : 0;
    T rhs[6];
    if (node) {
        const T* g = sg + el * S::GEO;
        const T* uo = sq + el * NP;
        // physical derivatives: D_d u = sum_k G[k][d] d_k u
        T du[6][DIM];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const T* u = uo + c * NE;
            T ud[3] = {T(0), T(0), T(0)};
#pragma unroll
            for (int m = 0; m < N1; ++m) {
                ud[0] += sD[ix * N1 + m] * u[i + m - ix];
                ud[1] += sD[iy * N1 + m] * u[i + N1 * (m - iy)];
                if constexpr (DIM == 3) ud[2] += sD[iz * N1 + m] * u[i + NFP * (m - iz)];
            }
#pragma unroll
            for (int dd = 0; dd < DIM; ++dd) {
                T v = g[dd] * ud[0] + g[DIM + dd] * ud[1];
                if constexpr (DIM == 3) v += g[2 * DIM + dd] * ud[2];
                du[c][dd] = v;
            }
        }
        const T ieps = g[S::GEO - 3], imu = g[S::GEO - 2], sig = g[S::GEO - 1];
        auto dd = [&](int c, int dir) { return dir < DIM ? du[c][dir < DIM ? dir : 0] : T(0); };
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            const int y = (x + 1) % 3, z = (x + 2) % 3;
            rhs[x] = ieps * (dd(3 + z, y) - dd(3 + y, z)) - sig * uo[x * NE + i];
            rhs[3 + x] = imu * (dd(y, z) - dd(z, y));
        }
        // lifted fluxes: face f's node on this node's normal line (its
        // numbering follows the face's vertex cycle), weight M1^-1[line
        // index][0 or p]
        auto lift = [&](int f, int line, int end, int b) {
            const T w = sMi[line * 2 + end];
            const T* fl = sf + el * 6 * FN + f * NFP + b;
#pragma unroll
            for (int c = 0; c < 6; ++c) rhs[c] += w * fl[c * FN];
        };
        if constexpr (DIM == 3) {
            lift(0, iz, 0, ix + N1 * (P - iy));
            lift(1, iy, 0, ix + N1 * iz);
            lift(2, ix, 1, iy + N1 * iz);
            lift(3, iy, 1, P - ix + N1 * iz);
            lift(4, ix, 0, P - iy + N1 * iz);
            lift(5, iz, 1, ix + N1 * iy);
        } else {
            lift(0, iy, 0, ix);
            lift(1, ix, 1, iy);
            lift(2, iy, 1, P - ix);
            lift(3, ix, 0, P - iy);
        }
    }
    __syncthreads();
    if (node) {
#pragma unroll
        for (int c = 0; c < 6; ++c) sf[c * NE + t] = rhs[c];
    }
    __syncthreads();

    // ---- stage update ----
    bool bad = false;
    v4 o, r2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const T v = sf[c0 * NE + first + r], qv = q[r];
        if constexpr (MODE == kModeMult) {
            o[r] = v;
        } else if constexpr (MODE == kModeLserk) {
            r2[r] = a.ca * rv[r] + a.dt * v;
            o[r] = qv + a.cb * r2[r];
        } else if constexpr (MODE == kModeRk1) {
            o[r] = qv + a.ca * v;
            r2[r] = qv + a.cb * v;
        } else if constexpr (MODE == kModeRk2 || MODE == kModeRk3) {
            o[r] = xv[r] + a.ca * v;
            r2[r] = rv[r] + a.cb * v;
        } else {
            o[r] = rv[r] + a.ca * v;
        }
        if constexpr (MODE == kModeLserk || MODE == kModeRk4) bad = bad || (first + r < cnt && unstable_entry(o[r]));
    }
    constexpr bool kRes = MODE != kModeMult && MODE != kModeRk4;
    const bool keep = MODE != kModeLserk || a.res_out;
    if (full) {
        if constexpr (kRes)
            if (keep) *reinterpret_cast<v4*>(a.res + off + first) = r2;
        *reinterpret_cast<v4*>(a.out + off + first) = o;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (first + r < cnt) {
                if constexpr (kRes)
                    if (keep) a.res[off + first + r] = r2[r];
                a.out[off + first + r] = o[r];
            }
    }
    if constexpr (MODE == kModeLserk || MODE == kModeRk4) report_unstable(a.unstable, bad);
}

template <typename T, int P, int DIM>
hipError_t tensor_launch(const StageArgs<T>& a, int mode, hipStream_t s)
{
    constexpr int EB = Tensor<P, DIM>::EB;
    const int blocks = (a.K + EB - 1) / EB;
    const dim3 g((unsigned)((blocks + 7) / 8 * 8)), b(kThreads);
    switch (mode) {
        case kModeMult: hipLaunchKernelGGL((tensor_stage<T, P, DIM, kModeMult>), g, b, 0, s, a); break;
        case kModeLserk: hipLaunchKernelGGL((tensor_stage<T, P, DIM, kModeLserk>), g, b, 0, s, a); break;
        case kModeRk1: hipLaunchKernelGGL((tensor_stage<T, P, DIM, kModeRk1>), g, b, 0, s, a); break;
        case kModeRk2: hipLaunchKernelGGL((tensor_stage<T, P, DIM, kModeRk2>), g, b, 0, s, a); break;
        case kModeRk3: hipLaunchKernelGGL((tensor_stage<T, P, DIM, kModeRk3>), g, b, 0, s, a); break;
        case kModeRk4: hipLaunchKernelGGL((tensor_stage<T, P, DIM, kModeRk4>), g, b, 0, s, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

template <typename T>
hipError_t launch_tensor_stage(int order, int dim, const StageArgs<T>& a, int mode, hipStream_t s)
{
    if (a.K <= 0) return hipErrorInvalidValue;
    switch (10 * dim + order) {
        case 21: return tensor_launch<T, 1, 2>(a, mode, s);
        case 22: return tensor_launch<T, 2, 2>(a, mode, s);
        case 23: return tensor_launch<T, 3, 2>(a, mode, s);
        case 24: return tensor_launch<T, 4, 2>(a, mode, s);
        case 25: return tensor_launch<T, 5, 2>(a, mode, s);
        case 31: return tensor_launch<T, 1, 3>(a, mode, s);
        case 32: return tensor_launch<T, 2, 3>(a, mode, s);
        case 33: return tensor_launch<T, 3, 3>(a, mode, s);
        case 34: return tensor_launch<T, 4, 3>(a, mode, s);
        case 35: return tensor_launch<T, 5, 3>(a, mode, s);
        default: return hipErrorInvalidValue;
    }
}

template hipError_t launch_tensor_stage<float>(int, int, const StageArgs<float>&, int, hipStream_t);
template hipError_t launch_tensor_stage<double>(int, int, const StageArgs<double>&, int, hipStream_t);

}  // namespace dgtd
