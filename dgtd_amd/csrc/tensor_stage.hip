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
// A block takes EB = 256 / Np elements:
//   1. state and records into LDS, a node per thread and its six components;
//      the threads that form fluxes start their chain neighbour id ->
//      neighbour node -> exterior trace before that;
//   2. per face node: jump (or the boundary / interior-condition weights of
//      the own trace), flux fluxE = a (dE - n (n . dE)) + n x dH, fluxH = a
//      (dH - n (n . dH)) - n x dE, scaled by fscale/2 and 1/eps or 1/mu, into
//      LDS (component-major: component-last tiles, a stride of six words, made
//      the banks collide); a = 1 on SMA faces whatever alpha, as the Global
//      operator assembles them;
//   3. per node: metric-weighted tensor derivatives of the six components,
//      the curl, the lifted face fluxes, -sigma/eps E and the stage update of
//      the node's six values.
// Large meshes run at the memory rate, small ones at the latency of that chain.
// An earlier form moved state and update in 16- and 32-byte accesses by six
// waves, one component each; the right-hand sides then crossed LDS behind two
// more barriers, a third of the waves idled in the products, and an FP64 lane's
// 32 bytes half-filled each access.  Per stage, that form -> this one, 8
// million unknowns: hexahedra order 1 FP64 106 -> 73 us (operator alone 97 ->
// 63), order 3 FP32 38 -> 29 and FP64 75 -> 55, order 5 FP64 79 -> 57 (66 ->
// 45); quadrilaterals order 3 FP32 29 -> 24 and FP64 54 -> 42, order 5 FP64
// 65 -> 42.  Order-5 hexahedra in FP32 below 20,000 unknowns lose: 4.9 -> 5.0.
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "stability.hpp"
#include "tensor_dev.hpp"

namespace dgtd {

namespace {

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
};

template <typename T, int P, int DIM, int MODE, int kThreads>
__global__ __launch_bounds__(kThreads) void tensor_stage(StageArgs<T> a)
{
    using S = Tensor<P, DIM>;
    constexpr int N1 = S::N1, NP = S::NP, NFP = S::NFP, NF = S::NF, EB = S::EB, NE = S::NE;
    __shared__ T sq[6 * NE];       // [c][el*NP + i]
    __shared__ T sf[6 * EB * NF];  // fluxes [el][c][f*NFP + b]
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
    const int cnt = ne * NP;

    // ---- loads (threads past the end repeat the last node's or face node's) ----
    // the longest chain first: neighbour and table row, neighbour node, trace
    constexpr int NS = (EB * NF + kThreads - 1) / kThreads;
    const int* fmask = a.tabs;      // [NFACE][NFP]
    const int* perm = a.tabs + NF;  // neighbour-node table rows of NFP
    int nb[NS], row[NS], own[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int s = min(t + kThreads * k, ne * NF - 1);
        const int el = s / NF, m = s - el * NF;
        const size_t rec = (size_t)(e0 + el) * S::CONN + m / NFP;
        nb[k] = a.conn[rec];
        row[k] = a.conn[rec + S::NFACE];
        own[k] = fmask[m];
    }
    const bool node = t < cnt;
    const size_t own0 = (size_t)e0 * NP + min(t, cnt - 1);
    T q[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) q[c] = a.qin[c * N + own0];
    constexpr int NGL = (EB * S::GEO + kThreads - 1) / kThreads;
    T gv[NGL];
#pragma unroll
    for (int k = 0; k < NGL; ++k) gv[k] = a.geo[(size_t)e0 * S::GEO + min(t + kThreads * k, ne * S::GEO - 1)];
    T d[NS][6];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int s = min(t + kThreads * k, ne * NF - 1);
        const int el = s / NF, m = s - el * NF;
        // a boundary face reads the element's own trace (replaced below)
        const int pn = perm[(nb[k] >= 0 ? row[k] : 0) * NFP + m % NFP];
        const size_t g = nb[k] >= 0 ? (size_t)nb[k] * NP + pn : (size_t)(e0 + el) * NP + own[k];
#pragma unroll
        for (int c = 0; c < 6; ++c) d[k][c] = a.qin[c * N + g];
    }
    // D1 row-major, then M1^-1 columns 0 and p
    if (t < N1 * N1) sD[t] = a.mats[t];
    if (t < N1 * 2) sMi[t] = a.mats[N1 * N1 + t];
    if (node) {
#pragma unroll
        for (int c = 0; c < 6; ++c) sq[c * NE + t] = q[c];
    }
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
        T* o = sf + el * 6 * NF + m;
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            const int y = (x + 1) % 3, z = (x + 2) % 3;
            o[x * NF] = se * (al * (dk[x] - n[x] * nE) + (n[y] * dk[3 + z] - n[z] * dk[3 + y]));
            o[(3 + x) * NF] = sh * (al * (dk[3 + x] - n[x] * nH) - (n[y] * dk[z] - n[z] * dk[y]));
        }
    }
    __syncthreads();

    // the update's operands, in flight during the products
    constexpr bool kNeedRes = MODE == kModeLserk || MODE == kModeLserkLast || MODE == kModeRk2 || MODE == kModeRk3 ||
                              MODE == kModeRk4;
    constexpr bool kNeedX = MODE == kModeRk2 || MODE == kModeRk3;
    T rv[6], xv[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        if constexpr (kNeedRes) rv[c] = a.res[c * N + own0];
        if constexpr (kNeedX) xv[c] = a.x[c * N + own0];
    }

    // ---- right-hand sides and stage update, a node per thread (the first NE threads) ----
    const int el = t / NP, i = t - el * NP;
    const int ix = i % N1, iy = i / N1 % N1, iz = DIM == 3 ? i / NFP : 0;
    bool bad = false;
    if (node) {
        T rhs[6];
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
        // lifted fluxes: face f's node on this node's normal line, weight
        // M1^-1[line index][0 or p]
        auto lift = [&](int f) {
            const int axis = tensor_face_axis(DIM, f);
            const T w = sMi[(axis == 0 ? ix : axis == 1 ? iy : iz) * 2 + tensor_face_end(DIM, f)];
            const T* fl = sf + el * 6 * NF + f * NFP + tensor_face_node(DIM, P, f, ix, iy, iz);
#pragma unroll
            for (int c = 0; c < 6; ++c) rhs[c] += w * fl[c * NF];
        };
        lift(0);
        lift(1);
        lift(2);
        lift(3);
        if constexpr (DIM == 3) {
            lift(4);
            lift(5);
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const size_t o = c * N + own0;
            if constexpr (MODE == kModeMult) {
                a.out[o] = rhs[c];
            } else if constexpr (is_lserk(MODE)) {
                T r = a.dt * rhs[c];
                if constexpr (MODE != kModeLserkFirst) r = a.ca * rv[c] + r;
                const T qn = q[c] + a.cb * r;
                if constexpr (MODE != kModeLserkLast) a.res[o] = r;
                a.out[o] = qn;
                bad = bad || unstable_entry(qn);
            } else if constexpr (MODE == kModeRk1) {
                a.out[o] = q[c] + a.ca * rhs[c];
                a.res[o] = q[c] + a.cb * rhs[c];
            } else if constexpr (MODE == kModeRk2 || MODE == kModeRk3) {
                a.out[o] = xv[c] + a.ca * rhs[c];
                a.res[o] = rv[c] + a.cb * rhs[c];
            } else {
                const T qn = rv[c] + a.ca * rhs[c];
                a.out[o] = qn;
                bad = bad || unstable_entry(qn);
            }
        }
    }
    if constexpr (is_lserk(MODE) || MODE == kModeRk4) report_unstable(a.unstable, bad);
}

template <typename T, int P, int DIM, int MODE, int kThreads>
hipError_t tensor_threads(const StageArgs<T>& a, int blocks, hipStream_t s)
{
    hipLaunchKernelGGL((tensor_stage<T, P, DIM, MODE, kThreads>), dim3((unsigned)((blocks + 7) / 8 * 8)),
                       dim3(kThreads), 0, s, a);
    return hipGetLastError();
}

// Four waves, enough for a node per thread, or six where those form the
// block's fluxes in one round fewer (hexahedra of orders 1, 3 and 4,
// quadrilaterals of order 2) and the mesh is small: up to two blocks per CU
// the round's latency counts (order 3 FP32, 1,331 hexahedra: 5.0 us with
// four, 4.6 with six, the operator alone; order 4, 729: 5.7 and 5.2), beyond that
// the idle waves of the products do (order 4, 10,648: 26.7 and 31.1).  Order
// 1 in FP64 needs 58 KB of LDS, two blocks per CU, and takes six waves up to
// one block per CU (10,648: 7.6 with four, 8.3 with six).  On order-2
// quadrilaterals a third of the second round's threads have work and one round
// stays ahead at every size (148,000, FP64: 38.2 with four, 35.9 with six).
template <typename T, int P, int DIM, int MODE>
hipError_t tensor_go(const StageArgs<T>& a, int cus, hipStream_t s)
{
    constexpr int EB = Tensor<P, DIM>::EB, F = EB * Tensor<P, DIM>::NF;
    constexpr bool kSaves = (F + 383) / 384 < (F + 255) / 256;
    const int blocks = (a.K + EB - 1) / EB;
    if constexpr (kSaves && DIM == 2) {
        return tensor_threads<T, P, DIM, MODE, 384>(a, blocks, s);
    } else {
        if constexpr (kSaves)
            if (blocks <= (P == 1 && sizeof(T) == 8 ? 1 : 2) * cus)
                return tensor_threads<T, P, DIM, MODE, 384>(a, blocks, s);
        return tensor_threads<T, P, DIM, MODE, 256>(a, blocks, s);
    }
}

template <typename T, int P, int DIM>
hipError_t tensor_launch(const StageArgs<T>& a, int mode, int cus, hipStream_t s)
{
    switch (lserk_mode(a, mode)) {
        case kModeMult: return tensor_go<T, P, DIM, kModeMult>(a, cus, s);
        case kModeLserk: return tensor_go<T, P, DIM, kModeLserk>(a, cus, s);
        case kModeLserkFirst: return tensor_go<T, P, DIM, kModeLserkFirst>(a, cus, s);
        case kModeLserkLast: return tensor_go<T, P, DIM, kModeLserkLast>(a, cus, s);
        case kModeRk1: return tensor_go<T, P, DIM, kModeRk1>(a, cus, s);
        case kModeRk2: return tensor_go<T, P, DIM, kModeRk2>(a, cus, s);
        case kModeRk3: return tensor_go<T, P, DIM, kModeRk3>(a, cus, s);
        case kModeRk4: return tensor_go<T, P, DIM, kModeRk4>(a, cus, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

template <typename T>
hipError_t launch_tensor_stage(int order, int dim, const StageArgs<T>& a, int mode, int cus, hipStream_t s)
{
    if (a.K <= 0) return hipErrorInvalidValue;
    switch (10 * dim + order) {
        case 21: return tensor_launch<T, 1, 2>(a, mode, cus, s);
        case 22: return tensor_launch<T, 2, 2>(a, mode, cus, s);
        case 23: return tensor_launch<T, 3, 2>(a, mode, cus, s);
        case 24: return tensor_launch<T, 4, 2>(a, mode, cus, s);
        case 25: return tensor_launch<T, 5, 2>(a, mode, cus, s);
        case 31: return tensor_launch<T, 1, 3>(a, mode, cus, s);
        case 32: return tensor_launch<T, 2, 3>(a, mode, cus, s);
        case 33: return tensor_launch<T, 3, 3>(a, mode, cus, s);
        case 34: return tensor_launch<T, 4, 3>(a, mode, cus, s);
        case 35: return tensor_launch<T, 5, 3>(a, mode, cus, s);
        default: return hipErrorInvalidValue;
    }
}

template hipError_t launch_tensor_stage<float>(int, int, const StageArgs<float>&, int, int, hipStream_t);
template hipError_t launch_tensor_stage<double>(int, int, const StageArgs<double>&, int, int, hipStream_t);

}  // namespace dgtd
