// Fused ADER step of the induction solver without the FV update: the stage
// sequence of src/induction_ader.hpp:343-359 (copy_ader, p+1 x Solve_E with
// p predictor updates, then update_B_solution) in p+2 launches, bit-exact
// with the stage kernels.
//
// What crosses HBM between launches is the raw edge field E of each element
// (compute_E's first variable, src/induction.cpp:139-208, before any face
// solve), FP64, for all time slices. A sweep launch works on a tile of
// consecutive elements (along x), all slices at once:
//   A. every edge point's face-solved value goes from HBM to LDS: upwinded
//      along the first face axis and then the second, exactly as the in-place
//      E_riemann_solver calls do (src/induction.cpp:509-560,
//      src/induction_ader.hpp:437-448). The upwind velocity is uniform, so the
//      solved value is one element's raw value (or, along an axis of zero
//      velocity, the mean of two) and the face solve is a choice of address;
//      boundary ghosts are resolved by index (periodic wrap, gradfree mirror)
//      as the SD trace fill makes them;
//   B. dB/dt at every face-B point (the derivative sums of
//      src/induction.cpp:331-356), kept in registers for all slices;
// then either the corrector into B (last launch, update_B_solution) or the
// predictor slices in LDS (update_B_prediction) and their raw E, written for
// the next launch.
// The zero-order guess makes every slice equal, so the first launch only
// computes the raw E of B, once per point, and the first sweep reads that one
// slice.
//
// The same kernels with R = float are the mixed-precision form: raw E, the
// face solves, the sp->fp interpolations and the predictor slices in FP32
// (with dfp_to_sp/h and invader*w*dt premultiplied), while the corrector forms
// dB/dt in FP64 from the FP32 edge values and accumulates B in FP64. Since
// every face-B update is a discrete curl of one set of edge values, div B
// stays at FP64 round-off.
//
// Only the upwind velocities of the face solves matter: they are the uniform
// advection velocity of the run (compute_E stores it per point, the face
// solve takes max(v_L, v_R) = v), and the other variables the stage path
// carries never reach B.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include "ctx.hpp"
#include "physics.hpp"

// Element tiles of the induction sweep in XCD-contiguous order (0: launch order).
#ifndef SPDK_ISWEEP_XCD
#define SPDK_ISWEEP_XCD 1
#endif

using namespace spdk;

namespace {

// Point counts of one configuration: N solution points per active axis; D = 3,
// or D = 2 with z inactive (one point along z).
template <int N, int D>
struct IG {
    static constexpr int M = N + 1;
    __host__ __device__ static constexpr int sp(int a) { return a < D ? N : 1; }
    __host__ __device__ static constexpr int fp(int a) { return a < D ? M : 1; }
    // face-B component d: flux points along d, solution points elsewhere
    __host__ __device__ static constexpr int bcnt(int d, int a) { return a == d ? fp(a) : sp(a); }
    // edge-E component e: solution points along e, flux points elsewhere
    __host__ __device__ static constexpr int ecnt(int e, int a) { return a == e ? sp(a) : fp(a); }
    __host__ __device__ static constexpr int bpts(int d) { return bcnt(d, 0) * bcnt(d, 1) * bcnt(d, 2); }
    __host__ __device__ static constexpr int epts(int e) { return ecnt(e, 0) * ecnt(e, 1) * ecnt(e, 2); }
    static constexpr int BP = bpts(0) + bpts(1) + bpts(2);
    static constexpr int EP = epts(0) + epts(1) + epts(2);
    __host__ __device__ static constexpr int boff(int d) { return d == 0 ? 0 : (d == 1 ? bpts(0) : bpts(0) + bpts(1)); }
    __host__ __device__ static constexpr int eoff(int e) { return e == 0 ? 0 : (e == 1 ? epts(0) : epts(0) + epts(1)); }
};

// A workgroup's tile: as many whole elements as its threads cover with one
// edge point of a component per thread, so that phases A and C run without a
// loop over points and phase B keeps one face-B point per component and
// thread (256 threads: 10 elements of 2-D p=3, 250 threads busy). The 100 edge
// points of 3-D p=3 fit 3 times into 320 threads and twice, 200 busy, into 256;
// a step with 320 and with 256, us: FP64 10 x 11 x 12 elements 65 and 70,
// 20^3 204 and 200, 56^3 4589 and 4338; mixed 14 x 15 x 16 71 and 74,
// 40 x 37 x 43 1096 and 992. So 320 is the better for meshes below some 20^3.
template <int N, int D, int T, class R>
struct Tile {
    using G = IG<N, D>;
    static constexpr int EMAX = G::epts(0) > G::epts(2) ? G::epts(0) : G::epts(2);
    static constexpr int THREADS = D == 3 && N == 4 ? 320 : 256;
    static constexpr int EPB = THREADS / EMAX;
    static_assert(EPB >= 1 && G::bpts(0) <= EMAX && G::bpts(2) <= EMAX, "one point per thread");
};

struct IArgs {
    void* Eout;           // raw E written by this launch (T, 3 components, elements, points)
    const void* Ein;      // raw E of the state this launch reads (element type R)
    double* B[3];         // face B, ghost-inclusive layout (1, 1, Nz, Ny, Nx, pts)
    const double* S2F;    // sp_to_fp (M x N)
    const double* Dm;     // dfp_to_sp (N x M)
    const double* inv;    // invader (T x T)
    const double* w;      // time weights (T)
    double vel[3];        // advection velocity
    double h[3];          // element widths
    double dt;
    int n[3];             // active elements per axis (1 on an inactive axis)
    int G[3];             // ghost-inclusive element counts
    int g[3];             // ghost elements per side (1 on active axes)
    int periodic[3];      // 1: periodic wrap, 0: gradfree mirror
    int nel;              // active elements
    int tin;              // slices present in Ein (1: every slice is slice 0)
    ConstDiv dh[3];       // division by h
};

// Raw-E slab of component e (all slices): T x nel x epts(e), components
// back to back.
template <int N, int D, int T>
__device__ __forceinline__ size_t eslab(int e, int nel) {
    using G = IG<N, D>;
    size_t o = 0;
    for (int c = 0; c < e; c++) o += (size_t)T * nel * G::epts(c);
    return o;
}

__device__ __forceinline__ void split_pt(int p, int nx, int ny, int pt[3]) {
    pt[0] = p % nx;
    p /= nx;
    pt[1] = p % ny;
    pt[2] = p / ny;
}

// Raw E (compute_E's first variable) of component e at point pt from B
// given by an accessor bget(d, point[3]): v1*b2 - v2*b1 with b1 = B_{e+1}
// interpolated sp->fp along e+2 and b2 = B_{e+2} along e+1 (an inactive axis
// takes the value as is).
template <int N, int D, class R, class BGet>
__device__ __forceinline__ R edge_e(int e, const int pt[3], const R* S2F, const R vel[3], BGet bget) {
    const int a1 = e == 2 ? 0 : e + 1, a2 = a1 == 2 ? 0 : a1 + 1;
    R b1 = 0, b2 = 0;
    int q[3] = {pt[0], pt[1], pt[2]};
    if (a2 < D) {
        for (int l = 0; l < N; l++) {
            q[a2] = l;
            b1 += bget(a1, q) * S2F[pt[a2] * N + l];
        }
        q[a2] = pt[a2];
    } else {
        b1 = bget(a1, q);
    }
    if (a1 < D) {
        for (int l = 0; l < N; l++) {
            q[a1] = l;
            b2 += bget(a2, q) * S2F[pt[a1] * N + l];
        }
    } else {
        b2 = bget(a2, q);
    }
    return vel[a1] * b2 - vel[a2] * b1;
}

// Face-solved E of component e (src/induction.cpp:509-560) at point pt of an
// element, for the slices: raw(off) reads raw values at an offset from the
// element's own point. lo[c] and hi[c] are the offsets of the points that
// share a lower / upper face point along c: the neighbour's opposite face
// point, or 0 where the ghost mirrors the element itself (gradfree).
// face(c) = -1 / +1 on a lower / upper face along c, else 0. dir[c] is the
// sign of the velocity along c; AVG: some dir is 0, where the solve takes the
// mean of both sides.
template <int e, int D, bool AVG, class V, class Raw>
__device__ __forceinline__ V edge_solved(const long lo[3], const long hi[3], const int dir[3], const int face[3],
                                         Raw raw) {
    constexpr int c1 = e == 0 ? 1 : 0, c2 = e == 2 ? 1 : 2;  // face axes, x before y before z
    auto shift = [&](int c) -> long {
        return c >= D ? 0 : (face[c] < 0 && dir[c] > 0 ? lo[c] : (face[c] > 0 && dir[c] < 0 ? hi[c] : 0));
    };
    if (!AVG) return raw(shift(c1) + shift(c2));
    auto first = [&](long base) -> V {
        if (c1 >= D || face[c1] == 0 || dir[c1] != 0) return raw(base + shift(c1));
        return mean(raw(base + (face[c1] < 0 ? lo[c1] : 0)), raw(base + (face[c1] < 0 ? 0 : hi[c1])));
    };
    if (c2 >= D || face[c2] == 0 || dir[c2] != 0) return first(shift(c2));
    return mean(first(face[c2] < 0 ? lo[c2] : 0), first(face[c2] < 0 ? 0 : hi[c2]));
}

// One point's value in every slice
template <class R, int T>
struct Slices {
    R v[T];
};
template <class R, int T>
__device__ __forceinline__ Slices<R, T> mean(const Slices<R, T>& l, const Slices<R, T>& r) {
    Slices<R, T> m;
#pragma unroll
    for (int t = 0; t < T; t++) m.v[t] = R(0.5) * (l.v[t] + r.v[t]);
    return m;
}

template <class F>
__device__ __forceinline__ void for_each_component(F f) {
    f(std::integral_constant<int, 0>{});
    f(std::integral_constant<int, 1>{});
    f(std::integral_constant<int, 2>{});
}

// Linear index of active element lin in the ghost-inclusive arrays
__device__ __forceinline__ size_t ghosted(const IArgs& a, int lin) {
    return ((size_t)(lin / (a.n[0] * a.n[1]) + a.g[2]) * a.G[1] + ((lin / a.n[0]) % a.n[1] + a.g[1])) * a.G[0] +
           (lin % a.n[0] + a.g[0]);
}

// Zero-order guess: the raw E of B, slice 0. The sweep's tile with B read once
// into LDS (reading each of the up to 8 B values of an edge point through the
// caches, over all components in one index, took 0.69 ms at 1024^2 p=3).
template <int N, int D, int T, class R>
__global__ void __launch_bounds__((Tile<N, D, T, R>::THREADS)) k_istart(IArgs a) {
    using G = IG<N, D>;
    using TL = Tile<N, D, T, R>;
    constexpr int EPB = TL::EPB, M = G::M;
    __shared__ R sB[EPB * G::BP];
    __shared__ R sS2F[M * N];
    const int e0 = blockIdx.x * EPB, tid = threadIdx.x, ne = min(EPB, a.nel - e0);
    for (int i = tid; i < M * N; i += TL::THREADS) sS2F[i] = (R)a.S2F[i];
    for_each_component([&](auto comp) {
        constexpr int d = comp.value, BPT = G::bpts(d);
        if (tid >= ne * BPT) return;
        const int q = tid / BPT, p = tid % BPT;
        sB[q * G::BP + G::boff(d) + p] = (R)a.B[d][ghosted(a, e0 + q) * BPT + p];
    });
    __syncthreads();
    const R vel[3] = {(R)a.vel[0], (R)a.vel[1], (R)a.vel[2]};
    for_each_component([&](auto comp) {
        constexpr int e = comp.value, EPT = G::epts(e);
        if (tid >= ne * EPT) return;
        const int q = tid / EPT, p = tid % EPT;
        int pt[3];
        split_pt(p, G::ecnt(e, 0), G::ecnt(e, 1), pt);
        const R* Bs = sB + q * G::BP;
        auto bget = [&](int d, const int r3[3]) -> R {
            return Bs[G::boff(d) + (r3[2] * G::bcnt(d, 1) + r3[1]) * G::bcnt(d, 0) + r3[0]];
        };
        ((R*)a.Eout)[eslab<N, D, T>(e, a.nel) + (size_t)(e0 + q) * EPT + p] = edge_e<N, D, R>(e, pt, sS2F, vel, bget);
    });
}

// One Picard sweep (CORR = false: predictor slices and their raw E; CORR =
// true: the corrector into B). The sweep moves each raw-E value of the tile
// once in and once out (2-D p=3: 4.6 KB per element, 1.1 ms at 1024^2 at the
// rate of a large copy); a thread owns one point of each component in every
// phase, with the slices unrolled, so that T loads are in flight per point,
// all index arithmetic is by compile-time constants and shared by the slices,
// and the sweep needs three barriers. Measured (1024^2 p=3 step): staging the
// raw E and solving faces LDS to LDS, with points in a runtime order, took
// 5.8 ms per sweep; this form 1.30 ms (3-D mixed 40 x 37 x 43: 1.04 -> 0.29 ms).
template <int N, int D, int T, bool CORR, class R>
__global__ void __launch_bounds__((Tile<N, D, T, R>::THREADS)) k_isweep(IArgs a) {
    using G = IG<N, D>;
    using TL = Tile<N, D, T, R>;
    constexpr bool PLAIN = std::is_same<R, double>::value;
    using Acc = typename std::conditional<PLAIN || CORR, double, float>::type;  // dB/dt
    constexpr int EPB = TL::EPB, M = G::M, TH = TL::THREADS;
    static_assert(G::BP <= G::EP, "the predictor slices fit in the edge buffer");
    __shared__ R sE[EPB * T * G::EP];  // face-solved E (element, slice, point), then the predictor slices
    __shared__ R sS2F[M * N];
    __shared__ double sDm[N * M], sInv[T * T], sW[T];
    __shared__ int sLow[TH / 64];
    __shared__ Acc sDmH[PLAIN ? 1 : D][PLAIN ? 1 : N * M];  // dfp_to_sp / h_axis
    __shared__ float sP[PLAIN ? 1 : T * T];                  // invader * w * dt
    // workgroups go to the 8 XCDs in turn; XCD x takes the x-th contiguous
    // eighth of the element tiles, so a tile's y (and z) neighbours, whose
    // face traces it reads, were mostly written through the same L2. The grid
    // is a multiple of 8; tiles past the end exit (uniform per block).
    const int blk = SPDK_ISWEEP_XCD ? (int)((blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8) : (int)blockIdx.x;
    const int e0 = blk * EPB;
    if (e0 >= a.nel) return;
    const int tid = threadIdx.x, ne = min(EPB, a.nel - e0);
    for (int i = tid; i < N * M; i += TH) {
        sDm[i] = a.Dm[i];
        sS2F[i] = (R)a.S2F[i];
        if (!PLAIN)
            for (int c = 0; c < D; c++) sDmH[c][i] = (Acc)(a.Dm[i] / a.h[c]);
    }
    if (tid < T * T) {
        sInv[tid] = a.inv[tid];
        if (!PLAIN) sP[tid] = (float)(a.inv[tid] * a.w[tid % T] * a.dt);
    }
    if (tid < T) sW[tid] = a.w[tid];
    const int dir[3] = {a.vel[0] == 0 ? 0 : (a.vel[0] > 0 ? 1 : -1), a.vel[1] == 0 ? 0 : (a.vel[1] > 0 ? 1 : -1),
                        a.vel[2] == 0 ? 0 : (a.vel[2] > 0 ? 1 : -1)};
    bool any_mean = false;
#pragma unroll
    for (int c = 0; c < D; c++) any_mean = any_mean || dir[c] == 0;

    // A. face-solved E of every slice
    int low = 0;  // smallest binary exponent of a nonzero value
    for_each_component([&](auto comp) {
        constexpr int e = comp.value, EPT = G::epts(e);
        if (tid >= ne * EPT) return;
        const int q = tid / EPT, p = tid % EPT, lin = e0 + q;
        int pt[3];
        split_pt(p, G::ecnt(e, 0), G::ecnt(e, 1), pt);
        const int el[3] = {lin % a.n[0], (lin / a.n[0]) % a.n[1], lin / (a.n[0] * a.n[1])};
        const int es[3] = {1, a.n[0], a.n[0] * a.n[1]};
        constexpr int ps[3] = {1, G::ecnt(e, 0), G::ecnt(e, 0) * G::ecnt(e, 1)};
        long lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
        int face[3] = {0, 0, 0};
#pragma unroll
        for (int c = 0; c < D; c++) {
            if (c == e) continue;
            face[c] = pt[c] == 0 ? -1 : (pt[c] == M - 1 ? 1 : 0);
            const bool first = el[c] == 0, last = el[c] == a.n[c] - 1;
            const long across = (long)(M - 1) * ps[c];
            lo[c] = first && !a.periodic[c] ? 0 : (long)(first ? a.n[c] - 1 : -1) * es[c] * EPT + across;
            hi[c] = last && !a.periodic[c] ? 0 : (long)(last ? 1 - a.n[c] : 1) * es[c] * EPT - across;
        }
        const size_t ss = (size_t)a.nel * EPT;
        const R* own = (const R*)a.Ein + eslab<N, D, T>(e, a.nel) + (size_t)lin * EPT + p;
        const int tin = a.tin;
        auto raw = [&](long off) {
            Slices<R, T> r;
#pragma unroll
            for (int t = 0; t < T; t++) r.v[t] = t < tin ? own[off + (long)(t * ss)] : r.v[0];
            return r;
        };
        const Slices<R, T> v = any_mean ? edge_solved<e, D, true, Slices<R, T>>(lo, hi, dir, face, raw)
                                        : edge_solved<e, D, false, Slices<R, T>>(lo, hi, dir, face, raw);
#pragma unroll
        for (int t = 0; t < T; t++)
            if (t < tin) {
                sE[(q * T + t) * G::EP + G::eoff(e) + p] = v.v[t];
                if (PLAIN) low = min(low, __builtin_amdgcn_frexp_exp((double)v.v[t]));
            }
    });
    // a zero sum may hold inexact quotients (div_small) only with such an edge value: matrix entries are zero or at
    // least 2^-200 (step())
    if (PLAIN) sLow[tid / 64] = __ballot(low <= -700) != 0;
    __syncthreads();

    const bool small = PLAIN && (sLow[0] | sLow[1] | sLow[2] | sLow[3] | sLow[TH / 64 - 1]);

    // B. dB/dt of every slice at the thread's face-B points
    Acc dBdt[3][T];
    for_each_component([&](auto comp) {
        constexpr int d = comp.value, BPT = G::bpts(d);
        constexpr int a1 = (d + 1) % 3, a2 = (d + 2) % 3;
#pragma unroll
        for (int t = 0; t < T; t++) dBdt[d][t] = 0;
        if (tid >= ne * BPT) return;
        const int q = tid / BPT, p = tid % BPT;
        int pt[3];
        split_pt(p, G::bcnt(d, 0), G::bcnt(d, 1), pt);
        // E1 = E_{d+1} differentiated along d+2, E2 = E_{d+2} along d+1
        constexpr int s1[3] = {1, G::ecnt(a1, 0), G::ecnt(a1, 0) * G::ecnt(a1, 1)};
        constexpr int s2[3] = {1, G::ecnt(a2, 0), G::ecnt(a2, 0) * G::ecnt(a2, 1)};
        const R* E1 = sE + q * T * G::EP + G::eoff(a1) + (pt[0] * s1[0] + pt[1] * s1[1] + pt[2] * s1[2] - pt[a2] * s1[a2]);
        const R* E2 = sE + q * T * G::EP + G::eoff(a2) + (pt[0] * s2[0] + pt[1] * s2[1] + pt[2] * s2[2] - pt[a1] * s2[a1]);
        Acc D1[M], D2[M];
#pragma unroll
        for (int l = 0; l < M; l++) {
            D1[l] = a2 < D ? (PLAIN ? (Acc)sDm[pt[a2] * M + l] : sDmH[PLAIN || a2 >= D ? 0 : a2][PLAIN ? 0 : pt[a2] * M + l]) : (Acc)0;
            D2[l] = a1 < D ? (PLAIN ? (Acc)sDm[pt[a1] * M + l] : sDmH[PLAIN || a1 >= D ? 0 : a1][PLAIN ? 0 : pt[a1] * M + l]) : (Acc)0;
        }
        const int tin = a.tin;
#pragma unroll
        for (int t = 0; t < T; t++) {
            if (t >= tin) {
                dBdt[d][t] = dBdt[d][0];
                continue;
            }
            Acc dB = 0;
#pragma unroll
            for (int l = 0; l < M; l++) {
                if (a2 < D) {
                    const Acc x = (Acc)E1[t * G::EP + l * s1[a2]] * D1[l];
                    dB += PLAIN ? (Acc)div_fast((double)x, a.dh[a2]) : x;
                }
                if (a1 < D) {
                    const Acc x = (Acc)E2[t * G::EP + l * s2[a1]] * D2[l];
                    dB -= PLAIN ? (Acc)div_fast((double)x, a.dh[a1]) : x;
                }
            }
            if (PLAIN && sum_recheck((double)dB) && (dB != 0 || small)) {
                dB = 0;
#pragma unroll 1
                for (int l = 0; l < M; l++) {
                    if (a2 < D) dB += (Acc)E1[t * G::EP + l * s1[a2]] * (Acc)sDm[pt[a2] * M + l] / (Acc)a.h[a2];
                    if (a1 < D) dB -= (Acc)E2[t * G::EP + l * s2[a1]] * (Acc)sDm[pt[a1] * M + l] / (Acc)a.h[a1];
                }
            }
            dBdt[d][t] = dB;
        }
    });

    // the corrector, or the predictor slices over the edge buffer
    if (!CORR) __syncthreads();
    for_each_component([&](auto comp) {
        constexpr int d = comp.value, BPT = G::bpts(d);
        if (tid >= ne * BPT) return;
        const int q = tid / BPT, p = tid % BPT;
        double* Bp = a.B[d] + ghosted(a, e0 + q) * BPT + p;
        const double B_old = *Bp;
        if (CORR) {
            double dB = 0;
#pragma unroll
            for (int t = 0; t < T; t++) dB += (double)dBdt[d][t] * sW[t] * a.dt;
            *Bp = B_old - dB;
            return;
        }
#pragma unroll
        for (int t = 0; t < T; t++) {
            Acc dB = 0;
            if (PLAIN) {
#pragma unroll
                for (int l = 0; l < T; l++) dB += dBdt[d][l] * sInv[t * T + l] * sW[l] * a.dt;
            } else {
#pragma unroll
                for (int l = 0; l < T; l++) dB += dBdt[d][l] * (Acc)sP[t * T + l];
            }
            sE[(q * T + t) * G::BP + G::boff(d) + p] = (R)B_old - (R)dB;
        }
    });
    if (CORR) return;
    __syncthreads();
    // C. the slices' raw E
    const R vel[3] = {(R)a.vel[0], (R)a.vel[1], (R)a.vel[2]};
    for_each_component([&](auto comp) {
        constexpr int e = comp.value, EPT = G::epts(e);
        if (tid >= ne * EPT) return;
        const int q = tid / EPT, p = tid % EPT;
        int pt[3];
        split_pt(p, G::ecnt(e, 0), G::ecnt(e, 1), pt);
        R* dst = (R*)a.Eout + eslab<N, D, T>(e, a.nel) + (size_t)(e0 + q) * EPT + p;
        const size_t ss = (size_t)a.nel * EPT;
#pragma unroll
        for (int t = 0; t < T; t++) {
            const R* Bs = sE + (q * T + t) * G::BP;
            auto bget = [&](int d, const int r3[3]) -> R {
                return Bs[G::boff(d) + (r3[2] * G::bcnt(d, 1) + r3[1]) * G::bcnt(d, 0) + r3[0]];
            };
            dst[t * ss] = edge_e<N, D, R>(e, pt, sS2F, vel, bget);
        }
    });
}

template <int N, int D, int T, class R>
size_t ws_bytes(int nel) {
    return 2 * (size_t)T * nel * IG<N, D>::EP * sizeof(R);
}

template <int N, int D, int T, class R>
int run_step(spdk_ctx* c, IArgs a, void* ws) {
    using TL = Tile<N, D, T, R>;
    const size_t half = (size_t)T * a.nel * IG<N, D>::EP;
    R* buf[2] = {(R*)ws, (R*)ws + half};
    const unsigned nstart = (unsigned)((a.nel + TL::EPB - 1) / TL::EPB);
    const unsigned nb = SPDK_ISWEEP_XCD ? (nstart + 7) / 8 * 8 : nstart;
    a.Eout = buf[0];
    a.Ein = nullptr;
    hipLaunchKernelGGL((k_istart<N, D, T, R>), dim3(nstart), dim3(TL::THREADS), 0, c->stream, a);
    SPDK_LAUNCH_CHECK("induction istart");
    for (int s = 0; s < T; s++) {
        a.Ein = buf[s & 1];
        a.Eout = buf[(s + 1) & 1];
        a.tin = s == 0 ? 1 : T;
        bool rec = c->timing && c->ev_used < spdk_ctx::kEvPool;
        if (rec) SPDK_CHECK(hipEventRecord(c->evs[c->ev_used][0], c->stream));
        if (s < T - 1) hipLaunchKernelGGL((k_isweep<N, D, T, false, R>), dim3(nb), dim3(TL::THREADS), 0, c->stream, a);
        else hipLaunchKernelGGL((k_isweep<N, D, T, true, R>), dim3(nb), dim3(TL::THREADS), 0, c->stream, a);
        SPDK_LAUNCH_CHECK("induction isweep");
        if (rec) SPDK_CHECK(hipEventRecord(c->evs[c->ev_used++][1], c->stream));
    }
    if (c->timing && c->ev_used > 0) {  // harvest the sweep timings (syncs the step)
        SPDK_CHECK(hipEventSynchronize(c->evs[c->ev_used - 1][1]));
        for (int i = 0; i < c->ev_used; i++) {
            float ms = 0;
            SPDK_CHECK(hipEventElapsedTime(&ms, c->evs[i][0], c->evs[i][1]));
            c->kernel_ms += ms;
            c->kernel_launches++;
        }
        c->ev_used = 0;
    }
    return SPDK_OK;
}

typedef int (*istep_fn)(spdk_ctx*, IArgs, void*);
typedef size_t (*iws_fn)(int);
struct IVariant {
    int n, dim, T;
    istep_fn step[2];  // FP64, mixed
    iws_fn ws[2];
};
#define SPDK_IVARIANT(Nn, D)                                                                  \
    {                                                                                         \
        Nn, D, Nn, {run_step<Nn, D, Nn, double>, run_step<Nn, D, Nn, float>},                 \
            {ws_bytes<Nn, D, Nn, double>, ws_bytes<Nn, D, Nn, float>}                        \
    }
const IVariant kIVariants[] = {SPDK_IVARIANT(2, 2), SPDK_IVARIANT(3, 2), SPDK_IVARIANT(4, 2), SPDK_IVARIANT(5, 2),
                               SPDK_IVARIANT(2, 3), SPDK_IVARIANT(3, 3), SPDK_IVARIANT(4, 3)};

const IVariant* find_ivariant(spdk_ctx* c) {
    if (!c->prm.active[0] || !c->prm.active[1]) return nullptr;
    int dim = c->prm.active[2] ? 3 : 2;
    if (c->prm.rk_order != 0) return nullptr;  // ADER only
    for (const IVariant& v : kIVariants)
        if (v.n == c->n && v.dim == dim && v.T == c->T) return &v;
    return nullptr;
}

bool bc_supported(spdk_ctx* c) {
    for (int d = 0; d < 3; d++)
        if (c->prm.active[d] && c->prm.bc[d] != SPDK_BC_PERIODIC && c->prm.bc[d] != SPDK_BC_GRADFREE) return false;
    return true;
}

size_t workspace_bytes(spdk_ctx* c, const int N[3], int mixed) {
    const IVariant* v = c ? find_ivariant(c) : nullptr;
    if (!v || !bc_supported(c)) {
        set_error("fused induction path: ADER, x-y or x-y-z active, p = 1..4 (1..3 in 3-D), periodic or gradfree "
                  "boundaries");
        return 0;
    }
    size_t nel = 1;
    for (int d = 0; d < 3; d++) nel *= (size_t)(c->prm.active[d] ? N[d] - 2 * c->ngh[d] : 1);
    if (nel == 0 || nel >= (1ull << 31)) { set_error("fused induction: element count"); return 0; }
    return v->ws[mixed]((int)nel);
}

int step(spdk_ctx* c, double* Bx, spdk_sd_shape sx, double* By, spdk_sd_shape sy, double* Bz, spdk_sd_shape sz, void* ws,
         double dt, int mixed) {
    if (!c || !Bx || !By || !Bz || !ws) { set_error("fused induction: null argument"); return SPDK_E_ARG; }
    const IVariant* v = find_ivariant(c);
    if (!v || !bc_supported(c)) { set_error("fused induction: unsupported configuration"); return SPDK_E_CONFIG; }
    const spdk_sd_shape* s[3] = {&sx, &sy, &sz};
    const int n = c->n, m = c->m;
    for (int d = 0; d < 3; d++) {
        const spdk_sd_shape& q = *s[d];
        int want[3];
        for (int a = 0; a < 3; a++) want[a] = c->prm.active[a] ? (a == d ? m : n) : 1;
        if (q.nt != 1 || q.nv != 1 || q.nx != want[0] || q.ny != want[1] || q.nz != want[2] || q.Nx != sx.Nx ||
            q.Ny != sx.Ny || q.Nz != sx.Nz) {
            set_error("fused induction: face-B shape");
            return SPDK_E_SHAPE;
        }
    }
    IArgs a;
    std::memset(&a, 0, sizeof(a));
    a.B[0] = Bx;
    a.B[1] = By;
    a.B[2] = Bz;
    a.S2F = c->mat[SPDK_M_SP_TO_FP];
    a.Dm = c->mat[SPDK_M_DFP_TO_SP];
    a.inv = c->mat[SPDK_M_INVADER];
    a.w = c->wt;
    a.dt = dt;
    const int Gd[3] = {sx.Nx, sx.Ny, sx.Nz};
    size_t nel = 1;
    for (int d = 0; d < 3; d++) {
        a.vel[d] = c->prm.vel[d];
        a.h[d] = c->prm.h[d];
        a.dh[d] = const_div(c->prm.h[d]);
        a.G[d] = Gd[d];
        a.g[d] = c->ngh[d];
        a.n[d] = Gd[d] - 2 * c->ngh[d];
        a.periodic[d] = c->prm.bc[d] == SPDK_BC_PERIODIC;
        if (a.n[d] < 1) { set_error("fused induction: axis needs ghost elements"); return SPDK_E_SHAPE; }
        nel *= (size_t)a.n[d];
    }
    // see k_isweep: with smaller matrix entries every quotient is formed by division
    for (double x : c->mat_host[SPDK_M_DFP_TO_SP])
        if (x != 0.0 && std::fabs(x) < 0x1p-200)
            for (int d = 0; d < 3; d++) a.dh[d].z = __builtin_nan("");
    if (nel >= (1ull << 31)) { set_error("fused induction: too many elements"); return SPDK_E_SHAPE; }
    a.nel = (int)nel;
    std::strncpy(c->kernel_name, "k_isweep", sizeof(c->kernel_name) - 1);
    return v->step[mixed](c, a, ws);
}

}  // namespace

extern "C" {

size_t spdk_induction_fused_workspace_bytes(spdk_ctx* c, const int N[3]) { return workspace_bytes(c, N, 0); }

int spdk_induction_step_fused(spdk_ctx* c, double* Bx, spdk_sd_shape sx, double* By, spdk_sd_shape sy, double* Bz,
                              spdk_sd_shape sz, void* ws, double dt) {
    return step(c, Bx, sx, By, sy, Bz, sz, ws, dt, 0);
}

size_t spdk_induction_mixed_workspace_bytes(spdk_ctx* c, const int N[3]) { return workspace_bytes(c, N, 1); }

int spdk_induction_step_mixed(spdk_ctx* c, double* Bx, spdk_sd_shape sx, double* By, spdk_sd_shape sy, double* Bz,
                              spdk_sd_shape sz, void* ws, double dt) {
    return step(c, Bx, sx, By, sy, Bz, sz, ws, dt, 1);
}

}  // extern "C"
