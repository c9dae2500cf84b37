// Fused element-tile path for the hydro SD step (plain FP64).
//
// One Picard sweep of ADER_step / one RK stage (src/hydro_ader.hpp:291-325)
// is one kernel over element tiles. A workgroup owns whole (element, time
// slice) units and keeps their flux-point fluxes in LDS; the only data that
// crosses elements are the face traces (the solution interpolated to the
// first and last flux point of every pencil), which each sweep writes for the
// next one. The Riemann flux of a face is evaluated by both elements that
// share it, from the same two traces, so both see identical bits.
//
// The arithmetic of every value (interpolation, Euler flux, LLF, the
// x/y/z-interleaved flux divergence, predictor and corrector sums, cv
// transform, dt) is performed in the same order as the stage kernels and the
// reference, so this path is bit-identical to the stage path.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include "ctx.hpp"
#include "physics.hpp"

using namespace spdk;

namespace {

constexpr int kMaxT = 8;

// Waves per SIMD the sweeps are compiled for (FACES: 3). At 4 (128 registers)
// the 3-D p=3 sweeps spill 2 to 10 registers and still gain over 3: predictor
// 5.58 -> 5.25 ms, corrector 4.61 -> 4.41 ms at 64^3 (4.6 and 4.5 since the
// matrices come by scalar loads), 2-D p=3 predictor
// 0.295 -> 0.239 ms at 256^2.
#ifndef SPDK_SWEEP_WAVES
#define SPDK_SWEEP_WAVES 4
#endif

template <int N, int DIM>
struct Tile {
    static constexpr int M = N + 1;                                // flux points per axis
    static constexpr int NT = DIM == 1 ? 1 : (DIM == 2 ? N : N * N);  // points per element face
    static constexpr int TPE = N * NT;                             // solution points per element
    static constexpr int EPB = TPE >= 256 ? 1 : 256 / TPE;         // units (elements, if of one slice) per workgroup
    static constexpr int BLOCK = 256;
    static constexpr int FSZ = M * NT;                             // flux points per axis per element
    static constexpr int LDS_U = NVP * TPE;                        // doubles: one state
    static constexpr int LDS_F = DIM * NVP * FSZ;                  // doubles: fluxes of every axis
    static_assert(EPB * TPE <= BLOCK && TPE <= BLOCK, "tile workgroups are 256 threads");
};

// What a sweep produces, and its units. PREDICT: the new predictor slices and
// their traces; CORRECT: the solution after the step or stage; FACES: the
// sub-cell face fluxes of the FV update; FLUXES: the flux-point fluxes.
enum { PREDICT = 0, CORRECT = 1, FACES = 2, FLUXES = 3 };

// S time slices of an element are units of one workgroup. S = T for the sweeps
// whose slices differ: the workgroup then holds fewer elements (one at 3-D
// p=3), every thread owns one point of one slice, and the slices meet once, in
// LDS, for the time contraction. That keeps one slice's divergence per thread
// in registers instead of T, makes the serial chain of a workgroup T times
// shorter and gives T times the workgroups (a 32^2 mesh, 1156 elements, has
// 289 for 256 CUs instead of 73). S = 1 where there is one slice: the first
// sweep from the zero-order guess and an SSP-RK stage; and for FACES, whose
// output rows run over elements, with a loop over the slices.
template <int N, int DIM, int T, int S, int MODE>
struct Unit {
    using G = Tile<N, DIM>;
    static constexpr int EL = G::EPB / S;  // elements per workgroup
    // doubles per unit: the fluxes, over which the exchanges go (two states; S = 1 PREDICT: all T new slices);
    // FACES: a scratch state ahead of them. + 4: the unit areas start 8 banks apart
    static constexpr int SCR = MODE == FACES ? G::LDS_U : 0;
    static constexpr int NEW = (S == 1 && MODE == PREDICT ? T : 2) * G::LDS_U;
    static constexpr int AREA = SCR + (G::LDS_F > NEW ? G::LDS_F : NEW) + 4;
    static constexpr int UNITS = EL * S;
    static constexpr int DOUBLES = UNITS * AREA + N * G::M;  // + dfp_to_sp
    static_assert(EL >= 1, "a workgroup holds every slice of an element");
};

struct SweepArgs {
    const double* U_sp;   // (1,6,E,TPE) solution (reference layout)
    double* U_sp_out;     // corrector output (same array)
    const double* U_in;   // (T,5,E,TPE) predictor state in (IN_ADER)
    double* U_out;        // (T,5,E,TPE) predictor state out (OUT_PRED)
    const double* tr_in[3];  // per axis (Tin,5,E,2,NT); Tin = 1 when traces are slice-independent
    double* tr_out[3];       // per axis (T,5,E,2,NT)
    double* U0;           // (5,E,TPE) RK step-start state
    double* W_cv;         // optional (1,6,E,TPE)
    double* F_x;          // optional (T,6,E,NT,M) x flux-point fluxes
    double* F_out[3];     // flux-only sweep: per axis (T,out_nv,E,FSZ) flux-point fluxes
    double* part;         // per-block dt minima
    const double* Dm;     // dfp_to_sp (N x M)
    const double* S2F;    // sp_to_fp  (M x N)
    const double* S2C;    // sp_to_cv  (N x N)
    const double* inv;    // invader (T x T)
    const double* w;      // time weights (T)
    int Ne[3];            // elements per axis incl. ghosts (x,y,z)
    int act[3], bc[3];
    int E;
    double h[3];
    ConstDiv dh[3];       // division by h
    double dt, gm, cfl, rk_a;
    int tin_slices;       // slices present in tr_in (1 or T)
    int in_nv;            // variables per slice of U_in
    int out_nv;           // variables per slice of F_out (slots past the physical ones get zero)
    double* Ffv[kMaxT][3];  // flux-only sweep: sub-cell face fluxes of slice t along axis d (FV layout)
    int fvn[3];           // FV cells per axis incl. ghost layers (an axis' face array has one more along it)
    int fgh[3];           // FV ghost layers per axis
    int in_ader;          // state from U_in (else U_sp broadcast to every slice)
    int rk_first;         // RK: write U0 = U_sp
    int want_dt;          // corrector: compute cv primitives and dt partials
    double g[3];          // constant gravity (hydro/g1..g3)
    int grav;             // any component nonzero
};

__device__ __forceinline__ int fidx(int d, int ll, int q, int N, int NT, int M) {
    // LDS index of flux point ll of pencil q along axis d (see header comment)
    if (d == 0) return q * M + ll;
    if (d == 1) return ((q / N) * M + ll) * N + (q % N);
    return ll * NT + q;
}

// Solution-point index of position ll along axis d of pencil q.
template <int N, int DIM>
__device__ __forceinline__ int spidx(int d, int ll, int q) {
    if (DIM == 1) return ll;
    if (DIM == 2) return d == 0 ? q * N + ll : ll * N + q;
    if (d == 0) return q * N + ll;                          // q = kk*N + jj
    if (d == 1) return ((q / N) * N + ll) * N + (q % N);   // q = kk*N + ii
    return ll * N * N + q;                                  // q = jj*N + ii
}

// Element block of a face-integral sweep workgroup: workgroups go to the 8
// XCDs in turn and XCD x takes the x-th contiguous eighth of the blocks, so
// the face rows that neighbouring blocks share (rows are not line-aligned)
// are written through one L2. The grid is padded to a multiple of 8.
__device__ __forceinline__ int face_sweep_block() {
    return (int)((blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8);
}

// face_integral of slice t for every active axis (src/transforms.cpp:378-481)
// from the element's flux-point fluxes in LDS (Fs, the fidx layout of each
// axis): each element writes the sub-cell faces of its cells' lower sides
// along d (the right ghost along d writes the domain's last face), so each
// FV face is written once, by the element whose copy face_integral reads.
// With both transverse axes active, the dim1 sweep u(f, o1, nn) = sum_ll
// F(f, ll, nn) S(o1, ll) goes through `scr` (the element's state area, free
// after the pencils) and the dim2 sum over nn of u S(o2, nn) is written;
// otherwise the single contraction of face_integral_ref. Sums in the
// reference's order, so the faces equal the stage kernels' bit for bit.
template <int N, int DIM, int AREA>
__device__ __forceinline__ void fv_faces(const SweepArgs& a, double* scr, double* Fs, int t, int s, bool live, int ei,
                                         int ej, int ek) {
    using G = Tile<N, DIM>;
    constexpr int M = G::M, NT = G::NT, TPE = G::TPE, FSZ = G::FSZ;
    // 3-D p=3: an element is a wave, so its two contractions need no block
    // barrier. An axis' faces then replace its fluxes (read for the last time by
    // its first contraction), and after one barrier per slice the block's four
    // elements (consecutive along x) write 16 consecutive faces per row, whole
    // 128-byte rows. With four barriers per axis instead, the waves waited 52%
    // of their time: 62 x 66 x 61 elements 5.92 -> 5.20 ms. At the other 3-D
    // degrees an element is not a wave (8 points: 8 to a wave; 27: across waves),
    // and two block barriers per axis stay.
    constexpr bool WAVE = TPE == 64 && DIM == 3;
    static_assert(!WAVE || TPE <= FSZ, "the faces fit over the fluxes");
    const double* S = a.S2C;
    const int ec[3] = {ei, ej, ek};
    const int o[3] = {s % N, DIM >= 2 ? (s / N) % N : 0, DIM == 3 ? s / (N * N) : 0};  // x fastest
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        bool own = live;
#pragma unroll
        for (int x = 0; x < DIM; x++) own = own && ec[x] >= 1 && ec[x] <= (x == d ? a.Ne[x] - 1 : a.Ne[x] - 2);
        const int f = o[d];
        const bool put = own && (ec[d] < a.Ne[d] - 1 || f == 0);
        const int dim1 = d == 0 ? 1 : (d == 1 ? 2 : 0), dim2 = dim1 == 0 ? 1 : (dim1 == 1 ? 2 : 0);
        const int nx = a.fvn[0] + (d == 0), ny = a.fvn[1] + (d == 1), nz = a.fvn[2] + (d == 2);
        const int I = o[0] + a.fgh[0] + (ei - 1) * N;
        const int J = DIM >= 2 ? o[1] + a.fgh[1] + (ej - 1) * N : 0;
        const int K = DIM == 3 ? o[2] + a.fgh[2] + (ek - 1) * N : 0;
        double* out = a.Ffv[t][d] + ((size_t)K * ny + J) * nx + I;
        const size_t vstride = (size_t)nz * ny * nx;
        if (DIM == 3) {
            {  // dim1 sweep: thread s -> (f, o1, nn)
                const int f1 = s / (N * N), o1 = (s / N) % N, nn = s % N;
                if (own)
#pragma unroll
                    for (int v = 0; v < NVP; v++) {
                        double u = 0;
#pragma unroll
                        for (int ll = 0; ll < N; ll++) {
                            const int q = d == 1 ? ll * N + nn : nn * N + ll;
                            u += Fs[(d * NVP + v) * FSZ + fidx(d, f1, q, N, NT, M)] * cload(S, o1 * N + ll);
                        }
                        scr[v * TPE + s] = u;
                    }
            }
            if (WAVE) elem_sync();
            else __syncthreads();
            if (own) {
                const int o1 = o[dim1], o2 = o[dim2];
#pragma unroll
                for (int v = 0; v < NVP; v++) {
                    double acc = 0;
#pragma unroll
                    for (int nn = 0; nn < N; nn++) acc += scr[v * TPE + (f * N + o1) * N + nn] * cload(S, o2 * N + nn);
                    if (WAVE) Fs[(d * NVP + v) * FSZ + s] = acc;
                    else if (put) out[(size_t)v * vstride] = acc;
                }
            }
            if (WAVE) elem_sync();
            else __syncthreads();
        } else if (put) {  // at most one transverse axis active: face_integral_ref
#pragma unroll
            for (int v = 0; v < NVP; v++) {
                double acc = 0;
                if (DIM == 1) {
                    acc += Fs[v * FSZ + fidx(0, f, 0, N, NT, M)];
                } else if (d == 0) {  // dim1 = y active, dim2 = z inactive
#pragma unroll
                    for (int ll = 0; ll < N; ll++) {
                        double x = Fs[v * FSZ + fidx(0, f, ll, N, NT, M)];
                        x *= cload(S, o[1] * N + ll);
                        acc += x;
                    }
                } else {  // d = 1: dim1 = z inactive, dim2 = x active
#pragma unroll
                    for (int nn = 0; nn < N; nn++) {
                        double x = Fs[(NVP + v) * FSZ + fidx(1, f, nn, N, NT, M)];
                        x *= cload(S, o[0] * N + nn);
                        acc += x;
                    }
                }
                out[(size_t)v * vstride] = acc;
            }
        }
    }
    if constexpr (WAVE) {
        static_assert(G::EPB == 4, "four elements per workgroup");
        __syncthreads();
        const int tid = threadIdx.x, xx = tid % 16, row = tid / 16;
        const int e2l = xx / N, ox = xx % N, oy = row % N, oz = row / N;
        const int e2 = face_sweep_block() * G::EPB + e2l;
        if (e2 >= a.E) return;
        const int ec2[3] = {e2 % a.Ne[0], (e2 / a.Ne[0]) % a.Ne[1], e2 / (a.Ne[0] * a.Ne[1])};
        const int o2[3] = {ox, oy, oz};
        const int I2 = ox + a.fgh[0] + (ec2[0] - 1) * N, J2 = oy + a.fgh[1] + (ec2[1] - 1) * N;
        const int K2 = oz + a.fgh[2] + (ec2[2] - 1) * N;
        const double* F2 = Fs + (long)(e2l - tid / TPE) * AREA + ox + N * (oy + N * oz);
#pragma unroll
        for (int d = 0; d < DIM; d++) {
            bool own2 = ec2[d] < a.Ne[d] - 1 || o2[d] == 0;
#pragma unroll
            for (int x = 0; x < DIM; x++)
                own2 = own2 && ec2[x] >= 1 && ec2[x] <= (x == d ? a.Ne[x] - 1 : a.Ne[x] - 2);
            if (!own2) continue;
            const int nx = a.fvn[0] + (d == 0), ny = a.fvn[1] + (d == 1), nz = a.fvn[2] + (d == 2);
            double* out = a.Ffv[t][d] + ((size_t)K2 * ny + J2) * nx + I2;
            const size_t vstride = (size_t)nz * ny * nx;
#pragma unroll
            for (int v = 0; v < NVP; v++) out[(size_t)v * vstride] = F2[(d * NVP + v) * FSZ];
        }
    }
}

// One pencil of axis D: state U (variables slabE apart) of element e, pencil q.
// Writes the fluxes at its M flux points to Fd (the fidx layout): interpolation
// to the flux points, Euler fluxes, and the LLF flux at the element faces
// (src/hydro.cpp:167-206, :368-418). ts: slice of the traces. The neighbours'
// face values are loaded first, with the ghost fill (src/boundary.cpp:48-113)
// as a choice of source: n0 is the value left of the lower face, or, in the
// left ghost, the fill that replaces its own upper face value; n1 likewise on
// the right. The outer face of a ghost has no neighbour: its own flux.
// lower_only: the upper face is not needed.
template <int N, int DIM, int D>
__device__ __forceinline__ void pencil(const SweepArgs& a, const double* U, size_t slabE, double* Fd, int q, size_t e,
                                       int ed, int ts, bool lower_only) {
    using G = Tile<N, DIM>;
    constexpr int M = G::M, NT = G::NT, TPE = G::TPE;
    const int Nd = a.Ne[D], type = a.bc[D];
    const bool per = type == SPDK_BC_PERIODIC;
    const size_t E = (size_t)a.E;
    const size_t stride = D == 0 ? 1 : (D == 1 ? (size_t)a.Ne[0] : (size_t)a.Ne[0] * a.Ne[1]);
    const size_t line = e - (size_t)ed * stride;  // element with ed = 0 on this line
    const bool lo = ed <= 1, hi = ed >= Nd - 2;
    const size_t el0 = line + (size_t)(lo ? (per ? Nd - 2 : 1) : ed - 1) * stride;
    const size_t el1 = line + (size_t)(hi ? (per ? 1 : Nd - 2) : ed + 1) * stride;
    const double* t0 = a.tr_in[D] + ((size_t)ts * NVP * E + el0) * 2 * NT + (lo && !per ? 0 : NT) + q;
    const double* t1 = a.tr_in[D] + ((size_t)ts * NVP * E + el1) * 2 * NT + (hi && !per ? NT : 0) + q;
    double n0[NVP], n1[NVP], p[NVP][N];
#pragma unroll
    for (int v = 0; v < NVP; v++) {
        n0[v] = t0[(size_t)v * E * 2 * NT];
        n1[v] = t1[(size_t)v * E * 2 * NT];
    }
    if (type == SPDK_BC_REFLECTIVE) {
        if (lo) n0[1 + D] = -1.0 * n0[1 + D];
        if (hi) n1[1 + D] = -1.0 * n1[1 + D];
    }
#pragma unroll
    for (int v = 0; v < NVP; v++)
#pragma unroll
        for (int l = 0; l < N; l++) p[v][l] = U[(size_t)v * slabE + e * TPE + spidx<N, DIM>(D, l, q)];
    auto at = [&](int f, double* u) {
#pragma unroll
        for (int v = 0; v < NVP; v++) {
            double x = 0;
#pragma unroll
            for (int l = 0; l < N; l++) x += p[v][l] * cload(a.S2F, f * N + l);
            u[v] = x;
        }
    };
    auto put = [&](int f, const double* fl) {
#pragma unroll
        for (int v = 0; v < NVP; v++) Fd[v * G::FSZ + fidx(D, f, q, N, NT, M)] = fl[v];
    };
#pragma unroll
    for (int f = 1; f < M - 1; f++) {
        double u[NVP], fl[NVP];
        at(f, u);
        state_flux<D>(u, fl, a.gm);
        put(f, fl);
    }
    const bool ghost0 = ed == 0, ghost1 = ed == Nd - 1;
    {
        double own[NVP], L[NVP], R[NVP], fl[NVP];
        at(0, own);
#pragma unroll
        for (int v = 0; v < NVP; v++) {
            L[v] = ghost0 ? own[v] : n0[v];
            R[v] = ghost1 ? n1[v] : own[v];
        }
        riemann_llf<D>(L, R, fl, a.gm, ghost0);
        put(0, fl);
    }
    if (lower_only) return;
    double own[NVP], L[NVP], R[NVP], fl[NVP];
    at(M - 1, own);
#pragma unroll
    for (int v = 0; v < NVP; v++) {
        L[v] = ghost0 ? n0[v] : own[v];
        R[v] = ghost1 ? own[v] : n1[v];
    }
    riemann_llf<D>(L, R, fl, a.gm, ghost1);
    put(M - 1, fl);
}

// Flux divergence of variable v at solution point s (src/transforms.cpp:301-307),
// whose sum `acc` of fast quotients is zero, small or NaN: formed again with
// divisions, unless it is a zero without inexact terms.
template <int N, int DIM>
__device__ __forceinline__ double divergence_recheck(const SweepArgs& a, const double* Fs, const double* sD, int v,
                                                     int ii, int jj, int kk, double acc) {
    using G = Tile<N, DIM>;
    constexpr int M = G::M, NT = G::NT;
    auto fx = [&](int l) { return Fs[v * G::FSZ + fidx(0, l, DIM == 3 ? kk * N + jj : jj, N, NT, M)]; };
    auto fy = [&](int l) { return Fs[(NVP + v) * G::FSZ + fidx(1, l, DIM == 3 ? kk * N + ii : ii, N, NT, M)]; };
    auto fz = [&](int l) { return Fs[(2 * NVP + v) * G::FSZ + fidx(2, l, jj * N + ii, N, NT, M)]; };
    bool redo = acc != 0.0;  // NaN: true
    if (!redo) {
        AnyBits any;
#pragma unroll
        for (int l = 0; l < M; l++) {
            any.add(fx(l));
            if (DIM >= 2) any.add(fy(l));
            if (DIM == 3) any.add(fz(l));
        }
#pragma unroll 1
        for (int l = 0; l < M && any.b; l++) {
            redo |= div_small(fx(l) * sD[ii * M + l]);
            if (DIM >= 2) redo |= div_small(fy(l) * sD[jj * M + l]);
            if (DIM == 3) redo |= div_small(fz(l) * sD[kk * M + l]);
        }
    }
    if (!redo) return acc;
    acc = 0;
#pragma unroll 1
    for (int l = 0; l < M; l++) {
        acc += fx(l) * sD[ii * M + l] / a.h[0];
        if (DIM >= 2) acc += fy(l) * sD[jj * M + l] / a.h[1];
        if (DIM == 3) acc += fz(l) * sD[kk * M + l] / a.h[2];
    }
    return acc;
}

// One sweep (see Unit). Three dependent phases, a barrier between each: the
// pencils' fluxes into LDS, the divergence at every point, and the output.
// Pencils are dealt to threads axis by axis over all units, so that a wave
// mostly works on one axis with all lanes (3-D p=3: 64 pencils per axis and
// workgroup; the fourth wave has none, and it is another wave in every
// workgroup and slice). What bounds it (3-D p=3, 64^3): FP64 issue, of which
// the divergence's divisions by h were 41% before they became three
// instructions each, and the latency of the phases. With the state read from
// memory by the pencils and one slice per thread the predictor needs 38.5 KB
// LDS and fits 4 workgroups per CU.
template <int N, int DIM, int T, int S, int MODE>
__global__ void __launch_bounds__(256, MODE == FACES ? 3 : SPDK_SWEEP_WAVES) k_sweep(SweepArgs a) {
    using G = Tile<N, DIM>;
    using X = Unit<N, DIM, T, S, MODE>;
    constexpr int M = G::M, NT = G::NT, TPE = G::TPE, EL = X::EL;
    extern __shared__ double lds[];
    double* const sD = lds + X::UNITS * X::AREA;
    const int tid = threadIdx.x;
    const int bx = MODE == FACES ? face_sweep_block() : (int)blockIdx.x;
    if (MODE == FACES && bx * EL >= a.E) return;  // padding of the XCD-ordered grid (uniform per block)
    // (element, slice) and solution point of this thread; the former is the
    // wave's where a slice fills it, and its addresses are then scalar
    const int unit = TPE == 64 ? __builtin_amdgcn_readfirstlane(tid / 64) : tid / TPE, s = tid % TPE;
    const int el = unit / S, ut = unit % S;
    const int e = bx * EL + el;
    const bool live = unit < X::UNITS && e < a.E;
    const size_t E = (size_t)a.E;
    const size_t slabE = E * TPE;  // one (t,v) plane of a state array
    double* const Fs = lds + (unit < X::UNITS ? unit : 0) * X::AREA + X::SCR;
    for (int i = tid; i < N * M; i += G::BLOCK) sD[i] = cload(a.Dm, i);

    int ei = 0, ej = 0, ek = 0;
    if (live) {
        ei = e % a.Ne[0];
        ej = (e / a.Ne[0]) % a.Ne[1];
        ek = e / (a.Ne[0] * a.Ne[1]);
    }
    const int ii = s % N, jj = DIM >= 2 ? (s / N) % N : 0, kk = DIM == 3 ? s / (N * N) : 0;

    constexpr int LOOP = MODE == FACES ? T : 1;  // slices one after the other
    double dudt[NVP] = {0, 0, 0, 0, 0};
#pragma unroll 1
    for (int tl = 0; tl < LOOP; tl++) {
        // ---- pencils
        for (int i = (tid + 64 * ((bx + tl) % 4)) % G::BLOCK; i < DIM * X::UNITS * NT; i += G::BLOCK) {
            const int d = i / (X::UNITS * NT), pu = i / NT % X::UNITS, q = i % NT;
            const int pe = bx * EL + pu / S, pt = MODE == FACES ? tl : pu % S;
            if (pe >= a.E) continue;
            const double* U = a.in_ader ? a.U_in + (size_t)pt * a.in_nv * slabE : a.U_sp;
            const int ts = a.tin_slices > 1 ? pt : 0;
            double* F = lds + pu * X::AREA + X::SCR;
            const int px = pe % a.Ne[0], py = (pe / a.Ne[0]) % a.Ne[1], pz = pe / (a.Ne[0] * a.Ne[1]);
            // the face integrals read faces 0..M-2 only: the upper face's
            // flux is formed when the flux-point array is written as well
            if (d == 0) pencil<N, DIM, 0>(a, U, slabE, F, q, pe, px, ts, MODE == FACES && !a.F_out[0]);
            if (DIM >= 2 && d == 1)
                pencil<N, DIM, 1>(a, U, slabE, F + NVP * G::FSZ, q, pe, py, ts, MODE == FACES && !a.F_out[1]);
            if (DIM == 3 && d == 2)
                pencil<N, DIM, 2>(a, U, slabE, F + 2 * NVP * G::FSZ, q, pe, pz, ts, MODE == FACES && !a.F_out[2]);
        }
        __syncthreads();
        if (MODE == FACES || MODE == FLUXES) {  // the stage flux-point layout (src/hydro_ader.hpp:278-289)
            const int t = MODE == FACES ? tl : ut;
            if (live) {
#pragma unroll
                for (int d = 0; d < DIM; d++)
                    for (int idx = s; a.F_out[d] && idx < G::FSZ; idx += TPE) {
                        double* o = a.F_out[d] + ((size_t)t * a.out_nv * E + e) * G::FSZ + idx;
#pragma unroll
                        for (int v = 0; v < NVP; v++) o[(size_t)v * E * G::FSZ] = Fs[(d * NVP + v) * G::FSZ + idx];
                        for (int v = NVP; v < a.out_nv; v++) o[(size_t)v * E * G::FSZ] = 0.0;
                    }
            }
            if (MODE == FACES) {  // last: its faces replace the fluxes
                fv_faces<N, DIM, X::AREA>(a, Fs - X::SCR, Fs, t, s, live, ei, ej, ek);
                __syncthreads();
            }
        }
    }
    if (MODE == FACES || MODE == FLUXES) return;

    // ---- flux divergence at the solution points (src/transforms.cpp:301-307)
    if (live) {
        const int qx = DIM == 3 ? kk * N + jj : jj;
        const int qy = DIM == 3 ? kk * N + ii : ii;
        const int qz = jj * N + ii;
        bool recheck = false;
#pragma unroll
        for (int v = 0; v < NVP; v++) {
            double acc = 0;
            AnyBits any;
            const double* Fx = Fs + v * G::FSZ;
            const double* Fy = Fs + (NVP + v) * G::FSZ;
            const double* Fz = Fs + (2 * NVP + v) * G::FSZ;
            auto flux = [&](double f) {
                if (v > DIM && v < 4) any.add(f);  // momentum along an inactive axis: zero in most flows
                return f;
            };
#pragma unroll
            for (int l = 0; l < M; l++) {
                acc += div_fast(flux(Fx[fidx(0, l, qx, N, NT, M)]) * sD[ii * M + l], a.dh[0]);
                if (DIM >= 2) acc += div_fast(flux(Fy[fidx(1, l, qy, N, NT, M)]) * sD[jj * M + l], a.dh[1]);
                if (DIM == 3) acc += div_fast(flux(Fz[fidx(2, l, qz, N, NT, M)]) * sD[kk * M + l], a.dh[2]);
            }
            dudt[v] = acc;
            if (v > DIM && v < 4) recheck = recheck || (sum_recheck(acc) && (any.b || acc != 0.0));
            else recheck = recheck || sum_recheck(acc);
        }
        if (recheck)
#pragma unroll
            for (int v = 0; v < NVP; v++)
                if (sum_recheck(dudt[v])) dudt[v] = divergence_recheck<N, DIM>(a, Fs, sD, v, ii, jj, kk, dudt[v]);
        if (a.grav && MODE == CORRECT) {
            // update_solution's gravity source (src/transforms.cpp:17-27,
            // :364-367) from the ADER slice: rho g and m . g
            const double* U = (a.in_ader ? a.U_in + (size_t)ut * a.in_nv * slabE : a.U_sp) + (size_t)e * TPE + s;
            const double rho = U[0], m1 = U[slabE], m2 = U[2 * slabE], m3 = U[3 * slabE];
            dudt[1] -= rho * a.g[0];
            dudt[2] -= rho * a.g[1];
            dudt[3] -= rho * a.g[2];
            dudt[4] -= m1 * a.g[0] + m2 * a.g[1] + m3 * a.g[2];
        }
        if (MODE == CORRECT && a.F_x) {  // x flux-point fluxes of the final sweep (outputs)
            for (int idx = s; idx < G::FSZ; idx += TPE) {
                size_t o = (((size_t)ut * NV) * E + e) * G::FSZ + idx;
#pragma unroll
                for (int v = 0; v < NVP; v++) a.F_x[o + (size_t)v * E * G::FSZ] = Fs[v * G::FSZ + idx];
                a.F_x[o + (size_t)NVP * E * G::FSZ] = 0.0;
            }
        }
    }
    double u_old[NVP];
#pragma unroll
    for (int v = 0; v < NVP; v++) u_old[v] = live ? a.U_sp[(size_t)v * slabE + (size_t)e * TPE + s] : 0.0;
    __syncthreads();  // the fluxes have been read

    // ---- the slices' divergences meet in the flux area of each element's units
    double* const mine = Fs;                    // this unit's divergence, then its exchange area
    const double* const own0 = Fs - ut * X::AREA;  // the element's unit of slice 0
    if (S > 1) {
        if (live)
#pragma unroll
            for (int v = 0; v < NVP; v++) mine[v * TPE + s] = dudt[v];
        __syncthreads();
    }
    auto rate = [&](int l, int v) -> double { return S > 1 ? own0[l * X::AREA + v * TPE + s] : dudt[v]; };

    if (MODE == PREDICT) {
        // ---- predictor (src/transforms.cpp:316-322): slices ut + k S of this thread
        constexpr int OWN = T / S;  // slices this thread forms
        constexpr int UO = S > 1 ? G::LDS_U : 0;  // new slices in LDS, behind the divergences
        auto slice_at = [&](int t) -> double* {   // area of new slice t of this element
            return S > 1 ? const_cast<double*>(own0) + t * X::AREA + UO : Fs + t * G::LDS_U;
        };
        if (!a.grav) {
#pragma unroll
            for (int k = 0; k < OWN; k++) {
                const int t = S > 1 ? ut : k;
                if (live)
#pragma unroll
                    for (int v = 0; v < NVP; v++) {
                        double du = 0;
#pragma unroll
                        for (int l = 0; l < T; l++) du += rate(l, v) * cload(a.inv, t * T + l) * cload(a.w, l) * a.dt;
                        const double un = u_old[v] - du;
                        a.U_out[((size_t)t * NVP + v) * slabE + (size_t)e * TPE + s] = un;
                        slice_at(t)[v * TPE + s] = un;
                    }
            }
        } else {
            // With gravity (src/transforms.cpp:17-27, :309-313) update_prediction
            // writes U_ader variable by variable and its source reads U_ader
            // back: the momenta's source takes the density just written, the
            // energy's the momenta just written. Each group goes through LDS.
#pragma unroll 1
            for (int grp = 0; grp < 3; grp++) {
                const int v0 = grp == 0 ? 0 : (grp == 1 ? 1 : 4), v1 = grp == 0 ? 1 : (grp == 1 ? 4 : 5);
                if (live)
#pragma unroll
                    for (int k = 0; k < OWN; k++) {
                        const int t = S > 1 ? ut : k;
#pragma unroll
                        for (int v = 0; v < NVP; v++) {
                            if (v < v0 || v >= v1) continue;
                            double du = 0;
#pragma unroll
                            for (int l = 0; l < T; l++) {
                                const double* n = slice_at(l) + s;
                                double r = rate(l, v);
                                if (v >= 1 && v <= 3) r -= n[0] * a.g[v - 1];
                                if (v == 4) r -= n[TPE] * a.g[0] + n[2 * TPE] * a.g[1] + n[3 * TPE] * a.g[2];
                                du += r * cload(a.inv, t * T + l) * cload(a.w, l) * a.dt;
                            }
                            const double un = u_old[v] - du;
                            a.U_out[((size_t)t * NVP + v) * slabE + (size_t)e * TPE + s] = un;
                            slice_at(t)[v * TPE + s] = un;
                        }
                    }
                __syncthreads();
            }
        }
        __syncthreads();
        // ---- traces of the new slices, axis by axis over (slice, element)
        for (int i = tid; i < DIM * T * EL * NT; i += G::BLOCK) {
            const int d = i / (T * EL * NT), t = i / (EL * NT) % T, pl = i / NT % EL, q = i % NT;
            const int pe = bx * EL + pl;
            if (pe >= a.E) continue;
            const double* un = S > 1 ? lds + (pl * S + t) * X::AREA + UO : lds + pl * X::AREA + t * G::LDS_U;
            const int l0 = d == 0 ? spidx<N, DIM>(0, 0, q) : (d == 1 ? spidx<N, DIM>(1, 0, q) : spidx<N, DIM>(2, 0, q));
            const int ls = d == 0 ? 1 : (d == 1 ? N : N * N);
            double* tr = d == 0 ? a.tr_out[0] : (d == 1 ? a.tr_out[1] : a.tr_out[2]);
#pragma unroll
            for (int v = 0; v < NVP; v++) {
                double p[N];
#pragma unroll
                for (int l = 0; l < N; l++) p[l] = un[v * TPE + l0 + l * ls];
                double x0 = 0, x1 = 0;
#pragma unroll
                for (int l = 0; l < N; l++) x0 += p[l] * cload(a.S2F, l);
#pragma unroll
                for (int l = 0; l < N; l++) x1 += p[l] * cload(a.S2F, (M - 1) * N + l);
                double* to = tr + (((size_t)t * NVP + v) * E + pe) * 2 * NT + q;
                to[0] = x0;
                to[NT] = x1;
            }
        }
        return;
    }

    // ---- corrector (src/transforms.cpp:354-372), optional SSP combine: the
    // element's slice-0 threads
    const bool lead = live && ut == 0;
    double un[NVP];
    if (lead) {
#pragma unroll
        for (int v = 0; v < NVP; v++) {
            double du = 0;
#pragma unroll
            for (int t = 0; t < T; t++) du += rate(t, v) * cload(a.w, t) * a.dt;
            un[v] = u_old[v] - du;
        }
        if (a.rk_a != 0.0) {  // combine_solution (src/transforms.cpp:252-261)
#pragma unroll
            for (int v = 0; v < NVP; v++) {
                double u0 = a.U0[(size_t)v * slabE + (size_t)e * TPE + s];
                un[v] = a.rk_a * u0 + (1.0 - a.rk_a) * un[v];
            }
        }
#pragma unroll
        for (int v = 0; v < NVP; v++) {
            if (a.rk_first) a.U0[(size_t)v * slabE + (size_t)e * TPE + s] = u_old[v];
            a.U_sp_out[(size_t)v * slabE + (size_t)e * TPE + s] = un[v];
        }
    }
    if (!a.want_dt) return;
    // ---- cv primitives: compute_primitives then sp->cv sweeps x, y, z, the
    // variables shared out over the element's units
    double* src = const_cast<double*>(own0) + G::LDS_U;  // clear of the divergences (slice 0's area)
    double* dst = const_cast<double*>(own0);
    if (lead) {
        double wv[NVP];
        prim(un, wv, a.gm);
#pragma unroll
        for (int v = 0; v < NVP; v++) src[v * TPE + s] = wv[v];
    }
    __syncthreads();
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        if (live) {
            const int id = d == 0 ? ii : (d == 1 ? jj : kk);
            for (int v = ut; v < NVP; v += S) {
                double x = 0;
#pragma unroll
                for (int l = 0; l < N; l++) {
                    int sl = d == 0 ? s - ii + l : (d == 1 ? s + (l - jj) * N : s + (l - kk) * N * N);
                    x += src[v * TPE + sl] * cload(a.S2C, id * N + l);
                }
                dst[v * TPE + s] = x;
            }
        }
        __syncthreads();
        double* tmp = src;
        src = dst;
        dst = tmp;
    }
    // src now holds W_cv of the element
    double r = __builtin_inf();
    if (lead) {
        double wc[NVP];
#pragma unroll
        for (int v = 0; v < NVP; v++) wc[v] = src[v * TPE + s];
        if (a.W_cv) {
#pragma unroll
            for (int v = 0; v < NVP; v++) a.W_cv[(size_t)v * slabE + (size_t)e * TPE + s] = wc[v];
            a.W_cv[(size_t)NVP * slabE + (size_t)e * TPE + s] = 0.0;
        }
        bool active = (!a.act[0] || (ei >= 1 && ei <= a.Ne[0] - 2)) && (!a.act[1] || (ej >= 1 && ej <= a.Ne[1] - 2)) &&
                      (!a.act[2] || (ek >= 1 && ek <= a.Ne[2] - 2));
        if (active) {  // src/hydro.cpp:226-256 (inviscid)
            double c_s = sound_speed(wc[0], wc[4], a.gm);
            double c_max = 0, dx_min = 1;
            if (a.act[0]) { c_max += (fabs(wc[1]) + c_s); dx_min = smin(dx_min, a.h[0]); }
            if (a.act[1]) { c_max += (fabs(wc[2]) + c_s); dx_min = smin(dx_min, a.h[1]); }
            if (a.act[2]) { c_max += (fabs(wc[3]) + c_s); dx_min = smin(dx_min, a.h[2]); }
            r = a.cfl * dx_min / c_max / N;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) r = nan_min(r, __shfl_xor(r, o));
    __syncthreads();
    if (tid % 64 == 0) lds[tid / 64] = r;
    __syncthreads();
    if (tid == 0) a.part[blockIdx.x] = nan_min(nan_min(lds[0], lds[1]), nan_min(lds[2], lds[3]));
}

// Face traces of slice blockIdx.y of U (in_nv variables per slice): of the
// solution U_sp (one slice), the input of a step's first sweep, or of given
// predictor slices.
template <int N, int DIM>
__global__ void __launch_bounds__(256) k_trace0(const double* __restrict__ U, int in_nv, double* tr0,
                                                               double* tr1, double* tr2, const double* __restrict__ S2F,
                                                               int Eint) {
    using G = Tile<N, DIM>;
    constexpr int M = G::M, NT = G::NT, TPE = G::TPE, EPB = G::EPB;
    __shared__ double us[EPB * NVP * TPE];
    const int tid = threadIdx.x, el = tid / TPE, s = tid % TPE;
    const int e = blockIdx.x * EPB + el;
    const bool live = el < EPB && e < Eint;
    const size_t E = (size_t)Eint, slabE = E * TPE, t = blockIdx.y;
    if (live)
#pragma unroll
        for (int v = 0; v < NVP; v++) us[(el * NVP + v) * TPE + s] = U[(t * in_nv + v) * slabE + (size_t)e * TPE + s];
    __syncthreads();
    for (int task = s; live && task < DIM * NT; task += TPE) {
        const int d = task / NT, q = task % NT;
        double* trd = d == 0 ? tr0 : (d == 1 ? tr1 : tr2);
#pragma unroll
        for (int v = 0; v < NVP; v++) {
            double x0 = 0, x1 = 0;
#pragma unroll
            for (int l = 0; l < N; l++) {
                double p = us[(el * NVP + v) * TPE + spidx<N, DIM>(d, l, q)];
                x0 += p * S2F[l];
            }
#pragma unroll
            for (int l = 0; l < N; l++) {
                double p = us[(el * NVP + v) * TPE + spidx<N, DIM>(d, l, q)];
                x1 += p * S2F[(M - 1) * N + l];
            }
            double* to = trd + (((t * NVP + v) * E + e) * 2) * NT + q;
            to[0] = x0;
            to[NT] = x1;
        }
    }
}

// Minimum of part[0, n) over the grid: out[blockIdx.x] per workgroup.
__global__ void __launch_bounds__(1024) k_partial_min(const double* part, int n, double* out) {
    __shared__ double red[16];
    double r = __builtin_inf();
    for (int i = blockIdx.x * 1024 + threadIdx.x; i < n; i += gridDim.x * 1024) r = nan_min(r, part[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) r = nan_min(r, __shfl_xor(r, o));
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = r;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++) r = nan_min(r, red[w]);
        out[blockIdx.x] = r;
    }
}

// ---------------------------------------------------------------------------
constexpr int kMinBlocks = 256;  // workgroups of the first of two dt reductions
struct Layout {
    size_t E = 0, tpe = 0, nt = 0, T = 0, dim = 0;
    size_t off_uader = 0, off_trA = 0, off_trB = 0, off_u0 = 0, off_part = 0, total = 0;
    size_t tr_axis = 0;  // doubles per axis per trace buffer
    unsigned blocks = 0;
};

template <int N, int DIM>
Layout layout_for(size_t E, int T) {
    using G = Tile<N, DIM>;
    Layout L;
    L.E = E;
    L.tpe = G::TPE;
    L.nt = G::NT;
    L.T = T;
    L.dim = DIM;
    L.blocks = (unsigned)((E + G::EPB / T - 1) / (G::EPB / T));  // of a sweep with every slice (T = 1: one)
    size_t st = (size_t)T * NVP * E * G::TPE;
    L.tr_axis = (size_t)T * NVP * E * 2 * G::NT;
    size_t o = 0;
    L.off_uader = o; o += st;
    L.off_trA = o; o += DIM * L.tr_axis;
    L.off_trB = o; o += DIM * L.tr_axis;
    L.off_u0 = o; o += (size_t)NVP * E * G::TPE;
    L.total = o;
    // the dt minima lie over the trace buffer that the last sweep (number
    // T - 1; even ones read buffer A) neither reads nor writes: at least 10 E
    // doubles, where at most E minima go, and 256 more above 16384 (kMinBlocks)
    L.off_part = T % 2 ? L.off_trB : L.off_trA;
    return L;
}

// The predictor slices (T, NVP, E, TPE) in the stage layout of U_ader (T, nv,
// E, TPE); slots past the physical variables are zero, as the stage
// predictor leaves them.
__global__ void k_export_ader(const double* __restrict__ Ua, double* __restrict__ out, int nv, size_t slabE,
                              size_t total) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t r = i % slabE, tv = i / slabE;
        const int v = (int)(tv % nv), t = (int)(tv / nv);
        out[i] = v < NVP ? Ua[((size_t)t * NVP + v) * slabE + r] : 0.0;
    }
}

// What a call produces instead of a whole step (all null: one step).
struct Extra {
    double* U_export = nullptr;  // the T-1 predictor sweeps from the zero-order guess, slices written here
    int nv_export = 0;
    double* F_out[3] = {nullptr, nullptr, nullptr};  // the predictor sweeps, then the flux evaluation of the
    int out_nv = 0;                                  // final slices written here (stage flux-point layout)
    const double* U_slices = nullptr;  // with F_out: the flux evaluation of these slices (stage layout), no
    int slices_nv = 0;                 // predictor; the workspace then holds only their traces
    double* const* Ffv = nullptr;      // the flux evaluation's sub-cell face fluxes, [t * 3 + d] (FV layout)
    int fvn[3] = {1, 1, 1}, fgh[3] = {0, 0, 0};
};

template <int N, int DIM>
size_t slice_trace_doubles(size_t E, int T) {
    return (size_t)DIM * T * NVP * E * 2 * Tile<N, DIM>::NT;
}

template <int N, int DIM, int T>
int run_step(spdk_ctx* c, double* U_sp, const int Ne[3], void* ws, double dt, double* W_cv, double* F_x,
             double* dt_next, const Extra* x) {
    using G = Tile<N, DIM>;
    size_t E = (size_t)Ne[0] * Ne[1] * Ne[2];
    Layout L = layout_for<N, DIM>(E, T);
    double* W = (double*)ws;
    double* trA[3] = {nullptr, nullptr, nullptr};
    double* trB[3] = {nullptr, nullptr, nullptr};
    for (int d = 0; d < DIM; d++) {
        trA[d] = W + L.off_trA + d * L.tr_axis;
        trB[d] = W + L.off_trB + d * L.tr_axis;
    }
    SweepArgs a;
    std::memset(&a, 0, sizeof(a));
    a.U_sp = U_sp;
    a.U_sp_out = U_sp;
    a.U0 = W + L.off_u0;
    a.part = W + L.off_part;
    a.Dm = c->mat[SPDK_M_DFP_TO_SP];
    a.S2F = c->mat[SPDK_M_SP_TO_FP];
    a.S2C = c->mat[SPDK_M_SP_TO_CV];
    a.inv = c->mat[SPDK_M_INVADER];
    a.w = c->wt;
    for (int d = 0; d < 3; d++) {
        a.Ne[d] = Ne[d];
        a.act[d] = c->prm.active[d];
        a.bc[d] = c->prm.bc[d];
        a.h[d] = c->prm.h[d];
        a.dh[d] = const_div(c->prm.h[d]);
    }
    a.E = (int)E;
    a.in_nv = NVP;
    a.dt = dt;
    a.gm = c->prm.gamma;
    a.cfl = c->prm.cfl;
    for (int d = 0; d < 3; d++) a.g[d] = c->prm.g[d];
    a.grav = (a.g[0] != 0.0 || a.g[1] != 0.0 || a.g[2] != 0.0);
    const unsigned eblocks = (unsigned)((E + G::EPB - 1) / G::EPB);  // workgroups of whole elements, one slice
    dim3 grid(eblocks), block(G::BLOCK);
    // timing: one event pair per sweep launch, harvested after the step's own sync
    auto launch_sweep = [&](auto mode_, const SweepArgs& args) -> int {
        constexpr int mode = decltype(mode_)::value;
        constexpr int ST = T > 1 ? T : 1;
        bool rec = c->timing && !x && c->ev_used < spdk_ctx::kEvPool;
        if (rec) SPDK_CHECK(hipEventRecord(c->evs[c->ev_used][0], c->stream));
        auto go = [&](auto slices) {
            constexpr int S = decltype(slices)::value;
            using X = Unit<N, DIM, T, S, mode>;
            unsigned nb = S == 1 ? eblocks : L.blocks;
            if (mode == FACES) nb = (nb + 7) / 8 * 8;
            hipLaunchKernelGGL((k_sweep<N, DIM, T, S, mode>), dim3(nb), block, sizeof(double) * X::DOUBLES, c->stream, args);
        };
        if constexpr (mode == FACES || ST == 1) go(std::integral_constant<int, 1>{});
        else if constexpr (mode == PREDICT) {
            if (args.in_ader) go(std::integral_constant<int, ST>{});
            else go(std::integral_constant<int, 1>{});
        } else go(std::integral_constant<int, ST>{});
        SPDK_LAUNCH_CHECK("k_sweep");
        if (rec) SPDK_CHECK(hipEventRecord(c->evs[c->ev_used++][1], c->stream));
        return SPDK_OK;
    };
    constexpr std::integral_constant<int, PREDICT> predict{};
    constexpr std::integral_constant<int, CORRECT> correct{};
    // the flux evaluation of the slices: face integrals, or flux-point arrays alone
    auto launch_fluxes = [&](const SweepArgs& args) -> int {
        if constexpr (T > 1) {
            if (args.Ffv[0][0]) return launch_sweep(std::integral_constant<int, FACES>{}, args);
            return launch_sweep(std::integral_constant<int, FLUXES>{}, args);
        }
        return SPDK_OK;
    };
    auto traces0 = [&]() -> int {
        hipLaunchKernelGGL((k_trace0<N, DIM>), grid, block, 0, c->stream, U_sp, NV, trA[0], trA[1], trA[2], a.S2F, (int)E);
        SPDK_LAUNCH_CHECK("k_trace0");
        return SPDK_OK;
    };
    int rc;
    const bool flux_out = x && (x->F_out[0] || x->Ffv);
    auto set_fv = [&](SweepArgs& sa) {
        if (!x || !x->Ffv) return;
        for (int t = 0; t < T; t++)
            for (int d = 0; d < 3; d++) sa.Ffv[t][d] = x->Ffv[t * 3 + d];
        for (int d = 0; d < 3; d++) { sa.fvn[d] = x->fvn[d]; sa.fgh[d] = x->fgh[d]; }
    };
    if (T > 1 && x && x->U_slices) {  // flux evaluation of given slices: their traces, then one flux sweep
        double* trS[3] = {nullptr, nullptr, nullptr};
        for (int d = 0; d < DIM; d++) trS[d] = W + (size_t)d * L.tr_axis;
        hipLaunchKernelGGL((k_trace0<N, DIM>), dim3(eblocks, T), block, 0, c->stream, x->U_slices, x->slices_nv, trS[0],
                           trS[1], trS[2], a.S2F, (int)E);
        SPDK_LAUNCH_CHECK("k_trace0");
        SweepArgs s = a;
        s.U0 = nullptr;
        s.part = nullptr;
        for (int d = 0; d < 3; d++) { s.tr_in[d] = trS[d]; s.tr_out[d] = nullptr; s.F_out[d] = x->F_out[d]; }
        s.tin_slices = T;
        s.in_ader = 1;
        s.U_in = x->U_slices;
        s.in_nv = x->slices_nv;
        s.out_nv = x->out_nv;
        set_fv(s);
        return launch_fluxes(s);
    }
    if (T > 1) {  // ADER: K = T sweeps, the last one with the corrector (or the flux evaluation)
        if ((rc = traces0())) return rc;
        const bool pred_only = x && x->U_export;
        for (int k = 0; k < (pred_only ? T - 1 : T); k++) {
            SweepArgs s = a;
            bool last = k == T - 1;
            double** tin = (k % 2 == 0) ? trA : trB;
            double** tout = (k % 2 == 0) ? trB : trA;
            for (int d = 0; d < 3; d++) { s.tr_in[d] = tin[d]; s.tr_out[d] = tout[d]; }
            s.tin_slices = k == 0 ? 1 : T;
            s.in_ader = k > 0;
            s.U_in = W + L.off_uader;
            s.U_out = W + L.off_uader;
            s.want_dt = last;
            s.W_cv = last ? W_cv : nullptr;
            s.F_x = last ? F_x : nullptr;
            if (last && flux_out) {
                s.want_dt = 0;
                s.W_cv = nullptr;
                s.F_x = nullptr;
                s.out_nv = x->out_nv;
                for (int d = 0; d < 3; d++) s.F_out[d] = x->F_out[d];
                set_fv(s);
                return launch_fluxes(s);
            }
            if constexpr (T > 1) {
                if ((rc = last ? launch_sweep(correct, s) : launch_sweep(predict, s))) return rc;
            }
        }
        if (pred_only) {
            const size_t slabE = E * G::TPE, total = (size_t)T * x->nv_export * slabE;
            hipLaunchKernelGGL(k_export_ader, dim3((unsigned)std::min<size_t>((total + 255) / 256, 65536)), dim3(256), 0,
                               c->stream, W + L.off_uader, x->U_export, x->nv_export, slabE, total);
            SPDK_LAUNCH_CHECK("k_export_ader");
            return SPDK_OK;
        }
    } else {  // SSP-RK stages (src/hydro_ader.hpp:313-325)
        int order = c->prm.rk_order;
        double rk[3] = {0, 0, 0};
        if (order == 2) rk[1] = 0.5;
        if (order == 3) { rk[1] = 0.75; rk[2] = 1.0 / 3.0; }
        for (int st = 0; st < order; st++) {
            if ((rc = traces0())) return rc;
            SweepArgs s = a;
            for (int d = 0; d < 3; d++) { s.tr_in[d] = trA[d]; s.tr_out[d] = nullptr; }
            s.tin_slices = 1;
            s.in_ader = 0;
            s.rk_a = rk[st];
            s.rk_first = st == 0 && order > 1;
            bool last = st == order - 1;
            s.want_dt = last;
            s.W_cv = last ? W_cv : nullptr;
            s.F_x = last ? F_x : nullptr;
            if constexpr (T == 1) {
                if ((rc = launch_sweep(correct, s))) return rc;
            }
        }
    }
    // one workgroup reads up to 16 k minima in about 5 us; more go through 256
    // first (64^3: 36 us in one). The result is written to the host's page.
    const double* mins = a.part;
    int nmin = (int)L.blocks;
    if (nmin > 16384) {
        hipLaunchKernelGGL(k_partial_min, dim3(kMinBlocks), dim3(1024), 0, c->stream, mins, nmin, a.part + L.blocks);
        SPDK_LAUNCH_CHECK("k_partial_min");
        mins = a.part + L.blocks;
        nmin = kMinBlocks;
    }
    hipLaunchKernelGGL(k_partial_min, dim3(1), dim3(1024), 0, c->stream, mins, nmin, c->red_host);
    SPDK_LAUNCH_CHECK("k_partial_min");
    SPDK_CHECK(hipStreamSynchronize(c->stream));
    if (dt_next) *dt_next = c->red_host[0];
    for (int i = 0; i < c->ev_used; i++) {
        float ms = 0;
        SPDK_CHECK(hipEventElapsedTime(&ms, c->evs[i][0], c->evs[i][1]));
        c->kernel_ms += ms;
        c->kernel_launches++;
    }
    c->ev_used = 0;
    return SPDK_OK;
}

typedef int (*step_fn)(spdk_ctx*, double*, const int*, void*, double, double*, double*, double*, const Extra*);
typedef Layout (*layout_fn)(size_t, int);
typedef size_t (*trace_fn)(size_t, int);

struct Variant {
    int n, dim;
    step_fn ader, rk;
    layout_fn layout;
    trace_fn slice_traces;
};
#define SPDK_VARIANT(Nn, D) {Nn, D, run_step<Nn, D, Nn>, run_step<Nn, D, 1>, layout_for<Nn, D>, slice_trace_doubles<Nn, D>}
const Variant kVariants[] = {SPDK_VARIANT(2, 1), SPDK_VARIANT(3, 1), SPDK_VARIANT(4, 1), SPDK_VARIANT(5, 1),
                             SPDK_VARIANT(2, 2), SPDK_VARIANT(3, 2), SPDK_VARIANT(4, 2), SPDK_VARIANT(5, 2),
                             SPDK_VARIANT(2, 3), SPDK_VARIANT(3, 3), SPDK_VARIANT(4, 3)};

const Variant* find_variant(spdk_ctx* c) {
    int dim = c->prm.active[0] + c->prm.active[1] + c->prm.active[2];
    // the fused tile assumes active axes are x, x-y or x-y-z
    if (!c->prm.active[0] || (c->prm.active[2] && !c->prm.active[1])) return nullptr;
    // the kernels are compiled for p+1 slices (ADER) or one (SSP-RK); grid and workspace follow c->T
    if (c->T != c->n && c->T != 1) return nullptr;
    for (const Variant& v : kVariants)
        if (v.n == c->n && v.dim == dim) return &v;
    return nullptr;
}

// Workspace of the allocation-free step entry: one array per GPU, resident
// until the process ends. A kernel takes its address as seen from the
// device, read per device with hipGetSymbolAddress (the array's name in host
// code is a host-side stand-in, not a device address).
constexpr size_t kScratchBytes = (size_t)64 << 20;
static __device__ __align__(256) double scratch[kScratchBytes / sizeof(double)];
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on the current device (looked up once per device).
int scratch_for_current_device(void** out) {
    int dev = -1;
    SPDK_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) { set_error("fused noalloc: device index out of range"); return SPDK_E_ARG; }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error(std::string("fused noalloc: hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
            return SPDK_E_HIP;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return SPDK_OK;
}

}  // namespace

extern "C" {

size_t spdk_fused_workspace_bytes(spdk_ctx* c, const int N[3]) {
    const Variant* v = c ? find_variant(c) : nullptr;
    if (!v) {
        set_error("fused path: no tile variant for this degree, dimensionality and slice count");
        return 0;
    }
    if (c->T > kMaxT || c->prm.nu != 0.0) {
        set_error("fused path covers the inviscid update");
        return 0;
    }
    Layout L = v->layout((size_t)N[0] * N[1] * N[2], c->T);
    return L.total * sizeof(double);
}

// Checks of a whole fused step on U_sp of shape s.
static int check_step_fused(spdk_ctx* c, const spdk_sd_shape& s, const Variant** vout) {
    if (c->prm.nu != 0.0) {
        set_error("fused path covers the inviscid update");
        return SPDK_E_CONFIG;
    }
    const Variant* v = find_variant(c);
    if (!v) { set_error("fused path: no tile variant for this degree, dimensionality and slice count"); return SPDK_E_CONFIG; }
    if (s.nv != NV || s.nt != 1 || s.nx != c->n || s.ny != (c->prm.active[1] ? c->n : 1) ||
        s.nz != (c->prm.active[2] ? c->n : 1)) {
        set_error("fused: U_sp shape");
        return SPDK_E_SHAPE;
    }
    for (int d = 0; d < 3; d++) {
        int Nd = d == 0 ? s.Nx : (d == 1 ? s.Ny : s.Nz);
        if (c->prm.active[d] && Nd < 3) { set_error("fused: axis needs ghost elements"); return SPDK_E_SHAPE; }
    }
    if ((uint64_t)s.Nx * s.Ny * s.Nz >= (1ull << 31)) { set_error("fused: too many elements"); return SPDK_E_SHAPE; }
    *vout = v;
    return SPDK_OK;
}

int spdk_hydro_step_fused(spdk_ctx* c, double* U_sp, spdk_sd_shape s, void* ws, double dt, double* W_cv, double* F_x,
                          double* dt_next) {
    if (!c || !U_sp || !ws) { set_error("fused: null argument"); return SPDK_E_ARG; }
    const Variant* v = nullptr;
    if (int rc = check_step_fused(c, s, &v)) return rc;
    int Ne[3] = {s.Nx, s.Ny, s.Nz};
    std::strncpy(c->kernel_name, "k_sweep", sizeof(c->kernel_name) - 1);
    if (c->T > 1) return v->ader(c, U_sp, Ne, ws, dt, W_cv, F_x, dt_next, nullptr);
    return v->rk(c, U_sp, Ne, ws, dt, W_cv, F_x, dt_next, nullptr);
}

size_t spdk_fused_noalloc_max_bytes(void) { return kScratchBytes; }

int spdk_hydro_step_fused_noalloc(spdk_ctx* c, double* U_sp, spdk_sd_shape s, double dt, double* W_cv, double* F_x,
                                  double* dt_next) {
    if (!c || !U_sp) { set_error("fused noalloc: null argument"); return SPDK_E_ARG; }
    const Variant* v = nullptr;
    if (int rc = check_step_fused(c, s, &v)) return rc;
    const size_t need = v->layout((size_t)s.Nx * s.Ny * s.Nz, c->T).total * sizeof(double);
    if (need > kScratchBytes) {
        set_error("fused noalloc: the step needs " + std::to_string(need) + " bytes of workspace, more than the " +
                  std::to_string(kScratchBytes) + " of the static scratch; use spdk_hydro_step_fused");
        return SPDK_E_SHAPE;
    }
    void* ws = nullptr;
    if (int rc = scratch_for_current_device(&ws)) return rc;
    int Ne[3] = {s.Nx, s.Ny, s.Nz};
    std::strncpy(c->kernel_name, "k_sweep", sizeof(c->kernel_name) - 1);
    if (c->T > 1) return v->ader(c, U_sp, Ne, ws, dt, W_cv, F_x, dt_next, nullptr);
    return v->rk(c, U_sp, Ne, ws, dt, W_cv, F_x, dt_next, nullptr);
}

int spdk_fused_predict(spdk_ctx* c, double* U_sp, spdk_sd_shape s, void* ws, double dt, double* U_ader,
                       spdk_sd_shape s_ader) {
    if (!c || !U_sp || !ws || !U_ader) { set_error("fused predict: null argument"); return SPDK_E_ARG; }
    if (c->prm.nu != 0.0 || c->T < 2) {
        set_error("fused predict covers the inviscid ADER predictor");
        return SPDK_E_CONFIG;
    }
    const Variant* v = find_variant(c);
    if (!v) { set_error("fused path: no tile variant for this degree, dimensionality and slice count"); return SPDK_E_CONFIG; }
    if (s.nv != NV || s.nt != 1 || s.nx != c->n || s.ny != (c->prm.active[1] ? c->n : 1) ||
        s.nz != (c->prm.active[2] ? c->n : 1) || s_ader.nt != c->T || s_ader.nv < NVP || s_ader.Nx != s.Nx ||
        s_ader.Ny != s.Ny || s_ader.Nz != s.Nz || s_ader.nx != s.nx || s_ader.ny != s.ny || s_ader.nz != s.nz) {
        set_error("fused predict: U_sp / U_ader shape");
        return SPDK_E_SHAPE;
    }
    for (int d = 0; d < 3; d++) {
        int Nd = d == 0 ? s.Nx : (d == 1 ? s.Ny : s.Nz);
        if (c->prm.active[d] && Nd < 3) { set_error("fused: axis needs ghost elements"); return SPDK_E_SHAPE; }
    }
    if ((uint64_t)s.Nx * s.Ny * s.Nz >= (1ull << 31)) { set_error("fused: too many elements"); return SPDK_E_SHAPE; }
    int Ne[3] = {s.Nx, s.Ny, s.Nz};
    std::strncpy(c->kernel_name, "k_sweep", sizeof(c->kernel_name) - 1);
    Extra x;
    x.U_export = U_ader;
    x.nv_export = s_ader.nv;
    return v->ader(c, U_sp, Ne, ws, dt, nullptr, nullptr, nullptr, &x);
}

// Checks shared by the flux-evaluation entries: the ADER slices shape and the
// flux-point arrays of the active axes.
static int check_flux_args(spdk_ctx* c, spdk_sd_shape s_ader, double* const F[3], const Variant** vout,
                           bool need_F = true) {
    if (c->prm.nu != 0.0 || c->T < 2) {
        set_error("fused flux evaluation covers the inviscid ADER step");
        return SPDK_E_CONFIG;
    }
    const Variant* v = find_variant(c);
    if (!v) { set_error("fused path: no tile variant for this degree, dimensionality and slice count"); return SPDK_E_CONFIG; }
    if (s_ader.nt != c->T || s_ader.nv < NVP || s_ader.nx != c->n || s_ader.ny != (c->prm.active[1] ? c->n : 1) ||
        s_ader.nz != (c->prm.active[2] ? c->n : 1)) {
        set_error("fused fluxes: slice shape");
        return SPDK_E_SHAPE;
    }
    for (int d = 0; d < 3; d++) {
        int Nd = d == 0 ? s_ader.Nx : (d == 1 ? s_ader.Ny : s_ader.Nz);
        if (c->prm.active[d] && Nd < 3) { set_error("fused: axis needs ghost elements"); return SPDK_E_SHAPE; }
        if (need_F && c->prm.active[d] && !F[d]) {
            set_error("fused fluxes: null flux array of an active axis");
            return SPDK_E_ARG;
        }
    }
    if ((uint64_t)s_ader.Nx * s_ader.Ny * s_ader.Nz >= (1ull << 31)) { set_error("fused: too many elements"); return SPDK_E_SHAPE; }
    *vout = v;
    return SPDK_OK;
}

int spdk_fused_predict_fluxes(spdk_ctx* c, double* U_sp, spdk_sd_shape s, void* ws, double dt, double* F_x,
                              double* F_y, double* F_z, spdk_sd_shape s_ader) {
    if (!c || !U_sp || !ws) { set_error("fused predict fluxes: null argument"); return SPDK_E_ARG; }
    double* F[3] = {F_x, F_y, F_z};
    const Variant* v = nullptr;
    int rc = check_flux_args(c, s_ader, F, &v);
    if (rc) return rc;
    if (s.nv != NV || s.nt != 1 || s.nx != s_ader.nx || s.ny != s_ader.ny || s.nz != s_ader.nz || s.Nx != s_ader.Nx ||
        s.Ny != s_ader.Ny || s.Nz != s_ader.Nz) {
        set_error("fused predict fluxes: U_sp shape");
        return SPDK_E_SHAPE;
    }
    int Ne[3] = {s.Nx, s.Ny, s.Nz};
    Extra x;
    for (int d = 0; d < 3; d++) x.F_out[d] = F[d];
    x.out_nv = s_ader.nv;
    std::strncpy(c->kernel_name, "k_sweep", sizeof(c->kernel_name) - 1);
    return v->ader(c, U_sp, Ne, ws, dt, nullptr, nullptr, nullptr, &x);
}

int spdk_fused_predict_fv_fluxes(spdk_ctx* c, double* U_sp, spdk_sd_shape s, void* ws, double dt, double* const* F_fv,
                                 spdk_fv_shape sc, double* F_x, spdk_sd_shape s_ader) {
    if (!c || !U_sp || !ws || !F_fv) { set_error("fused predict fv fluxes: null argument"); return SPDK_E_ARG; }
    double* F[3] = {F_x, nullptr, nullptr};  // flux-point arrays are optional here
    const Variant* v = nullptr;
    int rc = check_flux_args(c, s_ader, F, &v, false);
    if (rc) return rc;
    if (s.nv != NV || s.nt != 1 || s.nx != s_ader.nx || s.ny != s_ader.ny || s.nz != s_ader.nz || s.Nx != s_ader.Nx ||
        s.Ny != s_ader.Ny || s.Nz != s_ader.Nz) {
        set_error("fused predict fv fluxes: U_sp shape");
        return SPDK_E_SHAPE;
    }
    const int Ne[3] = {s.Nx, s.Ny, s.Nz}, nc[3] = {sc.Nx, sc.Ny, sc.Nz};
    for (int d = 0; d < 3; d++) {
        const bool act = c->prm.active[d] != 0;
        const bool ok = act ? (Ne[d] > 2 * c->ngh[d] && nc[d] == (Ne[d] - 2 * c->ngh[d]) * c->n + 2 * c->fgh[d] &&
                               c->ngh[d] == 1)
                            : (Ne[d] == 1 && nc[d] == 1);
        if (!ok || sc.nv != NV) {
            set_error("fused predict fv fluxes: FV cell shape disagrees with U_sp along axis " + std::to_string(d));
            return SPDK_E_SHAPE;
        }
        for (int t = 0; t < c->T; t++)
            if (act && !F_fv[t * 3 + d]) { set_error("fused predict fv fluxes: null face array"); return SPDK_E_ARG; }
    }
    Extra x;
    x.F_out[0] = F_x;  // optional: the x flux-point fluxes (outputs)
    x.out_nv = s_ader.nv;
    x.Ffv = F_fv;
    for (int d = 0; d < 3; d++) { x.fvn[d] = nc[d]; x.fgh[d] = c->fgh[d]; }
    std::strncpy(c->kernel_name, "k_sweep", sizeof(c->kernel_name) - 1);
    return v->ader(c, U_sp, Ne, ws, dt, nullptr, nullptr, nullptr, &x);
}

size_t spdk_fused_fluxes_workspace_bytes(spdk_ctx* c, const int N[3]) {
    const Variant* v = c ? find_variant(c) : nullptr;
    if (!v || c->T < 2) {
        set_error("fused fluxes: no tile variant for this degree, dimensionality and slice count, or not ADER");
        return 0;
    }
    return v->slice_traces((size_t)N[0] * N[1] * N[2], c->T) * sizeof(double);
}

int spdk_fused_fluxes(spdk_ctx* c, const double* U_ader, spdk_sd_shape s_ader, void* ws, double* F_x, double* F_y,
                      double* F_z) {
    if (!c || !U_ader || !ws) { set_error("fused fluxes: null argument"); return SPDK_E_ARG; }
    double* F[3] = {F_x, F_y, F_z};
    const Variant* v = nullptr;
    int rc = check_flux_args(c, s_ader, F, &v);
    if (rc) return rc;
    int Ne[3] = {s_ader.Nx, s_ader.Ny, s_ader.Nz};
    Extra x;
    for (int d = 0; d < 3; d++) x.F_out[d] = F[d];
    x.out_nv = s_ader.nv;
    x.U_slices = U_ader;
    x.slices_nv = s_ader.nv;
    std::strncpy(c->kernel_name, "k_sweep", sizeof(c->kernel_name) - 1);
    return v->ader(c, nullptr, Ne, ws, 0.0, nullptr, nullptr, nullptr, &x);
}

}  // extern "C"
