// Single large circuit instance on MI355X (gfx950): the whole Newton inner loop for one netlist of tens of
// thousands of unknowns, which does not fit the batched kernel's per-instance LDS region.
//
//   * device evaluation, one thread per device, every stamp to its own contribution cell in HBM
//     (models.h, the same functions the batched kernel runs);
//   * ordered gather: each matrix element and RHS entry sums its contributions in component order, then
//     stamp order -- the order Solver::update adds them (analysis.rs:153-168) -- without atomics;
//   * the KCL residual in FP64 and the reference's convergence test (analysis.rs:331-345);
//   * a multifrontal LU over the order large_sym.cpp fixes: fronts of up to SMALL_MAX entries a side
//     assembled and factored in one workgroup's LDS, many fronts per launch by elimination-tree levels;
//     larger fronts assembled in column blocks and factored by panels (a diagonal-block LU in LDS, then
//     the panel's L rows and U columns and the trailing update on the matrix cores);
//   * forward and backward sweeps front by front, level by level;
//   * the max-|dx| <= 1 clamp and update (analysis.rs:196-207), commit of device state on convergence.
// The Newton loop, the fixed-step Backward-Euler time loop and IC forcing (analysis.rs:489-574) are
// driven from the host with one 16-byte read-back per iteration.  Mixed precision factors and sweeps in
// FP32; evaluation, residual, update and the convergence test stay FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <unordered_map>
#include <vector>

#include "bsim4_eval.h"
#include "devmem.h"
#include "internal.h"
#include "large.h"
#include "models.h"

#define LCHECK(x)                                                                           \
    do {                                                                                    \
        hipError_t e_ = (x);                                                                \
        if (e_ != hipSuccess) s21::fail(S21_DEVICE, std::string("HIP: ") + hipGetErrorString(e_)); \
    } while (0)

namespace s21 {
namespace lg {

constexpr int TPB = 256;
constexpr int NB = 64;                   // panel width of the blocked factorisation of large fronts
constexpr int CB = 16;                   // column block of the large-front assembly
// Sides of the fronts that one wavefront factors and sweeps, and one workgroup; larger ones go by panels.  A 90 x 90
// grid's factorisation, FP64 / FP32 ms: up to 24 and 64 a side 1.01 / 0.85, 32 and 48 1.00 / 0.85, 32 and 64 1.03 /
// 0.87, 32 and 96 1.07 / 0.90, 48 and 128 1.21 / 1.03; on 72 x 72, 24 and 64 are 2 to 3 % ahead of 32 and 48.
constexpr int WAVE_MAX = 24, SMALL_MAX = 64;
constexpr size_t SMALL_LDS = 128 * 1024; // LDS bytes a small front may take, its children's maps included
constexpr int M1F = 11, M1C = 4, M1S = 7, DPF = 14, DSF = 4;

// Orders the LDS accesses of one wavefront's lanes (a wavefront executes its LDS operations in order; the
// fences keep the compiler from moving accesses across this point).
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

static_assert(WAVE_MAX <= 64 && SMALL_MAX <= TPB, "the small-front sweeps give every row of a front a thread of its own");

// ---------------------------------------------------------------------------------------------------
// Device evaluation
// ---------------------------------------------------------------------------------------------------
struct EvalArgs {
    int n_m1, n_d, n_lin, tran;
    double gmin, dt;
    const double* x;
    const int* m1_node;   // [n_m1][6] d g s b dp sp (-1 = ground)
    const double* m1_par; // [M1F + M1C][n_m1]
    const int* m1_caps;   // [n_m1] 1 when the device carries gate charge
    double* m1_state;     // [2 * M1S][n_m1]: committed op, then guess
    const int* m1_cb;     // [n_m1] first contribution cell
    const int* d_node;    // [n_d][3] p n r
    const double* d_par;  // [DPF][n_d]
    double* d_state;      // [DSF][n_d]: guess vd, guess charge, committed charge, vd the last load started from
    const int* d_cb;
    const int* l_node;    // [n_lin][3]
    const int* l_type;    // [n_lin] S21_COMP_*
    const double* l_val;  // [2][n_lin] operating-point and transient values
    const double* c_q;    // [n_lin] committed capacitor charge
    const int* l_cb;
    double* cv;           // contribution cells
    // trapezoidal integration: trap = 1 integrates by the trapezoidal rule, 2 by Backward Euler while
    // recording each charge's current (the first step, from an operating point whose capacitor currents
    // are zero), 0 by Backward Euler alone.  Per charge, the current at the last accepted point
    // (committed) and the one of the current guess.
    int trap;
    double* m1_icur;      // [4][n_m1]: committed gate-drain (tr.gs) and gate-bulk currents, then guesses
    double* d_icur;       // [2][n_d]: committed junction-charge current, then guess
    double* c_icur;       // [2][n_lin]: committed capacitor current, then guess
};

__device__ inline double xval(const double* x, int v) { return v < 0 ? 0.0 : x[v]; }

__global__ void __launch_bounds__(TPB) k_eval(EvalArgs E) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < E.n_m1) {
        const int j = t, nm = E.n_m1;
        const int* nd = E.m1_node + 6 * j;
        auto F = [&](int f) { return E.m1_par[(size_t)f * nm + j]; };
        Mos1Core P{F(0), F(1), F(2), F(3),  F(4),        F(5),       F(6),
                   F(7), F(8), F(9), F(10), F(7) / F(6), F(8) / F(6)};
        double* cv = E.cv + E.m1_cb[j];
        auto put = [&](int e, double v) { cv[e] = v; };
        const double vd = xval(E.x, nd[RD]), vg = xval(E.x, nd[RG]), vs = xval(E.x, nd[RS]), vb = xval(E.x, nd[RB]);
        if (!E.m1_caps[j]) {
            mos1_load<false>(P, nullptr, nullptr, vd, vg, vs, vb, E.gmin, E.dt, put, nullptr);
            return;
        }
        Mos1Caps K{F(M1F + 0), F(M1F + 1), F(M1F + 2), F(M1F + 3)};
        double* st = E.m1_state;
        Mos1State op{st[0 * nm + j], st[1 * nm + j], st[2 * nm + j], st[3 * nm + j],
                     st[4 * nm + j], st[5 * nm + j], st[6 * nm + j]};
        Mos1State gs{};
        if (E.tran) {
            if (E.trap) {
                const double ip[2] = {E.m1_icur[(size_t)0 * nm + j], E.m1_icur[(size_t)1 * nm + j]};
                double io[2];
                mos1_load<true>(P, &K, &op, vd, vg, vs, vb, E.gmin, E.dt, put, &gs, nullptr, E.trap == 1 ? ip : nullptr,
                                io);
                E.m1_icur[(size_t)2 * nm + j] = io[0];
                E.m1_icur[(size_t)3 * nm + j] = io[1];
            } else {
                mos1_load<true>(P, &K, &op, vd, vg, vs, vb, E.gmin, E.dt, put, &gs);
            }
        } else {
            mos1_load<false>(P, &K, &op, vd, vg, vs, vb, E.gmin, E.dt, put, &gs);
        }
        st[7 * nm + j] = gs.vgs;
        st[8 * nm + j] = gs.vgd;
        st[9 * nm + j] = gs.vgb;
        st[10 * nm + j] = gs.cgs;
        st[11 * nm + j] = gs.cgd;
        st[12 * nm + j] = gs.cgb;
        st[13 * nm + j] = gs.reversed;
        return;
    }
    if (t < E.n_m1 + E.n_d) {
        const int j = t - E.n_m1, nd_ = E.n_d;
        const int* nd = E.d_node + 3 * j;
        auto F = [&](int f) { return E.d_par[(size_t)f * nd_ + j]; };
        DiodeP P{F(0), F(1), F(2), F(3), F(4), F(5), F(6), F(7), F(8), F(9), F(10), F(11), F(12), F(13)};
        double* st = E.d_state;
        const double vd0 = st[0 * nd_ + j];
        double* cv = E.cv + E.d_cb[j];
        auto put = [&](int e, double v) { cv[e] = v; };
        DiodeGuess gs;
        const double vr = xval(E.x, nd[DR_]), vn = xval(E.x, nd[DN_]);
        if (E.tran && E.trap)
            diode_load<true>(P, vr, vn, E.gmin, E.dt, vd0, st[2 * nd_ + j], put, &gs,
                             E.trap == 1 ? E.d_icur + j : nullptr, E.d_icur + nd_ + j);
        else if (E.tran)
            diode_load<true>(P, vr, vn, E.gmin, E.dt, vd0, st[2 * nd_ + j], put, &gs);
        else
            diode_load<false>(P, vr, vn, E.gmin, E.dt, vd0, st[2 * nd_ + j], put, &gs);
        st[0 * nd_ + j] = gs.vd;
        st[1 * nd_ + j] = gs.charge;
        st[3 * nd_ + j] = vd0;
        return;
    }
    if (t < E.n_m1 + E.n_d + E.n_lin) {
        const int j = t - E.n_m1 - E.n_d;
        const int* nd = E.l_node + 3 * j;
        double* cv = E.cv + E.l_cb[j];
        const double val = E.l_val[(size_t)(E.tran ? 1 : 0) * E.n_lin + j];
        switch (E.l_type[j]) {
        case S21_COMP_R:
            cv[0] = val;
            cv[1] = val;
            cv[2] = -val;
            cv[3] = -val;
            break;
        case S21_COMP_C:
            if (!E.tran) {  // no stamps in the operating point (comps/mod.rs:205-209)
                for (int e = 0; e < C_NE; e++) cv[e] = 0.0;
            } else {
                cap_load_tran(val, xval(E.x, nd[0]) - xval(E.x, nd[1]), E.c_q[j], E.dt,
                              [&](int e, double v) { cv[e] = v; }, E.trap == 1 ? E.c_icur + j : nullptr,
                              E.trap ? E.c_icur + E.n_lin + j : nullptr);
            }
            break;
        case S21_COMP_V:
            cv[0] = 1.0;
            cv[1] = 1.0;
            cv[2] = -1.0;
            cv[3] = -1.0;
            cv[4] = val;
            break;
        default:
            cv[0] = val;
            cv[1] = -val;
        }
    }
}

// BSIM4, one thread per device (bsim4solver.rs:134-145, 3757-3769): Bsim4::op from the port voltages with
// limiting against the device's last guess, tran_op's Backward-Euler charge companions against the committed
// charges in a transient, then the 42 stamps into the device's contribution cells.  Parameters and state are
// structures of arrays in HBM (field-major, so consecutive threads read consecutive addresses): parameter
// field K of device j at par[K][j]; state [B4S_F][j]: the last load's limiting fields (vds vgs vbs vbd von)
// and charges (qg qd qb), then the committed charges.
constexpr int B4S_LIM = 0, B4S_Q = 5, B4S_QC = 8, B4S_F = 11;
struct B4Args {
    int n, tran;
    double gmin, dt;
    const double* x;
    const int* node;   // [n][4] d g s b (-1 = ground)
    const double* par; // [parameter doubles][n]
    double* st;        // [B4S_F][n]
    const int* cb;     // [n] first contribution cell
    double* cv;
};
// The parameter view of one device: field K read where it is stored.
struct B4Fields {
    const double* par;
    int n, j;
    template <int K>
    __device__ double get() const {
        return par[(size_t)K * n + j];
    }
};

__global__ void __launch_bounds__(128) k_eval_b4(B4Args A) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= A.n) return;
    const int* nd = A.node + 4 * j;
    const B4Fields P{A.par, A.n, j};
    const size_t n = A.n;
    b4::B4Op G;  // only the limiting fields of the last load's point are read
    G.vds = A.st[(B4S_LIM + 0) * n + j];
    G.vgs = A.st[(B4S_LIM + 1) * n + j];
    G.vbs = A.st[(B4S_LIM + 2) * n + j];
    G.vbd = A.st[(B4S_LIM + 3) * n + j];
    G.von = A.st[(B4S_LIM + 4) * n + j];
    b4::B4Op N;
    b4::op_eval(P, G, xval(A.x, nd[0]), xval(A.x, nd[1]), xval(A.x, nd[2]), xval(A.x, nd[3]), A.gmin, N);
    b4::B4Tran T{};
    if (A.tran) {
        b4::B4Op O;  // tran_op reads the committed point's charges only
        O.qg = A.st[(B4S_QC + 0) * n + j];
        O.qd = A.st[(B4S_QC + 1) * n + j];
        O.qb = A.st[(B4S_QC + 2) * n + j];
        b4::tran_eval(P, O, N, A.dt, T);
    }
    double* cv = A.cv + A.cb[j];
    b4::stamp(P, N, T, [&](int k, double v) { cv[k] = v; });
    A.st[(B4S_LIM + 0) * n + j] = N.vds;
    A.st[(B4S_LIM + 1) * n + j] = N.vgs;
    A.st[(B4S_LIM + 2) * n + j] = N.vbs;
    A.st[(B4S_LIM + 3) * n + j] = N.vbd;
    A.st[(B4S_LIM + 4) * n + j] = N.von;
    A.st[(B4S_Q + 0) * n + j] = N.qg;
    A.st[(B4S_Q + 1) * n + j] = N.qd;
    A.st[(B4S_Q + 2) * n + j] = N.qb;
}

__global__ void k_commit_b4(int n, double* __restrict__ st) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n)
        for (int f = 0; f < 3; f++) st[(size_t)(B4S_QC + f) * n + j] = st[(size_t)(B4S_Q + f) * n + j];
}

// Each matrix element (then each RHS entry) sums its contributions in component-then-stamp order.
__global__ void __launch_bounds__(TPB) k_gather(int n_slots, const int* __restrict__ ptr, const int* __restrict__ idx,
                                                const double* __restrict__ cv, double* __restrict__ out) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n_slots) return;
    double acc = 0.0;
    for (int q = ptr[s]; q < ptr[s + 1]; q++) acc = acc + cv[idx[q]];
    out[s] = acc;
}

// res = rhs - A x by rows of A (elements of each row in creation order); flags[0] |= 1 when some
// |res_i| > iabstol (false for NaN, as the reference's comparison); *resmax = max |res_i| (NaN skipped),
// as the bits of a non-negative double.
__global__ void __launch_bounds__(TPB) k_residual(int n, const int* __restrict__ rptr, const int* __restrict__ relem,
                                                  const int* __restrict__ ecol, const double* __restrict__ val,
                                                  const double* __restrict__ rhs, const double* __restrict__ x,
                                                  double* __restrict__ res, double iabstol, int* flags,
                                                  unsigned long long* resmax) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    double m = 0.0;
    if (r < n) {
        double acc = 0.0;
        for (int q = rptr[r]; q < rptr[r + 1]; q++) {
            const int e = relem[q];
            acc = acc + val[e] * x[ecol[e]];
        }
        const double v = rhs[r] - acc;
        res[r] = v;
        if (fabs(v) > iabstol) atomicOr(flags, 1);
        if (fabs(v) == fabs(v)) m = fabs(v);
    }
    for (int o = 32; o > 0; o >>= 1) {
        const double u = __shfl_xor(m, o, 64);
        m = u > m ? u : m;
    }
    if ((threadIdx.x & 63) == 0 && m > 0.0) atomicMax(resmax, (unsigned long long)__double_as_longlong(m));
}

// ---------------------------------------------------------------------------------------------------
// Multifrontal factorisation
// ---------------------------------------------------------------------------------------------------
// What a kernel needs of one front, in launch order: a workgroup reads its own with one scalar load instead of
// chasing the structure's arrays (a microsecond a hop on data that another XCD's kernel displaced).
struct FrontD {
    int64_t fo;    // offset in the pool
    int64_t w;     // offset of its sweep vector (F entries)
    int64_t r;     // offset of its rows below the pivots in r_idx
    int k, F;      // pivots, side
    int f, p;      // first internal column; first panel among all large fronts' panels
    int ch0, ch1;  // children (ChildD)
    int a0, a1;    // entries of A
    int m0, m1;    // its children's maps in c_map
};
// A child of a front: its update block in the pool, and its rows' positions in the parent.
struct ChildD {
    int64_t u;   // pool offset of the block's first entry
    int mc, Fc;  // side and leading dimension
    int map;     // offset in c_map, from the parent's m0
};
// A tile of a large front's assembly: 256 rows from r0 by CB columns from c0, the entries of A and the pieces of
// children's update blocks that fall into it.
struct AsmJob {
    int64_t fo;
    int F, r0, c0;
    int p0, p1, a0, a1;
};
struct AsmPiece {
    int64_t u;       // pool offset of the piece's first entry
    int Fc, ni, nj;  // leading dimension, rows, columns
    int mi, mj;      // c_map offsets of the rows' and the columns' positions
};

// Small fronts: assemble (zero, A entries, children's update blocks in order), partial LU, write back; one
// workgroup of NT threads per front, the front in LDS with its children's maps after it.  A front of a few dozen rows
// takes one wavefront, which needs no barriers.
template <int NT>
__device__ inline void front_sync() {
    if (NT == 64)
        wave_sync();
    else
        __syncthreads();
}
template <typename T, int NT>
__global__ void __launch_bounds__(NT) k_small(const FrontD* __restrict__ fr, const ChildD* __restrict__ child,
                                              const int* __restrict__ c_map, const int* __restrict__ a_elem,
                                              const int* __restrict__ a_off, const double* __restrict__ aval,
                                              T* __restrict__ pool, int* flags) {
    extern __shared__ char lds_raw[];
    constexpr int TX = NT == 64 ? 8 : 16, TY = NT / TX;
    const FrontD S = fr[blockIdx.x];
    const int k = S.k, F = S.F;
    T* L = (T*)lds_raw;
    int* M = (int*)(L + F * F);
    const int tid = threadIdx.x, ti = tid % TX, tj = tid / TX;
    for (int i = tid; i < S.m1 - S.m0; i += NT) M[i] = c_map[S.m0 + i];
    for (int i = tid; i < F * F; i += NT) L[i] = (T)0;
    front_sync<NT>();
    for (int q = S.a0 + tid; q < S.a1; q += NT) L[a_off[q]] = (T)aval[a_elem[q]];
    front_sync<NT>();
    for (int c = S.ch0; c < S.ch1; c++) {
        const ChildD C = child[c];
        const int* mp = M + C.map;
        const T* U = pool + C.u;
        for (int j = tj; j < C.mc; j += TY) {
            const int col = mp[j] * F;
            for (int i = ti; i < C.mc; i += TX) L[col + mp[i]] += U[(size_t)j * C.Fc + i];
        }
        front_sync<NT>();
    }
    for (int j = 0; j < k; j++) {
        const T piv = L[j * F + j];
        if (piv == (T)0 && tid == 0) atomicOr(flags, 2);
        for (int i = j + 1 + tid; i < F; i += NT) L[j * F + i] = L[j * F + i] / piv;
        front_sync<NT>();
        for (int c = j + 1 + tj; c < F; c += TY) {
            const T u = L[c * F + j];
            for (int i = j + 1 + ti; i < F; i += TX) L[c * F + i] = L[c * F + i] - L[j * F + i] * u;
        }
        front_sync<NT>();
    }
    T* out = pool + S.fo;
    for (int i = tid; i < F * F; i += NT) out[i] = L[i];
}

// Large fronts, assembly: one tile a workgroup, in LDS, thread = row.  A piece of a child's update block adds to
// distinct entries; the pieces follow each other in child order.  The next piece's entries are read while one is
// added.  Searching every child's map for its columns and adding in HBM took 110 us a level (200 x 200 grid, FP32);
// this takes 18 us.
template <typename T>
__global__ void __launch_bounds__(TPB) k_assemble(const AsmJob* __restrict__ job, const AsmPiece* __restrict__ piece,
                                                  const int* __restrict__ c_map, const int* __restrict__ a_elem,
                                                  const int* __restrict__ a_tile, const double* __restrict__ aval,
                                                  T* __restrict__ pool) {
    __shared__ T L[CB][TPB];
    const AsmJob J = job[blockIdx.x];
    const int t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < CB; q++) L[q][t] = (T)0;
    __syncthreads();
    for (int q = J.a0 + t; q < J.a1; q += TPB) L[a_tile[q] / TPB][a_tile[q] % TPB] = (T)aval[a_elem[q]];
    T v[CB];
    int m = 0;
    auto load = [&](int p) {
        const AsmPiece P = piece[p];
        if (t < P.ni) {
            m = c_map[P.mi + t] - J.r0;
#pragma unroll
            for (int q = 0; q < CB; q++) v[q] = q < P.nj ? pool[P.u + (int64_t)q * P.Fc + t] : (T)0;
        }
    };
    if (J.p0 < J.p1) load(J.p0);
    __syncthreads();
    for (int p = J.p0; p < J.p1; p++) {
        const AsmPiece P = piece[p];
        T w[CB];
        const int row = m;
#pragma unroll
        for (int q = 0; q < CB; q++) w[q] = v[q];
        if (p + 1 < J.p1) load(p + 1);
        if (t < P.ni)
#pragma unroll
            for (int q = 0; q < CB; q++)
                if (q < P.nj) L[c_map[P.mj + q] - J.c0][row] += w[q];
        __syncthreads();
    }
    const int i = J.r0 + t;
    T* A = pool + J.fo;
    if (i < J.F)
#pragma unroll
        for (int q = 0; q < CB; q++)
            if (J.c0 + q < J.F) A[(size_t)(J.c0 + q) * J.F + i] = L[q][t];
}

// Value of v in lane l (l the same for every lane), through the scalar unit.
__device__ inline double lane_value(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ inline float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// ---- matrix-core tiles ---------------------------------------------------------------------------
// 16 x 16 x 4 products in FP64 and FP32.  Lane l supplies A[l % 16][k] and B[k][l % 16] of the step's k for its
// group g = l / 16, and holds D[mfma_row(l, r)][l % 16] in register r.  As the k of a step may be any four columns,
// register r of a D is the B operand of the step whose k are mfma_row(., r).
template <typename T>
using Acc = T __attribute__((ext_vector_type(4)));
__device__ inline Acc<double> mfma(double a, double b, Acc<double> c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline Acc<float> mfma(float a, float b, Acc<float> c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
template <typename T>
__device__ inline int mfma_row(int g, int r) {
    return sizeof(T) == 8 ? 4 * r + g : 4 * g + r;
}

constexpr int SB = 16;                       // sub-block of a panel's diagonal block
constexpr int INV = 2 * (NB / SB) * SB * SB; // inverses kept per panel: the L, then the U sub-blocks on its diagonal
constexpr int DLD = NB + 1;                  // leading dimension of the diagonal block in LDS

// Inverse of the 16 x 16 L (or U) sub-block at column o of D, one column per lane of a wavefront's first sixteen:
// L by columns, U by rows (their readers' order).  rp: the pivots' reciprocals.
template <typename T, bool UPPER>
__device__ __attribute__((always_inline)) inline void invert_sub(const T* D, const T* rp, int o, T* __restrict__ inv) {
    const int col = threadIdx.x & 63;
    if (col >= SB) return;
    T x[SB];
#pragma unroll
    for (int i = 0; i < SB; i++) x[i] = i == col ? (T)1 : (T)0;
    if (!UPPER) {
#pragma unroll
        for (int j = 0; j < SB; j++)
#pragma unroll
            for (int i = j + 1; i < SB; i++) x[i] = fma(-D[(o + i) * DLD + o + j], x[j], x[i]);
#pragma unroll
        for (int i = 0; i < SB; i++) inv[(o + col) * SB + i] = x[i];
    } else {
#pragma unroll
        for (int j = SB - 1; j >= 0; j--) {
            x[j] = x[j] * rp[o + j];
#pragma unroll
            for (int i = 0; i < j; i++) x[i] = fma(-D[(o + i) * DLD + o + j], x[j], x[i]);
        }
#pragma unroll
        for (int i = 0; i < SB; i++) inv[(NB + o + i) * SB + col] = x[i];
    }
}

// LU of a panel's w x w diagonal block D (rows by DLD, in LDS, padded to 64 x 64 by the identity) by a workgroup
// of 256 threads, and the inverses of its 16 x 16 L and U diagonal sub-blocks.  A sub-block's 16 columns are
// eliminated by wavefront 0, lane i holding row i, the pivot rows broadcast by the scalar unit; the rows right of it are
// solved one column per lane; the rest is updated on the matrix cores, the next sub-block's columns first, so that
// wavefront 0 goes on while the others update what is right of them and invert the finished sub-block.
// Serial by nature, and bound by the chain from one pivot to the next -- its broadcast, a division, a multiply-add --
// and by the issue of one wavefront's instructions.  One wavefront holding all 64 columns spent 28 us (FP64) and 31 us
// (FP32) on a block; this takes 13.6 and 10.6 us in a launch of its own, and costs nothing beside a large trailing update.
// (With the pivot rows through LDS 15.3 and 11.8 us; not inlined, its LDS became generic memory: 7 us more.)  Every
// multiplier is a rounded quotient.  Two pivots at a time through their determinant took as long, 13.7 and 10.8 us, and the
// determinant leaves the range of FP32 for pivots of 1e-19 or 1e19, and loses digits in a nearly singular pair that the
// pair's own factors keep.
template <typename T>
__device__ __attribute__((always_inline)) inline void diag_lu(T* D, T* rp, int w, T* __restrict__ inv, int* flags) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, n = lane & 15;
    // tile (i0, j0) -= L(i0, c0) U(c0, j0), 16 columns of L
    auto update = [&](int c0, int i0, int j0) {
        Acc<T> acc;
#pragma unroll
        for (int r = 0; r < 4; r++) acc[r] = D[(i0 + mfma_row<T>(g, r)) * DLD + j0 + n];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int k = c0 + 4 * r + g;
            acc = mfma(-D[(i0 + n) * DLD + k], D[k * DLD + j0 + n], acc);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) D[(i0 + mfma_row<T>(g, r)) * DLD + j0 + n] = acc[r];
    };
    for (int c0 = 0; c0 < w; c0 += SB) {
        const int c1 = c0 + SB, nt = (NB - c1) / SB;
        if (wave == 0) {
            T r[SB];
#pragma unroll
            for (int q = 0; q < SB; q++) r[q] = D[lane * DLD + c0 + q];
#pragma unroll
            for (int j = 0; j < SB; j++) {
                // the pivot row reaches every lane through the scalar unit
                T u[SB];
#pragma unroll
                for (int q = j; q < SB; q++) u[q] = lane_value(r[q], c0 + j);
                if (lane == 0 && u[j] == (T)0) atomicOr(flags, 2);
                const T quot = r[j] / u[j];
                const T l = lane > c0 + j ? quot : (T)0;
                r[j] = lane > c0 + j ? l : r[j];
#pragma unroll
                for (int q = j + 1; q < SB; q++) r[q] = fma(-l, u[q], r[q]);
            }
            if (lane >= c0) {
#pragma unroll
                for (int q = 0; q < SB; q++) D[lane * DLD + c0 + q] = r[q];
            }
            wave_sync();
            if (lane < SB) rp[c0 + lane] = (T)1 / D[(c0 + lane) * DLD + c0 + lane];
        } else if (c0 > 0) {  // the rest of the previous sub-block's update, and its inverses
            for (int t = wave - 1; t < (nt + 1) * nt; t += 3)
                update(c0 - SB, c0 + (t % (nt + 1)) * SB, c1 + (t / (nt + 1)) * SB);
            if (wave == 2) invert_sub<T, false>(D, rp, c0 - SB, inv);
            if (wave == 3) invert_sub<T, true>(D, rp, c0 - SB, inv);
        }
        __syncthreads();
        if (c1 >= w) break;
        if (wave == 0 && lane < NB - c1) {  // rows [c0, c1) right of the sub-block: unit lower solve by columns
            T y[SB];
#pragma unroll
            for (int i = 0; i < SB; i++) y[i] = D[(c0 + i) * DLD + c1 + lane];
#pragma unroll
            for (int j = 0; j < SB; j++)
#pragma unroll
                for (int i = j + 1; i < SB; i++) y[i] = fma(-D[(c0 + i) * DLD + c0 + j], y[j], y[i]);
#pragma unroll
            for (int i = 0; i < SB; i++) D[(c0 + i) * DLD + c1 + lane] = y[i];
        }
        __syncthreads();
        if (wave < nt) update(c0, c1 + wave * SB, c1);  // the next sub-block's columns
        __syncthreads();
    }
    const int last = (w - 1) / SB * SB;
    if (wave == 0) invert_sub<T, false>(D, rp, last, inv);
    if (wave == 1) invert_sub<T, true>(D, rp, last, inv);
}

// The first panel's diagonal block of each large front (the later ones are factored by k_update_big).
template <typename T>
__global__ void __launch_bounds__(TPB) k_diag(const FrontD* __restrict__ fr, T* __restrict__ pool,
                                              T* __restrict__ inv, int* flags) {
    __shared__ T D[NB * DLD], rp[NB];
    const FrontD S = fr[blockIdx.x];
    const int F = S.F, w = min(NB, S.k);
    T* A = pool + S.fo;
    T v[NB * NB / TPB];  // every load on its way before the first is used
#pragma unroll
    for (int u = 0; u < NB * NB / TPB; u++) {
        const int i = threadIdx.x % NB, j = threadIdx.x / NB + u * (TPB / NB);
        v[u] = i < w && j < w ? A[(size_t)j * F + i] : i == j ? (T)1 : (T)0;
    }
#pragma unroll
    for (int u = 0; u < NB * NB / TPB; u++) D[(threadIdx.x % NB) * DLD + threadIdx.x / NB + u * (TPB / NB)] = v[u];
    __syncthreads();
    diag_lu<T>(D, rp, w, inv + (size_t)S.p * INV, flags);
    for (int q = threadIdx.x; q < NB * NB; q += TPB) {
        const int i = q % NB, j = q / NB;
        if (i < w && j < w) A[(size_t)j * F + i] = D[i * DLD + j];
    }
}

// Large fronts, the panel's L rows (x U11 = a) and U columns (L11 y = a): a wavefront solves 16 of them on the matrix
// cores, sub-block by sub-block: y_b = inv(M_bb) (a_b - sum_{c<b} M_bc y_c) with M = L11, or U11 transposed for
// rows (x^T is then a column).  The product by an inverse leaves a residual that grows with the sub-block's condition
// (networks with conductances of either sign: 3 times the error of substitution, and an operating point in mixed
// precision that did not converge), so y_b is corrected once by its own residual.  y_c comes out of one product in the
// layout the next takes it in.  Its 56 operand registers are loaded before the first product; grid.x * 4 wavefronts,
// grid.y the front.  One row or column per thread by substitution took 28 us a panel in FP64 and 37 in FP32, 2,000
// dependent multiply-adds through LDS; this takes 9.3 and 7.6 us, 7.4 and 6.2 without the correction.
template <typename T>
__global__ void __launch_bounds__(TPB) k_trsm(const FrontD* __restrict__ fr, int panel, T* __restrict__ pool,
                                              const T* __restrict__ invs) {
    const FrontD S = fr[blockIdx.y];
    const int k = S.k, F = S.F;
    const int c = panel * NB;
    if (c >= k) return;
    const int w = min(NB, k - c);
    const int r0 = c + w, units = (F - r0 + SB - 1) / SB;
    const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (unit >= 2 * units) return;
    const bool rows = unit < units;
    T* A = pool + S.fo;
    const T* inv = invs + ((size_t)S.p + panel) * INV + (rows ? (NB / SB) * SB * SB : 0);
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int o = r0 + (rows ? unit : unit - units) * SB + n;
    // loads are never under a mask (a mask costs more instructions than its load): rows past the front repeat its last
    // and are not stored, columns past a short last panel repeat the panel's last and are set to zero
    Acc<T> y[4];
    T off[6][4], dia[4][4], tri[4][4];
    const int oc = min(o, F - 1);
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = b * SB + mfma_row<T>(g, r), kk = min(m, w - 1);
            y[b][r] = rows ? A[(size_t)(c + kk) * F + oc] : A[(size_t)oc * F + c + kk];
            dia[b][r] = inv[m * SB + n];
            // M_bb itself: U11's sub-block transposed, or L11's with its unit diagonal
            const int i = min(b * SB + n, w - 1);
            const T e = rows ? A[(size_t)(c + i) * F + c + kk] : A[(size_t)(c + kk) * F + c + i];
            tri[b][r] = m < b * SB + n || (rows && m == b * SB + n) ? e : m == b * SB + n ? (T)1 : (T)0;
        }
#pragma unroll
    for (int b = 1, e = 0; b < 4; b++)
#pragma unroll
        for (int q = 0; q < b; q++, e++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = min(b * SB + n, w - 1), kk = min(q * SB + mfma_row<T>(g, r), w - 1);
                off[e][r] = rows ? A[(size_t)(c + m) * F + c + kk] : A[(size_t)(c + kk) * F + c + m];
            }
    if (w < NB) {
#pragma unroll
        for (int b = 0, e = 0; b < 4; b++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                y[b][r] = b * SB + mfma_row<T>(g, r) < w ? y[b][r] : (T)0;
                dia[b][r] = b * SB < w ? dia[b][r] : (T)0;
                tri[b][r] = b * SB + n < w && b * SB + mfma_row<T>(g, r) < w ? tri[b][r] : (T)0;
            }
#pragma unroll
            for (int q = 0; q < b; q++, e++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    off[e][r] = b * SB + n < w && q * SB + mfma_row<T>(g, r) < w ? off[e][r] : (T)0;
        }
    }
#pragma unroll
    for (int b = 0, e = 0; b < 4; b++) {
        Acc<T> t = y[b];
#pragma unroll
        for (int q = 0; q < b; q++, e++)
#pragma unroll
            for (int r = 0; r < 4; r++) t = mfma(-off[e][r], y[q][r], t);
        Acc<T> x = {0, 0, 0, 0};
#pragma unroll
        for (int r = 0; r < 4; r++) x = mfma(dia[b][r], t[r], x);
#pragma unroll
        for (int r = 0; r < 4; r++) t = mfma(-tri[b][r], x[r], t);
#pragma unroll
        for (int r = 0; r < 4; r++) x = mfma(dia[b][r], t[r], x);
        y[b] = x;
    }
    if (o < F) {
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int kk = b * SB + mfma_row<T>(g, r);
                if (kk < w) (rows ? A[(size_t)(c + kk) * F + o] : A[(size_t)o * F + c + kk]) = y[b][r];
            }
    }
}

// Large fronts, trailing update of panel [c, c + w): A22 -= L21 U12 in 64 x 64 tiles, a quarter per wavefront, K = 64
// in one go: all operands are loaded straight into the matrix cores' registers (group g takes k = 16 g .. 16 g + 15,
// contiguous in U12) before the first product.  The workgroup of tile (0, 0) then factors the next panel's diagonal
// block while the others work.  grid.x: tiles of the largest trailing block of the launch, grid.y: the front.
// The 4 x 4-per-thread vector version through LDS took 18 us (FP64, trailing blocks of up to 446) and 40 us (FP32,
// up to 4,176) a panel, besides the diagonal block's own launch (28 and 31 us); this takes 15 and 29 us with the next
// diagonal block in it.  The 200 x 200 grid's factorisation: FP32 12.7 -> 4.1 ms, FP64 15.5 -> 5.7 ms.
// The products are summed from zero and subtracted once: added one by one to an entry that they are small against, as
// to the diagonal of a network's matrix, each would round off in it (nearly singular networks of 300 nodes came out with
// 7e-13 relative error in FP64, this way with 1.6e-13).  FP64 keeps two wavefronts a SIMD without accumulation
// registers, whose moves took 2 % (200 x 200 grid); FP32 is 5 % slower with four instead of three.
template <typename T>
__global__ void __launch_bounds__(TPB, sizeof(T) == 8 ? 2 : 1) k_update_big(const FrontD* __restrict__ fr, int panel,
                                                    T* __restrict__ pool, T* __restrict__ invs, int* flags) {
    __shared__ T D[NB * DLD], rp[NB];
    const FrontD S = fr[blockIdx.y];
    const int k = S.k, F = S.F;
    const int c = panel * NB;
    if (c >= k) return;
    const int w = min(NB, k - c);
    const int r0 = c + w, rest = F - r0;
    const int tiles = (rest + NB - 1) / NB;
    if ((int)blockIdx.x >= tiles * tiles) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int i0 = r0 + (blockIdx.x % tiles) * NB + (wave & 1) * 32, j0 = r0 + (blockIdx.x / tiles) * NB + (wave >> 1) * 32;
    T* A = pool + S.fo;
    Acc<T> acc[2][2], at[2][2];
    T a[2][SB], b[2][SB];
    const bool full = i0 + 32 <= F && j0 + 32 <= F;  // all of the quarter inside the front
#pragma unroll
    for (int u = 0; u < 2; u++) {  // no load under a mask, as in k_trsm
        const int i = min(i0 + SB * u + n, F - 1), j = min(j0 + SB * u + n, F - 1);
        const T* pb = A + (size_t)j * F + c;
        const T* pa = A + (size_t)c * F + i;
        if (w == NB) {
#pragma unroll
            for (int q = 0; q < SB; q++) {
                b[u][q] = pb[SB * g + q];
                a[u][q] = pa[(size_t)(SB * g + q) * F];
            }
        } else {
#pragma unroll
            for (int q = 0; q < SB; q++) {
                const int kk = SB * g + q, kc = min(kk, w - 1);
                b[u][q] = pb[kc];
                a[u][q] = pa[(size_t)kc * F];
                b[u][q] = kk < w ? b[u][q] : (T)0;
                a[u][q] = kk < w ? a[u][q] : (T)0;
            }
        }
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int v = 0; v < 2; v++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                at[u][v][r] = A[(size_t)min(j0 + SB * v + mfma_row<T>(g, r), F - 1) * F + min(i0 + SB * u + n, F - 1)];
    // the tile transposed (D's columns are the block's rows), so that its loads and stores run along columns
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int v = 0; v < 2; v++) acc[u][v] = Acc<T>{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < SB; q++)
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int v = 0; v < 2; v++) acc[u][v] = mfma(b[v][q], a[u][q], acc[u][v]);
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int v = 0; v < 2; v++) acc[u][v] = at[u][v] - acc[u][v];
    // the next diagonal block [r0, r0 + wn) is stored factored
    const int wn = blockIdx.x == 0 ? min(NB, k - r0) : 0;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int v = 0; v < 2; v++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = i0 + SB * u + n, j = j0 + SB * v + mfma_row<T>(g, r);
                if ((full || (i < F && j < F)) && (i >= r0 + wn || j >= r0 + wn)) A[(size_t)j * F + i] = acc[u][v][r];
            }
    if (wn <= 0) return;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int v = 0; v < 2; v++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = i0 - r0 + SB * u + n, j = j0 - r0 + SB * v + mfma_row<T>(g, r);
                D[i * DLD + j] = i < wn && j < wn ? acc[u][v][r] : i == j ? (T)1 : (T)0;
            }
    __syncthreads();
    diag_lu<T>(D, rp, wn, invs + ((size_t)S.p + panel + 1) * INV, flags);
    __syncthreads();
    for (int q = threadIdx.x; q < NB * NB; q += TPB) {
        const int i = q % NB, j = q / NB;
        if (i < wn && j < wn) A[(size_t)(r0 + j) * F + r0 + i] = D[i * DLD + j];
    }
}

// ---------------------------------------------------------------------------------------------------
// Sweeps: fronts of a level per launch.  b is the internal right-hand side, which the sweeps only read; y becomes the
// forward solution, then the backward one; wbuf holds each front's sweep vector.  A row of a front starts from its own
// right-hand side and its children's updates, listed per row in child order (g_ptr, g_idx over the sweep vectors).
// Nothing orders the workgroups of a launch, and several of one front read the same right-hand side while one of them
// stores the solution: the two may not share an array.
// ---------------------------------------------------------------------------------------------------
template <typename T>
__device__ inline T sweep_start(const FrontD& S, int i, const int* __restrict__ g_ptr, const int* __restrict__ g_idx,
                                const T* __restrict__ b, const T* wbuf) {
    T acc = i < S.k ? b[S.f + i] : (T)0;
    const int e1 = g_ptr[S.w + i + 1];
    for (int e = g_ptr[S.w + i]; e < e1; e++) acc += wbuf[g_idx[e]];
    return acc;
}

// A front of at most 64 rows in one wavefront, lane = row, its value in a register; larger small fronts a thread per
// row, the vector in LDS.  A thread loads its entries of the next eight pivots' columns at once.
template <typename T, int NT>
__global__ void __launch_bounds__(NT) k_forward(const FrontD* __restrict__ fr, const int* __restrict__ g_ptr,
                                                const int* __restrict__ g_idx, const T* __restrict__ pool,
                                                const T* __restrict__ b, T* __restrict__ y, T* __restrict__ wbuf) {
    __shared__ T xs[NT];
    const FrontD S = fr[blockIdx.x];
    const int k = S.k, F = S.F, tid = threadIdx.x;
    const T* A = pool + S.fo;
    T x = tid < F ? sweep_start(S, tid, g_ptr, g_idx, b, wbuf) : (T)0;
    for (int j0 = 0; j0 < k; j0 += 8) {
        T a[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int j = j0 + u;
            a[u] = (j < k && tid > j && tid < F) ? A[(size_t)j * F + tid] : (T)0;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int j = j0 + u;
            if (j < k) {
                T xj;
                if (NT == 64) {
                    xj = lane_value(x, j);
                } else {
                    if (tid == j) xs[j] = x;
                    __syncthreads();
                    xj = xs[j];
                }
                if (tid > j && tid < F) x = x - a[u] * xj;
            }
        }
    }
    if (tid < k) y[S.f + tid] = x;
    if (tid >= k && tid < F) wbuf[S.w + tid] = x;
}

template <typename T, int NT>
__global__ void __launch_bounds__(NT) k_backward(const FrontD* __restrict__ fr, const int* __restrict__ r_idx,
                                                 const T* __restrict__ pool, T* __restrict__ y) {
    __shared__ T xs[NT];
    const FrontD S = fr[blockIdx.x];
    const int k = S.k, F = S.F, tid = threadIdx.x;
    const T* A = pool + S.fo;
    const int* R = r_idx + S.r;
    // x = y - U12 x_R (the ancestors' solution is final)
    T x = tid < k ? y[S.f + tid] : (T)0;
    if (NT == 64 && k <= 8) {  // few pivots: a column per lane, the rows' products summed across the wavefront
        const bool own = tid >= k && tid < F;
        const T yv = own ? y[R[tid - k]] : (T)0;
        T a[8];
#pragma unroll
        for (int j = 0; j < 8; j++) a[j] = own && j < k ? A[(size_t)tid * F + j] * yv : (T)0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (j >= k) break;
            T v = a[j];
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
            if (tid == j) x = x - v;
        }
    } else if (tid < k) {  // a row per thread, sixteen columns' loads in flight, subtracted in column order
        int c = k;
        for (; c + 15 < F; c += 16) {
            int ri[16];
            T a[16], yv[16];
#pragma unroll
            for (int u = 0; u < 16; u++) {
                ri[u] = R[c + u - k];
                a[u] = A[(size_t)(c + u) * F + tid];
            }
#pragma unroll
            for (int u = 0; u < 16; u++) yv[u] = y[ri[u]];
#pragma unroll
            for (int u = 0; u < 16; u++) x = x - a[u] * yv[u];
        }
        for (; c < F; c++) x = x - A[(size_t)c * F + tid] * y[R[c - k]];
    }
    for (int j0 = k - 1; j0 >= 0; j0 -= 8) {  // thread j loads the pivot itself
        T a[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int j = j0 - u;
            a[u] = (j >= 0 && tid <= j) ? A[(size_t)j * F + tid] : (T)1;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int j = j0 - u;
            if (j >= 0) {
                if (tid == j) x = x / a[u];
                T xj;
                if (NT == 64) {
                    xj = lane_value(x, j);
                } else {
                    if (tid == j) xs[j] = x;
                    __syncthreads();
                    xj = xs[j];
                }
                if (tid < j) x = x - a[u] * xj;
            }
        }
    }
    if (tid < k) y[S.f + tid] = x;
}

// Sweeps of large fronts, the fronts of a level per launch (grid.y), WP pivots at a time.
// Forward: every block solves L11 x = w[c, c + w) (unit lower) for itself, thread = row, 32 columns at a time: the
// wavefront that holds them passes each x_j from its lane through the scalar unit, the rows below take the 32 from
// LDS.  Block 0 stores x in y; every block then updates its 256 rows below: w_i -= L(i, c..c+w) x.  The next 32 columns'
// entries are always on their way.  The first launch of a front starts its sweep vector (sweep_start) in place.
// A launch of its own per 64 pivots and one for the start cost 8.0 us and 3.6 us each, of which the kernel's own
// start and its first loads are half: 36 us for 256 pivots against 20 us now (200 x 200 grid, FP32).
constexpr int WP = TPB;   // pivots per launch
constexpr int WC = 32;    // columns whose entries a thread holds at once
template <typename T>
__global__ void __launch_bounds__(TPB) k_fwd_panel(const FrontD* __restrict__ fr, int panel, const int* __restrict__ g_ptr,
                                                   const int* __restrict__ g_idx, const T* __restrict__ pool,
                                                   const T* __restrict__ rhs, T* __restrict__ y, T* wbuf) {
    __shared__ T xs[WP];
    const FrontD S = fr[blockIdx.y];
    const int k = S.k, F = S.F;
    const int c = panel * WP;
    if (c >= k) return;
    const int w = min(WP, k - c), r0 = c + w;
    if ((int)blockIdx.x > 0 && (int)blockIdx.x * TPB >= F - r0) return;
    const T* A = pool + S.fo + (int64_t)c * F;  // the panel's columns
    T* wv = wbuf + S.w;
    const int tid = threadIdx.x, wave = tid >> 6;
    const int i = r0 + blockIdx.x * TPB + tid;
    T a[WC], b[WC];
    // Column q of the panel at `row`; columns past the panel repeat the last (their x are zero), rows past the front
    // the last row (never stored), so that no load is under a mask.
    auto load = [&](T (&v)[WC], int q0, int row) {
#pragma unroll
        for (int u = 0; u < WC; u++) v[u] = A[(int64_t)min(q0 + u, w - 1) * F + row];
    };
    auto start = [&](int row) { return panel == 0 ? sweep_start(S, row, g_ptr, g_idx, rhs, wbuf) : wv[row]; };
    const int own = c + min(tid, w - 1), below = min(i, F - 1);
    load(a, 0, own);
    load(b, 0, below);
    T x = tid < w ? start(own) : (T)0, acc = start(below);
    xs[tid] = (T)0;
    __syncthreads();
    for (int q0 = 0; q0 < w; q0 += WC) {
        T n[WC];
        load(n, q0 + WC, own);
#pragma unroll
        for (int u = 0; u < WC; u++) a[u] = tid > q0 + u && tid < w ? -a[u] : (T)0;  // L11 below the diagonal
        if (wave == q0 >> 6) {
#pragma unroll
            for (int u = 0; u < WC; u++) x = fma(a[u], lane_value(x, (q0 & 63) + u), x);
            if (tid >= q0 && tid < q0 + WC) xs[tid] = x;
        }
        __syncthreads();
        if (wave > q0 >> 6)
#pragma unroll
            for (int u = 0; u < WC; u++) x = fma(a[u], xs[q0 + u], x);
#pragma unroll
        for (int u = 0; u < WC; u++) a[u] = n[u];
    }
    if (blockIdx.x == 0 && tid < w) y[S.f + c + tid] = x;
    if ((int)blockIdx.x * TPB >= F - r0) return;
    for (int q0 = 0; q0 < w; q0 += WC) {
        T n[WC];
        load(n, q0 + WC, below);
#pragma unroll
        for (int u = 0; u < WC; u++) acc = fma(-b[u], xs[q0 + u], acc);
#pragma unroll
        for (int u = 0; u < WC; u++) b[u] = n[u];
    }
    if (i < F) wv[i] = acc;
}

// Backward of large fronts: w_j = y_j - U12(j, :) x_R for the front's pivots.  A block of 1024 threads
// takes 64 pivots (grid.x): lane = pivot, its 16 wavefronts stride over the columns of R, and the 16
// partial sums are added in wavefront order.
template <typename T>
__global__ void __launch_bounds__(1024) k_bwd_init(const FrontD* __restrict__ fr, const int* __restrict__ r_idx,
                                                   const T* __restrict__ pool, const T* __restrict__ y,
                                                   T* __restrict__ wbuf) {
    __shared__ T part[16][64];
    const FrontD S = fr[blockIdx.y];
    const int k = S.k, F = S.F;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + lane;
    if ((int)blockIdx.x * 64 >= k) return;
    const T* A = pool + S.fo;
    const int* R = r_idx + S.r;
    T acc = (T)0;
    if (j < k) {
        int c = k + wv;
        for (; c + 16 * 7 < F; c += 16 * 8) {  // eight columns' loads in flight, added in column order
            int ri[8];
            T a[8], yv[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                ri[u] = R[c + 16 * u - k];
                a[u] = A[(size_t)(c + 16 * u) * F + j];
            }
#pragma unroll
            for (int u = 0; u < 8; u++) yv[u] = y[ri[u]];
#pragma unroll
            for (int u = 0; u < 8; u++) acc = acc + a[u] * yv[u];
        }
        for (; c < F; c += 16) acc = acc + A[(size_t)c * F + j] * y[R[c - k]];
    }
    part[wv][lane] = acc;
    __syncthreads();
    if (wv == 0 && j < k) {
        T sum = part[0][lane];
        for (int q = 1; q < 16; q++) sum = sum + part[q][lane];
        wbuf[S.w + j] = y[S.f + j] - sum;
    }
}

// Backward panel [c, c + w), panels from the last: U11 x = w[c, c + w) by every block (as forward, the columns from the
// last; a row's pivot divides as a reciprocal, all of which are taken at once), block 0 stores x in y, every block
// updates its rows above: w_i -= U(i, c..c+w) x.
template <typename T>
__global__ void __launch_bounds__(TPB) k_bwd_panel(const FrontD* __restrict__ fr, int panel, const T* __restrict__ pool,
                                                   T* __restrict__ y, T* __restrict__ wbuf) {
    __shared__ T xs[WP];
    const FrontD S = fr[blockIdx.y];
    const int k = S.k, F = S.F;
    const int c = panel * WP;
    if (c >= k) return;
    const int w = min(WP, k - c);
    if ((int)blockIdx.x > 0 && (int)blockIdx.x * TPB >= c) return;
    const T* A = pool + S.fo + (int64_t)c * F;
    T* wv = wbuf + S.w;
    const int tid = threadIdx.x, wave = tid >> 6;
    const int i = blockIdx.x * TPB + tid;
    T a[WC], b[WC];
    auto load = [&](T (&v)[WC], int q0, int row) {  // as forward
#pragma unroll
        for (int u = 0; u < WC; u++) v[u] = A[(int64_t)min(max(q0 + u, 0), w - 1) * F + row];
    };
    const int last = (w - 1) / WC * WC, own = c + min(tid, w - 1), above = min(i, max(c - 1, 0));
    load(a, last, own);
    load(b, last, above);
    const T rd = (T)1 / A[(int64_t)min(tid, w - 1) * F + own];
    T x = tid < w ? wv[own] : (T)0, acc = wv[above];
    xs[tid] = (T)0;
    __syncthreads();
    for (int q0 = last; q0 >= 0; q0 -= WC) {
        T n[WC];
        load(n, q0 - WC, own);
#pragma unroll
        for (int u = 0; u < WC; u++) a[u] = tid < q0 + u && q0 + u < w ? -a[u] : (T)0;  // U11 above the diagonal
        if (wave == q0 >> 6) {
            T z = x * rd;  // each lane's solution once its row is done
#pragma unroll
            for (int u = WC - 1; u >= 0; u--) {
                x = fma(a[u], lane_value(z, (q0 & 63) + u), x);
                z = x * rd;
            }
            if (tid >= q0 && tid < q0 + WC) xs[tid] = x = z;
        }
        __syncthreads();
        if (wave < q0 >> 6)
#pragma unroll
            for (int u = WC - 1; u >= 0; u--) x = fma(a[u], xs[q0 + u], x);
#pragma unroll
        for (int u = 0; u < WC; u++) a[u] = n[u];
    }
    if (blockIdx.x == 0 && tid < w) y[S.f + c + tid] = x;
    if ((int)blockIdx.x * TPB >= c) return;
    for (int q0 = last; q0 >= 0; q0 -= WC) {
        T n[WC];
        load(n, q0 - WC, above);
#pragma unroll
        for (int u = WC - 1; u >= 0; u--) acc = fma(-b[u], xs[q0 + u], acc);
#pragma unroll
        for (int u = 0; u < WC; u++) b[u] = n[u];
    }
    if (i < c) wv[i] = acc;
}

// internal right-hand side from the FP64 residual (rows in pivot order), and dx back in external order
template <typename T>
__global__ void k_permute_in(int n, const int* __restrict__ prow, const double* __restrict__ res, T* __restrict__ b) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a < n) b[a] = (T)res[prow[a]];
}
template <typename T>
__global__ void k_permute_out(int n, const int* __restrict__ perm, const T* __restrict__ y, double* __restrict__ dx) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < n) dx[perm[b]] = (double)y[b];
}

// max |dx| over the non-NaN entries (the reference's fold with f64::max), as ordered bit patterns;
// *nonfinite = 1 when some entry is NaN or infinite
__global__ void k_maxabs(int n, const double* __restrict__ dx, unsigned long long* out, int* nonfinite) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (i < n) {
        const double a = fabs(dx[i]);
        if (a == a) v = a;
        if (!(a <= 1.7976931348623157e308)) atomicOr(nonfinite, 1);
    }
    for (int o = 32; o > 0; o >>= 1) {
        const double u = __shfl_xor(v, o, 64);
        v = u > v ? u : v;
    }
    if ((threadIdx.x & 63) == 0 && v > 0.0) atomicMax(out, (unsigned long long)__double_as_longlong(v));
}
// clamp and update (analysis.rs:196-207); flags[0] |= 4 when some |dx| > reltol after the clamp.  A
// solve with reused factors whose dx is not finite is discarded whole (x unchanged, not converged): the
// iteration is repeated with fresh factors.
__global__ void k_update(int n, const double* __restrict__ dx, const unsigned long long* mxbits, double reltol,
                         double* __restrict__ x, int* flags, int reused, const int* __restrict__ nonfinite) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (reused && *nonfinite) {
        if (i == 0) atomicOr(flags, 4);
        return;
    }
    const double mx = __longlong_as_double((long long)*mxbits);
    double d = dx[i];
    if (mx > 1.0) d = d * 1.0 / mx;
    if (fabs(d) > reltol) atomicOr(flags, 4);
    x[i] = x[i] + d;
}

// commit (comps/*: guess -> op) at the accepted solution
__global__ void k_commit(EvalArgs E, double* c_q) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < E.n_m1) {
        if (!E.m1_caps[t]) return;
        for (int f = 0; f < M1S; f++) E.m1_state[(size_t)f * E.n_m1 + t] = E.m1_state[(size_t)(M1S + f) * E.n_m1 + t];
        for (int f = 0; f < 2; f++) E.m1_icur[(size_t)f * E.n_m1 + t] = E.m1_icur[(size_t)(2 + f) * E.n_m1 + t];
        return;
    }
    if (t < E.n_m1 + E.n_d) {
        const int j = t - E.n_m1;
        E.d_state[2 * E.n_d + j] = E.d_state[1 * E.n_d + j];
        E.d_icur[j] = E.d_icur[E.n_d + j];
        return;
    }
    if (t < E.n_m1 + E.n_d + E.n_lin) {
        const int j = t - E.n_m1 - E.n_d;
        if (E.l_type[j] != S21_COMP_C) return;
        const int* nd = E.l_node + 3 * j;
        c_q[j] = E.l_val[j] * (xval(E.x, nd[0]) - xval(E.x, nd[1]));  // guess.q = c * vd
        E.c_icur[j] = E.c_icur[E.n_lin + j];
    }
}

// Local truncation error of a trapezoidal step from the third divided difference DD3 of the node voltages
// over the last four accepted points (x, h1, h2, h3 at t0 > t1 > t2 > t3): the error is dt^3 / 12 times the
// third derivative, which is about 6 DD3.  *rmax = max over voltage unknowns of that error over
// trtol (reltol max(|x|, |h1|) + abstol).
__global__ void k_lte(int n, const int* __restrict__ kind, const double* __restrict__ x, const double* __restrict__ h1,
                      const double* __restrict__ h2, const double* __restrict__ h3, double t0, double t1, double t2,
                      double t3, double reltol, double abstol, double trtol, unsigned long long* rmax) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double r = 0.0;
    if (i < n && kind[i] == S21_VAR_V) {
        const double d01 = (x[i] - h1[i]) / (t0 - t1), d12 = (h1[i] - h2[i]) / (t1 - t2),
                     d23 = (h2[i] - h3[i]) / (t2 - t3);
        const double d012 = (d01 - d12) / (t0 - t2), d123 = (d12 - d23) / (t1 - t3);
        const double d3 = (d012 - d123) / (t0 - t3);
        const double dt = t0 - t1;
        const double lte = dt * dt * dt / 2.0 * fabs(d3);
        const double tol = trtol * (reltol * fmax(fabs(x[i]), fabs(h1[i])) + abstol);
        r = lte / tol;
        if (!(r == r)) r = 1e300;
    }
    for (int o = 32; o > 0; o >>= 1) {
        const double u = __shfl_xor(r, o, 64);
        r = u > r ? u : r;
    }
    if ((threadIdx.x & 63) == 0 && r > 0.0) atomicMax(rmax, (unsigned long long)__double_as_longlong(r));
}

// out = a + w (b - a): an output-grid point between two accepted points
__global__ void k_interp(int n, const double* __restrict__ a, const double* __restrict__ b, double w,
                         double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = a[i] + w * (b[i] - a[i]);
}

}  // namespace lg
}  // namespace s21

// ===================================================================================================
// Host runtime
// ===================================================================================================
namespace s21 {
namespace lg {

using Buf = DevMem;

template <typename V>
static void upload(Buf& b, const std::vector<V>& v) {
    b.alloc(std::max<size_t>(v.size(), 1) * sizeof(V));
    if (!v.empty()) LCHECK(hipMemcpy(b.p, v.data(), v.size() * sizeof(V), hipMemcpyHostToDevice));
}

// Launch lists of one elimination-tree level.
struct Level {
    int f0 = 0;                        // first front of the level's launch list: one-wavefront, one-workgroup, large
    int n_wave = 0, n_group = 0, n_big = 0;
    size_t lds_wave = 0, lds_group = 0;  // LDS bytes of the first two kinds' factorisation
    int job0 = 0, n_job = 0;           // range in the large-front assembly jobs
    int panels = 0;                    // most panels of a large front of the level
    int k_big = 0;                     // most pivots of a large front of the level
};

}  // namespace lg
}  // namespace s21

struct s21_large {
    // the netlist
    int n_vars = 0;
    std::vector<std::string> names;
    std::vector<int> kinds;
    std::vector<s21_comp> comps;
    std::vector<s21_params> mos1_models, mos1_insts, diode_models, diode_insts, bsim4_models, bsim4_insts;
    s21_options opts;
    int precision = S21_FP64;
    int device = 0;
    double relax = 0.1;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // the structure of the last analysis
    std::string prepared;
    s21::Topology t;
    s21::LargeSym S;
    int n_m1 = 0, n_d = 0, n_lin = 0, n_b4 = 0, n_cells = 0, n_elem = 0;
    std::vector<s21::lg::Level> levels;
    std::vector<s21::lg::FrontD> fronts;  // launch lists (host copy)
    int reuse = -1;             // factor reuse: 1 on, 0 off (factor every iteration), -1 = on in mixed precision
    bool has_bsim4 = false;     // BSIM4 devices present: no factor reuse
    bool have_factors = false;  // the pool holds factors of this structure
    int reused = 0;             // iterations since the last factorisation
    s21::lg::Buf m1_node, m1_par, m1_caps, m1_state, m1_cb, d_node, d_par, d_state, d_cb, l_node, l_type, l_val, c_q,
        l_cb, cv, g_ptr, g_idx, slots, r_ptr, r_elem, e_col, x, res, dx, flags, mxbits;
    s21::lg::Buf f_fr, f_child, f_map, f_ridx, f_aelem, f_aoff, f_job, f_piece, f_gptr, f_gidx, inv;
    s21::lg::Buf perm, prow, pool, bv, yv, wv;
    s21::lg::Buf wave;
    s21::lg::Buf b4_node, b4_par, b4_st, b4_cb;
    // trapezoidal integration: per-charge currents, unknown kinds, accepted-point history
    s21::lg::Buf m1_icur, d_icur, c_icur, kinds_dev, hist[4];
    int trap = 0;
    int64_t accepted = 0, rejected = 0;
    // results
    int status = S21_OK;
    int64_t iters = 0, npts = 0, factorisations = 0;
    std::vector<double> axis;
    double ms_total = 0, ms_factor = 0, ms_solve = 0, ms_eval = 0;
    ~s21_large() {
        if (ev0) (void)hipEventDestroy(ev0);
        if (ev1) (void)hipEventDestroy(ev1);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace s21 {
namespace lg {

inline int64_t ekey(int r, int c, int n) { return (int64_t)r * (int64_t)(n + 1) + c; }

// Stamp entries of one component and the slot each reaches: a matrix element, n_elem + row for an RHS
// entry, or -1 (ground, or an entry the analysis never stamps).
static int entry_targets(const Comp& c, const std::unordered_map<int64_t, int>& elem, int n, int n_elem, int* tgt) {
    const int* nd = c.node;
    auto M = [&](int r, int col) -> int {
        if (r < 0 || col < 0) return -1;
        return elem.at(ekey(r, col, n));
    };
    auto B = [&](int r) { return r < 0 ? -1 : n_elem + r; };
    switch (c.type) {
    case S21_COMP_MOS1:
        for (int e = 0; e < MOS1_NE; e++) {
            const int r = nd[mos1_entry_row(e)];
            tgt[e] = mos1_entry_col(e) < 0 ? B(r) : M(r, nd[mos1_entry_col(e)]);
        }
        return MOS1_NE;
    case S21_COMP_DIODE:
        for (int e = 0; e < DIODE_NE; e++) {
            const int r = nd[diode_entry_row(e)];
            tgt[e] = diode_entry_col(e) < 0 ? B(r) : M(r, nd[diode_entry_col(e)]);
        }
        return DIODE_NE;
    case S21_COMP_R:
    case S21_COMP_C:
        tgt[0] = M(nd[0], nd[0]);
        tgt[1] = M(nd[1], nd[1]);
        tgt[2] = M(nd[0], nd[1]);
        tgt[3] = M(nd[1], nd[0]);
        if (c.type == S21_COMP_R) return R_NE;
        tgt[4] = B(nd[0]);
        tgt[5] = B(nd[1]);
        return C_NE;
    case S21_COMP_V:
        tgt[0] = M(nd[0], nd[2]);
        tgt[1] = M(nd[2], nd[0]);
        tgt[2] = M(nd[1], nd[2]);
        tgt[3] = M(nd[2], nd[1]);
        tgt[4] = B(nd[2]);
        return V_NE;
    case S21_COMP_I:
        tgt[0] = B(nd[0]);
        tgt[1] = B(nd[1]);
        return I_NE;
    case S21_COMP_BSIM4:
        for (int k = 0; k < b4::B4_NS; k++) {
            const int r = nd[b4::b4_row(k)];
            tgt[k] = b4::b4_col(k) < 0 ? B(r) : M(r, nd[b4::b4_col(k)]);
        }
        return b4::B4_NS;
    default: fail(S21_INVALID, "the large-instance path takes R, C, V, I, Mos1, Diode and BSIM4 components");
    }
}

template <typename T>
static void set_lds_limits() {
    LCHECK(hipFuncSetAttribute((const void*)k_small<T, 64>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)SMALL_LDS));
    LCHECK(hipFuncSetAttribute((const void*)k_small<T, TPB>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)SMALL_LDS));
}

static EvalArgs eval_args(const s21_large* L, bool tran, double dt) {
    EvalArgs E;
    E.n_m1 = L->n_m1;
    E.n_d = L->n_d;
    E.n_lin = L->n_lin;
    E.tran = tran ? 1 : 0;
    E.gmin = L->opts.gmin;
    E.dt = dt;
    E.x = L->x.as<double>();
    E.m1_node = L->m1_node.as<int>();
    E.m1_par = L->m1_par.as<double>();
    E.m1_caps = L->m1_caps.as<int>();
    E.m1_state = L->m1_state.as<double>();
    E.m1_cb = L->m1_cb.as<int>();
    E.d_node = L->d_node.as<int>();
    E.d_par = L->d_par.as<double>();
    E.d_state = L->d_state.as<double>();
    E.d_cb = L->d_cb.as<int>();
    E.l_node = L->l_node.as<int>();
    E.l_type = L->l_type.as<int>();
    E.l_val = L->l_val.as<double>();
    E.c_q = L->c_q.as<double>();
    E.l_cb = L->l_cb.as<int>();
    E.cv = L->cv.as<double>();
    E.trap = L->trap;
    E.m1_icur = L->m1_icur.as<double>();
    E.d_icur = L->d_icur.as<double>();
    E.c_icur = L->c_icur.as<double>();
    return E;
}

// The structure of one analysis: components (IC forcing for a transient), derived parameters, the
// symbolic phase on the first iteration's matrix, gather lists and front maps, all uploaded.
static void prepare(s21_large* L, const s21_tran_options* tr) {
    Topology& t = L->t;
    t = Topology();
    build_comps(L->n_vars, L->names, L->kinds, L->comps, (int)L->mos1_models.size(), (int)L->mos1_insts.size(),
                (int)L->diode_models.size(), (int)L->diode_insts.size(), tr, t);
    topo_elements(t);
    const int n = t.n;
    const int ne = (int)t.erow.size();
    L->n_elem = ne;
    const bool tran = tr != nullptr;
    // devices by class, in component order; derived parameters
    HostInstance h0;
    std::vector<int> m1_node, d_node, l_node, l_type, m1_caps;
    std::vector<double> m1p, dpar, lval0, lval1;
    std::vector<int> m1_comp, d_comp, l_comp, b4_comp, b4_node;
    for (size_t ci = 0; ci < t.comps.size(); ci++) {
        const Comp& c = t.comps[ci];
        if (c.type == S21_COMP_BSIM4) {
            if (c.model < 0 || c.model >= (int)L->bsim4_models.size() || c.inst < 0 ||
                c.inst >= (int)L->bsim4_insts.size())
                fail(S21_ERR, "Parameters not defined");
            try {
                h0.b4.push_back(b4::derive_params(L->bsim4_models[c.model], L->bsim4_insts[c.inst]));
            } catch (const std::domain_error& e) {  // the reference panics here (bsim4inst.rs:200-223)
                fail(S21_ERR, e.what());
            }
            b4_comp.push_back((int)ci);
            for (int r = 0; r < 4; r++) b4_node.push_back(c.node[r]);
        } else if (c.type == S21_COMP_MOS1) {
            h0.m1.push_back(derive_mos1(L->mos1_models[c.model], L->mos1_insts[c.inst], L->opts));
            m1_comp.push_back((int)ci);
        } else if (c.type == S21_COMP_DIODE) {
            h0.dio.push_back(derive_diode(L->diode_models[c.model], L->diode_insts[c.inst], L->opts));
            d_comp.push_back((int)ci);
        } else if (c.type == S21_COMP_MOS0) {
            fail(S21_INVALID, "the large-instance path takes R, C, V, I, Mos1, Diode and BSIM4 components");
        } else {
            h0.lin_value.push_back(c.value);
            l_comp.push_back((int)ci);
        }
    }
    const int nm = (int)m1_comp.size(), nd = (int)d_comp.size(), nl = (int)l_comp.size(), nb4 = (int)b4_comp.size();
    L->n_b4 = nb4;
    L->n_m1 = nm;
    L->n_d = nd;
    L->n_lin = nl;
    m1p.assign((size_t)(M1F + M1C) * nm, 0.0);
    m1_caps.assign(nm, 0);
    for (int j = 0; j < nm; j++) {
        const Comp& c = t.comps[m1_comp[j]];
        for (int r = 0; r < 6; r++) m1_node.push_back(c.node[r]);
        const Mos1Derived& D = h0.m1[j];
        const double core[M1F] = {D.core.p,      D.core.vt0_t,  D.core.beta,   D.core.phi_t,
                                  D.core.gamma,  D.core.lambda, D.core.vtherm, D.core.isat_d,
                                  D.core.isat_s, D.core.grd,    D.core.grs};
        for (int f = 0; f < M1F; f++) m1p[(size_t)f * nm + j] = core[f];
        const double caps[M1C] = {D.caps.cox, D.caps.cgs_ov, D.caps.cgd_ov, D.caps.cgb_ov};
        for (int f = 0; f < M1C; f++) m1p[(size_t)(M1F + f) * nm + j] = caps[f];
        m1_caps[j] = D.has_caps && tran ? 1 : 0;
    }
    dpar.assign((size_t)DPF * nd, 0.0);
    for (int j = 0; j < nd; j++) {
        const Comp& c = t.comps[d_comp[j]];
        for (int r = 0; r < 3; r++) d_node.push_back(c.node[r]);
        const DiodeP& P = h0.dio[j];
        const double v[DPF] = {P.isat, P.vte, P.vcrit, P.gspr, P.bv, P.has_bv, P.cz,
                               P.cz2,  P.dep, P.f1,    P.f3,   P.tt, P.vj,     P.m};
        for (int f = 0; f < DPF; f++) dpar[(size_t)f * nd + j] = v[f];
    }
    lval0.resize(nl);
    lval1.resize(nl);
    for (int j = 0; j < nl; j++) {
        const Comp& c = t.comps[l_comp[j]];
        for (int r = 0; r < 3; r++) l_node.push_back(c.type == S21_COMP_V || r < 2 ? c.node[r] : -1);
        l_type.push_back(c.type);
        lval0[j] = c.value;
        lval1[j] = c.value_tran;
    }
    std::vector<double> lval(lval0);
    lval.insert(lval.end(), lval1.begin(), lval1.end());
    // contribution cells and the ordered gather lists (component order, then entry order)
    std::unordered_map<int64_t, int> elem;
    elem.reserve((size_t)ne * 2);
    for (int e = 0; e < ne; e++) elem[ekey(t.erow[e], t.ecol[e], n)] = e;
    std::vector<int> m1_cb(nm), d_cb(nd), l_cb(nl), b4_cb(nb4), comp_cb(t.comps.size(), -1);
    int cells = 0;
    for (int j = 0; j < nb4; j++) {
        b4_cb[j] = cells;
        comp_cb[b4_comp[j]] = cells;
        cells += b4::B4_NS;
    }
    for (int j = 0; j < nm; j++) {
        m1_cb[j] = cells;
        comp_cb[m1_comp[j]] = cells;
        cells += MOS1_NE;
    }
    for (int j = 0; j < nd; j++) {
        d_cb[j] = cells;
        comp_cb[d_comp[j]] = cells;
        cells += DIODE_NE;
    }
    for (int j = 0; j < nl; j++) {
        l_cb[j] = cells;
        comp_cb[l_comp[j]] = cells;
        cells += C_NE;  // the widest linear element
    }
    L->n_cells = cells;
    const int nslot = ne + n;
    std::vector<int> cnt(nslot + 1, 0);
    std::vector<std::pair<int, int>> contrib;  // (slot, cell) in component order
    int tg[b4::B4_NS > MOS1_NE ? b4::B4_NS : MOS1_NE];
    for (size_t ci = 0; ci < t.comps.size(); ci++) {
        const int k = entry_targets(t.comps[ci], elem, n, ne, tg);
        for (int e = 0; e < k; e++)
            if (tg[e] >= 0) contrib.push_back({tg[e], comp_cb[ci] + e});
    }
    for (auto& pc : contrib) cnt[pc.first + 1]++;
    for (int sl = 0; sl < nslot; sl++) cnt[sl + 1] += cnt[sl];
    std::vector<int> gidx(contrib.size()), fill(cnt.begin(), cnt.end() - 1);
    for (auto& pc : contrib) gidx[fill[pc.first]++] = pc.second;
    // residual rows: elements of each row in creation order
    std::vector<int> rptr(n + 1, 0), relem(ne);
    for (int e = 0; e < ne; e++) rptr[t.erow[e] + 1]++;
    for (int r = 0; r < n; r++) rptr[r + 1] += rptr[r];
    {
        std::vector<int> f2(rptr.begin(), rptr.end() - 1);
        for (int e = 0; e < ne; e++) relem[f2[t.erow[e]]++] = e;
    }
    // symbolic phase on the first Newton iteration's matrix (x = 0)
    std::vector<double> vals, rhs;
    host_assemble_op(t, h0, L->opts, std::vector<double>(n, 0.0), vals, rhs);
    large_symbolic(n, t.erow, t.ecol, &vals, L->S, L->relax);
    const LargeSym& S = L->S;
    // A's entries by front
    std::vector<int64_t> aptr(S.ns + 1, 0);
    std::vector<int> a_s(ne), a_loc(ne);
    for (int e = 0; e < ne; e++) {
        const int a = S.irow[t.erow[e]], b = S.icol[t.ecol[e]];
        const int lo = std::min(a, b);
        const int s = (int)(std::upper_bound(S.sn_first.begin(), S.sn_first.end(), lo) - S.sn_first.begin()) - 1;
        const int64_t o = large_entry_offset(S, a, b);
        if (o < 0) fail(S21_ERR, "matrix entry outside the symbolic structure");
        a_s[e] = s;
        a_loc[e] = (int)(o - S.front_off[s]);
        aptr[s + 1]++;
    }
    for (int s = 0; s < S.ns; s++) aptr[s + 1] += aptr[s];
    std::vector<int> aelem(ne), aoff(ne);
    {
        std::vector<int64_t> f2(aptr.begin(), aptr.end() - 1);
        for (int e = 0; e < ne; e++) {
            const int64_t q = f2[a_s[e]]++;
            aelem[q] = e;
            aoff[q] = a_loc[e];
        }
    }
    std::vector<int64_t> woff(S.ns + 1, 0);
    std::vector<int> Fs(S.ns), Ks(S.ns);
    for (int s = 0; s < S.ns; s++) {
        Ks[s] = S.sn_first[s + 1] - S.sn_first[s];
        Fs[s] = Ks[s] + (int)(S.r_ptr[s + 1] - S.r_ptr[s]);
        woff[s + 1] = woff[s] + Fs[s];
    }
    // children of each front in order, with their maps one after another; rows' contributions to the forward sweep
    std::vector<ChildD> child(S.child.size());
    std::vector<int> cmap, m0(S.ns + 1, 0), gptr((size_t)woff[S.ns] + 1, 0);
    if (woff[S.ns] >= (int64_t)1 << 31) fail(S21_INVALID, "circuit too large: sweep index");
    for (int s = 0; s < S.ns; s++) {
        m0[s] = (int)cmap.size();
        for (int c = S.child_ptr[s]; c < S.child_ptr[s + 1]; c++) {
            const int ch = S.child[c], mc = Fs[ch] - Ks[ch];
            child[c] = ChildD{S.front_off[ch] + (int64_t)Ks[ch] * Fs[ch] + Ks[ch], mc, Fs[ch], (int)cmap.size() - m0[s]};
            for (int q = 0; q < mc; q++) {
                const int at = S.ext_map[S.ext_ptr[ch] + q];
                cmap.push_back(at);
                gptr[woff[s] + at + 1]++;
            }
        }
    }
    m0[S.ns] = (int)cmap.size();
    for (int64_t q = 0; q < woff[S.ns]; q++) gptr[q + 1] += gptr[q];
    std::vector<int> gcontrib(cmap.size());
    {
        std::vector<int> at(gptr.begin(), gptr.end() - 1);
        for (int s = 0; s < S.ns; s++)
            for (int c = S.child_ptr[s]; c < S.child_ptr[s + 1]; c++) {
                const int ch = S.child[c];
                for (int q = 0; q < child[c].mc; q++)
                    gcontrib[at[woff[s] + cmap[m0[s] + child[c].map + q]]++] = (int)(woff[ch] + Ks[ch] + q);
            }
    }
    // level launch lists, and the assembly tiles of large fronts
    auto lds_of = [&](int s) {
        const size_t tsz = L->precision == S21_MIXED ? sizeof(float) : sizeof(double);
        return (size_t)Fs[s] * Fs[s] * tsz + (size_t)(m0[s + 1] - m0[s]) * sizeof(int);
    };
    auto kind = [&](int s) { return lds_of(s) > SMALL_LDS || Fs[s] > SMALL_MAX ? 2 : Fs[s] > WAVE_MAX ? 1 : 0; };
    std::vector<FrontD>& fr = L->fronts;
    fr.clear();
    std::vector<AsmJob> jobs;
    std::vector<AsmPiece> pieces;
    int panels = 0;
    L->levels.clear();
    for (size_t l = 0; l + 1 < S.lvl_ptr.size(); l++) {
        Level lv;
        lv.f0 = (int)fr.size();
        lv.job0 = (int)jobs.size();
        for (int want = 0; want < 3; want++)
            for (int q = S.lvl_ptr[l]; q < S.lvl_ptr[l + 1]; q++) {
                const int s = S.lvl_sn[q];
                if (kind(s) != want) continue;
                const int F = Fs[s], k = Ks[s];
                fr.push_back(FrontD{S.front_off[s], woff[s], S.r_ptr[s], k, F, S.sn_first[s], want == 2 ? panels : 0,
                                    S.child_ptr[s], S.child_ptr[s + 1], (int)aptr[s], (int)aptr[s + 1], m0[s], m0[s + 1]});
                if (want == 0) {
                    lv.n_wave++;
                    lv.lds_wave = std::max(lv.lds_wave, lds_of(s));
                    continue;
                }
                if (want == 1) {
                    lv.n_group++;
                    lv.lds_group = std::max(lv.lds_group, lds_of(s));
                    continue;
                }
                lv.n_big++;
                lv.panels = std::max(lv.panels, (k + NB - 1) / NB);
                lv.k_big = std::max(lv.k_big, k);
                panels += (k + NB - 1) / NB;
                // tiles row block by row block; A's entries sorted by tile, their offsets within it
                const int nr = (F + TPB - 1) / TPB, nc = (F + CB - 1) / CB, j0 = (int)jobs.size();
                std::vector<std::vector<std::pair<int, int>>> in_tile((size_t)nr * nc);  // (element, offset)
                for (int64_t e = aptr[s]; e < aptr[s + 1]; e++) {
                    const int col = aoff[e] / F, row = aoff[e] % F;
                    in_tile[(size_t)(row / TPB) * nc + col / CB].push_back({aelem[e], (col % CB) * TPB + row % TPB});
                }
                int at = (int)aptr[s];
                for (int r = 0; r < nr; r++)
                    for (int c = 0; c < nc; c++) {
                        AsmJob J{S.front_off[s], F, r * TPB, c * CB, 0, 0, at, at};
                        for (const auto& e : in_tile[(size_t)r * nc + c]) {
                            aelem[at] = e.first;
                            aoff[at++] = e.second;
                        }
                        J.a1 = at;
                        jobs.push_back(J);
                    }
                // a child's rows (and columns) of each tile are runs, its map being increasing
                std::vector<std::vector<AsmPiece>> in(in_tile.size());
                for (int c = S.child_ptr[s]; c < S.child_ptr[s + 1]; c++) {
                    const ChildD& C = child[c];
                    const int* mp = cmap.data() + m0[s] + C.map;
                    for (int i0 = 0; i0 < C.mc;) {
                        const int r = mp[i0] / TPB;
                        const int i1 = (int)(std::lower_bound(mp + i0, mp + C.mc, (r + 1) * TPB) - mp);
                        for (int c0 = 0; c0 < C.mc;) {
                            const int cb = mp[c0] / CB;
                            int c1 = c0;
                            while (c1 < C.mc && mp[c1] < (cb + 1) * CB) c1++;
                            in[(size_t)r * nc + cb].push_back(AsmPiece{C.u + (int64_t)c0 * C.Fc + i0, C.Fc, i1 - i0, c1 - c0,
                                                                       m0[s] + C.map + i0, m0[s] + C.map + c0});
                            c0 = c1;
                        }
                        i0 = i1;
                    }
                }
                for (size_t t2 = 0; t2 < in.size(); t2++) {
                    jobs[j0 + t2].p0 = (int)pieces.size();
                    pieces.insert(pieces.end(), in[t2].begin(), in[t2].end());
                    jobs[j0 + t2].p1 = (int)pieces.size();
                }
            }
        lv.n_job = (int)jobs.size() - lv.job0;
        L->levels.push_back(lv);
    }
    // upload
    upload(L->m1_node, m1_node);
    upload(L->m1_par, m1p);
    upload(L->m1_caps, m1_caps);
    upload(L->m1_cb, m1_cb);
    upload(L->d_node, d_node);
    upload(L->d_par, dpar);
    upload(L->d_cb, d_cb);
    upload(L->l_node, l_node);
    upload(L->l_type, l_type);
    upload(L->l_val, lval);
    upload(L->l_cb, l_cb);
    upload(L->b4_node, b4_node);
    {  // parameters field-major: field K of device j at [K][j]
        constexpr int D = (int)(sizeof(b4::B4Par) / sizeof(double));
        std::vector<double> par((size_t)D * nb4);
        for (int j = 0; j < nb4; j++)
            for (int k = 0; k < D; k++) par[(size_t)k * nb4 + j] = ((const double*)&h0.b4[j])[k];
        upload(L->b4_par, par);
    }
    upload(L->b4_cb, b4_cb);
    L->b4_st.alloc(std::max<size_t>((size_t)B4S_F * nb4, 1) * sizeof(double));
    L->m1_state.alloc(std::max<size_t>((size_t)2 * M1S * nm, 1) * sizeof(double));
    L->d_state.alloc(std::max<size_t>((size_t)DSF * nd, 1) * sizeof(double));
    L->c_q.alloc(std::max<size_t>(nl, 1) * sizeof(double));
    L->m1_icur.alloc(std::max<size_t>((size_t)4 * nm, 1) * sizeof(double));
    L->d_icur.alloc(std::max<size_t>((size_t)2 * nd, 1) * sizeof(double));
    L->c_icur.alloc(std::max<size_t>((size_t)2 * nl, 1) * sizeof(double));
    upload(L->kinds_dev, t.kinds);
    L->cv.alloc(std::max<size_t>(cells, 1) * sizeof(double));
    upload(L->g_ptr, cnt);
    upload(L->g_idx, gidx);
    L->slots.alloc((size_t)std::max(nslot, 1) * sizeof(double));
    upload(L->r_ptr, rptr);
    upload(L->r_elem, relem);
    upload(L->e_col, t.ecol);
    L->x.alloc((size_t)std::max(n, 1) * sizeof(double));
    L->res.alloc((size_t)std::max(n, 1) * sizeof(double));
    L->dx.alloc((size_t)std::max(n, 1) * sizeof(double));
    L->flags.alloc(8 * sizeof(int));  // 3 flags, the non-finite-dx flag, the residual's max |.| (8 bytes)
    L->mxbits.alloc(sizeof(unsigned long long));
    upload(L->f_fr, fr);
    upload(L->f_child, child);
    upload(L->f_map, cmap);
    upload(L->f_ridx, S.r_idx);
    upload(L->f_aelem, aelem);
    upload(L->f_aoff, aoff);
    upload(L->f_job, jobs);
    upload(L->f_piece, pieces);
    upload(L->f_gptr, gptr);
    upload(L->f_gidx, gcontrib);
    upload(L->perm, S.perm);
    upload(L->prow, S.prow);
    L->have_factors = false;
    const size_t tsz = L->precision == S21_MIXED ? sizeof(float) : sizeof(double);
    L->pool.alloc((size_t)std::max<int64_t>(S.pool, 1) * tsz);
    L->inv.alloc((size_t)std::max(panels, 1) * INV * tsz);
    L->bv.alloc((size_t)std::max(n, 1) * tsz);
    L->yv.alloc((size_t)std::max(n, 1) * tsz);
    L->wv.alloc((size_t)std::max<int64_t>(woff[S.ns], 1) * tsz);
    if (L->precision == S21_MIXED)
        set_lds_limits<float>();
    else
        set_lds_limits<double>();
}

static inline int blocks(int64_t n) { return (int)std::max<int64_t>((n + TPB - 1) / TPB, 1); }

template <typename T>
static void factor(s21_large* L) {
    const double* aval = L->slots.as<double>();
    T* pool = L->pool.as<T>();
    T* inv = L->inv.as<T>();
    int* flags = L->flags.as<int>();
    const FrontD* fr = L->f_fr.as<FrontD>();
    const ChildD* child = L->f_child.as<ChildD>();
    const int *cmap = L->f_map.as<int>(), *aelem = L->f_aelem.as<int>(), *aoff = L->f_aoff.as<int>();
    for (const Level& lv : L->levels) {
        if (lv.n_wave)
            hipLaunchKernelGGL((k_small<T, 64>), dim3(lv.n_wave), dim3(64), lv.lds_wave, L->stream, fr + lv.f0, child, cmap,
                               aelem, aoff, aval, pool, flags + 1);
        if (lv.n_group)
            hipLaunchKernelGGL((k_small<T, TPB>), dim3(lv.n_group), dim3(TPB), lv.lds_group, L->stream,
                               fr + lv.f0 + lv.n_wave, child, cmap, aelem, aoff, aval, pool, flags + 1);
        if (!lv.n_big) continue;
        const int b0 = lv.f0 + lv.n_wave + lv.n_group;
        const FrontD* big = fr + b0;
        hipLaunchKernelGGL(k_assemble<T>, dim3(lv.n_job), dim3(TPB), 0, L->stream, L->f_job.as<AsmJob>() + lv.job0,
                           L->f_piece.as<AsmPiece>(), cmap, aelem, aoff, aval, pool);
        hipLaunchKernelGGL(k_diag<T>, dim3(lv.n_big), dim3(TPB), 0, L->stream, big, pool, inv, flags + 1);
        for (int p = 0; p < lv.panels; p++) {
            int units = 0, tiles = 0;  // grid sizes for this panel: the largest over the level's large fronts
            for (int q = 0; q < lv.n_big; q++) {
                const FrontD& f = L->fronts[b0 + q];
                const int c = p * NB;
                if (c >= f.k) continue;
                const int w = std::min(NB, f.k - c), rest = f.F - c - w;
                units = std::max(units, 2 * ((rest + SB - 1) / SB));
                const int tl = (rest + NB - 1) / NB;
                tiles = std::max(tiles, tl * tl);
            }
            if (units > 0)
                hipLaunchKernelGGL(k_trsm<T>, dim3((units + 3) / 4, lv.n_big), dim3(TPB), 0, L->stream, big, p, pool, inv);
            if (tiles > 0)
                hipLaunchKernelGGL(k_update_big<T>, dim3(tiles, lv.n_big), dim3(TPB), 0, L->stream, big, p, pool, inv,
                                   flags + 1);
        }
    }
    LCHECK(hipGetLastError());
    L->factorisations++;
}

template <typename T>
static void solve(s21_large* L) {
    const int n = L->t.n;
    T* b = L->bv.as<T>();
    T* y = L->yv.as<T>();
    T* w = L->wv.as<T>();
    const T* pool = L->pool.as<T>();
    const FrontD* fr = L->f_fr.as<FrontD>();
    const int *gp = L->f_gptr.as<int>(), *gi = L->f_gidx.as<int>(), *ri = L->f_ridx.as<int>();
    hipLaunchKernelGGL(k_permute_in<T>, dim3(blocks(n)), dim3(TPB), 0, L->stream, n, L->prow.as<int>(),
                       L->res.as<double>(), b);
    for (const Level& lv : L->levels) {
        if (lv.n_wave)
            hipLaunchKernelGGL((k_forward<T, 64>), dim3(lv.n_wave), dim3(64), 0, L->stream, fr + lv.f0, gp, gi, pool, b, y,
                               w);
        if (lv.n_group)
            hipLaunchKernelGGL((k_forward<T, TPB>), dim3(lv.n_group), dim3(TPB), 0, L->stream, fr + lv.f0 + lv.n_wave, gp, gi,
                               pool, b, y, w);
        if (!lv.n_big) continue;
        const int b0 = lv.f0 + lv.n_wave + lv.n_group;
        for (int p = 0; p * WP < lv.k_big; p++) {
            int nb = 1;  // blocks of rows below the panel, the largest over the level's large fronts
            for (int q = 0; q < lv.n_big; q++) {
                const FrontD& f = L->fronts[b0 + q];
                if (p * WP < f.k) nb = std::max(nb, (f.F - std::min(f.k, (p + 1) * WP) + TPB - 1) / TPB);
            }
            hipLaunchKernelGGL(k_fwd_panel<T>, dim3(nb, lv.n_big), dim3(TPB), 0, L->stream, fr + b0, p, gp, gi, pool, b, y,
                               w);
        }
    }
    for (auto it = L->levels.rbegin(); it != L->levels.rend(); ++it) {
        const Level& lv = *it;
        if (lv.n_wave)
            hipLaunchKernelGGL((k_backward<T, 64>), dim3(lv.n_wave), dim3(64), 0, L->stream, fr + lv.f0, ri, pool, y);
        if (lv.n_group)
            hipLaunchKernelGGL((k_backward<T, TPB>), dim3(lv.n_group), dim3(TPB), 0, L->stream, fr + lv.f0 + lv.n_wave, ri,
                               pool, y);
        if (!lv.n_big) continue;
        const FrontD* big = fr + lv.f0 + lv.n_wave + lv.n_group;
        hipLaunchKernelGGL(k_bwd_init<T>, dim3((lv.k_big + 63) / 64, lv.n_big), dim3(1024), 0, L->stream, big, ri, pool, y, w);
        for (int p = (lv.k_big - 1) / WP; p >= 0; p--)
            hipLaunchKernelGGL(k_bwd_panel<T>, dim3(std::max(1, p), lv.n_big), dim3(TPB), 0, L->stream, big, p, pool, y, w);
    }
    hipLaunchKernelGGL(k_permute_out<T>, dim3(blocks(n)), dim3(TPB), 0, L->stream, n, L->perm.as<int>(), y,
                       L->dx.as<double>());
    LCHECK(hipGetLastError());
}

// Commit of every device's guess (Component::commit) at the accepted solution.
static void commit_state(s21_large* L, bool tran, double dt) {
    const EvalArgs E = eval_args(L, tran, dt);
    hipLaunchKernelGGL(k_commit, dim3(blocks(L->n_m1 + L->n_d + L->n_lin)), dim3(TPB), 0, L->stream, E,
                       L->c_q.as<double>());
    if (L->n_b4)
        hipLaunchKernelGGL(k_commit_b4, dim3(blocks(L->n_b4)), dim3(TPB), 0, L->stream, L->n_b4,
                           L->b4_st.as<double>());
    LCHECK(hipGetLastError());
}

// Evaluation, gather and residual at the current x; flags[0] set when the residual fails the test.
static void assemble_residual(s21_large* L, bool tran, double dt) {
    const int n = L->t.n, nslot = L->n_elem + n;
    const EvalArgs E = eval_args(L, tran, dt);
    hipLaunchKernelGGL(k_eval, dim3(blocks(L->n_m1 + L->n_d + L->n_lin)), dim3(TPB), 0, L->stream, E);
    if (L->n_b4) {
        B4Args A{L->n_b4,
                 tran ? 1 : 0,
                 L->opts.gmin,
                 dt,
                 L->x.as<double>(),
                 L->b4_node.as<int>(),
                 L->b4_par.as<double>(),
                 L->b4_st.as<double>(),
                 L->b4_cb.as<int>(),
                 L->cv.as<double>()};
        hipLaunchKernelGGL(k_eval_b4, dim3((L->n_b4 + 127) / 128), dim3(128), 0, L->stream, A);
    }
    hipLaunchKernelGGL(k_gather, dim3(blocks(nslot)), dim3(TPB), 0, L->stream, nslot, L->g_ptr.as<int>(),
                       L->g_idx.as<int>(), L->cv.as<double>(), L->slots.as<double>());
    LCHECK(hipMemsetAsync(L->flags.p, 0, sizeof(int), L->stream));
    LCHECK(hipMemsetAsync(L->flags.as<int>() + 4, 0, sizeof(unsigned long long), L->stream));
    hipLaunchKernelGGL(k_residual, dim3(blocks(n)), dim3(TPB), 0, L->stream, n, L->r_ptr.as<int>(),
                       L->r_elem.as<int>(), L->e_col.as<int>(), L->slots.as<double>(),
                       L->slots.as<double>() + L->n_elem, L->x.as<double>(), L->res.as<double>(), L->opts.iabstol,
                       L->flags.as<int>(), (unsigned long long*)(L->flags.as<int>() + 4));
    LCHECK(hipGetLastError());
}

// One Newton solve (Solver::solve, analysis.rs:169-210) from the current x.  Every iteration assembles
// and tests in FP64.  The FP64 path factors every iteration, as the reference does; with factor reuse on
// (the mixed path's default) an iteration keeps the FP32 factors of an earlier Jacobian -- of an earlier
// iteration or time point -- while the FP64 residual still falls at least fourfold per iteration (Newton
// as iterative refinement, converging to the same solution under the same test), and factors afresh
// otherwise, or after 32 reuses.
static int newton(s21_large* L, bool tran, double dt, bool commit = true) {
    const int n = L->t.n;
    bool prev_ok = true;  // dx starts at zero
    LCHECK(hipMemsetAsync(L->flags.p, 0, 8 * sizeof(int), L->stream));
    double res_prev = 0.0;
    bool last_reused = false;
    for (int it = 0; it < 100; it++) {  // analysis.rs:173
        L->iters++;
        assemble_residual(L, tran, dt);
        int hf[8];
        LCHECK(hipMemcpyAsync(hf, L->flags.p, sizeof(hf), hipMemcpyDeviceToHost, L->stream));
        LCHECK(hipStreamSynchronize(L->stream));
        if (hf[1]) return S21_PIVOT;  // the last factorisation met a zero pivot
        if (it > 0) prev_ok = hf[2] == 0;
        if (prev_ok && hf[0] == 0) {
            if (commit) commit_state(L, tran, dt);
            return S21_OK;
        }
        double res_now;
        {
            unsigned long long bits;
            std::memcpy(&bits, hf + 4, sizeof(bits));
            res_now = __builtin_bit_cast(double, bits);
        }
        // the first iteration of a solve has no residual of its own to compare with: it keeps the factors;
        // a reused solve that came out non-finite (hf[3]) was discarded and is repeated with fresh factors
        const bool refactor = !L->reuse || !L->have_factors || L->reused >= 32 || (hf[3] && last_reused) ||
                              (it > 0 && !(res_now <= 0.25 * res_prev));
        res_prev = res_now;
        LCHECK(hipMemsetAsync(L->flags.as<int>() + 1, 0, 3 * sizeof(int), L->stream));
        if (refactor) {
            if (L->precision == S21_MIXED)
                factor<float>(L);
            else
                factor<double>(L);
            L->have_factors = true;
            L->reused = 0;
        } else {
            L->reused++;
        }
        last_reused = !refactor;
        if (L->precision == S21_MIXED)
            solve<float>(L);
        else
            solve<double>(L);
        LCHECK(hipMemsetAsync(L->mxbits.p, 0, sizeof(unsigned long long), L->stream));
        hipLaunchKernelGGL(k_maxabs, dim3(blocks(n)), dim3(TPB), 0, L->stream, n, L->dx.as<double>(),
                           L->mxbits.as<unsigned long long>(), L->flags.as<int>() + 3);
        hipLaunchKernelGGL(k_update, dim3(blocks(n)), dim3(TPB), 0, L->stream, n, L->dx.as<double>(),
                           L->mxbits.as<unsigned long long>(), L->opts.reltol, L->x.as<double>(),
                           L->flags.as<int>() + 2, last_reused ? 1 : 0, L->flags.as<int>() + 3);
        LCHECK(hipGetLastError());
    }
    return S21_CONVERGENCE;
}

static void reset_state(s21_large* L) {
    for (Buf* b : {&L->m1_state, &L->d_state, &L->c_q, &L->x, &L->m1_icur, &L->d_icur, &L->c_icur, &L->b4_st})
        LCHECK(hipMemsetAsync(b->p, 0, b->bytes, L->stream));
    L->iters = 0;
    L->factorisations = 0;
    L->have_factors = false;  // each analysis starts from a fresh factorisation
}

}  // namespace lg
}  // namespace s21

namespace s21 {
namespace lg {

template <typename F>
static int lguard(F&& f) {
    try {
        f();
        return S21_OK;
    } catch (const Error& e) {
        set_last_error(e.what());
        return e.code;
    } catch (const std::bad_alloc&) {
        set_last_error("out of host memory");
        return S21_ERR;
    } catch (const std::exception& e) {
        set_last_error(e.what());
        return S21_ERR;
    }
}

static void check_current_device(const s21_large* L) {
    int dev = 0;
    LCHECK(hipGetDevice(&dev));
    if (dev != L->device) fail(S21_INVALID, "the current device is not the one the instance was created on");
}

}  // namespace lg
}  // namespace s21

using namespace s21;
using namespace s21::lg;

extern "C" {

int s21_large_create(const s21_netlist* net, const s21_options* opts, int32_t precision, s21_large** out) {
    return lguard([&] {
        if (!out || !net) fail(S21_INVALID, "s21_large_create: bad arguments");
        *out = nullptr;
        const s21_netlist& nl = *net;
        if (nl.n_vars < 0 || nl.n_comps < 0 || (nl.n_comps > 0 && !nl.comps)) fail(S21_INVALID, "malformed netlist");
        int n = 0;
        hipError_t e = hipGetDeviceCount(&n);
        if (e != hipSuccess || n == 0) fail(S21_DEVICE, "no HIP device available");
        std::unique_ptr<s21_large> L(new s21_large());
        LCHECK(hipGetDevice(&L->device));
        hipDeviceProp_t prop;
        LCHECK(hipGetDeviceProperties(&prop, L->device));
        if (std::string(prop.gcnArchName).rfind("gfx950", 0) != 0)
            fail(S21_DEVICE, std::string("engine is built for gfx950, device is ") + prop.gcnArchName);
        L->n_vars = nl.n_vars;
        for (int k = 0; k < nl.n_vars; k++) {
            L->names.push_back(nl.var_name && nl.var_name[k] ? nl.var_name[k] : ("v" + std::to_string(k)));
            L->kinds.push_back(nl.var_kind ? nl.var_kind[k] : S21_VAR_V);
        }
        L->comps.assign(nl.comps, nl.comps + nl.n_comps);
        auto take = [](int k, const s21_params* p, std::vector<s21_params>& v) {
            if (k > 0 && !p) fail(S21_INVALID, "malformed netlist");
            v.assign(p, p + std::max(k, 0));
        };
        take(nl.n_bsim4_models, nl.bsim4_models, L->bsim4_models);
        take(nl.n_bsim4_insts, nl.bsim4_insts, L->bsim4_insts);
        take(nl.n_mos1_models, nl.mos1_models, L->mos1_models);
        take(nl.n_mos1_insts, nl.mos1_insts, L->mos1_insts);
        take(nl.n_diode_models, nl.diode_models, L->diode_models);
        take(nl.n_diode_insts, nl.diode_insts, L->diode_insts);
        if (opts)
            L->opts = *opts;
        else
            s21_default_options(&L->opts);
        L->precision = precision == S21_MIXED ? S21_MIXED : S21_FP64;
        bool bsim4 = false;
        for (const s21_comp& c : L->comps) bsim4 = bsim4 || c.type == S21_COMP_BSIM4;
        L->has_bsim4 = bsim4;
        L->reuse = L->precision == S21_MIXED && !bsim4 ? 1 : 0;
        LCHECK(hipStreamCreateWithFlags(&L->stream, hipStreamNonBlocking));
        LCHECK(hipEventCreate(&L->ev0));
        LCHECK(hipEventCreate(&L->ev1));
        *out = L.release();
    });
}

void s21_large_free(s21_large* L) { delete L; }

int s21_large_op(s21_large* L) {
    return lguard([&] {
        if (!L) fail(S21_INVALID, "null instance");
        check_current_device(L);
        if (L->prepared != "op") {
            L->prepared.clear();
            prepare(L, nullptr);
            L->prepared = "op";
        }
        reset_state(L);
        L->trap = 0;
        const auto t0 = std::chrono::steady_clock::now();
        L->status = newton(L, false, 0.0);
        LCHECK(hipStreamSynchronize(L->stream));
        L->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        L->npts = 0;
        L->axis.clear();
    });
}

int s21_large_tran(s21_large* L, const s21_tran_options* tr) {
    return lguard([&] {
        if (!L || !tr) fail(S21_INVALID, "null argument");
        if (!(tr->tstep > 0.0) && tr->tstop > 0.0) fail(S21_INVALID, "tstep must be positive");
        check_current_device(L);
        const std::string key = prep_key(tr);
        if (L->prepared != key) {
            L->prepared.clear();
            prepare(L, tr);
            L->prepared = key;
        }
        reset_state(L);
        L->trap = 0;
        const int n = L->t.n;
        const int64_t npts = s21_tran_point_count(tr->tstep, tr->tstop);
        L->wave.alloc((size_t)npts * n * sizeof(double));
        const auto t0 = std::chrono::steady_clock::now();
        L->status = newton(L, false, 0.0);  // operating point with the ICs forced (analysis.rs:540-549)
        int64_t stored = 0;
        if (L->status == S21_OK) {
            LCHECK(hipMemcpyAsync(L->wave.as<double>(), L->x.p, n * sizeof(double), hipMemcpyDeviceToDevice, L->stream));
            stored = 1;
            for (int64_t p = 1; p < npts; p++) {  // t = tstep, 2 tstep, ... while t < tstop
                L->status = newton(L, true, tr->tstep);
                if (L->status != S21_OK) break;
                LCHECK(hipMemcpyAsync(L->wave.as<double>() + (size_t)p * n, L->x.p, n * sizeof(double),
                                      hipMemcpyDeviceToDevice, L->stream));
                stored = p + 1;
            }
        }
        LCHECK(hipStreamSynchronize(L->stream));
        L->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        L->npts = stored;
        L->axis.assign(stored, 0.0);
        double t = tr->tstep;
        for (int64_t p = 1; p < stored; p++) {
            L->axis[p] = t;
            t += tr->tstep;
        }
    });
}

int s21_large_tran_trap(s21_large* L, const s21_tran_options* tr, const s21_trap_options* o) {
    return lguard([&] {
        if (!L || !tr || !o) fail(S21_INVALID, "null argument");
        if (!(tr->tstep > 0.0) || !(tr->tstop >= 0.0)) fail(S21_INVALID, "tstep must be positive");
        check_current_device(L);
        for (const s21_comp& c : L->comps)
            if (c.type == S21_COMP_BSIM4)  // tran_op bakes ag0 = 1 / dt into its companions (tran.rs:86)
                fail(S21_INVALID, "BSIM4 devices integrate by Backward Euler only");
        const std::string key = prep_key(tr);
        if (L->prepared != key) {
            L->prepared.clear();
            prepare(L, tr);
            L->prepared = key;
        }
        reset_state(L);
        L->trap = 0;  // the operating point integrates nothing
        const int n = L->t.n;
        const int64_t npts = s21_tran_point_count(tr->tstep, tr->tstop);
        std::vector<double> axis(npts, 0.0);  // the reference's output grid (t += tstep)
        {
            double t = tr->tstep;
            for (int64_t p = 1; p < npts; p++) {
                axis[p] = t;
                t += tr->tstep;
            }
        }
        L->wave.alloc((size_t)npts * n * sizeof(double));
        for (Buf& h : L->hist) h.alloc((size_t)std::max(n, 1) * sizeof(double));
        L->accepted = L->rejected = 0;
        const auto t0 = std::chrono::steady_clock::now();
        L->status = newton(L, false, 0.0);
        int64_t stored = 0;
        double* W = L->wave.as<double>();
        auto copy = [&](double* dst, const void* src) {
            LCHECK(hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToDevice, L->stream));
        };
        if (L->status == S21_OK) {
            copy(W, L->x.p);
            stored = 1;
            const double dtmax = tr->tstep;
            const double dtmin = o->dt_min > 0.0 ? o->dt_min : dtmax * 1e-9;
            // hist[0] = x at the last accepted point (time th[0]), hist[1..3] the ones before
            int h[4] = {0, 1, 2, 3};
            double th[4] = {0.0, 0.0, 0.0, 0.0};
            int nh = 1;
            copy(L->hist[h[0]].as<double>(), L->x.p);
            double t = 0.0, dt = o->lte ? dtmax / 4.0 : dtmax;
            L->trap = 2;  // the first step is Backward Euler, as SPICE starts: the operating point's capacitor
                          // currents (zero) do not describe the circuit released from its IC forcing
            const double t_end = axis[npts - 1];
            int64_t k = 1;
            while (k < npts) {
                if (o->lte) dt = std::min(dt, t_end - t);
                const double tn = o->lte ? t + dt : axis[k];
                L->status = newton(L, true, dt, false);
                double r = 0.0;
                if (L->status == S21_OK && o->lte && nh >= 3) {
                    LCHECK(hipMemsetAsync(L->mxbits.p, 0, sizeof(unsigned long long), L->stream));
                    hipLaunchKernelGGL(k_lte, dim3(blocks(n)), dim3(TPB), 0, L->stream, n, L->kinds_dev.as<int>(),
                                       L->x.as<double>(), L->hist[h[0]].as<double>(), L->hist[h[1]].as<double>(),
                                       L->hist[h[2]].as<double>(), tn, th[0], th[1], th[2], o->reltol, o->abstol,
                                       o->trtol, L->mxbits.as<unsigned long long>());
                    unsigned long long bits = 0;
                    LCHECK(hipMemcpyAsync(&bits, L->mxbits.p, sizeof(bits), hipMemcpyDeviceToHost, L->stream));
                    LCHECK(hipStreamSynchronize(L->stream));
                    r = __builtin_bit_cast(double, bits);
                }
                if (L->status != S21_OK || r > 1.0) {  // reject: back to the last accepted point
                    if (!o->lte) break;
                    L->rejected++;
                    dt = L->status != S21_OK ? dt / 4.0 : dt * std::max(0.25, 0.9 * std::cbrt(1.0 / r));
                    copy(L->x.as<double>(), L->hist[h[0]].p);
                    if (dt < dtmin) {
                        L->status = S21_CONVERGENCE;
                        fail(S21_CONVERGENCE, "Timestep too small");
                    }
                    L->status = S21_OK;
                    continue;
                }
                commit_state(L, true, dt);
                L->accepted++;
                L->trap = 1;
                if (o->lte) {  // output-grid points in (t, tn], linearly between the accepted points
                    while (k < npts && axis[k] <= tn * (1.0 + 1e-12)) {
                        const double w = std::min(1.0, (axis[k] - t) / (tn - t));
                        hipLaunchKernelGGL(k_interp, dim3(blocks(n)), dim3(TPB), 0, L->stream, n,
                                           L->hist[h[0]].as<double>(), L->x.as<double>(), w, W + (size_t)k * n);
                        k++;
                    }
                } else {
                    copy(W + (size_t)k * n, L->x.p);
                    k++;
                }
                stored = k;
                // history: the new point in front
                const int last = h[3];
                for (int q = 3; q > 0; q--) {
                    h[q] = h[q - 1];
                    th[q] = th[q - 1];
                }
                h[0] = last;
                th[0] = tn;
                copy(L->hist[h[0]].as<double>(), L->x.p);
                nh = std::min(nh + 1, 4);
                t = tn;
                if (o->lte && nh >= 4) dt = std::min(dtmax, dt * (r > 0.0 ? std::min(2.0, 0.9 * std::cbrt(1.0 / r)) : 2.0));
            }
        }
        LCHECK(hipStreamSynchronize(L->stream));
        L->trap = 0;
        L->ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        L->npts = stored;
        L->axis.assign(axis.begin(), axis.begin() + stored);
    });
}

int s21_large_trap_stats(const s21_large* L, int64_t* accepted, int64_t* rejected) {
    return lguard([&] {
        if (!L) fail(S21_INVALID, "null instance");
        if (accepted) *accepted = L->accepted;
        if (rejected) *rejected = L->rejected;
    });
}

int32_t s21_large_n_vars(const s21_large* L) { return L ? (L->t.n ? L->t.n : L->n_vars) : 0; }

const char* s21_large_var_name(const s21_large* L, int32_t k) {
    if (!L || k < 0) return nullptr;
    const std::vector<std::string>& nm = L->t.n ? L->t.names : L->names;
    return k < (int)nm.size() ? nm[k].c_str() : nullptr;
}

int s21_large_get_x(const s21_large* L, double* out) {
    return lguard([&] {
        if (!L || !out || !L->t.n) fail(S21_INVALID, "no analysis has run");
        LCHECK(hipMemcpy(out, L->x.p, L->t.n * sizeof(double), hipMemcpyDeviceToHost));
    });
}

int s21_large_get_status(const s21_large* L, int32_t* status, int64_t* iters) {
    return lguard([&] {
        if (!L) fail(S21_INVALID, "null instance");
        if (status) *status = L->status;
        if (iters) *iters = L->iters;
    });
}

int64_t s21_large_n_points(const s21_large* L) { return L ? L->npts : 0; }

int s21_large_get_axis(const s21_large* L, double* out) {
    return lguard([&] {
        if (!L || !out) fail(S21_INVALID, "bad arguments");
        std::copy(L->axis.begin(), L->axis.end(), out);
    });
}

int s21_large_get_wave(const s21_large* L, int32_t n_sel, const int32_t* vars, double* out) {
    return lguard([&] {
        if (!L || !out || n_sel < 0 || (n_sel > 0 && !vars)) fail(S21_INVALID, "bad arguments");
        const int n = L->t.n;
        for (int j = 0; j < n_sel; j++)
            if (vars[j] < 0 || vars[j] >= n) fail(S21_INVALID, "variable out of range");
        std::vector<double> row(n);
        for (int64_t p = 0; p < L->npts; p++) {
            LCHECK(hipMemcpy(row.data(), L->wave.as<double>() + (size_t)p * n, n * sizeof(double),
                             hipMemcpyDeviceToHost));
            for (int j = 0; j < n_sel; j++) out[(size_t)p * n_sel + j] = row[vars[j]];
        }
    });
}

int s21_large_structure(const s21_large* L, int64_t* nnz_a, int64_t* nnz_lu, int64_t* fronts, int64_t* levels,
                        int64_t* max_front, double* flops_lu) {
    return lguard([&] {
        if (!L || !L->t.n) fail(S21_INVALID, "no analysis has run");
        if (nnz_a) *nnz_a = L->S.nnz_a;
        if (nnz_lu) *nnz_lu = L->S.nnz_lu;
        if (fronts) *fronts = L->S.ns;
        if (levels) *levels = (int64_t)L->levels.size();
        if (max_front) *max_front = L->S.max_front;
        if (flops_lu) *flops_lu = L->S.flops;
    });
}

int s21_large_timing(const s21_large* L, double* total_ms, int64_t* factorisations) {
    return lguard([&] {
        if (!L) fail(S21_INVALID, "null instance");
        if (total_ms) *total_ms = L->ms_total;
        if (factorisations) *factorisations = L->factorisations;
    });
}

int s21_large_set_reuse(s21_large* L, int32_t on) {
    return lguard([&] {
        if (!L) fail(S21_INVALID, "null instance");
        if (on && L->has_bsim4) fail(S21_INVALID, "factor reuse is not available with BSIM4 devices");
        L->reuse = on ? 1 : 0;
    });
}

int s21_large_time_factor(s21_large* L, int32_t reps, double* factor_ms, double* solve_ms) {
    return lguard([&] {
        if (!L || reps <= 0 || !L->t.n) fail(S21_INVALID, "bad arguments");
        check_current_device(L);
        float ms = 0.0f;
        LCHECK(hipEventRecord(L->ev0, L->stream));
        for (int r = 0; r < reps; r++) {
            if (L->precision == S21_MIXED)
                factor<float>(L);
            else
                factor<double>(L);
        }
        LCHECK(hipEventRecord(L->ev1, L->stream));
        LCHECK(hipEventSynchronize(L->ev1));
        LCHECK(hipEventElapsedTime(&ms, L->ev0, L->ev1));
        if (factor_ms) *factor_ms = ms / reps;
        LCHECK(hipEventRecord(L->ev0, L->stream));
        for (int r = 0; r < reps; r++) {
            if (L->precision == S21_MIXED)
                solve<float>(L);
            else
                solve<double>(L);
        }
        LCHECK(hipEventRecord(L->ev1, L->stream));
        LCHECK(hipEventSynchronize(L->ev1));
        LCHECK(hipEventElapsedTime(&ms, L->ev0, L->ev1));
        if (solve_ms) *solve_ms = ms / reps;
    });
}

int s21_large_host_check(int32_t n, int64_t ne, const int32_t* rows, const int32_t* cols, const double* vals,
                         const double* b, double relax, double* x, int64_t* nnz_lu, double* flops_lu) {
    return lguard([&] {
        if (n <= 0 || ne < 0 || (ne > 0 && (!rows || !cols || !vals)) || !b || !x) fail(S21_INVALID, "bad arguments");
        std::vector<int> r(rows, rows + ne), c(cols, cols + ne);
        std::vector<double> v(vals, vals + ne);
        LargeSym S;
        large_symbolic(n, r, c, &v, S, relax);
        std::vector<double> pool, xs;
        large_factor_host(S, r, c, v, pool);
        large_solve_host(S, pool, std::vector<double>(b, b + n), xs);
        std::copy(xs.begin(), xs.end(), x);
        if (nnz_lu) *nnz_lu = S.nnz_lu;
        if (flops_lu) *flops_lu = S.flops;
    });
}

}  // extern "C"
