// Shared device-side definitions of the MI355X GFN2-xTB engine.
//
// One workgroup owns one system (trajectory).  Per-system data lives in flat
// device arrays addressed through SysInfo offsets; per-system n x n matrices
// are stored row-major with a leading dimension ld = round_up(nao, 16) and
// zero padding, so that 16 x 16 FP64 MFMA tiles cover them exactly.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gfn2_params.h"

#define QX_BLOCK 512       // threads per system in the setup and gradient kernels
#define QX_SCC_BLOCK 512   // threads per system in the SCC kernel
#define QX_MAX_NAT 64
#define QX_MAX_NSH 128
#define QX_MAX_NAO 256
#define QX_MAX_REF 7
#define QX_PAIR_STRIDE 16  // doubles per ordered atom pair in the gradient pair buffer
#define QX_PAIR_KERN 3     // kernel planes per ordered atom pair

#ifndef QX_DEFAULT_EXTRAPOLATE
#define QX_DEFAULT_EXTRAPOLATE 4  // MD start of the SCC when the caller passes 0
#endif

#define QX_DEV __device__ __forceinline__

// Thread index of a phase.  The empty asm hides its origin from the compiler,
// so the addresses a phase derives from it are formed again each time the
// phase runs instead of being hoisted out of the SCC loop, where the
// addresses of all phases together overflowed the register file.  (The CPU
// emulation of the kernels compiles the plain index.)
QX_DEV int qx_tid()
{
    int t = threadIdx.x;
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+v"(t));
#endif
    return t;
}

// Wavefront index as a scalar: loops over it run on the scalar unit.
QX_DEV int qx_wave(int tid)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_readfirstlane(tid >> 6);
#else
    return tid >> 6;
#endif
}

// A value that is the same on every thread, as a scalar: what it decides is
// then branched on by the scalar unit, without execution masks to keep.
QX_DEV int qx_uniform(int v)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_readfirstlane(v);
#else
    return v;
#endif
}

// v of lane l, l the same on every lane: two scalar reads instead of the LDS
// crossbar of __shfl.
QX_DEV double qx_bcast(double v, int l)
{
#ifdef __HIP_DEVICE_COMPILE__
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
#else
    return __shfl(v, l, 64);
#endif
}

#ifdef __HIP_DEVICE_COMPILE__
template <int CTRL>
QX_DEV double qx_dpp(double v)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
#endif

// v of the next / previous lane; the last / first lane gets edge
QX_DEV double qx_lane_up(double v, double edge)
{
#ifdef __HIP_DEVICE_COMPILE__
    const long long b = __double_as_longlong(v), g = __double_as_longlong(edge);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp((int)g, (int)b, 0x130, 0xf, 0xf, false);  // wave_shl:1
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp((int)(g >> 32), (int)(b >> 32), 0x130, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
#else
    const int l = threadIdx.x & 63;
    const double x = __shfl(v, l < 63 ? l + 1 : l, 64);
    return l < 63 ? x : edge;
#endif
}
QX_DEV double qx_lane_down(double v, double edge)
{
#ifdef __HIP_DEVICE_COMPILE__
    const long long b = __double_as_longlong(v), g = __double_as_longlong(edge);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp((int)g, (int)b, 0x138, 0xf, 0xf, false);  // wave_shr:1
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp((int)(g >> 32), (int)(b >> 32), 0x138, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
#else
    const int l = threadIdx.x & 63;
    const double x = __shfl(v, l > 0 ? l - 1 : l, 64);
    return l > 0 ? x : edge;
#endif
}

// whether p holds on any lane of the wavefront
QX_DEV bool qx_any(bool p)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_ballot_w64(p) != 0;
#else
    int v = p;
    for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, 64);
    return v != 0;
#endif
}

// Keeps the instructions before it (a batch of loads) before those after it.
QX_DEV void qx_sched_fence()
{
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_sched_barrier(0);
#endif
}

struct QxAdd {
    QX_DEV static double op(double a, double b) { return a + b; }
};
struct QxMax {
    QX_DEV static double op(double a, double b) { return fmax(a, b); }
};

// Reduction over the 64 lanes, the result on every lane: quad permutations
// and row mirrors (data-parallel primitives, no LDS crossbar) inside the rows
// of 16 lanes, then the four rows' values by scalar reads.
template <class F>
QX_DEV double wave_reduce(double v)
{
#ifdef __HIP_DEVICE_COMPILE__
    v = F::op(v, qx_dpp<0xb1>(v));   // quad_perm 1 0 3 2
    v = F::op(v, qx_dpp<0x4e>(v));   // quad_perm 2 3 0 1
    v = F::op(v, qx_dpp<0x141>(v));  // mirrored half rows
    v = F::op(v, qx_dpp<0x140>(v));  // mirrored rows
    return F::op(F::op(qx_bcast(v, 0), qx_bcast(v, 16)), F::op(qx_bcast(v, 32), qx_bcast(v, 48)));
#else
    for (int o = 32; o > 0; o >>= 1) v = F::op(v, __shfl_xor(v, o, 64));
    return v;
#endif
}

// sum over the four lanes of a quad, on each of them
QX_DEV double quad_sum(double v)
{
#ifdef __HIP_DEVICE_COMPILE__
    v += qx_dpp<0xb1>(v);
    return v + qx_dpp<0x4e>(v);
#else
    v += __shfl_xor(v, 1, 64);
    return v + __shfl_xor(v, 2, 64);
#endif
}

QX_DEV double wave_sum(double v) { return wave_reduce<QxAdd>(v); }
QX_DEV double wave_max(double v) { return wave_reduce<QxMax>(v); }

struct ElemParams {
    int z, nsh, nprim[2], pqn[2];
    double alpha[2][6], coeff[2][6];  // scaled exponents, normalised contraction coefficients
    double slater[2], hself0[2], kcn[2], shpoly[2], refocc[2];  // self-energies/kcn in Eh
    double hard[2], third[2];                                     // shell hardness, Gamma_l
    double rep_alpha, rep_zeff, en, rad, dkernel, qkernel, mprad, mpvcn, nval, covrad;
    // D4
    int nref, refc[QX_MAX_REF];
    double refq[QX_MAX_REF], refcovcn[QX_MAX_REF], zeff, gam, r4r2, rcov_d4, en_d4;
};

struct DevTables {
    ElemParams e[gfn2::kElem];
    double c6ref[gfn2::kElem][QX_MAX_REF][gfn2::kElem][QX_MAX_REF];
};

extern __constant__ DevTables g_tab;
extern __constant__ double g_rad[118];  // QCxMS bond radii (covalent_radii.f90:89-114), Bohr

struct SysInfo {
    int nat, nsh, nao, ld, ndim, nx;
    int atom_off, shell_off, ref_off, x_off;
    long long mat_off;   // one ld*ld slot
    long long gam_off;   // nsh*nsh
    long long hist_off;  // Broyden history: 2*mem*nx + mem*mem
    long long pair_off;  // nat*nat*QX_PAIR_STRIDE gradient scratch
    int item_off;        // shell-pair work items: off-atom pairs first (grouped by
    int nitem_off;       // angular-momentum class), then same-atom pairs
    int nitem;
    int rowitem_off;     // the same pairs split into rows of the first shell's AOs
    int nrowitem;        // (rows of three AO pairs first), for the setup integrals
    int charge;
    double nel, kt;
};

struct SccOpts {
    double econv, pconv, damp, jacobi_tol;
    int maxiter, mem;
    int extrapolate;  // MD start: 1 linear 2 x(n-1) - x(n-2), 2 quadratic 3 (x(n-1) - x(n-2)) + x(n-3),
                      // 3 cubic 4 (x(n-1) + x(n-3)) - 6 x(n-2) - x(n-4),
                      // 4 quartic 5 (x(n-1) - x(n-4)) - 10 (x(n-2) - x(n-3)) + x(n-5)
    int keep;         // > 0: Broyden secant pairs kept across warm-started calls (ring of keep)
    int lds_doubles;  // dynamic LDS of the launch in doubles (set per launch by the host)
    int eig_mfma;     // 1: MFMA simultaneous-rotation eigen refinement before Jacobi
    int lds_max_m;    // systems of at most this (even) basis size keep their SCC matrices in
                      // LDS, the others in global memory (set per launch, <= qx::kFastM)
    int first_sys;    // system of workgroup 0 (a launch over a range of the batch's systems); -1: all
                      // systems in the batch's launch order
};

// Device-resident batch state.  Every pointer is a flat array over all systems.
struct BatchPtrs {
    int nsys;
    const SysInfo* info;
    const int* order; // systems by decreasing basis size: workgroup k of a setup, SCC, gradient or
                      // persistent MD launch over all takes order[k], so the longest run first
                      // and the short ones fill the end (launches over a range and k_dblocks
                      // keep the batch's order)
                      // (6 MD steps of 512 chains of 2 .. 11 heavy atoms: 28.9 -> 21.5 ms)
    const int* elem;  // per atom: element slot
    double* xyz;      // 3 per atom
    double* grad;     // 3 per atom
    double* qat;      // per atom
    double* cn;       // per atom (GFN2 CN)
    double* cnd4;     // per atom (D4 covalent CN)
    double* mrad;     // per atom
    double* dmrad;    // per atom
    double* hself;    // per shell
    double* gw;       // per D4 reference
    double* dgw;      // per D4 reference
    double* S;        // ld^2 per system
    double* H0;
    double* D;        // 3 ld^2 per system: dipole integral (mu, nu) about mu's atom at nu*ld+mu
    double* Q;        // 6 ld^2 per system: traceless quadrupole, same layout
    double* L;        // Cholesky factor of S (lower)
    double* X;        // L^-T (upper): X^T S X = 1
    double* C;        // eigenvectors (AO basis)
    double* T;        // scratch
    double* P;        // density
    double* W;        // energy-weighted density
    double* U;        // eigenvectors in the orthogonalised basis (warm start)
    double* E;        // scratch matrix of the MFMA eigen refinement (systems whose SCC
                      // matrices are in global memory)
    double* gam;      // nsh^2 per system
    double* x;        // mixing vector [qsh, dp, qp] (converged, warm start)
    double* xo;       // output moments of the last iteration
    double* vs;       // per shell potential at the output moments
    double* vd;       // 3 per atom
    double* vq;       // 6 per atom
    double* eps;      // orbital energies, ld per system
    double* focc;     // occupations, ld per system
    double* hist;     // Broyden history
    double* pairbuf;  // gradient scratch
    const int2* spitem;  // shell-pair work items (ia, ib), ia > ib or same shell
    double* spbuf;    // per shell pair (ia, ib): gradient on A (3), dE/dCN_A, dE/dCN_B
    double* pairk;    // QX_PAIR_KERN planes of nat x nat per system: damped multipole kernels
                      // 1/r^3 and 1/r^5, D4 pair damping
    double* dblk;     // stored derivative blocks per off-atom shell-pair item (null: recomputed)
    double* xprev;    // mixing vector of the step before (extrapolated MD start)
    double* xprev2;   // and of the step before that
    double* xprev3;   // and of the one before that (cubic extrapolation)
    double* xprev4;   // and of the one before that (quartic extrapolation)
    double* energy;   // per system: total
    double* eparts;   // per system: 10 parts (band, es2, es3, aes, axc, d4, atm, rep, ts, scc)
    int* iters;       // per system
    unsigned long long* iters_total;  // per system: SCC iterations summed over calls
    int* status;      // per system: 0 ok, -1 not converged
    int* warm;        // per system: 1 if U/x hold a previous solution
    const int* active;  // per system: 0 skips the system (finished trajectories), may be null
};

// Kernel arguments as the phases see them.  A kernel that takes one argument
// structure reads it through a pointer to the argument segment, so a phase
// loads (scalar loads) the pointers and options it needs when it runs,
// instead of all of them staying in scalar registers through the SCC loop.
// (Plain references in the CPU emulation.)
#ifdef __HIP_DEVICE_COMPILE__
#define QX_ARG(T) const __attribute__((address_space(4))) T&
template <class T>
QX_DEV QX_ARG(T) qx_args(const T&)
{
    return *(const __attribute__((address_space(4))) T*)__builtin_amdgcn_kernarg_segment_ptr();
}
#else
#define QX_ARG(T) const T&
template <class T>
QX_DEV QX_ARG(T) qx_args(const T& a)
{
    return a;
}
#endif
typedef QX_ARG(BatchPtrs) BatchRef;
typedef QX_ARG(SccOpts) OptRef;
// the batch pointers loaded anew from here on
QX_DEV BatchRef qx_fresh(BatchRef B)
{
#ifdef __HIP_DEVICE_COMPILE__
    auto p = &B;
    asm volatile("" : "+s"(p));
    return *p;
#else
    return B;
#endif
}

// The record of system sys in scalar registers (the MD changes kt, so the
// compiler would load it per lane).
QX_DEV SysInfo qx_info(BatchRef B, int sys)
{
#ifdef __HIP_DEVICE_COMPILE__
    static_assert(sizeof(SysInfo) % 4 == 0, "copied in words");
    const int* src = (const int*)(B.info + sys);
    int w[sizeof(SysInfo) / 4];
#pragma unroll
    for (int k = 0; k < (int)(sizeof(SysInfo) / 4); ++k) w[k] = src[k];
#pragma unroll
    for (int k = 0; k < (int)(sizeof(SysInfo) / 4); ++k) w[k] = qx_uniform(w[k]);
    SysInfo si;
    __builtin_memcpy(&si, w, sizeof(SysInfo));
    return si;
#else
    return B.info[sys];
#endif
}

// 1 / sqrt(x) to rounding: the hardware estimate and one third-order step
QX_DEV double qx_rsqrt(double x)
{
#ifdef __HIP_DEVICE_COMPILE__
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
#else
    return 1.0 / sqrt(x);
#endif
}

// Block barrier that orders LDS accesses only: global stores in flight stay
// in flight (__syncthreads waits for them too).
QX_DEV void qx_lds_barrier()
{
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#else
    __syncthreads();
#endif
}

QX_DEV int pad16(int n) { return (n + 15) & ~15; }

// block-wide sum (all threads must call); smem needs QX_BLOCK/64 doubles
QX_DEV double block_sum(double v, double* smem)
{
    v = wave_sum(v);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) smem[w] = v;
    __syncthreads();
    double s = 0.0;
    for (int i = 0; i < QX_BLOCK / 64; ++i) s += smem[i];
    __syncthreads();
    return s;
}

// Shell descriptor built per system in LDS
struct ShellDesc {
    int at, l, el, k, ao0, nao;  // k: shell index within the element
};

// Fill shell and AO tables of one system (called by all threads).
QX_DEV void build_shell_tables(const SysInfo& si, const int* elem, ShellDesc* sh, int* ao_at,
                               int* ao_sh)
{
    if (threadIdx.x == 0) {
        int is = 0, ia = 0;
        for (int a = 0; a < si.nat; ++a) {
            int el = elem[si.atom_off + a];
            for (int k = 0; k < g_tab.e[el].nsh; ++k) {
                ShellDesc d;
                d.at = a;
                d.l = k;
                d.el = el;
                d.k = k;
                d.ao0 = ia;
                d.nao = k ? 3 : 1;
                sh[is] = d;
                for (int c = 0; c < d.nao; ++c) {
                    ao_at[ia] = a;
                    ao_sh[ia] = is;
                    ++ia;
                }
                ++is;
            }
        }
    }
    __syncthreads();
}
