// Self-consistent charge iterations of GFN2-xTB, one workgroup per system,
// all iterations inside one launch (data-dependent iteration counts never
// leave the device).
//
// Per iteration: potentials from the mixed moments -> Fock matrix built from
// row-local potentials G (F = H0 - (G + G^T)/2, coalesced reads of the
// transposed moment integrals) -> A = C^T F C in the current orbital basis C
// (S-orthonormal) -> parallel cyclic threshold Jacobi on A with the rotations
// applied straight to the columns of C -> Fermi occupations (one wavefront,
// safeguarded Newton from the previous chemical potential) ->
// P = C diag(2f) C^T -> Mulliken shell charges, atomic dipole/quadrupole
// moments and the band energy as column sweeps -> energy -> modified Broyden
// mixing (Johnson, PRB 38, 12807 (1988)).
// The Jacobi tolerance follows the SCC: 1e-3 of the previous iteration's RMS
// moment change, never looser than 1e-6 and never tighter than the requested
// floor, so the converged iterate is diagonalised to the floor.
// Systems with at most opt.lds_max_m (<= kFastM) basis functions keep A, C,
// F and P in LDS; larger ones use per-system global scratch.  C starts as X U with X = L^-T
// and U the previous call's orthogonal basis (identity on a cold start).
#pragma once
#include "k_setup.h"

namespace qx {

constexpr int kNT = QX_SCC_BLOCK;  // threads of the SCC kernel
constexpr int kMaxNx = 128 + 9 * QX_MAX_NAT;
constexpr int kMaxRef = QX_MAX_REF * QX_MAX_NAT;
constexpr int kFastM = 56;
constexpr int kRs = 11;  // row sums per AO: S, D (3), Q (6), H0

// Opt-in per-phase cycle counters of the SCC kernel (build with
// -DQX_PHASE_TIMING); compiled out otherwise.  Rows are systems of the batch,
// whatever workgroup runs them.
#ifdef QX_PHASE_TIMING
constexpr int kPhaseSys = 1024, kPhaseSlots = 32;
__device__ unsigned long long g_phase[kPhaseSys * kPhaseSlots];
#define QX_PH_INIT unsigned long long ph_t = clock64();
#define QX_PH(sys, k)                                                              \
    do {                                                                           \
        __syncthreads();                                                           \
        if (threadIdx.x == 0 && (sys) < kPhaseSys) {                               \
            const unsigned long long t_ = clock64();                               \
            g_phase[(sys) * kPhaseSlots + (k)] += t_ - ph_t;                       \
            ph_t = t_;                                                             \
        }                                                                          \
    } while (0)
#define QX_PH_ADD(sys, k, v)                                                       \
    do {                                                                           \
        if (threadIdx.x == 0 && (sys) < kPhaseSys) g_phase[(sys) * kPhaseSlots + (k)] += (v); \
    } while (0)
#else
#define QX_PH_INIT
#define QX_PH(sys, k) \
    do {              \
    } while (0)
#define QX_PH_ADD(sys, k, v) \
    do {                     \
    } while (0)
#endif

typedef double qx_d4 __attribute__((ext_vector_type(4)));

// C[i][j] = sum_k opA[i][k] * d[k] * opB[k][j] on the FP64 matrix cores
// (v_mfma_f64_16x16x4f64).  Operands are given by their element strides:
// opA[i][k] at A[i * ai + k * ak], opB[k][j] at Bm[k * bk + j * bj].  A
// wavefront computes a strip of two 16 x 16 tiles sharing the A operand;
// operand lanes: A[i0 + l%16][k0 + l/16], B[k0 + l/16][j0 + l%16];
// accumulator element r of lane l is C[i0 + 4r + l/16][j0 + l%16].
// sym: the result is symmetric (M = N); only strips that reach the diagonal
// or lie above it are formed, and mirrored.  Lanes of rows and columns past
// the edge read the last row or column (their results are not stored); only
// the last k step is masked.  The operands of the next four k steps are
// loaded while the matrix cores work on the current four, so a strip waits
// for memory once.  Up to 56 columns a product is bound by that wait and the
// tail, above by the L1 traffic of the operands (16 lines per load of A).
// (A product of the eigenvector refinement with every strip formed -> now, in
// cycles: 58 columns 12.9 k -> 12.2 k, 88: 38 k -> 34 k, 132: 129 k -> 114 k,
// where the matrix cores need 43 k for all and half of it for the symmetric.)
QX_DEV void mfma_gemm(int M, int N, int K, const double* A, int ai, int ak, const double* Bm, int bk,
                      int bj, double* Cm, int ldc, const double* d, bool sym)
{
    constexpr int NU = 2;  // 16 x 16 tiles per strip
    constexpr int KS = 4;  // k steps per pass
    constexpr int NW = kNT / 64;
    const int tid = qx_tid(), lane = tid & 63, wave = qx_wave(tid);
    const int li = lane & 15, lk = lane >> 4;
    const int tm = (M + 15) >> 4, tc = (N + 16 * NU - 1) / (16 * NU);
    const int nblk = K / (4 * KS);
    int ti = 0, ts = wave;  // tile row, strip in the row counted from its first one
    auto row_strips = [&](int t) { return sym ? tc - t / NU : tc; };
    while (ti < tm) {
        const int ns = row_strips(ti);
        if (ts >= ns) {
            ts -= ns;
            ++ti;
            continue;
        }
        const int i0 = ti * 16, jc = (ts + tc - ns) * 16 * NU;
        ts += NW;
        const int i = i0 + li < M ? i0 + li : M - 1;
        const double* pa = A + i * ai + lk * ak;
        const double* pb[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int j = jc + 16 * u + li < N ? jc + 16 * u + li : N - 1;
            pb[u] = Bm + lk * bk + j * bj;
        }
        qx_d4 acc[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) acc[u] = qx_d4{0.0, 0.0, 0.0, 0.0};
        double a[KS], b[KS][NU];
        auto load = [&](int k0) {
#pragma unroll
            for (int q = 0; q < KS; ++q) {
                a[q] = pa[(k0 + 4 * q) * ak];
                if (d) a[q] *= d[k0 + 4 * q + lk];
#pragma unroll
                for (int u = 0; u < NU; ++u) b[q][u] = pb[u][(k0 + 4 * q) * bk];
            }
        };
        if (nblk) load(0);
        for (int kb = 0; kb < nblk; ++kb) {
            double ca[KS], cb[KS][NU];
#pragma unroll
            for (int q = 0; q < KS; ++q) {
                ca[q] = a[q];
#pragma unroll
                for (int u = 0; u < NU; ++u) cb[q][u] = b[q][u];
            }
            if (kb + 1 < nblk) load((kb + 1) * 4 * KS);
#pragma unroll
            for (int q = 0; q < KS; ++q)
#pragma unroll
                for (int u = 0; u < NU; ++u)
                    acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ca[q], cb[q][u], acc[u], 0, 0, 0);
        }
        // the rest, the last k step masked (lanes past K read k0 itself)
        for (int k0 = nblk * 4 * KS; k0 < K; k0 += 4) {
            const bool kin = k0 + lk < K;
            const int k = kin ? k0 : k0 - lk;
            double ta = pa[k * ak];
            if (d) ta *= d[k + lk];
            ta = kin ? ta : 0.0;
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const double tb = pb[u][k * bk];
                acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ta, kin ? tb : 0.0, acc[u], 0, 0, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = i0 + 4 * r + lk, col = jc + 16 * u + li;
                if (row < M && col < N && (!sym || (col >> 4) >= ti)) {
                    Cm[row * ldc + col] = acc[u][r];
                    if (sym && (col >> 4) > ti) Cm[col * ldc + row] = acc[u][r];
                }
            }
    }
}

QX_DEV double block_max(double v, double* smem)
{
    v = wave_max(v);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0) smem[w] = v;
    __syncthreads();
    double s = smem[0];
    for (int i = 1; i < kNT / 64; ++i) s = fmax(s, smem[i]);
    __syncthreads();
    return s;
}

// block-wide sums of K values at once (all threads call)
template <int K>
QX_DEV void block_sums(double* v, double* smem)
{
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_sum(v[k]);
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    __syncthreads();
    if (l == 0)
        for (int k = 0; k < K; ++k) smem[w * K + k] = v[k];
    __syncthreads();
    for (int k = 0; k < K; ++k) {
        double s = 0.0;
        for (int i = 0; i < kNT / 64; ++i) s += smem[i * K + k];
        v[k] = s;
    }
    __syncthreads();
}

// round-robin pairing: round r, slot k of m players (m even, r < m - 1)
QX_DEV void rr_pair(int m, int r, int k, int& p, int& q)
{
    if (k == 0) {
        p = r;
        q = m - 1;
    } else {
        p = r + k;
        if (p >= m - 1) p -= m - 1;
        q = r - k;
        if (q < 0) q += m - 1;
    }
}

// largest off-diagonal magnitude of the leading m x m block of A
QX_DEV double offdiag_max(const double* A, int m, int lda, double* red)
{
    double mx = 0.0;
    const int tid = qx_tid();
    for (int i = qx_wave(tid); i < m; i += kNT / 64)
        for (int j = tid & 63; j < m; j += 64)
            if (i != j) mx = fmax(mx, fabs(A[i * lda + j]));
    return block_max(mx, red);
}

// pair-ordered 2 x 2 block index b -> (P, R) with R <= P
QX_DEV void tri_index(int b, int& P, int& R)
{
    P = (int)((sqrtf(8.0f * (float)b + 1.0f) - 1.0f) * 0.5f);
    while (P * (P + 1) / 2 > b) --P;
    while ((P + 1) * (P + 2) / 2 <= b) ++P;
    R = b - P * (P + 1) / 2;
}

// Jacobi rotation (c, s) that zeroes a_pq: with d = a_qq - a_pp and
//   1/r = 1 / sqrt(d^2 + 4 a^2),  c^2 = (1 + |d| / r) / 2,
//   s = a sign(d) / (r c)   (c^2 + s^2 = 1)
// i.e. t = s / c = 2 a sign(d) / (|d| + r), the smaller root of
// t^2 + t d / a - 1 = 0.  Two reciprocal roots in a row and no division: the
// rotation is the critical path of a Jacobi round.
QX_DEV double2 jacobi_rotation(double app, double aqq, double apq)
{
    const double d = aqq - app, a2 = 2.0 * apq;
    const double ir = qx_rsqrt(d * d + a2 * a2);
    const double w = 0.5 + 0.5 * fabs(d) * ir;
    const double ic = qx_rsqrt(w);
    return make_double2(w * ic, (d >= 0.0 ? apq : -apq) * ir * ic);
}

// Rotated entries of the 2 x 2 block (P, R): input b00 = A[p][r],
// b01 = A[p][s], b10 = A[q][r], b11 = A[q][s] with (p, q) the pair of P and
// (r, s) the pair of R; on a rotated diagonal block (P == R) the off-diagonal
// entries become exact zeros.
QX_DEV void rotate_block(double2 rp, double2 rr, bool diag, const double b[4], double n[4])
{
    const double cp = rp.x, sp = rp.y, cr = rr.x, sr = rr.y;
    const double m00 = b[0] * cr - b[1] * sr, m01 = b[0] * sr + b[1] * cr;
    const double m10 = b[2] * cr - b[3] * sr, m11 = b[2] * sr + b[3] * cr;
    const bool zero = diag && sp != 0.0;
    n[0] = cp * m00 - sp * m10;
    n[1] = zero ? 0.0 : cp * m01 - sp * m11;
    n[2] = zero ? 0.0 : sp * m00 + cp * m10;
    n[3] = sp * m01 + cp * m11;
}

// Where the player of seat s (pair slot s / 2, p or q side) sits in the next
// round: the p players move one slot down, the q players one up, the ends
// turn round and q of slot 0 stays.
QX_DEV int rr_move(int half, int s)
{
    const int k = s >> 1;
    if (half == 1) return s;
    if ((s & 1) == 0) return k == 0 ? 3 : s - 2;
    if (k == 0) return s;
    return k == half - 1 ? s - 1 : s + 2;
}

// The players that meet in pair slot k of the next round: the p side comes
// from slot K1 (its q player if s1, else its p player), the q side from slot
// K2 (s2 likewise); K1 > K2 for half > 1.
QX_DEV void rr_next(int half, int k, int& K1, int& s1, int& K2, int& s2)
{
    if (k == 0) {
        K1 = half > 1 ? 1 : 0;
        s1 = 0;
        K2 = 0;
        s2 = 1;
    } else {
        K1 = k == half - 1 ? k : k + 1;
        s1 = k == half - 1 ? 1 : 0;
        K2 = k - 1;
        s2 = k == 1 ? 0 : 1;
    }
}

// The rotation of one pivot, the identity for pairs left alone
QX_DEV double2 pivot_rotation(double app, double aqq, double apq, double tol, double min_s)
{
    const double2 cs = jacobi_rotation(app, aqq, apq);
    const bool turn = !(fabs(apq) < tol) && fabs(cs.y) > min_s;
    return make_double2(turn ? cs.x : 1.0, turn ? cs.y : 0.0);
}

// Blocks per thread that the rounds with the blocks in LDS take (up to 132
// basis functions); above, the rounds work on global memory.  The LDS would
// hold the blocks of 172 functions, but a thread keeps its blocks in registers
// between the barriers.  (Six blocks: 136 functions 57.9 -> 36.1 ms and 144:
// 72.6 -> 39.5 ms, single rings of carbon, but 132: 33.3 -> 33.7 ms; as a
// further instantiation 104 to 132 functions take 0.5 % longer and the kernel
// spills 112 instead of 57 vector registers.)
constexpr int kMaxNB = 5;

// Working storage of the Jacobi sweeps
struct JacobiBuffers {
    double* blk;      // A as 2 x 2 blocks by seats: 4 planes of half (half + 1) / 2 doubles (LDS)
    double* gblk[2];  // two of them in global memory, for systems too large
    double2* log;     // rotations of a sweep: (m - 1) x m / 2
    double2* rot;     // rotations of two rounds (LDS)
    int* any;         // per round of a sweep: whether it rotates anything (LDS, m entries)
    double* red;
    bool lds;         // the blocks fit in LDS
    int sys;          // system (phase counters)
};

// The pivot of a lane in the next round: its two slots and their blocks
struct JacobiPivot {
    int K1, K2, i1, i2, i12;
    bool s1, s2;
    double d1[3], d2[3], b4[4];
    double2 r1, r2;

    QX_DEV void place(int half, int k)
    {
        int a, b;
        rr_next(half, k < half ? k : 0, K1, a, K2, b);
        s1 = a;
        s2 = b;
        i1 = K1 * (K1 + 1) / 2 + K1;
        i2 = K2 * (K2 + 1) / 2 + K2;
        i12 = K1 * (K1 + 1) / 2 + K2;
    }
    QX_DEV void load(const double* blk, int nblk, const double2* rf)
    {
        r1 = rf[K1];
        r2 = rf[K2];
        d1[0] = blk[i1];
        d1[1] = blk[nblk + i1];
        d1[2] = blk[3 * nblk + i1];
        d2[0] = blk[i2];
        d2[1] = blk[nblk + i2];
        d2[2] = blk[3 * nblk + i2];
#pragma unroll
        for (int e = 0; e < 4; ++e) b4[e] = blk[e * nblk + i12];
    }
    // the rotation, from the pivot's entries after this round (formed as the
    // threads that store them form them)
    QX_DEV double2 rotation(int half, double tol, double min_s) const
    {
        const double x1 = d1[0] * r1.x - d1[1] * r1.y, y1 = d1[0] * r1.y + d1[1] * r1.x;
        const double u1 = d1[1] * r1.x - d1[2] * r1.y, v1 = d1[1] * r1.y + d1[2] * r1.x;
        const double app = s1 ? r1.y * y1 + r1.x * v1 : r1.x * x1 - r1.y * u1;
        const double x2 = d2[0] * r2.x - d2[1] * r2.y, y2 = d2[0] * r2.y + d2[1] * r2.x;
        const double u2 = d2[1] * r2.x - d2[2] * r2.y, v2 = d2[1] * r2.y + d2[2] * r2.x;
        const double aqq = s2 ? r2.y * y2 + r2.x * v2 : r2.x * x2 - r2.y * u2;
        double nb[4];
        rotate_block(r1, r2, false, b4, nb);
        double apq = s1 ? (s2 ? nb[3] : nb[2]) : (s2 ? nb[1] : nb[0]);
        if (half == 1) apq = r1.y != 0.0 ? 0.0 : d1[1];
        return pivot_rotation(app, aqq, apq, tol, min_s);
    }
};

// Where the four entries of block b go in the next round (indices into the
// four planes)
QX_DEV void block_moves(int half, int nblk, int P, int R, int to[4])
{
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        // (1, 0) of a diagonal block is (0, 1) again
        const int x = rr_move(half, 2 * P + (P == R && e == 2 ? 0 : e >> 1));
        const int y = rr_move(half, 2 * R + (P == R && e == 2 ? 1 : e & 1));
        const int hi = (x >> 1) > (y >> 1) ? x : y, lo = hi == x ? y : x;
        const int Ph = hi >> 1, Rh = lo >> 1;
        const int plane = Ph == Rh ? (x == y ? 3 * (x & 1) : 1) : 2 * (hi & 1) + (lo & 1);
        to[e] = plane * nblk + Ph * (Ph + 1) / 2 + Rh;
    }
}

// The rounds of one sweep, blocks in LDS.  NB: blocks per thread of the
// wavefronts 1 ...; f: half of rot that holds the rotations of round 0.
// NR > 0 (m <= 64): the rows of Cv as well, two per pair of registers x[u],
// y[u] (rows_lane), a lane per pair slot: the rotation of a slot, then the
// players move to the next lane.  x holds the p players and y the q players,
// but in slot 0, whose q player stays, the other way round, so that x moves
// down and y up.  They run while wavefront 0 has the pivots.  NR = 0: the
// rotations are logged instead.
template <int NB, int NR>
QX_DEV void jacobi_rounds(const JacobiBuffers& jb, int m, int nrow, double tol, double min_s, double* x, double* y,
                          int& f)
{
    constexpr int kNU = kNT - 64, NW = kNT / 64 - 1, NK = NB > 3 ? 2 : 1;  // NK pivots per lane (half <= 64 NK)
    const int tid = qx_tid(), lane = tid & 63, wave = qx_wave(tid), ut = tid - 64;
    const int half = m / 2, nblk = half * (half + 1) / 2;
    double* blk = jb.blk;
    const int k = lane & 31;             // pair slot of the lane's rows
    JacobiPivot pv[NK];                  // wavefront 0
    int bPR[NB], to01[NB], to23[NB];     // the others: their blocks and where each entry goes
    if (wave == 0) {
#pragma unroll
        for (int j = 0; j < NK; ++j) pv[j].place(half, lane + 64 * j);
    } else {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            int P, R, to[4];
            tri_index(ut + j * kNU < nblk ? ut + j * kNU : 0, P, R);
            bPR[j] = P | (R << 16);
            block_moves(half, nblk, P, R, to);
            to01[j] = to[0] | (to[1] << 16);
            to23[j] = to[2] | (to[3] << 16);
        }
    }
    for (int r = 0; r < m - 1; ++r, f ^= 1) {
        const double2* rf = jb.rot + f * half;
        double nn[NB][4];
        int any = 0;
        if (wave == 0) {
#pragma unroll
            for (int j = 0; j < NK; ++j) pv[j].load(blk, nblk, rf);
        } else {
            if (NR) any = qx_uniform(jb.any[r]);
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const int b = ut + j * kNU;
                if (b >= nblk) continue;
                const int P = bPR[j] & 0xffff, R = bPR[j] >> 16;
                double bb[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) bb[e] = blk[e * nblk + b];
                if (P == R) bb[2] = bb[1];
                rotate_block(rf[P], rf[R], P == R, bb, nn[j]);
            }
        }
        qx_lds_barrier();
        if (wave == 0) {
            bool turn = false;
#pragma unroll
            for (int j = 0; j < NK; ++j) {
                const double2 cs = pv[j].rotation(half, tol, min_s);
                const int kp = lane + 64 * j;
                if (kp < half) {
                    turn = turn || cs.y != 0.0;
                    jb.rot[(f ^ 1) * half + kp] = cs;
                    if (!NR && r + 1 < m - 1) jb.log[(r + 1) * half + kp] = cs;
                }
            }
            turn = qx_any(turn);
            if (lane == 0) jb.any[r + 1] = turn;
        } else {
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                if (ut + j * kNU >= nblk) continue;
                blk[to01[j] & 0xffff] = nn[j][0];
                blk[(unsigned)to01[j] >> 16] = nn[j][1];
                blk[to23[j] & 0xffff] = nn[j][2];
                blk[(unsigned)to23[j] >> 16] = nn[j][3];
            }
            if (NR) {
                const double2 cs = rf[k < half ? k : 0];
                const double sg = k == 0 ? -cs.y : cs.y;
#pragma unroll
                for (int u = 0; u < NR; ++u) {
                    if (2 * (wave - 1 + NW * u) >= nrow) continue;
                    double px = x[u], py = y[u];
                    if (any) {
                        px = cs.x * x[u] - sg * y[u];
                        py = sg * x[u] + cs.x * y[u];
                    }
                    const double up = qx_lane_up(px, 0.0), down = qx_lane_down(py, 0.0);
                    x[u] = k == 0 ? px : k == half - 1 ? py : up;
                    y[u] = half == 1 ? py : k == 0 ? up : down;
                }
            }
        }
        qx_lds_barrier();
    }
}

// The same with the blocks in global memory (systems too large for LDS): read
// from one buffer, written to the other.
QX_DEV void jacobi_rounds_global(const JacobiBuffers& jb, int m, double tol, double min_s, int& f, int& g)
{
    constexpr int kNU = kNT - 64;
    const int tid = qx_tid(), lane = tid & 63, wave = qx_wave(tid), ut = tid - 64;
    const int half = m / 2, nblk = half * (half + 1) / 2;
    for (int r = 0; r < m - 1; ++r, f ^= 1, g ^= 1) {
        const double2* rf = jb.rot + f * half;
        const double* src = jb.gblk[g];
        double* dst = jb.gblk[g ^ 1];
        if (wave == 0) {
            bool turn = false;
            for (int k = lane; k < half; k += 64) {
                JacobiPivot pv;
                pv.place(half, k);
                pv.load(src, nblk, rf);
                const double2 cs = pv.rotation(half, tol, min_s);
                turn = turn || cs.y != 0.0;
                jb.rot[(f ^ 1) * half + k] = cs;
                if (r + 1 < m - 1) jb.log[(r + 1) * half + k] = cs;
            }
            turn = qx_any(turn);
            if (lane == 0) jb.any[r + 1] = turn;
        } else {
            for (int b = ut; b < nblk; b += kNU) {
                int P, R, to[4];
                tri_index(b, P, R);
                block_moves(half, nblk, P, R, to);
                double bb[4], nn[4];
                for (int e = 0; e < 4; ++e) bb[e] = src[e * nblk + b];
                if (P == R) bb[2] = bb[1];
                rotate_block(rf[P], rf[R], P == R, bb, nn);
                for (int e = 0; e < 4; ++e) dst[to[e]] = nn[e];
            }
        }
        __syncthreads();
    }
}

// Columns of the nrow x m matrix Cv rotated by the logged sweep, m <= 2 NL NS.
// 64 / NL rows share a wavefront, NL lanes each; a lane holds NS consecutive
// pair slots of its row in registers, the players as in jacobi_rounds (x the p and y
// the q players, in slot 0 the other way round), so that in the move after a
// round only one player of x and one of y change the lane and the others the
// register.  NR such sets of rows at a time.  Without barriers, and with one LDS
// read (whether the round rotates anything), a round is bound by the
// instructions issued.  More than one pair (m > 2: smaller systems have their
// rows in registers).
// (Cycles a round with one row per wavefront and slots 64 apart -> now: 132
// rows and columns 6.0 k -> 2.9 k, where the second set had used 2 lanes of 64;
// 88: 1.75 k -> 1.50 k.)
template <int NL, int NS, int NR>
QX_DEV void jacobi_replay(const JacobiBuffers& jb, double* Cv, int m, int nrow, int lda)
{
    constexpr int NG = 64 / NL, NW = kNT / 64;
    const int tid = qx_tid(), lane = tid & 63, wave = qx_wave(tid), half = m / 2;
    const int s0 = (lane & (NL - 1)) * NS;
    const bool first = s0 == 0;
    for (int i0 = 0; i0 < nrow; i0 += NG * NW * NR) {
        // lanes without a row read the wavefront's first one
        const int own = i0 + NG * wave;
        if (own >= nrow) break;
        double x[NR][NS], y[NR][NS];
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            const int row = i0 + NG * (wave + NW * u) + lane / NL, i = row < nrow ? row : own;
#pragma unroll
            for (int t = 0; t < NS; ++t) {
                const int k = s0 + t < half ? s0 + t : half - 1;
                x[u][t] = Cv[i * lda + (k == 0 ? m - 1 : k)];
                y[u][t] = Cv[i * lda + (k == 0 ? 0 : m - 1 - k)];
            }
        }
        double2 cs[NS];
        auto fetch = [&](int r) {
#pragma unroll
            for (int t = 0; t < NS; ++t) {
                const int k = s0 + t < half ? s0 + t : half - 1;
                cs[t] = jb.log[r * half + k];
            }
        };
        fetch(0);
        for (int r = 0; r < m - 1; ++r) {
            double2 cr[NS];
#pragma unroll
            for (int t = 0; t < NS; ++t) cr[t] = cs[t];
            if (first) cr[0].y = -cr[0].y;
            if (r + 1 < m - 1) fetch(r + 1);
            const bool any = qx_uniform(jb.any[r]);
#pragma unroll
            for (int u = 0; u < NR; ++u) {
                if (i0 + NG * (wave + NW * u) >= nrow) continue;
                double px[NS], py[NS];
#pragma unroll
                for (int t = 0; t < NS; ++t) {
                    px[t] = x[u][t];
                    py[t] = y[u][t];
                    if (any) {
                        px[t] = cr[t].x * x[u][t] - cr[t].y * y[u][t];
                        py[t] = cr[t].y * x[u][t] + cr[t].x * y[u][t];
                    }
                }
                const double xin = qx_lane_up(px[0], 0.0), yin = qx_lane_down(py[NS - 1], 0.0);
#pragma unroll
                for (int t = 0; t < NS; ++t) {
                    const double down = t + 1 < NS ? px[t + 1 < NS ? t + 1 : t] : xin;
                    const double up = t > 0 ? py[t > 0 ? t - 1 : 0] : yin;
                    x[u][t] = s0 + t == half - 1 ? py[t] : t == 0 && first ? px[0] : down;
                    y[u][t] = t == 0 && first ? px[1] : up;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            const int i = i0 + NG * (wave + NW * u) + lane / NL;
#pragma unroll
            for (int t = 0; t < NS; ++t) {
                const int k = s0 + t;
                if (i < nrow && k < half) {
                    Cv[i * lda + (k == 0 ? m - 1 : k)] = x[u][t];
                    Cv[i * lda + (k == 0 ? 0 : m - 1 - k)] = y[u][t];
                }
            }
        }
    }
}

// Parallel cyclic threshold Jacobi on symmetric A (m x m, m even, leading
// dimension lda).  Pairs with |a_pq| < tol, or whose rotation has |sin| <=
// min_s, are not rotated; the sweeps end when no off-diagonal element of the
// result reaches tol, at the latest after maxsweep.  The rotations are also
// applied to the columns of the nrow x m matrix Cv (leading dimension lda),
// so Cv ends as Cv V with A = V^T A_in V diagonal.
//
// What bounds a round is the latency of its rotations (two reciprocal roots
// in a row on one pivot per lane) and the number of instructions that the
// other wavefronts issue.  So A is kept as 2 x 2 blocks by seats of the
// round-robin: every address of a thread is the same in every round, a block
// is four conflict-free reads and four writes to where its players sit next.
// Wavefront 0 does nothing but the pivots: while the others apply round r it
// forms the three entries of each pivot of round r + 1 from the blocks they
// come from and their rotation.  One barrier keeps the reads of a round
// before its writes, one ends it.  Up to 64 columns the other wavefronts also
// rotate Cv, held in registers; above that the rotations of a sweep are
// logged and applied to Cv afterwards, without barriers.
template <int NB, int NR>
QX_DEV int jacobi(double* A, double* Cv, int m, int nrow, int lda, double tol, int maxsweep, double min_s,
                  const JacobiBuffers& jb)
{
    constexpr int NW = kNT / 64 - 1;
    constexpr bool LDS = NB > 0, rows = NR > 0;
    const int half = m / 2, nblk = half * (half + 1) / 2;
    if (qx_uniform(offdiag_max(A, m, lda, jb.red) < tol)) return 0;
    const int tid = qx_tid(), lane = tid & 63, wave = qx_wave(tid);
    int sweep = 0, f = 0, g = 0;
    double* blk = LDS ? jb.blk : jb.gblk[0];
    double x[NR ? NR : 1], y[NR ? NR : 1];
    // rows of Cv in registers (jacobi_rounds): row and columns of a lane
    auto rows_lane = [&](int u, int& i, int& cx, int& cy) {
        const int k = lane & 31;
        i = 2 * (wave - 1 + NW * u) + (lane >> 5);
        cx = k == 0 ? m - 1 : k;
        cy = k == 0 ? 0 : m - 1 - k;
        return wave > 0 && i < nrow && k < half;
    };
    for (int b = tid; b < nblk; b += kNT) {
        int P, R;
        int2 p, r;
        tri_index(b, P, R);
        rr_pair(m, 0, P, p.x, p.y);
        rr_pair(m, 0, R, r.x, r.y);
        blk[b] = A[p.x * lda + r.x];
        blk[nblk + b] = A[p.x * lda + r.y];
        blk[2 * nblk + b] = A[p.y * lda + r.x];
        blk[3 * nblk + b] = A[p.y * lda + r.y];
    }
    if (rows) {
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            int i, cx, cy;
            const bool in = rows_lane(u, i, cx, cy);
            x[u] = in ? Cv[i * lda + cx] : 0.0;
            y[u] = in ? Cv[i * lda + cy] : 0.0;
        }
    }
    __syncthreads();
    if (wave == 0) {
        bool turn = false;
        for (int k = lane; k < half; k += 64) {
            const int b = k * (k + 1) / 2 + k;
            const double2 cs = pivot_rotation(blk[b], blk[3 * nblk + b], blk[nblk + b], tol, min_s);
            turn = turn || cs.y != 0.0;
            jb.rot[k] = cs;
        }
        turn = qx_any(turn);
        if (lane == 0) jb.any[m - 1] = turn;
    }
    __syncthreads();
    while (sweep < maxsweep) {
        ++sweep;
        // round 0 of this sweep (its rotations come from the sweep before)
        if (!rows)
            for (int k = tid; k < half; k += kNT) jb.log[k] = jb.rot[f * half + k];
        if (tid == 0) jb.any[0] = jb.any[m - 1];
        __syncthreads();
        if constexpr (LDS) jacobi_rounds<NB, NR>(jb, m, nrow, tol, min_s, x, y, f);
        else jacobi_rounds_global(jb, m, tol, min_s, f, g);
        if (!LDS) blk = jb.gblk[g];
        if constexpr (!rows) {
            __syncthreads();
            // sizes of the instantiation (jacobi_any): up to 102, 132, 256; the
            // split that gives the longest wavefront the fewest rotations
            if constexpr (NB == 3) {
                if (m <= 96) jacobi_replay<16, 3, 3>(jb, Cv, m, nrow, lda);
                else jacobi_replay<8, 7, 2>(jb, Cv, m, nrow, lda);
            } else if constexpr (NB == kMaxNB) {
                jacobi_replay<16, 5, 5>(jb, Cv, m, nrow, lda);
            } else {
                jacobi_replay<16, 8, 2>(jb, Cv, m, nrow, lda);
            }
        }
        if (sweep < maxsweep) {
            double mx = 0.0;
            for (int b = tid; b < nblk; b += kNT) {
                int P, R;
                tri_index(b, P, R);
                mx = fmax(mx, fabs(blk[nblk + b]));
                if (P != R) mx = fmax(fmax(mx, fabs(blk[b])), fmax(fabs(blk[2 * nblk + b]), fabs(blk[3 * nblk + b])));
            }
            if (qx_uniform(block_max(mx, jb.red) < tol)) break;
        }
    }
    __syncthreads();
    for (int b = tid; b < nblk; b += kNT) {
        int P, R;
        int2 p, r;
        tri_index(b, P, R);
        rr_pair(m, 0, P, p.x, p.y);
        rr_pair(m, 0, R, r.x, r.y);
        const double n[4] = {blk[b], blk[nblk + b], blk[P == R ? nblk + b : 2 * nblk + b], blk[3 * nblk + b]};
        A[p.x * lda + r.x] = n[0];
        A[p.x * lda + r.y] = n[1];
        A[p.y * lda + r.x] = n[2];
        A[p.y * lda + r.y] = n[3];
        if (P == R) continue;
        A[r.x * lda + p.x] = n[0];
        A[r.y * lda + p.x] = n[1];
        A[r.x * lda + p.y] = n[2];
        A[r.y * lda + p.y] = n[3];
    }
    if (rows) {
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            int i, cx, cy;
            if (rows_lane(u, i, cx, cy)) {
                Cv[i * lda + cx] = x[u];
                Cv[i * lda + cy] = y[u];
            }
        }
    }
    __syncthreads();
    return sweep;
}

// jacobi() in the form for the system: rows of Cv in registers up to 64
// columns, blocks per thread by the number of blocks, or the blocks in global
// memory when they do not fit in LDS
template <bool FAST>
QX_DEV int jacobi_any(double* A, double* Cv, int m, int nrow, int lda, double tol, int maxsweep, double min_s,
                      const JacobiBuffers& jb)
{
    constexpr int kNU = kNT - 64, kRows = 2 * (kNT / 64 - 1);  // rows of Cv per register pair
    const int nblk = (m / 2) * (m / 2 + 1) / 2;
    if (FAST) return jacobi<1, (kFastM + kRows - 1) / kRows>(A, Cv, m, nrow, lda, tol, maxsweep, min_s, jb);
    if (!jb.lds) return jacobi<0, 0>(A, Cv, m, nrow, lda, tol, maxsweep, min_s, jb);
    if (m <= 64) return jacobi<2, (64 + kRows - 1) / kRows>(A, Cv, m, nrow, lda, tol, maxsweep, min_s, jb);
    if (nblk <= 3 * kNU) return jacobi<3, 0>(A, Cv, m, nrow, lda, tol, maxsweep, min_s, jb);
    return jacobi<kMaxNB, 0>(A, Cv, m, nrow, lda, tol, maxsweep, min_s, jb);
}

constexpr double kCoarseSin = 0.02;  // |sin| of the rotations a coarse sweep applies
constexpr int kCoarseSweeps = 3;      // coarse sweeps before the refinement gives up

// Eigenvectors of a symmetric A (m x m, leading dimension lda) to
// off-diagonals below tol, Cv <- Cv V (nrow x m).
//
// With T (a fifth matrix), simultaneous rotations by FP64 MFMA products come
// first.  Every pair (i, j) gets the angle of the Jacobi rotation that would
// zero a_ij alone; with K the antisymmetric matrix of the angles,
// Y = I + K (+ K^2 / 2 when max |K| > 1e-4 or <= 1e-5) is orthogonal up to
// O(K^2) (O(K^4)), and none, one or two Newton-Schulz steps
// R <- R (3 I - R^T R) / 2 make it orthogonal to rounding.  Then
// A <- R^T A R and Cv <- Cv R.  The off-diagonal decreases quadratically
// (errors of the simultaneous angles are second order in the off-diagonal
// over the eigenvalue gaps).  An angle above 0.1 (near-degenerate pairs with
// a relatively large coupling, typically at the first SCC iteration after
// the geometry moved: the series would need more terms) calls for a coarse
// Jacobi sweep that rotates only the pairs whose rotation has |sin| >
// kCoarseSin, up to kCoarseSweeps times; from the first one on, pairs with a
// coupling below tol are left alone, as Jacobi leaves them.  When the angles
// stay above 0.1, kRounds rounds did not suffice or there is no T, full
// Jacobi sweeps finish (or do it all).
// Y, Z, T: m x m scratch (leading dimension lda; T may be null).  Called by
// all threads.  Returns the number of full Jacobi sweeps.
constexpr int kRounds = 3;
template <bool EIG, bool FAST>
QX_DEV int eig_solve(double* A, double* Cv, int m, int nrow, int lda, double tol, double* Y, double* Z,
                     double* T, const JacobiBuffers& jb)
{
    double* red = jb.red;
    int coarse = 0, rounds = 0;
    bool refine = EIG && T;
    if (refine && qx_uniform(offdiag_max(A, m, lda, red) < tol)) return 0;
    for (;;) {
        const int tid = qx_tid();
        int sweeps = 50;
        double min_s = 0.0;
        if (refine && rounds < kRounds) {
            // one angle per pair i < j (K_ji = -K_ij): rows r and m - 1 - r of
            // the upper triangle together hold m - 1 pairs, so pair b maps to
            // (r, c) = (b / (m - 1), b % (m - 1)) without a square root (m even)
            double kmax = 0.0;
            for (int b = tid; b < (m / 2) * (m - 1); b += kNT) {
                const int r = b / (m - 1), c = b - r * (m - 1);
                const bool first = c < m - 1 - r;
                const int i = first ? r : m - 1 - r;
                const int j = first ? r + 1 + c : m - r + (c - (m - 1 - r));
                const double a = A[i * lda + j];
                const double d = A[j * lda + j] - A[i * lda + i];
                const double rr = sqrt(d * d + 4.0 * a * a);
                const double t = rr > 0.0 ? 2.0 * (d >= 0.0 ? a : -a) / (fabs(d) + rr) : 0.0;
                // after a coarse sweep, pairs below tol are left alone as Jacobi leaves them
                const double th = (coarse && fabs(a) < tol) ? 0.0 : atan(t);
                Y[i * lda + j] = th;
                Y[j * lda + i] = -th;
                kmax = fmax(kmax, fabs(th));
            }
            for (int i = tid; i < m; i += kNT) Y[i * lda + i] = 0.0;
            kmax = block_max(kmax, red);
            if (qx_uniform(kmax <= 0.1)) {
                // Y = I + K + K^2/2 has Y^T Y = I + K^4/4: with max |K| <= 1e-5
                // that is below rounding and no Newton-Schulz step is needed
                const bool quad = qx_uniform(kmax > 1e-4 || kmax <= 1e-5);
                const int nns = qx_uniform(kmax > 0.005 ? 2 : (kmax > 1e-5 ? 1 : 0));
                // the products one after the other (one copy of the product's
                // code): K K, then per Newton-Schulz step R^T R and R Z, then
                // A R, R^T (A R) and Cv R
                double* R = Y;
                double* W = T;
                const int last = 1 + 2 * nns + 3;
                for (int s = quad ? 0 : 1; s < last; ++s) {
                    const int k = s == 0 ? 0 : s < 1 + 2 * nns ? 1 + ((s - 1) & 1) : 3 + (s - 1 - 2 * nns);
                    if (s == 1) {
                        for (int p = tid; p < m * m; p += kNT) {
                            const int i = p / m, j = p - i * m, o = i * lda + j;
                            Y[o] = (i == j ? 1.0 : 0.0) + Y[o] + (quad ? 0.5 * Z[o] : 0.0);
                        }
                        __syncthreads();
                    }
                    const double* pa = k == 3 ? A : k == 5 ? Cv : R;
                    const bool ta = k == 1 || k == 4;
                    const double* pb = k == 2 ? Z : k == 4 ? W : R;
                    double* pc = k == 2 ? W : k == 3 ? W : k == 4 ? A : Z;
                    mfma_gemm(k == 5 ? nrow : m, m, m, pa, ta ? 1 : lda, ta ? lda : 1, pb, lda, 1, pc, lda, nullptr,
                                   k == 0 || k == 1 || k == 4);
                    if (k != 4) __syncthreads();  // Cv R reads nothing that R^T W writes
                    if (k == 1) {
                        for (int p = tid; p < m * m; p += kNT) {
                            const int i = p / m, j = p - i * m, o = i * lda + j;
                            Z[o] = (i == j ? 1.5 : 0.0) - 0.5 * Z[o];
                        }
                        __syncthreads();
                    } else if (k == 2) {
                        double* t = R;
                        R = W;
                        W = t;
                    }
                }
                for (int p = tid; p < nrow * m; p += kNT) {
                    const int i = p / m, j = p - i * m;
                    Cv[i * lda + j] = Z[i * lda + j];
                }
                __syncthreads();
                ++rounds;
                if (qx_uniform(offdiag_max(A, m, lda, red) < tol)) return 0;
                continue;
            }
            // strongly coupled pairs (near-degenerate orbitals after the
            // geometry moved): one Jacobi sweep over the pairs whose rotation
            // exceeds kCoarseSin, then the simultaneous rotations again
            if (coarse < kCoarseSweeps) {
                ++coarse;
                sweeps = 1;
                min_s = kCoarseSin;
            }
        }
        const int done = jacobi_any<FAST>(A, Cv, m, nrow, lda, tol, sweeps, min_s, jb);
        if (sweeps != 1) return done;
        QX_PH_ADD(jb.sys, 29, 1);
    }
}

// The Broyden weights of n secant pairs by the whole block: solves (B) x = g
// for the n x n symmetric positive definite B in rows 0 .. n - 1 of bt (lower
// triangle, leading dimension st) with g as row n, and returns x in gm.
// B = U D^-1 U^T column by column without roots (column j of U is the column
// as the elimination reaches it), one barrier per column; g eliminated along
// with it is the forward substitution.  The backward substitution is on
// wavefront 0, a lane per column (two for n > 64).  n <= 128.
QX_DEV void broyden_solve(double* bt, int st, double* gm, int n)
{
    const int tid = qx_tid(), lane = tid & 63;
    const int ti = tid >> 4, tk = tid & 15;
    for (int j = 0; j < n; ++j) {
        const double inv = 1.0 / bt[j * st + j];
        for (int i = j + 1 + ti; i <= n; i += kNT / 16) {
            const double l = bt[i * st + j] * inv;
            for (int k = j + 1 + tk; k <= i && k < n; k += 16) bt[i * st + k] -= l * bt[k * st + j];
        }
        __syncthreads();
    }
    if (tid < 64) {
        const int j0 = lane < n ? lane : n - 1, j1 = lane + 64 < n ? lane + 64 : n - 1;
        double y0 = bt[n * st + j0], y1 = bt[n * st + j1];
        const double d0 = 1.0 / bt[j0 * st + j0], d1 = 1.0 / bt[j1 * st + j1];
        for (int i = n - 1; i >= 0; --i) {
            const double x = i < 64 ? qx_bcast(y0 * d0, i) : qx_bcast(y1 * d1, i - 64);
            const double* u = bt + i * st;
            if (lane == 0) gm[i] = x;
            if (j0 < i) y0 -= u[j0] * x;
            if (j1 < i) y1 -= u[j1] * x;
        }
    }
    __syncthreads();
}

// Fermi occupations per spin on wavefront 0 for nalpha electrons; returns -TS.
// The chemical potential is found by Newton steps safeguarded by a bracket
// (bisection whenever a step leaves it), starting from mu_io when it lies
// inside the bracket, until the electron count is met to 1e-13 relative, and
// polished by one more Newton step; the root is written back to mu_io.
QX_DEV double fermi_wave(int n, const double* e, double kt, double nalpha, double* f, double& mu_io,
                         int& iters)
{
    const int l = threadIdx.x & 63;
    const double ikt = 1.0 / kt;
    double lo = 1e300, hi = -1e300;
    for (int i = l; i < n; i += 64) {
        lo = fmin(lo, e[i]);
        hi = fmax(hi, e[i]);
    }
    lo = -wave_max(-lo);
    hi = wave_max(hi);
    lo = lo - 50.0 * kt - 1.0;
    hi = hi + 50.0 * kt + 1.0;
    double mu = (mu_io > lo && mu_io < hi) ? mu_io : 0.5 * (lo + hi);
    iters = 0;
    for (int it = 0; it < 300; ++it) {
        ++iters;
        double s = 0.0, ds = 0.0;
        for (int i = l; i < n; i += 64) {
            const double fi = 1.0 / (1.0 + exp((e[i] - mu) * ikt));
            s += fi;
            ds += fi * (1.0 - fi);
        }
        s = wave_sum(s);
        ds = wave_sum(ds) * ikt;
        const double diff = nalpha - s;
        if (fabs(diff) <= 1e-13 * fmax(nalpha, 1.0)) {
            if (ds > 0.0) mu += diff / ds;  // final Newton polish
            break;
        }
        if (s > nalpha) hi = mu;
        else lo = mu;
        double mun = (ds > 0.0) ? mu + diff / ds : 0.5 * (lo + hi);
        if (!(mun > lo && mun < hi)) mun = 0.5 * (lo + hi);
        mu = mun;
        if (hi - lo <= 1e-15 * (fabs(mu) + 1.0)) break;
    }
    double ts = 0.0;
    for (int i = l; i < n; i += 64) {
        const double fi = 1.0 / (1.0 + exp((e[i] - mu) * ikt));
        f[i] = fi;
        if (fi > 0.0 && fi < 1.0) ts += fi * log(fi) + (1.0 - fi) * log(1.0 - fi);
    }
    mu_io = mu;
    return 2.0 * kt * wave_sum(ts);
}

struct SysShared {
    ShellDesc sh[QX_MAX_NSH];
    int ao_at[QX_MAX_NAO], ao_sh[QX_MAX_NAO];
    int shoff[QX_MAX_NAT + 1], aooff[QX_MAX_NAT + 1];  // shells/AOs of atom a: [off[a], off[a+1])
    int sel[QX_MAX_NAT], refoff[QX_MAX_NAT + 1];
    unsigned char refat[kMaxRef];          // atom of a D4 reference
    int eroff[gfn2::kElem + 1];            // D4 references of the elements present: [off[e], off[e+1])
    double sx[3 * QX_MAX_NAT];
    double mrad[QX_MAX_NAT];
    double qat[QX_MAX_NAT];
    // D4 references inside potentials(); between its calls the same LDS holds
    // the Jacobi rotations, its round flags and the Broyden weights
    union {
        struct {
            double zr[kMaxRef], dzr[kMaxRef], yr[kMaxRef];
        };
        struct {
            alignas(16) double rot[2 * QX_MAX_NAO];  // (c, s) pairs of two rounds
            int any[QX_MAX_NAO];
            double gm[128];  // at most `mem` <= 100 pairs
        };
    };
    double red[8 * (kNT / 64)];
    double eparts[6];  // es2, es3, aes, axc, d4, unused
};

// LDS doubles potentials() works in: inner D4 sums, multipole shares
inline __host__ __device__ int pot_lds(int nat)
{
    return gfn2::kElem * QX_MAX_REF * nat + (nat <= 32 ? 80 : 40) * nat;
}

// What a thread needs from the parameter tables in every call: of its D4
// reference (thread k: reference k), its shell's Coulomb row (from the last
// thread on) and its atom's on-site multipole kernels.
struct PotTables {
    double c, qref, zeff, gw, third, dk, qk;

    QX_DEV void load(const SysInfo& si, BatchRef B, const SysShared& ss)
    {
        static_assert(kMaxRef <= kNT && QX_MAX_NSH <= kNT - 256, "one reference and one shell per thread");
        const int tid = qx_tid();
        c = qref = zeff = gw = third = dk = qk = 0.0;
        if (tid < si.ndim) {
            const int a = ss.refat[tid];
            const ElemParams& e = g_tab.e[ss.sel[a]];
            c = e.gam * gfn2::kD4Gc;
            qref = e.refq[tid - ss.refoff[a]] + e.zeff;
            zeff = e.zeff;
            gw = B.gw[si.ref_off + tid];
        }
        const int a = kNT - 1 - tid;
        if (a < si.nsh) third = g_tab.e[ss.sh[a].el].third[ss.sh[a].k];
        if (tid < si.nat) {
            dk = g_tab.e[ss.sel[tid]].dkernel;
            qk = g_tab.e[ss.sel[tid]].qkernel;
        }
    }
};

// Potentials vs (per shell), vd (3 per atom), vq (6 per atom) and, with
// energy set, interaction energies (ES2, ES3, AES, AXC, D4 two-body) at
// moments x = [qsh, dp, qp].
// The D4 response of reference k of atom i is
//   y_k = gw_k sum_j disp_ij sum_(l of j) C6ref_kl gw_l z_l,
// whose inner sum depends on i through its element and reference number only:
// it is formed once per (element, reference, atom j), which leaves nat
// terms per reference instead of ndim, and nat^2 values to read instead of
// ndim^2.  The multipole terms read two damped kernels per atom pair (1/r^3
// and 1/r^5) and take the directions from the coordinates.  First the
// wavefronts 0 .. 3 sum the multipole terms of a share of the partners each
// (half-wavefronts up to 32 atoms) while the others form the inner D4 sums
// and the shell Coulomb potential gamma q; then the shares are added up, a
// thread per atom and term, and the outer D4 sums taken, four threads per
// reference; then the atoms' terms are put together.  A call is bound by the
// instructions on its longest wavefront, not by memory, so what is read from
// memory is under way before it is needed and the tables' values are kept in
// registers.  The AES energy is x . v_aes / 2 (the multipole energy is a
// symmetric bilinear form of the moments).  scr: LDS, pot_lds(nat) doubles.
// (26-atom C8H18+, 50 basis functions: 20-30 k cycles a call with one
// multipole wavefront, ten kernel planes and the ndim^2 response matrix, 15 k
// now, 18 k with the energies.)
QX_DEV void potentials(const SysInfo& si, BatchRef B, SysShared& ss, const PotTables& pt, const double* x, double* vs,
                       double* vd, double* vq, double* scr, bool energy)
{
    const int tid = qx_tid(), lane = tid & 63, wave = qx_wave(tid);
    const int nat = si.nat, nsh = si.nsh, nd = si.ndim, nn = nat * nat;
    const double* qsh = x;
    const double* dp = x + nsh;
    const double* qp = x + nsh + 3 * nat;
    constexpr int na = 4;          // multipole wavefronts
    const bool split = nat <= 32;  // two half-wavefronts of atoms
    const int nparts = split ? 2 * na : na;
    const int ner = qx_uniform(ss.eroff[gfn2::kElem]);
    double* tt = scr;             // ner x nat inner D4 sums
    double* pa = tt + ner * nat;  // nparts x 10 x nat multipole shares
    const double* pk = B.pairk + (size_t)si.pair_off / QX_PAIR_STRIDE * QX_PAIR_KERN;
    // what the first pass of each wavefront reads from memory, on its way
    // while the charges and D4 references are formed: kernels of the first
    // NJ partners, or the C6 row of the first inner D4 sum and the start of
    // the Coulomb row
    constexpr int NJ = 4, NB = 8;
    const int t0 = tid - 64 * na, nt = kNT - 64 * na;
    const int ai = split ? (lane & 31) : lane;
    const int part = split ? 2 * wave + (lane >> 5) : wave;
    const int len = (nat + nparts - 1) / nparts, pj0 = part * len, pj1 = pj0 + len < nat ? pj0 + len : nat;
    const double* G = B.gam + si.gam_off;
    const int ga = kNT - 1 - tid;  // Coulomb row, from the last thread on
    auto c6row = [&](int p) {
        const int er = p / nat, j = p - er * nat;
        int e = 0;
        while (ss.eroff[e + 1] <= er) ++e;
        return g_tab.c6ref[e][er - ss.eroff[e]][ss.sel[j]];
    };
    double h3[NJ], h5[NJ], c6[QX_MAX_REF], gr[NB];
    auto kernels = [&](int jb) {
#pragma unroll
        for (int u = 0; u < NJ; ++u) {
            const int j = jb + u < pj1 ? jb + u : ai;  // (i, i) is zero
            h3[u] = pk[j * nat + ai];
            h5[u] = pk[nn + j * nat + ai];
        }
    };
    auto coulomb = [&](int b0) {
#pragma unroll
        for (int u = 0; u < NB; ++u) gr[u] = G[(b0 + u < nsh ? b0 + u : b0) * nsh + ga];
    };
    if (wave < na) {
        if (ai < nat) kernels(pj0);
    } else {
        const double* c = c6row(t0 < ner * nat ? t0 : 0);
#pragma unroll
        for (int l = 0; l < QX_MAX_REF; ++l) c6[l] = c[l];
        if (ga < nsh) coulomb(0);
    }
    qx_sched_fence();
    for (int a = tid; a < nat; a += kNT) {
        double q = 0.0;
        for (int s = ss.shoff[a]; s < ss.shoff[a + 1]; ++s) q += qsh[s];
        ss.qat[a] = q;
    }
    __syncthreads();
    if (tid < nd) {
        double z, dz;
        d4_zeta_both(gfn2::kD4Ga, pt.c, pt.qref, ss.qat[ss.refat[tid]] + pt.zeff, z, dz);
        ss.zr[tid] = z * pt.gw;
        ss.dzr[tid] = dz * pt.gw;
    }
    __syncthreads();
    double eaes = 0.0, eaxc = 0.0, es2 = 0.0, es3 = 0.0, ed4 = 0.0;
    if (wave < na) {
        const int i = ai;
        double v0 = 0.0, d0 = 0.0, d1 = 0.0, d2 = 0.0;
        double w0 = 0.0, w1 = 0.0, w2 = 0.0, w3 = 0.0, w4 = 0.0, w5 = 0.0;
        if (i < nat) {
            const double x0 = ss.sx[3 * i], x1 = ss.sx[3 * i + 1], x2 = ss.sx[3 * i + 2];
            for (int jb = pj0; jb < pj1; jb += NJ) {
                if (jb > pj0) {
                    kernels(jb);
                    qx_sched_fence();
                }
#pragma unroll
                for (int u = 0; u < NJ; ++u) {
                    if (jb + u >= pj1) continue;
                    const int j = jb + u;
                    const double rv0 = x0 - ss.sx[3 * j], rv1 = x1 - ss.sx[3 * j + 1], rv2 = x2 - ss.sx[3 * j + 2];
                    const double r2 = rv0 * rv0 + rv1 * rv1 + rv2 * rv2;
                    const double g0 = h3[u] * rv0, g1 = h3[u] * rv1, g2 = h3[u] * rv2;
                    const double t0 = h5[u] * rv0, t1 = h5[u] * rv1;
                    const double g3 = t0 * rv0, g4 = t0 * rv1, g5 = t1 * rv1, g6 = t0 * rv2, g7 = t1 * rv2,
                                 g8 = h5[u] * rv2 * rv2, g9 = r2 * h5[u];
                    const double qj = ss.qat[j];
                    const double m0 = dp[3 * j], m1 = dp[3 * j + 1], m2 = dp[3 * j + 2];
                    const double* t = qp + 6 * j;
                    v0 += m0 * g0 + m1 * g1 + m2 * g2 + t[0] * g3 + 2.0 * t[1] * g4 + t[2] * g5 +
                          2.0 * t[3] * g6 + 2.0 * t[4] * g7 + t[5] * g8;
                    d0 += -qj * g0 + g9 * m0 - 3.0 * (g3 * m0 + g4 * m1 + g6 * m2);
                    d1 += -qj * g1 + g9 * m1 - 3.0 * (g4 * m0 + g5 * m1 + g7 * m2);
                    d2 += -qj * g2 + g9 * m2 - 3.0 * (g6 * m0 + g7 * m1 + g8 * m2);
                    w0 += qj * g3;
                    w1 += qj * g4;
                    w2 += qj * g5;
                    w3 += qj * g6;
                    w4 += qj * g7;
                    w5 += qj * g8;
                }
            }
            double* o = pa + part * 10 * nat + i;
            const double pv[10] = {v0, d0, d1, d2, w0, w1, w2, w3, w4, w5};
#pragma unroll
            for (int k = 0; k < 10; ++k) o[k * nat] = pv[k];
        }
    } else {
        for (int p = t0; p < ner * nat; p += nt) {
            if (p > t0) {
                const double* c = c6row(p);
#pragma unroll
                for (int l = 0; l < QX_MAX_REF; ++l) c6[l] = c[l];
            }
            const int j = p % nat, l0 = ss.refoff[j], nl = ss.refoff[j + 1] - l0;
            double s = 0.0;
#pragma unroll
            for (int l = 0; l < QX_MAX_REF; ++l)
                if (l < nl) s += c6[l] * ss.zr[l0 + l];
            tt[p] = s;
        }
        if (ga < nsh) {
            double v = 0.0;
            for (int b0 = 0; b0 < nsh; b0 += NB) {
                double g[NB];
#pragma unroll
                for (int u = 0; u < NB; ++u) g[u] = gr[u];
                if (b0 + NB < nsh) coulomb(b0 + NB);
                qx_sched_fence();
#pragma unroll
                for (int u = 0; u < NB; ++u)
                    if (b0 + u < nsh) v += g[u] * qsh[b0 + u];
            }
            const double q = qsh[ga];
            es2 += 0.5 * q * v;
            es3 += pt.third * q * q * q / 3.0;
            vs[ga] = v + pt.third * q * q;
        }
    }
    __syncthreads();
    // the multipole shares of one atom and term, into the first share
    for (int p = tid; p < 10 * nat; p += kNT) {
        double v = pa[p];
        for (int w = 1; w < nparts; ++w) v += pa[w * 10 * nat + p];
        pa[p] = v;
    }
    // the outer D4 sums: the four threads of a reference take a share of the
    // atoms each; -dz_k y_k replaces dz_k
    const int slen = (nat + 3) / 4;
    for (int p = kNT - 1 - tid; p < ((4 * nd + 63) & ~63); p += kNT) {  // whole wavefronts
        const int k = p < 4 * nd ? p >> 2 : nd - 1, seg = p & 3, i = ss.refat[k];
        const double* t = tt + (ss.eroff[ss.sel[i]] + k - ss.refoff[i]) * nat;
        const double* dsp = pk + 2 * nn + i;
        const int j0 = seg * slen, j1 = p >= 4 * nd ? j0 : j0 + slen < nat ? j0 + slen : nat;
        double y = 0.0;
        constexpr int ND = 8;
        for (int jb = j0; jb < j1; jb += ND) {
            double ds[ND];
#pragma unroll
            for (int u = 0; u < ND; ++u) ds[u] = dsp[(jb + u < j1 ? jb + u : jb) * nat];
            qx_sched_fence();
#pragma unroll
            for (int u = 0; u < ND; ++u)
                if (jb + u < j1) y += ds[u] * t[jb + u];
        }
        y = quad_sum(y);
        if (seg == 0 && p < 4 * nd) {
            ed4 += -0.5 * ss.zr[k] * y;
            ss.dzr[k] = -ss.dzr[k] * y;
        }
    }
    __syncthreads();
    if (wave == 0) {
        const int i = lane;
        if (i < nat) {
            const double v0 = pa[i], d0 = pa[nat + i], d1 = pa[2 * nat + i], d2 = pa[3 * nat + i];
            const double w0 = pa[4 * nat + i], w1 = 2.0 * pa[5 * nat + i], w2 = pa[6 * nat + i],
                         w3 = 2.0 * pa[7 * nat + i], w4 = 2.0 * pa[8 * nat + i], w5 = pa[9 * nat + i];
            const double qi = ss.qat[i];
            const double mi0 = dp[3 * i], mi1 = dp[3 * i + 1], mi2 = dp[3 * i + 2];
            const double* ti = qp + 6 * i;
            eaes = 0.5 * (qi * v0 + mi0 * d0 + mi1 * d1 + mi2 * d2 + ti[0] * w0 + ti[1] * w1 + ti[2] * w2 +
                          ti[3] * w3 + ti[4] * w4 + ti[5] * w5);
            const double dk = pt.dk, qk = pt.qk;
            eaxc = dk * (mi0 * mi0 + mi1 * mi1 + mi2 * mi2) +
                   qk * (ti[0] * ti[0] + ti[2] * ti[2] + ti[5] * ti[5] +
                         2.0 * (ti[1] * ti[1] + ti[3] * ti[3] + ti[4] * ti[4]));
            vd[3 * i + 0] = d0 + 2.0 * dk * mi0;
            vd[3 * i + 1] = d1 + 2.0 * dk * mi1;
            vd[3 * i + 2] = d2 + 2.0 * dk * mi2;
            vq[6 * i + 0] = w0 + 2.0 * qk * ti[0];
            vq[6 * i + 1] = w1 + 4.0 * qk * ti[1];
            vq[6 * i + 2] = w2 + 2.0 * qk * ti[2];
            vq[6 * i + 3] = w3 + 4.0 * qk * ti[3];
            vq[6 * i + 4] = w4 + 4.0 * qk * ti[4];
            vq[6 * i + 5] = w5 + 2.0 * qk * ti[5];
        }
    } else {
        for (int a = tid - 64; a < nsh; a += kNT - 64) {
            const int at = ss.sh[a].at, k0 = ss.refoff[at], nk = ss.refoff[at + 1] - k0;
            double vdisp = 0.0;
#pragma unroll
            for (int k = 0; k < QX_MAX_REF; ++k)
                if (k < nk) vdisp += ss.dzr[k0 + k];
            vs[a] += pa[at] + vdisp;
        }
    }
    if (energy) {
        double e5[5] = {es2, es3, eaes, eaxc, ed4};
        block_sums<5>(e5, ss.red);
        if (tid == 0)
            for (int k = 0; k < 5; ++k) ss.eparts[k] = e5[k];
    }
    __syncthreads();
}

QX_DEV void load_system(const SysInfo& si, BatchRef B, SysShared& ss)
{
    const int tid = qx_tid(), nt = blockDim.x, nat = si.nat;
    for (int i = tid; i < 3 * nat; i += nt) ss.sx[i] = B.xyz[3 * (size_t)si.atom_off + i];
    for (int i = tid; i < nat; i += nt) {
        ss.sel[i] = B.elem[si.atom_off + i];
        ss.mrad[i] = B.mrad[si.atom_off + i];
    }
    build_shell_tables(si, B.elem, ss.sh, ss.ao_at, ss.ao_sh);
    if (tid == 0) {
        int o = 0, so = 0, ao = 0;
        unsigned present = 0;
        for (int a = 0; a < nat; ++a) {
            const ElemParams& e = g_tab.e[ss.sel[a]];
            present |= 1u << ss.sel[a];
            ss.refoff[a] = o;
            ss.shoff[a] = so;
            ss.aooff[a] = ao;
            for (int r = 0; r < e.nref; ++r) ss.refat[o + r] = (unsigned char)a;
            o += e.nref;
            so += e.nsh;
            ao += (e.nsh == 2) ? 4 : 1;
        }
        ss.refoff[nat] = o;
        ss.shoff[nat] = so;
        ss.aooff[nat] = ao;
        o = 0;
        for (int e = 0; e < gfn2::kElem; ++e) {
            ss.eroff[e] = o;
            if (present >> e & 1) o += g_tab.e[e].nref;
        }
        ss.eroff[gfn2::kElem] = o;
    }
    __syncthreads();
}

struct SccBuffers {
    double *A, *C, *F, *P;  // m x m working matrices (LDS or global), leading dimension ld
    double* rs;             // kRs row sums per AO
    int ld;
    double* E;              // fifth m x m matrix (with LDS matrices: or null)
    double* lds;            // LDS that is free while xin is updated (with LDS matrices from A on)
    int nlds;               // its size in doubles
    double* pot;            // LDS that is free while the potentials are taken (pot_lds doubles)
};

// LDS of one system's SCC
struct SccLds {
    SysShared ss;
    double xin[kMaxNx], xout[kMaxNx], vs[QX_MAX_NSH], vd[3 * QX_MAX_NAT], vq[6 * QX_MAX_NAT];
    double eps[QX_MAX_NAO], focc[QX_MAX_NAO], f2[QX_MAX_NAO];
    double s_e[4];
};

// Modified Broyden update (Johnson) of xin from dq = xout - xin, which is left
// in xout; it: SCC iteration, hcount: secant pairs seen so far.
QX_DEV void broyden_step(const SysInfo& si, double* hist, OptRef opt, const SccBuffers& bf, double* xin,
                         double* xout, double* gm, double* red, int it, int& hcount)
{
    const int tid = qx_tid(), lane = tid & 63, wave = qx_wave(tid);
    const int nx = si.nx, mem = opt.mem;
    double* hdf = hist;
    double* hu = hist + (size_t)mem * nx;
    double* ha = hist + 2 * (size_t)mem * nx;
    double* hom = ha + mem * mem;
    double* hql = hom + mem;
    double* hdql = hql + nx;
    double* hbeta = hdql + nx;
    // secant pairs form a ring of `ring` slots; with opt.keep > 0 a warm
    // start continues from the pairs of the previous call
    const int ring = (opt.keep > 0 && opt.keep < mem) ? opt.keep : mem;
    if (it == 1 && hcount == 0) {
        for (int i = tid; i < nx; i += kNT) {
            const double dq = xout[i] - xin[i];
            hdql[i] = dq;
            hql[i] = xin[i];
            xin[i] = xin[i] + opt.damp * dq;
        }
        __syncthreads();
        return;
    }
    // a new secant pair from this call's previous iterate (it >= 2) into
    // ring slot k1; on the first iteration of a continued call only the
    // kept pairs enter
    const bool add = it >= 2;
    const int k1 = hcount % ring;
    if (add) {
        double nr[2] = {0.0, 0.0};
        for (int i = tid; i < nx; i += kNT) {
            const double dq = xout[i] - xin[i];
            xout[i] = dq;
            const double d = dq - hdql[i];
            hdf[k1 * nx + i] = d;
            nr[0] += d * d;
            nr[1] += dq * dq;
        }
        block_sums<2>(nr, red);
        const double inv = nr[0] > 0.0 ? 1.0 / sqrt(nr[0]) : 0.0;
        for (int i = tid; i < nx; i += kNT) {
            const double d = hdf[k1 * nx + i] * inv;
            hdf[k1 * nx + i] = d;
            hu[k1 * nx + i] = opt.damp * d + inv * (xin[i] - hql[i]);
        }
        if (tid == 0) {
            double w = sqrt(nr[1]);
            w = (w > 0.01 / 100000.0) ? 0.01 / w : 100000.0;
            if (w < 1.0) w = 1.0;
            hom[k1] = w;
        }
        ++hcount;
    } else {
        for (int i = tid; i < nx; i += kNT) xout[i] = xout[i] - xin[i];
    }
    const int it1 = hcount < ring ? hcount : ring;  // live pairs
    __syncthreads();
    // dot products df_i . df_k1 and df_i . dq: wavefront per i
    for (int i = wave; i < it1; i += kNT / 64) {
        double s = 0.0, c = 0.0;
        for (int j = lane; j < nx; j += 64) {
            const double di = hdf[i * nx + j];
            if (add) s += di * hdf[k1 * nx + j];
            c += di * xout[j];
        }
        s = wave_sum(s);
        c = wave_sum(c);
        if (lane == 0) {
            if (add) {
                ha[i * mem + k1] = s;
                ha[k1 * mem + i] = s;
            }
            gm[i] = c;
        }
    }
    __syncthreads();
    // (w0^2 I + diag(om) a diag(om)) x = diag(om) c and the weights
    // diag(om) x, in LDS when the matrix and the right-hand side below it
    // fit, else in global memory
    auto solve = [&](double* bt, int st) {
        for (int p = tid; p < (it1 + 1) * it1; p += kNT) {
            const int i = p / it1, j = p - i * it1;
            bt[i * st + j] = i == it1 ? hom[j] * gm[j] : hom[i] * hom[j] * ha[i * mem + j] + (i == j ? 1e-4 : 0.0);
        }
        __syncthreads();
        broyden_solve(bt, st, gm, it1);
    };
    if ((it1 + 1) * (it1 | 1) <= bf.nlds) solve(bf.lds, it1 | 1);
    else solve(hbeta, mem);
    for (int j = tid; j < nx; j += kNT) {
        const double dq = xout[j];
        double q = xin[j];
        hdql[j] = dq;
        hql[j] = q;
        q += opt.damp * dq;
        for (int i0 = 0; i0 < it1; i0 += 8) {
            double u[8], w[8];
#pragma unroll
            for (int v = 0; v < 8; ++v) {
                const int i = i0 + v < it1 ? i0 + v : i0;
                u[v] = hu[i * nx + j];
                w[v] = hom[i];
            }
            qx_sched_fence();
#pragma unroll
            for (int v = 0; v < 8; ++v)
                if (i0 + v < it1) q -= gm[i0 + v] * w[v] * u[v];
        }
        xin[j] = q;
    }
    __syncthreads();
}

template <bool FAST, bool EIG>
QX_DEV void scc_body(int sys, const SysInfo& si, BatchRef B0, OptRef opt, SysShared& ss, SccBuffers bf,
                     SccLds& L)
{
    const int nat = si.nat, nsh = si.nsh, n = si.nao, ld = si.ld, nx = si.nx;
    const int m = (n + 1) & ~1;
    const int lb = bf.ld;
    const int ms = ld * ld;
    const int warm = qx_uniform(B0.warm[sys]);
    double* A = bf.A;
    double* Cc = bf.C;
    double* Ft = bf.F;
    double* P = bf.P;
    double* rs = bf.rs;
    double* xin = L.xin;
    double* xout = L.xout;
    double *vs = L.vs, *vd = L.vd, *vq = L.vq;
    double* eps = L.eps;
    double* f2 = L.f2;

    QX_PH_INIT
    {
        // initial moments (polynomial extrapolation of order 1-4 over the
        // previous steps' converged moments in MD) and basis C = X U (padding
        // column zero)
        BatchRef B = qx_fresh(B0);
        const int tid = qx_tid();
        double* xg = B.x + si.x_off;
        double* xp = B.xprev + si.x_off;    // converged moments of the step before
        double* xpp = B.xprev2 + si.x_off;  // and of the one before that
        double* xp3 = B.xprev3 + si.x_off;  // and of the one before that
        double* xp4 = B.xprev4 + si.x_off;  // and of the one before that
        for (int i = tid; i < nx; i += kNT) {
            double v = 0.0;
            if (warm >= 5 && opt.extrapolate >= 4)
                v = 5.0 * (xg[i] - xp3[i]) - 10.0 * (xp[i] - xpp[i]) + xp4[i];
            else if (warm >= 4 && opt.extrapolate >= 3) v = 4.0 * (xg[i] + xpp[i]) - 6.0 * xp[i] - xp3[i];
            else if (warm >= 3 && opt.extrapolate >= 2) v = 3.0 * (xg[i] - xp[i]) + xpp[i];
            else if (warm >= 2 && opt.extrapolate >= 1) v = 2.0 * xg[i] - xp[i];
            else if (warm >= 1) v = xg[i];
            xin[i] = v;
            if (warm >= 4) xp4[i] = xp3[i];
            if (warm >= 3) xp3[i] = xpp[i];
            if (warm >= 2) xpp[i] = xp[i];
            if (warm >= 1) xp[i] = xg[i];
        }
        const double* X = B.X + si.mat_off;
        if (warm) {
            mfma_gemm(n, n, n, X, ld, 1, B.U + si.mat_off, ld, 1, Cc, lb, nullptr, false);
        } else {
            for (int p = tid; p < n * n; p += kNT) Cc[(p / n) * lb + p % n] = X[(p / n) * ld + p % n];
        }
        if (m > n)
            for (int i = tid; i < n; i += kNT) Cc[i * lb + n] = 0.0;
        if (tid == 0) L.s_e[1] = -1e300;
    }
    __syncthreads();
    QX_PH(sys, 11);

    PotTables pt;
    pt.load(si, qx_fresh(B0), ss);
    int hcount = 0;
    if (opt.keep > 0 && warm >= 1) {
        const double* hcnt = B0.hist + si.hist_off + 2 * (size_t)opt.mem * nx + 2 * (size_t)opt.mem * opt.mem +
                             2 * (size_t)opt.mem + 2 * (size_t)nx;
        hcount = qx_uniform((int)hcnt[0]);
    }
    const double nalpha = 0.5 * si.nel;
    double eold = 0.0, etot = 0.0, ts = 0.0, eband = 0.0, errp = 1e-3;
    int it = 1, conv = 0;
    // each iteration takes the potentials twice, at the input and at the
    // output moments (one copy of their code)
    for (bool out = false;; out = !out) {
        potentials(si, qx_fresh(B0), ss, pt, out ? xout : xin, vs, vd, vq, bf.pot, out);
        if (!out) {
            QX_PH(sys, 0);
            {
                // G^T (row nu holds G_{mu nu} over mu), then F = H0 - (G + G^T) / 2
                BatchRef B = qx_fresh(B0);
                const double* S = B.S + si.mat_off;
                const double* H = B.H0 + si.mat_off;
                const double* Dm = B.D + 3 * si.mat_off;  // transposed: (mu, nu) at nu * ld + mu
                const double* Qm = B.Q + 6 * si.mat_off;
                const int tid = qx_tid(), wave = qx_wave(tid);
                constexpr int NU = 3;  // rows per batch of loads
                for (int mu = tid & 63; mu < n; mu += 64) {
                    const int am = ss.ao_at[mu];
                    const double w0 = vs[ss.ao_sh[mu]], w1 = vd[3 * am], w2 = vd[3 * am + 1], w3 = vd[3 * am + 2];
                    const double* q = vq + 6 * am;
                    const double w4 = q[0], w5 = q[1], w6 = q[2], w7 = q[3], w8 = q[4], w9 = q[5];
                    for (int nu0 = wave; nu0 < n; nu0 += NU * (kNT / 64)) {
                        double g[NU][10];
#pragma unroll
                        for (int u = 0; u < NU; ++u) {
                            const int nu = nu0 + u * (kNT / 64);
                            const int o = (nu < n ? nu : nu0) * ld + mu;
                            g[u][0] = S[o];
#pragma unroll
                            for (int c = 0; c < 3; ++c) g[u][1 + c] = Dm[c * ms + o];
#pragma unroll
                            for (int c = 0; c < 6; ++c) g[u][4 + c] = Qm[c * ms + o];
                        }
                        qx_sched_fence();
#pragma unroll
                        for (int u = 0; u < NU; ++u) {
                            const int nu = nu0 + u * (kNT / 64);
                            if (nu < n)
                                Ft[nu * lb + mu] = g[u][0] * w0 + g[u][1] * w1 + g[u][2] * w2 + g[u][3] * w3 +
                                                   g[u][4] * w4 + g[u][5] * w5 + g[u][6] * w6 + g[u][7] * w7 +
                                                   g[u][8] * w8 + g[u][9] * w9;
                        }
                    }
                }
                __syncthreads();
                for (int p = tid; p < n * n; p += kNT) {
                    const int mu = p / n, nu = p - mu * n;
                    if (nu < mu) continue;
                    const double gmn = Ft[mu * lb + nu], gnm = Ft[nu * lb + mu];
                    const double f = H[mu * ld + nu] - 0.5 * (gmn + gnm);
                    Ft[mu * lb + nu] = f;
                    Ft[nu * lb + mu] = f;
                }
                __syncthreads();
            }
            QX_PH(sys, 1);
            // A = C^T F C (F C staged in the density buffer)
            for (int s = 0; s < 2; ++s) {
                mfma_gemm(n, n, n, s ? Cc : Ft, s ? 1 : lb, s ? lb : 1, s ? P : Cc, lb, 1, s ? A : P, lb, nullptr,
                          s != 0);
                if (s && m > n)
                    for (int j = qx_tid(); j < m; j += kNT) {
                        A[n * lb + j] = 0.0;
                        A[j * lb + n] = 0.0;
                    }
                __syncthreads();
            }
            QX_PH(sys, 2);
            double jtol = fmin(1e-6, 1e-3 * errp);
            if (jtol < opt.jacobi_tol) jtol = opt.jacobi_tol;
            const int nblk = (m / 2) * (m / 2 + 1) / 2;
            const bool blk_lds = FAST || (4 * nblk <= bf.nlds && nblk <= kMaxNB * (kNT - 64));
            const JacobiBuffers jb{FAST ? Ft : bf.lds, {Ft, bf.E}, (double2*)P, (double2*)ss.rot, ss.any, ss.red, blk_lds, sys};
            const int nsweep = eig_solve<EIG, FAST>(A, Cc, m, n, lb, jtol, Ft, P, bf.E, jb);
            QX_PH(sys, 3);
            QX_PH_ADD(sys, 12, nsweep);
            QX_PH_ADD(sys, 15, nsweep == 0);
            (void)nsweep;
            const int tid = qx_tid();
            for (int i = tid; i < n; i += kNT) eps[i] = A[i * lb + i];
            __syncthreads();
            if (tid < 64) {
                double mu = L.s_e[1];
                int fit = 0;
                const double t = fermi_wave(n, eps, si.kt, nalpha, L.focc, mu, fit);
                if (tid == 0) {
                    L.s_e[0] = t;
                    L.s_e[1] = mu;
                }
                QX_PH_ADD(sys, 14, fit);
                (void)fit;
                for (int i = tid; i < n; i += 64) f2[i] = 2.0 * L.focc[i];
            }
            __syncthreads();
            ts = L.s_e[0];
            QX_PH(sys, 4);
            mfma_gemm(n, n, n, Cc, lb, 1, Cc, 1, lb, P, lb, f2, true);
            __syncthreads();
            QX_PH(sys, 5);
            // row sums of P o M for M = S, D (3), Q (6), H0 as coalesced column
            // sweeps over all AOs (lanes): a wavefront takes every fourth matrix,
            // up to three that share the loads of P, over one half of the rows.
            // Every matrix is read once per iteration, which bounds large
            // systems; so P is read by four wavefronts and not by all eight.
            // (Cycles with a matrix or two per wavefront over all rows -> now: 58
            // AOs 52 k -> 30 k, 88: 105 k -> 62 k, 132: 184 k -> 114 k.)
            const bool split = n >= kRs;  // A holds n x kRs
            {
                static_assert(kNT / 64 == 8 && kRs <= 12, "three matrices by half the rows per wavefront");
                BatchRef B = qx_fresh(B0);
                const int tid = qx_tid(), lane = tid & 63, wave = qx_wave(tid), c0 = wave & 3;
                auto mat = [&](int c) {
                    return c == 0 ? B.S + si.mat_off
                           : c < 4 ? B.D + 3 * si.mat_off + (c - 1) * ms
                           : c < 10 ? B.Q + 6 * si.mat_off + (c - 4) * ms
                                    : B.H0 + si.mat_off;
                };
                const bool three = c0 + 8 < kRs;
                const double* M0 = mat(c0);
                const double* M1 = mat(c0 + 4);
                const double* M2 = mat(three ? c0 + 8 : c0);
                const int nh = split ? (n + 1) / 2 : n, nb = wave < 4 ? 0 : nh, ne = wave < 4 ? nh : n;
                double* o = wave < 4 ? rs : A;  // the second half's sums
                constexpr int NU = 7;           // rows per batch of loads
                for (int mu = lane; mu < n && nb < ne; mu += 64) {
                    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
                    for (int nu0 = nb; nu0 < ne; nu0 += NU) {
                        double x0[NU], x1[NU], x2[NU], p[NU];
#pragma unroll
                        for (int u = 0; u < NU; ++u) {
                            const int nu = nu0 + u < ne ? nu0 + u : nu0, q = nu * ld + mu;
                            x0[u] = M0[q];
                            x1[u] = M1[q];
                            if (three) x2[u] = M2[q];
                            p[u] = P[nu * lb + mu];
                        }
                        qx_sched_fence();
#pragma unroll
                        for (int u = 0; u < NU; ++u)
                            if (nu0 + u < ne) {
                                a0 += p[u] * x0[u];
                                a1 += p[u] * x1[u];
                                if (three) a2 += p[u] * x2[u];
                            }
                    }
                    o[mu * kRs + c0] = a0;
                    o[mu * kRs + c0 + 4] = a1;
                    if (three) o[mu * kRs + c0 + 8] = a2;
                }
            }
            __syncthreads();
            if (split) {
                for (int p = tid; p < n * kRs; p += kNT) rs[p] += A[p];
                __syncthreads();
            }
            for (int s = tid; s < nsh; s += kNT) {
                const ShellDesc d = ss.sh[s];
                double pop = 0.0;
                for (int a = 0; a < d.nao; ++a) pop += rs[(d.ao0 + a) * kRs];
                xout[s] = g_tab.e[d.el].refocc[d.k] - pop;
            }
            for (int t = tid; t < 9 * nat; t += kNT) {
                const int a = t / 9, c = t % 9;
                double v = 0.0;
                for (int mu = ss.aooff[a]; mu < ss.aooff[a + 1]; ++mu) v += rs[mu * kRs + 1 + c];
                if (c < 3) xout[nsh + 3 * a + c] = -v;
                else xout[nsh + 3 * nat + 6 * a + (c - 3)] = -v;
            }
            __syncthreads();
            QX_PH(sys, 6);
            continue;
        }
        QX_PH(sys, 7);
        double red2[2] = {0.0, 0.0};
        for (int mu = qx_tid(); mu < n; mu += kNT) red2[0] += rs[mu * kRs + 10];
        for (int i = qx_tid(); i < nx; i += kNT) {
            const double dd = xout[i] - xin[i];
            red2[1] += dd * dd;
        }
        block_sums<2>(red2, ss.red);
        eband = red2[0];
        etot = eband + ss.eparts[0] + ss.eparts[1] + ss.eparts[2] + ss.eparts[3] + ss.eparts[4] + ts;
        const double err = sqrt(red2[1] / nx);
        errp = err;
        const double de = etot - eold;
        eold = etot;
        if (qx_uniform(it > 1 && fabs(de) < opt.econv && err < opt.pconv)) {
            conv = 1;
            break;
        }
        if (it == opt.maxiter) break;
        QX_PH(sys, 8);
        broyden_step(si, qx_fresh(B0).hist + si.hist_off, opt, bf, xin, xout, ss.gm, ss.red, it, hcount);
        QX_PH(sys, 9);
        ++it;
    }
    QX_PH_ADD(sys, 13, it);
    BatchRef B = qx_fresh(B0);
    const int tid = qx_tid();
    if (opt.keep > 0 && tid == 0) {
        double* hcnt = B.hist + si.hist_off + 2 * (size_t)opt.mem * nx + 2 * (size_t)opt.mem * opt.mem +
                       2 * (size_t)opt.mem + 2 * (size_t)nx;
        hcnt[0] = (double)hcount;
    }
    // results: moments, charges, potentials at the output moments
    for (int i = tid; i < nx; i += kNT) {
        B.x[si.x_off + i] = xout[i];
        B.xo[si.x_off + i] = xout[i];
    }
    for (int a = tid; a < nat; a += kNT) B.qat[si.atom_off + a] = ss.qat[a];
    for (int s = tid; s < nsh; s += kNT) B.vs[si.shell_off + s] = vs[s];
    for (int i = tid; i < 3 * nat; i += kNT) B.vd[3 * (size_t)si.atom_off + i] = vd[i];
    for (int i = tid; i < 6 * nat; i += kNT) B.vq[6 * (size_t)si.atom_off + i] = vq[i];
    for (int i = tid; i < n; i += kNT) {
        B.eps[(size_t)sys * QX_MAX_NAO + i] = eps[i];
        B.focc[(size_t)sys * QX_MAX_NAO + i] = L.focc[i];
        f2[i] = 2.0 * L.focc[i] * eps[i];
    }
    if (FAST) {
        double* Pg = B.P + si.mat_off;
        for (int p = tid; p < n * n; p += kNT) Pg[(p / n) * ld + p % n] = P[(p / n) * lb + p % n];
    }
    __syncthreads();
    // W = C diag(2 f e) C^T ; U = L^T C for the next warm start
    mfma_gemm(n, n, n, Cc, lb, 1, Cc, 1, lb, B.W + si.mat_off, ld, f2, true);
    mfma_gemm(n, n, n, B.L + si.mat_off, 1, ld, Cc, lb, 1, B.U + si.mat_off, ld, nullptr, false);
    QX_PH(sys, 10);
    if (tid == 0) {
        double* ep = B.eparts + 10 * sys;
        ep[0] = eband;
        ep[1] = ss.eparts[0];
        ep[2] = ss.eparts[1];
        ep[3] = ss.eparts[2];
        ep[4] = ss.eparts[3];
        ep[5] = ss.eparts[4];
        ep[8] = ts;
        ep[9] = etot;
        B.energy[sys] = etot + ep[6] + ep[7];
        B.iters[sys] = it;
        B.iters_total[sys] += (unsigned long long)it;
        B.status[sys] = conv ? 0 : -1;
        B.warm[sys] = warm >= 5 ? 5 : warm + 1;
    }
}

// the whole SCC of system sys by the block (dyn: the launch's dynamic LDS)
//   EIG: with the MFMA eigen refinement
template <bool EIG>
QX_DEV void scc_system(BatchRef B, OptRef opt, int sys, SccLds& L, double* dyn)
{
    const SysInfo si = qx_info(B, sys);
    load_system(si, B, L.ss);
    const int m = (si.nao + 1) & ~1;
    if (m <= opt.lds_max_m) {
        // odd leading dimension: column-wise LDS accesses hit distinct banks
        const int mm = m * (m + 1);
        // a fifth matrix after the row sums when the launch's LDS holds it
        double* E = EIG && 5 * mm + kRs * m <= opt.lds_doubles ? dyn + 4 * mm + kRs * m : nullptr;
        // A and F are free at the potentials, P and the row sums are not
        double* pot = dyn + (pot_lds(si.nat) <= 2 * mm ? mm : 4 * mm + kRs * m);
        SccBuffers bf{dyn + mm, dyn, dyn + 2 * mm, dyn + 3 * mm, dyn + 4 * mm, m + 1, E, dyn + mm,
                      opt.lds_doubles - mm, pot};
        scc_body<true, EIG>(sys, si, B, opt, L.ss, bf, L);
    } else {
        // the energy-weighted density slot doubles as the row-sum scratch
        SccBuffers bf{B.T + si.mat_off, B.C + si.mat_off, B.U + si.mat_off, B.P + si.mat_off, B.W + si.mat_off,
                      si.ld, B.E + si.mat_off, dyn, opt.lds_doubles, dyn};
        scc_body<false, EIG>(sys, si, B, opt, L.ss, bf, L);
    }
}

struct SccArgs {
    BatchPtrs B;
    SccOpts opt;
};

template <bool EIG>
__global__ __launch_bounds__(kNT) void k_scc(SccArgs args)
{
    QX_ARG(SccArgs) a = qx_args(args);
    const int sys = qx_uniform(a.opt.first_sys < 0 ? a.B.order[blockIdx.x] : a.opt.first_sys + (int)blockIdx.x);
    if (a.B.active && !a.B.active[sys]) return;
    __shared__ SccLds L;
    extern __shared__ double dyn[];
    scc_system<EIG>(a.B, a.opt, sys, L, dyn);
}

}  // namespace qx
