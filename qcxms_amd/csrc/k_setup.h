// Geometry-dependent setup of one GFN2-xTB evaluation (one workgroup per
// system): coordination numbers, D4 reference weights, repulsion and ATM
// energies, S/H0/dipole/quadrupole integrals, the ES2 gamma matrix, the D4
// charge-response matrix and the Cholesky orthogonaliser X = L^-T of S.
#pragma once
#include "integrals.h"

namespace qx {

// x^(alp / 3) of the ATM damping, and the exponents of the repulsion are
// r^1 (H-H) and r^(3/2): roots instead of the general power
QX_DEV double d4_pow(double x)
{
    static_assert(gfn2::kD4Alp == 16.0 && gfn2::kRepKexp == 1.5 && gfn2::kRepKexpLight == 1.0,
                  "powers written as roots");
    const double x2 = x * x;
    return x2 * x2 * x * cbrt(x);
}

QX_DEV double d4_zeta(double a, double c, double qref, double qmod)
{
    if (qmod < 0.0) return exp(a);
    return exp(a * (1.0 - exp(c * (1.0 - qref / qmod))));
}
// both at once
QX_DEV void d4_zeta_both(double a, double c, double qref, double qmod, double& z, double& dz)
{
    if (qmod < 0.0) {
        z = exp(a);
        dz = 0.0;
        return;
    }
    const double e = exp(c * (1.0 - qref / qmod));
    z = exp(a * (1.0 - e));
    dz = -a * c * e * z * qref / (qmod * qmod);
}

// GFN2 coordination-number count and its derivative d(count)/dr
QX_DEV void gfn_count(double rc, double r, double& f, double& df)
{
    const double e1 = exp(-gfn2::kCnKa * (rc / r - 1.0));
    const double e2 = exp(-gfn2::kCnKb * ((rc + gfn2::kCnShift) / r - 1.0));
    const double f1 = 1.0 / (1.0 + e1), f2 = 1.0 / (1.0 + e2);
    const double r2 = r * r;
    const double d1 = -gfn2::kCnKa * rc * e1 * f1 * f1 / r2;
    const double d2 = -gfn2::kCnKb * (rc + gfn2::kCnShift) * e2 * f2 * f2 / r2;
    f = f1 * f2;
    df = d1 * f2 + f1 * d2;
}

// D4 covalent count (dftd4.f90:292-325) and derivative
QX_DEV void d4_count(const ElemParams& ei, const ElemParams& ej, double r, double& f, double& df)
{
    const double rco = ei.rcov_d4 + ej.rcov_d4;
    const double den0 = fabs(ei.en_d4 - ej.en_d4) + gfn2::kD4K5;
    const double den = gfn2::kD4K4 * exp(-den0 * den0 / gfn2::kD4K6);
    const double ex = exp(-gfn2::kD4K1 * (rco / r - 1.0));
    f = den / (1.0 + ex);
    df = (-gfn2::kD4K1 * rco * ex * den) / (r * r * (1.0 + ex) * (1.0 + ex));
}

QX_DEV void mp_radius(const ElemParams& e, double cn, double& r, double& drdcn)
{
    const double arg = cn - e.mpvcn - gfn2::kAesShift;
    const double t = exp(-gfn2::kAesKexp * arg);
    r = e.mprad + (gfn2::kAesRmax - e.mprad) / (1.0 + t);
    drdcn = (gfn2::kAesRmax - e.mprad) * gfn2::kAesKexp * t / ((1.0 + t) * (1.0 + t));
}

// K * X(EN) * Y(zeta) and Pi(R) with dPi/dR for an off-site shell pair
QX_DEV double h0_scale(const ElemParams& ea, int ka, const ElemParams& eb, int kb, double r,
                       double& pir, double& dpir, double& kxy)
{
    const double za = ea.slater[ka], zb = eb.slater[kb];
    const double yz = sqrt(2.0 * sqrt(za * zb) / (za + zb));  // wexp = 1/2
    const double den = ea.en - eb.en;
    const double xen = 1.0 + gfn2::kEnScale * den * den;
    const double rab = ea.rad + eb.rad;
    const double sq = sqrt(r / rab);
    const double fa = 1.0 + ea.shpoly[ka] * sq, fb = 1.0 + eb.shpoly[kb] * sq;
    pir = fa * fb;
    dpir = (r > 0.0) ? (ea.shpoly[ka] * fb + eb.shpoly[kb] * fa) * 0.5 / sqrt(r * rab) : 0.0;
    kxy = 0.5 * (gfn2::kShellK[ka] + gfn2::kShellK[kb]) * xen * yz;
    return kxy * pir;
}

QX_DEV double d4_disp(const ElemParams& ei, const ElemParams& ej, double r2, double* ddisp_dr)
{
    const double r4r2ij = 3.0 * ei.r4r2 * ej.r4r2;
    const double r0 = gfn2::kD4A1 * sqrt(r4r2ij) + gfn2::kD4A2;
    const double r02 = r0 * r0, r06 = r02 * r02 * r02;
    const double oor6 = 1.0 / (r2 * r2 * r2 + r06);
    const double oor8 = 1.0 / (r2 * r2 * r2 * r2 + r06 * r02);
    if (ddisp_dr) {
        const double r = sqrt(r2);
        const double door6 = -6.0 * r2 * r2 * r * oor6 * oor6;
        const double door8 = -8.0 * r2 * r2 * r2 * r * oor8 * oor8;
        *ddisp_dr = gfn2::kD4S6 * door6 + gfn2::kD4S8 * r4r2ij * door8;
    }
    return gfn2::kD4S6 * oor6 + gfn2::kD4S8 * r4r2ij * oor8;
}

struct IntegralOut {
    double *S, *H, *D, *Q;
    int ld;
    size_t ms;
};

// S, H0 (off-atom), D and Q blocks of one bra AO (component A) of a shell
// pair.  S and H0 are symmetric; the moment integrals are stored transposed:
// element (mu, nu), taken about the atom of mu, sits at nu * ld + mu.  A row
// writes element (A, b) at both places; for a shell paired with itself
// (same), row b writes element (b, A) itself, so row A writes only the
// transposed places and every address has one writer.
template <int LA, int LB, int A>
QX_DEV void setup_shell_row(const ShellDesc& sa, const ShellDesc& sb, const ElemParams& ea,
                            const ElemParams& eb, const double* ra, const double* rb,
                            const double t[3], double hs, bool off, bool same, const IntegralOut& io)
{
    double s[3], dpb[3][3], qpb[3][6];
    shell_row_values<LA, LB, A>(ea, sa.k, eb, sb.k, ra, rb, s, dpb, qpb);
    constexpr int NB = LB ? 3 : 1;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        double dpa[3], qpa[6], qta[6], qtb[6];
        shift_to_a(t, s[b], dpb[b], qpb[b], dpa, qpa);
        traceless6(qpa, qta);
        traceless6(qpb[b], qtb);
        const int mu = sa.ao0 + A, nu = sb.ao0 + b;
        const size_t o1 = (size_t)mu * io.ld + nu, o2 = (size_t)nu * io.ld + mu;
        io.S[o2] = s[b];
        if (off) io.H[o2] = hs * s[b];
#pragma unroll
        for (int c = 0; c < 3; ++c) io.D[c * io.ms + o2] = dpa[c];
#pragma unroll
        for (int k = 0; k < 6; ++k) io.Q[k * io.ms + o2] = qta[k];
        if (!same) {
            io.S[o1] = s[b];
            if (off) io.H[o1] = hs * s[b];
#pragma unroll
            for (int c = 0; c < 3; ++c) io.D[c * io.ms + o1] = dpb[b][c];
#pragma unroll
            for (int k = 0; k < 6; ++k) io.Q[k * io.ms + o1] = qtb[k];
        }
    }
}

// Cholesky factor L of S and X = L^-T in LDS: S = U D^-1 U^T column by column
// (column j of U is the column of S as the elimination reaches it), the
// identity eliminated along with it, so that after the last column it is the
// inverse of the unit factor.  Row i of a step has the same i + 1 entries in
// every step (0 .. j of the inverse, j + 1 .. i of S), half a wavefront takes
// a row, and there is one barrier per column.  Both triangles are packed by
// rows; a: n (n + 2) doubles.
// (26-atom C8H18+, 50 basis functions: 82 us as a right-looking Cholesky of two
// barriers per column followed by one thread per column of the inverse.  The
// whole setup of a C8H18+ step takes 372 k cycles instead of 490 k with it.)
QX_DEV void factor_lds(const double* S, double* Lg, double* Xg, int n, int ld, double* a)
{
    constexpr int NR = QX_BLOCK / 32;
    const int tid = qx_tid(), q0 = tid & 31, r0 = tid >> 5;
    double* e = a + n * (n + 1) / 2;
    double* rd = e + n * (n + 1) / 2;  // 1 / L_jj
    __syncthreads();
    for (int i = r0; i < n; i += NR)
        for (int q = q0; q <= i; q += 32) {
            a[i * (i + 1) / 2 + q] = S[i * ld + q];
            e[i * (i + 1) / 2 + q] = q == i ? 1.0 : 0.0;
        }
    __syncthreads();
    for (int j = 0; j < n - 1; ++j) {
        const double inv = 1.0 / a[j * (j + 1) / 2 + j];
        const double* ej = e + j * (j + 1) / 2;
        for (int i = j + 1 + r0; i < n; i += NR) {
            double* ai = a + i * (i + 1) / 2;
            double* ei = e + i * (i + 1) / 2;
            const double l = ai[j] * inv;
            for (int q = q0; q <= i; q += 32) {
                if (q <= j) ei[q] -= l * ej[q];
                else ai[q] -= l * a[q * (q + 1) / 2 + j];
            }
        }
        __syncthreads();
    }
    for (int j = tid; j < n; j += QX_BLOCK) rd[j] = 1.0 / sqrt(a[j * (j + 1) / 2 + j]);
    __syncthreads();
    for (int i = r0; i < ld; i += NR)
        for (int q = q0; q < ld; q += 32) {
            Lg[i * ld + q] = (i < n && q <= i) ? a[i * (i + 1) / 2 + q] * rd[q] : 0.0;
            // row q of X is column q of L^-1
            Xg[i * ld + q] = (q < n && i <= q) ? e[q * (q + 1) / 2 + i] * rd[q] : 0.0;
        }
}

// The same in global memory, for systems whose triangles do not fit in LDS:
// every element goes through the same operations in the same order, so L and X
// do not depend on where the triangles are.  They are kept by columns here
// (element (i, q) at q * ld + i), a lane per row and the columns dealt to the
// wavefronts, so that all accesses are contiguous or uniform; the loads of NC
// columns are under way together, since a step is bound by their latency.
// a, e: ld x ld scratch each; rd: n doubles of LDS.
// (The whole setup of a 36-atom ring of 144 basis functions: 1.66 ms with a
// right-looking Cholesky and one thread per column of the inverse, 1.35 ms now.)
QX_DEV void factor_global(const double* S, double* Lg, double* Xg, int n, int ld, double* a, double* e, double* rd)
{
    constexpr int NW = QX_BLOCK / 64, NC = 4;
    const int tid = qx_tid(), lane = tid & 63, wave = qx_wave(tid);
    __syncthreads();
    for (int q = wave; q < n; q += NW)
        for (int i = q + lane; i < n; i += 64) {
            a[q * ld + i] = S[i * ld + q];
            e[q * ld + i] = q == i ? 1.0 : 0.0;
        }
    __syncthreads();
    for (int j = 0; j < n - 1; ++j) {
        const double inv = 1.0 / a[j * ld + j];
        for (int i0 = j + 1; i0 < n; i0 += 64) {
            const int i = i0 + lane, ir = i < n ? i : j;  // (row j is not written)
            const double l = a[j * ld + ir] * inv;
            // columns 0 .. j of the inverse, j + 1 .. of S down to the diagonal
            const int qe = i0 + 64 < n ? i0 + 64 : n;
            for (int q = wave; q < qe; q += NC * NW) {
                double v[NC], x[NC];
#pragma unroll
                for (int u = 0; u < NC; ++u) {
                    const int c = q + u * NW < qe ? q + u * NW : q;
                    v[u] = (c <= j ? e : a)[c * ld + ir];
                    x[u] = c <= j ? e[c * ld + j] : a[j * ld + c];
                }
                qx_sched_fence();
#pragma unroll
                for (int u = 0; u < NC; ++u) {
                    const int c = q + u * NW;
                    if (c < qe && i < n && (c <= j || c <= i)) (c <= j ? e : a)[c * ld + i] = v[u] - l * x[u];
                }
            }
        }
        __syncthreads();
    }
    for (int j = tid; j < n; j += QX_BLOCK) rd[j] = 1.0 / sqrt(a[j * ld + j]);
    __syncthreads();
    for (int i = wave; i < ld; i += NW)
        for (int q = lane; q < ld; q += 64) {
            Lg[i * ld + q] = (i < n && q <= i) ? a[q * ld + i] * rd[q] : 0.0;
            Xg[i * ld + q] = (q < n && i <= q) ? e[i * ld + q] * rd[q] : 0.0;
        }
}

// ---------------------------------------------------------------------------
// LDS of one system's setup (the Cholesky factor uses the dynamic LDS)
struct SetupLds {
    ShellDesc sh[QX_MAX_NSH];
    int ao_at[QX_MAX_NAO], ao_sh[QX_MAX_NAO];
    double sx[3 * QX_MAX_NAT];
    int sel[QX_MAX_NAT];
    double scn[QX_MAX_NAT], scnd4[QX_MAX_NAT];
    int refoff[QX_MAX_NAT + 1];
    double red[QX_BLOCK / 64];
    // per D4 reference: zeta(q = 0) * gw
    double zg[QX_MAX_REF * QX_MAX_NAT];
};

// dyn: ndyn doubles of LDS for the factorisation
QX_DEV void setup_system(BatchRef B, int sys, int with_chol, SetupLds& Ls, double* dyn, int ndyn)
{
    const SysInfo si = qx_info(B, sys);
    const int tid = qx_tid();
    const int nat = si.nat, nsh = si.nsh, n = si.nao, ld = si.ld;
    ShellDesc* sh = Ls.sh;
    int* ao_at = Ls.ao_at;
    int* ao_sh = Ls.ao_sh;
    double* sx = Ls.sx;
    int* sel = Ls.sel;
    double* scn = Ls.scn;
    double* scnd4 = Ls.scnd4;
    int* refoff = Ls.refoff;
    double* red = Ls.red;

    const double* gx = B.xyz + 3 * (size_t)si.atom_off;
    for (int i = tid; i < 3 * nat; i += QX_BLOCK) sx[i] = gx[i];
    for (int i = tid; i < nat; i += QX_BLOCK) sel[i] = B.elem[si.atom_off + i];
    build_shell_tables(si, B.elem, sh, ao_at, ao_sh);
    if (tid == 0) {
        int o = 0;
        for (int a = 0; a < nat; ++a) {
            refoff[a] = o;
            o += g_tab.e[sel[a]].nref;
        }
        refoff[nat] = o;
    }
    // 1. coordination numbers: a wavefront per atom, a lane per partner,
    //    tree sums over the lanes
    __syncthreads();
    for (int a = tid >> 6; a < nat; a += QX_BLOCK / 64) {
        const int lane = tid & 63;
        const ElemParams& ea = g_tab.e[sel[a]];
        double cn = 0.0, cn4 = 0.0;
        for (int b = lane; b < nat; b += 64) {
            if (b == a) continue;
            const ElemParams& eb = g_tab.e[sel[b]];
            const double dx = sx[3 * a] - sx[3 * b], dy = sx[3 * a + 1] - sx[3 * b + 1],
                         dz = sx[3 * a + 2] - sx[3 * b + 2];
            const double r2 = dx * dx + dy * dy + dz * dz;
            const double r = sqrt(r2);
            double f, df;
            if (r2 <= gfn2::kCnCutoff * gfn2::kCnCutoff) {
                gfn_count(ea.covrad + eb.covrad, r, f, df);
                cn += f;
            }
            if (r2 <= gfn2::kD4CnThr) {
                d4_count(ea, eb, r, f, df);
                cn4 += f;
            }
        }
        cn = wave_sum(cn);
        cn4 = wave_sum(cn4);
        if (lane != 0) continue;
        scn[a] = cn;
        scnd4[a] = cn4;
        B.cn[si.atom_off + a] = cn;
        B.cnd4[si.atom_off + a] = cn4;
        double mr, dmr;
        mp_radius(ea, cn, mr, dmr);
        B.mrad[si.atom_off + a] = mr;
        B.dmrad[si.atom_off + a] = dmr;
    }
    __syncthreads();
    // 2. self-energies and D4 weights
    for (int s = tid; s < nsh; s += QX_BLOCK) {
        const ElemParams& e = g_tab.e[sh[s].el];
        B.hself[si.shell_off + s] = e.hself0[sh[s].k] - e.kcn[sh[s].k] * scn[sh[s].at];
    }
    for (int a = tid; a < nat; a += QX_BLOCK) {
        const ElemParams& e = g_tab.e[sel[a]];
        const double cn = scnd4[a];
        double norm = 0.0, dnorm = 0.0;
        for (int r = 0; r < e.nref; ++r)
            for (int k = 1; k <= e.refc[r]; ++k) {
                const double twf = k * gfn2::kD4Wf, d = cn - e.refcovcn[r];
                const double t = exp(-twf * d * d);
                norm += t;
                dnorm += 2.0 * twf * (e.refcovcn[r] - cn) * t;
            }
        norm = 1.0 / norm;
        double mx = -1e300;
        for (int r = 0; r < e.nref; ++r) mx = fmax(mx, e.refcovcn[r]);
        for (int r = 0; r < e.nref; ++r) {
            double ex = 0.0, dex = 0.0;
            for (int k = 1; k <= e.refc[r]; ++k) {
                const double twf = k * gfn2::kD4Wf, d = cn - e.refcovcn[r];
                const double t = exp(-twf * d * d);
                ex += t;
                dex += 2.0 * twf * (e.refcovcn[r] - cn) * t;
            }
            double g = ex * norm;
            if (g != g) g = (mx == e.refcovcn[r]) ? 1.0 : 0.0;
            double dg = dex * norm - ex * dnorm * norm * norm;
            if (dg != dg) dg = 0.0;
            B.gw[si.ref_off + refoff[a] + r] = g;
            B.dgw[si.ref_off + refoff[a] + r] = dg;
        }
    }
    // 3. clear the matrix slots (padding stays zero)
    const size_t ms = (size_t)ld * ld;
    double* S = B.S + si.mat_off;
    double* H = B.H0 + si.mat_off;
    double* D = B.D + 3 * si.mat_off;
    double* Q = B.Q + 6 * si.mat_off;
    for (size_t i = tid; i < ms; i += QX_BLOCK) {
        S[i] = 0.0;
        H[i] = 0.0;
    }
    for (size_t i = tid; i < 3 * ms; i += QX_BLOCK) D[i] = 0.0;
    for (size_t i = tid; i < 6 * ms; i += QX_BLOCK) Q[i] = 0.0;
    __syncthreads();
    // 4. integrals, one work item per row of a shell pair (the rows of a p
    //    shell are three items; rows of three AO pairs come first)
    for (int it = tid; it < si.nrowitem; it += QX_BLOCK) {
        const int2 pr = B.spitem[si.rowitem_off + it];
        const int ia = pr.x & 0xffff, row = pr.x >> 16, ib = pr.y;
        const ShellDesc sa = sh[ia], sb = sh[ib];
        const ElemParams& ea = g_tab.e[sa.el];
        const ElemParams& eb = g_tab.e[sb.el];
        const double* ra = sx + 3 * sa.at;
        const double* rb = sx + 3 * sb.at;
        const double t[3] = {rb[0] - ra[0], rb[1] - ra[1], rb[2] - ra[2]};
        double hs = 0.0;
        const bool off = sa.at != sb.at;
        if (off) {
            const double r = sqrt(t[0] * t[0] + t[1] * t[1] + t[2] * t[2]);
            double pir, dpir, kxy;
            hs = 0.5 * (B.hself[si.shell_off + ia] + B.hself[si.shell_off + ib]) *
                 h0_scale(ea, sa.k, eb, sb.k, r, pir, dpir, kxy);
        }
        const IntegralOut io{S, H, D, Q, ld, ms};
        const bool same = ia == ib;
        switch ((sa.l * 2 + sb.l) * 3 + row) {
        case 9: setup_shell_row<1, 1, 0>(sa, sb, ea, eb, ra, rb, t, hs, off, same, io); break;
        case 10: setup_shell_row<1, 1, 1>(sa, sb, ea, eb, ra, rb, t, hs, off, same, io); break;
        case 11: setup_shell_row<1, 1, 2>(sa, sb, ea, eb, ra, rb, t, hs, off, same, io); break;
        case 6: setup_shell_row<1, 0, 0>(sa, sb, ea, eb, ra, rb, t, hs, off, same, io); break;
        case 7: setup_shell_row<1, 0, 1>(sa, sb, ea, eb, ra, rb, t, hs, off, same, io); break;
        case 8: setup_shell_row<1, 0, 2>(sa, sb, ea, eb, ra, rb, t, hs, off, same, io); break;
        case 3: setup_shell_row<0, 1, 0>(sa, sb, ea, eb, ra, rb, t, hs, off, same, io); break;
        default: setup_shell_row<0, 0, 0>(sa, sb, ea, eb, ra, rb, t, hs, off, same, io); break;
        }
    }
    __syncthreads();
    for (int s = tid; s < nsh; s += QX_BLOCK)
        for (int a = 0; a < sh[s].nao; ++a) {
            const int mu = sh[s].ao0 + a;
            H[(size_t)mu * ld + mu] = B.hself[si.shell_off + s];
        }
    // 5. ES2 gamma matrix
    double* G = B.gam + si.gam_off;
    for (int p = tid; p < nsh * nsh; p += QX_BLOCK) {
        const int a = p / nsh, b = p % nsh;
        const double* ra = sx + 3 * sh[a].at;
        const double* rb = sx + 3 * sh[b].at;
        const double dx = ra[0] - rb[0], dy = ra[1] - rb[1], dz = ra[2] - rb[2];
        const double eta = 0.5 * (g_tab.e[sh[a].el].hard[sh[a].k] + g_tab.e[sh[b].el].hard[sh[b].k]);
        G[p] = 1.0 / sqrt(dx * dx + dy * dy + dz * dz + 1.0 / (eta * eta));
    }
    // 6. per D4 reference zeta(q = 0) gw, and the kernels of an ordered atom
    //    pair (i, j) at planes c * nat^2 + j * nat + i: the damped multipole
    //    kernels 1/r^3 and 1/r^5 and the D4 pair damping, zero for i = j
    const double* gw = B.gw + si.ref_off;
    double* zg = Ls.zg;
    __syncthreads();
    for (int a = tid; a < nat; a += QX_BLOCK) {
        const ElemParams& e = g_tab.e[sel[a]];
        for (int r = 0; r < e.nref; ++r) {
            const int k = refoff[a] + r;
            zg[k] = d4_zeta(gfn2::kD4Ga, e.gam * gfn2::kD4Gc, e.refq[r] + e.zeff, e.zeff) * gw[k];
        }
    }
    double* pk = B.pairk + (size_t)si.pair_off / QX_PAIR_STRIDE * QX_PAIR_KERN;
    const int nn = nat * nat;
    for (int p = tid; p < nn; p += QX_BLOCK) {
        const int j = p / nat, i = p - j * nat;
        double h3 = 0.0, h5 = 0.0, disp = 0.0;
        if (i != j) {
            const double dx = sx[3 * i] - sx[3 * j], dy = sx[3 * i + 1] - sx[3 * j + 1],
                         dz = sx[3 * i + 2] - sx[3 * j + 2];
            const double r2 = dx * dx + dy * dy + dz * dz;
            const double r = sqrt(r2);
            const double r0 = 0.5 * (B.mrad[si.atom_off + i] + B.mrad[si.atom_off + j]);
            const double r03 = r0 * r0 * r0;
            h3 = 1.0 / (r2 * r + 6.0 * r03);
            h5 = 1.0 / (r * (r2 * r2 + 6.0 * r03 * r0));
            if (r2 <= gfn2::kD4RThr) disp = d4_disp(g_tab.e[sel[i]], g_tab.e[sel[j]], r2, nullptr);
        }
        pk[p] = h3;
        pk[nn + p] = h5;
        pk[2 * nn + p] = disp;
    }
    __syncthreads();
    // 7. repulsion energy
    double erep = 0.0;
    for (int p = tid; p < nat * nat; p += QX_BLOCK) {
        const int i = p / nat, j = p % nat;
        if (j >= i) continue;
        const ElemParams& ei = g_tab.e[sel[i]];
        const ElemParams& ej = g_tab.e[sel[j]];
        const double dx = sx[3 * i] - sx[3 * j], dy = sx[3 * i + 1] - sx[3 * j + 1],
                     dz = sx[3 * i + 2] - sx[3 * j + 2];
        const double r = sqrt(dx * dx + dy * dy + dz * dz);
        if (r > gfn2::kRepCutoff) continue;
        erep += ei.rep_zeff * ej.rep_zeff / r *
                exp(-sqrt(ei.rep_alpha * ej.rep_alpha) * (ei.z <= 2 && ej.z <= 2 ? r : r * sqrt(r)));
    }
    erep = block_sum(erep, red);
    // 8. ATM energy at zero charges: pair C6 into scratch, then triples
    double* c60 = B.pairbuf + si.pair_off;  // nat*nat
    for (int p = tid; p < nat * nat; p += QX_BLOCK) {
        const int i = p / nat, j = p % nat;
        const ElemParams& ei = g_tab.e[sel[i]];
        const ElemParams& ej = g_tab.e[sel[j]];
        double c = 0.0;
        for (int ii = 0; ii < ei.nref; ++ii) {
            const double zi = zg[refoff[i] + ii];
            for (int jj = 0; jj < ej.nref; ++jj) c += zi * zg[refoff[j] + jj] * g_tab.c6ref[sel[i]][ii][sel[j]][jj];
        }
        c60[p] = c;
    }
    __syncthreads();
    // triples i > j > k in contiguous equal chunks per thread (the pair-wise
    // loop left half the threads idle and the rest unevenly loaded)
    double eatm = 0.0;
    {
        const long long ntri = (long long)nat * (nat - 1) * (nat - 2) / 6;
        const long long chunk = (ntri + QX_BLOCK - 1) / QX_BLOCK;
        long long t = (long long)tid * chunk;
        const long long tend = t + chunk < ntri ? t + chunk : ntri;
        // unrank t: i with C(i,3) <= t < C(i+1,3), then j with C(j,2) <= rest
        int i = 2, j = 1, k = 0;
        if (t < tend) {
            while ((long long)(i + 1) * i * (i - 1) / 6 <= t) ++i;
            long long rest = t - (long long)i * (i - 1) * (i - 2) / 6;
            j = 1;
            while ((long long)(j + 1) * j / 2 <= rest) ++j;
            k = (int)(rest - (long long)j * (j - 1) / 2);
        }
        for (; t < tend; ++t) {
            const double dij[3] = {sx[3 * i] - sx[3 * j], sx[3 * i + 1] - sx[3 * j + 1], sx[3 * i + 2] - sx[3 * j + 2]};
            const double u = dij[0] * dij[0] + dij[1] * dij[1] + dij[2] * dij[2];
            const double dik[3] = {sx[3 * i] - sx[3 * k], sx[3 * i + 1] - sx[3 * k + 1], sx[3 * i + 2] - sx[3 * k + 2]};
            const double djk[3] = {sx[3 * j] - sx[3 * k], sx[3 * j + 1] - sx[3 * k + 1], sx[3 * j + 2] - sx[3 * k + 2]};
            const double w = dik[0] * dik[0] + dik[1] * dik[1] + dik[2] * dik[2];
            const double v = djk[0] * djk[0] + djk[1] * djk[1] + djk[2] * djk[2];
            if (u <= gfn2::kD4AtmThr && w <= gfn2::kD4AtmThr && v <= gfn2::kD4AtmThr) {
                const ElemParams& ei = g_tab.e[sel[i]];
                const ElemParams& ej = g_tab.e[sel[j]];
                const ElemParams& ek = g_tab.e[sel[k]];
                const double cij = gfn2::kD4A1 * sqrt(3.0 * ei.r4r2 * ej.r4r2) + gfn2::kD4A2;
                const double cik = gfn2::kD4A1 * sqrt(3.0 * ei.r4r2 * ek.r4r2) + gfn2::kD4A2;
                const double cjk = gfn2::kD4A1 * sqrt(3.0 * ej.r4r2 * ek.r4r2) + gfn2::kD4A2;
                const double uvw = u * v * w, rijk = sqrt(uvw), cijk = cij * cjk * cik;
                const double aa = u + v - w, bb = u + w - v, cc = w + v - u;
                const double atm = (0.375 * aa * bb * cc / uvw + 1.0) / (rijk * rijk * rijk);
                const double x = d4_pow(cijk / rijk);
                const double fd = 1.0 / (1.0 + 6.0 * x);
                const double c9 = gfn2::kD4S9 * sqrt(c60[i * nat + j] * c60[j * nat + k] * c60[i * nat + k]);
                eatm += c9 * atm * fd;
            }
            // next triple in (i, j, k) lexicographic order with k < j < i
            if (++k == j) {
                k = 0;
                if (++j == i) {
                    j = 1;
                    ++i;
                }
            }
        }
    }
    eatm = block_sum(eatm, red);
    if (tid == 0) {
        B.eparts[10 * sys + 6] = eatm;
        B.eparts[10 * sys + 7] = erep;
    }
    if (!with_chol) return;
    // 9. Cholesky S = L L^T and X = L^-T (the SCC's scratch is free)
    static_assert(QX_MAX_REF * QX_MAX_NAT >= QX_MAX_NAO, "the pivots take the place of zg");
    if (n * (n + 2) <= ndyn) factor_lds(S, B.L + si.mat_off, B.X + si.mat_off, n, ld, dyn);
    else factor_global(S, B.L + si.mat_off, B.X + si.mat_off, n, ld, B.T + si.mat_off, B.C + si.mat_off, zg);
}

__global__ __launch_bounds__(QX_BLOCK) void k_setup(BatchPtrs B, int with_chol, int ndyn)
{
    const int sys = B.order[blockIdx.x];
    if (B.active && !B.active[sys]) return;
    __shared__ SetupLds Ls;
    extern __shared__ double dyn[];
    setup_system(qx_args(B), sys, with_chol, Ls, dyn, ndyn);
}

}  // namespace qx
