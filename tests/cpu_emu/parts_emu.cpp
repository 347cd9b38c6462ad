// Driver of the CPU-emulated build that runs single parts of the library: the
// setup of one system, the launch sizes of a trajectory ensemble, the
// eigensolver and the solution for the Broyden weights.
//   parts_emu setup in out
//     in : int32 nat, num[nat]; double xyz[3 nat]
//     out: int32 n, ld; then twice (triangles of the factorisation in LDS, in
//          global memory) double S, L, X [ld * ld] each
//   parts_emu launch in out
//     in : int32 ntraj, offsets[ntraj + 1], num[natoms]
//     out: int64 shmem, lds_doubles of the persistent launch, of the SCC
//          launch of a step, free: LDS bytes that a workgroup may take beside
//          the static ones with the reserve kept
//   parts_emu eig in out
//     in : int32 m, nrow, form (0 blocks in global memory, 1 in LDS, 2 matrices
//          of up to 56 columns in LDS), refine, maxsweep (0: eig_solve, else
//          jacobi_any); double tol, min_s, A [m * m], C [nrow * m]
//     out: int32 full sweeps; double A, C
//   parts_emu broyden in out
//     in : int32 n, st (0: in LDS); double B [n * n], g [n]
//     out: double x [n]
//   phase_emu phase in out
//     in : int32 nsys, max_nao of the first of two launches; offsets[nsys + 1],
//          num[natoms]; double xyz[3 natoms]
//     out: per system int32 SCC iterations, the phase counters' iterations
#include "_build/src/capi.hip"

#include <cstdlib>

template <class T>
static void rd(FILE* f, T* v, size_t n)
{
    if (std::fread(v, sizeof(T), n, f) != n) std::exit(2);
}

template <class T>
static std::vector<T> rdv(FILE* f, size_t n)
{
    std::vector<T> v(n);
    rd(f, v.data(), n);
    return v;
}

template <class T>
static void wr(FILE* f, const T* v, size_t n)
{
    if (std::fwrite(v, sizeof(T), n, f) != n) std::exit(2);
}

static void run_setup(FILE* in, FILE* out)
{
    int32_t nat;
    rd(in, &nat, 1);
    const auto num = rdv<int32_t>(in, nat);
    const auto xyz = rdv<double>(in, 3 * (size_t)nat);
    const int32_t off[2] = {0, nat}, charge = 0;
    qcxms_batch* b = qcxms_batch_create(1, off, num.data(), &charge, QCXMS_GFN2_XTB);
    if (!b) std::exit(3);
    std::memcpy(b->d.xyz, xyz.data(), sizeof(double) * 3 * nat);
    const SysInfo& si = b->info[0];
    const int32_t size[2] = {si.nao, si.ld};
    wr(out, size, 2);
    const size_t ms = (size_t)si.ld * si.ld;
    for (const int ndyn : {si.nao * (si.nao + 2), 0}) {
        for (size_t i = 0; i < ms; ++i) b->d.L[i] = b->d.X[i] = NAN;
        hipLaunchKernelGGL(qx::k_setup, dim3(1), dim3(QX_BLOCK), sizeof(double) * (size_t)ndyn, b->stream, b->d, 1,
                           ndyn);
        wr(out, b->d.S, ms);
        wr(out, b->d.L, ms);
        wr(out, b->d.X, ms);
    }
    qcxms_batch_destroy(b);
}

static int64_t g_fused[2], g_step[2];

static bool note_launch(const void* k, unsigned, unsigned, size_t shmem, const void* const* args)
{
    if (k == (const void*)&qx::k_md_fused<true>) {
        g_fused[0] = (int64_t)shmem;
        g_fused[1] = ((const qx::MdArgs*)args[0])->opt.lds_doubles;
    } else if (k == (const void*)&qx::k_scc<true>) {
        g_step[0] = (int64_t)shmem;
        g_step[1] = ((const qx::SccArgs*)args[0])->opt.lds_doubles;
    }
    return false;
}

static void run_launch(FILE* in, FILE* out)
{
    int32_t nt;
    rd(in, &nt, 1);
    const auto off = rdv<int32_t>(in, nt + 1);
    const size_t nat = off[nt];
    const auto num = rdv<int32_t>(in, nat);
    const std::vector<int32_t> charge(nt, 0), imass(nat, -1);
    const std::vector<double> one(nat, 1.0), x(3 * nat, 0.0), e(nt, 0.0);
    qx_emu::g_launch_hook = note_launch;
    for (int fused = 0; fused < 2; ++fused) {
        qcxms_md_params p{};
        p.tstep = 20.0;
        p.etempin = -1.0;
        p.nfragexit = 3;
        p.max_steps = 1;
        p.fused = fused;
        qcxms_md* md = qcxms_md_create(nt, off.data(), num.data(), charge.data(), one.data(), imass.data(), x.data(),
                                       x.data(), one.data(), e.data(), e.data(), &p);
        int32_t running;
        if (!md || qcxms_md_run(md, 1, &running) != QCXMS_OK) std::exit(3);
        qcxms_md_destroy(md);
    }
    hipFuncAttributes fa;
    hipFuncGetAttributes(&fa, nullptr);
    const int64_t lds = (int64_t)qx_emu::kMaxLds - (int64_t)fa.sharedSizeBytes - 8192;
    wr(out, g_fused, 2);
    wr(out, g_step, 2);
    wr(out, &lds, 1);
}

struct EigArgs {
    int m, nrow, lda, lds, maxsweep;
    double tol, min_s;
    double *A, *C, *Y, *Z, *T;  // m x m each (C: nrow x m), leading dimension lda
    int* done;
};

template <bool EIG, bool FAST>
static void k_eig(EigArgs a)
{
    __shared__ __align__(16) double rot[2 * QX_MAX_NAO];
    __shared__ int any[QX_MAX_NAO];
    __shared__ double red[8 * (qx::kNT / 64)];
    double* dyn = (double*)qx_emu::dyn_lds();
    const qx::JacobiBuffers jb{FAST ? a.Y : dyn, {a.Y, a.T}, (double2*)a.Z, (double2*)rot, any, red, a.lds != 0};
    const int n = a.maxsweep ? qx::jacobi_any<FAST>(a.A, a.C, a.m, a.nrow, a.lda, a.tol, a.maxsweep, a.min_s, jb)
                             : qx::eig_solve<EIG, FAST>(a.A, a.C, a.m, a.nrow, a.lda, a.tol, a.Y, a.Z, a.T, jb);
    if (threadIdx.x == 0) *a.done = n;
}

// the matrices' storage as the SCC has it: leading dimension m + 1 (LDS) or
// the next multiple of 16 (global memory), the blocks exactly in the LDS
static void run_eig(FILE* in, FILE* out)
{
    int32_t h[5];
    rd(in, h, 5);
    const int m = h[0], nrow = h[1], form = h[2], refine = h[3];
    double t[2];
    rd(in, t, 2);
    const int lda = form == 2 ? m + 1 : (m + 15) & ~15, rows = form == 2 ? m : lda;
    std::vector<double> mat[5];
    for (auto& v : mat) v.assign((size_t)rows * lda, NAN);
    for (int i = 0; i < m; ++i) rd(in, &mat[0][(size_t)i * lda], m);
    for (int i = 0; i < nrow; ++i) rd(in, &mat[1][(size_t)i * lda], m);
    int done = -1;
    const EigArgs a{m, nrow, lda, form != 0, h[4], t[0], t[1], mat[0].data(), mat[1].data(), mat[2].data(),
                    mat[3].data(), mat[4].data(), &done};
    const size_t blk = form == 1 ? sizeof(double) * (size_t)m * (m + 2) / 2 : 0;
    void (*k)(EigArgs) = form == 2 ? (refine ? k_eig<true, true> : k_eig<false, true>)
                                   : (refine ? k_eig<true, false> : k_eig<false, false>);
    hipLaunchKernelGGL(k, dim3(1), dim3(qx::kNT), blk, nullptr, a);
    const int32_t d = done;
    wr(out, &d, 1);
    for (int i = 0; i < m; ++i) wr(out, &mat[0][(size_t)i * lda], m);
    for (int i = 0; i < nrow; ++i) wr(out, &mat[1][(size_t)i * lda], m);
}

static void k_broyden(int n, int st, const double* B, const double* g, double* bt, double* x)
{
    __shared__ double gm[128];
    double* t = bt ? bt : (double*)qx_emu::dyn_lds();
    for (int p = threadIdx.x; p < (n + 1) * n; p += qx::kNT) t[p / n * st + p % n] = p / n == n ? g[p % n] : B[p];
    __syncthreads();
    qx::broyden_solve(t, st, gm, n);
    for (int i = threadIdx.x; i < n; i += qx::kNT) x[i] = gm[i];
}

static void run_broyden(FILE* in, FILE* out)
{
    int32_t h[2];
    rd(in, h, 2);
    const int n = h[0], st = h[1] ? h[1] : (n | 1);
    const auto B = rdv<double>(in, (size_t)n * n), g = rdv<double>(in, n);
    std::vector<double> bt((size_t)(n + 1) * st, NAN), x(n);
    hipLaunchKernelGGL(k_broyden, dim3(1), dim3(qx::kNT), h[1] ? 0 : sizeof(double) * bt.size(), nullptr, n, st,
                       B.data(), g.data(), h[1] ? bt.data() : nullptr, x.data());
    wr(out, x.data(), n);
}

#ifdef QX_PHASE_TIMING
static void run_phase(FILE* in, FILE* out)
{
    int32_t h[2];
    rd(in, h, 2);
    const int nsys = h[0];
    const auto off = rdv<int32_t>(in, nsys + 1), num = rdv<int32_t>(in, off[nsys]);
    const auto xyz = rdv<double>(in, 3 * (size_t)off[nsys]);
    const std::vector<int32_t> charge(nsys, 0);
    const std::vector<double> et(nsys, 300.0);
    const int32_t bins[2] = {h[1], 256}, eig[2] = {0, 0}, lds[2] = {1, 1};
    std::vector<double> e(nsys), g(3 * (size_t)off[nsys]), q(off[nsys]);
    std::vector<int32_t> st(nsys);
    if (qcxms_set_tuning(h[1] < 256 ? 2 : 1, bins, eig, lds, -1, 0) != QCXMS_OK) std::exit(3);
    qcxms_batch* b = qcxms_batch_create(nsys, off.data(), num.data(), charge.data(), QCXMS_GFN2_XTB);
    if (!b || qcxms_batch_egrad(b, xyz.data(), et.data(), e.data(), g.data(), q.data(), st.data()) != QCXMS_OK)
        std::exit(3);
    std::vector<unsigned long long> row((size_t)nsys * qx::kPhaseSlots);
    std::memcpy(row.data(), qx::g_phase, sizeof(row[0]) * row.size());
    for (int s = 0; s < nsys; ++s) {
        const int32_t n[2] = {b->d.iters[s], (int32_t)row[(size_t)s * qx::kPhaseSlots + 13]};
        wr(out, n, 2);
    }
    qcxms_batch_destroy(b);
}
#endif

int main(int argc, char** argv)
{
    if (argc != 4) {
        std::fprintf(stderr, "usage: %s setup|launch|eig|broyden|phase input output\n", argv[0]);
        return 2;
    }
    FILE* in = std::fopen(argv[2], "rb");
    FILE* out = std::fopen(argv[3], "wb");
    if (!in || !out) return 2;
    const std::string part = argv[1];
    if (part == "setup") run_setup(in, out);
    else if (part == "launch") run_launch(in, out);
    else if (part == "eig") run_eig(in, out);
    else if (part == "broyden") run_broyden(in, out);
#ifdef QX_PHASE_TIMING
    else if (part == "phase") run_phase(in, out);
#endif
    else return 2;
    std::fclose(in);
    return std::fclose(out) ? 2 : 0;
}
