// Driver of the CPU-emulated build that runs single parts of the library: the
// setup of one system, and the launch sizes of a trajectory ensemble.
//   parts_emu setup in out
//     in : int32 nat, num[nat]; double xyz[3 nat]
//     out: int32 n, ld; then twice (triangles of the factorisation in LDS, in
//          global memory) double S, L, X [ld * ld] each
//   parts_emu launch in out
//     in : int32 ntraj, offsets[ntraj + 1], num[natoms]
//     out: int64 shmem, lds_doubles of the persistent launch, of the SCC
//          launch of a step, free: LDS bytes that a workgroup may take beside
//          the static ones with the reserve kept
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

int main(int argc, char** argv)
{
    if (argc != 4) {
        std::fprintf(stderr, "usage: %s setup|launch input output\n", argv[0]);
        return 2;
    }
    FILE* in = std::fopen(argv[2], "rb");
    FILE* out = std::fopen(argv[3], "wb");
    if (!in || !out) return 2;
    const std::string part = argv[1];
    if (part == "setup") run_setup(in, out);
    else if (part == "launch") run_launch(in, out);
    else return 2;
    std::fclose(in);
    return std::fclose(out) ? 2 : 0;
}
