"""Single parts of the kernels and the launch sizes in the CPU emulation
(tests/cpu_emu/parts_emu.cpp: bounds-checked, LDS filled with NaN bytes), at
the sizes where they change their path, and whole systems above 64 basis
functions."""
import numpy as np
import pytest

import emu_bind as eb
import oracle_bind as ob
from qcxms_amd import workloads as W


def molecule(nao):
    """Saturated C/N/O chain of nao basis functions and at most 64 atoms
    (2 + 6 per heavy atom, 2 less per O, 1 less per N)."""
    n = -(-(nao - 2) // 6)
    while 3 * n + 2 - (6 * n + 2 - nao) > 64:
        n += 1
    less = 6 * n + 2 - nao
    backbone = [6] * n
    for k in range(less // 2):
        backbone[min(1 + 3 * k, n - 1)] = 8
    if less % 2:
        backbone[n - 2 if n > 1 else 0] = 7
    num, xyz = W.build_chain(backbone, noise=0.02, seed=nao)
    assert sum(1 if z == 1 else 4 for z in num) == nao and len(num) <= 64
    return num, xyz


@pytest.mark.timeout(900)
@pytest.mark.parametrize("nao", [6, 57, 64, 119, 134])
def test_factorisation_does_not_depend_on_where_the_triangles_are(nao):
    """L and X = L^-T of the overlap have the same bits with the triangles in
    LDS and in global memory, so a system's results do not depend on the LDS
    of its launch (the per-step and the persistent MD kernel, other systems in
    the batch).  L L^T = S to the Cholesky bound (n + 1) eps |L| |L^T| with unit
    diagonal of S, taken four times: 1e-13; L^T X = 1 to that times the
    condition of L (< 1e2): 1e-11."""
    num, xyz = molecule(nao)
    raw = eb.part("setup", np.array([len(num)], np.int32), np.asarray(num, np.int32), np.asarray(xyz, np.float64))
    n, ld = np.frombuffer(raw, np.int32, 2)
    assert n == nao
    m = np.frombuffer(raw, np.float64, offset=8).reshape(2, 3, ld, ld)
    for s, l, x in m:
        assert np.abs(l[:n, :n] @ l[:n, :n].T - s[:n, :n]).max() < 1e-13
        assert np.abs(l[:n, :n].T @ x[:n, :n] - np.eye(n)).max() < 1e-11
        for a in (l, x):
            assert np.all(a[n:] == 0.0) and np.all(a[:, n:] == 0.0)
    assert m[0].tobytes() == m[1].tobytes()


def launch(naos):
    mols = [molecule(n)[0] for n in naos]
    off = np.cumsum([0] + [len(m) for m in mols]).astype(np.int32)
    raw = eb.part("launch", np.array([len(mols)], np.int32), off, np.concatenate(mols).astype(np.int32))
    return np.frombuffer(raw, np.int64)


@pytest.mark.timeout(900)
def test_persistent_launch_keeps_its_lds_reserve():
    """Whatever the basis size, the persistent MD kernel's workgroup leaves
    8 KiB of the LDS free, as the SCC and setup kernels do."""
    for nao in (2 + 6 * 8, 56, 58, 111, 113, 115, 116, 117, 118, 119, 120, 121, 122, 132, 134):
        shmem, _, _, _, free = launch([nao])
        assert shmem <= free, nao


@pytest.mark.timeout(900)
@pytest.mark.parametrize("naos", [(50, 56), (52,), (52, 117), (52, 119), (54, 121), (58, 134)])
def test_scc_of_a_persistent_launch_has_the_lds_of_the_scc_kernel(naos):
    """The LDS that the SCC may use (which decides about the fifth matrix of
    the eigenvector refinement, so about the solver's path) is that of the
    SCC kernel of a step, whatever the setup of another trajectory takes."""
    shmem, doubles, step_shmem, step_doubles, _ = launch(naos)
    assert doubles == step_doubles and 8 * doubles == step_shmem <= shmem


def eig(a, form, refine=0, maxsweep=0, tol=1e-11, min_s=0.0):
    """The eigensolver on the n x n matrix a, padded to an even order by a
    zero row and column; C starts as the identity, so that it ends as V."""
    n = len(a)
    m = (n + 1) & ~1
    am, c = np.zeros((m, m)), np.zeros((n, m))
    am[:n, :n] = a
    c[:, :n] = np.eye(n)
    raw = eb.part("eig", np.array([m, n, form, refine, maxsweep], np.int32), np.array([tol, min_s]), am, c)
    out = np.frombuffer(raw, np.float64, offset=4)
    return int(np.frombuffer(raw, np.int32, 1)[0]), out[:m * m].reshape(m, m), out[m * m:].reshape(n, m)


def check_rotated(a, out, v, sweeps):
    """V orthogonal and A_out = V^T A V: every row takes m - 1 rotations a
    sweep, each within 4 eps of the norm (2 here), over at most 15 sweeps and
    256 columns 4e-12."""
    n = len(a)
    one = np.zeros(len(out))
    one[:n] = 1.0
    assert np.abs(v.T @ v - np.diag(one)).max() < 4e-12, sweeps
    assert np.abs(v.T @ a @ v - out).max() < 4e-12, sweeps


def dense(n):
    r = np.random.default_rng(n).standard_normal((n, n))
    return np.diag(np.linspace(-1.0, 1.0, n)) + 0.25 * (r + r.T) / np.sqrt(n)


def offdiag(a):
    return np.abs(a - np.diag(np.diag(a))).max()


@pytest.mark.timeout(900)
@pytest.mark.parametrize("n,form", [(2, 2), (3, 2), (21, 2), (21, 1), (66, 1), (66, 0)])
def test_jacobi_to_convergence(n, form):
    """Every form of the sweeps: rows of C in registers (up to 64 columns) or
    rotated by the logged sweep, blocks in LDS or in global memory."""
    a = dense(n)
    sweeps, out, v = eig(a, form)
    assert 0 < sweeps <= 15 and offdiag(out) < 1e-11
    check_rotated(a, out, v, sweeps)
    assert np.array_equal(out, out.T)


@pytest.mark.timeout(900)
@pytest.mark.parametrize("n,form,min_s", [(55, 2, 0.02), (56, 2, 0.0), (57, 1, 0.0), (64, 1, 0.02), (96, 1, 0.0),
                                          (97, 1, 0.02), (102, 1, 0.0), (104, 1, 0.02), (132, 1, 0.0),
                                          (134, 0, 0.02), (256, 0, 0.0)])
def test_two_jacobi_sweeps_at_the_limits_of_their_forms(n, form, min_s):
    """Two sweeps at the largest orders of the matrices in LDS, the rows in
    registers, the splits of the rotation replay and the blocks in LDS, and
    beyond; all rotations or (a coarse sweep) the large ones."""
    a = dense(n)
    sweeps, out, v = eig(a, form, maxsweep=2, min_s=min_s)
    assert sweeps == 2 and np.array_equal(out, out.T)
    # a sweep that rotates every pair does not increase the sum of squares
    assert np.sum(np.tril(out, -1) ** 2) < 0.5 * np.sum(np.tril(a, -1) ** 2)
    check_rotated(a, out, v, sweeps)


@pytest.mark.timeout(900)
@pytest.mark.parametrize("n,form,strong", [(50, 2, 3), (57, 1, 0), (66, 1, 3), (134, 0, 3)])
def test_eigenvector_refinement(n, form, strong):
    """The simultaneous rotations, from small couplings (no Jacobi sweep) and
    with near-degenerate, strongly coupled pairs (coarse sweeps first); the
    fifth matrix shares its storage with the blocks in global memory."""
    r = np.random.default_rng(n + strong).standard_normal((n, n))
    a = np.diag(np.linspace(-1.0, 1.0, n)) + 2e-5 * (r + r.T)
    for k in range(strong):
        i, j = 5 * k, 5 * k + 1
        a[i, j] = a[j, i] = 0.05
    sweeps, out, v = eig(a, form, refine=1)
    assert sweeps == 0 and offdiag(out) < 1e-11
    check_rotated(a, out, v, sweeps)


@pytest.mark.timeout(900)
@pytest.mark.parametrize("n,st", [(1, 0), (2, 0), (40, 0), (41, 100), (64, 0), (65, 100), (100, 100)])
def test_broyden_weights(n, st):
    """The solution for the weights of n secant pairs, the matrix in LDS or in
    global memory, against numpy: n eps times the condition (< 1e3) times 10."""
    rng = np.random.default_rng(n)
    g = rng.standard_normal((n, 3 * n))
    b = np.eye(n) + g @ g.T / (3 * n)
    assert np.linalg.cond(b) < 1e3
    rhs = rng.standard_normal(n)
    x = np.frombuffer(eb.part("broyden", np.array([n, st], np.int32), b, rhs), np.float64)
    ref = np.linalg.solve(b, rhs)
    assert np.abs(x - ref).max() < 1.2e-13 * n * np.abs(ref).max() * 10


@pytest.mark.timeout(900)
@pytest.mark.parametrize("first", [256, 4])
def test_phase_counters_belong_to_their_system(first):
    """Row s of the phase counters (builds with QX_PHASE_TIMING) is system s
    of the batch, in a launch that takes the systems by size and in one launch
    per run of systems of one bin."""
    mols = [(np.array([1, 1], np.int32), np.array([[0.0, 0.0, 0.0], [0.0, 0.0, 1.5]])), molecule(6)]
    off = np.cumsum([0] + [len(n) for n, _ in mols]).astype(np.int32)
    raw = eb.part("phase", np.array([len(mols), first], np.int32), off,
                  np.concatenate([n for n, _ in mols]).astype(np.int32), np.concatenate([x for _, x in mols]))
    iters, counted = np.frombuffer(raw, np.int32).reshape(-1, 2).T
    assert iters[0] != iters[1]
    assert np.array_equal(iters, counted)


@pytest.mark.timeout(900)
def test_emulated_large_systems_match_the_oracle():
    """Systems of 66, 104 and 134 basis functions in one launch with the
    eigenvector refinement, at the bars of the GPU parity tests."""
    eb.build()
    mols = [molecule(n) for n in (66, 104, 134)]
    systems, coords = [(num, 1) for num, _ in mols], [xyz for _, xyz in mols]
    rc, e, g, q, st, err = eb.egrad_batch(systems, coords, 5000.0, tuning=[(256, 1, 1)])
    assert rc == 0 and np.all(st == 0), err
    re, rg, rq, rst = ob.gfn2_egrad_batch(systems, coords, 5000.0, opts=ob.default_opts(econv=1e-12, pconv=1e-10))
    assert np.all(rst == 0)
    assert np.abs(e - re).max() <= 1e-8
    assert max(np.abs(a - b).max() for a, b in zip(g, rg)) <= 1e-6
    assert max(np.abs(a - b).max() for a, b in zip(q, rq)) <= 1e-6
