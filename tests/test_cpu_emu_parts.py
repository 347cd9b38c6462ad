"""Single parts of the kernels and the launch sizes in the CPU emulation
(tests/cpu_emu/parts_emu.cpp: bounds-checked, LDS filled with NaN bytes), at
the sizes where they change their path."""
import numpy as np
import pytest

import emu_bind as eb
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
