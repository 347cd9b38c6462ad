"""Basis sizes at which the SCC and setup kernels change their path, in one
batch that is not sorted by size, against the CPU oracle: the smallest (2), an
odd one, the limits of the matrices in LDS (56 | 58), of eigenvector rows in
registers (64 | 66), of the splits of the rotation replay (96 | 98, 102 | 104)
and of the Jacobi blocks in LDS (132 | 136).  The launch plans cover them
with the eigenvector refinement, with the matrices of all sizes in global
memory, and with Jacobi alone.  Tolerances: |dE| <= 1e-8 Eh, max |dg| <= 1e-6 Eh/bohr, max |dq| <=
1e-6 e, both sides converged well below them.
"""
import numpy as np
import pytest

import oracle_bind as ob
from qcxms_amd import workloads as W

pytestmark = pytest.mark.gpu

SIZES = (58, 136, 2, 96, 57, 104, 56, 132, 66, 98, 64, 102)


def system(nao):
    """Open-chain C/O/N cation (2 + 6 per heavy atom, 2 less per O, 1 less per
    N) of at most 64 atoms, or H2+."""
    if nao == 2:
        return np.array([1, 1], np.int32), np.array([[0.0, 0, 0], [0, 0, 1.9]])
    n = -(-(nao - 2) // 6)
    while 3 * n + 2 - (6 * n + 2 - nao) > 64:
        n += 1
    less = 6 * n + 2 - nao
    backbone = [6] * n
    for k in range(less // 2):
        backbone[1 + 3 * k] = 8
    if less % 2:
        backbone[n - 2] = 7
    return W.build_chain(backbone, noise=0.02, seed=nao)


@pytest.fixture(scope="module")
def reference():
    mols = [system(n) for n in SIZES]
    for n, (num, _) in zip(SIZES, mols):
        assert sum(1 if z == 1 else 4 for z in num) == n and len(num) <= 64
    r = ob.gfn2_egrad_batch([(num, 1) for num, _ in mols], [xyz for _, xyz in mols], 5000.0,
                            opts=ob.default_opts(econv=1e-12, pconv=1e-10))
    assert np.all(r[3] == 0)
    return mols, r


@pytest.mark.parametrize("eig,lds", [(1, 1), (1, 0), (0, 1)])
def test_sizes_at_the_limits_match_the_oracle(reference, eig, lds):
    import qcxms_amd
    mols, (re, rg, rq, _) = reference
    saved = qcxms_amd.get_tuning()
    try:
        qcxms_amd.set_tuning([(256, eig, lds)], (eig, lds))
        b = qcxms_amd.Batch([(num, 1) for num, _ in mols])
        b.set_scc(econv=1e-11, pconv=1e-9)
        e, g, q, st = b.egrad(np.concatenate([xyz for _, xyz in mols]), 5000.0)
        b.close()
    finally:
        qcxms_amd.set_tuning(*saved)
    assert np.all(st == 0)
    off = 0
    for i, n in enumerate(SIZES):
        k = slice(off, off + len(mols[i][0]))
        off = k.stop
        de, dg, dq = abs(e[i] - re[i]), np.abs(g[k] - rg[i]).max(), np.abs(q[k] - rq[i]).max()
        print(f"nao={n} dE={de:.2e} dg={dg:.2e} dq={dq:.2e}", flush=True)
        assert de <= 1e-8 and dg <= 1e-6 and dq <= 1e-6, n
