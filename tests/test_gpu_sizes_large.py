"""The largest systems, up to the library's limits (64 atoms, 256 basis
functions, so 128 shells, 448 D4 references and 704 mixed moments), and the
launch plan with Jacobi alone and the matrices of all sizes in global memory,
against the CPU oracle at the tolerances of test_gpu_sizes.py."""
import numpy as np
import pytest

import oracle_bind as ob
from test_gpu_sizes import SIZES, reference  # noqa: F401

pytestmark = pytest.mark.gpu


def ring(n):
    """Noisy cumulene ring of n carbon atoms (4 n basis functions)."""
    t = 2.0 * np.pi * np.arange(n) / n
    r = 1.30 / 0.529177 / (2.0 * np.sin(np.pi / n))
    xyz = np.stack([r * np.cos(t), r * np.sin(t), 0.0 * t], axis=1)
    return np.full(n, 6, np.int32), xyz + 0.02 * np.random.default_rng(n).standard_normal((n, 3))


def compare(mols, ref, eig, lds):
    import qcxms_amd
    re, rg, rq = ref[:3]
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
    for i, (num, _) in enumerate(mols):
        k = slice(off, off + len(num))
        off = k.stop
        de, dg, dq = abs(e[i] - re[i]), np.abs(g[k] - rg[i]).max(), np.abs(q[k] - rq[i]).max()
        print(f"nat={len(num)} dE={de:.2e} dg={dg:.2e} dq={dq:.2e}", flush=True)
        assert de <= 1e-8 and dg <= 1e-6 and dq <= 1e-6, i


def test_jacobi_alone_in_global_memory(reference):  # noqa: F811
    mols, ref = reference
    assert len(mols) == len(SIZES)
    compare(mols, ref, 0, 0)


@pytest.fixture(scope="module")
def rings():
    mols = [ring(n) for n in (48, 64, 36)]
    r = ob.gfn2_egrad_batch([(num, 1) for num, _ in mols], [xyz for _, xyz in mols], 5000.0,
                            opts=ob.default_opts(econv=1e-12, pconv=1e-10))
    assert np.all(r[3] == 0)
    return mols, r


@pytest.mark.parametrize("eig", [1, 0])
def test_largest_systems_match_the_oracle(rings, eig):
    compare(rings[0], rings[1], eig, 1)
