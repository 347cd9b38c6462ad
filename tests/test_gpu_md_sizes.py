"""The persistent MD kernel at the basis sizes around which its dynamic LDS
stops holding the setup's triangles (117 | 118) and the setup kernel's does
(133 | 134), in one uneven ensemble with a trajectory (52 functions) whose
eigenvector refinement would have its fifth matrix in the LDS of the largest:
the same bits as the per-step kernels, which guards the persistent kernel's
compilation at these sizes too, and the oracle's trajectory."""
import numpy as np
import pytest

import oracle_bind as ob
from qcxms_amd import workloads as W
from test_cpu_emu_parts import molecule

pytestmark = pytest.mark.gpu

SIZES = (52, 117, 118, 119, 121, 122, 132, 133, 134)
STEPS = 3


def test_persistent_kernel_equals_per_step_kernels_at_the_lds_limits():
    import qcxms_amd
    trajs = []
    for n in SIZES:
        num, xyz = molecule(n)
        mass = np.array([W.atomic_mass(int(z)) for z in num])
        trajs.append(dict(num=num, xyz=xyz, velo=W.maxwell_boltzmann(mass, 500.0, n), mass=mass, eimp=0.2,
                          tadd=100.0 * W.FSTOAU))
    outs = []
    for fused in (False, True):
        print("fused", fused, flush=True)
        md = qcxms_amd.MdEnsemble(trajs, max_steps=STEPS, fused=fused, econv=1e-11, pconv=1e-9)
        md.run(STEPS + 1)
        outs.append(md.read())
        off = md.offsets
        md.close()
    a, b = outs
    for t, n in enumerate(SIZES):
        sl = slice(off[t], off[t + 1])
        for key in ("xyz", "velo", "grad", "qat", "list"):
            assert np.array_equal(a[key][sl], b[key][sl]), (n, key)
        assert a["results"][t].nstep == b["results"][t].nstep == STEPS
        assert a["results"][t].epot == b["results"][t].epot, n
    # the bars of the MD parity tests, both sides converged well below them
    for n in (52, 119, 134):
        t = SIZES.index(n)
        sl = slice(off[t], off[t + 1])
        ref = ob.md_run(trajs[t], steps_limit=0, max_steps=STEPS, opts=ob.default_opts(econv=1e-12, pconv=1e-10))
        de = abs(b["results"][t].epot - ref["state"].epot)
        dx = np.abs(b["xyz"][sl] - ref["xyz"]).max()
        print(f"nao={n} dE={de:.2e} dx={dx:.2e}", flush=True)
        assert de < 1e-8 and dx < 1e-8
