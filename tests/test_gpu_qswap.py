"""qswap of a three-dimensional box in one launch against its three parts in
numpy, in the reference's order (src/parallel.F90:4877-5200): along i, j, k in
turn the halo copies, then the average of the duplicate nodes.  q is copies
and 0.5 (a + b), so it is exact; the primitives of every cell written are
q2fvar of its q, compared at 4 ulp of each operand's magnitude."""
import numpy as np
import pytest

import astr_gpu_amd as ag
from test_gpu_adjoint import test_adjoint_matches_torch_autograd as adjoint_matches

pytestmark = pytest.mark.gpu
HM = 5


def parts(q, n, npdc):
    """The three parts on a copy of the haloed q; the cells written."""
    q = q.copy()
    wr = np.zeros(q.shape[:3], bool)
    own = [slice(HM, HM + m + 1) for m in n]
    for d in range(3):
        if npdc[d] != 3:
            continue

        def at(c):
            s = list(own)
            s[d] = HM + c
            return tuple(s)

        for r in range(1, HM + 1):
            q[at(-r)] = q[at(n[d] - r)]
            q[at(n[d] + r)] = q[at(r)]
            wr[at(-r)] = wr[at(n[d] + r)] = True
        q[at(0)] = q[at(n[d])] = 0.5 * (q[at(0)] + q[at(n[d])])
        wr[at(0)] = wr[at(n[d])] = True
    return q, wr


@pytest.mark.parametrize("npdc", [(3, 3, 3), (3, 4, 3), (4, 3, 3), (3, 3, 4), (4, 4, 3), (3, 4, 4), (4, 3, 4)])
@pytest.mark.parametrize("dims", [(16, 16, 16), (17, 19, 23), (33, 16, 18), (64, 21, 17), (18, 65, 32)])
def test_one_launch_equals_the_parts(dims, npdc):
    print(f"case qswap {dims} {npdc}", flush=True)
    p = ag.default_params(dims, npdci=npdc[0], npdcj=npdc[1], npdck=npdc[2])
    s = ag.AstrSolver(p)
    s.upload_geom(*ag.box_metrics(p))
    st = ag.tgv_state(p)
    rng = np.random.default_rng(3)
    q = np.asfortranarray(1.0 + 0.1 * rng.random(st["q"].shape))
    q[..., 4] += 20.0
    prim = {"rho": 1.0, "vel": 2.0, "prs": 3.0, "tmp": 4.0}
    prim = {k: np.asfortranarray(np.full(st[k].shape, v)) for k, v in prim.items()}
    s.upload_state(q, prim["rho"], prim["vel"], prim["prs"], prim["tmp"])
    s.qswap()
    g = s.download_state()
    s.close()
    ref, wr = parts(q, dims, npdc)
    own = tuple(slice(HM, HM + m + 1) for m in dims)
    see = wr.copy()
    see[own] = True
    assert np.array_equal(g["q"][see], ref[see])
    rho = ref[..., 0]
    vel = ref[..., 1:4] / rho[..., None]
    ke = 0.5 * rho * (vel ** 2).sum(-1)
    const6 = 1.0 / (p.gamma - 1.0)
    prs = (ref[..., 4] - ke) / const6
    tmp = prs / rho * (p.gamma * p.mach ** 2)
    ulp = 4 * np.finfo(float).eps
    scale = (np.abs(ref[..., 4]) + ke) / const6
    assert np.array_equal(g["rho"][wr], rho[wr])
    assert np.all(np.abs(g["vel"] - vel)[wr] <= ulp * np.abs(vel)[wr])
    assert np.all(np.abs(g["prs"] - prs)[wr] <= ulp * scale[wr])
    assert np.all(np.abs(g["tmp"] - tmp)[wr] <= ulp * (scale / rho * p.gamma * p.mach ** 2 + tmp)[wr])
    # and nothing else
    rest = ~wr
    rest[:HM] = rest[-HM:] = False
    rest[:, :HM] = rest[:, -HM:] = rest[:, :, :HM] = rest[:, :, -HM:] = False
    for k, v in (("rho", 1.0), ("prs", 3.0), ("tmp", 4.0)):
        assert np.all(g[k][rest] == v)


@pytest.mark.parametrize("dims", [(16, 16, 16), (17, 23, 16), (34, 17, 19)])
def test_reversal_in_one_launch(dims):
    """The reversed parts in one launch, inside the whole reversal, against
    PyTorch's autograd of the same forward (its own bounds)."""
    adjoint_matches(1, 1, None, dims)
