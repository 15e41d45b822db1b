"""Layouts and kernels chosen by a rule, on both sides of its line: the samples
and states of every layout are the same bits, and those of the plain ones are
held to the CPU oracle by the other tests."""
import copy

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = {0: 1e-12, 1: 1e-5}   # against the oracle (FP32C against its FP64), as for every parity case


def layer(cases, nx, nz, sheet=None):
    w, h = 5.0 * nx, 5.0 * nz
    text = cases.problem_text(w, h, 0.4, 0.002, 0.1, 10, 2.5, [("p", 1000, "s", 500, 2000)], "WAVESV",
                              [0.6 * w, 0.6 * h, 0.5 * w, 0, 1, 0.2, 0.2, 1.0, 5.0])
    return cases.S.case_from_problem_text(text, sheet=sheet or (-3.3, w - 10.0, 4.1), name="layer")


def scattered(cases, case, n, seed):
    """n receivers at seeded points of the mesh, some in no element."""
    rng = np.random.default_rng(seed)
    out = copy.copy(case)
    e = rng.integers(0, case.nelems, n)
    c = case.mesh.corners()[e] - 1
    x0 = case.mesh.nodes[c[:, 0]]
    h = case.mesh.nodes[c[:, 2], 1] - x0[:, 1]
    out.recv_elem = np.where(rng.random(n) < 0.05, 0, e + 1).astype(np.int32)
    out.recv_xy = x0 + h[:, None] * rng.uniform(0.03, 0.97, (n, 2))
    out.recv_ff = cases.S.inside_soil(case.model, *out.recv_xy.T).astype(np.uint8)   # as the oracle does
    return out


# one workgroup up to 896 receivers, whole and partial groups of 256 above
@pytest.mark.parametrize("nrecv", [896, 897, 1024, 1025, 2500])
@pytest.mark.parametrize("prec", [0, 1])
def test_receivers_only_kernel(nrecv, prec):
    from damian_hip import cases, lib
    import oracle_ctypes as O
    case = scattered(cases, layer(cases, 60, 40), nrecv, nrecv)
    n = 90
    _, _, _, rec_o = O.run(case, nsteps=n, recv_interval=1)
    assert np.abs(rec_o).max() > 1e-3
    for tuning in ((128, 1, 0, 3), (256, 1, 0, 1)):
        print(f"nrecv={nrecv} prec={prec} tuning={tuning}", flush=True)
        s = lib.Solver(case, precision=prec)
        s.set_tuning(*tuning)
        # calls that end in the receivers-only kernel: whole launches
        rec = np.concatenate([s.run(k, noalloc=k == 6) for k in (30, 3, 3, 6, 48)])
        s.close()
        assert rel_l2(rec, rec_o) <= TOL[prec]
        assert not rec[:, case.recv_elem == 0].any()
