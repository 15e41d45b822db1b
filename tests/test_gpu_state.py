"""State downloads of one and of several chunks, by one and by several host
threads, against receivers that sit on nodes (bilinear weights 1, 0, 0, 0: the
sample is the node's displacement, bit for bit)."""
import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def on_nodes(case, n=300, seed=3):
    """The case with n receivers on corners 0 of random elements (and on those
    of the first and the last element); no free field is added."""
    m = case.mesh
    pick = np.random.default_rng(seed).integers(0, m.nelems, n)
    pick[:2] = 0, m.nelems - 1
    node = m.corners()[pick, 0] - 1
    out = copy.copy(case)
    out.recv_elem = (pick + 1).astype(np.int32)
    out.recv_xy = m.nodes[node].copy()
    out.recv_ff = np.zeros(n, np.uint8)
    return out, node


# nodes: 378 (hanging, one chunk per level), 141,969 (hanging, two) and 275,151
# (three, so that the ring of four is used again)
@pytest.mark.parametrize("which", ["f2", "c3", "layer"])
@pytest.mark.parametrize("prec", [0, 1])
def test_state_at_receivers(which, prec):
    from damian_hip import cases, lib
    if which == "layer":
        text = cases.problem_text(4250, 1610, 1.0, 0.002, 0.1, 10, 2.5, [("p", 1000, "s", 500, 2000)], "WAVESV",
                                  [4100, 1500, 2000, 0, 1, 0.3, 0.1, 1.0, 4.0])
        case = cases.S.case_from_problem_text(text, sheet=(0.0, 100.0, 50.0), name="layer")
    else:
        case = cases.BUILDERS[which]()
    case, node = on_nodes(case)
    print(f"which={which} nodes={case.mesh.nnodes} prec={prec}", flush=True)
    s = lib.Solver(case, precision=prec)
    s.run(90, record=False)
    rec = s.run(2)
    u, up, mf = s.state()
    u2, up2, mf2 = s.state()
    s.close()
    assert np.abs(u).max() > 0
    assert np.array_equal(u.reshape(-1, 2)[node], rec[1])
    assert np.array_equal(up.reshape(-1, 2)[node], rec[0])
    for a, b in ((u, u2), (up, up2), (mf, mf2)):
        assert np.array_equal(a, b)
    h = case.hanging.reshape(-1, 3) - 1
    for v in (u.reshape(-1, 2), up.reshape(-1, 2)):
        assert np.array_equal(v[h[:, 0]], (v[h[:, 1]] + v[h[:, 2]]) / 2)
    # each level, or the mass, alone
    import ctypes as C
    t = lib.Solver(case, precision=prec)
    t.run(92, record=False)
    for k, want in enumerate((u, up, mf)):
        one = np.zeros_like(u)
        args = [None, None, None]
        args[k] = one.ctypes.data_as(C.c_void_p)
        assert lib.lib().dmp_get_state(t.h, *args) == 0
        assert np.array_equal(one, want)
    t.close()
