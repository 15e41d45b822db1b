"""The library's host code without a device: error paths, launch shapes and
allocations, under the HIP runtime of host_hip/ (which notes launches and runs
no kernel)."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
PRELUDE = """
import ctypes, sys
sys.path.insert(0, {python!r})
import numpy as np
from damian_hip import cases, lib
hh = ctypes.CDLL("libamdhip64.so.7")
hh.hh_launches.restype = hh.hh_hostmallocs.restype = ctypes.c_char_p
def layer(nx, nz):
    w, h = 5.0 * nx, 5.0 * nz
    t = cases.problem_text(w, h, 0.4, 0.002, 0.1, 10, 2.5, [("p", 1000, "s", 500, 2000)], "WAVESV",
                           [0.6 * w, 0.6 * h, 0.5 * w, 0, 1, 0.2, 0.2, 1.0, 5.0])
    return cases.S.case_from_problem_text(t, sheet=(-3.3, w - 10.0, 19.1), name="layer")
def fronts(nx, nz, part, seed=7):
    # 10 m cells, halved everywhere but in the first `part` of the width, there at random
    w, h = 10.0 * nx, 10.0 * nz
    t = cases.problem_text(w, h, 1.0, 0.002, 0.2, 10, 5.0, [("p", 1000, "s", 500, 2000)], "WAVESV",
                           [0.6 * w, 0.6 * h, 0.5 * w, 0, 1, 0.3, 0.0, 1.0, 3.0])
    mdl = cases.S.build_model(cases.S.parse_problem(t))
    rng = np.random.default_rng(seed)
    m = cases.S.quadtree_mesh(mdl.totcols - 1, mdl.totrows - 1, mdl.blength, 2,
                              lambda x, z, s: (x >= part * w) | (rng.random(len(x)) < 0.5))
    return cases.S.finish_case(mdl, m, sheet=(-3.3, w - 10.0, 19.1), name="fronts")
def launches():
    return [l.split() for l in hh.hh_launches().decode().splitlines()]
def fail(name, n=1, times=1):
    hh.hh_fail(name.encode(), n, times)
"""


@pytest.fixture(scope="session")
def host_hip(tmp_path_factory):
    """Runs a script under that runtime; returns its standard output and the
    layouts that the library says it built (dicts of numbers)."""
    d = tmp_path_factory.mktemp("host_hip")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    HERE / "host_hip" / "host_hip.cpp", f"-Wl,--version-script={HERE / 'host_hip' / 'versions.map'}",
                    "-Wl,-soname,libamdhip64.so.7", "-o", d / "libamdhip64.so.7"], check=True)

    def run(script):
        prelude = PRELUDE.format(python=str(HERE.parent / "damian.par_amd" / "python"))
        r = subprocess.run([sys.executable, "-c", prelude + script], capture_output=True, text=True, timeout=300,
                           env=dict(os.environ, LD_LIBRARY_PATH=str(d), DMP_LAYOUT_STATS="1"))
        assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
        layouts = []
        for line in r.stderr.splitlines():
            if line.startswith("layout "):
                layouts.append({k: float(v) for k, v in (w.rstrip(",").split("=") for w in line.split() if w.count("=") == 1 and not w.startswith("hist="))})
        return r.stdout, layouts

    return run


@pytest.mark.parametrize("name", ["f1", "c1"])
def test_failed_call_leaves_last_run_ms(host_hip, name):
    """The device time of the last complete call, whether it is asked for before
    or after a call that fails part way (one tile, many tiles)."""
    host_hip(f"""
s = lib.Solver(cases.{name}())
s.set_tuning(64, 1, 0, 2)
s.run(10)
launches()
s.run(20)
want = len(launches())
for asked in (False, True):
    if asked:
        assert s.last_run_ms() == want
    fail("hipLaunchKernel", 4)
    try:
        s.run(30)
        raise SystemExit("not refused")
    except lib.DmpError as e:
        assert e.code == -3
    assert s.last_run_ms() == want, (asked, s.last_run_ms(), want)
s.run(6)
assert 0 < s.last_run_ms() < want
""")


def test_pinned_memory_is_coherent(host_hip):
    """The host reads the receiver ring and the completion word before the
    stream is idle, so both ask for coherent memory by name."""
    out, _ = host_hip("""
s = lib.Solver(cases.f1())
print(hh.hh_hostmallocs().decode())
""")
    mapped, coherent = 0x2, 0x40000000
    made = [(int(a), int(b)) for a, b in (l.split() for l in out.splitlines() if l)]
    assert sorted(n for n, _ in made)[0] == 4 and len(made) == 3
    assert all(f == mapped | coherent for _, f in made)


@pytest.mark.parametrize("name", ["f1", "f2"])
def test_shape_that_was_got_can_be_set(host_hip, name):
    """Setting the shape that dmp_get_tuning gave (a small mesh in one tile), or
    going back to dmp_init's, gives that layout again; where it is still in
    place nothing is built."""
    out, layouts = host_hip(f"""
s = lib.Solver(cases.{name}())
t = s.tuning()
s.set_tuning(*t)
s.set_tuning(64, 1, 0, 2)
s.set_tuning(*t)
lib.lib().dmp_set_tuning(s.h, None)
s.set_tuning(*t)
launches()
s.run(40)
print(len([l for l in launches() if "step_kernel" in l[0]]))
""")
    assert [(l["K"], l["whole"]) for l in layouts] == [(3, 1), (2, 0), (3, 1)]
    assert layouts[0] == layouts[2] and layouts[0]["depth"] > 8
    assert int(out) == -(-40 // layouts[0]["depth"])


def test_same_shape_of_a_large_mesh_is_not_built_again(host_hip):
    _, layouts = host_hip("""
s = lib.Solver(cases.c1())
s.set_tuning(256, 1, 0, 3)
s.set_tuning(256, 0, 12, 3)
lib.lib().dmp_set_tuning(s.h, None)
""")
    assert len(layouts) == 1


@pytest.mark.parametrize("what,n", [("hipLaunchKernel", 500), ("hipMalloc", 100)])
def test_failed_autotune_leaves_shape_and_state(host_hip, what, n):
    """A search that fails part way gives back the shape, the step and the
    state (a launch that fails; memory that runs out while a layout is built)."""
    host_hip(f"""
s = lib.Solver(cases.c1())
s.set_tuning(100, 0, 12, 2)
launches()
s.run(7, record=False)
want = s.tuning()
kernels = {{tuple(l) for l in launches() if "step_kernel" in l[0]}}
fail({what!r}, {n})
try:
    s.autotune(20)
    raise SystemExit("not refused")
except lib.DmpError as e:
    assert e.code in (-2, -3), e
assert s.tuning() == want, s.tuning()
step = ctypes.c_int()
lib.lib().dmp_get_step(s.h, ctypes.byref(step))
assert step.value == 7, step.value
launches()
out = s.run(6)
assert out.shape[0] == 6
assert {{tuple(l) for l in launches() if "step_kernel" in l[0]}} == kernels
""")


def test_no_launch_without_a_layout(host_hip):
    """Memory that runs out while a shape is built, and again while the one
    before is, leaves no layout: a run call builds it or fails, and launches
    nothing until it is there."""
    _, layouts = host_hip("""
s = lib.Solver(cases.c1())
s.set_tuning(128, 1, 0, 3)
want = s.tuning()
def refused(call, code):
    launches()
    try:
        call()
        raise SystemExit("not refused")
    except lib.DmpError as e:
        assert e.code == code, e
    assert not launches()
fail("hipMalloc", 5, 1000)
refused(lambda: s.set_tuning(64, 1, 0, 2), -2)
assert s.tuning() == want
refused(lambda: s.run(6), -2)
fail("hipMalloc", 10**9)
refused(lambda: s.run(6, noalloc=True), -5)
assert s.run(6).shape[0] == 7
assert s.run(6, noalloc=True).shape[0] == 6
s.close()
""")
    assert (layouts[-1]["B"], layouts[-1]["K"]) == (128, 3)


# one tile for many shapes; tiles between patches, which are no larger than 64
# or 128 nodes; neither
@pytest.mark.parametrize("case", ["cases.f1()", "cases.f2()", "layer(450, 440)", "fronts(400, 200, 0.5)", "cases.c1()"])
def test_autotune_builds_no_layout_twice(host_hip, case):
    _, layouts = host_hip(f"""
s = lib.Solver({case})
s.set_tuning(33, 1, 0, 2)
s.autotune(4)
""")
    searched = [tuple(sorted((k, v) for k, v in l.items() if k != "K" or not l["whole"])) for l in layouts[2:]]
    assert len(searched) > 8
    assert len(set(searched[:-1])) == len(searched) - 1   # the last is the one found, built again


def test_state_download_without_threads(host_hip):
    """Host threads only speed a large download up: where none can be started
    (no address space for a stack) the call still moves every byte."""
    host_hip("""
import os, resource
os.environ["DMP_THREADS"] = "1"
case = cases.c4_valley(200.0)
s = lib.Solver(case)
n = case.mesh.nnodes
a = [np.full(2 * n, np.nan) for _ in range(3)]
os.environ["DMP_THREADS"] = "8"
size = int(open("/proc/self/statm").read().split()[0]) * os.sysconf("SC_PAGE_SIZE")
resource.setrlimit(resource.RLIMIT_AS, (size + (2 << 20), resource.RLIM_INFINITY))
import threading
try:
    threading.Thread(target=int).start()
    raise SystemExit("a thread can be started: nothing is tested")
except RuntimeError:
    pass
rc = lib.lib().dmp_get_state(s.h, *[x.ctypes.data_as(ctypes.c_void_p) for x in a])
resource.setrlimit(resource.RLIMIT_AS, (resource.RLIM_INFINITY, resource.RLIM_INFINITY))
assert rc == 0, lib.last_error(s.h)
assert all(np.isfinite(x).all() for x in a)
""")


@pytest.mark.parametrize("nrecv,groups", [(1, 1), (896, 1), (897, 4), (2000, 8)])
def test_receivers_only_kernel_grows_with_its_receivers(host_hip, nrecv, groups):
    out, _ = host_hip(f"""
import copy
case = copy.copy(cases.c1())
case.recv_elem = np.resize(case.recv_elem, {nrecv})
case.recv_xy = np.resize(case.recv_xy, ({nrecv}, 2))
case.recv_ff = np.resize(case.recv_ff, {nrecv})
s = lib.Solver(case)
s.set_tuning(256, 1, 0, 3)
for noalloc in (False, True):
    launches()
    s.run(3, noalloc=noalloc)
    print(*[l[1:3] for l in launches() if "recv_kernel" in l[0]])
""")
    run, noalloc = [eval(l) for l in out.splitlines()]
    assert int(run[0]) == groups and int(run[0]) * int(run[1]) >= nrecv
    assert int(noalloc[0]) * int(noalloc[1]) >= nrecv > (int(noalloc[0]) - 1) * int(noalloc[1])


# 256 compute units: patches above 196,608 nodes
@pytest.mark.parametrize("case,tuning,want", [
    ("layer(443, 440)", (256, 1, 0, 1), dict(B=256, threads=256, patches=0)),       # 195,804 nodes
    ("layer(443, 440)", (64, 1, 0, 1), dict(B=64, threads=64, patches=0)),
    ("layer(450, 440)", (256, 1, 0, 1), dict(B=64, threads=256, patches=3134)),     # 198,891
    ("layer(450, 440)", (32, 1, 0, 1), dict(B=32, threads=256, patches=3134)),
    ("fronts(400, 200, 0.5)", (256, 1, 0, 1), dict(B=128, threads=256)),            # hanging nodes in half of it
    ("fronts(400, 200, 0.5)", (64, 1, 0, 1), dict(B=64, threads=128)),
    ("fronts(400, 200, 0.05)", (512, 1, 0, 1), dict(B=64, threads=256)),            # in a twentieth
    ("cases.c2()", (512, 1, 0, 1), dict(B=512, patches=0)),
])
def test_one_step_layouts(host_hip, case, tuning, want):
    _, layouts = host_hip(f"""
s = lib.Solver({case})
s.set_tuning(300, 1, 0, 2)
s.set_tuning(*{tuning})
""")
    got = layouts[-1]
    assert got["K"] == 1
    assert {k: got[k] for k in want} == want
    if "patches" not in want:
        assert got["patches"] > 100


# a mesh with uniform parts, one without
@pytest.mark.parametrize("case", ["cases.c2()", "fronts(60, 40, 1.0)"])
def test_one_step_tiles_that_do_not_fit(host_hip, case):
    """Tiles of a small mesh are as large as asked for; where those do not fit,
    the mesh is cut into patches and small tiles and the shape is taken."""
    _, layouts = host_hip(f"""
s = lib.Solver({case})
s.set_tuning(512, 1, 0, 1)
s.set_tuning(1024, 1, 0, 1)
assert s.tuning() == (1024, 1, 0, 1)
s.run(9)
""")
    assert [(l["B"], l["patches"] > 0) for l in layouts[-2:]] == [(512, False), (layouts[-1]["B"], case == "cases.c2()")]
    assert layouts[-1]["B"] in (64, 128)


# few patches among small tiles, which they would widen; most of the mesh in
# them; half of it, where plain tiles would need as many rounds or more
@pytest.mark.parametrize("case,tuning,patched", [
    ("cases.c2()", (64, 1, 0, 2), False),
    ("cases.c2()", (64, 1, 0, 3), False),
    ("cases.c2()", (64, 1, 0, 4), True),
    ("layer(300, 200)", (64, 1, 0, 2), False),
    ("layer(300, 200)", (128, 1, 0, 2), True),
    ("layer(300, 200)", (48, 1, 0, 8), True),
    ("fronts(200, 100, 0.4)", (64, 1, 0, 2), False),
    ("fronts(200, 100, 0.4)", (64, 1, 0, 3), True),
])
def test_block_patches_where_they_pay(host_hip, case, tuning, patched):
    _, layouts = host_hip(f"""
s = lib.Solver({case})
s.set_tuning(300, 1, 0, 1)
s.set_tuning(*{tuning})
""")
    assert (layouts[-1]["B"], layouts[-1]["K"]) == (tuning[0], tuning[3])
    assert (layouts[-1]["patches"] > 0) == patched


# the shapes of test_gpu_layouts.py
@pytest.mark.parametrize("case", ["layer(300, 200)", "cases.c4_valley(200.0, 'SV', 10.0)"])
def test_block_patch_shapes_of_the_gpu_tests(host_hip, case):
    from test_gpu_layouts import BLOCK_SHAPES
    _, layouts = host_hip(f"""
s = lib.Solver({case})
s.set_tuning(300, 1, 0, 1)
for t in {BLOCK_SHAPES}:
    try:
        s.set_tuning(*t)
    except lib.DmpError as e:
        assert e.code == -4 and t[3] > 4
        s.set_tuning(300, 1, 0, 1)
""")
    built = {(l["B"], l["K"]): l for l in layouts if l["K"] > 1}
    assert {k for _, k in built} >= {2, 3, 4}
    assert all(built[b, k]["patches"] > 0 for b, k in built if (b, k) in {(t[0], t[3]) for t in BLOCK_SHAPES})


# the shapes that test_gpu_patches.py::test_halved_tiles does not leave out
@pytest.mark.parametrize("case,built,halved", [
    ("cases.c4_valley(200.0, 'SV', 10.0)", [256, 200, 170, 140], [256, 200, 170]),
    ("cases.c2()", [256, 170, 140], [170]),
])
def test_halved_tiles_of_the_gpu_tests(host_hip, case, built, halved):
    out, layouts = host_hip(f"""
s = lib.Solver({case})
for t in ((256, 1, 0, 3), (200, 1, 0, 4), (170, 0, 12, 4), (140, 1, 0, 4)):
    s.set_tuning(300, 1, 0, 1)
    try:
        s.set_tuning(*t)
        print(t[0])
    except lib.DmpError as e:
        assert e.code == -4
""")
    assert [int(b) for b in out.split()] == built
    assert sorted({int(l["B"]) for l in layouts if l["K"] > 1 and l["halved"]}, reverse=True) == halved
