"""What the library does when device memory runs out, and what a failed solve
leaves, on the CPU: its entry points with a stand-in for the device of a set
capacity, on which kernels do not run (tests/host/fake_device.cpp)."""
import os
import subprocess

import pytest

from test_krylov_host import CLANG, HOST, ROOT, build_host

PKG = ROOT / "openstaple_amd"
SH = 2048  # half-sites of memory.cpp's 8^4 lattice
IP, VEC, ORDER = 512 * SH, 48 * SH, 4


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("memory")
    subprocess.run([CLANG, "-O1", "-std=c++17", "-I/opt/rocm/include", "-c", str(HOST / "fake_device.cpp"), "-o",
                    str(d / "fake.o")], check=True)
    build_host(HOST / "memory.cpp", d / "memory", str(d / "fake.o"), f"-L{PKG}", "-lopenstaple_amd", "-L/opt/rocm/lib",
               "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib")

    def go(*args):
        env = dict(os.environ)
        env["LD_LIBRARY_PATH"] = f"{os.environ.get('OSTP_HOST_TEST_LIB', PKG)}:{env.get('LD_LIBRARY_PATH', '')}"
        out = subprocess.run([str(d / "memory"), *map(str, args)], check=True, capture_output=True, text=True, env=env,
                             timeout=60).stdout
        return dict(line.split(" : ") for line in out.splitlines() if " : " in line and "WARNING" not in line)

    return go


def test_work_space_is_given_back(run):
    """With the gauge force's work space held and no memory beside it, the
    caller's allocations and the library's own get what they need."""
    got = run("given_back")
    assert set(got) == {"work space", "caller", "tables", "window", "again"}
    assert not {k: v for k, v in got.items() if v != "ok"}


def test_gauge_work_space_is_taken_whole(run):
    """Where there is room for the first of the gauge force's two buffers only,
    it is not kept; with room for both, both are."""
    assert run("refused") == {"refused": "ok", "taken": "ok"}


@pytest.mark.parametrize("after_gauge_force", [0, 1])
def test_force_in_little_memory(run, after_gauge_force):
    """The fermion force keeps the stout levels' QA and D_oe of the solutions
    where there is room.  In all memories from what it needs without them on,
    it succeeds, and no kernel is given memory that has been taken back."""
    extra = ["gauge"] if after_gauge_force else []
    (k, v), = run("force", 1 << 40).items()
    _, took, qa, hops = k.split()
    assert (v, qa, hops) == ("ok", "1", "1")
    # without: one level's QA and one source's D_oe instead of two
    least = int(took) - IP - ORDER * VEC
    kept = set()
    for room in list(range(least, 2 * int(took), VEC)) + list(range(2 * int(took), 7 * int(took), 8 * VEC)):
        (k, v), = run("force", room, *extra).items()
        assert v == "ok", (room - least, k, v)
        kept.add(tuple(k.split()[2:]))
    assert ("0", "0") in kept and ("1", "1") in kept, kept


def test_failed_multishift_leaves_no_old_solutions(run):
    """A solve that fails (its state does not advance) leaves zero solutions,
    with windows of residuals and with per-iteration updates."""
    assert run("failed_solve") == {"window 0": "ok", "window 1": "ok"}


@pytest.mark.parametrize("tens,first", [(12, 16), (13, 8)])  # 49152 half-sites, 53248
def test_short_solves_queue_few_iterations(run, tens, first):
    """A CG that takes 1 to 12 iterations: the first batch is shorter on large
    lattices, where an iteration queued in vain costs more than a batch's end;
    those that follow come from the rate of convergence, with a margin of a
    tenth and one iteration."""
    got = run("short", tens)
    assert len(got) == 12
    for k, v in got.items():
        stop, queued = map(int, k.split())
        assert int(v) == stop
        assert queued <= (first if stop <= first else stop + 4), (stop, queued)


@pytest.mark.parametrize("shape,tlsm,mode,force,moves", [
    ((8, 8, 8, 8), 1, 1, False, True), ((10, 10, 10, 10), 1, 1, False, True), ((16, 16, 16, 4), 1, 1, True, True),
    ((12, 18, 4, 14), 1, 1, False, True), ((16, 16, 16, 2), 1, 1, False, False), ((10, 10, 10, 8), 1, 1, False, False),
    ((64, 64, 2, 2), 1, 1, False, False), ((64, 64, 2, 2), 1, 2, True, True), ((8, 3, 4, 4), 1, 2, False, False),
    ((16, 16, 16, 8), 0, 1, False, False), ((16, 16, 16, 8), 0, 2, False, False), ((16, 16, 16, 8), 1, 0, False, False),
])
def test_gauge_force_kernels(run, shape, tlsm, mode, force, moves):
    """Which kernel forms the gauge force: by planes where that is faster or,
    asked for, possible; by links with the Wilson action, an odd extent, few
    sites a tile, and always where the staples are asked for (the integrator's
    last force)."""
    got = run("gauge", *shape, tlsm, mode)
    assert got["staples"] == "0 1 ok"
    f, m = ([int(v) for v in got[k].split()[:2]] for k in ("force", "moves"))
    assert all(v.endswith(" ok") for v in got.values())
    assert (f[0] > 0, f[1] > 0) == (force, not force)
    assert m == ([10, 1] if moves else [0, 11])
