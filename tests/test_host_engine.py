"""Error paths and launch decisions of the engine's host side, on the CPU:
libgfc.so runs against the HIP calls of tests/fake_hip_driver.cpp, whose device
memory is host memory and whose kernels do nothing."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "gaugefix-coulomb_amd", "lib")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None or not os.path.exists(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no host C++ compiler or no HIP headers")
    exe = str(tmp_path_factory.mktemp("fake_hip") / "fake_hip_driver")
    # -rdynamic: the driver's HIP calls are found before libamdhip64's
    subprocess.run([cxx, "-std=c++17", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROCM, "include"),
                    os.path.join(ROOT, "tests", "fake_hip_driver.cpp"), "-o", exe,
                    "-L", LIB, "-lgfc", "-Wl,-rpath," + LIB, "-lpthread"], check=True)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, (r.returncode, r.stdout[-2000:], r.stderr[-2000:])
        return r.stdout.splitlines()

    return run


def test_transfers_without_a_ring(driver):
    """16^3 x 32 (75 MB) would go through the ring of pinned slots; when that
    memory is not to be had, the plain copy takes its place and nothing of the
    failed request is left behind, neither HIP's last error (the launch check
    after the copy would report it) nor a message."""
    first, *log = driver("no_ring", 16, 32)
    assert first == "up 0 down 0 same 1 message []"
    assert [l for l in log if l.startswith("copy")] == ["copy 75497472"] * 2


@pytest.mark.parametrize("pinned", [0, 1])
@pytest.mark.parametrize("ns,nt", [(8, 16), (16, 32)])
def test_route_of_host_arrays(driver, ns, nt, pinned):
    """Small transfers and arrays in pinned memory are one plain copy; large
    pageable ones (75 MB) go through the ring's 8 MiB slots."""
    first, *log = driver("round_trip", ns, nt, pinned)
    assert first == "up 0 down 0 same 1 message []"
    n = ns ** 3 * nt * 576
    copies = [int(l.split()[1]) for l in log if l.startswith("copy")]
    if ns == 8 or pinned:
        assert copies == [n, n]
    else:
        assert sum(copies) == 2 * n and max(copies) == 8 << 20


def test_transfers_without_host_memory(driver):
    """No exception leaves a C entry: without memory for the copying threads the
    transfer is one plain copy."""
    first, *log = driver("round_trip", 16, 32, 0, 1)
    assert first == "up 0 down 0 same 1 message []"
    assert [l for l in log if l.startswith("copy")] == ["copy 75497472"] * 2


def _fix(driver, ns, nt, prec=0, sweeps=20, hits=2, group=0, lanes=0):
    first, *log = driver("fix", ns, nt, prec, sweeps, hits, group, lanes)
    assert first.startswith(f"fix -1 sweeps {sweeps} ")
    return log


@pytest.mark.parametrize("ns,nt,slices", [
    (2, 256, 1), (2, 258, 0), (2, 2000, 0), (4, 2, 1), (4, 512, 1), (4, 514, 0),
    (6, 256, 1), (6, 258, 0), (8, 2, 1), (8, 2000, 1), (10, 64, 0), (10, 130, 0),
    (10, 132, 1), (10, 256, 1), (10, 258, 0), (10, 1022, 0), (10, 1024, 1), (12, 16, 0)])
def test_route_of_small_lattices(driver, ns, nt, slices):
    """FP64 sweeps in one launch per host decision or in one per half-sweep, on
    both sides of each line of the rule."""
    log = _fix(driver, ns, nt)
    assert len([l for l in log if "k_sweep_slices" in l]) == slices
    launches = [l for l in log if "k_sweep" in l and "slices" not in l]
    assert len(launches) == 0 if slices else len(launches) >= 20


@pytest.mark.parametrize("nt,hits", [(16, 2), (4096, 2), (4096, 30), (16384, 2), (2, 100000)])
def test_work_of_a_launch_is_bounded(driver, nt, hits):
    """k_sweep_slices at ns = 8: the half-sweeps of a launch follow the
    timeslices that take turns on a CU and the hits, so that a launch stays near
    20 ms; together they are all of them, in order."""
    n = 5000
    log = _fix(driver, 8, nt, sweeps=n, hits=hits)
    runs = [tuple(map(int, l.split()[1:])) for l in log if l.startswith("sweeps")]
    assert runs[0][0] == 0 and runs[-1][1] == n
    assert all(a[1] == b[0] for a, b in zip(runs, runs[1:]))
    most = max(b - a for a, b in runs)
    us = -(-nt // 256) * (3.5 + 0.65 * hits)
    assert most == 1 or most * us < 20e3
    assert most * us > 5e3  # and no shorter than that either


@pytest.mark.parametrize("group,lanes,launches", [(0, 1, 20), (0, 2, 40), (0, 4, 80), (4, 0, 80),
                                                  (-1, 0, 20)])
def test_groups_and_streams_that_are_asked_for(driver, group, lanes, launches):
    """slice_group and slice_lanes are kept to where the default would be one
    launch (8^3 x 16, 20 half-sweeps): nt / lanes timeslices per group."""
    log = _fix(driver, 8, 16, group=group, lanes=lanes)
    sweeps = [l.split() for l in log if "k_sweep" in l]
    assert all("slices" not in l[1] for l in sweeps) and len(sweeps) == launches
    assert all(int(l[2]) == (16 if group < 0 else 16 // (lanes or 4)) for l in sweeps)


@pytest.mark.parametrize("sweeps,length,done", [
    (20, 20, -1), (20, 7, -1), (20, 40, -1), (20, 0, -1), (3000, 2500, -1), (2048, 2048, -1),
    (20, 20, 5), (20, 3, 5), (3000, 2500, 1024), (3000, 2500, 1030)])
def test_trace_of_a_fix_that_ends_anywhere(driver, sweeps, length, done):
    """Every value of the trace up to its length or the last half-sweep is set,
    and none behind it; a fix whose launch after half-sweep `done` fails leaves
    those it had."""
    rc, done = (-3, done) if done >= 0 else (-1, sweeps)
    assert driver("trace", 4, 2, sweeps, length, done if rc == -3 else -1)[0] == \
        f"trace {rc} set {min(length, done)} of {length}"


@pytest.mark.parametrize("ns,prec,retire,rc,why", [
    (16, 0, 0, -3, "hipGetLastError(): error"), (16, 1, 0, -3, "hipGetLastError(): error"),
    (16, 0, 1, -3, "hipGetLastError(): error"),
    (6, 0, 1, -6, "gfc_job_fix: retire_slices needs ns a multiple of 8")])
def test_failed_fix_leaves_the_identity(driver, ns, prec, retire, rc, why):
    """Whether a launch fails half way or the call is refused, the last thing
    written is G = 1, and the message is that of the failure."""
    first, *log = driver("fix", ns, 4, prec, 20, 2, 0, 0, retire, 7)
    assert first == f"fix {rc} sweeps 0 message [{why}]"
    assert "k_g_identity" in [l for l in log if l.startswith("launch")][-1]


def test_fixed_configuration_costs_no_frame(driver):
    """An FP64 fix whose input meets the tolerance looks at it, writes G = 1 and
    U, and builds nothing for sweeps."""
    first, *log = driver("fix", 16, 4, 0, 0, 2, 0, 0)
    assert first == "fix 0 sweeps 0 message []"
    names = [l.split()[1] for l in log if l.startswith("launch")]
    kernels = ("k_obs_aos", "k_reduce_final", "k_g_identity", "k_materialize")
    assert len(names) == 4 and all(k in n for k, n in zip(kernels, names))


def test_the_columns_are_walked_once(driver):
    """A fix walks the columns on its way into the axial frame (a thread per
    column) and leaves it site by site."""
    log = [l.split() for l in _fix(driver, 16, 4) if l.startswith("launch")]
    assert [l[2:] for l in log if "k_frame_begin" in l[1]] == [["16", "64"]]
    assert [l[2:] for l in log if "k_frame_end" in l[1]] == [["64", "256"]]


@pytest.mark.parametrize("offset", [0, 8])
def test_loads_by_the_alignment_of_a_callers_array(driver, offset):
    """16-byte loads straight to LDS only from addresses that allow them."""
    first, *log = driver("noalloc", offset)
    assert first == "noalloc 0"
    names = [l.split()[1] for l in log if "_aos" in l]
    # template arguments CHECK, ALIGNED of the residues, ALIGNED of the plaquettes
    lo = "ILb0ELb%dEE" % (offset == 0), "ILb%dEE" % (offset == 0)
    assert len(names) == 2 and all(t in n for t, n in zip(lo, names))
