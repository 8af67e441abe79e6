"""The library's sources built for the host under AddressSanitizer (no GPU).

tests/host_build compiles csrc/*.hip with the host compiler against a stand-in
for the HIP runtime (lanes are fibers, a workgroup is a host thread, device
allocations have exactly the asked size), so the library's own C entry points
run end to end: every launch form of every search, sorts, CSR builds and
batched queries.  tests/host_build/check.cpp holds the cases and compares with
serial references.
"""
import fcntl
import os
import shutil
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_build")
CXX = "/opt/rocm/llvm/bin/clang++"


@pytest.fixture(scope="module")
def check():
    if shutil.which(CXX) is None:
        pytest.skip("%s is not available" % CXX)
    with open(os.path.join(HERE, ".build.lock"), "w") as lk:
        fcntl.flock(lk, fcntl.LOCK_EX)
        subprocess.run(["make", "-s", "-j8", "-C", HERE], check=True)

    def run(*args):
        cmd = [os.path.join(HERE, "_build", "check")] + [str(a) for a in args]
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=300,
                           env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"))
        assert r.returncode == 0, "%s\n%s\n%s" % (" ".join(cmd[1:]), r.stdout[-1000:], r.stderr[-4000:])
        return r.stdout
    return run


@pytest.mark.parametrize("marks,wgs,tier", [(1, 1, 16), (0, 2, 100000), (1, 2, 100000), (0, 1, 16)])
def test_searches(check, marks, wgs, tier):
    """Every strategy and mode on paths, stars, skewed graphs (symmetric and
    directed) and a grid: claims on labels (marks 1) or on the bitmask, the
    narrow persistent kernel with pieces that spill (the star), the grid tier
    from `tier` edges on."""
    check("searches", marks, wgs, tier)


def test_wide_persistent(check):
    """More than 256 persistent workgroups: the form with the shared queue."""
    check("wide_persistent")


@pytest.mark.parametrize("case", ["sorts", "primitives", "builds", "scan_segments"])
def test_arrays_and_builds(check, case):
    """Sorts on both sides of the one-workgroup limit, scans, consecutive
    removals and CSR builds."""
    check(case)


@pytest.mark.parametrize("levels,persistent", [(0, 0), (3, 0), (2, 1)])
def test_batched(check, levels, persistent):
    """40 queries over four graphs in each form of a step, results taken in
    and against the order of submission."""
    check("batched", levels, persistent)


@pytest.mark.parametrize("levels", [1, 2, 3, 6, 8])
def test_strategies_share_a_problem(check, levels):
    """A direction-optimizing search with `levels` levels per host check, then
    every other strategy, on one problem: its partial sums, left behind, made
    captured expand-contract loops replay for ever."""
    check("shared_problem", levels)


def test_search_depth_with_a_late_first_workgroup(check):
    """Contract-expand in launches per level where workgroup 0 starts last: its
    plain store of the level before overwrote what the others had found."""
    check("late_first_workgroup")


@pytest.mark.parametrize("case", ["sort_few_resident", "sort_grouped"])
def test_sort_progress(check, case):
    """A place ends whatever waits for whatever: 20 workgroups at a time on a
    small device (blocks grouped by XCD ran into the bounded wait there), and the
    fewest with which blocks are grouped."""
    check(case)


def test_narrow_persistent_grid(check):
    """The narrow persistent kernel's grid follows its own occupancy."""
    check("narrow_occupancy")


def test_tuning_round_trip(check):
    """Setting the tuning that was read leaves the choices per graph alone."""
    check("tuning_round_trip")


def test_sort_after_a_failed_one(check):
    """A sort that fails after its launches keeps its report words until its
    kernels have run; they were given to the next sort at once."""
    check("sort_after_error")


def test_short_of_device_memory(check):
    """Sorts and builds that find no memory for the scratch they want go on with
    the little they need."""
    check("short_of_memory")


def test_no_memory_for_frontier_pieces(check):
    """Expand-contract without room for the narrow kernel's pieces."""
    check("no_frontier_pieces")


def test_tiny_queues(check):
    """A sizing factor that asks for less than one queue entry: no value array
    was allocated for an edge frontier's single one."""
    check("tiny_queues")


def test_orders_of_results(check):
    """Batched results taken in and out of the order of submission: out of it,
    every second window held a result that was not asked for next."""
    check("result_orders")


def test_average_duty(check):
    """Instrumented searches of every strategy and mode report a duty of at most
    one: hybrid's level launches counted as work but not as time."""
    check("duty")


def test_late_blocks(check):
    """Scans, removals and CSR builds where a block cannot start while the others wait for
    it (as beside a persistent kernel that holds the GPU): the call finishes what
    gave up; it failed."""
    check("late_blocks")


def test_late_sorts(check):
    """The same of sorts, where such a place failed and the later ones moved
    nothing; a serving workgroup may be the one that cannot start."""
    check("late_sorts")
