"""What the library's host code asks of the HIP runtime, from the log of
tests/cpp/fake_hip, which runs it over a runtime that runs nothing: devices,
streams, events, allocations and launches, without a GPU."""
import os
import subprocess

import pytest

PROG = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "fake_hip")


def log(*args):
    r = subprocess.run([PROG, *map(str, args)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    return r.stdout.splitlines()


def test_tree_freed_with_another_device_current():
    """The tree of device 1 is freed with device 0 current: the wait and the
    kept blocks' events belong to device 1, and device 0 is current again."""
    got = log("other_device", 300000, 4)
    assert "device_sync dev 1" in got
    records = [x for x in got if x.startswith("record")]
    assert records and all(x.startswith("record dev 1") for x in records)
    assert "current dev 0" in got


def test_tree_freed_during_a_capture():
    """Where the device may not be waited for, nothing is kept: the blocks'
    last uses are not known to have ended."""
    got = log("other_device_capturing", 300000, 4)
    assert sum(x.startswith("free dev 1") for x in got) == 2  # the tree's arrays and its scratch
    assert not any(x.startswith("record") for x in got)


def test_searches_on_two_streams():
    """An FP64 search that needs scratch (a query per lane) does not wait for
    one on another stream of the same tree, and a stream's later searches take
    the memory of its earlier ones."""
    got = log("two_streams", 300000, 4)
    assert sum("k_knn" in x for x in got) == 3
    assert not any(x.startswith(("wait", "host waits", "device_sync")) for x in got)
    assert not any(x.startswith("malloc") for x in got[got.index("again"):])


# 268.4 MB of fixed scratch, 8 bytes a particle of it for the densities, 94 MB
# for the search at its best
@pytest.mark.parametrize("n", [400000, 21000000, 27800000, 30000000, 33000000, 33554000])
def test_noalloc_search_with_little_scratch(n):
    """Once less than a third of the search's scratch is left, the search that
    needs none runs instead of a few workgroups."""
    got = log("noalloc", n, 8)
    lanes = [int(x.split("grid ")[1].split()[0]) for x in got if "k_knnILi3E" in x]
    waves = any("k_knn_wave" in x for x in got)
    assert "rc 0" in got and not any(x.startswith("malloc") for x in got)
    assert (lanes and min(lanes) >= 1360 and not waves) if n < 29600000 else (waves and not lanes)


# the fake device holds 4096 workgroups of the linking kernel
@pytest.mark.parametrize("n", [1, 64, 65, 262144, 524288, 524289, 4000000])
def test_fof_without_counters(n):
    """Up to two waves of particles per workgroup that fits, linking is a
    workgroup for each wave, and no counters are cleared for it."""
    got = log("fof", n)
    assert "rc 0" in got
    each = [x for x in got if "k_fof_each" in x]
    if n <= 524288:
        assert len(each) == 1 and f" grid {(n + 63) // 64} " in each[0]
        assert not any("k_fill_i32" in x or "5k_fofI" in x for x in got)
    else:
        assert not each and sum("5k_fofI" in x for x in got) == 1


# sizes at which the other kernel was the slower one
@pytest.mark.parametrize("what,n,k,form,kernel", [
    ("rows", 262144, 4, 0, "5k_knnI"), ("rows", 262144, 5, 0, "5k_knnI"), ("density", 262144, 6, 0, "5k_knnI"),
    ("rows", 262144, 7, 0, "5k_knnI"), ("density", 195112, 2, 0, "5k_knnI"), ("rows", 262144, 8, 0, "10k_knn_wave"),
    ("rows", 110592, 1, 0, "10k_knn_wave"), ("density", 204800, 4, 0, "10k_knn_wave"),
    ("density", 300000, 32, 1, "11k_knn_mixed"), ("density", 262144, 32, 1, "10k_knn_wave")])
def test_search_kernel(what, n, k, form, kernel):
    got = log(what, n, k, form)
    assert "rc 0" in got
    assert [x.split()[1][2:].startswith(kernel) for x in got if "k_knn" in x] == [True]


@pytest.mark.parametrize("n", [1000, (1 << 30) - 1, 1 << 30, (1 << 31) - 5000])
def test_adjoint_of_many_particles(n):
    """No launch of the adjoint has 2^32 threads, which none may have."""
    got = log("adjoint", n, 4)
    assert "rc 0" in got
    assert all(int(x.split("threads ")[1].split()[0]) < 1 << 32 for x in got if x.startswith("launch"))


def _build(n, form, gib=288):
    got = [x for x in log("build", n, form, gib) if x.startswith("tree ")][0].split()
    return int(got[1]), int(got[3]), int(got[5])  # made, most bytes at once, bytes held


# need: the sum of the tree's arrays
@pytest.mark.parametrize("n,form,need", [(2000000000, 0, 87516204768), (2000000000, 1, 124737430240)])
def test_large_trees_are_not_rounded_up(n, form, need):
    made, _, held = _build(n, form)
    assert made and held < need + (16 << 20)


@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("n", [200000000, 2000000000])
def test_build_gives_its_work_memory_back_first(n, form):
    """A build never holds the sort's work memory (32 bytes a particle and more)
    beside the tree's arrays, only the order (4 bytes a particle)."""
    made, peak, held = _build(n, form)
    assert made and peak < held + 5 * n


@pytest.mark.parametrize("gib,fits", [(131, True), (117, False)])
def test_build_on_a_full_device(gib, fits):
    """2e9 particles of the precision form: 124.7 GB of arrays and 8 of order."""
    assert _build(2000000000, 1, gib)[0] == fits


def test_trim_memory():
    """Everything kept goes back, on both devices, after the work that uses it."""
    got = log("trim", 300000, 4)
    f = [x for x in got if x.startswith("trimmed")][0].split()
    assert int(f[1]) > 0 and f[1] == f[3] and f[5] == "0" and f[7] == "0"
    assert "host waits for stream 0xa0" in got


def test_searches_on_a_full_device():
    """8 bytes a particle, a density's own need, are enough for every FP64
    call: where the lane search's scratch cannot be had, a wave per query runs."""
    got = log("full", 1000000, 4, 8)
    assert [x for x in got if " rc " in x] == ["rows rc 0", "density rc 0", "spline rc 0", "adjoint rc 0"]
    assert sum("k_knn_wave" in x for x in got) == 4 and not any("5k_knnI" in x for x in got)
    # with room for it the lane search runs
    got = log("full", 1000000, 4, 200)
    assert sum("5k_knnI" in x for x in got) == 4 and not any("k_knn_wave" in x for x in got)


def test_smoothed_velocities_memory():
    """Beside the rows (4 k bytes a particle) and a density's 8: densities and h
    16, means 32, dispersions 64, moments 64 and the buffer of the rest 72.  (The
    blocks of 8 bytes a particle are small enough to be kept, and rounded up by
    at most an eighth of 2^32.)"""
    n, k = 500000000, 4
    got = {x.split()[0]: x.split() for x in log("smooth", n, k) if " peak " in x}
    for what, own in (("mean", 120), ("disp", 184), ("moments", 248)):
        assert got[what][2] == "0" and int(got[what][4]) <= (4 * k + 8 + own) * n + 3 * (1 << 29) + (128 << 20), what
