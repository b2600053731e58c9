"""What the library's host side queues, without a GPU: tests/native/fake_device.cpp
defines the HIP calls that the library makes, so that launches, stream waits and
allocations are seen (and allocations can fail) while nothing runs."""
import os
import subprocess

import pytest

from astc_encoder_amd import _capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    exe = tmp_path_factory.mktemp("native") / "fake_device"
    libdir = os.path.dirname(_capi.LIB_PATH)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                    os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "native", "fake_device.cpp"), "-o",
                    str(exe), "-rdynamic", "-L", libdir, "-lastc_mi355x", f"-Wl,-rpath,{libdir}",
                    "-Wl,-rpath-link,/opt/rocm/lib"], check=True)

    def run(*args):
        r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
        return r.stdout

    return run


def fields(line):
    words = line.split()
    return dict(zip(words[::2], (int(w) for w in words[1::2])))


def test_batches_of_a_trace_with_overlapping_destinations_follow_each_other(fake):
    """Requests of different batches with one destination: the later batch's work is
    queued behind the earlier one's, whichever slots they run on.  Batches whose
    destinations lie apart stay free of each other."""
    got = fields(fake("one_destination"))
    assert got["rc"] == 0 and got["batches"] == 3 and got["peak_inflight"] == 3
    assert got["unordered"] == 0 and got["ordered"] > 0
    apart = fields(fake("own_destinations"))
    assert apart["rc"] == 0 and apart["batches"] == 3 and apart["ordered"] == 0


@pytest.mark.parametrize("k", range(12))
def test_a_failed_growth_of_the_work_lists_is_tried_again(fake, k):
    """Two slots of six buffers each: whichever allocation fails, the trace reports it
    and the next one grows the lists afresh."""
    got = fields(fake("growth_fails", k))
    assert got == {"first": -2, "second": 0}


@pytest.mark.parametrize("tuning,steps", [((8, 1, 1, 0, 1), (2, 2, 2)), ((8, 1, 1, 0, 2), (2, 2, 2)), ((1, 1, 0, 0, 1), (1, 1, 1)),
                                          ((8, 2, 1, 0, 1), (1, 1, 1)), ((8, 1, 1, 1, 1), (1, 1, 1))])
def test_one_workgroup_on_a_compute_unit(fake, tuning, steps):
    """workgroups_per_cu 1 with split_modes 0: no two workgroups of a kernel fit a compute
    unit's 160 KB of LDS, and 256 are reckoned with when the images are cut into chunks.
    Any other tuning leaves the launches alone."""
    lines = [fields(x) for x in fake("batch_tuning", *tuning).splitlines()]
    assert lines[0] == {"rc": 0} and len(lines) == 4
    tables = 4096  # the kernels' own LDS
    for got, k in zip(lines[1:], steps):
        assert got["grid"] == -(-400 * 250 // (256 * k))
        if tuning[1] == 1 and tuning[3] == 0:
            assert 160 << 10 >= got["lds"] + tables > 80 << 10
        else:
            assert got["lds"] == 0


@pytest.mark.parametrize("dim,flags,tuning,resident", [
    (6, 1, (1, 8, 1, 0, 0), 2), (6, 1, (2, 8, 1, 0, 0), 3), (6, 1, (1, 8, 0, 0, 1), 3), (6, 9, (1, 8, 0, 0, 1), 2),
    (6, 9, (2, 8, 1, 0, 0), 2), (4, 1, (1, 8, 1, 0, 0), 4), (4, 1, (1, 8, 0, 0, 1), 5), (4, 9, (1, 8, 0, 0, 1), 4)])
def test_a_plain_launch_fills_the_chip_once(fake, dim, flags, tuning, resident):
    """As many workgroups as the kernel that is launched has resident on 256 compute
    units, whatever the tuning asks for: the max-accumulation search (flag 8) runs one
    lane a block on unpacked texels."""
    step = 256 // (2 if tuning[0] == 2 and not flags & 8 else 1)
    got = fields(fake("plain_grid", dim, step * (256 * resident + 100), flags, *tuning))
    assert got == {"rc": 0, "grid": 256 * resident}


@pytest.mark.parametrize("dim,blocks,candidates", [(6, 1000, 2), (4, 1000, 1), (4, 262144 + 1, 3), (4, 8 * 262144, 7),
                                                   (6, 131072 + 1, 4), (6, 1 << 20, 14)])
def test_the_autotuner_times_each_plan_once(fake, dim, blocks, candidates):
    """Tunings that cut a batch into the same chunks launch the same: one of them is
    timed, with the smallest blocks_per_lane.  (1, 2, 4 and 8 steps with and without
    the next step's loads, twice where 6x6 blocks may take two lanes.)"""
    got = fields(fake("autotune", dim, blocks))
    assert got["rc"] == 0 and got["launches"] == 4 * candidates
    if candidates <= 2:
        assert got["blocks_per_lane"] == 1 and got["prefetch"] == 0


def test_an_image_of_nearly_2_31_blocks_is_cut_to_its_end(fake):
    """The chunk that would begin after the last passes 2^31."""
    blocks = 4194303 * 512
    assert fields(fake("batch_items", 4194303, 512)) == {"rc": 0, "blocks": blocks, "items": -(-blocks // 1024)}
