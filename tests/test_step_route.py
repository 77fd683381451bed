"""Which decode steps one workgroup per group makes, who sums the scores of others, and where arrivals are counted
(csrc/step_route.h, host code: compiled here by g++)."""
import ctypes
import os
import shutil
import subprocess

import pytest

import bench
from retrievalattention_amd._lib import DecodeStep

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _compiled(tmp_path_factory, function):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    where = tmp_path_factory.mktemp("route")
    (where / "route.cpp").write_text(f'#include "step_route.h"\nextern "C" int ask{function}\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "retrievalattention_amd", "csrc"), str(where / "route.cpp"), "-o",
                    str(where / "route.so")], check=True)
    return ctypes.CDLL(str(where / "route.so")).ask


@pytest.fixture(scope="module")
def is_one(tmp_path_factory):
    """What ri_decode_step asks: whether the kernel's form for one workgroup per group makes the step."""
    call = _compiled(tmp_path_factory, "(const ri_decode_step_t* s, int n) { return step_is_one(s, n); }")

    def one(static_len, zone=323, on_device=False, BG=129, gs=4, nc=512, np=9, es=118, page=8, max_pages=72, store=8192,
            sizes=True):
        step = DecodeStep(BG=BG, gs=gs, nc=nc, np=np, es=es, page=page, max_pages=max_pages, steady_stride=zone,
                          store_stride=store, static_len_dev=1 if on_device else None,
                          cluster_size_i32=1 if sizes else None, cluster_start=1 if sizes else None)
        return bool(call(ctypes.byref(step), static_len))
    return one


@pytest.mark.parametrize("gs", [1, 4, 5, 8])
def test_steps_that_one_workgroup_per_group_makes(is_one, gs):
    """Those of 129 to 256 groups, up to 512 clusters and eight heads, with up to 448 rows by the length at hand and the usual
    size of a cluster: the zone's end, pages and the store do not matter.  Up to 128 groups there are several workgroups."""
    assert not any(is_one(at, BG=BG, gs=gs) for at in (0, 69, 186) for BG in (1, 8, 64, 65, 128))
    for BG in (129, 200, 256):
        assert is_one(0, BG=BG, gs=gs) and is_one(186, BG=BG, gs=gs) and not is_one(187, BG=BG, gs=gs)
        assert is_one(186, BG=BG, gs=gs, zone=9000, on_device=True, max_pages=1 << 30, store=1 << 40)
        assert is_one(400, BG=BG, gs=gs, np=1, es=32) and not is_one(401, BG=BG, gs=gs, np=1, es=32)
        assert not is_one(98, BG=BG, gs=gs, nc=520) and not is_one(98, BG=BG, gs=gs, sizes=False)
    assert not is_one(98, gs=9) and not is_one(98, BG=257, gs=gs)


def test_who_sums_the_scores(tmp_path_factory):
    """Clusters up to which the selecting workgroups sum the scores themselves, by the heads and the groups.  More than eight heads
    have dist_kernel past 2048 clusters in any number of groups: eight clusters of sixteen heads to a thread are no form of
    the kernel's."""
    apart = _compiled(tmp_path_factory, "(int gs, int groups, int nc) { return step_sums_apart(gs, groups, nc); }")
    for gs in range(1, 17):
        for groups in (1, 8, 48, 49, 64, 65, 128, 129, 256, 4096):
            line = 2048 if gs > 8 or (gs > 6 and groups <= 64) else 4096
            assert not apart(gs, groups, line) and apart(gs, groups, line + 8), (gs, groups)
            for nc in (520, 2048, 2056, 4096, 4104, 16384):   # the launches that the benchmark names
                cfg = dict(B=groups, Hkv=1, gs=gs, nc=nc)
                assert bench.attending_launches(cfg) == ["dist_kernel"] * apart(gs, groups, nc) + ["select_attend_kernel"]


def test_arrival_counters_have_lines_of_their_own(tmp_path_factory):
    """Eight counters a group for the up to 128 groups that have more than one workgroup, in 4096 words: a line of 128 bytes each up
    to 16 groups, half a line up to 32."""
    pitch = _compiled(tmp_path_factory, "(int groups) { return attend_counter_pitch(groups); }")
    for groups in range(1, 129):
        assert groups * 8 * pitch(groups) <= 4096
        assert pitch(groups) >= (32 if groups <= 16 else 16 if groups <= 32 else 4)
