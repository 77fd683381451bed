"""Which decode steps one workgroup per group makes, and where arrivals are counted (csrc/step_route.h, host code: compiled here by
g++)."""
import ctypes
import os
import shutil
import subprocess

import pytest

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


def _route(tmp_path_factory, name):
    call = _compiled(tmp_path_factory, f"(const ri_decode_step_t* s, int n) {{ return step_{name}(s, n); }}")

    def short(static_len, zone=323, on_device=False, BG=8, gs=4, nc=512, np=9, es=118, page=8, max_pages=72, store=8192,
              sizes=True):
        step = DecodeStep(BG=BG, gs=gs, nc=nc, np=np, es=es, page=page, max_pages=max_pages, steady_stride=zone,
                          store_stride=store, static_len_dev=1 if on_device else None,
                          cluster_size_i32=1 if sizes else None, cluster_start=1 if sizes else None)
        return bool(call(ctypes.byref(step), static_len))
    return short


@pytest.fixture(scope="module")
def is_short(tmp_path_factory):
    return _route(tmp_path_factory, "is_short")


@pytest.fixture(scope="module")
def is_alone(tmp_path_factory):
    return _route(tmp_path_factory, "is_alone")


def test_limits(is_short):
    assert is_short(98) and is_short(98, gs=8)
    assert not is_short(98, nc=520) and not is_short(98, gs=9) and not is_short(98, BG=257) and not is_short(98, sizes=False)
    assert is_short(186) and not is_short(187)                      # 448 rows
    assert is_short(186, BG=256) and not is_short(187, BG=256)


@pytest.mark.parametrize("gs", [1, 4, 5, 8])
def test_length_on_the_device_grows_to_the_zone(is_short, gs):
    """A captured step serves every length up to the zone's: only where the attention by itself would have one workgroup
    as well (384 rows of up to four heads, 192 of eight, more than 128 groups) does the length at hand decide."""
    alone = gs <= 4
    for zone in (69 + 256, 69 + 1024):
        assert is_short(69, zone=zone, on_device=True, gs=gs) == alone
        assert is_short(122, zone=zone, on_device=True, gs=gs) == alone
        assert not is_short(123, zone=zone, on_device=True, gs=gs)
        assert is_short(123, zone=zone, on_device=False, gs=gs)
        assert is_short(123, zone=zone, on_device=True, gs=gs, BG=129)
    assert is_short(123, zone=186, on_device=True, gs=gs) and not is_short(123, zone=187, on_device=True, gs=gs)
    assert is_short(69, zone=1093, on_device=True, gs=gs, nc=128, np=2, es=30)


@pytest.mark.parametrize("gs", [4, 8])
def test_clusters_may_hold_what_the_page_limit_lets_them(is_short, gs):
    at = 170   # 432 rows if the clusters have their usual size
    assert is_short(at, gs=gs, max_pages=76) and not is_short(at, gs=gs, max_pages=77)     # 896 rows at most
    assert is_short(at, gs=gs, max_pages=1 << 30, store=608) and not is_short(at, gs=gs, max_pages=1 << 30, store=609)
    assert is_short(at, gs=gs, max_pages=1 << 30, BG=129)
    assert is_short(98, gs=gs, max_pages=1 << 30) == (gs == 4)


def test_captured_steps_of_many_groups_keep_one_workgroup_for_longer(is_alone):
    """Which short steps one workgroup per group makes: by the rows at hand, and captured ones by the zone's too."""
    for BG, line, end in ((1, 336, 420), (15, 336, 420), (16, 336, 512), (64, 336, 512), (65, 640, 800), (128, 640, 800)):
        assert is_alone(line - 90, BG=BG, np=4, es=26) and not is_alone(line - 89, BG=BG, np=4, es=26)
        assert is_alone(69, zone=end - 90, on_device=True, BG=BG, np=4, es=26)
        assert not is_alone(69, zone=end - 89, on_device=True, BG=BG, np=4, es=26)
        assert not is_alone(line - 89, zone=end - 90, on_device=True, BG=BG, np=4, es=26)
    assert is_alone(5000, BG=129)


def test_who_sums_the_scores(tmp_path_factory):
    """Clusters up to which the selecting workgroups sum the scores themselves, by the heads and the groups.  More than eight heads
    have dist_kernel past 2048 clusters in any number of groups: eight clusters of sixteen heads to a thread are no form of
    the kernel's."""
    apart = _compiled(tmp_path_factory, "(int gs, int groups, int nc) { return step_sums_apart(gs, groups, nc); }")
    for gs in range(1, 17):
        for groups in (1, 8, 48, 49, 64, 65, 128, 129, 256, 4096):
            line = 2048 if gs > 8 or (gs > 6 and groups <= 64) else 4096
            assert not apart(gs, groups, line) and apart(gs, groups, line + 8), (gs, groups)


def test_arrival_counters_have_lines_of_their_own(tmp_path_factory):
    """Eight counters a group for the up to 128 groups that have more than one workgroup, in 4096 words: a line of 128 bytes each up
    to 16 groups, half a line up to 32."""
    pitch = _compiled(tmp_path_factory, "(int groups) { return attend_counter_pitch(groups); }")
    for groups in range(1, 129):
        assert groups * 8 * pitch(groups) <= 4096
        assert pitch(groups) >= (32 if groups <= 16 else 16 if groups <= 32 else 4)
