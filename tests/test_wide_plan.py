"""Which form the launches of a wide prompt pass take (wide_plan in slai_amd/csrc/wide_plan.h), on the CPU."""
import ctypes as C
import os
import subprocess

import pytest

from test_gpu_prefill_share import DEALS

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LARGE, SMALL, SLIM4, SLIM8, SHARE = range(5)
WHOLE, SUMMED, READ = range(3)


class Plan:
    """form, ksplit; rounds, rest, mains, longest, whole: of the deal of tiles that the launch makes of its own row units."""

    def __init__(self, values):
        self.form, self.ksplit, self.rounds, self.rest, self.mains, self.longest, self.whole = values


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("plan") / "libwide_plan.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-I", os.path.join(ROOT, "slai_amd", "csrc"), os.path.join(HERE, "native", "wide_plan.cpp"), "-o", out])
    L = C.CDLL(out)

    def run(rows, ntokens, ncols, splits=WHOLE, gated=False, may_share=True):
        values = (C.c_uint32 * 7)()
        L.wide_plan_of((C.c_uint32 * len(rows))(*rows), len(rows), ntokens, (ncols + 255) // 256, splits, int(gated), int(may_share), values)
        return Plan(values)
    return run


@pytest.mark.parametrize("dim", [2048, 3584, 4096, 8192])
@pytest.mark.parametrize("gated", [False, True])
def test_what_is_shared_is_what_was_planned(plan, dim, gated):
    """A launch that shares tiles deals them out as the choice assumed: at most nine tenths of whole rounds, nobody with the rests of more than four tiles."""
    shared = 0
    for rows in list(range(dim, 5 * dim, 256)) + [4864, 17664, 11008, 18944, dim + 32, 2 * dim + 288]:
        for tokens in list(range(64, 1025, 48)) + [705, 801, 1024]:
            p = plan([rows], tokens, dim, WHOLE, gated)
            if p.form == SHARE:
                shared += 1
                assert p.ksplit == 1 and p.mains <= 4 and 10 * p.longest <= 9 * p.whole, (rows, tokens, p.rounds, p.rest, p.mains)
    assert shared > 50


@pytest.mark.parametrize("rows", [[4096], [1024, 1024, 4096], [11008]])
def test_nothing_is_shared_where_it_may_not(plan, rows):
    for tokens in range(9, 1025, 13):
        assert plan(rows, tokens, 4096, READ, may_share=False).form != SHARE


@pytest.mark.parametrize("deal", DEALS, ids=str)
def test_deals_of_the_gpu_tests(plan, deal):
    """The prompts that the GPU tests read reach the rounds and rests that they name."""
    _, hidden, n, rounds, rests = deal
    p = plan([hidden], n - 1, 2048, WHOLE, True)
    if rounds is None:
        assert p.form == LARGE and plan([2048, 2048, 2048], n - 1, 2048, READ).form == SHARE
    else:
        assert (p.form, p.rounds, p.mains) == (SHARE, rounds, rests)


@pytest.mark.parametrize("tokens,output,down", [(256, 1, 1), (257, 2, 4), (320, 2, 4), (321, 2, 2), (384, 2, 2), (385, 1, None)])
def test_ranges_of_the_gpu_tests(plan, tokens, output, down):
    """Slim launches of a model 2048 wide with 8704 hidden columns: the ranges of columns at the edges that test_gpu_prefill_ranges reads (with 8192, two)."""
    slim = (SLIM4, SLIM8)
    p = plan([2048], tokens, 2048, SUMMED)
    assert p.form in slim and p.ksplit == output
    for hidden, ranges in ((8704, down), (8192, down and min(down, 2))):
        p = plan([2048], tokens, hidden, SUMMED)
        assert (p.form in slim and p.ksplit == ranges) if ranges else p.ksplit != 2


# q/k/v of one format: large workgroups in two ranges fill the device once, three of 7B's 512-row units more tokens and they no longer do; ranges in two rounds
@pytest.mark.parametrize("rows,ncols,tokens,form,ranges", [([4096] * 3, 4096, 257, LARGE, 2), ([4096] * 3, 4096, 320, LARGE, 2), ([1024, 1024, 4096], 4096, 576, LARGE, 2), ([5120] * 3, 5120, 256, LARGE, 2),
                                                           ([4096] * 3, 4096, 353, SHARE, 1), ([512, 512, 3584], 3584, 801, SHARE, 1)])
def test_no_meeting_where_ranges_fill_the_device(plan, rows, ncols, tokens, form, ranges):
    p = plan(rows, tokens, ncols, READ)
    assert (p.form, p.ksplit) == (form, ranges)
