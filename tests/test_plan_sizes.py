"""The workspace of a context against what its calls write, for every size of both (CPU).

The rules of a call change with its tokens, so the largest need of a context of t_max tokens
is not always that of its largest call: 1279 tokens write more router partials than 1280.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG

SHIM = """
#include "qe_plan.h"
extern "C" {
long splits(int T) { return qe_router_splits(T); }
long rpart_rows(int t_max) { return (long)qe_rpart_rows(t_max); }
long item_pairs(int T, int used) { return used <= qe_item32_experts(T) ? 32 : QE_MFMA_MC; }
long max_items(int T) { return qe_max_items(T); }
long max_items_upto(int t_max) { return qe_max_items_upto(t_max); }
}
"""
T_END = 8300


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-std=c++17", "-I", os.path.join(PKG, "csrc"), str(d / "shim.cpp"), "-o",
                    str(d / "shim.so")], check=True)
    lib = ctypes.CDLL(str(d / "shim.so"))
    for f in ("splits", "rpart_rows", "item_pairs", "max_items", "max_items_upto"):
        getattr(lib, f).restype = ctypes.c_long
    return lib


def test_router_partials_of_every_call_fit(plan):
    ts = list(range(1, T_END)) + [16384, 65535, 65536]
    need = np.maximum.accumulate([T * plan.splits(T) for T in ts])
    have = np.array([plan.rpart_rows(T) for T in ts])
    assert np.all(have >= need)
    assert np.array_equal(have, need)  # and no larger than its largest call


def test_items_of_every_call_fit(plan):
    ts = list(range(1, T_END)) + [16384, 65535, 65536]
    need = np.maximum.accumulate([plan.max_items(T) for T in ts])
    have = np.array([plan.max_items_upto(T) for T in ts])
    assert np.array_equal(have, need)


def test_items_bound_covers_any_routing(plan):
    """Items of `used` experts: each has at least one pair and at most T, in items of item_pairs."""
    rng = np.random.default_rng(3)
    for T in (9, 16, 31, 100, 223, 224, 255, 256, 1000):
        np_ = T * 8
        for used in (8, 9, 32, 111, 112, 113, 200, 255, 256):
            if used > np_:
                continue
            tc = plan.item_pairs(T, used)
            for fill in ("even", "one item and one pair", "random"):
                if fill == "even":
                    c = np.full(used, np_ // used)
                    c[: np_ % used] += 1
                elif fill == "random":
                    c = 1 + rng.multinomial(np_ - used, rng.dirichlet(np.full(used, 0.3)))
                else:  # as many experts as go one pair past a whole item
                    c = np.ones(used, int)
                    left = np_ - used
                    for e in range(used):
                        k = min(left // tc * tc, (T - 1) // tc * tc)
                        c[e] += k
                        left -= k
                c = np.minimum(c, T)
                assert int(np.sum(-(-c // tc))) <= plan.max_items(T), (T, used, fill)
