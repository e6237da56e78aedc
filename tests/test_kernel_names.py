"""The names under which the engine times its step kernels: all of them are
documented, and bench.py has each one's bytes."""
import os
import re

import pytest

import bench
from fwiflow import models

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _names():
    with open(os.path.join(ROOT, "fwiflow.jl_amd", "csrc", "engine.hip")) as f:
        return sorted(set(re.findall(r'launch\("(\w+)"', f.read())))


def test_every_timed_kernel_is_documented():
    assert len(_names()) >= 8
    for doc in ("include/fwiflow.h", "INTEGRATION.md"):
        with open(os.path.join(ROOT, doc)) as f:
            text = f.read()
        assert not [n for n in _names() if n not in text], doc


def test_bench_knows_every_timed_kernel():
    c = models.case_small()
    for n in _names():
        assert n in bench.KERNEL_BYTES or n in bench.KERNEL_PARTS, n
        assert bench.kernel_launch_bytes(n, c, 2.0) == 2 * bench.kernel_launch_bytes(n, c, 1.0) > 0
        assert (n in bench.BACKWARD) == (not n.endswith("_fwd")), n


def test_bytes_of_a_whole_step():
    """Every field once in and once out where two launches read the other half's
    again; the memory variables of both halves."""
    c = models.case_small()
    g = bench.geometry_counts(c)
    two = bench.kernel_launch_bytes("stress_fwd", c, 1.0) + bench.kernel_launch_bytes("vel_fwd", c, 1.0)
    assert two - bench.kernel_launch_bytes("step_fwd", c, 1.0) == pytest.approx(20 * g["update"])
    two = bench.kernel_launch_bytes("bwd_pair_a", c, 1.0) + bench.kernel_launch_bytes("bwd_pair_b", c, 1.0)
    one = bench.kernel_launch_bytes("step_bwd", c, 1.0)
    assert two - one == pytest.approx(20 * g["ring_rect"] + 20 * g["update"])
