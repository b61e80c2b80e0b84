"""Conversion at the edges of its launches: super-windows about the segment
kernel's 4096 a step, counter arrays about the one-workgroup scan's 4096 and
16384, tiles about the number of compute units (wide workgroups up to it), and
rows about the 32- and 64-element windows; bit for bit against the oracle."""
import numpy as np
import pytest

from swtcf_checks import check_canonical
from test_gpu_convert import assert_same, convert_gpu

pytestmark = pytest.mark.gpu


def _check(oracle, dst, src, nd, ns, S):
    dst, src = np.asarray(dst, np.uint32), np.asarray(src, np.uint32)
    m, err, ng = convert_gpu(dst, src, nd, ns, S)
    ref = oracle.swtcf_convert(dst, src, nd, ns, S)
    assert err == 0 and ng == ref["numGroups"]
    assert_same(oracle, m, ref)
    return m


@pytest.mark.parametrize("order", ["rows", "shuffled"])
@pytest.mark.parametrize("windows", [1, 2, 4094, 4095, 4096, 4097, 8193])
def test_segments(gpu, oracle, windows, order):
    """S = 1: most of the super-windows are empty, the first and the last too."""
    nd, ns = 200, 8 * windows
    rng = np.random.default_rng(windows)
    key = np.sort(rng.choice(nd * ns, size=min(5000, nd * ns // 2), replace=False))
    if windows > 2:
        key = key[(key % ns >= 16) & (key % ns < ns - 16)]
    if order == "shuffled":
        rng.shuffle(key)
    _check(oracle, key // ns, key % ns, nd, ns, 1)


@pytest.mark.parametrize("windows", [14, 15, 16, 90, 91, 92])
def test_scan_steps(gpu, oracle, windows):
    """161 counters for each of 10 + windows tiles: 4025 and 4186, 16261 and 16422."""
    nd, ns = 700, 128 * windows
    key = np.sort(np.random.default_rng(windows).choice(nd * ns, size=40_960, replace=False))
    _check(oracle, key // ns, key % ns, nd, ns, 16)


@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_wide_workgroups(gpu, oracle, extra):
    import torch

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    nd, ns = 3000, 1000
    size = 4096 * cus + extra
    key = np.sort(np.random.default_rng(7).choice(nd * ns, size=size, replace=False))
    _check(oracle, key // ns, key % ns, nd, ns, 16)


@pytest.mark.parametrize("order", ["rows", "shuffled"])
@pytest.mark.parametrize("S", [8, 16, 32])
def test_row_lengths(gpu, oracle, S, order):
    """Rows of 1 to 8 S elements in one super-window, shuffled among short ones."""
    rng = np.random.default_rng(S)
    width, edges = 8 * S, []
    for r in range(600):
        length = [1, 7, 8, 9, 31, 32, 33, 34, 63, 64, 65, 66, width - 1, width, 2, 3][int(rng.integers(16))]
        cols = np.sort(rng.choice(width, size=min(length, width), replace=False)) + width * int(rng.integers(3))
        edges += [(r, int(c)) for c in cols]
    e = np.array(edges)
    if order == "shuffled":
        rng.shuffle(e)
    m = _check(oracle, e[:, 0], e[:, 1], 600, 3 * width, S)
    check_canonical(e[:, 0].astype(np.uint32), e[:, 1].astype(np.uint32), 3 * width, S, m)
