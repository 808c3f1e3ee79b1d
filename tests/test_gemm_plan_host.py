"""CPU: the GEMM's host planning (no launch is reached): the workspace size
query, what one launch requires, and the kernel it takes."""
from __future__ import annotations

import random

import pytest

from cubic_serve_amd import _native, linear

ROWS, PANEL, TILES, WIDE = range(4)  # CUBIC_GEMM_*


def launch_plan(m, members, n, k, bits, group, ldx=None):
    """(workspace bytes, kernel, K partitions) of one launch."""
    kernel, split = _native.ctypes.c_int(), _native.ctypes.c_int()
    need = _native.lib().cubic_gemm_launch_plan(m, members, n, k, bits, group, k if ldx is None else ldx,
                                                _native.ctypes.byref(kernel), _native.ctypes.byref(split))
    return need, kernel.value, split.value


@pytest.mark.parametrize("n,k,members,bits", [(4096, 12288, 1, 4), (6144, 4096, 1, 4), (12288, 4096, 2, 4),
                                              (12288, 4096, 2, 3), (4096, 4096, 1, 8), (2048, 1024, 4, 1)])
def test_workspace_covers_every_smaller_m(n, k, members, bits):
    """One workspace sized at the largest m serves every smaller one, at any
    group width and row stride."""
    size = _native.lib().cubic_gemm_group_workspace_bytes
    sizes = [size(m, members, n, k, bits) for m in range(1, 2400)]
    assert all(a <= b for a, b in zip(sizes, sizes[1:]))
    for m in (1, 4, 5, 16, 33, 64, 65, 128, 129, 500, 1024, 2048, 2399):
        for group in (32, 64, 128, 256):
            for ldx in (k, 1 << 24, 1 << 28):
                assert launch_plan(m, members, n, k, bits, group, ldx)[0] <= sizes[m - 1]


def test_random_launches_need_no_more_than_the_query():
    rng = random.Random(7)
    lib = _native.lib()
    for _ in range(20000):
        n, k = 16 * round(2 ** rng.uniform(0, 12)), 8 * round(2 ** rng.uniform(1, 12))
        m, members, bits = round(2 ** rng.uniform(0, 13)), rng.randint(1, 8), rng.randint(1, 8)
        size = lib.cubic_gemm_group_workspace_bytes(m, members, n, k, bits)
        small = rng.randint(1, m)
        assert lib.cubic_gemm_group_workspace_bytes(small, members, n, k, bits) <= size
        need = launch_plan(small, members, n, k, bits, rng.choice((32, 64, 96, 128, 256)),
                           rng.choice((k, 1 << 25, 1 << 28)))[0]
        assert 0 <= need <= size, (m, small, members, n, k, bits)


@pytest.mark.parametrize("m,stride,kernel", [(2048, 4096, WIDE), (2048, 1 << 28, TILES),
                                             (64, 4096, PANEL), (64, 1 << 25, TILES), (8, 1 << 27, TILES)])
def test_launch_takes_the_workspace_of_its_plan(m, stride, kernel):
    """The launch asks for exactly the plan's bytes, and row strides past the
    column-panel and wide kernels' offsets move it to the MFMA-tile kernel."""
    n, k = 6144, 4096
    need, got, split = launch_plan(m, 1, n, k, 4, 128, stride)
    assert got == kernel and split > 1
    assert need <= _native.lib().cubic_gemm_workspace_bytes(m, n, k, 4)
    assert (need == 0) == (kernel == WIDE)
    if need:  # one byte short: refused before anything is enqueued
        with pytest.raises(ValueError, match=f"workspace {need - 1} < {need} bytes"):
            _native.call("cubic_gemm", 16, stride, 16, 16, m, n, k, 4, 128, 0, 16, n, 16, need - 1, None)


def test_bound_launches_allocate_what_they_need():
    assert linear.gemm_workspace_bytes(2048, (6144,), 4096, 4) == 0
    assert linear._launch_workspace_bytes(2048, (6144,), 4096, 4, 128, 1 << 28) > 0
    # members of different widths run one after another
    assert linear.gemm_workspace_bytes(64, (6144, 4096), 4096, 4) == max(
        linear.gemm_workspace_bytes(64, (n,), 4096, 4) for n in (6144, 4096))
    with pytest.raises(ValueError, match="limited to two"):
        linear.gemm_workspace_bytes(64, (64, 128, 256), 4096, 4)
    assert launch_plan(64, 9, 6144, 4096, 4, 128)[0] == -1
    assert launch_plan(64, 1, 6144, 4096, 9, 128)[0] == -1
    assert launch_plan(64, 1, 6144, 4096, 4, 100)[0] == -1


# n per member, members, k, bits, group, m, us on the MFMA-tile kernel, us on the wide kernel
MEASURED = [
    (1616, 1, 768, 2, 64, 560, 12.2, 19.9), (3224, 1, 768, 2, 64, 281, 12.8, 19.5),
    (18768, 1, 1024, 1, 64, 899, 50.5, 66.2), (21480, 1, 2272, 4, 32, 428, 69.1, 83.1),
    (32768, 1, 1024, 4, 128, 384, 39.6, 44.2), (32768, 1, 1024, 4, 128, 777, 80.3, 87.2),
    (34928, 1, 2816, 4, 32, 246, 86.9, 98.7), (20248, 1, 1248, 2, 32, 1055, 84.4, 97.2),
    (10240, 1, 8192, 4, 128, 2048, 365.6, 388.2), (28672, 2, 8192, 4, 128, 777, 885.0, 935.5),
    (29152, 1, 6912, 4, 128, 1288, 630.5, 670.6), (34224, 1, 12736, 4, 128, 2055, 1844.4, 1992.1),
    (14896, 1, 20224, 4, 256, 2135, 1421.7, 1514.2),
    (4096, 1, 12288, 4, 128, 1024, 148.1, 176.0), (4096, 1, 12288, 4, 128, 512, 86.8, 162.1),
    (12288, 2, 4096, 4, 128, 300, 101.9, 121.7), (6144, 1, 4096, 4, 128, 384, 45.0, 59.4),
    (12288, 2, 4096, 4, 128, 256, 72.8, 61.4), (12288, 2, 4096, 4, 128, 2048, 478.1, 433.0),
    (6144, 1, 4096, 4, 128, 1024, 87.5, 62.7), (4096, 1, 12288, 4, 128, 2048, 272.4, 206.4),
    (6144, 2, 2048, 4, 128, 512, 64.8, 36.5), (3072, 1, 3072, 4, 128, 2048, 136.8, 53.5),
    (4096, 1, 4096, 3, 128, 1536, 87.0, 62.3), (12288, 2, 4096, 4, 32, 777, 298.5, 231.7),
    (12288, 2, 4096, 2, 32, 512, 168.4, 135.7), (32768, 1, 128, 4, 128, 2048, 85.8, 75.0),
    (151936, 1, 4096, 4, 32, 200, 468.5, 371.4), (151936, 1, 4096, 3, 128, 129, 302.3, 292.1),
]


@pytest.mark.parametrize("n,members,k,bits,group,m,tiles,wide", MEASURED)
def test_plan_takes_the_kernel_that_measured_faster(n, members, k, bits, group, m, tiles, wide):
    """Both kernels' times on an MI355X, 3 to 160% apart: the first thirteen
    were planned wide by a model without a tile's start and the last round's
    share."""
    assert launch_plan(m, members, n, k, bits, group)[1] == (WIDE if wide < tiles else TILES)
