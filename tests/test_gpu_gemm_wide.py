"""GPU: the wide GEMM (prompt-sized M, bits <= 4) against the small-M kernels.

The wide kernel computes the same MFMA sequence and adds the same K partitions
in the same order as the kernels that run at M <= 64, which the oracle covers:
every row of a wide launch must equal the same row of a 64-row launch bit for
bit.  The shapes walk its edges: a last row chunk of 1, 33, 255 and 256 rows,
a ragged N (a partial tile and a partial column block), K tails inside a
k-block, an odd number of k-blocks, one k-block, K partitions of one to eight
(folded in registers), groups of 32 to 256, bits 1 to 4, fp16, grouped members
whose boundary falls inside a column block, padded activation and output rows.
"""
from __future__ import annotations

import pytest
import torch

from cubic_serve_amd import linear, quantization as qz
from test_gemm_plan_host import TILES, WIDE, launch_plan
from test_gpu_gemm import random_matrix

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# n per member, members, k, group, bits, m, fp16
SHAPES = [
    (6144, 1, 2048, 128, 4, 1025, False),   # split 2 or more, last chunk of one row
    (6120, 1, 1096, 128, 4, 1535, False),   # ragged N, K tail of 72, odd k-blocks, 255 rows
    (4112, 2, 1152, 128, 3, 1313, True),    # member boundary inside a column block, 33 rows
    (8192, 1, 1024, 256, 2, 1024, False),   # two k-blocks per group, whole chunks
    (8200, 1, 1000, 32, 4, 1100, False),    # a group per quarter, quarters past K
    (8192, 1, 640, 64, 1, 1281, True),      # two groups per k-block, 5 k-blocks
    (32768, 1, 128, 128, 4, 600, False),    # one k-block
]


@pytest.mark.parametrize("n,members,k,group,bits,m,f16", SHAPES)
def test_wide_rows_equal_small_launches(n, members, k, group, bits, m, f16):
    print(f"wide n={n}x{members} k={k} g={group} bits={bits} m={m} f16={f16}", flush=True)
    dt = torch.float16 if f16 else torch.bfloat16
    parts = [linear.prepare_matrix(random_matrix(n, k, bits, group, qz.FMT_F32, seed=n + k + i).to(DEV), DEV, dt)
             for i in range(members)]
    prepared = parts[0] if members == 1 else linear.PreparedCubic(
        torch.cat([p.codes for p in parts]), torch.cat([p.meta for p in parts]), n * members, k, bits, group, dt)
    gen = torch.Generator(device=DEV).manual_seed(m)
    x = torch.zeros((m, k + 40), dtype=dt, device=DEV)  # padded rows
    x[:, :k] = torch.randn((m, k), generator=gen, device=DEV).to(dt)
    x[:, k:] = float("nan")  # never read into a sum
    x = x[:, :k]

    def run(rows):
        ys = [torch.full((rows.shape[0], n), float("nan"), dtype=dt, device=DEV) for _ in range(members)]
        linear.bind_prepared(rows, prepared, ys, (n,) * members).launch()
        return ys

    got = run(x)
    for r in range(0, m, 64):
        for a, b in zip(got, run(x[r:r + 64] if m - r > 4 else x[m - 64:])):
            rows = slice(r, min(m, r + 64)) if m - r > 4 else slice(m - 64, m)
            assert torch.equal(a[rows].view(torch.int16), b.view(torch.int16)), r


def test_wide_is_chosen_where_the_sizes_say():
    """These shapes take the wide kernel: no split-K workspace where the
    64-row launch of the same weight has one."""
    for n, k, m in ((6144, 4096, 2048), (4096, 12288, 2048), (6144, 2048, 1025), (8192, 1024, 1024)):
        assert linear.gemm_workspace_bytes(64, (n,), k, 4) > 0
        assert linear.gemm_workspace_bytes(m, (n,), k, 4) == 0, (n, k, m)
    # 128 wide tiles for 256 CUs and K partitions to use the rest
    assert linear.gemm_workspace_bytes(1024, (4096,), 12288, 4) > 0


def test_row_stride_past_the_wide_kernel_equals_contiguous_rows():
    """A row stride of 2^28 elements, past the wide kernel's offsets: the
    binding holds the MFMA-tile kernel's K partitions, and the rows equal the
    contiguous launch bit for bit."""
    n, members, k, m, stride = 6144, 2, 2048, 129, 1 << 28
    extent = ((m - 1) * stride + k) * 2
    if torch.cuda.mem_get_info()[0] < extent + (4 << 30):
        pytest.skip(f"needs {extent >> 30} GiB of free device memory")
    print(f"row stride {stride} m={m}", flush=True)
    assert launch_plan(m, members, n, k, 4, 128)[1] == WIDE
    need, kernel, split = launch_plan(m, members, n, k, 4, 128, stride)
    assert kernel == TILES and split > 1 and need > 0
    parts = [linear.prepare_matrix(random_matrix(n, k, 4, 128, qz.FMT_F32, seed=i).to(DEV), DEV) for i in range(members)]
    prepared = linear.PreparedCubic(torch.cat([p.codes for p in parts]), torch.cat([p.meta for p in parts]),
                                    n * members, k, 4, 128, torch.bfloat16)
    x = torch.randn((m, k), generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(torch.bfloat16)
    far = torch.empty(extent // 2, dtype=torch.bfloat16, device=DEV).as_strided((m, k), (stride, 1))
    far.copy_(x)
    got = []
    for rows in (x, far):
        ys = [torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(members)]
        linear.bind_prepared(rows, prepared, ys, (n,) * members).launch()
        got.append(torch.stack(ys).view(torch.int16))
    assert torch.equal(got[0], got[1])
