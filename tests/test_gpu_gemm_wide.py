"""GPU: the wide GEMM (prompt-sized M, bits <= 4) against the small-M kernels.

The wide kernel computes the same MFMA sequence and adds the same K partitions
in the same order as the kernels that run at 5 <= M <= 64, which the oracle
covers: every row of a wide launch must equal the same row of a 64-row launch
bit for bit.  The shapes walk its edges: a last row chunk of 1, 33, 255 and 256
rows, a ragged N (a partial tile and a partial column block), an N that is no
multiple of 8 (stored column by column), K tails inside a k-block (at 1 bit too,
where weights past K decode to a level), an odd number of k-blocks, one k-block,
one to eight K partitions but six (folded in registers), groups of 32 to 256,
bits 1 to 4, fp16, grouped members whose boundary falls inside a column block,
padded activation and output rows.  Each case asserts that the wide kernel is
planned.
"""
from __future__ import annotations

import pytest
import torch

from cubic_serve_amd import _native, linear, quantization as qz
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
    (32768, 1, 120, 128, 4, 2048, True),    # less than one k-block
    (32768, 1, 1016, 128, 3, 400, False),   # split 1, eight k-blocks, K tail
    (40000, 1, 584, 128, 4, 700, True),     # split 1, odd k-blocks, K tail
    (6144, 1, 1080, 128, 1, 1100, False),   # 1 bit with a K tail: levels past K
    (8192, 1, 616, 64, 1, 1281, False),     # the same with two groups per k-block
    (1696, 1, 1280, 32, 2, 936, False),     # split 5
    (2704, 1, 1768, 64, 4, 800, False),     # split 7, K tail
    (3072, 1, 3032, 128, 4, 1100, False),   # split 8, K tail
    (2048, 1, 2048, 128, 2, 1100, True),    # split 8 of two k-blocks
    (5003, 1, 2048, 128, 4, 1281, False),   # rows of 5003: no 16-byte segments
    (2067, 1, 1288, 32, 1, 1100, False),    # the same, 1 bit, quarters past K
]


def prepared_members(n, members, k, group, bits, dt):
    parts = [linear.prepare_matrix(random_matrix(n, k, bits, group, qz.FMT_F32, seed=n + k + i).to(DEV), DEV, dt)
             for i in range(members)]
    return parts[0] if members == 1 else linear.PreparedCubic(
        torch.cat([p.codes for p in parts]), torch.cat([p.meta for p in parts]), n * members, k, bits, group, dt)


def padded_rows(m, k, dt):
    """Activations in rows of k + 40 whose padding is NaN: never read into a sum."""
    x = torch.full((m, k + 40), float("nan"), dtype=dt, device=DEV)
    x[:, :k] = torch.randn((m, k), generator=torch.Generator(device=DEV).manual_seed(m), device=DEV).to(dt)
    return x[:, :k]


def test_wide_shapes_cover_the_partitions():
    splits = {launch_plan(m, members, n, k, bits, group)[2] for n, members, k, group, bits, m, _ in SHAPES}
    assert splits == {1, 2, 3, 4, 5, 7, 8}


@pytest.mark.parametrize("n,members,k,group,bits,m,f16", SHAPES)
def test_wide_rows_equal_small_launches(n, members, k, group, bits, m, f16):
    print(f"wide n={n}x{members} k={k} g={group} bits={bits} m={m} f16={f16}", flush=True)
    assert launch_plan(m, members, n, k, bits, group)[1] == WIDE
    dt = torch.float16 if f16 else torch.bfloat16
    prepared, x = prepared_members(n, members, k, group, bits, dt), padded_rows(m, k, dt)

    def run(rows):
        ys = [torch.full((rows.shape[0], n), float("nan"), dtype=dt, device=DEV) for _ in range(members)]
        linear.bind_prepared(rows, prepared, ys, (n,) * members).launch()
        return ys

    got = run(x)
    for r in range(0, m, 64):
        for a, b in zip(got, run(x[r:r + 64] if m - r > 4 else x[m - 64:])):
            rows = slice(r, min(m, r + 64)) if m - r > 4 else slice(m - 64, m)
            assert torch.equal(a[rows].view(torch.int16), b.view(torch.int16)), r


@pytest.mark.parametrize("n,members,k,bits,m,pads", [
    (6144, 2, 2048, 4, 257, (8, 3)),     # one member in 16-byte segments, one column by column
    (4112, 3, 1152, 3, 1057, (0, 5, 1)), # boundaries inside a column block
    (5003, 1, 2048, 2, 1281, (5,)),      # aligned rows, a ragged last segment
])
def test_padded_output_rows(n, members, k, bits, m, pads):
    """Output rows of n + pad: equal to contiguous ones, the padding and the
    rows past M untouched."""
    print(f"padded n={n}x{members} k={k} bits={bits} m={m} pads={pads}", flush=True)
    assert launch_plan(m, members, n, k, bits, 128)[:2] == (0, WIDE)
    dt = torch.bfloat16
    prepared, x = prepared_members(n, members, k, 128, bits, dt), padded_rows(m, k, dt)
    want = [torch.empty((m, n), dtype=dt, device=DEV) for _ in range(members)]
    linear.bind_prepared(x, prepared, want, (n,) * members).launch()
    ys = [torch.full((m + 1, n + pad), float("nan"), dtype=dt, device=DEV) for pad in pads]
    ptrs = (_native.ctypes.c_void_p * members)(*(y.data_ptr() for y in ys))
    ldys = (_native.ctypes.c_int64 * members)(*(y.stride(0) for y in ys))
    _native.call("cubic_gemm_group", x.data_ptr(), x.stride(0), prepared.codes.data_ptr(), prepared.meta.data_ptr(),
                 m, members, n, k, bits, 128, 0, ptrs, ldys, None, 0, _native.stream_of(torch.device(DEV)))
    for y, w in zip(ys, want):
        assert torch.equal(y[:m, :n].view(torch.int16), w.view(torch.int16))
        assert torch.isnan(y[:m, n:].float()).all() and torch.isnan(y[m].float()).all()


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
    prepared = prepared_members(n, members, k, 128, 4, torch.bfloat16)
    x = torch.randn((m, k), generator=torch.Generator(device=DEV).manual_seed(1), device=DEV).to(torch.bfloat16)
    far = torch.empty(extent // 2, dtype=torch.bfloat16, device=DEV).as_strided((m, k), (stride, 1))
    far.copy_(x)
    got = []
    for rows in (x, far):
        ys = [torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(members)]
        linear.bind_prepared(rows, prepared, ys, (n,) * members).launch()
        got.append(torch.stack(ys).view(torch.int16))
    assert torch.equal(got[0], got[1])
