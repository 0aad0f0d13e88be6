"""The prefill tiles (mxa_ptile.hip, mxa_iq4.hip) at the places where they can go wrong, against the oracle bit for
bit: remainders of the 32-row tiles on both sides, one block per row, rows whose blocks start at
2-byte boundaries, weights that start 4 bytes past a 16-byte boundary, each choice of workgroup, and
the largest integer sums of each type."""

import numpy as np
import pytest
import torch

from matricxon_amd import synthetic as S
from oracle import dequant as D
from tests.test_gpu_kernels import assert_within_tolerance, bits, dev, host

pytestmark = pytest.mark.gpu

TYPES = [D.Q4_K, D.Q6_K, D.Q8_0]


def check(gpu, oracle, t, w, x, n, k, shift=0):
    buf = torch.zeros(w.size + 64, dtype=torch.uint8, device="cuda")
    wd = buf[shift:shift + w.size].view(n, -1)
    wd.copy_(dev(w))
    assert wd.data_ptr() % 16 == shift
    got = host(gpu.matmul(t, wd, dev(x), n, k))
    rows = np.unique(np.concatenate([np.arange(min(n, 200)), np.arange(max(0, n - 200), n), np.arange(0, n, 37)]))
    want = oracle.gemm(t, w[rows], x, len(rows), k)
    assert np.array_equal(bits(got[:, rows]), bits(want))


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("n,k,m", [
    (1, 256, 65), (31, 256, 96), (33, 512, 97), (64, 768, 128), (129, 1280, 129), (257, 2816, 200),
    (1, 256, 17), (33, 512, 32), (70, 768, 33), (129, 1280, 40), (32, 2816, 64),  # a workgroup per tile
    (1000, 512, 1100),   # two waves, one tile
    (8200, 256, 400),    # four waves, two tiles
    (16500, 512, 300),   # eight waves, two tiles
])
def test_prefill_tiles_match_oracle(gpu, oracle, t, n, k, m) -> None:
    w = S.packed_weight(t, n, k, seed=n + k)
    check(gpu, oracle, t, w, S.activations(m, k, seed=m), n, k)


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("shift", [4, 8, 12])
@pytest.mark.parametrize("m", [70, 1100])
def test_prefill_weight_alignment(gpu, oracle, t, shift, m) -> None:
    n = 70 if m == 70 else 1000  # a workgroup per tile, waves of tiles
    w = S.packed_weight(t, n, 1280, seed=9)
    check(gpu, oracle, t, w, S.activations(m, 1280, seed=10), n, 1280, shift)


@pytest.mark.parametrize("t,q6_scale", [(D.Q4_K, 0), (D.Q6_K, -128), (D.Q6_K, -4), (D.Q8_0, 0)])
@pytest.mark.parametrize("sign", [1, -1])
def test_prefill_largest_sums(gpu, oracle, t, q6_scale, sign) -> None:
    """Every code, scale and activation at its largest magnitude, all products of one sign: the sums
    that the float conversion of the integer planes has to hold. Q6_K's value -32 times a scale of -128 is
    16 in the high plane and 0 in the low one, times -4 it is 1 and -128, that plane's largest."""
    n, k, m = 40, 1536, 80
    w = S.packed_weight(t, n, k, seed=1).reshape(n, -1)
    if t == D.Q4_K:
        b = w.reshape(-1, 144)
        b[:, 4:16] = 0xFF  # every scale and min 63
        b[:, 16:] = 0xFF  # every code 15
    elif t == D.Q6_K:
        b = w.reshape(-1, 210)
        b[:, :192] = 0  # every code 0, the value -32
        b[:, 192:208] = q6_scale & 0xFF
    else:
        w.reshape(-1, 34)[:, 2:] = 0x80  # every quant -128
    x = np.full((m, k), 127.0 * sign, dtype=np.float32)
    x[1::2] *= -1
    x[2::5, 3::7] *= -0.5
    check(gpu, oracle, t, w, x, n, k)


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("counts", [
    [0, 1, 31, 32, 33, 2],
    [5, 1, 31, 32, 33, 40],  # 32-row chunks (past 20 rows an expert on average)
    [0, 1, 64, 65, 33, 0, 129],  # 64-row chunks, the last one of some experts with one tile's rows
])
def test_grouped_prefill_tiles_match_oracle(gpu, oracle, t, counts) -> None:
    n, k, e = 300, 1280, len(counts)
    w = np.stack([S.packed_weight(t, n, k, seed=70 + i) for i in range(e)])
    x = S.activations(sum(counts), k, seed=71)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    got = host(gpu.matmul_moe(t, dev(w), dev(x), dev(off), max(counts), n, k))
    for i, c in enumerate(counts):
        if c:
            rows = slice(off[i], off[i + 1])
            assert np.array_equal(bits(got[rows]), bits(oracle.gemm(t, w[i], x[rows], n, k)))


@pytest.mark.parametrize("n,k,m,shift", [
    (1, 256, 17, 0), (33, 512, 33, 0), (70, 768, 64, 4), (70, 1280, 70, 8), (129, 768, 96, 12),
    (8200, 256, 400, 0),  # four waves, two tiles
    (16500, 512, 300, 0),  # eight waves, two tiles
])
def test_iq4_prefill_tiles_match_oracle(gpu, oracle, n, k, m, shift) -> None:
    """IQ4_XS on the bf16 tiles: rows whose blocks start at 8-byte multiples, weights at every dword
    of a 16-byte unit, remainders on both sides; within the type's tolerance."""
    w = S.packed_weight(D.IQ4_XS, n, k, seed=n + k)
    x = S.activations(m, k, seed=m)
    buf = torch.zeros(w.size + 64, dtype=torch.uint8, device="cuda")
    wd = buf[shift:shift + w.size].view(n, -1)
    wd.copy_(dev(w))
    got = host(gpu.matmul(D.IQ4_XS, wd, dev(x), n, k))
    rows = np.unique(np.concatenate([np.arange(min(n, 200)), np.arange(max(0, n - 200), n)]))
    assert_within_tolerance(got[:, rows], oracle.gemm(D.IQ4_XS, w[rows], x, len(rows), k))


@pytest.mark.parametrize("t", TYPES)
def test_grouped_prefill_expert_strides(gpu, oracle, t) -> None:
    """Experts 4 bytes further apart than their rows take: their blocks start at every dword of a 16-byte
    unit, the last expert's at the end of the allocation."""
    n, k, e = 300, 512, 5
    rb = gpu.row_bytes(t, k)
    stride = -(-n * rb // 16) * 16 + 4
    w = np.stack([S.packed_weight(t, n, k, seed=80 + i) for i in range(e)])
    flat = np.zeros((e - 1) * stride + n * rb, dtype=np.uint8)
    for i in range(e):
        flat[i * stride:i * stride + n * rb] = w[i].reshape(-1)
    counts = [33, 40, 1, 0, 64]
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    x = S.activations(sum(counts), k, seed=81)
    wd, xd, od = dev(flat), dev(x), dev(off)
    ws = torch.empty(gpu.workspace_bytes(t, sum(counts), k), dtype=torch.uint8, device="cuda")
    y = torch.empty((sum(counts), n), dtype=torch.float32, device="cuda")
    st = gpu._lib.mxa_gemm_moe(t, wd.data_ptr(), stride, e, xd.data_ptr(), od.data_ptr(), sum(counts), 64,
                               y.data_ptr(), n, k, ws.data_ptr(), ws.numel(),
                               torch.cuda.current_stream().cuda_stream)
    assert st == 0
    got = host(y)
    for i, c in enumerate(counts):
        if c:
            rows = slice(off[i], off[i + 1])
            assert np.array_equal(bits(got[rows]), bits(oracle.gemm(t, w[i], x[rows], n, k)))


@pytest.mark.parametrize("t", [D.Q8_0, D.IQ4_XS])
def test_prefill_rows_past_4_gib_apart(gpu, t) -> None:
    """Rows so long that a wave's last ones start more than 4 GiB past its first: they equal the same rows of
    a matrix of two, of which neither does."""
    k = 256 * (540_000 if t == D.Q8_0 else 1_080_000)
    rb, n, m = gpu.row_bytes(t, k), 32, 17
    assert 30 * rb > 1 << 32
    g = torch.Generator(device="cuda").manual_seed(5)
    w = torch.randint(0, 256, (n, rb), dtype=torch.uint8, device="cuda", generator=g)
    blocks = w.view(-1, 34 if t == D.Q8_0 else 136)
    blocks[:, 0] = torch.randint(0, 256, (blocks.shape[0],), dtype=torch.uint8, device="cuda", generator=g)
    blocks[:, 1] = 0x0C  # scales of 2^-12 to 2^-11
    x = torch.randn((m, k), device="cuda", generator=g)
    got = gpu.matmul(t, w, x, n, k)
    for r in (0, 30) if t == D.Q8_0 else (30,):
        assert torch.equal(got[:, r:r + 2].view(torch.int32), gpu.matmul(t, w[r:r + 2], x, 2, k).view(torch.int32))
    assert got.isfinite().all() and got[:, 31].count_nonzero() == m


def test_prefill_more_rows_than_a_grid_takes(gpu, oracle) -> None:
    """More than 65535 groups of 64 activation rows, the most of one launch's grid."""
    n, k, m = 3, 256, 65535 * 64 + 70
    w = S.packed_weight(D.Q4_K, n, k, seed=2)
    x = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(6))
    got = gpu.matmul(D.Q4_K, dev(w), x, n, k)
    for rows in (slice(0, 40), slice(m - 130, m)):
        assert np.array_equal(bits(host(got[rows])), bits(oracle.gemm(D.Q4_K, w, host(x[rows]), n, k)))


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("m", [4, 9, 16])
@pytest.mark.parametrize("shift", [0, 4])
def test_wide_matrices_of_few_rows(gpu, oracle, t, m, shift) -> None:
    """4 to 16 activation rows and 32768 weight rows or more, also where the weights' place or the length of a
    row keeps the batched-decode kernels from taking them."""
    n, k = 32800, 256 * 18
    w = S.packed_weight(t, 64, k, seed=3)
    w = np.ascontiguousarray(np.tile(w, (n // 64 + 1, 1))[:n])
    check(gpu, oracle, t, w, S.activations(m, k, seed=m), n, k, shift)
