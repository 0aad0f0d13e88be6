"""What the packed modules refuse and accept on the host, before any launch. Host-only: the library's
calls are replaced by stubs of the same results' shapes, CPU tensors stand in for the device's."""

import pytest
import torch

from matricxon_amd.device_packed import DevicePackedLinear
from matricxon_amd.fused_ops import HANDOFF
from matricxon_amd.gemm import HipGemm

K, N, Q4_K, ROW_BYTES = 256, 8, 12, 144


class _Stub:
    """HipGemm's calls on the forward path: every one is recorded and gives zeros."""

    def __init__(self) -> None:
        self.calls: list[tuple[str, int]] = []

    def matmul(self, t, packed, x, n, k):
        self.calls.append(("matmul", x.shape[0]))
        return torch.zeros(x.shape[0], n)

    def matmul_bf16(self, t, packed, x, n, k):
        self.calls.append(("matmul_bf16", x.shape[0]))
        return torch.zeros(x.shape[0], n, dtype=torch.bfloat16)

    def _gemm_bf16(self, t, packed, xb, y, m, n, k):
        assert xb.shape == (m, k) and xb.is_contiguous()
        self.calls.append(("_gemm_bf16", m))
        y.zero_()

    def matmul_q8k(self, t, packed, ws, x, y, m, n, k):
        self.calls.append(("matmul_q8k", m))
        y.zero_()

    def gemv_f32(self, t, packed, x, n, k):
        self.calls.append(("gemv_f32", x.shape[0]))
        return torch.zeros(x.shape[0], n)

    def dequantize(self, packed, t):
        return torch.zeros(N * K)


def _module(dtype, backend="native") -> tuple[DevicePackedLinear, _Stub]:
    mod = DevicePackedLinear(torch.zeros(N, ROW_BYTES, dtype=torch.uint8), K, Q4_K, None, dtype, backend=backend)
    mod._gemm = stub = _Stub()
    return mod, stub


@pytest.mark.parametrize("backend", ["native", "numba"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(3, K + 2), (1, 300), (300, K - 1), (4, K // 2), (2, 2 * K), (K + 1,), (2 * K,),
                                   (2, 3, K + 1), (2, 4, K // 2), (2, 2, 2 * K), ()])
@pytest.mark.parametrize("x_dtype", [torch.bfloat16, torch.float32])
def test_linear_refuses_a_wrong_width(backend, dtype, shape, x_dtype) -> None:
    """F.linear raises for these, also where the elements would fill whole rows."""
    mod, stub = _module(dtype, backend)
    with pytest.raises(RuntimeError):
        mod(torch.ones(shape, dtype=x_dtype))
    assert stub.calls == []


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(4, K // 2), (2, 2 * K), (2, 2, 2 * K)])
def test_linear_refuses_a_wrong_width_after_a_producer(dtype, shape) -> None:
    """The offered blocks of a result of another width are not multiplied, and stay offered."""
    mod, stub = _module(dtype)
    x, ws = torch.ones(shape, dtype=dtype), torch.empty(64, dtype=torch.uint8)
    HANDOFF.offer(x, ws)
    try:
        with pytest.raises(RuntimeError):
            mod(x)
        assert stub.calls == [] and HANDOFF.claim(x) is ws
    finally:
        HANDOFF.clear()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(K,), (1, K), (3, K), (2, 3, K), (0, K), (2, 0, K), (0, K + 2)])
def test_linear_result_shapes(dtype, shape) -> None:
    mod, _ = _module(dtype)
    y = mod(torch.ones(shape, dtype=dtype))
    assert y.shape == (*shape[:-1], N) and y.dtype == dtype


def test_linear_takes_views() -> None:
    """Transposed, strided and offset inputs reach the library as contiguous rows."""
    mod, stub = _module(torch.bfloat16)
    big = torch.ones(8 * K + 8, dtype=torch.bfloat16)
    for x in (big[:4 * K].view(K, 4).T, big[:8 * K].view(4, 2 * K)[:, K:], big[1:1 + 4 * K].view(4, K),
              big[:8 * K].view(8, K)[::2]):
        assert mod(x).shape == (4, N)
    assert stub.calls == [("_gemm_bf16", 4)] * 4


def test_finish_gives_the_leading_shape() -> None:
    """Rows that do not fill the leading shape are an error, never a result of another shape."""
    mod, _ = _module(torch.float32)
    assert mod.finish(torch.zeros(6, N), (2, 3)).shape == (2, 3, N)
    assert mod.finish(torch.zeros(6, N), (6,)).shape == (6, N)
    for lead in ((5,), (12,), (2, 2)):
        with pytest.raises(RuntimeError):
            mod.finish(torch.zeros(6, N), lead)


def test_supports_is_the_librarys_rule() -> None:
    """`HipGemm.supports` answers the common case itself; every answer is the library's."""
    gemm = HipGemm.get()
    for t in range(-1, 40):
        for k in (-256, 0, 1, 32, 255, 256, 288, 512, 2816, 4096, 4097, (1 << 31) - 256):
            assert gemm.supports(t, k) == bool(gemm._lib.mxa_supports(t, k)), (t, k)
