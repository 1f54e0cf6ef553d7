"""What the linears hand to the native library for views of activations and outputs
(CPU only: the native calls are recorded, not made)."""
import pytest
import torch

from helm_amd import kernels as hk

K, N = 64, 48


@pytest.fixture
def calls(monkeypatch):
    made = []
    monkeypatch.setattr(hk._native, "require_cuda", lambda *t, what: None)
    monkeypatch.setattr(hk._native, "stream_ptr", lambda device=None: 0)
    monkeypatch.setattr(hk._native, "call", lambda name, *args: made.append((name, args)))
    return made


def _half(*shape):
    return torch.randn(*shape).half()


VIEWS = {
    "contiguous row": lambda: _half(1, K),
    "transposed column": lambda: _half(K, 1).t(),
    "odd row stride": lambda: _half(2, K + 1)[:1, :K],
    "one row of overlapping rows": lambda: _half(3 * K).as_strided((1, K), (1, 1)),
    "one-dimensional": lambda: _half(K),
    "last position": lambda: _half(1, 5, K)[:, -1],
    "padded rows": lambda: _half(3, 2 * K)[:, :K],
    "odd padded rows": lambda: _half(3, K + 1)[:, :K],
    "batch and sequence": lambda: _half(2, 3, K).transpose(0, 1),
    "many rows": lambda: _half(20, K),
}


@pytest.mark.parametrize("view", VIEWS)
@pytest.mark.parametrize("fp16", [False, True], ids=["int8", "fp16"])
def test_row_operands_are_ones_the_kernels_take(calls, view, fp16):
    x = VIEWS[view]()
    rows = x.reshape(-1, K)
    if fp16:
        if rows.shape[0] > hk.GEMV_MAX_TOKENS:
            pytest.skip("a library product")
        y = hk.fp16_linear(x, _half(N, K))
    else:
        y = hk.int8_linear(x, torch.ones(N, K, dtype=torch.int8), _half(N))
    (name, args), = calls
    ptr, ldx = args[0], args[1]
    assert ldx >= K and ldx % 8 == 0 and ptr % 16 == 0
    # in place unless the rows are ones the kernels do not take
    if rows.data_ptr() == x.data_ptr() and rows.stride(0) % 8 == 0:
        assert ptr == x.data_ptr() and (ldx == rows.stride(0) or rows.shape[0] == 1)
    assert y.shape == (*x.shape[:-1], N)


@pytest.mark.parametrize("out", ["contiguous", "transposed column", "padded rows", "three dims"])
def test_output_views_are_written_in_place(calls, out):
    y = {"contiguous": lambda: _half(1, N), "transposed column": lambda: _half(N, 1).t(),
         "padded rows": lambda: _half(1, N + 8)[:, :N], "three dims": lambda: _half(1, 1, N)}[out]()
    r = hk.int8_linear(_half(1, K), torch.ones(N, K, dtype=torch.int8), _half(N), out=y)
    (name, args), = calls
    assert r is y and args[7] == y.data_ptr() and args[8] >= N
