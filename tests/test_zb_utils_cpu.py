"""The forward of elf_amd.zb_utils.LinearDX up to its kernel call: what reaches the kernel as the bias row, and what is refused."""

import pytest
import torch

from elf_amd import zb_utils


class _Layer:
	def _store_input(self, x):
		pass


@pytest.fixture
def rows(monkeypatch):
	seen = []

	def gemm(x, w, *, residual, **kw):
		seen.append(residual)
		return x @ w.t() + residual

	monkeypatch.setattr(zb_utils.kernels, "gemm", gemm)
	return seen


@pytest.mark.parametrize("form", ["dense", "one_row", "strided", "reversed_rows", "single"])
def test_linear_dx_hands_the_kernel_a_dense_bias_row(rows, form):
	x, w = torch.randn(4, 64), torch.randn(128, 64)
	bias = {"dense": torch.randn(128), "one_row": torch.randn(1, 128), "strided": torch.randn(256)[::2], "reversed_rows": torch.randn(2, 64).t(), "single": torch.randn(1)}[form]
	y = zb_utils.LinearDX.apply(x, w, bias, _Layer())
	assert rows[0].numel() == 128 and rows[0].is_contiguous()
	assert torch.equal(y, x @ w.t() + bias.reshape(1, -1))


@pytest.mark.parametrize("n", [64, 127, 256])
def test_linear_dx_refuses_a_bias_of_another_size(rows, n):
	with pytest.raises(RuntimeError, match="expanded size"):
		zb_utils.LinearDX.apply(torch.randn(4, 64), torch.randn(128, 64), torch.randn(n), _Layer())
	assert not rows
