"""elf_amd.zb_utils up to its kernel calls: what reaches the kernel of LinearDX.forward as the bias row, what is refused, and which way the W pass
of a list of layers goes."""

from contextlib import nullcontext
from types import SimpleNamespace

import pytest
import torch

from elf_amd import zb_utils
from elf_amd.execution.autograd_block import AutogradStageBlock


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


class _OnCpu:
	"""The W kernels as plain sums on the CPU, and what was asked of them."""

	def __init__(self, monkeypatch):
		self.asked = []
		for name in ("gemm", "colsum_", "linear_w_pass"):
			monkeypatch.setattr(zb_utils.kernels, name, getattr(self, name))

	def gemm(self, go, x, *, a_t, b_t, out, epilogue):
		assert a_t and b_t and epilogue == zb_utils.kernels.EPI_F32_ACC and go.is_contiguous() and x.is_contiguous()
		self.asked.append("one")
		out += (go.float().t() @ x.float()).to(out.dtype)

	def colsum_(self, go, out):
		out += go.float().sum(0).to(out.dtype)

	def linear_w_pass(self, layers):
		self.asked.append(len(layers))
		for go, x, acc, bias in layers:
			assert go.shape[0] == layers[0][0].shape[0] and all(t.is_contiguous() for t in (go, x, acc)) and acc.dtype == torch.float32
			acc += go.float().t() @ x.float()
			if bias is not None:
				bias += go.float().sum(0)


def _stashed(tokens=64, cls=None, bias=True, m=128, n=64):
	layer = (cls or zb_utils.LinearDW)(torch.nn.Linear(n, m, bias=bias).to(torch.bfloat16))
	layer.set("grad_output", 0, torch.randn(tokens // 32, 32, m).to(torch.bfloat16))
	layer.set("input", 0, torch.randn(tokens // 32, 32, n).to(torch.bfloat16))
	return layer


def _w_pass(layers):
	"""backward_params of a generic block that holds these layers; checks the gradients."""
	want = []
	for l in layers:
		go, x = l.ctx["grad_output"][0].flatten(0, -2).float(), l.ctx["input"][0].flatten(0, -2).float()
		want.append((go.t() @ x, go.sum(0)))
	block = SimpleNamespace(id=0, _timed=lambda name: nullcontext(), _layers_dw=lambda: layers)
	AutogradStageBlock.backward_params(block, 0)
	for l, (w, b) in zip(layers, want):
		assert l.is_empty("grad_output") and l.is_empty("input")
		tol = dict(rtol=1e-4, atol=1e-3) if l.weight.main_grad.dtype == torch.float32 else dict(rtol=2e-2, atol=2e-1)  # (bf16: one rounding, 2^-9)
		assert torch.allclose(l.weight.main_grad.float(), w, **tol)
		assert l.bias is None or torch.allclose(l.bias.main_grad.float(), b, rtol=1e-4, atol=1e-3)


def test_w_pass_takes_layers_over_the_same_tokens_together(monkeypatch):
	k = _OnCpu(monkeypatch)
	_w_pass([_stashed(64), _stashed(128), _stashed(64, bias=False), _stashed(128), _stashed(64)])
	assert k.asked == [3, 2]


@pytest.mark.parametrize("what", ["rows of the accumulator apart", "accumulator in bf16", "strided gradient", "strided input"])
def test_w_pass_of_a_layer_that_a_common_call_does_not_take(monkeypatch, what):
	"""It goes by itself, as before there was one; what has to be copied to dense rows is copied for one layer at a time."""
	k = _OnCpu(monkeypatch)
	odd = [_stashed(), _stashed()]
	for l in odd:
		if what == "rows of the accumulator apart":
			l.weight.main_grad = torch.zeros(128, 96)[:, :64]
		elif what == "accumulator in bf16":
			l.weight.main_grad = torch.zeros(128, 64, dtype=torch.bfloat16)
		else:
			q = "grad_output" if what == "strided gradient" else "input"
			l.ctx[q][0] = l.ctx[q][0].transpose(0, 1).contiguous().transpose(0, 1)
	_w_pass([odd[0], _stashed(), odd[1], _stashed()])
	assert k.asked == ["one", "one", 2]


def test_w_pass_asks_a_backward_that_is_not_linear_dws_own(monkeypatch):
	k, asked = _OnCpu(monkeypatch), []

	class Own(zb_utils.LinearDW):
		def backward(self, mb_id):
			asked.append("class")
			super().backward(mb_id)

	wrapped = _stashed()
	monkeypatch.setattr(wrapped, "backward", lambda mb: (asked.append("object"), zb_utils.LinearDW.backward(wrapped, mb)))
	_w_pass([_stashed(cls=Own), wrapped, _stashed()])
	assert asked == ["class", "object"] and k.asked == ["one", "one", 1]
	own = zb_utils.LinearDW.backward
	monkeypatch.setattr(zb_utils.LinearDW, "backward", lambda self, mb: (asked.append("patched"), own(self, mb)))
	_w_pass([_stashed(), _stashed()])
	assert asked[2:] == ["patched", "patched"]
