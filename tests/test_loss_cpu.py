"""The backward of ``losses.cross_entropy`` where what arrives is followed by something a kernel does not see: it must stay a
product of torch operations (no GPU needed, the kernel would fail on these tensors)."""

import types

import torch
import torch.autograd.forward_ad as fwAD
from torch.fx.experimental.proxy_tensor import make_fx

from elf_amd.losses import _CrossEntropy


def _backward(g):
	ctx = types.SimpleNamespace(grad=torch.arange(12, dtype=torch.bfloat16).view(3, 4), shape=(3, 4), per_row=False)
	return _CrossEntropy.backward(ctx, g)[0]


def test_tangent_of_the_incoming_gradient_is_carried_on():
	with fwAD.dual_level():
		value, tangent = fwAD.unpack_dual(_backward(fwAD.make_dual(torch.tensor(2.0), torch.tensor(0.5))))
		assert torch.equal(value, torch.arange(12, dtype=torch.bfloat16).view(3, 4) * 2)
		assert torch.equal(tangent, torch.arange(12, dtype=torch.bfloat16).view(3, 4) * 0.5)


def test_traced_backward_depends_on_the_incoming_gradient():
	traced = make_fx(_backward)(torch.tensor(1.0))
	for g in (torch.tensor(2.0), torch.tensor(-3.0)):
		assert torch.equal(traced(g), torch.arange(12, dtype=torch.bfloat16).view(3, 4) * g.to(torch.bfloat16))
