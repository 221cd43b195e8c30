"""Loss functions of a pipeline's last stage that run as one HIP kernel.

``cross_entropy`` has the call shape ``Engine.compute_loss`` uses for ``loss_fn`` —
``loss_fn(output, target, reduction="sum")`` (elf/execution/engine.py:374-410) — and the semantics of
the reference transformer's loss (benchmarks/models/simple.py:520-524): logits flattened to
``[rows, V]``, arithmetic in fp32, ``torch.nn.functional.cross_entropy`` reductions and
``ignore_index``.  Loss and gradient come out of a single pass over the logits; there is no CPU path.
"""

import torch
from torch.autograd import forward_ad

from . import _lib

_PAD = 64  # gradient rows are padded to this many columns, the layout the stage's head GEMM reads


_stream = _lib.raw_stream


def _rows_view(pred, V):
	"""``pred`` as (tensor whose memory the kernel reads, row stride) without copying when its rows are
	evenly strided and 16-byte aligned; otherwise a padded contiguous copy."""
	if pred.dtype != torch.bfloat16 or not pred.is_cuda:
		raise _lib.ElfStageError(f"cross_entropy: logits must be a bf16 GPU tensor, got {pred.dtype} on {pred.device}")
	if pred.shape[-1] != V:
		raise _lib.ElfStageError("cross_entropy: the last dimension of the logits must be the class dimension")
	p = pred if pred.dim() >= 2 else pred.unsqueeze(0)
	ld = p.stride(-2)
	ok = p.stride(-1) == 1 and ld % 8 == 0 and ld >= V and p.data_ptr() % 16 == 0
	expect = ld
	for size, stride in zip(reversed(p.shape[:-1]), reversed(p.stride()[:-1])):
		ok = ok and (size == 1 or stride == expect)
		expect *= size
	if ok:
		return p, ld
	ld = -(-V // 8) * 8
	buf = torch.zeros(p.numel() // V, ld, dtype=torch.bfloat16, device=pred.device)
	buf[:, :V] = p.reshape(-1, V)
	return buf, ld


def _check_target(target, rows):
	if target.dtype != torch.int64 or not target.is_cuda or target.numel() != rows:
		raise _lib.ElfStageError(f"cross_entropy: target must be an int64 GPU tensor of {rows} class indices (probabilities are not supported), got {tuple(target.shape)} {target.dtype} on {target.device}")
	return target.contiguous().view(-1)


_DENSE_MAX = 1024 * 16 * 8 - 7  # widest row elf_cross_entropy_dense holds in registers


def _run(pred, target, *, ignore_index, scale, reduction, want_grad, padded=True):
	"""(loss, grad or None).  The gradient is [rows, ld_out] bf16 with ``ld_out`` a multiple of 64, or, unless ``padded``, [rows, V]
	where V is a multiple of 8 or the logits are one dense block: rows that start at any address are then read in place (50257
	columns: the padded copy of the logits took half of a loss's time)."""
	if reduction not in ("sum", "mean", "none"):
		raise ValueError(f"{reduction} is not a valid value for reduction")
	V = pred.shape[-1]
	dense = V % 8 != 0 and not (want_grad and padded) and pred.dtype == torch.bfloat16 and pred.is_cuda and pred.is_contiguous() and not pred.is_neg() and pred.data_ptr() % 16 == 0 and 0 < V <= _DENSE_MAX
	src, ld = (pred, V) if dense else _rows_view(pred, V)
	rows = pred.numel() // V
	target = _check_target(target, rows)
	lib, stream = _lib.load(), _stream()
	dev = pred.device
	row_loss = torch.empty(rows, dtype=torch.float32, device=dev)
	grad, ld_out, dx = None, 0, None
	if want_grad:
		ld_out = V if dense or (V % 8 == 0 and not padded) else -(-V // _PAD) * _PAD
		grad = torch.empty(rows, ld_out, dtype=torch.bfloat16, device=dev)
		dx = grad.data_ptr()
	if reduction != "none":
		loss, scratch = torch.empty((), dtype=torch.float32, device=dev), torch.empty(2, dtype=torch.float32, device=dev)
		rc = lib.elf_cross_entropy_loss(src.data_ptr(), ld, dense, target.data_ptr(), rows, V, ignore_index, scale, reduction == "mean",
			row_loss.data_ptr(), loss.data_ptr(), dx, ld_out, scratch.data_ptr(), stream)
		_lib.check(rc, "elf_cross_entropy_loss")
		return loss, grad
	if dense:
		_lib.check(lib.elf_cross_entropy_dense(src.data_ptr(), target.data_ptr(), rows, V, ignore_index, scale, None, row_loss.data_ptr(), dx, stream), "elf_cross_entropy_dense")
	else:
		_lib.check(lib.elf_cross_entropy(src.data_ptr(), ld, target.data_ptr(), rows, V, ignore_index, scale, None, row_loss.data_ptr(), dx, ld_out, stream), "elf_cross_entropy")
	return row_loss.view(pred.shape[:-1]), grad


_has_storage, _wrapped, _dispatch_modes = torch._C._has_storage, torch._C._functorch.is_functorch_wrapped_tensor, torch._C._len_torch_dispatch_stack


def _plain(t):
	"""Whether a kernel may read ``t`` through its pointer: under vmap it is a batch without storage of its own, and a view
	such as ``z.conj().imag`` holds its values negated.  Nor may it where somebody follows the operations on ``t``: in a
	forward-mode level (a tangent) or under a dispatch mode (a trace)."""
	return (type(t) is torch.Tensor and _has_storage(t) and not _wrapped(t) and not t.is_neg() and not t._is_zerotensor()
	        and forward_ad._current_level < 0 and not _dispatch_modes())


class _CrossEntropy(torch.autograd.Function):
	@staticmethod
	def forward(ctx, pred, target, reduction, ignore_index):
		loss, ctx.grad = _run(pred, target, ignore_index=ignore_index, scale=1.0, reduction=reduction, want_grad=ctx.needs_input_grad[0], padded=False)
		ctx.shape, ctx.per_row = pred.shape, reduction == "none"
		return loss

	@staticmethod
	def backward(ctx, g):
		V = ctx.shape[-1]
		grad = ctx.grad
		if grad.shape[1] == V and g.dim() == 0 and g.dtype == torch.float32 and not (g.requires_grad and torch.is_grad_enabled()) and _plain(g):
			# one pass of 16-byte accesses with the same roundings (2048 x 50257: 60 us, 82 as a torch product of the strided view)
			out = torch.empty(ctx.shape, dtype=grad.dtype, device=grad.device)
			_lib.check(_lib.load().elf_scale_by_bf16(grad.data_ptr(), g.data_ptr(), out.data_ptr(), out.numel(), _stream()), "elf_scale_by_bf16")
			return out, None, None, None
		grad = grad[:, :V]
		grad = grad * (g.reshape(-1, 1) if ctx.per_row else g).to(grad.dtype)
		return grad.view(ctx.shape), None, None, None


def cross_entropy(pred, target, reduction="mean", ignore_index=-100):
	"""Drop-in for ``torch.nn.functional.cross_entropy(pred.float().view(-1, V), target.view(-1))`` on
	bf16 GPU logits ``[..., V]`` and int64 class indices ``[...]``; differentiable w.r.t. ``pred``."""
	if pred.requires_grad and torch.is_grad_enabled():
		return _CrossEntropy.apply(pred, target, reduction, ignore_index)
	return _run(pred, target, ignore_index=ignore_index, scale=1.0, reduction=reduction, want_grad=False)[0]


def _loss_and_grad(pred, target, reduction="sum", ignore_index=-100, scale=1.0):
	"""The loss and ``scale`` times its gradient w.r.t. ``pred`` from one kernel, without autograd.
	``Engine.compute_loss`` calls this when the loss function offers it.  The gradient is a view of a
	``[rows, V rounded up to 64]`` buffer whose extra columns are zero: the layout a last stage reads
	in place."""
	if reduction not in ("sum", "mean"):
		raise ValueError("loss_and_grad needs a scalar loss: reduction must be 'sum' or 'mean'")
	loss, grad = _run(pred, target, ignore_index=ignore_index, scale=scale, reduction=reduction, want_grad=True)
	V = pred.shape[-1]
	return loss, grad.view(*pred.shape[:-1], -1)[..., :V]


cross_entropy.loss_and_grad = _loss_and_grad
