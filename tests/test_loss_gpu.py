"""The one-kernel cross-entropy of a last stage (elf_cross_entropy) against the CPU oracle
(oracle/loss_ref.py: fp32 torch.nn.functional.cross_entropy on the upcast logits, as
benchmarks/models/simple.py:520-524).  Tolerances: per-row loss rel 1e-5 / abs 2e-5 (fp32 arithmetic
on identical bf16 inputs; only the summation order differs); gradient within one bf16 rounding of
the fp32 gradient (rel 2^-7 of the element, abs 1e-6 of the scale)."""

import pytest
import torch

from oracle import loss_ref as L

pytestmark = pytest.mark.gpu


def _case(rows, V, seed, ld=None, spread=4.0):
	g = torch.Generator().manual_seed(seed)
	x = (torch.randn(rows, V, generator=g) * spread).to(torch.bfloat16)
	t = torch.randint(0, V, (rows,), generator=g)
	t[::7] = -100
	t[1] = V - 1
	t[2] = 0
	if ld is None:
		return x, t, x.cuda()
	buf = torch.full((rows, ld), float("nan"), dtype=torch.bfloat16).cuda()  # what lies between rows must not matter
	buf[:, :V] = x.cuda()
	return x, t, buf[:, :V]


def _check_grad(got, want_f32, scale):
	got, want = got.float().cpu(), want_f32
	err = (got - want).abs()
	assert bool((err <= want.abs() * 2.0**-7 + 1e-6 * scale).all()), f"max err {err.max().item():.3e}"


# (rows, V, row stride): wave per row (two register depths), 4 / 16 waves per row, 16 chunks per lane,
# the two-read kernel for rows beyond the register budget, V not a multiple of 8 (padded copy), tiny rows
@pytest.mark.parametrize("rows,V,ld", [(37, 1000, 1024), (64, 1000, None), (16, 50257, None), (33, 4096, 4096), (9, 16384, 16400), (5, 65536, None), (6, 128256, None), (3, 150001, None), (3, 200000, None), (3, 8, None), (5, 3, None)])
def test_cross_entropy_loss_and_gradient(rows, V, ld):
	from elf_amd import losses

	x, t, xg = _case(rows, V, seed=rows + V, ld=ld)
	tg = t.cuda()
	want_rows = L.cross_entropy_ref(x, t, "none")
	for reduction in ("none", "sum", "mean"):
		got = losses.cross_entropy(xg, tg, reduction=reduction)
		want = L.cross_entropy_ref(x, t, reduction)
		assert torch.allclose(got.cpu(), want, rtol=1e-5, atol=2e-5 * (1 if reduction != "sum" else rows)), reduction
	# gradient, scaled in the kernel
	xf = x.float().requires_grad_()
	L.cross_entropy_ref(xf, t, "sum").backward()
	scale = 1.0 / 128
	loss, grad = losses.cross_entropy.loss_and_grad(xg, tg, reduction="sum", scale=scale)
	assert float(loss) == pytest.approx(float(want_rows.sum()), rel=1e-5)
	assert tuple(grad.shape) == (rows, V) and grad.stride(0) % 64 == 0
	_check_grad(grad, xf.grad * scale, scale)
	assert grad[t == -100].abs().max().item() == 0
	base = torch.as_strided(grad, (rows, grad.stride(0)), (grad.stride(0), 1))
	assert base[:, V:].abs().sum().item() == 0  # padding columns are zeros
	# mean: divides by the live rows, through autograd with an upstream factor
	xa = xg.detach().clone().requires_grad_()
	(losses.cross_entropy(xa, tg) * 3.0).backward()
	live = int((t != -100).sum())
	_check_grad(xa.grad, xf.grad * (3.0 / live), 3.0 / live)


@pytest.mark.parametrize("rows,V", [(2048, 1000), (2049, 1000), (2048, 4089), (2048, 4090), (2047, 4096), (66, 4097), (700, 48000)])
def test_mean_where_the_loss_kernel_counts_the_live_rows_and_where_it_does_not(rows, V):
	"""Up to 2048 rows of up to 4096 columns (a dense row may cover 7 more) every wave counts the rows that are not ignored, beyond
	that a launch before it does; logits from 2^25 elements up are read past the caches.  Mean and gradient against fp32 of PyTorch."""
	from elf_amd import losses

	x, t, xg = _case(rows, V, seed=rows * 7 + V)
	xa = xg.detach().clone().requires_grad_()
	loss = losses.cross_entropy(xa, t.cuda())
	loss.backward()
	xf = x.float().cuda().requires_grad_()
	want = torch.nn.functional.cross_entropy(xf, t.cuda())
	want.backward()
	assert float(loss.detach()) == pytest.approx(float(want.detach()), rel=1e-5)
	_check_grad(xa.grad, xf.grad.cpu(), 1.0 / int((t != -100).sum()))
	none = losses.cross_entropy(xg, torch.full_like(t, -100).cuda())
	assert torch.isnan(none)  # no live row, as torch


@pytest.mark.parametrize("rows,V", [(1800, 48000), (1800, 47999), (10239, 8192), (10240, 8192), (10250, 8191), (32800, 4096)])
def test_mean_of_logits_that_are_read_past_the_caches(rows, V):
	"""5 x 2^24 logits in long rows, 2^27 in narrower ones, and either side of these lines.  Bounds as above."""
	test_mean_where_the_loss_kernel_counts_the_live_rows_and_where_it_does_not(rows, V)


@pytest.mark.parametrize("rows,V", [(1024, 1000), (1025, 1000), (1024, 4089), (1024, 4090), (1023, 4096)])
def test_mean_on_both_sides_of_1024_rows(rows, V):
	"""The line up to which every wave counts the rows that are not ignored, at either end of the widths.  Bounds as above."""
	test_mean_where_the_loss_kernel_counts_the_live_rows_and_where_it_does_not(rows, V)


@pytest.mark.parametrize("rows,V,ld", [(9, 3, 8), (300, 1003, 1024), (37, 1230, 1232), (5, 4095, 4160), (7, 16381, 16384), (6, 20003, 20032), (3, 65533, 65536), (3, 100001, 100008)])
def test_last_columns_of_rows_no_chunk_divides(rows, V, ld):
	"""V that is no multiple of 8, in rows that lie ld apart with NaN between them: every register depth, the target and infinities
	in the last columns, and zeros from column V to the end of the gradient's rows."""
	from elf_amd import losses

	x, t, xg = _case(rows, V, seed=V, ld=ld)
	x[0, V - 1] = xg[0, V - 1] = float("-inf")
	t[0] = 1  # (not ignored)
	t[rows - 1] = V - 1
	xf = x.float().requires_grad_()
	L.cross_entropy_ref(xf, t, "sum").backward()
	loss, grad = losses.cross_entropy.loss_and_grad(xg, t.cuda(), reduction="sum")
	assert float(loss) == pytest.approx(float(L.cross_entropy_ref(x, t, "sum")), rel=1e-5)
	_check_grad(grad, xf.grad, 1.0)
	base = torch.as_strided(grad, (rows, grad.stride(0)), (grad.stride(0), 1))
	assert base[:, V:].float().abs().sum().item() == 0


# dense rows that start at every 2-byte phase (odd widths), at the widest of each register depth and one beyond it, and a base
# that is not 16-byte aligned (the padded copy)
@pytest.mark.parametrize("V", [1, 7, 9, 1017, 1018, 4089, 4091, 16377, 16379, 32761, 32763, 65529, 65531, 131065, 131067])
@pytest.mark.parametrize("offset", [0, 1])
def test_cross_entropy_dense_rows_of_any_width(V, offset):
	from elf_amd import losses

	rows = 11
	x, t, _ = _case(rows, V, seed=V)
	t[3] = V - 1  # the last column
	t[4] = 0
	buf = torch.zeros(rows * V + offset, dtype=torch.bfloat16).cuda()
	buf[offset:] = x.reshape(-1).cuda()
	xg = buf[offset:].view(rows, V).requires_grad_()
	xf = x.float().requires_grad_()
	want = L.cross_entropy_ref(xf, t, "mean")
	want.backward()
	got = losses.cross_entropy(xg, t.cuda())
	assert torch.allclose(got.detach().cpu(), want.detach(), rtol=1e-5, atol=2e-5)
	(grad,) = torch.autograd.grad(got, xg, retain_graph=True)
	live = int((t != -100).sum())
	_check_grad(grad, xf.grad, 1.0 / live)
	assert V == 1 or grad[t == -100].abs().max().item() == 0
	(twice,) = torch.autograd.grad(got, xg, grad_outputs=torch.tensor(-2.0).cuda())  # the kept gradient is not consumed
	assert torch.equal(twice, grad * -2)


@pytest.mark.parametrize("n", [1, 7, 8, 2047, 2048, 2049, 4103, (1 << 25) - 9, (1 << 25) - 1, 1 << 25, (1 << 25) + 4095, (1 << 25) + 8191])
def test_scaling_pass_at_the_edges_of_its_grids(n):
	"""Whole and partly filled workgroups of one and two chunks a thread, the last elements of no whole chunk, the step to the pass
	that goes past the caches: the bits of the torch product, nothing behind the end touched."""
	from elf_amd import _lib

	x = torch.randn(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(n)).to(torch.bfloat16)
	g, y = torch.tensor(-1.7, device="cuda"), torch.full((n + 4096,), 7.0, dtype=torch.bfloat16, device="cuda")
	_lib.check(_lib.load().elf_scale_by_bf16(x.data_ptr(), g.data_ptr(), y.data_ptr(), n, torch.cuda.current_stream().cuda_stream), "elf_scale_by_bf16")
	assert torch.equal(y[:n], x * g.to(torch.bfloat16)) and bool((y[n:] == 7).all())


@pytest.mark.parametrize("V", [1000, 1003])
def test_cross_entropy_gradients_for_a_batch_of_incoming_gradients(V):
	"""``is_grads_batched``: the backward is run once under vmap, with an incoming gradient that has no storage of its own; and an
	incoming gradient whose storage holds something else than its value."""
	from elf_amd import losses

	x, t, xg = _case(11, V, seed=V)
	xg = xg.detach().clone().requires_grad_()
	loss = losses.cross_entropy(xg, t.cuda())
	(one,) = torch.autograd.grad(loss, xg, retain_graph=True)
	g = torch.tensor([1.0, -2.0, 0.5]).cuda()
	(many,) = torch.autograd.grad(loss, xg, grad_outputs=g, is_grads_batched=True)
	assert tuple(many.shape) == (3, 11, V)
	for i in range(3):
		assert torch.equal(many[i], one * g[i].to(torch.bfloat16))
	lazy = torch.tensor(3 - 2j).cuda().conj().imag  # 2, kept as the negation of -2
	assert lazy.is_neg() and lazy.item() == 2
	(twice,) = torch.autograd.grad(loss, xg, grad_outputs=lazy)
	assert torch.equal(twice, one * 2)


def test_cross_entropy_rejects_what_it_cannot_run_and_flags_bad_targets():
	from elf_amd import _lib, losses

	x = torch.randn(4, 16).to(torch.bfloat16).cuda()
	t = torch.tensor([1, 2, 99, -100]).cuda()
	got = losses.cross_entropy(x, t, reduction="none")
	assert torch.isnan(got[2]) and not torch.isnan(got[[0, 1, 3]]).any() and got[3].item() == 0
	with pytest.raises(_lib.ElfStageError):
		losses.cross_entropy(x.float(), t)
	with pytest.raises(_lib.ElfStageError):
		losses.cross_entropy(x, t.int())
	with pytest.raises(_lib.ElfStageError):
		losses.cross_entropy(x.cpu(), t.cpu())
	with pytest.raises(ValueError):
		losses.cross_entropy(x, t, reduction="max")


def test_engine_compute_loss_takes_the_one_kernel_path():
	"""Engine.compute_loss with the library loss equals the oracle's restatement of the reference's
	compute_loss (sum over the micro-batch / elements per sample, gradient in bf16)."""
	from elf_amd import losses
	from elf_amd.execution.engine import compute_loss

	class _Block:
		compute_time = []

	mb, S, V = 4, 128, 1000
	g = torch.Generator().manual_seed(5)
	buf = (torch.randn(mb, S, 1024, generator=g) * 3).to(torch.bfloat16).cuda()
	out = buf[..., :V]  # the view a last stage hands out
	tgt = torch.randint(0, V, (mb, S), generator=g)
	want_loss, want_grad = L.compute_loss_ref(out.cpu(), tgt)
	loss, grad_fn = compute_loss(_Block, out, tgt.cuda(), losses.cross_entropy)
	(grad,) = grad_fn()
	assert float(loss) == pytest.approx(float(want_loss), rel=1e-5)
	assert not loss.requires_grad and grad.shape == out.shape
	xf = out.cpu().float().requires_grad_()
	(L.cross_entropy_ref(xf, tgt, "sum") / S).backward()
	_check_grad(grad, xf.grad, 1.0 / S)
	assert torch.equal(grad.cpu(), want_grad) or (grad.cpu().float() - want_grad.float()).abs().max().item() <= 2.0**-7 / S
