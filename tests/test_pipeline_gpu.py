"""``Pipeline`` over the native stage executor (reference API: elf/pipeline.py:97-295): two stages on
one rank under AFAB, and one stage under ZB-H1, against the oracle stages driven by hand with the
same loss.  Tolerances as for the stage tests (rel 2e-2 of max, 1e-2 Frobenius)."""

import pytest
import torch
import torch.nn.functional as F

from tests.helpers import assert_close, cfg_from_stage, oracle_params_from_stage, perturb_norms, product_grads

pytestmark = pytest.mark.gpu


def _stages(n):
	from elf_amd import models

	out = []
	for i in range(n):
		st = models.llama_stage(1, 256, 2, 1, 512, 128, head_dim=128, seed=20 + i)
		perturb_norms(st)
		out.append(st)
	return out


# (scheduler, placement, total batch, split): an even split, a batch the split size does not divide (short
# last micro-batch: elf/pipeline.py:497-500) and an explicit list of sizes (elf/pipeline.py:501-503)
@pytest.mark.parametrize("case", [("afab", [0, 0], 6, 2), ("zbh1", [0], 6, 2), ("afab", [0, 0], 5, 2), ("zbh1", [0], 5, [1, 2, 2])])
def test_pipeline_step_matches_oracle(case):
	from elf_amd.pipeline import Pipeline, PipelineConfig
	from oracle import stage_ref as R

	sched, placement, total, split = case
	mb = 2
	sizes = split if isinstance(split, list) else [mb] * (total // mb) + ([total % mb] if total % mb else [])
	nmb, starts = len(sizes), [sum(sizes[:i]) for i in range(len(sizes))]
	stages = _stages(len(placement))
	refs = [R.RefStage(cfg_from_stage(st, mb), oracle_params_from_stage(st), device="cuda") for st in stages]
	S, d = stages[0].seq_len, 256
	g = torch.Generator().manual_seed(7)
	batch = torch.randn(total, S, d, generator=g).to(torch.bfloat16).cuda()
	target = torch.randn(total, S, d, generator=g).to(torch.bfloat16).cuda()

	pipe = Pipeline(stages if len(stages) > 1 else stages[0], batch[:mb], config=PipelineConfig(scheduler=sched, partitioner=False, placement=placement))
	assert pipe.is_first() and pipe.is_last() and [b.id for b in pipe.blocks] == list(range(len(placement)))
	pipe.zero_grad()
	result, loss = pipe(batch, target, F.mse_loss, split_size=split)
	assert len(result) == nmb and pipe.last_nmb == nmb
	assert set(pipe.stats) == {"total", "idle", "start_idle", "end_idle", "bubble"}
	assert list(pipe.detailed_stats["memories"]) == [str(op) for op in pipe.schedule]

	want_loss = 0.0
	for m in range(nmb):
		x = batch[starts[m]:starts[m] + sizes[m]]
		for ref in refs:
			x = ref.forward(m, x)
		y = x.detach().float().requires_grad_()
		t = target[starts[m]:starts[m] + sizes[m]].float()
		l = F.mse_loss(y, t, reduction="sum") / (S * d)
		l.backward()
		want_loss += float(l.detach())
		assert_close(result[m].reshape(sizes[m], S, d), x, f"{sched} output[{m}]")
		dy = y.grad.to(torch.bfloat16)
		for ref in reversed(refs):
			dy = ref.backward_inputs(m, dy)
		for ref in refs:
			ref.backward_params(m)
	for ref in refs:
		ref.scale_grads(total)
	assert abs(float(loss) - want_loss / total) <= 2e-2 * abs(want_loss / total)
	for st, ref in zip(stages, refs):
		got, want = product_grads(st), ref.grads()
		for name in sorted(want):
			assert_close(got[name], want[name], f"{sched} grad {name}")

	# a second step with the same batch reuses the schedule and gives the same loss
	pipe.zero_grad()
	_, loss2 = pipe(batch, target, F.mse_loss, split_size=split)
	assert abs(float(loss2) - float(loss)) <= 1e-3 * abs(float(loss))
	assert sum(p.numel() for p in pipe.parameters()) == sum(p.numel() for st in stages for p in st.parameters())
	pipe.clear()


def test_pipeline_checkpoint_round_trip(tmp_path):
	"""The reference's per-rank checkpoint layout (elf/pipeline.py:346-368), written and read back: the
	restored weights are the ones the library computes with."""
	from elf_amd.pipeline import Pipeline

	stages = _stages(2)
	mb, S, d = 2, stages[0].seq_len, 256
	batch = torch.randn(mb * 2, S, d, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).cuda()
	pipe = Pipeline(stages, batch[:mb], scheduler="afab", partitioner=False, placement=[0, 0])
	out0, _ = pipe(batch, batch, F.mse_loss, split_size=mb)
	pipe.checkpoint(epoch="e1", dir_path=str(tmp_path))
	state = torch.load(tmp_path / "e1" / "dp0_pp0.pt", weights_only=True)
	assert {"rank", "pp", "dp", "epoch", "state_dict_0", "state_dict_1"} <= set(state) and state["epoch"] == "e1"
	assert set(state["state_dict_0"]) == set(stages[0].state_dict())
	with torch.no_grad():
		for p in pipe.parameters():
			p.mul_(0.5)
	out1, _ = pipe(batch, batch, F.mse_loss, split_size=mb)
	assert not torch.equal(out1[0], out0[0])
	pipe.load_checkpoint(epoch="e1", dir_path=str(tmp_path))
	out2, _ = pipe(batch, batch, F.mse_loss, split_size=mb)
	assert all(torch.equal(a, b) for a, b in zip(out2, out0))
	pipe.save(str(tmp_path / "full.pt"))
	full = torch.load(tmp_path / "full.pt", weights_only=True)
	assert set(full) == {n for n, _ in pipe.named_parameters()} and set(pipe.gather_parameters()) == set(full)


def test_pipeline_rejects_what_this_build_does_not_run():
	from elf_amd.pipeline import Pipeline

	st = _stages(1)[0]
	with pytest.raises(NotImplementedError):
		Pipeline(st, torch.zeros(2, 128, 256), scheduler="afab", placement=[0])  # default partitioner needs a tracer
	with pytest.raises(ValueError):
		Pipeline(st, None, scheduler="afab", partitioner=False, placement=[0])  # no sample, no mb_size
	pipe = Pipeline(st, None, scheduler="afab", partitioner=False, placement=[0], mb_size=2)
	with pytest.raises(ValueError):
		pipe(torch.zeros(6, 128, 256, dtype=torch.bfloat16, device="cuda"), None, None, split_size=3)  # larger than the stage was sized for


def test_memory_figures_of_one_allocator_query():
	from elf_amd.execution import engine as E

	keep = torch.empty(3 << 20, dtype=torch.uint8, device="cuda")
	del keep
	held = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
	assert E._mem() == (torch.cuda.memory_allocated(), torch.cuda.max_memory_allocated())
	torch.cuda.reset_peak_memory_stats()
	assert E._mem() == (torch.cuda.memory_allocated(), torch.cuda.max_memory_allocated())
	del held


def test_memory_figures_where_the_torch_library_does_not_load(monkeypatch, tmp_path):
	from elf_amd import _lib
	from elf_amd.execution import engine as E

	bad = tmp_path / "libelf_torch.so"
	bad.write_bytes(b"no library")
	held = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")
	monkeypatch.setattr(_lib, "TORCH_LIB_PATH", str(bad))
	monkeypatch.setattr(_lib, "_torch_allocated", None)
	for _ in range(2):
		assert E._mem() == (torch.cuda.memory_allocated(), torch.cuda.max_memory_allocated())
	del held


def test_steps_in_a_row_hand_over_their_own_outputs():
	"""Six steps on six batches without a wait in between: the host is never more than two steps' output copies ahead, and every
	step's outputs and loss are those the same step gives alone."""
	from elf_amd.pipeline import Pipeline, PipelineConfig

	g = torch.Generator().manual_seed(11)
	batches = [torch.randn(4, 128, 256, generator=g).to(torch.bfloat16).cuda() for _ in range(6)]
	target = torch.zeros_like(batches[0])
	pipe = Pipeline(_stages(2), batches[0][:2], config=PipelineConfig(scheduler="afab", partitioner=False, placement=[0, 0]))
	alone = []
	for b in batches:
		out, loss = pipe(b, target, F.mse_loss, split_size=2)
		torch.cuda.synchronize()
		alone.append(([o.clone() for o in out], float(loss)))
	got = []
	for b in batches:
		got.append(pipe(b, target, F.mse_loss, split_size=2))
		assert len(pipe.engine._output_copies) <= 2
	torch.cuda.synchronize()
	for (out, loss), (want, want_loss) in zip(got, alone):
		assert all(o.device.type == "cpu" and torch.equal(o, w) for o, w in zip(out, want)) and float(loss) == want_loss


@pytest.mark.parametrize("sched,n_stages,d,V", [("afab", 1, 256, 16384), ("full_remat", 1, 256, 16384), ("afab", 2, 1024, 1024), ("full_remat", 2, 1024, 1024)])
def test_every_micro_batch_hands_over_its_own_logits(sched, n_stages, d, V):
	"""Six micro-batches whose logits take longer to the host than the kernels in between: each one's are those it gives in a step of its own.
	While a copy waits its turn nothing else is written where it reads: not the next logits (one stage), not the gradient that the last
	stage's backward makes right behind (two, of the logits' size)."""
	from elf_amd import losses
	from elf_amd.models import EndStage, StageModule, TransformerBlock
	from elf_amd.pipeline import Pipeline

	S, n = 256, 6
	torch.manual_seed(5)
	with torch.device("cuda"):
		stages = [EndStage(StageModule([TransformerBlock(d, d // 64, 4 * d)], S), vocab_in=V if i == 0 else None, vocab_out=V if i == n_stages - 1 else None) for i in range(n_stages)]
	stages = [st.to(torch.bfloat16) for st in stages]
	ids = torch.randint(0, V, (4 * n, S + 1), generator=torch.Generator().manual_seed(6)).cuda()
	x, t = ids[:, :-1].contiguous(), ids[:, 1:].contiguous()
	pipe = Pipeline(stages, scheduler=sched, partitioner=False, placement=[0] * n_stages, mb_size=4)
	alone = []
	for i in range(n):
		logits, _ = pipe(x[4 * i : 4 * i + 4], t[4 * i : 4 * i + 4], losses.cross_entropy, split_size=4)
		torch.cuda.synchronize()
		alone.append(logits[0].clone())
	for _ in range(3):
		pipe.zero_grad()
		logits, _ = pipe(x, t, losses.cross_entropy, split_size=4)
		torch.cuda.synchronize()
		assert len(logits) == n and all(torch.equal(a, b) for a, b in zip(logits, alone))
