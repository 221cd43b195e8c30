"""The work users of this framework have it do, as a list of measurable cases.

Four kinds of case, each through the public entry points:

* ``stage``   the operation stream of one middle pipeline stage (``HipStageBlock`` driven by ``Engine.train_step``): forward,
              split backward, deferred weight gradients and gradient scale of every micro-batch, with the remat, lean-stash and
              offload options of the schedules; boundary tensors already on the GPU, as a pipeline's neighbours leave them;
* ``model``   a whole decoder through ``Pipeline``: token ids in, embedding, blocks, final norm, output head, cross-entropy,
              logits and every weight gradient out;
* ``layers``  the split backward of a generic module's linear layers (``AutogradStageBlock`` over ``LinearDW``);
* ``loss``    ``losses.cross_entropy`` as an ordinary differentiable function over logits of any vocabulary.

``listed()`` are fixed sizes, from a launch-bound toy to a 70B-shaped stage with activation offload; ``draw()`` gives more
sizes of the same ranges: widths, FFN sizes and layer sizes in steps of 64, sequences in steps of 128, one to eight
sequences per micro-batch with a shorter last one, any vocabulary."""

import math
import random

import torch
import torch.nn as nn

from elf_amd.benchmark_utils import get_checkpointed_scheduler, get_offloaded_scheduler
from elf_amd.execution import AutogradStageBlock, Engine, HipStageBlock
from elf_amd.losses import cross_entropy
from elf_amd.models import EndStage, LlamaBlock, StageModule, TransformerBlock
from elf_amd.partitioners.utils import sequential_signatures
from elf_amd.pipeline import Pipeline
from elf_amd.registry import COMM_SCHEDULERS, SCHEDULERS
from elf_amd.scheduling import add_comms

PLACEMENT = [0, 1, 2, 3]  # a stage's stream is block 1's of a four-stage pipeline: a middle stage
BLOCK_ID = 1
WEIGHT_STD = 0.02


def _llama(**kw):
	base = dict(kind="stage", arch="llama", blocks=1, d=4096, heads=32, kv_heads=8, head_dim=128, ffn=14336, seq=4096, mb=2, batch=8,
	            causal=True, scheduler="zbh1", remat="none", lean=0, offload=False)
	return dict(base, **kw)


def _gpt(**kw):
	base = dict(kind="stage", arch="gpt", blocks=3, d=768, heads=12, kv_heads=12, head_dim=64, ffn=3072, seq=1024, mb=8, batch=32,
	            causal=False, scheduler="1f1b", remat="none", lean=0, offload=False)
	return dict(base, **kw)


def listed():
	return [
		# the smallest stage of bench.py: every kernel is a few microseconds, the step is launches and host work
		_llama(name="stage_tiny", blocks=2, d=512, heads=4, kv_heads=2, ffn=768, seq=256, mb=2, batch=8),
		# the reference's own small decoder (4 layers of 256, vocabulary 1000, micro-batches of 4 x 128 tokens), two stages
		dict(name="decoder_small", kind="model", arch="gpt", stages=2, blocks=2, d=256, heads=4, kv_heads=4, head_dim=64, ffn=1024, seq=128,
		     mb=4, batch=32, vocab=1000, final_norm=False, scheduler="afab"),
		# an MLP that is no transformer block, at sizes no tile divides
		dict(name="mlp_odd", kind="layers", d_in=1600, d_hidden=4288, d_out=832, tokens=2112, n_mb=4, scheduler="zbh1"),
		# GPT-2-small stage, bidirectional attention, as bench.py runs it
		_gpt(name="gpt_small_stage"),
		# a GPT-2-small decoder with its vocabulary (50257 is odd: padded to 50304 = 393 x 128), head and loss
		dict(name="decoder_gpt_small", kind="model", arch="gpt", stages=1, blocks=3, d=768, heads=12, kv_heads=12, head_dim=64, ffn=3072, seq=1024,
		     mb=4, batch=8, vocab=50257, final_norm=True, scheduler="afab"),
		# a wider GPT stage whose width is no multiple of 256, sequences of 640 and a short last micro-batch
		_gpt(name="gpt_odd_stage", blocks=2, d=1600, heads=25, kv_heads=25, ffn=6400, seq=640, mb=3, batch=8, causal=True),
		# a 1B-class Llama stage: 2048 wide, FFN 5504
		_llama(name="llama_2k_stage", blocks=2, d=2048, heads=16, kv_heads=4, ffn=5504, seq=2048, mb=2, batch=8),
		# short ragged sequences through a Llama-3-8B-shaped block (fine-tuning on short samples), short last micro-batch
		_llama(name="llama_8b_short", seq=896, mb=3, batch=7, scheduler="1f1b"),
		# bench.py's headline stage, one block of it and four micro-batches
		_llama(name="llama_8b_stage"),
		# long sequences under a memory budget: full checkpointing over the lean stash
		_llama(name="llama_8b_long_remat", seq=8192, mb=1, batch=3, remat="full", lean=1, scheduler="1f1b"),
		# Llama-3-70B-shaped block with activation offload
		_llama(name="llama_70b_offload", d=8192, heads=64, ffn=28672, seq=8192, mb=1, batch=4, offload=True, scheduler="1f1b"),
		# the loss on its own: unpadded logits of a GPT-2 vocabulary straight out of a user's linear layer
		dict(name="loss_gpt_vocab", kind="loss", rows=2048, vocab=50257),
	]


# ------------------------------------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
	"""A whole number of [lo, hi], uniform over the logarithm."""
	return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _draw_blocks(rng, arch, d_max, tokens_max):
	if arch == "gpt":
		heads = _log(rng, 4, d_max // 64)
		shape = dict(d=64 * heads, heads=heads, kv_heads=heads, head_dim=64, ffn=64 * round(heads * rng.uniform(2, 4)))
	else:
		D = rng.choice([128, 128, 128, 64])
		kv = rng.choice([1, 2, 4, 8])
		groups = [g for g in (1, 2, 3, 4, 6, 8) if 512 <= g * kv * D <= d_max]
		heads = kv * rng.choice(groups or [max(1, 512 // (kv * D))])
		shape = dict(d=heads * D, heads=heads, kv_heads=kv, head_dim=D, ffn=64 * round(heads * D / 64 * rng.uniform(2, 3.5)))
	shape["seq"] = 128 * _log(rng, 1, min(64, tokens_max // 128))
	shape["mb"] = _log(rng, 1, max(1, min(8, tokens_max // shape["seq"])))
	return shape


def _draw_one(rng):
	pick = rng.random()
	if pick < 0.08:
		rows = _log(rng, 64, 8192)
		return dict(kind="loss", rows=rows, vocab=_log(rng, 1000, min(128256, 2**28 // rows)))
	if pick < 0.22:
		return dict(kind="layers", d_in=64 * _log(rng, 2, 96), d_hidden=64 * _log(rng, 4, 192), d_out=64 * _log(rng, 2, 96), tokens=64 * _log(rng, 2, 128),
		            n_mb=rng.randint(2, 4), scheduler=rng.choice(["1f1b", "zbh1"]))
	if pick < 0.4:
		arch = rng.choice(["gpt", "llama"])
		s = _draw_blocks(rng, arch, 2048, 8192)
		n = rng.randint(1, 4)
		return dict(kind="model", arch=arch, stages=rng.randint(1, 2), blocks=rng.randint(1, 2), vocab=_log(rng, 1000, 50257), final_norm=arch == "llama" or rng.random() < 0.5,
		            scheduler=rng.choice(["afab", "afab", "full_remat"]), batch=s["mb"] * n + rng.randrange(s["mb"]), **s)
	arch = "gpt" if pick < 0.62 else "llama"
	s = _draw_blocks(rng, arch, 2048 if arch == "gpt" else 8192, 16384)
	offload = arch == "llama" and rng.random() < 0.15
	remat = "none" if offload else rng.choice(["none", "none", "none", "selective", "simple" if arch == "gpt" else "full"])
	n = rng.randint(2, 4)
	return dict(kind="stage", arch=arch, blocks=rng.randint(1, 3), causal=arch == "llama" or rng.random() < 0.5, scheduler="1f1b" if offload else rng.choice(["1f1b", "zbh1", "afab"]),
	            remat=remat, lean=rng.choice([0, 0, 1, 2]), offload=offload, batch=s["mb"] * n + rng.randrange(s["mb"]), **s)


def draw(rng: random.Random):
	"""One more case of the ranges above, no dearer than the largest listed one."""
	most = max(work(c)["flops"] for c in listed())
	while True:
		case = _draw_one(rng)
		if work(case)["flops"] <= most:
			return case


# ------------------------------------------------------------------------------------------------ preparing
def _sizes(case):
	full, rest = divmod(case["batch"], case["mb"])
	return [case["mb"]] * full + ([rest] if rest else [])


def _init(module, gen):
	"""N(0, 0.02) weights and norm gains / shifts a little off 1 / 0, drawn on the GPU, in bf16.  The query and key projections
	are drawn wide enough for attention scores of unit spread at any width: heads that attend to something, as trained ones do
	(near-uniform attention would make the key and value gradients differences of almost equal sums)."""
	with torch.no_grad():
		for name, p in module.named_parameters():
			if p.dim() == 2:
				p.normal_(0.0, 1 / math.sqrt(p.shape[1]) if "q_proj" in name or "k_proj" in name else WEIGHT_STD, generator=gen)
			else:
				p.normal_(0.0, 0.1, generator=gen)
				if "norm" in name and name.endswith("weight"):
					p.add_(1.0)
	return module.to(torch.bfloat16)


def _chain(case):
	if case["arch"] == "llama":
		blocks = [LlamaBlock(case["d"], case["heads"], case["kv_heads"], case["ffn"], case["head_dim"]) for _ in range(case["blocks"])]
	else:
		blocks = [TransformerBlock(case["d"], case["heads"], case["ffn"], causal=case.get("causal", True)) for _ in range(case["blocks"])]
	return StageModule(blocks, case["seq"])


def _stream(case, n_mb):
	"""The stage's operation stream under the case's schedule."""
	sched = SCHEDULERS[case["scheduler"]]
	if case.get("offload"):
		sched = get_offloaded_scheduler(sched, 1)
	elif case.get("remat", "none") != "none":
		sched = get_checkpointed_scheduler(sched, case["remat"])
	ops = COMM_SCHEDULERS["pipelined"](add_comms(sched(PLACEMENT, n_mb), sequential_signatures(PLACEMENT)))
	return [op for op in ops if op.block_id == BLOCK_ID]


def _randn(gen, *shape):
	return torch.randn(*shape, device="cuda", generator=gen).to(torch.bfloat16)


def _tokens(gen, vocab, *shape):
	"""Token ids with the skew of text: uniform over the logarithm of the rank."""
	u = torch.rand(*shape, device="cuda", generator=gen)
	return (torch.exp(u * math.log(vocab)).long() - 1).clamp_(0, vocab - 1)


def prepare(case, seed):
	gen = torch.Generator(device="cuda").manual_seed(seed)
	kind = case["kind"]
	if kind == "loss":
		logits = (_randn(gen, case["rows"], case["vocab"]) * 4).requires_grad_(True)
		target = _tokens(gen, case["vocab"], case["rows"])
		target[torch.rand(case["rows"], device="cuda", generator=gen) < 0.05] = -100  # padding tokens
		return {"kind": kind, "logits": logits, "target": target}
	if kind == "model":
		with torch.device("cuda"):
			ends = [dict(vocab_in=case["vocab"] if i == 0 else None, vocab_out=case["vocab"] if i == case["stages"] - 1 else None) for i in range(case["stages"])]
			stages = [_init(EndStage(_chain(case), final_norm=bool(case["final_norm"] and e["vocab_out"]), **e), gen) for e in ends]
		ids = _tokens(gen, case["vocab"], case["batch"], case["seq"] + 1)
		pipe = Pipeline(stages, scheduler=case["scheduler"], partitioner=False, placement=[0] * case["stages"], mb_size=case["mb"])
		return {"kind": kind, "pipe": pipe, "ids": ids[:, :-1].contiguous(), "target": ids[:, 1:].contiguous(), "mb": case["mb"],
		        "params": list(pipe.named_parameters())}
	if kind == "layers":
		sizes = [1] * case["n_mb"]
		with torch.device("cuda"):
			module = _init(nn.Sequential(nn.Linear(case["d_in"], case["d_hidden"]), nn.GELU(), nn.Linear(case["d_hidden"], case["d_out"])), gen)
		block = AutogradStageBlock(module, BLOCK_ID, PLACEMENT, sequential_signatures(PLACEMENT)[BLOCK_ID])
		xs = [_randn(gen, case["tokens"], case["d_in"]) for _ in sizes]
		dys = [_randn(gen, case["tokens"], case["d_out"]) for _ in sizes]
	else:
		sizes = _sizes(case)
		with torch.device("cuda"):
			module = _init(_chain(case), gen)
		block = HipStageBlock(module, BLOCK_ID, PLACEMENT, sequential_signatures(PLACEMENT)[BLOCK_ID], mb_size=case["mb"], lean_stash=case["lean"])
		xs = [_randn(gen, n, case["seq"], case["d"]) for n in sizes]
		dys = [_randn(gen, n, case["seq"], case["d"]) for n in sizes]
	block.set_boundary(inputs=xs, grads=dys, keep_sent=True)
	return {"kind": kind, "block": block, "engine": Engine([block]), "stream": _stream(case, len(sizes)), "sizes": sizes,
	        "params": list(module.named_parameters())}


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
	kind = state["kind"]
	if kind == "loss":
		logits = state["logits"]
		logits.grad = None
		loss = cross_entropy(logits, state["target"])
		loss.backward()
		return {"loss": loss.detach(), "grad": logits.grad}
	if kind == "model":
		pipe = state["pipe"]
		pipe.zero_grad()
		logits, loss = pipe(state["ids"], state["target"], cross_entropy, split_size=state["mb"])
		return {"logits": list(logits), "loss": loss, "grads": [p.main_grad for _, p in state["params"]]}
	block = state["block"]
	block.zero_grad()
	state["engine"].train_step(None, None, None, state["stream"], state["sizes"])
	y, dx = block.sent_forward, block.sent_backward
	return {"y": [y[m] for m in sorted(y)], "dx": [dx[m] for m in sorted(dx)], "grads": [p.main_grad for _, p in state["params"]]}


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def work(case):
	kind = case["kind"]
	if kind == "loss":
		n = case["rows"] * case["vocab"]
		return {"bytes": 4 * n, "flops": 6 * n}  # logits read, gradient written; two exponentials' worth of arithmetic per logit
	if kind == "layers":
		params = case["d_in"] * case["d_hidden"] + case["d_hidden"] * case["d_out"]
		T = case["tokens"] * case["n_mb"]
		return {"bytes": 6 * params + 2 * T * 2 * (case["d_in"] + case["d_out"]), "flops": 6.0 * T * params}
	T, d, F = case["batch"] * case["seq"], case["d"], case["ffn"]
	nq, nkv = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
	per_block = d * (nq + 2 * nkv) + nq * d + d * F * (3 if case["arch"] == "llama" else 2)
	blocks = case["blocks"] * case.get("stages", 1)
	lin = 2.0 * T * per_block
	# attention: two products per direction and query-key pair forward, four backward; half of the pairs under a causal mask
	att = (2.0 if case.get("causal", True) else 4.0) * T * case["seq"] * nq
	remat = "full" if case["scheduler"] == "full_remat" else case.get("remat", "none")
	flops = blocks * (3 * (lin + att) + (lin + att if remat == "full" else att if remat == "selective" else 0.0))
	nbytes = blocks * per_block * (2 + 4)  # weights read, fp32 gradients written
	if kind == "model":
		V = case["vocab"]
		flops += 6.0 * T * d * V
		nbytes += d * V * (2 * 2 + 4 * 2) + 16 * T + 2 * T * V  # embedding and head with their gradients, ids and targets, logits
	else:
		nbytes += 4 * 2 * T * d  # boundary: x and dy read, y and dx written
	return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
	"""From the distance of each output to the same computation in PyTorch float32 on the same bf16 weights and inputs (36 listed
	and drawn cases, worst output of each): relative 2-norm 0.0031 for the single linear layers, 0.0028 for the loss gradient
	(one bf16 rounding), 0.005 to 0.012 for stages and decoders, which take some ten roundings to bf16 per block.  The bounds are
	about four times that, 0.03 at most.  Largest single differences seen: 0.004 of the value for the loss; of the root mean
	square 0.02 for the layers, 0.08 for stages and 0.65 for the embedding gradient, whose few frequent rows carry almost all of it."""
	if case["kind"] == "loss":
		return {"rel": 0.011, "max": 0.016}
	if case["kind"] == "layers":
		return {"rel": 0.0125, "max": 0.08}
	if case["kind"] == "model":
		return {"rel": 0.03, "max": 0.99}
	return {"rel": 0.03, "max": 0.35}
