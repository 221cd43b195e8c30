"""Parity of every HIP kernel (through the C ABI) against a plain PyTorch fp32 evaluation of
the same op on the same bf16-rounded inputs.  Tolerance: the path's bf16 bar (rel 2e-2 of the
reference's max magnitude per tensor), plus a much tighter Frobenius-norm bound that catches
systematic errors (a dropped term, a wrong sign or index)."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

REL_MAX = 2e-2   # elementwise, relative to max |ref|
REL_FRO = 6e-3   # Frobenius, bf16 output rounding is ~2^-9 relative


def _close(got, ref, rel_max=REL_MAX, rel_fro=REL_FRO, what=""):
	got = got.float()
	ref = ref.float()
	assert got.shape == ref.shape, f"{what}: shape {got.shape} vs {ref.shape}"
	assert torch.isfinite(got).all(), f"{what}: non-finite output"
	scale = ref.abs().max().item() + 1e-12
	err = (got - ref).abs().max().item()
	fro = ((got - ref).norm() / (ref.norm() + 1e-12)).item()
	assert err <= rel_max * scale, f"{what}: max err {err:.4g} vs scale {scale:.4g}"
	assert fro <= rel_fro, f"{what}: relative Frobenius error {fro:.4g}"


def _randn(*shape, seed=0, scale=1.0):
	g = torch.Generator(device="cpu").manual_seed(seed)
	return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16).cuda()


@pytest.fixture(scope="module")
def K():
	from elf_amd import kernels

	return kernels


@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
@pytest.mark.parametrize("shape", [(256, 256, 64), (512, 768, 256), (1024, 2304, 768), (2048, 1024, 4096)])
@pytest.mark.parametrize("tile_cfg", [0, 1, 2, 3, 5, 7, 8])
def test_gemm_layouts(K, layout, shape, tile_cfg):
	M, N, Kd = shape
	if tile_cfg in (1, 5, 7) and (M % 256 or N % 256):
		pytest.skip("tile does not divide")
	if tile_cfg == 8 and N % 256:
		pytest.skip("the 128x256 direct-to-LDS tile needs N % 256 == 0")
	A = _randn(M, Kd, seed=1)
	B = _randn(N, Kd, seed=2, scale=0.05)
	ref = A.float() @ B.float().t()
	if layout == "nt":
		out = K.gemm(A, B, tile_cfg=tile_cfg)
	elif layout == "nn":
		out = K.gemm(A, B.t().contiguous(), b_t=True, tile_cfg=tile_cfg)
	else:
		out = K.gemm(A.t().contiguous(), B.t().contiguous(), a_t=True, b_t=True, tile_cfg=tile_cfg)
	_close(out, ref, what=f"gemm {layout} {shape} cfg{tile_cfg}")


def test_gemm_epilogues(K):
	M, N, Kd = 512, 768, 512
	A = _randn(M, Kd, seed=3)
	B = _randn(N, Kd, seed=4, scale=0.05)
	R = _randn(M, N, seed=5)
	ref = A.float() @ B.float().t()
	_close(K.gemm(A, B, epilogue=K.EPI_BF16_RESID, residual=R), ref + R.float(), what="resid")
	_close(K.gemm(A, B, epilogue=K.EPI_F32_STORE), ref, rel_fro=1e-5, rel_max=1e-5, what="f32 store")
	# fp32 accumulation across calls (the deferred weight-gradient pattern), with and without split-K
	for ks in (1, 4):
		acc = torch.full((M, N), 0.25, dtype=torch.float32, device="cuda")
		for _ in range(3):
			K.gemm(A, B, out=acc, epilogue=K.EPI_F32_ACC, k_splits=ks)
		_close(acc, 3 * ref + 0.25, rel_fro=1e-5, rel_max=1e-5, what=f"f32 acc ks={ks}")


@pytest.mark.parametrize("tile_cfg", [7, 8])
@pytest.mark.parametrize("layout", ["nt", "tn", "nn"])
def test_gemm_direct_to_lds_epilogues_and_k_split(K, tile_cfg, layout):
	"""The direct-to-LDS kernels (256x256 and 128x256 tiles): every epilogue, short K (1 and
	2 slices: the loop's loads past the end of K), and the K split with fp32 atomics."""
	M, N = (384, 768) if tile_cfg == 8 else (512, 768)
	for Kd in (64, 128, 1024):
		A = _randn(M, Kd, seed=21)
		B = _randn(N, Kd, seed=22, scale=0.05)
		R = _randn(M, N, seed=23)
		ref = A.float() @ B.float().t()
		if layout == "nt":
			kw = dict(tile_cfg=tile_cfg)
			a, b = A, B
		elif layout == "nn":
			kw = dict(tile_cfg=tile_cfg, b_t=True)
			a, b = A, B.t().contiguous()
		else:
			kw = dict(tile_cfg=tile_cfg, a_t=True, b_t=True)
			a, b = A.t().contiguous(), B.t().contiguous()
		_close(K.gemm(a, b, **kw), ref, what=f"bf16 K={Kd}")
		_close(K.gemm(a, b, epilogue=K.EPI_BF16_RESID, residual=R, **kw), ref + R.float(), what=f"resid K={Kd}")
		_close(K.gemm(a, b, epilogue=K.EPI_F32_STORE, **kw), ref, rel_fro=1e-5, rel_max=1e-5, what=f"f32 store K={Kd}")
		for ks in (1, 2, 4):
			acc = torch.full((M, N), 0.25, dtype=torch.float32, device="cuda")
			for _ in range(2):
				K.gemm(a, b, out=acc, epilogue=K.EPI_F32_ACC, k_splits=ks, **kw)
			_close(acc, 2 * ref + 0.25, rel_fro=1e-5, rel_max=1e-5, what=f"f32 acc K={Kd} ks={ks}")


@pytest.mark.parametrize("dims,ks", [((1024, 1536, 8192), 0), ((768, 768, 8192), 0), ((2304, 768, 8192), 0), ((2048, 2048, 4096), 0), ((512, 768, 4096), 8), ((4096, 6144, 8192), 0), ((2048, 2304, 2048), 4)])
def test_gemm_k_split_is_bit_reproducible(K, dims, ks):
	"""Weight-gradient GEMMs whose tiles are shared by several workgroups along K (all tiles split, only the
	tail of the last round split, an explicit split): the workgroups of a tile add in turn, so repeated runs
	into equal accumulators give equal bits, and the sum is the unsplit one within fp32 rounding."""
	M, N, Kd = dims
	A = _randn(Kd, M, seed=71)
	B = _randn(Kd, N, seed=72, scale=0.05)
	start = torch.randn(M, N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(73))
	runs = []
	for _ in range(4):
		acc = start.clone()
		K.gemm(A, B, a_t=True, b_t=True, out=acc, epilogue=K.EPI_F32_ACC, k_splits=ks)
		runs.append(acc)
	for r in runs[1:]:
		assert torch.equal(r, runs[0]), "split-K accumulation must not depend on the order in which workgroups finish"
	one = start.clone()
	K.gemm(A, B, a_t=True, b_t=True, out=one, epilogue=K.EPI_F32_ACC, k_splits=1)
	assert ((runs[0] - one).norm() / one.norm()).item() <= 1e-5


@pytest.mark.parametrize("shape", [(256, 256, 128), (512, 768, 256), (4096, 1280, 1152), (8192, 4096, 1024), (2048, 28672, 256), (4352, 4352, 320), (4352, 8704, 448)])
def test_persistent_forward_gemm_equals_the_tile_kernel_bit_for_bit(K, monkeypatch, shape):
	"""Forward GEMMs on 256x256 tiles run as persistent workgroups that walk several tiles and store from registers
	(operands swapped on the MFMA, permuted weight rows); the one-tile-per-workgroup kernel with its LDS-staged epilogue
	(ELF_NO_PERSISTENT_GEMM=1) forms the same products in the same order: equal bits for every epilogue, from one tile
	per workgroup (1, 6 tiles) to several with a ragged last round (80, 512, 896 tiles; 289 and 578 with an odd number of K slices: the
	ring starts every other tile in its other half), also against fp32 torch."""
	M, N, Kd = shape
	a, w, r, bias = _randn(M, Kd, seed=61), _randn(N, Kd, seed=62, scale=0.05), _randn(M, N, seed=63), _randn(1, N, seed=64)
	F = N // 2
	S, D = 256, 128
	cs = K.rope_table(S, D, 5e5)
	n_rot = (N // D) // 2

	def run():
		return (K.gemm(a, w, tile_cfg=7), K.gemm(a, w, tile_cfg=7, epilogue=K.EPI_BF16_RESID, residual=r),
		        K.gemm(a, w, tile_cfg=7, epilogue=K.EPI_BF16_RESID, residual=bias, residual_ld=0), *K.gemm_act(a, w, K.ACT_SWIGLU), K.gemm_rope(a, w, cs, S, n_rot, D))

	new = run()
	monkeypatch.setenv("ELF_NO_PERSISTENT_GEMM", "1")
	old = run()
	monkeypatch.delenv("ELF_NO_PERSISTENT_GEMM")
	for i, (x, y) in enumerate(zip(new, old)):
		assert torch.equal(x, y), f"output {i} of the persistent kernel differs from the tile kernel's at {shape}"
	ref = a.float() @ w.float().t()
	_close(new[0], ref, what="persistent bf16")
	_close(new[1], ref + r.float(), what="persistent residual")
	_close(new[2], ref + bias.float(), what="persistent bias row")
	_close(new[4], torch.nn.functional.silu(new[3][:, :F].float()) * new[3][:, F:].float(), what="persistent swiglu")


@pytest.mark.parametrize("layout", ["nt", "nn", "tn"])
@pytest.mark.parametrize("tile_cfg,shape", [
	(7, (256, 320, 64)), (7, (320, 256, 192)), (7, (1984, 576, 128)), (8, (128, 256, 64)), (8, (192, 448, 320)),
	(9, (128, 128, 64)), (9, (192, 320, 192)), (9, (832, 1600, 320)), (10, (64, 192, 448)), (11, (192, 64, 448)), (12, (64, 64, 64)), (12, (192, 128, 1088)),
	(0, (64, 64, 64)), (0, (576, 832, 192)), (0, (1088, 3136, 128)),
])
def test_gemm_ragged_sizes_on_every_tile(K, tile_cfg, shape, layout):
	"""Sizes that are multiples of 64 but not of the tile (the last tile moves back over its neighbour's rows or columns), down
	to the smallest a tile takes, with fewer and more K slices than the ring holds: every epilogue, and a K split with more
	splits than slices.  Bounds: one bf16 rounding of the fp32 sum for bf16 outputs, fp32 summation for the others."""
	M, N, Kd = shape
	A, B, R, bias = _randn(M, Kd, seed=31), _randn(N, Kd, seed=32, scale=0.05), _randn(M, N, seed=33), _randn(1, N, seed=34)
	ref = A.float() @ B.float().t()
	a, b, kw = {"nt": (A, B, {}), "nn": (A, B.t().contiguous(), dict(b_t=True)), "tn": (A.t().contiguous(), B.t().contiguous(), dict(a_t=True, b_t=True))}[layout]
	kw["tile_cfg"] = tile_cfg
	big = torch.full((M + 64, N + 64), 7.0, dtype=torch.bfloat16, device="cuda")  # what lies around the output stays untouched
	K.gemm(a, b, out=big[:M, :N], **kw)
	_close(big[:M, :N], ref, what="bf16")
	assert (big[M:] == 7).all() and (big[:, N:] == 7).all()
	assert torch.equal(K.gemm(a, b, **kw), big[:M, :N])
	_close(K.gemm(a, b, epilogue=K.EPI_BF16_RESID, residual=R, **kw), ref + R.float(), what="resid")
	_close(K.gemm(a, b, epilogue=K.EPI_BF16_RESID, residual=bias, residual_ld=0, **kw), ref + bias.float(), what="bias")
	_close(K.gemm(a, b, epilogue=K.EPI_F32_STORE, **kw), ref, rel_fro=1e-5, rel_max=1e-5, what="f32 store")
	before = K.gemm_turn_giveups()
	for ks in (0, 1, 3, 20):
		acc = torch.full((M, N), 0.25, dtype=torch.float32, device="cuda")
		for _ in range(2):
			K.gemm(a, b, out=acc, epilogue=K.EPI_F32_ACC, k_splits=ks, **kw)
		_close(acc, 2 * ref + 0.25, rel_fro=1e-5, rel_max=1e-5, what=f"f32 acc ks={ks}")
	assert K.gemm_turn_giveups() == before, "every split finds its predecessor's turn"


def test_gemm_bits_do_not_depend_on_the_tile(K):
	"""Every tile adds an output's products in the same order: equal bits from all of them, ragged tiles included."""
	A, B = _randn(320, 704, seed=41), _randn(448, 704, seed=42, scale=0.05)
	for kw, a, b in (({}, A, B), (dict(b_t=True), A, B.t().contiguous())):
		want = K.gemm(a, b, tile_cfg=7, **kw)
		for cfg in (8, 9, 10, 11, 12):
			assert torch.equal(K.gemm(a, b, tile_cfg=cfg, **kw), want), f"tile config {cfg} {kw}"


@pytest.mark.parametrize("M,N,Kd", [(2112, 3968, 320), (2624, 4160, 320), (2624, 4160, 448), (4096, 3072, 2048), (896, 14336, 512)])
def test_gemm_tiles_between_128_and_256_rows(K, M, N, Kd):
	"""Sizes around those of the tiles of 160, 192 and 224 rows (the last takes 256-row ones; which takes which is pinned in
	test_gemm_every_epilogue_of_the_tiles_between_128_and_256_rows), with moved last tiles that end inside a wave's 32-row strip, and
	fewer and more K slices than a turn of the ring: the bits of the 64x64 tile for every epilogue (all tiles add the products in
	the same order), nothing written outside the output."""
	a, w, r, bias = _randn(M, Kd, seed=71), _randn(N, Kd, seed=72, scale=0.05), _randn(M, N, seed=73), _randn(1, N, seed=74)
	for kw, b in ((dict(), w), (dict(b_t=True), w.t().contiguous())):
		want = K.gemm(a, b, tile_cfg=12, **kw)
		big = torch.full((M + 64, N + 64), 7.0, dtype=torch.bfloat16, device="cuda")
		K.gemm(a, b, out=big[:M, :N], **kw)
		assert torch.equal(big[:M, :N], want) and (big[M:] == 7).all() and (big[:, N:] == 7).all()
		for res in (dict(residual=r), dict(residual=bias, residual_ld=0)):
			assert torch.equal(K.gemm(a, b, epilogue=K.EPI_BF16_RESID, **res, **kw), K.gemm(a, b, epilogue=K.EPI_BF16_RESID, tile_cfg=12, **res, **kw))
	S, D = 64, 128 if N % 128 == 0 else 64
	cs, n_rot = K.rope_table(S, D, 5e5), N // D // 2
	assert torch.equal(K.gemm_rope(a, w, cs, S, n_rot, D), K.gemm_rope(a, w, cs, S, n_rot, D, fused=False))
	if N % 128 == 0:
		gu, act = K.gemm_act(a, w, K.ACT_SWIGLU)
		assert torch.equal(gu, K.gemm(a, w, tile_cfg=12)) and torch.equal(act, K.swiglu_fwd(gu))
	g, wt = _randn(M, 2 * N, seed=75), w.t().contiguous()
	assert torch.equal(K.gemm_swiglu_bwd(a, wt, g), K.gemm_swiglu_bwd(a, wt, g, fused=False))


MID_TILES = [  # rows of the tile, product, M, N, K: moved last tiles in rows, in columns or both, 5, 7 and more K slices
	*[(160, w, *s) for w in ("forward", "dx", "rope") for s in ((6592, 1088, 320), (6656, 1088, 448), (1216, 6656, 512))],
	*[(192, w, *s) for w in ("forward", "dx", "rope") for s in ((6784, 1344, 320), (6784, 1344, 448), (1792, 5632, 512))],
	*[(224, w, *s) for w in ("forward", "dx", "rope") for s in ((6976, 1600, 2048), (6976, 1600, 2112), (1984, 6144, 2048))],
	(160, "swiglu", 576, 6592, 320), (160, "swiglu", 576, 6592, 448), (160, "swiglu", 576, 6656, 512),
	(192, "swiglu", 832, 5440, 320), (192, "swiglu", 832, 5568, 448), (192, "swiglu", 704, 6656, 512),
	(224, "swiglu", 832, 6592, 2048), (224, "swiglu", 832, 6592, 2112), (224, "swiglu", 832, 6656, 2048),
	(160, "swiglu_bwd", 6784, 1088, 320), (160, "swiglu_bwd", 5504, 1344, 448), (160, "swiglu_bwd", 1216, 6656, 512),
	(192, "swiglu_bwd", 6784, 1344, 320), (192, "swiglu_bwd", 6784, 1344, 448), (192, "swiglu_bwd", 1792, 5632, 512),
	(224, "swiglu_bwd", 6976, 1600, 1088), (224, "swiglu_bwd", 4864, 2368, 1536), (224, "swiglu_bwd", 2368, 5120, 1088),
]


@pytest.mark.parametrize("rows,product,M,N,Kd", MID_TILES)
def test_gemm_every_epilogue_of_the_tiles_between_128_and_256_rows(K, rows, product, M, N, Kd):
	"""Every epilogue on tiles of 160, 192 and 224 rows (the rule is asked first whether the size goes there): the bits of the
	64x64 tile followed by the pass of its own, nothing written outside a plain output."""
	D = 128 if N % 128 == 0 else 64
	way = {"forward": K.WAY_FORWARD, "dx": K.WAY_INPUT_GRADIENT, "rope": K.WAY_ROPE, "swiglu": K.WAY_SWIGLU, "swiglu_bwd": K.WAY_SWIGLU_BWD}[product]
	assert K.gemm_way(way, M, N, Kd, D) == (rows, 256)
	a, w = _randn(M, Kd, seed=76), _randn(2 * N if product == "swiglu" else N, Kd, seed=77, scale=0.05)
	if product in ("forward", "dx"):
		kw, b = (dict(), w) if product == "forward" else (dict(b_t=True), w.t().contiguous())
		big = torch.full((M + 64, N + 64), 7.0, dtype=torch.bfloat16, device="cuda")
		K.gemm(a, b, out=big[:M, :N], **kw)
		assert torch.equal(big[:M, :N], K.gemm(a, b, tile_cfg=12, **kw)) and (big[M:] == 7).all() and (big[:, N:] == 7).all()
		for res in (dict(residual=_randn(M, N, seed=78)), dict(residual=_randn(1, N, seed=79), residual_ld=0)):
			assert torch.equal(K.gemm(a, b, epilogue=K.EPI_BF16_RESID, **res, **kw), K.gemm(a, b, epilogue=K.EPI_BF16_RESID, tile_cfg=12, **res, **kw))
	elif product == "rope":
		cs, n_rot = K.rope_table(64, D, 5e5), N // D // 2
		assert torch.equal(K.gemm_rope(a, w, cs, 64, n_rot, D), K.rope_apply_(K.gemm(a, w, tile_cfg=12), cs, 64, n_rot, D))
	elif product == "swiglu":
		gu, act = K.gemm_act(a, w, K.ACT_SWIGLU)
		assert torch.equal(gu, K.gemm(a, w, tile_cfg=12)) and torch.equal(act, K.swiglu_fwd(gu))
	else:
		g, wt = _randn(M, 2 * N, seed=75), w.t().contiguous()
		assert torch.equal(K.gemm_swiglu_bwd(a, wt, g), K.swiglu_bwd(K.gemm(a, wt, b_t=True, tile_cfg=12), g))


@pytest.mark.parametrize("product", ["forward", "dx"])
@pytest.mark.parametrize("M,N,Kd", [(448, 9984, 512), (576, 8576, 512), (576, 8000, 512), (832, 5504, 512), (448, 9728, 512), (1088, 3968, 512), (576, 7232, 512), (576, 8128, 512)])
def test_gemm_tiles_of_192_columns_in_any_number(K, product, M, N, Kd):
	"""Tiles that 8 XCDs share with each remainder: every tile once, the bits of the 64x64 tile, nothing written outside the output."""
	assert K.gemm_way(K.WAY_FORWARD if product == "forward" else K.WAY_INPUT_GRADIENT, M, N, Kd) == (128, 192)
	a, w = _randn(M, Kd, seed=80), _randn(N, Kd, seed=81, scale=0.05)
	kw, b = (dict(), w) if product == "forward" else (dict(b_t=True), w.t().contiguous())
	big = torch.full((M + 64, N + 64), 7.0, dtype=torch.bfloat16, device="cuda")
	K.gemm(a, b, out=big[:M, :N], **kw)
	assert torch.equal(big[:M, :N], K.gemm(a, b, tile_cfg=12, **kw)) and (big[M:] == 7).all() and (big[:, N:] == 7).all()


def _guarded(*shape):
	"""A dense bf16 tensor with 4096 marked elements before and behind it, and the whole."""
	n = int(torch.Size(shape).numel())
	whole = torch.full((n + 8192,), 7.0, dtype=torch.bfloat16, device="cuda")
	return whole[4096 : 4096 + n].view(*shape), whole


@pytest.mark.parametrize("M,F,Kd", [(64, 64, 256), (64, 192, 320), (512, 1024, 256), (512, 768, 512), (320, 448, 1088)])
def test_epilogues_of_the_64x64_tile(K, M, F, Kd):
	"""The activations, their backwards and the rotary embedding on 64x64 tiles (the rule is asked first), on the ring of two slices (K = 256)
	and with fewer and more slices than the long one holds: the bits of the product followed by the pass of its own, nothing
	written before or behind an output."""
	from elf_amd import _lib

	lib, p, st = _lib.load(), lambda t: t.data_ptr(), _lib.raw_stream()
	a, w, w2, wt = _randn(M, Kd, seed=81), _randn(F, Kd, seed=82, scale=0.1), _randn(2 * F, Kd, seed=83, scale=0.1), _randn(Kd, F, seed=85, scale=0.1)
	for way, n in ((K.WAY_GELU, F), (K.WAY_GELU_BWD, F), (K.WAY_SWIGLU, F), (K.WAY_SWIGLU_BWD, F), (K.WAY_ROPE, 2 * F)):
		assert K.gemm_way(way, M, n, Kd) == (64, 64), way
	plain, d = K.gemm(a, w, tile_cfg=12), K.gemm(a, wt, b_t=True, tile_cfg=12)
	pre, gu = _randn(M, F, seed=86), _randn(M, 2 * F, seed=84)

	def check(outs, want, call):
		views, wholes = zip(*[_guarded(*o) for o in outs])
		_lib.check(call(*views), "call")
		for v, whole, x in zip(views, wholes, want):
			assert torch.equal(v, x)
			assert (whole[:4096] == 7).all() and (whole[-4096:] == 7).all()

	check([(M, F), (M, F)], [plain, K.gelu_fwd(plain)], lambda o, o2: lib.elf_gemm_act_bf16(K.ACT_GELU, M, F, Kd, p(a), Kd, p(w), Kd, p(o), F, p(o2), F, st))
	plain2 = K.gemm(a, w2, tile_cfg=12)
	check([(M, 2 * F), (M, F)], [plain2, K.swiglu_fwd(plain2)], lambda o, o2: lib.elf_gemm_act_bf16(K.ACT_SWIGLU, M, F, Kd, p(a), Kd, p(w2), Kd, p(o), 2 * F, p(o2), F, st))
	scratch = torch.empty_like(pre)
	check([(M, F)], [K.gelu_bwd(d, pre)], lambda o: lib.elf_gemm_gelu_bwd_bf16(M, F, Kd, p(a), p(wt), p(pre), p(o), p(scratch), st))
	check([(M, 2 * F)], [K.swiglu_bwd(d, gu)], lambda o: lib.elf_gemm_swiglu_bwd_bf16(M, F, Kd, p(a), Kd, p(wt), F, p(gu), 2 * F, p(o), 2 * F, p(scratch), st))
	cs, heads = K.rope_table(64, 64, 5e5), 2 * F // 64
	want = K.rope_apply_(plain2.clone(), cs, 64, heads // 2, 64)
	check([(M, 2 * F)], [want], lambda o: lib.elf_gemm_rope_bf16(M, 2 * F, Kd, p(a), Kd, p(w2), Kd, p(o), 2 * F, p(cs), 64, heads // 2, 64, st))


@pytest.mark.parametrize("M,F,Kd", [(256, 512, 64), (1024, 4096, 512), (2048, 3072, 768)])
def test_gelu_backward_of_larger_products_is_a_pass_of_its_own(K, M, F, Kd):
	dy, w2, pre = _randn(M, Kd, seed=87), _randn(Kd, F, seed=88, scale=0.1), _randn(M, F, seed=89)
	assert K.gemm_way(K.WAY_GELU_BWD, M, F, Kd) == (0, 0)
	assert torch.equal(K.gemm_gelu_bwd(dy, w2, pre), K.gemm_gelu_bwd(dy, w2, pre, fused=False))


@pytest.mark.parametrize("M,F,Kd", [(64, 64, 256), (128, 192, 320), (512, 768, 512), (1024, 640, 256), (320, 448, 1088)])
def test_small_products_with_their_activation_in_one_kernel(K, M, F, Kd):
	"""Products that go to 64x64 tiles with the activation, its backward or the rotary embedding in the epilogue (both rings of
	slices): the bits of the plain product followed by the pass of its own."""
	a, w, w2 = _randn(M, Kd, seed=81), _randn(F, Kd, seed=82, scale=0.1), _randn(2 * F, Kd, seed=83, scale=0.1)
	pre, act = K.gemm_act(a, w, K.ACT_GELU)
	assert torch.equal(pre, K.gemm(a, w, tile_cfg=12)) and torch.equal(act, K.gelu_fwd(pre))
	gu, act = K.gemm_act(a, w2, K.ACT_SWIGLU)
	assert torch.equal(gu, K.gemm(a, w2, tile_cfg=12)) and torch.equal(act, K.swiglu_fwd(gu))
	g, wt = _randn(M, 2 * F, seed=84), w.t().contiguous()
	assert torch.equal(K.gemm_swiglu_bwd(a, wt, g), K.swiglu_bwd(K.gemm(a, wt, b_t=True, tile_cfg=12), g))
	for D in (64, 128):
		if 2 * F % D == 0:
			cs, heads = K.rope_table(64, D, 5e5), 2 * F // D
			for n_rot in (0, heads // 2, heads):
				assert torch.equal(K.gemm_rope(a, w2, cs, 64, n_rot, D), K.gemm_rope(a, w2, cs, 64, n_rot, D, fused=False) if n_rot else K.gemm(a, w2, tile_cfg=12)), (D, n_rot)


@pytest.mark.parametrize("Kd", [64, 320, 512, 1088])
@pytest.mark.parametrize("shapes", [[(256, 256)], [(512, 768), (1536, 512), (512, 512), (1024, 512)], [(256, 1024)] * 16])
def test_weight_gradients_of_small_stages_in_one_launch(K, shapes, Kd):
	"""Groups of no more than a round of 128x128 tiles (one problem of the smallest size, one to sixteen, K slices fewer and more
	than the ring holds): the bits of a launch per layer without a K split, and of that followed by the gradient scale."""
	dy = [_randn(Kd, M, seed=91 + i) for i, (M, N) in enumerate(shapes)]
	x = [_randn(Kd, N, seed=191 + i) for i, (M, N) in enumerate(shapes)]
	start = [torch.randn(M, N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(291 + i)) for i, (M, N) in enumerate(shapes)]
	want = [s.clone() for s in start]
	for d, a, w in zip(dy, x, want):
		K.gemm(d, a, a_t=True, b_t=True, out=w, epilogue=K.EPI_F32_ACC, tile_cfg=12, k_splits=1)
	got = [s.clone() for s in start]
	K.gemm_dw_group(list(zip(dy, x, got)))
	assert all(torch.equal(g, w) for g, w in zip(got, want))
	got, bf = [s.clone() for s in start], [torch.empty(M, N, dtype=torch.bfloat16, device="cuda") for M, N in shapes]
	K.gemm_dw_group(list(zip(dy, x, got, bf)), scale=0.375)
	for g, b, w in zip(got, bf, want):
		assert torch.equal(g, w * 0.375) and torch.equal(b, (w * 0.375).to(torch.bfloat16))


@pytest.mark.parametrize("shape", [(64, 64, 15424), (256, 704, 14080), (512, 384, 10112), (1536, 192, 12608), (64, 5632, 13696), (128, 256, 192)])
def test_small_weight_gradients_are_split_along_the_tokens(K, shape):
	"""Outputs too small for the chip with long reductions: the choice left open runs about as fast as the best of a few explicit
	splits of the small tiles (2.5 times as long without a split), with fp32 sums and equal bits from run to run."""
	M, N, Kd = shape
	A, B = _randn(Kd, M, seed=61), _randn(Kd, N, seed=62, scale=0.05)
	before = K.gemm_turn_giveups()
	acc = [K.gemm(A, B, a_t=True, b_t=True, epilogue=K.EPI_F32_ACC) for _ in range(2)]
	assert torch.equal(acc[0], acc[1]) and K.gemm_turn_giveups() == before
	_close(acc[0], A.float().t() @ B.float(), rel_fro=1e-5, rel_max=1e-5, what=f"weight gradient {shape}")
	if Kd < 4096:
		return

	def ms(**kw):
		times = []
		for _ in range(5):
			e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
			e0.record()
			for _ in range(20):
				K.gemm(A, B, a_t=True, b_t=True, out=acc[0], epilogue=K.EPI_F32_ACC, **kw)
			e1.record()
			e1.synchronize()
			times.append(e0.elapsed_time(e1))
		return sorted(times)[2]

	best = min(ms(tile_cfg=12, k_splits=ks) for ks in (1, 2, 3, 4))
	assert ms() < 1.6 * best


def test_gemm_with_activation_whose_up_rows_lie_far_off(K):
	"""A weight whose up rows start 1.3 GB behind the gate rows, too far for the fused epilogue: the separate passes."""
	M, F, Kd, ldw = 192, 320, 64, 1 << 21
	a = _randn(M, Kd, seed=87)
	w = torch.empty(2 * F, ldw, dtype=torch.bfloat16, device="cuda")[:, :Kd]
	w.copy_(_randn(2 * F, Kd, seed=88, scale=0.05))
	gu, act = K.gemm_act(a, w, K.ACT_SWIGLU)
	assert torch.equal(gu, K.gemm(a, w.contiguous())) and torch.equal(act, K.swiglu_fwd(gu))


def test_gemm_takes_any_tile_choice_below_one_as_open(K):
	A, B = _randn(192, 128, seed=85), _randn(320, 128, seed=86, scale=0.05)
	assert torch.equal(K.gemm(A, B, tile_cfg=-1), K.gemm(A, B))
	acc = K.gemm(A, B, tile_cfg=-1, k_splits=-1, epilogue=K.EPI_F32_ACC)
	_close(acc, A.float() @ B.float().t(), rel_fro=1e-5, rel_max=1e-5, what="f32 acc")


@pytest.mark.parametrize("layout", ["nt", "nn"])
@pytest.mark.parametrize("Kd", [64, 128, 192, 256, 320])
@pytest.mark.parametrize("tile_cfg,mn", [(9, (448, 320)), (10, (192, 320)), (11, (320, 192)), (12, (192, 64))])
def test_short_reductions_on_the_small_tiles(K, tile_cfg, mn, Kd, layout):
	"""K of 64 to 256 runs on a ring of two slices, K of 320 on the deep one: the bits of the 64x64 tile's fp32 sums, rounded once."""
	M, N = mn
	A, B, R = _randn(M, Kd, seed=81), _randn(N, Kd, seed=82, scale=0.05), _randn(M, N, seed=83)
	b, kw = (B, {}) if layout == "nt" else (B.t().contiguous(), dict(b_t=True))
	want = K.gemm(A, b, epilogue=K.EPI_F32_STORE, tile_cfg=12, **kw)
	_close(want, A.float() @ B.float().t(), rel_fro=1e-5, rel_max=1e-5, what="f32 store")
	big = torch.full((M + 64, N + 64), 7.0, dtype=torch.bfloat16, device="cuda")
	K.gemm(A, b, out=big[:M, :N], tile_cfg=tile_cfg, **kw)
	assert torch.equal(big[:M, :N], want.to(torch.bfloat16)) and (big[M:] == 7).all() and (big[:, N:] == 7).all()
	assert torch.equal(K.gemm(A, b, epilogue=K.EPI_BF16_RESID, residual=R, tile_cfg=tile_cfg, **kw), (want + R.float()).to(torch.bfloat16))


PROF_ACT_FWD, PROF_ACT_BWD, PROF_ROPE = 5, 6, 7


def _launches(kind, call):
	"""``call()`` and how many kernels of a family (``elf_prof_launches``) it ran: none where a fused epilogue did the work."""
	from elf_amd import _lib

	lib = _lib.load()
	lib.elf_prof_enable(1)
	try:
		return call(), lib.elf_prof_launches(kind, None)
	finally:
		lib.elf_prof_enable(0)


@pytest.mark.parametrize("dims,fused", [((1024, 3072, 64), False), ((8448, 512, 512), False), ((3072, 2304, 768), False), ((8192, 7168, 512), True), ((4096, 4096, 4096), True)])
def test_swiglu_backward_is_fused_where_that_is_faster(K, dims, fused):
	"""The epilogue of a 256x256 tile takes 27 us a round: one partly filled round of few K slices is faster apart (1024 x 3072 x 64:
	13 us against 25), full rounds are faster fused (8192 x 14336 x 4096: 842 us against 932)."""
	M, F, Kd = dims
	dy, w2, gu = _randn(M, Kd, seed=71), _randn(Kd, F, seed=72, scale=0.05), _randn(M, 2 * F, seed=73)
	got, passes = _launches(PROF_ACT_BWD, lambda: K.gemm_swiglu_bwd(dy, w2, gu))
	assert (passes == 0) == fused
	assert torch.equal(got, K.gemm_swiglu_bwd(dy, w2, gu, fused=False))


@pytest.mark.parametrize("dims", [(4160, 5504, 128), (2880, 2880, 64), (320, 320, 128)])
def test_fused_epilogues_at_ragged_sizes_equal_the_separate_passes(K, dims):
	"""SwiGLU forward and backward and the rotary embedding in the GEMM epilogue on tiles that move back at the matrix's
	edges (and at sizes where the separate passes are taken): the bits of the GEMM followed by the pass."""
	T, F, Kd = dims
	S, D = 64, 64
	a, w, w2 = _randn(T, Kd, seed=51), _randn(2 * F, Kd, seed=52, scale=0.05), _randn(Kd, F, seed=53, scale=0.05)
	gu, act = K.gemm_act(a, w, K.ACT_SWIGLU)
	assert torch.equal(gu, K.gemm(a, w)) and torch.equal(act, K.swiglu_fwd(gu))
	dy = _randn(T, Kd, seed=54)
	assert torch.equal(K.gemm_swiglu_bwd(dy, w2, gu), K.gemm_swiglu_bwd(dy, w2, gu, fused=False))
	cs = K.rope_table(S, D, 1e4)
	n_rot = F // D - 1
	assert torch.equal(K.gemm_rope(a, w[:F], cs, S, n_rot, D), K.gemm_rope(a, w[:F], cs, S, n_rot, D, fused=False))


# (tokens, F, K), the head width, and whether the epilogue runs in the GEMM.  1984 x 3200 x 512: 208 tiles of 128x256, the last ones
# moved back by 64 rows and 128 columns (two heads of 64 or one of 128); 4160 x 11136 x 128: 256x256, moved back by 192 rows and 128 columns
@pytest.mark.parametrize("dims,D,fused", [((1984, 1600, 512), 64, True), ((1984, 1600, 512), 128, True), ((4160, 5568, 128), 128, True), ((320, 320, 128), 64, False)])
def test_fused_epilogues_on_moved_tiles(K, dims, D, fused):
	T, F, Kd = dims
	a, w = _randn(T, Kd, seed=55), _randn(2 * F, Kd, seed=56, scale=0.05)
	(gu, act), passes = _launches(PROF_ACT_FWD, lambda: K.gemm_act(a, w, K.ACT_SWIGLU))
	assert (passes == 0) == fused
	assert torch.equal(gu, K.gemm(a, w)) and torch.equal(act, K.swiglu_fwd(gu))
	cs, n_rot = K.rope_table(64, D, 1e4), 2 * F // D - 1
	got, passes = _launches(PROF_ROPE, lambda: K.gemm_rope(a, w, cs, 64, n_rot, D))
	assert (passes == 0) == fused
	assert torch.equal(got, K.gemm_rope(a, w, cs, 64, n_rot, D, fused=False))


def test_gemm_strided_views(K):
	# operands that are column slices of wider buffers (leading dimension > row length)
	big = _randn(512, 1024, seed=6)
	A = big[:, 128:640]                      # [512, 512], ld 1024
	Bw = _randn(256, 512, seed=7, scale=0.05)
	out = torch.zeros(512, 512, dtype=torch.bfloat16, device="cuda")
	K.gemm(A, Bw, out=out[:, 256:])          # writes a column slice
	_close(out[:, 256:], A.float() @ Bw.float().t(), what="strided")
	assert out[:, :256].abs().max().item() == 0


def test_gemm_rejects_bad_shapes(K):
	from elf_amd._lib import ElfStageError

	A = _randn(100, 64)
	B = _randn(64, 64)
	with pytest.raises(ElfStageError):
		K.gemm(A, B)
	with pytest.raises(ElfStageError):
		K.gemm(_randn(64, 72), _randn(64, 72))  # K not a multiple of 64
	with pytest.raises(ElfStageError):
		K.gemm(A.cpu(), B)


@pytest.mark.parametrize("d", [256, 768, 1024, 2048, 4096, 8192])
@pytest.mark.parametrize("kind", ["rms", "ln"])
def test_norm_fwd_bwd(K, d, kind):
	T = 515 if d <= 2048 else 130  # ragged row count on purpose
	x = _randn(T, d, seed=10) * 1.5 + 0.25
	x = x.to(torch.bfloat16)
	gamma = (1 + 0.1 * torch.randn(d, generator=torch.Generator().manual_seed(11))).to(torch.bfloat16).cuda()
	beta = (0.1 * torch.randn(d, generator=torch.Generator().manual_seed(12))).to(torch.bfloat16).cuda()
	dy = _randn(T, d, seed=13)
	dres = _randn(T, d, seed=14)
	eps = 1e-5
	xr = x.float().requires_grad_(True)
	gr = gamma.float().requires_grad_(True)
	br = beta.float().requires_grad_(True)
	if kind == "rms":
		yr = xr * torch.rsqrt(xr.pow(2).mean(-1, keepdim=True) + eps) * gr
	else:
		yr = torch.nn.functional.layer_norm(xr, (d,), gr, br, eps)
	yr.backward(dy.float())
	k = K.NORM_RMS if kind == "rms" else K.NORM_LAYER
	y, stats = K.norm_fwd(k, x, gamma, beta if kind == "ln" else None, eps)
	_close(y, yr.detach(), what="norm fwd")
	dgamma = torch.full((d,), 0.5, dtype=torch.float32, device="cuda")
	dbeta = torch.full((d,), -0.5, dtype=torch.float32, device="cuda")
	dx = K.norm_bwd(k, dy, x, gamma, stats, dgamma, dbeta if kind == "ln" else None, dres)
	_close(dx, xr.grad + dres.float(), what="norm dx")
	_close(dgamma - 0.5, gr.grad, rel_fro=1e-4, rel_max=1e-3, what="dgamma")
	if kind == "ln":
		_close(dbeta + 0.5, br.grad, rel_fro=1e-4, rel_max=1e-3, what="dbeta")
	dx2 = K.norm_bwd(k, dy, x, gamma, stats, dgamma, dbeta if kind == "ln" else None, None)
	_close(dx2, xr.grad, what="norm dx no residual")


@pytest.mark.parametrize("shape", [(64, 64, 64), (192, 320, 192), (512, 832, 128)])
def test_gemm_output_at_any_element(K, shape):
	"""Outputs and residuals that start at any element, with an odd leading dimension."""
	M, N, Kd = shape
	A, B = _randn(M, Kd, seed=51), _randn(N, Kd, seed=52, scale=0.05)
	R = _randn(M + 1, N + 3, seed=53)[1:, 1 : N + 1]
	want, want_r = K.gemm(A, B), K.gemm(A, B, epilogue=K.EPI_BF16_RESID, residual=R.contiguous())
	for epi, res, ref in ((K.EPI_BF16, None, want), (K.EPI_BF16_RESID, R, want_r)):
		big = torch.full((M + 2, N + 5), 7.0, dtype=torch.bfloat16, device="cuda")
		view = big[1 : M + 1, 3 : N + 3]
		K.gemm(A, B, out=view, epilogue=epi, residual=res)
		assert torch.equal(view, ref)
		big[1 : M + 1, 3 : N + 3] = 7
		assert (big == 7).all()


@pytest.mark.parametrize("tile_cfg,shape", [(7, (320, 576, 128)), (8, (192, 448, 192)), (9, (192, 320, 192)), (12, (64, 128, 320)), (0, (192, 320, 128))])
def test_gemm_output_at_any_element_on_every_kind_of_tile(K, tile_cfg, shape):
	"""The same on ragged tiles of both kernels, and for fp32 outputs (added to and stored, whole and in K ranges)."""
	M, N, Kd = shape
	A, B = _randn(M, Kd, seed=51), _randn(N, Kd, seed=52, scale=0.05)
	R = _randn(M + 1, N + 3, seed=53)[1:, 1 : N + 1]
	for epi, res, ks in ((K.EPI_BF16, None, 0), (K.EPI_BF16_RESID, R, 0), (K.EPI_F32_STORE, None, 0), (K.EPI_F32_ACC, None, 1), (K.EPI_F32_ACC, None, 2)):
		kw = dict(epilogue=epi, tile_cfg=tile_cfg, k_splits=ks)
		dt = torch.bfloat16 if res is not None or epi == K.EPI_BF16 else torch.float32
		want = torch.full((M, N), 7.0, dtype=dt, device="cuda")
		K.gemm(A, B, out=want, residual=res.contiguous() if res is not None else None, **kw)
		big = torch.full((M + 2, N + 5), 7.0, dtype=dt, device="cuda")
		view = big[1 : M + 1, 3 : N + 3]
		K.gemm(A, B, out=view, residual=res, **kw)
		assert torch.equal(view, want), (epi, ks)
		view.fill_(7)
		assert (big == 7).all(), (epi, ks)


@pytest.mark.parametrize("d", [1032, 1600, 2040, 2048])
@pytest.mark.parametrize("T", [1, 3, 513, 2047, 2050, 3075])
@pytest.mark.parametrize("kind", ["rms", "ln"])
def test_norm_bwd_two_rows_a_trip(K, d, T, kind):
	"""Rows of 1025 to 2048 columns, two a trip: one row alone, odd counts, a last trip that some workgroups miss, the step from
	one workgroup per compute unit to two, widths with idle threads.  The workspace of more rows is never smaller."""
	from elf_amd import _lib

	lib = _lib.load()
	assert all(lib.elf_norm_bwd_workspace_floats(t, d) <= lib.elf_norm_bwd_workspace_floats(t + 1, d) for t in range(max(1, T - 3), T + 3))
	x, dy, dres = _randn(T, d, seed=41) + 0.25, _randn(T, d, seed=42), _randn(T, d, seed=43)
	x = x.to(torch.bfloat16)
	gamma, beta = (1 + 0.1 * _randn(1, d, seed=44).float()).to(torch.bfloat16)[0], _randn(1, d, seed=45)[0]
	xr, gr, br = (t.double().requires_grad_(True) for t in (x, gamma, beta))
	yr = torch.nn.functional.layer_norm(xr, (d,), gr, br, 1e-5) if kind == "ln" else xr * torch.rsqrt(xr.pow(2).mean(-1, keepdim=True) + 1e-5) * gr
	yr.backward(dy.double())
	k = K.NORM_LAYER if kind == "ln" else K.NORM_RMS
	_, stats = K.norm_fwd(k, x, gamma, beta if kind == "ln" else None, 1e-5)
	dgamma, dbeta = torch.zeros(d, device="cuda"), torch.zeros(d, device="cuda") if kind == "ln" else None
	dx = K.norm_bwd(k, dy, x, gamma, stats, dgamma, dbeta, dres)
	_close(dx, (xr.grad + dres.double()).float(), what="dx")
	# fp32 sums of T products, each with the row statistics' few units of 2^-24
	_close(dgamma, gr.grad.float(), rel_fro=1e-5, rel_max=1e-4, what="dgamma")
	if kind == "ln":
		_close(dbeta, br.grad.float(), rel_fro=1e-5, rel_max=1e-4, what="dbeta")
	again = torch.zeros_like(dgamma)
	assert torch.equal(K.norm_bwd(k, dy, x, gamma, stats, again, torch.zeros_like(dgamma) if kind == "ln" else None, dres), dx)
	assert torch.equal(again, dgamma)


def test_gelu_swiglu(K):
	x = _randn(300, 1024, seed=20) * 2
	x = x.to(torch.bfloat16)
	dy = _randn(300, 1024, seed=21)
	xr = x.float().requires_grad_(True)
	yr = torch.nn.functional.gelu(xr)
	yr.backward(dy.float())
	_close(K.gelu_fwd(x), yr.detach(), what="gelu")
	_close(K.gelu_bwd(dy, x), xr.grad, what="gelu bwd")
	F = 512
	gu = x  # [300, 2F]
	dh = _randn(300, F, seed=22)
	gur = gu.float().requires_grad_(True)
	hr = torch.nn.functional.silu(gur[:, :F]) * gur[:, F:]
	hr.backward(dh.float())
	_close(K.swiglu_fwd(gu), hr.detach(), what="swiglu")
	_close(K.swiglu_bwd(dh, gu), gur.grad, what="swiglu bwd")


@pytest.mark.parametrize("act", ["gelu", "swiglu"])
@pytest.mark.parametrize("shape", [(2048, 6144, 128), (1024, 4096, 192), (1536, 8192, 64), (320, 1024, 128)])
def test_gemm_with_activation_epilogue(K, act, shape):
	"""Up-projection with its activation (SwiGLU: in the GEMM epilogue; GELU: GEMM + activation kernel
	behind the same entry point): against fp32 torch, and bit for bit against the GEMM followed by the
	activation kernel.  Shapes: 256x256 tiles, 128x256 tiles, a single K slice, and one the fused tiles
	do not cover (the library then runs the two kernels itself)."""
	M, N, Kd = shape
	A = _randn(M, Kd, seed=41)
	W = _randn(N, Kd, seed=42, scale=0.12)
	code = K.ACT_GELU if act == "gelu" else K.ACT_SWIGLU
	pre, out = K.gemm_act(A, W, code)
	ref_pre = A.float() @ W.float().t()
	_close(pre, ref_pre, what="pre-activation")
	p32 = pre.float()
	if act == "gelu":
		ref_out = torch.nn.functional.gelu(p32)
		two = K.gelu_fwd(K.gemm(A, W))
	else:
		F = N // 2
		ref_out = torch.nn.functional.silu(p32[:, :F]) * p32[:, F:]
		two = K.swiglu_fwd(K.gemm(A, W))
	_close(out, ref_out, what="activated")
	assert torch.equal(pre, K.gemm(A, W)), "pre-activation differs from the plain GEMM"
	assert torch.equal(out, two), "fused activation differs from the separate kernel"


@pytest.mark.parametrize("shape", [(8192, 2048, 256), (4096, 3072, 64), (512, 1024, 128)])
def test_gemm_with_swiglu_backward_epilogue(K, shape):
	"""dX of the down projection with the SwiGLU's backward in the GEMM epilogue: against fp32 torch autograd
	of silu(g) * u, and bit for bit against the GEMM followed by the activation-backward kernel.  Shapes: two the
	fused tiles cover (one with a single K slice) and one they do not (the library runs the two kernels itself)."""
	M, F, Kd = shape
	dY = _randn(M, Kd, seed=51)
	W2 = _randn(Kd, F, seed=52, scale=0.1)
	gu = _randn(M, 2 * F, seed=53)
	dgu = K.gemm_swiglu_bwd(dY, W2, gu)
	two = K.gemm_swiglu_bwd(dY, W2, gu, fused=False)
	assert torch.equal(dgu, two), "fused activation backward differs from the separate kernels"
	d = (dY.float() @ W2.float()).to(torch.bfloat16).float()
	g32 = gu.float().requires_grad_(True)
	(torch.nn.functional.silu(g32[:, :F]) * g32[:, F:]).backward(d)
	_close(dgu, g32.grad, what="gradient of [g | u]")


@pytest.mark.parametrize("shape", [(8192, 6144, 256, 4096, 32, 8, 128), (4096, 2048, 64, 1024, 12, 4, 64), (2048, 4096, 128, 512, 5, 3, 128), (512, 1024, 128, 256, 4, 2, 128)])
def test_gemm_with_rope_epilogue(K, shape):
	"""The packed q | k | v projection with the rotary embedding of its q and k heads in the GEMM epilogue:
	bit for bit against the GEMM followed by the RoPE kernel, and against an fp32 rotation (fp64 angles) of
	the rounded projection.  Shapes: 256x256 tiles with heads of 128 (the Llama-3-8B projection), 128x256
	tiles with heads of 64, an odd number of rotated heads (the v heads start in the middle of a tile), and
	one the fused tiles do not cover (the library runs the two kernels itself)."""
	M, N, Kd, S, Hq, Hkv, D = shape
	assert (Hq + 2 * Hkv) * D <= N
	A = _randn(M, Kd, seed=61)
	W = _randn(N, Kd, seed=62, scale=0.1)
	cs = K.rope_table(S, D, 5e5)
	got = K.gemm_rope(A, W, cs, S, Hq + Hkv, D)
	two = K.gemm_rope(A, W, cs, S, Hq + Hkv, D, fused=False)
	assert torch.equal(got, two), "fused rotation differs from the separate kernel"
	plain = K.gemm(A, W)
	nrot = (Hq + Hkv) * D
	assert torch.equal(got[:, nrot:], plain[:, nrot:]), "columns after the rotated heads must be the plain projection"
	ref = _rope_ref(plain[:, :nrot].float().view(M, Hq + Hkv, D), S, D, 5e5).reshape(M, nrot)
	_close(got[:, :nrot], ref, what="rotated projection")


@pytest.mark.parametrize("dims", [(1024, 2048, 128), (512, 4096, 1664), (256, 8192, 1024), (128, 128, 64), (192, 320, 128), (576, 192, 192)])
def test_gemm_with_activation_strided_outputs(K, dims):
	"""Outputs that are column slices of wider buffers, as a caller that packs activations would pass: at every M and F of at least
	128, also where the product and the activation one after the other are faster.  The same bits as those two."""
	from elf_amd import _lib

	M, F, Kd = dims
	A = _randn(M, Kd, seed=43)
	W = _randn(2 * F, Kd, seed=44, scale=0.12)
	pre = torch.zeros(M, 2 * F + 64, dtype=torch.bfloat16, device="cuda")
	out = torch.zeros(M, F + 64, dtype=torch.bfloat16, device="cuda")
	rc = _lib.load().elf_gemm_act_bf16(K.ACT_SWIGLU, M, F, Kd, A.data_ptr(), Kd, W.data_ptr(), Kd, pre.data_ptr(), pre.stride(0),
	                                   out.data_ptr(), out.stride(0), torch.cuda.current_stream().cuda_stream)
	_lib.check(rc, "elf_gemm_act_bf16")
	p2, o2 = K.gemm_act(A, W, K.ACT_SWIGLU)
	assert torch.equal(pre[:, : 2 * F], p2) and torch.equal(out[:, :F], o2)
	assert torch.equal(p2, K.gemm(A, W)) and torch.equal(o2, K.swiglu_fwd(p2))
	assert pre[:, 2 * F :].abs().max().item() == 0 and out[:, F:].abs().max().item() == 0


@pytest.mark.parametrize("dims", [(1024, 16640, 8192), (8192, 2304, 8192), (256, 256, 64), (320, 448, 128)])
@pytest.mark.parametrize("strided", [False, True])
def test_swiglu_backward_without_scratch_at_any_size_a_tile_fits(K, dims, strided):
	"""M and F of at least 256: neither scratch nor dense buffers are needed, also where the product and the activation backward
	one after the other are faster (1024 x 16640 x 8192: 260 tiles on 256 compute units).  The same bits as those two."""
	from elf_amd import _lib

	M, F, Kd = dims
	dy, w2, gu = _randn(M, Kd, seed=47), _randn(Kd, F, seed=48, scale=0.05), _randn(M, 2 * F, seed=49)
	pad = 8 if strided else 0
	gin, dgu = torch.zeros(M, 2 * F + pad, dtype=torch.bfloat16, device="cuda"), torch.zeros(M, 2 * F + pad, dtype=torch.bfloat16, device="cuda")
	gin[:, : 2 * F] = gu
	_lib.check(_lib.load().elf_gemm_swiglu_bwd_bf16(M, F, Kd, dy.data_ptr(), Kd, w2.data_ptr(), F, gin.data_ptr(), gin.stride(0), dgu.data_ptr(), dgu.stride(0), None,
	                                                torch.cuda.current_stream().cuda_stream), "elf_gemm_swiglu_bwd_bf16")
	assert torch.equal(dgu[:, : 2 * F], K.gemm_swiglu_bwd(dy, w2, gu, fused=False))
	assert dgu[:, 2 * F :].float().abs().sum().item() == 0


def _rope_ref(x, S, D, theta):
	# x: [T, H, D] fp32; half-split rotation, angles in fp64
	T = x.shape[0]
	pos = (torch.arange(T, device=x.device) % S).double()
	inv = theta ** (-torch.arange(0, D // 2, device=x.device).double() / (D // 2))
	ang = pos[:, None] * inv[None, :]
	cos, sin = ang.cos().float()[:, None, :], ang.sin().float()[:, None, :]
	a, b = x[..., : D // 2], x[..., D // 2 :]
	return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def test_rope(K):
	S, B, Hq, Hkv, D, theta = 256, 2, 4, 2, 128, 5e5
	T = B * S
	qkv = _randn(T, (Hq + 2 * Hkv) * D, seed=30)
	cs = K.rope_table(S, D, theta)
	ref = qkv.float().clone()
	nrot = Hq + Hkv
	ref[:, : nrot * D] = _rope_ref(ref[:, : nrot * D].reshape(T, nrot, D), S, D, theta).reshape(T, -1)
	out = qkv.clone()
	K.rope_apply_(out, cs, S, nrot, D)
	_close(out, ref, what="rope fwd")
	assert torch.equal(out[:, nrot * D :], qkv[:, nrot * D :]), "v columns must be untouched"
	# backward = inverse rotation: rotating the forward result back returns the input
	back = out.clone()
	K.rope_apply_(back, cs, S, nrot, D, backward=True)
	_close(back, qkv, what="rope inverse")


def test_scale_and_add(K):
	acc = torch.randn(1000003, device="cuda")
	ref = acc.clone() * 0.125
	out = torch.empty(1000003, dtype=torch.bfloat16, device="cuda")
	K.scale_grads_(acc, out, 0.125)
	assert torch.equal(acc, ref)
	assert torch.equal(out, ref.to(torch.bfloat16))
	a, b = _randn(4096, 64, seed=40), _randn(4096, 64, seed=41)
	assert torch.equal(K.add(a, b), (a.float() + b.float()).to(torch.bfloat16))


def _attn_ref(qkv, B, S, Hq, Hkv, D, causal, do=None):
	T = B * S
	x = qkv.float().requires_grad_(True)
	q = x[:, : Hq * D].reshape(B, S, Hq, D).transpose(1, 2)
	k = x[:, Hq * D : (Hq + Hkv) * D].reshape(B, S, Hkv, D).transpose(1, 2)
	v = x[:, (Hq + Hkv) * D :].reshape(B, S, Hkv, D).transpose(1, 2)
	G = Hq // Hkv
	k = k.repeat_interleave(G, dim=1)
	v = v.repeat_interleave(G, dim=1)
	s = (q @ k.transpose(-1, -2)) / math.sqrt(D)
	if causal:
		mask = torch.ones(S, S, dtype=torch.bool, device=x.device).tril()
		s = s.masked_fill(~mask, float("-inf"))
	lse = torch.logsumexp(s, dim=-1)
	o = (torch.softmax(s, dim=-1) @ v).transpose(1, 2).reshape(T, Hq * D)
	if do is not None:
		o.backward(do.float())
		return o.detach(), lse.detach(), x.grad
	return o.detach(), lse.detach(), None


@pytest.mark.parametrize("cfg", [
	(1, 128, 2, 2, 64, False), (2, 256, 4, 4, 64, False), (2, 256, 4, 2, 128, True),
	(1, 512, 8, 2, 128, True), (1, 384, 2, 1, 64, True), (2, 128, 4, 4, 128, False),
	(1, 1024, 4, 1, 128, True), (1, 1024, 3, 3, 64, False), (1, 640, 2, 2, 128, True),
])
def test_attention_fwd_bwd(K, cfg):
	B, S, Hq, Hkv, D, causal = cfg
	T = B * S
	qkv = _randn(T, (Hq + 2 * Hkv) * D, seed=50)
	do = _randn(T, Hq * D, seed=51)
	o_ref, lse_ref, dqkv_ref = _attn_ref(qkv, B, S, Hq, Hkv, D, causal, do)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	_close(o, o_ref, what=f"attn fwd {cfg}")
	_close(lse, lse_ref, rel_fro=1e-3, rel_max=1e-2, what="lse")
	dqkv = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal)
	for name, sl in (("dq", slice(0, Hq * D)), ("dk", slice(Hq * D, (Hq + Hkv) * D)), ("dv", slice((Hq + Hkv) * D, None))):
		_close(dqkv[:, sl], dqkv_ref[:, sl], rel_fro=1.5e-2, what=f"attn {name} {cfg}")
	# no atomics anywhere in the backward: a second run gives the same bits
	assert torch.equal(dqkv, K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal))
	# the backward of a rotary embedding on q and k, applied where dQ and dK are stored: the bits of the plain
	# backward followed by the RoPE kernel's backward pass
	cs = K.rope_table(S, D, 5e5)
	fused = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal, rope_cs=cs)
	assert torch.equal(fused, K.rope_apply_(dqkv.clone(), cs, S, Hq + Hkv, D, backward=True))


@pytest.mark.parametrize("cfg", [(1, 2176, 6, 1, 128, True), (1, 896, 6, 2, 128, False), (1, 1664, 12, 4, 64, True), (3, 640, 5, 5, 64, False), (2, 384, 16, 16, 128, True)])
def test_attention_backward_with_walks_shared_by_workgroups(K, cfg):
	"""Few key tiles and kv heads: the query heads of a group and the query tiles of a pass (in two and four parts that the
	tile count does not divide evenly) go to different workgroups, whose dK and dV meet as fp32 partial sums.  Against fp32
	autograd, equal bits from run to run, the rotation undone as by a pass of its own, and a workspace sized for a batch that
	also holds every smaller one."""
	from elf_amd import _lib

	B, S, Hq, Hkv, D, causal = cfg
	T = B * S
	qkv, do = _randn(T, (Hq + 2 * Hkv) * D, seed=55), _randn(T, Hq * D, seed=56)
	o_ref, _, dqkv_ref = _attn_ref(qkv, B, S, Hq, Hkv, D, causal, do)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	dqkv = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal)
	for name, sl in (("dq", slice(0, Hq * D)), ("dk", slice(Hq * D, (Hq + Hkv) * D)), ("dv", slice((Hq + Hkv) * D, None))):
		_close(dqkv[:, sl], dqkv_ref[:, sl], rel_fro=1.5e-2, what=f"attn {name} {cfg}")
	assert torch.equal(dqkv, K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal))
	cs = K.rope_table(S, D, 5e5)
	fused = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal, rope_cs=cs)
	assert torch.equal(fused, K.rope_apply_(dqkv.clone(), cs, S, Hq + Hkv, D, backward=True))
	sizes = [_lib.load().elf_attn_bwd_workspace_bytes(b, S, Hq, D, int(causal)) for b in range(1, 9)]
	assert sizes == sorted(sizes)


@pytest.mark.parametrize("cfg", [(1, 896, 4, 4, 64, False), (2, 1152, 4, 2, 64, True), (9, 256, 16, 16, 64, True), (6, 384, 20, 4, 64, False), (1, 2048, 3, 3, 64, True), (3, 1024, 48, 8, 64, True)])
def test_attention_backward_of_64_columns_over_256_keys_a_pass(K, cfg):
	"""Heads of 64 columns take 256 keys a pass from 896 tokens up, shorter ones where they fill the chip: sequences that 256 divides
	and odd multiples of 128 (half of the last pass lies past the end), one pass and many, walks whole, split by heads and by
	queries, more workgroups than compute units.  Bounds of the 128-key kernels above: the same bf16 roundings, half as many of dQ."""
	B, S, Hq, Hkv, D, causal = cfg
	T = B * S
	qkv, do = _randn(T, (Hq + 2 * Hkv) * D, seed=59), _randn(T, Hq * D, seed=60)
	o_ref, _, dqkv_ref = _attn_ref(qkv, B, S, Hq, Hkv, D, causal, do)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	dqkv = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal)
	for name, sl in (("dq", slice(0, Hq * D)), ("dk", slice(Hq * D, (Hq + Hkv) * D)), ("dv", slice((Hq + Hkv) * D, None))):
		_close(dqkv[:, sl], dqkv_ref[:, sl], rel_fro=1.5e-2, what=f"attn {name} {cfg}")
	assert torch.equal(dqkv, K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal))
	cs = K.rope_table(S, D, 5e5)
	fused = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal, rope_cs=cs)
	assert torch.equal(fused, K.rope_apply_(dqkv.clone(), cs, S, Hq + Hkv, D, backward=True))


@pytest.mark.parametrize("cfg", [(1, 128, 8, 2, 128, True), (3, 256, 4, 2, 128, True), (4, 512, 12, 12, 64, True), (1, 1152, 6, 3, 64, True), (1, 640, 12, 2, 128, True)])
def test_attention_backward_with_a_workgroup_per_key_tile(K, cfg):
	"""Causal, key tiles (one, two, an odd number) that all fit the chip at once: each goes to a workgroup of its own, with and
	without shared walks.  Against fp32 autograd, equal bits from run to run, the rotation undone as by a pass of its own."""
	B, S, Hq, Hkv, D, causal = cfg
	T = B * S
	qkv, do = _randn(T, (Hq + 2 * Hkv) * D, seed=57), _randn(T, Hq * D, seed=58)
	o_ref, _, dqkv_ref = _attn_ref(qkv, B, S, Hq, Hkv, D, causal, do)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	dqkv = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal)
	for name, sl in (("dq", slice(0, Hq * D)), ("dk", slice(Hq * D, (Hq + Hkv) * D)), ("dv", slice((Hq + Hkv) * D, None))):
		_close(dqkv[:, sl], dqkv_ref[:, sl], rel_fro=1.5e-2, what=f"attn {name} {cfg}")
	assert torch.equal(dqkv, K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal))
	cs = K.rope_table(S, D, 5e5)
	fused = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal, rope_cs=cs)
	assert torch.equal(fused, K.rope_apply_(dqkv.clone(), cs, S, Hq + Hkv, D, backward=True))


@pytest.mark.parametrize("cfg", [(1, 1, 1, 64, False), (3, 5, 5, 64, True), (2, 3, 3, 128, False), (1, 2, 2, 128, True), (9, 32, 32, 64, True), (9, 32, 32, 128, True), (8, 6, 2, 64, False),
                                 (16, 6, 3, 64, True), (17, 4, 2, 128, False), (14, 64, 8, 64, True)])
def test_attention_backward_of_128_tokens_in_one_kernel(K, cfg):
	"""One key tile: a head a workgroup and groups of two to eight, one workgroup, more than compute units, the fewest groups
	of a size that come here.  Bounds, repeated bits and rotation as above (dQ has one rounding less)."""
	B, Hq, Hkv, D, causal = cfg
	S, T = 128, B * 128
	qkv, do = _randn(T, (Hq + 2 * Hkv) * D, seed=61), _randn(T, Hq * D, seed=62)
	o_ref, _, dqkv_ref = _attn_ref(qkv, B, S, Hq, Hkv, D, causal, do)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	dqkv = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal)
	for name, sl in (("dq", slice(0, Hq * D)), ("dk", slice(Hq * D, (Hq + Hkv) * D)), ("dv", slice((Hq + Hkv) * D, None))):
		_close(dqkv[:, sl], dqkv_ref[:, sl], rel_fro=1.5e-2, what=f"attn {name} {cfg}")
	assert torch.equal(dqkv, K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal))
	cs = K.rope_table(S, D, 5e5)
	fused = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal, rope_cs=cs)
	assert torch.equal(fused, K.rope_apply_(dqkv.clone(), cs, S, Hq + Hkv, D, backward=True))


def _check_attn_bwd(K, cfg, way, seed):
	"""The way a shape takes, then gradients against fp32 autograd, equal bits from run to run and the rotation undone as by a pass of its own."""
	B, S, Hq, Hkv, D, causal = cfg
	T = B * S
	assert K.attn_bwd_way(*cfg) == way
	qkv, do = _randn(T, (Hq + 2 * Hkv) * D, seed=seed), _randn(T, Hq * D, seed=seed + 1)
	o_ref, _, dqkv_ref = _attn_ref(qkv, B, S, Hq, Hkv, D, causal, do)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	dqkv = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal)
	for name, sl in (("dq", slice(0, Hq * D)), ("dk", slice(Hq * D, (Hq + Hkv) * D)), ("dv", slice((Hq + Hkv) * D, None))):
		_close(dqkv[:, sl], dqkv_ref[:, sl], rel_fro=1.5e-2, what=f"attn {name} {cfg}")
	assert torch.equal(dqkv, K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal))
	cs = K.rope_table(S, D, 5e5)
	fused = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal, rope_cs=cs)
	assert torch.equal(fused, K.rope_apply_(dqkv.clone(), cs, S, Hq + Hkv, D, backward=True))


@pytest.mark.parametrize("cfg,way", [
	((8, 256, 1, 1, 128, True), (128, 1, 4, False)), ((9, 640, 8, 8, 128, True), (128, 1, 1, False)), ((11, 512, 7, 7, 128, True), (128, 1, 1, False)),
	((8, 384, 8, 8, 64, True), (128, 1, 1, False)), ((9, 384, 9, 9, 64, True), (128, 1, 1, False)),
	((1, 1152, 6, 3, 64, True), (256, 2, 4, False)), ((8, 1024, 16, 8, 64, True), (256, 1, 1, False)), ((9, 1024, 16, 8, 64, True), (256, 1, 1, False)),
])
def test_attention_backward_of_single_key_tiles_that_fit_at_once_or_do_not(K, cfg, way):
	"""Causal launches of single key tiles, of each kernel: 64 to 256 workgroups (a group's tiles side by side) and 288 to 360 (the longest
	walks first), groups in a multiple of eight (each on one XCD) and not."""
	_check_attn_bwd(K, cfg, way, 67)


@pytest.mark.parametrize("cfg,way", [
	((8, 2048, 32, 16, 64, True), (256, 1, 1, True)), ((8, 1920, 32, 8, 64, True), (256, 1, 1, True)), ((1, 3968, 16, 2, 64, True), (256, 8, 2, True)),
	((13, 384, 60, 10, 64, True), (128, 1, 1, True)),
])
def test_attention_backward_of_pairs_of_key_tiles_of_64_columns(K, cfg, way):
	"""Causal, a light and a heavy key tile one after the other in a workgroup: the second pass reuses the first one's LDS, takes a last tile
	that is half past the end (1920 and 3968 tokens are odd multiples of 128), leaves partial dK and dV, and follows the middle tile of three,
	which has no partner (384 tokens)."""
	_check_attn_bwd(K, cfg, way, 69)


@pytest.mark.parametrize("cfg,way", [
	((32, 128, 6, 2, 64, False), (0, 1, 1, False)), ((5, 128, 3, 3, 64, True), (0, 1, 1, False)), ((17, 128, 4, 2, 128, False), (0, 1, 1, False)),
	((5, 896, 2, 2, 64, False), (256, 1, 4, False)), ((2, 1152, 4, 2, 64, True), (256, 2, 4, False)), ((6, 384, 20, 4, 64, False), (256, 5, 1, False)),
])
def test_attention_backward_in_the_kernels_that_cases_stand_for(K, cfg, way):
	"""Without a mask, three heads of 64 a group in the one kernel (the fewest groups that go there; the walk over the heads reuses what
	the one before left in LDS) and 256 keys a pass where 128 tokens fewer would take 128: the way is asked, not supposed."""
	_check_attn_bwd(K, cfg, way, 75)


def _attn_bwd_separate(B, S, Hq, Hkv, D, causal, q, k, v, o, do, lse, rope_cs=None):
	"""dq, dk and dv of operands in buffers of their own ([B * S, heads * D] with any row stride)."""
	from elf_amd import _lib

	lib, T = _lib.load(), B * S
	n = lib.elf_attn_bwd_shared_workspace_bytes(B, S, Hq, Hkv, D, int(causal))
	ws = torch.empty(n, dtype=torch.uint8, device="cuda")
	dq, dk, dv = (torch.empty(T, h * D, dtype=torch.bfloat16, device="cuda") for h in (Hq, Hkv, Hkv))
	rc = lib.elf_attn_bwd_shared(*(t.data_ptr() for t in (q, k, v, o, do, lse, dq, dk, dv, ws)), n, *(t.stride(0) for t in (q, k, v, o, do, dq, dk, dv)),
	                             B, S, Hq, Hkv, D, int(causal), 1 / math.sqrt(D), rope_cs.data_ptr() if rope_cs is not None else None, torch.cuda.current_stream().cuda_stream)
	_lib.check(rc, "elf_attn_bwd_shared")
	return dq, dk, dv


_EACH_KERNEL = [((3, 128, 5, 5, 64, True), 0), ((2, 128, 3, 3, 128, False), 0), ((32, 128, 6, 2, 64, False), 0), ((2, 1152, 4, 2, 64, True), 256),
                ((5, 896, 2, 2, 64, False), 256), ((8, 384, 2, 1, 64, True), 128), ((3, 256, 4, 2, 128, True), 128)]


@pytest.mark.parametrize("cfg,keys", _EACH_KERNEL)
def test_attention_backward_of_operands_in_buffers_of_their_own(K, cfg, keys):
	"""Rows of q, k, v, o and dO with a stride of their own each: the bits of packed rows."""
	B, S, Hq, Hkv, D, causal = cfg
	T = B * S
	assert K.attn_bwd_way(*cfg)[0] == keys
	qkv, do = _randn(T, (Hq + 2 * Hkv) * D, seed=71), _randn(T, Hq * D, seed=72)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	want = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal)
	own = []
	for i, t in enumerate((*qkv.split([Hq * D, Hkv * D, Hkv * D], dim=1), o, do)):
		own.append(torch.full((T, t.shape[1] + 8 * (2 * i + 1)), float("nan"), dtype=torch.bfloat16, device="cuda")[:, : t.shape[1]])
		own[-1].copy_(t)
	got = _attn_bwd_separate(B, S, Hq, Hkv, D, causal, *own, lse)
	assert torch.equal(torch.cat(got, dim=1), want)


@pytest.mark.parametrize("cfg,keys", _EACH_KERNEL)
@pytest.mark.parametrize("what", [float("inf"), float("nan")])
def test_attention_backward_keeps_an_infinity_in_its_group(K, cfg, keys, what):
	"""An infinity or NaN in one dO row of one head: every other group of heads and sequence has the bits it has without, and of that head's dQ
	the rows of other queries too; that row's dQ is not finite, and no dV of a key it attends to is."""
	B, S, Hq, Hkv, D, causal = cfg
	T, G = B * S, Hq // Hkv
	assert K.attn_bwd_way(*cfg)[0] == keys
	qkv, do = _randn(T, (Hq + 2 * Hkv) * D, seed=73), _randn(T, Hq * D, seed=74)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	want = K.attn_bwd(qkv, o, do, lse, B, S, Hq, Hkv, D, causal)
	row, head = S // 2 + 5, Hq - 1  # of sequence 0
	bad = do.clone()
	bad[row, head * D + 3] = what
	got = K.attn_bwd(qkv, o, bad, lse, B, S, Hq, Hkv, D, causal)
	assert torch.equal(got[S:], want[S:])
	hk = head // G
	clean = torch.ones(got.shape[1], dtype=torch.bool, device="cuda")
	clean[head * D : (head + 1) * D] = False
	for first in (Hq + hk, Hq + Hkv + hk):
		clean[first * D : (first + 1) * D] = False
	assert torch.equal(got[:S, clean], want[:S, clean])
	others = torch.arange(S, device="cuda") != row
	dq = slice(head * D, (head + 1) * D)
	assert torch.equal(got[:S, dq][others], want[:S, dq][others])
	assert not torch.isfinite(got[row, dq].float()).any()
	dv = got[:S, (Hq + Hkv + hk) * D + 3].float()
	assert not torch.isfinite(dv[: row + 1] if causal else dv).any()


@pytest.mark.parametrize("D,causal", [(64, True), (128, False)])
@pytest.mark.parametrize("far", ["q", "v", "do"])
def test_attention_backward_of_128_tokens_whose_rows_lie_far_apart(K, D, causal, far):
	"""Rows of 2^24 + 2^20 elements: row 121 lies 4 GiB from the first, further than a 32-bit byte offset reaches.  Against fp32 autograd,
	within the bounds of dense rows."""
	B, S, H, ld = 1, 128, 2, (1 << 24) + (1 << 20)
	qkv, do = _randn(S, 3 * H * D, seed=63), _randn(S, H * D, seed=64)
	o_ref, _, ref = _attn_ref(qkv, B, S, H, H, D, causal, do)
	o, lse = K.attn_fwd(qkv, B, S, H, H, D, causal)
	ops = dict(zip("qkv", (t.contiguous() for t in qkv.split(H * D, dim=1))), do=do)
	rows = torch.empty(127 * ld + H * D, dtype=torch.bfloat16, device="cuda").as_strided((S, H * D), (ld, 1))
	rows.copy_(ops[far])
	ops[far] = rows
	got = _attn_bwd_separate(B, S, H, H, D, causal, ops["q"], ops["k"], ops["v"], o, ops["do"], lse)
	for name, g, r in zip(("dq", "dk", "dv"), got, ref.split(H * D, dim=1)):
		_close(g, r, rel_fro=1.5e-2, what=f"attn {name} with {far} rows far apart")


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("off", [0, 4])
def test_attention_backward_of_128_tokens_with_v_in_a_buffer_of_its_own(K, D, off):
	"""V on a 16-byte boundary and 8 bytes past one, in rows of its own width."""
	B, S, H = 3, 128, 2
	T = B * S
	qkv, do = _randn(T, 3 * H * D, seed=65), _randn(T, H * D, seed=66)
	o_ref, _, ref = _attn_ref(qkv, B, S, H, H, D, True, do)
	o, lse = K.attn_fwd(qkv, B, S, H, H, D, True)
	q, k, v = qkv.split(H * D, dim=1)
	own = torch.empty(T * H * D + 8, dtype=torch.bfloat16, device="cuda")[off : off + T * H * D].view(T, H * D)
	own.copy_(v)
	assert K.attn_bwd_way(B, S, H, H, D, True, v=own.data_ptr())[0] == (128 if D == 128 and off else 0)
	got = _attn_bwd_separate(B, S, H, H, D, True, q, k, own, o, do, lse)
	for name, g, r in zip(("dq", "dk", "dv"), got, ref.split(H * D, dim=1)):
		_close(g, r, rel_fro=1.5e-2, what=f"attn {name} with v {2 * off} bytes past a boundary")


@pytest.mark.parametrize("cfg", [(1, 4096, 4, 4, 64, False), (2, 2048, 8, 4, 64, False), (1, 896, 8, 1, 128, True)])
@pytest.mark.parametrize("ways", [None, 1, 2, 3, 64])
def test_attention_backward_stays_inside_its_workspace(K, cfg, ways):
	"""Shapes whose walks are shared where there is room: the entry point that is not told its workspace's size (ways None) keeps
	to the size the formula gives, elf_attn_bwd_shared to the partial sums of at most `ways` parts that it is given room for.
	What lies behind the workspace keeps its value; the gradients are those of autograd in fp32."""
	from elf_amd import _lib

	B, S, Hq, Hkv, D, causal = cfg
	lib, T = _lib.load(), B * S
	whole = lib.elf_attn_bwd_workspace_bytes(B, S, Hq, D, int(causal))
	assert lib.elf_attn_bwd_shared_workspace_bytes(B, S, Hq, Hkv, D, int(causal)) > whole, "a shape whose walks are shared"
	part = 8 * B * S * Hkv * D
	n = whole if ways in (None, 1) else whole + ways * part
	ws = torch.full((n + 8 * part,), 0x5A, dtype=torch.uint8, device="cuda")  # as much again as eight parts behind it
	qkv, do = _randn(T, (Hq + 2 * Hkv) * D, seed=57), _randn(T, Hq * D, seed=58)
	o_ref, _, dqkv_ref = _attn_ref(qkv, B, S, Hq, Hkv, D, causal, do)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	dqkv = torch.empty_like(qkv)
	ld, at = qkv.stride(0), [0, 2 * Hq * D, 2 * (Hq + Hkv) * D]  # q, k, v: byte offsets in a row
	stream = torch.cuda.current_stream().cuda_stream
	ptrs = [qkv.data_ptr() + a for a in at] + [o.data_ptr(), do.data_ptr(), lse.data_ptr()] + [dqkv.data_ptr() + a for a in at] + [ws.data_ptr()]
	rest = [ld, ld, ld, Hq * D, Hq * D, ld, ld, ld, B, S, Hq, Hkv, D, int(causal), 1 / math.sqrt(D)]
	if ways is None:
		_lib.check(lib.elf_attn_bwd(*ptrs, *rest, stream), "elf_attn_bwd")
	else:
		_lib.check(lib.elf_attn_bwd_shared(*ptrs, n, *rest, None, stream), "elf_attn_bwd_shared")
	assert bool((ws[n:] == 0x5A).all()), "wrote behind its workspace"
	for name, sl in (("dq", slice(0, Hq * D)), ("dk", slice(Hq * D, (Hq + Hkv) * D)), ("dv", slice((Hq + Hkv) * D, None))):
		_close(dqkv[:, sl], dqkv_ref[:, sl], rel_fro=1.5e-2, what=f"attn {name} {cfg} {ways}")


@pytest.mark.parametrize("D,causal,ramp,gain", [(128, True, 6.0, 1.0), (128, False, 6.0, 1.0), (64, True, 6.0, 1.0), (128, True, 0.0, 6.0),
                                               (128, False, -6.0, 3.0), (64, False, 0.0, 6.0)])
def test_attention_forward_with_scores_that_climb_along_the_keys(K, D, causal, ramp, gain):
	"""The forward's softmax takes its exponentials against a reference point that follows the running maximum only
	when it has to.  Here it has to, again and again: a component of k that grows (ramp > 0) or falls (ramp < 0) with the
	key position against a constant component of q moves the row maxima by many powers of two from tile to tile, and
	gain scales everything to scores of several hundred.  Output and log-sum-exp against the fp32 softmax."""
	B, S, Hq, Hkv = 2, 1024, 4, 2
	T = B * S
	qkv = _randn(T, (Hq + 2 * Hkv) * D, seed=60).float() * gain
	pos = (torch.arange(T, device="cuda") % S).float() / S  # 0 .. 1 along each sequence
	for h in range(Hq):
		qkv[:, h * D] = 4.0
	for h in range(Hkv):
		qkv[:, (Hq + h) * D] = ramp * pos * math.sqrt(D)  # adds ramp * 4 * pos to every score: up to 35 powers of two
	qkv = qkv.to(torch.bfloat16)
	o_ref, lse_ref, _ = _attn_ref(qkv, B, S, Hq, Hkv, D, causal)
	o, lse = K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)
	assert torch.isfinite(o.float()).all() and torch.isfinite(lse).all()
	_close(o, o_ref, what=f"attn fwd, climbing scores D={D} causal={causal} ramp={ramp} gain={gain}")
	_close(lse, lse_ref, rel_fro=1e-3, rel_max=1e-2, what="lse")
	assert torch.equal(o, K.attn_fwd(qkv, B, S, Hq, Hkv, D, causal)[0])


@pytest.mark.parametrize("T,N,ld", [(8192, 768, 768), (1000, 2304, 2304), (7, 64, 128), (4096, 8, 8), (333, 4104, 4104)])
def test_colsum_is_exact_to_rounding_and_repeatable(K, T, N, ld):
	"""The bias gradient of a split linear layer: column sums of a bf16 [T, N] view (row stride ld) added to an fp32
	accumulator, equal bits from run to run (one writer per column, slices added in a fixed order)."""
	buf = _randn(T, ld, seed=91)
	x = buf[:, :N]
	start = torch.randn(N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(92))
	runs = []
	for _ in range(3):
		acc = start.clone()
		K.colsum_(x, acc)
		runs.append(acc)
	assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2])
	want = start.double() + x.double().sum(0)
	assert ((runs[0].double() - want).abs().max() / want.abs().max()).item() <= 1e-5


@pytest.mark.parametrize("T,shapes", [
	(2112, [(4288, 1600, True), (832, 4288, True)]),                          # one launch of 256x256 tiles, the last ones split
	(512, [(512, 512, True), (1536, 512, False), (512, 768, True)]),          # one launch of 128x128 tiles
	(64, [(64, 128, True), (256, 64, True)]),                                 # narrower than 256: one launch each
	(192, [(320, 256, False), (64, 64, True), (256, 320, False)] * 6),        # more layers than a launch takes, mixed
])
def test_parameter_gradients_of_a_list_of_layers(K, T, shapes):
	"""Weight and bias gradients of several layers in one call, on top of what the accumulators hold: against fp64 sums (fp32 sums of
	T products: T * 2^-24 of their magnitude, far below the bound), bias sums the bits of a call each, equal bits from run to run; two
	layers that share their parameters both count."""
	layers, want = [], []
	for i, (M, N, bias) in enumerate(shapes):
		dy, x = _randn(T, M, seed=300 + i), _randn(T, N, seed=400 + i)
		acc = torch.randn(M, N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(500 + i))
		b = torch.randn(M, device="cuda", generator=torch.Generator(device="cuda").manual_seed(600 + i)) if bias else None
		layers.append((dy, x, acc, b))
		want.append((acc.double() + dy.double().t() @ x.double(), K.colsum_(dy, b.clone()) if bias else None))
	runs = []
	for _ in range(2):
		run = [(dy, x, acc.clone(), None if b is None else b.clone()) for dy, x, acc, b in layers]
		K.linear_w_pass(run)
		runs.append(run)
	for a, b, (w, wb) in zip(*runs, want):
		assert torch.equal(a[2], b[2])
		assert float((a[2].double() - w).norm() / w.norm()) <= 1e-5
		assert wb is None or (torch.equal(a[3], wb) and torch.equal(b[3], wb))
	dy, x, acc, b = layers[0]
	twice, bias = acc.clone(), torch.zeros(dy.shape[1], device="cuda")
	K.linear_w_pass([(dy, x, twice, bias), (dy, x, twice, bias)])
	w = acc.double() + 2 * (dy.double().t() @ x.double())
	assert float((twice.double() - w).norm() / w.norm()) <= 1e-5
	assert torch.allclose(bias.double(), 2 * dy.double().sum(0), rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("M,N", [(64, 64), (512, 512), (128, 2048), (64, 4096)])
@pytest.mark.parametrize("Kd", [64, 256, 320, 1024, 3136])
@pytest.mark.parametrize("b_t", [False, True])
def test_products_on_32x32_tiles_have_the_bits_of_larger_ones(K, M, N, Kd, b_t):
	"""Products of at most 256 tiles of 32x32: one tile and a full round of them, K of one slice, of the short ring's last and the deep
	ring's first, of many.  A tile adds its products in the order of K whatever its size: the bits of the 64x64 tile, without and with a
	residual and a bias, in rows of its own width and further apart."""
	a = _randn(M, Kd, seed=700)
	b = _randn(Kd, N, seed=701) if b_t else _randn(N, Kd, seed=701)
	res, bias = _randn(M, N, seed=702), _randn(1, N, seed=703)
	assert K.gemm_way(K.WAY_INPUT_GRADIENT if b_t else K.WAY_FORWARD, M, N, Kd) == (32, 32)
	for kw in ({}, {"epilogue": K.EPI_BF16_RESID, "residual": res}, {"epilogue": K.EPI_BF16_RESID, "residual": bias, "residual_ld": 0}):
		want = K.gemm(a, b, b_t=b_t, tile_cfg=12, **kw)
		assert torch.equal(K.gemm(a, b, b_t=b_t, **kw), want)
		wide = torch.full((M, N + 24), 7.0, dtype=torch.bfloat16, device="cuda")
		K.gemm(a, b, b_t=b_t, out=wide[:, 3 : N + 3], **kw)
		assert torch.equal(wide[:, 3 : N + 3], want) and float((wide[:, :3] - 7).abs().max()) == 0 and float((wide[:, N + 3 :] - 7).abs().max()) == 0
	ref = a.double() @ (b.double() if b_t else b.double().t())
	_close(K.gemm(a, b, b_t=b_t), ref.float(), what="32x32 tile")


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M, N, Kd", [(8192, 768, 768), (896, 6208, 4160), (2560, 1664, 320), (8128, 768, 1088)])
def test_products_on_128x192_tiles_have_the_bits_of_smaller_ones(K, M, N, Kd, b_t):
	"""Products of one round of 128x192 tiles: whole ones, a last column of tiles moved back by 64 and by 128 columns, a last row moved
	back, K of few slices and of a number that is no multiple of the ring.  The bits of the 64x64 tile, as above."""
	a = _randn(M, Kd, seed=710)
	b = _randn(Kd, N, seed=711) if b_t else _randn(N, Kd, seed=711)
	res, bias = _randn(M, N, seed=712), _randn(1, N, seed=713)
	assert K.gemm_way(K.WAY_INPUT_GRADIENT if b_t else K.WAY_FORWARD, M, N, Kd) == (128, 192)
	for kw in ({}, {"epilogue": K.EPI_BF16_RESID, "residual": res}, {"epilogue": K.EPI_BF16_RESID, "residual": bias, "residual_ld": 0}):
		want = K.gemm(a, b, b_t=b_t, tile_cfg=12, **kw)
		assert torch.equal(K.gemm(a, b, b_t=b_t, **kw), want)
		wide = torch.full((M, N + 24), 7.0, dtype=torch.bfloat16, device="cuda")
		K.gemm(a, b, b_t=b_t, out=wide[:, 3 : N + 3], **kw)
		assert torch.equal(wide[:, 3 : N + 3], want) and float((wide[:, :3] - 7).abs().max()) == 0 and float((wide[:, N + 3 :] - 7).abs().max()) == 0


def test_split_k_on_one_stream_never_gives_up_its_turn_and_wide_splits_are_refused(K):
	"""Back-to-back split-K launches on one stream keep their turns (the counter of waves that added out of turn does not
	move, which is what bit-reproducible weight gradients rest on), and a split count that would not fit the 8 bits the
	turn counters give it is refused."""
	from elf_amd import _lib

	M, N, Kd = 768, 768, 8192
	A, B = _randn(Kd, M, seed=130), _randn(Kd, N, seed=131, scale=0.05)
	before = K.gemm_turn_giveups()
	runs = []
	for _ in range(3):
		acc = torch.zeros(M, N, device="cuda")
		for cfg in (7, 8, 1):
			K.gemm(A, B, a_t=True, b_t=True, out=acc, epilogue=K.EPI_F32_ACC, k_splits=4, tile_cfg=cfg)
		runs.append(acc)
	torch.cuda.synchronize()
	assert K.gemm_turn_giveups() == before
	assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2])
	with pytest.raises(_lib.ElfStageError):
		K.gemm(A, B, a_t=True, b_t=True, out=runs[0], epilogue=K.EPI_F32_ACC, k_splits=256, tile_cfg=7)


def _dw_problems(shapes, Kd, seed):
	"""(dy [Kd, M], x [Kd, N], acc [M, N] with what earlier micro-batches left in it) per (M, N)."""
	out = []
	for i, (M, N) in enumerate(shapes):
		g = torch.Generator(device="cuda").manual_seed(seed + i)
		out.append((_randn(Kd, M, seed=seed + 10 * i), _randn(Kd, N, seed=seed + 10 * i + 1, scale=0.05), torch.randn(M, N, generator=g, device="cuda")))
	return out


def test_grouped_weight_gradients_equal_the_single_launches(K):
	"""Several layers' dW += dY^T X in one launch (the W pass of a stage) against one elf_gemm_bf16 call per layer that
	splits K the same way: whole tiles (K too short to split); the GPT-2-small layers at K = 4096, whose 108 tiles are all
	in the launch's only round and split two ways; and a large layer (256 whole tiles, one round) followed by two small
	ones whose 36 tiles make up the last round and are split four ways.  Bit for bit, run after run, no turn given up; and
	against fp32 torch."""
	before = K.gemm_turn_giveups()
	for shapes, Kd, splits in (
		(((256, 512), (768, 256), (512, 768), (256, 256)), 512, (1, 1, 1, 1)),
		(((768, 3072), (3072, 768), (768, 768), (2304, 768)), 4096, (2, 2, 2, 2)),
		(((4096, 4096), (768, 768), (768, 2304)), 4096, (1, 4, 4)),
	):
		print(f"[case] gemm_dw_group {shapes} K={Kd}", flush=True)
		problems = _dw_problems(shapes, Kd, seed=400)
		start = [acc.clone() for _, _, acc in problems]
		want = []
		for (dy, x, _), acc0, ks in zip(problems, start, splits):
			acc = acc0.clone()
			K.gemm(dy, x, a_t=True, b_t=True, out=acc, epilogue=K.EPI_F32_ACC, tile_cfg=7, k_splits=ks)
			want.append(acc)
		runs = []
		for _ in range(3):
			accs = [a.clone() for a in start]
			K.gemm_dw_group([(dy, x, acc) for (dy, x, _), acc in zip(problems, accs)])
			runs.append(accs)
		torch.cuda.synchronize()
		for i, (dy, x, _) in enumerate(problems):
			assert torch.equal(runs[0][i], want[i]), f"layer {i} {shapes[i]}: grouped launch differs from the single one"
			assert torch.equal(runs[1][i], want[i]) and torch.equal(runs[2][i], want[i]), f"layer {i}: not reproducible"
			ref = start[i].double() + dy.double().t() @ x.double()
			assert ((want[i].double() - ref).abs().max() / ref.abs().max()).item() <= 1e-5
	assert K.gemm_turn_giveups() == before


@pytest.mark.parametrize("shapes", [((2048, 2048), (2048, 2048), (2048, 2048), (3072, 3072)), ((4608, 4608),), ((768, 768),)], ids=["small_layers", "one_large_layer", "one_small_layer"])
def test_grouped_weight_gradients_with_the_split_boundary_inside_a_layer(K, shapes):
	"""The launch's last round may begin in the middle of a layer: 3 x 64 + 144 tiles (80 of the last layer's tiles split
	three ways; small layers, laid on the XCDs as contiguous runs), one layer of 324 tiles (68 split three ways; its own
	tile walk), and a lone 9-tile layer (all split).  Against fp64 torch, twice with equal bits, with the scale folded in."""
	Kd = 4096
	problems = _dw_problems(shapes, Kd, seed=700)
	before = K.gemm_turn_giveups()
	runs = []
	for _ in range(2):
		accs = [acc.clone() for _, _, acc in problems]
		g16 = [torch.empty_like(a, dtype=torch.bfloat16) for a in accs]
		K.gemm_dw_group([(dy, x, acc, h) for (dy, x, _), acc, h in zip(problems, accs, g16)], scale=0.25)
		runs.append((accs, g16))
	torch.cuda.synchronize()
	assert K.gemm_turn_giveups() == before
	for i, (dy, x, start) in enumerate(problems):
		ref = (start.double() + dy.double().t() @ x.double()) * 0.25
		got = runs[0][0][i]
		assert ((got.double() - ref).abs().max() / ref.abs().max()).item() <= 1e-5, f"layer {i} {shapes[i]}"
		assert torch.equal(runs[0][1][i], got.to(torch.bfloat16)), f"layer {i}: bf16 copy"
		assert torch.equal(runs[1][0][i], got) and torch.equal(runs[1][1][i], runs[0][1][i]), f"layer {i}: not reproducible"


def test_grouped_weight_gradients_with_the_gradient_scale(K):
	"""scale != 0: the accumulators leave multiplied by the scale with their bf16 copies written, from the epilogue for
	whole tiles and by a small kernel behind the launch for split ones (here: none split, all split, and a whole layer
	followed by a split one): all equal the unscaled launch followed by elf_scale_grads bit for bit."""
	for shapes, Kd in ((((256, 512), (768, 256)), 512), (((768, 3072), (768, 768)), 8192), (((4096, 4096), (768, 768)), 4096)):
		problems = _dw_problems(shapes, Kd, seed=500)
		plain = [acc.clone() for _, _, acc in problems]
		K.gemm_dw_group([(dy, x, acc) for (dy, x, _), acc in zip(problems, plain)])
		plain16 = [torch.empty_like(a, dtype=torch.bfloat16) for a in plain]
		for a, h in zip(plain, plain16):
			K.scale_grads_(a, h, 1 / 32)
		folded = [acc.clone() for _, _, acc in problems]
		folded16 = [torch.full_like(a, 7.0, dtype=torch.bfloat16) for a in folded]
		K.gemm_dw_group([(dy, x, acc, h) for (dy, x, _), acc, h in zip(problems, folded, folded16)], scale=1 / 32)
		torch.cuda.synchronize()
		for i in range(len(problems)):
			assert torch.equal(folded[i], plain[i]) and torch.equal(folded16[i], plain16[i]), f"layer {i} {shapes[i]} K={Kd}"


def test_grouped_weight_gradients_refuse_what_the_tiles_cannot_hold(K):
	from elf_amd import _lib

	ok = _dw_problems(((256, 256),), 512, seed=600)
	with pytest.raises(_lib.ElfStageError):
		K.gemm_dw_group(ok * 17)
	with pytest.raises(_lib.ElfStageError):
		K.gemm_dw_group(_dw_problems(((256, 320),), 512, seed=601))
	with pytest.raises(_lib.ElfStageError):
		K.gemm_dw_group(ok, scale=0.5)  # a scaling pass needs somewhere to put the bf16 gradients


def test_split_k_gemms_on_two_streams_stay_correct(K):
	"""Weight-gradient GEMMs launched concurrently on two streams share the turn counters of their split tiles; whatever
	the interleaving, every sum must be the right one to fp32 rounding (a workgroup that finds its counter taken by
	the other launch adds out of turn)."""
	M, N, Kd = 768, 768, 8192
	A = [_randn(Kd, M, seed=110 + i) for i in range(2)]
	B = [_randn(Kd, N, seed=120 + i, scale=0.05) for i in range(2)]
	ref = [A[i].float().t() @ B[i].float() for i in range(2)]
	acc = [torch.zeros(M, N, device="cuda") for _ in range(2)]
	streams = [torch.cuda.Stream(), torch.cuda.Stream()]
	torch.cuda.synchronize()
	reps = 12
	for _ in range(reps):
		for i in range(2):
			with torch.cuda.stream(streams[i]):
				K.gemm(A[i], B[i], a_t=True, b_t=True, out=acc[i], epilogue=K.EPI_F32_ACC, k_splits=4, tile_cfg=7 if i == 0 else 8)
	torch.cuda.synchronize()
	for i in range(2):
		assert ((acc[i] - reps * ref[i]).norm() / (reps * ref[i]).norm()).item() <= 1e-5
