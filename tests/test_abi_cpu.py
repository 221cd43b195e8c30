"""The C-ABI library without a GPU: it loads, exports every entry point the header declares,
rejects bad arguments before touching the device, and its pinned arena follows the reference's
placement policy (checked against oracle/pinned_pool.py and hand-worked sequences)."""

import ctypes
import os
import random
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
	from elf_amd import _lib

	return _lib.load()


def _declared():
	text = open(os.path.join(ROOT, "include", "elf_stage.h")).read()
	text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
	return sorted(set(re.findall(r"\b(elf_[a-z0-9_]+)\s*\(", text)))


def test_exports_every_declared_symbol(lib):
	names = _declared()
	assert len(names) >= 40
	for n in names:
		assert hasattr(lib, n), f"{n} is declared in include/elf_stage.h but not exported"


def test_bindings_cover_the_header():
	import elf_amd.execution  # noqa: F401  (registers the stage and pool signatures)
	from elf_amd import _lib

	assert set(_declared()) == set(_lib.exported_symbols())


def test_argument_errors_without_device(lib):
	from elf_amd import _lib

	assert lib.elf_abi_version() == 1
	rc = lib.elf_gemm_bf16(0, 0, 0, 64, 64, None, 64, None, 64, None, 64, 0, None, 0, 0, 0, None)
	assert rc == -1 and b"empty problem" in lib.elf_last_error()
	rc = lib.elf_gemm_bf16(0, 0, 64, 64, 70, 16, 64, 16, 64, 16, 64, 0, None, 0, 0, 0, None)
	assert rc == -1 and b"multiple of 64" in lib.elf_last_error()
	rc = lib.elf_attn_fwd(16, 16, 16, 16, 16, 64, 64, 64, 64, 1, 100, 4, 4, 64, 0, 0.125, None)
	assert rc == -1 and b"multiple of 128" in lib.elf_last_error()
	rc = lib.elf_attn_fwd(16, 16, 16, 16, 16, 64, 64, 64, 64, 1, 128, 6, 4, 64, 0, 0.125, None)
	assert rc == -1 and b"Hkv" in lib.elf_last_error()
	rc = lib.elf_norm_fwd(0, 16, 16, None, 16, 16, 4, 100, 1e-5, None)
	assert rc == -1
	with pytest.raises(_lib.ElfStageError):
		_lib.check(rc, "elf_norm_fwd")
	assert lib.elf_norm_bwd_workspace_floats(8192, 4096) == 512 * 2 * 4096
	# bf16 dQ partials of the 32 key tiles (causal: tile kt only meets the queries from 128 kt on) + two floats per (token, head)
	stats = 2 * (2 * 4096 * 32 * 4)
	assert lib.elf_attn_bwd_workspace_bytes(2, 4096, 32, 128, 0) == 2 * (32 * 4096) * 32 * 128 * 2 + stats
	assert lib.elf_attn_bwd_workspace_bytes(2, 4096, 32, 128, 1) == 2 * sum(4096 - 128 * kt for kt in range(32)) * 32 * 128 * 2 + stats


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [0, 1])
def test_attention_workspace_of_a_larger_shape_serves_the_smaller_ones(lib, D, causal):
	"""The size is the header's formula at every shape, whether its walks would be shared or not, and grows with every argument:
	elf_attn_bwd is not told how large its buffer is, and a caller keeps one for its longest sequence."""
	heads, batches, tiles = (1, 2, 4, 6, 8, 16, 32), (1, 2, 3, 4, 8), (1, 2, 3, 7, 15, 16, 17, 31, 32, 33, 64)
	size = {}
	for B in batches:
		for nkt in tiles:
			for Hq in heads:
				S = 128 * nkt
				rows = S * (nkt + 1) // 2 if causal else S * nkt
				size[B, nkt, Hq] = lib.elf_attn_bwd_workspace_bytes(B, S, Hq, D, causal)
				assert size[B, nkt, Hq] == B * rows * Hq * D * 2 + 8 * B * S * Hq, (B, S, Hq)
				for Hkv in (h for h in heads if Hq % h == 0):
					more = lib.elf_attn_bwd_shared_workspace_bytes(B, S, Hq, Hkv, D, causal) - size[B, nkt, Hq]
					# room for a whole number of splits, four per query head at most
					assert more >= 0 and more % (8 * B * S * Hkv * D) == 0 and more // (8 * B * S * Hkv * D) <= 4 * Hq // Hkv
	for (B, nkt, Hq), n in size.items():
		for axis, values in enumerate((batches, tiles, heads)):
			key = [B, nkt, Hq]
			i = values.index(key[axis])
			if i:
				key[axis] = values[i - 1]
				assert size[tuple(key)] < n
	assert lib.elf_attn_bwd_workspace_bytes(2, 4096, 8, D, 0) > lib.elf_attn_bwd_workspace_bytes(2, 4096, 8, D, 1)


@pytest.mark.parametrize("shape,ways", [((2, 128, 4, 4, 64), 4), ((7, 128, 1, 1, 64), 4), ((1, 128, 8, 8, 128), 2), ((3, 128, 48, 16, 128), 3), ((3, 128, 75, 25, 64), 3), ((7, 128, 36, 12, 128), 1)])
def test_attention_backward_shares_the_walks_of_one_key_tile(lib, shape, ways):
	"""Causal sequences of 128: the sharing that the whole call was measured to be fastest with (us, whole and shared: 18.9 and 16.7,
	19.0 and 16.4, 21.5 and 19.2, 34.8 and 31.2, 32.5 and 29.4, 37.8 and 40.6)."""
	B, S, Hq, Hkv, D = shape
	more = lib.elf_attn_bwd_shared_workspace_bytes(*shape, 1) - lib.elf_attn_bwd_workspace_bytes(B, S, Hq, D, 1)
	assert more == (ways * 8 * B * S * Hkv * D if ways > 1 else 0)


@pytest.mark.parametrize("shape,ways", [((8, 1408, 6, 2, 128), 3), ((4, 1920, 4, 4, 128), 2), ((10, 512, 12, 4, 128), 3), ((15, 1024, 4, 2, 128), 2), ((2, 384, 48, 16, 128), 3),
                                        ((9, 256, 24, 8, 128), 1), ((1, 256, 12, 12, 128), 1), ((2, 512, 16, 16, 64), 1)])
def test_attention_backward_shares_pairs_of_key_tiles_where_whole_walks_of_one_are_slower(lib, shape, ways):
	"""Causal, pairs of key tiles shared or every tile a whole walk: the faster of the two as measured (us, shared and whole: 161 and
	187, 94.3 and 99.0, 82.3 and 85.5, 111.5 and 115.0, 63.7 and 66.0; the last three 1.20, 1.29 and 1.18 x as fast whole)."""
	B, S, Hq, Hkv, D = shape
	more = lib.elf_attn_bwd_shared_workspace_bytes(*shape, 1) - lib.elf_attn_bwd_workspace_bytes(B, S, Hq, D, 1)
	assert more == (ways * 8 * B * S * Hkv * D if ways > 1 else 0)


def test_attention_backward_refuses_a_workspace_that_is_too_small(lib):
	n = lib.elf_attn_bwd_workspace_bytes(1, 128, 4, 64, 1)
	rc = lib.elf_attn_bwd_shared(*[16] * 10, n - 1, *[64 * 12] * 8, 1, 128, 4, 4, 64, 1, 0.125, None, None)
	assert rc == -1 and str(n).encode() in lib.elf_last_error()


def test_gemm_refuses_rows_too_far_apart_for_its_offsets(lib):
	"""The kernels reach a tile's rows with 32-bit byte offsets: 256 rows of 2^24 elements reach too far, 128 of 2^25,
	64 of 2^26."""
	for cfg, lda, ldb in ((7, 24, 6), (7, 6, 24), (8, 25, 6), (8, 6, 24), (9, 25, 6), (9, 6, 25), (10, 6, 25), (11, 25, 6), (12, 26, 6), (12, 6, 26), (0, 26, 6), (0, 6, 26)):
		rc = lib.elf_gemm_bf16(0, 0, 256, 256, 64, 16, 1 << lda, 16, 1 << ldb, 16, 256, 0, None, 0, cfg, 0, None)
		assert rc == -1 and b"leading dimension too large" in lib.elf_last_error(), (cfg, lda, ldb)
	rc = lib.elf_gemm_bf16(1, 1, 256, 256, 64, 16, 1 << 26, 16, 256, 16, 256, 2, None, 0, 0, 0, None)
	assert rc == -1 and b"leading dimension too large" in lib.elf_last_error()


def test_gemm_of_short_reductions_takes_tiles_of_160_rows_for_a_single_round_only(lib):
	"""The QKV product of a GPT-2-small stage (8192 x 2304 x 768), 468 tiles of 160 rows, is on 192; 1920 x 4800 x 1600, 228 of them, stays,
	and so does the SwiGLU product 15360 x 2 * 1664 x 512.  Over several rounds no plain product with K of at most 1024 takes them;
	longer ones and those with an epilogue (3 SwiGLU, 6 RoPE) do."""
	assert lib.elf_gemm_way(0, 8192, 2304, 768, 0) == 192 << 16 | 256
	assert lib.elf_gemm_way(0, 1920, 4800, 1600, 0) == 160 << 16 | 256
	assert lib.elf_gemm_way(3, 15360, 1664, 512, 0) == 160 << 16 | 256
	rng, seen = random.Random(3), set()
	for _ in range(8000):
		M, N, K = (64 * int(2 ** rng.uniform(0, 7.5)) for _ in range(3))
		for product, cols in ((0, N), (1, N), (3, 2 * N), (6, N)):
			if lib.elf_gemm_way(product, M, N, K, 64) >> 16 == 160:
				seen.add((product, K <= 1024, -(-M // 160) * -(-cols // 256) <= 256))
	assert seen == {(p, short, one) for p in (0, 1, 3, 6) for short in (False, True) for one in (False, True) if one or p > 1 or not short}


def test_stage_create_rejects_bad_configs(lib):
	from elf_amd.execution.block import StageConfig

	h = ctypes.c_void_p()
	bad = [
		dict(arch=7), dict(n_heads=5, n_kv_heads=2), dict(head_dim=96), dict(seq=100), dict(d_model=100),
		dict(arch=0, n_heads=4, n_kv_heads=2),
	]
	base = dict(arch=1, n_blocks=1, d_model=256, n_heads=4, n_kv_heads=2, head_dim=64, ffn=512, seq=128, mb=1, causal=1, eps=1e-5, rope_theta=5e5)
	for delta in bad:
		cfg = StageConfig(**{**base, **delta})
		assert lib.elf_stage_create(ctypes.byref(cfg), ctypes.byref(h)) == -1, delta
		assert lib.elf_last_error()


def _pool(host=True):
	from elf_amd.execution import PinnedHostTensorPool

	return PinnedHostTensorPool(host_backing=host)


def test_pinned_pool_hand_worked_sequence():
	p = _pool()
	a, pa, oa = p.allocate(100, "bf16")        # new parent of 128 elements
	assert (pa, oa) == (0, 0) and p.size() == 128 * 2
	b, pb, ob = p.allocate(20, "bf16")         # carved from the remaining (100, 28)
	assert (pb, ob) == (0, 100) and p.free_segments() == [[(120, 8)]]
	c, pc, oc = p.allocate(9, "bf16")          # does not fit in 8 -> second parent of 16
	assert (pc, oc) == (1, 0) and p.free_segments() == [[(120, 8)], [(9, 7)]]
	assert p.free(a)
	assert p.free_segments()[0] == [(0, 100), (120, 8)]
	d, pd, od = p.allocate(50, "bf16")         # first fit: start of the (0, 100) hole
	assert (pd, od) == (0, 0) and p.free_segments()[0] == [(50, 50), (120, 8)]
	assert p.free(b)                            # (100, 20) merges with both neighbours
	assert p.free_segments()[0] == [(50, 78)]
	e, pe, oe = p.allocate(5, "f32")           # other dtype -> its own parent
	assert (pe, oe) == (2, 0) and p.size() == 128 * 2 + 16 * 2 + 8 * 4
	assert not p.free(12345)                    # foreign blocks are ignored
	for blk in (c, d, e):
		assert p.free(blk)
	assert p.free_segments() == [[(0, 128)], [(0, 16)], [(0, 8)]]
	p.reserve(1000, "f32")                      # ceil(1000/4) = 250 -> 256 elements
	assert p.size() == 128 * 2 + 16 * 2 + 8 * 4 + 256 * 4
	f, pf, of = p.allocate(0, "f32")           # a request of 0 takes 1 element, first fit in parent 2
	assert (pf, of) == (2, 0)


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_pinned_pool_matches_policy_model(seed):
	from oracle.pinned_pool import PoolModel

	rng = random.Random(seed)
	p, m = _pool(), PoolModel()
	live = []
	sizes = {"bf16": 2, "f32": 4}
	for step in range(400):
		if live and rng.random() < 0.45:
			addr, pi, off, n, esz = live.pop(rng.randrange(len(live)))
			assert p.free(addr) and m.free(pi, off)
		else:
			dt = rng.choice(["bf16", "bf16", "f32"])
			n = rng.choice([1, 3, 17, 64, 100, 1000, 4096, rng.randrange(1, 5000)])
			addr, pi, off = p.allocate(n, dt)
			assert (pi, off) == m.allocate(n, dt), f"step {step}"
			live.append((addr, pi, off, n, sizes[dt]))
		assert p.free_segments() == [pp["free"] for pp in m.parents]
		# live blocks never overlap (byte ranges)
		spans = sorted((a, a + n * e) for a, _, _, n, e in live)
		assert all(spans[i][1] <= spans[i + 1][0] for i in range(len(spans) - 1))
	assert p.size() == m.size_bytes(sizes)
	for addr, pi, off, n, esz in live:
		assert p.free(addr)
	assert all(len(s) == 1 and s[0][0] == 0 for s in p.free_segments())
	assert all((s[0][1] & (s[0][1] - 1)) == 0 for s in p.free_segments()), "parent sizes are powers of two"


def _attn_way(lib, shape, causal, ld=None, workspace=None, v=None):
	from elf_amd import kernels

	return kernels.attn_bwd_way(*shape, causal, ld=ld, workspace=workspace, v=v)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_attention_backward_of_128_tokens_whose_rows_lie_far_apart_stays_out_of_one_kernel(lib, D, causal):
	"""The one kernel reaches 128 rows of Q and dO, and of V with heads of 128, with 32-bit byte offsets; the three kernels reach 32 rows of
	Q and dO and any of V."""
	shape, dense = (1, 128, 2, 2, D), 6 * D
	near, far = (((1 << 32) - 512) // 2 // 127) & ~7, 1 << 25
	assert 127 * near * 2 + 512 <= 1 << 32 < 127 * (near + 8) * 2 + 512
	assert _attn_way(lib, shape, causal, ld=(near, near, near))[0] == 0
	for ld in ((near + 8, dense, dense), (dense, dense, near + 8), (far, dense, dense), (dense, dense, far)):
		assert _attn_way(lib, shape, causal, ld=ld)[0] == 128
	for ldv in (near + 8, far):
		assert _attn_way(lib, shape, causal, ld=(dense, ldv, dense))[0] == (0 if D == 64 else 128)


@pytest.mark.parametrize("D", [64, 128])
def test_attention_backward_of_a_misaligned_v_stays_out_of_one_kernel(lib, D):
	"""Heads of 128: the one kernel brings V into LDS in 16-byte pieces, which the kernels of longer sequences do with Q, K and dO only."""
	shape = (1, 128, 2, 2, D)
	assert _attn_way(lib, shape, True, v=1 << 20)[0] == 0
	for off in (2, 4, 8):
		assert _attn_way(lib, shape, True, v=(1 << 20) + off)[0] == (0 if D == 64 else 128)


@pytest.mark.parametrize("given,both", [((), True), (("TORCH_DIR=/nonexistent",), False), (("PYTHON=false",), False)])
def test_the_stage_library_builds_without_pytorch(given, both):
	"""The default target, dry run: where the interpreter has no PyTorch, or one without headers, nothing of libelf_torch.so is asked for."""
	import subprocess
	import sys

	out = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "elf_amd", "csrc"), *(given or (f"PYTHON={sys.executable}",))], capture_output=True, text=True)
	assert out.returncode == 0 and "-o ../libelf_stage.so" in out.stdout
	assert ("allocator.cpp" in out.stdout) == both


def test_an_unusable_torch_library_leaves_the_figures_to_pytorch(monkeypatch, tmp_path):
	"""Missing, no library at all, without the symbols, built for another PyTorch: looked for once, and the caller gets None."""
	import torch

	from elf_amd import _lib

	assert _lib._torch_reader(), "the library that was built here is usable"
	bad = tmp_path / "libelf_torch.so"
	bad.write_bytes(b"no library")
	for path, version in ((str(tmp_path / "none.so"), None), (str(bad), None), (_lib.LIB_PATH, None), (_lib.TORCH_LIB_PATH, "0.0.0")):
		with monkeypatch.context() as m:
			m.setattr(_lib, "TORCH_LIB_PATH", path)
			m.setattr(_lib, "_torch_allocated", None)
			if version:
				m.setattr(torch, "__version__", version)
			assert _lib.torch_allocated(0) is None
			m.setattr(_lib, "_torch_reader", lambda: pytest.fail("looked for again"))
			assert _lib.torch_allocated(0) is None


@pytest.mark.parametrize("T,shapes,way", [
	(2112, [(4288, 1600), (832, 4288)], 256), (512, [(512, 512), (1536, 512), (512, 768)], 128), (256, [(2112, 1024), (384, 2112)], 128),
	(8192, [(1536, 1536), (1536, 256)], 0), (3008, [(1344, 384), (4544, 1344)], 0), (2048, [(4096, 960), (960, 2560)], 0), (4096, [(2048, 2048), (2048, 2048)], 0),
	(4544, [(5824, 7232), (1792, 5824)], 0), (2112, [(4288, 1600), (192, 4288)], 0), (512, [(512, 512)], 0),
])
def test_weight_gradients_share_a_launch_where_the_way_it_takes_is_faster(lib, T, shapes, way):
	"""Lists that the one launch does sooner, on 256x256 and on 128x128 tiles, and lists that it would do later on the tiles it takes (measured:
	123 us for 96, 79 for 68, 66 for 56, 102 for 94), that make more than a round of tiles or hold a layer no such launch takes."""
	from elf_amd.kernels import _LinearW

	layers = (_LinearW * len(shapes))()
	for q, (M, N) in zip(layers, shapes):
		q.dY, q.lddy, q.X, q.ldx, q.acc, q.M, q.N = 1 << 20, M, 1 << 20, N, 1 << 20, M, N
	assert lib.elf_linear_w_way(len(shapes), layers, T) == way


@pytest.mark.parametrize("B,Hq,Hkv,D,causal,one", [
	(32, 32, 8, 128, True, True), (33, 32, 8, 128, True, False), (38, 32, 8, 128, True, False), (40, 32, 8, 128, True, True), (33, 24, 8, 128, True, True), (33, 32, 8, 64, True, True),
	(28, 64, 8, 128, True, True), (32, 64, 8, 128, True, True), (33, 64, 8, 128, True, False), (28, 64, 8, 64, False, True), (32, 64, 8, 128, False, False),
])
def test_attention_backward_of_128_tokens_takes_the_faster_way(lib, B, Hq, Hkv, D, causal, one):
	"""One kernel or three, whichever was measured to be faster on operands past the caches: causal groups of four heads of 128 in a second
	round that is not a quarter full stay with three (264 groups 100.3 us and 104.1)."""
	assert (_attn_way(lib, (B, 128, Hq, Hkv, D), causal)[0] == 0) == one


@pytest.mark.parametrize("shape,way", [((2, 384, 44, 22, 128), (128, 1, 1, False)), ((18, 256, 16, 4, 128), (128, 1, 1, False)), ((11, 256, 12, 2, 128), (128, 3, 1, False)),
                                       ((2, 384, 48, 6, 128), (128, 4, 1, False)), ((6, 256, 48, 12, 128), (128, 1, 1, False))])
def test_attention_backward_shares_no_walks_into_a_second_round_that_is_nearly_empty(lib, shape, way):
	"""Causal, heads of 128, a few single key tiles more than compute units: the sharing before is faster as measured (us, shared into 264 and 288
	workgroups and as here: 61.2 and 55.4, 76.4 and 73.3, 58.2 and 50.0, 63.9 and 60.7, 77.6 and 73.1)."""
	assert _attn_way(lib, shape, True) == way


@pytest.mark.parametrize("shape,way", [((6, 512, 16, 2, 128), (128, 4, 1, False)), ((15, 768, 2, 1, 128), (128, 2, 1, False)), ((2, 512, 48, 12, 128), (128, 2, 1, False))])
def test_attention_backward_shares_short_walks_over_several_rounds_where_that_is_clearly_faster(lib, shape, way):
	"""Causal, heads of 128, up to six key tiles: shared further, into 360 and 384 workgroups, these took 83.3 us for 75.5, 60.1 for 56.1 and 77.6
	for 73.8."""
	assert _attn_way(lib, shape, True) == way


@pytest.mark.parametrize("shape,keys", [((3, 896, 24, 24, 64), 128), ((11, 1152, 5, 5, 64), 128), ((6, 640, 17, 17, 64), 128), ((13, 1664, 3, 1, 64), 128), ((4, 896, 68, 17, 64), 128),
                                        ((11, 384, 25, 25, 64), 128), ((9, 384, 15, 5, 64), 128),
                                        ((6, 384, 48, 12, 64), 256), ((1, 1152, 26, 13, 64), 256), ((12, 2688, 6, 2, 64), 256), ((3, 896, 21, 21, 64), 256), ((3, 896, 30, 30, 64), 256)])
def test_attention_backward_without_a_mask_makes_one_round_of_128_keys_rather_than_a_bit_more_of_256(lib, shape, keys):
	"""Heads of 64: 476 to 510 workgroups of 128 keys fit the chip at once, 272 to 306 of 256 keys do not (us: 75.8 and 93.0, 89.3 and 107, 62.6 and
	74.9, 125 and 148, 245 and 264).  384 tokens likewise for two rounds of the one and three of the other (80.5 and 89.6)."""
	assert _attn_way(lib, shape, False)[0] == keys


@pytest.mark.parametrize("shape,keys", [((1, 1024, 2, 2, 64), 128), ((2, 1024, 4, 1, 64), 128), ((1, 1280, 4, 1, 64), 128), ((1, 640, 24, 8, 64), 128), ((1, 896, 6, 6, 64), 128),
                                        ((5, 896, 2, 2, 64), 256), ((1, 640, 30, 10, 64), 256), ((1, 1408, 1, 1, 64), 256), ((8, 1024, 12, 12, 64), 256)])
def test_attention_backward_of_little_work_without_a_mask_stays_with_128_keys_a_pass(lib, shape, keys):
	"""Heads of 64: passes over 256 keys where they were measured to be no slower (us, 128 and 256 keys: 23.4 and 25.6, 31.9 and 33.7, 33.3 and
	34.0, 33.6 and 35.9, 27.4 and 28.1; 33.7 and 30.5, 39.7 and 34.1)."""
	assert _attn_way(lib, shape, False)[0] == keys
