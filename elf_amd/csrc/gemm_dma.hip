// Direct-to-LDS GEMMs (gemm_dma_tile.h): the grouped weight gradients of a W pass, the persistent forward kernel and the
// dispatch over layouts, tiles and epilogues.
#include "gemm_dma_tile.h"

namespace elf {

namespace dma {

// Several weight gradients in one launch (the W pass of a stage: every linear layer's dW += dY^T X over the same
// tokens).  The chip's workgroup slots refill across problem boundaries, so only the launch's last round is partly
// filled, and small problems that would each need their tiles split many ways to fill the chip fill it together.
//  * compact = 0 (a problem of 256 tiles or more among them): the workgroups of problem p are first[p] .. first[p] +
//    count[p] - 1, each first[p] a multiple of 8 so that a workgroup's index within its problem names its XCD as in a
//    launch of its own (the workgroups in the gaps leave at once); every problem keeps its own walk and its own tail.
//  * compact = 1 (small problems only): the tiles of all problems form one sequence (problem after problem, down the
//    rows first; first[p] = problem p's first tile in it) and XCD x takes a contiguous eighth of its whole tiles, then
//    of its split tiles with the `splits` workgroups of a tile side by side: the 32 tiles an XCD holds at a time are
//    neighbours that share their operand slabs in its L2 (taken in launch order, neighbouring tiles of a 3-row problem
//    land on different XCDs and every slab is fetched by all eight).
constexpr int GROUP_MAX = DW_GROUP_MAX;
struct GroupArgs {
	int n, compact;
	int tiles, tail, splits;  // compact: all tiles of the launch, how many of the last are split, and how many ways
	uint32_t turn_base;
	int first[GROUP_MAX], count[GROUP_MAX];
	Args a[GROUP_MAX];
};
template <int EPI, bool EDGE>
__global__ __launch_bounds__(512) void gemm_dw_group_kernel(GroupArgs ga) {
	int p = 0, pid, ksplit = 0, splits = 1, turn_slot = 0;
	if (ga.compact) {
		const int x = blockIdx.x & 7, slot = blockIdx.x >> 3;
		const int full = ga.tiles - ga.tail, chunk_f = (full + 7) >> 3, chunk_t = (ga.tail + 7) >> 3;
		int gt;
		if (slot < chunk_f) {
			gt = x * chunk_f + slot;
			if (gt >= full) return;
		} else {
			const int q = slot - chunk_f, tt = x * chunk_t + q / ga.splits;
			if (tt >= ga.tail) return;
			gt = full + tt;
			ksplit = q % ga.splits;
			splits = ga.splits;
			turn_slot = (int)(((uint32_t)tt + ga.turn_base) % (uint32_t)TURN_TILES);
		}
		for (int i = 1; i < ga.n; i++)
			if (gt >= ga.first[i]) p = i;
		p = __builtin_amdgcn_readfirstlane(p);
		pid = gt - ga.first[p];
	} else {
		for (int i = 1; i < ga.n; i++)
			if ((int)blockIdx.x >= ga.first[i]) p = i;
		p = __builtin_amdgcn_readfirstlane(p);
		const int bid = (int)blockIdx.x - ga.first[p];
		if (bid >= ga.count[p]) return;
		locate_tile(ga.a[p], bid, pid, ksplit, splits, turn_slot);
	}
	gemm_dma_tile<8, 4, true, true, EPI, EDGE>(ga.a[p], pid, ksplit, splits, turn_slot);
}

// The split tiles of a launch with the scaling accumulate epilogue: their workgroups add partial sums and none of them
// holds the finished tile, so the scale and the bf16 copy of those (few, at most 128) tiles are applied here, behind the
// GEMM on the same stream.  Eight workgroups per tile (32 rows each); tile index and origin as in the GEMM.
__global__ __launch_bounds__(256) void scale_tail_kernel(Args g) {
	const int ntiles = g.tiles_m * g.tiles_n;
	const int pid = ntiles - g.tail_tiles + (int)(blockIdx.x >> 3);
	int m0, n0;
	tile_origin<256>(g, pid, m0, n0);
	m0 += (int)(blockIdx.x & 7) * 32;
	float* C = reinterpret_cast<float*>(g.C);
	for (int i = threadIdx.x; i < 32 * 64; i += 256) {
		const int row = i >> 6, c4 = (i & 63) * 4;
		if (m0 + row >= g.M || n0 + c4 >= g.N) continue;  // ragged sizes
		float* c = C + (int64_t)(m0 + row) * g.ldc + n0 + c4;
		f32x4 v = *reinterpret_cast<const f32x4*>(c);
		v *= g.scale;
		bf16x4 o;
#pragma unroll
		for (int t = 0; t < 4; t++) o[t] = (bf16_t)v[t];
		*reinterpret_cast<f32x4*>(c) = v;
		*reinterpret_cast<bf16x4*>(g.C2 + (int64_t)(m0 + row) * g.ldc2 + n0 + c4) = o;
	}
}

// dW: both operands reduction-major
template <int NW, int RF>
static int launch_tt(const Args& a, int epi, hipStream_t stream) {
	switch (epi) {
		case EPI_BF16: return launch<NW, RF, true, true, EPI_BF16>(a, stream);
		case EPI_BF16_RESID: return launch<NW, RF, true, true, EPI_BF16_RESID>(a, stream);
		case EPI_F32_ACC: return launch<NW, RF, true, true, EPI_F32_ACC>(a, stream);
		case EPI_F32_STORE: return launch<NW, RF, true, true, EPI_F32_STORE>(a, stream);
	}
	if constexpr (NW == 8) {
		if (epi == EPI_F32_ACC_SCALE) return launch<NW, RF, true, true, EPI_F32_ACC_SCALE>(a, stream);
	}
	set_error("gemm: unknown epilogue %d", epi);
	return -1;
}

}  // namespace dma

// Waves of this file's kernels that stopped waiting for their turn since the library was loaded (this device).
int dma_turn_giveups(uint64_t* out) {
	*out = 0;
	if (int rc = dma::add_turn_giveups(out)) return rc;
	if (int rc = dma::rr_turn_giveups(out)) return rc;
	return dma::rt_turn_giveups(out);
}

// Arguments are validated by gemm_bf16() before it dispatches here.
int gemm_bf16_dma(int a_t, int b_t, int M, int N, int K, const void* A, int64_t lda, const void* B, int64_t ldb, void* C,
                  int64_t ldc, int epi, const void* R, int64_t ldr, int k_splits, int tail_tiles, int bm, hipStream_t stream,
                  void* C2, int64_t ldc2, const void* rope_cs, int rope_S, int rope_cols, int rope_D, float scale, int bn) {
	ELF_REQUIRE(bm == 256 || bm == 128 || (!a_t && gemm_mid_rows(bm)), "gemm (dma tile): 256- or 128-row tiles, 160, 192 or 224 rows with a k-contiguous A");
	ELF_REQUIRE(bn == dma::BN || (bn == 192 && !a_t && bm == 128 && (epi == EPI_BF16 || epi == EPI_BF16_RESID)),
	            "gemm (dma tile): 256 columns, 192 with 128 rows of a k-contiguous A and a bf16 output");
	ELF_REQUIRE(M >= bm && N >= bn && M % 64 == 0 && N % 64 == 0 && K % dma::BKS == 0, "gemm (dma tile): M at least %d, N at least %d, all sizes multiples of 64", bm, bn);
	const int tiles_m = (M + bm - 1) / bm, tiles_n = (N + bn - 1) / bn, ntiles = tiles_m * tiles_n;
	ELF_REQUIRE(gemm_reaches(a_t ? dma::BKS : bm, lda) && gemm_reaches(b_t ? dma::BKS : bn, ldb), "gemm (dma tile): leading dimension too large (%lld, %lld)", (long long)lda, (long long)ldb);
	// a tile's columns are taken in heads: the last one may only move back by whole heads
	ELF_REQUIRE(epi != EPI_BF16_ROPE || N % rope_D == 0, "gemm (dma tile): the RoPE epilogue needs N to be a multiple of the head width");
	ELF_REQUIRE(epi != EPI_BF16_SWIGLU || (C2 && !a_t && !b_t), "gemm (dma tile): the SwiGLU epilogue needs k-contiguous operands and a second output");
	// the paired rows of the SwiGLU epilogue are addressed with 32-bit byte offsets from the tile's first row
	ELF_REQUIRE(epi != EPI_BF16_SWIGLU || (int64_t)(N / 2 + 256) * ldb * 2 < (int64_t(1) << 31), "gemm (dma tile): weight too large for the paired-row epilogue");
	ELF_REQUIRE(epi != EPI_F32_ACC_SCALE || (C2 && a_t && b_t && bm == 256), "gemm (dma tile): the scaling accumulate epilogue needs reduction-major operands, 256-row tiles and a bf16 output");
	ELF_REQUIRE(epi != EPI_BF16_ROPE || (rope_cs && rope_S > 0 && !a_t && !b_t && (rope_D == 64 || rope_D == 128) && rope_cols % rope_D == 0 && rope_cols <= N),
	            "gemm (dma tile): the RoPE epilogue needs k-contiguous operands, a table and heads of 64 or 128 columns");
	dma::Args a{(const bf16_t*)A, (const bf16_t*)B, C, (const bf16_t*)R, (bf16_t*)C2, lda, ldb, ldc, ldr, ldc2, M, N, K, tiles_m, tiles_n, k_splits < 1 ? 1 : k_splits,
	            tail_tiles < 0 || tail_tiles > ntiles ? ntiles : tail_tiles, 0, (const float2*)rope_cs, rope_S, rope_cols, rope_D, 0, scale};
	// The band walk fetches every row slab of A from HBM in one round only and B once per band; the default
	// walk wants A in the 256 MB memory-side cache for the whole launch and streams B once.  Inside the stage's
	// stream (operands cold, per-shape times from a kernel trace) the bands are 0-5 % faster on every shape but
	// the one with a small A and a B beyond that cache (gate/up projection forward, 67 MB against 235 MB: 2 %
	// slower), which keeps the default.
	const int64_t big = int64_t(160) << 20;
	a.walk = !((int64_t)M * K * 2 < big && (int64_t)N * K * 2 >= big);
	if ((epi != EPI_F32_ACC && epi != EPI_F32_ACC_SCALE) || a.k_splits == 1) a.k_splits = 1, a.tail_tiles = 0;
	// split tiles add in a fixed order (bit-reproducible weight gradients) as long as each has a counter of its own
	a.turn_tag = a.tail_tiles > 0 && a.tail_tiles <= dma::TURN_TILES ? next_turn_tag() : 0;
	a.turn_base = a.turn_tag * 977u;  // consecutive launches on different counters
	if (a_t && !b_t) {
		set_error("gemm: layout A=T,B=R is not used by any stage contraction");
		return -1;
	}
	// k-contiguous A (forward, dX): four waves with 128x128 wave tiles; both operands reduction-major (dW): eight
	// waves with 64x128 wave tiles (with two transpose reads per fragment on both operands the lone wave wins on
	// some shapes by 2-3 % and loses on most by 1-10 %)
	if (!a_t && b_t) return dma::launch_rt(bm, bn, a, epi, stream);
	if (!a_t && bm == 256 && bn == 256 && K / dma::BKS >= 2 && (epi == EPI_BF16 || epi == EPI_BF16_RESID || epi == EPI_BF16_SWIGLU) && !getenv("ELF_NO_PERSISTENT_GEMM")) {
		// forward shapes: persistent workgroups, register epilogue (the QKV projection with its rotary epilogue stays on the
		// one-tile kernel: with the table fetches in a lone wave's register epilogue the persistent form ran 3 % slower)
		return dma::launch_pers(a, epi, stream);
	}
	if (!a_t) return dma::launch_rr(bm, bn, a, epi, stream);
	if (bm == 128) return dma::launch_tt<4, 4>(a, epi, stream);
	if (int rc = dma::launch_tt<8, 4>(a, epi, stream)) return rc;
	if (epi == EPI_F32_ACC_SCALE && a.tail_tiles > 0) {
		ELF_LAUNCH(dma::scale_tail_kernel, dim3(a.tail_tiles * 8), dim3(256), 0, stream, a);
		ELF_CHECK_HIP(hipGetLastError());
	}
	return 0;
}

bool gemm_dw_groupable(int M, int N, int K, const void* dY, int64_t lddy, const void* X, int64_t ldx, const void* acc) {
	return M >= 256 && N >= dma::BN && K > 0 && gemm_reaches(dma::BKS, lddy) && gemm_reaches(dma::BKS, ldx) && M % 64 == 0 && N % 64 == 0 && K % dma::BKS == 0 && lddy % 8 == 0 && ldx % 8 == 0 && lddy >= M && ldx >= N &&
	       ((uintptr_t)dY % 16) == 0 && ((uintptr_t)X % 16) == 0 && ((uintptr_t)acc % 16) == 0;
}

DwGroupWay gemm_dw_group_way(int n, const DwProblem* pr, int K) {
	DwGroupWay w;
	int64_t small = 0;
	for (int i = 0; i < n; i++) {
		w.tiles += (int64_t)((pr[i].M + 255) / 256) * ((pr[i].N + dma::BN - 1) / dma::BN);
		small += (int64_t)((pr[i].M + 127) / 128) * ((pr[i].N + 127) / 128);
	}
	// Whole tiles, one workgroup each, except in the launch's last round: when that round would fill at most half of the
	// chip, its tiles (the last ones of the last problems) are split along K so that proportionally shorter workgroups
	// fill it - at least 16 K slices each, and no more than 8 ways (the splits of a tile add with atomics, one after the
	// other: past that their adds cost more than the idle compute units).
	const int nk = K / dma::BKS;
	if (const int rem = (int)(w.tiles % 256); rem != 0 && rem <= 128 && rem <= dma::TURN_TILES) {
		w.splits = 256 / rem < 8 ? 256 / rem : 8;
		while (w.splits > 1 && nk / w.splits < 16) w.splits--;
		if (w.splits > 1) w.tail = rem;
	}
	// Little work: where the layers make no more than a round of 128x128 tiles, these are done sooner than a few 256x256 ones (us,
	// without and with the splits of the latter; fitted to launches over 128 to 8192 tokens).  Two blocks of a 512-wide Llama stage
	// over 512 tokens 23.7 -> 12.7 us, of a 256-wide GPT stage 21.4 -> 10.8, one over 2048 tokens 33.5 -> 18.4; with two rounds it
	// is one or the other (four layers of 768 over 1024 tokens 33.8 and 29.4, eight of 512 33.5 and 34.7).
	w.small = small <= 256 && nk * 0.35f + 7.5f < (float)((nk + w.splits - 1) / w.splits) * 1.05f + 12.f + 2.f * (w.splits - 1);
	return w;
}

int gemm_dw_group(int n, const DwProblem* pr, int K, float scale, hipStream_t stream) {
	ELF_REQUIRE(n > 0 && n <= dma::GROUP_MAX && pr, "gemm_dw_group: 1..%d problems", dma::GROUP_MAX);
	double flops = 0;
	bool edge = false;
	auto tiles_of = [](const DwProblem& q) { return ((q.M + 255) / 256) * ((q.N + dma::BN - 1) / dma::BN); };
	for (int i = 0; i < n; i++) {
		ELF_REQUIRE(pr[i].dY && pr[i].X && pr[i].acc && gemm_dw_groupable(pr[i].M, pr[i].N, K, pr[i].dY, pr[i].lddy, pr[i].X, pr[i].ldx, pr[i].acc),
		            "gemm_dw_group: problem %d (M=%d N=%d K=%d) needs M, N of at least 256, all sizes multiples of 64 and 16-byte aligned operands", i, pr[i].M, pr[i].N, K);
		ELF_REQUIRE(scale == 0.f || (pr[i].grad_bf16 && ((uintptr_t)pr[i].grad_bf16 % 8) == 0), "gemm_dw_group: a scaling pass needs the bf16 gradient buffers");
		edge = edge || pr[i].M % 256 || pr[i].N % dma::BN;
		flops += 2.0 * pr[i].M * pr[i].N * K;
	}
	const DwGroupWay way = gemm_dw_group_way(n, pr, K);
	if (way.small) {
		ProfScope prof(PROF_GEMM, flops, stream);
		return gemm_ring_dw_group(n, pr, K, scale, stream);
	}
	const int64_t tiles = way.tiles;
	const int splits = way.splits, tail = way.tail;
	dma::GroupArgs ga{};
	ga.n = n;
	ga.compact = 1;
	for (int i = 0; i < n; i++)
		if (tiles_of(pr[i]) >= 256) ga.compact = 0;
	ga.tiles = (int)tiles, ga.tail = tail, ga.splits = splits;
	const uint32_t tag = tail ? next_turn_tag() : 0;
	uint32_t turn_base = tag * 977u;
	ga.turn_base = turn_base;
	const int64_t big = int64_t(160) << 20;
	int64_t before = 0;  // tiles of the problems ahead of this one
	int next = 0;
	for (int i = 0; i < n; i++) {
		const DwProblem& q = pr[i];
		const int ntiles = tiles_of(q);
		// this problem's share of the launch's last `tail` tiles
		const int64_t tail_from = tiles - tail;
		const int tail_i = before + ntiles <= tail_from ? 0 : (int)(before + ntiles - (tail_from > before ? tail_from : before));
		dma::Args& a = ga.a[i];
		a = dma::Args{(const bf16_t*)q.dY, (const bf16_t*)q.X, q.acc, nullptr, (bf16_t*)q.grad_bf16, q.lddy, q.ldx, q.N, 0, q.N, q.M, q.N, K, (q.M + 255) / 256, (q.N + dma::BN - 1) / dma::BN,
		              tail_i ? splits : 1, tail_i, 0, nullptr, 0, 0, 0, tail_i ? tag : 0, scale, turn_base};
		a.walk = ga.compact ? 2 : !((int64_t)q.M * K * 2 < big && (int64_t)q.N * K * 2 >= big);
		turn_base += (uint32_t)tail_i;
		ga.first[i] = ga.compact ? (int)before : next;
		ga.count[i] = ntiles + tail_i * (splits - 1);
		next += (ga.count[i] + 7) & ~7;
		before += ntiles;
	}
	if (ga.compact) next = 8 * (int)((tiles - tail + 7) / 8 + (tail + 7) / 8 * splits);
	{
		ProfScope prof(PROF_GEMM, flops, stream);
		using Sh = dma::Shape<8, 4>;
		constexpr int ring = Sh::RING_BYTES, epi = 8 * 32 * 136 * 4;
		constexpr int smem = ring > epi ? ring : epi;
		auto kern = scale != 0.f ? (edge ? dma::gemm_dw_group_kernel<EPI_F32_ACC_SCALE, true> : dma::gemm_dw_group_kernel<EPI_F32_ACC_SCALE, false>)
		                         : (edge ? dma::gemm_dw_group_kernel<EPI_F32_ACC, true> : dma::gemm_dw_group_kernel<EPI_F32_ACC, false>);
		static bool attr_set[2][2] = {};
		if (bool& set = attr_set[scale != 0.f][edge]; !set) {
			ELF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
			set = true;
		}
		ELF_LAUNCH(kern, dim3(next), dim3(512), smem, stream, ga);
		ELF_CHECK_HIP(hipGetLastError());
	}
	// split tiles have no single epilogue that could scale them: a small kernel behind the launch does those
	if (scale != 0.f)
		for (int i = 0; i < n; i++)
			if (ga.a[i].tail_tiles > 0) {
				ELF_LAUNCH(dma::scale_tail_kernel, dim3(ga.a[i].tail_tiles * 8), dim3(256), 0, stream, ga.a[i]);
				ELF_CHECK_HIP(hipGetLastError());
			}
	return 0;
}

}  // namespace elf
