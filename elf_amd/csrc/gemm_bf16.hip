// Dispatch of the bf16 GEMM: C[M,N] (+)= sum_k A(m,k) * B(n,k), fp32 accumulation.
//
// The three contractions of a linear layer under the split backward:
//   forward  Y  = X  . W^T   A = X  [M,K] k-contiguous ("R"), B = W  [N,K] k-contiguous ("R")
//   dX       dX = dY . W     A = dY [M,K] k-contiguous ("R"), B = W  [K,N] n-contiguous ("T")
//   dW       dW += dY^T . X  A = dY [K,M] m-contiguous ("T"), B = X  [K,N] n-contiguous ("T")
// (reference semantics: elf/zb_utils.py:20 forward, :34-37 dX, :235-244 dW accumulate).
//
// The kernels are in gemm_dma_tile.h and gemm_dma_pers.hip (128 to 256 rows by 256 columns, 128x192) and gemm_ring.hip (128x128 .. 32x32
// tiles); all of them
// add the products of an output in the same order, so the choice of a tile never changes its bits (a split of K does).
#include <algorithm>
#include <atomic>

#include "common.h"
#include "kernels.h"

namespace elf {

constexpr int BK = 64;

// One sequence of tags for every launch of every GEMM kernel that splits tiles: a counter value left behind by any
// earlier launch then never equals a value a later launch waits for.
uint32_t next_turn_tag() {
	static std::atomic<uint32_t> launch_tag{0};
	return (launch_tag.fetch_add(1) % 0xFFFFFFu) + 1;
}
int dma_turn_giveups(uint64_t* out);   // gemm_dma.hip
int ring_turn_giveups(uint64_t* out);  // gemm_ring.hip
// Split-K workgroups / waves (both GEMM kernel families, this device) that stopped waiting for their turn and added out
// of turn since the library was loaded: the sums are right, only bit-reproducibility lapsed for those launches.
int gemm_turn_giveups(uint64_t* out) {
	uint64_t d = 0, r = 0;
	if (int rc = dma_turn_giveups(&d)) return rc;
	if (int rc = ring_turn_giveups(&r)) return rc;
	*out = d + r;
	return 0;
}

// ------------------------------------------------------------------------------------------
// Tile choice.  Estimated time of a product on tiles of bm x bn: rounds of 256 workgroups (one per compute unit) times the
// time of a K slice of 64 times the slices and what a round costs besides (filling the ring, the epilogue), plus what a launch
// costs once.  The constants are microseconds fitted to timings of every tile on some 10000 shapes (sizes spread over the
// logarithm from 64 to 16384, operands rotated through 1 GB).  For K beyond RING_SHORT_K the bf16 constants come from 226 of
// them: the tile that is picked takes 0.4 % longer than the best one on average, and more than 7 % longer for 5 of the 226.
// A large tile has the cheaper products (per slice and output: 18 ps on 256x256, 23 on 128x256, 30 on 128x128, 52 on 64x64: the
// smaller the tile, the more operand bytes go through the 64 B/clk path into LDS for each product) and loses where its tiles leave
// compute units idle.  The tiles of 160, 192 and 224 rows are for sizes of which 256-row tiles leave a round partly empty and
// 128-row ones make twice the rounds (without them the best tile takes 2.9 % longer on average): before -> after (us)
//   2688 x 4096 x 28672 (a Llama-3-8B block's input gradient over 3 x 896 tokens) 504 on 176 tiles of 256 rows, 463 on 224 of 192;
//   2688 x 4096 x 14336 with a residual 266 -> 231, 1920 x 4800 x 1600 32.1 on 152 tiles, 28.0 on 228 of 160,
//   8192 x 2304 x 768 42.4 on 288 tiles of 256 rows, 40.2 on 387 of 192, 4096 x 5504 x 2048 with the SwiGLU backward 131 on 352
//   tiles of 256 rows, 117 on 484 of 192; 1920 x 1600 x 1600 stays on 195 tiles of 128x128 (14.6; 24 on 84 of 160 rows).
// 160-row tiles fetch 30 % more operand bytes a product than 256-row ones (192: 17 %), which a stream at the power limit pays for in
// its other kernels.  For K of at most 1024 they are taken where the launch is one round: with the QKV product on 468 of them
// (39.0 us alone) a GPT-2-small stage took 8.06 ms where it takes 7.97 with 192 rows, on parts that clock low; 7.69 and 7.70 on others.
// For a longer K 192 rows take 5 to 10 % longer, and a Llama-3-8B block of 2688 tokens is as fast with either; with the rotary or SwiGLU
// epilogue the other tiles cost a stage more than that (three Llama blocks of 512 over 2 x 7680 tokens 7.31 ms, 7.35 with 256 rows).
struct TileTime {
	int bm, bn;
	float slice, round, launch;
};
static constexpr TileTime TILES_BF16[] = {{256, 256, 1.18f, 6.f, 0.f}, {128, 256, 0.739f, 5.f, 0.f}, {128, 128, 0.487f, 2.9f, 0.4f}, {64, 128, 0.32f, 2.2f, 0.9f},
                                          {128, 64, 0.341f, 1.9f, 1.f}, {64, 64, 0.213f, 1.5f, 1.3f}};
// the tiles between 128 and 256 rows (k-contiguous A and bf16 outputs only)
static constexpr TileTime TILES_MID[] = {{224, 256, 1.01f, 11.1f, 0.f}, {192, 256, 0.938f, 6.5f, 0.f}, {160, 256, 0.854f, 6.2f, 0.f}};
// 128x192: a k-contiguous A, bf16 outputs, no more tiles than compute units.  Outputs of which 128x256 tiles leave compute units idle (64 x 3
// of them for 8192 x 768) and 128x128 ones make a second round.  Best tile before -> now, k-contiguous B / reduction-major B (us): 8192 x 768 x
// 768 14.6 -> 13.7 / 15.0 -> 14.6, x 3072 42.3 -> 38.8 / 41.5 -> 39.1, 896 x 6208 x 4160 66.6 -> 61.3 / 64.4 -> 60.3, 2560 x 1664 x 320 9.3 ->
// 8.4 / 9.8 -> 8.8.  More than a round of them gained nothing on 25 sizes (15 % more operand bytes a product than 128x256), and
// 256x192 tiles nothing on 59 of 60.
static constexpr TileTime TILE_192 = {128, 192, 0.68f, 5.1f, 0.f};
// K of at most RING_SHORT_K: the small tiles on the ring of two slices
static constexpr TileTime TILES_SHORT[] = {{256, 256, 1.293f, 7.15f, 2.5f}, {128, 256, 0.996f, 4.9f, 0.44f}, {128, 128, 0.388f, 1.94f, 3.5f},
                                                  {64, 128, 0.285f, 0.93f, 3.7f}, {128, 64, 0.325f, 1.0f, 2.4f}, {64, 64, 0.184f, 0.55f, 2.9f}};
// 32x32 tiles, K beyond RING_SHORT_K and up to it: a k-contiguous A, bf16 outputs, no more tiles than compute units.  A slice of the 64x64
// tile is 16 KB through a compute unit's path into LDS, one of these 8, and four times as many units take part.  GPU time alone, 64x64 ->
// 32x32 (us): 512 x 512 x 1536 7.4 -> 4.8 (B reduction-major 7.7 -> 6.0), 512 x 512 x 512 4.2 -> 3.4, 512 x 256 x 1024 5.1 -> 3.9, 128 x
// 256 x 64 2.8 -> 2.6; with two rounds of them 1024 x 512 x 1024 5.8 and 5.6 (reduction-major 6.1 and 6.6), 768 x 768 x 768 5.3 and 6.9.
static constexpr TileTime TILE_TINY = {32, 32, 0.11f, 1.2f, 1.3f}, TILE_TINY_SHORT = {32, 32, 0.1f, 0.5f, 2.9f};
// weight gradients: both operands reduction-major, fp32 read-modify-write of the output
static constexpr TileTime TILES_F32[] = {{256, 256, 1.3f, 22.f, 0.f}, {128, 256, 0.757f, 12.9f, 0.f}, {128, 128, 0.537f, 9.9f, 0.f},
                                                {64, 128, 0.442f, 5.9f, 0.f}, {128, 64, 0.416f, 7.5f, 0.f}, {64, 64, 0.26f, 4.f, 0.f}};

struct Plan {
	int bm = 0, bn = 0, k_splits = 1;
	float us = 1e30f;
	bool dma() const { return bn >= 192; }
};

static float tile_us(const TileTime& t, int M, int N, int slices, int k_splits = 1) {
	const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * k_splits;
	const float rounds = (float)((tiles + 255) / 256);
	return rounds * ((slices + k_splits - 1) / k_splits * t.slice + t.round) + t.launch;
}

// The tile of a bf16 output with the smallest estimate.  mid: the tiles between 128 and 256 rows are to be had, plain: those of
// 32x32 and 128x192 (left out where a product and a pass are weighed against a fused epilogue, which saves more than those tiles do).  For an epilogue
// that only the 256-column tiles have: epi_extra, its time per round of 256x256 tiles, and ring_extra, the time of the pass of its
// own that the small ring tiles need instead.
static Plan plan_tiles(int M, int N, int K, bool mid = true, float ring_extra = 0.f, float epi_extra = 0.f, bool plain = false) {
	Plan best;
	auto weigh = [&](TileTime t) {
		if (M < t.bm || N < t.bn) return;
		if (t.bn == 256) t.round += epi_extra * t.bm / 256;
		const float us = tile_us(t, M, N, K / BK) + (t.bn == 256 ? 0.f : ring_extra);
		if (us < best.us) best = Plan{t.bm, t.bn, 1, us};
	};
	if (plain && (int64_t)(M / 32) * (N / 32) <= 256) weigh(K <= RING_SHORT_K ? TILE_TINY_SHORT : TILE_TINY);
	if (K <= RING_SHORT_K) {
		for (const TileTime& t : TILES_SHORT) weigh(t);
		return best;
	}
	for (const TileTime& t : TILES_BF16) weigh(t);
	if (plain && (int64_t)((M + 127) / 128) * ((N + 191) / 192) <= 256) weigh(TILE_192);
	if (mid)
		for (const TileTime& t : TILES_MID)
			if (t.bm > 160 || K > 1024 || epi_extra > 0.f || (int64_t)((M + 159) / 160) * ((N + 255) / 256) <= 256) weigh(t);
	return best;
}

// Weight gradients, with K split up to max_splits ways where that fills the chip.  The splits of a tile add with atomics, one
// after the other: 2 us per split, and more on the ring's tiles, which take a whole tile's turn at a time, and for a large output.
// Only 128x256 tiles used to be split since the register-staged kernel went; before -> after splitting them all (us):
// 256 x 704 x 14080 68 -> 31, 512 x 384 x 10112 54 -> 26, 64 x 5632 x 13696 83 -> 53, 1536 x 192 x 12608 68 -> 39.
static Plan plan_weight_gradient(int M, int N, int K, int max_splits = 16) {
	Plan best;
	for (const TileTime& t : TILES_F32) {
		if (M < t.bm || N < t.bn) continue;
		const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
		// (what was measured: three slices or more a split, little more than two rounds of workgroups)
		for (int ks = 1; ks <= max_splits && (ks == 1 || (K / BK / ks >= 3 && tiles * ks <= 600)); ks++) {
			const float add = ks == 1 ? 0.f : t.bn == 256 ? ks * (1.6f + 1.3e-6f * (float)M * N) : ks * (2.2f + 1.2e-4f * t.bm * t.bn + 7.4e-6f * (float)M * N);
			const float us = tile_us(t, M, N, K / BK, ks) + add;
			if (us < best.us) best = Plan{t.bm, t.bn, ks, us};
		}
	}
	return best;
}

// ring_extra of a product that a ring tile cannot do
constexpr float NO_RING = 1e20f;
// what a pass of its own over `bytes` costs (5 TB/s and a launch)
static float pass_us(double bytes) { return 2.f + (float)(bytes / 5e6); }
// Estimate for 64x64 ring tiles with an epilogue of `extra` us a round.  From K = 256 up, the narrowest a stage was measured at;
// below, products and passes stay apart.
static float small_us(int M, int N, int K, float extra) {
	TileTime t = K <= RING_SHORT_K ? TILES_SHORT[5] : TILES_BF16[5];
	t.round += extra;
	return M < 64 || N < 64 || M % 64 || N % 64 || K % BK || K < 256 ? 1e30f : tile_us(t, M, N, K / BK);
}
// What an epilogue adds to a round of 64x64 tiles.  Of the smallest products a pass of its own costs more than that whatever its
// size: a launch, 3 us on the GPU and as much on the host.  Product and pass, before -> after on one kernel (us): SwiGLU 512 x 768
// x 512 (M x F x K) 7.3 -> 5.3 and its backward 7.6 -> 6.3, GELU 512 x 1024 x 256 6.5 -> 5.6, RoPE 512 x 1024 x 512 7.2 -> 5.2;
// with more than a round of tiles the larger ones and a pass are as fast: GELU 1024 x 2048 x 512 11.5 and 11.4.
constexpr float SMALL_SWIGLU_US = 0.5f, SMALL_ROPE_US = 0.5f, SMALL_GELU_US = 1.2f, SMALL_GELU_BWD_US = 1.8f, SMALL_SWIGLU_BWD_US = 1.6f;
// what an epilogue adds to a round of 256x256 tiles (half of it to one of 128x256)
constexpr float SWIGLU_FWD_US = 4.f, ROPE_US = 5.f;

// K split of a weight gradient on 256x256 direct-to-LDS tiles when the caller leaves it open: *k_splits ways for the last
// *tail_tiles tiles (-1: all of them).
static void dw_split_plan(int M, int N, int K, int* k_splits, int* tail_tiles) {
	const int64_t tiles = (int64_t)((M + 255) / 256) * ((N + 255) / 256);
	const int nk = K / 64;
	*k_splits = 1;
	*tail_tiles = -1;
	if (tiles < 256) {
		// too few tiles for the chip: split them all, down to 32 slices per workgroup (shorter
		// ranges pay more in pipeline fill and atomics than the extra workgroups bring)
		while (tiles * *k_splits * 2 <= 256 && nk / (*k_splits * 2) >= 32 && *k_splits < 16) *k_splits *= 2;
	} else if (const int rem = (int)(tiles % 256); rem != 0 && rem <= 128) {
		// the last round of workgroups would leave at least half of the CUs idle: split just those
		// tiles so that they fill it with proportionally shorter workgroups
		*k_splits = rem <= 64 ? 4 : 2;
		*tail_tiles = rem;
		if (nk / *k_splits < 16) *k_splits = 1;
	}
}

int gemm_bf16(int a_t, int b_t, int M, int N, int K, const void* A, int64_t lda, const void* B, int64_t ldb,
              void* C, int64_t ldc, int epi, const void* R, int64_t ldr, int tile_cfg, int k_splits,
              hipStream_t stream) {
	ELF_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: empty problem M=%d N=%d K=%d", M, N, K);
	ELF_REQUIRE(K % BK == 0, "gemm: K must be a multiple of %d (K=%d)", BK, K);
	ELF_REQUIRE(A && B && C, "gemm: null operand");
	ELF_REQUIRE(lda % 8 == 0 && ldb % 8 == 0, "gemm: leading dimensions must be multiples of 8 elements");
	ELF_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)B % 16) == 0, "gemm: operands must be 16-byte aligned");
	ELF_REQUIRE(lda >= (a_t ? M : K) && ldb >= (b_t ? N : K) && ldc >= N, "gemm: leading dimension too small");
	// ldr == 0: R is one row of N values added to every row of C (the bias of a linear layer)
	ELF_REQUIRE(epi != EPI_BF16_RESID || (R != nullptr && (ldr >= N || ldr == 0)), "gemm: residual epilogue needs R");
	// the turn counters of split tiles hold the split index in 8 bits next to the launch tag
	ELF_REQUIRE(k_splits <= 255, "gemm: k_splits must be at most 255 (got %d)", k_splits);
	ProfScope prof(PROF_GEMM, 2.0 * M * N * K, stream);
	ELF_REQUIRE(M % 64 == 0 && N % 64 == 0, "gemm: M and N must be multiples of 64 (M=%d N=%d)", M, N);
	if (tile_cfg < 0) tile_cfg = 0;
	ELF_REQUIRE(tile_cfg <= 12 && tile_cfg != 4 && tile_cfg != 6, "gemm: unknown tile config %d", tile_cfg);
	int bm = 0, bn = 0, tail_tiles = -1;  // an explicit k_splits splits every tile
	switch (tile_cfg) {
		case 0: break;
		case 1: case 7: bm = 256, bn = 256; break;
		case 8: bm = 128, bn = 256; break;
		case 2: case 5: case 9: bm = 128, bn = 128; break;
		case 10: bm = 64, bn = 128; break;
		case 11: bm = 128, bn = 64; break;
		default: bm = bn = 64; break;
	}
	ELF_REQUIRE(M >= bm && N >= bn, "gemm: tile config %d needs M of at least %d and N of at least %d (M=%d N=%d)", tile_cfg, bm, bn, M, N);
	if (bm == 0) {
		Plan p;
		if (epi != EPI_F32_ACC) {
			const bool bf16_out = !a_t && (epi == EPI_BF16 || epi == EPI_BF16_RESID);
			p = plan_tiles(M, N, K, bf16_out, 0.f, 0.f, bf16_out);
		} else if (k_splits > 0) {
			p = plan_weight_gradient(M, N, K, 1);
		} else if (M >= 256 && N >= 256 && (int64_t)((M + 255) / 256) * ((N + 255) / 256) >= 192 && K >= 4096) {
			p = Plan{256, 256, 0};  // the split of the tail included, see below
		} else {
			p = plan_weight_gradient(M, N, K);
		}
		bm = p.bm, bn = p.bn;
		if (epi == EPI_F32_ACC && k_splits <= 0) k_splits = p.k_splits;
		// rows 16 MB apart and more (those that 64 rows of are out of reach are refused, a 32x32 tile or not)
		if (!gemm_reaches(a_t ? BK : std::max(bm, 64), lda) || !gemm_reaches(b_t ? BK : std::max(bn, 64), ldb)) bm = bn = 64;
	}
	if (epi != EPI_F32_ACC) k_splits = 1;
	if (bm == 256 && k_splits <= 0) dw_split_plan(M, N, K, &k_splits, &tail_tiles);
	if (bn >= 192) return gemm_bf16_dma(a_t, b_t, M, N, K, A, lda, B, ldb, C, ldc, epi, R, ldr, k_splits < 1 ? 1 : k_splits, tail_tiles, bm, stream, nullptr, 0, nullptr, 0, 0, 0, 1.f, bn);
	return gemm_bf16_ring(a_t, b_t, M, N, K, A, lda, B, ldb, C, ldc, epi, R, ldr, k_splits, bm, bn, stream);
}

// Whether the weight gradients of several layers are done sooner in one launch of gemm_dw_group, the way that takes them, than in a launch
// each on the best tile, and 2 us for that launch.  Constants in microseconds, fitted to 649 lists of 2 to 16 layers of at most a
// round of 256x256 tiles over 64 to 8192 tokens, operands past the caches; on 450 others no list that goes together takes 3 % longer than
// apart, and three that would be 4 to 6 % faster together stay apart.  us, apart and together: 2112 tokens, 4288 x 1600 and 832 x 4288 70 and 59; 1792,
// 1536 x 5184 and 3328 x 1536 75 and 60; 5312, 1216 x 896 and 1536 x 1216 88 and 57; 256, 2112 x 1024 and 384 x 2112 15.4 and 10.8.
// Staying apart: 8192, 1536 x 1536 and 1536 x 256 96 and 123; 3008, 1344 x 384 and 4544 x 1344 68 and 79; 2048, 4096 x 960 and 960 x 2560 56
// and 66; lists of more than a round, 4544 tokens, 5824 x 7232 and 1792 x 5824 465 and 480.
static bool group_pays(int n, const DwProblem* pr, int K) {
	const DwGroupWay way = gemm_dw_group_way(n, pr, K);
	if (way.tiles > 256) return false;
	float apart = 2.f * (n - 1);
	for (int i = 0; i < n; i++) apart += plan_weight_gradient(pr[i].M, pr[i].N, K).us;
	const int nk = K / BK;
	const float fill = way.tiles / 256.f;
	float group = nk * 0.45f + 9.9f;
	if (!way.small) {
		group = (nk + way.splits - 1) / way.splits * (0.8f + 0.8f * fill) + 18.f;
		if (way.splits > 1) group += 6.f * (way.splits - 1) + 30.f * way.splits * fill;  // the parts of a tile add one after the other
	}
	return group < 0.97f * apart;
}

int linear_w_way(int n, const LinearW* layers, int T) {
	ELF_REQUIRE(n > 0 && n <= DW_GROUP_MAX && layers && T > 0 && T % BK == 0, "linear_w_way: 1..%d layers over a multiple of %d tokens", DW_GROUP_MAX, BK);
	DwProblem pr[DW_GROUP_MAX];
	for (int i = 0; i < n; i++) {
		const LinearW& l = layers[i];
		if (!gemm_dw_groupable(l.M, l.N, T, l.dY, l.lddy, l.X, l.ldx, l.acc)) return 0;
		pr[i] = DwProblem{l.dY, l.lddy, l.X, l.ldx, l.acc, nullptr, l.M, l.N};
	}
	return n == 1 || !group_pays(n, pr, T) ? 0 : gemm_dw_group_way(n, pr, T).small ? 128 : 256;
}

int linear_w_pass(int n, const LinearW* layers, int T, float* workspace, hipStream_t stream) {
	ELF_REQUIRE(n > 0 && layers && T > 0, "linear_w_pass: no layers or no tokens");
	ELF_REQUIRE(T % BK == 0, "linear_w_pass: the tokens must be a multiple of %d (T=%d)", BK, T);
	bool biased = false;
	for (int i = 0; i < n; i++) {
		const LinearW& l = layers[i];
		ELF_REQUIRE(l.dY && l.X && l.acc && l.M > 0 && l.N > 0 && l.M % 64 == 0 && l.N % 64 == 0 && l.lddy % 8 == 0 && l.ldx % 8 == 0 && l.lddy >= l.M && l.ldx >= l.N &&
		                ((uintptr_t)l.dY % 16) == 0 && ((uintptr_t)l.X % 16) == 0,
		            "linear_w_pass: layer %d (M=%d N=%d) has a null operand, sizes that are no multiples of 64 or misaligned rows", i, l.M, l.N);
		biased = biased || l.bias;
	}
	ELF_REQUIRE(!biased || workspace, "linear_w_pass: bias sums need a workspace");
	DwProblem group[DW_GROUP_MAX];
	int ng = 0;
	auto alone = [&](const DwProblem& q) { return gemm_bf16(1, 1, q.M, q.N, T, q.dY, q.lddy, q.X, q.ldx, q.acc, q.N, EPI_F32_ACC, nullptr, 0, 0, 0, stream); };
	auto flush = [&]() -> int {
		const int m = ng;
		ng = 0;
		if (m > 1 && group_pays(m, group, T)) return gemm_dw_group(m, group, T, 0.f, stream);
		for (int i = 0; i < m; i++)
			if (int rc = alone(group[i])) return rc;
		return 0;
	};
	for (int i = 0; i < n; i++) {
		const LinearW& l = layers[i];
		const DwProblem q{l.dY, l.lddy, l.X, l.ldx, l.acc, nullptr, l.M, l.N};
		bool again = false;  // an accumulator that an earlier layer of the launch adds to as well: one after the other
		for (int j = 0; j < ng; j++) again = again || (q.acc < group[j].acc + (int64_t)group[j].M * group[j].N && group[j].acc < q.acc + (int64_t)q.M * q.N);
		if (again || ng == DW_GROUP_MAX) {
			if (int rc = flush()) return rc;
		}
		if (gemm_dw_groupable(l.M, l.N, T, l.dY, l.lddy, l.X, l.ldx, l.acc)) {
			group[ng++] = q;
		} else {
			// (behind what is waiting: it may add to the same accumulator)
			if (int rc = flush()) return rc;
			if (int rc = alone(q)) return rc;
		}
	}
	if (int rc = flush()) return rc;
	return biased ? colsum_group(n, layers, T, workspace, stream) : 0;
}

// The way of an up-projection with its activation: a 256-column tile (SwiGLU), a 64x64 ring tile, bm = 0: two passes.
static Plan act_plan(int act, int M, int F, int K, bool dense) {
	const int N = act == ACT_SWIGLU ? 2 * F : F;
	Plan best;
	best.us = plan_tiles(M, N, K).us + pass_us((act == ACT_SWIGLU ? 6.0 : 4.0) * M * F);
	if (act == ACT_SWIGLU) {
		const Plan p = plan_tiles(M, N, K, true, dense ? pass_us(6.0 * M * F) : NO_RING, SWIGLU_FWD_US);
		best.us = p.us;
		if (p.dma()) best = p;
	}
	const float small = dense ? small_us(M, N, K, act == ACT_SWIGLU ? SMALL_SWIGLU_US : SMALL_GELU_US) : 1e30f;
	return small < best.us ? Plan{64, 64, 1, small} : best;
}

int gemm_act_bf16(int act, int M, int F, int K, const void* A, int64_t lda, const void* W, int64_t ldw, void* pre,
                  int64_t ldpre, void* out, int64_t ldout, hipStream_t stream) {
	ELF_REQUIRE(act == ACT_GELU || act == ACT_SWIGLU, "gemm_act: unknown activation %d", act);
	ELF_REQUIRE(M > 0 && F > 0 && K > 0 && A && W && pre && out, "gemm_act: empty problem or null operand");
	const int N = act == ACT_SWIGLU ? 2 * F : F;
	// the SwiGLU epilogue pairs 64 gate with 64 up columns per wave, so a 256-column tile covers 128 outputs; it reaches the up rows
	// with 32-bit byte offsets from the gate rows
	Plan p;
	if (M % 64 == 0 && F % 64 == 0 && K % 64 == 0 && lda % 8 == 0 && ldw % 8 == 0 && ldpre >= N && ldout >= F && ldpre % 8 == 0 && ldout % 8 == 0 && ((uintptr_t)A % 16) == 0 &&
	    ((uintptr_t)W % 16) == 0 && ((uintptr_t)pre % 16) == 0 && ((uintptr_t)out % 16) == 0 && lda >= K && ldw >= K && gemm_reaches(256, lda) && (int64_t)(F + 256) * ldw * 2 < (int64_t(1) << 31))
		p = act_plan(act, M, F, K, ldpre == N && ldout == F);  // rows that lie further apart only the fused kernel of the large tiles writes
	if (p.bm == 64) {
		ProfScope prof(PROF_GEMM, 2.0 * M * N * K, stream);
		return gemm_ring_act(M, N, K, A, lda, W, ldw, pre, ldpre, act == ACT_SWIGLU ? EPI_BF16_SWIGLU : EPI_BF16_GELU, nullptr, 0, stream, out, ldout);
	}
	if (p.bm) {
		ProfScope prof(PROF_GEMM, 2.0 * M * N * K, stream);
		return gemm_bf16_dma(0, 0, M, N, K, A, lda, W, ldw, pre, ldpre, EPI_BF16_SWIGLU, nullptr, 0, 1, 0,
		                     p.bm, stream, out, ldout);
	}
	ELF_REQUIRE(ldpre == N && ldout == F, "gemm_act: the unfused path needs dense outputs");
	if (int rc = gemm_bf16(0, 0, M, N, K, A, lda, W, ldw, pre, ldpre, EPI_BF16, nullptr, 0, 0, 0, stream)) return rc;
	return act == ACT_SWIGLU ? swiglu_fwd(pre, out, M, F, stream) : gelu_fwd(pre, out, (int64_t)M * F, stream);
}

int gemm_dw_final(int M, int N, int K, const void* dY, int64_t lddy, const void* X, int64_t ldx, float* acc, void* grad_bf16, float scale,
                  hipStream_t stream) {
	ELF_REQUIRE(M > 0 && N > 0 && K > 0 && dY && X && acc && grad_bf16, "gemm_dw_final: bad argument");
	const bool fused = gemm_reaches(BK, lddy) && gemm_reaches(BK, ldx) && M % 64 == 0 && N % 64 == 0 && K % 64 == 0 && M >= 256 && N >= 256 && (int64_t)((M + 255) / 256) * ((N + 255) / 256) >= 192 && K >= 4096 && lddy % 8 == 0 && ldx % 8 == 0 && lddy >= M &&
	                   ldx >= N && ((uintptr_t)dY % 16) == 0 && ((uintptr_t)X % 16) == 0 && ((uintptr_t)acc % 16) == 0 && ((uintptr_t)grad_bf16 % 8) == 0;
	if (fused) {
		// the same K split as the plain weight gradient (same rounding); tiles shared by several workgroups along K have no
		// single epilogue that could scale them: a small kernel behind the GEMM does those
		int k_splits, tail_tiles;
		dw_split_plan(M, N, K, &k_splits, &tail_tiles);
		ProfScope prof(PROF_GEMM, 2.0 * M * N * K, stream);
		return gemm_bf16_dma(1, 1, M, N, K, dY, lddy, X, ldx, acc, N, EPI_F32_ACC_SCALE, nullptr, 0, k_splits, tail_tiles, 256, stream, grad_bf16, N, nullptr, 0, 0, 0, scale);
	}
	if (int rc = gemm_bf16(1, 1, M, N, K, dY, lddy, X, ldx, acc, N, EPI_F32_ACC, nullptr, 0, 0, 0, stream)) return rc;
	return scale_grads(acc, grad_bf16, (int64_t)M * N, scale, stream);
}

// The way of a projection with its rotary embedding: the rows of a 256-column tile, 64: a 64x64 ring tile, 0: two passes.
static int rope_tile_rows(int M, int N, int K, int D) {
	if (!(M >= 64 && N >= 64 && M % 64 == 0 && N % 64 == 0 && K % 64 == 0 && (D == 64 || D == 128) && N % D == 0)) return 0;
	const Plan p = plan_tiles(M, N, K, true, pass_us(4.0 * M * N), ROPE_US);
	if (small_us(M, N, K, SMALL_ROPE_US) < p.us) return 64;
	return p.dma() ? p.bm : 0;
}
bool gemm_rope_fused(int M, int N, int K, int D) {
	return rope_tile_rows(M, N, K, D) != 0;
}

int gemm_rope_bf16(int M, int N, int K, const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, const void* cs,
                   int S, int n_rot_heads, int D, hipStream_t stream) {
	ELF_REQUIRE(M > 0 && N > 0 && K > 0 && A && W && C && cs, "gemm_rope: empty problem or null operand");
	ELF_REQUIRE(S > 0 && M % S == 0 && n_rot_heads >= 0 && (int64_t)n_rot_heads * D <= N, "gemm_rope: bad head layout (S=%d, heads=%d, D=%d, N=%d)", S, n_rot_heads, D, N);
	if (gemm_rope_fused(M, N, K, D) && lda % 8 == 0 && ldw % 8 == 0 && ldc % 8 == 0 && lda >= K && ldw >= K && ldc >= N && ((uintptr_t)A % 16) == 0 &&
	    ((uintptr_t)W % 16) == 0 && ((uintptr_t)C % 16) == 0 && ((uintptr_t)cs % 16) == 0 && gemm_reaches(256, lda) && gemm_reaches(256, ldw)) {
		// the rotation's arithmetic is not counted: the figure stays the GEMM's
		ProfScope prof(PROF_GEMM, 2.0 * M * N * K, stream);
		const int bm = rope_tile_rows(M, N, K, D);
		if (bm == 64) return gemm_ring_act(M, N, K, A, lda, W, ldw, C, ldc, EPI_BF16_ROPE, nullptr, 0, stream, nullptr, 0, cs, S, n_rot_heads * D, D);
		return gemm_bf16_dma(0, 0, M, N, K, A, lda, W, ldw, C, ldc, EPI_BF16_ROPE, nullptr, 0, 1, 0, bm, stream, nullptr, 0, cs, S, n_rot_heads * D, D);
	}
	if (int rc = gemm_bf16(0, 0, M, N, K, A, lda, W, ldw, C, ldc, EPI_BF16, nullptr, 0, 0, 0, stream)) return rc;
	return n_rot_heads ? rope_apply(C, cs, M, S, (int)ldc, n_rot_heads, D, 0, stream) : 0;
}

// What the fused kernel can run at all (a caller without scratch or with strided buffers relies on it) ...
static bool swiglu_bwd_fits(int M, int F, int K) { return M >= 256 && F >= 256 && M % 64 == 0 && F % 64 == 0 && K % 64 == 0; }
// The tile it runs on.  The epilogue reads and writes four of d, g, u and their two gradients at 256 tiles a time: 20 us more per
// round of 256-row tiles than the plain one, and 4 us a launch (without these 3072 x 2304 x 768 took 33 us fused, 30.6 apart;
// with 12 us for the whole round 1024 x 3072 x 64 took 25 us fused, 13 apart, and 8448 x 512 x 512 32 and 20).
static Plan swiglu_bwd_tile(int M, int F, int K) {
	Plan best;
	auto weigh = [&](TileTime t) {
		if (M < t.bm) return;
		t.round += 20.f * t.bm / 256, t.launch += 4.f;
		const float us = tile_us(t, M, F, K / BK);
		if (us < best.us) best = Plan{t.bm, t.bn, 1, us};
	};
	weigh(TILES_BF16[0]);
	if (K > RING_SHORT_K)
		for (const TileTime& t : TILES_MID) weigh(t);
	return best;
}
// The faster way, dense buffers: the fused kernel on large tiles, on 64x64 ones, or the best tile of the plain product and the pass
// over d, g, u and their gradients.
enum { WAY_APART, WAY_LARGE, WAY_SMALL };
static int swiglu_bwd_way(int M, int F, int K) {
	const float apart = plan_tiles(M, F, K).us + pass_us(10.0 * M * F), large = swiglu_bwd_fits(M, F, K) ? swiglu_bwd_tile(M, F, K).us : 1e30f;
	// (of more than a round of 64x64 tiles the epilogue's five operands are not hidden: 896 x 1408 x 512 10.8 us apart, 11.1 fused)
	const bool one_round = (int64_t)(M / 64) * (F / 64) <= 256;
	if (one_round && small_us(M, F, K, SMALL_SWIGLU_BWD_US) < (large < apart ? large : apart)) return WAY_SMALL;
	return large < apart ? WAY_LARGE : WAY_APART;
}
bool gemm_swiglu_bwd_fused(int M, int F, int K) { return swiglu_bwd_way(M, F, K) != WAY_APART; }

int gemm_swiglu_bwd_bf16(int M, int F, int K, const void* dY, int64_t lddy, const void* W, int64_t ldw, const void* gu,
                         int64_t ldgu, void* dgu, int64_t lddgu, void* scratch, hipStream_t stream, void* act, int64_t ldact) {
	ELF_REQUIRE(M > 0 && F > 0 && K > 0 && dY && W && gu && dgu, "gemm_swiglu_bwd: empty problem or null operand");
	const bool dense = ldgu == 2 * F && lddgu == 2 * F && (!act || ldact == F);
	const bool fits = lddy >= K && ldw >= F && ldgu >= 2 * F && lddgu >= 2 * F && lddy % 8 == 0 && ldw % 8 == 0 && ldgu % 8 == 0 && lddgu % 8 == 0 && ((uintptr_t)dY % 16) == 0 &&
	                  ((uintptr_t)W % 16) == 0 && ((uintptr_t)gu % 16) == 0 && ((uintptr_t)dgu % 16) == 0 && gemm_reaches(256, lddy) && gemm_reaches(BK, ldw);
	int way = WAY_APART;
	if (fits) {
		way = dense ? swiglu_bwd_way(M, F, K) : WAY_APART;
		// what the separate passes cannot do goes to the large tiles wherever these fit
		if (way == WAY_APART && !(dense && scratch) && swiglu_bwd_fits(M, F, K)) way = WAY_LARGE;
	}
	if (way != WAY_APART) {
		// the activation backward's arithmetic is not counted: the figure stays the GEMM's
		ProfScope prof(PROF_GEMM, 2.0 * M * F * K, stream);
		ELF_REQUIRE(!act || (ldact >= F && ldact % 8 == 0 && ((uintptr_t)act % 16) == 0), "gemm_swiglu_bwd: bad activation output");
		if (way == WAY_SMALL) return gemm_ring_act(M, F, K, dY, lddy, W, ldw, dgu, lddgu, EPI_BF16_SWIGLU_BWD, gu, ldgu, stream, act, ldact);
		return gemm_bf16_dma(0, 1, M, F, K, dY, lddy, W, ldw, dgu, lddgu, EPI_BF16_SWIGLU_BWD, gu, ldgu, 1, 0, swiglu_bwd_tile(M, F, K).bm, stream, act, ldact);
	}
	ELF_REQUIRE(scratch, "gemm_swiglu_bwd: this shape needs a scratch buffer of M x F bf16");
	ELF_REQUIRE(ldgu == 2 * F && lddgu == 2 * F, "gemm_swiglu_bwd: the unfused path needs dense [M, 2F] buffers");
	if (int rc = gemm_bf16(0, 1, M, F, K, dY, lddy, W, ldw, scratch, F, EPI_BF16, nullptr, 0, 0, 0, stream)) return rc;
	ELF_REQUIRE(!act || ldact == F, "gemm_swiglu_bwd: the unfused path needs a dense activation output");
	return swiglu_bwd(scratch, gu, dgu, M, F, stream, act);
}

// GELU: fused on 64x64 tiles only (on larger ones the error function costs more than the pass it saves).
bool gemm_gelu_bwd_fused(int M, int F, int K) {
	return small_us(M, F, K, SMALL_GELU_BWD_US) < plan_tiles(M, F, K).us + pass_us(6.0 * M * F);
}

int gemm_gelu_bwd_bf16(int M, int F, int K, const void* dY, const void* W, const void* pre, void* dpre, void* scratch, hipStream_t stream) {
	ELF_REQUIRE(M > 0 && F > 0 && K > 0 && dY && W && pre && dpre, "gemm_gelu_bwd: empty problem or null operand");
	if (gemm_gelu_bwd_fused(M, F, K) && ((uintptr_t)dY % 16) == 0 && ((uintptr_t)W % 16) == 0 && ((uintptr_t)pre % 16) == 0 && ((uintptr_t)dpre % 16) == 0) {
		ProfScope prof(PROF_GEMM, 2.0 * M * F * K, stream);
		return gemm_ring_act(M, F, K, dY, K, W, F, dpre, F, EPI_BF16_GELU_BWD, pre, F, stream);
	}
	ELF_REQUIRE(scratch, "gemm_gelu_bwd: this shape needs a scratch buffer of M x F bf16");
	if (int rc = gemm_bf16(0, 1, M, F, K, dY, K, W, F, scratch, F, EPI_BF16, nullptr, 0, 0, 0, stream)) return rc;
	return gelu_bwd(scratch, pre, dpre, (int64_t)M * F, stream);
}

int gemm_way(int product, int M, int N, int K, int D) {
	Plan p;
	if (M < 64 || N < 64 || K < 64 || M % 64 || N % 64 || K % 64) return 0;
	switch (product) {
		case GEMM_WAY_FORWARD: case GEMM_WAY_INPUT_GRADIENT: p = plan_tiles(M, N, K, true, 0.f, 0.f, true); break;
		case GEMM_WAY_GELU: p = act_plan(ACT_GELU, M, N, K, true); break;
		case GEMM_WAY_SWIGLU: p = act_plan(ACT_SWIGLU, M, N, K, true); break;
		case GEMM_WAY_GELU_BWD: if (gemm_gelu_bwd_fused(M, N, K)) p = Plan{64, 64}; break;
		case GEMM_WAY_SWIGLU_BWD: {
			const int way = swiglu_bwd_way(M, N, K);
			if (way != WAY_APART) p = way == WAY_SMALL ? Plan{64, 64} : swiglu_bwd_tile(M, N, K);
			break;
		}
		case GEMM_WAY_ROPE:
			if (const int rows = rope_tile_rows(M, N, K, D)) p = Plan{rows, rows == 64 ? 64 : 256};
			break;
	}
	return p.bm << 16 | p.bn;
}

}  // namespace elf
