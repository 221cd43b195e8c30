// bf16 MFMA GEMM tile kernel (128 to 256 rows by 256 columns) with direct global->LDS loads, for gfx950.
//
// The contraction of gemm_bf16.hip (C (+)= sum_k A(m,k) B(n,k); "R" operands are
// k-contiguous, "T" operands reduction-major), different data movement:
//   * global_load_lds_dwordx4 moves 16 B per lane straight into LDS (no VGPR staging, no
//     ds_write); a ring of two or three 64-wide K slices of each operand (see Shape), fetched ahead
//     of their use.  64 bf16 = one full 128-byte cache line per operand row;
//   * a wave instruction fills 1 KiB of LDS contiguously, so tiles cannot be padded; bank
//     conflicts are avoided by an XOR swizzle of the 16-byte chunk index, applied on the global
//     side when choosing which chunk a lane fetches and undone when fragments are read;
//   * the contraction runs on v_mfma_f32_16x16x32_bf16; the 256x256 tile is worked by four waves with
//     128x128 sub-tiles (one per SIMD; k-contiguous A) or by eight with 64x128 sub-tiles (two per SIMD;
//     both operands reduction-major), the 128x256 tile by four with 64x128 sub-tiles.
// The DMA loads are issued through inline assembly: the compiler cannot see that they write
// LDS, which is what allows partial vmcnt waits (its own tracking would force vmcnt(0) before
// every LDS read).  Ordering is explicit: s_waitcnt vmcnt(n) for this wave's slice, then a
// workgroup barrier for the other waves' slices and for the reuse of the oldest stage.
#pragma once
#include "common.h"
#include "kernels.h"
#include "gemm_tile.h"

namespace elf {

namespace dma {

constexpr int BN = 256;  // columns of a tile (192 where a kernel says so)
constexpr int PERS_WORKGROUPS = 256;  // one per compute unit: the persistent kernel's grid

// Shape of one workgroup: NW waves arranged (NW / 2) x 2, each owning RF x 8 accumulator tiles of
// 16 x 16 (6 of them across in a tile of 192 columns), so the workgroup tile is BM x TN with BM = (NW / 2) * RF * 16.
template <int NW, int RF, int TN = BN>
struct Shape {
	static constexpr int B_BYTES = TN * BKS * 2;
	static constexpr int CH = TN / 64;  // 16-column slabs of a wave in either column half
	static constexpr int BM = (NW / 2) * RF * 16;
	static constexpr int STRIPS = (RF + 1) / 2;  // 32-row strips of a wave in the epilogue (the last of an odd RF has 16 rows)
	static constexpr int A_BYTES = BM * BKS * 2;
	// K slices in LDS: three of B and two or three of A, as far as the 160 KiB go (256 rows: all of them).  What bounds a
	// round of tiles on cold operands is how long before its use a slice is asked for.  With two slices of both, the last
	// loads of a slice went out half a slice before they had to have landed, and a slice took 1.2 to 1.3 us whatever its
	// rows (1.0 with the chip to itself); with a third slice of B, whose loads go out a slice earlier, only those of A are
	// late, by three quarters of a slice.  Cold operands, before -> after (us): input gradients 8192 x 4096 x 28672 1282 -> 1217,
	// 2688 x 4096 x 28672 595 -> 504, SwiGLU backward 8192 x 14336 x 4096 883 -> 810; W pass of a Llama-3-8B block over 8192
	// tokens 2667 -> 2523, over 2688 1082 -> 1002, of three GPT-2-small blocks over 8192 324 -> 294.
	static constexpr int NSA = BM <= 160 ? 3 : 2, NSB = 3, RING_BYTES = NSA * A_BYTES + NSB * B_BYTES;
	static constexpr int PERIOD = NSA == NSB ? NSB : NSA * NSB;  // slices after which the ring is back where it was
	// 1 KiB pieces (one wave instruction each) per wave, slice and operand
	static constexpr int LOADS_A = A_BYTES / 1024 / NW, LOADS_B = B_BYTES / 1024 / NW;
	static_assert(LOADS_B % 2 == 0 && RING_BYTES <= 160 * 1024, "the loads of a slice of B are issued in two halves");
};

struct Args {
	const bf16_t* A;
	const bf16_t* B;
	void* C;
	const bf16_t* R;
	bf16_t* C2;  // SwiGLU epilogue: the activated output
	int64_t lda, ldb, ldc, ldr, ldc2;
	int M, N, K;
	int tiles_m, tiles_n;
	int k_splits;    // K is split this many ways (fp32 atomics epilogue) for the last tail_tiles tiles
	int tail_tiles;  // tiles_m * tiles_n for a uniform split, 0 when nothing is split
	int walk;        // 1: all XCDs share one band of 16 tile rows at a time (see the tile assignment)
	// EPI_BF16_ROPE: (cos, sin) table [rope_S, rope_D / 2], columns below rope_cols are rotated, heads are rope_D wide
	const float2* rope_cs;
	int rope_S, rope_cols, rope_D;
	// split tiles: this launch's tag in the turn counters (see turn[] below); 0 = the splits add in any order
	uint32_t turn_tag;
	float scale;  // EPI_F32_ACC_SCALE
	uint32_t turn_base;  // split tiles: the first of this problem's turn counters
};

// Turn counters of split tiles.  The workgroups that share a tile along K add their parts with fp32 atomics; to make
// the sum independent of the order in which they finish, split s only starts adding when turn[slot] holds this
// launch's tag with count s, and publishes count s + 1 when its adds have been performed.  The tag changes with every
// launch, so a value left by an earlier launch never matches and nothing has to be cleared.  Workgroups are
// dispatched in index order and the splits of a tile have consecutive indices, so the one a workgroup waits for is
// always running or done; the wait is bounded all the same, and a workgroup that gives up (counters shared with a
// concurrent launch on another stream) adds out of turn: still the right sum, only its rounding may differ.
// A counter covers one 32-row strip of one wave (up to 16 per tile), so a split starts on a strip as soon as its
// predecessor is through with that strip and the splits of a tile overlap except for about one strip.
constexpr int TURN_TILES = 4096, TURN_PER_TILE = 16;
static __device__ uint32_t turn[TURN_TILES * TURN_PER_TILE];
// polls of ~1 us each: about a millisecond in all, several times what a predecessor's epilogue takes (the splits of a
// tile start together and run equal K ranges).  One budget per wave for the whole epilogue; a wave that uses it up is
// counted in turn_giveups (gemm_turn_giveups() reads it) and adds out of turn from then on.
constexpr int TURN_SPIN_LIMIT = 1 << 10;
static __device__ unsigned int turn_giveups;
__device__ __forceinline__ void note_turn_giveup() { atomicAdd(&turn_giveups, 1u); }
// Adds this translation unit's count (the counters, like the kernels that use them, are one set per layout of the operands).
static int add_turn_giveups(uint64_t* sum) {
	unsigned int n = 0;
	ELF_CHECK_HIP(hipMemcpyFromSymbol(&n, HIP_SYMBOL(turn_giveups), sizeof(n)));
	*sum += n;
	return 0;
}

// NW = 4, RF = 8: 256x256 workgroup tile, one wave per SIMD with a 128x128 wave tile: 16 fragment reads per
// k32 for 64 MFMAs, a third less LDS traffic per FLOP than the eight-wave shape, which on this power-limited
// part is worth 2-4 % (forward and dX GEMMs).  It needs two things a lone wave does not forgive: all 256
// accumulator registers are live, so the MFMAs are tied in place by hand (mfma_acc), and nothing else
// fills issue gaps, so the next half-step's fragment reads and the slice's loads are dealt between the
// MFMAs one at a time (half_step).  Left to the builtin and to bursts of reads it ran 12 % slower than
// the eight-wave shape.
// NW = 8, RF = 4: 256x256 workgroup tile, two waves per SIMD with 64x128 wave tiles (12 fragment reads per
// k32 and 32 MFMAs); the two waves fill each other's issue gaps and barrier waits.  Used when both
// operands are reduction-major (dW): each of their fragments costs two transpose reads and an address.
// NW = 4, RF = 4: 128x256 workgroup tile for outputs with too few 256x256 tiles to fill the chip.  One wave per SIMD
// as well, so it runs the same interleaved loop (+35-40 % on the GPT-2-small shapes over read bursts).
// Which of the `half` load pieces dealt over a half-step of `nm` MFMAs goes out after MFMA n (-1: none): piece k after
// MFMA 2 * floor(k * (nm / 2) / half) - always an even one, because the fragment reads go out after the odd ones and a
// read and a load behind the same MFMA do not fit under it.
constexpr int piece_in_slot(int n, int nm, int half) {
	for (int k = 0; k < half; k++)
		if (2 * ((k * (nm / 2)) / half) == n) return k;
	return -1;
}

// every piece has a slot of its own within the half-step
constexpr bool pieces_have_slots(int nm, int half) {
	for (int k = 0; k < half; k++) {
		int hits = 0;
		for (int n = 0; n < nm; n++) hits += piece_in_slot(n, nm, half) == k;
		if (hits != 1) return false;
	}
	return true;
}

// acc += a b as one in-place instruction on accumulator registers — the builtin leaves source and
// destination accumulators untied, and when all 256 accumulator registers are live (128x128 wave tiles) the
// allocator then copies accumulator tiles around inside the loop (192 copies per K slice).  Every
// accumulator tile is touched once per half-step, so consecutive MFMAs never depend on each other, and the
// epilogue reads the accumulators only after a wait and a workgroup barrier.
__device__ __forceinline__ void mfma_acc(f32x4& acc, const bf16x8& a, const bf16x8& b) {
	asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}


// Origin (m0, n0) of tile `pid` of the launch: see "Tile assignment" in gemm_dma_kernel for the two walks.
template <int BM, int TN = BN>
__device__ __forceinline__ void tile_origin(const Args& g, int pid, int& m0, int& n0) {
	if (g.walk == 2) {  // tiles in plain order, down the rows first (the launch places them on the XCDs itself)
		m0 = (pid % g.tiles_m) * BM;
		n0 = (pid / g.tiles_m) * TN;
		return;
	}
	const int ntiles = g.tiles_m * g.tiles_n;
	const int nsb = ntiles >> 5, nrem = nsb & 7;
	if (g.walk == 1 && (g.tiles_m & 7) == 0 && (g.tiles_n & 3) == 0 && (nrem == 0 || nrem == 1 || nrem == 2 || nrem == 4)) {
		const int x = pid & 7, i = pid >> 3, nfull = nsb >> 3;
		int sb, jj;
		if (i < nfull * 32) {
			sb = (i >> 5) * 8 + x;
			jj = i & 31;
		} else {
			const int k = 8 / nrem;
			sb = nfull * 8 + x / k;
			jj = (x % k) * (32 / k) + (i - nfull * 32);
		}
		const int nsb_n = g.tiles_n >> 2, nsb_m = g.tiles_m >> 3;
		const int band = sb / (2 * nsb_n), within = sb - band * 2 * nsb_n;
		const bool pair = 2 * band + 1 < nsb_m;
		const int sbm = 2 * band + (pair ? within & 1 : 0), sbn = pair ? within >> 1 : within;
		m0 = (sbm * 8 + (jj & 7)) * BM;
		n0 = (sbn * 4 + (jj >> 3)) * TN;
	} else {
		// (192 columns: also where 8 does not divide the tiles, the first XCDs then have one more.  These tiles take the place of ones of 256 columns, of
		// which a product may have a multiple of 8, and with the neighbours of a slab on all XCDs each of them fetches all of B.  us on operands in
		// the memory-side cache, 256 columns, 192 in plain order, 192 so: 768 x 8000 x 12544, B reduction-major 133, 174 and 122; 320 x 16320 x
		// 2752 31.8, 51.2 and 35.0; 448 x 9728 x 1984, B reduction-major 24.5, 27.3 and 21.9)
		if ((ntiles & 7) == 0 || TN != BN) pid = (pid & 7) * (ntiles >> 3) + min(pid & 7, ntiles & 7) + (pid >> 3);
		constexpr int GROUP_M = 8;
		const int per_group = GROUP_M * g.tiles_n;
		const int first_m = (pid / per_group) * GROUP_M;
		const int gsz = min(g.tiles_m - first_m, GROUP_M);
		m0 = (first_m + (pid % per_group) % gsz) * BM;
		n0 = ((pid % per_group) / gsz) * TN;
	}
}

// Ragged sizes: the last tile of a row or column of tiles moves back so that it ends with the matrix, and stores only what
// its neighbour does not (it needs M >= BM, N >= 256).  Every operand load stays inside the matrix without a bounds check
// in the K loop, and the partly empty tile multiplies rows its neighbour multiplies as well instead of padding.  (M, N
// multiples of 64: what is skipped are whole 32-row strips and whole 64-column halves.)
template <int BM, int TN = BN>
__device__ __forceinline__ void clip_tile(const Args& g, int& m0, int& n0) {
	m0 = min(m0, g.M - BM);
	n0 = min(n0, g.N - TN);
}

// Tile, K range and turn counter of workgroup `bid` of the problem `g` (the block index of a launch with one problem).
// The first ntiles - tail_tiles tiles are computed whole, one workgroup each; each of the last tail_tiles is shared by
// k_splits workgroups that take a K range each and add their part with atomics.  Splitting only the tail turns the
// last, partly filled round of workgroups of a launch into a full round of shorter ones.
__device__ __forceinline__ void locate_tile(const Args& g, const int bid, int& pid, int& ksplit, int& splits, int& turn_slot) {
	const int ntiles = g.tiles_m * g.tiles_n;
	const int full = ntiles - g.tail_tiles;
	pid = bid, ksplit = 0, splits = 1;
	if (pid >= full) {
		const int q = pid - full;
		splits = g.k_splits;
		if (((ntiles | full) & 7) == 0) {  // keep workgroup index = tile index (mod 8): same XCD as its neighbours
			const int rest = q >> 3;
			ksplit = rest % splits;
			pid = full + (rest / splits) * 8 + (q & 7);
		} else {
			ksplit = q % splits;
			pid = full + q / splits;
		}
	}
	// split tiles: the turn counter of this tile (tiles of one launch get distinct counters, consecutive launches different ones)
	turn_slot = (int)(((uint32_t)(pid - full) + g.turn_base) % (uint32_t)TURN_TILES);
}

// One workgroup: tile `pid` of the problem `g`, K range `ksplit` of `splits`; a split tile's turn counters are those of
// `turn_slot`.
// EDGE: M or N is no multiple of the tile (see clip_tile).
template <int NW, int RF, bool AT, bool BT, int EPI, bool EDGE, int TN = BN>
__device__ __forceinline__ void gemm_dma_tile(const Args& g, const int pid, const int ksplit, const int splits, const int turn_slot) {
	using Sh = Shape<NW, RF, TN>;
	constexpr int BM = Sh::BM, A_BYTES = Sh::A_BYTES, B_BYTES = Sh::B_BYTES, STRIPS = Sh::STRIPS;
	constexpr int CH = Sh::CH, WCOLS = TN / 2;  // columns of a wave
	static_assert(TN == BN || EPI == EPI_BF16 || EPI == EPI_BF16_RESID, "the other epilogues are written for 256 columns");
	constexpr int LOADS_A = Sh::LOADS_A, LOADS_B = Sh::LOADS_B, NSA = Sh::NSA, NSB = Sh::NSB;
	constexpr bool PAIRED = EPI == EPI_BF16_SWIGLU;
	static_assert(!PAIRED || !BT, "the paired row order is defined for a k-contiguous B");
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int wr = wave >> 1, wc = wave & 1;

	// Tile assignment (tile_origin).  Workgroup w runs on XCD w % 8, whose 32 CUs hold 32 tiles at a time (a round);
	// both walks give an XCD 8 tile rows x 4 tile columns per round (12 operand slabs through its L2 for
	// 32 tiles) and differ in where the 8 XCDs are relative to each other:
	//  * default: each XCD owns a contiguous run of tiles (8 tile rows at a time, along the columns).  The
	//    XCDs work on different row groups; a row slab of A is needed in as many rounds as the row has
	//    column groups, so A has to stay in the memory-side cache between them;
	//  * walk = 1: the 8 XCDs share a 16 x 16 block of tiles per round, bands of 16 tile rows walked along the
	//    columns; a row slab of A is live for one band only, B is fetched once per band (weight gradient of
	//    the gate/up projection, 28672 x 4096 at K = 8192, A = 470 MB: 5-7 % faster).  A last, partly filled
	//    round shares each 8 x 4 block between several XCDs.
	int m0, n0;
	tile_origin<BM, TN>(g, pid, m0, n0);
	m0 = __builtin_amdgcn_readfirstlane(m0);
	n0 = __builtin_amdgcn_readfirstlane(n0);
	const int m_lo = m0, n_lo = n0;  // first row and column this tile stores
	if constexpr (EDGE) clip_tile<BM, TN>(g, m0, n0);

	const int nk_total = g.K / BKS;
	const int nk_per = (nk_total + splits - 1) / splits;
	const int kt0 = ksplit * nk_per;
	const int nk = min(nk_total, kt0 + nk_per) - kt0;
	constexpr bool CAN_SPLIT = EPI == EPI_F32_ACC || EPI == EPI_F32_ACC_SCALE;
	if (nk <= 0) {  // (left out where it cannot happen, the main loop's first trip is conditional and its accumulators spill)
		// a split without a K range of its own still takes and passes its turn on every strip
		if (CAN_SPLIT && splits > 1 && g.turn_tag && lane == 0) {
			const uint32_t want = (g.turn_tag << 8) | (uint32_t)ksplit;
			int patience = TURN_SPIN_LIMIT;
			for (int i = 0; i < STRIPS; i++) {
				if (EDGE && m0 + wr * (RF * 16) + i * 32 < m_lo) continue;
				uint32_t* t = turn + turn_slot * TURN_PER_TILE + wave * STRIPS + i;
				int spin = 0;
				for (; ksplit > 0 && spin < patience && __hip_atomic_load(t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != want; spin++)
					__builtin_amdgcn_s_sleep(8);
				if (ksplit > 0 && spin >= patience) {
					if (patience > 0) note_turn_giveup();
					patience = 0;
				} else {
					patience -= spin;
				}
				__hip_atomic_store(t, want + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			}
		}
		return;
	}

	const bf16_t* Ap = AT ? g.A + (int64_t)kt0 * BKS * g.lda + m0 : g.A + (int64_t)m0 * g.lda + (int64_t)kt0 * BKS;
	// paired rows: tile column n0 of the (gate | up interleaved) product starts at operand row n0 / 2
	const bf16_t* Bp = BT ? g.B + (int64_t)kt0 * BKS * g.ldb + n0 : g.B + (int64_t)(PAIRED ? n0 / 2 : n0) * g.ldb + (int64_t)kt0 * BKS;
	const int64_t a_step = AT ? (int64_t)BKS * g.lda : BKS;
	const int64_t b_step = BT ? (int64_t)BKS * g.ldb : BKS;
	uint32_t aoff[LOADS_A], boff[LOADS_B];
	lane_offsets<AT, LOADS_A, false, BM>(wave, lane, g.lda, aoff);
	lane_offsets<BT, LOADS_B, PAIRED, TN>(wave, lane, g.ldb, boff, g.N / 2);

	// this wave's first 1 KiB piece of each operand in stage 0
	const uint32_t lds_a = lds_addr(smem) + wave * (LOADS_A * 1024);
	const uint32_t lds_b = lds_addr(smem) + NSA * A_BYTES + wave * (LOADS_B * 1024);

	// Loads of one operand's K slice `step`: its pointer and the LDS address of this wave's first piece in ring stage `stage`.
	// Piece P (compile-time) is one wave instruction filling 1 KiB.  A slice past the end of K is fetched from the last one,
	// into the stage that would be its own (nobody reads it any more), so that the main loop needs no branches around its
	// loads and the accumulators stay put in registers.
	struct Loads {
		const bf16_t* p;
		uint32_t lds;
	};
	auto loads_a = [&](int step, int stage) { return Loads{Ap + (int64_t)min(step, nk - 1) * a_step, lds_a + (uint32_t)stage * A_BYTES}; };
	auto loads_b = [&](int step, int stage) { return Loads{Bp + (int64_t)min(step, nk - 1) * b_step, lds_b + (uint32_t)stage * B_BYTES}; };
	auto piece_a = [&](const Loads& l, auto pc) { dma16_at<decltype(pc)::value * 1024>(l.p, aoff[decltype(pc)::value], l.lds); };
	auto piece_b = [&](const Loads& l, auto pc) { dma16_at<decltype(pc)::value * 1024>(l.p, boff[decltype(pc)::value], l.lds); };

	// 16x16 accumulator tiles: RF down, 8 across (the 16x16x32 MFMA moves half as many accumulator
	// registers per FLOP as the 32x32x16 one, and sustains a higher clock under the power limit)
	f32x4 acc[RF][2 * CH];
#pragma unroll
	for (int i = 0; i < RF; i++)
#pragma unroll
		for (int j = 0; j < 2 * CH; j++)
#pragma unroll
			for (int r = 0; r < 4; r++) acc[i][j][r] = 0.f;

	// Software pipeline.  A slice is four half-steps (k32 half kq = 0, 1 x column half h = 0, 1) of RF * 4
	// MFMAs; the fragments of a half-step are read during the one before it (B: four 16-column slabs
	// per half-step, ping-pong; A: RF slabs per k32 half, ping-pong).  The barrier that publishes slice
	// kt+1 sits before the LAST half-step of slice kt: by then every wave has read all of slice kt (its
	// last fragments are in registers), so the same barrier frees its stages: the fetch of A's next slice for that
	// stage goes out in the last half-step, that of B's in the first two of slice kt+1.
	static_assert(pieces_have_slots(RF * CH, LOADS_A) && pieces_have_slots(RF * CH, LOADS_B / 2), "a half-step has too few even MFMA slots for its loads");
	// slices 0 .. NSB-2 of B and 0 .. NSA-1 of A; slice 0 has to have landed
	static_for<NSB>([&](auto sc) {
		constexpr int S = decltype(sc)::value;
		if constexpr (S < NSA) static_for<LOADS_A>([&](auto pc) { piece_a(loads_a(S, S), pc); });
		if constexpr (S < NSB - 1) static_for<LOADS_B>([&](auto pc) { piece_b(loads_b(S, S), pc); });
	});
	wait_vmcnt<(NSA - 1) * LOADS_A + (NSB - 2) * LOADS_B>();
	__syncthreads();

	bf16x8 fa[2][RF], fb[2][CH];
	auto load_a = [&](int buf, int step, int kq) {
		const unsigned char* sa = smem + (step % NSA) * A_BYTES;
#pragma unroll
		for (int i = 0; i < RF; i++) fa[buf][i] = frag<AT, BM>(sa, wr * (RF * 16) + i * 16, kq, lane);
	};
	auto load_b = [&](int buf, int step, int kq, int h) {
		const unsigned char* sb = smem + NSA * A_BYTES + (step % NSB) * B_BYTES;
#pragma unroll
		for (int j = 0; j < CH; j++) fb[buf][j] = frag<BT, TN>(sb, wc * WCOLS + (h * CH + j) * 16, kq, lane);
	};
	// One half-step: RF * CH MFMAs with the fragment reads of the next half-step (one read per two MFMAs, or as many as it takes, B
	// slabs first: they are needed first) and, in two of the four half-steps, half of this wave's loads of a
	// slice dealt between them one at a time.  A lone wave per SIMD has nothing else to fill its issue
	// gaps, and a wave that issues its loads in one burst (64 KiB per slice through a 64 B/clk path) sits in
	// the queue for ~1000 cycles with its MFMAs behind it.  With two waves per SIMD the wave also raises
	// its issue priority for the length of the half-step: the one feeding the matrix pipe goes first.
	// Reduction-major operands in this loop: the two transpose-read addresses of every fragment are computed
	// once (k32 half 0 of stage 0); the k32 half and the stage are compile-time here (the loop is unrolled by
	// PERIOD slices, three or six) and go into the instructions' offset fields.  Those hold 16 bits: stage 2 of B lies 64 and
	// 80 KiB up and costs an add per read, a third of B's reads.
	uint32_t ta[AT ? RF : 1][2], tb[BT ? 2 * CH : 1][2];
	{
		if constexpr (AT)
#pragma unroll
			for (int i = 0; i < RF; i++) {
				frag_t_offsets<BM>(wr * (RF * 16) + i * 16, lane, ta[i]);
				ta[i][0] += lds_addr(smem), ta[i][1] += lds_addr(smem);
				// opaque from here on: folded into these, the tile's base would push the loop's offsets past 16 bits
				asm volatile("" : "+v"(ta[i][0]), "+v"(ta[i][1]));
			}
		if constexpr (BT)
#pragma unroll
			for (int i = 0; i < 2 * CH; i++) {
				frag_t_offsets<TN>(wc * WCOLS + i * 16, lane, tb[i]);
				tb[i][0] += lds_addr(smem) + NSA * A_BYTES, tb[i][1] += lds_addr(smem) + NSA * A_BYTES;
				asm volatile("" : "+v"(tb[i][0]), "+v"(tb[i][1]));
			}
	}
	auto half_step = [&](int abuf, int bbuf, auto hc, int pb_buf, auto pb_stage, int pb_kq, int pb_h, bool pa, int pa_buf, auto pa_stage, int pa_kq,
	                     const Loads& ld, auto dealt) {
		// dealt: which loads go out in this half-step (0: none, 1: a slice of A, 2 and 3: the halves of a slice of B)
		constexpr int DEALT = decltype(dealt)::value, NP = DEALT == 0 ? 0 : DEALT == 1 ? LOADS_A : LOADS_B / 2, H = decltype(hc)::value, NM = RF * CH;
		constexpr int SA = decltype(pa_stage)::value, SB = decltype(pb_stage)::value;
		const unsigned char* sa = smem + SA * A_BYTES;
		const unsigned char* sb = smem + NSA * A_BYTES + SB * B_BYTES;
		if constexpr (NW == 8) __builtin_amdgcn_s_setprio(1);
		static_for<NM>([&](auto nc) {
			constexpr int n = decltype(nc)::value, i = n / CH, j = n % CH;
			mfma_acc(acc[i][H * CH + j], fa[abuf][i], fb[bbuf][j]);
			// reads [r0, r1) ride behind this MFMA: one behind every odd one, or, where those are too few (64 x 96 wave tiles), evenly dealt
			constexpr bool ODD = NM / 2 >= CH + RF;
			constexpr int r0 = ODD ? n / 2 : n * (CH + RF) / NM, r1 = ODD ? (n % 2 == 1 ? n / 2 + 1 : n / 2) : (n + 1) * (CH + RF) / NM;
			static_for<r1 - r0>([&](auto rc) {
				constexpr int r = r0 + decltype(rc)::value;
				if constexpr (r < CH) {
					if constexpr (BT) fb[pb_buf][r] = frag_t_at(tb[pb_h * CH + r], (uint32_t)(SB * B_BYTES + pb_kq * (32 * TN * 2)));
					else fb[pb_buf][r] = frag<BT, TN>(sb, wc * WCOLS + (pb_h * CH + r) * 16, pb_kq, lane);
				} else if constexpr (r - CH < RF) {
					if (pa) {
						if constexpr (AT) fa[pa_buf][r - CH] = frag_t_at(ta[r - CH], (uint32_t)(SA * A_BYTES + pa_kq * (32 * BM * 2)));
						else fa[pa_buf][r - CH] = frag<AT, BM>(sa, wr * (RF * 16) + (r - CH) * 16, pa_kq, lane);
					}
				}
			});
			constexpr int piece = NP == 0 ? -1 : piece_in_slot(n, NM, NP);
			if constexpr (piece >= 0) {
				if constexpr (DEALT == 1) piece_a(ld, std::integral_constant<int, piece>{});
				else piece_b(ld, std::integral_constant<int, (DEALT - 2) * (LOADS_B / 2) + piece>{});
			}
			__builtin_amdgcn_sched_barrier(0);
		});
		if constexpr (NW == 8) __builtin_amdgcn_s_setprio(0);
	};
	// K slice kt, kt mod PERIOD = S
	auto slice = [&](auto sc, int kt) {
		constexpr int S = decltype(sc)::value;
		constexpr std::integral_constant<int, S % NSA> A_CUR{};
		constexpr std::integral_constant<int, S % NSB> B_CUR{};
		constexpr std::integral_constant<int, (S + 1) % NSA> A_NXT{};
		constexpr std::integral_constant<int, (S + 1) % NSB> B_NXT{};
		constexpr std::integral_constant<int, 0> H0{}, NONE{};
		constexpr std::integral_constant<int, 1> H1{}, SLICE_A{};
		constexpr std::integral_constant<int, 2> FIRST_B{};
		constexpr std::integral_constant<int, 3> SECOND_B{};
		// where the loads go: scalar work.  B: the stage that slice kt - 1 left free; A: the one this slice leaves free
		const Loads lb = loads_b(kt + NSB - 1, (S + NSB - 1) % NSB), la = loads_a(kt + NSA, S % NSA);
		half_step(0, 0, H0, 1, B_CUR, 0, 1, false, 0, A_CUR, 0, lb, FIRST_B);
		half_step(0, 1, H1, 0, B_CUR, 1, 0, true, 1, A_CUR, 1, lb, SECOND_B);
		half_step(1, 0, H0, 1, B_CUR, 1, 1, false, 0, A_CUR, 0, la, NONE);
		// vmcnt: slice kt+1 landed (what was issued after it may still be in flight); lgkmcnt(0): slice kt fully read
		wait_counters<(NSA - 2) * LOADS_A + (NSB - 2) * LOADS_B, 0>();
		__syncthreads();
		// with the loads of A into the stage the barrier just freed; past the end the fragment reads hit a stale stage and
		// their values are unused
		half_step(1, 1, H1, 0, B_NXT, 0, 0, true, 0, A_NXT, 0, la, SLICE_A);
	};

	load_a(0, 0, 0);
	load_b(0, 0, 0, 0);
	for (int kt = 0; kt < nk; kt += Sh::PERIOD) {
		slice(std::integral_constant<int, 0>{}, kt);
		if (kt + 1 < nk) slice(std::integral_constant<int, 1>{}, kt + 1);
		if (kt + 2 < nk) slice(std::integral_constant<int, 2>{}, kt + 2);
		if constexpr (Sh::PERIOD == 6) {
			if (kt + 3 < nk) slice(std::integral_constant<int, 3>{}, kt + 3);
			if (kt + 4 < nk) slice(std::integral_constant<int, 4>{}, kt + 4);
			if (kt + 5 < nk) slice(std::integral_constant<int, 5>{}, kt + 5);
		}
	}

	// Epilogue through LDS (free once every wave has left the main loop).  Register r of a 16x16
	// accumulator tile holds row (lane/16)*4 + r, column lane%16; each wave parks one 32 x 128 fp32 strip
	// (two rows of accumulator tiles) at a time in its own LDS region (row pitch 136 floats) and reads it
	// back row-wise, so that global accesses are 16 bytes per lane over 256..512 contiguous bytes per row
	// and accumulators leave the AGPRs only via ds_write.
	wait_vmcnt<0>();  // the loads past the end of K issued by the last iterations land in LDS too
	__syncthreads();
	constexpr int PITCH = 136;
	float* ws = reinterpret_cast<float*>(smem) + wave * (32 * PITCH);
	[[maybe_unused]] int turn_patience = TURN_SPIN_LIMIT;
	const int col_l = lane & 15;
	const int row_l = (lane >> 4) * 4;
	// ROW_CLIP: an odd number of 16-row slabs per wave; where the tile is moved back, the neighbour's rows may end inside a strip
	constexpr bool ROW_CLIP = EDGE && RF % 2 == 1;
#pragma unroll
	for (int i = 0; i < STRIPS; i++) {
		const int rows = RF - 2 * i < 2 ? 16 : 32;  // (a constant once unrolled)
#pragma unroll
		for (int ii = 0; ii < 2; ii++)
#pragma unroll
			for (int j = 0; j < 2 * CH; j++)
#pragma unroll
				for (int r = 0; r < 4; r++)
					if (ii * 16 < rows) ws[(ii * 16 + row_l + r) * PITCH + j * 16 + col_l] = acc[i * 2 + ii < RF ? i * 2 + ii : 0][j][r];
		const int grow0 = m0 + wr * (RF * 16) + i * 32;
		const int gcol0 = n0 + wc * WCOLS;
		if (EDGE && grow0 + (ROW_CLIP ? rows - 16 : 0) < m_lo) continue;  // the neighbouring tile's rows (the same strips for every K split of a tile)
		const int c_lo = EDGE ? n_lo - gcol0 : 0;  // columns of the wave's 128 below c_lo are the neighbouring tile's
		if constexpr (EPI == EPI_BF16_SWIGLU) {
			// the strip's columns are 64 gate columns then the 64 up columns of the same outputs: both go to
			// their places in C = [gate | up] (kept for the backward) and silu(gate) * up, computed from the
			// rounded values exactly as a separate pass over C would, to C2
			const int F = g.N / 2, cg0 = n0 / 2 + wc * 64;
			if (EDGE && cg0 < n_lo / 2) continue;
#pragma unroll
			for (int it = 0; it < rows / 8; it++) {
				const int row = it * 8 + (lane >> 3), c8 = (lane & 7) * 8;
				if (ROW_CLIP && grow0 + row < m_lo) continue;
				const float* w = ws + row * PITCH + c8;
				const f32x4 g0 = *reinterpret_cast<const f32x4*>(w), g1 = *reinterpret_cast<const f32x4*>(w + 4);
				const f32x4 u0 = *reinterpret_cast<const f32x4*>(w + 64), u1 = *reinterpret_cast<const f32x4*>(w + 68);
				bf16x8 og, ou, oa;
#pragma unroll
				for (int t = 0; t < 8; t++) {
					og[t] = (bf16_t)(t < 4 ? g0[t] : g1[t - 4]);
					ou[t] = (bf16_t)(t < 4 ? u0[t] : u1[t - 4]);
					oa[t] = (bf16_t)swiglu_f((float)og[t], (float)ou[t]);
				}
				bf16_t* c = reinterpret_cast<bf16_t*>(g.C) + (int64_t)(grow0 + row) * g.ldc + cg0 + c8;
				*reinterpret_cast<bf16x8*>(c) = og;
				*reinterpret_cast<bf16x8*>(c + F) = ou;
				*reinterpret_cast<bf16x8*>(g.C2 + (int64_t)(grow0 + row) * g.ldc2 + cg0 + c8) = oa;
			}
		} else if constexpr (EPI == EPI_BF16_SWIGLU_BWD) {
			// the tile is d = dY W over F columns; g and u of the same rows and columns lie F columns apart in R,
			// their gradients likewise in C.  All loads of the strip first (see the residual epilogue below); d is
			// rounded to bf16 before it is used, as a separate pass over a stored d would read it
			const int F = g.N;
			if (EDGE && (lane & 15) * 8 < c_lo) continue;
			bf16x8 gs[8], us[8];
#pragma unroll
			for (int it = 0; it < rows / 4; it++) {
				const bf16_t* r = g.R + (int64_t)(grow0 + it * 4 + (lane >> 4)) * g.ldr + gcol0 + (lane & 15) * 8;
				gs[it] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(r));  // the pre-activation is read this once in B
				us[it] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(r + F));
			}
#pragma unroll
			for (int it = 0; it < rows / 4; it++) {
				const int row = it * 4 + (lane >> 4), c8 = (lane & 15) * 8;
				if (ROW_CLIP && grow0 + row < m_lo) continue;
				const f32x4 lo = *reinterpret_cast<const f32x4*>(ws + row * PITCH + c8);
				const f32x4 hi = *reinterpret_cast<const f32x4*>(ws + row * PITCH + c8 + 4);
				bf16x8 og, ou;
#pragma unroll
				for (int t = 0; t < 8; t++) {
					const float d = (float)(bf16_t)(t < 4 ? lo[t] : hi[t - 4]);
					float dg, du;
					swiglu_bwd_f(d, (float)gs[it][t], (float)us[it][t], dg, du);
					og[t] = (bf16_t)dg;
					ou[t] = (bf16_t)du;
				}
				bf16_t* c = reinterpret_cast<bf16_t*>(g.C) + (int64_t)(grow0 + row) * g.ldc + gcol0 + c8;
				*reinterpret_cast<bf16x8*>(c) = og;
				*reinterpret_cast<bf16x8*>(c + F) = ou;
				if (g.C2) {
					// a stash that dropped the activation gets it back here, from the g and u this epilogue holds anyway (the
					// forward's own arithmetic: the bits of swiglu_fwd)
					bf16x8 oa;
#pragma unroll
					for (int t = 0; t < 8; t++) oa[t] = (bf16_t)swiglu_f((float)gs[it][t], (float)us[it][t]);
					*reinterpret_cast<bf16x8*>(g.C2 + (int64_t)(grow0 + row) * g.ldc2 + gcol0 + c8) = oa;
				}
			}
		} else if constexpr (EPI == EPI_BF16_ROPE) {
			// A 128-column strip holds whole heads (rope_D = 64 or 128).  A lane takes, for one row, 8 columns of a
			// head's first half and the 8 columns half a head further on: the (x_i, x_{i + D/2}) pairs of the rotation.
			// The accumulator is rounded to bf16 first, as the RoPE kernel would read it from memory.  The table
			// entries of the whole strip are fetched before the first store (see the residual epilogue below).
			const int half = g.rope_D >> 1, cph = half >> 3;  // chunks of 8 columns per half head
			const int j = lane & 7;
			const int h_lo = (j / cph) * g.rope_D + (j % cph) * 8, h_hi = h_lo + half;
			if (EDGE && h_lo < c_lo) continue;  // (a launch's tiles only overlap by whole heads: see gemm_bf16_dma)
			const bool rot = gcol0 + h_lo < g.rope_cols;
			f32x4 tab[4][4];
			if (rot) {
#pragma unroll
				for (int it = 0; it < rows / 8; it++) {
					const int pos = (grow0 + it * 8 + (lane >> 3)) % g.rope_S;
					const f32x4* tp = reinterpret_cast<const f32x4*>(g.rope_cs + (int64_t)pos * half + (j % cph) * 8);
#pragma unroll
					for (int q = 0; q < 4; q++) tab[it][q] = tp[q];
				}
			}
#pragma unroll
			for (int it = 0; it < rows / 8; it++) {
				const int row = it * 8 + (lane >> 3);
				if (ROW_CLIP && grow0 + row < m_lo) continue;
				const float* w = ws + row * PITCH;
				const f32x4 a0 = *reinterpret_cast<const f32x4*>(w + h_lo), a1 = *reinterpret_cast<const f32x4*>(w + h_lo + 4);
				const f32x4 b0 = *reinterpret_cast<const f32x4*>(w + h_hi), b1 = *reinterpret_cast<const f32x4*>(w + h_hi + 4);
				bf16x8 olo, ohi;
#pragma unroll
				for (int t = 0; t < 8; t++) {
					const float a = (float)(bf16_t)(t < 4 ? a0[t] : a1[t - 4]), b = (float)(bf16_t)(t < 4 ? b0[t] : b1[t - 4]);
					float ra = a, rb = b;
					if (rot) rope_rot(a, b, tab[it][t >> 1][(t & 1) * 2], tab[it][t >> 1][(t & 1) * 2 + 1], ra, rb);
					olo[t] = (bf16_t)ra;
					ohi[t] = (bf16_t)rb;
				}
				bf16_t* c = reinterpret_cast<bf16_t*>(g.C) + (int64_t)(grow0 + row) * g.ldc + gcol0;
				*reinterpret_cast<bf16x8*>(c + h_lo) = olo;
				*reinterpret_cast<bf16x8*>(c + h_hi) = ohi;
			}
		} else if constexpr (EPI == EPI_BF16 || EPI == EPI_BF16_RESID) {
			// the strip's residual values first, all loads in flight together: read inside the loop below each
			// one would be awaited (a full trip to HBM) before the store that follows it in program order
			if ((EDGE && (lane & 15) * 8 < c_lo) || (WCOLS < 128 && (lane & 15) * 8 >= WCOLS)) continue;
			bf16x8 rs[EPI == EPI_BF16_RESID ? 8 : 1];
			if constexpr (EPI == EPI_BF16_RESID) {
#pragma unroll
				for (int it = 0; it < rows / 4; it++)
					rs[it] = *reinterpret_cast<const bf16x8*>(g.R + (int64_t)(grow0 + it * 4 + (lane >> 4)) * g.ldr + gcol0 + (lane & 15) * 8);
			}
#pragma unroll
			for (int it = 0; it < rows / 4; it++) {
				const int row = it * 4 + (lane >> 4), c8 = (lane & 15) * 8;
				if (ROW_CLIP && grow0 + row < m_lo) continue;
				const f32x4 lo = *reinterpret_cast<const f32x4*>(ws + row * PITCH + c8);
				const f32x4 hi = *reinterpret_cast<const f32x4*>(ws + row * PITCH + c8 + 4);
				float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
				if constexpr (EPI == EPI_BF16_RESID) {
#pragma unroll
					for (int t = 0; t < 8; t++) v[t] += (float)rs[it][t];
				}
				bf16x8 o;
#pragma unroll
				for (int t = 0; t < 8; t++) o[t] = (bf16_t)v[t];
				*reinterpret_cast<bf16x8*>(reinterpret_cast<bf16_t*>(g.C) + (int64_t)(grow0 + row) * g.ldc + gcol0 + c8) = o;
			}
		} else {
			if (CAN_SPLIT && splits > 1) {  // (split tiles of a scaling launch are scaled by scale_tail_kernel)
				uint32_t* const my_turn = turn + turn_slot * TURN_PER_TILE + wave * STRIPS + i;
				if (g.turn_tag && ksplit > 0) {
					// wait for this split's turn on this strip (see turn[]); every lane polls the same word.  Plain
					// (cache-bypassing) loads: nothing is read after the wait, the adds are performed at the memory side
					const uint32_t want = (g.turn_tag << 8) | (uint32_t)ksplit;
					int spin = 0;
					for (; spin < turn_patience && __hip_atomic_load(my_turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != want; spin++)
						__builtin_amdgcn_s_sleep(8);
					// a wave that gave up once (its counters are shared with a concurrent launch) does not wait again
					if (spin >= turn_patience) {
						if (turn_patience > 0 && lane == 0) note_turn_giveup();
						turn_patience = 0;
					} else {
						turn_patience -= spin;
					}
				}
				// several workgroups add into this tile: fp32 atomics, one scalar per lane so that a wave
				// instruction covers two whole 128-byte rows of 32 columns (16 bytes per lane would touch a
				// quarter of eight lines per instruction and run at half the speed)
#pragma unroll
				for (int it = 0; it < rows / 2; it++) {
					const int row = it * 2 + (lane >> 5);
					float* c = reinterpret_cast<float*>(g.C) + (int64_t)(grow0 + row) * g.ldc + gcol0 + (lane & 31);
#pragma unroll
					for (int cg = 0; cg < 4; cg++)
						if (!EDGE || cg * 32 >= c_lo) unsafeAtomicAdd(c + cg * 32, ws[row * PITCH + cg * 32 + (lane & 31)]);
				}
				if (g.turn_tag) {
					// wait until this wave's adds have been performed (they complete in vmcnt; no cache write-back is
					// needed for atomics), then the next split may add to this strip
					wait_vmcnt<0>();
					if (lane == 0) __hip_atomic_store(my_turn, (g.turn_tag << 8) | (uint32_t)(ksplit + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				}
				continue;
			}
			// fp32 accumulate: the strip's 16 loads of C all in flight before the first store (left inside the
			// loop each load is awaited on its own, 16 trips to HBM in a row per strip: 43 k cycles of a
			// 360 k-cycle dW tile)
			constexpr bool ACCUM = CAN_SPLIT;
			static_assert(!ROW_CLIP, "an fp32 output is clipped by whole strips");
			if (EDGE && (lane & 31) * 4 < c_lo) continue;
			f32x4 cv[ACCUM ? 16 : 1];
			if constexpr (ACCUM) {
#pragma unroll
				for (int it = 0; it < rows / 2; it++)
					cv[it] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(g.C) + (int64_t)(grow0 + it * 2 + (lane >> 5)) * g.ldc + gcol0 + (lane & 31) * 4));
			}
#pragma unroll
			for (int it = 0; it < rows / 2; it++) {
				const int row = it * 2 + (lane >> 5), c4 = (lane & 31) * 4;
				f32x4 v = *reinterpret_cast<const f32x4*>(ws + row * PITCH + c4);
				float* c = reinterpret_cast<float*>(g.C) + (int64_t)(grow0 + row) * g.ldc + gcol0 + c4;
				if constexpr (ACCUM) v += cv[it];
				if constexpr (EPI == EPI_F32_ACC_SCALE) {
					// the step's last weight-gradient pass: the gradient scale and the bf16 copy that scale_grads would make
					// in a pass of its own over the accumulator (same operations on the same values: same bits)
					v *= g.scale;
					bf16x4 o;
#pragma unroll
					for (int t = 0; t < 4; t++) o[t] = (bf16_t)v[t];
					*reinterpret_cast<bf16x4*>(g.C2 + (int64_t)(grow0 + row) * g.ldc2 + gcol0 + c4) = o;
				}
				if constexpr (ACCUM) __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(c));  // next touched by the next W pass
				else *reinterpret_cast<f32x4*>(c) = v;
			}
		}
	}
}

template <int NW, int RF, bool AT, bool BT, int EPI, bool EDGE, int TN = BN>
__global__ __launch_bounds__(NW * 64) void gemm_dma_kernel(Args g) {
	int pid, ksplit, splits, turn_slot;
	locate_tile(g, (int)blockIdx.x, pid, ksplit, splits, turn_slot);
	gemm_dma_tile<NW, RF, AT, BT, EPI, EDGE, TN>(g, pid, ksplit, splits, turn_slot);
}

template <int NW, int RF, bool AT, bool BT, int EPI, bool EDGE, int TN = BN>
static int launch_sized(const Args& a, hipStream_t stream) {
	// the ring (the loads past the end of K go into its stages too) or, where that is more, the epilogue's 32 x 136 fp32 strip per wave
	using Sh = Shape<NW, RF, TN>;
	constexpr int ring = Sh::RING_BYTES, epi = NW * 32 * 136 * 4;
	constexpr int smem = ring > epi ? ring : epi;
	auto kern = gemm_dma_kernel<NW, RF, AT, BT, EPI, EDGE, TN>;
	static bool attr_set = false;
	if (!attr_set) {
		ELF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
		attr_set = true;
	}
	ELF_LAUNCH(kern, dim3(a.tiles_m * a.tiles_n + a.tail_tiles * (a.k_splits - 1)), dim3(NW * 64), smem, stream, a);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

template <int NW, int RF, bool AT, bool BT, int EPI>
static int launch(const Args& a, hipStream_t stream) {
	return a.M % Shape<NW, RF>::BM || a.N % BN ? launch_sized<NW, RF, AT, BT, EPI, true>(a, stream) : launch_sized<NW, RF, AT, BT, EPI, false>(a, stream);
}

// Tiles of bm rows with a k-contiguous A, by the layout of B (gemm_dma_rr.hip, gemm_dma_rt.hip), and the persistent kernel for
// EPI_BF16, EPI_BF16_RESID and EPI_BF16_SWIGLU (gemm_dma_pers.hip).
// (tn: 256 columns, or 192 with 128 rows, EPI_BF16 and EPI_BF16_RESID)
int launch_rr(int bm, int tn, const Args& a, int epi, hipStream_t stream);
int launch_rt(int bm, int tn, const Args& a, int epi, hipStream_t stream);
int launch_pers(const Args& a, int epi, hipStream_t stream);
int rr_turn_giveups(uint64_t* sum);
int rt_turn_giveups(uint64_t* sum);

}  // namespace dma

// the tiles between 128 and 256 rows
inline bool gemm_mid_rows(int bm) { return bm == 160 || bm == 192 || bm == 224; }

}  // namespace elf
