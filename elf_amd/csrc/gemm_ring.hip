// bf16 MFMA GEMM on small tiles (128x128, 64x128, 128x64, 64x64, 32x32) with a deep ring of K slices in LDS, for gfx950.
//
// Same contraction, layouts and order of products along K as gemm_dma_tile.h (v_mfma_f32_16x16x32_bf16, 64 wide K slices in
// ascending order), so a tile's bits do not depend on which of the kernels computed it.  These are the tiles of products
// too small to fill the chip with the 256-column tiles of gemm_dma_tile.h: a workgroup then has few K slices and every trip to
// memory shows.  The ring holds as many slices as LDS takes (eight of the 64x64 tile, four of the 128x128 one), all fetched
// before the first product; from then on a slice is fetched as soon as its predecessor in the same stage has been read.
//
// Bound: the 64 B/clk path into LDS (a slice of the 128x128 tile is 512 cycles of it and 512 of MFMA, of the 64x64 tile 256
// against 128) and LDS reads; results leave from registers, two neighbouring column slabs exchanged between lane groups so
// that a lane stores 16 bytes.  The activations and the rotary embedding of the smallest products ride in the epilogue of the
// 64x64 tile (gemm_ring_act: what bounds these is the number of launches).
// Against the register-staged tiles (global -> VGPR -> LDS, two stages) that these replace, cold operands: 1920 x 1600 x 1600 23.1 -> 19.9 us, 2112 x 832 x 4288 50 -> 31, 512 x 512 x 1536 14.2 -> 7.9; weight
// gradients: 1600 x 1600 x 1920 36.7 -> 25.6, 832 x 4288 x 2112 50 -> 29, 768 x 768 x 4096 31 -> 22.
#include "common.h"
#include "gemm_tile.h"
#include "kernels.h"

namespace elf {

namespace ring {

using dma::BKS;

struct Args {
	const bf16_t* A;
	const bf16_t* B;
	void* C;
	const bf16_t* R;
	int64_t lda, ldb, ldc, ldr;
	int M, N, K;
	int tiles_m, tiles_n;
	int k_splits;       // K is split this many ways (fp32 atomics, EPI_F32_ACC only)
	uint32_t turn_tag;  // this launch's tag in the turn counters, 0 = the splits add in any order
	// epilogues of gemm_ring_act
	bf16_t* C2;
	int64_t ldc2;
	const float2* rope_cs;
	int rope_S, rope_cols, rope_D;
	float scale;  // EPI_F32_ACC_SCALE
};

// Turn counters of split tiles, one per tile and wave (the scheme of gemm_dma.hip: split s adds when the counter holds this
// launch's tag with count s and publishes s + 1; splits of lower index are dispatched first; the wait is bounded).
constexpr int TURN_TILES = 4096;
static __device__ uint32_t turn[TURN_TILES * 4];
constexpr int TURN_SPIN_LIMIT = 1 << 10;
static __device__ unsigned int turn_giveups;

// SHORT: two slices, for a K of at most RING_SHORT_K and bf16 outputs.  A deep ring fetches all of its slices up front whether K
// has them or not, and holds the compute unit's LDS alone; of these, two to four workgroups share one, and the epilogue of one
// hides behind the loads of the next.  11392 x 640 x 64 10.0 -> 8.1 us, 7232 x 576 x 128 7.6 -> 6.3, 9344 x 896 x 256 13.0 -> 10.2;
// with five to eight slices of K the deep ring is 5 % ahead, with sixteen 30 %.
template <int BM, int BN, bool SHORT>
struct Shape {
	static constexpr int A_BYTES = BM * BKS * 2, B_BYTES = BN * BKS * 2, STAGE_BYTES = A_BYTES + B_BYTES;
	// 128 .. 144 KiB of slices (of the 32x32 tile 64, as many of them as of the 64x64 one; 32 KiB of it if SHORT)
	static constexpr int NST = SHORT ? BM == 32 ? 4 : 2 : BM <= 64 && BN <= 64 ? 8 : BM == 128 && BN == 128 ? 4 : 6;
	static constexpr int LOADS_A = A_BYTES / 4096, LOADS_B = B_BYTES / 4096, LOADS = LOADS_A + LOADS_B;  // 1 KiB pieces per wave and slice
	static constexpr int SMEM = NST * STAGE_BYTES + (LOADS_A > LOADS_B ? LOADS_A : LOADS_B) * 1024;
};

// acc = four consecutive columns (n) of one output row (m) per lane: the weight side feeds the MFMA's row operand.
__device__ __forceinline__ void mfma(f32x4& acc, const bf16x8& b, const bf16x8& a) { acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, acc, 0, 0, 0); }

// Two neighbouring 16-column slabs of a row hold columns 4 g .. 4 g + 3 in lane group g = lane / 16.  Afterwards lo, hi are
// the eight consecutive columns 16 (g % 2) + 8 (g / 2) .. + 7 of the 32: one 16-byte store per lane.
__device__ __forceinline__ void pair_slabs(f32x4& lo, f32x4& hi) {
#pragma unroll
	for (int r = 0; r < 4; r++) {
		const float l = lo[r], h = hi[r];  // (copies: a bit cast of a vector element would read element 0)
		const auto p = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, l), __builtin_bit_cast(uint32_t, h), false, false);
		const uint32_t pl = p[0], ph = p[1];
		lo[r] = __builtin_bit_cast(float, pl);
		hi[r] = __builtin_bit_cast(float, ph);
	}
}

// One workgroup: tile `pid`, K range `ksplit` of g.k_splits.
template <int BM, int BN, bool AT, bool BT, int EPI, bool SHORT>
__device__ __forceinline__ void gemm_ring_tile(const Args& g, const int pid, const int ksplit) {
	using Sh = Shape<BM, BN, SHORT>;
	constexpr int NST = Sh::NST, A_BYTES = Sh::A_BYTES, B_BYTES = Sh::B_BYTES, LOADS_A = Sh::LOADS_A, LOADS_B = Sh::LOADS_B, P = Sh::LOADS;
	constexpr int WM = BM / 2, WN = BN / 2, RF = WM / 16, CF = WN / 16, NM = RF * CF, NR = RF + CF;
	// A wave's columns are 16 columns (gate, or a head's first half) and the 16 that belong to them `pair` rows of B further on (up,
	// or its second half): both halves of a pair are in one lane's accumulators
	constexpr bool PAIRED = EPI == EPI_BF16_SWIGLU || EPI == EPI_BF16_ROPE;
	static_assert(!PAIRED || (BM == 64 && BN == 64 && !AT && !BT), "the paired row order is defined for 64x64 tiles of k-contiguous operands");
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int wr = wave >> 1, wc = wave & 1;

	int m0, n0;
	{
		constexpr int GROUP_M = 8;
		const int per_group = GROUP_M * g.tiles_n;
		const int first_m = (pid / per_group) * GROUP_M;
		const int gsz = min(g.tiles_m - first_m, GROUP_M);
		m0 = __builtin_amdgcn_readfirstlane((first_m + (pid % per_group) % gsz) * BM);
		n0 = __builtin_amdgcn_readfirstlane(((pid % per_group) / gsz) * BN);
	}
	// ragged sizes: the last tile moves back to end with the matrix and skips what its neighbour stores (64-row and
	// 64-column steps: whole waves for a 128-wide tile)
	const int m_lo = m0, n_lo = n0;
	m0 = min(m0, g.M - BM);
	n0 = min(n0, g.N - BN);

	const int nk_total = g.K / BKS;
	const int nk_per = (nk_total + g.k_splits - 1) / g.k_splits;
	const int kt0 = ksplit * nk_per;
	const int nk = min(nk_total, kt0 + nk_per) - kt0;
	uint32_t* const my_turn = turn + (((uint32_t)pid + g.turn_tag * 977u) % (uint32_t)TURN_TILES) * 4 + wave;
	const uint32_t turn_want = (g.turn_tag << 8) | (uint32_t)ksplit;
	auto take_turn = [&]() {
		if (g.turn_tag && ksplit > 0) {
			int spin = 0;
			for (; spin < TURN_SPIN_LIMIT && __hip_atomic_load(my_turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != turn_want; spin++)
				__builtin_amdgcn_s_sleep(8);
			if (spin >= TURN_SPIN_LIMIT && lane == 0) atomicAdd(&turn_giveups, 1u);
		}
	};
	auto pass_turn = [&]() {
		if (g.turn_tag) {
			wait_vmcnt<0>();  // the adds have been performed at the memory side
			if (lane == 0) __hip_atomic_store(my_turn, turn_want + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
		}
	};
	if (nk <= 0) {  // a split without a K range of its own takes and passes its turn
		take_turn();
		pass_turn();
		return;
	}

	const bf16_t* const Ap = AT ? g.A + (int64_t)kt0 * BKS * g.lda + m0 : g.A + (int64_t)m0 * g.lda + (int64_t)kt0 * BKS;
	// the tile's first column in C: a paired tile covers half as many gate columns, or two runs of 32 columns of one head
	const int c_lo = EPI == EPI_BF16_SWIGLU ? n0 / 2 : EPI == EPI_BF16_ROPE ? n0 / g.rope_D * g.rope_D + n0 % g.rope_D / 2 : n0;
	const int pair = EPI == EPI_BF16_SWIGLU ? g.N / 2 : EPI == EPI_BF16_ROPE ? g.rope_D / 2 : 0;
	const bf16_t* const Bp = BT ? g.B + (int64_t)kt0 * BKS * g.ldb + n0 : g.B + (int64_t)c_lo * g.ldb + (int64_t)kt0 * BKS;
	const int64_t a_step = AT ? (int64_t)BKS * g.lda : BKS;
	const int64_t b_step = BT ? (int64_t)BKS * g.ldb : BKS;
	uint32_t aoff[LOADS_A], boff[LOADS_B];
	dma::lane_offsets<AT, LOADS_A, false, BM>(wave, lane, g.lda, aoff);
	if constexpr (PAIRED) {
#pragma unroll
		for (int i = 0; i < LOADS_B; i++) {
			const int row = (wave * LOADS_B + i) * 8 + (lane >> 3), slot = lane & 7;
			const int64_t grow = (row >> 5) * 16 + (row & 15) + ((row >> 4) & 1) * (int64_t)pair;
			boff[i] = (uint32_t)((grow * g.ldb + ((slot ^ ((row >> 1) & 7)) << 3)) * 2);
		}
	} else {
		dma::lane_offsets<BT, LOADS_B, false, BN>(wave, lane, g.ldb, boff);
	}
	const uint32_t lds_a = lds_addr(smem) + wave * (LOADS_A * 1024);
	const uint32_t lds_b = lds_addr(smem) + NST * A_BYTES + wave * (LOADS_B * 1024);
	const uint32_t lds_dummy = lds_addr(smem) + NST * Sh::STAGE_BYTES;

	// loads of one slice; a slice past the end of K is fetched from the last one into a scratch area that nobody reads, so
	// that the number of loads in flight (and with it every partial wait) is the same in every trip
	struct SliceLoads {
		const bf16_t* pa;
		const bf16_t* pb;
		uint32_t la, lb;
	};
	auto slice_loads = [&](int step, int stage) {
		const bool ok = step < nk;
		const int sc = ok ? step : nk - 1;
		return SliceLoads{Ap + (int64_t)sc * a_step, Bp + (int64_t)sc * b_step, ok ? lds_a + stage * A_BYTES : lds_dummy, ok ? lds_b + stage * B_BYTES : lds_dummy};
	};
	auto issue_piece = [&](const SliceLoads& sl, auto pc) {
		constexpr int Q = decltype(pc)::value;
		if constexpr (Q < LOADS_A) dma16_at<Q * 1024>(sl.pa, aoff[Q], sl.la);
		else dma16_at<(Q - LOADS_A) * 1024>(sl.pb, boff[Q - LOADS_A], sl.lb);
	};
	dma::static_for<NST>([&](auto sc) {
		const SliceLoads sl = slice_loads(decltype(sc)::value, decltype(sc)::value);
		dma::static_for<P>([&](auto pc) { issue_piece(sl, pc); });
	});

	f32x4 acc[RF][CF];
#pragma unroll
	for (int i = 0; i < RF; i++)
#pragma unroll
		for (int j = 0; j < CF; j++)
#pragma unroll
			for (int r = 0; r < 4; r++) acc[i][j][r] = 0.f;

	// LDS addresses of the fragment reads in stage 0; stage and k32 half are compile-time offsets on top
	uint32_t a_lane[AT ? RF : 2][AT ? 2 : 1], b_lane[BT ? CF : 2][BT ? 2 : 1];
	{
		const int l15 = lane & 15, q4 = lane >> 4;
		if constexpr (AT) {
#pragma unroll
			for (int i = 0; i < RF; i++) {
				dma::frag_t_offsets<BM>(wr * WM + i * 16, lane, a_lane[i]);
				a_lane[i][0] += lds_addr(smem), a_lane[i][1] += lds_addr(smem);
				asm volatile("" : "+v"(a_lane[i][0]), "+v"(a_lane[i][1]));
			}
		} else {
#pragma unroll
			for (int kq = 0; kq < 2; kq++) {
				a_lane[kq][0] = lds_addr(smem) + (uint32_t)((wr * WM + l15) * 128 + (((4 * kq + q4) ^ ((l15 >> 1) & 7)) << 4));
				asm volatile("" : "+v"(a_lane[kq][0]));
			}
		}
		if constexpr (BT) {
#pragma unroll
			for (int j = 0; j < CF; j++) {
				dma::frag_t_offsets<BN>(wc * WN + j * 16, lane, b_lane[j]);
				b_lane[j][0] += lds_addr(smem) + NST * A_BYTES, b_lane[j][1] += lds_addr(smem) + NST * A_BYTES;
				asm volatile("" : "+v"(b_lane[j][0]), "+v"(b_lane[j][1]));
			}
		} else {
#pragma unroll
			for (int kq = 0; kq < 2; kq++) {
				b_lane[kq][0] = lds_addr(smem) + NST * A_BYTES + (uint32_t)((wc * WN + l15) * 128 + (((4 * kq + q4) ^ ((l15 >> 1) & 7)) << 4));
				asm volatile("" : "+v"(b_lane[kq][0]));
			}
		}
	}
	auto read_a = [&](auto stage, auto kq, auto ic) -> bf16x8 {
		constexpr int S = decltype(stage)::value, KQ = decltype(kq)::value, I = decltype(ic)::value;
		if constexpr (AT) return dma::frag_t_at(a_lane[I], S * A_BYTES + KQ * (32 * BM * 2));
		else return *reinterpret_cast<const bf16x8 ELF_LDS*>((uintptr_t)(a_lane[KQ][0] + (uint32_t)(S * A_BYTES + I * (16 * 128))));
	};
	auto read_b = [&](auto stage, auto kq, auto jc) -> bf16x8 {
		constexpr int S = decltype(stage)::value, KQ = decltype(kq)::value, J = decltype(jc)::value;
		if constexpr (BT) return dma::frag_t_at(b_lane[J], S * B_BYTES + KQ * (32 * BN * 2));
		else return *reinterpret_cast<const bf16x8 ELF_LDS*>((uintptr_t)(b_lane[KQ][0] + (uint32_t)(S * B_BYTES + J * (16 * 128))));
	};

	bf16x8 fa[2][RF], fb[2][CF];
	// One k32 half: RF x CF MFMAs, with the next half's fragment reads behind the first NR of them (B first: all of it is
	// needed by the first row of products) and, in the second half of a slice, the loads of slice kt + NST dealt over the rest.
	auto step = [&](auto cur_c, auto rd_stage, auto rd_kq, auto load_c, const SliceLoads& sl) {
		constexpr int CUR = decltype(cur_c)::value, NXT = 1 - CUR;
		constexpr bool LOAD = decltype(load_c)::value;
		dma::static_for<NM>([&](auto nc) {
			constexpr int n = decltype(nc)::value, i = n / CF, j = n % CF;
			mfma(acc[i][j], fb[CUR][j], fa[CUR][i]);
			constexpr int r0 = NR <= NM ? n : n * NR / NM, r1 = NR <= NM ? (n < NR ? n + 1 : n) : (n + 1) * NR / NM;
			dma::static_for<r1 - r0>([&](auto rc) {
				constexpr int r = r0 + decltype(rc)::value;
				if constexpr (r < CF) fb[NXT][r] = read_b(rd_stage, rd_kq, std::integral_constant<int, r>{});
				else fa[NXT][r - CF] = read_a(rd_stage, rd_kq, std::integral_constant<int, r - CF>{});
			});
			if constexpr (LOAD) {
				constexpr int p0 = n * P / NM, p1 = (n + 1) * P / NM;
				dma::static_for<p1 - p0>([&](auto pc) { issue_piece(sl, std::integral_constant<int, p0 + decltype(pc)::value>{}); });
			}
			__builtin_amdgcn_sched_barrier(0);
		});
	};
	constexpr std::integral_constant<int, 0> C0{};
	constexpr std::integral_constant<int, 1> C1{};
	auto slice = [&](auto sc, int kt) {
		constexpr int S = decltype(sc)::value;
		constexpr std::integral_constant<int, S> CUR{};
		constexpr std::integral_constant<int, (S + 1) % NST> NXT{};
		const SliceLoads sl = slice_loads(kt + NST, S);
		step(C0, CUR, C1, std::false_type{}, sl);
		wait_counters<(NST - 2) * P, 0>();  // slice kt + 1 landed; this wave has read all of slice kt
		__syncthreads();                    // ... and so have the others: the stage of slice kt is free
		// (past the end of K the fragments come from a stale stage and are not used)
		step(C1, NXT, C0, std::true_type{}, sl);
	};
	wait_vmcnt<(NST - 1) * P>();
	__syncthreads();
	dma::static_for<CF>([&](auto jc) { fb[0][decltype(jc)::value] = read_b(C0, C0, jc); });
	dma::static_for<RF>([&](auto ic) { fa[0][decltype(ic)::value] = read_a(C0, C0, ic); });
	for (int kt = 0; kt < nk; kt += NST)
		dma::static_for<NST>([&](auto sc) {
			if (kt + decltype(sc)::value < nk) slice(sc, kt + decltype(sc)::value);
		});

	// Epilogue from registers: row m of slab row i is lane % 16, columns 4 (lane / 16) .. + 3 of every 16-column slab
	const int row0 = m0 + wr * WM + (lane & 15), col0 = n0 + wc * WN;
	const bool mine = m0 + wr * WM >= m_lo && col0 >= n_lo;  // 64-wide tiles are never ragged
	const int g4 = lane >> 4;
	if constexpr (EPI == EPI_F32_ACC) {
		if (g.k_splits > 1) take_turn();
	}
	if (mine) {
		if constexpr (PAIRED) {
			// four consecutive columns of the first half (acc[i][0]) and the four that belong to them (acc[i][1]); the arithmetic is
			// that of the separate passes, on the rounded values they would read
			const int c = c_lo + wc * 16 + 4 * g4;
			f32x4 tab[RF][2];
			[[maybe_unused]] bool rot = false;
			if constexpr (EPI == EPI_BF16_ROPE) {
				rot = c < g.rope_cols;
				if (rot) {
#pragma unroll
					for (int i = 0; i < RF; i++) {
						const f32x4* tp = reinterpret_cast<const f32x4*>(g.rope_cs + (int64_t)((row0 + i * 16) % g.rope_S) * pair + c % g.rope_D);
						tab[i][0] = tp[0], tab[i][1] = tp[1];
					}
				}
			}
#pragma unroll
			for (int i = 0; i < RF; i++) {
				bf16x4 lo, hi, oa;
#pragma unroll
				for (int t = 0; t < 4; t++) {
					lo[t] = (bf16_t)acc[i][0][t];
					hi[t] = (bf16_t)acc[i][1][t];
					if constexpr (EPI == EPI_BF16_SWIGLU) {
						oa[t] = (bf16_t)swiglu_f((float)lo[t], (float)hi[t]);
					} else if (rot) {
						float rl, rh;
						rope_rot((float)lo[t], (float)hi[t], tab[i][t >> 1][(t & 1) * 2], tab[i][t >> 1][(t & 1) * 2 + 1], rl, rh);
						lo[t] = (bf16_t)rl;
						hi[t] = (bf16_t)rh;
					}
				}
				bf16_t* const cp = reinterpret_cast<bf16_t*>(g.C) + (int64_t)(row0 + i * 16) * g.ldc + c;
				*reinterpret_cast<bf16x4*>(cp) = lo;
				*reinterpret_cast<bf16x4*>(cp + pair) = hi;
				if constexpr (EPI == EPI_BF16_SWIGLU) *reinterpret_cast<bf16x4*>(g.C2 + (int64_t)(row0 + i * 16) * g.ldc2 + c) = oa;
			}
		} else if constexpr (EPI == EPI_BF16_GELU || EPI == EPI_BF16_GELU_BWD || EPI == EPI_BF16_SWIGLU_BWD) {
			const int c = col0 + 16 * (g4 & 1) + 8 * (g4 >> 1);
			constexpr bool SW = EPI == EPI_BF16_SWIGLU_BWD;
			bf16x8 p[RF][CF / 2], u[SW ? RF : 1][CF / 2];  // what the backwards read, all of it before the first store
			if constexpr (EPI != EPI_BF16_GELU) {
#pragma unroll
				for (int i = 0; i < RF; i++)
#pragma unroll
					for (int j = 0; j < CF; j += 2) {
						const bf16_t* r = g.R + (int64_t)(row0 + i * 16) * g.ldr + c + j * 16;
						p[i][j / 2] = *reinterpret_cast<const bf16x8*>(r);
						if constexpr (SW) u[i][j / 2] = *reinterpret_cast<const bf16x8*>(r + g.N);
					}
			}
#pragma unroll
			for (int i = 0; i < RF; i++)
#pragma unroll
				for (int j = 0; j < CF; j += 2) {
					pair_slabs(acc[i][j], acc[i][j + 1]);
					bf16x8 o, o2;
#pragma unroll
					for (int t = 0; t < 8; t++) {
						const float d = (float)(bf16_t)(t < 4 ? acc[i][j][t] : acc[i][j + 1][t - 4]);
						if constexpr (EPI == EPI_BF16_GELU) {
							o[t] = (bf16_t)d;
							o2[t] = (bf16_t)gelu_f(d);
						} else if constexpr (EPI == EPI_BF16_GELU_BWD) {
							o[t] = (bf16_t)(d * gelu_grad_f((float)p[i][j / 2][t]));
						} else {
							float dg, du;
							swiglu_bwd_f(d, (float)p[i][j / 2][t], (float)u[i][j / 2][t], dg, du);
							o[t] = (bf16_t)dg;
							o2[t] = (bf16_t)du;
						}
					}
					const int64_t row = row0 + i * 16;
					bf16_t* const cp = reinterpret_cast<bf16_t*>(g.C) + row * g.ldc + c + j * 16;
					*reinterpret_cast<bf16x8*>(cp) = o;
					if constexpr (SW) *reinterpret_cast<bf16x8*>(cp + g.N) = o2;
					if constexpr (EPI == EPI_BF16_GELU) *reinterpret_cast<bf16x8*>(g.C2 + row * g.ldc2 + c + j * 16) = o2;
					if constexpr (SW) {
						if (g.C2) {  // the activation again, for a stash that dropped it
							bf16x8 oa;
#pragma unroll
							for (int t = 0; t < 8; t++) oa[t] = (bf16_t)swiglu_f((float)p[i][j / 2][t], (float)u[i][j / 2][t]);
							*reinterpret_cast<bf16x8*>(g.C2 + row * g.ldc2 + c + j * 16) = oa;
						}
					}
				}
		} else if constexpr (EPI == EPI_BF16 || EPI == EPI_BF16_RESID) {
			if constexpr (CF == 1) {  // 32x32 tiles: one 16-column slab, four columns per lane
				static_assert(RF == 1, "one slab");
				bf16x4 rs{}, o;
				if constexpr (EPI == EPI_BF16_RESID) rs = *reinterpret_cast<const bf16x4*>(g.R + (int64_t)row0 * g.ldr + col0 + 4 * g4);
#pragma unroll
				for (int t = 0; t < 4; t++) {
					float v = acc[0][0][t];
					if constexpr (EPI == EPI_BF16_RESID) v += (float)rs[t];
					o[t] = (bf16_t)v;
				}
				*reinterpret_cast<bf16x4*>(reinterpret_cast<bf16_t*>(g.C) + (int64_t)row0 * g.ldc + col0 + 4 * g4) = o;
			} else {
			static_assert(CF % 2 == 0, "slabs are stored in pairs");
			const int c = col0 + 16 * (g4 & 1) + 8 * (g4 >> 1);
			bf16x8 rs[EPI == EPI_BF16_RESID ? RF : 1][CF / 2];
			if constexpr (EPI == EPI_BF16_RESID) {
#pragma unroll
				for (int i = 0; i < RF; i++)
#pragma unroll
					for (int j = 0; j < CF; j += 2) rs[i][j / 2] = *reinterpret_cast<const bf16x8*>(g.R + (int64_t)(row0 + i * 16) * g.ldr + c + j * 16);
			}
#pragma unroll
			for (int i = 0; i < RF; i++)
#pragma unroll
				for (int j = 0; j < CF; j += 2) {
					pair_slabs(acc[i][j], acc[i][j + 1]);
					bf16x8 o;
#pragma unroll
					for (int t = 0; t < 8; t++) {
						float v = t < 4 ? acc[i][j][t] : acc[i][j + 1][t - 4];
						if constexpr (EPI == EPI_BF16_RESID) v += (float)rs[i][j / 2][t];
						o[t] = (bf16_t)v;
					}
					*reinterpret_cast<bf16x8*>(reinterpret_cast<bf16_t*>(g.C) + (int64_t)(row0 + i * 16) * g.ldc + c + j * 16) = o;
					// a slab leaves before the next is read: left alone the scheduler may keep all stores for the end, 0.2 us of a
					// tile's 4 to 5 (128x64, K = 64: 128 x 9344 4.33 -> 4.50 us that way; a d = 256 GPT stage 2.80 -> 2.83 ms)
					__builtin_amdgcn_sched_barrier(0);
				}
			}
		} else {
			constexpr bool ACCUM = EPI == EPI_F32_ACC || EPI == EPI_F32_ACC_SCALE;
			float* const cp = reinterpret_cast<float*>(g.C) + (int64_t)row0 * g.ldc + col0 + 4 * g4;
			if (EPI == EPI_F32_ACC && g.k_splits > 1) {
#pragma unroll
				for (int i = 0; i < RF; i++)
#pragma unroll
					for (int j = 0; j < CF; j++)
#pragma unroll
						for (int t = 0; t < 4; t++) unsafeAtomicAdd(cp + (int64_t)i * 16 * g.ldc + j * 16 + t, acc[i][j][t]);
			} else {
				f32x4 cv[ACCUM ? RF : 1][CF];
				if constexpr (ACCUM) {  // every load of the wave's share before the first store
#pragma unroll
					for (int i = 0; i < RF; i++)
#pragma unroll
						for (int j = 0; j < CF; j++) cv[i][j] = *reinterpret_cast<const f32x4*>(cp + (int64_t)i * 16 * g.ldc + j * 16);
				}
#pragma unroll
				for (int i = 0; i < RF; i++)
#pragma unroll
					for (int j = 0; j < CF; j++) {
						if constexpr (ACCUM) acc[i][j] += cv[i][j];
						if constexpr (EPI == EPI_F32_ACC_SCALE) {  // as in gemm_dma_tile: the bits of scale_grads
							acc[i][j] *= g.scale;
							bf16x4 o;
#pragma unroll
							for (int t = 0; t < 4; t++) o[t] = (bf16_t)acc[i][j][t];
							*reinterpret_cast<bf16x4*>(g.C2 + (int64_t)(row0 + i * 16) * g.ldc2 + col0 + 4 * g4 + j * 16) = o;
						}
						*reinterpret_cast<f32x4*>(cp + (int64_t)i * 16 * g.ldc + j * 16) = acc[i][j];
					}
			}
		}
	}
	if constexpr (EPI == EPI_F32_ACC) {
		if (g.k_splits > 1) pass_turn();
	}
	wait_vmcnt<0>();  // the loads past the end of K land in LDS too
}

template <int BM, int BN, bool AT, bool BT, int EPI, bool SHORT>
__global__ __launch_bounds__(256) void gemm_ring_kernel(Args g) {
	// Workgroup w runs on XCD w % 8: every XCD takes a contiguous run of tiles (the splits of a tile side by side), walked in
	// groups of eight tile rows that share their columns' slabs of B in its L2.
	const int ntiles = g.tiles_m * g.tiles_n;
	int ksplit, pid;
	{
		const int chunk = (ntiles + 7) >> 3, x = blockIdx.x & 7, slot = blockIdx.x >> 3;
		ksplit = slot % g.k_splits;
		pid = x * chunk + slot / g.k_splits;
		if (slot / g.k_splits >= chunk || pid >= ntiles) return;
	}
	gemm_ring_tile<BM, BN, AT, BT, EPI, SHORT>(g, pid, ksplit);
}

// The weight gradients of a stage's layers in one launch, as gemm_dw_group_kernel of gemm_dma.hip, for stages so small that its
// 256x256 tiles leave most of the chip idle: the 128x128 tiles of all problems are one sequence, of which every XCD takes a
// contiguous eighth.  What bounds it: one tile's chain (ring fill, slices, read-modify-write),
// 12.7 us for two blocks of a 512-wide Llama stage over 512 tokens against 23.7 on 60 tiles of 256x256 (see gemm_dw_group()).
struct GroupArgs {
	int n, tiles;
	int first[DW_GROUP_MAX];  // problem p's first tile in the sequence
	Args a[DW_GROUP_MAX];
};
template <int EPI>
__global__ __launch_bounds__(256) void gemm_ring_dw_group_kernel(GroupArgs ga) {
	const int chunk = (ga.tiles + 7) >> 3, x = blockIdx.x & 7, slot = blockIdx.x >> 3, t = x * chunk + slot;
	if (slot >= chunk || t >= ga.tiles) return;
	int p = 0;
	for (int i = 1; i < ga.n; i++)
		if (t >= ga.first[i]) p = i;
	p = __builtin_amdgcn_readfirstlane(p);
	gemm_ring_tile<128, 128, true, true, EPI, false>(ga.a[p], t - ga.first[p], 0);
}

template <int BM, int BN, bool AT, bool BT, int EPI, bool SHORT>
static int launch(const Args& g, hipStream_t stream) {
	using Sh = Shape<BM, BN, SHORT>;
	auto kern = gemm_ring_kernel<BM, BN, AT, BT, EPI, SHORT>;
	static bool attr_set = false;
	if (!attr_set) {
		ELF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Sh::SMEM));
		attr_set = true;
	}
	const int ntiles = g.tiles_m * g.tiles_n;
	ELF_LAUNCH(kern, dim3(8 * ((ntiles + 7) / 8) * g.k_splits), dim3(256), (Sh::SMEM), stream, g);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

template <int BM, int BN, bool AT, bool BT>
static int launch_epi(const Args& g, int epi, hipStream_t stream) {
	if constexpr (!AT) {
		if (g.K <= RING_SHORT_K && epi == EPI_BF16) return launch<BM, BN, AT, BT, EPI_BF16, true>(g, stream);
		if (g.K <= RING_SHORT_K && epi == EPI_BF16_RESID) return launch<BM, BN, AT, BT, EPI_BF16_RESID, true>(g, stream);
	}
	switch (epi) {
		case EPI_BF16: return launch<BM, BN, AT, BT, EPI_BF16, false>(g, stream);
		case EPI_BF16_RESID: return launch<BM, BN, AT, BT, EPI_BF16_RESID, false>(g, stream);
		case EPI_F32_ACC: return launch<BM, BN, AT, BT, EPI_F32_ACC, false>(g, stream);
		case EPI_F32_STORE: return launch<BM, BN, AT, BT, EPI_F32_STORE, false>(g, stream);
	}
	set_error("gemm: unknown epilogue %d", epi);
	return -1;
}

// 32x32 tiles: bf16 outputs with a k-contiguous A
template <bool BT>
static int launch_tiny(const Args& g, int epi, hipStream_t stream) {
	if (epi == EPI_BF16) return g.K <= RING_SHORT_K ? launch<32, 32, false, BT, EPI_BF16, true>(g, stream) : launch<32, 32, false, BT, EPI_BF16, false>(g, stream);
	return g.K <= RING_SHORT_K ? launch<32, 32, false, BT, EPI_BF16_RESID, true>(g, stream) : launch<32, 32, false, BT, EPI_BF16_RESID, false>(g, stream);
}

template <int BM, int BN>
static int launch_layout(Args& g, int a_t, int b_t, int epi, hipStream_t stream) {
	ELF_REQUIRE(g.M >= BM && g.N >= BN, "gemm (ring tile): M at least %d and N at least %d", BM, BN);
	g.tiles_m = (g.M + BM - 1) / BM, g.tiles_n = (g.N + BN - 1) / BN;
	if (epi != EPI_F32_ACC || g.k_splits < 1) g.k_splits = 1;
	g.turn_tag = g.k_splits > 1 && g.tiles_m * g.tiles_n <= TURN_TILES ? next_turn_tag() : 0;
	if (!a_t && !b_t) return launch_epi<BM, BN, false, false>(g, epi, stream);
	if (!a_t && b_t) return launch_epi<BM, BN, false, true>(g, epi, stream);
	if (a_t && b_t) return launch_epi<BM, BN, true, true>(g, epi, stream);
	set_error("gemm: layout A=T,B=R is not used by any stage contraction");
	return -1;
}

}  // namespace ring

int ring_turn_giveups(uint64_t* out) {
	unsigned int n = 0;
	ELF_CHECK_HIP(hipMemcpyFromSymbol(&n, HIP_SYMBOL(ring::turn_giveups), sizeof(n)));
	*out = n;
	return 0;
}

// Arguments are validated by gemm_bf16() before it dispatches here.
int gemm_bf16_ring(int a_t, int b_t, int M, int N, int K, const void* A, int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc, int epi, const void* R,
                   int64_t ldr, int k_splits, int bm, int bn, hipStream_t stream) {
	ELF_REQUIRE(M % 64 == 0 && N % 64 == 0 && K % dma::BKS == 0, "gemm (ring tile): sizes must be multiples of 64");
	ELF_REQUIRE(gemm_reaches(a_t ? dma::BKS : bm, lda) && gemm_reaches(b_t ? dma::BKS : bn, ldb), "gemm (ring tile): leading dimension too large (%lld, %lld)", (long long)lda, (long long)ldb);
	ring::Args g{(const bf16_t*)A, (const bf16_t*)B, C, (const bf16_t*)R, lda, ldb, ldc, ldr, M, N, K, 0, 0, k_splits, 0, nullptr, 0, nullptr, 0, 0, 0, 0.f};
	if (bm == 128 && bn == 128) return ring::launch_layout<128, 128>(g, a_t, b_t, epi, stream);
	if (bm == 64 && bn == 128) return ring::launch_layout<64, 128>(g, a_t, b_t, epi, stream);
	if (bm == 128 && bn == 64) return ring::launch_layout<128, 64>(g, a_t, b_t, epi, stream);
	if (bm == 64 && bn == 64) return ring::launch_layout<64, 64>(g, a_t, b_t, epi, stream);
	if (bm == 32 && bn == 32) {
		g.tiles_m = M / 32, g.tiles_n = N / 32, g.k_splits = 1;
		if (!a_t && (epi == EPI_BF16 || epi == EPI_BF16_RESID)) return b_t ? ring::launch_tiny<true>(g, epi, stream) : ring::launch_tiny<false>(g, epi, stream);
	}
	set_error("gemm (ring tile): unknown tile %dx%d", bm, bn);
	return -1;
}

namespace ring {
template <bool BT, int EPI>
static int launch_act(const Args& g, hipStream_t stream) {
	return g.K <= RING_SHORT_K ? launch<64, 64, false, BT, EPI, true>(g, stream) : launch<64, 64, false, BT, EPI, false>(g, stream);
}
}  // namespace ring

int gemm_ring_act(int M, int N, int K, const void* A, int64_t lda, const void* B, int64_t ldb, void* C, int64_t ldc, int epi, const void* R, int64_t ldr,
                  hipStream_t stream, void* C2, int64_t ldc2, const void* rope_cs, int rope_S, int rope_cols, int rope_D) {
	const bool bt = epi == EPI_BF16_SWIGLU_BWD || epi == EPI_BF16_GELU_BWD;
	ELF_REQUIRE(M > 0 && N > 0 && M % 64 == 0 && N % 64 == 0 && K > 0 && K % dma::BKS == 0, "gemm (ring tile): sizes must be multiples of 64");
	// the rows of a pair are addressed with 32-bit byte offsets from the tile's first row
	const int brows = epi == EPI_BF16_SWIGLU ? N / 2 + 64 : epi == EPI_BF16_ROPE ? rope_D : 64;
	ELF_REQUIRE(gemm_reaches(64, lda) && gemm_reaches(brows, ldb), "gemm (ring tile): leading dimension too large (%lld, %lld)", (long long)lda, (long long)ldb);
	ELF_REQUIRE(epi != EPI_BF16_SWIGLU || N % 128 == 0, "gemm (ring tile): the SwiGLU epilogue needs F to be a multiple of 64");
	ELF_REQUIRE(epi != EPI_BF16_ROPE || (rope_cs && rope_S > 0 && (rope_D == 64 || rope_D == 128) && N % rope_D == 0 && rope_cols % rope_D == 0),
	            "gemm (ring tile): the RoPE epilogue needs a table and whole heads of 64 or 128 columns");
	ELF_REQUIRE((C2 || (epi != EPI_BF16_SWIGLU && epi != EPI_BF16_GELU)) && (R || !bt), "gemm (ring tile): an epilogue's operand is missing");
	ring::Args g{(const bf16_t*)A, (const bf16_t*)B, C, (const bf16_t*)R, lda, ldb, ldc, ldr, M, N, K, M / 64, N / 64, 1, 0,
	             (bf16_t*)C2, ldc2, (const float2*)rope_cs, rope_S, rope_cols, rope_D, 0.f};
	switch (epi) {
		case EPI_BF16_SWIGLU: return ring::launch_act<false, EPI_BF16_SWIGLU>(g, stream);
		case EPI_BF16_ROPE: return ring::launch_act<false, EPI_BF16_ROPE>(g, stream);
		case EPI_BF16_GELU: return ring::launch_act<false, EPI_BF16_GELU>(g, stream);
		case EPI_BF16_GELU_BWD: return ring::launch_act<true, EPI_BF16_GELU_BWD>(g, stream);
		case EPI_BF16_SWIGLU_BWD: return ring::launch_act<true, EPI_BF16_SWIGLU_BWD>(g, stream);
	}
	set_error("gemm (ring tile): unknown epilogue %d", epi);
	return -1;
}

// Arguments are validated by gemm_dw_group() before it dispatches here.
int gemm_ring_dw_group(int n, const DwProblem* pr, int K, float scale, hipStream_t stream) {
	ring::GroupArgs ga{};
	ga.n = n;
	for (int i = 0; i < n; i++) {
		const DwProblem& q = pr[i];
		ring::Args& a = ga.a[i];
		a = ring::Args{(const bf16_t*)q.dY, (const bf16_t*)q.X, q.acc, nullptr, q.lddy, q.ldx, q.N, 0, q.M, q.N, K, (q.M + 127) / 128, (q.N + 127) / 128, 1, 0,
		               (bf16_t*)q.grad_bf16, q.N, nullptr, 0, 0, 0, scale};
		ga.first[i] = ga.tiles;
		ga.tiles += a.tiles_m * a.tiles_n;
	}
	using Sh = ring::Shape<128, 128, false>;
	auto kern = scale != 0.f ? ring::gemm_ring_dw_group_kernel<EPI_F32_ACC_SCALE> : ring::gemm_ring_dw_group_kernel<EPI_F32_ACC>;
	static bool attr_set[2] = {};
	if (bool& set = attr_set[scale != 0.f]; !set) {
		ELF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Sh::SMEM));
		set = true;
	}
	ELF_LAUNCH(kern, dim3(8 * ((ga.tiles + 7) / 8)), dim3(256), (Sh::SMEM), stream, ga);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

}  // namespace elf
