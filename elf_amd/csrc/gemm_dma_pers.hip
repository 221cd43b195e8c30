// The persistent kernel of the forward products on 256x256 tiles.
#include "gemm_dma_tile.h"

namespace elf {

namespace dma {

// ------------------------------------------------------------------------------------------------------------
// Persistent forward kernel: both operands k-contiguous, 256x256 tiles, four waves with 128x128 wave tiles - the loop
// of gemm_dma_kernel<4, 8, false, false, .> with two changes that take the tile boundary out of the matrix pipe's way.
//
//  * The epilogue leaves from registers.  The MFMA operands are swapped (the weight rows feed the m side), so a lane
//    holds four consecutive columns of ONE output row per accumulator tile, and the order in which weight rows enter
//    the four column slabs of a half-step is permuted (slab jj, m slot 4 g + r  <-  column 32 (jj / 2) + 8 g + 4 (jj % 2) + r)
//    so that the lane's 16 values of a half-step are two runs of 8 consecutive columns: one 16-byte store each, the four
//    lane groups of a row together 64 contiguous bytes.  No LDS staging, no barrier, a quarter of the instructions.
//    For column slab jj of half h and k32 half kq lane l reads tile row wc * 128 + h * 64 + 32 (jj / 2) + 8 ((l % 16) / 4)
//    + 4 (jj % 2) + l % 4 at k = 32 kq + 8 (l / 16) .. + 7; the B tile's chunk swizzle follows these rows (rb_swz) so
//    that the 16 lanes of a k chunk still hit 16 different 16-byte bank groups.
//  * A workgroup walks tiles pid, pid + grid, ... and its K-slice pipeline never drains: the last two slices of a tile
//    fetch the first two of the next (the loop's "slice past the end of K" is the next tile's slice 0), the LDS ring is
//    not needed by the epilogue, and the first MFMAs of a tile write their accumulators (C = 0 form) instead of adding
//    to cleared ones.
// With the ring of two slices of A and three of B (see Shape), before -> after, cold operands: 8192 x 4096 x 14336 with a residual
// 691 -> 622 us, 8192 x 4096 x 4096 212 -> 198, 2688 x 4096 x 14336 327 -> 266, SwiGLU 8192 x 28672 x 4096 1365 -> 1332,
// 8192 x 50304 x 768 611 -> 556.  (K / 64 may be odd since the ring's position is kept at run time: with one code for every slice
// instead of one per stage.)  Leaving the tile before's stores in flight past its successor's first slice gave nothing.
// Results are bit-identical to gemm_dma_kernel's: same products, same accumulation order along K, same roundings.
__device__ __forceinline__ int rb_swz(int row) { return (((row >> 3) & 3) << 1) | ((row >> 1) & 1); }

template <bool PAIRED>
__device__ __forceinline__ void lane_offsets_rb(int wave, int lane, int64_t ld, uint32_t (&off)[8], int64_t pair_rows) {
#pragma unroll
	for (int i = 0; i < 8; i++) {
		const int q = wave * 8 + i;
		const int row = q * 8 + (lane >> 3), slot = lane & 7;
		const int64_t grow = PAIRED ? (row >> 7) * 64 + (row & 63) + ((row >> 6) & 1) * pair_rows : row;
		off[i] = (uint32_t)((grow * ld + ((slot ^ rb_swz(row)) << 3)) * 2);
	}
}

// acc = a b: the first MFMA of an accumulator tile in a tile's K loop
__device__ __forceinline__ void mfma_init(f32x4& acc, const bf16x8& a, const bf16x8& b) {
	asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc) : "v"(a), "v"(b));
}

template <int EPI, bool EDGE>
__global__ __launch_bounds__(256) void gemm_pers_kernel(Args g) {
	using Sh = Shape<4, 8>;
	constexpr int BM = 256, RF = 8, A_BYTES = Sh::A_BYTES, B_BYTES = Sh::B_BYTES, NSA = Sh::NSA, NSB = Sh::NSB;
	constexpr int LOADS_A = Sh::LOADS_A, LOADS_B = Sh::LOADS_B;
	constexpr bool PAIRED = EPI == EPI_BF16_SWIGLU;
	static_assert(NSA == 2 && NSB == 3 && LOADS_A == 8 && LOADS_B == 8, "ring of two slices of A and three of B, 32 KiB each");
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
	const int tid = threadIdx.x;
	const int lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int wr = wave >> 1, wc = wave & 1;
	const int ntiles = g.tiles_m * g.tiles_n;
	const int nk = g.K / BKS;  // at least 2

	uint32_t aoff[LOADS_A], boff[LOADS_B];
	lane_offsets<false, LOADS_A, false, BM>(wave, lane, g.lda, aoff);
	lane_offsets_rb<PAIRED>(wave, lane, g.ldb, boff, g.N / 2);
	const uint32_t lds_a = lds_addr(smem) + wave * (LOADS_A * 1024);
	const uint32_t lds_b = lds_addr(smem) + NSA * A_BYTES + wave * (LOADS_B * 1024);

	auto tile_ptrs = [&](int tile, int& m0, int& n0, const bf16_t*& Ap, const bf16_t*& Bp) {
		tile_origin<BM>(g, tile, m0, n0);
		m0 = __builtin_amdgcn_readfirstlane(m0);
		n0 = __builtin_amdgcn_readfirstlane(n0);
		if constexpr (EDGE) clip_tile<BM>(g, m0, n0);
		Ap = g.A + (int64_t)m0 * g.lda;
		Bp = g.B + (int64_t)(PAIRED ? n0 / 2 : n0) * g.ldb;
	};
	int tile = blockIdx.x, m0, n0, m0_n = 0, n0_n = 0;
	const bf16_t *Ap, *Bp, *Ap_n, *Bp_n;
	tile_ptrs(tile, m0, n0, Ap, Bp);
	Ap_n = Ap, Bp_n = Bp;
	bool has_next = false;

	// Loads of slice `step` of the current tile into ring stage `stage`; steps nk and nk + 1 are slices 0 and 1 of the next tile
	// or, behind the workgroup's last tile, loads of its own first slices that nobody reads, into stages that nobody reads
	// any more.
	struct Loads {
		const bf16_t* p;
		uint32_t lds;
	};
	auto loads_a = [&](int step, int stage) { return Loads{(step < nk ? Ap : Ap_n) + (int64_t)(step < nk ? step : step - nk) * BKS, lds_a + (uint32_t)stage * A_BYTES}; };
	auto loads_b = [&](int step, int stage) { return Loads{(step < nk ? Bp : Bp_n) + (int64_t)(step < nk ? step : step - nk) * BKS, lds_b + (uint32_t)stage * B_BYTES}; };
	auto piece_a = [&](const Loads& l, auto pc) { dma16_at<decltype(pc)::value * 1024>(l.p, aoff[decltype(pc)::value], l.lds); };
	auto piece_b = [&](const Loads& l, auto pc) { dma16_at<decltype(pc)::value * 1024>(l.p, boff[decltype(pc)::value], l.lds); };

	f32x4 acc[RF][8];
	bf16x8 fa[2][RF], fb[2][4];
	static_assert(pieces_have_slots(RF * 4, LOADS_A) && pieces_have_slots(RF * 4, LOADS_B / 2), "a half-step has too few even MFMA slots for its loads");
	static_for<2>([&](auto sc) {
		constexpr int S = decltype(sc)::value;
		static_for<LOADS_A>([&](auto pc) { piece_a(loads_a(S, S), pc); });
		static_for<LOADS_B>([&](auto pc) { piece_b(loads_b(S, S), pc); });
	});
	wait_vmcnt<LOADS_A + LOADS_B>();
	__syncthreads();
	// Per-lane LDS addresses of the fragment reads for the two k32 halves of a slice (the chunk swizzles only look at
	// lane bits); row slab and column slab are compile-time byte offsets in the read instructions.  The addresses move on by a
	// stage with every slice: a tile may start anywhere in the ring, whatever K is.
	uint32_t a_lane[2], b_lane[2];
	{
		const int l15 = lane & 15, q4 = lane >> 4;
#pragma unroll
		for (int kq = 0; kq < 2; kq++) {
			a_lane[kq] = lds_addr(smem) + (uint32_t)((wr * 128 + l15) * 128 + (((4 * kq + q4) ^ ((l15 >> 1) & 7)) << 4));
			b_lane[kq] = lds_addr(smem) + NSA * A_BYTES + (uint32_t)((wc * 128 + 8 * (l15 >> 2) + (l15 & 3)) * 128 + (((4 * kq + q4) ^ rb_swz(8 * (l15 >> 2) + (l15 & 3))) << 4));
			asm volatile("" : "+v"(a_lane[kq]), "+v"(b_lane[kq]));
		}
	}
	auto read_a = [&](int kq, auto ic) -> bf16x8 {
		constexpr uint32_t IMM = decltype(ic)::value * (16 * 128);
		return *reinterpret_cast<const bf16x8 ELF_LDS*>((uintptr_t)(a_lane[kq] + IMM));
	};
	auto read_b = [&](int kq, int h, auto jc) -> bf16x8 {
		constexpr int JJ = decltype(jc)::value;
		constexpr uint32_t IMM = (32 * (JJ >> 1) + 4 * (JJ & 1)) * 128;
		return *reinterpret_cast<const bf16x8 ELF_LDS*>((uintptr_t)(b_lane[kq] + IMM + (uint32_t)h * (64 * 128)));
	};
	static_for<RF>([&](auto ic) { fa[0][decltype(ic)::value] = read_a(0, ic); });
	static_for<4>([&](auto jc) { fb[0][decltype(jc)::value] = read_b(0, 0, jc); });

	// One half-step (see gemm_dma_kernel): RF * 4 MFMAs, the next half-step's fragment reads behind the odd ones, its share of
	// a slice's loads behind even ones (dealt 0: none, 1: a slice of A, 2 and 3: the halves of a slice of B).  FIRST: the
	// accumulator tiles of this half-step are written, not added to.
	auto half_step = [&](int abuf, int bbuf, auto hc, auto first, int pb_buf, int pb_kq, int pb_h, bool pa, int pa_buf, int pa_kq, const Loads& ld, auto dealt) {
		constexpr int DEALT = decltype(dealt)::value, NP = DEALT == 0 ? 0 : DEALT == 1 ? LOADS_A : LOADS_B / 2, H = decltype(hc)::value, NM = RF * 4;
		constexpr bool FIRST = decltype(first)::value;
		static_for<NM>([&](auto nc) {
			constexpr int n = decltype(nc)::value, i = n / 4, j = n % 4;
			if constexpr (FIRST) mfma_init(acc[i][H * 4 + j], fb[bbuf][j], fa[abuf][i]);
			else mfma_acc(acc[i][H * 4 + j], fb[bbuf][j], fa[abuf][i]);
			if constexpr (n % 2 == 1) {
				constexpr int r = n / 2;
				if constexpr (r < 4) {
					fb[pb_buf][r] = read_b(pb_kq, pb_h, std::integral_constant<int, r>{});
				} else if constexpr (r - 4 < RF) {
					if (pa) fa[pa_buf][r - 4] = read_a(pa_kq, std::integral_constant<int, r - 4>{});
				}
			}
			constexpr int piece = NP == 0 ? -1 : piece_in_slot(n, NM, NP);
			if constexpr (piece >= 0) {
				if constexpr (DEALT == 1) piece_a(ld, std::integral_constant<int, piece>{});
				else piece_b(ld, std::integral_constant<int, (DEALT - 2) * (LOADS_B / 2) + piece>{});
			}
			__builtin_amdgcn_sched_barrier(0);
		});
	};
	int stage_a = 0, stage_b = 0;  // of the current slice
	auto slice = [&](auto first, int kt) {
		constexpr std::integral_constant<int, 0> H0{}, NONE{};
		constexpr std::integral_constant<int, 1> H1{}, SLICE_A{};
		constexpr std::integral_constant<int, 2> FIRST_B{};
		constexpr std::integral_constant<int, 3> SECOND_B{};
		constexpr std::false_type ADD{};
		const Loads lb = loads_b(kt + 2, stage_b == 0 ? 2 : stage_b - 1), la = loads_a(kt + 2, stage_a);
		half_step(0, 0, H0, first, 1, 0, 1, false, 0, 0, lb, FIRST_B);
		half_step(0, 1, H1, first, 0, 1, 0, true, 1, 1, lb, SECOND_B);
		half_step(1, 0, H0, ADD, 1, 1, 1, false, 0, 0, la, NONE);
		wait_counters<LOADS_B, 0>();  // slice kt + 1 landed (and the previous tile's stores acknowledged); slice kt fully read
		__syncthreads();
		const uint32_t next_a = stage_a ? (uint32_t)-A_BYTES : (uint32_t)A_BYTES, next_b = stage_b == 2 ? (uint32_t)(-2 * B_BYTES) : (uint32_t)B_BYTES;
#pragma unroll
		for (int kq = 0; kq < 2; kq++) {
			a_lane[kq] += next_a;
			b_lane[kq] += next_b;
		}
		stage_a ^= 1;
		stage_b = stage_b == 2 ? 0 : stage_b + 1;
		half_step(1, 1, H1, ADD, 0, 0, 0, true, 0, 0, la, SLICE_A);
	};

	const int g4 = lane >> 4, rr = lane & 15;
	for (;;) {
		const int tile_n = tile + (int)gridDim.x;
		has_next = tile_n < ntiles;
		if (has_next) tile_ptrs(tile_n, m0_n, n0_n, Ap_n, Bp_n);

		slice(std::true_type{}, 0);
		for (int kt = 1; kt < nk; kt++) slice(std::false_type{}, kt);

		// Epilogue from registers, while the next tile's first two slices are on their way into the ring.  The MFMAs were
		// issued through inline assembly, so the compiler places no wait states between the last of them and the first
		// read of an accumulator: 32 of them here (an 8-pass MFMA needs 11).
		asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
		const int grow0 = m0 + wr * 128 + rr;
		const int gcol0 = n0 + wc * 128;
		// a tile that was moved back (clip_tile): 16-row groups below i_lo and 64-column halves below h_lo are its neighbour's
		const int i_lo = EDGE ? ((m0 + BM - 1) / BM * BM - m0 - wr * 128) >> 4 : 0;
		const int h_lo = EDGE ? (PAIRED ? ((n0 + BN - 1) / BN * BN - n0) / 2 - wc * 64 : (n0 + BN - 1) / BN * BN - n0 - wc * 128) >> 6 : 0;
		// row group i has not left the accumulator registers yet (the compiler would read all of them behind the K loop and spill)
		auto stay = [&](int i) {
#pragma unroll
			for (int j = 0; j < 8; j++) asm volatile("" : "+a"(acc[i][j]));
		};
		// the lane's run t (0..3) of 8 consecutive columns: columns (t / 2) * 64 + (t % 2) * 32 + 8 g4 .. + 7 of the wave's 128
		auto run = [&](int i, int t, float (&v)[8]) {
#pragma unroll
			for (int e = 0; e < 8; e++) v[e] = acc[i][(t >> 1) * 4 + (t & 1) * 2 + (e >> 2)][e & 3];
		};
		auto run_col = [&](int t) { return (t >> 1) * 64 + (t & 1) * 32 + g4 * 8; };
		if constexpr (EPI == EPI_BF16_SWIGLU) {
			// the wave's columns are 64 gate columns (first half-step) and the 64 up columns of the same outputs (second)
			const int F = g.N / 2, cg0 = n0 / 2 + wc * 64;
#pragma unroll
			for (int i = 0; i < RF; i++) {
				__builtin_amdgcn_sched_barrier(0);  // one row group at a time (see the residual epilogue below)
				stay(i);
				if (EDGE && (i < i_lo || h_lo > 0)) continue;
				const int64_t row = grow0 + i * 16;
#pragma unroll
				for (int t = 0; t < 2; t++) {
					float gv[8], uv[8];
					run(i, t, gv);
					run(i, 2 + t, uv);
					bf16x8 og, ou, oa;
#pragma unroll
					for (int e = 0; e < 8; e++) {
						og[e] = (bf16_t)gv[e];
						ou[e] = (bf16_t)uv[e];
						oa[e] = (bf16_t)swiglu_f((float)og[e], (float)ou[e]);
					}
					const int c = cg0 + t * 32 + g4 * 8;
					bf16_t* cp = reinterpret_cast<bf16_t*>(g.C) + row * g.ldc + c;
					*reinterpret_cast<bf16x8*>(cp) = og;
					*reinterpret_cast<bf16x8*>(cp + F) = ou;
					*reinterpret_cast<bf16x8*>(g.C2 + row * g.ldc2 + c) = oa;
				}
			}
		} else {
			static_assert(EPI == EPI_BF16 || EPI == EPI_BF16_RESID, "epilogues of the persistent forward kernel");
			// residual (or bias row, ldr = 0): every load of the wave's 128 x 128 share goes out before the first store (a lone
			// wave has nothing else to cover the trips to memory with; inside the store loop each would be awaited alone)
			bf16x8 rs[EPI == EPI_BF16_RESID ? RF : 1][4];
			if constexpr (EPI == EPI_BF16_RESID) {
#pragma unroll
				for (int i = 0; i < RF; i++)
#pragma unroll
					for (int t = 0; t < 4; t++) rs[i][t] = *reinterpret_cast<const bf16x8*>(g.R + (int64_t)(grow0 + i * 16) * g.ldr + gcol0 + run_col(t));
			}
			// (left to itself the scheduler reads all 256 accumulators into vector registers first and then has room for
			// two loads at a time: the row groups are fenced off from each other and from the loads)
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for (int i = 0; i < RF; i++) {
				__builtin_amdgcn_sched_barrier(0);
				stay(i);
				if (EDGE && i < i_lo) continue;
				bf16_t* cp = reinterpret_cast<bf16_t*>(g.C) + (int64_t)(grow0 + i * 16) * g.ldc + gcol0;
#pragma unroll
				for (int t = 0; t < 4; t++) {
					if (EDGE && (t >> 1) < h_lo) continue;
					float v[8];
					run(i, t, v);
					bf16x8 o;
#pragma unroll
					for (int e = 0; e < 8; e++) {
						if constexpr (EPI == EPI_BF16_RESID) v[e] += (float)rs[i][t][e];
						o[e] = (bf16_t)v[e];
					}
					*reinterpret_cast<bf16x8*>(cp + run_col(t)) = o;
				}
			}
		}
		if (!has_next) break;
		tile = tile_n, m0 = m0_n, n0 = n0_n, Ap = Ap_n, Bp = Bp_n;
		asm volatile("s_nop 7" ::: "memory");  // accumulator reads above, accumulator writes by the next tile's first MFMAs
	}
	wait_vmcnt<0>();  // the loads past the last tile land in LDS too
}

template <int EPI, bool EDGE>
static int launch_pers_sized(const Args& a, hipStream_t stream) {
	using Sh = Shape<4, 8>;
	constexpr int smem = Sh::RING_BYTES;
	auto kern = gemm_pers_kernel<EPI, EDGE>;
	static bool attr_set = false;
	if (!attr_set) {
		ELF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
		attr_set = true;
	}
	const int ntiles = a.tiles_m * a.tiles_n;
	ELF_LAUNCH(kern, dim3(ntiles < PERS_WORKGROUPS ? ntiles : PERS_WORKGROUPS), dim3(256), smem, stream, a);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}
template <int EPI>
static int launch_pers_epi(const Args& a, hipStream_t stream) {
	return a.M % 256 || a.N % BN ? launch_pers_sized<EPI, true>(a, stream) : launch_pers_sized<EPI, false>(a, stream);
}

int launch_pers(const Args& a, int epi, hipStream_t stream) {
	switch (epi) {
		case EPI_BF16: return launch_pers_epi<EPI_BF16>(a, stream);
		case EPI_BF16_RESID: return launch_pers_epi<EPI_BF16_RESID>(a, stream);
		default: return launch_pers_epi<EPI_BF16_SWIGLU>(a, stream);
	}
}

}  // namespace dma

}  // namespace elf
