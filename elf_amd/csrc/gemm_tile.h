// What the direct-to-LDS GEMM kernels share: the layout of an operand tile in LDS (64 wide K slices, filled by
// global_load_lds_dwordx4, unpadded and XOR-swizzled) and the reads of v_mfma_f32_16x16x32_bf16 operand fragments from it.
#pragma once
#include <type_traits>

#include "common.h"
#include "lds_dma.h"

namespace elf {
namespace dma {

constexpr int BKS = 64;  // K slice

// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>), unrolled at compile time.
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
	if constexpr (N > 0) {
		static_for<N - 1>(f);
		f(std::integral_constant<int, N - 1>{});
	}
}

// Byte offsets (relative to the tile origin of the current K slice) of the 16-byte chunks this
// lane fetches for one operand (< 2^31: 256 rows of at most 64 K elements).  "R" tiles are
// [256 rows][128 B], "T" tiles [64 k][512 B] ([64 k][256 B] for the 128 rows of A in a 128x256 tile); LDS chunk slot s of a row holds global chunk
// s ^ f(row) with f chosen so that the lanes of a fragment read spread over all banks: an "R"
// read takes one chunk from each of 32 rows (f = (row / 2) % 8), a "T" transpose read takes 64
// contiguous bytes from each of four k rows per half-wave (f = 4 * (k % 8): the four rows land in
// four different 64-byte bank groups; with 2 * (k % 8) pairs of rows shared one and the bank-conflict
// counter read half of the LDS-active cycles).
// chunk swizzle of reduction-major ("T") tiles as a function of the k row
// ROWS = 128 (a k row is 256 bytes, exactly one row of banks): the four k rows of a half-wave's transpose read
// are moved into four different 64-byte groups by (k % 4) * 4 chunks, rows k and k + 8 apart by two chunks; ROWS = 64
// (two k rows span the banks): the same for pairs of rows
template <int ROWS = 256>
__device__ __forceinline__ int t_swz(int k) {
	if constexpr (ROWS == 192) return (((k >> 1) & 1) << 1) | (((k >> 3) & 1) << 2);  // (rows k and k + 2 start at the same bank)
	if constexpr (ROWS == 32) return ((k >> 3) & 1) << 1;  // (four k rows span the banks: rows k and k + 8 take different halves)
	if constexpr (ROWS == 64) return (((k >> 1) & 1) << 2) ^ (((k >> 3) & 1) << 1);
	return ((k & (ROWS == 256 ? 7 : 3)) << 2) ^ (((k >> 3) & 1) << 1);
}

// PAIRED (k-contiguous operands only): the 256 tile rows are not 256 consecutive operand rows but, for
// each 128-row half, 64 consecutive rows followed by the 64 rows `pair_rows` further down — the gate and
// up rows of the same 64 SwiGLU columns, which thereby land in one wave's accumulators.
template <bool T, int LPO, bool PAIRED = false, int ROWS = 256>
__device__ __forceinline__ void lane_offsets(int wave, int lane, int64_t ld, uint32_t (&off)[LPO], int64_t pair_rows = 0) {
#pragma unroll
	for (int i = 0; i < LPO; i++) {
		const int q = wave * LPO + i;  // which 1 KiB piece of the operand tile
		if constexpr (!T) {
			const int row = q * 8 + (lane >> 3), slot = lane & 7;
			const int64_t grow = PAIRED ? (row >> 7) * 64 + (row & 63) + ((row >> 6) & 1) * pair_rows : row;
			off[i] = (uint32_t)((grow * ld + ((slot ^ ((row >> 1) & 7)) << 3)) * 2);
		} else {
			constexpr int CPR = ROWS / 8;  // 16-byte chunks per k row; a 1 KiB piece holds 64 of them
			const int krow = (q * 64 + lane) / CPR, slot = (q * 64 + lane) % CPR;
			off[i] = (uint32_t)((krow * ld + ((slot ^ t_swz<ROWS>(krow)) << 3)) * 2);
		}
	}
}

// Operand fragment of v_mfma_f32_16x16x32_bf16 for the 16-row slab at `row0` and the k32 half `kq`
// of the current slice: lane l holds row (or column) row0 + l % 16 at k = 32 kq + 8 (l / 16) .. + 7.
// "R" tiles give it with one 16-byte read; "T" tiles with two transpose reads, each of which hands
// the 16 lanes of a group the 4 (k) x 16 (rows) block they address row-wise.
template <bool T, int ROWS = 256>
__device__ __forceinline__ bf16x8 frag(const unsigned char* base, int row0, int kq, int lane) {
	if constexpr (!T) {
		const int r = row0 + (lane & 15);
		const int c = (4 * kq + (lane >> 4)) ^ ((r >> 1) & 7);
		return *reinterpret_cast<const bf16x8*>(base + r * 128 + c * 16);
	} else {
		const int j = lane & 15;
		const int m = row0 + 4 * (j & 3);
		const int kk = kq * 32 + 8 * (lane >> 4) + (j >> 2);
		const int c0 = (m >> 3) ^ t_swz<ROWS>(kk);
		const int c1 = (m >> 3) ^ t_swz<ROWS>(kk + 4);
		const unsigned char* p0 = base + kk * (ROWS * 2) + c0 * 16 + (j & 1) * 8;
		const unsigned char* p1 = base + (kk + 4) * (ROWS * 2) + c1 * 16 + (j & 1) * 8;
		s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(p0));
		s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(p1));
		return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
	}
}

// The two byte offsets (within the operand tile of stage 0, k32 half 0) that frag<true> reads for the
// 16-row slab at row0, and the fragment read from them for k32 half kq of the tile at `base`.
template <int ROWS = 256>
__device__ __forceinline__ void frag_t_offsets(int row0, int lane, uint32_t (&o)[2]) {
	const int j = lane & 15;
	const int m = row0 + 4 * (j & 3);
	const int kk = 8 * (lane >> 4) + (j >> 2);
	o[0] = (uint32_t)(kk * (ROWS * 2) + (((m >> 3) ^ t_swz<ROWS>(kk)) << 4) + (j & 1) * 8);
	o[1] = (uint32_t)((kk + 4) * (ROWS * 2) + (((m >> 3) ^ t_swz<ROWS>(kk + 4)) << 4) + (j & 1) * 8);
}
// o: LDS byte addresses; imm: a compile-time byte offset (stage and k32 half) that ends up in the
// instructions' offset fields.  t_swz only looks at k % 16, so the second k32 half of a tile lies 32 rows
// (of 2 * ROWS bytes) further on.
__device__ __forceinline__ bf16x8 frag_t_at(const uint32_t (&o)[2], uint32_t imm) {
	s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(uintptr_t)(o[0] + imm));
	s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(uintptr_t)(o[1] + imm));
	return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

}  // namespace dma
}  // namespace elf
