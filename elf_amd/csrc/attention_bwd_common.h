// What the attention backward kernels share (see attention_common.h for the layout conventions): their arguments, the walk of a
// workgroup, the layout of the partial dQ, operand tiles in LDS and the stores of dK and dV.
#pragma once
#include "attention_common.h"

namespace elf {
namespace attn {

struct AttnBwdArgs {
	const bf16_t* q;
	const bf16_t* k;
	const bf16_t* v;
	const bf16_t* dO;
	const float* nlse2;  // -lse * log2(e)
	const float* ndelta;  // -rowsum(dO * O)
	bf16_t* dq_part;  // per key tile partial dQ, see part_row0()
	bf16_t* dk;
	bf16_t* dv;
	int64_t ldq, ldk, ldv, lddo, lddk, lddv;
	int B, S, Hq, Hkv;
	float scale;
	// non-null: the q and k heads carry a rotary embedding whose backward (the inverse rotation) is applied to
	// dQ and dK before they are stored; (cos, sin) table [S, D / 2] of rope_table()
	const float2* rope_cs;
	// A pass's walk (query heads of the group x query tiles) shared by h_splits x q_splits workgroups, each of which leaves its
	// dK and dV as fp32 partial sums in dkv_part ([split][dK, dV][token][Hkv * D]) for the reduction kernel; 1 x 1: they are
	// stored as they are.  See split_walk().
	int h_splits, q_splits;
	float* dkv_part;
	int paired;  // causal: a workgroup takes two key tiles one after the other (see attn_bwd_kernel); 0: one
	int longest_first;  // of a causal launch's single key tiles, see locate_walk()
};

// The walk of one workgroup: query heads [h0, h0 + nh) and, per head, query tiles [q_lo, q_hi) of a pass.
struct Walk {
	int pair, b, hk, split, h0, nh;
	__device__ __forceinline__ void tiles(const AttnBwdArgs& a, int qt_first, int nqt, int& q_lo, int& q_hi) const {
		const int qs = split % a.q_splits, len = nqt - qt_first;
		q_lo = qt_first + len * qs / a.q_splits;
		q_hi = qt_first + len * (qs + 1) / a.q_splits;
	}
};
// causal: key tiles taken one by one (not in pairs) have walks of very different lengths; where there are more of them than compute units
// all first (longest) ones are dispatched first, then all second ones, so that a launch of several rounds ends on short ones (a.longest_first;
// one to two rounds 1.13 x as fast, 256-key passes 1.15, 128-key ones of 64 columns, two on a unit, 1.05 from 257 to 512 of them).  Where all
// fit at once a group's tiles stay side by side (us, longest first and so): 1536 tokens, 4 heads of 64 34.6 and 32.6; 10 x 384, one head
// of 128 27.0 and 25.7; 4 x 256, 3 heads of 64 21.0 and 20.1; 309 such shapes 0.5 % faster, between 4 % slower and 6 % faster.
__device__ __forceinline__ Walk locate_walk(const AttnBwdArgs& a, int npair, bool causal) {
	const int ns = a.h_splits * a.q_splits, per_group = npair * ns;
	const int ngroups = (int)(gridDim.x / per_group);
	// all workgroups of a (batch, kv head) group on one XCD (workgroup w runs on XCD w % 8)
	const bool by_xcd = ngroups % 8 == 0;
	const int slot = by_xcd ? blockIdx.x >> 3 : blockIdx.x, groups = by_xcd ? ngroups >> 3 : ngroups;
	int bh, rest;
	if (causal && a.longest_first) {
		const int per_tile = groups * ns, in_tile = slot % per_tile;
		bh = in_tile / ns;
		rest = slot / per_tile * ns + in_tile % ns;
	} else {
		bh = slot / per_group;
		rest = slot % per_group;
	}
	if (by_xcd) bh = (blockIdx.x & 7) + 8 * bh;
	Walk w;
	w.split = rest % ns;
	w.pair = rest / ns;
	w.hk = bh % a.Hkv, w.b = bh / a.Hkv;
	w.nh = a.Hq / a.Hkv / a.h_splits;
	w.h0 = w.hk * (a.Hq / a.Hkv) + (w.split / a.q_splits) * w.nh;
	return w;
}

// dQ partials.  Every 128-key tile contributes a [queries, Hq*D] partial dQ; the partials are written
// with plain stores, each by exactly one workgroup, rounded to bf16 (like the P and dS operands of the
// products they come from), and summed in fp32 in a fixed order by dq_reduce_kernel: no atomics, no
// zero fill, and a result that does not depend on the order in which workgroups run.  (Adding the
// tiles into one fp32 buffer with atomics costs a read-modify-write of a line that is never cache
// resident per 32 lanes: 0.3 T lanes/s chip-wide, 0.68 of 1.81 ms at the Llama-3-8B shape.)
// Layout per batch element: the slices of the key tiles one after the other; with a causal mask
// slice kt only holds the queries q >= 128 kt, so it starts at row kt S - 128 kt (kt - 1) / 2 and
// its row index is q - 128 kt.  (keys: those of a tile, 128 or 256.)
__host__ __device__ __forceinline__ int64_t part_row0(int kt, int S, bool causal, int keys) {
	return causal ? (int64_t)kt * S - keys / 2 * (int64_t)kt * (kt - 1) : (int64_t)kt * S;
}
__host__ __device__ __forceinline__ int64_t part_rows(int S, bool causal, int keys) { return part_row0((S + keys - 1) / keys, S, causal, keys); }

// Tiles fetched straight into LDS (lds_dma.h) are unpadded; the 16-byte chunk index of a row is
// XOR-swizzled with a function of the row chosen so that both access patterns are conflict
// free: row-wise fragment reads (16 consecutive rows, same chunk) and transpose reads (a
// half-wave takes 64 contiguous bytes from each of 4 consecutive rows).
template <int D>
struct BwdTile {
	static constexpr int ROW_BYTES = D * 2;
	static constexpr int CPR = D / 8;             // 16-byte chunks per row
	static constexpr int RPI = 1024 / ROW_BYTES;  // rows per DMA wave instruction
	__device__ static __forceinline__ int swz(int row) {
		// D = 128 (16 chunks per row, a row spans all banks): bits [3:2] from row % 4 put four consecutive
		// rows into four different 64-byte bank groups, bits [1:0] from row / 4 make 16 consecutive rows
		// distinct.  D = 64 (8 chunks, two rows span all banks): the same for row pairs, bit-reversed.
		return D == 128 ? (((row & 3) << 2) | ((row >> 2) & 3)) : ((((row >> 1) & 1) << 2) | (((row >> 2) & 1) << 1) | ((row >> 3) & 1));
	}
	// row-wise operand: rows row0 + lane%32, 8 consecutive columns from 16*ks + 8*(lane/32)
	__device__ static __forceinline__ bf16x8 rows(const unsigned char* t, int row0, int ks, int lane) {
		const int r = row0 + (lane & 31);
		return *reinterpret_cast<const bf16x8*>(t + r * ROW_BYTES + (((2 * ks + (lane >> 5)) ^ swz(r)) << 4));
	}
	// transposed operand: column m0 + lane%32 at the rows {kA..kA+3, kA+second..+3}, kA = k0 + 4*(lane/32)
	// (second = 8: accumulator row order) or kA = k0 + 8*(lane/32) (second = 4: natural order)
	template <bool ACC_ORDER>
	__device__ static __forceinline__ bf16x8 cols(const unsigned char* t, int k0, int m0, int lane) {
		const int j = lane & 15;
		const int kk = k0 + (ACC_ORDER ? 4 : 8) * (lane >> 5) + (j >> 2);
		const int k2 = kk + (ACC_ORDER ? 8 : 4);
		const int c = (m0 + 16 * ((lane & 31) >> 4) + 4 * (j & 3)) >> 3;
		const unsigned char* p0 = t + kk * ROW_BYTES + ((c ^ swz(kk)) << 4) + (j & 1) * 8;
		const unsigned char* p1 = t + k2 * ROW_BYTES + ((c ^ swz(k2)) << 4) + (j & 1) * 8;
		s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(p0));
		s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(p1));
		return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
	}
};

// 4 bytes per lane from a per-lane global address to LDS at lds_byte_addr + lane * 4.
__device__ __forceinline__ void dma4(const void* lane_addr, uint32_t lds_byte_addr) {
	asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off" ::"s"(lds_byte_addr), "v"(lane_addr) : "memory", "m0");
}

// dS^T tile in LDS: [key][q] bf16 with 64-byte rows (32 queries); the 16-byte chunk index is
// XOR-swizzled with (key >> 2) & 3 so that the 8-byte accumulator writes of 32 consecutive keys
// and the transpose reads of 4 consecutive keys both spread over all banks.
__device__ __forceinline__ int ds_t_offset(int key, int q) {  // q a multiple of 4
	return key * 64 + (((q >> 3) ^ ((key >> 2) & 3)) << 4) + ((q >> 2) & 1) * 8;
}
// A operand from the dS^T tile: row q = lane%32, keys k0 + 8*(lane/32) .. +7
__device__ __forceinline__ bf16x8 ds_t_frag(const unsigned char* t, int k0, int lane) {
	const int j = lane & 15;
	const int kk = k0 + 8 * (lane >> 5) + (j >> 2);
	const int q = 16 * ((lane & 31) >> 4) + 4 * (j & 3);
	s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(t + ds_t_offset(kk, q)));
	s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(t + ds_t_offset(kk + 4, q)));
	return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// dK^T, dV^T and dQ^T accumulators of one wave -> memory: register r of tile dt <-> d = dt*32 + (r/4)*8 + 4g + r%4, lane <-> token; p: the
// token's row at the tile's first column.
__device__ __forceinline__ void store_tile(const f32x16& acc, bf16_t* p, float scale, int g) {
#pragma unroll
	for (int r4 = 0; r4 < 4; r4++) {
		bf16x4 o;
#pragma unroll
		for (int u = 0; u < 4; u++) o[u] = (bf16_t)(acc[r4 * 4 + u] * scale);
		*reinterpret_cast<bf16x4*>(p + r4 * 8 + 4 * g) = o;
	}
}
// With a rotary embedding on the heads, the gradient (scaled and rounded to bf16, as a separate RoPE pass over the stored
// gradient would read it) is rotated back first; the partner of column d is d + D/2, same register of tile dt + DT/2.
template <int D>
__device__ __forceinline__ void store_tiles_rotated(const f32x16& acc_lo, const f32x16& acc_hi, bf16_t* p, float scale, int g, const float2* cs) {
#pragma unroll
	for (int r4 = 0; r4 < 4; r4++) {
		const int i = r4 * 8 + 4 * g;
		const f32x4 t0 = *reinterpret_cast<const f32x4*>(cs + i), t1 = *reinterpret_cast<const f32x4*>(cs + i + 2);
		bf16x4 lo4, hi4;
#pragma unroll
		for (int u = 0; u < 4; u++) {
			const float lo = (float)(bf16_t)(acc_lo[r4 * 4 + u] * scale), hi = (float)(bf16_t)(acc_hi[r4 * 4 + u] * scale);
			const float c = (u < 2 ? t0 : t1)[(u & 1) * 2], sn = (u < 2 ? t0 : t1)[(u & 1) * 2 + 1];
			float rl, rh;
			rope_rot(lo, hi, c, -sn, rl, rh);
			lo4[u] = (bf16_t)rl;
			hi4[u] = (bf16_t)rh;
		}
		*reinterpret_cast<bf16x4*>(p + i) = lo4;
		*reinterpret_cast<bf16x4*>(p + i + D / 2) = hi4;
	}
}
template <int D>
__device__ __forceinline__ void store_dk(const f32x16 (&acc)[D / 32], bf16_t* p, float scale, int g, const float2* cs_row) {
	constexpr int DT = D / 32;
	if (cs_row == nullptr) {
#pragma unroll
		for (int dt = 0; dt < DT; dt++) store_tile(acc[dt], p + dt * 32, scale, g);
	} else {
#pragma unroll
		for (int dt = 0; dt < DT / 2; dt++) store_tiles_rotated<D>(acc[dt], acc[dt + DT / 2], p + dt * 32, scale, g, cs_row + dt * 32);
	}
}
template <int D>
__device__ __forceinline__ void store_dv(const f32x16 (&acc)[D / 32], bf16_t* p, int g) {
#pragma unroll
	for (int dt = 0; dt < D / 32; dt++) store_tile(acc[dt], p + dt * 32, 1.f, g);
}
template <int D>
__device__ __forceinline__ void store_dk_dv(const f32x16 (&acc_dk)[D / 32], const f32x16 (&acc_dv)[D / 32], bf16_t* dkp, bf16_t* dvp, float scale, int g,
                                            const float2* cs_row) {
	store_dv<D>(acc_dv, dvp, g);
	store_dk<D>(acc_dk, dkp, scale, g, cs_row);
}

// The same accumulators as fp32 partial sums: dK at p, dV `stride` floats further on.
template <int D>
__device__ __forceinline__ void store_dkv_part(const f32x16 (&acc_dk)[D / 32], const f32x16 (&acc_dv)[D / 32], float* p, int64_t stride, int g) {
#pragma unroll
	for (int dt = 0; dt < D / 32; dt++) {
#pragma unroll
		for (int r4 = 0; r4 < 4; r4++) {
			f32x4 k4, v4;
#pragma unroll
			for (int u = 0; u < 4; u++) k4[u] = acc_dk[dt][r4 * 4 + u], v4[u] = acc_dv[dt][r4 * 4 + u];
			*reinterpret_cast<f32x4*>(p + dt * 32 + r4 * 8 + 4 * g) = k4;
			*reinterpret_cast<f32x4*>(p + stride + dt * 32 + r4 * 8 + 4 * g) = v4;
		}
	}
}

// attention_bwd_wide.hip: passes over 256 keys, heads of 64 columns
int launch_bwd_wide(const AttnBwdArgs& a, bool causal, dim3 grid, hipStream_t stream);
// attention_bwd_one.hip: sequences of 128 tokens, the whole call
int launch_bwd_one(const AttnBwdArgs& a, int D, bool causal, const bf16_t* o, const float* lse, bf16_t* dq, int64_t ldo, int64_t lddq, hipStream_t stream);

}  // namespace attn
}  // namespace elf
