// Attention backward kernels (see attention_common.h for the layout conventions).
#include "attention_bwd_common.h"
#include <type_traits>

namespace elf {
namespace attn {

// ------------------------------------------------------------------------------------------
// ndelta[b,h,s] = -sum_d dO * O and nlse2[b,h,s] = -lse * log2(e).  D/8 lanes share one (token, head)
// row, 16 bytes each, so a wave covers 4 (D = 128) or 8 (D = 64) rows per step.
__global__ __launch_bounds__(256) void attn_delta_kernel(const bf16_t* __restrict__ dO, const bf16_t* __restrict__ O,
                                                         const float* __restrict__ lse, float* __restrict__ ndelta,
                                                         float* __restrict__ nlse2, int64_t ldd, int64_t ldo, int B, int S,
                                                         int Hq, int D) {
	const int lpr = D / 8;  // lanes per row: 8 or 16
	const int rows_per_block = 256 / lpr;
	const int sub = threadIdx.x % lpr;
	const int64_t n = (int64_t)B * S * Hq;
	for (int64_t idx = (int64_t)blockIdx.x * rows_per_block + threadIdx.x / lpr; idx < n; idx += (int64_t)gridDim.x * rows_per_block) {
		const int h = (int)(idx % Hq);
		const int64_t tok = idx / Hq;
		const bf16x8 x = *reinterpret_cast<const bf16x8*>(dO + tok * ldd + h * D + sub * 8);
		const bf16x8 y = *reinterpret_cast<const bf16x8*>(O + tok * ldo + h * D + sub * 8);
		float s = 0.f;
#pragma unroll
		for (int j = 0; j < 8; j++) s += (float)x[j] * (float)y[j];
		for (int o = lpr >> 1; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
		if (sub == 0) {
			const int64_t b = tok / S, sp = tok % S;
			ndelta[(b * Hq + h) * S + sp] = -s;
			nlse2[(b * Hq + h) * S + sp] = -lse[(b * Hq + h) * S + sp] * LOG2E;
		}
	}
}

// One workgroup pass = 128 keys of one (batch, kv head); wave w owns keys [32w, 32w+32) and
// keeps their K / V rows (MFMA B operands) and dK^T / dV^T accumulators in registers while the
// workgroup walks over the 32-query tiles of every query head of the group.  Q and dO tiles
// arrive by direct-to-LDS loads one tile ahead.  Per tile and wave:
//   S = Q K^T, dP = dO V^T  (A operands: LDS rows)      P = exp2(S*sc - lse), dS = P (dP - delta)
//   dV^T += dO^T P, dK^T += Q^T dS  (A operands: LDS transpose reads; B: P / dS from registers)
// dS^T goes to LDS; after the next workgroup barrier each wave multiplies the whole 32x128 dS
// by its slice of K (held in registers as B operands) to get its slice of the dQ tile.  That
// product runs one tile behind, so a tile costs one barrier; the slice goes to this key tile's
// partial dQ buffer (bf16).  The softmax scale of dK and dQ is applied by the epilogue / the
// reduction kernel.  With a causal mask key tile kt meets 1 - kt/nkt of the query tiles: a workgroup
// takes one tile, or (a.paired) the tiles kt and nkt-1-kt one after the other, which is the same work
// for every workgroup: see split_walk().
// Heads of 64 columns come here where passes over 256 keys (attention_bwd_wide.hip) do not pay.
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void attn_bwd_kernel(AttnBwdArgs a) {
	using TL = BwdTile<D>;
	constexpr int BKV = 128, BQ = 32;
	constexpr int NF = D / 16;  // fragments per operand tile
	constexpr int DT = D / 32;
	constexpr int NQ = BKV / 16;  // fragments of the dQ product (all 128 keys); waves 0..DT-1 own one 32-column slice each
	constexpr int K_BYTES = BKV * TL::ROW_BYTES, Q_BYTES = BQ * TL::ROW_BYTES;
	constexpr int STAGE = 2 * Q_BYTES + 256;  // Q tile, dO tile, 32 nlse2 + 32 -delta floats
	constexpr int DS_BYTES = BKV * BQ * 2;
	constexpr int Q_LOADS = 8 / TL::RPI;  // DMA instructions per wave and tile (8 rows per wave)
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
	unsigned char* const sKt = smem_raw;            // K tile, [key][d]
	unsigned char* const sStage = sKt + K_BYTES;    // 2 x {Q [q][d], dO [q][d], nlse2, delta}
	unsigned char* const sdS = sStage + 2 * STAGE;  // 2 x dS^T [key][q]

	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int g = lane >> 5, kl = lane & 31;
	const int nkt = a.S / BKV;
	const int npair = CAUSAL && a.paired ? (nkt + 1) / 2 : nkt;
	const Walk wk = locate_walk(a, npair, CAUSAL);
	const int pair = wk.pair, hk = wk.hk, b = wk.b;
	const int64_t tok0 = (int64_t)b * a.S;
	const int64_t HqD = (int64_t)a.Hq * D;
	const float sc = a.scale * LOG2E;
	const bool dq_wave = DT == 4 || wave < DT;  // head_dim 64: two slices, waves 2 and 3 have no dQ share
	const int dq_dt = wave % DT;
	const int key_l = wave * 32 + kl;                        // this lane's key within the tile
	const int nqt_all = a.S / BQ;
	const int dq_lane = kl * (int)HqD + dq_dt * 32 + 4 * g;  // lane part of a dQ tile address (elements): query kl, first of 4 columns

	// DMA plan for one (Q, dO) tile pair: wave w moves rows [w*8, w*8+8) of each
	uint32_t qoff[Q_LOADS], dooff[Q_LOADS];
#pragma unroll
	for (int i = 0; i < Q_LOADS; i++) {
		const int row = wave * 8 + i * TL::RPI + lane / TL::CPR, slot = lane % TL::CPR;
		qoff[i] = (uint32_t)((row * a.ldq + ((slot ^ TL::swz(row)) << 3)) * 2);
		dooff[i] = (uint32_t)((row * a.lddo + ((slot ^ TL::swz(row)) << 3)) * 2);
	}
	auto zero_ds = [&](unsigned char* t) {
#pragma unroll
		for (int i = 0; i < 4; i++) *reinterpret_cast<u32x2*>(t + ds_t_offset(key_l, 8 * i + 4 * g)) = u32x2{0u, 0u};
	};
	// registers [r_lo, r_hi) of a dQ^T accumulator tile -> the partial buffer.  The dQ product is computed
	// transposed (rows d, columns q) so that a lane holds 4 consecutive columns of one query's row:
	// four 8-byte stores per tile and lane (2-byte stores, one per register, cost 500 cycles more per tile)
	auto dq_out = [&](bf16_t* tile, const f32x16& v, int r_lo, int r_hi) {
		if (!dq_wave) return;
#pragma unroll
		for (int j = 0; j < 4; j++)
			if (4 * j >= r_lo && 4 * j < r_hi) {
				bf16x4 o;
#pragma unroll
				for (int t = 0; t < 4; t++) o[t] = (bf16_t)v[4 * j + t];
				*reinterpret_cast<bf16x4*>(tile + dq_lane + 8 * j) = o;
			}
	};

	const int n_pass = (CAUSAL && a.paired && nkt - 1 - pair != pair) ? 2 : 1;
#pragma unroll 1
	for (int pass = 0; pass < n_pass; pass++) {
		const int kt_idx = pass == 0 ? pair : nkt - 1 - pair;
		const int key0 = kt_idx * BKV;       // first key of the pass
		const int wkey0 = key0 + wave * 32;  // first key of this wave
		if (pass > 0) __syncthreads();       // every wave is done with the LDS of the previous pass

		// K tile -> LDS; this wave moves rows [wave*32, wave*32+32)
		{
			const bf16_t* kb = a.k + (tok0 + key0) * a.ldk + hk * D;
#pragma unroll
			for (int i = 0; i < 32 / TL::RPI; i++) {
				const int row = wave * 32 + i * TL::RPI + lane / TL::CPR, slot = lane % TL::CPR;
				dma16(kb, (uint32_t)((row * a.ldk + ((slot ^ TL::swz(row)) << 3)) * 2),
				      __builtin_amdgcn_readfirstlane(lds_addr(sKt) + (wave * 32 + i * TL::RPI) * TL::ROW_BYTES));
			}
		}
		// own K and V rows as B operands (n = key, 8 consecutive d) in registers
		bf16x8 kf[NF], vf[NF];
		{
			const bf16_t* kp = a.k + (tok0 + wkey0 + kl) * a.ldk + hk * D + 8 * g;
			const bf16_t* vp = a.v + (tok0 + wkey0 + kl) * a.ldv + hk * D + 8 * g;
#pragma unroll
			for (int ks = 0; ks < NF; ks++) {
				kf[ks] = *reinterpret_cast<const bf16x8*>(kp + ks * 16);
				vf[ks] = *reinterpret_cast<const bf16x8*>(vp + ks * 16);
				// the pass-long B operands live in the accumulator half of the register file (the matrix
				// pipe reads them there directly): pinning them at their definition keeps the allocator from
				// copying them into the vector half before every product
				asm volatile("" : "+a"(kf[ks]), "+a"(vf[ks]));
			}
		}
		f32x16 acc_dk[DT], acc_dv[DT];
#pragma unroll
		for (int i = 0; i < DT; i++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc_dk[i][r] = acc_dv[i][r] = 0.f;

		// Walk over (query head in group, query tile); causal: only tiles that reach key0.
		const int qt_first = CAUSAL ? key0 / BQ : 0;
		int q_lo, q_hi;
		wk.tiles(a, qt_first, nqt_all, q_lo, q_hi);
		const int n_iter = wk.nh * (q_hi - q_lo);  // at least one: a pass has four query tiles or more, q_splits is at most four

		// tile whose loads are issued next: running pointers, recomputed when the walk moves to the next head
		int ld_h = wk.h0, ld_qt = q_lo;
		const bf16_t* ld_q;
		const bf16_t* ld_do;
		const float* ld_stat;  // lanes 0..31: nlse2 of the tile's queries, lanes 32..63: -delta
		auto seek = [&]() {
			const int64_t row = tok0 + ld_qt * BQ;
			ld_q = a.q + row * a.ldq + ld_h * D;
			ld_do = a.dO + row * a.lddo + ld_h * D;
			ld_stat = (lane < 32 ? a.nlse2 : a.ndelta) + ((int64_t)b * a.Hq + ld_h) * a.S + ld_qt * BQ + (lane & 31);
		};
		seek();
		const uint32_t lds_stage = lds_addr(sStage) + wave * 8 * TL::ROW_BYTES;
		auto issue = [&](int stage) {
			const uint32_t st = lds_stage + (uint32_t)stage * STAGE;
#pragma unroll
			for (int i = 0; i < Q_LOADS; i++) {
				dma16(ld_q, qoff[i], __builtin_amdgcn_readfirstlane(st + i * TL::RPI * TL::ROW_BYTES));
				dma16(ld_do, dooff[i], __builtin_amdgcn_readfirstlane(st + Q_BYTES + i * TL::RPI * TL::ROW_BYTES));
			}
			if (wave == 0) dma4(ld_stat, __builtin_amdgcn_readfirstlane(st + 2 * Q_BYTES));
			if (++ld_qt == q_hi) {
				ld_qt = q_lo;
				ld_h++;
				seek();
			} else {
				ld_q += BQ * a.ldq;
				ld_do += BQ * a.lddo;
				ld_stat += BQ;
			}
		};

		issue(0);
		zero_ds(sdS + DS_BYTES);  // the "previous tile" of the first iteration
		wait_vmcnt<0>();
		__syncthreads();
		// this wave's slice of K^T as A operands of the dQ^T product (rows d, k = key)
		bf16x8 ktf[NQ];
#pragma unroll
		for (int i = 0; i < NQ; i++) ktf[i] = TL::template cols<false>(sKt, i * 16, dq_dt * 32, lane);

		// position of the current tile; dq_prev_tile = where the dQ tile of iteration it-1 goes
		int cur_h = wk.h0, cur_qt = q_lo;
		// rows of this key tile's slice: first query of the slice = key0 (causal) or 0
		bf16_t* const part = a.dq_part + ((int64_t)b * part_rows(a.S, CAUSAL, BKV) + part_row0(kt_idx, a.S, CAUSAL, BKV) - qt_first * BQ) * HqD;
		bf16_t* dq_prev_tile = part + (int64_t)(q_lo * BQ) * HqD + cur_h * D;

		for (int it = 0; it < n_iter; it++) {
			if (it + 1 < n_iter) issue((it + 1) & 1);
			const unsigned char* sQ = sStage + (it & 1) * STAGE;
			const unsigned char* sdO = sQ + Q_BYTES;
			const float* sLse = reinterpret_cast<const float*>(sdO + Q_BYTES);
			const unsigned char* sdS_prev = sdS + ((it + 1) & 1) * DS_BYTES;
			unsigned char* sdS_cur = sdS + (it & 1) * DS_BYTES;
			const int q0 = cur_qt * BQ;

			bf16x8 bA[NF], bC[NF];
			f32x16 dq, s, dp;
#pragma unroll
			for (int r = 0; r < 16; r++) dq[r] = s[r] = dp[r] = 0.f;
			if constexpr (DT == 4) {
#pragma unroll
				for (int i = 0; i < NF; i++) bC[i] = ds_t_frag(sdS_prev, i * 16, lane);
#pragma unroll
				for (int i = 0; i < NF; i++) bA[i] = TL::rows(sQ, 0, i, lane);
				__builtin_amdgcn_sched_barrier(0);
				// dQ product of the previous tile, interleaved with S of this one
#pragma unroll
				for (int i = 0; i < NF; i++) {
					dq = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ktf[i], bC[i], dq, 0, 0, 0);
					s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bA[i], kf[i], s, 0, 0, 0);
				}
			} else {
#pragma unroll
				for (int i = 0; i < NF; i++) bA[i] = TL::rows(sQ, 0, i, lane);
				if (dq_wave) {
					bf16x8 bD[NQ];
#pragma unroll
					for (int i = 0; i < NQ; i++) bD[i] = ds_t_frag(sdS_prev, i * 16, lane);
#pragma unroll
					for (int i = 0; i < NQ; i++) dq = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ktf[i], bD[i], dq, 0, 0, 0);
				}
#pragma unroll
				for (int i = 0; i < NF; i++) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bA[i], kf[i], s, 0, 0, 0);
			}
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for (int i = 0; i < NF; i++) bC[i] = TL::rows(sdO, 0, i, lane);
			dq_out(dq_prev_tile, dq, 0, 4);
			__builtin_amdgcn_sched_barrier(0);
			// dP = dO V^T on the matrix pipe while the vector pipe turns S into P
#pragma unroll
			for (int i = 0; i < NF; i++) dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bC[i], vf[i], dp, 0, 0, 0);
			// dO^T fragments: rows d, k = queries in accumulator order
#pragma unroll
			for (int i = 0; i < NF; i++) bA[i] = TL::template cols<true>(sdO, (i / DT) * 16, (i % DT) * 32, lane);
			// causal mask: key > query  <=>  row index of the accumulator register < key - q0
			// (never true for a tile that lies wholly after the wave's keys; a wave whose keys lie
			// wholly after the tile gets P = 0 everywhere)
			const int kq = wkey0 + kl - q0 - 4 * g;
			float p[16];
			auto softmax = [&](auto masked) {
#pragma unroll
				for (int r4 = 0; r4 < 4; r4++) {
					const f32x4 l4 = *reinterpret_cast<const f32x4*>(sLse + r4 * 8 + 4 * g);
#pragma unroll
					for (int t = 0; t < 4; t++) {
						float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r4 * 4 + t], sc, l4[t]));
						if (decltype(masked)::value && r4 * 8 + t < kq) pr = 0.f;
						p[r4 * 4 + t] = pr;
					}
				}
			};
			// only the tiles on the diagonal (the wave's last key lies after the tile's first query) need the mask
			if (CAUSAL && wkey0 + 31 > q0) softmax(std::true_type{});
			else softmax(std::false_type{});
			const bf16x8 pf[2] = {pack8(p), pack8(p + 8)};
			dq_out(dq_prev_tile, dq, 4, 8);
			__builtin_amdgcn_sched_barrier(0);
			// dV^T[d][key] += dO^T[d][q] P[q][key] while the vector pipe forms dS = P (dP - delta)
#pragma unroll
			for (int i = 0; i < NF; i++) bC[i] = TL::template cols<true>(sQ, (i / DT) * 16, (i % DT) * 32, lane);
#pragma unroll
			for (int i = 0; i < NF; i++)
				acc_dv[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bA[i], pf[i / DT], acc_dv[i % DT], 0, 0, 0);
			float ds[16];
#pragma unroll
			for (int r4 = 0; r4 < 4; r4++) {
				const f32x4 d4 = *reinterpret_cast<const f32x4*>(sLse + 32 + r4 * 8 + 4 * g);
#pragma unroll
				for (int t = 0; t < 4; t++) ds[r4 * 4 + t] = p[r4 * 4 + t] * (dp[r4 * 4 + t] + d4[t]);
			}
			const bf16x8 dsf[2] = {pack8(ds), pack8(ds + 8)};
			// accumulator rows of register r: q = (r/4)*8 + 4g + r%4 -> four 8-byte groups per lane
#pragma unroll
			for (int u = 0; u < 2; u++) {
				const u32x4 w = __builtin_bit_cast(u32x4, dsf[u]);
				*reinterpret_cast<u32x2*>(sdS_cur + ds_t_offset(key_l, 16 * u + 4 * g)) = u32x2{w[0], w[1]};
				*reinterpret_cast<u32x2*>(sdS_cur + ds_t_offset(key_l, 16 * u + 8 + 4 * g)) = u32x2{w[2], w[3]};
			}
			dq_out(dq_prev_tile, dq, 8, 12);
			__builtin_amdgcn_sched_barrier(0);
			// dK^T[d][key] += Q^T[d][q] dS[q][key]
#pragma unroll
			for (int i = 0; i < NF; i++)
				acc_dk[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bC[i], dsf[i / DT], acc_dk[i % DT], 0, 0, 0);
			dq_out(dq_prev_tile, dq, 12, 16);
			dq_prev_tile = part + (int64_t)q0 * HqD + cur_h * D;
			if (++cur_qt == q_hi) {
				cur_qt = q_lo;
				cur_h++;
			}
			// the next tile's loads were issued before this step's 4 partial stores and vector memory
			// operations complete in order: waiting until 4 are left waits for the loads only
			if (dq_wave) wait_vmcnt<4>();
			else wait_vmcnt<0>();
			__syncthreads();  // the next tile is in LDS, dS^T of this tile is complete, everyone is done with this tile
		}
		// drain: dQ product and partial of the last tile
		{
			const unsigned char* sdS_prev = sdS + ((n_iter + 1) & 1) * DS_BYTES;
			f32x16 dq;
#pragma unroll
			for (int r = 0; r < 16; r++) dq[r] = 0.f;
#pragma unroll
			for (int i = 0; i < NQ; i++)
				dq = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ktf[i], ds_t_frag(sdS_prev, i * 16, lane), dq, 0, 0, 0);
			dq_out(dq_prev_tile, dq, 0, 16);
		}

		// dK^T / dV^T accumulators: register r <-> d = dt*32 + (r/4)*8 + 4g + r%4, lane <-> key
		if (a.dkv_part) {
			store_dkv_part<D>(acc_dk, acc_dv, a.dkv_part + (((int64_t)wk.split * 2 * a.B * a.S + tok0 + wkey0 + kl) * a.Hkv + hk) * D, (int64_t)a.B * a.S * a.Hkv * D, g);
			continue;
		}
		bf16_t* dkp = a.dk + (tok0 + wkey0 + kl) * a.lddk + hk * D;
		bf16_t* dvp = a.dv + (tok0 + wkey0 + kl) * a.lddv + hk * D;
		store_dk_dv<D>(acc_dk, acc_dv, dkp, dvp, a.scale, g, a.rope_cs ? a.rope_cs + (int64_t)(wkey0 + kl) * (D / 2) : nullptr);
	}
}

// The same pass for a wave that has its SIMD to itself (head_dim 128: K / V rows and accumulators fill the
// register file).  Nothing else fills its issue gaps, so the schedule is explicit: Q / dO tiles in a three-stage
// ring fetched two steps ahead, every fragment read issued one product ahead of its use into two buffers
// that alternate roles, and every MFMA pinned between its share of the reads and of the vector work.
// 2690 against 3650 cycles per tile; in the stream (between GEMMs) the call takes 1.04 against 1.13 ms.
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256) void attn_bwd_kernel_lone(AttnBwdArgs a) {
	using TL = BwdTile<D>;
	constexpr int BKV = 128, BQ = 32;
	constexpr int NF = D / 16;  // fragments per operand tile
	constexpr int DT = D / 32;
	constexpr int NQ = BKV / 16;  // fragments of the dQ product (all 128 keys); waves 0..DT-1 own one 32-column slice each
	constexpr int K_BYTES = BKV * TL::ROW_BYTES, Q_BYTES = BQ * TL::ROW_BYTES;
	constexpr int STAGE = 2 * Q_BYTES + 256;  // Q tile, dO tile, 32 nlse2 + 32 -delta floats
	constexpr int NSTAGE = 3;                 // tiles are fetched two steps ahead
	constexpr int DS_BYTES = BKV * BQ * 2;
	constexpr int Q_LOADS = 8 / TL::RPI;  // DMA instructions per wave and tile (8 rows per wave)
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
	unsigned char* const sKt = smem_raw;            // K tile, [key][d]
	unsigned char* const sStage = sKt + K_BYTES;       // NSTAGE x {Q [q][d], dO [q][d], nlse2, delta}
	unsigned char* const sdS = sStage + NSTAGE * STAGE;  // 2 x dS^T [key][q]

	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int g = lane >> 5, kl = lane & 31;
	const int nkt = a.S / BKV;
	const int npair = CAUSAL && a.paired ? (nkt + 1) / 2 : nkt;
	const Walk wk = locate_walk(a, npair, CAUSAL);
	const int pair = wk.pair, hk = wk.hk, b = wk.b;
	const int64_t tok0 = (int64_t)b * a.S;
	const int64_t HqD = (int64_t)a.Hq * D;
	const float sc = a.scale * LOG2E;
	const bool dq_wave = DT == 4 || wave < DT;  // head_dim 64: two slices, waves 2 and 3 have no dQ share
	const int dq_dt = wave % DT;
	const int key_l = wave * 32 + kl;                        // this lane's key within the tile
	const int nqt_all = a.S / BQ;
	const int dq_lane = kl * (int)HqD + dq_dt * 32 + 4 * g;  // lane part of a dQ tile address (elements): query kl, first of 4 columns

	// DMA plan for one (Q, dO) tile pair: wave w moves rows [w*8, w*8+8) of each
	uint32_t qoff[Q_LOADS], dooff[Q_LOADS];
#pragma unroll
	for (int i = 0; i < Q_LOADS; i++) {
		const int row = wave * 8 + i * TL::RPI + lane / TL::CPR, slot = lane % TL::CPR;
		qoff[i] = (uint32_t)((row * a.ldq + ((slot ^ TL::swz(row)) << 3)) * 2);
		dooff[i] = (uint32_t)((row * a.lddo + ((slot ^ TL::swz(row)) << 3)) * 2);
	}
	auto zero_ds = [&](unsigned char* t) {
#pragma unroll
		for (int i = 0; i < 4; i++) *reinterpret_cast<u32x2*>(t + ds_t_offset(key_l, 8 * i + 4 * g)) = u32x2{0u, 0u};
	};
	// registers [r_lo, r_hi) of a dQ accumulator tile -> the partial buffer (issued a few at a time
	// between other work: a long burst backs up the memory pipeline and stalls the wave)
	auto dq_out = [&](bf16_t* tile, const f32x16& v, int r_lo, int r_hi) {
		if (!dq_wave) return;
#pragma unroll
		for (int j = 0; j < 4; j++)
			if (4 * j >= r_lo && 4 * j < r_hi) {
				bf16x4 o;
#pragma unroll
				for (int t = 0; t < 4; t++) o[t] = (bf16_t)v[4 * j + t];
				*reinterpret_cast<bf16x4*>(tile + dq_lane + 8 * j) = o;
			}
	};

	const int n_pass = (CAUSAL && a.paired && nkt - 1 - pair != pair) ? 2 : 1;
#pragma unroll 1
	for (int pass = 0; pass < n_pass; pass++) {
		const int kt_idx = pass == 0 ? pair : nkt - 1 - pair;
		const int key0 = kt_idx * BKV;       // first key of the pass
		const int wkey0 = key0 + wave * 32;  // first key of this wave
		if (pass > 0) __syncthreads();       // every wave is done with the LDS of the previous pass

		// K tile -> LDS; this wave moves rows [wave*32, wave*32+32)
		{
			const bf16_t* kb = a.k + (tok0 + key0) * a.ldk + hk * D;
#pragma unroll
			for (int i = 0; i < 32 / TL::RPI; i++) {
				const int row = wave * 32 + i * TL::RPI + lane / TL::CPR, slot = lane % TL::CPR;
				dma16(kb, (uint32_t)((row * a.ldk + ((slot ^ TL::swz(row)) << 3)) * 2),
				      __builtin_amdgcn_readfirstlane(lds_addr(sKt) + (wave * 32 + i * TL::RPI) * TL::ROW_BYTES));
			}
		}
		// own K and V rows as B operands (n = key, 8 consecutive d) in registers
		bf16x8 kf[NF], vf[NF];
		{
			const bf16_t* kp = a.k + (tok0 + wkey0 + kl) * a.ldk + hk * D + 8 * g;
			const bf16_t* vp = a.v + (tok0 + wkey0 + kl) * a.ldv + hk * D + 8 * g;
#pragma unroll
			for (int ks = 0; ks < NF; ks++) {
				kf[ks] = *reinterpret_cast<const bf16x8*>(kp + ks * 16);
				vf[ks] = *reinterpret_cast<const bf16x8*>(vp + ks * 16);
				asm volatile("" : "+a"(kf[ks]), "+a"(vf[ks]));
			}
		}
		f32x16 acc_dk[DT], acc_dv[DT];
#pragma unroll
		for (int i = 0; i < DT; i++)
#pragma unroll
			for (int r = 0; r < 16; r++) acc_dk[i][r] = acc_dv[i][r] = 0.f;

		// Walk over (query head in group, query tile); causal: only tiles that reach key0.
		const int qt_first = CAUSAL ? key0 / BQ : 0;
		int q_lo, q_hi;
		wk.tiles(a, qt_first, nqt_all, q_lo, q_hi);
		const int n_iter = wk.nh * (q_hi - q_lo);  // at least one: a pass has four query tiles or more, q_splits is at most four

		// tile whose loads are issued next: running pointers, recomputed when the walk moves to the next head
		int ld_h = wk.h0, ld_qt = q_lo;
		const bf16_t* ld_q;
		const bf16_t* ld_do;
		const float* ld_stat;  // lanes 0..31: nlse2 of the tile's queries, lanes 32..63: -delta
		auto seek = [&]() {
			const int64_t row = tok0 + ld_qt * BQ;
			ld_q = a.q + row * a.ldq + ld_h * D;
			ld_do = a.dO + row * a.lddo + ld_h * D;
			ld_stat = (lane < 32 ? a.nlse2 : a.ndelta) + ((int64_t)b * a.Hq + ld_h) * a.S + ld_qt * BQ + (lane & 31);
		};
		seek();
		const uint32_t lds_stage = lds_addr(sStage) + wave * 8 * TL::ROW_BYTES;
		auto issue = [&](int stage) {
			const uint32_t st = lds_stage + (uint32_t)stage * STAGE;
#pragma unroll
			for (int i = 0; i < Q_LOADS; i++) {
				dma16(ld_q, qoff[i], __builtin_amdgcn_readfirstlane(st + i * TL::RPI * TL::ROW_BYTES));
				dma16(ld_do, dooff[i], __builtin_amdgcn_readfirstlane(st + Q_BYTES + i * TL::RPI * TL::ROW_BYTES));
			}
			if (wave == 0) dma4(ld_stat, __builtin_amdgcn_readfirstlane(st + 2 * Q_BYTES));
			if (++ld_qt == q_hi) {
				ld_qt = q_lo;
				ld_h++;
				seek();
			} else {
				ld_q += BQ * a.ldq;
				ld_do += BQ * a.lddo;
				ld_stat += BQ;
			}
		};

		issue(0);
		if (n_iter > 1) issue(1);
		zero_ds(sdS + DS_BYTES);  // the "previous tile" of the first iteration
		wait_vmcnt<0>();
		__syncthreads();
		// this wave's slice of K as B operands of the dQ product (n = d column, k = key)
		bf16x8 ktf[NQ];
#pragma unroll
		for (int i = 0; i < NQ; i++) ktf[i] = TL::template cols<false>(sKt, i * 16, dq_dt * 32, lane);

		// position of the current tile; dq_prev_tile = where the dQ tile of iteration it-1 goes
		int cur_h = wk.h0, cur_qt = q_lo;
		// rows of this key tile's slice: first query of the slice = key0 (causal) or 0
		bf16_t* const part = a.dq_part + ((int64_t)b * part_rows(a.S, CAUSAL, BKV) + part_row0(kt_idx, a.S, CAUSAL, BKV) - qt_first * BQ) * HqD;
		bf16_t* dq_prev_tile = part + (int64_t)(q_lo * BQ) * HqD + cur_h * D;

		// One step = one (head, 32-query tile).  Two fragment buffers alternate roles so that every LDS
		// read is issued one product ahead of the MFMAs that consume it (one wave per SIMD: nothing else
		// hides the latency): X enters holding the Q rows of this tile, read during the previous step
		// (the tile has been in LDS since the barrier before that step), and leaves free; Y leaves
		// holding the Q rows of the next tile, so the caller swaps the two for the next step.
		//   Y <- dS^T(prev)     | S  = X(Q) K^T
		//   X <- dO rows        | dQ(prev) = Y K            softmax on the vector pipe
		//   Y <- dO^T           | dP = X(dO) V^T
		//   X <- Q^T            | dV^T += Y(dO^T) P         dS on the vector pipe, dS^T -> LDS
		//   Y <- Q rows (next)  | dK^T += X(Q^T) dS
		int stage = 0;  // it % NSTAGE
		auto step = [&](bf16x8(&X)[NQ], bf16x8(&Y)[NQ], int it) {
			const int load_stage = stage == 0 ? 2 : stage - 1;  // (it + 2) % 3
			const unsigned char* sQ = sStage + stage * STAGE;
			const unsigned char* sdO = sQ + Q_BYTES;
			const float* sLse = reinterpret_cast<const float*>(sdO + Q_BYTES);
			stage = stage == NSTAGE - 1 ? 0 : stage + 1;
			const unsigned char* sQ_next = sStage + stage * STAGE;
			const unsigned char* sdS_prev = sdS + ((it + 1) & 1) * DS_BYTES;
			unsigned char* sdS_cur = sdS + (it & 1) * DS_BYTES;
			const int q0 = cur_qt * BQ;

			f32x16 dq, s, dp;
#pragma unroll
			for (int r = 0; r < 16; r++) dq[r] = s[r] = dp[r] = 0.f;
			// A single wave per SIMD issues in order, so matrix and vector work only overlap where the
			// program interleaves them: every product below is a loop of "one MFMA + its share of the
			// LDS reads and vector work that ride along", pinned by scheduling barriers.
			// causal mask: key > query  <=>  row index of the accumulator register < key - q0
			// (never true for a tile that lies wholly after the wave's keys; a wave whose keys lie
			// wholly after the tile gets P = 0 everywhere)
			const int kq = wkey0 + kl - q0 - 4 * g;
			f32x4 l4[4];
			// S = Q K^T, with the dS^T fragments of the previous tile on their way; the loads of the tile after
			// next and the reads of this tile's statistics go between the MFMAs too
#pragma unroll
			for (int i = 0; i < NF; i++) {
				if (dq_wave) {
#pragma unroll
					for (int j = i * (NQ / NF); j < (i + 1) * (NQ / NF); j++) Y[j] = ds_t_frag(sdS_prev, j * 16, lane);
				}
				s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(X[i], kf[i], s, 0, 0, 0);
				if (i == 0 && it + 2 < n_iter) issue(load_stage);
				if (i == NF / 2) {
#pragma unroll
					for (int r4 = 0; r4 < 4; r4++) l4[r4] = *reinterpret_cast<const f32x4*>(sLse + r4 * 8 + 4 * g);
				}
				__builtin_amdgcn_sched_barrier(0);
			}
			// dQ of the previous tile = dS K, with the dO rows on their way and P = exp2(S sc - lse) on the vector pipe
			float p[16];
			auto dq_and_softmax = [&](auto masked) {
#pragma unroll
				for (int i = 0; i < NQ; i++) {
					if (i < NF) X[i] = TL::rows(sdO, 0, i, lane);
					if (dq_wave) dq = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ktf[i], Y[i], dq, 0, 0, 0);
#pragma unroll
					for (int r = i * (16 / NQ); r < (i + 1) * (16 / NQ); r++) {
						float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], sc, l4[r >> 2][r & 3]));
						if (decltype(masked)::value && (r >> 2) * 8 + (r & 3) < kq) pr = 0.f;
						p[r] = pr;
					}
					__builtin_amdgcn_sched_barrier(0);
				}
			};
			// only the tiles on the diagonal (the wave's last key lies after the tile's first query) need the mask
			if (CAUSAL && wkey0 + 31 > q0) dq_and_softmax(std::true_type{});
			else dq_and_softmax(std::false_type{});
			const bf16x8 pf[2] = {pack8(p), pack8(p + 8)};
			f32x4 d4[4];
#pragma unroll
			for (int r4 = 0; r4 < 4; r4++) d4[r4] = *reinterpret_cast<const f32x4*>(sLse + 32 + r4 * 8 + 4 * g);
			// dP = dO V^T, with the dO^T fragments (rows d, k = queries in accumulator order) on their way and the
			// previous tile's dQ partial going out
#pragma unroll
			for (int i = 0; i < NF; i++) {
				Y[i] = TL::template cols<true>(sdO, (i / DT) * 16, (i % DT) * 32, lane);
				dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(X[i], vf[i], dp, 0, 0, 0);
				if ((i * 4) % NF == 0) dq_out(dq_prev_tile, dq, (i * 4 / NF) * 4, (i * 4 / NF) * 4 + 4);
				__builtin_amdgcn_sched_barrier(0);
			}
			// dV^T[d][key] += dO^T[d][q] P[q][key], with the Q^T fragments on their way and dS = P (dP - delta) on
			// the vector pipe
			// (dS in the first half of the slots, its packing and the dS^T writes in the next two)
			float ds[16];
			bf16x8 dsf[2];
#pragma unroll
			for (int i = 0; i < NF; i++) {
				X[i] = TL::template cols<true>(sQ, (i / DT) * 16, (i % DT) * 32, lane);
				acc_dv[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(Y[i], pf[i / DT], acc_dv[i % DT], 0, 0, 0);
				if (i < NF / 2) {
#pragma unroll
					for (int r = i * (32 / NF); r < (i + 1) * (32 / NF); r++) ds[r] = p[r] * (dp[r] + d4[r >> 2][r & 3]);
				} else if (i < NF / 2 + 2) {
					// accumulator rows of register r: q = (r/4)*8 + 4g + r%4 -> four 8-byte groups per lane
					const int u = i - NF / 2;
					dsf[u] = pack8(ds + 8 * u);
					const u32x4 w = __builtin_bit_cast(u32x4, dsf[u]);
					*reinterpret_cast<u32x2*>(sdS_cur + ds_t_offset(key_l, 16 * u + 4 * g)) = u32x2{w[0], w[1]};
					*reinterpret_cast<u32x2*>(sdS_cur + ds_t_offset(key_l, 16 * u + 8 + 4 * g)) = u32x2{w[2], w[3]};
				}
				__builtin_amdgcn_sched_barrier(0);
			}
			// dK^T[d][key] += Q^T[d][q] dS[q][key], with the Q rows of the next tile on their way (past the last
			// tile: a stale stage, values unused)
#pragma unroll
			for (int i = 0; i < NF; i++) {
				Y[i] = TL::rows(sQ_next, 0, i, lane);
				acc_dk[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(X[i], dsf[i / DT], acc_dk[i % DT], 0, 0, 0);
				__builtin_amdgcn_sched_barrier(0);
			}
			dq_prev_tile = part + (int64_t)q0 * HqD + cur_h * D;
			if (++cur_qt == q_hi) {
				cur_qt = q_lo;
				cur_h++;
			}
			// the loads of the tile after next were issued before this step's 4 partial stores and vector
			// memory operations complete in order: waiting until 4 are left waits for the loads only
			if (dq_wave) wait_counters<4, 0>();
			else wait_counters<0, 0>();
			__syncthreads();  // the tile after next is in LDS, dS^T of this tile is complete, everyone is done with this tile
		};

		bf16x8 fragA[NQ], fragB[NQ];
#pragma unroll
		for (int i = 0; i < NF; i++) fragA[i] = TL::rows(sStage, 0, i, lane);
		for (int it = 0; it < n_iter; it += 2) {
			step(fragA, fragB, it);
			if (it + 1 < n_iter) step(fragB, fragA, it + 1);
		}
		// drain: dQ product and partial of the last tile
		{
			const unsigned char* sdS_prev = sdS + ((n_iter + 1) & 1) * DS_BYTES;
			f32x16 dq;
#pragma unroll
			for (int r = 0; r < 16; r++) dq[r] = 0.f;
#pragma unroll
			for (int i = 0; i < NQ; i++)
				dq = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ktf[i], ds_t_frag(sdS_prev, i * 16, lane), dq, 0, 0, 0);
			dq_out(dq_prev_tile, dq, 0, 16);
		}

		// dK^T / dV^T accumulators: register r <-> d = dt*32 + (r/4)*8 + 4g + r%4, lane <-> key
		if (a.dkv_part) {
			store_dkv_part<D>(acc_dk, acc_dv, a.dkv_part + (((int64_t)wk.split * 2 * a.B * a.S + tok0 + wkey0 + kl) * a.Hkv + hk) * D, (int64_t)a.B * a.S * a.Hkv * D, g);
			continue;
		}
		bf16_t* dkp = a.dk + (tok0 + wkey0 + kl) * a.lddk + hk * D;
		bf16_t* dvp = a.dv + (tok0 + wkey0 + kl) * a.lddv + hk * D;
		store_dk_dv<D>(acc_dk, acc_dv, dkp, dvp, a.scale, g, a.rope_cs ? a.rope_cs + (int64_t)(wkey0 + kl) * (D / 2) : nullptr);
	}
}

// dq[b, q, :] (bf16, row stride ld) = scale * sum over the key tiles that meet q of their partial rows,
// added in fp32 in ascending tile order.  A thread takes 8 columns of a head's first half and the 8 columns
// half a head further on; with a rotary embedding on the q heads (cs non-null) these are the pairs of the
// rotation, which is undone on the scaled, bf16-rounded sums before they are stored (what a separate RoPE
// pass over the stored gradient would compute).
//
// dkv.splits > 1: the launch's last dkv.blocks workgroups add the fp32 partial sums of dK and dV in ascending split order,
// 8 + 8 columns per thread, scale (dK), round, undo the rotation (dK) and store them.
struct DkvReduce {
	const float* part;
	bf16_t *dk, *dv;
	int64_t lddk, lddv;
	int splits, Hkv, blocks;
};
__global__ __launch_bounds__(256) void dq_reduce_kernel(const bf16_t* __restrict__ part, bf16_t* __restrict__ dq, int B, int S, int cols,
                                                        int64_t ld, float scale, int causal, int keys, int D, const float2* __restrict__ cs, DkvReduce dkv) {
	const int dq_blocks = (int)gridDim.x - dkv.blocks;
	if ((int)blockIdx.x >= dq_blocks) {
		const int half = D / 2, cph = half / 8, ppr = dkv.Hkv * cph;  // chunk pairs per row
		const int64_t n = (int64_t)B * S * ppr, stride = (int64_t)B * S * dkv.Hkv * D;
		for (int64_t i = ((int64_t)blockIdx.x - dq_blocks) * 256 + threadIdx.x; i < 2 * n; i += (int64_t)dkv.blocks * 256) {
			const bool is_v = i >= n;
			const int64_t k = is_v ? i - n : i, row = k / ppr;
			const int pr = (int)(k - row * ppr), c = (pr / cph) * D + (pr % cph) * 8;
			const float* p = dkv.part + (is_v ? stride : 0) + row * dkv.Hkv * D + c;
			f32x4 s[4] = {};
			for (int t = 0; t < dkv.splits; t++, p += 2 * stride) {
#pragma unroll
				for (int u = 0; u < 4; u++) s[u] += __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p + (u >> 1) * half + (u & 1) * 4));
			}
			const float f = is_v ? 1.f : scale;
			bf16x8 lo, hi;
#pragma unroll
			for (int t = 0; t < 8; t++) {
				lo[t] = (bf16_t)(s[t >> 2][t & 3] * f);
				hi[t] = (bf16_t)(s[2 + (t >> 2)][t & 3] * f);
			}
			if (cs && !is_v) {
				const float2* tab = cs + (row % S) * half + (pr % cph) * 8;
#pragma unroll
				for (int t = 0; t < 8; t++) {
					float rl, rh;
					rope_rot((float)lo[t], (float)hi[t], tab[t].x, -tab[t].y, rl, rh);
					lo[t] = (bf16_t)rl;
					hi[t] = (bf16_t)rh;
				}
			}
			bf16_t* out = (is_v ? dkv.dv + row * dkv.lddv : dkv.dk + row * dkv.lddk) + c;
			*reinterpret_cast<bf16x8*>(out) = lo;
			*reinterpret_cast<bf16x8*>(out + half) = hi;
		}
		return;
	}
	const int half = D / 2, cph = half / 8;  // 8-column chunks per half head
	const int ppr = cols / 16;               // chunk pairs per row
	const int64_t n = (int64_t)B * S * ppr;
	const int nkt = (S + keys - 1) / keys;
	const int64_t rows_b = part_rows(S, causal, keys);
	for (int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; j < n; j += (int64_t)dq_blocks * blockDim.x) {
		// last rows first: under a causal mask they sum the most partials, and the launch then ends on the short ones
		const int64_t i = n - 1 - j;
		const int64_t row = i / ppr;
		const int pr = (int)(i - row * ppr);
		const int c = (pr / cph) * D + (pr % cph) * 8;
		const int b = (int)(row / S), q = (int)(row - (int64_t)b * S);
		const int ns = causal ? q / keys + 1 : nkt;
		float lo[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, hi[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
		const bf16_t* pb = part + (int64_t)b * rows_b * cols + c;
#pragma unroll 8
		for (int kt = 0; kt < ns; kt++) {
			const bf16_t* pr_row = pb + (part_row0(kt, S, causal, keys) + q - (causal ? keys * kt : 0)) * cols;
			// read once: no point in keeping the partials in the caches
			const bf16x8 v = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(pr_row)), w = __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(pr_row + half));
#pragma unroll
			for (int t = 0; t < 8; t++) {
				lo[t] += (float)v[t];
				hi[t] += (float)w[t];
			}
		}
		bf16x8 olo, ohi;
#pragma unroll
		for (int t = 0; t < 8; t++) {
			olo[t] = (bf16_t)(lo[t] * scale);
			ohi[t] = (bf16_t)(hi[t] * scale);
		}
		if (cs) {
			const float2* tab = cs + (int64_t)q * half + (pr % cph) * 8;
#pragma unroll
			for (int t = 0; t < 8; t++) {
				const float2 t2 = tab[t];
				float rl, rh;
				rope_rot((float)olo[t], (float)ohi[t], t2.x, -t2.y, rl, rh);
				olo[t] = (bf16_t)rl;
				ohi[t] = (bf16_t)rh;
			}
		}
		*reinterpret_cast<bf16x8*>(dq + row * ld + c) = olo;
		*reinterpret_cast<bf16x8*>(dq + row * ld + c + half) = ohi;
	}
}

template <int D, bool CAUSAL>
int launch_bwd(const AttnBwdArgs& a, dim3 grid, hipStream_t stream) {
	// K tile + the Q / dO ring (two stages, three for the lone-wave schedule) + two dS^T tiles
	constexpr bool LONE = D == 128;
	constexpr int smem = 128 * D * 2 + (LONE ? 3 : 2) * (2 * 32 * D * 2 + 256) + 2 * 128 * 32 * 2;
	auto kern = LONE ? attn_bwd_kernel_lone<D, CAUSAL> : attn_bwd_kernel<D, CAUSAL>;
	static bool attr_set = false;
	if (!attr_set) {
		ELF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
		attr_set = true;
	}
	ELF_LAUNCH(kern, grid, dim3(256), smem, stream, a);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

}  // namespace attn

using namespace attn;

// How the walks of a launch are shared out.  A workgroup's walk over the query heads of its group and their query tiles is
// serial (one 32-query tile per step), and B * Hkv * (key tiles) walks leave the chip idle where there are few of them: then the
// heads of a group and, after those, the query tiles are split, as long as the estimate gets smaller.  A split adds fp32 partial
// sums of dK and dV to write and to read again.  Causal: a workgroup takes one key tile (the long walks are dispatched first, see
// locate_walk()) or a light and a heavy one, where these make whole rounds.
struct Splits {
	int h = 1, q = 1;
	bool paired = true;
	bool wide = false;  // passes over 256 keys (attention_bwd_wide.hip)
};
static int64_t dkv_part_bytes(const Splits& sp, int B, int S, int Hkv, int D) { return sp.h * sp.q > 1 ? (int64_t)sp.h * sp.q * 2 * B * S * Hkv * D * 4 : 0; }

// Heads of 64 columns, short sequences in a launch that does not fill the chip: workgroups of 128 keys, two on a compute unit.
// Constants in microseconds as measured.  Causal with one key tile (128 tokens): a walk has four steps a head, what a step and a
// split cost beside the fixed part shows.  Constants of its own, fitted to every sharing of 250 such shapes (the one that is picked
// takes 0.2 % longer than the best on average, 7 % at most; with those of longer walks 1.8 and 16 %).  (Where one_kernel_pays() nothing is
// shared; the workspace query, which does not see strides and addresses, asks for the room that calls need whose rows or V stay out of it.)  The whole call in
// three kernels, whole -> as shared now (us): 2 x 128 tokens, 4 heads of 64 18.9 -> 16.7; 3 x 128, 48 / 16 heads of 128 34.8 -> 31.2; 7 x 128, 36 / 12 heads
// of 128 stay whole: 37.8, three ways 40.6.  Heads of 64, 256 to 1280 tokens: what is picked takes 1.2 and (causal) 1.5 % longer than the best
// sharing of 128-key passes over 75 and 79 shapes, 12 and 17 % at most.
static Splits split_short(int B, int S, int Hq, int Hkv, int D, bool causal, int64_t room, float* estimate = nullptr) {
	const int nkt = S / 128, G = Hq / Hkv;
	const bool one = causal && nkt == 1;
	const float slots = D == 128 ? 256.f : 512.f, step = one ? 1.6f : D == 128 ? 1.2f : 1.1f, fixed = 8.f;
	// a split: what it adds by itself, per split, and the partial sums at so many bytes a us; it has to be that much better than less sharing
	const float split = one ? 0.f : 2.f, per_split = one ? 0.4f : 0.f, rate = one ? 4e6f : 5e6f, margin = one ? 1.f : 0.95f;
	Splits best;
	float best_us = 1e30f;
	if (estimate) *estimate = best_us;
	if ((int64_t)B * S * Hq >= 1 << 18) return best;  // these fill the chip
	for (int paired = 1; paired >= (causal && nkt > 1 ? 0 : 1); paired--) {
		if (!paired) best_us += fixed;  // that of a pair's second tile, which all sharings of pairs have alike
		const bool two = causal && paired && nkt > 1;  // key tiles one after the other
		const int64_t walks = (int64_t)B * Hkv * (two ? (nkt + 1) / 2 : nkt);
		const int tiles = two ? (nkt + 1) * 4 : nkt * 4;  // query tiles of the longest walk and head (a pair of key tiles has nkt + 1 of four)
		for (int h = 1; h <= G; h++) {
			if (G % h) continue;
			for (int q = 1; q <= 4; q *= 2) {
				if (q > 1 && h < G) continue;
				const int ns = h * q;
				if (dkv_part_bytes(Splits{h, q}, B, S, Hkv, D) > room) continue;
				const float rounds = ceilf((float)(walks * ns) / slots);
				if (!paired && rounds > 1.f) continue;
				const float us = rounds * (fixed + (float)(G / h) * ((tiles + q - 1) / q) * step) + (ns > 1 ? split + ns * per_split + (float)ns * B * S * Hkv * D * 16 / rate : 0.f);
				if (us < best_us * (ns > 1 ? margin : 1.f)) best_us = us, best = Splits{h, q, paired != 0};
			}
		}
	}
	if (estimate) *estimate = best_us;
	return best;
}

// 128 tokens: one kernel for the whole call (attention_bwd_one.hip) or -delta, walks and sums in three.  A workgroup of the one kernel has a compute
// unit to itself and takes the query heads of its group in turn (4.3 us each for heads of 64, 7.3 of 128; 6 and 7 us besides), the walks
// are shared.  Whole call, three kernels -> one, on operands past the caches (us, causal / not; on operands in them both take 4 to 15 % less):
//   one head of 64 a group: 16 groups 18.3 -> 11.0 / 16.6 -> 11.3, 240 28.1 -> 16.6 / 23.7 -> 17.0, 272 34.6 -> 27.8 / 28.6 and 28.4, 800 68.4 -> 55.5 / 56.3 and 56.9
//   one of 128: 16 21.2 -> 16.2 / 21.2 -> 17.5, 240 34.4 -> 26.1 / 33.3 -> 28.5, 800 104.4 -> 87.6 / 100.5 -> 95.9
//   two of 128: 256 48.2 -> 38.6 / 47.2 -> 42.2, 512 85.4 -> 71.4 / 83.4 and 78.3; three: 256 58.6 -> 50.6 / 57.2 and 55.7, 264 83.6 -> 82.6 / 81.8 and 91.7
//   four of 64: 64 31.2 -> 29.3 / 28.5 and 29.9, 96 37.7 -> 29.8 / 31.4 -> 30.7, 320 69.0 -> 61.1 / 60.8 and 62.7
//   four of 128: 96 49.9 -> 49.1 / 48.5 and 53.1, 256 71.6 -> 63.3 / 70.2 and 68.8, 264 100.3 and 104.1, 288 101.8 and 105.9, 352 108.7 -> 107.6 / 105.4 and 117.8
//   eight of 64: 112 58.5 -> 52.8 / 52.1 and 53.6, 224 85.2 -> 57.7 / 76.6 -> 58.8, 252 90.3 -> 57.9 / 80.9 -> 59.2
//   eight of 128: 128 77.4 and 88.5 / 75.7 and 96.8, 224 105.0 -> 101.4 / 104.1 and 109.7, 252 112.8 -> 103.5 / 111.0 and 113.4, 272 161.6 and 180.9
//
// It addresses all 128 rows of Q, dO and (heads of 128) V with 32-bit byte offsets, where the three kernels take 32 rows of Q and dO and
// read V through 64-bit pointers: rows that far apart stay with those.  So do V's of 128 columns a head that are not 16-byte aligned: the one
// kernel brings them into LDS as it does Q, K and dO.  (128 rows of K are what either needs.)
static bool one_kernel_pays(int B, int S, int Hq, int Hkv, int D, bool causal) {
	const int64_t groups = (int64_t)B * Hkv, G = Hq / Hkv;
	if (S != 128 || G > 8 || groups < (causal && D == 64 ? 16 : 32) * (G - 1)) return false;
	if (causal) return groups <= 256 || G < 4 || (G == 4 && (D == 64 || groups >= 320));
	return D == 64 ? groups <= 256 : G == 1 || (G == 2 && groups <= 256);
}

// room: bytes there are for the partial sums.
//
// One workgroup on a compute unit (heads of 128 columns, and of 64 on passes over 256 keys).  The longest walk, or the average filling of the
// chip and half a walk's fixed part where there are several rounds; constants in microseconds fitted to every sharing of 189 shapes of heads of 128 and
// 232 of 64 from 512 tokens up: what is picked takes 0.1 and 0.5 % longer than the best.  Against pairs of key tiles in any case but where all single
// tiles fit the chip at once, and the 128-key kernel for heads of 64, these shapes take 0.96 and 0.80 of the time.  The whole call,
// before -> after (us): 8 x 1408 tokens, 6 / 2 heads of 128 161 -> 140 (single tiles, heads split 3 ways); 3 x 896, 32 / 8 heads of 128 134 -> 118;
// 4096 tokens, 64 / 8 heads of 128 1424 -> 1012 (128 whole pairs before, shared 2 ways now); 8 x 1024, 12 heads of 64 101 -> 65, not causal
// 130 -> 103; 8192 tokens, 16 heads of 64 559 -> 360.  Single tiles of 128 keys, a few more than fit: the last ones follow the shortest walks, which
// short sequences feel (2.2 walks of the last key tile; of 436 shapes of 256 to 4096 tokens 3 instead of 9 take 3 % longer than the
// sharing before these constants; 11 x 256, 12 / 2 heads of 128 shared 6 ways, 264 workgroups, 58, 3 ways 50; 2 x 384, 44 / 22 heads 61
// shared 2 ways, whole 55).  Pairs that make whole rounds stay: 4 x 4096, 32 / 8 heads of 128 2020, single tiles 2053.
static Splits split_walk(int B, int S, int Hq, int Hkv, int D, bool causal, int64_t room) {
	const int G = Hq / Hkv;
	// Heads of 64 columns: a pass of 256 keys has twice the fixed part of one of 128.  Short sequences take it where there is work for the
	// chip (heads x key tiles of 128), below 512 tokens if the passes fit at once or the 128-key ones do not either, long ones always (us, 128
	// and 256 keys).  Causal: 3 x 384 tokens, 31 heads 40 and 33, 512, 7 heads 22 and 23, 2 x 512, 6 / 1 heads 33 and 30.  Not: 3 x 256,
	// 16 heads 22 and 23, 5 x 384, 26 heads 42 and 57, 3 x 512, 8 heads 30 and 33, 640, 24 / 8 heads 33.6 and 35.9, 30 / 10 39.7 and 34.1, 1024,
	// 2 heads 23.4 and 25.6, 2 x 1024, 4 / 1 heads 31.9 and 33.7, 5 x 896, 2 heads 33.7 and 30.5, 1280, 4 / 1 heads 33.3 and 34.0, 1536, 4 / 2 34.3 either
	// way, 5 x 1536, 2 heads 48.7 and 40.1.
	const int64_t work = (int64_t)B * Hq * (S / 128), tiles128 = (int64_t)B * Hkv * (S / 128), tiles256 = (int64_t)B * Hkv * ((S + 255) / 256);
	const bool worth = causal ? S >= 896 || (S >= 512 && work >= 48) : S >= 1408 || (S >= 896 && work >= 70) || (S >= 512 && work >= 150);
	const bool wide = D == 64 && S >= 256 && (worth || (work >= 256 && (tiles256 <= 256 || tiles128 > 512)));
	if (S < 256 || (D == 64 && !wide)) return split_short(B, S, Hq, Hkv, D, causal, room);
	const int keys = wide ? 256 : 128, n = (S + keys - 1) / keys, tile = keys / 32, Q = S / 32;  // key tiles; query tiles of a key tile, of a sequence
	const float slots = 256.f, step = wide ? 1.f : 1.05f, fixed = wide ? 4.f : 9.f;
	const float split = wide ? 0.4f : 1.4f, per_split = wide ? 0.3f : 0.35f, rate = wide ? 4.8e6f : 8.5e6f, margin = 0.96f;
	Splits best;
	float best_us = 1e30f;
	for (int paired = 1; paired >= (causal && n > 1 ? 0 : 1); paired--) {
		for (int h = 1; h <= G; h++) {
			if (G % h) continue;
			for (int q = 1; q <= 4; q *= 2) {
				if (q > 1 && h < G) continue;
				const int ns = h * q;
				if (dkv_part_bytes(Splits{h, q}, B, S, Hkv, D) > room) continue;
				const float walks = (float)B * Hkv * ns, per = (float)(G / h) / q * step;
				float us;
				if (causal && paired && n > 1) us = ceilf(walks * ((n + 1) / 2) / slots) * (2.f * fixed + per * (2 * Q - tile * (n - 1)));
				else if (!causal || n == 1) us = ceilf(walks * n / slots) * (fixed + per * Q);
				else if (walks * n <= slots) us = fixed + per * Q;
				else us = fmaxf(fmaxf(fixed + per * Q, (wide ? 0.f : 2.2f) * (fixed + per * tile)), walks * (n * fixed + per * ((float)n * Q - tile * 0.5f * n * (n - 1))) / slots + 0.5f * fixed);
				if (ns > 1) us = (us + split + ns * per_split + (float)ns * B * S * Hkv * D * 16 / rate) / margin;
				// partial sums of short walks in a launch of several rounds take a little more than that: of 80 shapes that this decides 30 were
				// slower by more than 3 % than the sharing before these constants, none is now (us, without and with: 6 x 512, 16 / 2 heads of
				// 128 83.3 and 76.2, 2 x 512, 48 / 12 77.6 and 74.4; 13 x 640, 2 / 1 45.6 and 48.2)
				if (causal && !paired && !wide && ns > 1 && n <= 6 && walks * n > slots) us *= 1.05f;
				if (us < best_us) best_us = us, best = Splits{h, q, paired != 0, wide};
			}
		}
	}
	// Without a mask all walks are alike: 128-key tiles, two on a compute unit, that fit at once against 256-key ones, the last one perhaps half
	// empty, whose second round is.  The two estimates are of kernels of their own, 1.38 is where both took the same time (us, 128 and 256 keys:
	// 3 x 896, 24 heads 75.8 and 93.0, 11 x 1152, 5 heads 89.3 and 107, 6 x 640, 17 heads 62.6 and 74.9, 4 x 896, 68 / 17 245 and 264;
	// below it 1 x 1152, 26 / 13 heads 59.4 and 58.4).  384 tokens, of whose three tiles of 128 the two of 256 keys leave a quarter empty, from 1.1
	// on: 11 x 384, 25 heads 80.5 and 89.6, 9 x 384, 15 / 5 heads 48.3 and 54.2; 6 x 384, 48 / 12 heads, 1.09, 80.0 and 79.8.  From 2048 tokens up the longer pass makes up for the round: 12 x 2688, 6 / 2 heads 530 and 488.
	if (wide && !causal && S < 2048) {
		float short_us;
		const Splits sp = split_short(B, S, Hq, Hkv, D, causal, room, &short_us);
		if (short_us * (S < 512 ? 1.1f : 1.38f) < best_us) return sp;
	}
	return best;
}

// bf16 dQ partials of every key tile + delta + scaled log-sum-exp: what a backward whose walks stay whole needs.  It grows with
// each of its arguments, so a buffer for the largest of a caller's shapes serves the smaller ones.
int64_t attn_bwd_workspace_bytes(int B, int S, int Hq, int D, int causal) {
	return (int64_t)B * part_rows(S, causal != 0, 128) * Hq * D * 2 + 2 * (int64_t)B * S * Hq * 4;
}

// With the partial sums of the walks this shape shares: 2 x 2048 tokens, 16 / 4 heads of 128 143 + 67 MB; 2 x 4096, 32 / 8 heads
// 1109 MB, whole.  Not monotonic (a shape that shares needs more than the next larger one that does not).
int64_t attn_bwd_shared_workspace_bytes(int B, int S, int Hq, int Hkv, int D, int causal) {
	const int64_t whole = attn_bwd_workspace_bytes(B, S, Hq, D, causal);
	if (Hkv <= 0 || Hq % Hkv != 0) return whole;
	return whole + dkv_part_bytes(split_walk(B, S, Hq, Hkv, D, causal != 0, INT64_MAX), B, S, Hkv, D);
}

AttnBwdWay attn_bwd_way(const void* v, int64_t ldq, int64_t ldv, int64_t lddo, int B, int S, int Hq, int Hkv, int D, int causal, int64_t workspace_bytes) {
	const bool reached = gemm_reaches(128, ldq) && gemm_reaches(128, lddo) && (D == 64 || (gemm_reaches(128, ldv) && ((uintptr_t)v % 16) == 0));
	if (reached && one_kernel_pays(B, S, Hq, Hkv, D, causal != 0)) return AttnBwdWay{0, 1, 1, 0};
	const Splits sp = split_walk(B, S, Hq, Hkv, D, causal != 0, workspace_bytes - attn_bwd_workspace_bytes(B, S, Hq, D, causal));
	return AttnBwdWay{sp.wide ? 256 : 128, sp.h, sp.q, causal && sp.paired && S > (sp.wide ? 256 : 128)};
}

int attn_bwd(const void* q, const void* k, const void* v, const void* o, const void* dO, const void* lse, void* dq,
             void* dk, void* dv, void* workspace, int64_t ldq, int64_t ldk, int64_t ldv, int64_t ldo, int64_t lddo,
             int64_t lddq, int64_t lddk, int64_t lddv, int B, int S, int Hq, int Hkv, int D, int causal, float scale,
             hipStream_t stream, const void* rope_cs, int64_t workspace_bytes) {
	ELF_REQUIRE(q && k && v && o && dO && lse && dq && dk && dv && workspace, "attn_bwd: null pointer");
	ELF_REQUIRE(((uintptr_t)rope_cs % 16) == 0, "attn_bwd: misaligned rotary table");
	ELF_REQUIRE(B > 0 && S > 0 && S % 128 == 0, "attn_bwd: sequence length must be a multiple of 128 (S=%d)", S);
	ELF_REQUIRE(Hkv > 0 && Hq % Hkv == 0, "attn_bwd: Hq must be a multiple of Hkv (Hq=%d Hkv=%d)", Hq, Hkv);
	ELF_REQUIRE(D == 64 || D == 128, "attn_bwd: head_dim must be 64 or 128 (D=%d)", D);
	ELF_REQUIRE(ldq % 8 == 0 && ldk % 8 == 0 && ldv % 8 == 0 && ldo % 8 == 0 && lddo % 8 == 0 && lddq % 8 == 0 &&
	                lddk % 8 == 0 && lddv % 8 == 0,
	            "attn_bwd: strides must be multiples of 8");
	ELF_REQUIRE(((uintptr_t)workspace % 16) == 0, "attn_bwd: misaligned workspace");
	const int64_t whole = attn_bwd_workspace_bytes(B, S, Hq, D, causal);
	ELF_REQUIRE(workspace_bytes >= whole, "attn_bwd: a workspace of %lld bytes, %lld are needed", (long long)workspace_bytes, (long long)whole);
	ELF_REQUIRE(((uintptr_t)o % 16) == 0 && ((uintptr_t)dO % 16) == 0, "attn_bwd: o and dO must be 16-byte aligned");
	ProfScope prof(PROF_ATTN_BWD, (causal ? 4.0 : 8.0) * B * Hq * (double)S * S * D, stream);
	const int64_t T = (int64_t)B * S;
	const AttnBwdWay way = attn_bwd_way(v, ldq, ldv, lddo, B, S, Hq, Hkv, D, causal, workspace_bytes);
	if (way.keys == 0) {
		const AttnBwdArgs a{(const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, (const bf16_t*)dO, nullptr, nullptr, nullptr,
		                    (bf16_t*)dk, (bf16_t*)dv, ldq, ldk, ldv, lddo, lddk, lddv, B, S, Hq, Hkv, scale, (const float2*)rope_cs, 1, 1, nullptr, 0, 0};
		return launch_bwd_one(a, D, causal != 0, (const bf16_t*)o, (const float*)lse, (bf16_t*)dq, ldo, lddq, stream);
	}
	bf16_t* dq_part = (bf16_t*)workspace;
	float* ndelta = (float*)(dq_part + (int64_t)B * part_rows(S, causal != 0, 128) * Hq * D);
	float* nlse2 = ndelta + T * Hq;
	{
		const int64_t rows = T * Hq, per_block = 256 / (D / 8);
		const int64_t want = (rows + per_block - 1) / per_block;
		ELF_LAUNCH(attn_delta_kernel, dim3((unsigned)(want < 8192 ? want : 8192)), dim3(256), 0, stream, (const bf16_t*)dO,
	                   (const bf16_t*)o, (const float*)lse, ndelta, nlse2, lddo, ldo, B, S, Hq, D);
	}
	float* dkv_part = way.h_splits * way.q_splits > 1 ? nlse2 + T * Hq : nullptr;
	const int nkt = (S + way.keys - 1) / way.keys;
	const int64_t workgroups = (int64_t)B * Hkv * (way.paired ? (nkt + 1) / 2 : nkt) * way.h_splits * way.q_splits;
	const int longest_first = causal && !way.paired && nkt > 1 && workgroups > 256;
	AttnBwdArgs a{(const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, (const bf16_t*)dO, nlse2, ndelta, dq_part,
	              (bf16_t*)dk, (bf16_t*)dv, ldq, ldk, ldv, lddo, lddk, lddv, B, S, Hq, Hkv, scale, (const float2*)rope_cs, way.h_splits, way.q_splits, dkv_part, way.paired, longest_first};
	const dim3 grid((unsigned)workgroups), block(256);
	int rc;
	if (way.keys == 256) rc = launch_bwd_wide(a, causal != 0, grid, stream);
	else if (D == 128) rc = causal ? launch_bwd<128, true>(a, grid, stream) : launch_bwd<128, false>(a, grid, stream);
	else rc = causal ? launch_bwd<64, true>(a, grid, stream) : launch_bwd<64, false>(a, grid, stream);
	if (rc) return rc;
	const int64_t n16 = T * (Hq * D / 16);
	const int64_t blocks = (n16 + 255) / 256;
	DkvReduce dkv{dkv_part, (bf16_t*)dk, (bf16_t*)dv, lddk, lddv, way.h_splits * way.q_splits, Hkv, 0};
	if (dkv_part) {
		const int64_t want = (2 * T * Hkv * (D / 16) + 255) / 256;
		dkv.blocks = (int)(want < 4096 ? want : 4096);
	}
	ELF_LAUNCH(dq_reduce_kernel, dim3((unsigned)(blocks < 16384 ? blocks : 16384) + dkv.blocks), dim3(256), 0, stream, dq_part, (bf16_t*)dq, B, S,
	                   Hq * D, lddq, scale, causal, way.keys, D, (const float2*)rope_cs, dkv);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

}  // namespace elf
