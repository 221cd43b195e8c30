// Attention backward for heads of 64 columns: 256 keys per workgroup pass, 64 per wave.
#include "attention_bwd_common.h"
#include "gemm_tile.h"

namespace elf {
namespace attn {

// acc += a b in place, on accumulator registers: left to the builtin the accumulators of dK and dV lie in the vector half of the
// file, which the rest of a step needs, and are copied to and fro.  The compiler does not see a matrix product here: whoever
// reads the operands or the accumulator keeps the distance (two instructions after an operand is written; the accumulators are read
// behind a barrier).
__device__ __forceinline__ void mfma_acc(f32x16& acc, const bf16x8& a, const bf16x8& b) {
	asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

template <class T>
__device__ __forceinline__ T ELF_LDS* lds_ptr(uint32_t addr) { return (T ELF_LDS*)(uintptr_t)addr; }
__device__ __forceinline__ bf16x8 tr_frag(uint32_t lo_addr, uint32_t hi_addr, uint32_t imm) {
	s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(uintptr_t)(lo_addr + imm));
	s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 ELF_LDS*)(uintptr_t)(hi_addr + imm));
	return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// The pass of attn_bwd_kernel (attention_bwd.hip) over twice the keys: wave w owns keys [64w, 64w + 64) as two halves of 32, so
// that every Q and dO fragment read from LDS feeds two products.  At 64 columns that is what bounded the pass: with 32 keys per
// wave a 32-query step reads 30 KB of LDS (240 cycles of the compute unit's 128 B/clk, four waves at a time) for 640 cycles of
// MFMA and 500 of softmax arithmetic, and two waves per SIMD overlapped hardly any of it.  Here one wave has its SIMD to itself, and as
// in attn_bwd_kernel_lone the schedule is explicit: a step is 40 slots of one 32x32x16 MFMA each (or two of 16x16x32), with the LDS
// reads, the stores and the vector work dealt between them.  S runs a tile ahead, so that P of the first keys is formed while dK
// still multiplies.
//   slots  0- 7  dP   = dO V^T - delta      reads: dO^T, dS^T of the previous tile   vector: P of the last 32 keys
//          8-15  dV^T += dO^T P                                                             dS of the first 32 keys
//         16-23  dQ   = (K^T dS^T)(prev)    Q rows, lse of the next tile                    dS of the others, dS^T -> LDS
//         24-31  S    = Q K^T (next tile)   Q^T; dO rows of the next tile                   dQ out
//         32-39  dK^T += Q^T dS             delta of the next tile                          P of the next tile's first 32 keys
// A wave's share of dQ is 32 columns of 16 queries over all 256 keys: half as many partial sums as with 128 keys, to write, to read
// back and to round.  -delta is what the dP products start from, which saves a subtraction per element.  The ring of tiles has four
// stages and a step's code one of them, so that every LDS address is a constant of the lane and an offset field.
// Main kernel and whole call, by itself and over and over, 128 -> 256 keys (us): 8192 tokens, 16 heads, causal 486 -> 327 (0.71 -> 1.05 PFLOP/s of the five products) and
// 559 -> 360; 8 x 1024, 12 heads, not causal 128 -> 103 whole (1.5 rounds of workgroups; in a stage's pass the main kernel alone takes 96).  A step takes 2330 cycles, 1280 of them
// MFMA; the instructions of a lone wave issue one at a time (1370), an exponential holds the vector pipe for four (another 380).
// Dealing the exponentials evenly over the slots, with S two products earlier, or alternating the halves' products made no difference.
// Keys past the end of the sequence (S an odd multiple of 128: waves 2 and 3 of the last pass) are computed on the last ones that
// there are, with zeros for K in the dQ product, and nothing of them is stored.
template <bool CAUSAL>
__global__ __launch_bounds__(256) void attn_bwd_wide_kernel(AttnBwdArgs a) {
	constexpr int D = 64;
	using TL = BwdTile<D>;
	constexpr int BKV = 256, BQ = 32;
	constexpr int NF = D / 16;    // fragments per operand tile
	constexpr int DT = D / 32;
	constexpr int NQ = BKV / 32;  // 32-key steps of the dQ product
	constexpr int K_BYTES = BKV * TL::ROW_BYTES, Q_BYTES = BQ * TL::ROW_BYTES;
	constexpr int STAGE = 2 * Q_BYTES + 256;  // Q tile, dO tile, 32 nlse2 + 32 delta floats
	constexpr int NSTAGE = 4;                 // tiles are fetched three steps ahead
	constexpr int DS_BYTES = BKV * BQ * 2;
	constexpr int BUFFER_FLAGS = 0x00020000;  // a raw buffer descriptor: 32-bit data format, offsets checked against the size in bytes
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
	unsigned char* const sKt = smem_raw;                 // K tile, [key][d]
	unsigned char* const sStage = sKt + K_BYTES;         // NSTAGE x {Q [q][d], dO [q][d], nlse2, delta}
	unsigned char* const sdS = sStage + NSTAGE * STAGE;  // 2 x dS^T [key][q]

	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int g = lane >> 5, kl = lane & 31;
	const int nwt = (a.S + BKV - 1) / BKV;
	const int npair = CAUSAL && a.paired ? (nwt + 1) / 2 : nwt;
	const Walk wk = locate_walk(a, npair, CAUSAL);
	const int pair = wk.pair, hk = wk.hk, b = wk.b;
	const int64_t tok0 = (int64_t)b * a.S;
	const int64_t HqD = (int64_t)a.Hq * D;
	const float sc = a.scale * LOG2E;
	const int dq_dt = wave & 1, dq_half = wave >> 1;  // this wave's share of a dQ tile: 32 columns of 16 queries
	const int nqt_all = a.S / BQ;
	// lane part of a dQ tile address (bytes): one query, the first of 4 columns
	const int dq_lane = ((dq_half * 16 + (lane & 15)) * (int)HqD + dq_dt * 32 + 4 * (lane >> 4)) * 2;

	// LDS addresses of this lane, for ring stage 0 and dS^T buffer 0: everything else is a compile-time offset on top
	const uint32_t lds_stage0 = lds_addr(sStage), lds_ds = lds_addr(sdS);
	uint32_t row_r[NF], col_r[DT][2], ds_r[2], ds_w[4], st_r;
#pragma unroll
	for (int i = 0; i < NF; i++) row_r[i] = lds_stage0 + (uint32_t)(kl * TL::ROW_BYTES + (((2 * i + g) ^ TL::swz(kl)) << 4));
	{
		const int j = lane & 15, kk = 4 * g + (j >> 2);  // (the transpose reads of BwdTile::cols<true> and ds_t_frag)
#pragma unroll
		for (int m = 0; m < DT; m++) {
			const int c = (m * 32 + 16 * ((lane & 31) >> 4) + 4 * (j & 3)) >> 3;
#pragma unroll
			for (int u = 0; u < 2; u++) col_r[m][u] = lds_stage0 + (uint32_t)((kk + 8 * u) * TL::ROW_BYTES + ((c ^ TL::swz(kk + 8 * u)) << 4) + (j & 1) * 8);
		}
		// B operand of a 16x16x32 product: lane = query (of the wave's 16), keys 8 (lane / 16) .. + 7 of a step's 32
#pragma unroll
		for (int u = 0; u < 2; u++) ds_r[u] = lds_ds + (uint32_t)ds_t_offset(8 * (lane >> 4) + (j >> 2) + 4 * u, dq_half * 16 + 4 * (j & 3));
#pragma unroll
		for (int c = 0; c < 4; c++) ds_w[c] = lds_ds + (uint32_t)ds_t_offset(wave * 64 + kl, 8 * c + 4 * g);
		st_r = lds_stage0 + 2 * Q_BYTES + 16 * g;
	}
	// opaque: folded into these, the regions' bases would push the offsets past their 16 bits
#pragma unroll
	for (int i = 0; i < 4; i++) asm volatile("" : "+v"(row_r[i]), "+v"(col_r[i / 2][i % 2]), "+v"(ds_w[i]));
	asm volatile("" : "+v"(ds_r[0]), "+v"(ds_r[1]), "+v"(st_r));
	const uint32_t lds_stage = __builtin_amdgcn_readfirstlane(lds_stage0 + wave * 8 * TL::ROW_BYTES);

	// DMA plan for one (Q, dO) tile pair: wave w moves rows [w*8, w*8+8) of each
	uint32_t qoff, dooff;
	{
		const int row = wave * 8 + lane / TL::CPR, slot = lane % TL::CPR;
		qoff = (uint32_t)((row * a.ldq + ((slot ^ TL::swz(row)) << 3)) * 2);
		dooff = (uint32_t)((row * a.lddo + ((slot ^ TL::swz(row)) << 3)) * 2);
	}

	const int n_pass = (CAUSAL && a.paired && nwt - 1 - pair != pair) ? 2 : 1;
#pragma unroll 1
	for (int pass = 0; pass < n_pass; pass++) {
		const int kt_idx = pass == 0 ? pair : nwt - 1 - pair;
		const int key0 = kt_idx * BKV;  // first key of the pass
		const bool mine = key0 + wave * 64 < a.S;                      // this wave has keys of its own
		const int wkey0 = min(key0 + wave * 64, a.S - 64);             // first key of this wave
		if (pass > 0) __syncthreads();                                 // every wave is done with the LDS of the previous pass

		// K tile -> LDS; this wave moves its own 64 rows (zeros for keys past the end: they add nothing to dQ)
		if (mine) {
			const bf16_t* kb = a.k + (tok0 + wkey0) * a.ldk + hk * D;
#pragma unroll
			for (int i = 0; i < 64 / TL::RPI; i++) {
				const int row = i * TL::RPI + lane / TL::CPR, slot = lane % TL::CPR;  // (the swizzle repeats every 16 rows)
				dma16(kb, (uint32_t)((row * a.ldk + ((slot ^ TL::swz(row)) << 3)) * 2),
				      __builtin_amdgcn_readfirstlane(lds_addr(sKt) + (wave * 64 + i * TL::RPI) * TL::ROW_BYTES));
			}
		} else {
#pragma unroll
			for (int i = 0; i < 64 * TL::ROW_BYTES / 1024; i++) *lds_ptr<u32x4>(lds_addr(sKt) + wave * 64 * TL::ROW_BYTES + i * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
		}
		// own K and V rows as B operands (n = key, 8 consecutive d) in registers, in the accumulator half of the file (see attn_bwd_kernel)
		bf16x8 kf[2][NF], vf[2][NF];
#pragma unroll
		for (int h = 0; h < 2; h++) {
			const bf16_t* kp = a.k + (tok0 + wkey0 + h * 32 + kl) * a.ldk + hk * D + 8 * g;
			const bf16_t* vp = a.v + (tok0 + wkey0 + h * 32 + kl) * a.ldv + hk * D + 8 * g;
#pragma unroll
			for (int ks = 0; ks < NF; ks++) {
				kf[h][ks] = *reinterpret_cast<const bf16x8*>(kp + ks * 16);
				vf[h][ks] = *reinterpret_cast<const bf16x8*>(vp + ks * 16);
			}
		}
#pragma unroll
		for (int h = 0; h < 2; h++)
#pragma unroll
			for (int ks = 0; ks < NF; ks++) asm volatile("" : "+a"(kf[h][ks]), "+a"(vf[h][ks]));
		f32x16 acc_dk[2][DT], acc_dv[2][DT];
#pragma unroll
		for (int h = 0; h < 2; h++)
#pragma unroll
			for (int i = 0; i < DT; i++)
#pragma unroll
				for (int r = 0; r < 16; r++) acc_dk[h][i][r] = acc_dv[h][i][r] = 0.f;

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
		auto issue = [&](auto stage) {
			constexpr int ST = decltype(stage)::value;
			dma16_at<ST * STAGE>(ld_q, qoff, lds_stage);
			dma16_at<ST * STAGE + Q_BYTES>(ld_do, dooff, lds_stage);
			if (wave == 0) dma4(ld_stat, __builtin_amdgcn_readfirstlane(lds_stage + ST * STAGE + 2 * Q_BYTES));
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

		dma::static_for<NSTAGE - 1>([&](auto sc) {
			if (decltype(sc)::value < n_iter) issue(sc);
		});
#pragma unroll
		for (int h = 0; h < 2; h++)  // the "previous tile" of the first step
#pragma unroll
			for (int c = 0; c < 4; c++) *lds_ptr<u32x2>(ds_w[c] + DS_BYTES + h * 32 * 64) = u32x2{0u, 0u};
		wait_vmcnt<0>();
		__syncthreads();
		// this wave's 32 columns of K as A operands of the dQ^T product (rows d, k = key)
		bf16x8 ktf[2][NQ];
		{
			const int j = lane & 15, kk = 8 * (lane >> 4) + (j >> 2);
#pragma unroll
			for (int t = 0; t < 2; t++) {
				const int c = (dq_dt * 32 + t * 16 + 4 * (j & 3)) >> 3;
				uint32_t p[2];
#pragma unroll
				for (int u = 0; u < 2; u++) p[u] = lds_addr(sKt) + (uint32_t)((kk + 4 * u) * TL::ROW_BYTES + ((c ^ TL::swz(kk + 4 * u)) << 4) + (j & 1) * 8);
#pragma unroll
				for (int i = 0; i < NQ; i++) ktf[t][i] = tr_frag(p[0], p[1], i * 32 * TL::ROW_BYTES);
			}
		}
#pragma unroll
		for (int i = 0; i < NQ; i++) asm volatile("" : "+a"(ktf[0][i]), "+a"(ktf[1][i]));

		// the current tile and where its dQ goes; the one before it (dq_prev_bytes: its size; 0: the first step has none)
		int cur_qt = q_lo;
		const int64_t dq_step = BQ * HqD;
		bf16_t* dq_tile = a.dq_part + ((int64_t)b * part_rows(a.S, CAUSAL, BKV) + part_row0(kt_idx, a.S, CAUSAL, BKV) + (q_lo - qt_first) * BQ) * HqD + wk.h0 * D;
		const int64_t dq_next_head = D - (int64_t)(q_hi - q_lo) * dq_step;
		bf16_t* dq_prev_tile = dq_tile;
		int dq_prev_bytes = 0;
		// Two 8-byte stores per tile and lane, through a buffer descriptor of that tile: with a size of zero it drops them, so that
		// every step has the same stores in flight and no branch.
		auto dq_rsrc = [&]() { return __builtin_amdgcn_make_buffer_rsrc(dq_prev_tile, 0, dq_prev_bytes, BUFFER_FLAGS); };
		f32x4 dq[2];
		auto dq_out = [&](__amdgpu_buffer_rsrc_t rsrc, int t) {
			bf16x4 o;
#pragma unroll
			for (int r = 0; r < 4; r++) o[r] = (bf16_t)dq[t][r];
			__builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, o), rsrc, dq_lane + 32 * t, 0, 0);
		};
		auto dq_mfma = [&](int i, const bf16x8& ds) {
#pragma unroll
			for (int t = 0; t < 2; t++) {
				if (i == 0) dq[t] = f32x4{0.f, 0.f, 0.f, 0.f};
				dq[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ktf[t][i], ds, dq[t], 0, 0, 0);
			}
		};

		f32x16 s[2], dp[2];      // S, then P; dP - delta, then dS
		f32x16 nd;               // -delta of this lane's 16 rows: what the dP products start from
		f32x4 l4[4];             // -lse log2(e) of these rows
		bf16x8 qr[NF], dor[NF], pf[2][2], dsf[2][2];
		// P of a half: elements [lo, hi) of its 16 registers
		auto softmax = [&](int h, int lo, int hi) {
#pragma unroll
			for (int r = lo; r < hi; r++) s[h][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[h][r], sc, l4[r >> 2][r & 3]));
		};
		auto pack = [&](const f32x16& v, int u) {
			bf16x8 o;
#pragma unroll
			for (int t = 0; t < 8; t++) o[t] = (bf16_t)v[8 * u + t];
			return o;
		};
		auto read_nd = [&](int stage, int r4) {
			const f32x4 v = *lds_ptr<const f32x4>(st_r + stage * STAGE + 128 + r4 * 32);
#pragma unroll
			for (int t = 0; t < 4; t++) nd[4 * r4 + t] = v[t];
		};
		// before the first step: S of the first tile, P of its first 32 keys, dO rows and delta
		{
#pragma unroll
			for (int i = 0; i < NF; i++) qr[i] = *lds_ptr<const bf16x8>(row_r[i]), dor[i] = *lds_ptr<const bf16x8>(row_r[i] + Q_BYTES);
#pragma unroll
			for (int r4 = 0; r4 < 4; r4++) {
				l4[r4] = *lds_ptr<const f32x4>(st_r + r4 * 32);
				read_nd(0, r4);
			}
#pragma unroll
			for (int h = 0; h < 2; h++) {
#pragma unroll
				for (int r = 0; r < 16; r++) s[h][r] = 0.f;
#pragma unroll
				for (int i = 0; i < NF; i++) s[h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qr[i], kf[h][i], s[h], 0, 0, 0);
			}
			softmax(0, 0, 16);
		}
		// One step on the tile of ring stage ST (steps go round the ring: every LDS address is a lane's constant and an offset field)
		auto step = [&](auto stage, int it) {
			constexpr int ST = decltype(stage)::value, CUR = ST * STAGE, NEXT = (ST + 1) % NSTAGE * STAGE, DS_CUR = ST % 2 * DS_BYTES, DS_PREV = DS_BYTES - DS_CUR;
			const auto rsrc = dq_rsrc();
			if (it + NSTAGE - 1 < n_iter) issue(std::integral_constant<int, (ST + NSTAGE - 1) % NSTAGE>{});
			const int q0 = cur_qt * BQ;
			dq_prev_tile = dq_tile;
			dq_prev_bytes = BQ * (int)HqD * 2;
			dq_tile += dq_step;
			if (++cur_qt == q_hi) {
				cur_qt = q_lo;
				dq_tile += dq_next_head;
			}

			bf16x8 sf[NQ], dot[NF], qt[NF];
			// causal mask: key > query  <=>  row index of the accumulator register < key - q0; only tiles on the diagonal
			// (a half's last key lies after the tile's first query) need it
			auto mask = [&](int h) {
				if (CAUSAL && wkey0 + h * 32 + 31 > q0) {
					const int kq = wkey0 + h * 32 + kl - q0 - 4 * g;
#pragma unroll
					for (int r = 0; r < 16; r++)
						if ((r >> 2) * 8 + (r & 3) < kq) s[h][r] = 0.f;
				}
			};
			// accumulator rows of register r: q = (r/4)*8 + 4g + r%4 -> four 8-byte groups per lane
			auto write_ds = [&](int h, int u) {
				const u32x4 w = __builtin_bit_cast(u32x4, dsf[h][u]);
				*lds_ptr<u32x2>(ds_w[2 * u] + DS_CUR + h * 32 * 64) = u32x2{w[0], w[1]};
				*lds_ptr<u32x2>(ds_w[2 * u + 1] + DS_CUR + h * 32 * 64) = u32x2{w[2], w[3]};
			};
			// columns d of the dO (Q) tile, fragment f: queries (f / DT) * 16 .., columns (f % DT) * 32 ..
			auto cols = [&](int f, int tile) { return tr_frag(col_r[f % DT][0], col_r[f % DT][1], tile + (f / DT) * 16 * TL::ROW_BYTES); };
			dma::static_for<40>([&](auto nc) {
				constexpr int n = decltype(nc)::value, i = n % 8, h = i / 4, f = i % 4;
				// the matrix product of the slot
				if constexpr (n < 8) {
					dp[h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dor[f], vf[h][f], f == 0 ? nd : dp[h], 0, 0, 0);
				} else if constexpr (n < 16) {
					mfma_acc(acc_dv[h][f % DT], dot[f], pf[h][f / DT]);
				} else if constexpr (n < 24) {
					dq_mfma(i, sf[i]);  // (two of half the size)
				} else if constexpr (n < 32) {
					if constexpr (f == 0)
#pragma unroll
						for (int r = 0; r < 16; r++) s[h][r] = 0.f;
					s[h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qr[f], kf[h][f], s[h], 0, 0, 0);
				} else {
					mfma_acc(acc_dk[h][f % DT], qt[f], dsf[h][f / DT]);
				}
				// LDS reads, a group of products and more ahead of their use (past the last tile those of the next one hit a stale
				// stage; their values are not used)
				if constexpr (n < 4) dot[n] = cols(n, CUR + Q_BYTES);
				if constexpr (n >= 4 && n < 12) sf[n - 4] = tr_frag(ds_r[0], ds_r[1], DS_PREV + (n - 4) * 32 * 64);
				if constexpr (n >= 16 && n < 20) qr[n - 16] = *lds_ptr<const bf16x8>(row_r[n - 16] + NEXT);
				if constexpr (n >= 20 && n < 24) l4[n - 20] = *lds_ptr<const f32x4>(st_r + NEXT + (n - 20) * 32);
				if constexpr (n >= 24 && n < 28) qt[n - 24] = cols(n - 24, CUR);
				if constexpr (n >= 28 && n < 32) dor[n - 28] = *lds_ptr<const bf16x8>(row_r[n - 28] + NEXT + Q_BYTES);
				if constexpr (n >= 32 && n < 36) read_nd((ST + 1) % NSTAGE, n - 32);
				// vector work.  An operand of mfma_acc is formed two slots or more before the product that reads it
				if constexpr (n == 0) mask(0);
				if constexpr (n == 1 || n == 2) pf[0][n - 1] = pack(s[0], n - 1);
				if constexpr (n < 10) softmax(1, n * 16 / 10, (n + 1) * 16 / 10);
				if constexpr (n == 10) mask(1);
				if constexpr (n == 10 || n == 11) pf[1][n - 10] = pack(s[1], n - 10);
				if constexpr (n >= 12 && n < 20) {
#pragma unroll
					for (int r = n % 4 * 4; r < n % 4 * 4 + 4; r++) dp[(n - 12) / 4][r] *= s[(n - 12) / 4][r];
					if constexpr (n % 2 == 1) dsf[(n - 12) / 4][n % 4 / 2] = pack(dp[(n - 12) / 4], n % 4 / 2);
				}
				if constexpr (n == 16 || n == 17) write_ds(0, n - 16);
				if constexpr (n == 20 || n == 21) write_ds(1, n - 20);
				if constexpr (n == 26 || n == 27) dq_out(rsrc, n - 26);
				if constexpr (n >= 29) softmax(0, (n - 29) * 16 / 11, (n - 28) * 16 / 11);
				__builtin_amdgcn_sched_barrier(0);
			});
			asm volatile("" : "+v"(s[0]));  // formed here, not where the next step reads it
			// The tile after next has to have landed.  Vector memory operations complete in order, and behind its loads came the
			// two stores of the step before, the loads of one more tile (none near the end) and this step's two stores.  LDS
			// operations complete in order too: all but the last eight (the next tile's dO rows and delta) are waited for
			wait_counters<4, 8>();
			asm volatile("s_barrier" ::: "memory");  // dS^T of this tile is complete, everyone is done with this tile
			__builtin_amdgcn_sched_barrier(0);
		};
#pragma unroll 1
		for (int it = 0; it < n_iter; it += NSTAGE)
			dma::static_for<NSTAGE>([&](auto sc) {
				if (it + decltype(sc)::value < n_iter) step(sc, it + decltype(sc)::value);
			});
		// dQ product and partial of the last tile
		{
			const uint32_t last = (uint32_t)((n_iter - 1) & 1) * DS_BYTES;
#pragma unroll
			for (int i = 0; i < NQ; i++) dq_mfma(i, tr_frag(ds_r[0] + last, ds_r[1] + last, i * 32 * 64));
			const auto rsrc = dq_rsrc();
			dq_out(rsrc, 0);
			dq_out(rsrc, 1);
		}

		// dK^T / dV^T accumulators: register r <-> d = dt*32 + (r/4)*8 + 4g + r%4, lane <-> key
		if (!mine) continue;
#pragma unroll
		for (int h = 0; h < 2; h++) {
			const int key = wkey0 + h * 32 + kl;
			if (a.dkv_part) {
				store_dkv_part<D>(acc_dk[h], acc_dv[h], a.dkv_part + (((int64_t)wk.split * 2 * a.B * a.S + tok0 + key) * a.Hkv + hk) * D, (int64_t)a.B * a.S * a.Hkv * D, g);
				continue;
			}
			store_dk_dv<D>(acc_dk[h], acc_dv[h], a.dk + (tok0 + key) * a.lddk + hk * D, a.dv + (tok0 + key) * a.lddv + hk * D, a.scale, g,
			               a.rope_cs ? a.rope_cs + (int64_t)key * (D / 2) : nullptr);
		}
	}
}

template <bool CAUSAL>
static int launch_wide(const AttnBwdArgs& a, dim3 grid, hipStream_t stream) {
	constexpr int smem = 256 * 64 * 2 + 4 * (2 * 32 * 64 * 2 + 256) + 2 * 256 * 32 * 2;
	static bool attr_set = false;
	if (!attr_set) {
		ELF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(attn_bwd_wide_kernel<CAUSAL>), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
		attr_set = true;
	}
	ELF_LAUNCH((attn_bwd_wide_kernel<CAUSAL>), grid, dim3(256), smem, stream, a);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

int launch_bwd_wide(const AttnBwdArgs& a, bool causal, dim3 grid, hipStream_t stream) {
	return causal ? launch_wide<true>(a, grid, stream) : launch_wide<false>(a, grid, stream);
}

}  // namespace attn
}  // namespace elf
