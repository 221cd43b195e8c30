// Attention backward of 128-token sequences in one kernel (see attention_common.h for the layout conventions).
#include "attention_bwd_common.h"
#include <type_traits>

namespace elf {
namespace attn {

// One workgroup = the 128 tokens of one (batch, kv head): the one key tile there is, so dQ needs no partial sums and no second kernel,
// and every dO and O row is read by the workgroup that needs its -delta, so neither does that.  Waves w and w + 4 own keys
// [32w, 32w + 32) for S, dP, dV and dK, each with every other 32-query tile, and queries [32w, 32w + 32) for dQ.  Per query head Q and dO
// go to LDS whole, the query tiles are products without a barrier between them (dS stays in registers), and dS^T takes the place
// of Q and dO for the dQ product:
//   S = Q K^T, dP = dO V^T, P = exp2(S sc - lse), dS = P (dP - delta), dV^T += dO^T P, dK^T += Q^T dS | dQ^T = K^T dS^T
// At the end the waves of a pair swap: w adds the two dK, w + 4 the two dV.
// What bounds it is a chain: the tiles' way into LDS, two query tiles of five products a wave, dQ, the stores; four waves that take
// four tiles each were as slow for one head of 64 and 4 us slower for one of 128.  The call by itself, over and over on the same operands: 4 x
// 128 tokens, 4 heads of 64, causal 16.7 us in three kernels (and two launches more), 10.6; 4 heads of 128 20.0 -> 15.5; 8 x 128, 32 heads of 64
// 25.9 -> 13.6.  In the pass of a stage, between other kernels, the first takes 12.5 us of kernel.  dQ is rounded to bf16 once instead of
// twice: its error against 64 bits is 0.0026 for 0.0031 with heads of 128, and the same with those of 64, whose scale is a power of two.
template <int D, bool CAUSAL>
__global__ __launch_bounds__(512) void attn_bwd_one_kernel(AttnBwdArgs a, const bf16_t* __restrict__ O, const float* __restrict__ lse, bf16_t* dq, int64_t ldo, int64_t lddq) {
	using TL = BwdTile<D>;
	constexpr int S = 128, BQ = 32, NQT = S / BQ;
	constexpr int NF = D / 16, DT = D / 32;
	constexpr int T_BYTES = S * TL::ROW_BYTES, DS_BYTES = S * BQ * 2, SWAP_BYTES = 64 * 16 * DT * 4;
	constexpr int LPR = D / 8, RPS = 512 / LPR, STEPS = S / RPS;  // lanes per row, rows per step and steps of the delta pass
	constexpr bool KV_REGS = D == 64;  // K and V rows in registers; those of 128 columns do not fit beside the accumulators
	static_assert(NQT * DS_BYTES <= 2 * T_BYTES, "dS^T takes the place of Q and dO");
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];
	unsigned char* const sQ = smem_raw;
	unsigned char* const sdO = sQ + T_BYTES;
	unsigned char* const sK = sdO + T_BYTES;
	unsigned char* const sV = sK + T_BYTES;
	unsigned char* const sdS = sQ;  // [query tile][key][query]
	float* const sLse = reinterpret_cast<float*>(smem_raw + 8 * SWAP_BYTES);  // 128 nlse2, 128 -delta
	static_assert(4 * T_BYTES <= 8 * SWAP_BYTES, "the four tiles take the place of the swap");

	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kt = wave & 3, half = wave >> 2;
	const int g = lane >> 5, kl = lane & 31;
	const int G = a.Hq / a.Hkv, hk = (int)blockIdx.x % a.Hkv, b = (int)blockIdx.x / a.Hkv;
	const int64_t tok0 = (int64_t)b * S;
	const float sc = a.scale * LOG2E;
	const int key_l = kt * 32 + kl;

	f32x16 acc_dk[DT], acc_dv[DT];
#pragma unroll
	for (int i = 0; i < DT; i++)
#pragma unroll
		for (int r = 0; r < 16; r++) acc_dk[i][r] = acc_dv[i][r] = 0.f;
	bf16x8 kf[KV_REGS ? NF : 1], vf[KV_REGS ? NF : 1];

#pragma unroll 1
	for (int hh = 0; hh < G; hh++) {
		const int h = hk * G + hh;
		// (what a lane's addresses are made of, anew for every head and query tile: kept for the whole walk the addresses spill; without a mask
		// and with heads of 128 eleven registers do all the same, 48 bytes a lane)
		int ln = lane, id = tid;
		asm volatile("" : "+v"(ln), "+v"(id));
		// wave w moves rows [16w, 16w + 16) of a tile
		auto fetch = [&](const bf16_t* base, int64_t ld, unsigned char* tile) {
#pragma unroll
			for (int i = 0; i < 16 / TL::RPI; i++) {
				const int row = wave * 16 + i * TL::RPI + ln / TL::CPR, slot = ln % TL::CPR;
				dma16(base, (uint32_t)((row * ld + ((slot ^ TL::swz(row)) << 3)) * 2), __builtin_amdgcn_readfirstlane(lds_addr(tile) + (wave * 16 + i * TL::RPI) * TL::ROW_BYTES));
			}
		};
		if (hh > 0) __syncthreads();  // every wave is done with the dS^T of the head before
		fetch(a.q + tok0 * a.ldq + h * D, a.ldq, sQ);
		fetch(a.dO + tok0 * a.lddo + h * D, a.lddo, sdO);
		if (hh == 0) {
			fetch(a.k + tok0 * a.ldk + hk * D, a.ldk, sK);
			if constexpr (KV_REGS) {
				const bf16_t* kp = a.k + (tok0 + key_l) * a.ldk + hk * D + 8 * g;
				const bf16_t* vp = a.v + (tok0 + key_l) * a.ldv + hk * D + 8 * g;
#pragma unroll
				for (int ks = 0; ks < NF; ks++) kf[ks] = *reinterpret_cast<const bf16x8*>(kp + ks * 16), vf[ks] = *reinterpret_cast<const bf16x8*>(vp + ks * 16);
			} else {
				fetch(a.v + tok0 * a.ldv + hk * D, a.ldv, sV);
			}
		}
		// -delta = -rowsum(dO * O), LPR lanes a row (the order of attn_delta_kernel's sums)
		{
			bf16x8 x[STEPS], y[STEPS];
			const int sub = id % LPR, row0 = id / LPR;
#pragma unroll
			for (int i = 0; i < STEPS; i++) {
				x[i] = *reinterpret_cast<const bf16x8*>(a.dO + (tok0 + i * RPS + row0) * a.lddo + h * D + sub * 8);
				y[i] = *reinterpret_cast<const bf16x8*>(O + (tok0 + i * RPS + row0) * ldo + h * D + sub * 8);
			}
			if (id < S) sLse[id] = -lse[((int64_t)b * a.Hq + h) * S + id] * LOG2E;
#pragma unroll
			for (int i = 0; i < STEPS; i++) {
				float d = 0.f;
#pragma unroll
				for (int j = 0; j < 8; j++) d += (float)x[i][j] * (float)y[i][j];
#pragma unroll
				for (int o = LPR >> 1; o > 0; o >>= 1) d += __shfl_xor(d, o, 64);
				if (sub == 0) sLse[S + i * RPS + row0] = -d;
			}
		}
		wait_vmcnt<0>();
		__syncthreads();

		bf16x8 dsf[NQT / 2][2];
#pragma unroll
		for (int j = 0; j < NQT / 2; j++) {
			const int qt = 2 * j + half;
			if (CAUSAL && qt < kt) continue;  // every query of the tile lies before the wave's keys
			__builtin_amdgcn_sched_barrier(0);
			asm volatile("" : "+v"(ln));
			const unsigned char* const tq = sQ + qt * BQ * TL::ROW_BYTES;  // (32 rows on, the swizzle is the same)
			const unsigned char* const tdo = sdO + qt * BQ * TL::ROW_BYTES;
			const float* const stat = sLse + qt * BQ + 4 * g;
			f32x16 s, dp;
#pragma unroll
			for (int r = 0; r < 16; r++) s[r] = dp[r] = 0.f;
#pragma unroll
			for (int i = 0; i < NF; i++) {
				const bf16x8 k8 = KV_REGS ? kf[KV_REGS ? i : 0] : TL::rows(sK + kt * 32 * TL::ROW_BYTES, 0, i, ln);
				s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::rows(tq, 0, i, ln), k8, s, 0, 0, 0);
			}
#pragma unroll
			for (int i = 0; i < NF; i++) {
				const bf16x8 v8 = KV_REGS ? vf[KV_REGS ? i : 0] : TL::rows(sV + kt * 32 * TL::ROW_BYTES, 0, i, ln);
				dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::rows(tdo, 0, i, ln), v8, dp, 0, 0, 0);
			}
			// only the tile on the diagonal needs the mask: key > query  <=>  row index of the accumulator register < key - first query
			const int kq = kl - 4 * g;
			float p[16];
			auto softmax = [&](auto masked) {
#pragma unroll
				for (int r4 = 0; r4 < 4; r4++) {
					const f32x4 l4 = *reinterpret_cast<const f32x4*>(stat + r4 * 8);
#pragma unroll
					for (int t = 0; t < 4; t++) {
						float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r4 * 4 + t], sc, l4[t]));
						if (decltype(masked)::value && r4 * 8 + t < kq) pr = 0.f;
						p[r4 * 4 + t] = pr;
					}
				}
			};
			if (CAUSAL && qt == kt) softmax(std::true_type{});
			else softmax(std::false_type{});
			const bf16x8 pf[2] = {pack8(p), pack8(p + 8)};
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for (int i = 0; i < NF; i++)
				acc_dv[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::template cols<true>(tdo, (i / DT) * 16, (i % DT) * 32, ln), pf[i / DT], acc_dv[i % DT], 0, 0, 0);
			float ds[16];
#pragma unroll
			for (int r4 = 0; r4 < 4; r4++) {
				const f32x4 d4 = *reinterpret_cast<const f32x4*>(stat + S + r4 * 8);
#pragma unroll
				for (int t = 0; t < 4; t++) ds[r4 * 4 + t] = p[r4 * 4 + t] * (dp[r4 * 4 + t] + d4[t]);
			}
			dsf[j][0] = pack8(ds), dsf[j][1] = pack8(ds + 8);
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for (int i = 0; i < NF; i++)
				acc_dk[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::template cols<true>(tq, (i / DT) * 16, (i % DT) * 32, ln), dsf[j][i / DT], acc_dk[i % DT], 0, 0, 0);
		}
		__syncthreads();  // every wave is done with Q and dO
#pragma unroll
		for (int j = 0; j < NQT / 2; j++) {
			const int qt = 2 * j + half;
			if (CAUSAL && qt < kt) continue;  // (nothing reads these)
#pragma unroll
			for (int u = 0; u < 2; u++) {
				const u32x4 w = __builtin_bit_cast(u32x4, dsf[j][u]);
				*reinterpret_cast<u32x2*>(sdS + qt * DS_BYTES + ds_t_offset(key_l, 16 * u + 4 * g)) = u32x2{w[0], w[1]};
				*reinterpret_cast<u32x2*>(sdS + qt * DS_BYTES + ds_t_offset(key_l, 16 * u + 8 + 4 * g)) = u32x2{w[2], w[3]};
			}
		}
		__syncthreads();
		// dQ: the pair shares a query tile's columns.  Heads of 128: the column tiles (half, half + 2), which the rotation pairs; of 64:
		// one each, or with a rotation, which pairs the two, both by the first wave
		bf16_t* const dqp = dq + (tok0 + key_l) * lddq + h * D;
		const float2* const cs = a.rope_cs ? a.rope_cs + (int64_t)key_l * (D / 2) : nullptr;
		asm volatile("" : "+v"(ln));
		auto dq_tiles = [&](auto two, int dt0, int dt1) {
			f32x16 lo, hi;
#pragma unroll
			for (int r = 0; r < 16; r++) lo[r] = hi[r] = 0.f;
#pragma unroll
			for (int t = 0; t < NQT; t++) {
				if (CAUSAL && t > kt) continue;  // keys after the queries
#pragma unroll
				for (int i = 0; i < 2; i++) {
					const bf16x8 f = ds_t_frag(sdS + kt * DS_BYTES, t * 32 + i * 16, ln);
					lo = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::template cols<false>(sK, t * 32 + i * 16, dt0 * 32, ln), f, lo, 0, 0, 0);
					if constexpr (decltype(two)::value) hi = __builtin_amdgcn_mfma_f32_32x32x16_bf16(TL::template cols<false>(sK, t * 32 + i * 16, dt1 * 32, ln), f, hi, 0, 0, 0);
				}
			}
			if (decltype(two)::value && cs) {
				store_tiles_rotated<D>(lo, hi, dqp + dt0 * 32, a.scale, g, cs + dt0 * 32);
			} else {
				store_tile(lo, dqp + dt0 * 32, a.scale, g);
				if constexpr (decltype(two)::value) store_tile(hi, dqp + dt1 * 32, a.scale, g);
			}
		};
		if (DT == 4) dq_tiles(std::true_type{}, half, half + 2);
		else if (cs == nullptr) dq_tiles(std::false_type{}, half, 0);
		else if (half == 0) dq_tiles(std::true_type{}, 0, 1);
	}
	// the swap: a wave leaves what its partner adds, register by register
	__syncthreads();  // every wave is done with K and the last dS^T
	f32x4* const mine = reinterpret_cast<f32x4*>(smem_raw + wave * SWAP_BYTES) + lane;
	const f32x4* const other = reinterpret_cast<const f32x4*>(smem_raw + (wave ^ 4) * SWAP_BYTES) + lane;
	auto leave = [&](const f32x16(&acc)[DT]) {
#pragma unroll
		for (int i = 0; i < 4 * DT; i++) mine[i * 64] = f32x4{acc[i / 4][i % 4 * 4], acc[i / 4][i % 4 * 4 + 1], acc[i / 4][i % 4 * 4 + 2], acc[i / 4][i % 4 * 4 + 3]};
	};
	auto add = [&](f32x16(&acc)[DT]) {
#pragma unroll
		for (int i = 0; i < 4 * DT; i++) {
			const f32x4 v = other[i * 64];
#pragma unroll
			for (int t = 0; t < 4; t++) acc[i / 4][i % 4 * 4 + t] += v[t];
		}
	};
	if (half == 0) leave(acc_dv);
	else leave(acc_dk);
	__syncthreads();
	if (half == 0) {
		add(acc_dk);
		store_dk<D>(acc_dk, a.dk + (tok0 + key_l) * a.lddk + hk * D, a.scale, g, a.rope_cs ? a.rope_cs + (int64_t)key_l * (D / 2) : nullptr);
	} else {
		add(acc_dv);
		store_dv<D>(acc_dv, a.dv + (tok0 + key_l) * a.lddv + hk * D, g);
	}
}

template <int D, bool CAUSAL>
static int launch_one(const AttnBwdArgs& a, const bf16_t* o, const float* lse, bf16_t* dq, int64_t ldo, int64_t lddq, hipStream_t stream) {
	constexpr int smem = 8 * 64 * (D / 2) * 4 + 2 * 128 * 4;
	static bool attr_set = false;
	if (!attr_set) {
		ELF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(attn_bwd_one_kernel<D, CAUSAL>), hipFuncAttributeMaxDynamicSharedMemorySize, smem));
		attr_set = true;
	}
	ELF_LAUNCH((attn_bwd_one_kernel<D, CAUSAL>), dim3((unsigned)(a.B * a.Hkv)), dim3(512), smem, stream, a, o, lse, dq, ldo, lddq);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

int launch_bwd_one(const AttnBwdArgs& a, int D, bool causal, const bf16_t* o, const float* lse, bf16_t* dq, int64_t ldo, int64_t lddq, hipStream_t stream) {
	if (D == 128) return causal ? launch_one<128, true>(a, o, lse, dq, ldo, lddq, stream) : launch_one<128, false>(a, o, lse, dq, ldo, lddq, stream);
	return causal ? launch_one<64, true>(a, o, lse, dq, ldo, lddq, stream) : launch_one<64, false>(a, o, lse, dq, ldo, lddq, stream);
}

}  // namespace attn
}  // namespace elf
