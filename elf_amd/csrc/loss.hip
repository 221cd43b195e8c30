// Cross-entropy of a pipeline's last stage over bf16 logits [rows, V] (row stride ld), computed in
// fp32 as the reference's loss function does after its upcast (benchmarks/models/simple.py:520-524,
// called from Engine.compute_loss, elf/execution/engine.py:374-410):
//     loss[r]      = logsumexp(x[r, :]) - x[r, target[r]]            (0 for target == ignore_index)
//     dlogits[r,c] = (softmax(x[r, :])[c] - (c == target[r])) * scale (0 for ignored rows and for
//                    the padding columns V <= c < ld_out)
// Forward and backward are one kernel — 4 bytes per logit of HBM traffic instead of the 10+ of a
// log-softmax / gather / scatter chain.  Rows of up to 65536 columns, and most of up to 131072, are
// read once into registers, reduced, and their gradient written from the same registers; longer rows
// are read twice by their workgroup.
#include "common.h"
#include "kernels.h"

namespace elf {

namespace {

constexpr float LOG2E_F = 1.4426950408889634f;

// 2^x as the bare hardware instruction: no denormal-range fix-up (results below 2^-126 flush to zero,
// which a softmax term that small may do).
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

struct LossArgs {
	const bf16_t* x;
	int64_t ld;
	const int64_t* target;
	int64_t rows;
	int V;
	int64_t ignore_index;
	float scale;
	const float* dev_div;  // optional device scalar the gradient is divided by
	int count;             // != 0: the gradient is divided by the number of live rows, which every wave counts (G = 64 only)
	float* row_loss;       // optional
	bf16_t* dx;            // optional
	int64_t ld_out;
};

// Reductions over the G threads that share a row (G = 64: one wave; otherwise G / 64 waves of one
// workgroup, through LDS).
template <int G, bool MAX>
__device__ __forceinline__ float group_reduce(float v, float* red) {
	v = MAX ? wave_max(v) : wave_sum(v);
	if constexpr (G > 64) {
		constexpr int NW = G / 64;
		const int wave = threadIdx.x >> 6;
		__syncthreads();
		if ((threadIdx.x & 63) == 0) red[wave] = v;
		__syncthreads();
		v = red[0];
#pragma unroll
		for (int i = 1; i < NW; i++) v = MAX ? fmaxf(v, red[i]) : v + red[i];
	}
	return v;
}

__device__ __forceinline__ float grad_scale(const LossArgs& a) { return a.dev_div ? a.scale / *a.dev_div : a.scale; }

// Loss of one row from its statistics; NaN for a target outside [0, V) that is not ignore_index.
__device__ __forceinline__ float row_loss_of(const LossArgs& a, int64_t row, int64_t tgt, float m, float s) {
	if (tgt == a.ignore_index) return 0.f;
	if (tgt < 0 || tgt >= a.V) return __builtin_nanf("");
	return m + logf(s) - (float)a.x[row * a.ld + tgt];
}

// Launches of at most this many rows of at most COUNT_COLS columns count the live rows themselves, each wave under the loads of its own
// row, instead of reading what a launch before them counted.  Loss, gradient and its product with the incoming one, counted before and
// here (us): 64 x 1000 10.8 and 8.5, 512 x 1000 11.1 and 9.5, 1024 x 1000 11.9 and 11.2, 1024 x 4080 18.4 and 17.7, 1536 x 1000 13.1 and 13.3, 2048 x
// 512 12.1 and 13.2, 2048 x 4080 26.1 and 29.5.  Not wider rows: the registers are full there.
constexpr int COUNT_ROWS = 1024, COUNT_COLS = 64 * 8 * 8;

// G threads per row, C 16-byte chunks (8 logits) per thread: rows of up to G * C * 8 columns, read once into registers,
// reduced there, and their gradient written from the same registers.  Bound: HBM (4 bytes per logit) and, close behind, the two
// exponentials per logit.  Rows beyond 16384 columns used to be read twice by 256 threads, the second time from a cache that
// the rows in flight on the chip (2048 of 100 KB) do not fit; loss and gradient, before -> after: 4096 x 50304 235 -> 167 us
// (3.5 -> 4.9 TB/s), 8192 x 20000 168 -> 130, 2048 x 128256 262 -> 241.
//
// DENSE: rows of V columns one after the other, so that they start at any 2-byte address; x and dx lie alike modulo 16 bytes.
// A row is walked in the aligned 16-byte chunks that cover it.  The first and the last of them, where they are shared with the
// neighbouring rows (or with what lies behind the last column), are read and written element by element by lanes 0 and 1.
// Rows that lie apart have their last chunk to themselves: it is taken whole and masked (element by element 301 x 1350 took 5.7 us,
// 4.2 masked; 36 x 1014 5.0 and 3.7).
// STREAM: the logits are read past the caches, so that these hold the gradient for who reads it next.  Loss, gradient and its product with the
// incoming one, 4096 x 32000 186 -> 171 us, 1024 x 128256 213 -> 195, 2048 x 50257 161 -> 157; the gradient written past them as well 190, 205 and 167.
template <int G, int C, bool DENSE, bool STREAM>
__global__ __launch_bounds__(G < 256 ? 256 : G, G >= 256 ? 64 / C : 1) void cross_entropy_kernel(LossArgs a) {
	constexpr int BLOCK = G < 256 ? 256 : G;
	constexpr int ROWS = BLOCK / G;
	constexpr bool WIDE = G * C * 8 > 16384;
	__shared__ float red[BLOCK / 64];
	const int lane = ROWS == 1 ? (int)threadIdx.x : (int)threadIdx.x % G;
	const int64_t row = ROWS == 1 ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * ROWS + threadIdx.x / G;
	if (ROWS > 1 && row >= a.rows) return;  // whole waves leave together (G = 64 when ROWS > 1)
	const int rot = DENSE ? (int)(((uintptr_t)(a.x + row * a.ld) >> 1) & 7) : 0;  // columns of chunk 0 that belong to the row before
	const bf16_t* const xr = a.x + (row * a.ld - rot);  // chunk c holds columns c * 8 - rot .. + 7, at xr + c * 8
	// the chunks taken whole: those that lie inside the row; not DENSE, where a row's last chunk is the row's own, that one too
	const int cbeg = rot != 0, cend = DENSE ? (a.V + rot) / 8 : (a.V + 7) / 8;
	const int tail = DENSE || a.V % 8 == 0 ? -1 : cend - 1;  // its columns from V % 8 on are masked
	// the edge chunk of this lane, if any, and its elements inside the row
	const int ec = !DENSE ? -1 : lane == 0 && rot ? 0 : lane == 1 && (a.V + rot) % 8 && (cend > 0 || !rot) ? cend : -1;
	const int elo = ec == 0 ? rot : 0, ehi = min(8, a.V + rot - ec * 8);

	bf16x8 reg[C];
	float m = -INFINITY;
#pragma unroll
	for (int j = 0; j < C; j++) {
		const int c = j * G + lane;
		if (c >= cbeg && c < cend) {
			const bf16x8* p = reinterpret_cast<const bf16x8*>(xr + (int64_t)c * 8);
			reg[j] = STREAM ? __builtin_nontemporal_load(p) : *p;
		}
	}
	float live = 0.f;
	if constexpr (G == 64) {
		if (a.count) {
			for (int64_t r = lane; r < a.rows; r += 64) live += a.target[r] != a.ignore_index ? 1.f : 0.f;
			live = wave_sum(live);
		}
	}
	if (ec >= 0) {
		for (int i = elo; i < ehi; i++) m = fmaxf(m, (float)xr[(int64_t)ec * 8 + i]);
	}
#pragma unroll
	for (int j = 0; j < C; j++) {
		const int c = j * G + lane;
		if (c >= cbeg && c < cend) {
			if (!DENSE && c == tail) {
#pragma unroll
				for (int i = 1; i < 8; i++)
					if (i >= a.V % 8) reg[j][i] = (bf16_t)-INFINITY;
			}
#pragma unroll
			for (int i = 0; i < 8; i++) m = fmaxf(m, (float)reg[j][i]);
		}
	}
	m = group_reduce<G, true>(m, red);
	const float m2 = m * LOG2E_F;
	float s = 0.f;
#pragma unroll
	for (int j = 0; j < C; j++) {
		const int c = j * G + lane;
		if (c >= cbeg && c < cend) {
#pragma unroll
			for (int i = 0; i < 8; i++) s += fast_exp2(fmaf((float)reg[j][i], LOG2E_F, -m2));
		}
	}
	if (ec >= 0) {
		for (int i = elo; i < ehi; i++) s += fast_exp2(fmaf((float)xr[(int64_t)ec * 8 + i], LOG2E_F, -m2));
	}
	s = group_reduce<G, false>(s, red);

	const int64_t tgt = a.target[row];
	if (a.row_loss && lane == 0) a.row_loss[row] = row_loss_of(a, row, tgt, m, s);
	if (!a.dx) return;
	const float g = tgt != a.ignore_index ? G == 64 && a.count ? a.scale / live : grad_scale(a) : 0.f;
	bf16_t* const dr = a.dx + (row * a.ld_out - rot);
	const int tchunk = tgt >= 0 && tgt < a.V ? (int)((tgt + rot) >> 3) : -1, tcol = (int)((tgt + rot) & 7);
	// softmax * |g| of the wide rows = exp2(x*log2e - (m + log2(s) - log2|g|)), its sign by an exclusive or: no product per
	// logit; a zero factor (an ignored row) gives zeros whatever the logits are
	const bool zero = WIDE && g == 0.f;
	const float gs = g / s, shift = WIDE ? m2 + log2f(s) - log2f(fabsf(g)) : m2;
	const uint32_t sign = WIDE && g < 0.f ? 0x80000000u : 0u;
	auto softmax = [&](bf16_t x) {
		float v = fast_exp2(fmaf((float)x, LOG2E_F, -shift));
		if constexpr (WIDE) return zero ? 0.f : __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) ^ sign);
		return v * gs;
	};
#pragma unroll
	for (int j = 0; j < C; j++) {
		const int c = j * G + lane;
		if (c < cbeg || c >= cend) continue;
		float v[8];
#pragma unroll
		for (int i = 0; i < 8; i++) v[i] = softmax(reg[j][i]);
		if (c == tchunk) {
#pragma unroll
			for (int i = 0; i < 8; i++)
				if (i == tcol) v[i] -= g;
		}
		if (!DENSE && c == tail) {
#pragma unroll
			for (int i = 1; i < 8; i++)
				if (i >= a.V % 8) v[i] = 0.f;
		}
		bf16x8 o;
#pragma unroll
		for (int i = 0; i < 8; i++) o[i] = (bf16_t)v[i];
		*reinterpret_cast<bf16x8*>(dr + (int64_t)c * 8) = o;
	}
	if (ec >= 0) {
		for (int i = elo; i < ehi; i++) dr[(int64_t)ec * 8 + i] = (bf16_t)(softmax(xr[(int64_t)ec * 8 + i]) - (ec == tchunk && i == tcol ? g : 0.f));
	}
	if constexpr (!DENSE)
		for (int64_t c = cend + lane; c < a.ld_out / 8; c += G) *reinterpret_cast<bf16x8*>(dr + c * 8) = bf16x8{};  // padding columns
}

// Rows beyond those registers; of rows that start on 16-byte boundaries also those that do not fill them well (see
// cross_entropy()) and wide ones whose gradient nobody asked for (nothing is read twice then, and more and smaller workgroups
// hide the loads better: 4096 x 50304 82 us against 100, 2048 x 128256 99 against 129).  Dense rows have the kernel above only.
// G threads per row (one workgroup), an online max / sum over one read of the row, then a second read for the gradient.  The running maximum only
// rescales the partial sum when it grows, column masks are confined to the last chunk of a row, the 1/sum * scale factor rides
// in the exponent, and the target column is fixed up by the one thread that holds it.
template <bool MASKED>
__device__ __forceinline__ void online_chunk(const bf16x8& r, int c, int V, float& m, float& s) {
	float x[8];
#pragma unroll
	for (int i = 0; i < 8; i++) x[i] = (MASKED && c * 8 + i >= V) ? -INFINITY : (float)r[i];
	const float cm = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7]))) * LOG2E_F;
	if (cm > m) {  // rare after the first chunks; s is 0 while m is -inf
		s *= fast_exp2(m - cm);
		m = cm;
	}
#pragma unroll
	for (int i = 0; i < 8; i++) s += fast_exp2(fmaf(x[i], LOG2E_F, -m));  // exp2(-inf) = 0 for masked columns
}

template <int G>
__global__ __launch_bounds__(G) void cross_entropy_stream_kernel(LossArgs a) {
	__shared__ float red[G / 64];
	const int lane = threadIdx.x;
	const int64_t row = blockIdx.x;
	const bf16_t* xr = a.x + row * a.ld;
	const int vchunks = (a.V + 7) / 8;
	const int full = a.V / 8;  // chunks with all 8 columns inside the row
	float m = -INFINITY, s = 0.f;  // m is in units of log2: max(x) * log2(e)
	int c = lane;
	for (; c + G < full; c += 2 * G) {  // two loads in flight per thread
		const bf16x8 r0 = *reinterpret_cast<const bf16x8*>(xr + (int64_t)c * 8);
		const bf16x8 r1 = *reinterpret_cast<const bf16x8*>(xr + (int64_t)(c + G) * 8);
		online_chunk<false>(r0, c, a.V, m, s);
		online_chunk<false>(r1, c + G, a.V, m, s);
	}
	for (; c < vchunks; c += G) {
		const bf16x8 r = *reinterpret_cast<const bf16x8*>(xr + (int64_t)c * 8);
		if (c < full) online_chunk<false>(r, c, a.V, m, s);
		else online_chunk<true>(r, c, a.V, m, s);
	}
	const float gm = group_reduce<G, true>(m, red);
	s = (m == -INFINITY) ? 0.f : s * fast_exp2(m - gm);
	s = group_reduce<G, false>(s, red);
	const float mx = gm * (1.f / LOG2E_F);  // back to natural units for the loss

	const int64_t tgt = a.target[row];
	if (a.row_loss && lane == 0) a.row_loss[row] = row_loss_of(a, row, tgt, mx, s);
	if (!a.dx) return;
	const float g = tgt != a.ignore_index ? grad_scale(a) : 0.f;
	bf16_t* dr = a.dx + row * a.ld_out;
	const int ochunks = (int)(a.ld_out / 8);
	if (g == 0.f) {  // ignored row (or a zero scale): the whole row of the gradient is zero
		bf16x8 z;
#pragma unroll
		for (int i = 0; i < 8; i++) z[i] = (bf16_t)0.f;
		for (int c2 = lane; c2 < ochunks; c2 += G) *reinterpret_cast<bf16x8*>(dr + (int64_t)c2 * 8) = z;
		return;
	}
	// softmax * |g| = exp2(x*log2e - (m + log2(s) - log2|g|)); the sign of g is applied after
	const float shift = gm + log2f(s) - log2f(fabsf(g));
	const float sign = g < 0.f ? -1.f : 1.f;
	const int tchunk = (tgt >= 0 && tgt < a.V) ? (int)(tgt >> 3) : -1;
	for (int c2 = lane; c2 < ochunks; c2 += G) {
		float v[8];
		if (c2 < full) {
			const bf16x8 r = *reinterpret_cast<const bf16x8*>(xr + (int64_t)c2 * 8);
#pragma unroll
			for (int i = 0; i < 8; i++) v[i] = fast_exp2((float)r[i] * LOG2E_F - shift) * sign;
		} else if (c2 < vchunks) {
			const bf16x8 r = *reinterpret_cast<const bf16x8*>(xr + (int64_t)c2 * 8);
#pragma unroll
			for (int i = 0; i < 8; i++) v[i] = c2 * 8 + i < a.V ? fast_exp2((float)r[i] * LOG2E_F - shift) * sign : 0.f;
		} else {
#pragma unroll
			for (int i = 0; i < 8; i++) v[i] = 0.f;
		}
		if (c2 == tchunk) {
#pragma unroll
			for (int i = 0; i < 8; i++)
				if (i == (int)(tgt & 7)) v[i] -= g;
		}
		bf16x8 o;
#pragma unroll
		for (int i = 0; i < 8; i++) o[i] = (bf16_t)v[i];
		*reinterpret_cast<bf16x8*>(dr + (int64_t)c2 * 8) = o;
	}
}

// out[0] = sum of row_loss (skipped when row_loss is null), out[1] = number of rows whose target is
// not ignore_index; loss (optional) = out[0], or out[0] / out[1] if mean.  One workgroup, fixed summation order: the same inputs
// give the same bits.
__global__ __launch_bounds__(1024) void cross_entropy_reduce_kernel(const float* __restrict__ row_loss, const int64_t* __restrict__ target,
                                                                    int64_t rows, int64_t ignore_index, float* __restrict__ out,
                                                                    float* __restrict__ loss, int mean) {
	__shared__ float red[16];
	float s = 0.f, n = 0.f;
	for (int64_t r = threadIdx.x; r < rows; r += 1024) {
		if (row_loss) s += row_loss[r];
		n += target[r] != ignore_index ? 1.f : 0.f;
	}
	s = group_reduce<1024, false>(s, red);
	n = group_reduce<1024, false>(n, red);
	if (threadIdx.x == 0) {
		if (out) {
			if (row_loss) out[0] = s;
			out[1] = n;
		}
		if (loss) *loss = mean ? s / n : s;
	}
}

// Which logits are read past the caches: those that the memory-side cache does not hold, 2^27 of them, and from 84 M on in long rows, where
// the gradient then finds more room: of 8192 columns and more if they start on 128-byte lines, otherwise of 32768.  Loss, gradient and product, with
// what produces the logits before, as usual and past the caches (us): 3108 x 31552 206 and 188, 2680 x 46784 266 and 245, 4096 x 32000 273 and 254.  On
// the other side of the lines, loss and padded gradient: 4959 x 10592 78 and 84, 5736 x 11824 99 and 109, 6641 x 10176 97 and 102; of 200 runs from
// 2^25 up a third were 2 to 12 % slower past them.  Dense rows without a gradient only from 2^27 on: at 2^26 they take 3 % longer.
template <bool DENSE>
bool past_caches(const LossArgs& a) {
	const int64_t n = a.rows * a.V, columns = !DENSE && a.ld % 64 == 0 && ((uintptr_t)a.x & 127) == 0 ? 8192 : 32768;
	return n >= int64_t(1) << 27 || (n >= int64_t(5) << 24 && a.V >= columns && (!DENSE || a.dx));
}

template <int G, int C, bool DENSE>
void launch_rows(const LossArgs& a, hipStream_t s) {
	constexpr int BLOCK = G < 256 ? 256 : G;
	constexpr int ROWS = BLOCK / G;
	const dim3 grid((unsigned)((a.rows + ROWS - 1) / ROWS));
	if (past_caches<DENSE>(a)) ELF_LAUNCH((cross_entropy_kernel<G, C, DENSE, true>), grid, dim3(BLOCK), 0, s, a);
	else ELF_LAUNCH((cross_entropy_kernel<G, C, DENSE, false>), grid, dim3(BLOCK), 0, s, a);
}

// The narrowest group of threads whose registers hold a row of `width` columns; false: none does.
template <bool DENSE>
bool launch_resident(const LossArgs& a, int64_t width, hipStream_t s) {
	if (width <= 64 * 2 * 8) launch_rows<64, 2, DENSE>(a, s);
	else if (width <= 64 * 8 * 8) launch_rows<64, 8, DENSE>(a, s);
	else if (width <= 256 * 8 * 8) launch_rows<256, 8, DENSE>(a, s);
	else if (width <= 512 * 8 * 8) launch_rows<512, 8, DENSE>(a, s);
	else if (width <= 1024 * 8 * 8) launch_rows<1024, 8, DENSE>(a, s);
	else if (width <= 1024 * 16 * 8) launch_rows<1024, 16, DENSE>(a, s);
	else return false;
	return true;
}

// y = x * g, both factors and the product rounded to bf16 once (g is an fp32 scalar on the device).  U chunks of 16 bytes per
// thread.  Bound: HBM.  STREAM: past the caches, for arrays these do not hold; 4096 x 128256 464 us -> 352 (4.5 -> 6.0 TB/s; walked
// with a grid of 8192 workgroups before), 1024 x 151936 125 -> 89, 2048 x 50257 69 -> 60.  16 MB take 7.5 us either way, and stay
// in the caches for who reads the gradient next.
constexpr int64_t STREAM_ELEMS = int64_t(1) << 25;
template <int U, bool STREAM>
__global__ __launch_bounds__(256) void scale_by_kernel(const bf16_t* __restrict__ x, const float* __restrict__ g, bf16_t* __restrict__ y, int64_t n) {
	const float f = (float)(bf16_t)*g;
	const int64_t nchunks = n >> 3, first = (int64_t)blockIdx.x * (256 * U) + threadIdx.x;
	bf16x8 v[U];
#pragma unroll
	for (int u = 0; u < U; u++) {
		const bf16x8* p = reinterpret_cast<const bf16x8*>(x) + first + u * 256;
		if (first + u * 256 < nchunks) v[u] = STREAM ? __builtin_nontemporal_load(p) : *p;
	}
#pragma unroll
	for (int u = 0; u < U; u++) {
		if (first + u * 256 >= nchunks) continue;
#pragma unroll
		for (int j = 0; j < 8; j++) v[u][j] = (bf16_t)((float)v[u][j] * f);
		bf16x8* p = reinterpret_cast<bf16x8*>(y) + first + u * 256;
		if constexpr (STREAM) __builtin_nontemporal_store(v[u], p);
		else *p = v[u];
	}
	if (blockIdx.x == 0 && threadIdx.x < (n & 7)) y[nchunks * 8 + threadIdx.x] = (bf16_t)((float)x[nchunks * 8 + threadIdx.x] * f);
}

template <int U, bool STREAM>
void launch_scale_by(const bf16_t* x, const float* g, bf16_t* y, int64_t n, hipStream_t s) {
	const int64_t blocks = (n / 8 + 256 * U - 1) / (256 * U);
	ELF_LAUNCH((scale_by_kernel<U, STREAM>), dim3((unsigned)(blocks < 1 ? 1 : blocks)), dim3(256), 0, s, x, g, y, n);
}

}  // namespace

int cross_entropy(const void* logits, int64_t ld, const void* target, int64_t rows, int64_t V, int64_t ignore_index, float scale,
                  const void* dev_div, void* row_loss, void* dlogits, int64_t ld_out, hipStream_t s, bool count) {
	ELF_REQUIRE(logits && target && rows > 0 && V > 0 && V < (1ll << 30), "cross_entropy: bad argument");
	ELF_REQUIRE(rows < (1ll << 31), "cross_entropy: too many rows");
	ELF_REQUIRE(ld % 8 == 0 && ld >= V && ((uintptr_t)logits & 15) == 0,
	            "cross_entropy: logits rows must start on 16-byte boundaries (row stride %lld must be a multiple of 8 and >= V)", (long long)ld);
	ELF_REQUIRE(row_loss || dlogits, "cross_entropy: nothing to compute (no row_loss and no dlogits)");
	if (dlogits)
		ELF_REQUIRE(ld_out % 8 == 0 && ld_out >= V && ((uintptr_t)dlogits & 15) == 0,
		            "cross_entropy: gradient rows must start on 16-byte boundaries (row stride %lld must be a multiple of 8 and >= V)", (long long)ld_out);
	LossArgs a{(const bf16_t*)logits, ld, (const int64_t*)target, rows, (int)V, ignore_index, scale, (const float*)dev_div, count,
	           (float*)row_loss, (bf16_t*)dlogits, dlogits ? ld_out : 0};
	const int64_t width = dlogits && ld_out > V ? ld_out : V;
	ProfScope prof(PROF_LOSS, (dlogits ? 4.0 : 2.0) * rows * V, s);
	// 1024 threads with 16 chunks each leave room for one row per compute unit, the two-read kernel for two: it is the faster one
	// where the registers are little more than half filled (4096 x 70656 as fast, 136 x 67936 12.9 us against 14.5) and where rows
	// make a little more than one round (279 x 130568 44 against 54); 4096 x 100000 371 us against 356, 4096 x 128256 483 and 450
	const bool twice = width > 65536 && (width < 98304 || rows < 512);
	if (!dlogits && width > 16384 && width <= 65536) ELF_LAUNCH(cross_entropy_stream_kernel<256>, dim3((unsigned)rows), dim3(256), 0, s, a);
	else if ((!dlogits && width > 16384) || twice || !launch_resident<false>(a, width, s)) ELF_LAUNCH(cross_entropy_stream_kernel<1024>, dim3((unsigned)rows), dim3(1024), 0, s, a);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

int cross_entropy_dense(const void* logits, const void* target, int64_t rows, int64_t V, int64_t ignore_index, float scale, const void* dev_div,
                        void* row_loss, void* dlogits, hipStream_t s, bool count) {
	ELF_REQUIRE(logits && target && rows > 0 && rows < (1ll << 31) && V > 0, "cross_entropy_dense: bad argument");
	ELF_REQUIRE(V <= 1024 * 16 * 8 - 7, "cross_entropy_dense: rows of at most %d columns (V=%lld)", 1024 * 16 * 8 - 7, (long long)V);
	ELF_REQUIRE(row_loss || dlogits, "cross_entropy_dense: nothing to compute (no row_loss and no dlogits)");
	ELF_REQUIRE(((uintptr_t)logits & 1) == 0 && (!dlogits || ((uintptr_t)logits & 15) == ((uintptr_t)dlogits & 15)),
	            "cross_entropy_dense: logits and their gradient must lie alike modulo 16 bytes");
	LossArgs a{(const bf16_t*)logits, V, (const int64_t*)target, rows, (int)V, ignore_index, scale, (const float*)dev_div, count, (float*)row_loss, (bf16_t*)dlogits, V};
	ProfScope prof(PROF_LOSS, (dlogits ? 4.0 : 2.0) * rows * V, s);
	launch_resident<true>(a, V + 7, s);  // a row may cover one chunk more than V / 8
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

int scale_by_bf16(const void* x, const void* g_f32, void* y, int64_t n, hipStream_t s) {
	ELF_REQUIRE(x && g_f32 && y && n > 0, "scale_by: bad argument");
	ELF_REQUIRE(((uintptr_t)x & 15) == 0 && ((uintptr_t)y & 15) == 0 && ((uintptr_t)g_f32 & 3) == 0, "scale_by: pointers must be 16-byte aligned");
	ELF_REQUIRE(n < (int64_t(1) << 42), "scale_by: too many elements");
	if (n < STREAM_ELEMS) launch_scale_by<1, false>((const bf16_t*)x, (const float*)g_f32, (bf16_t*)y, n, s);
	else launch_scale_by<2, true>((const bf16_t*)x, (const float*)g_f32, (bf16_t*)y, n, s);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

int cross_entropy_reduce(const void* row_loss, const void* target, int64_t rows, int64_t ignore_index, void* out2, hipStream_t s) {
	ELF_REQUIRE(target && out2 && rows > 0, "cross_entropy_reduce: bad argument");
	ELF_LAUNCH(cross_entropy_reduce_kernel, dim3(1), dim3(1024), 0, s, (const float*)row_loss, (const int64_t*)target, rows,
	                   ignore_index, (float*)out2, nullptr, 0);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

int cross_entropy_loss(const void* logits, int64_t ld, bool dense, const void* target, int64_t rows, int64_t V, int64_t ignore_index, float scale, bool mean,
                       void* row_loss, void* loss, void* dlogits, int64_t ld_out, void* scratch2, hipStream_t s) {
	ELF_REQUIRE(row_loss && loss && scratch2, "cross_entropy_loss: null pointer");
	const bool divide = mean && dlogits, count = divide && rows <= COUNT_ROWS && (dense ? V + 7 : ld_out > V ? ld_out : V) <= COUNT_COLS;
	float* const out2 = (float*)scratch2;
	if (divide && !count)
		if (int rc = cross_entropy_reduce(nullptr, target, rows, ignore_index, out2, s)) return rc;
	const void* div = divide && !count ? out2 + 1 : nullptr;
	if (int rc = dense ? cross_entropy_dense(logits, target, rows, V, ignore_index, scale, div, row_loss, dlogits, s, count)
	                   : cross_entropy(logits, ld, target, rows, V, ignore_index, scale, div, row_loss, dlogits, ld_out, s, count))
		return rc;
	ELF_LAUNCH(cross_entropy_reduce_kernel, dim3(1), dim3(1024), 0, s, (const float*)row_loss, (const int64_t*)target, rows, ignore_index, (float*)nullptr, (float*)loss, (int)mean);
	ELF_CHECK_HIP(hipGetLastError());
	return 0;
}

}  // namespace elf
