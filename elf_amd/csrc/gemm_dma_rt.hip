// Direct-to-LDS GEMMs with a k-contiguous A and an n-contiguous B (input gradients).
#include "gemm_dma_tile.h"

namespace elf {

namespace dma {

// 128- and 256-row tiles: every epilogue of the layout, whole and ragged sizes
template <int RF>
static int launch_epi(const Args& a, int epi, hipStream_t stream) {
	switch (epi) {
		case EPI_BF16: return launch<4, RF, false, true, EPI_BF16>(a, stream);
		case EPI_BF16_RESID: return launch<4, RF, false, true, EPI_BF16_RESID>(a, stream);
		case EPI_F32_ACC: return launch<4, RF, false, true, EPI_F32_ACC>(a, stream);
		case EPI_F32_STORE: return launch<4, RF, false, true, EPI_F32_STORE>(a, stream);
	}
	if constexpr (RF == 8) {
		if (epi == EPI_BF16_SWIGLU_BWD) return launch<4, RF, false, true, EPI_BF16_SWIGLU_BWD>(a, stream);
	}
	set_error("gemm: unknown epilogue %d", epi);
	return -1;
}

// the tiles between them: bf16 outputs, always clipped (an aligned size loses nothing by it)
template <int RF>
static int launch_mid(const Args& a, int epi, hipStream_t stream) {
	switch (epi) {
		case EPI_BF16: return launch_sized<4, RF, false, true, EPI_BF16, true>(a, stream);
		case EPI_BF16_RESID: return launch_sized<4, RF, false, true, EPI_BF16_RESID, true>(a, stream);
		case EPI_BF16_SWIGLU_BWD: return launch_sized<4, RF, false, true, EPI_BF16_SWIGLU_BWD, true>(a, stream);
	}
	set_error("gemm: epilogue %d has no %d-row tile", epi, RF * 32);
	return -1;
}

// 128 rows and 192 columns: always clipped as well
static int launch_192(const Args& a, int epi, hipStream_t stream) {
	switch (epi) {
		case EPI_BF16: return launch_sized<4, 4, false, true, EPI_BF16, true, 192>(a, stream);
		case EPI_BF16_RESID: return launch_sized<4, 4, false, true, EPI_BF16_RESID, true, 192>(a, stream);
	}
	set_error("gemm: epilogue %d has no 192-column tile", epi);
	return -1;
}

int launch_rt(int bm, int tn, const Args& a, int epi, hipStream_t stream) {
	if (tn == 192) return launch_192(a, epi, stream);
	switch (bm) {
		case 128: return launch_epi<4>(a, epi, stream);
		case 160: return launch_mid<5>(a, epi, stream);
		case 192: return launch_mid<6>(a, epi, stream);
		case 224: return launch_mid<7>(a, epi, stream);
		default: return launch_epi<8>(a, epi, stream);
	}
}

int rt_turn_giveups(uint64_t* sum) { return add_turn_giveups(sum); }

}  // namespace dma

}  // namespace elf
