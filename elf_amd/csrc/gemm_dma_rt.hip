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

int launch_rt(int bm, const Args& a, int epi, hipStream_t stream) { return bm == 128 ? launch_epi<4>(a, epi, stream) : launch_epi<8>(a, epi, stream); }

int rt_turn_giveups(uint64_t* sum) { return add_turn_giveups(sum); }

}  // namespace dma

}  // namespace elf
