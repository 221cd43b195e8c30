// The two figures of PyTorch's caching allocator that the Engine books after every operation of a step, for callers that would
// otherwise build the allocator's whole statistics tree as Python dictionaries for them (5 us an operation; 0.5 us here).
#include <c10/hip/HIPCachingAllocator.h>

#include <cstdint>

// The PyTorch whose headers this was built against: the figures lie where that one keeps them.
extern "C" const char* elf_torch_built_for() { return ELF_TORCH_VERSION; }

// out[0] = bytes allocated on `device` now, out[1] = the peak.  -1: the allocator knows no such device.
extern "C" int elf_torch_allocated(int device, int64_t* out) {
	try {
		const auto stats = c10::hip::HIPCachingAllocator::getDeviceStats((c10::DeviceIndex)device);
		const auto& bytes = stats.allocated_bytes[(size_t)c10::CachingAllocator::StatType::AGGREGATE];
		out[0] = bytes.current;
		out[1] = bytes.peak;
		return 0;
	} catch (...) {
		return -1;
	}
}
