// Fused NTT kernels of one tile size (VK_TILE, log2 words) and one modulus
// class (VK_CLASS): the Makefile compiles this file once per pair.
#include "ntt_fused.h"

namespace vk {

template <>
const ClassKernels *fused_class_table<VK_TILE, VK_CLASS>() {
	static const std::array<ClassKernels, kFusedEntries> table =
		make_class_table<VK_TILE, VK_CLASS>(
				std::make_integer_sequence<int, kFusedEntries>());
	return table.data();
}

}  // namespace vk
