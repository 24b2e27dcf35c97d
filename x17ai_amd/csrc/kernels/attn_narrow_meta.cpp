// Prints the launch geometry of the attention kernel with sixteen queries per wavefront, configured by common.h, as JSON
// (reference: templates/attn/meta.cu).
#include "common.h"
#include "attn_narrow_tile.h"
#include <cstdio>

int main() {
	namespace nt = x17::attn_narrow_tile;
	std::printf("{\n");
	std::printf("\t\"THREADS_PER_BLOCK\": %u,\n", nt::THREADS_PER_BLOCK);
	std::printf("\t\"SMEM_BYTES\": %u,\n", nt::SMEM_BYTES);
	std::printf("\t\"Q_PER_BLOCK\": %u\n", nt::Q_PER_BLOCK);
	std::printf("}\n");
}
