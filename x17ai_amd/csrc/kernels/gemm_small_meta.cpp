// Prints the launch geometry of the small-tile GEMM kernel configured by common.h as JSON.
#include "common.h"
#include "gemm_small_tile.h"
#include <cstdio>

int main() {
	namespace st = x17::gemm_small_tile;
	std::printf("{\n");
	std::printf("\t\"THREADS_PER_BLOCK\": %u,\n", st::THREADS_PER_BLOCK);
	std::printf("\t\"SMEM_BYTES\": %u,\n", st::SMEM_BYTES);
	std::printf("\t\"M_PER_BLOCK\": %u,\n", st::M_PER_BLOCK);
	std::printf("\t\"N_PER_BLOCK\": %u\n", st::N_PER_BLOCK);
	std::printf("}\n");
}
