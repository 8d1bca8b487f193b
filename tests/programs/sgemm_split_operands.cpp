// NO_CPU_VARIANT (compared with float64 products)
// The fp32 sgemm program (tiramisu_amd/programs/sgemm.cpp) at sizes whose operands are split into bf16 parts: every tile of
// kernels/gemm_mfma_split.hip.h, whole and guarded.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/sgemm.cpp"
#undef main

int main()
{
    generate(704, 1088, 528);      // 64x64 tiles, an odd number of slices, not the same for every wavefront
    generate(1408, 2560, 416);     // 128x128, whole
    generate(1219, 2747, 611);     // 128x128, rows at every alignment, everything ends inside a tile
    generate(2560, 3584, 208);     // 256x256, whole
    generate(2560, 3584, 210);     // 256x256, guarded in K only
    generate(2701, 3915, 99);      // 256x256, guarded, three k in the last slice
    return 0;
}
