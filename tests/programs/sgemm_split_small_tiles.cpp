// NO_CPU_VARIANT (compared with float64 products)
// The fp32 sgemm program (tiramisu_amd/programs/sgemm.cpp) at sizes that take the small tiles of split operands beyond the whole
// 64 x 64 ones: guarded in every direction, and half as long again on one side.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/sgemm.cpp"
#undef main

int main()
{
    generate(446, 1497, 733);      // 64x64, guarded, thirteen k in the last slice
    generate(1001, 1503, 703);     // 64x96, guarded
    generate(1344, 1024, 176);     // 96x64, whole, some wavefronts with one slice, some with two
    return 0;
}
