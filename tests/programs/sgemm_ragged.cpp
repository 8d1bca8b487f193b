// NO_CPU_VARIANT (compared with float64 products)
// The fp32 sgemm program (tiramisu_amd/programs/sgemm.cpp) at sizes that no square of split operands covers well.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/sgemm.cpp"
#undef main

int main()
{
    generate(446, 1497, 733);
    generate(1001, 1503, 703);
    generate(1344, 1024, 176);     // whole tiles, few k
    return 0;
}
