// NO_CPU_VARIANT (compared with the oracle)
// The five-point sweep (tiramisu_amd/programs/heat2d.cpp) on planes whose strips have fewer than 11 rows per thread and whose rows end
// one cell short of a whole quad.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/heat2d.cpp"
#undef main

int main()
{
    generate(67, 23);      // 11 and 12 steps with strips of 4 rows, boundary tiles only
    generate(203, 15);     // 3 steps with 2 rows, 12 with 4
    generate(1367, 23);    // 11 steps with 5 rows, 12 with 6, interior tiles
    generate(1631, 12);    // 3 steps with 6 rows and slices of 3, 9 with 6
    return 0;
}
