// NO_CPU_VARIANT (compared with the loops of the oracle)
// The convolution program (tiramisu_amd/programs/conv2d.cpp) at sizes that take each of the tiles for gathered operands: one row or a few
// positions in the last tiles, a few k in the last slice, and whole ones.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/conv2d.cpp"
#undef main

int main()
{
    generate(2, 41, 33, 13);      // 32x32, four groups of wavefronts; one row in the second tiles
    generate(1, 64, 32, 8);       // 32x32, whole
    generate(1, 44, 15, 96);      // 32x64, four groups
    generate(3, 15, 8, 91);       // 32x128
    generate(8, 40, 50, 92);      // 64x64
    generate(7, 11, 35, 67);      // 64x128
    generate(1, 64, 64, 16);      // 32x32 where few 64x64 tiles would share slices between two groups
    generate(4, 64, 64, 64);      // such 64x64 tiles, one for every compute unit
    return 0;
}
