// NO_CPU_VARIANT (compared with float64 sums)
// The convolution program (tiramisu_amd/programs/conv2d.cpp) where the windowed kernel splits its operands into bf16 parts: four
// blocks of channels, 576 tiles for 512 workgroups, so that the last 64 are cut into pieces.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/conv2d.cpp"
#undef main

int main()
{
    generate(9, 32, 64, 128);
    return 0;
}
