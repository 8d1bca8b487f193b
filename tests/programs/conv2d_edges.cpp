// NO_CPU_VARIANT (compared with the loops of the oracle)
// The convolution program (tiramisu_amd/programs/conv2d.cpp) with channels and image widths that no tile, slice or 16-byte load
// divides.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/conv2d.cpp"
#undef main

int main()
{
    generate(2, 5, 7, 9);
    generate(1, 3, 33, 10);
    generate(3, 9, 17, 20);       // rows of whole 16-byte loads
    generate(2, 31, 64, 33);
    generate(1, 64, 50, 12);
    return 0;
}
