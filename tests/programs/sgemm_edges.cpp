// NO_CPU_VARIANT (compared with float64 products)
// The fp32 sgemm program (tiramisu_amd/programs/sgemm.cpp) at sizes that end inside a tile, a slice and a 16-byte piece of the
// operands.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/sgemm.cpp"
#undef main

int main()
{
    generate(300, 260, 1001);     // one k in the last slice, rows at every alignment
    generate(130, 4098, 131);     // the larger tiles
    generate(2001, 1501, 37);
    generate(65, 67, 33);
    generate(14, 1732, 433);      // fewer rows than a tile
    generate(9, 3, 66);           // fewer columns than a 16-byte load
    generate(37, 70, 3);          // fewer k than one
    generate(70, 45, 64);         // whole slices
    generate(96, 96, 64);         // whole 32x32 tiles
    generate(224, 160, 32);       // whole 32x32 tiles, slices of 32 k
    generate(416, 2592, 31);      // guarded slices of 32 k
    generate(130, 95, 9);
    return 0;
}
