// NO_CPU_VARIANT (compared with float64 products)
// The bf16 sgemm program (tiramisu_amd/programs/sgemm_bf16.cpp) at sizes that take the tiles between the squares, and slices in
// pairs: one row or a few columns in the last tiles, a few k in the last stage.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/sgemm_bf16.cpp"
#undef main

int main()
{
    generate(1793, 3842, 514);    // 128 x 256
    generate(1921, 2562, 578);    // 192 x 128
    generate(673, 3202, 1090);    // 96 x 128
    generate(1473, 642, 514);     // 64 x 128
    generate(33, 66, 194);        // 32 x 64
    generate(2000, 1500, 1010);   // 128 x 128, pairs: the last one begins its second slice
    generate(3842, 3970, 1278);   // 256 x 256, pairs
    generate(1920, 2560, 1024);   // whole tiles of 192 x 128
    generate(3841, 3074, 1088);   // 256 x 256, pairs: 192 tiles, rows of A at whole lines
    generate(2560, 3520, 1368);   // 256 x 256, slices one by one: 140 tiles
    generate(4096, 2560, 640);    // 128 x 128: rows at multiples of 16 bytes
    return 0;
}
