// NO_CPU_VARIANT (compared with float64 products)
// The bf16 sgemm program (tiramisu_amd/programs/sgemm_bf16.cpp) at sizes that end inside a tile, a slice and a 16-byte piece
// of the operands, for every tile that the back-end chooses among.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/sgemm_bf16.cpp"
#undef main

int main()
{
    generate(4002, 3998, 500);    // 256x256 tiles loaded straight into LDS; the last slice holds 20 of 32 k
    generate(2000, 1500, 1006);   // 128x128, rows 4 bytes off a 16-byte boundary, 14 k in the last slice
    generate(70, 66, 130);        // 64x64, 2 k in the last slice
    generate(66, 2, 6);           // less than one slice and one granule of B
    generate(2001, 1501, 1001);   // rows of an odd number of elements: 128x128 tiles through registers
    generate(65, 67, 193);        // 64x64 through registers, one k in the last slice
    generate(64, 65, 63);         // odd rows, a single partial slice
    generate(33, 3, 65);          // fewer than four columns
    generate(20480, 20480, 32);   // 256x256 tiles with one slice, three (fewer than the LDS ring has stages) and five
    generate(8192, 12288, 96);
    generate(8192, 8192, 160);
    generate(640, 704, 64);       // whole tiles, for the order of the instructions behind them
    return 0;
}
