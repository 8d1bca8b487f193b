// NO_CPU_VARIANT (compared with the loops of the oracle)
// The LSTM program (tiramisu_amd/programs/lstm.cpp) at sizes on both sides of the rule for tiles of recurrent cells.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/lstm.cpp"
#undef main

int main()
{
    generate(2, 33, 40, 5);       // a row in the second tiles, a remainder of k, columns a multiple of 8 only
    generate(3, 5, 24, 4);        // few rows, less than one slice of k
    generate(2, 9, 37, 3);        // columns that no tile of 32 holds whole units of: the cell update stays apart
    generate(1, 64, 384, 3);      // slices of 128, eight groups
    generate(2, 64, 512, 4);      // whole tiles, four groups
    generate(4, 64, 512, 5);      // two tiles for every compute unit: 64x32 as before
    return 0;
}
