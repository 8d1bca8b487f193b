// NO_CPU_VARIANT (compared with the loops of the oracle)
// The LSTM program (tiramisu_amd/programs/lstm.cpp) with batches and hidden sizes that no tile divides, so that the two product
// terms of a cell meet inside a slice, or inside a 16-byte load.
#define main main_of_all_sizes
#include "../../tiramisu_amd/programs/lstm.cpp"
#undef main

int main()
{
    generate(2, 5, 33, 3);
    generate(1, 35, 18, 2);
    generate(2, 14, 129, 3);
    generate(3, 33, 160, 2);
    generate(1, 70, 288, 2);
    return 0;
}
