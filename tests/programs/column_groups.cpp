// NO_CPU_VARIANT (compared with float64 products)
// A product whose columns are groups of H and a point-wise nest that adds the groups of every unit: out[i, u] = sum_g sum_k A[i, k] W[k, g H + u].
// The back-end fuses the two where a tile holds all groups of whole units, four neighbouring ones at least (W is contiguous along its columns).
// One generated function per number of rows, units, groups and k: column_groups_<M>x<H>x<G>x<K>.
#include <tiramisu/tiramisu.h>

using namespace tiramisu;

static void generate(int M, int H, int G, int K)
{
    const std::string name = "column_groups_" + std::to_string(M) + "x" + std::to_string(H) + "x" + std::to_string(G) + "x" + std::to_string(K);
    tiramisu::init(name);

    var i("i", 0, M), n("n", 0, G * H), u("u", 0, H), k("k", 0, K);
    buffer buf_a("buf_a", {M, K}, p_float32, a_input);
    buffer buf_w("buf_w", {K, G * H}, p_float32, a_input);
    buffer buf_p("buf_p", {M, G * H}, p_float32, a_temporary);
    buffer buf_out("buf_out", {M, H}, p_float32, a_output);

    input a("a", {i, k}, p_float32);
    input w("w", {k, n}, p_float32);
    computation p_init("p_init", {i, n}, expr((float)0));
    computation p("p", {i, n, k}, p_float32);
    p.set_expression(p(i, n, 0) + a(i, k) * w(k, n));
    expr sum = p(i, u, 0);
    for (int g = 1; g < G; g++) sum = sum + p(i, u + g * H, 0);
    computation out("out", {i, u}, sum);

    a.store_in(&buf_a);
    w.store_in(&buf_w);
    p_init.store_in(&buf_p, {i, n});
    p.store_in(&buf_p, {i, n});
    out.store_in(&buf_out);
    for (buffer *q : {&buf_a, &buf_w, &buf_p, &buf_out}) q->tag_gpu_global();
    var ib("ib"), it("it"), nb("nb"), nt("nt"), ub("ub"), ut("ut");
    p_init.gpu_tile(i, n, 16, 16, ib, nb, it, nt);
    p.gpu_tile(i, n, 16, 16, ib, nb, it, nt);
    out.gpu_tile(i, u, 16, 16, ib, ub, it, ut);
    p_init.then(p, nt).then(out, computation::root);
    tiramisu::codegen({&buf_a, &buf_w, &buf_out}, "build/" + name + ".o", true);
}

int main(int argc, char **argv)
{
    tiramisu::backend_options_from_command_line(argc, argv);
    generate(64, 32, 16, 96);     // sixteen groups: four units of 64 columns, two of 32
    generate(64, 128, 4, 96);     // four: eight units of 32 columns
    return 0;
}
