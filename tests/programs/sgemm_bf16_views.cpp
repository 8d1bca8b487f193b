// NO_CPU_VARIANT (compared with float64 products)
// C = A * B + C on bf16 operands that are parts or other orders of their buffers: rows taken backwards (a negative leading
// dimension) and overlapping rows.  One function per form, sgemm_bf16_<form>.
#include <tiramisu/tiramisu.h>

using namespace tiramisu;

// element (i, k) of A at row ar * i + a0, element (k, j) of B at row br * k + b0, of buffers of a_rows x lda and b_rows x ldb
struct form {
    const char *name;
    int M, N, K, lda, ldb, ar, a0, br, b0;
};

static void generate(const form &o, bool overlapping = false)
{
    const std::string name = std::string("sgemm_bf16_") + o.name;
    tiramisu::init(name);
    var i("i", 0, o.M), j("j", 0, o.N), k("k", 0, o.K);
    buffer b_A("b_A", {o.M, o.lda}, p_bfloat16, a_input), b_B("b_B", {o.K, o.ldb}, p_bfloat16, a_input);
    buffer b_C("b_C", {o.M, o.N}, p_float32, a_output);
    input A("A", {var("i", 0, o.M), var("k", 0, o.lda)}, p_bfloat16), B("B", {var("k", 0, o.K), var("j", 0, o.ldb)}, p_bfloat16);
    A.store_in(&b_A);
    B.store_in(&b_B);

    computation acc_init("acc_init", {i, j}, expr((float)0)), acc("acc", {i, j, k}, p_float32), C("C", {i, j}, p_float32);
    const expr bk = expr(o.br) * k + expr(o.b0);
    acc.set_expression(acc(i, j, 0) + cast(p_float32, A(expr(o.ar) * i + expr(o.a0), k)) *
                       cast(p_float32, overlapping ? B(0, 2 * k + j) : B(bk, j)));
    C.set_expression(acc(i, j, 0) + C(i, j));
    C.store_in(&b_C);

    b_A.tag_gpu_global();
    b_B.tag_gpu_global();
    b_C.tag_gpu_global();
    buffer acc_reg("acc_reg", {1}, p_float32, a_temporary);
    acc_reg.tag_gpu_register();
    computation decl("decl", {i, j}, allocate(acc_reg));
    acc_init.store_in(&acc_reg, {0});
    acc.store_in(&acc_reg, {0});
    var ib("ib"), jb("jb"), it("it"), jt("jt");
    block({&decl, &acc_init, &acc, &C}).gpu_tile(i, j, 16, 16, ib, jb, it, jt);
    decl.then(acc_init, jt).then(acc, jt).then(C, jt);
    tiramisu::codegen({&b_A, &b_B, &b_C}, "build/" + name + ".o", true);
}

int main()
{
    // name, M, N, K, lda, ldb, row of A, row of B
    generate({"a_backwards", 200, 150, 100, 100, 150, -1, 199, 1, 0});
    generate({"b_backwards", 200, 150, 100, 100, 150, 1, 0, -1, 99});
    generate({"a_backwards_whole", 128, 192, 128, 128, 192, -1, 127, 1, 0});
    generate({"b_backwards_whole", 128, 192, 128, 128, 192, 1, 0, -1, 127});
    generate({"odd_k", 200, 150, 101, 102, 150, 1, 0, 1, 0});
    generate({"odd_n", 200, 149, 100, 100, 150, 1, 0, 1, 0});
    generate({"odd_k_and_n", 129, 257, 33, 36, 258, 1, 0, 1, 0});
    generate({"b_overlapping", 66, 30, 50, 50, 130, 1, 0, 0, 0}, true);
    return 0;
}
