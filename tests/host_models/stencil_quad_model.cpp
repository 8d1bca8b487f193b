// The values that a thread of kernels/stencil2d_regs.hip.h loads at the edges of a plane: st_load_quad, compiled here as plain C++ with
// loads that read memory, against the cells themselves.  Planes of every number of columns from 1 to 23, and quads that begin
// before, in and behind the plane.  Exit status 0 only when every value is right.  (tests/test_stencil_address_model.py)
#include <cstdio>
#include <cstring>
#include <vector>

struct model_index { unsigned x, y, z; };
static model_index threadIdx, blockIdx;
#define __global__
#define __device__
#define __forceinline__ inline
#define __launch_bounds__(n)
#define __shared__ static
static inline void __syncthreads() {}
static inline int __builtin_amdgcn_update_dpp(int, int v, int, int, int, bool) { return v; }

typedef float model_f4 __attribute__((vector_size(16)));
static const float *begin, *end;            // of the plane
static long outside = 0;
static float model_load1(const float *p) {
    if (p < begin || p >= end) { outside++; return 0.f; }
    return *p;
}
static model_f4 model_load4(const void *q) {
    const float *p = static_cast<const float *>(q);
    return model_f4{model_load1(p), model_load1(p + 1), model_load1(p + 2), model_load1(p + 3)};
}
#define ST_HOST_MODEL 1
#define ST_CONSTEXPR const
#define ST_STATIC_ASSERT(cond, text)
#define ST_SKIP_ARITHMETIC 1
#define ST_GLOBAL_LOAD4(p, stream) model_load4(p)
#define ST_GLOBAL_LOAD1(p) model_load1(p)
#define ST_GLOBAL_STORE4(p, v, stream) ((void)0)
#define ST_GLOBAL_STORE1(p, v) ((void)0)
// (one instance of the kernel: only what it loads with is called)
#define ST_NY 64
#define ST_NX 64
#define ST_Y0 1
#define ST_Y1 62
#define ST_X0 1
#define ST_X1 62
#define ST_GX 1
#define ST_GY 1
#define ST_IBX0 0
#define ST_IBX1 0
#define ST_IBY0 1
#define ST_IBY1 0
#define ST_R 1
#define ST_MODE 0
#define ST_W 8
#define ST_MERGE 1
#define ST_XCD 1
#define ST_OCC 0
#define ST_STREAM 2
#define ST_RAD 1
#define ST_EXPR ST_AT(0, 0)
#define ST_NAME model
#define ST_NAME_EDGE model_edge
#define ST_RPT 2
#define ST_RPT_EDGE 2
#include "../../tiramisu_amd/csrc/kernels/stencil2d_regs.hip.h"

int main() {
    long wrong = 0, quads = 0;
    for (int nx = 1; nx <= 23; nx++) {
        const int ny = 5;
        std::vector<float> plane(ny * nx);
        for (int i = 0; i < ny * nx; i++) plane[i] = 1.f + i;
        begin = plane.data();
        end = begin + plane.size();
        for (int gy = -2; gy < ny + 2; gy++)
            for (int gx = -8; gx < nx + 8; gx += 4) {
                const st_f4 v = st_load_quad<true>(plane.data(), gy, gx, ny, nx);
                const bool whole = gy >= 0 && gy < ny && gx >= 0 && gx + 3 < nx;
                const st_f4 u = whole ? st_load_quad<false>(plane.data(), gy, gx, ny, nx) : v;
                quads++;
                for (int e = 0; e < 4; e++) {
                    const bool in = gy >= 0 && gy < ny && gx + e >= 0 && gx + e < nx;
                    const float expected = in ? plane[gy * nx + gx + e] : 0.f;
                    if (v[e] != expected || u[e] != expected) {
                        if (wrong++ < 20) std::printf("FAIL plane %d x %d, quad (%d, %d), cell %d: %g, %g instead of %g\n", ny, nx, gy, gx, e, v[e], u[e], expected);
                    }
                }
            }
    }
    std::printf("%ld quads, %ld wrong value(s), %ld load(s) outside the plane\n", quads, wrong, outside);
    return wrong || outside ? 1 : 0;
}
