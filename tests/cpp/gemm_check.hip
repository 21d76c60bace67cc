// Check of launch_gemm (scess_amd/csrc/triples_adjoint.hip) against sums on the host: batches, K splits and both, for rows
// that are 16-byte aligned and rows that are not (they take different kernels). Run by tests/test_gemm_gpu.py.
#include "triples_internal.h"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

using namespace scess;

static void hip(hipError_t e, const char *what) {
    if (e != hipSuccess) {
        std::printf("%s: %s\n", what, hipGetErrorString(e));
        std::exit(1);
    }
}

static double *device(const std::vector<double> &h) {
    double *d = nullptr;
    hip(hipMalloc((void **)&d, 8 * h.size()), "hipMalloc");
    hip(hipMemcpy(d, h.data(), 8 * h.size(), hipMemcpyHostToDevice), "hipMemcpy");
    return d;
}

// C[b][m][n] = c0 + alpha sum_k A[b][m][k1][k2] B[b][n][k1][k2]; rows of K2 elements `pitch` apart
static bool check(int prec, int batch, int splits, int M, int N, int K1, int K2, int pitch) {
    const int64_t ra = (int64_t)M * K1 * pitch, rb = (int64_t)N * K1 * pitch;
    uint64_t seed = 88172645463325252ull + (uint64_t)(batch * 131 + splits * 17 + M * 7 + N * 3 + K2);
    auto draw = [&]() {
        seed ^= seed << 13;
        seed ^= seed >> 7;
        seed ^= seed << 17;
        return (double)(int64_t)(seed >> 11) * 0x1p-52 - 1.0;
    };
    std::vector<double> A((size_t)(batch * ra)), B((size_t)(batch * rb)), C((size_t)batch * M * N);
    for (auto *x : {&A, &B, &C})
        for (auto &y : *x)
            y = draw();
    GemmArgs g{};
    g.M = M;
    g.N = N;
    g.alpha = -0.5;
    g.splits = splits;
    g.prec = prec;
    g.seg.K1 = K1;
    g.seg.K2 = K2;
    double *dA = device(A), *dB = device(B), *dC = device(C);
    double *scratch = device(std::vector<double>((size_t)splits * batch * M * N, NAN));
    g.seg.A = {dA, (int64_t)K1 * pitch, pitch, 1, ra};
    g.seg.B = {dB, (int64_t)K1 * pitch, pitch, 1, rb};
    g.C = dC;
    g.sCm = N;
    g.sCn = 1;
    g.sCb = (int64_t)M * N;
    g.scratch = scratch;
    hip(launch_gemm(g, batch, nullptr), "launch_gemm");
    std::vector<double> out(C.size());
    hip(hipMemcpy(out.data(), dC, 8 * out.size(), hipMemcpyDeviceToHost), "hipMemcpy");
    for (double *p : {dA, dB, dC, scratch})
        hip(hipFree(p), "hipFree");
    // FP64: K + 2 roundings of partial sums on each side; FP32: two rounded inputs and sums of 16 products in FP32
    const double unit = prec == P64 ? 2.0 * (K1 * K2 + 2) * 0x1p-53 : 18.0 * 0x1p-24;
    double worst = 0.0;
    for (int b = 0; b < batch; b++)
        for (int m = 0; m < M; m++)
            for (int n = 0; n < N; n++) {
                double s = 0.0, t = std::fabs(C[((size_t)b * M + m) * N + n]);
                for (int k1 = 0; k1 < K1; k1++)
                    for (int k = 0; k < K2; k++) {
                        const double p = A[(size_t)(b * ra + ((int64_t)m * K1 + k1) * pitch + k)] *
                                         B[(size_t)(b * rb + ((int64_t)n * K1 + k1) * pitch + k)];
                        s += p;
                        t += std::fabs(p);
                    }
                const size_t at = ((size_t)b * M + m) * N + n;
                const double err = std::fabs(out[at] - (C[at] - 0.5 * s)) / (unit * t);
                worst = err <= worst ? worst : err;  // NaN is kept
            }
    std::printf("prec %d batch %d splits %d M %d N %d K %d x %d pitch %d: %.3f of the bound\n", prec, batch, splits, M, N, K1,
                K2, pitch, worst);
    return worst <= 1.0;
}

int main() {
    bool ok = true;
    for (int prec : {(int)P64, (int)P32})
        for (int pitch : {36, 37})  // 16-byte aligned rows or not
            for (int batch : {1, 3})
                for (int splits : {1, 2, 5})
                    ok = check(prec, batch, splits, 70, 33, 3, 35, pitch) && ok;
    ok = check(P64, 4, 3, 130, 17, 5, 16, 16) && ok;
    std::printf(ok ? "all checks passed\n" : "failed\n");
    return ok ? 0 : 1;
}
