// Closed-shell CCSD residual engine on gfx950 (FP64).
//
// A device einsum engine with the semantics of the reference's compile-time
// Einsum (src/Tensor/TensorEinsum.h:9-17,137-205): labels shared by both
// operands and absent from the output are summed; labels of the output found
// in both operands are batch indices. Each contraction is evaluated as
// permute(A) -> [batch][M][K], permute(B) -> [batch][N][K], one FP64 MFMA GEMM
// (launch_gemm of triples_adjoint.hip), and a permuting accumulate into the
// output. On top of it, UpdateAmplitudes (src/Quantum/CC/RCCSD.cpp:101-237) is
// transcribed term by term; the particle-particle ladder sum_cd Wvvvv tau never
// forms a v^4 tensor when the Cholesky factor of (ac|bd) is given:
//   sum_cd (ac|bd) tau_ij^cd   from (ac|bd) tiles regenerated from L per (a,b) tile,
//   sum_cd (kd|ac) t_k^b tau_ij^cd and sum_cd (kc|bd) t_k^a tau_ij^cd
//                              through Z[k][a][i][j] = sum_cd (kd|ac) tau_ij^cd.
#include "ccsd_internal.h"

#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <string>

namespace scess {

// ------------------------------------------------------------------ kernels
constexpr int MAXD = 8;
struct PermArgs {
    int nd;
    int64_t odims[MAXD];   // output dims (row-major)
    int64_t istride[MAXD]; // input stride of each output dim
    const double *in;
    double *out;
    double alpha, beta;    // out = beta * out + alpha * in[perm]
    int64_t n;
    int64_t row, pitch;    // rows of `row` outputs start `pitch` apart (row 0: contiguous)
};

// Input offset of an output position: the output multi-index decomposed with 64-bit divisions. The
// loop runs over all MAXD dimensions, unrolled, with the ones past a.nd skipped, so the index lives in
// registers.
struct PermWalk {
    int64_t idx[MAXD];
    int64_t off;
    __device__ void init(const PermArgs &a, int64_t lin) {
        int64_t r = lin;
        off = 0;
#pragma unroll
        for (int d = MAXD - 1; d >= 0; d--) {
            idx[d] = 0;
            if (d >= a.nd)
                continue;
            idx[d] = r % a.odims[d];
            r /= a.odims[d];
            off += idx[d] * a.istride[d];
        }
    }
};

// One output per thread, so that the lanes of a wave store (and, with beta != 0, load) consecutive
// outputs: walking several consecutive outputs per thread saves index divisions but spreads every
// store instruction over 32-byte strides (a CCSD update spent about twice the time in permutes).
__global__ __launch_bounds__(256) void permute_kernel(PermArgs a) {
    const int64_t lin = element_id();
    if (lin >= a.n)
        return;
    PermWalk w;
    w.init(a, lin);
    const double x = a.alpha * a.in[w.off];
    const int64_t at = a.row ? lin / a.row * a.pitch + lin % a.row : lin;
    a.out[at] = a.beta == 0.0 ? x : a.beta * a.out[at] + x;
}

// Permute into pre-split BF16x3 rows: element (row, k) of the permuted operand (a.odims, flattened
// row * K + k) goes to row `row` of `out`, k padded to Kp (a multiple of 32) with zeros, as hi = bf16(x)
// and lo = bf16(x - hi) (round to nearest even) in groups of 8 k: 8 hi then 8 lo (32 bytes per group).
__device__ inline uint16_t bf16_rn(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// one thread per group of 8 k of one row (two 16-byte stores)
__global__ __launch_bounds__(256) void permute_split_kernel(PermArgs a, int64_t K, int64_t Kp, uint16_t *out,
                                                            int64_t nrows) {
    // one element per thread: the lanes of a wave read consecutive k of a row (walking eight k per thread and storing
    // 16-byte vectors spread each load over 64-byte strides: 1.2 times the time of a BF16x3 update's split permutes)
    const int64_t lin = element_id();
    if (lin >= nrows * Kp)
        return;
    const int64_t row = lin / Kp, k = lin - row * Kp;
    double x = 0.0;
    if (k < K) {
        PermWalk w;
        w.init(a, row * K + k);
        x = a.alpha * a.in[w.off];
    }
    const uint16_t hi = bf16_rn((float)x);
    const uint16_t lo = bf16_rn((float)(x - (double)__uint_as_float((uint32_t)hi << 16)));
    uint16_t *o = out + row * 2 * Kp + (k >> 3) * 16 + (k & 7);
    o[0] = hi;
    o[8] = lo;
}

// Packed operands of the FP64 particle-particle ladder (ladder_symmetric): over pairs c >= d (plus) and c > d (minus)
//   tau+_ij[cd] = (tau_ij^cd + tau_ij^dc) / 2 (tau_ij^cc for c = d), i >= j,   tau-_ij[cd] = (tau_ij^cd - tau_ij^dc) / 2, i > j
// at row i (i + 1) / 2 + j (i (i - 1) / 2 + j), column c (c + 1) / 2 + d (c (c - 1) / 2 + d). One work-group per (32 x 32
// tile pair, ij); the transposed tile goes through LDS.
__device__ inline int64_t tri(int64_t c) { return c * (c + 1) / 2; }

// plus[d <= c] and minus[d < c] of the v x v matrix x (row pitch ld) for its tile (tc, td), tc >= td: wx (x + x^T), with
// the diagonal wd x, and wx (x - x^T)
__device__ inline void pack_pair(const double *x, int64_t ld, int v, int tc, int td, double wx, double wd, double *plus,
                                 double *minus) {
    __shared__ double up[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8) {  // tile (td, tc), element (d, c)
        const int d = td * 32 + r, c = tc * 32 + tx;
        up[r][tx] = d < v && c < v ? x[d * ld + c] : 0.0;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int c = tc * 32 + r, d = td * 32 + tx;
        if (c >= v || d > c)
            continue;
        const double a = x[c * ld + d], b = up[tx][r];
        plus[tri(c) + d] = d == c ? wd * a : wx * (a + b);
        if (minus && d < c)
            minus[tri(c - 1) + d] = wx * (a - b);
    }
}

// tile pair number -> (tc, td), tc >= td
__device__ inline void tile_pair(int t, int &tc, int &td) {
    tc = (int)((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
    while (tri(tc + 1) <= t)
        tc++;
    while (tri(tc) > t)
        tc--;
    td = t - (int)tri(tc);
}

__global__ __launch_bounds__(256) void pack_tau_kernel(const double *tau, int o, int v, double *plus, int64_t lp,
                                                       double *minus, int64_t lm) {
    int tc, td, i, j;
    tile_pair(blockIdx.x, tc, td);
    tile_pair(blockIdx.y, i, j);
    pack_pair(tau + ((int64_t)i * o + j) * v * v, v, v, tc, td, 0.5, 1.0, plus + (tri(i) + j) * lp,
              i > j ? minus + (tri(i - 1) + j) * lm : nullptr);
}

// (ac|bd) +- (ad|bc) of one strip: I[(a - a0, c)][(b, d)] with nb values of b; row (a - a0) nb + b
__global__ __launch_bounds__(256) void pack_int_kernel(const double *I, int nb, int v, double *plus, int64_t lp,
                                                       double *minus, int64_t lm) {
    int tc, td;
    tile_pair(blockIdx.x, tc, td);
    const int64_t row = blockIdx.y, al = row / nb, b = row - al * nb;
    pack_pair(I + (al * v * nb + b) * v, (int64_t)nb * v, v, tc, td, 1.0, 1.0, plus + row * lp, minus + row * lm);
}

// R_ij^ab += R+ + R-, R_ji^ab += R+ - R- and R_ij^ba = R_ji^ab for a strip's rows (a, b <= a); one thread per (i >= j, row)
__global__ __launch_bounds__(256) void ladder_scatter_kernel(const double *rp, const double *rm, int a0, int nb, int rows,
                                                             int o, int v, double *R) {
    const int row = blockIdx.x * 256 + threadIdx.x;
    if (row >= rows)
        return;
    int i, j;
    tile_pair(blockIdx.y, i, j);
    const int al = row / nb, b = row - al * nb, a = a0 + al;
    if (b > a)
        return;
    const int64_t np = tri(o), nm = tri(o - 1), vv = (int64_t)v * v;
    const double p = rp[row * np + blockIdx.y], m = i > j ? rm[row * nm + tri(i - 1) + j] : 0.0;
    double *x = R + ((int64_t)i * o + j) * vv, *y = R + ((int64_t)j * o + i) * vv;
    const int64_t ab = (int64_t)a * v + b, ba = (int64_t)b * v + a;
    x[ab] += p + m;
    if (i != j)
        y[ab] += p - m;
    if (a != b) {
        x[ba] += p - m;
        if (i != j)
            y[ba] += p + m;
    }
}

// out[2 b] = max |t_ij^ab - t_ji^ba|, out[2 b + 1] = max |t_ij^ab| over the work of block b, as bit patterns (which order as
// the values, NaN above all); the (32 x 32 tile of a, b; pair i >= j) go round the blocks. Bound by one read of t; out is
// pinned host memory: one launch and no copy.
constexpr int kAsymBlocks = 1024;
__global__ __launch_bounds__(256) void pair_asymmetry_kernel(const double *t, int o, int v, int nt, unsigned long long *out) {
    __shared__ double ji[32][33];
    __shared__ unsigned long long best[2];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    if (threadIdx.x < 2)
        best[threadIdx.x] = 0;
    unsigned long long d = 0, m = 0;
    auto bits = [](double z) { return (unsigned long long)__double_as_longlong(fabs(z)); };
    const int64_t tiles = (int64_t)nt * nt, items = tri(o) * tiles;
    for (int64_t w = blockIdx.x; w < items; w += gridDim.x) {
        const int pair = (int)(w / tiles), tile = (int)(w - pair * tiles), ta = tile / nt, tb = tile - ta * nt;
        int i, j;
        tile_pair(pair, i, j);
        const double *x = t + ((int64_t)i * o + j) * v * v, *y = t + ((int64_t)j * o + i) * v * v;
        for (int r = ty; r < 32; r += 8) {
            const int b = tb * 32 + r, a = ta * 32 + tx;
            ji[r][tx] = a < v && b < v ? y[(int64_t)b * v + a] : 0.0;
        }
        __syncthreads();
        for (int r = ty; r < 32; r += 8) {
            const int a = ta * 32 + r, b = tb * 32 + tx;
            if (a < v && b < v) {
                const double p = x[(int64_t)a * v + b], q = ji[tx][r];
                d = max(d, bits(p - q));
                m = max(m, max(bits(p), bits(q)));
            }
        }
        __syncthreads();
    }
    __syncthreads();
    atomicMax(&best[0], d);
    atomicMax(&best[1], m);
    __syncthreads();
    if (threadIdx.x < 2)
        out[2 * blockIdx.x + threadIdx.x] = best[threadIdx.x];
}

// A whole einsum of a small system in one launch, straight from the operands: G lanes per output element, lane g
// summing k = g, g + G, ... (then a fixed xor tree). The operand offsets of up to KT values of the summed index are
// decomposed once per work-group into LDS. Bound by launches, not by the chip: the CCSD of a water-sized molecule is
// some 60 contractions of microseconds per iteration, which as permute, permute, zero fill, GEMM, permute with two
// allocations each took 39 ms for o=5, v=19 (11 iterations).
struct ContractArgs {
    int no, nk;                 // output and summed dimensions
    int od[MAXD], kd[MAXD];     // their extents, last fastest
    int64_t oa[MAXD], ob[MAXD], oc[MAXD];  // strides of the output dimensions in A, B (0 where absent) and C
    int64_t ka[MAXD], kb[MAXD];            // strides of the summed dimensions in A and B
    const double *A, *B;
    double *C;
    double alpha, beta;
    int n, K, glog;             // outputs, summed extent, log2 of G
};
constexpr int kContractTable = 2048;

__global__ __launch_bounds__(256) void contract_kernel(ContractArgs a) {
    __shared__ int ta[kContractTable], tb[kContractTable];
    const int G = 1 << a.glog, g = threadIdx.x & (G - 1);
    const int64_t out = (int64_t)blockIdx.x * (256 >> a.glog) + (threadIdx.x >> a.glog);
    const bool live = out < a.n;
    int64_t pa = 0, pb = 0, pc = 0;
    int r = live ? (int)out : 0;
    for (int d = a.no - 1; d >= 0; d--) {
        const int q = r / a.od[d], i = r - q * a.od[d];
        pa += i * a.oa[d];
        pb += i * a.ob[d];
        pc += i * a.oc[d];
        r = q;
    }
    double s = 0.0;
    for (int k0 = 0; k0 < a.K; k0 += kContractTable) {
        const int kn = min(a.K - k0, kContractTable);
        if (k0)
            __syncthreads();
        for (int k = threadIdx.x; k < kn; k += 256) {
            int q = k0 + k, xa = 0, xb = 0;  // the operands hold less than 2^31 elements here
            for (int d = a.nk - 1; d >= 0; d--) {
                const int t = q / a.kd[d], i = q - t * a.kd[d];
                xa += i * (int)a.ka[d];
                xb += i * (int)a.kb[d];
                q = t;
            }
            ta[k] = xa;
            tb[k] = xb;
        }
        __syncthreads();
#pragma unroll 8
        for (int k = g; k < kn; k += G)
            s += a.A[pa + ta[k]] * a.B[pb + tb[k]];
    }
    for (int m = G >> 1; m >= 1; m >>= 1)
        s += __shfl_xor(s, m, 64);
    if (live && g == 0)
        a.C[pc] = a.beta == 0.0 ? a.alpha * s : a.beta * a.C[pc] + a.alpha * s;
}

// out = alpha * x + beta * y (elementwise)
__global__ __launch_bounds__(256) void axpby_kernel(double *out, const double *x, const double *y, double alpha,
                                                    double beta, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n)
        out[i] = alpha * x[i] + (y ? beta * y[i] : 0.0);
}

// tau[i][j][a][b] = t2 + t1[i][a] t1[j][b]
__global__ __launch_bounds__(256) void tau_kernel(double *tau, const double *t2, const double *t1, int o, int v) {
    const int64_t n = (int64_t)o * o * v * v;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= n)
        return;
    const int b = (int)(idx % v);
    int64_t r = idx / v;
    const int a = (int)(r % v);
    r /= v;
    const int j = (int)(r % o), i = (int)(r / o);
    tau[idx] = t2[idx] + t1[(int64_t)i * v + a] * t1[(int64_t)j * v + b];
}

// t1 /= (e_i - e_a), t2 /= (e_i + e_j - e_a - e_b)   (RCCSD.cpp:235-236, :321-331)
__global__ __launch_bounds__(256) void jacobi_kernel(double *t1, double *t2, const double *e, int o, int v) {
    const int64_t n2 = (int64_t)o * o * v * v, n1 = (int64_t)o * v;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx < n2) {
        const int b = (int)(idx % v);
        int64_t r = idx / v;
        const int a = (int)(r % v);
        r /= v;
        const int j = (int)(r % o), i = (int)(r / o);
        t2[idx] /= (e[i] - e[o + a]) + (e[j] - e[o + b]);
    }
    if (idx < n1) {
        const int a = (int)(idx % v), i = (int)(idx / v);
        t1[idx] /= e[i] - e[o + a];
    }
}

// partial dot products, fixed order: part[block] = sum over the block's range
__device__ inline void dot_body(const double *x, const double *y, int64_t n, double *part) {
    __shared__ double rs[256], rc[256];
    const int64_t per = (n + gridDim.x - 1) / gridDim.x;
    const int64_t b0 = (int64_t)blockIdx.x * per, b1 = min(n, b0 + per);
    double s = 0.0, c = 0.0;
    for (int64_t t = b0 + threadIdx.x; t < b1; t += 256) {
        const double p = x[t] * y[t];
        const double u = s + p;
        if (fabs(s) >= fabs(p))
            c += (s - u) + p;
        else
            c += (p - u) + s;
        s = u;
    }
    rs[threadIdx.x] = s;
    rc[threadIdx.x] = c;
    __syncthreads();
    for (int m = 128; m > 0; m >>= 1) {
        if ((int)threadIdx.x < m) {
            const double a1 = rs[threadIdx.x], b1v = rs[threadIdx.x + m];
            const double ss = a1 + b1v, bp = ss - a1;
            rc[threadIdx.x] = rc[threadIdx.x] + rc[threadIdx.x + m] + ((a1 - (ss - bp)) + (b1v - bp));
            rs[threadIdx.x] = ss;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        part[blockIdx.x] = rs[0] + rc[0];
}

// dot_kernel of x with each of up to kMaxDots vectors y (blockIdx.y): the same ranges and order
constexpr int kDotBlocks = 256;
struct DotVecs {
    const double *y[Engine::kMaxDots];
};
__global__ __launch_bounds__(256) void dots_kernel(const double *x, DotVecs v, int64_t n, double *part) {
    dot_body(x, v.y[blockIdx.y], n, part + (int64_t)blockIdx.y * gridDim.x);
}

hipError_t ccsd_jacobi(double *t1, double *t2, const double *e, int o, int v, hipStream_t s) {
    const int64_t n = (int64_t)o * o * v * v;
    hipLaunchKernelGGL(jacobi_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, t1, t2, e, o, v);
    return hipGetLastError();
}

// ------------------------------------------------------------------- engine
DTensor::~DTensor() { release(); }

void DTensor::release() {
    if (p)
        home->put(p);
    p = nullptr;
}

DTensor::DTensor(DTensor &&o) noexcept : p(o.p), dims(std::move(o.dims)), home(o.home) { o.p = nullptr; }

DTensor &DTensor::operator=(DTensor &&o) noexcept {
    if (this != &o) {
        release();
        p = o.p;
        dims = std::move(o.dims);
        home = o.home;
        o.p = nullptr;
    }
    return *this;
}

int64_t DTensor::size() const {
    int64_t n = 1;
    for (auto d : dims)
        n *= d;
    return n;
}

static void check(hipError_t e, const char *what) {
    if (e != hipSuccess)
        throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

DTensor Engine::alloc(std::vector<int64_t> dims, bool zero) {
    DTensor t;
    t.dims = std::move(dims);
    t.home = blocks;
    const size_t bytes = sizeof(double) * (size_t)std::max<int64_t>(t.size(), 1);
    check(blocks->get((void **)&t.p, bytes, stream), "device allocation (CCSD tensor)");
    if (zero)
        check(hipMemsetAsync(t.p, 0, bytes, stream), "hipMemsetAsync");
    return t;
}

void Engine::upload(DTensor &t, const double *host) {
    check(copy_to_device(t.p, host, sizeof(double) * (size_t)t.size(), stream), "upload");
}

void Engine::download(const DTensor &t, double *host) {
    check(copy_to_host(host, t.p, sizeof(double) * (size_t)t.size(), stream), "download");
}

void Engine::copy(DTensor &dst, const DTensor &src) {
    check(hipMemcpyAsync(dst.p, src.p, sizeof(double) * (size_t)src.size(), hipMemcpyDeviceToDevice, stream), "copy");
}

void Engine::axpby(double *out, const double *x, const double *y, double alpha, double beta, int64_t n) {
    hipLaunchKernelGGL(axpby_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, out, x, y, alpha, beta, n);
    check(hipGetLastError(), "axpby");
}

// out (labels lo, row-major dims) = beta*out + alpha*in[permuted], in has labels li
static PermArgs perm_args(const std::string &li, const double *in, const std::vector<int64_t> &idims,
                          const std::string &lo, double *out, const std::vector<int64_t> &odims, double alpha,
                          double beta) {
    PermArgs a{};
    a.nd = (int)lo.size();
    if (a.nd > MAXD || (int)li.size() != a.nd)
        throw std::runtime_error("permute: rank");
    std::vector<int64_t> is(li.size());
    int64_t s = 1;
    for (int d = (int)li.size() - 1; d >= 0; d--) {
        is[d] = s;
        s *= idims[d];
    }
    a.n = 1;
    for (int d = 0; d < a.nd; d++) {
        const auto pos = li.find(lo[d]);
        if (pos == std::string::npos)
            throw std::runtime_error("permute: label " + std::string(1, lo[d]) + " missing");
        a.odims[d] = odims[d];
        a.istride[d] = is[pos];
        a.n *= odims[d];
    }
    a.in = in;
    a.out = out;
    a.alpha = alpha;
    a.beta = beta;
    return a;
}

void Engine::permute(const std::string &li, const double *in, const std::vector<int64_t> &idims,
                     const std::string &lo, double *out, const std::vector<int64_t> &odims, double alpha,
                     double beta, int64_t row, int64_t pitch) {
    PermArgs a = perm_args(li, in, idims, lo, out, odims, alpha, beta);
    if (a.n == 0)
        return;
    a.row = row == pitch ? 0 : row;
    a.pitch = pitch;
    hipLaunchKernelGGL(permute_kernel, element_grid(a.n), dim3(256), 0, stream, a);
    check(hipGetLastError(), "permute");
}

DTensor Engine::permute_split(const std::string &li, const double *in, const std::vector<int64_t> &idims,
                              const std::string &lo, const std::vector<int64_t> &odims, int64_t K) {
    const PermArgs a = perm_args(li, in, idims, lo, nullptr, odims, 1.0, 0.0);
    if (K < 1 || a.n % K)
        throw std::runtime_error("permute_split: K does not divide the operand");
    const int64_t Kp = (K + 31) / 32 * 32, nrows = a.n / K;
    DTensor out = alloc({nrows, Kp / 2});  // Kp bf16 pairs per row = Kp / 2 eight-byte slots
    if (nrows > 0) {
        hipLaunchKernelGGL(permute_split_kernel, element_grid(nrows * Kp), dim3(256), 0, stream, a,
                           K, Kp, (uint16_t *)out.p, nrows);
        check(hipGetLastError(), "permute_split");
    }
    return out;
}

static void parse_spec(const std::string &spec, std::string &la, std::string &lb, std::string &lc) {
    const auto arrow = spec.find("->");
    const auto comma = spec.find(',');
    if (arrow == std::string::npos)
        throw std::runtime_error("einsum: no ->");
    lc = spec.substr(arrow + 2);
    if (comma == std::string::npos || comma > arrow) {
        la = spec.substr(0, arrow);
        lb.clear();
    } else {
        la = spec.substr(0, comma);
        lb = spec.substr(comma + 1, arrow - comma - 1);
    }
}

// C = beta*C + alpha * einsum(spec, A, B)
void Engine::einsum(const std::string &spec, const DTensor &A, const DTensor *B, DTensor &C, double alpha,
                    double beta) {
    std::string la, lb, lc;
    parse_spec(spec, la, lb, lc);
    if (la.size() != A.dims.size() || lc.size() != C.dims.size() || (B && lb.size() != B->dims.size()))
        throw std::runtime_error("einsum " + spec + ": rank mismatch");
    auto dim_of = [&](char x) -> int64_t {
        auto p = la.find(x);
        if (p != std::string::npos)
            return A.dims[p];
        p = lb.find(x);
        if (B && p != std::string::npos)
            return B->dims[p];
        p = lc.find(x);
        return C.dims[p];
    };
    if (!B) {  // pure permutation
        permute(la, A.p, A.dims, lc, C.p, C.dims, alpha, beta);
        return;
    }
    std::string Lb, Lm, Ln, Lk;
    for (char x : lc) {
        const bool ina = la.find(x) != std::string::npos, inb = lb.find(x) != std::string::npos;
        if (ina && inb)
            Lb += x;
        else if (ina)
            Lm += x;
        else if (inb)
            Ln += x;
        else
            throw std::runtime_error("einsum " + spec + ": output label not in an operand");
    }
    for (char x : la) {
        const bool inb = lb.find(x) != std::string::npos, inc = lc.find(x) != std::string::npos;
        if (inb && !inc)
            Lk += x;
        else if (!inb && !inc)
            throw std::runtime_error("einsum " + spec + ": trace over a single operand is not supported");
    }
    for (char x : lb)
        if (la.find(x) == std::string::npos && lc.find(x) == std::string::npos)
            throw std::runtime_error("einsum " + spec + ": trace over a single operand is not supported");
    auto prod = [&](const std::string &ls) {
        int64_t n = 1;
        for (char x : ls)
            n *= dim_of(x);
        return n;
    };
    auto dims_of = [&](const std::string &ls) {
        std::vector<int64_t> d;
        for (char x : ls)
            d.push_back(dim_of(x));
        return d;
    };
    const int64_t nb = prod(Lb), M = prod(Lm), N = prod(Ln), K = prod(Lk);
    // Small FP64 contractions in one launch (contract_kernel). The line is where its products at some 0.5 TFLOP/s
    // cost what the GEMM path's extra launches do (about 40 us): 1 << 24 products. A longer sum than 16384 over few outputs
    // (Foo: o^2 of o v^2) fills only a few work-groups, where the GEMM splits it over the chip: an update at o=1, v=200 takes
    // 24.7 ms without that bound and 24.1 with it, o=2, v=150 9.0 / 8.6, o=10, v=100 6.2 / 6.0 (4096: 6.0, 65536: 6.0 but 9.0
    // at o=2, v=150; 1024 costs o=5, v=100 4.0 ms against 3.8).
    if (prec == P64 && K <= 16384 && nb * M * N * std::max<int64_t>(K, 1) <= (int64_t)1 << 24 &&
        A.size() < (int64_t)1 << 31 && B->size() < (int64_t)1 << 31) {
        contract(la, A, lb, *B, lc, Lk, C, alpha, beta);
        return;
    }
    if (M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff || nb > 65535)
        throw std::runtime_error("einsum " + spec + ": extent too large");
    auto splits_of = [&](int64_t batch, int64_t m, int64_t n, int64_t k, GemmArgs &g, DTensor &scr) {
        // few output tiles over a long K (e.g. Foo, the T1 terms): split K so that every CU has work; the partial
        // tiles are added in split order (deterministic)
        const int64_t e = prec == P64 ? 128 : 64, tiles = batch * ((m + e - 1) / e) * ((n + e - 1) / e);
        if (prec == P64 ? tiles < 512 && k >= 2048 : tiles < 256 && k >= 8192)
            g.splits = prec == P64 ? (int)std::min<int64_t>({1024 / tiles, k / 1024, 256})
                                   : (int)std::min<int64_t>({512 / tiles, k / 2048, 256});
        if (g.splits > 1) {
            scr = alloc({g.splits, batch, m, n});
            g.scratch = scr.p;
        } else {
            g.splits = 1;
        }
    };
    // A large FP64 operand whose last label is summed is read in place when its other labels are [K1][M] or
    // [Mo][K1][Mi] (runs of summed and free ones): rows of stride sr in K1 pieces of the last label, Mo as a batch. Only
    // the other operand is permuted. (At o=20, v=200 a permute of the 1.28 GB (kd|ac) costs 0.7-1.8 ms, the GEMM 0.4.)
    if (prec == P64 && nb == 1 && M > 0 && N > 0 && K > 0) {
        auto in_place = [&](const std::string &l, const DTensor &T, const std::string &l2, const DTensor &T2,
                            const std::string &Ln2) -> bool {
            if (l.size() < 3 || Lk.find(l.back()) == std::string::npos || T.size() < T2.size() || T.size() < 1 << 20)
                return false;
            std::string part[3];  // Mo, K1, Mi
            size_t at = 0;
            for (size_t d = 0; d + 1 < l.size(); d++) {
                const bool sum = Lk.find(l[d]) != std::string::npos;
                if (sum && at == 0)
                    at = 1;
                else if (!sum && at == 1)
                    at = 2;
                else if (sum && at == 2)
                    return false;
                part[at] += l[d];
            }
            const int64_t k2 = T.dims.back(), mo = prod(part[0]), k1 = prod(part[1]), mi = prod(part[2]);
            if (part[1].empty() || part[2].empty() || k2 < 8 || k2 % 2 || mo > 65535 || (mo > 1 && mi < 96))
                return false;  // (a batch of few rows would leave most of a 128-row tile empty)
            const int64_t n = prod(Ln2);
            const std::string lo2 = Ln2 + part[1] + l.back(), lx = part[0] + part[2] + Ln2;
            DTensor P2, X, scr;
            const double *p2 = T2.p;
            if (l2 != lo2) {
                P2 = alloc({n, K});
                permute(l2, T2.p, T2.dims, lo2, P2.p, dims_of(lo2), 1.0, 0.0);
                p2 = P2.p;
            }
            const bool direct = lc == lx && (beta == 0.0 || beta == 1.0);
            if (!direct)
                X = alloc({mo, mi, n});
            GemmArgs g{};
            g.M = (int)mi;
            g.N = (int)n;
            g.alpha = direct ? alpha : 1.0;
            g.ow = !direct || beta == 0.0;
            g.splits = 1;
            g.seg.K1 = (int)k1;
            g.seg.K2 = (int)k2;
            g.seg.A = {T.p, k2, mi * k2, 1, k1 * mi * k2};
            g.seg.B = {p2, K, k2, 1, 0};
            g.C = direct ? C.p : X.p;
            g.sCm = n;
            g.sCn = 1;
            g.sCb = mi * n;
            splits_of(mo, mi, n, K, g, scr);
            check(launch_gemm(g, (int)mo, stream), "einsum gemm");
            if (!direct)
                permute(lx, X.p, dims_of(lx), lc, C.p, C.dims, alpha, beta);
            return true;
        };
        if (in_place(la, A, lb, *B, Ln) || in_place(lb, *B, la, A, Lm))
            return;
    }
    // operands in [batch][M][K] and [batch][N][K]: FP64 rows of an even pitch (16-byte aligned), or (BF16x3 products)
    // pre-split rows of Ks = Kp / 2 eight-byte slots, written by the permute itself. An FP64 operand that has such
    // rows already is used as it is, with its own order of the free labels; of the orders of the summed labels, the one
    // in which more of it is.
    const bool split = prec == PB3 && M > 0 && N > 0 && K > 0;
    const int64_t Ks = split ? (K + 31) / 32 * 16 : prec == P64 ? (K + 1) / 2 * 2 : K;
    if (prec == P64 && Ks == K) {
        auto free_order = [&](const std::string &l, const std::string &Lf) {  // Lf in the order of l, if the batch leads
            std::string f;
            for (char x : l)
                if (Lf.find(x) != std::string::npos)
                    f += x;
            return f;
        };
        std::string Lk2;
        for (char x : lb)
            if (Lk.find(x) != std::string::npos)
                Lk2 += x;
        const std::string Lm2 = free_order(la, Lm), Ln2 = free_order(lb, Ln);
        const auto as_is = [&](const std::string &lk) {
            return (la == Lb + Lm2 + lk ? A.size() : 0) + (lb == Lb + Ln2 + lk ? B->size() : 0);
        };
        if (as_is(Lk2) > as_is(Lk))
            Lk = Lk2;
        // (another order of C's labels costs a permute of C, at most the operand's)
        if (la == Lb + Lm2 + Lk && (Lm2 == Lm || A.size() >= C.size()))
            Lm = Lm2;
        if (lb == Lb + Ln2 + Lk && (Ln2 == Ln || B->size() >= C.size()))
            Ln = Ln2;
    }
    // the GEMM writes (or adds to) C itself where C has the order [batch][M][N]
    const bool direct = lc == Lb + Lm + Ln && M > 0 && N > 0 && K > 0 && (beta == 0.0 || beta == 1.0);
    DTensor Ap, Bp, Cp;
    const double *pA = A.p, *pB = B->p;
    if (!direct)
        Cp = alloc({nb, M, N}, K == 0);
    if (split) {
        Ap = permute_split(la, A.p, A.dims, Lb + Lm + Lk, dims_of(Lb + Lm + Lk), K);
        Bp = permute_split(lb, B->p, B->dims, Lb + Ln + Lk, dims_of(Lb + Ln + Lk), K);
        pA = Ap.p;
        pB = Bp.p;
    } else {
        if (la != Lb + Lm + Lk || Ks != K) {
            Ap = alloc({nb, M, Ks});
            permute(la, A.p, A.dims, Lb + Lm + Lk, Ap.p, dims_of(Lb + Lm + Lk), 1.0, 0.0, K, Ks);
            pA = Ap.p;
        }
        if (lb != Lb + Ln + Lk || Ks != K) {
            Bp = alloc({nb, N, Ks});
            permute(lb, B->p, B->dims, Lb + Ln + Lk, Bp.p, dims_of(Lb + Ln + Lk), 1.0, 0.0, K, Ks);
            pB = Bp.p;
        }
    }
    if (M > 0 && N > 0 && K > 0) {
        GemmArgs g{};
        g.M = (int)M;
        g.N = (int)N;
        g.alpha = direct ? alpha : 1.0;
        g.ow = !direct || beta == 0.0;
        g.splits = 1;
        g.seg.K1 = 1;
        g.seg.K2 = (int)(split ? Ks : K);
        g.seg.A = {pA, Ks, 0, 1, M * Ks};
        g.seg.B = {pB, Ks, 0, 1, N * Ks};
        g.C = direct ? C.p : Cp.p;
        g.sCm = N;
        g.sCn = 1;
        g.sCb = M * N;
        g.prec = split ? PB3S : prec;
        DTensor scr;
        if (nb == 1)
            splits_of(1, M, N, K, g, scr);
        check(launch_gemm(g, (int)nb, stream), "einsum gemm");
    }
    if (!direct)
        permute(Lb + Lm + Ln, Cp.p, dims_of(Lb + Lm + Ln), lc, C.p, C.dims, alpha, beta);
}

// C = beta C + alpha sum over the labels lk of A B, by contract_kernel
void Engine::contract(const std::string &la, const DTensor &A, const std::string &lb, const DTensor &B,
                      const std::string &lc, const std::string &lk, DTensor &C, double alpha, double beta) {
    if (lc.size() > MAXD || lk.size() > MAXD)
        throw std::runtime_error("contract: rank");
    auto stride = [](const std::string &l, const DTensor &t, char x) -> int64_t {
        const auto p = l.find(x);
        if (p == std::string::npos)
            return 0;
        int64_t s = 1;
        for (size_t d = p + 1; d < t.dims.size(); d++)
            s *= t.dims[d];
        return s;
    };
    ContractArgs a{};
    a.no = (int)lc.size();
    a.nk = (int)lk.size();
    a.n = 1;
    a.K = 1;
    for (int d = 0; d < a.no; d++) {
        a.od[d] = (int)C.dims[d];
        a.n *= a.od[d];
        a.oa[d] = stride(la, A, lc[d]);
        a.ob[d] = stride(lb, B, lc[d]);
        a.oc[d] = stride(lc, C, lc[d]);
    }
    for (int d = 0; d < a.nk; d++) {
        a.kd[d] = (int)A.dims[la.find(lk[d])];
        a.K *= a.kd[d];
        a.ka[d] = stride(la, A, lk[d]);
        a.kb[d] = stride(lb, B, lk[d]);
    }
    if (a.n == 0)
        return;
    a.A = A.p;
    a.B = B.p;
    a.C = C.p;
    a.alpha = alpha;
    a.beta = beta;
    // lanes per output: up to 64, while a lane keeps 16 terms or more and the launch fewer than 2^18 lanes
    while (a.glog < 6 && (a.K >> a.glog) >= 32 && ((int64_t)a.n << a.glog) < (1 << 17))
        a.glog++;
    const int64_t per = 256 >> a.glog, blocks = (a.n + per - 1) / per;
    hipLaunchKernelGGL(contract_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, a);
    check(hipGetLastError(), "contract");
}

void Engine::dots(const double *x, const double *const *y, int m, int64_t n, double *out) {
    if (m < 1 || m > kMaxDots)
        throw std::runtime_error("dots: count");
    if (!dotbuf)
        check(hipMalloc((void **)&dotbuf, sizeof(double) * kDotBlocks * kMaxDots), "hipMalloc dot");
    DotVecs v{};
    for (int q = 0; q < m; q++)
        v.y[q] = y[q];
    hipLaunchKernelGGL(dots_kernel, dim3(kDotBlocks, m), dim3(256), 0, stream, x, v, n, dotbuf);
    check(hipGetLastError(), "dot");
    double h[kDotBlocks * kMaxDots];
    check(hipMemcpyAsync(h, dotbuf, sizeof(double) * kDotBlocks * m, hipMemcpyDeviceToHost, stream), "dot copy");
    check(hipStreamSynchronize(stream), "dot sync");
    for (int q = 0; q < m; q++) {
        double s = 0.0, c = 0.0;
        for (int i = 0; i < kDotBlocks; i++) {
            const double z = h[q * kDotBlocks + i], u = s + z;
            if (std::fabs(s) >= std::fabs(z))
                c += (s - u) + z;
            else
                c += (z - u) + s;
            s = u;
        }
        out[q] = s + c;
    }
}

double Engine::dot(const double *x, const double *y, int64_t n) {
    double r;
    dots(x, &y, 1, n, &r);
    return r;
}

Engine::~Engine() {
    if (dotbuf)
        (void)hipFree(dotbuf);
    if (asym)
        (void)hipHostFree(asym);
    if (asym_done)
        (void)hipEventDestroy(asym_done);
}

// ------------------------------------------------------------- CCSD update
void CcsdState::make_tau(Engine &E, const DTensor &t1, const DTensor &t2, DTensor &tau) {
    const int64_t n = t2.size();
    hipLaunchKernelGGL(tau_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, E.stream, tau.p, t2.p, t1.p, o, v);
    check(hipGetLastError(), "tau");
}

// R += X_ij^ab + X_ji^ba (scaled)
static void plus_transpose_add(Engine &E, DTensor &R, const DTensor &X, double alpha) {
    E.permute("ijab", X.p, X.dims, "ijab", R.p, R.dims, alpha, 1.0);
    E.permute("jiba", X.p, X.dims, "ijab", R.p, R.dims, alpha, 1.0);
}

void Engine::pair_check(const DTensor &t) {
    const int64_t o = t.dims[0], v = t.dims[2], nt = (v + 31) / 32;
    if (!asym) {
        check(hipEventCreateWithFlags(&asym_done, hipEventDisableTiming), "hipEventCreate");
        check(hipHostMalloc((void **)&asym, sizeof(double) * 2 * kAsymBlocks, hipHostMallocDefault), "hipHostMalloc");
    }
    asym_blocks = (int)std::min<int64_t>(o * (o + 1) / 2 * nt * nt, kAsymBlocks);
    hipLaunchKernelGGL(pair_asymmetry_kernel, dim3((unsigned)asym_blocks), dim3(256), 0, stream, t.p, (int)o, (int)v, (int)nt,
                       (unsigned long long *)asym);
    check(hipGetLastError(), "symmetry of t2");
    check(hipEventRecord(asym_done, stream), "hipEventRecord");
}

// well above what rounding leaves in the amplitudes of an update (o=5, v=24 to o=16, v=157: 2e-16, FP32 2e-8, BF16x3 5e-8
// of the largest), below the error of the products themselves
static double pair_tolerance(int prec) { return prec == P64 ? 1e-11 : prec == P32 ? 1e-6 : 1e-5; }

bool Engine::pair_symmetric() {
    check(hipEventSynchronize(asym_done), "symmetry of t2");
    double d = 0.0, m = 0.0;
    for (int b = 0; b < asym_blocks; b++) {
        d = asym[2 * b] <= d ? d : asym[2 * b];  // NaN is kept
        m = std::max(m, asym[2 * b + 1]);
    }
    return d <= pair_tolerance(prec) * m;
}

bool Engine::pair_symmetric(const double *t, int64_t o, int64_t v) const {
    double d = 0.0, m = 0.0;
    for (int64_t b = 0; b < v; b++)
        for (int64_t a = 0; a < v; a++)
            for (int64_t j = 0; j < o; j++)
                for (int64_t i = j; i < o; i++) {
                    const double p = t[i + o * (j + o * (a + v * b))], q = t[j + o * (i + o * (b + v * a))];
                    const double e = std::fabs(p - q);
                    d = e <= d ? d : e;  // NaN is kept
                    m = std::max(m, std::max(std::fabs(p), std::fabs(q)));
                }
    return d <= pair_tolerance(prec) * m;
}

// Particle-particle ladder sum_cd (ac|bd) tau_ij^cd from the Cholesky factor, (a,b) tiles of TAB x TAB
void CcsdState::ladder_from_factor(Engine &E, const DTensor &tau, DTensor &R) {
    // (a, b) tile edge: 64 fills the GEMM's 64-row tiles; smaller when one tile of integrals
    // (TAB^2 v^2 doubles) would pass 8 GiB
    int64_t TAB = 64;
    while (TAB > 16 && TAB * TAB * v * v * 8 > ((int64_t)8 << 30))
        TAB /= 2;
    const int64_t nP = naux;
    DTensor I = E.alloc({TAB, v, TAB, v});  // I[a][c][b][d] of one tile
    // BF16x3 products: the factor (rows (a, c), K = P), tau (rows (i, j, c), K = d) and each tile of I
    // (rows (a, c, b), K = d) in pre-split rows of Ps / Vs eight-byte slots
    const bool split = E.prec == PB3;
    const int64_t Ps = (nP + 31) / 32 * 16, Vs = (v + 31) / 32 * 16;
    DTensor Ls, taus;
    if (split) {
        Ls = E.permute_split("acP", Lvv.p, {v, v, nP}, "acP", {v, v, nP}, nP);
        taus = E.permute_split("ijcd", tau.p, {o, o, v, v}, "ijcd", {o, o, v, v}, v);
    }
    for (int64_t a0 = 0; a0 < v; a0 += TAB) {
        const int64_t ta = std::min(TAB, v - a0);
        for (int64_t b0 = 0; b0 < v; b0 += TAB) {
            const int64_t tb = std::min(TAB, v - b0);
            // I[(a,c)][(b,d)] = sum_P L[a][c][P] L[b][d][P]
            GemmArgs g{};
            g.M = (int)(ta * v);
            g.N = (int)(tb * v);
            g.alpha = 1.0;
            g.splits = 1;
            g.seg.K1 = 1;
            if (split) {
                g.seg.K2 = (int)Ps;
                g.seg.A = {Ls.p + a0 * v * Ps, Ps, 0, 1, 0};
                g.seg.B = {Ls.p + b0 * v * Ps, Ps, 0, 1, 0};
            } else {
                g.seg.K2 = (int)nP;
                g.seg.A = {Lvv.p + a0 * v * nP, nP, 0, 1, 0};  // rows (a, c), K = P contiguous
                g.seg.B = {Lvv.p + b0 * v * nP, nP, 0, 1, 0};
            }
            g.ow = 1;
            g.C = I.p;
            g.prec = split ? PB3S : E.prec;
            g.sCm = tb * v;
            g.sCn = 1;
            g.sCb = 0;
            check(launch_gemm(g, 1, E.stream), "ladder integrals");
            // R[i][j][a][b] += sum_{c,d} I[a][c][b][d] tau[i][j][c][d]; batch a, rows b, K = (c, d)
            GemmArgs h{};
            h.M = (int)tb;
            h.N = (int)(o * o);
            h.alpha = 1.0;
            h.splits = 1;
            h.seg.K1 = (int)v;
            DTensor Is;
            if (split) {  // I of this tile in pre-split rows (a, c, b), K = d
                Is = E.permute_split("acbd", I.p, {ta, v, tb, v}, "acbd", {ta, v, tb, v}, v);
                h.seg.K2 = (int)Vs;
                h.seg.A = {Is.p, Vs, tb * Vs, 1, v * tb * Vs};
                h.seg.B = {taus.p, v * Vs, Vs, 1, 0};
            } else {
                h.seg.K2 = (int)v;
                h.seg.A = {I.p, v, tb * v, 1, v * tb * v};
                h.seg.B = {tau.p, v * v, v, 1, 0};
            }
            h.prec = split ? PB3S : E.prec;
            h.C = R.p + a0 * v + b0;
            h.sCb = v;
            h.sCm = 1;
            h.sCn = v * v;
            check(launch_gemm(h, (int)ta, E.stream), "ladder contraction");
        }
    }
}

// The same ladder in FP64 at less than a third of the products. R_ij^ab = R_ji^ba (tau_ij^cd = tau_ji^dc), so only b <= a
// is regenerated and contracted, in strips of TA values of a; and with s+- = (ac|bd) +- (ad|bc) and tau+- (pack_tau_kernel)
//   R_ij^ab = sum_{c>=d} s+ tau+ + sum_{c>d} s- tau-,   R_ji^ab = the same with minus,
// so the sum over (c, d) and the pairs (i, j) halve: o^2 v^4 / 4 products for the contraction and naux v^4 / 2 for the
// integrals. Bound by the GEMMs' matrix pipes; the packing passes read a strip's integrals and write them once.
void CcsdState::ladder_symmetric(Engine &E, const DTensor &tau, DTensor &R) {
    const int64_t nP = naux, pp = v * (v + 1) / 2, pm = v * (v - 1) / 2, np = o * (o + 1) / 2, nm = o * (o - 1) / 2;
    const int64_t lp = (pp + 1) / 2 * 2, lm = std::max<int64_t>((pm + 1) / 2 * 2, 2);  // 16-byte rows
    // strips of at most 32 a and 512 MiB of integrals, of even width (their diagonal blocks are half wasted: 8 of 200 a
    // cost 52% of the full square, 32 cost 58%)
    const int64_t most = std::max<int64_t>(1, std::min<int64_t>(32, ((int64_t)512 << 20) / (8 * v * v * v)));
    const int64_t strips = (v + most - 1) / most;
    const int64_t TA = (v + strips - 1) / strips, nt = (v + 31) / 32;
    const unsigned tp = (unsigned)(nt * (nt + 1) / 2);
    DTensor tp_ = E.alloc({np, lp}), tm_ = E.alloc({std::max<int64_t>(nm, 1), lm});
    hipLaunchKernelGGL(pack_tau_kernel, dim3(tp, (unsigned)np), dim3(256), 0, E.stream, tau.p, (int)o, (int)v, tp_.p, lp,
                       tm_.p, lm);
    check(hipGetLastError(), "pack tau");
    DTensor I = E.alloc({TA, v, v, v}), sp = E.alloc({TA * v, lp}), sm = E.alloc({TA * v, lm});
    DTensor rp = E.alloc({TA * v, np}), rm = E.alloc({TA * v, std::max<int64_t>(nm, 1)});
    for (int64_t a0 = 0; a0 < v; a0 += TA) {
        const int64_t ta = std::min(TA, v - a0), nb = a0 + ta, rows = ta * nb;
        // I[(a,c)][(b,d)] = sum_P L[a][c][P] L[b][d][P], b < a0 + ta
        GemmArgs g{};
        g.M = (int)(ta * v);
        g.N = (int)(nb * v);
        g.alpha = 1.0;
        g.splits = 1;
        g.seg.K1 = 1;
        g.seg.K2 = (int)nP;
        g.seg.A = {Lvv.p + a0 * v * nP, nP, 0, 1, 0};
        g.seg.B = {Lvv.p, nP, 0, 1, 0};
        g.C = I.p;
        g.sCm = nb * v;
        g.sCn = 1;
        g.ow = 1;
        check(launch_gemm(g, 1, E.stream), "ladder integrals");
        hipLaunchKernelGGL(pack_int_kernel, dim3(tp, (unsigned)rows), dim3(256), 0, E.stream, I.p, (int)nb, (int)v, sp.p, lp,
                           sm.p, lm);
        check(hipGetLastError(), "pack integrals");
        auto contract = [&](const DTensor &S, const DTensor &T, int64_t ld, int64_t K, int64_t N, DTensor &out) {
            if (K < 1 || N < 1)
                return;
            GemmArgs h{};
            h.M = (int)rows;
            h.N = (int)N;
            h.alpha = 1.0;
            h.splits = 1;
            h.seg.K1 = 1;
            h.seg.K2 = (int)K;
            h.seg.A = {S.p, ld, 0, 1, 0};
            h.seg.B = {T.p, ld, 0, 1, 0};
            h.C = out.p;
            h.sCm = N;
            h.sCn = 1;
            h.ow = 1;
            const int64_t tiles = ((rows + 127) / 128) * ((N + 127) / 128);
            DTensor scr;
            if (tiles < 512 && K >= 2048) {  // two work-groups per CU
                h.splits = (int)std::max<int64_t>(1, std::min<int64_t>({1024 / tiles, K / 1024, 32}));
                if (h.splits > 1) {
                    scr = E.alloc({h.splits, rows, N});
                    h.scratch = scr.p;
                }
            }
            check(launch_gemm(h, 1, E.stream), "ladder contraction");
        };
        contract(sp, tp_, lp, pp, np, rp);
        contract(sm, tm_, lm, pm, nm, rm);
        if (pm == 0 && nm > 0)
            check(hipMemsetAsync(rm.p, 0, sizeof(double) * (size_t)rm.size(), E.stream), "memset R-");
        hipLaunchKernelGGL(ladder_scatter_kernel, dim3((unsigned)((rows + 255) / 256), (unsigned)np), dim3(256), 0, E.stream,
                           rp.p, rm.p, (int)a0, (int)nb, (int)rows, (int)o, (int)v, R.p);
        check(hipGetLastError(), "ladder scatter");
    }
}

void CcsdState::update(Engine &E, DTensor &t1, DTensor &t2, const std::function<bool()> &symmetric) {
    const int64_t O = o, Vv = v;
    DTensor tau = E.alloc({O, O, Vv, Vv});
    make_tau(E, t1, t2, tau);
    DTensor Foo = E.alloc({O, O}), Fvv = E.alloc({Vv, Vv}), Fov = E.alloc({O, Vv});
    E.einsum("kcld,ilcd->ki", L_ovov, &tau, Foo, 1.0, 0.0);
    E.einsum("kcld,klad->ac", L_ovov, &tau, Fvv, -1.0, 0.0);
    E.einsum("kcld,ld->kc", L_ovov, &t1, Fov, 1.0, 0.0);

    // -- T1 equation (RCCSD.cpp:117-138)
    DTensor t1n = E.alloc({O, Vv});
    E.einsum("ac,ic->ia", Fvv, &t1, t1n, 1.0, 0.0);
    E.einsum("ki,ka->ia", Foo, &t1, t1n, -1.0, 1.0);
    E.einsum("kc,kica->ia", Fov, &t2, t1n, 2.0, 1.0);
    E.einsum("kc,ikca->ia", Fov, &t2, t1n, -1.0, 1.0);
    {
        DTensor Fov_t1 = E.alloc({O, O});
        E.einsum("kc,ic->ki", Fov, &t1, Fov_t1, 1.0, 0.0);
        E.einsum("ki,ka->ia", Fov_t1, &t1, t1n, 1.0, 1.0);
    }
    E.einsum("kcai,kc->ia", ovvo, &t1, t1n, 2.0, 1.0);
    E.einsum("kiac,kc->ia", oovv, &t1, t1n, -1.0, 1.0);
    E.einsum("kdac,ikcd->ia", ovvv, &tau, t1n, 2.0, 1.0);
    E.einsum("kcad,ikcd->ia", ovvv, &tau, t1n, -1.0, 1.0);
    E.einsum("lcki,klac->ia", ovoo, &tau, t1n, -2.0, 1.0);
    E.einsum("kcli,klac->ia", ovoo, &tau, t1n, 1.0, 1.0);

    // -- T2 equation
    DTensor t2n = E.alloc({O, O, Vv, Vv});
    E.axpby(t2n.p, oovv_phys.p, t2driver.p, 1.0, 1.0, t2n.size());  // (no driver: a copy)
    {
        // tmp2(a,b,i,c) = -kibc,ka + (ia|cb); abic,jc->ijab, without forming the o v^3 tmp2:
        //   sum_c (ia|cb) t_j^c  and  -sum_k t_k^a sum_c (ki|bc) t_j^c
        DTensor X = E.alloc({O, O, Vv, Vv});
        E.einsum("iacb,jc->ijab", ovvv, &t1, X, 1.0, 0.0);
        DTensor M = E.alloc({O, O, Vv, O});  // M[k][i][b][j] = sum_c (ki|bc) t_j^c
        E.einsum("kibc,jc->kibj", oovv, &t1, M, 1.0, 0.0);
        E.einsum("kibj,ka->ijab", M, &t1, X, -1.0, 1.0);
        plus_transpose_add(E, t2n, X, 1.0);
    }
    {
        // tmp2(a,k,i,j) = kcai,jc + (ia|jk); akij,kb->ijab
        DTensor tmp = E.alloc({Vv, O, O, O});
        E.einsum("kcai,jc->akij", ovvo, &t1, tmp, 1.0, 0.0);
        E.einsum("iajk->akij", ovoo, nullptr, tmp, 1.0, 1.0);
        DTensor X = E.alloc({O, O, Vv, Vv});
        E.einsum("akij,kb->ijab", tmp, &t1, X, 1.0, 0.0);
        plus_transpose_add(E, t2n, X, -1.0);
    }

    DTensor Loo = E.alloc({O, O}), Lvv = E.alloc({Vv, Vv});
    E.copy(Loo, Foo);
    E.einsum("lcki,lc->ki", ovoo, &t1, Loo, 2.0, 1.0);
    E.einsum("kcli,lc->ki", ovoo, &t1, Loo, -1.0, 1.0);
    E.copy(Lvv, Fvv);
    E.einsum("kdac,kd->ac", ovvv, &t1, Lvv, 2.0, 1.0);
    E.einsum("kcad,kd->ac", ovvv, &t1, Lvv, -1.0, 1.0);

    {
        DTensor Woooo = E.alloc({O, O, O, O});
        E.copy(Woooo, oooo_phys);
        E.einsum("lcki,jc->klij", ovoo, &t1, Woooo, 1.0, 1.0);
        E.einsum("kclj,ic->klij", ovoo, &t1, Woooo, 1.0, 1.0);
        E.einsum("kcld,ijcd->klij", ovov, &tau, Woooo, 1.0, 1.0);
        E.einsum("klij,klab->ijab", Woooo, &tau, t2n, 1.0, 1.0);
    }
    // particle-particle ladder (RCCSD.cpp:177-180, :215-216)
    if (vvvv_phys.p) {
        DTensor Wvvvv = E.alloc({Vv, Vv, Vv, Vv});
        E.copy(Wvvvv, vvvv_phys);
        E.einsum("kdac,kb->abcd", ovvv, &t1, Wvvvv, -1.0, 1.0);
        E.einsum("kcbd,ka->abcd", ovvv, &t1, Wvvvv, -1.0, 1.0);
        E.einsum("abcd,ijcd->ijab", Wvvvv, &tau, t2n, 1.0, 1.0);
    } else {
        const bool sym = symmetric();  // tau_ij^cd = tau_ji^dc
        if (sym && E.prec == P64 && O * (O + 1) / 2 <= 65535)  // (pairs are a grid dimension)
            ladder_symmetric(E, tau, t2n);
        else  // (the other precisions keep their rounding: packing would split and round other values)
            ladder_from_factor(E, tau, t2n);
        DTensor Z = E.alloc({O, Vv, O, O});  // Z[k][a][i][j] = sum_cd (kd|ac) tau_ij^cd
        E.einsum("kdac,ijcd->kaij", ovvv, &tau, Z, 1.0, 0.0);
        E.einsum("kaij,kb->ijab", Z, &t1, t2n, -1.0, 1.0);
        if (sym) {  // sum_cd (kc|bd) tau_ij^cd = Z[k][b][j][i]
            E.einsum("kbji,ka->ijab", Z, &t1, t2n, -1.0, 1.0);
        } else {
            E.einsum("kcbd,ijcd->kbij", ovvv, &tau, Z, 1.0, 0.0);
            E.einsum("kbij,ka->ijab", Z, &t1, t2n, -1.0, 1.0);
        }
    }
    {
        DTensor X = E.alloc({O, O, Vv, Vv});
        E.einsum("ac,ijcb->ijab", Lvv, &t2, X, 1.0, 0.0);
        plus_transpose_add(E, t2n, X, 1.0);
        E.einsum("ki,kjab->ijab", Loo, &t2, X, 1.0, 0.0);
        plus_transpose_add(E, t2n, X, -1.0);
    }

    // ring and exchange terms (RCCSD.cpp:182-211, :221-233)
    DTensor Wvoov = E.alloc({Vv, O, O, Vv}), Wvovo = E.alloc({Vv, O, Vv, O});
    E.einsum("kcai->akic", ovvo, nullptr, Wvoov, 1.0, 0.0);
    E.einsum("kcad,id->akic", ovvv, &t1, Wvoov, 1.0, 1.0);
    E.einsum("kcli,la->akic", ovoo, &t1, Wvoov, -1.0, 1.0);
    E.einsum("ldkc,ilda->akic", ovov, &t2, Wvoov, -0.5, 1.0);
    E.einsum("lckd,ilad->akic", ovov, &t2, Wvoov, -0.5, 1.0);
    E.einsum("ldkc,ilad->akic", ovov, &t2, Wvoov, 1.0, 1.0);
    {
        DTensor tmp = E.alloc({O, O, Vv, O});
        E.einsum("ldkc,id->lkci", ovov, &t1, tmp, 1.0, 0.0);
        E.einsum("lkci,la->akic", tmp, &t1, Wvoov, -1.0, 1.0);
    }
    E.einsum("kiac->akci", oovv, nullptr, Wvovo, 1.0, 0.0);
    E.einsum("kdac,id->akci", ovvv, &t1, Wvovo, 1.0, 1.0);
    E.einsum("lcki,la->akci", ovoo, &t1, Wvovo, -1.0, 1.0);
    E.einsum("lckd,ilda->akci", ovov, &t2, Wvovo, -0.5, 1.0);
    {
        DTensor tmp = E.alloc({O, Vv, O, O});
        E.einsum("lckd,id->lcki", ovov, &t1, tmp, 1.0, 0.0);
        E.einsum("lcki,la->akci", tmp, &t1, Wvovo, -1.0, 1.0);
    }
    {
        DTensor X = E.alloc({O, O, Vv, Vv});
        E.einsum("akic,kjcb->ijab", Wvoov, &t2, X, 2.0, 0.0);
        E.einsum("akci,kjcb->ijab", Wvovo, &t2, X, -1.0, 1.0);
        plus_transpose_add(E, t2n, X, 1.0);
        E.einsum("akic,kjbc->ijab", Wvoov, &t2, X, 1.0, 0.0);
        plus_transpose_add(E, t2n, X, -1.0);
        E.einsum("bkci,kjac->ijab", Wvovo, &t2, X, 1.0, 0.0);
        plus_transpose_add(E, t2n, X, -1.0);
    }

    // Jacobi update with FP64 denominators (RCCSD.cpp:235-236)
    const int64_t n = t2n.size();
    hipLaunchKernelGGL(jacobi_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, E.stream, t1n.p, t2n.p, e.p, o,
                       v);
    check(hipGetLastError(), "jacobi");
    t1 = std::move(t1n);
    t2 = std::move(t2n);
}

double CcsdState::energy(Engine &E, const DTensor &t1, const DTensor &t2) {
    // sum_ijab (2 <ij|ab> - <ij|ba>) tau_ij^ab (RCCSD.cpp:85-89) (+ F12 coupling :91-98)
    DTensor tau = E.alloc({o, o, v, v});
    make_tau(E, t1, t2, tau);
    double Ecorr = E.dot(L_oovv_phys.p, tau.p, tau.size());
    if (f12energy.p) {
        DTensor Le = E.alloc({o, o, v, v});
        E.permute("ijab", f12energy.p, f12energy.dims, "ijab", Le.p, Le.dims, 2.0, 0.0);
        E.permute("ijba", f12energy.p, f12energy.dims, "ijab", Le.p, Le.dims, -1.0, 1.0);
        Ecorr += E.dot(Le.p, t2.p, t2.size());
    }
    return Ecorr;
}

}  // namespace scess
