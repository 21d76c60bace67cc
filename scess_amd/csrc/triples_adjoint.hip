// gfx950 kernels of the (T) adjoint: dE(T)/d(ovvv), d(ovoo), d(ovov), dt1, dt2.
//
// E = sum_ijk w_ijk sum_abc W r3(Y)/D with Y = W + V and w_ijk = 2/deg_ijk. Since
// r3 is symmetric,  G_W = dE/dW = w (r3(Y)/D + r3(W/D))  and  G_V = dE/dV = w r3(W/D).
// W is recomputed per ijk (the forward W-build), G is formed by an orbit kernel
// like the forward epilogue, and the six permutation terms
//   w(x,y,z; p,q,r) = sum_f X[p][x][y][f] T[r][q][z][f] + sum_m Rn[p][q][x][m] TM[r][y][z][m]
// are back-contracted on the FP64 MFMAs (back_kernel):
//   dX[p][x][y][f]  += sum_z     G(x,y,z) T[r][q][z][f]
//   dT[r][q][z][f]  += sum_{x,y} G(x,y,z) X[p][x][y][f]
//   dRn[p][q][x][m] += sum_{y,z} G(x,y,z) TM[r][y][z][m]
//   dTM[r][y][z][m] += sum_x     Rn[p][q][x][m] G(x,y,z)
// Occupied triples are processed in batches and every kernel writes each output
// element from one thread in a fixed order (partials are summed in order), so the
// gradients are deterministic.
#include "triples_internal.h"

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <vector>
#include <cstdlib>

namespace scess {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

__device__ inline void nadd_a(double &s, double &c, double x) {
    const double t = s + x;
    if (fabs(s) >= fabs(x))
        c += (s - t) + x;
    else
        c += (x - t) + s;
    s = t;
}

// ------------------------------------------------------------------ G kernel
// Orbit geometry as in the forward epilogue (8-wide virtual blocks).
struct OrbitRowA {
    bool own;
    int ga, gb, gc0;
    int off[5], step[5];
};

template <int PB, int PX, int PY>
__device__ inline OrbitRowA orbit_row_a(const int *orbits, int orb, int tid) {
    constexpr int EB = 8;
    OrbitRowA r;
    const int A = orbits[3 * orb], B = orbits[3 * orb + 1], C = orbits[3 * orb + 2];
    const int bl1 = B != A ? B : C;
    auto slot = [&](int blk) { return blk == A ? 0 : (blk == bl1 ? 1 : 2); };
    const int sB = slot(B), sC = slot(C);
    uint64_t map_lo = 0, map_hi = 0;
    uint32_t seen = 0;
    int nd = 0;
    const int d = tid >> 6, ap = (tid >> 3) & 7, bp = tid & 7;
    int P = 0, Q = 0, R = 0, sP = 0, sQ = 0, sR = 0;
    auto add = [&](int p0, int p1, int p2, int s0, int s1, int s2) {
        const int key = s0 * 9 + s1 * 3 + s2;
        if (!(seen >> key & 1u)) {
            seen |= 1u << key;
            if (key < 21)
                map_lo |= (uint64_t)nd << (3 * key);
            else
                map_hi |= (uint64_t)nd << (3 * (key - 21));
            if (nd == d) {
                P = p0;
                Q = p1;
                R = p2;
                sP = s0;
                sQ = s1;
                sR = s2;
            }
            nd++;
        }
    };
    add(A, B, C, 0, sB, sC);
    add(B, C, A, sB, sC, 0);
    add(C, A, B, sC, 0, sB);
    add(C, B, A, sC, sB, 0);
    add(A, C, B, 0, sC, sB);
    add(B, A, C, sB, 0, sC);
    auto dindex = [&](int s0, int s1, int s2) -> int {
        const int key = s0 * 9 + s1 * 3 + s2;
        return (int)((key < 21 ? map_lo >> (3 * key) : map_hi >> (3 * (key - 21))) & 7u);
    };
    r.own = d < nd;
    r.ga = P * EB + ap;
    r.gb = Q * EB + bp;
    r.gc0 = R * EB;
    r.off[0] = dindex(sQ, sR, sP) * PB + bp * PX + ap;  // (b, c, a)
    r.step[0] = PY;
    r.off[1] = dindex(sR, sP, sQ) * PB + ap * PY + bp;  // (c, a, b)
    r.step[1] = PX;
    r.off[2] = dindex(sR, sQ, sP) * PB + bp * PY + ap;  // (c, b, a)
    r.step[2] = PX;
    r.off[3] = dindex(sP, sR, sQ) * PB + ap * PX + bp;  // (a, c, b)
    r.step[3] = PY;
    r.off[4] = dindex(sQ, sP, sR) * PB + bp * PX + ap * PY;  // (b, a, c)
    r.step[4] = 1;
    return r;
}

constexpr int GK_THREADS = 384;

// G_W and G_V (row-major [vR][vR][vR], FP64) of the occupied triple blockIdx.y, with the weight dE 2 / deg. Triples with
// two equal indices come as i == j: their G_W is symmetric in its first two indices and the six terms of the
// back-contractions pair up, so G_W is doubled and one term of each pair is left out (back_terms).
template <typename AccT>
__global__ __launch_bounds__(GK_THREADS) void adjoint_g_kernel(EpiArgs a, double dE, double *GW, double *GV) {
    constexpr int EB = 8;
    constexpr int PY = 9, PX = EB * PY + 1, PB = EB * PX;
    __shared__ double Yl[6 * PB];
    __shared__ double Zl[6 * PB];
    const int tid = threadIdx.x;
    const int orb = blockIdx.x;
    const int *q = a.ijk + 3 * blockIdx.y;
    const int i = q[0], j = q[1], k = q[2];
    const int v = a.v, vR = a.vR, nbR = a.vR >> 3;
    const int64_t vr = (int64_t)v * vR;
    const double eocc = a.e[i] + a.e[j] + a.e[k];
    const double *U = a.U + blockIdx.y * 3 * vr;
    const AccT *W1b = (const AccT *)a.W1 + blockIdx.y * a.wstride;
    const AccT *W2b = i == j ? W1b : (const AccT *)a.W2 + blockIdx.y * a.wstride;
    const double wgt = i == j ? dE : 2.0 * dE, wgtw = 2.0 * dE;
    GW += blockIdx.y * a.wstride;
    GV += blockIdx.y * a.wstride;
    const int ap = (tid >> 3) & 7, bp = tid & 7, d = tid >> 6;

    const OrbitRowA r = orbit_row_a<PB, PX, PY>(a.orbits, orb, tid);
    double Y0[EB], Z0[EB], D0[EB];
    const bool rowok = r.own && r.ga < v && r.gb < v;
    if (rowok) {
        const int P = r.ga >> 3, Q = r.gb >> 3, R = r.gc0 >> 3;
        const AccT *W1 = W1b + (((int64_t)P * nbR + Q) * nbR + R) * 512 + (r.ga & 7) * 64 + (r.gb & 7) * 8;
        const AccT *W2 = W2b + (((int64_t)Q * nbR + P) * nbR + R) * 512 + (r.gb & 7) * 64 + (r.ga & 7) * 8;
        const double u0 = U[(int64_t)r.ga * vR + r.gb];
        const double *u1 = U + vr + (int64_t)r.ga * vR + r.gc0;
        const double *u2 = U + 2 * vr + (int64_t)r.gb * vR + r.gc0;
        const double *tk = a.t1 + (int64_t)k * vR + r.gc0;
        const double ti = a.t1[(int64_t)i * vR + r.ga], tj = a.t1[(int64_t)j * vR + r.gb];
        const double eab = eocc - a.ev[r.ga] - a.ev[r.gb];
#pragma unroll
        for (int cp = 0; cp < EB; cp++) {
            const bool ok = r.gc0 + cp < v;
            const double w = (double)W1[cp] + (double)W2[cp];
            const double Dv = eab - a.ev[r.gc0 + cp];
            Y0[cp] = ok ? w + u0 * tk[cp] + u1[cp] * tj + u2[cp] * ti : 0.0;
            Z0[cp] = ok ? w / Dv : 0.0;
            D0[cp] = ok ? Dv : 1.0;
        }
    } else {
#pragma unroll
        for (int cp = 0; cp < EB; cp++) {
            Y0[cp] = Z0[cp] = 0.0;
            D0[cp] = 1.0;
        }
    }
    if (r.own)
#pragma unroll
        for (int cp = 0; cp < EB; cp++) {
            Yl[d * PB + ap * PX + bp * PY + cp] = Y0[cp];
            Zl[d * PB + ap * PX + bp * PY + cp] = Z0[cp];
        }
    __syncthreads();
    if (rowok) {
        double *gw = GW + ((int64_t)r.ga * vR + r.gb) * vR + r.gc0;
        double *gv = GV + ((int64_t)r.ga * vR + r.gb) * vR + r.gc0;
        double ow[EB], oz[EB];
#pragma unroll
        for (int cp = 0; cp < EB; cp++) {
            double y3 = 0.0, z3 = 0.0;
            if (r.gc0 + cp < v) {
                y3 = 4.0 * Y0[cp] + Yl[r.off[0] + cp * r.step[0]] + Yl[r.off[1] + cp * r.step[1]] -
                     2.0 * (Yl[r.off[2] + cp * r.step[2]] + Yl[r.off[3] + cp * r.step[3]] + Yl[r.off[4] + cp * r.step[4]]);
                z3 = 4.0 * Z0[cp] + Zl[r.off[0] + cp * r.step[0]] + Zl[r.off[1] + cp * r.step[1]] -
                     2.0 * (Zl[r.off[2] + cp * r.step[2]] + Zl[r.off[3] + cp * r.step[3]] + Zl[r.off[4] + cp * r.step[4]]);
            }
            ow[cp] = wgtw * (y3 / D0[cp] + z3);
            oz[cp] = wgt * z3;
        }
#pragma unroll
        for (int cp = 0; cp < EB; cp += 2) {
            *(d2 *)(gw + cp) = d2{ow[cp], ow[cp + 1]};
            *(d2 *)(gv + cp) = d2{oz[cp], oz[cp + 1]};
        }
    }
}

hipError_t launch_adjoint_g(int prec, const EpiArgs &a, double dE, double *GW, double *GV, int nbatch, hipStream_t s) {
    const dim3 grid((unsigned)a.norb, (unsigned)nbatch);
    if (prec == P64 || prec == PI8)  // both build W in FP64
        hipLaunchKernelGGL(adjoint_g_kernel<double>, grid, dim3(GK_THREADS), 0, s, a, dE, GW, GV);
    else
        hipLaunchKernelGGL(adjoint_g_kernel<float>, grid, dim3(GK_THREADS), 0, s, a, dE, GW, GV);
    return hipGetLastError();
}

// -------------------------------------------------------------------- GEMM
// C[b][m][n] += alpha sum_k1 sum_k2 A(m, k1, k2) B(n, k1, k2); with splits > 1, split p handles a fixed contiguous
// range of the 16-deep K chunks and writes its partial to scratch[p]; gemm_reduce_kernel adds them in split order.
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmArgs g) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)g.M * g.N)
        return;
    const int m = (int)(idx / g.N), n = (int)(idx - (int64_t)m * g.N);
    const int64_t mn = (int64_t)g.M * g.N * gridDim.y;
    const double *src = g.scratch + (int64_t)blockIdx.y * g.M * g.N + idx;
    double s = 0.0;
    int p = 0;
    for (; p + 8 <= g.splits; p += 8) {  // eight loads in flight, added in split order
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            x[u] = src[(int64_t)(p + u) * mn];
#pragma unroll
        for (int u = 0; u < 8; u++)
            s += x[u];
    }
    for (; p < g.splits; p++)
        s += src[(int64_t)p * mn];
    double *cp = g.C + (int64_t)blockIdx.y * g.sCb + (int64_t)m * g.sCm + (int64_t)n * g.sCn;
    *cp = g.ow ? g.alpha * s : *cp + g.alpha * s;
}

// ------------------------------------------- GEMM with K-contiguous operands
// The same contraction when A.s2 == B.s2 == 1 (the inner K index is the
// contiguous one, as the einsum engine lays its operands out) and even strides: rows are read as
// 16-byte vectors (two doubles of K), staged through registers into a double-buffered LDS ring
// with the rows' vectors XOR-permuted (conflict-free 16-lane fragment reads), and each of the 2x2
// waves holds BLK x BLK MFMA 16x16 blocks. K tails and rows past M / N are zero-filled.
typedef double d2v __attribute__((ext_vector_type(2)));

__device__ inline int kswz(int r) { return (r ^ (r >> 3)) & 7; }

typedef float f4v __attribute__((ext_vector_type(4)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));

__device__ inline short bf16_bits(float f) {  // round to nearest even
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (short)(u >> 16);
}
__device__ inline float bf16_value(short h) { return __uint_as_float(((uint32_t)(uint16_t)h) << 16); }

// DMA: operand chunks go from global memory straight into LDS (global_load_lds_dwordx4, each lane fetching
// the logical vector its swizzled LDS slot holds), as in the W-build; vectors reaching past K2 load the
// row's first vector instead and are rewritten (value or zero) after the chunk has landed.
// WIDE = 2 (direct-to-LDS only): tiles of BM rows by 2 BM columns, each wave BLK x 2 BLK blocks, so a
// wave issues twice the MFMAs per chunk for 1.5x the staged bytes.
template <int BLK, bool VEC, int PREC, bool DMA, int WIDE>
__global__ __launch_bounds__(256) void gemm_kc_kernel(GemmArgs g) {
    constexpr int BM = 2 * BLK * 16;   // tile rows
    constexpr int BN = BM * WIDE;      // tile columns
    constexpr int BLKN = BLK * WIDE;   // MFMA blocks per wave along n
    constexpr int RB = 128;            // bytes of one 16-double K chunk of a row
    constexpr int NV = BM * 8 / 256;   // 16-byte vectors per thread per operand per chunk (square tiles)
    static_assert(!DMA || (VEC && BM * RB % 4096 == 0), "direct-to-LDS loads need 16-byte vectors, whole KiB");
    static_assert(WIDE == 1 || (WIDE == 2 && DMA), "wide tiles use the direct-to-LDS loads");
    __shared__ __attribute__((aligned(1024))) char lds[2][(BM + BN) * RB];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane & 15, lq = lane >> 4;
    const int ntn = (g.N + BN - 1) / BN;
    // tiles of one (batch, split) on one XCD, so the tiles sharing an operand panel share its L2
    const int nx = gridDim.x, ny = gridDim.y;
    const int lin = xcd_remap(blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z), nx * ny * gridDim.z);
    const int bx = lin % nx, byz = lin / nx;
    const int tm = bx / ntn, tn = bx - tm * ntn;
    const int m0 = tm * BM, n0 = tn * BN;
    const int beta = byz % ny, split = byz / ny;

    const GemmSeg &sg = g.seg;
    const int nk = (sg.K2 + 15) / 16, total = sg.K1 * nk;
    const int c_begin = (int)((int64_t)total * split / g.splits), c_end = (int)((int64_t)total * (split + 1) / g.splits);

    d4 acc[BLK][BLKN];
#pragma unroll
    for (int x = 0; x < BLK; x++)
#pragma unroll
        for (int y = 0; y < BLKN; y++)
            acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
    // MFMA blocks of this wave wholly past M or N are skipped (wave-uniform)
    bool vm[BLK], vn[BLKN];
#pragma unroll
    for (int x = 0; x < BLK; x++)
        vm[x] = m0 + wm * BLK * 16 + x * 16 < g.M;
#pragma unroll
    for (int y = 0; y < BLKN; y++)
        vn[y] = n0 + wn * BLKN * 16 + y * 16 < g.N;

    // thread t loads vectors q = t + 256 u (u < NV) of the BM x 8 vector tile: row q / 8, vector q % 8
    d2v ra[NV], rb[NV];
    auto fetch = [&](int ch) {
        const int k1 = ch / nk, k0 = (ch - k1 * nk) * 16;
        const double *pa = sg.A.base + (int64_t)beta * sg.A.sb + (int64_t)k1 * sg.A.s1;
        const double *pb = sg.B.base + (int64_t)beta * sg.B.sb + (int64_t)k1 * sg.B.s1;
#pragma unroll
        for (int u = 0; u < NV; u++) {
            const int q = tid + 256 * u, row = q >> 3, k = k0 + 2 * (q & 7);
            const int gm = m0 + row, gn = n0 + row;
            d2v a = {0.0, 0.0}, b = {0.0, 0.0};
            if (gm < g.M) {
                const double *p = pa + (int64_t)gm * sg.A.sr + k;
                if (VEC && k + 1 < sg.K2) {
                    a = *(const d2v *)p;
                } else {
                    if (k < sg.K2)
                        a.x = p[0];
                    if (k + 1 < sg.K2)
                        a.y = p[1];
                }
            }
            if (gn < g.N) {
                const double *p = pb + (int64_t)gn * sg.B.sr + k;
                if (VEC && k + 1 < sg.K2) {
                    b = *(const d2v *)p;
                } else {
                    if (k < sg.K2)
                        b.x = p[0];
                    if (k + 1 < sg.K2)
                        b.y = p[1];
                }
            }
            ra[u] = a;
            rb[u] = b;
        }
    };
    auto stash = [&](int buf) {
        char *As = lds[buf], *Bs = As + BM * RB;
#pragma unroll
        for (int u = 0; u < NV; u++) {
            const int q = tid + 256 * u, row = q >> 3, vec = q & 7;
            *(d2v *)(As + row * RB + ((vec ^ kswz(row)) << 4)) = ra[u];
            *(d2v *)(Bs + row * RB + ((vec ^ kswz(row)) << 4)) = rb[u];
        }
    };

    auto compute = [&](int buf) {
        const char *As = lds[buf], *Bs = As + BM * RB;
        // lane (lr, lq) holds k = 4 lq .. 4 lq + 3 of its row: vectors 2 lq and 2 lq + 1
        if constexpr (PREC == P64) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                d2v af[BLK], bf[BLKN];
#pragma unroll
                for (int b = 0; b < BLK; b++) {
                    const int rowa = wm * BLK * 16 + b * 16 + lr;
                    af[b] = *(const d2v *)(As + rowa * RB + (((2 * lq + h) ^ kswz(rowa)) << 4));
                }
#pragma unroll
                for (int b = 0; b < BLKN; b++) {
                    const int rowb = wn * BLKN * 16 + b * 16 + lr;
                    bf[b] = *(const d2v *)(Bs + rowb * RB + (((2 * lq + h) ^ kswz(rowb)) << 4));
                }
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int x = 0; x < BLK; x++)
                        if (vm[x])
#pragma unroll
                            for (int y = 0; y < BLKN; y++)
                                if (vn[y])
                                    acc[x][y] =
                                        __builtin_amdgcn_mfma_f64_16x16x4f64(af[x][t], bf[y][t], acc[x][y], 0, 0, 0);
            }
        } else if constexpr (PREC == PB3S) {
            // a 16-slot chunk holds 32 k of pre-split rows: vector 2 lq = the hi bf16 of k = 8 lq .. 8 lq + 7,
            // vector 2 lq + 1 their lo bf16 (the 16x16x32 operand layout); hi*hi + hi*lo + lo*hi in FP32 per
            // chunk, added to the FP64 accumulators
            b8v ah[BLK], al[BLK], bh[BLKN], bl[BLKN];
#pragma unroll
            for (int b = 0; b < BLK; b++) {
                const int rowa = wm * BLK * 16 + b * 16 + lr;
                ah[b] = *(const b8v *)(As + rowa * RB + (((2 * lq) ^ kswz(rowa)) << 4));
                al[b] = *(const b8v *)(As + rowa * RB + (((2 * lq + 1) ^ kswz(rowa)) << 4));
            }
#pragma unroll
            for (int b = 0; b < BLKN; b++) {
                const int rowb = wn * BLKN * 16 + b * 16 + lr;
                bh[b] = *(const b8v *)(Bs + rowb * RB + (((2 * lq) ^ kswz(rowb)) << 4));
                bl[b] = *(const b8v *)(Bs + rowb * RB + (((2 * lq + 1) ^ kswz(rowb)) << 4));
            }
#pragma unroll
            for (int x = 0; x < BLK; x++)
#pragma unroll
                for (int y = 0; y < BLKN; y++) {
                    if (!vm[x] || !vn[y])
                        continue;
                    f4v c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[x], bh[y], f4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[x], bl[y], c, 0, 0, 0);
                    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[x], bh[y], c, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        acc[x][y][r] += (double)c[r];
                }
        } else {
            // the lane's 4 k values of each block row, rounded (FP32) or split (hi + lo BF16)
            f4v a32[BLK], b32[BLKN];
#pragma unroll
            for (int b = 0; b < BLK; b++) {
                const int rowa = wm * BLK * 16 + b * 16 + lr;
                const d2v a0 = *(const d2v *)(As + rowa * RB + (((2 * lq) ^ kswz(rowa)) << 4));
                const d2v a1 = *(const d2v *)(As + rowa * RB + (((2 * lq + 1) ^ kswz(rowa)) << 4));
                a32[b] = f4v{(float)a0.x, (float)a0.y, (float)a1.x, (float)a1.y};
            }
#pragma unroll
            for (int b = 0; b < BLKN; b++) {
                const int rowb = wn * BLKN * 16 + b * 16 + lr;
                const d2v b0 = *(const d2v *)(Bs + rowb * RB + (((2 * lq) ^ kswz(rowb)) << 4));
                const d2v b1 = *(const d2v *)(Bs + rowb * RB + (((2 * lq + 1) ^ kswz(rowb)) << 4));
                b32[b] = f4v{(float)b0.x, (float)b0.y, (float)b1.x, (float)b1.y};
            }
            f4v c32[BLK][BLKN];
#pragma unroll
            for (int x = 0; x < BLK; x++)
#pragma unroll
                for (int y = 0; y < BLKN; y++)
                    c32[x][y] = f4v{0.f, 0.f, 0.f, 0.f};
            if constexpr (PREC == P32) {
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int x = 0; x < BLK; x++)
                        if (vm[x])
#pragma unroll
                            for (int y = 0; y < BLKN; y++)
                                if (vn[y])
                                    c32[x][y] =
                                        __builtin_amdgcn_mfma_f32_16x16x4f32(a32[x][t], b32[y][t], c32[x][y], 0, 0, 0);
            } else {
                s4v ah[BLK], al[BLK], bh[BLKN], bl[BLKN];
#pragma unroll
                for (int b = 0; b < BLK; b++)
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        ah[b][t] = bf16_bits(a32[b][t]);
                        al[b][t] = bf16_bits(a32[b][t] - bf16_value(ah[b][t]));
                    }
#pragma unroll
                for (int b = 0; b < BLKN; b++)
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        bh[b][t] = bf16_bits(b32[b][t]);
                        bl[b][t] = bf16_bits(b32[b][t] - bf16_value(bh[b][t]));
                    }
#pragma unroll
                for (int x = 0; x < BLK; x++)
#pragma unroll
                    for (int y = 0; y < BLKN; y++) {
                        if (!vm[x] || !vn[y])
                            continue;
                        c32[x][y] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(al[x], bh[y], c32[x][y], 0, 0, 0);
                        c32[x][y] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah[x], bl[y], c32[x][y], 0, 0, 0);
                        c32[x][y] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah[x], bh[y], c32[x][y], 0, 0, 0);
                    }
            }
#pragma unroll
            for (int x = 0; x < BLK; x++)
#pragma unroll
                for (int y = 0; y < BLKN; y++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        acc[x][y][r] += (double)c32[x][y][r];
        }
    };

    int buf = 0;
    if constexpr (DMA) {
        constexpr int OPB = BM * RB, NIW = OPB / 4096, NIWB = BN * RB / 4096;  // A bytes; wave loads of A, B
        // this lane's DMA units: tile row and the first k (even) of the logical vector its LDS slot holds
        // (units 0 .. NIW-1 of A; the B units are the same for u < NIW and continue the rows past it)
        int lrow[NIWB], lk[NIWB];
#pragma unroll
        for (int u = 0; u < NIWB; u++) {
            const int qq = (wave * NIWB + u) * 64 + lane, r = qq >> 3;
            lrow[u] = r;
            lk[u] = 2 * ((qq & 7) ^ kswz(r));
        }
        int larow[NIW], lak[NIW];
#pragma unroll
        for (int u = 0; u < NIW; u++) {
            const int qq = (wave * NIW + u) * 64 + lane, r = qq >> 3;
            larow[u] = r;
            lak[u] = 2 * ((qq & 7) ^ kswz(r));
        }
        auto issue = [&](int ch, int st) {
            const int k1 = ch / nk, k0 = (ch - k1 * nk) * 16;
            const double *pa = sg.A.base + (int64_t)beta * sg.A.sb + (int64_t)k1 * sg.A.s1;
            const double *pb = sg.B.base + (int64_t)beta * sg.B.sb + (int64_t)k1 * sg.B.s1;
            char *base = lds[st];
#pragma unroll
            for (int u = 0; u < NIW; u++) {
                const int k = k0 + lak[u], kk = k + 1 < sg.K2 ? k : 0;  // inside the row, else its first vector
                const int gm = min(m0 + larow[u], g.M - 1);
                __builtin_amdgcn_global_load_lds((const void *)(pa + (int64_t)gm * sg.A.sr + kk),
                                                 (lds_void *)(base + (wave * NIW + u) * 1024), 16, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < NIWB; u++) {
                const int k = k0 + lk[u], kk = k + 1 < sg.K2 ? k : 0;
                const int gn = min(n0 + lrow[u], g.N - 1);
                __builtin_amdgcn_global_load_lds((const void *)(pb + (int64_t)gn * sg.B.sr + kk),
                                                 (lds_void *)(base + OPB + (wave * NIWB + u) * 1024), 16, 0, 0);
            }
        };
        // after the chunk has landed: the vectors reaching past K2 get (x[k], 0) or (0, 0)
        auto fixup = [&](int ch, int st) {
            const int k1 = ch / nk, k0 = (ch - k1 * nk) * 16;
            if (k0 + 16 <= sg.K2)
                return false;
            const double *pa = sg.A.base + (int64_t)beta * sg.A.sb + (int64_t)k1 * sg.A.s1;
            const double *pb = sg.B.base + (int64_t)beta * sg.B.sb + (int64_t)k1 * sg.B.s1;
            char *base = lds[st];
#pragma unroll
            for (int u = 0; u < NIW; u++) {
                const int k = k0 + lak[u];
                if (k + 1 < sg.K2)
                    continue;
                const int gm = min(m0 + larow[u], g.M - 1);
                *(d2v *)(base + (wave * NIW + u) * 1024 + lane * 16) =
                    d2v{k < sg.K2 ? pa[(int64_t)gm * sg.A.sr + k] : 0.0, 0.0};
            }
#pragma unroll
            for (int u = 0; u < NIWB; u++) {
                const int k = k0 + lk[u];
                if (k + 1 < sg.K2)
                    continue;
                const int gn = min(n0 + lrow[u], g.N - 1);
                *(d2v *)(base + OPB + (wave * NIWB + u) * 1024 + lane * 16) =
                    d2v{k < sg.K2 ? pb[(int64_t)gn * sg.B.sr + k] : 0.0, 0.0};
            }
            return true;  // wave-uniform: every lane of the block sees the same chunk
        };
        if (c_begin < c_end)
            issue(c_begin, 0);
        for (int ch = c_begin; ch < c_end; ch++) {
            wait_vm<0>();
            __syncthreads();  // chunk ch is in LDS; the other stage is free again
            if (fixup(ch, buf))
                __syncthreads();
            if (ch + 1 < c_end)
                issue(ch + 1, buf ^ 1);
            compute(buf);
            buf ^= 1;
        }
    } else {
        if (c_begin < c_end)
            fetch(c_begin);
        for (int ch = c_begin; ch < c_end; ch++) {
            stash(buf);
            __syncthreads();
            if (ch + 1 < c_end)
                fetch(ch + 1);
            compute(buf);
            buf ^= 1;
        }
    }

#pragma unroll
    for (int x = 0; x < BLK; x++)
#pragma unroll
        for (int y = 0; y < BLKN; y++) {
            const int n = n0 + wn * BLKN * 16 + y * 16 + lr;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                // output layout of the 16x16 MFMAs: row lq + 4 r (FP64), 4 lq + r (FP32 accumulators)
                const int m = m0 + wm * BLK * 16 + x * 16 + (PREC == P64 ? lq + 4 * r : 4 * lq + r);
                if (m < g.M && n < g.N) {
                    if (g.splits == 1) {
                        double *cp = g.C + (int64_t)beta * g.sCb + (int64_t)m * g.sCm + (int64_t)n * g.sCn;
                        *cp = g.ow ? g.alpha * acc[x][y][r] : *cp + g.alpha * acc[x][y][r];
                    } else {
                        g.scratch[(((int64_t)split * ny + beta) * g.M + m) * g.N + n] = acc[x][y][r];
                    }
                }
            }
        }
}

// ------------------------------------------- FP64 GEMM with K-contiguous operands
// The same contraction for one segment of FP64 products whose rows are 16-byte aligned. Four waves own the quadrants of
// a tile of up to 128 x 128, two work-groups fill a CU (64 KiB of LDS, 256 registers). The ceil(M / 16) blocks of the
// rows are dealt out evenly over ceil(M / 128) tiles and a tile's blocks over its two halves, the columns alike, so no
// tile or wave is nearly empty (N = 400: 7 + 6 + 6 + 6 blocks; the 64 x 128 tiles of gemm_kc_kernel ran 3.1 tiles as 4).
// The loop is that of the FP64 W-build: bound by the matrix pipes, fragments read one k-step (4 of a chunk's 16 k) ahead
// of their MFMAs, one barrier per chunk before its last step, after which the freed stage takes the loads of the chunk
// after the next; the last chunk of a row runs only the k-steps that exist, its k past K2 set to zero in registers.
template <int RB, int CB> struct GemmNT {
    // state shared with the kernel
    const GemmArgs &g;
    char *lds;
    int lane, wave, wr, wc, m0, n0, rb, cb, beta, split;
    uint32_t so[4];
    uint32_t oa[4], ob[4];
    const double *pa, *pb;   // operand rows m0, n0 at the next chunk to load
    int k2c, nk2, left;      // its place in the row, chunks of a row, chunks left to load

    static constexpr int OPB = 128 * 128;  // bytes of an operand's stage

    // the next chunk into stage st: returns its k-steps, with bit 3 set when the last is partly past K2 (the lane
    // offsets of its vectors were clamped into the row)
    __device__ inline int issue(int st) {
        char *base = lds + st * 2 * OPB;
        const int rem = k2c == nk2 - 1 ? g.seg.K2 - 16 * k2c : 16;
        const int last = (rem - 1) & ~1;  // first k of the last vector of the row
#pragma unroll
        for (int h = 0; h < 4; h++) {
            const int u = wave + 4 * h, hf = u >> 3, bl = (u >> 1) & 3;  // LDS rows 8 u .. 8 u + 7: block bl of half hf
            const int r = 8 * (u & 7) + (lane >> 3), k = min(2 * ((lane & 7) ^ kswz(r)), last);
            if (bl < (rb + 1 - hf) >> 1)
                __builtin_amdgcn_global_load_lds((const void *)((const char *)pa + oa[h] + 8 * k),
                                                 (lds_void *)(base + u * 1024), 16, 0, 0);
            if (bl < (cb + 1 - hf) >> 1)
                __builtin_amdgcn_global_load_lds((const void *)((const char *)pb + ob[h] + 8 * k),
                                                 (lds_void *)(base + OPB + u * 1024), 16, 0, 0);
        }
        pa += 16;
        pb += 16;
        if (++k2c == nk2) {
            k2c = 0;
            pa += g.seg.A.s1 - 16 * nk2;
            pb += g.seg.B.s1 - 16 * nk2;
        }
        left--;
        return (rem + 3) >> 2 | (rem & 3 ? 8 : 0);
    }

    __device__ inline void run(int total, int cur, int nxt) {
        d4 acc[RB][CB];
        double fr[2][RB], fc[2][CB];
#pragma unroll
        for (int x = 0; x < RB; x++)
#pragma unroll
            for (int y = 0; y < CB; y++)
                acc[x][y] = d4{};
        lds_char *qa, *qb;
        auto tiles = [&](int st) {
            qa = (lds_char *)lds + st * 2 * OPB + wr * (OPB / 2);
            qb = (lds_char *)lds + st * 2 * OPB + OPB + wc * (OPB / 2);
        };
        auto read = [&](auto tc, int buf) {
            constexpr int t = decltype(tc)::value;
#pragma unroll
            for (int x = 0; x < RB; x++)
                fr[buf][x] = *(lds_double *)(qa + so[t ^ x] + x * 2048);
#pragma unroll
            for (int y = 0; y < CB; y++)
                fc[buf][y] = *(lds_double *)(qb + so[t ^ y] + y * 2048);
        };
        auto row = [&](int buf, int x) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int y = 0; y < CB; y++)
                acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr[buf][x], fc[buf][y], acc[x][y], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        // a k-step, with the fragments of the next one (t) read into the other buffer after its first row
        auto step = [&](int buf, auto tc) {
            row(buf, 0);
            read(tc, buf ^ 1);
#pragma unroll
            for (int x = 1; x < RB; x++)
                row(buf, x);
        };
        auto move = [&]() {  // buffer 0 to buffer 1
#pragma unroll
            for (int x = 0; x < RB; x++)
                fr[1][x] = fr[0][x];
#pragma unroll
            for (int y = 0; y < CB; y++)
                fc[1][y] = fc[0][y];
        };
        using std::integral_constant;
        const int lq = lane >> 4, keep = g.seg.K2 & 3;
        wait_vm_lgkm0();
        __syncthreads();
        tiles(0);
        read(integral_constant<int, 0>{}, 0);
        for (int c = 0; c < total; c++) {
            // all k-steps of chunk c but its last, whose fragments end up in buffer 1
            const int steps = cur & 7;
            if (steps >= 2) {
                step(0, integral_constant<int, 1>{});
                if (steps >= 3) {
                    step(1, integral_constant<int, 2>{});
                    if (steps == 4)
                        step(0, integral_constant<int, 3>{});
                    else
                        move();
                }
            } else {
                move();
            }
            const bool more = c + 1 < total;
            if (more) {
                // chunk c + 1, in flight since the last step of chunk c - 1, and this wave's reads of this stage
                wait_vm_lgkm0();
                __syncthreads();
            }
            if (cur & 8) {  // k past K2
#pragma unroll
                for (int x = 0; x < RB; x++)
                    fr[1][x] = lq < keep ? fr[1][x] : 0.0;
#pragma unroll
                for (int y = 0; y < CB; y++)
                    fc[1][y] = lq < keep ? fc[1][y] : 0.0;
            }
            row(1, 0);
            if (more) {
                tiles((c + 1) & 1);
                read(integral_constant<int, 0>{}, 0);
            }
            cur = nxt;
            if (left > 0)
                nxt = issue(c & 1);
#pragma unroll
            for (int x = 1; x < RB; x++)
                row(1, x);
        }
        int ln = lane;
        asm volatile("" : "+v"(ln));  // keeps the store addresses from being formed, and held, before the loop
        const int lr = ln & 15, lqs = ln >> 4;
        const int mw = m0 + wr * 16 * ((rb + 1) >> 1), nw = n0 + wc * 16 * ((cb + 1) >> 1);
        const int mend = min(g.M, m0 + 16 * rb), nend = min(g.N, n0 + 16 * cb);
#pragma unroll
        for (int x = 0; x < RB; x++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = mw + x * 16 + lqs + 4 * r;
#pragma unroll
                for (int y = 0; y < CB; y++) {
                    const int n = nw + y * 16 + lr;
                    if (m < mend && n < nend) {
                        if (g.splits == 1) {
                            double *cp = g.C + (int64_t)beta * g.sCb + (int64_t)m * g.sCm + (int64_t)n * g.sCn;
                            *cp = g.ow ? g.alpha * acc[x][y][r] : *cp + g.alpha * acc[x][y][r];
                        } else {
                            g.scratch[(((int64_t)split * gridDim.y + beta) * g.M + m) * g.N + n] = acc[x][y][r];
                        }
                    }
                }
            }
    }
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gemm_nt_kernel(GemmArgs g) {
    __shared__ __attribute__((aligned(1024))) char lds[4 * 128 * 128];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nbm = (g.M + 15) >> 4, nbn = (g.N + 15) >> 4, ntm = (nbm + 7) >> 3, ntn = (nbn + 7) >> 3;
    // tiles of one (batch, split) on one XCD, so the tiles sharing an operand panel share its L2
    const int nx = gridDim.x, ny = gridDim.y;
    const int lin = xcd_remap(blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z), nx * ny * gridDim.z);
    const int bx = lin % nx, byz = lin / nx;
    const int tm = bx / ntn, tn = bx - tm * ntn;
    const int beta = byz % ny, split = byz / ny;
    const int am = (int)((int64_t)tm * nbm / ntm), an = (int)((int64_t)tn * nbn / ntn);
    const int rb = (int)((int64_t)(tm + 1) * nbm / ntm) - am, cb = (int)((int64_t)(tn + 1) * nbn / ntn) - an;
    const int quad = wave ^ (lin & 3);  // the uneven quadrants of neighbouring tiles on different SIMDs
    const int nk2 = (g.seg.K2 + 15) >> 4, total = g.seg.K1 * nk2;
    const int c_begin = (int)((int64_t)total * split / g.splits), c_end = (int)((int64_t)total * (split + 1) / g.splits);
    const int k1 = c_begin / nk2, k2c = c_begin - k1 * nk2;
    const int nr = (rb + 1 - (quad >> 1)) >> 1, nc = (cb + 1 - (quad & 1)) >> 1;  // blocks of this wave's quadrant
    // Every wave passes the same barriers, one per chunk, whatever the form of its quadrant. A quadrant without
    // blocks (a tile of one block row or column) runs as one block whose results lie past the tile, and are not stored.
    auto go = [&](auto rbc, auto cbc) {
        GemmNT<decltype(rbc)::value, decltype(cbc)::value> w{g, lds};
        w.lane = lane;
        w.wave = wave;
        w.wr = quad >> 1;
        w.wc = quad & 1;
        w.m0 = 16 * am;
        w.n0 = 16 * an;
        w.rb = rb;
        w.cb = cb;
        w.beta = beta;
        w.split = split;
        w.k2c = k2c;
        w.nk2 = nk2;
        w.left = c_end - c_begin;
        const GemmOp &A = g.seg.A, &B = g.seg.B;
        w.pa = A.base + (int64_t)beta * A.sb + (int64_t)k1 * A.s1 + 16 * k2c + (int64_t)w.m0 * A.sr;
        w.pb = B.base + (int64_t)beta * B.sb + (int64_t)k1 * B.s1 + 16 * k2c + (int64_t)w.n0 * B.sr;
        const int lr = lane & 15, lq = lane >> 4;
#pragma unroll
        for (int u = 0; u < 4; u++)
            w.so[u] = lr * 128 + ((2 * u + (lq >> 1)) ^ kswz(lr)) * 16 + (lq & 1) * 8;
#pragma unroll
        for (int h = 0; h < 4; h++) {
            // rows past M (N) load the last one
            const int u = wave + 4 * h, hf = u >> 3, r = 8 * (u & 7) + (lane >> 3);
            w.oa[h] = (uint32_t)min(r + hf * 16 * ((rb + 1) >> 1), g.M - 1 - w.m0) * (uint32_t)(8 * A.sr);
            w.ob[h] = (uint32_t)min(r + hf * 16 * ((cb + 1) >> 1), g.N - 1 - w.n0) * (uint32_t)(8 * B.sr);
        }
        const int run_total = w.left;
        if (run_total == 0) {  // a split without chunks: zero partials
            w.run(0, 0, 0);
            return;
        }
        const int i0 = w.issue(0), i1 = w.left > 0 ? w.issue(1) : 0;
        w.run(run_total, i0, i1);
    };
    using std::integral_constant;
    auto cols = [&](auto rbc) {
        switch (nc) {
        case 4: go(rbc, integral_constant<int, 4>{}); break;
        case 3: go(rbc, integral_constant<int, 3>{}); break;
        case 2: go(rbc, integral_constant<int, 2>{}); break;
        default: go(rbc, integral_constant<int, 1>{}); break;
        }
    };
    switch (nr) {
    case 4: cols(integral_constant<int, 4>{}); break;
    case 3: cols(integral_constant<int, 3>{}); break;
    case 2: cols(integral_constant<int, 2>{}); break;
    default: cols(integral_constant<int, 1>{}); break;
    }
}

// 0: not K-contiguous; 1: K-contiguous; 2: K-contiguous with 16-byte aligned rows (vector loads)
static int k_contiguous(const GemmArgs &g) {
    int r = 2;
    for (const GemmOp *op : {&g.seg.A, &g.seg.B}) {
        if (op->s2 != 1)
            return 0;
        if ((op->sr & 1) || (op->s1 & 1) || (op->sb & 1) || (((uintptr_t)op->base) & 15))
            r = 1;
    }
    return r;
}

hipError_t launch_gemm(const GemmArgs &g, int batch, hipStream_t s) {
    {  // the kernels index K chunks (16 deep) with 32-bit integers
        if ((int64_t)g.seg.K1 * ((g.seg.K2 + 15) / 16) >= (int64_t)1 << 31)
            return hipErrorInvalidValue;
    }
    const int kc = k_contiguous(g);
    if (!kc)  // the callers lay their operands out with K contiguous
        return hipErrorInvalidValue;
    // FP64: 128 x 128 tiles, unless rows of a tile are too far apart for lane offsets of 32 bits
    const GemmSeg &s0 = g.seg;
    const double far = 128.0 * 8.0 * (double)std::max(s0.A.sr, s0.B.sr);
    if (g.prec == P64 && kc == 2 && s0.K2 >= 1 && s0.K1 >= 1 && g.M >= 1 && g.N >= 1 && s0.A.sr >= 0 &&
        s0.B.sr >= 0 && far < 4294967296.0) {
        const int64_t tiles = (int64_t)((g.M + 127) / 128) * ((g.N + 127) / 128);
        if (tiles > 0x7fffffff)
            return hipErrorInvalidValue;
        hipLaunchKernelGGL(gemm_nt_kernel, dim3((unsigned)tiles, (unsigned)batch, (unsigned)g.splits), dim3(256), 0, s, g);
    } else {
        // 64 x 64 tiles
        const int nt = ((g.M + 63) / 64) * ((g.N + 63) / 64);
        const dim3 grid((unsigned)nt, (unsigned)batch, (unsigned)g.splits);
        // direct-to-LDS loads when the rows are 16-byte vectors and at least two elements long (the first vector of every
        // row is then inside it); SCESS_GEMM_DMA=0 keeps the register-staged loads of the other precisions (tuning)
        bool dma = kc == 2 && g.M >= 1 && g.N >= 1 && g.seg.K2 >= 2;
        if (const char *e = std::getenv("SCESS_GEMM_DMA"))
            dma = dma && (g.prec == P64 || std::atoi(e) != 0);
        const bool vec = kc == 2 && (g.prec != P64 || dma);
        // 64 x 128 tiles for the direct-to-LDS pre-split BF16x3 products: twice the MFMAs per barrier for 1.5x the staged
        // bytes (CCSD update at o=50, v=500: 6.08 s against 7.14 s with 64 x 64). SCESS_GEMM_WIDE=0 keeps 64 x 64 (tuning).
        const char *ew = std::getenv("SCESS_GEMM_WIDE");
        const bool wide = dma && g.prec == PB3S && !(ew && std::atoi(ew) == 0);
#define SCESS_KC(V, P, D)                                                                         \
    if (vec == V && g.prec == P && dma == D) {                                                    \
        hipLaunchKernelGGL((gemm_kc_kernel<2, V, P, D, 1>), grid, dim3(256), 0, s, g);            \
    } else
        if (wide) {
            const dim3 gw((unsigned)(((g.M + 63) / 64) * ((g.N + 127) / 128)), (unsigned)batch, (unsigned)g.splits);
            hipLaunchKernelGGL((gemm_kc_kernel<2, true, PB3S, true, 2>), gw, dim3(256), 0, s, g);
        } else
        SCESS_KC(true, P64, true) SCESS_KC(true, P32, true) SCESS_KC(true, PB3, true) SCESS_KC(true, PB3S, true)
        SCESS_KC(true, PB3S, false) SCESS_KC(true, P32, false) SCESS_KC(true, PB3, false)
        SCESS_KC(false, P64, false) SCESS_KC(false, P32, false) SCESS_KC(false, PB3, false)
        return hipErrorInvalidValue;
#undef SCESS_KC
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || g.splits == 1)
        return e;
    const int64_t n = (int64_t)g.M * g.N;
    hipLaunchKernelGGL(gemm_reduce_kernel, dim3((unsigned)((n + 255) / 256), (unsigned)batch), dim3(256), 0, s, g);
    return hipGetLastError();
}

// -------------------------------------------------- back-contractions of a batch
// With c one of the three positions of a triple's G and a, b the others, the six terms of all four gradients read G in
// two ways only, each against two operands side by side as v8 + o8 columns (v, o rounded up to 8):
//   rows (x_p, x_b), K = x_c:  dX[p][x_p][x_b][f] | dTM[p][x_b][x_p][m] += G (T[c][b][x_c][f] | Rn[c][b][x_c][m])
//   rows x_c, K = (x_a, x_b):  dT[c][b][x_c][f]   | dRn[c][b][x_c][m]   += G (X[a][x_a][x_b][f] | TM[a][x_b][x_a][m])
// (p, b, c and a, b, c stand for a position and its occupied index). The first kind runs over all triples of the batch
// with the same p in one go: its output, the size of G, is read and written once per batch and p instead of once per
// term. The second kind is split over ranges of the outer K index into partials, added in order by back_reduce_kernel.
// A row group is 8 rows along the unit-stride position of G where that is a row (K otherwise). Position 2 may be p or b,
// and all terms of one output tile need the same row order: the terms with p at position 2 make a launch of their own.
//
// One work-group makes a tile of up to 8 x 8 blocks of 16; the four waves own its rows in slabs, all columns each. The
// loop is that of gemm_nt_kernel (look-ahead of one k-step, one barrier per 16 k, two work-groups per CU); a chunk of G is
// a [m][k] tile (128-byte rows, vectors swizzled by kswz) where k has unit stride, else a [k][m] tile like B's [k][n],
// with the pairs of odd k 16 elements apart from those of even k. Bound by the FP64 matrix pipes.
// Gradients of a shard (190 triples) of o=20, v=200: 141 ms in back_kernel, 57 TFLOP/s of useful products (one GEMM group
// per kind and triple before: 350 ms); o=10, v=75 (210 triples): 5.1 ms against 32 and 2520 fewer launches.
constexpr int kBackOp = 16 * 128 * 8;  // bytes of an operand's chunk

template <int RB, int CB> struct BackGemm {
    const BackArgs &a;
    char *lds;
    int lane, wave;
    // rows: groups of 8 with coordinates (X, Y); gx, gy of the four loads of a [m][k] chunk, lx, ly of a [k][m] one
    int gx[4], gy[4], lx, ly;
    int n;        // first of this lane's two columns
    int block0;   // first row block of the wave's slab
    bool rows2, second;  // second: the K = (x_a, x_b) kind; rows2: p at position 2
    // next chunk to load
    const BackSeg *sg;
    int segs, k1, k1n, k2c, nk2;
    bool mc;
    const double *pa[4], *pb;
    int64_t da, a1, b1, b2;  // advance of G per chunk and of G and B per outer k, B's per k

    __device__ inline int64_t pos(int q) const { return q == 0 ? (int64_t)a.vR * a.vR : q == 1 ? a.vR : 1; }

    __device__ inline void setup() {
        // a scalar load: the wait of a vector load would be one for the chunks in flight, too
        const auto *seg = (const __attribute__((address_space(4))) int *)(uintptr_t)sg;
        const int slot = seg[0], code = seg[1];
        const int64_t occ = seg[2], v = a.v;
        const int P = code & 3, B = (code >> 2) & 3, C = code >> 4;
        const double *G = a.G + slot * a.gstride;
        int64_t sX, sY, sk;
        const bool inv = n < a.v8;
        k2c = 0;
        if (!second) {
            mc = C != 2;
            sX = pos(rows2 ? B : P);
            sY = pos(rows2 ? P : B);
            sk = pos(C);
            a1 = b1 = 0;
            k1n = 1;
            b2 = inv ? a.vK : a.oK;
            pb = inv ? a.T + occ * v * a.vK + n : a.Rn + occ * v * a.oK + (n - a.v8);
        } else {
            // P: position of x_a; the inner K index is at position 2, or at 1 where that is the row
            mc = C == 2;
            const int in = mc ? 1 : 2;
            const bool ina = P == in;
            sX = 0;
            sY = pos(C);
            sk = pos(in);
            a1 = pos(ina ? B : P);
            const int64_t ba = inv ? v * a.vK : a.oK, bb = inv ? a.vK : v * a.oK;
            b2 = ina ? ba : bb;
            b1 = ina ? bb : ba;
            pb = inv ? a.X + occ * v * v * a.vK + n : a.TM + occ * v * v * a.oK + (n - a.v8);
            pb += k1 * b1;
            G += k1 * a1;
        }
        if (mc) {
            da = 16 * sk;
#pragma unroll
            for (int h = 0; h < 4; h++)
                pa[h] = G + lx * sX + ly + (wave + 4 * h) * sk;
        } else {
            da = 16;
#pragma unroll
            for (int h = 0; h < 4; h++) {
                const int r = 8 * (wave + 4 * h) + (lane >> 3);
                pa[h] = G + gx[h] * sX + (gy[h] + (lane >> 3)) * sY + 2 * ((lane & 7) ^ kswz(r & 15));
            }
        }
    }

    // the next chunk into stage st: returns its k-steps, bit 3: a [k][m] chunk, bit 4: there is another
    __device__ inline int issue(int st) {
        char *base = lds + st * 2 * kBackOp;
        const int left = a.v - 16 * k2c, ret = (min(left, 16) + 3) >> 2 | (mc ? 8 : 0);
#pragma unroll
        for (int h = 0; h < 4; h++) {
            const int u = wave + 4 * h;
            __builtin_amdgcn_global_load_lds((const void *)pa[h], (lds_void *)(base + u * 1024), 16, 0, 0);
            // k past v: the last row again, times zeros of G
            __builtin_amdgcn_global_load_lds((const void *)(pb + (int64_t)min(16 * k2c + u, a.v - 1) * b2),
                                             (lds_void *)(base + kBackOp + u * 1024), 16, 0, 0);
        }
#pragma unroll
        for (int h = 0; h < 4; h++)
            pa[h] += da;
        if (++k2c < nk2)
            return ret | 16;
        k2c = 0;
        if (++k1 < k1n) {
#pragma unroll
            for (int h = 0; h < 4; h++)
                pa[h] += a1 - nk2 * da;
            pb += b1;
            return ret | 16;
        }
        if (--segs == 0)
            return ret;
        sg++;
        k1 = 0;
        setup();
        return ret | 16;
    }

    template <class Store> __device__ inline void run(Store &&store) {
        d4 acc[RB][CB];
        double fr[2][RB], fc[2][CB];
#pragma unroll
        for (int x = 0; x < RB; x++)
#pragma unroll
            for (int y = 0; y < CB; y++)
                acc[x][y] = d4{};
        const int lr = lane & 15, lq = lane >> 4;
        uint32_t km[4], mk[RB], cn[2];
#pragma unroll
        for (int t = 0; t < 4; t++)
            km[t] = (block0 * 16 + lr) * 128 + ((2 * t + (lq >> 1)) ^ kswz(lr)) * 16 + (lq & 1) * 8;
#pragma unroll
        for (int x = 0; x < RB; x++)
            mk[x] = lq * 1024 + lr * 8 + ((block0 + x) ^ (lq & 1)) * 128;
#pragma unroll
        for (int y = 0; y < 2; y++)
            cn[y] = kBackOp + lq * 1024 + lr * 8 + (y ^ (lq & 1)) * 128;
        lds_char *q;
        auto read = [&](auto tc, int buf, int flags) {
            constexpr int t = decltype(tc)::value;
#pragma unroll
            for (int x = 0; x < RB; x++)
                fr[buf][x] = *(lds_double *)(q + (flags & 8 ? mk[x] + t * 4096 : km[t] + x * 2048));
#pragma unroll
            for (int y = 0; y < CB; y++)
                fc[buf][y] = *(lds_double *)(q + cn[y & 1] + (y & ~1) * 128 + t * 4096);
        };
        auto row = [&](int buf, int x) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int y = 0; y < CB; y++)
                acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr[buf][x], fc[buf][y], acc[x][y], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        int cur, nxt = 0;
        auto step = [&](int buf, auto tc) {
            row(buf, 0);
            read(tc, buf ^ 1, cur);
#pragma unroll
            for (int x = 1; x < RB; x++)
                row(buf, x);
        };
        auto move = [&]() {
#pragma unroll
            for (int x = 0; x < RB; x++)
                fr[1][x] = fr[0][x];
#pragma unroll
            for (int y = 0; y < CB; y++)
                fc[1][y] = fc[0][y];
        };
        using std::integral_constant;
        setup();
        cur = issue(0);
        if (cur & 16)
            nxt = issue(1);
        wait_vm_lgkm0();
        __syncthreads();
        q = (lds_char *)lds;
        read(integral_constant<int, 0>{}, 0, cur);
        for (int st = 0;; st ^= 1) {
            const int steps = cur & 7;
            if (steps >= 2) {
                step(0, integral_constant<int, 1>{});
                if (steps >= 3) {
                    step(1, integral_constant<int, 2>{});
                    if (steps == 4)
                        step(0, integral_constant<int, 3>{});
                    else
                        move();
                }
            } else {
                move();
            }
            const bool more = cur & 16;
            if (more) {
                wait_vm_lgkm0();
                __syncthreads();
            }
            row(1, 0);
            if (more) {
                q = (lds_char *)lds + (st ^ 1) * 2 * kBackOp;
                read(integral_constant<int, 0>{}, 0, nxt);
            }
            cur = nxt;
            if (more && (nxt & 16))
                nxt = issue(st);
#pragma unroll
            for (int x = 1; x < RB; x++)
                row(1, x);
            if (!more)
                break;
        }
        store(acc);
    }
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void back_kernel(BackArgs a) {
    __shared__ __attribute__((aligned(1024))) char lds[4 * kBackOp];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nc = a.v8 + a.o8, nbn = (nc + 15) >> 4, ntn = (nbn + 7) >> 3;
    const bool second = (int)blockIdx.x >= a.blocks1;
    // Blocks b, b + 8, ... run on one XCD. First kind: the column tiles of a row tile there, one after another (they share
    // its rows of G); second kind: all tiles of one K range.
    int tm, tn, nbm, ngy, ngrp, seg0, segs, k10 = 0, k1n = 1, id = 0, part = 0;
    if (!second) {
        const int t = (int)blockIdx.x / a.per, l = (int)blockIdx.x - t * a.per, slot = l >> 3;
        const BackTarget tg = a.tg[t];
        id = tg.id;
        seg0 = tg.seg0;
        segs = tg.nseg;
        ngy = a.v8 >> 3;
        ngrp = a.v * ngy;
        nbm = (ngrp + 1) >> 1;
        tm = slot / ntn * 8 + (l & 7);
        tn = slot % ntn;
    } else {
        ngy = ngrp = a.v8 >> 3;
        nbm = (ngrp + 1) >> 1;
        const int tiles = ((nbm + 7) >> 3) * ntn, l = (int)blockIdx.x - a.blocks1, slot = l >> 3, t = slot % tiles;
        part = slot / tiles * 8 + (l & 7);
        if (part >= a.nseg2 * a.splits)
            return;
        tm = t / ntn;
        tn = t % ntn;
        seg0 = a.seg2 + part / a.splits;
        segs = 1;
        const int sp = part % a.splits;
        k10 = (int)((int64_t)a.v * sp / a.splits);
        k1n = (int)((int64_t)a.v * (sp + 1) / a.splits);
    }
    const int ntm = (nbm + 7) >> 3;
    if (tm >= ntm)
        return;
    const int am = (int)((int64_t)tm * nbm / ntm), rb = (int)((int64_t)(tm + 1) * nbm / ntm) - am;
    const int an = (int)((int64_t)tn * nbn / ntn), cb = (int)((int64_t)(tn + 1) * nbn / ntn) - an;
    const int slab = (wave + (blockIdx.x >> 3)) & 3;  // the uneven slabs of neighbouring tiles on different SIMDs
    const int sb0 = slab * rb >> 2, nr = ((slab + 1) * rb >> 2) - sb0;
    auto go = [&](auto rbc, auto cbc) {
        constexpr int RB = decltype(rbc)::value, CB = decltype(cbc)::value;
        BackGemm<RB, CB> w{a, lds};
        w.lane = lane;
        w.wave = wave;
        w.second = second;
        w.rows2 = a.rows2;
        w.block0 = nr > 0 ? sb0 : 0;
        // column pair at slot `lane` of the rows of odd or even k (those of this wave), past the end: the last pair
        const int pair = lane ^ ((wave & 1) << 3);
        w.n = min(16 * an + 2 * pair, nc - 2);
        {
            const int g = min(2 * am + (pair >> 2), ngrp - 1);
            w.lx = g / ngy;
            w.ly = (g - w.lx * ngy) * 8 + ((2 * pair) & 7);
        }
#pragma unroll
        for (int h = 0; h < 4; h++) {
            const int g = min(2 * am + wave + 4 * h, ngrp - 1);
            w.gx[h] = g / ngy;
            w.gy[h] = (g - w.gx[h] * ngy) * 8;
        }
        w.sg = a.segs + seg0;
        w.segs = segs;
        w.k1 = k10;
        w.k1n = k1n;
        w.nk2 = (a.v + 15) >> 4;
        w.run([&](d4 (&acc)[RB][CB]) {
            if (nr == 0)  // ran for its loads and barriers
                return;
            int ln = lane;
            asm volatile("" : "+v"(ln));  // keeps the store addresses from being formed, and held, before the loop
            const int lr = ln & 15, lq = ln >> 4;
            const int n0 = 16 * an + lr;
#pragma unroll
            for (int x = 0; x < RB; x++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    // row lq + 4 r of the block: group 2 x + (r >> 1)
                    const int g = 2 * (am + sb0 + x) + (r >> 1);
                    const int X = g / ngy, Y = (g - X * ngy) * 8 + lq + 4 * (r & 1);
                    if (g >= ngrp || Y >= a.v)
                        continue;
                    double *c0, *c1;
                    if (second) {
                        c0 = c1 = a.scr + ((int64_t)part * a.v + Y) * nc + n0;
                    } else {
                        const int64_t xp = a.rows2 ? Y : X, xb = a.rows2 ? X : Y;
                        c0 = a.dX + ((id * (int64_t)a.v + xp) * a.v + xb) * a.vK + n0;
                        c1 = a.dTM + ((id * (int64_t)a.v + xb) * a.v + xp) * a.oK + (n0 - a.v8);
                    }
                    // the old values of the row in flight together
                    double old[CB];
#pragma unroll
                    for (int y = 0; y < CB; y++) {
                        const int n = n0 + 16 * y;
                        old[y] = 0.0;
                        if (!second && (n < a.v8 ? n < a.v : n - a.v8 < a.o))
                            old[y] = (n < a.v8 ? c0 : c1)[16 * y];
                    }
#pragma unroll
                    for (int y = 0; y < CB; y++) {
                        const int n = n0 + 16 * y;
                        if (n < a.v8 ? n < a.v : n - a.v8 < a.o)
                            (n < a.v8 ? c0 : c1)[16 * y] = old[y] + acc[x][y][r];
                    }
                }
        });
    };
    using std::integral_constant;
    auto cols = [&](auto rbc) {
        switch (cb) {
        case 8: go(rbc, integral_constant<int, 8>{}); break;
        case 7: go(rbc, integral_constant<int, 7>{}); break;
        case 6: go(rbc, integral_constant<int, 6>{}); break;
        case 5: go(rbc, integral_constant<int, 5>{}); break;
        case 4: go(rbc, integral_constant<int, 4>{}); break;
        case 3: go(rbc, integral_constant<int, 3>{}); break;
        case 2: go(rbc, integral_constant<int, 2>{}); break;
        default: go(rbc, integral_constant<int, 1>{}); break;
        }
    };
    if (nr == 2)
        cols(integral_constant<int, 2>{});
    else
        cols(integral_constant<int, 1>{});
}

// dT, dRn of target blockIdx.y += the partials of its segments, in order
__global__ __launch_bounds__(256) void back_reduce_kernel(BackArgs a, const BackTarget *tg, double *dT, double *dRn) {
    const int nc = a.v8 + a.o8;
    const int idx = blockIdx.x * 256 + threadIdx.x, m = idx / nc, n = idx - m * nc;
    if (m >= a.v || (n < a.v8 ? n >= a.v : n - a.v8 >= a.o))
        return;
    const BackTarget t = tg[blockIdx.y];
    const int64_t step = (int64_t)a.v * nc;
    const double *p = a.scr + (int64_t)(t.seg0 - a.seg2) * a.splits * step + idx;
    double s = 0.0;
    int q = 0;
    for (; q + 8 <= t.nseg * a.splits; q += 8) {
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            x[u] = p[(q + u) * step];
#pragma unroll
        for (int u = 0; u < 8; u++)
            s += x[u];
    }
    for (; q < t.nseg * a.splits; q++)
        s += p[q * step];
    double *c = n < a.v8 ? dT + ((int64_t)t.id * a.v + m) * a.vK + n : dRn + ((int64_t)t.id * a.v + m) * a.oK + n - a.v8;
    *c += s;
}

// The terms of triples work[0..n) (occupied indices, 3 each) as segments and targets
void back_terms(const int *ijk, int n, int o, BackTables &t, BackBatch &b) {
    // positions (P, B, C) of the six terms; with i == j (positions 0 and 1 alike) terms 4, 1, 3 equal 0, 2, 5
    static const int TERM[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 2, 0}, {2, 0, 1}, {1, 0, 2}, {2, 1, 0}};
    static const bool TWIN[6] = {true, false, true, false, false, true};
    struct Entry {
        int id;
        BackSeg s;
    };
    std::vector<Entry> e[3];  // first kind with p at position 0 or 1, first kind with p at position 2, second kind
    for (int w = 0; w < n; w++) {
        const int *q = ijk + 3 * w;
        for (int m = 0; m < 6; m++) {
            if (q[0] == q[1] && !TWIN[m])
                continue;
            const int P = TERM[m][0], B = TERM[m][1], C = TERM[m][2];
            const int code = P | B << 2 | C << 4;
            e[P == 2].push_back({q[P], {w, code, q[C] * o + q[B]}});
            e[2].push_back({q[C] * o + q[B], {w, code, q[P]}});
        }
    }
    BackRange *out[3] = {&b.rows, &b.rows2, &b.second};
    for (int k = 0; k < 3; k++) {
        std::stable_sort(e[k].begin(), e[k].end(), [](const Entry &x, const Entry &y) { return x.id < y.id; });
        out[k]->tg0 = (int)t.tg.size();
        out[k]->seg0 = (int)t.segs.size();
        for (const Entry &x : e[k]) {
            if ((int)t.tg.size() == out[k]->tg0 || t.tg.back().id != x.id)
                t.tg.push_back({x.id, (int)t.segs.size(), 0});
            t.tg.back().nseg++;
            t.segs.push_back(x.s);
        }
        out[k]->ntg = (int)t.tg.size() - out[k]->tg0;
        out[k]->nseg = (int)t.segs.size() - out[k]->seg0;
        if (k < 2)  // the longest first
            std::stable_sort(t.tg.begin() + out[k]->tg0, t.tg.end(),
                             [](const BackTarget &x, const BackTarget &y) { return x.nseg > y.nseg; });
    }
}

static int round8(int n) { return (n + 7) / 8 * 8; }
static int back_cols(int o, int v) { return ((round8(v) + round8(o) + 15) / 16 + 7) / 8; }  // column tiles
// Blocks of a target of the first kind: row tiles in eights (one per XCD) times column tiles
static int back_blocks(int o, int v) {
    const int64_t nbm = ((int64_t)v * (round8(v) / 8) + 1) / 2, ntm = (nbm + 7) / 8;
    return (int)((ntm + 7) / 8 * 8 * back_cols(o, v));
}
// Tiles of a term of the second kind
static int back_tiles(int o, int v) { return ((v + 15) / 16 + 7) / 8 * back_cols(o, v); }

// One round of the chip (o=10, v=75, 48 tiles: 12.7 ms spread, 13.0 not; o=20, v=200, 640 tiles: no difference)
bool back_spread(int o, int v) { return back_blocks(o, v) < 512; }

// K ranges of a term of the second kind: 3072 work-groups (six rounds of the chip) from n triples, at most v
int back_splits(int n, int o, int v) { return std::max(1, std::min(v, 3072 / (6 * n * back_tiles(o, v)))); }

hipError_t launch_back(const BackArgs &a0, const BackTarget *tg, const BackBatch &b, double *dT, double *dRn, hipStream_t s) {
    BackArgs a = a0;
    const int nc = a.v8 + a.o8, tiles2 = back_tiles(a.o, a.v);
    a.per = back_blocks(a.o, a.v);
    a.tg = tg + b.rows.tg0;
    a.blocks1 = b.rows.ntg * a.per;
    a.seg2 = b.second.seg0;
    a.nseg2 = b.second.nseg;
    const int blocks2 = (a.nseg2 * a.splits + 7) / 8 * 8 * tiles2;
    hipLaunchKernelGGL(back_kernel, dim3((unsigned)(a.blocks1 + blocks2)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(back_reduce_kernel, dim3((unsigned)(((int64_t)a.v * nc + 255) / 256), (unsigned)b.second.ntg), dim3(256),
                       0, s, a, tg + b.second.tg0, dT, dRn);
    a.rows2 = 1;
    a.tg = tg + b.rows2.tg0;
    a.blocks1 = b.rows2.ntg * a.per;
    hipLaunchKernelGGL(back_kernel, dim3((unsigned)a.blocks1), dim3(256), 0, s, a);
    return hipGetLastError();
}

// ------------------------------------------------------------- V backward
// V(a,b,c) = U0[a][b] t_k^c + U1[a][c] t_j^b + U2[b][c] t_i^a (U rows pitched vR, t1 rows vR):
//   dU0[a][b] = sum_c G_V t_k^c,  dU1[a][c] = sum_b G_V t_j^b,  dU2[b][c] = sum_a G_V t_i^a
//   dt_k^c = sum_ab G_V U0[a][b], dt_j^b = sum_ac G_V U1[a][c], dt_i^a = sum_bc G_V U2[b][c]
// sum_z f(z), z = 0..n-1, in order, with eight loads in flight
template <typename F> __device__ inline void nsum8(int n, F f, double &s, double &c) {
    int z = 0;
    for (; z + 8 <= n; z += 8) {
        double x[8];
#pragma unroll
        for (int q = 0; q < 8; q++)
            x[q] = f(z + q);
#pragma unroll
        for (int q = 0; q < 8; q++)
            nadd_a(s, c, x[q]);
    }
    for (; z < n; z++)
        nadd_a(s, c, f(z));
}

// dU (w = 0, 1, 2) and H[a][c] = sum_b G_V[a][b][c] U0[a][b] (w = 3, into H), one thread per output
// element; the threads of a wave take consecutive y, so every G_V read but dU0's is coalesced
__global__ __launch_bounds__(256) void vback_du_kernel(const double *GV, int64_t gstride, const double *t1,
                                                        const double *U, const int *ijk, int v, int vR, double *dU,
                                                        double *H) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t vv = (int64_t)v * v;
    if (idx >= 4 * vv)
        return;
    const int i = ijk[3 * blockIdx.y], j = ijk[3 * blockIdx.y + 1], k = ijk[3 * blockIdx.y + 2];
    GV += blockIdx.y * gstride;
    U += (int64_t)blockIdx.y * 3 * v * vR;
    dU += blockIdx.y * 3 * vv;
    H += blockIdx.y * vv;
    const int w = (int)(idx / vv);
    const int64_t xy = idx - w * vv;
    const int x = (int)(xy / v), y = (int)(xy - (int64_t)x * v);
    const int64_t R2 = (int64_t)vR * vR;
    double s = 0.0, c = 0.0;
    if (w == 0) {  // dU0[x=a][y=b]
        const double *g = GV + x * R2 + (int64_t)y * vR;
        const double *t = t1 + (int64_t)k * vR;
        nsum8(v, [&](int z) { return g[z] * t[z]; }, s, c);
    } else if (w == 1) {  // dU1[x=a][y=c]
        const double *t = t1 + (int64_t)j * vR;
        nsum8(v, [&](int z) { return GV[x * R2 + (int64_t)z * vR + y] * t[z]; }, s, c);
    } else if (w == 2) {  // dU2[x=b][y=c]
        const double *t = t1 + (int64_t)i * vR;
        nsum8(v, [&](int z) { return GV[z * R2 + (int64_t)x * vR + y] * t[z]; }, s, c);
    } else {  // H[x=a][y=c]
        const double *u0 = U + (int64_t)x * vR;
        nsum8(v, [&](int z) { return GV[x * R2 + (int64_t)z * vR + y] * u0[z]; }, s, c);
        H[xy] = s + c;
        return;
    }
    dU[idx] = s + c;
}

__global__ __launch_bounds__(256) void vback_dt_kernel(const double *GV, int64_t gstride, const double *U,
                                                        const double *H, int v, int vR, double *dt) {
    __shared__ double rs[256], rc[256];
    GV += blockIdx.y * gstride;
    U += (int64_t)blockIdx.y * 3 * v * vR;
    H += (int64_t)blockIdx.y * v * v;
    dt += (int64_t)blockIdx.y * 3 * v;
    const int w = blockIdx.x / v, x = blockIdx.x - w * v;
    const int64_t R2 = (int64_t)vR * vR, vr = (int64_t)v * vR;
    const int64_t n = w == 0 ? v : (int64_t)v * v;
    double s = 0.0, c = 0.0;
    // terms t = p v + q: dt_j[x=b] = sum_ac G[a][b][c] U1[a][c] (w = 1), dt_i[x=a] = sum_bc G[a][b][c]
    // U2[b][c] (w = 2); dt_k[x=c] = sum_a H[a][c] (w = 0, terms t = a, H from vback_du_kernel). This thread
    // takes t = tid, tid + 256, ... in order, eight loads in flight, (p, q) advanced without divisions
    const double *Uw = U + (int64_t)w * vr;
    int p = (int)(threadIdx.x / v), q = (int)(threadIdx.x % v);
    for (int64_t t0 = threadIdx.x; t0 < n; t0 += 256 * 8) {
        double xs[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            double term = 0.0;  // past the end: adds nothing
            if (t0 + 256 * u < n) {
                if (w == 0)
                    term = H[(t0 + 256 * u) * v + x];
                else
                    term = (w == 1 ? GV[p * R2 + (int64_t)x * vR + q] : GV[x * R2 + (int64_t)p * vR + q]) *
                           Uw[(int64_t)p * vR + q];
            }
            xs[u] = term;
            q += 256;
            while (q >= v) {
                q -= v;
                p++;
            }
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            nadd_a(s, c, xs[u]);
    }
    rs[threadIdx.x] = s;
    rc[threadIdx.x] = c;
    __syncthreads();
    for (int m = 128; m > 0; m >>= 1) {
        if ((int)threadIdx.x < m) {
            const double a1 = rs[threadIdx.x], b1 = rs[threadIdx.x + m];
            const double ss = a1 + b1, bp = ss - a1;
            rc[threadIdx.x] = rc[threadIdx.x] + rc[threadIdx.x + m] + ((a1 - (ss - bp)) + (b1 - bp));
            rs[threadIdx.x] = ss;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        dt[blockIdx.x] = rs[0] + rc[0];
}

// dS[p][q][x][y] = d/d(px|qy): of each triple in order the six updates dS[pq_u] += 1/2 dU[u / 2] (transposed for odd u),
// in u order, for the pair p o + q of target blockIdx.y; past the targets the row dt1[blockIdx.y - ntg] with a triple's k
// from dt[0..v), j from dt[v..2v), i from dt[2v..3v). One thread per output element, read and written once.
__global__ __launch_bounds__(256) void vback_acc_kernel(double *dS, double *dt1, const double *dU, const double *dt,
                                                         const int *ijk, int n, const BackTarget *tg, int ntg, int o, int v,
                                                         int vR) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t vv = (int64_t)v * v;
    double s = 0.0;
    if ((int)blockIdx.y >= ntg) {
        const int p = (int)blockIdx.y - ntg;
        if (idx >= v)
            return;
        double *out = dt1 + (int64_t)p * vR + idx;
        s = *out;
        for (int b = 0; b < n; b++)
#pragma unroll
            for (int u = 0; u < 3; u++)
                if (ijk[3 * b + 2 - u] == p)
                    s += dt[((int64_t)3 * b + u) * v + idx];
        *out = s;
        return;
    }
    if (idx >= vv)
        return;
    const int pq = tg[blockIdx.y].id, p = pq / o, q = pq - p * o;
    const int64_t x = idx / v, y = idx - x * v;
    double *out = dS + pq * vv + idx;
    s = *out;
    for (int b = 0; b < n; b++) {
        const int i = ijk[3 * b], j = ijk[3 * b + 1], k = ijk[3 * b + 2];
        const int P[6] = {i, j, i, k, j, k}, Q[6] = {j, i, k, i, k, j};
#pragma unroll
        for (int u = 0; u < 6; u++)
            if (P[u] == p && Q[u] == q)
                s += 0.5 * dU[(int64_t)(3 * b + u / 2) * vv + (u & 1 ? y * v + x : idx)];
    }
    *out = s;
}

hipError_t launch_vback(const double *GV, int64_t gstride, const double *U, const double *t1, const int *ijk, int n,
                        const BackTarget *tg, int ntg, int o, int v, int vR, double *dU, double *dt, double *H, double *dS,
                        double *dt1, hipStream_t s) {
    const int64_t vv = (int64_t)v * v;
    hipLaunchKernelGGL(vback_du_kernel, dim3((unsigned)((4 * vv + 255) / 256), (unsigned)n), dim3(256), 0, s, GV, gstride,
                       t1, U, ijk, v, vR, dU, H);
    hipLaunchKernelGGL(vback_dt_kernel, dim3((unsigned)(3 * v), (unsigned)n), dim3(256), 0, s, GV, gstride, U, H, v, vR,
                       dt);
    hipLaunchKernelGGL(vback_acc_kernel, dim3((unsigned)((std::max<int64_t>(vv, v) + 255) / 256), (unsigned)(ntg + o)),
                       dim3(256), 0, s, dS, dt1, dU, dt, ijk, n, tg, ntg, o, v, vR);
    return hipGetLastError();
}

// --------------------------------------------------------------- unpacking
// ColMajor host-layout gradients from the packed FP64 accumulators.
__global__ __launch_bounds__(256) void unpack_kernel(int mode, const double *A, const double *B, double *out, int o_,
                                                     int v_, int64_t vK, int64_t oK, int64_t vR) {
    const int64_t o = o_, v = v_;
    const int64_t gid = element_id();
    int64_t n = 0;
    switch (mode) {
    case 0: n = o * v * v * v; break;  // ovvv(p,x,y,f) = dX[p][x][y][f]
    case 1: n = o * v * o * o; break;  // ovoo(p,x,m,q) = -dRn[p][q][x][m]
    case 2: n = o * v * o * v; break;  // ovov(p,x,q,y) = dS[p][q][x][y]
    case 3: n = o * o * v * v; break;  // t2(q,r,z,f) = dT[q][r][z][f] + dTM[r][z][f][q]
    case 4: n = o * v; break;          // t1(k,c) = dt1[k][c]
    }
    if (gid >= n)
        return;
    double val = 0.0;
    switch (mode) {
    case 0: {
        const int64_t p = gid % o, t = gid / o, x = t % v, t2 = t / v, y = t2 % v, f = t2 / v;
        val = A[((p * v + x) * v + y) * vK + f];
    } break;
    case 1: {
        const int64_t p = gid % o, t = gid / o, x = t % v, t2 = t / v, m = t2 % o, q = t2 / o;
        val = -A[((p * o + q) * v + x) * oK + m];
    } break;
    case 2: {
        const int64_t p = gid % o, t = gid / o, x = t % v, t2 = t / v, q = t2 % o, y = t2 / o;
        val = A[((p * o + q) * v + x) * v + y];
    } break;
    case 3: {
        const int64_t q = gid % o, t = gid / o, r = t % o, t2 = t / o, z = t2 % v, f = t2 / v;
        val = A[((q * o + r) * v + z) * vK + f] + B[((r * v + z) * v + f) * oK + q];
    } break;
    case 4: {
        const int64_t kk = gid % o, c = gid / o;
        val = A[kk * vR + c];
    } break;
    }
    out[gid] = val;
}

hipError_t launch_unpack(int mode, const double *A, const double *B, double *out, int o, int v, int64_t vK, int64_t oK,
                         int64_t vR, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(unpack_kernel, element_grid(n), dim3(256), 0, s, mode, A, B, out, o, v, vK, oK,
                       vR);
    return hipGetLastError();
}

}  // namespace scess
