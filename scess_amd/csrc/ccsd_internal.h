// Device tensors, the einsum engine and the closed-shell CCSD state.
#pragma once

#include "buffers.h"
#include "triples_internal.h"

#include <cstdint>
#include <functional>
#include <string>
#include <vector>

namespace scess {

// Row-major FP64 device tensor owning its allocation.
struct DTensor {
    double *p = nullptr;
    std::vector<int64_t> dims;
    BlockCache *home = nullptr;  // where the allocation goes back to
    DTensor() = default;
    DTensor(const DTensor &) = delete;
    DTensor &operator=(const DTensor &) = delete;
    DTensor(DTensor &&o) noexcept;
    DTensor &operator=(DTensor &&o) noexcept;
    ~DTensor();
    void release();
    int64_t size() const;
};

// Stream-ordered tensor operations; errors are thrown as std::runtime_error.
struct Engine {
    hipStream_t stream = nullptr;
    BlockCache *blocks = nullptr;  // of the context; outlives every tensor
    double *dotbuf = nullptr;
    int prec = 0;  // product precision of the einsum contractions (P64, P32, PB3), see GemmArgs::prec
    ~Engine();
    DTensor alloc(std::vector<int64_t> dims, bool zero = false);
    void upload(DTensor &t, const double *host);
    void download(const DTensor &t, double *host);
    void copy(DTensor &dst, const DTensor &src);
    void axpby(double *out, const double *x, const double *y, double alpha, double beta, int64_t n);
    void permute(const std::string &li, const double *in, const std::vector<int64_t> &idims, const std::string &lo,
                 double *out, const std::vector<int64_t> &odims, double alpha, double beta, int64_t row = 0,
                 int64_t pitch = 0);  // rows of `row` outputs `pitch` apart (0: contiguous)
    // the permutation of `in` (labels li -> lo, output dims odims) written as pre-split BF16x3 rows of its
    // last K elements (rows padded to a multiple of 32 k); returned as rows x Kp/2 eight-byte slots
    DTensor permute_split(const std::string &li, const double *in, const std::vector<int64_t> &idims,
                          const std::string &lo, const std::vector<int64_t> &odims, int64_t K);
    // C = beta C + alpha einsum(spec, A, B); B == nullptr for a pure permutation
    void einsum(const std::string &spec, const DTensor &A, const DTensor *B, DTensor &C, double alpha, double beta);
    // one launch of a small einsum (labels lk summed), see contract_kernel
    void contract(const std::string &la, const DTensor &A, const std::string &lb, const DTensor &B, const std::string &lc,
                  const std::string &lk, DTensor &C, double alpha, double beta);
    double dot(const double *x, const double *y, int64_t n);  // compensated, deterministic
    // out[q] = dot(x, y[q]) for q < m <= kMaxDots, one launch and one copy
    static constexpr int kMaxDots = 8;
    void dots(const double *x, const double *const *y, int m, int64_t n, double *out);
    // Whether t (i, j, a, b) has t_ij^ab = t_ji^ba within the rounding of precision `prec`: pair_check() starts the
    // comparison on the device, pair_symmetric() waits for it; or at once, for a ColMajor t on the host
    void pair_check(const DTensor &t);
    bool pair_symmetric();
    bool pair_symmetric(const double *t, int64_t o, int64_t v) const;

private:
    double *asym = nullptr;  // pinned: max |t_ij^ab - t_ji^ba| and max |t_ij^ab| of each block of the comparison
    int asym_blocks = 0;
    hipEvent_t asym_done = nullptr;
};

// Resident integral blocks of SolveRCCSD_DIIS (src/Quantum/CC/RCCSD.cpp:31-44), row-major with
// the reference's index order, plus the optional Cholesky factor of (ac|bd).
struct CcsdState {
    bool have = false;
    int64_t o = 0, v = 0, naux = 0;  // naux: pitch of the rows of Lvv (even, zero padded)
    DTensor ovov, oovv, ovvo, ovvv, ovoo, oooo_phys, vvvv_phys, oovv_phys, L_oovv_phys, L_ovov, Lvv, e;
    DTensor t2driver, f12energy;
    void make_tau(Engine &E, const DTensor &t1, const DTensor &t2, DTensor &tau);
    void ladder_from_factor(Engine &E, const DTensor &tau, DTensor &R);
    void ladder_symmetric(Engine &E, const DTensor &tau, DTensor &R);
    // One Jacobi update (UpdateAmplitudes); symmetric: whether t_ij^ab = t_ji^ba, asked where the ladder without vvvv comes
    void update(Engine &E, DTensor &t1, DTensor &t2, const std::function<bool()> &symmetric);
    double energy(Engine &E, const DTensor &t1, const DTensor &t2);
};

// t1 /= e_i - e_a and t2 /= e_i + e_j - e_a - e_b in place (row-major)
hipError_t ccsd_jacobi(double *t1, double *t2, const double *e, int o, int v, hipStream_t s);

}  // namespace scess
