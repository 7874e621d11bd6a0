// Nodal solve of the HEM immittance system from explicit symmetric inverses
// (see nodal.hip): W = [[-Z_L, 0, A], [0, -Z_T, B], [A^T, B^T, 0]] stored as
// the two impedance blocks only.
#pragma once

#include <vector>

#include "lu.h"

namespace tags {

// The impedance blocks of one sample: -Z_L at Z, -Z_T at Z + m (m + 1), both
// m x m with row pitch m, which is what the fills and k_hem_apply address for
// a matrix of pitch m with zl_off = 0, zt_off = m.
inline long nodal_z_items(long m) { return (2 * m * m + m + 1) & ~1L; }

// Work space and state of the nodal solve of up to `cap` samples at once
// (every launch covers all of them). One arena, laid out anew for each
// (m, n, precision) and grown only when a layout does not fit.
struct NodalSolver {
    // refinement steps queued before the first check, and in all; the first
    // one solves for x itself
    static constexpr int kSpec64 = 2, kSpec32 = 3, kMaxSteps = 20;
    static constexpr long kNormStride = 4 * (kMaxSteps + 1);

    hipStream_t st = nullptr;
    Profiler* pr = nullptr;

    long m = 0, n = 0, N = 0, mp = 0, np = 0;
    bool f64 = false;
    int cap = 0, nb = 0;
    long inj = 0;
    HemOp op;  // node lists and offsets of the compact storage

    char* arena = nullptr;
    size_t arena_bytes = 0;
    // pinned host copies
    unsigned long long* hnorms = nullptr;
    c64* hu = nullptr;
    int* hactive = nullptr;
    int host_cap = 0;

    c64* Z = nullptr;   // impedance blocks, item stride sZ
    long sZ = 0;
    void *F = nullptr, *S = nullptr;    // factored blocks (2 per item), node systems
    void *tp = nullptr, *op_ = nullptr, *tt = nullptr, *P = nullptr;
    c64 *x = nullptr, *r = nullptr, *b = nullptr, *ysum = nullptr, *dg = nullptr, *cst = nullptr;
    void *v = nullptr, *z = nullptr, *f = nullptr, *y = nullptr, *h = nullptr, *c = nullptr;
    c64* u = nullptr;
    unsigned long long* norms = nullptr;
    int* active = nullptr;

    // bytes of `batch` items (without allocating)
    static size_t bytes(long m, long n, bool f64, int batch);
    int ensure(const HemOp& hem, bool f64, int batch);
    void release();
    ~NodalSolver() { release(); }

    // Queues the solve of nb samples whose Z is filled (or queued on st): unit
    // current at node inj. No host wait.
    int issue(int nb, long inj);
    // Called when st is idle. While samples still refine: queues one more step
    // for them, *complete false. Then per item: done steps, backward error,
    // forward estimate and whether it was accepted; u in hu, x in x.
    int advance(bool* complete);
    std::vector<int> steps, accepted, go;
    std::vector<double> berr, fwd;
    std::vector<double> hist;  // 8 per item

private:
    int step_ = 0;
    bool first_ = true;
    double norm_at(int q, int k, int i) const;
    double berr_at(int q, int k) const;
    double dx_at(int q, int k) const;
    double fwd_at(int q, int k) const;
    bool accept(int q) const;
    template <typename T>
    int factor();
    template <typename T>
    int queue_step(int k, bool masked);
    template <typename T>
    size_t partition(char* base, int batch);
};

}  // namespace tags
