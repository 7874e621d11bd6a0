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
    int parts = 1;  // parts that the solve in flight tells apart

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
    void *tp = nullptr, *op_ = nullptr, *P = nullptr;
    c64 *x = nullptr, *r = nullptr, *b = nullptr, *ysum = nullptr, *dg = nullptr, *cst = nullptr;
    void *v = nullptr, *z = nullptr, *f = nullptr, *y = nullptr, *h = nullptr, *c = nullptr;
    unsigned long long* norms = nullptr;
    int* active = nullptr;

    // bytes of `batch` items (without allocating)
    static size_t bytes(long m, long n, int parts, bool f64, int batch);
    int ensure(const HemOp& hem, bool f64, int batch);
    void release();
    ~NodalSolver() { release(); }

    // Queues the solve of nb samples whose Z is filled (or queued on st): unit
    // current at node inj. No host wait.
    int issue(int nb, long inj);
    // The same for one sample with the right-hand side in b (complex128 only).
    int issue_rhs();
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
    bool unit_ = true;  // the right-hand side is a unit current at inj
    int queue_spec();
    int queue_results();
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

// Explicit inverses of complex symmetric matrices without row exchanges, `items`
// of order dim: src row-major with pitch lds (the upper triangle is read, item
// stride ssrc), X with pitch ld = dim rounded up to 64 (both triangles, zero
// beyond dim, item stride ld ld). work: sym_inverse_bytes.
size_t sym_inverse_bytes(long dim, int items);
int sym_inverse(const c64* src, long lds, long ssrc, c64* X, long dim, int items, char* work,
                hipStream_t st);
// x += X r (n of them), the largest |X r| into *dmax (a max-reduction)
int sym_apply(const c64* X, long ld, long n, const c64* r, c64* x, unsigned long long* dmax,
              hipStream_t st);
// R -= I for `items` m x m matrices, the largest |entry| into *dmax
int sub_identity(c64* R, long m, int items, unsigned long long* dmax, hipStream_t st);
// upper triangles of X by rows (see copy_out_rows), items one after the other
int sym_pack(const c64* X, long ld, long m, int items, c64* out, hipStream_t st);

// Whether W (N x N, N = n + 2 m; lower triangle column-major) is an immittance
// matrix of the HEM in the reference order: out = start nodes (m), end nodes
// (m), the number of start and of end entries found per segment (2 m), and the
// count of entries that do not fit.
int imm_structure(const c64* W, long N, long m, long n, int* out, hipStream_t st);
// its impedance blocks in NodalSolver's storage
int imm_blocks(const c64* W, long N, long m, long n, c64* Z, hipStream_t st);

}  // namespace tags
