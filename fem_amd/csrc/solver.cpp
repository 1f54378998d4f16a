// Device-resident AMG hierarchy and the Krylov drivers of liblina_hip.
//
// The host setup (amg_setup.cpp) produces the hierarchy; this file uploads it
// once (CSR values in FP64 and an FP32 copy, LDS row-block schedules,
// colour permutations, level schedules) and runs the reference's solve
// algorithms with every vector operation on the device:
//
//   pcg        PCGS.c:163-233
//   AMG_solve  Multigrid.c:1863-1931
//   V-cycle    Multigrid.c:1536-1580
//
// The host only reads back the scalars that drive control flow (|R| per
// Krylov iteration, |f-Ax| per V-cycle).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <string>
#include <tuple>
#include <type_traits>
#include <vector>

#include "../../include/lina_hip.h"
#include "kernels.hpp"
#include "lina_internal.hpp"
#include "solver.hpp"

namespace lina {

// ------------------------------------------------------------ errors

static thread_local std::string g_err;

void set_error(const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_err = buf;
}

const char* last_error() { return g_err.c_str(); }

void hip_check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw HipError(std::string(what) + ": " + hipGetErrorString(e));
}

void Captured::reset() {
    if (exec_) (void)hipGraphExecDestroy(exec_);
    if (graph_) (void)hipGraphDestroy(graph_);
    exec_ = nullptr;
    graph_ = nullptr;
}

void Captured::capture(hipStream_t st, const std::function<void()>& record) {
    reset();
    hip_check(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal), "begin capture");
    try {
        record();
    } catch (...) {
        hipGraph_t g = nullptr;  // the stream leaves capture whatever happened
        (void)hipStreamEndCapture(st, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
    }
    hip_check(hipStreamEndCapture(st, &graph_), "end capture");
    hip_check(hipGraphInstantiate(&exec_, graph_, nullptr, nullptr, 0), "instantiate");
}

void Captured::launch(hipStream_t st) const { hip_check(hipGraphLaunch(exec_, st), "graph launch"); }

bool wait_status(const double* status, int k, hipStream_t st, double* r) {
    const double* s = status + 4 * (k % 4);
    bool idle = false;
    for (long spin = 1;; spin++) {
        double seen, norm, stop, again;
        __atomic_load(s, &seen, __ATOMIC_ACQUIRE);
        if (seen >= (double)k) {
            // iteration k + 4 may be writing the slot: its norm and flag come
            // before its number, so read them until the number has held still
            __atomic_load(s + 1, &norm, __ATOMIC_ACQUIRE);
            __atomic_load(s + 2, &stop, __ATOMIC_ACQUIRE);
            __atomic_load(s, &again, __ATOMIC_ACQUIRE);
            if (again != seen) continue;
            *r = norm;
            // a later iteration in the slot: k did not stop the loop
            return seen == (double)k && stop != 0.0;
        }
        if (idle) throw HipError("the loop test was not reported");
        if (spin % 4096) continue;
        const hipError_t e = hipStreamQuery(st);
        if (e == hipErrorNotReady) continue;
        hip_check(e, "loop test");
        idle = true;  // everything queued is done: one more look
    }
}

double LoopTrend::left() const {
    if (n_ < W) return 0.0;
    const double now = r_[(n_ - 1) % W], then = r_[n_ % W];
    if (!(now > target_)) return 0.0;
    if (!(now < then) || !(target_ > 0.0)) return 1e9;
    return std::log(now / target_) * (W - 1) / std::log(then / now);
}

// ------------------------------------------------------------ memory

DevBuffers::~DevBuffers() {
    for (void* p : ptrs) (void)hipFree(p);
}

DevBuffers& DevBuffers::operator=(DevBuffers&& o) {
    std::swap(ptrs, o.ptrs);
    std::swap(chunk, o.chunk);
    std::swap(left, o.left);
    return *this;
}

void DevBuffers::drop(void* p, size_t bytes) {
    if (bytes <= SHARED_MAX) return;  // part of a shared allocation
    const auto it = std::find(ptrs.begin(), ptrs.end(), p);
    if (it == ptrs.end()) return;
    (void)hipFree(p);
    ptrs.erase(it);
}

// row-block schedule over rows [begin, end): at most max_nnz products and
// max_rows rows per block; a row longer than max_nnz gets a block alone.
// (Blocks of up to 1024 rows for the prolongations, a few entries a row,
// measured no faster.)
// Appends the blocks' first rows to starts.
void build_blocks(const Csr& A, int begin, int end, int max_nnz, std::vector<int>& starts, int max_rows) {
    int r = begin;
    int nnz = 0, rows = 0;
    if (begin >= end) return;
    starts.push_back(begin);
    while (r < end) {
        int len = A.rp[r + 1] - A.rp[r];
        if (rows > 0 && (nnz + len > max_nnz || rows == max_rows)) {
            starts.push_back(r);
            nnz = 0;
            rows = 0;
        }
        nnz += len;
        rows++;
        r++;
    }
}

// (first row, first entry) of each block start (the list ends with A.n)
std::vector<int2> block_pairs(const Csr& A, const std::vector<int>& starts_with_end) {
    std::vector<int2> bk(starts_with_end.size());
    for (size_t b = 0; b < starts_with_end.size(); b++) {
        bk[b].x = starts_with_end[b];
        bk[b].y = A.rp[starts_with_end[b]];
    }
    return bk;
}

// every index a kernel will dereference must be inside its array
static void validate(const Csr& A, const std::vector<int>& starts, int max_nnz) {
    if ((int)A.rp.size() != A.n + 1 || A.rp[0] != 0) throw std::logic_error("upload: bad row pointer");
    for (int i = 0; i < A.n; i++)
        if (A.rp[i + 1] < A.rp[i]) throw std::logic_error("upload: row pointer not monotone");
    for (int c : A.ci)
        if (c < 0 || c >= A.ncols) throw std::logic_error("upload: column index outside the matrix");
    for (size_t b = 0; b + 1 < starts.size(); b++) {
        int r0 = starts[b], r1 = starts[b + 1];
        if (r0 >= r1 || r1 > A.n) throw std::logic_error("upload: bad row block");
        if (r1 - r0 > dev::BLOCK_ROWS) throw std::logic_error("upload: row block too tall");
        if (A.rp[r1] - A.rp[r0] > max_nnz && r1 - r0 != 1) throw std::logic_error("upload: row block too wide");
    }
}

// Prolongation rows may carry sparse_zero's (i,0.0) seed at a column i that
// is not a coarse index (rows left empty by the reference); a zero product
// adds nothing, so such entries are dropped before upload.
static Csr drop_outside_zeros(const Csr& A) {
    Csr B;
    B.n = A.n;
    B.ncols = A.ncols;
    B.rp.assign(A.n + 1, 0);
    for (int i = 0; i < A.n; i++) {
        for (int p = A.rp[i]; p < A.rp[i + 1]; p++) {
            if (A.ci[p] >= A.ncols) {
                if (A.v[p] != 0.0) throw std::logic_error("upload: nonzero entry outside the matrix");
                continue;
            }
            B.ci.push_back(A.ci[p]);
            B.v.push_back(A.v[p]);
        }
        B.rp[i + 1] = (int)B.ci.size();
    }
    return B;
}

// 16-bit column codes of a schedule (see dev::DMat::cs): per block, the
// sorted columns are split at their largest gap into at most two clusters;
// when each spans < 32768 the block gets bases (b0, b1) and codes
// sel << 15 | (column - base_sel), otherwise b0 = -1 (32-bit columns).
// Returns the number of entries coded in 16 bits.
static long column_codes(const Csr& A, const std::vector<int>& starts_with_end, std::vector<uint16_t>& cs,
                         std::vector<int2>& cb) {
    const int nblk = (int)starts_with_end.size() - 1;
    cb.assign(std::max(nblk, 1), make_int2(-1, -1));
    cs.assign(A.ci.size(), 0);
    long coded = 0;
    std::vector<int> c;
    for (int b = 0; b < nblk; b++) {
        const int k0 = A.rp[starts_with_end[b]], k1 = A.rp[starts_with_end[b + 1]];
        if (k1 <= k0) continue;
        c.assign(A.ci.begin() + k0, A.ci.begin() + k1);
        std::sort(c.begin(), c.end());
        size_t g = 0;  // clusters [c0, c[g]] and [c[g+1], c.back()]
        for (size_t i = 1; i < c.size(); i++)
            if (c[i] - c[i - 1] > c[g + 1] - c[g]) g = i - 1;
        int b0 = c.front(), b1 = c.front();
        if (c.back() - c.front() > 32767) {
            if (c[g] - c.front() > 32767 || c.back() - c[g + 1] > 32767) continue;
            b1 = c[g + 1];
        }
        cb[b] = make_int2(b0, b1);
        for (int k = k0; k < k1; k++) {
            const int col = A.ci[k];
            cs[k] = (b1 != b0 && col >= b1) ? (uint16_t)(0x8000 | (col - b1)) : (uint16_t)(col - b0);
        }
        coded += k1 - k0;
    }
    return coded;
}

// first and last system (seg: a batch's row offsets per system) of each row
// block's rows; row r of A is row row_ids[r] of the level (ascending in a block)
static std::vector<int2> block_systems(const std::vector<int>& starts_with_end, const std::vector<int>& seg,
                                       const int* row_ids) {
    const int nblk = (int)starts_with_end.size() - 1;
    std::vector<int2> bs(std::max(nblk, 1), make_int2(0, 0));
    auto sys = [&](int r) {
        const int i = row_ids ? row_ids[r] : r;
        return (int)(std::upper_bound(seg.begin(), seg.end(), i) - seg.begin()) - 1;
    };
    for (int b = 0; b < nblk; b++) {
        const int r0 = starts_with_end[b], r1 = starts_with_end[b + 1] - 1;
        const int s0 = sys(r0), s1 = sys(r1);
        bs[b] = make_int2(std::min(s0, s1), std::max(s0, s1));
    }
    return bs;
}

// The slices of a matrix (dev::Slices) or none: groups: row offsets that no
// slice may straddle (a colour-permuted copy's colours; empty: one group).
//
// T lanes a row.  free_order false: the block form's lanes_per_row, so that a
// row's products are added in its order (the same bits); with blocks given and
// T = 1 each workgroup also keeps the rows of one block, so that a product's
// block partials (P.Q of the outer CG) are the block form's.  free_order true:
// one lane for short rows (means up to 24 entries) unless that leaves most of
// the chip idle (below 1,024 wavefronts), then four of at least 3 entries
// each; for longer rows as many as make 4,096 wavefronts (16 per compute unit:
// 20k rows x 117 entries takes 14.0 us with 313 wavefronts, 5.0 us with 5,000;
// 148k x 38 is flat from 2,300 to 9,200, 8.7 us, and 10 us beyond), at least 6
// entries a lane.
//
// No slices where more than twice the entries would be read: those are the
// coarsest levels with a few rows many times the mean, which the block form
// splits evenly.  Nor where more than four times the entries and 1M (10 MB in
// FP64) would be stored: a step takes 64 entries however few rows its slice has,
// so many small groups of long rows (a clique's colours) cost up to 64 / T
// times what they read.
struct SlicePlan {
    std::vector<dev::SliceHead> head;
    std::vector<int> group;  // first slice of each group, then the slice count
    int lt = 0;
    size_t steps = 0;
};

static int log2_of(int lanes) {
    int t = 0;
    while ((1 << t) < lanes) t++;
    return t;
}

static int slice_lanes(const Csr& A, const std::vector<int>& groups, bool free_order) {
    if (A.n == 0) return 0;
    const double mean = (double)A.nnz() / A.n;
    int lt = 0;
    if (free_order) {
        const double waves = (double)A.n / std::max((int)groups.size() - 1, 1) / 64;
        auto more = [&]() { lt = lt == 0 ? 2 : lt + 1; };  // 1, 4, 8, 16 as in the block form
        if (mean > 24)
            while (lt < 4 && waves * (1 << lt) < 4096 && mean >= (lt == 0 ? 24 : 6 << (lt + 1))) more();
        else if (waves < 1024 && mean >= 12)
            more();
    } else {
        while ((1 << lt) < dev::lanes_per_row(mean)) lt++;
    }
    return lt;
}

// lt: log2 of the lanes a row
static SlicePlan plan_slices(const Csr& A, const std::vector<int>& groups, int lt,
                             const std::vector<int>* blocks = nullptr) {
    SlicePlan p;
    p.lt = lt;
    const long nnz = A.nnz();
    if (A.n == 0 || nnz == 0) return p;
    const std::vector<int> whole = {0, A.n};
    const bool per_block = blocks && p.lt == 0;
    const std::vector<int>& g = per_block ? *blocks : groups.empty() ? whole : groups;
    const int ng = (int)g.size() - 1, T = 1 << p.lt, R = 64 / T;
    size_t steps = 0;
    for (int q = 0; q < ng; q++) {
        p.group.push_back((int)p.head.size());
        for (int r = g[q]; r < g[q + 1]; r += R) {
            dev::SliceHead h;
            h.row0 = r;
            h.row1 = std::min(r + R, g[q + 1]);
            h.step0 = (int)steps;
            int w = 0;
            for (int i = r; i < h.row1; i++) w = std::max(w, A.rp[i + 1] - A.rp[i]);
            h.steps = (w + T - 1) / T;
            steps += h.steps;
            p.head.push_back(h);
        }
        while (per_block && p.head.size() % dev::SLICES_PER_BLOCK) {
            dev::SliceHead h;
            h.row0 = h.row1 = g[q + 1];
            h.step0 = (int)steps;
            p.head.push_back(h);
        }
    }
    p.group.push_back((int)p.head.size());
    p.steps = steps;
    // entries read: lanes past a slice's rows load nothing
    size_t read = 0;
    for (const dev::SliceHead& h : p.head) read += (size_t)h.steps * T * (h.row1 - h.row0);
    if (read > 2 * (size_t)nnz || 64 * steps > 4 * (size_t)nnz + (1 << 20)) {  // nnz < 2^31: step0 fits an int
        p.head.clear();
        p.group.clear();
        p.steps = 0;
    }
    return p;
}

// Whether the row kernels take a matrix faster from slices than from row
// blocks, by launch (a group each), in us.  A slice is a chain of its longest
// row's steps, 8 in flight; row blocks spread a long row over a workgroup.
// Measured (blocks, slices; FP32): 116k entries, 50 steps, 4.9, 6.9; 248k, 108,
// 7.7, 12.4; 638k, 407, 16.2, 37.1; 1.5M, 148, 11.3, 15.6; the other side 506k,
// 26 steps, 8.5, 4.9; 986k, 65, 12.1, 8.2.  FP64 streams of long rows are a
// little faster in blocks: 6.4M entries in rows of 95, 17.0, 19.5; 39M, 159,
// 82, 97; but 1.7M, 95, 14.8, 7.1 and 7.8M, 53, 19.2, 19.6.  A colour's sweep
// loads its rows' places, then their right-hand sides first (base).  Padding
// costs where it is much: a prolongation of 2.1M rows, 9.4M entries, 1.47 read
// an entry, FP64 35.5, 50.1, FP32 23.3, 24.7; 525k, 2.7M, 1.69, 12.4, 15.8; but
// 1.05M, 2.5M, 1.49, 15.9, 10.7.
static bool slices_pay(const Csr& A, const SlicePlan& p, bool fp64) {
    const double base = p.group.size() > 2 ? 3.0 : 2.0;
    double slices = 0, blocks = 0, read = 0;
    for (size_t g = 0; g + 1 < p.group.size(); g++) {
        int steps = 0;
        double ent = 0;
        for (int k = p.group[g]; k < p.group[g + 1]; k++) {
            const dev::SliceHead& h = p.head[k];
            steps = std::max(steps, h.steps);
            ent += A.rp[h.row1] - A.rp[h.row0];
            read += ((double)h.steps * (h.row1 - h.row0)) * (1 << p.lt);
        }
        slices += base + 0.72 * ((steps + 7) / 8);
        blocks += 4.0 + std::min(ent / 1e5, 8.0);
    }
    if (slices > blocks || (read > 1.4 * A.nnz() && read - A.nnz() > 1.5e6)) return false;
    return !(fp64 && A.nnz() >= 4000000 && A.nnz() >= 90.0 * A.n);
}

// the slices of a matrix's copy by the rules, or none
static SlicePlan rule_slices(const Csr& A, const std::vector<int>& groups, bool free_order, bool fp64) {
    SlicePlan p = plan_slices(A, groups, slice_lanes(A, groups, free_order));
    return slices_pay(A, p, fp64) ? p : SlicePlan();
}

static bool same_rows(const SlicePlan& a, const SlicePlan& b) {
    auto eq = [](const dev::SliceHead& x, const dev::SliceHead& y) {
        return x.row0 == y.row0 && x.row1 == y.row1 && x.step0 == y.step0 && x.steps == y.steps;
    };
    return a.lt == b.lt && a.steps == b.steps && a.head.size() == b.head.size() &&
           std::equal(a.head.begin(), a.head.end(), b.head.begin(), eq);
}

// every row in one slice whose steps hold its entries, every slice's steps in
// the plan's
static void validate(const Csr& A, const SlicePlan& p) {
    if (p.head.empty()) return;
    const int T = 1 << p.lt;
    int row = 0;
    size_t step = 0;
    for (const dev::SliceHead& h : p.head) {
        if (h.row0 != row || h.row1 < h.row0 || h.row1 > A.n || h.row1 - h.row0 > 64 / T)
            throw std::logic_error("upload: bad slice rows");
        if ((size_t)h.step0 != step || h.steps < 0) throw std::logic_error("upload: bad slice steps");
        for (int i = h.row0; i < h.row1; i++)
            if (A.rp[i + 1] - A.rp[i] > (long)h.steps * T) throw std::logic_error("upload: row longer than its slice");
        row = h.row1;
        step += h.steps;
    }
    if (row != A.n || step != p.steps) throw std::logic_error("upload: slices do not cover the matrix");
}

// steps in flight per lane: all of a short row, else the count that wastes
// least of its last round (7 for the 7 and 14 entries of the P1 stencils:
// 2.1M rows x 14 in FP64, 69 us with 8, 65 us with 7)
static int slice_unroll(double mean_steps) {
    const int w = (int)std::ceil(mean_steps);
    if (w <= 4) return 4;
    return (w + 6) / 7 * 7 < (w + 7) / 8 * 8 ? 7 : 8;
}

// D.sl's fields from the plan.  Large streams are loaded nontemporally: FP64
// from 64 MB (read once per Krylov iteration; 2.1M rows x 14, 79 -> 69 us, 1.05M
// x 7, 22.0 -> 20.4 us), FP32 from 128 MB (2.1M x 14, 40 -> 37 us; smaller ones
// stay in the last-level cache between sweeps and lose: 403k x 14, 8.6 -> 9.1 us).
template <typename VT>
static dev::Slices<VT> slice_shape(const SlicePlan& p) {
    dev::Slices<VT> S;
    S.ns = (int)p.head.size();
    S.lt = p.lt;
    S.steps = p.steps;
    S.unroll = slice_unroll((double)S.steps / std::max(S.ns, 1));
    S.nt = S.steps * 64 * (sizeof(VT) + 2) >= (sizeof(VT) == 8 ? 64u << 20 : 128u << 20);
    return S;
}

// D.sl from the plan (D's CSR uploaded); share: the other precision's copy of
// the same plan (same_rows), whose heads and codes are reused.
template <typename VT, typename OT>
static void make_slices(const SlicePlan& p, dev::DMat<VT>& D, DevBuffers& B, hipStream_t st,
                        const dev::DMat<OT>* share) {
    dev::Slices<VT>& S = D.sl;
    S = slice_shape<VT>(p);
    if (p.head.empty()) return;
    if (share && (share->sl.ns != S.ns || share->sl.lt != S.lt || share->sl.steps != S.steps))
        throw std::logic_error("slices shared between different plans");
    S.v = dalloc<VT>(S.steps * 64, B);
    if (share) {
        S.head = share->sl.head;
        S.cs = share->sl.cs;
    } else {
        S.head = dupload(p.head, B, st);
        S.cs = dalloc<uint16_t>(S.steps * 64, B);
        dev::slice_columns<VT>(st, D);
    }
    dev::slice_values<VT>(st, D);
    D.lpr = 1 << p.lt;
    D.idx_bytes = 2.0 * D.nnz + 24.0 * S.ns;  // 32 bytes a head, 8 of them counted as its bounds
}

// slices of a matrix without groups and systems (krylov.cpp's operators)
bool slice_matrix(const Csr& A, dev::DMat<double>& D, DevBuffers& B, hipStream_t st) {
    const SlicePlan p = rule_slices(A, {}, false, true);  // the ILU's Krylov loops take no partials from it
    make_slices<double, double>(p, D, B, st, nullptr);
    return D.sl.ns > 0;
}

// the slices' first rows, ending with A.n
static std::vector<int> slice_starts(const Csr& A, const SlicePlan& p) {
    std::vector<int> first;
    for (const dev::SliceHead& k : p.head) first.push_back(k.row0);
    first.push_back(A.n);
    return first;
}

// plan: the slices (none: empty), starts_with_end: the row blocks (none:
// empty); share: a copy of A with other values uploaded before; its row
// pointers and column indices are reused, its slices' heads and codes with
// share_slices (the same plan), its 16-bit offsets when its block schedule
// (share_starts) is the same
template <typename VT, typename OT = double>
static void upload_mat(const Csr& A, const SlicePlan& plan, const std::vector<int>& starts_with_end,
                       dev::DMat<VT>& D, DevBuffers& B, hipStream_t st, const dev::DMat<OT>* share = nullptr,
                       bool share_slices = false, const std::vector<int>* share_starts = nullptr,
                       const int* row_ids = nullptr, const std::vector<int>* seg = nullptr) {
    validate(A, starts_with_end, dev::block_nnz<VT>());
    validate(A, plan);
    D.active = nullptr;
    D.n = A.n;
    D.ncols = A.ncols;
    D.nnz = A.nnz();
    D.rp = share ? share->rp : dupload(A.rp, B, st);
    D.ci = share ? share->ci : dupload(A.ci, B, st);
    std::vector<VT> v(A.v.begin(), A.v.end());
    D.v = dupload(v, B, st);
    D.cs = nullptr;
    D.cb = nullptr;
    D.bspec = nullptr;
    D.sl = dev::Slices<VT>();
    D.nblk = std::max((int)starts_with_end.size() - 1, 0);
    if (D.nblk > 0) {
        D.bk = dupload(block_pairs(A, starts_with_end), B, st);
        if (share && share_starts && *share_starts == starts_with_end) {
            D.cs = share->cs;
            D.cb = share->cb;
            D.idx_bytes = share->idx_bytes;
        } else {
            std::vector<uint16_t> cs;
            std::vector<int2> cb;
            const long coded = A.nnz() > 0 ? column_codes(A, starts_with_end, cs, cb) : 0;
            D.idx_bytes = 4.0 * A.nnz();
            if (coded > 0) {
                D.cs = dupload(cs, B, st);
                D.cb = dupload(cb, B, st);
                D.idx_bytes = 2.0 * coded + 4.0 * (A.nnz() - coded) + 8.0 * D.nblk;
            }
        }
        D.lpr = dev::lanes_per_row(A.n > 0 ? (double)A.nnz() / A.n : 0.0);
    }
    if (!plan.head.empty()) make_slices<VT, OT>(plan, D, B, st, share_slices ? share : nullptr);
    if (seg)  // the systems of each slice, or of each block where there are no slices
        D.bspec = dupload(block_systems(plan.head.empty() ? starts_with_end : slice_starts(A, plan), *seg, row_ids), B, st);
    // diagonal positions (row r's own index: row_ids == nullptr) and l1 norms
    std::vector<int> dpos(A.n, -1);
    std::vector<VT> l1(A.n, (VT)0);
    for (int r = 0; r < A.n; r++) {
        int i = row_ids ? row_ids[r] : r;
        VT s = 0;
        for (int p = A.rp[r]; p < A.rp[r + 1]; p++) {
            if (A.ci[p] == i) dpos[r] = p;
            s += std::fabs((VT)A.v[p]);
        }
        l1[r] = s;
    }
    D.dpos = dupload(dpos, B, st);
    D.l1 = dupload(l1, B, st);
}

// entries per row block of a matrix with nnz entries: the kernels' maximum,
// halved (down to 256) until the matrix has about 2048 blocks -- 8 per CU, so
// that the small coarse levels and transfers are not left to a few CUs
static int block_cap(long nnz, int cap) {
    int m = cap;
    while (m > 256 && nnz / m < 2048) m /= 2;
    return m;
}

// block schedule of [0, A.n) for value type VT, ending with A.n
template <typename VT>
static std::vector<int> schedule(const Csr& A) {
    std::vector<int> starts;
    build_blocks(A, 0, A.n, block_cap(A.nnz(), dev::block_nnz<VT>()), starts);
    starts.push_back(A.n);
    if (A.n == 0) starts.assign(1, 0);
    return starts;
}

// the slices and row blocks of a matrix's FP64 and FP32 copies
struct PairPlan {
    SlicePlan p64, p32;
    std::vector<int> s64, s32;
    bool shared = false;  // one plan: the FP32 copy takes the FP64 copy's heads and codes
};

// free32: the FP32 rows may be summed in any order (see Solver::fixed_order);
// partials: the FP64 product's block partials are summed by a Krylov method
// (its row order is kept then, and its partials' too without free32); tuned:
// the autotuner's lanes
static PairPlan plan_pair(const Csr& A, bool batch, bool free32, bool partials, const TunedLanes* tuned = nullptr) {
    PairPlan q;
    // the FP64 finest matrix (partials) keeps a row's column order
    if (!tuned) {
        q.p64 = rule_slices(A, {}, !partials, true);
        q.p32 = rule_slices(A, {}, free32, false);
    } else {
        if (tuned->s64) q.p64 = plan_slices(A, {}, log2_of(tuned->l64));
        if (tuned->s32) q.p32 = plan_slices(A, {}, log2_of(tuned->l32));
    }
    if (partials && !free32 && !batch && !q.p64.head.empty() && q.p64.lt == 0) {
        // slices by row block where they fill their wavefronts (1.05M rows x
        // 7: 256-row blocks), else the block form beside them (2.1M x 14, 146
        // rows a block: 76 us, 87 us as slices of 64, 64 and 18 rows)
        q.s64 = schedule<double>(A);
        SlicePlan b = plan_slices(A, {}, 0, &q.s64);
        if (!b.head.empty() && A.n >= 0.9 * 64 * b.head.size()) {
            q.p64 = std::move(b);
            q.s64.clear();
        }
    }
    if (q.p64.head.empty()) q.s64 = schedule<double>(A);
    if (q.p32.head.empty()) q.s32 = schedule<float>(A);
    // the FP32 plan is cut every 64 rows, the FP64 plan now and then by row
    // block: as many slices need not be the same rows
    q.shared = same_rows(q.p64, q.p32);
    return q;
}

// upload A as FP64 + FP32 copies sharing the index arrays (options: see
// plan_pair); returns the largest workgroup count of a row kernel over either
// copy in either form
int upload_pair(const Csr& A0, dev::DMat<double>& D, dev::DMat<float>& F, DevBuffers& B, hipStream_t st,
                const std::vector<int>* seg, bool free32, bool partials, const TunedLanes* tuned) {
    Csr A = drop_outside_zeros(A0);
    const PairPlan q = plan_pair(A, seg != nullptr, free32, partials, tuned);
    upload_mat<double, double>(A, q.p64, q.s64, D, B, st, nullptr, false, nullptr, nullptr, seg);
    upload_mat(A, q.p32, q.s32, F, B, st, &D, q.shared, &q.s64, nullptr, seg);
    if (tuned) {
        if (!D.sl.ns) D.lpr = tuned->l64;
        if (!F.sl.ns) F.lpr = tuned->l32;
    }
    const int blocks = std::max((int)schedule<double>(A).size(), (int)schedule<float>(A).size()) - 1;
    return std::max({dev::row_blocks(D), dev::row_blocks(F), blocks});
}

// the rows of A colour by colour (natural order within one): perm the row of A
// in each place, rows the colours' offsets
static Csr colour_permuted(const Csr& A, const std::vector<int>& col, int nc, std::vector<int>& perm,
                           std::vector<int>& rows) {
    rows.assign(nc + 1, 0);
    for (int i = 0; i < A.n; i++) rows[col[i] + 1]++;
    for (int c = 0; c < nc; c++) rows[c + 1] += rows[c];
    perm.assign(A.n, 0);
    std::vector<int> fill(rows.begin(), rows.end() - 1);
    for (int i = 0; i < A.n; i++) perm[fill[col[i]]++] = i;
    Csr Ac;
    Ac.n = A.n;
    Ac.ncols = A.n;
    Ac.rp.assign(A.n + 1, 0);
    Ac.ci.reserve(A.nnz());
    Ac.v.reserve(A.nnz());
    for (int r = 0; r < A.n; r++) {
        const int i = perm[r];
        Ac.ci.insert(Ac.ci.end(), A.ci.begin() + A.rp[i], A.ci.begin() + A.rp[i + 1]);
        Ac.v.insert(Ac.v.end(), A.v.begin() + A.rp[i], A.v.begin() + A.rp[i + 1]);
        Ac.rp[r + 1] = (int)Ac.ci.size();
    }
    return Ac;
}

// the slices of a colour-permuted copy's two precisions
static PairPlan plan_colours(const Csr& Ac, const std::vector<int>& rows, bool free32,
                             const TunedLanes* tuned = nullptr) {
    PairPlan q;
    if (!tuned) {
        q.p64 = rule_slices(Ac, rows, true, true);
        q.p32 = rule_slices(Ac, rows, free32, false);
    } else {
        if (tuned->s64) q.p64 = plan_slices(Ac, rows, log2_of(tuned->l64));
        if (tuned->s32) q.p32 = plan_slices(Ac, rows, log2_of(tuned->l32));
    }
    q.shared = same_rows(q.p64, q.p32);
    return q;
}

std::vector<dev::SliceHead> slice_layout(const Csr& A, const int* colours, bool free32, bool partials, int precision,
                                         int* lt, size_t* steps) {
    PairPlan q;
    if (colours) {
        std::vector<int> col(colours, colours + A.n), perm, rows;
        const int nc = A.n > 0 ? *std::max_element(col.begin(), col.end()) + 1 : 0;
        for (int c : col)
            if (c < 0) throw std::invalid_argument("negative colour");
        q = plan_colours(colour_permuted(A, col, nc, perm, rows), rows, free32);
    } else {
        q = plan_pair(A, false, free32, partials);
    }
    const bool fp64 = precision == LINA_PREC_FP64;
    const SlicePlan& own = fp64 ? q.p64 : q.p32;
    *lt = own.lt;
    *steps = own.steps;
    return !fp64 && q.shared ? q.p64.head : own.head;
}

// level schedule of the lexicographic sweep: forward, level(i) = 1 + max over
// j<i with a_ij != 0; backward, over j>i
static void level_schedule(const Csr& A, bool backward, std::vector<int>& off, std::vector<int>& rows) {
    const int n = A.n;
    std::vector<int> lev(n, 0);
    int nl = 0;
    for (int t = 0; t < n; t++) {
        int i = backward ? n - 1 - t : t;
        int l = 0;
        for (int p = A.rp[i]; p < A.rp[i + 1]; p++) {
            int j = A.ci[p];
            if (A.v[p] == 0.0) continue;
            if ((!backward && j < i) || (backward && j > i)) l = std::max(l, lev[j] + 1);
        }
        lev[i] = l;
        nl = std::max(nl, l + 1);
    }
    off.assign(nl + 1, 0);
    for (int i = 0; i < n; i++) off[lev[i] + 1]++;
    for (int l = 0; l < nl; l++) off[l + 1] += off[l];
    rows.assign(n, 0);
    std::vector<int> fill(off.begin(), off.end() - 1);
    for (int i = 0; i < n; i++) rows[fill[lev[i]]++] = i;
}

// ------------------------------------------------------------ Solver

Solver::Solver() {}

Solver::~Solver() {
    if (stream_) (void)hipStreamSynchronize(stream_);
    iteration_.reset();
    if (ev0_) (void)hipEventDestroy(ev0_);
    if (ev1_) (void)hipEventDestroy(ev1_);
    for (auto& pr : evk_)
        for (hipEvent_t e : pr)
            if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : evr_)
        if (e) (void)hipEventDestroy(e);
    if (host_scal_) (void)hipHostFree(host_scal_);
    if (host_ring_) (void)hipHostFree(host_ring_);
    bufs_.reset();
    if (stream_) (void)hipStreamDestroy(stream_);
}

void Solver::setup_host(const Csr& A, const lina_amg_params& p) {
    prm_ = p;
    SetupParams sp;
    sp.dof = p.dof;
    sp.depth = p.depth;
    sp.smoothing_iterations = p.smoothing_iterations;
    sp.aggr_smoothing_iterations = p.aggr_smoothing_iterations;
    sp.coarsening = p.coarsening;
    sp.eps_minus = p.eps_minus;
    sp.eps_plus = p.eps_plus;
    sp.matrix_tol = p.matrix_tol;
    amg_setup(A, sp, H_);
    tuned_.clear();
    n_ = A.n;
    colours_.assign(H_.lv.size(), std::vector<int>());
    ncolours_.assign(H_.lv.size(), 0);
    for (size_t l = 1; l < H_.lv.size(); l++) colours_[l] = greedy_colouring(H_.lv[l].A, &ncolours_[l]);
}

// ------------------------------------------------------- autotuning

namespace {
constexpr int kLaneCandidates[] = {1, 4, 8, 16, 32};
}

// device arrays that the candidates of one tuning are laid out in, one after another
struct Solver::SliceScratch {
    DevBuffers bufs;
    size_t heads = 0, entries = 0;
    dev::SliceHead* head = nullptr;
    uint16_t* cs = nullptr;
    double* v = nullptr;  // or as many floats
    void hold(size_t nh, size_t ne) {
        if (nh <= heads && ne <= entries) return;
        heads = std::max(nh, 2 * heads);
        entries = std::max(ne, 2 * entries);
        bufs = DevBuffers();  // the last candidate's timing has ended
        head = dalloc<dev::SliceHead>(heads, bufs);
        cs = dalloc<uint16_t>(entries, bufs);
        v = dalloc<double>(entries, bufs);
    }
};

// The form of M (rows: A's) whose launches are fastest: a sliced copy with each
// lane count, laid out in scratch memory, and the row blocks with each where M
// has them.  groups: a colour-permuted copy's (offsets: its sweep's offsets of
// slices or blocks).  What M has stays unless another is 3 % faster.
template <typename VT>
Solver::Form Solver::tune_form(const Csr& A, const std::vector<int>& groups, const dev::DMat<VT>& M,
                               const std::vector<int>& offsets, SliceScratch& scratch,
                               const std::function<void(const dev::DMat<VT>&, const std::vector<int>&)>& run) {
    const Form have = form_of(M);
    if (M.n == 0 || M.nnz == 0) return have;
    auto timed = [&](const dev::DMat<VT>& T, const std::vector<int>& off) {
        run(T, off);
        float t = 1e30f;
        for (int rep = 0; rep < 2; rep++) {
            hip_check(hipEventRecord(ev0_, stream_), "event");
            for (int k = 0; k < 3; k++) run(T, off);
            hip_check(hipEventRecord(ev1_, stream_), "event");
            hip_check(hipEventSynchronize(ev1_), "event sync");
            float ms = 0;
            hip_check(hipEventElapsedTime(&ms, ev0_, ev1_), "elapsed");
            t = std::min(t, ms);
        }
        return t;
    };
    Form best = have;
    float best_t = 0.97f * timed(M, offsets);
    auto keep = [&](float t, Form f) {
        if (t < best_t) {
            best_t = t;
            best = f;
        }
    };
    for (int lanes : kLaneCandidates) {
        if (lanes > 4 && (double)lanes * M.n > M.nnz) break;  // less than an entry a lane
        if (!have.sliced && lanes != have.lanes) {
            dev::DMat<VT> T = M;
            T.lpr = lanes;
            keep(timed(T, offsets), {lanes, false});
        }
        if (have.sliced && lanes == have.lanes) continue;
        const SlicePlan p = plan_slices(A, groups, log2_of(lanes));
        if (p.head.empty()) continue;
        validate(A, p);
        scratch.hold(p.head.size(), p.steps * 64);
        dev::DMat<VT> T = M;
        T.bspec = nullptr;
        T.sl = slice_shape<VT>(p);
        T.sl.head = scratch.head;
        T.sl.cs = scratch.cs;
        T.sl.v = (VT*)scratch.v;
        hip_check(hipMemcpyAsync(T.sl.head, p.head.data(), p.head.size() * sizeof(dev::SliceHead),
                                 hipMemcpyHostToDevice, stream_), "h2d");
        dev::slice_columns<VT>(stream_, T);
        dev::slice_values<VT>(stream_, T);
        keep(timed(T, p.group), {lanes, true});
    }
    return best;
}

// M in another form; share: the other precision's copy where it has that form
template <typename VT, typename OT>
void Solver::adopt_form(const Csr& A, const std::vector<int>& groups, dev::DMat<VT>& M, Form f,
                        const dev::DMat<OT>* share, std::vector<int>* offsets, const std::vector<int>* seg,
                        const int* row_ids) {
    if (!f.sliced) {  // only where M has row blocks already
        M.lpr = f.lanes;
        return;
    }
    const SlicePlan p = plan_slices(A, groups, log2_of(f.lanes));
    make_slices<VT, OT>(p, M, *bufs_, stream_, share);
    if (offsets) *offsets = p.group;
    if (seg) M.bspec = dupload(block_systems(slice_starts(A, p), *seg, row_ids), *bufs_, stream_);
    hip_check(hipStreamSynchronize(stream_), "adopt");  // the host plan dies here
}

// both copies of a matrix in the forms timed fastest; the slices that neither
// reads any more are freed
void Solver::adopt_forms(const Csr& A, const std::vector<int>& groups, dev::DMat<double>& D, dev::DMat<float>& F,
                         Form a, Form b, std::vector<int>* off64, std::vector<int>* off32,
                         const std::vector<int>* seg, const int* row_ids) {
    const dev::Slices<double> d0 = D.sl;
    const dev::Slices<float> f0 = F.sl;
    auto same = [](Form x, Form y) { return x.sliced == y.sliced && x.lanes == y.lanes; };
    if (!same(a, form_of(D))) adopt_form<double, double>(A, groups, D, a, nullptr, off64, seg, row_ids);
    if (!same(b, form_of(F)))
        adopt_form<float, double>(A, groups, F, b, same(a, b) && a.sliced ? &D : nullptr, off32, seg, row_ids);
    auto drop = [&](void* p, size_t bytes) {
        if (p) bufs_->drop(p, bytes);
    };
    if (D.sl.head != d0.head && F.sl.head != d0.head) drop(d0.head, d0.ns * sizeof(dev::SliceHead));
    if (f0.head != d0.head && F.sl.head != f0.head) drop(f0.head, f0.ns * sizeof(dev::SliceHead));
    if (D.sl.v != d0.v) drop(d0.v, d0.steps * 64 * sizeof(double));
    if (F.sl.v != f0.v) drop(f0.v, f0.steps * 64 * sizeof(float));
    if (D.sl.cs != d0.cs && F.sl.cs != d0.cs) drop(d0.cs, d0.steps * 64 * sizeof(uint16_t));
    if (f0.cs != d0.cs && F.sl.cs != f0.cs) drop(f0.cs, f0.steps * 64 * sizeof(uint16_t));
}

// The row partition (slices or row blocks, lanes per row) of every matrix of the
// hierarchy, chosen by timing each candidate on the device: the SpMV-shaped kernels (residual,
// restriction, prolongation, Jacobi) take their matrix's choice, the
// multicolour sweeps the colour-permuted copy's.
void Solver::autotune() {
    hipStream_t st = stream_;
    tuned_.clear();
    SliceScratch scratch;
    auto note = [&](int l, char which, Form a, Form b) {
        tuned_.push_back({l, which, a.lanes, b.lanes, a.sliced, b.sliced});
    };
    auto product = [&](int l, char which, const Csr& M0, dev::DMat<double>& D, dev::DMat<float>& F, const double* x,
                       double* y, const float* xf, float* yf, const std::vector<int>* seg) {
        const Csr M = which == 'A' ? Csr() : drop_outside_zeros(M0);  // A has none
        const Csr& A = which == 'A' ? M0 : M;
        const Form a = tune_form<double>(A, {}, D, {}, scratch,
                                         [&](const dev::DMat<double>& T, const std::vector<int>&) {
            dev::spmv<double, double>(st, T, x, nullptr, y, dev::MODE_SET, nullptr, nullptr);
        });
        const Form b = tune_form<float>(A, {}, F, {}, scratch,
                                        [&](const dev::DMat<float>& T, const std::vector<int>&) {
            dev::spmv<float, float>(st, T, xf, nullptr, yf, dev::MODE_SET, nullptr, nullptr);
        });
        adopt_forms(A, {}, D, F, a, b, nullptr, nullptr, seg, nullptr);
        note(l, which, a, b);
    };
    auto segs = [&](size_t l) { return seg_off_.empty() ? nullptr : &seg_off_[l]; };
    for (size_t l = 0; l < L_.size(); l++) {
        DevLevel& d = L_[l];
        const HostLevel& h = H_.lv[l];
        for (double* v : {d.x, d.f, d.r, d.xo}) dev::fill<double>(st, d.n, v, 1.0);
        for (float* v : {d.xf, d.ff, d.rf, d.xof}) dev::fill<float>(st, d.n, v, 1.0f);
        product((int)l, 'A', h.A, d.A, d.Af, d.x, d.r, d.xf, d.rf, segs(l));
        if (l == 0) continue;
        DevLevel& c = L_[l - 1];
        for (double* v : {c.x, c.f}) dev::fill<double>(st, c.n, v, 1.0);
        for (float* v : {c.xf, c.ff}) dev::fill<float>(st, c.n, v, 1.0f);
        product((int)l, 'P', h.P, d.P, d.Pf, c.x, d.r, c.xf, d.rf, segs(l));
        product((int)l, 'R', h.R, d.R, d.Rf, d.r, c.f, d.rf, c.ff, segs(l - 1));
        dev::fill<double>(st, d.n, d.f, 0.0);
        dev::fill<float>(st, d.n, d.ff, 0.0f);
        if (d.ncolours == 0) continue;
        std::vector<int> perm, rows;
        const Csr Ac = colour_permuted(h.A, colours_[l], ncolours_[l], perm, rows);
        const Form a = tune_form<double>(Ac, rows, d.Ac, d.colour_blk, scratch,
                                         [&](const dev::DMat<double>& T, const std::vector<int>& cb) {
            for (int c = 0; c < d.ncolours; c++)
                dev::mcsor_colour(st, T, cb[c], cb[c + 1] - cb[c], d.perm, (const double*)d.f, d.x, 1.0);
        });
        const Form b = tune_form<float>(Ac, rows, d.Acf, d.colour_blk32, scratch,
                                        [&](const dev::DMat<float>& T, const std::vector<int>& cb) {
            for (int c = 0; c < d.ncolours; c++)
                dev::mcsor_colour(st, T, cb[c], cb[c + 1] - cb[c], d.perm, (const float*)d.ff, d.xf, 1.0f);
        });
        adopt_forms(Ac, rows, d.Ac, d.Acf, a, b, &d.colour_blk, &d.colour_blk32, segs(l), perm.data());
        note((int)l, 'C', a, b);
    }
    hip_check(hipStreamSynchronize(st), "autotune");
}

// the autotuner's lanes of a matrix, or nullptr before it has run
const TunedLanes* Solver::tuned_lanes(int l, char which, TunedLanes& t) const {
    for (const Tuned& q : tuned_)
        if (q.level == l && q.which == which) {
            t = {q.lpr64, q.lpr32, q.s64, q.s32};
            return &t;
        }
    return nullptr;
}

void Solver::set_hierarchy(HostHierarchy&& H, const lina_amg_params& p) {
    prm_ = p;
    H_ = std::move(H);
    tuned_.clear();
    n_ = H_.lv.back().A.n;
    colours_.assign(H_.lv.size(), std::vector<int>());
    ncolours_.assign(H_.lv.size(), 0);
    for (size_t l = 1; l < H_.lv.size(); l++) colours_[l] = greedy_colouring(H_.lv[l].A, &ncolours_[l]);
}

void Solver::upload() {
    if (!stream_) {
        hip_check(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking), "hipStreamCreate");
        hip_check(hipEventCreate(&ev0_), "hipEventCreate");
        hip_check(hipEventCreate(&ev1_), "hipEventCreate");
        hip_check(hipHostMalloc((void**)&host_scal_, dev::S_COUNT * sizeof(double)), "hipHostMalloc");
        hip_check(hipHostMalloc((void**)&host_ring_, 2 * dev::S_COUNT * sizeof(double)), "hipHostMalloc");
        for (hipEvent_t& e : evr_) hip_check(hipEventCreate(&e), "hipEventCreate");
    }
    // a re-upload (recompute) frees every earlier buffer, including the
    // BiCGStab work vectors allocated on first use
    hip_check(hipStreamSynchronize(stream_), "sync");
    iteration_.reset();
    if (bufs_ && (host_stale_ || host_top_stale_)) sync_host_levels();  // values of a device recompute
    rap_.reset();  // the device products' plans belong to the patterns uploaded before
    host_stale_ = false;
    host_top_stale_ = false;
    neg_rows_ = nullptr;
    iso_pos_ = nullptr;
    iso_val_ = nullptr;
    niso_pos_ = 0;
    iso_pos_host_.clear();
    bufs_.reset(new DevBuffers());
    for (double** p : {&bS_, &bPS_, &bPP_, &bAPP_, &bAPS_, &bR_, &bR0_, &bP_}) *p = nullptr;
    DevBuffers& B = *bufs_;
    hipStream_t st = stream_;
    const int depth = (int)H_.lv.size();
    L_.assign(depth, DevLevel());
    up_.assign(track_ ? depth : 0, UpLevel());
    int maxn = 1, maxblk = 1;
    for (int l = 0; l < depth; l++) {
        const HostLevel& h = H_.lv[l];
        DevLevel& d = L_[l];
        d.n = h.A.n;
        maxn = std::max(maxn, d.n);
        const std::vector<int>* segl = seg_off_.empty() ? nullptr : &seg_off_[l];
        TunedLanes tl;
        maxblk = std::max(maxblk, upload_pair(h.A, d.A, d.Af, B, st, segl, !fixed_order(), l == depth - 1,
                                              tuned_lanes(l, 'A', tl)));
        d.x = dalloc<double>(d.n, B);
        d.f = dalloc<double>(d.n, B);
        d.r = dalloc<double>(d.n, B);
        d.xo = dalloc<double>(d.n, B);
        d.xf = dalloc<float>(d.n, B);
        d.ff = dalloc<float>(d.n, B);
        d.rf = dalloc<float>(d.n, B);
        d.xof = dalloc<float>(d.n, B);
        d.nlim = (d.n / std::max(1, prm_.dof)) * std::max(1, prm_.dof);
        if (track_) {
            up_[l].rp = h.A.rp;
            up_[l].ci = h.A.ci;
        }
        if (l == 0) continue;
        maxblk = std::max(maxblk, upload_pair(h.P, d.P, d.Pf, B, st, segl, !fixed_order(), false,
                                              tuned_lanes(l, 'P', tl)));
        maxblk = std::max(maxblk, upload_pair(h.R, d.R, d.Rf, B, st, seg_off_.empty() ? nullptr : &seg_off_[l - 1],
                                              !fixed_order(), false, tuned_lanes(l, 'R', tl)));
        // colour-permuted copy for the multicolour sweeps
        const std::vector<int>& col = colours_[l];
        int nc = ncolours_[l];
        std::vector<int> perm;
        const Csr Ac = colour_permuted(h.A, col, nc, perm, d.colour_rows);
        // colour c's rows form the slices or blocks [colour_blk[c], colour_blk[c+1])
        auto colour_schedule = [&](int max_nnz, std::vector<int>& cb) {
            std::vector<int> starts;
            cb.assign(nc + 1, 0);
            for (int c = 0; c < nc; c++) {
                cb[c] = (int)starts.size();
                build_blocks(Ac, d.colour_rows[c], d.colour_rows[c + 1], max_nnz, starts);
            }
            cb[nc] = (int)starts.size();
            starts.push_back(d.n);
            return starts;
        };
        const TunedLanes* tuned = tuned_lanes(l, 'C', tl);
        PairPlan q = plan_colours(Ac, d.colour_rows, !fixed_order(), tuned);
        if (q.p64.head.empty()) q.s64 = colour_schedule(dev::block_nnz<double>(), d.colour_blk);
        else d.colour_blk = q.p64.group;
        if (q.p32.head.empty()) q.s32 = colour_schedule(dev::block_nnz<float>(), d.colour_blk32);
        else d.colour_blk32 = q.p32.group;
        upload_mat<double, double>(Ac, q.p64, q.s64, d.Ac, B, st, nullptr, false, nullptr, perm.data(), segl);
        upload_mat(Ac, q.p32, q.s32, d.Acf, B, st, &d.Ac, q.shared, &q.s64, perm.data(), segl);
        if (tuned && !d.Ac.sl.ns) d.Ac.lpr = tuned->l64;
        if (tuned && !d.Acf.sl.ns) d.Acf.lpr = tuned->l32;
        d.perm = dupload(perm, B, st);
        d.ncolours = nc;
        if (track_) {
            up_[l].colour = col;
            up_[l].perm = perm;
        }
        // level schedules of the exact lexicographic sweeps
        std::vector<int> off, rows;
        level_schedule(h.A, false, off, rows);
        d.nlv_f = (int)off.size() - 1;
        d.lvf_off = dupload(off, B, st);
        d.lvf_rows = dupload(rows, B, st);
        if (track_) {
            up_[l].lvf_off = off;
            up_[l].lvf_rows = rows;
        }
        level_schedule(h.A, true, off, rows);
        d.nlv_b = (int)off.size() - 1;
        d.lvb_off = dupload(off, B, st);
        d.lvb_rows = dupload(rows, B, st);
        if (track_) {
            up_[l].lvb_off = off;
            up_[l].lvb_rows = rows;
        }
        if (lex_smoothing()) build_sor_packs(l, B, false);
    }
    // finest-level extras
    signs_ = dupload(H_.signs, B, st);
    has_neg_signs_ = false;
    for (double s : H_.signs)
        if (s < 0) has_neg_signs_ = true;
    iso_rows_ = dupload(H_.iso_rows, B, st);
    iso_a_ = dupload(H_.iso_a, B, st);
    niso_ = (int)H_.iso_rows.size();
    // the isolated rows' diagonals by row for the fused preconditioner entry
    // and exit (a zero diagonal keeps the separate kernels)
    isa_ = nullptr;
    isb_ = nullptr;
    isa_ok_ = true;
    if (niso_ > 0) {
        std::vector<double> isa(n_, 0.0);
        std::vector<uint32_t> isb((n_ + 31) / 32, 0u);
        for (int k = 0; k < niso_; k++) {
            const int i = H_.iso_rows[k];
            if (H_.iso_a[k] == 0.0) isa_ok_ = false;
            isa[i] = H_.iso_a[k];
            isb[i >> 5] |= 1u << (i & 31);
        }
        if (isa_ok_) {
            isa_ = dupload(isa, B, st);
            isb_ = dupload(isb, B, st);
        }
    }
    // coarse LU inverse
    const CoarseLU& lu = H_.lu;
    nd_ = (int)lu.dense_idx.size();
    nt_ = (int)lu.trivial_idx.size();
    didx_ = dupload(lu.dense_idx, B, st);
    inv_ = dupload(lu.dense, B, st);
    cbatched_ = lu.blk_off.size() > 2;
    if (cbatched_) {
        // block-diagonal coarsest level of a batch: one inverse per block
        const int nb = (int)lu.blk_off.size() - 1;
        std::vector<int> rblk(nd_);
        int maxb = 0;
        for (int b = 0; b < nb; b++) {
            maxb = std::max(maxb, lu.blk_off[b + 1] - lu.blk_off[b]);
            for (int g = lu.blk_off[b]; g < lu.blk_off[b + 1]; g++) rblk[g] = b;
        }
        crblk_ = dupload(rblk, B, st);
        coff_ = dupload(lu.blk_off, B, st);
        cmoff_ = dupload(lu.mat_off, B, st);
        double* piv = dalloc<double>(nb, B);
        dev::batched_gauss_jordan_inverse(st, nd_, maxb, crblk_, coff_, cmoff_, inv_, piv);
    } else {
        cpiv_ = dalloc<double>(dev::gauss_jordan_work(nd_), B);
        dev::gauss_jordan_inverse(st, nd_, inv_, cpiv_);
    }
    up_dense_ = lu.dense_idx;
    up_trivial_ = lu.trivial_idx;
    // gathered right-hand side, padded with zeros to whole tiles of the FP32 inverse
    const int nbd = std::max((nd_ + dev::CT - 1) / dev::CT * dev::CT, dev::CT);
    cbd_ = dalloc<double>(nbd, B);
    dev::fill<double>(st, nbd, cbd_, 0.0);
    // dense index of each coarsest row (restriction epilogue) and whether the
    // dense and trivial rows cover the level (no zero fill needed)
    dinv_ = nullptr;
    ccover_ = false;
    if (!cbatched_) {
        const int n0 = L_[0].n;
        std::vector<int> dinv(n0, -1), seen(n0, 0);
        bool ok = true;
        for (int g = 0; g < nd_ && ok; g++) {
            const int r = lu.dense_idx[g];
            if (r < 0 || r >= n0 || seen[r]++) ok = false;
            else dinv[r] = g;
        }
        for (int t = 0; t < nt_ && ok; t++) {
            const int r = lu.trivial_idx[t];
            if (r < 0 || r >= n0 || seen[r]++) ok = false;
        }
        if (ok) {
            dinv_ = dupload(dinv, B, st);
            ccover_ = nd_ + nt_ == n0;
        }
    }
    ctiles_ = nullptr;
    nct_ = ntiles_ = 0;
    tidx_ = dupload(lu.trivial_idx, B, st);
    tdiag_ = dupload(lu.trivial_diag, B, st);
    // Krylov vectors and scratch
    const int n = n_;
    ftop_ = dalloc<double>(n, B);
    rtop_ = dalloc<double>(n, B);
    kR_ = dalloc<double>(n, B);
    kP_ = dalloc<double>(n, B);
    kQ_ = dalloc<double>(n, B);
    kZ_ = dalloc<double>(n, B);
    kW_ = dalloc<double>(n, B);
    kX_ = dalloc<double>(n, B);
    kB_ = dalloc<double>(n, B);
    // block partials: one per SpMV workgroup (any matrix, and any sliced operator
    // of this size: at least 2 rows a slice, 4 slices a workgroup) or per
    // reduction block
    int np = std::max({4096, maxblk + 16, n / (2 * dev::SLICES_PER_BLOCK) + 32});
    part_ = dalloc<double>(np + 3 * dev::DOT_PART_MAX, B);  // and three dots' partials beside a product's
    part_cap_ = np;
    scal_ = dalloc<double>(dev::S_COUNT, B);
    dev::fill(st, dev::S_COUNT, scal_, 0.0);
    hip_check(hipStreamSynchronize(st), "upload sync");
    ensure_ctiles();
    if (prm_.autotune && tuned_.empty()) autotune();  // later uploads keep its choices
}

void Solver::set_params(const lina_amg_params& p) { prm_ = p; }

void Solver::set_segments(std::vector<std::vector<int>> off) {
    if (!off.empty() && off.size() != H_.lv.size()) throw std::invalid_argument("segments: one offset list per level");
    seg_off_ = std::move(off);
}

void Solver::set_active(const double* active) {
    if (seg_off_.empty()) throw std::logic_error("set_active without segments");
    for (DevLevel& d : L_) {
        for (auto* m : {&d.A, &d.P, &d.R, &d.Ac}) m->active = m->bspec ? active : nullptr;
        for (auto* m : {&d.Af, &d.Pf, &d.Rf, &d.Acf}) m->active = m->bspec ? active : nullptr;
    }
    seg_active_ = active;
}

// The coarse inverse's upper triangle as FP64 tiles of CT x CT, read by
// both precisions' V-cycles (half the bytes of the full inverse, exactly
// symmetric).  FP32 tiles were measured: 35 % more CG iterations on the
// high-contrast adjoint system, none on the elasticity benchmark.
void Solver::ensure_ctiles() {
    if (ctiles_ || cbatched_ || nd_ == 0 || !uploaded()) return;
    nct_ = (nd_ + dev::CT - 1) / dev::CT;
    std::vector<int> ti, tj;
    for (int I = 0; I < nct_; I++)
        for (int J = I; J < nct_; J++) {
            ti.push_back(I);
            tj.push_back(J);
        }
    ntiles_ = (int)ti.size();
    cti_ = dupload(ti, *bufs_, stream_);
    ctj_ = dupload(tj, *bufs_, stream_);
    cpart_ = dalloc<double>((size_t)nct_ * nct_ * dev::CT, *bufs_);
    ctiles_ = dalloc<double>((size_t)ntiles_ * dev::CT * dev::CT, *bufs_);
    dev::inverse_to_tiles<double>(stream_, nd_, ntiles_, cti_, ctj_, inv_, ctiles_);
    hip_check(hipStreamSynchronize(stream_), "sync");
}

// whether any level sweeps with the exact lexicographic SOR / SSOR
bool Solver::lex_smoothing() const {
    auto lex = [](int sm) { return sm == LINA_SMOOTHER_SOR || sm == LINA_SMOOTHER_SSOR; };
    return lex(prm_.smoother) || lex(prm_.coarse_smoother);
}

// The level-packed forms (dev::SorPack) of level l's exact lexicographic
// sweeps, from the host matrix and the level schedules: new entries (earlier
// rows in the sweep's order, nonzero, as the schedule counts them) in the
// records (past 4 or 8 in overflow arrays), old entries (all, zero or not)
// in the slot-major lists and their overflow.  Not built (the level keeps
// k_sor_lex) when a row lacks its diagonal.  reuse: the device arrays of the
// level's packs are rewritten in place when their sizes still fit.
void Solver::build_sor_packs(int l, DevBuffers& B, bool reuse) {
    DevLevel& d = L_[l];
    reuse = reuse && d.sor_packed;
    d.sor_packed = false;
    const Csr& A = H_.lv[l].A;
    const int n = A.n;
    if (n == 0) return;
    hipStream_t st = stream_;
    std::vector<int> off, rows;
    int maxc = 0;
    for (int i = 0; i < n; i++) {
        int nl = 0, nu = 0, dg = 0;
        for (int p = A.rp[i]; p < A.rp[i + 1]; p++) {
            const int j = A.ci[p];
            if (j == i) dg++;
            else if (j < i) nl++;
            else nu++;
        }
        if (dg != 1) return;
        maxc = std::max(maxc, std::max(nl, nu));
    }
    const int maxp = maxc <= 4 ? 4 : 8;
    for (int back = 0; back < 2; back++) {
        level_schedule(A, back != 0, off, rows);
        const int nlv = (int)off.size() - 1;
        std::vector<int> pos(n), lev(n);
        for (int L = 0; L < nlv; L++)
            for (int t = off[L]; t < off[L + 1]; t++) {
                pos[rows[t]] = t;
                lev[rows[t]] = L;
            }
        const size_t N = (size_t)n;
        std::vector<int> full(std::max(nlv, 1), 0), ocnt(n), ocol(maxp * N, 0), ovp(n, 0), ovsrc, ooff(n, 0), oovc;
        std::vector<double> oval(maxp * N, 0.0), ovval, oovv;
        std::vector<char> rec(N * (maxp == 4 ? sizeof(dev::TriRec<4>) : sizeof(dev::TriRec<8>)));
        for (int t = 0; t < n; t++) {
            const int i = rows[t], L = lev[i], e = off[L + 1];
            double diag = 0;
            double val[8];
            int src[8];
            for (int k = 0; k < 8; k++) {
                val[k] = 0.0;
                src[k] = dev::TRI_RING;
            }
            int kn = 0, ko = 0;
            ovp[t] = (int)ovval.size();
            ooff[t] = (int)oovv.size();
            for (int p = A.rp[i]; p < A.rp[i + 1]; p++) {
                const int j = A.ci[p];
                if (j == i) {
                    diag = A.v[p];
                } else if ((j < i) != (back != 0)) {  // new value
                    if (A.v[p] == 0.0) continue;
                    int sj;
                    if (e - pos[j] <= dev::TRI_RING) {
                        sj = pos[j] & (dev::TRI_RING - 1);
                    } else {
                        sj = -(j + 1);
                        full[L] = 1;
                    }
                    if (kn < maxp) {
                        val[kn] = A.v[p];
                        src[kn] = sj;
                    } else {
                        ovval.push_back(A.v[p]);
                        ovsrc.push_back(sj);
                    }
                    kn++;
                } else {  // old value
                    if (ko < maxp) {
                        oval[ko * N + t] = A.v[p];
                        ocol[ko * N + t] = j;
                    } else {
                        oovv.push_back(A.v[p]);
                        oovc.push_back(j);
                    }
                    ko++;
                }
            }
            ocnt[t] = ko;
            if (maxp == 4) {
                dev::TriRec<4>& r = reinterpret_cast<dev::TriRec<4>*>(rec.data())[t];
                r.diag = diag;
                for (int k = 0; k < 4; k++) {
                    r.val[k] = val[k];
                    r.src[k] = src[k];
                }
                r.orow = i;
                r.cnt = kn;
            } else {
                dev::TriRec<8>& r = reinterpret_cast<dev::TriRec<8>*>(rec.data())[t];
                r.diag = diag;
                for (int k = 0; k < 8; k++) {
                    r.val[k] = val[k];
                    r.src[k] = src[k];
                }
                r.orow = i;
                r.cnt = kn;
            }
        }
        for (int L = 0; L < nlv; L++)
            if (full[L]) off[L] |= (int)0x80000000u;
        dev::SorPack& S = back ? d.sorb : d.sorf;
        std::vector<int>& used = back ? d.sor_sizes_b : d.sor_sizes_f;
        const std::vector<int> sizes = {(int)ovval.size(), (int)oovv.size()};
        if (reuse && used == sizes) {
            // same pattern and schedules (checked by the caller) and overflow sizes
            auto to = [&](const void* dst, const void* src, size_t bytes) {
                if (bytes)
                    hip_check(hipMemcpyAsync(const_cast<void*>(dst), src, bytes, hipMemcpyHostToDevice, st), "h2d");
            };
            to(S.p.off, off.data(), off.size() * sizeof(int));
            to(S.p.rec, rec.data(), rec.size());
            to(S.p.ovp, ovp.data(), ovp.size() * sizeof(int));
            to(S.p.ovval, ovval.data(), ovval.size() * sizeof(double));
            to(S.p.ovsrc, ovsrc.data(), ovsrc.size() * sizeof(int));
            to(S.row, rows.data(), rows.size() * sizeof(int));
            to(S.ocnt, ocnt.data(), ocnt.size() * sizeof(int));
            to(S.oval, oval.data(), oval.size() * sizeof(double));
            to(S.ocol, ocol.data(), ocol.size() * sizeof(int));
            to(S.ooff, ooff.data(), ooff.size() * sizeof(int));
            to(S.oovv, oovv.data(), oovv.size() * sizeof(double));
            to(S.oovc, oovc.data(), oovc.size() * sizeof(int));
            hip_check(hipStreamSynchronize(st), "sync");  // the host arrays die here
            continue;
        }
        used = sizes;
        S = dev::SorPack();
        S.p.n = n;
        S.p.nlv = nlv;
        S.p.maxp = maxp;
        S.p.off = dupload(off, B, st);
        S.p.rec = dupload(rec, B, st);
        S.p.ovp = dupload(ovp, B, st);
        S.p.ovval = dupload(ovval, B, st);
        S.p.ovsrc = dupload(ovsrc, B, st);
        S.row = dupload(rows, B, st);
        S.ocnt = dupload(ocnt, B, st);
        S.oval = dupload(oval, B, st);
        S.ocol = dupload(ocol, B, st);
        S.ooff = dupload(ooff, B, st);
        S.oovv = dupload(oovv, B, st);
        S.oovc = dupload(oovc, B, st);
        S.old_first = back;
        S.in = dalloc<double>(n, B);
        S.a = dalloc<double>(n, B);
        S.prod = dalloc<double>(maxp * N, B);
        S.prodov = dalloc<double>(std::max<size_t>(oovv.size(), 1), B);
        dev::fill<double>(st, (int)(maxp * N), S.prod, 0.0);
        hip_check(hipStreamSynchronize(st), "sync");  // the host arrays die here
    }
    d.sor_packed = true;
}

// host l1 norms of a matrix's rows as upload_mat forms them (VT arithmetic)
template <typename VT>
static std::vector<VT> row_l1(const Csr& A) {
    std::vector<VT> l1(A.n, (VT)0);
    for (int r = 0; r < A.n; r++) {
        VT s = 0;
        for (int p = A.rp[r]; p < A.rp[r + 1]; p++) s += std::fabs((VT)A.v[p]);
        l1[r] = s;
    }
    return l1;
}

void Solver::refresh_after_recompute() {
    const bool timing = getenv("LINA_RN_TIMING") != nullptr;  // read per call: recomputes are rare
    const auto t0 = std::chrono::steady_clock::now();
    for (size_t l = 1; l < H_.lv.size(); l++) colours_[l] = greedy_colouring(H_.lv[l].A, &ncolours_[l]);
    const auto t1 = std::chrono::steady_clock::now();
    bool vals = false;
    if (uploaded()) {
        vals = refresh_values();
        vals = refresh_isolated() && vals;  // a full upload takes the isolated rows' divisors too
        if (!vals) {
            track_ = true;  // from now on upload() keeps what a values-only refresh compares
            upload();
        }
    } else {
        refresh_isolated();
    }
    if (timing) {
        const auto t2 = std::chrono::steady_clock::now();
        auto s = [](auto a, auto b) { return std::chrono::duration<double>(b - a).count(); };
        fprintf(stderr, "[amg] recompute: colouring %.3fs, %s upload %.3fs\n", s(t0, t1), vals ? "values" : "full",
                s(t1, t2));
    }
}

// The values-only re-upload after a recompute: every level's A (FP64, FP32,
// the colour-permuted copies and their row l1 norms) and the coarse inverse
// and tiles, when each level's pattern, colouring and lexicographic level
// schedules and the coarse LU's row split are those on the device (P, R and
// the autotuned lane counts stay).  False, with nothing changed, otherwise.
bool Solver::refresh_values() {
    const int depth = (int)H_.lv.size();
    if ((int)up_.size() != depth || (int)L_.size() != depth || cbatched_ || !seg_off_.empty()) return false;
    for (int l = 0; l < depth; l++) {
        const Csr& A = H_.lv[l].A;
        const UpLevel& u = up_[l];
        if (A.rp != u.rp || A.ci != u.ci || A.nnz() != L_[l].A.nnz) return false;
        if (l == 0) continue;
        if (colours_[l] != u.colour) return false;
        std::vector<int> off, rows;
        level_schedule(A, false, off, rows);
        if (off != u.lvf_off || rows != u.lvf_rows) return false;
        level_schedule(A, true, off, rows);
        if (off != u.lvb_off || rows != u.lvb_rows) return false;
    }
    const CoarseLU& lu = H_.lu;
    if (lu.dense_idx != up_dense_ || lu.trivial_idx != up_trivial_ || !cpiv_) return false;
    hipStream_t st = stream_;
    std::vector<std::vector<double>> keep;  // host staging alive until the copies are done
    std::vector<std::vector<float>> keepf;
    auto put = [&](double* d, std::vector<double> h) {
        keep.push_back(std::move(h));
        hip_check(hipMemcpyAsync(d, keep.back().data(), keep.back().size() * sizeof(double), hipMemcpyHostToDevice,
                                 st), "h2d");
    };
    auto putf = [&](float* d, std::vector<float> h) {
        keepf.push_back(std::move(h));
        hip_check(hipMemcpyAsync(d, keepf.back().data(), keepf.back().size() * sizeof(float), hipMemcpyHostToDevice,
                                 st), "h2d");
    };
    for (int l = 0; l < depth; l++) {
        const Csr& A = H_.lv[l].A;
        DevLevel& d = L_[l];
        put(d.A.v, A.v);
        dev::pair_values(st, d.A, d.Af);
        put(d.A.l1, row_l1<double>(A));
        putf(d.Af.l1, row_l1<float>(A));
        if (l == 0) continue;
        const std::vector<int>& perm = up_[l].perm;
        Csr Ac;
        Ac.n = A.n;
        Ac.rp.assign(A.n + 1, 0);
        Ac.v.reserve(A.nnz());
        for (int r = 0; r < A.n; r++) {
            const int i = perm[r];
            Ac.v.insert(Ac.v.end(), A.v.begin() + A.rp[i], A.v.begin() + A.rp[i + 1]);
            Ac.rp[r + 1] = (int)Ac.v.size();
        }
        put(d.Ac.l1, row_l1<double>(Ac));
        putf(d.Acf.l1, row_l1<float>(Ac));
        put(d.Ac.v, std::move(Ac.v));
        dev::pair_values(st, d.Ac, d.Acf);
        if (d.sor_packed) {
            hip_check(hipStreamSynchronize(st), "sync");
            build_sor_packs(l, *bufs_, true);  // the packs hold values: rewritten in place
        }
    }
    put(inv_, lu.dense);
    dev::gauss_jordan_inverse(st, nd_, inv_, cpiv_);
    put(tdiag_, lu.trivial_diag);
    if (ctiles_) dev::inverse_to_tiles<double>(st, nd_, ntiles_, cti_, ctj_, inv_, ctiles_);
    hip_check(hipStreamSynchronize(st), "refresh sync");
    return true;
}

void Solver::recompute(const std::vector<double>& val) {
    Csr A = H_.lv.back().A;  // pattern of the finest (sign-adjusted) matrix
    if ((int)val.size() != A.nnz()) throw std::invalid_argument("recompute: value count differs from the pattern");
    for (int i = 0; i < A.n; i++)
        for (int p = A.rp[i]; p < A.rp[i + 1]; p++) A.v[p] = val[p] * (H_.signs[i] < 0 ? -1.0 : 1.0);
    const bool timing = getenv("LINA_RN_TIMING") != nullptr;  // read per call: recomputes are rare
    if (device_rap_ok()) {
        const auto t0 = std::chrono::steady_clock::now();
        const bool built = rap_ != nullptr;
        const bool ok = recompute_device(A);
        if (timing) {
            const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            fprintf(stderr, "[amg] recompute on the device: %s %.3fs%s\n", ok ? "done" : "pattern changed", s,
                    built ? "" : " (plan built)");
        }
        if (ok) {
            H_.lv.back().A = std::move(A);
            host_stale_ = true;
            if (!refresh_isolated()) {
                sync_host_levels();
                upload();
            }
            return;
        }
    }
    sync_host_levels();
    amg_recompute(H_, A);
    refresh_after_recompute();
}

void Solver::recompute_matrix(const Csr& M) {
    if (M.n != n_) throw std::invalid_argument("recompute: matrix size differs from the hierarchy");
    const Csr& F = H_.lv.back().A;
    if (M.rp == F.rp && M.ci == F.ci) {  // the finest pattern holds: the values-only path
        recompute(M.v);
        return;
    }
    Csr A = M;
    for (int i = 0; i < A.n; i++)
        if (H_.signs[i] < 0)
            for (int p = A.rp[i]; p < A.rp[i + 1]; p++) A.v[p] = -A.v[p];
    sync_host_levels();
    amg_recompute(H_, A);
    refresh_after_recompute();
}

// AMG_fix_isolated (Multigrid.c:1301-1319) divides by the first nonzero of
// each isolated finest row: new finest values change the divisors
bool Solver::refresh_isolated() {
    if (host_top_stale_ && !H_.iso_rows.empty()) fetch_isolated_rows();
    const Csr& A = H_.lv.back().A;
    bool zero = false;
    for (size_t k = 0; k < H_.iso_rows.size(); k++) {
        const int i = H_.iso_rows[k];
        double a = 0.0;
        for (int p = A.rp[i]; p < A.rp[i + 1]; p++)
            if (A.v[p] != 0.0) {
                a = A.v[p];
                break;
            }
        H_.iso_a[k] = a;
        zero = zero || a == 0.0;
    }
    if (!uploaded() || niso_ == 0) return true;
    if (zero && isa_ok_) return false;  // the fused entry/exit kernels need nonzero divisors
    hip_check(hipMemcpyAsync(iso_a_, H_.iso_a.data(), (size_t)niso_ * sizeof(double), hipMemcpyHostToDevice, stream_),
              "h2d");
    if (isa_) {
        std::vector<double> isa(n_, 0.0);
        for (int k = 0; k < niso_; k++) isa[H_.iso_rows[k]] = H_.iso_a[k];
        hip_check(hipMemcpyAsync(isa_, isa.data(), (size_t)n_ * sizeof(double), hipMemcpyHostToDevice, stream_),
                  "h2d");
    }
    hip_check(hipStreamSynchronize(stream_), "sync");
    return true;
}

void Solver::set_operator(DevMatrix* op) {
    if (op) {
        if (op->n() != n_) throw std::invalid_argument("operator size differs from the hierarchy");
        if (op->nblocks() + 16 > part_cap_) throw std::invalid_argument("operator has more row blocks than the "
                                                                        "solver's partial-sum buffer");
        // the operator's own stream must be idle: its kernels now run on ours
        hip_check(hipStreamSynchronize(op->stream()), "sync");
    }
    op_ = op;
}

void Solver::set_kernel_timing(bool on) {
    if (on && !evk_[0][0])
        for (auto& pr : evk_)
            for (hipEvent_t& e : pr) hip_check(hipEventCreate(&e), "hipEventCreate");
    ktime_ = on;
}

double* Solver::dalloc_public(size_t n) { return dalloc<double>(n, *bufs_); }

// dL/dtheta of P1 plane-strain elements (host arrays in and out)
void Solver::elasticity_gradient(int n_nodes, const double* xy, int n_elem, const int* tri, double nu,
                                 const double* scale, int blocked, const double* u, const double* lam,
                                 double* grad) {
    DevBuffers B;
    auto up = [&](const void* h, size_t bytes) {
        void* d = nullptr;
        hip_check(hipMalloc(&d, std::max<size_t>(bytes, 8)), "hipMalloc");
        B.ptrs.push_back(d);
        if (h && bytes) hip_check(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, stream_), "h2d");
        return d;
    };
    const int n = 2 * n_nodes;
    auto* dxy = (const double*)up(xy, 2 * (size_t)n_nodes * sizeof(double));
    auto* dtri = (const int*)up(tri, 3 * (size_t)n_elem * sizeof(int));
    auto* du = (const double*)up(u, (size_t)n * sizeof(double));
    auto* dl = (const double*)up(lam, (size_t)n * sizeof(double));
    auto* ds = scale ? (const double*)up(scale, (size_t)n_elem * sizeof(double)) : nullptr;
    auto* dg = (double*)up(nullptr, (size_t)n_elem * sizeof(double));
    dev::elast_grad(stream_, n_elem, dtri, dxy, n_nodes, du, dl, nu, ds, blocked, dg);
    hip_check(hipMemcpyAsync(grad, dg, (size_t)n_elem * sizeof(double), hipMemcpyDeviceToHost, stream_), "d2h");
    hip_check(hipStreamSynchronize(stream_), "sync");
}

double Solver::read_scalar(int slot) {
    hip_check(hipMemcpyAsync(host_scal_ + slot, scal_ + slot, sizeof(double), hipMemcpyDeviceToHost, stream_), "d2h");
    hip_check(hipStreamSynchronize(stream_), "sync");
    return host_scal_[slot];
}

// ----------------------------------------------------------- smoothing

template <typename T>
static inline const dev::DMat<T>& pickA(const DevLevel& d);
template <>
inline const dev::DMat<double>& pickA<double>(const DevLevel& d) { return d.A; }
template <>
inline const dev::DMat<float>& pickA<float>(const DevLevel& d) { return d.Af; }
template <typename T>
static inline const dev::DMat<T>& pickAc(const DevLevel& d);
template <>
inline const dev::DMat<double>& pickAc<double>(const DevLevel& d) { return d.Ac; }
template <>
inline const dev::DMat<float>& pickAc<float>(const DevLevel& d) { return d.Acf; }
template <typename T>
static inline const dev::DMat<T>& pickP(const DevLevel& d);
template <>
inline const dev::DMat<double>& pickP<double>(const DevLevel& d) { return d.P; }
template <>
inline const dev::DMat<float>& pickP<float>(const DevLevel& d) { return d.Pf; }
template <typename T>
static inline const dev::DMat<T>& pickR(const DevLevel& d);
template <>
inline const dev::DMat<double>& pickR<double>(const DevLevel& d) { return d.R; }
template <>
inline const dev::DMat<float>& pickR<float>(const DevLevel& d) { return d.Rf; }

template <typename T>
struct LevelVecs;
template <>
struct LevelVecs<double> {
    static double* x(DevLevel& d) { return d.x; }
    static double* f(DevLevel& d) { return d.f; }
    static double* r(DevLevel& d) { return d.r; }
    static double* xo(DevLevel& d) { return d.xo; }
};
template <>
struct LevelVecs<float> {
    static float* x(DevLevel& d) { return d.xf; }
    static float* f(DevLevel& d) { return d.ff; }
    static float* r(DevLevel& d) { return d.rf; }
    static float* xo(DevLevel& d) { return d.xof; }
};

// smoother and sweep count in effect on level l (coarse_smoother overrides
// the levels below the finest)
void Solver::level_smoother(int l, int& smoother, int& sweeps) const {
    smoother = prm_.smoother;
    if (l < (int)L_.size() - 1 && prm_.coarse_smoother >= 0) {
        smoother = prm_.coarse_smoother;
        sweeps = prm_.coarse_sweeps;
    }
    if (l > 0 && l < (int)L_.size() - 1 && l < 32 && ((prm_.skip_levels >> l) & 1u)) sweeps = 0;
}

// smoother kind and sweep count of level l's pre- and post-smoothing in the
// V-cycle (AMG_V_cycle's Iter[level] settings)
void Solver::vcycle_smoother(int l, int& smoother, int& sweeps) const {
    const int depth = (int)L_.size();
    sweeps = (prm_.coarsening == AGGRESSIVE && l == depth - 1) ? prm_.aggr_smoothing_iterations
                                                                : prm_.smoothing_iterations;
    level_smoother(l, smoother, sweeps);
}

static bool is_jacobi(int smoother) {
    return smoother == LINA_SMOOTHER_JACOBI || smoother == LINA_SMOOTHER_L1_JACOBI;
}

// xinit (Solver::XInit): X_GUESS: x holds the iterate; X_ZERO: x stands for
// the zero vector and is not initialised (a coarse level's guess in the
// V-cycle), the smoother writes every entry; X_J0: x holds the first Jacobi
// sweep from zero (written by the restriction's epilogue); X_SPARE: the
// iterate is in the level's spare vector (a prolongation written beside x).
// X_J0 and X_SPARE are for Jacobi smoothers only.
template <typename T>
void Solver::smooth(int l, const T* f, T* x, int sweeps, bool post, int xinit) {
    DevLevel& d = L_[l];
    hipStream_t st = stream_;
    const T omega = (T)prm_.omega;
    int smoother;
    level_smoother(l, smoother, sweeps);
    const bool jac = is_jacobi(smoother);
    if ((xinit == X_J0 || xinit == X_SPARE) && !(jac && sweeps > 0))
        throw std::logic_error("smooth: a fused first step without a Jacobi sweep");
    const bool mc = smoother == LINA_SMOOTHER_MC_SOR || smoother == LINA_SMOOTHER_MC_SSOR;
    // a forward multicolour sweep from zero starts with one elementwise pass
    // (the first colour's values, zeros elsewhere); a batch's skipped row
    // blocks keep the zero fill instead
    const bool mc_first = mc && xinit == X_ZERO && sweeps > 0 && d.ncolours > 0 &&
                          !(smoother == LINA_SMOOTHER_MC_SSOR && post) && pickAc<T>(d).bspec == nullptr;
    if (xinit == X_ZERO && !(jac && sweeps > 0) && !mc_first) dev::fill<T>(st, d.n, x, (T)0);
    switch (smoother) {
        case LINA_SMOOTHER_SOR:
        case LINA_SMOOTHER_SSOR: {
            bool back = (smoother == LINA_SMOOTHER_SSOR) && post;
            if (std::is_same<T, double>::value && d.sor_packed)
                dev::sor_packed(st, back ? d.sorb : d.sorf, (const double*)f, (double*)x, (double)omega, sweeps);
            else if (back)
                dev::sor_lex(st, pickA<T>(d), d.nlv_b, d.lvb_off, d.lvb_rows, f, x, LevelVecs<T>::xo(d), omega,
                             sweeps, 1);
            else
                dev::sor_lex(st, pickA<T>(d), d.nlv_f, d.lvf_off, d.lvf_rows, f, x, LevelVecs<T>::xo(d), omega,
                             sweeps, 0);
            break;
        }
        case LINA_SMOOTHER_MC_SOR:
        case LINA_SMOOTHER_MC_SSOR: {
            bool back = (smoother == LINA_SMOOTHER_MC_SSOR) && post;
            const std::vector<int>& cb = sizeof(T) == 8 ? d.colour_blk : d.colour_blk32;
            for (int s = 0; s < sweeps; s++)
                for (int cc = 0; cc < d.ncolours; cc++) {
                    int c = back ? d.ncolours - 1 - cc : cc;
                    if (s == 0 && cc == 0 && mc_first) {
                        dev::mcsor_first(st, pickAc<T>(d), d.colour_rows[1], d.perm, f, x, omega);
                        continue;
                    }
                    int b0 = cb[c], b1 = cb[c + 1];
                    dev::mcsor_colour(st, pickAc<T>(d), b0, b1 - b0, d.perm, f, x, omega);
                }
            break;
        }
        case LINA_SMOOTHER_JACOBI:
        case LINA_SMOOTHER_L1_JACOBI: {
            // ping-pong between x and the level's spare vector, ending in x
            // when the iterate starts where the caller put it for that
            // (otherwise one copy back).  From a zero guess the first sweep
            // is elementwise.
            int kind = smoother == LINA_SMOOTHER_JACOBI ? dev::JAC_REF : dev::JAC_L1;
            T* a = x;
            T* b = LevelVecs<T>::xo(d);
            int s = 0;
            if (xinit == X_ZERO && sweeps > 0) {
                dev::jacobi0(st, pickA<T>(d), kind, f, x, d.nlim);
                s = 1;
            } else if (xinit == X_J0) {
                s = 1;
            } else if (xinit == X_SPARE) {
                std::swap(a, b);
            }
            for (; s < sweeps; s++) {
                dev::jacobi(st, pickA<T>(d), kind, f, (const T*)a, b, d.nlim);
                std::swap(a, b);
            }
            if (a != x) dev::copy(st, d.n, (const T*)a, x);
            break;
        }
        default:
            throw std::invalid_argument("unknown smoother");
    }
}

// the coarsest level's dense right-hand side is gathered by the restriction
bool Solver::fused_gather() const { return !cbatched_ && nd_ > 0 && dinv_ != nullptr && L_.size() > 1; }

// AMG_V_cycle (Multigrid.c:1536-1580) with Iter[level] == 1.  xinit as for
// smooth: X_ZERO stands for the reference zeroing the coarse guess before the
// recursive call.  Two steps are fused into neighbouring kernels where the
// arithmetic allows: a coarse level's first Jacobi sweep from zero (and the
// coarsest level's gather) into the restriction's epilogue, and a Jacobi
// post-smoother with an odd sweep count reads the prolongation from the
// spare vector, so its last sweep lands in x without a copy.
template <typename T>
void Solver::vcycle(int l, const T* f, T* x, int xinit) {
    hipStream_t st = stream_;
    if (l == 0) {
        // the dense-row/trivial-row split need not cover every row
        if (xinit == X_ZERO && !ccover_) dev::fill<T>(st, L_[0].n, x, (T)0);
        if (cbatched_)
            dev::bcoarse_solve(st, nd_, crblk_, coff_, cmoff_, didx_, inv_, nt_, tidx_, tdiag_, f, x, seg_active_);
        else if (ctiles_)
            dev::coarse_solve_sym(st, nd_, nct_, ntiles_, cti_, ctj_, (const double*)ctiles_, cpart_, didx_, nt_,
                                  tidx_, tdiag_, f, x, cbd_, fused_gather());
        else
            dev::coarse_solve(st, nd_, didx_, inv_, nt_, tidx_, tdiag_, f, x, cbd_, fused_gather());
        return;
    }
    DevLevel& d = L_[l];
    DevLevel& c = L_[l - 1];
    int sm, sw;
    vcycle_smoother(l, sm, sw);
    // a level without smoothing (skip_levels) passes its right-hand side down
    // and the coarse correction up: x = P V(R f), no matrix of its own read
    const bool pass = sw == 0 && xinit == X_ZERO && l < (int)L_.size() - 1;
    T* r = LevelVecs<T>::r(d);
    if (!pass) {
        smooth<T>(l, f, x, sw, false, xinit);
        dev::spmv<T, T>(st, pickA<T>(d), x, f, r, dev::MODE_RES, nullptr, nullptr);
    }
    T* fc = LevelVecs<T>::f(c);
    T* xc = LevelVecs<T>::x(c);
    dev::Epi<T, T> e;
    bool epi = false;
    int cinit = X_ZERO;
    if (l - 1 == 0) {
        if (fused_gather()) {
            e.bd = cbd_;
            e.dinv = dinv_;
            epi = true;
        }
    } else {
        int csm, csw;
        vcycle_smoother(l - 1, csm, csw);
        if (is_jacobi(csm) && csw > 0) {
            const auto& Ac = pickA<T>(c);
            e.x0 = xc;
            e.dpos = Ac.dpos;
            e.dv = Ac.v;
            e.l1 = Ac.l1;
            e.nlim = c.nlim;
            e.kind = csm == LINA_SMOOTHER_JACOBI ? dev::JAC_REF : dev::JAC_L1;
            epi = true;
            cinit = X_J0;
        }
    }
    dev::spmv<T, T>(st, pickR<T>(d), pass ? f : r, nullptr, fc, epi ? dev::MODE_SETX : dev::MODE_SET, nullptr,
                    nullptr, epi ? &e : nullptr);
    vcycle<T>(l - 1, fc, xc, cinit);
    if (pass) {
        dev::spmv<T, T>(st, pickP<T>(d), xc, nullptr, x, dev::MODE_SET, nullptr, nullptr);
        return;
    }
    if (is_jacobi(sm) && sw % 2 == 1) {
        dev::spmv<T, T>(st, pickP<T>(d), xc, x, LevelVecs<T>::xo(d), dev::MODE_ADDB, nullptr, nullptr);
        smooth<T>(l, f, x, sw, true, X_SPARE);
    } else {
        dev::spmv<T, T>(st, pickP<T>(d), xc, nullptr, x, dev::MODE_ADD, nullptr, nullptr);
        smooth<T>(l, f, x, sw, true, X_GUESS);
    }
}

// AMG_full_multigrid / FMG_recursive (Multigrid.c:1582-1611) with the
// recursion unrolled: the right-hand side restricted to every level
// (sparse_mult of each restriction, the reference's CF), the coarsest level
// solved, then on each finer level x = P x_coarse (sparse_mult, replacing
// the level's iterate) followed by one V-cycle.  The reference also
// restricts the incoming iterate down the levels (Coarse_X = R X), but the
// coarsest solve overwrites it and every finer level's iterate is replaced
// by the prolongation, so it never reaches the result and is not formed.
// Each level's f/x vectors hold CF[l] and the level's iterate: the V-cycle
// on level l writes only the vectors of the levels below, which the pass
// no longer reads.
template <typename T>
void Solver::fmg(const T* f, T* x) {
    hipStream_t st = stream_;
    const int top = (int)L_.size() - 1;
    for (int l = top; l >= 1; l--) {
        DevLevel& d = L_[l];
        const T* fl = l == top ? f : LevelVecs<T>::f(d);
        // the coarsest level's gathered right-hand side comes from the
        // restriction's epilogue when the coarse solve expects it there
        dev::Epi<T, T> e;
        const bool epi = l == 1 && fused_gather();
        if (epi) {
            e.bd = cbd_;
            e.dinv = dinv_;
        }
        dev::spmv<T, T>(st, pickR<T>(d), fl, nullptr, LevelVecs<T>::f(L_[l - 1]),
                        epi ? dev::MODE_SETX : dev::MODE_SET, nullptr, nullptr, epi ? &e : nullptr);
    }
    vcycle<T>(0, LevelVecs<T>::f(L_[0]), LevelVecs<T>::x(L_[0]), X_ZERO);
    for (int l = 1; l <= top; l++) {
        DevLevel& d = L_[l];
        T* xl = l == top ? x : LevelVecs<T>::x(d);
        const T* fl = l == top ? f : LevelVecs<T>::f(d);
        dev::spmv<T, T>(st, pickP<T>(d), LevelVecs<T>::x(L_[l - 1]), nullptr, xl, dev::MODE_SET, nullptr, nullptr);
        vcycle<T>(l, fl, xl, X_GUESS);
    }
}

// |f - A x| on the finest level into scal[slot] (FP64 or the FP32 copy)
template <typename T>
double Solver::residual_norm(const T* f, const T* x, T* r, int slot) {
    DevLevel& d = L_.back();
    const auto& A = pickA<T>(d);
    int np = dev::spmv<T, T>(stream_, A, x, f, r, dev::MODE_RES, part_, nullptr);
    dev::finalize(stream_, np, part_, scal_, slot, 1);
    return read_scalar(slot);
}

// AMG_solve (Multigrid.c:1863-1931) with F, X device vectors of the finest
// size.  The diagnostic ILU residuals of the reference (res0, res) do not
// influence the result except through `res0 != 0`, which holds exactly when
// the first residual r0 is nonzero; they are not computed.  LINA_CYCLE_FULL
// (the FULL_AMG case): one full-multigrid pass, counted as one cycle.
int Solver::amg_solve_dev(const double* F, double* X, double* relres) {
    hipStream_t st = stream_;
    DevLevel& top = L_.back();
    const int n = top.n;
    const double* Ft = F;
    if (has_neg_signs_) {
        dev::signs(st, n, signs_, F, ftop_);
        Ft = ftop_;
    }
    dev::fix_isolated<double>(st, niso_, iso_rows_, iso_a_, Ft, X);
    int it = 0;
    // relres: |r|/|r0| after the last V-cycle (AMG_add_stat's record,
    // Multigrid.c:1918); 0 when r0 = 0, 1 after a full-multigrid pass (the
    // reference leaves r = r0 there).  The loop skips the residual after the
    // last permitted cycle; it is formed only when asked for.
    double rel = 0.0;
    if (prm_.precision == LINA_PREC_FP64) {
        double r0 = residual_norm<double>(Ft, X, rtop_, dev::S_T0);
        if (r0 == 0.0) {
            if (relres) *relres = 0.0;
            return 0;
        }
        double r = r0;
        if (prm_.cycle == LINA_CYCLE_FULL) {
            fmg<double>(Ft, X);
            it = 1;
        }
        else while (std::fabs(r / r0) > prm_.amg_eps && it < prm_.amg_max_iter) {
            vcycle<double>((int)L_.size() - 1, Ft, X);
            it++;
            if (it < prm_.amg_max_iter || relres) r = residual_norm<double>(Ft, X, rtop_, dev::S_T0);
        }
        rel = std::fabs(r / r0);
    } else {
        float* ff = top.ff;
        float* xf = top.xf;
        dev::convert<double, float>(st, n, Ft, ff);
        dev::convert<double, float>(st, n, X, xf);
        double r0 = residual_norm<float>(ff, xf, top.rf, dev::S_T0);
        if (r0 != 0.0) {
            double r = r0;
            if (prm_.cycle == LINA_CYCLE_FULL) {
                fmg<float>(ff, xf);
                it = 1;
            }
            else while (std::fabs(r / r0) > prm_.amg_eps && it < prm_.amg_max_iter) {
                vcycle<float>((int)L_.size() - 1, ff, xf);
                it++;
                if (it < prm_.amg_max_iter || relres) r = residual_norm<float>(ff, xf, top.rf, dev::S_T0);
            }
            dev::convert<float, double>(st, n, xf, X);
            rel = std::fabs(r / r0);
        }
    }
    if (relres) *relres = rel;
    vcycles_ += it;
    precon_calls_++;
    return it;
}

// AMG_solve from a zero guess with at most one V-cycle, without a host round
// trip.  The reference's first residual is r0 = |F - A*0| = |F|; only
// `r0 == 0` matters with one V-cycle (the loop test is r/r0 = 1 > eps
// otherwise), and it holds exactly when every F_i^2 underflows, in whatever
// order the squares are summed.  The V-cycle runs unconditionally and its
// result is replaced by the untouched guess on the device when r0 == 0.
// w != nullptr: also the block partials of w.X into part_ (their number in
// *np), the dot k_dot_part(w, X) would give.
int Solver::vcycle_once(const double* F, double* X, const double* w, int* np) {
    hipStream_t st = stream_;
    DevLevel& top = L_.back();
    const int n = top.n;
    const int lt = (int)L_.size() - 1;
    const double* Ft = F;
    if (has_neg_signs_) {
        dev::signs(st, n, signs_, F, ftop_);
        Ft = ftop_;
    }
    // without isolated rows the guess is exactly zero and the pre-smoother
    // writes it; otherwise AMG_fix_isolated sets those rows first
    const bool xz = niso_ == 0;
    const bool fp64 = prm_.precision == LINA_PREC_FP64;
    int npd = 0;
    if (isa_ok_) {
        // entry and exit fused into one elementwise kernel each
        int n0;
        if (fp64) n0 = dev::precon_in<double>(st, n, Ft, part_, xz ? nullptr : X, nullptr, nullptr, isb_, isa_);
        else n0 = dev::precon_in<float>(st, n, Ft, part_, nullptr, xz ? nullptr : top.xf, top.ff, isb_, isa_);
        dev::finalize(st, n0, part_, scal_, dev::S_AMG0, 0);
        if (fp64) {
            vcycle<double>(lt, Ft, X, xz ? X_ZERO : X_GUESS);
            npd = dev::precon_out<double>(st, n, nullptr, X, Ft, isb_, isa_, scal_, dev::S_AMG0, w, part_);
        } else {
            vcycle<float>(lt, top.ff, top.xf, xz ? X_ZERO : X_GUESS);
            npd = dev::precon_out<float>(st, n, top.xf, X, Ft, isb_, isa_, scal_, dev::S_AMG0, w, part_);
        }
    } else {
        int n0 = dev::dot_part<double>(st, n, Ft, Ft, part_);
        dev::finalize(st, n0, part_, scal_, dev::S_AMG0, 0);
        if (!xz) {
            dev::fill<double>(st, n, X, 0.0);
            dev::fix_isolated<double>(st, niso_, iso_rows_, iso_a_, Ft, X);
        }
        if (fp64) {
            vcycle<double>(lt, Ft, X, xz ? X_ZERO : X_GUESS);
        } else {
            dev::convert<double, float>(st, n, Ft, top.ff);
            if (!xz) dev::convert<double, float>(st, n, X, top.xf);
            vcycle<float>(lt, top.ff, top.xf, xz ? X_ZERO : X_GUESS);
            dev::convert<float, double>(st, n, top.xf, X);
        }
        dev::restore_if_zero(st, n, X, scal_, dev::S_AMG0, niso_, iso_rows_, iso_a_, Ft);
        if (w) npd = dev::dot_part<double>(st, n, w, X, part_);
    }
    if (np) *np = npd;
    vcycles_ += 1;
    precon_calls_++;
    return 1;
}

// the preconditioner runs without host round trips (pcg's iterations can then
// be queued ahead of the stop test)
bool Solver::precon_async() const {
    return prm_.zero_init && prm_.amg_max_iter == 1 && prm_.cycle == LINA_CYCLE_V;
}

// pcg_update can write the next preconditioner entry (vcycle_once's fused path;
// not with make_positive_diag signs, whose signed right-hand side precon_out
// would also need)
bool Solver::entry_prepared_ok() const { return precon_async() && isa_ok_ && !has_neg_signs_; }

int Solver::precon(const double* R, double* Z, const double* w, int* np) {
    if (precon_async()) return vcycle_once(R, Z, w, np);
    if (prm_.zero_init) dev::fill<double>(stream_, n_, Z, 0.0);
    int it = amg_solve_dev(R, Z);
    if (w) *np = dev::dot_part<double>(stream_, n_, w, Z, part_);
    return it;
}

// whether two parameter blocks make the same V-cycle of one hierarchy
static bool same_cycle(const lina_amg_params& a, const lina_amg_params& b) {
    auto key = [](const lina_amg_params& p) {
        return std::make_tuple(p.dof, p.depth, p.smoothing_iterations, p.aggr_smoothing_iterations, p.coarsening,
                               p.smoother, p.omega, p.amg_eps, p.amg_max_iter, p.zero_init, p.precision,
                               p.coarse_smoother, p.coarse_sweeps, p.autotune, p.cycle, p.skip_levels);
    };
    return key(a) == key(b);
}

// pcg (PCGS.c:163-233) on device vectors X, B (length n).  The loop test is
// evaluated on the device; with a preconditioner that needs no host round
// trip, iteration k+1 is queued before the host sees iteration k's test, and
// an iteration queued after the stop leaves X, R and the scalars untouched.
//
// A one-V-cycle preconditioner without row signs (fused) has three launches
// an iteration around its V-cycle and the product: the exit kernel with the
// loop test of the previous iteration, the direction and the update, each
// adding up the partial sums it needs; the first preconditioned residual is
// iteration 0's.  Other preconditioners keep a launch per sum.
int Solver::pcg_dev(double* X, double* B, double tol, int max_iter, int stop, lina_stats* stats) {
    hipStream_t st = stream_;
    const int n = n_;
    DevLevel& top = L_.back();
    vcycles_ = 0;
    precon_calls_ = 0;
    hip_check(hipEventRecord(ev0_, st), "event");
    dev::pcg_start(st, scal_, tol, stop == LINA_STOP_RELRES, std::max(max_iter, 1));
    // h = |B| (h==0 -> 1), B and X scaled by 1/h
    int np = dev::dot_part<double>(st, n, B, B, part_);
    dev::finalize(st, np, part_, scal_, dev::S_H, 1);
    dev::scale_by(st, n, B, scal_, dev::S_H, 1);
    dev::scale_by(st, n, X, scal_, dev::S_H, 1);
    double* R = kR_;
    double* P = kP_;
    double* Q = kQ_;
    double* Z = kZ_;
    const bool fused = entry_prepared_ok();
    const bool fp64 = prm_.precision == LINA_PREC_FP64;
    double* W = fused ? Z : kW_;
    if (!fused) {  // the preconditioner's starting vectors
        dev::fill<double>(st, n, W, 0.0);
        dev::fill<double>(st, n, Z, 0.0);
    }
    // R = B + (-1)*(A X) with the caller's matrix (rows of the stored finest
    // matrix carry the make_positive_diag signs)
    if (op_) {
        op_->launch_on(st, X, B, R, dev::MODE_RES, nullptr, nullptr);
    } else if (has_neg_signs_) {
        apply_A(X, Q);
        dev::copy(st, n, (const double*)B, R);
        dev::axpby(st, n, 1.0, R, -1.0, Q);
    } else {
        dev::spmv<double, double>(st, top.A, X, B, R, dev::MODE_RES, nullptr, nullptr);
    }
    precon(R, W, W, &np);
    dev::finalize(st, np, part_, scal_, dev::S_R0, 1);
    double r0 = read_scalar(dev::S_R0);
    if (r0 == 0) {
        // the reference returns here without undoing the 1/h scaling
        if (stats) {
            stats->iterations = 0;
            stats->residual = 0;
        }
        return 0;
    }
    const int relres = stop == LINA_STOP_RELRES;
    const int cap = std::max(max_iter, 1);  // the loop body runs at least once
    // kernel timing samples every fourth iteration's outer SpMV (the events
    // themselves cost a few microseconds)
    auto sampled = [&](int k) { return ktime_ && k % 4 == 0; };
    const bool timed = ktime_ && !has_neg_signs_ && !op_;
    const bool fixed = !fp64 && fixed_order();
    // Q = A P and the partials of P.Q in part
    auto product = [&](int k, double* part) {
        if (op_) return op_->launch_on(st, P, nullptr, Q, dev::MODE_OUTER, part, P);
        if (has_neg_signs_) {
            apply_A(P, Q);
            return dev::dot_part<double>(st, n, P, Q, part);
        }
        if (sampled(k))  // the events bracket the kernel itself
            return dev::spmv_outer_timed(st, top.A, P, Q, part, P, evk_[k % 2][0], evk_[k % 2][1], fixed);
        return dev::spmv<double, double>(st, top.A, P, nullptr, Q, dev::MODE_OUTER, part, P, nullptr, fixed);
    };
    double ksum = 0.0;
    int kcount = 0;
    auto sample = [&](int k) {
        float kms = 0;
        hip_check(hipEventSynchronize(evk_[k % 2][1]), "event sync");
        hip_check(hipEventElapsedTime(&kms, evk_[k % 2][0], evk_[k % 2][1]), "elapsed");
        ksum += kms;
        kcount++;
    };
    double r = 0.0, rw = 0.0;
    int i = 0;
    if (fused) {
        double *pq = part_, *rz = part_ + part_cap_, *rr = rz + dev::DOT_PART_MAX, *zz = rr + dev::DOT_PART_MAX;
        double* status = host_ring_;
        for (int j = 0; j < 16; j++) status[j] = -1.0;
        double* Y = X;
        const int lt = (int)L_.size() - 1, xinit = niso_ == 0 ? X_ZERO : X_GUESS;
        const int ndot = std::min(std::max((n + 255) / 256, 1), dev::DOT_PART_MAX);  // an elementwise kernel's partials
        auto finish = [&](int k, int nrz, bool first) {
            dev::pcg_direction(st, n, first, P, Z, scal_, rz, nrz);
            int m = product(k, pq);
            if (m > dev::PCG_PARTS) {  // many partials keep their launch
                dev::finalize(st, m, pq, scal_, dev::S_PQ, 0);
                m = 0;
            }
            const int nrr = fp64 ? dev::pcg_update<double>(st, n, Y, R, P, Q, scal_, pq, m, rr, nullptr,
                                                           niso_ == 0 ? nullptr : Z, isb_, isa_)
                                 : dev::pcg_update<float>(st, n, Y, R, P, Q, scal_, pq, m, rr, top.ff,
                                                          niso_ == 0 ? nullptr : top.xf, isb_, isa_);
            if (nrr != ndot) throw std::logic_error("pcg: unexpected partials");
        };
        auto later = [&](int k) {
            int nrz;
            if (fp64) {
                vcycle<double>(lt, R, Z, xinit);
                nrz = dev::precon_out_stop<double>(st, n, nullptr, Z, R, isb_, isa_, scal_, rr, ndot, status, rz, zz);
            } else {
                vcycle<float>(lt, top.ff, top.xf, xinit);
                nrz = dev::precon_out_stop<float>(st, n, top.xf, Z, R, isb_, isa_, scal_, rr, ndot, status, rz, zz);
            }
            finish(k, nrz, false);
        };
        // Long solves go on with replays of REPLAY captured iterations: the
        // host takes 2.7 us a launch (3.9 with the sliced kernels' arguments),
        // the GPU 1.8 a node and about 20 us a graph, so that replays of one
        // iteration lose (257^2 Poisson, 37 iterations: 3.58 -> 3.88 ms) and
        // those of several pay where launches bound an iteration: 200
        // iterations, without -> with replays, 4k rows 18.4 -> 16.3 ms, 66k 22.6
        // -> 20.9, 132k 47.4 -> 47.3, where the line is drawn.  An iteration
        // replayed past the stop is a whole V-cycle (five of them: 5 % of a
        // solve of 49), and a capture costs 0.5-0.9 ms, what 70-100 replayed
        // iterations gain: both only when the last norms say that the solve
        // goes on for longer.  Not under kernel timing, whose events are the
        // launch's own, nor for another operator's matrix.
        constexpr int EAGER = 48, REPLAY = 4, AHEAD = 16, FIRST = 96, ROWS = 1 << 17;
        const bool replay = !op_ && !ktime_ && n <= ROWS;
        LoopTrend trend(relres ? tol : tol * r0);
        finish(0, dev::dot_part<double>(st, n, R, Z, rz), true);
        int queued = 0;
        for (int k = 1;; k++) {
            // the test of iteration k - 1 comes in the middle of iteration k:
            // what follows can be queued then, but for a graph's latency
            for (;;) {
                const bool ready = iteration_.ready() && same_cycle(iteration_prm_, prm_);
                const double left = std::min(trend.left(), (double)(cap - k)) - (queued - k);
                if (replay && queued >= EAGER && queued < k + 2 && left > (ready ? AHEAD : FIRST)) {
                    if (Y != kX_) {  // captured iterations work on the solver's own iterate
                        dev::copy(st, n, (const double*)Y, kX_);
                        Y = kX_;
                    }
                    if (!ready) {
                        iteration_.capture(st, [&]() {
                            for (int q = 0; q < REPLAY; q++) later(0);
                        });
                        iteration_prm_ = prm_;
                    }
                    iteration_.launch(st);
                    queued += REPLAY;
                } else if (queued < k) {
                    later(++queued);
                } else {
                    break;
                }
            }
            double norm;
            const bool stopped = wait_status(status, k, st, &norm);  // iteration k - 1's loop test
            if (timed && sampled(k - 1)) sample(k - 1);
            if (stopped) break;
            trend.add(norm);
        }
        // M^-1 of the final R and its norm come from the iteration that found
        // the stop; the reference's calls: one before the loop, one an
        // iteration, one after it
        dev::finalize(st, ndot, zz, scal_, dev::S_T1, 1);
        if (X != Y) dev::copy(st, n, (const double*)Y, X);
        double* last = host_ring_ + 20;  // S_R ... S_IT
        hip_check(hipMemcpyAsync(last, scal_ + dev::S_R, (dev::S_IT - dev::S_R + 1) * sizeof(double),
                                 hipMemcpyDeviceToHost, st), "d2h");
        hip_check(hipStreamSynchronize(st), "sync");
        r = last[0];
        rw = last[dev::S_T1 - dev::S_R];
        i = (int)last[dev::S_IT - dev::S_R];
        precon_calls_ = vcycles_ = i + 2;
    } else {
        // one iteration: Z = M^-1 R with R.Z, P, Q = A P with P.Q, X and R
        // with |R| and the stop test; its state (S_R..S_IT) copied to ring slot k % 2
        auto enqueue = [&](int k) {
            int m = 0;
            precon(R, Z, R, &m);
            dev::finalize(st, m, part_, scal_, dev::S_S, 2);  // s_old = s; s = R.Z
            dev::pcg_p(st, n, P, Z, scal_, k == 0);
            m = product(k, part_);
            dev::finalize(st, m, part_, scal_, dev::S_PQ, 0);
            m = dev::pcg_xr(st, n, X, R, P, Q, scal_, part_);
            dev::finalize_stop(st, m, part_, scal_, tol, relres, cap);
            double* h = host_ring_ + (k % 2) * dev::S_COUNT;
            hip_check(hipMemcpyAsync(h + dev::S_R, scal_ + dev::S_R, (dev::S_IT - dev::S_R + 1) * sizeof(double),
                                     hipMemcpyDeviceToHost, st),
                      "d2h");
            hip_check(hipEventRecord(evr_[k % 2], st), "event");
        };
        const int ahead = precon_async() ? 2 : 1;
        int enq = 0, done = 0;
        for (;;) {
            while (enq < cap && enq - done < ahead) enqueue(enq++);
            hip_check(hipEventSynchronize(evr_[done % 2]), "event sync");
            const double* h = host_ring_ + (done % 2) * dev::S_COUNT;
            const int it_dev = (int)h[dev::S_IT];
            if (timed && sampled(done) && it_dev == done + 1) sample(done);
            r = h[dev::S_R];
            i = it_dev;
            done++;
            if (h[dev::S_STOP] != 0.0 || (done == enq && enq >= cap)) break;
        }
        // an iteration queued after the stop ran its V-cycle and nothing else
        vcycles_ -= enq - i;
        precon_calls_ -= enq - i;
        precon(R, W, W, &np);
        dev::finalize(st, np, part_, scal_, dev::S_T1, 1);
        rw = read_scalar(dev::S_T1);
    }
    const double relres_out = r;
    dev::scale_by(st, n, B, scal_, dev::S_H, 0);
    dev::scale_by(st, n, X, scal_, dev::S_H, 0);
    hip_check(hipEventRecord(ev1_, st), "event");
    hip_check(hipEventSynchronize(ev1_), "event sync");
    float ms = 0;
    hip_check(hipEventElapsedTime(&ms, ev0_, ev1_), "elapsed");
    pcg_residuum_ = rw / r0;
    if (stats) {
        stats->iterations = i;
        stats->precon_calls = precon_calls_;
        stats->vcycles = vcycles_;
        stats->residual = pcg_residuum_;
        stats->relres = relres_out;
        stats->t_solve_ms = ms;
        stats->spmv_ms = kcount ? ksum / kcount : 0.0;
        stats->spmv_launches = kcount;
    }
    if (std::isnan(rw / r0)) throw NumericError("pcg: NaN residual");
    return i;
}

int Solver::pcg_host(double* x, double* b, double tol, int max_iter, int stop, lina_stats* stats) {
    const size_t bytes = (size_t)n_ * sizeof(double);
    hip_check(hipMemcpyAsync(kX_, x, bytes, hipMemcpyHostToDevice, stream_), "h2d");
    hip_check(hipMemcpyAsync(kB_, b, bytes, hipMemcpyHostToDevice, stream_), "h2d");
    int it = pcg_dev(kX_, kB_, tol, max_iter, stop, stats);
    hip_check(hipMemcpyAsync(x, kX_, bytes, hipMemcpyDeviceToHost, stream_), "d2h");
    hip_check(hipMemcpyAsync(b, kB_, bytes, hipMemcpyDeviceToHost, stream_), "d2h");
    hip_check(hipStreamSynchronize(stream_), "sync");
    return it;
}

int Solver::amg_solve_host(const double* f, double* x, double* relres) {
    const size_t bytes = (size_t)n_ * sizeof(double);
    hip_check(hipMemcpyAsync(kB_, f, bytes, hipMemcpyHostToDevice, stream_), "h2d");
    hip_check(hipMemcpyAsync(kX_, x, bytes, hipMemcpyHostToDevice, stream_), "h2d");
    vcycles_ = 0;
    precon_calls_ = 0;
    int it = amg_solve_dev(kB_, kX_, relres);
    hip_check(hipMemcpyAsync(x, kX_, bytes, hipMemcpyDeviceToHost, stream_), "d2h");
    hip_check(hipStreamSynchronize(stream_), "sync");
    return it;
}

int Solver::spmv_host(int level, int precision, const double* x, double* y) {
    DevLevel& d = L_.at(level);
    const size_t bytes = (size_t)d.n * sizeof(double);
    hip_check(hipMemcpyAsync(d.xo, x, bytes, hipMemcpyHostToDevice, stream_), "h2d");
    if (precision == LINA_PREC_FP64) {
        dev::spmv<double, double>(stream_, d.A, d.xo, nullptr, d.r, dev::MODE_SET, nullptr, nullptr);
    } else {
        dev::convert<double, float>(stream_, d.n, d.xo, d.xof);
        dev::spmv<float, float>(stream_, d.Af, d.xof, nullptr, d.rf, dev::MODE_SET, nullptr, nullptr);
        dev::convert<float, double>(stream_, d.n, d.rf, d.r);
    }
    hip_check(hipMemcpyAsync(y, d.r, bytes, hipMemcpyDeviceToHost, stream_), "d2h");
    hip_check(hipStreamSynchronize(stream_), "sync");
    return 0;
}

double Solver::time_spmv(int level, int precision, int reps) {
    DevLevel& d = L_.at(level);
    dev::fill<double>(stream_, d.n, d.xo, 1.0);
    dev::fill<float>(stream_, d.n, d.xof, 1.0f);
    auto launch = [&]() {
        if (precision == LINA_PREC_FP64)
            dev::spmv<double, double>(stream_, d.A, d.xo, nullptr, d.r, dev::MODE_OUTER, nullptr, nullptr);
        else
            dev::spmv<float, float>(stream_, d.Af, d.xof, nullptr, d.rf, dev::MODE_OUTER, nullptr, nullptr);
    };
    for (int i = 0; i < 3; i++) launch();
    hip_check(hipEventRecord(ev0_, stream_), "event");
    for (int i = 0; i < reps; i++) launch();
    hip_check(hipEventRecord(ev1_, stream_), "event");
    hip_check(hipEventSynchronize(ev1_), "event sync");
    float ms = 0;
    hip_check(hipEventElapsedTime(&ms, ev0_, ev1_), "elapsed");
    return ms / reps;
}

double spmv_bytes(double n, double nnz, int precision) {
    if (precision == LINA_PREC_FP64) return 12.0 * nnz + 4.0 * (n + 1) + 16.0 * n;
    return 8.0 * nnz + 4.0 * (n + 1) + 8.0 * n;
}

// algorithmic bytes of one y = A x with the uploaded arrays: values, column
// indices (2-byte codes + 8 bytes of bases per slice or block, or 4 bytes),
// row pointers, slice or block pairs, x gathered once, y written once
template <typename VT>
static double mat_bytes(const dev::DMat<VT>& A) {
    return (double)sizeof(VT) * A.nnz + A.idx_bytes + 4.0 * (A.n + 1) + 8.0 * ((A.sl.ns ? A.sl.ns : A.nblk) + 1) +
           (double)sizeof(VT) * (A.ncols + A.n);
}

double Solver::spmv_bytes(int level, int precision) const {
    if (uploaded() && level >= 0 && level < (int)L_.size())
        return precision == LINA_PREC_FP64 ? mat_bytes(L_[level].A) : mat_bytes(L_[level].Af);
    const Csr& A = H_.lv.at(level).A;
    return lina::spmv_bytes(A.n, A.nnz(), precision);
}

// ------------------------------------------------------- DevMatrix

DevMatrix::DevMatrix(const Csr& A) : n_(A.n), nnz_(A.nnz()), bufs_(new DevBuffers) {
    hip_check(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking), "stream");
    hip_check(hipEventCreate(&ev0_), "event");
    hip_check(hipEventCreate(&ev1_), "event");
    upload_pair(A, A_, Af_, *bufs_, stream_, nullptr, true, true);
    prp_ = A.rp;
    pci_ = A.ci;
    x_ = dalloc<double>(n_, *bufs_);
    y_ = dalloc<double>(n_, *bufs_);
    xf_ = dalloc<float>(n_, *bufs_);
    yf_ = dalloc<float>(n_, *bufs_);
    hip_check(hipStreamSynchronize(stream_), "upload");
}

bool DevMatrix::update_values(const Csr& A0) {
    if (A0.n != n_ || A0.rp != prp_ || A0.ci != pci_) return false;
    const Csr A = drop_outside_zeros(A0);
    if (A.nnz() != A_.nnz) return false;
    hip_check(hipMemcpyAsync(A_.v, A.v.data(), A.v.size() * sizeof(double), hipMemcpyHostToDevice, stream_), "h2d");
    dev::pair_values(stream_, A_, Af_);
    hip_check(hipStreamSynchronize(stream_), "update");
    return true;
}

bool DevMatrix::update_values_device(const double* d_val, long nnz) {
    if (nnz != (long)A_.nnz || nnz_ != nnz) return false;
    hip_check(hipMemcpyAsync(A_.v, d_val, nnz * sizeof(double), hipMemcpyDeviceToDevice, stream_), "d2d");
    dev::pair_values(stream_, A_, Af_);
    hip_check(hipStreamSynchronize(stream_), "update");
    return true;
}

double DevMatrix::matrix_norm() const {
    std::vector<double> v(A_.nnz);
    hip_check(hipMemcpyAsync(v.data(), A_.v, v.size() * sizeof(double), hipMemcpyDeviceToHost, stream_), "d2h");
    hip_check(hipStreamSynchronize(stream_), "sync");
    double s = 0;
    for (double a : v) s += std::fabs(a);
    return s / n_;
}

DevMatrix::~DevMatrix() {
    if (stream_) (void)hipStreamSynchronize(stream_);
    bufs_.reset();
    if (ev0_) (void)hipEventDestroy(ev0_);
    if (ev1_) (void)hipEventDestroy(ev1_);
    if (stream_) (void)hipStreamDestroy(stream_);
}

void DevMatrix::apply(const double* x, double* y) {
    dev::spmv<double, double>(stream_, A_, x, nullptr, y, dev::MODE_OUTER, nullptr, nullptr);
}

int DevMatrix::launch(const double* x, const double* b, double* y, int mode, double* part, const double* w) {
    return dev::spmv<double, double>(stream_, A_, x, b, y, mode, part, w);
}

int DevMatrix::launch_on(hipStream_t st, const double* x, const double* b, double* y, int mode, double* part,
                         const double* w) {
    return dev::spmv<double, double>(st, A_, x, b, y, mode, part, w);
}

void DevMatrix::spmv_dev(const double* x, double* y) {
    apply(x, y);
    hip_check(hipStreamSynchronize(stream_), "spmv");
}

void DevMatrix::spmv_host(int precision, const double* x, double* y) {
    const size_t bytes = (size_t)n_ * sizeof(double);
    hip_check(hipMemcpyAsync(x_, x, bytes, hipMemcpyHostToDevice, stream_), "h2d");
    if (precision == LINA_PREC_FP64) {
        apply(x_, y_);
    } else {
        dev::convert<double, float>(stream_, n_, x_, xf_);
        dev::spmv<float, float>(stream_, Af_, xf_, nullptr, yf_, dev::MODE_OUTER, nullptr, nullptr);
        dev::convert<float, double>(stream_, n_, yf_, y_);
    }
    hip_check(hipMemcpyAsync(y, y_, bytes, hipMemcpyDeviceToHost, stream_), "d2h");
    hip_check(hipStreamSynchronize(stream_), "sync");
}

double DevMatrix::time_spmv(int precision, int reps) {
    dev::fill<double>(stream_, n_, x_, 1.0);
    dev::fill<float>(stream_, n_, xf_, 1.0f);
    auto launch = [&]() {
        if (precision == LINA_PREC_FP64)
            dev::spmv<double, double>(stream_, A_, x_, nullptr, y_, dev::MODE_OUTER, nullptr, nullptr);
        else
            dev::spmv<float, float>(stream_, Af_, xf_, nullptr, yf_, dev::MODE_OUTER, nullptr, nullptr);
    };
    for (int i = 0; i < 3; i++) launch();
    hip_check(hipEventRecord(ev0_, stream_), "event");
    for (int i = 0; i < reps; i++) launch();
    hip_check(hipEventRecord(ev1_, stream_), "event");
    hip_check(hipEventSynchronize(ev1_), "event sync");
    float ms = 0;
    hip_check(hipEventElapsedTime(&ms, ev0_, ev1_), "elapsed");
    return ms / reps;
}

double DevMatrix::bytes(int precision) const {
    return precision == LINA_PREC_FP64 ? mat_bytes(A_) : mat_bytes(Af_);
}

template void Solver::smooth<double>(int, const double*, double*, int, bool, int);
template void Solver::smooth<float>(int, const float*, float*, int, bool, int);
template void Solver::vcycle<double>(int, const double*, double*, int);
template void Solver::vcycle<float>(int, const float*, float*, int);
template void Solver::fmg<double>(const double*, double*);
template void Solver::fmg<float>(const float*, float*);

}  // namespace lina
