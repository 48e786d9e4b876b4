// Host side of the LDL preconditioner: a nested-dissection ordering from
// cell centres and the numeric LDL^T factorization of the permuted matrix.
//
// The reference builds this preconditioner once, when the solver is set up
// (opLDL(A) in Preconditioner{LDL}, preconditioners_0_types.jl:36-42, with
// LinearOperators 2.6.0 over LDLFactorizations 0.10.1), and never updates
// it (update_preconditioner! for LDL is a no-op,
// preconditioners_2_functions.jl:52-57): every later solve is preconditioned
// by the inverse of the set-up matrix.  The factorization is the up-looking
// LDL^T of Davis ("Algorithm 849: a concise sparse Cholesky factorization
// package", ACM TOMS 31(4), 2005), which LDLFactorizations restates; the
// ordering is our own (geometric nested dissection: recursive bisection at
// the median cell centre along the longer side, the cells next to the other
// half forming the separator, numbered last), where LDLFactorizations uses
// AMD.  Ordering and rounding therefore differ from the reference's; the
// preconditioner they approximate, A^-1 of the set-up matrix, does not.
#include "fvh_internal.h"

#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <exception>
#include <numeric>
#include <thread>
#include <vector>

#include "ldl_host.h"

namespace fvh {

namespace {

struct NdState {
    const int *rowptr, *col;
    const double *x, *y;
    std::vector<int> mark;  // per cell: side stamp of the current split
    int stamp = 0;
    std::vector<int> *out;
    std::vector<int> *bounds;  // end of every leaf and separator appended (or null)
};

// Dissection goes on to kNdLeaf cells (less fill); a part of at most kNdRange
// cells is one range, whose triangle one block inverts and applies: larger
// ranges trade bytes (the packed inverse, s^2 / 2 values) for depth.
constexpr int kNdLeaf = 48, kNdRange = kLdlLeaf;

void nd_split(NdState &S, std::vector<int> cells) {
    // explicit stack instead of recursion: (cells, state) frames
    struct Frame {
        std::vector<int> cells;
        int stage;  // 0: split; 1: append separator after children
        bool inside;  // part of a range whose end an enclosing frame marks
        std::vector<int> sep;
    };
    std::vector<Frame> st;
    st.push_back({std::move(cells), 0, false, {}});
    while (!st.empty()) {
        Frame &F = st.back();
        if (F.stage == 1) {
            S.out->insert(S.out->end(), F.sep.begin(), F.sep.end());
            if (S.bounds && !F.inside && S.bounds->back() < (int)S.out->size()) S.bounds->push_back((int)S.out->size());
            st.pop_back();
            continue;
        }
        if ((int)F.cells.size() <= kNdLeaf) {
            std::sort(F.cells.begin(), F.cells.end());
            S.out->insert(S.out->end(), F.cells.begin(), F.cells.end());
            if (S.bounds && !F.inside && !F.cells.empty()) S.bounds->push_back((int)S.out->size());
            st.pop_back();
            continue;
        }
        double x0 = 1e300, x1 = -1e300, y0 = 1e300, y1 = -1e300;
        for (int c : F.cells) {
            x0 = std::min(x0, S.x[c]);
            x1 = std::max(x1, S.x[c]);
            y0 = std::min(y0, S.y[c]);
            y1 = std::max(y1, S.y[c]);
        }
        const double *coord = (x1 - x0 >= y1 - y0) ? S.x : S.y;
        std::vector<int> v = F.cells;
        const size_t half = v.size() / 2;
        std::nth_element(v.begin(), v.begin() + half, v.end(), [&](int a, int b) {
            return coord[a] < coord[b] || (coord[a] == coord[b] && a < b);
        });
        const int sl = ++S.stamp, sr = ++S.stamp;
        for (size_t i = 0; i < v.size(); ++i) S.mark[v[i]] = i < half ? sl : sr;
        std::vector<int> left, right, sep;
        for (size_t i = 0; i < half; ++i) {
            const int c = v[i];
            bool touches = false;
            for (int p = S.rowptr[c]; p < S.rowptr[c + 1] && !touches; ++p) touches = S.mark[S.col[p]] == sr;
            (touches ? sep : left).push_back(c);
        }
        right.assign(v.begin() + half, v.end());
        std::sort(sep.begin(), sep.end());
        // (a part small enough for one range is marked once, after its separator)
        const bool inside = F.inside || (int)F.cells.size() <= kNdRange;
        F.stage = 1;
        F.sep = std::move(sep);
        F.cells.clear();
        F.cells.shrink_to_fit();
        // right is numbered after left: push it first (the stack pops left first)
        st.push_back({std::move(right), 0, inside, {}});
        st.push_back({std::move(left), 0, inside, {}});
    }
}

}  // namespace

void ldl_order(int n, const int *rowptr, const int *col, const double *x, const double *y, std::vector<int> &perm,
               std::vector<int> *bounds) {
    NdState S{rowptr, col, x, y, std::vector<int>(n, 0), 0, &perm, bounds};
    perm.clear();
    perm.reserve(n);
    if (bounds) bounds->assign(1, 0);
    std::vector<int> all(n);
    std::iota(all.begin(), all.end(), 0);
    nd_split(S, std::move(all));
}

int ldl_factor(int n, const int *rowptr, const int *col, const double *val, const std::vector<int> &perm, LdlHost &F) {
    if ((int)perm.size() != n) return set_error(FVH_ERR_ARG, "LDL: ordering of %zu rows for %d", perm.size(), n);
    std::vector<int> iperm(n, -1);
    for (int k = 0; k < n; ++k) {
        if (perm[k] < 0 || perm[k] >= n || iperm[perm[k]] >= 0) return set_error(FVH_ERR_ARG, "LDL: not a permutation");
        iperm[perm[k]] = k;
    }
    // A(r, c) from the upper triangle of A in its own numbering
    auto upper = [&](int r, int c) -> double {
        const int a = std::min(r, c), b = std::max(r, c);
        const int *lo = col + rowptr[a], *hi = col + rowptr[a + 1];
        const int *it = std::lower_bound(lo, hi, b);
        return (it != hi && *it == b) ? val[it - col] : 0.0;
    };
    // symbolic: elimination tree and column counts of L
    std::vector<int> parent(n, -1), flag(n), lnz(n, 0);
    for (int k = 0; k < n; ++k) {
        flag[k] = k;
        const int r = perm[k];
        for (int p = rowptr[r]; p < rowptr[r + 1]; ++p) {
            int i = iperm[col[p]];
            if (i >= k) continue;
            for (; flag[i] != k; i = parent[i]) {
                if (parent[i] == -1) parent[i] = k;
                lnz[i]++;
                flag[i] = k;
            }
        }
    }
    F.n = n;
    F.perm = perm;
    F.Lp.assign(n + 1, 0);
    for (int k = 0; k < n; ++k) F.Lp[k + 1] = F.Lp[k] + lnz[k];
    const int64_t nnzL = F.Lp[n];
    if (nnzL >= (int64_t)1 << 31) return set_error(FVH_ERR_SIZE, "LDL: %lld entries in L", (long long)nnzL);
    F.Li.assign(nnzL, 0);
    F.Lx.assign(nnzL, 0.0);
    F.D.assign(n, 0.0);
    // numeric: row k of L from a sparse triangular solve along the etree
    std::vector<double> yv(n, 0.0);
    std::vector<int> pattern(n), fill(n, 0);
    double *__restrict__ y = yv.data();
    const int *__restrict__ Li = F.Li.data();
    const double *__restrict__ Lx = F.Lx.data();
    for (int k = 0; k < n; ++k) {
        int top = n;
        flag[k] = k;
        const int r = perm[k];
        for (int p = rowptr[r]; p < rowptr[r + 1]; ++p) {
            int i = iperm[col[p]];
            if (i > k) continue;
            yv[i] += upper(r, col[p]);
            int len = 0;
            for (; flag[i] != k; i = parent[i]) {
                pattern[len++] = i;
                flag[i] = k;
            }
            while (len > 0) pattern[--top] = pattern[--len];
        }
        double d = yv[k];
        yv[k] = 0.0;
        for (; top < n; ++top) {
            const int i = pattern[top];
            const double yi = yv[i];
            yv[i] = 0.0;
            const int p1 = F.Lp[i], p2 = p1 + fill[i];
            for (int p = p1; p < p2; ++p) y[Li[p]] -= Lx[p] * yi;
            const double lki = yi / F.D[i];
            d -= lki * yi;
            F.Li[p2] = k;
            F.Lx[p2] = lki;
            fill[i]++;
        }
        if (d == 0.0 || !std::isfinite(d))
            return set_error(FVH_ERR_ARG, "LDL: pivot %d (row %d) is %g: the set-up matrix is singular", k, r, d);
        F.D[k] = d;
    }
    return FVH_OK;
}

// Inverse of the unit lower triangular block of s rows from r0, packed
// without its unit diagonal by rows (row i: columns 0 .. i-1) and by columns
// (column k: rows k+1 .. s-1), into the sides that read it so.  X: scratch.
// Where an entry is above kLdlGrowth, the row it is in goes to `cuts`: between
// two cuts every entry is within it.  (A diagonal block of the inverse is the
// inverse of that block.)
static void invert_range(const LdlHost &F, int r0, int s, std::vector<double> &X, bool whole, double *f, double *b,
                         std::vector<int> &cuts) {
    if (X.size() < (size_t)s * s) X.resize((size_t)s * s);
    // X starts as the block itself (below its diagonal); row i of the inverse
    // then replaces row i: -sum_k L_ik (row k of the inverse), k ascending (L_ik
    // stands until its turn)
    for (int i = 0; i < s; ++i) std::fill_n(&X[(size_t)i * s], i, 0.0);
    for (int k = 0; k < s; ++k)
        for (int p = F.Lp[r0 + k]; p < F.Lp[r0 + k + 1] && F.Li[p] < r0 + s; ++p)
            X[(size_t)(F.Li[p] - r0) * s + k] = F.Lx[p];
    int from = 0;
    for (int i = 1; i < s; ++i) {
        double *xi = &X[(size_t)i * s];
        for (int k = 0; k < i; ++k) {
            const double l = xi[k];
            if (l == 0.0) continue;
            const double *xk = &X[(size_t)k * s];
            for (int c = 0; c < k; ++c) xi[c] -= l * xk[c];
            xi[k] = -l;
        }
        for (int c = from; c < i; ++c)
            if (!(std::fabs(xi[c]) <= kLdlGrowth)) {  // (a NaN too)
                cuts.push_back(r0 + i);
                from = i;
                break;
            }
    }
    double *rows = whole ? b : f, *cols = whole ? f : b;  // a whole range: lane = row, column after column
    for (int i = 1; i < s; ++i)
        for (int k = 0; k < i; ++k) *rows++ = X[(size_t)i * s + k];
    for (int k = 0; k + 1 < s; ++k)
        for (int i = k + 1; i < s; ++i) *cols++ = X[(size_t)i * s + k];
}

// The blocks of the ranges between `cut`; rows that a range has to be cut at
// as well, for the growth of its inverse, go to `more`.
static void blocks_of(const LdlHost &F, const std::vector<int> &cut, LdlBlocks &out, std::vector<int> &more) {
    const int n = F.n, ng = (int)cut.size() - 1;
    std::vector<int> range_of(n);
    for (int g = 0; g < ng; ++g)
        for (int i = cut[g]; i < cut[g + 1]; ++i) range_of[i] = g;
    // the entries outside the ranges' own blocks, by column and by row
    LdlSide &f = out.f, &b = out.b;
    f.ptr.assign(n + 1, 0);
    b.ptr.assign(n + 1, 0);
    for (int j = 0; j < n; ++j)
        for (int p = F.Lp[j]; p < F.Lp[j + 1]; ++p)
            if (range_of[F.Li[p]] != range_of[j]) {
                f.ptr[F.Li[p] + 1]++;
                b.ptr[j + 1]++;
            }
    for (int i = 0; i < n; ++i) {
        f.ptr[i + 1] += f.ptr[i];
        b.ptr[i + 1] += b.ptr[i];
    }
    f.idx.resize(f.ptr[n]);
    f.val.resize(f.ptr[n]);
    b.idx.resize(b.ptr[n]);
    b.val.resize(b.ptr[n]);
    // heights: a range follows, forward, every range its outside columns
    // belong to, and backward every range its outside rows belong to
    std::vector<int> hf(ng, 0), hb(ng, 0), pos(f.ptr.begin(), f.ptr.end() - 1);
    for (int j = 0; j < n; ++j) {
        const int g = range_of[j];
        int q = b.ptr[j];
        for (int p = F.Lp[j]; p < F.Lp[j + 1]; ++p) {
            const int i = F.Li[p], gi = range_of[i];
            if (gi == g) continue;
            hf[gi] = std::max(hf[gi], hf[g] + 1);  // columns of g are all visited before those of gi
            f.idx[pos[i]] = j;
            f.val[pos[i]++] = F.Lx[p];
            b.idx[q] = i;
            b.val[q++] = F.Lx[p];
        }
    }
    for (int j = n - 1; j >= 0; --j) {
        const int g = range_of[j];
        for (int p = b.ptr[j]; p < b.ptr[j + 1]; ++p) hb[g] = std::max(hb[g], hb[range_of[b.idx[p]]] + 1);
    }
    // inverse blocks, the ranges dealt to a few threads (each writes its own
    // ranges' words)
    std::vector<char> whole(ng);
    std::vector<long long> off(ng + 1, 0);
    for (int g = 0; g < ng; ++g) {
        const long long s = cut[g + 1] - cut[g];
        whole[g] = s <= kLdlWhole || (s <= kLdlLeaf && hf[g] == 0);
        off[g + 1] = off[g] + s * (s - 1) / 2;
    }
    f.inv.resize(off[ng]);
    b.inv.resize(off[ng]);
    std::atomic<int> next{0};
    const int nt = off[ng] < (1 << 17) ? 1 : std::max(1, std::min(8, (int)std::thread::hardware_concurrency()));
    std::vector<std::vector<int>> cuts(nt);
    std::vector<std::exception_ptr> failed(nt);  // an exception must not leave a thread, nor pass running ones
    const auto invert = [&](int t) {
        try {
            std::vector<double> X;
            for (int g0; (g0 = next.fetch_add(64)) < ng;)
                for (int g = g0; g < std::min(g0 + 64, ng); ++g)
                    invert_range(F, cut[g], cut[g + 1] - cut[g], X, whole[g], f.inv.data() + off[g],
                                 b.inv.data() + off[g], cuts[t]);
        } catch (...) {
            failed[t] = std::current_exception();
            next = ng;
        }
    };
    {
        std::vector<std::thread> th;
        th.reserve(nt);
        try {
            for (int t = 1; t < nt; ++t) th.emplace_back(invert, t);
        } catch (...) {  // fewer threads then
        }
        invert(0);
        for (auto &t : th) t.join();
    }
    for (const auto &e : failed)
        if (e) std::rethrow_exception(e);
    for (const auto &c : cuts) more.insert(more.end(), c.begin(), c.end());
    if (!more.empty()) return;
    // a range's parent in the tree holds the first of its outside rows; a
    // block's gates are words of the (at most two highest) ranges right below
    // it (forward) or of the parent (backward)
    std::vector<int> parent(ng, -1);
    std::vector<std::array<int, 2>> child(ng, {-1, -1});
    for (int g = 0; g < ng; ++g) {
        int first = n;
        for (int p = b.ptr[cut[g]]; p < b.ptr[cut[g + 1]]; ++p) first = std::min(first, b.idx[p]);
        if (first == n) continue;
        parent[g] = range_of[first];
        std::array<int, 2> &c = child[parent[g]];
        if (c[0] < 0 || hf[g] >= hf[c[0]]) c = {g, c[0]};
        else if (c[1] < 0 || hf[g] > hf[c[1]]) c[1] = g;
    }
    const auto last_row = [&](int g) { return g < 0 ? -1 : cut[g + 1] - 1; };
    // blocks by height (a range's outside rows before its inverse rows, which
    // wait for the range's own last outside row)
    const auto list = [&](const std::vector<int> &h, bool fwd, std::vector<LdlBlock> &blk) {
        std::vector<int> order(ng);
        std::iota(order.begin(), order.end(), 0);
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return h[x] < h[y]; });
        for (int g : order) {
            const int r0 = cut[g], s = cut[g + 1] - r0;
            const int g0 = last_row(fwd ? child[g][0] : parent[g]), g1 = last_row(fwd ? child[g][1] : -1);
            if (whole[g]) {
                blk.push_back({0, r0, r0, s, {g0, g1}, off[g]});
                continue;
            }
            for (int i = 0; i < s; i += kLdlWaves) blk.push_back({1, r0 + i, r0, s, {g0, g1}, off[g]});
            for (int i = 0; i < s; i += kLdlWaves) blk.push_back({2, r0 + i, r0, s, {r0, r0 + s - 1}, off[g]});
        }
    };
    f.blocks.clear();
    b.blocks.clear();
    list(hf, true, f.blocks);
    list(hb, false, b.blocks);
}

void ldl_blocks(const LdlHost &F, const std::vector<int> &bounds, LdlBlocks &out) {
    std::vector<int> cut{0}, more;
    for (size_t g = 0; g + 1 < bounds.size(); ++g)
        for (int a = bounds[g]; a < bounds[g + 1]; a += kLdlRange) cut.push_back(std::min(a + kLdlRange, bounds[g + 1]));
    blocks_of(F, cut, out, more);
    if (more.empty()) return;
    cut.insert(cut.end(), more.begin(), more.end());
    std::sort(cut.begin(), cut.end());
    more.clear();
    blocks_of(F, cut, out, more);  // the same inverses in smaller pieces: nothing more to cut
}

}  // namespace fvh
