// LDL preconditioner on the device: y = P^T L^-T D^-1 L^-1 P x with the
// factor of the set-up matrix (ldl_host.cpp), frozen after the first
// update as the reference freezes opLDL (preconditioners_0_types.jl:36-42,
// preconditioners_2_functions.jl:52-57).
//
// The two triangular solves go range by range of the nested-dissection order
// with the ranges' own triangles inverted (k_ldl_blocks, below).
// FVH_LDL_RANGES=0 at the set-up keeps the sync-free row solves: one wave per
// row of L (forward, rows in factor order) or of L^T (backward, rows in
// reverse order), the lanes splitting the row's entries.
// In both, a row's inputs from elsewhere are results that other work-groups
// publish with device-coherent stores into an array filled with a
// signalling-NaN sentinel before the solve; a lane polls a value until it is
// no longer the sentinel.  Every work-group waits only for rows of
// work-groups dispatched before it, so the solve always drains; each poll is
// bounded, and a wait that runs out sets a fault word (pinned host memory)
// that the caller reports.  Per row (sync-free solves): lane l sums its
// entries l, l + 64, ... in order from 0, then the lanes are added by a
// fixed tree; a lane issues the loads of up to kLdlBatch inputs before it
// waits for any.
#include <algorithm>
#include <cstdlib>
#include <vector>

#include "fvh_eqn.h"
#include "ldl_host.h"

namespace fvh {

namespace {

constexpr unsigned long long kLdlSent = 0x7FF4DEAD5EA11A57ull;
constexpr int kLdlSpin = 1 << 20;  // polls (a few 100 ms) before a wait is declared lost
constexpr int kLdlRowWaves = 4;    // waves (rows) per work-group of the row solves
constexpr int kLdlBatch = 16;      // inputs per lane loaded before any is waited for

__device__ inline double ldl_load(const double *p) {
    return __builtin_bit_cast(double, __hip_atomic_load(reinterpret_cast<const unsigned long long *>(p),
                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ inline void ldl_store(double *p, double v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(p), __builtin_bit_cast(unsigned long long, v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline bool ldl_sent(double v) { return __builtin_bit_cast(unsigned long long, v) == kLdlSent; }

// Value of row j once published (bounded wait).
__device__ inline double ldl_wait(const double *y, int j, int *fault) {
    double v = ldl_load(y + j);
    for (int s = 0; ldl_sent(v); ++s) {
        if (s >= kLdlSpin) {
            __hip_atomic_store(fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            return 0.0;
        }
        __builtin_amdgcn_s_sleep(1);
        v = ldl_load(y + j);
    }
    return v;
}

__device__ inline double wave_sum(double a) {
    for (int off = 32; off > 0; off >>= 1) a = a + __shfl_down(a, off, 64);
    return a;
}

// DPP move of an FP64 value (both halves); lanes that read outside their
// row, and rows the row mask leaves out, get 0
template <int CTRL, int ROWS, bool BOUND>
__device__ inline double dpp_f64(double v) {
    const int2 b = __builtin_bit_cast(int2, v);
    int2 r;
    r.x = __builtin_amdgcn_update_dpp(0, b.x, CTRL, ROWS, 0xF, BOUND);
    r.y = __builtin_amdgcn_update_dpp(0, b.y, CTRL, ROWS, 0xF, BOUND);
    return __builtin_bit_cast(double, r);
}
// Sum of a wave's 64 lanes in a fixed order, without LDS: shifts by 1, 2,
// 4, 8 within each row of 16 lanes (lane 15 of a row then holds the row's
// sum), the sum of rows 0 and 2 broadcast into rows 1 and 3, then lane 31's
// into rows 2 and 3; lane 63 holds (row 2 + row 3) + (row 0 + row 1).
__device__ inline double wave_total(double a) {
    a = a + dpp_f64<0x111, 0xF, true>(a);   // row_shr:1
    a = a + dpp_f64<0x112, 0xF, true>(a);   // row_shr:2
    a = a + dpp_f64<0x114, 0xF, true>(a);   // row_shr:4
    a = a + dpp_f64<0x118, 0xF, true>(a);   // row_shr:8
    a = a + dpp_f64<0x142, 0xA, false>(a);  // row_bcast:15 into rows 1 and 3
    a = a + dpp_f64<0x143, 0xC, false>(a);  // row_bcast:31 into rows 2 and 3
    const int2 b = __builtin_bit_cast(int2, a);
    return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(b.x, 63), __builtin_amdgcn_readlane(b.y, 63)));
}

}  // namespace

// rhs[k] = x[perm[k]] (in FP64); the result arrays to the sentinel
template <typename T>
__global__ void k_ldl_prep(int n, const int *__restrict__ perm, const T *__restrict__ x, double *__restrict__ rhs,
                           double *__restrict__ y, double *__restrict__ z, double *__restrict__ r,
                           double *__restrict__ s, const KScal *ks) {
    if (ks && ks->done) return;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const double sent = __builtin_bit_cast(double, kLdlSent);
    rhs[k] = (double)x[perm[k]];
    y[k] = sent;
    z[k] = sent;
    if (r) r[k] = sent;
    if (s) s[k] = sent;
}

// BWD = false: y_r = rhs_r - sum_j L_rj y_j (rows of L in order);
// BWD = true:  z_r = y_r / D_r - sum_k L_kr z_k (rows of L^T, last first).
template <bool BWD>
__global__ void __launch_bounds__(64 * kLdlRowWaves)
    k_ldl_sweep(int n, const int *__restrict__ ptr, const int *__restrict__ idx, const double *__restrict__ val,
                const double *__restrict__ rhs, const double *__restrict__ D, const double *src, double *dst,
                int *fault, const KScal *ks) {
    if (ks && ks->done) return;
    const int w = blockIdx.x * kLdlRowWaves + (int)(threadIdx.x >> 6);
    if (w >= n) return;
    const int lane = threadIdx.x & 63;
    const int r = BWD ? n - 1 - w : w;
    const int p1 = ptr[r + 1];
    double acc = 0.0;
    // blocks of 64 * kLdlBatch entries: a lane loads all its inputs of a block
    // at once and then polls only those not yet published, so a row waits
    // about one load latency per block rather than one per entry
    for (int pb = ptr[r] + lane; pb < p1; pb += 64 * kLdlBatch) {
        double a[kLdlBatch], v[kLdlBatch];
        int c[kLdlBatch];
#pragma unroll
        for (int k = 0; k < kLdlBatch; ++k) {
            const int p = pb + 64 * k;
            c[k] = p < p1 ? idx[p] : 0;
            a[k] = p < p1 ? val[p] : 0.0;
        }
#pragma unroll
        for (int k = 0; k < kLdlBatch; ++k) v[k] = pb + 64 * k < p1 ? ldl_load(src + c[k]) : 0.0;
        for (int s = 0;; ++s) {
            bool missing = false;
#pragma unroll
            for (int k = 0; k < kLdlBatch; ++k) missing |= ldl_sent(v[k]);
            if (!missing) break;
            if (s >= kLdlSpin) {
                __hip_atomic_store(fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
#pragma unroll
            for (int k = 0; k < kLdlBatch; ++k)
                if (ldl_sent(v[k])) v[k] = ldl_load(src + c[k]);
        }
#pragma unroll
        for (int k = 0; k < kLdlBatch; ++k)
            if (pb + 64 * k < p1) acc = acc + a[k] * v[k];  // the lane's entries in order
    }
    const double s = wave_sum(acc);
    if (lane == 0) {
        const double base = BWD ? ldl_wait(rhs, r, fault) / D[r] : rhs[r];
        ldl_store(dst + r, base - s);
    }
}

// Block solves (the default; ldl_host.h has the algebra).  A range's rows do
// not wait for each other, so a solve is as deep as the dissection tree (one
// or two hand-overs between CUs per level), where the substitution was as deep
// as the separators are long.  Bound by those hand-overs' latency (about 5 us
// a level).  400 x 100 (1.3 M factor entries, 10 levels): 142 us an apply, the
// substitution range by range it replaces 1,990 us; 800 x 200: 240 us.
// Blocks of 8 waves:
//   kind 0: a range of at most 64 rows, or a leaf of at most 80, taken whole.
//     The waves take its rows' outside entries, four rows at once, r (backward:
//     s) into LDS; then thread = row, the columns of the inverse (in LDS,
//     loaded before the wait) split among the waves of a row group;
//     their sums are added in order;
//   kind 1: outside rows of a longer range, one wave each: r (s), published;
//   kind 2: its inverse rows, one wave each.
// A row's outside sum: lane l adds its entries l, l + 64, ... in order, then
// wave_total.  Whatever a block knows beforehand is loaded first.  Then one
// wave waits for the block's gates, the words of the nearest ranges in the
// tree, which are done last; behind them the inputs nearly always are all
// there (each is still tested, and polled if not).  When every wave polled all
// its inputs, or a word each, the requests to the few words that many blocks
// wait for held up the stores behind them: 10 us a level.
// Blocks are dispatched in list order and wait only for blocks before them, so
// the solve drains.
constexpr int kLdlPart = 2;  // entries per lane of a row loaded at once, four rows at a time ...
constexpr int kLdlLong = 6;  // ... or one row alone (6 measured best with four rows in flight)
constexpr int kLdlRows = 4;
constexpr int kLdlThreads = 64 * kLdlWaves;
constexpr int kLdlInv = kLdlLeaf * (kLdlLeaf - 1) / 2;  // words of a whole range's packed inverse
static_assert(kLdlWhole == 64 && kLdlLeaf <= 128 && kLdlWaves % 2 == 0, "thread = row, one or two groups of 64 rows");

// Part of a row: entries p0 + lane + 64 k < p1, k < P (c: -1 beyond).
template <int P>
struct LdlPart {
    int c[P];
    double a[P];
};
template <int P, class At>
__device__ inline void ldl_part(LdlPart<P> &q, int p0, int p1, const double *__restrict__ val, At at) {
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int p = p0 + (int)(threadIdx.x & 63) + 64 * k;
        q.c[k] = p < p1 ? at(p) : -1;
        q.a[k] = p < p1 ? val[p] : 0.0;
    }
}
// Adds the parts' products to acc, polling src until every input is there.
template <int N, int P>
__device__ inline void ldl_gather(const LdlPart<P> (&q)[N], const double *src, double (&acc)[N], int *lost) {
    double v[N][P];
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int k = 0; k < P; ++k) v[i][k] = q[i].c[k] >= 0 ? ldl_load(src + q[i].c[k]) : 0.0;
    for (int s = 0;; ++s) {
        bool missing = false;
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int k = 0; k < P; ++k) missing |= ldl_sent(v[i][k]);
        if (!missing) break;
        if (s >= kLdlSpin) {
            *lost = 1;
            break;
        }
        __builtin_amdgcn_s_sleep(2);
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int k = 0; k < P; ++k)
                if (ldl_sent(v[i][k])) v[i][k] = ldl_load(src + q[i].c[k]);
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int k = 0; k < P; ++k)
            if (q[i].c[k] >= 0) acc[i] = acc[i] + q[i].a[k] * v[i][k];
}
// Adds the parts after the first of row [p0, p1) to acc.
template <int P, class At>
__device__ inline double ldl_rest(double acc, int p0, int p1, const double *__restrict__ val, const double *src, At at,
                                  int *lost) {
    double a[1] = {acc};
    for (int p = p0 + 64 * P; p < p1; p += 64 * kLdlLong) {
        LdlPart<kLdlLong> q[1];
        ldl_part(q[0], p, p1, val, at);
        ldl_gather(q, src, a, lost);
    }
    return a[0];
}
// The block's gates (one wave), then the barrier behind which all go on.
__device__ inline void ldl_gates(const LdlBlock &b, const double *src, int *lost) {
    if (threadIdx.x < 2) {
        const int j = threadIdx.x ? b.gate[1] : b.gate[0];
        for (int s = 0; j >= 0 && ldl_sent(ldl_load(src + j)); ++s) {
            if (s >= kLdlSpin) {
                *lost = 1;
                break;
            }
            __builtin_amdgcn_s_sleep(4);
        }
    }
    __syncthreads();
}

template <bool BWD>
__global__ void __launch_bounds__(kLdlThreads)
    k_ldl_blocks(const LdlBlock *__restrict__ blocks, const int *__restrict__ ptr, const int *__restrict__ idx,
                 const double *__restrict__ val, const double *__restrict__ inv, const double *__restrict__ base,
                 const double *__restrict__ D, double *mid, double *out, int *fault, const KScal *ks) {
    if (ks && ks->done) return;
    constexpr int R = kLdlRows;
    __shared__ double loc[kLdlLeaf], sums[kLdlWaves][64], ivs[kLdlInv];
    const LdlBlock b = blocks[blockIdx.x];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, s = b.rows;
    const double *iv = inv + b.off;
    const auto at = [&](int p) { return idx[p]; };
    int lost = 0;
    if (b.kind == 0) {
        // ng row groups of 64; this wave: rows 64 rg + lane, columns k0 .. k0 + nc - 1
        // of the inverse (forward, column k holds rows k+1 .. s-1; backward, row k
        // holds columns 0 .. k-1)
        const int ng = s <= 64 ? 1 : 2, nc = (s * ng + kLdlWaves - 1) / kLdlWaves, row = 64 * (w % ng) + lane, k0 = (w / ng) * nc;
        for (int q = threadIdx.x; q < s * (s - 1) / 2; q += kLdlThreads) ivs[q] = iv[q];
        const bool outside = ptr[b.r0] < ptr[b.r0 + s];
        if (!outside) {
            if ((int)threadIdx.x < s) {
                const int r = b.r0 + threadIdx.x;
                loc[threadIdx.x] = BWD ? base[r] / D[r] : base[r];
            }
        } else {
            for (int i0 = w, first = 1; first || i0 - w < s; i0 += kLdlWaves * R, first = 0) {
                int p0[R], p1[R];
                double bs[R], acc[R];
                LdlPart<kLdlPart> part[R];
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    const int i = i0 + kLdlWaves * q, r = b.r0 + min(i, s - 1);
                    p0[q] = ptr[r];
                    p1[q] = i < s ? ptr[r + 1] : p0[q];
                    bs[q] = BWD ? base[r] / D[r] : base[r];
                    acc[q] = 0.0;
                }
#pragma unroll
                for (int q = 0; q < R; ++q) ldl_part(part[q], p0[q], p1[q], val, at);
                if (first) ldl_gates(b, out, &lost);
                ldl_gather(part, out, acc, &lost);
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    const double sum = wave_total(ldl_rest<kLdlPart>(acc[q], p0[q], p1[q], val, out, at, &lost));
                    const int i = i0 + kLdlWaves * q;
                    if (lane == 0 && i < s) loc[i] = bs[q] - sum;
                }
            }
        }
        __syncthreads();
        double t = 0.0;
#pragma unroll 4
        for (int q = 0; q < nc; ++q) {
            const int k = k0 + q;
            const bool in = k < s && row < s && (BWD ? row < k : row > k);
            const int o = BWD ? k * (k - 1) / 2 + row : k * (s - 1) - k * (k - 1) / 2 + (row - k - 1);
            t = t + (in ? ivs[o] * loc[k] : 0.0);
        }
        sums[w][lane] = t;
        __syncthreads();
        if (w < ng && row < s) {
            double y = loc[row];
            for (int k = w; k < kLdlWaves; k += ng) y = y + sums[k][lane];
            ldl_store(out + b.r0 + row, y);
        }
    } else {
        // kind 1: the outside entries of row r; kind 2: row i of the inverse
        // (forward: columns 0 .. i-1; backward: rows i+1 .. s-1 of column i)
        const int r = b.r + min(w, b.r0 + s - 1 - b.r), i = r - b.r0;
        const bool mine = b.r + w < b.r0 + s;
        const double *src = b.kind == 1 ? out : mid;
        LdlPart<kLdlLong> part[1];
        double acc[1] = {0.0};
        if (b.kind == 1) {
            const int p0 = ptr[r], p1 = ptr[r + 1];
            const double bs = BWD ? base[r] / D[r] : base[r];
            ldl_part(part[0], p0, p1, val, at);
            ldl_gates(b, src, &lost);
            ldl_gather(part, src, acc, &lost);
            const double sum = wave_total(ldl_rest<kLdlLong>(acc[0], p0, p1, val, src, at, &lost));
            if (lane == 0 && mine) ldl_store(mid + r, bs - sum);
        } else {
            const double *v = iv + (BWD ? i * (s - 1) - i * (i - 1) / 2 : i * (i - 1) / 2);
            const int first = BWD ? r + 1 : b.r0, len = BWD ? s - 1 - i : i;
            const auto in = [&](int p) { return first + p; };
            ldl_part(part[0], 0, len, v, in);
            ldl_gates(b, src, &lost);
            double own = ldl_load(mid + r);
            ldl_gather(part, src, acc, &lost);
            const double sum = wave_total(ldl_rest<kLdlLong>(acc[0], 0, len, v, src, in, &lost));
            if (ldl_sent(own)) own = ldl_wait(mid, r, fault);
            if (lane == 0 && mine) ldl_store(out + r, own + sum);
        }
    }
    if (lost) __hip_atomic_store(fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <typename T>
__global__ void k_ldl_out(int n, const int *__restrict__ perm, const double *__restrict__ z, T *__restrict__ out,
                          const KScal *ks) {
    if (ks && ks->done) return;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    out[perm[k]] = (T)z[k];
}

// Factor A (values of the equation the preconditioner reads) on the host,
// once, and upload L by rows (forward) and by columns (backward).
int ldl_setup(fvh_eqn *e, const double *val_dev) {
    fvh_mesh *m = e->m;
    LdlStore &S = e->ldl;
    if (S.ready) return FVH_OK;  // frozen after the set-up factorization
    if (m->cases) return set_error(FVH_ERR_UNSUPPORTED, "LDL preconditioner: not with independent cases");
    const int n = (int)m->n;
    std::vector<double> val(m->nnz), cx(n), cy(n);
    // the values may still be in assembly on the library's stream (a
    // non-blocking stream, which the synchronous copies below do not wait for)
    HIP_TRY(hipStreamSynchronize(stream()));
    HIP_TRY(hipMemcpy(val.data(), val_dev, sizeof(double) * m->nnz, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(cx.data(), m->ccx.p, sizeof(double) * n, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(cy.data(), m->ccy.p, sizeof(double) * n, hipMemcpyDeviceToHost));
    std::vector<int> perm, bounds;
    ldl_order(n, m->h_rowptr.data(), m->h_col.data(), cx.data(), cy.data(), perm, &bounds);
    LdlHost F;
    FVH_TRY(ldl_factor(n, m->h_rowptr.data(), m->h_col.data(), val.data(), perm, F));
    const char *env = std::getenv("FVH_LDL_RANGES");
    S.by_blocks = !(env && env[0] == '0' && env[1] == 0);
    if (S.by_blocks) {
        LdlBlocks B;
        ldl_blocks(F, bounds, B);
        for (int k = 0; k < 2; ++k) {
            const LdlSide &h = k ? B.b : B.f;
            LdlSideDev &d = k ? S.b : S.f;
            FVH_TRY(d.ptr.upload(h.ptr));
            FVH_TRY(d.idx.upload(h.idx));
            FVH_TRY(d.val.upload(h.val));
            FVH_TRY(d.inv.upload(h.inv));
            FVH_TRY(d.blocks.upload(h.blocks));
            d.nblocks = (int)h.blocks.size();
        }
        FVH_TRY(S.r.alloc(n));
        FVH_TRY(S.s.alloc(n));
    } else {
        // rows of L (strictly lower, columns ascending) from its columns
        const int nnzL = F.Lp[n];
        std::vector<int> rp(n + 1, 0), ri(nnzL);
        std::vector<double> rv(nnzL);
        for (int p = 0; p < nnzL; ++p) rp[F.Li[p] + 1]++;
        for (int i = 0; i < n; ++i) rp[i + 1] += rp[i];
        {
            std::vector<int> pos(rp.begin(), rp.end() - 1);
            for (int j = 0; j < n; ++j)
                for (int p = F.Lp[j]; p < F.Lp[j + 1]; ++p) {
                    const int q = pos[F.Li[p]]++;
                    ri[q] = j;
                    rv[q] = F.Lx[p];
                }
        }
        FVH_TRY(S.f.ptr.upload(rp));
        FVH_TRY(S.f.idx.upload(ri));
        FVH_TRY(S.f.val.upload(rv));
        FVH_TRY(S.b.ptr.upload(F.Lp));
        FVH_TRY(S.b.idx.upload(F.Li));
        FVH_TRY(S.b.val.upload(F.Lx));
        S.r.release();
        S.s.release();
    }
    FVH_TRY(S.perm.upload(F.perm));
    FVH_TRY(S.D.upload(F.D));
    FVH_TRY(S.rhs.alloc(n));
    FVH_TRY(S.y.alloc(n));
    FVH_TRY(S.z.alloc(n));
    if (!S.h_fault) {
        HIP_TRY(hipHostMalloc((void **)&S.h_fault, sizeof(int), hipHostMallocCoherent | hipHostMallocMapped));
        *S.h_fault = 0;
    }
    S.ready = true;
    return FVH_OK;
}

template <typename T>
int ldl_apply(fvh_eqn *e, const T *x, T *out, const KScal *ks) {
    LdlStore &S = e->ldl;
    if (!S.ready) return set_error(FVH_ERR_ARG, "LDL preconditioner applied before its set-up factorization");
    const int n = (int)e->m->n;
    int *fault = nullptr;
    HIP_TRY(hipHostGetDevicePointer((void **)&fault, S.h_fault, 0));
    hipLaunchKernelGGL((k_ldl_prep<T>), grid1d(n), dim3(256), 0, stream(), n, S.perm.p, x, S.rhs.p, S.y.p, S.z.p,
                       S.r.p, S.s.p, ks);
    HIP_TRY(hipGetLastError());
    if (S.by_blocks) {
        hipLaunchKernelGGL((k_ldl_blocks<false>), dim3((unsigned)S.f.nblocks), dim3(kLdlThreads), 0, stream(), S.f.blocks.p,
                           S.f.ptr.p, S.f.idx.p, S.f.val.p, S.f.inv.p, S.rhs.p, S.D.p, S.r.p, S.y.p, fault, ks);
        HIP_TRY(hipGetLastError());
        hipLaunchKernelGGL((k_ldl_blocks<true>), dim3((unsigned)S.b.nblocks), dim3(kLdlThreads), 0, stream(), S.b.blocks.p,
                           S.b.ptr.p, S.b.idx.p, S.b.val.p, S.b.inv.p, S.y.p, S.D.p, S.s.p, S.z.p, fault, ks);
        HIP_TRY(hipGetLastError());
    } else {
        const dim3 g((unsigned)((n + kLdlRowWaves - 1) / kLdlRowWaves));
        hipLaunchKernelGGL((k_ldl_sweep<false>), g, dim3(64 * kLdlRowWaves), 0, stream(), n, S.f.ptr.p, S.f.idx.p,
                           S.f.val.p, S.rhs.p, S.D.p, S.y.p, S.y.p, fault, ks);
        HIP_TRY(hipGetLastError());
        hipLaunchKernelGGL((k_ldl_sweep<true>), g, dim3(64 * kLdlRowWaves), 0, stream(), n, S.b.ptr.p, S.b.idx.p,
                           S.b.val.p, S.y.p, S.D.p, S.z.p, S.z.p, fault, ks);
        HIP_TRY(hipGetLastError());
    }
    hipLaunchKernelGGL((k_ldl_out<T>), grid1d(n), dim3(256), 0, stream(), n, S.perm.p, S.z.p, out, ks);
    HIP_TRY(hipGetLastError());
    return FVH_OK;
}
template int ldl_apply<double>(fvh_eqn *, const double *, double *, const KScal *);
template int ldl_apply<float>(fvh_eqn *, const float *, float *, const KScal *);

// A wait of the last solves ran out (reported once).
int ldl_check(fvh_eqn *e) {
    int *f = e->ldl.h_fault;
    if (f && __atomic_load_n(f, __ATOMIC_ACQUIRE)) {
        __atomic_store_n(f, 0, __ATOMIC_RELEASE);
        return set_error(FVH_ERR_HIP, "LDL solve: a row's input did not arrive in time");
    }
    return FVH_OK;
}

}  // namespace fvh
