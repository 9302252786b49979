// Kronecker ILUT preconditioner on the GPU: Y = (LU)^-1 X Minv_r^T.
//
// Restates kronlusol (kronecker.f90:130-178) and lusol (ilut.f:2383-2432).  The
// reference inverts the q x q temporal matrix A, runs q scalar forward/backward
// sweeps over the MSR factors of ilut and mixes the q results with inv(A).
// Here the temporal mix is applied first (it commutes with the spatial solve),
// and the q*R columns of every row are solved together: rows are grouped into
// dependency levels (level(i) = 1 + max level of the rows it reads), and each
// level is one launch in which lane (row, column) performs the reference's
// row update x_i = y_i - sum_k alu(k) x(jlu(k)) (backward: times the stored
// inverse diagonal) in the reference's entry order.
#include <algorithm>
#include <atomic>
#include <numeric>

#include "xt_common.h"

namespace xt {

template <typename T>
__global__ void __launch_bounds__(256)
trsv_level_kernel(int nrows, const int *__restrict__ rows, const int *__restrict__ rp,
                  const int *__restrict__ ci, const T *__restrict__ v,
                  const T *__restrict__ dinv, int c, const T *__restrict__ b, T *__restrict__ x) {
    long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)nrows * c) return;
    const int k = (int)(idx / c);
    const int col = (int)(idx - (long long)k * c);
    const int row = rows[k];
    const size_t o = (size_t)row * c + col;
    T s = b ? b[o] : x[o];
    const int e1 = rp[row + 1];
    for (int e = rp[row]; e < e1; ++e) s -= v[e] * x[(size_t)ci[e] * c + col];
    if (dinv) s *= dinv[row];
    x[o] = s;
}

// Both sweeps in one workgroup (small factors): the levels are walked in order with a
// barrier between levels instead of one launch per level, then the upper levels.
// Same per-row arithmetic and order as trsv_level_kernel.  XL: the solution vector
// lives in LDS during the sweeps (dynamic shared memory of n*c elements).
template <typename T, bool XL>
__global__ void __launch_bounds__(1024)
trsv_onewg_kernel(int n_, int nlevL, const int *__restrict__ lpL, const int *__restrict__ rowsL,
                  const int *__restrict__ rpL, const int *__restrict__ ciL,
                  const T *__restrict__ vL, int nlevU, const int *__restrict__ lpU,
                  const int *__restrict__ rowsU, const int *__restrict__ rpU,
                  const int *__restrict__ ciU, const T *__restrict__ vU,
                  const T *__restrict__ dinv, int c, const T *__restrict__ b, T *xg) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T *x = XL ? reinterpret_cast<T *>(smem_raw) : xg;
    for (int l = 0; l < nlevL; ++l) {
        const int r0 = lpL[l], n = (lpL[l + 1] - r0) * c;
        for (int idx = threadIdx.x; idx < n; idx += blockDim.x) {
            const int k = idx / c, col = idx - k * c;
            const int row = rowsL[r0 + k];
            const size_t o = (size_t)row * c + col;
            T s = b[o];
            const int e1 = rpL[row + 1];
            for (int e = rpL[row]; e < e1; ++e) s -= vL[e] * x[(size_t)ciL[e] * c + col];
            x[o] = s;
        }
        __syncthreads();
    }
    for (int l = 0; l < nlevU; ++l) {
        const int r0 = lpU[l], n = (lpU[l + 1] - r0) * c;
        for (int idx = threadIdx.x; idx < n; idx += blockDim.x) {
            const int k = idx / c, col = idx - k * c;
            const int row = rowsU[r0 + k];
            const size_t o = (size_t)row * c + col;
            T s = x[o];
            const int e1 = rpU[row + 1];
            for (int e = rpU[row]; e < e1; ++e) s -= vU[e] * x[(size_t)ciU[e] * c + col];
            x[o] = dinv[row] * s;
        }
        __syncthreads();
    }
    if (XL)
        for (int i = threadIdx.x; i < n_ * c; i += blockDim.x) xg[i] = x[i];
}

// Both sweeps of kSfCols columns in one workgroup without a barrier per level (the columns
// are independent, a workgroup for each kSfCols of them): each wave takes rows in level order
// (tasks w, w + nwaves, ... of the level-ordered rows of L, then of U) and starts a row as
// soon as the rows it reads are finished.  The forward and the backward results live in LDS
// and are their own flags: an entry holds a NaN of a reserved bit pattern until its value is
// stored, so one LDS read tells a lane both that its row is finished and its value.  Every
// row depends only on rows earlier in that order and each wave walks its rows in that order,
// so the earliest unfinished row can always proceed.  Half a wave works on a column: the
// entry whose row comes last in the order is left for the end, the next kSlot sit in a
// fixed-size slot in level order, one a lane, so a wave loads its next two rows' entries with
// no dependent address while it waits for and computes the current one, and their products
// are summed by DPP lane moves in a fixed order before the last entry is waited for.  Waits
// are bounded: a wave that waits past kSpinMax polls raises an abort flag that releases every
// wave, and the output is then NaN.
//
// What bounds it: the chain of levels, each a store to LDS, a poll that sees it and the last
// product, 220 to 280 ns.  6 columns: 975 rows, 286 + 243 levels 287 us (one workgroup for
// all columns, separate flags, 8 lanes a column) -> 148; 2727 rows, 1936 + 1808 levels,
// which did not fit one workgroup's LDS, 5 ms (a barrier a level) -> 0.84.  Without the last entry kept
// apart 149 and 1010; polls with pauses, 8 or 16 waves: no better.
constexpr int kSlot = 32;           // leading entries of a row kept in its fixed-size slot
constexpr int kSfCols = 64 / kSlot; // columns of a workgroup
constexpr int kSfMaxRows = 4096;    // slots are built for factors up to this order
constexpr int kSpinMax = 1 << 22;

// LDS: forward and backward results [(n + 1) kSfCols] each (row n: always finished, zero),
// abort flag.  (At most 131 KB.)
template <typename T>
static size_t sf_lds_bytes(int n) {
    return sizeof(T) * 2 * ((size_t)n + 1) * kSfCols + 16;
}

// An entry that is not finished yet; results never hold the pattern (they are NaN then, and
// a NaN of another pattern is stored).
template <typename T> struct Unfinished;
template <> struct Unfinished<double> {
    static constexpr int kHigh = 0x7FFADEAD;
    static __device__ __forceinline__ double pattern() { return __hiloint2double(kHigh, 0); }
    static __device__ __forceinline__ bool is(double v) { return __double2hiint(v) == kHigh; }
};
template <> struct Unfinished<float> {
    static constexpr int kBits = 0x7FDADEAD;
    static __device__ __forceinline__ float pattern() { return __int_as_float(kBits); }
    static __device__ __forceinline__ bool is(float v) { return __float_as_int(v) == kBits; }
};

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// Sum over each half of the wave, in its last 16 lanes: within each row of 16 lanes by
// swapping neighbours, pairs, quads and eights, then the lower row's sum to the upper.
template <typename T>
__device__ __forceinline__ T half_sum(T s) {
    s += dpp_move<0xB1>(s);     // quad_perm [1,0,3,2]
    s += dpp_move<0x4E>(s);     // quad_perm [2,3,0,1]
    s += dpp_move<0x141>(s);    // row_half_mirror
    s += dpp_move<0x140>(s);    // row_mirror
    return s + dpp_move<0x142>(s);   // row_bcast:15
}

template <typename V>
__device__ __forceinline__ V lds_load(const V *f) {
    return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// One triangle as the single-workgroup sweep reads it (device pointers): the first kSlot
// entries of each row in its slot, rows in level order (the column, n past the row; the row in
// bits 13 to 25, bit 30 set when it has more than kSlot entries; values, 0 past the row), and
// the CSR for the entries past the slot.
constexpr int kSfBits = 13;
static_assert(kSfMaxRows < (1 << kSfBits), "column and row share a word");
struct SfTri {
    const int *sci, *lci, *rp, *ci;
    const void *sv, *lv, *v;
};

template <typename T>
__global__ void __launch_bounds__(768)
trsv_sf_kernel(int n, int c, SfTri L, SfTri U, const T *__restrict__ dinv, const T *b, T *xg) {
    using Un = Unfinished<T>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T *xf = reinterpret_cast<T *>(smem_raw);
    T *xb = xf + (size_t)(n + 1) * kSfCols;
    int *abort_flag = reinterpret_cast<int *>(xb + (size_t)(n + 1) * kSfCols);
    const int tid = threadIdx.x, nt = blockDim.x;
    const int c0 = blockIdx.x * kSfCols, nc = min(kSfCols, c - c0);
    for (int i = tid; i < (n + 1) * kSfCols; i += nt) {
        xf[i] = i < n * kSfCols ? Un::pattern() : T(0);
        xb[i] = i < n * kSfCols ? Un::pattern() : T(0);
    }
    if (tid == 0) *abort_flag = 0;
    __syncthreads();
    const int lane = tid & 63, nw = nt >> 6, ntask = 2 * n;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane & (kSlot - 1), col = lane / kSlot;
    const int colb = col < nc ? col : 0;     // (a missing column repeats the first)
    auto sf_row = [](int w) { return (w >> kSfBits) & ((1 << kSfBits) - 1); };
    struct Task {
        int pc, lc;          // row and column of this lane's entry, column of the last one
        T pv, lv, own, di;   // their values; b of the row, inverse diagonal
    };
    // task t < n: forward row of level-ordered position t; t >= n: backward row at t - n.
    // Branch-free loads (t clamped to the last task) with no use here, so they stay in
    // flight while the wave works on earlier tasks.
    auto load_row = [&](int t, Task &k) {
        t = t < ntask ? t : ntask - 1;
        const bool up = t >= n;
        const int pos = up ? t - n : t;
        const size_t e = (size_t)pos * kSlot + q;
        k.pc = (up ? U.sci : L.sci)[e];
        k.pv = static_cast<const T *>(up ? U.sv : L.sv)[e];
        const int z = pos + (lane >> 6);     // (a vector load)
        k.lc = (up ? U.lci : L.lci)[z];
        k.lv = static_cast<const T *>(up ? U.lv : L.lv)[z];
    };
    auto load_own = [&](Task &k) {           // once its row is known
        const int row = sf_row(k.pc);
        k.own = b[(size_t)row * c + c0 + colb];
        k.di = dinv[row];
    };
    auto process = [&](int t, const Task &k) {
        const bool up = t >= n;
        const int row = sf_row(k.pc);
        T *xs = up ? xb : xf;
        const T *pe = xs + (k.pc & ((1 << kSfBits) - 1)) * kSfCols + col;
        // backward: the row's forward result as well (forward: the finished zero)
        const T *po = xf + (up ? row : n) * kSfCols + col;
        T v, own;
        int spins = 0;
        auto give_up = [&]() {   // after too many polls, or when another wave did
            if ((++spins & 63) == 0) {
                if (lds_load(abort_flag)) return true;
                if (spins >= kSpinMax) {
                    __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_WORKGROUP);
                    return true;
                }
            }
            return false;
        };
        for (;;) {
            v = lds_load(pe);
            own = lds_load(po);
            if (__all(!Un::is(v) && !Un::is(own)) || give_up()) break;
        }
        T s = k.pv * v;
        if (k.pc >> 30) {
            const int *rp = up ? U.rp : L.rp, *ci = up ? U.ci : L.ci;
            const T *va = static_cast<const T *>(up ? U.v : L.v);
            for (int e = rp[row] + kSlot + 1 + q; e < rp[row + 1]; e += kSlot) {
                const T *px = xs + ci[e] * kSfCols + col;
                while (v = lds_load(px), Un::is(v) && !give_up()) {}
                s += va[e] * v;
            }
        }
        const T part = (up ? own : k.own) - half_sum(s);
        const T *pl = xs + k.lc * kSfCols + col;
        for (;;) {
            v = lds_load(pl);
            if (__all(!Un::is(v)) || give_up()) break;
        }
        T r = part - k.lv * v;
        if (up) r *= k.di;
        if (Un::is(r)) r = T(__builtin_nan(""));
        if (q == kSlot - 1)
            __hip_atomic_store(xs + row * kSfCols + col, r, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    // three register sets in turn: the entries of tasks t + nw and t + 2 nw and the own
    // values of t + nw fly while task t is processed (compiler fences keep them issued
    // before the current task's work)
    Task A, B, C;
    load_row(wave, A);
    load_row(wave + nw, B);
    load_own(A);
#define XT_SF_STEP(T0, K, K1, K2)                                                              \
    load_row((T0) + 2 * nw, K2);                                                               \
    load_own(K1);                                                                              \
    __atomic_signal_fence(__ATOMIC_SEQ_CST);                                                   \
    process(T0, K);
    for (int t = wave; t < ntask; t += 3 * nw) {
        XT_SF_STEP(t, A, B, C)
        if (t + nw >= ntask) break;
        XT_SF_STEP(t + nw, B, C, A)
        if (t + 2 * nw >= ntask) break;
        XT_SF_STEP(t + 2 * nw, C, A, B)
    }
#undef XT_SF_STEP
    __syncthreads();
    const bool bad = lds_load(abort_flag) != 0;
    for (int i = tid; i < n * nc; i += nt) {
        const int row = i / nc, j = i - row * nc;
        xg[(size_t)row * c + c0 + j] = bad ? T(__builtin_nan("")) : xb[row * kSfCols + j];
    }
}

// Level schedule of a triangular CSR: forward (lower) or backward (upper).
static void build_levels(int n, const std::vector<int> &rp, const std::vector<int> &ci,
                         bool forward, std::vector<int> &lev_ptr, std::vector<int> &lev_rows) {
    std::vector<int> lev(n, 0);
    int nlev = 0;
    for (int t = 0; t < n; ++t) {
        const int i = forward ? t : n - 1 - t;
        int l = 0;
        for (int e = rp[i]; e < rp[i + 1]; ++e) l = std::max(l, lev[ci[e]] + 1);
        lev[i] = l;
        nlev = std::max(nlev, l + 1);
    }
    lev_ptr.assign(nlev + 1, 0);
    for (int i = 0; i < n; ++i) lev_ptr[lev[i] + 1]++;
    for (int l = 0; l < nlev; ++l) lev_ptr[l + 1] += lev_ptr[l];
    lev_rows.resize(n);
    std::vector<int> fill(lev_ptr.begin(), lev_ptr.end() - 1);
    for (int t = 0; t < n; ++t) {
        const int i = forward ? t : n - 1 - t;
        lev_rows[fill[lev[i]]++] = i;
    }
}

struct Tri {
    DevCSR m;                    // strict triangle, 0-based, reference entry order
    DevBuf lev_rows;             // rows sorted by level
    std::vector<int> lev_ptr;    // host copy of level boundaries
    DevBuf lev_ptr_dev;          // device copy (single-workgroup sweeps)
    std::vector<long long> lev_nnz;  // entries per level (algorithmic bytes)
    // single-workgroup sweeps (small factors only): level-ordered rows with the long-row
    // bit, fixed-size entry slots
    DevBuf last_ci, last_v64, last_v32, slot_ci, slot_v64, slot_v32;
};

}  // namespace xt

using namespace xt;

namespace xt {
std::atomic<unsigned long long> g_prec_ids{0};
}
struct xt_prec_s {
    unsigned long long id = ++xt::g_prec_ids;   // never reused, unlike the handle's address
    int p = 0;
    Tri L, U;                  // ILUT factors (level-scheduled solves)
    DevBuf dinv64, dinv32;
    DevBuf work;
    BandPrec *band = nullptr;  // or: exact banded factor (block sweeps)
    // shifted factors (K + s_g M)^-1 of the temporal split, and their gathered columns
    std::vector<double> shifts;
    std::vector<BandPrec *> shifted;
    DevBuf gin[2], gout[2];    // [0] FP64, [1] FP32
    // or: banded factors of runs of independent systems, run g on DOFs goff[g]..goff[g+1]-1
    std::vector<BandPrec *> groups;
    std::vector<int> goff;
    ~xt_prec_s() {
        if (band) band_delete(band);
        for (BandPrec *b : shifted) band_delete(b);
        for (BandPrec *b : groups) band_delete(b);
    }
};

namespace xt {

int prec_rows(xt_prec pr) { return pr ? pr->p : -1; }

static int upload_tri(int n, const std::vector<int> &rp, const std::vector<int> &ci,
                      const std::vector<double> &v, bool forward, Tri &T) {
    T.m.n = n;
    T.m.nnz = rp[n];
    XT_TRY(T.m.rowptr.upload(rp.data(), sizeof(int) * (n + 1)));
    // one zero entry past the end: the single-workgroup sweeps read it, branch-free, in
    // place of a missing entry
    std::vector<int> cp(ci);
    std::vector<double> vp(v);
    cp.push_back(0);
    vp.push_back(0.0);
    XT_TRY(T.m.col.upload(cp.data(), sizeof(int) * cp.size()));
    XT_TRY(T.m.val64.upload(vp.data(), sizeof(double) * vp.size()));
    std::vector<float> v32(vp.begin(), vp.end());
    XT_TRY(T.m.val32.upload(v32.data(), sizeof(float) * v32.size()));
    std::vector<int> lrows;
    build_levels(n, rp, ci, forward, T.lev_ptr, lrows);
    XT_TRY(T.lev_ptr_dev.upload(T.lev_ptr.data(), sizeof(int) * T.lev_ptr.size()));
    T.lev_nnz.assign(T.lev_ptr.size() - 1, 0);
    for (size_t l = 0; l + 1 < T.lev_ptr.size(); ++l)
        for (int k = T.lev_ptr[l]; k < T.lev_ptr[l + 1]; ++k)
            T.lev_nnz[l] += rp[lrows[k] + 1] - rp[lrows[k]];
    XT_TRY(T.lev_rows.upload(lrows.data(), sizeof(int) * n));
    if (n <= kSfMaxRows) {
        std::vector<int> sci((size_t)n * kSlot), lci(n), at(n);
        std::vector<double> sv((size_t)n * kSlot, 0.0), lv(n, 0.0);
        for (int k = 0; k < n; ++k) at[lrows[k]] = k;
        for (int k = 0; k < n; ++k) {
            const int r = lrows[k], len = rp[r + 1] - rp[r], flag = len > kSlot + 1 ? 1 << 30 : 0;
            int last = rp[r];                // among the first kSlot + 1 entries
            for (int e = rp[r]; e < rp[r] + std::min(len, kSlot + 1); ++e)
                if (at[ci[e]] > at[ci[last]]) last = e;
            lci[k] = len ? ci[last] : n;
            lv[k] = len ? v[last] : 0.0;
            for (int q = 0, e = rp[r]; q < kSlot; ++q, ++e) {
                if (e == last && len) ++e;
                const bool in = e < rp[r + 1];
                sci[(size_t)k * kSlot + q] = (in ? ci[e] : n) | r << kSfBits | flag;
                if (in) sv[(size_t)k * kSlot + q] = v[e];
            }
        }
        std::vector<float> sv32(sv.begin(), sv.end()), lv32(lv.begin(), lv.end());
        XT_TRY(T.last_ci.upload(lci.data(), sizeof(int) * n));
        XT_TRY(T.last_v64.upload(lv.data(), sizeof(double) * n));
        XT_TRY(T.last_v32.upload(lv32.data(), sizeof(float) * n));
        XT_TRY(T.slot_ci.upload(sci.data(), sizeof(int) * sci.size()));
        XT_TRY(T.slot_v64.upload(sv.data(), sizeof(double) * sv.size()));
        XT_TRY(T.slot_v32.upload(sv32.data(), sizeof(float) * sv32.size()));
    }
    XT_HIP(hipDeviceSynchronize());
    return XT_OK;
}

template <typename T>
static int run_tri(const Tri &tri, const T *vals, const T *dinv, int c, const T *b, T *x,
                   bool timed, hipStream_t s) {
    const int nlev = (int)tri.lev_ptr.size() - 1;
    const int *rows = tri.lev_rows.as<int>();
    for (int l = 0; l < nlev; ++l) {
        const int r0 = tri.lev_ptr[l], nr = tri.lev_ptr[l + 1] - r0;
        if (!nr) continue;
        long long n = (long long)nr * c;
        const bool prof = timed && prof_on(XT_PROF_TRSV);
        if (prof) prof_begin(XT_PROF_TRSV, s);
        hipLaunchKernelGGL(trsv_level_kernel<T>, dim3(ceil_div(n, 256)), dim3(256), 0, s, nr,
                           rows + r0, tri.m.rowptr.as<int>(), tri.m.col.as<int>(), vals, dinv,
                           c, b, x);
        if (prof) {   // level rows: values + column indices of their entries, row data, x
            const double nnz = (double)(tri.lev_nnz[l]);
            prof_end(XT_PROF_TRSV, s, nnz * (sizeof(T) + 4) + nr * 12.0 +
                                          (double)nr * c * sizeof(T) * (b ? 2 : 1) +
                                          nnz * c * sizeof(T), 2.0 * nnz * c);
        }
    }
    XT_HIP(hipGetLastError());
    return XT_OK;
}

// Sweeps whose work (factor entries + diagonal, times columns) is at most this run in a
// single workgroup.
constexpr long long kOneWgWork = 4LL << 20;
// ... and keep the solution vector in LDS when it fits this many bytes.
constexpr size_t kOneWgLds = 128 * 1024;
// Whether both sweeps in a workgroup for each two columns (trsv_sf_kernel) beat the kernels
// above, by estimates in us of what each is bound by (rl: mean entries of a factor row):
//   two columns a workgroup  its rows, 0.1 for both sweeps, or its levels, 0.2 + 0.006 rl
//                            (512 columns at a time)
//   one workgroup            a barrier a level and its longest row, 0.45 + 0.11 rl, and every
//                            entry and column, 0.45 ns
//   a launch a level         3.7 + 0.1 rl
// Two columns / the others, us, 6 columns: 4000 rows, 80 levels of 1 entry a row 404 / 65, 800
// levels 405 / 410, 7950 levels of 34 entries 3150 / 34500; 300 rows, 40 levels 36 / 25, 86
// levels 37 / 43; 975 rows, 529 levels of 17 entries 149 / 1105.  Over 1106 factors and column
// counts the choice takes 1.004 times the better one's time (1.36 by levels per row alone).
static bool two_columns_pay(const xt_prec_s &pr, int c) {
    const double p = pr.p, nnz = (double)(pr.L.m.nnz + pr.U.m.nnz), rl = nnz / (2 * p);
    const double levels = (double)(pr.L.lev_ptr.size() + pr.U.lev_ptr.size()) - 2;
    const double sf = std::max(6 + 0.1 * p, levels * (0.2 + 0.006 * rl)) * ceil_div(c, 512);
    const bool one = (nnz + 2 * p) * c <= kOneWgWork;
    return sf <= (one ? levels * (0.45 + 0.11 * rl) + 0.45e-3 * (nnz + 2 * p) * c
                      : levels * (3.7 + 0.1 * rl));
}
// ILUT sweeps Y = (LU)^-1 X Minv_r^T.  stage: p*q*R elements of device memory for the
// temporal mix (used only when minv is given); timed: per-launch HIP-event timing when
// enabled (it creates events, so the allocation-free entry point passes false).
template <typename T>
static int ilut_apply(xt_prec pr, int R, int q, const T *minv, const T *x, T *y, bool f32,
                      T *stage, bool timed, hipStream_t s) {
    const int c = q * R;
    const T *b = x;
    if (minv) {
        XT_TRY(temporal_mix<T, T>(pr->p, q, R, minv, x, stage, s));
        b = stage;
    }
    const T *lv = f32 ? (const T *)pr->L.m.val32.ptr : (const T *)pr->L.m.val64.ptr;
    const T *uv = f32 ? (const T *)pr->U.m.val32.ptr : (const T *)pr->U.m.val64.ptr;
    const T *dv = f32 ? (const T *)pr->dinv32.ptr : (const T *)pr->dinv64.ptr;
    // Factors with slots: both sweeps of two columns in one workgroup where that pays.  Others
    // of little work: one workgroup with a barrier per level; else one launch per level over
    // the whole device.
    const long long work = (pr->L.m.nnz + pr->U.m.nnz + 2LL * pr->p) * c;
    const bool slots = pr->L.slot_ci.ptr && pr->U.slot_ci.ptr && c <= 4096 &&
                       two_columns_pay(*pr, c);
    if (slots || work <= kOneWgWork) {
        const bool prof = timed && prof_on(XT_PROF_TRSV);
        if (prof) prof_begin(XT_PROF_TRSV, s);
        const size_t xl = sizeof(T) * (size_t)pr->p * c;
        if (slots) {
            auto tri = [&](const Tri &t, const T *vals) {
                SfTri w;
                w.sci = t.slot_ci.as<int>();
                w.sv = f32 ? t.slot_v32.ptr : t.slot_v64.ptr;
                w.lci = t.last_ci.as<int>();
                w.lv = f32 ? t.last_v32.ptr : t.last_v64.ptr;
                w.rp = t.m.rowptr.as<int>();
                w.ci = t.m.col.as<int>();
                w.v = vals;
                return w;
            };
            // (12 waves: levels up to 6 rows wide keep that many busy; 16 poll more, 8 are few
            // for the widest)
            hipLaunchKernelGGL(trsv_sf_kernel<T>, dim3(ceil_div(c, kSfCols)), dim3(768),
                               sf_lds_bytes<T>(pr->p), s, pr->p, c, tri(pr->L, lv),
                               tri(pr->U, uv), dv, b, y);
        } else {
#define XT_ONEWG(XLDS)                                                                      \
    hipLaunchKernelGGL((trsv_onewg_kernel<T, XLDS>), dim3(1), dim3(1024), XLDS ? xl : 0, s,  \
                       pr->p, (int)pr->L.lev_ptr.size() - 1, pr->L.lev_ptr_dev.as<int>(),     \
                       pr->L.lev_rows.as<int>(), pr->L.m.rowptr.as<int>(),                    \
                       pr->L.m.col.as<int>(), lv, (int)pr->U.lev_ptr.size() - 1,              \
                       pr->U.lev_ptr_dev.as<int>(), pr->U.lev_rows.as<int>(),                 \
                       pr->U.m.rowptr.as<int>(), pr->U.m.col.as<int>(), uv, dv, c, b, y)
            if (xl <= kOneWgLds) XT_ONEWG(true);
            else XT_ONEWG(false);
#undef XT_ONEWG
        }
        if (prof)
            prof_end(XT_PROF_TRSV, s,
                     (double)(pr->L.m.nnz + pr->U.m.nnz) * (sizeof(T) + 4 + c * sizeof(T)) +
                         (double)pr->p * c * sizeof(T) * 3,
                     2.0 * (pr->L.m.nnz + pr->U.m.nnz) * c);
        XT_HIP(hipGetLastError());
        return XT_OK;
    }
    XT_TRY(run_tri<T>(pr->L, lv, nullptr, c, b, y, timed, s));
    XT_TRY(run_tri<T>(pr->U, uv, dv, c, nullptr, y, timed, s));
    return XT_OK;
}

// Gathered column of split case t: g[base_t + dof * stride_t] = sum_j m2_t[j] X[dof][r_t q + j]
template <typename T>
__global__ void __launch_bounds__(256)
split_gather_kernel(int p, int q, int c, int ns, const int *__restrict__ cs,
                    const long long *__restrict__ base, const int *__restrict__ stride,
                    const T *__restrict__ m2v, const T *__restrict__ x, T *__restrict__ g) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)p * ns) return;
    const long long dof = idx / ns;
    const int t = (int)(idx - dof * ns);
    const T *m2 = m2v + (size_t)t * 2 * q;
    const T *xr = x + dof * c + (long long)cs[t] * q;
    T acc = 0;
    for (int j = 0; j < q; ++j) acc += m2[j] * xr[j];
    g[base[t] + dof * stride[t]] = acc;
}

// Y[dof][r_t q + j] += v_t[j] h[base_t + dof * stride_t] (each case is one t at most)
template <typename T>
__global__ void __launch_bounds__(256)
split_scatter_kernel(int p, int q, int c, int ns, const int *__restrict__ cs,
                     const long long *__restrict__ base, const int *__restrict__ stride,
                     const T *__restrict__ m2v, const T *__restrict__ h, T *__restrict__ y) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)p * ns) return;
    const long long dof = idx / ns;
    const int t = (int)(idx - dof * ns);
    const T *v = m2v + (size_t)t * 2 * q + q;
    const T hv = h[base[t] + dof * stride[t]];
    T *yr = y + dof * c + (long long)cs[t] * q;
    for (int j = 0; j < q; ++j) yr[j] += v[j] * hv;
}

template <typename T>
int prec_apply_t(xt_prec pr, int R, int q, const T *minv, const T *x, T *y, bool f32,
                 hipStream_t s, const ActiveCols *ac) {
    if (pr->band)
        return band_apply<T>(pr->band, R, q, minv, x, y, s, ac ? ac->Ra[0] : -1,
                             ac ? ac->dcols : nullptr);
    if (!pr->groups.empty()) {   // rows of run g: goff[g] .. goff[g+1]-1, all R q columns
        const long long c = (long long)q * R;
        for (size_t g = 0; g < pr->groups.size(); ++g)
            XT_TRY(band_apply<T>(pr->groups[g], R, q, minv, x + pr->goff[g] * c,
                                 y + pr->goff[g] * c, s, ac ? ac->Ra[g] : -1,
                                 ac ? ac->dcols + g * R : nullptr));
        return XT_OK;
    }
    T *stage = nullptr;
    if (minv) {   // sized for FP64, so switching precision does not reallocate
        XT_TRY(pr->work.reserve(sizeof(double) * (size_t)pr->p * q * R));
        stage = pr->work.as<T>();
    }
    return ilut_apply<T>(pr, R, q, minv, x, y, f32, stage, true, s);
}
unsigned long long prec_id(xt_prec pr) { return pr->id; }
void prec_runs(xt_prec pr, std::vector<long long> &off) {
    off.clear();
    if (pr->band) {
        off = {0, (long long)pr->p};
    } else {
        for (int o : pr->goff) off.push_back(o);
    }
}
bool prec_has_fp64(xt_prec pr) {
    for (const BandPrec *b : pr->groups)
        if (!band_has_fp64(b)) return false;
    return !pr->band || band_has_fp64(pr->band);
}

int prec_shifts(xt_prec pr, const double **shifts, bool *fp64) {
    if (shifts) *shifts = pr->shifts.empty() ? nullptr : pr->shifts.data();
    if (fp64) *fp64 = !pr->shifted.empty() && band_has_fp64(pr->shifted[0]);
    return (int)pr->shifts.size();
}

template <typename T>
int prec_apply_split(xt_prec pr, int R, int q, const T *minv, const PrecSplit *sp, const T *x,
                     T *y, hipStream_t s, const ActiveCols *ac) {
    const bool f32 = sizeof(T) == 4;
    if (!sp || sp->ns == 0 || !pr->band) return prec_apply_t<T>(pr, R, q, minv, x, y, f32, s, ac);
    const int pi = f32 ? 1 : 0, p = pr->p, ns = sp->ns, c = q * R;
    XT_TRY(pr->gin[pi].reserve(sizeof(T) * (size_t)p * ns));
    XT_TRY(pr->gout[pi].reserve(sizeof(T) * (size_t)p * ns));
    T *gi = pr->gin[pi].as<T>(), *go = pr->gout[pi].as<T>();
    const T *m2v = sp->m2v[pi].as<T>();
    const int nblk = ceil_div((long long)p * ns, 256);
    // the gather reads x before the K^-1 sweeps, which may write y over nothing it needs
    hipLaunchKernelGGL(split_gather_kernel<T>, dim3(nblk), dim3(256), 0, s, p, q, c, ns,
                       sp->dcase.as<int>(), sp->dbase.as<long long>(), sp->dstride.as<int>(), m2v,
                       x, gi);
    XT_HIP(hipGetLastError());
    XT_TRY(band_apply<T>(pr->band, R, q, minv, x, y, s, ac ? ac->Ra[0] : -1,
                         ac ? ac->dcols : nullptr));
    for (size_t g = 0; g + 1 < sp->goff.size(); ++g) {
        const int o = sp->goff[g], ng = sp->goff[g + 1] - o;
        XT_ARG(sp->gfac[g] >= 0 && sp->gfac[g] < (int)pr->shifted.size(), "split factor index");
        XT_TRY(band_apply<T>(pr->shifted[sp->gfac[g]], ng, 1, nullptr, gi + (size_t)o * p,
                             go + (size_t)o * p, s));
    }
    hipLaunchKernelGGL(split_scatter_kernel<T>, dim3(nblk), dim3(256), 0, s, p, q, c, ns,
                       sp->dcase.as<int>(), sp->dbase.as<long long>(), sp->dstride.as<int>(), m2v,
                       go, y);
    XT_HIP(hipGetLastError());
    return XT_OK;
}
template int prec_apply_split<double>(xt_prec, int, int, const double *, const PrecSplit *,
                                      const double *, double *, hipStream_t, const ActiveCols *);
template int prec_apply_split<float>(xt_prec, int, int, const float *, const PrecSplit *,
                                     const float *, float *, hipStream_t, const ActiveCols *);

template int prec_apply_t<double>(xt_prec, int, int, const double *, const double *, double *,
                                  bool, hipStream_t, const ActiveCols *);
template int prec_apply_t<float>(xt_prec, int, int, const float *, const float *, float *, bool,
                                 hipStream_t, const ActiveCols *);

// Staging of the allocation-free apply (xt_prec_apply_noalloc): one array per device,
// held until the process ends, shared by every call on that device.  Host code never
// passes the array's name to a kernel or a copy (on the host it is a stand-in, not a
// device address): it resolves the device address once per device with
// hipGetSymbolAddress and uses that.
static __device__ __align__(256) unsigned char scratch[XT_NOALLOC_SCRATCH_BYTES];
constexpr int kMaxDevices = 64;
static std::atomic<void *> g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device (resolved on the first call there).
static int scratch_ptr(void **out) {
    int dev = 0;
    XT_HIP(hipGetDevice(&dev));
    XT_ARG(dev >= 0 && dev < kMaxDevices, "device ordinal beyond the scratch table");
    void *ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        XT_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        XT_ARG(ptr != nullptr, "hipGetSymbolAddress returned no address for scratch");
        g_scratch_ptr[dev].store(ptr, std::memory_order_release);
    }
    *out = ptr;
    return XT_OK;
}

}  // namespace xt

extern "C" {

int xt_prec_create(int p, const double *alu, const int *jlu, const int *ju, xt_prec *out) {
    XT_ARG(out && p > 0 && alu && jlu && ju, "prec arguments");
    XT_HIP(hipFuncSetAttribute((const void *)trsv_onewg_kernel<double, true>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)kOneWgLds));
    XT_HIP(hipFuncSetAttribute((const void *)trsv_onewg_kernel<float, true>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)kOneWgLds));
    XT_HIP(hipFuncSetAttribute((const void *)trsv_sf_kernel<double>,
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)sf_lds_bytes<double>(kSfMaxRows)));
    XT_HIP(hipFuncSetAttribute((const void *)trsv_sf_kernel<float>,
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)sf_lds_bytes<float>(kSfMaxRows)));
    XT_ARG(jlu[0] == p + 2, "MSR factors must come from ilut (jlu(1) = n+2)");
    std::vector<int> lrp(p + 1, 0), urp(p + 1, 0), lci, uci;
    std::vector<double> lv, uv, dinv(p);
    for (int i = 0; i < p; ++i) {
        const int l0 = jlu[i] - 1, l1 = ju[i] - 1, u1 = jlu[i + 1] - 1;
        XT_ARG(l0 <= l1 && l1 <= u1, "inconsistent MSR row pointers");
        for (int k = l0; k < l1; ++k) {
            const int cidx = jlu[k] - 1;
            XT_ARG(cidx >= 0 && cidx < i, "L entry not strictly lower");
            lci.push_back(cidx);
            lv.push_back(alu[k]);
        }
        for (int k = l1; k < u1; ++k) {
            const int cidx = jlu[k] - 1;
            XT_ARG(cidx > i && cidx < p, "U entry not strictly upper");
            uci.push_back(cidx);
            uv.push_back(alu[k]);
        }
        lrp[i + 1] = (int)lci.size();
        urp[i + 1] = (int)uci.size();
        dinv[i] = alu[i];
    }
    xt_prec pr = new (std::nothrow) xt_prec_s;
    if (!pr) return XT_E_NOMEM;
    pr->p = p;
    int rc = upload_tri(p, lrp, lci, lv, true, pr->L);
    if (rc == XT_OK) rc = upload_tri(p, urp, uci, uv, false, pr->U);
    if (rc == XT_OK) rc = pr->dinv64.upload(dinv.data(), sizeof(double) * p);
    if (rc == XT_OK) {
        std::vector<float> d32(dinv.begin(), dinv.end());
        rc = pr->dinv32.upload(d32.data(), sizeof(float) * p);
        if (rc == XT_OK && hipDeviceSynchronize() != hipSuccess) rc = XT_E_HIP;
    }
    if (rc != XT_OK) { delete pr; return rc; }
    *out = pr;
    return XT_OK;
}

void xt_prec_destroy(xt_prec pr) { delete pr; }

int xt_prec_create_band(int p, const int *ia, const int *ja, const double *a, int block,
                        xt_prec *out) {
    XT_ARG(out && p > 0 && ia && ja && a, "prec_create_band arguments");
    xt_prec pr = new (std::nothrow) xt_prec_s;
    if (!pr) return XT_E_NOMEM;
    pr->p = p;
    int rc = band_build(p, ia, ja, a, block, &pr->band);
    if (rc != XT_OK) { delete pr; return rc; }
    *out = pr;
    return XT_OK;
}

int xt_prec_create_band_shifted(int p, const int *kia, const int *kja, const double *ka,
                                const int *mia, const int *mja, const double *ma, int nshift,
                                const double *shifts, int block, int flags, xt_prec *out) {
    XT_ARG(out && p > 0 && kia && kja && ka && nshift >= 0 && (nshift == 0 || (shifts && mia &&
           mja && ma)), "prec_create_band_shifted arguments");
    XT_ARG(kia[0] == 1 && (nshift == 0 || mia[0] == 1), "CSR must be 1-based");
    for (int g = 0; g < nshift; ++g) XT_ARG(shifts[g] > 0.0, "shifts must be positive");
    xt_prec pr = new (std::nothrow) xt_prec_s;
    if (!pr) return XT_E_NOMEM;
    pr->p = p;
    int rc = band_build(p, kia, kja, ka, block, &pr->band, !(flags & XT_BAND_FP32_ONLY));
    int b = 0;
    if (rc == XT_OK) band_dims(pr->band, &b, nullptr, nullptr);
    // K + s M row by row (both rows sorted by column: merged; K's pattern holds M's for a
    // mesh whose mass couples only DOFs that the stiffness couples, but any union works)
    auto sorted = [p](const int *ia_, const int *ja_) {
        for (int i = 0; i < p; ++i)
            for (int k = ia_[i]; k + 1 < ia_[i + 1]; ++k)
                if (ja_[k] <= ja_[k - 1]) return false;
        return true;
    };
    if (rc == XT_OK && nshift > 0 && (!sorted(kia, kja) || !sorted(mia, mja))) {
        set_error("prec_create_band_shifted: CSR rows must be sorted by column");
        rc = XT_E_ARG;
    }
    std::vector<int> ia(p + 1, 1), ja;
    std::vector<double> a;
    for (int g = 0; g < nshift && rc == XT_OK; ++g) {
        ja.clear();
        a.clear();
        for (int i = 0; i < p; ++i) {
            int k = kia[i] - 1, ke = kia[i + 1] - 1, m = mia[i] - 1, me = mia[i + 1] - 1;
            while (k < ke || m < me) {
                const int jk = k < ke ? kja[k] : 1 << 30, jm = m < me ? mja[m] : 1 << 30;
                if (jk == jm) { ja.push_back(jk); a.push_back(ka[k++] + shifts[g] * ma[m++]); }
                else if (jk < jm) { ja.push_back(jk); a.push_back(ka[k++]); }
                else { ja.push_back(jm); a.push_back(shifts[g] * ma[m++]); }
            }
            ia[i + 1] = (int)ja.size() + 1;
        }
        BandPrec *bp = nullptr;
        if (rc == XT_OK)
            rc = band_build(p, ia.data(), ja.data(), a.data(), b, &bp,
                            !(flags & XT_SHIFT_FP32_ONLY));
        if (rc == XT_OK) {
            pr->shifted.push_back(bp);
            pr->shifts.push_back(shifts[g]);
        }
    }
    if (rc != XT_OK) { delete pr; return rc; }
    *out = pr;
    return XT_OK;
}

// Runs of consecutive systems for xt_prec_create_band_seg: minimise over the partitions
// of the systems into runs  sum_runs (dofs of the run x its block size) + kRunCost,
// the factor entries an apply streams plus a launch cost per run in the same units
// (about 8 us of sweeps at the HBM rate, FP32: 8e-6 s x 5e12 B/s / 16 B per entry),
// with runs of several systems capped in size.
static void band_runs(const std::vector<long long> &n, const std::vector<int> &b,
                      std::vector<int> &cut) {
    constexpr double kRunCost = 2.5e6;
    // a run of several systems holds at most this many factor entries per block set (the
    // FP64 factorisation of a run needs about six such sets at once)
    constexpr double kRunMaxEntries = 1.0e9;
    const int S = (int)n.size();
    std::vector<double> best(S + 1, 0.0);
    std::vector<int> from(S + 1, 0);
    for (int j = 1; j <= S; ++j) {
        best[j] = 1e300;
        long long dofs = 0;
        int bmax = 0;
        for (int i = j - 1; i >= 0; --i) {   // run i..j-1
            dofs += n[i];
            bmax = std::max(bmax, b[i]);
            if (i < j - 1 && (double)dofs * bmax > kRunMaxEntries) break;
            const double c = best[i] + (double)dofs * bmax + kRunCost;
            if (c < best[j]) {
                best[j] = c;
                from[j] = i;
            }
        }
    }
    cut.clear();
    for (int j = S; j > 0; j = from[j]) cut.push_back(j);
    cut.push_back(0);
    std::reverse(cut.begin(), cut.end());
}

int xt_prec_create_band_seg(int p, const int *ia, const int *ja, const double *a, int nseg,
                            const int *seg_dof, int block, int flags, xt_prec *out) {
    XT_ARG(out && p > 0 && ia && ja && a && nseg > 0 && seg_dof && block >= 0,
           "prec_create_band_seg arguments");
    XT_ARG(ia[0] == 1, "CSR must be 1-based");
    XT_ARG(seg_dof[0] == 0 && seg_dof[nseg] == p, "seg_dof must run from 0 to p");
    for (int t = 0; t < nseg; ++t) XT_ARG(seg_dof[t + 1] > seg_dof[t], "empty or unordered segment");
    std::vector<long long> n(nseg);
    std::vector<int> b(nseg);
    for (int t = 0; t < nseg; ++t) {
        const int lo = seg_dof[t], hi = seg_dof[t + 1];
        int bw = 0;
        for (int i = lo; i < hi; ++i) {
            XT_ARG(ia[i + 1] >= ia[i] && ia[i + 1] <= ia[p], "CSR row pointers must not decrease");
            for (int k = ia[i] - 1; k < ia[i + 1] - 1; ++k) {
                const int j = ja[k] - 1;
                if (j < lo || j >= hi) {
                    set_error("prec_create_band_seg: row %d (segment %d) couples column %d "
                              "outside its segment", i + 1, t, j + 1);
                    return XT_E_ARG;
                }
                if (j <= i) bw = std::max(bw, i - j);
            }
        }
        n[t] = hi - lo;
        b[t] = (std::max(std::max(block, bw), 64) + 63) / 64 * 64;
    }
    std::vector<int> cut;
    band_runs(n, b, cut);
    xt_prec pr = new (std::nothrow) xt_prec_s;
    if (!pr) return XT_E_NOMEM;
    pr->p = p;
    int rc = XT_OK;
    std::vector<int> sia, sja;
    std::vector<double> sa;
    for (size_t g = 0; g + 1 < cut.size() && rc == XT_OK; ++g) {
        const int lo = seg_dof[cut[g]], hi = seg_dof[cut[g + 1]], pg = hi - lo;
        int bg = 0;
        for (int t = cut[g]; t < cut[g + 1]; ++t) bg = std::max(bg, b[t]);
        // the run's rows, columns shifted to the run (1-based)
        const long long k0 = ia[lo] - 1, k1 = ia[hi] - 1;
        sia.resize(pg + 1);
        for (int i = 0; i <= pg; ++i) sia[i] = (int)(ia[lo + i] - k0);
        sja.resize(k1 - k0);
        for (long long k = k0; k < k1; ++k) sja[k - k0] = ja[k] - lo;
        sa.assign(a + k0, a + k1);
        BandPrec *bp = nullptr;
        rc = band_build(pg, sia.data(), sja.data(), sa.data(), bg, &bp,
                        !(flags & XT_BAND_FP32_ONLY));
        if (rc == XT_OK) {
            pr->groups.push_back(bp);
            pr->goff.push_back(lo);
        }
    }
    if (rc != XT_OK) { delete pr; return rc; }
    pr->goff.push_back(p);
    *out = pr;
    return XT_OK;
}

int xt_prec_band_groups(xt_prec pr, int *ngroup, int *goff, int *gblock) {
    XT_ARG(pr && ngroup, "prec_band_groups arguments");
    if (!pr->groups.empty()) {
        *ngroup = (int)pr->groups.size();
        for (size_t g = 0; g < pr->groups.size(); ++g) {
            if (goff) goff[g] = pr->goff[g];
            if (gblock) band_dims(pr->groups[g], &gblock[g], nullptr, nullptr);
        }
        if (goff) goff[pr->groups.size()] = pr->p;
        return XT_OK;
    }
    *ngroup = pr->band ? 1 : 0;
    if (pr->band) {
        if (goff) { goff[0] = 0; goff[1] = pr->p; }
        if (gblock) band_dims(pr->band, &gblock[0], nullptr, nullptr);
    }
    return XT_OK;
}

int xt_prec_band_bytes(xt_prec pr, int fp32, long long *bytes) {
    XT_ARG(pr && bytes, "prec_band_bytes arguments");
    *bytes = pr->band ? band_bytes(pr->band, fp32 != 0) : 0;
    for (const BandPrec *g : pr->groups) *bytes += band_bytes(g, fp32 != 0);
    return XT_OK;
}

int xt_prec_shifts(xt_prec pr, int *nshift, double *shifts) {
    XT_ARG(pr, "prec");
    if (nshift) *nshift = (int)pr->shifts.size();
    if (shifts) std::copy(pr->shifts.begin(), pr->shifts.end(), shifts);
    return XT_OK;
}

int xt_prec_refactor_band(xt_prec pr, const int *ia, const int *ja, const double *a,
                          void *stream) {
    XT_ARG(pr && (pr->band || !pr->groups.empty()) && ia && ja && a,
           "prec_refactor_band arguments");
    if (!pr->groups.empty()) {
        set_error("xt_prec_refactor_band: a grouped factor is rebuilt with "
                  "xt_prec_create_band_seg");
        return XT_E_UNSUPPORTED;
    }
    if (!pr->shifted.empty()) {
        set_error("xt_prec_refactor_band: a preconditioner with shifted factors is rebuilt with "
                  "xt_prec_create_band_shifted");
        return XT_E_UNSUPPORTED;
    }
    return band_refactor(pr->band, ia, ja, a, (hipStream_t)stream);
}

int xt_prec_refresh_band(xt_prec pr, const int *ia, const int *ja, const double *a,
                         int first_row, void *stream) {
    XT_ARG(pr && pr->band && pr->groups.empty() && pr->shifted.empty() && ia && ja && a,
           "prec_refresh_band arguments (a plain banded factor)");
    XT_ARG(first_row >= 0 && first_row < pr->p, "prec_refresh_band: first_row out of range");
    return band_refactor(pr->band, ia, ja, a, (hipStream_t)stream, first_row);
}

int xt_prec_band_info(xt_prec pr, int *block, int *nblocks, int *bandwidth) {
    XT_ARG(pr && (pr->band || !pr->groups.empty()), "not a banded-factor preconditioner");
    if (pr->band) {
        band_dims(pr->band, block, nblocks, bandwidth);
        return XT_OK;
    }
    int bmax = 0, nbs = 0, bwmax = 0;
    for (const BandPrec *g : pr->groups) {
        int b = 0, nb = 0, bw = 0;
        band_dims(g, &b, &nb, &bw);
        bmax = std::max(bmax, b);
        nbs += nb;
        bwmax = std::max(bwmax, bw);
    }
    if (block) *block = bmax;
    if (nblocks) *nblocks = nbs;
    if (bandwidth) *bandwidth = bwmax;
    return XT_OK;
}

int xt_prec_levels(xt_prec pr, int *nlev_lower, int *nlev_upper) {
    XT_ARG(pr, "prec");
    if (pr->band || !pr->groups.empty()) {   // sequential block steps of each sweep
        int nb = 0;
        if (pr->band) band_dims(pr->band, nullptr, &nb, nullptr);
        for (size_t g = 0; g < pr->groups.size(); ++g) {   // the runs follow one another
            int nbg = 0;
            band_dims(pr->groups[g], nullptr, &nbg, nullptr);
            nb += nbg;
        }
        if (nlev_lower) *nlev_lower = nb;
        if (nlev_upper) *nlev_upper = nb;
        return XT_OK;
    }
    if (nlev_lower) *nlev_lower = (int)pr->L.lev_ptr.size() - 1;
    if (nlev_upper) *nlev_upper = (int)pr->U.lev_ptr.size() - 1;
    return XT_OK;
}

int xt_prec_apply(xt_prec pr, int R, int q, const void *minv, const void *x, void *y, int fp32,
                  void *stream) {
    XT_ARG(pr && R > 0 && q > 0 && x && y && x != y, "prec_apply arguments");
    hipStream_t s = (hipStream_t)stream;
    if (fp32)
        return prec_apply_t<float>(pr, R, q, (const float *)minv, (const float *)x, (float *)y,
                                   true, s);
    return prec_apply_t<double>(pr, R, q, (const double *)minv, (const double *)x, (double *)y,
                                false, s);
}

int xt_prec_apply_noalloc(xt_prec pr, int R, int q, const void *minv, const void *x, void *y,
                          int fp32, void *stream) {
    XT_ARG(pr && R > 0 && q > 0 && x && y && x != y, "prec_apply_noalloc arguments");
    if (pr->band || !pr->groups.empty()) {
        set_error("xt_prec_apply_noalloc: ILUT factors only (the banded factor keeps its own "
                  "workspace)");
        return XT_E_UNSUPPORTED;
    }
    const size_t need = (size_t)pr->p * q * R * (fp32 ? sizeof(float) : sizeof(double));
    if (minv && need > XT_NOALLOC_SCRATCH_BYTES) {
        set_error("xt_prec_apply_noalloc: p*q*R = %lld values need %zu bytes of staging, more "
                  "than the %zu-byte scratch; use xt_prec_apply",
                  (long long)pr->p * q * R, need, (size_t)XT_NOALLOC_SCRATCH_BYTES);
        return XT_E_ARG;
    }
    void *stage = nullptr;
    if (minv) XT_TRY(scratch_ptr(&stage));
    hipStream_t s = (hipStream_t)stream;
    if (fp32)
        return ilut_apply<float>(pr, R, q, (const float *)minv, (const float *)x, (float *)y,
                                 true, (float *)stage, false, s);
    return ilut_apply<double>(pr, R, q, (const double *)minv, (const double *)x, (double *)y,
                              false, (double *)stage, false, s);
}

}  // extern "C"
