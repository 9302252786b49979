// Exact factor preconditioner K^-1 for banded SPD K, applied as block sweeps.
//
// The reference's live solver preconditions GMRES with the exact factor of K (MUMPS
// LDL^T of the lower triangle, mumps.f90:22-145, applied to all q temporal blocks by
// mpilusol, kronecker_mumps.f90:120-183).  ILUT with lfil >= n and droptol = 0 is the
// same exact factor (ilut.f:2169-2170).  Here K (half-bandwidth w after the mesh
// numbering) is cut into nb diagonal blocks of b >= w rows, so it is block tridiagonal,
// and eliminated from both ends towards a middle block ("twisted" block Cholesky, FP64,
// device): the first nt blocks top down, the last nbt blocks bottom up, the middle block
// last.  The two eliminations are independent of each other, so every dependent step of
// the factorization and of the sweeps works on two blocks at once and there are half as
// many of them, with the operations of the one-sided factor.
//
// The bottom blocks are held with their rows reversed (row r of the factor's order is row
// nb b - 1 - r of K from the last row back), which makes the bottom chain the same
// computation as the top one: block i of a chain with its sub-diagonal block
// E_i = K_{i+1,i} L_ii^-T, D_i = L_ii^-1 and
//
//   forward   y_0 = D_0 x_0,   y_{i+1} = D_{i+1} x_{i+1} - G_i y_i,   G_i = D_{i+1} E_i
//   middle    y_m = D_m x_m - G_top y_top - G_bot y_bot,   z_m = D_m^T y_m
//   backward  z_i = D_i^T y_i - H_i z_{i+1},   H_i = (E_i D_i)^T
//
// E_i couples only the last w columns of block i with the first w rows of block i + 1, so
// G_i has w nonzero columns (the last) and H_i too (the first): both are stored b x kw,
// kw = w rounded up.  The D x and D^T y products of all blocks run in one batched launch.
// A recurrence w_v -= M_v w_{v-1} (v = 1..m) advances 2^L blocks per dependent step:
// pairing two steps,
//   w_v -= M_v w_{v-1}  for even v            (one batched launch: the new right-hand sides)
//   w_v -= M'_v w_{v-2} for v = 2, 4, .. in order,   M'_v = -M_v M_{v-1}
//   w_v -= M_v w_{v-1}  for odd v             (one batched launch: the blocks between)
// and the middle line is again such a recurrence over every second block, paired in
// turn for L levels.  The level matrices are formed once per factorization.  Where the
// blocks are at least twice the band (rc < b below), the chain runs on the kw rows the
// next block reads only, and one batched launch finishes the other rows.
// All matrix sets are stored row-major (the row of the operator a tile needs is
// contiguous) in FP64 and FP32.
//
// The factorization runs on the device once per K, and again at every refactorization
// (xt_prec_refactor_band: per slab when K follows the temperature; from the first
// changed block on after an element deletion): this file's panel kernels for the block
// Cholesky and the inverses D_i, rocBLAS gemm for G_i, H_i and the level matrices
// (b^3 products near the FP64 matrix-core peak).  None of it is on the per-iteration path.
#include <rocblas/rocblas.h>

#include <algorithm>
#include <cstring>
#include <new>
#include <type_traits>

#include "xt_common.h"

namespace xt {

// The sweeps of one apply are a fixed sequence of launches on fixed buffers for a given
// column count and precision: captured once into a HIP graph and replayed, they skip the
// per-launch host overhead.  Keyed on every pointer the launches use and on the factor's
// layout (a refactorization of a wider band changes kw and rc, and an array that was freed
// for it can come back at its old address), so a refactorization or a grown workspace
// captures anew.
constexpr int kLevels = 4;     // pairing levels of the block recurrences, at most
constexpr int kMinChain = 3;   // a level is added while its chain keeps this many steps
constexpr int kKey = 6 + 2 * kLevels;
struct SweepGraph {
    int c = 0, pi = -1, nl = 0;                          // columns, precision, levels used,
    int kw = 0, rc = 0;                                  // the factor's layout,
    long long epoch = -1;                                // knob epoch
    const void *key[kKey] = {};
    hipGraphExec_t exec = nullptr;
};

#define XT_RB(...)                                                                      \
    do {                                                                                \
        rocblas_status st_ = (__VA_ARGS__);                                             \
        if (st_ != rocblas_status_success) {                                            \
            ::xt::set_error("%s:%d %s -> rocblas status %d", __FILE__, __LINE__,        \
                            #__VA_ARGS__, (int)st_);                                    \
            return XT_E_HIP;                                                            \
        }                                                                               \
    } while (0)

struct RbHandle {
    rocblas_handle h = nullptr;
    ~RbHandle() { if (h) rocblas_destroy_handle(h); }
};

constexpr size_t kKeepScratch = 8ull << 30;

struct BandPrec {
    int p = 0, b = 0, nb = 0, bw = 0;
    int nt = 0, nbt = 0;         // blocks of the top and of the bottom chain (+ the middle)
    int kw = 0, rc = 0;          // columns of G and H; rows the chains run on (kw or b)
    // [.][0] FP64, [.][1] FP32.  Blocks in the factor's order (top chain, middle, bottom
    // chain).  Dl: D_i row-major (lower), Du: D_i^T row-major (upper).  G, H: the
    // top chain's nt, then the bottom chain's nbt.  Lv[dir][L - 1]: the level-L matrices
    // (rc x kw) of the forward (0) and backward (1) recurrence, the top chain's
    // steps(0, dir) >> L, then the bottom chain's (order: level_view).
    DevBuf Dl[2], Du[2], G[2], H[2];
    DevBuf Lv[2][kLevels][2];
    int nlev = 0;
    bool keep64 = true;          // false: the FP64 sets are released after the FP32 copies
    DevBuf w1, w2;
    // scratch of the factorization, kept from the first refactorization on while it is at
    // most kKeepScratch bytes (a refactorization per slab would spend 5 ms of 30 on its
    // allocations and frees), and the rocBLAS handle with it
    DevBuf sL, sE, sW, sK, sinfo;
    bool built = false;
    RbHandle *rb = nullptr;
    SweepGraph graph[4];
    int next_graph = 0;
    hipStream_t cap = nullptr;   // capture stream (non-blocking, default priority)
    BandPrec() = default;
    BandPrec(const BandPrec &) = delete;
    BandPrec &operator=(const BandPrec &) = delete;
    ~BandPrec() {
        for (SweepGraph &g : graph)
            if (g.exec) (void)hipGraphExecDestroy(g.exec);
        if (cap) (void)hipStreamDestroy(cap);
        delete rb;
    }
    int blocks(int side) const { return side == 0 ? nt : nbt; }
    // steps of a chain's recurrence: forward over its blocks, backward from the middle
    int steps(int side, int dir) const {
        const int n = blocks(side);
        return dir == 0 ? std::max(0, n - 1) : n;
    }
};

// ---------------------------------------------------------------------------
// Block products of the sweeps, batched over items z:
//   O_z = A_z V_z   or   O_z -= A_z V_z
// A_z: rows x kdim row-major (row stride lda); V_z, O_z: row-major with ld columns (a
// multiple of 16; the columns past the vectors' own are never read back).  Items z < n0 are the
// first chain's, A_z = A[0] + z as[0] and so on, the others the second chain's.
// tri = 1: A lower triangular (k <= r), tri = 2: upper (k >= r); the stored zeros of
// the other triangle are skipped where a whole tile lies there.
// ---------------------------------------------------------------------------
template <typename T>
struct Items {
    const T *A[2], *V[2];
    T *O[2];
    long long as[2], vs[2], os[2];
    int n0, n;
    // rows dup0.. of item dupz are also written to dup (NULL: none)
    T *dup = nullptr;
    int dupz = 0, dup0 = 0;
};

typedef float xt_f4m __attribute__((ext_vector_type(4)));
typedef double xt_d4m __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
    typedef xt_f4m acc_t;
    __device__ static acc_t step(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static int row(int g, int i) { return 4 * g + i; }
};
template <>
struct Mfma<double> {
    typedef xt_d4m acc_t;
    __device__ static acc_t step(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static int row(int g, int i) { return g + 4 * i; }
};

// Tile t = (w % 8) (grid / 8) + w / 8 of workgroup w: workgroups are dealt to the 8 XCDs
// round-robin, so each XCD gets a contiguous run of tiles (the grid is a multiple of 8).
__device__ __forceinline__ long long xcd_tile() {
    return (long long)(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
}

// Dependent steps and few-column passes: a workgroup computes a (16 RT) x (16 CT) output
// tile; its KW waves split the k range (whole chunks of 16) and their partial tiles are
// summed through LDS in a fixed order (deterministic, one launch, no partials in
// memory).  Each wave reads its operands straight from global memory into registers, PF
// chunks ahead of the products and with no barrier in the loop: one FP64 matrix-core
// step takes 64 cycles a SIMD, so RT CT of them cover the loads of a chunk; what bounds
// a step is the latency of the first loads and of the launch.
// Lane l = 16 g + t holds A[row t][4 g + s] and V[4 g + s][column t] in step s of a chunk
// (any assignment of k to lane groups gives the same sum): A rows are read 32 or 16
// bytes a lane, 128 contiguous bytes a row; column tiles go in pairs, lane t taking
// columns 2 t and 2 t + 1 of the 32.  Output layout of the 4 accumulators per lane: f32
// row 4 g + i, f64 row g + 4 i.
// FP32 with up to 16 columns (NA = 4): a sum of its own for each step of a chunk, and the waves'
// partial tiles added to one another and to the old value in FP64.  One FP32 chain a wave and
// FP32 sums of the waves had 1.2 times the error of a sum over 256 threads and a tree (the
// largest of y, mean of 72 factors, 6 columns; thermal ones 1.3 to 1.9); so it is 0.92, for 2
// of 105 us an apply (768-row thermal blocks).  All sums in FP64 from the waves on: 0.80, 4 us.
// nseg = 2: one item whose product is A[0] V[0] + A[1] V[1], half the waves each.
// Consecutive tiles are the column tiles of one row tile, so one XCD's L2 serves its A.
template <typename T, int RT, int CT, int KW, int PF, int NA>
__global__ void __launch_bounds__(64 * KW)
band_prod_kernel(Items<T> it, int rows, int lda, int kdim, int tri, int ld, int sub, int nseg) {
    using M = Mfma<T>;
    using acc_t = typename M::acc_t;
    constexpr int AV = 16 / sizeof(T);              // elements of a 16-byte load
    typedef T avec __attribute__((ext_vector_type(AV)));
    typedef T vpair __attribute__((ext_vector_type(2)));
    constexpr int CP = CT / 2;                      // column-tile pairs
    typedef std::conditional_t<NA == 4, double, T> sum_t;   // what the waves' sums are added in
    __shared__ T red[KW][RT * CT][4][64];
    const int ntx = rows / (16 * RT), nty = ld / (16 * CT);
    const long long tile = xcd_tile();
    if (tile >= (long long)ntx * nty * it.n) return;
    const int z = (int)(tile / (ntx * nty)), rem = (int)(tile - (long long)z * ntx * nty);
    const int r0 = rem / nty * (16 * RT), n0 = rem % nty * (16 * CT);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, t = lane & 15;
    const int sd = z < it.n0 ? 0 : 1, zi = sd ? z - it.n0 : z;
    const int parts = KW / nseg, part = wave % parts, sg = nseg == 2 ? wave / parts : sd;
    const T *A = it.A[sg] + (nseg == 2 ? 0 : zi * it.as[sg]);
    const T *V = it.V[sg] + (nseg == 2 ? 0 : zi * it.vs[sg]);
    T *O = it.O[sd] + zi * it.os[sd];
    int k0 = 0, k1 = kdim;
    if (tri == 1) k1 = r0 + 16 * RT;
    if (tri == 2) k0 = r0;
    const int nch = (k1 - k0) >> 4;                 // chunks; this wave's: c0 .. c0 + n - 1
    const int c0 = nch * part / parts, n = nch * (part + 1) / parts - c0;
    const T *ap = A + (size_t)(r0 + t) * lda + k0 + 16 * c0 + 4 * g;
    const T *vp = V + (size_t)(k0 + 16 * c0 + 4 * g) * ld + n0 + (CP ? 2 * t : t);
    const T *vq = V + (size_t)(k0 + 16 * c0 + 4 * g) * ld + n0 + 32 * CP + t;   // odd last tile
    // output unit u (accumulator e of 16 x 16 tile tl): summed and stored by wave u % KW,
    // whose old values are loaded ahead of the products
    constexpr int NU = RT * CT * 4, UW = (NU + KW - 1) / KW;
    auto out_at = [&](int u) {
        const int tl = u >> 2, e = u & 3, i = tl / CT, c = tl - i * CT;
        const int col = n0 + (c < 2 * CP ? 32 * (c >> 1) + 2 * t + (c & 1) : 16 * c + t);
        return O + (size_t)(r0 + 16 * i + M::row(g, e)) * ld + col;
    };
    T old[UW];
#pragma unroll
    for (int h = 0; h < UW; ++h) {
        old[h] = T(0);
        const int u = wave + h * KW;
        if (sub && u < NU) old[h] = *out_at(u);
    }
    acc_t acc[RT][CT][NA];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int s = 0; s < NA; ++s) acc[i][j][s] = acc_t{T(0), T(0), T(0), T(0)};
    T a[PF][RT][4], v[PF][CT][4];
    auto load = [&](int j, int ch) {
        const size_t ko = (size_t)16 * ch;
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int h = 0; h < 4 / AV; ++h) {
                const avec w = *reinterpret_cast<const avec *>(ap + (size_t)16 * i * lda + ko + AV * h);
#pragma unroll
                for (int e = 0; e < AV; ++e) a[j][i][AV * h + e] = w[e];
            }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int cp = 0; cp < CP; ++cp) {
                const vpair w = *reinterpret_cast<const vpair *>(vp + (ko + s) * ld + 32 * cp);
                v[j][2 * cp][s] = w[0];
                v[j][2 * cp + 1][s] = w[1];
            }
            if (CT & 1) v[j][CT - 1][s] = vq[(ko + s) * ld];
        }
    };
    auto mul = [&](int j) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int c = 0; c < CT; ++c)
                    acc[i][c][s % NA] = M::step(a[j][i][s], v[j][c][s], acc[i][c][s % NA]);
    };
    if (n > 0) {
#pragma unroll
        for (int j = 0; j < PF; ++j) load(j, min(j, n - 1));
        int i = 0;
        for (; i + 2 * PF <= n; i += PF) {
#pragma unroll
            for (int j = 0; j < PF; ++j) {
                mul(j);
                load(j, i + PF + j);
            }
        }
        if (n - i > PF) {
#pragma unroll
            for (int j = 0; j < PF; ++j) {
                mul(j);
                load(j, min(i + PF + j, n - 1));
            }
            i += PF;
        }
#pragma unroll
        for (int j = 0; j < PF; ++j)
            if (i + j < n) mul(j);
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                T sum[NA];
#pragma unroll
                for (int s = 0; s < NA; ++s) sum[s] = acc[i][c][s][e];
#pragma unroll
                for (int d = NA / 2; d > 0; d /= 2)
#pragma unroll
                    for (int s = 0; s < d; ++s) sum[s] += sum[s + d];
                red[wave][i * CT + c][e][lane] = sum[0];
            }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < UW; ++h) {
        const int u = wave + h * KW;
        if (u >= NU) break;
        sum_t sum = red[0][u >> 2][u & 3][lane];
#pragma unroll
        for (int w = 1; w < KW; ++w) sum += red[w][u >> 2][u & 3][lane];
        T *o = out_at(u);
        *o = (T)(sub ? old[h] - sum : sum);
        if (it.dup && z == it.dupz) {
            const long long at = o - (O + (size_t)it.dup0 * ld);
            if (at >= 0) it.dup[at] = (T)sum;
        }
    }
}

// Batched products of many blocks with more than 16 columns (the block-diagonal passes and
// the pairing levels' passes, where parallelism is plentiful and L2 bandwidth is the
// limit of the tile kernel above): a workgroup computes a TM x 64 output tile of one
// block.  TM = 64: each of its 4 waves a 32 x 32 quadrant as 2 x 2 matrix-core tiles;
// TM = 128 (large batches): each wave a 32 x 64 strip as 2 x 4 tiles, fewer operand reads
// per product.  k advances in chunks of 16 staged through LDS, double-buffered (the next
// chunk's global loads are in flight while the current chunk is multiplied), so every
// operand element fetched feeds TM or 64 outputs instead of 16.  In MFMA step s of a
// chunk, lane group g takes k = 4 g + s for both operands.  Columns past ld read a
// clamped column and are not stored.  The XCD mapping gives one L2 all tiles of a block
// (the A row tiles and V column tiles each tile shares with its neighbours).
template <typename T, int TM>
__global__ void __launch_bounds__(256)
band_tile_kernel(Items<T> it, int rows, int lda, int kdim, int tri, int ld, int sub) {
    using M = Mfma<T>;
    constexpr int KC = 16, AP = KC + 4, VP = 64 + 4;
    constexpr int AV = TM / 64;                    // A vec4 loads per thread per chunk
    constexpr int RT = 2, CT = TM == 64 ? 2 : 4;   // MFMA tiles per wave (rows, columns)
    typedef T vec4_t __attribute__((ext_vector_type(4)));
    __shared__ T As[2][TM][AP];
    __shared__ T Vs[2][KC][VP];
    const int ntx = rows / TM;
    const long long per_blk = (long long)ntx * ((ld + 63) / 64);
    const long long tile = xcd_tile();
    if (tile >= per_blk * it.n) return;
    const int z = (int)(tile / per_blk);
    const int rem = (int)(tile - z * per_blk);
    const int R0 = (rem % ntx) * TM, N0 = (rem / ntx) * 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, t = lane & 15;
    const int sd = z < it.n0 ? 0 : 1, zi = sd ? z - it.n0 : z;
    const T *A = it.A[sd] + zi * it.as[sd];
    const T *V = it.V[sd] + zi * it.vs[sd];
    T *O = it.O[sd] + zi * it.os[sd];
    int k0 = 0, k1 = kdim;
    if (tri == 1) k1 = R0 + TM;
    if (tri == 2) k0 = R0;
    const int ar = tid >> 2, ac = (tid & 3) * 4;   // A chunk: rows ar + 64 u, k ac..ac+3
    const int vr = tid >> 4, vc = (tid & 15) * 4;  // V chunk: k row vr, columns vc..vc+3
    const T *ap = A + (size_t)(R0 + ar) * lda + ac;  // 4-element aligned: lda % 16 == 0
    const T *vp = V + (size_t)vr * ld + min(N0 + vc, ld - 4);
    const int wr = TM == 64 ? (wave >> 1) * 32 : wave * 32;
    const int wc = TM == 64 ? (wave & 1) * 32 : 0;
    typename M::acc_t acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = typename M::acc_t{T(0), T(0), T(0), T(0)};
    vec4_t ga[AV];
#pragma unroll
    for (int u = 0; u < AV; ++u)
        ga[u] = *reinterpret_cast<const vec4_t *>(ap + (size_t)64 * u * lda + k0);
    vec4_t gv = *reinterpret_cast<const vec4_t *>(vp + (size_t)k0 * ld);
    int buf = 0;
    for (int kc = k0; kc < k1; kc += KC) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int u = 0; u < AV; ++u) As[buf][ar + 64 * u][ac + e] = ga[u][e];
            Vs[buf][vr][vc + e] = gv[e];
        }
        __syncthreads();
        if (kc + KC < k1) {
#pragma unroll
            for (int u = 0; u < AV; ++u)
                ga[u] = *reinterpret_cast<const vec4_t *>(ap + (size_t)64 * u * lda + kc + KC);
            gv = *reinterpret_cast<const vec4_t *>(vp + (size_t)(kc + KC) * ld);
        }
        T a[RT][4], bv[CT][4];
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2) {
#pragma unroll
            for (int i = 0; i < RT; ++i) a[i][s2] = As[buf][wr + 16 * i + t][4 * g + s2];
#pragma unroll
            for (int j = 0; j < CT; ++j) bv[j][s2] = Vs[buf][4 * g + s2][wc + 16 * j + t];
        }
#pragma unroll
        for (int s2 = 0; s2 < 4; ++s2)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j) acc[i][j] = M::step(a[i][s2], bv[j][s2], acc[i][j]);
        buf ^= 1;
    }
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        const int col = N0 + wc + 16 * j + t;
        if (col >= ld) continue;
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                T *o = O + (size_t)(R0 + wr + 16 * i + M::row(g, e)) * ld + col;
                *o = sub ? *o - acc[i][j][e] : acc[i][j][e];
                if (it.dup && z == it.dupz) {
                    const long long at = o - (O + (size_t)it.dup0 * ld);
                    if (at >= 0) it.dup[at] = acc[i][j][e];
                }
            }
    }
}

// Profile kind of the sweeps in precision T.
template <typename T>
constexpr int band_kind() { return sizeof(T) == 8 ? XT_PROF_BAND64 : XT_PROF_BAND; }

// Columns of the workspace for c columns: a multiple of 16 up to 16, else the least
// multiple of 32 or of 48 (two or three 16-column tiles a workgroup).
static int pad_cols(int c) {
    if (c <= 16) return 16;
    return std::min((c + 31) / 32 * 32, (c + 47) / 48 * 48);
}

// Workgroups from which a pass with more than 16 columns takes the LDS-staged tiles.
constexpr long long kBatchedTiles = 1536;

template <typename T>
static int launch_prod(const Items<T> &it, int rows, int lda, int kdim, int tri, int c, int ld,
                       bool sub, int nseg, hipStream_t s) {
    if (it.n <= 0 || rows <= 0) return XT_OK;
    const bool prof = prof_on(band_kind<T>());
    if (prof) prof_begin(band_kind<T>(), s);
    auto grid = [&](int tr, int tc) {
        return dim3((unsigned)(ceil_div((long long)(rows / tr) * ceil_div(ld, tc) * it.n, 8) * 8));
    };
    constexpr int few = sizeof(T) == 4 ? 4 : 1;   // sums a tile with up to 16 columns
#define XT_PROD(RT, CT, KW, PF, NA)                                                          \
    hipLaunchKernelGGL((band_prod_kernel<T, RT, CT, KW, PF, NA>), grid(16 * RT, 16 * CT),     \
                       dim3(64 * KW), 0, s, it, rows, lda, kdim, tri, ld, (int)sub, nseg)
    if (ld == 16) {
        // few columns: the matrix is streamed once; two row tiles share V's loads where
        // that leaves enough workgroups (4.3 TB/s in the passes over 92 768-row blocks)
        const int sk = tune_knob(XT_TUNE_BAND_SMALLC);
        const bool rt2 = sk == 2 || (sk != 1 && (long long)rows / 32 * it.n >= 512);
        if (rt2 && rows % 32 == 0) XT_PROD(2, 1, 4, 4, few);
        else if (tune_knob(XT_TUNE_BAND_CHAIN_FEW) == 2) XT_PROD(1, 1, 4, 4, few);
        else XT_PROD(1, 1, 8, 2, few);
    } else if (const long long tiles = (long long)(rows / 64) * ceil_div(ld, 64) * it.n;
               rows % 64 == 0 && nseg == 1 && tiles >= kBatchedTiles) {
        const int tk = tune_knob(XT_TUNE_BAND_TILE);
        const bool can128 = sizeof(T) == 4 && rows % 128 == 0;
        if (can128 && (tk == 128 || (tk == 0 && it.n >= 23)))
            hipLaunchKernelGGL((band_tile_kernel<T, 128>), grid(128, 64), dim3(256), 0, s, it, rows,
                               lda, kdim, tri, ld, (int)sub);
        else
            hipLaunchKernelGGL((band_tile_kernel<T, 64>), grid(64, 64), dim3(256), 0, s, it, rows,
                               lda, kdim, tri, ld, (int)sub);
    } else {
        // dependent steps: the tile with the least work on the fullest of the 256 CUs.  FP64 steps of two b x b blocks, us: b 768,
        // 192 columns 16.1 with 2 x 3 tiles (192 workgroups), 18.6 with 1 x 3, 19.2 with 2 x 2;
        // b 1856, 96 columns 31.0 with 2 x 3, 40.4 with 1 x 3; b 256, 192 columns 5.7 with
        // 1 x 2 (192 workgroups), 6.5 with 1 x 3, 8.6 with 2 x 3.
        // The second factor weighs the operand reads per product: with b 768 and 192 columns
        // 16 x 16 tiles would leave the CUs fuller (5 against 6 tiles each) but take 24.8 us.
        const int cm = ld % 48 == 0 ? 3 : 2;
        const int ck = tune_knob(XT_TUNE_BAND_CHAIN);
        int rt = 1, ct = 1;
        double best = 1e300;
        for (int r = 1; r <= 2; ++r)
            for (int k : {1, 2, 3}) {
                if (rows % (16 * r) || ld % (16 * k) || (r == 2 && k == 1)) continue;
                if ((ck == 1 && (r != 1 || k != 1)) || (ck == 2 && (r != 2 || k != cm)) ||
                    (ck == 3 && (r != 1 || k != cm)))
                    continue;
                const long long n = (long long)(rows / (16 * r)) * (ld / (16 * k)) * it.n;
                const double w = ceil_div(n, 256) * (r * k) * (1.0 + 0.25 / r + 0.25 / k);
                if (w < best) {
                    best = w;
                    rt = r;
                    ct = k;
                }
            }
        const bool one = (long long)(rows / (16 * rt)) * (ld / (16 * ct)) * it.n <= 256;
        // (a workgroup alone on its CU: 8 waves, two a SIMD, hide more of the loads)
        if (rt == 2 && ct == 3 && one) XT_PROD(2, 3, 8, 2, 1);
        else if (rt == 2 && ct == 3) XT_PROD(2, 3, 4, 2, 1);
        else if (rt == 2) XT_PROD(2, 2, 4, 2, 1);
        else if (ct == 3) XT_PROD(1, 3, 4, 3, 1);
        else if (ct == 2) XT_PROD(1, 2, 4, 3, 1);
        else XT_PROD(1, 1, 4, 4, 1);
    }
#undef XT_PROD
    if (prof) {
        const double mat = tri ? (double)rows * (rows + 1) / 2 : (double)rows * kdim * nseg;
        const double vec = (double)kdim * c * nseg + (double)rows * c * (sub ? 2 : 1);
        prof_end(band_kind<T>(), s, sizeof(T) * it.n * (mat + vec), 2.0 * it.n * mat * c, false);
    }
    return XT_OK;
}

// ---------------------------------------------------------------------------
// Setup kernels
// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// Blocked Cholesky of the band, 64-column panels (replaces potrf + trsm + syrk per block)
//
// Block i's column of the band is the tall panel [L_i; E_i] (diagonal block K_ii, then
// the sub-diagonal block K_{i+1,i}), both column-major b x b with leading dimension b.
// One launch per panel k (columns 64k..64k+63) of one or two eliminations (grid y), its
// workgroups independent of each other:
//   panel tiles (t, half): the diagonal tile (k, k) and half of row tile k + t take the
//     rank-64 update of panel k - 1, the diagonal tile is factored (identical arithmetic in
//     each workgroup, so identical results) and the rows solved against it, P = A_t L_kk^-T,
//     alongside.  t = 0 solves the identity instead, which gives D_kk = L_kk^-1 (nothing reads
//     L_kk again).  Results go to the scratch W; the matrix is only read.
//   trailing tiles: the rank-64 update of panel k - 1 on every tile right of column k: the
//     lower tiles of L_i, all tiles of E_i, and the lower tiles of the next diagonal
//     block (K_{i+1,i+1} -= E_i E_i^T, a piece per panel).
//   copies: panel k - 1's results from the other scratch Wp into its tiles of the matrix.
// Panel 0 of a block applies and copies the last panel of the block before it (pL, pE); a
// launch with k = nt only applies and copies the block's own last panel.
// What bounds it is the chain of panels, each the path through one workgroup: the launch,
// the tile loads (4,600 cycles), the rank-64 updates (6,600, 5,100 of FP64 matrix-core time on
// a CU) and four 16-column steps (5,200 cycles each, 3,900 of them the 16 x 16 block's
// chain): 22 us a panel on 768-row blocks.  Whole row tiles a workgroup: 9,600 for the updates;
// rows by forward substitution, four lanes a row, instead of by the block's inverse: 2,600
// more a step; a panel kernel (31.4 us) and an update kernel (18.9 us) after each other before.
// ---------------------------------------------------------------------------
constexpr int kCT = 64;   // panel width and tile size
constexpr int kCW = 8;    // waves of a workgroup

// One elimination's operands; a launch works on one or two of them (grid y).
struct CholSide {
    double *L = nullptr, *E = nullptr;     // diagonal and sub-diagonal block (E: NULL, none)
    double *Kn = nullptr;                  // next diagonal block (with E)
    double *pL = nullptr, *pE = nullptr;   // panel 0: the previous block
    const double *Wp = nullptr;            // tiles of the panel before this one (NULL: none)
    double *W = nullptr;                   // this panel's tiles
    int *info = nullptr;
};
struct CholSides {
    CholSide s[2];
};

// Work items of one launch: panel tiles, trailing tiles of L, E and Kn, copies.
struct CholItems {
    int np, nl, ne, nk, nc;
    __host__ __device__ int total() const { return np + nl + ne + nk + nc; }
};
__host__ __device__ inline CholItems chol_items(int nt, int k, bool E, bool Wp) {
    const int ntot = E ? 2 * nt : nt, T = nt - 1 - k;
    CholItems c;
    c.np = k < nt ? 2 * (ntot - k) : 0;
    c.nl = k < nt && Wp ? T * (T + 1) / 2 : 0;
    c.ne = k >= 1 && k < nt && E ? nt * T : 0;
    c.nk = k >= 1 && E ? nt * (nt + 1) / 2 : 0;
    c.nc = !Wp ? 0 : k == 0 ? nt + 1 : ntot - k + 1;
    return c;
}

__device__ inline double *tall_tile(double *L, double *E, int b, int nt, int rt, int ct) {
    double *base = rt < nt ? L + (size_t)rt * kCT : E + (size_t)(rt - nt) * kCT;
    return base + (size_t)ct * kCT * b;
}

// value of v in lane `src` of the wave (every lane gets it)
__device__ inline double lane_bcast(double v, int src) {
    const long long bits = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)bits, src);
    const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), src);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

typedef double xt_d4c __attribute__((ext_vector_type(4)));

// Block (16 I.., 16 J..) of P Q^T, P and Q 64 x 64 column-major tiles: accumulator i of
// lane (g, q) is element (16 I + q, 16 J + g + 4 i).
__device__ inline xt_d4c block_product(const double *P, const double *Q, int I, int J, int g,
                                       int q) {
    double pv[kCT / 4], qv[kCT / 4];
#pragma unroll
    for (int k4 = 0; k4 < kCT / 4; ++k4) {
        pv[k4] = P[(4 * k4 + g) * kCT + 16 * I + q];
        qv[k4] = Q[(4 * k4 + g) * kCT + 16 * J + q];
    }
    xt_d4c acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k4 = 0; k4 < kCT / 4; ++k4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(qv[k4], pv[k4], acc, 0, 0, 0);
    return acc;
}

// a_r += a_rJ t for the rows r0 + i (i < N), a_rJ lane J's value of each row of 16 lanes.  (Two
// wait states stand between a write of a register and its read by lane-crossing operands.)
#define XT_ELIM(i) "v_fmac_f64_dpp %" #i ", %" #i ", %[t] row_newbcast:%[j] row_mask:0xf bank_mask:0xf\n\t"
template <int J>
__device__ inline void eliminate1(double &a0, double t) {
    asm("s_nop 1\n\t" XT_ELIM(0) : "+&v"(a0) : [t] "v"(t), [j] "n"(J));
}
template <int J>
__device__ inline void eliminate5(double &a0, double &a1, double &a2, double &a3, double &a4,
                                  double t) {
    asm("s_nop 1\n\t" XT_ELIM(0) XT_ELIM(1) XT_ELIM(2) XT_ELIM(3) XT_ELIM(4)
        : "+&v"(a0), "+&v"(a1), "+&v"(a2), "+&v"(a3), "+&v"(a4) : [t] "v"(t), [j] "n"(J));
}
template <int J>
__device__ inline void eliminate4(double &a0, double &a1, double &a2, double &a3, double t) {
    asm("s_nop 1\n\t" XT_ELIM(0) XT_ELIM(1) XT_ELIM(2) XT_ELIM(3)
        : "+&v"(a0), "+&v"(a1), "+&v"(a2), "+&v"(a3) : [t] "v"(t), [j] "n"(J));
}
#undef XT_ELIM

// Elimination of column J of a symmetric 16 x 16 block, unscaled: lane q of every row of 16
// lanes holds column q, all 16 rows (the four rows of lanes do the same).  a_rc -= a_rJ a_Jc / p
// for the rows r > J; above them stand the rows of the identity eliminated along, x_rc in place
// of a_rc: row J becomes x_Jc = -a_Jc / p, the rows before it x_rc -= x_rJ a_Jc / p.
// Finished columns (q <= J) keep their values.  Row J + 1, which holds the next pivot, is
// eliminated at once, the other rows of column J - 1 (its t: tp) while 1 / p is on its way.
template <int J>
__device__ inline void chol_column(double (&a)[16], int q, double &tp) {
    const double p = lane_bcast(a[J], J);
    const double row = q > J ? -a[J] : 0.0;
    // 1 / p: the hardware estimate (relative error e ~ 2^-24) and a third-order step
    const double r = __builtin_amdgcn_rcp(p);
    constexpr int P = J - 1;   // rows P + 2 .. P + 15 (mod 16): all but P and P + 1
    auto at = [&](int k) -> double & { return a[(P + 2 + k) & 15]; };
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (J > 0) eliminate5<P>(at(0), at(1), at(2), at(3), at(4), tp);
    __builtin_amdgcn_sched_barrier(0);
    const double e = fma(-p, r, 1.0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (J > 0) eliminate5<P>(at(5), at(6), at(7), at(8), at(9), tp);
    __builtin_amdgcn_sched_barrier(0);
    const double f = fma(e, e, e);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (J > 0) eliminate4<P>(at(10), at(11), at(12), at(13), tp);
    __builtin_amdgcn_sched_barrier(0);
    const double t = row * fma(r, f, r);
    if constexpr (J < 15) eliminate1<J>(a[(J + 1) & 15], t);
    a[J] = q > J ? t : a[J];
    __builtin_amdgcn_sched_barrier(0);
    tp = t;
}

// The upper triangle of X = L^-T of the 16 x 16 block at columns c0 of the tile (lower
// triangle), L its Cholesky factor (X's other entries are left undefined), by one wave: the identity's rows eliminated along with the block, scaled by
// 1 / sqrt(pivot) at the end.  Returns the first non-positive pivot (1-based, 0: none).
// Bound by the dependent chain pivot -> 1 / pivot -> next pivot and some 26 instructions a
// column, without a root, an LDS access or a lane exchange on the chain but the pivot's:
// 3,900 cycles with the inverse and the block's way through LDS.  The rows of a column over
// the four rows of lanes, exchanged by lane swaps, 4,400; a column scaled by its root, its
// coefficients through lane reads and LDS, 5,900 without the inverse.
__device__ inline int chol16_inverse(const double (*sA)[kCT + 1], int c0, int lane,
                                     double (*X)[17]) {
    const int q = lane & 15;
    double a[16], tp = 0.0;
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = sA[c0 + max(r, q)][c0 + min(r, q)];
    chol_column<0>(a, q, tp);
    chol_column<1>(a, q, tp);
    chol_column<2>(a, q, tp);
    chol_column<3>(a, q, tp);
    chol_column<4>(a, q, tp);
    chol_column<5>(a, q, tp);
    chol_column<6>(a, q, tp);
    chol_column<7>(a, q, tp);
    chol_column<8>(a, q, tp);
    chol_column<9>(a, q, tp);
    chol_column<10>(a, q, tp);
    chol_column<11>(a, q, tp);
    chol_column<12>(a, q, tp);
    chol_column<13>(a, q, tp);
    chol_column<14>(a, q, tp);
    chol_column<15>(a, q, tp);
    // (column 15 has no columns behind it)
    double piv = a[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) piv = q >= r ? a[r] : piv;
    // 1 / sqrt(p): y (1 + e/2 + 3 e^2/8) with e = 1 - p y^2, error 0.3 e^3
    const double y = __builtin_amdgcn_rsq(piv), er = fma(-piv * y, y, 1.0);
    const double rd = fma(y * er, fma(0.375, er, 0.5), y);
    if (lane < 16) {   // (a wave's LDS accesses complete in order)
#pragma unroll
        for (int r = 0; r < 15; ++r) X[r][q] = a[r] * rd;
        X[q][q] = rd;
    }
    const unsigned long long bad = __ballot(!(piv > 0.0)) & 0xFFFF;
    return bad ? __ffsll(bad) : 0;
}

__global__ void __launch_bounds__(64 * kCW)
chol_step_kernel(int b, int nt, int k, CholSides cs) {
    // panel: the diagonal tile and this workgroup's row tile, [row][column]; trailing: P, Q
    __shared__ double lds[2][kCT][kCT + 1];
    __shared__ double sL[16][17];      // L^-T of the step's 16 x 16 diagonal block
    __shared__ int sbad;
    const CholSide &S = cs.s[blockIdx.y];
    double *L = S.L, *E = S.E;
    const double *Wp = S.Wp;
    const CholItems ci = chol_items(nt, k, E != nullptr, Wp != nullptr);
    int id = blockIdx.x;
    if (id >= ci.total()) return;      // (the two eliminations' counts can differ)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, q = lane & 15;
    constexpr size_t TS = (size_t)kCT * kCT;
    // tile of Wp that holds row tile rt of the panel before (panel 0: row i of the next block)
    auto wp = [&](int rt) { return Wp + TS * (k == 0 ? 1 + rt : rt - (k - 1)); };
    if (id >= ci.np) {                 // trailing tile or copy
        id -= ci.np;
        const int T = nt - 1 - k;
        double *C;
        const double *P, *Q;
        if (id < ci.nl) {              // lower tile (i, j) of L, k < j <= i
            int jj = 0, rem = id;
            while (rem >= T - jj) { rem -= T - jj; ++jj; }
            const int j = k + 1 + jj, i = j + rem;
            C = tall_tile(L, E, b, nt, i, j);
            P = wp(i);
            Q = wp(j);
        } else if ((id -= ci.nl) < ci.ne) {   // E tile (i, j), j > k
            const int i = id / T, j = k + 1 + (id - i * T);
            C = tall_tile(L, E, b, nt, nt + i, j);
            P = wp(nt + i);
            Q = wp(j);
        } else if ((id -= ci.ne) < ci.nk) {   // Kn lower tile (i, j): E's row tiles i, j
            int j = 0, rem = id;
            while (rem >= nt - j) { rem -= nt - j; ++j; }
            const int i = j + rem;
            C = S.Kn + (size_t)j * kCT * b + (size_t)i * kCT;
            P = wp(nt + i);
            Q = wp(nt + j);
        } else {                       // copy of the panel before: its tile id
            id -= ci.nk;
            double *dst = k == 0 ? tall_tile(S.pL, S.pE, b, nt, nt - 1 + id, nt - 1)
                                 : tall_tile(L, E, b, nt, k - 1 + id, k - 1);
            const double *src = Wp + TS * id;
            for (int e = tid; e < kCT * kCT; e += 64 * kCW)
                dst[(size_t)(e >> 6) * b + (e & 63)] = src[e];
            return;
        }
        double *sP = &lds[0][0][0], *sQ = &lds[1][0][0];
        for (int e = tid; e < kCT * kCT; e += 64 * kCW) {
            sP[e] = P[e];
            sQ[e] = Q[e];
        }
        // 16 x 16 blocks (I, J0) and (I, J0 + 2) by each wave; the lanes of a quarter wave hold
        // 16 consecutive rows of one column
        const int I = wave & 3, J0 = wave >> 2;
        double old[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                old[h][i] = C[(size_t)(16 * (J0 + 2 * h) + g + 4 * i) * b + 16 * I + q];
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const xt_d4c acc = block_product(sP, sQ, I, J0 + 2 * h, g, q);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                C[(size_t)(16 * (J0 + 2 * h) + g + 4 * i) * b + 16 * I + q] = old[h][i] - acc[i];
        }
        return;
    }
    constexpr int HR = kCT / 2;       // rows of a half row tile
    const int t = id >> 1, hr = (id & 1) * HR;
    double (*sA)[kCT + 1] = lds[0], (*sX)[kCT + 1] = lds[1];
    const double *D = tall_tile(L, E, b, nt, k, k);
    const double *At = tall_tile(L, E, b, nt, k + t, k) + hr;
    // the tile and the half row tile into registers and the panel before's tiles k and k + t
    // into LDS (every wave needs most of them: 16 loads of one wave's column instead of 64)
    constexpr int NE = kCT / kCW, NX = HR * kCT / (64 * kCW);   // loads a lane
    const int xr = tid & (HR - 1), xc = tid / HR;               // row and column of load 0
    double dv[NE], xv[NX];
#pragma unroll
    for (int e = 0; e < NE; ++e) dv[e] = D[(size_t)(wave + kCW * e) * b + lane];
#pragma unroll
    for (int e = 0; e < NX; ++e) {
        const int c = xc + e * (64 * kCW / HR);
        xv[e] = t > 0 ? At[(size_t)c * b + xr] : hr + xr == c ? 1.0 : 0.0;
    }
    // rank-64 update of the panel before: the half row tile's 8 blocks by waves 0 - 3 (panel 0
    // leaves the rows of E alone), the diagonal tile's lower 10 by waves 4 - 7, two or three
    // blocks a wave, of one block row (its operand is read from LDS once) but wave 7's third
    const bool upx = t > 0 && (k > 0 || t < nt);
    const bool xw = wave < 4, w3 = wave >= 6;   // of the row tile; three blocks
    auto block_row = [&](int h) { return xw ? wave >> 1 : wave < 6 ? 3 : wave == 6 ? 2 : h < 2; };
    auto block_col = [&](int h) { return wave < 6 ? 2 * (wave & 1) + h : wave == 6 ? h : h & 1; };
    constexpr int UW = 3;
    xt_d4c au[UW];
    if (Wp) {
        double *sk = &lds[0][0][0], *st = &lds[1][0][0];
        const double *Pk = wp(k), *Pt = wp(k + t) + hr;
        double pk[NE], pt[NX];
#pragma unroll
        for (int e = 0; e < NE; ++e) pk[e] = Pk[tid + 64 * kCW * e];
#pragma unroll
        for (int e = 0; e < NX; ++e)
            pt[e] = upx ? Pt[(xc + e * (64 * kCW / HR)) * kCT + xr] : 0.0;
#pragma unroll
        for (int e = 0; e < NE; ++e) sk[tid + 64 * kCW * e] = pk[e];
#pragma unroll
        for (int e = 0; e < NX; ++e) st[tid + 64 * kCW * e] = pt[e];
        __syncthreads();
        double pv[kCT / 4];
#pragma unroll
        for (int h = 0; h < UW; ++h) {
            if ((xw && !upx) || (h == 2 && !w3)) break;
            double qv[kCT / 4];
#pragma unroll
            for (int k4 = 0; k4 < kCT / 4; ++k4) qv[k4] = sk[(4 * k4 + g) * kCT + 16 * block_col(h) + q];
            if (h == 0 || (h == 2 && wave == 7)) {
                const double *P = (xw ? st + g * HR : sk + g * kCT) + 16 * block_row(h) + q;
                const int ps = 4 * (xw ? HR : kCT);
#pragma unroll
                for (int k4 = 0; k4 < kCT / 4; ++k4) pv[k4] = P[k4 * ps];
            }
            au[h] = xt_d4c{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k4 = 0; k4 < kCT / 4; ++k4)
                au[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(qv[k4], pv[k4], au[h], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) sA[lane][wave + kCW * e] = dv[e];
#pragma unroll
    for (int e = 0; e < NX; ++e) sX[xr][xc + e * (64 * kCW / HR)] = xv[e];
    if (tid == 0) sbad = 0;
    __syncthreads();
    if (Wp) {
#pragma unroll
        for (int h = 0; h < UW; ++h) {
            if ((xw && !upx) || (h == 2 && !w3)) break;
            double (*Cm)[kCT + 1] = xw ? sX : sA;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                Cm[16 * block_row(h) + q][16 * block_col(h) + g + 4 * i] -= au[h][i];
        }
        __syncthreads();
    }
    // rank-16 update of block (Ib, J) of the tile (or of the row tile) by step s's columns
    auto rank16 = [&](double (*Cm)[kCT + 1], int Ib, int J, int c0) {
        xt_d4c a4 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4) {
            const double pa = Cm[16 * Ib + q][c0 + 4 * k4 + g];
            const double qb = sA[16 * J + q][c0 + 4 * k4 + g];
            a4 = __builtin_amdgcn_mfma_f64_16x16x4f64(pa, qb, a4, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) Cm[16 * Ib + g + 4 * i][16 * J + q] -= a4[i];
    };
    // four 16-column steps: the inverse factor of the 16 x 16 diagonal block by wave 0 in
    // registers while the other waves finish the step before (the rank-16 updates past the
    // next 16 columns); then on the matrix cores the rows below it (and the row tile's) by
    // that inverse and the rank-16 update of the next 16 columns
    for (int s = 0; s < 4; ++s) {
        const int c0 = 16 * s;
        if (wave == 0) {
            const int bad = chol16_inverse(sA, c0, lane, sL);
            if (tid == 0 && bad && !sbad) sbad = c0 + bad;
        } else if (s > 0) {
            // blocks (Ib, J) of the tile with s < J <= Ib, then (0..1, J) of the row tile
            const int nj = 3 - s, n1 = nj * (nj + 1) / 2, n2 = 2 * nj;
            for (int u = wave - 1; u < n1 + n2; u += kCW - 1) {
                if (u < n1) {
                    const int J = u < nj ? s + 1 : s + 2, Ib = u < nj ? s + 1 + u : 3;
                    rank16(sA, Ib, J, c0 - 16);
                } else {
                    rank16(sX, (u - n1) & 1, s + 1 + ((u - n1) >> 1), c0 - 16);
                }
            }
        }
        __syncthreads();
        // the rows below the block in the tile and the row tile's: x = a L_s^-T
        {
            const int n1 = 3 - s;
            if (wave < n1 + 2) {
                double (*Cm)[kCT + 1] = wave < n1 ? sA : sX;
                const int r0 = wave < n1 ? c0 + 16 + 16 * wave : 16 * (wave - n1);
                double pa[4], qb[4];
#pragma unroll
                for (int k4 = 0; k4 < 4; ++k4) {
                    pa[k4] = Cm[r0 + q][c0 + 4 * k4 + g];
                    qb[k4] = 4 * k4 + g <= q ? sL[4 * k4 + g][q] : 0.0;
                }
                xt_d4c a4 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int k4 = 0; k4 < 4; ++k4)
                    a4 = __builtin_amdgcn_mfma_f64_16x16x4f64(pa[k4], qb[k4], a4, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) Cm[r0 + g + 4 * i][c0 + q] = a4[i];
            }
        }
        __syncthreads();
        if (s < 3) {   // the next 16 columns: blocks (s + 1..3, s + 1), the row tile's (0..1, s + 1)
            const int n1 = 3 - s;
            if (wave < n1) rank16(sA, s + 1 + wave, s + 1, c0);
            else if (wave < n1 + 2) rank16(sX, wave - n1, s + 1, c0);
            __syncthreads();
        }
    }
    if (id == 0 && tid == 0 && sbad && !S.info[0]) S.info[0] = k * kCT + sbad;   // (the first)
    double *wt = S.W + TS * t;
    if (t > 0) {
        for (int e = tid; e < HR * kCT; e += 64 * kCW) {
            const int c = e / HR, r = e & (HR - 1);
            wt[c * kCT + hr + r] = sX[r][c];
        }
    } else {                           // row r of the solved identity: column r of D_kk
        for (int e = tid; e < HR * kCT; e += 64 * kCW)
            wt[hr * kCT + e] = sX[e >> 6][e & 63];
    }
}

// D = L^-1 of column-major lower b x b blocks whose diagonal tiles already hold D_kk, in
// both layouts (du column-major, dl row-major), one 64 x 64 tile a workgroup: the tiles at
// distance d below the diagonal from those nearer to it,
//   D_ij = -D_ii (L_ij D_jj + ... + L_i,i-1 D_i-1,j),   j = i - d,
// the inner products accumulated in registers (operands straight from memory: L
// column-major gives the rows of A, dl row-major the columns of B as 128-byte runs), the
// sum and the result turned through LDS.  d = 0 copies the diagonal tiles and zeroes the
// others above.  nt - 1 launches over all blocks; matrix-core bound where there are many
// (93 blocks of 768 rows: 0.9 ms, the library's batched trtri and two transposing passes
// 5.2 ms).
__global__ void __launch_bounds__(256)
tri_inverse_kernel(int b, int nt, int d, const double *__restrict__ Lb, double *du, double *dl) {
    __shared__ double sm[kCT][kCT + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, q = lane & 15;
    const long long off = (long long)blockIdx.y * b * b;
    Lb += off;
    du += off;
    dl += off;
    if (d == 0) {   // tiles (i, j), j >= i
        int i = 0, rem = blockIdx.x;
        while (rem >= nt - i) { rem -= nt - i; ++i; }
        const int j = i + rem;
        for (int e = tid; e < kCT * kCT; e += 256) {
            const int c = e >> 6, r = e & 63;
            const double v = i == j ? Lb[(size_t)(j * kCT + c) * b + i * kCT + r] : 0.0;
            du[(size_t)(j * kCT + c) * b + i * kCT + r] = v;
            if (i == j) sm[r][c] = v;
        }
        __syncthreads();
        for (int e = tid; e < kCT * kCT; e += 256) {
            const int r = e >> 6, c = e & 63;
            dl[(size_t)(i * kCT + r) * b + j * kCT + c] = i == j ? sm[r][c] : 0.0;
        }
        return;
    }
    const int i = d + blockIdx.x, j = blockIdx.x;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;   // this wave's quadrant
    xt_d4c acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = xt_d4c{0.0, 0.0, 0.0, 0.0};
    // one 64-deep product: A(row, m) = a[m b + row], B(m, column) from the functor
    auto product = [&](const double *a, auto bval) {
#pragma unroll
        for (int m0 = 0; m0 < kCT / 4; m0 += 8) {
            double av[8][2], bv[8][2];
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const int m = 4 * (m0 + u) + g;
                    av[u][x] = a[(size_t)m * b + wr + 16 * x + q];
                    bv[u][x] = bval(m, wc + 16 * x + q);
                }
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 2; ++y)
                        acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u][x], bv[u][y],
                                                                         acc[x][y], 0, 0, 0);
        }
    };
    for (int k = j; k < i; ++k) {
        const double *B = dl + (size_t)k * kCT * b + j * kCT;
        product(Lb + (size_t)k * kCT * b + i * kCT,
                [&](int m, int c) { return B[(size_t)m * b + c]; });
    }
    auto to_lds = [&]() {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sm[wr + 16 * x + g + 4 * e][wc + 16 * y + q] = acc[x][y][e];
                    acc[x][y][e] = 0.0;
                }
        __syncthreads();
    };
    to_lds();
    product(Lb + (size_t)i * kCT * b + i * kCT, [&](int m, int c) { return sm[m][c]; });
    __syncthreads();
    to_lds();
    for (int e = tid; e < kCT * kCT; e += 256) {
        const int c = e >> 6, r = e & 63;
        dl[(size_t)(i * kCT + c) * b + j * kCT + r] = -sm[c][r];
        du[(size_t)(j * kCT + c) * b + i * kCT + r] = -sm[r][c];
    }
}

__global__ void __launch_bounds__(256)
to_f32_kernel(long long n, const double *__restrict__ s, float *__restrict__ d) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (long long)gridDim.x * 256)
        d[i] = (float)s[i];
}

template <typename T>
__global__ void __launch_bounds__(256)
fill_zero_kernel(long long n, T *d) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (long long)gridDim.x * 256)
        d[i] = T(0);
}

// Lower triangle of the 1-based CSR K into column-major b x b blocks in the factor's order:
// diagonal blocks from block f0 on (kd) and sub-diagonal blocks from index e0 on (ko; top
// chain's block i at index i, bottom chain's block j at nt + j).  One lane per row in entry
// order (a repeated entry: the last one stays).  A row i past the middle block is row
// split + total - 1 - i of the factor's order, where the roles of an entry's row and column
// change places; the last bottom block's couplings to the middle block keep the middle's
// row order.  The rows of the last block beyond p get a unit diagonal.  The blocks are zero
// on entry.  flags[0] set: an entry outside the blocks; flags[1]: the largest i - j.
__global__ void __launch_bounds__(256)
band_scatter_kernel(int p, int b, int nb, int nt, int f0, int e0, const int *__restrict__ ia,
                    const int *__restrict__ ja, const double *__restrict__ a, double *kd,
                    double *ko, int *flags) {
    const int i = f0 * b + blockIdx.x * 256 + threadIdx.x;
    const long long bb = (long long)b * b;
    const int total = nb * b, split = (nt + 1) * b;
    if (i >= total) return;
    const int pi = i < split ? i : split + total - 1 - i;
    const int bi = pi / b, li = pi - bi * b;
    if (i >= p) {
        kd[(bi - f0) * bb + (long long)li * b + li] = 1.0;
        return;
    }
    int wide = 0;
    for (int k = ia[i] - 1; k < ia[i + 1] - 1; ++k) {
        const int j = ja[k] - 1;
        if (j > i) continue;
        if (j < 0 || i - j > b) {   // not in the blocks this factor was sized for
            flags[0] = 1;
            continue;
        }
        wide = max(wide, i - j);
        const int pj = j < split ? j : split + total - 1 - j;
        const int bj = pj / b, lj = pj - bj * b;
        int row = li, col = lj, e = bj;      // off-diagonal block: index, row, column in it
        if (i >= split) {                    // (j in the middle block or past it)
            row = lj;
            col = li;
            e = bi - 1;
        }
        if (bi == bj) kd[(bi - f0) * bb + (long long)col * b + row] = a[k];
        else if (e >= e0) ko[(e - e0) * bb + (long long)col * b + row] = a[k];
    }
    if (wide > 0) atomicMax(flags + 1, wide);
}

// dst += src (n elements)
__global__ void __launch_bounds__(256)
add_block_kernel(long long n, const double *__restrict__ src, double *__restrict__ dst) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (long long)gridDim.x * 256)
        dst[i] += src[i];
}

static int zero_fill(double *d, long long n, hipStream_t s) {
    if (n <= 0) return XT_OK;
    hipLaunchKernelGGL(fill_zero_kernel<double>, dim3(8192), dim3(256), 0, s, n, d);
    XT_HIP(hipGetLastError());
    return XT_OK;
}

// Where the matrices of one chain's recurrence (dir 0 forward, 1 backward) sit in a level's
// array: cnt of them, es elements apart.  They are stored in ascending block order, which
// for the backward recurrence is the reverse of its steps: step v (1, 2, ..) uses entry
// v - 1 forward and cnt - v backward.  vrow / crow: first of the kw rows the next step
// reads and of the rc rows the chain runs on, in an entry of rows rows.
struct LevelView {
    long long base, es;
    int cnt, vrow, crow;
};
static LevelView level_view(const BandPrec &bp, int side, int dir, int L) {
    LevelView v;
    const int rows = L == 0 ? bp.b : bp.rc;
    v.es = (long long)rows * bp.kw;
    v.cnt = bp.steps(side, dir) >> L;
    v.base = side == 0 ? 0 : v.es * (L == 0 ? bp.nt : bp.steps(0, dir) >> L);
    v.vrow = dir == 0 ? rows - bp.kw : 0;
    v.crow = dir == 0 ? rows - bp.rc : 0;
    return v;
}

// Level-L matrices of direction dir of one chain, stored entries t0 <= t < t1:
// M^L_t = -(M^{L-1}_{2t+1} M^{L-1}_{2t}) in step order, M^0 = G forward and H backward.
// Row-major X is column-major X^T, so the row-major product is the column-major product
// of the stored blocks in the order M_{2t}, M_{2t+1}.
static int level_products(rocblas_handle h, const BandPrec &bp, int side, int dir, int L, int t0,
                          int t1, const double *below, double *out) {
    if (t1 <= t0) return XT_OK;
    const LevelView f = level_view(bp, side, dir, L - 1), v = level_view(bp, side, dir, L);
    const double minus = -1.0, zero = 0.0;
    // stored entries of M_{2t} and M_{2t+1} for the first t
    const long long lo = dir == 0 ? 2LL * t0 : f.cnt - 2LL * v.cnt + 2LL * t0 + 1;
    const long long hi = dir == 0 ? lo + 1 : lo - 1;
    const double *A = below + f.base + lo * f.es + (long long)f.vrow * bp.kw;
    const double *B = below + f.base + hi * f.es + (long long)f.crow * bp.kw;
    XT_RB(rocblas_dgemm_strided_batched(h, rocblas_operation_none, rocblas_operation_none, bp.kw,
                                        bp.rc, bp.kw, &minus, A, bp.kw, 2 * f.es, B, bp.kw,
                                        2 * f.es, &zero, out + v.base + t0 * v.es, bp.kw, v.es,
                                        t1 - t0));
    return XT_OK;
}

// G_i (row-major D_{i+1} E_i, its last kw columns) for n consecutive i: E the first E_i,
// Dn the first D_{i+1}, both column-major b x b, G the first G_i.  E_i's nonzero rows start
// at e0 (0 within a chain).
static int g_products(rocblas_handle h, const BandPrec &bp, const double *E, int e0,
                      const double *Dn, double *G, int n) {
    if (n <= 0) return XT_OK;
    const int b = bp.b, kw = bp.kw;
    const long long bb = (long long)b * b;
    const double one = 1.0, zero = 0.0;
    XT_RB(rocblas_dgemm_strided_batched(
        h, rocblas_operation_transpose, rocblas_operation_transpose, kw, b, kw, &one,
        E + e0 + (long long)(b - kw) * b, b, bb, Dn + (long long)e0 * b, b, bb, &zero, G, kw,
        (long long)b * kw, n));
    return XT_OK;
}
// H_i (row-major (E_i D_i)^T, the kw columns from E_i's row e0 on) for n consecutive i.
static int h_products(rocblas_handle h, const BandPrec &bp, const double *E, int e0,
                      const double *D, double *H, int n) {
    if (n <= 0) return XT_OK;
    const int b = bp.b, kw = bp.kw;
    const long long bb = (long long)b * b;
    const double one = 1.0, zero = 0.0;
    XT_RB(rocblas_dgemm_strided_batched(
        h, rocblas_operation_none, rocblas_operation_none, kw, b, kw, &one,
        E + e0 + (long long)(b - kw) * b, b, bb, D + (b - kw), b, bb, &zero, H, kw,
        (long long)b * kw, n));
    return XT_OK;
}

// FP32 copy of elements [off, off + n) of an FP64 set.
static int to_f32_range(DevBuf *set, long long off, long long n, hipStream_t s) {
    if (n <= 0 || !set[0].ptr) return XT_OK;
    hipLaunchKernelGGL(to_f32_kernel, dim3(4096), dim3(256), 0, s, n,
                       set[0].as<double>() + off, set[1].as<float>() + off);
    XT_HIP(hipGetLastError());
    return XT_OK;
}

// One elimination in progress: its two scratch panels (of 2 nt tiles each) and the panel
// that the next launch applies.
struct CholRun {
    double *W[2] = {nullptr, nullptr};
    int cur = 0;                      // W[cur]: the next panel's tiles
    bool have = false;                // W[1 - cur] holds a panel not yet applied
    double *pL = nullptr, *pE = nullptr;   // the block it belongs to, when it is that block's last
    CholSide side(double *L, double *E, double *Kn, int *info) const {
        CholSide c;
        c.L = L;
        c.E = E;
        c.Kn = Kn;
        c.pL = pL;
        c.pE = pE;
        c.Wp = have ? W[1 - cur] : nullptr;
        c.W = W[cur];
        c.info = info;
        return c;
    }
};

static int chol_launch(int b, int nt, int k, const CholSide *sides, int n, hipStream_t s) {
    CholSides cs;
    int total = 0;
    for (int i = 0; i < 2; ++i) {
        cs.s[i] = sides[std::min(i, n - 1)];
        total = std::max(total, chol_items(nt, k, cs.s[i].E != nullptr, cs.s[i].Wp != nullptr).total());
    }
    if (total > 0)
        hipLaunchKernelGGL(chol_step_kernel, dim3(total, n), dim3(64 * kCW), 0, s, b, nt, k, cs);
    XT_HIP(hipGetLastError());
    return XT_OK;
}

// The panels of one block of each of n eliminations (side i: block blk[i], run *run[i]).
static int factor_blocks(int b, const CholSide *blk, CholRun *const *run, int n, hipStream_t s) {
    const int nt = b / kCT;
    for (int k = 0; k < nt; ++k) {
        CholSide sd[2];
        for (int i = 0; i < n; ++i) {
            sd[i] = run[i]->side(blk[i].L, blk[i].E, blk[i].Kn, blk[i].info);
            run[i]->cur ^= 1;
            run[i]->have = true;
        }
        XT_TRY(chol_launch(b, nt, k, sd, n, s));
    }
    for (int i = 0; i < n; ++i) {
        run[i]->pL = blk[i].L;
        run[i]->pE = blk[i].E;
    }
    return XT_OK;
}
// Apply and store the last panel of an elimination's last block.
static int factor_flush(int b, const CholSide &blk, const CholRun &run, hipStream_t s) {
    const CholSide sd = run.side(blk.L, blk.E, blk.Kn, blk.info);
    return chol_launch(b, b / kCT, b / kCT, &sd, 1, s);
}

// Estimated time (us) of one chain pair's forward or backward recurrence with nl pairing
// levels: every launch costs a latency (the boundary and the first loads: 4.6 us for two
// 256-row blocks) plus the larger of streaming its matrices and its products, at the rates
// the sweeps reach (4.4 TB/s; 45 TFLOP/s in FP64, the products of the dependent steps and
// of the batched passes alike).  Levels halve the number of dependent steps and add a pass
// over half the blocks each way.
static double chain_cost(int rows, int kw, int m0, int m1, int nl, int ld, size_t sv) {
    auto launch = [&](double n) {
        const double e = n * rows * kw;
        return 4.6 + std::max(e * sv / 4.4e6, 2.0 * e * ld / (sv == 8 ? 45e6 : 90e6));
    };
    double t = 0.0;
    for (int L = 0; L < nl; ++L)
        t += launch((m0 >> L) / 2 + (m1 >> L) / 2) +
             launch(((m0 >> L) + 1) / 2 + ((m1 >> L) + 1) / 2);
    return t + std::max(m0 >> nl, m1 >> nl) * launch(2);
}
// Pairing levels, of at most most, with the least estimated time for ld columns.
static int chain_levels(const BandPrec &bp, int most, int ld, size_t sv) {
    int best = 0;
    double tb = 1e300;
    for (int nl = 0; nl <= most; ++nl) {
        const double t = chain_cost(bp.rc, bp.kw, bp.steps(0, 1), bp.steps(1, 1), nl, ld, sv);
        if (t < tb) {
            tb = t;
            best = nl;
        }
    }
    return best;
}

// Columns of G and H and rows of the chains for a half-bandwidth of bw.
static void set_band(BandPrec &bp, int bw) {
    bp.kw = std::min(bp.b, std::max(64, (bw + 63) / 64 * 64));
    bp.rc = 2 * bp.kw <= bp.b ? bp.kw : bp.b;
}

// Block Cholesky of K given as a 1-based CSR in device memory (lower triangle read).
// fb > 0 (a factor with its FP64 sets, K changed only in rows and columns of blocks fb..):
// the top chain's blocks before fb are kept and the factor is recomputed from there on,
// starting from E_{ft-1} = K_{ft,ft-1} D_{ft-1}^T and the Schur complement K_{ft,ft} - E E^T
// (ft = fb, or the middle block when fb is past it: the bottom chain, which starts at the
// last row, is always recomputed); the pairing levels are recomputed where they depend on
// a changed block.  The result equals a full factorization up to rounding.
static int factor_dev(BandPrec &bp, const int *dia, const int *dja, const double *da,
                      hipStream_t s, int fb = 0) {
    const int b = bp.b, nb = bp.nb, p = bp.p, nt = bp.nt, nbt = bp.nbt;
    const long long bb = (long long)b * b;
    if (fb >= nb || !band_has_fp64(&bp) || !bp.Dl[0].ptr) fb = 0;
    const int ft = std::min(fb, nt);              // first block factored here
    const int nr = nb - ft, e0 = std::max(0, ft - 1), ne = nb - 1 - e0;
    DevBuf &L = bp.sL, &E = bp.sE, &Wb = bp.sW, &Km = bp.sK, &info = bp.sinfo;
    struct Release {   // the scratch is freed on every way out unless it is kept
        BandPrec &bp;
        const bool again;   // a refactorization: the factor was built before this call
        ~Release() {
            DevBuf *b[5] = {&bp.sL, &bp.sE, &bp.sW, &bp.sK, &bp.sinfo};
            size_t sum = 0;
            for (DevBuf *d : b) sum += d->bytes;
            if (again && bp.keep64 && sum <= kKeepScratch) {
                // (the caller's stream may be gone by the next call)
                if (bp.rb && bp.rb->h) (void)rocblas_set_stream(bp.rb->h, nullptr);
                return;
            }
            for (DevBuf *d : b) d->release();
            delete bp.rb;
            bp.rb = nullptr;
        }
    } release{bp, bp.built};
    struct Band {      // a failed factorization leaves the old factor's layout
        BandPrec &bp;
        const int kw, rc;
        bool ok = false;
        ~Band() {
            if (!ok) {
                bp.kw = kw;
                bp.rc = rc;
            }
        }
    } band{bp, bp.kw, bp.rc};
    DevBuf E0;
    XT_TRY(L.reserve(sizeof(double) * bb * nr));
    XT_TRY(zero_fill(L.as<double>(), bb * nr, s));
    if (ne > 0) {
        XT_TRY(E.reserve(sizeof(double) * bb * ne));
        XT_TRY(zero_fill(E.as<double>(), bb * ne, s));
    }
    XT_TRY(info.reserve(sizeof(int) * (nb + 2)));
    XT_HIP(hipMemsetAsync(info.ptr, 0, sizeof(int) * (nb + 2), s));
    hipLaunchKernelGGL(band_scatter_kernel, dim3(ceil_div((long long)(nb - ft) * b, 256)), dim3(256),
                       0, s, p, b, nb, nt, ft, e0, dia, dja, da, L.as<double>(),
                       ne > 0 ? E.as<double>() : nullptr, info.as<int>() + nb);
    XT_HIP(hipGetLastError());
    {
        int flags[2] = {0, 0};
        XT_HIP(hipMemcpyAsync(flags, info.as<int>() + nb, 2 * sizeof(int), hipMemcpyDeviceToHost, s));
        XT_HIP(hipStreamSynchronize(s));
        if (flags[0]) {
            set_error("K has entries outside the band of width %d the factor was built for", b);
            return XT_E_ARG;
        }
        if (flags[1] > bp.kw) {   // a wider band than the factor had, within its blocks
            set_band(bp, flags[1]);
            if (ft > 0) {
                const int rc0 = factor_dev(bp, dia, dja, da, s, 0);
                band.ok = rc0 == XT_OK;
                return rc0;
            }
        }
    }
    XT_HIP(hipMemsetAsync(info.ptr, 0, sizeof(int) * (nb + 2), s));
    const int kw = bp.kw, rc = bp.rc;
    const long long bk = (long long)b * kw;
    double *Lp = L.as<double>(), *Ep = E.as<double>();
    auto Lat = [&](int beta) { return Lp + (beta - ft) * bb; };   // diagonal block beta
    auto Eat = [&](int e) { return Ep + (e - e0) * bb; };         // sub-diagonal block e
    if (!bp.rb) bp.rb = new (std::nothrow) RbHandle;
    if (!bp.rb) return XT_E_NOMEM;
    RbHandle &rb = *bp.rb;
    if (!rb.h) XT_RB(rocblas_create_handle(&rb.h));
    XT_RB(rocblas_set_stream(rb.h, s));
    XT_RB(rocblas_set_pointer_mode(rb.h, rocblas_pointer_mode_host));
    if (ft > 0) {
        // E_{ft-1} = K_{ft,ft-1} L_{ft-1}^-T = K_{ft,ft-1} D_{ft-1}^T (column-major, D kept
        // column-major in the backward set), in place of the K block; then the Schur
        // complement K_{ft,ft} -= E E^T (lower triangle)
        const double one = 1.0, zero = 0.0, minus = -1.0;
        XT_TRY(E0.reserve(sizeof(double) * bb));
        XT_RB(rocblas_dgemm(rb.h, rocblas_operation_none, rocblas_operation_transpose, b, b, b,
                            &one, Eat(ft - 1), b, bp.Du[0].as<double>() + (ft - 1) * bb, b, &zero,
                            E0.as<double>(), b));
        XT_HIP(hipMemcpyAsync(Eat(ft - 1), E0.ptr, sizeof(double) * bb, hipMemcpyDeviceToDevice, s));
        XT_RB(rocblas_dsyrk(rb.h, rocblas_fill_lower, rocblas_operation_none, b, b, &minus,
                            Eat(ft - 1), b, &one, Lat(ft), b));
    }
    // L_ii, E_i = K_{i+1,i} L_ii^-T and K_{i+1,i+1} -= E_i E_i^T, panel by panel, block st
    // of both chains at once; the last bottom block's update of the middle block goes to Km
    // (both chains may end in the same launch)
    int *ip = info.as<int>();
    const long long wsize = 2LL * (b / kCT) * kCT * kCT;
    XT_TRY(Wb.reserve(sizeof(double) * 4 * wsize));
    CholRun run[2];
    for (int sd = 0; sd < 2; ++sd)
        for (int h = 0; h < 2; ++h) run[sd].W[h] = Wb.as<double>() + (2 * sd + h) * wsize;
    if (nbt > 0) {
        XT_TRY(Km.reserve(sizeof(double) * bb));
        XT_TRY(zero_fill(Km.as<double>(), bb, s));
    }
    CholSide last;
    for (int st = 0; st < std::max(nt - ft, nbt); ++st) {
        CholSide blk[2];
        CholRun *rn[2];
        int n = 0;
        if (ft + st < nt) {
            blk[n].L = Lat(ft + st);
            blk[n].E = Eat(ft + st);
            blk[n].Kn = Lat(ft + st + 1);
            blk[n].info = ip + ft + st;
            rn[n++] = &run[0];
        }
        if (st < nbt) {
            const int beta = nt + 1 + st;
            blk[n].L = Lat(beta);
            blk[n].E = Eat(nt + st);
            blk[n].Kn = st + 1 < nbt ? Lat(beta + 1) : Km.as<double>();
            blk[n].info = ip + beta;
            last = blk[n];
            rn[n++] = &run[1];
        }
        XT_TRY(factor_blocks(b, blk, rn, n, s));
    }
    if (nbt > 0) {
        XT_TRY(factor_flush(b, last, run[1], s));
        hipLaunchKernelGGL(add_block_kernel, dim3(std::min<long long>(ceil_div(bb, 256), 4096)),
                           dim3(256), 0, s, bb, Km.as<const double>(), Lat(nt));
    }
    {
        CholSide mid;
        mid.L = Lat(nt);
        mid.info = ip + nt;
        CholRun *rn[1] = {&run[0]};
        XT_TRY(factor_blocks(b, &mid, rn, 1, s));
        XT_TRY(factor_flush(b, mid, run[0], s));
    }
    std::vector<int> hinfo(nb + 1);
    XT_HIP(hipMemcpyAsync(hinfo.data(), ip, sizeof(int) * nb, hipMemcpyDeviceToHost, s));
    XT_HIP(hipStreamSynchronize(s));
    for (int e = ft; e < nb; ++e) {   // the chains, then the middle block
        const int i = e < nt ? e : e + 1 < nb ? e + 1 : nt;
        if (hinfo[i] != 0) {   // (the bottom chain's rows run backwards)
            const int r = i * b + hinfo[i] - 1;
            set_error("K is not positive definite (elimination of row %d)",
                      i <= nt ? r : (nt + 1 + nb) * b - 1 - r);
            return XT_E_SINGULAR;
        }
    }
    // nothing can fail numerically from here on: the new blocks go into the factor's own
    // arrays (a full factorization's into new ones where those are missing or too small,
    // allocated before anything is overwritten); an apply still running on another stream
    // is waited for
    const bool full = ft == 0;
    int nlev = bp.nlev;
    DevBuf fresh[4 + 2 * kLevels];
    DevBuf *sets[4 + 2 * kLevels];
    size_t bytes[4 + 2 * kLevels] = {};
    for (int k = 0; k < 4 + 2 * kLevels; ++k)
        sets[k] = k == 0 ? bp.Dl : k == 1 ? bp.Du : k == 2 ? bp.G : k == 3 ? bp.H
                : bp.Lv[(k - 4) / kLevels][(k - 4) % kLevels];
    if (full) {
        // the levels that pay for the fewest columns (more columns use fewer of them);
        // XT_TUNE_BAND_LEVELS v: v - 1 levels (set before the factor is built)
        const int kn = tune_knob(XT_TUNE_BAND_LEVELS), maxlev = kn ? kn - 1 : kLevels;
        nlev = 0;
        while (nlev < maxlev && (nt >> (nlev + 1)) >= kMinChain) ++nlev;
        if (!kn) nlev = std::max(chain_levels(bp, nlev, 16, 8), chain_levels(bp, nlev, 16, 4));
        bytes[0] = bytes[1] = sizeof(double) * bb * nb;
        bytes[2] = bytes[3] = sizeof(double) * bk * (nb - 1);
        for (int dir = 0; dir < 2; ++dir)
            for (int l = 1; l <= nlev; ++l)
                bytes[4 + dir * kLevels + l - 1] = sizeof(double) * rc * (size_t)kw *
                    ((bp.steps(0, dir) >> l) + (bp.steps(1, dir) >> l));
        for (int k = 0; k < 4 + 2 * kLevels; ++k)
            if (bytes[k] > sets[k][0].bytes) XT_TRY(fresh[k].reserve(bytes[k]));
    }
    XT_HIP(hipDeviceSynchronize());
    auto dst = [&](int k) { return fresh[k].ptr ? fresh[k].as<double>() : sets[k][0].as<double>(); };
    double *Dlp = dst(0), *Dup = dst(1), *Gp = dst(2), *Hp = dst(3);
    // D_i = L_ii^-1: column-major lower = D_i^T row-major, the backward set, and row-major
    const int ntl = b / kCT;
    for (int d = 0; d < ntl; ++d)
        hipLaunchKernelGGL(tri_inverse_kernel, dim3(d == 0 ? ntl * (ntl + 1) / 2 : ntl - d, nr),
                           dim3(256), 0, s, b, ntl, d, (const double *)Lp, Dup + ft * bb,
                           Dlp + ft * bb);
    XT_HIP(hipGetLastError());
    auto Dat = [&](int beta) { return Dup + beta * bb; };
    // top chain: G_i from E_{ft-1} (with the new D_ft) on, H_i from block ft on; bottom chain:
    // all, its last block coupled to the middle block by the middle's last rows
    XT_TRY(g_products(rb.h, bp, Eat(e0), 0, Dat(e0 + 1), Gp + e0 * bk, nt - e0));
    XT_TRY(h_products(rb.h, bp, Eat(ft), 0, Dat(ft), Hp + ft * bk, nt - ft));
    XT_TRY(g_products(rb.h, bp, Eat(nt), 0, Dat(nt + 2), Gp + nt * bk, nbt - 1));
    XT_TRY(h_products(rb.h, bp, Eat(nt), 0, Dat(nt + 1), Hp + nt * bk, nbt - 1));
    if (nbt > 0) {
        XT_TRY(g_products(rb.h, bp, Eat(nb - 2), b - kw, Dat(nt), Gp + (nb - 2) * bk, 1));
        XT_TRY(h_products(rb.h, bp, Eat(nb - 2), b - kw, Dat(nb - 1), Hp + (nb - 2) * bk, 1));
    }
    // first changed stored entry of the top chain's levels: forward entries whose G range
    // reaches index ft - 1, backward entries whose H range reaches block ft
    int first[2][kLevels + 1] = {};
    for (int dir = 0; dir < 2; ++dir)
        for (int l = 1; l <= nlev; ++l) {
            const int cnt = bp.steps(0, dir) >> l;
            if (ft > 0)
                first[dir][l] = dir == 0 ? std::min(cnt, (ft - 1) >> l)
                                         : std::max(0, cnt - 1 - ((nt - 1 - ft) >> l));
            if (ft > 0 && dir == 1 && ft >= nt) first[dir][l] = cnt;   // no changed H
            const double *below = l == 1 ? (dir == 0 ? Gp : Hp) : dst(4 + dir * kLevels + l - 2);
            double *out = dst(4 + dir * kLevels + l - 1);
            XT_TRY(level_products(rb.h, bp, 0, dir, l, first[dir][l], cnt, below, out));
            XT_TRY(level_products(rb.h, bp, 1, dir, l, 0, bp.steps(1, dir) >> l, below, out));
        }
    if (!full) {
        XT_TRY(to_f32_range(bp.Du, ft * bb, bb * nr, s));
        XT_TRY(to_f32_range(bp.Dl, ft * bb, bb * nr, s));
        XT_TRY(to_f32_range(bp.G, e0 * bk, bk * (nb - 1 - e0), s));
        XT_TRY(to_f32_range(bp.H, ft * bk, bk * (nb - 1 - ft), s));
        for (int dir = 0; dir < 2; ++dir)
            for (int l = 1; l <= nlev; ++l) {
                const long long es = (long long)rc * kw, off = first[dir][l] * es;
                const long long n = es * ((bp.steps(0, dir) >> l) + (bp.steps(1, dir) >> l));
                XT_TRY(to_f32_range(bp.Lv[dir][l - 1], off, n - off, s));
            }
        XT_HIP(hipStreamSynchronize(s));
        band.ok = true;
        return XT_OK;
    }
    band.ok = true;
    bp.nlev = nlev;
    for (int k = 0; k < 4 + 2 * kLevels; ++k) {
        if (fresh[k].ptr) sets[k][0] = std::move(fresh[k]);
        if (bytes[k] == 0) continue;
        XT_TRY(sets[k][1].reserve(bytes[k] / 2));
        XT_TRY(to_f32_range(sets[k], 0, (long long)(bytes[k] / sizeof(double)), s));
    }
    XT_HIP(hipStreamSynchronize(s));
    if (!bp.keep64)
        for (DevBuf *set : sets) set[0].release();
    bp.built = true;
    return XT_OK;
}

// Host CSR: uploaded, then assembled into the blocks on the device (a few % of their bytes).
static int factor(BandPrec &bp, const int *ia, const int *ja, const double *a, hipStream_t s) {
    const long long nnz = ia[bp.p] - 1;
    DevBuf dia, dja, da;
    XT_TRY(dia.upload(ia, sizeof(int) * (bp.p + 1), s));
    XT_TRY(dja.upload(ja, sizeof(int) * nnz, s));
    XT_TRY(da.upload(a, sizeof(double) * nnz, s));
    return factor_dev(bp, dia.as<int>(), dja.as<int>(), da.as<double>(), s);
}

// Refactor with new values of a K whose lower-triangle pattern fits the existing band
// (the same mesh, e.g. new material or boundary conditions), CSR in device memory.
// first_row > 0: K is unchanged in rows and columns before first_row (0-based), and the
// blocks before first_row / b are kept (a factor without FP64 sets is refactored whole).
int band_refactor(BandPrec *bp, const int *dia, const int *dja, const double *da,
                  hipStream_t s, int first_row) {
    const int fb = first_row > 0 ? std::min(first_row / bp->b, bp->nb) : 0;
    return factor_dev(*bp, dia, dja, da, s, fb);
}

int band_build(int p, const int *ia, const int *ja, const double *a, int block, BandPrec **out,
               bool keep64) {
    XT_ARG(p > 0 && ia && ja && a && out, "band prec arguments");
    XT_ARG(ia[0] == 1, "CSR must be 1-based");
    int bw = 0;
    for (int i = 0; i < p; ++i) XT_ARG(ia[i + 1] >= ia[i], "CSR row pointers must not decrease");
    for (int i = 0; i < p; ++i)
        for (int k = ia[i] - 1; k < ia[i + 1] - 1; ++k) {
            const int j = ja[k] - 1;
            XT_ARG(j >= 0 && j < p, "column index out of range");
            if (j <= i) bw = std::max(bw, i - j);
        }
    int b = std::max(std::max(block, bw), 64);
    b = (b + 63) / 64 * 64;
    if (b > 4096) {
        set_error("bandwidth %d exceeds the supported block size 4096 (renumber the mesh)", bw);
        return XT_E_UNSUPPORTED;
    }
    const int nb = (p + b - 1) / b;
    // only the lower triangle is read (K symmetric); b >= bandwidth puts every lower
    // entry in a diagonal block or the sub-diagonal block below it
    BandPrec *bp = new (std::nothrow) BandPrec;
    if (!bp) return XT_E_NOMEM;
    bp->p = p;
    bp->b = b;
    bp->nb = nb;
    bp->bw = bw;
    bp->nt = nb / 2;
    bp->nbt = (nb - 1) / 2;
    set_band(*bp, bw);
    bp->keep64 = keep64;
    hipStream_t s = nullptr;
    int rc = factor(*bp, ia, ja, a, s);
    if (rc != XT_OK) { delete bp; return rc; }
    *out = bp;
    return XT_OK;
}

void band_delete(BandPrec *bp) { delete bp; }

void band_dims(const BandPrec *bp, int *b, int *nb, int *bw) {
    if (b) *b = bp->b;
    if (nb) *nb = bp->nb;
    if (bw) *bw = bp->bw;
}

bool band_has_fp64(const BandPrec *bp) { return bp->keep64; }

long long band_bytes(const BandPrec *bp, bool f32) {
    const long long b = bp->b, n = bp->nb;
    return (f32 ? 4 : 8) * (2 * b * b * n + 2 * b * bp->kw * (n - 1));
}

// x into the sweeps' workspace w (rows in the factor's order, ld columns): the temporal mix
// with minv (NULL: none) of the active cases a < Ra (case cols[a], NULL: a), slot a's q
// columns at a q; the rows past p zero.  n rows and slots from row first on, one thread each.
// Q: the q that is unrolled, 0 for any.  The sums run in the order of temporal_mix.
template <typename T, int Q>
__global__ void __launch_bounds__(256)
band_load_kernel(unsigned n, int first, int p, int split, int total, int R, int q, int Ra,
                 const int *__restrict__ cols, int ld, const T *__restrict__ minv,
                 const T *__restrict__ x, T *__restrict__ w) {
    constexpr int LM = Q ? 256 * Q : 1;
    __shared__ T Ms[LM];                      // the R q x q matrices, R q <= 256
    const bool staged = Q && minv && R * Q <= 256;
    if (staged) {
        for (int e = threadIdx.x; e < R * Q * Q; e += 256) Ms[e] = minv[e];
        __syncthreads();
    }
    const unsigned idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= n) return;
    const unsigned slot_row = idx / (unsigned)Ra;
    const int row = first + (int)slot_row, a = (int)(idx - slot_row * (unsigned)Ra);
    T *o = w + (size_t)row * ld + a * q;
    const int dof = row < split ? row : split + total - 1 - row;
    if (dof >= p) {
        for (int j = 0; j < q; ++j) o[j] = T(0);
        return;
    }
    const int r = cols ? cols[a] : a;
    const T *xr = x + ((size_t)dof * R + r) * q;
    if (!minv) {
        for (int j = 0; j < q; ++j) o[j] = xr[j];
        return;
    }
    if (Q) {
        T v[Q ? Q : 1];
#pragma unroll
        for (int j = 0; j < Q; ++j) v[j] = xr[j];
        const T *m = staged ? Ms + r * Q * Q : minv + (size_t)r * Q * Q;
#pragma unroll
        for (int i = 0; i < Q; ++i) {
            T sum = T(0);
#pragma unroll
            for (int j = 0; j < Q; ++j) sum += m[i * Q + j] * v[j];
            o[i] = sum;
        }
    } else {
        for (int i = 0; i < q; ++i) {
            const T *m = minv + ((size_t)r * q + i) * q;
            T sum = T(0);
            for (int j = 0; j < q; ++j) sum += m[j] * xr[j];
            o[i] = sum;
        }
    }
}

// The workspace's columns back to y: slot a's to case cols[a], zero for the cases listed
// from Ra on (inactive).  n DOFs and cases from DOF first on, one thread each.
template <typename T, int Q>
__global__ void __launch_bounds__(256)
band_store_kernel(unsigned n, int first, int split, int total, int R, int q, int Ra,
                  const int *__restrict__ cols, int ld, const T *__restrict__ w,
                  T *__restrict__ y) {
    const unsigned idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= n) return;
    const unsigned case_dof = idx / (unsigned)R;
    const int dof = first + (int)case_dof, a = (int)(idx - case_dof * (unsigned)R);
    const int row = dof < split ? dof : split + total - 1 - dof;
    T *o = y + ((size_t)dof * R + (cols ? cols[a] : a)) * q;
    const T *v = w + (size_t)row * ld + a * q;
    if (Q) {
        T u[Q ? Q : 1];
#pragma unroll
        for (int j = 0; j < Q; ++j) u[j] = a < Ra ? v[j] : T(0);
#pragma unroll
        for (int j = 0; j < Q; ++j) o[j] = u[j];
    } else {
        for (int j = 0; j < q; ++j) o[j] = a < Ra ? v[j] : T(0);
    }
}

template <typename T>
int band_apply(BandPrec *bp, int R, int q, const T *minv, const T *x, T *y, hipStream_t s,
               int Ra, const int *dcols) {
    const int b = bp->b, nb = bp->nb, nt = bp->nt, nbt = bp->nbt, kw = bp->kw, rc = bp->rc;
    const int pi = sizeof(T) == 4 ? 1 : 0;
    if (pi == 0 && !bp->keep64) {
        set_error("band factor kept in FP32 only: no FP64 sweeps");
        return XT_E_UNSUPPORTED;
    }
    const bool compact = dcols && Ra >= 0 && Ra < R;
    if (compact && Ra == 0) {   // no active case: P^-1 0 = 0
        hipLaunchKernelGGL(fill_zero_kernel<T>, dim3(ceil_div((long long)bp->p * q * R, 256)),
                           dim3(256), 0, s, (long long)bp->p * q * R, y);
        XT_HIP(hipGetLastError());
        return XT_OK;
    }
    if (!compact) {
        Ra = R;
        dcols = nullptr;
    }
    const int c = q * Ra, ld = pad_cols(c);
    // sized for FP64 sweeps when the factor has them, and for all cases, so switching
    // precision or the active set does not reallocate (captured graphs hold these
    // pointers); one block more than the factor's (the bottom chain's view of the middle)
    const size_t es = bp->keep64 ? sizeof(double) : sizeof(T);
    XT_TRY(bp->w1.reserve(es * (size_t)(nb + 1) * b * pad_cols(q * R)));
    XT_TRY(bp->w2.reserve(es * (size_t)(nb + 1) * b * pad_cols(q * R)));
    T *w1 = bp->w1.as<T>(), *w2 = bp->w2.as<T>();
    const int total = nb * b, split = (nt + 1) * b;
    // (a launch holds fewer than 2^32 threads: more rows and cases take several)
    auto in_launches = [](int rows, int cases, auto launch) {
        const long long most = std::max(1LL, (1LL << 31) / cases);   // rows of a launch
        for (long long first = 0; first < rows; first += most)
            launch((int)first, std::min(most, rows - first) * cases);
    };
    in_launches(total, Ra, [&](int first, long long n) {
#define XT_LOAD(Q)                                                                             \
    hipLaunchKernelGGL((band_load_kernel<T, Q>), dim3(ceil_div(n, 256)), dim3(256), 0, s,       \
                       (unsigned)n, first, bp->p, split, total, R, q, Ra, dcols, ld, minv, x, w1)
        if (q == 6) XT_LOAD(6);
        else if (q == 3) XT_LOAD(3);
        else XT_LOAD(0);
#undef XT_LOAD
    });
    XT_HIP(hipGetLastError());
    const long long bb = (long long)b * b, bk = (long long)b * kw, bc = (long long)b * ld;
    const T *Dl = bp->Dl[pi].as<T>(), *Du = bp->Du[pi].as<T>();
    const T *G = bp->G[pi].as<T>(), *H = bp->H[pi].as<T>();
    // pairing levels used by this apply (XT_TUNE_BAND_PAIR: 1 none, 2 all of the factor's)
    const int pk = tune_knob(XT_TUNE_BAND_PAIR);
    const int nlev = pk == 1 ? 0 : pk == 2 ? bp->nlev : chain_levels(*bp, bp->nlev, ld, sizeof(T));
    // Both chains' recurrences in step coordinates: block v of side sd at W0 + v S, its
    // step's level-L matrix at Mb[L] + (v - 1) MS[L].
    auto chain = [&](int dir, T *w, const T *M0, hipStream_t st) -> int {
        T *W0[2];
        long long S;
        const T *Mb[2][kLevels + 1];
        long long MS[kLevels + 1];
        int m[2];
        const LevelView v0 = level_view(*bp, 0, dir, 0);
        const long long vo = (long long)v0.vrow * ld, oo = (long long)v0.crow * ld;
        S = dir == 0 ? bc : -bc;
        for (int sd = 0; sd < 2; ++sd) {
            m[sd] = bp->steps(sd, dir);
            W0[sd] = w + (dir == 0 ? (sd == 0 ? 0 : nt + 1) : (sd == 0 ? nt : nb)) * bc;
            for (int L = 0; L <= nlev; ++L) {
                const LevelView v = level_view(*bp, sd, dir, L);
                // (a chain without forward steps has one stored G, for the middle block)
                const T *arr = L == 0 ? M0 : bp->Lv[dir][L - 1][pi].as<T>();
                Mb[sd][L] = arr + v.base + (dir == 0 ? 0 : (v.cnt - 1) * v.es) + (long long)v.crow * kw;
                MS[L] = dir == 0 ? v.es : -v.es;
            }
        }
        // items of both chains: a0 + i as, V = block v0 + i vs, O = block o0 + i vs
        auto launch = [&](int L, long long a0, long long as, long long vb, long long ob,
                          long long str, int cnt0, int cnt1) -> int {
            Items<T> it;
            const int cn[2] = {std::max(0, cnt0), std::max(0, cnt1)};
            for (int sd = 0; sd < 2; ++sd) {
                it.A[sd] = Mb[sd][L] + a0 * MS[L];
                it.as[sd] = as * MS[L];
                it.V[sd] = W0[sd] + vb * S + vo;
                it.O[sd] = W0[sd] + ob * S + oo;
                it.vs[sd] = it.os[sd] = str * S;
            }
            it.n0 = cn[0];
            it.n = cn[0] + cn[1];
            return launch_prod<T>(it, rc, kw, kw, 0, c, ld, true, 1, st);
        };
        for (int L = 0; L < nlev; ++L) {   // even steps of level L: the next level's rhs
            const long long d = 1LL << L;
            XT_TRY(launch(L, 1, 2, d, 2 * d, 2 * d, (m[0] >> L) / 2, (m[1] >> L) / 2));
        }
        const long long D = 1LL << nlev;   // the dependent chain of the top level
        for (int v = 1; v <= (std::max(m[0], m[1]) >> nlev); ++v)
            XT_TRY(launch(nlev, v - 1, 0, (v - 1) * D, v * D, 0, v <= (m[0] >> nlev),
                          v <= (m[1] >> nlev)));
        for (int L = nlev - 1; L >= 0; --L) {   // odd steps of level L, from the finished ones
            const long long d = 1LL << L;
            XT_TRY(launch(L, 0, 2, 0, d, 2 * d, ((m[0] >> L) + 1) / 2, ((m[1] >> L) + 1) / 2));
        }
        if (rc < b) {   // the rows no step reads
            Items<T> it;
            const int r0 = dir == 0 ? 0 : rc;
            for (int sd = 0; sd < 2; ++sd) {
                it.A[sd] = Mb[sd][0] + (long long)(r0 - v0.crow) * kw;
                it.as[sd] = MS[0];
                it.V[sd] = W0[sd] + vo;
                it.O[sd] = W0[sd] + S + (long long)r0 * ld;
                it.vs[sd] = it.os[sd] = S;
            }
            it.n0 = m[0];
            it.n = m[0] + m[1];
            XT_TRY(launch_prod<T>(it, b - rc, kw, kw, 0, c, ld, true, 1, st));
        }
        return XT_OK;
    };
    auto diagonal = [&](int tri, const T *D, const T *v, T *o, hipStream_t st) -> int {
        Items<T> it = {{D, D}, {v, v}, {o, o}, {bb, bb}, {bc, bc}, {bc, bc}, nb, nb};
        if (tri == 2 && nbt > 0) {   // the bottom chain starts from the middle block's last rows
            it.dup = o + nb * bc;
            it.dupz = nt;
            it.dup0 = b - kw;
        }
        return launch_prod<T>(it, b, b, b, tri, c, ld, false, 1, st);
    };
    auto sweeps = [&](hipStream_t st) -> int {
        // forward: w2 = D w1 (all blocks), the chains, then the middle block from both
        XT_TRY(diagonal(1, Dl, w1, w2, st));
        XT_TRY(chain(0, w2, G, st));
        if (nt > 0) {
            const long long vo = (long long)(b - kw) * ld;
            Items<T> it = {{G + (nt - 1) * bk, G + (nb - 2) * bk},
                           {w2 + (nt - 1) * bc + vo, w2 + (nb - 1) * bc + vo},
                           {w2 + nt * bc, w2 + nt * bc}, {0, 0}, {0, 0}, {0, 0}, 1, 1};
            XT_TRY(launch_prod<T>(it, b, kw, kw, 0, c, ld, true, nbt > 0 ? 2 : 1, st));
        }
        // backward: w1 = D^T w2 (all blocks), then the chains from the middle block
        XT_TRY(diagonal(2, Du, w2, w1, st));
        XT_TRY(chain(1, w1, H, st));
        return XT_OK;
    };
    hipStreamCaptureStatus capst = hipStreamCaptureStatusNone;
    XT_HIP(hipStreamIsCapturing(s, &capst));
    // (inside a caller's capture the sweeps join that graph as plain launches)
    if (graphs_on() && !prof_on(band_kind<T>()) && capst == hipStreamCaptureStatusNone) {
        const void *key[kKey] = {w1, w2, Dl, Du, G, H};
        for (int dir = 0; dir < 2; ++dir)
            for (int L = 0; L < kLevels; ++L) key[6 + dir * kLevels + L] = bp->Lv[dir][L][pi].ptr;
        SweepGraph *g = nullptr;
        for (SweepGraph &cand : bp->graph)
            if (cand.exec && cand.c == c && cand.pi == pi &&
                cand.epoch == tune_epoch() &&
                cand.nl == nlev && cand.kw == kw && cand.rc == rc &&
                std::equal(key, key + kKey, cand.key)) {
                g = &cand;
                break;
            }
        if (!g) {
            if (!bp->cap) XT_HIP(hipStreamCreateWithFlags(&bp->cap, hipStreamNonBlocking));
            g = &bp->graph[bp->next_graph];
            bp->next_graph = (bp->next_graph + 1) % 4;
            if (g->exec) {
                (void)hipGraphExecDestroy(g->exec);
                g->exec = nullptr;
            }
            XT_HIP(hipStreamBeginCapture(bp->cap, hipStreamCaptureModeThreadLocal));
            const int status = sweeps(bp->cap);
            hipGraph_t graph = nullptr;
            const hipError_t e = hipStreamEndCapture(bp->cap, &graph);
            if (status != XT_OK || e != hipSuccess) {
                if (graph) (void)hipGraphDestroy(graph);
                if (status != XT_OK) return status;
                XT_HIP(e);
            }
            const hipError_t ei = hipGraphInstantiate(&g->exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            if (ei != hipSuccess) g->exec = nullptr;
            XT_HIP(ei);
            g->c = c;
            g->pi = pi;
            g->epoch = tune_epoch();
            g->nl = nlev;
            g->kw = kw;
            g->rc = rc;
            std::copy(key, key + kKey, g->key);
        }
        XT_HIP(hipGraphLaunch(g->exec, s));
    } else {
        XT_TRY(sweeps(s));
        // algorithmic work of the apply: the unpaired block recurrences, each factor block
        // read once (D_i, D_i^T as triangles, G_i, H_i: b x kw), each vector block read and
        // written once per product (plus the read of the block it is subtracted from)
        const double tri = (double)b * (b + 1) / 2, gh = (double)b * kw, vb = (double)b * c;
        const double vg = (double)kw * c + 2.0 * vb;
        prof_alg(band_kind<T>(),
                 sizeof(T) * (2.0 * (nb * tri + (nb - 1) * gh) + 2.0 * (2.0 * nb * vb + (nb - 1) * vg)),
                 2.0 * (2.0 * nb * tri * c + 2.0 * (nb - 1) * gh * c));
    }
    XT_HIP(hipGetLastError());
    in_launches(bp->p, R, [&](int first, long long n) {
#define XT_STORE(Q)                                                                            \
    hipLaunchKernelGGL((band_store_kernel<T, Q>), dim3(ceil_div(n, 256)), dim3(256), 0, s,      \
                       (unsigned)n, first, split, total, R, q, Ra, dcols, ld, (const T *)w1, y)
        if (q == 6) XT_STORE(6);
        else if (q == 3) XT_STORE(3);
        else XT_STORE(0);
#undef XT_STORE
    });
    XT_HIP(hipGetLastError());
    return XT_OK;
}
template int band_apply<double>(BandPrec *, int, int, const double *, const double *, double *,
                                hipStream_t, int, const int *);
template int band_apply<float>(BandPrec *, int, int, const float *, const float *, float *,
                               hipStream_t, int, const int *);

}  // namespace xt
