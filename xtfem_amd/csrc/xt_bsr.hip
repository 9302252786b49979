// Node-block Kronecker operator for 3-DOF meshes: Y = alpha (K X A_r^T + M X B_r^T) + beta Y.
//
// Same operator as kronspmv/kronspgemv (kronecker.f90:19-127) for the mechanical
// system, whose spatial matrices are made of 3x3 node-pair blocks (a C3D8 element
// couples all 3 displacement components of its 8 nodes; consistent mass couples
// only equal components, elesubs.f90:51-53, so each M block is diagonal).
//
// Storage ("node slices"): node rows, in their natural order, are packed into
// slices of 64 consecutive nodes.  Inside a slice the entries are aligned by
// neighbour offset: the slice keeps the sorted set of offsets d = m - n that
// occur in any of its rows, and entry e of every slot refers to node n + d_e
// (a zero block where that neighbour is absent).  For a structured mesh the set
// is the 27-point stencil, so at every step the 64 lanes of a wave read 64
// consecutive blocks and gather 64 consecutive rows of X: all wave-wide loads
// are contiguous.  A slice whose offset set would be much longer than its
// longest row (irregular meshes) stores its rows by position instead.  Block e
// of slot k of slice s lives at index base[s] + e*64 + k and holds the 3x3 K
// values (row-major) and the 3 diagonal M values (12 numbers), plus one int32
// column-node index.
//
// Work mapping of the slices: one lane per (node row, load case r), or SPL lanes with the
// entries split between them.  The lane accumulates the 3 rows x 6 temporal columns of
// K X and M X for its node in registers (72 FMA per block), then applies the 6x6
// temporal matrices of its load case in registers and stores its outputs once.  With W
// lanes a node a slice's 64 slots fill W whole waves for any W, so loop bounds are
// wave-uniform without lanes left over.
//
// Storage ("node groups", kron_group_kernel, several load cases on enough nodes): kG
// consecutive nodes share the union of their neighbours; the blocks stand neighbour by
// neighbour (only the couplings that exist), so a wave whose lanes are columns reads each
// neighbour's rows of X once for all nodes of the group.  The order is far nodes, near ones
// (within a third of the way to the lowest neighbour), the group's own, each ascending: the
// kernel adds product by product (the slices a block's three together), and with the large
// diagonal block before half of the products the sums rounded more often than the slices'.
// Error in the 2-norm, random X, against more bits: slices 1.12e-7 (FP32) and 2.1e-16 (FP64),
// groups in sorted order 1.37e-7 and 2.6e-16, in this order 8.1e-8 and 1.5e-16.
// Time of 145323 nodes, 32 cases, FP64: sorted 685 us, so 697 (5 % more of the reads miss the
// L2), own nodes last and the others sorted 722 (FP32 389, 391, 395); 23735 nodes 117, 121,
// 118 (80, 80, 80); a block's three products summed before they are added (error as the
// slices') 715 (430) and 142 (93).
// The values of a precision are copied from the slices by the first apply that takes the
// groups, and kept up to date from then on: a program with one load case never holds them.
//
// The path is for q = 6 temporal functions (three quadratic temporal nodes, each with a
// sine enrichment: 2*nnte, main3d.f90:172).
#include <algorithm>
#include <mutex>
#include <vector>

#include "xt_common.h"

namespace xt {

struct BsrPlan {
    int nn = 0;             // nodes (block rows)
    int nslices = 0;
    long long nblocks = 0;  // stored blocks including padding
    long long nreal = 0;    // blocks without padding
    DevBuf slot_node;       // [nslices*64] node of each slot, -1 for empty slots
    DevBuf slice_base;      // [nslices] first block of each slice
    DevBuf slice_len;       // [nslices] blocks per slot
    DevBuf bcol;            // [nblocks] column node
    DevBuf bval32, bval64;  // [nblocks][12]
    DevBuf kmap, mmap;      // value position in bval of every CSR entry of K and of M
    long long nk = 0, nm = 0;
    // Group form: neighbours gptr[s] .. gptr[s + 1] - 1 of group s as (node, 16 b + mask of the
    // group's nodes it couples to), its blocks from gblk[s] + b on (nodes ascending); gof: group
    // block of each stored block, -1 for padding.  Values ([nreal][12]) by group_values, gmutex
    // held: applies of several threads may be the first.
    int ngroups = 0;
    long long ngnbr = 0;    // neighbours of all groups
    DevBuf gptr, gblk, gnbr, gof, gval32, gval64;
    bool no_gval[2] = {};   // no memory for the FP64 [0], FP32 [1] values: slices instead
    std::mutex gmutex;
    // Staged form: the distinct column nodes of each slice (its neighbour set, sorted),
    // unode[ubase[s] .. ubase[s] + ulen[s]), and for every stored block the position of
    // its column node in that list (uint16), so a workgroup can stage the slice's rows
    // of X in LDS once and read them from there.
    DevBuf unode, ubase, ulen, lidx;
    int umax = 0;           // longest neighbour set (0: no staged form)
};

static constexpr int kSlice = 64;
static constexpr int kG = 4;   // nodes of a group
static constexpr int kTS = 73;   // LDS stride of a case's temporal matrices (odd)

__global__ void __launch_bounds__(256) bsr_zero_kernel(long long n, double *d, float *f) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        d[i] = 0.0;
        f[i] = 0.0f;
    }
}
int bsr_set_values(BsrPlan &P, const double *kv, const double *mv, hipStream_t s);

// Build the node-slice form and the node groups' lists (kv, mv: the CSR values on the
// device); returns XT_E_UNSUPPORTED if K/M are not 3x3-blocked with diagonal M blocks.
int bsr_build(int p, const int *krp, const int *kci, const double *kv, const int *mrp,
              const int *mci, const double *mv, BsrPlan &P) {
    if (p % 3) return XT_E_UNSUPPORTED;
    const int nn = p / 3;
    // M must be block-diagonal per node pair (equal components only)
    for (int i = 0; i < p; ++i)
        for (int e = mrp[i]; e < mrp[i + 1]; ++e)
            if (mci[e] % 3 != i % 3) return XT_E_UNSUPPORTED;
    // block pattern of each node row: union of the column nodes of K and M
    std::vector<std::vector<int>> cols(nn);
    std::vector<int> mark(nn, -1);
    for (int a = 0; a < nn; ++a) {
        std::vector<int> &c = cols[a];
        for (int d = 0; d < 3; ++d) {
            const int i = 3 * a + d;
            for (int e = krp[i]; e < krp[i + 1]; ++e) {
                const int b = kci[e] / 3;
                if (mark[b] != a) { mark[b] = a; c.push_back(b); }
            }
            for (int e = mrp[i]; e < mrp[i + 1]; ++e) {
                const int b = mci[e] / 3;
                if (mark[b] != a) { mark[b] = a; c.push_back(b); }
            }
        }
        std::sort(c.begin(), c.end());
        if (c.empty()) c.push_back(a);  // keep a (zero) block so the row is well formed
    }
    const int nslices = ceil_div(nn, kSlice);
    std::vector<int> slot_node((size_t)nslices * kSlice, -1), base(nslices), len(nslices);
    std::vector<std::vector<int>> offs(nslices);  // aligned offsets (empty: by position)
    long long nb = 0;
    for (int s = 0; s < nslices; ++s) {
        int maxlen = 0;
        std::vector<int> u;
        for (int k = 0; k < kSlice; ++k) {
            const int a = s * kSlice + k;
            if (a >= nn) break;
            slot_node[a] = a;
            maxlen = std::max(maxlen, (int)cols[a].size());
            for (int b : cols[a]) u.push_back(b - a);
        }
        std::sort(u.begin(), u.end());
        u.erase(std::unique(u.begin(), u.end()), u.end());
        if ((int)u.size() * 4 <= maxlen * 5) offs[s] = u;
        len[s] = offs[s].empty() ? maxlen : (int)u.size();
        base[s] = (int)nb;
        nb += (long long)len[s] * kSlice;
    }
    if (nb * 12 > 0x7fffffffLL) return XT_E_UNSUPPORTED;
    std::vector<int> bcol(nb);
    std::vector<int> pos(nn, -1);   // entry of column node b in the row
    std::vector<int> kmap(krp[p]), mmap(mrp[p]), gof(nb, -1);
    // groups: merge the kG sorted neighbour lists, then far, near and own nodes; gpos: block of
    // each of row a's neighbours, from cfirst[a] on
    const int ngroups = ceil_div(nn, kG);
    std::vector<int> gptr(ngroups + 1, 0), gblk(ngroups + 1, 0), gnbr;
    std::vector<int> cfirst(nn + 1, 0);
    for (int a = 0; a < nn; ++a) cfirst[a + 1] = cfirst[a] + (int)cols[a].size();
    std::vector<int> gpos(cfirst[nn]);
    {
        struct Neighbour {
            int m, mask, at[kG];   // column node, coupled nodes of the group, their entries
        };
        std::vector<Neighbour> u;
        int blk = 0;
        for (int s = 0; s < ngroups; ++s) {
            const int a0 = s * kG, na = std::min(kG, nn - a0);
            Neighbour n{};
            u.clear();
            for (;;) {
                n.m = nn;
                for (int i = 0; i < na; ++i)
                    if (n.at[i] < (int)cols[a0 + i].size())
                        n.m = std::min(n.m, cols[a0 + i][n.at[i]]);
                if (n.m == nn) break;
                n.mask = 0;
                for (int i = 0; i < na; ++i)
                    if (n.at[i] < (int)cols[a0 + i].size() && cols[a0 + i][n.at[i]] == n.m)
                        n.mask |= 1 << i;
                u.push_back(n);
                for (int i = 0; i < na; ++i) n.at[i] += n.mask >> i & 1;
            }
            gblk[s] = blk;
            const int third = std::max(a0 - u[0].m, 0) / 3;
            auto kind = [&](int m) {
                return m >= a0 && m < a0 + na ? 2 : m >= a0 - third && m < a0 + na + third ? 1 : 0;
            };
            for (int k = 0; k < 3; ++k)
                for (const Neighbour &v : u) {
                    if (kind(v.m) != k) continue;
                    gnbr.push_back(v.m);
                    gnbr.push_back((blk - gblk[s]) << 4 | v.mask);
                    for (int i = 0; i < na; ++i)
                        if (v.mask >> i & 1) gpos[cfirst[a0 + i] + v.at[i]] = blk++;
                }
            gptr[s + 1] = (int)(gnbr.size() / 2);
        }
        gblk[ngroups] = blk;
    }
    long long nreal = 0;
    std::vector<int> klast(p, -1), mlast(p, -1);   // last entry of a column (of this row: >= its first)
    for (int s = 0; s < nslices; ++s)
        for (int k = 0; k < kSlice; ++k) {
            const int a = s * kSlice + k;
            const int L = len[s];
            if (a >= nn) {
                for (int e = 0; e < L; ++e) bcol[(long long)base[s] + (long long)e * kSlice + k] = 0;
                continue;
            }
            const std::vector<int> &c = cols[a];
            nreal += (long long)c.size();
            for (int e = 0; e < L; ++e) {
                const long long idx = (long long)base[s] + (long long)e * kSlice + k;
                if (!offs[s].empty()) {
                    // aligned slot: neighbour a + d_e, clamped into range when absent
                    const int m = a + offs[s][e];
                    bcol[idx] = std::min(std::max(m, 0), nn - 1);
                } else {
                    bcol[idx] = e < (int)c.size() ? c[e] : a;
                }
            }
            // entry index of every real neighbour
            if (!offs[s].empty()) {
                for (int b : c) {
                    const int e = (int)(std::lower_bound(offs[s].begin(), offs[s].end(), b - a) -
                                        offs[s].begin());
                    pos[b] = e;
                }
            } else {
                for (int e = 0; e < (int)c.size(); ++e) pos[c[e]] = e;
            }
            for (int e = 0; e < (int)c.size(); ++e)
                gof[(long long)base[s] + (long long)pos[c[e]] * kSlice + k] = gpos[cfirst[a] + e];
            for (int d = 0; d < 3; ++d) {
                const int i = 3 * a + d;
                for (int e = krp[i]; e < krp[i + 1]; ++e) {
                    const int b = kci[e] / 3, cd = kci[e] % 3;
                    const long long idx = (long long)base[s] + (long long)pos[b] * kSlice + k;
                    kmap[e] = (int)(idx * 12 + d * 3 + cd);
                    if (klast[kci[e]] >= krp[i]) kmap[klast[kci[e]]] = -1;   // the last one stands
                    klast[kci[e]] = e;
                }
                for (int e = mrp[i]; e < mrp[i + 1]; ++e) {
                    const int b = mci[e] / 3;
                    const long long idx = (long long)base[s] + (long long)pos[b] * kSlice + k;
                    mmap[e] = (int)(idx * 12 + 9 + d);
                    if (mlast[mci[e]] >= mrp[i]) mmap[mlast[mci[e]]] = -1;
                    mlast[mci[e]] = e;
                }
            }
            for (int b : c) pos[b] = -1;
        }
    // staged form: per slice the sorted distinct column nodes and each block's position
    {
        std::vector<int> unode, ub(nslices), ul(nslices);
        std::vector<unsigned short> li(nb);
        int umax = 0;
        bool ok = true;
        std::vector<int> tmp;
        for (int sl = 0; sl < nslices && ok; ++sl) {
            const long long b0 = base[sl], b1 = b0 + (long long)len[sl] * kSlice;
            tmp.assign(bcol.begin() + b0, bcol.begin() + b1);
            std::sort(tmp.begin(), tmp.end());
            tmp.erase(std::unique(tmp.begin(), tmp.end()), tmp.end());
            if (tmp.size() > 65535) { ok = false; break; }
            ub[sl] = (int)unode.size();
            ul[sl] = (int)tmp.size();
            umax = std::max(umax, (int)tmp.size());
            for (long long i = b0; i < b1; ++i)
                li[i] = (unsigned short)(std::lower_bound(tmp.begin(), tmp.end(), bcol[i]) -
                                         tmp.begin());
            unode.insert(unode.end(), tmp.begin(), tmp.end());
        }
        if (ok && !unode.empty()) {
            XT_TRY(P.unode.upload(unode.data(), sizeof(int) * unode.size()));
            XT_TRY(P.ubase.upload(ub.data(), sizeof(int) * nslices));
            XT_TRY(P.ulen.upload(ul.data(), sizeof(int) * nslices));
            XT_TRY(P.lidx.upload(li.data(), sizeof(unsigned short) * nb));
            P.umax = umax;
        }
    }
    P.nn = nn;
    P.nslices = nslices;
    P.nblocks = nb;
    P.nreal = nreal;
    XT_TRY(P.slot_node.upload(slot_node.data(), sizeof(int) * slot_node.size()));
    XT_TRY(P.slice_base.upload(base.data(), sizeof(int) * nslices));
    XT_TRY(P.slice_len.upload(len.data(), sizeof(int) * nslices));
    XT_TRY(P.bcol.upload(bcol.data(), sizeof(int) * nb));
    P.nk = krp[p];
    P.nm = mrp[p];
    if (P.nk) XT_TRY(P.kmap.upload(kmap.data(), sizeof(int) * P.nk));
    if (P.nm) XT_TRY(P.mmap.upload(mmap.data(), sizeof(int) * P.nm));
    XT_TRY(P.gof.upload(gof.data(), sizeof(int) * nb));
    P.ngroups = ngroups;
    P.ngnbr = gptr[ngroups];
    XT_TRY(P.gptr.upload(gptr.data(), sizeof(int) * gptr.size()));
    XT_TRY(P.gblk.upload(gblk.data(), sizeof(int) * gblk.size()));
    XT_TRY(P.gnbr.upload(gnbr.data(), sizeof(int) * gnbr.size()));
    // the values, from the CSR values already on the device
    const long long nv = nb * 12;
    XT_TRY(P.bval64.reserve(sizeof(double) * nv));
    XT_TRY(P.bval32.reserve(sizeof(float) * nv));
    hipLaunchKernelGGL(bsr_zero_kernel, dim3(ceil_div(nv, 256)), dim3(256), 0, 0, nv,
                       P.bval64.as<double>(), P.bval32.as<float>());
    XT_HIP(hipGetLastError());
    XT_TRY(bsr_set_values(P, kv, mv, 0));
    XT_HIP(hipDeviceSynchronize());
    return XT_OK;
}

template <typename T> struct Vec2;
template <> struct Vec2<float> { using type = float2; };
template <> struct Vec2<double> { using type = double2; };

// 12 block values (3x3 K + diagonal M) with 16-byte loads.  (Non-temporal loads
// were measured 40% slower here on gfx950 and are not used.)
typedef float xt_f4 __attribute__((ext_vector_type(4)));
typedef double xt_d2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void load_block(const float *bv, float *kv) {
    const xt_f4 *p = reinterpret_cast<const xt_f4 *>(bv);
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        const xt_f4 v = p[t];
        kv[4 * t + 0] = v.x;
        kv[4 * t + 1] = v.y;
        kv[4 * t + 2] = v.z;
        kv[4 * t + 3] = v.w;
    }
}
__device__ __forceinline__ void load_block(const double *bv, double *kv) {
    const xt_d2 *p = reinterpret_cast<const xt_d2 *>(bv);
#pragma unroll
    for (int t = 0; t < 6; ++t) {
        const xt_d2 v = p[t];
        kv[2 * t + 0] = v.x;
        kv[2 * t + 1] = v.y;
    }
}

// Workgroups are dealt to the 8 XCDs round-robin (workgroup b runs on XCD b % 8);
// renumber them so each XCD walks one contiguous eighth of the node range and its
// L2 holds that range's neighbour band of X.  The grid is a multiple of 8, which
// makes the renumbering a permutation of [0, grid).
__device__ __forceinline__ long long xcd_block(long long b, long long grid) {
    const long long per = grid / 8;
    return (b % 8) * per + b / 8;
}

// W: lanes per node, from the load cases of this launch on (R: past its last one, <= 64 of
// them), inv = ceil(2^31 / W); UNR: entries per pass (loads in flight).  Bound by the vector
// cache, whose load instructions cost the same for idle lanes, so W is the cases themselves
// and not the power of two above them.  W = power of two / cases, us:
//   4879 nodes, FP64  9 cases 29 / 20, 12: 30 / 24, 17: 57 / 37, 28: 59 / 57
//  13237 nodes, FP32  5 cases 21 / 19, 9: 40 / 28, 12: 41 / 33, 17: 77 / 47, 28: 79 / 71
// One lane below a power of two is the exception (slice_lanes).
template <typename T, int UNR>
__global__ void __launch_bounds__(256)
kron_bsr3_kernel(int nslices, const int *__restrict__ slot_node,
                 const int *__restrict__ slice_base, const int *__restrict__ slice_len,
                 const int *__restrict__ bcol, const T *__restrict__ bval, int W,
                 unsigned inv, int R, int r0, int c, const T *__restrict__ tmat, T alpha,
                 T beta, const T *__restrict__ x, T *__restrict__ y) {
    using V2 = typename Vec2<T>::type;
    // Lane f of the slice's 64 W: slot f / W, case f % W.  The quotients by inv are exact
    // below 2^31 / W for any W, below 2^31 for a power of two; with W not one, 2^25 waves
    // would need vectors of more than the card's memory.  The wave stays a vector value: with
    // s and its loop in scalar registers FP64 took 2 to 4% more.
    const int lane = threadIdx.x & 63;
    const int wave = (int)xcd_block(blockIdx.x, gridDim.x) * (int)(blockDim.x >> 6) +
                     (int)(threadIdx.x >> 6);
    const int s = (int)__umulhi(2u * (unsigned)wave, inv);
    if (s >= nslices) return;
    const int f = (wave - s * W) * 64 + lane, k = (int)__umulhi(2u * (unsigned)f, inv);
    const int r = r0 + (f - k * W);
    const int node = slot_node[s * kSlice + k];
    const bool act = node >= 0 && r < R;
    const int L = slice_len[s];
    const long long b0 = slice_base[s];
    T aK[3][6], aM[3][6];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) { aK[i][j] = T(0); aM[i][j] = T(0); }
    const int rc = act ? r * 6 : 0;
    // UNR entries per pass: their column indices, blocks and X rows are all loaded
    // before the products, so one pass costs two dependent memory latencies (column
    // index, then X) instead of two per entry.
    auto accumulate = [&](const T (&kv)[12], const T (&xv)[3][6]) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                aK[i][j] += kv[3 * i + 0] * xv[0][j] + kv[3 * i + 1] * xv[1][j] + kv[3 * i + 2] * xv[2][j];
                aM[i][j] += kv[9 + i] * xv[i][j];
            }
    };
    auto gather = [&](int m, T (&xv)[3][6]) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const T *xr = x + (size_t)(3 * m + d) * c + rc;
#pragma unroll
            for (int j = 0; j < 6; j += 2) {
                const V2 v = *reinterpret_cast<const V2 *>(xr + j);
                xv[d][j] = v.x;
                xv[d][j + 1] = v.y;
            }
        }
    };
    int e = 0;
    for (; e + UNR <= L; e += UNR) {
        int m[UNR];
        T kv[UNR][12], xv[UNR][3][6];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const long long idx = b0 + (long long)(e + u) * kSlice + k;
            m[u] = bcol[idx];
            load_block(bval + idx * 12, kv[u]);
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) gather(m[u], xv[u]);
#pragma unroll
        for (int u = 0; u < UNR; ++u) accumulate(kv[u], xv[u]);
    }
    for (; e < L; ++e) {
        const long long idx = b0 + (long long)e * kSlice + k;
        T kv[12], xv[3][6];
        load_block(bval + idx * 12, kv);
        gather(bcol[idx], xv);
        accumulate(kv, xv);
    }
    if (!act) return;
    const T *TA = tmat + (size_t)(r * 2 + 0) * 36;
    const T *TB = tmat + (size_t)(r * 2 + 1) * 36;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        T out[6];
#pragma unroll
        for (int o = 0; o < 6; ++o) {
            T sacc = T(0);
#pragma unroll
            for (int j = 0; j < 6; ++j) sacc += TA[o * 6 + j] * aK[i][j] + TB[o * 6 + j] * aM[i][j];
            out[o] = sacc;
        }
        T *yr = y + (size_t)(3 * node + i) * c + rc;
#pragma unroll
        for (int o = 0; o < 6; o += 2) {
            V2 v;
            if (beta == T(0)) {
                v.x = alpha * out[o];
                v.y = alpha * out[o + 1];
            } else {
                const V2 old = *reinterpret_cast<const V2 *>(yr + o);
                v.x = alpha * out[o] + beta * old.x;
                v.y = alpha * out[o + 1] + beta * old.y;
            }
            *reinterpret_cast<V2 *>(yr + o) = v;
        }
    }
}

// Staged variant for many load cases: one workgroup per (slice, chunk of CC columns =
// CC/6 load cases).  The workgroup first copies the rows of X of the slice's neighbour
// nodes, restricted to its columns, into LDS (16-byte loads; each row of X is read once
// per slice instead of once per neighbouring node row), then thread (slot k, case rl)
// walks the slot's entries reading the block values from memory (consecutive slots
// consecutive) and the neighbour's X rows from LDS through the block's position in the
// neighbour list.  Same products and summation order as kron_bsr3_kernel.
template <typename T, int CC>
__global__ void __launch_bounds__(64 * (CC / 6))
kron_bsr3_lds_kernel(int nslices, int nch, const int *__restrict__ slot_node,
                     const int *__restrict__ slice_base, const int *__restrict__ slice_len,
                     const int *__restrict__ unode, const int *__restrict__ ubase,
                     const int *__restrict__ ulen, const unsigned short *__restrict__ lidx,
                     const T *__restrict__ bval, int c, const T *__restrict__ tmat, T alpha,
                     T beta, const T *__restrict__ x, T *__restrict__ y) {
    using V2 = typename Vec2<T>::type;
    constexpr int VEC = 16 / sizeof(T);
    typedef T vec_t __attribute__((ext_vector_type(VEC)));
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T *xs = reinterpret_cast<T *>(smem_raw);          // [u][3][CC]
    const long long blk = xcd_block(blockIdx.x, gridDim.x);
    const int s = (int)(blk / nch), ch = (int)(blk - (long long)s * nch);
    if (s >= nslices) return;                           // (grid padded to a multiple of 8)
    const int col0 = ch * CC;
    const int U = ulen[s];
    const int *un = unode + ubase[s];
    constexpr int RPN = 3 * CC / VEC;                   // vector loads per neighbour node
    for (int t = threadIdx.x; t < U * RPN; t += blockDim.x) {
        const int u = t / RPN, v = t - u * RPN;
        const int d = v / (CC / VEC), cv = v - d * (CC / VEC);
        *reinterpret_cast<vec_t *>(xs + ((size_t)u * 3 + d) * CC + cv * VEC) =
            *reinterpret_cast<const vec_t *>(x + ((size_t)un[u] * 3 + d) * c + col0 + cv * VEC);
    }
    __syncthreads();
    const int k = threadIdx.x & 63, rl = threadIdx.x >> 6;
    const int r = ch * (CC / 6) + rl;
    const int node = slot_node[(size_t)s * kSlice + k];
    const int L = slice_len[s];
    const long long b0 = slice_base[s];
    T aK[3][6], aM[3][6];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) { aK[i][j] = T(0); aM[i][j] = T(0); }
    constexpr int UNR = 4;
    int e = 0;
    auto step = [&](const T (&kv)[12], int li) {
        T xv[3][6];
        const T *xr = xs + (size_t)li * 3 * CC + rl * 6;
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int j = 0; j < 6; j += 2) {
                const V2 v = *reinterpret_cast<const V2 *>(xr + d * CC + j);
                xv[d][j] = v.x;
                xv[d][j + 1] = v.y;
            }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                aK[i][j] += kv[3 * i + 0] * xv[0][j] + kv[3 * i + 1] * xv[1][j] + kv[3 * i + 2] * xv[2][j];
                aM[i][j] += kv[9 + i] * xv[i][j];
            }
    };
    for (; e + UNR <= L; e += UNR) {
        T kv[UNR][12];
        int li[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const long long idx = b0 + (long long)(e + u) * kSlice + k;
            li[u] = lidx[idx];
            load_block(bval + idx * 12, kv[u]);
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) step(kv[u], li[u]);
    }
    for (; e < L; ++e) {
        const long long idx = b0 + (long long)e * kSlice + k;
        T kv[12];
        load_block(bval + idx * 12, kv);
        step(kv, lidx[idx]);
    }
    if (node < 0) return;
    const T *TA = tmat + (size_t)(r * 2 + 0) * 36;
    const T *TB = tmat + (size_t)(r * 2 + 1) * 36;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        T out[6];
#pragma unroll
        for (int o = 0; o < 6; ++o) {
            T sacc = T(0);
#pragma unroll
            for (int j = 0; j < 6; ++j) sacc += TA[o * 6 + j] * aK[i][j] + TB[o * 6 + j] * aM[i][j];
            out[o] = sacc;
        }
        T *yr = y + (size_t)(3 * node + i) * c + r * 6;
#pragma unroll
        for (int o = 0; o < 6; o += 2) {
            V2 v;
            if (beta == T(0)) {
                v.x = alpha * out[o];
                v.y = alpha * out[o + 1];
            } else {
                const V2 old = *reinterpret_cast<const V2 *>(yr + o);
                v.x = alpha * out[o] + beta * old.x;
                v.y = alpha * out[o + 1] + beta * old.y;
            }
            *reinterpret_cast<V2 *>(yr + o) = v;
        }
    }
}

using F4 = float __attribute__((ext_vector_type(4)));

// Value of the neighbouring lane of a pair (2 k, 2 k + 1), by DPP.
static __device__ inline float pair_swap(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}
static __device__ inline double pair_swap(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

// Row I of a node's block times the neighbour's X, three columns: K += the row's three
// values times X, M += its mass value times X's row I.  Lane t of each row of 16 lanes
// holds value t of the block; the row broadcast is part of each multiply-add.  (Two wait
// states stand between a write of kv and its first use by a lane-crossing operand.)
template <int I>
static __device__ inline void block_row(double kv, const double (&x)[3][3], double (&k)[3],
                                        double (&m)[3]) {
#define XT_FMA(acc, val, xv)                                                                   \
    "v_fmac_f64_dpp " acc ", %6, " xv " row_newbcast:" val                                     \
    " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define XT_BLOCK_ROW                                                                     \
    asm("s_nop 1\n\t"                                                                          \
        XT_FMA("%0", "%16", "%7") XT_FMA("%1", "%16", "%8") XT_FMA("%2", "%16", "%9")          \
        XT_FMA("%3", "%19", "%20") XT_FMA("%4", "%19", "%21") XT_FMA("%5", "%19", "%22")       \
        XT_FMA("%0", "%17", "%10") XT_FMA("%1", "%17", "%11") XT_FMA("%2", "%17", "%12")       \
        XT_FMA("%0", "%18", "%13") XT_FMA("%1", "%18", "%14") XT_FMA("%2", "%18", "%15")       \
        : "+&v"(k[0]), "+&v"(k[1]), "+&v"(k[2]), "+&v"(m[0]), "+&v"(m[1]), "+&v"(m[2])               \
        : "v"(kv), "v"(x[0][0]), "v"(x[0][1]), "v"(x[0][2]), "v"(x[1][0]), "v"(x[1][1]),       \
          "v"(x[1][2]), "v"(x[2][0]), "v"(x[2][1]), "v"(x[2][2]), "n"(3 * I), "n"(3 * I + 1),  \
          "n"(3 * I + 2), "n"(9 + I), "v"(x[I][0]), "v"(x[I][1]), "v"(x[I][2]))
    XT_BLOCK_ROW;
#undef XT_FMA
}
template <int I>
static __device__ inline void block_row(float kv, const float (&x)[3][3], float (&k)[3],
                                        float (&m)[3]) {
#define XT_FMA(acc, val, xv)                                                                   \
    "v_fmac_f32_dpp " acc ", %6, " xv " row_newbcast:" val                                     \
    " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
    XT_BLOCK_ROW;
#undef XT_FMA
#undef XT_BLOCK_ROW
}

// Several load cases: 2 lanes per load case (three temporal columns each), so a group of kG
// nodes takes LPG lanes (2 per case, whole rows of 16) and a wave holds 64 / LPG groups
// ("slots").  Each neighbour's rows of X are read once for the group, two neighbours ahead,
// 16 bytes and 8 a lane so that a row costs the address unit 2 instructions of 16 cycles
// (24-byte pieces a lane cost 64 each, 8-byte ones three of 16).  The blocks are staged in
// LDS, CH neighbours (up to CH kG blocks) at a time; a row of 16 lanes reads a block's 12
// values, one a lane, and they enter the multiply-adds by row broadcast.  A wave goes on to
// its next groups, the first chunk of which is loaded during the last of the one before.
//
// 145323 nodes (241 x 201 x 3), 32 cases, FP64: 1704 us by the slice kernel (every lane loads
// its node's block and its neighbours' rows: 15 loads an entry through the CU's vector
// cache), 687 here (699 since each group's own nodes come last).  Block values through scalar
// loads, a column or three a lane: 1460, 1160 (a dependent scalar load a block); by LDS reads
// of 16 bytes at one address: 880; one neighbour ahead, one group a wave: 760.  What is left:
// the rows of X reach a CU at 8.8 TB/s over all CUs with 63 % of them missing the L2 (the
// vector cache waits on about 80 lines of 128 bytes at 660 cycles each), and the clock sinks
// to 1.7 - 1.9 GHz.  Groups taken in strips of the section rather than in order halve the
// misses for 10 % of the time, but need the section's width, which the pattern does not give.
template <typename T, int LPG>
struct GroupGeom {
    static constexpr int CH = LPG >= 48 ? 6 : 3;              // neighbours of a chunk
    static constexpr int PPB = 12 * sizeof(T) / 16;           // 16-byte pieces of a block
    static constexpr int VP = CH * kG * PPB;                  // pieces of a chunk, at most
    static constexpr int NQ = (VP + LPG - 1) / LPG;
    static constexpr int MIX = 18 * LPG * sizeof(T) / 16;     // a node's rows of K X and M X
    static constexpr int SLOT = (VP > MIX ? VP : MIX) + (CH + 3) / 2;
    static constexpr int NS = 64 / LPG;
    static constexpr int BPC = sizeof(T) == 4 ? 3 : 2;        // workgroups a CU
};

template <typename T, int LPG>
__global__ void __launch_bounds__(256, (GroupGeom<T, LPG>::BPC))
kron_group_kernel(int ngroups, int nn, const int *__restrict__ gptr,
                  const int *__restrict__ gblk, const int2 *__restrict__ gnbr,
                  const T *__restrict__ gval, int R, int per, int c,
                  const T *__restrict__ tmat, T alpha, T beta, const T *__restrict__ x,
                  T *__restrict__ y) {
    using G = GroupGeom<T, LPG>;
    constexpr int CH = G::CH, PPB = G::PPB;
    using T2 = T __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    extern __shared__ F4 smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool spare = lane >= G::NS * LPG;      // spare lanes repeat slot 0 and store nothing
    const int slot = spare ? 0 : lane / LPG;
    const int li = spare ? lane - G::NS * LPG : lane - slot * LPG;
    const int r0 = blockIdx.y * per, cc = min(R - r0, per) * 6;   // the chunk's columns
    F4 *sv = smem + (size_t)(wave * G::NS + slot) * G::SLOT;
    int2 *se = (int2 *)(sv + G::SLOT - (CH + 3) / 2);   // CH + 2 entries
    T *st = (T *)(smem + (size_t)4 * G::NS * G::SLOT);            // the chunk's temporal matrices
    // this wave's items of NS groups: each XCD has an eighth of them, its waves side by side
    const int items = (ngroups + G::NS - 1) / G::NS, perx = (items + 7) / 8;
    const int xcd = blockIdx.x & 7, step = (int)(gridDim.x >> 3) * 4;
    const int end = min(items, (xcd + 1) * perx);
    int item = xcd * perx + (int)(blockIdx.x >> 3) * 4 + wave;
    // a slot that fills the wave has uniform entries
    auto uni = [](int v) { return LPG == 64 ? __builtin_amdgcn_readfirstlane(v) : v; };
    // this lane's columns, wide and contiguous across the slot's lanes: two, then one
    const int p0 = 2 * li, p2 = 2 * LPG + li;
    const int c0 = p0 < cc ? p0 : 0, c2 = p2 < cc ? p2 : 0;
    const T *xc = x + (size_t)r0 * 6;
    auto gather = [&](int m, T (&xv)[3][3]) {
        const T *q = xc + (size_t)m * 3 * c;
#pragma unroll
        for (int d = 0; d < 3; ++d, q += c) {
            const T2 w = *(const T2 *)(q + c0);
            xv[d][0] = w[0];
            xv[d][1] = w[1];
            xv[d][2] = q[c2];
        }
    };
    struct Group {
        int grp, u0, u1, b0, b1;   // neighbours u0 .. u1 - 1, blocks b0 .. b1 - 1
    };
    auto group_of = [&](int it) {   // (the last group where there is none)
        Group g;
        const int q = it * G::NS + slot;
        g.grp = uni(q < ngroups ? q : ngroups - 1);
        g.u0 = gptr[g.grp];
        g.u1 = gptr[g.grp + 1];
        g.b0 = gblk[g.grp];
        g.b1 = gblk[g.grp + 1];
        return g;
    };
    F4 rq[G::NQ] = {};
    int2 re = {};
    // chunk of a group: neighbours from us on, blocks from the group's block off on
    auto fetch = [&](int us, int u1, int b0, int b1, int off) {
        re = gnbr[us + li < u1 ? us + li : u1 - 1];
        const F4 *vsrc = (const F4 *)(gval + (size_t)b0 * 12);
        const int last = max((b1 - b0) * PPB - 1, 0);
#pragma unroll
        for (int i = 0; i < G::NQ; ++i) {
            const int q = off * PPB + i * LPG + li;
            rq[i] = vsrc[q < last ? q : last];
        }
    };
    Group cur = group_of(item);
    fetch(cur.u0, cur.u1, cur.b0, cur.b1, 0);
    {   // (unrolled: the loads are in flight together, and with those above)
        T v[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const int e = threadIdx.x + 256 * q, k = e / 72, j = e - k * 72;
            if (k < per) v[q] = tmat[(size_t)(r0 + min(k, R - r0 - 1)) * 72 + j];
        }
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const int e = threadIdx.x + 256 * q, k = e / 72, j = e - k * 72;
            if (k < per) st[k * kTS + j] = v[q];
        }
    }
    __syncthreads();
    const int kc = min(li >> 1, per - 1), j0 = (li & 1) * 3;
    const T *own = st + kc * kTS + j0 * 7, *other = st + kc * kTS + j0 * 5 + 3;
    T *sm = (T *)sv;
    for (; item < end; item += step) {
        const Group next = group_of(item + step < end ? item + step : item);
        int us = cur.u0, trips = (cur.u1 - us + CH - 1) / CH;   // the longest slot's
#pragma unroll
        for (int o = 32; o >= LPG; o >>= 1) trips = max(trips, __shfl_xor(trips, o));
        trips = __builtin_amdgcn_readfirstlane(trips);
        T aK[kG][3][3], aM[kG][3][3];
#pragma unroll
        for (int g = 0; g < kG; ++g)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int n = 0; n < 3; ++n) { aK[g][i][n] = T(0); aM[g][i][n] = T(0); }
        auto stage = [&]() {
            __builtin_amdgcn_wave_barrier();   // (a wave's LDS accesses complete in order)
            if (li < CH + 2) se[li] = make_int2(re.x, us + li < cur.u1 ? re.y : 0);   // 0: past the end
#pragma unroll
            for (int i = 0; i < G::NQ; ++i)
                if (i * LPG + li < G::VP) sv[i * LPG + li] = rq[i];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        stage();
        T xv[3][3][3];   // two neighbours ahead
        gather(uni(se[0].x), xv[0]);
        gather(uni(se[1].x), xv[1]);
        for (;;) {
            {   // the next chunk, of this group or of the next
                const bool more = trips > 1;
                const int off = se[CH].y >> 4;
                fetch(more ? (us + CH < cur.u1 ? us + CH : cur.u1) : next.u0,
                      more ? cur.u1 : next.u1, more ? cur.b0 : next.b0, more ? cur.b1 : next.b1,
                      more ? off : 0);
            }
            const T *bv = (const T *)sv + min(lane & 15, 11);
            T kv = *bv;
            auto neighbour = [&](int mask, const T (&xv)[3][3]) {
#pragma unroll
                for (int g = 0; g < kG; ++g) {
                    if (!((mask >> g) & 1)) continue;
                    bv += 12;
                    const T nx = *bv;   // (past the last block: what stands behind it)
                    block_row<0>(kv, xv, aK[g][0], aM[g][0]);
                    block_row<1>(kv, xv, aK[g][1], aM[g][1]);
                    block_row<2>(kv, xv, aK[g][2], aM[g][2]);
                    kv = nx;
                }
            };
            int2 e0 = se[0], e1 = se[1];
#pragma unroll
            for (int t = 0; t < CH; ++t) {
                const int2 e2 = se[t + 2];
                gather(uni(e2.x), xv[(t + 2) % 3]);
                __builtin_amdgcn_sched_barrier(0);
                neighbour(uni(e0.y) & 15, xv[t % 3]);
                __builtin_amdgcn_sched_barrier(0);
                e0 = e1;
                e1 = e2;
            }
            if (--trips == 0) break;
            us += CH;
            stage();
        }
        // Y = K X A^T + M X B^T, a node at a time: through LDS to three consecutive columns a
        // lane (the case's other three are its pair lane's) and back.
        const bool out_slot = !spare && item * G::NS + slot < ngroups;
        T ta[3][6], tb[3][6];   // own columns first, then the pair lane's
#pragma unroll
        for (int g = 0; g < kG; ++g) {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                T *sk = sm + i * 6 * LPG;
                sk[p0] = aK[g][i][0];
                sk[p0 + 1] = aK[g][i][1];
                sk[p2] = aK[g][i][2];
                sk[3 * LPG + p0] = aM[g][i][0];
                sk[3 * LPG + p0 + 1] = aM[g][i][1];
                sk[3 * LPG + p2] = aM[g][i][2];
            }
            if (g == 0) {
#pragma unroll
                for (int n = 0; n < 3; ++n)
#pragma unroll
                    for (int j = 0; j < 6; ++j) {
                        const T *t = (j < 3 ? own : other) + n * 6 + (j < 3 ? j : j - 3);
                        ta[n][j] = t[0];
                        tb[n][j] = t[36];
                    }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                T *sk = sm + i * 6 * LPG + 3 * li;
                T out[3] = {T(0), T(0), T(0)};
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const T zk = sk[j], zm = sk[3 * LPG + j];
                    const T pk = pair_swap(zk), pm = pair_swap(zm);
#pragma unroll
                    for (int n = 0; n < 3; ++n) {
                        out[n] += ta[n][j] * zk + tb[n][j] * zm;
                        out[n] += ta[n][3 + j] * pk + tb[n][3 + j] * pm;
                    }
                }
                // (a row's values are read by the lanes that hold them before they are replaced)
#pragma unroll
                for (int n = 0; n < 3; ++n) sk[n] = alpha * out[n];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int node = cur.grp * kG + g;
            if (out_slot && node < nn) {
                T *yr = y + (size_t)node * 3 * c + (size_t)r0 * 6;
#pragma unroll
                for (int i = 0; i < 3; ++i, yr += c) {
                    const T *sk = sm + i * 6 * LPG;
                    if (p0 < cc) {
                        T2 o = {sk[p0], sk[p0 + 1]};
                        T2 *q = (T2 *)(yr + p0);
                        if (beta != T(0)) {
                            const T2 old = *q;
                            o[0] += beta * old[0];
                            o[1] += beta * old[1];
                        }
                        *q = o;
                    }
                    if (p2 < cc) yr[p2] = beta == T(0) ? sk[p2] : sk[p2] + beta * yr[p2];
                }
            }
        }
        cur = next;
    }
}

// Sum over aligned groups of 4 or 8 lanes with DPP moves (swap neighbours, swap pairs
// in a quad, mirror in the half-row): every lane of the group ends with the group's sum.
template <int CTRL>
__device__ __forceinline__ float quad_move(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double quad_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
template <int SPL, typename T>
__device__ __forceinline__ T group_sum(T v) {
    v += quad_move<0xB1>(v);                     // quad_perm [1,0,3,2]
    v += quad_move<0x4E>(v);                     // quad_perm [2,3,0,1]
    if (SPL == 8) v += quad_move<0x141>(v);      // row_half_mirror
    return v;
}

// One load case (R = 1): SPL lanes per node row, lane `sub` taking the slot's entries
// sub, sub + SPL, ...; the partial K X and M X sums are added across the SPL lanes, and
// lane i < 3 applies the temporal matrices to row i of the node.  SPL times the waves
// of the lane-per-node kernel, and 1/SPL of its dependent load chain per lane, for the
// small launches where that chain is the bound.
template <typename T, int SPL, int UNR>
__global__ void __launch_bounds__(256)
kron_bsr3_r1_kernel(int nslices, const int *__restrict__ slot_node,
                    const int *__restrict__ slice_base, const int *__restrict__ slice_len,
                    const int *__restrict__ bcol, const T *__restrict__ bval,
                    const T *__restrict__ tmat, T alpha, T beta, const T *__restrict__ x,
                    T *__restrict__ y) {
    using V2 = typename Vec2<T>::type;
    constexpr int NPW = 64 / SPL, c = 6;
    const int lane = threadIdx.x & 63, sub = lane % SPL;
    const long long blk = xcd_block(blockIdx.x, gridDim.x);
    const long long wave = blk * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const long long slot = wave * NPW + lane / SPL;
    const int s = (int)(slot / kSlice);
    if (s >= nslices) return;   // whole quads leave together
    const int k = (int)(slot - (long long)s * kSlice);
    const int node = slot_node[slot];
    const int L = slice_len[s];
    const long long b0 = slice_base[s];
    T aK[3][6], aM[3][6];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) { aK[i][j] = T(0); aM[i][j] = T(0); }
    auto accumulate = [&](const T (&kv)[12], const T (&xv)[3][6]) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 6; ++j) {
                aK[i][j] += kv[3 * i + 0] * xv[0][j] + kv[3 * i + 1] * xv[1][j] + kv[3 * i + 2] * xv[2][j];
                aM[i][j] += kv[9 + i] * xv[i][j];
            }
    };
    auto gather = [&](int m, T (&xv)[3][6]) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const T *xr = x + (size_t)(3 * m + d) * c;
#pragma unroll
            for (int j = 0; j < 6; j += 2) {
                const V2 v = *reinterpret_cast<const V2 *>(xr + j);
                xv[d][j] = v.x;
                xv[d][j + 1] = v.y;
            }
        }
    };
    int e = sub;
    for (; e + (UNR - 1) * SPL < L; e += UNR * SPL) {
        int m[UNR];
        T kv[UNR][12], xv[UNR][3][6];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const long long idx = b0 + (long long)(e + u * SPL) * kSlice + k;
            m[u] = bcol[idx];
            load_block(bval + idx * 12, kv[u]);
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) gather(m[u], xv[u]);
#pragma unroll
        for (int u = 0; u < UNR; ++u) accumulate(kv[u], xv[u]);
    }
    for (; e < L; e += SPL) {
        const long long idx = b0 + (long long)e * kSlice + k;
        T kv[12], xv[3][6];
        load_block(bval + idx * 12, kv);
        gather(bcol[idx], xv);
        accumulate(kv, xv);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            aK[i][j] = group_sum<SPL>(aK[i][j]);
            aM[i][j] = group_sum<SPL>(aM[i][j]);
        }
    if (node < 0 || sub >= 3) return;
    const T *TA = tmat, *TB = tmat + 36;
    T out[6];
#pragma unroll
    for (int o = 0; o < 6; ++o) {
        T sacc = T(0);
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            // row sub of the node: select without dynamic register indexing
            const T kk = sub == 0 ? aK[0][j] : sub == 1 ? aK[1][j] : aK[2][j];
            const T mm = sub == 0 ? aM[0][j] : sub == 1 ? aM[1][j] : aM[2][j];
            sacc += TA[o * 6 + j] * kk + TB[o * 6 + j] * mm;
        }
        out[o] = sacc;
    }
    T *yr = y + (size_t)(3 * node + sub) * c;
#pragma unroll
    for (int o = 0; o < 6; o += 2) {
        V2 v;
        if (beta == T(0)) {
            v.x = alpha * out[o];
            v.y = alpha * out[o + 1];
        } else {
            const V2 old = *reinterpret_cast<const V2 *>(yr + o);
            v.x = alpha * out[o] + beta * old.x;
            v.y = alpha * out[o + 1] + beta * old.y;
        }
        *reinterpret_cast<V2 *>(yr + o) = v;
    }
}

// K and M values (CSR entries in the order the plan was built from) into the node blocks,
// FP64 and FP32.
__global__ void __launch_bounds__(256)
bsr_scatter_kernel(long long n, const int *__restrict__ map, const double *__restrict__ v,
                   double *__restrict__ b64, float *__restrict__ b32) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int t = map[i];
    if (t < 0) return;   // an entry that a later one of the row replaces
    const double w = v[i];
    b64[t] = w;
    b32[t] = (float)w;
}

// The slices' blocks to the groups, a 16-byte piece a lane (PPB a block; n pieces).
template <int PPB>
__global__ void __launch_bounds__(256)
bsr_group_kernel(long long n, const int *__restrict__ gof, const F4 *__restrict__ b,
                 F4 *__restrict__ g) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int blk = (int)(i / PPB), u = gof[blk];
    if (u >= 0) g[(long long)u * PPB + (i - (long long)blk * PPB)] = b[i];
}
template <typename T>
static int copy_groups(const BsrPlan &P, const DevBuf &b, const DevBuf &g, hipStream_t s) {
    constexpr int PPB = 12 * sizeof(T) / 16;
    const long long n = P.nblocks * PPB;
    hipLaunchKernelGGL(bsr_group_kernel<PPB>, dim3(ceil_div(n, 256)), dim3(256), 0, s, n,
                       P.gof.as<int>(), b.as<F4>(), g.as<F4>());
    XT_HIP(hipGetLastError());
    return XT_OK;
}

int bsr_set_values(BsrPlan &P, const double *kv, const double *mv, hipStream_t s) {
    if (P.nk)
        hipLaunchKernelGGL(bsr_scatter_kernel, dim3(ceil_div(P.nk, 256)), dim3(256), 0, s, P.nk,
                           P.kmap.as<int>(), kv, P.bval64.as<double>(), P.bval32.as<float>());
    if (P.nm)
        hipLaunchKernelGGL(bsr_scatter_kernel, dim3(ceil_div(P.nm, 256)), dim3(256), 0, s, P.nm,
                           P.mmap.as<int>(), mv, P.bval64.as<double>(), P.bval32.as<float>());
    XT_HIP(hipGetLastError());
    std::lock_guard<std::mutex> lock(P.gmutex);
    if (P.gval64.ptr) XT_TRY(copy_groups<double>(P, P.bval64, P.gval64, s));
    if (P.gval32.ptr) XT_TRY(copy_groups<float>(P, P.bval32, P.gval32, s));
    return XT_OK;
}

// The groups' values in T (NULL: the slices are to be taken), copied by the first caller and
// complete when it returns, whatever streams the next ones use.  A graph capture allocates
// nothing, so an operator's first apply there takes the slices, as does one without memory
// for a second copy.
template <typename T>
static int group_values(BsrPlan &P, hipStream_t s, const T **out) {
    const bool f32 = sizeof(T) == 4;
    DevBuf &g = f32 ? P.gval32 : P.gval64;
    std::lock_guard<std::mutex> lock(P.gmutex);
    if (!g.ptr && !P.no_gval[f32]) {
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        XT_HIP(hipStreamIsCapturing(s, &capturing));
        if (capturing == hipStreamCaptureStatusNone) {
            if (g.reserve(sizeof(T) * 12 * (size_t)P.nreal) != XT_OK) {
                (void)hipGetLastError();   // (not an error of this call)
                P.no_gval[f32] = true;
            } else {
                int rc = copy_groups<T>(P, f32 ? P.bval32 : P.bval64, g, s);
                if (rc == XT_OK && hipStreamSynchronize(s) != hipSuccess) rc = XT_E_HIP;
                if (rc != XT_OK) {
                    g.release();
                    return rc;
                }
            }
        }
    }
    *out = g.as<T>();
    return XT_OK;
}

static constexpr int kR1Split = 4;   // lanes per node row for one load case (8: slower)

// Kernel variant of a launch: the tuning knobs, else the built-in choices (4 entries in
// flight for one load case in FP32, else 2: with several cases in FP32 two entries took
// 849 us against 909 at 32 cases and 233 against 271 at 8 on a 435,969-DOF operator; one
// wave per workgroup when four-wave workgroups would leave CUs idle; kR1Split lanes per
// node for one load case).
template <typename T>
static int spmm_unr(int R) {
    const int k = tune_knob(XT_TUNE_SPMM_UNR);
    return k ? k : (sizeof(T) == 4 && R == 1 ? 4 : 2);
}

// LDS budget of one staged workgroup (two fit a CU's 160 KB).
constexpr size_t kStageLds = 64 * 1024;

// Columns per staged workgroup: the largest of 48, 24, 12 (whole load cases, 16-byte
// rows) that divides c and whose neighbour rows fit kStageLds; 0 when none does.
template <typename T>
static int stage_cols(const BsrPlan &P, int c) {
    if (!P.umax) return 0;
    for (int cc : {48, 24, 12})
        if (c % cc == 0 && (size_t)P.umax * 3 * cc * sizeof(T) <= kStageLds) return cc;
    return 0;
}

// Lanes per node of the slice kernel: the cases, except that
// - up to one wave a CU nothing shares its vector cache, and a power of two's loads touch
//   fewer lines each (power of two / cases, us, FP64: 5 cases on 455 nodes 12.1 / 12.8, 17 there
//   12.2 / 12.5; past 256 waves 9 on 1155 nodes 13.8 / 12.8, 17 there 16.7 / 14.8);
// - a count one below a power of two gets an idle lane: a node's lanes then neither straddle
//   waves nor shift against the cache lines from node to node (cases / cases + 1, us, FP64:
//   3 on 23735 nodes 38 / 35, 7 there 74 / 65, 15 on 4879 nodes 32.7 / 32.0; FP32: 15 there
//   19.0 / 17.8, 31 33.1 / 30.9, but 3 on 32513 nodes 23 / 25).  Other odd counts lose by it
//   as often as they win (5 on 23735 nodes 53 / 61, 13 on 13237 69 / 67).
template <typename T>
static int slice_lanes(int R, int nslices) {
    int up = 1;
    while (up < R) up <<= 1;
    if ((long long)nslices * up <= 256) return up;
    return R + 1 == up && R > (sizeof(T) == 4 ? 3 : 1) ? up : R;
}

// The group kernel from enough work on: a wave takes 24 (64 lanes a group) to 36 us (16) for
// its first group, a chain of loads, whatever the number of groups (a group's neighbours
// shared by the four waves of a workgroup: 13 to 18 us, but slower at every size from 4879
// nodes on in FP64 and 13237 in FP32, and no better than slices below).  The slices' time
// grows with nodes times cases, the groups' with their neighbours, 26 a group (3 x 3 nodes in
// the section) to 51 (40 x 9), so the line lies in nodes times cases at 45 a group (work, in
// thousands below; a section 5 nodes across).  Slices / groups, us, at work (cases):
//   FP64  197 (4) 79 / 102, 275 (4) 125 / 117, 281 (4) 79 / 84, 340 (4) 77 / 72, 95 (8) 36 / 41,
//         134 (8) 55 / 55, 232 (8) 55 / 41, 267 (8) 104 / 109, 395 (8) 142 / 130, 106 (9) 42 / 45,
//         151 (9) 63 / 62, 184 (9) 42 / 33, 95 (16) 35 / 34, 132 (16) 53 / 45, 59 (20) 24 / 27,
//         83 (20) 35 / 35, 118 (20) 45 / 36, 106 (36) 40 / 36, 123 (36) 31 / 23
//   FP32  267 (8) 58 / 59, 327 (8) 36 / 32, 395 (8) 77 / 75, 200 (12) 40 / 52, 284 (12) 58 / 54,
//         166 (20) 34 / 40, 236 (20) 45 / 41, 166 (28) 33 / 31, 232 (28) 45 / 38, 213 (36) 42 / 41,
//         298 (36) 58 / 68, 425 (36) 77 / 74
// The groups' time goes in rounds of the waves that the card holds (16 lanes a group: 32768
// nodes in FP64, 49152 in FP32), so just above one they lose up to 15 % (FP64, 6 cases on 33900
// nodes: 79 / 90).  In FP32 the stored blocks times cases have to outweigh the neighbours times
// the lanes as well (share; 4 cases on 99972 nodes 82 / 103, 36 on 8400 59 / 68).  Over 2480
// operators (40 to 800 thousand nodes times cases, 2 to 64 cases, eight sections) the choice
// takes 1.005 times the better kernel's time, 1.32 at most (FP64, 14 cases on 3900 nodes).
static bool group_form(const BsrPlan &P, int R, bool f32) {
    const int k = tune_knob(XT_TUNE_SPMM_GROUP);
    if (R < 2 || k == 1) return false;
    if (k == 2) return true;
    if (R < (f32 ? 5 : 3)) return false;
    const int chunks = ceil_div(R, 32), per = ceil_div(R, chunks);
    const double share = f32 ? (per <= 8 ? 15 : per <= 16 ? 28 : 40) * chunks : 0;
    if ((double)R * P.nblocks <= share * P.ngnbr) return false;
    const double work = (double)P.nn * R * 45 * P.ngroups / P.ngnbr;
    if (f32) return work >= (R <= 16 ? 280000 : 200000);
    return work >= (R <= 4 ? 270000 : R <= 16 ? 115000 : 68000);
}

template <typename T>
int bsr_apply(BsrPlan &P, int R, const T *tmat, double alpha, double beta, const T *x,
              T *y, bool f32, hipStream_t s) {
    const T *bv = f32 ? (const T *)P.bval32.ptr : (const T *)P.bval64.ptr;
    const int c = 6 * R;
    // staged kernel: only when the tuning knob asks for it (2; measured slower than the
    // lane-per-case kernel on the structured meshes here at 32 load cases) and the groups
    // are not asked for as well
    const int lk = tune_knob(XT_TUNE_SPMM_LDS), gk = tune_knob(XT_TUNE_SPMM_GROUP);
    const int cc = (lk != 2 || gk == 2 || R < 2) ? 0 : stage_cols<T>(P, c);
    if (cc) {
        const int nch = c / cc;
        const int grid = (int)(((long long)P.nslices * nch + 7) / 8 * 8);
        const size_t lds = (size_t)P.umax * 3 * cc * sizeof(T);
        if (prof_on(XT_PROF_SPMM)) prof_begin(XT_PROF_SPMM, s);
#define XT_BSR_LDS(CCV)                                                                        \
    hipLaunchKernelGGL((kron_bsr3_lds_kernel<T, CCV>), dim3(grid), dim3(64 * (CCV / 6)), lds, s, \
                       P.nslices, nch, P.slot_node.as<int>(), P.slice_base.as<int>(),          \
                       P.slice_len.as<int>(), P.unode.as<int>(), P.ubase.as<int>(),            \
                       P.ulen.as<int>(), P.lidx.as<unsigned short>(), bv, c, tmat, (T)alpha,   \
                       (T)beta, x, y)
        if (cc == 48) XT_BSR_LDS(48);
        else if (cc == 24) XT_BSR_LDS(24);
        else XT_BSR_LDS(12);
#undef XT_BSR_LDS
        if (prof_on(XT_PROF_SPMM)) {
            // as the lane-per-case kernel's: the stored format read once, X read once,
            // Y written (and read when beta != 0); the neighbour lists (2 B per block
            // in place of the 4-byte column index, 4 B per listed node) are counted
            const double sv = sizeof(T);
            const double vec = (double)P.nn * 3 * c * sv;
            const double bytes = (double)P.nblocks * (12 * sv + 2) +
                                 (double)P.nslices * (kSlice * 4 + 16) +
                                 (double)(P.unode.bytes) + vec * (beta != 0 ? 3 : 2);
            const double flops = 2.0 * 12 * P.nreal * c + 2.0 * 2 * 6 * (3.0 * P.nn) * c;
            prof_end(XT_PROF_SPMM, s, bytes, flops);
        }
        XT_HIP(hipGetLastError());
        return XT_OK;
    }
    const T *gv = nullptr;
    if (group_form(P, R, f32)) XT_TRY(group_values<T>(P, s, &gv));
    if (gv) {
        // cases split evenly over launches' second dimension, at most 32 a wave
        const int nchunk = ceil_div(R, 32), per = ceil_div(R, nchunk);
        if (prof_on(XT_PROF_SPMM)) prof_begin(XT_PROF_SPMM, s);
#define XT_GROUP(LPG)                                                                          \
    {                                                                                          \
        using G = GroupGeom<T, LPG>;                                                           \
        const int need = ceil_div(P.ngroups, 4 * G::NS), most = std::max(1, 256 * G::BPC / nchunk); \
        hipLaunchKernelGGL((kron_group_kernel<T, LPG>),                                        \
                           dim3(ceil_div(std::min(need, most), 8) * 8, nchunk),                \
                           dim3(256), 64 * G::NS * G::SLOT + sizeof(T) * kTS * per, s,         \
                           P.ngroups, P.nn, P.gptr.as<int>(), P.gblk.as<int>(),                \
                           P.gnbr.as<const int2>(), gv, R, per, c, tmat, (T)alpha, (T)beta, x, \
                           y);                                                                 \
    }
        if (per <= 8) XT_GROUP(16)
        else if (per <= 16) XT_GROUP(32)
        else if (per <= 24) XT_GROUP(48)
        else XT_GROUP(64)
#undef XT_GROUP
        if (prof_on(XT_PROF_SPMM)) {
            // 12 values per block, the neighbour lists, X read, Y written (and read)
            const double sv = sizeof(T), vec = (double)P.nn * 3 * c * sv;
            const double bytes = (double)P.nreal * 12 * sv + (double)P.gnbr.bytes +
                                 8.0 * P.ngroups + vec * (beta != 0 ? 3 : 2);
            prof_end(XT_PROF_SPMM, s, bytes,
                     2.0 * 12 * P.nreal * c + 2.0 * 2 * 6 * (3.0 * P.nn) * c);
        }
        XT_HIP(hipGetLastError());
        return XT_OK;
    }
    for (int r0 = 0; r0 < R; r0 += 64) {
        const int Rc = std::min(64, R - r0);
        const long long slots = (long long)P.nslices * kSlice;
        const int W = slice_lanes<T>(Rc, P.nslices);
        const long long waves = (long long)P.nslices * W;
        const unsigned inv = (0x80000000u + W - 1) / W;
        const int wk = tune_knob(XT_TUNE_SPMM_WPB);
        const int wpb = wk ? wk : (waves >= 4 * 1024 ? 4 : 1);
        const int grid = (int)(((waves + wpb - 1) / wpb + 7) / 8 * 8);
        const int unr = spmm_unr<T>(R);
#define XT_BSR_LAUNCH(U)                                                                      \
    hipLaunchKernelGGL((kron_bsr3_kernel<T, U>), dim3(grid), dim3(64 * wpb), 0, s, P.nslices,  \
                       P.slot_node.as<int>(), P.slice_base.as<int>(), P.slice_len.as<int>(),  \
                       P.bcol.as<int>(), bv, W, inv, r0 + Rc, r0, c, tmat, (T)alpha, (T)beta, x, y)
#define XT_BSR_R1(S, U)                                                                       \
    hipLaunchKernelGGL((kron_bsr3_r1_kernel<T, S, U>), dim3(grid1), dim3(64), 0, s, P.nslices, \
                       P.slot_node.as<int>(), P.slice_base.as<int>(), P.slice_len.as<int>(),  \
                       P.bcol.as<int>(), bv, tmat, (T)alpha, (T)beta, x, y)
        if (prof_on(XT_PROF_SPMM)) prof_begin(XT_PROF_SPMM, s);
        if (R == 1) {   // spl lanes per node
            const int sk = tune_knob(XT_TUNE_SPMM_R1SPLIT);
            const int spl = sk ? sk : kR1Split;
            const int grid1 = (int)(((slots * spl / 64) + 7) / 8 * 8);
            if (spl == 8) {
                if (unr == 2) XT_BSR_R1(8, 2);
                else if (unr == 8) XT_BSR_R1(8, 8);
                else XT_BSR_R1(8, 4);
            } else {
                if (unr == 2) XT_BSR_R1(4, 2);
                else if (unr == 8) XT_BSR_R1(4, 8);
                else XT_BSR_R1(4, 4);
            }
        } else if (unr == 2) {
            XT_BSR_LAUNCH(2);
        } else if (unr == 8) {
            XT_BSR_LAUNCH(8);
        } else {
            XT_BSR_LAUNCH(4);
        }
#undef XT_BSR_R1
#undef XT_BSR_LAUNCH
        if (prof_on(XT_PROF_SPMM)) {
            // 12 values (3x3 K block + diagonal of the M block) + 1 column index per
            // stored block, slice tables, X read, Y written (and read when beta != 0)
            const double sv = sizeof(T);
            const double vec = (double)P.nn * 3 * 6 * Rc * sv;
            const double bytes = (double)P.nblocks * (12 * sv + 4) +
                                 (double)P.nslices * (kSlice * 4 + 8) + vec * (beta != 0 ? 3 : 2);
            const double flops = 2.0 * 12 * P.nreal * 6 * Rc + 2.0 * 2 * 6 * (3.0 * P.nn) * 6 * Rc;
            prof_end(XT_PROF_SPMM, s, bytes, flops);
        }
        XT_HIP(hipGetLastError());
    }
    return XT_OK;
}
template int bsr_apply<float>(BsrPlan &, int, const float *, double, double, const float *,
                              float *, bool, hipStream_t);
template int bsr_apply<double>(BsrPlan &, int, const double *, double, double,
                               const double *, double *, bool, hipStream_t);

}  // namespace xt

namespace xt {
BsrPlan *bsr_new() { return new BsrPlan; }
void bsr_delete(BsrPlan *p) { delete p; }
long long bsr_blocks(const BsrPlan *p, int real) { return real ? p->nreal : p->nblocks; }
}  // namespace xt
