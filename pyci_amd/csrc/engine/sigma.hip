// Sigma (Y = H X) over the stored full-pattern CSR: the GPU counterpart of the
// reference's Eigen SpMV in perform_op / perform_op_symm (sparseop.cpp:96-112).
// The symmetric operator is stored with both triangles, so one row-parallel
// streaming pass produces (L + L^T - D) x without scatter atomics.
//
// Layout: X is ncol x NV and Y is nrow x NV, row-major, so the NV values a column
// index points at share one cache line. One 64-lane wavefront per row; each lane
// streams column indices (4 B) and values (8 B FP64 or 4 B FP32) with a stride of
// 64 entries, so every load instruction of the wavefront is fully coalesced.
// Rows are handed to blocks in contiguous per-XCD chunks (see xcd_row_block).
#include <algorithm>

#include "internal.hpp"

namespace pe {

constexpr int SPMV_WAVES = 4;  // wavefronts (rows) per 256-thread block
constexpr i64 SPMV_LDS_MIN_NNZ = (i64)1 << 20;
constexpr i64 SPMV_LDS_MIN_SEG = 32;
constexpr int NUM_XCD = 8;

// Blocks are dispatched round-robin over the 8 XCDs (block b runs on XCD b % 8).
// Remap so that XCD x receives a contiguous range of row blocks: neighbouring
// rows of a CI matrix share most of their column targets, so each XCD's L2 then
// serves a compact slice of X.
__device__ inline i64 xcd_row_block(i64 b, i64 nblocks) {
    const i64 per = (nblocks + NUM_XCD - 1) / NUM_XCD;
    const i64 x = b % NUM_XCD, k = b / NUM_XCD;
    const i64 r = x * per + k;
    return r;
}

// Row-major X with NV values per column; the NV values of one column are read as
// 16-byte pieces (NV * sizeof(XT) / 16 of them), and every lane issues the
// column/value loads of U entries (non-temporal: the CSR is streamed once per
// sigma) before their U * NV gathers, so each wavefront keeps U * 64 entries in flight.
template <typename XT>
struct Vec16;
template <>
struct Vec16<double> {
    typedef double2 type;
    static constexpr int n = 2;
};
template <>
struct Vec16<float> {
    typedef float4 type;
    static constexpr int n = 4;
};

// waves_per_eu(1, 4) lets the compiler hold all U * NQ pieces in registers (at
// FullCI nbasis 12, 8 FP64 vectors: 11.9 ms against 16.8 ms with the default budget).
template <int NV, int U, typename VT, typename XT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 4)))
k_spmm(i64 nrow, i64 nblocks, const i64 *__restrict__ rowptr, const int32_t *__restrict__ cols,
       const VT *__restrict__ vals, const XT *__restrict__ X, XT *__restrict__ Y) {
    typedef typename Vec16<XT>::type V16;
    constexpr int PER = Vec16<XT>::n, NQ = NV / PER;  // XT values per piece, pieces per column
    static_assert(NV % PER == 0, "NV must fill whole 16-byte pieces");
    const int lane = threadIdx.x & 63;
    const i64 blk = xcd_row_block(blockIdx.x, nblocks);
    const i64 row = blk * SPMV_WAVES + (threadIdx.x >> 6);
    if (blk >= nblocks || row >= nrow) return;
    const i64 beg = rowptr[row], end = rowptr[row + 1];
    XT acc[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[j] = (XT)0;
    const V16 *__restrict__ X16 = reinterpret_cast<const V16 *>(X);
    i64 p = beg + lane;
    for (; p + (U - 1) * 64 < end; p += U * 64) {
        int c[U];
        VT v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c[u] = __builtin_nontemporal_load(&cols[p + u * 64]);
            v[u] = __builtin_nontemporal_load(&vals[p + u * 64]);
        }
        V16 x[U][NQ];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < NQ; ++q) x[u][q] = X16[(i64)c[u] * NQ + q];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const XT w = (XT)v[u];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const XT *e = reinterpret_cast<const XT *>(&x[u][q]);
#pragma unroll
                for (int t = 0; t < PER; ++t) acc[q * PER + t] += w * e[t];
            }
        }
    }
    for (; p < end; p += 64) {
        const int c = __builtin_nontemporal_load(&cols[p]);
        const XT w = (XT)__builtin_nontemporal_load(&vals[p]);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const V16 xv = X16[(i64)c * NQ + q];
            const XT *e = reinterpret_cast<const XT *>(&xv);
#pragma unroll
            for (int t = 0; t < PER; ++t) acc[q * PER + t] += w * e[t];
        }
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        XT v = acc[j];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        acc[j] = v;
    }
    if (lane < NV) {
        XT out = acc[0];
#pragma unroll
        for (int j = 1; j < NV; ++j)
            if (lane == j) out = acc[j];
        Y[row * NV + lane] = out;
    }
}

// Single vector, a row per wave: every lane issues the column and value loads of U entries
// (non-temporal: the CSR is streamed once per sigma and must not evict X), then their U
// gathers of X. A row's last chunk takes part with the lanes that have an entry: loads beyond
// the row cost requests, and an element of X that belongs to no entry may be an infinity or a
// NaN. The gathers bound it: an 8-byte element costs a 128-byte line from L2 unless L1 still
// holds it.
//   WAVES 16, U 1   rows of a full space, sorted in column order: 16 neighbouring rows (most
//                   with the same alpha string) walk the same lines of X in step, so L1 serves
//                   them; a wider window per lane spreads the waves over more lines than L1
//                   holds. nbasis 12 (18.6 GB): 3.99 ms (4.7 TB/s) against 5.18-6.4 with U
//                   2..16 and 4 waves; nbasis 10: 147 us against 156-200. And sets of short
//                   rows, two chunks at most (400,000 FullCI determinants of 32 entries a row
//                   114 us, 172 with 4 waves and U 3; DOCI of 74,613 rows of 97 33 us, 40).
//   WAVES 4, U 3    other sets, whose entries are too few or too thin for panels of X in LDS
//                   (100,000 GenCI determinants of 154 entries a row 90 us, 99 with 16 waves,
//                   94 with U 6; full spaces of 15,876 rows of 561 26.6 us, 27-28 with U 2..8,
//                   36 with U 1).
template <int U, int WAVES, typename VT, typename XT>
__global__ void __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(1, WAVES == 4 ? 4 : 8)))
k_spmv(i64 nrow, i64 nblocks, const i64 *__restrict__ rowptr, const int32_t *__restrict__ cols,
       const VT *__restrict__ vals, const XT *__restrict__ X, XT *__restrict__ Y) {
    const int lane = threadIdx.x & 63;
    const i64 blk = xcd_row_block(blockIdx.x, nblocks);
    const i64 row = blk * WAVES + (threadIdx.x >> 6);
    if (blk >= nblocks || row >= nrow) return;
    const i64 beg = rowptr[row];
    const int len = (int)(rowptr[row + 1] - beg);
    cols += beg;
    vals += beg;
    XT acc = (XT)0;
    int p = lane;
    for (; p - lane + U * 64 <= len; p += U * 64) {
        int c[U];
        VT v[U];
        XT x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c[u] = __builtin_nontemporal_load(&cols[p + u * 64]);
            v[u] = __builtin_nontemporal_load(&vals[p + u * 64]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = X[c[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) acc += (XT)v[u] * x[u];
    }
    if (p - lane < len) {
        int c[U];
        VT v[U];
        XT x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            c[u] = 0, v[u] = (VT)0, x[u] = (XT)0;
            if (p + u * 64 < len) {
                c[u] = __builtin_nontemporal_load(&cols[p + u * 64]);
                v[u] = __builtin_nontemporal_load(&vals[p + u * 64]);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (p + u * 64 < len) x[u] = X[c[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) acc += (XT)v[u] * x[u];
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane == 0) Y[row] = acc;
}

// Single vector with X in LDS: one block of 16 waves per CU takes a run of rows with an equal
// share of the entries and goes through the columns in panels of SPMV_PANEL; a panel of X is
// staged, then 16 lanes (or a wave) multiply a row's entries of that panel, whose places come
// from the plan, with the next row's entries loaded while the current row's gathers come out
// of LDS. Longer rows are taken by the whole block afterwards. For sets whose columns follow
// no order the gathers then cost LDS cycles instead of a 128-byte line of L2 each: 60,000
// GenCI determinants (32 M entries, 3 panels) 286 -> 119 us (3.3 TB/s), 100,000 FullCI ones
// (5 panels) 580 -> 221 us, 17,317 (one panel) 51 -> 22.5 us. Lanes beyond a row's entries
// multiply 0 by the 0 behind the panel: X may hold infinities and NaNs, which belong to the
// rows of their columns alone.
constexpr int SPMV_PANEL = 20000;
constexpr int SPMV_LDS_WAVES = 16;

template <int LANES, typename VT, typename XT>
__global__ void __launch_bounds__(SPMV_LDS_WAVES * 64)
k_spmv_lds(i64 ncol, int npanel, const i64 *__restrict__ rowptr, const int32_t *__restrict__ split,
           const int *__restrict__ bounds, i64 long_len, const int32_t *__restrict__ cols,
           const VT *__restrict__ vals, const XT *__restrict__ X, XT *__restrict__ Y) {
    constexpr int U = LANES == 16 ? 8 : 4, NT = SPMV_LDS_WAVES * 64, STEP = NT / LANES;
    extern __shared__ double lds[];
    XT *xs = reinterpret_cast<XT *>(lds);
    __shared__ XT red[STEP];
    __shared__ int nlong, longs[32];
    const int sub = threadIdx.x / LANES, l = threadIdx.x % LANES;  // STEP rows at a time
    const int r0 = bounds[blockIdx.x], r1 = bounds[blockIdx.x + 1];
    for (int p = 0; p < npanel; ++p) {
        const i64 pb = (i64)p * SPMV_PANEL;
        const int width = (int)min((i64)SPMV_PANEL, ncol - pb);
        __syncthreads();
        if (threadIdx.x == 0) nlong = 0, xs[SPMV_PANEL] = (XT)0;
        for (int t = threadIdx.x; t < width; t += NT) xs[t] = X[pb + t];
        __syncthreads();
        // entries [beg, beg + len) of a row in this panel
        auto segment = [&](int row, i64 &beg, int &len) {
            beg = 0, len = 0;
            if (row >= r1) return;
            const i64 a = rowptr[row];
            beg = p ? a + split[(i64)row * (npanel - 1) + p - 1] : a;
            const i64 end = p + 1 < npanel ? a + split[(i64)row * (npanel - 1) + p] : rowptr[row + 1];
            len = (int)(end - beg);
        };
        auto load = [&](i64 beg, int len, int at, int (&c)[U], VT (&v)[U]) {
            const int32_t *cp = cols + beg;
            const VT *vp = vals + beg;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int e = at + l + u * LANES;
                c[u] = (int)((unsigned)pb + SPMV_PANEL);
                v[u] = (VT)0;
                if (e < len) {
                    c[u] = __builtin_nontemporal_load(&cp[e]);
                    v[u] = __builtin_nontemporal_load(&vp[e]);
                }
            }
        };
        auto dot = [&](const int (&c)[U], const VT (&v)[U]) {
            XT s = (XT)0;
#pragma unroll
            for (int u = 0; u < U; ++u) s += (XT)v[u] * xs[(unsigned)c[u] - (unsigned)pb];
            return s;
        };
        int row = r0 + sub;
        i64 beg, nbeg;
        int len, nlen;
        segment(row, beg, len);
        segment(row + STEP, nbeg, nlen);
        XT y = (p && row < r1) ? Y[row] : (XT)0;
        int c[U], cn[U];
        VT v[U], vn[U];
        load(beg, len, 0, c, v);
        for (; row < r1; row += STEP) {
            const int nrow = row + STEP;
            load(nbeg, nlen, 0, cn, vn);
            i64 b2;
            int l2;
            segment(nrow + STEP, b2, l2);
            const XT yn = (p && nrow < r1) ? Y[nrow] : (XT)0;
            if (len > long_len) {
                if (l == 0) longs[atomicAdd(&nlong, 1)] = row;
            } else {
                XT s = dot(c, v);
                for (int at = U * LANES; at < len; at += U * LANES) {
                    int ce[U];
                    VT ve[U];
                    load(beg, len, at, ce, ve);
                    s += dot(ce, ve);
                }
                s = lanes_sum<LANES>(s);
                if (l == 0) Y[row] = y + s;
            }
            beg = nbeg, len = nlen, nbeg = b2, nlen = l2, y = yn;
#pragma unroll
            for (int u = 0; u < U; ++u) c[u] = cn[u], v[u] = vn[u];
        }
        __syncthreads();
        for (int t = 0; t < nlong; ++t) {
            const int lr = longs[t];
            segment(lr, beg, len);
            XT s = (XT)0;
            for (int at = sub * U * LANES; at < len; at += STEP * U * LANES) {
                load(beg, len, at, c, v);
                s += dot(c, v);
            }
            s = lanes_sum<LANES>(s);
            if (l == 0) red[sub] = s;
            __syncthreads();
            if (threadIdx.x == 0) {
                XT all = p ? Y[lr] : (XT)0;
                for (int w = 0; w < STEP; ++w) all += red[w];
                Y[lr] = all;
            }
            __syncthreads();
        }
    }
}

// Plan of k_spmv_lds: split[row][p - 1] = entries of a row with column < p SPMV_PANEL, and
// bounds[b] = first row of block b (rows by their first entry in equal shares of nnz).
__global__ void k_spmv_split(i64 nrow, int npanel, const i64 *rowptr, const int32_t *cols, int32_t *split) {
    const i64 t = (i64)blockIdx.x * 256 + threadIdx.x;
    if (t >= nrow * (npanel - 1)) return;
    const i64 row = t / (npanel - 1), limit = (t - row * (npanel - 1) + 1) * SPMV_PANEL;
    const i64 beg = rowptr[row];
    i64 lo = beg, hi = rowptr[row + 1];
    while (lo < hi) {
        const i64 mid = (lo + hi) >> 1;
        if ((i64)cols[mid] < limit)
            lo = mid + 1;
        else
            hi = mid;
    }
    split[t] = (int32_t)(lo - beg);
}

__global__ void k_spmv_bounds(i64 nrow, i64 nnz, int nblk, const i64 *rowptr, int *bounds) {
    const int b = blockIdx.x * 64 + threadIdx.x;
    if (b > nblk) return;
    const i64 want = (i64)((__int128)nnz * b / nblk);
    i64 lo = 0, hi = nrow;
    while (lo < hi && b < nblk) {
        const i64 mid = (lo + hi) >> 1;
        if (rowptr[mid] < want)
            lo = mid + 1;
        else
            hi = mid;
    }
    bounds[b] = (int)(b < nblk ? lo : nrow);
}

// Generic nvec: loops over vector chunks of 8.
template <typename VT, typename XT>
__global__ void __launch_bounds__(256) k_spmm_any(i64 nrow, i64 nblocks, int nv, const i64 *__restrict__ rowptr,
                                                  const int32_t *__restrict__ cols, const VT *__restrict__ vals,
                                                  const XT *__restrict__ X, XT *__restrict__ Y) {
    const int lane = threadIdx.x & 63;
    const i64 blk = xcd_row_block(blockIdx.x, nblocks);
    const i64 row = blk * SPMV_WAVES + (threadIdx.x >> 6);
    if (blk >= nblocks || row >= nrow) return;
    const i64 beg = rowptr[row], end = rowptr[row + 1];
    for (int j0 = 0; j0 < nv; j0 += 8) {
        const int cnt = min(8, nv - j0);
        XT acc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = (XT)0;
        for (i64 p = beg + lane; p < end; p += 64) {
            const int c = cols[p];
            const XT v = (XT)vals[p];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (j < cnt) acc[j] += v * X[(i64)c * nv + j0 + j];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            XT v = acc[j];
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
            acc[j] = v;
        }
        if (lane < cnt) {
            XT out = acc[0];
#pragma unroll
            for (int j = 1; j < 8; ++j)
                if (lane == j) out = acc[j];
            Y[row * nv + j0 + lane] = out;
        }
    }
}

template <int LANES, typename XT>
static void allow_lds() {
    PE_HIP(hipFuncSetAttribute((const void *)k_spmv_lds<LANES, XT, XT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)(sizeof(XT) * (SPMV_PANEL + 1))));
}

// Which single-vector product serves an operator's rows, and the plan of the one that
// needs one. Called when the rows are final (the operator's build).
void spmv_plan(pyci_op *op, bool column_ordered_space) {
    SpmvPlan &P = op->spmv;
    P = SpmvPlan();
    P.ordered = column_ordered_space;
    const i64 nrow = op->nrow, npanel = (op->ncol + SPMV_PANEL - 1) / SPMV_PANEL;
    if (column_ordered_space || nrow < 1 || op->nnz < SPMV_LDS_MIN_NNZ || op->nnz / (nrow * npanel) < SPMV_LDS_MIN_SEG ||
        nrow >= ((i64)1 << 31))
        return;
    hipStream_t s = op->ctx->stream;
    int cus = 0;
    PE_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, op->ctx->device));
    // a kernel's attribute belongs to a device: set for the operator's with every plan
    allow_lds<16, double>();
    allow_lds<64, double>();
    allow_lds<16, float>();
    allow_lds<64, float>();
    try {
        P.bounds.alloc((size_t)(cus + 1));
        P.split.alloc((size_t)(nrow * (npanel - 1)));  // up to 1 % of the entries' bytes
    } catch (const EngineError &e) {
        if (e.code != PYCI_ENOMEM) throw;
        (void)hipGetLastError();
        P = SpmvPlan();  // the product without panels serves any operator
        return;
    }
    P.npanel = (int)npanel;
    P.nblk = cus;
    k_spmv_bounds<<<grid_for(cus + 1, 64), 64, 0, s>>>(nrow, op->nnz, cus, op->rowptr.p, P.bounds.p);
    PE_LAUNCH_CHECK();
    if (npanel > 1) {
        k_spmv_split<<<grid_for(nrow * (npanel - 1), 256), 256, 0, s>>>(nrow, (int)npanel, op->rowptr.p, op->cols.p,
                                                                       P.split.p);
        PE_LAUNCH_CHECK();
    }
}

template <int LANES, typename VT, typename XT>
static void launch_lds(const pyci_op *op, const VT *vals, const XT *X, XT *Y, hipStream_t s) {
    const size_t lds = sizeof(XT) * (SPMV_PANEL + 1);
    const SpmvPlan &P = op->spmv;
    // at most 25 rows of a block are longer than a 24th of its share
    const i64 long_len = std::max<i64>(1024, op->nnz / ((i64)P.nblk * 24));
    k_spmv_lds<LANES, VT, XT><<<(unsigned)P.nblk, SPMV_LDS_WAVES * 64, lds, s>>>(
        op->ncol, P.npanel, op->rowptr.p, P.split.p, P.bounds.p, long_len, op->cols.p, vals, X, Y);
    PE_LAUNCH_CHECK();
}

template <typename VT, typename XT>
static void spmv(const pyci_op *op, const VT *vals, const XT *X, XT *Y, hipStream_t s) {
    const i64 nrow = op->nrow, mean = op->nnz / nrow;
    const i64 *rp = op->rowptr.p;
    const int32_t *c = op->cols.p;
    const SpmvPlan &P = op->spmv;
    if (P.npanel > 0) {
        // 16 lanes a row take 64 rows at a time with a quarter of the instructions per entry
        // (60,000 GenCI determinants 119 us, 160 with a wave a row). With few rows a block the
        // last of its rounds is mostly empty, and a wave a row is the better one where a row's
        // entries of a panel keep it busy (17,317 FullCI determinants 31 us, 22.5; 10,000
        // GenCI ones of 426 entries 14.6, 13.0), not where they leave most of it idle (30,000
        // FullCI ones of 2 x 41 entries 16.3, 29.4; the two meet near 200)
        if (nrow >= (i64)P.nblk * 160 || op->nnz < nrow * P.npanel * 200)
            launch_lds<16, VT, XT>(op, vals, X, Y, s);
        else
            launch_lds<64, VT, XT>(op, vals, X, Y, s);
        return;
    }
    auto launch = [&](auto kern, int waves) {
        const i64 nblocks = (nrow + waves - 1) / waves, grid = ((nblocks + NUM_XCD - 1) / NUM_XCD) * NUM_XCD;
        kern<<<(unsigned)grid, waves * 64, 0, s>>>(nrow, nblocks, rp, c, vals, X, Y);
        PE_LAUNCH_CHECK();
    };
    // below 4,096 rows blocks of 16 would not reach every CU
    if ((P.ordered && nrow >= 32768) || (mean <= 100 && nrow >= 4096))
        launch(k_spmv<1, 16, VT, XT>, 16);
    else
        launch(k_spmv<3, 4, VT, XT>, 4);
}

template <typename VT, typename XT>
static void spmm(const pyci_op *op, const VT *vals, int nvec, const XT *X, XT *Y, hipStream_t s) {
    const i64 nrow = op->nrow;
    if (nrow <= 0) return;
    const i64 nblocks = (nrow + SPMV_WAVES - 1) / SPMV_WAVES;
    const i64 grid = ((nblocks + NUM_XCD - 1) / NUM_XCD) * NUM_XCD;
    const i64 *rp = op->rowptr.p;
    const int32_t *c = op->cols.p;
    switch (nvec) {
        case 1: spmv<VT, XT>(op, vals, X, Y, s); return;
        case 2:
            // two FP64 values are one 16-byte piece; two FP32 values are not
            if constexpr (sizeof(XT) == 8)
                k_spmm<2, 4, VT, XT><<<(unsigned)grid, 256, 0, s>>>(nrow, nblocks, rp, c, vals, X, Y);
            else
                k_spmm_any<VT, XT><<<(unsigned)grid, 256, 0, s>>>(nrow, nblocks, nvec, rp, c, vals, X, Y);
            break;
        case 4: k_spmm<4, 4, VT, XT><<<(unsigned)grid, 256, 0, s>>>(nrow, nblocks, rp, c, vals, X, Y); break;
        case 8: k_spmm<8, 4, VT, XT><<<(unsigned)grid, 256, 0, s>>>(nrow, nblocks, rp, c, vals, X, Y); break;
        default: k_spmm_any<VT, XT><<<(unsigned)grid, 256, 0, s>>>(nrow, nblocks, nvec, rp, c, vals, X, Y); break;
    }
    PE_LAUNCH_CHECK();
}

void sigma_f64(const pyci_op *op, int nvec, const double *X, double *Y, hipStream_t s, int sector,
               DevBuf<unsigned char> *ws) {
    if (op->storage == PYCI_STORAGE_DIRECT) return direct_sigma<double>(op, nvec, X, Y, s, nullptr, sector, ws);
    spmm<double, double>(op, op->vals.p, nvec, X, Y, s);
}

void sigma_f32(const pyci_op *op, int nvec, const float *X, float *Y, hipStream_t s, int sector,
               DevBuf<unsigned char> *ws) {
    if (op->storage == PYCI_STORAGE_DIRECT) return direct_sigma<float>(op, nvec, X, Y, s, nullptr, sector, ws);
    spmm<float, float>(op, op->vals32.p, nvec, X, Y, s);
}

__global__ void k_to_f32(const double *a, float *b, i64 n) {
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x)
        b[i] = (float)a[i];
}

void ensure_vals32(pyci_op *op) {
    if (op->storage == PYCI_STORAGE_DIRECT) return;  // the matrix-free operator has FP32 integrals of its own
    if (op->vals32.p && op->vals32.n >= (size_t)op->nnz) return;
    op->vals32.alloc((size_t)op->nnz);
    if (op->nnz > 0) {
        k_to_f32<<<4096, 256, 0, op->ctx->stream>>>(op->vals.p, op->vals32.p, op->nnz);
        PE_LAUNCH_CHECK();
    }
}

}  // namespace pe

namespace pe {

__global__ void k_fill_random(double *x, i64 n, u64 seed) {
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x)
        x[i] = (double)(mix64(seed + (u64)i) >> 11) * 0x1p-53 - 0.5;
}

// Times nrep launches of the sigma kernel with HIP events on the context stream.
// Algorithmic bytes of one launch: every stored entry's column index and value,
// the row pointers, one read of X and one write of Y. For the matrix-free
// operator: one read of X, one write of Y, and one write and one read each of
// the pair-indexed intermediates D and E (npair values per determinant and vector).
void op_bench_sigma(pyci_op *op, i64 nvec, i64 nrep, int fp32, float *avg_ms, double *bytes) {
    hipStream_t s = op->ctx->stream;
    const i64 nr = op->nrow, nc = op->ncol;
    PE_REQUIRE(nvec >= 1 && nrep >= 1, PYCI_EINVAL, "nvec and nrep must be >= 1");
    const int vb = fp32 ? 4 : 8;
    if (fp32) ensure_vals32(op);
    DevBuf<double> x((size_t)(nc * nvec)), y((size_t)(nr * nvec));
    DevBuf<float> x32, y32;
    k_fill_random<<<1024, 256, 0, s>>>(x.p, nc * nvec, 12345);
    PE_LAUNCH_CHECK();
    if (fp32) {
        x32.alloc((size_t)(nc * nvec));
        y32.alloc((size_t)(nr * nvec));
        k_to_f32<<<1024, 256, 0, s>>>(x.p, x32.p, nc * nvec);
        PE_LAUNCH_CHECK();
    }
    auto launch = [&] {
        if (fp32)
            sigma_f32(op, (int)nvec, x32.p, y32.p, s);
        else
            sigma_f64(op, (int)nvec, x.p, y.p, s);
    };
    launch();  // warm-up
    PE_HIP(hipEventRecord(op->ctx->ev0, s));
    for (i64 r = 0; r < nrep; ++r) launch();
    PE_HIP(hipEventRecord(op->ctx->ev1, s));
    PE_HIP(hipEventSynchronize(op->ctx->ev1));
    float ms = 0.f;
    PE_HIP(hipEventElapsedTime(&ms, op->ctx->ev0, op->ctx->ev1));
    *avg_ms = ms / (float)nrep;
    if (op->storage == PYCI_STORAGE_DIRECT)
        *bytes = (double)vb * (double)nvec * (double)nr * (2.0 + 4.0 * (double)op->direct->npair);
    else
        *bytes = (double)op->nnz * (4.0 + vb) + 8.0 * (double)(nr + 1) + (double)vb * (double)nvec * (double)(nc + nr);
}

}  // namespace pe
