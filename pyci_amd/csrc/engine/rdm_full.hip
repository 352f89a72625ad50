// One- and two-particle density matrices of a state over the full FullCI space.
//
// Reference: compute_rdms for FullCIWfn (rdm.cpp:269-530). With the determinants in
// colex order the vector is a matrix C[alpha string][beta string], and every element
// is a contraction of that matrix instead of a scatter from each pair of determinants:
//
//   same spin   gamma = C C^T (alpha; C^T C for beta) is one matrix product, and
//               <a+_p a_r>, <a+_p a+_q a_s a_r> are sums of gamma[I][J] over the pairs of
//               strings that one or two excitations connect (k_gamma, k_same);
//   two spins   abab[p,q,r,s] = <E_pr E_qs> is, for each alpha string I, the product of
//               the rows C[J] of the strings J = E_pr I (nup (n - nup + 1) of them) with
//               the matrix Y[qs][K] = sum_K' <K|E_qs|K'> C[I][K'] (k_abab). Only q <= s is
//               formed: abab[p,q,r,s] = abab[r,s,p,q] for real vectors.
//
// All products run on v_mfma_f64_16x16x4f64. At nbasis 12 (6 alpha, 6 beta) the
// contractions are 6.9 GF (two spins) + 1.7 GF (same spin); the scatter kernel of
// rdm.hip, which stays for every other set, needs about 3e9 FP64 atomics there.
#include <algorithm>
#include <cmath>

#include "internal.hpp"
#include "rdm.hpp"

namespace pe {

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ inline f64x4 mfma4(double a, double b, f64x4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ inline u64 rf_string(int r, int n, int k, const i64 *binom) {
    u64 s = 0;
    i64 rank = r;
    for (int p = n - 1; k >= 1; --k, --p) {
        while (binom[p * 65 + k] > rank) --p;
        s |= 1ULL << p;
        rank -= binom[p * 65 + k];
    }
    return s;
}

__device__ inline int rf_bit(u64 x, int t) {
    for (int s = 0; s < t; ++s) x &= x - 1;
    return __builtin_ctzll(x);
}

// C and its transpose with padded rows, through a 32 x 32 LDS tile.
__global__ void __launch_bounds__(256) k_rf_pad(RfShape S, const double *__restrict__ c, double *__restrict__ C,
                                                double *__restrict__ Ct) {
    __shared__ double t[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int j0 = blockIdx.x * 32, i0 = blockIdx.y * 32;
    for (int y = ty; y < 32; y += 8) {
        const int i = i0 + y, j = j0 + tx;
        const double v = (i < S.na && j < S.nb) ? c[(i64)i * S.nb + j] : 0.0;
        if (i < S.na && j < S.ldc) C[(i64)i * S.ldc + j] = v;
        t[y][tx] = v;
    }
    __syncthreads();
    for (int y = ty; y < 32; y += 8) {
        const int j = j0 + y, i = i0 + tx;
        if (j < S.nb && i < S.ldt) Ct[(i64)j * S.ldt + i] = t[tx][y];
    }
}

// tab[qs][K] = rank of E_sq K | (negative phase) << 15, or nb (a zero of the staged row)
// where q is empty or s is occupied in K; pairs q <= s at s (s + 1) / 2 + q, rows past npr
// and strings past nb hold nb. The accumulators are cleared beside it.
__global__ void k_rf_table(RfShape S, int rows, uint16_t *__restrict__ tab, i64 nacc, double *__restrict__ acc) {
    const i64 e = (i64)blockIdx.x * 256 + threadIdx.x;
    if (e < nacc) acc[e] = 0.0;
    if (e >= (i64)rows * S.ldc) return;
    const int pair = (int)(e / S.ldc), K = (int)(e - (i64)pair * S.ldc);
    unsigned v = (unsigned)S.nb;
    if (pair < S.npr && K < S.nb) {
        int s = (int)((sqrtf(8.0f * (float)pair + 1.0f) - 1.0f) * 0.5f);
        while (s * (s + 1) / 2 > pair) --s;
        while ((s + 1) * (s + 2) / 2 <= pair) ++s;
        const int q = pair - s * (s + 1) / 2;
        const u64 d = rf_string(K, S.n, S.ndn, S.binom);
        if (((d >> q) & 1) && (q == s || !((d >> s) & 1))) {
            v = (unsigned)K;
            if (q != s)
                v = (unsigned)colex_rank(d ^ (1ULL << q) ^ (1ULL << s), S.binom) |
                    (phase1(d, q, s) < 0 ? 0x8000u : 0u);
        }
    }
    tab[e] = (uint16_t)v;
}

// Four consecutive elements of a row for each lane: the lane quarter g = lane / 16 takes
// elements 4g .. 4g+3 of a chunk of 16, and MFMA step j multiplies element j of each
// quarter. Both operands use this order, so each row is read in whole 128-byte pieces.
__device__ inline void load4(const double *p, double v[4]) {
    const double2 a = reinterpret_cast<const double2 *>(p)[0], b = reinterpret_cast<const double2 *>(p)[1];
    v[0] = a.x, v[1] = a.y, v[2] = b.x, v[3] = b.y;
}

// gamma = M M^T on and above the block diagonal, 64 x 64 per block and 32 x 32 per wave,
// operands straight from L2 (a chunk of 16 columns feeds 16 MFMAs of 64 cycles, so one
// chunk of lookahead covers the loads). Blocks of both spins run in one launch. Bound by
// the matrix cores' latency chain at these sizes: 240 blocks at nbasis 12.
__global__ void __launch_bounds__(256) k_rf_gamma(RfShape S, const double *__restrict__ C,
                                                  const double *__restrict__ Ct, double *__restrict__ ga,
                                                  double *__restrict__ gb) {
    const int ta = (S.na + 63) / 64, ntri = ta * (ta + 1) / 2;
    const bool beta = (int)blockIdx.x >= ntri;
    const int t = beta ? (int)blockIdx.x - ntri : (int)blockIdx.x;
    int tj = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while (tj * (tj + 1) / 2 > t) --tj;
    while ((tj + 1) * (tj + 2) / 2 <= t) ++tj;
    const int ti = t - tj * (tj + 1) / 2;
    const int rows = beta ? S.nb : S.na, ld = beta ? S.ldt : S.ldc;
    const double *M = beta ? Ct : C;
    double *g = beta ? gb : ga;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
    const int i0 = ti * 64 + (wave >> 1) * 32, j0 = tj * 64 + (wave & 1) * 32;
    const double *pa[2], *pb[2];
    for (int m = 0; m < 2; ++m) {
        pa[m] = M + (i64)min(i0 + 16 * m + lr, rows - 1) * ld + 4 * lk;
        pb[m] = M + (i64)min(j0 + 16 * m + lr, rows - 1) * ld + 4 * lk;
    }
    f64x4 acc[2][2] = {};
    double a[2][4], b[2][4];
    for (int m = 0; m < 2; ++m) load4(pa[m], a[m]), load4(pb[m], b[m]);
    for (int k = 0; k < ld; k += 16) {
        double an[2][4], bn[2][4];
        const int kn = k + 16 < ld ? k + 16 : 0;
        for (int m = 0; m < 2; ++m) load4(pa[m] + kn, an[m]), load4(pb[m] + kn, bn[m]);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int u = 0; u < 2; ++u) acc[m][u] = mfma4(a[m][q], b[u][q], acc[m][u]);
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int q = 0; q < 4; ++q) a[m][q] = an[m][q], b[m][q] = bn[m][q];
    }
    for (int m = 0; m < 2; ++m)
        for (int u = 0; u < 2; ++u)
            for (int r = 0; r < 4; ++r) {
                const int i = i0 + 16 * m + 4 * r + lk, j = j0 + 16 * u + lr;
                if (i < rows && j < rows) g[(i64)i * rows + j] = acc[m][u][r];
            }
}

// Same-spin elements from gamma: one block per string I, a thread per string J >= I that
// at most two excitations connect with it. Each unordered pair of strings is added once;
// k_rf_expand forms both orders and the antisymmetric images.
__global__ void __launch_bounds__(256) k_rf_same(RfShape S, const double *__restrict__ ga,
                                                 const double *__restrict__ gb, int R, double *__restrict__ acc) {
    const bool beta = (int)blockIdx.x >= S.na;
    const int I = beta ? (int)blockIdx.x - S.na : (int)blockIdx.x;
    const int n = S.n, no = beta ? S.ndn : S.nup, nv = n - no, rows = beta ? S.nb : S.na;
    const double *g = (beta ? gb : ga) + (i64)I * rows;
    double *base = acc + (i64)(blockIdx.x % R) * S.stride;
    double *one = base + (beta ? n * n : 0), *two = base + (beta ? S.obb : S.oaa);
    const int npd = S.npd;
    auto pair = [&](int p, int q) { return p < q ? q * (q - 1) / 2 + p : p * (p - 1) / 2 + q; };
    const u64 d = rf_string(I, n, no, S.binom), e = ~d & full_mask(n);
    const double v0 = g[I];
    for (int t = threadIdx.x; t < no * no; t += 256) {
        const int p = rf_bit(d, t / no), q = rf_bit(d, t % no);
        if (p == q)
            atomicAdd(&one[p * n + p], v0);
        else if (p < q)
            atomicAdd(&two[(i64)pair(p, q) * npd + pair(p, q)], v0);
    }
    const int ns = no * nv, npv = nv * (nv - 1) / 2, nd = (no * (no - 1) / 2) * npv;
    for (int t = threadIdx.x; t < ns + nd; t += 256) {
        if (t < ns) {
            const int i = rf_bit(d, t / nv), a = rf_bit(e, t % nv);
            const int J = (int)colex_rank(d ^ (1ULL << i) ^ (1ULL << a), S.binom);
            if (J < I) continue;
            const double v = g[J] * phase1(d, i, a);
            atomicAdd(&one[i * n + a], v);
            for (u64 x = d; x; x &= x - 1) {
                const int q = __builtin_ctzll(x);
                if (q == i) continue;
                const bool neg = (i < q) != (a < q);
                atomicAdd(&two[(i64)pair(i, q) * npd + pair(a, q)], neg ? -v : v);
            }
        } else {
            int i, k, a, l;
            tri_decode((t - ns) / npv, i, k);
            tri_decode((t - ns) % npv, a, l);
            i = rf_bit(d, i), k = rf_bit(d, k), a = rf_bit(e, a), l = rf_bit(e, l);
            const int J = (int)colex_rank(d ^ (1ULL << i) ^ (1ULL << k) ^ (1ULL << a) ^ (1ULL << l), S.binom);
            if (J > I) atomicAdd(&two[(i64)pair(i, k) * npd + pair(a, l)], g[J] * phase2(d, i, k, a, l));
        }
    }
}

// Two-spin elements: one block per alpha string I (and chunk of MT x 16 of its rows E_pr I
// and NT x 16 pairs qs). C[I] is staged in LDS with a zero behind it; the waves split the
// beta strings in chunks of 16, read the rows C[J] from L2 and gather Y[qs][K] from the
// staged row through the table, so no barrier stands between the first and the last MFMA.
// The waves' sums meet in LDS and go out as one atomic per element and block (3e6 at
// nbasis 12, into R copies). MT x NT of 3 x 5 is what the registers hold beside the next
// chunk's operands (120 accumulator registers) and covers nbasis 12 in one piece.
template <int MT, int NT>
__global__ void __launch_bounds__(256) k_rf_abab(RfShape S, const double *__restrict__ C,
                                                 const uint16_t *__restrict__ tab, int nchunk, int R,
                                                 double *__restrict__ acc_out) {
    extern __shared__ double lds[];  // C[I] and a zero, later the block's sums
    __shared__ int jrank[MT * 16], jout[MT * 16];
    const int I = blockIdx.x, mc = blockIdx.y / nchunk, nc = blockIdx.y - mc * nchunk;
    const int n = S.n, nv = n - S.nup, live = S.nup * (nv + 1);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
    if ((int)threadIdx.x < MT * 16) {
        const int t = mc * MT * 16 + (int)threadIdx.x;
        int rank = I, out = -1;
        if (t < live) {
            const u64 d = rf_string(I, n, S.nup, S.binom);
            const int r = rf_bit(d, t / (nv + 1)), v = t % (nv + 1);
            const int p = v ? rf_bit(~d & full_mask(n), v - 1) : r;
            out = (p * n + r) * 2;
            if (p != r) {
                rank = (int)colex_rank(d ^ (1ULL << p) ^ (1ULL << r), S.binom);
                out |= phase1(d, r, p) < 0;
            }
        }
        jrank[threadIdx.x] = rank;
        jout[threadIdx.x] = out;
    }
    for (int k = threadIdx.x; k <= S.nb; k += 256) lds[k] = k < S.nb ? C[(i64)I * S.ldc + k] : 0.0;
    __syncthreads();
    const double *pa[MT];
    const uint16_t *pt[NT];
#pragma unroll
    for (int m = 0; m < MT; ++m) pa[m] = C + (i64)jrank[m * 16 + lr] * S.ldc + 4 * lk;
#pragma unroll
    for (int u = 0; u < NT; ++u) pt[u] = tab + (i64)((nc * NT + u) * 16 + lr) * S.ldc + 4 * lk;
    f64x4 acc[MT][NT] = {};
    double a[MT][4], an[MT][4];
    uint2 w[NT], wn[NT];
    const int kfirst = 16 * wave;
    if (kfirst < S.ldc) {
#pragma unroll
        for (int m = 0; m < MT; ++m) load4(pa[m] + kfirst, a[m]);
#pragma unroll
        for (int u = 0; u < NT; ++u) w[u] = *reinterpret_cast<const uint2 *>(pt[u] + kfirst);
    }
    for (int k = kfirst; k < S.ldc; k += 64) {
        const int kn = k + 64 < S.ldc ? k + 64 : kfirst;
#pragma unroll
        for (int m = 0; m < MT; ++m) load4(pa[m] + kn, an[m]);
#pragma unroll
        for (int u = 0; u < NT; ++u) wn[u] = *reinterpret_cast<const uint2 *>(pt[u] + kn);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            double b[NT];
#pragma unroll
            for (int u = 0; u < NT; ++u) {
                const unsigned h = ((q & 2) ? w[u].y : w[u].x) >> (16 * (q & 1));
                const double v = lds[h & 0x7fffu];
                b[u] = (h & 0x8000u) ? -v : v;
            }
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int u = 0; u < NT; ++u) acc[m][u] = mfma4(a[m][q], b[u], acc[m][u]);
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int q = 0; q < 4; ++q) a[m][q] = an[m][q];
#pragma unroll
        for (int u = 0; u < NT; ++u) w[u] = wn[u];
    }
    __syncthreads();
    for (int t = threadIdx.x; t < MT * NT * 256; t += 256) lds[t] = 0.0;
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                atomicAdd(&lds[(16 * m + 4 * r + lk) * (NT * 16) + 16 * u + lr], acc[m][u][r]);
    __syncthreads();
    double *base = acc_out + (i64)(blockIdx.x % R) * S.stride + S.oab;
    for (int t = threadIdx.x; t < MT * NT * 256; t += 256) {
        const int row = t / (NT * 16), pair = nc * NT * 16 + t % (NT * 16), out = jout[row];
        if (out >= 0 && pair < S.npr) atomicAdd(&base[(i64)(out >> 1) * S.npr + pair], (out & 1) ? -lds[t] : lds[t]);
    }
}

// The reference's arrays from the accumulators (FullCI: rdm1 aa, bb; rdm2 aaaa, bbbb, abab;
// GenCI: rdm1, rdm2 of the one string).
__global__ void k_rf_expand(RfShape S, int R, const double *__restrict__ acc, double *__restrict__ out) {
    const i64 n = S.n, n2 = n * n, n4 = n2 * n2, none = (S.genci ? 1 : 2) * n2;
    const i64 t = (i64)blockIdx.x * 256 + threadIdx.x;
    if (t >= none + (S.genci ? 1 : 3) * n4) return;
    i64 at0, at1 = -1;
    double sign = 1.0;
    if (t < none) {
        const i64 x = t % n2, p = x / n, q = x - p * n;
        at0 = t;
        if (p != q) at1 = t - x + q * n + p;
    } else {
        const i64 u = t - none, blk = u / n4, x = u - blk * n4;
        int p = (int)(x / (n2 * n)), q = (int)(x / n2 % n), r = (int)(x / n % n), s = (int)(x % n);
        if (blk < 2) {
            if (p == q || r == s) {
                out[t] = 0.0;
                return;
            }
            if (p > q) {
                const int y = p;
                p = q, q = y, sign = -sign;
            }
            if (r > s) {
                const int y = r;
                r = s, s = y, sign = -sign;
            }
            const i64 P = q * (q - 1) / 2 + p, Q = s * (s - 1) / 2 + r, o = blk ? S.obb : S.oaa;
            at0 = o + P * S.npd + Q;
            if (P != Q) at1 = o + Q * S.npd + P;
        } else {
            if (q > s) {
                int y = q;
                q = s, s = y;
                y = p, p = r, r = y;
            }
            at0 = S.oab + ((i64)p * n + r) * S.npr + s * (s + 1) / 2 + q;
        }
    }
    double v = 0.0;
    for (int c = 0; c < R; ++c) {
        v += acc[(i64)c * S.stride + at0];
        if (at1 >= 0) v += acc[(i64)c * S.stride + at1];
    }
    out[t] = sign * v;
}

// Fills the sizes and the accumulator layout; C's strides are the full-space contractions' own.
RfShape rf_shape(const pyci_wfn *w) {
    RfShape S{};
    S.n = (int)w->nbasis, S.nup = (int)w->nup, S.ndn = (int)w->ndn;
    S.genci = w->kind == PYCI_WFN_GENCI;
    S.npd = S.n * (S.n - 1) / 2, S.npr = S.n * (S.n + 1) / 2;
    S.binom = w->ctx->binom.p;
    const i64 n2 = (i64)S.n * S.n, npd2 = (i64)S.npd * S.npd;
    S.oaa = S.genci ? n2 : 2 * n2, S.obb = S.oaa + npd2;
    S.oab = S.genci ? S.obb : S.obb + npd2;
    S.stride = S.genci ? S.obb : S.oab + n2 * S.npr;
    return S;
}

int rf_copies(const RfShape &S) {
    return (int)std::max<i64>(1, std::min<i64>(4, ((i64)256 << 20) / (S.stride * 8)));
}

// Expands the accumulators and brings the result to the caller: straight into page-locked memory
// of the context (one synchronisation and no staged copies); beyond 16 MB (FullCI nbasis
// 29, GenCI 38), or where there is none to be had, through device memory.
void rf_result(pyci_ctx *ctx, const RfShape &S, int R, const double *acc, double *rdm1, double *rdm2) {
    hipStream_t s = ctx->stream;
    const i64 n2 = (i64)S.n * S.n, s1 = (S.genci ? 1 : 2) * n2, nout = s1 + (S.genci ? 1 : 3) * n2 * n2;
    bool direct = nout <= (i64)2 << 20;
    DevBuf<double> dout;
    Lease<HostBuf<double>> out(ctx->rdm_out);
    HostBuf<double> &host = out.buf;
    if (direct) {
        try {
            host.ensure((size_t)nout);
        } catch (const EngineError &) {
            (void)hipGetLastError();
            direct = false;
        }
    }
    if (!direct) dout.alloc((size_t)nout);
    k_rf_expand<<<grid_for(nout, 256), 256, 0, s>>>(S, R, acc, direct ? host.p : dout.p);
    PE_LAUNCH_CHECK();
    if (direct) {
        PE_HIP(hipStreamSynchronize(s));
        std::copy(host.p, host.p + s1, rdm1);
        std::copy(host.p + s1, host.p + nout, rdm2);
    } else {
        PE_HIP(hipMemcpyAsync(rdm1, dout.p, sizeof(double) * s1, hipMemcpyDeviceToHost, s));
        PE_HIP(hipMemcpyAsync(rdm2, dout.p + s1, sizeof(double) * (nout - s1), hipMemcpyDeviceToHost, s));
        PE_HIP(hipStreamSynchronize(s));
    }
}

template <int MT>
static void launch_abab(int nt, dim3 grid, size_t lds, hipStream_t s, const RfShape &S, const double *C,
                        const uint16_t *tab, int nchunk, int R, double *acc) {
    switch (nt) {
        case 1: k_rf_abab<MT, 1><<<grid, 256, lds, s>>>(S, C, tab, nchunk, R, acc); break;
        case 2: k_rf_abab<MT, 2><<<grid, 256, lds, s>>>(S, C, tab, nchunk, R, acc); break;
        case 3: k_rf_abab<MT, 3><<<grid, 256, lds, s>>>(S, C, tab, nchunk, R, acc); break;
        case 4: k_rf_abab<MT, 4><<<grid, 256, lds, s>>>(S, C, tab, nchunk, R, acc); break;
        default: k_rf_abab<MT, 5><<<grid, 256, lds, s>>>(S, C, tab, nchunk, R, acc); break;
    }
    PE_LAUNCH_CHECK();
}

// Whether the full-space contractions serve this set: the staged row and the table's
// 15-bit index need nb <= 8,000 (64 KB of LDS), gamma of both spins then takes at most
// 1 GB. Per call, scatter kernel against contractions (with the copies of the vector and
// the result): 100 determinants 70 / 38 us, 1,225 85 / 51, 4,900 269 / 60, 15,876 932 / 71,
// 63,504 5,050 / 141, 853,776 121,200 / 535 us.
static bool full_rdm_applies(const pyci_wfn *w) {
    if (w->kind != PYCI_WFN_FULLCI || !w->colex || w->nup < 1 || w->ndn < 1) return false;
    const i64 na = binom_host(w->nbasis, w->nup), nb = binom_host(w->nbasis, w->ndn);
    return na <= 8000 && nb <= 8000;
}

// compute_rdms of a full FullCI space; false where it does not apply or its scratch memory (three
// copies of the vector and the string matrices) is not to be had. A vector with
// infinities or NaNs is left to the scatter kernel as well: in a contraction they would
// reach elements that no connected pair of determinants carries them to.
bool rdms_full_space(pyci_wfn *w, const double *coeffs_host, double *rdm1, double *rdm2) {
    if (!full_rdm_applies(w)) return false;
    hipStream_t s = w->ctx->stream;
    RfShape S = rf_shape(w);
    S.na = (int)binom_host(S.n, S.nup), S.nb = (int)binom_host(S.n, S.ndn);
    S.ldc = (S.nb + 15) & ~15, S.ldt = (S.na + 15) & ~15;
    const int R = rf_copies(S);
    // the rows and pairs of k_rf_abab in equal chunks of at most 3 and 5 tiles
    const int mtiles = (S.nup * (S.n - S.nup + 1) + 15) / 16, ntiles = (S.npr + 15) / 16;
    const int mch = (mtiles + 2) / 3, nch = (ntiles + 4) / 5;
    const int MT = (mtiles + mch - 1) / mch, NT = (ntiles + nch - 1) / nch;
    const int trows = nch * NT * 16;
    const i64 nC = (i64)S.na * S.ldc, nCt = (i64)S.nb * S.ldt, nga = (i64)S.na * S.na, ngb = (i64)S.nb * S.nb;
    const i64 ntab = ((i64)trows * S.ldc + 3) / 4;
    // one allocation: the vector, C and C^T, gamma of both spins, the table, the accumulators
    const i64 nacc = R * S.stride, even = (w->ndet + 1) & ~(i64)1;
    DevBuf<double> buf;
    try {
        buf.alloc((size_t)(even + nC + nCt + nga + ngb + ntab + nacc));
    } catch (const EngineError &e) {
        if (e.code != PYCI_ENOMEM) throw;
        (void)hipGetLastError();  // not to be reported against a later launch
        return false;             // the scatter kernel needs the vector and its accumulators only
    }
    double *c = buf.p, *C = c + even, *Ct = C + nC, *ga = Ct + nCt, *gb = ga + nga;
    double *acc = gb + ngb;
    uint16_t *tab = reinterpret_cast<uint16_t *>(acc + nacc);
    PE_HIP(hipMemcpyAsync(c, coeffs_host, sizeof(double) * w->ndet, hipMemcpyHostToDevice, s));
    const i64 nprep = std::max<i64>((i64)trows * S.ldc, nacc);
    k_rf_table<<<grid_for(nprep, 256), 256, 0, s>>>(S, trows, tab, nacc, acc);
    PE_LAUNCH_CHECK();
    k_rf_pad<<<dim3((S.ldc + 31) / 32, (S.ldt + 31) / 32), 256, 0, s>>>(S, c, C, Ct);
    PE_LAUNCH_CHECK();
    const unsigned ta = (S.na + 63) / 64, tb = (S.nb + 63) / 64;
    k_rf_gamma<<<ta * (ta + 1) / 2 + tb * (tb + 1) / 2, 256, 0, s>>>(S, C, Ct, ga, gb);
    PE_LAUNCH_CHECK();
    k_rf_same<<<(unsigned)(S.na + S.nb), 256, 0, s>>>(S, ga, gb, R, acc);
    PE_LAUNCH_CHECK();
    const size_t lds = sizeof(double) * (size_t)std::max(S.nb + 1, MT * NT * 256);
    const dim3 grid((unsigned)S.na, (unsigned)(mch * nch));
    if (MT == 1)
        launch_abab<1>(NT, grid, lds, s, S, C, tab, nch, R, acc);
    else if (MT == 2)
        launch_abab<2>(NT, grid, lds, s, S, C, tab, nch, R, acc);
    else
        launch_abab<3>(NT, grid, lds, s, S, C, tab, nch, R, acc);
    rf_result(w->ctx, S, R, acc, rdm1, rdm2);
    double trace = 0.0;  // a sum of every squared coefficient
    for (i64 p = 0; p < S.n; ++p) trace += rdm1[p * (S.n + 1)];
    return std::isfinite(trace);
}

}  // namespace pe
