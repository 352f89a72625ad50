// One- and two-particle reduced density matrices on the GPU.
//
// Reference: compute_rdms for DOCIWfn (rdm.cpp:20-65) and FullCIWfn
// (rdm.cpp:269-530; full FullCI spaces are contracted in rdm_full.hip): a loop over
// determinants I that visits every excitation J of I present in the wave function with
// J > I and scatters c_I c_J times the phase into the symmetric index permutations, plus
// the diagonal c_I^2 terms. Selected FullCI and GenCI sets find the connected pairs by
// testing pairs of determinants (k_rdm_pairs); the rest enumerate.
// GenCIWfn is computed from the operator algebra (every ordered pair I, J); the
// reference's GenCI routine (rdm.cpp:532-632) has index errors and is not
// reproduced.
//
// Enumeration: one wavefront per determinant; lanes take excitations from the same flat
// candidate index as the CSR builder. Accumulation uses hardware FP64 atomics
// into R replicated copies of the RDM arrays (block b uses copy b % R) to spread
// contention on hot elements, followed by a reduction over the copies.
#include <algorithm>

#include "internal.hpp"
#include "rdm.hpp"

namespace pe {

__device__ inline void aadd(double *p, double v) { atomicAdd(p, v); }

__device__ inline int nth_bit_r(u64 x, int t) {
    for (int s = 0; s < t && x; ++s) x &= x - 1;
    return x ? __builtin_ctzll(x) : 0;
}

__device__ inline void tri_decode_r(int t, int &i, int &k) {
    int kk = (int)((1.0f + sqrtf(1.0f + 8.0f * (float)t)) * 0.5f);
    while (kk * (kk - 1) / 2 > t) --kk;
    while ((kk + 1) * kk / 2 <= t) ++kk;
    k = kk;
    i = t - kk * (kk - 1) / 2;
}

// 8 antisymmetric images of a same-spin 2-body term X[p,q,r,s] for pair (p,q),(r,s) and its transpose
__device__ inline void same_spin8(double *X, int n, int ii, int kk, int jj, int ll, double v) {
    const i64 n1 = n, n2 = n1 * n1, n3 = n2 * n1;
    aadd(&X[ii * n3 + kk * n2 + jj * n1 + ll], v);
    aadd(&X[ii * n3 + kk * n2 + ll * n1 + jj], -v);
    aadd(&X[kk * n3 + ii * n2 + jj * n1 + ll], -v);
    aadd(&X[kk * n3 + ii * n2 + ll * n1 + jj], v);
    aadd(&X[jj * n3 + ll * n2 + ii * n1 + kk], v);
    aadd(&X[jj * n3 + ll * n2 + kk * n1 + ii], -v);
    aadd(&X[ll * n3 + jj * n2 + ii * n1 + kk], -v);
    aadd(&X[ll * n3 + jj * n2 + kk * n1 + ii], v);
}

// single i->j with spectator k of the same spin (rdm.cpp:331-349 pattern)
__device__ inline void same_spin_single(double *X, int n, int ii, int jj, int kk, double v) {
    const i64 n1 = n, n2 = n1 * n1, n3 = n2 * n1;
    aadd(&X[ii * n3 + kk * n2 + jj * n1 + kk], v);
    aadd(&X[ii * n3 + kk * n2 + kk * n1 + jj], -v);
    aadd(&X[kk * n3 + ii * n2 + kk * n1 + jj], v);
    aadd(&X[kk * n3 + ii * n2 + jj * n1 + kk], -v);
    aadd(&X[jj * n3 + kk * n2 + ii * n1 + kk], v);
    aadd(&X[jj * n3 + kk * n2 + kk * n1 + ii], -v);
    aadd(&X[kk * n3 + jj * n2 + ii * n1 + kk], -v);
    aadd(&X[kk * n3 + jj * n2 + kk * n1 + ii], v);
}

// Flat candidate index of one row (the CSR builder's order): alpha singles, 1-1
// doubles, alpha doubles, beta singles, beta doubles; c0..c4 are the class ends.
template <int KIND>
__device__ inline void exc_bounds(int nou, int nvu, int nod, int nvd, int &c0, int &c1, int &c2, int &c3, int &c4) {
    const int nsu = nou * nvu, nsd = nod * nvd;
    const int npv_u = nvu * (nvu - 1) / 2, npv_d = nvd * (nvd - 1) / 2;
    if (KIND == PYCI_WFN_FULLCI) {
        c0 = nsu;
        c1 = c0 + nsu * nsd;
        c2 = c1 + (nou * (nou - 1) / 2) * npv_u;
        c3 = c2 + nsd;
        c4 = c3 + (nod * (nod - 1) / 2) * npv_d;
    } else if (KIND == PYCI_WFN_DOCI) {
        c0 = c1 = c2 = c3 = c4 = nsu;
    } else {
        c0 = c1 = nsu;
        c2 = c3 = c4 = c1 + (nou * (nou - 1) / 2) * npv_u;
    }
}

// Candidate e of a row: its class and list positions (i, a: first occupied and
// virtual; k, l: second), in the lists each lane holds in `packed`.
__device__ inline void exc_decode(int e, int c0, int c1, int c2, int c3, int nvu, int nod, int nvd, int &cls, int &i,
                                  int &a, int &k, int &l) {
    const int nsd = nod * nvd, npv_u = nvu * (nvu - 1) / 2, npv_d = nvd * (nvd - 1) / 2;
    cls = i = a = k = l = 0;
    if (e < c0) {
        i = e / nvu;
        a = e - i * nvu;
    } else if (e < c1) {
        cls = 1;
        int t = e - c0, ia = t / nsd, kl = t - ia * nsd;
        i = ia / nvu;
        a = ia - i * nvu;
        k = kl / nvd;
        l = kl - k * nvd;
    } else if (e < c2) {
        cls = 2;
        int t = e - c1, po = t / npv_u, pv = t - po * npv_u;
        tri_decode_r(po, i, k);
        tri_decode_r(pv, a, l);
    } else if (e < c3) {
        cls = 3;
        int t = e - c2;
        i = t / nvd;
        a = t - i * nvd;
    } else {
        cls = 4;
        int t = e - c3, po = t / npv_d, pv = t - po * npv_d;
        tri_decode_r(po, i, k);
        tri_decode_r(pv, a, l);
    }
}

template <int KIND>
__global__ void __launch_bounds__(256) k_rdm(WfnView w, const double *c, int R, i64 stride, double *acc) {
    const int lane = threadIdx.x & 63;
    const i64 row = (i64)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= w.ndet) return;
    const int n = w.nb;
    const i64 n1 = n, n2 = n1 * n1, n3 = n2 * n1, n4 = n2 * n2;
    double *base = acc + (i64)(blockIdx.x % R) * stride;
    const u64 m = full_mask(n);
    const u64 up = w.dets[(i64)w.nkey * row];
    const u64 dn = (KIND == PYCI_WFN_FULLCI) ? w.dets[2 * row + 1] : 0ULL;
    const int nou = __popcll(up), nvu = n - nou, nod = __popcll(dn), nvd = n - nod;
    const int packed = nth_bit_r(up, lane) | (nth_bit_r(~up & m, lane) << 8) | (nth_bit_r(dn, lane) << 16) |
                       (nth_bit_r(~dn & m, lane) << 24);
    const double ci = c[row];
    // ---- diagonal terms (lane-parallel over occupied pairs) ----
    const double val1 = ci * ci;
    if (KIND == PYCI_WFN_DOCI) {
        double *d0 = base, *d2 = base + n2;
        for (int t = lane; t < nou * nou; t += 64) {
            const int a = t / nou, b = t - a * nou;
            const int p = nth_bit_r(up, a), q = nth_bit_r(up, b);
            if (a == b)
                aadd(&d0[p * (n + 1)], val1);
            else
                aadd(&d2[p * n1 + q], val1);
        }
    } else if (KIND == PYCI_WFN_FULLCI) {
        double *aa = base, *bb = base + n2, *aaaa = base + 2 * n2, *bbbb = aaaa + n4, *abab = bbbb + n4;
        for (int t = lane; t < nou * nou; t += 64) {
            const int a = t / nou, b = t - a * nou;
            const int p = nth_bit_r(up, a), q = nth_bit_r(up, b);
            if (a == b) {
                aadd(&aa[p * (n + 1)], val1);
            } else if (a < b) {
                aadd(&aaaa[p * n3 + q * n2 + p * n1 + q], val1);
                aadd(&aaaa[p * n3 + q * n2 + q * n1 + p], -val1);
                aadd(&aaaa[q * n3 + p * n2 + p * n1 + q], -val1);
                aadd(&aaaa[q * n3 + p * n2 + q * n1 + p], val1);
            }
        }
        for (int t = lane; t < nod * nod; t += 64) {
            const int a = t / nod, b = t - a * nod;
            const int p = nth_bit_r(dn, a), q = nth_bit_r(dn, b);
            if (a == b) {
                aadd(&bb[p * (n + 1)], val1);
            } else if (a < b) {
                aadd(&bbbb[p * n3 + q * n2 + p * n1 + q], val1);
                aadd(&bbbb[p * n3 + q * n2 + q * n1 + p], -val1);
                aadd(&bbbb[q * n3 + p * n2 + p * n1 + q], -val1);
                aadd(&bbbb[q * n3 + p * n2 + q * n1 + p], val1);
            }
        }
        for (int t = lane; t < nou * nod; t += 64) {
            const int a = t / nod, b = t - a * nod;
            const int p = nth_bit_r(up, a), q = nth_bit_r(dn, b);
            aadd(&abab[p * n3 + q * n2 + p * n1 + q], val1);
        }
    } else {
        double *r1 = base, *r2 = base + n2;
        for (int t = lane; t < nou * nou; t += 64) {
            const int a = t / nou, b = t - a * nou;
            const int p = nth_bit_r(up, a), q = nth_bit_r(up, b);
            if (a == b) {
                aadd(&r1[p * (n + 1)], val1);
            } else {
                aadd(&r2[p * n3 + q * n2 + p * n1 + q], val1);
                aadd(&r2[p * n3 + q * n2 + q * n1 + p], -val1);
            }
        }
    }
    // ---- off-diagonal terms ----
    int c0, c1, c2, c3, c4;
    exc_bounds<KIND>(nou, nvu, nod, nvd, c0, c1, c2, c3, c4);
    for (int e0 = 0; e0 < c4; e0 += 64) {
        const int e = e0 + lane;
        const bool valid = e < c4;
        int cls = 0, i = 0, a = 0, k = 0, l = 0;
        if (valid) exc_decode(e, c0, c1, c2, c3, nvu, nod, nvd, cls, i, a, k, l);
        const int pi = __shfl(packed, i), pa = __shfl(packed, a), pk = __shfl(packed, k), pl = __shfl(packed, l);
        if (!valid) continue;
        const bool alpha = cls <= 2;
        const int ii = alpha ? (pi & 255) : ((pi >> 16) & 255);
        const int jj = alpha ? ((pa >> 8) & 255) : ((pa >> 24) & 255);
        int kk, ll;
        if (cls == 1 || !alpha) {
            kk = (pk >> 16) & 255;
            ll = (pl >> 24) & 255;
        } else {
            kk = pk & 255;
            ll = (pl >> 8) & 255;
        }
        u64 nu = up, nd = dn;
        if (cls == 0) nu = up ^ (1ULL << ii) ^ (1ULL << jj);
        else if (cls == 1) {
            nu = up ^ (1ULL << ii) ^ (1ULL << jj);
            nd = dn ^ (1ULL << kk) ^ (1ULL << ll);
        } else if (cls == 2) nu = up ^ (1ULL << ii) ^ (1ULL << jj) ^ (1ULL << kk) ^ (1ULL << ll);
        else if (cls == 3) nd = dn ^ (1ULL << ii) ^ (1ULL << jj);
        else nd = dn ^ (1ULL << ii) ^ (1ULL << jj) ^ (1ULL << kk) ^ (1ULL << ll);
        const i64 col = wfn_lookup(w, nu, nd);
        if (col < 0 || col >= w.ndet) continue;
        if (KIND != PYCI_WFN_GENCI && col <= row) continue;
        const double cc = ci * c[col];
        if (KIND == PYCI_WFN_DOCI) {
            double *d0 = base;
            aadd(&d0[ii * n1 + jj], cc);
            aadd(&d0[jj * n1 + ii], cc);
        } else if (KIND == PYCI_WFN_FULLCI) {
            double *aa = base, *bb = base + n2, *aaaa = base + 2 * n2, *bbbb = aaaa + n4, *abab = bbbb + n4;
            if (cls == 0) {
                const double v = cc * phase1(up, ii, jj);
                aadd(&aa[ii * n1 + jj], v);
                aadd(&aa[jj * n1 + ii], v);
                for (u64 x = up; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x);
                    if (q != ii) same_spin_single(aaaa, n, ii, jj, q, v);
                }
                for (u64 x = dn; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x);
                    aadd(&abab[ii * n3 + q * n2 + jj * n1 + q], v);
                    aadd(&abab[jj * n3 + q * n2 + ii * n1 + q], v);
                }
            } else if (cls == 1) {
                const double v = cc * (double)(phase1(up, ii, jj) * phase1(dn, kk, ll));
                aadd(&abab[ii * n3 + kk * n2 + jj * n1 + ll], v);
                aadd(&abab[jj * n3 + ll * n2 + ii * n1 + kk], v);
            } else if (cls == 2) {
                same_spin8(aaaa, n, ii, kk, jj, ll, cc * phase2(up, ii, kk, jj, ll));
            } else if (cls == 3) {
                const double v = cc * phase1(dn, ii, jj);
                aadd(&bb[ii * n1 + jj], v);
                aadd(&bb[jj * n1 + ii], v);
                for (u64 x = up; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x);
                    aadd(&abab[q * n3 + ii * n2 + q * n1 + jj], v);
                    aadd(&abab[q * n3 + jj * n2 + q * n1 + ii], v);
                }
                for (u64 x = dn; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x);
                    if (q != ii) same_spin_single(bbbb, n, ii, jj, q, v);
                }
            } else {
                same_spin8(bbbb, n, ii, kk, jj, ll, cc * phase2(dn, ii, kk, jj, ll));
            }
        } else {
            double *r1 = base, *r2 = base + n2;
            if (cls == 0) {
                // ket J = this row, bra I = col: <I| a+_jj a_ii |J>
                const double v = cc * phase1(up, ii, jj);
                aadd(&r1[jj * n1 + ii], v);
                for (u64 x = up; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x);
                    if (q == ii) continue;
                    aadd(&r2[jj * n3 + q * n2 + ii * n1 + q], v);
                    aadd(&r2[q * n3 + jj * n2 + q * n1 + ii], v);
                    aadd(&r2[jj * n3 + q * n2 + q * n1 + ii], -v);
                    aadd(&r2[q * n3 + jj * n2 + ii * n1 + q], -v);
                }
            } else {
                const double v = cc * phase2(up, ii, kk, jj, ll);
                aadd(&r2[jj * n3 + ll * n2 + ii * n1 + kk], v);
                aadd(&r2[jj * n3 + ll * n2 + kk * n1 + ii], -v);
                aadd(&r2[ll * n3 + jj * n2 + ii * n1 + kk], -v);
                aadd(&r2[ll * n3 + jj * n2 + kk * n1 + ii], v);
            }
        }
    }
}

// Transition RDMs (rdm.cpp:634-899): every determinant I of set 1 (w1, c1) and
// its excitations J present in set 2 (w2, c2) add c1_I c2_J times the phase to
// the reference's index images, one term per ordered (I, J) -- no symmetric
// images, as <1|...|2> is not symmetric. Diagonal: I itself where it is in set 2.
// Element conventions: [p,q] = <1| a+_p a_q |2>, [p,q,r,s] = <1| a+_p a+_q a_s a_r |2>;
// GenCI by the operator algebra (the reference routine has index errors).
template <int KIND>
__global__ void __launch_bounds__(256) k_trdm(WfnView w1, WfnView w2, const double *c1, const double *c2, int R,
                                             i64 stride, double *acc) {
    const int lane = threadIdx.x & 63;
    const i64 row = (i64)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= w1.ndet) return;
    const int n = w1.nb;
    const i64 n1 = n, n2 = n1 * n1, n3 = n2 * n1, n4 = n2 * n2;
    double *base = acc + (i64)(blockIdx.x % R) * stride;
    const u64 m = full_mask(n);
    const u64 up = w1.dets[(i64)w1.nkey * row];
    const u64 dn = (KIND == PYCI_WFN_FULLCI) ? w1.dets[2 * row + 1] : 0ULL;
    const int nou = __popcll(up), nvu = n - nou, nod = __popcll(dn), nvd = n - nod;
    const int packed = nth_bit_r(up, lane) | (nth_bit_r(~up & m, lane) << 8) | (nth_bit_r(dn, lane) << 16) |
                       (nth_bit_r(~dn & m, lane) << 24);
    const double ci = c1[row];
    // the 4 antisymmetric images of a same-spin pair term (p,q | r,s)
    auto four = [&](double *X, int p, int q, int r, int t, double v) {
        aadd(&X[p * n3 + q * n2 + r * n1 + t], v);
        aadd(&X[p * n3 + q * n2 + t * n1 + r], -v);
        aadd(&X[q * n3 + p * n2 + r * n1 + t], -v);
        aadd(&X[q * n3 + p * n2 + t * n1 + r], v);
    };
    // ---- diagonal terms ----
    const i64 jd = wfn_lookup(w2, up, dn);
    if (jd >= 0 && jd < w2.ndet) {
        const double val1 = ci * c2[jd];
        if (KIND == PYCI_WFN_DOCI) {
            double *d0 = base, *d2 = base + n2;
            for (int t = lane; t < nou * nou; t += 64) {
                const int a = t / nou, b = t - a * nou;
                const int p = nth_bit_r(up, a), q = nth_bit_r(up, b);
                if (a == b)
                    aadd(&d0[p * (n + 1)], val1);
                else
                    aadd(&d2[p * n1 + q], val1);
            }
        } else {
            double *r1a = base, *r2a = base + (KIND == PYCI_WFN_FULLCI ? 2 * n2 : n2);
            for (int t = lane; t < nou * nou; t += 64) {
                const int a = t / nou, b = t - a * nou;
                const int p = nth_bit_r(up, a), q = nth_bit_r(up, b);
                if (a == b)
                    aadd(&r1a[p * (n + 1)], val1);
                else if (a < b)
                    four(r2a, p, q, p, q, val1);
            }
            if (KIND == PYCI_WFN_FULLCI) {
                double *bb = base + n2, *bbbb = base + 2 * n2 + n4, *abab = bbbb + n4;
                for (int t = lane; t < nod * nod; t += 64) {
                    const int a = t / nod, b = t - a * nod;
                    const int p = nth_bit_r(dn, a), q = nth_bit_r(dn, b);
                    if (a == b)
                        aadd(&bb[p * (n + 1)], val1);
                    else if (a < b)
                        four(bbbb, p, q, p, q, val1);
                }
                for (int t = lane; t < nou * nod; t += 64) {
                    const int a = t / nod, b = t - a * nod;
                    const int p = nth_bit_r(up, a), q = nth_bit_r(dn, b);
                    aadd(&abab[p * n3 + q * n2 + p * n1 + q], val1);
                }
            }
        }
    }
    // ---- excitations of I present in set 2 ----
    int c0, cb1, cb2, cb3, c4;
    exc_bounds<KIND>(nou, nvu, nod, nvd, c0, cb1, cb2, cb3, c4);
    for (int e0 = 0; e0 < c4; e0 += 64) {
        const int e = e0 + lane;
        const bool valid = e < c4;
        int cls = 0, i = 0, a = 0, k = 0, l = 0;
        if (valid) exc_decode(e, c0, cb1, cb2, cb3, nvu, nod, nvd, cls, i, a, k, l);
        const int pi = __shfl(packed, i), pa = __shfl(packed, a), pk = __shfl(packed, k), pl = __shfl(packed, l);
        if (!valid) continue;
        const bool alpha = cls <= 2;
        const int ii = alpha ? (pi & 255) : ((pi >> 16) & 255);
        const int jj = alpha ? ((pa >> 8) & 255) : ((pa >> 24) & 255);
        int kk, ll;
        if (cls == 1 || !alpha) {
            kk = (pk >> 16) & 255;
            ll = (pl >> 24) & 255;
        } else {
            kk = pk & 255;
            ll = (pl >> 8) & 255;
        }
        u64 nu = up, nd = dn;
        if (KIND == PYCI_WFN_DOCI) nu = up ^ (1ULL << ii) ^ (1ULL << jj);
        else if (cls == 0) nu = up ^ (1ULL << ii) ^ (1ULL << jj);
        else if (cls == 1) {
            nu = up ^ (1ULL << ii) ^ (1ULL << jj);
            nd = dn ^ (1ULL << kk) ^ (1ULL << ll);
        } else if (cls == 2) nu = up ^ (1ULL << ii) ^ (1ULL << jj) ^ (1ULL << kk) ^ (1ULL << ll);
        else if (cls == 3) nd = dn ^ (1ULL << ii) ^ (1ULL << jj);
        else nd = dn ^ (1ULL << ii) ^ (1ULL << jj) ^ (1ULL << kk) ^ (1ULL << ll);
        const i64 col = wfn_lookup(w2, nu, nd);
        if (col < 0 || col >= w2.ndet) continue;
        const double cc = ci * c2[col];
        if (KIND == PYCI_WFN_DOCI) {
            aadd(&base[ii * n1 + jj], cc);
        } else if (KIND == PYCI_WFN_GENCI || cls <= 2) {
            // alpha string (FullCI) or the only string (GenCI)
            double *r1 = base, *r2 = base + (KIND == PYCI_WFN_FULLCI ? 2 * n2 : n2);
            double *abab = base + 2 * n2 + 2 * n4;
            if (cls == 0) {
                const double v = cc * phase1(up, ii, jj);
                aadd(&r1[ii * n1 + jj], v);
                for (u64 x = up; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x);
                    if (q == ii) continue;
                    aadd(&r2[ii * n3 + q * n2 + jj * n1 + q], v);
                    aadd(&r2[ii * n3 + q * n2 + q * n1 + jj], -v);
                    aadd(&r2[q * n3 + ii * n2 + q * n1 + jj], v);
                    aadd(&r2[q * n3 + ii * n2 + jj * n1 + q], -v);
                }
                if (KIND == PYCI_WFN_FULLCI)
                    for (u64 x = dn; x; x &= x - 1) {
                        const int q = __builtin_ctzll(x);
                        aadd(&abab[ii * n3 + q * n2 + jj * n1 + q], v);
                    }
            } else if (cls == 1) {
                aadd(&abab[ii * n3 + kk * n2 + jj * n1 + ll], cc * (double)(phase1(up, ii, jj) * phase1(dn, kk, ll)));
            } else {
                four(r2, ii, kk, jj, ll, cc * phase2(up, ii, kk, jj, ll));
            }
        } else {
            double *bb = base + n2, *bbbb = base + 2 * n2 + n4, *abab = bbbb + n4;
            if (cls == 3) {
                const double v = cc * phase1(dn, ii, jj);
                aadd(&bb[ii * n1 + jj], v);
                for (u64 x = up; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x);
                    aadd(&abab[q * n3 + ii * n2 + q * n1 + jj], v);
                }
                for (u64 x = dn; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x);
                    if (q == ii) continue;
                    aadd(&bbbb[ii * n3 + q * n2 + jj * n1 + q], v);
                    aadd(&bbbb[ii * n3 + q * n2 + q * n1 + jj], -v);
                    aadd(&bbbb[q * n3 + ii * n2 + q * n1 + jj], v);
                    aadd(&bbbb[q * n3 + ii * n2 + jj * n1 + q], -v);
                }
            } else {
                four(bbbb, ii, kk, jj, ll, cc * phase2(dn, ii, kk, jj, ll));
            }
        }
    }
}

__global__ void k_sum_copies(const double *acc, int R, i64 stride, double *out) {
    for (i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x; t < stride; t += (i64)gridDim.x * blockDim.x) {
        double v = 0.0;
        for (int r = 0; r < R; ++r) v += acc[(i64)r * stride + t];
        out[t] = v;
    }
}

// Sizes of the two output arrays of a kind (rdm1, rdm2 element counts).
static void rdm_sizes(int kind, i64 n, i64 &s1, i64 &s2) {
    const i64 n2 = n * n, n4 = n2 * n2;
    if (kind == PYCI_WFN_DOCI) {
        s1 = n2;
        s2 = n2;
    } else if (kind == PYCI_WFN_FULLCI) {
        s1 = 2 * n2;
        s2 = 3 * n4;
    } else {
        s1 = n2;
        s2 = n4;
    }
}

void trdms_device(pyci_wfn *w1, pyci_wfn *w2, const double *c1_host, const double *c2_host, double *rdm1,
                  double *rdm2) {
    PE_REQUIRE(w1->ctx == w2->ctx, PYCI_EINVAL, "wave functions belong to different contexts");
    PE_REQUIRE(w1->kind == w2->kind && w1->nbasis == w2->nbasis && w1->nup == w2->nup && w1->ndn == w2->ndn,
               PYCI_EINVAL, "transition RDMs need two wave functions of the same kind, nbasis and occupations");
    hipStream_t s = w1->ctx->stream;
    i64 s1, s2;
    rdm_sizes(w1->kind, w1->nbasis, s1, s2);
    const i64 stride = s1 + s2;
    const i64 nd1 = w1->ndet, nd2 = w2->ndet;
    int R = (int)std::max<i64>(1, std::min<i64>(32, ((i64)256 << 20) / (stride * 8)));
    R = (int)std::min<i64>(R, std::max<i64>(1, (nd1 + 3) / 4));
    DevBuf<double> acc((size_t)(R * stride)), out((size_t)stride);
    DevBuf<double> d1((size_t)std::max<i64>(nd1, 1)), d2((size_t)std::max<i64>(nd2, 1));
    PE_HIP(hipMemsetAsync(acc.p, 0, sizeof(double) * R * stride, s));
    if (nd1 > 0 && nd2 > 0) {
        PE_HIP(hipMemcpyAsync(d1.p, c1_host, sizeof(double) * nd1, hipMemcpyHostToDevice, s));
        PE_HIP(hipMemcpyAsync(d2.p, c2_host, sizeof(double) * nd2, hipMemcpyHostToDevice, s));
        const WfnView v1 = view_of(w1), v2 = view_of(w2);
        const unsigned g = grid_for(nd1, 4);
        if (w1->kind == PYCI_WFN_DOCI)
            k_trdm<PYCI_WFN_DOCI><<<g, 256, 0, s>>>(v1, v2, d1.p, d2.p, R, stride, acc.p);
        else if (w1->kind == PYCI_WFN_FULLCI)
            k_trdm<PYCI_WFN_FULLCI><<<g, 256, 0, s>>>(v1, v2, d1.p, d2.p, R, stride, acc.p);
        else
            k_trdm<PYCI_WFN_GENCI><<<g, 256, 0, s>>>(v1, v2, d1.p, d2.p, R, stride, acc.p);
        PE_LAUNCH_CHECK();
    }
    k_sum_copies<<<(unsigned)std::min<i64>(4096, (stride + 255) / 256), 256, 0, s>>>(acc.p, R, stride, out.p);
    PE_LAUNCH_CHECK();
    PE_HIP(hipMemcpyAsync(rdm1, out.p, sizeof(double) * s1, hipMemcpyDeviceToHost, s));
    PE_HIP(hipMemcpyAsync(rdm2, out.p + s1, sizeof(double) * s2, hipMemcpyDeviceToHost, s));
    PE_HIP(hipStreamSynchronize(s));
}

// ---------------------------------------------------------------------------
// Selected FullCI and GenCI sets: the connected pairs of determinants by testing every pair
// (k_pair_rows of csr_build.hip has the same scan), each pair J > I once, into
// the compact accumulators of rdm.hpp, whose images k_rf_expand forms. k_rdm hashes and
// probes every excitation of every row, and adds each image of an element with an
// atomic of its own.
// ---------------------------------------------------------------------------
constexpr int RP_ROWS = 8;
constexpr int RP_COLS = 4096;

template <int KIND>
__global__ void __launch_bounds__(256) k_rdm_pairs(WfnView w, RfShape S, const double *__restrict__ c, i64 seglen,
                                                   int R, double *__restrict__ acc) {
    constexpr int NW = KIND == PYCI_WFN_FULLCI ? 2 : 1;
    __shared__ u64 hits[4][RP_ROWS][64];
    __shared__ int qcol[4][128];
    __shared__ unsigned char qrow[4][128];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const i64 ngroup = (w.ndet + RP_ROWS - 1) / RP_ROWS, group = (i64)blockIdx.x * 4 + wave;
    if (group >= ngroup) return;  // uniform per wavefront; no block barriers below
    const int nrows = (int)((w.ndet - group + ngroup - 1) / ngroup), n = S.n, npd = S.npd;
    const i64 cbeg = (i64)blockIdx.y * seglen, cend = min(w.ndet, cbeg + seglen);
    double *base_acc = acc + (i64)((blockIdx.x + blockIdx.y) % R) * S.stride;
    u64 ra[RP_ROWS], rb[RP_ROWS];
#pragma unroll
    for (int r = 0; r < RP_ROWS; ++r) {
        const i64 row = min(group + r * ngroup, w.ndet - 1);
        ra[r] = w.dets[NW * row];
        rb[r] = NW == 2 ? w.dets[NW * row + NW - 1] : 0ULL;
    }
    auto pair = [](int p, int q) { return p < q ? q * (q - 1) / 2 + p : p * (p - 1) / 2 + q; };
    auto emit = [&](int at) {
        const i64 col = qcol[wave][at], row = group + (i64)qrow[wave][at] * ngroup;
        const u64 up = w.dets[NW * row], dn = NW == 2 ? w.dets[NW * row + NW - 1] : 0ULL;
        const u64 cu = w.dets[NW * col], cd = NW == 2 ? w.dets[NW * col + NW - 1] : 0ULL;
        const u64 hu = up & ~cu, pu = cu & ~up, hd = dn & ~cd, pd = cd & ~dn;
        const int nu = __popcll(hu), nd = __popcll(hd);
        const double cc = c[row] * c[col];
        if (nu == 1 && nd == 1) {
            const int i = __builtin_ctzll(hu), a = __builtin_ctzll(pu), k = __builtin_ctzll(hd), l = __builtin_ctzll(pd);
            const double v = cc * (double)(phase1(up, i, a) * phase1(dn, k, l));
            // abab[i,k,a,l] = abab[a,l,i,k], held with the beta pair in order
            const i64 pr = k < l ? (i64)(i * n + a) * S.npr + l * (l + 1) / 2 + k
                                 : (i64)(a * n + i) * S.npr + k * (k + 1) / 2 + l;
            aadd(&base_acc[S.oab + pr], v);
            return;
        }
        const bool beta = nu == 0;
        const u64 d = beta ? dn : up, h = beta ? hd : hu, p = beta ? pd : pu;
        double *one = base_acc + (beta ? n * n : 0), *two = base_acc + (beta ? S.obb : S.oaa);
        const int i = __builtin_ctzll(h), a = __builtin_ctzll(p);
        const u64 h2 = h & (h - 1), p2 = p & (p - 1);
        if (h2) {
            const int k = __builtin_ctzll(h2), l = __builtin_ctzll(p2);
            aadd(&two[(i64)pair(i, k) * npd + pair(a, l)], cc * phase2(d, i, k, a, l));
            return;
        }
        const double v = cc * phase1(d, i, a);
        aadd(&one[i * n + a], v);
        for (u64 x = d; x; x &= x - 1) {
            const int q = __builtin_ctzll(x);
            if (q == i) continue;
            aadd(&two[(i64)pair(i, q) * npd + pair(a, q)], (i < q) != (a < q) ? -v : v);
        }
        if constexpr (KIND == PYCI_WFN_FULLCI) {
            if (beta) {
                const int s = max(i, a), t = min(i, a);
                for (u64 x = up; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x);
                    aadd(&base_acc[S.oab + (i64)(q * n + q) * S.npr + s * (s + 1) / 2 + t], v);
                }
            } else {
                for (u64 x = dn; x; x &= x - 1) {
                    const int q = __builtin_ctzll(x), qq = q * (q + 1) / 2 + q;
                    aadd(&base_acc[S.oab + (i64)(i * n + a) * S.npr + qq], v);
                    aadd(&base_acc[S.oab + (i64)(a * n + i) * S.npr + qq], v);
                }
            }
        }
    };
    auto settle = [] {
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
    };
    int qn = 0;
    for (i64 base = cbeg; base < cend; base += RP_COLS) {
        if (base + RP_COLS - 1 <= group) continue;  // no column beyond the first row
        const int nch = (int)min((i64)(RP_COLS / 64), (cend - base + 63) / 64);
        u64 mk[RP_ROWS] = {};
        auto fetch = [&](int t, u64 &a, u64 &b) {
            const i64 col = min(base + t * 64 + lane, cend - 1);
            a = w.dets[NW * col];
            b = NW == 2 ? w.dets[NW * col + NW - 1] : 0ULL;
        };
        u64 a, b, an, bn;
        fetch(0, a, b);
        for (int t = 0; t < nch; ++t) {
            fetch(min(t + 1, nch - 1), an, bn);
            const u64 valid = __ballot(base + t * 64 + lane < cend);
#pragma unroll
            for (int r = 0; r < RP_ROWS; ++r) {
                int d = __popcll(a ^ ra[r]);
                if (NW == 2) d += __popcll(b ^ rb[r]);
                const u64 h = __ballot(d <= 4) & valid;
                mk[r] = lane == t ? h : mk[r];
            }
            a = an, b = bn;
        }
#pragma unroll
        for (int r = 0; r < RP_ROWS; ++r) hits[wave][r][lane] = mk[r];
        settle();
        for (int r = 0; r < nrows; ++r) {
            u64 m = hits[wave][r][lane];
            // columns beyond the row only
            const i64 first = group + r * ngroup + 1 - (base + lane * 64);
            if (first > 0) m = first >= 64 ? 0ULL : m & (~0ULL << first);
            for (u64 act = __ballot(m != 0); act; act = __ballot(m != 0)) {
                if (m) {
                    const int slot = qn + __popcll(act & ((1ULL << lane) - 1ULL));
                    qcol[wave][slot] = (int)base + lane * 64 + __builtin_ctzll(m);
                    qrow[wave][slot] = (unsigned char)r;
                    m &= m - 1;
                }
                qn += __popcll(act);
                if (qn >= 64) {
                    settle();
                    qn -= 64;
                    emit(qn + lane);
                    settle();
                }
            }
        }
        settle();
    }
    if (lane < qn) emit(lane);
}

// The diagonal terms c_I^2 of the same accumulators: summed over a block's determinants in
// LDS first, because every determinant adds to the elements of the common orbitals.
template <int KIND>
__global__ void __launch_bounds__(256) k_rdm_diagonal(WfnView w, RfShape S, const double *__restrict__ c, int R,
                                                      double *__restrict__ acc) {
    constexpr int NW = KIND == PYCI_WFN_FULLCI ? 2 : 1;
    extern __shared__ double sums[];  // per string: n orbitals, npd pairs; FullCI: n x n mixed
    const int n = S.n, per = n + S.npd, total = NW * per + (NW == 2 ? n * n : 0);
    for (int t = threadIdx.x; t < total; t += 256) sums[t] = 0.0;
    __syncthreads();
    for (i64 row = (i64)blockIdx.x * 256 + threadIdx.x; row < w.ndet; row += (i64)gridDim.x * 256) {
        const double v = c[row] * c[row];
        for (int s = 0; s < NW; ++s) {
            const u64 d = w.dets[NW * row + s];
            for (u64 x = d; x; x &= x - 1) {
                const int p = __builtin_ctzll(x);
                atomicAdd(&sums[s * per + p], v);
                for (u64 y = x & (x - 1); y; y &= y - 1) {
                    const int q = __builtin_ctzll(y);
                    atomicAdd(&sums[s * per + n + q * (q - 1) / 2 + p], v);
                }
                if (NW == 2 && s == 0)
                    for (u64 y = w.dets[NW * row + 1]; y; y &= y - 1)
                        atomicAdd(&sums[NW * per + p * n + __builtin_ctzll(y)], v);
            }
        }
    }
    __syncthreads();
    double *base = acc + (i64)(blockIdx.x % R) * S.stride;
    for (int t = threadIdx.x; t < total; t += 256) {
        const double v = sums[t];
        if (v == 0.0) continue;
        const int s = t / per, u = t - s * per;
        if (t >= NW * per) {
            const int m = t - NW * per, p = m / n, q = m - p * n;
            aadd(&base[S.oab + (i64)(p * n + p) * S.npr + q * (q + 1) / 2 + q], v);
        } else if (u < n) {
            aadd(&base[s * n * n + u * n + u], v);
        } else {
            aadd(&base[(s ? S.obb : S.oaa) + (i64)(u - n) * S.npd + (u - n)], v);
        }
    }
}

// FullCI up to 60 orbitals: the sums of k_rdm_diagonal take 58 KB of the 64 KB of LDS there.
static bool rdms_pairs(pyci_wfn *wfn, const double *coeffs_host, double *rdm1, double *rdm2) {
    if (wfn->kind == PYCI_WFN_DOCI || (wfn->kind == PYCI_WFN_FULLCI && wfn->nbasis > 60) || !pairs_serve(wfn))
        return false;
    hipStream_t s = wfn->ctx->stream;
    const RfShape S = rf_shape(wfn);
    const int R = rf_copies(S);
    const i64 nd = wfn->ndet, nacc = R * S.stride;
    DevBuf<double> buf((size_t)(nacc + nd));
    double *acc = buf.p, *c = acc + nacc;
    PE_HIP(hipMemsetAsync(acc, 0, sizeof(double) * nacc, s));
    PE_HIP(hipMemcpyAsync(c, coeffs_host, sizeof(double) * nd, hipMemcpyHostToDevice, s));
    const WfnView w = view_of(wfn);
    const i64 groups = (nd + RP_ROWS - 1) / RP_ROWS;
    // split as in build_rows_pairs
    const i64 most = (nd + RP_COLS - 1) / RP_COLS, even = std::min<i64>(16, (nd + 8191) / 8192);
    const i64 want = std::max<i64>(1, std::min(std::max((4096 + groups - 1) / groups, even), most));
    const i64 seglen = ((nd + want - 1) / want + RP_COLS - 1) / RP_COLS * RP_COLS;
    const dim3 grid((unsigned)((groups + 3) / 4), (unsigned)((nd + seglen - 1) / seglen));
    const bool two = wfn->kind == PYCI_WFN_FULLCI;
    const size_t lds = sizeof(double) * (size_t)((two ? 2 : 1) * (S.n + S.npd) + (two ? S.n * S.n : 0));
    const unsigned dg = (unsigned)std::min<i64>(256, (nd + 255) / 256);
    if (two) {
        k_rdm_diagonal<PYCI_WFN_FULLCI><<<dg, 256, lds, s>>>(w, S, c, R, acc);
        PE_LAUNCH_CHECK();
        k_rdm_pairs<PYCI_WFN_FULLCI><<<grid, 256, 0, s>>>(w, S, c, seglen, R, acc);
    } else {
        k_rdm_diagonal<PYCI_WFN_GENCI><<<dg, 256, lds, s>>>(w, S, c, R, acc);
        PE_LAUNCH_CHECK();
        k_rdm_pairs<PYCI_WFN_GENCI><<<grid, 256, 0, s>>>(w, S, c, seglen, R, acc);
    }
    PE_LAUNCH_CHECK();
    rf_result(wfn->ctx, S, R, acc, rdm1, rdm2);
    return true;
}

void rdms_device(pyci_wfn *wfn, const double *coeffs_host, double *rdm1, double *rdm2) {
    if (rdms_full_space(wfn, coeffs_host, rdm1, rdm2) || rdms_pairs(wfn, coeffs_host, rdm1, rdm2)) return;
    hipStream_t s = wfn->ctx->stream;
    const i64 n = wfn->nbasis, n2 = n * n, n4 = n2 * n2;
    i64 s1, s2;
    if (wfn->kind == PYCI_WFN_DOCI) {
        s1 = n2;
        s2 = n2;
    } else if (wfn->kind == PYCI_WFN_FULLCI) {
        s1 = 2 * n2;
        s2 = 3 * n4;
    } else {
        s1 = n2;
        s2 = n4;
    }
    const i64 stride = s1 + s2;
    const i64 nd = wfn->ndet;
    int R = (int)std::max<i64>(1, std::min<i64>(32, ((i64)256 << 20) / (stride * 8)));
    R = (int)std::min<i64>(R, std::max<i64>(1, (nd + 3) / 4));
    DevBuf<double> acc((size_t)(R * stride)), out((size_t)stride), dc((size_t)std::max<i64>(nd, 1));
    PE_HIP(hipMemsetAsync(acc.p, 0, sizeof(double) * R * stride, s));
    if (nd > 0) {
        PE_HIP(hipMemcpyAsync(dc.p, coeffs_host, sizeof(double) * nd, hipMemcpyHostToDevice, s));
        WfnView w = view_of(wfn);
        unsigned g = grid_for(nd, 4);
        if (wfn->kind == PYCI_WFN_DOCI)
            k_rdm<PYCI_WFN_DOCI><<<g, 256, 0, s>>>(w, dc.p, R, stride, acc.p);
        else if (wfn->kind == PYCI_WFN_FULLCI)
            k_rdm<PYCI_WFN_FULLCI><<<g, 256, 0, s>>>(w, dc.p, R, stride, acc.p);
        else
            k_rdm<PYCI_WFN_GENCI><<<g, 256, 0, s>>>(w, dc.p, R, stride, acc.p);
        PE_LAUNCH_CHECK();
    }
    k_sum_copies<<<(unsigned)std::min<i64>(4096, (stride + 255) / 256), 256, 0, s>>>(acc.p, R, stride, out.p);
    PE_LAUNCH_CHECK();
    PE_HIP(hipMemcpyAsync(rdm1, out.p, sizeof(double) * s1, hipMemcpyDeviceToHost, s));
    PE_HIP(hipMemcpyAsync(rdm2, out.p + s1, sizeof(double) * s2, hipMemcpyDeviceToHost, s));
    PE_HIP(hipStreamSynchronize(s));
}

}  // namespace pe
