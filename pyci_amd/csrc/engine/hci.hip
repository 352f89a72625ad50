// Heat-bath CI selection on the GPU.
//
// Reference: add_hci (hci.cpp:252-279) with the per-determinant screening of
// hci.cpp:49-238. A candidate D' of source determinant D_i is added when the
// magnitude of its matrix element exceeds eps/|c_i| and D' is not yet in the
// wave function (singles use the full single-excitation element, 1-1 doubles
// |<ik|ab>|, same-spin doubles |<ik|ab> - <ik|ba>|, DOCI pair hops |v_kl|).
//
// The reference merges per-thread hash maps, so its append order depends on the
// hash table's iteration order. Here new determinants are appended in the order
// of their FIRST occurrence in the serial enumeration (source det ascending,
// then the reference's loop order inside a row), which is deterministic:
//   pass 1 counts passing new candidates (with repeats) to size a hash set,
//   pass 2 inserts each candidate's 64-bit key with the minimum position,
//   then the claimed slots, one per new determinant, are sorted by that
//   position (a radix sort) and written in that order.
// One block handles one source row: its waves walk the lists of excitations above the
// threshold (HbLists), and a candidate's position in the reference's loop order is known
// in closed form.
//
// The same passes also build a candidate pool for the learned selector: the
// insertion threshold is then a looser eps_pool, and each candidate records its
// heat-bath score max_i |H_ji c_i| and whether plain add_hci(eps) takes it.
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "internal.hpp"

#pragma clang fp contract(off)

namespace pe {

constexpr u64 EMPTY_KEY = ~0ULL;

// The hash set of new determinants, two words a slot in one 16-byte piece, so that a
// candidate touches one line of a table that is far larger than L2: the key, and the first
// position (add_hci) or the numerator sum_i H_ai c_i (ENPT2).
struct NewSet {
    u64 *slot;
    u64 cap;  // slots
    unsigned long long *unique;  // number of claimed slots
    int *overflow;
    u64 *score = nullptr;  // pool only: max |H_ji c_i| as double bits (nonnegative, so integer max)
    int *plain = nullptr;  // pool only: 1 when some source passes the plain threshold
};

// Two strings that fit one word are the key themselves; longer ones enter by their ranks.
__host__ __device__ inline bool strings_fit(int nb) { return nb <= 32; }

__device__ inline u64 set_key(const WfnView &w, u64 a, u64 b) {
    if (w.nkey == 1) return a;
    if (strings_fit(w.nb)) return a | (b << 32);
    return (u64)colex_rank(a, w.binom) * (u64)w.nsd + (u64)colex_rank(b, w.binom);
}

// String of colex rank r with k electrons in nb orbitals.
__device__ inline u64 colex_unrank(i64 r, int nb, int k, const i64 *binom) {
    u64 str = 0;
    int p = nb;
    for (int q = k; q >= 1; --q) {
        int t = p - 1;
        while (binom[t * 65 + q] > r) --t;
        str |= 1ULL << t;
        r -= binom[t * 65 + q];
        p = t;
    }
    return str;
}

// The determinant of a key.
__device__ inline void key_det(const WfnView &w, u64 key, u64 &a, u64 &b) {
    a = key, b = 0ULL;
    if (w.nkey == 1) return;
    if (strings_fit(w.nb)) {
        a = key & 0xffffffffULL;
        b = key >> 32;
    } else {
        const i64 ra = (i64)(key / (u64)w.nsd), rb = (i64)(key - (u64)ra * (u64)w.nsd);
        a = colex_unrank(ra, w.nb, w.nup, w.binom);
        b = colex_unrank(rb, w.nb, w.ndn, w.binom);
    }
}

// Finds or claims the slot of key (counted in claims); returns it, or ~0 on overflow. A table
// that has become too small is found out by the first lane that walks it to its end or, long
// before, by one that meets 4,096 other keys (at the intended load of 2/3 chains have some
// hundreds at most); the others see the flag and leave it too, so that a pass over a
// full table ends.
__device__ inline u64 set_insert(const NewSet &S, u64 key, int &claims) {
    u64 h = __umul64hi(mix64(key), S.cap);
    for (u64 step = 0; step < S.cap; ++step) {
        unsigned long long old = atomicCAS((unsigned long long *)&S.slot[2 * h], (unsigned long long)EMPTY_KEY,
                                           (unsigned long long)key);
        if (old == EMPTY_KEY) ++claims;
        if (old == EMPTY_KEY || old == key) return h;
        h = h + 1 < S.cap ? h + 1 : 0;
        if ((step & 63) == 63 &&
            (step >= 4095 || __hip_atomic_load(S.overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
            break;
    }
    atomicOr(S.overflow, 1);
    return ~0ULL;
}

#define GIX(p, q, r, s) ((((p) * n + (q)) * n + (r)) * n + (s))

// Heat-bath lists of a Hamiltonian (n <= 64 orbitals or spin orbitals). For every orbital
// pair p < q (pair index P = q (q - 1) / 2 + p) the pairs r < s ordered by |V| descending,
// V = two_mo[p][q][r][s] - two_mo[p][q][s][r] (the same-spin double of add_hci,
// hci.cpp:219-220, with the same operands, so the same bits), stored with its sign; for
// FullCI also, for every ordered pair (p, q), all (r, s) by |two_mo[p][q][r][s]|, the
// element of a double of both spins; for every (i, a) an upper bound of the
// single-excitation element: |h_ia| + sum over all q of
// |two_mo[i][q][a][q] - two_mo[i][q][q][a]| (FullCI: + |two_mo[i][q][a][q]|). A row then
// visits, per occupied pair, only the list prefix above eps / |c_i|, and computes a single's
// element only where the bound reaches it, instead of evaluating every excitation. FullCI sets
// too small to pay for the lists (lists_pay) go without them (v = nullptr).
struct HbLists {
    const double *v = nullptr;         // [P][npair]
    const double *vo = nullptr;        // [p * n + q][n * n] (FullCI)
    const double *sb = nullptr;        // [i][a]
    const double *top = nullptr, *topo = nullptr;  // |V| of each list's first entry
    const double *most = nullptr;      // the largest of sb, top and topo
    const unsigned short *rs = nullptr, *rso = nullptr;  // r | s << 8 of each entry
};
constexpr int HB_CAP = 2048;      // n (n - 1) / 2 <= 2016 for n <= 64
constexpr int HB_CAP_OPP = 4096;  // n n

template <bool OPP>
__global__ void __launch_bounds__(256) k_hb_lists(HamView H, int count, double *lv, unsigned short *lrs,
                                                  double *top) {
    constexpr int CAP = OPP ? HB_CAP_OPP : HB_CAP;
    __shared__ double key[CAP];
    __shared__ unsigned short idx[CAP];
    const int n = H.n, tid = threadIdx.x;
    const double *two = H.two;
    int p, q;
    if (OPP)
        p = blockIdx.x / n, q = blockIdx.x % n;
    else
        tri_decode((int)blockIdx.x, p, q);
    auto element = [&](int j, int &r, int &s) {
        if (OPP) {
            r = j / n, s = j % n;
            return two[GIX(p, q, r, s)];
        }
        tri_decode(j, r, s);
        return two[GIX(p, q, r, s)] - two[GIX(p, q, s, r)];
    };
    int N = 1;
    while (N < count) N <<= 1;
    for (int j = tid; j < N; j += 256) {
        int r, s;
        const double k = j < count ? fabs(element(j, r, s)) : -1.0;
        key[j] = k >= 0.0 ? k : -1.0;  // a NaN passes no threshold
        idx[j] = (unsigned short)j;
    }
    __syncthreads();
    // bitonic sort, descending by |V|
    for (int size = 2; size <= N; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int t = tid; t < N / 2; t += 256) {
                const int blk = t / stride, o = t - blk * stride;
                int a, b;
                if (stride == (size >> 1)) {
                    a = blk * size + o;
                    b = blk * size + size - 1 - o;
                } else {
                    a = blk * 2 * stride + o;
                    b = a + stride;
                }
                // padding (index >= count) stays behind NaNs of the same key
                if (key[a] < key[b] || (key[a] == key[b] && idx[a] > idx[b])) {
                    const double tk = key[a];
                    key[a] = key[b];
                    key[b] = tk;
                    const unsigned short ti = idx[a];
                    idx[a] = idx[b];
                    idx[b] = ti;
                }
            }
            __syncthreads();
        }
    }
    if (tid == 0) top[blockIdx.x] = key[0];
    const i64 base = (i64)blockIdx.x * count;
    for (int t = tid; t < count; t += 256) {
        int r, s;
        lv[base + t] = element(idx[t], r, s);
        lrs[base + t] = (unsigned short)(r | (s << 8));
    }
}

__global__ void k_hb_single_bound(HamView H, int opp, double *sb) {
    const int n = H.n, e = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (e >= n * n) return;
    const double *one = H.one, *two = H.two;
    const int i = e / n, a = e - i * n;
    double b = fabs(one[i * n + a]);
    for (int q = 0; q < n; ++q) {
        b += fabs(two[GIX(i, q, a, q)] - two[GIX(i, q, q, a)]);
        if (opp) b += fabs(two[GIX(i, q, a, q)]);
    }
    sb[e] = b;
}

// most = max of v[0 .. n) (negative entries, of lists without a number, do not count)
__global__ void __launch_bounds__(256) k_hb_most(const double *v, int n, double *most) {
    __shared__ double red[4];
    double m = 0.0;
    for (int t = threadIdx.x; t < n; t += 256) m = v[t] > m || v[t] != v[t] ? v[t] : m;
    for (int o = 32; o > 0; o >>= 1) {
        const double x = __shfl_xor(m, o);
        m = x > m || x != x ? x : m;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) m = red[w] > m || red[w] != red[w] ? red[w] : m;
        *most = m;
    }
}

// PASS 1: count, 2: insert, 5: ENPT2 numerators (insert, then add the signed
// H_ai c_i of every passing candidate). A block of 4 waves per row shares out the
// row's lists: the reference determinant's row alone holds a large part of all passing
// candidates and one wave would still walk it when the others are done. Counters leave a
// block in one atomic (one per wave and chunk on the same address took over half of the
// ENPT2 pass). A launch holds fewer than 2^32 threads, 16.7 million such blocks: beyond a
// million blocks a block takes several rows.
constexpr int HCI_WAVES = 4;
constexpr i64 HCI_BLOCKS = (i64)1 << 20;

// LISTS: there are lists (DOCI has none).
template <int KIND, int PASS, bool LISTS>
__global__ void __launch_bounds__(HCI_WAVES * 64) k_hci(WfnView w, HamView H, const double *coeffs, double eps, double eps_plain,
                                             i64 rows_stride, NewSet S, unsigned long long *count, HbLists L) {
    __shared__ unsigned long long sums[HCI_WAVES];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = H.n;
    const double *one = H.one, *two = H.two;
    const u64 m = full_mask(n);
    u64 local = 0;   // PASS 1: passing candidates of the wave
    int claims = 0;  // slots this lane has claimed
    for (i64 row = blockIdx.x; row < w.ndet; row += gridDim.x) {
        const u64 up = w.dets[(i64)w.nkey * row];
        const u64 dn = (KIND == PYCI_WFN_FULLCI) ? w.dets[2 * row + 1] : 0ULL;
        const int nou = __popcll(up), nvu = n - nou, nod = __popcll(dn), nvd = n - nod;
        const double cabs = fabs(coeffs[row]);
        const double eps_i = eps / cabs, eps_plain_i = eps_plain / cabs;
        // a row of the tail, whose threshold no element reaches
        if (LISTS && *L.most * (1.0 + 1e-12) <= eps_i) continue;  // uniform per block
        // lane q holds the q-th occupied / virtual orbital of each string
        auto nth = [](u64 x, int t) {
            for (int s = 0; s < t && x; ++s) x &= x - 1;
            return x ? __builtin_ctzll(x) : 0;
        };
        const int packed = nth(up, lane) | (nth(~up & m, lane) << 8) | (nth(dn, lane) << 16) | (nth(~dn & m, lane) << 24);

        // Evaluates one candidate; returns true when it passes and is new.
        auto consider = [&](bool valid, u64 nu, u64 nd, double val, u64 pos, int sg) {
            bool pass = false;
            u64 key = 0;
            if (valid && fabs(val) > eps_i) {
                if (wfn_lookup(w, nu, nd) < 0) {
                    pass = true;
                    key = set_key(w, nu, nd);
                }
            }
            if (PASS == 1) {
                local += __popcll(__ballot(pass));
            } else if (PASS == 5) {
                // the reference multiplies the element by (phase * c_i) (enpt2.cpp:122-205)
                if (pass) {
                    const u64 slot = set_insert(S, key, claims);
                    if (slot != ~0ULL)
                        atomicAdd(reinterpret_cast<double *>(&S.slot[2 * slot + 1]), val * ((double)sg * coeffs[row]));
                }
            } else if (PASS == 2) {
                if (pass) {
                    const u64 slot = set_insert(S, key, claims);
                    if (slot != ~0ULL)
                        atomicMin((unsigned long long *)&S.slot[2 * slot + 1], (unsigned long long)pos);
                    if (S.score != nullptr && slot != ~0ULL) {
                        atomicMax((unsigned long long *)&S.score[slot],
                                  (unsigned long long)__double_as_longlong(fabs(val) * cabs));
                        if (fabs(val) > eps_plain_i) atomicOr(&S.plain[slot], 1);
                    }
                }
            }
        };

        const u64 rbase = (u64)row * (u64)rows_stride;
        if constexpr (KIND == PYCI_WFN_DOCI) {
            const int total = nou * nvu;
            for (int e0 = wave * 64; e0 < total; e0 += HCI_WAVES * 64) {
                const int e = e0 + lane;
                const bool valid = e < total;
                const int i = valid ? e / nvu : 0, j = valid ? e - (e / nvu) * nvu : 0;
                const int pi = __shfl(packed, i), pj = __shfl(packed, j);
                const int k = pi & 255, l = (pj >> 8) & 255;
                double val = valid ? two[GIX(k, k, l, l)] : 0.0;
                consider(valid, up ^ (1ULL << k) ^ (1ULL << l), 0ULL, val, rbase + (u64)e, 1);
            }
        } else {
            // Position of a candidate in the reference's row order (alpha: for i, for j: single
            // (i, j), FullCI the doubles with a beta single (k, l), then the doubles (k > i,
            // l > j); beta after alpha, without the second kind): the single (i, j) at off(i, j).
            const i64 mixed = KIND == PYCI_WFN_FULLCI ? (i64)nod * nvd : 0;
            auto off = [](int no, int nv, i64 mid, int i, int j) -> i64 {
                const i64 hv = (i64)nv * (nv - 1) / 2;
                return ((i64)i * nv + j) * (1 + mid) + hv * ((i64)i * (no - 1) - (i64)i * (i - 1) / 2) +
                       (i64)(no - 1 - i) * ((i64)j * (nv - 1) - (i64)j * (j - 1) / 2);
            };
            const i64 beta0 = KIND == PYCI_WFN_FULLCI ? off(nou, nvu, mixed, nou, 0) : 0;
            // index of orbital r among the empty orbitals of string d
            auto hole = [](u64 d, int r) { return r - __popcll(d & ((1ULL << r) - 1ULL)); };
            int turn = 0;  // lists seen: the waves take them in turn
            // the pairs (r, s) of p and q whose element is above the threshold, in chunks of 64
            // lanes: the beginning of their list, or all elements where there are no lists
            auto walk = [&](auto same, int p, int q, auto &&take) {
                constexpr bool SAME = decltype(same)::value;
                const int len = SAME ? n * (n - 1) / 2 : n * n;
                const i64 at = (SAME ? (i64)(q * (q - 1) / 2 + p) : (i64)(p * n + q)) * len;
                for (int t0 = 0; t0 < len; t0 += 64) {
                    const int t = t0 + lane;
                    int r = 0, s2 = 0;
                    double V = 0.0;
                    if (LISTS) {
                        if (t < len) V = (SAME ? L.v : L.vo)[at + t];
                    } else if (t < len) {
                        if (SAME) {
                            tri_decode(t, r, s2);
                            V = two[GIX(p, q, r, s2)] - two[GIX(p, q, s2, r)];
                        } else {
                            r = t / n, s2 = t - r * n;
                            V = two[at + t];
                        }
                    }
                    const bool above = t < len && fabs(V) > eps_i;
                    if (__ballot(above) == 0) {
                        if (LISTS) break;  // sorted: nothing further passes
                        continue;
                    }
                    if (LISTS) {
                        const unsigned rs = above ? (SAME ? L.rs : L.rso)[at + t] : 0u;
                        r = (int)(rs & 255u), s2 = (int)(rs >> 8);
                    }
                    take(above, V, r, s2);
                }
            };
            // singles and same-spin doubles of one spin
            auto spin = [&](bool beta) {
                const u64 d = beta ? dn : up;
                const int no = beta ? nod : nou, nv = beta ? nvd : nvu, so = beta ? 16 : 0;
                const i64 mid = beta ? 0 : mixed;
                const u64 at0 = rbase + (u64)(beta ? beta0 : 0);
                // singles, unless the bound stays below the threshold (one that is NaN tells nothing)
                for (int e0 = wave * 64; e0 < no * nv; e0 += HCI_WAVES * 64) {
                    const int e = e0 + lane;
                    const bool in = e < no * nv;
                    const int ec = in ? e : 0, i = ec / nv, j = ec - i * nv;
                    const int ii = (__shfl(packed, i) >> so) & 255, jj = (__shfl(packed, j) >> (so + 8)) & 255;
                    const bool live = in && !(LISTS && L.sb[ii * n + jj] * (1.0 + 1e-12) <= eps_i);
                    double val = 0.0;
                    int sg = 1;
                    if (live) {
                        double v = one[ii * n + jj];
                        for (u64 x = up; x; x &= x - 1) {
                            const int q = __builtin_ctzll(x);
                            if (beta)
                                v += two[GIX(ii, q, jj, q)];
                            else
                                v += two[GIX(ii, q, jj, q)] - two[GIX(ii, q, q, jj)];
                        }
                        if (KIND == PYCI_WFN_FULLCI)
                            for (u64 x = dn; x; x &= x - 1) {
                                const int q = __builtin_ctzll(x);
                                if (beta)
                                    v += two[GIX(ii, q, jj, q)] - two[GIX(ii, q, q, jj)];
                                else
                                    v += two[GIX(ii, q, jj, q)];
                            }
                        val = v;
                        if (PASS == 5) sg = phase1(d, ii, jj);
                    }
                    const u64 x = d ^ (1ULL << ii) ^ (1ULL << jj);
                    consider(live, beta ? up : x, beta ? x : dn, val, at0 + (u64)off(no, nv, mid, i, j), sg);
                }
                // doubles: the occupied pairs whose list begins above the threshold, a lane each
                const int np = no * (no - 1) / 2;
                for (int p0 = 0; p0 < np; p0 += 64) {
                    int i = 0, k = 0;
                    if (p0 + lane < np) tri_decode(p0 + lane, i, k);
                    const int ii0 = (__shfl(packed, i) >> so) & 255, kk0 = (__shfl(packed, k) >> so) & 255;
                    u64 todo = __ballot(p0 + lane < np && !(LISTS && !(L.top[kk0 * (kk0 - 1) / 2 + ii0] > eps_i)));
                    for (; todo; todo &= todo - 1) {
                        if (turn++ % HCI_WAVES != wave) continue;
                        const int from = __builtin_ctzll(todo);
                        const int pi = __shfl(i, from), pk = __shfl(k, from);
                        const int ii = __shfl(ii0, from), kk = __shfl(kk0, from);
                        walk(std::true_type{}, ii, kk, [&](bool above, double V, int r, int s2) {
                            const bool free = above && !((d >> r) & 1ULL) && !((d >> s2) & 1ULL);
                            const int j = hole(d, r), l = hole(d, s2);
                            int sg = 1;
                            if (PASS == 5 && free) sg = phase2(d, ii, kk, r, s2);
                            const i64 o = off(no, nv, mid, pi, j) + 1 + mid + (i64)(pk - pi - 1) * (nv - 1 - j) + (l - j - 1);
                            const u64 x = d ^ (1ULL << ii) ^ (1ULL << kk) ^ (1ULL << r) ^ (1ULL << s2);
                            consider(free, beta ? up : x, beta ? x : dn, V, at0 + (u64)o, sg);
                        });
                    }
                }
            };
            spin(false);
            if constexpr (KIND == PYCI_WFN_FULLCI) {
                // doubles of both spins
                for (int p0 = 0; p0 < nou * nod; p0 += 64) {
                    const int e = p0 + lane < nou * nod ? p0 + lane : 0, i = e / nod, k = e - i * nod;
                    const int ii0 = __shfl(packed, i) & 255, kk0 = (__shfl(packed, k) >> 16) & 255;
                    u64 todo = __ballot(p0 + lane < nou * nod && !(LISTS && !(L.topo[ii0 * n + kk0] > eps_i)));
                    for (; todo; todo &= todo - 1) {
                        if (turn++ % HCI_WAVES != wave) continue;
                        const int from = __builtin_ctzll(todo);
                        const int pi = __shfl(i, from), pk = __shfl(k, from);
                        const int ii = __shfl(ii0, from), kk = __shfl(kk0, from);
                        walk(std::false_type{}, ii, kk, [&](bool above, double V, int r, int s2) {
                            const bool free = above && !((up >> r) & 1ULL) && !((dn >> s2) & 1ULL);
                            int sg = 1;
                            if (PASS == 5 && free) sg = phase1(up, ii, r) * phase1(dn, kk, s2);
                            const i64 o = off(nou, nvu, mixed, pi, hole(up, r)) + 1 + (i64)pk * nvd + hole(dn, s2);
                            consider(free, up ^ (1ULL << ii) ^ (1ULL << r), dn ^ (1ULL << kk) ^ (1ULL << s2), V,
                                     rbase + (u64)o, sg);
                        });
                    }
                }
                spin(true);
            }
        }
    }
    if (PASS != 1) {
        for (int o = 32; o > 0; o >>= 1) claims += __shfl_xor(claims, o);
        local = (u64)claims;
    }
    if (lane == 0) sums[wave] = local;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long all = 0;
        for (int v = 0; v < HCI_WAVES; ++v) all += sums[v];
        if (all) atomicAdd(PASS == 1 ? count : S.unique, all);
    }
}

// slots empty, with `second` in their second word
__global__ void k_set_clear(u64 *slot, u64 second, u64 *score, int *plain, i64 n) {
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x) {
        reinterpret_cast<ulonglong2 *>(slot)[i] = ulonglong2{EMPTY_KEY, second};
        if (score) {
            score[i] = 0ULL;
            plain[i] = 0;
        }
    }
}

// Whether a FullCI set is large enough for sorting the lists, which takes 1.1 ms at 64 orbitals
// and hardly less than 40 us at any size: the elements that a pass over the set would look at
// without them against those of the lists. ENPT2 without / with lists, us: 64 orbitals, 1 + 1
// electrons, one determinant 51 / 1,170, 882 determinants 434 / 1,670; 2 + 2 electrons, 500
// determinants 1,010 / 2,010 (walk : sort 0.5); 5 + 5 electrons, 100 determinants (0.7) 4,970 / 3,560;
// 48 orbitals, 5 + 5 electrons, 50 determinants (0.6) 2,500 / 1,870; 12 orbitals, 6 + 6 electrons, 100
// determinants 266 / 284 (700,000 elements); 24 orbitals, 5 + 5 electrons, 300 determinants 760 / 666,
// 3,000 determinants 1,070 / 710.
static bool lists_pay(const WfnView &w) {
    const double n2 = (double)w.nb * w.nb, np = (n2 - w.nb) / 2, nu = w.nup, nd = w.ndn;
    const double walk = (double)w.ndet * (nu * nd * n2 + (nu * (nu - 1) + nd * (nd - 1)) / 2 * np);
    return walk > 1 << 20 && 2 * walk > n2 * n2 + np * np;
}

// The heat-bath lists of a selection (HbLists), built for one call.
struct HbTables {
    DevBuf<double> v;
    DevBuf<unsigned short> rs;
    HbLists L;
    void build(const HamView &H, bool opp, hipStream_t s) {
        const int n = H.n, npair = n * (n - 1) / 2;
        PE_REQUIRE(npair <= HB_CAP, PYCI_EUNSUPPORTED, "too many orbitals for the heat-bath lists");
        const size_t np2 = (size_t)npair * npair, n2 = (size_t)n * n, n4 = opp ? n2 * n2 : 0;
        const size_t nto = opp ? n2 : 0;
        v.alloc(np2 + n4 + n2 + npair + nto + 1);
        rs.alloc(np2 + n4);
        double *vo = v.p + np2, *sb = vo + n4, *top = sb + n2, *topo = top + npair, *most = topo + nto;
        if (npair > 0) {
            k_hb_lists<false><<<(unsigned)npair, 256, 0, s>>>(H, npair, v.p, rs.p, top);
            PE_LAUNCH_CHECK();
        }
        if (opp) {
            k_hb_lists<true><<<(unsigned)n2, 256, 0, s>>>(H, (int)n2, vo, rs.p + np2, topo);
            PE_LAUNCH_CHECK();
        }
        k_hb_single_bound<<<grid_for((i64)n2, 256), 256, 0, s>>>(H, opp ? 1 : 0, sb);
        PE_LAUNCH_CHECK();
        k_hb_most<<<1, 256, 0, s>>>(sb, (int)(n2 + npair + nto), most);
        PE_LAUNCH_CHECK();
        L = HbLists{v.p, vo, sb, top, topo, most, rs.p, rs.p + np2};
    }
};

template <int PASS>
static void launch_hci(int kind, const WfnView &w, const HamView &H, const double *c, double eps, double eps_plain,
                       i64 stride, const NewSet &S, unsigned long long *count, hipStream_t s, const HbLists &L) {
    const unsigned g = (unsigned)std::min(w.ndet, HCI_BLOCKS), t = HCI_WAVES * 64;
    if (kind == PYCI_WFN_DOCI)
        k_hci<PYCI_WFN_DOCI, PASS, false><<<g, t, 0, s>>>(w, H, c, eps, eps_plain, stride, S, count, L);
    else if (kind == PYCI_WFN_FULLCI && L.v)
        k_hci<PYCI_WFN_FULLCI, PASS, true><<<g, t, 0, s>>>(w, H, c, eps, eps_plain, stride, S, count, L);
    else if (kind == PYCI_WFN_FULLCI)
        k_hci<PYCI_WFN_FULLCI, PASS, false><<<g, t, 0, s>>>(w, H, c, eps, eps_plain, stride, S, count, L);
    else
        k_hci<PYCI_WFN_GENCI, PASS, true><<<g, t, 0, s>>>(w, H, c, eps, eps_plain, stride, S, count, L);
    PE_LAUNCH_CHECK();
}

void wfn_index_append(pyci_wfn *w, i64 first);

// Claimed slots of the set as (first position, slot) pairs, in no particular order: one
// cursor increment per block and 4,096 slots.
constexpr int OWN_ITEMS = 16;

__global__ void __launch_bounds__(256) k_set_owners(NewSet S, i64 cap, unsigned long long *cursor, u64 *pos_out,
                                                    u64 *slot_out) {
    __shared__ unsigned long long base;
    __shared__ int wsum[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (i64 h0 = (i64)blockIdx.x * 256 * OWN_ITEMS; h0 < cap; h0 += (i64)gridDim.x * 256 * OWN_ITEMS) {
        u64 b[OWN_ITEMS];
        int n = 0;
#pragma unroll
        for (int t = 0; t < OWN_ITEMS; ++t) {
            const i64 h = h0 + t * 256 + threadIdx.x;
            b[t] = __ballot(h < cap && S.slot[2 * h] != EMPTY_KEY);
            n += __popcll(b[t]);
        }
        if (lane == 0) wsum[wave] = n;
        __syncthreads();
        if (threadIdx.x == 0) {
            const int all = wsum[0] + wsum[1] + wsum[2] + wsum[3];
            base = all ? atomicAdd(cursor, (unsigned long long)all) : 0ULL;
        }
        __syncthreads();
        unsigned long long o = base;
        for (int v = 0; v < wave; ++v) o += (unsigned long long)wsum[v];
#pragma unroll
        for (int t = 0; t < OWN_ITEMS; ++t) {
            if ((b[t] >> lane) & 1ULL) {
                const i64 h = h0 + t * 256 + threadIdx.x;
                const unsigned long long at = o + (unsigned long long)__popcll(b[t] & ((1ULL << lane) - 1ULL));
                pos_out[at] = S.slot[2 * h + 1];
                slot_out[at] = (u64)h;
            }
            o += (unsigned long long)__popcll(b[t]);
        }
        __syncthreads();
    }
}

// The determinants of the sorted owner slots.
__global__ void k_emit_owners(WfnView w, NewSet S, const u64 *slots, i64 n, u64 *out) {
    const i64 o = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= n) return;
    u64 a, b;
    key_det(w, S.slot[2 * slots[o]], a, b);
    out[w.nkey * o] = a;
    if (w.nkey == 2) out[2 * o + 1] = b;
}

// Slots for up to `upper` new determinants: half as many again, a multiple of 256. (The
// slot of a hash is its high product with the capacity, so any capacity will do; with powers
// of two the table was three times the candidates on average, and it is cleared, probed and
// scanned from HBM.) Grown where the cap of 2^29 candidates makes it too small.
static i64 set_capacity(unsigned long long upper) {
    const i64 want = (i64)std::min<unsigned long long>(upper, 1ULL << 29);
    return std::max<i64>(1024, (want + want / 2 + 255) / 256 * 256);
}

// The table's memory comes from the context, which keeps up to 4 GB between calls
// (allocating and freeing it on each call took longer than filling it).
using SetTable = Lease<DevBuf<u64>>;

// Passes 1-2 of the selection: the set of new candidates (|H_ji| > eps/|c_i|,
// not in the wave function) with their first-occurrence positions; then its
// claimed slots ordered by that position (a radix sort), which is the order of
// first occurrence in the serial enumeration: slots[0 .. nnew).
struct HciRun {
    SetTable table;
    DevBuf<u64> score, slots;
    DevBuf<int> plain, ovf;
    DevBuf<unsigned long long> cnt;
    NewSet S{};
    i64 stride = 0, nnew = 0;
    unsigned long long S_unique_host = 0;  // claimed slots after pass 2
    explicit HciRun(pyci_ctx *ctx) : table(ctx->hci_table) {}
};

static void hci_collect(pyci_ham *ham, pyci_wfn *wfn, const double *dc, double eps, double eps_plain, bool pool,
                        HciRun &R) {
    pyci_ctx *ctx = wfn->ctx;
    hipStream_t s = ctx->stream;
    const i64 nd = wfn->ndet;
    PE_REQUIRE(ham->nbasis == wfn->nbasis, PYCI_EINVAL, "operator and wave function have different nbasis");
    if (wfn->kind == PYCI_WFN_FULLCI) {
        long double tot = (long double)binom_host(wfn->nbasis, wfn->nup) * (long double)binom_host(wfn->nbasis, wfn->ndn);
        PE_REQUIRE(tot < 9.0e18L, PYCI_EUNSUPPORTED, "determinant space too large for the GPU selection keys");
    }
    // positions: row * stride + in-row index; stride >= candidates per row
    const i64 no = wfn->nup, nv = wfn->nbasis - wfn->nup, ndo = wfn->ndn, ndv = wfn->nbasis - wfn->ndn;
    R.stride = no * nv + no * nv * ndo * ndv + (no * (no - 1) / 2) * (nv * (nv - 1) / 2) + ndo * ndv +
               (ndo * (ndo - 1) / 2) * (ndv * (ndv - 1) / 2) + 1;
    PE_REQUIRE((long double)R.stride * (long double)nd < 1.8e19L, PYCI_EUNSUPPORTED, "selection too large");
    const WfnView w = view_of(wfn);
    const HamView H = view_of(ham);
    R.cnt.alloc(2);
    R.ovf.alloc(1);
    PE_HIP(hipMemsetAsync(R.cnt.p, 0, sizeof(unsigned long long) * 2, s));
    R.S = NewSet{nullptr, 0, R.cnt.p + 1, R.ovf.p};
    HbTables hb;
    if (wfn->kind == PYCI_WFN_GENCI || (wfn->kind == PYCI_WFN_FULLCI && lists_pay(w)))
        hb.build(H, wfn->kind == PYCI_WFN_FULLCI, s);
    launch_hci<1>(wfn->kind, w, H, dc, eps, eps_plain, R.stride, R.S, R.cnt.p, s, hb.L);
    unsigned long long upper = 0;
    PE_HIP(hipMemcpyAsync(&upper, R.cnt.p, sizeof(upper), hipMemcpyDeviceToHost, s));
    PE_HIP(hipStreamSynchronize(s));
    R.nnew = 0;
    if (upper == 0) return;
    i64 cap = set_capacity(upper);
    for (;;) {
        R.table.buf.ensure((size_t)(2 * cap));
        u64 *table = R.table.buf.p;
        if (pool) {
            R.score.alloc((size_t)cap);
            R.plain.alloc((size_t)cap);
        }
        k_set_clear<<<4096, 256, 0, s>>>(table, ~0ULL, pool ? R.score.p : nullptr, pool ? R.plain.p : nullptr,
                                         cap);
        PE_LAUNCH_CHECK();
        PE_HIP(hipMemsetAsync(R.cnt.p + 1, 0, sizeof(unsigned long long), s));
        PE_HIP(hipMemsetAsync(R.ovf.p, 0, sizeof(int), s));
        R.S = NewSet{table, (u64)cap, R.cnt.p + 1, R.ovf.p};
        if (pool) {
            R.S.score = R.score.p;
            R.S.plain = R.plain.p;
        }
        launch_hci<2>(wfn->kind, w, H, dc, eps, eps_plain, R.stride, R.S, nullptr, s, hb.L);
        unsigned long long uniq = 0;
        int of = 0;
        PE_HIP(hipMemcpyAsync(&uniq, R.cnt.p + 1, sizeof(uniq), hipMemcpyDeviceToHost, s));
        PE_HIP(hipMemcpyAsync(&of, R.ovf.p, sizeof(int), hipMemcpyDeviceToHost, s));
        PE_HIP(hipStreamSynchronize(s));
        if (!of && 3 * (i64)uniq <= 2 * cap) {
            R.S_unique_host = uniq;
            break;
        }
        PE_REQUIRE(cap < ((i64)1 << 34), PYCI_ENOMEM, "selection hash set too large");
        cap <<= 2;
    }
    // every claimed slot is one new determinant with its first position
    const i64 nnew = (i64)R.S_unique_host;
    R.nnew = nnew;
    if (nnew == 0) return;
    PE_REQUIRE(nnew < ((i64)1 << 31), PYCI_ENOMEM, "too many new determinants in one selection step");
    DevBuf<u64> pos_in((size_t)nnew), slot_in((size_t)nnew), pos_out((size_t)nnew);
    R.slots.alloc((size_t)nnew);
    PE_HIP(hipMemsetAsync(R.cnt.p, 0, sizeof(unsigned long long), s));
    k_set_owners<<<(unsigned)std::min<i64>(4096, grid_for(cap, 256 * OWN_ITEMS)), 256, 0, s>>>(R.S, cap, R.cnt.p,
                                                                                             pos_in.p, slot_in.p);
    PE_LAUNCH_CHECK();
    // positions are below nd * stride
    int end_bit = 1;
    while (end_bit < 64 && (long double)((unsigned long long)1 << end_bit) < (long double)nd * (long double)R.stride)
        ++end_bit;
    size_t tmp_bytes = 0;
    PE_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, pos_in.p, pos_out.p, slot_in.p, R.slots.p,
                                              (int)nnew, 0, end_bit, s));
    DevBuf<unsigned char> tmp(tmp_bytes);
    PE_HIP(hipcub::DeviceRadixSort::SortPairs(tmp.p, tmp_bytes, pos_in.p, pos_out.p, slot_in.p, R.slots.p,
                                              (int)nnew, 0, end_bit, s));
    PE_HIP(hipStreamSynchronize(s));  // the sort's buffers leave scope
}

i64 add_hci_device(pyci_ham *ham, pyci_wfn *wfn, const double *coeffs_host, double eps) {
    pyci_ctx *ctx = wfn->ctx;
    hipStream_t s = ctx->stream;
    const i64 nd = wfn->ndet;
    if (nd == 0) return 0;
    DevBuf<double> dc((size_t)nd);
    PE_HIP(hipMemcpyAsync(dc.p, coeffs_host, sizeof(double) * nd, hipMemcpyHostToDevice, s));
    HciRun R(ctx);
    hci_collect(ham, wfn, dc.p, eps, eps, false, R);
    const i64 nnew = R.nnew;
    if (nnew == 0) return 0;
    // grow the device det array, then write the new determinants in place
    const i64 need = (nd + nnew) * wfn->nkey;
    if ((size_t)need > wfn->dets.n) {
        DevBuf<u64> nb((size_t)(need + need / 2));
        PE_HIP(hipMemcpyAsync(nb.p, wfn->dets.p, sizeof(u64) * nd * wfn->nkey, hipMemcpyDeviceToDevice, s));
        PE_HIP(hipStreamSynchronize(s));
        wfn->dets = std::move(nb);
    }
    k_emit_owners<<<grid_for(nnew, 256), 256, 0, s>>>(view_of(wfn), R.S, R.slots.p, nnew,
                                                      wfn->dets.p + nd * wfn->nkey);
    PE_LAUNCH_CHECK();
    PE_HIP(hipStreamSynchronize(s));
    wfn->ndet = nd + nnew;
    wfn_index_append(wfn, nd);
    PE_HIP(hipStreamSynchronize(s));
    return nnew;
}

// dst[i] = src[i] for i < n, dst[n] = 0 (input of an exclusive scan).
__global__ void k_int_to_i64(const int *src, i64 n, i64 *dst) {
    const i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i <= n) dst[i] = (i < n) ? (i64)src[i] : 0;
}

// Score and plain flag of each pooled candidate, from its slot.
__global__ void k_pool_scores(NewSet S, const u64 *slots, i64 n, double *hb, int *plain) {
    const i64 o = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= n) return;
    const u64 slot = slots[o];
    hb[o] = __longlong_as_double((long long)S.score[slot]);
    plain[o] = S.plain[slot];
}

void hci_pool_device(pyci_ham *ham, pyci_wfn *wfn, const double *dc, double eps, double eps_pool, HciPool &P) {
    hipStream_t s = wfn->ctx->stream;
    P.n = 0;
    P.nplain = 0;
    if (wfn->ndet == 0) return;
    HciRun R(wfn->ctx);
    hci_collect(ham, wfn, dc, eps_pool, eps, true, R);
    if (R.nnew == 0) return;
    P.n = R.nnew;
    P.dets.alloc((size_t)(R.nnew * wfn->nkey));
    P.hb.alloc((size_t)R.nnew);
    P.plain.alloc((size_t)R.nnew);
    const WfnView w = view_of(wfn);
    k_emit_owners<<<grid_for(P.n, 256), 256, 0, s>>>(w, R.S, R.slots.p, P.n, P.dets.p);
    PE_LAUNCH_CHECK();
    k_pool_scores<<<grid_for(P.n, 256), 256, 0, s>>>(R.S, R.slots.p, P.n, P.hb.p, P.plain.p);
    PE_LAUNCH_CHECK();
    // number of candidates plain add_hci(eps) appends
    DevBuf<i64> cnt((size_t)(P.n + 1));
    k_int_to_i64<<<grid_for(P.n + 1, 256), 256, 0, s>>>(P.plain.p, P.n, cnt.p);
    PE_LAUNCH_CHECK();
    P.nplain = exclusive_scan(wfn->ctx, cnt.p, P.n + 1);
    PE_HIP(hipStreamSynchronize(s));
}

// ---------------------------------------------------------------------------
// Epstein-Nesbet PT2 (enpt2.cpp:342-370): the same candidate enumeration and
// screening as add_hci, with every passing external determinant a accumulating
// sum_i H_ai c_i in a device hash set (pass 5), then
// sum_a num_a^2 / (e - H_aa) over the set.
// ---------------------------------------------------------------------------

// H_aa in the reference's order (compute_enpt2_thread_gather, enpt2.cpp:37-70;
// GenCI :237-255): per occupied j, one_mo[j,j], same-spin pairs, then for FullCI
// the opposite-spin pairs; then the beta string's own terms. jk[j n + l] =
// two[j,l,j,l] - two[j,l,l,j] and jj[j n + l] = two[j,l,j,l] are staged in LDS: every
// external determinant reads about half its electron count squared of them.
__device__ inline double pt2_diag(int n, const double *h, const double *jk, const double *jj, u64 up, u64 dn) {
    double d = 0.0;
    for (u64 x = up; x; x &= x - 1) {
        const int j = __builtin_ctzll(x);
        d += h[j];
        for (u64 y = x & (x - 1); y; y &= y - 1) d += jk[j * n + __builtin_ctzll(y)];
        for (u64 y = dn; y; y &= y - 1) d += jj[j * n + __builtin_ctzll(y)];
    }
    for (u64 x = dn; x; x &= x - 1) {
        const int j = __builtin_ctzll(x);
        d += h[j];
        for (u64 y = x & (x - 1); y; y &= y - 1) d += jk[j * n + __builtin_ctzll(y)];
    }
    return d;
}

constexpr int PT2_BLOCKS = 1024;

// partial[b] = block b's sum of num^2 / (e - H_aa) over its slots (grid-stride,
// then a fixed-order tree in LDS, so the total does not depend on timing).
__global__ void __launch_bounds__(256) k_pt2_terms(WfnView w, NewSet S, i64 cap, HamView H, double e,
                                                   double *partial) {
    extern __shared__ double tab[];
    __shared__ double red[256];
    const int n = H.n;
    double *h = tab, *jk = h + n, *jj = jk + n * n;
    for (int t = threadIdx.x; t < n * n; t += 256) {
        const int j = t / n, l = t - j * n;
        const double c = H.two[GIX(j, l, j, l)];
        jk[t] = c - H.two[GIX(j, l, l, j)];
        if (w.nkey == 2) jj[t] = c;
        if (j == l) h[j] = H.one[j * (n + 1)];
    }
    __syncthreads();
    // claimed slots of a sparse table: a wave collects 64 of them before it evaluates any
    __shared__ ulonglong2 queue[4][128];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double acc = 0.0;
    auto term = [&](int at) {
        const ulonglong2 slot = queue[wave][at];
        u64 a, b;
        key_det(w, slot.x, a, b);
        const double x = __longlong_as_double((long long)slot.y);
        acc += x * x / (e - pt2_diag(n, h, jk, jj, a, b));
    };
    auto settle = [] {
        __builtin_amdgcn_wave_barrier();
        asm volatile("" ::: "memory");
    };
    int qn = 0;
    for (i64 s0 = (i64)blockIdx.x * 256 + wave * 64; s0 < cap; s0 += (i64)gridDim.x * 256) {  // cap: a multiple of 256
        const ulonglong2 slot = reinterpret_cast<const ulonglong2 *>(S.slot)[s0 + lane];
        const bool claimed = slot.x != EMPTY_KEY;
        const u64 b = __ballot(claimed);
        if (claimed) queue[wave][qn + __popcll(b & ((1ULL << lane) - 1ULL))] = slot;
        qn += __popcll(b);
        settle();
        if (qn >= 64) {
            qn -= 64;
            term(qn + lane);
            settle();
        }
    }
    if (lane < qn) term(lane);
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int v = 128; v > 0; v >>= 1) {
        if ((int)threadIdx.x < v) red[threadIdx.x] += red[threadIdx.x + v];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// (d) -> (d, d): the FullCI set of a DOCI set, in the same order (FullCIWfn(const
// DOCIWfn &), fullciwfn.cpp:26-35).
__global__ void k_doci_to_fullci(const u64 *src, i64 n, u64 *dst) {
    const i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[2 * i] = dst[2 * i + 1] = src[i];
}

double enpt2_device(pyci_ham *ham, pyci_wfn *wfn_in, const double *coeffs_host, double e, double eps, i64 *nterms) {
    pyci_ctx *ctx = wfn_in->ctx;
    hipStream_t s = ctx->stream;
    PE_REQUIRE(ham->nbasis == wfn_in->nbasis, PYCI_EINVAL, "operator and wave function have different nbasis");
    if (nterms) *nterms = 0;
    const i64 nd = wfn_in->ndet;
    if (nd == 0) return 0.0;
    // a DOCI set enters as the FullCI set of its (d, d) determinants (enpt2.cpp:382-386)
    pyci_wfn tmp;
    pyci_wfn *wfn = wfn_in;
    if (wfn_in->kind == PYCI_WFN_DOCI) {
        tmp.ctx = ctx;
        tmp.kind = PYCI_WFN_FULLCI;
        tmp.nbasis = wfn_in->nbasis;
        tmp.nup = tmp.ndn = wfn_in->nup;
        tmp.nkey = 2;
        tmp.nsd = binom_host(tmp.nbasis, tmp.ndn);
        tmp.ndet = nd;
        tmp.dets.alloc((size_t)(2 * nd));
        k_doci_to_fullci<<<grid_for(nd, 256), 256, 0, s>>>(wfn_in->dets.p, nd, tmp.dets.p);
        PE_LAUNCH_CHECK();
        wfn_build_index(&tmp);
        wfn = &tmp;
    }
    if (wfn->kind == PYCI_WFN_FULLCI) {
        long double tot = (long double)binom_host(wfn->nbasis, wfn->nup) * (long double)binom_host(wfn->nbasis, wfn->ndn);
        PE_REQUIRE(tot < 9.0e18L, PYCI_EUNSUPPORTED, "determinant space too large for the GPU selection keys");
    }
    DevBuf<double> dc((size_t)nd);
    PE_HIP(hipMemcpyAsync(dc.p, coeffs_host, sizeof(double) * nd, hipMemcpyHostToDevice, s));
    const WfnView w = view_of(wfn);
    const HamView H = view_of(ham);
    DevBuf<unsigned long long> cnt(2);
    DevBuf<int> ovf(1);
    PE_HIP(hipMemsetAsync(cnt.p, 0, sizeof(unsigned long long) * 2, s));
    NewSet S{nullptr, 0, cnt.p + 1, ovf.p};
    // pass 1: passing external candidates (with repeats) bound the set size
    HbTables hb;
    if (wfn->kind == PYCI_WFN_GENCI || lists_pay(w)) hb.build(H, wfn->kind == PYCI_WFN_FULLCI, s);
    launch_hci<1>(wfn->kind, w, H, dc.p, eps, eps, 0, S, cnt.p, s, hb.L);
    unsigned long long upper = 0;
    PE_HIP(hipMemcpyAsync(&upper, cnt.p, sizeof(upper), hipMemcpyDeviceToHost, s));
    PE_HIP(hipStreamSynchronize(s));
    if (upper == 0) return 0.0;
    i64 cap = set_capacity(upper);
    SetTable kept(ctx->hci_table);
    unsigned long long uniq = 0;
    for (;;) {
        kept.buf.ensure((size_t)(2 * cap));
        u64 *table = kept.buf.p;
        k_set_clear<<<4096, 256, 0, s>>>(table, 0ULL, nullptr, nullptr, cap);
        PE_LAUNCH_CHECK();
        PE_HIP(hipMemsetAsync(cnt.p + 1, 0, sizeof(unsigned long long), s));
        PE_HIP(hipMemsetAsync(ovf.p, 0, sizeof(int), s));
        S = NewSet{table, (u64)cap, cnt.p + 1, ovf.p};
        launch_hci<5>(wfn->kind, w, H, dc.p, eps, eps, 0, S, nullptr, s, hb.L);
        int of = 0;
        PE_HIP(hipMemcpyAsync(&uniq, cnt.p + 1, sizeof(uniq), hipMemcpyDeviceToHost, s));
        PE_HIP(hipMemcpyAsync(&of, ovf.p, sizeof(int), hipMemcpyDeviceToHost, s));
        PE_HIP(hipStreamSynchronize(s));
        if (!of && 3 * (i64)uniq <= 2 * cap) break;
        PE_REQUIRE(cap < ((i64)1 << 34), PYCI_ENOMEM, "ENPT2 hash set too large");
        cap <<= 2;
    }
    DevBuf<double> part(PT2_BLOCKS);
    const size_t lds = sizeof(double) * (size_t)(H.n + H.n * H.n * (w.nkey == 2 ? 2 : 1));
    // tables of two spins from 59 orbitals on, with the kernel's own 10 KB, are more than the
    // 64 KB that need no attribute: set for the largest, for callers on other threads
    PE_HIP(hipFuncSetAttribute((const void *)k_pt2_terms, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)(sizeof(double) * (64 + 2 * 64 * 64))));
    k_pt2_terms<<<PT2_BLOCKS, 256, lds, s>>>(w, S, cap, H, e, part.p);
    PE_LAUNCH_CHECK();
    std::vector<double> hp(PT2_BLOCKS);
    PE_HIP(hipMemcpyAsync(hp.data(), part.p, sizeof(double) * PT2_BLOCKS, hipMemcpyDeviceToHost, s));
    PE_HIP(hipStreamSynchronize(s));
    double corr = 0.0;
    for (double v : hp) corr += v;
    if (nterms) *nterms = (i64)uniq;
    return corr;
}

}  // namespace pe
