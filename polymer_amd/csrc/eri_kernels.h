// eri_kernels.h -- the shell-quartet kernel template of libpolyeri.
//
// One thread per contracted shell quartet (ab|cd) of one class: primitive
// loop, Boys + VRR + HRR (eri_engine.h), then the quartet's contribution
// to the Coulomb and exchange matrices with FP64 atomics (8-fold
// permutational symmetry: each unique quartet is computed once).  Each
// class is instantiated in its own translation unit (kgen_*.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>
#include <vector>

#include "eri_engine.h"

// MODE_JK32: J/K of the quartets below the mixed-precision cut, recursion in FP32.
// MODE_PBC: periodic lattice sums (pairs with cell offsets, no permutational
// symmetry, work item = (bra, ket, Q3) with Q3 innermost).
enum { MODE_JK = 0, MODE_SCHWARZ = 1, MODE_TENSOR = 2, MODE_JK32 = 3, MODE_PBC = 4 };

struct PairMeta {
    int prim_off, nprim, fa, fb;
};

// A segment of one bra row: items t0 .. t0 + n - 1 of the list, all with
// the bra pair of row `row`.  2^ls lanes of a wavefront share each item and
// divide its ket primitive pairs (k_eri_seg, k_eri_gc, k_eri_gck; in the Rys
// classes k_eri_rys, 2^ls groups of a member's lanes).
struct SegDesc {
    long long t0;
    int row;
    int n : 26, ls : 6;
};

struct EriArgs {
    const PrimPair* prims;
    const PairMeta* meta;
    const double* ab;          // 4 per pair: ABx ABy ABz 0
    const int* bra_ids;
    const int* ket_ids;
    const long long* row_off;  // nrows + 1
    int nrows;
    long long nwork;
    const int* rb_off;         // nrows x (nbucket+1): ket-bucket offsets inside each row
    const int* bucket_start;   // nbucket: first ket of each bucket in ket_ids
    const int* rb_first;       // nrows x nbucket: first ket of the row's range inside each
                               // bucket (null: every range starts at the bucket start)
    int nbucket;
    const double* boys;        // BOYS_NT x BOYS_NM (wavefront kernel)
    const double* boysA;       // aligned per-L tables (thread kernels)
    const double* D;
    double* J;
    double* K;
    int nbf;
    double* out;               // tensor (MODE_TENSOR, MODE_PBC) or Schwarz (MODE_SCHWARZ)
    int jk_copies;             // 1: one J/K (device-scope atomics); 8: one per XCD
    int tpack;                 // MODE_TENSOR: the pair-packed layout of TensorCb
    const int2* items;         // explicit (bra pair, ket position) items of a density-screened list, or null
    const unsigned* count;     // number of items (device), with items
    const double* ksoa;        // ket primitive pairs, bucket-interleaved fields (9 x kfs doubles)
    long long kfs;             // field stride of ksoa
    const int* bucket_soa;     // nbucket: offset of each ket bucket in ksoa
    // periodic (MODE_PBC): nwork = items x n3, Q3 = t % n3 - cel2
    int n3, cel1, cel2, both;  // both: digest every integral also with bra and ket roles exchanged
    double period;
    const int2* pcell;         // per pair {cell offset Q of the second shell, swap}
    const double* Dc;          // (2 cel1 + 1) x nbf^2 density cells, P(Q)[k][l] = P(k_0, l_Q)
    double *Jc, *Kc;           // jk_copies x (2 cel1 + 1) x nbf^2
    const SegDesc* segs;       // segment kernel: bra-row segments of the list
    int nseg;
    // segment kernel, density screening in the kernel (dtol > 0): skip items
    // with Q_ab Q_cd max|D| (six shell blocks) < dtol, count the rest in kept
    double dtol;
    const double* Qs;
    const int2* psh;           // shells of each pair
    const double* dsh;         // nsh x nsh shell-block maxima of |D|
    int nsh;
    unsigned* kept;
    // with dtol > 0: per segment the largest ket bound (segq, indexed like
    // segs) and the largest |D| block (*dmax); a segment with bra bound x
    // segq x dmax < dtol holds no surviving item and is skipped
    const double* segq;
    const double* dmax;
    // generally contracted lists (k_eri_gc): pair data, bra primitive pairs,
    // ket fields 8 .. 11 of ksoa = the member weights
    const GcMeta* gmeta;
    const GcPrim* gprims;
    double qtol;               // Schwarz threshold of the member quartets
    int qloop;                 // MODE_PBC J/K, thread kernel: Q3 values per thread (0: one, t = item x n3 + Q3)
};

// Number of work items of a launch: the device count of a screened list, or
// the static list size.
__device__ __forceinline__ long long work_count(const EriArgs& g) {
    return g.items ? (long long)*g.count : g.nwork;
}

// J/K accumulation.  With one copy per XCD (jk_copies == 8) a block adds into
// the copy of the XCD it runs on (hardware XCC_ID register, masked to 0..7)
// with workgroup-scope atomics, which complete in that XCD's L2; the copies
// are summed afterwards.  With one copy the atomics are device scope.
__device__ __forceinline__ int xcd_slot(int copies) {
    if (copies <= 1) return 0;
    const int xcc = __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20);   // HW_REG_XCC_ID[3:0]
    return xcc & (copies - 1);
}

__device__ __forceinline__ void jk_add(double* p, double v, int copies) {
    if (copies > 1)
        __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
        atomicAdd(p, v);
}

// Fixed-point accumulation (periodic J/K): the element holds a two's
// complement integer in units of 2^-JK_FX_BITS, each contribution is rounded
// to that grid and added with an integer atomic.  Integer addition is
// associative, so the sum (and the sum of the per-XCD copies) does not depend
// on the order in which the atomics arrive: two builds of the same density
// give bit-identical matrices.  Resolution 2^-50 = 8.9e-16 per contribution;
// the final elements must lie within +-2^13 (intermediate sums may wrap).
#define JK_FX_BITS 50
__device__ __forceinline__ void jk_add_fx(double* p, double v, int copies) {
    const unsigned long long x = (unsigned long long)__double2ll_rn(v * 0x1p50);
    if (copies > 1)
        __hip_atomic_fetch_add(reinterpret_cast<unsigned long long*>(p), x, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    else
        __hip_atomic_fetch_add(reinterpret_cast<unsigned long long*>(p), x, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
}

// Digestion with the quartet's six density / Fock blocks held in registers
// (light classes).  With s the permutational degeneracy weight:
// Jacc[ab] += s v D[cd], Jacc[cd] += s v D[ab], Kacc[ac] += s v D[bd],
// Kacc[ad] += s v D[bc], Kacc[bc] += s v D[ad], Kacc[bd] += s v D[ac];
// afterwards J = 2(Jacc + Jacc^T) and K = Kacc + Kacc^T.
template <int NA, int NB, int NC, int ND, typename real = double>
struct RegDigest {
    real Dab[NA * NB], Dcd[NC * ND], Dac[NA * NC], Dad[NA * ND], Dbc[NB * NC], Dbd[NB * ND];
    real Jab[NA * NB], Jcd[NC * ND], Kac[NA * NC], Kad[NA * ND], Kbc[NB * NC], Kbd[NB * ND];
    __device__ __forceinline__ void load(const double* __restrict__ D, int n, int fa, int fb, int fc, int fd) {
#pragma unroll
        for (int a = 0; a < NA; ++a) {
#pragma unroll
            for (int b = 0; b < NB; ++b) { Dab[a * NB + b] = (real)D[(size_t)(fa + a) * n + fb + b]; Jab[a * NB + b] = 0; }
#pragma unroll
            for (int c = 0; c < NC; ++c) { Dac[a * NC + c] = (real)D[(size_t)(fa + a) * n + fc + c]; Kac[a * NC + c] = 0; }
#pragma unroll
            for (int d = 0; d < ND; ++d) { Dad[a * ND + d] = (real)D[(size_t)(fa + a) * n + fd + d]; Kad[a * ND + d] = 0; }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int c = 0; c < NC; ++c) { Dbc[b * NC + c] = (real)D[(size_t)(fb + b) * n + fc + c]; Kbc[b * NC + c] = 0; }
#pragma unroll
            for (int d = 0; d < ND; ++d) { Dbd[b * ND + d] = (real)D[(size_t)(fb + b) * n + fd + d]; Kbd[b * ND + d] = 0; }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int d = 0; d < ND; ++d) { Dcd[c * ND + d] = (real)D[(size_t)(fc + c) * n + fd + d]; Jcd[c * ND + d] = 0; }
    }
    __device__ __forceinline__ void operator()(int a, int b, int c, int d, real x) {
        Jab[a * NB + b] += x * Dcd[c * ND + d];
        Jcd[c * ND + d] += x * Dab[a * NB + b];
        Kac[a * NC + c] += x * Dbd[b * ND + d];
        Kad[a * ND + d] += x * Dbc[b * NC + c];
        Kbc[b * NC + c] += x * Dad[a * ND + d];
        Kbd[b * ND + d] += x * Dac[a * NC + c];
    }
    __device__ __forceinline__ void flush(double* J, double* K, int n, int fa, int fb, int fc, int fd, double s,
                                          int copies) {
#pragma unroll
        for (int a = 0; a < NA; ++a) {
#pragma unroll
            for (int b = 0; b < NB; ++b) jk_add(&J[(size_t)(fa + a) * n + fb + b], s * (double)Jab[a * NB + b], copies);
#pragma unroll
            for (int c = 0; c < NC; ++c) jk_add(&K[(size_t)(fa + a) * n + fc + c], s * (double)Kac[a * NC + c], copies);
#pragma unroll
            for (int d = 0; d < ND; ++d) jk_add(&K[(size_t)(fa + a) * n + fd + d], s * (double)Kad[a * ND + d], copies);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int c = 0; c < NC; ++c) jk_add(&K[(size_t)(fb + b) * n + fc + c], s * (double)Kbc[b * NC + c], copies);
#pragma unroll
            for (int d = 0; d < ND; ++d) jk_add(&K[(size_t)(fb + b) * n + fd + d], s * (double)Kbd[b * ND + d], copies);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int d = 0; d < ND; ++d) jk_add(&J[(size_t)(fc + c) * n + fd + d], s * (double)Jcd[c * ND + d], copies);
    }
};

// Digestion for heavy classes: each integral goes straight to the six
// matrix elements it touches (density read through the cache), so no block
// of integrals or accumulators is held per thread.
struct StreamDigest {
    const double* __restrict__ D;
    double* J;
    double* K;
    int n, fa, fb, fc, fd;
    double s;
    int copies;
    __device__ __forceinline__ void operator()(int a, int b, int c, int d, double x) {
        const size_t A = fa + a, B = fb + b, C = fc + c, E = fd + d;
        const double sx = s * x;
        jk_add(&J[A * n + B], sx * D[C * n + E], copies);
        jk_add(&J[C * n + E], sx * D[A * n + B], copies);
        jk_add(&K[A * n + C], sx * D[B * n + E], copies);
        jk_add(&K[A * n + E], sx * D[B * n + C], copies);
        jk_add(&K[B * n + C], sx * D[A * n + E], copies);
        jk_add(&K[B * n + E], sx * D[A * n + C], copies);
    }
};

struct SchwarzCb {
    double m = 0.0;
    __device__ __forceinline__ void operator()(int a, int b, int c, int d, double x) {
        if (a == c && b == d) m = fmax(m, fabs(x));
    }
};

// Writes one integral (ij|kl) to every position of the ERI tensor it fills:
// the full n^4 tensor at ((i n + j) n + k) n + l (8 positions), or, pk, the
// tensor with the first pair packed, A(P, k, l) at (P n + k) n + l with
// P = max(i, j) (max(i, j) + 1) / 2 + min(i, j) (4 positions, half the size).
struct TensorCb {
    double* out;
    size_t n;
    int fa, fb, fc, fd;
    int pk;
    __device__ __forceinline__ void operator()(int a, int b, int c, int d, double x) {
        const size_t n1 = n, n2 = n1 * n, n3 = n2 * n;
        const size_t i = fa + a, j = fb + b, k = fc + c, l = fd + d;
        if (pk) {
            const size_t pij = i >= j ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i;
            const size_t pkl = k >= l ? k * (k + 1) / 2 + l : l * (l + 1) / 2 + k;
            out[pij * n2 + k * n1 + l] = x;
            out[pij * n2 + l * n1 + k] = x;
            out[pkl * n2 + i * n1 + j] = x;
            out[pkl * n2 + j * n1 + i] = x;
            return;
        }
        out[i * n3 + j * n2 + k * n1 + l] = x;
        out[j * n3 + i * n2 + k * n1 + l] = x;
        out[i * n3 + j * n2 + l * n1 + k] = x;
        out[j * n3 + i * n2 + l * n1 + k] = x;
        out[k * n3 + l * n2 + i * n1 + j] = x;
        out[l * n3 + k * n2 + i * n1 + j] = x;
        out[k * n3 + l * n2 + j * n1 + i] = x;
        out[l * n3 + k * n2 + j * n1 + i] = x;
    }
};

// Work item t of a class pair -> (bra pair, ket position, ket bucket).
// Rows are bra pairs in Schwarz order; inside a row the surviving kets are
// grouped in buckets of equal primitive-pair count (each bucket a Schwarz
// prefix, or a range from rb_first), so neighbouring threads run primitive
// loops of the same length.  The ket pair is ket_ids[pos].
// Item t of bra row `row` -> (ket position, ket bucket).
__device__ __forceinline__ void decode_in_row(const EriArgs& g, int row, long long t, int& pos, int& b) {
    const int local = (int)(t - g.row_off[row]);
    const int* rb = g.rb_off + (size_t)row * (g.nbucket + 1);
    b = 0;
    while (b + 1 < g.nbucket && rb[b + 1] <= local) ++b;
    const int first = g.rb_first ? g.rb_first[(size_t)row * g.nbucket + b] : 0;
    pos = g.bucket_start[b] + first + (local - rb[b]);
}

__device__ __forceinline__ void decode_work(const EriArgs& g, long long t, int& bp, int& pos, int& b) {
    int lo = 0, hi = g.nrows - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (g.row_off[mid] <= t) lo = mid; else hi = mid - 1;
    }
    bp = g.bra_ids[lo];
    decode_in_row(g, lo, t, pos, b);
}

// Bucket of ket position pos.
__device__ __forceinline__ int bucket_of(const EriArgs& g, int pos) {
    int b = 0;
    while (b + 1 < g.nbucket && g.bucket_start[b + 1] <= pos) ++b;
    return b;
}

// Periodic digestion of one integral (i_0 j_Q1 | k_Q3 l_Q3+Q2) (src/pfourindexdirect.f90:691-704):
// J(Q1)[i][j] += v P(Q2)[k][l]; K(Q3+Q2)[i][l] += v P(Q1-Q3)[k][j] when both
// cells are within [-cel1, cel1].
__device__ __forceinline__ void pbc_add(const EriArgs& g, double* J, double* K, int q1, int q2, int q3, int fi,
                                        int fj, int fk, int fl, double v) {
    const size_t n = g.nbf, n2 = n * n;
    const int c1 = g.cel1;
    jk_add_fx(&J[(size_t)(q1 + c1) * n2 + fi * n + fj], v * g.Dc[(size_t)(q2 + c1) * n2 + fk * n + fl], g.jk_copies);
    const int qk = q3 + q2, qd = q1 - q3;
    if (qk >= -c1 && qk <= c1 && qd >= -c1 && qd <= c1)
        jk_add_fx(&K[(size_t)(qk + c1) * n2 + fi * n + fl], v * g.Dc[(size_t)(qd + c1) * n2 + fk * n + fj],
               g.jk_copies);
}

// Lattice tensor store (MODE_PBC with out set, src/pfourindexstore.f90:258-747):
// T[i][Q1][j][Q3][k][Q2][l] = (i_0 j_Q1 | k_Q3 l_Q3+Q2), Q1 and Q2 in
// [-cel1, cel1] (the launch passes the reduced pair range), Q3 in
// [-cel2, cel2].  Each integral has exactly one producer, so plain stores.
__device__ __forceinline__ void pbc_store(const EriArgs& g, int q1, int q2, int q3, int fi, int fj, int fk, int fl,
                                          double v) {
    const size_t n = g.nbf, n1 = 2 * g.cel1 + 1;
    size_t x = (size_t)fi * n1 + (q1 + g.cel1);
    x = (x * n + fj) * g.n3 + (q3 + g.cel2);
    x = (x * n + fk) * n1 + (q2 + g.cel1);
    g.out[x * n + fl] = v;
}

// Integral (a b | c d) of a stored bra pair (first functions fa, fb; cells cb)
// and a stored ket pair (fc, fd; ck) translated by s cells: as the reference
// quartet with this bra and ket, and (both) as the one with the roles
// exchanged, which is the same integral translated by -s cells.
__device__ __forceinline__ void pbc_integral(const EriArgs& g, double* J, double* K, int2 cb, int2 ck, int s, int fa,
                                             int fb, int fc, int fd, int a, int b, int c, int d, double v) {
    const int fi = cb.y ? fb + b : fa + a, fj = cb.y ? fa + a : fb + b;
    const int fk = ck.y ? fd + d : fc + c, fl = ck.y ? fc + c : fd + d;
    if (g.out) {
        pbc_store(g, cb.x, ck.x, s, fi, fj, fk, fl, v);
        if (g.both) pbc_store(g, ck.x, cb.x, -s, fk, fl, fi, fj, v);
        return;
    }
    pbc_add(g, J, K, cb.x, ck.x, s, fi, fj, fk, fl, v);
    if (g.both) pbc_add(g, J, K, ck.x, cb.x, -s, fk, fl, fi, fj, v);
}

// Periodic digestion of one (quartet, Q3) in registers, one atomic per
// matrix element (the same sums as pbc_integral over the quartet's
// integrals).  SB / SK: the stored bra / ket pair is swapped, so the
// reference's i (cell 0) and j (cell Q1) functions are b and a (and l, k
// are c, d).  Blocks: J(Q1)[i][j] += v D(Q2)[k][l]; K(Q3+Q2)[i][l] += v
// D(Q1-Q3)[k][j]; with both roles also J(Q2)[k][l] += v D(Q1)[i][j] and
// K(Q1-Q3)[k][j] += v D(Q2+Q3)[i][l].
template <int NA, int NB, int NC, int ND, bool SB, bool SK>
__device__ __forceinline__ void pbc_digest(const EriArgs& g, const double* v, int fa, int fb, int fc, int fd, int q1,
                                           int q2, int s, double* J, double* K) {
    constexpr int NI = SB ? NB : NA, NJ = SB ? NA : NB, NK = SK ? ND : NC, NL = SK ? NC : ND;
    const int fi = SB ? fb : fa, fj = SB ? fa : fb, fk = SK ? fd : fc, fl = SK ? fc : fd;
    const size_t n = g.nbf, n2 = n * n;
    const int c1 = g.cel1, cp = g.jk_copies;
    auto V = [&](int i, int j, int k, int l) -> double {
        const int a = SB ? j : i, b = SB ? i : j, c = SK ? l : k, d = SK ? k : l;
        return v[((a * NB + b) * NC + c) * ND + d];
    };
    {
        const double* D = g.Dc + (size_t)(q2 + c1) * n2;
        double dkl[NK * NL], acc[NI * NJ];
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int l = 0; l < NL; ++l) dkl[k * NL + l] = D[(size_t)(fk + k) * n + fl + l];
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                double x = 0.0;
#pragma unroll
                for (int k = 0; k < NK; ++k)
#pragma unroll
                    for (int l = 0; l < NL; ++l) x += V(i, j, k, l) * dkl[k * NL + l];
                acc[i * NJ + j] = x;
            }
        double* Jq = J + (size_t)(q1 + c1) * n2;
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) jk_add_fx(&Jq[(size_t)(fi + i) * n + fj + j], acc[i * NJ + j], cp);
    }
    const int qk = s + q2, qd = q1 - s;
    if (qk >= -c1 && qk <= c1 && qd >= -c1 && qd <= c1) {
        const double* D = g.Dc + (size_t)(qd + c1) * n2;
        double dkj[NK * NJ], acc[NI * NL];
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int j = 0; j < NJ; ++j) dkj[k * NJ + j] = D[(size_t)(fk + k) * n + fj + j];
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                double x = 0.0;
#pragma unroll
                for (int j = 0; j < NJ; ++j)
#pragma unroll
                    for (int k = 0; k < NK; ++k) x += V(i, j, k, l) * dkj[k * NJ + j];
                acc[i * NL + l] = x;
            }
        double* Kq = K + (size_t)(qk + c1) * n2;
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int l = 0; l < NL; ++l) jk_add_fx(&Kq[(size_t)(fi + i) * n + fl + l], acc[i * NL + l], cp);
    }
    if (!g.both) return;
    {
        const double* D = g.Dc + (size_t)(q1 + c1) * n2;
        double dij[NI * NJ], acc[NK * NL];
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) dij[i * NJ + j] = D[(size_t)(fi + i) * n + fj + j];
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                double x = 0.0;
#pragma unroll
                for (int i = 0; i < NI; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) x += V(i, j, k, l) * dij[i * NJ + j];
                acc[k * NL + l] = x;
            }
        double* Jq = J + (size_t)(q2 + c1) * n2;
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int l = 0; l < NL; ++l) jk_add_fx(&Jq[(size_t)(fk + k) * n + fl + l], acc[k * NL + l], cp);
    }
    const int qk2 = q1 - s, qd2 = q2 + s;
    if (qk2 >= -c1 && qk2 <= c1 && qd2 >= -c1 && qd2 <= c1) {
        const double* D = g.Dc + (size_t)(qd2 + c1) * n2;
        double dil[NI * NL], acc[NK * NJ];
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int l = 0; l < NL; ++l) dil[i * NL + l] = D[(size_t)(fi + i) * n + fl + l];
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                double x = 0.0;
#pragma unroll
                for (int i = 0; i < NI; ++i)
#pragma unroll
                    for (int l = 0; l < NL; ++l) x += V(i, j, k, l) * dil[i * NL + l];
                acc[k * NJ + j] = x;
            }
        double* Kq = K + (size_t)(qk2 + c1) * n2;
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int j = 0; j < NJ; ++j) jk_add_fx(&Kq[(size_t)(fk + k) * n + fj + j], acc[k * NJ + j], cp);
    }
}

// Periodic J/K of one (bra, ket) item over Q3 in [s0, s1] in one thread:
// J(Q1) (and, with both roles, J(Q2)) is the same matrix block for every
// Q3, so it is summed in registers and added once; the exchange blocks go
// to a different cell per Q3 and are added per Q3.  Same sums as
// pbc_digest.
template <int LA, int LB, int LC, int LD, bool SB, bool SK>
__device__ __forceinline__ void pbc_loop(const EriArgs& g, int bp, int kp, const PairMeta& mb, const PairMeta& mk,
                                         int q1, int q2, int s0, int s1) {
    constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
    constexpr int NI = SB ? NB : NA, NJ = SB ? NA : NB, NK = SK ? ND : NC, NL = SK ? NC : ND;
    const int fi = SB ? mb.fb : mb.fa, fj = SB ? mb.fa : mb.fb, fk = SK ? mk.fb : mk.fa, fl = SK ? mk.fa : mk.fb;
    const size_t n = g.nbf, n2 = n * n;
    const int c1 = g.cel1, cp = g.jk_copies;
    const size_t off = (size_t)xcd_slot(cp) * (2 * c1 + 1) * n2;
    double* J = g.Jc + off;
    double* K = g.Kc + off;
    double dkl[NK * NL], jij[NI * NJ], dij[NI * NJ], jkl[NK * NL];
    {
        const double* D = g.Dc + (size_t)(q2 + c1) * n2;
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int l = 0; l < NL; ++l) dkl[k * NL + l] = D[(size_t)(fk + k) * n + fl + l];
        const double* E = g.Dc + (size_t)(q1 + c1) * n2;
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                dij[i * NJ + j] = g.both ? E[(size_t)(fi + i) * n + fj + j] : 0.0;
                jij[i * NJ + j] = 0.0;
            }
#pragma unroll
        for (int i = 0; i < NK * NL; ++i) jkl[i] = 0.0;
    }
    const double ABx = g.ab[4 * bp], ABy = g.ab[4 * bp + 1], ABz = g.ab[4 * bp + 2];
    const double CDx = g.ab[4 * kp], CDy = g.ab[4 * kp + 1], CDz = g.ab[4 * kp + 2];
    for (int s = s0; s <= s1; ++s) {
        double v[NA * NB * NC * ND];
        StoreCb<NB, NC, ND, double> st{v};
        const ShiftKet kv{g.prims + mk.prim_off, s * g.period};
        quartet<double, LA, LB, LC, LD>(g.prims + mb.prim_off, mb.nprim, kv, mk.nprim, ABx, ABy, ABz, CDx, CDy, CDz,
                                        g.boysA, st);
        auto V = [&](int i, int j, int k, int l) -> double {
            const int a = SB ? j : i, b = SB ? i : j, c = SK ? l : k, d = SK ? k : l;
            return v[((a * NB + b) * NC + c) * ND + d];
        };
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                double x = 0.0;
#pragma unroll
                for (int k = 0; k < NK; ++k)
#pragma unroll
                    for (int l = 0; l < NL; ++l) x += V(i, j, k, l) * dkl[k * NL + l];
                jij[i * NJ + j] += x;
            }
        const int qk = s + q2, qd = q1 - s;
        if (qk >= -c1 && qk <= c1 && qd >= -c1 && qd <= c1) {
            const double* D = g.Dc + (size_t)(qd + c1) * n2;
            double dkj[NK * NJ];
#pragma unroll
            for (int k = 0; k < NK; ++k)
#pragma unroll
                for (int j = 0; j < NJ; ++j) dkj[k * NJ + j] = D[(size_t)(fk + k) * n + fj + j];
            double* Kq = K + (size_t)(qk + c1) * n2;
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int l = 0; l < NL; ++l) {
                    double x = 0.0;
#pragma unroll
                    for (int j = 0; j < NJ; ++j)
#pragma unroll
                        for (int k = 0; k < NK; ++k) x += V(i, j, k, l) * dkj[k * NJ + j];
                    jk_add_fx(&Kq[(size_t)(fi + i) * n + fl + l], x, cp);
                }
        }
        if (!g.both) continue;
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int l = 0; l < NL; ++l) {
                double x = 0.0;
#pragma unroll
                for (int i = 0; i < NI; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) x += V(i, j, k, l) * dij[i * NJ + j];
                jkl[k * NL + l] += x;
            }
        const int qk2 = q1 - s, qd2 = q2 + s;
        if (qk2 >= -c1 && qk2 <= c1 && qd2 >= -c1 && qd2 <= c1) {
            const double* D = g.Dc + (size_t)(qd2 + c1) * n2;
            double dil[NI * NL];
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int l = 0; l < NL; ++l) dil[i * NL + l] = D[(size_t)(fi + i) * n + fl + l];
            double* Kq = K + (size_t)(qk2 + c1) * n2;
#pragma unroll
            for (int k = 0; k < NK; ++k)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    double x = 0.0;
#pragma unroll
                    for (int i = 0; i < NI; ++i)
#pragma unroll
                        for (int l = 0; l < NL; ++l) x += V(i, j, k, l) * dil[i * NL + l];
                    jk_add_fx(&Kq[(size_t)(fk + k) * n + fj + j], x, cp);
                }
        }
    }
    double* J1 = J + (size_t)(q1 + c1) * n2;
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) jk_add_fx(&J1[(size_t)(fi + i) * n + fj + j], jij[i * NJ + j], cp);
    if (!g.both) return;
    double* J2 = J + (size_t)(q2 + c1) * n2;
#pragma unroll
    for (int k = 0; k < NK; ++k)
#pragma unroll
        for (int l = 0; l < NL; ++l) jk_add_fx(&J2[(size_t)(fk + k) * n + fl + l], jkl[k * NL + l], cp);
}

// Work index t = item x nchunk + chunk, chunk of g.qloop Q3 values.
template <int LA, int LB, int LC, int LD>
__device__ __forceinline__ void pbc_item_loop(const EriArgs& g, long long t) {
    const int nchunk = (g.n3 + g.qloop - 1) / g.qloop;
    const long long u = t / nchunk;
    const int chunk = (int)(t - u * nchunk);
    const int s0 = -g.cel2 + chunk * g.qloop, s1 = min(s0 + g.qloop - 1, g.cel2);
    int bp, pos, b;
    decode_work(g, u, bp, pos, b);
    const int kp = g.ket_ids[pos];
    const PairMeta mb = g.meta[bp], mk = g.meta[kp];
    const int2 cb = g.pcell[bp], ck = g.pcell[kp];
    switch (cb.y * 2 + ck.y) {
    case 0: pbc_loop<LA, LB, LC, LD, false, false>(g, bp, kp, mb, mk, cb.x, ck.x, s0, s1); break;
    case 1: pbc_loop<LA, LB, LC, LD, false, true>(g, bp, kp, mb, mk, cb.x, ck.x, s0, s1); break;
    case 2: pbc_loop<LA, LB, LC, LD, true, false>(g, bp, kp, mb, mk, cb.x, ck.x, s0, s1); break;
    default: pbc_loop<LA, LB, LC, LD, true, true>(g, bp, kp, mb, mk, cb.x, ck.x, s0, s1); break;
    }
}

template <int LA, int LB, int LC, int LD>
__device__ __forceinline__ void pbc_item(const EriArgs& g, long long t) {
    const long long u = t / g.n3;
    const int s = (int)(t - u * g.n3) - g.cel2;
    int bp, pos, b;
    decode_work(g, u, bp, pos, b);
    const int kp = g.ket_ids[pos];
    const PairMeta mb = g.meta[bp], mk = g.meta[kp];
    constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
    double v[NA * NB * NC * ND];
    StoreCb<NB, NC, ND, double> st{v};
    const ShiftKet kv{g.prims + mk.prim_off, s * g.period};
    quartet<double, LA, LB, LC, LD>(g.prims + mb.prim_off, mb.nprim, kv, mk.nprim, g.ab[4 * bp], g.ab[4 * bp + 1],
                                    g.ab[4 * bp + 2], g.ab[4 * kp], g.ab[4 * kp + 1], g.ab[4 * kp + 2], g.boysA, st);
    const size_t off = (size_t)xcd_slot(g.jk_copies) * (2 * g.cel1 + 1) * g.nbf * g.nbf;
    double* J = g.Jc + off;
    double* K = g.Kc + off;
    const int2 cb = g.pcell[bp], ck = g.pcell[kp];
    if (g.out) {   // lattice tensor: one store per integral
        for (int a = 0; a < NA; ++a)
            for (int bb = 0; bb < NB; ++bb)
                for (int c = 0; c < NC; ++c)
                    for (int d = 0; d < ND; ++d)
                        pbc_integral(g, J, K, cb, ck, s, mb.fa, mb.fb, mk.fa, mk.fb, a, bb, c, d,
                                     v[((a * NB + bb) * NC + c) * ND + d]);
        return;
    }
    switch (cb.y * 2 + ck.y) {
    case 0: pbc_digest<NA, NB, NC, ND, false, false>(g, v, mb.fa, mb.fb, mk.fa, mk.fb, cb.x, ck.x, s, J, K); break;
    case 1: pbc_digest<NA, NB, NC, ND, false, true>(g, v, mb.fa, mb.fb, mk.fa, mk.fb, cb.x, ck.x, s, J, K); break;
    case 2: pbc_digest<NA, NB, NC, ND, true, false>(g, v, mb.fa, mb.fb, mk.fa, mk.fb, cb.x, ck.x, s, J, K); break;
    default: pbc_digest<NA, NB, NC, ND, true, true>(g, v, mb.fa, mb.fb, mk.fa, mk.fb, cb.x, ck.x, s, J, K); break;
    }
}

template <int LA, int LB, int LC, int LD, int MODE>
__device__ __forceinline__ void eri_item(const EriArgs& g, long long t) {
    if (MODE == MODE_PBC) {
        if (g.qloop) pbc_item_loop<LA, LB, LC, LD>(g, t);
        else pbc_item<LA, LB, LC, LD>(g, t);
        return;
    }
    int bp, kp, pos = 0, b = 0;
    if (MODE == MODE_SCHWARZ) {
        bp = kp = g.bra_ids[t];
    } else {
        if (g.items) {
            const int2 it = g.items[t];
            bp = it.x; pos = it.y;
            b = bucket_of(g, pos);
        } else {
            decode_work(g, t, bp, pos, b);
        }
        kp = g.ket_ids[pos];
    }
    const PairMeta mb = g.meta[bp], mk = g.meta[kp];
    constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
    const double ABx = g.ab[4 * bp], ABy = g.ab[4 * bp + 1], ABz = g.ab[4 * bp + 2];
    const double CDx = g.ab[4 * kp], CDy = g.ab[4 * kp + 1], CDz = g.ab[4 * kp + 2];
    const PrimPair* bra = g.prims + mb.prim_off;
    const PrimPair* ket = g.prims + mk.prim_off;
    const int fa = mb.fa, fb = mb.fb, fc = mk.fa, fd = mk.fb;
    const int n = g.nbf;
    if (MODE == MODE_SCHWARZ) {
        SchwarzCb cb;
        quartet_fp64<LA, LB, LC, LD>(bra, mb.nprim, ket, mk.nprim, ABx, ABy, ABz, CDx, CDy, CDz, g.boysA, cb);
        g.out[bp] = sqrt(cb.m);
        return;
    }
    const SoaKet kv{g.ksoa + g.bucket_soa[b] + (pos - g.bucket_start[b]), g.bucket_start[b + 1] - g.bucket_start[b],
                    g.kfs};
    if (MODE == MODE_TENSOR) {
        TensorCb cb{g.out, (size_t)n, fa, fb, fc, fd, g.tpack};
        quartet<double, LA, LB, LC, LD>(bra, mb.nprim, kv, mk.nprim, ABx, ABy, ABz, CDx, CDy, CDz, g.boysA, cb);
    } else {
        const double s = (fa == fb ? 0.5 : 1.0) * (fc == fd ? 0.5 : 1.0) * (bp == kp ? 0.5 : 1.0);
        // light classes only (heavier ones run in kcoop.hip): the (ab|cd)
        // block in registers, then the six J/K blocks
        using real = typename std::conditional<MODE == MODE_JK32, float, double>::type;
        real v[NA * NB * NC * ND];
        StoreCb<NB, NC, ND, real> st{v};
        quartet<real, LA, LB, LC, LD>(bra, mb.nprim, kv, mk.nprim, ABx, ABy, ABz, CDx, CDy, CDz, g.boysA, st);
        RegDigest<NA, NB, NC, ND, real> cb;
        cb.load(g.D, n, fa, fb, fc, fd);
        const size_t off = (size_t)xcd_slot(g.jk_copies) * n * n;
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int d = 0; d < ND; ++d) cb(a, b, c, d, v[((a * NB + b) * NC + c) * ND + d]);
        cb.flush(g.J + off, g.K + off, n, fa, fb, fc, fd, s, g.jk_copies);
    }
}

// One thread per work item; grid-stride, so a density-screened list (item
// count known only on the device) runs with a fixed grid.
template <int LA, int LB, int LC, int LD, int MODE>
__global__ void __launch_bounds__(256) k_eri(EriArgs g) {
    const long long nw = work_count(g);
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < nw;
         t += (long long)gridDim.x * blockDim.x)
        eri_item<LA, LB, LC, LD, MODE>(g, t);
}

// Primitive pairs at an address that is the same for the whole wavefront,
// through the scalar cache.  In a loop with J/K atomics the compiler takes a
// plain load of them for a vector one (the atomics might write there): in
// k_eri_gc that was 26 registers and eleven loads a primitive quartet, each
// returning the same words to 64 lanes ((ps|ss) of (H2O)16 2.56 -> 2.21 ms).
typedef const __attribute__((address_space(4))) double* ScalarDoubles;
__device__ __forceinline__ PrimPair scalar_pair(ScalarDoubles x) {
    PrimPair r;
    r.zeta = x[0]; r.K = x[1]; r.Px = x[2]; r.Py = x[3]; r.Pz = x[4];
    r.PAx = x[5]; r.PAy = x[6]; r.PAz = x[7]; r.h = x[8]; r.a2 = x[9];
    return r;
}
__device__ __forceinline__ PrimPair scalar_load(const PrimPair* p) {
    static_assert(sizeof(PrimPair) == 10 * sizeof(double), "field order of scalar_pair");
    return scalar_pair((ScalarDoubles)p);
}
__device__ __forceinline__ GcPrim scalar_load(const GcPrim* p) {
    static_assert(sizeof(GcPrim) == 14 * sizeof(double), "field order");
    const ScalarDoubles x = (ScalarDoubles)p;
    GcPrim r;
    r.pp = scalar_pair(x);
    for (int i = 0; i < 4; ++i) r.w[i] = x[10 + i];
    return r;
}

// Sums over the lanes that share one item.  The 2^ls lanes of an item are
// those that differ in lane bits 5, 4, .. 6 - ls, so step S of a reduction
// exchanges with the lane whose bit 5 - S differs, whatever ls is.
// halve: two values x (kept by lanes with the bit clear) and y (kept by the
// others); returns the kept one summed over the pair of lanes.  On the two
// widest steps one v_permlane swap per 32-bit half moves both.
// full: x summed over the pair, in both lanes.
template <int S>
__device__ __forceinline__ unsigned lane_xchg(unsigned v) {
    if constexpr (S == 2) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, true);        // row_ror:8 = lane ^ 8
    else if constexpr (S == 3) return __builtin_amdgcn_ds_swizzle(v, (4 << 10) | 0x1f);     // lane ^ 4
    else if constexpr (S == 4) return __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, true);    // quad_perm [2,3,0,1]
    else return __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, true);                          // quad_perm [1,0,3,2]
}
template <int S>
__device__ __forceinline__ double lane_halve(double x, double y, int lane) {
    const unsigned long long a = __builtin_bit_cast(unsigned long long, x);
    const unsigned long long b = __builtin_bit_cast(unsigned long long, y);
    if constexpr (S < 2) {
        const auto swap = [](unsigned p, unsigned q) {
            if constexpr (S == 0) return __builtin_amdgcn_permlane32_swap(p, q, false, false);
            else return __builtin_amdgcn_permlane16_swap(p, q, false, false);
        };
        const auto lo = swap((unsigned)a, (unsigned)b), hi = swap((unsigned)(a >> 32), (unsigned)(b >> 32));
        return __builtin_bit_cast(double, (unsigned long long)hi[0] << 32 | lo[0]) +
               __builtin_bit_cast(double, (unsigned long long)hi[1] << 32 | lo[1]);
    } else {
        const bool up = lane >> (5 - S) & 1;
        const unsigned long long send = up ? a : b;
        const unsigned lo = lane_xchg<S>((unsigned)send), hi = lane_xchg<S>((unsigned)(send >> 32));
        return (up ? y : x) + __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
    }
}
template <int S>
__device__ __forceinline__ double lane_full(double x, int lane) {
    return lane_halve<S>(x, x, lane);
}

// acc holds N values for each of M2 x M1 members (member (i, j) at
// (i M1 + j) N).  Sums over the item's lanes, the first steps halving the
// j range a lane keeps, the next the i range, the last plain sums: afterwards
// the lane holds members i0 .. i0 + ni - 1, j0 .. j0 + nj - 1 at indices
// from (0, 0); of the lanes left with equal members one has first = true.
template <int M2, int M1, int N, int S = 0>
__device__ __forceinline__ void lane_reduce(double* acc, int ls, int lane, int& i0, int& ni, int& j0, int& nj,
                                            bool& first) {
    constexpr int LJ = M1 == 4 ? 2 : M1 == 2 ? 1 : 0, LI = M2 == 4 ? 2 : M2 == 2 ? 1 : 0;
    static_assert(M1 == 1 << LJ && M2 == 1 << LI, "member counts are 1, 2 or 4");
    if (S >= ls) return;
    const int up = lane >> (5 - S) & 1;
    if constexpr (S < LJ) {
        constexpr int h = M1 >> (S + 1);
#pragma unroll
        for (int i = 0; i < M2; ++i)
#pragma unroll
            for (int j = 0; j < h; ++j)
#pragma unroll
                for (int e = 0; e < N; ++e)
                    acc[(i * M1 + j) * N + e] =
                        lane_halve<S>(acc[(i * M1 + j) * N + e], acc[(i * M1 + j + h) * N + e], lane);
        nj = h;
        j0 += up * h;
    } else if constexpr (S < LJ + LI) {
        constexpr int h = M2 >> (S - LJ + 1);
#pragma unroll
        for (int i = 0; i < h; ++i)
#pragma unroll
            for (int e = 0; e < N; ++e)
                acc[i * M1 * N + e] = lane_halve<S>(acc[i * M1 * N + e], acc[(i + h) * M1 * N + e], lane);
        ni = h;
        i0 += up * h;
    } else {
#pragma unroll
        for (int e = 0; e < N; ++e) acc[e] = lane_full<S>(acc[e], lane);
        first = first && !up;
    }
    if constexpr (S < 5) lane_reduce<M2, M1, N, S + 1>(acc, ls, lane, i0, ni, j0, nj, first);
}

// Segment kernel for the light classes (J/K modes): one block per segment of
// a bra row, so every item of the block shares the bra pair (a b|.  The
// exchange contributions of a quartet all land in the rows of the two bra
// shells (K[a][c], K[a][d], K[b][c], K[b][d]) and J_ab in one fixed block:
// those are summed in LDS (rows NA + NB of width nbf, LDS atomics) and in
// registers (J_ab, reduced over the wavefront), and added to the XCD's J/K
// copy once per segment, one atomic per nonzero element.  Only J_cd is added
// per quartet.  LDS: ((NA + NB) nbf + NA NB) doubles.
// Bound by the loads and atomics of the digestion (texture data path 29-66 %
// busy, FP64 VALU 16-46 %, over the classes of (H2O)16 cc-pVDZ).  With the ket primitive outside, the bra's in
// scalar registers and the Boys rows in LDS no vector load is left in the
// inner loop: C16H34 6-31G** (ss|ss) 0.69 -> 0.44, (ps|ss) 1.18 -> 0.89 ms,
// (H2O)16 cc-pVDZ (pp|ss) 1.38 -> 0.95, (pp|ps) 1.63 -> 1.49 ms.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// SHARE: the form for lists in which some segments share items between
// lanes; without it every item has one lane.  BT: the block copies the
// coarse Boys rows of its L into LDS, in front of the rows, and reads them
// there.
template <int LA, int LB, int LC, int LD, bool SHARE, bool BT>
__global__ void __launch_bounds__(256) k_eri_seg(EriArgs g) {
    constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
    constexpr int NE = ((LA + LB + 1) * (LA + LB + 2) * (LA + LB + 3) - LA * (LA + 1) * (LA + 2)) / 6;
    constexpr int NF = ((LC + LD + 1) * (LC + LD + 2) * (LC + LD + 3) - LC * (LC + 1) * (LC + 2)) / 6;
    extern __shared__ double lds_all[];
    const double* btab = g.boysA;
    double* seg_lds = lds_all;
    if (BT) {
        const double* src = g.boys + BOYS_COFF + (size_t)(LA + LB + LC + LD) * BOYS_CROWS;
        for (int i = threadIdx.x; i < BOYS_CROWS; i += blockDim.x) lds_all[i] = src[i];
        btab = lds_all;
        seg_lds = lds_all + BOYS_CROWS;      // the first zeroing pass below is followed by a barrier
    }
    const int n = g.nbf;
    double* Kr = seg_lds;                        // rows fa.. (NA) then fb.. (NB), width n
    double* Jl = seg_lds + (size_t)(NA + NB) * n;
    const int total = (NA + NB) * n + NA * NB;
    const size_t off = (size_t)xcd_slot(g.jk_copies) * n * n;
    double* J = g.J + off;
    double* K = g.K + off;
    const int lane = threadIdx.x & 63;
    for (int sg = blockIdx.x; sg < g.nseg; sg += gridDim.x) {
        const SegDesc seg = g.segs[sg];
        const int bp = g.bra_ids[seg.row];
        if (g.dtol > 0.0 && g.segq && g.Qs[bp] * g.segq[sg] * g.dmax[0] < g.dtol) continue;   // block-uniform
        for (int i = threadIdx.x; i < total; i += blockDim.x) seg_lds[i] = 0.0;
        __syncthreads();
        const PairMeta mb = g.meta[bp];
        const int fa = mb.fa, fb = mb.fb;
        const double ABx = g.ab[4 * bp], ABy = g.ab[4 * bp + 1], ABz = g.ab[4 * bp + 2];
        const PrimPair* bra = g.prims + mb.prim_off;
        double jab[NA * NB];
#pragma unroll
        for (int i = 0; i < NA * NB; ++i) jab[i] = 0.0;
        const bool screen = g.dtol > 0.0;
        const int ls = SHARE ? seg.ls : 0, ipw = 64 >> ls, sub = SHARE ? lane >> (6 - ls) : 0;
        const int slot = SHARE ? (threadIdx.x >> 6) * ipw + (lane & (ipw - 1)) : threadIdx.x;
        for (long long t0 = seg.t0; t0 < seg.t0 + seg.n; t0 += blockDim.x >> ls) {
            const long long t = t0 + slot;
            bool live = t < seg.t0 + seg.n;
            if (!SHARE && !screen && !live) continue;
            int pos, b;
            decode_in_row(g, seg.row, live ? t : seg.t0, pos, b);
            const int kp = g.ket_ids[pos];
            if (screen && live) {
                const int2 ab = g.psh[bp], cd = g.psh[kp];
                const size_t ns = g.nsh, a = ab.x, bb = ab.y, c = cd.x, d = cd.y;
                double m = fmax(g.dsh[c * ns + d], g.dsh[a * ns + bb]);
                m = fmax(m, fmax(g.dsh[bb * ns + d], g.dsh[bb * ns + c]));
                m = fmax(m, fmax(g.dsh[a * ns + d], g.dsh[a * ns + c]));
                live = g.Qs[bp] * g.Qs[kp] * m >= g.dtol;
            }
            if (screen) {
                const unsigned long long mask = __ballot(live && sub == 0);
                if (lane == 0 && mask) atomicAdd(g.kept, (unsigned)__popcll(mask));
            }
            if ((!SHARE || ls == 0) && !live) continue;   // with shared items every lane takes part in the sums
            const int nkp = !SHARE || live ? g.meta[kp].nprim : 0;
            const SoaKet kv{g.ksoa + g.bucket_soa[b] + (pos - g.bucket_start[b]),
                            g.bucket_start[b + 1] - g.bucket_start[b], g.kfs};
            double acc[NE * NF];
#pragma unroll
            for (int i = 0; i < NE * NF; ++i) acc[i] = 0.0;
            // ket primitive outer (its fields stay in registers), bra inner
            // (the same for the whole block: scalar loads)
            for (int q = sub; q < nkp; q += 1 << ls) {
                const PrimPair kq = kv.load(q);
                for (int p = 0; p < mb.nprim; ++p)
                    prim_vrr<double, LA, LB, LC, LD, BT>(scalar_load(bra + p), kq, btab, acc);
            }
            if constexpr (SHARE) {
                if (ls) {
                    int i0 = 0, ni = 1, j0 = 0, nj = 1;
                    lane_reduce<1, 1, NE * NF>(acc, ls, lane, i0, ni, j0, nj, live);
                    if (!live) continue;
                }
            }
            const PairMeta mk = g.meta[kp];
            const int fc = mk.fa, fd = mk.fb;
            double v[NA * NB * NC * ND];
            StoreCb<NB, NC, ND, double> st{v};
            ClassCode<LA, LB, LC, LD, double>::hrr(ABx, ABy, ABz, g.ab[4 * kp], g.ab[4 * kp + 1], g.ab[4 * kp + 2],
                                                   acc, st);
            RegDigest<NA, NB, NC, ND, double> cb;
            cb.load(g.D, n, fa, fb, fc, fd);
#pragma unroll
            for (int a = 0; a < NA; ++a)
#pragma unroll
                for (int bb = 0; bb < NB; ++bb)
#pragma unroll
                    for (int c = 0; c < NC; ++c)
#pragma unroll
                        for (int d = 0; d < ND; ++d) cb(a, bb, c, d, v[((a * NB + bb) * NC + c) * ND + d]);
            const double s = (fa == fb ? 0.5 : 1.0) * (fc == fd ? 0.5 : 1.0) * (bp == kp ? 0.5 : 1.0);
#pragma unroll
            for (int i = 0; i < NA * NB; ++i) jab[i] += s * (double)cb.Jab[i];
#pragma unroll
            for (int a = 0; a < NA; ++a) {
#pragma unroll
                for (int c = 0; c < NC; ++c) atomicAdd(&Kr[(size_t)a * n + fc + c], s * (double)cb.Kac[a * NC + c]);
#pragma unroll
                for (int d = 0; d < ND; ++d) atomicAdd(&Kr[(size_t)a * n + fd + d], s * (double)cb.Kad[a * ND + d]);
            }
#pragma unroll
            for (int bb = 0; bb < NB; ++bb) {
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    atomicAdd(&Kr[(size_t)(NA + bb) * n + fc + c], s * (double)cb.Kbc[bb * NC + c]);
#pragma unroll
                for (int d = 0; d < ND; ++d)
                    atomicAdd(&Kr[(size_t)(NA + bb) * n + fd + d], s * (double)cb.Kbd[bb * ND + d]);
            }
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int d = 0; d < ND; ++d)
                    jk_add(&J[(size_t)(fc + c) * n + fd + d], s * (double)cb.Jcd[c * ND + d], g.jk_copies);
        }
#pragma unroll
        for (int i = 0; i < NA * NB; ++i) {
            const double w = wave_sum(jab[i]);
            if (lane == 0) atomicAdd(&Jl[i], w);
        }
        __syncthreads();
        for (int i = threadIdx.x; i < (NA + NB) * n; i += blockDim.x) {
            const double x = Kr[i];
            if (x != 0.0) {
                const int r = i / n, col = i - r * n;
                const int f = r < NA ? fa + r : fb + (r - NA);
                jk_add(&K[(size_t)f * n + col], x, g.jk_copies);
            }
        }
        for (int i = threadIdx.x; i < NA * NB; i += blockDim.x)
            jk_add(&J[(size_t)(fa + i / NB) * n + fb + i % NB], Jl[i], g.jk_copies);
        __syncthreads();
    }
}

// Segment kernel of the generally contracted lists, classes (ls|l's): as
// k_eri_seg, but an item is a pair of generally contracted pairs (GcMeta)
// and computes all member quartets from one primitive loop: for each ket
// primitive, the primitive quartets' [a0|c0] blocks are summed over the bra
// primitives with each bra member's weights, and that sum is added to every
// member quartet with the ket members' weights.  Each member quartet
// that passes the Schwarz test is digested with its own degeneracy weight; a
// list row whose bra equals the ket visits both orders of two different
// members, each at half weight.  LDS: the exchange rows of the up to two
// shells of each bra group ((2 NA + 2) nbf doubles) and J_ab of every bra
// member (MB NA doubles).  (H2O)16 cc-pVDZ: (ss|ss) 2.9 -> 1.2 ms with shared
// items and scalar bra loads, (ps|ss) 3.1 -> 2.2, (ps|ps) 2.6 -> 1.9; texture
// data path 41-77 % busy, FP64 VALU 33-51 %.
// Largest shell-block density maximum between shells {x0, x1} and {y0, y1}
// (x1 / y1 < 0: absent).
__device__ __forceinline__ double gc_dmax(const EriArgs& g, int x0, int x1, int y0, int y1) {
    const size_t ns = g.nsh;
    double m = g.dsh[x0 * ns + y0];
    if (y1 >= 0) m = fmax(m, g.dsh[x0 * ns + y1]);
    if (x1 >= 0) {
        m = fmax(m, g.dsh[x1 * ns + y0]);
        if (y1 >= 0) m = fmax(m, g.dsh[x1 * ns + y1]);
    }
    return m;
}

// The j-th member bound (a select: j differs between lanes).
__device__ __forceinline__ double gc_pick(const double (&q)[4], int j) {
    return j == 0 ? q[0] : j == 1 ? q[1] : j == 2 ? q[2] : q[3];
}

// With density screening (dtol > 0) an item is skipped when the group
// bound (largest member Q of each side times the largest density block over
// the groups' shells) is below dtol, and a member quartet is digested only
// when its own bound Q_ab Q_cd max|D| (six shell blocks) reaches dtol, the
// test the shell-pair lists apply; digested member quartets are counted in
// kept.  BT: the block copies the coarse Boys rows of its L into LDS (in
// front of the rows) and reads them there instead of the aligned global
// table, whose row gathers miss the L1 on most primitive iterations.
// TS: each member quartet's integrals are written to the ERI tensor g.out
// (TensorCb, layout g.tpack) instead of digested; no LDS rows, no J/K.
template <int LA, int LC, bool BT, bool TS = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LA + LC < 2 ? 3 : 2)))
k_eri_gc(EriArgs g) {
    constexpr int NA = ncart(LA), NC = ncart(LC), NI = NA * NC;
    constexpr int MB = LA == 0 ? 4 : 2, MK = LC == 0 ? 4 : 2;
    extern __shared__ double lds_all[];
    const double* btab = g.boysA;
    double* seg_lds = lds_all;
    if (BT) {
        const double* src = g.boys + BOYS_COFF + (size_t)(LA + LC) * BOYS_CROWS;
        for (int i = threadIdx.x; i < BOYS_CROWS; i += blockDim.x) lds_all[i] = src[i];
        btab = lds_all;
        seg_lds = lds_all + BOYS_CROWS;      // the first zeroing pass below is followed by a barrier
    }
    const int n = g.nbf;
    double* Kr = seg_lds;                        // rows fa0.. fa1.. (NA each), fb0, fb1
    double* Jl = seg_lds + (size_t)(2 * NA + 2) * n;
    const int total = (2 * NA + 2) * n + MB * NA;
    const size_t off = (size_t)xcd_slot(g.jk_copies) * n * n;
    double* J = g.J + off;
    double* K = g.K + off;
    const int lane = threadIdx.x & 63;
    const long long fs = g.kfs;
    for (int sg = blockIdx.x; sg < g.nseg; sg += gridDim.x) {
        const SegDesc seg = g.segs[sg];
        const int bp = g.bra_ids[seg.row];
        const GcMeta mb = g.gmeta[bp];
        if (g.dtol > 0.0 && g.segq &&
            fmax(fmax(mb.q[0], mb.q[1]), fmax(mb.q[2], mb.q[3])) * g.segq[sg] * g.dmax[0] < g.dtol)
            continue;   // block-uniform: no item of the segment survives
        if constexpr (!TS)
            for (int i = threadIdx.x; i < total; i += blockDim.x) seg_lds[i] = 0.0;
        __syncthreads();
        const GcPrim* bra = g.gprims + mb.prim_off;
        double jab[MB * NA];
#pragma unroll
        for (int i = 0; i < MB * NA; ++i) jab[i] = 0.0;
        const bool screen = g.dtol > 0.0;
        unsigned nkept = 0;
        const int ls = seg.ls, ipw = 64 >> ls, sub = lane >> (6 - ls);
        const int slot = (threadIdx.x >> 6) * ipw + (lane & (ipw - 1));
        for (long long t0 = seg.t0; t0 < seg.t0 + seg.n; t0 += blockDim.x >> ls) {
            const long long t = t0 + slot;
            bool live = t < seg.t0 + seg.n;
            int pos, b;
            decode_in_row(g, seg.row, live ? t : seg.t0, pos, b);
            const int kp = g.ket_ids[pos];
            if (screen && live) {
                const GcMeta mk = g.gmeta[kp];
                double qb = 0.0, qk = 0.0;
#pragma unroll
                for (int i = 0; i < 4; ++i) { qb = fmax(qb, mb.q[i]); qk = fmax(qk, mk.q[i]); }
                double m = gc_dmax(g, mk.sa0, mk.sa1, mk.sb0, mk.sb1);
                m = fmax(m, gc_dmax(g, mb.sa0, mb.sa1, mb.sb0, mb.sb1));
                m = fmax(m, gc_dmax(g, mb.sb0, mb.sb1, mk.sb0, mk.sb1));
                m = fmax(m, gc_dmax(g, mb.sb0, mb.sb1, mk.sa0, mk.sa1));
                m = fmax(m, gc_dmax(g, mb.sa0, mb.sa1, mk.sb0, mk.sb1));
                m = fmax(m, gc_dmax(g, mb.sa0, mb.sa1, mk.sa0, mk.sa1));
                live = qb * qk * m >= g.dtol;
            }
            if (ls == 0 && !live) continue;       // with shared items every lane takes part in the sums
            const int nkp = live ? g.gmeta[kp].nprim : 0;
            const int nk = g.bucket_start[b + 1] - g.bucket_start[b];
            const double* kb = g.ksoa + g.bucket_soa[b] + (pos - g.bucket_start[b]);
            double acc[MB * MK * NI];
#pragma unroll
            for (int i = 0; i < MB * MK * NI; ++i) acc[i] = 0.0;
            // ket primitive outer (its fields stay in registers), bra inner
            // (the same for the whole block: scalar loads)
            for (int q = sub; q < nkp; q += 1 << ls) {
                const double* x = kb + (long long)q * nk;
                PrimPair kq;
                kq.zeta = x[0]; kq.K = x[fs]; kq.Px = x[2 * fs]; kq.Py = x[3 * fs]; kq.Pz = x[4 * fs];
                kq.PAx = x[5 * fs]; kq.PAy = x[6 * fs]; kq.PAz = x[7 * fs];
                kq.h = 0.0;                     // kets (s s| and (p s| do not enter it
                // sum over the bra primitives with the bra members' weights,
                // then apply the ket members' weights once per ket primitive
                double sb[MB * NI];
#pragma unroll
                for (int i = 0; i < MB * NI; ++i) sb[i] = 0.0;
                for (int p = 0; p < mb.nprim; ++p) {
                    const GcPrim bq = scalar_load(bra + p);
                    double tv[NI];
#pragma unroll
                    for (int i = 0; i < NI; ++i) tv[i] = 0.0;
                    prim_vrr<double, LA, 0, LC, 0, BT>(bq.pp, kq, btab, tv);
#pragma unroll
                    for (int i = 0; i < MB; ++i)
#pragma unroll
                        for (int e = 0; e < NI; ++e) sb[i * NI + e] += bq.w[i] * tv[e];
                }
#pragma unroll
                for (int j = 0; j < MK; ++j) {
                    const double wk = x[(8 + j) * fs];
#pragma unroll
                    for (int i = 0; i < MB; ++i)
#pragma unroll
                        for (int e = 0; e < NI; ++e) acc[(i * MK + j) * NI + e] += wk * sb[i * NI + e];
                }
            }
            int i0 = 0, ni = MB, j0 = 0, nj = MK;
            lane_reduce<MB, MK, NI>(acc, ls, lane, i0, ni, j0, nj, live);
            if (!live) continue;
            // both pairs' data again: keeping the bra's 28 scalars across the
            // primitive loops spilled them
            int kp2 = kp, bp2 = __builtin_amdgcn_readfirstlane(bp);
            asm volatile("" : "+v"(kp2), "+s"(bp2));
            const GcMeta mk = g.gmeta[kp2], mb = g.gmeta[bp2];
            const double sq = bp == kp ? 0.5 : 1.0;
            // ket member outer: its J_cd block is summed over the lane's bra
            // members in registers and added once
#pragma unroll
            for (int jj = 0; jj < MK; ++jj) {
                if (jj >= nj) break;
                const int j = j0 + jj;
                if (j >= mk.m) break;
                const double qkj = gc_pick(mk.q, j);
                const int kc = (mk.code >> (2 * j)) & 1, kd = (mk.code >> (2 * j + 1)) & 1;
                const int fc = kc ? mk.fa1 : mk.fa0, fd = kd ? mk.fb1 : mk.fb0;
                double jcd[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) jcd[c] = 0.0;
                bool any = false;
#pragma unroll
                for (int ii = 0; ii < MB; ++ii) {
                    if (ii >= ni) break;
                    const int i = i0 + ii;
                    if (i >= mb.m) continue;
                    const double qij = gc_pick(mb.q, i) * qkj;
                    if (qij < g.qtol) continue;
                    const int ia = (mb.code >> (2 * i)) & 1, ib = (mb.code >> (2 * i + 1)) & 1;
                    const int fa = ia ? mb.fa1 : mb.fa0, fb = ib ? mb.fb1 : mb.fb0;
                    if (screen) {
                        const size_t ns = g.nsh;
                        const int a = ia ? mb.sa1 : mb.sa0, bb = ib ? mb.sb1 : mb.sb0;
                        const int c = kc ? mk.sa1 : mk.sa0, d = kd ? mk.sb1 : mk.sb0;
                        double m = fmax(g.dsh[c * ns + d], g.dsh[a * ns + bb]);
                        m = fmax(m, fmax(g.dsh[bb * ns + d], g.dsh[bb * ns + c]));
                        m = fmax(m, fmax(g.dsh[a * ns + d], g.dsh[a * ns + c]));
                        if (qij * m < g.dtol) continue;
                        nkept += bp != kp || j <= i;   // both orders of a bra == ket row are one quartet
                    }
                    double v[NI];
                    StoreCb<1, NC, 1, double> st{v};
                    ClassCode<LA, 0, LC, 0, double>::hrr(0.0, 0.0, 0.0, 0.0, 0.0, 0.0, acc + (ii * MK + jj) * NI, st);
                    if constexpr (TS) {
                        TensorCb tc{g.out, (size_t)n, fa, fb, fc, fd, g.tpack};
#pragma unroll
                        for (int a = 0; a < NA; ++a)
#pragma unroll
                            for (int c = 0; c < NC; ++c) tc(a, 0, c, 0, v[a * NC + c]);
                        continue;
                    }
                    RegDigest<NA, 1, NC, 1, double> cb;
                    cb.load(g.D, n, fa, fb, fc, fd);
#pragma unroll
                    for (int a = 0; a < NA; ++a)
#pragma unroll
                        for (int c = 0; c < NC; ++c) cb(a, 0, c, 0, v[a * NC + c]);
                    const double s = (fa == fb ? 0.5 : 1.0) * (fc == fd ? 0.5 : 1.0) * sq;
#pragma unroll
                    for (int a = 0; a < NA; ++a) {
                        // a lane of a shared item keeps other members than 0 .. ni - 1
#pragma unroll
                        for (int x = 0; x < MB; ++x) jab[x * NA + a] += x == i ? s * cb.Jab[a] : 0.0;
                        double* row = Kr + (size_t)(ia * NA + a) * n;
#pragma unroll
                        for (int c = 0; c < NC; ++c) atomicAdd(&row[fc + c], s * cb.Kac[a * NC + c]);
                        atomicAdd(&row[fd], s * cb.Kad[a]);
                    }
                    double* rowb = Kr + (size_t)(2 * NA + ib) * n;
#pragma unroll
                    for (int c = 0; c < NC; ++c) atomicAdd(&rowb[fc + c], s * cb.Kbc[c]);
                    atomicAdd(&rowb[fd], s * cb.Kbd[0]);
#pragma unroll
                    for (int c = 0; c < NC; ++c) jcd[c] += s * cb.Jcd[c];
                    any = true;
                }
                if (any) {
#pragma unroll
                    for (int c = 0; c < NC; ++c) jk_add(&J[(size_t)(fc + c) * n + fd], jcd[c], g.jk_copies);
                }
            }
        }
        if constexpr (!TS) {
#pragma unroll
            for (int i = 0; i < MB * NA; ++i) {
                const double w = wave_sum(jab[i]);
                if (lane == 0 && i < mb.m * NA) atomicAdd(&Jl[i], w);
            }
        }
        if (screen) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) nkept += __shfl_xor(nkept, o, 64);
            if (lane == 0 && nkept) atomicAdd(g.kept, nkept);
        }
        __syncthreads();
        if constexpr (!TS) {
            for (int i = threadIdx.x; i < (2 * NA + 2) * n; i += blockDim.x) {
                const double x = Kr[i];
                if (x != 0.0) {
                    const int r = i / n, col = i - r * n;
                    const int f =
                        r < 2 * NA ? (r < NA ? mb.fa0 + r : mb.fa1 + (r - NA)) : (r == 2 * NA ? mb.fb0 : mb.fb1);
                    jk_add(&K[(size_t)f * n + col], x, g.jk_copies);
                }
            }
            for (int i = threadIdx.x; i < mb.m * NA; i += blockDim.x) {
                const int j = i / NA, a = i - j * NA;
                const int fa = ((mb.code >> (2 * j)) & 1) ? mb.fa1 : mb.fa0;
                const int fb = ((mb.code >> (2 * j + 1)) & 1) ? mb.fb1 : mb.fb0;
                jk_add(&J[(size_t)(fa + a) * n + fb], Jl[i], g.jk_copies);
            }
        }
        __syncthreads();
    }
}

// Segment kernel for classes (ab|c s) whose bra is a shell pair and whose
// kets are generally contracted pairs ((pp|ss) (pp|ps) (ds|ps) (dp|ss)):
// bra and ket classes differ, so no bra-ket symmetry is involved.  For each
// ket primitive the VRR sums over the bra primitives (the block's shared
// bra), and that block is added to every ket member with its weight; after
// the loops the bra HRR runs per ket member, whose quartet is digested as in
// k_eri_seg when it passes Q_ab q_cd >= qtol (and, screened, the density
// test of the shell-pair lists).  LDS as k_eri_seg.
// One member quartet of k_eri_gck: bra HRR of its [e0|c0] block, then the
// segment kernel's digestion (exchange rows of the bra shells in LDS, J_ab
// in jab, J_cd to the global copy).
template <int LA, int LB, int LC>
__device__ __forceinline__ void gck_digest(const EriArgs& g, const double* acc, double ABx, double ABy, double ABz,
                                           int fa, int fb, int fc, int fd, double* Kr, double* J, double* jab) {
    constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC);
    const int n = g.nbf;
    double v[NA * NB * NC];
    StoreCb<NB, NC, 1, double> st{v};
    ClassCode<LA, LB, LC, 0, double>::hrr(ABx, ABy, ABz, 0.0, 0.0, 0.0, acc, st);
    RegDigest<NA, NB, NC, 1, double> cb;
    cb.load(g.D, n, fa, fb, fc, fd);
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int bb = 0; bb < NB; ++bb)
#pragma unroll
            for (int c = 0; c < NC; ++c) cb(a, bb, c, 0, v[(a * NB + bb) * NC + c]);
    const double s = (fa == fb ? 0.5 : 1.0) * (fc == fd ? 0.5 : 1.0);
#pragma unroll
    for (int i = 0; i < NA * NB; ++i) jab[i] += s * cb.Jab[i];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
#pragma unroll
        for (int c = 0; c < NC; ++c) atomicAdd(&Kr[(size_t)a * n + fc + c], s * cb.Kac[a * NC + c]);
        atomicAdd(&Kr[(size_t)a * n + fd], s * cb.Kad[a]);
    }
#pragma unroll
    for (int bb = 0; bb < NB; ++bb) {
#pragma unroll
        for (int c = 0; c < NC; ++c) atomicAdd(&Kr[(size_t)(NA + bb) * n + fc + c], s * cb.Kbc[bb * NC + c]);
        atomicAdd(&Kr[(size_t)(NA + bb) * n + fd], s * cb.Kbd[bb]);
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) jk_add(&J[(size_t)(fc + c) * n + fd], s * cb.Jcd[c], g.jk_copies);
}

// BT: the coarse Boys rows in LDS, as in k_eri_gc.
template <int LA, int LB, int LC, bool BT>
__global__ void __launch_bounds__(256) k_eri_gck(EriArgs g) {
    constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC);
    constexpr int NE = ((LA + LB + 1) * (LA + LB + 2) * (LA + LB + 3) - LA * (LA + 1) * (LA + 2)) / 6;
    constexpr int NF = ncart(LC);
    constexpr int MK = LC == 0 ? 4 : 2;
    extern __shared__ double lds_all[];
    const double* btab = g.boysA;
    double* seg_lds = lds_all;
    if (BT) {
        const double* src = g.boys + BOYS_COFF + (size_t)(LA + LB + LC) * BOYS_CROWS;
        for (int i = threadIdx.x; i < BOYS_CROWS; i += blockDim.x) lds_all[i] = src[i];
        btab = lds_all;
        seg_lds = lds_all + BOYS_CROWS;      // the first zeroing pass below is followed by a barrier
    }
    const int n = g.nbf;
    double* Kr = seg_lds;                        // rows fa.. (NA) then fb.. (NB), width n
    double* Jl = seg_lds + (size_t)(NA + NB) * n;
    const int total = (NA + NB) * n + NA * NB;
    const size_t off = (size_t)xcd_slot(g.jk_copies) * n * n;
    double* J = g.J + off;
    double* K = g.K + off;
    const int lane = threadIdx.x & 63;
    const long long fs = g.kfs;
    for (int sg = blockIdx.x; sg < g.nseg; sg += gridDim.x) {
        const SegDesc seg = g.segs[sg];
        const int bp = g.bra_ids[seg.row];
        if (g.dtol > 0.0 && g.segq && g.Qs[bp] * g.segq[sg] * g.dmax[0] < g.dtol) continue;   // block-uniform
        for (int i = threadIdx.x; i < total; i += blockDim.x) seg_lds[i] = 0.0;
        __syncthreads();
        const PairMeta mb = g.meta[bp];
        const int fa = mb.fa, fb = mb.fb;
        const double ABx = g.ab[4 * bp], ABy = g.ab[4 * bp + 1], ABz = g.ab[4 * bp + 2];
        const PrimPair* bra = g.prims + mb.prim_off;
        const double qb = g.Qs[bp];
        const bool screen = g.dtol > 0.0;
        double jab[NA * NB];
#pragma unroll
        for (int i = 0; i < NA * NB; ++i) jab[i] = 0.0;
        unsigned nkept = 0;
        const int ls = seg.ls, ipw = 64 >> ls, sub = lane >> (6 - ls);
        const int slot = (threadIdx.x >> 6) * ipw + (lane & (ipw - 1));
        for (long long t0 = seg.t0; t0 < seg.t0 + seg.n; t0 += blockDim.x >> ls) {
            const long long t = t0 + slot;
            bool live = t < seg.t0 + seg.n;
            int pos, b;
            decode_in_row(g, seg.row, live ? t : seg.t0, pos, b);
            const int kp = g.ket_ids[pos];
            const int2 ab = screen ? g.psh[bp] : make_int2(0, 0);
            if (screen && live) {
                const GcMeta mk = g.gmeta[kp];
                double qk = 0.0;
#pragma unroll
                for (int i = 0; i < 4; ++i) qk = fmax(qk, mk.q[i]);
                double m = gc_dmax(g, mk.sa0, mk.sa1, mk.sb0, mk.sb1);
                m = fmax(m, g.dsh[(size_t)ab.x * g.nsh + ab.y]);
                m = fmax(m, gc_dmax(g, ab.y, -1, mk.sb0, mk.sb1));
                m = fmax(m, gc_dmax(g, ab.y, -1, mk.sa0, mk.sa1));
                m = fmax(m, gc_dmax(g, ab.x, -1, mk.sb0, mk.sb1));
                m = fmax(m, gc_dmax(g, ab.x, -1, mk.sa0, mk.sa1));
                live = qb * qk * m >= g.dtol;
            }
            if (ls == 0 && !live) continue;       // with shared items every lane takes part in the sums
            const int nkp = live ? g.gmeta[kp].nprim : 0;
            const int nk = g.bucket_start[b + 1] - g.bucket_start[b];
            const double* kb = g.ksoa + g.bucket_soa[b] + (pos - g.bucket_start[b]);
            double acc[MK * NE * NF];
#pragma unroll
            for (int i = 0; i < MK * NE * NF; ++i) acc[i] = 0.0;
            for (int q = sub; q < nkp; q += 1 << ls) {
                const double* x = kb + (long long)q * nk;
                PrimPair kq;
                kq.zeta = x[0]; kq.K = x[fs]; kq.Px = x[2 * fs]; kq.Py = x[3 * fs]; kq.Pz = x[4 * fs];
                kq.PAx = x[5 * fs]; kq.PAy = x[6 * fs]; kq.PAz = x[7 * fs];
                kq.h = 0.0;                     // kets (s s| and (p s| do not enter it
                double sb[NE * NF];
#pragma unroll
                for (int i = 0; i < NE * NF; ++i) sb[i] = 0.0;
                for (int p = 0; p < mb.nprim; ++p) prim_vrr<double, LA, LB, LC, 0, BT>(scalar_load(bra + p), kq, btab, sb);
#pragma unroll
                for (int j = 0; j < MK; ++j) {
                    const double wk = x[(8 + j) * fs];
#pragma unroll
                    for (int e = 0; e < NE * NF; ++e) acc[j * NE * NF + e] += wk * sb[e];
                }
            }
            int i0 = 0, ni = 1, j0 = 0, nj = MK;
            lane_reduce<1, MK, NE * NF>(acc, ls, lane, i0, ni, j0, nj, live);
            if (!live) continue;
            const GcMeta mk = g.gmeta[kp];
            // one digestion instance: the lane's next member is always in
            // acc[0 ..), the accumulators move down one member after each step
#pragma unroll 1
            for (int jj = 0; jj < nj; ++jj) {
                const int j = j0 + jj;
                if (j >= mk.m) break;
                const double qkj = gc_pick(mk.q, j);
                const int kc = (mk.code >> (2 * j)) & 1, kd = (mk.code >> (2 * j + 1)) & 1;
                const int fc = kc ? mk.fa1 : mk.fa0, fd = kd ? mk.fb1 : mk.fb0;
                bool keep = qb * qkj >= g.qtol;
                if (screen && keep) {
                    const size_t ns = g.nsh;
                    const int c = kc ? mk.sa1 : mk.sa0, d = kd ? mk.sb1 : mk.sb0;
                    double m = fmax(g.dsh[c * ns + d], g.dsh[ab.x * ns + ab.y]);
                    m = fmax(m, fmax(g.dsh[ab.y * ns + d], g.dsh[ab.y * ns + c]));
                    m = fmax(m, fmax(g.dsh[ab.x * ns + d], g.dsh[ab.x * ns + c]));
                    keep = qb * qkj * m >= g.dtol;
                    nkept += keep;
                }
                if (keep) gck_digest<LA, LB, LC>(g, acc, ABx, ABy, ABz, fa, fb, fc, fd, Kr, J, jab);
#pragma unroll
                for (int x = 0; x + 1 < MK; ++x)
#pragma unroll
                    for (int e = 0; e < NE * NF; ++e) acc[x * NE * NF + e] = acc[(x + 1) * NE * NF + e];
            }
        }
#pragma unroll
        for (int i = 0; i < NA * NB; ++i) {
            const double w = wave_sum(jab[i]);
            if (lane == 0) atomicAdd(&Jl[i], w);
        }
        if (screen) {
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) nkept += __shfl_xor(nkept, o, 64);
            if (lane == 0 && nkept) atomicAdd(g.kept, nkept);
        }
        __syncthreads();
        for (int i = threadIdx.x; i < (NA + NB) * n; i += blockDim.x) {
            const double x = Kr[i];
            if (x != 0.0) {
                const int r = i / n, col = i - r * n;
                const int f = r < NA ? fa + r : fb + (r - NA);
                jk_add(&K[(size_t)f * n + col], x, g.jk_copies);
            }
        }
        for (int i = threadIdx.x; i < NA * NB; i += blockDim.x)
            jk_add(&J[(size_t)(fa + i / NB) * n + fb + i % NB], Jl[i], g.jk_copies);
        __syncthreads();
    }
}

typedef void (*EriKernel)(EriArgs);
// Getter modes of polyeri_class_kernel beyond the k_eri modes: the segment
// kernel (MODE_JK), the one with items shared between lanes, and the latter
// with the Boys rows read from global memory (the first two need BOYS_CROWS
// doubles more LDS).
enum { GET_SEG_JK = 5, GET_SEG_SHARE = 6, GET_SEG_SHARE_G = 7 };
// Strided batched FP64 products on the MFMA units (kgemm.hip):
// C_b(m,n) = sum_k A_b(m,k) B_b(k,n), X_b(r,c) = X[b*sX + r*sXr + c*sXc].
enum { GEMM_F64 = 1, GEMM_BF16X3 = 2 };
int polyeri_gemm_launch(int mode, int M, int N, int K, const double* A, long sam, long sak, long sA, const double* B,
                        long sbk, long sbn, long sB, double* C, long scm, long scn, long sC, int batch,
                        hipStream_t stream);
// Planar complex products C_b = A_b B_b (A real when Ai is null), same
// strides for the real and imaginary planes, k contiguous in A and n in B
// (kgemm.hip; C linkage for its test).  nci > 0 splits the columns of B and C as (n / nci, n % nci)
// with outer strides sbo / sco, mci > 0 the rows of C as (m / mci, m % mci)
// with outer stride smo.
extern "C" int polyeri_zgemm_launch(int mode, int M, int N, int K, const double* Ar, const double* Ai, long sam,
                                    long sA, const double* Br, const double* Bi, long sbk, long sB, double* Cr,
                                    double* Ci, long scm, long scn, long sC, int batch, hipStream_t stream,
                                    int nci = 0, long sbo = 0, long sco = 0, int mci = 0, long smo = 0);
// Density screening (kscreen.hip): shell-block maxima of |D|, and the
// compaction of one work list to the items whose bound
// Q_ab Q_cd max(|D| over the six blocks the quartet reads) reaches tol.
int polyeri_shell_dmax(const double* D, int nbf, const int* shell_f0, const int* shell_nf, int nsh,
                       double* dsh, hipStream_t stream);
// *out = the largest of the n values x (one block).
int polyeri_max_reduce(const double* x, size_t n, double* out, hipStream_t stream);
int polyeri_screen_list(const EriArgs& a, const double* Q, const int2* pair_shells, const double* dsh,
                        int nsh, double tol, int2* items, unsigned* count, hipStream_t stream);
// Cooperative (one wavefront per quartet, LDS-resident recursion) kernels;
// primitive quartets are prepared in batches of 2^pbs (pbs 0..3).
int polyeri_coop_nslot(int la, int lb, int lc, int ld, int pbs);
int polyeri_coop_launch(const EriArgs& a, int mode, int la, int lb, int lc, int ld, int pbs, int max_grid,
                        hipStream_t stream);
// default batch: eight for the classes whose LDS is small enough that the
// records cost no occupancy, one otherwise
inline int polyeri_coop_default_pbs(int nint) { return nint < 200 ? 3 : 0; }
// Generally contracted segment kernel (kgc.hip): LDS bytes, whether the
// class (la s|lc s) has one, and the launch over a.segs (grid blocks).
size_t polyeri_gc_lds_bytes(int la, int nbf);
bool polyeri_gc_class(int la, int lc);
int polyeri_gc_launch(const EriArgs& a, int la, int lc, int block, int grid, hipStream_t stream, bool tensor = false);
// The same for k_eri_gck (shell-pair bra (la lb|, generally contracted kets |lc s)).
size_t polyeri_gck_lds_bytes(int la, int lb, int nbf);
bool polyeri_gck_class(int la, int lb, int lc);
int polyeri_gck_launch(const EriArgs& a, int la, int lb, int lc, int block, int grid, hipStream_t stream);
// Rys-quadrature segment kernels (krys.hip) for the classes (dp|pp) (dp|dp)
// (dd|pp) (dd|ds) (dd|dp) (dd|dd): J/K over bra-row segments, mode MODE_JK
// or MODE_JK32 (FP32 recursion).
bool polyeri_rys_class(int la, int lb, int lc, int ld);
size_t polyeri_rys_lds_bytes(int la, int lb, int nbf);
int polyeri_rys_launch(const EriArgs& a, int mode, int la, int lb, int lc, int ld, int block, int max_grid,
                       hipStream_t stream);
// Nodes u[0..n-1] and weights w[0..n-1] of the n-point Rys rule at T, n <= 5
// (host evaluation of the kernels' tables).
int polyeri_rys_nodes_host(int n, double T, double* u, double* w);
// One primitive quartet's Cartesian block through the kernels' per-lane Rys
// code on the host (0; -1 bad class or pointer; -2 an integral not produced
// exactly once).
int polyeri_rys_block_host(int la, int lb, int lc, int ld, const double* xyz, const double* ex, double* out);

// Two-electron part of the nuclear gradient (kgrad.hip): per shell its atom,
// first function and centre, the density in the library's basis (nbf x nbf)
// and its largest |element| per shell block (nsh x nsh), the threshold on
// Q_ab Q_cd and on Q_ab Q_cd max |Gamma|, the exchange scale.
// Shell pairs (pa[i], pb[i]) with L(pa) >= L(pb), their Schwarz bounds and
// their primitive pairs prims[pp0[i]] .. + pn[i] - 1, grouped by pair class
// ((ss) (ps) (pp) (ds) (dp) (dd) = 0 .. 5: pairs seg[X] .. seg[X + 1] - 1),
// by primitive count inside a class; the quartets of class pair X >= Y run
// as one launch of the kernel for that class.
struct GradArgs {
    int nsh, natom, nbf, npair;
    int seg[7];
    const int *atom, *f0;
    const int *pa, *pb, *pp0, *pn;
    const PrimPair* prims;
    const double* xyz;
    const double* D;
    const double* dsh;
    const double* Qp;
    double tol, xfac;
    // the Schwarz survivors of one class pair as chunks: chunk c holds lanes
    // coff[c] .. coff[c + 1] - 1, cij[3c + 2] to a quartet of bra pair x0 +
    // cij[3c] and ket pairs y0 + cij[3c + 1] + 0, 1, ..
    const unsigned long long* coff = nullptr;
    const int* cij = nullptr;
    int nchunk = 0;
};
// One root of a primitive quartet is a unit of work in the classes of this
// many integrals and more, a whole primitive quartet below.
constexpr bool grad_root_units(int nint) { return nint >= 36; }

// Shells and primitives for the host's Schwarz bounds, ptol the primitive
// pair threshold.
struct GradShells {
    const int *L, *p0, *np;
    const double *xyz, *alpha, *coef;
    double ptol;
};

// Schwarz-surviving quartets of every class pair (X, Y <= X) of pairs sorted
// by polyeri_grad_sort_pairs: inside a class, pairs of one primitive count
// class (a group) are in descending bound order, so the kets of a group that
// survive with a given bra are a prefix of the group.  Class pair k = 6X + Y
// has n[k] chunks, offsets off[off0[k]] .. off[off0[k] + n[k]] (in lanes) and
// (row, first column, lanes a quartet) triples ij[ij0[k] ..].
struct GradChunks {
    std::vector<unsigned long long> off;
    std::vector<int> ij;
    size_t off0[36], ij0[36];
    int n[36];
    unsigned long long nlane[36];
    double units[36];
};
// grad (3 natom, zeroed by the caller) += dE2/dR on the device: the chunks ch
// (with d_off / d_ij its off / ij arrays on the device), the class pairs dealt
// over the ns streams, costliest first.
int polyeri_grad_launch(const GradArgs& g, double* d_grad, const hipStream_t* streams, int ns, const GradChunks& ch,
                        const unsigned long long* d_off, const int* d_ij);
// Orders the pairs of every class segment by primitive count class
// (descending) and, inside one, by bound (descending); pa, pb, qp, pp0 and pn
// permuted together.  False (nothing changed) when a bound is not finite.
bool polyeri_grad_sort_pairs(int* pa, int* pb, double* qp, int* pp0, int* pn, const int* seg);
// The chunks of the pairs whose bound product is >= tol (sorted = false: of
// all pairs, in their order), with the lanes each quartet gets.
void polyeri_grad_chunks(const double* qp, const int* pn, const int* seg, double tol, bool sorted,
                         GradChunks& ch);
// the same sum on the host (host pointers), grad overwritten, Schwarz bounds
// from gs
int polyeri_grad_host(const GradArgs& g, const GradShells& gs, double* grad);
// One record of the reference's .ao files (kstored.hip): packed cells,
// packed 1-based indices I J K L, the integral.
struct StoredEri {
    int32_t cells, ijkl;
    double v;
};
// J/K blocks (reference layout, 2 cel1 + 1 cells or 1) from n records.
int polyeri_jk_stored_launch(const StoredEri* rec, long long n, int nc, int cel1, int cel2, const double* P, double* J,
                             double* K, hipStream_t s);
// Internal-function AO tensor of a molecule from n records.
int polyeri_tensor_stored_launch(const StoredEri* rec, long long n, const int* inv, const double* scale, int nbf,
                                 double* T, hipStream_t s);
// Classes with more than this many integrals per quartet run cooperatively.
#define POLYERI_COOP_MIN_INTEGRALS 108
// Kernel of class (la lb|lc ld) and mode, or nullptr (generated getters).
EriKernel polyeri_class_kernel(int la, int lb, int lc, int ld, int mode);
