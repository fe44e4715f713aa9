// Batched per-sector factorisations in FP64: SVD (one-sided Jacobi), QR (Householder, with the
// reflector convention of Eigen::HouseholderQR), inverse Cholesky factors and symmetric eigen
// (parallel cyclic Jacobi).
//
// One workgroup owns one sector block.  Blocks that fit the LDS budget are factorised entirely in
// LDS; larger ones use a global-memory working copy with the same algorithm, except for the SVD,
// whose larger blocks go to block Jacobi (bjsvd.hip).
//
// The reference calls Eigen per sector (PlainInterface::svd, PlainInterface_Eigen_impl.cpp:116-127;
// MatrixInterface::qr, MatrixInterface_Eigen_impl.cpp:249-255; MatrixInterface::eigh,
// MatrixInterface_Eigen_impl.hpp:242-247), serially over sectors (Tensor.cpp:510-519, 762-777,
// 782-803).
#include <algorithm>
#include <cfloat>
#include <cstring>
#include <iterator>
#include <type_traits>

#include "device.hpp"

using xh::check;
using xh::guard;

namespace {

constexpr int F_THREADS = 256;
constexpr int MAX_SWEEPS = 60;

__device__ __forceinline__ int rr_player(int pos, int step, int n2)
{
    // circle method: position 0 is fixed, the others rotate by one each step (step < n2 - 1)
    if(pos == 0) return 0;
    const int q = pos + step;
    return q >= n2 ? q - (n2 - 1) : q;
}

// total orders over doubles for rank-based sorting: NaN below (above) every number
__device__ __forceinline__ double nan_low(double x) { return x == x ? x : -DBL_MAX * 2.0; }
__device__ __forceinline__ double nan_high(double x) { return x == x ? x : DBL_MAX * 2.0; }

struct FactorArgs {
    const xh_factor_item* items;
    const double* A;
    double* U;
    double* S;
    double* Vt;
    double* scratch;
    int64_t scratch_stride;
    int use_lds;
    int* status;
};

// The working set of a workgroup: dynamic LDS, or its slice of the global scratch.  Resolved at
// compile time, so that LDS accesses compile to LDS instructions (a pointer that may point to
// either space compiles to flat loads and stores, which wait on both memory counters).
template <bool LDS>
__device__ __forceinline__ double* work_base(double* smem, const FactorArgs& fa)
{
    if constexpr(LDS)
        return smem;
    else
        return fa.scratch + int64_t(blockIdx.x) * fa.scratch_stride;
}

// One-sided Jacobi SVD of a block worked on as mm x nn (mm >= nn, transposed where needed), one
// workgroup per block.  Working set in LDS: W (nn columns of ldw), V (nn columns of ldv), sigma
// (nn), order (nn ints).
//
// The kernel is a serial chain of (nn - 1) steps per sweep, each the latency of one rotation: the
// columns of a pair read from LDS, an inner product, the angle, the update, a barrier.  So G = 16
// lanes own a pair (two rows each per 16-byte LDS access; 64 lanes in tall blocks, SVD_TALL) and
// reduce by DPP; the columns of W stay in registers between the inner product and the update (RM > 0:
// rows <= 32 RM; RM = 0: any number, read twice); V is read only when the pair rotates.  Squared
// column norms are kept beside W, moved with each rotation, summed afresh where a rotation takes
// most of a column away and for every column before each sweep, so the last sweep, which finds
// every pair orthogonal, judges by fresh norms.  A block of more than BJ_MIN_COLS columns with a
// non-finite sum of squares is refused, as block Jacobi refuses it.
//
// Range: the block is scaled by a power of two to a largest finite entry of [2^229, 2^230).  Squared
// norms are then at most 2^475, and the products of two of them in range unless both columns are
// tiny; such a pair is scaled once more for its test and its angle, in a copy of the steps for blocks
// that have tiny columns (asked for each pair, it took 3 to 6 % more).  Only columns below
// sqrt(SVD_ZERO), 2e-214 of the largest entry, are left alone.
// (64 to 8 lanes per pair, three reductions through ds_bpermute, IEEE divisions and square roots
// took 542 us for the 9 blocks, 32 x 32 the largest, of a two-site tensor at bond 64; three DPP
// reductions and refined quotients 220 us; this takes 180 us.)
constexpr int SVD_THREADS = 1024;

// Blocks with more columns than this (after transposition) use the block Jacobi path: any block of
// a call where some block has to (a block of 65 to 98 columns then adds nothing to steps that run
// anyway, but 1.4 ms by itself), and only those that do not fit LDS in a call of smaller blocks
// (15 sectors of up to 74 columns: 0.46 ms by themselves, 1.07 ms with block Jacobi and its products).
constexpr int BJ_MIN_COLS = 64, BJ_MIN_COLS_ALONE = 98;

__host__ __device__ inline int svd_ld(int rows) { return (rows + 1) & ~1; }
__host__ __device__ inline int64_t svd_work_doubles(int64_t mm, int64_t nn)
{
    return nn * (svd_ld(int(mm)) + svd_ld(int(nn))) + nn + (nn + 1) / 2 + 2;
}

typedef double d2 __attribute__((ext_vector_type(2)));

constexpr int SVD_EXP = 230;            // the largest entry is scaled to below 2^SVD_EXP
constexpr double SVD_ZERO = 0x1p-960;   // squared norm of a column taken as zero
constexpr double SVD_SMALL = 0x1p-450;  // tiny: two such squared norms have their product scaled
constexpr double SVD_NEAR = 1e-14;      // squared cosine below which a sweep counts as nearly converged

// al, be and ga of a pair with al be < SVD_SMALL^2 times a power of two: the larger norm to about 2^400,
// the smaller one, at least SVD_ZERO, then above 2^-621
__device__ __forceinline__ void scale_pair(double& al, double& be, double& ga)
{
    if(al * be >= SVD_SMALL * SVD_SMALL) return;
    int e;
    frexp(fmax(al, be), &e);
    al = ldexp(al, 400 - e);
    be = ldexp(be, 400 - e);
    ga = ldexp(ga, 400 - e);
}

template <int RM, int VM, int G = 16>
__global__ __launch_bounds__(SVD_THREADS) void k_svd_jacobi(FactorArgs fa)
{
    extern __shared__ __attribute__((aligned(16))) double smem[];
    __shared__ int rotated, far;  // a pair was rotated this sweep; one by more than SVD_NEAR
    __shared__ int s_tiny;        // a column was tiny at the start of a sweep
    __shared__ double s_max[SVD_THREADS / 64], s_sq[SVD_THREADS / 64];
    const xh_factor_item it = fa.items[blockIdx.x];
    const int m = it.m, n = it.n;
    if(m == 0 || n == 0) return;
    const bool tr = m < n;
    const int mm = tr ? n : m, nn = tr ? m : n;
    const int ldw = svd_ld(mm), ldv = svd_ld(nn);
    double* W = smem;
    double* V = W + int64_t(ldw) * nn;
    double* sig = V + int64_t(ldv) * nn;
    int* ord = reinterpret_cast<int*>(sig + nn);
    constexpr int RR = RM > 0 ? RM : 1;
    constexpr bool WIDE = 32 * VM > BJ_MIN_COLS;  // may hold blocks that are refused where not finite
    const int tid = threadIdx.x, gl = tid % G, grp = tid / G, ngroups = blockDim.x / G;
    double mx = 0.0, sq = 0.0;
    for(int j = grp; j < nn; j += ngroups) {
        for(int i = gl; i < ldw; i += G) {
            const double v = i >= mm ? 0.0 : tr ? fa.A[it.a_off + j + int64_t(i) * m] : fa.A[it.a_off + i + int64_t(j) * m];
            W[j * ldw + i] = v;
            mx = fmax(mx, isfinite(v) ? fabs(v) : 0.0);
            sq = fma(v, v, sq);
        }
        for(int i = gl; i < ldv; i += G) V[j * ldv + i] = i == j ? 1.0 : 0.0;
    }
    for(int o = 32; o > 0; o >>= 1) {
        mx = fmax(mx, __shfl_xor(mx, o));
        if constexpr(WIDE) sq += __shfl_xor(sq, o);
    }
    if((tid & 63) == 0) {
        s_max[tid >> 6] = mx;
        if constexpr(WIDE) s_sq[tid >> 6] = sq;
    }
    __syncthreads();
    sq = 0.0;
    for(int w = 0; w < int(blockDim.x >> 6); ++w) {
        mx = fmax(mx, s_max[w]);
        if constexpr(WIDE) sq += s_sq[w];
    }
    if(WIDE && nn > BJ_MIN_COLS && !isfinite(sq)) {  // the same in every thread
        if(tid == 0) atomicOr(fa.status, XH_EINVAL);
        return;
    }
    int ex = 0;
    if(mx > 0.0) frexp(mx, &ex);
    ex -= SVD_EXP;

    const int n2 = nn + (nn & 1);
    const int npairs = n2 / 2;
    const double tol = fmax(1.0, sqrt(static_cast<double>(mm))) * DBL_EPSILON, tol2 = tol * tol;
    const int nw = (ldw >> 1) - gl, nv = (ldv >> 1) - gl;  // this lane's row pairs: 0, G, 2 G, ... below these
    auto norm2 = [&](int j) {
        double s = 0.0;
        const d2* w = reinterpret_cast<const d2*>(W + j * ldw) + gl;
        for(int k = 0; k < nw; k += G) {
            const d2 a = w[k];
            s = fma(a[0], a[0], s);
            s = fma(a[1], a[1], s);
        }
        return xh::lanes_sum<G>(s);
    };
    for(int j = grp; j < nn; j += ngroups)
        for(int i = gl; i < ldw; i += G) W[j * ldw + i] = ldexp(W[j * ldw + i], -ex);
    // the pair of positions (grp, n2 - 1 - grp) of the circle: position 0 keeps its column, the
    // others move on by one each step and are back after the n2 - 1 steps of a sweep
    int a = grp, b = n2 - 1 - grp;
    // the n2 - 1 steps of a sweep
    auto steps = [&](auto has_tiny) {
        constexpr bool tiny = decltype(has_tiny)::value;
        for(int step = 0; step < n2 - 1; ++step) {
            if(grp < npairs && max(a, b) < nn) {  // a dummy column fills an odd count
                d2* wi = reinterpret_cast<d2*>(W + __mul24(a, ldw)) + gl;
                d2* wj = reinterpret_cast<d2*>(W + __mul24(b, ldw)) + gl;
                const double al = sig[a], be = sig[b];
                d2 x[RR], y[RR];
                double ga = 0;
                if constexpr(RM > 0) {
#pragma unroll
                    for(int k = 0; k < RM; ++k) {
                        x[k] = d2{0.0, 0.0};
                        y[k] = d2{0.0, 0.0};
                        if(k * G < nw) {
                            x[k] = wi[k * G];
                            y[k] = wj[k * G];
                        }
                    }
#pragma unroll
                    for(int k = 0; k < RM; ++k) {
                        ga = fma(x[k][0], y[k][0], ga);
                        ga = fma(x[k][1], y[k][1], ga);
                    }
                } else {
                    for(int k = 0; k < nw; k += G) {
                        const d2 p = wi[k], q = wj[k];
                        ga = fma(p[0], q[0], ga);
                        ga = fma(p[1], q[1], ga);
                    }
                }
                ga = xh::lanes_sum<G>(ga);
                double sa = al, sb = be, sg = ga;  // scaled where the products would underflow
                if constexpr(tiny) scale_pair(sa, sb, sg);
                if(fmin(al, be) > SVD_ZERO && sg * sg > tol2 * (sa * sb)) {
                    d2* vi = reinterpret_cast<d2*>(V + __mul24(a, ldv)) + gl;
                    d2* vj = reinterpret_cast<d2*>(V + __mul24(b, ldv)) + gl;
                    d2 u[VM], v[VM];
#pragma unroll
                    for(int k = 0; k < VM; ++k)
                        if(k * G < nv) {
                            u[k] = vi[k * G];
                            v[k] = vj[k * G];
                        }
                    double c, s;
                    xh::jacobi_rotation(0.5 * (sb - sa), sg, c, s);
                    if constexpr(RM > 0) {
#pragma unroll
                        for(int k = 0; k < RM; ++k) {
                            const d2 p = x[k];
                            x[k] = c * p - s * y[k];
                            y[k] = s * p + c * y[k];
                            if(k * G < nw) {
                                wi[k * G] = x[k];
                                wj[k * G] = y[k];
                            }
                        }
                    } else {
                        for(int k = 0; k < nw; k += G) {
                            const d2 p = wi[k], q = wj[k];
                            wi[k] = c * p - s * q;
                            wj[k] = s * p + c * q;
                        }
                    }
#pragma unroll
                    for(int k = 0; k < VM; ++k)
                        if(k * G < nv) {
                            vi[k * G] = c * u[k] - s * v[k];
                            vj[k * G] = s * u[k] + c * v[k];
                        }
                    const double g2 = 2.0 * s * c * ga;
                    double na = fma(c * c, al, fma(s * s, be, -g2)), nb = fma(s * s, al, fma(c * c, be, g2));
                    if(fmin(na, nb) < 1e-3 * fmin(al, be)) {  // cancellation (rare): sum afresh
                        na = norm2(a);
                        nb = norm2(b);
                    }
                    if(gl == 0) {
                        sig[a] = na;
                        sig[b] = nb;
                        rotated = 1;
                        if(sg * sg > SVD_NEAR * (sa * sb)) far = 1;
                    }
                }
            }
            if(grp != 0) a = a == n2 - 1 ? 1 : a + 1;
            b = b == n2 - 1 ? 1 : b + 1;
            __syncthreads();
        }
    };
    int sweep = 0;
    if(tid == 0) s_tiny = 0;
    if(nn > 1) {
        for(sweep = 0; sweep < MAX_SWEEPS; ++sweep) {
            __syncthreads();
            for(int j = grp; j < nn; j += ngroups) {
                const double s = norm2(j);
                if(gl == 0) {
                    sig[j] = s;
                    if(s > 0.0 && s < SVD_SMALL) s_tiny = 1;
                }
            }
            if(tid == 0) rotated = far = 0;
            __syncthreads();
            const bool tiny = __builtin_amdgcn_readfirstlane(s_tiny) != 0;
            if(tiny)
                steps(std::true_type{});
            else
                steps(std::false_type{});
            if(!rotated) break;
            // Every angle of this sweep was small, so the next one will most likely find all pairs
            // orthogonal: test them all at once, without the steps' barriers (same test).
            if(!far) {
                for(int j = grp; j < nn; j += ngroups) {
                    const double s = norm2(j);
                    if(gl == 0) sig[j] = s;
                }
                __syncthreads();
                if(tid == 0) rotated = 0;
                __syncthreads();
                for(int i = grp; i < nn; i += ngroups)
                    for(int d = 1; d <= nn / 2; ++d) {
                        const int j = i + d < nn ? i + d : i + d - nn;
                        const d2* wi = reinterpret_cast<const d2*>(W + i * ldw) + gl;
                        const d2* wj = reinterpret_cast<const d2*>(W + j * ldw) + gl;
                        double ga = 0.0;
                        for(int k = 0; k < nw; k += G) {
                            const d2 p = wi[k], q = wj[k];
                            ga = fma(p[0], q[0], ga);
                            ga = fma(p[1], q[1], ga);
                        }
                        ga = xh::lanes_sum<G>(ga);
                        double al = sig[i], be = sig[j];
                        const bool live = fmin(al, be) > SVD_ZERO;
                        if(tiny) scale_pair(al, be, ga);
                        if(gl == 0 && live && ga * ga > tol2 * (al * be)) rotated = 1;
                    }
                __syncthreads();
                if(!rotated) break;
            }
        }
    }
    if(sweep >= MAX_SWEEPS && tid == 0) atomicOr(fa.status, XH_ENOTCONV);
    // column norms
    for(int j = grp; j < nn; j += ngroups) {
        const double* wj = W + j * ldw;
        double s = 0;
        for(int r = gl; r < mm; r += G) s = fma(wj[r], wj[r], s);
        s = xh::lanes_sum<G>(s);
        if(gl == 0) sig[j] = sqrt(s);  // of the scaled block
    }
    __syncthreads();
    // descending order, ties broken by column index; NaN (from non-finite input) sorts last so
    // that the ranks stay a permutation of 0..nn-1 for any input
    for(int j = tid; j < nn; j += blockDim.x) {
        const double sj = nan_low(sig[j]);
        int rank = 0;
        for(int k = 0; k < nn; ++k) {
            const double sk = nan_low(sig[k]);
            rank += (sk > sj) || (sk == sj && k < j);
        }
        ord[rank] = j;
    }
    __syncthreads();
    for(int r = tid; r < nn; r += blockDim.x) fa.S[it.s_off + r] = ldexp(sig[ord[r]], ex);
    // U (m x nn) and Vt (nn x n): W / sigma on the long side, V on the other
    for(int r = grp; r < nn; r += ngroups) {
        const int c = ord[r];
        const double s = sig[c];
        for(int i = gl; i < mm; i += G) {
            const double v = s > 0.0 ? W[i + c * ldw] / s : 0.0;
            if(!tr)
                fa.U[it.u_off + i + int64_t(r) * m] = v;
            else
                fa.Vt[it.vt_off + r + int64_t(i) * nn] = v;
        }
        for(int i = gl; i < nn; i += G) {
            const double v = V[i + c * ldv];
            if(!tr)
                fa.Vt[it.vt_off + r + int64_t(i) * nn] = v;
            else
                fa.U[it.u_off + i + int64_t(r) * m] = v;
        }
    }
}

// Householder QR with Eigen's reflector convention (Eigen/src/Householder/Householder.h
// makeHouseholder: beta = -sign(c0) * ||x||, tau = (beta - c0) / beta, v = [1, x_tail / (c0 - beta)]).
// Q has `q_cols` columns (the tensor's middle dimension; columns beyond m are zero) and R has
// `q_cols` rows (rows beyond min(m, n) are zero).  Item fields: u_off -> Q, vt_off -> R,
// s_off -> q_cols (reused as an integer).
//
// Both kernels are a serial chain of min(m, n) reflectors, bound by the latency of one reflector
// and by LDS reads, not by flops.  A group of G lanes owns a column (column j: group j mod the
// number of groups) and its lane l the rows l, l + G, ..., so dot products end in a lane
// reduction inside the group.  The group that owns column k + 1 applies reflector k and at once
// makes reflector k + 1 from the values it still holds: one barrier per reflector.  Q is made
// column by column without barriers, from reflector min(c, kmax - 1) down, since the later ones
// leave e_c alone.
//
// k_qr (at most G * RM rows): NC columns per group live in registers from their load to their
// store, and only the reflectors V are in LDS (or, when they do not fit, in global memory), full
// columns with zeros above and a one on the diagonal, padded with zeros to G * RM rows, so that a
// step reads RM values per lane without conditions for all NC columns.  More than NC columns per
// group run in panels; a panel first takes all reflectors of the panels before it.
// k_qr_tall (any number of rows): the working copy is in LDS or global memory (qr_in_memory).
//
// k_qr takes all rows of a column through a reflector, the zeros of v included, and through identities
// (tau = 0).  An infinity or a NaN would be spread by that to rows that the reflector does not reach,
// so a block with one is left to qr_in_memory, which touches a reflector's own rows only.  (Both in
// one set of steps, or a second copy of them, made finite blocks 7 to 8 % slower by their registers;
// the look at every value costs 2 %.)
//
// One thread per trailing column, serial over its rows, took 2864 us for the 9 blocks (132 x 85
// the largest) of a U(1) matrix product tensor at bond 300; columns kept in LDS by such groups
// 550 us (48 LDS operations per column and reflector); k_qr takes 163 us.
constexpr int QR_THREADS = 1024;

__host__ __device__ inline int64_t qr_work_doubles(int64_t m, int64_t n, int64_t rows) { return (m < n ? m : n) * (rows + 1) + 1; }
__host__ __device__ inline int64_t qr_tall_work_doubles(int64_t m, int64_t n) { return m * n + (m < n ? m : n) + 1; }

// beta, tau and 1 / (c0 - beta) of the reflector of a column with diagonal entry c0 and squared
// norm `tail` below it; tau = 0 (H = I) when nothing is below
__device__ __forceinline__ void make_householder(double c0, double tail, double& beta, double& t, double& inv)
{
    beta = c0;
    t = 0.0;
    inv = 1.0;
    if(!(tail <= DBL_MIN)) {
        beta = sqrt(c0 * c0 + tail);
        if(c0 >= 0.0) beta = -beta;
        t = (beta - c0) / beta;
        inv = 1.0 / (c0 - beta);
    }
}

// Q and R of a block with its columns in memory: Wk, m x n of leading dimension ld, is the working copy,
// tau min(m, n) doubles.  Wk may be R itself (then ld is R's rows).
__device__ __forceinline__ void qr_in_memory(const FactorArgs& fa, const xh_factor_item& it, double* Wk, int64_t ld, double* tau)
{
    const int m = it.m, n = it.n;
    const int qc = static_cast<int>(it.s_off);
    constexpr int G = 64, NG = QR_THREADS / G;
    const int kmax = min(m, n);
    const int tid = threadIdx.x, lane = tid % G, grp = tid / G;
    for(int j = grp; j < n; j += NG)
        for(int r = lane; r < m; r += G) Wk[j * ld + r] = fa.A[it.a_off + int64_t(j) * m + r];
    auto reflector = [&](int k) {  // from column k, whose rows this group's lanes wrote themselves
        double* col = Wk + k * ld;
        double tail = 0.0, c0 = 0.0;
        for(int r = lane; r < m; r += G) {
            const double y = col[r];
            if(r > k) tail = fma(y, y, tail);
            if(r == k) c0 = y;
        }
        tail = xh::lanes_sum<G>(tail);
        c0 = xh::lanes_sum<G>(c0);
        double beta, t, inv;
        make_householder(c0, tail, beta, t, inv);
        for(int r = lane; r < m; r += G)
            if(r >= k) col[r] = r == k ? beta : col[r] * inv;
        if(lane == 0) tau[k] = t;
    };
    auto apply = [&](int k, double t, double* c) {  // c -= tau (v^T c) v, v = [1; column k below k]
        const double* col = Wk + k * ld;
        double w = 0.0;
        for(int r = lane; r < m; r += G)
            if(r >= k) w = fma(r == k ? 1.0 : col[r], c[r], w);
        w = xh::lanes_sum<G>(w) * t;
        for(int r = lane; r < m; r += G)
            if(r >= k) c[r] = fma(-w, r == k ? 1.0 : col[r], c[r]);
    };
    if(grp == 0) reflector(0);
    for(int k = 0; k < kmax; ++k) {
        __syncthreads();  // reflector k is there
        const double t = tau[k];
        const int first = k + 1;
        for(int j = first + ((grp - first) % NG + NG) % NG; j < n; j += NG) {
            if(t != 0.0) apply(k, t, Wk + j * ld);
            if(j == first && first < kmax) reflector(first);
        }
    }
    __syncthreads();
    for(int c = grp; c < qc; c += NG) {
        double* qcol = fa.U + it.u_off + int64_t(c) * m;
        for(int r = lane; r < m; r += G) qcol[r] = (r == c) ? 1.0 : 0.0;
        if(c < m)
            for(int k = min(c, kmax - 1); k >= 0; --k)
                if(tau[k] != 0.0) apply(k, tau[k], qcol);
    }
    __syncthreads();
    // R: qc x n, upper triangle of the working copy (rows beyond min(m, n) are zero)
    for(int64_t e = tid; e < int64_t(qc) * n; e += QR_THREADS) {
        const int r = static_cast<int>(e % qc), c = static_cast<int>(e / qc);
        fa.Vt[it.vt_off + e] = (r < m && r <= c) ? Wk[r + c * ld] : 0.0;
    }
}

template <bool LDS, int G, int RM, int NC>
__global__ __launch_bounds__(QR_THREADS) void k_qr(FactorArgs fa)
{
    extern __shared__ double smem[];
    const xh_factor_item it = fa.items[blockIdx.x];
    const int m = it.m, n = it.n;
    const int qc = static_cast<int>(it.s_off);
    if(m == 0 || n == 0) return;
    constexpr int NG = QR_THREADS / G, LD = G * RM, PC = NG * NC;
    const int kmax = min(m, n);
    double* V = work_base<LDS>(smem, fa);  // reflectors: kmax columns of LD rows
    double* tau = V + int64_t(LD) * kmax;  // kmax
    const int lane = threadIdx.x % G, grp = threadIdx.x / G;
    double x[NC][RM], v[RM];
    auto load_panel = [&](int p0) {
#pragma unroll
        for(int q = 0; q < NC; ++q) {
            const int j = p0 + grp + q * NG;
#pragma unroll
            for(int i = 0; i < RM; ++i) {
                const int r = lane + i * G;
                x[q][i] = j < n && r < m ? fa.A[it.a_off + int64_t(j) * m + r] : 0.0;
            }
        }
    };
    load_panel(0);
    bool ok = true;
#pragma unroll
    for(int q = 0; q < NC; ++q)
#pragma unroll
        for(int i = 0; i < RM; ++i) ok = ok && isfinite(x[q][i]);
    for(int64_t e = int64_t(PC) * m + threadIdx.x; e < int64_t(m) * n; e += QR_THREADS) ok = ok && isfinite(fa.A[it.a_off + e]);
    if(!__syncthreads_and(ok)) {
        if(n <= m)
            qr_in_memory(fa, it, V, m, V + m * n);  // (m + 1) n doubles, as k_qr's work area has
        else
            qr_in_memory(fa, it, fa.Vt + it.vt_off, qc, tau);
        return;
    }
    auto load_v = [&](int k) {
        const double* col = V + int64_t(k) * LD + lane;
#pragma unroll
        for(int i = 0; i < RM; ++i) v[i] = col[i * G];
    };
    // x -= tau (v^T x) v for the group's columns first + q NG > after (those up to `after` are finished)
    auto apply = [&](double t, int first, int after) {
        double w[NC];
#pragma unroll
        for(int q = 0; q < NC; ++q) {
            w[q] = 0.0;
#pragma unroll
            for(int i = 0; i < RM; ++i) w[q] = fma(v[i], x[q][i], w[q]);
        }
#pragma unroll
        for(int q = 0; q < NC; ++q) w[q] = xh::lanes_sum<G>(w[q]) * t;
#pragma unroll
        for(int q = 0; q < NC; ++q)
            if(first + q * NG > after)
#pragma unroll
                for(int i = 0; i < RM; ++i) x[q][i] = fma(-w[q], v[i], x[q][i]);
    };
    // makes reflector k from the column xc, leaving beta on xc's diagonal
    auto reflector = [&](int k, double (&xc)[RM]) {
        double tail = 0.0, c0 = 0.0;
        int d = k - lane;  // row lane + i G lies below the diagonal for i G > d
#pragma unroll
        for(int i = 0; i < RM; ++i) {
            tail = fma(i * G > d ? xc[i] : 0.0, xc[i], tail);
            c0 = i * G == d ? xc[i] : c0;
        }
        tail = xh::lanes_sum<G>(tail);
        c0 = xh::lanes_sum<G>(c0);
        double beta, t, inv;
        make_householder(c0, tail, beta, t, inv);
        asm("" : "+v"(d));  // compare again: 2 RM lane masks kept over the square root would spill
        double* col = V + int64_t(k) * LD + lane;
#pragma unroll
        for(int i = 0; i < RM; ++i) {
            col[i * G] = i * G > d ? xc[i] * inv : (i * G == d ? 1.0 : 0.0);
            xc[i] = i * G == d ? beta : xc[i];
        }
        if(lane == 0) tau[k] = t;
    };
    for(int p0 = 0; p0 < n; p0 += PC) {
        if(p0 > 0) load_panel(p0);
        for(int k = 0; k < min(p0, kmax); ++k) {
            load_v(k);
            apply(tau[k], p0 + grp, -1);
        }
        const int p1 = min(p0 + PC, kmax);
        if(grp == 0 && p0 < kmax) reflector(p0, x[0]);
        for(int k = p0; k < p1; ++k) {
            __syncthreads();  // reflector k is there
            const double t = tau[k];
            if(k + 1 < min(p0 + PC, n)) {
                load_v(k);
                apply(t, p0 + grp, k);
                if(k + 1 < p1) {
#pragma unroll
                    for(int q = 0; q < NC; ++q)
                        if(p0 + grp + q * NG == k + 1) reflector(k + 1, x[q]);
                }
            }
        }
        // R: qc x n, the rows up to the diagonal (rows beyond min(m, n) are zero)
#pragma unroll
        for(int q = 0; q < NC; ++q) {
            const int j = p0 + grp + q * NG;
            if(j >= n) continue;
            double* out = fa.Vt + it.vt_off + int64_t(j) * qc;
#pragma unroll
            for(int i = 0; i < RM; ++i) {
                const int r = lane + i * G;
                if(r < qc) out[r] = r < m && r <= j ? x[q][i] : 0.0;
            }
            for(int r = lane + LD; r < qc; r += G) out[r] = 0.0;
        }
    }
    __syncthreads();
    // Q columns 0..qc-1: Q e_c = H_0 H_1 ... H_{kmax-1} e_c (zero for c >= m)
    for(int c0 = 0; c0 < qc; c0 += PC) {
#pragma unroll
        for(int q = 0; q < NC; ++q)
#pragma unroll
            for(int i = 0; i < RM; ++i) x[q][i] = lane + i * G == c0 + grp + q * NG ? 1.0 : 0.0;
        // a column beyond m holds its one outside the block (or nowhere): no reflector reaches it
        for(int k = min(c0 + grp + (NC - 1) * NG, kmax - 1); k >= 0; --k) {
            load_v(k);
            apply(tau[k], c0 + grp, -1);
        }
#pragma unroll
        for(int q = 0; q < NC; ++q) {
            const int c = c0 + grp + q * NG;
            if(c >= qc) continue;
            double* out = fa.U + it.u_off + int64_t(c) * m;
#pragma unroll
            for(int i = 0; i < RM; ++i) {
                const int r = lane + i * G;
                if(r < m) out[r] = x[q][i];
            }
        }
    }
}

template <bool LDS>
__global__ __launch_bounds__(QR_THREADS) void k_qr_tall(FactorArgs fa)
{
    extern __shared__ double smem[];
    const xh_factor_item it = fa.items[blockIdx.x];
    if(it.m == 0 || it.n == 0) return;
    double* Wk = work_base<LDS>(smem, fa);
    qr_in_memory(fa, it, Wk, it.m, Wk + int64_t(it.m) * it.n);
}

// Inverse of the upper Cholesky factor of a Gram block G + shift * trace(G) * I (the building
// block of shifted CholeskyQR, Fukaya, Kannan, Nakatsukasa, Yamamoto & Yanagisawa, SIAM J. Sci.
// Comput. 42 (2020) A477).  Item: a_off -> G (n x n), u_off -> X = R^-1 (n x n, upper), s_off ->
// index of the item's relative shift in fa.S.  A pivot that does not exceed 64 eps times its
// column's original diagonal marks a numerically dependent column: its row and column of X are
// zero, so Y X has a zero column there.
//
// One workgroup per block, in 16 x 16 tiles on the matrix cores.  The time is the serial chain of
// ceil(n / 16) diagonal tiles and of the barriers between them, not the n^3 / 3 flops (which one CU
// does in a few microseconds at n = 74), so a panel has two barriers:
//   solve     R_pj = R_pp^-T A_pj for the tiles right of the diagonal, one per wave;
//   update    A_ij -= R_pi^T R_pj; wave 0 takes the next diagonal tile first and factorises it
//             while the other waves update the rest.
// Then X R = I by block columns J: S = sum_l X_il R_lJ, X_iJ = -S R_JJ^-1, one tile row per wave.
// Multiplying by the explicit inverse of a diagonal tile is followed by one step of refinement
// with the tile itself, which gives back the stability of substitution.
//
// The tiles (i, j), i <= j, are packed by columns in LDS (n <= 192) or in a global working copy.
// Element (r, c) of a tile is at 16 r + (c ^ r), so that a wave reads and writes rows, columns and
// transposes without bank conflicts, and so that one set of four offsets per lane serves the A
// operand R^T, the B operand and the accumulators of v_mfma_f64_16x16x4f64: an accumulator is the
// B operand of the next product as it is.  A factorised diagonal tile holds R above and X^T = R^-T
// on and below its diagonal, with R's diagonal in rdiag; X is kept transposed, in LDS in the place
// of R's block column once that is used up, beyond LDS in the output itself.
// (One barrier per pivot and 16 lanes per dot product of X: 134 us at n = 74, 673 us at n = 190;
// these tiles 30 and 98 us, 2286 -> 227 us at n = 250.)
constexpr int CI_THREADS = 1024;
constexpr int CI_MAX_N = 40000;

__host__ __device__ inline int64_t chol_tiles(int64_t n) { return ((n + 15) / 16) * ((n + 15) / 16 + 1) / 2; }
__host__ __device__ inline int64_t chol_work_doubles(int64_t n) { return chol_tiles(n) * 256 + 2 * ((n + 15) / 16) * 16; }

typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double lane_value(double x, int lane)
{
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), lane), hi = __builtin_amdgcn_readlane(__double2hiint(x), lane);
    return __hiloint2double(hi, lo);
}

template <bool LDS>
__global__ __launch_bounds__(CI_THREADS) void k_chol_inv(FactorArgs fa)
{
    extern __shared__ __attribute__((aligned(16))) double smem[];
    __shared__ double s_part[CI_THREADS / 64];
    const xh_factor_item it = fa.items[blockIdx.x];
    const int n = it.n;
    if(n == 0) return;
    const int nt = (n + 15) / 16;
    const int64_t ntri = chol_tiles(n);
    double* W = work_base<LDS>(smem, fa);
    double* rd = W + ntri * 256;                     // shifted original diagonal (dependence threshold)
    double* rdiag = rd + nt * 16;                    // diagonal of R
    constexpr int NW = CI_THREADS / 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, row0 = lane >> 4;     // element (row0 + 4 q, col) of a tile for q = 0 .. 3
    int o[4], ot[4];                                 // its offset, and that of its mirror image
#pragma unroll
    for(int q = 0; q < 4; ++q) {
        const int r = row0 + 4 * q;
        o[q] = r * 16 + (col ^ r);
        ot[q] = col * 16 + (r ^ col);
    }
    auto tri = [](int i, int j) { return (int64_t(j) * (j + 1) / 2 + i) * 256; };
    auto tile = [&](int i, int j) { return W + tri(i, j); };
    // the identity continues G beyond n
    const double* G = fa.A + it.a_off;
    double tr = 0.0;
    for(int j = 0; j < nt; ++j)
        for(int i = (wave + NW - j % NW) % NW; i <= j; i += NW) {
            double* t = tile(i, j);
#pragma unroll
            for(int q = 0; q < 4; ++q) {  // lanes along a column of G
                const int gi = 16 * i + col, gj = 16 * j + row0 + 4 * q;
                const double v = gj < n && gi <= gj ? G[gi + int64_t(gj) * n] : (gi == gj ? 1.0 : 0.0);
                t[ot[q]] = v;
                if(gi == gj && gj < n) tr += v;
            }
        }
    for(int k = 32; k > 0; k >>= 1) tr += __shfl_xor(tr, k);
    if(lane == 0) s_part[wave] = tr;
    __syncthreads();
    {
        double t = 0.0;
        for(int w = 0; w < NW; ++w) t += s_part[w];
        const double shift = fa.S[it.s_off] * t;
        for(int k = threadIdx.x; k < 16 * nt; k += CI_THREADS) {
            double* d = tile(k / 16, k / 16) + (k & 15) * 16;  // (r, r) is at 16 r + 0
            if(k < n) *d += shift;
            rd[k] = *d;
        }
    }
    __syncthreads();

    // Cholesky factor and inverse of a diagonal tile by one wave: lane j holds column j of the
    // tile, lane 16 + j column j of the identity, and both take the same row operations
    auto factor = [&](int p) {
        double* t = tile(p, p);
        double x[16];
#pragma unroll
        for(int i = 0; i < 16; ++i) x[i] = lane < 16 ? t[i * 16 + (col ^ i)] : lane < 32 && i == col ? 1.0 : 0.0;
        const double thr = 64.0 * DBL_EPSILON * rd[16 * p + col];
        double diag = 0.0;
#pragma unroll
        for(int k = 0; k < 16; ++k) {
            const double d = lane_value(x[k], k);
            const bool ok = d > lane_value(thr, k) && d <= DBL_MAX;
            // 1 / sqrt(d): the hardware estimate and its second-order correction
            const double y = __builtin_amdgcn_rsq(ok ? d : 1.0);
            const double e = fma(-d * y, y, 1.0);
            const double s = ok ? fma(y * e, fma(e, 0.375, 0.5), y) : 0.0;
            x[k] *= s;
            if(lane == k) diag = ok ? x[k] : 0.0;  // a rejected pivot may be infinite or NaN
#pragma unroll
            for(int i = k + 1; i < 16; ++i) x[i] = fma(-lane_value(x[k], i), x[k], x[i]);
        }
        if(lane < 32) {
#pragma unroll
            for(int i = 0; i < 16; ++i)
                if(lane < 16 ? i < col : i >= col) t[i * 16 + (col ^ i)] = x[i];
            if(lane < 16) rdiag[16 * p + col] = diag;
        }
    };
    // a diagonal tile as A operands: X_pp^T and R_pp^T
    auto load_diag = [&](int p, double (&x)[4], double (&r)[4]) {
        const double* t = tile(p, p);
        const double dg = rdiag[16 * p + col];
#pragma unroll
        for(int q = 0; q < 4; ++q) {
            const int k = row0 + 4 * q;
            const double a = t[ot[q]], b = t[o[q]];
            x[q] = k <= col ? a : 0.0;
            r[q] = k < col ? b : (k == col ? dg : 0.0);
        }
    };
    auto mfma = [](double a, double b, d4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); };
    // sign * X_pp^T c with one refinement against R_pp^T
    auto solve = [&](const double (&x)[4], const double (&r)[4], const d4 c, double sign) {
        d4 y = {0, 0, 0, 0};
#pragma unroll
        for(int q = 0; q < 4; ++q) y = mfma(x[q], c[q], y);
        d4 res = c;
#pragma unroll
        for(int q = 0; q < 4; ++q) res = mfma(-r[q], y[q], res);
#pragma unroll
        for(int q = 0; q < 4; ++q) y = mfma(x[q], res[q], y);
        return sign * y;
    };
    auto update = [&](int p, int i, int j) {
        const double *a = tile(p, i), *b = tile(p, j);
        double* t = tile(i, j);
        d4 c;
        double u[4], v[4];
#pragma unroll
        for(int q = 0; q < 4; ++q) {
            c[q] = t[o[q]];
            u[q] = a[o[q]];
            v[q] = b[o[q]];
        }
#pragma unroll
        for(int q = 0; q < 4; ++q) c = mfma(-u[q], v[q], c);
#pragma unroll
        for(int q = 0; q < 4; ++q) t[o[q]] = c[q];
    };
    double* X = fa.U + it.u_off;
    // element q of this lane of tile (i, j), i < j, of X^T outside LDS: rows and columns below n unless j is the
    // last, which no later column reads
    auto out_at = [&](int i, int j, int q) -> double* { return X + (16 * i + col) + int64_t(16 * j + row0 + 4 * q) * n; };
    if(wave == 0) factor(0);
    __syncthreads();
    for(int p = 0; p + 1 < nt; ++p) {
        if(p + 1 + wave < nt) {
            double x[4], r[4];
            load_diag(p, x, r);
            for(int j = p + 1 + wave; j < nt; j += NW) {
                double* t = tile(p, j);
                d4 c;
#pragma unroll
                for(int q = 0; q < 4; ++q) c[q] = t[o[q]];
                c = solve(x, r, c, 1.0);
#pragma unroll
                for(int q = 0; q < 4; ++q) t[o[q]] = c[q];
            }
        }
        __syncthreads();
        if(wave == 0) {
            update(p, p + 1, p + 1);
            // factor's lanes read elements that other lanes of this wave have just stored
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            factor(p + 1);
        } else {
            int left = wave;  // tiles of the trailing triangle by columns; number 0 is wave 0's
            for(int j = p + 1; j < nt; ++j) {
                for(; left <= j - p - 1; left += NW - 1) update(p, p + 1 + left, j);
                left -= j - p;
            }
        }
        __syncthreads();
    }
    for(int J = 1; J < nt; ++J) {
        d4 c = {0, 0, 0, 0};
        if(wave < J) {
            double x[4], r[4];
            load_diag(J, x, r);
            for(int i = wave; i < J; i += NW) {
                c = d4{0, 0, 0, 0};  // S^T = sum_l R_lJ^T X_il^T
                for(int l = i; l < J; ++l) {
                    const double *a = tile(l, J), *b = tile(i, l);  // R's diagonal tile holds X^T's
                    double u[4], v[4];
#pragma unroll
                    for(int q = 0; q < 4; ++q) {
                        u[q] = a[o[q]];
                        v[q] = LDS || l == i ? b[o[q]] : *out_at(i, l, q);
                    }
#pragma unroll
                    for(int q = 0; q < 4; ++q) c = mfma(u[q], l > i || row0 + 4 * q >= col ? v[q] : 0.0, c);
                }
                c = solve(x, r, c, -1.0);
                if constexpr(!LDS) {
#pragma unroll
                    for(int q = 0; q < 4; ++q)
                        if(16 * J + row0 + 4 * q < n) *out_at(i, J, q) = c[q];
                }
            }
        }
        __syncthreads();
        if constexpr(LDS) {  // at most NW tile rows: one per wave
            if(wave < J) {
#pragma unroll
                for(int q = 0; q < 4; ++q) tile(wave, J)[o[q]] = c[q];
            }
            __syncthreads();
        }
    }
    // X to the output, zeros below its diagonal
    for(int t = wave; t < nt * nt; t += NW) {
        const int i = t % nt, j = t / nt;
        if(!LDS && i < j) continue;  // there already
        const double* b = i <= j ? tile(i, j) : nullptr;
#pragma unroll
        for(int q = 0; q < 4; ++q) {
            const int gi = 16 * i + col, gj = 16 * j + row0 + 4 * q;
            if(gi < n && gj < n) X[gi + int64_t(gj) * n] = gi <= gj ? b[o[q]] : 0.0;
        }
    }
}

// Symmetric eigen-decomposition by parallel cyclic Jacobi.  Item: a_off (n x n), s_off -> eigenvalues,
// u_off -> eigenvectors (columns), ascending order.
template <bool LDS>
__global__ __launch_bounds__(F_THREADS) void k_eigh(FactorArgs fa)
{
    extern __shared__ double smem[];
    __shared__ int rotated;
    const xh_factor_item it = fa.items[blockIdx.x];
    const int n = it.m;
    if(n == 0) return;
    double* Am = work_base<LDS>(smem, fa);
    double* V = Am + int64_t(n) * n;
    double* cs = V + int64_t(n) * n;  // per pair: c, s  (n entries)
    int* pr = reinterpret_cast<int*>(cs + n + 1);  // per pair: p, q (n ints)
    double* ev = cs;  // reused after the sweeps
    int* ord = pr;
    const int tid = threadIdx.x;
    for(int64_t e = tid; e < int64_t(n) * n; e += F_THREADS) {
        // symmetrise from the lower triangle as SelfAdjointEigenSolver reads it
        const int i = static_cast<int>(e % n), j = static_cast<int>(e / n);
        Am[e] = (i >= j) ? fa.A[it.a_off + e] : fa.A[it.a_off + j + int64_t(i) * n];
        V[e] = (i == j) ? 1.0 : 0.0;
    }
    __syncthreads();
    const int n2 = n + (n & 1), npairs = n2 / 2;
    int sweep = 0;
    if(n > 1) {
        for(sweep = 0; sweep < MAX_SWEEPS; ++sweep) {
            if(tid == 0) rotated = 0;
            __syncthreads();
            for(int step = 0; step < n2 - 1; ++step) {
                for(int p = tid; p < npairs; p += F_THREADS) {
                    int i = rr_player(p, step, n2), j = rr_player(n2 - 1 - p, step, n2);
                    if(i > j) {
                        int t = i;
                        i = j;
                        j = t;
                    }
                    double c = 1.0, s = 0.0;
                    if(j < n) {
                        const double apq = Am[i + int64_t(j) * n];
                        const double app = Am[i + int64_t(i) * n], aqq = Am[j + int64_t(j) * n];
                        if(fabs(apq) > DBL_EPSILON * sqrt(fabs(app) * fabs(aqq)) && fabs(apq) > 1e-300) {
                            const double theta = (aqq - app) / (2.0 * apq);
                            const double t = copysign(1.0, theta) / (fabs(theta) + sqrt(theta * theta + 1.0));
                            c = 1.0 / sqrt(t * t + 1.0);
                            s = t * c;
                            rotated = 1;
                        }
                    } else {
                        i = -1;
                    }
                    cs[2 * p] = c;
                    cs[2 * p + 1] = s;
                    pr[2 * p] = i;
                    pr[2 * p + 1] = j;
                }
                __syncthreads();
                // columns: A <- A J, V <- V J
                for(int64_t e = tid; e < int64_t(npairs) * n; e += F_THREADS) {
                    const int p = static_cast<int>(e / n), r = static_cast<int>(e % n);
                    const int i = pr[2 * p], j = pr[2 * p + 1];
                    if(i < 0) continue;
                    const double c = cs[2 * p], s = cs[2 * p + 1];
                    if(s == 0.0) continue;
                    double x = Am[r + int64_t(i) * n], y = Am[r + int64_t(j) * n];
                    Am[r + int64_t(i) * n] = c * x - s * y;
                    Am[r + int64_t(j) * n] = s * x + c * y;
                    x = V[r + int64_t(i) * n];
                    y = V[r + int64_t(j) * n];
                    V[r + int64_t(i) * n] = c * x - s * y;
                    V[r + int64_t(j) * n] = s * x + c * y;
                }
                __syncthreads();
                // rows: A <- J^T A
                for(int64_t e = tid; e < int64_t(npairs) * n; e += F_THREADS) {
                    const int p = static_cast<int>(e / n), col = static_cast<int>(e % n);
                    const int i = pr[2 * p], j = pr[2 * p + 1];
                    if(i < 0) continue;
                    const double c = cs[2 * p], s = cs[2 * p + 1];
                    if(s == 0.0) continue;
                    const double x = Am[i + int64_t(col) * n], y = Am[j + int64_t(col) * n];
                    Am[i + int64_t(col) * n] = c * x - s * y;
                    Am[j + int64_t(col) * n] = s * x + c * y;
                }
                __syncthreads();
            }
            const int any = rotated;
            __syncthreads();
            if(!any) break;
        }
    }
    if(sweep >= MAX_SWEEPS && tid == 0) atomicExch(fa.status, XH_ENOTCONV);
    for(int j = tid; j < n; j += F_THREADS) ev[j] = Am[j + int64_t(j) * n];
    __syncthreads();
    for(int j = tid; j < n; j += F_THREADS) {
        const double vj = nan_high(ev[j]);
        int rank = 0;
        for(int k = 0; k < n; ++k) rank += (nan_high(ev[k]) < vj) || (nan_high(ev[k]) == vj && k < j);
        ord[rank] = j;
    }
    __syncthreads();
    for(int r = tid; r < n; r += F_THREADS) fa.S[it.s_off + r] = ev[ord[r]];
    for(int64_t e = tid; e < int64_t(n) * n; e += F_THREADS) {
        const int i = static_cast<int>(e % n), r = static_cast<int>(e / n);
        fa.U[it.u_off + e] = V[i + int64_t(ord[r]) * n];
    }
}

struct Launch {
    std::vector<xh_factor_item> lds_items, glb_items;
    int64_t lds_bytes = 0, glb_stride = 0;
};

size_t lds_budget(xh_ctx* ctx)
{
    static size_t cached = 0;
    if(cached == 0) {
        hipDeviceProp_t prop;
        check(hipGetDeviceProperties(&prop, ctx->device), "hipGetDeviceProperties");
        cached = prop.sharedMemPerBlock;
        if(cached > 160 * 1024) cached = 160 * 1024;
    }
    return cached - 1024;  // leave room for the static shared variables
}

template <typename Need>
void run_factor(xh_ctx* ctx, void (*kern_lds)(FactorArgs), void (*kern_global)(FactorArgs), const std::vector<xh_factor_item>& items, Need need_doubles,
                const double* A, double* U, double* S, double* Vt)
{
    const size_t budget = lds_budget(ctx);
    std::vector<xh_factor_item> small, big;
    int64_t small_max = 0, big_max = 0;
    for(const auto& it : items) {
        if(it.m < 0 || it.n < 0) throw xh::Error(XH_EINVAL, "factor: negative extent");
        if(it.m == 0 || it.n == 0) continue;
        const int64_t nd = need_doubles(it);
        if(size_t(nd) * sizeof(double) <= budget) {
            small.push_back(it);
            small_max = std::max(small_max, nd);
        } else {
            big.push_back(it);
            big_max = std::max(big_max, nd);
        }
    }
    int* d_status = nullptr;
    check(xh::dmalloc(ctx, reinterpret_cast<void**>(&d_status), sizeof(int)), "hipMallocAsync");
    check(hipMemsetAsync(d_status, 0, sizeof(int), ctx->stream), "hipMemsetAsync");
    auto go = [&](const std::vector<xh_factor_item>& v, bool lds, int64_t maxd) {
        if(v.empty()) return;
        xh_factor_item* d_items = xh::dev_upload(ctx, v);
        double* scratch = nullptr;
        if(!lds) check(xh::dmalloc(ctx, reinterpret_cast<void**>(&scratch), size_t(maxd) * v.size() * sizeof(double)), "hipMallocAsync");
        FactorArgs fa{d_items, A, U, S, Vt, scratch, maxd, lds ? 1 : 0, d_status};
        auto* kern = lds ? kern_lds : kern_global;
        const size_t shmem = lds ? size_t(maxd) * sizeof(double) : 0;
        if(lds && shmem > 64 * 1024) check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, int(shmem)), "hipFuncSetAttribute");
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(v.size())), dim3(F_THREADS), shmem, ctx->stream, fa);
        xh::launch_check("factor kernel");
        check(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
        xh::dev_free(ctx, d_items);
        xh::dev_free(ctx, scratch);
    };
    go(small, true, small_max);
    go(big, false, big_max);
    int status = 0;
    check(hipMemcpyAsync(&status, d_status, sizeof(int), hipMemcpyDeviceToHost, ctx->stream), "hipMemcpyAsync");
    check(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
    xh::dev_free(ctx, d_status);
    if(status != 0) throw xh::Error(XH_ENOTCONV, "Jacobi iteration did not converge within the sweep limit");
}

}  // namespace

// Rows from which a call's pairs of up to 32 columns are worked on by 64 lanes instead of 16, which
// then read a column four times as fast: 2000 x 8 429 us with 16 lanes, 165 with 64 (296 with three
// reductions through ds_bpermute and IEEE divisions), 300 x 32 456 and 423, 20000 x 1 418 and 126.  Below,
// the longer reduction and the fewer blocks per CU cost more: 140 x 32 320 and 372, 300 blocks of
// 200 x 30 481 and 689.
constexpr int SVD_TALL = 257;

namespace {
// The single-workgroup Jacobi kernel on blocks whose working set fits LDS: one launch, in the
// variant of the tallest and widest block.  The singular values are read back by every caller, so
// the convergence status waits with them.
void small_svd(xh_ctx* ctx, const std::vector<xh_factor_item>& v, const double* A, double* U, double* S, double* Vt)
{
    if(v.empty()) return;
    int mm = 0, nn = 0;
    int64_t maxd = 0;
    for(const auto& it : v) {
        const int a = std::max(it.m, it.n), b = std::min(it.m, it.n);
        mm = std::max(mm, a);
        nn = std::max(nn, b);
        maxd = std::max(maxd, svd_work_doubles(a, b));
    }
    void (*kern)(FactorArgs) = nullptr;
    int G = 16;  // lanes per pair of columns
    if(nn <= 32 && mm >= SVD_TALL) {
        kern = k_svd_jacobi<0, 1, 64>;
        G = 64;
    } else if(nn <= 32)
        kern = mm <= 32 ? k_svd_jacobi<1, 1> : mm <= 64 ? k_svd_jacobi<2, 1> : mm <= 128 ? k_svd_jacobi<4, 1> : k_svd_jacobi<0, 1>;
    else if(nn <= 64)
        kern = mm <= 64 ? k_svd_jacobi<2, 2> : mm <= 128 ? k_svd_jacobi<4, 2> : k_svd_jacobi<0, 2>;
    else
        kern = mm <= 128 ? k_svd_jacobi<4, 4> : k_svd_jacobi<0, 4>;
    static_assert(BJ_MIN_COLS_ALONE <= 128, "k_svd_jacobi's V rows");
    const int npairs = (nn + 1) / 2;
    const int threads = std::min(SVD_THREADS, (npairs * G + 63) / 64 * 64);
    int* d_status = nullptr;
    check(xh::dmalloc(ctx, reinterpret_cast<void**>(&d_status), sizeof(int)), "hipMallocAsync");
    check(hipMemsetAsync(d_status, 0, sizeof(int), ctx->stream), "hipMemsetAsync");
    xh_factor_item* d_items = xh::dev_upload(ctx, v);
    FactorArgs fa{d_items, A, U, S, Vt, nullptr, 0, 1, d_status};
    const size_t shmem = size_t(maxd) * sizeof(double);
    if(shmem > 64 * 1024)
        check(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, int(shmem)), "hipFuncSetAttribute");
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(v.size())), dim3(threads), shmem, ctx->stream, fa);
    xh::launch_check("k_svd_jacobi");
    int status = 0;
    check(hipMemcpyAsync(&status, d_status, sizeof(int), hipMemcpyDeviceToHost, ctx->stream), "hipMemcpyAsync");
    check(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
    xh::dev_free(ctx, d_items);
    xh::dev_free(ctx, d_status);
    static_assert((XH_EINVAL & XH_ENOTCONV) == 0, "status bits");
    if(status & XH_EINVAL) throw xh::Error(XH_EINVAL, "block SVD: non-finite input block");
    if(status != 0) throw xh::Error(XH_ENOTCONV, "Jacobi iteration did not converge within the sweep limit");
}
}  // namespace

extern "C" int xh_block_svd(xh_ctx* ctx, const xh_factor_item* items, int64_t nitems, const double* A, double* U, double* S, double* Vt)
{
    return guard(ctx, [&] {
        // small blocks: one workgroup each, in LDS; larger ones: block Jacobi over grouped GEMMs
        std::vector<xh_factor_item> v, big;
        const size_t budget = lds_budget(ctx);
        for(int64_t i = 0; i < nitems; ++i) {
            const xh_factor_item& it = items[i];
            if(it.m <= 0 || it.n <= 0) continue;
            const int mn = std::min(it.m, it.n), mx = std::max(it.m, it.n);
            if(mn > BJ_MIN_COLS_ALONE || size_t(svd_work_doubles(mx, mn)) * sizeof(double) > budget)
                big.push_back(it);
            else
                v.push_back(it);
        }
        if(!big.empty()) {
            auto wide = [](const xh_factor_item& it) { return std::min(it.m, it.n) > BJ_MIN_COLS; };
            std::copy_if(v.begin(), v.end(), std::back_inserter(big), wide);
            v.erase(std::remove_if(v.begin(), v.end(), wide), v.end());
        }
        block_jacobi_svd(ctx, big, A, U, S, Vt);
        small_svd(ctx, v, A, U, S, Vt);
    });
}

extern "C" int xh_block_qr(xh_ctx* ctx, const xh_factor_item* items, int64_t nitems, const double* A, double* Q, double* R)
{
    // asynchronous: there is no status to read back, so no host synchronisation
    return guard(ctx, [&] {
        const size_t budget = lds_budget(ctx);
        // a kernel per range of rows, the narrowest that holds a block; its reflectors in LDS where
        // they fit; from 1025 rows the kernel with a working copy
        struct Class {
            void (*kern)(FactorArgs);
            int rows;  // most rows; 0: any
            bool lds;
            std::vector<xh_factor_item> v;
            int64_t maxd;
        };
        Class cls[] = {{k_qr<true, 16, 4, 4>, 64, true, {}, 0},   {k_qr<true, 16, 8, 2>, 128, true, {}, 0},    {k_qr<true, 16, 12, 2>, 192, true, {}, 0},
                       {k_qr<true, 16, 16, 1>, 256, true, {}, 0}, {k_qr<true, 64, 16, 1>, 1024, true, {}, 0},  {k_qr<false, 16, 16, 1>, 256, false, {}, 0},
                       {k_qr<false, 64, 16, 1>, 1024, false, {}, 0}, {k_qr_tall<true>, 0, true, {}, 0},     {k_qr_tall<false>, 0, false, {}, 0}};
        auto need = [&](const Class& c, const xh_factor_item& it) {
            return c.rows ? qr_work_doubles(it.m, it.n, c.rows) : qr_tall_work_doubles(it.m, it.n);
        };
        auto fits = [&](const Class& c, const xh_factor_item& it) {
            return (!c.rows || it.m <= c.rows) && (!c.lds || size_t(need(c, it)) * sizeof(double) <= budget);
        };
        for(int64_t i = 0; i < nitems; ++i) {
            const xh_factor_item& it = items[i];
            if(it.m < 0 || it.n < 0) throw xh::Error(XH_EINVAL, "factor: negative extent");
            if(it.m == 0 || it.n == 0) continue;
            for(Class& c : cls)
                if(fits(c, it)) {
                    c.v.push_back(it);
                    break;
                }
        }
        // one launch for the 16-lane classes where the widest of them can hold every block: a few
        // blocks run beside each other on different CUs, and the largest sets the time either way
        // (9 blocks of 31 to 132 rows: 174 + 109 + 21 us in three launches)
        Class* wide = nullptr;
        for(int c = 0; c < 4; ++c)
            if(!cls[c].v.empty()) wide = &cls[c];
        for(int c = 0; c < 4; ++c) {
            if(&cls[c] == wide || cls[c].v.empty()) continue;
            if(!std::all_of(cls[c].v.begin(), cls[c].v.end(), [&](const xh_factor_item& it) { return fits(*wide, it); })) continue;
            wide->v.insert(wide->v.end(), cls[c].v.begin(), cls[c].v.end());
            cls[c].v.clear();
        }
        for(Class& c : cls)
            for(const auto& it : c.v) c.maxd = std::max(c.maxd, need(c, it));
        for(Class& c : cls) {
            if(c.v.empty()) continue;
            xh_factor_item* d_items = xh::dev_upload(ctx, c.v);
            double* scratch = nullptr;
            if(!c.lds) check(xh::dmalloc(ctx, reinterpret_cast<void**>(&scratch), size_t(c.maxd) * c.v.size() * sizeof(double)), "hipMallocAsync");
            FactorArgs fa{d_items, A, Q, nullptr, R, scratch, c.maxd, c.lds ? 1 : 0, nullptr};
            const size_t shmem = c.lds ? size_t(c.maxd) * sizeof(double) : 0;
            if(shmem > 64 * 1024)
                check(hipFuncSetAttribute(reinterpret_cast<const void*>(c.kern), hipFuncAttributeMaxDynamicSharedMemorySize, int(shmem)), "hipFuncSetAttribute");
            hipLaunchKernelGGL(c.kern, dim3(static_cast<unsigned>(c.v.size())), dim3(QR_THREADS), shmem, ctx->stream, fa);
            xh::launch_check("k_qr");
            xh::dev_free(ctx, d_items);
            xh::dev_free(ctx, scratch);
        }
    });
}

extern "C" int xh_block_eigh(xh_ctx* ctx, const xh_factor_item* items, int64_t nitems, const double* A, double* W, double* V)
{
    return guard(ctx, [&] {
        std::vector<xh_factor_item> v(items, items + nitems);
        for(auto& it : v)
            if(it.m != it.n) throw xh::Error(XH_EINVAL, "eigh: blocks must be square");
        run_factor(
            ctx, k_eigh<true>, k_eigh<false>, v, [](const xh_factor_item& it) { return 2 * int64_t(it.m) * it.m + 2 * int64_t(it.m) + 4; }, A, V, W, nullptr);
    });
}

extern "C" int xh_block_chol_inv(xh_ctx* ctx, const xh_factor_item* items, int64_t nitems, const double* G, double* X, const double* shift_rel)
{
    // asynchronous: no status to read back, so no host synchronisation
    return guard(ctx, [&] {
        const size_t budget = lds_budget(ctx);
        std::vector<xh_factor_item> small, big;
        std::vector<double> sh;
        int64_t small_max = 0, big_max = 0;
        for(int64_t i = 0; i < nitems; ++i) {
            xh_factor_item it = items[i];
            if(it.m != it.n) throw xh::Error(XH_EINVAL, "chol_inv: blocks must be square");
            if(it.n < 0 || it.a_off < 0 || it.u_off < 0) throw xh::Error(XH_EINVAL, "chol_inv: negative extent or offset");
            if(it.n > CI_MAX_N) throw xh::Error(XH_EINVAL, "chol_inv: block larger than 40000");
            if(it.n == 0) continue;
            it.s_off = static_cast<int64_t>(sh.size());
            sh.push_back(shift_rel ? shift_rel[i] : 0.0);
            if(it.n <= 16 * (CI_THREADS / 64) && size_t(chol_work_doubles(it.n)) * sizeof(double) <= budget) {
                small.push_back(it);
                small_max = std::max(small_max, chol_work_doubles(it.n));
            } else {
                big.push_back(it);
                big_max = std::max(big_max, chol_work_doubles(it.n));
            }
        }
        if(sh.empty()) return;
        xh::PackedUpload up;
        const size_t o_small = up.add(small), o_big = up.add(big), o_sh = up.add(sh);
        up.upload(ctx);
        double* d_sh = up.ptr<double>(o_sh);
        if(!small.empty()) {
            const size_t shmem = size_t(small_max) * sizeof(double);
            if(shmem > 64 * 1024)
                check(hipFuncSetAttribute(reinterpret_cast<const void*>(k_chol_inv<true>), hipFuncAttributeMaxDynamicSharedMemorySize, int(shmem)), "hipFuncSetAttribute");
            FactorArgs fa{up.ptr<xh_factor_item>(o_small), G, X, d_sh, nullptr, nullptr, 0, 1, nullptr};
            hipLaunchKernelGGL(k_chol_inv<true>, dim3(static_cast<unsigned>(small.size())), dim3(CI_THREADS), shmem, ctx->stream, fa);
            xh::launch_check("k_chol_inv");
        }
        if(!big.empty()) {
            double* scratch = nullptr;
            check(xh::dmalloc(ctx, reinterpret_cast<void**>(&scratch), size_t(big_max) * big.size() * sizeof(double)), "hipMallocAsync");
            FactorArgs fa{up.ptr<xh_factor_item>(o_big), G, X, d_sh, nullptr, scratch, big_max, 0, nullptr};
            hipLaunchKernelGGL(k_chol_inv<false>, dim3(static_cast<unsigned>(big.size())), dim3(CI_THREADS), 0, ctx->stream, fa);
            xh::launch_check("k_chol_inv");
            xh::dev_free(ctx, scratch);
        }
        up.release_deferred(ctx);
    });
}

