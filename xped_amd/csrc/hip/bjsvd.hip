// FP64 SVD of large sector blocks by parallel one-sided block Jacobi.
//
// Each block A (m x n, worked on as A^T when m < n, so that it is rows x cols with rows >= cols)
// is copied into W and V = I is kept beside it, W = A V throughout.  The columns of W are cut
// into column blocks of width BJ_W; a sweep pairs every two column blocks once (round-robin
// tournament).  A step handles all pairs of all sector blocks at once:
//   G = [W_a W_b]^T [W_a W_b]          one grouped GEMM, one 2w x 2w tile per pair
//   G = J diag J^T                      k_bj_pair: cyclic Jacobi eigen-solve of G in LDS
//   [W_a W_b] <- [W_a W_b] J, same for V   one grouped GEMM that also moves the updated column
//                                       blocks to where the next step wants its pairs adjacent
// A pair whose columns are already orthogonal (|g_ij| <= tol sqrt(g_ii g_jj), the one-sided
// Jacobi test with tol = 8 sqrt(rows) sqrt(2w) eps to sit above the rounding noise of the Gram
// and update GEMMs; columns of norm below rows eps ||A||_F are numerical zeros and exempt) keeps
// J = I; a block is converged after a sweep without a rotation.  Then sigma_j = ||W_j||, U_j = W_j / sigma_j and V are
// read off in descending order of sigma.  The rotations are orthogonal transformations of the
// columns of A itself, so the result has the backward stability of one-sided Jacobi (Demmel &
// Veselic, SIAM J. Matrix Anal. Appl. 13 (1992) 1204; block form: Becka, Oksa & Vajtersic,
// Parallel Comput. 28 (2002) 243).
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <numeric>
#include <utility>

#include "device.hpp"

using xh::check;

namespace {

constexpr int BJ_W = 32;          // column block width; pairs are 64 columns wide
constexpr int BJ_THREADS = 1024;
constexpr int BJ_MAX_SWEEPS = 60;
constexpr int BJ_INNER_SWEEPS = 2;  // inexact pair solves: the outer sweeps finish the job

struct BjPair {
    int64_t g;       // offset of the pair's n2 x n2 Gram matrix (and of its J)
    int32_t n2;      // width of the pair
    int32_t sector;  // index of the block (for the rotation flag)
    int32_t rows;    // rows of the working matrix (convergence tolerance)
    int32_t pad;
    double z;        // squared norm below which a column counts as numerically zero
};

// Eigen-decomposition G = J diag(g) J^T of one pair's Gram matrix, eigenvalues descending: cyclic
// two-sided Jacobi in LDS, at most BJ_INNER_SWEEPS sweeps of np - 1 steps (np = n2 rounded up to
// even; a padding row and column of zeros never rotates).
//
// A step turns np / 2 disjoint planes at once and is bound by its latency and by LDS traffic.  The
// rows of A are kept by position in the tournament, so that the plane of pair P is always that
// of positions P and np - 1 - P; a step writes its result to the other of two buffers, every row
// already at its position of the next step (q -> q - 1, 1 -> np - 1, 0 -> 0).  So the addresses a
// thread reads and writes never change, and are computed once.  By symmetry only the 2 x 2 blocks
// of pairs I < J are kept (row in I, column in J), one per thread, and the diagonal blocks apart.
// V never touches LDS: half a wave holds two rows of it, lane k the entries at positions k and
// np - 1 - k, so a rotation stays inside a lane and the move to the next step is a shift by one
// lane (DPP).  Between two barriers one half wave turns the diagonal blocks into (c, s) while all
// waves apply the rotations of the step before to V and fetch their blocks of A; between the next
// two they turn the blocks.
// (256 threads, each rotating columns, then rows, of a square A in place, with 16 lanes of a wave
// on one bank in the row pass: 313 us per call at bond 701, up to two sweeps at n2 = 64; V in LDS
// and the blocks of A as here 102 us; this takes 76 us.)
constexpr int BJ_NMAX = 2 * BJ_W;
constexpr int BJ_LD = BJ_NMAX;
constexpr int BJ_BUF = BJ_NMAX * BJ_LD + 3 * BJ_W;  // one buffer: blocks, then app, aqq, apq per pair
constexpr double BJ_FAR = 1e-16;  // squared cosine above which another sweep follows
typedef double d2 __attribute__((ext_vector_type(2)));

__global__ __launch_bounds__(BJ_THREADS) void k_bj_pair(const BjPair* __restrict__ pairs, const double* __restrict__ G, double* __restrict__ J,
                                                         int* __restrict__ flags)
{
    extern __shared__ __attribute__((aligned(16))) double sm[];
    __shared__ int need, far;
    __shared__ double s_diag[BJ_NMAX];
    const BjPair pr = pairs[blockIdx.x];
    const int n = pr.n2;
    const int np = n + (n & 1), P = np / 2;
    double* buf0 = sm;                                  // two buffers
    d2* cs = reinterpret_cast<d2*>(buf0 + 2 * BJ_BUF);  // per pair, of an even and an odd step
    int* rank = reinterpret_cast<int*>(cs + 2 * BJ_W);
    const int tid = threadIdx.x;
    const double* Gp = G + pr.g;
    // offset of element (x, y) of A, by position, in a buffer: a block of pairs I < J, or the diagonal
    auto pair_of = [&](int x) { return min(x, np - 1 - x); };
    auto place = [&](int x, int y) {
        const int a = pair_of(x), b = pair_of(y);
        if(a != b) return a < b ? x * BJ_LD + y : y * BJ_LD + x;
        return BJ_NMAX * BJ_LD + 3 * a + (x != y ? 2 : (x < P ? 0 : 1));
    };
    auto next = [&](int x) { return x == 0 ? 0 : x == 1 ? np - 1 : x - 1; };  // position after a step
    if(tid == 0) need = far = 0;
    if(tid < BJ_NMAX) s_diag[tid] = tid < n ? Gp[tid + tid * n] : 0.0;
    __syncthreads();
    // scaled by a power of two to a largest diagonal entry of [1/2, 1): J does not change
    double mx = fabs(s_diag[tid & 63]);
    for(int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
    int ex = 0;
    if(mx > 0.0 && mx <= DBL_MAX) frexp(mx, &ex);
    // a computed inner product carries rounding noise of about sqrt(rows) eps relative to the
    // column norms, and the GEMM update of a pair adds about sqrt(n2) eps: pairs are orthogonal
    // once below a small multiple of both
    const double tol2 = 64.0 * fmax(1, pr.rows) * double(n) * DBL_EPSILON * DBL_EPSILON;
    const double z = ldexp(pr.z, -ex);
    const int ti = tid & 63, tj = tid >> 6;  // row, and first column, of this thread's entries
    for(int j = tj; j < np; j += BJ_THREADS / 64)
        if(ti >= j && ti < np) {  // the lower triangle of G
            const double g = ti < n ? ldexp(Gp[ti + j * n], -ex) : 0.0;
            buf0[place(ti, j)] = g;
            const double gi = ldexp(s_diag[ti], -ex), gj = ldexp(s_diag[j], -ex);
            if(ti > j && gi > z && gj > z && g * g > tol2 * (gi * gj)) need = 1;
        }
    __syncthreads();
    const int todo = need;
    double* cur = buf0;
    double* nxt = buf0 + BJ_BUF;
    // rows vrow, vrow + 2, ... of V at positions vk and np - 1 - vk
    constexpr int VR = BJ_NMAX * 32 / BJ_THREADS;
    const int vk = tid & 31, vrow = (tid >> 6) * 2 * VR + ((tid >> 5) & 1);
    double vt[VR], vb[VR];
#pragma unroll
    for(int q = 0; q < VR; ++q) {
        vt[q] = vrow + 2 * q == vk ? 1.0 : 0.0;
        vb[q] = vrow + 2 * q == np - 1 - vk ? 1.0 : 0.0;
    }
    if(todo) {
        if(tid == 0) atomicOr(flags + pr.sector, 1);
        // this thread's block of pairs I < J: blocks of one I on consecutive lanes
        const int nblk = P * (P - 1) / 2;
        int I = 0, Jb = 0, rd[4] = {}, wr[4] = {};
        if(tid < nblk) {
            int t = tid;
            while(t >= P - 1 - I) t -= P - 1 - I++;
            Jb = I + 1 + t;
            const int xi[2] = {I, np - 1 - I}, yj[2] = {Jb, np - 1 - Jb};
            for(int k = 0; k < 4; ++k) {
                rd[k] = place(xi[k >> 1], yj[k & 1]);
                wr[k] = place(next(xi[k >> 1]), next(yj[k & 1]));
            }
        }
        // the diagonal block of pair dg, on the last threads of the workgroup
        const int dg = tid - (BJ_THREADS - P);
        int dwr[3] = {};
        if(dg >= 0) {
            const int x = dg, y = np - 1 - dg;
            dwr[0] = place(next(x), next(x));
            dwr[1] = place(next(y), next(y));
            dwr[2] = place(next(x), next(y));
        }
        // the rotations r of a step applied to V, and its entries moved to the next step's positions
        auto turn_v = [&](const d2 r) {
#pragma unroll
            for(int q = 0; q < VR; ++q) {
                const double t = r[0] * vt[q] - r[1] * vb[q], b = r[1] * vt[q] + r[0] * vb[q];
                const double up = xh::dpp_mov<0x130>(t), down = xh::dpp_mov<0x138>(b);  // of lane vk + 1, of lane vk - 1
                vt[q] = vk == 0 ? t : vk == P - 1 ? b : up;
                vb[q] = vk == 0 ? (P > 1 ? up : b) : down;
            }
        };
        d2* cs_now = cs;
        d2* cs_last = cs + BJ_W;
        for(int sweep = 0; sweep < BJ_INNER_SWEEPS; ++sweep) {
            for(int step = 0; step < np - 1; ++step) {
                double app = 0, aqq = 0, apq = 0, c = 1.0, s = 0.0;
                if(dg >= 0) {
                    __builtin_amdgcn_s_setprio(3);  // everyone waits for these lanes
                    const double* D = cur + BJ_NMAX * BJ_LD + 3 * dg;
                    app = D[0];
                    aqq = D[1];
                    apq = D[2];
                    const double q2 = apq * apq, pq = fabs(app * aqq);
                    if(q2 > DBL_EPSILON * DBL_EPSILON * pq && q2 > 1e-280) {
                        xh::jacobi_rotation(0.5 * (aqq - app), apq, c, s);
                        if(q2 > BJ_FAR * pq) far = 1;
                    }
                    cs_now[dg] = d2{c, s};
                    __builtin_amdgcn_s_setprio(0);
                }
                double x[4];
                if(tid < nblk)
#pragma unroll
                    for(int k = 0; k < 4; ++k) x[k] = cur[rd[k]];
                if(step > 0) turn_v(cs_last[vk]);
                __syncthreads();
                if(tid < nblk) {
                    const d2 ci = cs_now[I], cj = cs_now[Jb];
                    // rows by the rotation of I, then columns by that of J
                    const double y0 = ci[0] * x[0] - ci[1] * x[2], y2 = ci[1] * x[0] + ci[0] * x[2];
                    const double y1 = ci[0] * x[1] - ci[1] * x[3], y3 = ci[1] * x[1] + ci[0] * x[3];
                    nxt[wr[0]] = cj[0] * y0 - cj[1] * y1;
                    nxt[wr[1]] = cj[1] * y0 + cj[0] * y1;
                    nxt[wr[2]] = cj[0] * y2 - cj[1] * y3;
                    nxt[wr[3]] = cj[1] * y2 + cj[0] * y3;
                }
                if(dg >= 0) {
                    const double cc = c * c, ss = s * s, sc = s * c;
                    nxt[dwr[0]] = cc * app - 2.0 * sc * apq + ss * aqq;
                    nxt[dwr[1]] = ss * app + 2.0 * sc * apq + cc * aqq;
                    nxt[dwr[2]] = sc * (app - aqq) + (cc - ss) * apq;
                }
                std::swap(cur, nxt);
                std::swap(cs_now, cs_last);
                __syncthreads();
            }
            turn_v(cs_last[vk]);
            const int again = far;
            __syncthreads();
            if(!again) break;
            if(tid == 0) far = 0;
            __syncthreads();
        }
    }
    // descending eigenvalues (NaN last), ties by index; J columns in that order.  A sweep ends with
    // every row back at its own position.
    if(tid < n) {
        const double v = cur[place(tid, tid)];
        s_diag[tid] = v == v ? v : -2.0 * DBL_MAX;
    }
    // V by columns through the buffer that is free
#pragma unroll
    for(int q = 0; q < VR; ++q)
        if(vk < P && vrow + 2 * q < np) {
            nxt[vk * BJ_LD + vrow + 2 * q] = vt[q];
            nxt[(np - 1 - vk) * BJ_LD + vrow + 2 * q] = vb[q];
        }
    __syncthreads();
    for(int j = tid >> 4; j < n; j += BJ_THREADS / 16) {  // 16 lanes count the values above value j
        const double vj = s_diag[j];
        int r = 0;
        for(int k = tid & 15; k < n; k += 16) r += (s_diag[k] > vj) || (s_diag[k] == vj && k < j);
        for(int o = 8; o > 0; o >>= 1) r += __shfl_xor(r, o);
        if((tid & 15) == 0) rank[r] = j;
    }
    __syncthreads();
    for(int c = tj; c < n; c += BJ_THREADS / 64)
        if(ti < n) J[pr.g + ti + c * n] = todo ? nxt[ti + rank[c] * BJ_LD] : (ti == c ? 1.0 : 0.0);
}

__global__ void k_set_ones(const int64_t* __restrict__ pos, int64_t n, double* __restrict__ x)
{
    for(int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) x[pos[i]] = 1.0;
}

struct Sec {
    xh_factor_item it;
    bool tr;
    int rows, cols;    // working matrix rows x cols, rows >= cols
    int nb, np, L;     // column blocks, players (even), steps per sweep
    int64_t w, v;      // offsets of W (rows x cols) and V (cols x cols) in the work buffers
    double z = 0.0;    // (rows eps ||A||_F)^2: columns of smaller squared norm are numerical zeros
    int done = 0;      // 0 active, 1 or 2: converged with the result in buffer 0 or 1
    int width(int b) const { return std::min(BJ_W, cols - b * BJ_W); }
    // ordered blocks of step s (pairs adjacent, the dummy player dropped) and pair boundaries
    void layout(int s, std::vector<int>& order, std::vector<std::pair<int, int>>& pairs) const
    {
        order.clear();
        pairs.clear();
        for(int p = 0; p < np / 2; ++p) {
            int a = bj_host_player(p, s), b = bj_host_player(np - 1 - p, s);
            if(a > b) std::swap(a, b);
            if(b >= nb) b = -1;
            pairs.emplace_back(a, b);
            order.push_back(a);
            if(b >= 0) order.push_back(b);
        }
    }
    std::vector<int64_t> col_offsets(int s) const
    {
        std::vector<int> order;
        std::vector<std::pair<int, int>> pairs;
        layout(s, order, pairs);
        std::vector<int64_t> off(nb, 0);
        int64_t c = 0;
        for(int b : order) {
            off[b] = c;
            c += width(b);
        }
        return off;
    }
    int bj_host_player(int pos, int step) const
    {
        if(np == 1) return 0;
        if(pos == 0) return 0;
        return ((pos - 1 + step) % (np - 1)) + 1;
    }
};

struct PlanSet {
    xh_ctx* ctx;
    std::vector<xh_gemm_plan*> gram, update;
    std::vector<int64_t> pair_begin, pair_count;
    int64_t n_pairs = 0;
    BjPair* d_pairs = nullptr;
    ~PlanSet() { clear(); }
    void clear()
    {
        for(auto* p : gram)
            if(p) xh_gemm_plan_destroy(ctx, p);
        for(auto* p : update)
            if(p) xh_gemm_plan_destroy(ctx, p);
        gram.clear();
        update.clear();
        pair_begin.clear();
        pair_count.clear();
        n_pairs = 0;
        xh::dev_free(ctx, d_pairs);
        d_pairs = nullptr;
    }
};

void gemm_plan(xh_ctx* ctx, const std::vector<xh_gemm_item>& items, int ta, int tb, xh_gemm_plan** out)
{
    *out = nullptr;
    if(items.empty()) return;
    const int rc = xh_gemm_plan_create(ctx, items.data(), static_cast<int64_t>(items.size()), ta, tb, out);
    if(rc != XH_OK) throw xh::Error(rc, std::string("block Jacobi plan: ") + xh_last_error(ctx));
}

// Plans for the T steps of one global sweep over the active blocks; block q runs step t mod L_q
// and leaves its columns where its next step wants them.  Returns the Gram buffer size needed.
int64_t build_plans(xh_ctx* ctx, std::vector<Sec>& secs, int T, int64_t nw, PlanSet& ps)
{
    ps.clear();
    // every operand of every item must lie inside its buffer (W/V work buffers of nw doubles,
    // Gram/J buffers of the returned size)
    auto inside = [](int64_t off, int64_t len, int64_t cap) { return off >= 0 && len >= 0 && off + len <= cap; };
    std::vector<BjPair> all_pairs;
    int64_t gsize = 0;
    for(int t = 0; t < T; ++t) {
        std::vector<xh_gemm_item> gram, upd;
        int64_t g = 0;
        ps.pair_begin.push_back(static_cast<int64_t>(all_pairs.size()));
        for(std::size_t q = 0; q < secs.size(); ++q) {
            const Sec& c = secs[q];
            if(c.done) continue;
            const int s = t % c.L, s_next = ((t + 1) % T) % c.L;
            std::vector<int> order;
            std::vector<std::pair<int, int>> pairs;
            c.layout(s, order, pairs);
            const std::vector<int64_t> off = c.col_offsets(s), off_next = c.col_offsets(s_next);
            for(const auto& [a, b] : pairs) {
                const int wa = c.width(a), wb = b >= 0 ? c.width(b) : 0, n2 = wa + wb;
                const int64_t panel_w = c.w + off[a] * c.rows, panel_v = c.v + off[a] * c.cols;
                gram.push_back(xh_gemm_item{panel_w, panel_w, g, n2, n2, c.rows});
                all_pairs.push_back(BjPair{g, n2, static_cast<int32_t>(q), c.rows, 0, c.z});
                upd.push_back(xh_gemm_item{panel_w, g, c.w + off_next[a] * c.rows, c.rows, wa, n2});
                upd.push_back(xh_gemm_item{panel_v, g, c.v + off_next[a] * c.cols, c.cols, wa, n2});
                if(wb) {
                    upd.push_back(xh_gemm_item{panel_w, g + int64_t(wa) * n2, c.w + off_next[b] * c.rows, c.rows, wb, n2});
                    upd.push_back(xh_gemm_item{panel_v, g + int64_t(wa) * n2, c.v + off_next[b] * c.cols, c.cols, wb, n2});
                }
                g += int64_t(n2) * n2;
            }
        }
        ps.pair_count.push_back(static_cast<int64_t>(all_pairs.size()) - ps.pair_begin.back());
        gsize = std::max(gsize, g);
        for(const auto& it : gram)
            if(!inside(it.a_off, int64_t(it.m) * it.k, nw) || !inside(it.c_off, int64_t(it.m) * it.n, g))
                throw xh::Error(XH_EINVAL, "block Jacobi: Gram item out of range");
        for(const auto& it : upd)
            if(!inside(it.a_off, int64_t(it.m) * it.k, nw) || !inside(it.b_off, int64_t(it.k) * it.n, g) || !inside(it.c_off, int64_t(it.m) * it.n, nw))
                throw xh::Error(XH_EINVAL, "block Jacobi: update item out of range");
        xh_gemm_plan *pg = nullptr, *pu = nullptr;
        gemm_plan(ctx, gram, 1, 0, &pg);
        ps.gram.push_back(pg);
        gemm_plan(ctx, upd, 0, 0, &pu);
        ps.update.push_back(pu);
    }
    ps.n_pairs = static_cast<int64_t>(all_pairs.size());
    ps.d_pairs = xh::dev_upload(ctx, all_pairs);
    return gsize;
}

}  // namespace

// Called by xh_block_svd for blocks too large for the single-workgroup Jacobi kernel.
void block_jacobi_svd(xh_ctx* ctx, const std::vector<xh_factor_item>& items, const double* A, double* U, double* S, double* Vt)
{
    if(items.empty()) return;
    std::vector<Sec> secs;
    int64_t nw = 0;
    for(const auto& it : items) {
        Sec c{};
        c.it = it;
        c.tr = it.m < it.n;
        c.rows = std::max(it.m, it.n);
        c.cols = std::min(it.m, it.n);
        c.nb = (c.cols + BJ_W - 1) / BJ_W;
        c.np = c.nb + (c.nb & 1);
        if(c.nb == 1) c.np = 2;
        c.L = c.np - 1;
        c.w = nw;
        nw += int64_t(c.rows) * c.cols;
        c.v = nw;
        nw += int64_t(c.cols) * c.cols;
        secs.push_back(c);
    }
    double *buf[2] = {nullptr, nullptr}, *G = nullptr, *Jm = nullptr;
    int* d_flags = nullptr;
    int64_t* d_ones = nullptr;
    auto cleanup = [&] {
        xh::dev_free(ctx, buf[0]);
        xh::dev_free(ctx, buf[1]);
        xh::dev_free(ctx, G);
        xh::dev_free(ctx, Jm);
        xh::dev_free(ctx, d_flags);
        xh::dev_free(ctx, d_ones);
    };
    PlanSet ps{ctx};
    try {
        check(xh::dmalloc(ctx, reinterpret_cast<void**>(&buf[0]), size_t(nw) * sizeof(double)), "hipMallocAsync");
        check(xh::dmalloc(ctx, reinterpret_cast<void**>(&buf[1]), size_t(nw) * sizeof(double)), "hipMallocAsync");
        check(xh::dmalloc(ctx, reinterpret_cast<void**>(&d_flags), sizeof(int) * secs.size()), "hipMallocAsync");
        // W = A (or A^T) in the layout of step 0, V = the matching column permutation of I
        std::vector<xh_copy_rect> rects;
        std::vector<int64_t> ones;
        for(const auto& c : secs) {
            const std::vector<int64_t> off = c.col_offsets(0);
            for(int b = 0; b < c.nb; ++b) {
                const int wb = c.width(b);
                if(!c.tr)
                    rects.push_back(xh_copy_rect{c.it.a_off + int64_t(b) * BJ_W * c.it.m, c.it.m, c.w + off[b] * c.rows, c.rows, c.rows, wb, 1.0, 0});
                else
                    rects.push_back(xh_copy_rect{c.it.a_off + int64_t(b) * BJ_W, c.it.m, c.w + off[b] * c.rows, c.rows, c.rows, wb, 1.0, 1});
                for(int k = 0; k < wb; ++k) ones.push_back(c.v + (b * BJ_W + k) + (off[b] + k) * int64_t(c.cols));
            }
        }
        {
            std::vector<int64_t> off, len;
            for(const auto& c : secs) {
                off.push_back(c.it.a_off);
                len.push_back(int64_t(c.it.m) * c.it.n);
            }
            std::vector<double> nrm(secs.size());
            const int rc0 = xh_range_sumsq(ctx, off.data(), len.data(), static_cast<int64_t>(off.size()), A, nrm.data());
            if(rc0 != XH_OK) throw xh::Error(rc0, "block Jacobi: block norms");
            for(std::size_t q = 0; q < secs.size(); ++q) {
                if(!std::isfinite(nrm[q])) throw xh::Error(XH_EINVAL, "block SVD: non-finite input block");
                const double f = double(secs[q].rows) * DBL_EPSILON;
                secs[q].z = f * f * nrm[q];
            }
        }
        int rc = xh_copy_rects(ctx, A, buf[0], rects.data(), static_cast<int64_t>(rects.size()));
        if(rc != XH_OK) throw xh::Error(rc, "block Jacobi: initial copy");
        for(const auto& c : secs) check(hipMemsetAsync(buf[0] + c.v, 0, size_t(c.cols) * c.cols * sizeof(double), ctx->stream), "hipMemsetAsync");
        d_ones = xh::dev_upload(ctx, ones);
        hipLaunchKernelGGL(k_set_ones, dim3(static_cast<unsigned>(std::min<int64_t>((ones.size() + 255) / 256, 65535))), dim3(256), 0, ctx->stream, d_ones,
                           static_cast<int64_t>(ones.size()), buf[0]);
        xh::launch_check("k_set_ones");
        const size_t pair_lds = size_t(2 * BJ_BUF + 4 * BJ_W + BJ_NMAX / 2) * sizeof(double);
        check(hipFuncSetAttribute(reinterpret_cast<const void*>(k_bj_pair), hipFuncAttributeMaxDynamicSharedMemorySize, int(pair_lds)), "hipFuncSetAttribute");
        int cur = 0;
        int64_t gcap = 0;
        bool rebuild = true;
        int T = 0;
        for(int sweep = 0;; ++sweep) {
            if(rebuild) {
                T = 0;
                for(const auto& c : secs)
                    if(!c.done) T = std::max(T, c.L);
                const int64_t gsize = build_plans(ctx, secs, T, nw, ps);
                if(static_cast<int>(ps.gram.size()) != T || static_cast<int>(ps.pair_begin.size()) != T)
                    throw xh::Error(XH_EINVAL, "block Jacobi: inconsistent step plans");
                if(gsize > gcap) {
                    xh::dev_free(ctx, G);
                    xh::dev_free(ctx, Jm);
                    check(xh::dmalloc(ctx, reinterpret_cast<void**>(&G), size_t(gsize) * sizeof(double)), "hipMallocAsync");
                    check(xh::dmalloc(ctx, reinterpret_cast<void**>(&Jm), size_t(gsize) * sizeof(double)), "hipMallocAsync");
                    gcap = gsize;
                }
                rebuild = false;
            }
            check(hipMemsetAsync(d_flags, 0, sizeof(int) * secs.size(), ctx->stream), "hipMemsetAsync");
            for(int t = 0; t < T; ++t) {
                if(ps.gram[t]) {
                    rc = xh_gemm(ctx, ps.gram[t], buf[cur], buf[cur], G, 1.0, 0.0, XH_FP64);
                    if(rc != XH_OK) throw xh::Error(rc, std::string("block Jacobi Gram: ") + xh_last_error(ctx));
                }
                if(ps.pair_begin[t] < 0 || ps.pair_begin[t] + ps.pair_count[t] > ps.n_pairs) throw xh::Error(XH_EINVAL, "block Jacobi: pair range");
                if(ps.pair_count[t]) {
                    hipLaunchKernelGGL(k_bj_pair, dim3(static_cast<unsigned>(ps.pair_count[t])), dim3(BJ_THREADS), pair_lds, ctx->stream,
                                       ps.d_pairs + ps.pair_begin[t], G, Jm, d_flags);
                    xh::launch_check("k_bj_pair");
                }
                if(ps.update[t]) {
                    rc = xh_gemm(ctx, ps.update[t], buf[cur], Jm, buf[1 - cur], 1.0, 0.0, XH_FP64);
                    if(rc != XH_OK) throw xh::Error(rc, std::string("block Jacobi update: ") + xh_last_error(ctx));
                }
                cur = 1 - cur;
            }
            std::vector<int> flags(secs.size());
            check(hipMemcpyAsync(flags.data(), d_flags, sizeof(int) * secs.size(), hipMemcpyDeviceToHost, ctx->stream), "hipMemcpyAsync");
            check(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
            bool active = false;
            for(std::size_t q = 0; q < secs.size(); ++q) {
                if(secs[q].done) continue;
                if(!flags[q]) {
                    secs[q].done = 1 + cur;
                    rebuild = true;
                } else {
                    active = true;
                }
            }
            if(!active) break;
            if(sweep + 1 >= BJ_MAX_SWEEPS) throw xh::Error(XH_ENOTCONV, "block Jacobi SVD did not converge within the sweep limit");
        }
        // singular values = column norms; outputs in descending order
        std::vector<int64_t> roff[2], rlen[2];
        std::vector<std::pair<int, int>> where[2];  // (sector, column)
        for(std::size_t q = 0; q < secs.size(); ++q) {
            const Sec& c = secs[q];
            const int b = c.done - 1;
            for(int j = 0; j < c.cols; ++j) {
                roff[b].push_back(c.w + int64_t(j) * c.rows);
                rlen[b].push_back(c.rows);
                where[b].emplace_back(static_cast<int>(q), j);
            }
        }
        std::vector<std::vector<double>> sig(secs.size());
        for(std::size_t q = 0; q < secs.size(); ++q) sig[q].assign(secs[q].cols, 0.0);
        for(int b = 0; b < 2; ++b) {
            if(roff[b].empty()) continue;
            std::vector<double> nrm(roff[b].size());
            rc = xh_range_sumsq(ctx, roff[b].data(), rlen[b].data(), static_cast<int64_t>(roff[b].size()), buf[b], nrm.data());
            if(rc != XH_OK) throw xh::Error(rc, "block Jacobi: column norms");
            for(std::size_t k = 0; k < nrm.size(); ++k) {
                if(!std::isfinite(nrm[k])) throw xh::Error(XH_EHIP, "block Jacobi SVD: non-finite column norm");
                sig[where[b][k].first][where[b][k].second] = std::sqrt(nrm[k]);
            }
        }
        std::vector<xh_copy_rect> out[2];
        for(std::size_t q = 0; q < secs.size(); ++q) {
            const Sec& c = secs[q];
            const int b = c.done - 1;
            std::vector<int> ord(c.cols);
            std::iota(ord.begin(), ord.end(), 0);
            const std::vector<double>& s = sig[q];
            std::stable_sort(ord.begin(), ord.end(), [&](int x, int y) { return s[x] > s[y]; });
            std::vector<double> sv(c.cols);
            for(int r = 0; r < c.cols; ++r) {
                const int col = ord[r];
                const double sr = s[col];
                sv[r] = sr;
                const double inv = sr > 0.0 ? 1.0 / sr : 0.0;
                const int64_t wcol = c.w + int64_t(col) * c.rows, vcol = c.v + int64_t(col) * c.cols;
                const int m = c.it.m, n = c.it.n;
                if(!c.tr) {
                    out[b].push_back(xh_copy_rect{wcol, c.rows, c.it.u_off + int64_t(r) * m, m, m, 1, inv, 0});
                    out[b].push_back(xh_copy_rect{vcol, c.cols, c.it.vt_off + r, c.cols, 1, n, 1.0, 1});
                } else {
                    out[b].push_back(xh_copy_rect{vcol, c.cols, c.it.u_off + int64_t(r) * m, m, m, 1, 1.0, 0});
                    out[b].push_back(xh_copy_rect{wcol, c.rows, c.it.vt_off + r, m, 1, n, inv, 1});
                }
            }
            check(hipMemcpyAsync(S + c.it.s_off, sv.data(), sizeof(double) * sv.size(), hipMemcpyHostToDevice, ctx->stream), "hipMemcpyAsync");
            check(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
        }
        // U and Vt are written from one buffer at a time; both are disjoint outputs
        for(int b = 0; b < 2; ++b) {
            if(out[b].empty()) continue;
            std::vector<xh_copy_rect> ru, rv;
            for(std::size_t k = 0; k < out[b].size(); k += 2) {
                ru.push_back(out[b][k]);
                rv.push_back(out[b][k + 1]);
            }
            rc = xh_copy_rects(ctx, buf[b], U, ru.data(), static_cast<int64_t>(ru.size()));
            if(rc == XH_OK) rc = xh_copy_rects(ctx, buf[b], Vt, rv.data(), static_cast<int64_t>(rv.size()));
            if(rc != XH_OK) throw xh::Error(rc, "block Jacobi: outputs");
        }
        check(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
    } catch(...) {
        ps.clear();
        hipStreamSynchronize(ctx->stream);
        cleanup();
        throw;
    }
    ps.clear();
    cleanup();
}
