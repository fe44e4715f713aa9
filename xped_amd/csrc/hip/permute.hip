// Grouped block-sparse permute: one launch moves every subblock of a tensor.
//
// The reference walks sectors x domain trees x codomain trees on the host and, per subblock,
// copies it out of its sector block, shuffles it with Eigen and adds it (scaled by the
// recoupling coefficient) into the output block (src/Core/Tensor.cpp:179-212, with
// PlainInterface::tensor_from_matrix_block / shuffle / add_to_block_from_tensor).
//
// Here the host builds a gather plan once: every output subblock ("task") knows its sources
// and coefficients.  The kernel walks the concatenated output element space in tiles; each
// output element is written exactly once (accumulated over its sources in the reference's
// order, each product rounded or fused with its sum), so abelian permutes are bit-exact
// copies/negations.
//
// The index arithmetic, not the bytes, bounds the gather, so the plan leaves the kernel little of it
// (compact tasks): legs of extent 1 are dropped and legs that lie behind one another in output and
// source alike are joined, which leaves one to five of the seven legs of a CTMRG intermediate.
// Tasks whose first output leg maps to a unit-stride source leg are copied with coalesced
// reads and writes.  Tasks where the leading output leg is strided in the source (a real
// transpose) go through a 64x64 LDS tile so that both the global loads and the global stores
// are coalesced.
#include <algorithm>
#include <cstring>

#include "device.hpp"
#include "../common/pool.hpp"

using xh::check;
using xh::guard;

namespace {

constexpr int PT_THREADS = 256;
constexpr int PT_TILE = 2048;  // output elements per workgroup in the gather path
constexpr int TR_DIM = 64;     // transpose tile edge

struct TaskMeta {
    int64_t dst_off, dst_ld;
    uint32_t rows, rmagic, rshift, pad;  // rmagic / rshift: magic-number division by rows
    int32_t nsrc, src_begin;
};
// (row, column) of element el of a task's column-major output subblock, without an integer divide
__device__ __forceinline__ void split_el(const TaskMeta& tm, uint32_t el, uint32_t& row, uint32_t& col)
{
    col = xh::fdiv(el, tm.rmagic, tm.rshift);
    row = el - col * tm.rows;
}

using xh::leg_cstride;
using xh::leg_rstride;
using xh::leg_shift;
using xh::LegInfo;

struct PermDev {
    int nlegs, new_rank;
    int64_t ntasks, total;
    const TaskMeta* meta;
    const LegInfo* legs;  // ntasks * nlegs
    const int64_t* prefix;  // ntasks + 1 (element prefix of gather tasks)
    const int32_t* tile_first;  // gather tiles: first task of each tile (+1 sentinel)
    const xh_permute_source* src;
    // transpose path
    int64_t ntr_tiles;
    const int4* tr_tiles;  // (task, tile index along the contiguous-source leg, tile index along rows, rest index)
};

// Source row / column offsets of the output element (row, col) of a task: every output leg's
// index is peeled off the output row (domain legs) or column (codomain legs) and mapped through
// its source stride.
__device__ __forceinline__ void decode_src(const LegInfo* __restrict__ L, int nlegs, int new_rank, uint32_t row, uint32_t col, int64_t& srow,
                                           int64_t& scol)
{
    srow = 0;
    scol = 0;
    for(int k = 0; k < nlegs; ++k) {
        const LegInfo li = L[k];
        const bool is_row = k < new_rank;
        const uint32_t x = is_row ? row : col;
        const uint32_t q = xh::fdiv(x, li.magic, leg_shift(li));
        const uint32_t j = x - q * li.ext;
        if(is_row)
            row = q;
        else
            col = q;
        srow += int64_t(j) * leg_rstride(li);
        scol += int64_t(j) * leg_cstride(li);
    }
}

__device__ __forceinline__ double gather_one(const PermDev& p, const TaskMeta& tm, const double* __restrict__ src, int64_t srow, int64_t scol)
{
    double acc = 0.0;
    for(int s = 0; s < tm.nsrc; ++s) {
        const xh_permute_source so = p.src[tm.src_begin + s];
        const double v = src[so.src_off + srow + scol * so.src_ld];
        acc = __dadd_rn(acc, __dmul_rn(so.coeff, v));
    }
    return acc;
}

// A gather task with its legs joined: nl legs of extent > 1 in a plan-wide stride of nlegs records.
// The index of output element el (column-major in its subblock) along each is peeled off el leg by
// leg; the last needs no division.
struct TaskC {
    int64_t dst_off, dst_ld, src_off;  // src_off: of the task's only source (single-source plans)
    double coeff;                      // its coefficient
    uint32_t rows, rmagic, rshift, nl;
    int32_t nsrc, src_begin;
};
struct LegC {
    uint32_t ext, magic, shift;  // shift: bit 8 set for a source column leg (plans with several sources)
    uint32_t stride;             // in source elements (single-source), else in source rows or columns
};
struct PermC {
    int32_t nlegs, ordered;     // ordered: the tasks' source ranges follow one another
    int64_t total;
    const TaskC* task;
    const LegC* legs;           // ntasks * nlegs
    const int64_t* prefix;      // ntasks + 1
    const int32_t* tile_first;  // first task of each tile (+1 sentinel)
    const xh_permute_source* src;
};

// Gather of compact tasks.  A workgroup covers 256 PER consecutive output elements (in task order,
// each task column-major in its output subblock); thread i handles elements i, i + 256, ...  The
// records of the tile's tasks are staged in LDS and an element finds its task by binary search
// over their first elements.  All source offsets of a thread are computed first, then its PER loads
// go out back to back, then the scaled stores; with several sources per task (recoupling sums) the
// loop over sources is outermost, so that PER loads are in flight per source, and each element
// accumulates in the reference's order.  0 + c v keeps the sign of zero of that accumulation.
// PER: 4 (8 was slower: 73 us in the first example below, 143 with several sources, by registers and
// LDS), or 2 for small tensors, whose time is the latency of one workgroup.
// Bound by the loads of 8 bytes at L2 line granularity and by the decode: 16.8 M elements of a
// seven-leg tensor in 46508 tasks 68 us (3.9 TB/s, a copy of the size takes 56), 15.5 M elements from
// 26.8 M sources of an eight-leg SU(2) tensor 112 us.  (All legs decoded per element from int64
// strides, a thread's elements one after the other where they have several sources: 88 and 148.)
constexpr int MC_CAP = 48;    // tasks of a tile whose records are staged in LDS
constexpr int MC_LEGS = 8;    // legs of a staged task
constexpr int SRC_CAP = 192;  // their sources (several per task)

// A tile inside one task: its records are the same for every lane and come through scalar loads, a leg at a
// time for all elements of a thread.  6 M elements of ten legs that do not join, in 102 tasks: 24 us with one
// source and 48 with four (from LDS or global memory like the other tiles 46 and 79; before there were
// compact tasks 33 and 50).
template <bool SINGLE, int PER>
__device__ __forceinline__ void one_task(const PermC& p, int t, int64_t e0, int n_here, const double* __restrict__ src, double* __restrict__ dst)
{
    const TaskC tk = p.task[t];
    const LegC* L = p.legs + int64_t(t) * p.nlegs;
    uint32_t x[PER];
    int64_t dpos[PER], off[PER];
    uint32_t row[SINGLE ? 1 : PER], col[SINGLE ? 1 : PER];
    const int64_t base = e0 - p.prefix[t];
#pragma unroll
    for(int i = 0; i < PER; ++i) {
        const int r = threadIdx.x + i * PT_THREADS;
        // an element past the end is taken as the first of the tile, and not stored
        x[i] = static_cast<uint32_t>(base + (r < n_here ? r : 0));
        const uint32_t c = xh::fdiv(x[i], tk.rmagic, tk.rshift);
        dpos[i] = tk.dst_off + (x[i] - c * tk.rows) + int64_t(c) * tk.dst_ld;
        off[i] = tk.src_off;
        if constexpr(!SINGLE) row[i] = col[i] = 0;
    }
    for(uint32_t k = 0; k < tk.nl; ++k) {
        const LegC l = L[k];
#pragma unroll
        for(int i = 0; i < PER; ++i) {
            const uint32_t q = xh::fdiv(x[i], l.magic, l.shift & 255u), d = x[i] - q * l.ext;
            if constexpr(SINGLE)
                off[i] += uint64_t(d) * l.stride;
            else if(l.shift & 256u)
                col[i] += d * l.stride;
            else
                row[i] += d * l.stride;
            x[i] = q;
        }
    }
    double val[PER];
    if constexpr(SINGLE) {
#pragma unroll
        for(int i = 0; i < PER; ++i) val[i] = src[off[i]];
#pragma unroll
        for(int i = 0; i < PER; ++i) val[i] = __dadd_rn(0.0, __dmul_rn(tk.coeff, val[i]));
    } else {
#pragma unroll
        for(int i = 0; i < PER; ++i) val[i] = 0.0;
        for(int s = 0; s < tk.nsrc; ++s) {
            const xh_permute_source so = p.src[tk.src_begin + s];
            double v[PER];
#pragma unroll
            for(int i = 0; i < PER; ++i) v[i] = src[so.src_off + row[i] + int64_t(col[i]) * so.src_ld];
#pragma unroll
            for(int i = 0; i < PER; ++i) val[i] = __dadd_rn(val[i], __dmul_rn(so.coeff, v[i]));
        }
    }
#pragma unroll
    for(int i = 0; i < PER; ++i)
        if(int(threadIdx.x) + i * PT_THREADS < n_here) dst[dpos[i]] = val[i];
}

template <bool SINGLE, int PER>
__global__ __launch_bounds__(PT_THREADS) void k_permute_compact(PermC p, const double* __restrict__ src, double* __restrict__ dst)
{
    constexpr int TILE = PER * PT_THREADS;
    __shared__ int32_t start[TILE + 1];
    __shared__ TaskC s_task[MC_CAP];
    __shared__ LegC s_legs[MC_CAP * MC_LEGS];
    __shared__ xh_permute_source s_src[SINGLE ? 1 : SRC_CAP];
    const int64_t e0 = int64_t(blockIdx.x) * TILE;
    const int n_here = static_cast<int>(min(int64_t(TILE), p.total - e0));
    const int t_lo = p.tile_first[blockIdx.x], t_hi = p.tile_first[blockIdx.x + 1];
    if(t_lo == t_hi) {
        one_task<SINGLE, PER>(p, __builtin_amdgcn_readfirstlane(t_lo), e0, n_here, src, dst);
        return;
    }
    // tasks t_lo .. t_hi intersect the tile; at most TILE + 1 since every task holds an element
    const int nt = t_hi - t_lo + 1, nl_max = p.nlegs;
    const bool staged = nt <= MC_CAP && nl_max <= MC_LEGS;  // uniform over the workgroup
    for(int j = threadIdx.x; j < nt; j += PT_THREADS) start[j] = static_cast<int32_t>(p.prefix[t_lo + j] - e0);  // a task holds less than 2^31 elements
    int s_first = 0, s_count = 0;
    if(staged) {
        for(int j = threadIdx.x; j < nt; j += PT_THREADS) s_task[j] = p.task[t_lo + j];
        for(int j = threadIdx.x; j < nt * nl_max; j += PT_THREADS) s_legs[j] = p.legs[int64_t(t_lo) * nl_max + j];
        if constexpr(!SINGLE) {
            s_first = p.task[t_lo].src_begin;
            s_count = p.ordered ? p.task[t_hi].src_begin + p.task[t_hi].nsrc - s_first : SRC_CAP + 1;
            if(s_count <= SRC_CAP)
                for(int j = threadIdx.x; j < s_count; j += PT_THREADS) s_src[j] = p.src[s_first + j];
        }
    }
    __syncthreads();
    const bool src_staged = !SINGLE && staged && s_count <= SRC_CAP;
    int64_t dpos[PER], soff[SINGLE ? PER : 1];
    uint32_t srow[SINGLE ? 1 : PER], scol[SINGLE ? 1 : PER];
    double val[PER], coef[SINGLE ? PER : 1];
    int ns[SINGLE ? 1 : PER], sb[SINGLE ? 1 : PER];
    auto decode = [&](int i, const TaskC& tk, const LegC* L, uint32_t el) {
        const uint32_t col = xh::fdiv(el, tk.rmagic, tk.rshift);
        dpos[i] = tk.dst_off + (el - col * tk.rows) + int64_t(col) * tk.dst_ld;
        uint32_t x = el;
        if constexpr(SINGLE) {
            int64_t off = tk.src_off;
            for(uint32_t k = 0; k + 1 < tk.nl; ++k) {
                const uint32_t q = xh::fdiv(x, L[k].magic, L[k].shift);
                off += uint64_t(x - q * L[k].ext) * L[k].stride;
                x = q;
            }
            if(tk.nl > 0) off += uint64_t(x) * L[tk.nl - 1].stride;
            soff[i] = off;
            coef[i] = tk.coeff;
        } else {
            uint32_t r = 0, c = 0;  // source row and column: below 2^31 (checked at plan creation)
            for(uint32_t k = 0; k < tk.nl; ++k) {
                const LegC l = L[k];
                const uint32_t q = xh::fdiv(x, l.magic, l.shift & 255u), d = (x - q * l.ext) * l.stride;
                r += (l.shift & 256u) ? 0 : d;
                c += (l.shift & 256u) ? d : 0;
                x = q;
            }
            srow[i] = r;
            scol[i] = c;
            ns[i] = tk.nsrc;
            sb[i] = tk.src_begin;
        }
    };
    auto find_task = [&](int r) {
        int lo = 0, hi = nt - 1;  // last j with start[j] <= r
        while(lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if(start[mid] <= r)
                lo = mid;
            else
                hi = mid - 1;
        }
        return lo;
    };
#pragma unroll
    for(int i = 0; i < PER; ++i) {
        const int r = threadIdx.x + i * PT_THREADS;
        dpos[i] = -1;
        val[i] = 0.0;
        if constexpr(SINGLE) {
            soff[i] = 0;
            coef[i] = 0.0;
        } else {
            ns[i] = 0;
            sb[i] = 0;
            srow[i] = scol[i] = 0;
        }
        if(r < n_here) {
            const int t = find_task(r);
            if(staged)
                decode(i, s_task[t], s_legs + t * nl_max, static_cast<uint32_t>(r - start[t]));
            else
                decode(i, p.task[t_lo + t], p.legs + int64_t(t_lo + t) * nl_max, static_cast<uint32_t>(e0 + r - p.prefix[t_lo + t]));
        }
    }
    if constexpr(SINGLE) {
        // inactive elements load src[0]: a single-source plan reads at least one source element
#pragma unroll
        for(int i = 0; i < PER; ++i) val[i] = src[soff[i]];
#pragma unroll
        for(int i = 0; i < PER; ++i) val[i] = __dadd_rn(0.0, __dmul_rn(coef[i], val[i]));
    } else {
        int most = 0;
#pragma unroll
        for(int i = 0; i < PER; ++i) most = max(most, ns[i]);
        for(int s = 0; s < most; ++s) {
            double v[PER], c[PER];
#pragma unroll
            for(int i = 0; i < PER; ++i) {
                v[i] = c[i] = 0.0;
                if(s < ns[i]) {
                    const xh_permute_source so = src_staged ? s_src[sb[i] + s - s_first] : p.src[sb[i] + s];
                    c[i] = so.coeff;
                    v[i] = src[so.src_off + srow[i] + int64_t(scol[i]) * so.src_ld];
                }
            }
#pragma unroll
            for(int i = 0; i < PER; ++i)
                if(s < ns[i]) val[i] = __dadd_rn(val[i], __dmul_rn(c[i], v[i]));
        }
    }
#pragma unroll
    for(int i = 0; i < PER; ++i)
        if(dpos[i] >= 0) dst[dpos[i]] = val[i];
}

// Gather of plans that compact tasks cannot hold (a source index or stride of 2^31 and more): every
// leg of an element decoded from the task's records in global memory.
template <bool SINGLE_SRC>
__global__ __launch_bounds__(PT_THREADS) void k_permute_gather(PermDev p, const double* __restrict__ src, double* __restrict__ dst)
{
    constexpr int PER = PT_TILE / PT_THREADS;
    const int64_t e0 = int64_t(blockIdx.x) * PT_TILE;
    const int n_here = static_cast<int>(min(int64_t(PT_TILE), p.total - e0));
    const int t_lo = p.tile_first[blockIdx.x], t_hi = p.tile_first[blockIdx.x + 1];
    int64_t soff[PER], dpos[PER];
    double coef[PER], val[PER];
#pragma unroll
    for(int i = 0; i < PER; ++i) {
        const int r = threadIdx.x + i * PT_THREADS;
        dpos[i] = -1;
        soff[i] = 0;
        coef[i] = 0.0;
        val[i] = 0.0;
        if(r < n_here) {
            int lo = t_lo, hi = t_hi;  // last task that starts at or before the element
            while(lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if(p.prefix[mid] <= e0 + r)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            const TaskMeta tm = p.meta[lo];
            uint32_t row, col;
            split_el(tm, static_cast<uint32_t>(e0 + r - p.prefix[lo]), row, col);
            int64_t srow, scol;
            dpos[i] = tm.dst_off + row + int64_t(col) * tm.dst_ld;
            decode_src(p.legs + int64_t(lo) * p.nlegs, p.nlegs, p.new_rank, row, col, srow, scol);
            if constexpr(SINGLE_SRC) {
                const xh_permute_source so = p.src[tm.src_begin];
                soff[i] = so.src_off + srow + scol * so.src_ld;
                coef[i] = so.coeff;
            } else {
                val[i] = gather_one(p, tm, src, srow, scol);
            }
        }
    }
    if constexpr(SINGLE_SRC) {
        // inactive elements load src[0]: a single-source plan reads at least one source element
#pragma unroll
        for(int i = 0; i < PER; ++i) val[i] = src[soff[i]];
#pragma unroll
        for(int i = 0; i < PER; ++i) val[i] = __dadd_rn(0.0, __dmul_rn(coef[i], val[i]));
    }
#pragma unroll
    for(int i = 0; i < PER; ++i)
        if(dpos[i] >= 0) dst[dpos[i]] = val[i];
}

// Transpose path.  For a task whose output leg 0 is not the unit-stride source leg, let leg u be
// the output leg that reads source stride 1.  A tile covers TR_DIM values of output leg 0 (the
// contiguous direction of the output) times TR_DIM values of leg u (the contiguous direction of
// the source) at one fixed value of every other leg.  Loads run along leg u, stores along leg 0.
struct TrTaskInfo {
    int32_t task, u;  // task id and the output leg with unit source stride
    uint32_t ext0, extu;
    int64_t rest;  // number of combinations of the remaining legs
};

__global__ __launch_bounds__(PT_THREADS) void k_permute_transpose(PermDev p, const TrTaskInfo* __restrict__ info, const double* __restrict__ src,
                                                                  double* __restrict__ dst)
{
    __shared__ double tile[TR_DIM][TR_DIM + 1];
    const int4 tt = p.tr_tiles[blockIdx.x];
    const TrTaskInfo ti = info[tt.x];
    const int t = ti.task;
    const TaskMeta tm = p.meta[t];
    const LegInfo* L = p.legs + int64_t(t) * p.nlegs;
    const int u = ti.u;
    const uint32_t i0 = uint32_t(tt.z) * TR_DIM;  // along output leg 0
    const uint32_t iu = uint32_t(tt.y) * TR_DIM;  // along output leg u
    // Decode the fixed remaining-leg index (every leg except 0 and u) into base offsets.
    uint32_t rest = uint32_t(tt.w);
    int64_t base_srow = 0, base_scol = 0;
    // output position contributions of the remaining legs: row (domain legs) and col (codomain legs)
    int64_t base_row = 0, base_col = 0;
    int64_t rmul = 1, cmul = 1;
    for(int k = 0; k < p.nlegs; ++k) {
        const LegInfo li = L[k];
        const bool is_row = k < p.new_rank;
        int64_t mult = is_row ? rmul : cmul;
        if(k != 0 && k != u) {
            uint32_t q = xh::fdiv(rest, li.magic, leg_shift(li));
            uint32_t j = rest - q * li.ext;
            rest = q;
            base_srow += int64_t(j) * leg_rstride(li);
            base_scol += int64_t(j) * leg_cstride(li);
            if(is_row)
                base_row += int64_t(j) * mult;
            else
                base_col += int64_t(j) * mult;
        }
        if(is_row)
            rmul *= li.ext;
        else
            cmul *= li.ext;
    }
    // output multiplier of leg u
    int64_t umul = 1;
    {
        const bool urow = u < p.new_rank;
        int64_t m = 1;
        for(int k = urow ? 0 : p.new_rank; k < u; ++k) m *= L[k].ext;
        umul = m;
    }
    const bool urow = u < p.new_rank;
    const LegInfo l0 = L[0];
    const LegInfo lu = L[u];
    const int tx = threadIdx.x & 63;
    const int ty = threadIdx.x >> 6;  // 0..3
    // load: rows of the tile indexed by leg-0 value a, columns by leg-u value b; b runs along lanes
    for(int a = ty; a < TR_DIM; a += 4) {
        const uint32_t j0 = i0 + a, ju = iu + tx;
        double v = 0.0;
        if(j0 < ti.ext0 && ju < ti.extu) {
            const int64_t srow = base_srow + int64_t(j0) * leg_rstride(l0) + int64_t(ju) * leg_rstride(lu);
            const int64_t scol = base_scol + int64_t(j0) * leg_cstride(l0) + int64_t(ju) * leg_cstride(lu);
            v = gather_one(p, tm, src, srow, scol);
        }
        tile[a][tx] = v;
    }
    __syncthreads();
    // store: a runs along lanes (output leg 0 is the contiguous output direction)
    for(int b = ty; b < TR_DIM; b += 4) {
        const uint32_t j0 = i0 + tx, ju = iu + b;
        if(j0 < ti.ext0 && ju < ti.extu) {
            int64_t row = base_row + j0;  // leg 0 is a domain leg with multiplier 1 (new_rank >= 1 here)
            int64_t col = base_col;
            if(urow)
                row += int64_t(ju) * umul;
            else
                col += int64_t(ju) * umul;
            dst[tm.dst_off + row + col * tm.dst_ld] = tile[tx][b];
        }
    }
}

}  // namespace

struct xh_permute_plan : xh::PlanLife {
    PermDev dev{};
    PermC cdev{};          // gather tasks of a compact plan (dev then holds the transpose tasks alone)
    bool compact = false;
    int per = 4;           // output elements per thread of the compact gather
    xh::PackedUpload up;
    int64_t ngather_tiles = 0;
    bool single_src = true;  // every gather task has exactly one source
    double bytes = 0.0;
    const TrTaskInfo* trinfo = nullptr;
};

extern "C" int xh_permute_plan_create(xh_ctx* ctx, const xh_permute_desc* desc, xh_permute_plan** out)
{
    *out = nullptr;
    auto* plan = new xh_permute_plan();
    int rc = guard(ctx, [&] {
        xh::refuse_under_capture(ctx, "plan creation");
        const int NL = desc->nlegs;
        if(NL < 0 || NL > XH_MAXLEGS) throw xh::Error(XH_EINVAL, "permute plan: too many legs");
        if(desc->new_rank < 0 || desc->new_rank > NL) throw xh::Error(XH_EINVAL, "permute plan: invalid new_rank");
        const int64_t NT = desc->ntasks;
        if(NT < 0 || NT > 0x7fffffff || desc->nsources < 0) throw xh::Error(XH_EINVAL, "permute plan: invalid task or source count");
        // pass 1: validate every task and pick its kernel (-1: gather, u > 0: transpose via leg u),
        // in chunks on the host worker pool for large plans; slot and tile0 are first numbered
        // within the chunk and shifted by the chunk's base once all chunks are counted
        std::vector<int32_t> route(static_cast<size_t>(NT));
        std::vector<int64_t> slot(static_cast<size_t>(NT)), tile0(static_cast<size_t>(NT), 0);  // table row; first transpose tile
        struct ChunkCount {
            int64_t ngather = 0, ntr = 0, ntr_tiles = 0, total = 0;
            double moved = 0.0, read = 0.0;
            bool single = true;
            bool ordered = true;   // source ranges follow one another
            bool near = true;      // source indices of every gather task below 2^31
            int nl1 = 0, nl2 = 0;  // most joined legs of a gather task, with absolute strides and with row / column strides
        };
        // The legs of a task joined (LegC): absolute source strides (abs: one source, its leading
        // dimension folded in), or source row and column strides.  Leg q joins the one before it (of extent >
        // 1) if it goes on where that one ends, so that no leg waits for the products of earlier ones, and
        // there are no branches, which would be guessed wrong for about every leg.  Pass 1 keeps a bit for
        // each leg that starts a joined one, pass 2 visits these alone.
        struct LegJoin {
            int64_t end = 0;       // where the leg before ends
            uint32_t heads = 0;    // legs that start a joined leg
            bool col = false;      // kind of the leg before
            bool far = false;      // a stride of 2^31 or more
            void add(int q, uint32_t e, int64_t st, bool c)
            {
                const bool one = e == 1, head = !one & ((heads == 0) | (st != end) | (c != col));
                heads |= uint32_t(head) << q;
                far |= head & (uint64_t(st) >= (uint64_t(1) << 31));
                end = one ? end : st * e;
                col = one ? col : c;
            }
        };
        std::vector<uint32_t> heads(static_cast<size_t>(NT));
        // largest source row and column of a task with row and column strides
        auto far_reach = [NL](const xh_permute_task& tk) {
            int64_t reach[2] = {0, 0};
            for(int q = 0; q < NL; ++q) reach[tk.is_col[q] != 0] += (int64_t(tk.ext[q]) - 1) * tk.sstride[q];
            return std::max(reach[0], reach[1]) >= (int64_t(1) << 31);
        };
        // on several host threads from 16384 tasks on: they sleep between plans, and waking them for a few
        // thousand tasks takes longer than it gains (first permute of a seven-leg tensor with some 6000
        // tasks: 1428 us with threads from 2048 tasks on, 820 so)
        const size_t nchunk = NT >= 16384 ? std::max<size_t>(1, std::min<size_t>(xp::WorkerPool::get().size(), size_t(NT) / 4096)) : 1;
        std::vector<ChunkCount> cc(nchunk);
        auto chunk_lo = [&](size_t c) { return int64_t(size_t(NT) * c / nchunk); };
        auto classify = [&](size_t c) {
            ChunkCount& k = cc[c];
            for(int64_t t = chunk_lo(c); t < chunk_lo(c + 1); ++t) {
                const xh_permute_task& tk = desc->tasks[t];
                // a record is 304 bytes, read in parts, and often written by another thread
                const char* ahead = reinterpret_cast<const char*>(desc->tasks + std::min(t + 6, chunk_lo(c + 1) - 1));
                __builtin_prefetch(ahead);
                __builtin_prefetch(ahead + 64);
                __builtin_prefetch(ahead + offsetof(xh_permute_task, sstride));
                __builtin_prefetch(ahead + offsetof(xh_permute_task, is_col));
                if(tk.rows < 0 || tk.cols < 0 || tk.rows * tk.cols >= (int64_t(1) << 31))
                    throw xh::Error(XH_EINVAL, "permute plan: subblock too large for 32-bit indexing");
                if(tk.nsrc < 0 || tk.src_begin < 0 || tk.src_begin + tk.nsrc > desc->nsources)
                    throw xh::Error(XH_EINVAL, "permute plan: source range out of bounds");
                if(t > 0 && tk.src_begin < desc->tasks[t - 1].src_begin + desc->tasks[t - 1].nsrc) k.ordered = false;
                // one source: most likely of every task, so row and column strides are joined only if they turn
                // out to be needed
                const bool abs = tk.nsrc == 1;
                const int64_t ld = abs ? desc->sources[tk.src_begin].src_ld : 1;
                int64_t rprod = 1, cprod = 1;
                LegJoin join;
                for(int q = 0; q < NL; ++q) {
                    if(tk.ext[q] == 0) throw xh::Error(XH_EINVAL, "permute plan: zero extent");
                    if(tk.sstride[q] < 0 || tk.sstride[q] >= (int64_t(1) << 31)) throw xh::Error(XH_EINVAL, "permute plan: source stride out of range");
                    (q < desc->new_rank ? rprod : cprod) *= tk.ext[q];
                    const bool is_col = tk.is_col[q] != 0;
                    join.add(q, tk.ext[q], is_col ? tk.sstride[q] * ld : tk.sstride[q], !abs & is_col);
                }
                if(rprod != tk.rows || cprod != tk.cols) throw xh::Error(XH_EINVAL, "permute plan: leg extents do not match the subblock shape");
                const double elems = double(tk.rows) * double(tk.cols);
                k.moved += elems;
                k.read += elems * tk.nsrc;
                // transpose path when output leg 0 is a real leg (ext >= 16) whose source stride is
                // not 1 and some other leg with ext >= 16 has unit source stride
                int u = -1;
                if(desc->new_rank >= 1 && NL >= 2 && tk.nsrc >= 1 && tk.sstride[0] != 1 && !tk.is_col[0] && tk.ext[0] >= 16) {
                    for(int q = 1; q < NL; ++q)
                        if(tk.sstride[q] == 1 && !tk.is_col[q] && tk.ext[q] >= 16) {
                            u = q;
                            break;
                        }
                }
                route[t] = u;
                if(u <= 0 && tk.nsrc != 1) k.single = false;
                if(u > 0) {
                    int64_t rest = 1;
                    for(int q = 0; q < NL; ++q)
                        if(q != 0 && q != u) rest *= tk.ext[q];
                    slot[t] = k.ntr;  // offset by ngather below
                    tile0[t] = k.ntr_tiles;
                    k.ntr_tiles += rest * ((tk.ext[0] + TR_DIM - 1) / TR_DIM) * ((tk.ext[u] + TR_DIM - 1) / TR_DIM);
                    ++k.ntr;
                } else {
                    slot[t] = k.ngather;
                    ++k.ngather;
                    k.total += tk.rows * tk.cols;
                    heads[t] = join.heads;
                    int& nl = abs ? k.nl1 : k.nl2;
                    nl = std::max(nl, __builtin_popcount(join.heads));
                    if(join.far || (!abs && far_reach(tk))) k.near = false;
                }
            }
        };
        if(nchunk > 1)
            xp::WorkerPool::get().run(nchunk, classify);
        else
            classify(0);
        std::vector<ChunkCount> base(nchunk);  // per chunk: counts of the chunks before it
        int64_t ngather = 0, ntr = 0, ntr_tiles = 0, total = 0;
        double moved = 0.0, read = 0.0;
        for(size_t c = 0; c < nchunk; ++c) {
            base[c].ngather = ngather;
            base[c].ntr = ntr;
            base[c].ntr_tiles = ntr_tiles;
            base[c].total = total;
            ngather += cc[c].ngather;
            ntr += cc[c].ntr;
            ntr_tiles += cc[c].ntr_tiles;
            total += cc[c].total;
            moved += cc[c].moved;
            read += cc[c].read;
            if(!cc[c].single) plan->single_src = false;
        }
        const bool single = plan->single_src;
        if(!single)  // tasks with one source among tasks with several
            for(int64_t t = 0; t < NT; ++t)
                if(route[t] <= 0 && desc->tasks[t].nsrc == 1) {
                    const xh_permute_task& tk = desc->tasks[t];
                    LegJoin join;
                    for(int q = 0; q < NL; ++q) join.add(q, tk.ext[q], tk.sstride[q], tk.is_col[q] != 0);
                    heads[t] = join.heads;
                    cc[0].nl2 = std::max(cc[0].nl2, __builtin_popcount(join.heads));
                    if(join.far || far_reach(tk)) cc[0].near = false;
                }
        int nl = 0;
        bool ordered = true;
        plan->compact = ngather > 0;
        for(const ChunkCount& k : cc) {
            ordered = ordered && k.ordered;
            if(!k.near) plan->compact = false;
            nl = std::max(nl, single ? k.nl1 : k.nl2);
        }
        const bool compact = plan->compact;
        // small tensors in small tiles: a workgroup's time is then its latency, and more of them run
        // beside one another (37214 elements: 4.1 us in tiles of 512 against 6.0 in tiles of 2048);
        // at 16.8 M elements tiles of 512 take 77 us against 70
        plan->per = total >= int64_t(2) * std::max(ctx->num_cu, 1) * PT_TILE ? 4 : 2;
        const int64_t tile = compact ? int64_t(plan->per) * PT_THREADS : PT_TILE;
        if(ntr_tiles > 0x7fffffff) throw xh::Error(XH_EINVAL, "permute: too many tiles");
        const int64_t ntiles = (total + tile - 1) / tile;
        if(ntiles > 0x7fffffff) throw xh::Error(XH_EINVAL, "permute: too many tiles");
        // pass 2: write the device tables straight into the upload buffer; gather tasks first,
        // then the transpose tasks (their metadata follows the gather metadata)
        const int64_t nc = compact ? ngather : 0, nmeta = ngather + ntr - nc;
        xh::PackedUpload& up = plan->up;
        const size_t bytes = xh::PackedUpload::packed_bytes(
            {size_t(nmeta) * sizeof(TaskMeta), size_t(nmeta * NL) * sizeof(LegInfo), size_t(ngather + 1) * sizeof(int64_t), size_t(ntiles + 1) * sizeof(int32_t),
             size_t(desc->nsources) * sizeof(xh_permute_source), size_t(ntr_tiles) * sizeof(int4), size_t(ntr) * sizeof(TrTaskInfo),
             size_t(nc) * sizeof(TaskC), size_t(nc * nl) * sizeof(LegC)});
        if(bytes >= (size_t(1) << 18)) up.begin_pinned(ctx, bytes);  // large plans: straight into pinned staging
        const size_t o_meta = up.reserve<TaskMeta>(nmeta), o_legs = up.reserve<LegInfo>(nmeta * NL), o_prefix = up.reserve<int64_t>(ngather + 1),
                     o_tiles = up.reserve<int32_t>(ntiles + 1), o_src = up.reserve<xh_permute_source>(desc->nsources),
                     o_tr = up.reserve<int4>(ntr_tiles), o_trinfo = up.reserve<TrTaskInfo>(ntr), o_taskc = up.reserve<TaskC>(nc),
                     o_legc = up.reserve<LegC>(nc * nl);
        TaskMeta* meta = up.host_ptr<TaskMeta>(o_meta);
        LegInfo* legs = up.host_ptr<LegInfo>(o_legs);
        int64_t* prefix = up.host_ptr<int64_t>(o_prefix);
        int32_t* tile_first = up.host_ptr<int32_t>(o_tiles);
        int4* trtiles = up.host_ptr<int4>(o_tr);
        TrTaskInfo* trinfo = up.host_ptr<TrTaskInfo>(o_trinfo);
        TaskC* taskc = up.host_ptr<TaskC>(o_taskc);
        LegC* legc = up.host_ptr<LegC>(o_legc);
        // second pass over the same chunks: final slots and first transpose tiles, the element
        // prefix of the gather tasks (in table order), the first task of every gather tile (the
        // tiles that start inside a task) and the per-task device tables
        auto place = [&](size_t c) {
            int64_t e = base[c].total;
            for(int64_t t = chunk_lo(c); t < chunk_lo(c + 1); ++t) {
                const xh_permute_task& tk = desc->tasks[t];
                const int u = route[t];
                if(u > 0) {
                    slot[t] += base[c].ntr;
                    tile0[t] += base[c].ntr_tiles;
                } else {
                    slot[t] += base[c].ngather;
                    prefix[slot[t]] = e;
                    const int64_t e_end = e + tk.rows * tk.cols;
                    const int64_t i0 = (e + tile - 1) / tile, i1 = (e_end + tile - 1) / tile;
                    if(i0 < i1) std::fill(tile_first + i0, tile_first + i1, static_cast<int32_t>(slot[t]));
                    e = e_end;
                    if(compact) {
                        const xh_permute_source* so = single ? desc->sources + tk.src_begin : nullptr;
                        const xh::FastDiv fd = xh::make_fastdiv(uint32_t(std::max<int64_t>(tk.rows, 1)));
                        LegC* L = legc + slot[t] * nl;
                        int n = 0;
                        for(uint32_t m = heads[t]; m; ++n) {  // joined legs: from a head to the next, past legs of extent 1
                            const int q = __builtin_ctz(m);
                            m &= m - 1;
                            uint32_t ext = tk.ext[q];
                            for(int k = q + 1, next = m ? __builtin_ctz(m) : NL; k < next; ++k) ext *= tk.ext[k];
                            const bool is_col = tk.is_col[q] != 0;
                            const xh::FastDiv d = xh::make_fastdiv(ext);
                            L[n] = LegC{ext, d.magic, d.shift | (!so && is_col ? 256u : 0u), static_cast<uint32_t>(so && is_col ? tk.sstride[q] * so->src_ld : tk.sstride[q])};
                        }
                        for(int k = n; k < nl; ++k) L[k] = LegC{1, 1, 0, 0};
                        taskc[slot[t]] = TaskC{tk.dst_off, tk.dst_ld, so ? so->src_off : 0, so ? so->coeff : 0.0, uint32_t(tk.rows), fd.magic, fd.shift, uint32_t(n),
                                               tk.nsrc, tk.src_begin};
                        continue;
                    }
                }
                const int64_t idx = u > 0 ? ngather - nc + slot[t] : slot[t];
                const xh::FastDiv fd = xh::make_fastdiv(uint32_t(std::max<int64_t>(tk.rows, 1)));
                meta[idx] = TaskMeta{tk.dst_off, tk.dst_ld, uint32_t(tk.rows), fd.magic, fd.shift, 0, tk.nsrc, tk.src_begin};
                LegInfo* L = legs + idx * NL;
                for(int k = 0; k < NL; ++k) L[k] = xh::make_leg(tk.ext[k], tk.sstride[k], tk.is_col[k] != 0);
                if(u > 0) {
                    int64_t rest = 1;
                    for(int k = 0; k < NL; ++k)
                        if(k != 0 && k != u) rest *= tk.ext[k];
                    const int64_t ti = slot[t];
                    trinfo[ti] = TrTaskInfo{static_cast<int32_t>(idx), u, tk.ext[0], tk.ext[u], rest};
                    const int n0 = (tk.ext[0] + TR_DIM - 1) / TR_DIM, nu = (tk.ext[u] + TR_DIM - 1) / TR_DIM;
                    int64_t tt = tile0[t];
                    for(int64_t r = 0; r < rest; ++r)
                        for(int a = 0; a < n0; ++a)
                            for(int b = 0; b < nu; ++b) trtiles[tt++] = int4{static_cast<int>(ti), b, a, static_cast<int>(r)};
                }
            }
        };
        if(nchunk > 1)
            xp::WorkerPool::get().run(nchunk, place);
        else
            place(0);
        prefix[ngather] = total;
        tile_first[ntiles] = static_cast<int32_t>(ngather > 0 ? ngather - 1 : 0);  // sentinel: the last gather task
        if(desc->nsources > 0)
            std::memcpy(up.host_ptr<xh_permute_source>(o_src), desc->sources, size_t(desc->nsources) * sizeof(xh_permute_source));
        plan->dev.nlegs = NL;
        plan->dev.new_rank = desc->new_rank;
        plan->dev.ntasks = nmeta;
        plan->dev.total = total;
        up.upload(ctx);
        plan->dev.meta = up.ptr<const TaskMeta>(o_meta);
        plan->dev.legs = up.ptr<const LegInfo>(o_legs);
        plan->dev.prefix = up.ptr<const int64_t>(o_prefix);
        plan->dev.tile_first = up.ptr<const int32_t>(o_tiles);
        plan->dev.src = up.ptr<const xh_permute_source>(o_src);
        plan->dev.ntr_tiles = ntr_tiles;
        plan->dev.tr_tiles = up.ptr<const int4>(o_tr);
        plan->trinfo = up.ptr<const TrTaskInfo>(o_trinfo);
        plan->ngather_tiles = ntiles;
        plan->cdev = PermC{nl, ordered ? 1 : 0, total, up.ptr<const TaskC>(o_taskc), up.ptr<const LegC>(o_legc), plan->dev.prefix, plan->dev.tile_first, plan->dev.src};
        plan->bytes = 8.0 * (moved + read);
    });
    if(rc != XH_OK) {
        xh_permute_plan_destroy(ctx, plan);
        return rc;
    }
    *out = plan;
    return XH_OK;
}

namespace {
void permute_plan_release(xh_ctx* ctx, xh::PlanLife* p)
{
    auto* plan = static_cast<xh_permute_plan*>(p);
    plan->up.release(ctx);
    delete plan;
}
}  // namespace

extern "C" int xh_permute_plan_destroy(xh_ctx* ctx, xh_permute_plan* plan)
{
    if(!plan) return XH_OK;
    return guard(ctx, [&] {
        if(plan->pins > 0) {
            plan->dead = true;  // a live graph reads its tables: freed by the last xh_graph_destroy
            return;
        }
        permute_plan_release(ctx, plan);
    });
}

extern "C" int xh_permute_plan_bytes(const xh_permute_plan* plan, double* bytes)
{
    if(!plan || !bytes) return XH_EINVAL;
    *bytes = plan->bytes;
    return XH_OK;
}

namespace {
void launch_gather(xh_ctx* ctx, const xh_permute_plan* plan, const double* src, double* dst)
{
    const dim3 grid(static_cast<unsigned>(plan->ngather_tiles)), block(PT_THREADS);
    if(plan->compact) {
        auto* kern = plan->single_src ? (plan->per == 4 ? k_permute_compact<true, 4> : k_permute_compact<true, 2>)
                                      : (plan->per == 4 ? k_permute_compact<false, 4> : k_permute_compact<false, 2>);
        hipLaunchKernelGGL(kern, grid, block, 0, ctx->stream, plan->cdev, src, dst);
    } else {
        auto* kern = plan->single_src ? k_permute_gather<true> : k_permute_gather<false>;
        hipLaunchKernelGGL(kern, grid, block, 0, ctx->stream, plan->dev, src, dst);
    }
}
}  // namespace

extern "C" int xh_permute(xh_ctx* ctx, const xh_permute_plan* plan, const double* src, double* dst)
{
    return guard(ctx, [&] {
        if(!plan) throw xh::Error(XH_EINVAL, "null permute plan");
        if(plan->dead) throw xh::Error(XH_EINVAL, "permute plan used after xh_permute_plan_destroy");
        xh::pin_for_capture(ctx, const_cast<xh_permute_plan*>(plan), permute_plan_release);
        const bool timed = ctx->perm_timing && (plan->ngather_tiles > 0 || plan->dev.ntr_tiles > 0);
        if(timed) xh::perm_timer_begin(ctx);
        if(plan->ngather_tiles > 0) {
            if(plan->ngather_tiles > 0x7fffffff) throw xh::Error(XH_EINVAL, "permute: too many tiles");
            launch_gather(ctx, plan, src, dst);
            xh::launch_check("k_permute_gather");
        }
        if(plan->dev.ntr_tiles > 0) {
            if(plan->dev.ntr_tiles > 0x7fffffff) throw xh::Error(XH_EINVAL, "permute: too many tiles");
            hipLaunchKernelGGL(k_permute_transpose, dim3(static_cast<unsigned>(plan->dev.ntr_tiles)), dim3(PT_THREADS), 0, ctx->stream, plan->dev,
                               plan->trinfo, src, dst);
            xh::launch_check("k_permute_transpose");
        }
        if(timed) xh::perm_timer_end(ctx, plan->bytes);
    });
}
