// mi_rows.hip -- power-iteration step of levels without long rows: one launch
// per iteration (eigensolve_kokkos.h:102-206, with the vector helpers of
// :14-58 and the product KokkosSparse::spmv), under the plain Laplacian (the
// normalised one keeps the streaming step's order of sums, see k_power_small).
//
// The streaming step (mi_eigen.hip) sums flat ranges of entries, whatever the
// rows look like, and so takes a second kernel that joins the pieces of rows,
// a row id per entry and a scan over the lanes per 512 entries.  Where every
// row is short, one lane sums a row whole, and the kernel that has the row's
// sum forms y and the sums of y right away.
//
// Layout: 64 rows, one per lane, are a slice; the entries of a slice lie group
// by group, GROUP consecutive entries of each lane's row in one 16-byte load
// of columns (sliced ELLPACK with sorting windows: SELL-C-sigma, Kreutzer et
// al., SIAM J. Sci. Comput. 36, 2014).  Rows are taken in windows of WIN, sorted
// by their number of groups, so that the rows of a slice have about the same
// number and padding stays small, while the vector values they touch stay
// within the window's lines.  Padding entries have weight 0 and the column n,
// where the vectors hold a zero.
//
// The deflation and normalisation of an iteration are never written back (as
// in the streaming step): the next one reads its input as x = (y - a) s.  Here
// the gathers read y as it is, and A x = s (A y - a wdeg), so that the first
// slice is summed before a and s are known: the previous launch's sums arrive
// meanwhile.  Sums per launch: S1 = sum y, S2 = sum y^2, S3 = sum x y, taken
// over y before it is rounded to the vector's type; with FP32 vectors a
// fourth, sum x^2, normalises the dot product.  Every sum has a fixed order:
// results are bit-identical run to run.
#include "mi_kernels.hpp"

#include <algorithm>
#include <cmath>

namespace mi {

namespace {

constexpr int NW = BLOCK / WAVE;         // wavefronts per workgroup
constexpr int GROUP = 4;                 // entries of a row that a lane loads together
constexpr uint32_t WIN = 2048;           // rows per sorting window
constexpr uint32_t WSL = WIN / WAVE;     // its slices
constexpr int SBLOCK = 1024;             // workgroup that sorts a window: a thread per compared pair
constexpr uint32_t SLICE_COST = 2;       // cost of a slice besides its groups, in groups (spans)
constexpr uint32_t MAXF = 1024;          // workgroups whose sums an iteration adds, at most
constexpr int NSUM = 4;                  // sums per workgroup (the last with FP32 vectors only)
template <class V>
constexpr int sums_of = sizeof(V) == 4 ? 4 : 3;
constexpr int W_UNIT = 0, W_U16 = 1, W_U32 = 2;  // weight formats

inline unsigned grid1(uint64_t n) { return (unsigned)ceil_div(n ? n : 1, BLOCK); }

// longest row and largest weight: out[0], out[1] (zeroed before).  A workgroup
// that meets a row past SHORT_ROW, which decides the matter, leaves the weights
// (a product with its plan on R-MAT-20, edge factor 6: 0.81 ms, 0.76 ms so).
__global__ void __launch_bounds__(BLOCK) k_extremes(uint32_t n, uint64_t m, const uint32_t* __restrict__ rowptr,
                                                    const uint32_t* __restrict__ w, uint32_t* __restrict__ out)
{
    __shared__ uint32_t lds[BLOCK / WAVE];
    const uint64_t t = (uint64_t)blockIdx.x * BLOCK + threadIdx.x, step = (uint64_t)gridDim.x * BLOCK;
    uint32_t len = 0, wm = 0;
    for (uint64_t r = t; r < n; r += step) {
        const uint32_t d = rowptr[r + 1] - rowptr[r];
        len = d > len ? d : len;
    }
    len = block_max_u32(len, lds);
    if (w && len <= SHORT_ROW)
        for (uint64_t e = t; e < m; e += step) wm = w[e] > wm ? w[e] : wm;
    wm = block_max_u32(wm, lds);
    if (threadIdx.x == 0) {
        if (len) atomicMax(&out[0], len);
        if (wm) atomicMax(&out[1], wm);
    }
}

// One workgroup per window of rows: by descending number of groups (equal ones
// in order); order[WIN window + j] = the j-th row (INF: none), sgroups[slice] =
// groups of the slice's longest.
__global__ void __launch_bounds__(SBLOCK) k_window_sort(uint32_t n, const uint32_t* __restrict__ rowptr,
                                                        uint32_t* __restrict__ order, uint32_t* __restrict__ sgroups)
{
    __shared__ uint32_t key[WIN];
    const uint32_t w = blockIdx.x, tid = threadIdx.x, r0 = w * WIN;
    const uint32_t cnt = n - r0 < WIN ? n - r0 : WIN;
    for (uint32_t j = tid; j < WIN; j += SBLOCK) {
        uint32_t k = INF;
        if (j < cnt) {
            const uint32_t len = rowptr[r0 + j + 1] - rowptr[r0 + j];
            k = (255u - (len + GROUP - 1) / GROUP) << 16 | j;  // (at most SHORT_ROW / GROUP = 32 groups)
        }
        key[j] = k;
    }
    __syncthreads();
    for (uint32_t k = 2; k <= WIN; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            const uint32_t t = tid, i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), p = i | j;
            const uint32_t u = key[i], v = key[p];
            if ((u > v) == ((i & k) == 0)) {
                key[i] = v;
                key[p] = u;
            }
            // (pairs at most 64 apart lie in the 128 elements of one wavefront)
            if (j > WAVE || (j == 1 && k > WAVE))
                __syncthreads();
            else
                wave_fence();
        }
    }
    __syncthreads();
    for (uint32_t j = tid; j < WIN; j += SBLOCK) {
        const uint32_t k = key[j];
        order[(size_t)w * WIN + j] = k == INF ? INF : r0 + (k & 0xffffu);
        if (j % WAVE == 0) sgroups[w * WSL + j / WAVE] = k == INF ? 0u : 255u - (k >> 16);
    }
}

// GROUP consecutive words; they lie at a word's alignment only
struct __attribute__((packed, aligned(4))) Words {
    uint32_t x[GROUP];
};

// The entries of every slice, one wavefront per slice; past a row's end the
// column n with weight 0.
template <class WT>
__global__ void __launch_bounds__(BLOCK) k_fill(uint32_t n, uint32_t nslices, const uint32_t* __restrict__ soff,
                                                const uint32_t* __restrict__ order,
                                                const uint32_t* __restrict__ rowptr,
                                                const uint32_t* __restrict__ col, const uint32_t* __restrict__ w,
                                                uint32_t* __restrict__ out, WT* __restrict__ wout)
{
    const uint32_t s = uniform((blockIdx.x * BLOCK + threadIdx.x) / WAVE), lane = threadIdx.x & (WAVE - 1);
    if (s >= nslices) return;
    const uint32_t g0 = soff[s], ng = soff[s + 1] - g0;
    const uint32_t r = order[(size_t)s * WAVE + lane];
    uint32_t e0 = 0, len = 0;
    if (r != INF) {
        e0 = rowptr[r];
        len = rowptr[r + 1] - e0;
    }
    for (uint32_t g = 0; g < ng; g++) {
        const size_t at = ((size_t)(g0 + g) * WAVE + lane) * GROUP;
        const uint32_t k0 = g * GROUP;
        Words cs, ws = {};
        if (k0 + GROUP <= len) {
            cs = *reinterpret_cast<const Words*>(col + e0 + k0);
            if (w) ws = *reinterpret_cast<const Words*>(w + e0 + k0);
        } else {
#pragma unroll
            for (int u = 0; u < GROUP; u++) {
                const bool in = k0 + u < len;
                cs.x[u] = in ? col[e0 + k0 + u] : n;
                ws.x[u] = in && w ? w[e0 + k0 + u] : 0u;
            }
        }
        *reinterpret_cast<uint4*>(out + at) = make_uint4(cs.x[0], cs.x[1], cs.x[2], cs.x[3]);
        if (!w) continue;
        if (sizeof(WT) == 2)
            *reinterpret_cast<uint2*>(wout + at) = make_uint2(ws.x[0] | ws.x[1] << 16, ws.x[2] | ws.x[3] << 16);
        else
            *reinterpret_cast<uint4*>(wout + at) = make_uint4(ws.x[0], ws.x[1], ws.x[2], ws.x[3]);
    }
}

// span[k] = the first slice whose cost, the groups and SLICE_COST per slice
// before it, reaches k / parts of the whole, k = 0 .. parts
__global__ void k_spans(uint32_t nslices, const uint32_t* __restrict__ soff, uint32_t parts,
                        uint32_t* __restrict__ span)
{
    const uint32_t k = blockIdx.x * BLOCK + threadIdx.x;
    if (k > parts) return;
    const uint64_t all = (uint64_t)soff[nslices] + (uint64_t)SLICE_COST * nslices;
    const uint64_t want = (all * k + parts - 1) / parts;
    uint32_t lo = 0, hi = nslices;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if ((uint64_t)soff[mid] + (uint64_t)SLICE_COST * mid < want)
            lo = mid + 1;
        else
            hi = mid;
    }
    span[k] = lo;
}

// ------------------------------------------------------------------ step
// Input transform of this iteration from the previous one's sums, and
// the convergence decision for the previous iteration (eigensolve_kokkos.h:
// 155-189).  Every workgroup computes the same values in the same order;
// workgroup 0 records them.  Returns false when the loop has ended, in every
// wavefront of a workgroup alike: the flag of an end found before is read once
// per workgroup, since workgroup 0 of this launch may set it meanwhile.
template <int NS>
__device__ __forceinline__ bool iteration_start(const RowStep& A, double& a, double& s)
{
    a = 0.0;
    s = 1.0;
    if (A.mode != 0) return true;
    __shared__ uint32_t ended;
    __shared__ double lds[NS][NW];
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    const uint32_t iter = A.cnt[A.itr] + 1u;  // 1-based index of this launch
    const uint32_t lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
    if (threadIdx.x == 0) ended = A.cnt[CT_DONE];
    double v[NS] = {}, T[NS];
#pragma unroll
    for (uint32_t j = 0; j < MAXF / BLOCK; j++) {
        const uint32_t b = threadIdx.x + j * BLOCK;
        if (b < A.nblk)
#pragma unroll
            for (int k = 0; k < NS; k++) v[k] += A.fprev[(size_t)b * NSUM + k];
    }
#pragma unroll
    for (int k = 0; k < NS; k++) {
        v[k] = wave_sum(v[k]);
        if (lane == 0) lds[k][wid] = v[k];
    }
    __syncthreads();
    if (ended) return false;
    if (iter < 2) {
        if (lead) {
            A.scal[SC_A] = 0.0;
            A.scal[SC_S] = 1.0;
        }
        return true;
    }
#pragma unroll
    for (int k = 0; k < NS; k++) {
        double t = 0.0;
#pragma unroll
        for (int j = 0; j < NW; j++) t += lds[k][j];
        T[k] = t;
    }
    const double mult = T[0] * A.c;  // dot(v, vec1)
    const double an = mult * A.c;    // subtracted from every entry
    const double nrm2 = T[1] - 2.0 * an * T[0] + an * an * (double)A.n;
    const double sn = 1 / sqrt(nrm2);
    double dot = T[2] * sn;
    if (NS == 4) dot /= sqrt(T[NS - 1]);
    const unsigned long long itn = iter - 1;                  // iterations done
    const double lastd = A.scal[SC_DOT + (iter & 1u)];         // dot of iteration iter - 2
    const bool go_on = (fabs(dot - lastd) > A.tol) && (itn < A.iter_max);
    if (lead) {
        A.scal[SC_DOT + ((iter - 1) & 1u)] = dot;
        if (go_on) {
            A.scal[SC_A] = an;
            A.scal[SC_S] = sn;
        } else {
            A.cnt[CT_DONE] = 1u;
            A.cnt[CT_MAXR] = itn >= A.iter_max ? 1u : 0u;
            *A.niter = itn;
            if (A.hdone) __hip_atomic_store(A.hdone, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    a = an;
    s = sn;
    return go_on;
}

__device__ __forceinline__ double fma_v(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float fma_v(float a, float b, float c) { return fmaf(a, b, c); }

// One lane's group as loaded.
struct Group {
    uint4 c, w;
};

template <int WF>
__device__ __forceinline__ void load_group(const RowStep& A, size_t group, Group& q)
{
    const size_t at = (group * WAVE + (threadIdx.x & (WAVE - 1))) * GROUP;
    q.c = *reinterpret_cast<const uint4*>(A.col + at);
    if (WF == W_U16) {
        const uint2 v = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(A.w) + at);
        q.w.x = v.x;
        q.w.y = v.y;
    }
    if (WF == W_U32) q.w = *reinterpret_cast<const uint4*>(static_cast<const uint32_t*>(A.w) + at);
}

__device__ __forceinline__ uint32_t word_of(const uint4& v, int u)
{
    return u == 0 ? v.x : u == 1 ? v.y : u == 2 ? v.z : v.w;
}

// weight u of a loaded group (unpacked here: a shift at the load would wait for it)
template <int WF>
__device__ __forceinline__ uint32_t weight_of(const Group& q, int u)
{
    if (WF != W_U16) return word_of(q.w, u);
    const uint32_t x = u < 2 ? q.w.x : q.w.y;
    return u & 1 ? x >> 16 : x & 0xffffu;
}

// A word that no kernel writes while this one runs, at a uniform address: a
// scalar load, which does not queue behind the wavefront's vector loads.
__device__ __forceinline__ uint32_t scalar_word(const uint32_t* p)
{
    using Const = const __attribute__((address_space(4))) uint32_t*;
    return uniform(*(Const)(uintptr_t)p);
}

// One row: y from z = A y_prev (the shifted product of the reference), stored,
// and its terms of the sums.
template <class V>
__device__ __forceinline__ void emit_row(const RowStep& A, uint32_t r, V z, V yr, uint32_t wd, uint32_t gb, double a,
                                         double s, double (&S)[sums_of<V>])
{
    const double x = ((double)yr - a) * s;
    const double ax = s * ((double)z - a * (double)wd);
    if (A.ax) A.ax[r] = ax;  // the last one written is A u of the returned u
    const double y = fma((double)(uint32_t)(gb - wd), x, ax);
    static_cast<V*>(A.ynew)[r] = (V)y;
    S[0] += y;
    S[1] = fma(y, y, S[1]);
    S[2] = fma(x, y, S[2]);
    if (sums_of<V> == 4) S[sums_of<V> - 1] = fma(x, x, S[sums_of<V> - 1]);
}

template <int NS>
__device__ __forceinline__ void leave_sums(const RowStep& A, const double (&S)[NS])
{
    if (A.mode != 0) return;
    __shared__ double red[NS][NW];
    double tot[NS];
    block_sum_k<NS>(S, tot, red);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NS; k++) A.fcur[(size_t)blockIdx.x * NSUM + k] = tot[k];
    }
}

// Bound by memory on large levels and by the chain counter, sums, entries,
// gathers on small ones (the kernel of a level of 8,000 to 20,000 vertices
// takes 4 to 6 us, an iteration with its launch 6.5 at least).  us per
// iteration, the streaming step's two launches before and this one: 3d grid
// 128^3 in FP64 73 and 47 (2.2 TB/s of the layout and vectors; the gathers of
// neighbours a plane away miss L1), its level of 628,115 vertices 44 and 35,
// random geometric graph of 150,000 vertices 37 and 28, 12,882 vertices 15.9
// and 11.4.
// Wavefront k of the logical grid takes the slices span[k] ..
// span[k + 1].  The first slice is summed before a and s are known.
template <int WF, class V>
__global__ void __launch_bounds__(BLOCK) k_power_rows(RowStep A)
{
    const V* yp = static_cast<const V*>(A.yprev);
    const uint32_t lane = threadIdx.x & (WAVE - 1), k = uniform(logical_block() * NW + threadIdx.x / WAVE);
    uint32_t sl = scalar_word(A.span + k);
    const uint32_t end = scalar_word(A.span + k + 1);
    const uint32_t gb = *A.gbp;
    V z = 0, yr = 0;
    uint32_t row = INF, wd = 0;
    auto slice = [&]() {
        row = A.row[(size_t)sl * WAVE + lane];
        const uint32_t g0 = scalar_word(A.soff + sl), g1 = scalar_word(A.soff + sl + 1);
        yr = row != INF ? yp[row] : (V)0;
        wd = row != INF ? A.wdeg[row] : 0u;
        z = 0;
        if (g0 < g1) {
            Group q, nx;
            load_group<WF>(A, g0, nx);
            for (uint32_t g = g0; g < g1; g++) {
                q = nx;
                // (the values are asked for before the next group: loads
                // return in order)
                V yv[GROUP];
#pragma unroll
                for (int u = 0; u < GROUP; u++) yv[u] = yp[word_of(q.c, u)];
                if (g + 1 < g1) load_group<WF>(A, g + 1, nx);
#pragma unroll
                for (int u = 0; u < GROUP; u++) z = WF == W_UNIT ? z + yv[u] : fma_v((V)weight_of<WF>(q, u), yv[u], z);
            }
        }
    };
    if (sl < end) slice();
    double a, s;
    if (!iteration_start<sums_of<V>>(A, a, s)) return;
    double S[sums_of<V>] = {};
    while (sl < end) {
        if (row != INF) emit_row<V>(A, row, z, yr, wd, gb, a, s, S);
        sl++;
        if (sl < end) slice();
    }
    leave_sums<sums_of<V>>(A, S);
    // (the counter that this launch's workgroups read stays as it is)
    if (A.mode == 0 && blockIdx.x == 0 && threadIdx.x == 0) A.cnt[A.itw] = A.cnt[A.itr] + 1u;
}

template <class V>
__global__ void k_pad_copy(uint32_t n, const double* __restrict__ x, V* __restrict__ y)
{
    const uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i <= n) y[i] = i < n ? (V)x[i] : (V)0;
}

template <class V>
void launch(Ctx& c, const RowStep& A)
{
    if (A.wfmt == W_UNIT)
        k_power_rows<W_UNIT, V><<<A.nblk, BLOCK, 0, c.stream>>>(A);
    else if (A.wfmt == W_U16)
        k_power_rows<W_U16, V><<<A.nblk, BLOCK, 0, c.stream>>>(A);
    else
        k_power_rows<W_U32, V><<<A.nblk, BLOCK, 0, c.stream>>>(A);
    MI_HIP(hipGetLastError());
}

}  // namespace

bool plan_rows(Ctx& c, const DGraph& g, RowPlan& p)
{
    const uint32_t n = g.n, m = g.m;
    // (power-law levels of longer rows on average hold some past SHORT_ROW: they
    // are not searched for one, some 15 us.  Regular stencils of 33 to 128
    // entries a row stay with the streaming step that way, though this one is
    // faster on them: 49,729 vertices, 40 entries a row 12.6 us per iteration and
    // 7.1, 60 a row 18.7 and 8.4; 199,809, 60 a row 40 and 19.)
    if (!m || (uint64_t)m > (uint64_t)(SHORT_ROW / 4) * n) return false;
    const uint32_t ncu = c.num_cu > 0 ? (uint32_t)c.num_cu : 256u;
    // longest row, and (at once where that is little to read) largest weight
    uint32_t ext[2] = {0, 0};
    const auto look = [&](bool weights) {
        DBuf<uint32_t> x(&c.pool, 2);
        fill_u32(c, x.get(), 2, 0u);
        const uint64_t work = std::max<uint64_t>(n, weights ? m : 0);
        // (two atomics per workgroup on the same words: few workgroups)
        k_extremes<<<(unsigned)std::min<uint64_t>(ncu, ceil_div(work, 4 * BLOCK)), BLOCK, 0, c.stream>>>(
            n, m, g.R(), weights ? g.W() : nullptr, x.get());
        MI_HIP(hipGetLastError());
        read_words(c, x.get(), ext, 8);
    };
    const bool once = g.unit || m <= (1u << 24);
    look(!g.unit && once);
    if (ext[0] > SHORT_ROW) return false;
    if (!once) look(true);
    p.w16 = !g.unit && ext[1] <= 0xffffu;  // (exact: weights are integers)
    const uint32_t nwin = (uint32_t)ceil_div(n, WIN);
    p.nslices = (uint32_t)ceil_div(n, WAVE);
    DBuf<uint32_t> sg(&c.pool, (uint64_t)nwin * WSL);
    p.row = DBuf<uint32_t>(&c.pool, (uint64_t)nwin * WIN);
    p.soff = DBuf<uint32_t>(&c.pool, (uint64_t)p.nslices + 1);
    k_window_sort<<<nwin, SBLOCK, 0, c.stream>>>(n, g.R(), p.row.get(), sg.get());
    MI_HIP(hipGetLastError());
    scan_exclusive_u32(c, sg.get(), p.soff.get(), p.nslices, p.soff.get() + p.nslices);
    uint32_t groups = 0;
    read_words(c, p.soff.get() + p.nslices, &groups, 4);
    p.slots = (uint64_t)groups * WAVE * GROUP;
    p.col = DBuf<uint32_t>(&c.pool, p.slots);
    if (!g.unit) p.w = DBuf<uint32_t>(&c.pool, p.w16 ? p.slots / 2 : p.slots);
    const unsigned grid = (unsigned)ceil_div((uint64_t)p.nslices * WAVE, BLOCK);
    if (p.w16)
        k_fill<uint16_t><<<grid, BLOCK, 0, c.stream>>>(n, p.nslices, p.soff.get(), p.row.get(), g.R(), g.Cc(), g.W(),
                                                       p.col.get(), reinterpret_cast<uint16_t*>(p.w.get()));
    else
        k_fill<uint32_t><<<grid, BLOCK, 0, c.stream>>>(n, p.nslices, p.soff.get(), p.row.get(), g.R(), g.Cc(),
                                                       g.unit ? nullptr : g.W(), p.col.get(), p.w.get());
    MI_HIP(hipGetLastError());
    // at most MAXF workgroups, whose sums the next launch adds
    p.nblk = (uint32_t)std::min<uint64_t>(MAXF, ceil_div(p.nslices, NW));
    p.fsum = DBuf<double>(&c.pool, 2ull * NSUM * MAXF);
    const uint32_t parts = p.nblk * NW;
    p.span = DBuf<uint32_t>(&c.pool, (uint64_t)parts + 1);
    k_spans<<<grid1((uint64_t)parts + 1), BLOCK, 0, c.stream>>>(p.nslices, p.soff.get(), parts, p.span.get());
    MI_HIP(hipGetLastError());
    p.on = true;
    return true;
}

RowStep rows_step(Ctx& c, const DGraph& g, const RowPlan& p, const uint32_t* wdeg, const uint32_t* gb,
                  const void* yprev, void* ynew, double tol, int mode, int parity)
{
    RowStep A;
    A.n = g.n;
    A.wfmt = g.unit ? W_UNIT : p.w16 ? W_U16 : W_U32;
    A.col = p.col.get();
    A.w = p.w.get();
    A.row = p.row.get();
    A.soff = p.soff.get();
    A.span = p.span.get();
    A.wdeg = wdeg;
    A.gbp = gb;
    A.nblk = p.nblk;
    A.fprev = p.fsum.get() + NSUM * MAXF * (parity ^ 1);
    A.fcur = p.fsum.get() + NSUM * MAXF * parity;
    A.yprev = yprev;
    A.ynew = ynew;
    A.c = 1 / std::sqrt((double)g.n);
    A.tol = tol;
    A.iter_max = 100000000000000ull / (unsigned long long)g.n;
    A.mode = mode;
    A.cnt = c.cnt;
    A.itr = parity ? CT_ITER2 : CT_ITER;
    A.itw = parity ? CT_ITER : CT_ITER2;
    A.scal = c.scal;
    A.niter = c.niter;
    A.hdone = nullptr;
    A.ax = nullptr;
    return A;
}

void launch_rows(Ctx& c, bool f32, const RowStep& A)
{
    if (f32)
        launch<float>(c, A);
    else
        launch<double>(c, A);
}

template <class V>
void pad_copy(Ctx& c, uint32_t n, const double* x, V* out)
{
    k_pad_copy<V><<<grid1((uint64_t)n + 1), BLOCK, 0, c.stream>>>(n, x, out);
    MI_HIP(hipGetLastError());
}
template void pad_copy<double>(Ctx&, uint32_t, const double*, double*);
template void pad_copy<float>(Ctx&, uint32_t, const double*, float*);

}  // namespace mi
