// mi_small.hip -- the FP64 power iterations of consecutive small levels of a
// hierarchy (eigensolve_kokkos.h:102-206, 1493-1558), coarsest first, in one
// workgroup and one launch, under the plain Laplacian (the normalised one keeps
// the order of sums of k_power_small_lds, mi_eigen.hip).
//
// A small level has up to a few thousand rows and takes hundreds of
// iterations, each far shorter than a kernel launch.  What bounds one is the
// instructions its wavefronts issue and the latency of the scalar chain sum
// -> inverse square root -> stop test, which every wavefront runs.  So a level
// lies in the LDS and registers of one workgroup, takes ONE barrier per
// iteration (none when one wavefront holds it).
//
// As in the two-kernel loop, x = (y - a) s is never stored: with
//   z = A y,  A x = s (z - a wdeg)   (A 1 = wdeg, the row sums)
// the gathers read y itself and need not wait for a and s.  An iteration is:
// sums of the previous one -> a, s, stop test; row sums z; y' = (gb - wdeg) x
// + A x; its sums S1 = sum y, S2 = sum y^2, S3 = sum x y.  The two-kernel
// loop's S4 = sum x is 0 but for rounding (x is orthogonal to 1), and enters
// the dot product times a, itself of rounding size: it is left out.
//
// Layout.  Rows are renumbered by descending length.  A row is summed by T
// lanes (T a power of two); 64 / T consecutive rows make a slice, its entries
// stored as L steps of 64 lane words, padded with zero weights (rows of one
// slice have nearly equal lengths, so padding stays small).  Slice s goes to
// wavefront s % (wavefronts), whose slices lie one after another in its
// stream.  An entry is one word, column in the low 13 bits and weight above
// (levels with a weight of 2^19 or more: two words).
//  - Register form (4 and 8 wavefronts): every wavefront's stream fits in
//    registers and is read once per level; T the same for every row, or, when
//    that makes a stream too long, growing with the row length.
//  - Streamed form (4 and 16 wavefronts), for the others (long rows, many
//    entries): T grows with the row length, the stream is read from LDS, or
//    from global memory (L2) when it does not fit there, four steps at a time
//    with the next four in flight.
// Which one a level takes follows from its rows and weights alone; the
// workgroup has 4, 8 or 16 wavefronts by the level's size (waves_of), 16 also
// where the registers of 8 turn out not to hold it.  Every sum has a fixed
// order (the sort key ends in the row id), so results are bit-identical run
// to run, and the same whether a level is solved alone, in a chain or in a
// batch of chains.
#include "mi_kernels.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mi {

namespace {

constexpr uint32_t SMALL_MAX_N = 7168;        // two vectors and the degrees of a level fit in LDS
constexpr uint32_t SMALL_MAX_M = 1u << 18;    // (a row length must fit the sort key's 19 bits)
constexpr uint32_t COL_BITS = 13;             // n <= 7168 < 2^13
constexpr uint32_t COL_MASK = (1u << COL_BITS) - 1u;
constexpr uint32_t LEN_MAX = (1u << (32 - COL_BITS)) - 1u;
// Slices: at most one per row with n <= 1024; above, the rows of T = 1 fill
// n / 64 of them, and rows of T lanes have more than 8 T entries, so theirs
// fill at most m / 8 / 64 = 512, and each of the seven T may add a part one.
constexpr uint32_t MAX_SLICES = 1152;
constexpr uint32_t GROUP = 4;                 // steps per load group

// The workgroup sizes.
template <int NWV>
struct Form;
template <>
struct Form<4> {
    static constexpr uint32_t MAX_N = 1024;
    static constexpr uint32_t STEPS = 64;     // register form: steps per wavefront at most
    static constexpr bool F64W = true;        // ... weights kept as doubles (512 registers per lane)
    static constexpr uint32_t POOL = 48 * 1024;
};
template <>
struct Form<8> {
    static constexpr uint32_t MAX_N = SMALL_MAX_N;
    static constexpr uint32_t STEPS = 128;
    static constexpr bool F64W = false;       // 256 registers: one packed word per step
    // 160 KB less the slice table, the sums and the small words
    static constexpr uint32_t POOL = 160 * 1024 - MAX_SLICES * 8 - 2 * 4 * 16 * 8 - 512;
};
template <>
struct Form<16> {
    static constexpr uint32_t MAX_N = SMALL_MAX_N;
    static constexpr uint32_t STEPS = 0;      // no register form
    static constexpr bool F64W = false;
    // 160 KB less the slice table, the sums and the small words
    static constexpr uint32_t POOL = 160 * 1024 - MAX_SLICES * 8 - 2 * 4 * 16 * 8 - 512;
};

// Lanes per row: 2^t with t the smallest that is at least t0 and leaves at
// most `lcap` steps (64 lanes at most).
struct Split {
    uint32_t t0, lcap;
};

// Largest T (at most 2^tmax) with all rows in one pass over `lanes` lanes.
__device__ __forceinline__ uint32_t one_pass(uint32_t n, uint32_t lanes, uint32_t tmax)
{
    uint32_t t = 0;
    while (t < tmax && (n << (t + 1)) <= lanes) t++;
    return t;
}

__device__ __forceinline__ uint32_t lanes_log2(Split sp, uint32_t deg)
{
    uint32_t t = sp.t0;
    while (t < 6 && (deg + (1u << t) - 1u) >> t > sp.lcap) t++;
    return t;
}

struct SmallLevel {
    uint32_t n, m;
    const uint32_t* rowptr;
    const uint32_t* col;
    const uint32_t* w;      // null: unit weights
    const uint32_t* vcmap;  // this level's vertices -> the previous (coarser) level's; null: none
    unsigned long long iter_max;
};

struct SmallResult {
    unsigned long long iters;
    unsigned long long ticks;
    uint32_t max_reached, done;
    uint32_t to16, pad;  // to16: the registers of eight wavefronts do not hold the level
};

// Where a launch that ran out of its iterations left the loop.
struct SmallState {
    uint32_t level;
    uint32_t iter;  // 1-based index of the next iteration of that level (0: not begun)
    double T[3], dot0, dot1, last_a, last_s;
};

struct SmallJob {
    const SmallLevel* lv;
    SmallResult* res;
    uint32_t nlv, waves;
    const double* start;
    const SmallResult* after;  // the last level of the chain that computes `start` (null: none)
    double* v[2];   // the vector of level k of the chain goes to v[k & 1]
    double* y[2];   // both y vectors, between launches
    uint32_t* ord;  // row of each position
    uint32_t* deg;  // weighted degrees by position
    uint32_t* ent;  // the matrix when it is not kept in LDS
    SmallState* st;
};

// One level's layout.
struct Layout {
    double* y;         // two vectors, `span` apart
    uint32_t* wd;      // weighted degrees by position
    uint32_t* ent_l;   // the matrix in LDS (streamed form)
    uint2* slice;      // first position | (rows - 1) << 13 | log2 T << 19, and L
    double* red;       // the wavefronts' sums, of two iterations
    uint32_t* words;   // small words: class sizes, [16..32) steps per wavefront, [64..) reductions
    uint32_t n, span, nslices, gb;
    uint32_t wstep;    // wavefronts that hold the level
    uint32_t base, steps, total;  // this wavefront's first step and steps; all steps
    uint32_t t;        // log2 T when it is the same for every row (uni)
    bool regs, uni, in_lds, wide;
};

template <int CTRL>
__device__ __forceinline__ double dpp_move_f64(double v)
{
    const unsigned long long b = __double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ double readlane_d(double v, int lane)
{
    const unsigned long long b = __double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Sum over aligned groups of 2^t lanes, in every lane of the group (t
// uniform): exchanges inside quads, then mirrored halves, whose lanes hold
// equal sums, then the rows of 16.
__device__ __forceinline__ double group_sum(double z, uint32_t t)
{
    if (t >= 1) z += dpp_move_f64<0xB1>(z);   // quad_perm 1,0,3,2
    if (t >= 2) z += dpp_move_f64<0x4E>(z);   // quad_perm 2,3,0,1
    if (t >= 3) z += dpp_move_f64<0x141>(z);  // row_half_mirror
    if (t >= 4) z += dpp_move_f64<0x140>(z);  // row_mirror
    if (t >= 5) z += __shfl_xor(z, 16, WAVE);
    if (t >= 6) z += __shfl_xor(z, 32, WAVE);
    return z;
}

// Max / sum over the workgroup, in every thread.
template <int NWV>
__device__ __forceinline__ uint32_t max_all(uint32_t v, uint32_t* lds)
{
    v = wave_max_u32(v);
    __syncthreads();
    if ((threadIdx.x & (WAVE - 1)) == 0) lds[threadIdx.x / WAVE] = v;
    __syncthreads();
    uint32_t m = 0;
    for (int k = 0; k < NWV; k++) m = lds[k] > m ? lds[k] : m;
    return m;
}

template <int NWV>
__device__ __forceinline__ double sum_all(double v, double* red)
{
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & (WAVE - 1)) == 0) red[threadIdx.x / WAVE] = v;
    __syncthreads();
    double t = 0.0;
    for (int k = 0; k < NWV; k++) t += red[k];
    return t;
}

// 1 / sqrt(v) by the hardware estimate and two Newton steps (r += r/2 (1 - v
// r^2), each squaring the estimate's relative error of about 2^-23): a third
// of the dependent operations of a square root and a division.  v = 0 gives
// NaN instead of infinity; either ends the loop, the dot product being 0 / 0.
__device__ __forceinline__ double inv_sqrt(double v)
{
    double r = __builtin_amdgcn_rsq(v);
#pragma unroll
    for (int k = 0; k < 2; k++) r = fma(0.5 * r, fma(-(v * r), r, 1.0), r);
    return r;
}

// Rows that the LDS arrays of a level are laid out for (the sort keys of a
// tiny level fill one wavefront).
__host__ __device__ inline uint32_t span_of(uint32_t n) { return n < 64 ? 64u : n; }

// The level's layout: order, slices, matrix, degrees.
template <int NWV>
__device__ __forceinline__ void build_layout(const SmallLevel& V, const SmallJob& J, double* pool, Layout& S)
{
    using F = Form<NWV>;
    constexpr uint32_t NT = NWV * WAVE;
    const uint32_t n = V.n, tid = threadIdx.x, lane = tid & (WAVE - 1), wid = uniform(tid / WAVE);
    const uint32_t span = span_of(n);
    S.n = n;
    S.y = pool;
    // rows by (descending length, row): bitonic sort of (2^19 - 1 - length,
    // row) in the space of y
    uint32_t* key = reinterpret_cast<uint32_t*>(pool);
    uint16_t* inv = reinterpret_cast<uint16_t*>(pool + span);  // (the keys fill n2 <= 2 span words)
    uint32_t n2 = 64;
    while (n2 < n) n2 <<= 1;
    uint32_t mw = V.w ? 0u : 1u;
    if (V.w)
        for (uint32_t e = tid; e < V.m; e += NT) mw = V.w[e] > mw ? V.w[e] : mw;
    for (uint32_t i = tid; i < n2; i += NT)
        key[i] = i < n ? ((LEN_MAX - (V.rowptr[i + 1] - V.rowptr[i])) << COL_BITS) | i : INF;
    mw = max_all<NWV>(mw, S.words + 64);  // (with its barriers)
    S.wide = mw > LEN_MAX;
    for (uint32_t k = 2; k <= n2; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t t = tid; t < n2 / 2; t += NT) {
                const uint32_t i = ((t & ~(j - 1)) << 1) | (t & (j - 1)), p = i | j;
                const uint32_t u = key[i], v = key[p];
                if ((u > v) == ((i & k) == 0)) {
                    key[i] = v;
                    key[p] = u;
                }
            }
            // (pairs at most 64 apart lie in the 128 elements of one wavefront)
            if (j > WAVE || (j == 1 && k > WAVE))
                __syncthreads();
            else
                wave_fence();
        }
    }
    __syncthreads();
    // the slices: first as the register form wants them, then, when a
    // wavefront's steps or the weights do not fit, as the streamed form does
    uint32_t steps = 0;
    for (int attempt = F::STEPS ? 0 : 2;; attempt++) {
        S.regs = attempt < 2;
        Split sp;
        if (S.regs) {
            sp.t0 = n <= WAVE ? one_pass(n, WAVE, 4) : one_pass(n, NT, 4);
            sp.lcap = attempt == 0 ? INF : 24u;
        } else {
            sp.t0 = n <= WAVE ? one_pass(n, WAVE, 4) : one_pass(n, NT, 3);
            sp.lcap = n <= WAVE ? 16u : n <= 1024u ? 6u : 16u;
        }
        S.uni = attempt == 0;
        S.t = sp.t0;
        if (tid < 8) S.words[tid] = 0;
        __syncthreads();
        if (S.uni) {
            if (tid == 0) S.words[sp.t0] = n;
        } else {
            for (uint32_t i = tid; i < n; i += NT)
                atomicAdd(&S.words[lanes_log2(sp, LEN_MAX - (key[i] >> COL_BITS))], 1u);
        }
        __syncthreads();
        // rows of each T and where they start, longest rows (largest T) first
        uint32_t cstart[8], sstart[8];  // class c: T = 2^(6 - c)
        {
            uint32_t r = 0, s = 0;
#pragma unroll
            for (int c = 0; c < 7; c++) {
                cstart[c] = r;
                sstart[c] = s;
                const uint32_t cnt = S.words[6 - c], per = 64u >> (6 - c);
                r += cnt;
                s += (cnt + per - 1) / per;
            }
            cstart[7] = r;
            sstart[7] = s;
        }
        const uint32_t ns = sstart[7];
        S.nslices = ns;
        S.wstep = ns <= 2 ? 1u : (uint32_t)NWV;  // one wavefront holds a level of two slices: no barriers
        for (uint32_t s = tid; s < ns; s += NT) {
            uint32_t c = 0;
            uint32_t c0 = cstart[0], c1 = cstart[1], s0 = sstart[0];
#pragma unroll
            for (int q = 1; q < 7; q++)
                if (s >= sstart[q]) {
                    c = q;
                    c0 = cstart[q];
                    c1 = cstart[q + 1];
                    s0 = sstart[q];
                }
            const uint32_t t = 6 - c, per = 64u >> t, r0 = c0 + (s - s0) * per;
            const uint32_t rows = c1 - r0 < per ? c1 - r0 : per;
            const uint32_t deg = LEN_MAX - (key[r0] >> COL_BITS);
            uint32_t L = (deg + (1u << t) - 1u) >> t;
            if (S.regs) L = L ? (L + GROUP - 1) / GROUP * GROUP : GROUP;  // whole groups
            S.slice[s] = make_uint2(r0 | (rows - 1) << 13 | t << 19, L);
        }
        __syncthreads();
        // steps of each wavefront, a multiple of GROUP
        steps = 0;
        if (wid < S.wstep)
            for (uint32_t s = wid + S.wstep * lane; s < ns; s += S.wstep * WAVE) steps += S.slice[s].y;
        steps = wave_sum_u32(steps);
        steps = (steps + GROUP - 1) / GROUP * GROUP;
        if (lane == 0) S.words[16 + wid] = steps;
        __syncthreads();
        uint32_t most = 0;
        for (int k = 0; k < NWV; k++) most = S.words[16 + k] > most ? S.words[16 + k] : most;
        if (!S.regs || (most <= F::STEPS && (!S.uni || ns <= S.wstep * 16u) && (F::F64W || mw <= 0xffffu))) break;
        __syncthreads();  // (the words are set again)
    }
    // the row of every position, for the start vector and the result; its
    // inverse, for the columns
    for (uint32_t i = tid; i < n; i += NT) {
        const uint32_t r = key[i] & COL_MASK;
        J.ord[i] = r;
        inv[r] = (uint16_t)i;
    }
    S.steps = uniform(steps);
    S.base = 0;
    S.total = 0;
    for (uint32_t k = 0; k < (uint32_t)NWV; k++) {
        if (k == wid) S.base = S.total;
        S.total += S.words[16 + k];
    }
    S.base = uniform(S.base);
    S.span = S.regs ? F::MAX_N : span;
    S.wd = reinterpret_cast<uint32_t*>(pool + 2 * S.span);
    S.ent_l = S.wd + S.span;
    S.in_lds = !S.regs && !S.wide && 20u * span + 4u * WAVE * S.total <= F::POOL;
    __syncthreads();
    // the entries, slice by slice, and the degrees (parked in global memory
    // until the sort's space is no longer read)
    uint32_t* out = S.in_lds ? S.ent_l : J.ent;
    uint32_t pos = S.base;
    uint32_t gbm = 0;
    for (uint32_t s = wid < S.wstep ? wid : S.nslices; s < S.nslices; s += S.wstep) {
        const uint2 d = S.slice[s];
        const uint32_t t = uniform(d.x >> 19), L = uniform(d.y), i = lane >> t, sub = lane & ((1u << t) - 1u);
        const bool valid = i <= ((d.x >> 13) & 63u);
        const uint32_t p = (d.x & COL_MASK) + (valid ? i : 0u);
        const uint32_t r = key[p] & COL_MASK;
        const uint32_t e0 = V.rowptr[r], e1 = valid ? V.rowptr[r + 1] : e0;
        uint32_t wsum = 0;
        for (uint32_t k = 0; k < L; k++) {
            const uint32_t e = e0 + (k << t) + sub;
            const bool in = e < e1;
            const uint32_t c = in ? inv[V.col[e]] : p;
            const uint32_t w = in ? (V.w ? V.w[e] : 1u) : 0u;
            wsum += w;
            const uint32_t at = (pos + k) * WAVE + lane;
            if (S.wide) {
                out[2 * at] = c;
                out[2 * at + 1] = w;
            } else {
                out[at] = c | w << COL_BITS;
            }
        }
        pos += L;
#pragma unroll
        for (uint32_t o = 1; o < WAVE; o <<= 1)
            if (o < (1u << t)) wsum += __shfl_xor(wsum, o, WAVE);
        if (valid && sub == 0) J.deg[p] = wsum;
        const uint32_t g = (uint32_t)(2.0 * (double)wsum);
        gbm = g > gbm ? g : gbm;
    }
    for (; pos < S.base + S.steps; pos++) {
        const uint32_t at = pos * WAVE + lane;
        if (S.wide) {
            out[2 * at] = 0;
            out[2 * at + 1] = 0;
        } else {
            out[at] = 0;
        }
    }
    const uint32_t gb = max_all<NWV>(gbm, S.words + 64);  // (its barriers: every read of inv and the keys is done)
    S.gb = gb < 2u ? 2u : gb;
    for (uint32_t i = tid; i < n; i += NT) S.wd[i] = J.deg[i];
    __syncthreads();
}

// The loop's scalars: the input transform of the next iteration from the
// sums of the one before, and the stop test for that one
// (eigensolve_kokkos.h:155-189).
struct Loop {
    double T[3], dot0, dot1, last_a, last_s;
    uint32_t iter, budget, parity;
    bool stopped;
};

template <class Z>
__device__ __forceinline__ bool next_input(Z& z, double c, double n, double tol, unsigned long long iter_max, double& a,
                                           double& s)
{
    a = 0.0;
    s = 1.0;
    if (z.iter >= 2) {
        const double an = z.T[0] * c * c;
        const double sn = inv_sqrt(z.T[1] - 2.0 * an * z.T[0] + an * an * n);
        const double dot = z.T[2] * sn;
        const unsigned long long itn = z.iter - 1;
        const double lastd = (z.iter & 1u) ? z.dot1 : z.dot0;
        const bool go_on = (fabs(dot - lastd) > tol) && (itn < iter_max);
        if ((z.iter - 1) & 1u)
            z.dot1 = dot;
        else
            z.dot0 = dot;
        if (!go_on) {
            z.stopped = true;
            return false;
        }
        a = an;
        s = sn;
    }
    z.last_a = a;
    z.last_s = s;
    return true;
}

// The sums of the workgroup, in a fixed order: each wavefront's through LDS
// ([sum][wavefront], one value per lane when read back), or this wavefront's
// alone.  The barrier also orders the y of this iteration.
template <int NWV>
__device__ __forceinline__ void share_sums(double (&sum)[3], double* red, bool one, double (&T)[3])
{
    const uint32_t lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
#pragma unroll
    for (int k = 0; k < 3; k++) sum[k] = wave_sum(sum[k]);
    if (one) {
        wave_fence();
#pragma unroll
        for (int k = 0; k < 3; k++) T[k] = sum[k];
        return;
    }
    if (lane < 3) red[lane * NWV + wid] = lane == 0 ? sum[0] : lane == 1 ? sum[1] : sum[2];
    __syncthreads();
    double v = red[lane < 3 * NWV ? lane : 0];
    v += dpp_move_f64<0xB1>(v);
    v += dpp_move_f64<0x4E>(v);
    if (NWV >= 8) v += dpp_move_f64<0x141>(v);
    if (NWV >= 16) v += dpp_move_f64<0x140>(v);
#pragma unroll
    for (int k = 0; k < 3; k++) T[k] = readlane_d(v, NWV * k);
}

// One row's y and its terms of the sums.
__device__ __forceinline__ double row_value(double z, double yr, uint32_t wd, uint32_t gb, double a, double s,
                                            double (&sum)[3], bool mine)
{
    const double x = (yr - a) * s;
    const double ax = s * (z - a * (double)wd);
    const double y = fma((double)(uint32_t)(gb - wd), x, ax);
    const double ym = mine ? y : 0.0, xm = mine ? x : 0.0;
    sum[0] += ym;
    sum[1] = fma(ym, ym, sum[1]);
    sum[2] = fma(xm, ym, sum[2]);
    return y;
}

// Register form.  UNI: T is the same for every row, so that the wavefront's
// slices follow one another at a fixed distance and their lengths fit two
// scalar registers (one byte each); else the slice table is read along (a
// fifth slower on meshes, but it keeps levels with long rows in registers).
template <int NWV, bool WIDE, bool UNI>
__device__ __forceinline__ void iterate_regs(const SmallLevel& V, const Layout& S, const uint32_t* __restrict__ ent,
                                             double tol, Loop& Z)
{
    using F = Form<NWV>;
    constexpr uint32_t NS = F::STEPS, NG = NS / GROUP;
    const uint32_t lane = threadIdx.x & (WAVE - 1), wid = uniform(threadIdx.x / WAVE);
    const bool one = S.wstep == 1;
    const double c = 1 / sqrt((double)S.n), dn = (double)S.n;
    const uint32_t groups = S.steps / GROUP;
    // the matrix: byte offset into y and weight
    uint32_t off[NS];
    double wt[F::F64W ? NS : 1];
#pragma unroll
    for (uint32_t k = 0; k < NS; k++) {
        uint32_t cc = 0, w = 0;
        if (k < S.steps) {
            if (WIDE) {
                const uint2 v = *reinterpret_cast<const uint2*>(ent + 2 * (k * WAVE + lane));
                cc = v.x;
                w = v.y;
            } else {
                const uint32_t v = ent[k * WAVE + lane];
                cc = v & COL_MASK;
                w = v >> COL_BITS;
            }
        }
        if (F::F64W) {
            off[k] = cc * 8;
            wt[k] = (double)w;
        } else {
            off[k] = cc * 8 | w << 16;  // (n * 8 < 2^16, w < 2^16)
        }
    }
    // groups of each of this wavefront's slices
    unsigned long long gl = 0, gh = 0;
    if (UNI) {
        for (uint32_t k = 0, s = wid; s < S.nslices; s += S.wstep, k++) {
            const unsigned long long g = uniform(S.slice[s].y) / GROUP;
            if (k < 8)
                gl |= g << (8 * k);
            else
                gh |= g << (8 * (k - 8));
        }
    }
    const uint32_t per = WAVE >> S.t;  // rows per slice
    const uint32_t pos0 = wid * per + (lane >> S.t);
    const bool lead = (lane & ((1u << S.t) - 1u)) == 0;
    auto step = [&](auto parity) {
        constexpr uint32_t P = decltype(parity)::value;
        if (Z.budget == 0) return false;
        double a, s;
        // (the first gathers do not wait for a and s)
        const char* yo = reinterpret_cast<const char*>(S.y + P * F::MAX_N);
        double* yn = S.y + (1 - P) * F::MAX_N;
        double nx[GROUP];
        auto gather = [&](uint32_t g) {
#pragma unroll
            for (uint32_t u = 0; u < GROUP; u++) {
                // (an opaque value: its two halves, invariant over the
                // iterations, would otherwise be kept in registers as well)
                if (!F::F64W) asm volatile("" : "+v"(off[g * GROUP + u]));
                const uint32_t o = off[g * GROUP + u];
                nx[u] = *reinterpret_cast<const double*>(yo + (F::F64W ? o : (o & 0xffffu)));
            }
        };
        gather(0);
        // the open slice; with the table, the next one's entry too
        uint32_t sl = wid, t = S.t, left, pos, wd;
        bool mine;
        double yr;
        unsigned long long gls = gl, ghs = gh;
        uint2 nd = make_uint2(0u, GROUP);
        pos = pos0;
        if (!UNI && sl < S.nslices) nd = S.slice[sl];
        auto open = [&]() {
            if (UNI) {
                left = (uint32_t)gls & 0xffu;
                gls = gls >> 8 | ghs << 56;
                ghs >>= 8;
                mine = lead && pos < S.n;
            } else {
                t = uniform(nd.x >> 19);
                left = uniform(nd.y) / GROUP;
                pos = (nd.x & COL_MASK) + (lane >> t);
                mine = (lane & ((1u << t) - 1u)) == 0 && (lane >> t) <= ((nd.x >> 13) & 63u);
                sl += S.wstep;
                nd = sl < S.nslices ? S.slice[sl] : make_uint2(0u, GROUP);  // (past the last: not used)
            }
            const uint32_t row = mine ? pos : 0u;
            yr = *reinterpret_cast<const double*>(yo + 8 * row);
            wd = S.wd[row];
        };
        open();
        if (!next_input(Z, c, dn, tol, V.iter_max, a, s)) return false;
        double sum[3] = {0.0, 0.0, 0.0};
        double z0 = 0.0, z1 = 0.0;
#pragma unroll
        for (uint32_t g = 0; g < NG; g++) {
            if (g >= groups) break;
            double yv[GROUP];
#pragma unroll
            for (uint32_t u = 0; u < GROUP; u++) yv[u] = nx[u];
            if (g + 1 < NG) gather(g + 1);  // (past the last group: offset 0)
#pragma unroll
            for (uint32_t u = 0; u < GROUP; u++) {
                const double w = F::F64W ? wt[g * GROUP + u] : (double)(off[g * GROUP + u] >> 16);
                if (u & 1)
                    z1 = fma(w, yv[u], z1);
                else
                    z0 = fma(w, yv[u], z0);
            }
            if (--left == 0) {
                const double y = row_value(group_sum(z0 + z1, t), yr, wd, S.gb, a, s, sum, mine);
                if (mine) yn[pos] = y;
                z0 = z1 = 0.0;
                if (UNI) pos += S.wstep * per;
                open();
            }
        }
        share_sums<NWV>(sum, S.red + P * 64, one, Z.T);
        Z.iter++;
        Z.budget--;
        return true;
    };
    // (a launch starts with the current y in the first buffer)
    for (;;) {
        Z.parity = 0;
        if (!step(std::integral_constant<uint32_t, 0>{})) break;
        Z.parity = 1;
        if (!step(std::integral_constant<uint32_t, 1>{})) break;
    }
}

// One group of matrix words of a wavefront's stream.
template <bool WIDE>
struct Words {
    uint32_t c[GROUP], w[GROUP];
};

template <bool WIDE>
__device__ __forceinline__ void load_group(const uint32_t* p, Words<WIDE>& q)
{
#pragma unroll
    for (uint32_t u = 0; u < GROUP; u++) {
        if (WIDE) {
            const uint2 v = *reinterpret_cast<const uint2*>(p + 2 * u * WAVE);
            q.c[u] = v.x;
            q.w[u] = v.y;
        } else {
            const uint32_t v = p[u * WAVE];
            q.c[u] = v & COL_MASK;
            q.w[u] = v >> COL_BITS;
        }
    }
}

// Streamed form; `ent`: lane 0's first word of this wavefront's stream.
template <int NWV, bool WIDE>
__device__ __forceinline__ void iterate_stream(const SmallLevel& V, const Layout& S, const uint32_t* __restrict__ ent,
                                               double tol, Loop& Z)
{
    const uint32_t lane = threadIdx.x & (WAVE - 1), wid = uniform(threadIdx.x / WAVE);
    const bool one = S.wstep == 1;
    const double c = 1 / sqrt((double)S.n), dn = (double)S.n;
    const uint32_t ngroups = S.steps / GROUP;
    constexpr uint32_t stride = WAVE * GROUP * (WIDE ? 2 : 1);
    const uint32_t* lp = ent + (WIDE ? 2 : 1) * lane;
    for (; Z.budget > 0; Z.iter++, Z.budget--) {
        double a, s;
        if (!next_input(Z, c, dn, tol, V.iter_max, a, s)) break;
        const double* yo = S.y + (Z.parity ? S.span : 0u);
        double* yn = S.y + (Z.parity ? 0u : S.span);
        double sum[3] = {0.0, 0.0, 0.0};
        uint32_t sl = wid, t = 0, left = INF, pos = 0, wd = 0;
        bool mine = false;
        double yr = 0.0, z = 0.0;
        // the next slice of this wavefront (none: the rest of the stream is padding)
        auto open = [&]() {
            left = INF;
            if (sl >= S.nslices) return;
            const uint2 d = S.slice[sl];
            t = uniform(d.x >> 19);
            left = uniform(d.y);
            pos = (d.x & COL_MASK) + (lane >> t);
            mine = (lane & ((1u << t) - 1u)) == 0 && (lane >> t) <= ((d.x >> 13) & 63u);
            yr = yo[mine ? pos : 0u];
            wd = S.wd[mine ? pos : 0u];
        };
        auto close = [&]() {
            const double y = row_value(group_sum(z, t), yr, wd, S.gb, a, s, sum, mine);
            if (mine) yn[pos] = y;
            z = 0.0;
            sl += S.wstep;
            open();
        };
        open();
        while (left == 0) close();  // rows without entries
        if (ngroups) {
            Words<WIDE> q, nx;
            load_group<WIDE>(lp, nx);
            for (uint32_t g = 0; g < ngroups; g++) {
                q = nx;
                if (g + 1 < ngroups) load_group<WIDE>(lp + (size_t)(g + 1) * stride, nx);
                double yv[GROUP];
#pragma unroll
                for (uint32_t u = 0; u < GROUP; u++) yv[u] = yo[q.c[u]];
#pragma unroll
                for (uint32_t u = 0; u < GROUP; u++) {
                    z = fma((double)q.w[u], yv[u], z);
                    left--;
                    while (left == 0) close();
                }
            }
        }
        share_sums<NWV>(sum, S.red + (Z.parity ? 64 : 0), one, Z.T);
        Z.parity ^= 1u;
    }
}

// One workgroup per chain.  A launch runs at most `chunk` iterations of each
// chain and leaves its place in the chain's state; the next one continues
// with the same values.  A chain whose start another one computes (`after`)
// waits for a launch that finds that one done.
// A level that the registers of eight wavefronts do not hold (rows of hundreds
// of entries whose padding does not fit, or weights past 16 bits) is left to
// sixteen, which the host launches when it sees that: eight hide its loads
// worse when they stream it (R-MAT level of 388 vertices and 49,268 entries
// 15.6 us per iteration against 10.0; 400 and 37,654 with heavy weights 11.4
// against 7.6; 200 and 15,374 4.6 against 3.4).
template <int NWV>
__global__ void __launch_bounds__(NWV * WAVE, NWV / 4)
    k_small_chain(const SmallJob* __restrict__ jobs, uint32_t chunk, double tol)
{
    using F = Form<NWV>;
    constexpr uint32_t NT = NWV * WAVE;
    __shared__ double pool[F::POOL / 8];
    __shared__ uint2 slice[MAX_SLICES];
    __shared__ double red[2 * 4 * 16];
    __shared__ uint32_t words[128];
    const SmallJob J = jobs[blockIdx.x];
    if (J.after && !J.after->done) return;
    const uint32_t tid = threadIdx.x, wid = uniform(tid / WAVE);
    SmallState st = *J.st;
    uint32_t budget = chunk;
    uint32_t k = st.level;
    for (; k < J.nlv; k++) {
        // (sixteen wavefronts launched for a run of eight: the levels passed on)
        if (NWV == 8 && J.res[k].to16) break;
        if (NWV == 16 && J.waves == 8 && !J.res[k].to16) break;
        const SmallLevel V = J.lv[k];
        const uint32_t n = V.n;
        const unsigned long long tick = wall_clock64();
        Layout S;
        S.slice = slice;
        S.red = red;
        S.words = words;
        build_layout<NWV>(V, J, pool, S);
        if (NWV == 8 && !S.regs) {
            if (tid == 0) J.res[k].to16 = 1u;
            break;
        }
        if (st.iter == 0) {
            // the start vector, orthogonalised against 1n = 1/sqrt(n) and
            // normalised (eigensolve_kokkos.h:118-150)
            const double c = 1 / sqrt((double)n);
            const double* start = k == 0 ? J.start : J.v[(k - 1) & 1];
            double p0 = 0.0;
            for (uint32_t i = tid; i < n; i += NT) {
                const uint32_t r = J.ord[i];
                const double u = start[V.vcmap ? V.vcmap[r] : r];
                S.y[i] = u;
                p0 += u * c;
            }
            const double shift = sum_all<NWV>(p0, red) * c;
            double q = 0.0;
            for (uint32_t i = tid; i < n; i += NT) {
                const double u = S.y[i] - shift;
                S.y[i] = u;
                q += u * u;
            }
            const double inv = 1 / sqrt(sum_all<NWV>(q, red));
            for (uint32_t i = tid; i < n; i += NT) S.y[i] = S.y[i] * inv;
            st.iter = 1;
            st.T[0] = st.T[1] = st.T[2] = 0.0;
            st.dot0 = st.dot1 = st.last_a = 0.0;
            st.last_s = 1.0;
        } else {
            for (uint32_t i = tid; i < n; i += NT) {
                S.y[i] = J.y[0][i];
                S.y[S.span + i] = J.y[1][i];
            }
        }
        __syncthreads();
        Loop Z;
#pragma unroll
        for (int q = 0; q < 3; q++) Z.T[q] = st.T[q];
        Z.dot0 = st.dot0;
        Z.dot1 = st.dot1;
        Z.last_a = st.last_a;
        Z.last_s = st.last_s;
        Z.iter = st.iter;
        Z.budget = budget;
        Z.parity = 0;
        Z.stopped = false;
        if (wid < S.wstep) {
            if constexpr (F::STEPS > 0) {
                if (S.regs) {
                    if (F::F64W && S.wide)
                        iterate_regs<NWV, F::F64W, false>(V, S, J.ent + 2 * WAVE * S.base, tol, Z);
                    else if (S.uni)
                        iterate_regs<NWV, false, true>(V, S, J.ent + WAVE * S.base, tol, Z);
                    else
                        iterate_regs<NWV, false, false>(V, S, J.ent + WAVE * S.base, tol, Z);
                }
            }
            if constexpr (NWV != 8) {
                if (!S.regs) {
                    if (S.in_lds)
                        iterate_stream<NWV, false>(V, S, S.ent_l + WAVE * S.base, tol, Z);
                    else if (!S.wide)
                        iterate_stream<NWV, false>(V, S, J.ent + WAVE * S.base, tol, Z);
                    else
                        iterate_stream<NWV, true>(V, S, J.ent + 2 * WAVE * S.base, tol, Z);
                }
            }
        }
        // the loop's outcome, for the wavefronts that took no part
        __syncthreads();
        if (tid == 0) {
            words[0] = Z.stopped ? 1u : 0u;
            words[1] = Z.budget;
            words[2] = Z.iter;
            words[3] = Z.parity;
            red[0] = Z.last_a;
            red[1] = Z.last_s;
        }
        __syncthreads();
        const bool stopped = words[0] != 0;
        budget = words[1];
        const uint32_t iter = words[2], parity = words[3];
        const double* ynow = S.y + (parity ? S.span : 0u);
        const double* ybefore = S.y + (parity ? 0u : S.span);
        if (!stopped) {
            for (uint32_t i = tid; i < n; i += NT) {
                J.y[0][i] = ynow[i];
                J.y[1][i] = ybefore[i];
            }
            if (tid == 0) {
                st.level = k;
                st.iter = Z.iter;
#pragma unroll
                for (int q = 0; q < 3; q++) st.T[q] = Z.T[q];
                st.dot0 = Z.dot0;
                st.dot1 = Z.dot1;
                st.last_a = Z.last_a;
                st.last_s = Z.last_s;
                *J.st = st;
                J.res[k].ticks += wall_clock64() - tick;
            }
            return;
        }
        // the reference returns the input of the last iteration (eigensolve_kokkos.h:157)
        const double la = red[0], ls = red[1];
        double* out = J.v[k & 1];
        for (uint32_t i = tid; i < n; i += NT) out[J.ord[i]] = (ybefore[i] - la) * ls;
        if (tid == 0) {
            J.res[k].iters = iter - 1;
            J.res[k].ticks += wall_clock64() - tick;
            J.res[k].max_reached = iter - 1 >= V.iter_max ? 1u : 0u;
            J.res[k].done = 1u;
        }
        st.iter = 0;
        __syncthreads();
    }
    if (tid == 0) {
        J.st->level = k;
        J.st->iter = st.iter;
    }
}

// Matrix words of a level outside LDS at most.  A slice is padded to its
// longest row; rows are sorted, so all of a class but the first slice hold at
// most the entries of the slice before.  That first one has 64 lanes of at most
// 28 steps (one T for every row: 128), or rows of 64 lanes, which need no
// padding among each other.  Rounding rows up to whole steps or groups adds at
// most m / 3 (rows of T lanes have more than 3 T entries, in whole groups more
// than 12 T) and, for the rows of the smallest T, 4 n or 2,048; the last group of
// each wavefront 3 steps.  Together below 4/3 m + 4 n + 16384 words; wide
// entries take two.
uint64_t matrix_words(const DGraph& g)
{
    const uint64_t words = 2ull * g.m + 8ull * g.n + 16384;
    return g.unit ? words : 2 * words;
}

template <int NWV>
void launch_chain(Ctx& c, const SmallJob* jobs, unsigned grid, double tol)
{
    k_small_chain<NWV><<<grid, NWV * WAVE, 0, c.stream>>>(jobs, c.small_chunk, tol);
}

}  // namespace

bool small_level(const Ctx& c, const DGraph& g, bool mixed, int normLap)
{
    if (normLap) return !mixed && small_lds_level(c, g);
    return !mixed && g.m > 0 && g.n <= SMALL_MAX_N && g.m <= std::min(c.small_max_m, SMALL_MAX_M);
}

void solve_small_chains(Ctx& c, std::vector<SmallChain>& chains, int normLap, double tol)
{
    if (normLap) {
        solve_lds_chains(c, chains, normLap, tol);
        return;
    }
    // runs of levels of one workgroup size, each a job; a chain's runs follow
    // one another in launches of their own (`depth`)
    struct Run {
        size_t chain, k0, k1, depth;
        int waves;
        uint64_t at, nmax;
    };
    // the workgroup size: four wavefronts while a row costs each SIMD less than
    // the loop's scalar chain (3d grid of 1000 vertices, 5400 entries: 1.5 us
    // per iteration against 1.7 with eight; R-MAT of 461 and 9592: 3.0 against
    // 2.2); eight while the rows, padded to whole groups, about fit their
    // registers (3d grid of 5832, 33048 entries: 4.8 us against 8.5 with
    // sixteen; R-MAT of 2992, 53434, which does not fit: 11.6 against 7.4)
    const auto waves_of = [](const SmallChainLevel& l) {
        const uint32_t n = l.g->n, m = l.g->m;
        if (n <= Form<4>::MAX_N && m <= 5120) return 4;
        return m + 4 * n <= 61440 ? 8 : 16;
    };
    std::vector<Run> runs;
    size_t depths = 0;
    uint64_t words = 0;  // 8-byte words of workspace
    for (size_t j = 0; j < chains.size(); j++) {
        const std::vector<SmallChainLevel>& lv = chains[j].lv;
        MI_CHECK(!lv.empty(), ST_INTERNAL, "empty chain of small levels");
        size_t depth = 0;
        for (size_t k = 0; k < lv.size(); depth++) {
            Run r{j, k, k, depth, waves_of(lv[k]), words, 1};
            uint64_t ent = 0;
            for (; r.k1 < lv.size() && waves_of(lv[r.k1]) == r.waves; r.k1++) {
                const DGraph& g = *lv[r.k1].g;
                MI_CHECK(g.n <= SMALL_MAX_N && g.m <= SMALL_MAX_M && g.m > 0, ST_INTERNAL,
                         "level does not fit the one-workgroup form");
                r.nmax = std::max<uint64_t>(r.nmax, g.n);
                ent = std::max(ent, matrix_words(g));
            }
            k = r.k1;
            // four vectors (both level vectors, both y), order and degrees, matrix
            words += 5 * r.nmax + (ent + 1) / 2;
            runs.push_back(r);
        }
        depths = std::max(depths, depth);
    }
    const size_t R = runs.size();
    if (!R) return;
    // jobs of one launch together
    std::stable_sort(runs.begin(), runs.end(), [](const Run& x, const Run& y) {
        return x.depth != y.depth ? x.depth < y.depth : x.waves < y.waves;
    });
    // one table: the jobs, the levels chain by chain, states (zero: not begun) and results
    std::vector<size_t> first(chains.size() + 1, 0);
    for (size_t j = 0; j < chains.size(); j++) first[j + 1] = first[j] + chains[j].lv.size();
    const size_t nlv = first.back();
    const size_t o_lv = R * sizeof(SmallJob), o_st = o_lv + nlv * sizeof(SmallLevel),
                 o_res = o_st + R * sizeof(SmallState), bytes = o_res + nlv * sizeof(SmallResult);
    static_assert(sizeof(SmallJob) % 8 == 0 && sizeof(SmallLevel) % 8 == 0 && sizeof(SmallState) % 8 == 0 &&
                      sizeof(SmallResult) % 8 == 0,
                  "the table's parts are 8-byte aligned");
    std::vector<uint64_t> host(bytes / 8, 0);
    char* hp = reinterpret_cast<char*>(host.data());
    DBuf<uint64_t> table(&c.pool, bytes / 8), work(&c.pool, words);
    char* dp = reinterpret_cast<char*>(table.get());
    SmallJob* jobs = reinterpret_cast<SmallJob*>(hp);
    SmallLevel* lv = reinterpret_cast<SmallLevel*>(hp + o_lv);
    SmallResult* hres = reinterpret_cast<SmallResult*>(hp + o_res);
    SmallResult* dres = reinterpret_cast<SmallResult*>(dp + o_res);
    unsigned long long cap = 0;
    std::vector<double*> last(chains.size(), nullptr);  // where the run before left its vector
    for (size_t i = 0; i < R; i++) {
        const Run& r = runs[i];
        const SmallChain& ch = chains[r.chain];
        const uint32_t L = (uint32_t)(r.k1 - r.k0);
        double* w = reinterpret_cast<double*>(work.get() + r.at);
        SmallJob& q = jobs[i];
        q.lv = reinterpret_cast<const SmallLevel*>(dp + o_lv) + first[r.chain] + r.k0;
        q.res = dres + first[r.chain] + r.k0;
        q.nlv = L;
        q.waves = (uint32_t)r.waves;
        q.start = r.k0 ? last[r.chain] : ch.start;
        q.after = r.k0 ? q.res - 1 : nullptr;
        double* out = r.k1 == ch.lv.size() ? ch.out : w + r.nmax;
        last[r.chain] = out;
        q.v[(L - 1) & 1] = out;
        q.v[L & 1] = w;
        q.y[0] = w + 2 * r.nmax;
        q.y[1] = w + 3 * r.nmax;
        q.ord = reinterpret_cast<uint32_t*>(w + 4 * r.nmax);
        q.deg = q.ord + r.nmax;
        q.ent = reinterpret_cast<uint32_t*>(w + 5 * r.nmax);
        q.st = reinterpret_cast<SmallState*>(dp + o_st) + i;
        unsigned long long run_cap = 0;
        for (size_t k = r.k0; k < r.k1; k++) {
            const SmallChainLevel& l = ch.lv[k];
            SmallLevel& d = lv[first[r.chain] + k];
            d.n = l.g->n;
            d.m = l.g->m;
            d.rowptr = l.g->R();
            d.col = l.g->Cc();
            d.w = l.g->W();
            d.vcmap = l.vcmap;
            d.iter_max = 100000000000000ull / (unsigned long long)l.g->n;
            run_cap += d.iter_max;
        }
        cap = std::max(cap, run_cap);
    }
    MI_HIP(hipMemcpyAsync(table.get(), host.data(), bytes, hipMemcpyHostToDevice, c.stream));
    const size_t res_bytes = nlv * sizeof(SmallResult);
    bool passed_on = false;  // some level awaits sixteen wavefronts
    for (unsigned long long launched = 0;; launched += c.small_chunk) {
        MI_CHECK(launched / depths <= cap + c.small_chunk, ST_INTERNAL,
                 "power iteration did not stop at its iteration cap");
        for (size_t i = 0; i < R;) {
            size_t e = i;
            while (e < R && runs[e].depth == runs[i].depth && runs[e].waves == runs[i].waves) e++;
            const SmallJob* dj = reinterpret_cast<const SmallJob*>(dp) + i;
            const unsigned grid = (unsigned)(e - i);
            if (runs[i].waves == 4)
                launch_chain<4>(c, dj, grid, tol);
            else if (runs[i].waves == 8)
                launch_chain<8>(c, dj, grid, tol);
            // (before any level is passed on: none of that size)
            if (runs[i].waves == 16 || (runs[i].waves == 8 && passed_on)) launch_chain<16>(c, dj, grid, tol);
            MI_HIP(hipGetLastError());
            i = e;
        }
        MI_HIP(hipMemcpyAsync(hres, dres, res_bytes, hipMemcpyDeviceToHost, c.stream));
        MI_HIP(hipStreamSynchronize(c.stream));
        bool all = true;
        passed_on = false;
        for (size_t k = 0; k < nlv; k++) {
            all = all && hres[k].done;
            passed_on = passed_on || (hres[k].to16 && !hres[k].done);
        }
        if (all) break;
    }
    int khz = 0;
    MI_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, c.device));
    for (size_t j = 0; j < chains.size(); j++) {
        for (size_t k = 0; k < chains[j].lv.size(); k++) {
            const SmallResult& r = hres[first[j] + k];
            SmallChainLevel& l = chains[j].lv[k];
            l.iters = r.iters;
            l.max_reached = r.max_reached != 0;
            l.ms = khz > 0 ? (double)r.ticks / khz : 0.0;
        }
    }
}

}  // namespace mi
