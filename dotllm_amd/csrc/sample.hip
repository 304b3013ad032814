// sample.hip -- Sampler.Sample (src/Llmdot.Core/Sampling/Sampler.cs:24-170) on
// the device, for a logits vector already in HBM.
//
//   scale:    logits * (1f / Temperature)                   (Sampler.cs:30-34)
//   penalty:  the last RepeatPenaltyWindowSize history tokens, applied once per
//             occurrence: x > 0 ? x / p : x * p, then the same scale
//             (ApplyRepeatPenalty, Sampler.cs:64-81); each workgroup penalises
//             the tokens of its own slice of the vocabulary
//   top-k:    (0 < TopK < n, Sampler.cs:36-42) the k largest, sorted by (value
//             desc, index asc), VectorMath.Softmax over them in the reference's
//             summation order, then the sequential draw (SampleFromProbabilities,
//             Sampler.cs:158-170).  k <= TOPK_TREE: every workgroup selects its
//             slice's k largest, one workgroup those of all slices; above, one
//             workgroup radix-selects over all n
//   softmax:  (otherwise) VectorMath.Softmax over all n in the reference's
//             summation order: the probabilities bit for bit
//   top-p:    (TopP < 1, Sampler.cs:44-61, FindNucleus 129-156) the reference
//             as written: its selection-sort order (ties included), the values
//             it writes into the buffer it still reads from, the sequential
//             float running sum that closes the nucleus, the renormalised draw,
//             and the fall-through draw over the rewritten buffer that returns
//             a rank; candidates located by a histogram of the mass (fp64 radix
//             descent where its bins are too coarse), so a full sort runs only
//             when they do not suffice
//   no top-p: the draw over the probabilities in index order (Sampler.cs:61),
//             placed with fp64 running sums
//
// The uniform draw r (Random.NextSingle() in the reference, Sampler.cs:160-161)
// is an input, read from rvals[step - 1], so the caller owns the generator.
// In the top-k path exact ties between values are resolved toward the smaller
// index.
#include "common.h"
#include "kernels.h"

namespace llmdot {

namespace {

constexpr int SWG = 1024;          // the single-workgroup kernels
constexpr int NWAVE = SWG / 64;

// Order-preserving 32-bit key of a float (larger float, larger key) and back.
__device__ __forceinline__ uint32_t fkey(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float keyf(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// Exclusive prefix sum over the workgroup in thread order; *total gets the sum.
template <typename V>
__device__ V block_excl_scan(V v, V* tmp, V* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    V incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const V u = __shfl_up(incl, o, 64);
        if (lane >= o) incl += u;
    }
    if (lane == 63) tmp[wave] = incl;
    __syncthreads();
    if (wave == 0) {
        V w = lane < NWAVE ? tmp[lane] : V(0);
        V wi = w;
#pragma unroll
        for (int o = 1; o < NWAVE; o <<= 1) {
            const V u = __shfl_up(wi, o, 64);
            if (lane >= o) wi += u;
        }
        if (lane < NWAVE) tmp[NWAVE + lane] = wi - w;   // exclusive offset of each wavefront
        if (lane == NWAVE - 1) tmp[2 * NWAVE] = wi;
    }
    __syncthreads();
    const V r = tmp[NWAVE + wave] + incl - v;
    *total = tmp[2 * NWAVE];
    __syncthreads();
    return r;
}

struct Descent {
    uint32_t key;     // key of the element reached
    double above;     // weight of all elements with a larger key
    int cnt_above;    // how many there are
    int n_eq;         // elements with this key
};

// Radix descent over keys (largest first): the element at which the running
// weight, in (key desc, index asc) order, first reaches T.  MASS: weight = the
// value (non-negative); otherwise weight = 1 per element (a rank).  With T
// beyond the total the last element is reached.  Workgroup-uniform result.
// Values are x[i] * f (rounded to float).
template <bool MASS>
__device__ Descent descend(const float* x, float f, int n, double T) {
    __shared__ int cnt[256];
    __shared__ double wsum[256];
    __shared__ uint32_t s_digit;
    __shared__ double s_above;
    __shared__ int s_cabove, s_neq;
    const int t = threadIdx.x, lane = t & 63;
    uint32_t prefix = 0, mask = 0;
    double above = 0.0;
    int cabove = 0, neq = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
        for (int i = t; i < 256; i += SWG) { cnt[i] = 0; wsum[i] = 0.0; }
        __syncthreads();
        for (int i = t; i < n; i += SWG) {
            const float v = x[i] * f;
            const uint32_t k = fkey(v);
            if ((k & mask) == prefix) {
                const int d = (k >> shift) & 255;
                atomicAdd(&cnt[d], 1);
                if (MASS) atomicAdd(&wsum[d], (double)v);
            }
        }
        __syncthreads();
        if (t < 64) {
            // lane l holds digits 255 - 4l .. 252 - 4l (descending)
            int c[4];
            double w[4], lw = 0.0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int d = 255 - 4 * lane - q;
                c[q] = cnt[d];
                w[q] = MASS ? wsum[d] : (double)c[q];
                lw += w[q];
            }
            double incl = lw;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const double u = __shfl_up(incl, o, 64);
                if (lane >= o) incl += u;
            }
            double run = above + (incl - lw);
            int crun = 0;
            int hit = -1;
            double hit_above = 0.0;
            int hit_c = 0;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                if (hit < 0 && c[q] > 0 && run + w[q] >= T) { hit = q; hit_above = run; hit_c = crun; }
                run += w[q];
                crun += c[q];
            }
            // counts above this lane's digits
            int ci = crun;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int u = __shfl_up(ci, o, 64);
                if (lane >= o) ci += u;
            }
            const int cexcl = ci - crun;
            const uint64_t found = __ballot(hit >= 0);
            // nonempty digits, for the case T lies beyond the total
            int last_q = -1;
#pragma unroll
            for (int q = 0; q < 4; q++) if (c[q] > 0) last_q = q;
            const uint64_t nonempty = __ballot(last_q >= 0);
            int src;
            if (found) src = __ffsll((unsigned long long)found) - 1;
            else src = 63 - __clzll((long long)nonempty);
            if (lane == src) {
                int q = hit;
                double ab = hit_above;
                int cb = hit_c;
                if (!found) {   // the last nonempty digit, with everything before it above
                    q = last_q;
                    ab = above + (incl - lw);
                    cb = 0;
                    for (int j = 0; j < q; j++) { ab += w[j]; cb += c[j]; }
                }
                s_digit = (uint32_t)(255 - 4 * lane - q);
                s_above = ab;
                s_cabove = cabove + cexcl + cb;
                s_neq = c[q];
            }
        }
        __syncthreads();
        prefix |= s_digit << shift;
        mask |= 255u << shift;
        above = s_above;
        cabove = s_cabove;
        neq = s_neq;
        __syncthreads();
    }
    return Descent{prefix, above, cabove, neq};
}

constexpr int PEN_LDS = 1024;      // penalty windows up to this many tokens are read from LDS

// ApplyRepeatPenalty (Sampler.cs:64-81) on the last `window` history tokens
// that lie in [b0, b1), then the temperature scale: set(token, value) once per
// distinct token.  Called by the whole workgroup; sh holds PEN_LDS ints.
template <typename F>
__device__ void penalise(const SampleArgs& a, int b0, int b1, int* sh, F set) {
    const int L = a.hist_base + *a.step - 1;   // tokens before this draw
    const int w0 = max(0, L - a.window), W = L - w0;
    if (W <= 0) return;
    const int* hp = a.hist + w0;
    if (W <= PEN_LDS) {
        for (int i = threadIdx.x; i < W; i += blockDim.x) sh[i] = hp[i];
        __syncthreads();
        hp = sh;
    }
    for (int j = threadIdx.x; j < W; j += blockDim.x) {
        const int tok = hp[j];
        if (tok < b0 || tok >= b1) continue;
        int before = 0, c = 0;   // occurrences before j; from j on
#pragma unroll 8
        for (int i = 0; i < W; i++) {
            const int eq = hp[i] == tok;
            before += i < j ? eq : 0;
            c += i < j ? 0 : eq;
        }
        if (before) continue;
        float x = a.logits[tok];
        for (int i = 0; i < c; i++) x = x > 0.f ? x / a.penalty : x * a.penalty;
        set(tok, x * a.inv_temp);
    }
}

__device__ __forceinline__ bool penalised(const SampleArgs& a) { return a.penalty != 1.f && a.window > 0 && a.hist; }

// work = scaled and penalised logits, a slice of `chunk` per workgroup; the
// slice's maximum into smax; the mass histogram cleared for samp_exp_kernel.
__global__ __launch_bounds__(256) void samp_scale_kernel(SampleArgs a, int chunk) {
    __shared__ int sh[PEN_LDS];
    __shared__ float red[4];
    const int t = threadIdx.x, b0 = blockIdx.x * chunk, b1 = min(a.n, b0 + chunk);
    float m = -INFINITY;
    for (int i = b0 + t; i < b1; i += 256) {
        const float x = a.logits[i] * a.inv_temp;
        a.work[i] = x;
        m = fmaxf(m, x);
    }
    if (penalised(a)) {
        __syncthreads();
        penalise(a, b0, b1, sh, [&](int tok, float x) { a.work[tok] = x; });
        __syncthreads();
        m = -INFINITY;
        for (int i = b0 + t; i < b1; i += 256) m = fmaxf(m, a.work[i]);
    }
    m = wave_max(m);
    if ((t & 63) == 0) red[t >> 6] = m;
    SampleScratch* sc = sample_scratch(a.work, a.n);
    for (int i = blockIdx.x * 256 + t; i < SAMPLE_BINS; i += gridDim.x * 256) { sc->mass[i] = 0; sc->count[i] = 0; }
    __syncthreads();
    if (t == 0) sc->smax[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

__device__ void publish(const SampleArgs& a, int token) {
    const int s = *a.step - 1;
    *a.token_out = token;
    if (a.token_log && s >= 0 && s < a.log_cap) a.token_log[s] = token;
    if (a.hist_out) a.hist_out[a.hist_base + s] = token;
}

// VectorMath.Softmax over the k selected values, sorted in cand (VM:215-258):
// max, exponentials, eight interleaved partial sums, their horizontal sum, the
// tail; then SampleFromProbabilities' running sum and the draw.  Every thread
// of the workgroup calls it after a barrier behind cand.
__device__ void topk_draw(const SampleArgs& a, const uint64_t* cand, float* pv, int k) {
    __shared__ float s_part[8];
    const int t = threadIdx.x;
    const float M = keyf((uint32_t)(cand[0] >> 32));
    const int k8 = k & ~7;
    for (int j = t; j < k; j += blockDim.x) {
#pragma clang fp contract(off)
        const float d = keyf((uint32_t)(cand[j] >> 32)) - M;
        pv[j] = j < k8 ? exp_approx(d) : expf(d);
    }
    __syncthreads();
    if (t < 8) {
        float vs = 0.f;
#pragma unroll 8
        for (int j = t; j < k8; j += 8) vs += pv[j];
        s_part[t] = vs;
    }
    __syncthreads();
    if (t == 0) {
        float sum = ((s_part[0] + s_part[1]) + (s_part[2] + s_part[3])) + ((s_part[4] + s_part[5]) + (s_part[6] + s_part[7]));
        for (int j = k8; j < k; j++) sum += pv[j];
        const float inv = 1.0f / sum;
        const float r = a.rvals[*a.step - 1];
        float cum = 0.f;
        int pick = k - 1;
        bool open = true;
        // whole runs of 8, so that their loads do not wait on the running sum
        for (int j0 = 0; j0 < k && open; j0 += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = j0 + u < k ? pv[j0 + u] : 0.f;
#pragma unroll
            for (int u = 0; u < 8; u++) {
#pragma clang fp contract(off)
                const float pj = v[u] * inv;   // Scale(input, invSum), then the running sum
                cum += pj;
                if (open && j0 + u < k && r <= cum) { pick = j0 + u; open = false; }
            }
        }
        publish(a, (int)(0xFFFFFFFFu - (uint32_t)(cand[pick] & 0xFFFFFFFFu)));
    }
}

// The k largest of the workgroup's NT x EPT entries into out[0, k), in no
// particular order; an entry is (key, low) with low = ~index, so that of equal
// keys the smaller indices win; (0, 0) is no entry and fills up where there are
// fewer than k.  The k-th key is found bit by bit: EPT compares and wave
// ballots, one barrier per bit, until exactly k entries are at or above.
template <int NT, int EPT>
__device__ void block_topk(const uint32_t (&key)[EPT], const uint32_t (&low)[EPT], int k, uint64_t* out) {
    __shared__ int cnt[2][NT / 64];
    __shared__ int s_o;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int turn = 0;
    // entries for which the predicate holds, over the workgroup
    auto count = [&](auto pred) {
        int w = 0;
#pragma unroll
        for (int e = 0; e < EPT; e++) w += __popcll(__ballot(pred(key[e], low[e])));
        if (lane == 0) cnt[turn][wave] = w;
        __syncthreads();
        int tot = 0;
#pragma unroll
        for (int i = 0; i < NT / 64; i++) tot += cnt[turn][i];
        turn ^= 1;   // the next count's writes do not meet this one's reads
        return tot;
    };
    uint32_t T = 0, Lw = 0;   // take key > T, and key == T with low >= Lw
    bool exact = false;
    for (int bit = 31; bit >= 0 && !exact; bit--) {
        const uint32_t c = T | (1u << bit);
        const int tot = count([&](uint32_t q, uint32_t) { return q >= c; });
        if (tot >= k) { T = c; exact = tot == k; }
    }
    if (!exact) {   // several entries equal the k-th, or fewer than k entries
        const int need = k - count([&](uint32_t q, uint32_t) { return q > T; });
        bool done = false;
        for (int bit = 31; bit >= 0 && !done; bit--) {
            const uint32_t c = Lw | (1u << bit);
            const int tot = count([&](uint32_t q, uint32_t l) { return q == T && l >= c; });
            if (tot >= need) { Lw = c; done = tot == need; }
        }
    }
    if (t == 0) s_o = 0;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < EPT; e++)
        if ((key[e] | low[e]) && (key[e] > T || (key[e] == T && low[e] >= Lw))) {
            const int o = atomicAdd(&s_o, 1);
            if (o < k) out[o] = ((uint64_t)key[e] << 32) | low[e];
        }
    __syncthreads();
    for (int o = s_o + t; o < k; o += NT) out[o] = 0;
}

// Top-k over many workgroups: one selection by a single workgroup took 226 us
// for k = 40 of 128256 logits (five passes of 125 elements per thread behind
// LDS histogram atomics that collide in few exponents) behind 16 us of scaling
// and penalties; slices over the chip, penalties included, take 13.8 us and one
// selection among their winners 11.8.  Bound by latency: a barrier per key bit.
// The second
// selection holds TOPK_PARTS x TOPK_TREE entries in registers, which is where
// the limits lie.
constexpr int TOPK_TREE = 128;     // largest k
constexpr int TOPK_PARTS = 64;     // most slices
static_assert(TOPK_PARTS * TOPK_TREE * sizeof(uint64_t) <= sizeof(SampleScratch::cand), "candidate scratch");

template <int EPT>
__global__ __launch_bounds__(256) void samp_topk_part_kernel(SampleArgs a) {
    __shared__ float v[256 * EPT];
    __shared__ int sh[PEN_LDS];
    const int t = threadIdx.x, b0 = blockIdx.x * 256 * EPT, len = min(256 * EPT, a.n - b0);
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = t + 256 * e;
        if (i < len) v[i] = a.logits[b0 + i] * a.inv_temp;
    }
    if (penalised(a)) {
        __syncthreads();
        penalise(a, b0, b0 + len, sh, [&](int tok, float x) { v[tok - b0] = x; });
        __syncthreads();
    }
    uint32_t key[EPT], low[EPT];
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = t + 256 * e;
        key[e] = i < len ? fkey(v[i]) : 0u;
        low[e] = i < len ? ~(uint32_t)(b0 + i) : 0u;
    }
    block_topk<256, EPT>(key, low, a.top_k, sample_scratch(a.work, a.n)->cand + (size_t)blockIdx.x * a.top_k);
}

template <int EPT>
__global__ __launch_bounds__(512) void samp_topk_final_kernel(SampleArgs a, int ncand) {
    __shared__ uint64_t cand[TOPK_TREE], sorted[TOPK_TREE];
    __shared__ float pv[TOPK_TREE];
    const int t = threadIdx.x, k = a.top_k;
    const uint64_t* in = sample_scratch(a.work, a.n)->cand;
    uint32_t key[EPT], low[EPT];
#pragma unroll
    for (int e = 0; e < EPT; e++) {
        const int i = t + 512 * e;
        const uint64_t c = i < ncand ? in[i] : 0;
        key[e] = (uint32_t)(c >> 32);
        low[e] = (uint32_t)c;
    }
    block_topk<512, EPT>(key, low, k, cand);
    __syncthreads();
    if (t < k) {   // distinct entries: the rank is the number of larger ones
        const uint64_t c = cand[t];
        int r = 0;
#pragma unroll 8
        for (int j = 0; j < k; j++) r += cand[j] > c;
        sorted[r] = c;
    }
    __syncthreads();
    topk_draw(a, sorted, pv, k);
}

// Top-k path, one workgroup (k > TOPK_TREE or very large n): select, gather in index order, sort, softmax, draw.
__global__ __launch_bounds__(SWG) void samp_topk_kernel(SampleArgs a) {
    __shared__ uint64_t cand[SAMPLE_MAX_K];
    __shared__ float pv[SAMPLE_MAX_K];
    __shared__ int tmp[2 * NWAVE + 1];
    const int n = a.n, k = a.top_k, t = threadIdx.x;
    const Descent D = descend<false>(a.work, 1.0f, n, (double)k);
    const uint32_t K = D.key;
    const int need_eq = k - D.cnt_above;   // elements equal to the k-th value that are kept

    // stable gather: thread t walks [t * seg, ...) twice
    const int seg = (n + SWG - 1) / SWG;
    const int b = t * seg, e = min(n, b + seg);
    int ng = 0, ne = 0;
    for (int i = b; i < e; i++) {
        const uint32_t kk = fkey(a.work[i]);
        ng += kk > K;
        ne += kk == K;
    }
    int tot;
    const int eq_off = block_excl_scan<int>(ne, tmp, &tot);
    const int keep_eq = max(0, min(ne, need_eq - eq_off));
    const int out_off = block_excl_scan<int>(ng + keep_eq, tmp, &tot);
    {
        int o = out_off, r = 0;
        for (int i = b; i < e; i++) {
            const uint32_t kk = fkey(a.work[i]);
            const bool take = kk > K || (kk == K && r++ < keep_eq);
            if (take && o < SAMPLE_MAX_K) cand[o++] = ((uint64_t)kk << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)i);
        }
    }
    int P = 1;
    while (P < k) P <<= 1;
    for (int i = k + t; i < P; i += SWG) cand[i] = 0;
    __syncthreads();
    // bitonic sort, descending
    for (int size = 2; size <= P; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = t; i < P / 2; i += SWG) {
                const int lo = 2 * i - (i & (stride - 1));
                const int hi = lo + stride;
                const bool desc = (lo & size) == 0;
                const uint64_t x = cand[lo], y = cand[hi];
                if ((x < y) == desc) { cand[lo] = y; cand[hi] = x; }
            }
            __syncthreads();
        }
    }
    topk_draw(a, cand, pv, k);
}

// The numerators of VectorMath.Softmax over all n (VM:215-258) into work: the
// maximum (FindMax, VM:260-284: the same value whatever the order), ExpApprox
// on the first 8 floor(n/8), expf on the tail; and their histogram by the top
// 12 bits (an eighth of an octave per bin): counts, and masses in 2^-40 units
// (integer sums, so the same whatever the order).
__global__ __launch_bounds__(256) void samp_exp_kernel(SampleArgs a, int nmax) {
    __shared__ unsigned long long mass[SAMPLE_BINS];
    __shared__ int count[SAMPLE_BINS];
    __shared__ float red[4];
    const int t = threadIdx.x, n = a.n, n8 = n & ~7;
    SampleScratch* sc = sample_scratch(a.work, n);
    for (int i = t; i < SAMPLE_BINS; i += 256) { mass[i] = 0; count[i] = 0; }
    float m = -INFINITY;
    for (int i = t; i < nmax; i += 256) m = fmaxf(m, sc->smax[i]);
    m = wave_max(m);
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    for (int i = blockIdx.x * 256 + t; i < n; i += gridDim.x * 256) {
        float ev;
        {
#pragma clang fp contract(off)
            const float d = a.work[i] - m;
            ev = i < n8 ? exp_approx(d) : expf(d);
        }
        a.work[i] = ev;
        const int bin = min((int)(__float_as_uint(ev) >> 20), SAMPLE_BINS - 1);
        atomicAdd(&count[bin], 1);
        atomicAdd(&mass[bin], ev >= 0.f && ev <= 1.5f ? (unsigned long long)(ev * 1099511627776.0f) : 0ull);
    }
    __syncthreads();
    for (int i = t; i < SAMPLE_BINS; i += 256)
        if (count[i]) {
            atomicAdd(&sc->count[i], count[i]);
            atomicAdd(&sc->mass[i], mass[i]);
        }
}

// ---- top-p: FindNucleus (Sampler.cs:129-156) with the reference's buffers ----
//
// The reference sorts token ids by probability with a selection sort (strict
// `>`, so among equal values the first in the array's current order wins) and
// then writes values[i] = probabilities[indices[i]] into the same buffer the
// probabilities live in (Sampler.cs:30, 48-50): a rank i whose id indices[i]
// is below i reads the value rank indices[i] already wrote.  Following
// a = indices[a] while indices[a] < a therefore gives rank i's value,
// p[indices[a]] (each link lowers a, so the chain ends).  The running float sum
// of those values, in rank order, closes the nucleus; when it never reaches
// TopP the fall-through draw walks the rewritten buffer and returns a rank.
//
// Selection order: distinct values leave in descending order.  Equal values
// leave together, in the order of the array positions they hold when the
// first of them is selected; positions change only by the sort's swaps: at
// step s the selected element's old position src[s] receives the element that
// stood at s.  An element e still unselected at step s therefore stands at the
// end of e, src[e], src[src[e]], ... (followed while below s), and the members
// of a run of equal values keep their positions while the run is selected.
//
// Candidates: every element down to a value at which the mass surely reaches
// TopP + 1e-4 (whole runs of equal values): the lower edge of the histogram bin
// in which it does, or, where that would be too many, the element itself
// (fp64 radix descent).  The aliased values are at least
// the true ones and float addition is monotonic, so the aliased running sum
// reaches TopP no later than the true one; if it still has not within the
// candidates the kernel repeats the work over all n (global scratch).

constexpr int NUC_LDS = 4096;   // candidates sorted in LDS (fast path)
constexpr int ZCH = 8192;       // numerators summed per LDS stage
constexpr int ZLD = ZCH / 8 + 4;   // floats per lane sequence in a stage

// Ascending bitonic sort of a[0, P) (P a power of two) by the whole workgroup.
__device__ void bitonic_asc(uint64_t* a, int P, bool global) {
    const int t = threadIdx.x;
    for (int size = 2; size <= P; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = t; i < P / 2; i += SWG) {
                const int lo = 2 * i - (i & (stride - 1));
                const int hi = lo + stride;
                const bool up = (lo & size) == 0;
                const uint64_t x = a[lo], y = a[hi];
                if ((x > y) == up) { a[lo] = y; a[hi] = x; }
            }
            if (global) __threadfence();
            __syncthreads();
        }
    }
}

// Position at step s of element e (unselected before s).
__device__ __forceinline__ int position_at(const int* src, int e, int s) {
    int q = e;
    while (q < s) q = src[q];
    return q;
}

// The selection-sort order of K candidates whose (~key, id) pairs are sorted
// ascending in comp[0, K): ids[r] = the id selected at step r.  Positions
// (src[r] = where the element selected at step r stood then) are computed up
// to the end of the last run of equal values, the only steps whose order
// depends on positions; comp[K, 3K) is the scratch of the runs' sorts.
__device__ void selection_order(uint64_t* comp, int K, int* ids, int* src, bool global) {
    __shared__ int s_last, s_i, s_i1;
    const int t = threadIdx.x;
    if (t == 0) { s_last = 0; s_i = 0; }
    __syncthreads();
    for (int i = t; i < K; i += SWG) {
        ids[i] = (int)(uint32_t)comp[i];
        if (i + 1 < K && (comp[i] >> 32) == (comp[i + 1] >> 32)) atomicMax(&s_last, i + 2);
    }
    if (global) __threadfence();
    __syncthreads();
    const int R = s_last;   // ranks [0, R) need positions; [R, K) follow the value order
    uint64_t* tmp = comp + K;
    while (R > 0) {
        if (t == 0) {
            // singleton steps in order, up to the next run of equal values
            int i = s_i, i1 = i;
            while (i < R) {
                i1 = i + 1;
                const uint64_t k = comp[i] >> 32;
                while (i1 < K && (comp[i1] >> 32) == k) i1++;
                if (i1 - i > 1) break;
                src[i] = position_at(src, ids[i], i);
                i++;
            }
            s_i = i;
            s_i1 = i1;
        }
        if (global) __threadfence();
        __syncthreads();
        const int i = s_i, i1 = s_i1;
        if (i >= R) break;
        // the run [i, i1): members leave in the order of their positions at step i
        const int g = i1 - i;
        int P = 1;
        while (P < g) P <<= 1;
        for (int j = t; j < P; j += SWG) {
            uint64_t v = ~0ull;
            if (j < g) {
                const int e = ids[i + j];
                v = ((uint64_t)(uint32_t)position_at(src, e, i) << 32) | (uint32_t)e;
            }
            tmp[j] = v;
        }
        if (global) __threadfence();
        __syncthreads();
        bitonic_asc(tmp, P, global);
        for (int j = t; j < g; j += SWG) {
            ids[i + j] = (int)(uint32_t)tmp[j];
            src[i + j] = (int)(tmp[j] >> 32);
        }
        if (global) __threadfence();
        __syncthreads();
        if (t == 0) s_i = i1;
        __syncthreads();
    }
    __syncthreads();
}

// Rank r's value as the reference writes it (the aliased chain), for r < K.
__device__ __forceinline__ float aliased_value(const float* e, float inv, const int* ids, int r) {
    int a = r;
    while (ids[a] < a) a = ids[a];
    return e[ids[a]] * inv;
}

// Running float sum of v[0, K) in order, from 0: the first index at which
// stop(sum) holds (K if none), and the sum there.  Runs of 8, so that their
// loads do not wait on the sum.
template <typename F>
__device__ int running_sum(const float* v, int K, float scale, float* sum, F stop) {
    float c = 0.f;
    for (int i0 = 0; i0 < K; i0 += 8) {
        float x[8];
#pragma unroll
        for (int u = 0; u < 8; u++) x[u] = i0 + u < K ? v[i0 + u] : 0.f;
#pragma unroll
        for (int u = 0; u < 8; u++) {
#pragma clang fp contract(off)
            if (i0 + u >= K) break;
            const float y = x[u] * scale;
            c += y;
            if (stop(c)) { *sum = c; return i0 + u; }
        }
    }
    *sum = c;
    return K;
}

// FindNucleus over K candidates (comp: (~key, id) pairs sorted in [0, K), 3K
// slots; ids, val: K each), then the draw; probabilities are e[i] * inv.
// Returns the token (or the rank, when the nucleus spans all n), or -1 when
// the running sum does not reach TopP within K < n.
__device__ int nucleus_draw(const float* e, float inv, int n, uint64_t* comp, int K, int* ids, float* val, float top_p,
                            float r, bool global) {
    __shared__ int s_res;
    const int t = threadIdx.x;
    int* src = reinterpret_cast<int*>(val);   // positions first, values after
    selection_order(comp, K, ids, src, global);
    for (int i = t; i < K; i += SWG) val[i] = aliased_value(e, inv, ids, i);
    if (global) __threadfence();
    __syncthreads();
    if (t == 0) {
        // FindNucleus's running sum (Sampler.cs:146-154)
        float sum, c;
        int count = running_sum(val, K, 1.0f, &sum, [&](float x) { return x >= top_p; }) + 1;
        if (count > K) count = K == n ? n : -1;
        int res = -1;
        if (count > 0 && count < n) {
            // Sampler.cs:51-57: sum (the same adds as above), Scale(1f / sum), the draw over the nucleus
            const int pick = running_sum(val, count, 1.0f / sum, &c, [&](float x) { return r <= x; });
            res = ids[min(pick, count - 1)];
        } else if (count == n) {
            // Sampler.cs:61 over the rewritten buffer: a rank is returned
            res = min(running_sum(val, n, 1.0f, &c, [&](float x) { return r <= x; }), n - 1);
        }
        s_res = res;
    }
    __syncthreads();
    return s_res;
}

// The softmax's denominator, then the top-p nucleus and the draw (Sampler.cs:44-61),
// over the numerators in work[0, n); the rest of work is scratch
// (sample_work_floats).  The denominator is the reference's sum (VM:238-250):
// lane l adds numerators l, l + 8, ... in order, the eight sums fold as
// ((l0 + l1) + (l2 + l3)) + ((l4 + l5) + (l6 + l7)), the tail follows in order:
// n / 8 dependent adds, which bound the kernel for large n.  At 32000 logits
// the top-p launches take 39 us (scale 7, exp 5, this one 27) against 130 when
// one workgroup did each pass over n and loads waited in the sum.  Wavefront 0 adds
// from LDS while the others stage the next 8192 numerators there, each lane's
// sequence contiguous (four numerators per LDS read), and list the candidates.
__global__ __launch_bounds__(SWG) void samp_nucleus_kernel(SampleArgs a) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[3 * NUC_LDS * 8 + NUC_LDS * 8];
    static_assert(2 * 8 * ZLD * 4 <= 3 * NUC_LDS * 8, "sum stages");
    uint64_t* const l_comp = reinterpret_cast<uint64_t*>(lds);
    int* const l_ids = reinterpret_cast<int*>(lds + 3 * NUC_LDS * 8);
    float* const l_val = reinterpret_cast<float*>(lds + 3 * NUC_LDS * 8 + NUC_LDS * 4);
    float* const stage = reinterpret_cast<float*>(lds);   // before the candidates' sort
    __shared__ double dtmp[2 * NWAVE + 1];
    __shared__ unsigned long long utmp[2 * NWAVE + 1];
    __shared__ int itmp[2 * NWAVE + 1];
    __shared__ float s_lane[8];
    __shared__ float s_inv;
    __shared__ int s_pick, s_cnt, s_edge, s_kc;
    const int n = a.n, t = threadIdx.x, n8 = n & ~7;
    const float* e = a.work;
    const float rf = a.rvals[*a.step - 1];
    const bool nucleus = a.top_p < 1.f;
    // the histogram bin in which the mass from the top reaches TopP + 1e-4
    if (nucleus) {
        static_assert(SAMPLE_BINS == SWG, "one bin per thread");
        const SampleScratch* sc = sample_scratch(a.work, n);
        const int bin = SAMPLE_BINS - 1 - t;
        const unsigned long long mb = sc->mass[bin];
        const int cb = sc->count[bin];
        if (t == 0) { s_edge = 0; s_kc = n; s_cnt = 0; }
        unsigned long long total;
        int ctotal;
        const unsigned long long above = block_excl_scan<unsigned long long>(mb, utmp, &total);
        const int cabove = block_excl_scan<int>(cb, itmp, &ctotal);
        const double T = ((double)a.top_p + 1e-4) * (double)total;
        if ((double)above < T && (double)(above + mb) >= T) { s_edge = bin; s_kc = cabove + cb; }
        __syncthreads();
    }
    const float edge = nucleus ? __uint_as_float((uint32_t)s_edge << 20) : 0.f;
    const float edge_lo = edge * (1.0f - 0x1p-22f);   // below any numerator whose probability equals the edge's
    const bool list = nucleus && s_kc <= NUC_LDS;
    float acc = 0.f;   // wavefront 0, lanes 0..7
    const int nst = (n + ZCH - 1) / ZCH;
    for (int c = 0; c <= nst; c++) {
        if (t >= 64 && c < nst) {
            float* st = stage + (c & 1) * 8 * ZLD;
            for (int q = t - 64; q < ZCH; q += SWG - 64) {
                const int i = c * ZCH + q;
                if (i >= n) break;
                const float v = e[i];
                st[(q & 7) * ZLD + (q >> 3)] = v;
                if (list && v >= edge_lo) {
                    const int o = atomicAdd(&s_cnt, 1);
                    if (o < NUC_LDS) l_ids[o] = i;
                }
            }
        } else if (t < 8 && c > 0) {
            const float* st = stage + ((c - 1) & 1) * 8 * ZLD + t * ZLD;
            const int m = min(n8 - (c - 1) * ZCH, ZCH) >> 3;   // numerators of this lane in the stage
            int j = 0;
            for (; j + 16 <= m; j += 16) {
                float4 v[4];
#pragma unroll
                for (int u = 0; u < 4; u++) v[u] = *reinterpret_cast<const float4*>(st + j + 4 * u);
#pragma unroll
                for (int u = 0; u < 4; u++) { acc += v[u].x; acc += v[u].y; acc += v[u].z; acc += v[u].w; }
            }
            for (; j < m; j++) acc += st[j];
        }
        __syncthreads();
    }
    if (t < 8) s_lane[t] = acc;
    __syncthreads();
    if (t == 0) {
        float z = ((s_lane[0] + s_lane[1]) + (s_lane[2] + s_lane[3])) + ((s_lane[4] + s_lane[5]) + (s_lane[6] + s_lane[7]));
        for (int j = n8; j < n; j++) z += e[j];
        s_inv = 1.0f / z;
        s_pick = 0;
    }
    __syncthreads();
    const float inv = s_inv;   // probabilities: e[i] * inv, the reference's bit for bit
    if (nucleus) {
        int res = -1, K = 0;
        bool fits = list && s_cnt <= NUC_LDS;
        if (fits) {
            // the listed numerators whose probability is at least the edge's
            const float pe = edge * inv;
            const int cnt = s_cnt;
            for (int o = t; o < cnt; o += SWG) {
                const int i = l_ids[o];
                const float p = e[i] * inv;
                if (p >= pe) l_comp[atomicAdd(&s_pick, 1)] = ((uint64_t)(~fkey(p)) << 32) | (uint32_t)i;
            }
        } else {
            // every element at or above the value where the fp64 mass reaches TopP + 1e-4
            const Descent D = descend<true>(e, inv, n, (double)a.top_p + 1e-4);
            fits = D.cnt_above + D.n_eq <= NUC_LDS;
            if (fits)
                for (int i = t; i < n; i += SWG) {
                    const uint32_t k = fkey(e[i] * inv);
                    if (k >= D.key) {
                        const int o = atomicAdd(&s_pick, 1);
                        if (o < NUC_LDS) l_comp[o] = ((uint64_t)(~k) << 32) | (uint32_t)i;
                    }
                }
        }
        __syncthreads();
        K = s_pick;
        if (fits && K > 0 && K <= NUC_LDS) {
            int P = 1;
            while (P < K) P <<= 1;
            for (int i = K + t; i < P; i += SWG) l_comp[i] = ~0ull;
            __syncthreads();
            bitonic_asc(l_comp, P, false);
            res = nucleus_draw(e, inv, n, l_comp, K, l_ids, l_val, a.top_p, rf, false);
        }
        if (res < 0) {
            // all n in global scratch
            int P = 1;
            while (P < n) P <<= 1;
            uint64_t* comp = reinterpret_cast<uint64_t*>(a.work + sample_comp_offset(n));
            int* ids = reinterpret_cast<int*>(a.work + sample_comp_offset(n) + 6 * (size_t)n);
            float* val = a.work + sample_comp_offset(n) + 7 * (size_t)n;
            for (int i = t; i < P; i += SWG)
                comp[i] = i < n ? ((uint64_t)(~fkey(e[i] * inv)) << 32) | (uint32_t)i : ~0ull;
            __threadfence();
            __syncthreads();
            bitonic_asc(comp, P, true);
            res = nucleus_draw(e, inv, n, comp, n, ids, val, a.top_p, rf, true);
        }
        if (t == 0) publish(a, res < 0 ? n - 1 : res);
        return;
    }
    // SampleFromProbabilities over all n in index order (Sampler.cs:61)
    const double r = (double)rf;
    const int seg = (n + SWG - 1) / SWG;
    const int b = t * seg, b1 = min(n, b + seg);
    double sum = 0.0;
    for (int i = b; i < b1; i++) sum += (double)(e[i] * inv);
    double total;
    const double off = block_excl_scan<double>(sum, dtmp, &total);
    if (t == 0) s_pick = n - 1;
    __syncthreads();
    if (off < r && r <= off + sum) {
        double c = off;
        for (int i = b; i < b1; i++) {
            c += (double)(e[i] * inv);
            if (r <= c) { s_pick = i; break; }
        }
    } else if (t == 0 && r <= 0.0) {
        s_pick = 0;
    }
    __syncthreads();
    if (t == 0) publish(a, s_pick < 0 ? n - 1 : s_pick);
}

}  // namespace

bool sample_supported(int n, int top_k) { return n > 0 && !(top_k > SAMPLE_MAX_K && top_k < n); }

hipError_t launch_sample(const SampleArgs& a, hipStream_t s) {
    if (!sample_supported(a.n, a.top_k) || a.inv_temp <= 0.f) return hipErrorInvalidValue;
    if (a.top_k > 0 && a.top_k < a.n && a.top_k <= TOPK_TREE && a.n <= TOPK_PARTS * 256 * 32) {
        // slices of 2048, 4096 or 8192: the smallest that gives at most TOPK_PARTS
        const int ept = a.n <= TOPK_PARTS * 256 * 8 ? 8 : a.n <= TOPK_PARTS * 256 * 16 ? 16 : 32;
        const int parts = (a.n + 256 * ept - 1) / (256 * ept), ncand = parts * a.top_k;
        if (ept == 8) samp_topk_part_kernel<8><<<parts, 256, 0, s>>>(a);
        else if (ept == 16) samp_topk_part_kernel<16><<<parts, 256, 0, s>>>(a);
        else samp_topk_part_kernel<32><<<parts, 256, 0, s>>>(a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        if (ncand <= 512 * 4) samp_topk_final_kernel<4><<<1, 512, 0, s>>>(a, ncand);
        else samp_topk_final_kernel<16><<<1, 512, 0, s>>>(a, ncand);
        return hipGetLastError();
    }
    // at most SAMPLE_SLICES slices of whole multiples of 1024
    const int chunk = ((a.n + SAMPLE_SLICES - 1) / SAMPLE_SLICES + 1023) / 1024 * 1024;
    const int g = (a.n + chunk - 1) / chunk;
    samp_scale_kernel<<<g, 256, 0, s>>>(a, chunk);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (a.top_k > 0 && a.top_k < a.n) {
        samp_topk_kernel<<<1, SWG, 0, s>>>(a);
        return hipGetLastError();
    }
    samp_exp_kernel<<<g, 256, 0, s>>>(a, g);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    samp_nucleus_kernel<<<1, SWG, 0, s>>>(a);
    return hipGetLastError();
}

}  // namespace llmdot
