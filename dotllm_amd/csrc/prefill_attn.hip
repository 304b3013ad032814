// prefill_attn.hip -- causal attention of a chunk's queries over a KV cache in
// registers: 16 queries of one head per workgroup, its wavefronts taking
// different keys.
//
// The 64-query kernels of prefill.hip share each K / V tile through LDS among
// four wavefronts of queries and walk all keys in sequence: right when there
// are workgroups for every CU, but a short turn behind a long conversation or
// a small model has only a few (23 tokens x 32 heads: 32 workgroups of 29
// key tiles each).  Here no tile is shared: a wavefront loads its keys' K and
// V rows straight into MFMA operands, so the keys of one query block spread
// over the workgroup's W wavefronts, and the row maxima (VectorMath.Softmax
// needs the exact maximum before any exponential,
// src/Llmdot.Core/Tensors/Numeric/VectorMath.cs:215-258) and the partial sums
// meet in LDS: one launch, no scores in memory.  Bound by the latency of the
// row loads (the next step's are in flight while a step computes).  Measured
// per layer: 23 tokens behind 1800, 32 heads of 128, fp16: 136 -> 40 us; 512
// tokens, 32 heads of 64, fp16: 35 -> 19; 301 tokens, 8 heads of 128, fp32:
// 121 (fp32 vector arithmetic, scores through memory) -> 20.
//
// Scores are computed transposed (A = K rows, B = q), which leaves lane
// (lr, lk) = (lane & 15, lane >> 4) with keys 4 lk .. 4 lk + 3 of each 16-key
// tile for query lr: the A operand of e . V.
//   fp16 cache: v_mfma_f32_16x16x32_f16; q and e enter as two fp16 planes
//     (22-bit significands), like the 64-query kernels, same scores bit for
//     bit.  V: a lane loads DPL consecutive dims (8 or 4 bytes) of its 8 keys
//     and turns them into the B operands of DPL output tiles with v_perm;
//     output tile j of a 16 DPL-wide slice holds dims DPL lr + j.
//   fp32 cache: v_mfma_f32_16x16x4_f32, plain fp32 products and sums; the key
//     operand takes dims 16 j + 4 lk + i (one 16-byte load for 4 MFMAs), the
//     value operand the same dims DPL lr + j.
#include "common.h"
#include "kernels.h"

#include <algorithm>

namespace llmdot {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr int QB = 16;   // queries per workgroup

template <int HD, bool F16>
struct Attn {
    static constexpr int DPL = HD % 64 == 0 ? 4 : 2;   // dims per lane of a V load
    static constexpr int NC = HD / (16 * DPL);         // slices of a V row
    static constexpr int KT = F16 ? 2 : 1;             // 16-key tiles per step
    static constexpr int KSTEP = 16 * KT;
    static constexpr int KS = HD / 32;                 // fp16 MFMA steps per score
    static constexpr int KJ = HD / 16;                 // fp32: 4 MFMAs each

    h8 qh[F16 ? KS : 1], ql[F16 ? KS : 1];
    f4 qf[F16 ? 1 : KJ];
    float oscale;

    // one step's K rows: fp16 dims 32 ks + 8 lk .. + 7, fp32 dims 16 j + 4 lk .. + 3, of key row kt * 16 + lr
    struct KFrag {
        v4u r[F16 ? KT * KS : KJ];
    };

    __device__ __forceinline__ void load_q(const PfAttnArgs& a, int tq, int h, int lk) {
        const float* qrow = a.qr + (int64_t)tq * (a.heads * HD) + h * HD;
        if constexpr (F16) {
            float qv[KS][8];
            float amax = 0.f;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const f4 u = *reinterpret_cast<const f4*>(qrow + 32 * ks + 8 * lk);
                const f4 v = *reinterpret_cast<const f4*>(qrow + 32 * ks + 8 * lk + 4);
#pragma unroll
                for (int i = 0; i < 4; i++) { qv[ks][i] = u[i]; qv[ks][4 + i] = v[i]; }
#pragma unroll
                for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(qv[ks][i]));
            }
            amax = fmaxf(amax, fx(lane_xor16, amax));
            amax = fmaxf(amax, fx(lane_xor32, amax));
            int e = 0;
            if (amax > 0.f) {
                (void)frexpf(amax, &e);
                e = 15 - e;
                e = e > 126 ? 126 : (e < -126 ? -126 : e);
            }
            const float sq = ldexpf(1.0f, e);
#pragma unroll
            for (int ks = 0; ks < KS; ks++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float x = qv[ks][i] * sq;
                    const _Float16 hi = (_Float16)x;
                    qh[ks][i] = hi;
                    ql[ks][i] = (_Float16)(x - (float)hi);
                }
            oscale = (1.0f / sqrtf((float)HD)) * ldexpf(1.0f, -e);
        } else {
#pragma unroll
            for (int j = 0; j < KJ; j++) qf[j] = *reinterpret_cast<const f4*>(qrow + 16 * j + 4 * lk);
            oscale = 1.0f / sqrtf((float)HD);
        }
    }

    // rows past the last key repeat it (their scores are masked)
    __device__ __forceinline__ static void load_k(KFrag& f, const void* kc, int64_t base, int j0, int nkeys, int lr,
                                                  int lk) {
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            const int64_t row = base + (int64_t)min(j0 + 16 * kt + lr, nkeys - 1) * HD;
            if constexpr (F16) {
                const _Float16* p = reinterpret_cast<const _Float16*>(kc) + row + 8 * lk;
#pragma unroll
                for (int ks = 0; ks < KS; ks++) f.r[kt * KS + ks] = *reinterpret_cast<const v4u*>(p + 32 * ks);
            } else {
                const float* p = reinterpret_cast<const float*>(kc) + row + 4 * lk;
#pragma unroll
                for (int j = 0; j < KJ; j++) f.r[j] = *reinterpret_cast<const v4u*>(p + 16 * j);
            }
        }
    }

    // one step's V rows, dims 16 DPL c + DPL lr .. + DPL - 1 of each:
    // fp16 keys 16 (i / 4) + 4 lk + i % 4 (i < 8), fp32 keys 4 lk + i
    static constexpr int VK = F16 ? 8 : 4, VW = F16 ? DPL / 2 : DPL;
    struct VFrag {
        uint32_t w[NC][VK][VW];
    };
    __device__ __forceinline__ static void load_v(VFrag& f, const void* vc, int64_t base, int j0, int nkeys, int lr,
                                                  int lk) {
#pragma unroll
        for (int i = 0; i < VK; i++) {
            const int key = min(j0 + 16 * (i >> 2) + 4 * lk + (i & 3), nkeys - 1);
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const int64_t el = base + (int64_t)key * HD + 16 * DPL * c + DPL * lr;
                const uint8_t* p = reinterpret_cast<const uint8_t*>(vc) + el * (F16 ? 2 : 4);
                if constexpr (VW == 4) {
                    const v4u x = *reinterpret_cast<const v4u*>(p);
#pragma unroll
                    for (int k = 0; k < 4; k++) f.w[c][i][k] = x[k];
                } else if constexpr (VW == 2) {
                    const uint2 x = *reinterpret_cast<const uint2*>(p);
                    f.w[c][i][0] = x.x;
                    f.w[c][i][1] = x.y;
                } else {
                    f.w[c][i][0] = *reinterpret_cast<const uint32_t*>(p);
                }
            }
        }
    }

    // scores of keys j0 + 16 kt + 4 lk + r for query lr
    __device__ __forceinline__ f4 scores(const KFrag& f, int kt) const {
        f4 c = f4{0.f, 0.f, 0.f, 0.f};
        if constexpr (F16) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const h8 kf = __builtin_bit_cast(h8, f.r[kt * KS + ks]);
                c = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qh[ks], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, ql[ks], c, 0, 0, 0);
            }
        } else {
            f4 c2 = c;   // two chains: a dependent MFMA waits for its predecessor's last pass
#pragma unroll
            for (int j = 0; j < KJ; j++) {
                const f4 kf = __builtin_bit_cast(f4, f.r[j]);
                c = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[0], qf[j][0], c, 0, 0, 0);
                c2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[1], qf[j][1], c2, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[2], qf[j][2], c, 0, 0, 0);
                c2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[3], qf[j][3], c2, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) c[r] += c2[r];
        }
#pragma unroll
        for (int r = 0; r < 4; r++) c[r] = c[r] * oscale;
        return c;
    }
};

// MODE: all of it, or with the keys also spread over blockIdx.y of a.splits
// workgroups, the maxima (to a.part_max) and then the sums (to a.part_out and
// a.part_z, added up where they are read) as a launch each: a CU reads rows at
// about 50 GB/s, so with few query blocks only more CUs shorten it.
enum AttnMode { ATTN_ALL = 0, ATTN_MAX = 1, ATTN_SUM = 2 };

template <int HD, bool F16, int W, int MODE>
__global__ __launch_bounds__(64 * W) void pf_attn_wave_kernel(PfAttnArgs a) {
    using A = Attn<HD, F16>;
    constexpr int DPL = A::DPL, NC = A::NC, KT = A::KT, KSTEP = A::KSTEP, NT = HD / 16;
    __shared__ float mx[W][QB];
    __shared__ float ob[W / 2][NT * 4 + 1][64];
    // causal work grows with the block: the heaviest first
    const int nqb = (a.T + QB - 1) / QB, L = (int)blockIdx.x;
    // consecutive workgroups (on different XCDs) take different kv heads, so
    // with 8 kv heads the heads that share K and V rows share an XCD's L2
    const int x = L % a.heads, kvh = x % a.kv_heads, h = kvh * (a.heads / a.kv_heads) + x / a.kv_heads;
    const int t0 = (nqb - 1 - L / a.heads) * QB;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tq = t0 + lr, tqc = min(tq, a.T - 1);
    A at;
    at.load_q(a, tqc, h, lk);
    const int last = tq < a.T ? a.pos0 + tq : -1;   // the query's last key
    // SlidingWindow (IE:385-387): the query's first key, and the block's first step
    const int window = F16 ? a.window : 0;   // fp16 caches only (launch_prefill_attn_wave)
    const int first = window > 0 ? max(0, a.pos0 + tqc + 1 - window) : 0;
    const int jstart = window > 0 ? max(0, a.pos0 + t0 + 1 - window) / KSTEP * KSTEP : 0;
    // the window's first 8 floor(len/8) keys are the Softmax's vector lanes
    const int n8 = first + ((a.pos0 + tqc + 1 - first) & ~7);
    const int nkeys = a.pos0 + min(t0 + QB, a.T);
    const int64_t base = (int64_t)kvh * a.context * HD;
    const int split = MODE == ATTN_ALL ? 0 : (int)blockIdx.y;
    const int j_step = (MODE == ATTN_ALL ? W : W * a.splits) * KSTEP;
    const int j_first = jstart + (split * W + wv) * KSTEP;

    // pass 1: the queries' maxima over this wavefront's keys
    float m = -INFINITY;
    if constexpr (MODE != ATTN_SUM) {
        typename A::KFrag cur, nxt;
        A::load_k(nxt, a.kcache, base, j_first, nkeys, lr, lk);
        for (int j0 = j_first; j0 < nkeys; j0 += j_step) {
            cur = nxt;
            A::load_k(nxt, a.kcache, base, j0 + j_step, nkeys, lr, lk);
#pragma unroll
            for (int kt = 0; kt < KT; kt++) {
                const f4 c = at.scores(cur, kt);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int key = j0 + kt * 16 + 4 * lk + r;
                    if (key <= last && key >= first) m = fmaxf(m, c[r]);
                }
            }
        }
    }
    float mq;
    if constexpr (MODE != ATTN_SUM) {
        m = fmaxf(m, fx(lane_xor16, m));
        m = fmaxf(m, fx(lane_xor32, m));
        if (lk == 0) mx[wv][lr] = m;
        __syncthreads();
        mq = mx[0][lr];
#pragma unroll
        for (int w = 1; w < W; w++) mq = fmaxf(mq, mx[w][lr]);
        if constexpr (MODE == ATTN_MAX) {
            if (tid < QB && tq < a.T) a.part_max[((int64_t)split * a.heads + h) * a.T + tq] = mq;
            return;
        }
    } else {
        mq = -INFINITY;
        for (int i = 0; i < a.splits; i++) mq = fmaxf(mq, a.part_max[((int64_t)i * a.heads + h) * a.T + tqc]);
    }

    // pass 2: the same scores, softmax numerators (ExpApprox on the vector
    // lanes, expf on the tail, VM:215-258), their sum and e . V
    const float P14 = 16384.0f;
    f4 acc[NC][DPL];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int j = 0; j < DPL; j++) acc[c][j] = f4{0.f, 0.f, 0.f, 0.f};
    float z = 0.f;
    typename A::KFrag kn, kf;
    typename A::VFrag vn, vf;
    A::load_k(kn, a.kcache, base, j_first, nkeys, lr, lk);
    A::load_v(vn, a.vcache, base, j_first, nkeys, lr, lk);
    for (int j0 = j_first; j0 < nkeys; j0 += j_step) {
        kf = kn;
        vf = vn;
        A::load_k(kn, a.kcache, base, j0 + j_step, nkeys, lr, lk);
        A::load_v(vn, a.vcache, base, j0 + j_step, nkeys, lr, lk);
        float ev[KT][4];
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            const f4 c = at.scores(kf, kt);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int key = j0 + kt * 16 + 4 * lk + r;
                float e = 0.f;
                if (key <= last && key >= first) {
#pragma clang fp contract(off)
                    const float x = c[r] - mq;
                    e = key < n8 ? exp_approx(x) : expf(x);
                }
                z += e;
                ev[kt][r] = e;
            }
        }
        if constexpr (F16) {
            h8 eh, el;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float xs = ev[(i >> 2) % KT][i & 3] * P14;
                const _Float16 hi = (_Float16)xs;
                eh[i] = hi;
                el[i] = (_Float16)(xs - (float)hi);
            }
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int j = 0; j < DPL; j++) {
                    v4u w;
#pragma unroll
                    for (int k = 0; k < 4; k++)
                        w[k] = __builtin_amdgcn_perm(vf.w[c][(2 * k + 1) % A::VK][j / 2], vf.w[c][(2 * k) % A::VK][j / 2],
                                                     j & 1 ? 0x07060302u : 0x05040100u);
                    const h8 vh = __builtin_bit_cast(h8, w);
                    acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(eh, vh, acc[c][j], 0, 0, 0);
                    acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(el, vh, acc[c][j], 0, 0, 0);
                }
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int c = 0; c < NC; c++)
#pragma unroll
                    for (int j = 0; j < DPL; j++)
                        acc[c][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                            ev[0][r], __uint_as_float(vf.w[c][r][j % A::VW]), acc[c][j], 0, 0, 0);
        }
    }

    // the wavefronts' sums, halving their number each round
#pragma unroll
    for (int s = W / 2; s >= 1; s /= 2) {
        __syncthreads();
        if (wv >= s && wv < 2 * s) {
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int j = 0; j < DPL; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) ob[wv - s][(c * DPL + j) * 4 + r][lane] = acc[c][j][r];
            ob[wv - s][NT * 4][lane] = z;
        }
        __syncthreads();
        if (wv < s) {
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int j = 0; j < DPL; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[c][j][r] += ob[wv][(c * DPL + j) * 4 + r][lane];
            z += ob[wv][NT * 4][lane];
        }
    }
    if (wv != 0) return;
    z = xor32_add(xor16_add(z));   // lanes lr, lr + 16, ... hold query lr's sum
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int ql = 4 * lk + r;
        const float zq = __shfl(z, ql, 64);
        const int t = t0 + ql;
        if (t < a.T) {
            const float inv = MODE == ATTN_SUM ? 1.0f : 1.0f / zq;
            float* const out = MODE == ATTN_SUM ? a.part_out + split * a.part_stride : a.out;
            if (MODE == ATTN_SUM && lr == 0) a.part_z[((int64_t)split * a.T + t) * a.heads + h] = zq;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                float* o = out + (int64_t)t * (a.heads * HD) + h * HD + 16 * DPL * c + DPL * lr;
#pragma unroll
                for (int j = 0; j < DPL; j++) o[j] = (F16 ? acc[c][j][r] * (1.0f / P14) : acc[c][j][r]) * inv;
            }
        }
    }
}

template <int HD, bool F16>
hipError_t launch_wave(const PfAttnArgs& a, hipStream_t s) {
    const unsigned grid = (unsigned)((a.T + QB - 1) / QB) * (unsigned)a.heads;
    // 8 wavefronts a workgroup where there is one workgroup a CU at most (128
    // tokens behind 3900: 88 us against 103 with 4), else 4 (256 tokens, 512
    // workgroups: 16 against 20)
    if (a.splits > 1) {
        pf_attn_wave_kernel<HD, F16, 8, ATTN_MAX><<<dim3(grid, a.splits), 512, 0, s>>>(a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        pf_attn_wave_kernel<HD, F16, 8, ATTN_SUM><<<dim3(grid, a.splits), 512, 0, s>>>(a);
    } else if (grid <= 256) {
        pf_attn_wave_kernel<HD, F16, 8, ATTN_ALL><<<grid, 512, 0, s>>>(a);
    } else {
        pf_attn_wave_kernel<HD, F16, 4, ATTN_ALL><<<grid, 256, 0, s>>>(a);
    }
    return hipGetLastError();
}

}  // namespace

int prefill_attn_splits(int T, int pos0, int heads, int kv_fp16, int window) {
    const int wgs = (T + QB - 1) / QB * heads;
    // where at least half of the CUs have no workgroup: 64 workgroups of 1823 keys
    // (23 tokens, 32 heads of 128) 42 us, in 4 splits 10 + 15; with a workgroup
    // on every CU the row loads are already spread
    if (wgs > 128) return 1;
    // steps of 32 (16) keys per wavefront; two are left to each
    const int keys = window > 0 ? std::min(pos0 + T, window + QB) : pos0 + T, step = kv_fp16 ? 32 : 16;
    const int per_wave = (keys + 8 * step - 1) / (8 * step);
    return std::max(1, std::min({16, 256 / wgs, per_wave / 2}));
}

hipError_t launch_prefill_attn_wave(const PfAttnArgs& a, hipStream_t s) {
    if (a.splits > 1 && (!a.part_max || !a.part_out || !a.part_z || a.part_stride < (int64_t)a.T * a.heads * a.head_dim))
        return hipErrorInvalidValue;
    if (!a.kv_fp16 && a.window > 0) return hipErrorInvalidValue;
    switch (a.head_dim) {
    case 64: return a.kv_fp16 ? launch_wave<64, true>(a, s) : launch_wave<64, false>(a, s);
    case 96: return a.kv_fp16 ? launch_wave<96, true>(a, s) : launch_wave<96, false>(a, s);
    case 128: return a.kv_fp16 ? launch_wave<128, true>(a, s) : launch_wave<128, false>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace llmdot
