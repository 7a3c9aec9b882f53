// Flash-attention forward for gfx950: O = softmax(Q K^T * scale) V and the
// per-row log-sum-exp, one pass over K/V with an online softmax.
//
// Follows the algorithm of attention_flash.cu:17-89 (online softmax, causal
// tile break, LSE = m + ln l at :85-87), re-tiled for CDNA4:
//   * workgroup = 4 waves = 128 queries of one (batch, head); each wave owns
//     32 queries, whose Q rows sit in registers as MFMA B operands (64 and
//     16 on grids too small to fill the GPU otherwise);
//   * K/V advance 64 keys per stage through double-buffered LDS, filled by
//     direct global->LDS loads issued one stage ahead;
//   * scores are computed transposed, S^T = K Q^T, so each lane owns one query
//     column: the running max / sum stay per lane and only the max needs a
//     cross-lane reduction (two permlane swaps);
//   * the output is accumulated transposed, O^T = V^T P^T, so the per-query
//     rescale factor is a per-lane scalar as well;
//   * exponentials are base 2: the fp32 scores are multiplied by scale
//     log2(e) (bf16, which keeps Q exact) or Q is (fp32, fwd_split_entry);
//   * after the first stage the running max is only raised (and O and the sum
//     rescaled) when some p of a row exceeds 2^16 (fwd_stage_lazy), detected
//     from the per-lane row sums without computing a row maximum;
//   * only stages that straddle the causal diagonal or the end of the sequence
//     run the masking code (a separate instantiation of the stage body).
#include <type_traits>

#include "fa_device.h"
#include "fa_launch.h"

namespace mxfa {

// Masking of a stage's scores, one compare per score: key k0 + 32 blk +
// bidx(t, g, r) is masked when it is past the lane's query position (causal)
// or past the last key, i.e. when its offset from the lane's first key of the
// stage, 32 blk + bidx(t, g, r) - bidx(0, g, 0) (a compile-time constant), is
// above the lane's limit below.
template <class Pol, bool CAUSAL>
__device__ __forceinline__ int fwd_mask_limit(int qpos, int k0, int Nk, int g) {
    return (CAUSAL ? min(qpos, Nk - 1) : Nk - 1) - k0 - Pol::bidx(0, g, 0);
}
template <class Pol>
__device__ __forceinline__ constexpr int fwd_mask_offset(int blk, int t, int g, int r) {
    return 32 * blk + Pol::bidx(t, g, r) - Pol::bidx(0, g, 0);
}

// One 64-key stage for one wave: scores in log2 units (x xmul: qf holds Q
// itself), online-softmax update,
// O^T += V^T P^T. PRIO: the matrix products run at raised wave priority.
// qpos0: position of the wave's first query row; Nk: key rows. EMPTY_ROWS:
// rows may have every key of the stage masked (a key split's first stage).
// after_k runs once K has been read, before_v before V is (fwd_few_entry's
// loads and waits).
struct FwdNothing {
    __device__ __forceinline__ void operator()() const {}
};
template <class Pol, int QT, bool CAUSAL, bool MASK, bool PRIO = false, bool EMPTY_ROWS = false,
          class AfterK = FwdNothing, class BeforeV = FwdNothing>
__device__ __forceinline__ void fwd_stage(f32x4 (&acc)[Pol::D / 16][QT], float (&m)[QT], float (&lsum)[QT],
                                          const typename Pol::Frag (&qf)[QT][Pol::NC],
                                          const typename Pol::T *sk, const typename Pol::T *sv, int k0, int qpos0,
                                          int Nk, int g, int l16, float xmul, AfterK after_k = {},
                                          BeforeV before_v = {}) {
    using Frag = typename Pol::Frag;
    constexpr int NC = Pol::NC, XT = Pol::D / 16;
    f32x4 s[2][2][QT];  // [block][t][qt]
    wave_priority<PRIO>(1);
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            Frag a[NC];
            Pol::lds_row_frags(a, sk, 32 * blk + Pol::arow(t, l16), g);
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                f32x4 c = zero4();
#pragma unroll
                for (int kc = 0; kc < NC; ++kc) c = Pol::mma(a[kc], qf[qt][kc], c);
                s[blk][t][qt] = c;
            }
        }
    }
    wave_priority<PRIO>(0);
    after_k();
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int lim = fwd_mask_limit<Pol, CAUSAL>(qpos0 + 16 * qt + l16, k0, Nk, g);
        float mx = -INFINITY;
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = s[blk][t][qt][r] * xmul;
                    if constexpr (MASK) v = fwd_mask_offset<Pol>(blk, t, g, r) > lim ? -INFINITY : v;
                    s[blk][t][qt][r] = v;
                    mx = fmaxf(mx, v);
                }
            }
        }
        mx = xg_max(mx);
        const float mnew = fmaxf(m[qt], mx);
        // a row with every key of the stage masked keeps m = -inf and gets
        // p = 0 (2^(-inf - 0)), not 2^(-inf - -inf) = NaN
        const float mref = EMPTY_ROWS && mnew == -INFINITY ? 0.f : mnew;
        const float corr = fast_exp2(m[qt] - mref);
        m[qt] = mnew;
        float ls = lsum[qt] * corr;
#pragma unroll
        for (int xt = 0; xt < XT; ++xt) acc[xt][qt] *= corr;
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float pv = fast_exp2(s[blk][t][qt][r] - mref);
                    s[blk][t][qt][r] = pv;
                    ls += pv;
                }
            }
        }
        lsum[qt] = ls;
    }
    before_v();
    wave_priority<PRIO>(1);
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
        typename Pol::ChainB cb[QT];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) cb[qt] = Pol::pack(s[blk][0][qt], s[blk][1][qt]);
#pragma unroll
        for (int xt = 0; xt < XT; ++xt) {
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                acc[xt][qt] = Pol::chain(acc[xt][qt], cb[qt], sv, 16 * xt, 32 * blk, g, l16);
            }
        }
    }
    wave_priority<PRIO>(0);
}

// fwd_stage for every stage after the first, with lazy rescaling. Key 0 is
// visible to every query (pos0 >= 0), so after the first stage m is finite for
// every row; a key split's work-group may leave a row at m = -inf after its
// first stage only when the row precedes every key of the split (causal), so
// every later stage masks the whole row (p = 0, nothing to rescale). The scores come out of the MFMAs relative to the running max m
// (the accumulators start at -m), and p = 2^(s - m) is taken optimistically
// with the old m. A lane's per-row sum of its p over the stage (16 keys)
// bounds each of them, so when no such sum exceeds kLazySum no p does either:
// O and the row sums then simply accumulate (m stays within log2(kLazySum) of
// the row's true running max, so nothing overflows or underflows in fp32 and
// the largest p of a row stays in [1, kLazySum]). Otherwise (an overflow shows
// as an infinite sum) the stage is redone exactly: the scores are recomputed
// from LDS, m rises to the row's max, O and the sum are rescaled, and the
// exponentials are taken again. LSE = m + log2(l) holds for any m used
// consistently, so the result is the online softmax's up to rounding. No row
// maximum is computed on the common path.
constexpr float kLazySum = 65536.0f;

// Scores of one 64-key stage relative to m: s = K Q^T scale log2(e) - m, with
// masked keys (MASK) at -inf: the accumulators start at -m / xmul and the
// fp32 result is multiplied by xmul = scale log2(e).
template <class Pol, int QT, bool CAUSAL, bool MASK, bool PRIO = false>
__device__ __forceinline__ void fwd_scores(f32x4 (&s)[2][2][QT], const float (&m)[QT],
                                           const typename Pol::Frag (&qf)[QT][Pol::NC], const typename Pol::T *sk,
                                           int k0, int qpos0, int Nk, int g, int l16, float xmul) {
    using Frag = typename Pol::Frag;
    constexpr int NC = Pol::NC;
    const float im = 1.0f / xmul;
    f32x4 nm[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const float n = -m[qt] * im;
        nm[qt] = f32x4{n, n, n, n};
    }
    wave_priority<PRIO>(1);
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            Frag a[NC];
            Pol::lds_row_frags(a, sk, 32 * blk + Pol::arow(t, l16), g);
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                f32x4 c = nm[qt];
#pragma unroll
                for (int kc = 0; kc < NC; ++kc) c = Pol::mma(a[kc], qf[qt][kc], c);
                s[blk][t][qt] = c * xmul;
            }
        }
    }
    wave_priority<PRIO>(0);
    if constexpr (MASK) {
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            const int lim = fwd_mask_limit<Pol, CAUSAL>(qpos0 + 16 * qt + l16, k0, Nk, g);
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (fwd_mask_offset<Pol>(blk, t, g, r) > lim) s[blk][t][qt][r] = -INFINITY;
                    }
                }
            }
        }
    }
}

// p = 2^s in place, added to l (row qt of this lane).
template <int QT>
__device__ __forceinline__ void fwd_exp_sum(f32x4 (&s)[2][2][QT], float (&l)[QT]) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        float ls = l[qt];
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float pv = fast_exp2(s[blk][t][qt][r]);
                    s[blk][t][qt][r] = pv;
                    ls += pv;
                }
            }
        }
        l[qt] = ls;
    }
}

template <class Pol, int QT, bool CAUSAL, bool MASK, bool PRIO = false>
__device__ __forceinline__ void fwd_stage_lazy(f32x4 (&acc)[Pol::D / 16][QT], float (&m)[QT], float (&lsum)[QT],
                                               const typename Pol::Frag (&qf)[QT][Pol::NC],
                                               const typename Pol::T *sk, const typename Pol::T *sv, int k0,
                                               int qpos0, int Nk, int g, int l16, float xmul) {
    constexpr int XT = Pol::D / 16;
    f32x4 s[2][2][QT];  // [block][t][qt]
    fwd_scores<Pol, QT, CAUSAL, MASK, PRIO>(s, m, qf, sk, k0, qpos0, Nk, g, l16, xmul);
    float l0[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) l0[qt] = lsum[qt];
    fwd_exp_sum(s, lsum);
    bool over = false;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) over = over || lsum[qt] > l0[qt] + kLazySum;
    if (__builtin_amdgcn_ballot_w64(over) != 0) {
        // some p of the wave exceeded kLazySum: redo the stage with m raised to
        // each row's max (rows whose max did not rise keep shift 0)
        fwd_scores<Pol, QT, CAUSAL, MASK, PRIO>(s, m, qf, sk, k0, qpos0, Nk, g, l16, xmul);
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            float v = -INFINITY;
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) v = fmaxf(v, s[blk][t][qt][r]);
                }
            }
            const float shift = fmaxf(xg_max(v), 0.f);
            const float corr = fast_exp2(-shift);
            m[qt] += shift;
#pragma unroll
            for (int xt = 0; xt < XT; ++xt) acc[xt][qt] *= corr;
            lsum[qt] = l0[qt] * corr;
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[blk][t][qt][r] -= shift;
                }
            }
        }
        fwd_exp_sum(s, lsum);
    }
    wave_priority<PRIO>(1);
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
        typename Pol::ChainB cb[QT];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) cb[qt] = Pol::pack(s[blk][0][qt], s[blk][1][qt]);
#pragma unroll
        for (int xt = 0; xt < XT; ++xt) {
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                acc[xt][qt] = Pol::chain(acc[xt][qt], cb[qt], sv, 16 * xt, 32 * blk, g, l16);
            }
        }
    }
    wave_priority<PRIO>(0);
}

// One work-group of the forward, grid (B Hq, query blocks). QT: 16-query
// tiles per wave (the work-group takes 64 QT queries); the kernels are
// compiled for a number of waves per SIMD (the names' w*). PAGED: K/V rows
// through Params::block_table (the kernels named *_pg). SPLIT (kernels *_sp,
// grid.z = the splits): work-group z takes stages [z nsteps / S, (z + 1)
// nsteps / S) of its query block's keys and writes its unnormalised O and
// its rows' running max and sum to Params::fwd_part; fwd_merge adds the
// splits.
template <class Pol, bool CAUSAL, int QT, bool PAGED = false, bool SPLIT = false>
__device__ __forceinline__ void fwd_entry(const Params &p) {
    using T = typename Pol::T;
    using Frag = typename Pol::Frag;
    constexpr int D = Pol::D, NC = Pol::NC, XT = D / 16;
    constexpr int BQ = 64 * QT, BK = Pol::ROWS;
    // the matrix products at raised wave priority, the softmax at normal
    // (A/B on one box: cfg4 78.1 -> 74.3 us, cfg5 d = 128 51.0 -> 47.2,
    // non-causal B2 H12 N4096 112.2 -> 109.7; the 64-query d = 64 launches
    // lost 1-3% with it)
    constexpr bool kPrio = QT == 2 || D == 128;

    __shared__ __attribute__((aligned(16))) T sK[2][BK * D];
    __shared__ __attribute__((aligned(16))) T sV[2][BK * D];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, l16 = lane & 15;
    const int N = p.N, Nk = p.Nk, pos0 = p.pos0;
    const int nqb = (N + BQ - 1) / BQ;
    // causal: heaviest first, in the order balanced per CU over the work-groups
    // resident at once (cu_order_wg; ranks are heads fastest)
    const int rank = CAUSAL ? cu_order_wg((int)(blockIdx.y * gridDim.x + blockIdx.x), p.cu_run, p.cu_runs)
                            : (int)(blockIdx.y * gridDim.x + blockIdx.x);
    const int bh = rank % (int)gridDim.x;
    const int qb = CAUSAL ? nqb - 1 - rank / (int)gridDim.x : rank / (int)gridDim.x;
    const int b = bh / p.Hq, h = bh % p.Hq, kvh = h / p.group;
    const T *Q = static_cast<const T *>(p.q) + b * p.q_bs + h * p.q_hs;
    const size_t kvoff = b * p.kv_bs + kvh * p.kv_hs;
    const T *K = static_cast<const T *>(p.k) + kvoff;
    const T *V = static_cast<const T *>(p.v) + kvoff;
    const int q0 = qb * BQ + wave * 16 * QT;
    const int qpos0 = pos0 + q0;  // position of the wave's first query row
    wg_time(0);

    Frag qf[QT][NC];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) Pol::gmem_row_frags(qf[qt], Q, q0 + 16 * qt + l16, N, p.q_rs, g);
    f32x4 acc[XT][QT];
    float m[QT], lsum[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
#pragma unroll
        for (int xt = 0; xt < XT; ++xt) acc[xt][qt] = zero4();
        m[qt] = -INFINITY;
        lsum[qt] = 0.f;
    }

    const int kend = CAUSAL ? min(Nk, pos0 + qb * BQ + BQ) : Nk;
    const int nsteps = (kend + BK - 1) / BK;
    // this work-group's stages [s_lo, s_hi) (SPLIT: its share; the first one
    // it runs takes the plain softmax body, the running max starting at -inf)
    const int s_lo = SPLIT ? (int)((long long)blockIdx.z * nsteps / gridDim.z) : 0;
    const int s_hi = SPLIT ? (int)((long long)(blockIdx.z + 1) * nsteps / gridDim.z) : nsteps;
    wg_info(2, qb, s_hi - s_lo);

    const RowPlan<Pol> plan(tid);
    // PAGED: the table entries of stage 0 now, then each stage fetches those
    // of the stage after the one it stages
    PagedRows<Pol> paged;
    auto stage_next = [&](T *sk, T *sv, int k0) __attribute__((always_inline)) {
        if constexpr (PAGED) {
            paged.stage(sk, sv, K, V, k0, Nk, p.bs_shift, plan, wave, p.kv_rs);
            if (k0 + BK < Nk) paged.fetch(p.block_table, p.bs_shift, k0 + BK, Nk, plan);
        } else {
            stage_kv<Pol>(sk, sv, K, V, k0, Nk, plan, wave, p.kv_rs);
        }
    };
    if (!SPLIT || s_lo < s_hi) {
        if constexpr (PAGED) paged.fetch(p.block_table, p.bs_shift, s_lo * BK, Nk, plan);
        stage_next(sK[0], sV[0], s_lo * BK);
    }
    wait_stage();
    __syncthreads();
    wg_time(1);

    // Leading stages that no wave masks (all their keys exist and precede the
    // workgroup's first query position) run in pairs with the LDS buffer a
    // compile-time constant, so the tile addresses fold into the instructions'
    // immediate offsets; the rest choose buffer and masking at run time.
    // The first stage runs the plain online-softmax body (the running max
    // starts at -inf); later ones the lazy-rescaling body.
    auto main_stage = [&](auto buf, auto first, int st) __attribute__((always_inline)) {
        constexpr int B = decltype(buf)::value;
        if (st + 1 < s_hi) stage_next(sK[B ^ 1], sV[B ^ 1], (st + 1) * BK);
        if constexpr (decltype(first)::value) {
            fwd_stage<Pol, QT, CAUSAL, false, kPrio>(acc, m, lsum, qf, sK[B], sV[B], st * BK, qpos0, Nk, g, l16,
                                                     p.scale_log2);
        } else {
            fwd_stage_lazy<Pol, QT, CAUSAL, false, kPrio>(acc, m, lsum, qf, sK[B], sV[B], st * BK, qpos0, Nk, g, l16,
                                                          p.scale_log2);
        }
        wait_stage();
        __syncthreads();
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    const int nmain = min(min(s_hi, Nk / BK), CAUSAL ? (pos0 + qb * BQ + 1) / BK : s_hi);
    int st = s_lo;
    if (nmain > st) main_stage(B0{}, std::true_type{}, st++);
    for (; st + 1 < nmain; st += 2) {
        main_stage(B1{}, std::false_type{}, st);
        main_stage(B0{}, std::false_type{}, st + 1);
    }
    if (st < nmain) main_stage(B1{}, std::false_type{}, st++);
    // the remaining stages may straddle the diagonal or the end of the keys:
    // one masked body each for the first stage and the later ones (a wave
    // that skips a stage skips every later one, so its first run stage is
    // the work-group's first)
    for (; st < s_hi; ++st) {
        const int cur = (st - s_lo) & 1;
        if (st + 1 < s_hi) stage_next(sK[cur ^ 1], sV[cur ^ 1], (st + 1) * BK);
        const int k0 = st * BK;
        // a wave whose queries all precede the stage's keys has nothing to do
        if (!CAUSAL || k0 <= qpos0 + 16 * QT - 1) {
            if (st == s_lo) {
                fwd_stage<Pol, QT, CAUSAL, true, kPrio, SPLIT>(acc, m, lsum, qf, sK[cur], sV[cur], k0, qpos0, Nk, g,
                                                               l16, p.scale_log2);
            } else {
                fwd_stage_lazy<Pol, QT, CAUSAL, true, kPrio>(acc, m, lsum, qf, sK[cur], sV[cur], k0, qpos0, Nk, g, l16,
                                                             p.scale_log2);
            }
        }
        wait_stage();
        __syncthreads();
    }

    wg_time(2);
    if constexpr (SPLIT) {
        // the split's partial: O unnormalised, then (running max, sum) per row
        const size_t rows = (size_t)gridDim.z * p.B * p.Hq * N;
        const size_t r0 = ((size_t)blockIdx.z * p.B * p.Hq + bh) * N;
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            const int qi = q0 + 16 * qt + l16;
            const float ltot = xg_sum(lsum[qt]);
            if (qi < N) {
                float *po = p.fwd_part + (r0 + qi) * D;
#pragma unroll
                for (int xt = 0; xt < XT; ++xt) store4<float>(po + 16 * xt + 4 * g, acc[xt][qt], 1.0f);
                if (g == 0) {
                    float *pml = p.fwd_part + rows * D + 2 * (r0 + qi);
                    *reinterpret_cast<float2 *>(pml) = make_float2(m[qt], ltot);
                }
            }
        }
        wg_time_after_stores();
        return;
    }
    T *O = static_cast<T *>(p.o) + b * p.o_bs + h * p.o_hs;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int qi = q0 + 16 * qt + l16;
        const float ltot = xg_sum(lsum[qt]);
        const float inv = 1.0f / ltot;
        // 16 bytes per lane (rows start on 16-byte boundaries)
        T *row = O + (size_t)min(qi, N - 1) * p.o_rs;
#pragma unroll
        for (int xt = 0; xt < XT; xt += 2)
            store8_pair_bf16(row, 16 * xt, g, acc[xt][qt], acc[xt + 1][qt], inv, qi < N);
        if (qi < N && p.lse != nullptr && g == 0) p.lse[(size_t)bh * N + qi] = (m[qt] + fast_log2(ltot)) * kLn2;
    }
    wg_time_after_stores();
}

// The forward of a few query rows (at most 16 per head: a token's GQA group, or
// a handful of tokens) over a KV cache, bf16. All NW waves hold the same rows;
// each takes 64-key stages of its own (the work-group's stages [s_lo, s_hi),
// every NW-th), staged into its own LDS tiles with no barrier between waves, and
// the waves' running maxima, sums and O are merged through LDS at the end.
//
// Bound: the loads. A work-group has NW x 64 keys of K and V in flight (128 KB,
// one work-group per CU), where the 64-query form holds one stage ahead and
// leaves three of its four waves without rows. Kernel-trace medians of one
// token with its keys split, us: 14/2 heads after 65535 20.2 -> 9.0 (3.7 TB/s;
// 128 splits instead of 32), 32/4 heads after 4095, paged, 5.0 -> 4.6.
constexpr int kFewRows = 16;

template <class Pol, int NW>
union FwdFewSmem {
    struct {
        typename Pol::T k[NW][Pol::ROWS * Pol::D], v[NW][Pol::ROWS * Pol::D];
    } t;
    struct {
        float acc[NW][kFewRows][Pol::D + 4];
        float ml[NW][kFewRows][2];
    } merge;
};

template <class Pol, int NW, bool PAGED, bool SPLIT>
__device__ __forceinline__ void fwd_few_entry(const Params &p) {
    using T = typename Pol::T;
    constexpr int D = Pol::D, XT = D / 16, BK = Pol::ROWS;
    __shared__ __attribute__((aligned(16))) FwdFewSmem<Pol, NW> sm;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, l16 = lane & 15;
    const int N = p.N, Nk = p.Nk, bh = blockIdx.x;
    const int b = bh / p.Hq, h = bh % p.Hq, kvh = h / p.group;
    const size_t kvoff = b * p.kv_bs + kvh * p.kv_hs;
    const T *K = static_cast<const T *>(p.k) + kvoff, *V = static_cast<const T *>(p.v) + kvoff;
    T *sk = sm.t.k[wave], *sv = sm.t.v[wave];
    wg_time(0);
    const int nsteps = (min(Nk, p.pos0 + N) + BK - 1) / BK;
    const int s_lo = SPLIT ? (int)((long long)blockIdx.z * nsteps / gridDim.z) : 0;
    const int s_hi = SPLIT ? (int)((long long)(blockIdx.z + 1) * nsteps / gridDim.z) : nsteps;
    wg_info(2, 0, s_hi - s_lo);

    const RowPlan<Pol, 64> plan(lane);
    PagedRows<Pol, 64> paged;
    constexpr int NL = RowPlan<Pol, 64>::NK;  // loads of a tile
    auto load = [&](T *tile, const T *base, int st) __attribute__((always_inline)) {
        if constexpr (PAGED) {
            paged.stage_one(tile, base, st * BK, Nk, p.bs_shift, plan, 0, p.kv_rs);
        } else {
            stage_rows<Pol, 64>(tile, base + (size_t)(st * BK) * p.kv_rs, Nk - st * BK, plan, 0, p.kv_rs);
        }
    };
    auto fetch = [&](int st) __attribute__((always_inline)) {
        if constexpr (PAGED) paged.fetch(p.block_table, p.bs_shift, st * BK, Nk, plan);
    };
    int st = s_lo + wave;
    if (st < s_hi) {
        fetch(st);
        load(sk, K, st);
        load(sv, V, st);
    }
    typename Pol::Frag qf[1][Pol::NC];
    Pol::gmem_row_frags(qf[0], static_cast<const T *>(p.q) + b * p.q_bs + h * p.q_hs, l16, N, p.q_rs, g);
    f32x4 acc[XT][1];
#pragma unroll
    for (int xt = 0; xt < XT; ++xt) acc[xt][0] = zero4();
    float m[1] = {-INFINITY}, lsum[1] = {0.f};
    // The wave's next stage: its K goes out once this one's K has been read, its
    // V once this one's V has, so one tile is in flight at any time. At least
    // NL loads follow K's when it is waited for (this stage's V), and V's (the
    // next K): vmcnt counts in order.
    for (; st < s_hi; st += NW) {
        const bool more = st + NW < s_hi;
        if (more) fetch(st + NW);
        wait_loads<NL>();
        fwd_stage<Pol, 1, true, true, false, true>(
            acc, m, lsum, qf, sk, sv, st * BK, p.pos0, Nk, g, l16, p.scale_log2,
            [&]() __attribute__((always_inline)) {
                wait_lds();
                if (more) load(sk, K, st + NW);
            },
            [&]() __attribute__((always_inline)) {
                if (more) {
                    wait_loads<NL>();
                } else {
                    wait_loads<0>();
                }
            });
        wait_lds();
        if (more) load(sv, V, st + NW);
    }
    const float lw = xg_sum(lsum[0]);
    __syncthreads();  // every wave is done with the tiles
    wg_time(2);
#pragma unroll
    for (int xt = 0; xt < XT; ++xt)
        *reinterpret_cast<f32x4 *>(&sm.merge.acc[wave][l16][16 * xt + 4 * g]) = acc[xt][0];
    if (g == 0) *reinterpret_cast<float2 *>(sm.merge.ml[wave][l16]) = make_float2(m[0], lw);
    __syncthreads();
    for (int i = tid; i < N * (D / 4); i += 64 * NW) {
        const int r = i / (D / 4), c = 4 * (i % (D / 4));
        float M = -INFINITY, L = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) M = fmaxf(M, sm.merge.ml[w][r][0]);
        const float mref = M == -INFINITY ? 0.f : M;  // a split with no key of the row: weight 0
        f32x4 o = zero4();
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float x = fast_exp2(sm.merge.ml[w][r][0] - mref);
            L += x * sm.merge.ml[w][r][1];
            o += *reinterpret_cast<const f32x4 *>(&sm.merge.acc[w][r][c]) * x;
        }
        if constexpr (SPLIT) {
            const size_t rows = (size_t)gridDim.z * p.B * p.Hq * N;
            const size_t r0 = ((size_t)blockIdx.z * p.B * p.Hq + bh) * N + r;
            store4<float>(p.fwd_part + r0 * D + c, o, 1.0f);
            if (c == 0) *reinterpret_cast<float2 *>(p.fwd_part + rows * D + 2 * r0) = make_float2(M, L);
        } else {
            T *O = static_cast<T *>(p.o) + b * p.o_bs + h * p.o_hs + (size_t)r * p.o_rs;
            store4<T>(O + c, o, 1.0f / L);
            if (p.lse != nullptr && c == 0) p.lse[(size_t)bh * N + r] = (M + fast_log2(L)) * kLn2;
        }
    }
    wg_time_after_stores();
}

// The fp32 forward (d = 64) with its products in bf16 parts (Split3): NW waves
// of 16 queries, 64 keys per stage. K and V pass through registers, loaded one
// stage ahead, and are split once per work-group into one 48 KB LDS buffer;
// NW = 4: three work-groups per CU (162 VGPRs), NW = 8: two (114 VGPRs), whose
// splitting, softmax and products overlap.
//
// Bound: a wave's stage is 96 MFMAs (1536 cycles, each hiding two VALU
// instructions), 48 KB of LDS reads and about 340 (NW = 4) or 250 VALU
// instructions, over half of them the splitting. Event medians on one card,
// us, against v_mfma_f32_16x16x4_f32 on the same tiles: causal B4 H12 N1024
// 79.5 -> 54, B4 H12 N4096 806 -> 523 (197 TFLOP/s), non-causal B1 H12 N4096
// 411 -> 318, B1 H1 N256 16.0 -> 14.1. Error of O against 64 bits: causal
// N1000 3.4e-7 -> 2.1e-7, N4096 5.1e-7 -> 3.8e-7, non-causal N4096 1.2e-6 ->
// 1.0e-6, N256 4.4e-7 -> 2.6e-7. Two 16-query tiles per wave, the waves in pairs over half a stage's
// keys each (half the LDS reads) ran 54.6, 570, 338 and 14.6: 250 VGPRs leave
// two waves per SIMD.
struct FwdSplitSmem {
    SplitTile k, v;
    uint32_t flags[8];
};

// The work-group's rows again in plain fp32 arithmetic, for operands outside
// the parts' range: thread t takes elements 16 (t % 4) .. + 15 of row t / 4.
template <int NW, bool CAUSAL, bool PAGED, bool SPLIT>
__device__ __forceinline__ void fwd_plain(const Params &p, int bh, int qb, int key0, int key1) {
    constexpr int D = 64;
    const int qi = qb * 16 * NW + (int)(threadIdx.x >> 2), c = 16 * (int)(threadIdx.x & 3), row = min(qi, p.N - 1);
    const int b = bh / p.Hq, h = bh % p.Hq, kvh = h / p.group;
    const float *Q = static_cast<const float *>(p.q) + b * p.q_bs + h * p.q_hs + (size_t)row * p.q_rs + c;
    const size_t kvoff = b * p.kv_bs + kvh * p.kv_hs + c;
    float q[16], acc[16], m = -INFINITY, l = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        q[e] = Q[e] * p.scale_log2;
        acc[e] = 0.f;
    }
    const int kend = min(key1, CAUSAL ? min(p.Nk, p.pos0 + row + 1) : p.Nk);  // the same for a row's 4 threads
    for (int k = key0; k < kend; ++k) {
        size_t r = k;
        if constexpr (PAGED) r = ((size_t)p.block_table[k >> p.bs_shift] << p.bs_shift) + (k & ((1 << p.bs_shift) - 1));
        const float *K = static_cast<const float *>(p.k) + kvoff + r * (size_t)p.kv_rs;
        const float *V = static_cast<const float *>(p.v) + kvoff + r * (size_t)p.kv_rs;
        const float s = dot16(q, K), mn = fmaxf(m, s), mref = mn == -INFINITY ? 0.f : mn;
        const float corr = fast_exp2(m - mref), pv = fast_exp2(s - mref);
        m = mn;
        l = l * corr + pv;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = __builtin_fmaf(pv, V[e], acc[e] * corr);
    }
    if (qi >= p.N) return;
    if constexpr (SPLIT) {
        const size_t rows = (size_t)gridDim.z * p.B * p.Hq * p.N;
        const size_t r0 = ((size_t)blockIdx.z * p.B * p.Hq + bh) * p.N + qi;
#pragma unroll
        for (int e = 0; e < 16; ++e) p.fwd_part[r0 * D + c + e] = acc[e];
        if (c == 0) *reinterpret_cast<float2 *>(p.fwd_part + rows * D + 2 * r0) = make_float2(m, l);
    } else {
        float *O = static_cast<float *>(p.o) + b * p.o_bs + h * p.o_hs + (size_t)qi * p.o_rs + c;
#pragma unroll
        for (int e = 0; e < 16; ++e) O[e] = acc[e] / l;
        if (p.lse != nullptr && c == 0) p.lse[(size_t)bh * p.N + qi] = (m + fast_log2(l)) * kLn2;
    }
}

template <int NW, bool CAUSAL, bool PAGED, bool SPLIT>
__device__ __forceinline__ void fwd_split_entry(const Params &p) {
    constexpr int D = 64, XT = 4, BQ = 16 * NW, BK = 64, NT = 64 * NW;
    using PL = PolBF16<64>;  // the parts' layout
    using Stage = SplitStage<NT>;
    __shared__ FwdSplitSmem sm;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, l16 = lane & 15;
    const int N = p.N, Nk = p.Nk, pos0 = p.pos0;
    const int nqb = (N + BQ - 1) / BQ;
    const int rank = CAUSAL ? cu_order_wg((int)(blockIdx.y * gridDim.x + blockIdx.x), p.cu_run, p.cu_runs)
                            : (int)(blockIdx.y * gridDim.x + blockIdx.x);
    const int bh = rank % (int)gridDim.x;
    const int qb = CAUSAL ? nqb - 1 - rank / (int)gridDim.x : rank / (int)gridDim.x;
    const int b = bh / p.Hq, h = bh % p.Hq, kvh = h / p.group;
    const size_t kvoff = b * p.kv_bs + kvh * p.kv_hs;
    const float *K = static_cast<const float *>(p.k) + kvoff;
    const float *V = static_cast<const float *>(p.v) + kvoff;
    const int q0 = qb * BQ + wave * 16, qi = q0 + l16;
    wg_time(0);

    const int nsteps = ((CAUSAL ? min(Nk, pos0 + qb * BQ + BQ) : Nk) + BK - 1) / BK;
    const int s_lo = SPLIT ? (int)((long long)blockIdx.z * nsteps / gridDim.z) : 0;
    const int s_hi = SPLIT ? (int)((long long)(blockIdx.z + 1) * nsteps / gridDim.z) : nsteps;
    wg_info(2, qb, s_hi - s_lo);

    // this thread's chunks of a tile: row and first column
    int srow[Stage::NK], scol[Stage::NK], blk[Stage::NK];
#pragma unroll
    for (int k = 0; k < Stage::NK; ++k) {
        PL::chunk_at(k * NT + tid, srow[k], scol[k]);
        scol[k] *= 8;
    }
    // rows past the last key re-read it (their scores are masked)
    auto fetch = [&](int st) __attribute__((always_inline)) {
        if constexpr (PAGED) {
#pragma unroll
            for (int k = 0; k < Stage::NK; ++k) blk[k] = p.block_table[min(st * BK + srow[k], Nk - 1) >> p.bs_shift];
        }
    };
    Stage xk, xv;
    auto load = [&](int st) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < Stage::NK; ++k) {
            const int t = min(st * BK + srow[k], Nk - 1);
            const size_t row = PAGED ? ((size_t)blk[k] << p.bs_shift) + (size_t)(t & ((1 << p.bs_shift) - 1)) : (size_t)t;
            const size_t off = row * (size_t)p.kv_rs + scol[k];
            xk.load(k, K + off);
            xv.load(k, V + off);
        }
        if (st + 1 < s_hi) fetch(st + 1);
    };
    if (s_lo < s_hi) {
        fetch(s_lo);
        load(s_lo);
    }

    Split3 qf[1][2];
    const bool low = split_row(qf[0], static_cast<const float *>(p.q) + b * p.q_bs + h * p.q_hs + (size_t)min(qi, N - 1) * p.q_rs,
                               g, p.scale_log2 * kPartDown, qi < N);
    f32x4 acc[XT];
#pragma unroll
    for (int xt = 0; xt < XT; ++xt) acc[xt] = zero4();
    float m = -INFINITY, lsum = 0.f;

    // One stage: the online softmax of fwd_stage (FIRST) or, after the
    // work-group's first stage, fwd_stage_lazy's: m raised only where a lane's sum
    // of p passes kLazySum. m is subtracted from the finished sums: started at -m,
    // they are rounded at its size, and not evenly up and down, so the splits of a
    // long context got weights that were off. kApart: a stage's part of O is summed
    // from zero and added once, instead of 12 roundings at O's size. Error of O,
    // relative, rms over 24 draws, with neither, the first, both: one token after
    // 65535 9.8e-7, 9.1e-7, 3.0e-7 (the fp32 matrix instructions 8.8e-7), after
    // 4095 3.5e-7, 2.2e-7, 1.9e-7 (4.0e-7). kApart costs 3% of a call and the wide
    // form's registers (12 to 24 spilled, 49 -> 58 us for 500 tokens after 3584),
    // where 3.5e-7 against 6.1e-7 is enough without. A row that precedes
    // every key of the first stage (a key split) has m = -inf, and then
    // precedes all later ones too; with finite operands whose first scores all
    // overflow to -inf it does not, and the rows are run again (below).
    constexpr bool kApart = SPLIT && NW == 4;
    auto compute = [&](auto first, bool edge, int k0) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first)::value;
        f32x4 s[2][2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                Split3 a[1][2];
                f32x4 c[1][1] = {{zero4()}};
                sm.k.row_frags(a[0], 32 * u + PL::arow(t, l16), g);
                mma_split_tiles<2, 1, 1>(c, a, qf);
                s[u][t] = c[0][0];
            }
        }
        if (edge) {
            const int lim = (CAUSAL ? min(pos0 + qi, Nk - 1) : Nk - 1) - k0 - PL::bidx(0, g, 0);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (32 * u + PL::bidx(t, 0, r) > lim) s[u][t][r] = -INFINITY;
                    }
                }
            }
        }
        const float base = m == -INFINITY ? 0.f : m;  // what p is relative to
        f32x4 pv[2][2];
        auto exps = [&](float sub) __attribute__((always_inline)) {
            float ls = 0.f;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float e = fast_exp2(s[u][t][r] - sub);
                        pv[u][t][r] = e;
                        ls += e;
                    }
                }
            }
            return ls;
        };
        auto raise = [&]() __attribute__((always_inline)) {  // m to the stage's max, O and the sum rescaled
            float mx = -INFINITY;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[u][t][r]);
                }
            }
            mx = fmaxf(xg_max(mx), m);
            const float to = mx == -INFINITY ? 0.f : mx;
            if constexpr (!FIRST) {
                const float corr = fast_exp2(base - to);
                lsum *= corr;
#pragma unroll
                for (int xt = 0; xt < XT; ++xt) acc[xt] *= corr;
            }
            m = mx;
            lsum += exps(to);
        };
        if constexpr (FIRST) {
            raise();
        } else {
            const float ls = exps(base);
            if (__builtin_amdgcn_ballot_w64(ls > kLazySum) != 0) {
                raise();
            } else {
                lsum += ls;
            }
        }
        if constexpr (kApart) {
            const Split3 pf[2][1] = {{split3(pv[0][0], pv[0][1])}, {split3(pv[1][0], pv[1][1])}};
#pragma unroll
            for (int xt = 0; xt < XT; ++xt) {
                f32x4 c = zero4();
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const Split3 a[1] = {sm.v.chain_a(16 * xt, 32 * u, g, l16)};
                    c = mma_split<1>(a, pf[u], c);
                }
                acc[xt] += c;
            }
        } else {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const Split3 pf[1] = {split3(pv[u][0], pv[u][1])};
#pragma unroll
                for (int xt = 0; xt < XT; ++xt) {
                    const Split3 a[1] = {sm.v.chain_a(16 * xt, 32 * u, g, l16)};
                    acc[xt] = mma_split<1>(a, pf, acc[xt]);
                }
            }
        }
    };
    // stages from `nmain` on have keys that some wave masks; a wave whose
    // queries all precede a stage's keys skips it, and every later one
    const int nmain = min(Nk / BK, CAUSAL ? (pos0 + qb * BQ + 1) / BK : nsteps);
    auto stage = [&](auto first, int st) __attribute__((always_inline)) {
        if (st > s_lo) barrier_lds();  // every wave is done with the stage before
        xk.write(sm.k, tid);
        xv.write(sm.v, tid);
        if (st + 1 < s_hi) load(st + 1);
        barrier_lds();
        if (!CAUSAL || st * BK <= pos0 + q0 + 15) compute(first, st >= nmain, st * BK);
    };
    if (s_lo < s_hi) stage(std::true_type{}, s_lo);
    wg_time(1);
    for (int st = s_lo + 1; st < s_hi; ++st) stage(std::false_type{}, st);
    wg_time(2);

    const float ltot = xg_sum(lsum);
    float z = 0.f * ltot;
#pragma unroll
    for (int xt = 0; xt < XT; ++xt) z += zero_of(acc[xt]);
    // a row with keys here whose first stage's scores all overflowed to -inf: m
    // stayed there, and O and the sum hold the later stages relative to 0
    if (m == -INFINITY && s_lo < s_hi && (!CAUSAL || s_lo * BK <= pos0 + qi)) z = NAN;
    if (low) z = NAN;
    if (any_nonfinite<NW>(z, sm.flags, wave, lane)) {
        fwd_plain<NW, CAUSAL, PAGED, SPLIT>(p, bh, qb, s_lo * BK, s_hi * BK);
    } else if (qi < N) {
        if constexpr (SPLIT) {
            const size_t rows = (size_t)gridDim.z * p.B * p.Hq * N;
            const size_t r0 = ((size_t)blockIdx.z * p.B * p.Hq + bh) * N + qi;
#pragma unroll
            for (int xt = 0; xt < XT; ++xt) store4<float>(p.fwd_part + r0 * D + 16 * xt + 4 * g, acc[xt], kPartDown);
            if (g == 0) *reinterpret_cast<float2 *>(p.fwd_part + rows * D + 2 * r0) = make_float2(m, ltot);
        } else {
            float *O = static_cast<float *>(p.o) + b * p.o_bs + h * p.o_hs + (size_t)qi * p.o_rs;
            const float inv = kPartDown / ltot;
#pragma unroll
            for (int xt = 0; xt < XT; ++xt) store4<float>(O + 16 * xt + 4 * g, acc[xt], inv);
            if (p.lse != nullptr && g == 0) p.lse[(size_t)bh * N + qi] = (m + fast_log2(ltot)) * kLn2;
        }
    }
    wg_time_after_stores();
}

// Adds the S key splits of a split forward (fwd_entry<..., SPLIT>): with M the
// largest of the splits' running maxima (log2 units), O = sum_s 2^(m_s - M)
// O_s / sum_s 2^(m_s - M) l_s, written as the forward writes O. A split that
// holds no key of the row has m = -inf and weight 0. Two forms:
//  * one thread per four elements of a row, every split's loads issued before
//    the first is used, so a call costs one memory latency (fwd_merge_body;
//    MAXS = 8 keeps the registers of the common case low, the 32-split form
//    takes 205): up to kMergeThread splits, and more with many rows;
//  * a work-group per row, its groups of threads over the splits
//    (fwd_merge_row_body), for more splits of at most kMergeRow elements of O:
//    with a thread per four elements one token's 32 rows are two work-groups, each
//    reading 131 KB (32 splits 4.7 -> 3.1 us; the 128 splits of 14 rows 3.6).
// The line, us a call, a work-group per row against a thread per four elements:
// d = 64, 1000 rows of 12 splits 9.5 / 9.9 and of 32 16.2 / 17.2, 1200 of 10 9.7 /
// 9.9, 1400 of 9 10.3 / 10.1, 4000 of 12 17.8 / 16.7, 7000 of 9 (fp32) 40.7 / 39.1;
// d = 128, 400 of 32 13.1 / 14.4, 1000 of 32 19.6 / 19.5, 3600 of 9 24.0 / 23.0.
constexpr int kFwdMaxSplits = 32;   // of 64-query work-groups
constexpr int kFewMaxSplits = 128;  // of fwd_few_entry's
constexpr int kMergeThread = 8;
constexpr size_t kMergeRow = 1 << 16;

template <class T, int D, int MAXS>
__device__ __forceinline__ void fwd_merge_body(const Params &p, int S) {
    constexpr int C = D / 4;
    const size_t rows = (size_t)p.B * p.Hq * p.N;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= rows * C) return;
    const size_t r = t / C;
    const int c = (int)(t % C);
    const float2 *ml = reinterpret_cast<const float2 *>(p.fwd_part + (size_t)S * rows * D);
    float2 v[MAXS];
    float4 a[MAXS];
#pragma unroll
    for (int sp = 0; sp < MAXS; ++sp) {
        if (sp < S) {
            v[sp] = ml[sp * rows + r];
            a[sp] = *reinterpret_cast<const float4 *>(p.fwd_part + (sp * rows + r) * D + 4 * c);
        }
    }
    // the split holding key 0 (visible to every row) makes M finite
    float M = -INFINITY;
#pragma unroll
    for (int sp = 0; sp < MAXS; ++sp) M = sp < S ? fmaxf(M, v[sp].x) : M;
    float L = 0.f;
    f32x4 o = zero4();
#pragma unroll
    for (int sp = 0; sp < MAXS; ++sp) {
        if (sp < S) {
            const float w = fast_exp2(v[sp].x - M);
            L += w * v[sp].y;
            o[0] += w * a[sp].x;
            o[1] += w * a[sp].y;
            o[2] += w * a[sp].z;
            o[3] += w * a[sp].w;
        }
    }
    const int bh = (int)(r / p.N), qi = (int)(r % p.N);
    const int b = bh / p.Hq, h = bh % p.Hq;
    T *O = static_cast<T *>(p.o) + b * p.o_bs + h * p.o_hs + (size_t)qi * p.o_rs + 4 * c;
    store4<T>(O, o, 1.0f / L);
    if (p.lse != nullptr && c == 0) p.lse[r] = (M + fast_log2(L)) * kLn2;
}

template <class T, int D, int MAXS>
__device__ __forceinline__ void fwd_merge_row_body(const Params &p, int S) {
    constexpr int NT = 8 * MAXS, NW = NT / 64;
    constexpr int C = D / 4, G = NT / C, PER = MAXS / G;  // threads per row of O, groups of splits, splits per group
    static_assert(PER * G == MAXS && 64 % C == 0, "whole groups, and whole waves of them");
    __shared__ float sm[NW], sl[NW];
    __shared__ __attribute__((aligned(16))) f32x4 so[NW][C];
    const size_t rows = (size_t)p.B * p.Hq * p.N, r = blockIdx.x;
    const int tid = threadIdx.x, wave = tid / 64, c = tid % C, grp = tid / C;
    const float2 *ml = reinterpret_cast<const float2 *>(p.fwd_part + (size_t)S * rows * D);
    float2 v[PER];
    f32x4 a[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int sp = grp + G * i;
        v[i] = make_float2(-INFINITY, 0.f);
        a[i] = zero4();
        if (sp < S) {
            v[i] = ml[sp * rows + r];
            a[i] = *reinterpret_cast<const f32x4 *>(p.fwd_part + (sp * rows + r) * D + 4 * c);
        }
    }
    float M = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; ++i) M = fmaxf(M, v[i].x);
#pragma unroll
    for (int k = 32; k >= C; k >>= 1) M = fmaxf(M, __shfl_xor(M, k, 64));
    if (tid % 64 == 0) sm[wave] = M;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, sm[w]);  // finite: the split of key 0
    float L = 0.f;
    f32x4 o = zero4();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const float w = fast_exp2(v[i].x - M);
        L += w * v[i].y;
        o += a[i] * w;
    }
    // the wave's groups, then the waves
#pragma unroll
    for (int k = 32; k >= C; k >>= 1) {
        L += __shfl_xor(L, k, 64);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += __shfl_xor(o[e], k, 64);
    }
    if (tid % 64 < C) so[wave][c] = o;
    if (tid % 64 == 0) sl[wave] = L;
    __syncthreads();
    if (tid >= C) return;
#pragma unroll
    for (int w = 1; w < NW; ++w) {
        o += so[w][c];
        L += sl[w];
    }
    const int bh = (int)(r / p.N), qi = (int)(r % p.N);
    const int b = bh / p.Hq, h = bh % p.Hq;
    T *O = static_cast<T *>(p.o) + b * p.o_bs + h * p.o_hs + (size_t)qi * p.o_rs + 4 * c;
    store4<T>(O, o, 1.0f / L);
    if (p.lse != nullptr && c == 0) p.lse[r] = (M + fast_log2(L)) * kLn2;
}

// The code object's forward kernels (fa_kernels.h): policy, causal, waves
// per SIMD, query tiles per wave.
#if defined(__HIP_DEVICE_COMPILE__)
#define MXFA_FWD(NAME, POL, CAUSAL, WPS, QT)                                                            \
    extern "C" __global__ __launch_bounds__(256, WPS) void NAME(Params p) { fwd_entry<POL, CAUSAL, QT>(p); }
#define MXFA_FWD_PG(NAME, POL, WPS, QT)                                                                 \
    extern "C" __global__ __launch_bounds__(256, WPS) void NAME(Params p) { fwd_entry<POL, true, QT, true>(p); }
MXFA_FWD(mxfa_fwd_b64_c_w3_q2, PolBF16<64>, true, 3, 2)
MXFA_FWD(mxfa_fwd_b64_c_w3_q1, PolBF16<64>, true, 3, 1)
MXFA_FWD(mxfa_fwd_b64_n_w2_q2, PolBF16<64>, false, 2, 2)
MXFA_FWD(mxfa_fwd_b64_n_w3_q1, PolBF16<64>, false, 3, 1)
MXFA_FWD(mxfa_fwd_b128_c_w2_q2, PolBF16<128>, true, 2, 2)
MXFA_FWD(mxfa_fwd_b128_c_w2_q1, PolBF16<128>, true, 2, 1)
MXFA_FWD(mxfa_fwd_b128_n_w2_q2, PolBF16<128>, false, 2, 2)
// fp32
#define MXFA_FWD_F(NAME, NW, CAUSAL, PG, SP)                                                            \
    extern "C" __global__ __launch_bounds__(64 * NW, NW == 8 ? 4 : 3) void NAME(Params p) {              \
        fwd_split_entry<NW, CAUSAL, PG, SP>(p);                                                          \
    }
MXFA_FWD_F(mxfa_fwd_f64_c, 4, true, false, false)
MXFA_FWD_F(mxfa_fwd_f64_n, 4, false, false, false)
MXFA_FWD_F(mxfa_fwd_f64_c_g8, 8, true, false, false)
MXFA_FWD_F(mxfa_fwd_f64_n_g8, 8, false, false, false)
MXFA_FWD_F(mxfa_fwd_f64_c_pg, 4, true, true, false)
MXFA_FWD_F(mxfa_fwd_f64_c_pg_g8, 8, true, true, false)
MXFA_FWD_F(mxfa_fwd_f64_c_sp, 4, true, false, true)
MXFA_FWD_F(mxfa_fwd_f64_c_pg_sp, 4, true, true, true)
MXFA_FWD_F(mxfa_fwd_f64_c_sp_g8, 8, true, false, true)
MXFA_FWD_F(mxfa_fwd_f64_c_pg_sp_g8, 8, true, true, true)
// the prefill over a paged cache (causal, as the prefill always is)
// (the table entry and row address take registers: the 128-query d = 128 form
// would spill in its loop, so paged launches use 64-query work-groups there;
// the 128-query d = 64 form spills 9, outside its main loop and twice per masked
// stage pair)
MXFA_FWD_PG(mxfa_fwd_b64_c_w3_q2_pg, PolBF16<64>, 3, 2)
MXFA_FWD_PG(mxfa_fwd_b64_c_w3_q1_pg, PolBF16<64>, 3, 1)
MXFA_FWD_PG(mxfa_fwd_b128_c_w2_q1_pg, PolBF16<128>, 2, 1)
// the prefill split over its keys (causal, 64-query work-groups) and the
// merge of the splits
#define MXFA_FWD_SP(NAME, POL, WPS, PG)                                                                \
    extern "C" __global__ __launch_bounds__(256, WPS) void NAME(Params p) { fwd_entry<POL, true, 1, PG, true>(p); }
MXFA_FWD_SP(mxfa_fwd_b64_c_w3_q1_sp, PolBF16<64>, 3, false)
MXFA_FWD_SP(mxfa_fwd_b128_c_w2_q1_sp, PolBF16<128>, 2, false)
MXFA_FWD_SP(mxfa_fwd_b64_c_w3_q1_pg_sp, PolBF16<64>, 3, true)
MXFA_FWD_SP(mxfa_fwd_b128_c_w2_q1_pg_sp, PolBF16<128>, 2, true)
#define MXFA_FWD_MERGE(NAME, T, D, MAXS)                                                               \
    extern "C" __global__ __launch_bounds__(256) void NAME(Params p, int splits) {                     \
        fwd_merge_body<T, D, MAXS>(p, splits);                                                         \
    }
MXFA_FWD_MERGE(mxfa_fwd_merge8_b64, u16, 64, kMergeThread)
MXFA_FWD_MERGE(mxfa_fwd_merge8_b128, u16, 128, kMergeThread)
MXFA_FWD_MERGE(mxfa_fwd_merge8_f64, float, 64, kMergeThread)
MXFA_FWD_MERGE(mxfa_fwd_merge32t_b64, u16, 64, kFwdMaxSplits)
MXFA_FWD_MERGE(mxfa_fwd_merge32t_b128, u16, 128, kFwdMaxSplits)
MXFA_FWD_MERGE(mxfa_fwd_merge32t_f64, float, 64, kFwdMaxSplits)
#define MXFA_FWD_MERGE_ROW(NAME, T, D, MAXS)                                                           \
    extern "C" __global__ __launch_bounds__(8 * MAXS) void NAME(Params p, int splits) {                \
        fwd_merge_row_body<T, D, MAXS>(p, splits);                                                     \
    }
MXFA_FWD_MERGE_ROW(mxfa_fwd_merge32_b64, u16, 64, kFwdMaxSplits)
MXFA_FWD_MERGE_ROW(mxfa_fwd_merge32_b128, u16, 128, kFwdMaxSplits)
MXFA_FWD_MERGE_ROW(mxfa_fwd_merge32_f64, float, 64, kFwdMaxSplits)
MXFA_FWD_MERGE_ROW(mxfa_fwd_merge128_b64, u16, 64, kFewMaxSplits)
MXFA_FWD_MERGE_ROW(mxfa_fwd_merge128_b128, u16, 128, kFewMaxSplits)
#define MXFA_FWD_FEW(NAME, D, NW, PG, SP)                                                              \
    extern "C" __global__ __launch_bounds__(64 * NW) void NAME(Params p) {                             \
        fwd_few_entry<PolBF16<D>, NW, PG, SP>(p);                                                      \
    }
MXFA_FWD_FEW(mxfa_fwd_b64_few, 64, 8, false, false)
MXFA_FWD_FEW(mxfa_fwd_b64_few_pg, 64, 8, true, false)
MXFA_FWD_FEW(mxfa_fwd_b64_few_sp, 64, 8, false, true)
MXFA_FWD_FEW(mxfa_fwd_b64_few_pg_sp, 64, 8, true, true)
MXFA_FWD_FEW(mxfa_fwd_b128_few, 128, 4, false, false)
MXFA_FWD_FEW(mxfa_fwd_b128_few_pg, 128, 4, true, false)
MXFA_FWD_FEW(mxfa_fwd_b128_few_sp, 128, 4, false, true)
MXFA_FWD_FEW(mxfa_fwd_b128_few_pg_sp, 128, 4, true, true)
#undef MXFA_FWD
#undef MXFA_FWD_F
#undef MXFA_FWD_PG
#undef MXFA_FWD_SP
#undef MXFA_FWD_MERGE
#undef MXFA_FWD_MERGE_ROW
#undef MXFA_FWD_FEW
#endif

// The kernel of (policy, causal) with `qt` query tiles per wave (one of the list
// above); paged: its *_pg form (causal kernels only). bf16 only; fp32 goes
// through launch_fwd_f32.
template <class Pol, bool CAUSAL>
static KernelId fwd_kernel_id(int qt, bool paged) {
    if constexpr (Pol::D == 64) {
        if (CAUSAL && paged) return qt == 1 ? k_mxfa_fwd_b64_c_w3_q1_pg : k_mxfa_fwd_b64_c_w3_q2_pg;
        if (CAUSAL) return qt == 1 ? k_mxfa_fwd_b64_c_w3_q1 : k_mxfa_fwd_b64_c_w3_q2;
        return qt == 1 ? k_mxfa_fwd_b64_n_w3_q1 : k_mxfa_fwd_b64_n_w2_q2;
    } else {
        if (CAUSAL && paged) return k_mxfa_fwd_b128_c_w2_q1_pg;
        if (CAUSAL) return qt == 1 ? k_mxfa_fwd_b128_c_w2_q1 : k_mxfa_fwd_b128_c_w2_q2;
        return k_mxfa_fwd_b128_n_w2_q2;
    }
}

template <class Pol, bool CAUSAL, int QT>
static hipError_t launch_fwd_qt(Params p, hipStream_t stream) {
    const dim3 grid(p.B * p.Hq, (p.N + 64 * QT - 1) / (64 * QT));
    const KernelId id = fwd_kernel_id<Pol, CAUSAL>(QT, p.block_table != nullptr);
    if (CAUSAL) cu_balance(&p, id, (long long)grid.x * grid.y);
    void *args[] = {&p};
    return launch_kernel(id, grid, dim3(256), args, stream);
}

// bf16 launches whose 128-query work-groups would not fill every resident
// slot (256 CUs x the 128-query kernel's waves per SIMD: 3 at d = 64, 2 at
// d = 128) take 64-query work-groups (one 16-query tile per wave): twice the
// work-groups and half the critical path (the heaviest block's keys times its
// queries), for twice the LDS reads per MFMA. Measured on the MI355X: causal
// B1 H12 N4096 d64 54.3 -> 40.3 us, B1 H8 N2048 d128 43.4 -> 28.8 us,
// non-causal B1 H12 N4096 d64 74.6 -> 65.5 us; at 768 work-groups (causal B1
// H12 N8192 d64) 125 against 135 us keeps 128 queries, and so does d = 128 at
// 512 (causal B1 H32 Hkv4 N2048: 44.6 against 45.5 us). Non-causal d = 128
// keeps them (B1 H8 N4096: 77.2 against 80.2 us). A d = 128 prefill takes
// 64-query work-groups at any grid, as its paged form must (the 128-query
// d = 128 kernel would spill with the block-table registers): the wave's
// rows decide when the lazy rescale redoes a stage, so both tilings must match
// for the paged prefill to give the contiguous one's bits.
template <class Pol, bool CAUSAL>
static hipError_t launch_fwd_t(const Params &p, hipStream_t stream) {
    if constexpr (CAUSAL || Pol::D == 64) {
        constexpr long long kSlots = 256LL * Pol::kWavesFwdCausal;
        const long long wg = (long long)p.B * p.Hq * ((p.N + 127) / 128);
        if (wg < kSlots || (Pol::D == 128 && p.prefill != 0))
            return launch_fwd_qt<Pol, CAUSAL, 1>(p, stream);
    }
    return launch_fwd_qt<Pol, CAUSAL, 2>(p, stream);
}

// The fp32 forward: 8 waves and 128 queries per work-group where those fill the
// two that a CU holds (each K and V element is then split half as often: B4 H12
// N4096 causal 590 -> 523 us); 4 waves and 64 queries on smaller grids (B4 H12
// N1024 causal 60 -> 54, B1 H1 N256 16.8 -> 14.1; 384 of 128 queries, B1 H12
// N4096, 310 and 318 non-causal, 192 both causal). A last block of 128 with at
// most 64 rows leaves half its waves idle, which costs more than that saves in
// heads of 1, 3 or 5 blocks of 64 (512 heads of 64 rows 9.5 us against 11.2, of
// 192 32.0 / 37.5, of 320 64.7 / 69.1; of 256 46.6 / 43.9). The same waves, so
// the same bits.
static hipError_t launch_fwd_f32(Params p, int causal, hipStream_t stream) {
    const bool pg = p.block_table != nullptr;
    const int nb64 = (p.N + 63) / 64;
    const int nw = (long long)p.B * p.Hq * ((p.N + 127) / 128) >= 512 && (nb64 % 2 == 0 || nb64 > 5) ? 8 : 4;
    const dim3 grid(p.B * p.Hq, (p.N + 16 * nw - 1) / (16 * nw));
    const KernelId id = nw == 8 ? (pg ? k_mxfa_fwd_f64_c_pg_g8 : causal ? k_mxfa_fwd_f64_c_g8 : k_mxfa_fwd_f64_n_g8)
                                : (pg ? k_mxfa_fwd_f64_c_pg : causal ? k_mxfa_fwd_f64_c : k_mxfa_fwd_f64_n);
    if (causal && nw == 4) cu_balance(&p, id, (long long)grid.x * grid.y);
    void *args[] = {&p};
    return launch_kernel(id, grid, dim3(64 * nw), args, stream);
}

// Few query rows of a prefill, unsplit (bh rows' blocks; the same rule for a
// paged cache, so that both give the same bits). fwd_few_entry's work-groups
// take a CU each:
//  * more than 256 of them run in rounds, where the 64-query form holds two or
//    three a CU (8 tokens, d = 64, 16 stages: 288 heads 1.3 times its time, 512
//    1.3, 256 1.16), and with one stage nothing is gained (3.9 -> 4.2 us);
//  * up to one stage per wave of all 256 (8 waves; d = 128: 4) they read faster:
//    us, 8 tokens, 128 heads of 16 stages 0.76 times, 8 heads of 125 0.51;
//  * beyond that the caches set the time: as fast up to 192 blocks at d = 64
//    (0.94-1.04; paged 0.83-0.97; 256: 1.25), and at d = 128 up to 64 (0.90;
//    96 and 128 0.94-1.12, 160 1.08-1.17).
static bool few_rows(const Params &p, int dtype_bf16) { return dtype_bf16 && p.prefill != 0 && p.N <= kFewRows; }
static long long key_stages(const Params &p) { return (std::min(p.Nk, p.pos0 + p.N) + 63) / 64; }
static bool fwd_few(const Params &p, int dtype_bf16, int d) {
    const long long stages = key_stages(p), bh = (long long)p.B * p.Hq;
    return few_rows(p, dtype_bf16) && stages > 1 && bh <= 256 &&
           (bh * stages <= 256 * (d == 128 ? 4 : 8) || bh <= (d == 128 ? 64 : 192));
}
// Split: up to 7/8 of a stage per wave of the 256 work-groups that fit at once
// (0.72-1.0 times the 64-query form's time; at a whole one 0.9-1.11, and with
// two 1.0-1.2 at d = 64); below 8 blocks, which the 64-query form splits into
// fewer work-groups than CUs, up to two stages (one token, 1 to 7 heads, d = 64:
// 0.26-0.89 times).
static bool fwd_few_split(const Params &p, int dtype_bf16, int d) {
    const long long bh = (long long)p.B * p.Hq, waves = 256 * (d == 128 ? 4 : 8);
    return few_rows(p, dtype_bf16) && bh * key_stages(p) <= (bh < 8 ? 2 * waves : waves / 8 * 7);
}

static hipError_t launch_fwd_few(const Params &p, int d, int splits, hipStream_t stream) {
    const bool pg = p.block_table != nullptr, sp = splits > 1;
    static constexpr KernelId ids[2][2][2] = {
        {{k_mxfa_fwd_b64_few, k_mxfa_fwd_b64_few_sp}, {k_mxfa_fwd_b64_few_pg, k_mxfa_fwd_b64_few_pg_sp}},
        {{k_mxfa_fwd_b128_few, k_mxfa_fwd_b128_few_sp}, {k_mxfa_fwd_b128_few_pg, k_mxfa_fwd_b128_few_pg_sp}}};
    void *args[] = {const_cast<Params *>(&p)};
    return launch_kernel(ids[d == 128][pg][sp], dim3(p.B * p.Hq, 1, splits), dim3(d == 128 ? 256 : 512), args, stream);
}

// Splits of the prefill's keys: none (1) when the 64-query work-groups
// already fill the resident slots (256 CUs x waves per SIMD) halfway, or when
// the heaviest query block has under 16 key stages (bf16; 8 for fp32), where
// the merging launch costs more than the split saves (measured on the MI355X,
// Qwen2.5 heads, 512 tokens at position 0, 8 stages: bf16 19.7 -> 24.6 us
// with 2 splits, fp32 36.5 -> 32.6 us); else enough to fill them, with at
// least 2 key stages per split and at most kFwdMaxSplits splits.
static int fwd_splits_64(const Params &p, int dtype_bf16, int d, long long most) {
    const long long wgs = (long long)p.B * p.Hq * ((p.N + 63) / 64);
    const long long slots = 256LL * (dtype_bf16 && d == 64 ? 3 : 2);
    if (2 * wgs >= slots) return 1;
    const long long stages = key_stages(p);  // the heaviest block's
    if (stages < (dtype_bf16 ? 16 : 8)) return 1;
    return (int)std::min({(slots + wgs - 1) / wgs, std::max(1LL, stages / 2), most});
}

// fp32 chunks of more than 64 rows split over 8-wave work-groups of 128 queries
// (launch_fwd_f32's reason) where there are stages enough to fill the 512 that
// fit at once and the blocks alone leave half of them empty: us a call, 14/2
// heads, 500 tokens after 3584 65 -> 56 (9 splits; 5 of 4-wave work-groups), 70
// after 8000 40 -> 31; 4/2 heads, 100 after 2000, which cannot fill them,
// 13.5 against 15.6.
static bool fwd_f32_wide(const Params &p, int dtype_bf16) {
    if (dtype_bf16 || p.N <= 64) return false;
    const long long stages = key_stages(p), bh = (long long)p.B * p.Hq;
    return stages >= 16 && bh * ((p.N + 127) / 128) < 256 &&
           bh * ((p.N + 63) / 64) * std::min(stages / 2, (long long)kFwdMaxSplits) >= 512;
}

// The forms that split into one round of the work-groups that fit at once:
// those, and fwd_few_entry's 256; else fwd_splits_64's.
int fwd_splits(const Params &p, int dtype_bf16, int d) {
    const long long stages = key_stages(p), bh = (long long)p.B * p.Hq;
    if (fwd_f32_wide(p, dtype_bf16))
        return (int)std::min({512 / (bh * ((p.N + 127) / 128)), stages / 2, (long long)kFwdMaxSplits});
    const bool few = fwd_few_split(p, dtype_bf16, d);
    const int s = fwd_splits_64(p, dtype_bf16, d, few ? kFewMaxSplits : kFwdMaxSplits);
    return few ? (int)std::min<long long>(s, std::max(1LL, 256 / bh)) : s;
}

int fwd_splits_in(const Params &p, int dtype_bf16, int d, size_t bytes) {
    const int want = fwd_splits(p, dtype_bf16, d), must = fwd_splits_64(p, dtype_bf16, d, kFwdMaxSplits);
    if (want <= 1) return 1;  // no workspace is reported for it, so none is asked for
    const size_t one = (size_t)p.B * p.Hq * p.N * (size_t)(d + 2) * sizeof(float);
    const int fit = (int)std::min<size_t>(bytes / one, (size_t)want);
    if (must <= 1) return std::max(fit, 1);
    return fit >= std::min(want, must) ? fit : 0;
}

size_t fwd_split_workspace_bytes(const Params &p, int d, int splits) {
    if (splits <= 1) return 0;
    return (size_t)splits * p.B * p.Hq * p.N * (size_t)(d + 2) * sizeof(float);
}

hipError_t launch_fwd_split(const Params &p, int dtype_bf16, int d, int splits, hipStream_t stream) {
    const bool few = fwd_few_split(p, dtype_bf16, d), pg = p.block_table != nullptr;
    if (p.fwd_part == nullptr || splits < 2 || splits > (few ? kFewMaxSplits : kFwdMaxSplits)) return hipErrorInvalidValue;
    const int nw = fwd_f32_wide(p, dtype_bf16) ? 8 : 4;
    const KernelId kf =
        dtype_bf16 ? (d == 64 ? (pg ? k_mxfa_fwd_b64_c_w3_q1_pg_sp : k_mxfa_fwd_b64_c_w3_q1_sp)
                              : (pg ? k_mxfa_fwd_b128_c_w2_q1_pg_sp : k_mxfa_fwd_b128_c_w2_q1_sp))
        : nw == 8  ? (pg ? k_mxfa_fwd_f64_c_pg_sp_g8 : k_mxfa_fwd_f64_c_sp_g8)
                   : (pg ? k_mxfa_fwd_f64_c_pg_sp : k_mxfa_fwd_f64_c_sp);
    const size_t rows = (size_t)p.B * p.Hq * p.N;
    // 0, 1: a thread per four elements; 2, 3: a work-group per row (3: few rows, bf16)
    const int mi = splits <= kMergeThread ? 0 : splits > kFwdMaxSplits ? 3 : rows * d > kMergeRow ? 1 : 2;
    static constexpr KernelId merge[3][4] = {
        {k_mxfa_fwd_merge8_b64, k_mxfa_fwd_merge32t_b64, k_mxfa_fwd_merge32_b64, k_mxfa_fwd_merge128_b64},
        {k_mxfa_fwd_merge8_b128, k_mxfa_fwd_merge32t_b128, k_mxfa_fwd_merge32_b128, k_mxfa_fwd_merge128_b128},
        {k_mxfa_fwd_merge8_f64, k_mxfa_fwd_merge32t_f64, k_mxfa_fwd_merge32_f64, k_mxfa_fwd_merge32_f64}};
    const KernelId km = merge[!dtype_bf16 ? 2 : d == 128 ? 1 : 0][mi];
    Params q = p;
    void *args[] = {&q};
    hipError_t e = few ? launch_fwd_few(p, d, splits, stream)
                       : launch_kernel(kf, dim3(p.B * p.Hq, (p.N + 16 * nw - 1) / (16 * nw), splits), dim3(64 * nw), args, stream);
    if (e != hipSuccess) return e;
    int s = splits;
    void *margs[] = {&q, &s};
    const unsigned groups = (unsigned)(mi <= 1 ? (rows * (d / 4) + 255) / 256 : rows);
    return launch_kernel(km, dim3(groups), dim3(mi == 3 ? 8 * kFewMaxSplits : 256), margs, stream);
}

hipError_t launch_fwd(const Params &p, int dtype_bf16, int d, int causal, hipStream_t stream) {
    if (p.block_table != nullptr && !causal) return hipErrorInvalidValue;  // paged kernels are causal
    if (causal && fwd_few(p, dtype_bf16, d)) return launch_fwd_few(p, d, 1, stream);
    if (!dtype_bf16) return d == 64 ? launch_fwd_f32(p, causal, stream) : hipErrorInvalidValue;
    if (d == 64) return causal ? launch_fwd_t<PolBF16<64>, true>(p, stream) : launch_fwd_t<PolBF16<64>, false>(p, stream);
    if (d == 128)
        return causal ? launch_fwd_t<PolBF16<128>, true>(p, stream) : launch_fwd_t<PolBF16<128>, false>(p, stream);
    return hipErrorInvalidValue;
}

}  // namespace mxfa
