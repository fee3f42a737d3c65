// Forward attention kernel for gfx950: O = softmax(Q K^T * sm_scale + bias) V, LSE saved.
//
// Replaces _attn_fwd / _attn_fwd_inner of the reference (/root/reference/flash_attention.py:12-194)
// together with the host-side bias pre-scale (flash_attention.py:660-663), which is folded into
// the kernel as an fp32 multiply.
//
// Work split.  One work-group (4 waves) owns 128 query rows of one (batch, head); each wave
// owns 32 of them for the whole kernel.  Keys/values are streamed through LDS in steps of 64 keys (32 with an
// fp32 bias or ALiBi, and above head dim 64 with any bias: StreamCfg, fwd_stream_kind), consumed 32 at a time.
// Scores are computed TRANSPOSED, S^T = K Q^T, so that in the MFMA accumulator a lane holds one
// query row (column l%32 of S^T) and 16 of the 32 keys: the row maximum and row sum of the online
// softmax are then per-lane loops plus a single exchange with lane l^32, the reference point of the exponentials, the
// running sum and the rescale factor are one scalar per lane, and P^T is already laid out as the
// B operand of O^T += V^T P^T.  V^T is gathered from the row-major V rows with
// ds_read_b64_tr_b16.
//
// Memory -> LDS.  The K and V rows of a step (double buffered, one step ahead, where a step has 64 keys or the bias is in fp32; else a
// ring of 3 slots, two ahead) and the bias slice of each wave (32 rows x 32 or 64 keys, a wave-private ring: of 4 slots,
// three steps ahead, 3 in fp32, 2 where a step has 64 keys) arrive through direct global -> LDS copies that the compiler
// does not see; their completion is counted by hand (copies complete in issue order and every step issues the same number).
// The bias is a pure HBM stream: a queue of 96 (64) keys a row keeps enough bytes in flight.
#include <type_traits>

#include "fa_common.hpp"
#include "fa_params.hpp"

namespace fa {

// Sum of a lane's exponentials of a block (or half of one) beyond which their reference point is raised to the maximum.
// No higher: after a raise the largest weight is 1, which rounding to 16 bits leaves as it is, and where few keys carry a row
// its rounding is most of the error.  Scores of standard deviation 8, D=64: out off by 1.87e-3 of its norm in bf16 and 2.36e-4 in
// fp16, with limits of 2^32 and 2^14 2.27e-3 and 2.61e-4 (a running maximum raised at 2^8: 1.95e-3, 2.47e-4).  The accumulators
// keep their range too (values of V up to about 2^119).  Random scores of deviation 1 never reach either limit; biases that
// grow take the higher ones 4 to 13 % faster (ALiBi at M=1024 N=8192 H=32 D=128 167 -> 182 us, as with a running maximum).
constexpr float kRaise = 0x1p8f;

// Biases that grow along the keys block after block (a distance penalty: ALiBi, its tensor, slope * key index in a
// row-broadcast bias).  Taking the exponentials first and again once their sum is over the limit then costs a second set
// of them per raise, in the heads with steep slopes in every block.
//   kRowMax  the maximum of each block is formed first, and the reference point raised when it lies 2^8 above: ALiBi, where
//            every row grows towards its diagonal: causal, and where a block's matrix work is small next to it (D <= 64).
//   kAfter   the maximum is formed first in the block that follows a raise, as long as that raises again.  Not where the
//            branch itself costs more than it saves: it takes 2 to 5 % from the causal kernels of a bias tile up to D = 64
//            and from those of a tile or a row-broadcast bias at 128 (B=1 H=16 M=N=4096 bf16 tensor 186.5 -> 190.7).
//   kSum     neither.
// Forward, us, kSum -> the rule here, both with a limit of 2^32 (B=2 H=16 M=N=2048 or, marked *, B=1 H=16 M=N=4096):
//   ALiBi causal D=32* 93.2 -> 71.4, D=64* 94.3 -> 82.4, D=128* 120.1 -> 112.8; not causal D=32 60.7 -> 54.0, D=64 72.0 -> 64.1;
//   as a tensor D=32 67.1 -> 61.6, fp16 D=64 74.0 -> 67.4; slope * key as a row D=32 60.7 -> 56.8.  Biases without a trend lose at
//   most 2 % (row-broadcast not causal D=32 79.3 -> 80.7*, D=64 97.8 -> 99.3*).
enum Growth { kSum, kAfter, kRowMax };
constexpr Growth growth_rule(int bias, int D, bool causal) {
    if (bias == 5) return causal || D <= 64 ? kRowMax : kAfter;
    const bool tile = bias >= 2 && bias <= 4;
    return (tile && D <= 64 && !causal) || (bias == 6 && D <= 64) || ((tile || bias == 6) && D > 128) ? kAfter : kSum;
}

// The K/V stream of a row-broadcast bias (kinds 6, 7) is tiled like that without a bias up to head dim 64 (so that it takes
// the steps, and the bits, of the same mask written out), above like that of ALiBi, in steps of 32 keys: the bias values of a
// block need the registers that 64-key steps spend on a second block of scores.
constexpr int fwd_stream_kind(int bias, int D) { return bias >= 6 && D <= 64 ? 0 : bias >= 5 ? 6 : bias; }

template <typename T, int D, int BIAS, bool CAUSAL>
__global__ __launch_bounds__(256, (StreamCfg<D, fwd_stream_kind(BIAS, D), true>::MIN_BLOCKS)) void fa_fwd_kernel(const FwdParams p) {
    constexpr int TB = tile_kind(BIAS);  // kind of bias tile that is streamed (none for ALiBi)
    typedef StreamCfg<D, fwd_stream_kind(BIAS, D), true> C;
    typedef Swz<D> SW;
    typedef typename VecOf<T>::v8 T8;
    typedef typename VecOf<T>::v4 T4;
    typedef typename BiasElem<tile_kind(BIAS)>::type E;
    constexpr int BM = C::BM, BK = C::BK, OS = C::OS, CPR = C::CPR;

    constexpr bool ROWB = BIAS >= 6;     // the same bias for every query row, kept as an fp32 row in LDS
    constexpr bool BOOLROW = BIAS == 7;  // ... a bool mask: the row holds 0 or the mask term, in log2 units
    constexpr bool BY_DWORD = BIAS == 4 && D <= 64;

    __shared__ __align__(1024) unsigned char smem[C::LOOP_BYTES + (ROWB ? kRowBiasKeys * 4 : 0)];
    const float* row_lds = reinterpret_cast<const float*>(smem + C::LOOP_BYTES);

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int r = lane & 31, g = lane >> 5;

    int mt, bh;
    // (ALiBi, and a row-broadcast bias up to D = 64: longest first in any grid, pairing took 4 to 8 % from them)
    constexpr bool PAIRS = !(BIAS == 5 || (BIAS == 6 && D <= 64));
    decode_block<CAUSAL, typename std::conditional<PAIRS, C, OnePerCu>::type>(blockIdx.x, p.n_mtiles * p.n_splits, p.B * p.H, mt, bh);
    // With the keys split between work-groups (never when causal) this one sees keys key0 ..
    // key0 + N - 1 as if they were all there are; only ALiBi needs to know better.
    const int split = mt % p.n_splits;
    mt /= p.n_splits;
    const int key0 = split * p.keys_per_split;
    if (CAUSAL) mt = p.n_mtiles - 1 - mt;  // longest rows first
    const int b = bh / p.H, h = bh % p.H;
    const int M = p.M;
    const int N = p.n_splits > 1 ? (p.N - key0 < p.keys_per_split ? p.N - key0 : p.keys_per_split) : p.N;
    const int m0 = mt * BM;
    const int mw = m0 + wave * 32;  // first query row of this wave
    const int my_m = mw + r;

    const T* qp = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.sq.b + (int64_t)h * p.sq.h;
    const T* kp = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.sk.b + (int64_t)h * p.sk.h + (int64_t)key0 * p.sk.s;
    const T* vp = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.sv.b + (int64_t)h * p.sv.h + (int64_t)key0 * p.sv.s;
    const E* bp = nullptr;
    if (TB != 0) bp = reinterpret_cast<const E*>(p.bias) + (int64_t)b * p.sbias.b + (int64_t)h * p.sbias.h + (int64_t)key0 * p.sbias.n;
    // ALiBi: the slope of this head and the position of this lane's query row on the key axis
    float neg_slope = 0.f, ratio = 0.f;
    // ... and, for unmasked steps, the slope in units of the dot product (its distances reach N)
    float raw_slope = 0.f;
    bool raw_ok = true;
    if (BIAS == 5) {
        neg_slope = -reinterpret_cast<const float*>(p.bias)[h];
        ratio = (float)p.N / (float)p.M;
        raw_slope = neg_slope / p.sm_scale;
        raw_ok = __builtin_fabsf(raw_slope) * (float)p.N < 1e30f;
    }

    const LiveChunks chunks{p.d_qk / 8, p.qk_inv};
    const unsigned rows_l = SW::rows_lane(lane), cols_l = SW::cols_lane(lane);
    typedef KeyStream<T, D, fwd_stream_kind(BIAS, D), true, true> KS;
    KS ks_;
    ks_.init(smem, kp, vp, bp, p.sk.s, p.sv.s, p.sbias.m, p.sbias.n, M, N, mw, wave, lane, chunks, p.d_v / 8);

    // Q^T as B operand: column my_m, k = d
    // (Rows through LDS, as in the dQ kernel, lose as much as they gain in this one, which needs them once and has its K and V
    // copies to wait for anyway.  us, the lanes' own loads / LDS, no bias: D=128 B=16 H=12 S=197 16.5 / 15.8, B=32 S=192 21.0 /
    // 21.4, causal 21.2 / 22.4, B=12 H=16 S=577 causal 36.4 / 38.3, H=16 S=2000 causal 36.1 / 37.0; D=256 H=32 S=1001 44.0 / 46.8,
    // B=12 H=16 S=577 116.5 / 120; D=80 B=4 H=8 S=512 12.4 / 13.2, B=16 H=12 S=197 14.0 / 13.3.)
    typedef WaveRows<T, D> WR;
    T8 qreg[C::KSTEPS];
#pragma unroll
    for (int ks = 0; ks < C::KSTEPS; ks++) {
        i32x4 raw = {0, 0, 0, 0};
        if (my_m < M) raw = gld16(qp + (int64_t)my_m * p.sq.s + (D <= 128 ? chunks.wrap(2 * ks + g) : 2 * ks + g) * 8);
        qreg[ks] = as_vec<T8>(raw);
    }
    auto split_q = [&]() {
        if (D <= 128 && p.d_qk < D) {
#pragma unroll
            for (int ks = 0; ks < C::KSTEPS; ks++) qreg[ks] = chunks.part(qreg[ks], 2 * ks + g, C::CPR);
        }
    };
    if constexpr (TB != 0) split_q();  // (kernels of a bias tile have no registers for it later)

    int n_steps = (N + BK - 1) / BK;
    if (CAUSAL) {
        int last = (m0 + BM - 1) / BK + 1;  // steps holding keys <= last row of this work-group
        n_steps = n_steps < last ? n_steps : last;
    }

    const float qk_scale = p.sm_scale * kLog2e;
    // (the lowest number, not -inf: keys whose bias is -inf then have exponentials of 0 also where no other key has been
    // seen yet, as in a share of the keys that is padding from end to end)
    float m_i = kLowest, l_i = 0.f;
    constexpr Growth GROWTH = growth_rule(BIAS, D, CAUSAL);
    bool rising = GROWTH == kRowMax;  // (the same in every lane) the next block's maximum is formed before its exponentials
    f32x16 o_acc[C::DB];
#pragma unroll
    for (int db = 0; db < C::DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o_acc[db][i] = 0.f;

    auto stage_row = [&]() {
        if (ROWB)
            stage_row_bias(reinterpret_cast<float*>(smem + C::LOOP_BYTES), p.bias, p.row_bias_kind,
                           (int64_t)b * p.sbias.b + (int64_t)h * p.sbias.h + (int64_t)key0 * p.sbias.n, p.sbias.n, N, tid);
    };

    // raises the reference point of this row's exponentials to mx (log2 units) where it is lower
    auto raise = [&](float mx) {
        const float alpha = mx > m_i ? fast_exp2(m_i - mx) : 1.f;
        m_i = mx > m_i ? mx : m_i;
        l_i *= alpha;
#pragma unroll
        for (int db = 0; db < C::DB; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) o_acc[db][i] *= alpha;
    };

    // One step of the K/V stream.  Interior steps (every key in range and visible to every row of
    // the work-group) run with STEP_MASKED = false: no range checks, no mask arithmetic.  BV: the
    // bias slices come by copy (rows that allow aligned 16-byte chunks), else element by element.
    // LEAN: the copies of the step need no clamps (KeyStream::issue_ahead_lean).
    auto kv_step = [&](int k, auto step_tag, auto bv_tag, auto lean_tag) {
        constexpr bool STEP_MASKED = decltype(step_tag)::value;
        constexpr int BV = decltype(bv_tag)::value;
        constexpr bool LEAN = decltype(lean_tag)::value;
        auto issue_ahead = [&]() {
            if constexpr (LEAN) ks_.template issue_ahead_lean<BV>(k);
            else ks_.template issue_ahead<BV>(k);
        };
        const int n0 = k * BK;
        ks_.template begin_step<BV>(k);
        const unsigned k_rows = ks_.k_addr(k) + rows_l, v_cols = ks_.v_addr(k) + cols_l;  // operand reads by address
        const unsigned char* b_slot = ks_.b_lds(k);
        // Interior steps of two blocks: the matrix instructions of one block are issued between
        // the exponentials of the other, S of block 1 under the exponentials of block 0 and the PV product
        // of block 0 under those of block 1, one fenced slot per two score elements.  Their LDS operands are
        // fetched a phase ahead; head dim 256 has no registers for that and fetches them one slot ahead.  (Bound by
        // the matrix and the vector pipeline together: per block 512 clocks of the one and about 440 of the other
        // at D = 128.  With the maximum gone and this order, B=2 H=16 M=N=4096 bf16 without a bias takes 0.257 ms
        // where it took 0.274 at D = 128, 0.570 / 0.609 ms at B=4 H=32 D = 64, 0.330 / 0.355 at H=8 D = 256.)
        if constexpr (!STEP_MASKED && C::NH == 2) {
            constexpr int NS = C::KSTEPS, NP = 2 * C::DB;  // matrix instructions of S and of PV per block
            constexpr bool AHEAD = D <= 128;
            constexpr int NSS = AHEAD ? NS : NS / 8, NPS = AHEAD ? NP : NP / 8;  // operands fetched at a time
            // units of the scores once their bias is in: raw dot product without one, log2 with a mask, else natural
            constexpr bool LOG2 = TB == 1 || BOOLROW, RAW = TB == 0 && !ROWB;
            const float to_log2 = RAW ? qk_scale : LOG2 ? 1.f : kLog2e;
            T8 ka[2][NSS], va[2][NPS];
            f32x16 sc[2];
            auto load_k = [&](int nb, int slot) {  // operands slot * NSS .. of S of block nb
#pragma unroll
                for (int i = 0; i < NSS; i++)
                    ka[AHEAD ? nb : slot & 1][i] = SW::template row8_at<T8>(k_rows, nb * 32, slot * NSS + i);
            };
            auto load_v = [&](int nb, int slot) {
#pragma unroll
                for (int i = 0; i < NPS; i++) {
                    const int at = slot * NPS + i;
                    va[AHEAD ? 0 : slot & 1][i] = SW::template col8_at<T8>(v_cols, nb * 32 + (at / C::DB) * 16, at % C::DB);
                }
            };
            // the matrix instructions of slot j of 8 of S and of PV
            auto mma_s = [&](int nb, int j) {
                if (!AHEAD && j < 7) load_k(nb, j + 1);
#pragma unroll
                for (int ks = j * NS / 8; ks < (j + 1) * NS / 8; ks++)
                    sc[nb] = mfma32(ka[AHEAD ? nb : j & 1][AHEAD ? ks : ks - j * NSS], qreg[ks], sc[nb]);
            };
            auto mma_pv = [&](int nb, const T8 (&pv)[2], int j) {
                if (!AHEAD && j < 7) load_v(nb, j + 1);
#pragma unroll
                for (int i = j * NP / 8; i < (j + 1) * NP / 8; i++)
                    o_acc[i % C::DB] = mfma32(va[AHEAD ? 0 : j & 1][AHEAD ? i : i - j * NPS], pv[i / C::DB], o_acc[i % C::DB]);
            };
            // the exponentials of a block against the current m_i; after(j) is called behind pair j of 8
            auto exps = [&](const f32x16& x, T8 (&out)[2], auto&& after) {
                float rs = 0.f;
#pragma unroll
                for (int j = 0; j < 8; j++) {
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const int i = 2 * j + e;
                        const float pv = LOG2 ? fast_exp2(x[i] - m_i) : fast_exp2(__builtin_fmaf(x[i], to_log2, -m_i));
                        rs += pv;
                        out[i >> 3][i & 7] = (T)pv;
                    }
                    after(j);
                }
                return rs;
            };
            auto settle = [&](const f32x16& x, T8 (&out)[2], float rs) {
                if (__builtin_amdgcn_ballot_w64(!(rs <= kRaise)) != 0) {
                    float mx = -INFINITY;
#pragma unroll
                    for (int i = 0; i < 16; i++) mx = fmaxf(mx, x[i]);
                    raise(pair_max(mx) * to_log2);
                    rs = exps(x, out, [](int) {});
                    if (GROWTH == kAfter) rising = k > 0;
                }
                l_i += rs;
            };
            auto add_bias = [&](f32x16& x, int nb) {
                if constexpr (ROWB) {
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) {
                        const f32x4 w = *reinterpret_cast<const f32x4*>(row_lds + n0 + nb * 32 + 8 * q4 + 4 * g);
#pragma unroll
                        for (int e = 0; e < 4; e++) x[q4 * 4 + e] = x[q4 * 4 + e] * (LOG2 ? qk_scale : p.sm_scale) + w[e];
                    }
                } else if constexpr (TB != 0) {
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) {
                        const unsigned char* at = b_slot + nb * C::BBLOCK + ks_.b_off(r, 8 * q4 + 4 * g);
                        if constexpr (TB == 1) {
                            const unsigned int w = *reinterpret_cast<const unsigned int*>(at);
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                const int i = q4 * 4 + e;
                                x[i] = ((w >> (8 * e)) & 0xffu) != 0 ? x[i] * qk_scale : x[i] * qk_scale + kMask;
                            }
                        } else {
                            const typename VecOf<E>::v4 hv = *reinterpret_cast<const typename VecOf<E>::v4*>(at);
#pragma unroll
                            for (int e = 0; e < 4; e++) x[q4 * 4 + e] = x[q4 * 4 + e] * p.sm_scale + (float)hv[e];
                        }
                    }
                }
            };
            auto look_ahead = [&](const f32x16& x) {
                float mx = -INFINITY;
#pragma unroll
                for (int i = 0; i < 16; i++) mx = fmaxf(mx, x[i]);
                mx = pair_max(mx) * to_log2;
                const bool higher = __builtin_amdgcn_ballot_w64(mx > m_i + 8.f) != 0;
                if (higher) raise(mx);
                if (GROWTH == kAfter) rising = higher;
            };
            load_k(0, 0);
            if (AHEAD) load_k(1, 0);
#pragma unroll
            for (int nb = 0; nb < 2; nb++)
#pragma unroll
                for (int i = 0; i < 16; i++) sc[nb][i] = 0.f;
#pragma unroll
            for (int j = 0; j < 8; j++) mma_s(0, j);
            issue_ahead();  // in the shadow of the MFMAs just issued
            if (!AHEAD) load_k(1, 0);
            if (AHEAD) load_v(0, 0);
            add_bias(sc[0], 0);
            if (GROWTH != kSum && rising) look_ahead(sc[0]);
            __builtin_amdgcn_sched_barrier(0);
            T8 p0[2], p1[2];
            float rs = exps(sc[0], p0, [&](int j) {
                __builtin_amdgcn_sched_barrier(0);
                mma_s(1, j);
                __builtin_amdgcn_sched_barrier(0);
            });
            if (!AHEAD) load_v(0, 0);
            settle(sc[0], p0, rs);
            add_bias(sc[1], 1);
            if (GROWTH != kSum && rising) {
                // (the point may be raised here: what block 0 adds, relative to the one it had, must be in O before)
#pragma unroll
                for (int j = 0; j < 8; j++) mma_pv(0, p0, j);
                look_ahead(sc[1]);
                rs = exps(sc[1], p1, [](int) {});
            } else {
                rs = exps(sc[1], p1, [&](int j) {
                    __builtin_amdgcn_sched_barrier(0);
                    mma_pv(0, p0, j);
                    __builtin_amdgcn_sched_barrier(0);
                });
            }
            load_v(1, 0);
            settle(sc[1], p1, rs);
#pragma unroll
            for (int j = 0; j < 8; j++) mma_pv(1, p1, j);
            return;
        }
#pragma unroll
        for (int nb = 0; nb < C::NH; nb++) {
        const int nh = nb * 32;  // first key of this block inside the step
        const unsigned char* b_lds = b_slot + nb * C::BBLOCK;
        __builtin_amdgcn_sched_barrier(0);  // keep the blocks apart
        // blocks entirely above this wave's diagonal or past the last key contribute nothing
        if (STEP_MASKED && ((CAUSAL && n0 + nh > mw + 31) || n0 + nh >= N)) {
            if (nb == 0) issue_ahead();  // every wave issues its copies in every step
            continue;
        }
        const bool need_mask = STEP_MASKED && ((n0 + nh + 32 > N) || (CAUSAL && n0 + nh + 31 > mw));

        // ---- S^T = K Q^T : s[i] is key n0 + nh + 8 (i/4) + 4 g + i%4, query my_m ----
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.f;
#pragma unroll
        for (int ks = 0; ks < C::KSTEPS; ks++) {
            T8 a = SW::template row8_at<T8>(k_rows, nh, ks);
            s = mfma32(a, qreg[ks], s);
        }
        if (nb == 0) issue_ahead();  // in the shadow of the MFMAs just issued

        // ---- online softmax step.  `masked` steps (ragged edge, causal diagonal) and a
        // non-positive scale follow the reference's arithmetic term by term: scaled score,
        // plus additive -1e6 terms in log2 units, plus bias (flash_attention.py:39-53); keys past N get the lowest
        // number.  Interior steps skip the mask terms and fold the scale into the exponent.
        // The reference point m_i of the exponentials is arbitrary (out = acc / l and LSE = m + log2 l do
        // not depend on it), so no running maximum is kept: the exponentials are taken against the m_i at
        // hand, and only when the sum of a lane's 8 or 16 of them exceeds kRaise (as at the first keys, where m_i is
        // the lowest number) or is no number is m_i raised to the maximum, O rescaled and they are taken again.  The test is one comparison on a sum that is needed anyway.
        auto softmax_step = [&](auto masked_tag) {
            constexpr bool MASKED = decltype(masked_tag)::value;
            // units of s[i] below: raw dot product (no bias), natural (float bias), log2 (MASKED, bool masks)
            constexpr bool RAW = !MASKED && (BIAS == 0 || BIAS == 5);
            constexpr bool NAT = !MASKED && BIAS >= 2 && !BOOLROW && !RAW;
            const float to_log2 = RAW ? qk_scale : (NAT ? kLog2e : 1.f);
            const float mf = (float)my_m, nf0 = (float)(key0 + n0 + nh + 4 * g);  // ALiBi: row and first key as floats
            // (unmasked: the distance to a key is that to the lane's first less a constant, and the slope goes into one
            // fused multiply-add: 2 instructions per score, 4 with the bias formed first; with the same in the backward kernels a training
            // step at M=1024 N=8192 H=32 D=128 718 -> 697 us)
            const float dist0 = __builtin_fmaf(mf, ratio, -nf0);
#pragma unroll
            for (int q4 = 0; q4 < 4; q4++) {
                const int nl = 8 * q4 + 4 * g;            // first of 4 consecutive keys
                float bv[4] = {0.f, 0.f, 0.f, 0.f};       // bias in natural units
                bool keep[4] = {true, true, true, true};
                if constexpr (BIAS == 1) {
                    unsigned int w = *reinterpret_cast<const unsigned int*>(b_lds + ks_.b_off(r, nl));
#pragma unroll
                    for (int e = 0; e < 4; e++) keep[e] = ((w >> (8 * e)) & 0xffu) != 0;
                } else if constexpr (BIAS == 2 || BIAS == 3) {
                    typedef typename VecOf<E>::v4 B4;
                    B4 hv = *reinterpret_cast<const B4*>(b_lds + ks_.b_off(r, nl));
#pragma unroll
                    for (int e = 0; e < 4; e++) bv[e] = (float)hv[e];
                } else if constexpr (BIAS == 4) {
                    f32x4 w = *reinterpret_cast<const f32x4*>(b_lds + ks_.b_off(r, nl));
#pragma unroll
                    for (int e = 0; e < 4; e++) bv[e] = w[e];
                } else if constexpr (BIAS == 5 && RAW) {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        s[q4 * 4 + e] = __builtin_fmaf(__builtin_fabsf(dist0 - (float)(8 * q4 + e)), raw_slope, s[q4 * 4 + e]);
                } else if constexpr (BIAS == 5) {
#pragma unroll
                    for (int e = 0; e < 4; e++) bv[e] = alibi_bias(neg_slope, ratio, mf, nf0 + (float)(8 * q4 + e));
                } else if constexpr (ROWB) {
                    f32x4 w = *reinterpret_cast<const f32x4*>(row_lds + n0 + nh + nl);
#pragma unroll
                    for (int e = 0; e < 4; e++) bv[e] = w[e];
                }
                if constexpr (!RAW) {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int i = q4 * 4 + e;
                        float x;
                        if constexpr (MASKED) {
                            x = __fmul_rn(s[i], qk_scale);
                            const int n = n0 + nh + nl + e;
                            const float t = CAUSAL && my_m < n ? kMask : 0.f;
                            float add = 0.f;
                            if (BIAS == 1) add = keep[e] ? 0.f : kMask;
                            if (BOOLROW) add = bv[e];
                            if (BIAS >= 2 && !BOOLROW) add = __fmul_rn(bv[e], kLog2e);
                            x = __fadd_rn(x, __fadd_rn(t, add));
                            x = n < N ? x : kLowest;  // (not an additive term: a float bias may mask a whole row below any)
                        } else if constexpr (BIAS == 1) {
                            x = keep[e] ? s[i] * qk_scale : s[i] * qk_scale + kMask;
                        } else if constexpr (BOOLROW) {
                            x = s[i] * qk_scale + bv[e];
                        } else {
                            x = s[i] * p.sm_scale + bv[e];
                        }
                        s[i] = x;
                    }
                }
            }
            // ---- P and O^T += V^T P^T (A = V^T gathered down the columns of the V rows), 16 keys
            // at a time: the MFMAs of the first 16 keys run while the exponentials of the second 16
            // are computed (head dim 256: all 32 at once, there are no registers for a second copy of the
            // rescaling) ----
            constexpr int PARTS = D <= 128 ? 2 : 1, PL = 16 / PARTS;
            if (GROWTH != kSum && rising) {
                float mx = -INFINITY;
#pragma unroll
                for (int i = 0; i < 16; i++) mx = fmaxf(mx, s[i]);
                mx = pair_max(mx) * to_log2;
                const bool higher = __builtin_amdgcn_ballot_w64(mx > m_i + 8.f) != 0;
                if (higher) raise(mx);
                if (GROWTH == kAfter) rising = higher;
            }
#pragma unroll
            for (int part = 0; part < PARTS; part++) {
                float pv[PL], rs;
                auto exps = [&]() {
                    rs = 0.f;
#pragma unroll
                    for (int j = 0; j < PL; j++) {
                        const int i = part * PL + j;
                        if constexpr (RAW || NAT) pv[j] = fast_exp2(__builtin_fmaf(s[i], to_log2, -m_i));
                        else pv[j] = fast_exp2(s[i] - m_i);
                        rs += pv[j];
                    }
                };
                exps();
                if (GROWTH != kRowMax && __builtin_amdgcn_ballot_w64(!(rs <= kRaise)) != 0) {
                    float mx = -INFINITY;
#pragma unroll
                    for (int i = part * PL; i < 16; i++) mx = fmaxf(mx, s[i]);
                    raise(pair_max(mx) * to_log2);
                    exps();
                    if (GROWTH == kAfter) rising = k > 0;  // (the first block always raises)
                }
                l_i += rs;  // per-lane partial sum; the two halves of a row are added at the end
#pragma unroll
                for (int kk = part * 2 / PARTS; kk < (part + 1) * 2 / PARTS; kk++) {
                    T8 pb;
#pragma unroll
                    for (int j = 0; j < 8; j++) pb[j] = (T)pv[kk * 8 + j - part * PL];
#pragma unroll
                    for (int db = 0; db < C::DB; db++) {
                        T8 a = SW::template col8_at<T8>(v_cols, nh + kk * 16, db);
                        o_acc[db] = mfma32(a, pb, o_acc[db]);
                    }
                }
            }
        };
        if constexpr (STEP_MASKED && D > 128) {
            // (head dim 256: one form of the softmax step in the edge loop; a second copy of the
            // 32 matrix products of a block there costs the registers that the interior loops need)
            softmax_step(std::true_type{});
        } else if constexpr (STEP_MASKED) {
            if (need_mask || !(qk_scale > 0.f) || !raw_ok) softmax_step(std::true_type{});
            else softmax_step(std::false_type{});
        } else {
            softmax_step(std::false_type{});
        }
        }
    };

    int n_fast = N / BK;  // leading steps that need no masks
    if (CAUSAL) n_fast = n_fast < (m0 + 1) / BK ? n_fast : (m0 + 1) / BK;
    if (n_fast > n_steps) n_fast = n_steps;
    if (!(qk_scale > 0.f) || !raw_ok) n_fast = 0;

    auto run = [&](auto bv_tag) {
        constexpr int BV = decltype(bv_tag)::value;
        stage_row();
        // The loads of this lane's rows issued above are the compiler's own.  Left in flight, they would
        // make it wait for "all vector-memory operations" at their first use inside EVERY step of the
        // loops (it cannot know that they land once), and that wait drains the queue of copies issued
        // steps ahead.  Waiting for them here keeps the loops free of it.
        wait_vmcnt<0>();
        // (After the wait and not before the loads, where it would be one for the first copies too.  B=32 H=12 M=N=197 D=64, us
        // per call, after / before: padding mask 13.45 / 13.96; no bias, B=8 H=16 S=512 15.4 / 15.9.)
        ks_.template prologue<BV>();
        if constexpr (TB == 0) split_q();  // (while the first copies are on their way)
        // the leading fast steps whose copies stay inside the tensors issue them without clamps
        const int n_lean = (BV != kByElement || TB == 0) ? ks_.lean_steps(n_fast) : 0;
        int k = 0;
        if (n_lean > 0) {
            ks_.template run_start<BV>(C::LA, C::NBS - 1);
#pragma unroll 1
            for (; k < n_lean; k++) kv_step(k, std::false_type{}, bv_tag, std::true_type{});
        }
#pragma unroll 1
        for (; k < n_fast; k++) kv_step(k, std::false_type{}, bv_tag, std::false_type{});
#pragma unroll 1
        for (; k < n_steps; k++) kv_step(k, std::true_type{}, bv_tag, std::false_type{});
    };
    if constexpr (TB == 0) {
        run(RowsTag<kByElement>{});
    } else {
        if constexpr (BY_DWORD) {
            if (p.bias_vec == kByChunk) run(RowsTag<kByChunk>{});
            else if (p.bias_vec == kByDword) run(RowsTag<kByDword>{});
            else run(RowsTag<kByElement>{});
        } else {
            if (p.bias_vec == kByChunk) run(RowsTag<kByChunk>{});
            else run(RowsTag<kByElement>{});
        }
    }

    // ---- epilogue (flash_attention.py:188-194) ----
    const float l_tot = pair_sum(l_i);
    // one of several shares of the keys: output and LSE go to this share's slice of the scratch (a share without a
    // visible key: zeros, and an LSE of -inf, which gives it no weight)
    const bool shared = p.n_splits > 1;
    const float inv_l = shared && l_tot == 0.f ? 0.f : 1.f / l_tot;
    float* lse_out = shared ? p.part_lse + ((int64_t)split * p.B * p.H + bh) * M : p.lse + ((int64_t)b * p.H + h) * M;
    // (the row index passes through an empty asm so that the store address is formed here and not
    // kept in two registers across the loops)
    int my_m_late = my_m;
    asm volatile("" : "+v"(my_m_late));
    if (g == 0 && my_m_late < M) lse_out[my_m_late] = m_i + fast_log2(l_tot);

    ks_.drain();  // K/V slots are dead and no copy is in flight: reuse their LDS for the output tile
    if (shared) {
        // a share stays in fp32 (the merge rounds once, like an unsplit run): 16 bytes per lane straight
        // from the accumulators (only problems with few query tiles come here)
        float* pf = reinterpret_cast<float*>(p.part_o) + (((int64_t)split * p.B * p.H + bh) * M + my_m_late) * D;
        if (my_m_late < M) {
#pragma unroll
            for (int db = 0; db < C::DB; db++) {
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const int d = db * 32 + 8 * q4 + 4 * g;
                    if (d < D) {
                        f32x4 w;
#pragma unroll
                        for (int e = 0; e < 4; e++) w[e] = o_acc[db][q4 * 4 + e] * inv_l;
                        *reinterpret_cast<f32x4*>(pf + d) = w;
                    }
                }
            }
        }
        return;
    }
    T* o_lds = reinterpret_cast<T*>(smem) + wave * 32 * OS;
#pragma unroll
    for (int db = 0; db < C::DB; db++) {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) {
            T4 pk;
#pragma unroll
            for (int e = 0; e < 4; e++) pk[e] = (T)(o_acc[db][q4 * 4 + e] * inv_l);
            *reinterpret_cast<T4*>(o_lds + r * OS + db * 32 + 8 * q4 + 4 * g) = pk;
        }
    }
    T* op = reinterpret_cast<T*>(p.o) + (int64_t)b * p.so.b + (int64_t)h * p.so.h;
    lds_wave_order();  // (a wave's own rows: no barrier)
    if constexpr (BIAS == 5 && CAUSAL && D == 64) {
        // (One read after the other.  With all of them in flight the compiler turned the order of this kernel's LOOPS: every LDS
        // read waited for by itself, us, H=16 S=1024 21.5 / 23.9, S=2048 39.4 / 44.6, H=64 62.7 / 63.0.)
        for (int c = lane; c < 32 * CPR; c += 64) {
            const int row = c / CPR, ch = c % CPR;
            if (mw + row < M && ch * 8 < p.d_v) gst16(op + (int64_t)(mw + row) * p.so.s + ch * 8, lds_read16(o_lds + row * OS + ch * 8));
        }
    } else {
        int lane_late = lane;  // (nothing formed of it here is kept in registers from the first copies on)
        asm volatile("" : "+v"(lane_late));
        i32x4 out[WR::COPIES];  // (all reads in flight together)
#pragma unroll
        for (int it = 0; it < WR::COPIES; it++)
            out[it] = lds_read16(o_lds + (it * 64 + lane_late) / CPR * OS + (it * 64 + lane_late) % CPR * 8);
#pragma unroll
        for (int it = 0; it < WR::COPIES; it++) {
            const int row = (it * 64 + lane_late) / CPR, ch = (it * 64 + lane_late) % CPR;
            if (mw + row < M && ch * 8 < p.d_v) gst16(op + (int64_t)(mw + row) * p.so.s + ch * 8, out[it]);
        }
    }
}

// out = sum over the shares of 2^(lse_s - lse) out_s with lse = log2 sum 2^lse_s: the softmax over
// all keys from the softmaxes over the shares.  One thread per 8 head-dim elements of a row.
template <typename T, int D> __global__ __launch_bounds__(256) void fa_fwd_merge_kernel(const FwdParams p) {
    typedef typename VecOf<T>::v8 T8;
    constexpr int TPR = D / 8;
    const int64_t rows = (int64_t)p.B * p.H * p.M;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = idx / TPR;
    const int c = (int)(idx % TPR);
    if (row >= rows || c * 8 >= p.d_v) return;
    // (unrolled: up to 32 shares, whose loads would be a chain of latencies)
    float mx = -INFINITY;
#pragma unroll 8
    for (int s = 0; s < p.n_splits; s++) mx = fmaxf(mx, p.part_lse[s * rows + row]);
    float sum = 0.f;
#pragma unroll 8
    for (int s = 0; s < p.n_splits; s++) sum += fast_exp2(p.part_lse[s * rows + row] - mx);
    const float lse = mx + fast_log2(sum);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 0; s < p.n_splits; s++) {
        const float w = fast_exp2(p.part_lse[s * rows + row] - lse);
        const float* src = reinterpret_cast<const float*>(p.part_o) + (s * rows + row) * D + c * 8;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(src), hi = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            acc[e] += w * lo[e];
            acc[4 + e] += w * hi[e];
        }
    }
    const int m = (int)(row % p.M);
    const int64_t bh = row / p.M;
    const int b = (int)(bh / p.H), h = (int)(bh % p.H);
    T8 o8;
#pragma unroll
    for (int e = 0; e < 8; e++) o8[e] = (T)acc[e];
    gst16(reinterpret_cast<T*>(p.o) + (int64_t)b * p.so.b + (int64_t)h * p.so.h + (int64_t)m * p.so.s + c * 8, as_raw(o8));
    if (c == 0) p.lse[row] = lse;
}

template <typename T, int D, int BIAS, bool CAUSAL> static hipError_t launch_one(const FwdParams& p, hipStream_t st) {
    dim3 grid((unsigned)(p.n_mtiles * p.n_splits * p.B * p.H));
    hipLaunchKernelGGL((fa_fwd_kernel<T, D, BIAS, CAUSAL>), grid, dim3(256), 0, st, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.n_splits == 1) return e;
    const int64_t threads = (int64_t)p.B * p.H * p.M * (D / 8);
    hipLaunchKernelGGL((fa_fwd_merge_kernel<T, D>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, p);
    return hipGetLastError();
}

template <typename T, int D> static hipError_t launch_bias(const FwdParams& p, int bias, bool causal, hipStream_t st) {
#define FA_CASE(BK)                                                        \
    case BK:                                                               \
        return causal ? launch_one<T, D, BK, true>(p, st) : launch_one<T, D, BK, false>(p, st);
    // a bias without a row dimension is staged once per work-group instead of streamed
    if (p.row_bias_kind != 0) bias = p.row_bias_kind == 1 ? 7 : 6;
    switch (bias) {
        FA_CASE(0)
        FA_CASE(1)
        FA_CASE(2)
        FA_CASE(3)
        FA_CASE(4)
        FA_CASE(5)
        FA_CASE(6)
        FA_CASE(7)
    }
#undef FA_CASE
    return hipErrorInvalidValue;
}

// This file is compiled once per head dimension (-DFA_HEAD_DIM=16 ... 256, 96 for those of 128 that are no larger); each object exports
// launch_fwd_d<FA_HEAD_DIM>.  dtype: 0 = fp16, 1 = bf16.  The caller has validated every argument.
#ifndef FA_HEAD_DIM
#error "compile with -DFA_HEAD_DIM=<16|32|64|96|128|256>"
#endif
template <int D> hipError_t launch_fwd_d(const FwdParams& p, int dtype, int bias, bool causal, hipStream_t st);
template <> hipError_t launch_fwd_d<FA_HEAD_DIM>(const FwdParams& p, int dtype, int bias, bool causal, hipStream_t st) {
    if (dtype == 0) return launch_bias<_Float16, FA_HEAD_DIM>(p, bias, causal, st);
    return launch_bias<__bf16, FA_HEAD_DIM>(p, bias, causal, st);
}

}  // namespace fa
