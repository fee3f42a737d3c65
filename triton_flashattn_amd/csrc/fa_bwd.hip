// Backward attention kernels for gfx950: dK, dV, dBias in one kernel over key tiles, dQ in a
// second kernel over query tiles.  Every output element has exactly one writer, so results are
// reproducible run to run, like the reference's (no atomics).
//
// Replaces _attn_bwd_preprocess, _attn_bwd_dkdv and _attn_bwd_dq of the reference
// (/root/reference/flash_attention.py:197-646) and the host-side K / bias pre-scales
// (flash_attention.py:699-704), which become fp32 multiplies inside the kernels.
//
//   fa_bwd_prep_kernel   delta[b,h,m] = sum_d o * do                  (flash_attention.py:215-227)
//   fa_bwd_kernel        dK, dV, dBias of 128 (or 64) keys per work-group, head dims 128 and 256 (flash_attention.py:237-454;
//                        fa_bwd_narrow.hip holds the kernel of the smaller ones, but for the biases of pair_of_waves)
//   fa_bwd_dq_kernel     dQ of 128 query rows per work-group          (flash_attention.py:458-646)
#include <type_traits>

#include "fa_common.hpp"
#include "fa_params.hpp"

namespace fa {

// ---------------------------------------------------------------------------------------------
// delta of one row: every 16-byte chunk c of the row is summed element by element with fused
// multiply-adds, then the D / 8 chunk sums are added pairwise, c with c ^ w for w = D / 16, ..., 2, 1.
// (fa_bwd_dq_kernel forms the same sums in the same order when it stands in for this kernel.)
template <typename T, int D>
__global__ __launch_bounds__(256) void fa_bwd_prep_kernel(const BwdParams p) {
    constexpr int LPR = D / 8;         // lanes per row (16 bytes each)
    constexpr int RPB = 256 / LPR;     // rows per block
    typedef typename VecOf<T>::v8 T8;
    const int64_t rows = (int64_t)p.B * p.H * p.M;
    const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / LPR;
    const int c = threadIdx.x % LPR;
    float acc = 0.f;
    if (row < rows && c * 8 < p.d_v) {
        const int m = (int)(row % p.M);
        const int bh = (int)(row / p.M);
        const int b = bh / p.H, h = bh % p.H;
        const T* op = reinterpret_cast<const T*>(p.o) + (int64_t)b * p.so.b + (int64_t)m * p.so.s + (int64_t)h * p.so.h;
        const T* dp = reinterpret_cast<const T*>(p.dout) + (int64_t)b * p.sdo.b + (int64_t)m * p.sdo.s + (int64_t)h * p.sdo.h;
        T8 ov = as_vec<T8>(gld16(op + c * 8));
        T8 dv = as_vec<T8>(gld16(dp + c * 8));
#pragma unroll
        for (int e = 0; e < 8; e++) acc = __builtin_fmaf((float)ov[e], (float)dv[e], acc);
    }
#pragma unroll
    for (int w = LPR / 2; w >= 1; w >>= 1) acc += __shfl_xor(acc, w, 64);
    if (row < rows && c == 0) p.delta[row] = acc;
}

// ---------------------------------------------------------------------------------------------
// dQ kernel: a work-group owns 128 query rows (Q^T and dO^T in registers), streams K / V rows
// and recomputes S^T = K Q^T and dP^T = V dO^T, so that dS^T sits in the accumulator layout that
// dQ^T += K^T dS^T wants as its B operand.  K, V and the bias slices arrive through the same
// counted direct-to-LDS copy rings as in the forward kernel.  Replaces _attn_bwd_dq
// (flash_attention.py:458-646).
//
// FROM_DS: when the key-tile kernel has just written dBias in the element type of q, that tensor IS
// dS rounded exactly as the reference rounds it before this product (flash_attention.py:516-520);
// an fp32 dBias is dS itself and is rounded here.  The kernel then reads the dBias slices through
// the bias ring instead of the bias, skips both recomputed products, the exponentials and the V
// rows, and is one product instead of three.
template <typename T, int D, int BIAS, bool CAUSAL, bool FROM_DS = false>
__global__ __launch_bounds__(256, (StreamCfg<D, stream_kind(BIAS)>::MIN_BLOCKS)) void fa_bwd_dq_kernel(const BwdParams p) {
    static_assert(!FROM_DS || BIAS == 4 || (BIAS == 2 && __is_same(T, _Float16)) || (BIAS == 3 && __is_same(T, __bf16)),
                  "dS can stand in for the recomputation only in fp32 or in the element type of q");
    constexpr int TB = tile_kind(BIAS);  // kind of bias tile that is streamed (none for ALiBi)
    typedef StreamCfg<D, stream_kind(BIAS)> C;
    typedef Swz<D> SW;
    typedef typename VecOf<T>::v8 T8;
    typedef typename VecOf<T>::v4 T4;
    typedef typename BiasElem<tile_kind(BIAS)>::type E;
    constexpr int BM = C::BM, BK = C::BK, OS = C::OS, CPR = C::CPR;
    constexpr bool ROWB = BIAS >= 6;     // the same bias for every query row, kept as an fp32 row in LDS
    constexpr bool BOOLROW = BIAS == 7;  // ... a bool mask: the row holds 0 or the mask term, in log2 units
    static_assert(!(FROM_DS && ROWB), "a row-broadcast bias has no dense dS");

    // Q and dO rows come through LDS (WaveRows) where StreamCfg has a place for them.  A place for dO beside that of Q where it
    // costs no work-group on a CU; else one after the other.  Not causal ALiBi at head dim 128 and a causal fp32 tile at 64 (us,
    // the lanes' own loads / LDS: ALiBi H=16 S=2000 53.2 / 56.1, B=2 H=8 S=2048 55.5 / 57.6, H=32 S=1001 33.4 / 34.4, but B=16 H=12
    // S=197 20.4 / 18.0; fp32 B=2 H=4 S=128 9.3 / 10.0, B=4 H=8 S=512 17.7 / 18.2, B=8 H=8 S=256 for all batches 13.0 / 13.9).
    typedef WaveRows<T, D> WR;
    constexpr bool STAGED = C::STAGE != C::kNowhere && !FROM_DS && !(CAUSAL && ((BIAS == 5 && D == 128) || (BIAS == 4 && D == 64)));
    constexpr bool BESIDE = STAGED && !ROWB && (C::LDS_BYTES + 4 * WR::BYTES) * C::ROOM <= 163840;
    constexpr int LDS_BYTES = STAGED ? C::LDS_BYTES : C::LOOP_BYTES;
    __shared__ __align__(1024) unsigned char smem[LDS_BYTES + (ROWB ? kRowBiasKeys * 4 : 0) + (BESIDE ? 4 * WR::BYTES : 0)];
    const float* row_lds = reinterpret_cast<const float*>(smem + LDS_BYTES);

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int r = lane & 31, g = lane >> 5;

    int mt, bh;
    // (ALiBi at D = 32: longest first in any grid, 76.1 -> 69.6 us at B=1 H=16 S=4096; at 16, 64 and 128 pairing is 1 to 4 % faster)
    constexpr bool PAIRS = !(BIAS == 5 && D == 32);
    decode_block<CAUSAL, typename std::conditional<PAIRS, C, OnePerCu>::type>(blockIdx.x, p.n_mtiles * p.dq_splits, p.B * p.H, mt, bh);
    // With the keys split between work-groups (never when causal) this one sees keys key0 ..
    // key0 + N - 1 as if they were all there are (its dq is a share, summed afterwards); only ALiBi
    // needs to know better.
    const int split = mt % p.dq_splits;
    mt /= p.dq_splits;
    const int key0 = split * p.dq_keys_per_split;
    if (CAUSAL) mt = p.n_mtiles - 1 - mt;  // longest rows first
    const int b = bh / p.H, h = bh % p.H;
    const int M = p.M;
    const int N = p.dq_splits > 1 ? (p.N - key0 < p.dq_keys_per_split ? p.N - key0 : p.dq_keys_per_split) : p.N;
    const int m0 = mt * BM;
    const int mw = m0 + wave * 32;  // first query row of this wave
    const int my_m = mw + r;

    const T* qp = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.sq.b + (int64_t)h * p.sq.h;
    const T* kp = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.sk.b + (int64_t)h * p.sk.h + (int64_t)key0 * p.sk.s;
    const T* vp = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.sv.b + (int64_t)h * p.sv.h + (int64_t)key0 * p.sv.s;
    const E* bp = nullptr;
    if (TB != 0) bp = reinterpret_cast<const E*>(p.bias) + (int64_t)b * p.sbias.b + (int64_t)h * p.sbias.h + (int64_t)key0 * p.sbias.n;
    float neg_slope = 0.f, ratio = 0.f;  // ALiBi: slope of this head, key positions per query row
    if (BIAS == 5) {
        neg_slope = -reinterpret_cast<const float*>(p.bias)[h];
        ratio = (float)p.N / (float)p.M;
    }
    const float log2_slope = neg_slope * kLog2e;
    if (FROM_DS) bp = reinterpret_cast<const E*>(p.dbias) + (int64_t)b * p.sdbias.b + (int64_t)h * p.sdbias.h + (int64_t)key0 * p.sdbias.n;

    const LiveChunks chunks{p.d_qk / 8, p.qk_inv};
    const unsigned rows_l = SW::rows_lane(lane), cols_l = SW::cols_lane(lane);
    typedef KeyStream<T, D, stream_kind(BIAS), !FROM_DS> KS;
    KS ks_;
    ks_.init(smem, kp, vp, bp, p.sk.s, p.sv.s, FROM_DS ? p.sdbias.m : p.sbias.m, FROM_DS ? p.sdbias.n : p.sbias.n, M, N,
             mw, wave, lane, chunks, p.d_v / 8);
    constexpr bool BY_DWORD = BIAS == 4 && D <= 64 && !FROM_DS;

    // Q^T and dO^T as B operands: column my_m, k = d
    const T* dop = reinterpret_cast<const T*>(p.dout) + (int64_t)b * p.sdo.b + (int64_t)h * p.sdo.h;
    const T* outp = reinterpret_cast<const T*>(p.o) + (int64_t)b * p.so.b + (int64_t)h * p.so.h;
    T8 qreg[C::KSTEPS], doreg[C::KSTEPS];
    auto load_rows = [&]() {
#pragma unroll
        for (int ks = 0; ks < C::KSTEPS; ks++) {
            i32x4 rq = {0, 0, 0, 0}, rd = {0, 0, 0, 0};
            const int d = ks * 16 + 8 * g;
            if (!FROM_DS && my_m < M) rq = gld16(qp + (int64_t)my_m * p.sq.s + (D <= 128 ? chunks.wrap(2 * ks + g) * 8 : d));
            if (!FROM_DS && my_m < M && d < p.d_v) rd = gld16(dop + (int64_t)my_m * p.sdo.s + d);
            qreg[ks] = as_vec<T8>(rq);
            doreg[ks] = as_vec<T8>(rd);
        }
    };
    if constexpr (!STAGED) load_rows();
    auto split_q = [&]() {
        if (D <= 128 && !FROM_DS && p.d_qk < D) {
#pragma unroll
            for (int ks = 0; ks < C::KSTEPS; ks++) qreg[ks] = chunks.part(qreg[ks], 2 * ks + g, C::CPR);
        }
    };
    // LSE (log2 units) and delta of this lane's query row
    float lse_i = 0.f, delta_i = 0.f;
    if (!FROM_DS && my_m < M) {
        lse_i = p.lse[((int64_t)b * p.H + h) * M + my_m];
        if (!p.dq_makes_delta) delta_i = p.delta[((int64_t)b * p.H + h) * M + my_m];
    }
    // Where this kernel runs first it forms delta = sum_d o * do itself (flash_attention.py:215-227), bit for bit as
    // fa_bwd_prep_kernel does: a chunk of 8 by fused multiply-adds, then chunk c with chunk c ^ w for w = D / 16, ..., 1.  The
    // dK/dV kernel reads what is stored.
    // O in the order of a WaveRows tile: chunk c = 64 it + l of the 32 rows to lane l, which finds dO's beside it in LDS
    constexpr bool O_AS_TILE = STAGED && D != 96;
    i32x4 o_raw[O_AS_TILE ? WR::COPIES : 1];
    auto o_chunk = [&](int it, int& row, int& src) {
        row = (it * 64 + lane) / CPR;
        src = ((it * 64 + lane) % CPR) ^ SW::f(row);
    };
    auto load_o = [&]() {
        if constexpr (O_AS_TILE) {
#pragma unroll
            for (int it = 0; it < WR::COPIES; it++) {
                int row, src;
                o_chunk(it, row, src);
                const int m = mw + row < M ? mw + row : M - 1;
                o_raw[it] = i32x4{0, 0, 0, 0};
                if (p.dq_makes_delta && src * 8 < p.d_v) o_raw[it] = gld16(outp + (int64_t)m * p.so.s + src * 8);
            }
        }
    };
    auto make_delta = [&](unsigned do_tile, auto tile_tag) {  // tile_tag: dO stands in LDS
        if (!p.dq_makes_delta) return;
        if constexpr (O_AS_TILE && decltype(tile_tag)::value) {
            constexpr int RPI = 64 / CPR;  // rows of a copy
            float sum[WR::COPIES];
#pragma unroll
            for (int it = 0; it < WR::COPIES; it++) {
                int row, src;
                o_chunk(it, row, src);
                const T8 ov = as_vec<T8>(o_raw[it]), dv = as_vec<T8>(lds_read16_at(do_tile + 1024 * it + 16 * lane));
                float a = 0.f;
#pragma unroll
                for (int e = 0; e < 8; e++) a = __builtin_fmaf((float)ov[e], (float)dv[e], a);
                sum[it] = src * 8 < p.d_v ? a : 0.f;
            }
#pragma unroll
            for (int w = CPR / 2; w >= 1; w >>= 1)
#pragma unroll
                for (int it = 0; it < WR::COPIES; it++) sum[it] += __shfl_xor(sum[it], w, 64);
#pragma unroll
            for (int it = 0; it < WR::COPIES; it++) {
                const float x = __shfl(sum[it], r % RPI * CPR, 64);
                if (r / RPI == it) delta_i = x;
            }
        } else {
            constexpr int NP = D == 96 ? 8 : C::KSTEPS;  // (delta of D = 96 is formed like that of 128, whose last chunks are zero)
            float part[NP];
#pragma unroll
            for (int ks = C::KSTEPS; ks < NP; ks++) part[ks] = 0.f;
#pragma unroll
            for (int ks = 0; ks < C::KSTEPS; ks++) {
                i32x4 ro = {0, 0, 0, 0};
                if (my_m < M && ks * 16 + 8 * g < p.d_v) ro = gld16(outp + (int64_t)my_m * p.so.s + ks * 16 + 8 * g);
                const T8 ov = as_vec<T8>(ro);
                float a = 0.f;
#pragma unroll
                for (int e = 0; e < 8; e++) a = __builtin_fmaf((float)ov[e], (float)doreg[ks][e], a);
                part[ks] = a;
            }
#pragma unroll
            for (int hs = NP / 2; hs >= 1; hs >>= 1)
#pragma unroll
                for (int ks = 0; ks < hs; ks++) part[ks] = part[ks] + part[ks + hs];
            delta_i = part[0] + __shfl_xor(part[0], 32, 64);
        }
        if (g == 0 && my_m < M && split == 0) p.delta[((int64_t)b * p.H + h) * M + my_m] = delta_i;
    };
    if constexpr (!STAGED && !FROM_DS) {
        if constexpr (TB != 0) split_q();  // (kernels of a bias tile have no registers for it later)
        make_delta(0, std::false_type{});
    }

    int n_steps = (N + BK - 1) / BK;
    if (CAUSAL) {
        int last = (m0 + BM - 1) / BK + 1;  // steps holding keys <= last row of this work-group
        n_steps = n_steps < last ? n_steps : last;
    }

    const float qk_scale = p.sm_scale * kLog2e;
    // bool mask, unmasked steps: the two values that the offset of a score's exponent can take (the lane
    // is one query row), so that an element costs a select and not a select and a subtraction
    const float neg_lse = 0.f - lse_i, mask_lse = kMask - lse_i;
    f32x16 dq_acc[C::DB];  // dQ^T: rows = head dim, column = my_m
#pragma unroll
    for (int db = 0; db < C::DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) dq_acc[db][i] = 0.f;

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
        const unsigned k_tile = ks_.k_addr(k), v_tile = ks_.v_addr(k);  // operand reads by address
        const unsigned char* b_lds = ks_.b_lds(k);
        static_assert(TB == 0 || C::NH == 1, "a bias slot covers one 32-key block");
        // Interior steps of two blocks (no bias tile), as in the forward kernel: S and dP of block 1 are issued between the
        // element-wise work of block 0, and the dQ product of block 0 between that of block 1, one fenced slot per two
        // elements.  Operands are fetched a phase ahead, above head dim 64 one slot ahead.  Same bits; us, one block after
        // the other -> this: B=4 H=16 S=2048 D=64 causal 65.1 -> 60.9, B=1 H=16 S=6001 D=128 causal 218 -> 206, B=2 H=16
        // M=N=4096 D=128 362 -> 350.  Not with a staged bias row up to head dim 64, whose reads between the fences it waits for:
        // B=2 H=8 M=N=577 D=32 11.0 -> 11.9, B=4 H=16 S=2048 D=64 causal 63 -> 65.
        if constexpr (!STEP_MASKED && C::NH == 2 && !FROM_DS && !(ROWB && D <= 64)) {
            constexpr int NS = 2 * C::KSTEPS, NP = 2 * C::DB;  // matrix instructions of S and dP, and of dQ, per block
            constexpr bool AHEAD = D <= 64;
            constexpr int NSS = AHEAD ? NS : (NS + 7) / 8, NPS = AHEAD ? NP : (NP + 7) / 8;  // operands fetched at a time
            auto fence = []() { __builtin_amdgcn_sched_barrier(0); };
            T8 ra[AHEAD ? 1 : 2][NSS], ca[AHEAD ? 1 : 2][NPS];
            f32x16 sc[2], dpc[2];
            auto load_rows = [&](int nb, int slot) {  // operands of S and dP of block nb: of slot `slot` of 8, or all
                const int first = AHEAD ? 0 : slot * NS / 8, last = AHEAD ? NS : (slot + 1) * NS / 8;
#pragma unroll
                for (int at = first; at < last; at++) {
                    ra[AHEAD ? 0 : slot & 1][at - first] = at < C::KSTEPS ? SW::template row8_at<T8>(k_tile + rows_l, nb * 32, at)
                                                                 : SW::template row8_at<T8>(v_tile + rows_l, nb * 32, at - C::KSTEPS);
                }
            };
            auto load_cols = [&](int nb, int slot) {
                const int first = AHEAD ? 0 : slot * NP / 8, last = AHEAD ? NP : (slot + 1) * NP / 8;
#pragma unroll
                for (int at = first; at < last; at++) {
                    ca[AHEAD ? 0 : slot & 1][at - first] = SW::template col8_at<T8>(k_tile + cols_l, nb * 32 + (at / C::DB) * 16, at % C::DB);
                }
            };
            // the matrix instructions of slot j of 8 of S and dP, and of dQ
            auto mma_s = [&](int nb, int j) {
                if (!AHEAD && j < 7) load_rows(nb, j + 1);
#pragma unroll
                for (int i = j * NS / 8; i < (j + 1) * NS / 8; i++) {
                    const T8 a = ra[AHEAD ? 0 : j & 1][AHEAD ? i : i - j * NS / 8];
                    if (i < C::KSTEPS) sc[nb] = mfma32(a, qreg[i], sc[nb]);
                    else dpc[nb] = mfma32(a, doreg[i - C::KSTEPS], dpc[nb]);
                }
            };
            auto mma_dq = [&](int nb, const T8 (&ds)[2], int j) {
                if (!AHEAD && j < 7) load_cols(nb, j + 1);
#pragma unroll
                for (int i = j * NP / 8; i < (j + 1) * NP / 8; i++)
                    dq_acc[i % C::DB] = mfma32(ca[AHEAD ? 0 : j & 1][AHEAD ? i : i - j * NP / 8], ds[i / C::DB], dq_acc[i % C::DB]);
            };
            auto elements = [&](int nb, T8 (&ds)[2], auto&& between) {
                f32x4 bias4;
#pragma unroll
                for (int j = 0; j < 8; j++) {
#pragma unroll
                    for (int i = 2 * j; i < 2 * j + 2; i++) {
                        float off = -lse_i;
                        if constexpr (ROWB) {
                            if (i % 4 == 0) bias4 = *reinterpret_cast<const f32x4*>(row_lds + n0 + nb * 32 + 2 * i + 4 * g);
                            off = BOOLROW ? bias4[i & 3] - lse_i : __builtin_fmaf(bias4[i & 3], kLog2e, -lse_i);
                        }
                        const float pv = fast_exp2(__builtin_fmaf(sc[nb][i], qk_scale, off));
                        ds[i >> 3][i & 7] = (T)(pv * (dpc[nb][i] - delta_i));
                    }
                    fence();
                    between(j);
                    fence();
                }
            };
#pragma unroll
            for (int nb = 0; nb < 2; nb++)
#pragma unroll
                for (int i = 0; i < 16; i++) sc[nb][i] = dpc[nb][i] = 0.f;
            load_rows(0, 0);
#pragma unroll
            for (int j = 0; j < 8; j++) mma_s(0, j);
            issue_ahead();  // in the shadow of the MFMAs just issued
            load_rows(1, 0);
            fence();
            T8 ds0[2], ds1[2];
            elements(0, ds0, [&](int j) { mma_s(1, j); });
            load_cols(0, 0);
            fence();
            elements(1, ds1, [&](int j) { mma_dq(0, ds0, j); });
            load_cols(1, 0);
#pragma unroll
            for (int j = 0; j < 8; j++) mma_dq(1, ds1, j);
            return;
        }
        // The step is consumed 32 keys at a time, so that only one 32 x 32 score block is live.
#pragma unroll
        for (int nb = 0; nb < C::NH; nb++) {
            const int nh = nb * 32;  // first key of this block inside the step
            __builtin_amdgcn_sched_barrier(0);  // keep the blocks apart
            // blocks entirely above this wave's diagonal or past the last key contribute nothing
            if (STEP_MASKED && ((CAUSAL && n0 + nh > mw + 31) || n0 + nh >= N)) {
                if (nb == 0) issue_ahead();  // every wave issues its copies in every step
                continue;
            }
            const bool need_mask = STEP_MASKED && ((n0 + nh + 32 > N) || (CAUSAL && n0 + nh + 31 > mw));
            T8 dsb[2];
            if constexpr (FROM_DS) {
                // dS^T of the block straight from the dBias slice: 4 consecutive keys per read, in
                // accumulator order; keys past N hold whatever column 0 holds and count as zero
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const int nl = 8 * q4 + 4 * g;
                    T4 hv;
                    if constexpr (BIAS == 4) {
                        const f32x4 w = *reinterpret_cast<const f32x4*>(b_lds + ks_.b_off(r, nl));
#pragma unroll
                        for (int e = 0; e < 4; e++) hv[e] = (T)w[e];
                    } else {
                        hv = *reinterpret_cast<const T4*>(b_lds + ks_.b_off(r, nl));
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int i = q4 * 4 + e;
                        T val = hv[e];
                        if (STEP_MASKED && n0 + nh + nl + e >= N) val = (T)0.f;
                        dsb[i >> 3][i & 7] = val;
                    }
                }
            } else {

            // ---- S^T = K Q^T : s[i] is key n0 + nh + 8 (i/4) + 4 g + i%4, query my_m ----
            f32x16 s;
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] = 0.f;
#pragma unroll
            for (int ks = 0; ks < C::KSTEPS; ks++) {
                T8 a = SW::template row8_at<T8>(k_tile + rows_l, nh, ks);
                s = mfma32(a, qreg[ks], s);
            }

            // ---- dP^T = V dO^T ----
            f32x16 dp;
#pragma unroll
            for (int i = 0; i < 16; i++) dp[i] = 0.f;
#pragma unroll
            for (int ks = 0; ks < C::KSTEPS; ks++) {
                T8 a = SW::template row8_at<T8>(v_tile + rows_l, nh, ks);
                dp = mfma32(a, doreg[ks], dp);
            }
            if (nb == 0) issue_ahead();  // in the shadow of the MFMAs just issued

            // ---- P = 2^(S*scale + bias - LSE), dS = P (dP - delta) (flash_attention.py:497-517).
            // Masked tiles follow the reference's additive -1e6 arithmetic term by term; keys past N have P = 0.
            auto ds_step = [&](auto masked_tag) {
                constexpr bool MASKED = decltype(masked_tag)::value;
                const float nf0 = (float)(key0 + n0 + nh + 4 * g);              // ALiBi: the lane's first key,
                const float dist0 = __builtin_fmaf((float)my_m, ratio, -nf0);  // and the distance to it
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const int nl = 8 * q4 + 4 * g;  // first of 4 consecutive keys of the block
                    float bv[4] = {0.f, 0.f, 0.f, 0.f};  // bias in natural units
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
                    } else if constexpr (BIAS == 5 && MASKED) {
#pragma unroll
                        for (int e = 0; e < 4; e++) bv[e] = alibi_bias(neg_slope, ratio, (float)my_m, nf0 + (float)(8 * q4 + e));
                    } else if constexpr (ROWB) {
                        f32x4 w = *reinterpret_cast<const f32x4*>(row_lds + n0 + nh + nl);
#pragma unroll
                        for (int e = 0; e < 4; e++) bv[e] = w[e];
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int i = q4 * 4 + e;
                        float pv;
                        if constexpr (MASKED) {
                            const int n = n0 + nh + nl + e;
                            const float t = CAUSAL && my_m < n ? kMask : 0.f;
                            float add = 0.f;
                            if (BIAS == 1) add = keep[e] ? 0.f : kMask;
                            if (BOOLROW) add = bv[e];
                            if (BIAS >= 2 && !BOOLROW) add = __fmul_rn(bv[e], kLog2e);
                            pv = fast_exp2(__fadd_rn(__fmul_rn(s[i], qk_scale), __fadd_rn(t, add)) - lse_i);
                            pv = n < N ? pv : 0.f;  // (not an additive term: the LSE may lie below any)
                        } else if constexpr (BIAS == 0) {
                            pv = fast_exp2(__builtin_fmaf(s[i], qk_scale, -lse_i));
                        } else if constexpr (BIAS == 5) {
                            const float dist = dist0 - (float)(8 * q4 + e);
                            pv = fast_exp2(__builtin_fmaf(__builtin_fabsf(dist), log2_slope, __builtin_fmaf(s[i], qk_scale, -lse_i)));
                        } else if constexpr (BIAS == 1) {
                            pv = fast_exp2(__builtin_fmaf(s[i], qk_scale, keep[e] ? neg_lse : mask_lse));
                        } else if constexpr (BOOLROW) {
                            pv = fast_exp2(__builtin_fmaf(s[i], qk_scale, bv[e] - lse_i));
                        } else {
                            pv = fast_exp2(__builtin_fmaf(bv[e], kLog2e, __builtin_fmaf(s[i], qk_scale, -lse_i)));
                        }
                        dsb[i >> 3][i & 7] = (T)(pv * (dp[i] - delta_i));
                    }
                }
            };
            if constexpr (STEP_MASKED) {
                if (need_mask || !(qk_scale > 0.f)) ds_step(std::true_type{});
                else ds_step(std::false_type{});
            } else {
                ds_step(std::false_type{});
            }
            }

            // ---- dQ^T += K^T dS^T : A = K^T gathered down the columns of the K tile ----
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
#pragma unroll
                for (int db = 0; db < C::DB; db++) {
                    T8 a = SW::template col8_at<T8>(k_tile + cols_l, nh + kk * 16, db);
                    dq_acc[db] = mfma32(a, dsb[kk], dq_acc[db]);
                }
            }
            if (FROM_DS && nb == 0) issue_ahead();  // in the shadow of the MFMAs just issued
        }
    };

    int n_fast = N / BK;  // leading steps that need no masks
    if (CAUSAL) n_fast = n_fast < (m0 + 1) / BK ? n_fast : (m0 + 1) / BK;
    if (n_fast > n_steps) n_fast = n_steps;
    // (query rows past M need no mask: a lane is one row, and such a row is not stored.  Run in masked steps, a
    // ragged last tile was the longest of a causal grid: B=1 H=16 M=N=6001 D=128 0.298 -> 0.218 ms)
    if (!(qk_scale > 0.f)) n_fast = 0;
    // Up to 64 rows, half of a tile or less: the lanes' own loads.  Waves without rows of their own copy the last one over and
    // over, and the longer way to the first step is all of such a call.  From head dim 64 on (us, LDS / own loads: D=128 B=2 H=4
    // S=64 no bias 8.7 / 7.9, byte mask 9.4 / 8.7, row mask 9.4 / 8.3, causal fp32 10.1 / 9.1, H=8 M=32 N=1024 12.6 / 11.5; D=80 bf16
    // B=2 H=4 S=64 10.0 / 9.2; D=64 no bias 6.2 / 5.6, fp32 for all batches 7.4 / 6.4; at 128 rows the two are even).
    const bool few_rows = STAGED && D >= 64 && M <= 64;
    auto run = [&](auto bv_tag) {
        constexpr int BV = decltype(bv_tag)::value;
        auto stage_row = [&]() {
            if (ROWB)
                stage_row_bias(reinterpret_cast<float*>(smem + LDS_BYTES), p.bias, p.row_bias_kind,
                               (int64_t)b * p.sbias.b + (int64_t)h * p.sbias.h + (int64_t)key0 * p.sbias.n, p.sbias.n, N, tid);
        };
        if (STAGED && few_rows) {
            load_rows();
            split_q();
            make_delta(0, std::false_type{});
            stage_row();
            wait_vmcnt<0>();
            ks_.template prologue<BV>();
        } else if constexpr (STAGED) {
            constexpr bool FIRST_KV = C::STAGE != C::kOwnRing;  // the first copies of the stream need not wait for the rows
            constexpr int PRO = FIRST_KV ? KS::template prologue_copies<BV>() : 0;
            const unsigned q_tile = ks_.stage_addr(), do_tile = BESIDE ? ks_.lds_kv + LDS_BYTES + ks_.wave_s * WR::BYTES : q_tile;
            auto copy = [&](bool is_q) {
                const unsigned saved_m0 = lds_copy_begin();
                if (is_q) WR::issue(qp, p.sq.s, mw, M, q_tile, lane, [&](int c) { return D <= 128 ? chunks.wrap(c) : c; });
                else WR::issue(dop, p.sdo.s, mw, M, do_tile, lane, [&](int c) { return live_chunk(c, p.d_v / 8); });
                lds_copy_end(saved_m0);
            };
            load_o();
            copy(true);
            if constexpr (BESIDE) copy(false);
            if constexpr (FIRST_KV) ks_.template prologue<BV>();
            WR::template arrived<PRO + (BESIDE ? WR::COPIES : 0)>();
#pragma unroll
            for (int ks = 0; ks < C::KSTEPS; ks++) qreg[ks] = SW::template row8_at<T8>(q_tile + rows_l, 0, ks);
            if constexpr (!BESIDE) {
                WR::done();
                copy(false);
                WR::template arrived<0>();
            } else {
                WR::template arrived<PRO>();
            }
#pragma unroll
            for (int ks = 0; ks < C::KSTEPS; ks++) {
                const i32x4 x = as_raw(SW::template row8_at<T8>(do_tile + rows_l, 0, ks));
                doreg[ks] = as_vec<T8>(ks * 16 + 8 * g < p.d_v ? x : i32x4{0, 0, 0, 0});
            }
            split_q();
            make_delta(do_tile, std::true_type{});
            if constexpr (!FIRST_KV) {
                WR::done();
                ks_.template prologue<BV>();
            }
            stage_row();
        }
        // The loads of this lane's rows issued above are the compiler's own.  Left in flight, they would
        // make it wait for "all vector-memory operations" at their first use inside EVERY step of the
        // loops (it cannot know that they land once), and that wait drains the queue of copies issued
        // steps ahead.  Waiting for them here keeps the loops free of it.
        wait_vmcnt<0>();
        if constexpr (!STAGED) {
            stage_row();
            ks_.template prologue<BV>();
            if constexpr (TB == 0 && !FROM_DS) split_q();  // (while the first copies are on their way)
        }
        // the leading fast steps whose copies stay inside the tensors issue them without clamps (not at head dim 256 in the
        // work-groups with the last rows of a bias, which have no registers for offsets that are clamped to them: us, without /
        // with, bf16 tile H=32 S=1001 causal 73.3 / 82.2, B=12 H=16 S=577 causal 158 / 166, H=8 M=32 N=1024 23.1 / 25.9)
        const bool last_rows = D > 128 && TB != 0 && !FROM_DS && m0 + BM > M;
        const int n_lean = (BV != kByElement || TB == 0) && !last_rows ? ks_.lean_steps(n_fast) : 0;
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
    if constexpr (FROM_DS) {
        run(RowsTag<kByChunk>{});
    } else if constexpr (TB == 0) {
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

    // ---- epilogue: dq = dQ * sm_scale (flash_attention.py:644-646) ----
    ks_.drain();  // K/V slots are dead and no copy is in flight: reuse their LDS for the output tile
    if (p.dq_splits > 1) {
        // one of several shares of the keys: into this share's slice of the scratch, in fp32 (the sum
        // rounds once, like an unsplit run), 16 bytes per lane straight from the accumulators
        float* pf = reinterpret_cast<float*>(p.part_dq) + (((int64_t)split * p.B * p.H + bh) * M + my_m) * D;
        if (my_m < M) {
#pragma unroll
            for (int db = 0; db < C::DB; db++) {
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const int d = db * 32 + 8 * q4 + 4 * g;
                    if (d < D) {
                        f32x4 w;
#pragma unroll
                        for (int e = 0; e < 4; e++) w[e] = dq_acc[db][q4 * 4 + e] * p.sm_scale;
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
            for (int e = 0; e < 4; e++) pk[e] = (T)(dq_acc[db][q4 * 4 + e] * p.sm_scale);
            *reinterpret_cast<T4*>(o_lds + r * OS + db * 32 + 8 * q4 + 4 * g) = pk;
        }
    }
    T* op = reinterpret_cast<T*>(p.dq) + (int64_t)b * p.sdq.b + (int64_t)h * p.sdq.h;
    // Nothing formed of the lane here is kept in registers through the loops.  (It was, up to 60 of them, some of those that the
    // loops need: D=256 from dS B=2 H=4 S=1024 22.5 -> 20.8 us, B=2 H=16 S=2048 108 -> 102, no bias B=4 H=4 S=512 32.4 -> 31, from
    // fp32 dS D=32 B=2 H=8 S=1024 17.1 -> 16.3, causal row mask D=64 there 25.3 -> 22.8.  The kernels of a row up to D=32 had them
    // to spare, and there the loop of causal ones lost its order with them: 18 -> 21.)
    int lane_late = lane;
    if constexpr (!(ROWB && D <= 32)) asm volatile("" : "+v"(lane_late));
    lds_wave_order();  // (a wave's own rows: no barrier)
    i32x4 out[WR::COPIES];  // (all reads in flight together)
#pragma unroll
    for (int it = 0; it < WR::COPIES; it++)
        out[it] = lds_read16(o_lds + (it * 64 + lane_late) / CPR * OS + (it * 64 + lane_late) % CPR * 8);
#pragma unroll
    for (int it = 0; it < WR::COPIES; it++) {
        const int row = (it * 64 + lane_late) / CPR, ch = (it * 64 + lane_late) % CPR;
        if (mw + row < M && ch * 8 < p.d_qk) gst16(op + (int64_t)(mw + row) * p.sdq.s + ch * 8, out[it]);
    }
}

// dq = sum of the shares that the work-groups of a split dQ kernel left in part_dq, added in fp32 in
// a fixed order.  One thread per 8 head-dim elements of a row.
template <typename T, int D> __global__ __launch_bounds__(256) void fa_bwd_dq_sum_kernel(const BwdParams p) {
    typedef typename VecOf<T>::v8 T8;
    constexpr int TPR = D / 8;
    const int64_t rows = (int64_t)p.B * p.H * p.M;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = idx / TPR;
    const int c = (int)(idx % TPR);
    if (row >= rows || c * 8 >= p.d_qk) return;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 0; s < p.dq_splits; s++) {
        const float* src = reinterpret_cast<const float*>(p.part_dq) + (s * rows + row) * D + c * 8;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(src), hi = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            acc[e] += lo[e];
            acc[4 + e] += hi[e];
        }
    }
    const int m = (int)(row % p.M);
    const int64_t bh = row / p.M;
    const int b = (int)(bh / p.H), h = (int)(bh % p.H);
    T8 o8;
#pragma unroll
    for (int e = 0; e < 8; e++) o8[e] = (T)acc[e];
    gst16(reinterpret_cast<T*>(p.dq) + (int64_t)b * p.sdq.b + (int64_t)h * p.sdq.h + (int64_t)m * p.sdq.s + c * 8, as_raw(o8));
}


// ---------------------------------------------------------------------------------------------
// The bias of 4 consecutive query rows at one key, as the dK/dV kernel reads it from a row-major
// slice (32 keys per row) in LDS; get(e) is the additive term of row e: natural units for a float
// bias, log2 units (0 or the mask value) for a bool mask.
template <int BIAS> struct BiasQuad;
template <> struct BiasQuad<0> {
    __device__ __forceinline__ void load(const unsigned char*, int, int, int) {}
    __device__ __forceinline__ float get(int) const { return 0.f; }
};
template <> struct BiasQuad<1> {
    unsigned char v[4];
    __device__ __forceinline__ void load(const unsigned char* slice, int row0, int key, int) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = slice[(row0 + e) * 32 + key];
    }
    __device__ __forceinline__ float get(int e) const { return v[e] ? 0.f : kMask; }
};
template <> struct BiasQuad<2> {
    i16x4 raw;  // 4 rows of one key column in one transposing read
    __device__ __forceinline__ void load(const unsigned char* slice, int row0, int, int lane) {
        raw = lds_read_tr4(reinterpret_cast<const _Float16*>(slice) + tr_offset(lane, row0, 0, 32));
    }
    __device__ __forceinline__ float get(int e) const { return (float)__builtin_bit_cast(f16x4, raw)[e]; }
};
template <> struct BiasQuad<3> {
    i16x4 raw;
    __device__ __forceinline__ void load(const unsigned char* slice, int row0, int, int lane) {
        raw = lds_read_tr4(reinterpret_cast<const __bf16*>(slice) + tr_offset(lane, row0, 0, 32));
    }
    __device__ __forceinline__ float get(int e) const { return (float)__builtin_bit_cast(bf16x4, raw)[e]; }
};
template <> struct BiasQuad<5> {  // ALiBi: nothing to read, the kernel computes the term from the indices
    __device__ __forceinline__ void load(const unsigned char*, int, int, int) {}
    __device__ __forceinline__ float get(int) const { return 0.f; }
};
template <> struct BiasQuad<6> : BiasQuad<5> {};  // row-broadcast bias: one value per key, held by the kernel
template <> struct BiasQuad<7> : BiasQuad<5> {};
template <> struct BiasQuad<4> {
    float v[4];
    __device__ __forceinline__ void load(const unsigned char* slice, int row0, int key, int) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = reinterpret_cast<const float*>(slice)[(row0 + e) * 32 + key];
    }
    __device__ __forceinline__ float get(int e) const { return v[e]; }
};

// ---------------------------------------------------------------------------------------------
// W, waves per role: four pairs of waves on a 128-key tile; two on a 64-key tile for head dim 256, where a wave needs the
// whole register file of its SIMD (128 accumulator registers and 64 of the resident operand before anything streams), and for
// few query rows at 128, where two such work-groups share a CU (short_rows below).
constexpr int bwd_waves(int D) { return D > 128 ? 2 : 4; }
// Biases that this kernel takes up to head dim 64, by the rule of pair_of_waves
constexpr bool pair_built(int D, int bias, int dbias) {
    return (D <= 64 && ((bias >= 2 && bias <= 4 && dbias == 1) || (bias == 4 && dbias == 0))) || (D == 64 && bias == 1 && dbias == 0);
}
template <int D, int BIAS, int W = bwd_waves(D)> struct BwdCfg {
    static constexpr int WPR = W;
    static constexpr bool HALF = D <= 128 && W == 2;  // half of a CU's LDS
    static constexpr int BN = 32 * WPR, NT = 128 * WPR;
    static constexpr int LDS_LIMIT = HALF ? 81920 : 163840;
    static constexpr int BMI = 32;                         // rows of a query block
    static constexpr int DB = D < 32 ? 1 : D / 32;
    static constexpr int KSTEPS = D / 16;
    static constexpr int CPR = D / 8;
    static constexpr int DSS = BMI + 4;                    // dS^T tile: elements between two keys
    static constexpr int ES = BIAS == 0 ? 0 : (BIAS == 1 ? 1 : (BIAS == 4 ? 4 : 2));
    static constexpr int EPC = ES > 0 ? 16 / ES : 8;       // bias elements per 16-byte chunk
    static constexpr int BCPR = 2 * ES;                    // 16-byte chunks per 32-key bias row
    static constexpr int BCH = (BMI * BCPR + 63) / 64;     // bias copies per S-wave per block
    static constexpr int Q_BYTES = BMI * D * 2;
    static constexpr int NQD = Q_BYTES / 1024;             // 1 KB copies per Q (or dO) block
    static constexpr int QD = NQD >= WPR ? NQD / WPR : 1;  // of which each wave of a role issues this many
    // Q, dO, LSE, delta and the bias slices reach LDS through direct global -> LDS copies issued
    // LA blocks ahead of their use (Q, LSE and bias by the S-waves, dO and delta by the dP-waves);
    // a copy has LA - 1 whole steps and the rest of its own to land before the barrier that
    // publishes it.
    static constexpr int DS_BYTES = (BIAS == 2 || BIAS == 3) ? BN * DSS * 2 : 0;  // dS^T tiles (dBias)
    // The LSE (delta) values of a block: a copy is 64 lanes wide, so a slot is 64 floats; with 32-row
    // blocks the upper lanes copy the same 32 values again (no lane mask, no branch around the copy).
    static constexpr int STAT_BYTES = 64 * 4;
    static constexpr int P_BYTES = 4 * 64 * 16 * WPR;         // P hand-off: 16 floats per lane
    static constexpr int BT_BYTES = BMI * 32 * ES;         // bias slice of one S-wave
    // LDS bytes with copies la blocks ahead: la + 1 dO buffers and bias slots, la + 2 Q buffers and
    // one more if the dK product of a block is deferred by a step (so that it does not wait for
    // the dS of the same step)
    static constexpr int lds_total(int la, int defer) {
        return (2 * la + 3 + defer) * (Q_BYTES + STAT_BYTES) + DS_BYTES + 2 * P_BYTES + WPR * (la + 1) * BT_BYTES;
    }
    static constexpr int LA = D > 128 ? 1 : HALF ? (lds_total(2, 1) <= LDS_LIMIT ? 2 : 1) : (lds_total(3, 1) <= LDS_LIMIT ? 3 : 2);
    static constexpr bool DEFER_DK = D <= 128 && lds_total(LA, 1) <= LDS_LIMIT;
    static constexpr int NDOB = LA + 1;                    // dO (+delta) buffers
    static constexpr int RING = LA + 1;                    // bias slots per S-wave
    static constexpr int NQB = LA + 2 + (DEFER_DK ? 1 : 0);  // Q (+LSE) buffers
    static constexpr int OFF_DO = NQB * Q_BYTES;
    static constexpr int OFF_DS = OFF_DO + NDOB * Q_BYTES;
    static constexpr int OFF_P = OFF_DS + DS_BYTES;        // two hand-off buffers
    static constexpr int OFF_LSE = OFF_P + 2 * P_BYTES;
    static constexpr int OFF_DELTA = OFF_LSE + NQB * STAT_BYTES;
    static constexpr int OFF_BIAS = OFF_DELTA + NDOB * STAT_BYTES;
    static constexpr int LOOP_BYTES = OFF_BIAS + WPR * RING * BT_BYTES;
    static constexpr int LDS_BYTES = LOOP_BYTES;
    static_assert(LDS_BYTES <= LDS_LIMIT, "LDS budget of the configuration");
    static constexpr int WAVES_PER_SIMD = D > 128 ? 1 : 2;
};

// Work split inside a work-group of 8 waves.  Waves 0-3 ("S-waves") and waves 4-7 ("dP-waves")
// pair up on the four 32-key blocks of the tile (waves w and w + 4 run on the same SIMD; for head
// dim 256 a work-group is two such pairs on a 64-key tile, one wave per SIMD):
//   S-wave : S = Q K^T, P = 2^(S*scale + bias - LSE)  -> hands P to its partner through LDS,
//            dV^T += dO^T P, and the global -> LDS copies of the Q / LSE / bias blocks
//   dP-wave: dP = dO V^T, dS = P (dP - delta) (+ dBias through an LDS tile), dK^T += Q^T dS,
//            and the global -> LDS copies of the dO / delta blocks
// The roles are skewed by one query block so that a step needs a single barrier and nothing a
// wave does inside a step depends on what its partner does in the same step:
//   step t : S-wave : P(t+1) from Q(t+1), then dV += dO(t)^T P(t)        (P(t) kept in registers)
//            dP-wave: dS(t) from dO(t) and the P(t) handed over in step t-1, dK += Q(t-1)^T dS(t-1)
// While one wave of a SIMD runs exponentials or products the other issues MFMAs.
// DBIAS: 0 = the bias is not trainable; 1 = dBias is written densely, (B, H, M, N) in the bias dtype
// (flash_attention.py:307-308); 2 = reduced in the kernel: for a float bias the sums of dS over the
// query rows, one fp32 per (batch, head, key), for ALiBi the gradient of the slope, one fp32 per
// (batch, head, key tile, wave); a second small kernel sums those over the broadcast dimensions.
template <typename T, int D, int BIAS, bool CAUSAL, int DBIAS, int W>
__global__ __launch_bounds__((BwdCfg<D, tile_kind(BIAS), W>::NT), (BwdCfg<D, tile_kind(BIAS), W>::WAVES_PER_SIMD)) void fa_bwd_kernel(const BwdParams p) {
    constexpr int TB = tile_kind(BIAS);  // kind of bias tile that is streamed (none for ALiBi)
    static_assert(D > 96 || pair_built(D, BIAS, DBIAS), "fa_bwd_narrow.hip");
    typedef BwdCfg<D, TB, W> C;
    typedef Swz<D> SW;
    typedef typename VecOf<T>::v8 T8;
    typedef typename VecOf<T>::v4 T4;
    typedef typename BiasElem<tile_kind(BIAS)>::type E;
    constexpr int BN = C::BN, BMI = C::BMI, CPR = C::CPR, DSS = C::DSS;
    // dBias leaves through the dS tile (16-byte row stores) when it has the element type of dS
    constexpr bool DB_VIA_LDS = DBIAS == 1 && ((BIAS == 2 && __is_same(T, _Float16)) || (BIAS == 3 && __is_same(T, __bf16)));
    // an fp32 dBias leaves through LDS too, as fp32: the dP-wave turns its part of the P hand-off buffer,
    // which it has just read and which is not written again before the next step, into a row-major
    // 32 x 32 tile (4-byte stores, one per element) and stores 16 bytes per lane from there
    constexpr bool DB_VIA_LDS32 = DBIAS == 1 && BIAS == 4;

    __shared__ __align__(1024) unsigned char smem[C::LDS_BYTES];

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int r = lane & 31, g = lane >> 5;
    const bool s_wave = wave < C::WPR;  // role
    const int kb = __builtin_amdgcn_readfirstlane(wave % C::WPR);  // 32-key block of this wave (scalar)
    const unsigned lds_base = lds_addr_of(smem);

    int nt, bh;
    decode_block<CAUSAL>(blockIdx.x, p.n_ntiles, p.B * p.H, nt, bh);
    const int b = bh / p.H, h = bh % p.H;
    const int M = p.M, N = p.N;
    const int n0 = nt * BN;
    const int nw = n0 + kb * 32;
    const int my_n = nw + r;

    const T* qp = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.sq.b + (int64_t)h * p.sq.h;
    const T* kp = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.sk.b + (int64_t)h * p.sk.h;
    const T* vp = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.sv.b + (int64_t)h * p.sv.h;
    const T* dop = reinterpret_cast<const T*>(p.dout) + (int64_t)b * p.sdo.b + (int64_t)h * p.sdo.h;
    const float* lsep = p.lse + ((int64_t)b * p.H + h) * M;
    const float* deltap = p.delta + ((int64_t)b * p.H + h) * M;
    const E* bp = nullptr;
    E* dbp = nullptr;
    if (TB != 0) bp = reinterpret_cast<const E*>(p.bias) + (int64_t)b * p.sbias.b + (int64_t)h * p.sbias.h;
    if (DBIAS == 1) dbp = reinterpret_cast<E*>(p.dbias) + (int64_t)b * p.sdbias.b + (int64_t)h * p.sdbias.h;
    float neg_slope = 0.f, ratio = 0.f;  // ALiBi: slope of this head, key positions per query row
    if (BIAS == 5) {
        neg_slope = -reinterpret_cast<const float*>(p.bias)[h];
        ratio = (float)p.N / (float)p.M;
    }
    const float log2_slope = neg_slope * kLog2e;
    // row-broadcast bias: the term of this lane's key, natural units (6) or 0 / mask value in log2 units (7)
    float row_bv = 0.f;
    if (BIAS == 6 || BIAS == 7) {
        if (my_n < N) {
            const int64_t idx = (int64_t)b * p.sbias.b + (int64_t)h * p.sbias.h + (int64_t)my_n * p.sbias.n;
            switch (p.row_bias_kind) {
                case 1: row_bv = reinterpret_cast<const unsigned char*>(p.bias)[idx] ? 0.f : kMask; break;
                case 2: row_bv = (float)reinterpret_cast<const _Float16*>(p.bias)[idx]; break;
                case 3: row_bv = (float)reinterpret_cast<const __bf16*>(p.bias)[idx]; break;
                default: row_bv = reinterpret_cast<const float*>(p.bias)[idx]; break;
            }
        }
    }
    constexpr bool NATURAL = BIAS >= 2 && BIAS != 7;  // the bias term is in natural units (else log2 units)
    unsigned char* ring_lds = smem + C::OFF_BIAS + kb * C::RING * C::BT_BYTES;
    float* p_lds = reinterpret_cast<float*>(smem + C::OFF_P) + kb * 64 * 16;  // + buffer * P_BYTES / 4

    // ---- this wave's 32 keys as B operand (column my_n, k = d): K for an S-wave, V for a dP-wave.  Up to head dim 128 they come
    // through LDS with the first copies (WaveRows): K through the hand-off buffers, V through the Q and dO slots that those
    // copies leave free.  A tile spent 14 000 clocks before its first step and 6 000 after its last one, a quarter of it at 1024
    // rows.  With this and the way back at the end, us, before -> after, D = 128: B=8 H=12 S=512 44.9 -> 38.5, with dBias 63.5 ->
    // 58, S=1024 causal with a byte mask 95.6 -> 87.6, H=32 M=1024 N=8192 with dBias 552 -> 528, M=N=4096 843 -> 833; the way
    // back alone, D = 256 B=4 H=8 S=1024 104.5 -> 99.4. ----
    typedef WaveRows<T, D> WR;
    constexpr bool STAGED = D <= 128;
    T8 opreg[C::KSTEPS];
    if constexpr (!STAGED) {
        const T* src = s_wave ? kp + (int64_t)my_n * p.sk.s : vp + (int64_t)my_n * p.sv.s;
#pragma unroll
        for (int ks = 0; ks < C::KSTEPS; ks++) {
            i32x4 v = {0, 0, 0, 0};
            if (my_n < N && ks * 16 + 8 * g < (s_wave ? p.d_qk : p.d_v)) v = gld16(src + ks * 16 + 8 * g);
            opreg[ks] = as_vec<T8>(v);
        }
    }

    // dV^T (S-wave) or dK^T (dP-wave) of this wave's 32 keys: rows = head dim, columns = keys
    f32x16 acc[C::DB];
#pragma unroll
    for (int db = 0; db < C::DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[db][i] = 0.f;

    const float qk_scale = p.sm_scale * kLog2e;
    const int n_mblocks = (M + BMI - 1) / BMI;
    // causal: query blocks that end above the first key of this tile see none of its keys
    const int mb_first = CAUSAL ? (n0 / BMI) : 0;
    constexpr bool BY_DWORD = BIAS == 4 && D <= 64;
    const bool bias_vec = TB != 0 && p.bias_vec;
    const bool dbias_vec = DBIAS == 1 && p.dbias_vec;

    // blocks skipped by the causal schedule still owe zeros to dBias
    if (DBIAS == 1 && CAUSAL && !s_wave) {
        const int rows_skipped = mb_first * BMI < M ? mb_first * BMI : M;
        for (int c = lane; c < rows_skipped * C::BCPR; c += 64) {
            const int m = c / C::BCPR, nn = nw + (c % C::BCPR) * C::EPC;
            E* dst = dbp + (int64_t)m * p.sdbias.m + (int64_t)nn * p.sdbias.n;
            if (dbias_vec && nn + C::EPC <= N) {
                i32x4 z = {0, 0, 0, 0};
                gst16(dst, z);
            } else {
                for (int e = 0; e < C::EPC; e++)
                    if (nn + e < N) dst[(int64_t)e * p.sdbias.n] = (E)0.f;
            }
        }
    }

    // ---- global -> LDS copies of Q (+LSE), dO (+delta) and bias blocks ----
    // A block is NQD copies of 1 KB; copy ci fills bytes [1024 ci, 1024 ci + 1024) of the swizzled
    // tile, so lane l of it fetches the 16-byte chunk that lives at tile position 64 ci + l.  Each
    // wave of the issuing role issues QD of them (more than once where a block has fewer than four), every step the
    // same number: completion is counted (s_waitcnt vmcnt) and copies complete in issue order.
    // Rows past M re-read the last row: their P and dS are exactly zero.
    unsigned cq_off[C::QD], cdo_off[C::QD];
    int c_idx[C::QD];
#pragma unroll
    for (int i = 0; i < C::QD; i++) {
        c_idx[i] = (kb * C::QD + i) % C::NQD;
        const int c = c_idx[i] * 64 + lane;
        const int row = c / CPR, src = (c % CPR) ^ SW::f(row);
        cq_off[i] = (unsigned)(row * (int)p.sq.s * 2 + live_chunk(src, p.d_qk / 8) * 16);
        cdo_off[i] = (unsigned)(row * (int)p.sdo.s * 2 + live_chunk(src, p.d_v / 8) * 16);
    }
    auto issue_rows = [&](const T* base, int64_t row_stride, int chunks, const unsigned (&off)[C::QD], int mb, unsigned dst) {
        // a block past the end is the last row over and over: offsets never go negative
        const int m0 = mb * BMI < M ? mb * BMI : M - 1;
        const uint64_t blk = uniform_ptr(base + (int64_t)m0 * row_stride);
        const bool full = m0 + BMI <= M;
#pragma unroll
        for (int i = 0; i < C::QD; i++) {
            unsigned o = off[i];
            if (!full) {
                // (rare: the lane index passes through an empty asm so that these per-lane values are
                // formed here and not kept in registers across the loops)
                int lane_here = lane;
                asm volatile("" : "+v"(lane_here));
                const int c = c_idx[i] * 64 + lane_here;
                int row = c / CPR;
                const int src = (c % CPR) ^ SW::f(row);
                row = row < M - m0 ? row : M - 1 - m0;
                o = (unsigned)(row * (int)row_stride * 2 + live_chunk(src, chunks) * 16);
            }
            lds_copy16(blk, o, dst + c_idx[i] * 1024);
        }
    };
    // one float per row
    auto issue_stat = [&](const float* src, int mb, unsigned dst) {
        int m = mb * BMI + lane % BMI;
        m = m < M ? m : M - 1;
        lds_copy4(uniform_ptr(src), (unsigned)m * 4u, dst);
    };
    // bias slice (BMI rows x 32 keys) of query block mb -> ring slot.  Chunk c = 64 it + lane of the
    // slice (row c / BCPR, 16-byte chunk c % BCPR) lands at byte 16 c of the slot, i.e. the slot
    // is the row-major slice.  Rows past M re-read row M - 1 (masked where they are used) and chunks that start past N
    // re-read column 0 (a lane is a key: what such a lane forms is not stored).
    auto issue_bias = [&](int mb, auto bv_tag) {
        if constexpr (TB != 0) {
            const unsigned dst = lds_base + C::OFF_BIAS + (kb * C::RING + (mb - mb_first) % C::RING) * C::BT_BYTES;
            const uint64_t base = uniform_ptr(bp);
            if constexpr (decltype(bv_tag)::value == kByDword) {
#pragma unroll
                for (int it = 0; it < 16; it++) {
                    int m = mb * BMI + 2 * it + g;
                    m = m < M ? m : M - 1;
                    lds_copy4(base, (unsigned)(((int64_t)m * p.sbias.m + (my_n < N ? my_n : N - 1)) * 4), dst + it * 256);
                }
                return;
            }
#pragma unroll
            for (int it = 0; it < C::BCH; it++) {
                const int c = it * 64 + lane;
                int m = mb * BMI + c / C::BCPR;
                int nn = nw + (c % C::BCPR) * C::EPC;
                m = m < M ? m : M - 1;
                nn = nn < N ? nn : 0;
                // a (batch, head) slice that takes this path is smaller than 2 GiB
                lds_copy16(base, (unsigned)(((int64_t)m * p.sbias.m + nn) * C::ES), dst + it * 1024);
            }
        }
    };
    // block mb of Q with its LSE (QD + 1 copies) / block mb of dO with its delta (QD + 1 copies);
    // all four waves of a role copy the 32 or 64 floats, which keeps their counts alike
    auto issue_q = [&](int mb) {
        issue_rows(qp, p.sq.s, p.d_qk / 8, cq_off, mb, lds_base + (mb % C::NQB) * C::Q_BYTES);
        issue_stat(lsep, mb, lds_base + C::OFF_LSE + (mb % C::NQB) * C::STAT_BYTES);
    };
    auto issue_do = [&](int mb) {
        issue_rows(dop, p.sdo.s, p.d_v / 8, cdo_off, mb, lds_base + C::OFF_DO + (mb % C::NDOB) * C::Q_BYTES);
        issue_stat(deltap, mb, lds_base + C::OFF_DELTA + (mb % C::NDOB) * C::STAT_BYTES);
    };
    // Issuing a copy stalls the wave while the memory pipeline of the CU is backed up, so the
    // copies are dealt out between the roles: Q and the bias go with the S-waves, dO with the
    // dP-waves.
    constexpr bool Q_BY_S = true, DO_BY_S = false;
    static_assert(Q_BY_S && !DO_BY_S, "the running pointers of the interior steps are laid out for this deal");
    // Interior steps (every block they touch is whole, in range and unmasked: all but the first and
    // the last few of a tile) walk the query blocks in order, so their copies keep running block
    // pointers in scalar registers, one 64-bit add per block, and need no clamps; run_start() points
    // them at the first blocks an interior loop issues.
    const int n_full = M / BMI;  // blocks whose rows all exist
    uint64_t run_rows = 0, run_stat = 0, run_bias = 0;  // Q and LSE (role that issues Q) or dO and delta; bias slices
    unsigned bias_off0 = 0;  // this lane's byte offset in the first bias copy of a block, from the block's first row
    if constexpr (TB != 0) {
        int nn = nw + (lane % C::BCPR) * C::EPC;
        nn = nn < N ? nn : 0;
        bias_off0 = (unsigned)(((int64_t)(lane / C::BCPR) * p.sbias.m + nn) * C::ES);
        if (BY_DWORD && p.bias_vec == kByDword) bias_off0 = (unsigned)(((int64_t)g * p.sbias.m + (my_n < N ? my_n : N - 1)) * 4);
    }
    auto run_start = [&](const T* rows, int64_t row_stride, const float* stat, int mb, int mb_bias) {
        run_rows = uniform_ptr(rows + (int64_t)mb * BMI * row_stride);
        run_stat = uniform_ptr(stat + (int64_t)mb * BMI);
        if constexpr (TB != 0) run_bias = uniform_ptr(bp + (int64_t)mb_bias * BMI * p.sbias.m);
    };
    // the next block of Q (or dO) with its LSE (or delta): QD + 1 copies, like issue_q / issue_do
    // (the caller has passed the running pointers through settle_ptrs() since they were last advanced)
    auto issue_next_rows = [&](int64_t row_stride, const unsigned (&off)[C::QD], unsigned dst, unsigned stat_dst) {
#pragma unroll
        for (int i = 0; i < C::QD; i++) lds_copy16(run_rows, off[i], dst + c_idx[i] * 1024);
        run_rows += (uint64_t)(BMI * 2) * (uint64_t)row_stride;
        // (the lane index passes through an empty asm so that the offset is formed here, two
        // instructions, and does not hold a register across the loop)
        unsigned lane_here = (unsigned)lane;
        asm volatile("" : "+v"(lane_here));
        lds_copy4(run_stat, (lane_here % BMI) * 4u, stat_dst);
        run_stat += BMI * 4;
    };
    auto issue_next_q = [&](int mb) {
        const unsigned slot = (unsigned)mb % C::NQB;
        issue_next_rows(p.sq.s, cq_off, lds_base + slot * C::Q_BYTES, lds_base + C::OFF_LSE + slot * C::STAT_BYTES);
    };
    auto issue_next_do = [&](int mb) {
        const unsigned slot = (unsigned)mb % C::NDOB;
        issue_next_rows(p.sdo.s, cdo_off, lds_base + C::OFF_DO + slot * C::Q_BYTES, lds_base + C::OFF_DELTA + slot * C::STAT_BYTES);
    };
    auto issue_next_bias = [&](int mb, auto bv_tag) {
        if constexpr (TB != 0) {
            constexpr int N_COPIES = decltype(bv_tag)::value == kByDword ? 16 : C::BCH;
            const unsigned dst = lds_base + C::OFF_BIAS + (kb * C::RING + (unsigned)(mb - mb_first) % C::RING) * C::BT_BYTES;
            const unsigned rows_step = (unsigned)(BMI / N_COPIES * (int)p.sbias.m * C::ES);  // the rows one copy covers
#pragma unroll
            for (int it = 0; it < N_COPIES; it++) {
                if constexpr (N_COPIES == C::BCH) lds_copy16(run_bias, bias_off0 + it * rows_step, dst + it * 1024);
                else lds_copy4(run_bias, bias_off0 + it * rows_step, dst + it * 256);
            }
            run_bias += (uint64_t)(BMI * C::ES) * (uint64_t)p.sbias.m;
        }
    };
    // per-element path for bias rows that cannot be copied in aligned 16-byte chunks
    auto load_bias_scalar = [&](int mb, unsigned char* dst) {
        if constexpr (TB != 0) {
            // all loads of the block in flight together (clamped addresses instead of
            // branches; what lies outside the bias is masked where it is used)
            const int m0 = mb * BMI;
            const int nn = my_n < N ? my_n : N - 1;
            E vals[16];
#pragma unroll
            for (int j = 0; j < 16; j++) {
                int m = m0 + 2 * j + g;
                m = m < M ? m : M - 1;
                vals[j] = bp[(int64_t)m * p.sbias.m + (int64_t)nn * p.sbias.n];
            }
#pragma unroll
            for (int j = 0; j < 16; j++) reinterpret_cast<E*>(dst)[(2 * j + g) * 32 + r] = vals[j];
        }
    };

    // ---- prologue: this wave's keys, the first LA blocks of Q and LA - 1 blocks of dO ----
    unsigned op_tile = 0;
    if constexpr (STAGED) {
        constexpr int FREE_Q = C::NQB - C::LA;  // Q slots without a block yet, and two of dO
        static_assert(2 * C::P_BYTES >= C::WPR * WR::BYTES && FREE_Q + 2 >= C::WPR && C::Q_BYTES == WR::BYTES, "room for the keys");
        if (s_wave) op_tile = lds_base + C::OFF_P + (unsigned)kb * WR::BYTES;
        else if (kb < FREE_Q) op_tile = lds_base + (unsigned)((mb_first + C::LA + kb) % C::NQB) * C::Q_BYTES;
        else op_tile = lds_base + C::OFF_DO + (unsigned)((mb_first + C::LA - 1 + kb - FREE_Q) % C::NDOB) * C::Q_BYTES;
        op_tile = __builtin_amdgcn_readfirstlane(op_tile);
    }
    {
        const unsigned saved_m0 = lds_copy_begin();
        if constexpr (STAGED) {
            const int chunks = (s_wave ? p.d_qk : p.d_v) / 8;
            WR::issue(s_wave ? kp : vp, s_wave ? p.sk.s : p.sv.s, nw, N, op_tile, lane, [&](int c) { return live_chunk(c, chunks); });
        }
#pragma unroll 1
        for (int i = 0; i < C::LA; i++) {
            if (s_wave == Q_BY_S) issue_q(mb_first + i);
            if constexpr (BY_DWORD) {
                if (s_wave && p.bias_vec == kByDword) issue_bias(mb_first + i, RowsTag<kByDword>{});
                else if (s_wave && bias_vec) issue_bias(mb_first + i, RowsTag<kByChunk>{});
            } else {
                if (s_wave && TB != 0 && bias_vec) issue_bias(mb_first + i, RowsTag<kByChunk>{});
            }
            if (s_wave == DO_BY_S && i < C::LA - 1) issue_do(mb_first + i);
        }
        lds_copy_end(saved_m0);
    }
    WR::template arrived<0>();
    if constexpr (STAGED) {  // (of a key past the end, the last one again: nothing of such a lane is stored)
#pragma unroll
        for (int ks = 0; ks < C::KSTEPS; ks++) {
            const i32x4 x = as_raw(SW::template row8_at<T8>(op_tile + SW::rows_lane(lane), 0, ks));
            opreg[ks] = as_vec<T8>(ks * 16 + 8 * g < (s_wave ? p.d_qk : p.d_v) ? x : i32x4{0, 0, 0, 0});
        }
    }
    __syncthreads();

    T8 op_cur[2];  // P^T (S-wave) or dS^T (dP-wave) of the block whose accumulation is still due
#pragma unroll
    for (int kk = 0; kk < 2; kk++) op_cur[kk] = as_vec<T8>(i32x4{0, 0, 0, 0});

    // A wave issues its instructions in order and only two waves share a SIMD, so every LDS round
    // trip that sits between two dependent pieces of a step is dead time.  A step therefore
    // fetches what it needs from LDS into registers at its top (PRELOAD): the A operands of both
    // products and the inputs of the element-wise work, each ahead of work that hides the trip.
    // With D = 256 there is no register room for that and the compiler places the reads.
    constexpr bool PRELOAD = D <= 128;
    constexpr int NR = C::KSTEPS;  // A operands of a row product: 32 rows x 16 of the head dim each
    constexpr int NA = 2 * C::DB;  // A operands of a column product: 32 of the head dim x 16 rows each
    // tiles are named by their LDS byte address (scalar); the two per-lane address constants of
    // Swz cover every operand read of the loop
    const unsigned rows_l = SW::rows_lane(lane), cols_l = SW::cols_lane(lane);
    auto load_rows = [&](unsigned tile, T8 (&a)[NR]) {
        const unsigned base = tile + rows_l;
#pragma unroll
        for (int ks = 0; ks < C::KSTEPS; ks++) a[ks] = SW::template row8_at<T8>(base, 0, ks);
    };
    // sacc = rows(tile) x opreg: S = Q K^T (S-wave) or dP = dO V^T (dP-wave)
    auto mma_rows = [&](const T8 (&a)[NR], f32x16& sacc) {
#pragma unroll
        for (int i = 0; i < 16; i++) sacc[i] = 0.f;
#pragma unroll
        for (int ks = 0; ks < C::KSTEPS; ks++) sacc = mfma32(a[ks], opreg[ks], sacc);
    };
    // the A operands of acc^T += tile^T op are columns of the tile, gathered with ds_read_b64_tr_b16
    auto load_cols = [&](unsigned tile, T8 (&a)[NA]) {
        const unsigned base = tile + cols_l;
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
#pragma unroll
            for (int db = 0; db < C::DB; db++) a[kk * C::DB + db] = SW::template col8_at<T8>(base, kk * 16, db);
    };
    // acc^T += tile^T op: dV^T += dO^T P (S-wave) or dK^T += Q^T dS (dP-wave)
    auto mma_cols = [&](const T8 (&a)[NA], const T8 (&op)[2]) {
#pragma unroll
        for (int kk = 0; kk < 2; kk++)
#pragma unroll
            for (int db = 0; db < C::DB; db++) acc[db] = mfma32(a[kk * C::DB + db], op[kk], acc[db]);
    };
    // ring slots of a block index that may run one or two blocks below zero at the first steps
    auto q_tile = [&](int mb) { return lds_base + (unsigned)(((mb < 0 ? 0 : mb) % C::NQB) * C::Q_BYTES); };
    auto do_tile = [&](int mb) { return lds_base + (unsigned)(C::OFF_DO + ((mb < 0 ? 0 : mb) % C::NDOB) * C::Q_BYTES); };
    // the same for the interior steps, whose block indices are never negative
    auto q_tile_in = [&](int mb) { return lds_base + ((unsigned)mb % C::NQB) * C::Q_BYTES; };
    auto do_tile_in = [&](int mb) { return lds_base + C::OFF_DO + ((unsigned)mb % C::NDOB) * C::Q_BYTES; };

    if (s_wave) {
        // ================================ S-wave ================================
        auto s_loop = [&](auto bv_tag) {
        constexpr int BV = decltype(bv_tag)::value;                    // bias slices come by copy
        constexpr int BIAS_COPIES = BV == kByElement ? 0 : BV == kByDword ? 16 : C::BCH;
        constexpr int OPS = BIAS_COPIES + ((Q_BY_S ? 1 : 0) + (DO_BY_S ? 1 : 0)) * (C::QD + 1);  // copies per step
        // S_AHEAD: the scores of a block are formed at the END of the step before the one that turns
        // them into P, so that a step of this role opens with vector work (exponentials) while the
        // partner wave on the same SIMD opens with matrix products, and closes with matrix products
        // while the partner does its vector work.  It needs the Q block one step earlier, i.e. a copy
        // look-ahead of at least three blocks.  Measured: 3 % on the kernel that writes dBias (whose
        // dP-wave has the most vector work), a loss of 5 % with a bias that is only read and of 4 %
        // without one, which keep the plain order.
        constexpr bool S_AHEAD = TB != 0 && C::LA >= 3 && DBIAS == 1;
        f32x16 sacc;
        if constexpr (S_AHEAD) {
            T8 a_rows[NR];
            load_rows(q_tile(mb_first), a_rows);
            mma_rows(a_rows, sacc);
        }
        auto s_step = [&](int t, auto in_tag) {
            // IN: an interior step: blocks t .. t + 2 + LA are whole and in range, block t + 1 needs no mask
            constexpr bool IN = decltype(in_tag)::value;
            const int nb = t + 1;  // the block whose P is produced in this step
            T8 op_next[2];
            // Copies for the steps to come (their buffers were last read one step ago).  With a bias
            // they are issued behind the LDS reads of the step, whose round trip they cover; without
            // one right after the barrier: measured, each way is a few per cent better in its case.
            auto issue_copies = [&]() {
                const unsigned saved_m0 = lds_copy_begin();
                if constexpr (IN) {
                    settle_ptrs(run_rows, run_stat, run_bias);
                    if constexpr (Q_BY_S) issue_next_q(nb + C::LA);
                    if constexpr (BV != kByElement) issue_next_bias(nb + C::LA, bv_tag);
                    if constexpr (DO_BY_S) issue_next_do(t + C::LA);
                } else {
                    if constexpr (Q_BY_S) issue_q(nb + C::LA);
                    if constexpr (BV != kByElement) issue_bias(nb + C::LA, bv_tag);
                    if constexpr (DO_BY_S) issue_do(t + C::LA);
                }
                lds_copy_end(saved_m0);
            };
            const unsigned char* bt_lds = ring_lds + ((nb - mb_first) % C::RING) * C::BT_BYTES;
            const float* lse_lds = reinterpret_cast<const float*>(smem + C::OFF_LSE) + (IN ? (unsigned)nb % C::NQB : nb % C::NQB) * (C::STAT_BYTES / 4);
            // inputs of P: LSE of 4 consecutive rows and the bias of those rows at this lane's key
            f32x4 lse_in[4];
            BiasQuad<BIAS> bias_in[4];
            auto load_p_inputs = [&]() {
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const int ml0 = 8 * q4 + 4 * g;  // first of 4 consecutive rows
                    lse_in[q4] = *reinterpret_cast<const f32x4*>(lse_lds + ml0);
                    bias_in[q4].load(bt_lds, ml0, r, lane);
                }
            };
            // ---- P (flash_attention.py:281-294) of block nb from its scores; register i
            // is row m0 + 8 (i/4) + 4 g + i%4, the lane is key my_n.  Blocks that touch the
            // last rows or the causal diagonal follow the reference's additive -1e6 arithmetic term
            // by term, and rows past M have none; interior blocks fold everything into one exponent. ----
            auto make_p = [&](auto&& after_pair) {
                const int m0 = nb * BMI;
                // (keys past N need no mask: the lane is the key, and nothing of such a lane is stored.  A ragged
                // last tile so runs interior steps like any other: B=1 H=16 M=N=6001 D=128 0.607 -> 0.540 ms)
                const bool need_mask = !IN && ((m0 + BMI > M) || (CAUSAL && m0 < n0 + BN - 1));
                const float mf0 = (float)(m0 + 4 * g);  // ALiBi: first row of this lane's registers, as a float,
                const float dist0 = __builtin_fmaf(mf0, ratio, -(float)my_n);  // and its distance to the lane's key
                float* p_out = p_lds + (nb & 1) * (C::P_BYTES / 4);
                auto p_step = [&](auto masked_tag) {
                    constexpr bool MASKED = decltype(masked_tag)::value;
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) {
                        const int ml0 = 8 * q4 + 4 * g;
                        const f32x4 lse4 = lse_in[q4];
                        f32x4 p4;
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const int i = q4 * 4 + e;
                            // bool mask: the additive term in log2 units; float bias: natural units
                            float bv = bias_in[q4].get(e);
                            if constexpr (BIAS == 5) bv = alibi_bias(neg_slope, ratio, mf0 + (float)(ml0 - 4 * g + e), (float)my_n);
                            if constexpr (BIAS == 6 || BIAS == 7) bv = row_bv;
                            float pv;
                            if constexpr (MASKED) {
                                const int m = m0 + ml0 + e;
                                const float tmask = CAUSAL && m < my_n ? kMask : 0.f;
                                const float add = NATURAL ? __fmul_rn(bv, kLog2e) : bv;
                                // (no row, no weight.  Not an additive term: the LSE read again may lie below any; and selected here, not
                                // behind the exponential, which took 2 to 3 % where dBias leaves element by element)
                                const float lse = m < M ? lse4[e] : __builtin_inff();
                                pv = fast_exp2(__fadd_rn(__fmul_rn(sacc[i], qk_scale), __fadd_rn(tmask, add)) - lse);
                            } else {
                                // (without a bias the offset is the negated LSE itself: written as 0 - lse it
                                // would cost a subtraction per element, +0 - x not being -x)
                                const float off = BIAS == 0   ? -lse4[e]
                                                  : BIAS == 5 ? __builtin_fmaf(__builtin_fabsf(__builtin_fmaf((float)(8 * q4 + e), ratio, dist0)), log2_slope, -lse4[e])
                                                              : (NATURAL ? __builtin_fmaf(bv, kLog2e, -lse4[e]) : bv - lse4[e]);
                                pv = fast_exp2(__builtin_fmaf(sacc[i], qk_scale, off));
                            }
                            p4[e] = pv;
                            op_next[i >> 3][i & 7] = (T)pv;
                            if (e & 1) after_pair(i >> 1);
                        }
                        // hand P to the dP-wave of the same keys: same lane, same register order
                        *reinterpret_cast<f32x4*>(p_out + (q4 * 64 + lane) * 4) = p4;
                    }
                };
                if constexpr (IN) {
                    p_step(std::false_type{});
                } else {
                    if (need_mask) p_step(std::true_type{});
                    else p_step(std::false_type{});
                }
            };
            if constexpr (TB != 0 && BV == kByElement) {
                if (nb < n_mblocks) load_bias_scalar(nb, ring_lds + ((nb - mb_first) % C::RING) * C::BT_BYTES);
            }
            if constexpr (S_AHEAD) {
                // vector work first: P(nb) from the scores formed at the end of the last step
                T8 a_cols[NA], a_rows[NR];
                if constexpr (PRELOAD) {
                    load_p_inputs();
                    __builtin_amdgcn_sched_barrier(0);
                }
                issue_copies();  // behind the reads, whose round trip they cover
                if constexpr (!PRELOAD) load_p_inputs();
                if (IN || nb < n_mblocks) make_p([](int) {});
                if constexpr (PRELOAD) __builtin_amdgcn_sched_barrier(0);
                load_cols((IN ? do_tile_in(t) : do_tile(t)), a_cols);
                load_rows((IN ? q_tile_in(nb + 1) : q_tile(nb + 1)), a_rows);  // lands while the first product runs
                if constexpr (PRELOAD) __builtin_amdgcn_sched_barrier(0);
                // dV^T += dO(t)^T P(t), then the scores of block nb + 1 for the next step
                if (IN || (t >= mb_first && t < n_mblocks)) mma_cols(a_cols, op_cur);
                if (IN || nb + 1 < n_mblocks) mma_rows(a_rows, sacc);
            } else {
                T8 a_cols[NA], a_rows[NR];
                if constexpr (TB == 0) issue_copies();
                load_cols((IN ? do_tile_in(t) : do_tile(t)), a_cols);
                load_rows((IN ? q_tile_in(nb) : q_tile(nb)), a_rows);
                if constexpr (PRELOAD) {
                    load_p_inputs();
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (TB != 0) issue_copies();
                // Interior steps: the scores first, then the dV product (its operands do not depend on this
                // step) one MFMA at a time between the exponentials of two score elements, so that the wave
                // has vector work to issue while its matrix instructions execute (measured 2-3 % on the
                // kernels of head dim 128 without a bias and with a bias that is only read; the same interleaving of
                // the dK product into the dS arithmetic of the dP-wave costs 1-4 %).
                constexpr bool FUSE = IN && D == 128;
                if constexpr (FUSE) {
                    mma_rows(a_rows, sacc);
                    __builtin_amdgcn_sched_barrier(0);
                    make_p([&](int j) {
                        __builtin_amdgcn_sched_barrier(0);
                        acc[j % C::DB] = mfma32(a_cols[j], op_cur[j / C::DB], acc[j % C::DB]);
                        __builtin_amdgcn_sched_barrier(0);
                    });
                } else {
                // dV^T += dO(t)^T P(t) first: its operands do not depend on this step
                if (IN || (t >= mb_first && t < n_mblocks)) mma_cols(a_cols, op_cur);
                if (IN || nb < n_mblocks) {
                    mma_rows(a_rows, sacc);
                    if constexpr (!PRELOAD) load_p_inputs();
                    make_p([](int) {});
                }
                }
            }
#pragma unroll
            for (int kk = 0; kk < 2; kk++) op_cur[kk] = op_next[kk];
            // The barrier publishes the copies that the next step reads.  Copies complete in issue
            // order (Q rows, then the bias slice of the same step).  S_AHEAD: the next step reads the
            // Q rows issued one step ago, so only the bias slice issued behind them and this step's
            // copies may still be in flight; else everything but the last LA - 1 steps has landed.
            // Without a bias the compiler is kept from moving work of the step across its closing
            // barrier (it sinks matrix instructions below it where it can): measured 3 % faster at head
            // dim 128 without a bias, slower or equal everywhere else, so only there.
            if constexpr (BIAS == 0 && D == 128) __builtin_amdgcn_sched_barrier(0);
            if constexpr (S_AHEAD) wait_vmcnt<BIAS_COPIES + OPS*(C::LA - 2)>();
            else wait_vmcnt<OPS*(C::LA - 1)>();
            lds_barrier();
        };
        // interior steps: t >= mb_first (block t is accumulated), the copied blocks up to t + 1 + LA are
        // whole, and block t + 1 lies below the causal diagonal of every key of the tile
        // Both roles run steps mb_first - 1 .. n_mblocks, whatever part of them is interior.
        const int t_end = n_mblocks + 1;
        int t_in = mb_first, t_out = n_full - C::LA - 1;
        if (CAUSAL) t_in = (n0 + BN - 1 + BMI - 1) / BMI - 1 > t_in ? (n0 + BN - 1 + BMI - 1) / BMI - 1 : t_in;
        if (TB != 0 && BV == kByElement) t_out = t_in;  // bias element by element: no interior
        t_in = t_in < t_end ? t_in : t_end;
        t_out = t_out < t_in ? t_in : (t_out < t_end ? t_out : t_end);
        // (two passes over ONE copy of the general loop, the interior loop between them)
        int t = mb_first - 1, stop = t_in;
#pragma unroll 1
        for (int pass = 0; pass < 2; pass++) {
#pragma unroll 1
            for (; t < stop; t++) s_step(t, std::false_type{});
            if (pass == 0 && t_in < t_out) {
                run_start(qp, p.sq.s, lsep, t_in + 1 + C::LA, t_in + 1 + C::LA);
#pragma unroll 1
                for (; t < t_out; t++) s_step(t, std::true_type{});
            }
            stop = t_end;
        }
        };
        if constexpr (BY_DWORD) {
            if (p.bias_vec == kByDword) s_loop(RowsTag<kByDword>{});
            else if (bias_vec) s_loop(RowsTag<kByChunk>{});
            else s_loop(RowsTag<kByElement>{});
        } else {
            if (TB != 0 && bias_vec) s_loop(RowsTag<kByChunk>{});
            else s_loop(RowsTag<kByElement>{});
        }
    } else {
        // ================================ dP-wave ================================
        // dS^T tile of this wave: 32 keys x BMI rows.  A lane writes its 4 consecutive rows of one key
        // with one 8-byte store, and ds_read_b64_tr_b16 hands a lane 4 consecutive keys of one row.
        T* ds_lds = reinterpret_cast<T*>(smem + C::OFF_DS) + kb * 32 * DSS;
        // lane -> row 16 ((lane/16)%2) + lane%16, keys 8 (lane/32 + 2 it) .. + 7 of the slice
        const int db_row = 16 * ((lane >> 4) & 1) + (lane & 15);
        const int db_src = (8 * (lane >> 5) + ((lane & 15) >> 2)) * DSS + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        // dBias rows that are whole aligned 16-byte chunks leave through unconditional buffer
        // stores (chunks outside the tensor get an offset outside the view): a loop without
        // branches around its stores lets the loads of the next blocks stay in flight across them.
        const bool db_fast = (DB_VIA_LDS && dbias_vec && (N % 8 == 0)) || (DB_VIA_LDS32 && dbias_vec && (N % 4 == 0));
        __amdgpu_buffer_rsrc_t db_rsrc = make_buffer(nullptr, 0);
        int db_off[2];
        const int db_row_bytes = (DB_VIA_LDS || DB_VIA_LDS32) ? (int)p.sdbias.m * C::ES : 0;
        // fp32: lane -> row 8 it + lane / 8, keys 4 (lane % 8) .. + 3 of the slice, it = 0 .. 3
        const int db32_row = lane >> 3, db32_key = 4 * (lane & 7);
        if (db_fast) {
            db_rsrc = make_buffer(dbp, ((int64_t)(M - 1) * p.sdbias.m + N) * C::ES);
            if constexpr (DB_VIA_LDS32) {
                db_off[0] = nw + db32_key < N ? db32_row * db_row_bytes + (nw + db32_key) * 4 : (int)0x80000000;
                db_off[1] = 0;
            } else {
#pragma unroll
                for (int it = 0; it < 2; it++) {
                    const int nn = nw + 8 * ((lane >> 5) + 2 * it);
                    db_off[it] = nn < N ? db_row * db_row_bytes + nn * 2 : (int)0x80000000;
                }
            }
        }
        float red_acc = 0.f;  // DBIAS == 2: this lane's share of the reduced gradient
        auto dp_loop = [&](auto fast_tag) {
        constexpr bool DB_FAST = decltype(fast_tag)::value;
        // copies per step; the dBias stores that may sit between them in the queue are not
        // counted, which only makes the wait at the end of a step stricter
        constexpr int COPIES = ((Q_BY_S ? 0 : 1) + (DO_BY_S ? 0 : 1)) * (C::QD + 1);
        auto dp_step = [&](int t, auto in_tag) {
            // IN: an interior step: blocks t - 1 .. t + LA are whole and in range
            constexpr bool IN = decltype(in_tag)::value;
            auto issue_copies = [&]() {
                if constexpr (COPIES > 0) {
                    const unsigned saved_m0 = lds_copy_begin();
                    if constexpr (IN) {
                        settle_ptrs(run_rows, run_stat, run_bias);
                        issue_next_do(t + C::LA);
                    } else {
                        if constexpr (!Q_BY_S) issue_q(t + 1 + C::LA);
                        if constexpr (!DO_BY_S) issue_do(t + C::LA);
                    }
                    lds_copy_end(saved_m0);
                }
            };
            const bool live = IN || (t >= mb_first && t < n_mblocks);
            const int m0 = t * BMI;
            const float* delta_lds = reinterpret_cast<const float*>(smem + C::OFF_DELTA) + (IN ? (unsigned)t % C::NDOB : (t < 0 ? 0 : t) % C::NDOB) * (C::STAT_BYTES / 4);
            const float* p_in = p_lds + (t & 1) * (C::P_BYTES / 4);
            T8 a_cols[NA], a_rows[NR];
            f32x4 del_in[4], p_vals[4];
            auto load_ds_inputs = [&]() {
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    del_in[q4] = *reinterpret_cast<const f32x4*>(delta_lds + 8 * q4 + 4 * g);
                    p_vals[q4] = *reinterpret_cast<const f32x4*>(p_in + (q4 * 64 + lane) * 4);
                }
            };
            if constexpr (TB == 0) issue_copies();
            // operands of both products up front: Q(t-1)^T for dK, the rows of dO(t) for dP
            if constexpr (C::DEFER_DK) load_cols((IN ? q_tile_in(t - 1) : q_tile(t - 1)), a_cols);
            load_rows((IN ? do_tile_in(t) : do_tile(t)), a_rows);
            if constexpr (PRELOAD && TB == 0) __builtin_amdgcn_sched_barrier(0);
            if constexpr (TB != 0) issue_copies();  // behind the reads, whose round trip they cover
            if (C::DEFER_DK && (IN || t - 1 >= mb_first)) mma_cols(a_cols, op_cur);  // dK^T += Q(t-1)^T dS(t-1)
            if (live) {
                f32x16 sacc;
                if constexpr (PRELOAD) {
                    load_ds_inputs();  // land while the products run
                    __builtin_amdgcn_sched_barrier(0);
                }
                mma_rows(a_rows, sacc);
                if constexpr (!PRELOAD) load_ds_inputs();
                // ---- dS = P (dP - delta) (flash_attention.py:303-308) ----
                i32x2 pk_even = {0, 0};
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const int ml0 = 8 * q4 + 4 * g;
                    const f32x4 del4 = del_in[q4];
                    const f32x4 p4 = p_vals[q4];
                    T4 d4;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int i = q4 * 4 + e;
                        const float dsv = p4[e] * (sacc[i] - del4[e]);
                        d4[e] = (T)dsv;
                        if constexpr (DBIAS == 2) {
                            // rows past M have P = 0 exactly, hence dS = 0
                            if constexpr (BIAS == 5)  // d bias / d slope = -|i N / M - j|
                                red_acc -= dsv * __builtin_fabsf(__builtin_fmaf((float)(m0 + 4 * g) + (float)(ml0 - 4 * g + e), ratio, -(float)my_n));
                            else red_acc += dsv;
                        }
                        if constexpr (DBIAS == 1 && !DB_VIA_LDS && !DB_VIA_LDS32) {
                            const int m = m0 + ml0 + e;
                            if (m < M && my_n < N) dbp[(int64_t)m * p.sdbias.m + (int64_t)my_n * p.sdbias.n] = (E)dsv;
                        }
                        // (p_in is this wave's part of the hand-off buffer read at the top of the step)
                        if constexpr (DB_VIA_LDS32) const_cast<float*>(p_in)[(ml0 + e) * 32 + r] = dsv;
                    }
                    // the operand of the dK product is made of the same packed words that go to the dS
                    // tile (assembled as integers: element-wise inserts made the compiler convert
                    // every value a second time, one by one, and merge the halves with permutes)
                    const i32x2 pk = __builtin_bit_cast(i32x2, d4);
                    if (q4 & 1) op_cur[q4 >> 1] = __builtin_bit_cast(T8, (i32x4){pk_even[0], pk_even[1], pk[0], pk[1]});
                    else pk_even = pk;
                    if constexpr (DB_VIA_LDS) *reinterpret_cast<T4*>(ds_lds + r * DSS + ml0) = d4;
                }
                // ---- dBias rows of this wave's 32 keys, 16 bytes per lane, out of the dS^T tile ----
                if constexpr (DB_VIA_LDS) {
#pragma unroll
                    for (int it = 0; it < 2; it++) {
                        const i16x4 lo = lds_read_tr4(ds_lds + db_src + it * 16 * DSS);
                        const i16x4 hi = lds_read_tr4(ds_lds + db_src + it * 16 * DSS + 4 * DSS);
                        typedef short i16x8 __attribute__((ext_vector_type(8)));
                        const i32x4 v = __builtin_bit_cast(i32x4, (i16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                        const int m = m0 + db_row, nn = nw + 8 * ((lane >> 5) + 2 * it);
                        if constexpr (DB_FAST) {
                            // rows past M: m0 * row bytes alone is past the view only if the view is
                            // tight, so the row test is explicit
                            const int off = (IN || m < M) ? db_off[it] + m0 * db_row_bytes : (int)0x80000000;
                            buf_store16(db_rsrc, v, off);
                        } else if (m < M && nn < N) {
                            E* dst = dbp + (int64_t)m * p.sdbias.m + (int64_t)nn * p.sdbias.n;
                            if (dbias_vec && nn + 8 <= N) {
                                gst16(dst, v);
                            } else {
                                const T8 v8 = as_vec<T8>(v);
#pragma unroll
                                for (int e = 0; e < 8; e++)
                                    if (nn + e < N) dst[(int64_t)e * p.sdbias.n] = __builtin_bit_cast(E, (T)v8[e]);
                            }
                        }
                    }
                }
                if constexpr (DB_VIA_LDS32) {
#pragma unroll
                    for (int it = 0; it < 4; it++) {
                        const int row = 8 * it + db32_row;
                        const f32x4 w = *reinterpret_cast<const f32x4*>(p_in + row * 32 + db32_key);
                        const i32x4 v = __builtin_bit_cast(i32x4, w);
                        const int m = m0 + row, nn = nw + db32_key;
                        if constexpr (DB_FAST) {
                            const int off = (IN || m < M) ? db_off[0] + (m0 + 8 * it) * db_row_bytes : (int)0x80000000;
                            buf_store16(db_rsrc, v, off);
                        } else if (m < M && nn < N) {
                            float* dst = reinterpret_cast<float*>(dbp) + (int64_t)m * p.sdbias.m + (int64_t)nn * p.sdbias.n;
                            if (dbias_vec && nn + 4 <= N) {
                                gst16(dst, v);
                            } else {
#pragma unroll
                                for (int e = 0; e < 4; e++)
                                    if (nn + e < N) dst[(int64_t)e * p.sdbias.n] = w[e];
                            }
                        }
                    }
                }
                if constexpr (!C::DEFER_DK) {  // dK^T += Q(t)^T dS(t)
                    load_cols((IN ? q_tile_in(t) : q_tile(t)), a_cols);
                    mma_cols(a_cols, op_cur);
                }
            }
            if constexpr (COPIES > 0) wait_vmcnt<COPIES*(C::LA - 1)>();
            lds_barrier();
        };
        // interior steps: block t - 1 was accumulated into dS (t - 1 >= mb_first) and the copied block t + LA is whole
        const int t_end = n_mblocks + 1;
        int t_in = mb_first + 1, t_out = n_full - C::LA;
        t_in = t_in < t_end ? t_in : t_end;
        t_out = t_out < t_in ? t_in : (t_out < t_end ? t_out : t_end);
        // (two passes over ONE copy of the general loop, the interior loop between them)
        int t = mb_first - 1, stop = t_in;
#pragma unroll 1
        for (int pass = 0; pass < 2; pass++) {
#pragma unroll 1
            for (; t < stop; t++) dp_step(t, std::false_type{});
            if (pass == 0 && t_in < t_out) {
                run_start(dop, p.sdo.s, deltap, t_in + C::LA, 0);
#pragma unroll 1
                for (; t < t_out; t++) dp_step(t, std::true_type{});
            }
            stop = t_end;
        }
        };
        if constexpr (DB_VIA_LDS || DB_VIA_LDS32) {
            if (db_fast) dp_loop(std::true_type{});
            else dp_loop(std::false_type{});
        } else {
            dp_loop(std::false_type{});
        }
        if constexpr (DBIAS == 2) {
            if constexpr (BIAS == 5) {
                // slope gradient of this wave's 32 keys: one float per (batch, head, key tile, wave), summed
                // over the lanes in a fixed order
                float s = my_n < N ? red_acc : 0.f;
#pragma unroll
                for (int w = 32; w >= 1; w >>= 1) s += __shfl_xor(s, w, 64);
                if (lane == 0) p.partials[((int64_t)bh * p.n_ntiles + nt) * C::WPR + kb] = s;
            } else {
                // column sums: lanes l and l + 32 hold different rows of the same key
                const float s = pair_sum(red_acc);
                if (g == 0 && my_n < N) p.partials[(int64_t)bh * N + my_n] = s;
            }
        }
    }
    // ---- dV (S-wave) or dK (dP-wave) of this wave's 32 keys (flash_attention.py:449-454) ----
    wait_vmcnt<0>();
    lds_barrier();  // (the rings are dead and no copy is in flight)
    static_assert(2 * C::WPR * WR::BYTES <= C::LDS_BYTES, "room for the way back");
    T* dst = s_wave ? reinterpret_cast<T*>(p.dv) + (int64_t)b * p.sdv.b + (int64_t)h * p.sdv.h
                    : reinterpret_cast<T*>(p.dk) + (int64_t)b * p.sdk.b + (int64_t)h * p.sdk.h;
    const unsigned own = lds_base + (unsigned)__builtin_amdgcn_readfirstlane(wave) * WR::BYTES;
    WR::store(acc, s_wave ? 1.f : p.sm_scale, own, dst, s_wave ? p.sdv.s : p.sdk.s, nw, N, s_wave ? p.d_v : p.d_qk, lane);
}

// ---------------------------------------------------------------------------------------------
// Few query rows at head dim 128: tiles of 64 keys, two work-groups to a CU.  What a tile costs beyond its steps (its operands,
// its first copies, two steps of skew, its stores: about 16 us) is then spent next to the steps of another one.  us, 128 -> 64
// keys: no bias B=8 H=12 S=512 53.0 -> 44.7, M=256 N=4096 H=32 83.3 -> 76.0; causal S=1024 95.7 -> 85.1, with a byte mask 108.6 ->
// 97.5, causal B=2 H=8 S=512 24.1 -> 17.3; read-only bf16 bias B=8 H=12 S=512 54.9 -> 45.2, B=64 491 -> 496.  (With the delta pass:) padding
// mask B=8 H=12 S=512 59.5 -> 53.1, B=64 H=16 498 -> 482, causal B=32 H=16 S=1024 575 -> 550; bf16 row and its gradient 63.3 -> 56.5, 517 ->
// 496, 617 -> 570; a trainable table for all batches 61.4 -> 53.4, 503 -> 496, 590 -> 545.  With more rows the
// second reading of Q and dO costs as much (B=4 H=16 S=2048 289 -> 293, byte mask B=2 H=16 S=1024 51.6 -> 52.6), and where dBias is
// written the shallow rings cost more (M=N=4096 712 -> 928).  An fp32 bias is copied one step ahead only in these rings, which costs
// more where a CU has many tiles, whose reads overlap anyway: B=8 H=12 S=512 56 -> 47, B=64 H=16 S=512 493 -> 513, causal 432 -> 460;
// causal B=8 H=12 S=1024 115 -> 112, B=32 H=16 565 -> 642.  Up to 320 rows in any number: M=N=257 B=32 H=16 135 -> 117, M=256 N=8192
// H=32 196 -> 190.
static bool short_rows(const BwdParams& p, int bias, bool causal) {
    if (bias == 4 && (int64_t)((p.N + 127) / 128) * p.B * p.H > (causal ? 4 : 2) * (int64_t)p.cus) return p.M <= 320;
    return p.M <= 512 || (causal && p.M <= 1024);
}
constexpr bool short_rows_built(int bias, int dbias) { return dbias == 0 || (dbias == 2 && bias >= 5); }

// Up to head dim 64: which of the kernels takes a bias tile.  A pair of waves keeps two waves per SIMD and the bias of three
// blocks in flight where a CU gets one tile only, and streams an fp32 bias and its gradient at the copy rate with one tile per
// CU (two of fa_bwd_narrow.hip read and write twice as many rows at a time: 4.6 TB/s).  us, one wave -> pair, D = 64:
//   one tile to a CU: fp32 read M=N=1024 H=32 37 -> 33, M=N=2048 H=8 62 -> 50; bf16 and dBias M=N=1500 H=8 57 -> 51, M=N=577 B=2
//     H=8 27 -> 24, 512 rows the same; at 256 tiles of 2048 rows 73 -> 82.  Below 512 rows the ends of a tile count for more
//     (fp32 read B=2 H=4 M=N=77 7 -> 8) but for fp32 and dBias, causal, whose tiles are few steps long: B=4 H=8 S=197 17 -> 16.  Long
//     ones of these that leave few CUs idle end up waiting for memory (with the delta pass: S=1500, 156 tiles 67 -> 61, 192 the
//     same, 216 91 -> 95, S=2000, 192 tiles 105 -> 109).
//   more, fp32 and dBias, not causal, any D: pairs of long tiles, whose last round of one to a CU is nearly full (with the delta
//     pass: M=N=2016 H=32 233 -> 218, D=32 222 -> 207, M=1280 N=1024 H=64 D=32 144 -> 140, 1.75 rounds the same, 1.25 or 2.5
//     rounds 122 -> 125 and 202 -> 209; 1024 rows, two rounds, 126 -> 128; M=600 N=1000 H=40 52 -> 63); where they are very
//     long the last round, then alone with the memory, matters less (M=N=4096, 1.5 rounds 343 -> 334, M=4096 N=512, 2.5 rounds 637
//     -> 613; M=2048 N=1024, 2.5 rounds 305 -> 308).  Causal, where long tiles are paired with short ones, B=2 H=16 M=N=2048 193 -> 230.
//   D = 16, one tile to a CU (with the delta pass, N=512, us): more than 1024 rows in 51 tiles and more, fp32 read, H=32 M=2304 60 ->
//     53 (32 tiles of 1088 rows 29 -> 30), and 16 bits and dBias where most CUs are idle, H=16 M=2304 57 -> 53 (128 tiles of 4096
//     rows 106 -> 130); fp32 and dBias the same either way.  At D = 32 none gains 5 %.
//   a byte mask, not causal, one tile to a CU of 1500 rows and more (N=512, H=16): M=1536 46.2 -> 44.5, M=4096 108 -> 101, 1088 rows
//     35.0 -> 34.5; causal S=2000 57.6 -> 58.7.
//   a dBias of the other 16-bit type: always one wave (M=N=1024 H=32 48 -> 37).
// A dBias whose rows allow no aligned 16-byte accesses, or a bias that is read element by element: always a pair, whose stores
// go out of registers, 32 keys of a row each, and which has 16 loads of a lane in flight, not 8 (fp32 dBias B=2 H=8 M=N=577 57
// -> 38, bf16 q and fp16 dBias B=2 H=16 M=N=1023 131 -> 59).
// fp32 rows that are fetched 4 bytes to a lane (kByDword): by the lines above, though a block takes 16 copies there, not 4.  Of 144
// cases (head dims 16 to 64, 8 to 960 tiles of 77 to 2049 rows, read only and dBias, causal and not) the other kernel is faster by
// more than 3 % in 22, 10 % at most (one wave / pair: D=64 M=511 N=515 H=8 21.6 / 19.7, D=16 B=2 H=12 M=N=1001 dBias 45.5 / 41.4;
// D=16 H=8 M=2049 N=2047 49.2 / 53.0, where the line takes the pair); with more tiles than CUs the pair loses up to half.
// (measured at 256 CUs, B=1 where none is given)
static bool pair_of_waves(const BwdParams& p, int D, int bias, int dbias, bool own_type, bool causal) {
    const int64_t tiles = (int64_t)p.n_ntiles * p.B * p.H;
    if (bias == 1) return !causal && p.bias_vec && p.M >= 1500 && tiles <= p.cus;
    if (!p.bias_vec || (dbias == 1 && !p.dbias_vec)) return true;
    if (bias != 4 && !own_type) return false;
    const bool fp32_dbias = bias == 4 && dbias == 1;
    if (tiles > p.cus) {
        if (!fp32_dbias || causal) return false;
        const int64_t last = tiles % p.cus;
        return (p.M >= 1280 && (last == 0 || 4 * last >= 3 * (int64_t)p.cus)) || (p.M > 2048 && 2 * tiles >= 3 * (int64_t)p.cus);
    }
    if (D == 16) {
        const bool long_tiles = !causal && p.M > 1024 && 5 * tiles >= p.cus;
        return long_tiles && !fp32_dbias && (bias == 4 ? 4 * tiles <= 3 * (int64_t)p.cus : 8 * tiles <= 3 * (int64_t)p.cus);
    }
    if (D != 64) return false;
    if (p.M < 512) return fp32_dbias && causal;
    if (fp32_dbias && causal && p.M >= 1500 && 4 * tiles >= 3 * (int64_t)p.cus) return false;
    return bias == 4 || tiles < p.cus || p.M < 2048;
}

template <typename T, int D, int BIAS, bool CAUSAL, int DBIAS, int W = bwd_waves(D)>
static hipError_t launch_main(const BwdParams& p, hipStream_t st) {
    // (the host has put 64-key tiles into p: short_rows)
    if constexpr (D == 128 && W == 4 && short_rows_built(BIAS, DBIAS)) {
        if (p.waves_per_role == 2) return launch_main<T, D, BIAS, CAUSAL, DBIAS, 2>(p, st);
    }
    dim3 grid((unsigned)(p.n_ntiles * p.B * p.H));
    hipLaunchKernelGGL((fa_bwd_kernel<T, D, BIAS, CAUSAL, DBIAS, W>), grid, dim3((BwdCfg<D, tile_kind(BIAS), W>::NT)), 0, st, p);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Second pass of the reduced dBias modes (DBIAS == 2), one thread per output element, sums in a
// fixed order: every output has one writer and the result is reproducible run to run.
//   float bias: dbias[b', h', 0, n] = sum over the broadcast batches / heads of colsum[b, h, n]
template <typename E>
__global__ __launch_bounds__(256) void fa_bwd_colsum_reduce_kernel(const BwdParams p) {
    const int nb_out = p.sdbias.b == 0 ? 1 : p.B, nh_out = p.sdbias.h == 0 ? 1 : p.H;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (int64_t)nb_out * nh_out * p.N) return;
    const int n = (int)(idx % p.N);
    const int ho = (int)((idx / p.N) % nh_out), bo = (int)(idx / ((int64_t)p.N * nh_out));
    float s = 0.f;
    for (int b = (nb_out == 1 ? 0 : bo); b < (nb_out == 1 ? p.B : bo + 1); b++)
        for (int h = (nh_out == 1 ? 0 : ho); h < (nh_out == 1 ? p.H : ho + 1); h++)
            s += p.partials[((int64_t)b * p.H + h) * p.N + n];
    reinterpret_cast<E*>(p.dbias)[(int64_t)bo * p.sdbias.b + (int64_t)ho * p.sdbias.h + (int64_t)n * p.sdbias.n] = (E)s;
}
//   ALiBi: dslope[h] = sum over batches, key tiles and waves of the partial slope gradients
// (a template so that the per-head-dim compile units may each hold a copy)
template <int LANES>
__global__ __launch_bounds__(LANES) void fa_bwd_slope_reduce_kernel(const BwdParams p) {
    static_assert(LANES == 64, "one wave");
    const int h = blockIdx.x, lane = threadIdx.x;
    const int per_bh = p.n_ntiles * p.waves_per_role;
    float s = 0.f;
    for (int b = 0; b < p.B; b++)
        for (int i = lane; i < per_bh; i += 64) s += p.partials[((int64_t)b * p.H + h) * per_bh + i];
#pragma unroll
    for (int w = 32; w >= 1; w >>= 1) s += __shfl_xor(s, w, 64);
    if (lane == 0) reinterpret_cast<float*>(p.dbias)[h] = s;
}

// fa_bwd_narrow.hip: dK, dV and dBias up to head dim 96
template <int D> hipError_t launch_bwd_narrow_d(const BwdParams& p, int dtype, int bias, bool causal, int dbias, hipStream_t st);

// dbias: 0 = none, 1 = dense, 2 = reduced in the kernels (see fa_bwd_kernel), 3 = of a shared bias (not here)
template <typename T, int D> static hipError_t launch_all(const BwdParams& p, int bias, bool causal, int dbias, int stages, hipStream_t st) {
    constexpr int PREP_D = D == 96 ? 128 : D;  // (a power of two of chunks per row)
    constexpr int RPB = 256 / (PREP_D / 8);
    const int64_t rows = (int64_t)p.B * p.H * p.M;
    dim3 rgrid((unsigned)((rows + RPB - 1) / RPB));
    hipError_t e = hipSuccess;
    // dBias in fp32 or in the element type of q, written densely a moment ago by the key-tile kernel
    // in rows of whole 16-byte chunks, is the dS the dQ product needs.  Only when that kernel ran in
    // this very call (or the caller vouches for the contents of dbias, bit 8) is it read.
    constexpr int DS_BIAS = __is_same(T, _Float16) ? 2 : 3;
    const bool ds_valid = dbias == 1 && ((stages & 2) || (stages & 8));
    const bool from_ds = (stages & 4) && ds_valid && (bias == DS_BIAS || bias == 4) && p.dbias_vec;
    // A dQ kernel that recomputes dS depends on nothing but delta.  When delta and dQ are asked for in one
    // call it runs FIRST and forms delta itself, bit for bit as fa_bwd_prep_kernel would, which saves a
    // launch and a pass over o and do; the dK/dV kernel then reads the delta it has stored.
    const bool dq_first = (stages & 5) == 5 && !from_ds;
    auto launch_dq = [&](bool makes_delta) -> hipError_t {
        // The one-product form runs at the rate of the dS stream: it gains from more work-groups only where the tiles
        // leave half of the CUs without one, that is where they are split in four or more (D = 128, H=8, N=8192, whole training
        // step, ms: M=64 0.153 -> 0.079, M=512 0.204 -> 0.154; one tile per CU, H=32 M=1024: this kernel 0.137 -> 0.161).
        BwdParams pq = p;
        pq.dq_makes_delta = makes_delta ? 1 : 0;
        if (from_ds && pq.dq_splits < 4) pq.dq_splits = 1;
        dim3 qgrid((unsigned)(pq.n_mtiles * pq.dq_splits * pq.B * pq.H));
        if (from_ds) {
            if constexpr (D == 96) {
                return hipErrorInvalidValue;  // (a dense dBias runs at 128)
            } else if (bias == DS_BIAS) {
                if (causal) hipLaunchKernelGGL((fa_bwd_dq_kernel<T, D, DS_BIAS, true, true>), qgrid, dim3(256), 0, st, pq);
                else hipLaunchKernelGGL((fa_bwd_dq_kernel<T, D, DS_BIAS, false, true>), qgrid, dim3(256), 0, st, pq);
            } else {
                if (causal) hipLaunchKernelGGL((fa_bwd_dq_kernel<T, D, 4, true, true>), qgrid, dim3(256), 0, st, pq);
                else hipLaunchKernelGGL((fa_bwd_dq_kernel<T, D, 4, false, true>), qgrid, dim3(256), 0, st, pq);
            }
        } else {
#define FA_CASE(BK)                                                                                               \
    case BK:                                                                                                      \
        if (causal) hipLaunchKernelGGL((fa_bwd_dq_kernel<T, D, BK, true>), qgrid, dim3(256), 0, st, pq);           \
        else hipLaunchKernelGGL((fa_bwd_dq_kernel<T, D, BK, false>), qgrid, dim3(256), 0, st, pq);                 \
        break;
            // a bias without a row dimension whose keys (of one share) fit the LDS row is staged once per
            // work-group instead of streamed
            const int keys_per_wg = pq.dq_splits > 1 ? pq.dq_keys_per_split : pq.N;
            const int qbias = (p.row_bias_kind != 0 && keys_per_wg <= kRowBiasKeys) ? (p.row_bias_kind == 1 ? 7 : 6) : bias;
            switch (qbias) {
                FA_CASE(0)
                FA_CASE(1)
                FA_CASE(2)
                FA_CASE(3)
                FA_CASE(4)
                FA_CASE(5)
                FA_CASE(6)
                FA_CASE(7)
                default: return hipErrorInvalidValue;
            }
#undef FA_CASE
        }
        hipError_t eq = hipGetLastError();
        if (eq == hipSuccess && pq.dq_splits > 1) {
            const int64_t threads = (int64_t)p.B * p.H * p.M * (D / 8);
            hipLaunchKernelGGL((fa_bwd_dq_sum_kernel<T, D>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, pq);
            eq = hipGetLastError();
        }
        return eq;
    };
    if ((stages & 1) && !dq_first) {
        hipLaunchKernelGGL((fa_bwd_prep_kernel<T, PREP_D>), rgrid, dim3(256), 0, st, p);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (dq_first) {
        e = launch_dq(true);
        if (e != hipSuccess) return e;
    }
    if (stages & 2) {
    // a bias that is the same for every query row is one register per key for this kernel
    // (dbias 3, the gradient of a shared bias, is a kernel of its own: here the bias is only read)
    const int kbias = (p.row_bias_kind != 0 && dbias != 1) ? (p.row_bias_kind == 1 ? 7 : 6) : bias;
    const int kdbias = dbias == 3 ? 0 : dbias;
    BwdParams pk = p;
    if (D == 128 && short_rows_built(kbias, kdbias) && short_rows(p, kbias, causal)) {
        pk.n_ntiles = (p.N + 63) / 64;
        pk.waves_per_role = 2;
    }
    if constexpr (D <= 96) {
        bool pair = false;
        if constexpr (D <= 64) {
            pair = pair_built(D, kbias, kdbias) && pair_of_waves(p, D, kbias, kdbias, kbias == DS_BIAS, causal);
            if (pair) e = hipErrorInvalidValue;  // (until one of these has it)
#define FA_CASE(BK, DBK)                                                                                      \
    if (pair && kbias == BK && kdbias == DBK)                                                                  \
        e = causal ? launch_main<T, D, BK, true, DBK>(p, st) : launch_main<T, D, BK, false, DBK>(p, st);
            FA_CASE(2, 1)
            FA_CASE(3, 1)
            FA_CASE(4, 1)
            FA_CASE(4, 0)
#undef FA_CASE
            if constexpr (D == 64) {
                if (pair && kbias == 1) e = launch_main<T, D, 1, false, 0>(p, st);
            }
        }
        if (!pair) e = launch_bwd_narrow_d<D>(p, __is_same(T, __bf16), kbias, causal, kdbias, st);
    } else {
#define FA_CASE(BK, DBK)                                                                                      \
    if (kbias == BK && kdbias == DBK)                                                                          \
        e = causal ? launch_main<T, D, BK, true, DBK>(pk, st) : launch_main<T, D, BK, false, DBK>(pk, st);
    FA_CASE(0, 0)
    else FA_CASE(6, 0)
    else FA_CASE(6, 2)
    else FA_CASE(7, 0)
    else FA_CASE(1, 0)
    else FA_CASE(2, 0)
    else FA_CASE(2, 1)
    else FA_CASE(2, 2)
    else FA_CASE(3, 0)
    else FA_CASE(3, 1)
    else FA_CASE(3, 2)
    else FA_CASE(4, 0)
    else FA_CASE(4, 1)
    else FA_CASE(4, 2)
    else FA_CASE(5, 0)
    else FA_CASE(5, 2)
    else return hipErrorInvalidValue;
#undef FA_CASE
    }
        if (e != hipSuccess) return e;
        if (dbias == 2) {
            if (bias == 5) {
                hipLaunchKernelGGL((fa_bwd_slope_reduce_kernel<64>), dim3((unsigned)p.H), dim3(64), 0, st, pk);
            } else {
                const int64_t outs = (int64_t)(p.sdbias.b == 0 ? 1 : p.B) * (p.sdbias.h == 0 ? 1 : p.H) * p.N;
                dim3 g((unsigned)((outs + 255) / 256));
                if (bias == 2) hipLaunchKernelGGL((fa_bwd_colsum_reduce_kernel<_Float16>), g, dim3(256), 0, st, p);
                else if (bias == 3) hipLaunchKernelGGL((fa_bwd_colsum_reduce_kernel<__bf16>), g, dim3(256), 0, st, p);
                else hipLaunchKernelGGL((fa_bwd_colsum_reduce_kernel<float>), g, dim3(256), 0, st, p);
            }
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    if ((stages & 4) && !dq_first) e = launch_dq(false);
    return e;
}

// This file is compiled once per head dimension (-DFA_HEAD_DIM=16 ... 256, 96 for those of 128 that are no larger); each object exports
// launch_bwd_d<FA_HEAD_DIM>.
#ifndef FA_HEAD_DIM
#error "compile with -DFA_HEAD_DIM=<16|32|64|96|128|256>"
#endif
template <int D> hipError_t launch_bwd_d(const BwdParams& p, int dtype, int bias, bool causal, int dbias, int stages, hipStream_t st);
template <> hipError_t launch_bwd_d<FA_HEAD_DIM>(const BwdParams& p, int dtype, int bias, bool causal, int dbias, int stages, hipStream_t st) {
    if (dtype == 0) return launch_all<_Float16, FA_HEAD_DIM>(p, bias, causal, dbias, stages, st);
    return launch_all<__bf16, FA_HEAD_DIM>(p, bias, causal, dbias, stages, st);
}

}  // namespace fa

