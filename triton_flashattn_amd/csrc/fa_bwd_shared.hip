// Gradient of a bias that is shared by batches or heads but not by query rows (a table of relative positions,
// (1, H, M, N); a mask-like (B, 1, M, N); one (M, N) for everything): the sum of dS over the pairs that share it.
// The reference writes dS for every (batch, head) and leaves that sum to autograd (flash_attention.py:307-308).
//
// Here no dS of a single pair is written.  A work-group owns one 128 x 64 tile of the gradient and walks the
// (batch, head) pairs that share it: S^T = K Q^T and dP^T = V dO^T of the tile, dS = P (dP - delta) added to
// accumulators that stay in registers in fp32; the tile of the bias, the same for every pair, stays there too.
// Recomputing the two products costs 4 D operations per score where writing dS, reading it back and adding it up
// moves three times its bytes: at D = 64 and an fp32 bias 0.25 us against 2.5 us per million scores at this
// card's rates, and there is no scratch of the size of dS.
//
// A pass over a pair is 48 KB of rows through LDS, whose reads (1024 clocks per pair and tile) and the vector
// work (900) bound it together; the rows arrive through direct global -> LDS copies two pairs ahead (LDS for three
// pairs, one work-group per CU).  Head dims above 64 are taken in slices of 64.  Few tiles: the pairs are split
// between work-groups, whose shares in fp32 a second kernel adds in a fixed order.
// Measured: 32 batches, 12 heads, M=N=197, D=64, fp32 table: 0.023 ms and 0.005 for the shares; 24 batches, 16 heads,
// M=N=577: 0.122 ms (0.167 with addresses formed from the indices and every copy behind the barrier).  Before, one
// backward per batch with its dS written and added up: the whole training step at 32 batches took 2.1 ms, now 0.11.
// Few pairs: a tile then costs what stands around its pairs.  With the bias and the gradient accessed one element at a
// time, each load behind the one before, and products formed for a pair behind the last that was 10 us of a tile at
// D = 128 (2 us per pair); whole training steps with bf16 tables, two batches, us, one backward per batch / that / now:
// H=16 M=N=4096 D=64 2575 / 2734 / 1868, H=16 M=N=2048 D=128 723 / 849 / 616, causal 698 / 550 / 389, D=256 causal
// 860 / 972 / 731, D=256 1106 / 1594 / 1318: there the four slices of a pair are what bounds it, 1.5 us each, whatever
// the order of their copies, products and tiles.
#include "fa_common.hpp"
#include "fa_params.hpp"

namespace fa {

constexpr int kSharedM = kSharedTileM, kSharedN = kSharedTileN;

template <int D> struct SharedCfg {
    static constexpr int DC = D < 64 ? D : 64, CHUNKS = D / DC;  // slices of the head dim
    static constexpr int CPR = DC / 8, KS = DC / 16;
    static constexpr int Q_BYTES = kSharedM * DC * 2, K_BYTES = kSharedN * DC * 2;
    static constexpr int QCP = Q_BYTES / 1024, KCP = K_BYTES / 1024;        // 1 KB copies per tensor
    static constexpr int NQ = QCP >= 8 ? QCP / 8 : 1, NK = KCP >= 8 ? KCP / 8 : 1;  // of which a wave issues so many
    static constexpr int COPIES = 2 * NQ + 2 * NK + 1;
    static_assert(COPIES <= 8, "one copy per slot of a pair");
    static constexpr int OFF_DO = Q_BYTES, OFF_K = 2 * Q_BYTES, OFF_V = OFF_K + K_BYTES, OFF_STAT = OFF_V + K_BYTES;
    static constexpr int STAGE = OFF_STAT + 1024;  // LSE and delta of 128 rows
    static constexpr int STAGES = 3;
};

// elements (m, n .. n + 3) of slice (bo, ho) of the gradient
template <typename E> __device__ __forceinline__ void store_grad4(const BwdParams& p, int64_t at, int n, f32x4 v) {
    typedef E E4 __attribute__((ext_vector_type(4)));
    E* dst = reinterpret_cast<E*>(p.dbias) + at;
    if (p.dbias_quads && n + 4 <= p.N) {
        const E4 w = {(E)v[0], (E)v[1], (E)v[2], (E)v[3]};
        *reinterpret_cast<E4*>(dst) = w;
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (n + e < p.N) dst[(int64_t)e * p.sdbias.n] = (E)v[e];
}
__device__ __forceinline__ void store_grad4(const BwdParams& p, int bo, int ho, int m, int n, f32x4 v) {
    if (m >= p.M) return;
    const int64_t at = (int64_t)bo * p.sdbias.b + (int64_t)ho * p.sdbias.h + (int64_t)m * p.sdbias.m + (int64_t)n * p.sdbias.n;
    if (p.bias_kind == 2) store_grad4<_Float16>(p, at, n, v);
    else if (p.bias_kind == 3) store_grad4<__bf16>(p, at, n, v);
    else store_grad4<float>(p, at, n, v);
}

// A lane's 16 elements of a bias row in log2 units: i is key n + 8 (i/4) + i%4.  The kind is chosen once around all loads:
// chosen per element, each load waits for the one before it.
template <typename E> __device__ __forceinline__ void load_bias16(const BwdParams& p, int64_t row, int n, bool quads, float (&out)[16]) {
    typedef E E4 __attribute__((ext_vector_type(4)));
    const E* src = reinterpret_cast<const E*>(p.bias) + row;
    E4 raw[4];
    if (quads) {
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) raw[q4] = *reinterpret_cast<const E4*>(src + n + 8 * q4);
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int at = n + 8 * (i / 4) + i % 4;
            raw[i / 4][i % 4] = src[(int64_t)(at < p.N ? at : p.N - 1) * p.sbias.n];
        }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) out[i] = (float)raw[i / 4][i % 4] * kLog2e;
}

// Output slice and tile number `tile` (slice-major, rows of tiles inside a slice).
struct SharedPlace {
    int m0, n0, bo, ho;
};
__device__ __forceinline__ SharedPlace shared_place(const BwdParams& p, int tile) {
    SharedPlace w;
    const int nt = (p.N + kSharedN - 1) / kSharedN, mt = (p.M + kSharedM - 1) / kSharedM;
    w.n0 = (tile % nt) * kSharedN;
    w.m0 = (tile / nt % mt) * kSharedM;
    const int slice = tile / (nt * mt), nh = p.sdbias.h == 0 ? 1 : p.H;
    w.ho = slice % nh;
    w.bo = slice / nh;
    return w;
}

template <typename T, int D>
__global__ __launch_bounds__(512, 2) void fa_bwd_shared_bias_kernel(const BwdParams p) {
    typedef SharedCfg<D> C;
    typedef Swz<C::DC> SW;
    typedef typename VecOf<T>::v8 T8;
    __shared__ __align__(1024) unsigned char smem[C::STAGES * C::STAGE];

    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Work-groups are dealt round-robin to the 8 XCDs: each XCD takes a run of neighbours in the order (slice, share,
    // tile), which walk the same pairs at about the same time, so that their rows come from its L2 (2 % at 24 batches,
    // 16 heads, M=N=577, D=64).
    const int per_slice = ((p.N + kSharedN - 1) / kSharedN) * ((p.M + kSharedM - 1) / kSharedM), splits = p.shared_splits;
    const int place = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    if (place >= p.shared_tiles * splits) return;
    const int split = place / per_slice % splits, tile = place / (per_slice * splits) * per_slice + place % per_slice;
    const SharedPlace at = shared_place(p, tile);
    const int m0 = at.m0, n0 = at.n0, M = p.M, N = p.N;
    const int my_m = m0 + (wave >> 1) * 32 + r, nb = (wave & 1) * 32;  // this lane's query row, first key of the wave's block
    const bool over_b = p.sdbias.b == 0 && p.B > 1, over_h = p.sdbias.h == 0 && p.H > 1;
    const int heads = over_h ? p.H : 1, pairs = (over_b ? p.B : 1) * heads;
    const int per = (pairs + splits - 1) / splits;
    const int r0 = split * per, r1 = pairs < r0 + per ? pairs : r0 + per;

    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.f;

    // causal: a tile above the diagonal has no dS
    if (r0 < r1 && !(p.causal && n0 > m0 + kSharedM - 1)) {
        // the bias of the tile: register i is key n0 + nb + 8 (i/4) + 4 g + i%4
        float bias2[16];
        {
            const int64_t row = (int64_t)at.bo * p.sbias.b + (int64_t)at.ho * p.sbias.h + (int64_t)(my_m < M ? my_m : M - 1) * p.sbias.m;
            const bool quads = p.bias_quads && n0 + kSharedN <= N;
            if (p.bias_kind == 2) load_bias16<_Float16>(p, row, n0 + nb + 4 * g, quads, bias2);
            else if (p.bias_kind == 3) load_bias16<__bf16>(p, row, n0 + nb + 4 * g, quads, bias2);
            else load_bias16<float>(p, row, n0 + nb + 4 * g, quads, bias2);
        }
        // Copies: of the 1 KB pieces of a tensor's tile this wave issues NQ (Q, dO) or NK (K, V); lane l of piece ci
        // fetches the chunk at tile position 64 ci + l.  Rows past the end re-read the last one: what they give
        // is not stored.
        unsigned q_off[C::NQ], do_off[C::NQ], k_off[C::NK], v_off[C::NK];
        auto piece = [&](int i, int n, int total) { return (wave * n + i) % total; };
        auto offset = [&](int ci, int first, int count, int64_t stride) {
            const int c = ci * 64 + lane;
            int row = c / C::CPR;
            const int src = (c % C::CPR) ^ SW::f(row);
            row = first + row < count ? row : count - 1 - first;
            return (unsigned)(row * (int)stride * 2 + src * 16);
        };
#pragma unroll
        for (int i = 0; i < C::NQ; i++) {
            q_off[i] = offset(piece(i, C::NQ, C::QCP), m0, M, p.sq.s);
            do_off[i] = offset(piece(i, C::NQ, C::QCP), m0, M, p.sdo.s);
        }
#pragma unroll
        for (int i = 0; i < C::NK; i++) {
            k_off[i] = offset(piece(i, C::NK, C::KCP), n0, N, p.sk.s);
            v_off[i] = offset(piece(i, C::NK, C::KCP), n0, N, p.sv.s);
        }
        // waves 0, 1: LSE of rows 0 .. 63, 64 .. 127; waves 2, 3: delta (the other four again)
        const int stat_part = wave & 3;
        int stat_row = m0 + (stat_part & 1) * 64 + lane;
        stat_row = stat_row < M ? stat_row : M - 1;
        const unsigned lds_base = lds_addr_of(smem);

        // The copies walk the pairs with running 64-bit addresses in scalar registers (formed from the pair's indices
        // they would cost 150 scalar instructions per pair, in front of the copies): Q, dO, K, V, LSE or delta.
        const int pair0 = r0;
        const int b0 = over_b ? pair0 / heads : at.bo, h0 = over_h ? pair0 % heads : at.ho;
        const float* stat_src = stat_part < 2 ? p.lse : p.delta;
        uint64_t run[5] = {
            uniform_ptr(reinterpret_cast<const T*>(p.q) + (int64_t)b0 * p.sq.b + (int64_t)h0 * p.sq.h + (int64_t)m0 * p.sq.s),
            uniform_ptr(reinterpret_cast<const T*>(p.dout) + (int64_t)b0 * p.sdo.b + (int64_t)h0 * p.sdo.h + (int64_t)m0 * p.sdo.s),
            uniform_ptr(reinterpret_cast<const T*>(p.k) + (int64_t)b0 * p.sk.b + (int64_t)h0 * p.sk.h + (int64_t)n0 * p.sk.s),
            uniform_ptr(reinterpret_cast<const T*>(p.v) + (int64_t)b0 * p.sv.b + (int64_t)h0 * p.sv.h + (int64_t)n0 * p.sv.s),
            uniform_ptr(stat_src + ((int64_t)b0 * p.H + h0) * M)};
        // bytes to the next pair: one head on, or from the last head of a batch to the first of the next
        const int64_t sh[5] = {p.sq.h * 2, p.sdo.h * 2, p.sk.h * 2, p.sv.h * 2, (int64_t)M * 4};
        const int64_t sb[5] = {p.sq.b * 2, p.sdo.b * 2, p.sk.b * 2, p.sv.b * 2, (int64_t)p.H * M * 4};
        int64_t to_head[5], to_batch[5];
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const int64_t back = i < 4 ? (int64_t)(C::CHUNKS - 1) * C::DC * 2 : 0;
            to_head[i] = sh[i] - back;
            to_batch[i] = sb[i] - (heads - 1) * sh[i] - back;
        }
        int heads_left = heads - (over_h ? h0 : 0), chunk = 0, left = (r1 - r0) * C::CHUNKS;
        unsigned slot_in = 0, slot_out = 0;  // byte offsets of the stages that are filled and read next
        auto next_slot = [](unsigned slot) { return slot == (C::STAGES - 1) * C::STAGE ? 0u : slot + C::STAGE; };
        // copy number c of a stage
        auto copy = [&](int c) __attribute__((always_inline)) {
            const unsigned dst = __builtin_amdgcn_readfirstlane(lds_base + slot_in);
            const unsigned saved_m0 = lds_copy_begin();
            if (c < 2 * C::NQ) {
                const int at_c = piece(c / 2, C::NQ, C::QCP) * 1024;
                if (c % 2 == 0) lds_copy16(run[0], q_off[c / 2], dst + at_c);
                else lds_copy16(run[1], do_off[c / 2], dst + C::OFF_DO + at_c);
            } else if (c < C::COPIES - 1) {
                const int i = (c - 2 * C::NQ) / 2, at_c = piece(i, C::NK, C::KCP) * 1024;
                if (c % 2 == 0) lds_copy16(run[2], k_off[i], dst + C::OFF_K + at_c);
                else lds_copy16(run[3], v_off[i], dst + C::OFF_V + at_c);
            } else {
                lds_copy4(run[4], (unsigned)stat_row * 4u, dst + C::OFF_STAT + stat_part * 256);
            }
            lds_copy_end(saved_m0);
        };
        auto settle = [&]() __attribute__((always_inline)) {
            settle_ptrs(run[0], run[1], run[2]);
            settle_ptrs(run[3], run[4], run[0]);
        };
        // after the last copy of a stage: on to the next
        auto advance = [&]() __attribute__((always_inline)) {
            slot_in = next_slot(slot_in);
            if (--left <= 0) return;  // (past the end: the last one again, never read)
            if (C::CHUNKS > 1 && ++chunk < C::CHUNKS) {
#pragma unroll
                for (int i = 0; i < 4; i++) run[i] += C::DC * 2;
                return;
            }
            chunk = 0;
            const bool wrap = --heads_left == 0;
            if (wrap) heads_left = heads;
#pragma unroll
            for (int i = 0; i < 5; i++) run[i] += (uint64_t)(wrap ? to_batch[i] : to_head[i]);
        };
        wait_vmcnt<0>();  // the bias loads above: left in flight, the compiler would wait for every copy with them
        const float qk_scale = p.sm_scale * kLog2e;
        const unsigned rows_l = SW::rows_lane(lane);
        const bool masked = p.causal && n0 + kSharedN - 1 > m0;
        T8 ops[4][C::KS];  // rows of K, Q, V and dO of a stage
        f32x16 xa[2], xb[2];  // scores and dP of the pair whose dS is due, and of the one after it
        float lse = 0.f, delta = 0.f, lse_next, delta_next;
        auto issue = [&]() __attribute__((always_inline)) {
            settle();
#pragma unroll
            for (int c = 0; c < C::COPIES; c++) copy(c);
            advance();
        };
        // the next stage: waits for it and fetches its operands
        auto begin = [&]() __attribute__((always_inline)) {
            wait_vmcnt<C::COPIES>();  // all but the copies of the next stage have landed
            lds_barrier();            // ... for every wave; and the stage before it has been read
            const unsigned base = lds_base + slot_out + rows_l;
            const unsigned q_at = base + (unsigned)((wave >> 1) * 32 * SW::RB), k_at = base + C::OFF_K + (unsigned)(nb * SW::RB);
#pragma unroll
            for (int ks = 0; ks < C::KS; ks++) {
                ops[0][ks] = SW::template row8_at<T8>(k_at, 0, ks);
                ops[1][ks] = SW::template row8_at<T8>(q_at, 0, ks);
            }
#pragma unroll
            for (int ks = 0; ks < C::KS; ks++) {
                ops[2][ks] = SW::template row8_at<T8>(k_at + (C::OFF_V - C::OFF_K), 0, ks);
                ops[3][ks] = SW::template row8_at<T8>(q_at + C::OFF_DO, 0, ks);
            }
            const float* stat = reinterpret_cast<const float*>(smem + slot_out + C::OFF_STAT) + (wave >> 1) * 32 + r;
            lse_next = stat[0];
            delta_next = stat[128];
            slot_out = next_slot(slot_out);
        };
        // matrix instruction j of 2 KS: S = K Q^T, then dP = V dO^T
        auto mma = [&](f32x16 (&x)[2], int j) {
            const int half = j / C::KS, ks = j % C::KS;
            x[half] = mfma32(ops[2 * half][ks], ops[2 * half + 1][ks], x[half]);
        };
        // element i of the dS of the pair whose scores are in `cur`
        auto add_ds = [&](const f32x16 (&cur)[2], int i, auto masked_tag) __attribute__((always_inline)) {
            float x = __builtin_fmaf(cur[0][i], qk_scale, bias2[i]);
            if (decltype(masked_tag)::value && my_m < n0 + nb + 8 * (i / 4) + 4 * g + i % 4) x += kMask;
            acc[i] = __builtin_fmaf(fast_exp2(x - lse), cur[1][i] - delta, acc[i]);
        };
        // the products of a slice of the head dim, the copies of a stage between them
        auto slice = [&](f32x16 (&x)[2]) __attribute__((always_inline)) {
            begin();
            settle();
#pragma unroll
            for (int j = 0; j < 2 * C::KS || j < C::COPIES; j++) {
                if (j < 2 * C::KS) mma(x, j);
                if (j < C::COPIES) copy(j);
            }
            advance();
        };
        // One pair: the products of the NEXT one are issued between the element-wise work of this one, whose scores
        // are in `cur` (what bounds a pass would otherwise be the sum of the two and of the LDS reads).
        auto pair_step = [&](f32x16 (&cur)[2], f32x16 (&next)[2], auto masked_tag) __attribute__((always_inline)) {
            begin();
            settle();
#pragma unroll
            for (int i = 0; i < 16; i++) next[0][i] = next[1][i] = 0.f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                __builtin_amdgcn_sched_barrier(0);
                add_ds(cur, 2 * j, masked_tag);
                add_ds(cur, 2 * j + 1, masked_tag);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = j * 2 * C::KS / 8; k < (j + 1) * 2 * C::KS / 8; k++) mma(next, k);
                // (a copy holds its wave while those of the others drain: one per slot, behind a matrix instruction)
                if (j < C::COPIES) copy(j);
            }
            advance();
            __builtin_amdgcn_sched_barrier(0);
            lse = lse_next;
            delta = delta_next;
#pragma unroll
            for (int c = 1; c < C::CHUNKS; c++) slice(next);
        };
        issue();
        issue();
#pragma unroll
        for (int i = 0; i < 16; i++) xa[0][i] = xa[1][i] = 0.f;
#pragma unroll
        for (int c = 0; c < C::CHUNKS; c++) slice(xa);
        lse = lse_next;
        delta = delta_next;
        auto walk = [&](auto masked_tag) {
            int n = r1 - r0;  // pairs whose dS is due
#pragma unroll 1
            for (; n > 2; n -= 2) {
                pair_step(xa, xb, masked_tag);
                pair_step(xb, xa, masked_tag);
            }
            if (n == 2) {
                pair_step(xa, xb, masked_tag);
                xa[0] = xb[0];
                xa[1] = xb[1];
            }
#pragma unroll
            for (int i = 0; i < 16; i++) add_ds(xa, i, masked_tag);  // the last one: no products behind it
        };
        if (masked) walk(BoolTag<true>{});
        else walk(BoolTag<false>{});
        wait_vmcnt<0>();  // nothing may land in LDS after the work-group has ended
    }

#pragma unroll
    for (int q4 = 0; q4 < 4; q4++) {
        const f32x4 v = {acc[4 * q4], acc[4 * q4 + 1], acc[4 * q4 + 2], acc[4 * q4 + 3]};
        if (splits > 1)
            reinterpret_cast<f32x4*>(p.partials)[(((int64_t)tile * splits + split) * 8 + wave) * 256 + q4 * 64 + lane] = v;
        else
            store_grad4(p, at.bo, at.ho, my_m, n0 + nb + 8 * q4 + 4 * g, v);
    }
}

// Adds the shares of a tile in their order and stores the sums: one thread per four elements, 16 blocks per tile.
template <int NT> __global__ __launch_bounds__(NT) void fa_bwd_shared_bias_sum_kernel(const BwdParams p) {
    constexpr int QUADS = kSharedM * kSharedN / 4;
    static_assert(QUADS % NT == 0, "blocks of whole tiles");
    const int tile = blockIdx.x / (QUADS / NT);
    const SharedPlace at = shared_place(p, tile);
    const int quad = (blockIdx.x % (QUADS / NT)) * NT + threadIdx.x;
    const int wave = quad >> 8, q4 = (quad >> 6) & 3, lane = quad & 63;
    const f32x4* share = reinterpret_cast<const f32x4*>(p.partials) + (int64_t)tile * p.shared_splits * QUADS + quad;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 0; s < p.shared_splits; s++) sum += share[(int64_t)s * QUADS];
    store_grad4(p, at.bo, at.ho, at.m0 + (wave >> 1) * 32 + (lane & 31), at.n0 + (wave & 1) * 32 + 8 * q4 + 4 * (lane >> 5), sum);
}

template <typename T, int D> static hipError_t launch_shared(const BwdParams& p, hipStream_t st) {
    const unsigned groups = (unsigned)(p.shared_tiles * p.shared_splits);
    hipLaunchKernelGGL((fa_bwd_shared_bias_kernel<T, D>), dim3((groups + 7) / 8 * 8), dim3(512), 0, st, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.shared_splits == 1) return e;
    hipLaunchKernelGGL((fa_bwd_shared_bias_sum_kernel<128>), dim3((unsigned)p.shared_tiles * (kSharedM * kSharedN / 512)), dim3(128), 0, st, p);
    return hipGetLastError();
}

// This file is compiled once per head dimension (-DFA_HEAD_DIM=16 ... 256); each object exports
// launch_bwd_shared_d<FA_HEAD_DIM>.
#ifndef FA_HEAD_DIM
#error "compile with -DFA_HEAD_DIM=<16|32|64|128|256>"
#endif
template <int D> hipError_t launch_bwd_shared_d(const BwdParams& p, int dtype, hipStream_t st);
template <> hipError_t launch_bwd_shared_d<FA_HEAD_DIM>(const BwdParams& p, int dtype, hipStream_t st) {
    return dtype == 0 ? launch_shared<_Float16, FA_HEAD_DIM>(p, st) : launch_shared<__bf16, FA_HEAD_DIM>(p, st);
}

}  // namespace fa
