// dK, dV and dBias for head dims up to 64, and up to 96 without a bias tile (flash_attention.py:237-454).
//
// A work-group of 4 waves owns 128 keys, a wave 32 of them with everything that belongs to them: K and V as operands in
// registers, the scores, dP, and the accumulators of dK^T and dV^T (128 registers at D = 64).  Query rows stream through
// LDS in steps of 64 or 32.  Scores are not transposed: a lane holds one KEY and 16 query rows of a 32 x 32 block, so
// P and dS are, as they leave the registers, the B operands of dV^T += dO^T P and dK^T += Q^T dS.
//
// Why one wave does both halves here and a pair of waves at D = 128 (fa_bwd_kernel): what the pair hands over, P in fp32,
// and the values per row that both of its halves read are as large as the operands of the products at D = 64 (32 KB of
// LDS traffic per 32 x 32 block, 512 clocks of a CU's LDS for its four SIMDs, as much as the matrix work).  One wave needs
// 21 KB, no step of skew at either end of a tile, and half the waves, so that two tiles fit a CU with 256 registers per
// lane; at D = 128 it would have a SIMD to itself (0.51 -> 0.54 ms at B=2 H=16 M=N=4096).  Bound by the matrix pipeline
// under the power limit where tiles are long (1.1 PFLOP/s), by the ends of tiles where they are short.
// us, pair of waves -> this kernel, D = 64 bf16: B=4 H=32 M=N=4096 1221 -> 1000; B=4 H=16 S=2048 causal 110 -> 84; ALiBi there
// 128 -> 94; byte mask B=8 H=12 S=1024 causal 76 -> 54; B=32 H=12 M=N=192 with an fp32 bias that is read 41 -> 32; bf16 bias
// and dBias B=2 H=16 M=N=4096 584 -> 511 (2.2 GB: HBM); D = 32, B=8 H=32 S=2048 463 -> 338.
#include <type_traits>

#include "fa_common.hpp"
#include "fa_params.hpp"

namespace fa {

// BIAS: kind of bias tile that is streamed (0 none, 1 bytes, 2 / 3 16 bits, 4 fp32)
template <int D, int BIAS> struct NarrowCfg {
    static constexpr int ES = BIAS == 0 ? 0 : (BIAS == 1 ? 1 : (BIAS == 4 ? 4 : 2));
    // 32-row blocks per step, and steps the copies run ahead.  Two blocks to a barrier wherever two work-groups fit a CU
    // with them (with three steps of one block ahead in the same LDS, bf16 bias and dBias at B=2 H=16 M=N=4096 D=64:
    // 0.511 -> 0.569 ms; without a bias, two steps ahead 1.05 -> 1.08 ms at B=4 H=32).
    static constexpr int NB = ES == 4 ? 1 : 2;
    static constexpr int LA = ES == 4 ? 2 : 1;
    static constexpr int BN = 128, NT = 256, SR = 32 * NB;
    static constexpr int DB = D < 32 ? 1 : D / 32;       // 32-wide blocks of the head dim
    static constexpr int KSTEPS = D / 16;
    static constexpr int CPR = D / 8;                    // 16-byte chunks per row
    static constexpr int NS = LA + 1;                    // slots of every ring
    static constexpr int ROWS_BYTES = SR * D * 2;        // the Q (or dO) rows of a step, swizzled
    static constexpr int NQD = ROWS_BYTES / 1024;        // 1 KB copies of them
    static constexpr int QD = (NQD + 3) / 4;             // of which each wave issues this many
    static constexpr int STAT_BYTES = 64 * 4;            // LSE (or delta) of a step: a copy is 64 lanes wide
    static constexpr int EPC = ES > 0 ? 16 / ES : 8;     // bias elements per 16-byte chunk
    static constexpr int BCPR = 2 * ES;                  // 16-byte chunks per bias row of 32 keys
    static constexpr int BBLOCK = 32 * 32 * ES;          // bias of one wave and 32 rows
    static constexpr int BSLOT = NB * BBLOCK;            // ... and of a step
    static constexpr int BCH = BSLOT / 1024;             // copies of that
    static constexpr int DSS = 36;                       // dS^T tile: elements between two keys
    static constexpr int DS_BYTES = ES == 2 ? 32 * DSS * 2 : 0;  // of one wave
    static constexpr int OFF_DO = NS * ROWS_BYTES;
    static constexpr int OFF_STAT = 2 * NS * ROWS_BYTES;
    static constexpr int OFF_BIAS = OFF_STAT + NS * 2 * STAT_BYTES;
    static constexpr int OFF_DS = OFF_BIAS + NS * 4 * BSLOT;
    static constexpr int LOOP_BYTES = OFF_DS + 4 * DS_BYTES;
    // Where the K and V rows of a wave stand before the first step (WaveRows): in the slots that the first copies leave free, of
    // Q and dO rows, half a slot to a wave, or in the wave's own bias slot; else behind everything else.  (V beside an fp32
    // bias at D = 64: nowhere, there the lanes load it.  At D = 16, half a kilobyte to a wave, neither: us, LDS / own loads, fp32 for
    // all batches 32 x 12 pairs of 192 rows 18.8 / 17.2, 16 x 12 of 197 14.3 / 13.3, fp32 H=8 M=32 N=1024 5.6 / 5.3, 192 rows 21.4 / 20.0,
    // no bias B=12 H=16 S=577 causal 21.8 / 20.9.)
    enum Stage { kHalfSlots, kBiasSlot, kBehind, kNowhere };
    static constexpr Stage K_STAGE = D == 16 ? kNowhere : ES == 4 ? kBiasSlot : kHalfSlots;
    static constexpr Stage V_STAGE = D == 16 ? kNowhere : ES == 4 ? (128 * D <= BSLOT ? kBiasSlot : kNowhere) : 64 * D <= BSLOT ? kBiasSlot : kBehind;
    static constexpr int LDS_BYTES = LOOP_BYTES + (V_STAGE == kBehind ? 256 * D : 0);
    static constexpr int MIN_BLOCKS = D <= 32 && ES <= 1 ? 3 : 2;  // work-groups per CU
    static_assert(LDS_BYTES * MIN_BLOCKS <= 163840, "LDS of a CU");
};

// An LDS address formed here: the compiler would add the constants of every access to it once per kernel, and keep them all
// in registers, instead of in the offset field.
__device__ __forceinline__ unsigned formed_here(unsigned addr) {
    asm volatile("" : "+v"(addr));
    return addr;
}

// The bias of a lane's key in the 16 rows of a block that the lane holds, from a row-major slice (32 keys per row);
// get(i): the additive term of register i, natural units for a float bias, log2 units (0 or the mask value) for bytes.
template <int BIAS> struct BiasBlock {
    __device__ __forceinline__ void load(unsigned, int) {}
    __device__ __forceinline__ float get(int) const { return 0.f; }
};
template <> struct BiasBlock<1> {
    i32x2 w[2];
    // ds_read_b64_tr_b8: within each group of 16 lanes, lane s supplies the address of 8 consecutive bytes, row s/2,
    // columns 8 (s%2) .. + 7 of an 8 x 16 matrix; lane i of the group receives its column i
    __device__ __forceinline__ void load(unsigned slice, int lane) {
        typedef i32x2 __attribute__((address_space(3))) * lds_ptr;
        const int row = ((lane & 15) >> 1), first = 4 * (lane >> 5) + (row & 3) + 8 * (row >> 2);
        const unsigned at = formed_here(slice + (unsigned)(first * 32 + 16 * ((lane >> 4) & 1) + 8 * (lane & 1)));
        w[0] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr)(uintptr_t)at);
        w[1] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr)(uintptr_t)(at + 16 * 32));
    }
    __device__ __forceinline__ float get(int i) const { return ((w[i >> 3][(i >> 2) & 1] >> (8 * (i & 3))) & 0xff) != 0 ? 0.f : kMask; }
};
template <typename V4> struct BiasBlock16 {
    i16x4 raw[4];
    __device__ __forceinline__ void load(unsigned slice, int lane) {
        const unsigned at = formed_here(slice + 2u * (unsigned)tr_offset(lane, 4 * (lane >> 5), 0, 32));
#pragma unroll
        for (int q4 = 0; q4 < 4; q4++) raw[q4] = lds_read_tr4_at(at + 512 * q4);
    }
    __device__ __forceinline__ float get(int i) const { return (float)__builtin_bit_cast(V4, raw[i >> 2])[i & 3]; }
};
template <> struct BiasBlock<2> : BiasBlock16<f16x4> {};
template <> struct BiasBlock<3> : BiasBlock16<bf16x4> {};
template <> struct BiasBlock<4> {
    unsigned at;  // (read where they are used: 16 registers more are not there)
    __device__ __forceinline__ void load(unsigned slice, int lane) { at = formed_here(slice + 512u * (unsigned)(lane >> 5) + 4u * (unsigned)(lane & 31)); }
    __device__ __forceinline__ float get(int i) const {
        typedef const float __attribute__((address_space(3))) * lds_ptr;
        return *(lds_ptr)(uintptr_t)(at + 128u * (unsigned)(8 * (i >> 2) + (i & 3)));
    }
};

// The same with the values in registers before they are used (an fp32 bias only: the others' are after load()).
template <int BIAS> struct BiasAhead : BiasBlock<BIAS> {
    __device__ __forceinline__ void fetch(const BiasBlock<BIAS>& from) { *static_cast<BiasBlock<BIAS>*>(this) = from; }
};
template <> struct BiasAhead<4> {
    float v[16];
    __device__ __forceinline__ void fetch(const BiasBlock<4>& from) {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = from.get(i);
    }
    __device__ __forceinline__ float get(int i) const { return v[i]; }
};

// Value that lane 16 (l / 16) + i holds, for lane l: a modifier of the instruction that uses it, no instruction of its own.
template <int I> __device__ __forceinline__ float row_bcast(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + I, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_bcast(float x, int i) {
    switch (i) {
#define FA_LANE(I) case I: return row_bcast<I>(x);
        FA_LANE(0) FA_LANE(1) FA_LANE(2) FA_LANE(3) FA_LANE(4) FA_LANE(5) FA_LANE(6) FA_LANE(7)
        FA_LANE(8) FA_LANE(9) FA_LANE(10) FA_LANE(11) FA_LANE(12) FA_LANE(13) FA_LANE(14)
#undef FA_LANE
    }
    return row_bcast<15>(x);
}

// DBIAS as in fa_bwd_kernel: 0 = the bias is not trainable; 1 = dBias is written densely (its rows allow aligned 16-byte
// accesses, and those of the bias come by copies, of 16 bytes or of 4: fa_bwd_kernel takes the others); 2 = reduced: the sums of dS over the query rows, or (ALiBi) the slope's
// gradient, one fp32 per (batch, head, key tile, wave).
template <typename T, int D, int BIAS, bool CAUSAL, int DBIAS>
__global__ __launch_bounds__(256, (NarrowCfg<D, tile_kind(BIAS)>::MIN_BLOCKS)) void fa_bwd_narrow_kernel(const BwdParams p) {
    constexpr int TB = tile_kind(BIAS);
    typedef NarrowCfg<D, TB> C;
    typedef Swz<D> SW;
    typedef typename VecOf<T>::v8 T8;
    typedef typename VecOf<T>::v4 T4;
    typedef typename BiasElem<TB>::type E;
    constexpr int SR = C::SR, NB = C::NB, LA = C::LA, BN = C::BN;
    constexpr bool DB16 = DBIAS == 1 && C::ES == 2, DB32 = DBIAS == 1 && C::ES == 4;
    constexpr bool NATURAL = BIAS >= 2 && BIAS != 7;  // the bias term is in natural units (else log2 units)

    __shared__ __align__(1024) unsigned char smem[C::LDS_BYTES];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 31, g = lane >> 5;
    const unsigned lds_base = lds_addr_of(smem);

    int nt, bh;
    decode_block<CAUSAL, C>(blockIdx.x, p.n_ntiles, p.B * p.H, nt, bh);
    const int b = bh / p.H, h = bh % p.H;
    const int M = p.M, N = p.N;
    const int n0 = nt * BN, nw = n0 + wave * 32, my_n = nw + r;
    // A wave without keys only copies blocks for the others.  (Without K, V and results of its own, too, us: D=64 64 x 12 pairs of 50
    // keys causal, no bias 13.2 -> 12.4, bf16 14.0 -> 13.2, B=2 H=2 33 keys 6.5 -> 6.0.)
    const bool live = nw < N;

    const T* qp = reinterpret_cast<const T*>(p.q) + (int64_t)b * p.sq.b + (int64_t)h * p.sq.h;
    const T* kp = reinterpret_cast<const T*>(p.k) + (int64_t)b * p.sk.b + (int64_t)h * p.sk.h;
    const T* vp = reinterpret_cast<const T*>(p.v) + (int64_t)b * p.sv.b + (int64_t)h * p.sv.h;
    const T* dop = reinterpret_cast<const T*>(p.dout) + (int64_t)b * p.sdo.b + (int64_t)h * p.sdo.h;
    // waves 0 and 1 copy the LSE of a step, waves 2 and 3 its delta
    const float* statp = (wave < 2 ? p.lse : p.delta) + ((int64_t)b * p.H + h) * M;
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
    if ((BIAS == 6 || BIAS == 7) && my_n < N) {
        const int64_t idx = (int64_t)b * p.sbias.b + (int64_t)h * p.sbias.h + (int64_t)my_n * p.sbias.n;
        switch (p.row_bias_kind) {
            case 1: row_bv = reinterpret_cast<const unsigned char*>(p.bias)[idx] ? 0.f : kMask; break;
            case 2: row_bv = (float)reinterpret_cast<const _Float16*>(p.bias)[idx]; break;
            case 3: row_bv = (float)reinterpret_cast<const __bf16*>(p.bias)[idx]; break;
            default: row_bv = reinterpret_cast<const float*>(p.bias)[idx]; break;
        }
    }

    // K and V of this wave's keys as B operands (column my_n, k = d), through LDS with the first copies (WaveRows).  With this and
    // the way back at the end, us, before -> after: padding mask B=32 H=12 S=197 D=64 25.6 -> 21.9, with an fp32 table 31.1 ->
    // 27.6, B=8 H=16 S=257 D=80 22.1 -> 19.3, B=4 H=16 S=2048 D=64 causal 81.6 -> 78.2, B=4 H=32 M=N=4096 1105 -> 1078.
    typedef WaveRows<T, D> WR;
    constexpr bool K_STAGED = C::K_STAGE != C::kNowhere, V_STAGED = C::V_STAGE != C::kNowhere;
    static_assert(K_STAGED || !V_STAGED, "V comes with K");
    T8 kreg[C::KSTEPS], vreg[C::KSTEPS];
    if constexpr (!V_STAGED) {
#pragma unroll
        for (int ks = 0; ks < C::KSTEPS; ks++) {
            i32x4 rv = {0, 0, 0, 0};
            const int d = ks * 16 + 8 * g;
            if constexpr (!K_STAGED) {
                i32x4 rk = {0, 0, 0, 0};
                if (my_n < N && d < p.d_qk) rk = gld16(kp + (int64_t)my_n * p.sk.s + d);
                kreg[ks] = as_vec<T8>(rk);
            }
            if (my_n < N && d < p.d_v) rv = gld16(vp + (int64_t)my_n * p.sv.s + d);
            vreg[ks] = as_vec<T8>(rv);
        }
    }
    // At head dim 96, up to 64 keys (half of a tile or less): the lanes' own loads and stores.  The longer ways to the first step and
    // from the last are all that such a call notices.  us, LDS / own: D=80 B=2 H=4 S=64 no bias 7.3 / 6.7,
    // causal 7.7 / 6.4, ALiBi 7.3 / 6.5, row mask 7.3 / 6.1, B=2 H=2 33 keys 7.0 / 6.1; 128 keys are even.  (At head dim 64 such calls gain 0.3
    // us and longer ones lose 1 %.)
    const bool few_keys = K_STAGED && D == 96 && N <= 64;
    f32x16 dk[C::DB], dv[C::DB];  // dK^T, dV^T: rows = head dim, column = my_n
#pragma unroll
    for (int db = 0; db < C::DB; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) dk[db][i] = dv[db][i] = 0.f;

    const float qk_scale = p.sm_scale * kLog2e;
    // causal: steps that end above the first key of this tile see none of its keys
    const int t0 = CAUSAL ? n0 / SR : 0, t_end = (M + SR - 1) / SR;
    constexpr bool BY_DWORD = TB == 4;

    // rows above the diagonal block of a wave are not visited and owe zeros to dBias
    if (DBIAS == 1 && CAUSAL) {
        const int rows_skipped = nw < M ? nw : M;
        for (int c = lane; c < rows_skipped * C::BCPR; c += 64) {
            const int m = c / C::BCPR, nn = nw + (c % C::BCPR) * C::EPC;
            E* dst = dbp + (int64_t)m * p.sdbias.m + nn;
            if (nn + C::EPC <= N) {
                gst16(dst, i32x4{0, 0, 0, 0});
            } else {
                for (int e = 0; e < C::EPC; e++)
                    if (nn + e < N) dst[e] = (E)0.f;
            }
        }
    }

    // ---- global -> LDS copies of a step: Q and dO rows, LSE and delta, this wave's bias slice.  Copy ci fills bytes
    // [1024 ci, 1024 ci + 1024) of a swizzled slot; every wave issues the same number in every step, completion is counted
    // (they complete in issue order).  Rows past M re-read the last row: p_value gives them zero. ----
    unsigned cq_off[C::QD], cdo_off[C::QD];
    int c_idx[C::QD];
#pragma unroll
    for (int i = 0; i < C::QD; i++) {
        c_idx[i] = (wave * C::QD + i) % C::NQD;
        const int c = c_idx[i] * 64 + lane;
        const int row = c / C::CPR, src = (c % C::CPR) ^ SW::f(row);
        cq_off[i] = (unsigned)(row * (int)p.sq.s * 2 + live_chunk(src, p.d_qk / 8) * 16);
        cdo_off[i] = (unsigned)(row * (int)p.sdo.s * 2 + live_chunk(src, p.d_v / 8) * 16);
    }
    const unsigned stat_dst = lds_base + C::OFF_STAT + (unsigned)(wave >> 1) * C::STAT_BYTES;
    const unsigned bias_dst = lds_base + C::OFF_BIAS + (unsigned)wave * C::BSLOT;
    auto slot_of = [&](int t) { return (unsigned)t % C::NS; };
    auto issue = [&](int t, auto bv_tag) {
        constexpr int BV = decltype(bv_tag)::value;
        const unsigned slot = slot_of(t);
        const int m0 = t * SR < M ? t * SR : M - 1;  // a step past the end is the last row over and over
        const uint64_t qb = uniform_ptr(qp + (int64_t)m0 * p.sq.s), dob = uniform_ptr(dop + (int64_t)m0 * p.sdo.s);
        const bool full = m0 + SR <= M;
#pragma unroll
        for (int i = 0; i < C::QD; i++) {
            unsigned oq = cq_off[i], od = cdo_off[i];
            if (!full) {
                // (rare: the lane index passes through an empty asm so that these per-lane values are
                // formed here and not kept in registers across the loops)
                int lane_here = lane;
                asm volatile("" : "+v"(lane_here));
                int over = (c_idx[i] * 64 + lane_here) / C::CPR - (M - 1 - m0);
                over = over > 0 ? over : 0;
                oq -= (unsigned)(over * (int)p.sq.s * 2);
                od -= (unsigned)(over * (int)p.sdo.s * 2);
            }
            lds_copy16(qb, oq, lds_base + slot * C::ROWS_BYTES + c_idx[i] * 1024);
            lds_copy16(dob, od, lds_base + C::OFF_DO + slot * C::ROWS_BYTES + c_idx[i] * 1024);
        }
        int m = t * SR + lane % SR;
        m = m < M ? m : M - 1;
        lds_copy4(uniform_ptr(statp), (unsigned)m * 4u, stat_dst + slot * 2 * C::STAT_BYTES);
        if constexpr (TB != 0) {
            if constexpr (BV == kByDword) {
                const uint64_t base = uniform_ptr(bp);
#pragma unroll
                for (int it = 0; it < 16; it++) {
                    int mb = t * SR + 2 * it + g;
                    mb = mb < M ? mb : M - 1;
                    lds_copy4(base, (unsigned)(((int64_t)mb * p.sbias.m + (my_n < N ? my_n : N - 1)) * 4), bias_dst + slot * 4 * C::BSLOT + it * 256);
                }
            } else if constexpr (BV == kByChunk) {
                const uint64_t base = uniform_ptr(bp);
#pragma unroll
                for (int it = 0; it < C::BCH; it++) {
                    const int c = it * 64 + lane;
                    int mb = t * SR + c / C::BCPR, nn = nw + (c % C::BCPR) * C::EPC;
                    mb = mb < M ? mb : M - 1;
                    nn = nn < N ? nn : 0;  // (such a lane's key does not exist: nothing of it is stored)
                    // a (batch, head) slice that takes this path is smaller than 2 GiB
                    lds_copy16(base, (unsigned)(((int64_t)mb * p.sbias.m + nn) * C::ES), bias_dst + slot * 4 * C::BSLOT + it * 1024);
                }
            }
        }
    };
    // Steps whose copies are whole walk the rows with running addresses in scalar registers, without clamps.
    uint64_t run_q = 0, run_do = 0, run_stat = 0, run_bias = 0;
    unsigned bias_off0 = 0;  // this lane's byte offset in the first bias copy of a step
    if constexpr (TB != 0) {
        int nn = nw + (lane % C::BCPR) * C::EPC;
        nn = nn < N ? nn : 0;
        bias_off0 = (unsigned)(((int64_t)(lane / C::BCPR) * p.sbias.m + nn) * C::ES);
        if (BY_DWORD && p.bias_vec == kByDword) bias_off0 = (unsigned)(((int64_t)g * p.sbias.m + (my_n < N ? my_n : N - 1)) * 4);
    }
    auto run_start = [&](int t) {
        run_q = uniform_ptr(qp + (int64_t)t * SR * p.sq.s);
        run_do = uniform_ptr(dop + (int64_t)t * SR * p.sdo.s);
        run_stat = uniform_ptr(statp + (int64_t)t * SR);
        if constexpr (TB != 0) run_bias = uniform_ptr(bp + (int64_t)t * SR * p.sbias.m);
    };
    auto issue_next = [&](int t, auto bv_tag) {
        settle_ptrs(run_q, run_do, run_stat);
        if constexpr (TB != 0) run_bias = uniform_ptr(reinterpret_cast<const void*>(run_bias));
        const unsigned slot = slot_of(t);
#pragma unroll
        for (int i = 0; i < C::QD; i++) {
            lds_copy16(run_q, cq_off[i], lds_base + slot * C::ROWS_BYTES + c_idx[i] * 1024);
            lds_copy16(run_do, cdo_off[i], lds_base + C::OFF_DO + slot * C::ROWS_BYTES + c_idx[i] * 1024);
        }
        unsigned lane_here = (unsigned)lane;
        asm volatile("" : "+v"(lane_here));
        lds_copy4(run_stat, (lane_here % SR) * 4u, stat_dst + slot * 2 * C::STAT_BYTES);
        run_q += (uint64_t)(SR * 2) * (uint64_t)p.sq.s;
        run_do += (uint64_t)(SR * 2) * (uint64_t)p.sdo.s;
        run_stat += SR * 4;
        if constexpr (TB != 0) {
            constexpr int N_COPIES = decltype(bv_tag)::value == kByDword ? 16 : C::BCH;
            const unsigned rows_step = (unsigned)(SR / N_COPIES * (int)p.sbias.m * C::ES);  // the rows one copy covers
#pragma unroll
            for (int it = 0; it < N_COPIES; it++) {
                if constexpr (N_COPIES == C::BCH) lds_copy16(run_bias, bias_off0 + it * rows_step, bias_dst + slot * 4 * C::BSLOT + it * 1024);
                else lds_copy4(run_bias, bias_off0 + it * rows_step, bias_dst + slot * 4 * C::BSLOT + it * 256);
            }
            run_bias += (uint64_t)(SR * C::ES) * (uint64_t)p.sbias.m;
        }
    };
    // bias rows that cannot be copied in aligned 16-byte chunks: element by element, 8 loads in flight together (as many as
    // there are registers for; clamped addresses, what lies outside the bias is masked or not stored)
    auto load_bias_scalar = [&](int t) {
        if constexpr (TB != 0) {
            E* dst = reinterpret_cast<E*>(smem + C::OFF_BIAS + (slot_of(t) * 4 + (unsigned)wave) * C::BSLOT);
            const int nn = my_n < N ? my_n : N - 1;
#pragma unroll 1
            for (int j0 = 0; j0 < 16 * NB; j0 += 8) {
                E vals[8];
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    int m = t * SR + 2 * (j0 + j) + g;
                    m = m < M ? m : M - 1;
                    vals[j] = bp[(int64_t)m * p.sbias.m + (int64_t)nn * p.sbias.n];
                }
#pragma unroll
                for (int j = 0; j < 8; j++) dst[(2 * (j0 + j) + g) * 32 + r] = vals[j];
            }
        }
    };

    // ---- where dBias goes.  16 bits: through a dS^T tile of the wave (8-byte stores of 4 rows of a key,
    // ds_read_b64_tr_b16 hands a lane 8 keys of a row).  fp32: over the bias values just read, whose place a lane's dS
    // takes, and out row by row.  Either way 16 bytes per lane. ----
    const unsigned ds_tile = lds_base + C::OFF_DS + (unsigned)wave * C::DS_BYTES;
    // lane -> row 16 ((lane/16)%2) + lane%16, keys 8 (lane/32 + 2 it) .. + 7 of the slice
    const int db_row = 16 * ((lane >> 4) & 1) + (lane & 15);
    const int db_src = 2 * ((8 * g + ((lane & 15) >> 2)) * C::DSS + 16 * ((lane >> 4) & 1) + 4 * (lane & 3));  // (bytes)
    // fp32: lane -> row 8 it + lane / 8, keys 4 (lane % 8) .. + 3, it = 0 .. 3
    const int db32_row = lane >> 3, db32_key = 4 * (lane & 7);
    // rows of whole aligned chunks leave through unconditional buffer stores (chunks outside the tensor get an offset
    // outside the view), so that the loop has no branch around its stores and can count them.  (16 bits: of rows that end inside a
    // chunk, all but the wave that holds the last keys; B=2 H=12 M=N=1001 D=32 34.6 -> 33.3 us.  fp32 there 48.4 -> 49.2, and the
    // pair of waves gains nothing: D=64 bf16 38.4 / 38.5, fp32 47.5 / 50.)
    const bool db_fast = DBIAS == 1 && (N % C::EPC == 0 || (DB16 && nw + 32 <= N));
    __amdgpu_buffer_rsrc_t db_rsrc = make_buffer(nullptr, 0);
    int db_off[2] = {0, 0};
    const int db_row_bytes = DBIAS == 1 ? (int)p.sdbias.m * C::ES : 0;
    if (DBIAS == 1 && db_fast) {
        db_rsrc = make_buffer(dbp, ((int64_t)(M - 1) * p.sdbias.m + N) * C::ES);
        if constexpr (DB32) {
            db_off[0] = nw + db32_key < N ? db32_row * db_row_bytes + (nw + db32_key) * 4 : (int)0x80000000;
        } else {
#pragma unroll
            for (int it = 0; it < 2; it++) {
                const int nn = nw + 8 * (g + 2 * it);
                db_off[it] = nn < N ? db_row * db_row_bytes + nn * 2 : (int)0x80000000;
            }
        }
    }
    constexpr int STORES = DB16 ? 2 * NB : DB32 ? 4 * NB : 0;  // dBias stores of a whole step
    float red_acc = 0.f;  // DBIAS == 2: this lane's share of the reduced gradient
    const unsigned rows_l = SW::rows_lane(lane), cols_l = SW::cols_lane(lane);

    auto run = [&](auto bv_tag, auto fast_tag) {
        constexpr int BV = decltype(bv_tag)::value;          // how bias slices come (BiasRows)
        constexpr bool DB_FAST = decltype(fast_tag)::value;
        constexpr int OPS = 2 * C::QD + 1 + (BV == kByElement ? 0 : BV == kByDword ? 16 : C::BCH);  // copies per wave and step
        {
            const unsigned free_slot = slot_of(t0 + LA);
            const unsigned half_slot = lds_base + (wave < 2 ? 0u : (unsigned)C::OFF_DO) + free_slot * C::ROWS_BYTES + (unsigned)(wave & 1) * WR::BYTES;
            const unsigned bias_slot = bias_dst + free_slot * 4 * C::BSLOT;
            const unsigned k_tile = C::K_STAGE == C::kBiasSlot ? bias_slot : half_slot;
            const unsigned v_tile = C::V_STAGE == C::kBehind ? lds_base + C::LOOP_BYTES + (unsigned)wave * WR::BYTES
                                                             : bias_slot + (C::K_STAGE == C::kBiasSlot ? WR::BYTES : 0);
            const unsigned saved_m0 = lds_copy_begin();
            if (few_keys) {
#pragma unroll
                for (int ks = 0; ks < C::KSTEPS; ks++) {
                    const int d = ks * 16 + 8 * g;
                    i32x4 rk = {0, 0, 0, 0}, rv = {0, 0, 0, 0};
                    if (my_n < N && d < p.d_qk) rk = gld16(kp + (int64_t)my_n * p.sk.s + d);
                    if (my_n < N && d < p.d_v) rv = gld16(vp + (int64_t)my_n * p.sv.s + d);
                    kreg[ks] = as_vec<T8>(rk);
                    vreg[ks] = as_vec<T8>(rv);
                }
            } else {
                if (K_STAGED && live) WR::issue(kp, p.sk.s, nw, N, k_tile, lane, [&](int c) { return live_chunk(c, p.d_qk / 8); });
                if (V_STAGED && live) WR::issue(vp, p.sv.s, nw, N, v_tile, lane, [&](int c) { return live_chunk(c, p.d_v / 8); });
            }
#pragma unroll
            for (int i = 0; i < LA; i++) issue(t0 + i, bv_tag);
            lds_copy_end(saved_m0);
            // (the compiler's own loads, too: left in flight, it would wait for everything in every step)
            WR::template arrived<0>();
            // (of a key past the end the last one again: nothing of such a lane is stored)
            if (!few_keys)
#pragma unroll
            for (int ks = 0; ks < C::KSTEPS; ks++) {
                const int d = ks * 16 + 8 * g;
                if constexpr (K_STAGED) {
                    const i32x4 rk = as_raw(SW::template row8_at<T8>(k_tile + rows_l, 0, ks));
                    kreg[ks] = as_vec<T8>(d < p.d_qk ? rk : i32x4{0, 0, 0, 0});
                }
                if constexpr (V_STAGED) {
                    const i32x4 rv = as_raw(SW::template row8_at<T8>(v_tile + rows_l, 0, ks));
                    vreg[ks] = as_vec<T8>(d < p.d_v ? rv : i32x4{0, 0, 0, 0});
                }
            }
        }
        int whole = 0;  // steps since one that may have stored less than STORES

        auto step = [&](int t, auto masked_tag, auto lean_tag) {
            constexpr bool MASKED = decltype(masked_tag)::value;  // some rows may be past M or above the diagonal
            constexpr bool LEAN = decltype(lean_tag)::value;      // the copies issued here are whole
            // the copies of step t were issued LA steps ago; later ones and the stores behind them may be in flight
            if constexpr (STORES > 0 && DB_FAST) {
                if (whole >= LA) wait_vmcnt<OPS*(LA - 1) + STORES * LA>();
                else wait_vmcnt<OPS*(LA - 1)>();
            } else {
                wait_vmcnt<OPS*(LA - 1)>();
            }
            lds_barrier();
            {
                const unsigned saved_m0 = lds_copy_begin();
                if constexpr (LEAN) issue_next(t + LA, bv_tag);
                else issue(t + LA, bv_tag);
                lds_copy_end(saved_m0);
            }
            whole = MASKED ? 0 : whole + 1;
            if (MASKED && !live) return;
            if constexpr (TB != 0 && BV == kByElement) load_bias_scalar(t);
            const unsigned slot = slot_of(t);
            const unsigned q_tile = lds_base + slot * C::ROWS_BYTES, do_tile = q_tile + C::OFF_DO;
            const float* stat = reinterpret_cast<const float*>(smem + C::OFF_STAT + slot * 2 * C::STAT_BYTES);
            const unsigned b_tile = lds_base + C::OFF_BIAS + (slot * 4 + (unsigned)wave) * C::BSLOT;

            // delta of the lane's rows: lane 16 j + i holds that of row 8 (i/4) + 4 (j/2) + i%4, and register i takes it from there
            auto load_delta = [&](int nb) { return stat[C::STAT_BYTES / 4 + nb * 32 + 8 * ((lane & 15) >> 2) + 4 * g + (lane & 3)]; };
            auto load_lse = [&](int nb, int q4) { return *reinterpret_cast<const f32x4*>(stat + nb * 32 + 8 * q4 + 4 * g); };
            // ---- P (flash_attention.py:281-294); register i is row m0 + 8 (i/4) + 4 g + i%4, the lane is key my_n.  Blocks
            // that touch the last rows or the causal diagonal follow the reference's additive -1.0e6 arithmetic term by
            // term, and rows past M have none; the others fold everything into one exponent.  (Keys past N need no mask:
            // nothing of them is stored.) ----
            auto p_value = [&](auto mk_tag, int m0, int i, float s, float lse, const auto& bias) {
                constexpr bool MK = decltype(mk_tag)::value;
                float bv = bias.get(i);
                if constexpr (BIAS == 5) bv = alibi_bias(neg_slope, ratio, (float)(m0 + 4 * g) + (float)(8 * (i >> 2) + (i & 3)), (float)my_n);
                if constexpr (BIAS == 6 || BIAS == 7) bv = row_bv;
                if constexpr (MK) {
                    const int m = m0 + 8 * (i >> 2) + 4 * g + (i & 3);
                    const float tmask = CAUSAL && m < my_n ? kMask : 0.f;
                    const float add = NATURAL ? __fmul_rn(bv, kLog2e) : bv;
                    const float pv = fast_exp2(__fadd_rn(__fmul_rn(s, qk_scale), __fadd_rn(tmask, add)) - lse);
                    return m < M ? pv : 0.f;  // (not an additive term: the LSE read again may lie below any)
                } else {
                    float off = BIAS == 0 ? -lse : (NATURAL ? __builtin_fmaf(bv, kLog2e, -lse) : bv - lse);
                    if constexpr (BIAS == 5) {  // distance of the lane's first row to its key, and from there to row i
                        const float dist0 = __builtin_fmaf((float)(m0 + 4 * g), ratio, -(float)my_n);
                        off = __builtin_fmaf(__builtin_fabsf(__builtin_fmaf((float)(8 * (i >> 2) + (i & 3)), ratio, dist0)), log2_slope, -lse);
                    }
                    return fast_exp2(__builtin_fmaf(s, qk_scale, off));
                }
            };
            auto reduce = [&](int m0, int i, float dsv) {
                // (rows past M have P = 0 exactly, hence dS = 0)
                if constexpr (DBIAS == 2 && BIAS == 5)  // d bias / d slope = -|i N / M - j|
                    red_acc -= dsv * __builtin_fabsf(__builtin_fmaf((float)(m0 + 4 * g) + (float)(8 * (i >> 2) + (i & 3)), ratio, -(float)my_n));
                else if constexpr (DBIAS == 2) red_acc += dsv;
            };
            auto store_dbias = [&](int nb, int m0) {
                if constexpr (DB16) {
                    const unsigned at = formed_here(ds_tile + (unsigned)db_src);
#pragma unroll
                    for (int it = 0; it < 2; it++) {
                        const i16x4 lo = lds_read_tr4_at(at + it * 32 * C::DSS), hi = lds_read_tr4_at(at + it * 32 * C::DSS + 8 * C::DSS);
                        typedef short i16x8 __attribute__((ext_vector_type(8)));
                        const i32x4 v = __builtin_bit_cast(i32x4, (i16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                        const int m = m0 + db_row, nn = nw + 8 * (g + 2 * it);
                        if constexpr (DB_FAST) {
                            buf_store16(db_rsrc, v, !MASKED || m < M ? db_off[it] + m0 * db_row_bytes : (int)0x80000000);
                        } else if (m < M && nn < N) {
                            E* dst = dbp + (int64_t)m * p.sdbias.m + nn;
                            if (nn + 8 <= N) {
                                gst16(dst, v);
                            } else {
#pragma unroll
                                for (int e = 0; e < 8; e++)
                                    if (nn + e < N) dst[e] = __builtin_bit_cast(E, (short)(v[e >> 1] >> (16 * (e & 1))));
                            }
                        }
                    }
                }
                if constexpr (DB32) {
                    const unsigned at = formed_here(b_tile + nb * C::BBLOCK + 128u * (unsigned)db32_row + 4u * (unsigned)db32_key);
#pragma unroll
                    for (int it = 0; it < 4; it++) {
                        const int row = 8 * it + db32_row;
                        const f32x4 w = __builtin_bit_cast(f32x4, lds_read16_at(at + it * 1024));
                        const int m = m0 + row, nn = nw + db32_key;
                        if constexpr (DB_FAST) {
                            buf_store16(db_rsrc, __builtin_bit_cast(i32x4, w), !MASKED || m < M ? db_off[0] + (m0 + 8 * it) * db_row_bytes : (int)0x80000000);
                        } else if (m < M && nn < N) {
                            float* dst = reinterpret_cast<float*>(dbp) + (int64_t)m * p.sdbias.m + nn;
                            if (nn + 4 <= N) {
                                gst16(dst, __builtin_bit_cast(i32x4, w));
                            } else {
#pragma unroll
                                for (int e = 0; e < 4; e++)
                                    if (nn + e < N) dst[e] = w[e];
                            }
                        }
                    }
                }
            };

            // Steps in the middle of a tile, D = 64 without a bias tile: the matrix instructions of one block are issued
            // between the exponentials and the dS arithmetic of the other, their operands fetched a phase ahead.
            if constexpr (!MASKED && NB == 2 && D == 64 && TB == 0 && !(BIAS == 5 && DBIAS == 2)) {
                constexpr int KS = C::KSTEPS, NP = 2 * C::DB;
                auto fence = []() { __builtin_amdgcn_sched_barrier(0); };
                T8 q_op[KS], do_op[KS], do_col[NP], q_col[NP];
                f32x16 s[2], dp[2];
                float del[2], pf[16];
                f32x4 lse[4];
                T8 pb[2], ds[2];
                const BiasBlock<BIAS> no_bias{};
                const int m0 = t * SR;
                auto load_rows = [&](int nb) {
#pragma unroll
                    for (int i = 0; i < KS; i++) q_op[i] = SW::template row8_at<T8>(q_tile + rows_l, nb * 32, i);
#pragma unroll
                    for (int i = 0; i < KS; i++) do_op[i] = SW::template row8_at<T8>(do_tile + rows_l, nb * 32, i);
                };
                auto load_cols = [&](unsigned tile, int nb, T8 (&a)[NP]) {
#pragma unroll
                    for (int i = 0; i < NP; i++) a[i] = SW::template col8_at<T8>(tile + cols_l, nb * 32 + (i / C::DB) * 16, i % C::DB);
                };
                auto load_stat = [&](int nb) {
                    del[nb] = load_delta(nb);
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) lse[q4] = load_lse(nb, q4);
                };
                // the exponentials (dS) of a block, two elements at a time, between(j) behind pair j of 8
                auto exps = [&](int nb, auto&& between) {
#pragma unroll
                    for (int j = 0; j < 8; j++) {
#pragma unroll
                        for (int i = 2 * j; i < 2 * j + 2; i++) {
                            pf[i] = p_value(std::false_type{}, m0 + 32 * nb, i, s[nb][i], lse[i >> 2][i & 3], no_bias);
                            pb[i >> 3][i & 7] = (T)pf[i];
                        }
                        fence();
                        between(j);
                        fence();
                    }
                };
                auto dss = [&](int nb, auto&& between) {
#pragma unroll
                    for (int j = 0; j < 8; j++) {
#pragma unroll
                        for (int i = 2 * j; i < 2 * j + 2; i++) {
                            const float dsv = pf[i] * (dp[nb][i] - row_bcast(del[nb], i));
                            ds[i >> 3][i & 7] = (T)dsv;
                            reduce(m0 + 32 * nb, i, dsv);
                        }
                        fence();
                        between(j);
                        fence();
                    }
                };
                auto mma_dv = [&](int j) {  // slot j of 8
#pragma unroll
                    for (int i = j * NP / 8; i < (j + 1) * NP / 8; i++) dv[i % C::DB] = mfma32(do_col[i], pb[i / C::DB], dv[i % C::DB]);
                };
                auto mma_dk = [&](int j) {
#pragma unroll
                    for (int i = j * NP / 8; i < (j + 1) * NP / 8; i++) dk[i % C::DB] = mfma32(q_col[i], ds[i / C::DB], dk[i % C::DB]);
                };
#pragma unroll
                for (int nb = 0; nb < 2; nb++)
#pragma unroll
                    for (int i = 0; i < 16; i++) s[nb][i] = dp[nb][i] = 0.f;
                load_rows(0);
                load_stat(0);
#pragma unroll
                for (int i = 0; i < KS; i++) s[0] = mfma32(q_op[i], kreg[i], s[0]);
#pragma unroll
                for (int i = 0; i < KS; i++) dp[0] = mfma32(do_op[i], vreg[i], dp[0]);
                load_rows(1);
                load_cols(do_tile, 0, do_col);
                fence();
                exps(0, [&](int j) {
#pragma unroll
                    for (int i = j * KS / 4; i < (j + 1) * KS / 4; i++) {
                        if (i < KS) s[1] = mfma32(q_op[i], kreg[i], s[1]);
                        else dp[1] = mfma32(do_op[i - KS], vreg[i - KS], dp[1]);
                    }
                });
                load_cols(q_tile, 0, q_col);
                load_stat(1);
                fence();
                dss(0, mma_dv);
                load_cols(do_tile, 1, do_col);
                fence();
                exps(1, mma_dk);
                load_cols(q_tile, 1, q_col);
                fence();
                dss(1, mma_dv);
#pragma unroll
                for (int j = 0; j < 8; j++) mma_dk(j);
                return;
            }

#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
                const int m0 = t * SR + nb * 32;
                __builtin_amdgcn_sched_barrier(0);  // keep the blocks apart
                if (MASKED && ((CAUSAL && m0 + 31 < nw) || m0 >= M)) continue;
                const bool need_mask = MASKED && (m0 + 32 > M || (CAUSAL && m0 < nw + 31));
                // Up to head dim 32 there are registers for everything that a block reads from LDS, fetched ahead of where it is
                // used: operands of the first two products, then, under them, LSE, bias and the operands of the other two.  Left to
                // the compiler, each read waited for the one before it in some of these kernels.  us, before -> after: D=32, fp32 and
                // dBias B=2 H=12 M=N=1024 39.1 -> 36.2, B=8 154.8 -> 141.2; bf16 and dBias B=2 30.7 -> 29.5, causal H=8 28.0 -> 26.6;
                // fp32 read B=16 H=8 M=N=256 10.6 -> 10.2; D=16, fp32 and dBias 38.0 -> 36.5.  (A 16-bit tile at D=16 has
                // registers for three work-groups on a CU without them and for two with them.  Fetched ahead / not: read only, B=8 H=12
                // M=N=1024 50.5 / 46, 16 x 12 pairs of 576 rows 36.8 / 33.7; dBias, 32 x 12 pairs of 192 rows 22.6 / 19.6, causal 23.6 /
                // 19.7, but where few tiles end alone H=16 M=N=1024 29.1 / 29.4, B=12 H=16 S=577 77.9 / 77.3, B=8 H=12 2048 355 / 374.)
                constexpr bool AHEAD = C::MIN_BLOCKS == 2 && (D == 32 || (D == 16 && C::ES == 4));
                constexpr bool BIAS_AHEAD = AHEAD || (D == 64 && TB == 4 && DBIAS == 0);  // (16 registers)
                constexpr int NP = 2 * C::DB;
                auto fence = [&]() {
                    if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
                };
                T8 q_op[C::KSTEPS], do_op[C::KSTEPS], do_col[NP], q_col[NP];
                f32x4 lse_ahead[4];
                BiasBlock<BIAS> bias;
                BiasAhead<BIAS> bias_ahead;
                const float del = load_delta(nb);
                f32x16 s, dp;
#pragma unroll
                for (int i = 0; i < 16; i++) s[i] = dp[i] = 0.f;
                if constexpr (AHEAD) {
#pragma unroll
                    for (int ks = 0; ks < C::KSTEPS; ks++) q_op[ks] = SW::template row8_at<T8>(q_tile + rows_l, nb * 32, ks);
#pragma unroll
                    for (int ks = 0; ks < C::KSTEPS; ks++) do_op[ks] = SW::template row8_at<T8>(do_tile + rows_l, nb * 32, ks);
                    fence();
#pragma unroll
                    for (int ks = 0; ks < C::KSTEPS; ks++) s = mfma32(q_op[ks], kreg[ks], s);
#pragma unroll
                    for (int ks = 0; ks < C::KSTEPS; ks++) dp = mfma32(do_op[ks], vreg[ks], dp);
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) lse_ahead[q4] = load_lse(nb, q4);
                    bias.load(b_tile + nb * C::BBLOCK, lane);
                    bias_ahead.fetch(bias);
#pragma unroll
                    for (int i = 0; i < NP; i++) {
                        do_col[i] = SW::template col8_at<T8>(do_tile + cols_l, nb * 32 + (i / C::DB) * 16, i % C::DB);
                        q_col[i] = SW::template col8_at<T8>(q_tile + cols_l, nb * 32 + (i / C::DB) * 16, i % C::DB);
                    }
                    fence();
                } else {
#pragma unroll
                    for (int ks = 0; ks < C::KSTEPS; ks++) s = mfma32(SW::template row8_at<T8>(q_tile + rows_l, nb * 32, ks), kreg[ks], s);
#pragma unroll
                    for (int ks = 0; ks < C::KSTEPS; ks++) dp = mfma32(SW::template row8_at<T8>(do_tile + rows_l, nb * 32, ks), vreg[ks], dp);
                    bias.load(b_tile + nb * C::BBLOCK, lane);
                    if constexpr (BIAS_AHEAD) {
                        bias_ahead.fetch(bias);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                T8 pb[2], ds[2];
                auto elements = [&](auto mk_tag) {
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) {
                        const f32x4 lse = AHEAD ? lse_ahead[q4] : load_lse(nb, q4);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const int i = q4 * 4 + e;
                            float pv;
                            if constexpr (BIAS_AHEAD) pv = p_value(mk_tag, m0, i, s[i], lse[e], bias_ahead);
                            else pv = p_value(mk_tag, m0, i, s[i], lse[e], bias);
                            pb[i >> 3][i & 7] = (T)pv;
                            dp[i] = pv * (dp[i] - row_bcast(del, i));  // dS (flash_attention.py:303-308)
                            ds[i >> 3][i & 7] = (T)dp[i];
                            reduce(m0, i, dp[i]);
                        }
                    }
                };
                if constexpr (MASKED) {
                    if (need_mask) elements(std::true_type{});
                    else elements(std::false_type{});
                } else {
                    elements(std::false_type{});
                }
                if constexpr (DB16) {
                    typedef typename VecOf<E>::v4 E4;
                    typedef E4 __attribute__((address_space(3))) * lds_ptr;
                    const unsigned at = formed_here(ds_tile + (unsigned)(2 * (r * C::DSS + 4 * g)));
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) {
                        E4 d4;
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            if constexpr (__is_same(T, E)) d4[e] = ds[q4 >> 1][(q4 & 1) * 4 + e];
                            else d4[e] = (E)dp[q4 * 4 + e];
                        }
                        *(lds_ptr)(uintptr_t)(at + 16 * q4) = d4;
                    }
                }
                if constexpr (DB32) {
                    typedef float __attribute__((address_space(3))) * lds_ptr;
#pragma unroll
                    for (int i = 0; i < 16; i++) *(lds_ptr)(uintptr_t)(bias.at + 128u * (unsigned)(8 * (i >> 2) + (i & 3))) = dp[i];
                }
                store_dbias(nb, m0);
#pragma unroll
                for (int kk = 0; kk < 2; kk++)
#pragma unroll
                    for (int db = 0; db < C::DB; db++) {
                        if constexpr (!AHEAD) {
                            do_col[kk * C::DB + db] = SW::template col8_at<T8>(do_tile + cols_l, nb * 32 + kk * 16, db);
                            q_col[kk * C::DB + db] = SW::template col8_at<T8>(q_tile + cols_l, nb * 32 + kk * 16, db);
                        }
                        dv[db] = mfma32(do_col[kk * C::DB + db], pb[kk], dv[db]);
                        dk[db] = mfma32(q_col[kk * C::DB + db], ds[kk], dk[db]);
                    }
            }
        };

        // steps in the middle of the tile: below the diagonal of all of its keys, every row of the step and of the copies
        // issued in it exists
        int t_in = CAUSAL ? (n0 + BN - 1 + SR - 1) / SR : t0;
        t_in = t_in < t_end ? t_in : t_end;
        int t_out = M / SR - LA;
        if ((TB != 0 && BV == kByElement) || !live || t_out < t_in) t_out = t_in;
        // (two passes over ONE copy of the general loop, the others between them)
        int t = t0, stop = t_in;
#pragma unroll 1
        for (int pass = 0; pass < 2; pass++) {
#pragma unroll 1
            for (; t < stop; t++) step(t, std::true_type{}, std::false_type{});
            if (pass == 0 && t < t_out) {
                run_start(t + LA);
#pragma unroll 1
                for (; t < t_out; t++) step(t, std::false_type{}, std::true_type{});
            }
            stop = t_end;
        }
        wait_vmcnt<0>();  // nothing may land in LDS once the work-group is gone
    };
    auto run_rows = [&](auto fast_tag) {
        if constexpr (TB == 0) {
            run(RowsTag<kByElement>{}, fast_tag);
        } else {
            if constexpr (BY_DWORD && DBIAS == 1) {
                if (p.bias_vec == kByDword) run(RowsTag<kByDword>{}, fast_tag);
                else run(RowsTag<kByChunk>{}, fast_tag);
            } else if constexpr (DBIAS == 1) {
                run(RowsTag<kByChunk>{}, fast_tag);
            } else if constexpr (BY_DWORD) {
                if (p.bias_vec == kByChunk) run(RowsTag<kByChunk>{}, fast_tag);
                else if (p.bias_vec == kByDword) run(RowsTag<kByDword>{}, fast_tag);
                else run(RowsTag<kByElement>{}, fast_tag);
            } else {
                if (p.bias_vec == kByChunk) run(RowsTag<kByChunk>{}, fast_tag);
                else run(RowsTag<kByElement>{}, fast_tag);
            }
        }
    };
    if constexpr (DBIAS == 1) {
        if (db_fast) run_rows(std::true_type{});
        else run_rows(std::false_type{});
    } else {
        run_rows(std::false_type{});
    }

    if constexpr (DBIAS == 2 && BIAS == 5) {
        // slope gradient of this wave's 32 keys, summed over the lanes in a fixed order
        float s = my_n < N ? red_acc : 0.f;
#pragma unroll
        for (int w = 32; w >= 1; w >>= 1) s += __shfl_xor(s, w, 64);
        if (lane == 0) p.partials[((int64_t)bh * p.n_ntiles + nt) * 4 + wave] = s;
    } else if constexpr (DBIAS == 2) {
        // column sums: lanes l and l + 32 hold different rows of the same key
        const float s = pair_sum(red_acc);
        if (g == 0 && my_n < N) p.partials[(int64_t)bh * N + my_n] = s;
    }
    // ---- dV and dK of this wave's keys (flash_attention.py:449-454) ----
    T* dvp = reinterpret_cast<T*>(p.dv) + (int64_t)b * p.sdv.b + (int64_t)h * p.sdv.h;
    T* dkp = reinterpret_cast<T*>(p.dk) + (int64_t)b * p.sdk.b + (int64_t)h * p.sdk.h;
    if (few_keys) {
        if (my_n < N) {
#pragma unroll
            for (int db = 0; db < C::DB; db++)
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const int d = db * 32 + 8 * q4 + 4 * g;
                    T4 v4, k4;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        v4[e] = (T)dv[db][q4 * 4 + e];
                        k4[e] = (T)(dk[db][q4 * 4 + e] * p.sm_scale);
                    }
                    if (d < p.d_v) *reinterpret_cast<T4*>(dvp + (int64_t)my_n * p.sdv.s + d) = v4;
                    if (d < p.d_qk) *reinterpret_cast<T4*>(dkp + (int64_t)my_n * p.sdk.s + d) = k4;
                }
        }
        return;
    }
    lds_barrier();  // (the rings are dead and no copy is in flight)
    static_assert(8 * WR::BYTES <= C::LDS_BYTES, "room for the way back");
    if (!live) return;
    const unsigned own = lds_base + 2u * (unsigned)wave * WR::BYTES;
    WR::store(dv, 1.f, own, dvp, p.sdv.s, nw, N, p.d_v, lane);
    WR::store(dk, p.sm_scale, own + WR::BYTES, dkp, p.sdk.s, nw, N, p.d_qk, lane);
}

// This file is compiled once per head dimension (-DFA_HEAD_DIM=16, 32, 64, 96); each object exports
// launch_bwd_narrow_d<FA_HEAD_DIM>.  bias: 0 ... 7, dbias: 0, 1 or 2, as the kernel takes them.
#ifndef FA_HEAD_DIM
#error "compile with -DFA_HEAD_DIM=<16|32|64|96>"
#endif
template <typename T, int BIAS, int DBIAS> static hipError_t launch_one(const BwdParams& p, bool causal, hipStream_t st) {
    const dim3 grid((unsigned)(p.n_ntiles * p.B * p.H));
    if (causal) hipLaunchKernelGGL((fa_bwd_narrow_kernel<T, FA_HEAD_DIM, BIAS, true, DBIAS>), grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL((fa_bwd_narrow_kernel<T, FA_HEAD_DIM, BIAS, false, DBIAS>), grid, dim3(256), 0, st, p);
    return hipGetLastError();
}
template <typename T> static hipError_t launch_typed(const BwdParams& p, int bias, bool causal, int dbias, hipStream_t st) {
#define FA_CASE(B, DB) \
    if (bias == B && dbias == DB) return launch_one<T, B, DB>(p, causal, st);
    FA_CASE(0, 0)
    FA_CASE(5, 0)
    FA_CASE(5, 2)
    FA_CASE(6, 0)
    FA_CASE(6, 2)
    FA_CASE(7, 0)
#if FA_HEAD_DIM <= 64
    // (at 96 there are no registers for a bias tile: fa_bwd_kernel at 128 takes those)
    FA_CASE(1, 0)
    FA_CASE(2, 0)
    FA_CASE(2, 1)
    FA_CASE(2, 2)
    FA_CASE(3, 0)
    FA_CASE(3, 1)
    FA_CASE(3, 2)
    FA_CASE(4, 0)
    FA_CASE(4, 1)
    FA_CASE(4, 2)
#endif
#undef FA_CASE
    return hipErrorInvalidValue;
}
template <int D> hipError_t launch_bwd_narrow_d(const BwdParams& p, int dtype, int bias, bool causal, int dbias, hipStream_t st);
template <> hipError_t launch_bwd_narrow_d<FA_HEAD_DIM>(const BwdParams& p, int dtype, int bias, bool causal, int dbias, hipStream_t st) {
    if (dbias == 1 && !(p.bias_vec && p.dbias_vec)) return hipErrorInvalidValue;  // (fa_bwd_kernel's)
    return dtype == 0 ? launch_typed<_Float16>(p, bias, causal, dbias, st) : launch_typed<__bf16>(p, bias, causal, dbias, st);
}

}  // namespace fa
