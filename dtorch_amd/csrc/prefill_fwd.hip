// Flash-style attention forward for gfx950 (bf16 / fp16 MFMA), with per-row LSE.
//
// Replaces the arithmetic of SdpaOp::Compute (the libtorch call at
// dtorch/core/operators/standard/scaled_dot_product_attention_op.cc:107-109) on the GPU.
//
// Work decomposition
//   One workgroup = 4 waves = 4*QT*32 consecutive query rows of one (batch, query head).  Each wave
//   owns QT tiles of 32 queries and keeps their Q fragments in registers for the whole kernel.
//   Key/value tiles of 64 rows are staged through LDS and shared by the 4 waves.
//
// Layout trick
//   The score tile is computed transposed, S^T = K Q^T, with v_mfma_f32_32x32x16_{bf16,f16}: the
//   accumulator column (lane % 32) is the query, so each lane holds 16 keys of one query row and the
//   row max needs one cross-half exchange (v_permlane32_swap) instead of a 32-lane reduction.  The
//   output is accumulated transposed as well, O^T = V^T P^T: P^T comes straight from the score
//   registers (the MFMA reduction index is a free permutation, matched on both operands), and the V^T
//   operand is read from the row-major V tile with ds_read_b64_tr_b16 (LDS transpose read).  The
//   per-query rescale factor is then a per-lane scalar.
//
// LDS: K and V tiles of 64 rows, double-buffered, filled by direct buffer->LDS loads (no VGPR
// staging); 16-byte chunk c of row r sits at chunk c ^ kswz(r), which keeps both the 16-byte K reads
// and the 8-byte transposed V reads free of bank conflicts.
//
// Pipeline per key tile j (one barrier per tile):
//   wait own loads + barrier | K[j+1], V[j+1] -> LDS (async) | S^T = K[j] Q^T | softmax |
//   O^T += V^T(j) P^T(j)
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "dtattn_common.hpp"
#include "prefill_params.hpp"

namespace dtattn {

// XOR swizzle of the 16-byte chunk index of LDS row r (K and V tiles).  It is distinct over any 16
// consecutive rows (the 16-byte K reads take one chunk of 16 rows per step) and differs above the
// low two bits for 4 consecutive rows (a transposed V read takes 4 aligned chunks of 4 rows).  With
// 128-byte rows (D = 64) two rows share a 256-byte bank row, so the pattern is applied per row pair.
template <int D>
__device__ __forceinline__ int kswz(int r) {
    return D >= 128 ? 4 * (r & 3) + ((r >> 2) & 3) : 4 * ((r >> 1) & 1) + ((r >> 2) & 3);
}

// PAD: the real head dims are below D (any multiple of 8, Dv may differ from D); Q/K chunks past
// p.qk_ch and V chunks past p.v_ch load as zeros, and O chunks past p.v_ch are not stored.
// KG: key groups, 1 or 2.  KG * 4 waves share the 128 query rows, group g takes key tiles g, g + KG, ... through its own
// LDS buffers, and the groups' (O, max, sum) are merged in fp32 through LDS: for grids that leave CUs idle otherwise.
// SUMC: the row max only where the sums of P ask for it (below).
template <typename T, int D, int QT, bool CAUSAL, int MASKED, bool PAD, int KG, bool SUMC>
__global__ void __launch_bounds__(256 * KG, 2) prefill_fwd_kernel(const PrefillParams p) {
    static_assert(KG == 1 || KG == 2, "the merge holds one more group");
    constexpr int NW = 4;
    constexpr int BN = 64;
    constexpr int BM = NW * 32;
    constexpr int DCH = D / 8;            // 16-byte chunks per row
    constexpr int KSTEPS = D / 16;        // MFMA k-steps of S^T = K Q^T
    constexpr int DT = D / 32;            // 32-row d tiles of O^T
    constexpr int KT = BN / 32;           // 32-key tiles per key block
    constexpr int PVS = BN / 16;          // MFMA k-steps of O^T = V^T P^T
    static_assert(QT == 1, "one 32-query tile per wave");
    typedef typename Elem<T>::vec8 V8;
    typedef typename Elem<T>::vec4 V4;
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

    // K and V tiles, double-buffered, each [64 keys][D] with 16-byte chunk c of row r at c ^ kswz(r).
    // Four distinct LDS objects so the compiler's alias analysis can tell an in-flight load into one
    // buffer from the reads of the others.
    __shared__ __attribute__((aligned(16))) T Ka_[KG * BN * D];
    __shared__ __attribute__((aligned(16))) T Kb_[KG * BN * D];
    __shared__ __attribute__((aligned(16))) T Va_[KG * BN * D];
    __shared__ __attribute__((aligned(16))) T Vb_[KG * BN * D];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);  // wave-uniform: LDS bases stay scalar
    const int kg = KG > 1 ? __builtin_amdgcn_readfirstlane(tid >> 8) : 0;
    T* const Ka = Ka_ + kg * BN * D;
    T* const Kb = Kb_ + kg * BN * D;
    T* const Va = Va_ + kg * BN * D;
    T* const Vb = Vb_ + kg * BN * D;
    const int l32 = lane & 31;
    const int hf = lane >> 5;

    const BlockCoord bc = block_coord<CAUSAL>(p);
    const int qb = bc.qb, b = bc.b, hq = bc.hq, hk = bc.hk;
    if constexpr (MASKED != kMaskNone)
        if (p.spans != nullptr && p.spans[b].y >= 0) return;  // run as a key span (prefill_rows64.hip)

    const T* qp = reinterpret_cast<const T*>(p.q) + b * p.qs_b + hq * p.qs_h;
    const T* kp = reinterpret_cast<const T*>(p.k) + b * p.ks_b + hk * p.ks_h;
    const T* vp = reinterpret_cast<const T*>(p.v) + b * p.vs_b + hk * p.vs_h;

    const int q0 = qb * BM;
    const int wq0 = q0 + wave * 32;

    int kend = p.Sk;
    if (CAUSAL) {
        const int lim = q0 + BM + p.delta;  // keys < lim can be visible
        kend = lim < 0 ? 0 : (lim < p.Sk ? lim : p.Sk);
    }
    const int nt = (kend + BN - 1) / BN;

    V8 qf[KSTEPS];  // Q fragments (B operand of S^T = K Q^T), loaded after tile 0's loads are issued

    f32x16 oacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
    float mrow = kNegInf, lrow = 0.f;
    // The VALU work of the softmax, not the MFMAs, bounds head dim 64, and the row max is a tenth of it.  SUMC (non-causal
    // kernels without a mask) computes it only when it has to move: a tile is exponentiated with the max so far, and only
    // if some lane's sum of its 32 P then exceeds 2^8 (no sum up to it holds a P above the bound that the rescale rule
    // keeps) are the row max, the rescale and the exponentials done over; also while a row has no max yet.  2x24x4429
    // fp16 286 -> 271 us; with the causal or masked kernels' registers it cost 2-6%.  sum_check_pays() has the grids.
    static_assert(!SUMC || (D == 64 && !CAUSAL && MASKED == kMaskNone), "the kernels of the form");
    constexpr float kSumLimit = 256.f;  // 2^kRescaleThreshold
    bool fresh = true;

    const int krow = (int)(p.ks_s * (int64_t)sizeof(T));  // row pitch in bytes (< 2^25, host-checked)
    const int vrow = (int)(p.vs_s * (int64_t)sizeof(T));

    // Tile t of K or V -> LDS by direct buffer->LDS loads: one wave instruction fills 1 KB of LDS (lane
    // l -> byte 16*l), i.e. 1024/(2*D) rows, so lane l loads the global chunk that belongs at its LDS
    // slot, c = slot ^ kswz(row).  The buffer resource covers the tile's valid rows; rows past Sk
    // read zeros, and so do chunks at or past valid_ch (PAD), whose offset is the resource's size.
    auto dma = [&](T* dst, const T* base, int pitch, int64_t stride, int t, int valid_ch) {
        constexpr int ROWS_PER_INSTR = 1024 / (2 * D);
        constexpr int INSTR = BN / ROWS_PER_INSTR / NW;  // per wave
        const int rows = min(BN, p.Sk - t * BN);
        // the resource ends where the tile's last valid row ends (its real width under PAD)
        const uint32_t nbytes = (uint32_t)((rows - 1) * pitch + (PAD ? valid_ch * 16 : D * (int)sizeof(T)));
        const auto rs = make_rsrc(base + (int64_t)t * BN * stride, nbytes);
#pragma unroll
        for (int i = 0; i < INSTR; ++i) {
            const int r0 = (wave * INSTR + i) * ROWS_PER_INSTR;
            const int r = r0 + lane / DCH;
            const int c = (lane % DCH) ^ kswz<D>(r);
            const uint32_t off = (PAD && c >= valid_ch) ? nbytes : (uint32_t)(r * pitch + c * 16);
            buf_ld16_lds_async(rs, dst + r0 * D, off);
        }
    };

    // V^T fragments for the PV MFMA come straight from the row-major V tile with ds_read_b64_tr_b16:
    // within each 16-lane block, lane 4j+a addresses key K0+j, d-segment D0+4a, and lane i then
    // receives V[K0..K0+3][D0+i] -- one d and four consecutive keys, the A-operand slot layout.
    const int blk = lane >> 4, bl = lane & 15;
    const int tr_key = bl >> 2;                 // j
    const int tr_d = 16 * (blk & 1) + 4 * (bl & 3);  // D0 offset within the 32-d tile + 4a
    const int tr_k4 = 4 * (blk >> 1);           // 4 * hf

    // MASKED: lane (l32, hf) reads, for query row wq0 + l32, the four consecutive keys of each of its 4 groups per
    // 32-key tile.
    const auto mslab = [&] {
        if constexpr (MASKED != kMaskNone) return MaskSlab<MASKED>(p, b, hq, wq0 + l32);
        else return 0;
    }();

    // One key tile.  Kc/Vc hold tile t; Kn/Vn receive the group's next tile.
    auto tile = [&](const T* Kc, const T* Vc, T* Kn, T* Vn, int t) {
        wait_vmem();
        lds_barrier();  // tile t landed everywhere; every wave finished tile t-1 (so Kn/Vn are free)
        auto next_tile = [&]() {
            if (t + KG < nt) {
                dma(Kn, kp, krow, p.ks_s, t + KG, p.qk_ch);
                dma(Vn, vp, vrow, p.vs_s, t + KG, p.v_ch);
            }
        };
        if (KG > 1 && t >= nt) return;  // a group's last round may be short
        // Issue point of the next tile's loads: at the tile start in the causal kernel; after this tile's
        // S block in the non-causal one (measured +2.5% at 256-512 keys, neutral on long rows; the causal
        // kernel would spill); masked kernels after the mask add (the compiler's wait for the mask values
        // would otherwise also wait for the tile loads).
        constexpr bool kLateLoads = MASKED != kMaskNone || !CAUSAL;
        if constexpr (!kLateLoads) next_tile();
        const int kbase = t * BN;
        if (CAUSAL && kbase > wq0 + 31 + p.delta) {  // every row of this wave precedes the tile
            if constexpr (kLateLoads) next_tile();
            return;
        }
        const bool need_mask = (kbase + BN > p.Sk) || (CAUSAL && (kbase + BN - 1 > wq0 + p.delta));
        typename MaskSlab<MASKED>::Group mraw[MASKED != kMaskNone ? KT * 4 : 1];
        if constexpr (MASKED != kMaskNone) {
#pragma unroll
            for (int g = 0; g < KT * 4; ++g)  // keys kbase + 32*(g/4) + 8*(g%4) + 4*hf .. +3
                mraw[g] = mslab.load(kbase + 32 * (g >> 2) + 8 * (g & 3) + 4 * hf);
        }

        f32x16 s[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 16; ++i) s[kt][i] = 0.f;
        // key tile kt=0 completes first, so its row max can overlap the MFMAs of kt=1
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks) {
                const int r = kt * 32 + l32;
                const int c = ks * 2 + hf;
                const V8 a = *reinterpret_cast<const V8*>(Kc + r * D + 8 * (c ^ kswz<D>(r)));
                s[kt] = Elem<T>::mfma32(a, qf[ks], s[kt]);
            }
        }
        // K fragment reads run 4 MFMAs ahead of their use
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
        for (int i = 0; i < KT * KSTEPS - 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
        // A tile whose keys a bool mask keeps for every row of the wave needs no adds (s + 0): most tiles of a
        // padding mask.
        bool add_mask = MASKED != kMaskNone;
        if constexpr (MASKED == kMaskBool) {
            uint32_t all = mslab.bytes(mraw[0]);
#pragma unroll
            for (int g = 1; g < KT * 4; ++g) all &= mslab.bytes(mraw[g]);
            add_mask = !__all(all == 0x01010101u);
        }
        if (add_mask) {
            if constexpr (MASKED != kMaskNone) {
#pragma unroll
                for (int g = 0; g < KT * 4; ++g) {
                    float s0 = s[g >> 2][4 * (g & 3) + 0], s1 = s[g >> 2][4 * (g & 3) + 1];
                    float s2 = s[g >> 2][4 * (g & 3) + 2], s3 = s[g >> 2][4 * (g & 3) + 3];
                    mslab.add(mraw[g], p.inv_scale, s0, s1, s2, s3);
                    s[g >> 2][4 * (g & 3) + 0] = s0, s[g >> 2][4 * (g & 3) + 1] = s1;
                    s[g >> 2][4 * (g & 3) + 2] = s2, s[g >> 2][4 * (g & 3) + 3] = s3;
                }
            }
        }
        if constexpr (kLateLoads) next_tile();
        if (need_mask) {
            // Element i of key tile kt holds key kbase + kt*32 + 8*(i/4) + 4*hf + i%4; it is visible
            // iff its compile-time offset kt*32 + 8*(i/4) + i%4 is <= lim.
            int lim = p.Sk - 1 - kbase;
            if (CAUSAL) lim = min(lim, wq0 + l32 + p.delta - kbase);
            lim -= 4 * hf;
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (kt * 32 + 8 * (i >> 2) + (i & 3) > lim) s[kt][i] = kNegInf;
        }
        V8 pb[PVS];
        // P = exp2(s c - base) and its row sum over the lane's keys, from `ls` on (fp32: a sum of the rounded P would cost
        // up to 2^-9 relative in the LSE of rows with few keys)
        auto exponentials = [&](float base, float ls) {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    V8 pk;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float pv = fast_exp2(__builtin_fmaf(s[kt][8 * half + e], p.c, -base));
                        ls += pv;
                        pk[e] = Elem<T>::from_f32(pv);
                    }
                    pb[2 * kt + half] = pk;
                }
            }
            return ls;
        };
        // Moves the row max where it grew by more than 2^threshold for some row of the wave.
        auto rescale = [&](float threshold) {
            float mx = kNegInf;
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kt][i]);
            mx = max_xor32(mx);
            const float mcand = fmaxf(mrow, mx * p.c);
            if (__any(mcand - mrow > threshold)) {  // wave-uniform
                const float alpha = fast_exp2(mrow - (mcand == kNegInf ? 0.f : mcand));
                // A lane whose max is still -inf has seen no visible key: its O and l are exactly 0.  When
                // that holds for the whole wave (its first tile) the multiply is skipped.
                if (!__all(mrow == kNegInf)) {
                    lrow *= alpha;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                        for (int i = 0; i < 16; ++i) oacc[dt][i] *= alpha;
                }
                mrow = mcand;
            }
        };
        // Wave priority: raised over the exponential/PV block of the non-causal kernel only.  Measured
        // A/B on one MI355X: MMDiT 1x24x4608 +4.5% against raising it over both blocks; the causal
        // kernels ran 1-3% faster with no raise at all.
        if constexpr (SUMC) {
            float ls = 0.f;
            bool done = false;
            if (!fresh) {
                __builtin_amdgcn_s_setprio(1);
                ls = exponentials(mrow, 0.f);
                done = !__any(ls > kSumLimit);
            }
            if (!done) {
                rescale(0.f);  // any growth moves it: a sum past the limit has some
                fresh = __any(mrow == kNegInf);
                ls = exponentials(mrow == kNegInf ? 0.f : mrow, 0.f);
            }
            lrow += ls;
        } else {
            rescale(kRescaleThreshold);
            if constexpr (!CAUSAL) __builtin_amdgcn_s_setprio(1);
            lrow = exponentials(mrow == kNegInf ? 0.f : mrow, lrow);
        }

        // k-step outer: the four MFMAs of step ks need only P chunk ks, so they can run while the
        // exponentials of the later chunks are still being computed
#pragma unroll
        for (int ks = 0; ks < PVS; ++ks) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const int d = dt * 32 + tr_d;
                const int k1 = ks * 16 + tr_k4 + tr_key;  // slots 0-3: keys 16ks + 4hf + j
                const int k2 = k1 + 8;                    // slots 4-7: keys 16ks + 8 + 4hf + j
                const V4 lo = __builtin_bit_cast(
                    V4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(Vc + k1 * D + 8 * ((d >> 3) ^ kswz<D>(k1)) + (d & 7))));
                const V4 hi = __builtin_bit_cast(
                    V4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(Vc + k2 * D + 8 * ((d >> 3) ^ kswz<D>(k2)) + (d & 7))));
                const V8 a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                oacc[dt] = Elem<T>::mfma32(a, pb[ks], oacc[dt]);
            }
        }
        // Issue order of this block: the V^T reads of step 0 and P chunk 0, then each PV MFMA
        // followed by two V^T reads and a slice of the next chunk's exponentials.
        __builtin_amdgcn_sched_group_barrier(0x100, 4 * DT, 0);
        __builtin_amdgcn_sched_group_barrier(0x402, 28, 0);
#pragma unroll
        for (int i = 0; i < (PVS - 1) * DT; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x402, 7, 0);
        }
#pragma unroll
        for (int i = 0; i < DT; ++i) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if constexpr (!CAUSAL) __builtin_amdgcn_s_setprio(0);
    };

    if (kg < nt) {
        dma(Ka, kp, krow, p.ks_s, kg, p.qk_ch);
        dma(Va, vp, vrow, p.vs_s, kg, p.v_ch);
    }
    // Q fragments: lane holds query l32, d = ks*16 + hf*8 .. +8.  Issued after tile 0's loads so that
    // the two share one memory latency.  The loads are unconditional, so they issue back to back (a
    // branch per load made the compiler wait for each in turn: 8 round trips, ~3.7 us of a C2
    // workgroup's start).  Rows past Sq read row Sq-1 and chunks past qk_ch read chunk 0; the mask
    // zeroes both.
    {
        const int qrow = wq0 + l32;
        const bool row_ok = qrow < p.Sq;
        const T* qsrc = qp + (int64_t)(row_ok ? qrow : p.Sq - 1) * p.qs_s;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
            const bool ok = row_ok && (!PAD || 2 * ks + hf < p.qk_ch);
            const u32x4 w = ld16(qsrc + (ok ? ks * 16 + hf * 8 : 0));
            qf[ks] = __builtin_bit_cast(V8, q_bits(w, ok ? p.q_and : 0u, ok ? p.q_xor : 0u));
        }
    }
    // Q fragments (and tile 0) complete here, visibly to the compiler, so that it inserts no load
    // waits inside the loop (where they would also drain the asynchronous tile loads).
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    for (int t = 0; t < nt; t += 2 * KG) {  // unrolled by two so each tile names its buffers statically
        tile(Ka, Va, Kb, Vb, t + kg);
        if (t + KG < nt) tile(Kb, Vb, Ka, Va, t + KG + kg);
    }
    if constexpr (KG > 1) {
        // The second group leaves its 16 DT accumulators, max and sum per lane in LDS; the first merges them.
        __syncthreads();
        float* const part = reinterpret_cast<float*>((wave < 2 ? Ka_ : Kb_) + (wave & 1) * BN * D);  // [16 DT][64 lanes]
        float* const ml = reinterpret_cast<float*>(Vb_) + wave * 128;
        if (kg > 0) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) part[(16 * dt + i) * 64 + lane] = oacc[dt][i];
            ml[lane] = mrow;
            ml[64 + lane] = lrow;
        }
        __syncthreads();
        if (kg == 0) {
            const float mg = ml[lane], lg = ml[64 + lane];
            const float mm = fmaxf(mrow, mg), mb = mm == kNegInf ? 0.f : mm;  // -inf: no visible key, weight 0
            const float a0 = fast_exp2(mrow - mb), ag = fast_exp2(mg - mb);
            mrow = mm;
            lrow = lrow * a0 + lg * ag;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) oacc[dt][i] = oacc[dt][i] * a0 + part[(16 * dt + i) * 64 + lane] * ag;
        }
    }

    // Epilogue: normalise, stage O through LDS (wave w in a 32-row slab of Ka/Kb; 16-byte chunk c of
    // row r at c ^ (r % DCH)) for 16-byte coalesced row stores, and write the LSE.
    __syncthreads();
    if (KG > 1 && kg > 0) return;
    T* Os = (wave < 2 ? Ka : Kb) + (wave & 1) * 32 * D;
    {
        const float l = sum_xor32(lrow);
        const float inv = l > 0.f ? 1.f / l : 0.f;
        const int row = l32;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                V4 o4;
#pragma unroll
                for (int e = 0; e < 4; ++e) o4[e] = Elem<T>::from_f32(oacc[dt][4 * i4 + e] * inv);
                const int c = dt * 4 + i4;
                *reinterpret_cast<V4*>(Os + row * D + 8 * (c ^ (row % DCH)) + 4 * hf) = o4;
            }
        if (p.lse != nullptr && hf == 0) {
            const int qrow = wq0 + row;
            if (qrow < p.Sq) {
                const float lse = l > 0.f ? (mrow + __log2f(l)) * kLn2 : kNegInf;
                p.lse[b * p.lses_b + hq * p.lses_h + qrow] = lse;
            }
        }
    }
    __syncthreads();
    T* op = reinterpret_cast<T*>(p.o) + b * p.os_b + hq * p.os_h;
#pragma unroll
    for (int it = 0; it < 32 * DCH / 64; ++it) {
        const int id = it * 64 + lane;
        const int row = id / DCH, c = id % DCH;
        const int qrow = wq0 + row;
        // non-temporal: measured +1.3 to 2.5% on short sequences (16x512, 32x256), +0.2 to 0.3% on long ones,
        // against plain stores, with back-to-back launches
        if (qrow < p.Sq && (!PAD || c < p.v_ch))
            __builtin_nontemporal_store(ld16(Os + row * D + 8 * (c ^ (row % DCH))),
                                        reinterpret_cast<u32x4*>(op + (int64_t)qrow * p.os_s + c * 8));
    }
}

// ------------------------------------------------------------------------------------------------

template <typename T, int D, int QT, bool CAUSAL, int MASKED, bool PAD, int KG = 1, bool SUMC = false>
static int launch_prefill(const PrefillParams& prm, hipStream_t stream) {
    constexpr int BM = 4 * QT * 32;
    PrefillParams p = prm;
    p.n_qblocks = (p.Sq + BM - 1) / BM;
    const int64_t grid = (int64_t)p.n_qblocks * p.B * p.Hq;
    if (grid == 0) return DTATTN_OK;
    if (grid > 0x7fffffff) return fail(DTATTN_ERR_UNSUPPORTED, "prefill grid too large (%lld blocks)", (long long)grid);
    hipLaunchKernelGGL((prefill_fwd_kernel<T, D, QT, CAUSAL, MASKED, PAD, KG, SUMC>), dim3((unsigned)grid), dim3(256 * KG), 0, stream, p);
    return check_launch("prefill_fwd_kernel");
}

static int stream_device(hipStream_t stream, int* dev) {
    return (stream == nullptr ? hipGetDevice(dev) : hipStreamGetDevice(stream, dev)) == hipSuccess ? DTATTN_OK
                                                                                               : DTATTN_ERR_DEVICE;
}

// Whether a head-dim-64 call without mask or causal rule takes the form that checks the sums of P.  With r workgroups of
// 128 rows per CU (three fit at once), times with the row max first over times with the check, bf16 / fp16:
//   r up to 2: 1.03-1.37 from 512 keys on, 0.94-1.00 at 77 to 256 keys
//   2 < r <= 3: 0.96-0.99 at r = 2.25, 0.96-1.00 at 2.5, 0.98-1.01 at 2.75 and 3, at any number of keys
//   3 < r <= 4: 1.02-1.10 at 3.25; at 3.75 and 4 1.01-1.07 up to 256 keys, 0.95-0.97 at 512 and 768, 0.96-1.01 above
//   r above 4: 1.00-1.08 (one 0.97)
static bool sum_check_pays(const PrefillParams& p, hipStream_t stream) {
    int dev = 0;
    dtattn_device_peaks pk;
    if (stream_device(stream, &dev) != DTATTN_OK || dtattn_get_device_peaks(dev, &pk) != DTATTN_OK) return true;
    const int64_t grid = ((int64_t)p.Sq + 127) / 128 * p.B * p.Hq, cus = pk.cu_count;
    if (grid > 4 * cus) return true;
    if (grid > 3 * cus) return 8 * grid <= 27 * cus || p.Sk <= 256;
    return grid <= 2 * cus && p.Sk > 256;
}

template <typename T, int MASKED, bool PAD>
static int dispatch_prefill_m(const PrefillParams& p, int D, bool causal, int kg, hipStream_t stream) {
    if constexpr (MASKED == kMaskNone && !PAD) {
        if (kg > 1 && D == 128)
            return causal ? launch_prefill<T, 128, 1, true, MASKED, PAD, 2>(p, stream)
                          : launch_prefill<T, 128, 1, false, MASKED, PAD, 2>(p, stream);
        if (kg > 1 && D == 64)
            return causal ? launch_prefill<T, 64, 1, true, MASKED, PAD, 2>(p, stream)
                          : launch_prefill<T, 64, 1, false, MASKED, PAD, 2, true>(p, stream);
    }
    if (D == 128) {
        return causal ? launch_prefill<T, 128, 1, true, MASKED, PAD>(p, stream)
                      : launch_prefill<T, 128, 1, false, MASKED, PAD>(p, stream);
    }
    if (D == 64) {
        if constexpr (MASKED == kMaskNone)
            if (!causal && sum_check_pays(p, stream)) return launch_prefill<T, 64, 1, false, MASKED, PAD, 1, true>(p, stream);
        return causal ? launch_prefill<T, 64, 1, true, MASKED, PAD>(p, stream)
                      : launch_prefill<T, 64, 1, false, MASKED, PAD>(p, stream);
    }
    return fail(DTATTN_ERR_UNSUPPORTED, "prefill: kernel head dim %d not supported (64, 128, 256 or 512)", D);
}

int prefill_rows64(const PrefillParams& p, bool causal, bool f16, void* ws, size_t ws_bytes, hipStream_t stream);
bool prefill_rows64_fits(const PrefillParams& p);
int prefill_rows64_spans(const PrefillParams& p, bool causal, bool f16, hipStream_t stream);
bool prefill_rows64_streamk(const PrefillParams& p, bool causal, hipStream_t stream);
size_t rows64_sk_workspace(const dtattn_prefill_args* a, int device);

// Kernel head dim of a bf16/fp16 call: the smallest of 64, 128, 256, 512 holding both real head dims.
static int kernel_head_dim(int64_t D, int64_t Dv) {
    const int64_t dmax = D > Dv ? D : Dv;
    return dmax <= 64 ? 64 : dmax <= 128 ? 128 : dmax <= 256 ? 256 : dmax <= 512 ? 512 : 0;
}

// The key span of each batch (PrefillParams::spans) of a mask that is one row of keys for all queries and heads, and,
// unless `rows` is NULL, that row in fp32 (0 and -inf for a bool mask) at rows + batch * pitch.  One workgroup per batch;
// the row is a few KB, so this is one short launch ahead of a call of 40 us or more.
__global__ void __launch_bounds__(256) mask_spans_kernel(const void* mask, int kind, int64_t ms_b, int Sk, float inv_scale,
                                                         int2* spans, float* rows, int64_t pitch) {
    __shared__ int red[4][4];
    const int64_t off = (int64_t)blockIdx.x * ms_b;
    int first = Sk, last = -1, count = 0, other = 0;
    constexpr int NB = 8;  // loads in flight: one memory latency per 2048 keys
    for (int j0 = threadIdx.x; j0 < Sk; j0 += 256 * NB) {
        float mv[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int64_t at = off + min(j0 + 256 * i, Sk - 1);
            if (kind == DTATTN_BOOL) mv[i] = reinterpret_cast<const uint8_t*>(mask)[at] != 0 ? 0.f : kNegInf;
            else if (kind == DTATTN_BF16) mv[i] = (float)reinterpret_cast<const bf16_t*>(mask)[at];
            else if (kind == DTATTN_FP16) mv[i] = (float)reinterpret_cast<const f16_t*>(mask)[at];
            else mv[i] = reinterpret_cast<const float*>(mask)[at];
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int j = j0 + 256 * i;
            if (j >= Sk) break;
            const float m = mv[i];
            if (rows != nullptr) rows[blockIdx.x * pitch + j] = m;
            if (m * inv_scale != kNegInf) {  // not hidden
                first = min(first, j);
                last = max(last, j);
                ++count;
                other |= m != 0.f;  // NaN too
            }
        }
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        first = min(first, __shfl_xor(first, d, 64));
        last = max(last, __shfl_xor(last, d, 64));
        count += __shfl_xor(count, d, 64);
        other |= __shfl_xor(other, d, 64);
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) red[0][w] = first, red[1][w] = last, red[2][w] = count, red[3][w] = other;
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int i = 1; i < 4; ++i) {
        first = min(first, red[0][i]);
        last = max(last, red[1][i]);
        count += red[2][i];
        other |= red[3][i];
    }
    spans[blockIdx.x] = count == 0 ? make_int2(0, 0)
                        : other == 0 && count == last + 1 - first ? make_int2(first, last + 1) : make_int2(0, -1);
}

// Whether mask_spans_kernel runs ahead of a masked call, and the workspace it needs: bf16 / fp16 calls at D = Dv = 128
// (the span kernel's) whose mask is the same for every query and head, from 2.4e10 operations on, not causal from 3e10.
// A call none of whose batches has a span pays 5-7 us for the two launches that find that out.  us without spans, with
// them for left padding up to half, with them for a mask with a hole: causal 4x32/8x850 (2.4e10) 53, 35, 62, not causal
// 8x32/8x400 (2.1e10) 40, 36, 43, 4x32/8x600 (2.4e10) 40, 41, 45, 4x32/8x700 (3.2e10) 49, 45, 50, 4x32/8x850 (4.7e10)
// 64, 51, 67; causal 4x32/8x1000 65, 40, 72 (bool) and 67, 40, 72 (fp32).
//
// Not causal, batches without a span read a 16-bit or bool mask from fp32 rows (4x32/8x2000 bool 280 -> 270 us, bf16
// 298 -> 270); causal they read it as stored (bool 226 -> 209, bf16 225 -> 219), and fp32 masks always (2x32/8x1000 42 -> 36).
struct MaskSpans {
    size_t bytes = 0, rows = 0;  // of the workspace; where the rows start, or 0
    int64_t pitch = 0;           // of the rows, in elements
};
static MaskSpans mask_spans_plan(const dtattn_prefill_args* a, const dtattn_mask* mk) {
    MaskSpans m;
    if (a->dtype != DTATTN_BF16 && a->dtype != DTATTN_FP16) return m;
    if (a->B <= 0 || a->B > 0x7fffffff || a->Hq <= 0 || a->Sq <= 1 || a->Sk <= 0 || a->D != 128 || a->Dv != 128) return m;
    if (mk->stride[1] != 0 || mk->stride[2] != 0) return m;
    const double ops = 512.0 * (double)a->B * (double)a->Hq * (double)a->Sq * (double)a->Sk * (a->causal != 0 ? 0.5 : 1.0);
    if (ops < (a->causal != 0 ? 2.4e10 : 3e10)) return m;
    m.bytes = (size_t)a->B * sizeof(int2);
    if (a->causal == 0 && mk->dtype != DTATTN_FP32) {
        m.rows = (m.bytes + 255) & ~(size_t)255;
        m.pitch = (a->Sk + 3) / 4 * 4;
        m.bytes = m.rows + (size_t)a->B * m.pitch * sizeof(float);
    }
    return m;
}

// Key groups of prefill_fwd_kernel for a call without mask or padding, or 0: the grid is large enough for the kernels
// with 64 rows per wave (head dim 128).  A workgroup ends no sooner than its own key tiles, and a 64-row wave takes
// 1.35 us a tile against 0.95 us here, so up to two workgroups per CU 128-row blocks of one head end first (causal
// 1x32/8x512 18.0 -> 13.8 us, 2x32/8x777 23.1 -> 20.4, 4x32/8x512 18.3 -> 15.8; 16x32/8x128 not causal 11.8 -> 9.5); a
// non-causal grid of long rows is as good on the 64-row kernel already (1x32/8x1500 42.6 against 40.6; two workgroups per CU,
// 64-row time over this one's at 640, 896 and 1024 keys: 1.10, 1.06, 1.04 for 16 kv heads, 1.05, 1.00, 0.97 where the 64-row
// kernel shares a kv head's tiles among 4 query heads).  Two key groups
// halve the chain of tiles, for 128 KB of LDS at head dim 128 and a merge worth 1-2 us: from 8 tiles on, on grids of one
// workgroup per CU (causal 1x32/8x1024 22.3 -> 20.9, 777 18.2 -> 16.7, 400 11.9 both; D = 64 1x12x1024 15.8 -> 13.4) and
// on causal ones of two where the second round is the short blocks of many (1x32/8x1500 32.0 -> 28.8, D = 64 1x12x4096
// 51.5 -> 39.7; of 7 blocks, 1x64/8x777, 20.1 -> 24.5).  A prompt that continues a long context is long rows again: between
// one and two workgroups per CU (r), the 64-row kernel over this one by the tiles of its first block times r over its
// blocks: 2.3 to 3.4 1.02-1.12, 4.5 0.96-1.08 (2x32/8x900 behind 1000 keys 52.7 / 55.0), above 0.88-1.02 (3x32/8x512 behind
// 3000 85 / 96, 4x32/8x512 behind 1000 46.5 / 49.5); with less than 16 tiles in the first block 0.99-1.17.
static int key_groups(const PrefillParams& p, int D, bool causal, hipStream_t stream) {
    int dev = 0;
    dtattn_device_peaks pk;
    if (stream_device(stream, &dev) != DTATTN_OK || dtattn_get_device_peaks(dev, &pk) != DTATTN_OK) return D == 128 ? 0 : 1;
    const int64_t blocks = ((int64_t)p.Sq + 127) / 128, grid = blocks * p.B * p.Hq;
    int64_t keys = p.Sk;  // of the longest workgroup
    if (causal) keys = std::max<int64_t>(0, std::min<int64_t>(keys, (int64_t)p.Sq + p.delta));
    const int64_t tiles = (keys + 63) / 64;
    if (grid <= pk.cu_count) return tiles >= 8 ? 2 : 1;
    if (grid <= 2 * pk.cu_count) {
        if (causal) {
            const int64_t first = (std::max<int64_t>(0, std::min<int64_t>(p.Sk, 128 + p.delta)) + 63) / 64;  // tiles of rows 0..127
            if (D == 128 && first >= 16 && 2 * first * grid >= 9 * blocks * pk.cu_count) return 0;
            return tiles >= 8 && blocks >= 12 ? 2 : 1;
        }
        if (tiles <= (p.group >= 4 && p.group % 4 == 0 ? 13 : 16)) return 1;
    }
    return D == 128 ? 0 : 1;
}

// D is the kernel's head dim (64 or 128); pad: the real head dims are below it.  Head dim 128 without mask or
// padding runs the 64-rows-per-wave kernel (prefill_rows64.hip) on grids that fill the chip, which returns the same
// bits as prefill_fwd_kernel at 4-9% (non-causal) and 4-14% (causal) more throughput.
template <typename T>
static int dispatch_prefill(PrefillParams p, int D, bool causal, bool pad, void* ws, size_t ws_bytes, hipStream_t stream) {
    // Row masks with key spans (head dim 128): the batches that have one run as shorter calls without a mask, on the
    // faster kernel and without the hidden tiles; prefill_fwd_kernel then runs the others and leaves at once for these
    // (about 4 us of a call).  4x32/8x2000, left padding up to half: causal 219 -> 103 us, not causal 264 -> 186 us.
    if (p.spans != nullptr) {
        const int st = prefill_rows64_spans(p, causal, __is_same(T, f16_t), stream);
        if (st != DTATTN_OK) return st;
    }
    int kg = 1;
    if (!pad && p.mask == nullptr) {
        const bool fits64 = D == 128 && prefill_rows64_fits(p);
        kg = key_groups(p, D, causal, stream);
        if (fits64 && (kg == 0 || prefill_rows64_streamk(p, causal, stream)))
            return prefill_rows64(p, causal, __is_same(T, f16_t), ws, ws_bytes, stream);
    }
    const MaskMode mode = mask_mode(p);
    auto run = [&](auto pad_c) {
        constexpr bool PAD = decltype(pad_c)::value;
        switch (mode) {
            case kMaskF32: return dispatch_prefill_m<T, kMaskF32, PAD>(p, D, causal, kg, stream);
            case kMaskBool: return dispatch_prefill_m<T, kMaskBool, PAD>(p, D, causal, kg, stream);
            case kMaskBf16: return dispatch_prefill_m<T, kMaskBf16, PAD>(p, D, causal, kg, stream);
            case kMaskF16: return dispatch_prefill_m<T, kMaskF16, PAD>(p, D, causal, kg, stream);
            default: return dispatch_prefill_m<T, kMaskNone, PAD>(p, D, causal, kg, stream);
        }
    };
    return pad ? run(std::true_type{}) : run(std::false_type{});
}

int prefill_fp8(const dtattn_prefill_args* a, float c, int32_t delta, uint32_t q_and, uint32_t q_xor,
                hipStream_t stream);
size_t prefill_fp8_workspace_size(const dtattn_prefill_args* a, int device);
int prefill_f32(const PrefillParams& p, int D, bool causal, bool pad, hipStream_t stream);
int prefill_wide(const PrefillParams& p, int D, bool causal, bool bf16, bool pad, hipStream_t stream);
int wide_key_splits(int64_t B, int64_t Hq, int64_t Sq, int64_t Sk, int D, int cu_count);

// Key blocks of a wide-head call on `device` (1: unsplit) and the workspace their partials need:
// O parts [splits][B][Hq][Sq][Dv] in the input dtype, then (256-byte aligned) LSE parts
// [splits][B][Hq][Sq] fp32.
static int wide_plan(const dtattn_prefill_args* a, int device, size_t* bytes, size_t* lse_off) {
    *bytes = 0;
    *lse_off = 0;
    if (a->dtype != DTATTN_BF16 && a->dtype != DTATTN_FP16) return 1;
    if (a->D % 8 != 0 || a->Dv % 8 != 0 || a->B <= 0 || a->Sq <= 0 || a->Sk <= 0) return 1;
    const int Dk = kernel_head_dim(a->D, a->Dv);
    if (Dk < 256) return 1;
    dtattn_device_peaks pk;
    if (dtattn_get_device_peaks(device, &pk) != DTATTN_OK) return 1;
    const int splits = wide_key_splits(a->B, a->Hq, a->Sq, a->Sk, Dk, pk.cu_count);
    if (splits <= 1) return 1;
    const size_t o_bytes = (size_t)splits * a->B * a->Hq * a->Sq * a->Dv * 2;
    *lse_off = (o_bytes + 255) & ~(size_t)255;
    *bytes = *lse_off + (size_t)splits * a->B * a->Hq * a->Sq * sizeof(float);
    return splits;
}

static int mask_element_size(int32_t dtype) {
    return dtype == DTATTN_BOOL ? 1 : dtype == DTATTN_BF16 || dtype == DTATTN_FP16 ? 2 : dtype == DTATTN_FP32 ? 4 : 0;
}

static bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

}  // namespace dtattn

using namespace dtattn;

// dtattn_prefill_fwd with the mask either in `a` (fp32) or in `mk`, as the caller holds it.
static int prefill_entry(const dtattn_prefill_args* a, const dtattn_mask* mk, void* stream_) {
    if (a == nullptr) return fail(DTATTN_ERR_INVALID_ARGUMENT, "prefill: args is NULL");
    hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
    if (a->B < 0 || a->Hq <= 0 || a->Hkv <= 0 || a->Sq < 0 || a->Sk < 0)
        return fail(DTATTN_ERR_INVALID_ARGUMENT, "prefill: bad sizes B=%lld Hq=%lld Hkv=%lld Sq=%lld Sk=%lld",
                    (long long)a->B, (long long)a->Hq, (long long)a->Hkv, (long long)a->Sq, (long long)a->Sk);
    if (a->Hq % a->Hkv != 0)
        return fail(DTATTN_ERR_INVALID_ARGUMENT, "prefill: Hq=%lld is not a multiple of Hkv=%lld", (long long)a->Hq,
                    (long long)a->Hkv);
    if (a->D <= 0 || a->Dv <= 0)
        return fail(DTATTN_ERR_INVALID_ARGUMENT, "prefill: bad head dims D=%lld Dv=%lld", (long long)a->D,
                    (long long)a->Dv);
    const bool sixteen_bit = a->dtype == DTATTN_BF16 || a->dtype == DTATTN_FP16;
    if (a->D != a->Dv && !sixteen_bit && a->dtype != DTATTN_FP32)
        return fail(DTATTN_ERR_UNSUPPORTED, "prefill: D=%lld != Dv=%lld is supported for bf16/fp16/fp32 only",
                    (long long)a->D, (long long)a->Dv);
    if (sixteen_bit && (a->D % 8 != 0 || a->Dv % 8 != 0))
        return fail(DTATTN_ERR_UNSUPPORTED, "prefill: head dims must be multiples of 8 (D=%lld, Dv=%lld)",
                    (long long)a->D, (long long)a->Dv);
    if (a->dtype == DTATTN_FP32 && (a->D % 4 != 0 || a->Dv % 4 != 0 || a->D > 512 || a->Dv > 512))
        return fail(DTATTN_ERR_UNSUPPORTED,
                    "prefill: fp32 head dims must be multiples of 4 up to 512 (D=%lld, Dv=%lld)", (long long)a->D,
                    (long long)a->Dv);
    // Sequence lengths up to 2^29 keep every causal index expression of the kernels in int32.
    if (a->Sq > (1 << 29) || a->Sk > (1 << 29) || a->B * a->Hq > 0x3fffffff)
        return fail(DTATTN_ERR_UNSUPPORTED, "prefill: sequence length exceeds 2^29");
    if (a->B == 0 || a->Sq == 0) return DTATTN_OK;
    if (a->q == nullptr || a->o == nullptr || (a->Sk > 0 && (a->k == nullptr || a->v == nullptr)))
        return fail(DTATTN_ERR_INVALID_ARGUMENT, "prefill: null tensor pointer");
    const int64_t* strides[4] = {a->q_stride, a->k_stride, a->v_stride, a->o_stride};
    const int esz_in = a->dtype == DTATTN_FP8_E4M3FN ? 1 : (a->dtype == DTATTN_FP32 ? 4 : 2);
    const int esz_out = a->o_dtype == DTATTN_FP32 ? 4 : 2;
    for (int i = 0; i < 4; ++i) {
        const int esz = i == 3 ? esz_out : esz_in;
        for (int j = 0; j < 3; ++j)
            if ((strides[i][j] * esz) % 16 != 0)
                return fail(DTATTN_ERR_UNSUPPORTED,
                            "prefill: tensor %d stride[%d]=%lld is not a multiple of 16 bytes", i, j,
                            (long long)strides[i][j]);
    }
    if (!aligned16(a->q) || !aligned16(a->k) || !aligned16(a->v) || !aligned16(a->o))
        return fail(DTATTN_ERR_UNSUPPORTED, "prefill: tensors must be 16-byte aligned");
    // key/value tiles are addressed with 32-bit byte offsets: 64 rows x row pitch < 2^31
    if (a->k_stride[2] * esz_in * 64 >= (int64_t)1 << 31 || a->v_stride[2] * esz_in * 64 >= (int64_t)1 << 31)
        return fail(DTATTN_ERR_UNSUPPORTED, "prefill: key/value row pitch exceeds 32 MB");
    ScalePlan sp;
    {
        const uint32_t sign = a->dtype == DTATTN_FP32 ? kSign32 : a->dtype == DTATTN_FP8_E4M3FN ? kSign8 : kSign16;
        const int st = plan_scale(a->scale, a->D, sign, &sp);
        if (st != DTATTN_OK) return st;
    }
    const float scale = sp.scale;
    const float c = scale * kLog2e;
    int64_t delta64 = a->q_offset - a->k_offset;
    const int64_t lim = a->Sq + a->Sk + 1;
    if (delta64 > lim) delta64 = lim;
    if (delta64 < -lim) delta64 = -lim;
    const int32_t delta = (int32_t)delta64;

    if (mk != nullptr) {
        if (a->mask != nullptr) return fail(DTATTN_ERR_INVALID_ARGUMENT, "prefill: two masks");
        const int esz = mask_element_size(mk->dtype);
        if (esz == 0)
            return fail(DTATTN_ERR_UNSUPPORTED, "prefill: mask dtype %d not supported (bool, bf16, fp16, fp32)", mk->dtype);
        if (a->dtype == DTATTN_FP8_E4M3FN)
            return fail(DTATTN_ERR_UNSUPPORTED, "prefill: an attention mask is not supported with fp8 inputs");
        if (kernel_head_dim(a->D, a->Dv) > 128)
            return fail(DTATTN_ERR_UNSUPPORTED, "prefill: a mask as stored needs head dims up to 128 (D=%lld, Dv=%lld)",
                        (long long)a->D, (long long)a->Dv);
        for (int j = 0; j < 3; ++j)
            if (mk->stride[j] < 0)
                return fail(DTATTN_ERR_UNSUPPORTED, "prefill: mask stride[%d]=%lld is negative", j, (long long)mk->stride[j]);
        if (mk->data == nullptr || reinterpret_cast<uintptr_t>(mk->data) % (uintptr_t)esz != 0)
            return fail(DTATTN_ERR_INVALID_ARGUMENT, "prefill: mask pointer is null or not aligned to its elements");
        if (((a->Sq - 1) * mk->stride[2] + a->Sk + 64) * esz + 64 >= ((int64_t)1 << 32))
            return fail(DTATTN_ERR_UNSUPPORTED, "prefill: mask slab of one (batch, head) exceeds 4 GB");
    }
    if (a->mask != nullptr) {
        if (a->dtype == DTATTN_FP8_E4M3FN)
            return fail(DTATTN_ERR_UNSUPPORTED, "prefill: an attention mask is not supported with fp8 inputs");
        for (int j = 0; j < 3; ++j)
            if (a->mask_stride[j] < 0 || a->mask_stride[j] % 4 != 0)
                return fail(DTATTN_ERR_UNSUPPORTED, "prefill: mask stride[%d]=%lld must be a non-negative multiple of 4",
                            j, (long long)a->mask_stride[j]);
        if ((reinterpret_cast<uintptr_t>(a->mask) & 15u) != 0)
            return fail(DTATTN_ERR_UNSUPPORTED, "prefill: mask must be 16-byte aligned");
        // one (b, h) slab of the mask is addressed with 32-bit byte offsets
        if (((a->Sq - 1) * a->mask_stride[2] + a->Sk + 64) * 4 >= ((int64_t)1 << 32))
            return fail(DTATTN_ERR_UNSUPPORTED, "prefill: mask slab of one (batch, head) exceeds 4 GB");
    }
    if (a->dtype == DTATTN_FP8_E4M3FN) {
        if (a->o_dtype != DTATTN_BF16 && a->o_dtype != DTATTN_FP16)
            return fail(DTATTN_ERR_UNSUPPORTED, "prefill fp8: output must be bf16 or fp16");
        if (a->q_descale == nullptr || a->k_descale == nullptr || a->v_descale == nullptr)
            return fail(DTATTN_ERR_INVALID_ARGUMENT, "prefill fp8: descale pointers are required");
        return prefill_fp8(a, c, delta, sp.q_and, sp.q_xor, stream);
    }
    if (a->dtype != DTATTN_BF16 && a->dtype != DTATTN_FP16 && a->dtype != DTATTN_FP32)
        return fail(DTATTN_ERR_UNSUPPORTED, "prefill: dtype %d not supported (bf16, fp16, fp32, fp8_e4m3fn)",
                    a->dtype);
    if (a->o_dtype != a->dtype) return fail(DTATTN_ERR_UNSUPPORTED, "prefill: output dtype must equal input dtype");

    PrefillParams p;
    p.q = a->q;
    p.k = a->k;
    p.v = a->v;
    p.o = a->o;
    p.lse = a->lse;
    p.qs_b = a->q_stride[0], p.qs_h = a->q_stride[1], p.qs_s = a->q_stride[2];
    p.ks_b = a->k_stride[0], p.ks_h = a->k_stride[1], p.ks_s = a->k_stride[2];
    p.vs_b = a->v_stride[0], p.vs_h = a->v_stride[1], p.vs_s = a->v_stride[2];
    p.os_b = a->o_stride[0], p.os_h = a->o_stride[1], p.os_s = a->o_stride[2];
    p.lses_b = a->lse ? a->lse_stride[0] : 0;
    p.lses_h = a->lse ? a->lse_stride[1] : 0;
    p.B = (int32_t)a->B;
    p.Hq = (int32_t)a->Hq;
    p.Hkv = (int32_t)a->Hkv;
    p.Sq = (int32_t)a->Sq;
    p.Sk = (int32_t)a->Sk;
    p.group = (int32_t)(a->Hq / a->Hkv);
    p.n_qblocks = 0;
    p.delta = delta;
    p.c = c;
    p.xcd_map = (p.B * p.Hkv) % 8 == 0 ? 1 : 0;
    p.mask = mk != nullptr ? mk->data : a->mask;
    const int64_t* ms = mk != nullptr ? mk->stride : a->mask_stride;
    p.ms_b = ms[0], p.ms_h = ms[1], p.ms_l = ms[2];
    p.mask_kind = mk != nullptr ? mk->dtype : DTATTN_FP32;
    p.spans = nullptr;
    p.inv_scale = 1.0f / scale;
    p.nsplit = 1;
    p.kblock = (int32_t)(a->Sk > 0 ? a->Sk : 1);
    p.os_split = 0;
    p.lses_split = 0;
    p.q_and = sp.q_and;
    p.q_xor = sp.q_xor;
    const bool causal = a->causal != 0;
    if (mk != nullptr && a->workspace != nullptr && (reinterpret_cast<uintptr_t>(a->workspace) & 255u) == 0) {
        const MaskSpans m = mask_spans_plan(a, mk);
        if (m.bytes > 0 && m.bytes <= a->workspace_bytes && prefill_rows64_fits(p)) {
            int2* spans = reinterpret_cast<int2*>(a->workspace);
            float* rows = m.rows > 0 ? reinterpret_cast<float*>(static_cast<char*>(a->workspace) + m.rows) : nullptr;
            hipLaunchKernelGGL(mask_spans_kernel, dim3((unsigned)a->B), dim3(256), 0, stream, mk->data, mk->dtype,
                               mk->stride[0], p.Sk, p.inv_scale, spans, rows, m.pitch);
            const int st = check_launch("mask_spans_kernel");
            if (st != DTATTN_OK) return st;
            p.spans = spans;
            if (rows != nullptr) {
                p.mask = rows;
                p.mask_kind = DTATTN_FP32;
                p.ms_b = m.pitch;
            }
        }
    }
    if (a->dtype == DTATTN_FP32) {
        // kernel head dim 64, 128, 256 or 512 (the last two on the wide fp32 kernel); smaller real dims
        // (multiples of 4, D and Dv independent) are padded
        const int Dk = kernel_head_dim(a->D, a->Dv);
        p.qk_ch = (int32_t)(a->D / 4);
        p.v_ch = (int32_t)(a->Dv / 4);
        return prefill_f32(p, Dk, causal, a->D != Dk || a->Dv != Dk, stream);
    }
    // bf16 / fp16: the kernel head dim is the smallest of 64, 128, 256, 512 that holds both real head
    // dims; smaller real dims (multiples of 8, D and Dv independent) run the padded instantiations.
    const int Dk = kernel_head_dim(a->D, a->Dv);
    if (Dk == 0)
        return fail(DTATTN_ERR_UNSUPPORTED, "prefill: head dim %lld exceeds 512",
                    (long long)(a->D > a->Dv ? a->D : a->Dv));
    p.qk_ch = (int32_t)(a->D / 8);
    p.v_ch = (int32_t)(a->Dv / 8);
    const bool pad = a->D != Dk || a->Dv != Dk;
    if (Dk >= 256) {
        int splits = 1;
        size_t need = 0, lse_off = 0;
        if (a->workspace != nullptr && a->workspace_bytes > 0 && (reinterpret_cast<uintptr_t>(a->workspace) & 255u) == 0) {
            int dev = 0;
            if (stream_device(stream, &dev) != DTATTN_OK) return fail(DTATTN_ERR_DEVICE, "prefill: stream device");
            splits = wide_plan(a, dev, &need, &lse_off);
            if (need > a->workspace_bytes) splits = 1;
        }
        if (splits <= 1) return prefill_wide(p, Dk, causal, a->dtype == DTATTN_BF16, pad, stream);
        // Key blocks in one launch, then their (O, LSE) merged by LSE into the caller's outputs.
        const int64_t tiles = (a->Sk + 31) / 32;
        p.kblock = (int32_t)((tiles + splits - 1) / splits * 32);
        p.nsplit = (int32_t)((a->Sk + p.kblock - 1) / p.kblock);
        char* ws = static_cast<char*>(a->workspace);
        p.o = ws;
        p.os_b = a->Hq * a->Sq * a->Dv, p.os_h = a->Sq * a->Dv, p.os_s = a->Dv;
        p.os_split = a->B * a->Hq * a->Sq * a->Dv;
        p.lse = reinterpret_cast<float*>(ws + lse_off);
        p.lses_b = a->Hq * a->Sq, p.lses_h = a->Sq;
        p.lses_split = a->B * a->Hq * a->Sq;
        const int st = prefill_wide(p, Dk, causal, a->dtype == DTATTN_BF16, pad, stream);
        if (st != DTATTN_OK) return st;
        dtattn_merge_args m;
        memset(&m, 0, sizeof(m));
        m.n_blocks = p.nsplit;
        for (int i = 0; i < p.nsplit; ++i) {
            m.o_blocks[i] = ws + (size_t)i * p.os_split * 2;
            m.lse_blocks[i] = reinterpret_cast<const float*>(ws + lse_off) + (size_t)i * p.lses_split;
        }
        m.B = a->B, m.H = a->Hq, m.S = a->Sq, m.D = a->Dv;
        m.block_o_stride[0] = p.os_b, m.block_o_stride[1] = p.os_h, m.block_o_stride[2] = p.os_s;
        m.block_lse_stride[0] = p.lses_b, m.block_lse_stride[1] = p.lses_h;
        m.block_dtype = a->dtype;
        m.o = a->o;
        m.o_stride[0] = a->o_stride[0], m.o_stride[1] = a->o_stride[1], m.o_stride[2] = a->o_stride[2];
        m.lse = a->lse;
        m.lse_stride[0] = a->lse_stride[0], m.lse_stride[1] = a->lse_stride[1];
        m.o_dtype = a->o_dtype;
        return dtattn_lse_merge(&m, stream);
    }
    if (a->dtype == DTATTN_BF16) return dispatch_prefill<bf16_t>(p, Dk, causal, pad, a->workspace, a->workspace_bytes, stream);
    return dispatch_prefill<f16_t>(p, Dk, causal, pad, a->workspace, a->workspace_bytes, stream);
}

extern "C" int dtattn_prefill_fwd(const dtattn_prefill_args* a, void* stream) { return prefill_entry(a, nullptr, stream); }

extern "C" int dtattn_prefill_masked(const dtattn_prefill_args* a, const dtattn_mask* mask, void* stream) {
    return prefill_entry(a, mask, stream);
}

extern "C" size_t dtattn_prefill_masked_workspace_size(const dtattn_prefill_args* a, const dtattn_mask* mask) {
    return a == nullptr || mask == nullptr ? 0 : mask_spans_plan(a, mask).bytes;
}

extern "C" size_t dtattn_prefill_workspace_size(const dtattn_prefill_args* a) {
    if (a == nullptr) return 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (a->dtype == DTATTN_FP8_E4M3FN) return prefill_fp8_workspace_size(a, dev);
    size_t bytes = 0, lse_off = 0;
    wide_plan(a, dev, &bytes, &lse_off);
    const size_t sk = rows64_sk_workspace(a, dev);
    return bytes > sk ? bytes : sk;
}
