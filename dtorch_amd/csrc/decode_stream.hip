// Single-token decode of larger batches, streaming form (bf16 / fp16, head dim 128, groups of up to 8 query heads).
//
// Semantics and callers are decode_splitkv.hip's (SdpaOp::Compute's arithmetic,
// dtorch/core/operators/standard/scaled_dot_product_attention_op.cc:107-109, at Lq = 1 over the true lengths).
//
// Bound by HBM: the cache is read once.  The split kernel's workgroups load one split each into registers, so a
// workgroup has bytes in flight for a third of its life (then it computes on the VALU and combines its waves), and half
// of a mixed batch's grid is splits past a sequence's end (5.3 TB/s).  Here four single-wave workgroups per CU stay for
// the whole call.  All (kv head, sequence, 32-token unit) triples are laid end to end by a prefix sum of the lengths and
// cut in equal shares, one per wave, and a wave streams its share through a ring of two 16 KB stages in LDS (direct
// buffer->LDS loads with the non-temporal hint, without which it reads 5.7 instead of 6.3 TB/s), refilling a stage as
// soon as it has read it into registers.  Scores and P V run on the matrix cores (16 columns hold up to 8 query heads of
// the kv head, so larger groups cost no second read): about 15% of a wave's time, so nothing but the loads shows.
// Waves never meet: what a share cuts (at most its first and its last sequence) goes to a record per head, which
// decode_stream_merge_kernel merges by LSE; sequences inside one share are written directly.
//
// 64 sequences of 512 to 8192 tokens, 8 kv heads: 16-token pages 32 heads 217 -> 180 us (5.25 -> 6.3 TB/s), 64 heads
// 328 -> 185 us, contiguous 202 -> 179 us; 28 heads over 4 kv heads 390 -> 96 us.
#include <algorithm>

#include "decode_params.hpp"
#include "dtattn_common.hpp"

namespace dtattn {

namespace {

constexpr int kUnit = 32;      // tokens per stage of the ring
constexpr int kStreamHeads = 8;  // query heads of a kv head held in LDS
constexpr int kStreamD = 128;

// 16-byte chunk c of LDS row r sits at c ^ sswz(r): conflict-free for the 16-byte K reads (16 rows, one chunk) and the
// 8-byte transposed V reads (8 rows, two chunks).
__device__ __forceinline__ int sswz(int r) { return 2 * (r & 7) + ((r >> 3) & 1); }

__device__ __forceinline__ f32x4 mfma16(typename Elem<bf16_t>::vec8 a, typename Elem<bf16_t>::vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(typename Elem<f16_t>::vec8 a, typename Elem<f16_t>::vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int units_of(const DecodeParams& p, int64_t b) {
    return (min(max(p.lengths[b], 0), p.S_max) + kUnit - 1) / kUnit;
}

// Inclusive prefix sum over the wave's lanes.
__device__ __forceinline__ int wave_scan(int v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    return v;
}

// V units in `n` shares of V / n or one more (all the longer ones first); the host keeps V below 2^31.
struct Shares {
    int n, q, rem;
    __device__ __forceinline__ Shares(int V, int grid) {
        n = min(grid, max(1, V / 2));  // of two units or more
        q = V / n;
        rem = V - q * n;
    }
    __device__ __forceinline__ int start(int r) const { return r * q + min(r, rem); }
    __device__ __forceinline__ int of(int x) const {  // the share of unit x
        const int big = rem * (q + 1);
        return x < big ? x / (q + 1) : rem + (x - big) / q;
    }
};

}  // namespace

template <typename T, bool PAGED>
__global__ void __launch_bounds__(64, 1) decode_stream_kernel(const DecodeParams p) {
    typedef typename Elem<T>::vec8 V8;
    typedef typename Elem<T>::vec4 V4;
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    constexpr int D = kStreamD, NI = kUnit / 4;  // NI: 1 KB loads per stage of K and of V
    __shared__ __attribute__((aligned(16))) T kv[2][2][kUnit * D];
    __shared__ __attribute__((aligned(16))) T qs[2][kStreamHeads * D];

    const int lane = threadIdx.x;
    const int col = lane & 15, g4 = lane >> 4;
    const int G = p.group;
    // units of all sequences (the first 64 are kept: their prefix finds the share's start)
    const int own0 = lane < p.B ? units_of(p, lane) : 0;
    const int pre0 = wave_scan(own0);
    int U = __shfl(pre0, 63, 64);
    for (int j0 = 64; j0 < p.B; j0 += 64) U += __shfl(wave_scan(j0 + lane < p.B ? units_of(p, j0 + lane) : 0), 63, 64);
    U = __builtin_amdgcn_readfirstlane(U);
    if (U == 0) return;
    const Shares sh(U * p.Hkv, (int)gridDim.x);
    const int r = blockIdx.x;
    if (r >= sh.n) return;
    const int u0 = sh.start(r), n = sh.start(r + 1) - u0;  // first unit and units of this wave

    // The share's first sequence and token
    struct At {
        int hk, b, tok, L;
        bool first;  // the unit starts a segment
    };
    At at;
    at.hk = u0 / U;
    int x = u0 - at.hk * U;
    at.b = 0;
    for (int j0 = 0;; j0 += 64) {
        const int own = j0 == 0 ? own0 : j0 + lane < p.B ? units_of(p, j0 + lane) : 0;
        const int s = j0 == 0 ? pre0 : wave_scan(own);
        const uint64_t hit = __ballot(s > x);  // sequences ending past x
        if (hit != 0) {
            const int l = __builtin_ctzll(hit);
            at.b = __builtin_amdgcn_readfirstlane(j0 + l);
            x -= __builtin_amdgcn_readfirstlane(__shfl(s - own, l, 64));
            break;
        }
        x -= __builtin_amdgcn_readfirstlane(__shfl(s, 63, 64));
    }
    at.tok = x * kUnit;
    // lengths and page ids in the loop are scalar loads: a vector load's wait would drain the ring
    typedef const __attribute__((address_space(4))) int32_t cint32;
    cint32* const lengths = (cint32*)p.lengths;
    cint32* const table = (cint32*)p.block_table;
    auto length = [&](int b) { return min(max(lengths[b], 0), p.S_max); };
    at.L = length(at.b);
    at.first = true;
    auto next = [&](At a) {
        a.tok += kUnit;
        a.first = false;
        if (a.tok >= a.L) {
            a.tok = 0;
            a.first = true;
            do {  // a unit follows, so a sequence with tokens does
                if (++a.b == p.B) a.b = 0, ++a.hk;
                a.L = length(a.b);
            } while (a.L == 0);
        }
        return a;
    };

    const uint32_t kpitch = (uint32_t)(p.ks_s * sizeof(T)), vpitch = (uint32_t)(p.vs_s * sizeof(T));
    uint32_t koff[NI], voff[NI];  // of this lane's 16 bytes in load i: row 4 i + lane / 16, the chunk of its LDS slot
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int row = 4 * i + g4;
        const uint32_t c = (uint32_t)((col ^ sswz(row)) * 16);
        koff[i] = (uint32_t)(PAGED ? row & 15 : row) * kpitch + c;
        voff[i] = (uint32_t)(PAGED ? row & 15 : row) * vpitch + c;
    }
    uint32_t qoff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = 4 * i + g4;
        qoff[i] = row < G ? (uint32_t)(row * p.qs_h * (int64_t)sizeof(T)) + (uint32_t)((col ^ sswz(row)) * 16) : 0xfffffff0u;
    }
    auto issue = [&](int buf, const At& a) {
        if (a.first) {
            const auto qrs = make_rsrc(reinterpret_cast<const T*>(p.q) + a.b * p.qs_b + (int64_t)a.hk * G * p.qs_h,
                                       (uint32_t)((G - 1) * p.qs_h * (int64_t)sizeof(T)) + D * (uint32_t)sizeof(T));
#pragma unroll
            for (int i = 0; i < 2; ++i) buf_ld16_lds_async(qrs, &qs[buf][4 * i * D], qoff[i]);
        }
        const int rows = a.L - a.tok;  // valid rows of the unit, or more
        const T* kb = reinterpret_cast<const T*>(p.k) + (int64_t)a.hk * p.ks_h;
        const T* vb = reinterpret_cast<const T*>(p.v) + (int64_t)a.hk * p.vs_h;
        if constexpr (PAGED) {
            // 16 tokens lie in one page
            const int last = p.S_max - 1, mask = (1 << p.page_shift) - 1;
            const auto krs = make_rsrc(kb, p.kspan);
            const auto vrs = make_rsrc(vb, p.vspan);
            uint32_t kp[2], vp[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int t = min(a.tok + 16 * h, last);
                const int id = table[a.b * p.bt_s + (t >> p.page_shift)];
                const uint32_t pg = (uint32_t)min(max(id, 0), p.num_pages - 1), row = (uint32_t)((a.tok + 16 * h) & mask);
                kp[h] = pg * (uint32_t)(p.ks_b * sizeof(T)) + row * kpitch;
                vp[h] = pg * (uint32_t)(p.vs_b * sizeof(T)) + row * vpitch;
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const bool ok = 4 * i + g4 < rows;  // rows past the sequence end load as zeros
                buf_ld16_lds_async_nt(krs, &kv[buf][0][4 * i * D], ok ? kp[i / 4] + koff[i] : p.kspan);
                buf_ld16_lds_async_nt(vrs, &kv[buf][1][4 * i * D], ok ? vp[i / 4] + voff[i] : p.vspan);
            }
        } else {
            const int m = min(rows, kUnit) - 1;
            const uint32_t kn = (uint32_t)m * kpitch + D * (uint32_t)sizeof(T), vn = (uint32_t)m * vpitch + D * (uint32_t)sizeof(T);
            const auto krs = make_rsrc(kb + a.b * p.ks_b + a.tok * p.ks_s, kn);
            const auto vrs = make_rsrc(vb + a.b * p.vs_b + a.tok * p.vs_s, vn);
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const bool ok = 4 * i + g4 < rows;
                buf_ld16_lds_async_nt(krs, &kv[buf][0][4 * i * D], ok ? koff[i] : kn);
                buf_ld16_lds_async_nt(vrs, &kv[buf][1][4 * i * D], ok ? voff[i] : vn);
            }
        }
    };

    float M = kNegInf, m = kNegInf, l = 0.f;  // running max, base of acc, row sum (base M)
    f32x4 acc[8];
    V8 qf[4];
    int start = 0;        // the segment's first token
    bool cut_first = true;  // the segment is the share's first
    At cur = at, ahead = at;
    issue(0, ahead);
    if (n > 1) {
        ahead = next(ahead);
        issue(1, ahead);
    }
    At nxt = ahead;
    for (int s = 0; s < n; ++s) {
        const int buf = s & 1;
        // stage s has landed when at most the 16 loads of stage s + 1 are left
        if (s + 1 < n) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (cur.first || s == 0) {
            const int row = col & 7;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                qf[k] = __builtin_bit_cast(V8, q_bits(ld16(&qs[buf][row * D + 8 * ((4 * k + g4) ^ sswz(row))]), p.q_and, p.q_xor));
            M = m = kNegInf;
            l = 0.f;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
            start = cur.tok;
            cut_first = s == 0;
        }
        const T* K = kv[buf][0];
        const T* Vt = kv[buf][1];
        V8 kf[2][4], vf[8];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int row = 16 * tt + col;
                kf[tt][k] = __builtin_bit_cast(V8, ld16(K + row * D + 8 * ((4 * k + g4) ^ sswz(row))));
            }
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
            const int R = 4 * g4 + (col >> 2), c = (2 * dt + ((col & 3) >> 1)) ^ sswz(R);
            const int off = R * D + 8 * c + 4 * (col & 1);
            const V4 lo = __builtin_bit_cast(V4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(Vt + off)));
            const V4 hi = __builtin_bit_cast(V4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(Vt + off + 16 * D)));
            vf[dt] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage is in registers: its buffer takes stage s + 2
        if (s + 2 < n) {
            ahead = next(ahead);
            issue(buf, ahead);
        }
        f32x4 sc[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            sc[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 4; ++k) sc[tt] = mfma16(kf[tt][k], qf[k], sc[tt]);
        }
        const int left = cur.L - cur.tok;
        if (left < kUnit) {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (16 * tt + 4 * g4 + i >= left) sc[tt][i] = kNegInf;
        }
        float mx = kNegInf;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sc[tt][i]);
        mx = max_across_groups<16>(mx);
        // acc's base is the unit's own max, not the running one, so that its largest P is 1 and rounds exactly (error of O
        // against 64 bits at the sizes above 2.0e-3; with the running max 2.2e-3; the split form 2.1e-3); at most 2^24
        // below the running max, which keeps alpha and O finite.  The row sum stays on the running max: rescaled every
        // unit it would collect an exponential's rounding each time.
        const float Mnew = fmaxf(M, mx * p.c);
        const float mnew = fmaxf(mx * p.c, Mnew - 24.f);
        const float mbase = mnew == kNegInf ? 0.f : mnew;
        const float alpha = fast_exp2(m - mbase);
        m = mnew;
        float us = 0.f;
        V8 pk;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float pv = fast_exp2(__builtin_fmaf(sc[tt][i], p.c, -mbase));
                us += pv;
                pk[4 * tt + i] = Elem<T>::from_f32(pv);
            }
        const float Mbase = Mnew == kNegInf ? 0.f : Mnew;
        l = __builtin_fmaf(us, fast_exp2(m - Mbase), l * fast_exp2(M - Mbase));
        M = Mnew;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
            acc[dt] *= alpha;
            acc[dt] = mfma16(vf[dt], pk, acc[dt]);
        }
        const bool ends = left <= kUnit;  // the sequence's last unit
        if (ends || s + 1 == n) {
            const float lt = sum_across_groups<16>(l);
            float inv = 1.f / (lt * fast_exp2(M - m));
            if (col < G) {
                const int hq = cur.hk * G + col;
                const float lse = __builtin_fmaf(M, kLn2, __log2f(lt) * kLn2);
                if (ends && start == 0) {  // the whole sequence
                    T* o = reinterpret_cast<T*>(p.o) + cur.b * p.os_b + hq * p.os_h;
#pragma unroll
                    for (int dt = 0; dt < 8; ++dt) {
                        V4 o4;
#pragma unroll
                        for (int i = 0; i < 4; ++i) o4[i] = Elem<T>::from_f32(acc[dt][i] * inv);
                        *reinterpret_cast<V4*>(o + 16 * dt + 4 * g4) = o4;
                    }
                    if (p.lse != nullptr && g4 == 0) p.lse[cur.b * p.lses_b + hq] = lse;
                } else {
                    const int64_t rec = (int64_t)(2 * r + (cut_first ? 0 : 1)) * G + col;
                    if (lt == 0.f) inv = 0.f;  // every score is -inf: O = 0, not 0 / 0, at the LSE of -inf that drops it
#pragma unroll
                    for (int dt = 0; dt < 8; ++dt)
                        *reinterpret_cast<f32x4*>(p.part_o + rec * D + 16 * dt + 4 * g4) = acc[dt] * inv;
                    if (g4 == 0) p.part_lse[rec] = lse;
                }
            }
        }
        cur = nxt;
        nxt = ahead;
    }
}

// Merges the records of the shares that cut a sequence, one (b, query head) per W waves; W = 4 for small batches, whose
// sequences are cut often (one of 32768 tokens into 128 pieces per head: 36.1 -> 30.0 us a call).
template <typename T, int W>
__global__ void __launch_bounds__(256) decode_stream_merge_kernel(const DecodeParams p, int shares) {
    constexpr int D = kStreamD;
    __shared__ float red[W > 1 ? W : 1][D];
    const int lane = threadIdx.x & 63, wave = W > 1 ? threadIdx.x >> 6 : 0;
    const int64_t pair = W > 1 ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (pair >= (int64_t)p.B * p.Hq) return;
    const int b = (int)(pair / p.Hq), hq = (int)(pair % p.Hq), hk = hq / p.group;
    int U = 0, before = 0, own = 0;
    for (int j0 = 0; j0 < p.B; j0 += 64) {
        const int u = j0 + lane < p.B ? units_of(p, j0 + lane) : 0;
        const int s = wave_scan(u);
        if (b >= j0 && b < j0 + 64) {
            own = __shfl(u, b - j0, 64);
            before = U + __shfl(s, b - j0, 64) - own;
        }
        U += __shfl(s, 63, 64);
    }
    T* op = reinterpret_cast<T*>(p.o) + b * p.os_b + hq * p.os_h;
    if (own == 0) {  // empty sequence: O = 0, LSE = -inf
        if (wave == 0) {
            op[2 * lane] = op[2 * lane + 1] = Elem<T>::from_f32(0.f);
            if (p.lse != nullptr && lane == 0) p.lse[b * p.lses_b + hq] = kNegInf;
        }
        return;
    }
    const Shares sh(U * p.Hkv, shares);
    const int x0 = hk * U + before, r0 = sh.of(x0), r1 = sh.of(x0 + own - 1);
    if (r0 == r1) return;
    const int ns = r1 - r0 + 1;
    // share r0 holds this sequence in its first segment only if it begins with it
    const int slot0 = sh.start(r0) < x0 ? 1 : 0;
    auto rec = [&](int j) { return (int64_t)(2 * (r0 + j) + (j == 0 ? slot0 : 0)) * p.group + hq % p.group; };
    float mx = kNegInf;
    for (int j = lane; j < ns; j += 64) mx = fmaxf(mx, p.part_lse[rec(j)]);
    mx = wave_max(mx);
    float sum = 0.f;
    for (int j = lane; j < ns; j += 64) sum += __expf(p.part_lse[rec(j)] - mx);
    sum = wave_sum(sum);
    const float inv = 1.f / sum;
    float a0 = 0.f, a1 = 0.f;
    constexpr int MB = 8;  // records in flight
    for (int j0 = wave; j0 < ns; j0 += W * MB) {
        float lw[MB], v0[MB], v1[MB];
#pragma unroll
        for (int j = 0; j < MB; ++j) {
            const int64_t q = rec(min(j0 + W * j, ns - 1));
            lw[j] = p.part_lse[q];
            v0[j] = p.part_o[q * D + 2 * lane];
            v1[j] = p.part_o[q * D + 2 * lane + 1];
        }
#pragma unroll
        for (int j = 0; j < MB; ++j) {
            const float w = j0 + W * j < ns ? __expf(lw[j] - mx) * inv : 0.f;
            a0 = __builtin_fmaf(w, v0[j], a0);
            a1 = __builtin_fmaf(w, v1[j], a1);
        }
    }
    if constexpr (W > 1) {
        red[wave][2 * lane] = a0;
        red[wave][2 * lane + 1] = a1;
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int w = 1; w < W; ++w) a0 += red[w][2 * lane], a1 += red[w][2 * lane + 1];
    }
    op[2 * lane] = Elem<T>::from_f32(a0);
    op[2 * lane + 1] = Elem<T>::from_f32(a1);
    if (p.lse != nullptr && lane == 0) p.lse[b * p.lses_b + hq] = mx + __logf(sum);
}

int stream_cus(hipStream_t stream) {
    int dev = 0;
    dtattn_device_peaks pk;
    if ((stream == nullptr ? hipGetDevice(&dev) : hipStreamGetDevice(stream, &dev)) != hipSuccess) return 0;
    return dtattn_get_device_peaks(dev, &pk) == DTATTN_OK ? pk.cu_count : 0;
}

// Shares (workgroups of one wave): four per CU, and no more than the records of two cut sequences each that the
// split form's workspace holds.
static int stream_shares(const DecodeParams& p, hipStream_t stream) {
    return (int)std::min<int64_t>(4 * (int64_t)stream_cus(stream), (int64_t)p.B * p.Hkv * ((p.S_max + 127) / 128) / 2);
}

// Units per CU from which it is faster, by the capacity (the host does not know the lengths).  Its fixed cost is about 3 us
// above the split form's, which reads a chunk twice for 8 heads, three times for 6 and 3, and 5 and 7 times for 5 and 7, and
// keeps up longest where every head reads its own cache.  A line is where the form wins on full caches and loses little
// on half-full ones.  us, 384-token splits (the form's own alternative above 2560 tokens) / streaming, full and half full:
//   1: contiguous 16x8192 340 / 339 and 16x512 in 8192 30 / 33, 64x512 91 / 101: never; pages of 16 tokens 64x512 99 / 86,
//      64x2048 365 / 329, 16x2048 mixed 53 / 49
//   2: 64x2048 94 / 88, 16x8192 mixed 53 / 50 (128 units); 16x2048 26.7 / 27.3 (32)
//   3: 4x3072 16.8 / 17.1 and 11.7 / 12.3 (12 units); 4x3840 20.9 / 17.4 and 11.8 / 12.6, 16x960 21.6 / 17.8 and 14.1 / 13.0 (15)
//   4: 4x2912 15.1 / 17.3 (11); 4x3680 20.9 / 17.6 and 13.7 / 13.2 (14); up to 384 tokens 64x384 19.8 / 23.3 (24), 3: 64x256
//      19.8 / 23.4 (16): never
//   5: 4x2048 16.9 / 16.3 and 9.8 / 12.0 (8); 4x3072 22.4 / 17.3 and 13.1 / 12.4 (12);  6: 4x2048 16.6 / 16.2 and 11.4 / 12.0 (8);
//      4x3072 20.0 / 17.3 and 12.2 / 12.5 (12)
//   7: 4x2048 14.9 / 16.2 (4); 4x3072 20.1 / 16.1 and 12.3 / 11.9, 64x192 20.1 / 11.7 (6)
//   8: 4x1536 14.2 / 16.2 (6); 2x3936 19.8 / 16.8 and 12.4 / 12.8, 16x448 19.1 / 15.4 (7)
// Lengths far below the capacity (a sixteenth and less) cost it up to 3.5 us (7: 1x2048 in 32768 8.3 / 10.0; 3: 4x256 in 4096
// 6.3 / 9.6), in groups of 4 and 8 nothing (4: 1x2048 in 32768 11.9 / 9.9).
bool decode_stream_pays(int64_t B, int64_t Hkv, int64_t S_max, int64_t group, bool paged, hipStream_t stream) {
    if (group > kStreamHeads || (group == 1 && !paged)) return false;
    if (group <= 4 && S_max <= 384) return false;  // one split per sequence and no merge
    const int64_t per_cu = group == 8 ? 7 : group == 7 ? 6 : group >= 5 ? 12 : group >= 3 ? 15 : 124;
    const int cus = stream_cus(stream);
    return cus > 0 && B * Hkv * ((S_max + kUnit - 1) / kUnit) >= per_cu * cus;
}

bool decode_stream_fits(const DecodeParams& p, int32_t dtype, size_t ws_bytes, hipStream_t stream) {
    if ((dtype != DTATTN_BF16 && dtype != DTATTN_FP16) || p.d_real != kStreamD || p.group > kStreamHeads) return false;
    if (p.block_table != nullptr && (p.kspan == 0 || p.page_shift < 4)) return false;
    // 16-byte loads straight into LDS and 8-byte stores (the entry points check strides, not pointers)
    if (((reinterpret_cast<uintptr_t>(p.q) | reinterpret_cast<uintptr_t>(p.k) | reinterpret_cast<uintptr_t>(p.v)) & 15u) != 0) return false;
    if ((reinterpret_cast<uintptr_t>(p.o) & 7u) != 0 || p.os_b % 4 != 0 || p.os_h % 4 != 0) return false;
    if (p.qs_h < 0 || p.qs_h * p.group >= (1 << 28) || p.ks_s < 0 || p.vs_s < 0) return false;
    if (!decode_stream_pays(p.B, p.Hkv, p.S_max, p.group, p.block_table != nullptr, stream)) return false;
    if ((int64_t)p.B * p.Hkv * ((p.S_max + kUnit - 1) / kUnit) >= ((int64_t)1 << 31)) return false;
    const int n = stream_shares(p, stream);
    return n > 0 && (size_t)(2 * n) * p.group * (kStreamD + 1) * sizeof(float) <= ws_bytes;
}

template <typename T>
static int launch_stream(const DecodeParams& p, int n, hipStream_t stream) {
    if (p.block_table != nullptr)
        hipLaunchKernelGGL((decode_stream_kernel<T, true>), dim3((unsigned)n), dim3(64), 0, stream, p);
    else
        hipLaunchKernelGGL((decode_stream_kernel<T, false>), dim3((unsigned)n), dim3(64), 0, stream, p);
    const int st = check_launch("decode_stream_kernel");
    if (st != DTATTN_OK) return st;
    const int64_t pairs = (int64_t)p.B * p.Hq;
    if (pairs <= 256)
        hipLaunchKernelGGL((decode_stream_merge_kernel<T, 4>), dim3((unsigned)pairs), dim3(256), 0, stream, p, n);
    else
        hipLaunchKernelGGL((decode_stream_merge_kernel<T, 1>), dim3((unsigned)((pairs + 3) / 4)), dim3(256), 0, stream, p, n);
    return check_launch("decode_stream_merge_kernel");
}

int decode_stream(const DecodeParams& p0, int32_t dtype, void* ws, hipStream_t stream) {
    DecodeParams p = p0;
    const int n = stream_shares(p, stream);
    p.part_o = reinterpret_cast<float*>(ws);
    p.part_lse = p.part_o + (int64_t)2 * n * p.group * kStreamD;
    return dtype == DTATTN_BF16 ? launch_stream<bf16_t>(p, n, stream) : launch_stream<f16_t>(p, n, stream);
}

}  // namespace dtattn
