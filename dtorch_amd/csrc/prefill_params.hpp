// Launch parameters shared by the bf16/fp16 and fp32 prefill kernels (prefill_fwd.hip,
// prefill_f32.hip): pointers, [B, H, S] element strides, sizes and the softmax constants, filled once
// by dtattn_prefill_fwd.
#pragma once

#include "dtattn_common.hpp"

namespace dtattn {

struct PrefillParams {
    const void* q;
    const void* k;
    const void* v;
    void* o;
    float* lse;
    int64_t qs_b, qs_h, qs_s;
    int64_t ks_b, ks_h, ks_s;
    int64_t vs_b, vs_h, vs_s;
    int64_t os_b, os_h, os_s;
    int64_t lses_b, lses_h;
    int32_t B, Hq, Hkv, Sq, Sk, group;
    int32_t n_qblocks;
    int32_t delta;  // key j visible to query i iff j <= i + delta (causal only)
    float c;        // softmax scale * log2(e)
    int32_t xcd_map;  // 1: group the workgroups of each (batch, kv head) slice on one XCD
    // additive attention mask (MASKED kernels): element (b, h, i, j) at index b*ms_b + h*ms_h + i*ms_l + j of
    // `mask` (key stride 1); it enters the raw scores as m / scale, so -inf and the dtype-minimum fills both
    // hide a key.  mask_kind: its element type (DTATTN_FP32, BF16, FP16 or BOOL); base and rows need no alignment
    // beyond the element's.
    const void* mask;
    int64_t ms_b, ms_h, ms_l;
    int32_t mask_kind;
    // Key spans of a mask that is one row for all queries and heads (mask_spans_kernel), or NULL: entry b is the
    // [first, last + 1) visible keys of batch b when the mask hides every key outside and adds nothing inside,
    // else (0, -1).  The head-dim-128 kernels run the first kind as shorter calls, prefill_fwd_kernel the rest.
    const int2* spans;
    float inv_scale;
    // Head dims below the kernel's D (PAD kernels): Q/K rows hold qk_ch valid 16-byte chunks and V/O rows
    // v_ch; the chunks past them load as zeros (adding nothing to the scores, giving O columns that are
    // never stored).
    int32_t qk_ch, v_ch;
    // Key blocks (wide kernel): workgroup (x, y) takes keys [y kblock, (y + 1) kblock) and writes its
    // partial O and LSE at o + y os_split, lse + y lses_split; nsplit = 1 is the unsplit launch.
    int32_t nsplit, kblock;
    int64_t os_split, lses_split;
    // q's words pass through (w & q_and) ^ q_xor at load: negation or zeroing for scales <= 0
    uint32_t q_and, q_xor;
};

// Lazy rescaling: the running max only moves (and O, l are only rescaled) when some row's max grew
// by more than 2^8; otherwise P is taken against the stale max (values up to 2^8, exact in the
// normalisation, which uses the same max for O and l).
constexpr float kRescaleThreshold = 8.0f;

// How a kernel instantiation reads its mask: none, fp32, or as stored.  One instantiation per type: choosing it per
// element costs 100 instructions a tile at 64 keys (dense bf16 mask, 4x32x2000 at D = 128: 396 against 346 us for
// the fp32 form and its conversion).
enum MaskMode { kMaskNone = 0, kMaskF32 = 1, kMaskBool = 2, kMaskBf16 = 3, kMaskF16 = 4 };

inline MaskMode mask_mode(const PrefillParams& p) {
    if (p.mask == nullptr) return kMaskNone;
    switch (p.mask_kind) {
        case DTATTN_BOOL: return kMaskBool;
        case DTATTN_BF16: return kMaskBf16;
        case DTATTN_FP16: return kMaskF16;
        default: return kMaskF32;
    }
}

// The mask slab of one (batch, head) for a lane that reads its own query row, four consecutive keys at a time.
// fp32: one 16-byte load per group.  As stored: rows start at any byte, so a group is the two (bool) or three
// aligned words around it, shifted into place when they are used; the resource ends with the word that holds
// the slab's last element.  Reads past it return 0; those keys are hidden by the ragged-tail mask anyway.
template <int MODE>
struct MaskSlab {
    static constexpr int kWords = MODE == kMaskBool ? 2 : MODE == kMaskF32 ? 4 : 3;
    typedef uint32_t Group __attribute__((ext_vector_type(kWords)));
    __amdgpu_buffer_rsrc_t rs;
    uint32_t row;    // byte offset of the lane's row in the resource, at its first word
    uint32_t shift;  // of the row's first element in that word (groups of 4 keys keep it)

    __device__ __forceinline__ MaskSlab(const PrefillParams& p, int b, int hq, int qrow) {
        constexpr int esz = MODE == kMaskBool ? 1 : MODE == kMaskF32 ? 4 : 2;
        const uint64_t base = (uint64_t)(uintptr_t)p.mask + (uint64_t)((b * p.ms_b + hq * p.ms_h) * esz);
        const uint32_t mis = (uint32_t)base & 3u;
        const uint64_t bytes = (uint64_t)((int64_t)(p.Sq - 1) * p.ms_l + p.Sk) * (uint64_t)esz;
        rs = make_rsrc(reinterpret_cast<const void*>((uintptr_t)(base - mis)), (uint32_t)((bytes + mis + 3) & ~(uint64_t)3));
        row = (uint32_t)((int64_t)min(qrow, p.Sq - 1) * p.ms_l * esz) + mis;
        shift = row & 3u;
        row &= ~3u;
    }
    // keys key .. key + 3; key is a multiple of 4
    __device__ __forceinline__ Group load(int key) const {
        if constexpr (MODE == kMaskBool)
            return __builtin_bit_cast(Group, __builtin_amdgcn_raw_buffer_load_b64(rs, row + (uint32_t)key, 0, 0));
        else if constexpr (MODE == kMaskF32)
            return buf_ld16(rs, row + (uint32_t)(key * 4));
        else
            return __builtin_bit_cast(Group, __builtin_amdgcn_raw_buffer_load_b96(rs, row + (uint32_t)(key * 2), 0, 0));
    }
    // The group's four bytes of a bool mask, in key order.
    __device__ __forceinline__ uint32_t bytes(Group g) const { return __builtin_amdgcn_alignbyte(g[1], g[0], shift); }
    // s0..s3 += mask / scale
    __device__ __forceinline__ void add(Group g, float inv_scale, float& s0, float& s1, float& s2, float& s3) const {
        if constexpr (MODE == kMaskBool) {
            // Any non-zero byte keeps its key: bit 7 of `nz` says so for each byte (the sum cannot carry into the next
            // one); sign-extended and inverted over -inf's bits it is +0 or -inf
            const uint32_t w = bytes(g);
            const int nz = (int)(((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w);
            auto m = [](int keep) { return __builtin_bit_cast(float, (uint32_t)~keep & 0xff800000u); };
            s0 += m(nz << 24 >> 31), s1 += m(nz << 16 >> 31), s2 += m(nz << 8 >> 31), s3 += m(nz >> 31);
        } else if constexpr (MODE == kMaskF32) {
            const f32x4 m = __builtin_bit_cast(f32x4, g);
            s0 += m.x * inv_scale, s1 += m.y * inv_scale, s2 += m.z * inv_scale, s3 += m.w * inv_scale;
        } else {
            const uint32_t lo = __builtin_amdgcn_alignbyte(g[1], g[0], shift);
            const uint32_t hi = __builtin_amdgcn_alignbyte(g[2], g[1], shift);
            if constexpr (MODE == kMaskBf16) {
                s0 += __builtin_bit_cast(float, lo << 16) * inv_scale;
                s1 += __builtin_bit_cast(float, lo & 0xffff0000u) * inv_scale;
                s2 += __builtin_bit_cast(float, hi << 16) * inv_scale;
                s3 += __builtin_bit_cast(float, hi & 0xffff0000u) * inv_scale;
            } else {
                const f16x2 a = __builtin_bit_cast(f16x2, lo), c = __builtin_bit_cast(f16x2, hi);
                s0 += (float)a.x * inv_scale, s1 += (float)a.y * inv_scale;
                s2 += (float)c.x * inv_scale, s3 += (float)c.y * inv_scale;
            }
        }
    }
};

template <bool CAUSAL>
__device__ __forceinline__ BlockCoord block_coord(const PrefillParams& p) {
    return block_coord<CAUSAL>(p.B, p.Hq, p.Hkv, p.group, p.n_qblocks, p.xcd_map);
}

}  // namespace dtattn
