// Parameters of the decode kernels (decode_splitkv.hip, decode_stream.hip).
#pragma once
#include "dtattn_common.hpp"

namespace dtattn {

struct DecodeParams {
    const void* q;
    const void* k;
    const void* v;
    const int32_t* lengths;
    void* o;
    float* lse;
    float* part_o;    // [B, Hq, nsplit, D]
    float* part_lse;  // [B, Hq, nsplit]
    int64_t qs_b, qs_h;
    int64_t ks_b, ks_h, ks_s;
    int64_t vs_b, vs_h, vs_s;
    int64_t os_b, os_h;
    int64_t lses_b;
    int32_t B, Hq, Hkv, S_max, group;
    int32_t chunk, nsplit;
    float c;  // scale * log2(e)
    // paged cache: token t of sequence b is row t & (2^page_shift - 1) of page
    // block_table[b * bt_s + (t >> page_shift)]; ks_b / vs_b are then the page strides
    const int32_t* block_table;
    int64_t bt_s;
    int32_t page_shift, num_pages;
    // bytes from a kv head's base to the end of its last page row (K, V), when every page offset fits 32 bits
    // (strides >= 0, span < 2^32): the paged loads then go through buffer resources; 0: 64-bit flat loads
    uint32_t kspan, vspan;
    // real head dim (<= the kernel's D; a multiple of 16 bytes of elements) and its 16-byte chunks
    int32_t d_real, d_ch;
    uint32_t q_and, q_xor;  // applied to q's words at load, as in ScalePlan
};

// CUs of the stream's device (0: unknown).
int stream_cus(hipStream_t stream);
// Whether a 16-bit call at head dim 128 is large enough for the streaming form.
bool decode_stream_pays(int64_t B, int64_t Hkv, int64_t S_max, int64_t group, bool paged, hipStream_t stream);
// The streaming form (decode_stream.hip): whether a call on the current device takes it (its partials fit `ws_bytes`),
// and its two launches.
bool decode_stream_fits(const DecodeParams& p, int32_t dtype, size_t ws_bytes, hipStream_t stream);
int decode_stream(const DecodeParams& p, int32_t dtype, void* ws, hipStream_t stream);

}  // namespace dtattn
