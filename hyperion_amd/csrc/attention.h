// Parameters shared by the attention kernels (attention.hip: decode, the merges and the
// dispatch; attention_chunk.hip: chunks).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace hyperion::hip {

constexpr uint32_t kKeyBlock = 32;
constexpr float kLog2e = 1.4426950408889634f;

struct AttnParams {
    const uint16_t* q;      // [L][H][D]
    const uint16_t* k;      // [L][KVH][D]: the chunk, or null when it is in the cache
    const uint16_t* v;
    const uint16_t* ck;     // [cap][KVH][D]: the cache
    const uint16_t* cv;
    uint16_t* out;          // [L][H][D]
    float* part_o;          // split partials: [splits][L * H][D]
    float* part_ml;         // [splits][L * H][2]
    uint32_t L, H, KVH, G, cap, offset, prefix, window;
    uint32_t splits, keys_per_split;
    const uint32_t* pos;    // non-null: offset = *pos, read on the device (graph replays)
    // The decode form with the prepare folded in (L = 1): q is the raw projection; each
    // wave normalises and rotates its query rows, and the wave whose keys hold the new
    // token forms its K/V from k_raw/v_raw and writes them to the cache slot.
    const float2* rope_cs;  // (cos, sin) [positions][D / 2]
    const uint16_t* q_w;    // [D]
    const uint16_t* k_w;    // [D]
    const uint16_t* k_raw;  // [KVH][D]
    const uint16_t* v_raw;  // [KVH][D], or null: V = v_norm(k_raw)
    uint16_t* ck_out;       // the cache, written at the new token's slot
    uint16_t* cv_out;
    float eps;
};

// Graph-replay form: the position comes from device memory, the prefix and the split
// length follow from it as the host computes them (prefix = min(window, offset) with a
// window, offset without; keys split evenly in whole key blocks over the fixed grid).
__device__ __forceinline__ void resolve_position(AttnParams& p) {
    if (p.pos == nullptr) return;
    p.offset = *p.pos;
    p.prefix = p.window != 0u ? min(p.window, p.offset) : p.offset;
    const uint32_t T = p.prefix + p.L;
    p.keys_per_split = ((T + p.splits - 1u) / p.splits + kKeyBlock - 1u) / kKeyBlock * kKeyBlock;
}

// The chunk form (attention_chunk.hip): workgroups of kChunkRows query rows of one kv head,
// each row tile's keys over p.splits workgroups.
constexpr uint32_t kChunkRows = 128;
void launch_attn_chunk(const AttnParams& p, uint32_t head_dim, hipStream_t stream);

}  // namespace hyperion::hip
