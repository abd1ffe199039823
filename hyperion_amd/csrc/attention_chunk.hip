// Attention of a chunk of query tokens (prefill, and any call with more than 16 query rows
// per KV head) on gfx950: the semantics of attention.hip, flash-attention style on
// v_mfma_f32_32x32x16_bf16.
//
// A workgroup (4 waves) takes kChunkRows = 128 query rows of one kv head - row r is token
// r / G, head-in-group r % G - and walks their visible keys in blocks of 32, each wave with
// 32 rows of its own:
//  * Scores are formed transposed, S^T = K Q^T: K rows are the A operand (read from LDS), the
//    wave's Q rows the B operand, in registers for the whole walk. A lane then holds 16 of
//    the block's keys for one query row, so the row maximum and sum are in-lane chains and
//    one exchange with lane ^ 32.
//  * The output is transposed too, O^T = V^T P^T: the 16 probabilities of a lane, rounded to
//    bf16, are its B operand as they stand (no trip through LDS), for the key order
//    16 t + 8 (e / 4) + 4 (lane / 32) + e % 4 of step t's element e; the V^T operand takes the
//    same keys by transposing reads (ds_read_b64_tr_b16) of V rows as loaded.
//  * K and V rows go straight to LDS (16-byte loads with the LDS as destination), two stages,
//    one barrier per block: the next block lands while this one computes. Rows are not
//    padded; their 16-byte chunks are XOR-swizzled (k_swz, v_swz) so that the rows one read
//    touches lie on different banks.
//  * Online softmax: up to head_dim 256 O is rescaled to the running maximum on every block,
//    each tile in the shadow of the products before its own. At head_dim 512 O is in
//    accumulation registers (three instructions a value), and is rescaled only when some
//    row's maximum has grown by more than 2^kRescaleLog2 since the last time. The largest
//    probability is then no longer the exact 1 of a running maximum: rounded to bf16 against an
//    unrounded denominator it would leave a row that one key dominates an error of 2.3e-3
//    where the running maximum's is 1.7e-3 (128 keys, the key 4 to 8 octaves above those before
//    it). So every probability enters as two bf16 terms (1.66e-3 there, and 4% below the
//    running maximum on random rows), at 364 us against 324 with second terms for half of the
//    keys, on the first case below (the other half's behind a test of whether one of them can
//    dominate, with V read again for it: 364 as well, and 73 against 65 us for 203 tokens
//    behind 3000). A block that outgrows the reference takes its score products
//    twice: 2048 tokens behind 2048 in 391 us on random rows, 453 with their scores' deviation
//    four times that, 632 where every block of every row does.
//  * Operands are read from LDS four products ahead of their use, and the next block's loads
//    go out between the score products.
//
// What bounds it: each wave reads every K and V byte of a block from LDS (64 KB a block and
// wave at head_dim 512 for 3072 matrix-core cycles), so the 32 rows a wave holds - the most
// its 512 registers allow at head_dim 512: 256 of O, 128 of Q - set the LDS traffic. With one
// wave per SIMD at head_dim 512 the softmax between the two products is exposed. Measured, the
// whole call with its merge, against 16 rows per wave on 16x16x32 products with V transposed
// or read behind each product: 16 heads, 2048 tokens behind 2048 at head_dim 512 (one kv head)
// 1110 -> 364 us (186 -> 566 TFLOP/s); 1000 behind 700 at head_dim 256 (8 kv heads, window 1024)
// 118 -> 44 us. Without the reads ahead of use a third slower.
#include "attention.h"
#include "attention_plan.h"
#include "common.h"
#include "kernels.h"

namespace hyperion::hip {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));
typedef short short4_t __attribute__((ext_vector_type(4)));

constexpr uint32_t kThreads = 256;
constexpr uint32_t kWaveRows = 32;
constexpr float kRescaleLog2 = 8.0f;

#define HYP_LDS __attribute__((address_space(3)))
#define HYP_GLOBAL __attribute__((address_space(1)))

template <uint32_t D>
struct ChunkLds {
    static constexpr uint32_t kRow = D * 2u;                 // one K or V row (bytes)
    static constexpr uint32_t kChunks = D / 8u;              // its 16-byte chunks
    static constexpr uint32_t kV = kKeyBlock * kRow;         // V behind K in a stage
    static constexpr uint32_t kStage = 2u * kKeyBlock * kRow;
    static constexpr uint32_t kOutRow = D * 2u + 16u;        // output staging rows (padded)
    static constexpr uint32_t kOut = kChunkRows * kOutRow;
    static constexpr uint32_t kBytes = 2u * kStage > kOut ? 2u * kStage : kOut;
    // K operand reads touch 32 rows at one logical chunk; V operand reads 4 or 8 rows (key
    // 4 h + 0..3) at 32 or 64 bytes.
    static constexpr uint32_t k_swz(uint32_t row) { return (row & 15u) & (kChunks - 1u); }
    static constexpr uint32_t v_swz(uint32_t row) { return (((row & 3u) << 2) | ((row >> 1) & 2u)) & (kChunks - 1u); }
};

// The other half-wave's value (lane ^ 32) combined with this lane's.
__device__ __forceinline__ float half_max(float v) {
    float u = v, c = v;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(u), "+v"(c));
    return fmaxf(u, c);
}

__device__ __forceinline__ float half_sum(float v) {
    float u = v, c = v;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(u), "+v"(c));
    return u + c;
}

__device__ __forceinline__ bf16x8_t lds_read16(uint32_t at) {
    return *reinterpret_cast<const HYP_LDS bf16x8_t*>(at);
}

// A transposing read. The pointer is restrict so that the read carries alias information:
// without any, the compiler puts a wait for the loads to LDS in flight (the next block's)
// ahead of it. The block's own loads are waited for explicitly.
__device__ __forceinline__ short4_t lds_read_tr4(HYP_LDS short4_t* __restrict at) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(at);
}

// 8 keys of one dim per lane (two transposing reads of 4 keys, `hi` bytes apart).
__device__ __forceinline__ bf16x8_t lds_read_tr(uint32_t at, uint32_t hi) {
    const short4_t a = lds_read_tr4(reinterpret_cast<HYP_LDS short4_t*>(at));
    const short4_t b = lds_read_tr4(reinterpret_cast<HYP_LDS short4_t*>(at + hi));
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Eight probabilities rounded to bf16, a lane's operand of one product.
__device__ __forceinline__ bf16x8_t round_p(const float* p) {
    return __builtin_bit_cast(bf16x8_t, make_uint4(cvt_pk_bf16(p[0], p[1]), cvt_pk_bf16(p[2], p[3]),
                                                   cvt_pk_bf16(p[4], p[5]), cvt_pk_bf16(p[6], p[7])));
}

// One query row again, over its visible keys [j0, j1) of this split alone, against the same
// reference: the matrix products take masked keys with a probability of 0, which a value of V
// that is not finite turns into NaN (and the two terms of a probability make NaN of an
// infinity). Four keys at a time, one per 16 lanes, the next four in flight; fp32 throughout.
// The sums stay unnormalised, dims 64 c + 4 (lane % 16) + e of o[c][e], in every lane. Rare and
// slow: 2048 tokens behind 2048 at head_dim 512 with one such value 18 ms.
template <uint32_t D>
__device__ __forceinline__ void row_alone(const AttnParams& p, uint32_t hk, size_t orow, uint32_t j0, uint32_t j1,
                                          float ref, uint32_t lane, float (&o)[D / 64u][4]) {
    constexpr uint32_t kC = D / 64u;
    const uint32_t at = (lane & 15u) * 4u;
    const uint16_t *ck = p.ck, *cv = p.cv, *pk = p.k, *pv = p.v;   // (selected by value, not through memory)
    const auto load = [&](const uint16_t* row, uint2 (&raw)[kC]) {
#pragma unroll
        for (uint32_t c = 0; c < kC; ++c) raw[c] = *reinterpret_cast<const uint2*>(row + 64u * c + at);
    };
    const auto value = [](const uint2& w, int e) {
        const uint32_t two = e < 2 ? w.x : w.y;
        return (e & 1) != 0 ? __uint_as_float(two & 0xFFFF0000u) : bf16_bits_to_f32(two & 0xFFFFu);
    };
    const auto load_keys = [&](uint32_t jb, uint2 (&k)[kC], uint2 (&v)[kC]) {
        const uint32_t j = min(jb + (lane >> 4), j1 - 1u);
        const bool cached = pk == nullptr || j < p.prefix;
        const size_t row = (static_cast<size_t>(cached ? (p.offset - p.prefix + j) % p.cap : j - p.prefix) * p.KVH + hk) * D;
        load((cached ? ck : pk) + row, k);
        load((cached ? cv : pv) + row, v);
    };
    uint2 q[kC], k[kC], v[kC];
    load(p.q + orow * D, q);
#pragma unroll
    for (uint32_t c = 0; c < kC; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[c][e] = 0.0f;
    if (j0 < j1) load_keys(j0, k, v);
    for (uint32_t jb = j0; jb < j1; jb += 4u) {
        uint2 k_next[kC], v_next[kC];
        load_keys(jb + 4u, k_next, v_next);   // (past the end: the last key again)
        float s = 0.0f;
#pragma unroll
        for (uint32_t c = 0; c < kC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) s = fmaf(value(q[c], e), value(k[c], e), s);
#pragma unroll
        for (int d = 1; d < 16; d *= 2) s += __shfl_xor(s, d);
        if (jb + (lane >> 4) < j1) {
            const float w = s == s ? __builtin_amdgcn_exp2f(fmaf(s, kLog2e, -ref)) : 0.0f;   // (a NaN score weighs 0)
#pragma unroll
            for (uint32_t c = 0; c < kC; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[c][e] = fmaf(w, value(v[c], e), o[c][e]);
        }
#pragma unroll
        for (uint32_t c = 0; c < kC; ++c) {
            k[c] = k_next[c];
            v[c] = v_next[c];
        }
    }
#pragma unroll
    for (uint32_t c = 0; c < kC; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[c][e] += __shfl_xor(o[c][e], 16);
            o[c][e] += __shfl_xor(o[c][e], 32);
        }
}

template <uint32_t D, bool WIDE>
__global__ __launch_bounds__(kThreads, D >= 512u ? 1 : 2) void attn_chunk_kernel(AttnParams p) {
    resolve_position(p);
    using Lds = ChunkLds<D>;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds_mem[];
    const uint32_t lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((HYP_LDS uint8_t*)lds_mem));
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 31u;   // this lane's query row of the wave
    const uint32_t h = lane >> 5;

    // kv head fastest (with 8 of them each XCD works on one head's keys), then the row tiles
    // longest first, then the key splits.
    const uint32_t rows = p.L * p.G;
    const uint32_t tiles = (rows + kChunkRows - 1u) / kChunkRows;
    const uint32_t id = blockIdx.x;
    const uint32_t hk = id % p.KVH;
    const uint32_t rest = id / p.KVH;
    const uint32_t split = rest / tiles;
    const uint32_t tile = tiles - 1u - (rest - split * tiles);
    const uint32_t row0 = tile * kChunkRows;

    // Keys any row of the tile sees, and this split's share of their blocks.
    const uint32_t t_lo = row0 / p.G;
    const uint32_t t_hi = (min(row0 + kChunkRows, rows) - 1u) / p.G;
    uint32_t j_lo = 0u;
    if (p.window != 0u && p.prefix + t_lo + 1u > p.window) j_lo = p.prefix + t_lo + 1u - p.window;
    const uint32_t j_end = p.prefix + t_hi + 1u;
    const uint32_t blocks = (j_end - j_lo + kKeyBlock - 1u) / kKeyBlock;
    const uint32_t b0 = split_first_block(blocks, split, p.splits);
    const uint32_t b1 = split_first_block(blocks, split + 1u, p.splits);

    // This wave's rows: their tokens' range, and this lane's last visible key.
    const uint32_t wrow0 = row0 + wave * kWaveRows;
    const uint32_t w_lo = p.prefix + min(wrow0, rows - 1u) / p.G;                     // last keys of the first
    const uint32_t w_hi = p.prefix + min(wrow0 + kWaveRows - 1u, rows - 1u) / p.G;    // and last row
    const uint32_t qrow = min(wrow0 + n, rows - 1u);   // rows past the end repeat the last (not stored)
    const uint32_t qt = qrow / p.G;
    const uint32_t last_key = p.prefix + qt;
    const uint32_t first_key = p.window != 0u && last_key + 1u > p.window ? last_key + 1u - p.window : 0u;
    const size_t orow = static_cast<size_t>(qt) * p.H + hk * p.G + (qrow - qt * p.G);   // [L][H] row

    constexpr uint32_t kSteps = D / 16u;
    constexpr uint32_t kDTiles = D / 32u;
    bf16x8_t q[kSteps];
    {
        const uint16_t* src = p.q + orow * D + h * 8u;
#pragma unroll
        for (uint32_t st = 0; st < kSteps; ++st) q[st] = *reinterpret_cast<const bf16x8_t*>(src + st * 16u);
    }

    // Block b into stage s: 1 KB units of 512 / D rows, wave w takes units w, w + 4, ... of K
    // and of V; lane l fills physical chunk l % kChunks of row l / kChunks of the unit. Rows
    // past j_end repeat its last row (their scores are masked, no unwritten slot is read).
    constexpr uint32_t kUnitRows = 512u / D;
    constexpr uint32_t kUnits = kKeyBlock / kUnitRows / 4u;   // per wave
    const uint32_t ring_base = p.offset - p.prefix;
    const uint32_t row_stride = p.KVH * D;
    const uint32_t cache_bytes = (p.cap * p.KVH - hk) * D * 2u;   // (narrow: below 2^32)
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.ck + hk * D), static_cast<short>(0), static_cast<int>(cache_bytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.cv + hk * D), static_cast<short>(0), static_cast<int>(cache_bytes), 0x00020000);
    const auto load_unit = [&](uint32_t jb, uint32_t slot0, uint32_t s, uint32_t i) {
        uint32_t ln = lane;
        asm volatile("" : "+v"(ln));   // per-lane addresses formed here, not kept in registers over the walk
        {
            const uint32_t unit = wave + 4u * i;
            const uint32_t r = unit * kUnitRows + ln / Lds::kChunks;
            const uint32_t j = min(jb + r, j_end - 1u);
            const uint32_t phys = ln % Lds::kChunks;
            const bool cached = !WIDE || p.k == nullptr || j < p.prefix;
            uint32_t slot = slot0 + (j - jb);
            slot = slot >= p.cap ? slot - p.cap : slot;
            HYP_LDS void* kd = reinterpret_cast<HYP_LDS void*>(lds + s * Lds::kStage + unit * 1024u);
            HYP_LDS void* vd = reinterpret_cast<HYP_LDS void*>(lds + s * Lds::kStage + Lds::kV + unit * 1024u);
            if constexpr (WIDE) {
                const uint64_t at = static_cast<uint64_t>(cached ? slot : j - p.prefix) * row_stride + hk * D;
                const uint16_t* kp = (cached ? p.ck : p.k) + at + (phys ^ Lds::k_swz(r)) * 8u;
                const uint16_t* vp = (cached ? p.cv : p.v) + at + (phys ^ Lds::v_swz(r)) * 8u;
                __builtin_amdgcn_global_load_lds((const HYP_GLOBAL void*)kp, kd, 16, 0, 0);
                __builtin_amdgcn_global_load_lds((const HYP_GLOBAL void*)vp, vd, 16, 0, 0);
            } else {
                const uint32_t at = slot * row_stride * 2u;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(kr, kd, 16, static_cast<int>(at + (phys ^ Lds::k_swz(r)) * 16u), 0, 0, 0);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(vr, vd, 16, static_cast<int>(at + (phys ^ Lds::v_swz(r)) * 16u), 0, 0, 0);
            }
        }
    };

    f32x16_t o[kDTiles];
#pragma unroll
    for (uint32_t t = 0; t < kDTiles; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] = 0.0f;
    float m = -__builtin_huge_valf();   // the softmax reference (log2 domain) of row n
    float l = 0.0f;                     // the sum over this lane's keys

    // K operand: row n, logical chunk 2 st + h at physical chunk (2 st + h) ^ k_swz(n).
    const uint32_t k_at = lds + n * Lds::kRow + ((h ^ Lds::k_swz(n)) << 4);
    constexpr uint32_t kSpan = Lds::kChunks < 16u ? Lds::kChunks : 16u;   // chunks a swizzle permutes
    constexpr uint32_t kAhead = 4u;
    // V operand of dim tile dt, step t: 16-lane group g reads key rows 16 t + 4 h + 0..3 (then
    // + 8) at dims 32 dt + 16 (g % 2) + 0..15.
    const uint32_t j16 = lane & 15u;
    const uint32_t vrow = 4u * h + (j16 >> 2);
    const uint32_t vchunk = 2u * ((lane >> 4) & 1u) + ((j16 >> 1) & 1u);
    const uint32_t v_at = lds + Lds::kV + vrow * Lds::kRow + ((vchunk ^ Lds::v_swz(vrow)) << 4) + (j16 & 1u) * 8u;

    if (b0 < b1) {
        const uint32_t jb = j_lo + b0 * kKeyBlock;
        const uint32_t slot0 = (ring_base + jb) % p.cap;
#pragma unroll
        for (uint32_t i = 0; i < kUnits; ++i) load_unit(jb, slot0, 0u, i);
    }
    // Product u of O (dim tile u / 2, step u % 2): its V operand.
    const auto v_read = [&](uint32_t stage, uint32_t u) {
        const uint32_t c = 4u * (u / 2u);
        const uint32_t at = ((v_at + stage) ^ ((c % kSpan) << 4)) + (c / kSpan) * kSpan * 16u;
        return lds_read_tr(at + 16u * (u % 2u) * Lds::kRow, 8u * Lds::kRow);
    };
    constexpr uint32_t kProducts = 2u * kDTiles;
    constexpr bool kLazy = D >= 512u;
    float mx = 0.0f;
    // kLazy: blocks run in the inner loop while no row's maximum has outgrown its reference; one
    // that has ends it before it touches O, the outer loop rescales, and the inner loop takes
    // the same block again. (A branch around the rescaling inside the block loop made the
    // compiler copy all of O on every block.)
    uint32_t b = b0;
    bool again = false;
    do {
    for (; b < b1; ++b) {
        const uint32_t stage = ((b - b0) & 1u) * Lds::kStage;
        if (!again) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();   // block b has landed, and every wave has left the other stage
        }
        again = false;
        // The next block's loads go out between this one's score products (the last block, and
        // one taken again, load what they loaded before once more: the same bytes).
        const uint32_t jn = j_lo + min(b + 1u, b1 - 1u) * kKeyBlock;
        const uint32_t slot_n = (ring_base + jn) % p.cap;
        const uint32_t stage_n = (b + 1u - b0) & 1u;
        const uint32_t jb = j_lo + b * kKeyBlock;
        // Fragments are read kAhead products ahead (the scheduling hints keep that order).
        const auto k_read = [&](uint32_t st) {
            const uint32_t c = 2u * st;
            return lds_read16(((k_at + stage) ^ ((c % kSpan) << 4)) + (c / kSpan) * kSpan * 16u);
        };
        f32x16_t s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
        bf16x8_t kf[kAhead];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t st = 0; st < kAhead; ++st) kf[st] = k_read(st);
#pragma unroll
        for (uint32_t st = 0; st < kSteps; ++st) {
            __builtin_amdgcn_sched_barrier(0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[st % kAhead], q[st], s, 0, 0, 0);
            if (st + kAhead < kSteps) kf[st % kAhead] = k_read(st + kAhead);
            if (st % (kSteps / kUnits) == 0u) load_unit(jn, slot_n, stage_n, st / (kSteps / kUnits));
        }
        __builtin_amdgcn_sched_barrier(0);
        bf16x8_t vf[kAhead];
        if constexpr (D != 256u) {   // (at 256 their registers are short)
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u) vf[u] = v_read(stage, u);
            __builtin_amdgcn_sched_barrier(0);
        }

        // s[i] is key jb + 8 (i / 4) + 4 h + i % 4 of row n.
        if (jb + kKeyBlock - 1u > w_lo || (p.window != 0u && jb + p.window <= w_hi)) {
#pragma unroll
            for (uint32_t i = 0; i < 16u; ++i) {
                const uint32_t j = jb + 8u * (i / 4u) + 4u * h + (i & 3u);
                s[i] = j - first_key <= last_key - first_key ? s[i] : -__builtin_huge_valf();
            }
        }
        mx = -__builtin_huge_valf();   // (an all-NaN block leaves it there)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
        mx = half_max(mx) * kLog2e;
        if constexpr (kLazy) m = m == -__builtin_huge_valf() ? mx : m;   // O is still zero: nothing to rescale
        float alpha = 1.0f;
        if constexpr (kLazy) {
            if (__any(mx > m + kRescaleLog2)) {
                again = true;
                break;
            }
        } else {
            const float m_new = fmaxf(m, mx);
            alpha = m_new > m ? __builtin_amdgcn_exp2f(m - m_new) : 1.0f;
            m = m_new;
            l *= alpha;
        }
        const float ref = m > -__builtin_huge_valf() ? m : 0.0f;
        float pr[16];
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            pr[i] = __builtin_amdgcn_exp2f(fmaf(s[i], kLog2e, -ref));
            sum += pr[i];
        }
        if (__any(sum != sum)) {   // a NaN score is a masked one (and an infinite one keeps its NaN)
            sum = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if (s[i] != s[i]) pr[i] = 0.0f;
                sum += pr[i];
            }
        }
        l += sum;
        bf16x8_t pb[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) pb[t] = round_p(pr + 8 * t);
        bf16x8_t pl[2];
        if constexpr (kLazy) {
#pragma unroll
            for (int i = 0; i < 16; ++i) pr[i] -= bf16_bits_to_f32(__builtin_bit_cast(u16x8_t, pb[i / 8])[i % 8]);
#pragma unroll
            for (int t = 0; t < 2; ++t) pl[t] = round_p(pr + 8 * t);
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) o[0][i] *= alpha;
        }
        if constexpr (D == 256u) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u) vf[u] = v_read(stage, u);
        }
#pragma unroll
        for (uint32_t u = 0; u < kProducts; ++u) {
            __builtin_amdgcn_sched_barrier(0);
            o[u / 2u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[u % kAhead], pb[u % 2u], o[u / 2u], 0, 0, 0);
            if constexpr (kLazy)
                o[u / 2u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[u % kAhead], pl[u % 2u], o[u / 2u], 0, 0, 0);
            if (u + kAhead < kProducts) vf[u % kAhead] = v_read(stage, u + kAhead);
            if (!kLazy && u / 2u + 1u < kDTiles) {   // the next tile, half of it in each product's shadow
#pragma unroll
                for (uint32_t i = 0; i < 8u; ++i) o[u / 2u + 1u][8u * (u % 2u) + i] *= alpha;
            }
        }
    }
    if (again) {
        const float m_new = fmaxf(m, mx);
        const float alpha = m_new > m ? __builtin_amdgcn_exp2f(m - m_new) : 1.0f;
        m = m_new;
        l *= alpha;
#pragma unroll
        for (uint32_t t = 0; t < kDTiles; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[t][i] *= alpha;
    }
    } while (again);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last loads: none writes LDS past here
    l = half_sum(l);

    // Rows with a value that is not finite are formed again, by themselves (row_alone), once they
    // are out.
    float zero = 0.0f;
#pragma unroll
    for (uint32_t dt = 0; dt < kDTiles; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) zero = fmaf(o[dt][i], 0.0f, zero);
    const uint64_t odd_lanes = __ballot(zero != 0.0f && wrow0 + n < rows);
    const uint32_t odd_rows = static_cast<uint32_t>(odd_lanes) | static_cast<uint32_t>(odd_lanes >> 32);
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;

    // o[dt][i] is dim 32 dt + 8 (i / 4) + 4 h + i % 4 of row n.
    if (p.splits > 1u) {
        const size_t prow = static_cast<size_t>(split) * p.L * p.H + orow;
        if (wrow0 + n < rows) {
#pragma unroll
            for (uint32_t dt = 0; dt < kDTiles; ++dt)
#pragma unroll
                for (uint32_t u = 0; u < 4u; ++u)
                    *reinterpret_cast<float4*>(p.part_o + prow * D + 32u * dt + 8u * u + 4u * h) =
                        make_float4(o[dt][4 * u], o[dt][4 * u + 1], o[dt][4 * u + 2], o[dt][4 * u + 3]);
            if (h == 0u) {
                p.part_ml[prow * 2u] = m;
                p.part_ml[prow * 2u + 1u] = l;
            }
        }
    } else {
        // The wave's rows through LDS (its own part of the stages, once every wave has left
        // them), then out as 16-byte pieces of whole rows.
        __syncthreads();
        const uint32_t out_lds = lds + wave * kWaveRows * Lds::kOutRow;
#pragma unroll
        for (uint32_t dt = 0; dt < kDTiles; ++dt)
#pragma unroll
            for (uint32_t u = 0; u < 4u; ++u) {
                u32x2_t w;
                w.x = cvt_pk_bf16(o[dt][4 * u] * inv, o[dt][4 * u + 1] * inv);
                w.y = cvt_pk_bf16(o[dt][4 * u + 2] * inv, o[dt][4 * u + 3] * inv);
                *reinterpret_cast<HYP_LDS u32x2_t*>(out_lds + n * Lds::kOutRow + (32u * dt + 8u * u + 4u * h) * 2u) = w;
            }
        __syncthreads();
        for (uint32_t c = lane; c < kWaveRows * Lds::kChunks; c += 64u) {
            const uint32_t r = c / Lds::kChunks;
            const uint32_t gr = wrow0 + r;
            if (gr >= rows) break;
            const uint32_t t = gr / p.G;
            const size_t dst = (static_cast<size_t>(t) * p.H + hk * p.G + (gr - t * p.G)) * D + (c % Lds::kChunks) * 8u;
            *reinterpret_cast<u32x4_t*>(p.out + dst) =
                *reinterpret_cast<const HYP_LDS u32x4_t*>(out_lds + r * Lds::kOutRow + (c % Lds::kChunks) * 16u);
        }
    }
    if (odd_rows == 0u) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the wave's own stores of these rows are done
    for (uint32_t todo = odd_rows; todo != 0u; todo &= todo - 1u) {
        const int r = __builtin_ctz(todo);
        const uint32_t t = (wrow0 + r) / p.G;
        const size_t row = static_cast<size_t>(t) * p.H + hk * p.G + (wrow0 + r - t * p.G);
        const uint32_t last = p.prefix + t;
        const uint32_t first = p.window != 0u && last + 1u > p.window ? last + 1u - p.window : 0u;
        const float ref = __shfl(m, r);
        const float scale = __shfl(inv, r);
        float a[D / 64u][4];
        row_alone<D>(p, hk, row, max(first, j_lo + b0 * kKeyBlock), min(last + 1u, j_lo + b1 * kKeyBlock),
                     ref > -__builtin_huge_valf() ? ref : 0.0f, lane, a);
        if (lane >= 16u) continue;
#pragma unroll
        for (uint32_t c = 0; c < D / 64u; ++c) {
            const uint32_t dim = 64u * c + 4u * lane;
            if (p.splits > 1u) {
                *reinterpret_cast<float4*>(p.part_o + (static_cast<size_t>(split) * p.L * p.H + row) * D + dim) =
                    make_float4(a[c][0], a[c][1], a[c][2], a[c][3]);
            } else {
                *reinterpret_cast<uint2*>(p.out + row * D + dim) = make_uint2(
                    cvt_pk_bf16(a[c][0] * scale, a[c][1] * scale), cvt_pk_bf16(a[c][2] * scale, a[c][3] * scale));
            }
        }
    }
}

template <uint32_t D>
void launch_chunk_d(AttnParams p, hipStream_t stream) {
    constexpr size_t lds = ChunkLds<D>::kBytes;
    static_assert(lds <= 160u * 1024u, "attention LDS");
    if (lds > 65536u) {
        static thread_local int configured_device = -1;
        int dev = 0;
        HYP_HIP_CHECK(hipGetDevice(&dev));
        if (configured_device != dev) {
            for (const void* f : {reinterpret_cast<const void*>(attn_chunk_kernel<D, false>),
                                  reinterpret_cast<const void*>(attn_chunk_kernel<D, true>)})
                HYP_HIP_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
            configured_device = dev;
        }
    }
    const uint32_t tiles = (p.L * p.G + kChunkRows - 1u) / kChunkRows;
    const uint64_t grid = static_cast<uint64_t>(tiles) * p.KVH * p.splits;
    HYP_REQUIRE(grid <= 0x7fffffffull, HYP_STATUS_INVALID_ARGUMENT, "attention: too many rows");
    // A chunk without a prefix is a cache of its own. Keys in one buffer below 4 GiB (a cache
    // that holds the chunk, or such a chunk) load with 32-bit offsets; a larger cache, or a
    // chunk beside its cached prefix, with a 64-bit address per lane.
    if (p.k != nullptr && p.prefix == 0u) {
        p.ck = p.k;
        p.cv = p.v;
        p.k = p.v = nullptr;
        p.cap = p.L;
        p.offset = 0u;
    }
    const bool wide = p.k != nullptr || static_cast<uint64_t>(p.cap) * p.KVH * D * 2u >= (1ull << 32);
    auto kernel = wide ? attn_chunk_kernel<D, true> : attn_chunk_kernel<D, false>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(grid)), dim3(kThreads), lds, stream, p);
    HYP_HIP_CHECK(hipGetLastError());
}

}  // namespace

void launch_attn_chunk(const AttnParams& p, uint32_t head_dim, hipStream_t stream) {
    switch (head_dim) {
        case 64: launch_chunk_d<64>(p, stream); break;
        case 128: launch_chunk_d<128>(p, stream); break;
        case 256: launch_chunk_d<256>(p, stream); break;
        case 512: launch_chunk_d<512>(p, stream); break;
        default: throw NativeError(HYP_STATUS_UNSUPPORTED, "attention: head_dim must be 64, 128, 256 or 512");
    }
}

}  // namespace hyperion::hip
