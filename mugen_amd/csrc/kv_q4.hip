// kv_q4.hip -- append to the 4-bit group KV store (KVCache::append,
// src/core/memory/kv_cache.cpp:163-216).
//
// Layout per sequence: Q4 groups of every quantised token at its absolute
// position ([max_seq_len][vpt/32][20 B]) and an f16 ring of `ring` token
// rows (a power of two) holding the newest ones (token t at slot
// t % ring).  Appending n_new
// tokens to a sequence holding T tokens of which n_q4 are quantised leaves
// the newest fp16_preserve_last in f16 and quantises the ones that age out:
// positions n_q4 .. n_q4 + q - 1 with q = max(0, T - n_q4 + n_new -
// preserve), exactly the tokens the reference's one-token appends quantise.
// With ring >= preserve + n_new, the ring slots read by those quantisations
// and the slots written by the new tokens are distinct, so one launch does
// both.
//
// Grid (2 * n_new, n_seq), two waves per job, one for K and one for V: job j <
// n_new writes new token j to its ring slot (unless it is quantised right
// away), job n_new + j quantises aged token n_q4 + j (from the ring, or from the
// new tokens when preserve < n_new), four lanes per 32-value group, 8 values
// (one 16-byte load, one dword of nibbles) each:
//   quantize_group (kv_cache.cpp:21-56): min / max over the 32 f16 values,
//   scale = f16(range / 15) (0 for a constant group), nibble =
//   min(15, roundf((v - min) / scale)), value 2i in the low nibble of byte i.
// Bound: latency -- the lengths, the row, 8 IEEE divisions per lane.  One lane
// per group did K's and V's 64 divisions one after the other with a quarter of
// the lanes: one token for 16 sequences, 512 values a row, 6.7 us (now 4.0).
#include "common.h"
#include "kernels.h"

namespace mugen_attn {

// values 8 * (lane % 4) .. +7 of a group at src; every lane of the wave calls it
// (store: this lane's group exists)
__device__ __forceinline__ void quantize_group_part(const uint16_t* src, uint8_t* dst, int part, bool store) {
#pragma clang fp contract(off)
    const u32x4_t w = load16(src);
    float x[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        x[2 * i] = lo_f32<DT_F16>(w[i]);
        x[2 * i + 1] = hi_f32<DT_F16>(w[i]);
    }
    // the reference scans the group from its first value with strict compares:
    // the first occurrence of the extremes wins, and a NaN past the first value
    // is passed over.  So part 0 starts from its first value, the others from
    // no value, and a later part wins only by a strict compare
    float lo = part == 0 ? x[0] : -kNegInf, hi = part == 0 ? x[0] : kNegInf;
    uint32_t lo_bits = w[0] & 0xffffu;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if (x[i] < lo) {
            lo = x[i];
            lo_bits = (i & 1) ? (w[i >> 1] >> 16) : (w[i >> 1] & 0xffffu);
        }
        hi = x[i] > hi ? x[i] : hi;
    }
    auto merge = [&](auto m) {  // with the lane xor M: the part with bit M clear comes first
        constexpr int M = decltype(m)::value;
        const float plo = dpp_xor<M>(lo), phi = dpp_xor<M>(hi);
        const uint32_t pb = __float_as_uint(dpp_xor<M>(__uint_as_float(lo_bits)));
        const bool first = (part & M) == 0;
        const float alo = first ? lo : plo, blo = first ? plo : lo;
        const uint32_t ab = first ? lo_bits : pb, bb = first ? pb : lo_bits;
        const float ahi = first ? hi : phi, bhi = first ? phi : hi;
        lo = blo < alo ? blo : alo;
        lo_bits = blo < alo ? bb : ab;
        hi = bhi > ahi ? bhi : ahi;
    };
    merge(std::integral_constant<int, 1>{});
    merge(std::integral_constant<int, 2>{});
    const float range = hi - lo;
    const uint32_t sbits = range == 0.0f ? 0u : uint32_t(from_f32<DT_F16>(range / 15.0f));
    const float sf = to_f32<DT_F16>(uint16_t(sbits)), mf = to_f32<DT_F16>(uint16_t(lo_bits));
    uint32_t packed = 0u;
    if (sf > 0.0f) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float a = fminf(15.0f, roundf((x[2 * i] - mf) / sf));
            const float c = fminf(15.0f, roundf((x[2 * i + 1] - mf) / sf));
            packed |= ((uint32_t(c) << 4) | uint32_t(a)) << (8 * i);
        }
    }
    if (!store) return;
    // 20 bytes at a 4-byte aligned address: scale and min, then a dword a part
    uint32_t* d = reinterpret_cast<uint32_t*>(dst);
    if (part == 0) d[0] = sbits | (lo_bits << 16);
    d[1 + part] = packed;
}

__global__ __launch_bounds__(128) void kv_q4_append_kernel(KvQ4AppendParams p) {
    const int b = blockIdx.y, job = blockIdx.x, lane = threadIdx.x & 63;
    const bool is_v = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) != 0;
    // lengths clamped to the store: a device value past max_seq_len (or
    // negative) never indexes outside it
    const int T = clamp_len(p.seq_lens[b], p.max_seq_len), nq = clamp_len(p.n_q4[b], T);
    const int q = max(0, T - nq + p.n_new - p.preserve);
    const uint16_t* fresh = (is_v ? p.v_new : p.k_new) + (int64_t)b * p.n_new * p.vpt;
    uint16_t* ring = (is_v ? p.ring_v : p.ring_k) + (int64_t)b * p.ring_seq_stride;
    // tokens at positions >= max_seq_len are dropped, so they are not counted
    if (job == 0 && threadIdx.x == 0) p.n_q4_out[b] = min(nq + q, p.max_seq_len);
    if (job < p.n_new) {
        const int t = T + job;
        if (t < nq + q || t >= p.max_seq_len) return;  // quantised right away / past the cache
        uint16_t* dst = ring + (int64_t)(t & (p.ring - 1)) * p.vpt;
        for (int i = 8 * lane; i < p.vpt; i += 8 * 64)
            *reinterpret_cast<u32x4_t*>(dst + i) = load16(fresh + (int64_t)job * p.vpt + i);
        return;
    }
    const int j = job - p.n_new;
    if (j >= q) return;
    const int t = nq + j;
    if (t >= p.max_seq_len) return;
    const uint16_t* src = t < T ? ring + (int64_t)(t & (p.ring - 1)) * p.vpt : fresh + (int64_t)(t - T) * p.vpt;
    const int groups = p.vpt / 32;
    uint8_t* row = (is_v ? p.q4v : p.q4k) + (int64_t)b * p.q4_seq_stride + (int64_t)t * groups * 20;
    for (int g0 = 0; g0 < groups; g0 += 16) {  // every lane in step: the merges read their neighbours
        const int g = g0 + (lane >> 2), gc = min(g, groups - 1);
        quantize_group_part(src + 32 * gc + 8 * (lane & 3), row + 20 * gc, lane & 3, g < groups);
    }
}

hipError_t launch_kv_q4_append(const KvQ4AppendParams& p, int n_seq, hipStream_t st, KernelTimer* t) {
    return launch_k(t, "kv_q4_append", kv_q4_append_kernel, dim3(2 * p.n_new, n_seq), dim3(128), st, p);
}

}  // namespace mugen_attn
