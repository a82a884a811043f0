// gqa_prefill_rows.hip -- causal GQA prefill over flattened (token, head) rows.
//
// Semantics: as gqa_prefill.hip (flash_prefill_attention,
// src/metal/kernel_sources.h:2769-2896).
//
// The query heads of one kv head read the same keys, so the (token, head)
// pairs of a group are stacked into one list of rows, row r = head r % G of
// token r / G, and cut into blocks of 128 rows whatever G is: no head slot
// stays empty (the blocks of 16 tokens x 4 or 8 heads leave 1 of 8 empty at
// 7 heads per kv head, 2 of 4 at 2).
//  * workgroup = (128-row block, kv head[, key range]), 4 waves of 32 rows.
//    A wave does its rows' whole attention: S^T = K . Q^T on
//    v_mfma_f32_32x32x16, the softmax, O^T += V^T . P^T.  In the 32x32 layout
//    a lane holds one row (its column) of S^T and of O^T, so the row max, sum
//    and re-base factor never cross lanes except for one swap of the wave's
//    halves, and S^T's registers are the PV product's B operand as they
//    stand (the PV key order is S^T's register order; the V^T reads follow
//    it): P never goes through LDS;
//  * 32-key tiles of K and V reach LDS by DMA into a 5-slot ring, up to four
//    tiles ahead, one barrier per tile.  Two workgroups share a CU up to
//    head_dim 128 (80 KiB of LDS and half the registers each): the waves of a
//    SIMD belong to different workgroups, so one's softmax runs beside the
//    other's MFMAs without any ordering between them;
//  * K rows and V rows are XOR-swizzled separately (16-byte chunks): the K
//    operand reads (ds_read_b128, rows = lanes) and the V^T transpose reads
//    (4 rows x 64 bytes per half wave) are both free of bank conflicts, and
//    the V^T swizzle depends on row bits 0-1 only, so one address register per
//    32 output columns serves the whole tile;
//  * S runs one tile ahead: an interval reads K(j + 1) beside the PV product
//    of tile j - 1 and computes S(j + 1) beside the softmax of tile j, so a
//    wave's MFMAs, LDS reads and VALU work overlap inside the wave.
//
// Bound up to head_dim 128 (two waves per SIMD): the SIMDs' issue slots -- per
// 32-key tile and 32 rows 16 MFMAs of 32 cycles and ~80 VALU instructions at
// head_dim 128, ~0.51 us per tile and wave against 0.26 of MFMAs; leaving out
// the DMA, the LDS reads or the softmax takes 14 / 10 / 9% off (timing builds).
// Against the warp-specialised kernel (gqa_prefill.hip), f16, us: 28 / 4 heads
// at head_dim 128 N = 3072 / 4096 / 8192 90 / 148 / 557 -> 82 / 132 / 490, 8 / 8
// heads N = 4096 129 -> 83, 32 / 8 heads at head_dim 64 (bf16) N = 4096 / 8192
// 107 / 391 -> 84 / 300.
// Blocks of 256 rows (8 waves, a 10-slot ring) measured the same, and constant
// ring slots (the loop unrolled over the ring) 1% faster at N = 8192 for four
// times the code.
//
// Bound at head_dim 256: the chain of one wave per SIMD, on half of them (16 / 8
// heads N = 1021: 128 workgroups, the longest 32 tiles at ~1.1 us, of which the
// matrix pipes take 0.45 (32 MFMAs of 32 cycles); a wave issues in half of its
// cycles, waits on memory or LDS for 28% and for its turn for 23%).  16 / 8 heads,
// f16, one prompt: N = 1021 523 -> 38 us (16 -> 226 TFLOP/s), N = 2048 1890 -> 70 us,
// 100 tokens after 1500 172 -> 26 us; before, every (token, kv head) pair walked its
// keys in its own workgroup.
#include "common.h"
#include "kernels.h"

namespace mugen_attn {

namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// A: lane l holds A[l % 32][8(l / 32) .. +8]; B alike (column l % 32); D:
// lane l holds D[8(i / 4) + 4(l / 32) + i % 4][l % 32], i = 0..15
template <int DT>
__device__ __forceinline__ f32x16_t mfma32x32x16(u32x4_t a, u32x4_t b, f32x16_t c) {
    if constexpr (DT == DT_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b),
                                                      c, 0, 0, 0);
}

// One row without matrix products, over keys [k, end): a lane's dot product per
// key, the weights handed round, each lane its output columns.  Nothing of a key
// past `end` is read.  (m, l) as the rows of the main loop
template <int D, int DT>
__device__ __forceinline__ void row_by_hand(const GqaPrefillParams& p, const uint16_t* q, const uint16_t* kb,
                                            const uint16_t* vb, int hd, int k, int end, float (&o)[D / 64], float& m,
                                            float& l) {
    const int lane = threadIdx.x & 63;
    m = kNegInf;
    l = 0.f;
#pragma unroll
    for (int c = 0; c < D / 64; c++) o[c] = 0.f;
#pragma unroll 1
    for (; k < end; k += 64) {
        float s = kNegInf;
        if (k + lane < end) {
            const uint16_t* kr = kb + (int64_t)(k + lane) * p.row_stride;
            s = 0.f;
#pragma unroll 1
            for (int c = 0; c < hd; c += 8) {
                const u32x4_t x = load16(q + c), y = load16(kr + c);
#pragma unroll
                for (int e = 0; e < 4; e++)
                    s += lo_f32<DT>(x[e]) * lo_f32<DT>(y[e]) + hi_f32<DT>(x[e]) * hi_f32<DT>(y[e]);
            }
            s *= p.scale_log2;
        }
        const float mn = fmaxf(m, wave_max(s)), ref = mn == kNegInf ? 0.f : mn;
        const float alpha = m == kNegInf ? 0.f : fast_exp2(m - ref);
        const float w = fast_exp2(s - ref);
        m = mn;
        l = l * alpha + w;
#pragma unroll
        for (int c = 0; c < D / 64; c++) o[c] *= alpha;
        const int n = min(64, end - k);
#pragma unroll 1
        for (int i = 0; i < n; i++) {
            const float wi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), i));
            const uint16_t* vr = vb + (int64_t)(k + i) * p.row_stride;
#pragma unroll
            for (int c = 0; c < D / 64; c++)
                if (lane + 64 * c < hd) o[c] += wi * to_f32<DT>(vr[lane + 64 * c]);
        }
    }
    l = wave_sum(l);
}

// 16-byte chunk c of K (and q) tile row r is stored at chunk c ^ rk_swz(r).
// LDS has 64 banks x 4 B: a phase of a ds_read_b128 covers 16 lanes whose
// rows differ in bits 0, 1, 3, 4 (lane quads of equal parity), and a row is
// half the banks (D = 64) or all of them.
template <int D>
__device__ constexpr int rk_swz(int r) {
    if constexpr (D == 64) return (((r >> 1) & 1) << 2) | ((r >> 3) & 3);
    else return ((r & 3) << 2) | ((r >> 3) & 3);
}
// V rows: a transpose read's phase covers 4 consecutive rows x 4 chunks
template <int D>
__device__ constexpr int rv_swz(int r) {
    if constexpr (D == 64) return ((r >> 1) & 1) << 2;
    else return (r & 3) << 2;
}

// wait until at most `left` DMA groups of OPK operations are in flight (left
// <= MAX; MAX, the steady state, is tested first)
template <int OPK, int MAX>
__device__ __forceinline__ void wait_ops(int left) {
    if (left >= MAX) {
        vm_wait<MAX * OPK>();
        return;
    }
    switch (left) {
#define ROWS_WAIT(n) case n: vm_wait<(n < MAX ? n : 0) * OPK>(); break;
        ROWS_WAIT(1) ROWS_WAIT(2) ROWS_WAIT(3) ROWS_WAIT(4) ROWS_WAIT(5) ROWS_WAIT(6) ROWS_WAIT(7) ROWS_WAIT(8)
        ROWS_WAIT(9) ROWS_WAIT(10) ROWS_WAIT(11) ROWS_WAIT(12) ROWS_WAIT(13) ROWS_WAIT(14) ROWS_WAIT(15)
#undef ROWS_WAIT
        default: vm_wait<0>(); break;
    }
    static_assert(MAX <= 16, "wait cases");
}

// chunk c of a head narrower than D: the chunks past hd re-read chunk
// c mod (hd / 8) (in bounds; q is zero there and O's columns are not stored)
__device__ __forceinline__ int alias_chunk(int c, int hd) {
    const int ch = hd >> 3;
    return c < ch ? c : c % ch;
}

}  // namespace

// PAD: head_dim hd < D.  SPLIT: the workgroup takes keys [s kchunk, (s+1)
// kchunk) of its block and stores partials (see GqaPrefillParams).
template <int D, int DTI, int OUT_DT, bool PAD, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D > 128 ? 1 : 2))) void gqa_prefill_rows_kernel(
    GqaPrefillParams p, int nblk, int Hk) {
    constexpr int DT = DTI == kDtBf16V16 ? DT_BF16 : DTI;  // q and K
    // bf16 inputs: P.V in fp16 with V converted (by this kernel, in LDS, or
    // by the caller's pre-pass); above head_dim 128 P as bf16 hi + lo
    constexpr bool VCVT = DTI == DT_BF16 && D <= 128;
    constexpr int PDT = (VCVT || DTI == kDtBf16V16) ? DT_F16 : DT;
    constexpr int NP = p_terms<PDT>();
    constexpr int NW = 4, BR = 32 * NW;      // waves, rows per block
    constexpr int TK = 32;                   // keys per tile
    constexpr int KK = D / 16;               // k-steps of S over head_dim
    constexpr int DB = D / 32;               // 32-column blocks of O
    constexpr int NT = DB < 4 ? DB : 4;      // V^T address registers
    constexpr int RB = 2 * D, CR = D / 8;    // bytes and 16-byte chunks per tile row
    constexpr int MAT = TK * RB;             // bytes of one K or V tile
    constexpr int NSLOT = 5;                 // tiles per ring
    constexpr int QS = NW / 2;               // slots of each ring that first hold q
    constexpr int VRING = NSLOT * MAT;       // the V ring follows the K ring
    constexpr int OPK = MAT / 1024 / NW;     // 1-KiB DMA ops per wave per tile of one matrix
    constexpr float kClampW = 32768.f;       // re-base when a lane's weights of one tile sum past 2^15
    __shared__ __attribute__((aligned(1024))) char ring[2 * VRING];

    const int hd = PAD ? p.hd : D;
    const int G = p.G;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c32 = lane & 31, h = lane >> 5;

    // (block, kv head, key range) of this workgroup.  Workgroups are dealt to
    // the 8 XCDs round-robin: a group -- one kv head's (range of) keys -- stays
    // on as few XCDs as the group count allows, so that their L2s hold its K
    // and V rows; inside that, the longest blocks first
    const int groups = SPLIT ? Hk * p.ksplit : Hk;
    int grp, bi;
    if (groups < 8 && 8 % groups == 0) {
        const int x = blockIdx.x & 7, r = 8 / groups;
        grp = x % groups;
        bi = (int)(blockIdx.x >> 3) * r + x / groups;
    } else if (groups % 8 == 0) {
        const int x = blockIdx.x & 7, i = blockIdx.x >> 3, gpx = groups >> 3;
        if (SPLIT) {  // blocks of equal length: one group after the other
            grp = x + 8 * (i / nblk);
            bi = i % nblk;
        } else {
            grp = x * gpx + i % gpx;
            bi = i / gpx;
        }
    } else {
        grp = blockIdx.x % groups;
        bi = blockIdx.x / groups;
    }
    if (bi >= nblk) return;
    const int blk = nblk - 1 - bi;
    const int ks_id = SPLIT ? grp / Hk : 0;
    const int kvh = SPLIT ? grp - ks_id * Hk : grp;

    const int R = p.N * G;                    // rows of the group
    const int r0 = blk * BR + 32 * w;         // this wave's first row
    auto lim = [&](int tok) { return p.causal ? min(p.start_pos + tok + 1, p.kv_len) : p.kv_len; };
    int kend = lim((min(blk * BR + BR, R) - 1) / G);
    const int k_beg = SPLIT ? ks_id * p.kchunk : 0;
    if (SPLIT) kend = min(kend, k_beg + p.kchunk);
    const int nt = kend > k_beg ? (kend - k_beg + TK - 1) / TK : 0;  // tiles
    const int row = min(r0 + c32, R - 1);     // (rows past the last: clamped, never stored)
    const int tok = row / G, hi = row - tok * G;
    const int row_lim = lim(tok);
    // the wave's keys: none visible from w_end on, all visible below mask_from
    const int w_end = r0 < R ? min(kend, lim((min(r0 + 32, R) - 1) / G)) : 0;
    const int mask_from = min(lim(min(r0, R - 1) / G), kend);

    const uint32_t ring_base = lds_addr(&ring[0]);
    const int rs_bytes = p.row_stride * 2;
    const uint16_t* kb = p.k + (int64_t)kvh * hd;
    const uint16_t* vb = p.v + (int64_t)kvh * hd;

    // tile DMA: op o = w + NW k moves tile rows (64 o + lane) / CR
    int t_row[OPK];
    uint32_t k_off[OPK], v_off[OPK];
#pragma unroll
    for (int k = 0; k < OPK; k++) {
        t_row[k] = (64 * (w + NW * k) + lane) / CR;
        const int ck = (lane % CR) ^ rk_swz<D>(t_row[k]), cv = (lane % CR) ^ rv_swz<D>(t_row[k]);
        k_off[k] = (uint32_t)t_row[k] * rs_bytes + (uint32_t)(PAD ? alias_chunk(ck, hd) : ck) * 16;
        v_off[k] = (uint32_t)t_row[k] * rs_bytes + (uint32_t)(PAD ? alias_chunk(cv, hd) : cv) * 16;
    }
    // one tile of one matrix into its slot; rows past the block's last key
    // re-read it (masked)
    const uint32_t ring_w = ring_base + w * 1024;
    auto issue = [&](const uint16_t* src, const uint32_t* col, int dst, int it) {
        const int kt = k_beg + it * TK;
        const char* sp = reinterpret_cast<const char*>(src) + (int64_t)kt * rs_bytes;
        const int last = kend - 1 - kt;
        if (last >= TK - 1) {
#pragma unroll
            for (int k = 0; k < OPK; k++) dma16s(ring_w + dst + k * NW * 1024, sp, col[k]);
        } else {
#pragma unroll
            for (int k = 0; k < OPK; k++)
                dma16s(ring_w + dst + k * NW * 1024, sp, col[k] - (uint32_t)max(t_row[k] - last, 0) * rs_bytes);
        }
    };
    auto issue_k = [&](int it, int slot) {
        if (it < nt) issue(kb, k_off, slot * MAT, it);
    };
    auto issue_v = [&](int it, int slot) {
        if (it < nt) issue(vb, v_off, VRING + slot * MAT, it);
    };

    // q rows of this wave by DMA too (a compiler-tracked load would be waited
    // for behind the tiles): one slot's worth, into a slot whose first tile
    // comes after barrier P
    char* qst = &ring[(w / QS) * VRING + (NSLOT - QS + w % QS) * MAT];
    if (nt > 0) {
        const int tok0 = min(r0, R - 1) / G;
        const uint16_t* qb = p.q + ((int64_t)tok0 * p.H + kvh * G) * hd;
#pragma unroll
        for (int k = 0; k < MAT / 1024; k++) {
            const int qr = (64 * k + lane) / CR;
            const int rr = min(r0 + qr, R - 1);
            const int tk = rr / G;
            const int cq = (lane % CR) ^ rk_swz<D>(qr);
            const uint32_t off = (uint32_t)(((tk - tok0) * p.H + (rr - tk * G)) * hd) * 2 +
                                 (uint32_t)(PAD ? alias_chunk(cq, hd) : cq) * 16;
            dma16s(lds_addr(qst) + k * 1024, qb, off);
        }
    }
    // tile order: K(0), then V(i), K(i + 1)
    constexpr int PRE = NSLOT - QS;  // tiles of each matrix requested before barrier P
    issue_k(0, 0);
#pragma unroll
    for (int i = 0; i < PRE - 1; i++) {
        issue_v(i, i);
        issue_k(i + 1, i + 1);
    }
    issue_v(PRE - 1, PRE - 1);
    // operand addresses inside a slot: K row c32, chunk 2kk + h; V^T column
    // block t, rows 4h + (c32 % 16) / 4 (+ 16m + 8x as constant offsets)
    uint32_t a_off[KK], t_off[NT];
#pragma unroll
    for (int kk = 0; kk < KK; kk++) a_off[kk] = c32 * RB + ((2 * kk + h) ^ rk_swz<D>(c32)) * 16;
    {
        const int i = lane & 15, vr = 4 * h + (i >> 2);
#pragma unroll
        for (int t = 0; t < NT; t++)
            t_off[t] = vr * RB + ((4 * t + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1)) ^ rv_swz<D>(vr)) * 16 + 8 * (i & 1);
    }
    // ops of the tiles issued behind K(0) (before barrier P) and behind the
    // pair (V(j), K(j + 1)) (before barrier j) that may stay in flight
    u32x4_t qf[KK];
    if (nt > 0) {
        // the q rows and K(0), first in the queue (VCVT: and V(0))
        wait_ops<OPK, 2 * PRE - 1 - VCVT>(2 * min(nt, PRE) - 1 - VCVT);
#pragma unroll
        for (int kk = 0; kk < KK; kk++) {
            qf[kk] = *reinterpret_cast<const u32x4_t*>(qst + a_off[kk]);
            if (PAD && 16 * kk + 8 * h >= hd) qf[kk] = u32x4_t{0, 0, 0, 0};
        }
    }

    // V conversion (VCVT): a wave converts the V chunks its own DMA moved, in
    // the interval before the tile is read
    auto cv_addr = [&](int slot, int k) {
        return reinterpret_cast<u32x4_t*>(&ring[VRING + slot * MAT + (w + NW * k) * 1024 + lane * 16]);
    };
    u32x4_t cv[OPK];
    auto cv_read = [&](int slot) {
#pragma unroll
        for (int k = 0; k < OPK; k++) cv[k] = *cv_addr(slot, k);
    };
    auto cv_write = [&](int slot) {
#pragma unroll
        for (int k = 0; k < OPK; k++) {
            u32x4_t y;
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = pack2<DT_F16>(lo_f32<DT_BF16>(cv[k][e]), hi_f32<DT_BF16>(cv[k][e]));
            *cv_addr(slot, k) = y;
        }
    };

    f32x16_t o[DB];
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[d][i] = 0.f;
    float m_run = kNegInf, l_part = 0.f;
    u32x4_t kf[KK], vf[2][DB], pf[2][NP];
#pragma unroll
    for (int m = 0; m < 2; m++) {
#pragma unroll
        for (int d = 0; d < DB; d++) vf[m][d] = u32x4_t{0, 0, 0, 0};
#pragma unroll
        for (int pp = 0; pp < NP; pp++) pf[m][pp] = u32x4_t{0, 0, 0, 0};
    }
    const lds_char_t* ka[KK];
    const lds_char_t* va[NT];
    auto addr_k = [&](int slot) {
#pragma unroll
        for (int kk = 0; kk < KK; kk++) ka[kk] = lds_ptr(ring_base + slot * MAT + a_off[kk]);
    };
    auto addr_v = [&](int slot) {
#pragma unroll
        for (int t = 0; t < NT; t++) va[t] = lds_ptr(ring_base + VRING + slot * MAT + t_off[t]);
    };
    auto read_k = [&]() {
#pragma unroll
        for (int kk = 0; kk < KK; kk++) kf[kk] = lds_read_b128(ka[kk]);
    };
    auto read_v = [&]() {
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int d = 0; d < DB; d++) {
                const int off = (d / NT) * 256 + 16 * m * RB;
                const u32x2_t lo = lds_read_tr16(va[d % NT] + off);
                const u32x2_t up = lds_read_tr16(va[d % NT] + off + 8 * RB);
                vf[m][d] = u32x4_t{lo[0], lo[1], up[0], up[1]};
            }
    };
    auto pv = [&]() {
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int pp = 0; pp < NP; pp++)
#pragma unroll
                for (int d = 0; d < DB; d++) o[d] = mfma32x32x16<PDT>(vf[m][d], pf[m][pp], o[d]);
    };
    auto scores = [&](f32x16_t& r) {
#pragma unroll
        for (int i = 0; i < 16; i++) r[i] = 0.f;
#pragma unroll
        for (int kk = 0; kk < KK; kk++) r = mfma32x32x16<DT>(kf[kk], qf[kk], r);
    };
    // lane: row c32, keys kt + 8(i / 4) + 4h + i % 4
    auto mask = [&](f32x16_t& r, int kt) {
        const int lim0 = row_lim - kt - 4 * h;
#pragma unroll
        for (int i = 0; i < 16; i++)
            if (8 * (i >> 2) + (i & 3) >= lim0) r[i] = kNegInf;
    };
    const int nw = w_end > k_beg ? (w_end - k_beg + TK - 1) / TK : 0;  // the wave's own tiles (a prefix)
    const int jmask = max(mask_from - k_beg, 0) / TK;                  // the first of them that needs the mask
    f32x16_t s0, s1;  // scores of two tiles in turn
    int slot = 0;     // of tile j
    if (nt > 0) {
        if constexpr (VCVT) {
            cv_read(0);
            cv_write(0);
        }
        lds_barrier();  // P: K(0) from every wave; every q row is in registers
#pragma unroll
        for (int i = PRE; i < NSLOT; i++) {
            issue_k(i, i);
            if (i < NSLOT - 1) issue_v(i, i);
        }
        if (nw > 0) {
            addr_k(0);
            read_k();
            scores(s0);
            if (jmask == 0) mask(s0, k_beg);
            // the first tile sets the row's reference max
            float mx = s0[0];
#pragma unroll
            for (int i = 1; i < 16; i++) mx = fmaxf(mx, s0[i]);
            m_run = max_x32(mx) * p.scale_log2;
        }
    }
    // tile j of slot u: S(j + 1) runs ahead into sn while the softmax of s
    // and the PV product of tile j - 1 are under way
    auto step = [&](int j, f32x16_t& s, f32x16_t& sn, bool first) {
        const int u = slot, un = u == NSLOT - 1 ? 0 : u + 1, up = u == 0 ? NSLOT - 1 : u - 1;
        slot = un;
        // V(j) and K(j + 1) landed (VCVT: and V(j + 1), whose conversion is due
        // now); what was issued after them stays in flight
        const int left = nt - 1 - j;
        constexpr int NP1 = NSLOT - 2;
        // behind (V(j), K(j + 1)): V(j + 1 .. j + NP1), K(j + 2 .. j + 1 + NP1);
        // behind V(j + 1): one of each pair less, K(j + 2) first
        if (VCVT) wait_ops<OPK, 2 * NP1 - 1>(left > NP1 ? 2 * NP1 - 1 : max(2 * left - 2, 0));
        else wait_ops<OPK, 2 * NP1>(left > NP1 ? 2 * NP1 : max(2 * left - 1, 0));
        lds_barrier();  // j
        issue_v(j + NSLOT - 1, up);
        issue_k(j + NSLOT, u);
        if (VCVT && left > 0) cv_read(un);
        if (j >= nw) {  // wave-uniform: no row of the wave sees tile j
            if (VCVT && left > 0) cv_write(un);
            return;
        }
        if (!first && __builtin_expect(j >= jmask, 0)) mask(s, k_beg + j * TK);
        float nm = m_run == kNegInf ? 0.f : -m_run;
        addr_k(un);
        addr_v(u);
        // head_dim 256 (one wave per SIMD): the MFMAs spread over the softmax and
        // the LDS reads by hand; left to itself the scheduler spills (16 / 8
        // heads, N = 1021: 42.7 -> 38.3 us, N = 2048 96 -> 71).  At 128 the
        // second wave fills the gaps and the hints change nothing
        if constexpr (D > 128) __builtin_amdgcn_sched_barrier(0);
        read_k();  // (past the wave's last tile the scores are never used)
        pv();
        read_v();
        float x[16], ps = 0.f;
        scores(sn);
#pragma unroll
        for (int i = 0; i < 16; i++) x[i] = fast_exp2(fmaf(s[i], p.scale_log2, nm));
        {
            float a[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = (x[i] + x[4 + i]) + (x[8 + i] + x[12 + i]);
            ps = (a[0] + a[1]) + (a[2] + a[3]);
        }
        if constexpr (D > 128) {
            constexpr int kMfma = 0x8, kValu = 0x402, kLdsRead = 0x100;
#pragma unroll
            for (int i = 0; i < 4; i++) {  // PV beside K's reads
                __builtin_amdgcn_sched_group_barrier(kLdsRead, KK / 4, 0);
                __builtin_amdgcn_sched_group_barrier(kMfma, 2 * DB * NP / 4, 0);
                __builtin_amdgcn_sched_group_barrier(kValu, 6, 0);
            }
#pragma unroll
            for (int i = 0; i < KK; i++) {  // S beside V's reads and the softmax
                __builtin_amdgcn_sched_group_barrier(kLdsRead, 4 * DB / KK, 0);
                __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                __builtin_amdgcn_sched_group_barrier(kValu, 40 / KK, 0);
            }
        }
        // re-base only when a lane's weights sum past kClampW (every weight
        // >= 0, so any weight past it shows).  A row without a visible key
        // in the first tile sees no later key
        if (!first && __builtin_expect(__any(!(ps <= kClampW)), 0)) {
            float mt = kNegInf;
#pragma unroll
            for (int i = 0; i < 16; i++) mt = fmaxf(mt, fmaf(s[i], p.scale_log2, nm));
            mt = max_x32(mt);
            const float shift = fmaxf(mt, 0.f);  // rows under their reference keep it
            const float alpha = fast_exp2(-shift);
            l_part *= alpha;
#pragma unroll
            for (int d = 0; d < DB; d++) o[d] *= alpha;
            m_run = (m_run == kNegInf ? 0.f : m_run) + shift;
            nm -= shift;
            ps = 0.f;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                x[i] = fast_exp2(fmaf(s[i], p.scale_log2, nm));
                ps += x[i];
            }
        }
        l_part += ps;
#pragma unroll
        for (int m = 0; m < 2; m++) split_p<PDT, NP>(x + 8 * m, pf[m]);
        // the first tile: what rounding took off its weights, through the same
        // V^T.  Rows of few keys have the largest outputs, and most of their keys
        // here; the per-pair kernel's four reference weights of exactly 1 a row
        // (here one) had a smaller error without it.  Against 64 bits, f16, 16 / 8
        // heads d256, per pair / without / with: N = 150 2.34 / 2.43 / 2.16e-4, 1021
        // 2.50 / 2.60 / 2.43e-4, 700 after 1500 2.907 / 2.910 / 2.891e-4; 28 / 4 heads
        // d128 N = 3072, warp-specialised / without / with 2.63 / 2.65 / 2.51e-4
        if (NP == 1 && first) {
#pragma unroll
            for (int m = 0; m < 2; m++) {
                u32x4_t hl[2];
                split_p<PDT, 2>(x + 8 * m, hl);
#pragma unroll
                for (int d = 0; d < DB; d++) o[d] = mfma32x32x16<PDT>(vf[m][d], hl[1], o[d]);
            }
        }
        if (VCVT && left > 0) cv_write(un);
    };
    // the first tile on its own: no mask or re-base to test for, and the loop
    // without its extra product (in the loop: 472 -> 475 us at 28 / 4 heads d128 N =
    // 8192).  Padded heads above 128 keep it in the loop, whose schedule suffers from
    // the copy (16 / 8 heads d192 N = 2048 78 against 84 us)
    if constexpr (PAD && D > 128) {
        for (int j = 0; j < nt; j += 2) {
            step(j, s0, s1, j == 0);
            if (j + 1 < nt) step(j + 1, s1, s0, false);
        }
    } else {
        if (nt > 0) step(0, s0, s1, true);
        for (int j = 1; j < nt; j += 2) {
            step(j, s1, s0, false);
            if (j + 1 < nt) step(j + 1, s0, s1, false);
        }
    }
    if (nw > 0) pv();

    // partials: fp16 up to head_dim 128 (a convex combination of V rows, inside
    // V's +-65504), fp32 above
    constexpr int SDT = SPLIT ? (D > 128 ? DT_F32 : DT_F16) : OUT_DT;
    // A key that a row does not see has weight 0 in the wave's tiles from mask_from
    // on, and 0 x an infinity or a NaN of its V is a NaN.  A wave with such a V row
    // works its rows again, each over its own keys; looked for only where the output
    // is not finite (a NaN from a visible key costs the look, not the rows).  Above
    // head_dim 128 only, where the per-pair kernel never read such a key: it is
    // free there (16 / 8 heads d256 N = 1021 39.5 us either way), at 128 it takes 0.7%
    // of 472 us, and the kernels beside it do as this one
    if constexpr (D > 128) {
        float z4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < DB; d++)
#pragma unroll
            for (int i = 0; i < 16; i++) z4[i & 3] = fmaf(0.f, o[d][i], z4[i & 3]);
        float z = (z4[0] + z4[1]) + (z4[2] + z4[3]);
        bool hidden = false;
        if (__builtin_expect(__any(z != 0.f), 0)) {
            z = 0.f;
#pragma unroll 1
            for (int t = max(mask_from, k_beg), t_end = min(k_beg + nw * TK, kend); t < t_end; t++)
#pragma unroll 1
                for (int c = lane; c < hd; c += 64) z = fmaf(0.f, to_f32<DT>(vb[(int64_t)t * p.row_stride + c]), z);
            hidden = __any(z != 0.f);
        }
        if (__builtin_expect(hidden, 0)) {
#pragma unroll 1
            for (int r = r0; r < min(r0 + 32, R); r++) {
                const int t = r / G;
                const int64_t at = (int64_t)t * p.H + kvh * G + (r - t * G);
                float oc[D / 64], m, l;
                row_by_hand<D, DT>(p, p.q + at * hd, kb, vb, hd, k_beg, min(lim(t), kend), oc, m, l);
                const float inv = l > 0.f ? 1.f / l : 0.f;
                const int64_t slot_at = SPLIT ? at * p.ksplit + ks_id : at;
                if (SPLIT && lane == 0) *reinterpret_cast<f32x2v_t*>(p.ws_ml + slot_at * 2) = f32x2v_t{m, l};
                void* base = SPLIT ? static_cast<void*>(p.ws_o) : p.out;
#pragma unroll
                for (int c = 0; c < D / 64; c++)
                    if (lane + 64 * c < hd) store_out<SDT>(base, slot_at * hd + lane + 64 * c, oc[c] * inv);
            }
            return;
        }
    }

    // ---- store.  Lane: row c32, columns 32d + 8a + 4h + i in o[d][4a + i]
    if (r0 + c32 >= R) return;
    const float l = sum_x32(l_part);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const int64_t orow = (int64_t)tok * p.H + kvh * G + hi;
    if (SPLIT && h == 0)
        *reinterpret_cast<f32x2v_t*>(p.ws_ml + (orow * p.ksplit + ks_id) * 2) = f32x2v_t{m_run, l};
    char* dst = SPLIT ? reinterpret_cast<char*>(p.ws_o) + (orow * p.ksplit + ks_id) * hd * (SDT == DT_F32 ? 4 : 2)
                      : static_cast<char*>(p.out) + orow * hd * (SDT == DT_F32 ? 4 : 2);
#pragma unroll
    for (int d = 0; d < DB; d++) {
        o[d] *= inv;
        if constexpr (SDT == DT_F32) {
#pragma unroll
            for (int a = 0; a < 4; a++) {
                const int c = 32 * d + 8 * a + 4 * h;
                if (!PAD || c < hd)
                    *reinterpret_cast<f32x4_t*>(dst + 4 * c) =
                        f32x4_t{o[d][4 * a], o[d][4 * a + 1], o[d][4 * a + 2], o[d][4 * a + 3]};
            }
        } else {
            // two quads of each half swapped across the halves: 8 consecutive
            // columns per lane, one 16-byte store
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int e = 8 * q;
                const auto x0 = __builtin_amdgcn_permlane32_swap(pack2<SDT>(o[d][e], o[d][e + 1]),
                                                                 pack2<SDT>(o[d][e + 4], o[d][e + 5]), false, false);
                const auto x1 = __builtin_amdgcn_permlane32_swap(pack2<SDT>(o[d][e + 2], o[d][e + 3]),
                                                                 pack2<SDT>(o[d][e + 6], o[d][e + 7]), false, false);
                const int c = 32 * d + 16 * q + 8 * h;
                if (!PAD || c < hd) *reinterpret_cast<u32x4_t*>(dst + 2 * c) = u32x4_t{x0[0], x1[0], x0[1], x1[1]};
            }
        }
    }
}

// ------------------------------------------------------------------ launch

template <int D, int DT, int OUT_DT, bool PAD>
static hipError_t launch_rows_t(const GqaPrefillParams& p, int Hk, hipStream_t st, KernelTimer* t) {
    const int nblk = (int)(((int64_t)p.N * p.G + 127) / 128);
    const int groups = Hk * (p.ksplit > 1 ? p.ksplit : 1);
    // (the kernel's deal of blocks to XCDs)
    const int grid = groups < 8 && 8 % groups == 0 ? 8 * ((nblk * groups + 7) / 8) : nblk * groups;
    if constexpr (D > 128)
        if (p.ksplit > 1)
            return launch_k(t, "gqa_prefill", gqa_prefill_rows_kernel<D, DT, DT_F32, PAD, true>, dim3(grid), dim3(256),
                            st, p, nblk, Hk);
    return launch_k(t, "gqa_prefill", gqa_prefill_rows_kernel<D, DT, OUT_DT, PAD, false>, dim3(grid), dim3(256), st, p,
                    nblk, Hk);
}

template <int D, int DT, bool PAD>
static hipError_t launch_rows_o(const GqaPrefillParams& p, int Hk, int out_dt, hipStream_t st, KernelTimer* t) {
    if (out_dt == DT_F32) return launch_rows_t<D, DT, DT_F32, PAD>(p, Hk, st, t);
    if (out_dt == DT_F16) return launch_rows_t<D, DT, DT_F16, PAD>(p, Hk, st, t);
    return launch_rows_t<D, DT, DT_BF16, PAD>(p, Hk, st, t);
}

template <int D, bool PAD>
static hipError_t launch_rows_d(const GqaPrefillParams& p, int Hk, int dt, int out_dt, hipStream_t st, KernelTimer* t) {
    if (dt == DT_F16) return launch_rows_o<D, DT_F16, PAD>(p, Hk, out_dt, st, t);
    if constexpr (D <= 128)
        if (dt == kDtBf16V16) return launch_rows_o<D, kDtBf16V16, PAD>(p, Hk, out_dt, st, t);
    return launch_rows_o<D, DT_BF16, PAD>(p, Hk, out_dt, st, t);
}

hipError_t launch_gqa_prefill_rows(const GqaPrefillParams& p, int Hk, int dt, int out_dt, hipStream_t st,
                                   KernelTimer* t) {
    if (p.hd > 128)
        return p.hd != 256 ? launch_rows_d<256, true>(p, Hk, dt, out_dt, st, t)
                           : launch_rows_d<256, false>(p, Hk, dt, out_dt, st, t);
    if (p.ksplit > 1) return hipErrorInvalidValue;  // split ranges: the warp-specialised kernel
    if (p.hd > 64)
        return p.hd != 128 ? launch_rows_d<128, true>(p, Hk, dt, out_dt, st, t)
                           : launch_rows_d<128, false>(p, Hk, dt, out_dt, st, t);
    return p.hd != 64 ? launch_rows_d<64, true>(p, Hk, dt, out_dt, st, t)
                      : launch_rows_d<64, false>(p, Hk, dt, out_dt, st, t);
}

}  // namespace mugen_attn
