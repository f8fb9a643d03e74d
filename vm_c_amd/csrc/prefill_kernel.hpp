// prefill_kernel.hpp -- causal flash-attention prefill on MFMA, with optional fused
// quantize-on-append of the K/V rows into the paged cache.
//
// Replaces vm_c::flash_attention_prefill_local (include/vm_c/cuda/
// kernels_flash_attn.h:81-93, src/cuda/flash_attn_v2_kernels.cu:262-393: one
// serial thread block per (token, head)).  Semantics: each sequence's tokens
// are contiguous with positions 0..n-1, so token t attends keys
// [t - pos(t), t]; GQA kv head = q head / (Hq / Hkv).
//
// Tiling (gfx950, wave64, v_mfma_f32_32x32x16_{bf16,f16}):
//   workgroup = 8 waves = up to 4 query heads of one KV head x 32-row query
//   blocks, so every K/V tile of 64 keys in LDS serves 256 query rows.  Tiles
//   arrive by load-to-LDS transfers in a 3-slot ring (rows of 256 B, 16-byte
//   chunk ch of row r at position ch ^ swz(r)); before a tile is published
//   each wave transposes the V rows it loaded into an fp16 V^T tile.
//   S^T[64 kv x 32 q] = K . Q^T per wave: 16 MFMAs, Q^T held in registers,
//     the two 32-key chains interleaved with K operand reads two steps
//     ahead.  One query row per lane column: the row max / sum of the online
//     softmax are in-lane plus one cross-half shuffle.
//   O[32 q x 128] += P . V per wave: 16 fp16 MFMAs.  P is fed straight from
//     the S^T registers: the contraction index k of an MFMA may be any
//     permutation of the 16 keys as long as A and B agree, so logical k =
//     8h + e maps to kv 16c + 8(e/4) + 4h + e%4, which is what lane half h
//     already holds; V^T stores each 16-key block in that order, so a B
//     operand is one 16-byte read.
//   Per-row rescale factors reach the O rows through a small LDS scratch.
// bf16 V that fp16 would overflow (|v| >= 65536), or rows of V entirely
// below 2^-8 with values fp16 keeps only on its subnormal grid, are caught
// in the V^T pass; the workgroup then reruns in an exact mode: raw bf16 V
// rows as B operands, P in fp32 split into bf16 hi + lo, two bf16 MFMAs per
// product.
// Fused append: head group 0 of each KV head writes the block's K/V rows into
// the paged cache with the same block encoders as vmc_reshape_and_cache
// (bit-identical pages).
#pragma once

#include "kv_quant.hpp"
#include "prefill_dev.hpp"
#include "tq_lut.hpp"
#include "vmc_tq.hpp"

namespace vmc {

constexpr int kD = 128;
constexpr int NW = 8;      // waves per workgroup (32 query rows each)
constexpr int BN = 64;     // kv rows per tile
constexpr int NSLOT = 3;   // K/V tile slots in LDS
constexpr int kBsP = 16;   // tokens per page (paged sources)
constexpr float kNegInf = -__builtin_inff();
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// K/V sources of the kernel: this step's contiguous rows, or the paged cache
// (f16 / bf16 pages by load-to-LDS transfers; q8_0 / q4_0 and TurboQuant
// pages (key / value bits 3/3, 4/4, 3/4; fp8 keys with 4-bit values)
// dequantized to fp16 through registers)
constexpr int SRC_LOCAL = 0, SRC_PAGED = 1, SRC_Q8 = 2, SRC_Q4 = 3, SRC_TQ33 = 4, SRC_TQ44 = 5, SRC_TQ34 = 6,
              SRC_K8 = 7;

struct PrefillParams {
    uint16_t* out;
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    const int32_t* pos;
    // paged sources: pools, block tables [seq][max_blocks], token -> sequence
    const uint8_t* kp;
    const uint8_t* vp;
    const int32_t* bt;
    const int32_t* tok_seq;
    int64_t max_blocks, page_bytes;
    int num_seqs;        // rows of a sequence outside [0, num_seqs) get no keys
    int q_bf16;          // paged: q / out (TurboQuant: and the stored halves) are bf16
    // TurboQuant slots: Lloyd-Max centroids, 1 / sqrt(d), field offsets
    float cent[16];
    uint32_t sq_plane[16];  // cent[i]^2 / sq_unit, rounded: byte planes (tq_lut.hpp)
    float sq_unit;
    float rot_c;
    int mse_bytes, key_packed, val_data;
    int norm_corr;  // keys scaled by 1 / ||C[codes]|| (else by the stored norm alone)
    int fp8_e4b15;  // fp8 keys: e4b15 (1) or e4m3 (0) codes
    int T, Hq, Hkv, G;
    float scale_log2;
    int ntiles;          // query blocks of qb rows
    int hw, rb, qb;      // heads per workgroup, 32-row blocks per head, rows per block
    int ks;              // parts of a tile's keys, a wave each (1 or 2)
    int hgroups;         // workgroups per KV head and query block (G / hw)
    // fused append
    uint8_t* kc;
    uint8_t* vc;
    const int64_t* slots;
    int64_t bs, E, stride;
    int hnd;
    // local K/V with a workspace: the V^T tiles of every 64-key tile of the
    // step (vt_prep_kernel) and their exact-mode flags, vt_tiles per KV head
    const uint8_t* vt;
    const uint8_t* vt_flag;
    int vt_tiles;
};

// The kernel of (bf16, fmt, src, vt), one translation unit per key split:
// KS = 1, a wave takes a tile's 64 keys; KS = 2, the halves of a tile go to
// two waves (prefill_split.hip).  fmt: the fused append's format or -1; src:
// SRC_*; vt: prebuilt V^T tiles (local bf16 K/V).
int launch_prefill_whole(PrefillParams& prm, bool bf16, int fmt, int src, bool vt, hipStream_t s);
int launch_prefill_split(PrefillParams& prm, bool bf16, int fmt, int src, bool vt, hipStream_t s);

namespace {

// All LDS of the kernel: the per-wave exchange, the fp16 V^T tiles (128
// rows of 64 keys, 16-byte chunk i of row d at position i ^ ((d >> 1) & 7)),
// then the K / raw V tile ring (rows of 256 B, 16-byte chunk ch of row r
// stored at chunk position ch ^ swz(r)).  In that order every V^T read and
// the K reads of slot 0 sit below 64 KB, where their constant part fits the
// 16-bit offset of the LDS instruction (above it, each address costs a
// vector add: 704-710 vs 712-720 us on the 4 x 4096 prefill).  swz(r) rotates the low
// 4 row bits by two: a bijection on 16 consecutive rows (the 32-row K
// operand reads spread over all banks) whose bits 2-3 differ for 4
// consecutive rows (the transpose reads of 4 rows x 16 dims spread too).
struct PrefillLds {
    float scratch[2][NW][32];            // [alpha, l][wave][row]
    alignas(8) uint8_t wide[NSLOT][NW];  // bf16: wave w's V rows of the tile need the exact mode
    float tq_base[2][16];                // TurboQuant: key centroids, value codes 0 .. 15
    uint32_t tq_sq[16];                  // squared centroids, 32-bit fixed point, as byte planes
    alignas(16) uint8_t vtr[NSLOT][kD * BN * 2];  // [slot][dim][kv position] fp16 V^T
    uint8_t tile[NSLOT][2][BN * 256];             // [slot][K, V][row][position]
};

__device__ __forceinline__ int swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

__device__ __forceinline__ int wave_max_int(int v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = max(v, __shfl_xor(v, m, kWave));
    return v;
}

// Workgroup = 8 waves = hw query heads of one KV head x rb blocks of 32
// query rows (hw * rb = 8): every K/V tile in LDS serves 256 query rows,
// which halves the tile traffic from L2 against 4-wave, one-head
// workgroups.  Grid: query block (largest first) x KV head x head group.
// BF16 is the type of the S MFMA and of V (paged: the page type; q8_0 /
// q4_0 pages dequantize to fp16).
template <bool BF16, int APPEND_FMT, int SRC, bool VT, int KS>
__global__ void __launch_bounds__(512, 1)
prefill_kernel(PrefillParams p) {
    using M = MT<BF16>;
    using V8 = typename M::v8;
    constexpr bool kPaged = SRC != SRC_LOCAL;
    __shared__ PrefillLds lds;

    const int tid = threadIdx.x;
    const int w = tid >> 6, lane = tid & 63;
    const int c32 = lane & 31, h = lane >> 5;
    const int per_blk = p.Hkv * p.hgroups;
    const int qblk = p.ntiles - 1 - (int)(blockIdx.x / per_blk);
    const int gi = (int)blockIdx.x % per_blk;
    const int g = gi / p.hgroups, hgrp = gi % p.hgroups;
    // wave w: head and row block w % (NW / KS), key part w / (NW / KS)
    const int wb = w & (NW / KS - 1);
    const int kh = __builtin_amdgcn_readfirstlane(w / (NW / KS));
    const int hq = g * p.G + hgrp * p.hw + wb / p.rb;  // this wave's query head
    const int T = p.T;
    const int q0 = qblk * p.qb;
    const int q_end = min(q0 + p.qb, T);
    // q / out dtype: the MFMA type for local rows, the caller's for pages
    const bool qbf = kPaged ? p.q_bf16 != 0 : BF16;

    // this lane's query row
    const int wr = 32 * (wb % p.rb);  // this wave's rows: q0 + wr .. +31
    const int row = q0 + wr + c32;
    const bool row_ok = row < T;
    const int wrow0 = q0 + wr;

    // pass state: the workgroup's kv range [kv_lo, kv_end) in ntile tiles,
    // this lane's key window [lo, hi] (hi < 0: none) and the wave's bounds of
    // both; rows [cur, rend) are the pass's.  Local rows: one pass, kv index =
    // token index, window [row - pos(row), row].  Pages: one pass per
    // sequence among the workgroup's rows, kv index = position, window
    // [0, pos(row)] through that sequence's block table.
    int kv_lo = 0, kv_end = 0, ntile = 0, lo = 0, hi = -1;
    int wlo_min = 0, wlo_max = 0, whi_min = -1, whi_max = -1;
    int cur = q0, rend = q_end;
    // block-table row of the pass's sequence, read through the constant
    // address space so that wave-uniform lookups are scalar loads (a vector
    // load would need a vmcnt wait, which also waits for the tile transfers)
    using cint = const __attribute__((address_space(4))) int32_t;
    cint* bt_row = (cint*)p.bt;
    int last_page = 0;

    // ---- Q^T operand: lane (col = row, half h) holds dims 16s + 8h .. +7.
    // A negative scale flips Q's sign bits (exact) so that c = |scale| log2 e
    // is positive and the largest raw score is the largest scaled one.  Paged
    // q of the other half type is rounded to the MFMA type.
    const float csc = fabsf(p.scale_log2);
    const uint32_t qflip = p.scale_log2 < 0.0f ? 0x80008000u : 0u;
    V8 qb[8];
    {
        const uint16_t* qp = p.q + ((int64_t)row * p.Hq + hq) * kD + 8 * h;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            u32x4 wv = {0u, 0u, 0u, 0u};
            if (row_ok) wv = *reinterpret_cast<const u32x4*>(qp + 16 * s);
            if constexpr (kPaged) {
                if (qbf != BF16) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float f0 = qbf ? __builtin_bit_cast(float, wv[e] << 16) : f16_bits_to_f32(wv[e] & 0xffff);
                        const float f1 = qbf ? __builtin_bit_cast(float, wv[e] & 0xffff0000u) : f16_bits_to_f32(wv[e] >> 16);
                        wv[e] = BF16 ? ((uint32_t)f32_to_bf16_bits(f0) | ((uint32_t)f32_to_bf16_bits(f1) << 16))
                                     : ((uint32_t)f32_to_f16_bits(f0) | ((uint32_t)f32_to_f16_bits(f1) << 16));
                    }
                }
            }
            qb[s] = as_v8<V8>(u32x4{wv[0] ^ qflip, wv[1] ^ qflip, wv[2] ^ qflip, wv[3] ^ qflip});
        }
    }
    if constexpr (SRC >= SRC_TQ33 && SRC != SRC_K8) {
        // TurboQuant keys are stored rotated: q_rot = H q / sqrt(d), in fp32
        // from the raw q.  Dim 16 s + 8 h + e: butterflies over e (half-widths
        // 1, 2, 4) and s (16, 32, 64) in the lane, over h (8) with the lane
        // 32 apart; then fp16.
        const uint16_t* qp = p.q + ((int64_t)row * p.Hq + hq) * kD + 8 * h;
        float y[8][8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            u32x4 wv = {0u, 0u, 0u, 0u};
            if (row_ok) wv = *reinterpret_cast<const u32x4*>(qp + 16 * s);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[s][2 * e] = qbf ? __builtin_bit_cast(float, wv[e] << 16) : f16_bits_to_f32(wv[e] & 0xffff);
                y[s][2 * e + 1] = qbf ? __builtin_bit_cast(float, wv[e] & 0xffff0000u) : f16_bits_to_f32(wv[e] >> 16);
            }
        }
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int hw = 1; hw < 8; hw <<= 1)
#pragma unroll
                for (int i = 0; i < 8; i += 2 * hw)
#pragma unroll
                    for (int j = i; j < i + hw; ++j) {
                        const float a = y[s][j], b = y[s][j + hw];
                        y[s][j] = a + b;
                        y[s][j + hw] = a - b;
                    }
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float o = shfl_xor(y[s][e], 32);
                y[s][e] = h ? o - y[s][e] : y[s][e] + o;
            }
#pragma unroll
        for (int hw = 1; hw < 8; hw <<= 1)
#pragma unroll
            for (int i = 0; i < 8; i += 2 * hw)
#pragma unroll
                for (int j = i; j < i + hw; ++j)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float a = y[j][e], b = y[j + hw][e];
                        y[j][e] = a + b;
                        y[j + hw][e] = a - b;
                    }
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            uint32_t wd[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                wd[e] = ((uint32_t)f32_to_f16_bits(y[s][2 * e] * p.rot_c) |
                         ((uint32_t)f32_to_f16_bits(y[s][2 * e + 1] * p.rot_c) << 16)) ^ qflip;
            qb[s] = as_v8<V8>(u32x4{wd[0], wd[1], wd[2], wd[3]});
        }
        if (tid < 32) lds.tq_base[tid >> 4][tid & 15] = tid < 16 ? p.cent[tid] : (float)(tid & 15);
        if (tid < 16) lds.tq_sq[tid] = p.sq_plane[tid];
        __syncthreads();
    }

    f32x16 o[4];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[m][i] = 0.0f;
    // m_run: the row's reference max (log2 units); it moves only when a score
    // exceeds it by more than 8, so P <= 256 and most tiles skip the rescale
    float m_run = kNegInf, m_thr = kNegInf, l_part = 0.0f;

    // ---- tile loads: load-to-LDS, 2 rounds of 32 rows per tensor; lane
    // (wave w, lane L) of round i fills row 32 i + 4 w + L / 16 at chunk
    // position L % 16, i.e. source chunk (L % 16) ^ swz(row)
    const int ld_row = 4 * w + (lane >> 4);
    const uint32_t ld_col = 16u * (uint32_t)((lane & 15) ^ swz(ld_row));
    const int64_t row_stride = (int64_t)p.Hkv * kD * 2;  // bytes between kv rows
    const uint8_t* kg = reinterpret_cast<const uint8_t*>(p.k) + (int64_t)g * kD * 2 + ld_col;
    const uint8_t* vg = reinterpret_cast<const uint8_t*>(p.v) + (int64_t)g * kD * 2 + ld_col;
    // pages: the 4 rows a 16-lane group covers lie in one page, so round i's
    // page is wave-uniform (a scalar block-table read); a hole reads page 0
    // and its keys are masked
    const int wu = __builtin_amdgcn_readfirstlane(w);
    auto page_at = [&](int k) __attribute__((always_inline)) {
        const int32_t pg = bt_row[min(k >> 4, last_page)];
        return max(pg, 0);
    };
    // byte offset of kv row k (< kv_end) inside its page
    auto row_in_page = [&](int k) __attribute__((always_inline)) {
        const int r = k & (kBsP - 1);
        return p.hnd ? (int64_t)(g * kBsP + r) * p.E : (int64_t)(r * p.Hkv + g) * p.E;
    };
    // local K/V: this lane's row of a tile starting at key k0 is k0 + ld_row
    // (+ 32 in the second round); the LDS rows of this wave in slot 0 (the
    // other slots and the V half at fixed offsets)
    // the fast path's transfers: uniform bases (this KV head's dims at the
    // tile's rows) plus this lane's row and chunk as a 32-bit offset
    const uint32_t ld_off = (uint32_t)ld_row * (uint32_t)row_stride + ld_col;
    const uint8_t* const kgu = reinterpret_cast<const uint8_t*>(p.k) + (int64_t)g * kD * 2;
    const uint8_t* const vgu = reinterpret_cast<const uint8_t*>(p.v) + (int64_t)g * kD * 2;
    const uint32_t lds_w = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)&lds.tile[0][0][1024 * w]);
    constexpr uint32_t kSlotB = 2 * BN * 256, kPartB = BN * 256;
    // prebuilt V^T tiles: wave w fetches bytes 2048 w .. + 2047 of the tile
    // into the same bytes of the slot's V^T tile
    const uint32_t vt_w = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)&lds.vtr[0][2048 * w]);
    const uint32_t lane16 = 16u * (uint32_t)lane;
    auto load_tile = [&](int t, auto slot_c, auto vt_c) __attribute__((always_inline)) {
        constexpr int SL = decltype(slot_c)::value;
        constexpr bool FROM_VT = decltype(vt_c)::value;
        const int k0 = kv_lo + t * BN;
        if constexpr (FROM_VT) {
            // kv_lo is a multiple of BN here, so the tile is prebuilt tile k0 / BN
            const uint8_t* src = p.vt + (((int64_t)g * p.vt_tiles + (k0 / BN)) << 14) + 2048 * wu;
            dma16s(src, lane16, vt_w + SL * (uint32_t)(kD * BN * 2));
            dma16s(src + 1024, lane16, vt_w + SL * (uint32_t)(kD * BN * 2) + 1024u);
        }
        if constexpr (SRC == SRC_LOCAL) {
            if (k0 + BN <= kv_end) {  // uniform: every row of the tile in range
                const int64_t toff = (int64_t)k0 * row_stride;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int64_t off = toff + (int64_t)(32 * i) * row_stride;
                    dma16s(kgu + off, ld_off, lds_w + SL * kSlotB + 8192u * i);
                    if constexpr (!FROM_VT) dma16s(vgu + off, ld_off, lds_w + SL * kSlotB + kPartB + 8192u * i);
                }
                return;
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            // rows past the range re-read the last row (masked later)
            const int kk = min(k0 + 32 * i + ld_row, kv_end - 1);
            if constexpr (SRC == SRC_LOCAL) {
                const int64_t off = (int64_t)kk * row_stride;
                dma16m(kg + off, lds_w + SL * kSlotB + 8192u * i);
                if constexpr (!FROM_VT) dma16m(vg + off, lds_w + SL * kSlotB + kPartB + 8192u * i);
            } else {
                const int64_t off = (int64_t)page_at(min(k0 + 32 * i + 4 * wu, kv_end - 1)) * p.page_bytes +
                                    row_in_page(kk) + ld_col;
                dma16m(p.kp + off, lds_w + SL * kSlotB + 8192u * i);
                dma16m(p.vp + off, lds_w + SL * kSlotB + kPartB + 8192u * i);
            }
        }
    };
    // q8_0 / q4_0 pages: lane L of wave w holds 32-dim block L & 3 of row
    // 32 (r >> 2) + 4 w + (r & 3), r = (L >> 2) & 7, of K (L < 32) or V --
    // the rows whose V this wave transposes -- as the block's bytes read
    // from their 4-byte floor (a block is 2-byte aligned; the read stays in
    // the entry)
    constexpr bool kTQ = SRC >= SRC_TQ33;
    constexpr bool kK8 = SRC == SRC_K8;  // fp8 keys: one byte per dim, 4-byte aligned
    constexpr int TKB = SRC == SRC_TQ44 ? 4 : kK8 ? 8 : 3, TVB = SRC == SRC_TQ33 ? 3 : 4;
    constexpr int kBE = SRC == SRC_Q8 ? 34 : 18;        // block bytes
    // words read per lane: GGUF block from its 4-byte floor; TurboQuant:
    // the 32 codes (12 / 16 / 32 bytes) from their floor, TKB + 1 words for K
    // lanes and TVB + 1 for V lanes (the reads end inside the slot), then the
    // norm (K) or the scale and zero (V) as 16-bit reads
    constexpr int kNC = kTQ ? (4 * (TKB > TVB ? TKB : TVB)) / 4 + 1 : 0;
    constexpr int kNW = SRC == SRC_Q8 ? 9 : SRC == SRC_Q4 ? 5 : kTQ ? kNC + 1 : 1;
    const int qr = 32 * ((lane >> 4) & 1) + 4 * w + ((lane >> 2) & 3);
    const int qblk_ = lane & 3;
    uint32_t qraw[kPaged && SRC != SRC_PAGED ? kNW : 1];
    uint32_t tq_sh = 0;  // TurboQuant: the code run's offset past its 4-byte floor (0 or 2)
    auto issue_q = [&](int t) __attribute__((always_inline)) {
        if constexpr (kTQ) {
            const int k0 = kv_lo + t * BN;
            const int kk = min(k0 + qr, kv_end - 1);
            const int pg0 = page_at(min(k0 + 4 * wu, kv_end - 1));
            const int pg1 = page_at(min(k0 + 32 + 4 * wu, kv_end - 1));
            const int pg = (lane & 16) ? pg1 : pg0;
            // slot fields: K codes at 0, the norm at mse_bytes, V codes at
            // key_packed, scale and zero at key_packed + val_data; block b's
            // codes at 4 bits b (the field offsets are multiples of 4 but for
            // key_packed, and a slot is 2-byte aligned)
            const uint8_t* slot = p.kp + (int64_t)pg * p.page_bytes + row_in_page(kk);
            const uint8_t* codes = lane < 32 ? slot + 4 * TKB * qblk_ : slot + p.key_packed + 4 * TVB * qblk_;
            const uint8_t* halves = lane < 32 ? slot + p.mse_bytes : slot + p.key_packed + p.val_data;
            tq_sh = (uint32_t)((uintptr_t)codes & 2u);
            const uint32_t* c4 = reinterpret_cast<const uint32_t*>((uintptr_t)codes & ~(uintptr_t)3);
            const uint16_t* h2 = reinterpret_cast<const uint16_t*>(halves);
#pragma unroll
            for (int i = 0; i < kNC; ++i) qraw[i] = (lane < 32 ? i <= TKB : i <= TVB) ? c4[i] : 0u;
            qraw[kNC] = (uint32_t)h2[0] | (lane < 32 ? 0u : (uint32_t)h2[1] << 16);
        } else if constexpr (SRC == SRC_Q8 || SRC == SRC_Q4) {
            const int k0 = kv_lo + t * BN;
            const int kk = min(k0 + qr, kv_end - 1);
            const int pg0 = page_at(min(k0 + 4 * wu, kv_end - 1));
            const int pg1 = page_at(min(k0 + 32 + 4 * wu, kv_end - 1));
            const int pg = (lane & 16) ? pg1 : pg0;
            // entries are whole dwords (136 / 72 bytes), so block b starts
            // 2 (b & 1) bytes past a dword
            const uint8_t* src = (lane < 32 ? p.kp : p.vp) + (int64_t)pg * p.page_bytes + row_in_page(kk) +
                                 kBE * qblk_ - 2 * (qblk_ & 1);
            const uint32_t* w4 = reinterpret_cast<const uint32_t*>(src);
#pragma unroll
            for (int i = 0; i < kNW; ++i) qraw[i] = w4[i];
        }
    };
    // dequantize the held block into the K or V tile of slot SL (fp16 rows
    // in the swizzled layout of the load-to-LDS path).  The 16 lanes of a
    // 16-byte write pass hold 4 rows x 4 blocks; written in order, lane
    // (row e, block b) puts chunk j at position 4 (b ^ e) + (j ^ const): 4
    // distinct positions, a 4-way bank conflict.  TurboQuant rows write chunk
    // (j + e) & 3 at step j instead: 16 distinct positions, all 64 banks.
    auto store_q = [&](auto slot_c) __attribute__((always_inline)) {
        if constexpr (SRC == SRC_Q8 || SRC == SRC_Q4 || kTQ) {
            constexpr int SL = decltype(slot_c)::value;
            if constexpr (kTQ && !kK8) {
                // A row's K (or V) holds at most 8 or 16 distinct fp16 values:
                // C[i] * norm / ||C[codes]|| (C[i] * norm without the norm
                // correction), or i * scale + zero.  They are computed once per
                // lane and block, split into low and high bytes, and looked up
                // four codes at a time by byte permutes (tq_lut.hpp): 1403 us
                // on 2048 tokens over a 30720-token prefix of 3-bit slots (4-bit
                // 1547), of which 1497 against 1687 came with the tables alone:
                // one LDS gather, multiply and conversion per code before.
                constexpr int NB = TKB > TVB ? TKB : TVB;
                using Lut = TqLut<NB>;
                const bool kpart = lane < 32;
                uint32_t c[NB];
#pragma unroll
                for (int i = 0; i < NB; ++i) c[i] = __builtin_amdgcn_alignbyte(qraw[i + 1], qraw[i], tq_sh);
                const uint32_t hw2 = qraw[kNC];
                auto half_f = [&](uint32_t b) {
                    return qbf ? __builtin_bit_cast(float, b << 16) : f16_bits_to_f32(b & 0xffffu);
                };
                // chunk j = codes 8j .. 8j+7; at step j this lane converts
                // chunk (j + rot) & 3, by two selects on the bits of rot (a
                // select by the chunk index compiles to divergent branches)
                const int rot = qr & 3;
                const bool r0 = (rot & 1) != 0, r1 = (rot & 2) != 0;
                auto turn = [&](uint32_t (&x)[4]) __attribute__((always_inline)) {
                    const uint32_t y0 = r0 ? x[1] : x[0], y1 = r0 ? x[2] : x[1];
                    const uint32_t y2 = r0 ? x[3] : x[2], y3 = r0 ? x[0] : x[3];
                    x[0] = r1 ? y2 : y0, x[1] = r1 ? y3 : y1, x[2] = r1 ? y0 : y2, x[3] = r1 ? y1 : y3;
                };
                uint32_t sel[4][2];
                {
                    uint32_t x3[4], x4[4];
                    if constexpr (TKB == 3) {
                        tq_chunks<3>(c, x3);
                        turn(x3);
                    }
                    if constexpr (NB == 4) {
                        tq_chunks<4>(c, x4);
                        turn(x4);
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        uint32_t s3[2] = {}, s4[2] = {};
                        if constexpr (TKB == 3) tq_spread<3>(x3[j], s3);
                        if constexpr (NB == 4) tq_spread<4>(x4[j], s4);
#pragma unroll
                        for (int u = 0; u < 2; ++u)
                            sel[j][u] = NB == 3 ? s3[u] : TKB == 4 ? s4[u] : kpart ? s3[u] : s4[u];
                    }
                }
                // ||C[codes]||^2 as a sum of 32-bit fixed-point squares (exact
                // integers; the four lanes of a quad hold the row's four blocks)
                float f = half_f(hw2), add = 0.0f;
                {
                    constexpr int NS = 1 << TKB;  // dwords: 2^TKB entries
                    uint32_t sq[NS];
#pragma unroll
                    for (int i = 0; i < NS; ++i) sq[i] = lds.tq_sq[i];
                    const float nrm = __builtin_amdgcn_rsqf(
                        __builtin_fmaf(tq_row_squares<TKB>(sel, sq, lane), p.sq_unit, 1e-16f));
                    if (kpart) {
                        f *= p.norm_corr ? nrm : 1.0f;
                    } else {
                        add = half_f(hw2 >> 16);
                    }
                }
                Lut lut;
                {
                    float base[1 << NB];
#pragma unroll
                    for (int i = 0; i < (1 << NB); ++i) base[i] = lds.tq_base[lane >> 5][i];
                    lut.build(base, f, add);
                }
                uint8_t* dst = lds.tile[SL][lane >> 5] + qr * 256;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const u32x2 a = lut.pick(sel[j][0]), b = lut.pick(sel[j][1]);
                    const u32x4 x = {a[0], a[1], b[0], b[1]};
                    *reinterpret_cast<u32x4*>(dst + 16 * ((4 * qblk_ + ((j + rot) & 3)) ^ swz(qr))) = x;
                }
            } else if constexpr (kK8) {
                // fp8 keys: each of the lane's 32 bytes is exact in fp16;
                // V = code * scale + zero
                u32x4 kw[4];
                constexpr int NC = 4 * TKB / 4;  // code dwords
                uint32_t c[NC];
#pragma unroll
                for (int i = 0; i < NC; ++i) c[i] = __builtin_amdgcn_alignbyte(qraw[i + 1], qraw[i], tq_sh);
                const uint32_t hw2 = qraw[kNC];
                auto half_f = [&](uint32_t b) {
                    return qbf ? __builtin_bit_cast(float, b << 16) : f16_bits_to_f32(b & 0xffffu);
                };
                if (lane < 32) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int b = 8 * j + 2 * e;  // bytes b and b + 1 share a word
                            const uint32_t wv = c[b >> 2] >> (8 * (b & 3));
                            kw[j][e] = (uint32_t)fp8_f16_bits(wv, p.fp8_e4b15) |
                                       ((uint32_t)fp8_f16_bits(wv >> 8, p.fp8_e4b15) << 16);
                        }
                } else {
                    const float vs = half_f(hw2), vz = half_f(hw2 >> 16);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const uint32_t b = c[j] >> (8 * e);
                            kw[j][e] = (uint32_t)f32_to_f16_bits(__builtin_fmaf((float)(b & 15u), vs, vz)) |
                                       ((uint32_t)f32_to_f16_bits(__builtin_fmaf((float)((b >> 4) & 15u), vs, vz)) << 16);
                        }
                }
                // chunk (j + rot) & 3 at step j, by two selects on the bits
                // of rot (a select by the chunk index compiles to divergent
                // branches)
                uint8_t* dst = lds.tile[SL][lane >> 5] + qr * 256;
                const int rot = qr & 3;
                const bool b0 = (rot & 1) != 0, b1 = (rot & 2) != 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    u32x4 x;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t t0 = b0 ? kw[(j + 1) & 3][e] : kw[j][e];
                        const uint32_t t1 = b0 ? kw[(j + 3) & 3][e] : kw[(j + 2) & 3][e];
                        x[e] = b1 ? t1 : t0;
                    }
                    *reinterpret_cast<u32x4*>(dst + 16 * ((4 * qblk_ + ((j + rot) & 3)) ^ swz(qr))) = x;
                }
            } else {
                // q8_0 / q4_0: each chunk written as soon as it is converted,
                // in order (measured faster here than the conflict-free order,
                // which needs all four chunks held)
                const bool off2 = (qblk_ & 1) != 0;
                constexpr int NC = SRC == SRC_Q8 ? 8 : 4;  // code dwords
                uint32_t c[NC];
#pragma unroll
                for (int i = 0; i < NC; ++i)
                    c[i] = off2 ? qraw[i + 1] : __builtin_amdgcn_alignbyte(qraw[i + 1], qraw[i], 2);
                const uint32_t d16 = off2 ? qraw[0] >> 16 : qraw[0] & 0xffffu;
                const f16x2 d2 = __builtin_bit_cast(f16x2, d16 * 0x10001u);
                uint8_t* dst = lds.tile[SL][lane >> 5] + qr * 256;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    u32x4 kw;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if constexpr (SRC == SRC_Q8) {
                            const uint32_t wv = c[2 * j + (e >> 1)];  // values 8j + 2e, +1
                            kw[e] = q8_pair_f16((e & 1) ? wv >> 16 : wv, d2);
                        } else {
                            const uint32_t wv = c[2 * (j & 1) + (e >> 1)];  // byte i: value i | value i+16 << 4
                            kw[e] = q4_pair_f16((e & 1) ? wv >> 16 : wv, j >= 2 ? 4 : 0, d2);
                        }
                    }
                    *reinterpret_cast<u32x4*>(dst + 16 * ((4 * qblk_ + j) ^ swz(qr))) = kw;
                }
            }
        }
    };

    // ---- this wave's keys of a tile: NKB blocks of 32 from 32 NKB kh on, NC
    // P V chunks of 16
    constexpr int NKB = 2 / KS, NC = 2 * NKB;
    // ---- loop-invariant LDS read offsets
    // K (S^T A operand): lane reads row 32 kb + c32, chunk 2 s + h
    int k_rd[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) k_rd[s] = c32 * 256 + 16 * ((2 * s + h) ^ swz(c32));
    // V^T (PV B operand): lane (n = c32, h) reads dim 32 m + n, kv positions
    // 16 c + 8 h .. +7 = 16-byte chunk 2 c + h of the 128-byte row, stored at
    // chunk (2 c + h) ^ ((dim >> 1) & 7); m enters as an immediate offset
    int vt_rd[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) vt_rd[c] = c32 * 128 + 16 * ((2 * (NC * kh + c) + h) ^ ((c32 >> 1) & 7));
    // transposing LDS reads: lane (e, q) of a 16-lane group addresses row
    // base + e, dims 4q .. 4q+3 of a 16-dim block; lane j receives dim j of
    // the 4 rows
    const int tq_e = (lane >> 2) & 3, tq_q = lane & 3, tq_j = lane & 15;

    auto process = [&](int t, auto slot_c, auto exact_c) __attribute__((always_inline)) {
        constexpr int SL = decltype(slot_c)::value;
        constexpr bool EXACT = decltype(exact_c)::value;
        const int k0 = kv_lo + t * BN + 32 * NKB * kh;
        // skip: keys entirely after this wave's last key, or before its first window
        const bool active = k0 <= whi_max && k0 + 32 * NKB - 1 >= wlo_min;
        if (!active) return;
        const uint8_t* kt = lds.tile[SL][0] + 32 * NKB * 256 * kh;
        const uint8_t* vtt = lds.vtr[SL];
        // pages: bit q set when page q of the keys is a hole (its keys masked)
        uint32_t holes = 0;
        if constexpr (kPaged) {
            // loaded together, before any is looked at (a page past the last
            // one counts as the last one; its keys are masked anyway).  One by
            // one, each scalar load was waited for: 1516 against 1487 us on
            // 2048 tokens over a 30720-token prefix of 3-bit slots.
            int32_t pg[NC];
#pragma unroll
            for (int q = 0; q < NC; ++q) pg[q] = bt_row[min((k0 >> 4) + q, last_page)];
#pragma unroll
            for (int q = 0; q < NC; ++q) holes |= ((uint32_t)pg[q] >> 31) << q;
        }
        const bool need_mask = (k0 + 32 * NKB - 1 > whi_min) || (k0 < wlo_max) || holes != 0;
        // ---- S^T = K Q^T, 32-row kv blocks
        f32x16 sacc[NKB];
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i) sacc[kb][i] = 0.0f;
        {
            // the kv blocks' chains interleaved; K operands read two steps
            // ahead of their MFMAs (with one block the compiler drops the
            // group barriers' order, so each step is fenced)
            u32x4 ka[8][NKB];
            auto read_k = [&](int s) __attribute__((always_inline)) {
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb)
                    ka[s][kb] = *reinterpret_cast<const u32x4*>(kt + kb * 32 * 256 + k_rd[s]);
            };
            if constexpr (NKB == 1) {
#pragma unroll
                for (int s = 0; s < 3; ++s) read_k(s);
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    __builtin_amdgcn_sched_barrier(0);
                    sacc[0] = M::mma(as_v8<V8>(ka[s][0]), qb[s], sacc[0]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (s + 3 < 8) read_k(s + 3);
                }
            } else {
#pragma unroll
                for (int s = 0; s < 8; ++s) read_k(s);
#pragma unroll
                for (int s = 0; s < 8; ++s)
#pragma unroll
                    for (int kb = 0; kb < NKB; ++kb) sacc[kb] = M::mma(as_v8<V8>(ka[s][kb]), qb[s], sacc[kb]);
                __builtin_amdgcn_sched_group_barrier(0x100, 2 * NKB, 0);
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    if (s < 6) __builtin_amdgcn_sched_group_barrier(0x100, NKB, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, NKB, 0);
                }
            }
        }
        // ---- online softmax (log2 domain), one query row per lane column;
        // masked scores become -inf (only tiles that cross a window edge)
        if (need_mask) {
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int kv = k0 + kb * 32 + 8 * (j >> 2) + 4 * h + (j & 3);
                    const bool ok = kv <= hi && kv >= lo && !((holes >> (2 * kb + (j >> 3))) & 1u);
                    sacc[kb][j] = ok ? sacc[kb][j] : kNegInf;
                }
        }
        float mloc = kNegInf;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int j = 0; j < 16; ++j) mloc = fmaxf(mloc, sacc[kb][j]);
        if (__ballot(mloc * csc > m_thr)) {  // wave-uniform; rare after the first tiles
            const float mrow = fmaxf(mloc, shfl_xor(mloc, 32)) * csc;
            const bool upd = mrow > m_thr;  // the same in both halves of the row
            const float m_new = upd ? mrow : m_run;
            const float alpha = upd ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;  // 0 from -inf
            l_part *= alpha;
            m_run = m_new;
            m_thr = m_run + 8.0f;
            // rescale O rows by their query rows' alpha (rows 8b + 4h + i)
            float* sc = lds.scratch[0][w];
            if (h == 0) sc[c32] = alpha;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            float al[16];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const f32x4 a4 = *reinterpret_cast<const f32x4*>(sc + 8 * b + 4 * h);
#pragma unroll
                for (int i = 0; i < 4; ++i) al[4 * b + i] = a4[i];
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[m][i] *= al[i];
        }
        const float m_use = m_run == kNegInf ? 0.0f : m_run;
        if constexpr (EXACT) {
            // ---- exact mode (bf16 V that fp16 cannot hold): P = 2^(s c - m)
            // in fp32 splits into bf16 hi + lo (16 significant bits, fp32
            // range), the row sum adds the same parts, and O += P V runs as two
            // bf16 MFMAs on the raw bf16 V rows, read by transposing reads:
            // lane (n = c32, h) gets kv 16c + 4h + 0..3 and 16c + 8 + 4h + 0..3
            // at dim 32m + n, the k order of the fp16 path.  Row
            // 16c + 8sec + 4h + e has swz = 4e + ((2 sec + h) & 3), so chunk
            // 4m + cb sits at 4 (m ^ e) + (cb ^ h ^ 2 sec).  The lane id is
            // opaque here so that none of this is computed ahead, in
            // registers the fast pass needs.
            uint32_t phi[NC][4], plo[NC][4];
            float psum = 0.0f;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const int kb = c >> 1;
                    const int j0 = 4 * (2 * (c & 1) + (e >> 2)) + (e & 3);
                    uint32_t hb[2], lb[2];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][j0 + u], csc, -m_use));
                        hb[u] = __builtin_bit_cast(uint32_t, pv) & 0xffff0000u;
                        const float r = pv - __builtin_bit_cast(float, hb[u]);  // exact
                        lb[u] = __builtin_bit_cast(uint32_t, r) & 0xffff0000u;
                        psum += __builtin_bit_cast(float, hb[u]) + __builtin_bit_cast(float, lb[u]);
                    }
                    phi[c][e >> 1] = (hb[0] >> 16) | hb[1];
                    plo[c][e >> 1] = (lb[0] >> 16) | lb[1];
                }
            l_part += psum;
            int ln = lane;
            asm volatile("" : "+v"(ln));
            const int le = (ln >> 2) & 3, lq = ln & 3, lh = ln >> 5;
            const int cbh = (2 * ((ln >> 4) & 1) + (lq >> 1)) ^ lh;
            const uint32_t vbase = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)
                                       lds.tile[SL][1] +
                                   (uint32_t)((4 * lh + le) * 256 + 8 * (lq & 1) + 32 * NKB * 256 * kh);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const bf16x8 ah = as_v8<bf16x8>(u32x4{phi[c][0], phi[c][1], phi[c][2], phi[c][3]});
                const bf16x8 al = as_v8<bf16x8>(u32x4{plo[c][0], plo[c][1], plo[c][2], plo[c][3]});
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    s16x4 part[2];
#pragma unroll
                    for (int sec = 0; sec < 2; ++sec) {
                        const uint32_t a = vbase + (uint32_t)(4096 * c + 2048 * sec + 64 * (m ^ le) +
                                                              16 * (cbh ^ (2 * sec)));
                        part[sec] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (__attribute__((address_space(3))) s16x4*)(uintptr_t)a);
                    }
                    const u32x2 p0 = __builtin_bit_cast(u32x2, part[0]);
                    const u32x2 p1 = __builtin_bit_cast(u32x2, part[1]);
                    const bf16x8 vb = as_v8<bf16x8>(u32x4{p0[0], p0[1], p1[0], p1[1]});
                    o[m] = MT<true>::mma(ah, vb, o[m]);
                    o[m] = MT<true>::mma(al, vb, o[m]);
                }
            }
        } else {
            // P = 2^(s c - m) in fp16 (11 bits, also for bf16 inputs) as MFMA A
            // operands, chunk c = kv rows 16c .. 16c+15; the row sum adds the
            // rounded values the MFMA uses
            uint32_t pw[NC][4];
            float psum = 0.0f;
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const int kb = c >> 1;
                    const int j0 = 4 * (2 * (c & 1) + (e >> 2)) + (e & 3);
                    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][j0], csc, -m_use));
                    const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[kb][j0 + 1], csc, -m_use));
                    const f16x2 ph = {(_Float16)p0, (_Float16)p1};
                    psum = __builtin_amdgcn_fdot2(ph, f16x2{(_Float16)1.0f, (_Float16)1.0f}, psum, false);
                    pw[c][e >> 1] = __builtin_bit_cast(uint32_t, ph);
                }
            l_part += psum;
            // ---- O += P V (fp16): k = 8h + e <-> kv 16c + 8(e/4) + 4h + e%4 (the
            // S^T registers' order); V arrives transposed, output column n = dim 32m + n
            u32x4 vb[NC][4];
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    vb[c][m] = *reinterpret_cast<const u32x4*>(vtt + m * 32 * 128 + vt_rd[c]);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const f16x8 pa = as_v8<f16x8>(u32x4{pw[c][0], pw[c][1], pw[c][2], pw[c][3]});
#pragma unroll
                for (int m = 0; m < 4; ++m) o[m] = MT<false>::mma(pa, as_v8<f16x8>(vb[c][m]), o[m]);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
            for (int i = 0; i < 4 * NC; ++i) {
                if (i < 4 * NC - 2) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
        }
    };

    // V^T pass: each wave transposes the 8 V rows its own transfers wrote
    // (rows 32 rs + 4 w + 0..3, rs = 0, 1) into the fp16 V^T tile, by
    // transpose reads (16-lane group: 4 rows x 16 dims) and 8-byte writes.
    // Within each 16-key block, kv 8a + 4h + e sits at position 8h + 4a + e,
    // so the PV B operand of lane half h is one contiguous 16-byte chunk.
    // bf16 inputs are converted to fp16 here, which keeps every bit for
    // 2^-17 <= |v| < 65536 and rounds smaller magnitudes to the subnormal
    // grid (absolute error <= 2^-25).  The wave's rows are marked in
    // lds.wide (exact mode for the workgroup) when they hold |v| >= 65536 or
    // a NaN, or when they hold a value below 2^-17 but none of 2^-8 or more;
    // otherwise the rounding error is at most 2^-17 of their largest |v|.
    auto v_transpose = [&](auto slot_c) __attribute__((always_inline)) {
        constexpr int SL = decltype(slot_c)::value;
        const uint8_t* vr = lds.tile[SL][1];
        uint8_t* vtt = lds.vtr[SL];
        u16x2 amax = {0, 0}, amin1 = {0xffff, 0xffff};  // |bits|, |bits| - 1 (0 wraps)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int combo = 4 * i + (lane >> 4);
            const int rs = combo & 1, dblk = combo >> 1;
            const int r = 32 * rs + 4 * w + tq_e;
            const int chunk = 2 * dblk + (tq_q >> 1);
            const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) s16x4*)(vr + r * 256 + 16 * (chunk ^ swz(r)) + 8 * (tq_q & 1)));
            u32x2 y = __builtin_bit_cast(u32x2, x);
            if constexpr (BF16) {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const u16x2 a = __builtin_bit_cast(u16x2, y[e] & 0x7fff7fffu);
                    amax = __builtin_elementwise_max(amax, a);
                    amin1 = __builtin_elementwise_min(amin1, a - u16x2{1, 1});
                    const f16x2 hh = {(_Float16)__builtin_bit_cast(float, y[e] << 16),
                                      (_Float16)__builtin_bit_cast(float, y[e] & 0xffff0000u)};
                    y[e] = __builtin_bit_cast(uint32_t, hh);
                }
            }
            const int dim = 16 * dblk + tq_j;
            const int ci = 2 * (2 * rs + (w >> 2)) + (w & 1);
            *reinterpret_cast<u32x2*>(vtt + dim * 128 + 16 * (ci ^ ((dim >> 1) & 7)) + 8 * ((w >> 1) & 1)) = y;
        }
        if constexpr (BF16) {
            // bf16 bit patterns: 0x477f = 65280 (largest below 2^16),
            // 0x3700 = 2^-17, 0x3b80 = 2^-8
            const uint32_t mx = max((uint32_t)amax[0], (uint32_t)amax[1]);
            const uint32_t mn1 = min((uint32_t)amin1[0], (uint32_t)amin1[1]);
            const bool ovf = __ballot(mx > 0x477fu) != 0;
            const bool small = __ballot(mn1 < 0x36ffu) != 0;
            const bool big = __ballot(mx >= 0x3b80u) != 0;
            if (lane == 0) lds.wide[SL][w] = ovf || (small && !big);
        }
    };

    // ---- NSLOT LDS slots: tile t in slot t % NSLOT; the next NSLOT - 1 tiles
    // are in flight while t runs.  Before tile t each wave waits until only
    // the transfers of tiles t+1 .. t+NSLOT-2 are outstanding (4 per tile:
    // vmcnt retires loads in order), converts its own V chunks, and the
    // barrier makes the tile visible and shows slot (t-1) % NSLOT free, which
    // then receives tile t + NSLOT - 1.
    // bf16: when a tile's V is not fp16-exact (a flag every wave reads after
    // the tile's barrier) the pass returns true and the workgroup starts over
    // in the exact mode, which skips the V^T pass and multiplies the raw bf16
    // rows.  The pass runs to its end rather than leaving early: an early
    // exit costs the common case registers.
    // Quantized pages instead hold the next tile in registers while a tile
    // runs and dequantize it into its slot before that tile's barrier.  The
    // two waves of a SIMD do so at opposite ends of the interval: waves 0 .. 3
    // after their products of tile t, waves 4 .. 7 before them, so that one's
    // vector work runs beside the other's matrix work (the slot of tile t + 1
    // was last read before the barrier of tile t - 1).  All eight after the
    // products: 1518 against 1444 us on 2048 tokens over a 30720-token prefix
    // of 3-bit slots, 1275 against 1264 us over q8_0 pages.
    // With prebuilt V^T tiles (FROM_VT) the transfers bring the V^T tile
    // instead of the raw V rows and there is no V^T pass; the exact mode was
    // decided before the pass from the tiles' flags.
    static_assert(NSLOT == 3, "wait counts below assume three slots");
    constexpr bool kDma = SRC == SRC_LOCAL || SRC == SRC_PAGED;
    const bool early = !kDma && wu >= NW / 2;
    auto run = [&](auto exact_c, auto vt_c) __attribute__((always_inline)) {
        constexpr bool EXACT = decltype(exact_c)::value;
        constexpr bool FROM_VT = decltype(vt_c)::value;
        bool redo = false;
        if constexpr (kDma) {
            load_tile(0, std::integral_constant<int, 0>{}, vt_c);
            if (1 < ntile) load_tile(1, std::integral_constant<int, 1>{}, vt_c);
        } else {
            issue_q(0);
        }
        for (int t0 = 0; t0 < ntile; t0 += NSLOT) {
            static_for<NSLOT>([&](auto sc) __attribute__((always_inline)) {
                constexpr int S = decltype(sc)::value;
                const int t = t0 + S;
                if (t < ntile) {  // uniform over the workgroup
                    if constexpr (kDma) {
                        if (t + 1 < ntile) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
                        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                        if constexpr (!EXACT && !FROM_VT) v_transpose(sc);
                    } else if (!early || t == 0) {
                        store_q(sc);
                        v_transpose(sc);
                        if (early && 1 < ntile) issue_q(1);
                    }
                    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    if constexpr (BF16 && !EXACT && !FROM_VT) {
                        const uint64_t wf = *reinterpret_cast<const uint64_t*>(lds.wide[S]);
                        redo |= (__builtin_amdgcn_readfirstlane((uint32_t)wf) |
                                 __builtin_amdgcn_readfirstlane((uint32_t)(wf >> 32))) != 0;
                    }
                    if constexpr (kDma) {
                        if (t + 2 < ntile) load_tile(t + 2, std::integral_constant<int, (S + 2) % NSLOT>{}, vt_c);
                    } else if (!early) {
                        if (t + 1 < ntile) issue_q(t + 1);
                    } else if (t + 1 < ntile) {
                        constexpr std::integral_constant<int, (S + 1) % NSLOT> nx{};
                        store_q(nx);
                        v_transpose(nx);
                        if (t + 2 < ntile) issue_q(t + 2);
                    }
                    process(t, sc, exact_c);
                }
            });
        }
        if constexpr (kDma) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        return redo;
    };
    auto run_pass = [&]() __attribute__((always_inline)) {
        if (run(std::false_type{}, std::false_type{})) {
            if constexpr (BF16) {
                __syncthreads();  // every wave is past its last read of the ring
                // the pass's rows start over: O rows 8b + 4h + i, this lane's row
#pragma unroll
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = wrow0 + 8 * b + 4 * h + i;
                        if (r >= cur && r < rend) {
#pragma unroll
                            for (int m = 0; m < 4; ++m) o[m][4 * b + i] = 0.0f;
                        }
                    }
                if (row >= cur && row < rend) {
                    m_run = kNegInf;
                    m_thr = kNegInf;
                    l_part = 0.0f;
                }
                run(std::true_type{}, std::false_type{});
            }
        }
    };

    if constexpr (SRC == SRC_LOCAL) {
        kv_lo = __builtin_amdgcn_readfirstlane(max(0, q0 - p.pos[q0]));  // uniform: scalar tile addresses
        kv_end = q_end;
        ntile = (kv_end - kv_lo + BN - 1) / BN;
        lo = row_ok ? row - p.pos[row] : 0;
        hi = row_ok ? row : -1;
        if (wrow0 < T) {  // rows increase, and so do their window starts
            const int wrow1 = min(wrow0 + 31, T - 1);
            whi_min = wrow0;
            whi_max = wrow1;
            wlo_min = wrow0 - p.pos[wrow0];
            wlo_max = wrow1 - p.pos[wrow1];
        }
        // prebuilt V^T tiles serve a workgroup whose tiles start on a 64-key
        // boundary; a workgroup whose sequence starts elsewhere transposes
        // its own tiles
        bool prebuilt = false;
        if constexpr (VT) {
            if ((kv_lo % BN) == 0) {
                bool flagged = false;
                const uint8_t* fl = p.vt_flag + (int64_t)g * p.vt_tiles + kv_lo / BN;
                for (int t0 = 0; t0 < ntile; t0 += 64)
                    flagged |= __ballot(t0 + lane < ntile && fl[t0 + lane] != 0) != 0;
                if (flagged) run(std::true_type{}, std::false_type{});  // the exact mode
                else run(std::false_type{}, std::true_type{});
                prebuilt = true;
            }
        }
        if (!prebuilt) run_pass();
    } else {
        // runs of rows of one sequence: every wave scans the workgroup's rows
        // and finds the same runs
        while (cur < q_end) {
            const int sq = p.tok_seq[cur];
            rend = q_end;
            int pmax = -1;
            for (int r0 = cur; r0 < rend; r0 += 64) {
                const int r = r0 + lane;
                const int sr = r < rend ? p.tok_seq[r] : sq;
                const uint64_t diff = __ballot(sr != sq);
                if (diff) rend = r0 + (int)__builtin_ctzll(diff);
                pmax = max(pmax, wave_max_int(r < rend ? p.pos[r] : -1));
            }
            pmax = __builtin_amdgcn_readfirstlane(pmax);
            if (sq >= 0 && sq < p.num_seqs && pmax >= 0) {
                kv_lo = 0;
                kv_end = pmax + 1;
                ntile = (kv_end + BN - 1) / BN;
                bt_row = (cint*)(p.bt + (int64_t)sq * p.max_blocks);
                last_page = min((kv_end - 1) >> 4, (int)p.max_blocks - 1);
                const bool in = row_ok && row >= cur && row < rend;
                hi = in ? p.pos[row] : -1;
                lo = 0;
                whi_max = __builtin_amdgcn_readfirstlane(wave_max_int(hi));
                whi_min = __builtin_amdgcn_readfirstlane(-wave_max_int(-hi));
                wlo_min = 0;
                wlo_max = 0;
                __syncthreads();  // the previous pass's last tiles are read before the ring refills
                run_pass();
            }
            cur = rend;
        }
    }

    // ---- normalise and store: lane holds rows 8b + 4h + i, dims 32m + c32.
    // Two key parts meet in LDS: the second's wave leaves its O (over the tile
    // ring), running max and sum, the first's adds them.
    {
        const float l_tot = l_part + shfl_xor(l_part, 32);
        float f0 = l_tot, f1 = 0.0f;
        f32x4* const other = reinterpret_cast<f32x4*>(lds.tile[0][0]) + 1024 * wb + lane;
        if constexpr (KS == 2) {
            __syncthreads();  // every wave is past its last read of the ring
            if (kh) {
#pragma unroll
                for (int m = 0; m < 4; ++m)
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        other[64 * (4 * m + b)] = f32x4{o[m][4 * b], o[m][4 * b + 1], o[m][4 * b + 2], o[m][4 * b + 3]};
                if (h == 0) {
                    lds.scratch[0][w][c32] = m_run;
                    lds.scratch[1][w][c32] = l_tot;
                }
            }
            __syncthreads();
            const float m1 = lds.scratch[0][wb + NW / 2][c32], l1 = lds.scratch[1][wb + NW / 2][c32];
            const float mx = fmaxf(m_run, m1), m_use = mx == kNegInf ? 0.0f : mx;
            const float a0 = __builtin_amdgcn_exp2f(m_run - m_use), a1 = __builtin_amdgcn_exp2f(m1 - m_use);
            const float l = __builtin_fmaf(a1, l1, a0 * l_tot);
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            f0 = a0 * inv;
            f1 = a1 * inv;
        } else {
            f0 = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
        }
        if (kh == 0) {
            float* sc = lds.scratch[0][w];
            float* sc1 = lds.scratch[1][w];
            if (h == 0) {
                sc[c32] = f0;
                if constexpr (KS == 2) sc1[c32] = f1;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const f32x4 g0 = *reinterpret_cast<const f32x4*>(sc + 8 * b + 4 * h);
                f32x4 g1, x1[4];
                if constexpr (KS == 2) {
                    g1 = *reinterpret_cast<const f32x4*>(sc1 + 8 * b + 4 * h);
#pragma unroll
                    for (int m = 0; m < 4; ++m) x1[m] = other[64 * (4 * m + b)];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = wrow0 + 8 * b + 4 * h + i;
                    if (r >= T) continue;
                    uint16_t* op = p.out + ((int64_t)r * p.Hq + hq) * kD + c32;
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        float x = o[m][4 * b + i] * g0[i];
                        if constexpr (KS == 2) x = __builtin_fmaf(x1[m][i], g1[i], x);
                        op[32 * m] = qbf ? f32_to_bf16_bits(x) : f32_to_f16_bits(x);
                    }
                }
            }
        }
    }

    // ---- fused quantize-on-append of this tile's K/V rows (once per KV head)
    if constexpr (APPEND_FMT >= 0) {
        if (hgrp == 0) {
            const int nrow = min(p.qb, T - q0);
            for (int item = tid; item < 2 * p.qb * 4; item += NW * 64) {  // [tensor][row][block]
                const int tensor = item / (p.qb * 4);
                const int r = (item >> 2) % p.qb;
                const int blk = item & 3;
                if (r >= nrow) continue;
                const int64_t slot = p.slots[q0 + r];
                if (slot < 0) continue;
                const uint16_t* src = (tensor ? p.v : p.k) + ((int64_t)(q0 + r) * p.Hkv + g) * kD + 32 * blk;
                uint8_t* dst = (tensor ? p.vc : p.kc) +
                               kv_entry_offset(slot, g, p.bs, p.Hkv, p.E, p.stride, p.hnd != 0);
                append_block32<APPEND_FMT, BF16>(src, dst, blk);
            }
        }
    }
}

template <bool BF16, int FMT, int SRC, bool VT, int KS>
int launch_prefill(PrefillParams& prm, hipStream_t stream) {
    auto kern = prefill_kernel<BF16, FMT, SRC, VT, KS>;
    const int64_t grid = (int64_t)prm.ntiles * prm.Hkv * prm.hgroups;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * NW), 0, stream, prm);
    VMC_LAUNCH_CHECK();
    return VMC_OK;
}

template <bool BF16, bool VT, int KS>
int launch_prefill_local(PrefillParams& prm, int fmt, hipStream_t s) {
    switch (fmt) {
        case -1: return launch_prefill<BF16, -1, SRC_LOCAL, VT, KS>(prm, s);
        case VMC_KV_F16: return launch_prefill<BF16, VMC_KV_F16, SRC_LOCAL, VT, KS>(prm, s);
        case VMC_KV_BF16: return launch_prefill<BF16, VMC_KV_BF16, SRC_LOCAL, VT, KS>(prm, s);
        case VMC_KV_Q8_0: return launch_prefill<BF16, VMC_KV_Q8_0, SRC_LOCAL, VT, KS>(prm, s);
        case VMC_KV_Q4_0: return launch_prefill<BF16, VMC_KV_Q4_0, SRC_LOCAL, VT, KS>(prm, s);
        default: return VMC_EINVAL;
    }
}

template <int KS>
int launch_prefill_any(PrefillParams& prm, bool bf16, int fmt, int src, bool vt, hipStream_t s) {
    switch (src) {
        case SRC_LOCAL:
            if (vt) return bf16 ? launch_prefill_local<true, true, KS>(prm, fmt, s) : VMC_EINVAL;
            return bf16 ? launch_prefill_local<true, false, KS>(prm, fmt, s)
                        : launch_prefill_local<false, false, KS>(prm, fmt, s);
        case SRC_PAGED:
            return bf16 ? launch_prefill<true, -1, SRC_PAGED, false, KS>(prm, s)
                        : launch_prefill<false, -1, SRC_PAGED, false, KS>(prm, s);
        case SRC_Q8: return launch_prefill<false, -1, SRC_Q8, false, KS>(prm, s);
        case SRC_Q4: return launch_prefill<false, -1, SRC_Q4, false, KS>(prm, s);
        case SRC_TQ33: return launch_prefill<false, -1, SRC_TQ33, false, KS>(prm, s);
        case SRC_TQ44: return launch_prefill<false, -1, SRC_TQ44, false, KS>(prm, s);
        case SRC_TQ34: return launch_prefill<false, -1, SRC_TQ34, false, KS>(prm, s);
        case SRC_K8: return launch_prefill<false, -1, SRC_K8, false, KS>(prm, s);
        default: return VMC_EINVAL;
    }
}

}  // namespace
}  // namespace vmc
