// prefill_hd.hip -- causal flash-attention prefill of head_dim 64 and 256 over
// this step's K/V rows, on MFMA.  The rows and their windows are
// gen_attn_kernel's (generic_attn.hip: token t attends tokens t - pos[t] .. t),
// which keeps operands that are not 16-byte aligned and the shortest steps.
//
// What bounds it: the matrix cores (4 D flops per query, key and head; P V
// counts three times, see below).  The one-wave-per-row kernel had no
// products and read K/V once per row (22.9 ms for 10,752 tokens in 4 prompts,
// 16/2 heads, head_dim 256, bf16: 12.5 TFLOP/s); this one takes 535 us (533
// TFLOP/s of the attention's own flops, 1.07 PFLOP/s on the matrix cores).
// Workgroup = 8 waves = up to 4 query heads of one KV head x 32-row query
// blocks, as prefill_kernel (prefill.hip), so a K/V tile of 64 keys in LDS
// serves 256 query rows; 4 waves and 128 rows where workgroups are few
// (prefill_hd).  Tiles arrive by load-to-LDS transfers: three slots
// at head_dim 64 (two tiles in flight), two at 256 (128 KB, one in flight).
//   S^T[32 keys x 32 rows] = K . Q^T, O^T[D x 32 rows] += V^T . P^T on
//   v_mfma_f32_32x32x16: a query row is one lane column in both, so its
//   running max, rescale and final division stay in the lane (and its partner
//   32 lanes on).  V^T operands come from the row-major tile by transposing
//   LDS reads; the contraction index is permuted as P leaves the S registers
//   (k = 8h + e <-> key 16c + 8 (e / 4) + 4h + e % 4).  Their LDS time hides
//   under the products, which take three MFMAs for each operand read.
// Head_dim 256 runs the softmax per 32 keys and 64 per 64: O, Q and S then
// fit the 256 registers of a wave at two waves per SIMD.
//
// Weights keep their 24 bits: P is the sum of three rounded 16-bit terms of V's
// own type, an MFMA each (weight_terms.hpp; fp16: scaled by 2^7 against
// underflow).  Two bf16 terms took 475 instead of 590 us on the case above with
// its append, the same error against 64 bits in the bf16 output (1.6e-3) but
// five times the wrongly rounded values (2.4e-3 of them against 4.4e-4; three
// terms 3.1e-4).  Two fp16 terms took 166 instead of 204 us (head_dim 64, 32/8
// heads, 4096 tokens) and 261 instead of 330 us (256, 16/2); they leave 22 bits
// of a weight, which no N(0, 1) input showed in the fp16 output (both round
// 1.8e-3 of the values wrongly at 256, the one-wave kernel 3.8e-3).  V of either
// type enters
// exactly.  A row whose sums are not finite reruns key by key (gen_row): its
// products met an infinity or a NaN, or bf16 V so large that weights of up to
// 2^8 (the reference max lags by that much) overflow where weights of 1 do not.
#include "device_cus.hpp"
#include "generic_row.hpp"
#include "prefill_dev.hpp"
#include "prefill_hd.hpp"
#include "weight_terms.hpp"

namespace vmc {
namespace {

constexpr int kHdBN = 64;  // keys per tile
// Steps of no more rows stay with the one-wave-per-row kernel, whatever their
// prompts (bf16, us there / here: head_dim 64, 14/2 heads, 8 rows 4.7 / 5.6, 17
// rows 6.2 / 5.5; 256, 16/2, 8 rows 7.9 / 9.8, 17 rows 9.0 / 10.6, 32 rows
// 12.2 / 12.2)
__host__ __device__ constexpr int hd_min_rows(int D) { return D == 256 ? 24 : 16; }

struct PrefillHdParams {
    uint16_t* out;
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    const int32_t* pos;
    int T, Hq, Hkv, G;
    float scale;
    int ntiles;       // query blocks of qb rows
    int hw, rb, qb;   // heads per workgroup, 32-row blocks per head, rows per block
    int hgroups;      // workgroups per KV head and query block
};

// chunk swizzle of a tile row of 2 D bytes: 16-byte chunk ch of row r sits at
// ch ^ swz(r).  16 consecutive rows x one chunk (K operands) and 4 rows x 64
// bytes (transposing V reads) each cover the 64 banks once.
template <int D>
__device__ __forceinline__ int hd_tile_swz(int r) {
    return D == 256 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
}

// One query head's row over keys k0 .. k1 - 1 by gen_row.  A call, not inlined:
// its registers stay out of the tile loop's.
template <int D, bool BF>
__device__ __noinline__ void prefill_row_exact(uint16_t* out, const uint16_t* q, const uint16_t* k, const uint16_t* v,
                                               int row_halfs, float scale, int n, float* qs) {
    const int lane = threadIdx.x & 63;
    GenArgs a = {};
    a.scale = scale;
    const TQTables none = {};
    wave_sync();
#pragma unroll
    for (int i = 0; i < D / 64; ++i) qs[lane + 64 * i] = half_to_f32<BF>(q[lane + 64 * i]);
    wave_sync();
    auto key_at = [&](int kk, const uint8_t*& ke, const uint8_t*& ve) __attribute__((always_inline)) {
        ke = reinterpret_cast<const uint8_t*>(k + (int64_t)kk * row_halfs);
        ve = reinterpret_cast<const uint8_t*>(v + (int64_t)kk * row_halfs);
        return true;
    };
    float m, l, acc[D / 64];
    gen_row<D, GEN_LOCAL, 0, 0, BF>(a, none, qs, lane, 0, n, key_at, m, l, acc);
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int i = 0; i < D / 64; ++i) out[lane + 64 * i] = f32_to_half<BF>(acc[i] * inv);
    wave_sync();
}

__device__ __forceinline__ int hd_wave_min(int v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = min(v, __shfl_xor(v, m, kWave));
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ int hd_wave_max(int v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = max(v, __shfl_xor(v, m, kWave));
    return __builtin_amdgcn_readfirstlane(v);
}

template <int D, bool BF, int W>
__global__ void __launch_bounds__(64 * W, D == 256 && W == 4 ? 1 : 2) prefill_hd_kernel(PrefillHdParams p) {
    using M = MT<BF>;
    using V8 = typename M::v8;
    constexpr int NS = D == 256 ? 2 : 3;        // tile slots
    constexpr int ROW = 2 * D, TILE = kHdBN * ROW;
    constexpr int NTR = TILE / (1024 * W);      // transfers per wave and tensor
    constexpr int NTERM = WeightTerms<BF>::n;   // 16-bit terms of a weight
    constexpr int HB = D == 256 ? 1 : 2;        // 32-key blocks per softmax round
    constexpr int KA = D == 256 && W == 4 ? 6 : 2, VA = D == 256 && W == 4 ? 4 : 1;  // operand reads ahead
    constexpr float kOff = BF ? 0.0f : 7.0f;    // weights are 2^(s - m + kOff), at most 2^15
    struct Lds {
        uint8_t tile[NS][2][TILE];  // [slot][K, V]
        float qs[W][D];             // rows that rerun key by key
    };
    __shared__ __attribute__((aligned(1024))) Lds lds;

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int c32 = lane & 31, h = lane >> 5;
    const int per_blk = p.Hkv * p.hgroups;
    const int qblk = p.ntiles - 1 - (int)(blockIdx.x / per_blk);  // long windows first
    const int gi = (int)blockIdx.x % per_blk;
    const int g = gi / p.hgroups, hgrp = gi % p.hgroups;
    const int hq = g * p.G + hgrp * p.hw + w / p.rb;
    const int T = p.T, q0 = qblk * p.qb, q_end = min(q0 + p.qb, T);
    const int wrow0 = q0 + 32 * (w % p.rb), row = wrow0 + c32;
    const bool row_ok = row < T;

    // ---- windows: this lane's [lo, hi] (hi < lo: none), the wave's bounds and
    // the workgroup's first key (each wave finds the same one)
    int first = q_end;
    for (int r = q0 + lane; r < q_end; r += 64) {
        const int ps = p.pos[r];
        if (ps >= 0) first = min(first, r - ps);
    }
    const int kv_lo = max(0, hd_wave_min(first)), kv_end = q_end;
    int lo = 0, hi = -1;
    if (row_ok) {
        const int ps = p.pos[row];
        if (ps >= 0) {
            lo = max(0, row - ps);
            hi = row;
        }
    }
    const int whi_max = hd_wave_max(hi), whi_min = hd_wave_min(hi);
    const int wlo_min = hd_wave_min(hi < 0 ? 0x7fffffff : lo), wlo_max = hd_wave_max(lo);
    const int ntile = kv_lo < kv_end ? (kv_end - kv_lo + kHdBN - 1) / kHdBN : 0;

    // ---- Q^T operand: lane (row c32, half h) holds dims 16s + 8h .. + 7; a
    // negative scale flips Q's signs, so that the largest score is the largest
    // scaled one
    const float sl2 = p.scale * kLog2e, csc = fabsf(sl2);
    const uint32_t qflip = sl2 < 0.0f ? 0x80008000u : 0u;
    V8 qf[D / 16];
    {
        const uint16_t* qp = p.q + ((int64_t)min(row, T - 1) * p.Hq + hq) * D + 8 * h;
#pragma unroll
        for (int s = 0; s < D / 16; ++s) {
            const u32x4 x = *reinterpret_cast<const u32x4*>(qp + 16 * s);
            qf[s] = as_v8<V8>(u32x4{x[0] ^ qflip, x[1] ^ qflip, x[2] ^ qflip, x[3] ^ qflip});
        }
    }

    // ---- tile transfers: wave w fills 64 / W rows, 1 KB (2 or 8 rows) at a time; lane L's 16 bytes land at position L of that KB
    const int64_t row_stride = (int64_t)p.Hkv * ROW;  // bytes between keys
    const uint8_t* kg = reinterpret_cast<const uint8_t*>(p.k) + (int64_t)g * ROW;
    const uint8_t* vg = reinterpret_cast<const uint8_t*>(p.v) + (int64_t)g * ROW;
    int tr_row[NTR];
    uint32_t tr_col[NTR];
#pragma unroll
    for (int i = 0; i < NTR; ++i) {
        tr_row[i] = kHdBN / W * w + i * (1024 / ROW) + lane / (D / 8);
        tr_col[i] = 16u * (uint32_t)((lane % (D / 8)) ^ hd_tile_swz<D>(tr_row[i]));
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)&lds.tile[0][0][0]);
    auto load_tile = [&](int t, uint32_t slot) __attribute__((always_inline)) {
        const int k0 = kv_lo + t * kHdBN;
        const uint32_t dst = lds0 + slot * (2u * TILE) + 1024u * NTR * (uint32_t)w;
        const uint8_t* kb = kg + (int64_t)k0 * row_stride;
        const uint8_t* vb = vg + (int64_t)k0 * row_stride;
        const int last = kv_end - 1 - k0;  // keys past the range re-read the last one (masked)
#pragma unroll
        for (int i = 0; i < NTR; ++i) {
            const uint32_t off = (uint32_t)min(tr_row[i], last) * (uint32_t)row_stride + tr_col[i];
            dma16s(kb, off, dst + 1024u * i);
            dma16s(vb, off, dst + TILE + 1024u * i);
        }
    };

    // ---- operand reads.  K: row 32 kb + c32, chunk 2s + h.  V (transposing):
    // lane (e, x) of a 16-lane group addresses 8 bytes of row e of 4, and gets
    // one dim of the 4 rows: dims 32 m + c32, keys 16 c + 8 sec + 4 h + 0 .. 3
    // The chunk's bits above its lane part (2s of a K chunk, 4m of a V chunk)
    // enter by an exclusive or on the address, or as an offset past the swizzle
    const uint32_t k_lane = lds0 + (uint32_t)(c32 * ROW + 16 * (h ^ hd_tile_swz<D>(c32)));
    const int te = (lane >> 2) & 3, tx = lane & 3, cb = (lane >> 4) & 1;
    uint32_t v_lane[2];
#pragma unroll
    for (int sec = 0; sec < 2; ++sec) {
        const int r = 8 * sec + 4 * h + te;
        v_lane[sec] = lds0 + TILE + (uint32_t)(r * ROW + 8 * (tx & 1) + 16 * ((2 * cb + (tx >> 1)) ^ hd_tile_swz<D>(r)));
    }
    auto lds128 = [](uint32_t a) __attribute__((always_inline)) {
        return *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>((uintptr_t)a);
    };
    auto lds_tr = [](uint32_t a) __attribute__((always_inline)) {
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                             (__attribute__((address_space(3))) s16x4*)(uintptr_t)a));
    };

    f32x16 o[D / 32];
#pragma unroll
    for (int m = 0; m < D / 32; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[m][i] = 0.0f;
    // reference max (log2 units): moves only when a score passes it by more than 8
    float m_run = -__builtin_inff(), m_thr = -__builtin_inff(), l_part = 0.0f;

    auto process = [&](int t, uint32_t slot) __attribute__((always_inline)) {
        const int kt = kv_lo + t * kHdBN;
        const uint32_t k_slot = k_lane + slot * (2u * TILE);
        const uint32_t v_slot[2] = {v_lane[0] + slot * (2u * TILE), v_lane[1] + slot * (2u * TILE)};
#pragma unroll
        for (int r = 0; r < 2 / HB; ++r) {
            const int k0 = kt + 32 * HB * r;
            // after this wave's last key, or before its first
            if (k0 > whi_max || k0 + 32 * HB - 1 < wlo_min) continue;
            const bool need_mask = k0 + 32 * HB - 1 > whi_min || k0 < wlo_max;
            f32x16 sacc[HB];
#pragma unroll
            for (int b = 0; b < HB; ++b)
#pragma unroll
                for (int i = 0; i < 16; ++i) sacc[b][i] = 0.0f;
            // K operands are read two steps ahead of their products, V operands
            // one.  Fixed by scheduling barriers: left alone, the compiler
            // issues each read right before the product that waits for it (593
            // against 565 us on the 4 prompts named above, with the store).
            u32x4 ka[KA + 1][HB];
            auto read_k = [&](int s) __attribute__((always_inline)) {
#pragma unroll
                for (int b = 0; b < HB; ++b)
                    ka[s % (KA + 1)][b] = lds128((k_slot ^ (uint32_t)(32 * (s & 7))) +
                                          (uint32_t)((HB * r + b) * 32 * ROW + 256 * (s >> 3)));
            };
#pragma unroll
            for (int s = 0; s < KA; ++s) read_k(s);
#pragma unroll
            for (int s = 0; s < D / 16; ++s) {
                if (s + KA < D / 16) read_k(s + KA);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < HB; ++b) sacc[b] = M::mma(as_v8<V8>(ka[s % (KA + 1)][b]), qf[s], sacc[b]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (need_mask) {
#pragma unroll
                for (int b = 0; b < HB; ++b)
#pragma unroll
                    for (int j = 0; j < 16; ++j) {
                        const int kv = k0 + 32 * b + 8 * (j >> 2) + 4 * h + (j & 3);
                        sacc[b][j] = kv <= hi && kv >= lo ? sacc[b][j] : -__builtin_inff();
                    }
            }
            float mloc = sacc[0][0];
#pragma unroll
            for (int b = 0; b < HB; ++b)
#pragma unroll
                for (int j = 0; j < 16; ++j) mloc = fmaxf(mloc, sacc[b][j]);
            if (__ballot(mloc * csc > m_thr)) {  // rare after the first tiles
                const float mrow = fmaxf(mloc, shfl_xor(mloc, 32)) * csc;
                const bool upd = mrow > m_thr;  // the same in both halves of the row
                const float alpha = upd ? __builtin_amdgcn_exp2f(m_run - mrow) : 1.0f;  // 0 from -inf
                m_run = upd ? mrow : m_run;
                m_thr = m_run + 8.0f;
                l_part *= alpha;
#pragma unroll
                for (int m = 0; m < D / 32; ++m)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[m][i] *= alpha;
            }
            const float ref = m_run == -__builtin_inff() ? 0.0f : m_run - kOff;
            u32x4 pt[NTERM][2 * HB];  // [term][16-key chunk]
            float sum = 0.0f;
#pragma unroll
            for (int c = 0; c < 2 * HB; ++c)
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const int j = 4 * (2 * (c & 1) + (e >> 2)) + (e & 3);
                    float x0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[c >> 1][j], csc, -ref));
                    float x1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[c >> 1][j + 1], csc, -ref));
                    sum += x0 + x1;
                    uint32_t x[NTERM];
                    WeightTerms<BF>::split(x0, x1, x);
#pragma unroll
                    for (int u = 0; u < NTERM; ++u) pt[u][c][e >> 1] = x[u];
                }
            l_part += sum;
            // O^T += V^T P^T, V operands (two transposing reads each) one ahead
            u32x2 va[VA + 1][2];
            auto read_v = [&](int i) __attribute__((always_inline)) {
                const int c = i / (D / 32), m = i % (D / 32);
                const int vo = (2 * HB * r + c) * 16 * ROW + 256 * (m >> 2);
#pragma unroll
                for (int sec = 0; sec < 2; ++sec)
                    va[i % (VA + 1)][sec] = lds_tr((v_slot[sec] ^ (uint32_t)(64 * (m & 3))) + (uint32_t)vo);
            };
            constexpr int NV = 2 * HB * (D / 32);
#pragma unroll
            for (int i = 0; i < VA; ++i) read_v(i);
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                if (i + VA < NV) read_v(i + VA);
                __builtin_amdgcn_sched_barrier(0);
                const int c = i / (D / 32), m = i % (D / 32);
                const u32x2* vi = va[i % (VA + 1)];
                const V8 x = as_v8<V8>(u32x4{vi[0][0], vi[0][1], vi[1][0], vi[1][1]});
#pragma unroll
                for (int u = 0; u < NTERM; ++u) o[m] = M::mma(x, as_v8<V8>(pt[u][c]), o[m]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    // ---- tile t in slot t % NS; the next NS - 1 tiles in flight while it runs.
    // The barrier makes tile t visible and shows slot (t - 1) % NS free, which
    // then receives tile t + NS - 1 (2 NTR transfers a tile; vmcnt retires
    // loads in order)
    if (ntile > 0) load_tile(0, 0);
    if (NS == 3 && ntile > 1) load_tile(1, 1);
    uint32_t slot = 0, fill = NS - 1;
    for (int t = 0; t < ntile; ++t) {
        if (NS == 3 && t + 1 < ntile) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NTR) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (t + NS - 1 < ntile) load_tile(t + NS - 1, fill);
        process(t, slot);
        slot = slot == NS - 1 ? 0 : slot + 1;
        fill = fill == NS - 1 ? 0 : fill + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- normalise and store: dims 32 m + 8 b + 4 h + i of this lane's row
    const float l = l_part + shfl_xor(l_part, 32);
    bool bad = !(l == l);
#pragma unroll
    for (int m = 0; m < D / 32; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) bad |= !(fabsf(o[m][i]) < __builtin_inff());
    uint64_t badb = __ballot(bad && row_ok);
    badb = (badb | (badb >> 32)) & 0xffffffffull;  // a row is the lane and its partner
    if (row_ok && !((badb >> c32) & 1)) {
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        uint16_t* op = p.out + ((int64_t)row * p.Hq + hq) * D + 4 * h;
#pragma unroll
        for (int m = 0; m < D / 32; ++m)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                uint32_t x[2];
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    x[i] = (uint32_t)M::cvt(o[m][4 * b + 2 * i] * inv) |
                           ((uint32_t)M::cvt(o[m][4 * b + 2 * i + 1] * inv) << 16);
                *reinterpret_cast<u32x2*>(op + 32 * m + 8 * b) = u32x2{x[0], x[1]};
            }
    }
    while (badb) {
        const int c = (int)__builtin_ctzll(badb);
        badb &= badb - 1;
        const int r = wrow0 + c, n = min(p.pos[r], r) + 1;
        const int64_t kr = ((int64_t)(r - n + 1) * p.Hkv + g) * D, qr = ((int64_t)r * p.Hq + hq) * D;
        prefill_row_exact<D, BF>(p.out + qr, p.q + qr, p.k + kr, p.v + kr, p.Hkv * D, p.scale, n, lds.qs[w]);
    }
}

template <int W>
int launch_prefill_hd(const PrefillHdParams& prm, int D, bool bf, hipStream_t s) {
    const dim3 grid((unsigned)((int64_t)prm.ntiles * prm.Hkv * prm.hgroups)), block(64 * W);
    if (D == 64 && bf) hipLaunchKernelGGL((prefill_hd_kernel<64, true, W>), grid, block, 0, s, prm);
    else if (D == 64) hipLaunchKernelGGL((prefill_hd_kernel<64, false, W>), grid, block, 0, s, prm);
    else if (bf) hipLaunchKernelGGL((prefill_hd_kernel<256, true, W>), grid, block, 0, s, prm);
    else hipLaunchKernelGGL((prefill_hd_kernel<256, false, W>), grid, block, 0, s, prm);
    VMC_LAUNCH_CHECK();
    return VMC_OK;
}

PrefillHdParams hd_params(const GenArgs& a, int waves) {
    PrefillHdParams prm = {};
    prm.out = reinterpret_cast<uint16_t*>(a.out);
    prm.q = reinterpret_cast<const uint16_t*>(a.q);
    prm.k = a.k;
    prm.v = a.v;
    prm.pos = a.pos;
    prm.T = a.rows;
    prm.Hq = a.Hq;
    prm.Hkv = a.Hkv;
    prm.G = a.Hq / a.Hkv;
    prm.scale = a.scale;
    // heads per workgroup: 4, 2 or 1, dividing G; 32-row blocks per head fill the waves
    prm.hw = prm.G % 4 == 0 ? 4 : (prm.G % 2 == 0 ? 2 : 1);
    prm.rb = waves / prm.hw;
    prm.qb = 32 * prm.rb;
    prm.hgroups = prm.G / prm.hw;
    prm.ntiles = (a.rows - 1) / prm.qb + 1;
    return prm;
}

}  // namespace

bool prefill_hd_takes(const GenArgs& a) {
    if (a.src != GEN_LOCAL || (a.D != 64 && a.D != 256) || a.rows <= hd_min_rows(a.D) || a.rows > 0x7fffffff - 1024)
        return false;
    const PrefillHdParams prm = hd_params(a, 8);
    return (int64_t)prm.ntiles * prm.Hkv * prm.hgroups <= 0x7fffffff &&
           (int64_t)kHdBN * a.Hkv * 2 * a.D <= 0x7fffffff &&  // a tile's 32-bit offsets
           (((uintptr_t)a.q | (uintptr_t)a.out | (uintptr_t)a.k | (uintptr_t)a.v) & 15) == 0;
}

int prefill_hd(const GenArgs& a, hipStream_t s) {
    // Four waves while their workgroups fit the CUs, one each at head_dim 256
    // (128 KB of tiles) and four at 64: shorter blocks see fewer tiles of their
    // neighbours' keys, and half as many waves load, multiply and store on a CU.
    // bf16, us for eight waves / four: 256, 16/2 heads, 8 prompts of 20 tokens 20.0
    // / 14.8, one of 1000 90.5 / 76.6 (past the line: 8 of 500 62 / 86); 64, 32/8,
    // 8 of 20 10.0 / 6.4, one of 4096 197 / 170 (past the line: one of 8000 555 /
    // 575).
    const PrefillHdParams half = hd_params(a, 4);
    if ((int64_t)half.ntiles * half.Hkv * half.hgroups <= (int64_t)num_cus() * (a.D == 64 ? 4 : 1))
        return launch_prefill_hd<4>(half, a.D, a.q_bf16 != 0, s);
    return launch_prefill_hd<8>(hd_params(a, 8), a.D, a.q_bf16 != 0, s);
}

}  // namespace vmc
