// prefill.hip -- entry points of the causal flash-attention prefill
// (prefill_kernel.hpp), and the V^T tiles its local form may prebuild.
#include "device_cus.hpp"
#include "generic_attn.hpp"
#include "prefill_api.hpp"
#include "prefill_hd.hpp"
#include "prefill_kernel.hpp"

namespace vmc {

int launch_prefill_whole(PrefillParams& prm, bool bf16, int fmt, int src, bool vt, hipStream_t s) {
    return launch_prefill_any<1>(prm, bf16, fmt, src, vt, s);
}

namespace {

// ---- V^T tiles of the local prefill, built once per (64-key tile, KV head)
// rather than by every workgroup that reads the tile.  Tile tau of head g is
// the byte image of prefill_kernel's LDS V^T tile: fp16 V[64 tau + 16c + 8a
// + 4h + e][d] at byte d * 128 + 16 * ((2c + h) ^ ((d >> 1) & 7)) + 8a + 2e
// (keys past the step: zero).  flag[g][tau] = 1 when some row of the tile
// holds |v| >= 65536 or a NaN, or a value below 2^-17 and none of 2^-8 or more
// (per row: every case the kernel's own pass flags for its rows' groups is
// flagged).
__global__ void __launch_bounds__(256) vt_prep_kernel(const uint16_t* __restrict__ v, uint8_t* __restrict__ vt,
                                                      uint8_t* __restrict__ flag, int T, int Hkv, int ntT) {
    // rows padded to 65 dwords: the 8 lanes that gather one dim from 8 rows
    // of the tile hit 8 banks in pairs, not one bank
    __shared__ alignas(16) uint16_t tl[BN][kD + 2];
    const int tau = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
    bool fl = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = tid + 256 * i;
        const int r = c >> 4, cc = c & 15;  // row of the tile, 16-byte chunk of the row
        const int k = BN * tau + r;
        u32x4 w = {0u, 0u, 0u, 0u};
        if (k < T) w = *reinterpret_cast<const u32x4*>(v + ((int64_t)k * Hkv + g) * kD + 8 * cc);
        uint32_t mx = 0, mn1 = 0xffffu;
        u16x2 amax = {0, 0}, amin1 = {0xffff, 0xffff};  // |bits|, |bits| - 1 (0 wraps)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const u16x2 a = __builtin_bit_cast(u16x2, w[e] & 0x7fff7fffu);
            amax = __builtin_elementwise_max(amax, a);
            amin1 = __builtin_elementwise_min(amin1, a - u16x2{1, 1});
            const f16x2 hh = {(_Float16)__builtin_bit_cast(float, w[e] << 16),
                              (_Float16)__builtin_bit_cast(float, w[e] & 0xffff0000u)};
            w[e] = __builtin_bit_cast(uint32_t, hh);
        }
        mx = max((uint32_t)amax[0], (uint32_t)amax[1]);
        mn1 = min((uint32_t)amin1[0], (uint32_t)amin1[1]);
        // a row's 16 chunks sit in lanes 16j .. 16j + 15
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) {
            mx = max(mx, (uint32_t)__shfl_xor((int)mx, m, kWave));
            mn1 = min(mn1, (uint32_t)__shfl_xor((int)mn1, m, kWave));
        }
        // bf16 bit patterns: 0x477f = 65280 (largest below 2^16), 0x3700 =
        // 2^-17, 0x3b80 = 2^-8
        fl |= mx > 0x477fu || (mn1 < 0x36ffu && mx < 0x3b80u);
#pragma unroll
        for (int e = 0; e < 4; ++e) *reinterpret_cast<uint32_t*>(&tl[r][8 * cc + 2 * e]) = w[e];
    }
    const int any = __syncthreads_or(fl ? 1 : 0);
    if (tid == 0) flag[(int64_t)g * ntT + tau] = any ? 1 : 0;
    // the tile's 16 KB as 1024 chunks, chunk q = tid + 256 i (consecutive
    // lanes, consecutive bytes): dim row d = q >> 3 at position q & 7, which
    // holds logical chunk ci = (q & 7) ^ ((d >> 1) & 7)
    uint8_t* out = vt + (((int64_t)g * ntT + tau) << 14);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int q = tid + 256 * i, d = q >> 3;
        const int ci = (q & 7) ^ ((d >> 1) & 7), c = ci >> 1, h = ci & 1;
        uint32_t x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = tl[16 * c + 8 * (u >> 2) + 4 * h + (u & 3)][d];
        const u32x4 o = {x[0] | (x[1] << 16), x[2] | (x[3] << 16), x[4] | (x[5] << 16), x[6] | (x[7] << 16)};
        *reinterpret_cast<u32x4*>(out + 16 * q) = o;
    }
}

// workspace of the local prefill's prebuilt V^T tiles: 16 KB per (64-key
// tile, KV head), then one flag byte each
size_t vt_workspace_bytes(int64_t num_tokens, int64_t num_kv_heads) {
    const int64_t n = (num_tokens + BN - 1) / BN * num_kv_heads;
    return (size_t)(n * (kD * BN * 2) + ((n + 255) & ~(int64_t)255));
}

// workgroup shape shared by the local and paged entry points; whole_alone: see
// the rule at the end
void set_tiling(PrefillParams& prm, int num_tokens, int num_heads, int num_kv_heads, float scale, bool whole_alone) {
    prm.T = num_tokens;
    prm.Hq = num_heads;
    prm.Hkv = num_kv_heads;
    prm.G = num_heads / num_kv_heads;
    prm.scale_log2 = scale * kLog2e;
    // heads per workgroup: 4, 2 or 1, dividing G; 32-row blocks per head and
    // key parts fill 8 waves
    prm.hw = prm.G % 4 == 0 ? 4 : (prm.G % 2 == 0 ? 2 : 1);
    prm.hgroups = prm.G / prm.hw;
    auto shape = [&](int ks) {
        prm.ks = ks;
        prm.rb = NW / (prm.hw * ks);
        prm.qb = 32 * prm.rb;
        prm.ntiles = (int)(((int64_t)num_tokens + prm.qb - 1) / prm.qb);
        return (int64_t)prm.ntiles * prm.Hkv * prm.hgroups;
    };
    // Two waves share a tile's keys where that still gives one workgroup a CU
    // at most: twice the workgroups, each through a tile in about 0.7 of the
    // time (32/8 heads over a 4096-token prefix, us for one wave / two: q8_0
    // 64 tokens 148 / 112, 512 166 / 127, 1024 184 / 146; fp16 pages 512 142 /
    // 101; 3-bit slots 512 201 / 168; a 1024-token prompt 39 / 32).  Past
    // that the workgroups take turns and each tile is fetched twice as often
    // (q8_0 1536 tokens 205 / 252, 2048 245 / 281).
    // No more workgroups come of it where one block holds all rows, and with one
    // head a workgroup the four waves of 128 rows already sit on four SIMDs:
    // over this step's K/V and over slots with 4-bit values the second wave then
    // costs more than it brings (28/4 heads, us for one wave / two: a 64-token
    // prompt 6.1 / 7.0; 64 tokens over a 4096-token prefix, 4-bit slots 157 / 172,
    // 3/4-bit 153 / 168, k8v4 207 / 225; but 3-bit slots of 100 tokens 160 / 152,
    // q8_0 of 64 107 / 100, fp16 96 / 85).
    const int64_t split = shape(2);
    if (split > num_cus() || (whole_alone && prm.hw == 1 && prm.ntiles == 1)) shape(1);
}

int launch_tiled(PrefillParams& prm, bool bf16, int fmt, int src, bool vt, hipStream_t s) {
    return prm.ks == 2 ? launch_prefill_split(prm, bf16, fmt, src, vt, s)
                       : launch_prefill_whole(prm, bf16, fmt, src, vt, s);
}

}  // namespace

int tq_prefill_tiled(void* out, const void* query, const void* kv_cache, const int32_t* block_tables,
                     const int32_t* token_to_seq, const int32_t* token_positions, int num_tokens, int num_heads,
                     int num_kv_heads, float scale, int64_t max_blocks, const vmc_tq_config* cfg, int half_dtype,
                     hipStream_t stream) {
    if (!tq_config_valid(cfg) || cfg->head_dim != kD || cfg->group_size != 0) return VMC_EINVAL;
    if (half_dtype != VMC_DTYPE_F16 && half_dtype != VMC_DTYPE_BF16) return VMC_EINVAL;
    if (num_tokens < 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads != 0 || max_blocks <= 0 ||
        max_blocks > 0x7fffffff)
        return VMC_EINVAL;
    if (num_tokens == 0) return VMC_OK;
    if (!out || !query || !kv_cache || !block_tables || !token_to_seq || !token_positions) return VMC_EINVAL;
    if (((uintptr_t)kv_cache & 3) != 0) return VMC_EINVAL;
    PrefillParams prm = {};
    prm.out = reinterpret_cast<uint16_t*>(out);
    prm.q = reinterpret_cast<const uint16_t*>(query);
    prm.pos = token_positions;
    set_tiling(prm, num_tokens, num_heads, num_kv_heads, scale, cfg->value_quant_bits == 4);
    prm.kp = prm.vp = reinterpret_cast<const uint8_t*>(kv_cache);
    prm.bt = block_tables;
    prm.tok_seq = token_to_seq;
    prm.max_blocks = max_blocks;
    prm.num_seqs = 0x7fffffff;  // the rows' sequences are the caller's to keep in the table
    prm.E = cfg->slot_size_aligned;
    prm.page_bytes = (int64_t)kBsP * num_kv_heads * prm.E;
    prm.hnd = 0;
    prm.q_bf16 = half_dtype == VMC_DTYPE_BF16;
    if (!cfg->key_fp8) {
        const TQTables& tab = tq_tables(kD, cfg->key_quant_bits);
        for (int i = 0; i < 16; ++i) prm.cent[i] = i < tab.n_centroids ? tab.centroids[i] : 0.0f;
        prm.sq_unit = tq_square_planes(prm.cent, cfg->key_quant_bits, prm.sq_plane);
        prm.rot_c = tab.rot_c;
    }
    prm.fp8_e4b15 = cfg->fp8_e4b15 ? 1 : 0;
    prm.mse_bytes = cfg->mse_bytes;
    prm.key_packed = cfg->key_packed_size;
    prm.val_data = cfg->val_data_bytes;
    prm.norm_corr = cfg->norm_correction != 0;
    if ((int64_t)prm.ntiles * prm.Hkv * prm.hgroups > 0x7fffffffLL) return VMC_EINVAL;
    const int kb = cfg->key_quant_bits, vb = cfg->value_quant_bits;
    if (cfg->key_fp8) return vb == 4 ? launch_tiled(prm, false, -1, SRC_K8, false, stream) : VMC_EINVAL;
    if (kb == 3 && vb == 3) return launch_tiled(prm, false, -1, SRC_TQ33, false, stream);
    if (kb == 4 && vb == 4) return launch_tiled(prm, false, -1, SRC_TQ44, false, stream);
    if (kb == 3 && vb == 4) return launch_tiled(prm, false, -1, SRC_TQ34, false, stream);
    return VMC_EINVAL;
}

}  // namespace vmc

using namespace vmc;

extern "C" int vmc_flash_attention_prefill_v2(void* output, const void* query, const void* key_cache,
                                              const void* value_cache, int num_tokens, int num_heads,
                                              int num_kv_heads, int head_dim, float scale, int block_size,
                                              int max_num_blocks_per_req, const int32_t* block_tables,
                                              const int32_t* seq_lens, const int32_t* token_to_seq,
                                              const int32_t* token_positions, int num_reqs, int q_dtype,
                                              int kv_format, int layout, vmc_stream_t stream) {
    (void)seq_lens;  // a token's keys are positions 0 .. token_positions[t]
    if (generic_head_dim(head_dim)) {
        // head_dim 64 / 256: one wave per (token, query head), any block size
        if (num_tokens < 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads != 0 ||
            block_size <= 0 || max_num_blocks_per_req <= 0 || num_reqs < 0)
            return VMC_EINVAL;
        if (q_dtype != VMC_DTYPE_F16 && q_dtype != VMC_DTYPE_BF16) return VMC_EINVAL;
        if (layout != VMC_LAYOUT_NHD && layout != VMC_LAYOUT_HND) return VMC_EINVAL;
        if (kv_format != VMC_KV_F16 && kv_format != VMC_KV_BF16 && kv_format != VMC_KV_Q8_0 &&
            kv_format != VMC_KV_Q4_0)
            return VMC_EINVAL;
        if (num_tokens == 0 || num_reqs == 0) return VMC_OK;
        if (!output || !query || !key_cache || !value_cache || !block_tables || !token_to_seq ||
            !token_positions)
            return VMC_EINVAL;
        GenArgs a = {};
        a.out = output;
        a.q = query;
        a.q_bf16 = q_dtype == VMC_DTYPE_BF16;
        a.src = kv_format == VMC_KV_F16 ? GEN_F16 : kv_format == VMC_KV_BF16 ? GEN_BF16
              : kv_format == VMC_KV_Q8_0 ? GEN_Q8 : GEN_Q4;
        a.kp = reinterpret_cast<const uint8_t*>(key_cache);
        a.vp = reinterpret_cast<const uint8_t*>(value_cache);
        a.entry = vmc_kv_entry_bytes(kv_format, head_dim);
        a.hnd = layout == VMC_LAYOUT_HND;
        a.bs = block_size;
        a.bt = block_tables;
        a.max_blocks = max_num_blocks_per_req;
        a.tok_seq = token_to_seq;
        a.pos = token_positions;
        a.num_seqs = num_reqs;
        a.rows = num_tokens;
        a.Hq = num_heads;
        a.Hkv = num_kv_heads;
        a.D = head_dim;
        a.scale = scale;
        return gen_attention(a, reinterpret_cast<hipStream_t>(stream));
    }
    if (head_dim != kD || block_size != kBsP || num_tokens < 0 || num_heads <= 0 || num_kv_heads <= 0 ||
        num_heads % num_kv_heads != 0 || max_num_blocks_per_req <= 0 || num_reqs < 0)
        return VMC_EINVAL;
    if (q_dtype != VMC_DTYPE_F16 && q_dtype != VMC_DTYPE_BF16) return VMC_EINVAL;
    if (layout != VMC_LAYOUT_NHD && layout != VMC_LAYOUT_HND) return VMC_EINVAL;
    if (kv_format != VMC_KV_F16 && kv_format != VMC_KV_BF16 && kv_format != VMC_KV_Q8_0 &&
        kv_format != VMC_KV_Q4_0)
        return VMC_EINVAL;
    if (num_tokens == 0 || num_reqs == 0) return VMC_OK;
    if (!output || !query || !key_cache || !value_cache || !block_tables || !token_to_seq ||
        !token_positions)
        return VMC_EINVAL;
    // pages are read in 16-byte (f16 / bf16) and 4-byte (q8_0 / q4_0) units
    if ((((uintptr_t)key_cache | (uintptr_t)value_cache) & 15) != 0) return VMC_EINVAL;
    PrefillParams prm = {};
    prm.out = reinterpret_cast<uint16_t*>(output);
    prm.q = reinterpret_cast<const uint16_t*>(query);
    prm.pos = token_positions;
    set_tiling(prm, num_tokens, num_heads, num_kv_heads, scale, false);
    prm.kp = reinterpret_cast<const uint8_t*>(key_cache);
    prm.vp = reinterpret_cast<const uint8_t*>(value_cache);
    prm.bt = block_tables;
    prm.tok_seq = token_to_seq;
    prm.max_blocks = max_num_blocks_per_req;
    prm.num_seqs = num_reqs;
    prm.E = vmc_kv_entry_bytes(kv_format, head_dim);
    prm.page_bytes = (int64_t)kBsP * num_kv_heads * prm.E;
    prm.hnd = layout == VMC_LAYOUT_HND;
    prm.q_bf16 = q_dtype == VMC_DTYPE_BF16;
    if ((int64_t)prm.ntiles * prm.Hkv * prm.hgroups > 0x7fffffffLL) return VMC_EINVAL;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (kv_format) {
        case VMC_KV_F16: return launch_tiled(prm, false, -1, SRC_PAGED, false, s);
        case VMC_KV_BF16: return launch_tiled(prm, true, -1, SRC_PAGED, false, s);
        case VMC_KV_Q8_0: return launch_tiled(prm, false, -1, SRC_Q8, false, s);
        default: return launch_tiled(prm, false, -1, SRC_Q4, false, s);
    }
}

namespace {
// the local prefill; with a workspace (ws != NULL) the V^T tiles of a bf16 step
// are built once by vt_prep_kernel and the attention kernel fetches them.  In
// fp16 a workgroup's own transpose needs no conversion and no range check and
// costs less than the extra launch saves, 32/8 heads, us prebuilt / own: 64
// tokens 13.8 / 9.6, 512 tokens 20.9 / 18.1, 1024 tokens 31.3 / 28.1, 4096
// tokens 157 / 154, 2 x 4096 tokens 301 / 297 (64/8 heads 571 / 576; bf16, 2 x
// 4096 tokens: 296 / 319)
int local_prefill(void* output, const void* query, const void* key, const void* value, int num_tokens,
                  int num_heads, int num_kv_heads, int head_dim, float scale, const int32_t* token_positions,
                  int dtype, void* key_cache, void* value_cache, const int64_t* slot_mapping, int64_t block_size,
                  int kv_format, int layout, void* ws, size_t ws_bytes, vmc_stream_t stream) {
    if (generic_head_dim(head_dim)) {
        // head_dim 64 / 256: the append by vmc_reshape_and_cache, then
        // prefill_hd.hip, or for operands it does not take one wave per
        // (token, query head) over this step's K/V
        if (num_tokens < 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads != 0)
            return VMC_EINVAL;
        if (dtype != VMC_DTYPE_F16 && dtype != VMC_DTYPE_BF16) return VMC_EINVAL;
        if (num_tokens == 0) return VMC_OK;
        if (!output || !query || !key || !value || !token_positions) return VMC_EINVAL;
        if (key_cache) {
            const int64_t E = vmc_kv_entry_bytes(kv_format, head_dim);
            if (E < 0 || block_size <= 0) return VMC_EINVAL;
            const int rc = vmc_reshape_and_cache(key, value, key_cache, value_cache, slot_mapping, num_tokens,
                                                 num_kv_heads, head_dim, block_size,
                                                 block_size * num_kv_heads * E, kv_format, dtype, layout,
                                                 stream);
            if (rc != VMC_OK) return rc;
        }
        GenArgs a = {};
        a.out = output;
        a.q = query;
        a.q_bf16 = dtype == VMC_DTYPE_BF16;
        a.src = GEN_LOCAL;
        a.k = reinterpret_cast<const uint16_t*>(key);
        a.v = reinterpret_cast<const uint16_t*>(value);
        a.pos = token_positions;
        a.num_seqs = -1;
        a.rows = num_tokens;
        a.Hq = num_heads;
        a.Hkv = num_kv_heads;
        a.D = head_dim;
        a.scale = scale;
        if (prefill_hd_takes(a)) return prefill_hd(a, reinterpret_cast<hipStream_t>(stream));
        return gen_attention(a, reinterpret_cast<hipStream_t>(stream));
    }
    if (head_dim != kD || num_tokens < 0 || num_heads <= 0 || num_kv_heads <= 0 ||
        num_heads % num_kv_heads != 0)
        return VMC_EINVAL;
    if (dtype != VMC_DTYPE_F16 && dtype != VMC_DTYPE_BF16) return VMC_EINVAL;
    if (num_tokens == 0) return VMC_OK;
    if (!output || !query || !key || !value || !token_positions) return VMC_EINVAL;
    PrefillParams prm = {};
    prm.out = reinterpret_cast<uint16_t*>(output);
    prm.q = reinterpret_cast<const uint16_t*>(query);
    prm.k = reinterpret_cast<const uint16_t*>(key);
    prm.v = reinterpret_cast<const uint16_t*>(value);
    prm.pos = token_positions;
    set_tiling(prm, num_tokens, num_heads, num_kv_heads, scale, true);
    int fmt = -1;
    if (key_cache) {
        const int64_t E = vmc_kv_entry_bytes(kv_format, head_dim);
        if (E < 0 || !value_cache || !slot_mapping || block_size <= 0) return VMC_EINVAL;
        if (layout != VMC_LAYOUT_NHD && layout != VMC_LAYOUT_HND) return VMC_EINVAL;
        prm.kc = reinterpret_cast<uint8_t*>(key_cache);
        prm.vc = reinterpret_cast<uint8_t*>(value_cache);
        prm.slots = slot_mapping;
        prm.bs = block_size;
        prm.E = E;
        prm.stride = block_size * num_kv_heads * E;
        prm.hnd = layout == VMC_LAYOUT_HND;
        fmt = kv_format;
    }
    if ((int64_t)prm.ntiles * prm.Hkv * prm.hgroups > 0x7fffffffLL) return VMC_EINVAL;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const bool bf = dtype == VMC_DTYPE_BF16;
    if (ws) {
        if (ws_bytes < vt_workspace_bytes(num_tokens, num_kv_heads)) return VMC_ENOMEM;
        if (((uintptr_t)ws & 15) != 0) return VMC_EINVAL;
    }
    if (!ws || !bf) return launch_tiled(prm, bf, fmt, SRC_LOCAL, false, s);
    const int ntT = (num_tokens + BN - 1) / BN;
    prm.vt = reinterpret_cast<const uint8_t*>(ws);
    prm.vt_flag = prm.vt + (int64_t)ntT * num_kv_heads * (kD * BN * 2);
    prm.vt_tiles = ntT;
    uint8_t* vt = reinterpret_cast<uint8_t*>(ws);
    uint8_t* flag = vt + (int64_t)ntT * num_kv_heads * (kD * BN * 2);
    const dim3 vgrid((unsigned)ntT, (unsigned)num_kv_heads);
    hipLaunchKernelGGL(vt_prep_kernel, vgrid, dim3(256), 0, s, prm.v, vt, flag, num_tokens, num_kv_heads, ntT);
    VMC_LAUNCH_CHECK();
    return launch_tiled(prm, true, fmt, SRC_LOCAL, true, s);
}
}  // namespace

extern "C" int vmc_flash_attention_prefill(void* output, const void* query, const void* key,
                                           const void* value, int num_tokens, int num_heads,
                                           int num_kv_heads, int head_dim, float scale,
                                           const int32_t* token_positions, int dtype,
                                           void* key_cache, void* value_cache,
                                           const int64_t* slot_mapping, int64_t block_size,
                                           int kv_format, int layout, vmc_stream_t stream) {
    return local_prefill(output, query, key, value, num_tokens, num_heads, num_kv_heads, head_dim, scale,
                         token_positions, dtype, key_cache, value_cache, slot_mapping, block_size, kv_format,
                         layout, nullptr, 0, stream);
}

extern "C" size_t vmc_flash_attention_prefill_workspace_size(int num_tokens, int num_kv_heads, int head_dim) {
    if (head_dim != kD || num_tokens <= 0 || num_kv_heads <= 0) return 0;
    return vt_workspace_bytes(num_tokens, num_kv_heads);
}

extern "C" int vmc_flash_attention_prefill_ws(void* output, const void* query, const void* key,
                                              const void* value, int num_tokens, int num_heads,
                                              int num_kv_heads, int head_dim, float scale,
                                              const int32_t* token_positions, int dtype, void* key_cache,
                                              void* value_cache, const int64_t* slot_mapping,
                                              int64_t block_size, int kv_format, int layout,
                                              void* workspace, size_t workspace_bytes, vmc_stream_t stream) {
    // head_dim 64 / 256 take no workspace (their kernel has no tiles)
    if (head_dim == kD && num_tokens > 0 && !workspace) return VMC_EINVAL;
    return local_prefill(output, query, key, value, num_tokens, num_heads, num_kv_heads, head_dim, scale,
                         token_positions, dtype, key_cache, value_cache, slot_mapping, block_size, kv_format,
                         layout, head_dim == kD ? workspace : nullptr, workspace_bytes, stream);
}
