// paged_decode_hd.hip -- split-KV paged decode on MFMA for head_dim 64 and 256:
// f16 / bf16 pages read with q of the same type, q8_0 / q4_0 pages with
// either; block size 16, at most 16 query heads per KV head, any number of KV
// heads.  The semantics and the arithmetic's precision are gen_attn_kernel's
// (generic_attn.hip), which keeps the shapes outside these limits.
//
// What bounds it: HBM.  The one-wave-per-row kernel read every page once per
// query head, one wave per row (4.06 ms for 32 sequences of 256 .. 8192
// tokens, 32/8 heads, head_dim 64, bf16: 43 GB/s; this kernel and its merge
// 47 us, 3.7 TB/s); here
//  * a wave is one (page range, KV head) unit: all G query heads share each
//    page it reads, and the ranges (decode_plan.hpp) cut long sequences, so
//    that a CU holds 12 (head_dim 64) or 8 units whatever the batch, as far as
//    the workspace has room for their partial rows (paged_decode_hd; the size
//    query is by rows of 128 dims: at head_dim 256, 16/2 heads, 519 of the 1024
//    ranges; 8/4 heads 259 of 512);
//  * waves share nothing and meet no barrier: each finds its sequences by a
//    scan of seq_lens, keeps 64 block-table entries in its lanes, and holds
//    the next step's pages (32 tokens at head_dim 64, 16 at 256: 8 or 16 KB)
//    in registers while this step runs from its own LDS tile, so one wave's
//    loads overlap the others' arithmetic.
// S^T = K . Q^T and O^T = V^T . P^T, so a query head stays one lane column
// throughout: the running max, the rescale and the final division need no
// exchange between lanes but the max over the column's four lane groups.  V^T
// operands come from the row-major tile by transposing LDS reads.  Tile rows
// keep 16-byte chunk ch of row r at ch ^ f(r): conflict-free for the 16-row
// K reads (f is a bijection on the rows that share banks) and for the
// transposing reads of 8 rows x 32 bytes.
//
// Weights keep their 24 bits: P enters the products as a sum of three 16-bit
// terms (weight_terms.hpp), fp16 against fp16 V (the largest weight scaled to
// 2^15: whole down to 2^-16, off by at most 2^-40 below), bf16 otherwise.  q8_0 / q4_0
// codes are integers of at most 8 bits, exact in either type; a block's scale
// multiplies its partial score (K) or the weights (V) in fp32.
#include "decode_plan.hpp"
#include "generic_row.hpp"
#include "paged_decode_hd.hpp"
#include "weight_terms.hpp"

namespace vmc {
namespace {

// the MFMA operand type and products of one 16-bit type
template <bool BF>
struct HdT {
    using v8 = f16x8;
    static __device__ __forceinline__ f32x4 mma32(u32x4 a, u32x4 b, f32x4 c) {
        return mfma16x16x32(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c);
    }
    static __device__ __forceinline__ f32x4 mma16(u32x2 a, u32x2 b, f32x4 c) {
        return mfma16x16x16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c);
    }
};
template <>
struct HdT<true> {
    using v8 = bf16x8;
    static __device__ __forceinline__ f32x4 mma32(u32x4 a, u32x4 b, f32x4 c) {
        return mfma16x16x32(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c);
    }
    static __device__ __forceinline__ f32x4 mma16(u32x2 a, u32x2 b, f32x4 c) {
        return mfma16x16x16(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c);
    }
};

template <bool BF>
__device__ __forceinline__ uint32_t pack_half2(float a, float b) {
    return (uint32_t)f32_to_half<BF>(a) | ((uint32_t)f32_to_half<BF>(b) << 16);
}

template <int D, int FMT>
struct HdGeo {
    static constexpr bool gguf = FMT == FMT_Q8_0 || FMT == FMT_Q4_0;
    static constexpr int waves = D == 64 ? 4 : 2;  // per workgroup
    static constexpr int pg = D == 64 ? 2 : 1;     // pages per step
    static constexpr int tok = 16 * pg;
    static constexpr int row = 2 * D;              // bytes of a tile row
    static constexpr int tile = tok * row;
    static constexpr int nblk = D / 32;
    static constexpr int be = FMT == FMT_Q8_0 ? 34 : 18;  // GGUF block bytes
    static constexpr int nw = FMT == FMT_Q8_0 ? 9 : 5;    // dwords from a block's 4-byte floor
    static constexpr int nld = gguf ? tok * nblk / 64 : tok * row / 1024;  // blocks / chunks per lane and tensor
    static constexpr int scales = gguf ? 2 * pg * nblk * 16 : 0;           // floats: K then V, [page][block][token]
};

// chunk swizzle of a tile row (see the top): 16 chunk positions in one
// 256-byte bank cycle at head_dim 256, two rows of 8 at 64
template <int D>
__device__ __forceinline__ int hd_swz(int r) {
    return D == 256 ? (((r & 7) << 1) | ((r >> 3) & 1)) : ((((r >> 1) & 3) << 1) | ((r >> 3) & 1));
}

// One query head over keys k0 .. k1 - 1 by gen_row, into its output row or its
// partial row.  A call, not inlined: its registers stay out of the page loop's.
template <int D, int FMT, bool QBF>
__device__ __noinline__ void hd_row_exact(const uint16_t* q, const uint8_t* kc, const uint8_t* vc, const int32_t* bt,
                                          int64_t page_bytes, uint32_t entry, uint32_t row0, uint32_t row_step,
                                          float scale, int k0, int k1, float* qs, uint16_t* out, float* part) {
    constexpr int SRC = FMT == FMT_F16 ? GEN_F16 : FMT == FMT_BF16 ? GEN_BF16 : FMT == FMT_Q8_0 ? GEN_Q8 : GEN_Q4;
    const int lane = threadIdx.x & 63;
    GenArgs a = {};
    a.scale = scale;
    const TQTables none = {};
    wave_sync();
#pragma unroll
    for (int i = 0; i < D / 64; ++i) qs[lane + 64 * i] = half_to_f32<QBF>(q[lane + 64 * i]);
    wave_sync();
    auto key_at = [&](int k, const uint8_t*& ke, const uint8_t*& ve) __attribute__((always_inline)) {
        const int32_t id = bt[k >> 4];
        const int64_t off = (int64_t)id * page_bytes + (int64_t)(row0 + (uint32_t)(k & 15) * row_step) * entry;
        ke = kc + off;
        ve = vc + off;
        return id >= 0;
    };
    float m, l, acc[D / 64];
    gen_row<D, SRC, 0, 0, QBF>(a, none, qs, lane, k0, k1, key_at, m, l, acc);
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int i = 0; i < D / 64; ++i) {
        if (out) out[lane + 64 * i] = f32_to_half<QBF>(acc[i] * inv);
        else part[lane + 64 * i] = acc[i];
    }
    if (!out && lane == 0) *reinterpret_cast<float2*>(part + D) = make_float2(m * kLog2e, l);
    wave_sync();
}

template <int D, int FMT, bool QBF>
__global__ void __launch_bounds__((D == 64 ? 256 : 128), (D == 64 ? 3 : 2)) paged_decode_hd_kernel(DecodeParams p) {
    using GE = HdGeo<D, FMT>;
    constexpr int PG = GE::pg, TOK = GE::tok, NT = D / 16, NP = 4 * PG;
    constexpr bool kGguf = GE::gguf;
    constexpr bool VBF = kGguf || FMT == FMT_BF16;  // type of the V operand and the weights' terms
    constexpr int kTerms = WeightTerms<VBF>::n;
    constexpr float kOff = VBF ? 0.0f : 15.0f;  // weights are 2^(s - m + kOff)
    struct WaveLds {
        uint8_t k[GE::tile], v[GE::tile];
        float sc[kGguf ? GE::scales : 4];
    };
    __shared__ __attribute__((aligned(16))) WaveLds lds_all[GE::waves];
    WaveLds& lds = lds_all[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63, r16 = lane & 15, grp = lane >> 4;
    const int unit = __builtin_amdgcn_readfirstlane(blockIdx.x * GE::waves + (threadIdx.x >> 6));
    const int w = unit / p.Hkv, g = unit % p.Hkv;
    if (w >= p.grid) return;

    // ---- loads of one step into registers, and from there into the tile
    uint32_t kraw[GE::nld][kGguf ? GE::nw : 4], vraw[GE::nld][kGguf ? GE::nw : 4];
    auto row_off = [&](int r) __attribute__((always_inline)) {  // row r & 15 of a page, this KV head
        return (uint32_t)(p.hnd ? g * kBs + (r & 15) : (r & 15) * p.Hkv + g) * (uint32_t)p.entry_bytes;
    };
    auto issue = [&](int pg0, int pg1) __attribute__((always_inline)) {
        const int64_t o0 = (int64_t)pg0 * p.page_bytes, o1 = (int64_t)pg1 * p.page_bytes;
#pragma unroll
        for (int i = 0; i < GE::nld; ++i) {
            if constexpr (kGguf) {
                // lane: block idx % nblk of row idx / nblk, from its 4-byte
                // floor (odd blocks start 2 bytes past one); the last dword
                // stays inside the entry
                const int idx = 64 * i + lane, r = idx / GE::nblk, blk = idx % GE::nblk;
                const int64_t off = (PG == 2 && r >= 16 ? o1 : o0) + row_off(r) + GE::be * blk - 2 * (blk & 1);
                const uint32_t* ks = reinterpret_cast<const uint32_t*>(p.kc + off);
                const uint32_t* vs = reinterpret_cast<const uint32_t*>(p.vc + off);
#pragma unroll
                for (int e = 0; e < GE::nw; ++e) {
                    kraw[i][e] = ks[e];
                    vraw[i][e] = vs[e];
                }
            } else {
                // lane: 16-byte chunk idx % (D / 8) of row idx / (D / 8); a
                // load covers rows of one page
                const int idx = 64 * i + lane, r = idx / (D / 8);
                const int64_t ob = PG == 2 && i >= GE::nld / 2 ? o1 : o0;
                const uint32_t off = row_off(r) + 16u * (uint32_t)(idx % (D / 8));
                const u32x4 kw = *reinterpret_cast<const u32x4*>(p.kc + ob + off);
                const u32x4 vw = *reinterpret_cast<const u32x4*>(p.vc + ob + off);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    kraw[i][e] = kw[e];
                    vraw[i][e] = vw[e];
                }
            }
        }
    };
    // nv0 / nv1: tokens of the step's pages that count; the V rows (GGUF: the
    // V scales) of the others become zero
    auto stage = [&](int nv0, int nv1) __attribute__((always_inline)) {
        const bool full = nv0 == 16 && (PG == 1 || nv1 == 16);
#pragma unroll
        for (int i = 0; i < GE::nld; ++i) {
            if constexpr (kGguf) {
                const int idx = 64 * i + lane, r = idx / GE::nblk, blk = idx % GE::nblk;
                const bool odd = (blk & 1) != 0;
                const bool ok = (r & 15) < (PG == 2 && r >= 16 ? nv1 : nv0);
                auto block = [&](const uint32_t (&raw)[GE::nw], uint8_t* tile, float* sc, bool live, auto bf_c)
                    __attribute__((always_inline)) {
                    constexpr bool BF = decltype(bf_c)::value;
                    constexpr int NC = GE::nw - 1;
                    uint32_t c[NC];
#pragma unroll
                    for (int e = 0; e < NC; ++e)
                        c[e] = odd ? raw[e + 1] : __builtin_amdgcn_alignbyte(raw[e + 1], raw[e], 2);
                    const float d = f16_bits_to_f32((uint16_t)(odd ? raw[0] >> 16 : raw[0] & 0xffffu));
                    sc[((r >> 4) * GE::nblk + blk) * 16 + (r & 15)] = live ? d : 0.0f;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {  // chunk j: values 8j .. 8j + 7
                        u32x4 x;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            float f[2];
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                const int q = 8 * j + 2 * e + u;
                                if constexpr (FMT == FMT_Q8_0)
                                    f[u] = (float)(int)(int8_t)(c[q >> 2] >> (8 * (q & 3)));
                                else  // byte i: value i | value i + 16 << 4
                                    f[u] = (float)((int)((c[(q & 15) >> 2] >> (8 * (q & 3) + (q >= 16 ? 4 : 0))) & 15u) - 8);
                            }
                            x[e] = pack_half2<BF>(f[0], f[1]);
                        }
                        *reinterpret_cast<u32x4*>(tile + r * GE::row + 16 * ((4 * blk + j) ^ hd_swz<D>(r & 15))) = x;
                    }
                };
                block(kraw[i], lds.k, lds.sc, true, std::integral_constant<bool, QBF>{});
                block(vraw[i], lds.v, lds.sc + GE::scales / 2, ok, std::integral_constant<bool, VBF>{});
            } else {
                const int idx = 64 * i + lane, r = idx / (D / 8);
                const int at = r * GE::row + 16 * ((idx % (D / 8)) ^ hd_swz<D>(r & 15));
                u32x4 vw = {vraw[i][0], vraw[i][1], vraw[i][2], vraw[i][3]};
                if (!full) {  // uniform
                    const bool ok = (r & 15) < (PG == 2 && i >= GE::nld / 2 ? nv1 : nv0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) vw[e] = ok ? vw[e] : 0u;
                }
                *reinterpret_cast<u32x4*>(lds.k + at) = u32x4{kraw[i][0], kraw[i][1], kraw[i][2], kraw[i][3]};
                *reinterpret_cast<u32x4*>(lds.v + at) = vw;
            }
        }
        wave_sync();
    };

    // ---- LDS operand addresses
    const int k_sw = hd_swz<D>(r16);
    const int te = (lane >> 2) & 3, tq = lane & 3, v_row = 4 * grp + te;  // transposing reads
    const int v_sw = hd_swz<D>(v_row);
    const uint32_t v_lds = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)lds.v +
                           (uint32_t)(v_row * GE::row + 8 * (tq & 1));
    auto v_tr = [&](int t, int pg) __attribute__((always_inline)) {  // dims 16t + r16, tokens 4 grp .. + 3 of page pg
        const uint32_t a = v_lds + (uint32_t)(16 * pg * GE::row + 16 * ((2 * t + (tq >> 1)) ^ v_sw));
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                             (__attribute__((address_space(3))) s16x4*)(uintptr_t)a));
    };

    u32x4 qf[D / 32];
    f32x4 o[NT];
    float m_run, l_part;
    const float csc = p.scale_log2;

    auto compute = [&](int nv0, int nv1) __attribute__((always_inline)) {
        // ---- S^T: tokens 4 grp + i of page pg, head r16
        float s[NP];
#pragma unroll
        for (int pg = 0; pg < PG; ++pg) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < D / 32; ++st) {
                const u32x4 a = *reinterpret_cast<const u32x4*>(lds.k + (16 * pg + r16) * GE::row +
                                                                16 * ((4 * st + grp) ^ k_sw));
                if constexpr (kGguf) {
                    const f32x4 part = HdT<QBF>::mma32(a, qf[st], f32x4{0.f, 0.f, 0.f, 0.f});
                    const f32x4 d = *reinterpret_cast<const f32x4*>(lds.sc + (pg * GE::nblk + st) * 16 + 4 * grp);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(d[i], part[i], acc[i]);
                } else {
                    acc = HdT<QBF>::mma32(a, qf[st], acc);
                }
            }
            const int nv = pg ? nv1 : nv0;
#pragma unroll
            for (int i = 0; i < 4; ++i) s[4 * pg + i] = 4 * grp + i < nv ? acc[i] * csc : kNegInf;
        }
        // ---- online softmax (log2 domain), exact running max per head
        float mx = s[0];
#pragma unroll
        for (int i = 1; i < NP; ++i) mx = fmaxf(mx, s[i]);
        mx = fmaxf(m_run, max_over_groups(mx));
        if (__ballot(mx > m_run)) {  // some head's max moved
            const float alpha = mx > m_run ? __builtin_amdgcn_exp2f(m_run - mx) : 1.0f;  // 0 from -inf
            m_run = mx;
            l_part *= alpha;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[t][i] *= alpha;
        }
        const float ref = m_run == kNegInf ? 0.0f : m_run - kOff;
        float pr[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            pr[i] = __builtin_amdgcn_exp2f(s[i] - ref);
            l_part += pr[i];
        }
        // ---- O^T += V^T . P^T, the weights as kTerms 16-bit terms
        uint32_t pt[kTerms][NP / 2];
        auto split = [&](float (&x)[NP]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NP; i += 2) {
                uint32_t w[kTerms];
                WeightTerms<VBF>::split(x[i], x[i + 1], w);
#pragma unroll
                for (int u = 0; u < kTerms; ++u) pt[u][i / 2] = w[u];
            }
        };
        if constexpr (!kGguf) split(pr);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            // (head_dim 256: no reads ahead across groups of tiles, registers)
            if (D == 256 && t % 4 == 0) __builtin_amdgcn_sched_barrier(0);
            if constexpr (kGguf) {
                if (t % 2 == 0) {  // two tiles to a block
                    float x[NP];
#pragma unroll
                    for (int pg = 0; pg < PG; ++pg) {
                        const f32x4 d = *reinterpret_cast<const f32x4*>(lds.sc + GE::scales / 2 +
                                                                        (pg * GE::nblk + t / 2) * 16 + 4 * grp);
#pragma unroll
                        for (int i = 0; i < 4; ++i) x[4 * pg + i] = pr[4 * pg + i] * d[i];
                    }
                    split(x);
                }
            }
            if constexpr (PG == 2) {
                const u32x2 a0 = v_tr(t, 0), a1 = v_tr(t, 1);
                const u32x4 a = {a0[0], a0[1], a1[0], a1[1]};
#pragma unroll
                for (int u = 0; u < kTerms; ++u)
                    o[t] = HdT<VBF>::mma32(a, u32x4{pt[u][0], pt[u][1], pt[u][NP / 2 - 2], pt[u][NP / 2 - 1]}, o[t]);
            } else {
                const u32x2 a = v_tr(t, 0);
#pragma unroll
                for (int u = 0; u < kTerms; ++u) o[t] = HdT<VBF>::mma16(a, u32x2{pt[u][0], pt[u][1]}, o[t]);
            }
        }
        wave_sync();  // the tile is read before the next step's rows replace it
    };

    const uint16_t* qbase = p.q + (int64_t)g * p.G * D;
    uint16_t* obase = reinterpret_cast<uint16_t*>(p.out) + (int64_t)g * p.G * D;
    // ---- pages pa .. pb - 1 of query row b (length L); slot: partial rows of
    // a cut sequence (-1: the output rows)
    auto piece = [&](int b, int pa, int pb, int L, int64_t slot) __attribute__((always_inline)) {
        const int32_t* bt = p.bt + (int64_t)(p.row_seq ? p.row_seq[b] : b) * p.max_blocks;
        const int np = pb - pa;
        auto bt_chunk = [&](int i0) __attribute__((always_inline)) {  // entries of pages pa + i0 + lane
            return i0 + lane < np ? bt[pa + i0 + lane] : -1;
        };
        int bt_cur = bt_chunk(0), bt_nxt = bt_chunk(64);
        // page i of the piece: its id (0 for a hole or past the end) and the
        // tokens of it that count
        auto page = [&](int i, int* nv) __attribute__((always_inline)) {
            const int id = __builtin_amdgcn_readlane(bt_cur, i & 63);
            *nv = i < np && id >= 0 ? min(16, L - 16 * (pa + i)) : 0;
            return max(id, 0);
        };
        int nv0, nv1 = 0;
        int id0 = page(0, &nv0), id1 = PG == 2 ? page(1, &nv1) : 0;
        issue(id0, id1);
#pragma unroll
        for (int st = 0; st < D / 32; ++st) {
            qf[st] = u32x4{0u, 0u, 0u, 0u};
            if (r16 < p.G)
                qf[st] = *reinterpret_cast<const u32x4*>(qbase + ((int64_t)b * p.Hq + r16) * D + 32 * st + 8 * grp);
        }
        m_run = kNegInf;
        l_part = 0.0f;
#pragma unroll
        for (int t = 0; t < NT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int i = 0; i < np; i += PG) {
            const int c0 = nv0, c1 = nv1;
            stage(c0, c1);
            if (i + PG < np) {
                if (((i + PG) & 63) == 0) {
                    bt_cur = bt_nxt;
                    bt_nxt = bt_chunk(i + PG + 64);
                }
                id0 = page(i + PG, &nv0);
                if constexpr (PG == 2) id1 = page(i + PG + 1, &nv1);
                issue(id0, id1);
            }
            compute(c0, c1);
        }
        const float l = sum_over_groups(l_part);
        // an infinity or a NaN in the products (0 * inf for a key of weight 0
        // included) shows as a NaN here: those heads rerun key by key
        bool bad = !(l == l);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) bad |= !(o[t][i] == o[t][i]);
        const uint64_t badb = __ballot(bad && r16 < p.G);
        constexpr uint64_t kCol = 0x0001000100010001ull;  // the four lanes of column 0
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        if (r16 < p.G && !((badb >> r16) & kCol)) {
            if (slot < 0) {
                uint16_t* op = obase + ((int64_t)b * p.Hq + r16) * D + 4 * grp;
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    *reinterpret_cast<u32x2*>(op + 16 * t) = u32x2{pack_half2<QBF>(o[t][0] * inv, o[t][1] * inv),
                                                                   pack_half2<QBF>(o[t][2] * inv, o[t][3] * inv)};
            } else {
                float* pp = p.part + (slot * p.Hq + (int64_t)g * p.G + r16) * (D + 4);
#pragma unroll
                for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(pp + 16 * t + 4 * grp) = o[t];
                // o and l hold weights of 2^(s - m_run + kOff): the reference they go with
                if (grp == 0) *reinterpret_cast<float2*>(pp + D) = make_float2(m_run - kOff, l);
            }
        }
        if (badb) {
            for (int c = 0; c < p.G; ++c) {
                if (!((badb >> c) & kCol)) continue;
                const int64_t r = (int64_t)b * p.Hq + (int64_t)g * p.G + c;
                hd_row_exact<D, FMT, QBF>(p.q + r * D, p.kc, p.vc, bt, p.page_bytes, (uint32_t)p.entry_bytes,
                                          (uint32_t)(p.hnd ? g * kBs : g), (uint32_t)(p.hnd ? 1 : p.Hkv),
                                          p.scale_log2 / kLog2e, 16 * pa, min(16 * pb, L),
                                          reinterpret_cast<float*>(lds.k),
                                          slot < 0 ? reinterpret_cast<uint16_t*>(p.out) + r * D : nullptr,
                                          slot < 0 ? nullptr : p.part + (slot * p.Hq + (int64_t)g * p.G + c) * (D + 4));
            }
        }
    };

    // ---- the unit's pages: range w of the batch's, or (per_seq) row w's
    int p_lo = 0, p_hi = 0, b0 = 0;
    if (p.per_seq) {
        int L = 0;
        p_hi = seq_pages(p, w, &L);
        b0 = w;
        if (p_hi == 0 && r16 < p.G) {
            uint16_t* op = obase + ((int64_t)w * p.Hq + r16) * D + 4 * grp;
#pragma unroll
            for (int t = 0; t < NT; ++t) *reinterpret_cast<u32x2*>(op + 16 * t) = u32x2{0u, 0u};
        }
    } else {
        const int T = total_pages(p, lane);
        if (T == 0) return;  // the merge writes the zero rows
        const int n = effective_wgs(p, T, p.grid);
        if (w >= n) return;
        p_lo = range_lo(p, w, n, T);
        p_hi = range_lo(p, w + 1, n, T);
    }
    int carry = 0;
    for (; b0 < p.B && carry < p_hi; b0 += 64) {
        int L = 0;
        const int pgs = b0 + lane < p.B ? seq_pages(p, b0 + lane, &L) : 0;
        const int incl = wave_incl_scan(pgs, lane);
        const int ps = carry + incl - pgs;
        uint64_t hit = __ballot(pgs > 0 && ps < p_hi && ps + pgs > p_lo);
        while (hit) {
            const int j = (int)__builtin_ctzll(hit);
            hit &= hit - 1;
            const int s0 = __builtin_amdgcn_readlane(ps, j), sn = __builtin_amdgcn_readlane(pgs, j);
            const int Lj = __builtin_amdgcn_readlane(L, j);
            const int64_t slot = s0 < p_lo ? 2 * (int64_t)w : s0 + sn > p_hi ? 2 * (int64_t)w + 1 : -1;
            piece(b0 + j, max(p_lo - s0, 0), min(p_hi - s0, sn), Lj, slot);
        }
        carry += __builtin_amdgcn_readlane(incl, 63);
    }
}

template <int D, int FMT, bool QBF>
int launch_hd(DecodeParams& prm, hipStream_t stream) {
    const int64_t units = (int64_t)prm.grid * prm.Hkv;
    constexpr int W = HdGeo<D, FMT>::waves;
    hipLaunchKernelGGL((paged_decode_hd_kernel<D, FMT, QBF>), dim3((unsigned)((units + W - 1) / W)), dim3(64 * W), 0,
                       stream, prm);
    VMC_LAUNCH_CHECK();
    if (!prm.per_seq) {
        hipLaunchKernelGGL((decode_merge_rows_kernel<D, true>), dim3(prm.B, merge_rows_y(prm.B, prm.Hq)), dim3(256), 0,
                           stream, prm);
        VMC_LAUNCH_CHECK();
    }
    return VMC_OK;
}

template <int D>
int dispatch_hd(DecodeParams& prm, int kv_format, hipStream_t s) {
    switch (kv_format) {
        case VMC_KV_F16: return launch_hd<D, FMT_F16, false>(prm, s);
        case VMC_KV_BF16: return launch_hd<D, FMT_BF16, true>(prm, s);
        case VMC_KV_Q8_0: return prm.q_bf16 ? launch_hd<D, FMT_Q8_0, true>(prm, s) : launch_hd<D, FMT_Q8_0, false>(prm, s);
        case VMC_KV_Q4_0: return prm.q_bf16 ? launch_hd<D, FMT_Q4_0, true>(prm, s) : launch_hd<D, FMT_Q4_0, false>(prm, s);
        default: return VMC_EINVAL;
    }
}

}  // namespace

bool paged_decode_hd_takes(const GenArgs& a) {
    const bool own = a.src == GEN_F16 ? !a.q_bf16 : a.src == GEN_BF16 ? a.q_bf16 != 0 : a.src == GEN_Q8 || a.src == GEN_Q4;
    return own && (a.D == 64 || a.D == 256) && a.bs == kBs && a.Hq / a.Hkv <= 16 && a.rows <= (1 << 24) &&
           (int64_t)a.rows * a.Hkv <= 0x7fffffff && a.max_blocks <= 0x7fffffff / kBs &&
           kBs * a.Hkv * a.entry <= 0x7fffffff &&
           (((uintptr_t)a.q | (uintptr_t)a.out | (uintptr_t)a.kp | (uintptr_t)a.vp) & 15) == 0;
}

int paged_decode_hd(const GenArgs& a, int max_splits, void* ws, size_t ws_bytes, hipStream_t stream) {
    DecodeParams prm = {};
    prm.out = a.out;
    prm.q = reinterpret_cast<const uint16_t*>(a.q);
    prm.kc = a.kp;
    prm.vc = a.vp;
    prm.bt = a.bt;
    prm.seq_lens = a.seq_lens;
    prm.row_seq = a.tok_seq;
    prm.row_pos = a.pos;
    prm.B = a.rows;
    prm.Hq = a.Hq;
    prm.Hkv = a.Hkv;
    prm.G = a.Hq / a.Hkv;
    prm.max_blocks = (int)a.max_blocks;
    prm.scale_log2 = a.scale * kLog2e;
    prm.q_bf16 = a.q_bf16;
    prm.entry_bytes = (int)a.entry;
    prm.page_bytes = kBs * a.Hkv * a.entry;
    prm.hnd = a.hnd;
    prm.part = reinterpret_cast<float*>(ws);
    prm.pps_min = kPpsMin;
    prm.max_splits = max_splits;
    // Page ranges: 12 units per CU at head_dim 64, 8 at 256: one resident wave
    // of them (registers; 32 x 256 .. 8192 tokens at head_dim 64: 47.2 us,
    // 16 per CU 49.8, 24 per CU 53.0, 16 resident at 128 registers 57.6), no
    // more than the workspace has partial rows for.
    // One range per row instead (no partial rows, no merge):
    //  * where a wave walks the longest row the table allows in four steps, about
    //    what the merge takes (100 rows of up to 50 keys, 32/8 heads of 64: 15.8
    //    us in ranges, 5.4; 16/2 heads of 256: 19.8, 11.4);
    //  * from 1024 rows on: a wave each fills the chip or half of it, while every
    //    unit and merge workgroup would scan all rows' lengths (10,000 rows of up
    //    to 300 keys, 32/8 heads of 64: 264 us; in ranges, with a merge workgroup
    //    per row and head, 8.1 ms, and the one-wave kernel 4.1 ms);
    //  * without room for as many ranges as rows or units.  The entry points take
    //    a call without a workspace here, and one sized for rows of 128 dims.
    const int64_t pages = (int64_t)a.rows * a.max_blocks;
    int64_t n = std::max<int64_t>(1, (int64_t)num_cus() * (a.D == 64 ? 12 : 8) / a.Hkv);
    n = std::min<int64_t>(n, (pages + kPpsMin - 1) / kPpsMin);
    if (max_splits > 1) n = std::min<int64_t>(n, (int64_t)a.rows * max_splits);
    const int64_t room =
        ws && ((uintptr_t)ws & 15) == 0 ? (int64_t)(ws_bytes / ((size_t)2 * a.Hq * (a.D + 4) * sizeof(float))) : 0;
    prm.per_seq = max_splits == 1 || a.max_blocks <= (a.D == 64 ? 8 : 4) || a.rows >= 1024 || pages > 0x7fffffff ||
                  room < std::min<int64_t>(n, a.rows) || room < 2;
    prm.grid = prm.per_seq ? a.rows : (int)std::min(n, room);
    const int fmt = a.src == GEN_F16 ? VMC_KV_F16 : a.src == GEN_BF16 ? VMC_KV_BF16 : a.src == GEN_Q8 ? VMC_KV_Q8_0 : VMC_KV_Q4_0;
    return a.D == 64 ? dispatch_hd<64>(prm, fmt, stream) : dispatch_hd<256>(prm, fmt, stream);
}

}  // namespace vmc
