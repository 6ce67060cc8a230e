// attention.hip — paged decode attention (K9), varlen causal prefill attention (K7) and the
// prefix-cached paged prefill variant (K8) for gfx950.
// reference: Attention::flash_attention_decode / compute_attention_with_cache / gather_cached_kv,
// src/layers/attention.rs:225-235,264-318; flash_attention_varlen + causal mask :177-208,321-339;
// GQA mapping kv = h / (H/KVH), :419-435; scale 1/sqrt(D), :45.  Semantics per SURVEY.md A-8/A-9:
// query t sees exactly ctx_lens[t] keys, softmax in f32.
//
// The decode step is HBM-bound (114 688 B of K/V per cached token per step for
// Qwen3-0.6B, 76 % of all decode bytes at ctx 1024), so the kernel is built around the load path:
//  * K and V rows of one kv head are 2·D contiguous bytes; a wave reads whole rows, 16 B per lane,
//    D/8 lanes per row (4 rows = 1 KiB per wave-instruction at D=128) — full 128-B lines, straight
//    to VGPRs (no LDS round trip for a once-read stream), U such loads of K and of V requested back to back.
//  * q·k: v_dot2_f32_f16 on the lane's 8-element slice, then a butterfly over the D/8 lanes of the
//    row; softmax is online (running max / sum per wave, f32), p·v accumulates the lane's slice.
//  * split-KV: one workgroup = WAVES waves owns (query, kv head, partition); its waves interleave
//    row groups and merge through LDS.  With one partition the workgroup writes the fp16 result
//    itself; otherwise f32 partials go to a workspace and a second tiny kernel merges them.
//  * all G = H/KVH query heads of a kv head are processed together so K/V are read once.
#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <type_traits>
#include "kernels.h"
#include "device_utils.h"
#include "../common.h"

namespace nvr { namespace NVR_DT_NS {

struct AttnParams {
    const half_t *q; int64_t ldq;
    const half_t *k, *v; int64_t ldkv;
    const int32_t *ctx_lens, *seq_of_q, *kv_base, *block_tables;
    int32_t max_blocks, block_size, bs_shift;
    int32_t H, KVH;
    float scale;
    int32_t part_size, num_parts;
    int32_t part0, kv0;                // shared-prefix decode: partitions 0..part0-1 hold the batch's shared keys [0, kv0) (written by
                                       // flash_shared_prefix); this launch covers partition part0 + i = keys [kv0 + i*part_size, ..)
    const int32_t *kv0_rows;           // per-query kv0 (shared-prefix groups: members shared_len, others 0) or null = p.kv0 for all
    float *part_o; float *part_ml;     // [nq, H, num_parts, D], [nq, H, num_parts, 2]
    half_t *out;                       // [nq, H, D]
    unsigned int *tickets;             // FUSE: one arrival counter per (query, kv head), zero between launches (the last arriver re-arms it)
};
struct OwnRows { const half_t *qn_w, *kn_w; float qk_eps; const int64_t *pos; const int32_t *slots; const float *cos_t, *sin_t; };   // QKN (AttnArgs)
struct AttnParamsOwn : AttnParams, OwnRows {};         // (a type of its own: the arguments of the other instances stay as short as they were)
struct OutRows { const half_t *w; float *slabs; int64_t stride; int32_t N; };       // OUTP: the output product's weights [N][H D] and its slabs, one per kv head, `stride` elements apart
struct AttnParamsOut : AttnParams, OwnRows, OutRows {};
template <bool QKN, bool OUTP = false> struct AttnParamsOf { using type = AttnParams; };
template <> struct AttnParamsOf<true, false> { using type = AttnParamsOwn; };
template <bool QKN> struct AttnParamsOf<QKN, true> { using type = AttnParamsOut; };

// One 8-element piece of a head of 128 held by 16 lanes (dc = lane % 16, elements dc * 8 ..): RMSNorm over the head and rotation as qknorm_rope_store_kernel does them — its sums' pairs, its
// roundings, nothing contracted: the same bits.  g: the norm's weights of the piece, c / s: cosines and sines of pairs (dc % 8) * 8 ..
__device__ __forceinline__ half8_t norm_rotate_piece(half8_t x, half8_t g, const float4_t (&c)[2], const float4_t (&s)[2], float eps, int dc) {
#pragma clang fp contract(off)
    auto partner = [](half8_t v) {                      // the other half's piece, 8 lanes away inside the row of 16
        int4 w = __builtin_bit_cast(int4, v);
        w.x = __builtin_amdgcn_update_dpp(0, w.x, 0x128, 0xF, 0xF, false); w.y = __builtin_amdgcn_update_dpp(0, w.y, 0x128, 0xF, 0xF, false);
        w.z = __builtin_amdgcn_update_dpp(0, w.z, 0x128, 0xF, 0xF, false); w.w = __builtin_amdgcn_update_dpp(0, w.w, 0x128, 0xF, 0xF, false);
        return __builtin_bit_cast(half8_t, w);
    };
    const bool low = dc < 8;
    const half8_t px = partner(x);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float a = (float)(low ? x[e] : px[e]), b = (float)(low ? px[e] : x[e]), aa = a * a, bb = b * b, ab = aa + bb;
        ss = ss + ab;
    }
    ss = head_sum<8>(ss);
    const float rms = sqrtf(ss / 128.0f + eps);
    half8_t n, o;
#pragma unroll
    for (int e = 0; e < 8; ++e) n[e] = to_half_rn(__fmul_rn(__fdiv_rn((float)x[e], rms), (float)g[e]));
    const half8_t pn = partner(n);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float cc = c[e >> 2][e & 3], sn = s[e >> 2][e & 3];
        o[e] = low ? to_half_rn(mul_sub_unfused((float)n[e], cc, (float)pn[e], sn)) : to_half_rn(mul_add_unfused((float)n[e], cc, (float)pn[e], sn));
    }
    return o;
}

// a * b rounded, then + c rounded: never contracted into an fma, whatever kernel this is inlined into
__device__ __forceinline__ float mul_then_add(float a, float b, float c) {
#pragma clang fp contract(off)
    return a * b + c;
}

template <bool NT>
__device__ __forceinline__ half8_t load_row16(const half_t *p) {
    if (NT) return __builtin_nontemporal_load(reinterpret_cast<const half8_t *>(p));
    return *reinterpret_cast<const half8_t *>(p);
}

// sum / max over the 64/LPR row groups of the wave (lanes with equal lane % LPR), result in every lane
template <int LPR>
__device__ __forceinline__ float groups_sum(float x) {
    if (LPR == 8) x = dpp_add<0x128>(x);                                   // row_ror:8 inside the 16-lane row
    return xor32_partner_sum(xor16_partner_sum(x));
}
template <int LPR>
__device__ __forceinline__ float groups_max(float x) {
    if (LPR == 8) x = fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xF, 0xF, false)));
    return xor32_partner_max(xor16_partner_max(x));
}

// A wave-instruction reads one ROW GROUP: RPI = 64/(D/8) consecutive tokens of one kv head, 16 B per lane (1 KiB).
// The partition is cut into chunks of U row groups (TPI = U*RPI consecutive tokens); in a FULL round every wave of
// the workgroup takes one complete chunk (chunk r*WAVES + wave: the waves' loads are neighbours in memory) and
// requests its U groups of K and of V back to back before any arithmetic, with no validity tests.  What is left
// after the last full round (< WAVES*U groups, the last one possibly partial) is dealt out group by group
// (group j -> wave j % WAVES) and requested BEFORE the arithmetic of the last full round, so the remainder costs no
// extra exposed memory round trip and no wave has more than one group more than another.
// NT: non-temporal loads.  UB: block_size is a multiple of TPI, so a chunk lies inside ONE cache block: its
// block-table entry is a scalar read (v_readlane) from a register copy of the table (lane j holds entry
// 64*c + j) and the row address is scalar base + small lane offset -- no dependent table load sits between the row
// loads.
// out = sum_p e^(m_p-M) o_p / sum_p e^(m_p-M) l_p over partitions [0, np) of ONE (query, head), 4 columns per thread: the partials of up
// to 8 partitions are requested together (a runtime-count loop of dependent loads would pay one round trip per partition); sums run over
// the partitions in ascending order for every column.  load_ml(i) / load_o(i): (max, sum) and the 4 columns of partition i — plain loads
// in the merge kernel, sc1 loads in the last arriver of the fused form (the same arithmetic: the two forms agree bit for bit).
template <class LoadML, class LoadO>
__device__ __forceinline__ half4_t merge_partitions(int np, LoadML load_ml, LoadO load_o) {
    float M = -INFINITY;
    float4_t o = {0.f, 0.f, 0.f, 0.f};
    float L = 0.f;
    for (int i0 = 0; i0 < np; i0 += 8) {
        float2_t ml[8]; float4_t po[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = min(i0 + u, np - 1);
            ml[u] = load_ml(i);
            po[u] = load_o(i);
        }
        float Mn = M;
#pragma unroll
        for (int u = 0; u < 8; ++u) if (i0 + u < np) Mn = fmaxf(Mn, ml[u][0]);
        if (i0 > 0 && Mn != M) { const float r = __expf(M - Mn); o *= r; L *= r; }     // (more than 8 partitions: rescale what is summed)
        M = Mn;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (i0 + u < np) {
                const float w = __expf(ml[u][0] - M);
                // (spelled out as fused multiply-adds: under -ffp-contract=fast hipcc decides per INSTANTIATION whether "a += w * b" becomes an fma,
                //  and this function is inlined into three kernels whose results are promised to agree bit for bit; fma is what the merge kernel got)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = __fmaf_rn(w, po[u][e], o[e]);
                L = __fmaf_rn(w, ml[u][1], L);
            }
        }
    }
    half4_t hv;
#pragma unroll
    for (int e = 0; e < 4; ++e) hv[e] = (half_t)(L > 0.f ? o[e] / L : 0.f);
    return hv;
}

// FUSE (split-KV, no shared-prefix pass): the merge of a (query, kv head)'s partitions rides on the LAST ARRIVER of its partition workgroups
// instead of a second launch (cdna guide Guideline 16, counter form): every workgroup publishes its partials write-through (sc1), drains,
// and one lane draws a ticket from the pair's counter; the workgroup whose ticket says it came last reads all partials back with sc1 loads
// and merges them with merge_partitions — nobody polls.  On a tensor-parallel rank (1-2 kv heads) every kernel of the decode step sits on the
// launch floor: one launch less per layer.
// SHM (shared-prefix decode where EVERY query shares the prefix and its own keys fit one partition): the partials of the shared
// partitions [0, part0) were written by the launch in front of this one (flash_shared_prefix), so the single own-partition workgroup of a (query, kv head) IS
// the last arriver by stream order: it merges the pair itself (own partial through LDS, the same merge_partitions: the merge launch's bits) — no merge launch.
// QKN (heads of 128, UB): the step's own rows come raw — RMSNorm over q and k heads, rotation and the store of the new key and value row ride here instead of a launch of their own in front
// (4.6 us a layer at a few rows, as much as this whole kernel over short contexts): the first waves form the G query heads and the key row, 16 lanes a head, while every wave's first keys are on
// their way; all read them back from LDS.  The row of the last key is taken from there, not from the cache; the workgroup whose keys end with it stores it.
// OUTP (one workgroup's worth of keys per pair, few queries): the output product rides here.  blockIdx.y = OUTP (64 or 128) of its rows: the workgroups of a pair all form the pair's G heads (its keys come from
// one XCD's L2, where the pairs' workgroups meet) and multiply them, rounded as the launch between the two rounded them, with their rows of the G D columns of W that belong to the pair, requested behind
// the first keys; the pair's sums go to slab g, added up by the norm that reads the slabs.  Launches bound such a step: one sequence of 128 keys, 16 heads, 1024 columns, attention 6.9 and product
// 4.1 us, so 6.5 (attn_out_rides).
constexpr int OUT_ROWS = 64;                              // (128 where 64 would put two workgroups on a CU)
template <int D, int G, bool PAGED, bool DIRECT_OUT, int U, int WAVES, bool NT, bool UB, bool FUSE = false, bool SHM = false, bool QKN = false, int OUTP = 0>
__global__ __launch_bounds__(WAVES * 64) void attn_rows_kernel(typename AttnParamsOf<QKN, (OUTP > 0)>::type own) {
    const AttnParams &p = own;                          // (a type that does not depend on the instance: hipcc drops the host stub otherwise)
    static_assert(!QKN || (D == 128 && PAGED && UB && !SHM && G < 4 * WAVES), "QKN: paged heads of 128");
    static_assert(!OUTP || (PAGED && DIRECT_OUT && WAVES == 8 && G * D <= 512), "OUTP: a wave takes eight rows of up to 64 pieces of the product");
    constexpr int LPR = D / 8;          // lanes per K/V row
    constexpr int RPI = 64 / LPR;       // rows per wave-instruction (= tokens per row group)
    constexpr int TPI = RPI * U;        // tokens per chunk
    const int lparts = p.num_parts - p.part0;        // partitions of this launch
    const int part = p.part0 + blockIdx.x % lparts, g = (blockIdx.x / lparts) % p.KVH;
    const int t = blockIdx.x / (lparts * p.KVH);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int dc = lane % LPR, tg = lane / LPR;
    const int p0 = (p.kv0_rows ? p.kv0_rows[t] : p.kv0) + (part - p.part0) * p.part_size;

    const int32_t *bt = PAGED ? p.block_tables + (int64_t)(p.seq_of_q ? p.seq_of_q[t] : t) * p.max_blocks : nullptr;
    int bt_chunk = -1, bt_reg = 0;                   // UB: register copy of 64 block-table entries
    auto load_bt_chunk = [&](int c) {
        bt_chunk = c;
        const int idx = (c << 6) + lane;
        bt_reg = idx < p.max_blocks ? bt[idx] : 0;
    };
    if (PAGED && UB) {                               // requested together with ctx and q, ahead of their use
        const int b0 = p.bs_shift >= 0 ? p0 >> p.bs_shift : p0 / p.block_size;
        load_bt_chunk(b0 >> 6);
    }

    // SHM: the shared partitions' partials [G heads][part0][D] (+ their (max, sum) pairs) go straight into LDS by LDS-DMA, requested HERE, with ctx and
    // the block table: as loads of the merge at the end of the kernel they were a third dependent round trip in the life of a workgroup whose own
    // keys are two chunks per wave (configs[4]: 4096 workgroups of ~94 own tokens, 43 us per layer = 0.57 of HBM; profiles/r05_priced_levers.txt 7.)
    constexpr int SHP = 4;                            // shared partitions whose partials are staged (more: the merge reads them from global memory)
    __shared__ __attribute__((aligned(16))) float shm_po[SHM ? G * SHP * D : 4];
    __shared__ float shm_pml[SHM ? G * SHP * 2 : 1];
    const bool staged = SHM && p.part0 <= SHP;
    if (SHM && staged) {
        const int per_head = p.part0 * (D / 4), total = G * per_head;            // 16-byte pieces, lane-linear in LDS: [head][partition][D]
        const float *src0 = p.part_o + ((int64_t)t * p.H + (int64_t)g * G) * p.num_parts * D;
        for (int x0 = wave * 64; x0 < total; x0 += WAVES * 64) {
            const int x = x0 + lane;
            if (x < total) {
                const int i = x / per_head, rem = x - i * per_head;
                __builtin_amdgcn_global_load_lds(src0 + ((int64_t)i * p.num_parts * (D / 4) + rem) * 4,
                                                 (__attribute__((address_space(3))) void *)(shm_po + x0 * 4), 16, 0, 0);
            }
        }
        if (wave == WAVES - 1 && lane < G * p.part0 * 2) {
            const int i = lane / (p.part0 * 2), rem = lane - i * (p.part0 * 2);
            __builtin_amdgcn_global_load_lds(p.part_ml + (((int64_t)t * p.H + (int64_t)g * G + i) * p.num_parts) * 2 + rem,
                                             (__attribute__((address_space(3))) void *)shm_pml, 4, 0, 0);
        }
    }
    // QKN: head item wave * 4 + tg (G query heads, then the key head) of the step's row, and the value row's piece
    const half_t *own_row = QKN ? p.q + (int64_t)t * p.ldq : nullptr;
    const int hi = wave * 4 + tg;
    int own_slot = -1;
    const bool forms = QKN && wave * 4 <= G;                              // (uniform)
    half8_t hx, hg, own_k, own_v; float4_t hc[2], hs[2];
    __shared__ half8_t own_lds[QKN ? (G + 1) * 16 : 1];
    if constexpr (QKN) {
        if (own.slots) own_slot = own.slots[t];
        const int64_t at = own.pos[t] * (D / 2) + (dc & 7) * 8;
        if (forms) {
            const int hh = min(hi, G);
            hx = *reinterpret_cast<const half8_t *>(own_row + (hh < G ? g * G + hh : p.H + g) * D + dc * 8);
            hg = *reinterpret_cast<const half8_t *>((hh < G ? own.qn_w : own.kn_w) + dc * 8);
#pragma unroll
            for (int x = 0; x < 2; ++x) { hc[x] = *reinterpret_cast<const float4_t *>(own.cos_t + at + 4 * x); hs[x] = *reinterpret_cast<const float4_t *>(own.sin_t + at + 4 * x); }
        }
        own_v = *reinterpret_cast<const half8_t *>(own_row + (p.H + p.KVH + g) * D + dc * 8);
    }
    // q slice of this lane for the G heads of kv head g (fp16 pairs for v_dot2); requested in front of ctx's first use
    half2_t qv[G][4];
    if constexpr (!QKN) {
        const half_t *qrow = p.q + (int64_t)t * p.ldq + (int64_t)g * G * D + dc * 8;
#pragma unroll
        for (int i = 0; i < G; ++i) {
            half8_t h = *reinterpret_cast<const half8_t *>(qrow + i * D);
#pragma unroll
            for (int j = 0; j < 4; ++j) qv[i][j] = (half2_t){h[2 * j], h[2 * j + 1]};
        }
    }
    const int ctx = p.ctx_lens[t];
    if (p0 >= ctx && !(DIRECT_OUT) && !SHM) return;  // empty partition: the merge kernel skips it too (SHM: this workgroup still merges the shared partitions)
    const int pend = max(p0, min(ctx, p0 + p.part_size));
    const int64_t base_row = PAGED ? 0 : (int64_t)p.kv_base[t];
    const int row_elems = p.KVH * D;

    // element offset of (scalar token tb, kv head g, d = 0) through the register copy of the block table
    auto block_base = [&](int tb) -> int64_t {
        int bi, bo;
        if (p.bs_shift >= 0) { bi = tb >> p.bs_shift; bo = tb & (p.block_size - 1); }
        else { bi = tb / p.block_size; bo = tb - bi * p.block_size; }
        if ((bi >> 6) != bt_chunk) load_bt_chunk(bi >> 6);
        const int blk = __builtin_amdgcn_readlane(bt_reg, bi & 63);
        return (((int64_t)blk * p.block_size + bo) * p.KVH + g) * D;
    };
    // per-lane form (contiguous K/V, or block sizes that are no multiple of the chunk)
    auto lane_row = [&](int tok) -> int64_t {
        if (PAGED) {
            int bi, bo;
            if (p.bs_shift >= 0) { bi = tok >> p.bs_shift; bo = tok & (p.block_size - 1); }
            else { bi = tok / p.block_size; bo = tok - bi * p.block_size; }
            return (((int64_t)bt[bi] * p.block_size + bo) * p.KVH + g) * D + dc * 8;
        }
        return (base_row + tok) * p.ldkv + (int64_t)g * D + dc * 8;
    };

    // online softmax state per head AND per row-group slot of the wave (the 64/LPR lane groups never exchange data
    // inside the loop; they are merged once at the end)
    float m[G], l[G], acc[G][8];
#pragma unroll
    for (int i = 0; i < G; ++i) {
        m[i] = -INFINITY; l[i] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = 0.f;
    }

    // scores, online softmax and p.v for U row groups; CHECK: slot u holds token tok0 + u*WAVES*RPI + tg, valid < pend
    auto process = [&](auto check, const half8_t (&kk)[U], const half8_t (&vv)[U], int tok0) {
        constexpr bool CHECK = decltype(check)::value;
        float s[U][G];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool valid = !CHECK || tok0 + u * (WAVES * RPI) + tg < pend;
#pragma unroll
            for (int i = 0; i < G; ++i) {
                float d = 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    d = dot2((half2_t){kk[u][2 * j], kk[u][2 * j + 1]}, qv[i][j], d);
                d = row_sum<LPR>(d);
                s[u][i] = valid ? d * p.scale : -INFINITY;
            }
        }
#pragma unroll
        for (int i = 0; i < G; ++i) {
            float mx = s[0][i];
#pragma unroll
            for (int u = 1; u < U; ++u) mx = fmaxf(mx, s[u][i]);
            const float mn = fmaxf(m[i], mx);
            const float ms = (CHECK && mn == -INFINITY) ? 0.f : mn;   // a slot that has seen no valid token yet
            const float alpha = __expf(m[i] - ms);                    // m = -inf on first use -> 0
            m[i] = mn;
            float ps = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[i][j] *= alpha;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float pr = __expf(s[u][i] - ms);
                ps += pr;
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[i][j] = fmaf(pr, (float)vv[u][j], acc[i][j]);
            }
            l[i] = __fmaf_rn(l[i], alpha, ps);                         // (pinned: see the cross-wave merge below)
        }
    };

    const int ng = (pend - p0 + RPI - 1) / RPI;      // row groups of this partition, the last one possibly partial
    const int R = (pend - p0) / (TPI * WAVES);       // full rounds: every wave gets a complete chunk
    const int gt0 = R * (WAVES * U) + wave;          // this wave's remainder groups: gt0, gt0 + WAVES, ..
    auto issue_remainder = [&](half8_t (&kt)[U], half8_t (&vt)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int gt = gt0 + u * WAVES;
            if (gt < ng) {                           // uniform
                const int tb = p0 + gt * RPI;
                if (PAGED && UB) {
                    const int64_t base = block_base(tb);
                    const unsigned lo = (unsigned)(min(tg, pend - 1 - tb) * row_elems + dc * 8);
                    kt[u] = load_row16<NT>(p.k + base + lo); vt[u] = load_row16<NT>(p.v + base + lo);
                } else {
                    const int64_t off = lane_row(min(tb + tg, pend - 1));
                    kt[u] = load_row16<NT>(p.k + off); vt[u] = load_row16<NT>(p.v + off);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) { kt[u][j] = (half_t)0.f; vt[u][j] = (half_t)0.f; }
            }
        }
    };

    half8_t kt[U], vt[U];
    if (R == 0) issue_remainder(kt, vt);
    // OUTP: LW lanes hold a row's G D columns, a wave's 64 / LW groups of lanes OL consecutive rows each
    constexpr int LW = OUTP ? G * D / 8 : 64, OL = OUTP == 128 ? LW / 4 : LW / 8;
    half8_t ow[OUTP ? OL : 1];
    const int on = blockIdx.y * OUTP + wave * (OUTP / 8) + lane / LW * OL;
    auto request_out = [&]() {
        if constexpr (OUTP > 0) {
            const half_t *w = own.w + (int64_t)on * (p.H * D) + g * (G * D) + lane % LW * 8;
#pragma unroll
            for (int u = 0; u < OL; ++u) ow[u] = *reinterpret_cast<const half8_t *>(w + (int64_t)u * (p.H * D));
        }
    };
    if constexpr (OUTP > 0 && !QKN) {
        half8_t kk[U], vv[U];
        auto issue_round = [&](int tb) {
            if constexpr (UB) {
                const int64_t base = block_base(tb);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const unsigned lo = (unsigned)((u * RPI + tg) * row_elems + dc * 8);
                    kk[u] = load_row16<NT>(p.k + base + lo); vv[u] = load_row16<NT>(p.v + base + lo);
                }
            } else {
                int64_t off[U];
#pragma unroll
                for (int u = 0; u < U; ++u) off[u] = lane_row(tb + u * RPI + tg);
#pragma unroll
                for (int u = 0; u < U; ++u) { kk[u] = load_row16<NT>(p.k + off[u]); vv[u] = load_row16<NT>(p.v + off[u]); }
            }
        };
        if (R > 0) issue_round(p0 + wave * TPI);
        asm volatile("" ::: "memory");
        request_out();
        for (int r = 0; r < R; ++r) {
            if (r > 0) issue_round(p0 + (r * WAVES + wave) * TPI);
            if (r == R - 1) issue_remainder(kt, vt);
            process(std::false_type{}, kk, vv, 0);
        }
    } else if constexpr (QKN) {
        half8_t kk[U], vv[U];
        auto issue_round = [&](int tb) {
            const int64_t base = block_base(tb);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const unsigned lo = (unsigned)((u * RPI + tg) * row_elems + dc * 8);
                kk[u] = load_row16<NT>(p.k + base + lo); vv[u] = load_row16<NT>(p.v + base + lo);
            }
        };
        if (R > 0) issue_round(p0 + wave * TPI);
        asm volatile("" ::: "memory");                                    // the requests stay in front of the norm
        request_out();
        if (forms) {
            const half8_t o = norm_rotate_piece(hx, hg, hc, hs, own.qk_eps, dc);
            if (hi <= G) own_lds[hi * 16 + dc] = o;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                // (LDS alone: __syncthreads may wait for the keys as well)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const half8_t h = own_lds[i * 16 + dc];
#pragma unroll
            for (int j = 0; j < 4; ++j) qv[i][j] = (half2_t){h[2 * j], h[2 * j + 1]};
        }
        own_k = own_lds[G * 16 + dc];
        if (wave == WAVES - 1 && tg == 0 && own_slot >= 0 && pend == ctx && p0 < ctx && (!OUTP || blockIdx.y == 0)) {
            const int64_t dst = ((int64_t)own_slot * p.KVH + g) * D + dc * 8;
            *reinterpret_cast<half8_t *>(const_cast<half_t *>(p.k) + dst) = own_k;
            *reinterpret_cast<half8_t *>(const_cast<half_t *>(p.v) + dst) = own_v;
        }
        // the pieces of token ctx - 1 among rows tb + step * u + tg (clamped to the partition's last one: those lanes' weights are 0, but what they are multiplied with has to be a number)
        auto take_own = [&](half8_t (&ka)[U], half8_t (&va)[U], int tb, int step) {
            if (own_slot >= 0)
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (min(tb + step * u + tg, pend - 1) == ctx - 1) { ka[u] = own_k; va[u] = own_v; }
        };
        for (int r = 0; r < R; ++r) {
            const int tb = p0 + (r * WAVES + wave) * TPI;
            if (r > 0) issue_round(tb);
            if (r == R - 1) issue_remainder(kt, vt);
            if (tb + TPI >= ctx) take_own(kk, vv, tb, RPI);
            process(std::false_type{}, kk, vv, 0);
        }
        if (gt0 < ng && p0 + (gt0 + (U - 1) * WAVES + 1) * RPI >= ctx) take_own(kt, vt, p0 + gt0 * RPI, WAVES * RPI);
    } else {
        // (a loop of its own: with its requests in the lambda above, hipcc forms the addresses otherwise, and a launch is slower: 24 x 700 keys 15.6 / 16.0 us, 32 x 2048 of 32 heads 45.8 / 46.1,
        // 256 x 1024 161 / 162)
        for (int r = 0; r < R; ++r) {
            const int tb = p0 + (r * WAVES + wave) * TPI;
            half8_t kk[U], vv[U];
            if (PAGED && UB) {
                const int64_t base = block_base(tb);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const unsigned lo = (unsigned)((u * RPI + tg) * row_elems + dc * 8);
                    kk[u] = load_row16<NT>(p.k + base + lo); vv[u] = load_row16<NT>(p.v + base + lo);
                }
            } else {
                int64_t off[U];
#pragma unroll
                for (int u = 0; u < U; ++u) off[u] = lane_row(tb + u * RPI + tg);
#pragma unroll
                for (int u = 0; u < U; ++u) { kk[u] = load_row16<NT>(p.k + off[u]); vv[u] = load_row16<NT>(p.v + off[u]); }
            }
            if (r == R - 1) issue_remainder(kt, vt);
            process(std::false_type{}, kk, vv, 0);
        }
    }
    if (gt0 < ng) process(std::true_type{}, kt, vt, p0 + gt0 * RPI);

    // bring the row-group slots of the wave to their common max and sum them, then merge the waves through LDS
    constexpr bool ONE = SHM && WAVES == 1;                               // one wave per workgroup: its sums ARE the partition's partial (the cross-wave
                                                                          // merge below would multiply them by exp(0) = 1 and add them to 0)
    __shared__ float sm_acc[ONE ? 1 : WAVES][ONE ? 1 : G][ONE ? 1 : D];
    __shared__ float sm_ml[WAVES][G][2];
    __shared__ float shm_o[SHM ? G : 1][SHM ? D : 1];                     // SHM: this workgroup's own partial, merged below with the shared partitions'
    __shared__ float shm_ml[SHM ? G : 1][2];
#pragma unroll
    for (int i = 0; i < G; ++i) {
        const float M = groups_max<LPR>(m[i]);
        const float w = (m[i] == -INFINITY) ? 0.f : __expf(m[i] - M);
        l[i] = groups_sum<LPR>(l[i] * w);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = groups_sum<LPR>(acc[i][j] * w);
        if (tg == 0) {
            if constexpr (ONE) {
#pragma unroll
                for (int j = 0; j < 8; ++j) shm_o[i][dc * 8 + j] = acc[i][j];
                if (dc == 0) { shm_ml[i][0] = M; shm_ml[i][1] = l[i]; }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) sm_acc[wave][i][dc * 8 + j] = acc[i][j];
                if (dc == 0) { sm_ml[wave][i][0] = M; sm_ml[wave][i][1] = l[i]; }
            }
        }
    }
    if constexpr (!ONE) __syncthreads();
    // the pair's partials are contiguous: [G heads][num_parts][D] (and [..][2]); buffer offsets stay small whatever the workspace size
    const int64_t pair0 = DIRECT_OUT ? 0 : ((int64_t)t * p.H + (int64_t)g * G) * p.num_parts;
    const auto rs_o = __builtin_amdgcn_make_buffer_rsrc(DIRECT_OUT ? nullptr : p.part_o + pair0 * D, 0, DIRECT_OUT ? 0 : (int)(G * p.num_parts * D * 4), 0x00020000);
    const auto rs_ml = __builtin_amdgcn_make_buffer_rsrc(DIRECT_OUT ? nullptr : p.part_ml + pair0 * 2, 0, DIRECT_OUT ? 0 : (int)(G * p.num_parts * 2 * 4), 0x00020000);
    constexpr int AUX = FUSE ? 16 : 0;                                    // sc1: write-through, so the hand-off needs no release fence
    __shared__ __attribute__((aligned(16))) half_t heads[OUTP ? G * D : 8];
    if constexpr (!ONE)
    for (int idx = threadIdx.x; idx < G * D; idx += WAVES * 64) {
        const int i = idx / D, d = idx % D;
        float M = sm_ml[0][i][0];
#pragma unroll
        for (int w2 = 1; w2 < WAVES; ++w2) M = fmaxf(M, sm_ml[w2][i][0]);
        float o = 0.f, L = 0.f;
#pragma unroll
        for (int w2 = 0; w2 < WAVES; ++w2) {
            const float mw = sm_ml[w2][i][0];
            const float wgt = (mw == -INFINITY) ? 0.f : __expf(mw - M);
            // (multiply, THEN add, spelled out: left to -ffp-contract=fast the SHM instantiation of this loop got fmas where the instantiation in front of
            //  the merge launch got v_pk_mul + v_add — a 1-ulp difference that flipped ~1 output in 10^5 between two forms promised to be bit-identical
            //  (r05, found at 300 sequences; the 9-sequence test was too small to see it).  Unfused is what the partial-writing instantiations always were;
            //  HIP's __fmul_rn / __fadd_rn are plain * and + and contract like them, hence the helper with contraction switched off.)
            o = mul_then_add(wgt, sm_acc[w2][i][d], o);
            L = mul_then_add(wgt, sm_ml[w2][i][1], L);
        }
        const int h = g * G + i;
        if constexpr (OUTP > 0) {
            heads[idx] = (half_t)(L > 0.f ? o / L : 0.f);
        } else if (DIRECT_OUT) {
            p.out[((int64_t)t * p.H + h) * D + d] = (half_t)(L > 0.f ? o / L : 0.f);
        } else if (SHM) {
            shm_o[i][d] = o;
            if (d == 0) { shm_ml[i][0] = M; shm_ml[i][1] = L; }
        } else {
            const int slot = i * p.num_parts + part;                     // inside the pair's region
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), rs_o, (slot * D + d) * 4, 0, AUX);
            if (d == 0) { __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(M), rs_ml, slot * 8, 0, AUX);
                          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(L), rs_ml, slot * 8 + 4, 0, AUX); }
        }
    }
    if constexpr (OUTP > 0) {
        __syncthreads();
        const half8_t x = *reinterpret_cast<const half8_t *>(heads + lane % LW * 8);
        float y[OL];
#pragma unroll
        for (int u = 0; u < OL; ++u) {
            float d = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) d = dot2((half2_t){x[2 * j], x[2 * j + 1]}, (half2_t){ow[u][2 * j], ow[u][2 * j + 1]}, d);
            d = row_sum<LW < 16 ? LW : 16>(d);
            if (LW >= 32) d = xor16_partner_sum(d);
            if (LW >= 64) d = xor32_partner_sum(d);
            y[u] = d;
        }
        if (lane % LW == 0) {
            float *const to = own.slabs + g * own.stride + (int64_t)t * own.N + on;
#pragma unroll
            for (int u = 0; u < OL; ++u) to[u] = y[u];
        }
    }
    if constexpr (!DIRECT_OUT) {
        constexpr int TPH = D / 4;                                // merging threads per head: 4 columns each (merge_partitions)
        static_assert(G * TPH <= WAVES * 64, "one pass over the (head, column group) pairs");
        if constexpr (SHM) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                  // the LDS-DMA requests of the shared partitions' partials (long landed)
            __syncthreads();
            if (threadIdx.x < G * TPH) {
                const int i = threadIdx.x / TPH, d = (threadIdx.x % TPH) * 4;
                const int own = part;                                         // = part0: the one partition of this launch
                const int np = own + (ctx > p0 ? 1 : 0);                      // shared partitions, then the own one if the query has own keys
                const int64_t base = ((int64_t)t * p.H + g * G + i) * p.num_parts;
                const float2_t own_ml = {shm_ml[i][0], shm_ml[i][1]};
                const float4_t own_o = {shm_o[i][d], shm_o[i][d + 1], shm_o[i][d + 2], shm_o[i][d + 3]};
                half4_t hv;
                if (staged)
                    hv = merge_partitions(np,
                        [&](int pi) { return pi < own ? *reinterpret_cast<const float2_t *>(shm_pml + (i * own + pi) * 2) : own_ml; },
                        [&](int pi) { return pi < own ? *reinterpret_cast<const float4_t *>(shm_po + (i * own + pi) * D + d) : own_o; });
                else
                    hv = merge_partitions(np,
                        [&](int pi) { return pi < own ? *reinterpret_cast<const float2_t *>(p.part_ml + (base + pi) * 2) : own_ml; },
                        [&](int pi) { return pi < own ? *reinterpret_cast<const float4_t *>(p.part_o + (base + pi) * D + d) : own_o; });
                *reinterpret_cast<half4_t *>(p.out + ((int64_t)t * p.H + g * G + i) * D + d) = hv;
            }
        }
        if constexpr (FUSE) {
            __shared__ unsigned int ticket_s;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                  // every storing wave drains its stores ...
            __syncthreads();
            unsigned int *cnt = p.tickets + (int64_t)t * p.KVH + g;
            if (threadIdx.x == 0) ticket_s = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ... one ticket
            __syncthreads();
            const int np = min(p.num_parts, (ctx + p.part_size - 1) / p.part_size);   // non-empty partitions of this query
            if (ticket_s != (unsigned)(np - 1)) return;                       // not the last partition of this pair to finish: done
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");            // keeps the sc1 loads below the ticket
            if (threadIdx.x < G * TPH) {
                const int i = threadIdx.x / TPH, d = (threadIdx.x % TPH) * 4;
                const half4_t hv = merge_partitions(np,
                    [&](int pi) { return __builtin_bit_cast(float2_t, __builtin_amdgcn_raw_buffer_load_b64(rs_ml, (i * p.num_parts + pi) * 8, 0, 16)); },
                    [&](int pi) { return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rs_o, ((i * p.num_parts + pi) * D + d) * 4, 0, 16)); });
                *reinterpret_cast<half4_t *>(p.out + ((int64_t)t * p.H + g * G + i) * D + d) = hv;
            }
            if (threadIdx.x == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // re-arm for the next launch
        }
    }
}

// merge split-KV partitions: out = sum_p e^(m_p-M) o_p / sum_p e^(m_p-M) l_p
// 32 (D = 128) or 16 (D = 64) threads per (query, head), 4 columns each; the partials of up to 8 partitions are requested together
// (a runtime-count loop of dependent loads would pay one round trip per partition).  Sums run over the partitions in ascending
// order for every column, as before.
template <int D>
__global__ __launch_bounds__(256) void attn_merge_kernel(const float *__restrict__ part_o, const float *__restrict__ part_ml,
                                                         const int32_t *__restrict__ ctx_lens, int H, int part_size, int num_parts,
                                                         int part0, int kv0, const int32_t *__restrict__ kv0_rows, int64_t pairs,
                                                         half_t *__restrict__ out) {
    constexpr int TPP = D / 4;                                   // threads per (query, head) pair
    const int64_t pair = (int64_t)blockIdx.x * (256 / TPP) + threadIdx.x / TPP;
    if (pair >= pairs) return;
    const int t = (int)(pair / H), d = (threadIdx.x % TPP) * 4;
    const int my_kv0 = kv0_rows ? kv0_rows[t] : kv0;
    const int first = (part0 > 0 && my_kv0 == 0) ? part0 : 0;   // a query outside the sharing group has no partials in the shared slots
    const int np = min(num_parts, part0 + (max(ctx_lens[t] - my_kv0, 0) + part_size - 1) / part_size) - first;
    const int64_t base = pair * num_parts + first;
    const half4_t hv = merge_partitions(np,
        [&](int i) { return *reinterpret_cast<const float2_t *>(part_ml + (base + i) * 2); },
        [&](int i) { return *reinterpret_cast<const float4_t *>(part_o + (base + i) * D + d); });
    *reinterpret_cast<half4_t *>(out + pair * D + d) = hv;
}

// ---- work-balanced form ---------------------------------------------------------------------------------------
// attn_rows_kernel gives every (query, kv head) pair its own workgroup(s): 264 pairs on 256 CUs (33 sequences x 8 kv heads) run as one full round and a tail,
// 35.6 us per layer where 256 pairs take 24.5.  Here the launch is nw shares x KVH workgroups and the WORK is cut evenly: the keys of all queries, in units of
// CH = WAVES * TPI keys (one full round of a workgroup), query after query, form one line of utot units; share w walks the units [w * utot / nw, (w + 1) * utot / nw)
// — a suffix of one query's keys, whole queries, a prefix of another — once per kv head: the KVH workgroups of a share read the same cache rows at the same time.
// A (query, kv head) pair that lies inside one share is written directly; a pair cut by share boundaries leaves one f32 partial per share (slot = share index -
// first share of the pair) and the LAST of its shares to finish merges them (the ticket scheme of FUSE above: sc1 partials, one counter per pair, nobody polls;
// merge_partitions: the same arithmetic).  Paged K/V through block tables whose block size is a power of two >= TPI (the scalar block-table form), nt loads.
// What bounds it is the stream of K and V; what kept it from that, and what stands against it here:
//  * a segment (one query's keys in one share) costs a start and a cross-wave merge of its own, about two units' time: every query is charged CHARGE units in
//    front of its keys, so that a share of many short queries holds fewer keys (27 sequences of 64..8100 keys 40.9 -> 38.7 us, 64 of 64..4096 54.5 -> 49.1;
//    one unit 39.1 / 51.9, four 39.0 / 50.7);
//  * one trip per round: a segment starts with two rounds requested and asks for the next one behind each (the block-table reload, which would make hipcc wait for everything at each
//    round, waits for itself).  For groups of 4 and 8 heads, whose arithmetic fills the time of a round, and heads of 64, whose rows are short, the requests are held in front of it (AHEAD); the
//    waves of smaller groups of 128 are at the memory's rate without, and requests held cost them 6 % of it;
//  * one share per CU: with those two, twice the shares only double the starts and merges (64 of 64..4096 keys: 49.1 us with one, 52.6 with two per CU).
// us a launch of 8 kv heads of 128, before these (one or two shares per CU, whichever is less) / with requests past a segment's end / now: 27 sequences of 64..8100 keys 43.3 / 35.9 / 35.1, 64 of
// 64..4096 59.7 / 47.4 / 45.0, 40 of 32..2000 28.0 / 21.0 / 21.0, 33 of 4000 84.9 / 90.8 / 83.6-86.5 (6.3 TB/s), 48 of 4000 117.4 / 124.6 / 117.9, 65 of 4000 159 / 172 / 160, 74 of 1500
// 74.2 / 79.8 / 75.5, 48 of 1500 50.2 / 50.4 / 48.9, 33 of 700 23.6 / 21.7 / 22.2.  Groups of 4, not AHEAD / AHEAD: 40 of 1500 keys 55.1 / 49.5, 33 of 4000 102.6 / 91.7, 27 of 64..8100
// 44.5 / 39.8; heads of 64, 4 kv heads, 66 of 4000 keys: groups of 8 111.4 / 98.3, of 4 74.1 / 60.5, of 2 63.0 / 45.4.
// QKN (27 sequences of 64 .. 8100 keys: a step of Qwen3-0.6B 1950 -> 1922 us): as in attn_rows_kernel, the step's own rows come raw; a segment's query heads (and key row, where it holds the query's last key) are formed when it is opened, behind its first requests.
template <int D, int G, int U, int WAVES, bool QKN = false>
__global__ __launch_bounds__(WAVES * 64) void attn_share_kernel(typename AttnParamsOf<QKN>::type own, int nq, int nw) {
    const AttnParams &p = own;
    static_assert(!QKN || (D == 128 && G < 4 * WAVES), "QKN: heads of 128");
    constexpr int LPR = D / 8, RPI = 64 / LPR, TPI = RPI * U, CH = TPI * WAVES;
    static_assert(G * D <= WAVES * 64 && G * (D / 4) <= WAVES * 64, "one pass over the (head, column) pairs");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int dc = lane % LPR, tg = lane / LPR;
    constexpr int CHARGE = 2;
    constexpr bool AHEAD = D == 64 || G >= 4;
    __shared__ int pre[1025];                               // pre[t] = units of the queries in front of t, their charges included
    __shared__ int cx[1024];                                // ctx_lens[t]
    __shared__ float sm_acc[WAVES][G][D];
    __shared__ float sm_ml[WAVES][G][2];
    __shared__ unsigned int ticket_s;
    if (wave == 0) {
        int base = 0;
        for (int k = 0; k < nq; k += 64) {
            const int t = k + lane;
            const int c = t < nq ? p.ctx_lens[t] : 0;
            int un = c > 0 ? (c + CH - 1) / CH + CHARGE : 0;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_up(un, o, 64); if (lane >= o) un += v; }
            if (t < nq) { pre[t + 1] = base + un; cx[t] = c; }
            base += __shfl(un, 63, 64);
        }
        if (lane == 0) pre[0] = 0;
    }
    __syncthreads();
    const int g = blockIdx.x % p.KVH, ws = blockIdx.x / p.KVH;
    const long long utot = pre[nq];
    // no more shares than units: behind a share without a unit the slots of a cut query would count a share that never draws its ticket (few queries with keys, many without)
    nw = (int)min((long long)nw, max(utot, 1ll));
    const long long ub = min(ws * utot / nw, utot), ue = min((ws + 1) * utot / nw, utot);
    // a query without keys owns no unit: its output row is zero, as in attn_rows_kernel (L == 0)
    for (int t0 = blockIdx.x; t0 < nq; t0 += gridDim.x)
        if (cx[t0] == 0)
            for (int x = threadIdx.x; x < p.H * D; x += WAVES * 64) p.out[(int64_t)t0 * p.H * D + x] = (half_t)0.f;
    long long u = ub;
    const int row_elems = p.KVH * D;

    // ---- state of the segment being streamed (set by `open`, which also REQUESTS its first K/V rows: a segment is opened under the tail of the one in front) ----
    int t = 0, np = 1, slot = 0, p0 = 0, pend = 0, R = 0, bt_chunk = -1, bt_reg = 0;
    const int32_t *bt = p.block_tables;
    half2_t qv[G][4];
    half8_t ka[U], va[U], kb[U], vb[U];                     // the wave's even / odd rounds: two are always requested ahead
    __shared__ half8_t own_lds[2][QKN ? (G + 1) * 16 : 1];  // (two: a wave may open the second segment while another still reads the first one's; behind it the tails' barriers stand between)
    half8_t own_k, own_v;
    int own_j = -1, opened = 0;                             // own_j: the segment's last key where it is the step's own row and has a slot
    auto block_base = [&](int tb) -> int64_t {              // element offset of (scalar token tb, kv head g, d = 0)
        const int bi = tb >> p.bs_shift, bo = tb & (p.block_size - 1);
        if ((bi >> 6) != bt_chunk) {
            bt_chunk = bi >> 6; const int idx = (bt_chunk << 6) + lane; bt_reg = idx < p.max_blocks ? bt[idx] : 0;
            asm volatile("" : "+v"(bt_reg));                // waited for HERE: at the readlane below hipcc would wait for every K/V request in flight, on every round
        }
        const int blk = __builtin_amdgcn_readlane(bt_reg, bi & 63);
        return (((int64_t)blk * p.block_size + bo) * p.KVH + g) * D;
    };
    // round r of the wave: a wave without keys asks for the segment's first row, and rows past the segment's end are its last row.  No branch stands around an AHEAD request (hipcc would then wait
    // for all that is in flight): past the wave's last round all its lanes ask for one 16-byte piece of that round, for all of it again they read 4 rounds too many per 66 of 4000 keys
    auto load_round = [&](int r, half8_t (&kk)[U], half8_t (&vv)[U]) {
        const int tb = R > 0 ? p0 + (min(r, R - 1) * WAVES + wave) * TPI : p0;
        const int64_t base = block_base(tb);
#pragma unroll
        for (int x = 0; x < U; ++x) {
            unsigned off = (unsigned)(min(x * RPI + tg, pend - 1 - tb) * row_elems + dc * 8);
            if (AHEAD) off &= r < R ? ~0u : 0u;
            kk[x] = load_row16<true>(p.k + base + off); vv[x] = load_row16<true>(p.v + base + off);
        }
    };
    // opens the next segment of the share, if there is one: the rest of a query's units, or as many as the share still holds
    auto open = [&]() -> bool {
        int lu = 0, seg = 0;
        for (;;) {
            if (u >= ue) return false;
            int lo = 0, hi = nq;                            // the query of unit u: the last t with pre[t] <= u (queries without keys own no unit)
            while (hi - lo > 1) { const int mid = (lo + hi) >> 1; if (pre[mid] <= u) lo = mid; else hi = mid; }
            t = lo;
            const int e = (int)min((long long)pre[t + 1], ue) - pre[t];
            lu = max((int)(u - pre[t]) - CHARGE, 0); seg = e - CHARGE - lu;
            u = pre[t] + e;
            if (seg > 0) break;                             // (else the share ends inside the query's charge)
        }
        // shares that touch this query's keys: unit x belongs to share floor(((x + 1) * nw - 1) / utot)
        const int wf = (int)(((pre[t] + CHARGE + 1ll) * nw - 1) / utot), wl = (int)(((long long)pre[t + 1] * nw - 1) / utot);
        np = wl - wf + 1; slot = ws - wf;
        p0 = lu * CH; pend = min(cx[t], (lu + seg) * CH);
        R = max(pend - p0 - wave * TPI + CH - 1, 0) / CH;   // rounds in which this wave has a key
        bt = p.block_tables + (int64_t)t * p.max_blocks;
        bt_chunk = (p0 >> p.bs_shift) >> 6;
        int64_t own_pos = 0; int own_slot = -1;
        if constexpr (QKN) { own_pos = own.pos[t]; own_slot = own.slots ? own.slots[t] : -1; }
        { const int idx = (bt_chunk << 6) + lane; bt_reg = idx < p.max_blocks ? bt[idx] : 0; asm volatile("" : "+v"(bt_reg)); }
        half8_t hx, hg; float4_t hc[2], hs[2];
        if constexpr (QKN) {
            const half_t *row = p.q + (int64_t)t * p.ldq;
            if (wave * 4 <= G) {
                const int hh = min(wave * 4 + tg, G);
                const int64_t at = own_pos * (D / 2) + (dc & 7) * 8;
                hx = *reinterpret_cast<const half8_t *>(row + (hh < G ? g * G + hh : p.H + g) * D + dc * 8);
                hg = *reinterpret_cast<const half8_t *>((hh < G ? own.qn_w : own.kn_w) + dc * 8);
#pragma unroll
                for (int x = 0; x < 2; ++x) { hc[x] = *reinterpret_cast<const float4_t *>(own.cos_t + at + 4 * x); hs[x] = *reinterpret_cast<const float4_t *>(own.sin_t + at + 4 * x); }
            }
            own_v = *reinterpret_cast<const half8_t *>(row + (p.H + p.KVH + g) * D + dc * 8);
        } else {
            const half_t *qrow = p.q + (int64_t)t * p.ldq + (int64_t)g * G * D + dc * 8;
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const half8_t h = *reinterpret_cast<const half8_t *>(qrow + i * D);
#pragma unroll
                for (int j = 0; j < 4; ++j) qv[i][j] = (half2_t){h[2 * j], h[2 * j + 1]};
            }
        }
        load_round(0, ka, va); load_round(1, kb, vb);
        if constexpr (QKN) {
            asm volatile("" ::: "memory");
            half8_t *lds = own_lds[opened & 1];
            if (wave * 4 <= G) {
                const half8_t o = norm_rotate_piece(hx, hg, hc, hs, own.qk_eps, dc);
                if (wave * 4 + tg <= G) lds[(wave * 4 + tg) * 16 + dc] = o;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const half8_t h = lds[i * 16 + dc];
#pragma unroll
                for (int j = 0; j < 4; ++j) qv[i][j] = (half2_t){h[2 * j], h[2 * j + 1]};
            }
            own_k = lds[G * 16 + dc];
            own_j = own_slot >= 0 && pend == cx[t] ? pend - 1 : -1;
            if (wave == WAVES - 1 && tg == 0 && own_j >= 0) {
                const int64_t dst = ((int64_t)own_slot * p.KVH + g) * D + dc * 8;
                *reinterpret_cast<half8_t *>(const_cast<half_t *>(p.k) + dst) = own_k;
                *reinterpret_cast<half8_t *>(const_cast<half_t *>(p.v) + dst) = own_v;
            }
            ++opened;
        }
        asm volatile("" ::: "memory");                      // the requests stay HERE: hipcc would sink them to their first use, behind the tail of the segment in front
        return true;
    };

    bool more = open();
    while (more) {
        float m[G], l[G], acc[G][8];
#pragma unroll
        for (int i = 0; i < G; ++i) {
            m[i] = -INFINITY; l[i] = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[i][j] = 0.f;
        }
        auto process = [&](half8_t (&kk)[U], half8_t (&vv)[U], int r) {
            const int left = pend - p0 - (r * WAVES + wave) * TPI;      // keys of the segment from the round's first one on
            if (QKN && own_j >= 0 && left <= TPI)                       // the round that holds the step's own row (and, clamped to it, rows past the segment's end)
#pragma unroll
                for (int x = 0; x < U; ++x)
                    if (x * RPI + tg >= left - 1) { kk[x] = own_k; vv[x] = own_v; }
            float sc[U][G];
#pragma unroll
            for (int x = 0; x < U; ++x) {
                const bool valid = x * RPI + tg < left;
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    float d = 0.f;
#pragma unroll
                    for (int j = 0; j < 4; ++j) d = dot2((half2_t){kk[x][2 * j], kk[x][2 * j + 1]}, qv[i][j], d);
                    d = row_sum<LPR>(d);
                    sc[x][i] = valid ? d * p.scale : -INFINITY;
                }
            }
#pragma unroll
            for (int i = 0; i < G; ++i) {
                float mx = sc[0][i];
#pragma unroll
                for (int x = 1; x < U; ++x) mx = fmaxf(mx, sc[x][i]);
                const float mn = fmaxf(m[i], mx);
                const float ms = (mn == -INFINITY) ? 0.f : mn;
                const float alpha = __expf(m[i] - ms);
                m[i] = mn;
                float ps = 0.f;
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[i][j] *= alpha;
#pragma unroll
                for (int x = 0; x < U; ++x) {
                    const float pr = __expf(sc[x][i] - ms);
                    ps += pr;
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[i][j] = fmaf(pr, (float)vv[x][j], acc[i][j]);
                }
                l[i] = __fmaf_rn(l[i], alpha, ps);
            }
        };
        for (int r = 0; r < R; r += 2) {
            process(ka, va, r);
            if (r + 1 >= R) break;
            if (AHEAD || r + 2 < R) load_round(r + 2, ka, va);
            if (AHEAD) { asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); }   // the requests stay in front of the other round's arithmetic
            process(kb, vb, r + 1);
            if (AHEAD || r + 3 < R) load_round(r + 3, kb, vb);
            if (AHEAD) { asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); }
        }

        // the segment is in the accumulators: what its tail needs of the state, then the NEXT segment is opened (its query, block table and first K/V rows
        // are on their way while this one is merged and handed over)
        const int st = t, snp = np, sslot = slot;
        more = open();

        // row-group slots of the wave -> the wave's sums; waves -> the segment's partial (attn_rows_kernel's arithmetic)
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const float M = groups_max<LPR>(m[i]);
            const float w = (m[i] == -INFINITY) ? 0.f : __expf(m[i] - M);
            l[i] = groups_sum<LPR>(l[i] * w);
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[i][j] = groups_sum<LPR>(acc[i][j] * w);
            if (tg == 0) {
#pragma unroll
                for (int j = 0; j < 8; ++j) sm_acc[wave][i][dc * 8 + j] = acc[i][j];
                if (dc == 0) { sm_ml[wave][i][0] = M; sm_ml[wave][i][1] = l[i]; }
            }
        }
        __syncthreads();
        const int64_t pair0 = ((int64_t)st * p.H + (int64_t)g * G) * p.num_parts;
        const auto rs_o = __builtin_amdgcn_make_buffer_rsrc(p.part_o + pair0 * D, 0, (int)(G * p.num_parts * D * 4), 0x00020000);
        const auto rs_ml = __builtin_amdgcn_make_buffer_rsrc(p.part_ml + pair0 * 2, 0, (int)(G * p.num_parts * 2 * 4), 0x00020000);
        if (threadIdx.x < G * D) {
            const int i = threadIdx.x / D, d = threadIdx.x % D;
            float M = sm_ml[0][i][0];
#pragma unroll
            for (int w2 = 1; w2 < WAVES; ++w2) M = fmaxf(M, sm_ml[w2][i][0]);
            float o = 0.f, L = 0.f;
#pragma unroll
            for (int w2 = 0; w2 < WAVES; ++w2) {
                const float mw = sm_ml[w2][i][0];
                const float wgt = (mw == -INFINITY) ? 0.f : __expf(mw - M);
                o = mul_then_add(wgt, sm_acc[w2][i][d], o);
                L = mul_then_add(wgt, sm_ml[w2][i][1], L);
            }
            if (snp == 1) {
                p.out[((int64_t)st * p.H + g * G + i) * D + d] = (half_t)(L > 0.f ? o / L : 0.f);
            } else {
                const int sl = i * p.num_parts + sslot;
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), rs_o, (sl * D + d) * 4, 0, 16);
                if (d == 0) { __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(M), rs_ml, sl * 8, 0, 16);
                              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(L), rs_ml, sl * 8 + 4, 0, 16); }
            }
        }
        if (snp > 1) {                                                        // (workgroup-uniform)
            constexpr int TPH = D / 4;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                  // every storing wave drains its stores (and the next segment's first rows land) ...
            __syncthreads();
            unsigned int *cnt = p.tickets + (int64_t)st * p.KVH + g;
            if (threadIdx.x == 0) ticket_s = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // ... one ticket
            __syncthreads();
            if (ticket_s == (unsigned)(snp - 1)) {                            // the last of the pair's shares to finish merges it
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");        // keeps the sc1 loads below the ticket
                if (threadIdx.x < G * TPH) {
                    const int i = threadIdx.x / TPH, d = (threadIdx.x % TPH) * 4;
                    const half4_t hv = merge_partitions(snp,
                        [&](int pi) { return __builtin_bit_cast(float2_t, __builtin_amdgcn_raw_buffer_load_b64(rs_ml, (i * p.num_parts + pi) * 8, 0, 16)); },
                        [&](int pi) { return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(rs_o, ((i * p.num_parts + pi) * D + d) * 4, 0, 16)); });
                    *reinterpret_cast<half4_t *>(p.out + ((int64_t)st * p.H + g * G + i) * D + d) = hv;
                }
                if (threadIdx.x == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // re-arm for the next launch
            }
        }
        __syncthreads();                                                      // sm_acc / sm_ml / ticket_s are the next segment's too
    }
}

// ---- launch configuration ------------------------------------------------------------------------
static int share_mode() { static const int v = getenv("NVR_ATTN_SHARE") ? atoi(getenv("NVR_ATTN_SHARE")) : 1; return v; }   // 0: never, 1: by the rule, 2: whenever it can run (probes)
static bool share_enabled() { return share_mode() != 0; }
static int share_workgroups() {                                           // one workgroup per CU of the current device
    static const int v = [] { int dev = 0, n = 0; if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256; return n; }();
    return v;
}
static inline int parts_for(int64_t nq, int64_t KVH, int64_t max_ctx, int waves, int *part_size) {
    // aim at ~4096 waves over the 256 CUs; partitions are multiples of 64 tokens
    const int64_t want_wgs = 4096 / waves;
    int64_t want = (want_wgs + nq * KVH - 1) / (nq * KVH);
    int64_t max_parts = (max_ctx + 63) / 64;
    if (want > max_parts) want = max_parts;
    if (want < 1) want = 1;
    int64_t ps = ((max_ctx + want - 1) / want + 63) / 64 * 64;
    if (ps < 64) ps = 64;
    *part_size = (int)ps;
    return (int)((max_ctx + ps - 1) / ps);
}

// Longest context of up to 128 pairs that one workgroup per pair takes without partitions: a round of 128 keys and half a chunk.  A second round costs more than the partitions' hand-off
// does from about 144 keys on while there are enough CUs for the partitions; from 129 pairs on the partitions fill the chip more than once and it pays up to 256 keys.  Groups of 8 merge
// for longer than they stream.  Qwen3-0.6B (8 kv heads), us a step in partitions / without: 1 sequence of 128 keys 728 / 716, 136 735 / 734, 144 741 / 739, 152 740 / 754, 201 736 / 778;
// 4 sequences of 128 816 / 786, 201 822 / 853; 16 of 128 932 / 881, 251 952 / 973; 17 of 251 1026 / 995, 23 1080 / 1044.  8 groups of 4 heads, us a launch: 128 keys 6.3 / 6.1, 140 6.7 / 6.9;
// of 8 heads: 128 keys 9.0 / 10.1
int64_t attn_brief_context(int64_t nq, int64_t H, int64_t KVH) { return nq * KVH <= 128 && H <= 4 * KVH ? 136 : 0; }

size_t attn_workspace_bytes(int64_t nq, int64_t H, int64_t D, int64_t max_ctx) {
    int64_t max_parts = (max_ctx + 63) / 64;
    if (max_parts > 1024) max_parts = 1024;
    if (max_parts < 1) max_parts = 1;
    return (size_t)(nq * H * max_parts * (D + 2) * sizeof(float));
}

// ---- a batch behind one shared prefix, in one launch --------------------------------------------------------------
// A workgroup takes the G query heads of a kv head for NS sequences: its eight waves walk the shared keys in chunks of 32 on the matrix cores, every query row of the workgroup on one column
// (S^T = K Q^T, O^T += V^T P^T, both operands through a wave's own LDS image: fragments straight from the pages would be 16 rows x 64 bytes a request, whose lanes' addresses take four times as long), then 8 / NS waves walk each sequence's own keys as attn_rows_kernel
// does; all of a row's partials meet in LDS.  Against a launch for the shared keys and one for the own ones (flash_shared_prefix, SHM) there is one start-up, no partials in memory, and no merge of
// them: a workgroup reads the shared keys again (from its XCD's L2), which is what bounds the launch beside the own keys: 512 bytes a key and workgroup at 82 GB/s.
// The weights of shared keys are rounded to 16 bits for the product as there, their sum is that of the rounded weights; own keys' weights stay in f32.
constexpr int PRE_CH = 32, PRE_VS = 128 * 2 + 32, PRE_OS = 128 + 4;        // keys of a chunk; bytes of an image row, f32 numbers of a partial row (conflict-free strides)
template <int G, int NS>
constexpr size_t prefix_lds() { return std::max<size_t>((size_t)8 * PRE_CH * PRE_VS, ((size_t)8 * G * NS + 8 * G) * PRE_OS * 4); }
template <int G, int NS>
__global__ __launch_bounds__(512) void attn_prefix_kernel(AttnParams p, int nq, int shared_len) {
    constexpr int D = 128, R = G * NS, WPS = 8 / NS, U = 4;
    static_assert(R <= 16 && 8 % NS == 0, "the rows of a workgroup are columns of one product");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    __shared__ float sh_ml[8][R][2], own_ml[8][G][2];
    const int g = blockIdx.x % p.KVH, t0 = (blockIdx.x / p.KVH) * NS;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lm = lane & 15, lq = lane >> 4;
    const float scale2 = p.scale * 1.44269504088896340736f;
    const int row_elems = p.KVH * D;
    // this wave's sequence: its block table from the shared keys on, its length, its queries for the own keys (lm: the lane's 16-byte piece, lq: its row of a group of four)
    const int ts = min(t0 + wave / WPS, nq - 1), wsub = wave % WPS;
    const int32_t *bt = p.block_tables + (int64_t)ts * p.max_blocks;
    const int b0 = shared_len >> p.bs_shift;
    int bt_base = b0, bt_reg = bt[min(b0 + lane, p.max_blocks - 1)];
    const int ctx = p.ctx_lens[ts];
    half2_t qv[G][4];
    {
        const half_t *q = p.q + (int64_t)ts * p.ldq + (int64_t)g * G * D + lm * 8;
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const half8_t h = *reinterpret_cast<const half8_t *>(q + i * D);
#pragma unroll
            for (int j = 0; j < 4; ++j) qv[i][j] = (half2_t){h[2 * j], h[2 * j + 1]};
        }
    }
    half8_t qf[4];                                                            // column lm of the products: row lm of the workgroup (the columns behind the last repeat it)
    {
        const int r = min(lm, R - 1), t = min(t0 + r / G, nq - 1);
        const half_t *q = p.q + (int64_t)t * p.ldq + (int64_t)(g * G + r % G) * D + lq * 8;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) qf[ks] = *reinterpret_cast<const half8_t *>(q + ks * 32);
    }
    auto block_row = [&](int tok) -> int64_t {                                // cache row of a key of this sequence's own blocks (uniform)
        const int bi = tok >> p.bs_shift;
        if (bi >= bt_base + 64) { bt_base = bi; bt_reg = bt[min(bi + lane, p.max_blocks - 1)]; }
        return (int64_t)__builtin_amdgcn_readlane(bt_reg, bi - bt_base) * p.block_size + (tok & (p.block_size - 1));
    };
    const int ngroups = (max(ctx - shared_len, 0) + 3) >> 2;                  // groups of four own keys, dealt to the sequence's waves in turn
    half8_t kk[U], vv[U];
    auto request_own = [&](int first) {                                       // groups first, first + WPS, ..
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int tok = shared_len + (min(first + u * WPS, ngroups - 1) << 2);
            const int64_t at = (block_row(tok) + min(lq, ctx - 1 - tok)) * row_elems + g * D + lm * 8;
            kk[u] = load_row16<true>(p.k + at); vv[u] = load_row16<true>(p.v + at);
        }
    };
    if (wsub < ngroups) request_own(wsub);
    // ---- shared keys
    char *img = smem + wave * PRE_CH * PRE_VS;
    float m = -INFINITY, l = 0.f;
    float4_t o[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) o[t] = (float4_t){0.f, 0.f, 0.f, 0.f};
    half8_t kx[8], vx[8];                                                     // a chunk as it comes from the pages: row 4 i + lq, 16-byte piece lm
    auto request_shared = [&](int x) {
        const int base = x * PRE_CH;
        const int64_t row0 = (int64_t)p.block_tables[base >> p.bs_shift] * p.block_size + (base & (p.block_size - 1));
        const int64_t at = (row0 + lq) * row_elems + g * D + lm * 8;
#pragma unroll
        for (int u = 0; u < 8; ++u) kx[u] = *reinterpret_cast<const half8_t *>(p.k + at + u * 4 * row_elems);
#pragma unroll
        for (int u = 0; u < 8; ++u) vx[u] = *reinterpret_cast<const half8_t *>(p.v + at + u * 4 * row_elems);
    };
    const int chunks = shared_len / PRE_CH;
    if (wave < chunks) request_shared(wave);
    for (int x = wave; x < chunks; x += 8) {
        half8_t kf[2][4];
#pragma unroll
        for (int u = 0; u < 8; ++u) { const int row = 4 * u + lq; *reinterpret_cast<half8_t *>(img + row * 256 + ((lm ^ (row & 15)) << 4)) = kx[u]; }
        asm volatile("" ::: "memory");                                        // (a wave's LDS requests are served in order: what is written is read behind it, and written again behind that)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) kf[mt][ks] = *reinterpret_cast<const half8_t *>(img + (mt * 16 + lm) * 256 + (((ks * 4 + lq) ^ lm) << 4));
        asm volatile("" ::: "memory");
#pragma unroll
        for (int u = 0; u < 8; ++u) *reinterpret_cast<half8_t *>(img + (4 * u + lq) * PRE_VS + lm * 16) = vx[u];
        asm volatile("" ::: "memory");
        if (x + 8 < chunks) request_shared(x + 8);
        float4_t s[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
            s[mt] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) s[mt] = mfma16(kf[mt][ks], qf[ks], s[mt]);
        }
        float mx = -INFINITY;                                                 // scores of row lm: keys base + mt * 16 + lq * 4 + e
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int e = 0; e < 4; ++e) { s[mt][e] *= scale2; mx = fmaxf(mx, s[mt][e]); }
        mx = xor32_partner_max(xor16_partner_max(mx));
        const float mn = fmaxf(m, mx), ms = mn == -INFINITY ? 0.f : mn, alpha = __builtin_amdgcn_exp2f(m - ms);      // (only keys of score -inf so far: weights of 0)
        const bool moved = mn != m;
        m = mn;
        half8_t pf;
        float rs = 0.f;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int e = 0; e < 4; ++e) { const half_t w = (half_t)__builtin_amdgcn_exp2f(s[mt][e] - ms); rs += (float)w; pf[mt * 4 + e] = w; }
        l = fmaf(l, alpha, rs);
        if (__any(moved)) {
#pragma unroll
            for (int t = 0; t < 8; ++t) o[t] *= alpha;
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const char *at = img + (lq * 4 + (lm >> 2)) * PRE_VS + t * 32 + (lm & 3) * 8;
            const half4_t a0 = lds_read_tr16(at), a1 = lds_read_tr16(at + 16 * PRE_VS);
            o[t] = mfma16(__builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7), pf, o[t]);
        }
        asm volatile("" ::: "memory");
    }
    // ---- own keys
    float om[G], ol[G], acc[G][8];
#pragma unroll
    for (int i = 0; i < G; ++i) {
        om[i] = -INFINITY; ol[i] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = 0.f;
    }
    for (int first = wsub; first < ngroups; first += WPS * U) {
        float sc[U][G];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool valid = first + u * WPS < ngroups && shared_len + ((first + u * WPS) << 2) + lq < ctx;
#pragma unroll
            for (int i = 0; i < G; ++i) {
                float d = 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j) d = dot2((half2_t){kk[u][2 * j], kk[u][2 * j + 1]}, qv[i][j], d);
                sc[u][i] = valid ? row_sum<16>(d) * scale2 : -INFINITY;
            }
        }
#pragma unroll
        for (int i = 0; i < G; ++i) {
            float mx = sc[0][i];
#pragma unroll
            for (int u = 1; u < U; ++u) mx = fmaxf(mx, sc[u][i]);
            const float mn = fmaxf(om[i], mx), ms = mn == -INFINITY ? 0.f : mn, alpha = __builtin_amdgcn_exp2f(om[i] - ms);
            om[i] = mn;
            float ps = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[i][j] *= alpha;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float pr = __builtin_amdgcn_exp2f(sc[u][i] - ms);
                ps += pr;
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[i][j] = fmaf(pr, (float)vv[u][j], acc[i][j]);
            }
            ol[i] = fmaf(ol[i], alpha, ps);
        }
        if (first + WPS * U < ngroups) request_own(first + WPS * U);
    }
    // ---- partials of every row: [wave][row] of the shared keys, [wave][head] of the own ones
    l = xor32_partner_sum(xor16_partner_sum(l));
    __syncthreads();                                                          // every wave is done with its image
    float *sh_o = reinterpret_cast<float *>(smem), *own_o = sh_o + 8 * R * PRE_OS;
    if (lm < R) {
#pragma unroll
        for (int t = 0; t < 8; ++t) *reinterpret_cast<float4_t *>(sh_o + (wave * R + lm) * PRE_OS + t * 16 + lq * 4) = o[t];
        if (lq == 0) { sh_ml[wave][lm][0] = m; sh_ml[wave][lm][1] = l; }
    }
#pragma unroll
    for (int i = 0; i < G; ++i) {
        const float M = xor32_partner_max(xor16_partner_max(om[i])), w = om[i] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(om[i] - M);
        const float L = xor32_partner_sum(xor16_partner_sum(ol[i] * w));
        float4_t a[2];
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j >> 2][j & 3] = xor32_partner_sum(xor16_partner_sum(acc[i][j] * w));
        if (lq == 0) {
            float *at = own_o + (wave * G + i) * PRE_OS + lm * 8;
            *reinterpret_cast<float4_t *>(at) = a[0]; *reinterpret_cast<float4_t *>(at + 4) = a[1];
            if (lm == 0) { own_ml[wave][i][0] = M; own_ml[wave][i][1] = L; }
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < R * (D / 4); idx += 512) {
        const int r = idx / (D / 4), c = (idx % (D / 4)) * 4, sq = r / G, i = r % G;
        if (t0 + sq >= nq) continue;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < 8; ++w) M = fmaxf(M, sh_ml[w][r][0]);
#pragma unroll
        for (int w = 0; w < WPS; ++w) M = fmaxf(M, own_ml[sq * WPS + w][i][0]);
        float4_t v = {0.f, 0.f, 0.f, 0.f};
        float L = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            const float f = __builtin_amdgcn_exp2f(sh_ml[w][r][0] - M);      // (a wave without a chunk: 2^-inf = 0)
            v += *reinterpret_cast<const float4_t *>(sh_o + (w * R + r) * PRE_OS + c) * f;
            L = fmaf(sh_ml[w][r][1], f, L);
        }
#pragma unroll
        for (int w = 0; w < WPS; ++w) {
            const float f = __builtin_amdgcn_exp2f(own_ml[sq * WPS + w][i][0] - M);
            v += *reinterpret_cast<const float4_t *>(own_o + ((sq * WPS + w) * G + i) * PRE_OS + c) * f;
            L = fmaf(own_ml[sq * WPS + w][i][1], f, L);
        }
        half4_t hv;
#pragma unroll
        for (int e = 0; e < 4; ++e) hv[e] = (half_t)(L > 0.f ? v[e] / L : 0.f);      // (as merge_partitions: no key of a finite score, or NaN among them)
        *reinterpret_cast<half4_t *>(p.out + ((int64_t)(t0 + sq) * p.H + g * G + i) * D + c) = hv;
    }
}

template <int D, int G, int U, int WAVES, bool NT>
static void launch_cfg(const AttnParams &p, bool paged, bool direct, int64_t nwg, hipStream_t s, bool fuse = false, bool shm = false, const OwnRows *own = nullptr) {
    dim3 grid((unsigned)nwg), block(WAVES * 64);
    if constexpr (D == 128 && G <= 4 && WAVES >= 4 && NT)
        if (own) {
            const AttnParamsOwn po{p, *own};
            if (direct) attn_rows_kernel<D, G, true, true, U, WAVES, NT, true, false, false, true><<<grid, block, 0, s>>>(po);
            else attn_rows_kernel<D, G, true, false, U, WAVES, NT, true, true, false, true><<<grid, block, 0, s>>>(po);
            return;
        }
    constexpr int TPI = 64 / (D / 8) * U;
    const bool ub = paged && p.block_size % TPI == 0 && (p.num_parts == 1 || p.part_size % TPI == 0);
    if constexpr (WAVES <= 4 && NT) {                                     // (only instantiated where launch_attn can ask for it)
        if (shm) {                                                        // (paged, split, every query behind the shared prefix: launch_attn)
            if (ub) attn_rows_kernel<D, G, true, false, U, WAVES, NT, true, false, true><<<grid, block, 0, s>>>(p);
            else attn_rows_kernel<D, G, true, false, U, WAVES, NT, false, false, true><<<grid, block, 0, s>>>(p);
            return;
        }
    }
    if constexpr (NT) {                                                   // the cache through block tables (every paged call site streams: nt loads)
        if (ub) {
            if (direct) attn_rows_kernel<D, G, true, true, U, WAVES, NT, true><<<grid, block, 0, s>>>(p);
            else if (fuse) attn_rows_kernel<D, G, true, false, U, WAVES, NT, true, true><<<grid, block, 0, s>>>(p);
            else attn_rows_kernel<D, G, true, false, U, WAVES, NT, true><<<grid, block, 0, s>>>(p);
        } else if (paged) {
            if (direct) attn_rows_kernel<D, G, true, true, U, WAVES, NT, false><<<grid, block, 0, s>>>(p);
            else if (fuse) attn_rows_kernel<D, G, true, false, U, WAVES, NT, false, true><<<grid, block, 0, s>>>(p);
            else attn_rows_kernel<D, G, true, false, U, WAVES, NT, false><<<grid, block, 0, s>>>(p);
        }
    } else {                                           // contiguous K / V (prefill): rows re-read from L2, 4-wave workgroups only
        if (direct) attn_rows_kernel<D, G, false, true, U, WAVES, NT, false><<<grid, block, 0, s>>>(p);
        else attn_rows_kernel<D, G, false, false, U, WAVES, NT, false><<<grid, block, 0, s>>>(p);
    }
}

static int own_rows(const AttnArgs &a, hipStream_t s) {                    // what QKN does inside the attention, by the launch of its own
    if (!a.qn_w) return 0;
    return rope_store_kv(const_cast<half_bits *>(a.q), a.pos, a.slots, a.nq, a.H, a.KVH, a.D, a.cos_t, a.sin_t, const_cast<half_bits *>(a.k), const_cast<half_bits *>(a.v), s, a.qn_w, a.kn_w, a.qk_eps);
}

static bool own_rows_aligned(const AttnArgs &a) {
    return a.qn_w && a.ldq % 8 == 0 && (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.qn_w | (uintptr_t)a.kn_w | (uintptr_t)a.cos_t | (uintptr_t)a.sin_t) & 15) == 0;
}
static OwnRows own_rows_params(const AttnArgs &a) { return OwnRows{(const half_t *)a.qn_w, (const half_t *)a.kn_w, a.qk_eps, a.pos, a.slots, a.cos_t, a.sin_t}; }

// A whole batch behind its prefix in one launch or two.  One: as many sequences a workgroup (NS: 1, 2, 4 or 8) as give every CU one workgroup.  It saves the second launch (5 us) and has no partials in
// memory, but every workgroup reads the shared keys (256 of them 1.6 us, 0.5-0.85 in the launch of their own), and a sequence's own keys are walked by 8 / NS waves, where the two launches give each pair four and
// cut long ones over the idle CUs: the longest sequence is waited for.  So the bound on its own keys goes by NS, a little further where all are long (then the bytes count on either side), half as far
// (NS 4 and 8: three quarters) beyond 512 shared keys: over 2520 shapes the choice is 0.5 % above the better of the two, one launch throughout 14.6 %, two 14.4 %.  us a launch, two / one, groups of 2 of 8 kv heads behind 512 keys; all of so many own keys; one of them among 15:
//   16 sequences (NS 1) 256 own 19.0 / 15.0, 512 21.1 / 19.6, 1000 behind 256 23.9 / 29.7; one of 2000 behind 256 27.6 / 48.4
//   33 (NS 2) 64 14.5 / 11.2, 192 18.5 / 17.2, 256 20.4 / 20.2; one of 192 14.6 / 14.9, of 256 15.7 / 17.5
//   64 (NS 2) 64 16.8 / 11.8, 256 25.6 / 21.3; one of 192 16.3 / 15.2, of 256 17.2 / 17.6, of 2000 behind 256 47 / 87
//   65 (NS 4) 64 17.3 / 14.0, 128 21.1 / 19.8, 192 24.8 / 25.8; one of 96 16.4 / 14.8, of 128 16.1 / 17.3, of 256 17.2 / 27.5
//   128 (NS 4) 64 20.0 / 14.6, 192 31.4 / 27.1; one of 128 17.4 / 17.4, of 192 17.7 / 22.5
//   129 (NS 8) 64 20.7 / 19.7, 128 27.0 / 31.5; one of 64 18.5 / 17.2, of 96 18.6 / 22.0
//   256 (NS 8) 64 25.4 / 21.1, 128 35.2 / 33.8; one of 64 19.2 / 17.5, of 96 19.5 / 22.2
// and behind 1024: 33 of 96 17.2 / 16.5, of 192 18.8 / 20.3; 128 of 64 21.3 / 17.9, one of 128 19.2 / 20.1.  Below 32 pairs the launch of the shared keys is cut over idle CUs too: 2 sequences of 2 kv
// heads behind 512, 75 own 11.4 / 9.3, 250 11.8 / 12.8, behind 1024, 75 own 12.4 / 13.0.
int32_t attn_prefix_launches(int64_t nq, int64_t H, int64_t KVH, int64_t shared_len, int64_t longest, int64_t mean) {
    const int64_t G = H / std::max<int64_t>(KVH, 1), pairs = nq * KVH, cus = share_workgroups(), prefix = pairs < 32 ? 2 * shared_len : shared_len;
    if (prefix > 1024 || pairs > cus * (G <= 2 ? 8 : 4)) return 2;
    const int64_t bound = pairs <= cus ? (pairs < 96 ? 256 : 384) : pairs <= 2 * cus ? std::min<int64_t>(192 + mean / 2, 256) : pairs <= 4 * cus ? 96 + mean / 2 : 64;
    return longest <= (prefix <= 512 ? bound : pairs <= 2 * cus ? bound / 2 : bound * 3 / 4) ? 1 : 2;
}
static bool prefix_in_one_launch(const AttnArgs &a) {
    return !a.shared_rows && (a.block_size & (a.block_size - 1)) == 0 && a.block_size % 64 == 0 && a.ldq % 8 == 0 && (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.out) & 15) == 0 &&
           (int64_t)a.nq * a.KVH <= (int64_t)share_workgroups() * (a.H / a.KVH <= 2 ? 8 : 4) &&
           (a.prefix_launches ? a.prefix_launches : attn_prefix_launches(a.nq, a.H, a.KVH, a.shared_len, a.max_ctx - a.shared_len, 0)) == 1;
}
template <int G, int NS>
static int launch_prefix(const AttnParams &p, int nq, int shared_len, hipStream_t s) {
    if (int rc = attn_prepare()) return rc;                                   // (callers without a runner)
    attn_prefix_kernel<G, NS><<<dim3((unsigned)((nq + NS - 1) / NS * p.KVH)), dim3(512), prefix_lds<G, NS>(), s>>>(p, nq, shared_len);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "attention (shared prefix) launch failed: %s", hipGetErrorString(e));
    return 0;
}

// Whether a decode step's attention takes the output product along (OUTP): no more workgroups than CUs (two on a CU wait for each other's registers: 4 sequences of 128 keys 767 / 835 us a step), which 128 rows a workgroup
// allow twice as many sequences as 64, and contexts of up to two rounds of keys, since every workgroup of a pair walks all of them; four sequences, which each have 128 rows' workgroups, of one round only.
// Qwen3-0.6B, us a step whose keys are new to the caches, two launches / one, float16: 1 sequence of 40 keys 667 / 630, 128 699 / 672, 200 708 / 699, 254 743 / 731; 2 of 40 701 / 662, 128 723 / 706,
// 254 771 / 770; 3 of 128 746 / 730, 254 796 / 796; 4 of 40 743 / 729, 128 772 / 766, 254 822 / 834; with q / k norms (bfloat16) 1 of 40 677 / 643, 200 711 / 693, 254 733 / 724; 2 of 40 723 / 693, 128
// 736 / 716, 254 781 / 787; 3 of 128 749 / 736, 254 794 / 794; 4 of 40 771 / 754, 128 783 / 779, 254 832 / 839.  (The same step again and again, whose keys the last-level cache holds, gains more:
// 1 of 128 694 / 645, 4 of 255 with norms 797 / 761.)
bool attn_out_rides(int64_t nq, int64_t H, int64_t KVH, int64_t D, int64_t N, int64_t max_ctx) {
    if (KVH <= 0 || H % KVH || nq > 4 || max_ctx > (nq < 4 ? 256 : attn_brief_context(nq, H, KVH)) || nq * KVH * (N / (N % 128 ? 64 : 128)) > share_workgroups()) return false;
    const int64_t G = H / KVH;
    return (D == 64 || D == 128) && (G == 1 || G == 2 || G == 4) && (KVH == 2 || KVH == 4 || KVH == 8) && N % OUT_ROWS == 0;
}
template <int D, int G, int R>
static int launch_attn_out_rows(const AttnArgs &a, AttnParamsOut &p, hipStream_t s) {
    constexpr int U = D == 128 ? 4 : 2, TPI = 64 / (D / 8) * U;
    const dim3 grid((unsigned)(a.nq * a.KVH), (unsigned)(a.out_n / R));
    const bool ub = a.block_size % TPI == 0;
    bool in_it = false;
    if constexpr (D == 128)
        if (ub && own_rows_aligned(a)) {
            static_cast<OwnRows &>(p) = own_rows_params(a);
            attn_rows_kernel<D, G, true, true, U, 8, false, true, false, false, true, R><<<grid, dim3(512), 0, s>>>(p);
            in_it = true;
        }
    if (!in_it) {
        if (int rc = own_rows(a, s)) return rc;
        if (ub) attn_rows_kernel<D, G, true, true, U, 8, false, true, false, false, false, R><<<grid, dim3(512), 0, s>>>(p);
        else attn_rows_kernel<D, G, true, true, U, 8, false, false, false, false, false, R><<<grid, dim3(512), 0, s>>>(p);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "attention + output product launch failed: %s", hipGetErrorString(e));
    return 0;
}

template <int D, int G>
static int launch_attn_out(const AttnArgs &a, hipStream_t s) {
    if (!attn_out_rides(a.nq, a.H, a.KVH, D, a.out_n, a.max_ctx) || a.shared_len > 0 || a.seq_of_q || ((uintptr_t)a.out_w & 15))
        return nvr::fail(NVR_ERR_INVALID_ARG, "attention + output product: %d queries, %d / %d heads of %d, %d columns, contexts up to %d", a.nq, a.H, a.KVH, D, a.out_n, a.max_ctx);
    AttnParamsOut p{};
    p.q = (const half_t *)a.q; p.ldq = a.ldq; p.k = (const half_t *)a.k; p.v = (const half_t *)a.v;
    p.ctx_lens = a.ctx_lens; p.block_tables = a.block_tables; p.max_blocks = a.max_blocks; p.block_size = a.block_size;
    p.bs_shift = (a.block_size > 0 && (a.block_size & (a.block_size - 1)) == 0) ? __builtin_ctz(a.block_size) : -1;
    p.H = a.H; p.KVH = a.KVH; p.scale = a.scale; p.part_size = 0x3fffffff; p.num_parts = 1;
    p.w = (const half_t *)a.out_w; p.slabs = a.out_slabs; p.stride = (int64_t)a.nq * a.out_n; p.N = a.out_n;
    const int64_t pairs = (int64_t)a.nq * a.KVH;
    if (pairs * (a.out_n / OUT_ROWS) > share_workgroups() && a.out_n % 128 == 0) return launch_attn_out_rows<D, G, 128>(a, p, s);
    return launch_attn_out_rows<D, G, 64>(a, p, s);
}

template <int D, int G>
static int launch_attn(const AttnArgs &a, bool paged, hipStream_t s) {
    if constexpr (G <= 4)
        if (paged && a.out_w) return launch_attn_out<D, G>(a, s);
    AttnParams p{};
    p.q = (const half_t *)a.q; p.ldq = a.ldq; p.k = (const half_t *)a.k; p.v = (const half_t *)a.v; p.ldkv = a.ldkv;
    p.ctx_lens = a.ctx_lens; p.seq_of_q = a.seq_of_q; p.kv_base = a.kv_base; p.block_tables = a.block_tables;
    p.max_blocks = a.max_blocks; p.block_size = a.block_size;
    p.bs_shift = (a.block_size > 0 && (a.block_size & (a.block_size - 1)) == 0) ? __builtin_ctz(a.block_size) : -1;
    p.H = a.H; p.KVH = a.KVH; p.scale = a.scale; p.out = (half_t *)a.out;
    constexpr int DU = (D == 128) ? 4 : 2;           // default: 16 tokens per wave iteration
    // Geometry (measured on MI355X at B=32, ctx 1044, KVH=8, D=128, profiles/r01_attn_tune.txt): one 8-wave
    // workgroup per (query, kv head) = one per CU, each wave with 2 row groups of K and of V in flight (32 KiB per
    // CU), non-temporal loads and no split (23.6 us, 5.8 TB/s) beats 16 waves x 4 groups (25.0 us: more bytes in
    // flight per CU is slower, as for a plain streaming read) and 4-wave workgroups over 4 partitions + merge
    // kernel (29.6 us).  So: when there is enough work for >= ~192 such workgroups use them (splitting only to reach
    // ~256 workgroups), otherwise fall back to 4-wave workgroups over 64-token-granular partitions.
    const int64_t mc = a.max_ctx > 0 ? a.max_ctx : 1;
    const int64_t pairs = (int64_t)a.nq * a.KVH;
    // 8-wave workgroups whenever ~256 of them can be given >= 64 tokens each; with fewer than ~192 (query, kv head) pairs
    // (small batches, tensor-parallel ranks that hold 1-4 kv heads) the context is cut into ceil(256 / pairs)
    // 64-token-granular partitions + merge kernel (B=32, ctx 1044: KVH=1 10.9 us vs 14.6 us for the 4-wave path, KVH=2
    // 12.7 vs 14.6, KVH=4 17.5 vs 19.7; scratch/attn_tp_shape.py)
    int waves = (paged && a.workspace && pairs * ((mc + 63) / 64) >= 256) ? 8 : 4;
    // Waves per workgroup when there are >= 2048 pairs (batches of >= 256 sequences at 8 kv heads): enough for the chip's ~4096 waves, and by the bound
    // on the keys a workgroup walks (the 256-token context bucket: the contexts themselves are shorter) — with eight waves on a short context a
    // workgroup's life is mostly start-up, barriers and the cross-wave merge, not K/V requests (scratch/attn_batch_shape.py, ragged contexts, us per
    // launch at 8 / 4 / 2 / 1 waves: 512 x <= 100: 45.0 / 37.0 / 35.7 / 32.8; 1024 x <= 100: 83.9 / 70.1 / 64.7 / 63.4; 256 x <= 200: 37.9 / 35.9 /
    // 33.8 / 42.3; 512 x <= 300: 92.3 / 89.2 / 90.0 / 91.1; 256 x 1024: 149 / 153 / 152 / 161; configs[4]'s own partitions, bound 256: 2 waves 3.23, 1 wave 3.13 ms / step)
    constexpr int min_waves = (G * (D / 4) + 63) / 64;                    // the merge takes one pass over (head, 4-column group)
    auto waves_for = [&](int64_t wgs, int64_t keys, int cap) {
        const int64_t want = std::max<int64_t>({(4096 + wgs - 1) / wgs, keys <= 256 ? 1 : keys <= 512 ? 4 : 8, (int64_t)min_waves});
        int w = 1;
        while (w < want && w < cap) w *= 2;
        return w;
    };
    if (paged && a.workspace && a.shared_len <= 0 && pairs >= 2048) waves = waves_for(pairs, mc, 8);
    int part_size = 0x3fffffff, np = 1, sparts = 0, shared_part = 0;
    const bool shared = a.shared_len > 0;
    if (shared) {
        // partitions of shared_len tokens: number 0 (the same K/V for every query) goes through the MFMA kernel, 1.. through
        // the row kernel below; always merged (np >= 2 keeps the partial format even when nobody has own tokens yet)
        if (!paged || !a.workspace || a.seq_of_q || a.shared_len % a.block_size || a.shared_len % 64)
            return nvr::fail(NVR_ERR_INVALID_ARG, "attention: shared_len needs paged decode with a workspace (shared_len %d, block_size %d)", a.shared_len, a.block_size);
        // the shared keys [0, shared_len) are cut into sparts equal partitions (64-key granularity) until the MFMA launch has ~256
        // workgroups; the keys behind them are partitioned like a context of their own (one partition per pair when there are
        // enough pairs, else ~256 workgroups)
        const int qb = flash_tile_positions(a.H, a.KVH);
        const int64_t wgs = (int64_t)((a.nq + qb - 1) / qb) * a.KVH, n64 = a.shared_len / 64;
        int64_t c = std::min<int64_t>(std::max<int64_t>(1, (256 + wgs - 1) / wgs), n64);
        while (n64 % c) --c;
        sparts = (int)c;
        const bool grouped = a.shared_rows != nullptr;
        if (grouped && (!a.shared_kv0 || !a.shared_count)) return nvr::fail(NVR_ERR_INVALID_ARG, "attention: shared_rows / shared_kv0 / shared_count come together");
        const int64_t rest = std::max<int64_t>(grouped ? mc : mc - a.shared_len, 64);   // a query outside the group reads its whole context
        // the workspace holds cap partials per (query, head) (nvr_paged_attn_workspace_bytes: one per 64 tokens of the context bound):
        // the shared partitions and the remainder's together must fit
        const int64_t cap = a.workspace_bytes ? (int64_t)(a.workspace_bytes / ((size_t)a.nq * a.H * (D + 2) * sizeof(float))) : (mc + 63) / 64;
        if (cap < 2) return nvr::fail(NVR_ERR_INVALID_ARG, "attention: workspace too small for the shared-prefix pass");
        while (sparts > 1 && sparts > cap / 2) { --sparts; while (n64 % sparts) --sparts; }
        shared_part = a.shared_len / sparts;
        int64_t want = pairs >= 192 ? 1 : (256 + pairs - 1) / pairs;
        want = std::max<int64_t>(1, std::min<int64_t>(want, cap - sparts));
        part_size = (int)(((rest + want - 1) / want + 63) / 64 * 64);
        np = sparts + (int)((rest + part_size - 1) / part_size);
        // waves per (query, kv head, own partition) workgroup: 4 while that gives the chip its ~4096 waves; with more workgroups than that
        // (configs[4]: 512 x 8 pairs of ~94 own keys) a workgroup's life is mostly the part with no K/V request in flight — cross-wave merge,
        // two barriers, the partition merge behind 24 keys per wave (r05 stamps: ~4 of ~9 us, four rounds of 1024 workgroups) — so one wave
        // streams the whole partition and 16 independent waves per CU cover each other's tails
        const int64_t own_wgs = pairs * (np - sparts);
        waves = own_wgs >= 2048 ? waves_for(own_wgs, part_size, 4) : 4;
    } else if (a.workspace) {
        if (waves >= 8) {
            int64_t want = pairs >= 192 ? 1 : (256 + pairs - 1) / pairs;
            int64_t ps = ((mc + want - 1) / want + 63) / 64 * 64;
            part_size = (int)ps; np = (int)((mc + ps - 1) / ps);
        } else np = parts_for(a.nq, a.KVH, mc, waves, &part_size);
    }
    // Few pairs over short contexts (a chat's first hundred tokens): the partitions' hand-off — partials out, a ticket, partials back — costs more than the keys: ONE workgroup of
    // eight waves per pair, whose round is 128 keys (attn_brief_context).
    const bool brief = paged && a.workspace && !shared && mc <= (pairs <= 128 ? attn_brief_context(a.nq, a.H, a.KVH) : pairs < 192 ? 256 : 0);
    if (brief) { np = 1; waves = 8; }
    // Work-balanced form (attn_share_kernel): a pair count whose last round of one-workgroup-per-pair launches would be mostly empty — 257..2047 pairs with
    // >= 15 % of the rounds' slots unused (33..37 and 65..74 sequences at 8 kv heads, ...), contexts long enough for the stream to matter — or a RAGGED batch
    // (ragged: the caller knows the sum of the contexts; per-pair launches size every pair's partitions by the LONGEST context and leave the short sequences'
    // workgroups idle, or — with several pairs per CU — end on the long sequences' workgroups: 32 sequences of 256..8192 keys 4.09 -> 2.43 ms per Qwen3-0.6B step,
    // 64 of 64..4096 keys 3.26 -> 2.78).  NVR_ATTN_SHARE=0: off.
    if constexpr (G * D <= 512)
    if (!brief && !shared && paged && a.workspace && a.tickets && !a.seq_of_q && waves == 8 && p.bs_shift >= 0 && a.block_size >= 8 && a.nq <= 1024 && share_enabled()) {
        const int64_t cus = share_workgroups(), rounds = (pairs + cus - 1) / cus, units = (mc + 63) / 64;
        const int64_t cap = a.workspace_bytes ? (int64_t)(a.workspace_bytes / ((size_t)a.nq * a.H * (D + 2) * sizeof(float))) : units;
        const bool by_count = pairs > cus && rounds * cus * 100 >= pairs * 115 && mc >= 256;
        if ((by_count || a.ragged || share_mode() == 2) && pairs < 2048 && cap >= units) {
            p.part_size = 64; p.num_parts = (int32_t)cap;
            p.part_o = (float *)a.workspace; p.part_ml = p.part_o + (int64_t)a.nq * a.H * cap * D;
            p.part0 = 0; p.kv0 = 0; p.kv0_rows = nullptr; p.tickets = a.tickets;
            const int shares = (int)std::max<int64_t>(1, cus / a.KVH);                      // one workgroup per CU
            bool in_it = false;
            // (the step's own rows in this launch up to three pairs for two CUs: a share opens more segments beyond, and each waits for its norms.  Qwen3-0.6B with norms, us a step by a launch in
            // front / here: 33 sequences of 32..700 keys 1436 / 1388, 40 of 64..4000 1960 / 1922, 48 of 64..2000 1834 / 1780, 56 of 64..2000 1926 / 1992, 64 of 64..3000 2317 / 2308, 80 of 32..700
            // 1853 / 1890, 96 of 64..2000 2488 / 2514, 128 of 32..700 2244 / 2309, 200 of 32..1000 2730 / 2737)
            if constexpr (D == 128 && G <= 4)
                if (own_rows_aligned(a) && 2 * pairs <= 3 * (int64_t)cus) {
                    attn_share_kernel<D, G, DU / 2, 8, true><<<dim3((unsigned)(shares * a.KVH)), dim3(512), 0, s>>>(AttnParamsOwn{p, own_rows_params(a)}, (int)a.nq, shares);
                    in_it = true;
                }
            if (!in_it) {
                if (int rc = own_rows(a, s)) return rc;
                attn_share_kernel<D, G, DU / 2, 8><<<dim3((unsigned)(shares * a.KVH)), dim3(512), 0, s>>>(p, (int)a.nq, shares);
            }
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "attention (work-balanced) launch failed: %s", hipGetErrorString(e));
            return 0;
        }
    }
    if constexpr (D == 128 && G <= 4)
        if (shared && prefix_in_one_launch(a)) {
            if (int rc = own_rows(a, s)) return rc;
            const int64_t ns = (pairs + share_workgroups() - 1) / share_workgroups();     // sequences of a workgroup: one workgroup per CU
            if (ns <= 1) return launch_prefix<G, 1>(p, a.nq, a.shared_len, s);
            if (ns <= 2) return launch_prefix<G, 2>(p, a.nq, a.shared_len, s);
            if (ns <= 4) return launch_prefix<G, 4>(p, a.nq, a.shared_len, s);
            if constexpr (G <= 2) return launch_prefix<G, 8>(p, a.nq, a.shared_len, s);
        }
    const bool direct = np <= 1;
    if (!direct && a.workspace_bytes && (size_t)a.nq * a.H * np * (D + 2) * sizeof(float) > a.workspace_bytes)
        return nvr::fail(NVR_ERR_INVALID_ARG, "attention: %d partitions of %d queries x %d heads need %zu workspace bytes, %zu given",
                         np, a.nq, a.H, (size_t)a.nq * a.H * np * (D + 2) * sizeof(float), a.workspace_bytes);
    if (direct) { p.part_size = 0x3fffffff; p.num_parts = 1; }
    else {
        p.part_size = part_size; p.num_parts = np;
        p.part_o = (float *)a.workspace;
        p.part_ml = p.part_o + (int64_t)a.nq * a.H * np * D;
    }
    p.part0 = sparts; p.kv0 = shared ? a.shared_len : 0; p.kv0_rows = shared ? a.shared_kv0 : nullptr;
    const int64_t nwg = (int64_t)(p.num_parts - p.part0) * a.KVH * a.nq;
    // split-KV without a shared-prefix pass: the last partition workgroup of a (query, kv head) to finish merges the pair (no merge launch)
    const bool fuse = !direct && !shared && paged && a.tickets != nullptr;
    p.tickets = a.tickets;
    // ... and with a shared-prefix pass in front whose group is the whole batch, one own partition per pair: that workgroup merges (SHM)
    const bool shm = shared && paged && !a.shared_rows && np - sparts == 1 && a.tickets != nullptr;
    // the step's own rows (QKN): in this launch where four or eight waves walk a pair's keys in blocks of whole chunks and there is a CU for every pair (beyond, the start of every pair's workgroup
    // pays for it again: Qwen3-0.6B with norms at 300 keys, us a step by a launch in front / here: 1 sequence 764 / 721, 2 833 / 784, 4 896 / 826, 8 975 / 912, 16 1062 / 998, 32 1159 / 1115,
    // 64 1674 / 1677, 128 2243 / 2249; 256 of 1024 keys 6069 / 6090)
    const int tpi = 64 / (D / 8) * (brief || waves == 4 ? DU : DU / 2);
    const bool qkn = D == 128 && G <= 4 && !shared && paged && pairs <= share_workgroups() && (waves == 8 || waves == 4) && (direct || fuse) && p.block_size % tpi == 0 && (p.num_parts == 1 || p.part_size % tpi == 0) && own_rows_aligned(a);
    const OwnRows own_params = own_rows_params(a), *const own = qkn ? &own_params : nullptr;
    if (!qkn) if (int rc = own_rows(a, s)) return rc;
    if (shared)
        if (int rc = flash_shared_prefix(a.q, a.ldq, a.k, a.v, a.block_tables, a.max_blocks, a.block_size, a.nq, a.H, a.KVH, a.D, a.scale,
                                         shared_part, sparts, np, p.part_o, p.part_ml, s, a.shared_rows, a.shared_count)) return rc;
    {
        if (brief) {
            const bool ub = p.block_size % (64 / (D / 8) * DU) == 0;
            if (qkn) launch_cfg<D, G, DU, 8, true>(p, true, true, nwg, s, false, false, own);
            else if (ub) attn_rows_kernel<D, G, true, true, DU, 8, true, true><<<dim3((unsigned)nwg), dim3(512), 0, s>>>(p);
            else attn_rows_kernel<D, G, true, true, DU, 8, true, false><<<dim3((unsigned)nwg), dim3(512), 0, s>>>(p);
        } else if (waves == 8) launch_cfg<D, G, DU / 2, 8, true>(p, paged, direct, nwg, s, fuse, false, own);  // K/V streamed once: nt loads
        else if (paged && waves == 1) { if constexpr (G * (D / 4) <= 64) launch_cfg<D, G, DU, 1, true>(p, paged, direct, nwg, s, fuse, shm); }   // (U = 2: 3.18-3.20 against 3.14-3.17 ms per configs[4] step)
        else if (paged && waves == 2) { if constexpr (G * (D / 4) <= 128) launch_cfg<D, G, DU, 2, true>(p, paged, direct, nwg, s, fuse, shm); }
        else if (paged) launch_cfg<D, G, DU, 4, true>(p, paged, direct, nwg, s, fuse, shm, own);
        else launch_cfg<D, G, DU, 4, false>(p, paged, direct, nwg, s);                     // prefill: rows re-read from L2
    }
    if (!direct && !fuse && !shm)
        attn_merge_kernel<D><<<dim3((unsigned)(((int64_t)a.H * a.nq + 256 / (D / 4) - 1) / (256 / (D / 4)))), dim3(256), 0, s>>>(
            p.part_o, p.part_ml, a.ctx_lens, a.H, part_size, np, p.part0, p.kv0, p.kv0_rows, (int64_t)a.H * a.nq, p.out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "attention launch failed: %s", hipGetErrorString(e));
    return 0;
}

int attention(const AttnArgs &a, bool paged, hipStream_t s) {
    if (a.nq == 0) return 0;
    if (a.H % a.KVH) return nvr::fail(NVR_ERR_INVALID_ARG, "attention: H=%d not a multiple of KVH=%d", a.H, a.KVH);
    const int G = a.H / a.KVH;
#define NVR_ATTN_CASE(DD, GG) if (a.D == DD && G == GG) return launch_attn<DD, GG>(a, paged, s);
    NVR_ATTN_CASE(128, 1) NVR_ATTN_CASE(128, 2) NVR_ATTN_CASE(128, 4) NVR_ATTN_CASE(128, 8)
    NVR_ATTN_CASE(64, 1) NVR_ATTN_CASE(64, 2) NVR_ATTN_CASE(64, 4) NVR_ATTN_CASE(64, 8)
#undef NVR_ATTN_CASE
    return nvr::fail(NVR_ERR_UNSUPPORTED, "attention: unsupported head_dim=%d / group=%d (D in {64,128}, G in {1,2,4,8})",
                     a.D, G);
}

// (more than 64 KiB of LDS are opted in for each instance, in front of a runner's first step of this form: the step may be captured.  Not at the runner's creation: with the opt-in there a step of one
// sequence of 128 keys, which has none of these kernels, took 672 us instead of 661)
int attn_prepare() {
    static std::atomic<bool> done{false};
    if (done.load(std::memory_order_acquire)) return 0;
#define NVR_PREFIX_ATTR(G_, NS_)                                                                                                                                                                  \
    {                                                                                                                                                                                             \
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&attn_prefix_kernel<G_, NS_>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)prefix_lds<G_, NS_>());            \
        if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "attention (shared prefix): LDS opt-in failed: %s", hipGetErrorString(e));                                                             \
    }
    NVR_PREFIX_ATTR(1, 1) NVR_PREFIX_ATTR(1, 2) NVR_PREFIX_ATTR(1, 4) NVR_PREFIX_ATTR(1, 8) NVR_PREFIX_ATTR(2, 1) NVR_PREFIX_ATTR(2, 2) NVR_PREFIX_ATTR(2, 4) NVR_PREFIX_ATTR(2, 8)
    NVR_PREFIX_ATTR(4, 1) NVR_PREFIX_ATTR(4, 2) NVR_PREFIX_ATTR(4, 4)
#undef NVR_PREFIX_ATTR
    done.store(true, std::memory_order_release);
    return 0;
}

}}  // namespace nvr::k / nvr::kb (NVR_DT_NS)
