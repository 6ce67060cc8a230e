// linear.hip — y[T,N] = x[T,K] · W[N,K]^T on MFMA (K3/K10/K12/K14/K16), with the two epilogue fusions of
// the decode path: gate_up -> SiluAndMul (K12+K13) and qkv -> RoPE + KV store (K3+K4+K5+K6).
// reference call sites: QKVParallelLinear::forward src/layers/linear.rs:354-356 (+split_qkv :331-340),
// RowParallelLinear :228-239, MergedColumnParallelLinear :437-439 (+SiluAndMul activation.rs:46-63),
// ParallelLMHead::compute_logits src/layers/embed_head.rs:292-306; all `candle_nn::Linear::forward`,
// x·Wᵀ with W [out, in]; RoPE src/layers/rotary_embedding.rs:23-48; store_kv_cache attention.rs:150-174.
//
// Weight-streaming kernel for the decode regime (T <= 64: every weight byte is read once from HBM
// and the kernel is HBM/latency-bound).  Roofline: algorithmic bytes = 2·N·K (weights)
// + 2·T·K (x) + out; MFMA is used only because T=32 tokens x 8 k per 16-byte weight load exceeds
// the VALU rate at HBM speed (cdna_hip_programming.md §5 "GEMV / M <= 16" row: weights straight to
// VGPRs, no LDS round trip).
//
// Tiling: v_mfma_f32_16x16x32_f16 with A = W tile (16 output columns n x 32 k: each lane loads 16
// contiguous bytes of one W row, 4 lanes cover 64 B of the row) and B = x tile (16 tokens x 32 k,
// L2 resident).  A workgroup = WAVES waves owns NT*16 output columns for MT*16 tokens; its waves
// interleave 32-wide k steps (together they read 64·WAVES contiguous bytes per W row per step, all
// k-steps of a small GEMM in flight at once) and reduce their f32 partials through LDS.
// Grid = (N/(16 NT), ceil(T/(16 MT))): for large T the same kernel re-streams W from L2 per 16·MT-token
// slab (correct, not yet the tiled prefill GEMM).
//
// Rounding points mirror the oracle (oracle/model_oracle.py): the f32 accumulator is rounded to fp16
// where the unfused graph stores an fp16 tensor (qkv, gate_up), then the epilogue math runs in f32
// without FMA contraction and is rounded again.
#include <algorithm>
#include <cstdlib>
#include "kernels.h"
#include "device_utils.h"
#include "slab_walk.h"
#include "../common.h"

namespace nvr { namespace NVR_DT_NS {

enum { EPI_F16 = 0, EPI_F32 = 1, EPI_SILU = 2, EPI_ROPE = 3, EPI_SLAB = 4, EPI_CLAMP = 5 };
// rows up to which a decode step's add + norm rides on the product behind it: every workgroup reads every row's slabs again (16 KB a row at K = 1024), so the launch it saves pays for a few
// rows — Qwen3-0.6B at 300 keys, us a step apart / riding: 802 / 727 at one row, 822 / 760 at two, 840 / 792 at three, 863 / 826 at four (as many as NORM_ELEMS holds of that width)
constexpr int64_t NORM_ROWS = 4;

struct LinEpi {
    // EPI_SILU, EPI_CLAMP: N is the intermediate size I; W holds gate rows [0,I) and up rows [I,2I)
    // EPI_ROPE: qkv output [T, (H+2KVH)*D] + caches
    const int64_t *pos; const int32_t *slots; const float *cos_t, *sin_t;
    half_t *kc, *vc;
    int32_t H, KVH, D;
    // EPI_SLAB: blockIdx.z owns k in [z*kslice, (z+1)*kslice) and writes its f32 partial tile to slab z
    int32_t kslice; int64_t slab_stride;
    // W is the TILED copy [N/16][K/32][16][32] (retile_weight): one wave-instruction reads 1 KiB contiguous
    int32_t tiled;
    int32_t gelu;                          // EPI_SILU: gelu (tanh form) instead of silu; EPI_F16: gelu (error function) of the product
};
// What single instances need beyond it stays out of the others' arguments
struct LinEpiNorm : LinEpi { NormIn norm; };                       // NORM instances: x is formed by the workgroup itself
struct LinEpiClamp : LinEpi { float limit, alpha; int64_t ldy; };  // EPI_CLAMP: min(g, limit) sigmoid(alpha min(g, limit)) (clamp(u, +-limit) + 1); row stride of y
// NORM: slabs that an instance has room for (0: it takes its rows as they are)
template <int EPI, int NORM> struct LinArgs { using type = LinEpiNorm; };
template <int EPI> struct LinArgs<EPI, 0> { using type = LinEpi; };
template <> struct LinArgs<EPI_CLAMP, 0> { using type = LinEpiClamp; };

// W row handled by local row r (0..15) of n-tile i of workgroup bx
template <int EPI>
__device__ __forceinline__ int w_row(int bx, int i, int NT, int r, int N, const LinEpi &e) {
    if (EPI == EPI_SILU || EPI == EPI_CLAMP) return (i == 0 ? 0 : N) + bx * 16 + r;             // N == I here
    if (EPI == EPI_ROPE) {
        const int tph = e.D / 16, head = bx / tph, c = bx % tph;            // tiles per head
        if (head < e.H + e.KVH) return head * e.D + (r < 8 ? c * 8 + r : e.D / 2 + c * 8 + (r - 8));
        return head * e.D + c * 16 + r;
    }
    int n = (bx * NT + i) * 16 + r;
    return n < N ? n : N - 1;
}

// NORM (MT = 1, T <= NORM_ROWS, T K <= NORM_ELEMS): the rows are RMSNorm(h + sum of the split-k slabs) (what add_rmsnorm_slabs leaves in memory, with its roundings: 16-bit sum of
// the slabs, 16-bit residual add, 16-bit normalised row), formed by every workgroup in LDS while its first weight pieces are on the way, so that the add + norm launch in front of
// the product disappears; workgroup 0 writes the new residual rows to norm.h_out, a second buffer, since the others still read the old ones.
constexpr int NORM_ELEMS = 4096;
template <int NT, int MT, int WAVES, int EPI, int NORM = 0>
__global__ __launch_bounds__(WAVES * 64) void linear_skinny_kernel(const half_t *__restrict__ x, int64_t ldx,
                                                                   const half_t *__restrict__ W, int T, int K, int N,
                                                                   void *__restrict__ y, typename LinArgs<EPI, NORM>::type epi) {
    constexpr int U = 4;                                    // k-steps in flight per wave
    extern __shared__ __attribute__((aligned(16))) char norm_lds[];   // NORM: the normalised rows [T][K + 8]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;
    const int m0 = blockIdx.y * (16 * MT);

    const half_t *wrow[NT];
    const half_t *xrow[MT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        if (epi.tiled) {
            // tile index in the tiled copy: SiLU — gate tile bx, up tile I/16 + bx; RoPE — tile bx of the permuted row order;
            // else tile bx*NT + i (clamped like w_row clamps its rows)
            int64_t tile = EPI == EPI_SILU || EPI == EPI_CLAMP ? (i == 0 ? (int64_t)blockIdx.x : (int64_t)(N / 16) + blockIdx.x) : (int64_t)blockIdx.x * NT + i;
            if (EPI != EPI_SILU && EPI != EPI_CLAMP && EPI != EPI_ROPE && tile > N / 16 - 1) tile = N / 16 - 1;
            wrow[i] = W + tile * (int64_t)(K / 32) * 512 + r * 32 + q * 8;
        } else wrow[i] = W + (int64_t)w_row<EPI>(blockIdx.x, i, NT, r, N, epi) * K + q * 8;
    }
    const int kmul = epi.tiled ? 16 : 1;                            // k -> element offset: (k / 32) * 512 in the tiled copy
#pragma unroll
    for (int i = 0; i < MT; ++i) { int m = m0 + i * 16 + r; if (m > T - 1) m = T - 1; xrow[i] = x + (int64_t)m * ldx + q * 8; }

    float4_t acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};

    // Loads come back in the order they were requested.  EPI_ROPE: the epilogue of token tile j runs on wave j; its position and slot are requested first, its cosines and sines (which wait for the
    // position) behind the first weight pieces, all ahead of their use after the reduction barrier.
    float4_t rope_cs = (float4_t){0.f, 0.f, 0.f, 0.f}, rope_sn = rope_cs;
    int rope_slot = -1;
    int64_t rope_p = 0;
    const int rope_tph = EPI == EPI_ROPE ? epi.D / 16 : 1, rope_head = blockIdx.x / rope_tph;
    if (EPI == EPI_ROPE && wave < MT) {
        const int m = m0 + wave * 16 + r;
        rope_p = epi.pos[m < T ? m : T - 1];
        if (rope_head >= epi.H && epi.slots && m < T) rope_slot = epi.slots[m];
    }
    auto rope_request = [&]() {
        if (EPI == EPI_ROPE && wave < MT && rope_head < epi.H + epi.KVH) {
            const int64_t at = rope_p * (epi.D / 2) + (blockIdx.x % rope_tph) * 8 + (q & 1) * 4;
            rope_cs = *reinterpret_cast<const float4_t *>(epi.cos_t + at);
            rope_sn = *reinterpret_cast<const float4_t *>(epi.sin_t + at);
        }
    };
    constexpr int KS = 32 * WAVES;
    constexpr bool AHEAD = NORM > 0 || EPI == EPI_ROPE;
    half8_t a_first[U][NT], b_first[U][MT];                  // AHEAD: the first pieces of the weights (and rows)
    auto first_request = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kk = min(wave * 32 + u * KS, K - 32);
#pragma unroll
            for (int i = 0; i < NT; ++i) a_first[u][i] = __builtin_nontemporal_load(reinterpret_cast<const half8_t *>(wrow[i] + (int64_t)kk * kmul));
            if constexpr (NORM == 0)
#pragma unroll
                for (int j = 0; j < MT; ++j) b_first[u][j] = *reinterpret_cast<const half8_t *>(xrow[j] + kk);
        }
        asm volatile("" ::: "memory");
    };
    if constexpr (AHEAD && NORM == 0) { first_request(); rope_request(); }
    if constexpr (NORM > 0) {
        static_assert(MT == 1, "one row block");
        constexpr int NI = NORM_ELEMS / 4 / (WAVES * 64);     // 4-column pieces per thread
        __shared__ float ss_w[NI * WAVES];                    // sums of squares of 64 neighbouring pieces (K is a multiple of 256: inside one row)
        half_t *xs = reinterpret_cast<half_t *>(norm_lds);
        const NormIn &nm = epi.norm;
        const int per_row = K / 4, total = T * per_row;
        half4_t hv[NI], gv[NI]; float4_t sv[NI][NORM];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int idx = i * (WAVES * 64) + (int)threadIdx.x;
            if (idx < total) {
                const int row = idx / per_row, c = (idx - row * per_row) * 4;
                const int64_t o = (int64_t)row * K + c;
                hv[i] = *reinterpret_cast<const half4_t *>((const half_t *)nm.h_in + o); gv[i] = *reinterpret_cast<const half4_t *>((const half_t *)nm.w + c);
#pragma unroll
                for (int z = 0; z < NORM; ++z) sv[i][z] = z < nm.S ? *reinterpret_cast<const float4_t *>(nm.slabs + z * nm.stride + o) : (float4_t){0.f, 0.f, 0.f, 0.f};
            }
        }
        asm volatile("" ::: "memory");
        first_request();                                      // the weights behind the rows: in front of them, the norm would start when they
                                                              // have arrived (one row: qkv of 4096 columns 6.5 -> 5.5 us, gate_up of 3072 6.6 -> 5.8)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int idx = i * (WAVES * 64) + (int)threadIdx.x;
            if (idx - lane < total) {                         // (wave-uniform: total is a multiple of 64)
                float ss = 0.f;
                float4_t a = sv[i][0];
#pragma unroll
                for (int z = 1; z < NORM; ++z) a += sv[i][z];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hv[i][e] = to_half_rn((float)hv[i][e] + (float)to_half_rn(a[e]));
                    const float f = (float)hv[i][e]; ss += f * f;
                }
                ss = wave_sum(ss);
                if (lane == 0) ss_w[i * WAVES + wave] = ss;
            }
        }
        rope_request();
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int idx = i * (WAVES * 64) + (int)threadIdx.x;
            if (idx < total) {
                const int row = idx / per_row, c = (idx - row * per_row) * 4;
                float tot = 0.f;
                const int np = per_row / 64;
                for (int k0 = 0; k0 < np; k0 += 4) {           // (four requested together, added in their order)
                    float p[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) p[k] = ss_w[row * np + min(k0 + k, np - 1)];
#pragma unroll
                    for (int k = 0; k < 4; ++k) if (k0 + k < np) tot += p[k];
                }
                const float rms = sqrtf(tot / (float)K + nm.eps);
                half4_t o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = to_half_rn(__fmul_rn(__fdiv_rn((float)hv[i][e], rms), (float)gv[i][e]));
                *reinterpret_cast<half4_t *>(xs + row * (K + 8) + c) = o;
                if (blockIdx.x == 0) *reinterpret_cast<half4_t *>((half_t *)nm.h_out + (int64_t)row * K + c) = hv[i];
            }
        }
        __syncthreads();
        xrow[0] = xs + (int64_t)min(r, T - 1) * (K + 8) + q * 8;
    }
    constexpr bool SLABBED = EPI == EPI_SLAB;
    const int kbeg = SLABBED ? blockIdx.z * epi.kslice : 0;
    if (SLABBED) K = min(K, kbeg + epi.kslice);
    for (int k = kbeg + wave * 32; k < K; k += KS * U) {
        half8_t a[U][NT], b[U][MT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kk = k + u * KS;
            if (kk < K) {
#pragma unroll
                for (int i = 0; i < NT; ++i) {
                    if (AHEAD && k == kbeg + wave * 32) a[u][i] = a_first[u][i];
                    else a[u][i] = __builtin_nontemporal_load(reinterpret_cast<const half8_t *>(wrow[i] + (int64_t)kk * kmul));
                }
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    if (AHEAD && NORM == 0 && k == kbeg + wave * 32) b[u][j] = b_first[u][j];
                    else b[u][j] = *reinterpret_cast<const half8_t *>(xrow[j] + kk);
                }
            } else {
#pragma unroll
                for (int i = 0; i < NT; ++i) a[u][i] = (half8_t)(half_t)0;
#pragma unroll
                for (int j = 0; j < MT; ++j) b[u][j] = (half8_t)(half_t)0;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j)
                    acc[i][j] = mfma16(a[u][i], b[u][j], acc[i][j]);
    }

    // cross-wave (split-k) reduction through LDS: part[wave][tile][lane] as float4
    __shared__ float4_t part[WAVES][NT * MT][64];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) part[wave][i * MT + j][lane] = acc[i][j];
    __syncthreads();

    auto reduce = [&](int tile) {
        float4_t s = part[0][tile][lane];
#pragma unroll
        for (int w2 = 1; w2 < WAVES; ++w2) { float4_t pz = part[w2][tile][lane]; s += pz; }
        return s;
    };
    // C layout of the 16x16 MFMA: row (n) = q*4 + reg, col (token) = r
    if (EPI == EPI_F16 || EPI == EPI_F32 || EPI == EPI_SLAB) {
        for (int tile = wave; tile < NT * MT; tile += WAVES) {
            float4_t s = reduce(tile);
            if (EPI == EPI_F16 && epi.gelu)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = gelu_erf_fast(s[e]);
            const int i = tile / MT, j = tile % MT;
            const int n = (blockIdx.x * NT + i) * 16 + q * 4, m = m0 + j * 16 + r;
            if (m < T && n < N) {
                if (EPI == EPI_F32) {
                    *reinterpret_cast<float4_t *>(reinterpret_cast<float *>(y) + (int64_t)m * N + n) = s;
                } else if (EPI == EPI_SLAB) {
                    *reinterpret_cast<float4_t *>(reinterpret_cast<float *>(y) + blockIdx.z * epi.slab_stride + (int64_t)m * N + n) = s;
                } else {
                    half4_t h = {(half_t)s[0], (half_t)s[1], (half_t)s[2], (half_t)s[3]};
                    *reinterpret_cast<half4_t *>(reinterpret_cast<half_t *>(y) + (int64_t)m * N + n) = h;
                }
            }
        }
    } else if (EPI == EPI_SILU || EPI == EPI_CLAMP) {
        // tiles (0,j) = gate, (1,j) = up for the same 16 columns: act = fp16(silu(fp16 g) * fp16 u)
        for (int j = wave; j < MT; j += WAVES) {
            const float4_t g4 = reduce(j), u4 = reduce(MT + j);
            const int n = blockIdx.x * 16 + q * 4, m = m0 + j * 16 + r;
            if (m < T) {
                half4_t h;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float gf = (float)to_half_rn(g4[e]), uf = (float)to_half_rn(u4[e]);
                    if constexpr (EPI == EPI_CLAMP) {
                        const float g = fminf(gf, epi.limit), u = fminf(fmaxf(uf, -epi.limit), epi.limit);
                        h[e] = to_half_rn(g / (1.0f + expf(-epi.alpha * g)) * (u + 1.0f));
                    } else {
                        const float sg = gate_factor(gf, epi.gelu);
                        h[e] = to_half_rn(__fmul_rn(__fmul_rn(gf, sg), uf));
                    }
                }
                if constexpr (EPI == EPI_CLAMP) *reinterpret_cast<half4_t *>(reinterpret_cast<half_t *>(y) + (int64_t)m * epi.ldy + n) = h;
                else *reinterpret_cast<half4_t *>(reinterpret_cast<half_t *>(y) + (int64_t)m * N + n) = h;
            }
        }
    } else {   // EPI_ROPE: NT == 1
        const int tph = epi.D / 16, head = blockIdx.x / tph, c = blockIdx.x % tph, half_d = epi.D / 2;
        const int64_t ldq = (int64_t)(epi.H + 2 * epi.KVH) * epi.D;
        for (int j = wave; j < MT; j += WAVES) {
            const float4_t s = reduce(j);
            const int m = m0 + j * 16 + r;
            const int mc = m < T ? m : T - 1;
            float v[4], pv[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) { v[e] = (float)to_half_rn(s[e]); pv[e] = __shfl_xor(v[e], 32, 64); }
            half4_t h;
            int col;                                           // first of the lane's 4 consecutive head columns
            if (head < epi.H + epi.KVH) {
                const int jj = c * 8 + (q & 1) * 4;            // index inside the half dimension
                float4_t cs = rope_cs, sn = rope_sn;
                if (MT > WAVES) {                               // never instantiated: every token tile has its own wave
                    cs = *reinterpret_cast<const float4_t *>(epi.cos_t + epi.pos[mc] * half_d + jj);
                    sn = *reinterpret_cast<const float4_t *>(epi.sin_t + epi.pos[mc] * half_d + jj);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // rotary_embedding.rs:36-44: out1 = x1*c - x2*s ; out2 = x2*c + x1*s
                    h[e] = (q < 2) ? to_half_rn(mul_sub_unfused(v[e], cs[e], pv[e], sn[e]))
                                   : to_half_rn(mul_add_unfused(v[e], cs[e], pv[e], sn[e]));
                }
                col = (q < 2) ? jj : half_d + jj;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = to_half_rn(s[e]);
                col = c * 16 + q * 4;
            }
            if (m < T) {
                *reinterpret_cast<half4_t *>(reinterpret_cast<half_t *>(y) + (int64_t)m * ldq + head * epi.D + col) = h;
                const int slot = MT > WAVES ? (epi.slots ? epi.slots[m] : -1) : rope_slot;
                if (slot >= 0 && head >= epi.H) {
                    const bool is_k = head < epi.H + epi.KVH;
                    const int kvh = is_k ? head - epi.H : head - epi.H - epi.KVH;
                    half_t *dst = (is_k ? epi.kc : epi.vc) + ((int64_t)slot * epi.KVH + kvh) * epi.D + col;
                    *reinterpret_cast<half4_t *>(dst) = h;
                }
            }
        }
    }
}

// Two products of a decode step that do not wait for each other, of rows x and x2 of one length, in one launch: the first `units` workgroups of a row block form the clamped gated unit of I columns
// (EPI_CLAMP), the others the plain product of N (EPI_F16).  Both sum as linear_skinny_kernel does, and have its bits; a body of its own, since the instances of that kernel come out otherwise with
// a function that they share.
template <int NT, int MT, int WAVES>
__device__ __forceinline__ void few_rows_sums(const half_t *__restrict__ x, int64_t ldx, const half_t *(&wrow)[NT], int m0, int T, int K, float4_t (&part)[WAVES][2 * MT][64]) {
    constexpr int U = 4, KS = 32 * WAVES;                   // k-steps in flight per wave
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const half_t *xrow[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) xrow[j] = x + (int64_t)min(m0 + j * 16 + r, T - 1) * ldx + q * 8;
    float4_t acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
    for (int k = wave * 32; k < K; k += KS * U) {
        half8_t a[U][NT], b[U][MT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kk = k + u * KS;
            if (kk < K) {
#pragma unroll
                for (int i = 0; i < NT; ++i) a[u][i] = __builtin_nontemporal_load(reinterpret_cast<const half8_t *>(wrow[i] + kk));
#pragma unroll
                for (int j = 0; j < MT; ++j) b[u][j] = *reinterpret_cast<const half8_t *>(xrow[j] + kk);
            } else {
#pragma unroll
                for (int i = 0; i < NT; ++i) a[u][i] = (half8_t)(half_t)0;
#pragma unroll
                for (int j = 0; j < MT; ++j) b[u][j] = (half8_t)(half_t)0;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) acc[i][j] = mfma16(a[u][i], b[u][j], acc[i][j]);
    }
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) part[wave][i * MT + j][lane] = acc[i][j];
    __syncthreads();
}
template <int MT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void linear_beside_unit_kernel(const half_t *__restrict__ x, const half_t *__restrict__ x2, int64_t ldx, const half_t *__restrict__ W, const half_t *__restrict__ W2,
                                                                        int T, int K, int N, int I, half_t *__restrict__ y, half_t *__restrict__ y2, int64_t ldy2, float limit, float alpha) {
    __shared__ float4_t part[WAVES][2 * MT][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int m0 = blockIdx.y * (16 * MT), units = I / 16;
    auto reduce = [&](int tile) {
        float4_t s = part[0][tile][lane];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) s += part[w][tile][lane];
        return s;
    };
    const int m = m0 + wave * 16 + r;                       // (row tile j is finished by wave j)
    if ((int)blockIdx.x < units) {
        const half_t *wrow[2] = {W2 + ((int64_t)blockIdx.x * 16 + r) * K + q * 8, W2 + ((int64_t)I + blockIdx.x * 16 + r) * K + q * 8};
        few_rows_sums<2, MT, WAVES>(x2, ldx, wrow, m0, T, K, part);
        if (wave < MT && m < T) {
            const float4_t g4 = reduce(wave), u4 = reduce(MT + wave);
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float g = fminf((float)to_half_rn(g4[e]), limit), u = fminf(fmaxf((float)to_half_rn(u4[e]), -limit), limit);
                h[e] = to_half_rn(g / (1.0f + expf(-alpha * g)) * (u + 1.0f));
            }
            *reinterpret_cast<half4_t *>(y2 + (int64_t)m * ldy2 + blockIdx.x * 16 + q * 4) = h;
        }
    } else {
        const int n0 = ((int)blockIdx.x - units) * 16;
        const half_t *wrow[1] = {W + ((int64_t)n0 + r) * K + q * 8};
        few_rows_sums<1, MT, WAVES>(x, ldx, wrow, m0, T, K, part);
        if (wave < MT && m < T) {
            const float4_t s = reduce(wave);
            *reinterpret_cast<half4_t *>(y + (int64_t)m * N + n0 + q * 4) = (half4_t){(half_t)s[0], (half_t)s[1], (half_t)s[2], (half_t)s[3]};
        }
    }
}

// The split-k products of large weights (linear_splitk: 64 columns a workgroup, eight waves, slab blockIdx.z): what linear_skinny_kernel<4, MT, 8, EPI_SLAB> computes, with its sums' order.  A wave has
// several rounds of requests there (12 steps of 32 k at K = 12288 in four slices), and each round waited for the one in front of it; here three sets of two steps take turns, two of them on their way
// while the third is multiplied.  Slices: slab_takes.  Qwen3-8B, us a step, linear_skinny_kernel / so: 32 sequences of 2048 keys 5087 / 5051, 24 of 300 3740 / 3714, up to 16 sequences the same.
template <int MT>
__global__ __launch_bounds__(512) void linear_slab_kernel(const half_t *__restrict__ x, int64_t ldx, const half_t *__restrict__ W, int T, int K, int N, float *__restrict__ y, int kslice, int64_t slab_stride,
                                                          int tiled) {
    constexpr int NT = 4, WAVES = SLAB_WAVES, U = SLAB_SET;
    __shared__ float4_t part[WAVES][NT * MT][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int m0 = blockIdx.y * (16 * MT), k0 = slab_column(kslice, (int)blockIdx.z, wave), sets = slab_steps(kslice) / U;
    const int64_t step = tiled ? (int64_t)(SLAB_STEP / 32) * 512 : SLAB_STEP;
    const half_t *wrow[NT], *xrow[MT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int tile = (int)blockIdx.x * NT + i;
        wrow[i] = tiled ? W + ((int64_t)tile * (K / 32) + k0 / 32) * 512 + r * 32 + q * 8 : W + ((int64_t)tile * 16 + r) * K + k0 + q * 8;
    }
#pragma unroll
    for (int j = 0; j < MT; ++j) xrow[j] = x + (int64_t)min(m0 + j * 16 + r, T - 1) * ldx + k0 + q * 8;
    float4_t acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
    struct Set { half8_t a[U][NT], b[U][MT]; } s0, s1, s2 = {};
    auto request = [&](Set &s, int set) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = set * U + u;
#pragma unroll
            for (int i = 0; i < NT; ++i) s.a[u][i] = __builtin_nontemporal_load(reinterpret_cast<const half8_t *>(wrow[i] + k * step));
#pragma unroll
            for (int j = 0; j < MT; ++j) s.b[u][j] = *reinterpret_cast<const half8_t *>(xrow[j] + (int64_t)k * SLAB_STEP);
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](const Set &s) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) acc[i][j] = mfma16(s.a[u][i], s.b[u][j], acc[i][j]);
        __builtin_amdgcn_sched_barrier(0);
    };
    request(s0, 0); request(s1, 1);                                       // (two sets at least)
    int i = 0;                                                            // sets i and i + 1 are on their way
    for (; i + 5 <= sets; i += 3) {
        request(s2, i + 2); multiply(s0);
        request(s0, i + 3); multiply(s1);
        request(s1, i + 4); multiply(s2);
    }
    const int left = sets - i;                                            // 2, 3 or 4
    if (left > 2) request(s2, i + 2);
    multiply(s0);
    if (left > 3) request(s0, i + 3);
    multiply(s1);
    if (left > 2) multiply(s2);
    if (left > 3) multiply(s0);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) part[wave][i * MT + j][lane] = acc[i][j];
    __syncthreads();
    for (int tile = wave; tile < NT * MT; tile += WAVES) {
        float4_t s = part[0][tile][lane];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) s += part[w][tile][lane];
        const int n = ((int)blockIdx.x * NT + tile / MT) * 16 + q * 4, m = m0 + tile % MT * 16 + r;
        if (m < T) *reinterpret_cast<float4_t *>(y + blockIdx.z * slab_stride + (int64_t)m * N + n) = s;
    }
}

template <int NT, int MT, int WAVES, int EPI>
static void launch(const half_t *x, int64_t ldx, const half_t *W, int T, int K, int N, void *y, const typename LinArgs<EPI, 0>::type &e,
                   unsigned gx, hipStream_t s, unsigned gz = 1) {
    dim3 grid(gx, (unsigned)((T + 16 * MT - 1) / (16 * MT)), gz);
    linear_skinny_kernel<NT, MT, WAVES, EPI><<<grid, dim3(WAVES * 64), 0, s>>>(x, ldx, W, T, K, N, y, e);
}

// 256x256 kernel or 128x128 kernel?  The 128x128 kernel takes 9.4 K/1024 + 3.5 us while its tiles fit one per CU (K = 1024 13.3 us, 2048 22, 4096 42, 12288 118), beyond that 8 K/1024 + 1.2 per 256
// tiles (768 tiles 31, 1152 45, 2048 73 at K = 1024).  The line for the 256x256 kernel is a round of its tiles for a round of its time, whatever their number.  The kernel itself takes less for a round
// of few tiles, but so do the 128-row tiles that compete for it: over 424 sizes (512..8192 rows by 128, the projections of Qwen3-0.6B and Qwen3-8B, weights from HBM) the rows that these lines deal take within
// 1 % of the best dealing at all but 3, those of a line that follows a round's tiles ((17.5 + 6 max(0, n - 128) / 128) K/1024 + 1.5, a launch 5.5) at all but 15, and 0.06 % and 0.12 % over the best in
// all (gate and up of 0.6B, 6272..6528 rows: 76.3..76.8 us so, 79.8..80.5 by that line; 3328 rows 48.9 and 47.4).  us of the two kernels, 256 / 128: qkv of 0.6B 25.4 / 19.8 at 2048 tokens, 25.9 / 28.9 at
// 2560, 49.4 / 45.6 at 4608; o_proj 44.4 / 36.8 at 8192; 8B qkv 76.1 / 65.0 at 1280, 78.9 / 104 at 1536, 166 / 163 at 3072.  N = W rows
static double cost_256(int64_t T, int64_t K, int64_t N) {
    const int64_t tiles = ((N + 255) / 256) * ((T + 255) / 256);
    return (double)((tiles + 255) / 256) * (18.5 * (double)K / 1024.0 + 8.0);
}
static double cost_128(int64_t T, int64_t K, int64_t N) {
    const int64_t tiles = ((N + 127) / 128) * ((T + 127) / 128);
    const double kk = (double)K / 1024.0, rounds = (double)tiles / 256.0;
    if (tiles <= 256) return 9.4 * kk + 3.5;
    // (two workgroups share a CU: up to 512 tiles a last part of a round is one of the two; what begins a third round lasts a whole one.  us of a Qwen3-0.6B prompt, a last part of any round counted
    // half / so: 1408 tokens 3703 / 3650, 2176 4944 / 4675, 2304 5022 / 4766; 8B, 2900 tokens 39160 / 38850)
    return (tiles <= 512 ? 0.5 * (rounds + (double)((tiles + 255) / 256)) : (double)((tiles + 255) / 256)) * (8.0 * kk + 1.2) + 2.0;
}
static inline bool prefer_256(int64_t T, int64_t K, int64_t N) { return cost_256(T, K, N) < cost_128(T, K, N); }
bool gemm256_preferred(int64_t T, int64_t K, int64_t N, int64_t ldx) { return gemm256_ok(T, K, N, ldx) && prefer_256(T, K, N); }
// Rows [0, r) of a product on 256x256 tiles and the others on 128x128 ones (0: all on the latter, T: all on the former).  A last round of 256x256 tiles costs as much as a full one however few
// they are, so the rows that do not fill one go to the small tiles where that is estimated 4 % cheaper: both kernels sum a row's products in the same order, and a row has the same bits on either.
// us, the better kernel for all rows / split: 8B qkv 163 / 137 at 3072 rows, o_proj 168 / 136 at 4608, down_proj 482 / 380 at 4608, 489 / 416 at 5120; 0.6B gate_up 46.8 / 42.0 at 3072, qkv 44.1 / 38.8
// at 4352, 45.6 / 40.2 at 4608, o_proj 78.6 / 62.8 at 17000.
static int64_t rows_on_256(int64_t T, int64_t K, int64_t N) {
    const double c256 = cost_256(T, K, N), c128 = cost_128(T, K, N);
    int64_t best = c256 < c128 ? T : 0;
    double least = 0.96 * std::min(c256, c128);
    const int64_t tn = (N + 255) / 256;
    for (int64_t rounds = 1; rounds * 256 / tn * 256 <= T - 65; ++rounds) {
        const int64_t r = rounds * 256 / tn * 256;
        const double c = r > 0 ? cost_256(r, K, N) + cost_128(T - r, K, N) : 1e30;
        if (c < least) { least = c; best = r; }
    }
    return best;
}
// where the 256x256 kernel was estimated the faster one before both kernels' times were fitted anew: what nvr_linear_add_residual takes does not move with them
static bool former_256(int64_t T, int64_t K, int64_t N) {
    const int64_t t256 = ((N + 255) / 256) * ((T + 255) / 256), t128 = ((N + 127) / 128) * ((T + 127) / 128);
    const double kk = (double)K / 1024.0, c128 = (t128 <= 256 ? 15.0 * kk : (double)((t128 + 511) / 512) * 21.0 * kk) + 5.0;
    return (double)((t256 + 255) / 256) * (17.0 * kk + 20.0) < c128;
}
bool linear_add_residual_ok(int64_t T, int64_t K, int64_t N, int64_t ldx) { return gemm256_ok(T, K, N, ldx) && former_256(T, K, N); }
// a product with an epilogue that the 256x256 kernel alone has (GELU, max(y, 0)^2): elsewhere it is a launch of its own that reads and writes the rows again, so the line lies where either estimate
// prefers the kernel.  us of product and GELU, tiles and a launch of its own / so: 4096 columns, K = 1024 1800 rows 32.3 / 32.6, 2064 40.6 / 31.9, 2304 40.5 / 30.8; 8192 columns, K = 2048 2064 rows
// 97.8 / 92.6, 2560 109 / 95.1
bool gemm256_epilogue_preferred(int64_t T, int64_t K, int64_t N, int64_t ldx) { return gemm256_ok(T, K, N, ldx) && (prefer_256(T, K, N) || former_256(T, K, N)); }
int64_t stream_row_limit() { return 64; }
// split-k GEMMs of the N = hidden projections: LDS tiles beyond the streaming kernels' rows — and from 33 rows on over large weights, where the
// streaming split-k kernel walks the weights once per 32-row block (Qwen3-8B bs 64: o + down 92 us per layer against 46 us at bs 128 on the tiles;
// up to 32 rows the streaming kernel stays ahead: Qwen3-8B bs 32 / 16 5.00 / 4.20 ms per step against 5.10 / 4.38 on 32-token tiles, 8 slices)
bool splitk_prefers_tiles(int64_t T, int64_t K, int64_t N) { return T > stream_row_limit() || (T > 32 && N * K * 2 >= (24ll << 20)); }
// ... and with 8 slices whatever the weights: 64 rows, N = 1024, K = 2048 / 3072 5.3 / 6.6 us as two blocks and 2 slices, 4.4 / 5.5 on the tiles
constexpr int64_t TILE_SLICES = 8;
// k-slices of the N = hidden GEMMs of a decode-sized step (linear_splitk): reach ~256 workgroups with slices of >= 256 columns that are
// multiples of 64
int decode_splitk_slices(int64_t T, int64_t K, int64_t N) {
    int64_t S = 1;
    const int64_t tiles = (N / 16) * ((T + 31) / 32);
    while (S < 4 && tiles * S < 256 && K % (32 * S * 2) == 0 && K / (S * 2) >= 128) S *= 2;
    return (int)S;
}
bool stream_preferred(int64_t T, int64_t N) {
    // up to 64 rows the weight-streaming kernel; beyond, the LDS-tiled kernel with 32- / 64-token tiles (ctx 256: bs 66 2.20 -> 1.83 ms/step, bs 96 2.48 -> 2.15, bs 128 2.82 -> 2.23) from
    // 192 Ki outputs on.  us, streamed / tiles, widths of 256 to 4096 columns: K = 1024 7.0 / 7.0 at 200-240 Ki outputs, 9.3 / 7.0 at 290-380 Ki (80 rows of 4096 columns 9.1 / 7.9, 96 rows
    // 10.0 / 7.9), K = 2048 12.2 / 11.2 and 17.2 / 11.3, K = 4096 21.7 / 20.5 and 31.5 / 21; K = 512 4.2-4.8 / 4.9 and 5.9 / 4.9: there the line could lie at 260 Ki, but one line keeps prompts of
    // like sizes on one kernel.
    return T <= stream_row_limit() || T * N <= 192 * 1024;
}
static inline int waves_for(int64_t K) { return K >= 2048 ? 16 : (K >= 1024 ? 8 : 4); }

static int launch_check(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "%s launch failed: %s", what, hipGetErrorString(e));
    return 0;
}

// outputs up to which a product with GELU stays on the streaming kernel: on tiles the product is rounded before GELU, by a launch of its own.  us a layer, tiles and that launch / so: 200 / 300 /
// 384 rows of 1024 columns, K = 256 49.0 50.6 50.8 / 44.4 46.4 49.1, 100 / 192 rows of 2048, K = 512 53.9 55.5 / 49.9 53.2, 72 / 96 rows of 4096, K = 1024 68.5 69.5 / 67.0 68.9
constexpr int64_t GELU_STREAM = 384 * 1024;
// gelu (not null): in, whether y = gelu(x . W^T) is wanted; out, whether the kernel this shape takes has applied it
static int linear_routed(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, void *y, bool y_f32, hipStream_t s, const half_bits *Wt, bool *gelu) {
    const bool act = gelu && *gelu;
    if (K % 32 || N % 16 || ldx % 8)
        return nvr::fail(NVR_ERR_UNSUPPORTED, "linear: K=%ld must be a multiple of 32, N=%ld of 16, ldx=%ld of 8",
                         (long)K, (long)N, (long)ldx);
    if (T == 0) return 0;
    // prompts: rows_on_256; up to 64 rows and for small T * N the weight-streaming kernel over blocks of 32 rows
    if (!y_f32 && gemm256_ok(T, K, N, ldx)) {
        if (act) { if (gemm256_epilogue_preferred(T, K, N, ldx)) return gemm256_gelu(x, ldx, W, T, K, N, (half_bits *)y, s); }
        else if (const int64_t r = rows_on_256(T, K, N)) {
            if (int rc = gemm256(x, ldx, W, r, K, N, (half_bits *)y, s)) return rc;
            return r == T ? 0 : gemm_tiled(x + r * ldx, ldx, W, T - r, K, N, (half_bits *)y + r * N, s, Wt);
        }
    }
    if (gelu) *gelu = false;                               // (the tiled and the streaming kernel have no such epilogue)
    if (!y_f32 && gemm_tiled_ok(T, K, N, ldx) && !stream_preferred(T, N) && !(act && T * N <= GELU_STREAM)) return gemm_tiled(x, ldx, W, T, K, N, (half_bits *)y, s, Wt);
    if (!y_f32 && linear_stream_ok(T, K, N, ldx)) return linear_stream(x, ldx, W, T, K, N, (half_bits *)y, s, Wt);   // large weights
    const half_t *xx = (const half_t *)x, *ww = (const half_t *)(Wt ? Wt : W);
    const int t = (int)T, k = (int)K, n = (int)N;
    LinEpi e{};
    e.tiled = Wt != nullptr;
    if (act && !y_f32) { e.gelu = 1; *gelu = true; }
    const int64_t mtiles = (T + 31) / 32;
    // wide GEMMs (LM head, prefill slabs): 64 columns per workgroup amortise the x fragments; narrow ones keep
    // 16 columns per workgroup (more workgroups) and split k over more waves (more bytes in flight per CU)
    const bool wide = (N / 64) * (T <= 16 ? 1 : mtiles) >= 1024;
    const int wv = waves_for(K);
#define NVR_LIN(NT_, MT_, WV_)                                                                      \
    do {                                                                                            \
        const unsigned gx = (unsigned)((N + 16 * NT_ - 1) / (16 * NT_));                            \
        if (y_f32) launch<NT_, MT_, WV_, EPI_F32>(xx, ldx, ww, t, k, n, y, e, gx, s);               \
        else launch<NT_, MT_, WV_, EPI_F16>(xx, ldx, ww, t, k, n, y, e, gx, s);                     \
    } while (0)
    // narrow outputs (N/16 < 128 column tiles: the row-parallel GEMMs of a tensor-parallel rank) with 17..32 tokens: 16-token
    // workgroups double the workgroup count (the W tile of a column block is read by both token blocks from the same XCD's L2):
    // 6.1 vs 8.2 us at K = 2048, N = 1024 (scratch/gemm_chain.py)
    const bool mt1 = T <= 16 || (!wide && T <= 32 && N / 16 < 128);
    if (mt1) {
        if (wide) NVR_LIN(4, 1, 4);
        else if (wv == 16) NVR_LIN(1, 1, 16);
        else if (wv == 8) NVR_LIN(1, 1, 8);
        else NVR_LIN(1, 1, 4);
    } else {
        if (wide) NVR_LIN(4, 2, 4);
        else if (wv == 16) NVR_LIN(1, 2, 16);
        else if (wv == 8) NVR_LIN(1, 2, 8);
        else NVR_LIN(1, 2, 4);
    }
#undef NVR_LIN
    return launch_check("linear");
}

int linear(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, void *y,
           bool y_f32, hipStream_t s, const half_bits *Wt) {
    return linear_routed(x, ldx, W, T, K, N, y, y_f32, s, Wt, nullptr);
}

int linear_gelu(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, half_bits *y, bool *applied, hipStream_t s) {
    *applied = true;
    return linear_routed(x, ldx, W, T, K, N, y, false, s, nullptr, applied);
}

bool linear_resid_ok(int64_t T, int64_t K, int64_t N, int64_t ldx) { return gemm_tiled_ok(T, K, N, ldx) && !stream_preferred(T, N) && N % 8 == 0; }
int linear_resid(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, half_bits *h, hipStream_t s, const half_bits *Wt) {
    if (!linear_resid_ok(T, K, N, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "linear_resid: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    const int64_t r = gemm256_ok(T, K, N, ldx) ? rows_on_256(T, K, N) : 0;
    if (r > 0) if (int rc = gemm256_resid(x, ldx, W, r, K, N, h, s)) return rc;
    return r == T ? 0 : gemm_tiled_resid(x + r * ldx, ldx, W, T - r, K, N, h + r * N, s, Wt);
}

// split-k over S workgroups per tile: slabs[z][T][N] f32 partial sums (summed by add_rmsnorm_slabs); the narrow
// row-parallel GEMMs of the decode step (o_proj, down_proj: N = hidden) reach all 256 CUs this way
int linear_splitk(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, int64_t S,
                  float *slabs, hipStream_t s, const half_bits *Wt) {
    if (K % (32 * S) || N % 16 || ldx % 8 || S < 1)
        return nvr::fail(NVR_ERR_UNSUPPORTED, "linear_splitk: K=%ld must be a multiple of 32*S (S=%ld), N=%ld of 16", (long)K, (long)S, (long)N);
    if (T == 0) return 0;
    if ((splitk_prefers_tiles(T, K, N) || (T > 32 && S >= TILE_SLICES)) && gemm_tiled_splitk_ok(T, K, N, S, ldx)) return gemm_tiled_splitk(x, ldx, W, T, K, N, S, slabs, s, Wt);   // LDS tiles
    LinEpi e{};
    e.kslice = (int32_t)(K / S); e.slab_stride = T * N;
    if (Wt) { W = Wt; e.tiled = 1; }
    const unsigned gx = (unsigned)(N / 16);
    if (N * K * 2 >= (24ll << 20) && N % 64 == 0) {
        // large weights (Qwen3-8B o/down: N = 4096): 64 output columns per workgroup so that an x fragment feeds four weight
        // tiles (x costs half the weight bytes instead of twice), 8 waves; with S = 4: 10.8 / 29.5 us vs 15.5 / 45 us for the
        // 16-column kernel at K = 4096 / 12288 (scratch/splitk_8b.py)
        if (!slab_takes(e.kslice)) {
            if (T <= 16) launch<4, 1, 8, EPI_SLAB>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K, (int)N, slabs, e, (unsigned)(N / 64), s, (unsigned)S);
            else launch<4, 2, 8, EPI_SLAB>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K, (int)N, slabs, e, (unsigned)(N / 64), s, (unsigned)S);
            return launch_check("linear_splitk");
        }
        const int mt = T <= 16 ? 1 : 2;
        const dim3 grid((unsigned)(N / 64), (unsigned)((T + 16 * mt - 1) / (16 * mt)), (unsigned)S);
        if (mt == 1) linear_slab_kernel<1><<<grid, dim3(512), 0, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K, (int)N, slabs, e.kslice, e.slab_stride, e.tiled);
        else linear_slab_kernel<2><<<grid, dim3(512), 0, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K, (int)N, slabs, e.kslice, e.slab_stride, e.tiled);
        return launch_check("linear_splitk");
    }
    if (T <= 16) launch<1, 1, 4, EPI_SLAB>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K, (int)N, slabs, e, gx, s, (unsigned)S);
    else launch<1, 2, 4, EPI_SLAB>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K, (int)N, slabs, e, gx, s, (unsigned)S);
    return launch_check("linear_splitk");
}

// 56 rows and more of weights that the large-weight kernel does not take: the two blocks of 32 rows each read x for every 16 columns.  us of 56 / 64 rows, blocks | tiles: K = 512, I = 2304
// 5.2 5.4 | 5.3 5.9, 3840 6.1 6.3 | 6.2 6.3, 4864 7.6 7.8 | 6.4 6.4; K = 768, I = 2304 7.0 7.4 | 7.0 7.4, 3840 8.1 8.5 | 7.5 7.6; K = 1024, I = 2304 8.3 8.7 | 8.3 8.4, 3072 8.9 9.3 | 8.3 8.4,
// 4864 11.9 12.5 | 9.0 9.2; K = 2560, I = 3072 20.4 21.3 | 17.1 17.5, 4864 29.5 31.1 | 19.7 19.9
static bool glu_on_tiles(int64_t T, int64_t K, int64_t I, int64_t ldx) {
    return gemm_tiled_ok(T, K, I, ldx) && I % 64 == 0 && (!stream_preferred(T, 2 * I) || (T >= 56 && T * I > (K >= 768 ? 128 : 256) * 1024 && !linear_stream_silu_ok(T, K, I, ldx)));
}
Ahead linear_silu_ahead(const half_bits *W, int64_t T, int64_t K, int64_t I, const half_bits *Wt) {
    if (2 * I * K * 2 > 24ll << 20 || K % 32 || I % 128) return {};
    if (gemm256_silu_ok(T, K, I, K) && rows_on_256(T, K, 2 * I) > 0) return {};
    return glu_on_tiles(T, K, I, K) ? gemm_tiled_silu_ahead(Wt ? Wt : W, T, K, I) : Ahead{};
}

// gate_up GEMM + SiluAndMul: W [2I, K] (gate rows then up rows), out [T, I]
static int linear_glu(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t I,
                      half_bits *out, hipStream_t s, const half_bits *Wt, bool gelu) {
    if (K % 32 || I % 16 || ldx % 8)
        return nvr::fail(NVR_ERR_UNSUPPORTED, "linear_silu_mul: K=%ld must be a multiple of 32, I=%ld of 16", (long)K, (long)I);
    if (T == 0) return 0;
    if (const int64_t r = gemm256_silu_ok(T, K, I, ldx) ? rows_on_256(T, K, 2 * I) : 0) {
        if (int rc = gelu ? gemm256_gelu_mul(x, ldx, W, r, K, I, out, s) : gemm256_silu_mul(x, ldx, W, r, K, I, out, s)) return rc;
        return r == T ? 0 : gemm_tiled_silu_mul(x + r * ldx, ldx, W, T - r, K, I, out + r * I, s, gelu, Wt);
    }
    if (glu_on_tiles(T, K, I, ldx)) return gemm_tiled_silu_mul(x, ldx, W, T, K, I, out, s, gelu, Wt);
    if (linear_stream_silu_ok(T, K, I, ldx)) return linear_stream_silu_mul(x, ldx, W, T, K, I, out, s, Wt, gelu);              // large weights
    const half_t *xx = (const half_t *)x, *ww = (const half_t *)(Wt ? Wt : W);
    LinEpi e{};
    e.tiled = Wt != nullptr; e.gelu = gelu ? 1 : 0;
    const unsigned gx = (unsigned)(I / 16);
    const int wv = waves_for(K);
    // few column tiles (the shard of a tensor-parallel rank): 16-token workgroups double the workgroup count (the second token
    // block finds its W tile in the XCD's L2) and long rows are split over 16 waves — same rule as linear()
    const bool narrow = I / 16 < 128 && T <= 32;
    if (narrow && wv == 16) {
        launch<2, 1, 16, EPI_SILU>(xx, ldx, ww, (int)T, (int)K, (int)I, out, e, gx, s);
    } else if (T <= 16 || narrow) {
        if (wv >= 8) launch<2, 1, 8, EPI_SILU>(xx, ldx, ww, (int)T, (int)K, (int)I, out, e, gx, s);
        else launch<2, 1, 4, EPI_SILU>(xx, ldx, ww, (int)T, (int)K, (int)I, out, e, gx, s);
    } else {
        if (wv >= 8) launch<2, 2, 8, EPI_SILU>(xx, ldx, ww, (int)T, (int)K, (int)I, out, e, gx, s);
        else launch<2, 2, 4, EPI_SILU>(xx, ldx, ww, (int)T, (int)K, (int)I, out, e, gx, s);
    }
    return launch_check("linear_silu_mul");
}
int linear_silu_mul(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t I, half_bits *out, hipStream_t s, const half_bits *Wt) {
    return linear_glu(x, ldx, W, T, K, I, out, s, Wt, false);
}
// the same with gelu (tanh form) in silu's place
int linear_gelu_mul(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t I, half_bits *out, hipStream_t s) {
    return linear_glu(x, ldx, W, T, K, I, out, s, nullptr, true);
}

// gate_up GEMM + the clamped gated unit of a layer list: W [2I, K] (gate rows, then up rows), out [T, ldo].  Few rows, whose product the weight-row kernel takes: the unit
// is a launch of its own otherwise, and a launch behind a launch is about 5 us whatever it holds (16 rows of 1024, I = 3072: 11.3 -> 6.3 us together).  Shapes of the LDS tiles, routed as linear()
// routes the plain product: the unit by itself reads both halves of every row again and the product writes twice the columns (1024 wide, I = 3072: 16384 rows 178 + 63 us -> 195, 4096 52 + 17 -> 67;
// the unit on v_rcp and the fast exponential was 24 us faster at 16384, but then a row's unit would depend on the size of its step, and be off by a few last places of f32 more).
static bool clamped_glu_on_tiles(int64_t T, int64_t K, int64_t I, int64_t ldx) {
    return K % 32 == 0 && I % 64 == 0 && gemm_tiled_ok(T, K, I, ldx) && ((gemm256_silu_ok(T, K, I, ldx) && rows_on_256(T, K, 2 * I) > 0) || !stream_preferred(T, 2 * I));
}
bool linear_clamped_glu_ok(const half_bits *x, int64_t ldx, int64_t T, int64_t K, int64_t I, const half_bits *out, int64_t ldo) {
    if (((uintptr_t)x | (uintptr_t)out) % 16 == 0 && ldo % 8 == 0 && ldo >= I && clamped_glu_on_tiles(T, K, I, ldx)) return true;
    return T <= 32 && K % 32 == 0 && I % 16 == 0 && ldx % 8 == 0 && ldo % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)out % 8 == 0 && !linear_stream_silu_ok(T, K, I, ldx);
}
int linear_clamped_glu(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t I, float limit, float alpha, half_bits *out, int64_t ldo, hipStream_t s) {
    if (!linear_clamped_glu_ok(x, ldx, T, K, I, out, ldo)) return nvr::fail(NVR_ERR_UNSUPPORTED, "linear_clamped_glu: T=%ld K=%ld I=%ld", (long)T, (long)K, (long)I);
    if (T == 0) return 0;
    if (T > 32) {
        const int64_t r = gemm256_silu_ok(T, K, I, ldx) ? rows_on_256(T, K, 2 * I) : 0;
        if (r > 0) if (int rc = gemm256_clamped_glu(x, ldx, W, r, K, I, limit, alpha, out, ldo, s)) return rc;
        return r == T ? 0 : gemm_tiled_clamped_glu(x + r * ldx, ldx, W, T - r, K, I, limit, alpha, out + r * ldo, ldo, s);
    }
    LinEpiClamp e{};
    e.limit = limit; e.alpha = alpha; e.ldy = ldo;
    const unsigned gx = (unsigned)(I / 16);
    const half_t *xx = (const half_t *)x, *ww = (const half_t *)W;
    const int wv = waves_for(K);
    if (T <= 16 || I / 16 < 128) {
        if (wv >= 8) launch<2, 1, 8, EPI_CLAMP>(xx, ldx, ww, (int)T, (int)K, (int)I, out, e, gx, s);
        else launch<2, 1, 4, EPI_CLAMP>(xx, ldx, ww, (int)T, (int)K, (int)I, out, e, gx, s);
    } else {
        if (wv >= 8) launch<2, 2, 8, EPI_CLAMP>(xx, ldx, ww, (int)T, (int)K, (int)I, out, e, gx, s);
        else launch<2, 2, 4, EPI_CLAMP>(xx, ldx, ww, (int)T, (int)K, (int)I, out, e, gx, s);
    }
    return launch_check("linear_clamped_glu");
}

// y = x . W^T [T, N] and the clamped gated unit of x2 . W2^T [T, ldo] in one launch, where both take the kernel of few rows with the same rows and waves to a workgroup: the routes of linear() and
// linear_clamped_glu().  A launch of 5-7 us a layer is
// saved: us a request batch of a 4-layer list (width 1024, I = 3072), two launches / one: 1 request of 64 + 32 tokens 5009 / 4598, 8 of 100 + 32 5774 / 5380, 16 of 1024 + 32 10334 / 9920, 24 of 100 + 32
// 7405 / 7025.
bool linear_beside_clamped_glu_ok(const half_bits *x, const half_bits *x2, int64_t ldx, int64_t T, int64_t K, int64_t N, int64_t I, const half_bits *y, const half_bits *out, int64_t ldo) {
    if (((uintptr_t)x & 15) || ((uintptr_t)y & 7) || T < 1 || T > 32 || K % 32 || N % 16 || ldx % 8 || waves_for(K) == 16 || !linear_clamped_glu_ok(x2, ldx, T, K, I, out, ldo)) return false;
    if ((N / 64) * (T <= 16 ? 1 : (T + 31) / 32) >= 1024 || linear_stream_ok(T, K, N, ldx) || gemm256_ok(T, K, N, ldx)) return false;
    return (T <= 16 || N / 16 < 128) == (T <= 16 || I / 16 < 128);
}
int linear_beside_clamped_glu(const half_bits *x, const half_bits *x2, int64_t ldx, const half_bits *W, const half_bits *W2, int64_t T, int64_t K, int64_t N, int64_t I, float limit, float alpha, half_bits *y,
                              half_bits *out, int64_t ldo, hipStream_t s) {
    if (!linear_beside_clamped_glu_ok(x, x2, ldx, T, K, N, I, y, out, ldo))
        return nvr::fail(NVR_ERR_UNSUPPORTED, "linear beside linear_clamped_glu: T=%ld K=%ld N=%ld I=%ld", (long)T, (long)K, (long)N, (long)I);
    const bool mt1 = T <= 16 || I / 16 < 128;
    const dim3 grid((unsigned)(I / 16 + N / 16), (unsigned)((T + (mt1 ? 15 : 31)) / (mt1 ? 16 : 32)));
#define NVR_PAIR(MT_, WV_) linear_beside_unit_kernel<MT_, WV_><<<grid, dim3(64 * WV_), 0, s>>>((const half_t *)x, (const half_t *)x2, ldx, (const half_t *)W, (const half_t *)W2, (int)T, (int)K, (int)N, \
                                                                                              (int)I, (half_t *)y, (half_t *)out, ldo, limit, alpha)
    if (waves_for(K) == 8) { if (mt1) NVR_PAIR(1, 8); else NVR_PAIR(2, 8); }
    else { if (mt1) NVR_PAIR(1, 4); else NVR_PAIR(2, 4); }
#undef NVR_PAIR
    return launch_check("linear beside linear_clamped_glu");
}

// qkv GEMM + RoPE on q,k heads + store of k,v rows into the paged caches
int linear_qkv_rope_store(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t H,
                          int64_t KVH, int64_t D, const int64_t *positions, const int32_t *slots, const float *cos_t,
                          const float *sin_t, half_bits *qkv, half_bits *k_cache, half_bits *v_cache, hipStream_t s, const half_bits *Wt,
                          bool kv_cache_only) {
    if (K % 32 || D % 16 || ldx % 8)
        return nvr::fail(NVR_ERR_UNSUPPORTED, "linear_qkv_rope_store: K=%ld must be a multiple of 32, D=%ld of 16", (long)K, (long)D);
    if (T == 0) return 0;
    if (const int64_t r = gemm256_rope_ok(T, K, H, KVH, D, ldx) ? rows_on_256(T, K, (H + 2 * KVH) * D) : 0) {
        if (int rc = gemm256_qkv_rope_store(x, ldx, W, r, K, H, KVH, D, positions, slots, cos_t, sin_t, qkv, k_cache, v_cache, s, kv_cache_only)) return rc;
        return r == T ? 0 : gemm_tiled_qkv_rope_store(x + r * ldx, ldx, W, T - r, K, H, KVH, D, positions + r, slots ? slots + r : nullptr, cos_t, sin_t, qkv + r * (H + 2 * KVH) * D, k_cache, v_cache, s, Wt, kv_cache_only);
    }
    if (gemm_tiled_ok(T, K, (H + 2 * KVH) * D, ldx) && 128 % D == 0 && !stream_preferred(T, (H + 2 * KVH) * D))
        return gemm_tiled_qkv_rope_store(x, ldx, W, T, K, H, KVH, D, positions, slots, cos_t, sin_t, qkv, k_cache, v_cache, s, Wt, kv_cache_only);
    if (linear_stream_rope_ok(T, K, H, KVH, D, ldx))                                                                  // large weights
        return linear_stream_qkv_rope_store(x, ldx, W, T, K, H, KVH, D, positions, slots, cos_t, sin_t, qkv, k_cache, v_cache, s, Wt);
    const half_t *xx = (const half_t *)x, *ww = (const half_t *)(Wt ? Wt : W);
    LinEpi e{};
    e.tiled = Wt != nullptr;
    e.pos = positions; e.slots = slots; e.cos_t = cos_t; e.sin_t = sin_t; e.kc = (half_t *)k_cache; e.vc = (half_t *)v_cache;
    e.H = (int32_t)H; e.KVH = (int32_t)KVH; e.D = (int32_t)D;
    const int N = (int)((H + 2 * KVH) * D);
    const unsigned gx = (unsigned)(N / 16);
    const int wv = waves_for(K);
    const bool narrow = N / 16 < 128 && T <= 32;                 // see linear_silu_mul
    if (narrow && wv == 16) {
        launch<1, 1, 16, EPI_ROPE>(xx, ldx, ww, (int)T, (int)K, N, qkv, e, gx, s);
    } else if (T <= 16 || narrow) {
        if (wv >= 8) launch<1, 1, 8, EPI_ROPE>(xx, ldx, ww, (int)T, (int)K, N, qkv, e, gx, s);
        else launch<1, 1, 4, EPI_ROPE>(xx, ldx, ww, (int)T, (int)K, N, qkv, e, gx, s);
    } else {
        if (wv >= 8) launch<1, 2, 8, EPI_ROPE>(xx, ldx, ww, (int)T, (int)K, N, qkv, e, gx, s);
        else launch<1, 2, 4, EPI_ROPE>(xx, ldx, ww, (int)T, (int)K, N, qkv, e, gx, s);
    }
    return launch_check("linear_qkv_rope_store");
}

// As linear() routes the plain product: a last norm's launch behind it read and wrote every row once more (509 rows of 16 + 8 + 8 heads 4.2 us, 3815 rows 14.6, 3062 rows of 32 + 8 + 8 18.7).
bool linear_qkv_norm_rope_store_ok(int64_t T, int64_t K, int64_t H, int64_t KVH, int64_t D, int64_t ldx) {
    const int64_t N = (H + 2 * KVH) * D;
    return D == 128 && K % 32 == 0 && gemm_tiled_ok(T, K, N, ldx) && ((gemm256_rope_ok(T, K, H, KVH, D, ldx) && rows_on_256(T, K, N) > 0) || !stream_preferred(T, N));
}
int linear_qkv_norm_rope_store(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t H, int64_t KVH, int64_t D, const int64_t *positions, const int32_t *slots,
                               const float *cos_t, const float *sin_t, half_bits *qkv, half_bits *k_cache, half_bits *v_cache, const QkNorm &norm, hipStream_t s, const half_bits *Wt, bool kv_cache_only) {
    const uintptr_t at = (uintptr_t)qkv | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)norm.q_w | (uintptr_t)norm.k_w | (uintptr_t)cos_t | (uintptr_t)sin_t;
    if (!linear_qkv_norm_rope_store_ok(T, K, H, KVH, D, ldx) || (at & 15)) return nvr::fail(NVR_ERR_UNSUPPORTED, "linear_qkv_norm_rope_store: T=%ld K=%ld D=%ld", (long)T, (long)K, (long)D);
    const int64_t N = (H + 2 * KVH) * D, r = gemm256_rope_ok(T, K, H, KVH, D, ldx) ? rows_on_256(T, K, N) : 0;
    if (r > 0) if (int rc = gemm256_qkv_rope_store(x, ldx, W, r, K, H, KVH, D, positions, slots, cos_t, sin_t, qkv, k_cache, v_cache, s, kv_cache_only, &norm)) return rc;
    return r == T ? 0 : gemm_tiled_qkv_rope_store(x + r * ldx, ldx, W, T - r, K, H, KVH, D, positions + r, slots ? slots + r : nullptr, cos_t, sin_t, qkv + r * N, k_cache, v_cache, s, Wt, kv_cache_only, &norm);
}

// ---- products of a decode step of few rows whose workgroups form RMSNorm(h + slabs) themselves (linear_skinny_kernel, NORM)
// (three and four rows: from the width on at which the products behind a launch of its own split k over the same eight waves, so that the step's bits are theirs)
// (slabs: 2 or 4 of a split product; in front of the gate and up product also 8, one per kv head, of an attention with the output product in it)
static bool norm_linear_ok(int64_t T, int64_t K, int64_t S, int64_t most) {
    return T >= 1 && T <= NORM_ROWS && (T <= 2 || waves_for(K) == 8) && K % 256 == 0 && T * K <= NORM_ELEMS && (S == 2 || S == 4 || S == 8) && S <= most;
}
template <int NT, int EPI>
static int norm_launch(const NormIn &nm, const half_bits *W, int64_t T, int64_t K, int64_t N, void *y, const LinEpi &le, int64_t gx, bool tiled, hipStream_t s, const char *what) {
    if (!norm_linear_ok(T, K, nm.S, EPI == EPI_SILU ? 8 : 4)) return nvr::fail(NVR_ERR_UNSUPPORTED, "%s: T=%ld K=%ld, %d slabs", what, (long)T, (long)K, nm.S);
    LinEpiNorm e{};
    static_cast<LinEpi &>(e) = le;
    e.norm = nm; e.tiled = tiled;
    if constexpr (EPI == EPI_SILU)
        if (nm.S > 4) {
            linear_skinny_kernel<NT, 1, 8, EPI, 8><<<dim3((unsigned)gx), dim3(512), (size_t)(T * (K + 8) * 2), s>>>(nullptr, 0, (const half_t *)W, (int)T, (int)K, (int)N, y, e);
            return launch_check(what);
        }
    linear_skinny_kernel<NT, 1, 8, EPI, 4><<<dim3((unsigned)gx), dim3(512), (size_t)(T * (K + 8) * 2), s>>>(nullptr, 0, (const half_t *)W, (int)T, (int)K, (int)N, y, e);
    return launch_check(what);
}
// which products of these shapes take the weight-streaming kernel above at so few rows (large weights have a kernel of their own)
bool norm_linear_plain_ok(int64_t T, int64_t K, int64_t N, int64_t S) { return norm_linear_ok(T, K, S, 4) && N % 16 == 0 && !linear_stream_ok(T, K, N, K); }
bool norm_linear_silu_ok(int64_t T, int64_t K, int64_t I, int64_t S) { return norm_linear_ok(T, K, S, 8) && I % 16 == 0 && !linear_stream_silu_ok(T, K, I, K); }
bool norm_linear_rope_ok(int64_t T, int64_t K, int64_t H, int64_t KVH, int64_t D, int64_t S) { return norm_linear_ok(T, K, S, 4) && D % 16 == 0 && !linear_stream_rope_ok(T, K, H, KVH, D, K); }
int norm_linear(const NormIn &nm, const half_bits *W, int64_t T, int64_t K, int64_t N, half_bits *y, hipStream_t s, const half_bits *Wt) {
    return norm_launch<1, EPI_F16>(nm, Wt ? Wt : W, T, K, N, y, LinEpi{}, N / 16, Wt != nullptr, s, "norm + linear");
}
int norm_linear_silu_mul(const NormIn &nm, const half_bits *W, int64_t T, int64_t K, int64_t I, half_bits *out, hipStream_t s, const half_bits *Wt) {
    return norm_launch<2, EPI_SILU>(nm, Wt ? Wt : W, T, K, I, out, LinEpi{}, I / 16, Wt != nullptr, s, "norm + gate_up + silu");
}
int norm_linear_qkv_rope_store(const NormIn &nm, const half_bits *W, int64_t T, int64_t K, int64_t H, int64_t KVH, int64_t D, const int64_t *positions, const int32_t *slots,
                               const float *cos_t, const float *sin_t, half_bits *qkv, half_bits *k_cache, half_bits *v_cache, hipStream_t s, const half_bits *Wt) {
    LinEpi e{};
    e.pos = positions; e.slots = slots; e.cos_t = cos_t; e.sin_t = sin_t; e.kc = (half_t *)k_cache; e.vc = (half_t *)v_cache;
    e.H = (int32_t)H; e.KVH = (int32_t)KVH; e.D = (int32_t)D;
    const int64_t N = (H + 2 * KVH) * D;
    return norm_launch<1, EPI_ROPE>(nm, Wt ? Wt : W, T, K, N, qkv, e, N / 16, Wt != nullptr, s, "norm + qkv + rope");
}

}}  // namespace nvr::k / nvr::kb (NVR_DT_NS)
