// gemm_tiled.hip — LDS-tiled MFMA GEMM for the prefill regime (T >= 128 tokens): y[T,N] = x[T,K]·W[N,K]^T
// with the same three epilogues as the decode kernel (plain fp16, gate_up -> SiluAndMul, qkv -> RoPE + KV store).
// reference call sites as in linear.hip (linear.rs:354-356,228-239,437-439; activation.rs:46-63;
// rotary_embedding.rs:23-48; attention.rs:150-174).  Bound: MFMA (dense contraction, SURVEY §8d:
// 880.8 MFLOP per prefill token for Qwen3-0.6B).
//
// Structure:
//   workgroup = 4 waves = 128 (n) x 128 / 64 / 32 (m) output tile, BK = 64; wave (wn, wm) owns 64 x 64 / 32 / 16, MFMA tiles of v_mfma_f32_16x16x32_f16 (A = W rows, B = x rows, both
//   K-contiguous in memory);
//   both operand tiles are staged global -> LDS by global_load_lds_dwordx4 (16 B per lane, no VGPR round trip) into a ring of 2..4 K-tiles behind counted waits, and the fragments of a
//   k-step of 32 are read from LDS while the k-step in front of it is multiplied, so that one wave per SIMD keeps requests, LDS reads and products going at once (with the reads of a
//   K-tile in front of its products: K = 2048, N = 1024, 3814 tokens 24.3 us, this way 21.8, 2048 / 1000 tokens as two slices 11.1 / 9.4);
//   the tiles of a launch are dealt to the XCDs in compact blocks (TileMap: the same product 18.9);
//   what bounds it: a CU takes operand bytes in at 80-87 GB/s (loads alone take 22.4 us of K = 3072's 26.3, products and reads alone 20.1).
//   LDS image = [row][8 chunks of 16 B] with chunk' = chunk ^ (row & 7): the swizzle is applied to the per-lane
//   SOURCE address (the LDS destination of glds is lane-linear) and again on the ds_read_b128 address, so a
//   16-lane fragment read touches 8 distinct 16-B slots (2-way instead of 16-way conflicts).
//   A tiled copy of W (retile_weight) is read where there is one: a K-tile of 16 rows is then 2 KiB in a row in memory instead of 16 pieces of 128 B, 3-6 % of a launch whose weights come from
//   HBM (509 tokens, us: qkv 9.9 -> 9.5, down_proj in 4 slices 9.5 -> 9.2; 3814 tokens down_proj 32.4 -> 30.0).
// Row mapping of the A operand lets one lane hold what its epilogue needs: for SiluAndMul a wave's 4 n-tiles are
// [gate c, gate c+16, up c, up c+16]; for RoPE an n-tile is 8 columns of the first half of a head and their 8
// partners of the second half (the partner of lane l sits in lane l^32).
#include <cstdlib>
#include <type_traits>
#include "kernels.h"
#include "device_utils.h"
#include "../common.h"

namespace nvr { namespace NVR_DT_NS {

enum { TEPI_F16 = 0, TEPI_SILU = 2, TEPI_ROPE = 3, TEPI_LMHEAD = 4, TEPI_SLAB = 5, TEPI_RESID = 6, TEPI_QKN = 7, TEPI_CLAMP = 8 };     // RESID: y <- y + x.W^T, the product rounded first; QKN: heads of 128, RMSNorm over the columns of every q and k head, rotation, store

// Where a launch's tiles lie: nx column tiles (W rows) x ny token tiles x nz k-slices, numbered slice by slice, within a slice in strips of `width` column tiles, within a strip
// token tile by token tile.  Workgroups are dealt to the 8 XCDs in turn and each XCD has an L2 of its own, so XCD c takes the c-th eighth of that line: a compact block of tiles,
// whose rows of W and x it fetches once.
struct TileMap { int32_t nx, ny, width; };
struct TileAt { int32_t x, y, z; };
__device__ __forceinline__ TileAt tile_of(const TileMap &m) {
    const unsigned n = gridDim.x, xcd = blockIdx.x & 7, rem = n & 7;
    unsigned t = xcd * (n >> 3) + min(xcd, rem) + (blockIdx.x >> 3);
    TileAt at;
    const unsigned slice = (unsigned)m.nx * m.ny;
    at.z = t / slice; t -= at.z * slice;
    const unsigned strip = t / ((unsigned)m.width * m.ny), first = strip * m.width;
    t -= first * m.ny;
    const unsigned w = min((unsigned)m.width, m.nx - first);
    at.y = t / w; at.x = first + (t - at.y * w);
    return at;
}

struct TileEpi {
    const int64_t *pos; const int32_t *slots; const float *cos_t, *sin_t;
    half_t *kc, *vc;
    int32_t H, KVH, D, kv_cache_only;      // kv_cache_only: k and v go to the caches alone
    // TEPI_LMHEAD: f32 logits [T, N] (nullable) and the greedy arg-max of every row over this workgroup's 128 columns:
    // pval / pidx [column tile][T] (maximum, lowest index), merged by argmax_partials
    float *logits; float *pval; int32_t *pidx;
    // TEPI_SLAB: k-slice z owns k in [z*kslice, (z+1)*kslice) and writes its f32 partial tile to slabs[z][T][N]
    float *slabs; int64_t slab_stride; int32_t kslice;
    int32_t gelu;                          // TEPI_SILU: gelu (tanh form) instead of silu
    TileMap map;
    int32_t tiled;                         // W is the copy [rows/16][K/32][16][32] (retile_weight; TEPI_ROPE: its 16-row tiles are the n-tiles)
};
// What single instances need beyond it stays out of the others' arguments (Qwen3-0.6B in float16, us a step with / without the three numbers and two pointers in all of them: 33 sequences of 64..200
// keys 1336 / 1320, 48 of 64..300 1475 / 1461, 64 of 300 1631 / 1615)
struct TileEpiNorm : TileEpi { const half_t *qn_w, *kn_w; float qk_eps; };      // TEPI_QKN: the norms' weights
struct TileEpiClamp : TileEpi { float limit, alpha; int64_t ldo; };             // TEPI_CLAMP
template <int EPI> struct TileArgs { using type = TileEpi; };
template <> struct TileArgs<TEPI_QKN> { using type = TileEpiNorm; };
template <> struct TileArgs<TEPI_CLAMP> { using type = TileEpiClamp; };

constexpr int BM = 128, BN = 128, BK = 64;
constexpr int RING96 = 3;                                                 // K-tiles in the LDS ring of the 96-row kernel

// s_waitcnt vmcnt(N)
template <int N>
__device__ __forceinline__ void wait_requests() {
    static_assert(N <= 63, "vmcnt is a 6-bit count");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// K-tile kt has landed once at most the PER requests per thread of each of the `younger` (0..3) K-tiles behind it are outstanding
template <int PER>
__device__ __forceinline__ void wait_ring(int younger) {
    switch (younger) {
    case 0: wait_requests<0>(); break;
    case 1: wait_requests<PER>(); break;
    case 2: wait_requests<2 * PER>(); break;
    default: wait_requests<3 * PER>(); break;
    }
}

constexpr bool t_glu(int epi) { return epi == TEPI_SILU || epi == TEPI_CLAMP; }      // gate and up rows in one tile (CLAMP: clamped_unit, rows of y ldo apart)

// W row of local row r (0..15) of the workgroup's 16-row n-tile `t` (0..7)
template <int EPI>
__device__ __forceinline__ int tile_w_row(int bx, int t, int r, int N, const TileEpi &e) {
    if (t_glu(EPI)) {                             // N == I; the workgroup owns 64 output columns
        const int wn = t >> 2, nt = t & 3;
        return (nt >> 1) * N + bx * 64 + wn * 32 + (nt & 1) * 16 + r;
    }
    if (EPI == TEPI_ROPE) {
        const int g = bx * 8 + t, tph = e.D / 16, head = g / tph, c = g % tph;
        if (head < e.H + e.KVH) return head * e.D + (r < 8 ? c * 8 + r : e.D / 2 + c * 8 + (r - 8));
        return head * e.D + c * 16 + r;
    }
    return bx * BN + t * 16 + r;
}

// the same n-tile in the tiled copy
template <int EPI>
__device__ __forceinline__ int tile_w_block(int bx, int t, int N) {
    if (t_glu(EPI)) return ((t & 3) >> 1) * (N >> 4) + bx * 4 + (t >> 2) * 2 + (t & 1);
    return bx * 8 + t;
}

// NS: K-tiles in the LDS ring (tiled_launch).  MT: 16-token m-tiles per wave, 4 = the 128-token tile, 2 / 1 = a 64- / 32-token tile for batches of 65..~1000 rows, where 128 x 128 tiles
// leave half the CUs without a workgroup.
template <int EPI, int NS, int MT = 4>
__global__ __launch_bounds__(256, 2) void gemm_tiled_kernel(const half_t *__restrict__ x, int64_t ldx,
                                                         const half_t *__restrict__ W, int T, int K, int N, int NW,
                                                         half_t *__restrict__ y, typename TileArgs<EPI>::type epi) {
    // one LDS array (cdna guide §5 item 4a): [NS buffers][A 16 KiB | B 16 or 8 KiB]
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int BMt = 32 * MT;                                          // tokens per workgroup
    constexpr int BUF = (BN + BMt) * BK * 2;                              // bytes of one LDS buffer
    const TileAt at = tile_of(epi.map);
    static_assert(NS >= 2 && NS <= 4, "wait_ring counts up to three younger K-tiles");
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;
    const int wn = wave >> 1, wm = wave & 1;
    const int m0 = at.y * BMt;

    // staging: thread t copies 16-byte piece idx = i*256 + t (row = idx/8, LDS chunk c' = idx%8) of each operand tile
    const int kmul = epi.tiled ? 16 : 1;                                  // k -> element offset: (k / 32) * 512 in the tiled copy
    const half_t *asrc[4], *bsrc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int idx = i * 256 + threadIdx.x, row = idx >> 3, c = (idx & 7) ^ (row & 7);
        int wr = tile_w_row<EPI>(at.x, row >> 4, row & 15, N, epi);
        if (wr > NW - 1) wr = NW - 1;
        int xr = m0 + row; if (xr > T - 1) xr = T - 1;
        if (epi.tiled) asrc[i] = W + ((int64_t)min(tile_w_block<EPI>(at.x, row >> 4, N), NW / 16 - 1) * (K / 32) + (c >> 2)) * 512 + (row & 15) * 32 + (c & 3) * 8;
        else asrc[i] = W + (int64_t)wr * K + c * 8;
        bsrc[i] = x + (int64_t)xr * ldx + c * 8;                          // (rows >= BMt: unused)
        if (EPI == TEPI_SLAB) { asrc[i] += (int64_t)at.z * epi.kslice * kmul; bsrc[i] += (int64_t)at.z * epi.kslice; }
    }
    auto stage = [&](int buf, int k0) {
        char *a_dst = smem + buf * BUF, *b_dst = a_dst + BN * BK * 2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int piece = (i * 256 + wave * 64) * 16;               // wave-uniform LDS base; hardware adds lane*16
            __builtin_amdgcn_global_load_lds(asrc[i] + k0 * kmul, (__attribute__((address_space(3))) void *)(a_dst + piece), 16, 0, 0);
            if (i < MT) __builtin_amdgcn_global_load_lds(bsrc[i] + k0, (__attribute__((address_space(3))) void *)(b_dst + piece), 16, 0, 0);
        }
    };

    float4_t acc[4][MT];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};

    // TEPI_ROPE: the epilogue's inputs arrive UNDER the K loop instead of as three dependent round trips behind it (position -> cos / sin row -> rotate; cache
    // slot -> store).  Positions and slots are requested here, in front of the first operand tile, the cos / sin pieces once the positions are in.  A wave's four
    // n-tiles need 128 consecutive bytes of each table per token; lanes q and q + 2 need the same ones, so each requests two n-tiles' pieces and they trade them.
    // TEPI_QKN: a workgroup's columns are one head; behind the K loop a thread takes row j * 32 + tid / 8 and the pair of pieces tid % 8 (its positions, cosines, sines and norm weights are
    // requested here in the same way).
    constexpr bool QKN = EPI == TEPI_QKN, ROPE = EPI == TEPI_ROPE || QKN;
    int64_t rope_pos[MT];
    int rope_slot[MT];
    float4_t pre_cs[MT][2], pre_sn[MT][2];
    const int tph = EPI == TEPI_ROPE ? epi.D / 16 : 1, tsh = 31 - __clz(tph), heads = epi.H + 2 * epi.KVH;      // n-tiles per head: 1, 2, 4 or 8
    const int rope_head = QKN ? at.x : ROPE ? (at.x * 8 + wn * 4) >> tsh : 0;          // the head of the first of this wave's four n-tiles
    const bool rope_rot = ROPE && rope_head < epi.H + epi.KVH;
    half8_t norm_w[2];
    if (ROPE) {
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            // (as inline asm: a compiler-visible load makes hipcc drain vmcnt(0) at its first use, operand tiles in flight included; the values are complete
            //  once the first operand tile is, which is younger — see the pin there)
            const int m = m0 + (QKN ? j * 32 + ((int)threadIdx.x >> 3) : wm * (16 * MT) + j * 16 + r), mc = m < T ? m : T - 1;
            const int64_t *src = epi.pos + mc;
            asm volatile("global_load_dwordx2 %0, %1, off" : "=v"(rope_pos[j]) : "v"(src) : "memory");
            const int32_t *ss = epi.slots ? epi.slots + mc : reinterpret_cast<const int32_t *>(src);      // (no branch: a value in flight would be copied at its end)
            asm volatile("global_load_dword %0, %1, off" : "=v"(rope_slot[j]) : "v"(ss) : "memory");
        }
    }

    const int KT = (EPI == TEPI_SLAB ? epi.kslice : K) / BK;
    auto read_a = [&](const char *buf, int ks, int i) {
        const int arow = wn * 64 + i * 16 + r;
        return *reinterpret_cast<const half8_t *>(buf + (arow * 8 + ((ks * 4 + q) ^ (arow & 7))) * 16);
    };
    auto read_b = [&](const char *buf, int ks, int j) {
        const int brow = wm * (16 * MT) + j * 16 + r;
        return *reinterpret_cast<const half8_t *>(buf + BN * BK * 2 + (brow * 8 + ((ks * 4 + q) ^ (brow & 7))) * 16);
    };
    // A K-tile is two k-steps of 32, each with its fragments in registers.  While one k-step is multiplied the fragments of the next are read from LDS, so that with one
    // wave per SIMD neither the LDS reads nor the requests for later K-tiles stand in front of the matrix cores.
    half8_t fa[2][4], fb[2][MT];
    auto read_frag = [&](int slot, int ks) {
        const char *buf = smem + slot * BUF;
#pragma unroll
        for (int i = 0; i < 4; ++i) fa[ks][i] = read_a(buf, ks, i);
#pragma unroll
        for (int j = 0; j < MT; ++j) fb[ks][j] = read_b(buf, ks, j);
    };
    auto multiply = [&](int ks, bool reads) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j)
                acc[i][j] = mfma16(fa[ks][i], fb[ks][j], acc[i][j]);
        if (reads) {                                                      // the reads between the first products, so that they land under the later ones
            constexpr int P = MT > 1 ? MT / 2 : 1;
            __builtin_amdgcn_sched_group_barrier(0x8, P, 0); __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, P, 0); __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, P, 0); __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, P, 0); __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 4 * MT - 4 * P, 0);
        }
    };
#pragma unroll
    for (int st = 0; st < NS; ++st) if (st < KT) stage(st, st * BK);
    wait_ring<4 + MT>(min(NS - 1, KT - 1));
    if (ROPE) {
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            asm volatile("" : "+v"(rope_pos[j]), "+v"(rope_slot[j]));     // uses stay behind the counted wait (volatile asm keeps its order)
            if (!epi.slots) rope_slot[j] = -1;
        }
    }
    constexpr int PRE = QKN && MT == 4 ? 2 : MT;                          // (registers: the 128-token tile's other two behind the K loop)
    auto request_angles = [&](int j) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int64_t at_pos = rope_pos[j] * 64 + (threadIdx.x & 7) * 8 + u * 4;
            pre_cs[j][u] = *reinterpret_cast<const float4_t *>(epi.cos_t + at_pos);
            pre_sn[j][u] = *reinterpret_cast<const float4_t *>(epi.sin_t + at_pos);
        }
    };
    if constexpr (QKN)
        if (rope_rot) {
            const half_t *w = (rope_head < epi.H ? epi.qn_w : epi.kn_w) + (threadIdx.x & 7) * 8;
            norm_w[0] = *reinterpret_cast<const half8_t *>(w); norm_w[1] = *reinterpret_cast<const half8_t *>(w + 64);
#pragma unroll
            for (int j = 0; j < PRE; ++j) request_angles(j);
        }
    if (!QKN && rope_rot) {
        const int half_d = epi.D / 2;
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int jj = ((at.x * 8 + wn * 4 + (q >> 1) * 2 + u) & (tph - 1)) * 8 + (q & 1) * 4;
                pre_cs[j][u] = *reinterpret_cast<const float4_t *>(epi.cos_t + rope_pos[j] * half_d + jj);
                pre_sn[j][u] = *reinterpret_cast<const float4_t *>(epi.sin_t + rope_pos[j] * half_d + jj);
            }
    }
    __builtin_amdgcn_s_barrier();
    read_frag(0, 0);
    int slot = 0;
    // first k-step of a K-tile; behind it this wave has read the whole tile
    auto first_half = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        read_frag(slot, 1);
        multiply(0, true);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);                               // lgkmcnt(0)
    };
    auto second_half = [&](int next) {
        read_frag(next, 0);
        multiply(1, true);
        slot = next;
    };
    int kt = 0;
    for (; kt + NS < KT; ++kt) {
        first_half();
        // K-tile kt + 1 has landed once at most the 4 + MT requests per thread of each of the NS - 2 younger K-tiles are outstanding (the cos / sin requests of a rotating
        // TEPI_ROPE wave are younger than K-tiles 1 .. NS - 1 and may stay in flight with them)
        if (rope_rot && kt + 1 < NS) wait_requests<(NS - 2) * (4 + MT) + 4 * PRE + (QKN ? 2 : 0)>();
        else wait_requests<(NS - 2) * (4 + MT)>();
        __builtin_amdgcn_s_barrier();                                     // every thread's pieces of K-tile kt + 1 are in, and every wave has read K-tile kt: its slot is free
        __builtin_amdgcn_sched_barrier(0);
        stage(slot, (kt + NS) * BK);
        second_half(slot + 1 == NS ? 0 : slot + 1);
    }
    for (; kt + 1 < KT; ++kt) {                                           // the last NS - 1 K-tiles but one: nothing left to request
        first_half();
        wait_ring<4 + MT>(KT - 2 - kt);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        second_half(slot + 1 == NS ? 0 : slot + 1);
    }
    first_half();
    multiply(1, false);
    if (EPI == TEPI_SLAB) {                                                // f32 partial sums, C layout: 4 consecutive columns of token r
        float *sl = epi.slabs + (int64_t)at.z * epi.slab_stride;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int m = m0 + wm * (16 * MT) + j * 16 + r;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = at.x * BN + wn * 64 + i * 16 + q * 4;
                if (m < T && n < N) *reinterpret_cast<float4_t *>(sl + (int64_t)m * N + n) = acc[i][j];
            }
        }
        return;
    }
    if (EPI == TEPI_LMHEAD) {
        // C layout: row (n) = q*4 + reg, col (token) = r.  f32 logits go out as they are (embed_head.rs:292-306, A-21); the
        // row maxima are taken over the f32 accumulators in increasing column order (ties keep the lowest index, A-12)
        float *sv = reinterpret_cast<float *>(smem);                      // [2 (wn)][BMt tokens]
        int *si = reinterpret_cast<int *>(smem + 2 * BMt * 4);
        __syncthreads();                                                  // (the operand buffers are read by every wave)
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int ml = wm * (16 * MT) + j * 16 + r, m = m0 + ml;
            float bv = -INFINITY; int bi = 0x7fffffff;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = at.x * BN + wn * 64 + i * 16 + q * 4;
                if (epi.logits && m < T && n < N) *reinterpret_cast<float4_t *>(epi.logits + (int64_t)m * N + n) = acc[i][j];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = acc[i][j][e];
                    if (n + e < N && (v > bv || (v == bv && n + e < bi))) { bv = v; bi = n + e; }
                }
            }
#pragma unroll
            for (int o = 16; o <= 32; o <<= 1) {                          // the four q groups of a token
                const float v = __shfl_xor(bv, o, 64); const int i2 = __shfl_xor(bi, o, 64);
                if (v > bv || (v == bv && i2 < bi)) { bv = v; bi = i2; }
            }
            if (q == 0) { sv[wn * BMt + ml] = bv; si[wn * BMt + ml] = bi; }
        }
        __syncthreads();
        if (threadIdx.x < BMt && m0 + threadIdx.x < T) {
            float bv = sv[threadIdx.x]; int bi = si[threadIdx.x];
            const float v = sv[BMt + threadIdx.x]; const int i2 = si[BMt + threadIdx.x];
            if (v > bv || (v == bv && i2 < bi)) { bv = v; bi = i2; }
            epi.pval[(int64_t)at.x * T + m0 + threadIdx.x] = bv;
            epi.pidx[(int64_t)at.x * T + m0 + threadIdx.x] = bi;
        }
        return;
    }
    if constexpr (QKN) {
        // the products, rounded, as [token][16 pieces ^ token & 15] over the operand buffers; then every row's norm, rotation and stores (head_norm: 8 lanes a row)
        if (PRE < MT && rope_rot) {
#pragma unroll
            for (int j = PRE; j < MT; ++j) request_angles(j);
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int ml = wm * (16 * MT) + j * 16 + r;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int col = wn * 64 + i * 16 + q * 4;
                *reinterpret_cast<half4_t *>(smem + ml * 256 + ((((col >> 3) ^ (ml & 15)) << 4) | ((col & 4) << 1))) =
                    (half4_t){(half_t)acc[i][j][0], (half_t)acc[i][j][1], (half_t)acc[i][j][2], (half_t)acc[i][j][3]};
            }
        }
        __syncthreads();
        const int pc = threadIdx.x & 7;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int ml = j * 32 + ((int)threadIdx.x >> 3), m = m0 + ml;
            half8_t x1 = *reinterpret_cast<const half8_t *>(smem + ml * 256 + ((pc ^ (ml & 15)) << 4));
            half8_t x2 = *reinterpret_cast<const half8_t *>(smem + ml * 256 + (((8 + pc) ^ (ml & 15)) << 4));
            if (rope_rot) {
                head_norm<8>(x1, x2, norm_w[0], norm_w[1], epi.qk_eps);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float a = (float)x1[e], b = (float)x2[e], cc = pre_cs[j][e >> 2][e & 3], sn = pre_sn[j][e >> 2][e & 3];
                    x1[e] = to_half_rn(mul_sub_unfused(a, cc, b, sn));
                    x2[e] = to_half_rn(mul_add_unfused(b, cc, a, sn));
                }
            }
            if (m >= T) continue;
            if (rope_head < epi.H || !epi.kv_cache_only) {
                half_t *row = y + (int64_t)m * N + rope_head * 128 + pc * 8;
                *reinterpret_cast<half8_t *>(row) = x1; *reinterpret_cast<half8_t *>(row + 64) = x2;
            }
            if (rope_head >= epi.H && rope_slot[j] >= 0) {
                half_t *row = (rope_rot ? epi.kc : epi.vc) + ((int64_t)rope_slot[j] * epi.KVH + rope_head - epi.H - (rope_rot ? 0 : epi.KVH)) * 128 + pc * 8;
                *reinterpret_cast<half8_t *>(row) = x1; *reinterpret_cast<half8_t *>(row + 64) = x2;
            }
        }
        return;
    }
    // epilogue: C layout row (n) = q*4 + reg, col (token) = r: a lane holds 4 consecutive columns of one token in each n-tile.  Two neighbouring n-tiles trade the
    // odd 16-lane rows of one for the even rows of the other (v_permlane16_swap), after which a lane holds 8 consecutive columns of one of them: 16-byte stores,
    // 64 consecutive bytes of a token row per instruction, without a pass through LDS (3814 tokens, us: gate_up 52.0 -> 50.3, qkv 35.3 -> 34.8; 4672 tokens with the rotation 68.0 -> 60.0).
    auto pair8 = [&](half4_t x, half4_t y) -> half8_t {
        union { half4_t h; unsigned u[2]; } a, b;
        union { half8_t h; unsigned u[4]; } o;
        a.h = x; b.h = y;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const auto t = __builtin_amdgcn_permlane16_swap(a.u[e], b.u[e], false, false);
            o.u[e] = t[0]; o.u[2 + e] = t[1];
        }
        return o.h;
    };
    const int col_in_pair = (q & 1) * 16 + (q >> 1) * 8;                  // first column a lane holds of a pair of n-tiles whose 32 columns are consecutive
    half8_t resid[MT][2];                                                 // TEPI_RESID: what the products are added to, all of it requested at once
    if (EPI == TEPI_RESID) {
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                resid[j][i] = *reinterpret_cast<const half8_t *>(y + (int64_t)min(m0 + wm * (16 * MT) + j * 16 + r, T - 1) * N + min(at.x * BN + wn * 64 + i * 32 + col_in_pair, N - 8));
    }
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int m = m0 + wm * (16 * MT) + j * 16 + r;
        if (EPI == TEPI_F16 || EPI == TEPI_RESID) {
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                half4_t h[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) h[u] = (half4_t){(half_t)acc[i + u][j][0], (half_t)acc[i + u][j][1], (half_t)acc[i + u][j][2], (half_t)acc[i + u][j][3]};
                half8_t v8 = pair8(h[0], h[1]);
                const int n = at.x * BN + wn * 64 + i * 16 + col_in_pair;
                if (EPI == TEPI_RESID) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v8[e] = to_half_rn((float)resid[j][i >> 1][e] + (float)v8[e]);
                }
                if (m < T && n < N) *reinterpret_cast<half8_t *>(y + (int64_t)m * N + n) = v8;
            }
        } else if (t_glu(EPI)) {
            half4_t h[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {                                 // tiles i (gate) and i+2 (up), same 16 columns
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float gf = (float)to_half_rn(acc[i][j][e]), uf = (float)to_half_rn(acc[i + 2][j][e]);
                    if constexpr (EPI == TEPI_CLAMP) h[i][e] = to_half_rn(clamped_unit(gf, uf, epi.limit, epi.alpha));
                    else {
                        const float sg = gate_factor(gf, epi.gelu);
                        h[i][e] = to_half_rn(__fmul_rn(__fmul_rn(gf, sg), uf));
                    }
                }
            }
            const half8_t v8 = pair8(h[0], h[1]);
            const int n = at.x * 64 + wn * 32 + col_in_pair;
            int64_t ldo = N;
            if constexpr (EPI == TEPI_CLAMP) ldo = epi.ldo;
            if (m < T && n < N) *reinterpret_cast<half8_t *>(y + (int64_t)m * ldo + n) = v8;
        } else {                                                          // TEPI_ROPE
            const int half_d = epi.D / 2;
            const int64_t ldy = (int64_t)heads * epi.D;
            float4_t cs[4], sn[4];
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const auto tc = __builtin_amdgcn_permlane32_swap(__float_as_uint(pre_cs[j][u][e]), __float_as_uint(pre_cs[j][u][e]), false, false);
                    const auto ts = __builtin_amdgcn_permlane32_swap(__float_as_uint(pre_sn[j][u][e]), __float_as_uint(pre_sn[j][u][e]), false, false);
                    cs[u][e] = __uint_as_float(tc[0]); cs[2 + u][e] = __uint_as_float(tc[1]);
                    sn[u][e] = __uint_as_float(ts[0]); sn[2 + u][e] = __uint_as_float(ts[1]);
                }
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                half4_t h[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const bool rot = ((at.x * 8 + wn * 4 + i + u) >> tsh) < epi.H + epi.KVH;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float v = (float)to_half_rn(acc[i + u][j][e]);
                        const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
                        const float pv = __uint_as_float(q < 2 ? t[1] : t[0]);                        // the partner column: the same register of lane ^ 32
                        // rotary_embedding.rs:36-44: out1 = x1*c - x2*s ; out2 = x2*c + x1*s
                        const float f = !rot ? v : (q < 2) ? mul_sub_unfused(v, cs[i + u][e], pv, sn[i + u][e]) : mul_add_unfused(v, cs[i + u][e], pv, sn[i + u][e]);
                        h[u][e] = to_half_rn(f);
                    }
                }
                const half8_t v8 = pair8(h[0], h[1]);
                const int g = at.x * 8 + wn * 4 + i + (q & 1), head = g >> tsh, c = g & (tph - 1);    // of the n-tile whose columns the lane now holds
                const bool rot = head < epi.H + epi.KVH;
                // rotated heads: an n-tile is 8 columns of the first half of the head (lanes q < 2) and their 8 partners
                const int col = rot ? c * 8 + (q >> 1) * half_d : c * 16 + (q >> 1) * 8;
                if (m < T && head < heads) {
                    if (head < epi.H || !epi.kv_cache_only) *reinterpret_cast<half8_t *>(y + (int64_t)m * ldy + head * epi.D + col) = v8;
                    if (head >= epi.H && rope_slot[j] >= 0) {
                        const int kvh = rot ? head - epi.H : head - epi.H - epi.KVH;
                        *reinterpret_cast<half8_t *>((rot ? epi.kc : epi.vc) + ((int64_t)rope_slot[j] * epi.KVH + kvh) * epi.D + col) = v8;
                    }
                }
            }
        }
    }
}

// gate_up + SiluAndMul on 96 W rows (48 gate + 48 up = 48 output columns) x 128 tokens (r05).  At T = 512 the 128 x 128
// tiles above give the gate_up GEMM of Qwen3-0.6B 48 x 4 = 192 workgroups — 64 CUs idle — and a launch of these GEMMs is paced by the operand
// bytes a CU takes in through its L2 -> LDS path (profiles/r04_mid_batch_gemm.txt: ~52 GB/s per CU): 64 x 4 = 256 workgroups of (96 + 128) rows
// x 2 KB = 458 KB each instead of 192 of 524 KB.  Four waves side by side over the tokens (wave w: tokens 32 w .. 32 w + 31, all six n-tiles:
// 12 MFMA tiles per wave and k-step), the four-buffer ring with counted waits of gemm_tiled_kernel<.., 4, ..>, the same K order per output as
// every other tiling of this file (same bits as the 128-row tiles and as the unfused GEMM + SiluAndMul).
constexpr int S96_A = 96 * BK * 2, S96_BUF = S96_A + BM * BK * 2;        // bytes of the A image / of one ring buffer
__global__ __launch_bounds__(256, 2) void gemm_tiled_silu96_kernel(const half_t *__restrict__ x, int64_t ldx, const half_t *__restrict__ W, int T, int K, int I,
                                                                half_t *__restrict__ y, int tiled) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int NS = RING96;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;
    const int m0 = blockIdx.y * BM;
    const int kmul = tiled ? 16 : 1;
    const half_t *asrc[3], *bsrc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int idx = i * 256 + threadIdx.x, row = idx >> 3, c = (idx & 7) ^ (row & 7);
        if (i < 3) {                                                      // A: local row = 16 t + rr, t = 0..2 gate tiles, 3..5 up tiles of the same columns
            const int t = row >> 4, rr = row & 15;
            const int blk = (t < 3 ? 0 : I / 16) + (int)blockIdx.x * 3 + t % 3;
            asrc[i] = W + (tiled ? ((int64_t)blk * (K / 32) + (c >> 2)) * 512 + rr * 32 + (c & 3) * 8 : (int64_t)(blk * 16 + rr) * K + c * 8);
        }
        int xr = m0 + row; if (xr > T - 1) xr = T - 1;
        bsrc[i] = x + (int64_t)xr * ldx + c * 8;
    }
    auto stage = [&](int buf, int k0) {
        char *a_dst = smem + buf * S96_BUF, *b_dst = a_dst + S96_A;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int piece = (i * 256 + wave * 64) * 16;               // wave-uniform LDS base; hardware adds lane*16
            if (i < 3) __builtin_amdgcn_global_load_lds(asrc[i] + k0 * kmul, (__attribute__((address_space(3))) void *)(a_dst + piece), 16, 0, 0);
            __builtin_amdgcn_global_load_lds(bsrc[i] + k0, (__attribute__((address_space(3))) void *)(b_dst + piece), 16, 0, 0);
        }
    };
    float4_t acc[6][2];
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
    const int KT = K / BK;
    half8_t fa[2][6], fb[2][2];                                           // fragments of the two k-steps of a K-tile: one multiplied, the other being read, as in gemm_tiled_kernel
    auto read_frag = [&](int slot, int ks) {
        const char *a_lds = smem + slot * S96_BUF, *b_lds = a_lds + S96_A;
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const int arow = i * 16 + r;
            fa[ks][i] = *reinterpret_cast<const half8_t *>(a_lds + (arow * 8 + ((ks * 4 + q) ^ (arow & 7))) * 16);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int brow = wave * 32 + j * 16 + r;
            fb[ks][j] = *reinterpret_cast<const half8_t *>(b_lds + (brow * 8 + ((ks * 4 + q) ^ (brow & 7))) * 16);
        }
    };
    auto multiply = [&](int ks, bool reads) {
#pragma unroll
        for (int i = 0; i < 6; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = mfma16(fa[ks][i], fb[ks][j], acc[i][j]);
        if (reads) {
            __builtin_amdgcn_sched_group_barrier(0x8, 2, 0); __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 2, 0); __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 2, 0); __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 6, 0);
        }
    };
#pragma unroll
    for (int st = 0; st < NS; ++st) if (st < KT) stage(st, st * BK);
    wait_ring<7>(min(NS - 1, KT - 1));
    __builtin_amdgcn_s_barrier();
    read_frag(0, 0);
    int slot = 0;
    for (int kt = 0; kt < KT; ++kt) {
        __builtin_amdgcn_sched_barrier(0);
        read_frag(slot, 1);
        multiply(0, true);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);                               // lgkmcnt(0)
        if (kt + 1 == KT) break;
        wait_ring<7>(min(NS - 2, KT - 2 - kt));
        __builtin_amdgcn_s_barrier();                                     // K-tile kt + 1 is in, and every wave has read K-tile kt
        __builtin_amdgcn_sched_barrier(0);
        if (kt + NS < KT) stage(slot, (kt + NS) * BK);
        slot = slot + 1 == NS ? 0 : slot + 1;
        read_frag(slot, 0);
        multiply(1, true);
    }
    multiply(1, false);
    __syncthreads();                                                      // the epilogue reuses the operand buffers
    // act = fp16(silu(fp16 g) * fp16 u) (activation.rs:46-63; the rounding points of the unfused graph), staged in LDS and written as 16-byte pieces
    constexpr int OST = 112;                                              // bytes per staged row (48 fp16 + pad)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int ml = wave * 32 + j * 16 + r;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            half4_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float gf = (float)to_half_rn(acc[c][j][e]), uf = (float)to_half_rn(acc[c + 3][j][e]);
                const float sg = sigmoid_fast(gf);
                h[e] = to_half_rn(__fmul_rn(__fmul_rn(gf, sg), uf));
            }
            *reinterpret_cast<half4_t *>(smem + ml * OST + (c * 16 + q * 4) * 2) = h;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < (BM * 6) / 256; ++i) {                            // 6 pieces per row
        const int pidx = i * 256 + threadIdx.x, row = pidx / 6, ch = pidx % 6;
        const int m = m0 + row;
        if (m >= T) continue;
        *reinterpret_cast<half8_t *>(y + (int64_t)m * I + blockIdx.x * 48 + ch * 8) = *reinterpret_cast<const half8_t *>(smem + row * OST + ch * 16);
    }
}

static int tiled_check(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "%s launch failed: %s", what, hipGetErrorString(e));
    return 0;
}

// Token tile of a launch with `cols` = column tiles x k-slices: 128, 64 or 32 tokens (4, 2, 1 m-tiles per wave).  A CU is fed through its L2 -> LDS path at 80-87 GB/s whatever the
// tile (loads alone, no products: 0.25 / 0.30 / 0.375 us per K-tile of 20 / 24 / 32 KiB), so a launch costs its fullest CU's workgroups times that.  Measured, us: 200 tokens x 4096
// columns, K = 1024 6.8 on 224 tiles of 32 tokens / 7.7 on 128 of 64; 300 tokens 8.4 on 320 of 32 / 7.6 on 160 of 64; 1000 tokens 12.5 on 512 of 64 / 11.6 on 256 of 128; 509 tokens of
// gate_up (48 column tiles) 13.3 on 384 of 64 or 192 of 128, 15.9 on 768 of 32.
static int tiled_mt(int64_t T, int64_t cols) {
    auto cost = [&](int mt, int us) { return (cols * ((T + 32 * mt - 1) / (32 * mt)) + 255) / 256 * us; };
    int mt = 4;
    if (cost(2, 300) < cost(mt, 375)) mt = 2;
    if (cost(1, 250) < cost(mt, mt == 4 ? 375 : 300)) mt = 1;
    return mt;
}
// Strips of a launch's tiles (TileMap): as many as keep the rows of W and x that one XCD reads fewest.  3814 tokens, us in 1 / 2 / 4 / 8 strips: o_proj (8 column tiles) 19.0 / 18.9 /
// 19.0 / 21.8, qkv (32) 35.2 / 33.0 / 33.2 / 33.3, gate_up (48) 56.4 / 51.4 / 50.5 / 50.3; in the order of a 2-d grid, 8 token tiles apart on one XCD, o_proj 21.8.
static TileMap tile_map(int64_t nx, int64_t ny, int64_t nz, int64_t tokens) {
    const int64_t xcds = nz >= 8 ? 1 : 8 / nz;                            // XCDs of a k-slice
    int64_t strips = 1, best = INT64_MAX;
    for (int64_t a = 1; a <= xcds && a <= nx; a *= 2) {
        const int64_t rows = (nx + a - 1) / a * BN + (ny * a + xcds - 1) / xcds * tokens;
        if (rows < best) { best = rows; strips = a; }
    }
    return TileMap{(int32_t)nx, (int32_t)ny, (int32_t)((nx + strips - 1) / strips)};
}
constexpr size_t kStageBytes = 2 * BM * BK * 2;                          // MT = 4
constexpr size_t kStageBytes64 = (BN + 64) * BK * 2;                     // MT = 2
constexpr size_t kStageBytes32 = (BN + 32) * BK * 2;                     // MT = 1
// K-tiles in flight: two of the 128-token tiles when two workgroups share a CU (64 KiB each), three when one is alone on it; three or (a long K loop, one workgroup per CU) four of the 64-token
// tiles, four of the 32-token tiles.  More are slower: 512 tokens x 4096 columns 8.2 us with three, 8.3 with four, 8.7 with six (a launch's LDS takes time to be given out).
template <int EPI>
static void tiled_launch(int64_t nx, int64_t nz, const half_bits *x_, int64_t ldx, const half_bits *W_, const half_bits *Wt, int64_t T, int64_t K, int64_t N, int64_t NW, half_t *y, typename TileArgs<EPI>::type e, hipStream_t s) {
    const half_t *x = (const half_t *)x_, *W = (const half_t *)(Wt ? Wt : W_);
    e.tiled = Wt != nullptr;
    const int mt = tiled_mt(T, nx * nz);
    const int64_t ny = (T + 32 * mt - 1) / (32 * mt), wgs = nx * ny * nz;
    e.map = tile_map(nx, ny, nz, 32 * mt);
    const dim3 grid((unsigned)wgs), block(256);
#define NVR_TILED(NS_, MT_, BYTES_) gemm_tiled_kernel<EPI, NS_, MT_><<<grid, block, (NS_) * (BYTES_), s>>>(x, ldx, W, (int)T, (int)K, (int)N, (int)NW, y, e)
    if (mt == 4) { if (wgs <= 256) NVR_TILED(3, 4, kStageBytes); else NVR_TILED(2, 4, kStageBytes); }
    else if (mt == 2) { if (wgs <= 256) NVR_TILED(4, 2, kStageBytes64); else NVR_TILED(3, 2, kStageBytes64); }
    else NVR_TILED(4, 1, kStageBytes32);
#undef NVR_TILED
}
// > 64 KiB of dynamic LDS needs an opt-in per kernel instance; called at runner creation (never inside a stream capture)
int gemm_tiled_prepare() {
    static bool done = false;
    if (done) return 0;
#define NVR_TILED_ATTR1(EPI_, NS_, MT_, BYTES_)                                                                                                                   \
    { hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_tiled_kernel<EPI_, NS_, MT_>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)(NS_ * BYTES_)); \
      if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "gemm_tiled: LDS opt-in failed: %s", hipGetErrorString(e)); }
#define NVR_TILED_ATTR(EPI_) NVR_TILED_ATTR1(EPI_, 3, 4, kStageBytes) NVR_TILED_ATTR1(EPI_, 4, 2, kStageBytes64) NVR_TILED_ATTR1(EPI_, 3, 2, kStageBytes64) NVR_TILED_ATTR1(EPI_, 4, 1, kStageBytes32)
    NVR_TILED_ATTR(TEPI_F16) NVR_TILED_ATTR(TEPI_SILU) NVR_TILED_ATTR(TEPI_ROPE) NVR_TILED_ATTR(TEPI_LMHEAD) NVR_TILED_ATTR(TEPI_SLAB) NVR_TILED_ATTR(TEPI_RESID) NVR_TILED_ATTR(TEPI_QKN) NVR_TILED_ATTR(TEPI_CLAMP)
#undef NVR_TILED_ATTR
#undef NVR_TILED_ATTR1
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_tiled_silu96_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, RING96 * S96_BUF) != hipSuccess)
        return nvr::fail(NVR_ERR_HIP, "gemm_tiled: LDS opt-in failed (96-row SiLU tiles)");
    done = true;
    return 0;
}

static constexpr bool tiled_enabled() { return true; }
// LM head for more than 32 rows (large decode batches, many-sequence prefills): weights streamed once per 128-row block
bool gemm_tiled_lm_head_ok(int64_t T, int64_t K, int64_t N, int64_t ldx) {
    return tiled_enabled() && T > 32 && T <= 65536 && K % BK == 0 && N % 16 == 0 && ldx % 8 == 0 && (N + BN - 1) / BN <= LM_HEAD_MAX_PARTS &&
           N < (1ll << 31);
}
int gemm_tiled_lm_head(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, float *logits,
                       float *part_val, int32_t *part_idx, int32_t *nparts, hipStream_t s, const half_bits *Wt) {
    if (!gemm_tiled_lm_head_ok(T, K, N, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm_tiled_lm_head: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    TileEpi e{};
    e.logits = logits; e.pval = part_val; e.pidx = part_idx;
    *nparts = (int32_t)((N + BN - 1) / BN);
    if (int rc = gemm_tiled_prepare()) return rc;
    tiled_launch<TEPI_LMHEAD>(*nparts, 1, x, ldx, W, Wt, T, K, N, N, nullptr, e, s);
    return tiled_check("gemm_tiled_lm_head");
}

// split-k form for the narrow row-parallel GEMMs (o_proj / down_proj) at 65..1024 rows: slabs[z][T][N] f32, S slices of K
bool gemm_tiled_splitk_ok(int64_t T, int64_t K, int64_t N, int64_t S, int64_t ldx) {
    return tiled_enabled() && T > 32 && S >= 1 && K % (S * BK) == 0 && N % 16 == 0 && ldx % 8 == 0;
}
int gemm_tiled_splitk(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, int64_t S, float *slabs, hipStream_t s, const half_bits *Wt) {
    if (!gemm_tiled_splitk_ok(T, K, N, S, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm_tiled_splitk: T=%ld K=%ld N=%ld S=%ld", (long)T, (long)K, (long)N, (long)S);
    if (int rc = gemm_tiled_prepare()) return rc;
    TileEpi e{};
    e.slabs = slabs; e.slab_stride = T * N; e.kslice = (int32_t)(K / S);
    tiled_launch<TEPI_SLAB>((N + BN - 1) / BN, S, x, ldx, W, Wt, T, K, N, N, nullptr, e, s);
    return tiled_check("gemm_tiled_splitk");
}

bool gemm_tiled_ok(int64_t T, int64_t K, int64_t N, int64_t ldx) { return tiled_enabled() && T > 32 && K % BK == 0 && N % 16 == 0 && ldx % 8 == 0; }

int gemm_tiled(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, half_bits *y, hipStream_t s, const half_bits *Wt) {
    if (!gemm_tiled_ok(T, K, N, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm_tiled: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    if (int rc = gemm_tiled_prepare()) return rc;
    tiled_launch<TEPI_F16>((N + BN - 1) / BN, 1, x, ldx, W, Wt, T, K, N, N, (half_t *)y, TileEpi{}, s);
    return tiled_check("gemm_tiled");
}
int gemm_tiled_resid(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, half_bits *h, hipStream_t s, const half_bits *Wt) {
    if (!gemm_tiled_ok(T, K, N, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm_tiled_resid: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    if (int rc = gemm_tiled_prepare()) return rc;
    tiled_launch<TEPI_RESID>((N + BN - 1) / BN, 1, x, ldx, W, Wt, T, K, N, N, (half_t *)h, TileEpi{}, s);
    return tiled_check("gemm_tiled_resid");
}
// 96-row tiles when they put a workgroup on (nearly) every CU where the 128-row tiles leave a quarter of them idle (T = 512, I = 3072: 256 against 192; T = 321..384: 192 against 144)
static bool on_96_rows(int64_t T, int64_t I) {
    const int64_t ty = (T + BM - 1) / BM, w128 = (I / 64) * ty, w96 = (I / 48) * ty;
    return I % 48 == 0 && tiled_mt(T, I / 64) == 4 && w96 <= 256 && w96 > w128 && w128 * 8 <= w96 * 7;
}
// the weights of gemm_tiled_silu_mul by the XCD that reads them: workgroup x of the 96-row tiles takes 48 gate and 48 up rows; of the others an XCD takes an eighth of both where that is a strip
Ahead gemm_tiled_silu_ahead(const half_bits *W, int64_t T, int64_t K, int64_t I) {
    if (on_96_rows(T, I)) return (I / 48) % 8 ? Ahead{} : Ahead{W, (int32_t)(2 * I / 48), (int32_t)(48 * K / 8)};
    const int64_t nx = I / 64, mt = tiled_mt(T, nx);
    if (nx % 8 || tile_map(nx, (T + 32 * mt - 1) / (32 * mt), 1, 32 * mt).width * 8 != nx) return {};
    return {W, 16, (int32_t)(I / 8 * K / 8)};
}
int gemm_tiled_silu_mul(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t I, half_bits *out, hipStream_t s, bool gelu, const half_bits *Wt) {
    if (!gemm_tiled_ok(T, K, I, ldx) || I % 64) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm_tiled_silu_mul: T=%ld K=%ld I=%ld", (long)T, (long)K, (long)I);
    if (int rc = gemm_tiled_prepare()) return rc;
    if (!gelu && on_96_rows(T, I)) {
        gemm_tiled_silu96_kernel<<<dim3((unsigned)(I / 48), (unsigned)((T + BM - 1) / BM)), dim3(256), RING96 * S96_BUF, s>>>((const half_t *)x, ldx, (const half_t *)(Wt ? Wt : W), (int)T, (int)K, (int)I, (half_t *)out, Wt != nullptr);
        return tiled_check("gemm_tiled_silu_mul (96-row tiles)");
    }
    TileEpi e{}; e.gelu = gelu ? 1 : 0;
    tiled_launch<TEPI_SILU>(I / 64, 1, x, ldx, W, Wt, T, K, I, 2 * I, (half_t *)out, e, s);
    return tiled_check("gemm_tiled_silu_mul");
}
int gemm_tiled_clamped_glu(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t I, float limit, float alpha, half_bits *out, int64_t ldo, hipStream_t s) {
    if (!gemm_tiled_ok(T, K, I, ldx) || I % 64 || ldo % 8 || ldo < I) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm_tiled_clamped_glu: T=%ld K=%ld I=%ld", (long)T, (long)K, (long)I);
    if (int rc = gemm_tiled_prepare()) return rc;
    TileEpiClamp e{}; e.limit = limit; e.alpha = alpha; e.ldo = ldo;
    tiled_launch<TEPI_CLAMP>(I / 64, 1, x, ldx, W, nullptr, T, K, I, 2 * I, (half_t *)out, e, s);
    return tiled_check("gemm_tiled_clamped_glu");
}
int gemm_tiled_qkv_rope_store(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t H, int64_t KVH, int64_t D,
                              const int64_t *positions, const int32_t *slots, const float *cos_t, const float *sin_t, half_bits *qkv,
                              half_bits *k_cache, half_bits *v_cache, hipStream_t s, const half_bits *Wt, bool kv_cache_only, const QkNorm *norm) {
    const int64_t N = (H + 2 * KVH) * D;
    if (norm && D != 128) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm_tiled_qkv_rope_store: head norms with D=%ld", (long)D);
    if (!gemm_tiled_ok(T, K, N, ldx) || D % 16 || 128 % D) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm_tiled_qkv_rope_store: T=%ld K=%ld D=%ld", (long)T, (long)K, (long)D);
    TileEpiNorm e{};
    e.pos = positions; e.slots = slots; e.cos_t = cos_t; e.sin_t = sin_t; e.kc = (half_t *)k_cache; e.vc = (half_t *)v_cache;
    e.H = (int32_t)H; e.KVH = (int32_t)KVH; e.D = (int32_t)D;
    e.kv_cache_only = kv_cache_only && slots && k_cache && v_cache;
    if (int rc = gemm_tiled_prepare()) return rc;
    if (norm) {
        e.qn_w = (const half_t *)norm->q_w; e.kn_w = (const half_t *)norm->k_w; e.qk_eps = norm->eps;
        tiled_launch<TEPI_QKN>(N / BN, 1, x, ldx, W, Wt, T, K, N, N, (half_t *)qkv, e, s);
    } else tiled_launch<TEPI_ROPE>((N / 16 + 7) / 8, 1, x, ldx, W, Wt, T, K, N, N, (half_t *)qkv, e, s);
    return tiled_check("gemm_tiled_qkv_rope_store");
}

}}  // namespace nvr::k / nvr::kb (NVR_DT_NS)
