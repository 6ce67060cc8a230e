// gemm256.hip — 256x256x64 four-wave MFMA GEMM for the prefill regime (T >= 256 tokens): y[T,N] = x[T,K]·W[N,K]^T,
// with the three epilogues of the decode kernels (plain fp16, gate_up -> SiluAndMul, qkv -> RoPE + KV store).
// reference call sites as in linear.hip (linear.rs:354-356,228-239,437-439; activation.rs:46-63;
// rotary_embedding.rs:23-48; attention.rs:150-174).  Bound: MFMA (880.8 MFLOP per prefill token of Qwen3-0.6B).
//
// Structure:
//   * workgroup = 4 waves (2 along n x 2 along m), one per SIMD with all of its 512 registers, = 256 W rows (A operand) x 256 tokens (B operand), BK = 64.
//     Each operand tile is two HALF-TILES of 128 rows (16 KiB: [row][8 chunks of 16 B], chunk' = chunk ^ (row & 7),
//     conflict-free for the 4 x 16 lane groups of ds_read_b128).  LDS = 2 K-tile buffers x {A0, A1, B0, B1} = 128 KiB.
//   * a wave owns 64 rows of EACH half, so its 128 x 128 output (256 accumulation registers) splits into four quadrants (A half, B half) of 32 MFMAs
//     (v_mfma_f32_16x16x32_f16, 4 n-tiles x 4 m-tiles x 2 k-steps): one quadrant per PHASE.  A fragment read from LDS feeds eight products (eight waves of 128 x 64: 5.3, with 1.5 times the LDS reads).
//   * fragments of all four half-tiles fit in registers (128), so a phase brings in the half-tile that the NEXT one (A0: the one after) adds, and requests (LDS-DMA, 4 x 16 B per thread) a half-tile of
//     the K-tile after next into a slot whose last reader is a barrier back:
//         phase 0: quadrant (A0,B0)  reads B1        requests A0''        phase 2: quadrant (A1,B1)  reads A0'       requests B1''
//         phase 1: quadrant (A0,B1)  reads A1        requests B0''        phase 3: quadrant (A1,B0)  reads B0'       requests A1''
//     ending with s_waitcnt vmcnt(20) (the five youngest half-tiles stay in flight: a request has five phases of 512 clocks to land) and ONE barrier.
//   * results leave straight from the accumulators as 16-byte pieces: the W rows of a half-tile are laid into LDS in the order that gives a lane eight neighbouring columns, and epilogue partners are
//     in ONE lane (SiLU: A0 = gate rows, A1 = up rows of the same 128 columns; RoPE: A0 = first halves, A1 = second halves of the same heads).  No barrier, and the next tile's requests are under way.
// What bounds it: power.  With operands of zeros a K-tile takes 1.05 us at 2.4 GHz however many CUs run (2520 clocks: 128 products of 17 and the ~120 other instructions of a wave, which nothing overlaps), with
// random ones 1.07 us on 32 CUs and 1.45 on 256: the clock falls to what the part's power allows.  us, eight waves of 128 x 64 with 8 barriers a K-tile and results through LDS / so: 4096 x 12288 x 4096
// (T K N) 294 / 281, 32768 x 3072 x 1024 + residual 183 / 162, 32768 x 2048 x 1024 113 / 101, 32768 x 1024 x 4096 231 / 221, gate and up of 3072 columns 362 / 347, of 12288 at 3062 x 4096 478 / 451,
// qkv with RoPE and store 265 / 245, with head norms 298 / 274, of 3815 rows 36.8 / 35.7; rows grouped by expert, 32768 of 1024 to 768 and back 101 + 53 / 89 + 48, 2048 26 + 19.5 / 25 + 20.  A wave without
// another beside it pays for its epilogue's arithmetic in full: single rounds of 144..256 tiles with K <= 1024 whose epilogue computes much take 1 to 4 % more (with head norms, 160 tiles 32.1 / 33.4;
// heads of 64 31.3 / 32.0; the clamped unit at K = 512 21.7 / 22.6).  Registers: 476 to 512 of 512 a lane; the head norms' instance keeps one more in scratch memory (a store and a load a tile), the
// head's 29 scalar ones in lanes of a vector register, the others nothing.  (One barrier a K-tile with all requests behind it: the same rate alone, but 15 % less where the operands come from memory.)
#include <cstdlib>
#include <type_traits>
#include "kernels.h"
#include "device_utils.h"
#include "../common.h"

namespace nvr { namespace NVR_DT_NS {

enum { GEPI_F16 = 0, GEPI_RESID = 1, GEPI_SILU = 2, GEPI_ROPE = 3, GEPI_LMHEAD = 4, GEPI_RELU2 = 5, GEPI_GELU = 6, GEPI_GELU_ERF = 7, GEPI_QKN = 8, GEPI_CLAMP = 9 };   // GELU_ERF: y = gelu(x·Wᵀ) with the error function (from the unrounded product); RELU2: y = max(x·Wᵀ, 0)² (the product rounded to 16 bits first, as the unfused pair of launches does)
constexpr bool g_rope(int epi) { return epi == GEPI_ROPE || epi == GEPI_QKN; }      // QKN: RMSNorm over the columns of every q and k head in front of the rotation
constexpr bool g_glu(int epi) { return epi == GEPI_SILU || epi == GEPI_GELU || epi == GEPI_CLAMP; }      // gate and up rows in one tile, out = act(gate) * up (GELU: the tanh form; CLAMP: clamped_unit, rows of y ldo apart)
//   // RESID: y is the residual stream: y <- fp16(y + fp16(x·Wᵀ)) (qwen3.rs:382,389)
// LMHEAD (r06): the LM head over >= 128 rows (ParallelLMHead::compute_logits, embed_head.rs:292-306, + the greedy branch of Sampler::forward,
// sampler.rs:109-112): W = the [V, hidden] head, nothing is written as fp16 — every tile leaves (max, lowest vocabulary index) of its 256
// columns per token row (pval / pidx [column tile][T], merged by argmax_partials) and, on demand, the f32 logits straight from the accumulators;
// the vocabulary need not be a multiple of 256 (the last column tile clamps its row loads and masks its columns)

struct G256Epi {
    const int64_t *pos; const int32_t *slots; const float *cos_t, *sin_t;
    half_t *kc, *vc;
    int32_t H, KVH, D;
    int32_t kv_cache_only;             // GEPI_ROPE: k and v rows go to the caches only (the attention that follows reads them there)
    float *logits; float *pval; int32_t *pidx;   // GEPI_LMHEAD: f32 logits [T][N] (nullable), arg-max partials [tiles_x][T]
    const int32_t *row_w; int64_t w_stride; const int32_t *rows_used;      // (rows_used, on the device: rows behind it are nobody's; null: all T) GRP (rows grouped by expert): row block rb of 256 rows multiplies the matrix W + row_w[rb] * w_stride
};
// What single instances need beyond it stays out of the others' arguments
struct G256EpiNorm : G256Epi { const half_t *qn_w, *kn_w; float qk_eps; };      // GEPI_QKN: the norms' weights [D]
struct G256EpiClamp : G256Epi { float limit, alpha; int64_t ldo; };             // GEPI_CLAMP
template <int EPI> struct G256Args { using type = G256Epi; };
template <> struct G256Args<GEPI_QKN> { using type = G256EpiNorm; };
template <> struct G256Args<GEPI_CLAMP> { using type = G256EpiClamp; };

constexpr int G_BK = 64, G_HT = 128, G_HALF = G_HT * G_BK * 2;          // 16 KiB per half-tile
constexpr int G_BUF = 4 * G_HALF;                                         // A0 A1 B0 B1
constexpr int G_THREADS = 256;

// 1 KiB of an operand into LDS: 16 bytes a lane from base + off, lane-linear at the byte that M0 holds (set an instruction before, by the hardware's rule).  Inline asm: hipcc drains the
// builtin in front of LDS reads that it cannot tell apart from it; the requests are counted by hand.  M0 travels from g_aim to g_dma as a value of the compiler's own, which keeps the register free
// between the two.
__device__ __forceinline__ unsigned g_aim(unsigned lds, int piece) { unsigned at; asm volatile("s_add_u32 %0, %1, %2" : "={m0}"(at) : "s"(lds), "i"(piece) : "scc"); return at; }
__device__ __forceinline__ void g_dma(unsigned at, unsigned off, const char *base) { asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(at) : "memory"); }

// 4 bytes a lane from a pointer each
__device__ __forceinline__ void g_dma4(unsigned lds, const void *src) { asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "{m0}"(lds) : "memory"); }

template <int EPI, int RD = 0, bool GRP = false>
__global__ __launch_bounds__(G_THREADS, 1) void gemm256_kernel(const half_t *__restrict__ x, int64_t ldx, const half_t *__restrict__ W,
                                                      int T, int K, int N, int NW, half_t *__restrict__ y, typename G256Args<EPI>::type epi,
                                                      int tiles_x, int tiles_y, int PW) {
    extern __shared__ __attribute__((aligned(16))) char smem[];           // 2 x G_BUF, then what an epilogue needs
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 15, q = lane >> 4;
    const int wn = wave >> 1, wm = wave & 1;

    // Persistent workgroup.  The K-tile stream runs ACROSS its tiles: K-tile g of the stream lives in buffer g & 1, and the
    // last two K-tiles of a tile already stage K-tiles 0 and 1 of the next one, so those loads fly during the epilogue.
    // Tile order: column panels of PW tiles, each walked row block by row block; the line of tiles is cut into eight equal pieces, one per XCD (workgroup w runs on XCD w % 8, each XCD has its own
    // 4 MiB L2).  The 32 workgroups of an XCD are then at about PW columns x 32 / PW row blocks at any time, and fetch PW + 32 / PW half-megabyte slices of either operand for a K-tile instead of
    // the 18 or 33 of a plain order (us, one box each: 4096 x 12288 x 4096 278 -> 272; 32768 x 1024 x 4096 230 -> 221; 32768 x 2048 x 1024 112 -> 103).
    const int rows_y = GRP && epi.rows_used ? min(tiles_y, (__builtin_amdgcn_readfirstlane(*epi.rows_used) + 255) / 256) : tiles_y, tiles_total = tiles_x * rows_y;
    const int xcd = blockIdx.x & 7, step = gridDim.x >> 3, u_end = tiles_total / 8 * (xcd + 1) + min(xcd + 1, tiles_total % 8);
    int u = tiles_total / 8 * xcd + min(xcd, tiles_total % 8) + (int)(blockIdx.x >> 3);
    if (u >= u_end) return;
    struct Tile { int bx, by; };
    auto tile_of = [&](int uu) {
        const int panel = uu / (PW * rows_y), rem = uu - panel * (PW * rows_y), width = min(PW, tiles_x - panel * PW), by = rem / width;
        return Tile{panel * PW + rem - by * width, by};
    };

    constexpr int hd2 = g_rope(EPI) ? RD / 2 : 1;
    constexpr int OUTC = g_glu(EPI) ? 128 : 256;                          // output columns of a tile
    // Staging: a request is 32 rows (8 lanes a row) of a half-tile; LDS row rho = r0 + 32 i.  W row behind LDS row rho of A half hA: the 32 rows of a group lie in the order in which the
    // accumulators of two neighbouring 16-row tiles give a lane eight neighbouring columns (LDS row 16 b + 4 a + e holds row 8 a + 4 b + e), so that results leave as 16-byte pieces straight from
    // the registers; groups by column: plain bx*256 + hA*128 + ..   gate / up: hA*N + bx*128 + ..   RoPE: half hA of the tile's 256 / D heads, group by group; of two heads of 128 a wave gets the
    // same 32 columns of both (GEPI_ROPE: one set of sines serves the two; loading them for each head took 13 us of 259 at 32768 x 1024 x 4096) or one head whole (GEPI_QKN: its norm is then the wave's own).
    const int r0 = tid >> 3, pr = ((r0 & 15) >> 2) * 8 + (r0 >> 4) * 4 + (r0 & 3);
    const unsigned cch = (unsigned)(((tid & 7) ^ (r0 & 7)) * 16);         // swizzled 16-byte chunk of the row
    constexpr int PH = EPI == GEPI_QKN ? 2 : 1;                           // 32-column groups that a wave has of a half head
    auto w_row = [&](int i) { return !g_rope(EPI) ? i * 32 + pr : RD == 64 ? i * 64 + pr : PH == 2 ? (i >> 1) * 128 + (i & 1) * 32 + pr : (i & 1) * 128 + (i >> 1) * 32 + pr; };
    const int64_t half_w = (int64_t)(g_glu(EPI) ? N : g_rope(EPI) ? hd2 : 128) * K;      // from an A half's rows to the other's
    unsigned va[EPI == GEPI_LMHEAD ? 8 : 4], vb[8];                       // byte offsets of the thread's pieces from the tile's rows
    const char *pa0 = nullptr, *pa1 = nullptr, *pb = nullptr;             // next K-tile to request
#pragma unroll
    for (int i = 0; i < 4; ++i) va[i] = (unsigned)w_row(i) * (unsigned)K * 2u + cch;
    auto set_sources = [&](Tile t) {
        const int bx = t.bx, m0 = t.by * 256;
        const half_t *wb = W + (int64_t)bx * OUTC * K;
        if (GRP) wb += (int64_t)__builtin_amdgcn_readfirstlane(epi.row_w[t.by]) * epi.w_stride;
        pa0 = (const char *)wb;
        pa1 = (const char *)(wb + half_w);
        pb = (const char *)(x + (int64_t)m0 * ldx);
        const int rows_left = T - 1 - m0;                                 // ragged last row block: its last row again
#pragma unroll
        for (int i = 0; i < 8; ++i) vb[i] = (unsigned)min(i * 32 + r0, rows_left) * (unsigned)ldx * 2u + cch;
        if constexpr (EPI == GEPI_LMHEAD) {                               // (a ragged vocabulary block likewise; both halves count from its first row)
            pa1 = pa0;
            const int wrows_left = N - 1 - bx * 256;
#pragma unroll
            for (int i = 0; i < 8; ++i) va[i] = (unsigned)min(i * 32 + pr, wrows_left) * (unsigned)K * 2u + cch;
        }
    };
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char *)smem, lds_w = lds0 + (unsigned)wave * 1024u;
    // piece i = 0..3 of half-tile ht (0 = A0, 1 = A1, 2 = B0, 3 = B1)
    auto aim = [&](int ht, int i, unsigned lds) { return g_aim(lds, ht * G_HALF + i * 4096); };
    auto request = [&](int ht, int i, unsigned at) {
        if (ht < 2) g_dma(at, va[EPI == GEPI_LMHEAD ? ht * 4 + i : i], ht ? pa1 : pa0);
        else g_dma(at, vb[(ht - 2) * 4 + i], pb);
    };
    auto request_all = [&](int g) {                                       // a whole K-tile, in the order of the phases: A0, B0, B1, A1
#pragma unroll
        for (int n = 0; n < 16; ++n) {
            const int ht = n < 4 ? 0 : n < 8 ? 2 : n < 12 ? 3 : 1;
            const unsigned at = aim(ht, n & 3, lds_w + (unsigned)((g & 1) * G_BUF));
            asm volatile("s_nop 0");
            request(ht, n & 3, at);
        }
    };
    // RoPE: positions (low dwords of the int64 entries) and cache slots of a tile's 256 token rows travel to LDS behind the K-tile ring by LDS-DMA, 4 bytes per lane (64 rows a wave), into one
    // of two 2 KiB slots by tile parity, one tile ahead.
    auto request_rows = [&](Tile t, int slot) {
        if (g_rope(EPI)) {
            int m = t.by * 256 + wave * 64 + lane; if (m > T - 1) m = T - 1;
            const unsigned dst = lds0 + (unsigned)(2 * G_BUF + slot * 2048 + wave * 256);
            g_dma4(dst, epi.pos + m);
            if (epi.slots) g_dma4(dst + 1024, epi.slots + m);
        }
    };

    float4_t acc[2][4][2][4];                                             // [A half][n-tile][B half][m-tile]
    half8_t fa[2][4][2], fb[2][4][2];                                     // [half][tile][k-step]
    const int sw = (q ^ (r & 7)) * 16;
    const int a_lane = (wn * 64 + r) * 128 + sw, b_lane = 2 * G_HALF + (wm * 64 + r) * 128 + sw;
    auto read = [&](half8_t (&f)[4][2], int e, int half, int lane_at, int g) {      // fragment e of the 8 of half-tile `half` of an operand: tile e / 2, k-step e & 1 (chunk + 4, i.e. ^ 64)
        f[e >> 1][e & 1] = *reinterpret_cast<const half8_t *>(smem + (g & 1) * G_BUF + half * G_HALF + (e >> 1) * 2048 + (lane_at ^ ((e & 1) * 64)));
    };
    // One phase: the 32 products of quadrant (A half HA, B half HB) of a K-tile, B's fragments outermost.  A product leaves its wave room for three instructions: the 8 fragments of the half-tile that
    // the phase brings into registers (F of READ_G, one behind every fourth product, or behind the products of the B fragment that they replace) and the four pieces of the half-tile that it
    // requests (two instructions each) go between them.  Own requests that the next phase reads have landed (all but the youngest five half-tiles), own reads of the phase before are back, barrier.
#define G256_PHASE(HA_, HB_, F_, FH_, LANE_, READ_G_, RHT_, VM_, REQ_)                                                                          \
    unsigned at_##RHT_ = 0;                                                                                                                \
    _Pragma("unroll") for (int n = 0; n < 32; ++n) {                                                                                       \
        constexpr bool behind = (RHT_) == 1;                              /* phase 3 */                                                    \
        if (!behind && n % 3 == 0 && n < 24) read(F_[FH_], n / 3, FH_, LANE_, READ_G_);                                                    \
        if (behind && n >= 8 && n % 8 == 0) { read(F_[FH_], n / 4 - 2, FH_, LANE_, READ_G_); }                                             \
        if (behind && n >= 8 && n % 8 == 1) { read(F_[FH_], n / 4 - 1, FH_, LANE_, READ_G_); }                                             \
        if ((REQ_) && n % 8 == 4) at_##RHT_ = aim(RHT_, n / 8, req_lds);                                                                              \
        if ((REQ_) && n % 8 == 5) request(RHT_, n / 8, at_##RHT_);                                                                                            \
        __builtin_amdgcn_sched_barrier(0);                                                                                                 \
        acc[HA_][n & 3][HB_][n >> 3] = mfma16(fa[HA_][n & 3][(n >> 2) & 1], fb[HB_][n >> 3][(n >> 2) & 1], acc[HA_][n & 3][HB_][n >> 3]);  \
        __builtin_amdgcn_sched_barrier(0);                                                                                                 \
    }                                                                                                                                      \
    if ((RHT_) == 1) { read(F_[FH_], 6, FH_, LANE_, READ_G_); read(F_[FH_], 7, FH_, LANE_, READ_G_); }                                     \
    asm volatile("" ::: "memory");                                                                                                         \
    __builtin_amdgcn_s_waitcnt(((VM_) & 15) | 0x70 | ((RHT_) == 1 ? 2 << 8 : 0) | ((VM_) >> 4) << 14);                                     \
    __builtin_amdgcn_s_barrier();                                                                                                          \
    asm volatile("" ::: "memory");
#define G256_KTILE(V0_, V1_, V2_, V3_, REQ_)                                                                                                \
    {                                                                                                                                      \
        const unsigned req_lds = lds_w + (unsigned)((g & 1) * G_BUF);                                                                      \
        (void)req_lds;                                                                                                                     \
        G256_PHASE(0, 0, fb, 1, b_lane, g, 0, V0_, REQ_)                                                                                   \
        G256_PHASE(0, 1, fa, 1, a_lane, g, 2, V1_, REQ_)                                                                                   \
        G256_PHASE(1, 1, fa, 0, a_lane, g + 1, 3, V2_, REQ_)                                                                               \
        G256_PHASE(1, 0, fb, 0, b_lane, g + 1, 1, V3_, REQ_)                                                                               \
        if (REQ_) advance();                                                                                                               \
        ++g;                                                                                                                               \
    }

    const int KT = K / G_BK;
    Tile tile = tile_of(u);
    int su = u, skt = 0;                               // su, skt: tile and K-tile that the next requests are for
    auto advance = [&]() {
        pa0 += 2 * G_BK; pa1 += 2 * G_BK; pb += 2 * G_BK;
        if (++skt == KT) {
            skt = 0;
            if (su + step < u_end) { su += step; set_sources(tile_of(su)); }
        }
    };
    set_sources(tile);
    request_rows(tile, 0);
    request_all(0);
    advance();
    request_all(1);
    advance();
    asm volatile("s_waitcnt vmcnt(20)" ::: "memory");                     // (the rows and) A0, B0 and B1 of K-tile 0
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int e = 0; e < 8; ++e) { read(fa[0], e, 0, a_lane, 0); read(fb[0], e, 0, b_lane, 0); }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                                         // (phase 0 refills A0)
    asm volatile("" ::: "memory");

    const int64_t ldy = [&]() -> int64_t { if constexpr (EPI == GEPI_CLAMP) return epi.ldo; else return g_rope(EPI) ? (int64_t)(epi.H + 2 * epi.KVH) * RD : (int64_t)N; }();

    // Stores that a whole tile's epilogue leaves behind every request that is under way then: the first K-tile of the next tile need not wait for them (they are counted in order with the requests;
    // 32768 x 1024 x 4096: 231 -> 223 us).  RoPE's stores may be left out (slots), the LM head's are not told.
    constexpr int SLACK = g_rope(EPI) || EPI == GEPI_LMHEAD ? 0 : g_glu(EPI) ? 16 : 32;
    bool whole = false;                                                   // the tile before this one was a whole one
    int tile_no = 0;
    for (int g = 0;; ) {
        const bool have_next = u + step < u_end;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[a][i][b][j] = (float4_t){0.f, 0.f, 0.f, 0.f};
        // (in accumulation registers from here on: 256 is all there are, and any temporary among them has hipcc move accumulators about within the loop; a tile's first products without an addend need such)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                asm volatile("" : "+a"(acc[a][i][0][0]), "+a"(acc[a][i][0][1]), "+a"(acc[a][i][0][2]), "+a"(acc[a][i][0][3]), "+a"(acc[a][i][1][0]), "+a"(acc[a][i][1][1]), "+a"(acc[a][i][1][2]), "+a"(acc[a][i][1][3]));
        // (a workgroup's last two K-tiles request nothing: what is still under way is counted down)
        int kt = have_next ? KT : KT - 2;
        if (SLACK > 0 && whole && kt > 0) { G256_KTILE(20 + SLACK, 20 + SLACK, 20 + SLACK, 20 + SLACK, true) --kt; }
        for (; kt > 0; --kt) G256_KTILE(20, 20, 20, 20, true)
        if (!have_next) {
            G256_KTILE(16, 12, 8, 4, false)
            G256_KTILE(0, 0, 0, 0, false)
        }
        whole = tile.by * 256 + 256 <= T;
        // ---- epilogue of `tile`, straight from the accumulators: lane (r, q) has of token row m0 + hB*128 + wm*64 + j*16 + r the eight columns q*8 .. of every 32-column group wn*2 + p of either
        // A half (tiles 2p and 2p + 1).  No LDS, no barrier: the requests of the next tile's first two K-tiles are under way.
        {
        const int bx = tile.bx, m0 = tile.by * 256;
        // (the thread coordinates come from a value that the compiler cannot see through: otherwise it hoists the epilogue's address arithmetic out of the tile loop, where it has no registers)
        int elane = lane;
        asm volatile("" : "+v"(elane));
        const int r = elane & 15, q = elane >> 4;
        const int mrow = wm * 64 + r;                                     // + hB*128 + j*16
        // (the accumulators of a token tile stay in accumulation registers up to here: hipcc would bring all 256 over in front of the epilogue, and spill)
        auto hold = [&](int b, int j) {
            asm volatile("" : "+a"(acc[0][0][b][j]), "+a"(acc[0][1][b][j]), "+a"(acc[0][2][b][j]), "+a"(acc[0][3][b][j]), "+a"(acc[1][0][b][j]), "+a"(acc[1][1][b][j]), "+a"(acc[1][2][b][j]), "+a"(acc[1][3][b][j]));
        };
        auto eight = [&](int a, int p, int b, int j) {
            const float4_t lo = acc[a][2 * p][b][j], hi = acc[a][2 * p + 1][b][j];
            return (half8_t){(half_t)lo[0], (half_t)lo[1], (half_t)lo[2], (half_t)lo[3], (half_t)hi[0], (half_t)hi[1], (half_t)hi[2], (half_t)hi[3]};
        };
        if constexpr (EPI == GEPI_LMHEAD) {
            // Per token row: (max, lowest index) over this lane's 32 entries in ascending column order (strict >: the first maximum stays),
            // then over the 4 lanes of the token (larger value, else lower index), then over the two wave columns through LDS.
            // A wave has its SIMD to itself, so nothing runs beside this: three instructions an entry, the bound in the vocabulary's last tile alone and the lane's first column behind the loop (with
            // both in it, us without logits at N = 151936, K = 1024, with / so: 192 rows 112 / 107, 256 97 / 91, 512 150 / 144, 2048 530 / 505; K = 4096, 256 rows 316 / 309)
            float *sv = reinterpret_cast<float *>(smem + 2 * G_BUF); int *si = reinterpret_cast<int *>(smem + 2 * G_BUF + 1024);
            int lim = N - (bx * 256 + wn * 64 + q * 8);                   // vocabulary entries from the lane's first one on (opaque: no row of compares is kept over the K loop)
            int nv = N, tv = T;
            asm volatile("" : "+v"(lim), "+v"(nv), "+v"(tv));
            const int n_base = nv - lim;
            float bestv[2][4]; int besti[2][4];
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int ml = b * 128 + mrow + j * 16, m = m0 + ml;
                    hold(b, j);
                    float bv = -INFINITY; int bi = 0x7fffffff;
                    if (epi.logits) {
                        float *lrow = epi.logits + (int64_t)m * nv + n_base;
                        const int out = m < tv ? lim : 0;
#pragma unroll
                        for (int a = 0; a < 2; ++a)
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                if (const int c0 = a * 128 + (i >> 1) * 32 + (i & 1) * 4; c0 < out) *reinterpret_cast<float4_t *>(lrow + c0) = acc[a][i][b][j];
                    }
                    auto largest = [&](auto ragged) {
#pragma unroll
                        for (int a = 0; a < 2; ++a)
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const int c0 = a * 128 + (i >> 1) * 32 + (i & 1) * 4;
                                const float4_t v = acc[a][i][b][j];
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    const bool more = (!decltype(ragged)::value || c0 + e < lim) && v[e] > bv;
                                    bv = more ? v[e] : bv; bi = more ? c0 + e : bi;
                                }
                            }
                    };
                    if (bx * 256 + 256 <= N) largest(std::false_type{});
                    else largest(std::true_type{});
                    if (bi != 0x7fffffff) bi += n_base;
#pragma unroll
                    for (int o = 16; o < 64; o <<= 1) {
                        const float v2 = __shfl_xor(bv, o, 64); const int i2 = __shfl_xor(bi, o, 64);
                        const bool other = (v2 > bv) | ((v2 == bv) & (i2 < bi));
                        bv = other ? v2 : bv; bi = other ? i2 : bi;
                    }
                    bestv[b][j] = bv; besti[b][j] = bi;
                    if (wn == 1 && q == 0) { sv[ml] = bv; si[ml] = bi; }
                    __builtin_amdgcn_sched_barrier(0);
                }
            __syncthreads();
            if (wn == 0 && q == 0) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int ml = b * 128 + mrow + j * 16, m = m0 + ml;
                        float bv = bestv[b][j]; int bi = besti[b][j];
                        const float v2 = sv[ml]; const int i2 = si[ml];
                        if (v2 > bv || (v2 == bv && i2 < bi)) { bv = v2; bi = i2; }
                        if (m < tv) { epi.pval[(int64_t)bx * tv + m] = bv; epi.pidx[(int64_t)bx * tv + m] = bi; }
                    }
            }
            __syncthreads();                                              // (the next tile's partials go to the same place)
        } else if constexpr (g_rope(EPI)) {
            // Partners are in one lane: columns c .. c + 7 of a head's first half (A half 0) and the same ones of its second half (A half 1).  The products are rounded to 16 bits, then rotated.
            if (have_next) request_rows(tile_of(u + step), (tile_no + 1) & 1);
            const int *lds_pos = reinterpret_cast<const int *>(smem + 2 * G_BUF + (tile_no & 1) * 2048), *lds_slot = lds_pos + 256;
            const int head0 = bx * (256 / RD) + (RD == 64 ? wn * 2 : PH == 2 ? wn : 0);      // head of the wave's group p: head0 + (PH == 2 ? 0 : p)
            half8_t g1[2], g2[2];
            if constexpr (EPI == GEPI_QKN) {
                const half_t *w = head0 < epi.H ? epi.qn_w : epi.kn_w;
#pragma unroll
                for (int p = 0; p < 2; ++p) { g1[p] = *reinterpret_cast<const half8_t *>(w + p * 32 + q * 8); g2[p] = *reinterpret_cast<const half8_t *>(w + 64 + p * 32 + q * 8); }
            }
            const int cc0 = (RD == 128 && PH == 1 ? wn * 32 : 0) + q * 8; // column in the half head (PH == 2: + p*32)
            // rows of the caches and of y, from o1 (first half) and o2 (second half) of group p
            auto leave = [&](int t, int p, bool rot, half8_t o1, half8_t o2) {
                const int ml = (t >> 2) * 128 + mrow + (t & 3) * 16, m = m0 + ml, head = head0 + (PH == 2 ? 0 : p), c = (PH == 2 ? p * 32 : 0) + cc0;
                if (m >= T) return;
                if (head < epi.H || !epi.kv_cache_only) {
                    half_t *yrow = y + (int64_t)m * ldy + (int64_t)head * RD + c;
                    *reinterpret_cast<half8_t *>(yrow) = o1;
                    *reinterpret_cast<half8_t *>(yrow + hd2) = o2;
                }
                if (head >= epi.H) {
                    const int slot = epi.slots ? lds_slot[ml] : -1;
                    if (slot < 0) return;
                    half_t *crow = (rot ? epi.kc : epi.vc) + ((int64_t)slot * epi.KVH + (rot ? head - epi.H : head - epi.H - epi.KVH)) * RD + c;
                    *reinterpret_cast<half8_t *>(crow) = o1;
                    *reinterpret_cast<half8_t *>(crow + hd2) = o2;
                }
            };
            if (head0 < epi.H + epi.KVH) {                                // q and k heads rotate, v heads pass through
                constexpr int AHEAD = 4 - PH;                             // sines of a token tile's rows, requested three (QKN: two) tiles ahead
                float4_t cs[AHEAD][PH][2], sn[AHEAD][PH][2];
                auto sines = [&](int t) {
                    const int64_t at = (int64_t)lds_pos[(t >> 2) * 128 + mrow + (t & 3) * 16] * hd2 + cc0;
#pragma unroll
                    for (int p = 0; p < PH; ++p)
#pragma unroll
                        for (int hh = 0; hh < 2; ++hh) {
                            cs[t % AHEAD][p][hh] = *reinterpret_cast<const float4_t *>(epi.cos_t + at + p * 32 + hh * 4);
                            sn[t % AHEAD][p][hh] = *reinterpret_cast<const float4_t *>(epi.sin_t + at + p * 32 + hh * 4);
                        }
                };
#pragma unroll
                for (int t = 0; t < AHEAD; ++t) sines(t);
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const int b = t >> 2, j = t & 3;
                    half8_t x1[2], x2[2];
#pragma unroll
                    for (int p = 0; p < 2; ++p) { x1[p] = eight(0, p, b, j); x2[p] = eight(1, p, b, j); }
                    if constexpr (EPI == GEPI_QKN) head_norm_pieces(x1, x2, g1, g2, epi.qk_eps);
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const bool rot = PH == 2 || head0 + p < epi.H + epi.KVH;
                        half8_t o1 = x1[p], o2 = x2[p];
                        if (rot) {
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                const float f1 = (float)x1[p][e], f2 = (float)x2[p][e], cc = cs[t % AHEAD][PH == 2 ? p : 0][e >> 2][e & 3], ss = sn[t % AHEAD][PH == 2 ? p : 0][e >> 2][e & 3];
                                o1[e] = to_half_rn(mul_sub_unfused(f1, cc, f2, ss));
                                o2[e] = to_half_rn(mul_add_unfused(f2, cc, f1, ss));
                            }
                        }
                        leave(t, p, rot, o1, o2);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if (t + AHEAD < 8) sines(t + AHEAD);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int t = 0; t < 8; ++t) {
#pragma unroll
                    for (int p = 0; p < 2; ++p) leave(t, p, false, eight(0, p, t >> 2, t & 3), eight(1, p, t >> 2, t & 3));
                }
            }
        } else {
            constexpr int NA = g_glu(EPI) ? 1 : 2;
            half_t *yt = y + (int64_t)m0 * ldy + (int64_t)bx * OUTC + wn * 64;
            const unsigned lane_off = (unsigned)(mrow * ldy) + q * 8;
            half8_t res[EPI == GEPI_RESID ? 8 : 1][2][2];                 // RESID: the rows that are added to, requested four token tiles ahead
            auto residual = [&](int t) {
                const int b = t >> 2, j = t & 3;
                const bool in = m0 + b * 128 + mrow + j * 16 < T;
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int p = 0; p < 2; ++p)
                        res[EPI == GEPI_RESID ? t : 0][a][p] = in ? *reinterpret_cast<const half8_t *>(yt + (int64_t)(b * 128 + j * 16) * ldy + lane_off + a * 128 + p * 32) : (half8_t)(half_t)0;
            };
            if (EPI == GEPI_RESID) {
#pragma unroll
                for (int t = 0; t < 4; ++t) residual(t);
            }
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int b = t >> 2, j = t & 3;
                if (EPI == GEPI_RESID && t < 4) residual(t + 4);
                hold(b, j);
                const bool in = m0 + b * 128 + mrow + j * 16 < T;
                half_t *yrow = yt + (int64_t)(b * 128 + j * 16) * ldy + lane_off;
#pragma unroll
                for (int a = 0; a < NA; ++a)
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        half8_t o;
                        if constexpr (g_glu(EPI)) {
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                const float gf = (float)to_half_rn(acc[0][2 * p + (e >> 2)][b][j][e & 3]), uf = (float)to_half_rn(acc[1][2 * p + (e >> 2)][b][j][e & 3]);
                                if constexpr (EPI == GEPI_CLAMP) o[e] = to_half_rn(clamped_unit(gf, uf, epi.limit, epi.alpha));
                                else {
                                    const float sg = gate_factor(gf, EPI == GEPI_GELU);
                                    o[e] = to_half_rn(__fmul_rn(__fmul_rn(gf, sg), uf));
                                }
                            }
                        } else if constexpr (EPI == GEPI_RELU2) {
                            const half8_t v = eight(a, p, b, j);
#pragma unroll
                            for (int e = 0; e < 8; ++e) { const float f = fmaxf((float)v[e], 0.f); o[e] = (half_t)(f * f); }
                        } else if constexpr (EPI == GEPI_GELU_ERF) {
#pragma unroll
                            for (int e = 0; e < 8; ++e) o[e] = (half_t)gelu_erf_fast(acc[a][2 * p + (e >> 2)][b][j][e & 3]);
                        } else if constexpr (EPI == GEPI_RESID) {
                            // h <- fp16(h + fp16(acc)): the rounding points of add_rmsnorm's add
                            const half8_t v = eight(a, p, b, j);
#pragma unroll
                            for (int e = 0; e < 8; ++e) o[e] = to_half_rn((float)res[t][a][p][e] + (float)v[e]);
                        } else o = eight(a, p, b, j);
                        if (in) *reinterpret_cast<half8_t *>(yrow + a * 128 + p * 32) = o;
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        }   // epilogue scope
        ++tile_no;
        if (!have_next) break;
        u += step;
        tile = tile_of(u);
    }
#undef G256_PHASE
#undef G256_KTILE
}

static int g256_prepare() {                                               // 128 KiB of dynamic LDS: opt-in once
    static bool done = false;
    if (done) return 0;
    const void *fns[] = {reinterpret_cast<const void *>(&gemm256_kernel<GEPI_F16>), reinterpret_cast<const void *>(&gemm256_kernel<GEPI_SILU>),
                         reinterpret_cast<const void *>(&gemm256_kernel<GEPI_ROPE, 128>), reinterpret_cast<const void *>(&gemm256_kernel<GEPI_ROPE, 64>),
                         reinterpret_cast<const void *>(&gemm256_kernel<GEPI_RESID>), reinterpret_cast<const void *>(&gemm256_kernel<GEPI_LMHEAD>),
                         reinterpret_cast<const void *>(&gemm256_kernel<GEPI_F16, 0, true>), reinterpret_cast<const void *>(&gemm256_kernel<GEPI_SILU, 0, true>),
                         reinterpret_cast<const void *>(&gemm256_kernel<GEPI_RELU2>), reinterpret_cast<const void *>(&gemm256_kernel<GEPI_GELU>),
                         reinterpret_cast<const void *>(&gemm256_kernel<GEPI_GELU_ERF>), reinterpret_cast<const void *>(&gemm256_kernel<GEPI_QKN, 128>),
                         reinterpret_cast<const void *>(&gemm256_kernel<GEPI_CLAMP>)};
    for (const void *f : fns) {
        hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * G_BUF + 4096);
        if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "gemm256: hipFuncSetAttribute: %s", hipGetErrorString(e));
    }
    done = true;
    return 0;
}
static int g256_grid(int tiles) { return tiles < 256 ? (tiles + 7) / 8 * 8 : 256; }   // one persistent workgroup per CU (128 KiB of LDS each), as many on every XCD
static int g256_panel(int tiles_x) { const int panels = (tiles_x + 7) / 8; return (tiles_x + panels - 1) / panels; }   // columns of a panel: 8, or the next smaller number that makes the panels alike
static int g256_check(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return nvr::fail(NVR_ERR_HIP, "%s launch failed: %s", what, hipGetErrorString(e));
    return 0;
}
static constexpr bool g256_enabled() { return true; }

bool gemm256_ok(int64_t T, int64_t K, int64_t N, int64_t ldx) {
    return g256_enabled() && T >= 256 && K % G_BK == 0 && K >= 2 * G_BK && N % 256 == 0 && ldx % 8 == 0;
}
bool gemm256_silu_ok(int64_t T, int64_t K, int64_t I, int64_t ldx) {
    return g256_enabled() && T >= 256 && K % G_BK == 0 && K >= 2 * G_BK && I % 128 == 0 && ldx % 8 == 0;
}
bool gemm256_rope_ok(int64_t T, int64_t K, int64_t H, int64_t KVH, int64_t D, int64_t ldx) {
    return g256_enabled() && T >= 256 && K % G_BK == 0 && K >= 2 * G_BK && (D == 128 || D == 64) && ((H + 2 * KVH) * D) % 256 == 0 && ldx % 8 == 0;
}

int gemm256(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, half_bits *y, hipStream_t s) {
    if (!gemm256_ok(T, K, N, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    if (int rc = g256_prepare()) return rc;
    const int tx = (int)(N / 256), tt = tx * (int)((T + 255) / 256);
    gemm256_kernel<GEPI_F16><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                        (int)N, (int)N, (half_t *)y, G256Epi{}, tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256");
}
// y = max(x . W^T, 0)^2: a dense feed-forward's up product with its squared ReLU in the epilogue
int gemm256_relu2(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, half_bits *y, hipStream_t s) {
    if (!gemm256_ok(T, K, N, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_relu2: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    if (int rc = g256_prepare()) return rc;
    const int tx = (int)(N / 256), tt = tx * (int)((T + 255) / 256);
    gemm256_kernel<GEPI_RELU2><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                          (int)N, (int)N, (half_t *)y, G256Epi{}, tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256_relu2");
}
// y = gelu(x . W^T) with the error function, of the unrounded product
int gemm256_gelu(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, half_bits *y, hipStream_t s) {
    if (!gemm256_ok(T, K, N, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_gelu: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    if (int rc = g256_prepare()) return rc;
    const int tx = (int)(N / 256), tt = tx * (int)((T + 255) / 256);
    gemm256_kernel<GEPI_GELU_ERF><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                             (int)N, (int)N, (half_t *)y, G256Epi{}, tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256_gelu");
}
// Rows grouped by expert (a mixture of experts over many tokens): T is a multiple of 256 and row block rb multiplies the matrix W + row_w[rb] * w_stride
// (row_w on the device: the host does not know how many rows an expert got).  y = x . W_e^T, or out = silu(gate) * up with W_e = [gate rows; up rows].
int gemm256_grouped(const half_bits *x, int64_t ldx, const half_bits *W, int64_t w_stride, const int32_t *row_w, int64_t T, int64_t K, int64_t N, half_bits *y, hipStream_t s, const int32_t *rows_used) {
    if (!gemm256_ok(T, K, N, ldx) || T % 256) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_grouped: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    if (int rc = g256_prepare()) return rc;
    G256Epi e{}; e.row_w = row_w; e.w_stride = w_stride; e.rows_used = rows_used;
    const int tx = (int)(N / 256), tt = tx * (int)(T / 256);
    gemm256_kernel<GEPI_F16, 0, true><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K, (int)N, (int)N, (half_t *)y, e, tx,
                                                                                                  tt / tx, g256_panel(tx));
    return g256_check("gemm256_grouped");
}
int gemm256_grouped_silu_mul(const half_bits *x, int64_t ldx, const half_bits *W, int64_t w_stride, const int32_t *row_w, int64_t T, int64_t K, int64_t I, half_bits *out, hipStream_t s, const int32_t *rows_used) {
    if (!gemm256_silu_ok(T, K, I, ldx) || T % 256) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_grouped_silu_mul: T=%ld K=%ld I=%ld", (long)T, (long)K, (long)I);
    if (int rc = g256_prepare()) return rc;
    G256Epi e{}; e.row_w = row_w; e.w_stride = w_stride; e.rows_used = rows_used;
    const int tx = (int)(I / 128), tt = tx * (int)(T / 256);
    gemm256_kernel<GEPI_SILU, 0, true><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K, (int)I, (int)(2 * I), (half_t *)out, e,
                                                                                                   tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256_grouped_silu_mul");
}
// h[T,N] <- fp16(h + fp16(x·Wᵀ)): the row-parallel GEMM with the residual add of qwen3.rs:382,389 in its epilogue (prefill steps on one
// rank: the following norm then reads ONE tensor instead of h and the projection)
int gemm256_resid(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, half_bits *h, hipStream_t s) {
    if (!gemm256_ok(T, K, N, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_resid: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    if (int rc = g256_prepare()) return rc;
    const int tx = (int)(N / 256), tt = tx * (int)((T + 255) / 256);
    gemm256_kernel<GEPI_RESID><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                          (int)N, (int)N, (half_t *)h, G256Epi{}, tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256_resid");
}
int gemm256_silu_mul(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t I, half_bits *out, hipStream_t s) {
    if (!gemm256_silu_ok(T, K, I, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_silu_mul: T=%ld K=%ld I=%ld", (long)T, (long)K, (long)I);
    if (int rc = g256_prepare()) return rc;
    const int tx = (int)(I / 128), tt = tx * (int)((T + 255) / 256);
    gemm256_kernel<GEPI_SILU><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                         (int)I, (int)(2 * I), (half_t *)out, G256Epi{}, tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256_silu_mul");
}
// out = gelu(gate) * up with the tanh form of gelu
int gemm256_gelu_mul(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t I, half_bits *out, hipStream_t s) {
    if (!gemm256_silu_ok(T, K, I, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_gelu_mul: T=%ld K=%ld I=%ld", (long)T, (long)K, (long)I);
    if (int rc = g256_prepare()) return rc;
    const int tx = (int)(I / 128), tt = tx * (int)((T + 255) / 256);
    gemm256_kernel<GEPI_GELU><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                         (int)I, (int)(2 * I), (half_t *)out, G256Epi{}, tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256_gelu_mul");
}
// the clamped gated unit, rows of out ldo apart
int gemm256_clamped_glu(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t I, float limit, float alpha, half_bits *out, int64_t ldo, hipStream_t s) {
    if (!gemm256_silu_ok(T, K, I, ldx) || ldo % 8 || ldo < I) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_clamped_glu: T=%ld K=%ld I=%ld", (long)T, (long)K, (long)I);
    if (int rc = g256_prepare()) return rc;
    G256EpiClamp e{}; e.limit = limit; e.alpha = alpha; e.ldo = ldo;
    const int tx = (int)(I / 128), tt = tx * (int)((T + 255) / 256);
    gemm256_kernel<GEPI_CLAMP><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                          (int)I, (int)(2 * I), (half_t *)out, e, tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256_clamped_glu");
}
int gemm256_qkv_rope_store(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t H, int64_t KVH, int64_t D,
                           const int64_t *positions, const int32_t *slots, const float *cos_t, const float *sin_t, half_bits *qkv,
                           half_bits *k_cache, half_bits *v_cache, hipStream_t s, bool kv_cache_only, const QkNorm *norm) {
    if (norm && D != 128) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_qkv_rope_store: head norms with D=%ld", (long)D);
    if (!gemm256_rope_ok(T, K, H, KVH, D, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_qkv_rope_store: T=%ld K=%ld D=%ld", (long)T, (long)K, (long)D);
    if (int rc = g256_prepare()) return rc;
    const int64_t N = (H + 2 * KVH) * D;
    G256EpiNorm e{};
    e.pos = positions; e.slots = slots; e.cos_t = cos_t; e.sin_t = sin_t; e.kc = (half_t *)k_cache; e.vc = (half_t *)v_cache;
    e.H = (int32_t)H; e.KVH = (int32_t)KVH; e.D = (int32_t)D;
    e.kv_cache_only = (kv_cache_only && slots && k_cache && v_cache) ? 1 : 0;
    const int tx = (int)(N / 256), tt = tx * (int)((T + 255) / 256);
    if (norm) {
        e.qn_w = (const half_t *)norm->q_w; e.kn_w = (const half_t *)norm->k_w; e.qk_eps = norm->eps;
        gemm256_kernel<GEPI_QKN, 128><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF + 4096, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                                  (int)N, (int)N, (half_t *)qkv, e, tx, tt / tx, g256_panel(tx));
    } else if (D == 128)
        gemm256_kernel<GEPI_ROPE, 128><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF + 4096, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                                  (int)N, (int)N, (half_t *)qkv, e, tx, tt / tx, g256_panel(tx));
    else
        gemm256_kernel<GEPI_ROPE, 64><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF + 4096, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                                 (int)N, (int)N, (half_t *)qkv, e, tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256_qkv_rope_store");
}

// LM head over >= G256_LM_MIN_T (192) rows (large decode batches: 512 sequences — and many-sequence prefills): f32 logits on demand,
// one (max, lowest index) partial per 256-column tile and row; N any multiple of 16
constexpr int64_t G256_LM_MIN_T = 192;     // (us without logits, K = 1024, N = 151936: 128x128 tiles 78 at 128 rows, 129 at 160..192, 132 at 256; these tiles 90..107 at 192..256; K = 4096: 270, 470, 483; 298..309)
bool gemm256_lm_head_ok(int64_t T, int64_t K, int64_t N, int64_t ldx) {
    return g256_enabled() && T >= G256_LM_MIN_T && T <= 65536 && K % G_BK == 0 && K >= 2 * G_BK && N % 16 == 0 && N >= 256 && ldx % 8 == 0 &&
           (N + 255) / 256 <= LM_HEAD_MAX_PARTS && N < (1ll << 31) && ((N + 255) / 256) * ((T + 255) / 256) < (1ll << 30);
}
int gemm256_lm_head(const half_bits *x, int64_t ldx, const half_bits *W, int64_t T, int64_t K, int64_t N, float *logits, float *part_val,
                    int32_t *part_idx, int32_t *nparts, hipStream_t s) {
    if (!gemm256_lm_head_ok(T, K, N, ldx)) return nvr::fail(NVR_ERR_UNSUPPORTED, "gemm256_lm_head: T=%ld K=%ld N=%ld", (long)T, (long)K, (long)N);
    if (int rc = g256_prepare()) return rc;
    G256Epi e{};
    e.logits = logits; e.pval = part_val; e.pidx = part_idx;
    const int tx = (int)((N + 255) / 256), tt = tx * (int)((T + 255) / 256);
    *nparts = tx;
    gemm256_kernel<GEPI_LMHEAD><<<dim3((unsigned)g256_grid(tt)), dim3(G_THREADS), 2 * G_BUF + 2048, s>>>((const half_t *)x, ldx, (const half_t *)W, (int)T, (int)K,
                                                                                           (int)N, (int)N, nullptr, e, tx, tt / tx, g256_panel(tx));
    return g256_check("gemm256_lm_head");
}

}}  // namespace nvr::k / nvr::kb (NVR_DT_NS)
