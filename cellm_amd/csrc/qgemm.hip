// MLX 4-bit GEMM on MFMA for prefill and batched decode over f16 activations (gfx950).
//
//   Y[M,N] = X[M,K] . dequant(W)[N,K]^T        (f16 X, f32 accumulate, f32 Y)
//
// Reference: there is no batched or GEMM path in cellm (prefill runs the GEMV
// token by token, crates/cellm-model/src/llama.rs:214-233).  The per-element
// oracle is cpu_kernels::matmul_f32 (cpu_kernels.rs:36-63) over the dequantized
// weight, summed over k ascending.
//
// Weights are dequantized to f16 with the converter's rounding,
// h = RNE_f16(f32(q)*s + b) (tools/convert/src/main.rs:4435-4436): into LDS
// tiles by qgemm_kernel, in registers right before each MFMA by the q4 kernel
// for K % 128 == 0.  For f16 or bf16 scales, f32(q)*s is exact in f32, so
// fma(q, s, b) rounds exactly as the reference's mul-then-add does; f32
// scales take a separate mul and add.
//
// Tiling: 256 threads = 4 waves in a 2x2 grid; block tile 128x128, wave tile
// 64x64 = 4x4 v_mfma_f32_16x16x32_f16 tiles; BK = 64 per LDS stage.  The next
// stage's global data is prefetched into registers during the MFMA loop.
// Split-K over blockIdx.z writes f32 partials to a workspace that a second
// kernel sums in a fixed order (deterministic).
#include <mutex>
#include <utility>
#include <vector>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "lds_dma.hpp"

namespace cellm {

namespace {

constexpr int BM = 128, BN = 128, BK = 64;
constexpr int LDS_STRIDE = BK + 8;  // halves; 144-byte rows break LDS bank aliasing
constexpr int kThreads = 256;
constexpr int kStages = 4;  // register prefetch depth (K stages of 64 in flight)

template <int SBT>
__device__ __forceinline__ h8_t dequant_word_f16(uint32_t w, float s, float b)
{
    h8_t h;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float q = (float)((w >> (4 * k)) & 0xFu);
        float v;
        if constexpr (SBT == DT_F32) {
#pragma clang fp contract(off)
            const float t = q * s;
            v = t + b;
        } else {
            v = __builtin_fmaf(q, s, b);  // q*s exact: same bits as mul-then-add
        }
        // Keep the f32 rounding: without this barrier the compiler folds the
        // fma and the f16 narrowing into one v_fma_mix*_f16, which rounds once
        // instead of the reference's twice (f32, then f16).
        asm volatile("" : "+v"(v));
        h[k] = (_Float16)v;
    }
    return h;
}

// One K stage (BK = 64) of global data held in registers by one thread:
// its 32-element halves of one X row and one W row, plus the W row's scale
// and bias bits for that group (raw, converted when the tile is stored).
struct StageRegs {
    u4_t x[4];
    u4_t w;  // 32 nibbles
    uint32_t s, b;
};

// q4 affine (u32 words).  NS = register prefetch depth.
template <int SBT, int NS>
__global__ __launch_bounds__(kThreads) void qgemm_kernel(const void* __restrict__ W, const void* __restrict__ S,
                                                         const void* __restrict__ Bz, int group_size,
                                                         const _Float16* __restrict__ X, float* __restrict__ Y,
                                                         int M, int N, int K, int k_per_split)
{
    // two LDS buffers: stage s is stored into buffer s&1 while no wave can
    // still read it (every wave passed the barrier after its compute of s-2)
    __shared__ __align__(16) _Float16 xs[2][BM * LDS_STRIDE];
    __shared__ __align__(16) _Float16 ws[2][BN * LDS_STRIDE];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int kbeg = blockIdx.z * k_per_split;
    const int kend = min(K, kbeg + k_per_split);
    const int nsteps = kend > kbeg ? (kend - kbeg) / BK : 0;  // K % 64 == 0, k_per_split % 64 == 0

    // global -> register assignment: thread = (row, 32-element half of the stage)
    const int ld_row = tid >> 1;
    const int ld_half = tid & 1;
    // Rows past M or N are clamped to the last valid row: their loads stay in
    // bounds without a branch and their results are never stored.
    const int xm = min(m0 + ld_row, M - 1), wn_row = min(n0 + ld_row, N - 1);
    const int gshift = __builtin_ctz((unsigned)group_size);
    const int gpr = (K + group_size - 1) >> gshift;
    const u4_t* w4 = reinterpret_cast<const u4_t*>(W);

    auto load_stage = [&](int step, StageRegs& r) {
        const int kc = kbeg + min(step, nsteps - 1) * BK + ld_half * 32;  // clamped: tail slots reload the last stage
#pragma unroll
        for (int i = 0; i < 4; ++i) r.x[i] = *reinterpret_cast<const u4_t*>(X + (size_t)xm * K + kc + i * 8);
        r.w = __builtin_nontemporal_load(w4 + ((size_t)wn_row * K + kc) / 32);
        const size_t gi = (size_t)wn_row * gpr + (kc >> gshift);
        r.s = load_raw<SBT>(S, gi);
        r.b = load_raw<SBT>(Bz, gi);
    };

    auto store_stage = [&](const StageRegs& r, int buf) {
        _Float16* xd = xs[buf] + ld_row * LDS_STRIDE + ld_half * 32;
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<u4_t*>(xd + i * 8) = r.x[i];
        _Float16* wd = ws[buf] + ld_row * LDS_STRIDE + ld_half * 32;
        const float sc = raw_to_f32<SBT>(r.s), bi = raw_to_f32<SBT>(r.b);
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<h8_t*>(wd + i * 8) = dequant_word_f16<SBT>(r.w[i], sc, bi);
    };

    f4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};

    const int frag_row = lane & 15;
    const int frag_k = (lane >> 4) * 8;
    auto compute = [&](int buf) {
#pragma unroll
        for (int kk = 0; kk < BK; kk += 32) {
            h8_t a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                a[i] = *reinterpret_cast<const h8_t*>(xs[buf] + (wm * 64 + i * 16 + frag_row) * LDS_STRIDE + kk + frag_k);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                b[j] = *reinterpret_cast<const h8_t*>(ws[buf] + (wn * 64 + j * 16 + frag_row) * LDS_STRIDE + kk + frag_k);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };

    if (nsteps > 0) {
        // Software pipeline.  Stage s is in LDS buffer s&1 when step s starts;
        // step s dequantizes and stores stage s+1 into the other buffer while
        // its own MFMAs run (same basic block, so VALU issues in the MFMA
        // shadow), then one barrier, then the freed ring slot is refilled with
        // stage s+1+NS.  Buffer (s+1)&1 last held stage s-1, which every wave
        // finished reading before the barrier that ended step s-1.
        StageRegs ring[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) load_stage(j, ring[j]);
        store_stage(ring[0], 0);
        __syncthreads();
        load_stage(NS, ring[0]);
        for (int s0 = 0; s0 < nsteps; s0 += NS) {
#pragma unroll
            for (int j = 0; j < NS; ++j) {
                const int s = s0 + j;
                if (s < nsteps) {
                    // past the end this stores a clamped copy of the last stage
                    // into the idle buffer; nobody reads it
                    store_stage(ring[(j + 1) % NS], (s + 1) & 1);
                    compute(s & 1);
                }
                // The barrier and the reload run on every path (s is block-uniform and
                // the reload is clamped), so each unrolled step issues the same loads
                // and the compiler's vmcnt stays partial across the loop back edge.
                __syncthreads();
                load_stage(s + 1 + NS, ring[(j + 1) % NS]);
            }
        }
    }

    // C fragment: lane holds rows 4*(lane/16)+e, column lane%16 of each 16x16 tile.
    float* out = Y + (size_t)blockIdx.z * M * N;
    const int crow = (lane >> 4) * 4;
    const int ccol = lane & 15;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = n0 + wn * 64 + j * 16 + ccol;
        if (n >= N) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + wm * 64 + i * 16 + crow + e;
                if (m < M) out[(size_t)m * N + n] = acc[i][j][e];
            }
        }
    }
}

// Sum split-K partials [splits][M*N] in split order.
__global__ void splitk_reduce_kernel(const float* __restrict__ part, float* __restrict__ y, int splits, int M, int N)
{
    const size_t total = (size_t)M * N;
    if ((N & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {
        // four columns of one row per thread: 16-byte loads of every split's partials
        const size_t n4 = total >> 2;
        for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x) {
            reinterpret_cast<f4_t*>(y)[i] = sum_splits_f4(reinterpret_cast<const f4_t*>(part) + i, n4, splits);
        }
        return;
    }
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        float v = part[i];
        for (int s = 1; s < splits; ++s) v += part[(size_t)s * total + i];
        y[i] = v;
    }
}

// ---------------------------------------------------------------------------
// Direct-to-LDS helpers for the q4 qGEMM below (K % 128 == 0): LDS tiles hold
// rows of 16 chunks of 8 halves, chunk position XOR-swizzled by (row & 15) so
// that the 16 rows a fragment read touches fall in 16 distinct 4-bank groups.
// ---------------------------------------------------------------------------
namespace dma {

using namespace ldsdma;

constexpr int BK = 128;
constexpr int kStageHalves = BM * BK;       // one f16 X or W tile

__device__ __forceinline__ int slot(int r, int c) { return r * 16 + (c ^ (r & 15)); }

// ---------------------------------------------------------------------------
// q4 affine qGEMM, dequant at the MFMA (K % 128 == 0).
//
// 512 threads = 8 waves, two per SIMD; block tile 128 (M) x 128 (N).  Wave
// (kh, ns) owns a 128 x 32 tile (four v_mfma_f32_32x32x16_f16 accumulators)
// over k half kh of every 128-wide k-step; the two halves are added through
// LDS after the loop.  X (f16) and the raw nibbles of W go global -> LDS by
// global_load_lds_dwordx4 through a ring of three stages (stage = one k-step:
// X 128 x 128 halves, swizzled as above, and W 128 columns x 64 bytes),
// issued two steps ahead; the f16 weights never touch LDS.  Lane
// (r32 = lane % 32, h32 = lane / 32) owns column n0 + 32 ns + r32 and the 32 k
// starting at 64 kh + 32 h32 of each step (16 bytes of nibbles, one LDS read).
// The MFMA's k order is free as long as X and W agree, so k-slot group h32 of
// substep ks is k = 64 kh + 32 h32 + 8 ks + 0..7: one nibble word of the lane,
// dequantized right before its MFMAs, and chunk 8 kh + 4 h32 + ks of the X row.
// Every weight is dequantized once, by the lane that multiplies it, and LDS
// carries no f16 weight tile.
// Dequant: bytes of (w & 0x0F0F0F0F) and ((w >> 4) & 0x0F0F0F0F) convert with
// v_cvt_f32_ubyteN, then fma(q, s, b) in f32 (mul then add for f32 scales)
// and a round-to-nearest-even pack to f16: the converter's
// RNE_f16(f32(q) * s + b).
// The loop holds no compiler-visible global access (the DMA is inline asm
// waited for by explicit counts): a register prefetch of W made the compiler
// copy the loaded registers between iterations behind a vmcnt(0), which
// drained every load in flight at each step.  Measured per k-step on the box:
// X fragment reads plus DMA (~170 KB of LDS traffic per CU) 0.48 us, with the
// MFMAs 0.82 us, everything 1.04 us; one wave per SIMD (4 waves, 128 x 32
// tiles over the whole step) took 1.36 us.
// ---------------------------------------------------------------------------
constexpr int kRegThreads = 512;
constexpr int kRegStages = 3;
constexpr int kRawStepBytes = BN * BK / 2;                           // W nibbles of one k-step
constexpr int kRegStageBytes = kStageHalves * 2 + kRawStepBytes;    // 40 KB
constexpr size_t kRegFixedLds = (size_t)kRegStages * kRegStageBytes;
constexpr size_t kRegExchangeBytes = 8 * 2 * 16 * 64 * 4;  // k-half exchange after the loop (64 KB)

struct RegArgs {
    Q4FusedSeg seg[3];
    int tile0[3];  // first column tile of each segment; of an absent one, past every tile
    int gshift, M, K, k_per_split, act;
    const _Float16* X;
    float* part;   // split sums [split][M][N] of the one segment, or nullptr
};

// REG_MANY: up to three matrices share X, column tiles of one grid, with their biases.  REG_ACT: segments 0 and 1
// are gate and up, a tile's four 32-column slices are gate, up, gate, up of the same 64 outputs, and
// h = act(gate) * up leaves the tile (both unsplit only).  At 512 rows of 896, 2 x 4864 columns took 13.2 us twice
// and 5 us for the activation over three f32 matrices, now 26.3 (304 tiles are two rounds of 256 blocks); q/k/v of
// 896 and 2 x 16 columns 32.2 -> 11.6.  One matrix has an instance of its own, without the selects and the bias:
// with them 10.9 -> 11.3 us at 512 x 896 x 896.
enum RegMode { REG_ONE, REG_MANY, REG_ACT };

template <int SBT, RegMode MODE>
__global__ __launch_bounds__(kRegThreads) void qgemm_q4_regw_kernel(const RegArgs a)
{
    constexpr bool ACT = MODE == REG_ACT;
    extern __shared__ __align__(16) unsigned char smem[];
    // stage t: X tile at t * kRegStageBytes, W raw at + kStageHalves * 2; then the scales/biases
    uint32_t* sbl = reinterpret_cast<uint32_t*>(smem + kRegFixedLds);  // [BN][groups] as in the DMA kernel
    // wn through readfirstlane: the DMA's LDS bases derived from it stay scalar arithmetic.  Wave
    // wn = (kh, ns): k half kh of every step, 32-column slice ns of the tile.
    const int tid = threadIdx.x, lane = tid & 63, wn = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kh = wn >> 2, ns = wn & 3;
    const int r32 = lane & 31, h32 = lane >> 5;
    const int M = a.M, K = a.K, gshift = a.gshift, vt = blockIdx.x;
    // selects between arguments that are all loaded at once, not a chain of loads through an index
    const Q4FusedSeg su = a.seg[1];
    Q4FusedSeg sg = a.seg[0];
    int tile0 = 0;
    if constexpr (MODE == REG_MANY) {
        const Q4FusedSeg s2 = a.seg[2];
        const int t1 = a.tile0[1], t2 = a.tile0[2];
        const bool c1 = vt >= t1, c2 = vt >= t2;
        const auto pick = [&](auto x0, auto x1, auto x2) { return c2 ? x2 : c1 ? x1 : x0; };
        sg = Q4FusedSeg{pick(sg.w, su.w, s2.w),    pick(sg.S, su.S, s2.S), pick(sg.B, su.B, s2.B),
                        pick(sg.bias, su.bias, s2.bias), pick(sg.y, su.y, s2.y), pick(sg.n, su.n, s2.n)};
        tile0 = pick(0, t1, t2);
    }
    const int N = sg.n;
    const int n0 = ACT ? vt * (BN / 2) : (vt - tile0) * BN, m0 = blockIdx.y * BM;
    // tile column -> matrix column past n0
    const auto column = [](int c) { return ACT ? (c >> 6) * 32 + (c & 31) : c; };
    const int kbeg = blockIdx.z * a.k_per_split;
    const int kend = min(K, kbeg + a.k_per_split);
    const int nsteps = (kend - kbeg) / BK;
    float* o = a.part ? a.part + (size_t)blockIdx.z * M * N : sg.y;
    if (nsteps <= 0) return;  // the launcher never makes an empty split
    const int last = nsteps - 1;
    const int gpr = (K + (1 << gshift) - 1) >> gshift;
    const int g0 = kbeg >> gshift;
    const int ng = ((kend - 1) >> gshift) - g0 + 1;

    // X DMA: 4 per wave per stage, load j covers tile rows (wn * 4 + j) * 4 .. +4; byte offsets from
    // X + 2 kbeg (the launcher keeps M K 2 below 2^32)
    uint32_t xoff[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = (wn * 4 + j) * 4 + (lane >> 4);
        const int c = (lane & 15) ^ (r & 15);
        xoff[j] = (uint32_t)((size_t)min(m0 + r, M - 1) * K * 2 + 16 * c);
    }
    // W DMA: 1 per wave per stage, covering columns wn * 16 .. +16, 64 bytes each (columns past N
    // re-read the last one: computed, never stored); byte offsets from W + kbeg / 2
    const uint32_t woff =
        (uint32_t)((size_t)min(n0 + column(wn * 16 + (lane >> 2)), N - 1) * (K / 2) + 16 * (lane & 3));
    const unsigned char* xbase = reinterpret_cast<const unsigned char*>(a.X) + (size_t)kbeg * 2;
    const unsigned char* wbase = reinterpret_cast<const unsigned char*>(ACT && (wn & 2) ? su.w : sg.w) + kbeg / 2;
    const uint32_t lds0 = lds_addr(smem);
    auto issue = [&](int step) {
        const int sc = min(step, last), st = step % kRegStages;
        const uint32_t base = lds0 + st * kRegStageBytes;
        const unsigned char* xs_ = xbase + (size_t)sc * BK * 2;
        const unsigned char* ws_ = wbase + (size_t)sc * (BK / 2);
#pragma unroll
        for (int j = 0; j < 4; ++j) dma16_s(xoff[j], xs_, base + (wn * 4 + j) * 1024);
        dma16_s(woff, ws_, base + kStageHalves * 2 + wn * 1024);
    };

    issue(0);
    {
        // scales/biases of this split's groups, loads batched before any use
        constexpr int PB = 8;
        const int total = BN * ng;
        for (int base = tid; base < total; base += PB * kRegThreads) {
            uint32_t sv[PB], bv[PB];
#pragma unroll
            for (int u = 0; u < PB; ++u) {
                const int i = min(base + u * kRegThreads, total - 1);
                const int col = i / ng, gi = i - col * ng;
                const size_t idx = (size_t)min(n0 + column(col), N - 1) * gpr + g0 + gi;
                sv[u] = load_raw<SBT>(ACT && (col & 32) ? su.S : sg.S, idx);
                bv[u] = load_raw<SBT>(ACT && (col & 32) ? su.B : sg.B, idx);
            }
#pragma unroll
            for (int u = 0; u < PB; ++u) {
                // unconditional (slots past the end rewrite the last one with its own value): a load
                // consumed only under a branch stays pending for the compiler on the other path, and
                // the first reuse of its register inside the k-loop became a vmcnt(0) drain per step
                const int i = min(base + u * kRegThreads, total - 1);
                if constexpr (SBT == DT_F32) {
                    sbl[2 * i] = sv[u];
                    sbl[2 * i + 1] = bv[u];
                } else {
                    sbl[i] = sv[u] | (bv[u] << 16);
                }
            }
        }
    }
    __syncthreads();
    issue(1);

    const int lcol = ns * 32 + r32;
    auto scale_bias = [&](int k) {
        const int gi = ((kbeg + k) >> gshift) - g0;
        float sc, bi;
        if constexpr (SBT == DT_F32) {
            sc = __builtin_bit_cast(float, sbl[2 * (lcol * ng + gi)]);
            bi = __builtin_bit_cast(float, sbl[2 * (lcol * ng + gi) + 1]);
        } else {
            const uint32_t sb = sbl[lcol * ng + gi];
            sc = raw_to_f32<SBT>(sb & 0xFFFFu);
            bi = raw_to_f32<SBT>(sb >> 16);
        }
        return make_float2(sc, bi);
    };

    f16v_t acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f16v_t{};
    for (int s = 0; s < nsteps; ++s) {
        // Stage s was issued two steps ago; only stage s + 1 (5 loads per thread) may stay in flight.
        // A bare s_barrier: __syncthreads()'s release fence waits for vmcnt(0), i.e. for every DMA in
        // flight.  The asm waits carry memory clobbers, so no LDS access moves across them.
        wait_vmcnt<5>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();  // stage s complete everywhere; stage s - 1 no longer read
        issue(s + 2);                  // into the ring slot of stage s - 1
        const unsigned char* sbase = smem + (s % kRegStages) * kRegStageBytes;
        const _Float16* xa = reinterpret_cast<const _Float16*>(sbase);
        // this lane's 32 k of the step: k = 64 kh + 32 h32 + 8 ks + 0..7 (substep ks = 0..3)
        const u4_t w = *reinterpret_cast<const u4_t*>(sbase + kStageHalves * 2 + lcol * 64 + 32 * kh + 16 * h32);
        const float2 sb = scale_bias(s * BK + 64 * kh + 32 * h32);
        // A fragments are read one substep ahead of their MFMAs
        h8_t a[2][4];
        auto read_a = [&](int ks, h8_t (&dst)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                dst[i] = *reinterpret_cast<const h8_t*>(xa + slot(i * 32 + r32, 8 * kh + 4 * h32 + ks) * 8);
        };
        read_a(0, a[0]);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            if (ks + 1 < 4) read_a(ks + 1, a[(ks + 1) & 1]);
            const h8_t b = dequant_word_bytes<SBT>(w[ks], sb.x, sb.y);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks & 1][i], b, acc[i], 0, 0, 0);
        }
    }
    // drain the trailing (re-read) DMA before the stage memory is reused
    wait_vmcnt<0>();
    __syncthreads();

    // The two k halves meet through LDS: wave (kh, ns) hands the row tiles the other half keeps to
    // its partner (kh = 0 keeps rows 0..63, kh = 1 rows 64..127) and adds what it receives; lane l
    // exchanges with lane l of the partner, 8 KB per wave.  All partner values are read before any
    // add or store (one LDS round trip instead of one per store).
    float* xch = reinterpret_cast<float*>(smem);
    const int ncol = n0 + column(lcol);
    auto finish = [&](auto keep_c) {
        constexpr int KEEP = decltype(keep_c)::value, GIVE = 2 - KEEP;  // constant indices: no scratch
        // arrived before the stores: a load still pending there makes every guarded store wait for the one
        // before it (10.9 against 14.0 us at 512 x 896 x 896)
        float bias = MODE == REG_MANY && sg.bias ? sg.bias[min(ncol, N - 1)] : 0.0f;
        asm volatile("" : "+v"(bias));
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) xch[(((wn * 2 + t) * 16 + r) * 64) + lane] = acc[GIVE + t][r];
        __syncthreads();
        float other[2][16];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) other[t][r] = xch[((((wn ^ 4) * 2 + t) * 16 + r) * 64) + lane];
        if constexpr (ACT) {
            // every wave's sums back to LDS, then half a gate tile and its up tile for each: the waves that hold
            // the gate slices sit on two of the four SIMDs, which took 15.4 us at 65 x 896 x 2 x 896, this 12.9
            float* mine = xch + kRegExchangeBytes / 4 + (size_t)wn * 2 * 16 * 64;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) mine[(t * 16 + r) * 64 + lane] = acc[KEEP + t][r] + other[t][r];
            __syncthreads();
            const int t = ns & 1, n = n0 + (ns >> 1) * 32 + r32;
            const float* gate = xch + kRegExchangeBytes / 4 + (size_t)((wn & ~1) * 2 + t) * 16 * 64 + lane;
            const float* up = gate + 2 * 16 * 64;
            if (n >= N) return;
            const auto rows = [&](auto act) {
#pragma unroll 8
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + (KEEP + t) * 32 + (r >> 2) * 8 + h32 * 4 + (r & 3);
                    const float v = act_mul(decltype(act)::value, gate[r * 64], up[r * 64]);
                    if (m < M) __builtin_nontemporal_store(v, o + (size_t)m * N + n);
                }
            };
            if (a.act == ACT_GELU_TANH)
                rows(std::integral_constant<int, ACT_GELU_TANH>{});
            else
                rows(std::integral_constant<int, ACT_SILU>{});
            return;
        }
        if (ncol >= N) return;
        const bool biased = MODE == REG_MANY && sg.bias;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                // register r of a 32x32 tile: row (r/4)*8 + (lane/32)*4 + r%4, column lane%32
                const int m = m0 + (KEEP + t) * 32 + (r >> 2) * 8 + h32 * 4 + (r & 3);
                const float v = acc[KEEP + t][r] + other[t][r];
                if (m < M) __builtin_nontemporal_store(biased ? v + bias : v, o + (size_t)m * N + ncol);
            }
    };
    if (kh == 0)
        finish(std::integral_constant<int, 0>{});
    else
        finish(std::integral_constant<int, 2>{});
}

#ifndef CELLM_QGEMM_MIN_SPLIT_STEPS
#define CELLM_QGEMM_MIN_SPLIT_STEPS 4
#endif
constexpr int kMinSplitSteps = CELLM_QGEMM_MIN_SPLIT_STEPS;  // k-steps per split at least

struct Plan {
    int splits;
    int k_per_split;
    size_t lds;
};

// Split-K so the grid covers the 256 CUs (each split >= 4 steps), and enough
// splits that a split's scales/biases fit the LDS left by the tiles.
Plan plan(int M, int N, int K, int group, int sbt, size_t fixed_lds)
{
    Plan p{0, 0, 0};
    if (K <= 0 || K % BK != 0 || group < 32) return p;
    const int tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    const int steps = K / BK;
    int splits = 1;
    while (tiles * splits * 2 <= 256 && steps / (splits * 2) >= kMinSplitSteps) splits *= 2;
    const size_t sb_bytes = sbt == DT_F32 ? 8 : 4;
    for (;;) {
        const int sps = (steps + splits - 1) / splits;
        const int kps = sps * BK;
        const int ng = (kps + group - 1) / group + 1;  // + 1: a split may start mid-group
        const size_t lds = fixed_lds + (size_t)BN * ng * sb_bytes;
        if (lds <= kMaxLds) {
            p.splits = (steps + sps - 1) / sps;  // no empty split
            p.k_per_split = kps;
            p.lds = lds;
            return p;
        }
        if (sps == 1) return Plan{0, 0, 0};
        ++splits;
    }
}

}  // namespace dma

}  // namespace

// Choose the split-K factor so the grid covers the chip: 256 CUs.
int qgemm_splits(int M, int N, int K)
{
    const int tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    const int ksteps = (K + BK - 1) / BK;
    int splits = 1;
    // one round of blocks on 256 CUs; each split keeps >= 8 stages so the
    // prefetch ring has something to overlap
    while (tiles * splits * 2 <= 256 && ksteps / (splits * 2) >= 8) splits *= 2;
    return splits;
}

size_t qgemm_workspace_bytes(int M, int N, int K, int group_size, int sbt)
{
    const dma::Plan p = dma::plan(M, N, K, group_size, sbt, dma::kRegFixedLds);
    if (p.splits > 0) return p.splits > 1 ? (size_t)p.splits * M * N * sizeof(float) : 0;
    const int splits = qgemm_splits(M, N, K);
    return splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
}

// Dynamic LDS above 64 KB needs the per-function limit raised once per device and kernel (keyed by the
// kernel itself: every instantiation of a kernel template has the same pointer type).
template <typename Kern>
static hipError_t allow_lds(Kern kern, size_t bytes)
{
    static std::mutex mu;
    static std::vector<std::pair<int, const void*>> done;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const void* fn = reinterpret_cast<const void*>(kern);
    std::lock_guard<std::mutex> lk(mu);
    for (const auto& d : done)
        if (d.first == dev && d.second == fn) return hipSuccess;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)dma::kMaxLds);
    if (e == hipSuccess) done.emplace_back(dev, fn);
    (void)bytes;
    return e;
}

template <dma::RegMode MODE>
static hipError_t launch_q4_regw(const dma::RegArgs& a, int sbt, int vtiles, int splits, size_t lds, hipStream_t st)
{
    auto go = [&](auto kern) {
        const hipError_t e = allow_lds(kern, lds);
        if (e != hipSuccess) return e;
        const dim3 grid(vtiles, (a.M + BM - 1) / BM, splits);
        hipLaunchKernelGGL(kern, grid, dim3(dma::kRegThreads), lds, st, a);
        return hipGetLastError();
    };
    return sbt == DT_F16   ? go(dma::qgemm_q4_regw_kernel<DT_F16, MODE>)
           : sbt == DT_F32 ? go(dma::qgemm_q4_regw_kernel<DT_F32, MODE>)
                           : go(dma::qgemm_q4_regw_kernel<DT_BF16, MODE>);
}

// LDS of an unsplit tile, 0 if its scales and biases do not fit
static size_t fused_lds(int K, int group, int sbt)
{
    const size_t lds = dma::kRegFixedLds + (size_t)BN * ((K + group - 1) / group) * (sbt == DT_F32 ? 8 : 4);
    return lds <= dma::kMaxLds ? std::max(lds, dma::kRegExchangeBytes * 2) : 0;
}

bool qgemm_q4_fused_supported(const Q4FusedSeg* segs, int nseg, bool act, int sbt, int group, const _Float16* x, int M,
                              int K)
{
    if (M < 1 || K <= 0 || K % dma::BK != 0 || group < 32 || (reinterpret_cast<uintptr_t>(x) & 15) != 0 ||
        (uint64_t)M * K * 2 >= (1ull << 32) || !fused_lds(K, group, sbt) || (act && segs[0].n != segs[1].n))
        return false;
    int64_t tiles = 0;
    for (int i = 0; i < nseg; ++i) {
        if (segs[i].n <= 0 || (reinterpret_cast<uintptr_t>(segs[i].w) & 15) != 0 ||
            (uint64_t)segs[i].n * K / 2 >= (1ull << 32))
            return false;
        tiles += (segs[i].n + BN - 1) / BN;
    }
    tiles *= (M + BM - 1) / BM;
    // unsplit: 1.04 us per 128 k, against launches of their own with split sums where tiles are few
    return K / dma::BK <= 20 || tiles >= 128;
}

hipError_t launch_qgemm_q4_fused(const Q4FusedSeg* segs, int nseg, int act, int sbt, int group, const _Float16* x, int M,
                                 int K, hipStream_t st)
{
    dma::RegArgs a{};
    int vtiles = 0;
    for (int i = 0; i < 3; ++i) {
        a.tile0[i] = i < nseg ? vtiles : INT32_MAX;
        if (i >= nseg) continue;
        a.seg[i] = segs[i];
        vtiles += (segs[i].n + BN - 1) / BN;
    }
    if (act >= 0) vtiles = (segs[0].n + BN / 2 - 1) / (BN / 2);
    a.gshift = __builtin_ctz((unsigned)group);
    a.M = M;
    a.K = K;
    a.k_per_split = K;
    a.act = act;
    a.X = x;
    const size_t lds = fused_lds(K, group, sbt);
    return act >= 0 ? launch_q4_regw<dma::REG_ACT>(a, sbt, vtiles, 1, lds, st)
                    : launch_q4_regw<dma::REG_MANY>(a, sbt, vtiles, 1, lds, st);
}

static hipError_t launch_qgemm_common(const void* W, const void* S, const void* B, int sbt, int group_size,
                                      const _Float16* X, float* Y, int M, int N, int K, float* workspace,
                                      hipStream_t st)
{
    const int splits = workspace ? qgemm_splits(M, N, K) : 1;
    const int ksteps = (K + BK - 1) / BK;
    const int k_per_split = ((ksteps + splits - 1) / splits) * BK;
    const dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM, splits);
    float* out = splits > 1 ? workspace : Y;
#define CELLM_QGEMM(SBT_)                                                                                          \
    hipLaunchKernelGGL((qgemm_kernel<SBT_, kStages>), grid, dim3(kThreads), 0, st, W, S, B, group_size, X, out, M, N, K, \
                       k_per_split)
    if (sbt == DT_F32) CELLM_QGEMM(DT_F32);
    else if (sbt == DT_F16) CELLM_QGEMM(DT_F16);
    else CELLM_QGEMM(DT_BF16);
#undef CELLM_QGEMM
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const size_t total = (size_t)M * N;
    unsigned blocks = (unsigned)((total + 255) / 256);
    if (blocks > 4096) blocks = 4096;
    if (splits > 1) {
        hipLaunchKernelGGL(splitk_reduce_kernel, dim3(blocks), dim3(256), 0, st, workspace, Y, splits, M, N);
        e = hipGetLastError();
    }
    return e;
}

hipError_t launch_qgemm_q4_affine_ws(const uint32_t* wq, const void* S, const void* B, int sbt, int group_size,
                                     const _Float16* x, float* y, int M, int N, int K, float* workspace,
                                     hipStream_t st)
{
    dma::Plan p = dma::plan(M, N, K, group_size, sbt, dma::kRegFixedLds);
    p.lds = std::max(p.lds, dma::kRegExchangeBytes);
    const bool offsets_fit = (uint64_t)M * K * 2 < (1ull << 32) && (uint64_t)N * K / 2 < (1ull << 32);
    if (p.splits > 0 && (p.splits == 1 || workspace) && offsets_fit) {
        dma::RegArgs a{};
        a.seg[0] = Q4FusedSeg{wq, S, B, nullptr, y, N};
        a.tile0[1] = a.tile0[2] = INT32_MAX;
        a.gshift = __builtin_ctz((unsigned)group_size);
        a.M = M;
        a.K = K;
        a.k_per_split = p.k_per_split;
        a.X = x;
        a.part = p.splits > 1 ? workspace : nullptr;
        const hipError_t e = launch_q4_regw<dma::REG_ONE>(a, sbt, (N + BN - 1) / BN, p.splits, p.lds, st);
        if (e != hipSuccess || p.splits == 1) return e;
        const size_t total = (size_t)M * N;
        unsigned blocks = (unsigned)((total + 255) / 256);
        if (blocks > 4096) blocks = 4096;
        hipLaunchKernelGGL(splitk_reduce_kernel, dim3(blocks), dim3(256), 0, st, workspace, y, p.splits, M, N);
        return hipGetLastError();
    }
    return launch_qgemm_common(wq, S, B, sbt, group_size, x, y, M, N, K, workspace, st);
}

}  // namespace cellm
