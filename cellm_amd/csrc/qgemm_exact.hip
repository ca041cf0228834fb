// Multi-row GEMM on f16 MFMA whose weights are exact in f16 (gfx950):
//
//   Y[m,n] = (sum_k w[n,k] x[m,k]) * scale[n] (+ bias[n]),   w (or q - 8) exact in f16
//
// for M >= 5 rows of f32 activations over int8, symmetric 4-bit and f16 weights
// (cpu_kernels::matmul_i8_f32, matmul_i4_f32, matmul_f16_f32,
// crates/cellm-kernels/src/cpu_kernels.rs:66-243, run once per prompt token by the
// reference, crates/cellm-model/src/llama.rs:214-233) and MLX 4-bit affine ones
// (crates/cellm-model/src/lfm.rs:985-1066).
//
// Group-scaled nibbles (w = q s + b or (q - 8) s, one scale per 64 k or a multiple)
// multiply as the exact q - 8: every K step's sum is folded as
// s acc + (b + 8 s) sum(x'), the sums of x' coming from the split kernel and
// the step's scales and biases with the weights through the DMA ring.  With q - 8
// in place of q the step's two terms do not cancel (b is near -7.5 s).
//
// f32 activations are two f16 parts, 23 bits of the 24: a first kernel scales each
// row by the power of two that puts its largest |x| in [2^13, 2^14) and splits it
// into hi = RNE_f16(x') and lo = RNE_f16(x' - hi); x' - hi - lo is at most 2^-23 |x'|,
// and elements below 2^-15 of the row's largest are held to 2^-38 of that.  Both
// parts are rows of the GEMM's A operand over one weight tile, so every weight is
// fetched and unpacked once for the two.  Products of f16 values are exact in f32.
// The MFMA chain rounds its f32 accumulator once per 8 or 16 products, so a chain
// over the whole K carries more rounding error than the tree sums of the
// one-wave-per-row kernels: accumulators run over one K step (64 k), low parts
// before high ones, the sums of two steps are added and then join the total.  Error
// against 64 bits, int8 at 512 rows, K = 960 / 2560 / 4096 / 8192: 8.4e-8 / 1.0e-7 /
// 1.1e-7 / 1.2e-7 (each step added to the total by itself 8.6e-8 / 1.0e-7 / 1.3e-7 /
// 1.3e-7, chains over two steps 9.7e-8 / 1.1e-7 / 1.2e-7, over four 1.3e-7 / 1.4e-7 /
// 1.4e-7, the one-wave-per-row kernels 9.7e-8 / 1.3e-7 / 1.7e-7 / 2.1e-7); against
// chains over four steps this costs 4-5 % of the wide shapes' time.  At few K the
// split of x and the MFMA's own rounding show: 300 rows, K = 256 / 576 / 896 / 1024,
// this and the row kernels, f16 weights 9.5e-8 and 6.8e-8 / 9.8e-8 and 8.6e-8 /
// 9.7e-8 and 9.1e-8 / 9.9e-8 and 9.4e-8, int8 9.1e-8 and 8.2e-8 / 9.3e-8 and 9.0e-8 /
// 9.1e-8 and 9.1e-8 / 9.3e-8 and 9.6e-8; i4 and q4 are below the row kernels there
// already.  Shorter chains, added as a tree, change nothing.
// Results that are not finite (an infinity or NaN in x or w, or an overflow) are
// recomputed by plain f32 sums where these may differ (kPlain).
//
// Measured, int8 at 512 rows (us, one-wave-per-row kernel -> this one with its
// split of x): 960 -> 960 1963 -> 20, 2560 -> 960 5098 -> 25, 4096 -> 4096
// 8034 -> 60; 16 rows of 1152 -> 1536 35 -> 15; 2048 rows of 2048 -> 8192 164,
// 839 TFLOP/s of MFMA work; 16 rows of 2560 -> 960, i4 109 -> 14, f16 63 -> 14; MLX
// q4 with f32 scales, 512 rows of 4096 -> 4096, 1480 -> 67 (error 1.6e-7 -> 1.1e-7).  The
// small ones are bound by three dependent launches and the latency of a few K steps,
// the wide ones by the MFMAs.
//
// Tile: WM x WN waves of (32 TA) x (32 TB); X parts and raw weights go
// global -> LDS by DMA through a ring of NST stages of 64 k, one barrier per
// step.  Weights stay raw in LDS and are unpacked right before their MFMAs by
// the lane that multiplies them.  A lane (r32 = lane % 32, h32 = lane / 32)
// supplies k = 32 h32 + 8 ks + 0..7 of the step to substep ks = 0..3: the MFMA's
// k order is free as long as X and W agree, and this one makes a lane's weights
// of a step contiguous.  LDS rows are XOR-swizzled in 16-byte chunks so that the
// eight rows of a read phase fall in different banks.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"
#include "launch_util.hpp"
#include "lds_dma.hpp"

namespace cellm {

namespace {

using namespace ldsdma;

constexpr int kBK = 64;

struct XgArgs {
    XgSeg seg[3];
    int tile0[3];  // first column tile of each segment; of an absent one, past every tile
    const _Float16* xp;   // [M][P][Kp] activation parts
    const int32_t* xe;    // [M] row exponents e (x' = x 2^e); P == 2
    const void* x;        // the caller's activations [M][K], for the recomputed sums
    const float* xsum;    // XG_Q4: sum of x' over the 64 k of each step, [steps][M]
    float* part;          // [splits][M][vcols] raw sums, or nullptr (unsplit)
    int M, K, Kp;
    int steps_per_split;
    int vcols;            // column tiles * BN
    int sdt;
    int group, gpr;       // XG_Q4: elements per scale, scales per row
    int act;              // ACT: h = act(seg 0) * seg 1, written to seg 0's y
};

// The segment of column tile vt and its first tile: selects between arguments that are all loaded at once, not
// a chain of loads through an index
__device__ __forceinline__ XgSeg segment_of(const XgArgs& a, int vt, int& tile0)
{
    const XgSeg s0 = a.seg[0], s1 = a.seg[1], s2 = a.seg[2];
    const int t1 = a.tile0[1], t2 = a.tile0[2];
    const bool c1 = vt >= t1, c2 = vt >= t2;
    const auto pick = [&](auto x0, auto x1, auto x2) { return c2 ? x2 : c1 ? x1 : x0; };
    tile0 = pick(0, t1, t2);
    return XgSeg{pick(s0.w, s1.w, s2.w), pick(s0.s, s1.s, s2.s), pick(s0.bias, s1.bias, s2.bias), pick(s0.y, s1.y, s2.y),
                 pick(s0.n, s1.n, s2.n), pick(s0.s_stride, s1.s_stride, s2.s_stride), pick(s0.gs, s1.gs, s2.gs),
                 pick(s0.gb, s1.gb, s2.gb)};
}

template <int FMT>
struct Fmt;
template <>
struct Fmt<XG_I8> {
    static constexpr int kStepBytes = 64;  // of a weight row per K step
    static constexpr bool kPairs = false;  // x in k order
};
template <>
struct Fmt<XG_I4> {
    static constexpr int kStepBytes = 32;
    static constexpr bool kPairs = true;  // each 8 x as 0,4,1,5,2,6,3,7: the order nib8 unpacks a word in
};
template <>
struct Fmt<XG_Q4> : Fmt<XG_I4> {};
template <>
struct Fmt<XG_F16> {
    static constexpr int kStepBytes = 128;
    static constexpr bool kPairs = false;
};

constexpr int stage_bytes(int fmt, int P, int bm, int bn, int step_bytes)
{
    return bm * P * 128 + bn * step_bytes + (fmt == XG_Q4 ? 8 * bn + 4 * (bm > 64 ? bm : 64) : 0);
}

template <int FMT>
__device__ __forceinline__ size_t row_bytes(int K)
{
    return (size_t)K * Fmt<FMT>::kStepBytes / kBK;
}

// eight consecutive int8 weights as f16, in order: bytes biased to u8 land under 0x64 (1024 + u8), minus 1152
__device__ __forceinline__ h8_t i8x8(uint32_t w0, uint32_t w1)
{
    const uint32_t b0 = w0 ^ 0x80808080u, b1 = w1 ^ 0x80808080u, hi = 0x64646464u;
    const h2_t off = {(_Float16)1152.0f, (_Float16)1152.0f};
    const h2_t a0 = as_h2(__builtin_amdgcn_perm(hi, b0, 0x04010400u)) - off;
    const h2_t a1 = as_h2(__builtin_amdgcn_perm(hi, b0, 0x04030402u)) - off;
    const h2_t a2 = as_h2(__builtin_amdgcn_perm(hi, b1, 0x04010400u)) - off;
    const h2_t a3 = as_h2(__builtin_amdgcn_perm(hi, b1, 0x04030402u)) - off;
    return h8_t{a0[0], a0[1], a1[0], a1[1], a2[0], a2[1], a3[0], a3[1]};
}

// the eight nibbles of a word minus 8 as f16, in the order 0,4,1,5,2,6,3,7: the low nibble of a byte
// lands as 1024 + q, the high one as 1024 + 16 q, which one fma takes to q - 8
__device__ __forceinline__ h8_t nib8(uint32_t w)
{
    const uint32_t mlo = 0x000F000Fu, mhi = 0x00F000F0u, magic = 0x64006400u;
    const h2_t off = {(_Float16)1032.0f, (_Float16)1032.0f}, off16 = {(_Float16)-72.0f, (_Float16)-72.0f},
               inv = {(_Float16)0.0625f, (_Float16)0.0625f};
    const uint32_t v = w >> 8;
    const h2_t a0 = as_h2(and_or(w, mlo, magic)) - off;
    const h2_t a1 = __builtin_elementwise_fma(as_h2(and_or(w, mhi, magic)), inv, off16);
    const h2_t a2 = as_h2(and_or(v, mlo, magic)) - off;
    const h2_t a3 = __builtin_elementwise_fma(as_h2(and_or(v, mhi, magic)), inv, off16);
    return h8_t{a0[0], a0[1], a1[0], a1[1], a2[0], a2[1], a3[0], a3[1]};
}

// LDS position of 16-byte chunk c of row r: rows of RB bytes, the eight rows of a read phase in
// different banks
template <int RB>
__device__ __forceinline__ int swz(int r, int c)
{
    if constexpr (RB == 128) return c ^ (r & 7);
    else if constexpr (RB == 64) return c ^ ((r >> 2) & 3);
    else return c;
}

__device__ __forceinline__ float scale_at(const void* s, int sdt, size_t i)
{
    return sdt == DT_F32 ? load_f32<DT_F32>(s, i) : sdt == DT_F16 ? load_f32<DT_F16>(s, i) : load_f32<DT_BF16>(s, i);
}

// Results that MFMA leaves non-finite may be finite or another infinity in a plain sum where the weights' side can
// be infinite (f16 weights, group scales): inf * lo, or s inf - 8 s inf.  int8 and i4 under row scales are what a plain
// sum gives: exact finite weights, lo = 0 beside an infinite hi, one product each.
template <int FMT>
constexpr bool kPlain = FMT == XG_F16 || FMT == XG_Q4;

// sum_k w[n,k] x[m,k] by plain f32 sums, eight chains: the results that MFMA left non-finite.  Where every output of
// 512 x 2048 x 2048 was one, a loop of single elements took 5.9 ms (f16 weights) and 19 (q4), this 0.72 and 1.3 (the
// one-wave-per-row kernels 1.6 and 0.76 at any input); one infinite weight 0.076 and 0.19 ms for 0.23 and 0.66.
template <int FMT, int P, int UNROLL>
__device__ __forceinline__ float plain_dot(const XgArgs& a, const XgSeg& g, int m, int n)
{
#pragma clang fp contract(off)
    const int K = a.K;
    float acc[8] = {};
    for (int k0 = 0; k0 < K; k0 += kBK) {
        float s = 1.0f, b = 0.0f;
        if constexpr (FMT == XG_Q4) {
            const size_t i = (size_t)n * a.gpr + k0 / a.group;
            s = scale_at(g.gs, a.sdt, i);
            if (g.gb) b = scale_at(g.gb, a.sdt, i);
        }
        const int end = min(k0 + kBK, K);  // K % 8 == 0
#pragma unroll UNROLL
        for (int k = k0; k < end; k += 8) {
            float x[8], w[8];
            if constexpr (P == 2) {
                const f4_t* p = reinterpret_cast<const f4_t*>(static_cast<const float*>(a.x) + (size_t)m * K + k);
                const f4_t x0 = p[0], x1 = p[1];
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = i < 4 ? x0[i & 3] : x1[i & 3];
            } else {
                const h8_t h = *reinterpret_cast<const h8_t*>(static_cast<const _Float16*>(a.x) + (size_t)m * K + k);
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = (float)h[i];
            }
            if constexpr (FMT == XG_F16) {
                const h8_t h = *reinterpret_cast<const h8_t*>(static_cast<const _Float16*>(g.w) + (size_t)n * K + k);
#pragma unroll
                for (int i = 0; i < 8; ++i) w[i] = (float)h[i];
            } else {
                const uint32_t q = static_cast<const uint32_t*>(g.w)[((size_t)n * K + k) / 8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float v = (float)(q >> (4 * i) & 15u);
                    w[i] = g.gb ? v * s + b : (v - 8.0f) * s;
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] = acc[i] + w[i] * x[i];
        }
    }
    return ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
}

__device__ __forceinline__ bool finite_f32(float v) { return (__builtin_bit_cast(uint32_t, v) & 0x7F800000u) != 0x7F800000u; }

__device__ __forceinline__ float column_scale(const XgSeg& g, int sdt, int n)
{
    return g.s ? scale_at(g.s, sdt, (size_t)n * g.s_stride) : 1.0f;
}

template <int FMT, int P, bool ACT, int UNROLL>
__device__ __forceinline__ float plain_output(const XgArgs& a, const XgSeg& g, const XgSeg& gu, int m, int n)
{
    const float v = plain_dot<FMT, P, UNROLL>(a, g, m, n) * column_scale(g, a.sdt, n) + (g.bias ? g.bias[n] : 0.0f);
    if constexpr (!ACT) return v;
    return act_mul(a.act, v, plain_dot<FMT, P, UNROLL>(a, gu, m, n) * column_scale(gu, a.sdt, n) + (gu.bias ? gu.bias[n] : 0.0f));
}

// S16: XG_Q4's scales are 16 bits wide.  FOLD: the sums of two K steps (int8 over f16 rows: four) meet before they
// join the total, else one chain over K.  ACT: segments 0 and 1 are gate and up; each wave's 64 columns are 32
// gate columns and the same 32 up columns, so both sums of an output end in one lane.
template <int FMT, bool S16, int P, bool FOLD, int TA, int TB, int WM, int WN, int NST, bool ACT>
__global__ __launch_bounds__(64 * WM * WN, 2) void qgemm_exact_kernel(const XgArgs a)
{
    constexpr int NW = WM * WN, BM = 32 * TA * WM, BN = 32 * TB * WN, RB = Fmt<FMT>::kStepBytes;
    constexpr bool GROUPED = FMT == XG_Q4;
    static_assert(FOLD || !GROUPED, "group scales are folded per step");
    static_assert(!ACT || TB == 2, "a gate and an up tile per wave");
    // a stage: X parts, raw weights, and the step's group scales, group biases and sums of x'
    constexpr int kXBytes = BM * P * 128, kWBytes = BN * RB, kGroupAt = kXBytes + kWBytes, kSumAt = kGroupAt + 8 * BN;
    constexpr int kStage = stage_bytes(FMT, P, BM, BN, RB);
    constexpr int XD = kXBytes / 1024 / NW, WD = kWBytes / 1024 / NW;  // DMA loads per wave and step
    constexpr int GD = GROUPED ? 2 * BN / 64 / NW : 0;                 // of 64 scales or biases
    constexpr int NDMA = XD + WD + GD + (GROUPED ? 1 : 0), LA = NST - 1;
    static_assert(!GROUPED || GD * NW * 64 == 2 * BN, "whole DMA loads per wave");
    static_assert(XD * NW * 1024 == kXBytes && WD * NW * 1024 == kWBytes, "whole DMA loads per wave");
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN, r32 = lane & 31, h32 = lane >> 5;
    const int vt = blockIdx.x, m0 = blockIdx.y * BM;
    const int step0 = blockIdx.z * a.steps_per_split, total = a.Kp / kBK;
    const int nsteps = min(a.steps_per_split, total - step0);
    if (nsteps <= 0) return;  // the launcher makes no empty split
    int tile0 = 0;
    const XgSeg gu = a.seg[1], g = ACT ? a.seg[0] : segment_of(a, vt, tile0);
    const int n0 = (vt - tile0) * (ACT ? BN / 2 : BN);
    const size_t rbytes = row_bytes<FMT>(a.K);

    // X DMA: load j of a wave covers 8 part rows (128 bytes each); part row p BM + i is part p of row
    // m0 + i, rows past M re-read the last one (computed, never stored)
    uint32_t xoff[XD];
#pragma unroll
    for (int j = 0; j < XD; ++j) {
        const int pr = (wave * XD + j) * 8 + (lane >> 3);
        const int p = pr / BM, i = min(pr % BM, a.M - 1 - m0);
        xoff[j] = (uint32_t)(i * P + p) * (uint32_t)(a.Kp * 2) + 16 * ((lane & 7) ^ (pr & 7));
    }
    // W DMA: load j covers 1024 / RB rows.  In the last step of a K that is no multiple of 64, chunks
    // past the row's end re-read its last one (they meet the zeros that pad X)
    constexpr int RPD = 1024 / RB, CPR = RB / 16;
    uint32_t woff[WD], woff_tail[WD];
    const unsigned char* wbase[WD];
    const int tail_chunks = (int)(rbytes - (size_t)(total - 1) * RB) / 16;
#pragma unroll
    for (int j = 0; j < WD; ++j) {
        const int r = (wave * WD + j) * RPD + lane / CPR;
        const int c = swz<RB>(r, lane % CPR);
        // a load's rows lie in one 32-row slice: for ACT, slices alternate between gate and up
        const int slice = (wave * WD + j) * RPD / 32, col = ACT ? (slice >> 1) * 32 + (r & 31) : r;
        wbase[j] = static_cast<const unsigned char*>(ACT && (slice & 1) ? gu.w : g.w) + (size_t)n0 * rbytes;
        const uint32_t row = (uint32_t)min(col, g.n - 1 - n0) * (uint32_t)rbytes;
        woff[j] = row + 16 * c;
        woff_tail[j] = row + 16 * min(c, tail_chunks - 1);
    }
    const unsigned char* xbase = reinterpret_cast<const unsigned char*>(a.xp) + (size_t)m0 * P * a.Kp * 2;
    // scale and bias DMA: load j of a wave covers 64 columns of either (symmetric weights fetch their scales
    // twice); x' sums: 64 rows per load, waves past the tile's rows repeat one
    uint32_t goff[GROUPED ? GD : 1], soff = 0;
    const unsigned char* gbase[GROUPED ? GD : 1];
    constexpr int SB = S16 ? 2 : 4;
    const int sum_at = (wave % (BM > 64 ? BM / 64 : 1)) * 64;
    if constexpr (GROUPED) {
#pragma unroll
        for (int j = 0; j < GD; ++j) {
            // ACT: the gate columns' scales, then the up columns', the same for the biases
            constexpr int PER = ACT ? BN / 128 : BN / 64;
            const int q = wave * GD + j, c = (q % PER) * 64 + lane;
            const XgSeg& h = ACT && (q / PER & 1) ? gu : g;
            goff[j] = (uint32_t)min(c, g.n - 1 - n0) * (uint32_t)(a.gpr * SB);
            gbase[j] = static_cast<const unsigned char*>(q < BN / 64 || !h.gb ? h.gs : h.gb) + (size_t)n0 * a.gpr * SB;
        }
        soff = (uint32_t)min(sum_at + lane, a.M - 1 - m0) * 4u;
    }
    const uint32_t lds0 = lds_addr(smem);
    const bool ragged = tail_chunks < CPR;
    auto issue = [&](int s, int slot) {
        const int t = step0 + min(s, nsteps - 1);
        const uint32_t base = lds0 + slot * kStage;
        const unsigned char* xs = xbase + (size_t)t * 128;
        const size_t wt = (size_t)t * RB;
#pragma unroll
        for (int j = 0; j < XD; ++j) dma16_s(xoff[j], xs, base + (wave * XD + j) * 1024);
        if (ragged && t == total - 1) {
#pragma unroll
            for (int j = 0; j < WD; ++j) dma16_s(woff_tail[j], wbase[j] + wt, base + kXBytes + (wave * WD + j) * 1024);
        } else {
#pragma unroll
            for (int j = 0; j < WD; ++j) dma16_s(woff[j], wbase[j] + wt, base + kXBytes + (wave * WD + j) * 1024);
        }
        if constexpr (GROUPED) {
            const size_t gi = (size_t)(t * kBK / a.group) * SB;
#pragma unroll
            for (int j = 0; j < GD; ++j) {
                const uint32_t to = base + kGroupAt + (wave * GD + j) * 256;
                if constexpr (S16) dma2_s(goff[j], gbase[j] + gi, to);
                else dma4_s(goff[j], gbase[j] + gi, to);
            }
            dma4_s(soff, a.xsum + (size_t)t * a.M + m0, base + kSumAt + sum_at * 4);
        }
    };
#pragma unroll
    for (int j = 0; j < LA; ++j) issue(j, j);

    f16v_t sum[TA][TB];
#pragma unroll
    for (int i = 0; i < TA; ++i)
#pragma unroll
        for (int j = 0; j < TB; ++j) sum[i][j] = f16v_t{};

    int slot = 0;
    // K step s into acc: onto it, or (grouped) the step's scaled sum added to pair
    auto step = [&](int s, f16v_t(&acc)[TA][TB], f16v_t(&pair)[TA][TB]) {
        // stage s landed in this wave's share of the slot; only the LA - 1 stages after it may be in
        // flight.  A bare s_barrier: __syncthreads()'s release fence waits for every DMA in flight.
        wait_vmcnt<(LA - 1) * NDMA>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();  // stage s complete everywhere; stage s - 1 no longer read
        issue(s + LA, slot == 0 ? NST - 1 : slot - 1);  // into the slot of stage s - 1
        const unsigned char* xs = smem + slot * kStage;
        const unsigned char* ws = xs + kXBytes;
        slot = slot + 1 == NST ? 0 : slot + 1;
        h8_t b[TB][4];
#pragma unroll
        for (int j = 0; j < TB; ++j) {
            const int r = (wn * TB + j) * 32 + r32;
            if constexpr (FMT == XG_I8) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const u4_t w = *reinterpret_cast<const u4_t*>(ws + r * RB + 16 * swz<RB>(r, 2 * h32 + c));
                    b[j][2 * c] = i8x8(w[0], w[1]);
                    b[j][2 * c + 1] = i8x8(w[2], w[3]);
                }
            } else if constexpr (FMT == XG_F16) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    b[j][c] = *reinterpret_cast<const h8_t*>(ws + r * RB + 16 * swz<RB>(r, 4 * h32 + c));
            } else {
                const u4_t w = *reinterpret_cast<const u4_t*>(ws + r * RB + 16 * h32);
#pragma unroll
                for (int c = 0; c < 4; ++c) b[j][c] = nib8(w[c]);
            }
        }
#pragma unroll
        for (int p = P - 1; p >= 0; --p)  // low parts first
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                h8_t x[TA];
#pragma unroll
                for (int i = 0; i < TA; ++i) {
                    const int r = p * BM + (wm * TA + i) * 32 + r32;
                    x[i] = *reinterpret_cast<const h8_t*>(xs + r * 128 + 16 * swz<128>(r, 4 * h32 + ks));
                }
#pragma unroll
                for (int i = 0; i < TA; ++i)
#pragma unroll
                    for (int j = 0; j < TB; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[i], b[j][ks], acc[i][j], 0, 0, 0);
            }
        if constexpr (GROUPED) {
            // w = q s + b = (q - 8) s + (b + 8 s): the step's sum of (q - 8) x' times s, plus (b + 8 s) times
            // its sum of x'
            const uint32_t* gs = reinterpret_cast<const uint32_t*>(xs + kGroupAt);
            const f4_t* sums = reinterpret_cast<const f4_t*>(xs + kSumAt);
            float sc[TB], bi[TB];
#pragma unroll
            for (int j = 0; j < TB; ++j) {
                const int c = ACT ? j * (BN / 2) + wn * 32 + r32 : (wn * TB + j) * 32 + r32;
                const uint32_t s = gs[c], b = gs[BN + c];
                if constexpr (S16) {
                    sc[j] = a.sdt == DT_F16 ? raw_to_f32<DT_F16>(s) : raw_to_f32<DT_BF16>(s);
                    bi[j] = a.sdt == DT_F16 ? raw_to_f32<DT_F16>(b) : raw_to_f32<DT_BF16>(b);
                } else {
                    sc[j] = raw_to_f32<DT_F32>(s);
                    bi[j] = raw_to_f32<DT_F32>(b);
                }
                bi[j] = g.gb ? __builtin_fmaf(8.0f, sc[j], bi[j]) : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < TA; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f4_t xv = sums[(wm * TA + i) * 8 + q * 2 + h32];
#pragma unroll
                    for (int j = 0; j < TB; ++j)
#pragma unroll
                        for (int c = 0; c < 4; ++c)
                            pair[i][j][4 * q + c] = __builtin_fmaf(
                                sc[j], acc[i][j][4 * q + c], __builtin_fmaf(bi[j], xv[c], pair[i][j][4 * q + c]));
                }
        }
    };
    if constexpr (FOLD) {
        if constexpr (P == 1 && !GROUPED) {
            for (int s = 0; s < nsteps; s += 4) {
                f16v_t few[TA][TB] = {};
                step(s, few, few);
#pragma unroll
                for (int u = 1; u < 4; ++u) {
                    if (s + u >= nsteps) break;
                    f16v_t a0[TA][TB] = {};
                    step(s + u, a0, a0);
#pragma unroll
                    for (int i = 0; i < TA; ++i)
#pragma unroll
                        for (int j = 0; j < TB; ++j) few[i][j] += a0[i][j];
                }
#pragma unroll
                for (int i = 0; i < TA; ++i)
#pragma unroll
                    for (int j = 0; j < TB; ++j) sum[i][j] += few[i][j];
            }
        } else
        for (int s = 0; s < nsteps; s += 2) {
            f16v_t a0[TA][TB] = {}, a1[TA][TB] = {};
            if constexpr (GROUPED) {
                step(s, a0, a1);
                if (s + 1 < nsteps) {
                    f16v_t a2[TA][TB] = {};
                    step(s + 1, a2, a1);
                }
            } else {
                step(s, a0, a0);
                if (s + 1 < nsteps) step(s + 1, a1, a1);
            }
#pragma unroll
            for (int i = 0; i < TA; ++i)
#pragma unroll
                for (int j = 0; j < TB; ++j) {
                    if constexpr (GROUPED) sum[i][j] += a1[i][j];
                    else sum[i][j] += a0[i][j] + a1[i][j];
                }
        }
    } else {
        for (int s = 0; s < nsteps; ++s) step(s, sum, sum);
    }
    wait_vmcnt<0>();  // the trailing (re-read) DMA, before the block's LDS is given back

    // register r of a 32x32 tile: row (r / 4) * 8 + h32 * 4 + r % 4, column r32
    if (a.part) {
#pragma unroll
        for (int i = 0; i < TA; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + (wm * TA + i) * 32 + (r >> 2) * 8 + h32 * 4 + (r & 3);
                float* row = a.part + ((size_t)blockIdx.z * a.M + m) * a.vcols + (size_t)vt * BN + wn * TB * 32 + r32;
                if (m < a.M)
#pragma unroll
                    for (int j = 0; j < TB; ++j) row[j * 32] = sum[i][j][r];
            }
        return;
    }
    int e[TA][16];
    if constexpr (P == 2) {
#pragma unroll
        for (int i = 0; i < TA; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                e[i][r] = -a.xe[min(m0 + (wm * TA + i) * 32 + (r >> 2) * 8 + h32 * 4 + (r & 3), a.M - 1)];
    }
    // output tile j of the wave: columns at n; with ACT the gate tile's columns hold the outputs
    constexpr int TO = ACT ? 1 : TB;
    const auto out_col = [&](int j) { return n0 + (ACT ? wn : wn * TB + j) * 32 + r32; };
    const auto value = [](float v, int ev, float sc, float bi) { return (P == 2 ? ldexpf(v, ev) : v) * sc + bi; };
    // every load of the epilogue before its first store: one still pending there makes each guarded store wait for
    // the one before it (int8 over f16 rows, 2048 x 12288 x 4096: 237 -> 223 us)
    float sc[TO], bi[TO], sc1 = 1.0f, bi1 = 0.0f;
#pragma unroll
    for (int j = 0; j < TO; ++j) {
        const int n = min(out_col(j), g.n - 1);
        sc[j] = column_scale(g, a.sdt, n);
        bi[j] = g.bias ? g.bias[n] : 0.0f;
        if constexpr (ACT) {
            sc1 = column_scale(gu, a.sdt, n);
            bi1 = gu.bias ? gu.bias[n] : 0.0f;
        }
    }
#pragma unroll
    for (int j = 0; j < TO; ++j) asm volatile("" : "+v"(sc[j]), "+v"(bi[j]));
    asm volatile("" : "+v"(sc1), "+v"(bi1));
    if constexpr (P == 2) {
#pragma unroll
        for (int i = 0; i < TA; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(e[i][r]));
    }
    bool bad = false;
    const auto store = [&](auto act) {
#pragma unroll
        for (int j = 0; j < TO; ++j) {
            const int n = out_col(j);
            if (n >= g.n) continue;
#pragma unroll
            for (int i = 0; i < TA; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + (wm * TA + i) * 32 + (r >> 2) * 8 + h32 * 4 + (r & 3);
                    const int ev = P == 2 ? e[i][r] : 0;
                    float v = value(sum[i][j][r], ev, sc[j], bi[j]);
                    if constexpr (ACT)
                        v = act_mul(decltype(act)::value, v, value(sum[i][TB - 1][r], ev, sc1, bi1));
                    if (m < a.M) {
                        g.y[(size_t)m * g.n + n] = v;
                        if constexpr (kPlain<FMT>) bad |= !finite_f32(v);
                    }
                }
        }
    };
    if (ACT && a.act == ACT_GELU_TANH)  // outside the loops: no branch between neighbouring values
        store(std::integral_constant<int, ACT_GELU_TANH>{});
    else
        store(std::integral_constant<int, ACT_SILU>{});
    if constexpr (kPlain<FMT>) {
        if (!bad) return;
        // rolled and rare: this lane's non-finite results again (a non-finite gate or up sum makes h non-finite)
        for (int t = 0; t < TA * TO * 16; ++t) {
            const int i = t / (16 * TO), j = (t / 16) % TO, r = t & 15;
            const int m = m0 + (wm * TA + i) * 32 + (r >> 2) * 8 + h32 * 4 + (r & 3), n = out_col(j);
            if (m >= a.M || n >= g.n || finite_f32(g.y[(size_t)m * g.n + n])) continue;
            g.y[(size_t)m * g.n + n] = plain_output<FMT, P, ACT, 4>(a, g, gu, m, n);
        }
    }
}

// y of a split GEMM: the splits' sums added in split order, then the epilogue above.  A thread owns four
// neighbouring outputs of one row.
template <int FMT, int P, bool ACT>
__global__ __launch_bounds__(256) void qgemm_exact_reduce_kernel(const XgArgs a, int splits, int bn)
{
    const int quads = a.vcols / (ACT ? 8 : 4);
    const size_t stride = (size_t)a.M * (a.vcols / 4);
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < (size_t)a.M * quads; t += (size_t)gridDim.x * 256) {
        const int m = (int)(t / quads), c0 = (int)(t - (size_t)m * quads) * 4;
        int tile0 = 0;
        const XgSeg gu = a.seg[1], g = ACT ? a.seg[0] : segment_of(a, c0 / bn, tile0);
        const int n = c0 - tile0 * bn, vc = ACT ? c0 / 32 * 64 + c0 % 32 : c0;  // ACT: 32 gate, then their 32 up columns
        if (n >= g.n) continue;
        const f4_t* part = reinterpret_cast<const f4_t*>(a.part + (size_t)m * a.vcols + vc);
        const f4_t v = sum_splits_f4(part, stride, splits);
        f4_t u{};
        if constexpr (ACT) u = sum_splits_f4(part + 8, stride, splits);
        const int e = P == 2 ? -a.xe[m] : 0;
        float* y = g.y + (size_t)m * g.n + n;
        f4_t o;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int nc = min(n + c, g.n - 1);
            o[c] = (P == 2 ? ldexpf(v[c], e) : v[c]) * column_scale(g, a.sdt, nc) + (g.bias ? g.bias[nc] : 0.0f);
            if constexpr (ACT)
                o[c] = act_mul(a.act, o[c],
                               (P == 2 ? ldexpf(u[c], e) : u[c]) * column_scale(gu, a.sdt, nc) +
                                   (gu.bias ? gu.bias[nc] : 0.0f));
        }
        if ((g.n & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0) {
            *reinterpret_cast<f4_t*>(y) = o;
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (n + c < g.n) y[c] = o[c];
        }
        if constexpr (kPlain<FMT>) {
            if (finite_f32(o[0]) && finite_f32(o[1]) && finite_f32(o[2]) && finite_f32(o[3])) continue;
#pragma unroll 1
            for (int c = 0; c < min(4, g.n - n); ++c)
                if (!finite_f32(y[c])) y[c] = plain_output<FMT, P, ACT, 1>(a, g, gu, m, n + c);  // 4: 110 registers for 72
        }
    }
}

// f16 rows zero-padded to Kp (K % 8 == 0)
__global__ __launch_bounds__(256) void pad_x_kernel(const _Float16* __restrict__ x, int K, int Kp, size_t units,
                                                    _Float16* __restrict__ xp)
{
    const int per_row = Kp / 8;
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < units; t += (size_t)gridDim.x * 256) {
        const size_t m = t / per_row;
        const int u = (int)(t - m * per_row);
        u4_t v = {0u, 0u, 0u, 0u};
        if (u * 8 < K) v = *reinterpret_cast<const u4_t*>(x + m * K + u * 8);
        reinterpret_cast<u4_t*>(xp)[t] = v;
    }
}

// One block per row of x: its parts, zero-padded to Kp, and its exponent.  Eight elements per thread
// and round; rows of up to 8192 stay in registers between the maximum and the split.
constexpr int kSplitUnits = 4;
template <bool PAIRS, bool SUMS>
__global__ __launch_bounds__(256) void split_x_kernel(const float* __restrict__ x, int K, int Kp,
                                                      _Float16* __restrict__ xp, int32_t* __restrict__ xe,
                                                      float* __restrict__ xsum)
{
    __shared__ float wmax[4];
    const int m = blockIdx.x, tid = threadIdx.x, units = Kp / 8;
    const float* row = x + (size_t)m * K;
    f4_t v[kSplitUnits][2];
    auto load = [&](int u, f4_t (&d)[2]) {
        const bool in = u * 8 < K;  // K % 8 == 0
        const f4_t* p = reinterpret_cast<const f4_t*>(row + (in ? u * 8 : 0));
        d[0] = p[0];
        d[1] = p[1];
        if (!in) d[0] = d[1] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    };
    auto largest = [](const f4_t (&d)[2], float mx) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float q = fabsf(d[i >> 2][i & 3]);
            mx = finite_f32(q) ? fmaxf(mx, q) : mx;
        }
        return mx;
    };
    const bool held = units <= kSplitUnits * 256;
    float mx = 0.0f;
    if (held) {
#pragma unroll
        for (int j = 0; j < kSplitUnits; ++j) load(min(tid + j * 256, units - 1), v[j]);
#pragma unroll
        for (int j = 0; j < kSplitUnits; ++j) mx = largest(v[j], mx);
    } else {
        for (int u = tid; u < units; u += 256) {
            load(u, v[0]);
            mx = largest(v[0], mx);
        }
    }
    mx = group_max<64>(mx);
    if ((tid & 63) == 0) wmax[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const int top = (int)(__builtin_bit_cast(uint32_t, mx) >> 23);  // biased exponent; 0: zero or subnormal
    const int e = mx > 0.0f ? 13 - (max(top, 1) - 127) : 0;
    if (tid == 0) xe[m] = e;
    _Float16* out = xp + (size_t)m * 2 * Kp;
    auto store = [&](int u, const f4_t (&d)[2]) {
        h8_t hi, lo;
        if constexpr (SUMS) {  // eight threads hold a step's 64 (Kp / 8 is a multiple of 8, so all or none are here)
            const f4_t q = d[0] + d[1];
            const float sum = oct_sum(ldexpf((q[0] + q[1]) + (q[2] + q[3]), e));
            if ((u & 7) == 0) xsum[(size_t)(u >> 3) * gridDim.x + m] = sum;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = PAIRS ? (i >> 1) + 4 * (i & 1) : i;
            const float s = ldexpf(d[k >> 2][k & 3], e);
            hi[i] = (_Float16)s;
            lo[i] = finite_f32(s) ? (_Float16)(s - (float)hi[i]) : (_Float16)0.0f;
        }
        *reinterpret_cast<h8_t*>(out + u * 8) = hi;
        *reinterpret_cast<h8_t*>(out + Kp + u * 8) = lo;
    };
    if (held) {
#pragma unroll
        for (int j = 0; j < kSplitUnits; ++j)
            if (tid + j * 256 < units) store(tid + j * 256, v[j]);
    } else {
        for (int u = tid; u < units; u += 256) {
            load(u, v[0]);
            store(u, v[0]);
        }
    }
}

// f16 rows in the nibbles' order, zero-padded to Kp, with each step's sum (K % 8 == 0): a thread per eight
// elements, eight threads per step
__global__ __launch_bounds__(256) void pair_x_kernel(const _Float16* __restrict__ x, int M, int K, int Kp,
                                                     _Float16* __restrict__ xp, float* __restrict__ xsum)
{
    const int per_row = Kp / 8;
    const size_t units = (size_t)M * per_row;  // a multiple of 8: a step's threads are all here or none
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < units; t += (size_t)gridDim.x * 256) {
        const int m = (int)(t / per_row), u = (int)(t - (size_t)m * per_row);
        h8_t v = {};
        if (u * 8 < K) v = *reinterpret_cast<const h8_t*>(x + (size_t)m * K + u * 8);
        const float s = oct_sum((((float)v[0] + (float)v[1]) + ((float)v[2] + (float)v[3])) +
                                (((float)v[4] + (float)v[5]) + ((float)v[6] + (float)v[7])));
        if ((u & 7) == 0) xsum[(size_t)(u >> 3) * M + m] = s;
        reinterpret_cast<h8_t*>(xp)[t] = h8_t{v[0], v[4], v[1], v[5], v[2], v[6], v[3], v[7]};
    }
}

// The tile forms, rows x columns: f32 x 32 x 128 (2 waves), 64 x 128 (4 waves), 128 x 256 (8 waves); f16 x
// 32 x 128, 128 x 128, 256 x 256 (with second accumulators for the sums of steps, 128 x 256).
struct XgPlan {
    int form, bm, bn, vtiles, steps_per_split, splits;
    size_t xp_off, sum_off, part_off, bytes;  // workspace: exponents, parts, sums of x', split sums
};

// f16 rows over int8 in place run one chain over K, as in the tile kernel that took them before (error at 4096 k,
// 2048 rows, 4.2e-7 in both).  k % 64 != 0 came from the one-wave-per-row kernel's tree sums (976 / 2032 / 4080 /
// 8176 k: 8.3e-8 / 9.3e-8 / 1.1e-7 / 1.5e-7), which sums of four steps keep (8.4e-8 / 9.4e-8 / 1.1e-7 / 1.3e-7) and a
// chain does not (2.1e-7 / 2.9e-7 / 4.1e-7 / 5.7e-7); four steps need tiles of half the rows (2048 rows of 8176 ->
// 8192 260 us chained, 344 so; single rows take tens of ms).  q4 over f16 rows: a step at a time onto the total 1.2e-7
// / 1.4e-7 / 2.0e-7 / 2.9e-7 at 992 / 2016 / 4064 / 8160 k, in pairs 7.7e-8 / 8.7e-8 / 1.1e-7 / 1.6e-7 (single rows
// 9.7e-8 / 1.2e-7 / 1.6e-7 / 2.1e-7), 3 to 5 % slower.
bool xg_chained(int fmt, int P, int K) { return P == 1 && fmt == XG_I8 && K % kBK == 0; }

XgPlan xg_plan(int fmt, int P, const XgSeg* segs, int nseg, bool act, int M, int K)
{
    XgPlan p{};
    const int steps = (K + kBK - 1) / kBK;
    const bool chained = xg_chained(fmt, P, K);
    auto tiles = [&](int bm, int bn) {
        int t = 0;
        if (act) t = (segs[0].n + bn / 2 - 1) / (bn / 2);
        else
            for (int i = 0; i < nseg; ++i) t += (segs[i].n + bn - 1) / bn;
        p.bm = bm, p.bn = bn, p.vtiles = t;
        return (int64_t)t * ((M + bm - 1) / bm);
    };
    int64_t blocks = tiles(chained ? 256 : 128, 256);
    p.form = 2;
    // up to 64 rows keep tiles of their own height however many columns there are: 5 rows of 1152 -> 262144 took 165 /
    // 166 / 152 / 185 us (int8 / f16 / i4 / q4) in tiles of 128 rows, 75 / 111 / 57 / 87 so, 64 rows 171 / 182 / 159 / 199
    // and 111 / 156 / 95 / 120 (single rows' kernels at 5 rows 886 / 591 / 1047 / 308)
    if (blocks < 192 || M <= 64) {
        p.form = M > 32 ? 1 : 0;
        blocks = p.form ? tiles(P == 2 ? 64 : 128, 128) : tiles(32, 128);
    }
    int splits = 1;
    // f16 x: a second block per CU does not pay for the split sums (2048 rows of 2048 -> 2048 34.5 us unsplit on
    // 256 blocks, 43.0 split in two); f32 x: it does or is even (512 rows of 960 -> 960 20.0 against 20.3)
    const int64_t want = p.form == 2 || P == 1 ? 256 : 512;
    while (blocks * splits * 2 <= want && steps / (splits * 2) >= 4) splits *= 2;
    p.steps_per_split = (steps + splits - 1) / splits;
    p.splits = (steps + p.steps_per_split - 1) / p.steps_per_split;
    const auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    p.xp_off = P == 2 ? up((size_t)M * 4) : 0;
    p.sum_off = p.xp_off + (P == 2 || K % kBK || fmt == XG_Q4 ? up((size_t)M * P * steps * kBK * 2) : 0);
    p.part_off = p.sum_off + (fmt == XG_Q4 ? up((size_t)M * steps * 4) : 0);
    p.bytes = p.part_off + (p.splits > 1 ? (size_t)p.splits * M * p.vtiles * p.bn * 4 : 0);
    return p;
}

template <int FMT, bool S16, int P, bool FOLD, int TA, int TB, int WM, int WN, int NST, bool ACT>
hipError_t launch_form(const XgArgs& a, const XgPlan& p, hipStream_t st)
{
    constexpr int lds = NST * stage_bytes(FMT, P, 32 * TA * WM, 32 * TB * WN, Fmt<FMT>::kStepBytes);
    auto kern = qgemm_exact_kernel<FMT, S16, P, FOLD, TA, TB, WM, WN, NST, ACT>;
    if constexpr (lds > 64 * 1024) {
        const hipError_t e = allow_big_lds(kern, lds);
        if (e != hipSuccess) return e;
    }
    const dim3 grid(p.vtiles, (a.M + p.bm - 1) / p.bm, p.splits);
    hipLaunchKernelGGL(kern, grid, dim3(64 * WM * WN), lds, st, a);
    return hipGetLastError();
}

template <int FMT, bool S16, int P, bool ACT, bool FOLD = true>
hipError_t launch_act(const XgArgs& a, const XgPlan& p, hipStream_t st)
{
    // f16 rows are twice the bytes: two stages keep two blocks (form 1) or one (form 2) on a CU
    constexpr int NST = FMT == XG_F16 ? 2 : 3, T1 = P == 2 ? 1 : 2, T2 = FOLD ? 2 : 4;
    hipError_t e = p.form == 2   ? launch_form<FMT, S16, P, FOLD, T2, 2, 2, 4, NST, ACT>(a, p, st)
                   : p.form == 1 ? launch_form<FMT, S16, P, FOLD, T1, 2, 2, 2, NST, ACT>(a, p, st)
                                 : launch_form<FMT, S16, P, FOLD, 1, 2, 1, 2, 3, ACT>(a, p, st);
    if (e != hipSuccess || p.splits == 1) return e;
    const size_t quads = (size_t)a.M * a.vcols / (ACT ? 8 : 4);
    const unsigned blocks = (unsigned)std::min<size_t>((quads + 255) / 256, 4096);
    hipLaunchKernelGGL((qgemm_exact_reduce_kernel<FMT, P, ACT>), dim3(blocks), dim3(256), 0, st, a, p.splits, p.bn);
    return hipGetLastError();
}

template <int FMT, bool S16>
hipError_t launch_f32x(const XgArgs& a, const XgPlan& p, bool act, int32_t* xe, _Float16* xp, float* xsum,
                       hipStream_t st)
{
    hipLaunchKernelGGL((split_x_kernel<Fmt<FMT>::kPairs, FMT == XG_Q4>), dim3(a.M), dim3(256), 0, st,
                       static_cast<const float*>(a.x), a.K, a.Kp, xp, xe, xsum);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if constexpr (FMT != XG_F16)
        if (act) return launch_act<FMT, S16, 2, true>(a, p, st);
    return launch_act<FMT, S16, 2, false>(a, p, st);
}

}  // namespace

bool qgemm_exact_supported(const XgCall& c, int M, int K)
{
    const bool nibbles = c.fmt == XG_I4 || c.fmt == XG_Q4;
    // weight rows start on 16-byte boundaries; a K step has one scale
    if (M < (c.x_f16 && c.fmt == XG_I8 ? 1 : 5) || K <= 0 || K % (nibbles ? 32 : c.fmt == XG_I8 ? 16 : 8) != 0) return false;
    if (c.fmt == XG_Q4 && (c.group <= 0 || c.group % kBK != 0)) return false;
    if (c.x_f16 && c.fmt != XG_I8 && (c.fmt != XG_Q4 || !c.segs[0].gb)) return false;
    if (c.act >= 0 && (c.fmt == XG_F16 || c.nseg != 2 || c.segs[0].n != c.segs[1].n)) return false;
    int64_t n = 0;
    for (int i = 0; i < c.nseg; ++i) {
        if (c.segs[i].n <= 0 || (reinterpret_cast<uintptr_t>(c.segs[i].w) & 15) != 0) return false;
        // group scales and biases are fetched as whole elements
        if (((reinterpret_cast<uintptr_t>(c.segs[i].gs) | reinterpret_cast<uintptr_t>(c.segs[i].gb)) & 3) != 0) return false;
        n += c.segs[i].n;
    }
    if ((reinterpret_cast<uintptr_t>(c.x) & 15) != 0 || (M + 31) / 32 > 65535) return false;
    // a tile's byte offsets are 32-bit
    if ((uint64_t)K * 1024 >= (1ull << 31) || n >= (1 << 30)) return false;
    if (c.x_f16 && (c.fmt == XG_I8 ? K % kBK == 0 : M > 64)) return true;  // x in place; over the tile kernels of f16 weights
    // The kernels of single rows walk the rows one after the other (f16: four at a time), so they take
    // longer with M K (a wave's walk) and with M K N (the whole work); the three launches here take 14-17
    // us at small sizes.  Measured, row kernels against these (us, rows x outputs x k):
    //   int8  5 x 960 x 960 10.7 / 16.2, 5 x 576 x 1536 15.2 / 14.4, 5 x 8192 x 960 22.8 / 17.4
    //   i4    5 x 960 x 960 16.0 / 16.0, 8 x 960 x 960 24.4 / 15.3
    //   f16   8 x 960 x 960 11.3 / 14.9, 12 x 2560 x 960 21.2 / 14.9, 5 x 8192 x 960 19.5 / 14.9
    //   q4    16 x 2560 x 960 13.3 / 17.7, 24 x 1024 x 1024 14.6 / 13.3, 5 x 16384 x 960 17.5 / 17.4
    const bool affine = c.fmt == XG_Q4 && c.segs[0].gb;
    const int64_t walk = affine ? 24000 : c.fmt == XG_F16 ? 10000 : nibbles ? 5000 : 7000;
    const double work = affine ? 78e6 : 35e6;
    return (int64_t)M * K * c.nseg >= walk || (double)M * K * n >= work;
}

size_t qgemm_exact_workspace_bytes(const XgCall& c, int M, int K)
{
    return xg_plan(c.fmt, c.x_f16 ? 1 : 2, c.segs, c.nseg, c.act >= 0, M, K).bytes;
}

hipError_t launch_qgemm_exact(const XgCall& c, int M, int K, void* ws, hipStream_t st)
{
    const bool act = c.act >= 0;
    XgPlan p = xg_plan(c.fmt, c.x_f16 ? 1 : 2, c.segs, c.nseg, act, M, K);
    if (!ws && p.splits > 1) {  // x in place and no workspace for split sums
        p.steps_per_split *= p.splits;
        p.splits = 1;
    }
    XgArgs a{};
    for (int i = 0, t = 0; i < 3; ++i) {
        a.tile0[i] = i < c.nseg && !act ? t : INT32_MAX;
        if (i >= c.nseg) continue;
        a.seg[i] = c.segs[i];
        t += (c.segs[i].n + p.bn - 1) / p.bn;
    }
    unsigned char* base = static_cast<unsigned char*>(ws);
    int32_t* xe = reinterpret_cast<int32_t*>(base);
    _Float16* xp = reinterpret_cast<_Float16*>(base + p.xp_off);
    float* xsum = reinterpret_cast<float*>(base + p.sum_off);
    a.xe = xe;
    a.xp = xp;
    a.xsum = xsum;
    a.x = c.x;
    a.part = p.splits > 1 ? reinterpret_cast<float*>(base + p.part_off) : nullptr;
    a.M = M;
    a.K = K;
    a.Kp = (K + kBK - 1) / kBK * kBK;
    a.steps_per_split = p.steps_per_split;
    a.vcols = p.vtiles * p.bn;
    a.sdt = c.sdt;
    a.group = c.group;
    a.gpr = c.gpr;
    a.act = c.act;
    if (c.x_f16 && c.fmt == XG_Q4) {
        const size_t units = (size_t)M * a.Kp / 8;
        hipLaunchKernelGGL(pair_x_kernel, dim3((unsigned)std::min<size_t>((units + 255) / 256, 4096)), dim3(256), 0, st,
                           static_cast<const _Float16*>(c.x), M, K, a.Kp, xp, xsum);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        if (c.sdt == DT_F32) return act ? launch_act<XG_Q4, false, 1, true>(a, p, st) : launch_act<XG_Q4, false, 1, false>(a, p, st);
        return act ? launch_act<XG_Q4, true, 1, true>(a, p, st) : launch_act<XG_Q4, true, 1, false>(a, p, st);
    }
    if (c.x_f16 && xg_chained(c.fmt, 1, K)) {
        a.xp = static_cast<const _Float16*>(c.x);
        return act ? launch_act<XG_I8, false, 1, true, false>(a, p, st) : launch_act<XG_I8, false, 1, false, false>(a, p, st);
    }
    if (c.x_f16) {
        const size_t units = (size_t)M * a.Kp / 8;
        hipLaunchKernelGGL(pad_x_kernel, dim3((unsigned)std::min<size_t>((units + 255) / 256, 4096)), dim3(256), 0, st,
                           static_cast<const _Float16*>(c.x), K, a.Kp, units, xp);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        return act ? launch_act<XG_I8, false, 1, true>(a, p, st) : launch_act<XG_I8, false, 1, false>(a, p, st);
    }
    switch (c.fmt) {
        case XG_I8: return launch_f32x<XG_I8, false>(a, p, act, xe, xp, xsum, st);
        case XG_I4: return launch_f32x<XG_I4, false>(a, p, act, xe, xp, xsum, st);
        case XG_F16: return launch_f32x<XG_F16, false>(a, p, act, xe, xp, xsum, st);
        case XG_Q4:
            return c.sdt == DT_F32 ? launch_f32x<XG_Q4, false>(a, p, act, xe, xp, xsum, st)
                                   : launch_f32x<XG_Q4, true>(a, p, act, xe, xp, xsum, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace cellm
