// GQA attention over paged f16 K/V on f16 MFMA (gfx950): prompts, many sessions
// and long contexts (attention_single_token_gqa_f32,
// crates/cellm-cache/src/kvcache.rs:710-789; the sliding windows of
// crates/cellm-model/src/gemma.rs:747-780).
//
// A block computes up to 16 query vectors ("columns") that read the same K and V
// over a range of positions, so each K and V element is fetched once for all:
//   - the G query heads of one (row, kv head), or
//   - one query head of up to 16 neighbouring rows whose block tables agree over
//     their positions: the tokens of a prompt.
// Which of the two is found on the device: a row joins its 16-row tile's set if
// its table equals the table of the tile's furthest row over its own positions,
// and the set is worth sharing (rule below).  A set is computed in units of one
// query head and one range of positions, spread over the blocks of the tile's
// rows; any other row by its own blocks.  Sessions with pages of their own differ
// in their first page, which one load per row shows.
//
// Wave w of 4 takes chunks of 32 positions, w, w + 4, ...  A chunk is
//   S^T [32 positions][16 columns] = K . Q^T       v_mfma_f32_16x16x32_f16
//   O^T [HD][16 columns] += V^T . P^T
// with K straight from the pages as the A operand and V through wave-private LDS,
// transposed.  S^T leaves lane (column c, group g) with positions 4 g + 0..3 of
// both halves of the chunk; the k order of the second product is free as long as
// V^T and P^T agree, so those eight weights are its B operand as they are.
// Each wave keeps a running maximum, sum and O^T; the waves meet in LDS once.
//
// q and the softmax weights are two f16 parts each, 23 bits of their 24: hi =
// RNE_f16(v') and lo = RNE_f16(v' - hi), of v scaled by a power of two (q: its
// largest |q| to [2^13, 2^14); weights: by 2^13), multiplied one after the other.
// Elements below 2^-15 of the head's largest |q| are held to 2^-38 of that, weights
// below 2^-15 to 2^-38.
// K and V are f16 and exact.  Scores, exponentials and sums are f32.  Sums of a
// block that are not finite (an infinity or NaN in q, K or V: inf * lo may be NaN
// where inf * v is not, and a masked position's 0 * inf is) are computed again by
// plain f32 sums over the block's positions.
//
// Long contexts split their positions over blocks, a row's and a set's: partial
// sums (HD values, the maximum, the sum) go to the workspace with agent-coherent
// stores and the last block of the row's or of the set's head adds them in split
// order, as in attn_partial_kernel.
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "kernels.hpp"

#pragma clang fp contract(off)

namespace cellm {

namespace {

typedef float f2_t __attribute__((ext_vector_type(2)));

constexpr int kWaves = 4, kThreads = kWaves * 64, kCols = 16, kChunk = 32;
constexpr int kMinSplit = kWaves * kChunk;  // positions: a chunk per wave
// rows share where their own positions have no splits, or up to kShareSplits of at least kSharePositions
constexpr int kShareSplits = 6, kSharePositions = 1024;
constexpr int kMinTileSplit = 256, kMaxTileSplits = 32;  // positions of a set's split, splits
constexpr float kWeightScale = 8192.0f;  // of the softmax weights (two f16 parts), and so of the sums l and O
constexpr int kVStride = kChunk + 4;  // halves between the dims of a transposed V chunk

struct AttnArgs {
    const float* q;
    const uint16_t* kc;
    const uint16_t* vc;
    const int32_t* pos;
    const uint32_t* bt;
    int max_blocks, total_blocks, n_layers, tpb, tpb_shift;  // tpb_shift: log2(tpb), or -1
    int rows, n_heads, n_kv, group, layer, window, tiles;
    float scale, soft_cap;
    int nsplit, cap;        // splits of a row's positions at most; positions of a table
    int tsplit, tsplit_last, slots;  // splits of a full and of the last, ragged tile's set at most; slots in `part`
    int busy;               // rows of a shared tile whose blocks have a unit of it, at most
    float* part;            // [row][kv head][slot][group][HD + 2]
    uint32_t* counters;     // per (row, kv head): splits done, zero between calls
    float* out;
};

__device__ __forceinline__ bool finite_f32(float v) { return (__builtin_bit_cast(uint32_t, v) & 0x7F800000u) != 0x7F800000u; }
__device__ __forceinline__ void st_agent(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float ld_agent(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ f2_t ld_agent2(const float* p)  // 8-byte aligned
{
    return __builtin_bit_cast(f2_t, __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ int first_position(int seq, int window) { return window > 0 ? max(seq - window, 0) : 0; }
// LDS of one wave, written and read across its lanes: the wave's LDS operations run in order, and the
// compiler moves none across this
__device__ __forceinline__ void wave_lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// element offset of position t of `layer` in the cache, or -1 where its page is missing
__device__ __forceinline__ long long page_base(const AttnArgs& a, int row, int t, int kvd)
{
    const int b = a.tpb_shift >= 0 ? t >> a.tpb_shift : t / a.tpb;
    if (b >= a.max_blocks) return -1;
    const uint32_t blk = a.bt[(size_t)row * a.max_blocks + b];
    if (blk >= (uint32_t)a.total_blocks) return -1;
    return (((long long)blk * a.n_layers + a.layer) * a.tpb + (t - b * a.tpb)) * kvd;
}

__device__ __forceinline__ float capped(const AttnArgs& a, float s)
{
    return a.soft_cap > 0.0f ? tanhf(s / a.soft_cap) * a.soft_cap : s;  // kvcache.rs:768-770
}

// e^x for x <= 0 to the accuracy of the hardware exponential: x log2(e) in two parts, the second folded in
// to first order.  -inf gives NaN (callers select masked positions away).
__device__ __forceinline__ float exp_neg(float x)
{
    const float kLog2e = 1.4426950216293335f, kLog2eLo = 1.9259629911266175e-8f, kLn2 = 0.6931471805599453f;
    const float h = x * kLog2e;
    const float r = __builtin_fmaf(x, kLog2eLo, __builtin_fmaf(x, kLog2e, -h));
    const float e = __builtin_amdgcn_exp2f(h);
    return __builtin_fmaf(e, r * kLn2, e);
}

// Positions lo..up of one (row, head) by plain f32 sums, the whole block: maximum m, sum l of e^(score - m) and, in
// threads below HD, the weighted sum of V (returned).  256 positions at a time: a score per thread, then HD threads
// per position.  A range without a score above -inf has weights of 0 where other ranges follow (`part`).  With a NaN in its
// first page a prompt of 512 tokens, 14/2 heads of 64, takes 0.34 ms (0.015 without; the vector kernels 0.1), 8 sessions
// at 8192 positions 0.33 (0.057; 0.09).
template <int HD>
__device__ __forceinline__ float plain_range(const AttnArgs& a, int row, int head, int lo, int up, bool part,
                                             unsigned char* lds, float& m, float& l)
{
    long long* const bases = reinterpret_cast<long long*>(lds);
    float* const red = reinterpret_cast<float*>(bases + kThreads);
    float* const ws = red + kThreads;
    const int t = threadIdx.x, kvd = a.n_kv * HD, kvh = head / a.group;
    const float* qr = a.q + ((size_t)row * a.n_heads + head) * HD;
    const auto score = [&](long long b) {
        float d = 0.0f;
        if (b >= 0) {
            const u4_t* src = reinterpret_cast<const u4_t*>(a.kc + b + (long long)kvh * HD);
            u4_t k[HD / 8];
#pragma unroll
            for (int i = 0; i < HD / 8; ++i) k[i] = src[i];
#pragma unroll
            for (int i = 0; i < HD / 8; ++i) {
                const h8_t h = __builtin_bit_cast(h8_t, k[i]);
#pragma unroll
                for (int j = 0; j < 8; ++j) d = d + qr[8 * i + j] * (float)h[j];
            }
        }
        return capped(a, d * a.scale);
    };
    const auto reduce = [&](float v, auto op) {  // over the block
        __syncthreads();
        red[t] = v;
        __syncthreads();
        for (int o = kThreads / 2; o > 0; o >>= 1) {
            if (t < o) red[t] = op(red[t], red[t + o]);
            __syncthreads();
        }
        return red[0];
    };
    float mt = -INFINITY;
#pragma unroll 1
    for (int p = lo + t; p < up; p += kThreads) mt = fmaxf(mt, score(page_base(a, row, p, kvd)));
    m = reduce(mt, [](float x, float y) { return fmaxf(x, y); });
    constexpr int NP = kThreads / HD, UN = 16;
    const int d = t % HD;
    float lt = 0.0f, o = 0.0f;
#pragma unroll 1
    for (int p0 = lo; p0 < up; p0 += kThreads) {
        const int n = min(kThreads, up - p0);
        long long b = -1;
        float w = 0.0f;
        if (t < n) {
            b = page_base(a, row, p0 + t, kvd);
            const float s = score(b);
            w = part && m == -INFINITY && s == -INFINITY ? 0.0f : expf(s - m);
        }
        lt = lt + w;
        __syncthreads();
        bases[t] = b;
        ws[t] = w;
        __syncthreads();
#pragma unroll 1
        for (int j0 = t / HD; j0 < n; j0 += NP * UN) {
            uint16_t v[UN];
#pragma unroll
            for (int i = 0; i < UN; ++i) {
                const long long bj = bases[min(j0 + i * NP, kThreads - 1)];
                v[i] = a.vc[max(bj, 0ll) + (long long)kvh * HD + d];
            }
#pragma unroll
            for (int i = 0; i < UN; ++i) {
                const int j = j0 + i * NP;
                if (j < n) o = o + ws[j] * (bases[j] >= 0 ? (float)__builtin_bit_cast(_Float16, v[i]) : 0.0f);
            }
        }
    }
    l = reduce(lt, [](float x, float y) { return x + y; });
    __syncthreads();
    red[t] = o;
    __syncthreads();
    o = 0.0f;
    for (int j = 0; j < NP; ++j) o = o + red[j * HD + d];
    __syncthreads();
    return o;
}

// Row of the i-th block of a kv head: of all tiles the rows whose blocks have the units of a set's first split (one
// per query head), then those of its other splits, then those whose blocks then leave at once, and the last tile
// first (in a prompt its rows see the most positions).  Blocks go to the XCDs in turn: with the rows in order one
// XCD in four had half the others' work (a 2048-token prompt of 14 / 2 heads 126 us in row order, 74 so), and with
// the rows of all splits together sets that have no splits fill half the XCDs (855 tokens of 4 / 1 heads of 128 at
// 1100 positions, window 512, 26.7 us, 20.5 so).
__device__ __forceinline__ int block_row(const AttnArgs& a, int i)
{
    const int full = a.rows / kCols, rem = a.rows - full * kCols;
    int lo = 0, hi = a.group, first = min(rem, hi);
    for (int next = a.busy;; next = kCols) {
        const int n = full * (hi - lo) + first;
        if (i < n) break;
        i -= n;
        lo = hi;
        hi = next;
        first = max(0, min(rem, hi) - lo);
    }
    if (i < first) return full * kCols + lo + i;
    const int j = i - first, w = hi - lo;
    return (full - 1 - j / w) * kCols + lo + j % w;
}

// Registers: four waves per SIMD at HD 64 (a 2048-token prompt of 14 / 2 heads 74 us at three, 67 at four); HD 128
// needs the registers of three.  Measured, us, vector kernels -> this: prompts of 512 and 2048 tokens, 14 / 2 heads
// of 64, 90 -> 13 and 589 -> 61; 1024 tokens at 2048 positions, 32 / 8 heads of 128, 1586 -> 182; 8 sessions at
// 4096..8192 positions, 32 / 8 heads of 128, 82 -> 54 (3.7 TB/s), 16 sessions at 8192..16384, 8 / 8 heads of 128,
// 190 -> 176 (4.6 TB/s).  Prompts are bound by the latency of a chunk (page, K, scores, maximum, weights, V in LDS)
// at about two waves per SIMD, long contexts by memory.  The error against 64 bits is 0.92 of the vector
// kernels' over 70 calls of both directions and none larger by more than 5 % (8 sessions at 4096..8192, by the seed,
// 3.7e-7 / 3.8e-7 and 4.5e-7 / 4.3e-7).
template <int HD, bool CAP>
__global__ __launch_bounds__(kThreads, HD == 64 ? 4 : 3) void attn_mma_kernel(const AttnArgs a)
{
    constexpr int KK = HD / 32, DT = HD / 16;         // 32-wide k steps of Q.K, 16-wide tiles of O^T
    constexpr int VU = HD / 32;                       // V units (two positions x 8 dims) per lane and chunk
    constexpr int OS = HD + 4;                        // floats between the columns of a wave's O^T in LDS
    constexpr int kWaveLds = HD * kVStride * 2 > kCols * OS * 4 ? HD * kVStride * 2 : kCols * OS * 4;
    __shared__ __align__(16) unsigned char wave_lds[kWaves * kWaveLds];
    constexpr int QS = HD + 8;                        // halves between the columns of a q part
    __shared__ __align__(16) _Float16 qs[2][kCols * QS];
    __shared__ int es[kCols];
    __shared__ long long bases_s[kWaves][kChunk];
    __shared__ float ml[kWaves][2][kCols];
    __shared__ uint32_t flags;                        // tile rows that differ; then columns to sum plainly
    __shared__ int last, splits_s;                    // splits_s: of this pass (a scalar register fewer over the loop)

    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int c = lane & 15, g4 = lane >> 4;
    const int r = block_row(a, blockIdx.x / a.n_kv), kvh = blockIdx.x % a.n_kv, sp = blockIdx.y;
    const int cap = a.cap, kvd = a.n_kv * HD;

    // ---- positions and first pages of the tile's rows, and the first chunk's page entry
    const int tile0 = r & ~(kCols - 1), sub = r & (kCols - 1), nr = min(kCols, a.rows - tile0);
    const int jr = tile0 + min(c, nr - 1);
    const auto block_of = [&](int p) { return a.tpb_shift >= 0 ? p >> a.tpb_shift : p / a.tpb; };
    const int b_first = min(block_of(wave * kChunk + (lane & 31)), a.max_blocks - 1);
    const int pos_c = a.pos[a.tiles ? jr : r];
    const uint32_t first = a.bt[(size_t)(a.tiles ? jr : r) * a.max_blocks];
    const uint32_t own_first = a.bt[(size_t)r * a.max_blocks + b_first];
    uint32_t lead_first = own_first;
    const int pj = !a.tiles || c < nr ? min(pos_c + 1, cap) : 0;  // positions of tile row c (of row r without tiles)
    const int seq_own = __builtin_amdgcn_readlane(pj, a.tiles ? sub : 0);

    // ---- which rows of the tile share their pages
    const int most_splits = nr == kCols ? a.tsplit : a.tsplit_last;
    uint32_t members = 0;  // of the shared set, by row of the tile
    int leader = sub, seq_lead = 0;
    if (a.tiles) {
        int best = (pj << 4) | (15 - c);
        best = max(best, __shfl_xor(best, 8));
        best = max(best, __shfl_xor(best, 4));
        best = max(best, __shfl_xor(best, 2));
        best = max(best, __shfl_xor(best, 1));
        best = __builtin_amdgcn_readfirstlane(best);
        leader = 15 - (best & 15);
        seq_lead = best >> 4;
        const uint32_t* lead = a.bt + (size_t)(tile0 + leader) * a.max_blocks;
        lead_first = lead[b_first];
        members = (uint32_t)__ballot(pj > 0 && first == (uint32_t)__builtin_amdgcn_readlane((int)first, leader)) & 0xFFFFu;
        // Worth sharing: a row by itself fills `group` of the 16 columns, a set one per row, and its last block adds
        // 16 columns where a row's adds `group`.  us, each row by itself / a set, 1 set and 2 and 4 (16, 32, 64 rows of
        // one session): 14/2 heads of 64, 8192 positions 20.6 / 28.1, 25.7 / 29.7, 38.2 / 33.9; 2048 16.7 / 17.3, 17.8 /
        // 18.4, 19.1 / 19.6; 32/8 of 128, 8192 64.9 / 42.8, 110 / 51, 154 / 73; 1024 20.4 / 21.4, 27.0 / 22.9, 26.7 / 26.7.
        // Two rows of 14/2 heads at 8192 positions took 371 us as a set with one block per head, 17 so.
        const int span = a.window > 0 ? min(seq_lead, a.window) : seq_lead;
        if (__popc(members) < max(a.group, 2) ||
            (a.nsplit > 1 && (a.nsplit > kShareSplits || span < a.nsplit * kSharePositions)))
            members = 0;
        if (members) {
            // whole tables: thread t compares entries t / 16, t / 16 + 16, ... of tile row t % 16 (that is c); of
            // every candidate where this block needs the set, of its own row where that is all
            if (t == 0) flags = 0;
            __syncthreads();
            const bool mine = (members >> c & 1) && c != leader && (c == sub || sub < a.group || sub == leader || most_splits > 1);
            const int nb = mine ? (pj + a.tpb - 1) / a.tpb : 0;
            const uint32_t* own = a.bt + (size_t)jr * a.max_blocks;
            bool differ = false;
            for (int b = t >> 4; b < nb; b += 4 * (kThreads / 16)) {
                uint32_t x[4], y[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int bi = min(b + i * (kThreads / 16), nb - 1);
                    x[i] = own[bi];
                    y[i] = lead[bi];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) differ |= x[i] != y[i];
            }
            const unsigned long long bits = __ballot(differ);
            uint32_t rows = (uint32_t)bits | (uint32_t)(bits >> 32);
            rows = (rows | rows >> 16) & 0xFFFFu;
            if (lane == 0 && rows) atomicOr(&flags, rows);
            __syncthreads();
            members &= ~flags;
        }
        if (__popc(members) < 2) members = 0;
        members = __builtin_amdgcn_readfirstlane(members);
    }

    unsigned char* const my_lds = wave_lds + wave * kWaveLds;
    _Float16* const vt = reinterpret_cast<_Float16*>(my_lds);
    const bool in_set = members >> sub & 1;

    // The shared set: positions lo_set..seq_lead in `tsplits` parts, one unit per query head and part
    int lo_set = 0, tsplits = 1, tper = 0;
    if (members) {
        if (a.window > 0) {
            lo_set = members >> c & 1 ? first_position(pj, a.window) : cap;
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) lo_set = min(lo_set, __shfl_xor(lo_set, o));
            lo_set = __builtin_amdgcn_readfirstlane(lo_set) & ~(kChunk - 1);
        }
        const int len = seq_lead - lo_set;
        const int n = len < 4 * kMinTileSplit ? 1 : max(1, min(most_splits, len / kMinTileSplit));
        tper = __builtin_amdgcn_readfirstlane(((len + n - 1) / n + kChunk - 1) & ~(kChunk - 1));
        tsplits = __builtin_amdgcn_readfirstlane((len + tper - 1) / tper);
    }
    const int units = members ? a.group * tsplits : 0;

    // the set's units, spread over the blocks of the tile's rows, then this row's heads if it is not in the set
    for (int u = sub + nr * sp;; u += nr * a.nsplit) {
        const bool solo = u >= units;
        if (solo && in_set) break;
        const int ts = solo ? sp : __builtin_amdgcn_readfirstlane(u / a.group), h = solo ? 0 : u - ts * a.group;
        // column c: its positions, and those of the whole block
        const bool has = solo ? c < a.group : members >> c & 1;
        const int seq_c = has ? (solo ? seq_own : pj) : 0;
        const int s0_c = first_position(seq_c, a.window);
        const int hi = solo ? seq_own : seq_lead;
        if (hi <= 0) break;  // no position: nothing written
        const int table = solo ? r : tile0 + leader;
        int t0 = solo ? first_position(hi, a.window) & ~(kChunk - 1) : lo_set, t1 = hi, splits = tsplits, per = tper;
        if (solo) {
            // Rows past half their table take shares of the table, the others (and windows) spread their own
            // positions over all splits.  us, shares / spread: 8 rows, 32/8 heads of 128, table of 8192, positions
            // 500 16.1 / 13.1, 2000 29.3 / 23.5, 4096..8191 56.4 / 57.6; 16 rows, 8/8 of 128, 9000 of 16384 116 /
            // 122; 1 row, 14/2 of 64, 1000 of 32768 14.9 / 11.3 (at least 256 a split 12.6); 16 rows, 32/8 of 128,
            // window 2048 of 8192 47.3 / 33.9
            const int len = hi - t0, over = 2 * len >= a.cap ? a.cap : len;
            // (the divisions run on the vector unit: their results go back to scalars)
            per = __builtin_amdgcn_readfirstlane(
                max(kMinSplit, ((over + a.nsplit - 1) / a.nsplit + kChunk - 1) & ~(kChunk - 1)));
            splits = __builtin_amdgcn_readfirstlane((len + per - 1) / per);
            if (sp >= splits) break;
        }
        t0 += ts * per;
        t1 = min(hi, t0 + per);
        if (t == 0) splits_s = splits;  // read after the barriers below

        // ---- q: two f16 parts of every column in LDS (wave 0; lane (c, g4): dims 32 kk + 8 g4 + 0..7)
        if (wave == 0) {
            const int row = solo ? r : jr, head = kvh * a.group + (solo ? min(c, a.group - 1) : h);
            const f4_t* src = reinterpret_cast<const f4_t*>(a.q + ((size_t)row * a.n_heads + head) * HD + 8 * g4);
            f4_t qv[KK][2];
#pragma unroll
            for (int kk = 0; kk < KK; ++kk)
#pragma unroll
                for (int i = 0; i < 2; ++i) qv[kk][i] = src[kk * 8 + i];
            float mx = 0.0f;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float x = fabsf(qv[kk][i >> 2][i & 3]);
                    mx = finite_f32(x) ? fmaxf(mx, x) : mx;
                }
            mx = fmaxf(mx, lane_xor<16>(mx, 64));
            mx = fmaxf(mx, lane_xor<32>(mx, 64));
            const int top = (int)(__builtin_bit_cast(uint32_t, mx) >> 23);
            const int e = mx > 0.0f ? 13 - (max(top, 1) - 127) : 0;
            if (g4 == 0) es[c] = e;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                h8_t hi8, lo8;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float x = ldexpf(qv[kk][i >> 2][i & 3], e);
                    hi8[i] = (_Float16)x;
                    lo8[i] = finite_f32(x) ? (_Float16)(x - (float)hi8[i]) : (_Float16)0.0f;
                }
                *reinterpret_cast<h8_t*>(&qs[0][c * QS + 32 * kk + 8 * g4]) = hi8;
                *reinterpret_cast<h8_t*>(&qs[1][c * QS + 32 * kk + 8 * g4]) = lo8;
            }
        }
        __syncthreads();
        const float qscale = ldexpf(a.scale, -es[c]);
        const _Float16* const qc = &qs[0][c * QS + 8 * g4];

        f4_t o[DT];
#pragma unroll
        for (int d = 0; d < DT; ++d) o[d] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
        float m = -INFINITY, l = 0.0f;
        // the page entry of position p + lane % 32, loaded a chunk ahead of its use and as it is (every load
        // below has an address in range and no branch before it, so that none waits for another)
        const uint32_t* const bt = a.bt + (size_t)table * a.max_blocks;
        int b_next = block_of(t0 + wave * kChunk + (lane & 31));
        uint32_t blk_next = solo ? own_first : lead_first;
        if (t0 > 0) blk_next = bt[min(b_next, a.max_blocks - 1)];
        const uint16_t* const kh = a.kc + kvh * HD + 8 * g4;
        const uint16_t* const vh = a.vc + kvh * HD;
        for (int p0 = t0 + wave * kChunk; p0 < t1; p0 += kWaves * kChunk) {
            bool missing;
            {
                const int pp = p0 + (lane & 31);
                const bool ok = pp < t1 && b_next < a.max_blocks && blk_next < (uint32_t)a.total_blocks;
                const long long own =
                    (((long long)blk_next * a.n_layers + a.layer) * a.tpb + (pp - b_next * a.tpb)) * kvd;
                wave_lds_fence();
                if (lane < kChunk) bases_s[wave][lane] = ok ? own : -1;
                missing = __ballot(!ok) != 0;
                wave_lds_fence();
            }
            b_next = block_of(p0 + kWaves * kChunk + (lane & 31));
            blk_next = bt[min(b_next, a.max_blocks - 1)];
            u4_t kraw[2][KK], vraw[VU][2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const long long b = bases_s[wave][16 * j + c];
                const u4_t* src = reinterpret_cast<const u4_t*>(kh + max(b, 0ll));
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) kraw[j][kk] = src[kk * 4];
            }
            // V unit u: positions 2 (u / (HD / 8)) + 0, 1, dims 8 (u % (HD / 8)) + 0..7
#pragma unroll
            for (int i = 0; i < VU; ++i) {
                const int u = lane + 64 * i, vg = u % (HD / 8), vp = u / (HD / 8);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const long long b = bases_s[wave][2 * vp + j];
                    vraw[i][j] = *reinterpret_cast<const u4_t*>(vh + max(b, 0ll) + 8 * vg);
                }
            }
            asm volatile("" ::: "memory");  // every load issued, in this order, before any is used
            // a missing page counts as zeros, and so do the positions past the range that pad the last chunk
            // (their weights are 0)
            if (missing) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int kk = 0; kk < KK; ++kk) kraw[j][kk] = bases_s[wave][16 * j + c] >= 0 ? kraw[j][kk] : u4_t{0, 0, 0, 0};
            }
            // scores of positions p0 + 16 j + 4 g4 + i: the low parts, then the high ones
            f4_t s[2] = {};
#pragma unroll
            for (int part = 1; part >= 0; --part)
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) {
                    const h8_t qv = *reinterpret_cast<const h8_t*>(qc + part * kCols * QS + 32 * kk);
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        s[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, kraw[j][kk]), qv, s[j], 0, 0, 0);
                }
            // positions that some column does not attend to
            const bool partial = __ballot(has && (p0 < s0_c || p0 + kChunk > seq_c)) != 0;
            float mc = -INFINITY;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[j][i] = s[j][i] * qscale;
                    if constexpr (CAP) s[j][i] = capped(a, s[j][i]);
                    if (partial) {
                        const int p = p0 + 16 * j + 4 * g4 + i;
                        s[j][i] = p >= s0_c && p < seq_c ? s[j][i] : -INFINITY;
                    }
                    mc = fmaxf(mc, s[j][i]);
                }
            mc = fmaxf(mc, lane_xor<16>(mc, 64));
            mc = fmaxf(mc, lane_xor<32>(mc, 64));
            if (missing) {
#pragma unroll
                for (int i = 0; i < VU; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        vraw[i][j] = bases_s[wave][2 * ((lane + 64 * i) / (HD / 8)) + j] >= 0 ? vraw[i][j] : u4_t{0, 0, 0, 0};
            }
            // transposed V
#pragma unroll
            for (int i = 0; i < VU; ++i) {
                const int u = lane + 64 * i, vg = u % (HD / 8), vp = u / (HD / 8);
                uint32_t* dst = reinterpret_cast<uint32_t*>(vt + (size_t)vg * 8 * kVStride + 2 * vp);
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    dst[(2 * w) * (kVStride / 2)] = __builtin_amdgcn_perm(vraw[i][1][w], vraw[i][0][w], 0x05040100u);
                    dst[(2 * w + 1) * (kVStride / 2)] = __builtin_amdgcn_perm(vraw[i][1][w], vraw[i][0][w], 0x07060302u);
                }
            }
            // weights times 2^13 (and so the sums l and O: the factor leaves with their quotient)
            const float mn = fmaxf(m, mc);
            const float shrink = mn > m && m > -INFINITY ? exp_neg(m - mn) : 1.0f;  // from -inf: l and O are 0
            m = mn;
            h8_t ph, pl;
            float lc = 0.0f;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float w = exp_neg(s[j][i] - mn) * kWeightScale;
                    if (partial) {
                        const int p = p0 + 16 * j + 4 * g4 + i;
                        w = p >= s0_c && p < seq_c ? w : 0.0f;
                    }
                    lc = lc + w;
                    ph[4 * j + i] = (_Float16)w;
                    pl[4 * j + i] = (_Float16)(w - (float)ph[4 * j + i]);
                }
            l = l * shrink + lc;
            wave_lds_fence();
            // the chunk's product by itself, then onto O^T: one rounding of the running sums per chunk
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const _Float16* src = vt + (size_t)(d * 16 + c) * kVStride + 4 * g4;
                const h4_t v0 = *reinterpret_cast<const h4_t*>(src), v1 = *reinterpret_cast<const h4_t*>(src + 16);
                const h8_t v = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                f4_t acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, pl, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, ph, acc, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) o[d][i] = __builtin_fmaf(o[d][i], shrink, acc[i]);
            }
        }
        l = l + lane_xor<16>(l, 64);
        l = l + lane_xor<32>(l, 64);

        // ---- the waves meet: O^T over the V chunks' LDS, maxima and sums beside it
        __syncthreads();
        float* ow = reinterpret_cast<float*>(my_lds) + c * OS + 4 * g4;
#pragma unroll
        for (int d = 0; d < DT; ++d) *reinterpret_cast<f4_t*>(ow + d * 16) = o[d];
        if (g4 == 0) {
            ml[wave][0][c] = m;
            ml[wave][1][c] = l;
        }
        if (t == 0) flags = 0;
        __syncthreads();
        const int nsp = __builtin_amdgcn_readfirstlane(splits_s);
        const bool split = nsp > 1;
        // column oc's partials of split 0, and the floats between splits
        const auto partial_of = [&](int oc) {
            const int row = solo ? r : tile0 + oc, head = solo ? oc : h;
            return a.part + ((size_t)(row * a.n_kv + kvh) * a.slots * a.group + head) * (HD + 2);
        };
        const size_t split_step = (size_t)a.group * (HD + 2);
        for (int i = t; i < kCols * (HD / 4); i += kThreads) {
            const int oc = i / (HD / 4), d4 = i % (HD / 4);
            if (solo ? oc >= a.group : !(members >> oc & 1)) continue;
            float mm = ml[0][0][oc];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) mm = fmaxf(mm, ml[w][0][oc]);
            float ll = 0.0f;
            f4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const float ew = ml[w][0][oc] > -INFINITY ? expf(ml[w][0][oc] - mm) : 0.0f;
                ll = ll + ml[w][1][oc] * ew;
                acc = acc + *reinterpret_cast<const f4_t*>(reinterpret_cast<const float*>(wave_lds + w * kWaveLds) + oc * OS + 4 * d4) * ew;
            }
            if (split) {
                float* p = partial_of(oc) + ts * split_step;
#pragma unroll
                for (int k = 0; k < 4; ++k) st_agent(p + 4 * d4 + k, acc[k]);
                if (d4 == 0) {
                    st_agent(p + HD, mm);
                    st_agent(p + HD + 1, ll);
                }
            } else {
                acc = acc * (ll > 0.0f ? 1.0f / ll : 0.0f);
                const int row = solo ? r : tile0 + oc, head = kvh * a.group + (solo ? oc : h);
                *reinterpret_cast<f4_t*>(a.out + ((size_t)row * a.n_heads + head) * HD + 4 * d4) = acc;
            }
            if (!(finite_f32(acc[0]) && finite_f32(acc[1]) && finite_f32(acc[2]) && finite_f32(acc[3])) || !finite_f32(ll))
                atomicOr(&flags, 1u << oc);
        }
        __syncthreads();
        const uint32_t again = flags;
        if (again) {  // rare: columns that are not finite over this block's positions
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // their first values are written
            __syncthreads();
#pragma unroll 1
            for (int oc = 0; oc < kCols; ++oc) {
                if (!(again >> oc & 1)) continue;
                const int row = solo ? r : tile0 + oc, head = kvh * a.group + (solo ? oc : h);
                const int seq = min(a.pos[row] + 1, cap);
                float mm, ll;
                const float o_c = plain_range<HD>(a, row, head, max(t0, first_position(seq, a.window)), min(t1, seq), split,
                                                  wave_lds, mm, ll);
                if (split) {
                    float* p = partial_of(oc) + ts * split_step;
                    if (t < HD) st_agent(p + t, o_c * kWeightScale);
                    if (t == 0) {
                        st_agent(p + HD, mm);
                        st_agent(p + HD + 1, ll * kWeightScale);
                    }
                } else if (t < HD) {
                    a.out[((size_t)row * a.n_heads + head) * HD + t] = o_c * (ll > 0.0f ? 1.0f / ll : 0.0f);
                }
            }
        }
        if (split) {
            // this block's partials are performed at the coherence point before it counts itself.  A row counts on its
            // own counter; head h of a set on byte h % 4 of the counter of the set's first row, or second for h >= 4
            // (a set has two rows or more, and they count nothing of their own)
            const uint32_t rest = members & (members - 1);
            const int crow = solo ? r : tile0 + __builtin_ctz(h < 4 ? members : rest), shift = solo ? 0 : 8 * (h & 3);
            uint32_t* const counter = a.counters + crow * a.n_kv + kvh;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (t == 0)
                last = (__hip_atomic_fetch_add(counter, 1u << shift, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> shift & 255u) ==
                       (uint32_t)(nsp - 1);
            __syncthreads();
            if (!last) {
                if (solo) break;
                continue;
            }
            // split maxima and sums to LDS, then weights e^(m_k - M), then HD values per column, eight loads at a time
            const int n = nsp, cols = solo ? a.group : kCols;
            float* mk = reinterpret_cast<float*>(wave_lds);   // [column][n], then the weights
            float* lk = mk + cols * n;
            for (int i = t; i < cols * n; i += kThreads) {
                const int oc = i / n;
                if (!solo && !(members >> oc & 1)) continue;
                const float* p = partial_of(oc) + (size_t)(i - oc * n) * split_step + HD;
                mk[i] = ld_agent(p);
                lk[i] = ld_agent(p + 1);
            }
            __syncthreads();
            for (int oc = wave; oc < cols; oc += kWaves) {
                if (!solo && !(members >> oc & 1)) continue;
                float mm = -INFINITY, ll = 0.0f;
                for (int k = lane; k < n; k += 64) mm = fmaxf(mm, mk[oc * n + k]);
                mm = group_max<64>(mm);
                for (int k = lane; k < n; k += 64) {
                    const float ew = expf(mk[oc * n + k] - mm);
                    ll = ll + lk[oc * n + k] * ew;
                    mk[oc * n + k] = ew;
                }
                ll = group_sum<64>(ll);
                if (lane == 0) ml[0][0][oc] = ll;
            }
            __syncthreads();
            for (int i = t; i < cols * (HD / 2); i += kThreads) {
                const int oc = i / (HD / 2), d = 2 * (i % (HD / 2));
                if (!solo && !(members >> oc & 1)) continue;
                const float* p = partial_of(oc) + d;
                f2_t acc = {0.0f, 0.0f};
                for (int k = 0; k < n; k += 8) {
                    f2_t v[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = ld_agent2(p + (size_t)min(k + j, n - 1) * split_step);
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (k + j < n) acc = acc + v[j] * mk[oc * n + k + j];
                }
                const float ll = ml[0][0][oc];
                acc = acc * (ll > 0.0f ? 1.0f / ll : 0.0f);
                const int row = solo ? r : tile0 + oc, head = kvh * a.group + (solo ? oc : h);
                *reinterpret_cast<f2_t*>(a.out + ((size_t)row * a.n_heads + head) * HD + d) = acc;
            }
            if (t == 0) __hip_atomic_fetch_sub(counter, (uint32_t)n << shift, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (solo) break;
        __syncthreads();
    }
}

}  // namespace

hipError_t launch_attention_mma(const float* q, const uint16_t* kcache, const uint16_t* vcache,
                                const uint32_t* block_tables, int max_blocks, int total_blocks, const int32_t* pos,
                                int rows, int n_heads, int n_kv_heads, int head_dim, int n_layers, int tokens_per_block,
                                int layer, float scale, float soft_cap, int window, int max_splits, float* part,
                                uint32_t* counters, float* out, hipStream_t st)
{
    AttnArgs a{};
    a.q = q;
    a.kc = kcache;
    a.vc = vcache;
    a.pos = pos;
    a.bt = block_tables;
    a.max_blocks = max_blocks;
    a.total_blocks = total_blocks;
    a.n_layers = n_layers;
    a.tpb = tokens_per_block;
    a.tpb_shift = (tokens_per_block & (tokens_per_block - 1)) == 0 ? __builtin_ctz((unsigned)tokens_per_block) : -1;
    a.rows = rows;
    a.n_heads = n_heads;
    a.n_kv = n_kv_heads;
    a.group = n_heads / n_kv_heads;
    a.layer = layer;
    a.window = window;
    a.tiles = rows > 1 ? 1 : 0;
    a.scale = scale;
    a.soft_cap = soft_cap;
    const int cap = max_blocks * tokens_per_block;
    // at least 512 positions of the table per split (four chunks per wave), and no more splits than make 512
    // blocks: a split that has no work still reads positions and pages (4 rows of 15 / 5 heads over 2048 positions: 256 / 512 / 1024
    // per split 17.3 / 15.3 / 21.5 us; 8 rows of 32 / 8 heads of 128 over 8192: 512 / 768 / 1024 65 / 64 / 60 us;
    // a 2048-token prompt of 14 / 2 heads with four splits 186 us, with one 126)
    const int want = std::min(max_splits, std::max(1, 512 / (rows * n_kv_heads)));
    a.nsplit = std::min(want, (cap + 511) / 512);
    a.slots = (cap + 63) / 64;  // as attention_workspace_bytes counts them
    // Sets of all tiles' heads: 512 blocks, where the table or the window is long enough for splits.  A full tile's
    // set has a block for each of its units; a ragged last one has fewer blocks, which take several units each
    // where that is the shorter walk.  Where it is not the launch ends with that tile, and the others' splits only
    // cost: us, without / with them, 8/1 heads of 128, 300 rows at 2048 positions 44 / 48, 16/2, 200 rows at 3008
    // 60 / 67; without a ragged tile, 8/1, 400 rows at 4096, 78 / 66; 300 there 78, 89 with the last tile unsplit, 76 so.
    const int tiles = (rows + kCols - 1) / kCols, ragged = rows % kCols;
    const int span = window > 0 ? std::min(window + kCols, cap) : cap;
    a.tsplit = a.tsplit_last = 1;
    if (max_splits > 1 && span >= 4 * kMinTileSplit) {
        const int most = std::min({kMaxTileSplits, a.slots, std::max(1, 512 / (tiles * n_heads))});
        const int blocks = ragged * a.nsplit;
        // a block's walk, in positions: its units' own and what a unit takes besides (8 us of 4096 positions' 79 at
        // heads of 128, 12 with the adding of splits)
        const auto walk = [&](int n) { return (a.group * n + blocks - 1) / blocks * (span / n + (n > 1 ? 700 : 450)); };
        a.tsplit = std::min(most, std::max(1, kCols * a.nsplit / a.group));
        if (ragged >= std::max(a.group, 2)) {
            a.tsplit_last = std::min(most, blocks / a.group);
            for (int n = 2; n <= most && blocks < 2 * a.group; ++n)
                if (walk(n) < walk(a.tsplit_last)) a.tsplit_last = n;
            if (a.tsplit_last == 1) a.tsplit = 1;
        } else if (ragged > 0 && a.nsplit == 1) {
            a.tsplit = 1;  // its rows stay by themselves, unsplit
        }
    }
    a.busy = std::min(kCols, a.group * std::max(a.tsplit, a.tsplit_last));
    a.cap = cap;
    a.part = part;
    a.counters = counters;
    a.out = out;
    const dim3 grid((unsigned)(rows * n_kv_heads), (unsigned)a.nsplit);
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(kThreads), 0, st, a); };
    if (head_dim == 64) soft_cap > 0.0f ? go(attn_mma_kernel<64, true>) : go(attn_mma_kernel<64, false>);
    else soft_cap > 0.0f ? go(attn_mma_kernel<128, true>) : go(attn_mma_kernel<128, false>);
    return hipGetLastError();
}

}  // namespace cellm
