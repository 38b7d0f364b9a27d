// Rotary embedding and GQA tree attention over the prefix-trie rows.
//
// Reference: k_rope (src/tensor.cu:2180-2197) behind apply_rope_tree_gpu
// (src/tensor.cu:3342-3359), and k_attention_tree_gqa4 (src/tensor.cu:
// 2407-2633) behind attention_tree_gpu (src/tensor.cu:3361-3377).  A row is
// a trie node: its RoPE position is its depth and its keys are its ancestor
// chain (the last SLIDING_WINDOW of it), so attention runs on deduplicated
// rows without expanding them back to tokens.
//
// Arithmetic kept from the reference kernel, operation for operation, so the
// result is the reference's to the bit (up to the double exp below):
//   score of key w for query head g:
//     a_j = fma chain over d = j, j + 4, ... ascending (j < 4), +0 init
//     s_w = ((a_0 + a_1) + (a_2 + a_3)) * (1 / sqrtf(head_dim))
//   m = max_w s_w;  e_w = (float)exp((double)(s_w - m));
//   den = fp32 sum of e_w over w ascending (one lane per head);  p_w = e_w / den
//   out[d] = fma chain over w ascending of p_w * v[key w][d]
// exp is ROCm's double exp (the reference: CUDA's); both are within an ulp of
// double, so the float e_w agree except when a double lands within an ulp of
// a float rounding boundary.
//
// gfx950 mapping.  k_attention_group takes the rows four at a time on the
// matrix cores (its own comment has the mapping); k_attention_tree serves
// windows whose scores do not fit LDS that way, and unaligned arrays: one
// 256-thread workgroup per (row, KV head) serves the four query heads of the
// group, as in the reference.  Scores: a thread owns a key and reads its
// 128-float row as 16-byte vectors, one element per partial sum a_0..a_3
// (the four partials are exactly the four lanes of a float4), against the
// four query rows broadcast from LDS.  The order-critical denominator runs
// on four lanes (one per head) of one wave.  Values: a thread owns one
// dimension d of two heads and walks the keys in order, V rows read
// coalesced (128 threads = one 512-byte row).
#include "common.hpp"

namespace aps {
namespace {

constexpr int kHeadDim = 128;
constexpr int kGroup = 4;            // query heads per KV head (GQA-4)
constexpr int kAttnThreads = 256;

typedef float af4 __attribute__((ext_vector_type(4)));
typedef float af2 __attribute__((ext_vector_type(2)));

// q and k in one launch: a row holds q_heads + kv_heads heads of half / P
// runs of P pairs (j, j + half).  P = 4 (16-byte accesses) when the head
// dimension and the alignment allow, else 1.  Bound by the traffic (4.7 TB/s
// at 4,096 and more rows).  Measured, 43 / 4,096 / 10,240 rows: 5 / 16 / 35 us,
// against 10 / 24 / 56 us in two launches of one pair per thread.
template <int P>
__global__ void __launch_bounds__(256)
k_rope_tree(float* __restrict__ q, float* __restrict__ k, const uint32_t* __restrict__ row_pos, int64_t rows,
            int q_heads, int kv_heads, int half, const float* __restrict__ cosv, const float* __restrict__ sinv,
            int64_t max_seq) {
    typedef float rv_t __attribute__((ext_vector_type(P)));
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int runs = half / P, heads = q_heads + kv_heads;
    const int64_t rh = i / runs;   // row * heads + head
    const int64_t row = rh / heads;
    if (row >= rows) return;
    const int j = static_cast<int>(i - rh * runs) * P, head = static_cast<int>(rh - row * heads);
    const uint32_t pos = row_pos[row];
    if (pos >= max_seq) return;  // outside the table: left as is (the C++ layer checks positions)
    float* base = head < q_heads ? q + (row * q_heads + head) * (2 * half)
                                 : k + (row * kv_heads + (head - q_heads)) * (2 * half);
    const int64_t t = static_cast<int64_t>(pos) * half + j;
    auto ld = [](const float* p) { return *reinterpret_cast<const rv_t*>(p); };
    const rv_t c = ld(cosv + t), s = ld(sinv + t), x0 = ld(base + j), x1 = ld(base + j + half);
    rv_t o0, o1;
#pragma unroll
    for (int e = 0; e < P; ++e) {
        o0[e] = __fmaf_rn(x0[e], c[e], -__fmul_rn(x1[e], s[e]));
        o1[e] = __fmaf_rn(x1[e], c[e], __fmul_rn(x0[e], s[e]));
    }
    *reinterpret_cast<rv_t*>(base + j) = o0;
    *reinterpret_cast<rv_t*>(base + j + half) = o1;
}

// ---------------------------------------------------------------------------
// Row groups on the matrix cores.  Rows are taken 4 at a time (group g =
// rows 4g .. 4g+3); a group is worked off in runs of rows that lie on the
// ancestor chain of the run's last row (tree: anc[last][pos[r]] == r; packed:
// one sequence), so each row's keys are a contiguous range of that one chain.
// Most groups are one run; a trie branch or a sequence's end splits one.
constexpr int kGroupRows = 4;
constexpr int kGroupQueries = kGroupRows * kGroup;   // 16: query q = 4 row + head
constexpr int kKeyTile = 16;                         // keys per score tile / value group

// Bit 4 l + r: row r0 + r (r < l < nr) lies on the chain of row r0 + l.  pos:
// in lanes 4 l .. 4 l + 3 the position of row r0 + l.
template <bool PACKED>
__device__ inline uint32_t chain_pairs(const uint32_t* __restrict__ row_pos, const uint32_t* __restrict__ anc,
                                       int64_t anc_stride, int64_t r0, int nr, int lane, int& pos) {
    const int r = lane & 3, l = (lane >> 2) & 3;
    const uint32_t most = anc_stride < 0x7FFFFFFF ? static_cast<uint32_t>(anc_stride - 1) : 0x7FFFFFFEu;
    bool ok = false;
    pos = 0;
    if (lane < 16 && l < nr) {
        const int64_t row = r0 + r, last = r0 + l;
        uint32_t pr = r < l ? row_pos[row] : 0u, pl = row_pos[last];
        pr = pr < most ? pr : most;
        pl = pl < most ? pl : most;
        pos = static_cast<int>(pl);
        ok = r < l && pr <= pl && (PACKED ? anc[row] == anc[last] : anc[last * anc_stride + pr] == static_cast<uint32_t>(row));
    }
    return static_cast<uint32_t>(__ballot(ok));
}

typedef float ag4_t __attribute__((ext_vector_type(4)));

// Scores s[0 .. n) of one query -> probabilities: p = e / den in the window
// [l0, h0], 0 elsewhere; by the query's 16 threads (part: thread % 16), which
// are in one wave.
__device__ inline void window_softmax(float* srow, int l0, int h0, int n, float mq, int part) {
    // e = (float)exp((double)(s - m)) over the window, in place
    int w = l0 + part;
    for (; w + 48 <= h0; w += 64) {
        float x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = srow[w + 16 * u];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            srow[w + 16 * u] = static_cast<float>(exp(static_cast<double>(__fsub_rn(x[u], mq))));
    }
    for (; w <= h0; w += 16) srow[w] = static_cast<float>(exp(static_cast<double>(__fsub_rn(srow[w], mq))));
    // the denominator in key order on the query's first lane (the
    // wave's LDS accesses complete in program order), 16 reads ahead;
    // the wave barrier keeps the compiler from moving the other lanes'
    // stores past that lane's reads (they communicate through LDS)
    __builtin_amdgcn_wave_barrier();
    float den = 0.0f;
    if (part == 0) {
        int x = l0;
        for (; x + 16 <= h0 + 1; x += 16) {
            float e[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) e[u] = srow[x + u];
#pragma unroll
            for (int u = 0; u < 16; ++u) den = __fadd_rn(den, e[u]);
        }
        for (; x <= h0; ++x) den = __fadd_rn(den, srow[x]);
    }
    den = __shfl(den, static_cast<int>(threadIdx.x & 63) & ~15);
    // p = e / den in the window, 0 elsewhere over the tiles
    int x = part;
    for (; x + 48 < n; x += 64) {
        float e[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) e[u] = srow[x + 16 * u];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int xu = x + 16 * u;
            srow[xu] = (xu >= l0 && xu <= h0) ? __fdiv_rn(e[u], den) : 0.0f;
        }
    }
    for (; x < n; x += 16) srow[x] = (x >= l0 && x <= h0) ? __fdiv_rn(srow[x], den) : 0.0f;
}

// One row and KV head by one wave: the same arithmetic on the same MFMAs with
// the four heads' rows of the query operand repeated, so that lane l ends with
// head l / 16.  Keys in blocks of 64, a lane per key's row offset, read a block
// ahead and passed on by shuffles; K goes two tiles ahead into the registers a
// tile has used up, V two groups of 16 keys.  sc: this wave's 4 score rows.
// LDS is the wave's own: no workgroup barrier.
template <bool PACKED>
__device__ inline void attend_row(const float* __restrict__ q, const float* __restrict__ k,
                                  const float* __restrict__ v, float* __restrict__ out,
                                  const uint32_t* __restrict__ anc, int64_t anc_stride, int64_t rows, int q_heads,
                                  int kv_heads, int wmax, float scale, float* sc, int sw, int kh, int64_t row,
                                  int64_t pos) {
    const int lane = threadIdx.x & 63, qq = lane & 15, qj = lane >> 4;
    const int64_t begin = pos + 1 > wmax ? pos + 1 - wmax : 0;
    const int W = static_cast<int>(pos - begin + 1);
    const int ntiles = (W + kKeyTile - 1) / kKeyTile;
    const uint32_t kvs_bytes = static_cast<uint32_t>(kv_heads) * kHeadDim * sizeof(float);
    const int64_t first = (PACKED ? static_cast<int64_t>(anc[row]) : row * anc_stride) + begin;
    // byte offset of key w's K / V row (past the window: the last key's)
    auto key = [&](int w) __attribute__((always_inline)) {
        w = w < W ? w : W - 1;
        const int64_t a = PACKED ? first + w : static_cast<int64_t>(anc[first + w]);
        return static_cast<uint32_t>(a < rows ? a : rows - 1) * kvs_bytes;
    };
    auto pick = [&](const ag4_t& x) { return qj == 0 ? x[0] : qj == 1 ? x[1] : qj == 2 ? x[2] : x[3]; };
    float* const srow = sc + qj * sw;   // this lane's head

    // ---- scores ----
    const af4* qsrc =
        reinterpret_cast<const af4*>(q + (row * q_heads + kh * kGroup + qq % kGroup) * kHeadDim + 4 * qj);
    af4 qv[8];
#pragma unroll
    for (int a = 0; a < 8; ++a) qv[a] = qsrc[4 * a];
    float m = -3.402823466e+38f;
    {
        const char* const kbase = reinterpret_cast<const char*>(k + kh * kHeadDim) + 16 * qj;
        uint32_t cur = key(lane), next = key(kWave + lane);
        auto ksrc = [&](uint32_t block, int t) __attribute__((always_inline)) {
            return reinterpret_cast<const af4*>(kbase + __shfl(block, 16 * t + qq));
        };
        af4 kb[2][8];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const af4* src = ksrc(cur, t);
#pragma unroll
            for (int a = 0; a < 8; ++a) kb[t][a] = src[4 * a];
            __builtin_amdgcn_sched_barrier(0);
        }
        for (int t0 = 0; t0 < ntiles; t0 += 4) {
            const uint32_t after = key(16 * t0 + 2 * kWave + lane);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t0 + t >= ntiles) break;   // wave-uniform
                const af4* src = ksrc(t < 2 ? cur : next, (t + 2) & 3);
                ag4_t acc[4] = {};
#pragma unroll
                for (int a = 0; a < 8; ++a) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[a][j], kb[t & 1][a][j], acc[j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    kb[t & 1][a] = src[4 * a];
                    __builtin_amdgcn_sched_barrier(0);
                }
                const int w = 16 * (t0 + t) + qq;
                const float s = __fmul_rn(__fadd_rn(__fadd_rn(pick(acc[0]), pick(acc[1])),
                                                    __fadd_rn(pick(acc[2]), pick(acc[3]))), scale);
                srow[w] = s;
                if (w < W) m = fmaxf(m, s);
            }
            cur = next;
            next = after;
        }
    }
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    __builtin_amdgcn_wave_barrier();   // (the wave's LDS accesses complete in order)

    // ---- softmax and values, the first 32 keys' loads under the softmax ----
    const char* const vbase = reinterpret_cast<const char*>(v + kh * kHeadDim) + 32 * qq;   // this lane's 8 dimensions
    uint32_t cur = key(lane), next = key(kWave + lane);
    af4 vb[2][4][2];
    auto vload = [&](af4 (&d)[4][2], uint32_t block, int g) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const af4* src = reinterpret_cast<const af4*>(vbase + __shfl(block, 16 * g + 4 * u + qj));
            d[u][0] = src[0];
            d[u][1] = src[1];
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    vload(vb[0], cur, 0);
    vload(vb[1], cur, 1);
    window_softmax(srow, 0, W - 1, ntiles * kKeyTile, m, qq);
    __builtin_amdgcn_wave_barrier();
    const float* const prow = sc + (qq % kGroup) * sw + qj;   // A: query lane % 16, key lane / 16 of a step
    ag4_t o[8] = {};   // register t of o[i]: head t, dimension 8 (lane % 16) + i
    for (int g0 = 0; g0 < ntiles; g0 += 4) {
        const uint32_t after = key(16 * g0 + 2 * kWave + lane);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (g0 + g >= ntiles) break;   // wave-uniform
            const int w0 = 16 * (g0 + g);
            af4 (&d)[4][2] = vb[g & 1];
            float pa[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) pa[u] = prow[w0 + 4 * u];
            if (w0 + 16 > W) {   // the last tile's padding: no value at all
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (w0 + 4 * u + qj >= W) d[u][0] = d[u][1] = af4{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    o[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[u], d[u][i / 4][i % 4], o[i], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            vload(d, g < 2 ? cur : next, (g + 2) & 3);
        }
        cur = next;
        next = after;
    }
    float* const dst = out + (row * q_heads + kh * kGroup + qj) * kHeadDim + 8 * qq;   // 8-byte aligned
#pragma unroll
    for (int i = 0; i < 8; i += 2) *reinterpret_cast<af2*>(dst + i) = af2{pick(o[i]), pick(o[i + 1])};
}

// One workgroup = one row group x one KV head.  Per run of rows: 16 queries
// (up to 4 rows x the KV head's 4 query heads) against the keys chain[dlo ..
// dhi] of the run's last row; row r attends to chain[begin_r .. pos_r].  The arithmetic is the
// row kernel's, operation for operation:
//   scores on v_mfma_f32_16x16x4_f32, whose products join the accumulator one
//     after the other (chain_mfma.hpp): one accumulator per partial chain a_j
//     over d = j, j + 4, .., 16 queries x 16 keys; then s = ((a0 + a1) + (a2 +
//     a3)) * scale in registers, into LDS;
//   per query over its window: m = max s, e = (float)exp((double)(s - m)),
//     den = sum of e in key order (one lane per query), p = e / den;
//   out[d] = chain over keys of p v[d] on the same MFMA, 16 queries x 16
//     dimensions, four keys a step.
// Every score is computed once: the run's 16 x window scores sit in LDS.
// Keys after a row's window take p = 0, which leaves its value chains
// unchanged except that a -0 would turn +0; keys before it keep the chain
// at its +0 start; the last tile's padding has p = 0 and v = 0.  Infinite and
// NaN values of a key outside a row's window would turn its output NaN
// (0 * inf): a wave with a NaN output in a run of several rows does its
// dimensions again row by row, each row on its own keys alone.
//   K and V go from global memory straight to registers (LDS holds only the
// scores and the chain's key rows, so two workgroups fit a CU at 1,024-key
// windows, and three at key spans up to 784).  Scores: wave w takes the
// 16-key tiles w, w + 4, ..; a lane (key lane % 16, k slot lane / 16) loads 16
// bytes, elements 16 a + 4 (lane / 16) .. + 3 for a < 8, which are the operands of
// the four partial chains at one step: no lane transposes.  The tile two
// ahead goes into the registers a step has used up.  Softmax: the 16 threads
// of query q are in wave q / 4, so exp, the ordered denominator and p = e /
// den need no workgroup barrier.  Values: wave w takes dimensions 32 w .. 32 w
// + 31, two per lane, one 8-byte load per four keys, 64 keys ahead; the K / V
// row offsets are 32-bit byte offsets off a uniform base.
//   Bound by the fp32 MFMAs with the vector work that cannot run beside them
// (exp, division, addresses).  Measured, 4,096 rows of 512-token prompts: 249
// us -> 177; 10,240 rows, 16 prompts of 1,024 with shared halves: 1345 -> 1016,
// against the K = 1 MFMA with its operands transposed across lanes and the
// values on two of the four waves.  Serving every group here instead of
// leaving branching groups to a second launch over all rows saves that launch:
// 9.7 and 22 us, and 14 -> 8 us for 43 rows.  Groups that branch much go row by
// row (attend_row): 4,096 single-token prompts 68 us in two launches, 150 run by
// run, 56 row by row; 4,096 leaves of a 1,000-token prompt 1650, 1990, 1430, of
// a 100-token prompt 207, 328, 222.
template <bool PACKED>
__global__ void __launch_bounds__(256, 3)
k_attention_group(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                  float* __restrict__ out, const uint32_t* __restrict__ row_pos, const uint32_t* __restrict__ anc,
                  int64_t anc_stride, int64_t rows, int q_heads, int kv_heads, int wmax, float scale, int sw) {
    extern __shared__ __align__(16) float gdyn[];
    float* sc = gdyn;                                                     // [16 queries][sw]: s, then e
    uint32_t* chain = reinterpret_cast<uint32_t*>(sc + kGroupQueries * sw);   // [sw - 1] key rows
    __shared__ int qlo[kGroupQueries], qhi[kGroupQueries];   // window of each query, relative to dlo
    __shared__ float wmx[4][kGroupQueries];                  // per-wave maxima

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // groups in reverse row order: later rows (longer chains in trie and
    // packed order) start first, so the short ones fill the last round
    const int64_t g0 = static_cast<int64_t>(gridDim.x / kv_heads - 1 - blockIdx.x / kv_heads) * kGroupRows;
    const int kh = static_cast<int>(blockIdx.x % kv_heads);
    const int gn = static_cast<int>(rows - g0 < kGroupRows ? rows - g0 : kGroupRows);
    int group_pos;
    const uint32_t pairs = __builtin_amdgcn_readfirstlane(
        chain_pairs<PACKED>(row_pos, anc, anc_stride, g0, gn, threadIdx.x & 63, group_pos));
    // of the group's row i (32 bits: scalar compares)
    auto pos_of = [&](int i) { return __builtin_amdgcn_readlane(group_pos, 4 * i); };
    // the longest run from row i0 whose key range, from its first row's
    // window on, fits the LDS (sw - 1 keys: a single row always does)
    auto run_rows = [&](int i0) __attribute__((always_inline)) {
        const int p0 = pos_of(i0);
        int nr = gn - i0;
        for (; nr > 1; --nr) {
            const int l = i0 + nr - 1;
            const uint32_t need = ((1u << nr) - 1u) >> 1 << i0;   // rows i0 .. l - 1
            bool fits = ((pairs >> (4 * l)) & need) == need &&
                        pos_of(l) - (p0 + 1 > wmax ? p0 + 1 - wmax : 0) + 1 <= sw - 1;
            for (int r = 1; r + 1 < nr; ++r) fits = fits && pos_of(i0 + r) >= p0;
            if (fits) break;
        }
        return nr;
    };
    int runs = 0;
    uint32_t run_at = 0;   // 4 bits per row: the rows of the run that starts there
    int longest = 0;
    for (int i0 = 0; i0 < gn; ++runs) {
        const int nr = run_rows(i0);
        run_at |= static_cast<uint32_t>(nr) << (4 * i0);
        i0 += nr;
        const int p = pos_of(i0 - 1);
        longest = p > longest ? p : longest;
    }
    // Rows of several runs one per wave: always with four runs, with fewer while
    // the windows are short and the runs' latencies, one after the other,
    // weigh more than the repeated query rows.  us by run -> by row at windows of
    // 33 / 101 / 201 / 501 keys, leaves of a shared prompt: four runs (512 rows)
    // 33 -> 20, 53 -> 35, 79 -> 57, 152 -> 121; three 33 -> 27, 53 -> 51, 82 -> 83,
    // 160 -> 180; two 34 -> 34, 54 -> 64, 80 -> 108, 152 -> 241.
    const int window = longest + 1 < wmax ? longest + 1 : wmax;
    const bool by_row = runs == 4 || (runs == 3 && window <= 160) || (runs == 2 && window <= 32);
    for (int i0 = 0, nr; !by_row && i0 < gn;) {
    const int64_t r0 = g0 + i0;
    // (opaque per run: addresses hoisted out of the loop cost spills)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    nr = (run_at >> (4 * i0)) & 15;
    const int64_t last = r0 + nr - 1;
    const int p0 = pos_of(i0);
    const int dlo = p0 + 1 > wmax ? p0 + 1 - wmax : 0;
    const int dhi = pos_of(i0 + nr - 1);
    const int W = dhi - dlo + 1;
    const int ntiles = (W + kKeyTile - 1) / kKeyTile;   // 16-key tiles (at most capacity / 16)
    const int64_t seg = PACKED ? static_cast<int64_t>(anc[last]) : 0;
    if (tid < kGroupQueries) {
        const int r = tid / kGroup;
        int pr = p0;
#pragma unroll
        for (int i = 1; i < kGroupRows; ++i)
            if (r == i) pr = pos_of(i0 + i);
        if (r < nr) {
            qhi[tid] = pr - dlo;
            qlo[tid] = (pr + 1 > wmax ? pr + 1 - wmax : 0) - dlo;
        } else {
            qhi[tid] = -1;   // a padding row: an empty window
            qlo[tid] = 0;
        }
    }
    // q operand: lane l -> query l % 16 (row (l % 16) / 4, head (l % 16) % 4),
    // elements 16 a + 4 (l / 16) .. + 3, one per partial chain (loads in
    // flight during the staging)
    const int qq = lane & 15, qj = lane >> 4;
    const int qrow = qq / kGroup;
    const int64_t qr = r0 + (qrow < nr ? qrow : nr - 1);
    const af4* qsrc = reinterpret_cast<const af4*>(q + (qr * q_heads + kh * kGroup + qq % kGroup) * kHeadDim + 4 * qj);
    af4 qv[8];
#pragma unroll
    for (int a = 0; a < 8; ++a) qv[a] = qsrc[4 * a];
    // the chain's key rows (clamped to the chain and the rows) in LDS, as
    // byte offsets of the key's K / V row (below 2^32: the launcher's check)
    const uint32_t kvs_bytes = static_cast<uint32_t>(kv_heads) * kHeadDim * sizeof(float);
    for (int i = tid; i < ntiles * 16; i += 256) {
        const int d = dlo + i < dhi ? dlo + i : dhi;
        const int64_t a = PACKED ? seg + d : static_cast<int64_t>(anc[last * anc_stride + d]);
        chain[i] = static_cast<uint32_t>(a < rows ? a : rows - 1) * kvs_bytes;
    }
    __syncthreads();
    // this lane's four score queries 4 qj + t: windows
    int lo[4], hi[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        lo[t] = qlo[4 * qj + t];
        hi[t] = qhi[4 * qj + t];
    }

    // ---- scores: tiles wave, wave + 4, .. ----
    const char* const kbase = reinterpret_cast<const char*>(k + kh * kHeadDim);
    auto ksrc = [&](int t) __attribute__((always_inline)) {
        return reinterpret_cast<const af4*>(kbase + (chain[16 * t + qq] + 16u * qj));
    };
    float m[4] = {-3.402823466e+38f, -3.402823466e+38f, -3.402823466e+38f, -3.402823466e+38f};
    // the loads of every step are unconditional (a step past the end reloads
    // the last tile): the compiler's wait counts then leave the other
    // buffer's loads in flight
    auto tclamp = [&](int t) { return t < ntiles ? t : ntiles - 1; };
    auto tile = [&](int t, af4* buf) __attribute__((always_inline)) {
        const af4* next = ksrc(tclamp(t + 8));
        ag4_t acc[4] = {};   // partial chain j
#pragma unroll
        for (int a = 0; a < 8; ++a) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[a][j], buf[a][j], acc[j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            buf[a] = next[4 * a];   // this wave's tile two ahead into the freed registers
            __builtin_amdgcn_sched_barrier(0);
        }
        // register u of chain j: partial j of query 4 qj + u, key lane % 16
        const int w = 16 * t + qq;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float sx = __fmul_rn(__fadd_rn(__fadd_rn(acc[0][u], acc[1][u]), __fadd_rn(acc[2][u], acc[3][u])), scale);
            sc[(4 * qj + u) * sw + w] = sx;
            if (w >= lo[u] && w <= hi[u]) m[u] = fmaxf(m[u], sx);
        }
    };
    if (wave < ntiles) {
        af4 kb0[8], kb1[8];
        const af4* s0 = ksrc(wave);
        const af4* s1 = ksrc(tclamp(wave + 4));
#pragma unroll
        for (int a = 0; a < 8; ++a) kb0[a] = s0[4 * a];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int a = 0; a < 8; ++a) kb1[a] = s1[4 * a];
        __builtin_amdgcn_sched_barrier(0);
        int t = wave;
        for (; t + 4 < ntiles; t += 8) {
            tile(t, kb0);
            tile(t + 4, kb1);
        }
        if (t < ntiles) tile(t, kb0);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int o = 8; o >= 1; o >>= 1) m[u] = fmaxf(m[u], __shfl_xor(m[u], o));
        if (qq == 0) wmx[wave][4 * qj + u] = m[u];
    }
    __syncthreads();

    // ---- softmax, per query on the 16 threads of one wave (queries
    // 4 w .. 4 w + 3 on wave w), so it needs no workgroup barrier ----
    const int qi = tid / 16, part = tid % 16;
    const char* const vbase = reinterpret_cast<const char*>(v + kh * kHeadDim);   // uniform: 32-bit lane offsets
    const uint32_t dbytes = static_cast<uint32_t>(32 * wave + 2 * qq) * sizeof(float);   // this lane's two dimensions
    auto vload = [&](int g, af2* vb) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            vb[u] = *reinterpret_cast<const af2*>(vbase + (chain[16 * g + 4 * u + qj] + dbytes));
    };
    af2 vb0[4], vb1[4], vb2[4], vb3[4];
    auto gclamp = [&](int g) { return g < ntiles ? g : ntiles - 1; };
    vload(0, vb0);   // the first 64 keys' values go out now
    vload(gclamp(1), vb1);
    vload(gclamp(2), vb2);
    vload(gclamp(3), vb3);
    {
        const float mq = fmaxf(fmaxf(wmx[0][qi], wmx[1][qi]), fmaxf(wmx[2][qi], wmx[3][qi]));
        window_softmax(sc + qi * sw, qlo[qi], qhi[qi], ntiles * kKeyTile, mq, part);
    }
    __syncthreads();

    // ---- values: out[q][d] = chain over keys of p v[d] ----
    ag4_t o[2] = {};   // register t of o[i]: query 4 (lane / 16) + t, dimension 32 wave + 2 (lane % 16) + i
    {
        const float* prow = sc + qq * sw + qj;   // A: query lane % 16, key lane / 16 of a step
        float pa[2][4];
        auto pload = [&](int g, float* p) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < 4; ++u) p[u] = prow[16 * g + 4 * u];
        };
        auto group = [&](int g, af2* vb, int s) __attribute__((always_inline)) {
            pload(gclamp(g + 1), pa[s ^ 1]);
            if (g < ntiles) {   // wave-uniform
                if (16 * g + 16 > W) {   // the last tile's padding: no value at all
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (16 * g + 4 * u + qj >= W) vb[u] = af2{0.0f, 0.0f};
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        o[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa[s][u], vb[u][i], o[i], 0, 0, 0);
            }
            vload(gclamp(g + 4), vb);   // unconditional, as for the scores
        };
        pload(0, pa[0]);
        for (int g = 0; g < ntiles; g += 4) {
            group(g, vb0, 0);
            group(g + 1, vb1, 1);
            group(g + 2, vb2, 0);
            group(g + 3, vb3, 1);
        }
    }
    // (lane group qj holds row qj's four heads)
    bool nan = false;
#pragma unroll
    for (int t = 0; t < 4; ++t) nan = nan || o[0][t] != o[0][t] || o[1][t] != o[1][t];
    if (nr > 1 && __ballot(nan && qj < nr) != 0) {   // wave-uniform: this wave's dimensions again, row by row
        for (int r = 0; r < nr; ++r) {
            const int l0 = qlo[kGroup * r], h0 = qhi[kGroup * r];
            ag4_t own[2] = {};
            for (int g = l0 / kKeyTile; g <= h0 / kKeyTile; ++g) {
                vload(g, vb0);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int w = 16 * g + 4 * u + qj;
                    if (w < l0 || w > h0) vb0[u] = af2{0.0f, 0.0f};
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        own[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(sc[qq * sw + w], vb0[u][i], own[i], 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
                if (qj == r) o[i] = own[i];
        }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)   // head t
        if (qj < nr)
            *reinterpret_cast<af2*>(out + ((r0 + qj) * q_heads + kh * kGroup + t) * kHeadDim + 32 * wave + 2 * qq) =
                af2{o[0][t], o[1][t]};
    __syncthreads();   // the next run writes the chain and the scores
    i0 += nr;
    }
    if (by_row && wave < gn)   // wave-uniform
        attend_row<PACKED>(q, k, v, out, anc, anc_stride, rows, q_heads, kv_heads, wmax, scale,
                           sc + wave * kGroup * sw, sw, kh, g0 + wave, pos_of(wave));
}

// Dynamic LDS: scores [wmax][4] fp32, then chain [wmax] u32.
// PACKED: the rows are packed token sequences (reference k_attention_grouped_gqa4,
// src/tensor.cu:2267-2405, which the tree kernel restates with an index
// indirection): `anc` holds each row's segment start seg_offset[row], the
// keys of a row are the contiguous rows seg_offset + begin .. seg_offset +
// pos, and anc_stride is the longest segment.  Otherwise the keys are the
// ancestor chain anc[row][begin .. pos] of a trie node.
template <bool PACKED>
__global__ void __launch_bounds__(kAttnThreads)
k_attention_tree(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                 float* __restrict__ out, const uint32_t* __restrict__ row_pos, const uint32_t* __restrict__ anc,
                 int64_t anc_stride, int64_t rows, int q_heads, int kv_heads, int wmax, float scale) {
    extern __shared__ __align__(16) float dyn[];
    float* sc = dyn;                                                  // [w][g]
    uint32_t* chain = reinterpret_cast<uint32_t*>(dyn + static_cast<int64_t>(wmax) * kGroup);
    __shared__ __align__(16) float qs[kHeadDim][kGroup];              // [d][g]
    __shared__ float red[kAttnThreads / kWave][kGroup];
    __shared__ float stat[2][kGroup];                                 // max, denominator
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row = blockIdx.x / kv_heads;
    const int kh = static_cast<int>(blockIdx.x % kv_heads);
    // Positions past the ancestor table and key rows past the end are
    // clamped, for memory safety only: the C++ layer checks them (through
    // RowIndexBuffer::max_row and the packed segment table), and direct
    // C-ABI callers must keep them in range.
    int64_t pos = row_pos[row];
    pos = pos < anc_stride ? pos : anc_stride - 1;
    const int64_t begin = pos + 1 > wmax ? pos + 1 - wmax : 0;
    const int window = static_cast<int>(pos - begin + 1);
    const int64_t seg = PACKED ? static_cast<int64_t>(anc[row]) : 0;
    for (int i = tid; i < window; i += kAttnThreads) {
        const int64_t a = PACKED ? seg + begin + i : static_cast<int64_t>(anc[row * anc_stride + begin + i]);
        chain[i] = static_cast<uint32_t>(a < rows ? a : rows - 1);
    }
    for (int i = tid; i < kGroup * kHeadDim; i += kAttnThreads) {
        const int g = i / kHeadDim, d = i % kHeadDim;
        qs[d][g] = q[(row * q_heads + kh * kGroup + g) * kHeadDim + d];
    }
    __syncthreads();

    // ---- scores and the per-head maximum ----
    float mx[kGroup];
#pragma unroll
    for (int g = 0; g < kGroup; ++g) mx[g] = -3.402823466e+38f;
    for (int w = tid; w < window; w += kAttnThreads) {
        const af4* kr = reinterpret_cast<const af4*>(k + (static_cast<int64_t>(chain[w]) * kv_heads + kh) * kHeadDim);
        float a[kGroup][4];
#pragma unroll
        for (int g = 0; g < kGroup; ++g) a[g][0] = a[g][1] = a[g][2] = a[g][3] = 0.0f;
#pragma unroll 4
        for (int i = 0; i < kHeadDim / 4; ++i) {
            const af4 kv = kr[i];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const af4 qv = *reinterpret_cast<const af4*>(&qs[4 * i + j][0]);  // the four heads at d = 4i + j
                a[0][j] = __fmaf_rn(qv[0], kv[j], a[0][j]);
                a[1][j] = __fmaf_rn(qv[1], kv[j], a[1][j]);
                a[2][j] = __fmaf_rn(qv[2], kv[j], a[2][j]);
                a[3][j] = __fmaf_rn(qv[3], kv[j], a[3][j]);
            }
        }
        af4 s;
#pragma unroll
        for (int g = 0; g < kGroup; ++g) {
            s[g] = __fmul_rn(__fadd_rn(__fadd_rn(a[g][0], a[g][1]), __fadd_rn(a[g][2], a[g][3])), scale);
            mx[g] = fmaxf(mx[g], s[g]);
        }
        *reinterpret_cast<af4*>(sc + 4 * w) = s;
    }
#pragma unroll
    for (int g = 0; g < kGroup; ++g) {
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) mx[g] = fmaxf(mx[g], __shfl_xor(mx[g], o));
        if (lane == 0) red[wave][g] = mx[g];
    }
    __syncthreads();
    if (tid < kGroup) {
        float m = red[0][tid];
#pragma unroll
        for (int w = 1; w < kAttnThreads / kWave; ++w) m = fmaxf(m, red[w][tid]);
        stat[0][tid] = m;
    }
    __syncthreads();

    // ---- exponentials (elementwise: any thread), then the ordered denominator ----
    for (int i = tid; i < window * kGroup; i += kAttnThreads)
        sc[i] = static_cast<float>(exp(static_cast<double>(__fsub_rn(sc[i], stat[0][i & 3]))));
    __syncthreads();
    if (tid < kGroup) {
        float den = 0.0f;
        int w = 0;
        for (; w + 8 <= window; w += 8) {
            float e[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) e[u] = sc[4 * (w + u) + tid];
#pragma unroll
            for (int u = 0; u < 8; ++u) den = __fadd_rn(den, e[u]);
        }
        for (; w < window; ++w) den = __fadd_rn(den, sc[4 * w + tid]);
        stat[1][tid] = den;
    }
    __syncthreads();
    for (int i = tid; i < window * kGroup; i += kAttnThreads) sc[i] = __fdiv_rn(sc[i], stat[1][i & 3]);
    __syncthreads();

    // ---- values: thread = (dimension d, head pair), keys in order ----
    const int d = tid & (kHeadDim - 1);
    const int g0 = 2 * (tid >> 7);
    const float* vcol = v + static_cast<int64_t>(kh) * kHeadDim + d;
    const int64_t vstride = static_cast<int64_t>(kv_heads) * kHeadDim;
    float o0 = 0.0f, o1 = 0.0f;
    int w = 0;
    for (; w + 8 <= window; w += 8) {
        float vv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) vv[u] = vcol[static_cast<int64_t>(chain[w + u]) * vstride];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            o0 = __fmaf_rn(sc[4 * (w + u) + g0], vv[u], o0);
            o1 = __fmaf_rn(sc[4 * (w + u) + g0 + 1], vv[u], o1);
        }
    }
    for (; w < window; ++w) {
        const float vv = vcol[static_cast<int64_t>(chain[w]) * vstride];
        o0 = __fmaf_rn(sc[4 * w + g0], vv, o0);
        o1 = __fmaf_rn(sc[4 * w + g0 + 1], vv, o1);
    }
    float* orow = out + (row * q_heads + kh * kGroup + g0) * kHeadDim + d;
    orow[0] = o0;
    orow[kHeadDim] = o1;
}

// Packed-sequence attention for head layouts other than GQA-4 (reference
// k_attention, src/tensor.cu:2209-2274, launched by attention_gpu,
// :3316-3340, when q_heads != 4 kv_heads).  One 128-thread workgroup per
// (row, query head); the arithmetic is the reference kernel's:
//   s_w = (fma chain over d ascending of q[d] k_w[d], from +0) * scale
//   m = max_w s_w;  e_w = (float)exp((double)(s_w - m));
//   den = fp32 sum of e_w, w ascending (one lane);  p_w = e_w / den
//   out[d] = fma chain over w ascending of p_w v_w[d]
// The scores and exps of different keys are independent, so threads take
// keys w = tid, tid + 128, ...; only the denominator is a serial sum.  Keys
// are the rows seg_offset[row] + begin .. seg_offset[row] + pos of the row's
// own sequence, begin = max(0, pos + 1 - window).  Dynamic LDS: wmax scores.
constexpr int kAnyThreads = 128;

__global__ void __launch_bounds__(kAnyThreads)
k_attention_any(const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
                float* __restrict__ out, const uint32_t* __restrict__ seg_offset, const uint32_t* __restrict__ seg_pos,
                int64_t rows, int q_heads, int kv_heads, int head_dim, int64_t max_seq, int wmax, float scale) {
    extern __shared__ float sc[];
    __shared__ float qs[kAnyThreads];
    __shared__ float red[kAnyThreads / kWave];
    __shared__ float den_s;
    const int tid = threadIdx.x;
    const int64_t task = blockIdx.x;
    const int64_t row = task / q_heads;
    const int qh = static_cast<int>(task % q_heads);
    const int kh = qh / (q_heads / kv_heads);
    // positions and segment starts clamped for memory safety only (the C++
    // layer builds them from the sequence lengths)
    int64_t pos = seg_pos[row];
    pos = pos < max_seq ? pos : max_seq - 1;
    const int64_t begin = pos + 1 > wmax ? pos + 1 - wmax : 0;
    const int window = static_cast<int>(pos - begin + 1);
    const int64_t first = static_cast<int64_t>(seg_offset[row]) + begin;
    auto key_row = [&](int w) {
        const int64_t r = first + w;
        return r < rows ? r : rows - 1;
    };
    const float* qrow = q + (row * q_heads + qh) * static_cast<int64_t>(head_dim);
    if (tid < head_dim) qs[tid] = qrow[tid];
    __syncthreads();
    float m = -3.402823466e+38F;
    for (int w = tid; w < window; w += kAnyThreads) {
        const float* kr = k + (key_row(w) * kv_heads + kh) * static_cast<int64_t>(head_dim);
        float a = 0.0f;
        for (int d = 0; d < head_dim; ++d) a = __fmaf_rn(qs[d], kr[d], a);
        const float sw = __fmul_rn(a, scale);
        sc[w] = sw;
        m = fmaxf(m, sw);
    }
    // the window's maximum (order-independent)
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    m = fmaxf(red[0], red[1]);
    for (int w = tid; w < window; w += kAnyThreads)
        sc[w] = static_cast<float>(exp(static_cast<double>(__fsub_rn(sc[w], m))));
    __syncthreads();
    if (tid == 0) {
        float den = 0.0f;
        for (int w = 0; w < window; ++w) den = __fadd_rn(den, sc[w]);
        den_s = den;
    }
    __syncthreads();
    const float den = den_s;
    for (int w = tid; w < window; w += kAnyThreads) sc[w] = __fdiv_rn(sc[w], den);
    __syncthreads();
    if (tid < head_dim) {
        float o = 0.0f;
        for (int w = 0; w < window; ++w)
            o = __fmaf_rn(sc[w], v[(key_row(w) * kv_heads + kh) * static_cast<int64_t>(head_dim) + tid], o);
        out[(row * q_heads + qh) * static_cast<int64_t>(head_dim) + tid] = o;
    }
}

}  // namespace

hipError_t launch_rope_tree(float* q, float* k, const uint32_t* row_pos, int64_t rows, int q_heads, int kv_heads,
                            int head_dim, const float* cosv, const float* sinv, int64_t max_seq, hipStream_t s) {
    const int half = head_dim / 2;
    if (kv_heads > 0 && q < k + rows * kv_heads * head_dim && k < q + rows * q_heads * head_dim) {
        const hipError_t e = launch_rope_tree(q, q, row_pos, rows, q_heads, 0, head_dim, cosv, sinv, max_seq, s);
        return e != hipSuccess
                   ? e
                   : launch_rope_tree(k, k, row_pos, rows, kv_heads, 0, head_dim, cosv, sinv, max_seq, s);
    }
    const uintptr_t addr = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                           reinterpret_cast<uintptr_t>(cosv) | reinterpret_cast<uintptr_t>(sinv);
    const bool vec = half % 4 == 0 && (addr & 15u) == 0;
    // (a launch of 2^32 threads or more would drop the rest without an error)
    const int64_t per_row = static_cast<int64_t>(q_heads + kv_heads) * (vec ? half / 4 : half);
    const int64_t most = (int64_t(1) << 31) / per_row > 0 ? (int64_t(1) << 31) / per_row : 1;
    for (int64_t r0 = 0; r0 < rows; r0 += most) {
        const int64_t nr = rows - r0 < most ? rows - r0 : most;
        hipLaunchKernelGGL(vec ? k_rope_tree<4> : k_rope_tree<1>,
                           dim3(static_cast<unsigned>(ceil_div(nr * per_row, 256))), dim3(256), 0, s,
                           q + r0 * q_heads * head_dim, k + r0 * kv_heads * head_dim, row_pos + r0, nr, q_heads,
                           kv_heads, half, cosv, sinv, max_seq);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_attention_tree(const float* q, const float* k, const float* v, float* out, const uint32_t* row_pos,
                                 const uint32_t* anc, int64_t anc_stride, int64_t rows, int q_heads, int kv_heads,
                                 int head_dim, int window_max, bool packed, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (head_dim != kHeadDim || q_heads != kGroup * kv_heads || anc_stride <= 0 || window_max <= 0)
        return hipErrorInvalidValue;
    const int64_t keys = anc_stride < window_max ? anc_stride : window_max;
    if (keys > kAttnMaxWindow) return hipErrorInvalidValue;
    const int wmax = static_cast<int>(keys);
    // 1 / sqrtf(head_dim), both correctly rounded, as the reference kernel computes it
    const float root = sqrtf(static_cast<float>(head_dim));
    const float scale = 1.0f / root;
    // path groups on the matrix cores when their scores fit in LDS (16
    // queries x the group's key range), q, k, v are 16-byte and out 8-byte
    // aligned; the rest per row
    const int64_t span = ceil_div(keys + kGroupRows - 1, kKeyTile) * kKeyTile;
    const int sw = static_cast<int>(span) | 1;   // odd row stride: 16 queries, 16 bank groups
    const size_t glds = static_cast<size_t>(kGroupQueries + 1) * sw * sizeof(float);
    const bool group = glds <= 150 * 1024 && rows * kv_heads * kHeadDim * static_cast<int64_t>(sizeof(float)) <= 0xFFFFFFFFll &&
                       ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                         reinterpret_cast<uintptr_t>(v)) & 15u) == 0 &&
                       (reinterpret_cast<uintptr_t>(out) & 7u) == 0;
    if (group) {
        // (splitting one launch into a long- and a short-range launch lost
        // more to the first one's tail than the short ranges gained)
        auto gk = packed ? &k_attention_group<true> : &k_attention_group<false>;
        if (glds > 65536) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gk),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(glds));
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(gk, dim3(static_cast<unsigned>(ceil_div(rows, kGroupRows) * kv_heads)), dim3(256), glds, s,
                           q, k, v, out, row_pos, anc, anc_stride, rows, q_heads, kv_heads, wmax, scale, sw);
        return hipGetLastError();
    }
    const size_t lds = static_cast<size_t>(wmax) * (kGroup * sizeof(float) + sizeof(uint32_t));
    // dynamic LDS past 64 KB needs the function's limit raised first
    auto kern = packed ? &k_attention_tree<true> : &k_attention_tree<false>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(rows * kv_heads)), dim3(kAttnThreads), lds, s, q, k, v, out,
                       row_pos, anc, anc_stride, rows, q_heads, kv_heads, wmax, scale);
    return hipGetLastError();
}

hipError_t launch_attention_any(const float* q, const float* k, const float* v, float* out, const uint32_t* seg_offset,
                                const uint32_t* seg_pos, int64_t max_seq, int64_t rows, int q_heads, int kv_heads,
                                int head_dim, int window_max, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (kv_heads <= 0 || q_heads <= 0 || q_heads % kv_heads != 0 || head_dim <= 0 || head_dim > kAnyThreads ||
        max_seq <= 0 || window_max <= 0 || rows * q_heads > 0x7FFFFFFFll)
        return hipErrorInvalidValue;
    const int64_t keys = max_seq < window_max ? max_seq : window_max;
    if (keys > kAttnMaxWindow) return hipErrorInvalidValue;
    const int wmax = static_cast<int>(keys);
    const size_t lds = static_cast<size_t>(wmax) * sizeof(float);
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_attention_any),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
        if (e != hipSuccess) return e;
    }
    const float root = sqrtf(static_cast<float>(head_dim));
    const float scale = 1.0f / root;
    hipLaunchKernelGGL(k_attention_any, dim3(static_cast<unsigned>(rows * q_heads)), dim3(kAnyThreads), lds, s, q, k,
                       v, out, seg_offset, seg_pos, rows, q_heads, kv_heads, head_dim, max_seq, wmax, scale);
    return hipGetLastError();
}

}  // namespace aps
