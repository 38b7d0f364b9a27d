// fp32 Linear on the matrix cores, bit for bit the reference's FMA chain.
//
// y[m][n] = (fp32 FMA chain over k ascending of x[m][k] w[n][k]) + bias[n]:
// the decoder's projections and the LM head.  Reference: Linear::forward
// (src/layer.cu:30-42) -> matmul_transposed_bias_gpu (src/tensor.cu:3120-3143)
// -> k_matmul_transposed_8x8 (src/tensor.cu:715-800): one accumulator per
// output walked over k ascending, the bias added once in the epilogue.
// chain_mfma.hpp states why the fp32 MFMAs give those bits.
//
// Two kernels:
//  * k_linear_mfma, many rows: 128-row x 128- (or 64-) column blocks, four
//    waves of 64 x 64 on v_mfma_f32_32x32x2_f32;
//  * k_linear_small, few rows: 16- to 64-row blocks on v_mfma_f32_16x16x4_f32.
// The launcher's cost rule takes the one whose busiest CU is done first, or for a
// short K that is not a multiple of 32 the SIMT blocks of ffn_f32.hip.
#include "chain_mfma.hpp"

#include <utility>

namespace aps {
namespace {

constexpr int kLRows = 128;               // x rows per block
constexpr int kLStageK = 32;              // k per stage: one 128-byte row

__device__ inline void l_wait_vm0() { chain_wait_vm<0>(); }
__device__ inline void l_barrier() { asm volatile("s_barrier" ::: "memory"); }

template <int V>
struct LInt {
    static constexpr int value = V;
};

constexpr int kLXcds = 8;   // XCDs of an MI355X

// Up to three outputs of one x in one grid (the reference's
// matmul_pair_bias_gpu pairs k and v): segment s owns column tiles
// t0[s] .. t0[s + 1] - 1 of the grid's column dimension.
struct LinSegs {
    const float* w[3];
    const float* b[3];
    float* y[3];
    int n[3];
    int t0[4];
};
__device__ inline int seg_of(const LinSegs& g, int tc) { return tc >= g.t0[1] ? (tc >= g.t0[2] ? 2 : 1) : 0; }

// WN: columns per wave (64, or 32 for grids that would otherwise leave CUs
// idle).  A block is 128 rows x 2 WN columns, four waves of 64 x WN as 2 x
// WN / 32 tiles of v_mfma_f32_32x32x2_f32.  A stage is 32 k deep: 128 x rows
// and 2 WN weight rows of 128 bytes, copied with global_load_lds_dwordx4 into
// two LDS slots (64 KB with WN = 64: two blocks per CU).
// Bound by the fp32 MFMA rate under the card's power limit: 145 to 149
// TFLOP/s with nothing but MFMAs on all CUs (157 nominal), so everything else
// stays out of the vector ALU (chain_mfma.hpp) and in the MFMAs' shadow:
//  * operands are read in MFMA order, a chunk of 4 k (two steps) ahead, one
//    ds_read2_b32 behind each of the first MFMAs of a chunk.  In one burst
//    they hold the MFMAs up until the LDS has taken them all;
//  * the stage hand-over (all copies of stage kt + 1 landed, one barrier) sits
//    before the last chunk's MFMAs; the refill of the freed slot goes out
//    between them;
//  * source pointers move once per two stages (the copies' immediate offset
//    reaches the second), LDS addresses are registers.
// Measured, 4096 x 4096 -> 2048: 472 us (145 TFLOP/s); 10,240 rows 1168 us
// (147).  The K = 1 MFMA form before it (every B operand read twice, b128
// reads that the compiler waited for in full, two barriers a stage, each
// store of the epilogue behind a wait for the one before): 546 and 1540 us.
// The grid is one-dimensional over the row-tile-major tile order.
// Workgroups are dealt to the 8 XCDs round robin (workgroup b runs on XCD
// b % 8).  Taken in launch order (tile b), XCD x holds the column tiles
// c = x mod 8 of every row tile: it reads an eighth of W and all of x.  With
// xcd_rows, workgroup b takes tile (b % 8) * per + b / 8 instead: XCD x holds
// a contiguous run of tiles, the column tiles of a row tile sharing its x
// rows in one L2, and reads about an eighth of x and all of W.  The
// launcher picks xcd_rows when x is the larger operand by 3x or more.
template <int WN>
__global__ void __launch_bounds__(256, 2)
k_linear_mfma(const float* __restrict__ x, const LinSegs segs, int64_t M, int K, int row_tiles, int xcd_rows) {
    constexpr int kBRows = 2 * WN;                        // weight rows per block
    constexpr int kStageRows = kLRows + kBRows;
    constexpr int kLStageBytes = kStageRows * 128;
    constexpr int kSlots = kStageRows / 32;               // copies per wave per stage
    constexpr int NJ = WN / 32;                           // column tiles per wave
    // one LDS object for both slots: with two, the compiler's tracking of the
    // in-flight copies made every stage's first read wait for all of them
    // (the next stage's included); the waits here are explicit
    __shared__ __align__(16) uint8_t ring[2][kLStageBytes];
    const int ncol = segs.t0[3];
    const int64_t per = (static_cast<int64_t>(row_tiles) * ncol + kLXcds - 1) / kLXcds;
    const int64_t t = xcd_rows ? static_cast<int64_t>(blockIdx.x % kLXcds) * per + blockIdx.x / kLXcds
                               : static_cast<int64_t>(blockIdx.x);
    if (t >= static_cast<int64_t>(row_tiles) * ncol) return;
    const int tc = static_cast<int>(t % ncol);
    const int64_t m0 = (t / ncol) * kLRows;
    const int sg = seg_of(segs, tc);
    const float* __restrict__ w = segs.w[sg];
    const float* __restrict__ bias = segs.b[sg];
    float* __restrict__ y = segs.y[sg];
    const int N = segs.n[sg];
    const int n0 = (tc - segs.t0[sg]) * kBRows;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KT = K / kLStageK;

    // copies: instruction s of wave w fills stage rows 32s + 8w .. +7; lane
    // i writes row 32s + 8w + i/8, physical chunk i & 7, i.e. logical chunk
    // (i & 7) ^ ((row >> 1) & 7).  Rows 0..127 are x rows m0.., the rest
    // weight rows n0..; rows past the end re-read the last one (their
    // results are not stored).
    const float* src[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        const int row = 32 * s + 8 * wave + (lane >> 3);
        const int chunk = (lane & 7) ^ ((row >> 1) & 7);
        if (32 * s < kLRows) {
            const int64_t r = m0 + row < M ? m0 + row : M - 1;
            src[s] = x + r * K + 4 * chunk;
        } else {
            const int64_t r = n0 + (row - kLRows) < N ? n0 + (row - kLRows) : N - 1;
            src[s] = w + r * K + 4 * chunk;
        }
    }
    // the stage at src (+ one stage for slot 1) into its slot; the copy's
    // immediate offset moves both addresses
    auto issue_one = [&](auto slotc, int s) __attribute__((always_inline)) {
        constexpr int P = decltype(slotc)::value;
        __builtin_amdgcn_global_load_lds(APS_CGP(src[s]), APS_CLP(ring[P] + (32 * s + 8 * wave) * 128 - 128 * P), 16,
                                         128 * P, 0);
    };
    auto issue = [&](auto slotc) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < kSlots; ++s) issue_one(slotc, s);
    };

    const int aR = (wave & 1) * 64;            // this wave's x rows in the stage
    const int bR = kLRows + (wave >> 1) * WN;  // its weight rows
    cf16_t acc[2][NJ];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    // this lane's bias of each column tile, loaded before the main loop
    float bb[NJ];
    int col[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        col[j] = n0 + (wave >> 1) * WN + 32 * j + (lane & 31);
        bb[j] = bias != nullptr ? bias[col[j] < N ? col[j] : N - 1] : 0.0f;
    }

    // this lane's LDS addresses: 16-byte chunk c of its row of tile 0, at the
    // k half (lane / 32) of a step; the tiles lie 4096 bytes apart (the
    // swizzle repeats every 16 rows), step 2 c + 1 8 bytes after step 2 c
    uint32_t aa[2][8], ba[2][8];   // [slot]
    const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(APS_CLP(&ring[0][0]))) + 4 * (lane >> 5);
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            aa[p][c] = base + p * kLStageBytes + chain_swz(aR + (lane & 31), c);
            ba[p][c] = base + p * kLStageBytes + chain_swz(bR + (lane & 31), c);
            // kept as they are: derived from one another they would cost a
            // vector add before every read
            asm volatile("" : "+v"(aa[p][c]), "+v"(ba[p][c]));
        }
    typedef const __attribute__((address_space(3))) float* lds_t;
    // one stage: 8 chunks of 4 k (two steps); a chunk's operands are read one
    // chunk ahead of its MFMAs
    float a[2][2][2], b[2][2][NJ];   // [set][step][tile]
    auto load_a = [&](auto slotc, auto cc, int p, int i) __attribute__((always_inline)) {
        constexpr int sl = decltype(slotc)::value, c = decltype(cc)::value;
#pragma unroll
        for (int h = 0; h < 2; ++h) a[p][h][i] = *reinterpret_cast<lds_t>(aa[sl][c] + (4096 * i + 8 * h));
    };
    auto load_b = [&](auto slotc, auto cc, int p, int j) __attribute__((always_inline)) {
        constexpr int sl = decltype(slotc)::value, c = decltype(cc)::value;
#pragma unroll
        for (int h = 0; h < 2; ++h) b[p][h][j] = *reinterpret_cast<lds_t>(ba[sl][c] + (4096 * j + 8 * h));
    };
    auto load = [&](auto slotc, auto cc, int p) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) load_a(slotc, cc, p, i);
#pragma unroll
        for (int j = 0; j < NJ; ++j) load_b(slotc, cc, p, j);
    };
    // the MFMAs of set p, after(n) behind the n-th
    auto mma = [&](int p, auto after) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[p][h][i], b[p][h][j], acc[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    after((h * 2 + i) * NJ + j);
                    __builtin_amdgcn_sched_barrier(0);
                }
    };
    // a stage whose first chunk's operands are read already; `more`: another
    // follows; `refill`: its slot takes the stage after that, once every wave
    // has read it (the barrier before its last MFMAs)
    auto stage = [&](auto par, bool more, bool refill) __attribute__((always_inline)) {
        constexpr int P = decltype(par)::value;
        [&]<int... C>(std::integer_sequence<int, C...>) __attribute__((always_inline)) {
            (
                [&] {
                    chain_wait_lgkm0();   // chunk C's operands
                    mma(C & 1, [&](int n) __attribute__((always_inline)) {
                        if (n < 2) load_a(par, LInt<C + 1>{}, (C + 1) & 1, n);
                        else if (n < 2 + NJ) load_b(par, LInt<C + 1>{}, (C + 1) & 1, n - 2);
                    });
                }(),
                ...);
        }(std::make_integer_sequence<int, 7>{});
        chain_wait_lgkm0();
        if (more) {
            l_wait_vm0();
            l_barrier();
        }
        mma(1, [&](int n) __attribute__((always_inline)) {
            if (!more) return;
            if (n < 2) load_a(LInt<P ^ 1>{}, LInt<0>{}, 0, n);
            else if (n < 2 + NJ) load_b(LInt<P ^ 1>{}, LInt<0>{}, 0, n - 2);
            if (refill) {
#pragma unroll
                for (int s = n * kSlots / (4 * NJ); s < (n + 1) * kSlots / (4 * NJ); ++s) issue_one(par, s);
            }
        });
    };
    auto advance = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < kSlots; ++s) src[s] += 2 * kLStageK;
    };
    issue(LInt<0>{});
    if (KT > 1) issue(LInt<1>{});
    advance();
    if (KT > 1) chain_wait_vm<kSlots>();
    else l_wait_vm0();
    l_barrier();
    load(LInt<0>{}, LInt<0>{}, 0);
    int kt = 0;
    for (; kt + 3 < KT; kt += 2) {
        stage(LInt<0>{}, true, true);
        stage(LInt<1>{}, true, true);
        advance();
    }
    // one, two or three stages left
    stage(LInt<0>{}, kt + 1 < KT, kt + 2 < KT);
    if (kt + 1 < KT) stage(LInt<1>{}, kt + 2 < KT, false);
    if (kt + 2 < KT) stage(LInt<0>{}, false, false);

    // epilogue: register v of acc[i][j] is row 32 i + 8 (v / 4) + 4 (lane /
    // 32) + v % 4 of the wave tile, column 32 j + lane % 32; the 32 lanes of
    // a row store 128 contiguous bytes.  (The empty asm waits for the bias
    // once: left to its uses, every store waited for the store before it.)
#pragma unroll
    for (int j = 0; j < NJ; ++j) asm volatile("" : "+v"(bb[j]));
    const int64_t row0 = m0 + aR + 4 * (lane >> 5);
    auto store = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const int64_t row = row0 + 32 * i + 8 * (v / 4) + (v % 4);
                    const float o = bias != nullptr ? __fadd_rn(acc[i][j][v], bb[j]) : acc[i][j][v];
                    if (decltype(whole)::value || (row < M && col[j] < N)) y[row * N + col[j]] = o;
                }
    };
    if (m0 + kLRows <= M && n0 + kBRows <= N) store(LInt<1>{});   // block-uniform
    else store(LInt<0>{});
}

// Few rows: ChainRing blocks of 16 RT WR rows x 16 CT WC columns
// (chain_mfma.hpp).  Tiles in row-fastest order, so that the blocks that share
// weight columns run together.  Rows and columns past the end re-read the
// last one; their results are not stored.  Bound by the length of the chain
// (14 us at K = 4096) or, for the LM head, by W's bytes.  Measured against
// 128 x 64 blocks, which computed 128 rows whatever their number: 16 rows of
// 4096 -> 2048 139 -> 22 us, 333 rows 146 -> 72 us, 333 rows of 2048 -> 4096
// 82 -> 64 us; the LM head (4096 -> 32064, 525 MB) on 8 rows 279 -> 111 us
// (4.7 TB/s), on 40 rows 283 -> 141 us.
template <int RT, int CT, int WR, int WC, int S>
__global__ void __launch_bounds__(64 * WR * WC)
k_linear_small(const float* __restrict__ x, const LinSegs segs, int64_t M, int K, int row_tiles) {
    using Ring = ChainRing<RT, CT, WR, WC, S>;
    __shared__ __align__(16) uint8_t ring[Ring::kBytes];
    const int tc = static_cast<int>(blockIdx.x / row_tiles);
    const int64_t m0 = static_cast<int64_t>(blockIdx.x % row_tiles) * Ring::kARows;
    const int sg = seg_of(segs, tc);
    const float* __restrict__ w = segs.w[sg];
    const float* __restrict__ bias = segs.b[sg];
    float* __restrict__ y = segs.y[sg];
    const int N = segs.n[sg];
    const int n0 = (tc - segs.t0[sg]) * Ring::kBRows;
    const int lane = threadIdx.x & 63;
    const int wave = WR * WC > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    cf4_t acc[RT][CT];
    Ring::run(
        ring,
        [&](int r) __attribute__((always_inline)) {
            if (r < Ring::kARows) return x + (m0 + r < M ? m0 + r : M - 1) * K;
            const int c = n0 + r - Ring::kARows;
            return w + static_cast<int64_t>(c < N ? c : N - 1) * K;
        },
        K, acc);
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        const int c = n0 + (wave / WR) * 16 * CT + 16 * j + 4 * (lane >> 4);
        if (c >= N) continue;   // N % 4 == 0: a column group is all in or all out
        cf4_t bv = {0.0f, 0.0f, 0.0f, 0.0f};
        if (bias != nullptr) bv = *reinterpret_cast<const cf4_t*>(bias + c);
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const int64_t r = m0 + (wave % WR) * 16 * RT + 16 * i + (lane & 15);
            if (r >= M) continue;
            cf4_t o = acc[i][j];
            if (bias != nullptr)
#pragma unroll
                for (int v = 0; v < 4; ++v) o[v] = __fadd_rn(o[v], bv[v]);
            *reinterpret_cast<cf4_t*>(y + r * N + c) = o;
        }
    }
}

// Fills the segment table for column tiles of `bc` columns; returns the tiles.
int fill_segs(LinSegs& segs, int count, const float* const* w, const float* const* bias, float* const* y,
              const int* out_f, int bc) {
    int t = 0;
    for (int i = 0; i < 3; ++i) {
        segs.t0[i] = t;
        if (i < count) {
            segs.w[i] = w[i];
            segs.b[i] = bias[i];
            segs.y[i] = y[i];
            segs.n[i] = out_f[i];
            t += static_cast<int>(ceil_div(out_f[i], bc));
        }
    }
    segs.t0[3] = t;
    for (int i = count; i < 3; ++i) segs.t0[i] = t;   // empty segments past the last
    return t;
}

}  // namespace

bool linear_mfma_fits(int64_t rows, int in_f, int out_f) {
    return rows > 0 && in_f > 0 && in_f % 16 == 0 && out_f > 0 && out_f % 4 == 0 &&
           (rows + kLRows - 1) / kLRows <= 65535;
}

hipError_t launch_linear_mfma_multi(const float* x, int64_t rows, int in_f, int count, const float* const* w,
                                    const float* const* bias, float* const* y, const int* out_f, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (count < 1 || count > 3) return hipErrorInvalidValue;
    for (int i = 0; i < count; ++i)
        if (!linear_mfma_fits(rows, in_f, out_f[i])) return hipErrorInvalidValue;
    // Blocks on the busiest CU x the time of one block, in us at K = 4096 as
    // measured with one to eight blocks per CU.  A small block's MFMAs alone
    // take 14, 29, 57 us, and 114 and 228 for the two block kernels; the
    // rest is what its operand reads and copies add.
    const int64_t cus = num_cus(), rt = ceil_div(rows, kLRows);
    auto cost = [&](int br, int bc, double us) {
        int64_t t = 0;
        for (int i = 0; i < count; ++i) t += ceil_div(out_f[i], bc);
        return static_cast<double>(ceil_div(ceil_div(rows, br) * t, cus)) * us;
    };
    LinSegs segs{};
#define APS_SMALL(RT, CT, WR, WC, S)                                                                              \
    do {                                                                                                           \
        const int64_t tt = fill_segs(segs, count, w, bias, y, out_f, 16 * CT * WC);                                \
        const int64_t rtt = ceil_div(rows, 16 * RT * WR);                                                          \
        hipLaunchKernelGGL((k_linear_small<RT, CT, WR, WC, S>), dim3(static_cast<unsigned>(tt * rtt)),              \
                           dim3(64 * WR * WC), 0, s, x, segs, rows, in_f, static_cast<int>(rtt));                  \
        return hipGetLastError();                                                                                  \
    } while (0)
    // one-wave blocks of one tile: at most 16 rows (W streams past once), or
    // so few tiles that every wave has a SIMD, and half the CU's LDS ports,
    // to itself
    int64_t waves = 0;
    for (int i = 0; i < count; ++i) waves += ceil_div(out_f[i], 16) * ceil_div(rows, 16);
    if (rows <= 16 || waves <= 2 * cus) APS_SMALL(1, 1, 1, 1, 8);
    // A short K that ends in half a stage (in_f % 32 == 16) on many blocks is
    // bound by y's stores, and the ring's 64 KB of LDS leave two blocks to a CU:
    // SIMT blocks of 64 x 64 there.  us, ring -> SIMT: 20,000 rows of 16 -> 4096 236
    // -> 66, of 48 -> 4096 273 -> 132, of 112 -> 11008 935 -> 735; 333 rows of 16 ->
    // 4096 7.6 -> 4.2; past the line 17 rows of 48 -> 11008 4.5 -> 5.0, 4,096 rows of
    // 176 -> 1000 24 -> 26.
    bool simt = in_f % kLStageK != 0 && in_f <= 144;
    for (int i = 0; i < count; ++i) {
        const int64_t blocks = ceil_div(out_f[i], kF32BN) * ceil_div(rows, kF32BM);
        simt = simt && out_f[i] >= kF32BN && 8 * blocks >= 3 * cus && 70 * blocks >= cus * in_f;
    }
    if (simt) {
        for (int i = 0; i < count; ++i) {
            const hipError_t e = launch_linear_any_f32(x, w[i], bias[i], y[i], rows, in_f, out_f[i], s, true);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    const bool whole = in_f % kLStageK == 0;   // the block kernels take whole stages only
    const double c11 = cost(32, 32, 22.5), c12 = cost(32, 64, 38.5), c22 = cost(64, 64, 63.5);
    const double c64 = whole ? cost(128, 64, 121.0) : 1e300, c128 = whole ? cost(128, 128, 230.0) : 1e300;
    const double small = c11 < c12 ? (c11 < c22 ? c11 : c22) : (c12 < c22 ? c12 : c22);
    if (small < c64 && small < c128) {
        if (small == c22) APS_SMALL(2, 2, 2, 2, 4);
        if (small == c12) APS_SMALL(1, 2, 2, 2, 4);
        APS_SMALL(1, 1, 2, 2, 4);
    }
#undef APS_SMALL
    const bool wide = c128 <= c64;
    const int t = fill_segs(segs, count, w, bias, y, out_f, wide ? 128 : 64);
    const int64_t tiles = static_cast<int64_t>(t) * rt;
    int64_t wcols = 0;
    for (int i = 0; i < count; ++i) wcols += out_f[i];
    const int xr = rows >= 3 * wcols ? 1 : 0;   // x bytes >= 3 x W bytes (both rows x in_f fp32)
    const dim3 grid(static_cast<unsigned>(ceil_div(tiles, kLXcds) * kLXcds));
    if (wide) hipLaunchKernelGGL(k_linear_mfma<64>, grid, dim3(256), 0, s, x, segs, rows, in_f, static_cast<int>(rt), xr);
    else hipLaunchKernelGGL(k_linear_mfma<32>, grid, dim3(256), 0, s, x, segs, rows, in_f, static_cast<int>(rt), xr);
    return hipGetLastError();
}

hipError_t launch_linear_mfma_f32(const float* x, const float* w, const float* bias, float* y, int64_t rows,
                                  int in_f, int out_f, hipStream_t s) {
    return launch_linear_mfma_multi(x, rows, in_f, 1, &w, &bias, &y, &out_f, s);
}

}  // namespace aps
