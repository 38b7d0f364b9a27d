// Grouped expert FFN in fp32 with the reference's accumulation order.
//
// Reference: k_moe_pair_silu_8x8 (src/tensor.cu:1838-1966) and
// k_moe_matmul_8x8 (src/tensor.cu:1740-1836) give every output ONE fp32
// accumulator walked over k ascending with FMA (nvcc contracts
// `acc += a * b`), and the SiLU epilogue evaluates exp in double:
// a = g / (1 + (float)exp((double)-g)) * u.
//
// These kernels keep exactly that arithmetic, so for fp32 weights the result
// equals the CPU oracle bit for bit (the only libm call, exp in double, is
// rounded to float afterwards).  The chains run on the fp32 MFMAs, which give
// the same bits (chain_mfma.hpp); arrays that are not 16-byte aligned, and
// Linear shapes those do not take, run on SIMT kernels.
#include "chain_mfma.hpp"

namespace aps {
namespace {

constexpr int kBK = 16;
constexpr int kFXcds = 8;   // XCDs of an MI355X

// The work of a grouped kernel: expert e's rows in tiles of bm positions
// against ncol column blocks.  Workgroup b runs on XCD b % 8, so the column
// blocks (e, c) are dealt to the XCDs by (e ncol + c) % 8 and an XCD walks
// them with the row tiles innermost: the row tiles that read the same weights
// follow one another in one L2, and every XCD gets the same number of columns
// (to one).  b / 8 counts an XCD's items; false past its last.
struct GroupTile {
    int expert, col;
    uint32_t m0, end;
};
__device__ inline bool locate_group_tile(const uint32_t* __restrict__ offsets, int E, int bm, int ncol, GroupTile& g) {
    const int lane = threadIdx.x & 63;
    const int xcd = blockIdx.x % kFXcds, item = blockIdx.x / kFXcds;
    const uint32_t lo = lane < E ? offsets[lane] : 0u;
    uint32_t hi = __shfl_down(lo, 1);
    if (lane == E - 1) hi = offsets[E];
    const int nt = lane < E ? static_cast<int>((hi - lo + bm - 1) / bm) : 0;
    const int c0 = (xcd + kFXcds * ncol - lane * (ncol % kFXcds)) & (kFXcds - 1);   // first column of this XCD
    const int nc = c0 < ncol ? (ncol - 1 - c0) / kFXcds + 1 : 0;
    int incl = nt * nc;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(incl, d);
        if (lane >= d) incl += v;
    }
    const uint64_t m = __ballot(lane < E && incl > item);
    if (m == 0) return false;
    const int e = __ffsll(static_cast<unsigned long long>(m)) - 1;
    const int i = item - (__shfl(incl, e) - __shfl(nt * nc, e));
    const int ent = __shfl(nt, e);
    g.expert = e;
    g.col = __shfl(c0, e) + kFXcds * (i / ent);
    g.m0 = __shfl(lo, e) + static_cast<uint32_t>(i % ent) * bm;
    g.end = __shfl(hi, e);
    return true;
}

// a = g / (1 + (float)exp((double)-g)) * u, each operation rounded on its own
// (src/tensor.cu:1961-1963, src/layer.cu:8-11).
__device__ inline float swiglu_exact(float g, float u) {
    const float ex = static_cast<float>(exp(-static_cast<double>(g)));
    return __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, ex)), u);
}

// act = SwiGLU of the gate and up chains, blocks of 16 RT WR positions.
// CT = 2: a wave's two column tiles are w1's and w3's same 16 columns, so that
// the gate and the up value meet in one lane; 16 WC columns per block.  CT = 1
// (WC = 2): the first column of waves computes gate, the second up, and they
// meet in LDS; 16 columns per block, half the chain length per wave.
template <int RT, int CT, int WR, int WC, int S>
__global__ void __launch_bounds__(64 * WR * WC)
k_ffn_up_f32(const float* __restrict__ x, const uint32_t* __restrict__ offsets,
             const uint32_t* __restrict__ assignment_rows, const float* __restrict__ w1,
             const float* __restrict__ w3, float* __restrict__ act, int H, int F, int E) {
    using Ring = ChainRing<RT, CT, WR, WC, S>;
    static_assert(CT == 2 || (CT == 1 && WC == 2), "gate and up tiles");
    constexpr int kCols = CT == 2 ? 16 * WC : 16;
    __shared__ __align__(16) uint8_t ring[Ring::kBytes];
    GroupTile g;
    if (!locate_group_tile(offsets, E, Ring::kARows, F / kCols, g)) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = g.col * kCols;
    cf4_t acc[RT][CT];
    Ring::run(
        ring,
        [&](int r) __attribute__((always_inline)) {
            if (r < Ring::kARows) {   // positions past the end re-read the last one; their rows are not stored
                const uint32_t p = g.m0 + r < g.end ? g.m0 + r : g.end - 1;
                return x + static_cast<int64_t>(assignment_rows[p]) * H;
            }
            const int b = r - Ring::kARows, t = b / 16;
            const int c = n0 + (CT == 2 ? (t / 2) * 16 : 0) + b % 16;
            return (t % 2 ? w3 : w1) + (static_cast<int64_t>(g.expert) * F + c) * H;
        },
        H, acc);
    const int row = (wave % WR) * 16 * RT + (lane & 15), c4 = 4 * (lane >> 4);
    auto put = [&](int i, int col, const cf4_t& gate, const cf4_t& up) __attribute__((always_inline)) {
        const uint32_t p = g.m0 + row + 16 * i;
        if (p >= g.end) return;
        cf4_t o;
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] = swiglu_exact(gate[v], up[v]);
        *reinterpret_cast<cf4_t*>(act + static_cast<int64_t>(p) * F + col + c4) = o;
    };
    if constexpr (CT == 2) {
#pragma unroll
        for (int i = 0; i < RT; ++i) put(i, n0 + (wave / WR) * 16, acc[i][0], acc[i][1]);
    } else {
        __syncthreads();   // every wave is done with the ring
        auto* up = reinterpret_cast<cf4_t*>(ring) + (wave % WR) * RT * 64 + lane;
        if (wave / WR == 1)
#pragma unroll
            for (int i = 0; i < RT; ++i) up[64 * i] = acc[i][0];
        __syncthreads();
        if (wave / WR == 0)
#pragma unroll
            for (int i = 0; i < RT; ++i) put(i, n0, acc[i][0], up[64 * i]);
    }
}

// y = act . w2^T, blocks of 16 RT WR positions x 16 CT WC hidden columns.
template <int RT, int CT, int WR, int WC, int S>
__global__ void __launch_bounds__(64 * WR * WC)
k_ffn_down_f32(const float* __restrict__ act, const uint32_t* __restrict__ offsets,
               const float* __restrict__ w2, float* __restrict__ y, int H, int F, int E) {
    using Ring = ChainRing<RT, CT, WR, WC, S>;
    __shared__ __align__(16) uint8_t ring[Ring::kBytes];
    GroupTile g;
    if (!locate_group_tile(offsets, E, Ring::kARows, H / Ring::kBRows, g)) return;
    const int lane = threadIdx.x & 63;
    const int wave = WR * WC > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int n0 = g.col * Ring::kBRows;
    cf4_t acc[RT][CT];
    Ring::run(
        ring,
        [&](int r) __attribute__((always_inline)) {
            if (r < Ring::kARows) {
                const uint32_t p = g.m0 + r < g.end ? g.m0 + r : g.end - 1;
                return act + static_cast<int64_t>(p) * F;
            }
            return w2 + (static_cast<int64_t>(g.expert) * H + n0 + r - Ring::kARows) * F;
        },
        F, acc);
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const uint32_t p = g.m0 + (wave % WR) * 16 * RT + 16 * i + (lane & 15);
        if (p >= g.end) continue;
#pragma unroll
        for (int j = 0; j < CT; ++j)
            *reinterpret_cast<cf4_t*>(y + static_cast<int64_t>(p) * H + n0 + (wave / WR) * 16 * CT + 16 * j +
                                      4 * (lane >> 4)) = acc[i][j];
    }
}

// ---- any alignment ---------------------------------------------------------
// The same chains on the vector ALU with 4-byte accesses, for arrays that the
// ring's 16-byte copies cannot take (and, k_linear_any, for Linear shapes it
// does not): 64 x 64 blocks, 4 x 4 outputs per thread and operand, 16 k of
// each operand k-major in LDS.
constexpr int kAnyPitch = kF32BM + 4;   // a wave's transposing stores hit 64 banks
static_assert(kF32BM == 64 && kF32BN == 64, "one row of A and of each B per four threads");

template <int NB>
struct AnyStage {
    float a[kBK][kAnyPitch], b[NB][kBK][kAnyPitch];
};

// acc[n][r][c] += the chain of row 4 (tid / 16) + r of A against row 4 (tid %
// 16) + c of B n.  a, b: this thread's staging row (tid / 4) of each, null past
// the end: read as zero, as is k past K.  A padded step adds the exact product
// 0 * 0 to an accumulator that is never -0 (it starts at +0, and a sum that
// cancels exactly rounds to +0), so it changes no bit.  VEC: 16-byte accesses, K
// % 4 == 0.
template <int NB, bool VEC = false>
__device__ inline void any_chains(AnyStage<NB>& st, const float* a, const float* const (&b)[NB], int K,
                                  float (&acc)[NB][4][4]) {
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4, sr = tid >> 2, sk = (tid & 3) * 4;
    for (int k0 = 0; k0 < K; k0 += kBK) {
        cf4_t av = {}, bv[NB] = {};
        if constexpr (VEC) {
            const int k = k0 + sk;
            if (a && k < K) av = *reinterpret_cast<const cf4_t*>(a + k);
#pragma unroll
            for (int n = 0; n < NB; ++n)
                if (b[n] && k < K) bv[n] = *reinterpret_cast<const cf4_t*>(b[n] + k);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = k0 + sk + i;
                av[i] = a && k < K ? a[k] : 0.0f;
#pragma unroll
                for (int n = 0; n < NB; ++n) bv[n][i] = b[n] && k < K ? b[n][k] : 0.0f;
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            st.a[sk + i][sr] = av[i];
#pragma unroll
            for (int n = 0; n < NB; ++n) st.b[n][sk + i][sr] = bv[n][i];
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kBK; ++kk) {
            const cf4_t ar = *reinterpret_cast<const cf4_t*>(&st.a[kk][ty * 4]);
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const cf4_t br = *reinterpret_cast<const cf4_t*>(&st.b[n][kk][tx * 4]);
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[n][r][c] = __builtin_fmaf(ar[r], br[c], acc[n][r][c]);
            }
        }
    }
}

// UP: act as k_ffn_up_f32 (w = w1, w' = w3, rows by assignment_rows); else y as
// k_ffn_down_f32 (w = w2, rows by position).  [N][K]: an expert's weight matrix.
template <bool UP>
__global__ void __launch_bounds__(256)
k_ffn_any(const float* __restrict__ in, const uint32_t* __restrict__ offsets,
          const uint32_t* __restrict__ assignment_rows, const float* __restrict__ w, const float* __restrict__ w3,
          float* __restrict__ out, int K, int N, int E) {
    constexpr int NB = UP ? 2 : 1;
    __shared__ __align__(16) AnyStage<NB> st;
    GroupTile g;
    if (!locate_group_tile(offsets, E, kF32BM, N / kF32BN, g)) return;
    const int tid = threadIdx.x, sr = tid >> 2, n0 = g.col * kF32BN;
    const uint32_t p = g.m0 + sr;
    const float* a = nullptr;
    if (p < g.end) a = in + static_cast<int64_t>(UP ? assignment_rows[p] : p) * K;
    const int64_t brow = (static_cast<int64_t>(g.expert) * N + n0 + sr) * K;
    const float* b[NB];
    b[0] = w + brow;
    if constexpr (UP) b[1] = w3 + brow;
    float acc[NB][4][4] = {};
    any_chains<NB>(st, a, b, K, acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint32_t pr = g.m0 + (tid >> 4) * 4 + r;
        if (pr >= g.end) continue;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            out[static_cast<int64_t>(pr) * N + n0 + (tid & 15) * 4 + c] =
                UP ? swiglu_exact(acc[0][r][c], acc[NB - 1][r][c]) : acc[0][r][c];
    }
}

// y[m][n] = (fp32 FMA chain over k ascending of x[m][k] w[n][k]) + bias[n] for
// any K, N and alignment (the reference's fallback for shapes its fast kernels
// do not take, k_matmul_transposed_tiled, src/tensor.cu:433-461).  Row tiles
// are walked grid-stride over gridDim.y.  VEC: 16-byte aligned, K and N multiples
// of four.
template <bool VEC>
__global__ void __launch_bounds__(256)
k_linear_any(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
             float* __restrict__ y, int64_t M, int K, int N) {
    __shared__ __align__(16) AnyStage<1> st;
    const int n0 = blockIdx.x * kF32BN;
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4, sr = tid >> 2;
    const float* const b[1] = {n0 + sr < N ? w + static_cast<int64_t>(n0 + sr) * K : nullptr};
    cf4_t bv = {};
    if constexpr (VEC)
        if (bias && n0 + tx * 4 < N) bv = *reinterpret_cast<const cf4_t*>(bias + n0 + tx * 4);
    for (int64_t m0 = static_cast<int64_t>(blockIdx.y) * kF32BM; m0 < M;
         m0 += static_cast<int64_t>(gridDim.y) * kF32BM) {
        float acc[1][4][4] = {};
        any_chains<1, VEC>(st, m0 + sr < M ? x + (m0 + sr) * K : nullptr, b, K, acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = m0 + ty * 4 + r;
            if (row >= M) continue;
            if constexpr (VEC) {
                const int col = n0 + tx * 4;   // N % 4 == 0: a column group is all in or all out
                if (col >= N) continue;
                cf4_t o;
#pragma unroll
                for (int c = 0; c < 4; ++c) o[c] = bias ? __fadd_rn(acc[0][r][c], bv[c]) : acc[0][r][c];
                *reinterpret_cast<cf4_t*>(y + row * N + col) = o;
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int col = n0 + tx * 4 + c;
                    if (col >= N) continue;
                    y[row * N + col] = bias ? __fadd_rn(acc[0][r][c], bias[col]) : acc[0][r][c];
                }
            }
        }
    }
}

// The ring copies rows of `a` 16 bytes at a time and the epilogue stores 16
// bytes of `b`; the library's own weight arrays are always aligned.
bool aligned16(const float* a, const float* b) {
    return ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15u) == 0;
}

}  // namespace

hipError_t launch_linear_any_f32(const float* x, const float* w, const float* bias, float* y, int64_t rows, int in_f,
                                 int out_f, hipStream_t s, bool vec) {
    if (rows <= 0) return hipSuccess;
    if (in_f <= 0 || out_f <= 0 || (vec && (in_f % 4 != 0 || out_f % 4 != 0))) return hipErrorInvalidValue;
    const int64_t ty = ceil_div(rows, kF32BM);
    const dim3 grid(static_cast<unsigned>(ceil_div(out_f, kF32BN)), static_cast<unsigned>(ty < 65535 ? ty : 65535));
    hipLaunchKernelGGL(vec ? k_linear_any<true> : k_linear_any<false>, grid, dim3(256), 0, s, x, w, bias, y, rows,
                       in_f, out_f);
    return hipGetLastError();
}

// Rows per block by the mean number of positions per expert.
#define APS_GROUPED(KERNEL, RT, CT, WR, WC, S, NCOL, ...)                                                        \
    do {                                                                                                          \
        const int64_t t = max_row_tiles(2 * rows, 16 * RT * WR, experts) * ceil_div(NCOL, kFXcds) * kFXcds;        \
        hipLaunchKernelGGL((KERNEL<RT, CT, WR, WC, S>), dim3(static_cast<unsigned>(t)), dim3(64 * WR * WC), 0, s, \
                           __VA_ARGS__, hidden, ffn, experts);                                                    \
        return hipGetLastError();                                                                                 \
    } while (0)

hipError_t launch_ffn_up_f32(const float* x, const uint32_t* offsets,
                             const uint32_t* assignment_rows, const float* w1,
                             const float* w3, float* act, int64_t rows, int hidden, int ffn,
                             int experts, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (hidden % kBK != 0 || ffn % 64 != 0) return hipErrorInvalidValue;
    if (!aligned16(x, act)) {
        const int64_t t = max_row_tiles(2 * rows, kF32BM, experts) * ceil_div(ffn / kF32BN, kFXcds) * kFXcds;
        hipLaunchKernelGGL(k_ffn_any<true>, dim3(static_cast<unsigned>(t)), dim3(256), 0, s, x, offsets,
                           assignment_rows, w1, w3, act, hidden, ffn, experts);
        return hipGetLastError();
    }
    const int64_t mean = ceil_div(2 * rows, experts);
    // us at hidden 4096, ffn 448, 16 experts, for 1 / 43 / 512 / 1,024 / 2,048
    // tokens; the SIMT kernel before these took 468 to 476 us up to 512
    //   16 rows x 16 columns, gate and up on two waves   23  52 136 225 428
    //   32 x 16, the same                                26  53 114 177 332
    //   32 x 32, gate and up in a lane                   41  57 121 165 307
    //   64 x 32                                          66  78 141 203 279
    // Few rows are bound by the length of a chain or by the weights (235 MB,
    // 48 us), many by the MFMAs on rows that pad each expert's last tile.
    if (mean <= 8) APS_GROUPED(k_ffn_up_f32, 1, 1, 1, 2, 8, ffn / 16, x, offsets, assignment_rows, w1, w3, act);
    if (mean <= 96) APS_GROUPED(k_ffn_up_f32, 1, 1, 2, 2, 4, ffn / 16, x, offsets, assignment_rows, w1, w3, act);
    if (mean <= 192) APS_GROUPED(k_ffn_up_f32, 1, 2, 2, 2, 4, ffn / 32, x, offsets, assignment_rows, w1, w3, act);
    APS_GROUPED(k_ffn_up_f32, 2, 2, 2, 2, 4, ffn / 32, x, offsets, assignment_rows, w1, w3, act);
}

hipError_t launch_ffn_down_f32(const float* act, const uint32_t* offsets, const float* w2,
                               float* y, int64_t rows, int hidden, int ffn, int experts,
                               hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (ffn % kBK != 0 || hidden % 64 != 0) return hipErrorInvalidValue;
    if (!aligned16(act, y)) {
        const int64_t t = max_row_tiles(2 * rows, kF32BM, experts) * ceil_div(hidden / kF32BN, kFXcds) * kFXcds;
        hipLaunchKernelGGL(k_ffn_any<false>, dim3(static_cast<unsigned>(t)), dim3(256), 0, s, act, offsets, nullptr,
                           w2, nullptr, y, ffn, hidden, experts);
        return hipGetLastError();
    }
    const int64_t mean = ceil_div(2 * rows, experts);
    // as above; the SIMT kernel took 63 us for 43 tokens, 89 for 512
    //   16 rows x 64 columns    8  25  60 107 199
    //   32 x 64                 9  27  54  92 175
    //   64 x 64                12  39  58  93 160
    if (mean <= 16) APS_GROUPED(k_ffn_down_f32, 1, 2, 1, 2, 4, hidden / 64, act, offsets, w2, y);
    if (mean <= 192) APS_GROUPED(k_ffn_down_f32, 1, 2, 2, 2, 4, hidden / 64, act, offsets, w2, y);
    APS_GROUPED(k_ffn_down_f32, 2, 2, 2, 2, 4, hidden / 64, act, offsets, w2, y);
}
#undef APS_GROUPED

}  // namespace aps
