// Split-bf16 Linear on the bf16 matrix cores: the reference's optional
// tensor-core projection path.
//
// Reference: Tensor::prepare_cuda_bf16_weight and k_pack_bf16_weight
// (src/tensor.cu:124-177: W = W_hi + W_lo, W_hi = bf16(w), W_lo = bf16(w -
// W_hi), round to nearest even), k_matmul_transposed_bf16_wmma
// (src/tensor.cu:514-584: x split the same way on the fly; per 16-k step
// acc += x_hi W_hi + x_hi W_lo + x_lo W_hi, and x_lo W_lo as well under
// USE_TC_ALL; fp32 accumulation), its dispatch in matmul_transposed_gpu
// (src/tensor.cu:3042-3055) and the bias added after the product
// (matmul_transposed_bias_gpu, src/tensor.cu:3121-3142).  The sum is an
// approximation of the fp32 product (the dropped lo x lo term and the
// residual of lo are about 2^-16 of a product), accumulated in a different
// order than the fp32 chain, so it is compared with the fp32 oracle under a
// tolerance, not bit for bit.
//
// gfx950 mapping.
//  * x is split once into bf16 x_hi and x_lo row-major arrays (k_split_bf16,
//    shared by every projection of one input), W once at preparation into
//    swizzled tile images: 128 rows x 32 k, each 128-byte row the 32 hi values
//    and then the 32 lo values, so that a stage row of the MFMA ring
//    (mfma_ring.hpp) holds both halves of its operand.
//  * A block computes 128 rows x 256, 128 or 64 columns with four waves of 64
//    x 128, 64 x 64 or 32 x 64 (v_mfma_f32_32x32x16_bf16).  A fragment pair (hi,
//    lo) feeds 3 or 4 products, and the products go round all of a wave's
//    tiles before the next one, so no MFMA waits for the one before it.
//  * Rows past M and columns past N read clamped rows / zero-padded images
//    and are not stored.
//  Bound by the bf16 MFMAs and their operand reads.  Measured, 10,240 rows,
//  four products: q, k and v (4096 -> 3072) 989 -> 817 us (1.26 PFLOP/s), output
//  projection (2048 -> 4096) 665 -> 539 us, against 128 x 128 blocks in two 64 KB
//  stages, which drained every copy at a barrier per stage and read each
//  step's operands right before its MFMAs.
#include "mfma_ring.hpp"

namespace aps {
namespace {

constexpr int kTcRows = 128;                 // x rows per block
constexpr int kTcK = 32;                     // k per stage

__device__ inline uint16_t bf16_bits(float v) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(v)); }
__device__ inline float bf16_value(uint16_t b) { return __uint_as_float(static_cast<uint32_t>(b) << 16); }

// hi = bf16(v), lo = bf16(v - hi): v - hi is exact in fp32.
__device__ inline void split2(float v, uint16_t& hi, uint16_t& lo) {
    hi = bf16_bits(v);
    lo = bf16_bits(v - bf16_value(hi));
}

// x [n] fp32 -> hi, lo bf16; 8 elements per thread (n % 8 == 0).
__global__ void __launch_bounds__(256)
k_split_bf16(const float* __restrict__ x, uint16_t* __restrict__ hi, uint16_t* __restrict__ lo, int64_t n8) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n8) return;
    const float4 a = reinterpret_cast<const float4*>(x)[2 * i];
    const float4 b = reinterpret_cast<const float4*>(x)[2 * i + 1];
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint16_t h[8], l[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) split2(v[j], h[j], l[j]);
    u32x4_t ph, pl;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        ph[j] = static_cast<uint32_t>(h[2 * j]) | (static_cast<uint32_t>(h[2 * j + 1]) << 16);
        pl[j] = static_cast<uint32_t>(l[2 * j]) | (static_cast<uint32_t>(l[2 * j + 1]) << 16);
    }
    reinterpret_cast<u32x4_t*>(hi)[i] = ph;
    reinterpret_cast<u32x4_t*>(lo)[i] = pl;
}

// W [N][K] fp32 -> images: image (nb * KT + kt) holds rows 128 nb .. + 127,
// k 32 kt .. + 31, swizzled: logical 16-byte chunks 0..3 of a row are hi, 4..7
// lo; rows past N are zero.  One thread per (hi, lo) element pair.
__global__ void __launch_bounds__(256)
k_pack_split(const float* __restrict__ w, uint16_t* __restrict__ img, int N, int K, int64_t pairs) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= pairs) return;
    const int KT = K / kTcK;
    const int kk = static_cast<int>(i & (kTcK - 1));
    const int r = static_cast<int>((i >> 5) & 127);   // image row
    const int64_t t = i >> 12;                        // image index nb * KT + kt
    const int64_t n = t / KT * 128 + r;
    const float v = n < N ? w[n * K + t % KT * kTcK + kk] : 0.0f;
    uint16_t h, l;
    split2(v, h, l);
    uint16_t* image = img + t * (kImageBytes / 2);
    image[swz(r, kk >> 3) / 2 + (kk & 7)] = h;
    image[swz(r, 4 + (kk >> 3)) / 2 + (kk & 7)] = l;
}

// The ring's operand format: 16 k per step, a fragment is the hi and the lo
// half of 32 rows x 16 k; three products (four with ALL) per fragment pair.
template <bool ALL>
struct SplitFmt {
    static constexpr int kSub = 2, kParts = 2, kProd = ALL ? 4 : 3;
    static constexpr int kAStep = kTcK * 2;   // x_hi and x_lo rows advance 32 k per stage
    struct frag_t {
        bf16x8_t h[2];   // hi, lo
    };
    __device__ static void load_part(frag_t& f, const uint8_t* st, int row, int kk, int lane, int part) {
        f.h[part] = __builtin_bit_cast(
            bf16x8_t, *reinterpret_cast<const u32x4_t*>(st + swz(row, 4 * part + 2 * kk + (lane >> 5))));
    }
    // products in the order x_hi W_hi, x_hi W_lo, x_lo W_hi, x_lo W_lo
    __device__ static f32x16_t mma(const frag_t& w, const frag_t& x, f32x16_t c, int prod) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(w.h[prod & 1], x.h[prod >> 1], c, 0, 0, 0);
    }
};

// Up to three outputs of one input (q, k and v): segment j is y[j]
// [M][n[j]] from packed weights w[j], column blocks t0[j] .. t0[j + 1] - 1 of
// the grid's x dimension.
struct TcSegs {
    const uint16_t* w[3];
    const float* b[3];
    float* y[3];
    int n[3];
    int t0[4];
};

// One-dimensional grid over the row-tile-major tile order, dealt to XCDs as
// k_linear_mfma's (workgroup b on XCD b % 8): tile b, or with xcd_rows tile
// (b % 8) * per + b / 8, so that the column tiles of a row tile share its x
// rows in one L2 (picked when x is the larger operand by 3x or more).
constexpr int kTcXcds = 8;

template <class Sh, bool ALL>
__global__ void __launch_bounds__(256, 1)
k_linear_tc(const uint16_t* __restrict__ xhi, const uint16_t* __restrict__ xlo, const TcSegs segs, int64_t M,
            int K, int row_tiles, int xcd_rows) {
    typedef PDims<Sh> D;
    typedef SplitFmt<ALL> Fmt;
    constexpr int MI = Sh::MI, NJ = Sh::NJ;
    static_assert(D::RA == kTcRows, "128-row blocks");
    __shared__ __align__(16) Ring3 ring;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ncol = segs.t0[3];
    const int64_t per = (static_cast<int64_t>(row_tiles) * ncol + kTcXcds - 1) / kTcXcds;
    const int64_t t = xcd_rows ? static_cast<int64_t>(blockIdx.x % kTcXcds) * per + blockIdx.x / kTcXcds
                               : static_cast<int64_t>(blockIdx.x);
    if (t >= static_cast<int64_t>(row_tiles) * ncol) return;
    const int64_t m0 = (t / ncol) * kTcRows;
    // this block's segment (selects, so the argument block stays in scalar registers)
    const int bx = static_cast<int>(t % ncol);
    const int sg = (bx >= segs.t0[1]) + (bx >= segs.t0[2]);
    const uint16_t* __restrict__ img = sg == 0 ? segs.w[0] : sg == 1 ? segs.w[1] : segs.w[2];
    const float* __restrict__ bias = sg == 0 ? segs.b[0] : sg == 1 ? segs.b[1] : segs.b[2];
    float* __restrict__ y = sg == 0 ? segs.y[0] : sg == 1 ? segs.y[1] : segs.y[2];
    const int N = sg == 0 ? segs.n[0] : sg == 1 ? segs.n[1] : segs.n[2];
    const int n0 = (bx - (sg == 0 ? segs.t0[0] : sg == 1 ? segs.t0[1] : segs.t0[2])) * D::RB;
    const int KT = K / kTcK, images = (N + 127) / 128;

    // A slots: chunks 0..3 of a stage row from x_hi, 4..7 from x_lo.  B slots:
    // 8 rows of an image, copied verbatim (a stage row and its image row share
    // their swizzle); images past the last re-read it.
    Slots sl;
#pragma unroll
    for (int s = 0; s < D::NS; ++s) {
        if (s < D::NA) {
            const int row = slot_row(s, wave, lane), c = slot_chunk(row, lane);
            const int64_t xr = m0 + row < M ? m0 + row : M - 1;
            sl.p[s] = reinterpret_cast<const uint8_t*>((c < 4 ? xhi : xlo) + xr * K + 8 * (c & 3));
        } else {
            const int col = n0 + 32 * (s - D::NA) + 8 * wave;   // the slot's first output column
            const int im = col / 128 < images ? col / 128 : images - 1;
            sl.p[s] = reinterpret_cast<const uint8_t*>(img) + static_cast<int64_t>(im) * KT * kImageBytes +
                      (col % 128) * kRowBytes + lane * 16;
        }
    }
    const int aR = (wave % Sh::WM) * MI * 32, bR = (wave / Sh::WM) * NJ * 32;
    f32x16_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x16_t{};
    pmainloop<Sh, Fmt>(ring, sl, KT, wave, lane, aR, D::RA + bR, acc);

    // W first in the MFMA: lane % 32 is an x row, register group q = v / 4
    // holds output columns 8 q + 4 (lane / 32) .. +3 of the 32-column tile
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int64_t row = m0 + aR + 32 * i + (lane & 31);
        if (row >= M) continue;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int col = n0 + bR + 32 * j + 8 * q + 4 * (lane >> 5);
                if (col >= N) continue;   // N % 4 == 0: a group is all in or all out
                float4 o = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                                       acc[i][j][4 * q + 3]);
                if (bias) {
                    const float4 b = *reinterpret_cast<const float4*>(bias + col);
                    o = make_float4(__fadd_rn(o.x, b.x), __fadd_rn(o.y, b.y), __fadd_rn(o.z, b.z), __fadd_rn(o.w, b.w));
                }
                *reinterpret_cast<float4*>(y + row * N + col) = o;
            }
    }
}

}  // namespace

int64_t linear_tc_packed_elems(int out_f, int in_f) {
    // ceil(out / 128) * (in / 32) images of 128 rows x (32 hi + 32 lo)
    return ceil_div(out_f, 128) * (in_f / kTcK) * 128 * 64;
}

hipError_t launch_linear_tc_prepare(const float* w, int out_f, int in_f, uint16_t* packed, hipStream_t s) {
    if (out_f <= 0 || in_f <= 0 || in_f % 64 != 0) return hipErrorInvalidValue;
    const int64_t pairs = linear_tc_packed_elems(out_f, in_f) / 2;
    hipLaunchKernelGGL(k_pack_split, dim3(static_cast<unsigned>(ceil_div(pairs, 256))), dim3(256), 0, s, w, packed,
                       out_f, in_f, pairs);
    return hipGetLastError();
}

hipError_t launch_split_bf16(const float* x, int64_t n, uint16_t* hi, uint16_t* lo, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (n % 8 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_split_bf16, dim3(static_cast<unsigned>(ceil_div(n / 8, 256))), dim3(256), 0, s, x, hi, lo,
                       n / 8);
    return hipGetLastError();
}

hipError_t launch_linear_tc_multi(const uint16_t* xhi, const uint16_t* xlo, int count, const uint16_t* const* packed,
                                  const float* const* bias, float* const* y, const int* out_f, int64_t rows, int in_f,
                                  bool all_terms, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (count < 1 || count > 3 || in_f <= 0 || in_f % 64 != 0 || ceil_div(rows, kTcRows) > 65535)
        return hipErrorInvalidValue;
    // The block width whose busiest CU is done first: blocks per CU x the time
    // of one, relative to a 64-column block.  Measured (four products), q, k
    // and v of K = 4096 at 64 / 128 / 256 columns: 512 rows 64 / 84 / 150 us, 1,024
    // rows 125 / 99 / 158, 2,048 rows 201 / 195 / 178, 4,096 rows 392 / 323 / 350, 10,240
    // rows 1085 / 861 / 819; the output projection at 4,096 rows 276 / 224 / 213;
    // the LM head on 8 rows 142 / 104 / 147.
    const int64_t cus = num_cus(), rt = ceil_div(rows, kTcRows);
    auto cost = [&](int bc, double block) {
        int64_t t = 0;
        for (int j = 0; j < count; ++j) t += ceil_div(out_f[j], bc);
        return static_cast<double>(ceil_div(rt * t, cus)) * block;
    };
    const double c256 = cost(256, 2.65), c128 = cost(128, 1.55), c64 = cost(64, 1.0);
    const int bc = c256 <= c128 && c256 <= c64 ? 256 : c128 <= c64 ? 128 : 64;
    TcSegs segs{};
    int t = 0;
    for (int j = 0; j < 3; ++j) {
        segs.t0[j] = t;
        const int jj = j < count ? j : 0;   // unused segments: never selected (their t0 is the tile count)
        if (out_f[jj] <= 0 || out_f[jj] % 4 != 0) return hipErrorInvalidValue;
        segs.w[j] = packed[jj];
        segs.b[j] = bias[jj];
        segs.y[j] = y[jj];
        segs.n[j] = out_f[jj];
        if (j < count) t += static_cast<int>(ceil_div(out_f[j], bc));
    }
    segs.t0[3] = t;
    for (int j = count; j < 3; ++j) segs.t0[j] = t;
    int64_t wcols = 0;
    for (int j = 0; j < count; ++j) wcols += out_f[j];
    const int xr = rows >= 3 * wcols ? 1 : 0;   // x bytes >= 3 x W bytes (both hi + lo bf16)
    const dim3 grid(static_cast<unsigned>(ceil_div(rt * t, kTcXcds) * kTcXcds));
#define APS_TC_LAUNCH(KIND)                                                                                            \
    do {                                                                                                               \
        if (all_terms)                                                                                                 \
            hipLaunchKernelGGL((k_linear_tc<PShape<KIND>, true>), grid, dim3(256), 0, s, xhi, xlo, segs, rows, in_f,   \
                               static_cast<int>(rt), xr);                                                              \
        else                                                                                                           \
            hipLaunchKernelGGL((k_linear_tc<PShape<KIND>, false>), grid, dim3(256), 0, s, xhi, xlo, segs, rows, in_f,  \
                               static_cast<int>(rt), xr);                                                              \
    } while (0)
    if (bc == 256) APS_TC_LAUNCH(kPieceW);
    else if (bc == 128) APS_TC_LAUNCH(kPieceS);
    else APS_TC_LAUNCH(kPieceQ);
#undef APS_TC_LAUNCH
    return hipGetLastError();
}

hipError_t launch_linear_tc(const uint16_t* xhi, const uint16_t* xlo, const uint16_t* packed, const float* bias,
                            float* y, int64_t rows, int in_f, int out_f, bool all_terms, hipStream_t s) {
    return launch_linear_tc_multi(xhi, xlo, 1, &packed, &bias, &y, &out_f, rows, in_f, all_terms, s);
}

}  // namespace aps
