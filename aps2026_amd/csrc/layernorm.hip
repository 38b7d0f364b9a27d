// LayerNorm of the decoder layer, the producer of the MoE block's input:
// y = (v - mean) * inv * w + b with v = x (+ residual, written back to x).
//
// Reference: k_layer_norm / k_add_layer_norm (src/tensor.cu:2121-2178) with
// ln_moments, ln_serial_sum, ln_serial_var and ln_write (src/tensor.cu:
// 2032-2119).  Both row sums run on ONE thread in ascending j, because the
// router downstream quantises its logits at 1e-3 with a 2e-2 tie margin and a
// last-ulp change of a LayerNorm output can flip an expert.  The arithmetic,
// operation for operation (nvcc contracts `var += t * t` and `... * w + b`):
//   sum  = fp32 adds of v[j], j ascending       mean = sum / h
//   var  = fma(t, t, var), t = v[j] - mean      inv  = 1 / sqrt(var / h + eps)
//   y[j] = fma((v[j] - mean) * inv, w[j], b[j])
// (this library is built with -ffp-contract=off and IEEE division / square
// root, so every other operation is rounded on its own).
//
// gfx950 mapping.  The sums are dependent chains of h additions: their length,
// not bandwidth, sets the time, and only one lane can hold a row's sum.  A row
// belongs to the 16 lanes of a DPP row (a wave owns 4 rows): lane i holds the
// elements 16 i .. 16 i + 15 of each 256-column chunk, and the running sum
// walks through the lanes.  Every lane runs the same 16 additions on its own
// registers 16 times over; before each round the accumulators rotate one lane
// (DPP row_ror:1, folded into the add in pass 1), so after round i lane i's
// accumulator is the sum up to its last element and the others' are unused.
// A step is one vector instruction on registers, with no LDS reads and no
// broadcasts, and the deviation v - mean, elementwise, is taken 16 lanes at a
// time before the variance chain.
//   A row of 16 chunks (h = 4096) stays in its lanes' registers from the first
// load to the last store (256 VGPRs, one wave per SIMD), so x is read once;
// other widths stream the chunks again for each pass.
//   Bound by the two chains up to one wave per SIMD (4,096 rows), by the row
// traffic with them past that.  Measured at h = 4096 (with the residual):
// 43 rows 27 (29) us, 4,096 rows 39 (52), 10,240 rows 99 (149: 4.5 TB/s).
// One lane per row reading staged rows from LDS four values at a time, three
// passes over memory, took 64 (65), 78 (80), 162 (193) us; loading and storing
// in the chains' layout (64 bytes apart across lanes) 28 (29), 49 (69), 123
// (182) us.  Streamed widths, at 16,384 rows, one lane per row -> chains' layout
// -> here: h = 256 10 -> 16 -> 8.5 (14 -> 21 -> 12) us, 768 29 -> 35 -> 22 (46 -> 51
// -> 44), 2048 95 -> 82 -> 62 (131 -> 149 -> 127), 5120 242 -> 269 -> 206 (386 -> 410
// -> 355); at 64 rows, h = 512, 10 -> 5.0 -> 5.3 (8.6 -> 5.4 -> 5.8).
#include "common.hpp"

namespace aps {
namespace {

constexpr int kLnRows = 4;       // rows per wave, one per 16-lane DPP row
constexpr int kLnElems = 16;     // consecutive elements per lane and chunk
constexpr int kLnChunk = 256;    // columns per chunk (16 lanes x 16 elements)
constexpr int kLnResident = 16;  // chunks of a row that stays in registers
constexpr int kLnAhead = 4;      // chunks of loads in flight

typedef float lf4 __attribute__((ext_vector_type(4)));

// lane 15's value in every lane of its row
__device__ inline float ln_last(float v) {
    const int i = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, 0x15F, 0xF, 0xF, true));
}

struct LnChunk {
    lf4 q[kLnElems / 4];
};

// The chains over one chunk: on entry lane 15 (or, at the first chunk, every
// lane) holds the sum so far, on exit lane 15 holds the new one.
__device__ inline float ln_sum(float acc, const LnChunk& v) {
#pragma unroll 4
    for (int i = 0; i < 16; ++i) {
        acc = __fadd_rn(row_ror1(acc), v.q[0][0]);
#pragma unroll
        for (int e = 1; e < kLnElems; ++e) acc = __fadd_rn(acc, v.q[e / 4][e % 4]);
    }
    return acc;
}
__device__ inline float ln_sum_sq(float acc, const LnChunk& t) {
#pragma unroll 4
    for (int i = 0; i < 16; ++i) {
        acc = row_ror1(acc);
#pragma unroll
        for (int e = 0; e < kLnElems; ++e) acc = __fmaf_rn(t.q[e / 4][e % 4], t.q[e / 4][e % 4], acc);
    }
    return acc;
}

__device__ inline lf4 ln_add(lf4 v, lf4 r) {
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = __fadd_rn(v[k], r[k]);
    return v;
}
__device__ inline void ln_deviation(LnChunk& v, float mean) {
#pragma unroll
    for (int p = 0; p < kLnElems / 4; ++p)
#pragma unroll
        for (int k = 0; k < 4; ++k) v.q[p][k] = __fsub_rn(v.q[p][k], mean);
}
__device__ inline float ln_inv(float var, int h, float eps) {
    // sqrtf, not __fsqrt_rn: under -fhip-fp32-correctly-rounded-divide-sqrt
    // sqrtf is correctly rounded (v_sqrt_f32 plus a neighbour check),
    // while __fsqrt_rn lowers to the bare v_sqrt_f32, off by an ulp at
    // times (rows of a GPU test disagreed with the oracle by one ulp)
    return __fdiv_rn(1.0f, sqrtf(__fadd_rn(__fdiv_rn(var, static_cast<float>(h)), eps)));
}

// row k's value, from its DPP row, in every lane
__device__ inline float ln_row(float v, int k) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 16 * k));
}

// Memory is read and written whole 1 KB row chunks at a time (lane s holds 16
// bytes of each of the 4 rows); LDS turns a chunk between that layout and the
// chains' (64 consecutive bytes of one row per lane).  Lane s's 16 bytes are
// columns io .. io + 3 of the chunk, slot s; the piece p of chain lane L lies in
// slot 4 L + (p ^ (L / 4)), so that 16 chain lanes read 16 different bank groups.
__device__ inline int ln_slot(int p) {
    const int L = threadIdx.x & 15;
    return 4 * L + (p ^ (L >> 2));
}
__device__ inline void ln_turned(LnChunk& v, const lf4 (&turn)[kLnRows][64]) {
#pragma unroll
    for (int p = 0; p < 4; ++p) v.q[p] = turn[threadIdx.x >> 4][ln_slot(p)];
}
struct LnLane {
    int s, io, nr;
    int64_t at[kLnRows];   // rows past the end load the last one and store nothing
    __device__ LnLane(int64_t rows, int h) {
        s = threadIdx.x;
        io = 16 * (s >> 2) + 4 * ((s & 3) ^ ((s >> 4) & 3));
        const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kLnRows;
        nr = rows - r0 < kLnRows ? static_cast<int>(rows - r0) : kLnRows;   // wave-uniform
#pragma unroll
        for (int k = 0; k < kLnRows; ++k) at[k] = (r0 + (k < nr ? k : nr - 1)) * h + io;
    }
};

// h = 4096: the row in registers throughout.
template <bool ADD>
__global__ void __launch_bounds__(64, 1)
k_layer_norm_resident(float* __restrict__ x, const float* __restrict__ residual, const float* __restrict__ w,
                      const float* __restrict__ b, float* __restrict__ y, int64_t rows, float eps) {
    constexpr int NC = kLnResident, h = NC * kLnChunk;
    __shared__ lf4 turn[2][kLnRows][64];
    const LnLane l(rows, h);
    const int s = l.s, io = l.io, nr = l.nr;
    const int64_t (&at)[kLnRows] = l.at;
    auto ld = [](const float* p) __attribute__((always_inline)) { return *reinterpret_cast<const lf4*>(p); };

    LnChunk v[NC];
    lf4 xs[kLnAhead][kLnRows], rs[ADD ? kLnAhead : 1][kLnRows];
    auto load = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kLnRows; ++k) {
            xs[c % kLnAhead][k] = ld(x + at[k] + c * kLnChunk);
            if (ADD) rs[c % kLnAhead][k] = ld(residual + at[k] + c * kLnChunk);
        }
        __builtin_amdgcn_sched_barrier(0);   // chunk order, so that a chunk's wait leaves the later ones in flight
    };
    // chunk c as it was loaded (+ residual, written back to x) into its chain lanes' registers
    auto take = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kLnRows; ++k) {
            lf4 u = xs[c % kLnAhead][k];
            if (ADD) {
                u = ln_add(u, rs[c % kLnAhead][k]);
                if (k < nr) *reinterpret_cast<lf4*>(x + at[k] + c * kLnChunk) = u;
            }
            turn[c & 1][k][s] = u;
        }
        __builtin_amdgcn_wave_barrier();
        ln_turned(v[c], turn[c & 1]);
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int c = 0; c < kLnAhead; ++c) load(c);
    take(0);
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if (c + kLnAhead < NC) load(c + kLnAhead);
        if (c + 1 < NC) take(c + 1);
        acc = ln_sum(acc, v[c]);
        __builtin_amdgcn_sched_barrier(0);
    }
    const float mean = __fdiv_rn(ln_last(acc), static_cast<float>(h));
    // w and b in the loads' layout, the first chunks' under the variance chain
    lf4 wv[kLnAhead], bv[kLnAhead];
    auto load_wb = [&](int c) __attribute__((always_inline)) {
        wv[c % kLnAhead] = ld(w + c * kLnChunk + io);
        bv[c % kLnAhead] = ld(b + c * kLnChunk + io);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int c = 0; c < kLnAhead; ++c) load_wb(c);
    float var = 0.0f;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        ln_deviation(v[c], mean);
        var = ln_sum_sq(var, v[c]);
        __builtin_amdgcn_sched_barrier(0);
    }
    const float inv_row = ln_inv(ln_last(var), h, eps);
    float inv[kLnRows];
#pragma unroll
    for (int k = 0; k < kLnRows; ++k) inv[k] = ln_row(inv_row, k);
    // chunk c of t into the loads' layout, one chunk ahead of its use
    lf4 t[2][kLnRows];
    auto turn_back = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 4; ++p) turn[c & 1][s >> 4][ln_slot(p)] = v[c].q[p];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < kLnRows; ++k) t[c & 1][k] = turn[c & 1][k][s];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    turn_back(0);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if (c + 1 < NC) turn_back(c + 1);
#pragma unroll
        for (int k = 0; k < kLnRows; ++k) {
            lf4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[j] = __fmaf_rn(__fmul_rn(t[c & 1][k][j], inv[k]), wv[c % kLnAhead][j], bv[c % kLnAhead][j]);
            if (k < nr) *reinterpret_cast<lf4*>(y + at[k] + c * kLnChunk) = o;
        }
        if (c + kLnAhead < NC) load_wb(c + kLnAhead);
    }
}

// Any h (a multiple of 256): the chunks are read again for each pass, AHEAD of
// them in flight, in the same layout; only the two chains' passes turn them.
template <bool ADD, int AHEAD>
__global__ void __launch_bounds__(64)
k_layer_norm(float* __restrict__ x, const float* __restrict__ residual, const float* __restrict__ w,
             const float* __restrict__ b, float* __restrict__ y, int64_t rows, int h, float eps) {
    __shared__ lf4 turn[2][kLnRows][64];
    const LnLane l(rows, h);
    const int NC = h / kLnChunk;
    auto ld = [](const float* p) __attribute__((always_inline)) { return *reinterpret_cast<const lf4*>(p); };
    // f(c, x of chunk c, a second operand of chunk c loaded by also); loads past
    // the end re-read the last chunk, so that every load is unconditional and a
    // chunk's wait leaves the later ones in flight
    auto each = [&](auto also, auto f) __attribute__((always_inline)) {
        lf4 xs[AHEAD][kLnRows];
        decltype(also(0)) as[AHEAD];
        auto load = [&](int d, int c) __attribute__((always_inline)) {
            c = c < NC ? c : NC - 1;
#pragma unroll
            for (int k = 0; k < kLnRows; ++k) xs[d][k] = ld(x + l.at[k] + c * kLnChunk);
            as[d] = also(c);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) load(d, d);
        for (int c0 = 0; c0 < NC; c0 += AHEAD) {
#pragma unroll
            for (int d = 0; d < AHEAD; ++d) {
                if (c0 + d >= NC) break;   // wave-uniform
                f(c0 + d, xs[d], as[d]);
                load(d, c0 + d + AHEAD);
            }
        }
    };
    struct Four {
        lf4 r[kLnRows];
    };
    struct None {};
    const auto none = [](int) { return None{}; };
    auto turned = [&](int c, const lf4 (&u)[kLnRows]) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kLnRows; ++k) turn[c & 1][k][l.s] = u[k];
        __builtin_amdgcn_wave_barrier();
        LnChunk v;
        ln_turned(v, turn[c & 1]);
        __builtin_amdgcn_wave_barrier();
        return v;
    };
    float acc = 0.0f;
    if constexpr (ADD) {
        each([&](int c) __attribute__((always_inline)) {
            Four r;
#pragma unroll
            for (int k = 0; k < kLnRows; ++k) r.r[k] = ld(residual + l.at[k] + c * kLnChunk);
            return r;
        }, [&](int c, lf4 (&u)[kLnRows], const Four& r) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < kLnRows; ++k) {
                u[k] = ln_add(u[k], r.r[k]);
                if (k < l.nr) *reinterpret_cast<lf4*>(x + l.at[k] + c * kLnChunk) = u[k];
            }
            acc = ln_sum(acc, turned(c, u));
        });
    } else {
        each(none, [&](int c, lf4 (&u)[kLnRows], None) __attribute__((always_inline)) { acc = ln_sum(acc, turned(c, u)); });
    }
    const float mean = __fdiv_rn(ln_last(acc), static_cast<float>(h));
    float var = 0.0f;
    each(none, [&](int c, lf4 (&u)[kLnRows], None) __attribute__((always_inline)) {
        LnChunk v = turned(c, u);
        ln_deviation(v, mean);
        var = ln_sum_sq(var, v);
    });
    const float inv_row = ln_inv(ln_last(var), h, eps);
    float m[kLnRows], inv[kLnRows];
#pragma unroll
    for (int k = 0; k < kLnRows; ++k) {
        m[k] = ln_row(mean, k);
        inv[k] = ln_row(inv_row, k);
    }
    struct Two {
        lf4 w, b;
    };
    each([&](int c) __attribute__((always_inline)) {
        return Two{ld(w + c * kLnChunk + l.io), ld(b + c * kLnChunk + l.io)};
    }, [&](int c, lf4 (&u)[kLnRows], const Two& p) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < kLnRows; ++k) {
            lf4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[j] = __fmaf_rn(__fmul_rn(__fsub_rn(u[k][j], m[k]), inv[k]), p.w[j], p.b[j]);
            if (k < l.nr) *reinterpret_cast<lf4*>(y + l.at[k] + c * kLnChunk) = o;
        }
    });
}

}  // namespace

hipError_t launch_layer_norm(float* x, const float* residual, const float* weight, const float* bias, float* y,
                             int64_t rows, int hidden, float eps, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (hidden <= 0 || hidden % kLnChunk != 0) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(ceil_div(rows, kLnRows)));
    if (hidden == kLnResident * kLnChunk) {
        if (residual)
            hipLaunchKernelGGL(k_layer_norm_resident<true>, grid, dim3(64), 0, s, x, residual, weight, bias, y, rows, eps);
        else
            hipLaunchKernelGGL(k_layer_norm_resident<false>, grid, dim3(64), 0, s, x, residual, weight, bias, y, rows, eps);
    } else {
        const int nc = hidden / kLnChunk;
        auto kern = residual ? (nc == 1 ? k_layer_norm<true, 1> : nc < 4 ? k_layer_norm<true, 2> : k_layer_norm<true, 4>)
                             : (nc == 1 ? k_layer_norm<false, 1> : nc < 4 ? k_layer_norm<false, 2> : k_layer_norm<false, 4>);
        hipLaunchKernelGGL(kern, grid, dim3(64), 0, s, x, residual, weight, bias, y, rows, hidden, eps);
    }
    return hipGetLastError();
}

}  // namespace aps
