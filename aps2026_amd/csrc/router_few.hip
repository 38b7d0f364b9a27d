// Router for few tokens: the logits, routes and x copies of router.hip, bit
// for bit, one workgroup per token.
//
// The logits are the same serial FMA chains (router.hip has the reference and
// the reason), so the time is one chain's latency however few the tokens.
// With few tokens there are more lanes than chains: a chain (token, expert)
// takes the 16 lanes of a DPP row.  Lane i holds elements 32 i .. 32 i + 31 of each
// 512-step chunk of x and of the expert's gate row, and the accumulator walks
// through the lanes as in layernorm.hip: every lane runs 32 FMAs on its own
// registers 16 times over, the accumulators rotating one lane (row_ror:1)
// before each round.  A step is one v_fmac on registers, without the LDS read
// per four steps and the stage barriers of the token-major kernel, and the
// loop is short: straight-line code of a whole stage is fetched for every
// launch here and runs once.
//   Bound by the chain (4096 steps: 11 us).  Measured at H = 4096, against the
// token-major kernel: bf16 x 19 -> 14 us, with its fp8 codes 27 -> 15.5 us, fp32 x 24
// -> 16 us; any count up to 256 tokens.  Past that workgroups share SIMDs (bf16
// block of 300 tokens 81 -> 88 us, 613 85 -> 105).
//   A workgroup's four waves are the 16 experts of one token.  The fp8 codes
// of x come from further workgroups of the same launch, beside the chains
// instead of after them.
#include "chain_mfma.hpp"

namespace aps {
namespace {

constexpr int kRfElems = 32;                  // chain steps per lane and chunk
constexpr int kRfChunk = 16 * kRfElems;       // 512
constexpr int kRfMaxE = 16;

typedef uint32_t rf_u4 __attribute__((ext_vector_type(4)));
typedef float rf_f4 __attribute__((ext_vector_type(4)));

// This lane's operands of a chunk.
template <bool XBF16>
struct RfRegs {
    static constexpr int kX = kRfElems * (XBF16 ? 2 : 4) / 16;   // 16-byte pieces of x
    rf_f4 g[kRfElems / 4];
    rf_u4 x[kX];
};

// fp32 x: a wave's ring slot holds the chunk of its four gate rows and of x (16
// lanes x 128 bytes each), copied whole lines at a time; the 16-byte pieces are
// swizzled so that 16 lanes reading theirs hit 16 different bank groups.
struct RfSlot {
    static constexpr int kCopies = 10;   // per wave and chunk
    uint8_t row[5][16 * 128];            // gate rows, x
    // physical piece of lane i's logical piece p
    __device__ static int piece(int i, int p) { return p ^ ((i >> 1) & 7); }
};

// Blocks 0 .. rows - 1: one token each; with xq, four rows of x per further block.
template <bool XBF16>
__global__ void __launch_bounds__(256)
k_router_few(const void* __restrict__ xv, const float* __restrict__ gate, int64_t rows, int H, int E,
             float* __restrict__ logits, uint8_t* __restrict__ routes, bf16_t* __restrict__ xcopy,
             uint8_t* __restrict__ xq, float* __restrict__ xq_scale) {
    constexpr int kElt = XBF16 ? 2 : 4;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (blockIdx.x >= rows) {   // block-uniform
        if constexpr (XBF16) {
            const int64_t row = (blockIdx.x - rows) * 4 + wave;
            if (row < rows)
                e4m3_quant_row<8>(static_cast<const bf16_t*>(xv) + row * H, H, xq + row * H, H, xq_scale + row, lane);
        }
        return;
    }
    // one LDS object, a ring per wave (no barriers): with a second object the
    // compiler tracks the copies and waits for all of them before each read
    __shared__ __align__(16) RfSlot ring[XBF16 ? 1 : 4][XBF16 ? 1 : 3];
    float* lg = reinterpret_cast<float*>(&ring[0][0]);   // after the chains
    const int64_t t = blockIdx.x;
    const int i = lane & 15, row = lane >> 4, e = 4 * wave + row;
    const int NC = H / kRfChunk;
    float acc = 0.0f;
    auto chain = [&](const RfRegs<XBF16>& d, int c) __attribute__((always_inline)) {
        float xe[kRfElems];
#pragma unroll
        for (int k = 0; k < kRfElems; ++k) {
            if constexpr (XBF16) {
                const uint32_t w = d.x[k / 8][k % 8 / 2];
                xe[k] = k % 2 ? bf16w_hi(w) : bf16w_lo(w);
            } else {
                xe[k] = __uint_as_float(d.x[k / 4][k % 4]);
            }
        }
        if constexpr (!XBF16) {
            // the FFN's bf16 copy: each chunk by one row of wave 0
            if (xcopy && wave == 0 && row == (c & 3)) {
#pragma unroll
                for (int k = 0; k < kRfElems; k += 8)
                    *reinterpret_cast<rf_u4*>(xcopy + t * H + c * kRfChunk + kRfElems * i + k) =
                        rf_u4{pack2_bf16(xe[k], xe[k + 1]), pack2_bf16(xe[k + 2], xe[k + 3]),
                              pack2_bf16(xe[k + 4], xe[k + 5]), pack2_bf16(xe[k + 6], xe[k + 7])};
            }
        }
#pragma unroll 1
        for (int r = 0; r < 16; ++r) {
            acc = row_ror1(acc);
#pragma unroll
            for (int k = 0; k < kRfElems; ++k) acc = __fmaf_rn(xe[k], d.g[k / 4][k % 4], acc);
        }
    };
    // Operands one chunk ahead of the chain.  Chunks past the end re-read the
    // last, so that every load and copy is unconditional and can be counted.
    RfRegs<XBF16> regs[2];
    if constexpr (XBF16) {
        // straight into registers, two chunks in flight
        const uint8_t* xsrc = static_cast<const uint8_t*>(xv) + (t * H + kRfElems * i) * kElt;
        const float* gsrc = gate + static_cast<int64_t>(e < E ? e : E - 1) * H + kRfElems * i;
        auto load = [&](RfRegs<XBF16>& d, int c) __attribute__((always_inline)) {
            c = c < NC ? c : NC - 1;
#pragma unroll
            for (int k = 0; k < RfRegs<XBF16>::kX; ++k)
                d.x[k] = *reinterpret_cast<const rf_u4*>(xsrc + c * kRfChunk * kElt + 16 * k);
#pragma unroll
            for (int k = 0; k < kRfElems / 4; ++k) d.g[k] = *reinterpret_cast<const rf_f4*>(gsrc + c * kRfChunk + 4 * k);
            __builtin_amdgcn_sched_barrier(0);
        };
        load(regs[0], 0);
        load(regs[1], 1);
        for (int c = 0; c < NC; c += 2) {
            chain(regs[0], c);
            __builtin_amdgcn_sched_barrier(0);
            load(regs[0], c + 2);
            if (c + 1 < NC) {   // wave-uniform
                chain(regs[1], c + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            load(regs[1], c + 3);
        }
        __syncthreads();
    } else {
        // through the ring: with twice the x, loads of 64 separate lines an
        // instruction took longer than the chain (20 us against 16)
        // copy j covers half a row, lanes 8 (j % 2) .. + 7 of row j / 2: this copy
        // lane's source is the piece that its place holds
        const uint8_t* src[RfSlot::kCopies];
#pragma unroll
        for (int j = 0; j < RfSlot::kCopies; ++j) {
            const int ge = 4 * wave + j / 2, l = 8 * (j & 1) + (lane >> 3);
            const uint8_t* base = j < 8 ? reinterpret_cast<const uint8_t*>(gate + static_cast<int64_t>(ge < E ? ge : E - 1) * H)
                                        : static_cast<const uint8_t*>(xv) + t * H * kElt;
            src[j] = base + 128 * l + 16 * RfSlot::piece(l, lane & 7);
        }
        auto issue = [&](int c) __attribute__((always_inline)) {
            uint8_t* to = &ring[wave][c % 3].row[0][0];
            c = c < NC ? c : NC - 1;
#pragma unroll
            for (int j = 0; j < RfSlot::kCopies; ++j)
                __builtin_amdgcn_global_load_lds(APS_CGP(src[j] + c * 4 * kRfChunk), APS_CLP(to + 1024 * j), 16, 0, 0);
        };
        // (by LDS address: through the ring object the compiler would wait for
        // every copy in flight before each read)
        typedef const __attribute__((address_space(3))) rf_f4* lds_f4;
        typedef const __attribute__((address_space(3))) rf_u4* lds_u4;
        const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(APS_CLP(&ring[wave][0]))) + 128u * i;
        auto read = [&](RfRegs<XBF16>& d, int c) __attribute__((always_inline)) {
            const uint32_t s = base + (c % 3) * static_cast<uint32_t>(sizeof(RfSlot));
#pragma unroll
            for (int p = 0; p < kRfElems / 4; ++p)
                d.g[p] = *reinterpret_cast<lds_f4>(s + (2048u * row + 16u * RfSlot::piece(i, p)));
#pragma unroll
            for (int p = 0; p < RfRegs<XBF16>::kX; ++p)
                d.x[p] = *reinterpret_cast<lds_u4>(s + (8192u + 16u * RfSlot::piece(i, p)));
        };
        // chunk c: chunk c + 1's copies have landed when at most those of c + 2 are
        // in flight (stores of x copies in between are waited for too); its
        // operands are read under the chain, and chunk c + 3 takes c's slot
        issue(0);
        issue(1);
        issue(2);
        chain_wait_vm<2 * RfSlot::kCopies>();
        __builtin_amdgcn_wave_barrier();
        read(regs[0], 0);
        auto step = [&](auto par, int c) __attribute__((always_inline)) {
            constexpr int P = decltype(par)::value;
            chain_wait_vm<RfSlot::kCopies>();
            chain_wait_lgkm0();   // chunk c's reads: its slot is free
            __builtin_amdgcn_sched_barrier(0);
            issue(c + 3);
            read(regs[P ^ 1], c + 1);
            __builtin_amdgcn_sched_barrier(0);
            chain(regs[P], c);
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int c = 0; c < NC; c += 2) {
            step(std::integral_constant<int, 0>{}, c);
            if (c + 1 < NC) step(std::integral_constant<int, 1>{}, c + 1);   // wave-uniform
        }
        chain_wait_vm<0>();   // no copy outlives its slot
        __syncthreads();   // every wave has read its chunks: lg takes a slot
    }
    // the row's last lane holds the logit
    if (i == 15) {
        lg[e] = acc;
        if (e < E) logits[t * E + e] = acc;
    }
    __syncthreads();
    if (wave != 0) return;
    const float q = route_quantise(lg[i]);
    float qs[kRfMaxE];
#pragma unroll
    for (int k = 0; k < kRfMaxE; ++k)
        qs[k] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, q), k));
    int first, second;
    route_greedy_top2<kRfMaxE>(qs, E, first, second);
    if (lane == 0) {
        routes[2 * t] = static_cast<uint8_t>(first);
        routes[2 * t + 1] = static_cast<uint8_t>(second);
    }
}

}  // namespace

bool router_few_fits(int64_t rows, int hidden, int experts) {
    return rows <= kDispatchFewRows && experts >= 2 && experts <= kRfMaxE && hidden % kRfChunk == 0;
}

hipError_t launch_router_few(const void* x, bool x_bf16, const float* gate, int64_t rows, int hidden, int experts,
                             float* logits, uint8_t* routes, bf16_t* x_copy, uint8_t* xq, float* xq_scale,
                             hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (!router_few_fits(rows, hidden, experts) || (x_copy && x_bf16) || (xq && (!x_bf16 || !xq_scale || hidden > 4096)))
        return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(rows + (xq ? ceil_div(rows, 4) : 0)));
    if (x_bf16)
        hipLaunchKernelGGL(k_router_few<true>, grid, dim3(256), 0, s, x, gate, rows, hidden, experts, logits, routes,
                           x_copy, xq, xq_scale);
    else
        hipLaunchKernelGGL(k_router_few<false>, grid, dim3(256), 0, s, x, gate, rows, hidden, experts, logits, routes,
                           x_copy, xq, xq_scale);
    return hipGetLastError();
}

}  // namespace aps
