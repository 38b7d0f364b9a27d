// fp32 FMA chains on the matrix cores, shared by the kernels that must give
// the reference's bits: one accumulator per output, k ascending, one fused
// multiply-add per step.
//
// gfx950's v_mfma_f32_16x16x4_f32 and v_mfma_f32_32x32x2_f32 add their four
// (two) products to the accumulator one after the other, k ascending, with
// one rounding each: a sequence of them over k IS the fmaf chain.  Checked on
// gfx950 over 4096-step chains against fmaf on the host: operands N(0, 1),
// with exponents spread over 2^-20 .. 2^20, with products around FLT_MIN and
// with cancelling terms: no output of 256 (1024) differs, while 149 to 247 of
// 256 differ from the unfused chain.
//
// Rates measured (cycles per instruction, dependent accumulators included):
// 16x16x4 32, 32x32x2 64, so both run at the fp32 matrix rate of 256 FLOP per
// clock per CU, and one 16x16x4 advances 256 chains by four steps in 32
// cycles: 8 cycles per chain step, where a dependent v_fmac chain takes 6.1 to
// 6.3 (measured) for 64 chains.  The K = 1 forms run at the same rate but read
// every B operand twice (two or four blocks share it).
//
// What a kernel around them has to know (measured, one and two waves per
// SIMD): vector ALU instructions do NOT run beside an fp32 MFMA, of the same
// wave or another's.  Each one between two MFMAs adds its 4 cycles (8 for a
// v_permlane swap) and the first after an MFMA about 12 more; LDS reads,
// direct-to-LDS copies, scalar instructions and waits cost nothing.  So the
// operands come out of LDS in MFMA order, one ds_read_b32 per operand and
// step, from addresses that are registers plus immediates: no lane
// transposes, no address arithmetic in the loop.
//
// Operand layout: lane l holds row (A) or column (B) l % 16 (l % 32) at k =
// l / 16 (l / 32) of the step; register v of the result is row 4 (l / 16) +
// v, column l % 16 (16x16x4), row 8 (v / 4) + 4 (l / 32) + v % 4, column
// l % 32 (32x32x2).
#pragma once

#include "common.hpp"

#include <type_traits>
#include <utility>

namespace aps {

typedef float cf4_t __attribute__((ext_vector_type(4)));
typedef float cf16_t __attribute__((ext_vector_type(16)));

#define APS_CGP(p) ((const __attribute__((address_space(1))) void*)(p))
#define APS_CLP(p) ((__attribute__((address_space(3))) void*)(p))

// Byte offset of 16-byte chunk `chunk` of 128-byte stage row `row` (32 k of
// fp32): XOR-swizzled by row pair, so that the 16 lanes of an operand read
// (16 consecutive rows, one chunk) hit 16 distinct bank groups.
__device__ inline int chain_swz(int row, int chunk) { return row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4); }

template <int N>
__device__ inline void chain_wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (0xF << 8) | ((N >> 4) << 14));
}

// Every LDS read issued so far has returned.  Stated before the next reads go
// out, it keeps the compiler from waiting for those as well: with
// direct-to-LDS copies in flight it only ever waits for lgkmcnt(0).
__device__ inline void chain_wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xF | (0x7 << 4) | (0x0 << 8) | (0x3 << 14)); }

// acc[i][j] of each wave = the chains over k = 0 .. 32 KT - 1 of its RT x CT
// tiles of 16 x 16 outputs, in a workgroup of WR x WC waves: 16 RT WR rows (A)
// against 16 CT WC columns (B).  Wave w is at (w % WR, w / WR).
//
// Tiles this small are for grids that 128 x 128 blocks would leave mostly
// idle: a wave needs 8 RT CT cycles per k, so a 4096-step chain of one tile
// takes 14 us.  The operands go through a ring of S stages of 32 k (a 128-byte
// row per A row and per B column) filled by global_load_lds_dwordx4, S - 1
// stages ahead.  A wave reads stage kt + 1's operands under the MFMAs of stage
// kt.  One barrier per stage; a one-wave workgroup needs none.  The loop runs
// a round of S stages at a time, so that every slot is an immediate and the
// source pointers move once per round.
//   row(r): the address of stage row r's data (A rows first, then B rows),
//   16-byte aligned, K floats readable; K % 16 == 0.
// B goes into the first operand slot: a lane then holds row l % 16 and the
// four consecutive columns 4 (l / 16) .. + 3 of every tile.
template <int RT, int CT, int WR, int WC, int S>
struct ChainRing {
    static constexpr int kWaves = WR * WC;
    static constexpr int kARows = 16 * RT * WR, kBRows = 16 * CT * WC;
    static constexpr int kStageBytes = (kARows + kBRows) * 128;
    static constexpr int kCopies = (kARows + kBRows) / 8 / kWaves;   // per wave per stage
    static_assert(kCopies * 8 * kWaves == kARows + kBRows, "stage rows split evenly over the waves");
    static_assert(kCopies * (S - 1) < 64, "vmcnt range");
    static constexpr int kBytes = S * kStageBytes;
    static_assert(kBytes <= 65536 && S >= 2, "LDS offsets are 16-bit immediates");

    struct Frags {
        float a[8][RT], b[8][CT];   // [step of 4 k]
    };

    // wait until at most n (0 .. S - 2) stages' copies are in flight
    __device__ static void wait_stages(int n) {
        [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
            ((n == I ? chain_wait_vm<kCopies * I>() : (void)0), ...);
        }(std::make_integer_sequence<int, S - 1>{});
    }

    template <class Row>
    __device__ static void run(uint8_t* ring, Row row, int K, cf4_t (&acc)[RT][CT]) {
        const int KT = K / 32;
        const int lane = threadIdx.x & 63;
        const int wave = kWaves > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
        // copy s of wave w fills stage rows 8 q .. 8 q + 7, q = w + kWaves s;
        // lane i writes 16 bytes at row 8 q + i / 8, physical chunk i % 8
        const float* src[kCopies];
#pragma unroll
        for (int s = 0; s < kCopies; ++s) {
            const int r = 8 * (wave + kWaves * s) + (lane >> 3);
            src[s] = row(r) + 4 * ((lane & 7) ^ ((r >> 1) & 7));
        }
        // stage `slot` of the round src points at into its slot.  The copy's
        // immediate offset moves both addresses.
        auto issue = [&](auto slotc) __attribute__((always_inline)) {
            constexpr int slot = decltype(slotc)::value;
#pragma unroll
            for (int s = 0; s < kCopies; ++s)
                __builtin_amdgcn_global_load_lds(
                    APS_CGP(src[s]),
                    APS_CLP(ring + slot * kStageBytes + (wave + kWaves * s) * 1024 - 128 * slot), 16, 128 * slot, 0);
        };
        auto next_round = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < kCopies; ++s) src[s] += 32 * S;
        };
        // LDS byte addresses of this lane's element of step s (chunk s); the
        // tiles of a wave lie 2048 bytes apart (the swizzle repeats every 16
        // rows)
        const int ar = (wave % WR) * 16 * RT + (lane & 15), br = kARows + (wave / WR) * 16 * CT + (lane & 15);
        uint32_t aa[8], ba[8];
        const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(APS_CLP(ring))) + 4 * (lane >> 4);
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            aa[s] = base + chain_swz(ar, s);
            ba[s] = base + chain_swz(br, s);
        }
        typedef const __attribute__((address_space(3))) float* lds_t;
        auto read = [&](Frags& f, int slot, int s) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < CT; ++j) f.b[s][j] = *reinterpret_cast<lds_t>(ba[s] + (slot * kStageBytes + 2048 * j));
#pragma unroll
            for (int i = 0; i < RT; ++i) f.a[s][i] = *reinterpret_cast<lds_t>(aa[s] + (slot * kStageBytes + 2048 * i));
        };
        auto mma = [&](const Frags& f, int s) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int j = 0; j < CT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.b[s][j], f.a[s][i], acc[i][j], 0, 0, 0);
        };
        // the MFMAs of f with the reads of n from `slot` in their shadow: two
        // steps' reads after each of the first four steps' MFMAs (in one burst
        // the reads hold the MFMAs up until the LDS has taken them all)
        auto mma_read = [&](const Frags& f, Frags& n, int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                mma(f, s);
                __builtin_amdgcn_sched_barrier(0);
                if (s < 4) {
                    read(n, slot, 2 * s);
                    read(n, slot, 2 * s + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        auto barrier = [&]() __attribute__((always_inline)) {
            if (kWaves > 1) asm volatile("s_barrier" ::: "memory");
            else __builtin_amdgcn_wave_barrier();
        };
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) acc[i][j] = cf4_t{0.0f, 0.0f, 0.0f, 0.0f};
        auto for_slots = [&](auto body) __attribute__((always_inline)) {
            [&]<int... U>(std::integer_sequence<int, U...>) __attribute__((always_inline)) {
                (body(std::integral_constant<int, U>{}), ...);
            }(std::make_integer_sequence<int, S>{});
        };
        // round 0 into the S slots
        for_slots([&](auto u) __attribute__((always_inline)) {
            if (decltype(u)::value < KT) issue(u);
        });
        next_round();
        Frags f[2];
        if (KT > 0) {
            if (KT >= S) chain_wait_vm<kCopies*(S - 1)>();
            else wait_stages(KT - 1);
            barrier();
#pragma unroll
            for (int s = 0; s < 8; ++s) read(f[0], 0, s);
        }
        // stage kt + 1 has landed when at most the S - 2 stages after it are
        // in flight; past its barrier every wave has read stage kt, whose slot
        // takes stage kt + S
        int kt = 0;
        static_assert(S % 2 == 0, "the operand sets alternate");
        for (; kt + 2 * S <= KT; kt += S) {
            for_slots([&](auto u) __attribute__((always_inline)) {
                constexpr int U = decltype(u)::value;
                chain_wait_lgkm0();   // stage kt's operands
                chain_wait_vm<kCopies*(S - 2)>();
                barrier();
                issue(u);
                mma_read(f[U & 1], f[(U + 1) & 1], (U + 1) % S);
            });
            next_round();
        }
        // the last S .. 2 S - 1 stages (fewer in all when KT < S)
        auto last = [&](auto u) __attribute__((always_inline)) {
            constexpr int U = decltype(u)::value;
            if (kt >= KT) return;   // wave-uniform
            chain_wait_lgkm0();
            if (kt + 1 < KT) {
                wait_stages(KT - 2 - kt < S - 2 ? KT - 2 - kt : S - 2);
                barrier();
                if (kt + S < KT) issue(u);
                mma_read(f[U & 1], f[(U + 1) & 1], (U + 1) % S);
            } else {
#pragma unroll
                for (int s = 0; s < 8; ++s) mma(f[U & 1], s);
            }
            ++kt;
        };
        for_slots(last);
        for_slots(last);
        if (K % 32 != 0) {   // the last 16 k, straight from memory
            const int at = K - 16 + (lane >> 4);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
#pragma unroll
                for (int j = 0; j < CT; ++j) f[0].b[s][j] = row(br + 16 * j)[at + 4 * s];
#pragma unroll
                for (int i = 0; i < RT; ++i) f[0].a[s][i] = row(ar + 16 * i)[at + 4 * s];
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) mma(f[0], s);
        }
    }
};

}  // namespace aps
