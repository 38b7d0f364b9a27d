// The LDS stage ring of the bf16 and fp8 MFMA GEMMs: direct-to-LDS copies
// into three 48 KB stages, operand fragments read one MFMA step ahead, every
// copy and read placed behind an MFMA.  Used by the grouped expert GEMMs
// (ffn_mfma.hip, which describes the tiling) and the split-bf16 Linear
// (linear_tc.hip).
//
// A format Fmt states kSub (MFMA k steps per 128-byte stage row), frag_t,
// kParts / load_part (the LDS reads of one fragment), kProd and mma<P> (the
// MFMAs per fragment pair and step: 1, or the hi / lo products of split bf16)
// and kAStep (bytes an A row advances per stage).
#pragma once

#include "common.hpp"

namespace aps {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));
// native vectors (not HIP's uint4 struct, whose copies become memcpy through
// a stack slot): 16 bytes = one ds_read_b128 / global_load_dwordx4
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kRowBytes = 128;                 // one stage row: 8 chunks of 16 bytes
constexpr int kImageBytes = 128 * kRowBytes;   // one packed weight tile image

// Byte offset of 16-byte chunk `chunk` (0..7) of stage row `row`.  gfx950's
// LDS has 64 four-byte banks (a 256-byte bank row = two stage rows) and
// serves a ds_read_b128 16 lanes at a time.  An MFMA operand fetch reads the
// same logical chunk from 16 consecutive rows, so the physical chunk is
// chunk ^ ((row >> 1) & 7): rows 2m and 2m+1 sit in the two halves of a bank
// row, and the eight pairs of a 16-row group get eight different chunks --
// sixteen distinct 16-byte bank groups, no conflict.
__device__ inline int swz(int row, int chunk) { return row * kRowBytes + ((chunk ^ ((row >> 1) & 7)) << 4); }

// silu(g) * u for the MFMA paths: fp32 math with the hardware exp2 and
// reciprocal (the result is rounded to bf16, far coarser than their error).
__device__ inline float swiglu(float g, float u) {
    return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
}

#define APS_GP(p) ((const __attribute__((address_space(1))) void*)(p))
#define APS_LP(p) ((__attribute__((address_space(3))) void*)(p))
#define APS_PIN() __builtin_amdgcn_sched_barrier(0)

// One direct-to-LDS copy: lane i writes LDS bytes [16i, 16i+16) of the
// wave-uniform 1 KB slot at lds_slot (eight stage rows).
__device__ inline void dma16(const uint8_t* src, uint8_t* lds_slot) {
    __builtin_amdgcn_global_load_lds(APS_GP(src), APS_LP(lds_slot), 16, 0, 0);
}

// s_waitcnt vmcnt(n) lgkmcnt(0) (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] |
// lgkmcnt[11:8] | vmcnt[5:4] at bits [15:14]); n must be a constant.
template <int N>
__device__ inline void wait_vm_lgkm0() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (0x0 << 8) | ((N >> 4) << 14));
}

// s_waitcnt lgkmcnt(0) alone (vmcnt and expcnt left at their maximum).
__device__ inline void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xF | (0x7 << 4) | (0x0 << 8) | (0x3 << 14)); }

// A raw s_barrier: __syncthreads() adds a workgroup fence, which drains every
// in-flight load (vmcnt(0)) and would serialise the ring.
__device__ inline void raw_barrier() { asm volatile("s_barrier" ::: "memory"); }

// ---------------------------------------------------------------------------
// Operand formats.  kSub MFMA k steps per 128-byte stage row; a fragment is
// one lane's share of a 32-row MFMA operand: lane l holds row l % 32 and the
// k half (l / 32) of the step, the same for A and B.
struct Bf16Fmt {
    static constexpr int kSub = 4;             // 32x32x16: 16 k = 32 bytes per step
    static constexpr int kElt = 2;
    static constexpr int kProd = 1, kAStep = kRowBytes;
    typedef bf16x8_t frag_t;
    __device__ static frag_t load(const uint8_t* st, int row, int kk, int lane) {
        return __builtin_bit_cast(frag_t, *reinterpret_cast<const u32x4_t*>(st + swz(row, 2 * kk + (lane >> 5))));
    }
    // a fragment is one ds_read_b128; load_part(.., 0) is load()
    static constexpr int kParts = 1;
    __device__ static void load_part(frag_t& f, const uint8_t* st, int row, int kk, int lane, int) {
        f = load(st, row, kk, lane);
    }
    __device__ static f32x16_t mma(const frag_t& a, const frag_t& b, f32x16_t c, int = 0) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    // The register-resident w2 kernel pins its operands: accumulators in
    // VGPRs, the resident act fragments (second operand) in AGPRs, which
    // the MFMA reads directly.  Left to the allocator, the 224 act registers
    // plus 128 accumulators overflow the VGPR file and every step shuffles
    // operands between the two files.
    static constexpr bool kPinned = true;
    // NOP: three wait states in the same statement first, for a VALU write
    // of an operand register that the compiler may place right before it
    // (the hazard recognizer does not look into inline asm; 2 are needed)
    template <bool NOP = false>
    __device__ static void mma_pinned(f32x16_t& c, const frag_t& b, const frag_t& a) {
        if constexpr (NOP) asm("s_nop 2\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(b), "a"(a));
        else asm("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(b), "a"(a));
    }
    // the first k step of a tile: c = b x a + 0 (no zeroed accumulators)
    template <bool NOP = false>
    __device__ static void mma_pinned_first(f32x16_t& c, const frag_t& b, const frag_t& a) {
        if constexpr (NOP) asm("s_nop 2\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(b), "a"(a));
        else asm("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(b), "a"(a));
    }
};

struct Fp8Fmt {
    static constexpr int kSub = 2;             // 32x32x64: 64 k = 64 bytes per step
    static constexpr int kElt = 1;
    static constexpr int kProd = 1, kAStep = kRowBytes;
    typedef i32x8_t frag_t;
    __device__ static frag_t load(const uint8_t* st, int row, int kk, int lane) {
        const int c = 4 * kk + 2 * (lane >> 5);
        const i32x4_t lo = *reinterpret_cast<const i32x4_t*>(st + swz(row, c));
        const i32x4_t hi = *reinterpret_cast<const i32x4_t*>(st + swz(row, c + 1));
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
    // a fragment is two ds_read_b128 (its low and high 16 bytes), issued
    // separately by the interleaved main loop
    static constexpr int kParts = 2;
    __device__ static void load_part(frag_t& f, const uint8_t* st, int row, int kk, int lane, int part) {
        const int c = 4 * kk + 2 * (lane >> 5) + part;
        const i32x4_t v = *reinterpret_cast<const i32x4_t*>(st + swz(row, c));
        const i32x4_t lo = __builtin_shufflevector(f, f, 0, 1, 2, 3);
        const i32x4_t hi = __builtin_shufflevector(f, f, 4, 5, 6, 7);
        f = part == 0 ? __builtin_shufflevector(v, hi, 0, 1, 2, 3, 4, 5, 6, 7)
                      : __builtin_shufflevector(lo, v, 0, 1, 2, 3, 4, 5, 6, 7);
    }
    // e4m3 x e4m3 (format code 0 for both operands), unit scales
    __device__ static f32x16_t mma(const frag_t& a, const frag_t& b, f32x16_t c, int = 0) {
        return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
    }
    // The register-resident w2 kernel pins its operands as for bf16:
    // accumulators in VGPRs, the resident act fragments in AGPRs, so that
    // the epilogue reads the accumulators without v_accvgpr_read (128 VALU
    // moves per column block, which add to the MFMA time on a SIMD).
    static constexpr bool kPinned = true;
    template <bool NOP = false>
    __device__ static void mma_pinned(f32x16_t& c, const frag_t& b, const frag_t& a) {
        if constexpr (NOP) asm("s_nop 2\n\tv_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, %0" : "+v"(c) : "v"(b), "a"(a));
        else asm("v_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, %0" : "+v"(c) : "v"(b), "a"(a));
    }
    template <bool NOP = false>
    __device__ static void mma_pinned_first(f32x16_t& c, const frag_t& b, const frag_t& a) {
        if constexpr (NOP) asm("s_nop 2\n\tv_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, 0" : "=&v"(c) : "v"(b), "a"(a));
        else asm("v_mfma_f32_32x32x64_f8f6f4 %0, %1, %2, 0" : "=&v"(c) : "v"(b), "a"(a));
    }
};

// ---------------------------------------------------------------------------
// Stage ring.  A stage holds kStageRows = 384 rows of 128 bytes: RA rows of
// A (token rows) followed by 384 - RA rows of B (packed weight tile rows).
constexpr int kStageRows = 384;
constexpr int kStageBytes = kStageRows * kRowBytes;  // 48 KB
constexpr int kStages = 3;                           // 3 x 48 KB = 144 KB of LDS

struct Ring3 {
    uint8_t s[kStages][kStageBytes];
};

// Load slot s (0..11) of wave w copies stage rows 32s + 8w .. +8 (1 KB).
// A slots advance one 128-byte row chunk per stage, B slots one tile image.
struct Slots {
    const uint8_t* p[12];
};

// Stage row and logical chunk of this lane in a load slot: lane i lands at
// physical chunk i & 7 of row 8 * (slot row group) + i / 8, so it fetches
// the logical chunk that swz() places there.
__device__ inline int slot_row(int s, int wave, int lane) { return 32 * s + 8 * wave + (lane >> 3); }
__device__ inline int slot_chunk(int row, int lane) { return (lane & 7) ^ ((row >> 1) & 7); }

enum PieceKind { kPieceW = 0, kPieceT = 1, kPieceS = 2, kPieceQ = 3 };

template <int KIND>
struct PShape;
template <>
struct PShape<kPieceW> { static constexpr int WM = 2, WN = 2, MI = 2, NJ = 4; };
template <>
struct PShape<kPieceT> { static constexpr int WM = 4, WN = 1, MI = 2, NJ = 4; };
template <>
struct PShape<kPieceS> { static constexpr int WM = 2, WN = 2, MI = 2, NJ = 2; };
template <>
struct PShape<kPieceQ> { static constexpr int WM = 4, WN = 1, MI = 1, NJ = 2; };

template <class Sh>
struct PDims {
    static constexpr int RA = Sh::WM * Sh::MI * 32;      // A rows (positions) per stage
    static constexpr int RB = Sh::WN * Sh::NJ * 32;      // B rows (packed weight rows) per stage
    static constexpr int NA = RA / 32;                   // A load slots per wave
    static constexpr int NS = (RA + RB) / 32;            // load slots per wave
    static constexpr int M = Sh::MI * Sh::NJ;            // MFMAs per step
    static constexpr int NR = Sh::MI + Sh::NJ;           // fragments per step
    static constexpr int kCols = Sh::WN * Sh::NJ / 2 * 32;  // act columns of the piece
    static_assert(RA + RB <= kStageRows, "stage fits the ring");
};

template <class Fmt, class Sh>
struct PFrags {
    typename Fmt::frag_t a[Sh::MI];
    typename Fmt::frag_t b[Sh::NJ];
};

// Part `part` of fragment o of a wave's step-kk operands, in the order the
// step's MFMAs first need them: a0, b0 .. b(NJ-1), a1 .. a(MI-1).
template <class Fmt, class Sh>
__device__ inline void pload(PFrags<Fmt, Sh>& f, const uint8_t* st, int kk, int lane, int aR, int bR, int o,
                             int part) {
    if (o == 0) Fmt::load_part(f.a[0], st, aR + (lane & 31), kk, lane, part);
    else if (o <= Sh::NJ) Fmt::load_part(f.b[o - 1], st, bR + (o - 1) * 32 + (lane & 31), kk, lane, part);
    else Fmt::load_part(f.a[o - Sh::NJ], st, aR + (o - Sh::NJ) * 32 + (lane & 31), kk, lane, part);
}

// MFMA q of a step, product q / (MI NJ) of tile t = q % (MI NJ):
// acc[t / NJ][t % NJ] += b[t % NJ] x a[t / NJ].
template <class Fmt, class Sh>
__device__ inline void pmma(const PFrags<Fmt, Sh>& f, f32x16_t (&acc)[Sh::MI][Sh::NJ], int q) {
    const int t = q % PDims<Sh>::M, i = t / Sh::NJ, j = t % Sh::NJ;
    acc[i][j] = Fmt::mma(f.b[j], f.a[i], acc[i][j], q / PDims<Sh>::M);
}

// Copies of load slots [lo, hi) of stage kt (A slots advance one 128-byte
// row chunk per stage, B slots one 16 KB tile image).
template <class Sh, class Fmt>
__device__ inline void pissue(uint8_t* stage, const Slots& sl, int kt, int wave, int lo, int hi) {
#pragma unroll
    for (int s = lo; s < hi; ++s) {
        const int64_t adv = s < PDims<Sh>::NA ? static_cast<int64_t>(kt) * Fmt::kAStep
                                              : static_cast<int64_t>(kt) * kImageBytes;
        dma16(sl.p[s] + adv, stage + (32 * s + 8 * wave) * kRowBytes);
    }
}

// One stage of the three-stage ring.  Every MFMA is issued with the fragment
// reads and stage copies of its shadow after it, so that the matrix pipe
// keeps working while the wave issues them (issued in a burst between groups
// of MFMAs, they left the pipe idle for about a quarter of each step).  A
// step s < kSub - 1 issues MFMA q and then: for q < MR, its share of the
// next step's fragments (MR = 3 of 8 MFMAs, fewer for small pieces); for
// q >= MR, its share of this step's refill copies (REFILL).  The compiler
// drains lgkmcnt before a step's first MFMA (it cannot count LDS reads past
// in-flight LDS DMA), so the reads go first, well before that wait.  The
// last step (the stage hand-over) issues MFMAs 0 .. MB - 1, waits for stage
// kt + 1 (vmcnt) and its own fragments, passes one s_barrier, and reads
// stage kt + 1's first fragments in the shadow of the remaining MFMAs.
// REFILL: this stage refills the slot of stage kt - 1 with stage kt + 2;
// NEXT: a stage kt + 1 exists; PEND: stage kt + 2's copies are in flight at
// the hand-over.  Only the issue order is chosen here: every output element
// accumulates its MFMAs in k order.
template <class Sh, class Fmt, bool REFILL, bool NEXT, bool PEND>
__device__ inline void pstage(Ring3& ring, const Slots& sl, int kt, int wave, int lane, int aR, int bR,
                              PFrags<Fmt, Sh> (&f)[2], f32x16_t (&acc)[Sh::MI][Sh::NJ]) {
    typedef PDims<Sh> D;
    constexpr int kSub = Fmt::kSub, P = Fmt::kParts;
    constexpr int M = D::M * Fmt::kProd, NR = D::NR, NS = D::NS;
    // MFMAs carrying the reads: early in the step, but (several products per
    // fragment) no more than one read per MFMA, the LDS rate of four waves
    constexpr int MR = Fmt::kProd > 1 ? M / 2 : M >= 8 ? 3 : (M >= 4 ? 2 : 1);
    constexpr int MB = M >= 8 ? 2 : 1;                  // MFMAs before the hand-over barrier
    const uint8_t* st = ring.s[kt % 3];
#pragma unroll
    for (int s = 0; s < kSub; ++s) {
        const PFrags<Fmt, Sh>& fc = f[s & 1];
        PFrags<Fmt, Sh>& fn = f[(s + 1) & 1];
        if (s + 1 < kSub) {
            const int c0 = NS * s / (kSub - 1), nc = NS * (s + 1) / (kSub - 1) - c0;
#pragma unroll
            for (int q = 0; q < M; ++q) {
                pmma<Fmt, Sh>(fc, acc, q);
                APS_PIN();
                if (q < MR) {
#pragma unroll
                    for (int o = q * NR * P / MR; o < (q + 1) * NR * P / MR; ++o)
                        pload<Fmt, Sh>(fn, st, s + 1, lane, aR, bR, o / P, o % P);
                }
                if (REFILL) {
#pragma unroll
                    for (int c = 0; c < nc; ++c) {
                        const int qc = M > MR ? MR + c * (M - MR) / nc : M - 1;
                        if (qc == q) pissue<Sh, Fmt>(ring.s[(kt + 2) % 3], sl, kt + 2, wave, c0 + c, c0 + c + 1);
                    }
                }
                APS_PIN();
            }
        } else {
#pragma unroll
            for (int q = 0; q < MB; ++q) {
                pmma<Fmt, Sh>(fc, acc, q);
                APS_PIN();
            }
            if (NEXT) {
                if (PEND) wait_vm_lgkm0<NS>();
                else wait_vm_lgkm0<0>();
                raw_barrier();
            } else {
                wait_lgkm0();
            }
            APS_PIN();
            const uint8_t* sn = ring.s[(kt + 1) % 3];
            // MFMAs carrying the next stage's reads
            constexpr int MRn = Fmt::kProd > 1 ? M / 2 : M - MB < 3 ? M - MB : 3;
#pragma unroll
            for (int q = MB; q < M; ++q) {
                pmma<Fmt, Sh>(fc, acc, q);
                APS_PIN();
                if (NEXT && q - MB < MRn) {
                    const int k = q - MB;
#pragma unroll
                    for (int o = k * NR * P / MRn; o < (k + 1) * NR * P / MRn; ++o)
                        pload<Fmt, Sh>(f[0], sn, 0, lane, aR, bR, o / P, o % P);
                }
                APS_PIN();
            }
        }
    }
}

// acc += A x B over KT stages of the three-stage ring.  Stage kt lives in
// slot kt % 3; stages 0..2 are copied up front, stage kt + 2 during stage kt
// (1 <= kt <= KT - 3).
template <class Sh, class Fmt>
__device__ inline void pmainloop(Ring3& ring, const Slots& sl, int KT, int wave, int lane, int aR, int bR,
                                 f32x16_t (&acc)[Sh::MI][Sh::NJ]) {
    typedef PDims<Sh> D;
    constexpr int P = Fmt::kParts, NS = D::NS;
    pissue<Sh, Fmt>(ring.s[0], sl, 0, wave, 0, NS);
    if (KT > 1) pissue<Sh, Fmt>(ring.s[1], sl, 1, wave, 0, NS);
    if (KT > 2) pissue<Sh, Fmt>(ring.s[2], sl, 2, wave, 0, NS);
    if (KT > 2) wait_vm_lgkm0<2 * NS>();
    else if (KT > 1) wait_vm_lgkm0<NS>();
    else wait_vm_lgkm0<0>();
    raw_barrier();
    PFrags<Fmt, Sh> f[2];
#pragma unroll
    for (int o = 0; o < D::NR; ++o)
#pragma unroll
        for (int part = 0; part < P; ++part) pload<Fmt, Sh>(f[0], ring.s[0], 0, lane, aR, bR, o, part);
    APS_PIN();
    if (KT == 1) {
        pstage<Sh, Fmt, false, false, false>(ring, sl, 0, wave, lane, aR, bR, f, acc);
        return;
    }
    if (KT > 2) pstage<Sh, Fmt, false, true, true>(ring, sl, 0, wave, lane, aR, bR, f, acc);
    else pstage<Sh, Fmt, false, true, false>(ring, sl, 0, wave, lane, aR, bR, f, acc);
    for (int kt = 1; kt + 2 < KT; ++kt) pstage<Sh, Fmt, true, true, true>(ring, sl, kt, wave, lane, aR, bR, f, acc);
    if (KT > 2) pstage<Sh, Fmt, false, true, false>(ring, sl, KT - 2, wave, lane, aR, bR, f, acc);
    pstage<Sh, Fmt, false, false, false>(ring, sl, KT - 1, wave, lane, aR, bR, f, acc);
}

}  // namespace aps
