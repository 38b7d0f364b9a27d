// Grouped expert FFN for few rows per expert (a decode step, a small serving
// batch): the same products as ffn_mfma.hip, bit for bit, in one-wave tiles.
//
// With a handful of rows per expert the GEMMs are bound by the weights' bytes
// (bf16, 16 experts: 117 MB for w1||w3, 59 MB for w2), or for one or two
// active experts by how many CUs share them and by latency.  The row tiles of
// ffn_mfma.hip stage 128 or 256 activation rows whatever their number, two
// bytes of copies for every byte of weights, through a ring that holds 16 KB
// of weights per CU.  Here a wave owns 32 rows x 32 packed weight rows over
// the whole K and loads both MFMA operands straight into registers, several
// stages ahead: no LDS, no barriers, 4 KB of weights in flight per stage, and
// rows past the expert's end re-read its last row (the same cache lines).
//  * w1||w3: 16 gate rows and the same 16 up rows, so that SwiGLU closes inside
//    each lane.  Eight stages of 128 bytes per row in flight: 64 loads, what
//    the wave can count (twelve were slower).
//  * w2: 32 hidden columns; K = F is short enough for every operand fragment
//    of the tile to be in flight at once.
// Every output element accumulates the same MFMA sequence over k ascending as
// in ffn_mfma.hip, so a row's bits do not depend on its batch.
//   Measured on weights that are in no cache (three sets in turn, traced), bf16:
// 37 tokens w1||w3 36 -> 27 us (4.4 TB/s), w2 20 -> 13 us (4.6 TB/s); one token 24 ->
// 14 and 13 -> 4.0 us.  fp8, 65 tokens: 21 -> 18 us, w2 with its combine 38 -> 13 us.
// (One set in a loop, which the memory-side cache holds: 37 tokens 27 -> 21 and 19 ->
// 11 us.)
//
// The packed images are read at their swizzled 16-byte chunks: the four (bf16)
// reads of a 128-byte image row follow each other and share its cache line.
#include "mfma_ring.hpp"

namespace aps {
namespace {

constexpr int kSmRows = 32;      // rows per tile
constexpr int kSmXcds = 8;
constexpr int kSmAhead = 8;      // w1||w3 stages in flight

struct SmallTile {
    int expert, col;             // expert, column group
    uint32_t m0, end;            // first position, expert's end
};

// Tile b of the list expert -> column group -> 32-row tile, dealt to the XCDs
// in contiguous slices (workgroup b runs on XCD b % 8), so that the row tiles
// of an expert read a weight tile in one L2.  lo, hi: this lane's expert's
// positions (lane = expert, 0 past the last); `bn`: column groups.  A block of
// `blocks` takes every (blocks / 8)-th tile of its slice; the grid covers 2
// rows assignments in one round, a caller's plan may hold more.
template <class Body>
__device__ inline void each_small(uint32_t lo, uint32_t hi, int bn, int blocks, Body body) {
    const int lane = threadIdx.x & 63;
    const int tiles = static_cast<int>((hi - lo + kSmRows - 1) / kSmRows);
    int incl = tiles * bn;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(incl, d);
        if (lane >= d) incl += v;
    }
    const int total = __shfl(incl, 63);
    const int per = (total + kSmXcds - 1) / kSmXcds;
    const int first = static_cast<int>(blockIdx.x % kSmXcds) * per;
    for (int l = static_cast<int>(blockIdx.x) / kSmXcds; l < per; l += blocks / kSmXcds) {
        const int t = first + l;
        if (t >= total) return;
        const int e = __ffsll(static_cast<unsigned long long>(__ballot(incl > t))) - 1;
        const int i = t - (e > 0 ? __shfl(incl, e - 1) : 0);
        const int n = __shfl(tiles, e);
        SmallTile u;
        u.expert = __builtin_amdgcn_readfirstlane(e);
        u.col = __builtin_amdgcn_readfirstlane(i / n);
        u.m0 = __builtin_amdgcn_readfirstlane(__shfl(lo, e) + static_cast<uint32_t>(i % n) * kSmRows);
        u.end = __builtin_amdgcn_readfirstlane(__shfl(hi, e));
        body(u);
    }
}

// ---- the routing plan inside the w1||w3 launch ------------------------------
// After the few-token router the plan (dispatch.hip states it) is a stable sort
// of at most 512 route bytes: every wave of the w1||w3 launch counts the routes
// itself and ranks those of its own expert, and two further blocks write the
// plan and its tile histograms out, for the kernels after it and for callers.  That saves the dispatch's launch between
// the router and the GEMM for 1 us in it: one bf16 token 35.0 -> 33.2 us a block,
// 37 tokens 52.0 -> 49.9, fp8 65 tokens 45.9 -> 43.6 (one weight set in a loop).
constexpr int kPlanTiles = static_cast<int>(kDispatchFewRows / kWave);

struct Routes {
    int first[kPlanTiles], second[kPlanTiles];   // token 64 k + lane (255: none)
    int nt;                                      // 64-token tiles
    __device__ void load(const uint8_t* __restrict__ routes, int64_t rows) {
        nt = static_cast<int>((rows + kWave - 1) / kWave);
#pragma unroll
        for (int k = 0; k < kPlanTiles; ++k) {
            const int64_t t = kWave * k + (threadIdx.x & 63);
            first[k] = t < rows ? routes[2 * t] : 255;
            second[k] = t < rows ? routes[2 * t + 1] : 255;
        }
    }
    __device__ uint64_t slot0(int k, int e) const { return __ballot(first[k] == e); }
    __device__ uint64_t slot1(int k, int e) const { return __ballot(second[k] == e); }
};

// This lane's expert's positions [lo, hi), counted from the routes.
__device__ inline void plan_counts(const Routes& r, int E, uint32_t& lo, uint32_t& hi) {
    const int lane = threadIdx.x & 63;
    uint32_t run = 0;
    lo = hi = 0;
    for (int e = 0; e < E; ++e) {
        uint32_t n = 0;
#pragma unroll
        for (int k = 0; k < kPlanTiles; ++k)
            if (k < r.nt) n += static_cast<uint32_t>(__popcll(r.slot0(k, e)) + __popcll(r.slot1(k, e)));
        if (lane == e) {
            lo = run;
            hi = run + n;
        }
        run += n;
    }
}

// The whole plan, by one wave (router's routes: two distinct experts a token).
__device__ inline void plan_write(const Routes& r, int64_t rows, int E, uint32_t lo, uint32_t hi, const SmallPlan& p) {
    const int lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t p0[kPlanTiles], p1[kPlanTiles], i0[kPlanTiles], i1[kPlanTiles];
    for (int e = 0; e < E; ++e) {
        uint32_t at = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(lo), e));
        uint32_t n0 = 0;
#pragma unroll
        for (int k = 0; k < kPlanTiles; ++k)
            if (k < r.nt) n0 += static_cast<uint32_t>(__popcll(r.slot0(k, e)));
        uint32_t l0 = at, l1 = at + n0;   // slot-0 routes of e, then its slot-1 routes
        if (lane == 0 && p.slot1) p.slot1[e] = l1;
#pragma unroll
        for (int k = 0; k < kPlanTiles; ++k) {
            if (k >= r.nt) continue;   // wave-uniform
            const uint64_t m0 = r.slot0(k, e), m1 = r.slot1(k, e);
            const uint32_t b0 = static_cast<uint32_t>(__popcll(m0 & below)), b1 = static_cast<uint32_t>(__popcll(m1 & below));
            if (r.first[k] == e) {
                p0[k] = at + b0 + b1;
                i0[k] = l0 + b0;
            }
            if (r.second[k] == e) {
                p1[k] = at + b0 + b1;
                i1[k] = l1 + b1;
            }
            at += static_cast<uint32_t>(__popcll(m0) + __popcll(m1));
            l0 += static_cast<uint32_t>(__popcll(m0));
            l1 += static_cast<uint32_t>(__popcll(m1));
        }
    }
    if (lane < E) {
        p.counts[lane] = hi - lo;
        p.offsets[lane] = lo;
        if (lane == E - 1) p.offsets[E] = hi;
    }
#pragma unroll
    for (int k = 0; k < kPlanTiles; ++k) {
        const uint32_t t = static_cast<uint32_t>(kWave * k + lane);
        if (t >= rows) continue;
        p.assignment_rows[p0[k]] = t;
        p.assignment_rows[p1[k]] = t;
        p.route_positions[2 * t] = p0[k];
        p.route_positions[2 * t + 1] = p1[k];
        if (p.slot1) {
            p.slot_rows[i0[k]] = p0[k];
            p.slot_tokens[i0[k]] = t;
            p.slot_rows[i1[k]] = p1[k];
            p.slot_tokens[i1[k]] = t;
        }
    }
}

// The plan's tile histograms, by one wave.
__device__ inline void plan_histograms(const Routes& r, int E, const SmallPlan& p) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < kPlanTiles; ++k) {
        if (k >= r.nt) continue;   // wave-uniform
        uint64_t m0 = 0, m1 = 0;
        for (int e = 0; e < E; ++e) {
            mask_to_lane(m0, r.slot0(k, e), e);
            mask_to_lane(m1, r.slot1(k, e), e);
        }
        if (lane >= E) continue;
        p.tile_counts[k * E + lane] = tile_word(m0, m1);
        if (p.slot1) p.tile_counts0[k * E + lane] = tile_word(m0, 0);
    }
}

// Token of row (lane % 32) of tile u, through tok[32] in LDS; rows past the
// expert's end get its last token.
__device__ inline uint32_t plan_token(const Routes& r, uint32_t expert_lo, const SmallTile& u, uint32_t* tok) {
    const int lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t at = expert_lo;
    __builtin_amdgcn_wave_barrier();   // the previous tile's reads come first
#pragma unroll
    for (int k = 0; k < kPlanTiles; ++k) {
        if (k >= r.nt) continue;   // wave-uniform
        const uint64_t m = r.slot0(k, u.expert) | r.slot1(k, u.expert);
        const uint32_t i = at + static_cast<uint32_t>(__popcll(m & below)) - u.m0;   // wraps for rows before m0
        if ((m >> lane & 1) && i < static_cast<uint32_t>(kSmRows)) tok[i] = static_cast<uint32_t>(kWave * k + lane);
        at += static_cast<uint32_t>(__popcll(m));
    }
    __builtin_amdgcn_wave_barrier();   // (a wave's LDS accesses complete in order)
    const uint32_t n = u.end - u.m0, row = lane & 31;
    return tok[row < n ? row : n - 1];
}

// One 128-byte stage of a lane's row: kSub fragments, each 16 (bf16) or 32
// (fp8) bytes of the k half lane / 32.
template <class Fmt>
struct SmallStage {
    typename Fmt::frag_t f[Fmt::kSub];
};
// Byte offset of part p of fragment kk in a row's stage (logical chunk order).
template <class Fmt>
__device__ inline int small_chunk(int kk, int p, int lane) {
    return (8 / Fmt::kSub) * kk + Fmt::kParts * (lane >> 5) + p;
}
template <class Fmt, class At>
__device__ inline void small_load(SmallStage<Fmt>& d, At at) {
#pragma unroll
    for (int kk = 0; kk < Fmt::kSub; ++kk) {
        u32x4_t v[Fmt::kParts];
#pragma unroll
        for (int p = 0; p < Fmt::kParts; ++p) v[p] = *reinterpret_cast<const u32x4_t*>(at(kk, p));
        if constexpr (Fmt::kParts == 1) d.f[kk] = __builtin_bit_cast(typename Fmt::frag_t, v[0]);
        else
            d.f[kk] = __builtin_bit_cast(typename Fmt::frag_t, __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7));
    }
}

// act[p][n], as ffn_mfma.hip's up_piece.  ROUTES: the plan comes from
// plan.routes and the last two blocks write it out; else from offsets and
// assignment_rows.
template <class Fmt, bool ROUTES>
__global__ void __launch_bounds__(64, 1)
k_ffn_up_small(const uint8_t* __restrict__ x, uint32_t x_row_bytes, const uint32_t* __restrict__ offsets,
               const uint32_t* __restrict__ assignment_rows, const SmallPlan plan, int64_t rows,
               const uint8_t* __restrict__ w13, bf16_t* __restrict__ act, int H, int F, int E,
               const float* __restrict__ sx, const float* __restrict__ s1, const float* __restrict__ s3) {
    constexpr bool kFp8 = Fmt::kElt == 1;
    __shared__ uint32_t tok[ROUTES ? kSmRows : 1];
    const int lane = threadIdx.x, r = lane & 31, h = lane >> 5;
    const int blocks = static_cast<int>(gridDim.x) - (ROUTES ? 2 : 0);
    uint32_t lo, hi;
    Routes routes;
    if constexpr (ROUTES) {
        routes.load(plan.routes, rows);
        if (static_cast<int>(blockIdx.x) > blocks) {   // block-uniform
            plan_histograms(routes, E, plan);
            return;
        }
        plan_counts(routes, E, lo, hi);
        if (static_cast<int>(blockIdx.x) == blocks) {   // block-uniform
            plan_write(routes, rows, E, lo, hi, plan);
            return;
        }
    } else {
        lo = lane < E ? offsets[lane] : 0u;
        hi = lane < E ? offsets[lane + 1] : 0u;
    }
    each_small(lo, hi, F / 16, blocks, [&](const SmallTile& u) __attribute__((always_inline)) {
    const int KT = H * Fmt::kElt / kRowBytes;
    const uint32_t p = u.m0 + r < u.end ? u.m0 + r : u.end - 1;
    uint32_t token;
    if constexpr (ROUTES)
        token = plan_token(routes, static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(lo), u.expert)), u,
                           tok);
    else token = assignment_rows[p];
    // image row of this lane: gate row 16 (col % 4) + r, then the same up rows
    const int ir = 16 * (u.col & 3) + (r < 16 ? r : 64 + (r - 16));
    const uint8_t* image = w13 + (static_cast<int64_t>(u.expert) * (F / 64) + u.col / 4) * KT * kImageBytes;
    uint32_t ao[Fmt::kSub][Fmt::kParts], bo[Fmt::kSub][Fmt::kParts];
#pragma unroll
    for (int kk = 0; kk < Fmt::kSub; ++kk)
#pragma unroll
        for (int q = 0; q < Fmt::kParts; ++q) {
            ao[kk][q] = token * x_row_bytes + 16u * small_chunk<Fmt>(kk, q, lane);
            bo[kk][q] = static_cast<uint32_t>(swz(ir, small_chunk<Fmt>(kk, q, lane)));
        }
    SmallStage<Fmt> a[kSmAhead], b[kSmAhead];
    // unconditional (a stage past the end re-reads the last), so that the
    // waits count the stages in flight
    auto load = [&](int d, int kt) __attribute__((always_inline)) {
        kt = kt < KT ? kt : KT - 1;
        const uint8_t* xb = x + static_cast<int64_t>(kt) * kRowBytes;
        const uint8_t* wb = image + static_cast<int64_t>(kt) * kImageBytes;
        small_load<Fmt>(b[d], [&](int kk, int q) __attribute__((always_inline)) { return wb + bo[kk][q]; });
        small_load<Fmt>(a[d], [&](int kk, int q) __attribute__((always_inline)) { return xb + ao[kk][q]; });
        APS_PIN();
    };
#pragma unroll
    for (int d = 0; d < kSmAhead; ++d) load(d, d);
    f32x16_t acc = {};
    for (int k0 = 0; k0 < KT; k0 += kSmAhead)
#pragma unroll
        for (int d = 0; d < kSmAhead; ++d) {
            if (k0 + d < KT)   // wave-uniform
#pragma unroll
                for (int kk = 0; kk < Fmt::kSub; ++kk) acc = Fmt::mma(b[d].f[kk], a[d].f[kk], acc);
            APS_PIN();
            load(d, k0 + d + kSmAhead);
        }
    // lane: row r; register 4 q + v: packed row 8 q + 4 h + v, i.e. gate column
    // 8 q + 4 h + v for q < 2 and its up value at q + 2
    if (u.m0 + r >= u.end) return;
    const int c0 = 16 * u.col + 4 * h;
    const float rs = kFp8 ? sx[token] : 1.0f;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        float g[4], up[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            g[v] = acc[4 * q + v];
            up[v] = acc[4 * (q + 2) + v];
            if constexpr (kFp8) {
                const int at = u.expert * F + c0 + 8 * q + v;
                g[v] = g[v] * rs * s1[at];
                up[v] = up[v] * rs * s3[at];
            }
        }
        *reinterpret_cast<u32x2_t*>(act + static_cast<int64_t>(p) * F + c0 + 8 * q) =
            u32x2_t{pack2_bf16(swiglu(g[0], up[0]), swiglu(g[1], up[1])),
                    pack2_bf16(swiglu(g[2], up[2]), swiglu(g[3], up[3]))};
    }
    });
}

// y[p][n], as ffn_mfma.hip's w2 GEMM.  KT: 128-byte stages of an act row.
template <class Fmt, int KT>
__global__ void __launch_bounds__(64, 2)
k_ffn_down_small(const uint8_t* __restrict__ act, int64_t act_row_bytes, const uint32_t* __restrict__ offsets,
                 const uint8_t* __restrict__ w2, bf16_t* __restrict__ y, int H, int E, const float* __restrict__ sa,
                 const float* __restrict__ s2) {
    constexpr bool kFp8 = Fmt::kElt == 1;
    const int lane = threadIdx.x, r = lane & 31, h = lane >> 5;
    const uint32_t lo = lane < E ? offsets[lane] : 0u, hi = lane < E ? offsets[lane + 1] : 0u;
    each_small(lo, hi, H / 32, static_cast<int>(gridDim.x), [&](const SmallTile& u) __attribute__((always_inline)) {
    const uint32_t p = u.m0 + r < u.end ? u.m0 + r : u.end - 1;
    const uint8_t* image = w2 + (static_cast<int64_t>(u.expert) * (H / 128) + u.col / 4) * KT * kImageBytes;
    const uint8_t* arow = act + static_cast<int64_t>(p) * act_row_bytes;
    const int ir = 32 * (u.col & 3) + r;
    SmallStage<Fmt> a[KT], b[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
        small_load<Fmt>(b[kt], [&](int kk, int q) __attribute__((always_inline)) {
            return image + kt * kImageBytes + swz(ir, small_chunk<Fmt>(kk, q, lane));
        });
        small_load<Fmt>(a[kt], [&](int kk, int q) __attribute__((always_inline)) {
            return arow + kt * kRowBytes + 16 * small_chunk<Fmt>(kk, q, lane);
        });
        APS_PIN();
    }
    f32x16_t acc = {};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int kk = 0; kk < Fmt::kSub; ++kk) acc = Fmt::mma(b[kt].f[kk], a[kt].f[kk], acc);
    if (u.m0 + r >= u.end) return;
    const int c0 = 32 * u.col + 4 * h;
    const float rs = kFp8 ? sa[p] : 1.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float o[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            o[v] = acc[4 * q + v];
            if constexpr (kFp8) o[v] = o[v] * rs * s2[u.expert * H + c0 + 8 * q + v];
        }
        *reinterpret_cast<u32x2_t*>(y + static_cast<int64_t>(p) * H + c0 + 8 * q) =
            u32x2_t{pack2_bf16(o[0], o[1]), pack2_bf16(o[2], o[3])};
    }
    });
}

typedef void (*down_small_fn)(const uint8_t*, int64_t, const uint32_t*, const uint8_t*, bf16_t*, int, int,
                              const float*, const float*);
// The w2 kernel for KT stages, or null (the operands of longer rows do not fit
// the registers).
template <class Fmt>
down_small_fn down_small_kernel(int KT) {
    constexpr int kMax = Fmt::kElt == 1 ? 4 : 7;
    switch (KT) {
        case 1: return k_ffn_down_small<Fmt, 1>;
        case 2: return k_ffn_down_small<Fmt, 2>;
        case 3: return k_ffn_down_small<Fmt, 3>;
        case 4: return k_ffn_down_small<Fmt, 4>;
        case 5: return kMax >= 5 ? k_ffn_down_small<Fmt, (kMax >= 5 ? 5 : 1)> : nullptr;
        case 6: return kMax >= 6 ? k_ffn_down_small<Fmt, (kMax >= 6 ? 6 : 1)> : nullptr;
        case 7: return kMax >= 7 ? k_ffn_down_small<Fmt, (kMax >= 7 ? 7 : 1)> : nullptr;
        default: return nullptr;
    }
}

// Blocks of a tile list of 2 rows assignments: every expert's last tile may be
// partly filled, and an expert has a tile only if it has a row.
dim3 grid_small(int64_t rows, int experts, int bn) {
    const int64_t some = 2 * rows < experts ? 2 * rows : experts;
    const int64_t tiles = (2 * rows) / kSmRows + some;
    return dim3(static_cast<unsigned>(ceil_div(tiles * bn, kSmXcds) * kSmXcds));
}

int small_kt(bool fp8, int ffn) { return static_cast<int>(fp8 ? ceil_div(ffn, 128) : ffn / 64); }

}  // namespace

// Up to 12 rows per expert on average in bf16, 24 in fp8, whose MFMAs and w2
// passes weigh less against the weights' bytes: a tile reads its weights for
// 32 rows, so more rows read them again.  Whole MoE block, 16 experts (one weight
// set in a loop), us with the row tiles of ffn_mfma.hip -> here, even (Zipf 1.1) expert loads:
//   bf16  1 token 60 -> 40 (60 -> 40), 37 69 -> 56 (68 -> 56), 96 70 -> 58 (69 ->
//         64), 128 69 -> 59 (70 -> 78), 256 70 -> 83 (73 -> 84)
//   fp8   1 token 74 -> 44 (73 -> 44), 65 86 -> 58 (86 -> 61), 192 87 -> 63 (87 ->
//         71), 384 87 -> 82 (91 -> 83), 613 88 -> 114 (95 -> 117)
//   Past 128 blocks of 64 columns over all experts (E F > 8192) the row tiles
// fill the chip by themselves, and a skewed load sends many rows to an expert
// while the mean is low: there up to 8 experts' worth.  us row tiles -> here, 64
// experts, hidden 2048, even (Zipf 1.1 / 2.2) loads: F = 448 bf16 64 tokens 99 -> 105
// (88 -> 98 / 68 -> 68), 256 tokens 114 -> 123 (113 -> 136 / 83 -> 113), fp8 512 tokens
// 90 -> 98 (94 -> 117 / 85 -> 103); F = 64, hidden 4096, bf16 256 tokens 101 -> 91 (103 ->
// 94 / 101 -> 92); 24 experts of 448, hidden 4096, bf16 96 tokens 90 -> 87 (92 -> 94 /
// 83 -> 92).
bool ffn_small_fits(bool fp8, int64_t rows, int ffn, int experts) {
    const int64_t mean = fp8 ? 24 : 12, E = experts;
    return 2 * rows <= mean * E && (E * ffn <= 8192 || 2 * rows <= mean * 8) && small_kt(fp8, ffn) <= (fp8 ? 4 : 7);
}

// w2's whole K is in flight at once and its tiles read less again, so it gains
// up to 24 rows per expert in bf16 and 32, a full tile, in fp8.  Whole block, 16
// experts, us with the row tiles of w2 -> here, even (Zipf 1.1) loads:
//   bf16  97 tokens 75 -> 69 (75 -> 73), 192 77 -> 72 (77 -> 76), 256 78 -> 77 (83 ->
//         85), 512 83 -> 91 (95 -> 100)
//   fp8   224 tokens 56 -> 51 (57 -> 54), 256 56 -> 53 (59 -> 58), 384 69 -> 70 (73 ->
//         73), 613 71 -> 77 (78 -> 80)
//   Many experts keep the mean low whatever the load: past 512 bf16 tokens (and
// 8192 columns, as above) an expert that takes them all reads its weights too
// often.  64 experts, hidden 4096, us row tiles -> here, even / Zipf 1.1 / every
// token to two experts: 512 tokens 230 -> 218 / 252 -> 253 / 107 -> 118, 768 tokens
// 231 -> 228 / 257 -> 263 / 108 -> 129.
bool ffn_down_small_fits(bool fp8, int64_t rows, int ffn, int experts) {
    if (!fp8 && rows > 512 && static_cast<int64_t>(experts) * ffn > 8192) return false;
    return 2 * rows <= (fp8 ? 32 : 24) * static_cast<int64_t>(experts) && small_kt(fp8, ffn) <= (fp8 ? 4 : 7);
}

hipError_t launch_ffn_up_small(bool fp8, const uint8_t* x, const float* sx, const uint32_t* offsets,
                               const uint32_t* assignment_rows, const SmallPlan* plan, const uint8_t* w13,
                               const float* s1, const float* s3, bf16_t* act, int64_t rows, int hidden, int ffn,
                               int experts, hipStream_t s) {
    if (plan && (rows > kDispatchFewRows || experts > kWave)) return hipErrorInvalidValue;
    dim3 grid = grid_small(rows, experts, ffn / 16);
    const uint32_t row_bytes = static_cast<uint32_t>(hidden) * (fp8 ? 1u : 2u);
    if (plan) grid.x += 2;
    auto kern = fp8 ? (plan ? k_ffn_up_small<Fp8Fmt, true> : k_ffn_up_small<Fp8Fmt, false>)
                    : (plan ? k_ffn_up_small<Bf16Fmt, true> : k_ffn_up_small<Bf16Fmt, false>);
    hipLaunchKernelGGL(kern, grid, dim3(64), 0, s, x, row_bytes, offsets, assignment_rows, plan ? *plan : SmallPlan{},
                       rows, w13, act, hidden, ffn, experts, sx, s1, s3);
    return hipGetLastError();
}

hipError_t launch_ffn_down_small(bool fp8, const uint8_t* act, const float* sa, const uint32_t* offsets,
                                 const uint8_t* w2, const float* s2, bf16_t* y, int64_t rows, int hidden, int ffn,
                                 int experts, hipStream_t s) {
    const int KT = small_kt(fp8, ffn);
    const down_small_fn kern = fp8 ? down_small_kernel<Fp8Fmt>(KT) : down_small_kernel<Bf16Fmt>(KT);
    if (!kern) return hipErrorInvalidValue;
    hipLaunchKernelGGL(kern, grid_small(rows, experts, hidden / 32), dim3(64), 0, s, act,
                       static_cast<int64_t>(fp8 ? KT * 128 : ffn * 2), offsets, w2, y, hidden, experts, sa, s2);
    return hipGetLastError();
}

}  // namespace aps
