// The part of the kernels' host interface that does not depend on the Element type: scheduler
// sizing, the slot kernel, the launch of a planned persistent kernel, and the switch over the
// Element type in front of the launchers that kernels_f32.hip, kernels_bf16.hip and kernels_f16.hip
// instantiate (kernels_impl.hpp).
#include <cmath>

#include "kernels_impl.hpp"

namespace kleos_amd {

KLEOS_EXTERN_ELEMENT(float)
KLEOS_EXTERN_ELEMENT(tf32_t)
KLEOS_EXTERN_ELEMENT(bf16_t)
KLEOS_EXTERN_ELEMENT(f16_t)

namespace {
__global__ __launch_bounds__(kPhaseThreads) void slot_kernel(const LayerParams p) {
    extern __shared__ uint32_t slot_smem[];
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t tile = blockIdx.x * 4 + wave;
    slot_tile<false>(p, tile, tile < p.n_gate_tiles, slot_smem + wave * slot_tile_words(p.E, kWave), threadIdx.x % kWave, kWave);
    if (blockIdx.x == 0)
        for (uint32_t e = threadIdx.x; e < p.E; e += kPhaseThreads) p.expert_count[e] = routed_count(p, e);
    // the coarse counts of the other epoch are free now: clear them for the next launch
    uint32_t* other = p.super_count + size_t((p.epoch & 1u) ^ 1u) * p.n_super * p.E;
    for (uint32_t i = blockIdx.x * kPhaseThreads + threadIdx.x; i < p.n_super * p.E; i += gridDim.x * kPhaseThreads)
        other[i] = 0u;
}

__global__ __launch_bounds__(kPhaseThreads) void dense_rows_kernel(const LayerParams p) {
    const uint32_t first = blockIdx.x * kPhaseThreads + threadIdx.x, stride = gridDim.x * kPhaseThreads;
    dense_rows(p, first, stride);
    uint32_t* other = p.super_count + size_t((p.epoch & 1u) ^ 1u) * p.n_super;
    for (uint32_t i = first; i < p.n_super; i += stride) other[i] = 0u;
}
}  // namespace

const char* unsupported_reason(uint32_t E, uint32_t k) {
    if (E > kMaxExperts) return "num_experts > 512 is not supported by this build (LDS tables of the persistent kernel)";
    if (E > 16 * kMaxGateGroups && k > kWideGateMaxK)
        return "expert_top_k > 32 with num_experts > 256 is not supported by the gate kernel of this build";
    return nullptr;
}

uint32_t sched_error_word() { return kSchedError; }


size_t sched_words(uint32_t E, uint32_t cap_rows) {
    return kSchedReady + size_t(E) * ceil_div_u32(cap_rows, 64) + 64;
}

namespace {
// What a tile of bm x bn costs per value of K (us, a CU's share of the device while all of them stream), and how
// many of them the CUs go through one after another.
struct TileCost { uint32_t bm, bn; double per_k, fixed; };
double projection_us(const LayerParams& p, const TileCost& t, uint32_t N, uint32_t K, uint32_t rows, double slots, bool whole_rounds) {
    double rounds = double(p.E) * ceil_div_u32(rows, t.bm) * ceil_div_u32(N, t.bn) / slots;
    rounds = whole_rounds ? double(uint64_t(rounds + 0.999999)) : (rounds < 1.0 ? 1.0 : rounds);
    return rounds * (K * t.per_k + t.fixed);
}
double projections_us(const LayerParams& p, const TileCost& t, uint32_t rows, double slots, bool whole_rounds) {
    return projection_us(p, t, p.I, p.H, rows, slots, whole_rounds) + projection_us(p, t, p.H, p.I, rows, slots, whole_rounds);
}
// Rows an expert holds on average.
uint32_t mean_rows(const LayerParams& p) {
    const uint32_t cap = p.EC < p.cap_rows ? p.EC : p.cap_rows;
    uint32_t rows = ceil_div_u32(p.S * p.k, p.E);
    if (rows > cap) rows = cap;
    return rows < 1 ? 1u : rows;
}
// Rows an expert may hold, and for which share of the experts.
struct RowShare { double rows, share; };
// Routing that favours nobody gives an expert its mean, give or take the root of it. Where the capacity leaves room for
// more than that (two and a half times the mean) one expert in ten is taken to be hot and hold twice the mean (of the shares and factors tried the one that loses to
// the capacity rule at the fewest of the layers below); a single expert holds what it holds.
int row_shares(const LayerParams& p, RowShare out[4]) {
    const double cap = p.EC < p.cap_rows ? p.EC : p.cap_rows;
    double mean = double(p.S) * p.k / p.E;
    if (mean > cap) mean = cap;
    auto held = [&](double rows) { return rows < 1.0 ? 1.0 : (rows > cap ? cap : rows); };
    if (p.E == 1) { out[0] = RowShare{held(mean), 1.0}; return 1; }
    const bool hot = cap >= 2.5 * mean;
    const double all = hot ? 1.1 : 1.0, sigma = std::sqrt(mean);
    out[0] = RowShare{held(mean - sigma), 0.25 / all};
    out[1] = RowShare{held(mean), 0.5 / all};
    out[2] = RowShare{held(mean + sigma), 0.25 / all};
    if (hot) out[3] = RowShare{held(2.0 * mean), 0.1 / all};
    return hot ? 4 : 3;
}
// A 16-bit tile by what a CU loads and multiplies (the figures at choose_tiles). The rows a tile has beyond the expert's
// read one row of zeros and are not charged: charged like the others, the rule does 0.2 % better in the mean of the layers
// below and loses to the capacity rule at some more of them.
TileCost tile16_cost(uint32_t bm, uint32_t bn, uint32_t rows) {
    const uint32_t r = rows < bm ? rows : bm;
    const double load = (r + bn) * 2.0 / 47e3, multiply = 2.0 * (ceil_div_u32(r, 16) * 16) * bn / 5.1e6;
    return TileCost{bm, bn, load > multiply ? load : multiply, 5.0};
}
}  // namespace

// The variants differ in how many rows and columns a tile has, so in how many rounds the CUs need for all of a
// layer's tiles, and in the bytes and operations of a round. The estimate below, of both projections, decides:
//   - an expert holds the rows of row_shares, so many row blocks on average;
//   - a CU takes in about 47 KB a microsecond whatever it loads (fitted to times of all 16-bit variants), a tile rows +
//     columns of 2 bytes per value of K; 256 x 256 tiles also come close to the matrix rate, 5.1 GFLOP a millisecond and CU;
//   - a tile costs 5 us besides (look-ups, first slices, epilogue);
//   - the weights pass at no more than 6.2 TB/s (tiles that share weights read them with the default policy, whose
//     rate for weights read once is an eighth lower), and of two variants bound by that the one considered first is taken:
//     the large tile, then as below.
// Measured against every variant at 487 layers drawn between 128 and 15 616 tokens, 1 and 511 experts, with and without
// dropping and skew (profiles/tile_choice_16bit_layers.txt): 3.2 % from the best of them in the mean, more than 10 % at 59 of them; 15 % faster in the mean than a
// choice by capacity alone (variant 1 up to 128 rows, 2 from 1 024, else 0), more than 3 % slower at seven (13 with
// every expert at its mean). Where it moves a layer from the
// 256- and 128-row tiles to the smaller ones: 640 tokens, 8 experts top-2, 704 x 512: 58 -> 37 us per forward; 2 176
// tokens, 16 experts top-2, 2 048 x 512: 91 -> 75; 2 048 tokens, one expert, 1 024 x 4 096: 148 -> 108.
// (The figures above are from before the wavefronts of a SIMD took turns in the 256-row tiles. With them, and the tall tiles below, the choice lies 4 % from the
// best at 155 other layers drawn alike; all constants fitted anew brought 1.9 %, at layers that other rules here are pinned to, and were not taken.)
// tf32: 256 x 256 tiles on the 16-bit matrix cores, 128 clocks per value of K, one on a CU, against 64 x 64 tiles on the fp32 ones,
// 32 clocks, two on a CU in turn. The large tile takes what it is charged (607 us per forward at 8 192 tokens, 64 experts top-2, 2 048 x
// 2 048, four rounds: 133 clocks; 272 at 2 048 tokens, 8 experts, one round each way: 123), bound by its loads; the 32 are the small one's
// matrix time, of which it reaches two thirds to three quarters (2 729 and 722 us: 43 and 47 clocks), so the line lies too high. Of
// 28 layers around it, timed on both, the rule takes the better tile at 17, with all that it gives to the large tile among them (4 096
// tokens, 8 experts top-2, 1 024 x 1 024: 171 against 392 us; 16 384, 64 experts top-1, 320 x 320: 119 against 132); 11 just below
// it would gain from the large one (2 048 tokens, 8 experts top-2, 1 024 x 1 024: 225 against 154; 1 024, 2 048 x 2 048: 398 against 257;
// 2 048, 64 experts, 2 048 x 2 048: 729 against 517), others not (512 tokens, one expert, 1 024 x 4 096: 206 against 287).
void choose_tiles(LayerParams& p, int dtype, int num_cus) {
    const uint32_t cap = p.EC < p.cap_rows ? p.EC : p.cap_rows;
    const uint32_t rows = mean_rows(p);
    p.tile_variant = 0u;
    p.down_small = 0u;
    p.tall = 0u;
    if (dtype == 0 || dtype == 1) {
        const double split = projections_us(p, TileCost{256, 256, 128.0, 0.0}, rows, num_cus, true);
        const double plain = projections_us(p, TileCost{64, 64, 32.0, 0.0}, rows, num_cus, false);
        if (dtype == 1 && split < plain) p.tile_variant = 3u;
        // The 32 x 32 tile takes 12 clocks per value of K on a busy CU (its loads); a tile costs some 3 us besides. Its row
        // blocks need a readiness counter each, of which there is one per 64 rows that an expert's arrays hold: that, not
        // a measurement, keeps it to experts of at most 64 rows.
        const double medium = projections_us(p, TileCost{64, 64, 32.0, 6500.0}, rows, num_cus, false);
        const double small = projections_us(p, TileCost{32, 32, 12.0, 6500.0}, rows, num_cus, false);
        if (p.tile_variant == 0u && small < medium && ceil_div_u32(cap, 32) <= ceil_div_u32(p.cap_rows, 64)) p.tile_variant = 7u;
        return;
    }
    // (bm x bn tiles, the down-projection on dm x dn tiles)
    RowShare shares[4];
    const int n_shares = row_shares(p, shares);
    auto row_blocks = [&](uint32_t bm) {   // of an expert, in the mean
        double blocks = 0.0;
        for (int i = 0; i < n_shares; ++i) blocks += shares[i].share * std::ceil(shares[i].rows / bm - 1e-9);
        return blocks;
    };
    auto projection = [&](uint32_t bm, uint32_t bn, uint32_t N, uint32_t K) {
        const double rounds = p.E * row_blocks(bm) * ceil_div_u32(N, bn) / num_cus;
        const TileCost t = tile16_cost(bm, bn, rows);
        return double(uint64_t(rounds + 0.999999)) * (K * t.per_k + t.fixed);
    };
    auto estimate = [&](uint32_t bm, uint32_t bn, uint32_t dm, uint32_t dn, bool streams) {
        const double tiles = projection(bm, bn, p.I, p.H) + projection(dm, dn, p.H, p.I);
        double memory = 4.0 * p.E * p.H * double(p.I) / 6.2e6;
        if (!streams && rows <= bm) memory *= 1.12;
        return (tiles > memory ? tiles : memory) + 0.1 * tiles;
    };
    // The smaller tile in the down-projection: a workgroup that goes over to it empties its pipeline once, and layers
    // bound by their weights gain nothing (256 tokens, 17 experts of 1 088 x 2 048: 59 -> 66 us without this allowance).
    // The best tiles without it against those with it, of the layers named above: 2 048 tokens, one expert, 1 024 x 4 096, dense:
    // 67 -> 63 us; 6 400 tokens, 896 x 2 496, dense: 112 -> 100; 2 432 tokens, 11 experts top-3, 640 x 12 544: 472 -> 422;
    // 1 024 tokens, 64 experts top-2, 320 x 9 216: 229 -> 218; 3 200 tokens, 320 x 14 144, dense: 215 -> 178.
    auto two_tiles = [&](uint32_t bm, uint32_t bn, uint32_t dm, uint32_t dn, bool streams) { return 1.06 * estimate(bm, bn, dm, dn, streams) + 5.0; };
    double us = 1e30;
    auto consider = [&](uint32_t variant, uint32_t small, double estimated) {
        if (estimated < us) { us = estimated; p.tile_variant = variant; p.down_small = small; }
    };
    // Experts of several row blocks each, one and more to an XCD: the 256-row tiles, which share their weights through
    // an L2 and mix heights, without asking; the estimate does not know of the sharing. (4 096 tokens, 8 experts top-2,
    // 1 024 x 1 024: 75 us against 90 with 128 x 128 tiles; 8 192 tokens, 12 experts, 768 x 3 072: 211 against 292; the
    // smallest lose, 53 against 47 at 512 x 512. Where exactly the line should lie, below 8 experts and 512 rows, is not measured.)
    const bool many = cap >= kSharedRows && rows >= kSharedRows / 2 && p.E >= 8;
    const bool narrow = rows <= kNarrowRows, shared = cap >= kSharedRows;
    if (narrow) {
        consider(1, 0, estimate(128, 256, 128, 256, true));
        consider(1, 1, two_tiles(128, 256, 128, 128, true));
    }
    if (!narrow || cap > kNarrowRows) consider(shared ? 2 : 0, 0, estimate(256, 256, 256, 256, !shared));
    if (!narrow && !many) consider(2, 1, two_tiles(256, 256, 128, 256, false));   // (variant 2 halves the last tiles of many rows anyway)
    if (many) return;
    // 64 rows: the weights non-temporally (6) where an expert reads them once and they bound the layer. Where no expert is
    // likely to hold more, a tile of 128 takes in no more rows and gains nothing on one of 64, which then comes first (40 such
    // layers: 4 to 7 % faster than on 128).
    const bool single = rows <= 64, likely = rows <= 32 || cap <= 64;
    auto low = [&] {
        consider(5, 0, estimate(64, 128, 64, 128, false));
        if (single) consider(6, 0, estimate(64, 128, 64, 128, true));
    };
    if (likely) low();
    consider(4, 0, estimate(128, 128, 128, 128, false));
    consider(4, 1, two_tiles(128, 128, 64, 128, false));
    if (!likely) low();
    // Variant 4 on tiles of 256 x 128 where experts hold more than 128 rows and whole rounds of what a value of K takes on either
    // tile (GemmTurns, 1 290 clocks per 64, against GemmKSplit, 1 010) come to less: half as many tiles in whatever runs on them. Row blocks of another
    // height also lie differently on the XCDs, and a layer whose fullest queue takes longer than the grid would is handed out (set_up in the persistent
    // kernel), which costs some 10 us at these sizes. Us per forward on tall and on 128-row tiles: 2 304 tokens, 4 experts top-4, 384 x 384, strided on tall ones
    // only 48.3 / 68.5; 3 072 tokens, one expert, 2 240 x 832, strided on 128-row ones only 93.3 / 73.3; 2 048 tokens, one expert, 1 024 x 4 096 70.3 / 76.2.
    // Of 540 layers of variant 4, timed on both (weights from HBM), the choice lies 1.2 % from the better tile in the mean; without the 10 us 2.4, without tall tiles 5.1,
    // with nothing but tall ones 2.8. It loses more than 5 % to 128-row tiles at 20 (29 without the 10 us, 27 % at most).
    if (p.tile_variant == 4u && rows > 128u) {
        auto rounds_us = [&](uint32_t bm, double per_k) {
            const double blocks = row_blocks(bm), queue = p.E == 1 ? std::ceil(blocks / kXcds - 1e-6) : double(ceil_div_u32(p.E, kXcds)) * blocks;
            const double small = row_blocks(64), small_queue = p.E == 1 ? queue * (bm / 64) : double(ceil_div_u32(p.E, kXcds)) * small;
            auto rounds = [&](double tiles) { return std::ceil(tiles / num_cus - 1e-6); };
            auto fits = [&](double of_queue, double of_all, uint32_t columns) { return rounds(of_queue * kXcds * columns) <= rounds(of_all * columns); };
            const uint32_t up = ceil_div_u32(p.I, 128), down = ceil_div_u32(p.H, 128);
            double us = rounds(p.E * blocks * up) * (p.H * per_k + 5.0);
            if (!p.down_small) us += rounds(p.E * blocks * down) * (p.I * per_k + 5.0);
            const bool strided = fits(queue, p.E * blocks, up) && (p.down_small ? fits(small_queue, p.E * small, down) : fits(queue, p.E * blocks, down));
            return strided ? us : us + 10.0;
        };
        p.tall = rounds_us(256, 0.0115) < rounds_us(128, 0.0085);
    }
}

uint32_t gate_splits_for(uint32_t S, uint32_t H, uint32_t E, uint32_t PX, int dtype, int num_cus) {
    if ((dtype != 2 && dtype != 3) || E <= 64) return 0;
    const uint32_t tiles = (S / kGateTileM) * ceil_div_u32(PX, kGateTileN);
    uint32_t splits = ceil_div_u32(uint32_t(num_cus), tiles ? tiles : 1u);
    const uint32_t slices = H / 64;
    if (splits > slices) splits = slices;
    if (splits > kGateMaxSplits) splits = kGateMaxSplits;
    return splits < 1 ? 1u : splits;
}

// Calls go(Element{}) for the Element type of a torch_dtype value (kleos_amd.h: 0 fp32, 1 tf32, 2 bf16, 3 fp16).
template <typename F>
hipError_t dispatch_dtype(int dtype, F&& go) {
    switch (dtype) {
        case 1: return go(tf32_t{});
        case 2: return go(bf16_t{});
        case 3: return go(f16_t{});
        default: return go(float{});
    }
}

void tile_sizes(const LayerParams& p, int dtype, uint32_t sizes[4]) {
    (void)dispatch_dtype(dtype, [&](auto tag) {
        using T = decltype(tag);
        return dispatch_variant<T>(p, [&](auto variant) {
            constexpr int V = decltype(variant)::value;
            const bool small = small_down<T, V>(p);
            sizes[0] = TileShape<T, V>::BM; sizes[1] = TileShape<T, V>::BN;
            sizes[2] = small ? kNarrowTileRows<V> : sizes[0]; sizes[3] = small ? kNarrowTileCols<V> : sizes[1];
            return hipSuccess;
        });
    });
}

hipError_t launch_gate(const LayerParams& p, int dtype, int num_cus, hipStream_t s) {
    return dispatch_dtype(dtype, [&](auto tag) { return launch_gate_t<decltype(tag)>(p, num_cus, s); });
}

hipError_t launch_slots(const LayerParams& p, hipStream_t s) {
    const uint32_t grid = ceil_div_u32(p.n_gate_tiles, 4);
    hipLaunchKernelGGL(slot_kernel, dim3(grid), dim3(kPhaseThreads), 4 * slot_tile_words(p.E, kWave) * sizeof(uint32_t), s, p);
    return hipGetLastError();
}

hipError_t launch_dense_rows(const LayerParams& p, hipStream_t s) {
    hipLaunchKernelGGL(dense_rows_kernel, dim3(ceil_div_u32(p.S, kPhaseThreads)), dim3(kPhaseThreads), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_expert_gemm(const LayerParams& p, int dtype, int kind, int num_cus, hipStream_t s) {
    return dispatch_dtype(dtype, [&](auto tag) { return launch_expert_gemm_t<decltype(tag)>(p, kind, num_cus, s); });
}

hipError_t launch_combine(const LayerParams& p, int dtype, hipStream_t s) {
    return dispatch_dtype(dtype, [&](auto tag) { return launch_combine_t<decltype(tag)>(p, s); });
}

hipError_t plan_fused(const LayerParams& p, int dtype, int num_cus, FusedPlan* plan) {
    return dispatch_dtype(dtype, [&](auto tag) { return plan_fused_t<decltype(tag)>(p, num_cus, plan); });
}

hipError_t launch_fused(const LayerParams& p, const FusedPlan& plan, uint32_t fused_seq, int schedule, hipStream_t s) {
    uint32_t seq = fused_seq;
    uint32_t mt_max = plan.mt_max, lag = plan.lag, policy = uint32_t(schedule);
    LayerParams pc = p;
    void* args[] = {&pc, &seq, &mt_max, &lag, &policy};
    // A cooperative launch makes the runtime verify that the whole grid can be resident at once
    // (it fails with hipErrorCooperativeLaunchTooLarge otherwise); it costs about 14 us per launch.
    if (plan.cooperative) return hipLaunchCooperativeKernel(plan.kernel, dim3(plan.nwg), dim3(plan.threads), args, plan.smem, s);
    return hipLaunchKernel(plan.kernel, dim3(plan.nwg), dim3(plan.threads), args, plan.smem, s);
}


// ------------------------------------------------------------------------------------ probe
namespace {
template <int TILE>
__global__ __launch_bounds__(512, 1) void mfma_probe_kernel(const uint32_t* data, float* sink, uint32_t iterations) {
    // eight operand fragments of each kind per lane, as a 128 x 64 wavefront tile keeps them around
    bf16x8 fa[8], fb[8];
    const u32x4* pool = reinterpret_cast<const u32x4*>(data);
    constexpr uint32_t kMask = uint32_t(kMfmaProbeWords / 4 - 1);
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
        fa[i] = __builtin_bit_cast(bf16x8, pool[(blockIdx.x * 512u + threadIdx.x + i * 4096u) & kMask]);
        fb[i] = __builtin_bit_cast(bf16x8, pool[(blockIdx.x * 512u + threadIdx.x + i * 4096u + 77777u) & kMask]);
    }
    float total = 0.f;
    if constexpr (TILE == 32) {
        f32x16 acc[2][4] = {};
        for (uint32_t it = 0; it < iterations; ++it)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int m = 0; m < 4; ++m)
                        acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[(n + 2 * ks) & 7], fa[(m + ks) & 7], acc[n][m], 0, 0, 0);
        for (int n = 0; n < 2; ++n) for (int m = 0; m < 4; ++m) for (int i = 0; i < 16; ++i) total += acc[n][m][i];
    } else {
        f32x4 acc[4][8] = {};
        for (uint32_t it = 0; it < iterations; ++it)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int m = 0; m < 8; ++m)
                        acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[(n + 4 * ks) & 7], fa[(m + ks) & 7], acc[n][m], 0, 0, 0);
        for (int n = 0; n < 4; ++n) for (int m = 0; m < 8; ++m) for (int i = 0; i < 4; ++i) total += acc[n][m][i];
    }
    if (total == 12345.678f) *sink = total;   // keeps the loop alive; never true in practice
}

__global__ void mfma_probe_fill_kernel(uint32_t* data, size_t words, uint32_t zero) {
    for (size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x; i < words; i += size_t(gridDim.x) * blockDim.x) {
        uint32_t h = uint32_t(i) * 2654435761u + 12345u;
        h ^= h >> 15; h *= 2246822519u; h ^= h >> 13; h *= 3266489917u; h ^= h >> 16;
        // two bf16: sign and 7 mantissa bits random, exponent 0x7e or 0x7f (0.5 <= |v| < 2)
        const uint32_t lo = (h & 0x80ffu) | 0x3f00u, hi = ((h >> 16) & 0x80ffu) | 0x3f00u;
        data[i] = zero ? 0u : (lo | (hi << 16));
    }
}
}  // namespace

hipError_t launch_mfma_probe(int tile, uint32_t iterations, const uint32_t* data, float* sink, int num_cus, double* flop,
                             hipStream_t s) {
    if (tile != 16 && tile != 32) return hipErrorInvalidValue;
    // per iteration and wavefront: a 128 x 64 tile advanced by 64 values of K
    if (flop) *flop = double(num_cus) * 8.0 * double(iterations) * 2.0 * 128.0 * 64.0 * 64.0;
    if (tile == 32) hipLaunchKernelGGL(mfma_probe_kernel<32>, dim3(num_cus), dim3(512), 0, s, data, sink, iterations);
    else hipLaunchKernelGGL(mfma_probe_kernel<16>, dim3(num_cus), dim3(512), 0, s, data, sink, iterations);
    return hipGetLastError();
}

hipError_t launch_mfma_probe_fill(uint32_t* data, size_t words, bool zero, hipStream_t s) {
    hipLaunchKernelGGL(mfma_probe_fill_kernel, dim3(2048), dim3(256), 0, s, data, words, zero ? 1u : 0u);
    return hipGetLastError();
}

}  // namespace kleos_amd
