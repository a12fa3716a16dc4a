// Gate: logits GEMM fused with softmax, top-k and the per-tile expert histogram, then the
// token-order slot assignment with capacity drop.
//
// Replaces gate::FusedGate / gate::forward of the reference (csrc/include/kleos/moe/gate.cuh:
// 474-720, 729-789). Differences that matter:
//   * one wavefront quad of lanes owns a token, so softmax and top-k are register + cross-lane
//     shuffle work; the reference bounces the accumulator through shared memory to get one
//     thread per token (gate.cuh:560-572);
//   * every expert count is handled inside one workgroup: up to 256 experts with the logits in
//     registers, more in passes of 256 (the reference chains
//     64-expert blocks through global-memory mailboxes, gate.cuh:93-468);
//   * slots are assigned in token order from per-tile histograms and their prefix sums, which
//     makes dropping deterministic; the reference takes a tile's base slot from atomicAdd arrival
//     order (gate.cuh:699).
#pragma once
#include <type_traits>

#include "device_common.hpp"

namespace kleos_amd {

template <typename T>
struct GateK {
    static constexpr int kElemsPer16B = 16 / sizeof(T);
    // K consumed by one mma16_step: each of the 4 lane groups brings 16 bytes
    static constexpr int kStepK = 4 * kElemsPer16B;
};

// Token blocks (16 tokens each) one gate unit works on together: the fragments of the gate weights
// are loaded once per unit and used by every block, which halves the L2 traffic of the weights.
// With 16 expert groups (E > 128) the accumulators of two blocks no longer fit the register file.
// NG = 0 stands for the wide gate (E > 256), which works in passes of 16 groups.
template <int NG>
constexpr int gate_unit_blocks() { return NG == 0 || NG >= 16 ? 1 : 2; }

__host__ __device__ inline uint32_t gate_group_words(uint32_t E, uint32_t k, bool training);
// Softmax, top-k, outputs and histogram of a 16-token tile by a group of four wavefronts (below).
template <typename T, int NL>
__device__ __forceinline__ void gate_group_finish(const LayerParams& p, uint32_t tile, bool valid, f32x4 (&acc)[NL], uint32_t* gsm, uint32_t gtid);
// Up to 64 experts (four groups) and a multiple of four wavefronts: the epilogue of a block is
// shared out over a group of four wavefronts instead of run by one.
template <int NG>
constexpr bool gate_unit_grouped(int kw) { return NG >= 1 && NG <= 4 && kw % 4 == 0; }
// Row stride of the parked partial sums in the grouped epilogue: one word more than a wavefront
// writes, so that the reads, which walk the rows four at a time, spread over all banks.
constexpr int kGateParkStride = kWave + 1;
// LDS floats needed by gate_unit with KW wavefronts: the partial accumulators (4*NG registers of
// 64 lanes) of the KW shares of the hidden dimension of the block being reduced, in padded rows (its epilogue's scratch
// takes their place, 33 words an expert at most); up to 64 experts those of both blocks, and the scratch of the groups.
template <int NG>
constexpr int gate_smem_floats(int kw) {
    if (gate_unit_grouped<NG>(kw)) return 2 * kw * NG * 4 * kGateParkStride + (kw / 4) * int(kGateTileTokens * 64 + 64 + kGateTileTokens * 64);
    return kw * (NG == 0 ? 16 : NG) * kGateParkStride * 4;
}
constexpr uint32_t kWideGateMaxK = 32, kWideGateMaxE = 512;   // of the gate of more than 256 experts

// Sums of the K steps s0 .. s1-1 of TB token blocks against NG groups of 16 experts, from zero: logits^T, experts are
// the matrix-core rows, tokens its columns (gate.cuh:526-534). `xrow`, `wrow`: the lane's own row at its chunk of a step.
// The loads of U steps are in flight together: the activation rows stream from HBM once and this is what
// keeps enough of them in flight. They are issued in halves of U / 2 steps, and a half is
// requested again (for U steps further on) as soon as its matrix instructions have read it, so
// the memory pipeline never runs empty between one batch and the next (worth 0.5 us of 12.5 per
// workgroup at the 64-expert shape with a hidden size of 2048: the loop runs at what a CU gets
// of the memory system while all CUs stream, about 32 GB/s). Fewer than U steps that are left over are one more
// batch, of just their loads. (Filled up to U with
// repeated loads such a batch cost more than it saved: gate phase of 15 616 tokens of 512 values, 27 experts, 25.4 against
// 16.7 us; of 4 096 tokens of 256 values, 16 experts, 12.6 against 8.9.)
template <typename T, int NG, int TB, int U>
__device__ __forceinline__ void gate_accumulate(const T* (&xrow)[TB], const T* wrow, uint32_t H, uint32_t s0, uint32_t s1, f32x4 (&acc)[TB][NG]) {
    constexpr int kStepK = GateK<T>::kStepK;
    constexpr int UH = U >= 2 ? U / 2 : 1;
#pragma unroll
    for (int b = 0; b < TB; ++b)
#pragma unroll
        for (int g = 0; g < NG; ++g) acc[b][g] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 xb[U][TB], wa[U][NG];
    auto load_step = [&](int u, uint32_t step) {
        const uint32_t off = step * kStepK;
#pragma unroll
        for (int b = 0; b < TB; ++b) xb[u][b] = load16(xrow[b] + off);
#pragma unroll
        for (int g = 0; g < NG; ++g) wa[u][g] = load16(wrow + size_t(g) * 16 * H + off);
    };
    auto multiply_step = [&](int u) {
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int b = 0; b < TB; ++b) acc[b][g] = mma16_step(wa[u][g], xb[u][b], acc[b][g], T{});
    };
    uint32_t s = s0;
    if constexpr (U >= 2) {
        auto issue = [&](auto first_slot, uint32_t s_first) {
            constexpr int u0 = decltype(first_slot)::value;
#pragma unroll
            for (int u = 0; u < UH; ++u) load_step(u0 + u, s_first + u);
            __builtin_amdgcn_sched_barrier(0);   // the loads stay where they are written
        };
        auto consume = [&](auto first_slot) {
            constexpr int u0 = decltype(first_slot)::value;
#pragma unroll
            for (int u = 0; u < UH; ++u) multiply_step(u0 + u);
            __builtin_amdgcn_sched_barrier(0);
        };
        constexpr std::integral_constant<int, 0> lower{};
        constexpr std::integral_constant<int, UH> upper{};
        if (s + U <= s1) {
            issue(lower, s);
            issue(upper, s + UH);
            for (; s + 2 * U <= s1; s += U) {
                consume(lower);
                issue(lower, s + U);
                consume(upper);
                issue(upper, s + U + UH);
            }
            consume(lower);
            consume(upper);
            s += U;
        }
        // left over: runs of U / 2, U / 4, ... 1 steps, as its bits say; run R in the slots from U - 2 R on
        const uint32_t left = s1 - s;
        auto runs = [&](auto&& f) {
            uint32_t at = s;
            auto run = [&](auto size) {
                constexpr int R = decltype(size)::value;
                if (R >= 1 && (left & uint32_t(R))) {
#pragma unroll
                    for (int u = 0; u < R; ++u) f(U - 2 * R + u, at + u);
                    at += R;
                }
            };
            run(std::integral_constant<int, U / 2>{});
            run(std::integral_constant<int, U / 4>{});
            run(std::integral_constant<int, U / 8>{});
            run(std::integral_constant<int, U / 16>{});
        };
        runs([&](int u, uint32_t step) { load_step(u, step); });
        __builtin_amdgcn_sched_barrier(0);
        runs([&](int u, uint32_t) { multiply_step(u); });
    } else {
        for (; s < s1; ++s) {
            load_step(0, s);
            multiply_step(0);
        }
    }
}

// One gate unit: TB consecutive 16-token tiles (gate_unit_blocks<NG>(), or one where the tiles are fewer than workgroups), computed by KW wavefronts of the
// workgroup (all of them, or one of several such groups, each with a unit and LDS of its own), which
// split the hidden dimension. Wavefront b then reduces the partial sums of block
// b in a fixed order and runs its epilogue. Every thread of the workgroup must call the function
// (it contains workgroup barriers); `smem` holds gate_smem_floats<NG>(KW) floats and may be reused
// after the call.
template <typename T, int NG, int KW, int TB = gate_unit_blocks<NG>()>
__device__ __forceinline__ void gate_unit(const LayerParams& p, uint32_t unit, float* smem) {
    static_assert(TB <= KW);
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)) % KW, lane = threadIdx.x & 63;
    const int col = lane & 15;       // token inside a block / expert row inside a group
    const int chunk = lane >> 4;     // which 16-byte K chunk of a step this lane loads
    const uint32_t H = p.H;
    constexpr int kStepK = GateK<T>::kStepK;
    constexpr int kPer = GateK<T>::kElemsPer16B;
    const uint32_t steps = H / kStepK;
    // Wavefront w works on share (w + unit / 8) % KW of the hidden dimension: the units that run on
    // one XCD at the same time (unit numbers 8 apart) then ask its L2 for different lines of the
    // gate weights at any moment instead of all for the same ones.
    const uint32_t part = (uint32_t(wave) + (unit >> 3)) % uint32_t(KW);
    // (a unit past the last one, which a group is handed when the units run out, sums nothing)
    const uint32_t s0 = (steps * part) / KW, s1 = unit * TB < p.n_gate_tiles ? (steps * (part + 1)) / KW : s0;

    const T* xrow[TB];
    bool live[TB];
#pragma unroll
    for (int b = 0; b < TB; ++b) {
        const uint32_t tile = unit * TB + b;
        live[b] = tile < p.n_gate_tiles;
        // a block past the end re-reads the last tile; nothing of it is written
        const uint32_t token = (live[b] ? tile : p.n_gate_tiles - 1) * kGateTileTokens + col;
        xrow[b] = static_cast<const T*>(p.x) + size_t(token) * H + chunk * kPer;
    }
    const T* wrow = static_cast<const T*>(p.wg) + size_t(col) * H + chunk * kPer;

    f32x4 acc[TB][NG];
    gate_accumulate<T, NG, TB, (NG <= 2 ? 8 : (NG <= 4 ? 4 : (NG <= 8 ? 2 : 1)))>(xrow, wrow, H, s0, s1, acc);

    if constexpr (gate_unit_grouped<NG>(KW)) {
        // Every wavefront parks the partial sums of its share of both blocks in LDS; block b then
        // belongs to group b of four wavefronts (one group: block after block), 16 lanes per token
        // and four experts per lane, which add the shares in ascending order (a fixed order: the
        // logits depend neither on timing nor on which wavefront worked on which share).
        static_assert(TB <= 2);
        constexpr int kShare = NG * 4 * kGateParkStride;
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            float* dst = smem + (b * KW + part) * kShare;
#pragma unroll
            for (int g = 0; g < NG; ++g)
#pragma unroll
                for (int v = 0; v < 4; ++v) dst[(g * 4 + v) * kGateParkStride + lane] = acc[b][g][v];
        }
        __syncthreads();
        constexpr int kGroups = KW / 4;
        const uint32_t group = uint32_t(wave) >> 2, gtid = threadIdx.x & 255u;
        uint32_t* gsm = reinterpret_cast<uint32_t*>(smem + TB * KW * kShare) + group * gate_group_words(p.E, p.k, p.is_training != 0);
        const int sub = lane & 15;                              // experts 4 sub .. 4 sub + 3
        const int tl = 4 * (wave & 3) + (lane >> 4);            // token inside the block
#pragma unroll
        for (int b0 = 0; b0 < TB; b0 += kGroups) {
            const uint32_t b = b0 + group;
            const uint32_t tile = unit * TB + b;
            const bool valid = b < uint32_t(TB) && tile < p.n_gate_tiles;
            f32x4 sum[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
            if (valid && sub < 4 * NG) {
                // expert 4 sub + v sits in row 4 (sub / 4) + v of a share, at lane 16 (sub % 4) + token
                const float* src = smem + (b * KW) * kShare + ((sub >> 2) * 4) * kGateParkStride + 16 * (sub & 3) + tl;
#pragma unroll
                for (int v = 0; v < 4; ++v) sum[0][v] = src[v * kGateParkStride];
#pragma unroll
                for (int w = 1; w < KW; ++w)
#pragma unroll
                    for (int v = 0; v < 4; ++v) sum[0][v] += src[w * kShare + v * kGateParkStride];
            }
            gate_group_finish<T, 1>(p, tile, valid, sum, gsm, gtid);
        }
        return;
    }
    // More experts, block after block: every wavefront parks the partial sums of its share in LDS, one group of four adds
    // them in ascending order, each lane four experts of every 64, and finishes the block. Softmax and top-k by a single
    // wavefront, whose lanes each held a quarter of a token's experts, were a chain of some 3 000 instructions beside idle
    // wavefronts, with 2 053 to 2 110 registers spilled at 128 experts. 32-bit Elements, us per forward (256 columns up): 1 024 tokens of
    // 1 024 values, 128 experts top-2, fp32 180 -> 129, 256 experts top-8 307 -> 247; 15 616 tokens of 512 values, 128 experts
    // top-2, fp32 406 -> 298, tf32 391 -> 198, 256 experts top-4, tf32 497 -> 300; 4 096 tokens of 2 048, 256 experts, fp32 542 -> 490.
    static_assert(gate_unit_grouped<NG>(KW) || NG % 4 == 0);   // the reads below take whole runs of four groups
    constexpr int NL = (NG + 3) / 4;
    const uint32_t group = uint32_t(wave) >> 2, gtid = threadIdx.x & 255u;
    uint32_t* gsm = reinterpret_cast<uint32_t*>(smem) + group * gate_group_words(p.E, p.k, p.is_training != 0);
    const int sub = lane & 15;                              // experts 64 j + 4 sub .. + 3
    const int tl = 4 * (wave & 3) + (lane >> 4);            // token inside the block
#pragma unroll
    for (int b = 0; b < TB; ++b) {
        constexpr int kShare = NG * 4 * kGateParkStride;
        float* dst = smem + part * kShare;
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v) dst[(g * 4 + v) * kGateParkStride + lane] = acc[b][g][v];
        __syncthreads();
        const bool mine = live[b] && group == 0;
        f32x4 sum[NL];
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            sum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (!mine) continue;
            const float* src = smem + (16 * j + (sub & 12)) * kGateParkStride + 16 * (sub & 3) + tl;
#pragma unroll
            for (int v = 0; v < 4; ++v) sum[j][v] = src[v * kGateParkStride];
#pragma unroll
            for (int w = 1; w < KW; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) sum[j][v] += src[w * kShare + v * kGateParkStride];
        }
        __syncthreads();   // the sums are in registers: their LDS is the epilogue's
        gate_group_finish<T, NL>(p, unit * TB + b, mine, sum, gsm, gtid);
    }
}

// Few tokens leave most CUs without a gate unit, and a unit's loop runs at what one CU gets of the memory system (128
// tokens of 4 096 values, 8 experts: four units, 16 us, spread 8; 768 tokens of 4 224 32-bit values, 256 experts: 422 us,
// spread 114). The tiles are then spread: a virtual workgroup of KW wavefronts
// takes KW / ways shares of the hidden dimension of one 16-token tile and, above 64 experts (32-bit Elements), 64 of the
// experts. Every wavefront writes the sums of its share through the L2, and the workgroup that arrives last at a tile
// adds the shares in the order of gate_unit - the logits have the same bits - and finishes the tile.
// The sums lie in `y`, which nobody needs before the experts run. The arrivals are counted, without ever being reset, in
// the spare words of 32 lines that hold one counter of the scheduler each (`lines`): tile t in line t % 32.
constexpr uint32_t kArrivalLines = 32, kArrivalLineWords = 32;
template <int NG> constexpr uint32_t gate_spread_quarters() { return NG > 4 ? NG / 4 : 1; }
// ways (a power of two): as many workgroups a tile as keep the grid to one round. 0: whole units, where they fill the grid
// themselves (a tile by a single workgroup gains nothing either) or the sums do not fit. `groups`: the grid, in virtual workgroups.
template <typename T, int NG, int KW>
__device__ __forceinline__ uint32_t gate_spread_ways(const LayerParams& p, uint32_t groups) {
    if constexpr (NG == 0) return 0u;
    constexpr uint32_t Q = gate_spread_quarters<NG>(), TB = gate_unit_blocks<NG>();
    if ((p.n_gate_tiles + TB - 1) / TB >= groups || p.n_gate_tiles > kArrivalLines * (kArrivalLineWords - 1)) return 0u;
    if (size_t(p.n_gate_tiles) * KW * NG * 1024 > size_t(p.E) * y_expert_elems(p.cap_rows, p.H, sizeof(T)) * sizeof(T)) return 0u;
    uint32_t ways = 1;
    while (ways < uint32_t(KW) && p.n_gate_tiles * Q * ways * 2 <= groups) ways *= 2;
    // The sums' way through memory costs about 3 us, which 32 KB a microsecond and CU have to bring back: 2 048 tokens
    // of 1 024 values (one expert, 66 KB less a unit) lose 1 us, 1 920 of 1 472 (24 experts, 118 KB less) gain 2.7. Units of
    // four wavefronts load at half the rate: 128 tokens of 256 32-bit values (40 KB less) gain 1 us.
    constexpr uint32_t G = NG > 4 ? 4 : NG;
    if (p.H * uint32_t(sizeof(T)) * ((16 * TB + 16 * NG) - (16 + 16 * G) / ways) < 10u * KW * 1024u) return 0u;
    return ways * Q >= 2 ? ways : 0u;
}

// Virtual workgroup `group` (0 .. groups-1) of the spread gate; every thread of every workgroup must call it. `smem`:
// gate_smem_floats<NG>(KW) floats of the virtual workgroup's own.
template <typename T, int NG, int KW>
__device__ __forceinline__ void gate_spread(const LayerParams& p, uint32_t ways, uint32_t group, uint32_t groups, uint32_t* lines, float* smem) {
    constexpr uint32_t Q = gate_spread_quarters<NG>();
    constexpr int G = NG > 4 ? 4 : NG;                   // groups of 16 experts a wavefront works on
    constexpr int U = G == 1 ? 16 : 8;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)) % KW, lane = threadIdx.x & 63;
    const int col = lane & 15, chunk = lane >> 4;
    constexpr int kPer = GateK<T>::kElemsPer16B;
    const uint32_t steps = p.H / GateK<T>::kStepK, shares = KW / ways, total = p.n_gate_tiles * Q * ways;
    uint32_t* flag = reinterpret_cast<uint32_t*>(smem);
    const uint32_t rounds = (total + groups - 1) / groups;
    for (uint32_t round = 0; round < rounds; ++round) {
        const uint32_t item = group + round * groups;    // (the workgroups of an XCD get the same shares where ways is 8)
        const bool valid = item < total;
        const uint32_t sub = item % ways, rest = item / ways;
        const uint32_t tile = valid ? rest % p.n_gate_tiles : 0u, quarter = rest / p.n_gate_tiles;
        const coherent_rows_t sums = coherent_rows(static_cast<const char*>(p.y) + size_t(tile) * KW * NG * 1024);
        if (valid && uint32_t(wave) < shares) {
            const uint32_t share = sub * shares + uint32_t(wave);
            const T* xrow[1] = {static_cast<const T*>(p.x) + size_t(tile * kGateTileTokens + col) * p.H + chunk * kPer};
            const T* wrow = static_cast<const T*>(p.wg) + size_t(quarter * 16 * G + col) * p.H + chunk * kPer;
            f32x4 acc[1][G];
            gate_accumulate<T, G, 1, U>(xrow, wrow, p.H, (steps * share) / KW, (steps * (share + 1)) / KW, acc);
#pragma unroll
            for (int g = 0; g < G; ++g)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[0][g]), sums,
                                                       int(((share * NG + quarter * G + g) * kWave + lane) * 16), 0, 16);
        }
        wait_vmcnt<0>();
        __syncthreads();
        if (valid && wave == 0 && lane == 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            const uint32_t arrived = atomic_add_agent(lines + (tile % kArrivalLines) * kArrivalLineWords + 1 + tile / kArrivalLines, 1u) + 1u;
            *flag = uint32_t(arrived % (ways * Q) == 0u);
        }
        __syncthreads();
        const bool last = valid && *flag != 0u;
        asm volatile("" ::: "memory");   // the sums are read behind the arrival
        const uint32_t part = uint32_t(wave) >> 2, gtid = threadIdx.x & 255u;
        uint32_t* gsm = reinterpret_cast<uint32_t*>(smem) + kWave + part * gate_group_words(p.E, p.k, p.is_training != 0);
        constexpr int NL = (NG + 3) / 4;
        const int sub16 = lane & 15;                            // experts 64 j + 4 sub16 .. + 3
        const int tl = 4 * (wave & 3) + (lane >> 4);            // token inside the tile
        f32x4 sum[NL];
#pragma unroll
        for (int j = 0; j < NL; ++j) sum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const bool mine = last && part == 0;
        if (mine && sub16 < 4 * NG) {
#pragma unroll
            for (int j = 0; j < NL; ++j) {
                // expert 64 j + 4 sub16 + v is word v of lane 16 (sub16 % 4) + token of the share's group 4 j + sub16 / 4
                u32x4 v[KW];
#pragma unroll
                for (int w = 0; w < KW; ++w)
                    v[w] = load16_coherent(sums, uint32_t(((w * NG + 4 * j + (sub16 >> 2)) * kWave + 16 * (sub16 & 3) + tl) * 16));
                sum[j] = __builtin_bit_cast(f32x4, v[0]);
#pragma unroll
                for (int w = 1; w < KW; ++w) sum[j] += __builtin_bit_cast(f32x4, v[w]);
            }
        }
        gate_group_finish<T, NL>(p, tile, mine, sum, gsm, gtid);
    }
}

// The gate of 32-bit Elements for more than 256 experts: one 16-token block per unit, the experts in passes of 256.
// Every pass is the K loop of gate_unit with 16 groups; a group of four wavefronts adds the shares in ascending order, keeps them (each
// lane four experts of every 64) and finishes the block when all passes are done. Before, one wavefront stored the logits and read them
// back once and more for every pick, alone in its workgroup: 4 992 tokens of 256 values, 360 experts top-4, tf32: 221 us of 1 062.
// Every thread of the workgroup must call the function; `smem` holds gate_smem_floats<0>(KW) floats.
template <typename T, int KW>
__device__ __forceinline__ void gate_unit_wide(const LayerParams& p, uint32_t unit, float* smem) {
    constexpr int NG = 16, kPasses = int(kWideGateMaxE) / (16 * NG), NL = kPasses * NG / 4;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)) % KW, lane = threadIdx.x & 63;
    const int col = lane & 15, chunk = lane >> 4;
    const uint32_t H = p.H;
    constexpr int kStepK = GateK<T>::kStepK;
    constexpr int kPer = GateK<T>::kElemsPer16B;
    const uint32_t steps = H / kStepK;
    const uint32_t part = (uint32_t(wave) + (unit >> 3)) % uint32_t(KW);
    const uint32_t s0 = (steps * part) / KW, s1 = unit < p.n_gate_tiles ? (steps * (part + 1)) / KW : s0;
    const uint32_t tile = unit;
    const bool live = tile < p.n_gate_tiles;
    const uint32_t token = (live ? tile : p.n_gate_tiles - 1) * kGateTileTokens + col;
    const T* xrow = static_cast<const T*>(p.x) + size_t(token) * H + chunk * kPer;
    const uint32_t group = uint32_t(wave) >> 2, gtid = threadIdx.x & 255u;
    const int sub = lane & 15;                              // experts 64 j + 4 sub .. + 3
    const int tl = 4 * (wave & 3) + (lane >> 4);            // token inside the block
    const bool mine = live && group == 0;
    constexpr int kShare = NG * 4 * kGateParkStride;
    f32x4 sum[NL];

#pragma unroll
    for (int pass = 0; pass < kPasses; ++pass) {
        const uint32_t e0 = uint32_t(pass) * 16 * NG;
        f32x4 acc[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g) acc[g] = f32x4{0.f, 0.f, 0.f, 0.f};
        // weight rows past the padded expert count re-read its last row; their logits are never stored
        auto wrow = [&](int g) {
            const uint32_t r = e0 + 16 * g + col;
            return static_cast<const T*>(p.wg) + size_t(r < p.PX ? r : p.PX - 1) * H + chunk * kPer;
        };
        for (uint32_t s = s0; s < s1; ++s) {
            const uint32_t off = s * kStepK;
            const u32x4 xb = load16(xrow + off);
            u32x4 wa[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) wa[g] = load16(wrow(g) + off);
#pragma unroll
            for (int g = 0; g < NG; ++g) acc[g] = mma16_step(wa[g], xb, acc[g], T{});
        }
        float* dst = smem + part * kShare;
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v) dst[(g * 4 + v) * kGateParkStride + lane] = acc[g][v];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NG / 4; ++j) {
            f32x4 total{0.f, 0.f, 0.f, 0.f};
            if (mine) {
                const float* src = smem + (16 * j + (sub & 12)) * kGateParkStride + 16 * (sub & 3) + tl;
#pragma unroll
                for (int v = 0; v < 4; ++v) total[v] = src[v * kGateParkStride];
#pragma unroll
                for (int w = 1; w < KW; ++w)
#pragma unroll
                    for (int v = 0; v < 4; ++v) total[v] += src[w * kShare + v * kGateParkStride];
            }
            sum[pass * (NG / 4) + j] = total;
        }
        __syncthreads();
    }
    gate_group_finish<T, NL>(p, tile, mine, sum, reinterpret_cast<uint32_t*>(smem) + group * gate_group_words(p.E, p.k, p.is_training != 0), gtid);
}

// ------------------------------------------------------------------------------------------------
// Gate of the 16-bit Elements with more than 64 experts: the logits come from a tiled product
// (128 tokens x 256 experts per workgroup, the hidden dimension split into p.gate_splits ranges
// whose fp32 sums land in p.gate_partial[split][token][PX]), so the gate weights are read once per
// 128 tokens instead of once per 16 or 32. After a grid-wide barrier the 16-token tiles are
// reduced by a group of four wavefronts each: the
// ranges are added in ascending order (a fixed order: the logits do not depend on timing or on the
// launch mode), then softmax, top-k and the tile's histogram as in the other gates.
// ------------------------------------------------------------------------------------------------
// A tile worked on by a group of four wavefronts (256 threads): wavefront w of
// the group takes tokens 4 w .. 4 w + 3 of the tile, 16 lanes per token, each lane the experts
// 64 j + 4 (lane % 16) + v (j < NL, NL * 64 >= PX, v < 4). Against one wavefront per tile every per-lane
// loop over the experts is four times shorter, and the partial sums, logits and gate outputs move
// in runs of 256 and 128 bytes per token. The tile's picks meet in LDS: every pick counts the picks
// of its expert by earlier tokens for its in-tile rank and adds itself to the tile's histogram,
// which the group then writes out.
// `gsm`: gate_group_words(p) words of LDS private to the group. Every thread of the workgroup must
// call the function the same number of times (it contains workgroup barriers); a group without a
// tile passes valid = false.
__host__ __device__ inline uint32_t gate_group_words(uint32_t E, uint32_t k, bool training) {
    return kGateTileTokens * k + E + (training ? kGateTileTokens * E : 0u);
}
template <typename T, int NL>
__device__ __forceinline__ void gate_reduce_group(const LayerParams& p, uint32_t tile, bool valid, uint32_t* gsm, uint32_t gtid) {
    const int lane = gtid & 63, sub = lane & 15;
    const uint32_t tl = 4 * (gtid >> 6) + (lane >> 4);
    f32x4 acc[NL];
#pragma unroll
    for (int j = 0; j < NL; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (valid) {
        const uint32_t token = tile * kGateTileTokens + tl;
        const coherent_rows_t partial = coherent_rows(p.gate_partial);
        // range by range, in ascending order; the loads of eight ranges in flight together (two at a time the sixteen ranges of 128 tokens of 7 168
        // values, 256 experts, were eight trips to memory)
        constexpr uint32_t kRanges = NL > 4 ? 4 : 8;   // (at most 128 registers)
        for (uint32_t s0 = 0; s0 < p.gate_splits; s0 += kRanges) {
            u32x4 v[kRanges][NL];
#pragma unroll
            for (uint32_t u = 0; u < kRanges; ++u) {
                const uint32_t s = s0 + u < p.gate_splits ? s0 + u : s0;
                const uint32_t row = ((s * p.S + token) * p.PX + 4 * sub) * 4u;
#pragma unroll
                for (int j = 0; j < NL; ++j) v[u][j] = uint32_t(64 * j) < p.PX && s0 + u < p.gate_splits ? load16_coherent(partial, row + 256u * j) : u32x4{0, 0, 0, 0};
            }
#pragma unroll
            for (uint32_t u = 0; u < kRanges; ++u) {
                if (s0 + u < p.gate_splits) {
#pragma unroll
                    for (int j = 0; j < NL; ++j) acc[j] += __builtin_bit_cast(f32x4, v[u][j]);
                }
            }
        }
    }
    gate_group_finish<T, NL>(p, tile, valid, acc, gsm, gtid);
}

// The part of the group's work that follows the logits: `acc[j][v]` of a lane is the logit of expert
// 64 j + 4 (lane % 16) + v of its token (anything for experts past the padded count).
template <typename T, int NL>
__device__ __forceinline__ void gate_group_finish(const LayerParams& p, uint32_t tile, bool valid, f32x4 (&acc)[NL], uint32_t* gsm, uint32_t gtid) {
    constexpr uint32_t kGroupThreads = 4 * kWave;
    const int lane = gtid & 63, sub = lane & 15;
    const uint32_t gw = gtid >> 6, tl = 4 * gw + (lane >> 4);
    const uint32_t E = p.E, k = p.k;
    uint32_t* s_sel = gsm;                                   // [16][k] expert picked by token t in round r
    uint32_t* s_hist = gsm + kGateTileTokens * k;            // [E]
    float* s_prob = reinterpret_cast<float*>(s_hist + E);    // [16][E], training only
    for (uint32_t e = gtid; e < E; e += kGroupThreads) s_hist[e] = 0u;
    if (valid) {
        const uint32_t token = tile * kGateTileTokens + tl;
        const float kNegInf = -__builtin_inff();
        float m = kNegInf;
        const bool whole_quads = (E & 3u) == 0u;   // a lane's four experts are all real or all padding
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const uint32_t e0 = 64 * j + 4 * sub;
            if (whole_quads && e0 < E) *reinterpret_cast<f32x4*>(p.logits + size_t(token) * E + e0) = acc[j];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const uint32_t e = e0 + v;
                if (e >= E) acc[j][v] = kNegInf;   // softmax domain = the E real experts only (gate.cuh:550)
                else if (!whole_quads) p.logits[size_t(token) * E + e] = acc[j][v];
                m = fmaxf(m, acc[j][v]);
            }
        }
        m = row16_allreduce(m, [](float a, float b) { return fmaxf(a, b); });
        float d = 0.f;
#pragma unroll
        for (int j = 0; j < NL; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) d += __expf(acc[j][v] - m);
        d = row16_allreduce(d, [](float a, float b) { return a + b; });
        const float inv_d = 1.0f / d;
        auto prob = [&](float logit) { return __expf(logit - m) * inv_d; };
        // gateOut[t, e] = Element(p) (gate.cuh:590-605); padded columns are zero
        T* grow = static_cast<T*>(p.gate_out) + size_t(token) * p.PX;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            T o[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const uint32_t e = 64 * j + 4 * sub + v;
                o[v] = float_to_elem<T>(e < E ? prob(acc[j][v]) : 0.f);
                if (p.is_training && e < E) s_prob[tl * E + e] = prob(acc[j][v]);
            }
            // the padded row length is a multiple of 64: the four columns are inside the row together
            using Quad = std::conditional_t<sizeof(T) == 2, uint2, f32x4>;
            static_assert(sizeof(Quad) == 4 * sizeof(T));
            Quad raw;
            __builtin_memcpy(&raw, o, sizeof(Quad));
            if (uint32_t(64 * j) < p.PX) *reinterpret_cast<Quad*>(grow + 64 * j + 4 * sub) = raw;
        }
        // top-k: k rounds of arg-max, equal values go to the lower expert index (gate.cuh:654-670);
        // a picked expert becomes -inf in the working copy. A logit of -inf or NaN counts as the lowest finite value there, so that a
        // token that holds such logits picks k distinct experts too; so does what lies past the last expert, behind all of them by its index.
        f32x4 w[NL];
#pragma unroll
        for (int j = 0; j < NL; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) w[j][v] = fmaxf(acc[j][v], -__FLT_MAX__);
        float den = 0.f;
        constexpr uint32_t kNone = 0x7fffffffu;   // of a lane whose experts are taken
        for (uint32_t r = 0; r < k; ++r) {
            float best = kNegInf;
            uint32_t bi = kNone;
#pragma unroll
            for (int j = 0; j < NL; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (w[j][v] > best) {
                        best = w[j][v];
                        bi = 64 * j + 4 * sub + v;
                    }
            // (the rule is symmetric in the two candidates, so the lanes of a pair agree after a step)
            auto better = [&](float ob, uint32_t oi) {
                if (oi != kNone && (bi == kNone || ob > best || (ob == best && oi < bi))) {
                    best = ob;
                    bi = oi;
                }
            };
            { const float ob = row16_peer<0>(best); const uint32_t oi = row16_peer<0>(bi); better(ob, oi); }
            { const float ob = row16_peer<1>(best); const uint32_t oi = row16_peer<1>(bi); better(ob, oi); }
            { const float ob = row16_peer<2>(best); const uint32_t oi = row16_peer<2>(bi); better(ob, oi); }
            { const float ob = row16_peer<3>(best); const uint32_t oi = row16_peer<3>(bi); better(ob, oi); }
            // every lane of the token knows the winner and its logit (some expert is left: k <= E)
            const float pv = prob(best);
            den += pv;   // mCw, accumulated in selection order (gate.cuh:669)
#pragma unroll
            for (int j = 0; j < NL; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (uint32_t(64 * j + 4 * sub + v) == bi) w[j][v] = kNegInf;
            if (sub == 0) {
                store_through(p.topk_expert + size_t(token) * k + r, int32_t(bi));
                store_through(p.topk_prob + size_t(token) * k + r, pv);
                s_sel[tl * k + r] = bi;
            }
        }
        if (sub == 0) store_through(p.combine_den + token, den);
    }
    __syncthreads();
    // in-tile ranks (gate.cuh:678-696): pick r of token t ranks behind the picks of the same expert
    // by the tokens before t (a token's own picks are distinct experts). One pick per thread, the
    // earlier picks read four at a time (every lane reads the same words: broadcasts); the reads
    // may run up to three words past the picks of the earlier tokens, which stays inside the
    // group's LDS and is masked out.
    if (valid) {
        for (uint32_t i = gtid; i < kGateTileTokens * k; i += kGroupThreads) {
            const uint32_t e = s_sel[i];
            const uint32_t before = (i / k) * k;
            uint32_t rank = 0;
            if (e < E) {
                for (uint32_t j = 0; j < before; j += 4) {
                    const uint32_t a = s_sel[j], b = s_sel[j + 1], c = s_sel[j + 2], d = s_sel[j + 3];
                    rank += uint32_t(a == e) + uint32_t(b == e && j + 1 < before) + uint32_t(c == e && j + 2 < before) +
                            uint32_t(d == e && j + 3 < before);
                }
                atomicAdd(s_hist + e, 1u);
            }
            store_through(p.topk_slot + size_t(tile) * kGateTileTokens * k + i, int32_t(rank));
        }
    }
    __syncthreads();
    if (valid) {
        uint32_t* super = p.super_count + size_t(p.epoch & 1u) * p.n_super * E + size_t(tile / kSuperTiles) * E;
        for (uint32_t e = gtid; e < E; e += kGroupThreads) {
            const uint32_t cnt = s_hist[e];
            store_through(p.tile_count + size_t(tile) * E + e, cnt);
            if (cnt) atomic_add_agent(super + e, cnt);
            if (p.is_training) {
                // column sums of the tile's probabilities for the load-balancing loss (gate.cuh:608-635)
                float col_sum = 0.f;
                for (uint32_t t = 0; t < kGateTileTokens; ++t) col_sum += s_prob[t * E + e];
                store_through(p.tile_prob + size_t(tile) * E + e, col_sum);
            }
        }
    }
    __syncthreads();   // the next tile clears the histogram
}

// Slot assignment for one 16-token tile, by a group of `gsize` threads (whole wavefronts). Every thread of the workgroup must call
// it (it contains workgroup barriers); a group without work passes valid = false. `part` is LDS scratch of
// slot_tile_words(E, gsize) words private to the group. Must run after every gate tile has finished
// and released its results; what the gate tiles wrote is read with device-coherent loads.
//   slot = (tokens routed to e in all earlier tiles) + (rank inside this tile); a token keeps its
//   expert iff slot < EC (gate.cuh:710-716).
// What bounds it: trips to memory that other XCDs wrote, well over a microsecond each. The rows of counts before a tile (31 of its
// block and the coarse ones) are shared out over the threads that a workgroup of 512 has per expert (SHARED: four up to 128 experts, two up to 256), so that they are one trip or two; by a single wavefront, 64
// experts after the other, they were eight with 256 experts. Up to 64 experts a single wavefront's two trips are the shorter way (the
// shares cost a sum per pair and more code, all of it executed once: 8 192 tokens, 64 experts: 8.3 us for the phase, 8.9 shared out).
// The phase with its barrier, with 256 experts: 128 tokens top-8 29 -> 8 us, 4 096 38 -> 12. Us per forward: 2 048 tokens, 128 experts
// top-3, 448 x 448: 72 -> 61; 1 280, 256 experts top-2, 2 304 x 576: 311 -> 284; 384, 128 experts top-2, 4 544 x 704: 331 -> 318.
__host__ __device__ inline uint32_t slot_tile_words(uint32_t E, uint32_t gsize) { return E > gsize ? E : gsize; }
template <bool SHARED>
__device__ __forceinline__ void slot_tile(const LayerParams& p, uint32_t tile, bool valid, uint32_t* part, uint32_t gtid, uint32_t gsize) {
    const uint32_t E = p.E;
    const uint32_t* super = p.super_count + size_t(p.epoch & 1u) * p.n_super * E;
    // The tile's (token, expert) pairs are requested first: they do not depend on the counts.
    const uint32_t pairs = kGateTileTokens * p.k;
    constexpr uint32_t kInline = 4;            // pairs per thread kept in registers
    uint32_t pe[kInline];
    int32_t pr[kInline];
#pragma unroll
    for (uint32_t u = 0; u < kInline; ++u) {
        const uint32_t i = gtid + u * gsize;
        pe[u] = 0; pr[u] = 0;
        if (valid && i < pairs) {
            pe[u] = uint32_t(load_coherent(p.topk_expert + size_t(tile) * pairs + i));
            pr[u] = load_coherent(p.topk_slot + size_t(tile) * pairs + i);
        }
    }
    // expert e's rows of counts: thread e of every run of 2^lg threads, run g taking the rows g, g + runs, ...
    const uint32_t lg = SHARED && E > 1 ? 32u - uint32_t(__builtin_clz(E - 1)) : 0u;
    const uint32_t most = SHARED ? gsize >> lg : 1u, runs = most ? most : 1u, g = runs > 1 ? gtid >> lg : 0u;
    if (valid) {
        const uint32_t sup = tile / kSuperTiles;
        const uint32_t first = sup * kSuperTiles;
        // The coarse rows before this tile's block and the tile rows inside it form one list of
        // n rows, summed per expert in batches of 16 loads that are in flight together (the row
        // index is clamped instead of branching, so the loads of a batch issue back to back).
        const uint32_t n = sup + (tile - first);
        auto row_ptr = [&](uint32_t r) {
            return r < sup ? super + size_t(r) * E : p.tile_count + size_t(first + (r - sup)) * E;
        };
        for (uint32_t e = runs > 1 ? gtid & ((1u << lg) - 1u) : gtid; e < E && g < runs; e += runs > 1 ? E : gsize) {
            uint32_t acc = 0;
            constexpr uint32_t kBatch = 16;
            for (uint32_t r0 = g; r0 < n; r0 += kBatch * runs) {
                uint32_t v[kBatch];
#pragma unroll
                for (uint32_t u = 0; u < kBatch; ++u) {
                    const uint32_t r = r0 + u * runs;
                    v[u] = load_coherent(row_ptr(r < n ? r : n - 1) + e);
                }
#pragma unroll
                for (uint32_t u = 0; u < kBatch; ++u) acc += r0 + u * runs < n ? v[u] : 0u;
            }
            part[g * E + e] = acc;
            // training: the group of a block's first tile also sums the block's probability rows
            if (p.is_training && tile == first && g == 0) {
                const uint32_t rows = p.n_gate_tiles - first < uint32_t(kSuperTiles) ? p.n_gate_tiles - first
                                                                                      : uint32_t(kSuperTiles);
                float total = 0.f;
                for (uint32_t r0 = 0; r0 < rows; r0 += 16) {
                    float v[16];
#pragma unroll
                    for (uint32_t u = 0; u < 16; ++u)
                        v[u] = load_coherent(p.tile_prob + size_t(first + (r0 + u < rows ? r0 + u : rows - 1)) * E + e);
#pragma unroll
                    for (uint32_t u = 0; u < 16; ++u) total += r0 + u < rows ? v[u] : 0.f;
                }
                store_through(p.super_prob + size_t(sup) * E + e, total);
            }
        }
    }
    __syncthreads();
    if (valid) {
        auto assign = [&](uint32_t i, uint32_t e, int32_t rank) {
            const size_t idx = size_t(tile) * pairs + i;
            const uint32_t token = tile * kGateTileTokens + i / p.k;
            const bool real = e < E;   // (always: the rounds of the gate pick experts; anything else would have no place)
            e = real ? e : 0u;
            uint32_t slot = uint32_t(rank);
            for (uint32_t r = 0; r < runs; ++r) slot += part[r * E + e];
            const bool keep = real && slot < p.EC && slot < p.cap_rows;
            store_through(p.topk_slot + idx, keep ? int32_t(slot) : -1);
            if (keep) store_through(p.slot_token + size_t(e) * p.cap_rows + slot, int32_t(token));
        };
#pragma unroll
        for (uint32_t u = 0; u < kInline; ++u)
            if (gtid + u * gsize < pairs) assign(gtid + u * gsize, pe[u], pr[u]);
        for (uint32_t i = gtid + kInline * gsize; i < pairs; i += gsize)
            assign(i, uint32_t(load_coherent(p.topk_expert + size_t(tile) * pairs + i)),
                   load_coherent(p.topk_slot + size_t(tile) * pairs + i));
    }
    __syncthreads();
}

// Training mode, one wavefront, after the slot phase has been released: mean probability and mean
// routed count per expert and their scaled dot product (gate.cuh:763-773). Every sum has a fixed
// order, so the loss does not depend on timing.
__device__ __forceinline__ void gate_loss_finalize(const LayerParams& p) {
    const uint32_t lane = threadIdx.x & 63, E = p.E;
    const float inv_s = 1.0f / float(p.S);
    float dot = 0.f;
    for (uint32_t e0 = 0; e0 < E; e0 += kWave) {
        const uint32_t e = e0 + lane;
        float prod = 0.f;
        if (e < E) {
            float total = 0.f;
            for (uint32_t r0 = 0; r0 < p.n_super; r0 += 16) {
                float v[16];
#pragma unroll
                for (uint32_t u = 0; u < 16; ++u)
                    v[u] = load_coherent(p.super_prob + size_t(r0 + u < p.n_super ? r0 + u : p.n_super - 1) * E + e);
#pragma unroll
                for (uint32_t u = 0; u < 16; ++u) total += r0 + u < p.n_super ? v[u] : 0.f;
            }
            const float mean_prob = total * inv_s;
            const float mean_count = float(load_coherent(p.expert_count + e)) * inv_s;
            p.gate_loss[e] = mean_prob;
            p.gate_loss[E + e] = mean_count;
            prod = mean_prob * mean_count;
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) prod += __shfl_xor(prod, off);
        dot += prod;
    }
    if (lane == 0) p.gate_loss[2 * E] = dot / float(E);
}

}  // namespace kleos_amd
