// Expert projections of the tf32 Element on the 16-bit matrix cores: GemmHalf, one fp16 product per pair of operands, and
// GemmSplit, four bf16 products, for the tiles whose operands do not fit fp16.
//
// A tf32 operand has 11 significant bits. Its upper 8 are a bf16 value (the upper half of the word) and
// the remainder, at most 3 bits, is exactly one too: v = hi + lo. A product of two operands is then the sum
// of four bf16 products, each exact in fp32 as the tf32 product itself is, and all four are added: nothing
// is dropped, the sums are fp32 sums of exact products as on the fp32 matrix instructions. The bf16
// instructions have sixteen times the fp32 rate, so four products per pair of operands leave a factor of four.
// Two kinds of operands do not split: an infinity, whose product with a remainder of zero is NaN, and a value below
// 2^-123, whose remainder has bits below the last of a bf16 subnormal (2^-133). A wavefront that finds a NaN among its
// sums, or sums so small that such lost bits could show in them, computes its part of the tile again on the fp32
// matrix instructions. (Noticing the lost bits takes 17 of a slice's 364 vector instructions: 953 -> 959 us at the
// layer below, the mean of two runs, when every tile was GemmSplit's.)
#pragma once
#include "expert_gemm.hpp"

namespace kleos_amd {

// Where a tile's results go.
struct TileOut32 {
    float* c_base;
    uint32_t ldc, m_valid, n_valid;
};

// ------------------------------------------------------------------------------------------------
// BM x BN tile, WAVES_M x WAVES_N wavefronts, K in slices of 32 values (128-byte rows) through two LDS
// stages that direct loads fill with the 32-bit Elements as they are in memory, with the swizzle of
// Gemm16. Before a slice is multiplied, every wavefront splits the rows that its own loads brought, in
// place: sixteen consecutive values of a row (64 bytes) become [16 hi | 16 lo] in bf16. A fragment of one
// 16x16x32 instruction - 16 bytes of a row per lane - is then [hi | lo] of sixteen values of K. With the
// weight fragment's halves doubled inside the registers ([hi | hi] and [lo | lo]: half a wavefront swapped
// with the other half), two instructions against one activation fragment [hi | lo] give the four products.
//
// Why the split happens in LDS: split on the way out of LDS, a weight would be split by WAVES_M
// wavefronts and an activation by WAVES_N of them (3 500 clocks of vector instructions for the 4 096 clocks of
// matrix instructions of a slice); split on the way in, through registers, the 64 KB of a slice would hold
// 32 registers of every lane while they are in flight, beside 128 accumulators. In place it costs a slice
// 1 500 clocks of vector instructions in the shadow of the matrix ones, and LDS traffic of 128 KB beside the 192 KB
// of fragment reads.
//
// The pipeline of a slice kt, per wavefront (128 matrix instructions in sixteen groups of eight, the groups
// walking the activation fragments):
//   top       the workgroup meets: slice kt is split in LDS, everybody has left slice kt-1
//   group 0.. the activation rows of slice kt+1 are requested, into the stage of slice kt-1
//   group 8   every wavefront holds its last weight fragments of slice kt: behind a barrier the weight rows of
//             slice kt+2 are requested, a slice and a half before they are split (they come from memory; the
//             activation rows, shared by the column tiles of an expert, from the L2)
//   group 8.. slice kt+1 is split, the weight rows first
//
// Measured with all tiles on it (8 192 tokens, 64 experts top-2, 2 048 x 2 048): 2 729 us per forward with the 64 x 64 tiles on the
// fp32 matrix cores, 975 with these; the expert phase took 870 us, 1 240 TFLOP/s of bf16 products, the rate the
// bf16 tiles reach at the compute-bound shapes. Same distance from the layer computed in 64 bits (4.6e-4, the
// rounding of the rows to tf32). It runs now where GemmHalf's tile does not fit fp16, behind that product.
// ------------------------------------------------------------------------------------------------
template <int BM, int BN, int WAVES_M, int WAVES_N>
struct GemmSplit {
    static constexpr int kWaves = WAVES_M * WAVES_N;
    static constexpr int kThreads = kWaves * kWave;
    static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
    static constexpr int TM = WM / 16, TN = WN / 16;
    static constexpr int kSliceK = 32, kSteps = 2;                 // a K step: 16 values, one fragment
    static constexpr int kRowBytes = kSliceK * 4, kRowsPerLoad = 8, kChunks = 8;
    static constexpr int kABytes = BM * kRowBytes, kBBytes = BN * kRowBytes, kStage = kABytes + kBBytes;
    static constexpr int kBiasBytes = BN * 4, kBiasOffset = 2 * kStage;
    static constexpr int kLostOffset = kBiasOffset + 2 * kBiasBytes;   // a word per bias slot: whether an operand of the tile lost bits
    static constexpr int kSmemBytes = kLostOffset + 16;
    static constexpr int LA = BM / (kRowsPerLoad * kWaves), LB = BN / (kRowsPerLoad * kWaves);
    static_assert(TM == 8 && TN == 4 && LA == 4 && LB == 4, "the groups below are counted for these");
    static_assert(kWaves * 4096 <= kStage && kBiasBytes <= 1024);

    struct Tile {
        const float* pa[LA];
        const float* pb[LB];
        const float* a_base;                     // the rows as `recompute` finds them
        const int32_t* a_row_index;
        const float* b_base;
        uint32_t a_rows, lda, ldb;
        float* c_base;
        uint32_t ldc, m_valid, n_valid, k_tiles, act, k_first;
        int stage0, bias_slot;
    };
    typedef f32x4 Acc[TN][TM];

    static __device__ __forceinline__ int swizzle(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }
    static __device__ __forceinline__ int stage_of(const Tile& t, uint32_t kt) { return (t.stage0 + kt) & 1; }
    static __device__ __forceinline__ int last_stage(const Tile& t) { return stage_of(t, t.k_tiles - 1); }
    static __device__ __forceinline__ int next_stage0(const Tile& t) { return stage_of(t, t.k_tiles); }

    static __device__ __forceinline__ uint32_t first_value(const Tile& t, uint32_t kt) {
        const uint32_t slice = kt + t.k_first;
        return (slice >= t.k_tiles ? slice - t.k_tiles : slice) * kSliceK;
    }
    static __device__ __forceinline__ void load_a(const Tile& t, uint32_t stage_lds, uint32_t k0, int i) {
        direct_load16<false>(t.pa[i] + k0, stage_lds + 1024 * kWaves * i);
    }
    static __device__ __forceinline__ void load_b(const Tile& t, uint32_t stage_lds, uint32_t k0, int i) {
        direct_load16<true>(t.pb[i] + k0, stage_lds + kABytes + 1024 * kWaves * i);
    }
    static __device__ __forceinline__ uint32_t stage_lds(const Tile& t, char* smem, uint32_t kt) {
        return lds_address(smem) + stage_of(t, kt) * kStage + 1024 * wave_index();
    }

    // As Gemm16::begin; requests slice 0, weight rows first.
    static __device__ __forceinline__ void begin(Tile& t, const GemmTileArgs<float>& g, int stage0, int bias_slot, char* smem) {
        const uint32_t tid = local_tid();
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const int ld_r = lane / kChunks, ld_p = lane % kChunks;
        if (wave == 0 && lane < kBiasBytes / 16) {
            const uint32_t n = uint32_t(lane) * 4 < g.n_valid ? uint32_t(lane) * 4 : 0u;
            direct_load16<false>(g.bias + n, lds_address(smem) + kBiasOffset + bias_slot * kBiasBytes);
        }
        // (last read by the epilogue of the tile before the previous one, written again behind the main loop's barriers)
        if (tid == 0) *lost_word(smem, bias_slot) = 0u;
        t.a_base = g.a_base; t.a_row_index = g.a_row_index; t.a_rows = g.a_rows; t.lda = g.lda;
        t.b_base = g.b_base; t.ldb = g.ldb;
        t.c_base = g.c_base; t.ldc = g.ldc;
        t.m_valid = g.m_valid; t.n_valid = g.n_valid; t.k_tiles = g.K / kSliceK;
        // Known to be scalar, it takes the slices' offsets off the vector unit: 364 instead of 381 vector instructions a
        // slice, 32 registers spilled instead of 48. Against the tree that did not look for lost bits, in turn on one box,
        // 981 -> 997 us per forward at the layer above, all tiles GemmSplit's, without this, 949 -> 958 and 957 -> 959 with it.
        t.k_first = __builtin_amdgcn_readfirstlane(g.k_first < t.k_tiles ? g.k_first : 0u);
        t.act = g.act; t.stage0 = stage0; t.bias_slot = bias_slot;
        const uint32_t k0 = first_value(t, 0), dst = stage_lds(t, smem, 0);
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int row = kRowsPerLoad * (wave + kWaves * i) + ld_r;
            const uint32_t r = row < int(g.n_valid) ? row : g.n_valid - 1;
            t.pb[i] = g.b_base + size_t(r) * g.ldb + ((ld_p ^ swizzle(row)) << 2);
            load_b(t, dst, k0, i);
        }
        uint32_t src[LA];
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int row = kRowsPerLoad * (wave + kWaves * i) + ld_r;
            src[i] = row < int(g.m_valid) ? row : g.m_valid - 1;
        }
        if (g.a_row_index) {
#pragma unroll
            for (int i = 0; i < LA; ++i) src[i] = uint32_t(load_coherent(g.a_row_index + src[i]));
#pragma unroll
            for (int i = 0; i < LA; ++i) src[i] = src[i] < g.a_rows ? src[i] : g.a_rows - 1;
        }
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int row = kRowsPerLoad * (wave + kWaves * i) + ld_r;
            const float* from = g.a_base + size_t(src[i]) * g.lda;
            if (g.a_pad && row >= int(g.m_valid)) from = g.a_pad;
            t.pa[i] = from + ((ld_p ^ swizzle(row)) << 2);
            load_a(t, dst, k0, i);
        }
    }

    // ---- the split of the 1 KB (8 rows) that one direct load of this wavefront brought
    // `raw`: the lane's four values, as they landed at 16 * lane. `split_hi`: where their hi halves go inside
    // the 1 KB (their lo halves: two chunks further, i.e. at split_hi ^ 32).
    static __device__ __forceinline__ uint32_t split_offset() {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        const int r = lane >> 3, sw = swizzle(kRowsPerLoad * wave + r);   // (the loads of a wavefront are 8 * kRowsPerLoad rows apart: one swizzle)
        const int c = (lane & 7) ^ sw;                                    // values 4 c .. 4 c + 3 of the row
        const int hi_chunk = (c & 4) + ((c & 3) >> 1);
        return uint32_t(r * kRowBytes + ((hi_chunk ^ sw) << 4) + (c & 1) * 8);
    }
    // `lost`: what the remainders split by this thread had in their lower halves, which bf16 does not hold.
    static __device__ __forceinline__ uint32_t* lost_word(char* smem, int bias_slot) { return reinterpret_cast<uint32_t*>(smem + kLostOffset) + bias_slot; }
    static __device__ __forceinline__ void report_lost(const Tile& t, char* smem, uint32_t lost) {
        if (lost & 0xffffu) *lost_word(smem, t.bias_slot) = 1u;
    }
    static __device__ __forceinline__ void split_store(char* kilobyte, uint32_t split_hi, u32x4 raw, uint32_t& lost) {
        u32x2 hi, lo;
        uint32_t rest[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t word = raw[j];   // (a scalar: the compiler takes a bit cast of a vector's element to mean its first)
            const float v = __builtin_bit_cast(float, word & 0xffffe000u), h = __builtin_bit_cast(float, word & 0xffff0000u);
            rest[j] = __builtin_bit_cast(uint32_t, v - h);
        }
        lost |= rest[0] | rest[1] | rest[2] | rest[3];
        // the upper halves of two words, packed
        hi[0] = __builtin_amdgcn_perm(raw[1], raw[0], 0x07060302u);
        hi[1] = __builtin_amdgcn_perm(raw[3], raw[2], 0x07060302u);
        lo[0] = __builtin_amdgcn_perm(rest[1], rest[0], 0x07060302u);
        lo[1] = __builtin_amdgcn_perm(rest[3], rest[2], 0x07060302u);
        *reinterpret_cast<u32x2*>(kilobyte + split_hi) = hi;
        *reinterpret_cast<u32x2*>(kilobyte + (split_hi ^ 32u)) = lo;
    }
    // Kilobyte i of this wavefront's share of a stage: weight rows 0 .. LB-1, then activation rows.
    static __device__ __forceinline__ char* kilobyte(char* stage, int i) {
        return stage + 1024 * (threadIdx.x >> 6) + (i < LB ? kABytes + 1024 * kWaves * i : 1024 * kWaves * (i - LB));
    }

    static __device__ __forceinline__ bool rows_absent_of(uint32_t m_valid, int wm) { return uint32_t(wm * WM) >= m_valid; }
    static __device__ __forceinline__ bool rows_absent(const Tile& t, int wm) { return rows_absent_of(t.m_valid, wm); }

    template <typename Hook>
    static __device__ __forceinline__ void mainloop(const Tile& t, Acc& acc, char* smem, Hook&& after_first_barrier) {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        const int wm = wave / WAVES_N, wn = wave % WAVES_N;
        const uint32_t split_hi = split_offset();
        uint32_t lost = 0u;
        // every wavefront has left the previous tile's epilogue, staged where slice 1 goes
        asm volatile("s_barrier" ::: "memory");
        if (t.k_tiles > 1) {
            const uint32_t dst = stage_lds(t, smem, 1), k0 = first_value(t, 1);
#pragma unroll
            for (int i = 0; i < LB; ++i) load_b(t, dst, k0, i);
            wait_vmcnt<LB>();
        } else {
            wait_vmcnt<0>();
        }
        asm volatile("" ::: "memory");
        {
            char* st = smem + stage_of(t, 0) * kStage;
            u32x4 raw[LA + LB];
#pragma unroll
            for (int i = 0; i < LA + LB; ++i) raw[i] = load16(kilobyte(st, i) + 16 * lane);
#pragma unroll
            for (int i = 0; i < LA + LB; ++i) split_store(kilobyte(st, i), split_hi, raw[i], lost);
        }
        // The workgroup meets in front of a slice once this wavefront's split rows are in LDS.
        auto top = [&](uint32_t kt) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (kt == 0) after_first_barrier();
        };
        if (rows_absent(t, __builtin_amdgcn_readfirstlane(wave) / WAVES_N)) {
            // None of this wavefront's rows exist: it brings and splits its share of every slice between
            // the same barriers, and multiplies nothing.
            for (uint32_t kt = 0; kt < t.k_tiles; ++kt) {
                top(kt);
                const bool next = kt + 1 < t.k_tiles, next2 = kt + 2 < t.k_tiles;
                if (next) {
                    const uint32_t dst = stage_lds(t, smem, kt + 1), k0 = first_value(t, kt + 1);
#pragma unroll
                    for (int i = 0; i < LA; ++i) load_a(t, dst, k0, i);
                }
                if (next2) {
                    asm volatile("s_barrier" ::: "memory");
                    const uint32_t dst = stage_lds(t, smem, kt + 2), k0 = first_value(t, kt + 2);
#pragma unroll
                    for (int i = 0; i < LB; ++i) load_b(t, dst, k0, i);
                    wait_vmcnt<LB>();
                } else {
                    wait_vmcnt<0>();
                }
                asm volatile("" ::: "memory");
                if (next) {
                    char* st = smem + stage_of(t, kt + 1) * kStage;
#pragma unroll
                    for (int i = 0; i < LA + LB; ++i) split_store(kilobyte(st, i), split_hi, load16(kilobyte(st, i) + 16 * lane), lost);
                }
            }
            report_lost(t, smem, lost);
            return;
        }
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int mi = 0; mi < TM; ++mi) acc[ni][mi] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int fr_row = lane & 15, fr_part = lane >> 4;
        const int rx = wm * WM + fr_row, rw = wn * WN + fr_row;
        const int base_x = rx * kRowBytes + ((fr_part ^ swizzle(rx)) << 4);
        const int base_w = kABytes + rw * kRowBytes + ((fr_part ^ swizzle(rw)) << 4);

        constexpr int kRing = 4;       // activation fragments on their way or in use
        u32x4 fx[kRing], fw[TN];       // [hi | lo]; the weight fragments of the next K step
        bf16x8 wh[TN], wl[TN];         // [hi | hi] and [lo | lo] of the K step being multiplied
        auto read_x = [&](const char* st, int q) {   // q: group of the slice, 8 ks + mi
            fx[q % kRing] = load16(st + (base_x ^ ((q / TM) << 6)) + (q % TM) * 16 * kRowBytes);
        };
        auto read_w = [&](const char* st, int ks, int ni) { fw[ni] = load16(st + (base_w ^ (ks << 6)) + ni * 16 * kRowBytes); };
        auto double_w = [&]() {
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) {
                u32x4 h, l;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const auto both = __builtin_amdgcn_permlane32_swap(fw[ni][v], fw[ni][v], false, false);
                    h[v] = both[0];
                    l[v] = both[1];
                }
                wh[ni] = __builtin_bit_cast(bf16x8, h);
                wl[ni] = __builtin_bit_cast(bf16x8, l);
            }
        };
        auto slice = [&](uint32_t kt, auto next_tag, auto next2_tag) {
            constexpr bool NEXT = decltype(next_tag)::value, NEXT2 = decltype(next2_tag)::value;
            top(kt);
            const char* st = smem + stage_of(t, kt) * kStage;
            char* st1 = smem + stage_of(t, kt + 1) * kStage;
            const uint32_t dst1 = stage_lds(t, smem, kt + 1), k1 = first_value(t, kt + 1);
            const uint32_t dst2 = stage_lds(t, smem, kt), k2 = NEXT2 ? first_value(t, kt + 2) : 0u;
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) read_w(st, 0, ni);
#pragma unroll
            for (int q = 0; q < kRing - 1; ++q) read_x(st, q);
            u32x4 raw{};
#pragma unroll
            for (int q = 0; q < kSteps * TM; ++q) {
                const int ks = q / TM, o = q % TM;
                if (o == 0) double_w();
                __builtin_amdgcn_sched_barrier(0);
                const bf16x8 x = __builtin_bit_cast(bf16x8, fx[q % kRing]);
#pragma unroll
                for (int ni = 0; ni < TN; ++ni) {
                    acc[ni][o] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wh[ni], x, acc[ni][o], 0, 0, 0);
                    if (ni == 0) {
                        if (q + kRing - 1 < kSteps * TM) read_x(st, q + kRing - 1);
                        if (ks == 0 && o >= TM - TN) read_w(st, 1, o - (TM - TN));
                    }
                }
                if (NEXT && ks == 0 && o < LA) load_a(t, dst1, k1, o);
                if (NEXT2 && ks == 1 && o >= 1 && o <= LB) load_b(t, dst2, k2, o - 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int ni = 0; ni < TN; ++ni) acc[ni][o] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wl[ni], x, acc[ni][o], 0, 0, 0);
                if (NEXT && ks == 1) {
                    // kilobyte o of slice kt+1: its values asked for here, split a group later. In flight at o = 0: its
                    // weight rows, then its activation rows; from o = LB on: those, then the weight rows of slice kt+2.
                    if (o > 0) split_store(kilobyte(st1, o - 1), split_hi, raw, lost);
                    if (o == 0) wait_vmcnt<LA>();
                    if (o == LB) wait_vmcnt<NEXT2 ? LB : 0>();
                    asm volatile("" ::: "memory");
                    raw = load16(kilobyte(st1, o) + 16 * lane);
                }
                if (NEXT2 && ks == 1 && o == 0) asm volatile("s_barrier" ::: "memory");   // the weight rows of this stage are free
                __builtin_amdgcn_sched_barrier(0);
            }
            if (NEXT) split_store(kilobyte(st1, TM - 1), split_hi, raw, lost);
        };
        const uint32_t ahead = t.k_tiles >= 2 ? t.k_tiles - 2 : 0u;
        for (uint32_t kt = 0; kt < ahead; ++kt) slice(kt, std::true_type{}, std::true_type{});
        if (t.k_tiles >= 2) slice(t.k_tiles - 2, std::true_type{}, std::false_type{});
        slice(t.k_tiles - 1, std::false_type{}, std::false_type{});
        report_lost(t, smem, lost);
    }

    // Bias, activation, rounding to tf32, rows written through the L2 in whole lines: panels of 32 rows x 32
    // columns go through 4 KB of the wavefront's own of `stage`.
    static __device__ __forceinline__ void finish(const Tile& t, Acc& acc, char* smem) {
        float largest = 0.f;
        const bool lost = *lost_word(smem, t.bias_slot) != 0u;   // the same in every wavefront
        if (lost) largest = largest_operand(t, smem);
        if (rows_absent(t, __builtin_amdgcn_readfirstlane(int(local_tid() >> 6)) / WAVES_N)) return;
        bool nan = false;
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int mi = 0; mi < TM; ++mi)
#pragma unroll
                for (int j = 0; j < 4; ++j) nan |= acc[ni][mi][j] != acc[ni][mi][j];
        if (lost) nan |= small_sums(t, acc, largest);
        const TileOut32 out{t.c_base, t.ldc, t.m_valid, t.n_valid};
        const char* bias = smem + kBiasOffset + t.bias_slot * kBiasBytes;
        char* stage = smem + last_stage(t) * kStage;
        if (__builtin_amdgcn_ballot_w64(nan) != 0u) recompute(t, smem);
        else if (t.act == 0) finish_act<0>(out, acc, bias, stage);
        else if (t.act == 1) finish_act<1>(out, acc, bias, stage);
        else finish_act<2>(out, acc, bias, stage);
    }
    // The largest operand of the tile, from the rows in memory: every thread looks at what it loaded for the main loop, the
    // stage that the last slice is not in takes the results. Called by all wavefronts or none.
    static __device__ __forceinline__ float largest_operand(const Tile& t, char* smem) {
        float largest = 0.f;
#pragma unroll 1
        for (uint32_t k = 0; k < t.k_tiles * kSliceK; k += kSliceK) {
            // (four loads at a time: the sums of the tile occupy half of the registers)
            u32x4 v[4];
            auto look = [&] {
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t word = v[i][j] & 0x7fffffffu;
                        largest = __builtin_fmaxf(largest, __builtin_bit_cast(float, word));
                    }
                __builtin_amdgcn_sched_barrier(0);
            };
#pragma unroll
            for (int i = 0; i < LA; ++i) v[i] = load16(t.pa[i] + k);
            look();
#pragma unroll
            for (int i = 0; i < LB; ++i) v[i] = load16(t.pb[i] + k);
            look();
        }
        float* words = reinterpret_cast<float*>(smem + (last_stage(t) ^ 1) * kStage);
        words[threadIdx.x] = largest;
        __syncthreads();
#pragma unroll 1
        for (int i = 0; i < kThreads; ++i) largest = __builtin_fmaxf(largest, words[i]);
        __syncthreads();   // the next tile's first loads go to that stage
        return largest;
    }
    // Whether a sum of this lane is so small that bits lost in the split could show in it. A product loses less than 2^-133
    // times the largest operand, a sum K times that; what is below the 26th bit of a sum disappears in its fp32 rounding.
    static __device__ __forceinline__ bool small_sums(const Tile& t, const Acc& acc, float largest) {
        const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63;
        const float visible = largest * float(t.k_tiles * kSliceK) * 0x1p-107f;
        float least = __builtin_huge_valf();   // of the sums of rows that exist
#pragma unroll
        for (int mi = 0; mi < TM; ++mi) {
            float v = __builtin_huge_valf();
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) {
                asm("v_min3_f32 %0, %0, |%1|, |%2|" : "+v"(v) : "v"(acc[ni][mi][0]), "v"(acc[ni][mi][1]));
                asm("v_min3_f32 %0, %0, |%1|, |%2|" : "+v"(v) : "v"(acc[ni][mi][2]), "v"(acc[ni][mi][3]));
            }
            if (uint32_t((wave / WAVES_N) * WM + mi * 16 + (lane & 15)) < t.m_valid) least = __builtin_fminf(least, v);
        }
        return !(least > visible);
    }
    // This wavefront's part of the tile once more, on the fp32 matrix instructions from the rows in memory: what infinities,
    // NaN and the smallest operands give is what the 64 x 64 tiles give. Rows and columns past the last one repeat it
    // and are not written. A row block against all four column blocks, ten loads in flight: bound by their round trips,
    // about 0.6 ms per projection where it happens (one expert of 2 048 x 2 048, 8 192 tokens, an infinity in one token:
    // 592 -> 1 784 us per forward; 3 160 a column block at a time; 2 190 with the 64 x 64 tiles throughout).
    static __device__ __forceinline__ void recompute(const Tile& t, const char* smem) {
        const uint32_t tid = local_tid();
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const uint32_t m0 = uint32_t(wave / WAVES_N) * WM, n0 = uint32_t(wave % WAVES_N) * WN;
        const uint32_t fr_row = lane & 15, fr_part = lane >> 4, K = t.k_tiles * kSliceK;
        const char* bias = smem + kBiasOffset + t.bias_slot * kBiasBytes;
#pragma unroll 1
        for (uint32_t mi = 0; mi < uint32_t(TM); ++mi) {
            const uint32_t m = m0 + mi * 16 + fr_row;
            uint32_t row = m < t.m_valid ? m : t.m_valid - 1;
            if (t.a_row_index) {
                row = uint32_t(load_coherent(t.a_row_index + row));
                row = row < t.a_rows ? row : t.a_rows - 1;
            }
            const float* x = t.a_base + size_t(row) * t.lda + 4 * fr_part;
            const float* w[TN];
            f32x4 sum[TN];
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) {
                const uint32_t n = n0 + ni * 16 + fr_row;
                w[ni] = t.b_base + size_t(n < t.n_valid ? n : t.n_valid - 1) * t.ldb + 4 * fr_part;
                sum[ni] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll 1
            for (uint32_t k = 0; k < K; k += kSliceK) {
                u32x4 xv[2], wv[2][TN];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    xv[h] = load16(x + k + 16 * h);
#pragma unroll
                    for (int ni = 0; ni < TN; ++ni) wv[h][ni] = load16(w[ni] + k + 16 * h);
                }
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int ni = 0; ni < TN; ++ni) sum[ni] = mma16_step(wv[h][ni], xv[h], sum[ni], tf32_t{});
            }
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) {
                const uint32_t n = n0 + ni * 16 + 4 * fr_part;
                const f32x4 b4 = *reinterpret_cast<const f32x4*>(bias + n * 4);
                f32x4 v;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float s = sum[ni][j] + b4[j];
                    v[j] = tf32_round(t.act == 0 ? activate<0, tf32_t>(s) : (t.act == 1 ? activate<1, tf32_t>(s) : activate<2, tf32_t>(s)));
                }
                if (m < t.m_valid && n < t.n_valid) store16_through(t.c_base + size_t(m) * t.ldc + n, __builtin_bit_cast(u32x4, v));
            }
        }
    }
    template <int ACT>
    static __device__ __forceinline__ void finish_act(const TileOut32& t, Acc& acc, const char* bias_mem, char* stage) {
        const uint32_t tid = local_tid();
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const int wm = wave / WAVES_N, wn = wave % WAVES_N;
        const int fr_row = lane & 15, fr_part = lane >> 4;
        char* stg = stage + wave * 4096;
        const char* bias = bias_mem + (wn * WN + 4 * fr_part) * 4;
#pragma unroll
        for (int pm = 0; pm < TM / 2; ++pm)
#pragma unroll
            for (int pn = 0; pn < TN / 2; ++pn) {
#pragma unroll
                for (int ml = 0; ml < 2; ++ml)
#pragma unroll
                    for (int nl = 0; nl < 2; ++nl) {
                        const int ni = 2 * pn + nl, r = ml * 16 + fr_row;
                        const f32x4 b4 = *reinterpret_cast<const f32x4*>(bias + ni * 16 * 4);
                        f32x4 v;
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[j] = tf32_round(activate<ACT, tf32_t>(acc[ni][2 * pm + ml][j] + b4[j]));
                        *reinterpret_cast<f32x4*>(stg + r * 128 + (((4 * nl + fr_part) ^ ((r >> 1) & 7)) << 4)) = v;
                    }
#pragma unroll
                for (int it = 0; it < 4; ++it) {
                    const int id = it * kWave + lane, r = id >> 3, c = id & 7;
                    const u32x4 v = load16(stg + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
                    const uint32_t m = wm * WM + pm * 32 + r, n = wn * WN + pn * 32 + c * 4;
                    constexpr int kAgentScope = 16;   // sc1
                    if (m < t.m_valid && n < t.n_valid)
                        __builtin_amdgcn_raw_buffer_store_b128(v, coherent_rows(t.c_base), int((size_t(m) * t.ldc + n) * 4), 0, kAgentScope);
                }
            }
    }
};

// ------------------------------------------------------------------------------------------------
// The same tile with one fp16 product instead of four bf16 ones. An fp16 value holds the 11 significant bits of a tf32
// operand; what it lacks is range. Every row of the tile is therefore scaled by a power of two of its own, chosen from the
// row's values in the tile's first slice (of an activation row their largest goes to 2^9 .. 2^10, so that the row may hold values 64 times
// as large and keeps all bits of those down to 2^-24 of it, of a weight row, which is seldom sparse, to 2^12 .. 2^13, 8 times and 2^-27;
// a row of zeros there takes after the rows beside it), and the epilogue
// scales the sums back: scaling is exact, a truncating conversion to fp16 cuts a value to what the tf32 instructions read of
// it, a product of two such values is exact in fp32. A row that outgrows its scale gets a smaller one on the way, and its sums with
// it (`refit`). What does not fit is noticed, and the whole tile then computed by GemmSplit:
//   - an infinity, a row whose first slice goes beyond 2^40 or that outgrows it by more than 2^38;
//   - a value below 2^-14 once scaled, which may lose bits below 2^-24. One in some ten million of a random operand does. What
//     the values of a row lose at most is added up, and the tile is kept if for every single one of its sums this stays below 2^-24 of
//     the magnitudes of that sum's own products: less than adding them up in fp32 may lose anyway (`hidden`).
// (A NaN needs no care: it makes the same sums NaN.)
//
// K in slices of 32 values (128-byte rows). Four wavefronts bring the weight rows of a slice, four the activation rows, as
// direct loads into rings of LDS of their own: two slices for weights, which come from memory, one for activations, which the
// column tiles of an expert share in the L2 (vmcnt counts loads in order: a wavefront that brought both would wait for the weights
// in front of its activations). A wavefront converts what it brought, eight rows at a time, from its ring into the one
// slice that is multiplied; a ring slot is requested anew as soon as it has been read, without a barrier. The twelve
// fragments of a slice fit the registers beside the accumulators, so that the converted slice is free early. Per slice kt:
//   top       the workgroup meets: slice kt is converted
//   group 0   all fragments of slice kt are read; behind a second barrier the converted slice may change
//   group i   four matrix instructions of slice kt, between the request for eight rows of slice kt+1 and their conversion
//
// What bounds it: the weights, which have 64 KB a CU in flight (with all weight tiles read from one place, 477 us of 549), then the
// way of a slice through LDS and its conversion (454 us with the activations resident in L2 as well, 419 without the matrix instructions; LDS
// busy 26 % of the launch, bank conflicts 30 % of that, matrix cores 21 %). Measured, expert phase at 8 192 tokens, 64 experts top-2,
// 2 048 x 2 048: GemmSplit 890 us, this as first built, with sums spilled behind the main loop, 574, now 549 (970 -> 650 -> 607 us per
// forward). On the way: both operands in one ring of 12 kilobytes a wavefront, the kernel still spilling, 640; raw rows converted in place
// in two stages 737; loads to registers one slice ahead 761.
//
// What other values cost, us per forward of the same layer, GemmSplit throughout / when one row that outgrew its scale had the whole tile
// multiplied again / now: random ones 953 / 653 / 607; h with 70, 90, 95 and 99 % zeros 979 / 705 / 660, 934 / 1 022 / 654, 931 / 1 039 / 664,
// 916 / 1 025 / 807; x with a channel 200 times the others 825 / 931 / 590, with six of 100 to 1 000 times 815 / 925 / 671, with 90 %
// zeros 1 068 / 1 051 / 763, with rows between 2^-20 and 2^20 1 143 / 792 / 778; w_up with 90 % zeros 946 / 1 120 / 715. Behind GELU, whose
// small values are many, the channel gives 833 before and 792 now, the six 854 and 877. With weight rows at 2^9 like the others, so that one
// in twenty tiles holds a weight that loses bits instead of one in 160: 99 % zeros, where most products of a sum are zero and such a
// loss is not seen to be covered, 1 024, 90 % 717, random values 620, the channel behind GELU 853.
// ------------------------------------------------------------------------------------------------
template <int BM, int BN, int WAVES_M, int WAVES_N>
struct GemmHalf {
    static __device__ __forceinline__ uint32_t scalar(uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); }
    template <typename P>
    static __device__ __forceinline__ P* scalar(P* p) {
        const uint64_t a = reinterpret_cast<uint64_t>(p);
        return reinterpret_cast<P*>((uint64_t(scalar(uint32_t(a >> 32))) << 32) | scalar(uint32_t(a)));
    }
    // A tile's arguments in scalar registers: they live through the main loop.
    static __device__ __forceinline__ GemmTileArgs<float> scalar(const GemmTileArgs<float>& g) {
        GemmTileArgs<float> s;
        s.a_base = scalar(g.a_base); s.a_row_index = scalar(g.a_row_index); s.a_rows = scalar(g.a_rows); s.a_pad = scalar(g.a_pad);
        s.b_base = scalar(g.b_base); s.bias = scalar(g.bias); s.c_base = scalar(g.c_base);
        s.lda = scalar(g.lda); s.ldb = scalar(g.ldb); s.ldc = scalar(g.ldc); s.K = scalar(g.K); s.k_first = scalar(g.k_first);
        s.m_valid = scalar(g.m_valid); s.n_valid = scalar(g.n_valid); s.act = scalar(g.act);
        return s;
    }
    typedef GemmSplit<BM, BN, WAVES_M, WAVES_N> Split;
    static constexpr int kWaves = Split::kWaves, kThreads = Split::kThreads, kSliceK = Split::kSliceK;
    static constexpr int WM = Split::WM, WN = Split::WN, TM = Split::TM, TN = Split::TN, kRowsPerLoad = Split::kRowsPerLoad;
    static constexpr int kLoaders = kWaves / 2;                          // wavefronts that bring the rows of one operand
    static constexpr int L = BM / (kRowsPerLoad * kLoaders);             // kilobytes of a slice a wavefront brings
    static_assert(BM == BN && L == TM, "the groups below are counted for these");
    // LDS: the converted slice [BM rows | BN rows] of 64 bytes, then the rings that the loads land in: kRingX kilobytes for every wavefront
    // that brings activations, kRingW for the others
    static constexpr int kRowBytes = kSliceK * 2, kABytes = BM * kRowBytes, kConverted = (BM + BN) * kRowBytes;
    static constexpr int kRingX = L, kRingW = 2 * L;
    static constexpr int kRings = kLoaders * (kRingX + kRingW) * 1024;
    static constexpr int kExponents = Split::kSmemBytes;                 // powers of two that scale a sum back: int32 [BM rows | BN columns]
    static constexpr int kLargest = kExponents + (BM + BN) * 4;          // of every scaled row: its largest value (bits of a float)
    static constexpr int kLoss = kLargest + (BM + BN) * 4;               // what its values lose at most, in units of 2^-34 (hidden)
    static constexpr int kDrops = kLoss + (BM + BN) * 4;                 // by how much its scale has come down since the first slice (exponents)
    static constexpr int kRangeOffset = kDrops + (BM + BN) * 4;          // per bias slot: the Range words
    static constexpr int kRangeWords = 4 + 2 * kWaves;
    static constexpr int kSmemBytes = kRangeOffset + 2 * kRangeWords * 4;
    static_assert(kConverted + kRings <= 2 * Split::kStage && kWaves * 4096 <= kConverted);
    typedef typename Split::Acc Acc;
    struct Tile {
        GemmTileArgs<float> g;
        const float* rows[L];      // this lane's rows of the operand its wavefront brings, at its chunk of a slice
        uint32_t k_tiles;
        int bias_slot;
    };

    // words of a tile's range: what it holds that calls for a second look, whether a row has outgrown its scale in the slice converted last,
    // then for every wavefront in which slices (their number modulo 64, two words) the rows it brings have values that lose bits
    enum : uint32_t { kSeen = 0, kOutgrown = 1, kSlices = 4 };
    enum : uint32_t { kOutOfRange = 1, kLossy = 2, kInDoubt = 4 };
    static __device__ __forceinline__ uint32_t* range_words(char* smem, int bias_slot) {
        return reinterpret_cast<uint32_t*>(smem + kRangeOffset) + bias_slot * kRangeWords;
    }

    static __device__ __forceinline__ uint32_t* lossy_slices(char* smem, int bias_slot) { return range_words(smem, bias_slot) + kSlices + 2 * wave_index(); }

    static __device__ __forceinline__ int next_stage0(const Tile&) { return 0; }
    static __device__ __forceinline__ uint32_t first_value(const Tile& t, uint32_t kt) {
        const uint32_t slice = kt + t.g.k_first;
        return (slice >= t.k_tiles ? slice - t.k_tiles : slice) * kSliceK;
    }
    // Odd wavefronts bring weight rows, even ones activation rows.
    static __device__ __forceinline__ uint32_t brings_w() { return wave_index() & 1u; }
    static __device__ __forceinline__ uint32_t loader() { return wave_index() >> 1; }
    static __device__ __forceinline__ uint32_t ring_offset() { return kConverted + 1024 * (brings_w() ? kLoaders * kRingX + loader() * kRingW : loader() * kRingX); }
    // A direct load with the policy of the wavefront's operand (non-temporal for weights), and the wait for all but W or X of a
    // wavefront's loads. One statement each, so that the compiler sees no branch between the matrix instructions.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    static __device__ __forceinline__ void load(const float* src, uint32_t lds, uint32_t w) {
        asm volatile("s_mov_b32 m0, %0\n\ts_cmp_lg_u32 %2, 0\n\ts_cbranch_scc1 1f\n\tglobal_load_lds_dwordx4 %1, off\n\ts_branch 2f\n"
                     "1:\n\tglobal_load_lds_dwordx4 %1, off nt\n2:" ::"s"(lds), "v"(src), "s"(w) : "memory", "m0", "scc");
    }
#pragma clang diagnostic pop
    template <int X, int W>
    static __device__ __forceinline__ void wait(uint32_t w) {
        if constexpr (X == W) {
            wait_vmcnt<X>();
            asm volatile("" ::: "memory");
        } else {
            asm volatile("s_cmp_lg_u32 %0, 0\n\ts_cbranch_scc1 1f\n\ts_waitcnt vmcnt(%1)\n1:\n\ts_waitcnt vmcnt(%2)" ::"s"(w), "i"(X), "i"(W) : "memory", "scc");
            static_assert(W > X);
        }
    }
    // The word of a per-row array that belongs to the row whose values of kilobyte i lie in this lane.
    static __device__ __forceinline__ uint32_t* row_word(char* smem, int array, int i) {
        const uint32_t row = kRowsPerLoad * (loader() + kLoaders * i) + ((threadIdx.x & 63) >> 3);
        return reinterpret_cast<uint32_t*>(smem + array) + (brings_w() ? BM : 0) + row;
    }
    // This lane's rows of the operand that its wavefront brings, at its chunk of a slice.
    static __device__ __forceinline__ void locate(const GemmTileArgs<float>& g, const float* (&rows)[L]) {
        const uint32_t tid = local_tid();
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const int ld_r = lane >> 3, ld_c = lane & 7;
        const bool w = wave & 1;
        const int valid = w ? g.n_valid : g.m_valid;
        uint32_t src[L];
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int row = kRowsPerLoad * ((wave >> 1) + kLoaders * i) + ld_r;
            src[i] = row < valid ? row : valid - 1;
        }
        if (!w && g.a_row_index) {
#pragma unroll
            for (int i = 0; i < L; ++i) src[i] = uint32_t(load_coherent(g.a_row_index + src[i]));
#pragma unroll
            for (int i = 0; i < L; ++i) src[i] = src[i] < g.a_rows ? src[i] : g.a_rows - 1;
        }
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int row = kRowsPerLoad * ((wave >> 1) + kLoaders * i) + ld_r;
            const float* from = w ? g.b_base + size_t(src[i]) * g.ldb : g.a_base + size_t(src[i]) * g.lda;
            if (!w && g.a_pad && row >= valid) from = g.a_pad;
            rows[i] = from + 4 * ld_c;
        }
    }
    // As Gemm16::begin; requests as many slices as the wavefront's ring holds.
    static __device__ __forceinline__ void begin(Tile& t, const GemmTileArgs<float>& args, int, int bias_slot, char* smem) {
        const GemmTileArgs<float> g = scalar(args);
        const uint32_t tid = local_tid();
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        if (wave == 0 && lane < Split::kBiasBytes / 16) {
            const uint32_t n = uint32_t(lane) * 4 < g.n_valid ? uint32_t(lane) * 4 : 0u;
            direct_load16<false>(g.bias + n, lds_address(smem) + Split::kBiasOffset + bias_slot * Split::kBiasBytes);
        }
        // (last read by the epilogue of the tile before the previous one, written again behind the main loop's barriers)
        if (tid < uint32_t(kRangeWords)) range_words(smem, bias_slot)[tid] = 0u;
        t.g = g;
        t.k_tiles = g.K / kSliceK;
        t.g.k_first = g.k_first < t.k_tiles ? g.k_first : 0u;
        t.bias_slot = bias_slot;
        locate(g, t.rows);
        if ((lane & 7) == 0) {   // written by this wavefront alone, last read by the previous tile in front of a barrier
#pragma unroll
            for (int i = 0; i < L; ++i) *row_word(smem, kLargest, i) = *row_word(smem, kDrops, i) = 0u;
        }
        const uint32_t ring = lds_address(smem) + ring_offset();
#pragma unroll
        for (int i = 0; i < L; ++i) load(t.rows[i] + first_value(t, 0), ring + 1024 * i, brings_w());
        if (brings_w() && t.k_tiles > 1) {
#pragma unroll
            for (int i = 0; i < L; ++i) load(t.rows[i] + first_value(t, 1), ring + 1024 * (L + i), brings_w());
        }
    }

    // ---- the conversion of a kilobyte
    static __device__ __forceinline__ int swizzle(int r) { return (r >> 2) & 3; }
    // Where the lane's four values go inside the 512 bytes that a kilobyte becomes.
    static __device__ __forceinline__ uint32_t half_offset() {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        const int r = lane >> 3, c = lane & 7;      // (the kilobytes of a wavefront are kLoaders * kRowsPerLoad rows apart: one swizzle)
        return uint32_t(r * kRowBytes + (((c >> 1) ^ swizzle(kRowsPerLoad * (wave >> 1) + r)) << 4) + (c & 1) * 8);
    }
    static __device__ __forceinline__ uint32_t halves(float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b)); }
    // A scaled value loses bits if it is not zero, and below 2^-14, the least normal fp16 value: if 2 * bits - 1 is less than this.
    static constexpr uint32_t kSmall = (0x38800000u << 1) - 1u;
    // `largest`: of the scaled values that this thread has seen of the row. `least`: 2 * bits - 1 of those of the slice.
    static __device__ __forceinline__ void convert(char* to, u32x4 raw, float scale, float& largest, uint32_t& least) {
        float v[4];
        uint32_t u[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t word = raw[j];
            v[j] = __builtin_bit_cast(float, word) * scale;
            u[j] = (__builtin_bit_cast(uint32_t, v[j]) << 1) - 1u;
        }
        asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(largest) : "v"(v[0]), "v"(v[1]));
        asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(largest) : "v"(v[2]), "v"(v[3]));
        asm("v_min3_u32 %0, %0, %1, %2" : "+v"(least) : "v"(u[0]), "v"(u[1]));
        asm("v_min3_u32 %0, %0, %1, %2" : "+v"(least) : "v"(u[2]), "v"(u[3]));
        *reinterpret_cast<u32x2*>(to) = u32x2{halves(v[0], v[1]), halves(v[2], v[3])};
    }
    static constexpr float kTooLarge = 65536.f;   // (a value of 11 bits below it is one of fp16)
    // The largest of what the eight lanes of a row hold (bits of a magnitude).
    static __device__ __forceinline__ uint32_t row_max(uint32_t largest) {
        auto with = [&](uint32_t peer) { largest = peer > largest ? peer : largest; };
        with(row16_peer<0>(largest));
        with(row16_peer<1>(largest));
        with(row16_peer<2>(largest));   // (the three steps combine aligned groups of eight lanes)
        return largest;
    }
    static __device__ __forceinline__ int exponent(uint32_t magnitude) { return int(magnitude >> 23) - 127; }
    // Sums times 2^(row + column), as the array of exponents has them.
    static __device__ __forceinline__ void scale_sums(Acc& acc, const int* exponents) {
        const int wave = int(wave_index()), lane = threadIdx.x & 63, wm = wave / WAVES_N, wn = wave % WAVES_N;
        u32x4 col[TN];
#pragma unroll
        for (int ni = 0; ni < TN; ++ni) col[ni] = load16(exponents + BM + wn * WN + ni * 16 + 4 * (lane >> 4));
#pragma unroll
        for (int mi = 0; mi < TM; ++mi) {
            const int row = exponents[wm * WM + mi * 16 + (lane & 15)];
#pragma unroll
            for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t c = col[ni][j];
                    acc[ni][mi][j] = __builtin_amdgcn_ldexpf(acc[ni][mi][j], row + int(c));
                }
        }
    }

    template <typename Hook>
    static __device__ __forceinline__ void mainloop(const Tile& t, Acc& acc, char* smem, Hook&& after_first_barrier) {
        const int wave = int(wave_index()), lane = threadIdx.x & 63;
        const int wm = wave / WAVES_N, wn = wave % WAVES_N;
        float scale[L], largest[L];
#pragma unroll
        for (int i = 0; i < L; ++i) largest[i] = 0.f;
        const int target = brings_w() ? 12 : 9;   // the largest value of a row's first slice goes to 2^target
        uint64_t lossy = 0;   // slices (modulo 64) in which a value loses bits
        auto note_lossy = [&](uint32_t least, uint32_t s) { lossy |= uint64_t(scalar(uint32_t(__builtin_amdgcn_ballot_w64(least < kSmall) != 0u))) << (s & 63u); };
        uint32_t* const words = range_words(smem, t.bias_slot);
        const uint32_t w = brings_w(), ring = lds_address(smem) + ring_offset();
        const char* const ring_lane = smem + ring_offset() + 16 * lane;
        char* const to = smem + (w ? kABytes : 0) + 512 * loader() + half_offset();
        // Slice kt of the ring's slots: an activation slice takes the one place there is, a weight slice the place kt % 2.
        auto place = [&](uint32_t kt) { return (kt & w) * (L * 1024u); };
        // How far the loads have got when slice s is converted. Kilobyte i of it makes way for that of the slice one (activations) or two
        // (weights) later. kBoth: slice s+2 exists; kOne: s+1 does; kNone: s is the last.
        enum { kBoth, kOne, kNone };
        u32x4 raw[2];   // kilobyte i of the slice being converted, and the one behind it
        auto request = [&](auto stage_tag, auto i_tag, uint32_t s) {
            constexpr int S = decltype(stage_tag)::value, i = decltype(i_tag)::value;
            if constexpr (S == kBoth) wait<kRingX - 1, kRingW - 1>(w);
            else if constexpr (S == kOne) wait<kRingX - 1, (kRingW - 1 - i > kRingX - 1 ? kRingW - 1 - i : kRingX - 1)>(w);
            else wait<L - 1 - i, L - 1 - i>(w);
            raw[i & 1] = load16(ring_lane + place(s) + 1024 * i);
        };
        // The kilobyte's values are in registers: its slot takes the later one.
        auto reload = [&](auto stage_tag, auto i_tag, uint32_t s) {
            constexpr int S = decltype(stage_tag)::value, i = decltype(i_tag)::value;
            asm volatile("" : "+v"(raw[i & 1]));
            if constexpr (S == kBoth) load(t.rows[i] + first_value(t, s + 1 + w), ring + place(s) + 1024 * i, w);
            else if constexpr (S == kOne) { if (!w) load(t.rows[i] + first_value(t, s + 1), ring + 1024 * i, 0u); }
        };
        // Kilobytes 0 .. L-1 of slice s, the first of them requested: `between(i)` runs while number i + 1 is on its way.
        auto convert_slice = [&](auto stage_tag, uint32_t s, auto&& between) {
            uint32_t least = ~0u;
            static_for<L>([&](auto i_tag) {
                constexpr int i = decltype(i_tag)::value;
                reload(stage_tag, i_tag, s);
                if constexpr (i + 1 < L) request(stage_tag, std::integral_constant<int, (i + 1 < L ? i + 1 : 0)>{}, s);
                between(i);
                convert(to + 512 * kLoaders * i, raw[i & 1], scale[i], largest[i], least);
            });
            note_lossy(least, s);
            float most = largest[0];
#pragma unroll
            for (int i = 1; i < L; i += 2) asm("v_max3_f32 %0, %0, %1, %2" : "+v"(most) : "v"(largest[i]), "v"(largest[i + 1 < L ? i + 1 : i]));
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(most >= kTooLarge) != 0u, 0)) {
                if (!(scalar(words[kSeen]) & kOutOfRange)) words[kOutgrown] = 1u;
            }
        };
        // Slice s is converted, and a row has outgrown its scale in it: the row's largest value goes to 2^14 .. 2^15 (one that towers over
        // the others leaves them the more bits), the slice is converted once more, and kLoss says how the sums follow. Their last place lies at 2^-48 or above, and a row and a column
        // together come down by 2^76 at most: a sum stays a normal number and keeps its bits. Every wavefront calls it, and meets the others behind it.
        auto refit = [&](uint32_t s) {
            uint32_t least = ~0u, flags = 0u;
            static_for<L>([&](auto i_tag) {
                constexpr int i = decltype(i_tag)::value;
                const uint32_t most = row_max(__builtin_bit_cast(uint32_t, largest[i]));
                int down = __builtin_bit_cast(float, most) >= kTooLarge ? exponent(most) - 14 : 0;
                uint32_t* const drops = row_word(smem, kDrops, i);
                if (int(*drops) + down > 38) { flags |= kOutOfRange; down = 0; }   // (an infinity among them)
                if ((lane & 7) == 0) {
                    *drops += uint32_t(down);
                    *row_word(smem, kExponents, i) += uint32_t(down);
                    *row_word(smem, kLoss, i) = uint32_t(-down);
                }
                scale[i] = __builtin_amdgcn_ldexpf(scale[i], -down);
                largest[i] = __builtin_amdgcn_ldexpf(largest[i], -down);
                if (scale[i] < 1.f) flags |= kLossy;
                if (__builtin_amdgcn_ballot_w64(down != 0) != 0u) convert(to + 512 * kLoaders * i, load16(t.rows[i] + first_value(t, s)), scale[i], largest[i], least);
            });
            note_lossy(least, s);
            if (flags) atomicOr(words + kSeen, flags);
        };
        auto stages = [&](uint32_t s, auto&& f) {
            if (s + 2 < t.k_tiles) f(std::integral_constant<int, kBoth>{});
            else if (s + 1 < t.k_tiles) f(std::integral_constant<int, kOne>{});
            else f(std::integral_constant<int, kNone>{});
        };
        using First = std::integral_constant<int, 0>;
        meet();   // every wavefront has left the previous tile's epilogue, staged where the converted rows go; the tile's words are clear
        stages(0, [&](auto stage_tag) {
            u32x4 slice0[L];
            request(stage_tag, First{}, 0u);
            static_for<L>([&](auto i_tag) {
                constexpr int i = decltype(i_tag)::value;
                reload(stage_tag, i_tag, 0u);
                slice0[i] = raw[i & 1];
                if constexpr (i + 1 < L) request(stage_tag, std::integral_constant<int, (i + 1 < L ? i + 1 : 0)>{}, 0u);
            });
            uint32_t row[L], rows = 0u;   // the largest magnitude of the row, and of the wavefront's rows
#pragma unroll
            for (int i = 0; i < L; ++i) {
                row[i] = 0u;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t word = slice0[i][j] & 0x7fffffffu;
                    row[i] = word > row[i] ? word : row[i];
                }
                row[i] = row_max(row[i]);
                rows = row[i] > rows ? row[i] : rows;
            }
#pragma unroll
            for (int other = 8; other < kWave; other *= 2) {
                const uint32_t peer = __shfl_xor(rows, other);
                rows = peer > rows ? peer : rows;
            }
            // Zeros say nothing of what follows them: such a row may hold four times the largest value of the rows beside it, or is taken to be
            // of ordinary size. (Small values in front are left to refit: taken for a sparse row's, they cost rows that are small throughout
            // more, 772 -> 899 us where rows lie between 2^-20 and 2^20, than they save a layer with 90 % zeros, 717 -> 711.)
            const int guess = rows != 0u ? exponent(rows) - 13 + target : 0;
            uint32_t least = ~0u, flags = 0u;
            static_for<L>([&](auto i_tag) {
                constexpr int i = decltype(i_tag)::value;
                int e = row[i] != 0u ? exponent(row[i]) : guess;
                if (e > 40) { flags |= kOutOfRange; e = 40; }
                e = e < -40 ? -40 : e;
                scale[i] = __builtin_bit_cast(float, uint32_t(target - e + 127) << 23);
                if (e > target) flags |= kLossy;
                if ((lane & 7) == 0) *row_word(smem, kExponents, i) = uint32_t(e - target);
                convert(to + 512 * kLoaders * i, slice0[i], scale[i], largest[i], least);
            });
            note_lossy(least, 0u);
            if (flags) atomicOr(words + kSeen, flags);
        });
        auto top = [&](uint32_t kt) {
            meet();
            if (kt == 0) after_first_barrier();
        };
        auto report = [&] {
            uint32_t flags = 0u;
            if (lossy != 0u) {
                flags = kLossy;
                if (lane < 2) lossy_slices(smem, t.bias_slot)[lane] = uint32_t(lossy >> (32 * lane));
            }
#pragma unroll
            for (int i = 0; i < L; ++i) {
                if (largest[i] >= kTooLarge) flags |= kOutOfRange;
                atomicMax(row_word(smem, kLargest, i), __builtin_bit_cast(uint32_t, largest[i]));
            }
            if (flags) atomicOr(words + kSeen, flags);
        };
        if (Split::rows_absent_of(t.g.m_valid, wm)) {
            // None of this wavefront's rows exist: it brings and converts its share of every slice between
            // the same barriers, and multiplies nothing.
            for (uint32_t kt = 0; kt < t.k_tiles; ++kt) {
                top(kt);
                if (scalar(words[kOutgrown]) != 0u) {
                    refit(kt);
                    meet();
                }
                if (kt + 1 < t.k_tiles) {
                    asm volatile("s_barrier" ::: "memory");
                    stages(kt + 1, [&](auto stage_tag) {
                        request(stage_tag, First{}, kt + 1);
                        convert_slice(stage_tag, kt + 1, [](int) {});
                    });
                }
            }
            report();
            return;
        }
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int mi = 0; mi < TM; ++mi) acc[ni][mi] = f32x4{0.f, 0.f, 0.f, 0.f};
        // The lane's place in a fragment of 16 rows, the same for all, and the wavefront's first fragments: one vector register through the
        // main loop, and no more (a spilled one is loaded behind all that is on its way)
        const uint32_t from = lds_address(smem) + (lane & 15) * kRowBytes + (((lane >> 4) ^ swizzle(lane & 15)) << 4);
        auto slice = [&](uint32_t kt, auto next_tag, auto stage_tag) {
            constexpr bool NEXT = decltype(next_tag)::value;
            top(kt);
            f16x8 fw[TN], fx[TM];
            auto read = [&] {
                uint32_t x = uint32_t(wm * WM * kRowBytes), y = uint32_t(kABytes + wn * WN * kRowBytes);
                asm volatile("" : "+s"(x), "+s"(y));
                const auto from_x = (const __attribute__((address_space(3))) char*)uintptr_t(from + x), from_w = (const __attribute__((address_space(3))) char*)uintptr_t(from + y);
                auto load16 = [](const __attribute__((address_space(3))) char* at) { return *(const __attribute__((address_space(3))) u32x4*)at; };
#pragma unroll
                for (int ni = 0; ni < TN; ++ni) fw[ni] = __builtin_bit_cast(f16x8, load16(from_w + ni * 16 * kRowBytes));
#pragma unroll
                for (int mi = 0; mi < TM; ++mi) fx[mi] = __builtin_bit_cast(f16x8, load16(from_x + mi * 16 * kRowBytes));
            };
            const uint32_t larger = words[kOutgrown];   // (in front of the fragments, which are waited for anyway)
            read();
            __builtin_amdgcn_sched_barrier(0);
            if (__builtin_expect(scalar(larger) != 0u, 0)) {
                refit(kt);
                meet();
                if (threadIdx.x == 0) words[kOutgrown] = 0u;   // everybody has read it; set again behind the next barrier
                scale_sums(acc, reinterpret_cast<const int*>(smem + kLoss));
                read();
                __builtin_amdgcn_sched_barrier(0);
            }
            auto group = [&](int o) {
#pragma unroll
                for (int ni = 0; ni < TN; ++ni) acc[ni][o] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[ni], fx[o], acc[ni][o], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            if constexpr (NEXT) {
                // Behind a barrier in front of the first conversion every wavefront has its fragments of slice kt in registers.
                request(stage_tag, First{}, kt + 1);
                group(0);
                __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
                asm volatile("s_barrier" ::: "memory");
                convert_slice(stage_tag, kt + 1, [&](int i) { if (i + 1 < TM) group(i + 1); });
            } else {
#pragma unroll
                for (int o = 0; o < TM; ++o) group(o);
            }
        };
        using Both = std::integral_constant<int, kBoth>; using One = std::integral_constant<int, kOne>; using None = std::integral_constant<int, kNone>;
        const uint32_t both = t.k_tiles >= 3 ? t.k_tiles - 3 : 0u;
        for (uint32_t kt = 0; kt < both; ++kt) slice(kt, std::true_type{}, Both{});
        if (t.k_tiles >= 3) slice(t.k_tiles - 3, std::true_type{}, One{});
        if (t.k_tiles >= 2) slice(t.k_tiles - 2, std::true_type{}, None{});
        slice(t.k_tiles - 1, std::false_type{}, None{});
        report();
    }

    // Whether, in every sum of this wavefront, what small values lost (kLoss) stays below 2^-24 of the magnitudes of the products: whether
    // the products of some of the slices alone, converted one beside the other in LDS, are 2^24 of it.
    static __device__ __forceinline__ bool covered(const GemmTileArgs<float>& g, const char* smem, uint32_t samples) {
        const int wave = int(wave_index()), lane = threadIdx.x & 63, wm = wave / WAVES_N, wn = wave % WAVES_N, part = lane >> 4;
        if (Split::rows_absent_of(g.m_valid, wm)) return true;
        const int rx = wm * WM + (lane & 15), rw = wn * WN + (lane & 15);
        const char* const from_x = smem + rx * kRowBytes + ((part ^ swizzle(rx)) << 4);
        const char* const from_w = smem + kABytes + rw * kRowBytes + ((part ^ swizzle(rw)) << 4);
        auto magnitudes = [](const char* from) {
            u32x4 v = load16(from);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] &= 0x7fff7fffu;
            return __builtin_bit_cast(f16x8, v);
        };
        // Where the scale is below one, a value of less than 2^-149 once scaled is zero then, and nobody has seen it.
        const float unseen = float(g.K) * 0x1p-126f;
        // The largest value of a row, and 2^24 of what it lost. A row that is not there, or is all zeros, loses nothing.
        auto row = [&](uint32_t r, bool exists, float& most, float& lost) {
            const float a = __builtin_bit_cast(float, reinterpret_cast<const uint32_t*>(smem + kLargest)[r]);
            const float b = 0x1p-10f * float(reinterpret_cast<const uint32_t*>(smem + kLoss)[r]) + (reinterpret_cast<const int*>(smem + kExponents)[r] > 0 ? unseen : 0.f);
            most = exists ? a : 0.f;
            lost = most > 0.f ? b : 0.f;
        };
        float margin = 0.f;
#pragma unroll 1
        for (int ni = 0; ni < TN; ++ni) {
            float most_w[4], lost_w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t n = wn * WN + ni * 16 + 4 * part + j;
                row(BM + n, n < g.n_valid, most_w[j], lost_w[j]);
            }
#pragma unroll 2
            for (int mi = 0; mi < TM; ++mi) {
                const uint32_t m = wm * WM + mi * 16 + (lane & 15);
                float most_x, lost_x;
                row(m, m < g.m_valid, most_x, lost_x);
                f32x4 sum{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                for (uint32_t q = 0; q < samples; ++q)
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(magnitudes(from_w + q * kConverted + ni * 16 * kRowBytes), magnitudes(from_x + q * kConverted + mi * 16 * kRowBytes), sum, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) margin = __builtin_fminf(margin, sum[j] - (lost_x * most_w[j] + most_x * lost_w[j]));
            }
        }
        return margin >= 0.f;
    }
    // The workgroup meets, what it wrote to LDS is there. (Does not wait for what is on its way from memory: the next tile's ticket.)
    static __device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
    // Whether it holds for all wavefronts, each of which calls this; `verdict`: the bit that says it does not.
    static __device__ __forceinline__ bool all(bool holds, uint32_t* words, uint32_t verdict) {
        if (!holds) atomicOr(words + kSeen, verdict);
        meet();
        return !(scalar(words[kSeen]) & verdict);
    }
    static __device__ __forceinline__ uint64_t lossy_of(char* smem, int bias_slot) {
        const uint32_t* mask = lossy_slices(smem, bias_slot);
        return uint64_t(scalar(mask[1])) << 32 | scalar(mask[0]);
    }
    // Whether the losses are covered for sure, without another look at the operands: against the slice that is still in LDS, all values of
    // a row taken to be small in the slices where one that its wavefront brought was. Every wavefront calls it behind the main loop. In
    // loops, as `hidden`: both are rarely called, and take as long as their instructions take to fetch.
    static __device__ __forceinline__ bool hidden_for_sure(const GemmTileArgs<float>& g, int bias_slot, char* smem) {
        const uint32_t most = uint32_t(__builtin_popcountll(lossy_of(smem, bias_slot))) * ((g.K / kSliceK + 63u) / 64u) * kSliceK << 10;
#pragma unroll 1
        for (int i = 0; i < L; ++i) *row_word(smem, kLoss, i) = most;
        meet();
        return all(covered(g, smem, 1), range_words(smem, bias_slot), kInDoubt);
    }
    // What the small values lost, against four slices spread over K.
    static __device__ __forceinline__ bool hidden(const GemmTileArgs<float>& g, int bias_slot, char* smem) {
        const uint32_t k_tiles = g.K / kSliceK;
        const uint64_t lossy = lossy_of(smem, bias_slot);
        const float* rows[L];
        locate(g, rows);
        float scale[L];
#pragma unroll
        for (int i = 0; i < L; ++i) scale[i] = __builtin_amdgcn_ldexpf(1.f, -int(*row_word(smem, kExponents, i)));
        constexpr uint32_t kSamples = 4;
        static_assert(int(kSamples) * kConverted <= Split::kBiasOffset);
        const uint32_t samples = k_tiles < kSamples ? k_tiles : kSamples;
        char* const to = smem + (brings_w() ? kABytes : 0) + 512 * loader() + half_offset();
#pragma unroll 1
        for (uint32_t q = 0; q < samples; ++q) {
            u32x4 raw[L];
#pragma unroll
            for (int i = 0; i < L; ++i) raw[i] = load16(rows[i] + k_tiles * q / samples * kSliceK);
#pragma unroll
            for (int i = 0; i < L; ++i) {
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t word = raw[i][j];
                    v[j] = __builtin_bit_cast(float, word) * scale[i];
                }
                *reinterpret_cast<u32x2*>(to + q * kConverted + 512 * kLoaders * i) = u32x2{halves(v[0], v[1]), halves(v[2], v[3])};
            }
        }
        float lost[L];   // less than 2^-24 a value, and no more than itself
#pragma unroll
        for (int i = 0; i < L; ++i) lost[i] = 0.f;
        const uint32_t k_first = g.k_first < k_tiles ? g.k_first : 0u;
#pragma unroll 1
        for (uint32_t s = 0; s < k_tiles; ++s) {
            if (!((lossy >> (s & 63u)) & 1u)) continue;
            const uint32_t slice = s + k_first >= k_tiles ? s + k_first - k_tiles : s + k_first;
            u32x4 raw[L];
#pragma unroll
            for (int i = 0; i < L; ++i) raw[i] = load16(rows[i] + slice * kSliceK);
#pragma unroll
            for (int i = 0; i < L; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t word = raw[i][j];
                    const float v = __builtin_fabsf(__builtin_bit_cast(float, word) * scale[i]);
                    lost[i] += v < 0x1p-14f ? __builtin_fminf(v, 0x1p-24f) : 0.f;
                }
        }
#pragma unroll
        for (int i = 0; i < L; ++i) {   // the eight lanes of a row; rounded up, which covers the rounding of K additions as well
            lost[i] += row16_peer<0>(lost[i]);
            lost[i] += row16_peer<1>(lost[i]);
            lost[i] += row16_peer<2>(lost[i]);
            if ((threadIdx.x & 7) == 0) *row_word(smem, kLoss, i) = lost[i] > 0.f ? uint32_t(lost[i] * 0x1.04p34f) + 1u : 0u;
        }
        meet();
        return all(covered(g, smem, samples), range_words(smem, bias_slot), kOutOfRange);
    }

    // The end of a tile whose words call for a second look: its sums if they stand, the tile by GemmSplit if they do not. A function of its own:
    // its registers are not those of the main loop's tile. The caller lays the sums in memory for it, because the compiler has sums
    // that live across a call there from the main loop to the epilogue of every tile, called or not: 64 MB per round of
    // tiles, 785 us per forward of the layer above where this took 620.
    static __device__ __attribute__((noinline)) void settle(GemmTileArgs<float> args, uint32_t slot, uint32_t lds, const Acc* sums) {
        const GemmTileArgs<float> g = scalar(args);
        const int bias_slot = int(scalar(slot));
        char* smem = (char*)(__attribute__((address_space(3))) char*)uintptr_t(scalar(lds));
        if (!(scalar(range_words(smem, bias_slot)[kSeen]) & kOutOfRange) && hidden(g, bias_slot, smem)) {
            Acc acc;
#pragma unroll
            for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                for (int mi = 0; mi < TM; ++mi) acc[ni][mi] = (*sums)[ni][mi];
            write(g, acc, bias_slot, smem);
            return;
        }
        typename Split::Tile t;
        Acc acc;
        Split::begin(t, g, 0, bias_slot, smem);
        Split::mainloop(t, acc, smem, [] {});
        __syncthreads();
        Split::finish(t, acc, smem);
        __syncthreads();   // the next tile's loads land where the other wavefronts stage their rows
    }
    static __device__ __forceinline__ void finish(const Tile& t, Acc& acc, char* smem) {
        const uint32_t seen = scalar(range_words(smem, t.bias_slot)[kSeen]);   // the same in every wavefront
        if (__builtin_expect(seen != 0u && ((seen & kOutOfRange) || !hidden_for_sure(t.g, t.bias_slot, smem)), 0)) {
            Acc sums;
#pragma unroll
            for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                for (int mi = 0; mi < TM; ++mi) sums[ni][mi] = acc[ni][mi];
            settle(t.g, t.bias_slot, uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)smem)), &sums);
        } else {
            write(t.g, acc, t.bias_slot, smem);
        }
    }
    static __device__ __forceinline__ void write(const GemmTileArgs<float>& g, Acc& acc, int bias_slot, char* smem) {
        if (Split::rows_absent_of(g.m_valid, int(wave_index()) / WAVES_N)) return;
        scale_sums(acc, reinterpret_cast<const int*>(smem + kExponents));
        const TileOut32 out{g.c_base, g.ldc, g.m_valid, g.n_valid};
        const char* bias = smem + Split::kBiasOffset + bias_slot * Split::kBiasBytes;
        if (g.act == 0) Split::template finish_act<0>(out, acc, bias, smem);
        else if (g.act == 1) Split::template finish_act<1>(out, acc, bias, smem);
        else Split::template finish_act<2>(out, acc, bias, smem);
    }
};

}  // namespace kleos_amd
