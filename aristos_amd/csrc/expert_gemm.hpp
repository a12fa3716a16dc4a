// Expert projections: C[m, n] = act(sum_k A[m, k] * W[n, k] + bias[n]) on one output tile, with
// the rows of A optionally gathered through the slot->token table, so the dispatch of the
// reference (packet::dispatch row copy into a per-expert heap cell, csrc/include/kleos/os/
// packet.cuh:151-160) never materialises: the gather happens while the tile is staged into LDS.
//
// Replaces processor::fGET + BlockMM + FAA (csrc/include/kleos/os/processor/processor.cuh:358-489,
// gemm.cuh:22-107). Rounding points are the reference's: fp32 accumulate, fp32 bias add and
// activation, one round-to-nearest-even to Element on store (processor.cuh:475).
#pragma once
#include <type_traits>
#include "device_common.hpp"

namespace kleos_amd {

// ------------------------------------------------------------------------------------------------
// 16-bit Elements (bf16, fp16), matrix cores. WAVES_M x WAVES_N wavefronts over a BM x BN tile.
//
// K is walked in slices of BK through a ring of LDS stages that the wavefronts fill with direct
// global->LDS loads (global_load_lds_dwordx4: each lane names a 16-byte global source, the 64 lanes
// of the instruction land in 1 KB of consecutive LDS). They never occupy a vector register. Rows of
// A are gathered through the slot->token table by giving each lane its token's row address.
// Slice kt+STAGES-1 is requested during slice kt, into the stage slice kt-1 was read from, its loads
// placed one by one behind the matrix instructions of the slice's first quarters (a slice's matrix
// instructions run in four equal quarters: one K step each with 32x32x16, half a K step with 16x16x32).
// With two stages the loads can instead run two slices ahead (AHEAD2): slice kt+2 is requested
// into the stage of slice kt as soon as every wavefront has read its last fragments of slice kt (a
// second workgroup barrier per slice, inside the third quarter, whose matrix instructions
// the loads then follow one by one), so the memory pipeline holds requests across the wait for
// slice kt+1 instead of running empty at every slice boundary.
//
// LDS layout of a stage: rows of BK*2 bytes, 16-byte chunk c of row r stored at chunk position
// c ^ swizzle(r). The LDS of gfx950 has 64 banks of 4 bytes and serves a 16-byte access of 16 lanes
// per clock; the swizzle (128-byte rows: ((r>>1)&7) ^ ((r&1)<<2), 64-byte rows: (r>>2)&3) makes any
// 16 consecutive rows read at one chunk index cover all 64 banks. Because the LDS destination of a
// direct load is fixed by the lane number, the swizzle is applied on the global side: the lane
// that lands on position p of row r fetches chunk p ^ swizzle(r).
//
// The weight rows feed the matrix core's row operand and the activation rows its column operand,
// i.e. the core computes C^T: a lane then owns 4 consecutive output columns of one output row.
//
// The tile computation is split into the pieces a persistent workgroup overlaps across tiles:
//   begin()    per-lane source addresses + the loads of the bias and of the first STAGES-1 slices
//   mainloop() all K slices
//   finish()   bias, activation, rounding, transposition through LDS, coalesced stores
// A workgroup calls finish() of a tile, then begin() of its next one: the stores enter the memory
// pipeline ahead of the next tile's loads (measured: 2 % faster than the other order, in which the
// stores queue behind a slice of loads and hold the wavefronts that issue them), and the stage ring
// keeps turning across tiles (finish() stages its output in the stage of the last slice, which
// every wavefront has left; begin() follows behind a workgroup barrier of the caller).
// ------------------------------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void* lds_ptr;

// One direct global->LDS load: every lane names 16 bytes of global memory, and the 64 lanes' bytes
// land in the 1 KB of LDS at `dst` (the same address in all lanes; the instruction takes it from M0)
// in lane order. Written as inline assembly, not as the compiler's builtin, on purpose: the compiler
// cannot see the `s_waitcnt vmcnt` this file places by hand, so it takes every direct load it knows
// of for pending for ever, and in front of any later LDS read whose address it cannot tell apart
// from the loads' destinations it waits for all of them (`vmcnt(0)`) - which empties the pipeline of
// loads that run one or two K slices ahead. Whether it could tell them apart turned out to depend on
// the surrounding code (the same main loop lost 11 % inside one kernel and nothing inside another).
// The ordering these loads need is all explicit here: a wait for the wavefront's own loads, then a
// workgroup barrier, before anybody reads a stage; a barrier behind everybody's last read before a
// stage is written again. Loads the compiler does not know of only make its own waits stricter.
// (M0 is a register the compiler sets up itself right in front of each instruction that reads it
// and keeps nothing in; it warns about any statement that names it)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// `lds`: the LDS address of the 1 KB, a value the compiler holds in a scalar register (lds_address()
// plus offsets that are the same in all lanes).
template <bool NON_TEMPORAL>
__device__ __forceinline__ void direct_load16(const void* src, uint32_t lds) {
    // (one wait state between the write of M0 and the load that reads it)
    if constexpr (NON_TEMPORAL)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(lds), "v"(src) : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory", "m0");
}
// Brings the 128-byte line that every lane names into the L2. (4 bytes of each land in LDS, 256 bytes at `lds`, where nobody reads them.)
__device__ __forceinline__ void touch_lines(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(src) : "memory", "m0");
}
#pragma clang diagnostic pop
// The LDS address of a pointer into the workgroup's LDS, in a scalar register.
__device__ __forceinline__ uint32_t lds_address(const char* p) {
    return __builtin_amdgcn_readfirstlane(uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)p)));
}
// The wavefront's index within the workgroup, in a scalar register.
__device__ __forceinline__ uint32_t wave_index() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// A 16-bit Element seen only as storage: addresses are computed in units of it, values are
// interpreted by the Element type the tile is instantiated with.
typedef uint16_t elem16_t;

// What one output tile needs, in scalar form (identical in every lane). U: an Element as storage.
template <typename U>
struct GemmTileArgs {
    const U* a_base;               // A rows (gathered through a_row_index when it is not null)
    const int32_t* a_row_index;
    uint32_t a_rows;               // rows behind a_base: gathered indices are clamped below it
    const U* a_pad;                // K zeros that stand in for the rows past m_valid (null: they re-read the last valid row)
    const U* b_base;               // first of the tile's weight rows
    const U* bias;                 // first of the tile's bias entries
    U* c_base;                     // output element (row 0, column 0) of the tile
    uint32_t lda, ldb, ldc, K;
    uint32_t k_first;              // K slice the tile starts with (it wraps around); below K / BK
    uint32_t m_valid, n_valid;     // rows / columns of the tile that exist
    uint32_t act;                  // 0 relu, 1 erf-gelu, 2 identity
};

// Where a tile's results go.
struct TileOut {
    elem16_t* c_base;              // output element (row 0, column 0) of the tile
    uint32_t ldc, m_valid, n_valid, act;
};

// The lane's thread index as a value the optimiser cannot trace back to threadIdx: whatever a
// phase derives from it is computed when the phase starts and dies when it ends, instead of
// being shared with the main loop and kept (or spilled) across it.
__device__ __forceinline__ uint32_t local_tid() {
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// Epilogue of a WAVES_M x WAVES_N wavefront grid whose wavefronts each hold a WM x WN block of the
// C^T accumulators, in 16 x 16 matrix-core tiles: acc[ni][mi][v] is output column n = wn*WN + ni*16 + 4*(lane/16) + v
// of output row m = wm*WM + mi*16 + lane%16, i.e. a lane owns 4 consecutive columns per tile.
// Bias, activation and the rounding to Element happen in registers; the wavefront
// then transposes 32-row x 64-column panels through a private LDS region of 4 KB at
// stage_mem + wave * 4096 (rows of 128 bytes, 16-byte chunk c of row r at position
// c ^ ((r >> 1) & 7)) so that the global stores are 16 bytes per lane and cover whole 128-byte
// lines of the output rows. The bias comes from LDS (bias_mem: the tile's BN entries): the epilogue
// issues no global load, so nothing in it ever waits for the stores it has in flight.
constexpr int kEpiloguePanelRows = 32;
// The output rows are stored with the agent-scope (sc1) policy, which writes them through the L2
// instead of leaving dirty lines there: other workgroups read them later in the same launch, on
// any XCD, and nothing then has to write a whole L2 back before it may tell them so. It also pays
// by itself where a launch writes far more output than the L2 holds (256-expert top-8 shape: 3.03
// against 3.11 ms per forward); neutral on the other shapes measured.
// STREAM_OUT adds the non-temporal hint: the rows pass through the L2 without staying there. For
// layers of many small experts, whose intermediate and output rows are many times the L2 and are
// read long after they were written (256-expert top-8 shape: 2 865 against 2 950 us per forward with
// both outputs streamed, 2 913 with the intermediate rows alone, 2 953 with the output rows alone);
// where the rows are read back soon, from the L2 that took them, it costs (64-expert shape 293
// against 287 us, 16-expert shape 154 against 146 us).
// The matrix cores are idle meanwhile. What bounds it is vector work (an addition, the activation, half a conversion a value,
// 4 clocks an instruction, two wavefronts a SIMD) and trips to LDS, so the bias is read once and not in front of every panel
// (behind whose writes the compiler will not move it), and the four reads of a panel are in flight together: 1 900 clocks
// less of the 8 100 between the main loops of two 256 x 256 tiles, 2 000 of 11 300 where all CUs store at once. 2 304 tokens, 16 experts top-1,
// 4 096 x 4 096: 234 -> 231.5 us per forward; 8 192, 64 experts top-2, 2 048 x 2 048, skewed: 281.5 -> 279.
template <typename E, int WM, int WN, int WAVES_N, int ACT, bool STREAM_OUT>
__device__ __forceinline__ void epilogue16_act(const TileOut& t, f32x4 (&acc)[WN / 16][WM / 16], char* stage_mem,
                                               const char* bias_mem) {
    typedef typename Elem16<E>::vec4 vec4;
    constexpr int kPanelRows = kEpiloguePanelRows;
    const uint32_t tid = local_tid();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int fr_row = lane & 15, fr_part = lane >> 4;
    char* stg = stage_mem + wave * (kPanelRows * 128);
    const char* bias_lane = bias_mem + (wn * WN + 4 * fr_part) * 2;
    f32x4 bias[WN / 16];
#pragma unroll
    for (int ni = 0; ni < WN / 16; ++ni) {
        const vec4 b4 = *reinterpret_cast<const vec4*>(bias_lane + ni * 16 * 2);
#pragma unroll
        for (int j = 0; j < 4; ++j) bias[ni][j] = float(b4[j]);
    }
    const coherent_rows_t rows = coherent_rows(t.c_base);
#pragma unroll
    for (int pm = 0; pm < WM / 32; ++pm) {
        if (uint32_t(wm * WM + pm * 32) >= t.m_valid) break;   // (the same in all lanes)
#pragma unroll
        for (int pn = 0; pn < WN / 64; ++pn) {
#pragma unroll
            for (int ml = 0; ml < 2; ++ml) {
                const int r = ml * 16 + fr_row;   // row of the panel
#pragma unroll
                for (int nl = 0; nl < 4; ++nl) {
                    const int ni = pn * 4 + nl;
                    vec4 o;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        o[j] = static_cast<E>(activate<ACT, E>(acc[ni][pm * 2 + ml][j] + bias[ni][j]));
                    // columns nl*16 + 4*fr_part .. + 3 of the panel: chunk 2*nl + fr_part/2, half fr_part%2
                    *reinterpret_cast<vec4*>(stg + r * 128 + (((2 * nl + (fr_part >> 1)) ^ ((r >> 1) & 7)) << 4) + (fr_part & 1) * 8) = o;
                }
            }
            constexpr int kStores = kPanelRows * 8 / kWave;
            u32x4 v[kStores];
#pragma unroll
            for (int it = 0; it < kStores; ++it) {
                const int r = (it * kWave + lane) >> 3, c = lane & 7;
                v[it] = load16(stg + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
            }
#pragma unroll
            for (int it = 0; it < kStores; ++it) {
                const int r = (it * kWave + lane) >> 3, c = lane & 7;
                const uint32_t m = wm * WM + pm * 32 + r, n = wn * WN + pn * 64 + c * 8;
                constexpr int kAgentScope = STREAM_OUT ? 16 + 2 : 16;   // sc1 (+ nt)
                // (a tile's rows lie within 2 GiB of its first element: 256 rows of at most 2^22 bytes)
                if (m < t.m_valid && n < t.n_valid)
                    __builtin_amdgcn_raw_buffer_store_b128(v[it], rows, int((size_t(m) * t.ldc + n) * sizeof(E)), 0, kAgentScope);
            }
        }
    }
}
template <typename E, int WM, int WN, int WAVES_N, bool STREAM_OUT>
__device__ __forceinline__ void epilogue16(const TileOut& t, f32x4 (&acc)[WN / 16][WM / 16], char* stage_mem,
                                           const char* bias_mem) {
    if (t.act == 0) epilogue16_act<E, WM, WN, WAVES_N, 0, STREAM_OUT>(t, acc, stage_mem, bias_mem);
    else if (t.act == 1) epilogue16_act<E, WM, WN, WAVES_N, 1, STREAM_OUT>(t, acc, stage_mem, bias_mem);
    else epilogue16_act<E, WM, WN, WAVES_N, 2, STREAM_OUT>(t, acc, stage_mem, bias_mem);
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>), in this order.
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// STREAM_B: the weight rows are loaded with the non-temporal cache policy: read once (or by a
// neighbour at the same moment), they pass through the L2 without displacing the activation rows
// that are shared (7.0 against 6.4 TB/s on a read-only stream of this shape).
// AHEAD2 (two stages only): the loads run two slices ahead, at the price of a second workgroup
// barrier per slice. The fragments of a slice's second K step are read behind the matrix instructions of the
// first, so a wavefront has finished with the stage half a slice before it finishes the slice: the barrier that frees the stage
// sits kReleaseAt matrix instructions into the third quarter (the last reads have returned by then), and the loads of slice kt+2
// follow it, half of them in the third and half in the last quarter. Every load has between one and one and a half slices to land.
// MI: the matrix-core tile. 32: 32x32x16 instructions (16 values of K each, 16 accumulator registers), which the gate's product uses;
// 16: 16x16x32 instructions (32 values of K, 4 accumulator registers). The smaller tile reads and
// writes half as many accumulator registers per multiply-add and draws less power for the same work
// (instruction loops on random bf16 operands held in registers, whole device: 2.08 against 1.84
// PFLOP/s at the same 1.31 kW), which is what bounds these kernels.
// STREAM_OUT: the output rows are stored with the non-temporal hint (see the epilogue above).
// GROUPS: more than one when several groups of WAVES_M x WAVES_N wavefronts of a workgroup each run this on
// LDS of their own (GemmKSplit); the wavefront numbers below are then those within a group.
template <typename E, int BM, int BN, int WAVES_M, int WAVES_N, int BK, int STAGES, bool STREAM_B, bool AHEAD2, int MI = 16,
          bool STREAM_OUT = false, int GROUPS = 1>
struct Gemm16 {
    typedef E Element;
    static constexpr int kBM = BM, kBN = BN, kWavesN = WAVES_N, kStages = STAGES;
    static constexpr bool kAhead2 = AHEAD2;
    static constexpr int kMI = MI;
    // a wavefront's number within its group, and the same from a scalar register
    static __device__ __forceinline__ int group_wave(int wave) { return GROUPS == 1 ? wave : wave % (WAVES_M * WAVES_N); }
    static __device__ __forceinline__ uint32_t scalar_wave() { return GROUPS == 1 ? wave_index() : wave_index() % uint32_t(WAVES_M * WAVES_N); }
    typedef typename Elem16<E>::vec8 vec8;
    typedef typename Elem16<E>::vec4 vec4;
    static constexpr int kWaves = WAVES_M * WAVES_N;
    static constexpr int kThreads = kWaves * kWave;
    static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;     // wavefront tile
    static constexpr int TM = WM / MI, TN = WN / MI;               // matrix-core tiles per wavefront
    static constexpr int KI = MI == 32 ? 16 : 32;                  // values of K one matrix instruction consumes
    static constexpr int kRowBytes = BK * 2;
    static constexpr int kRowsPerLoad = 1024 / kRowBytes;          // rows one direct load covers
    static constexpr int kChunks = kRowBytes / 16;                 // 16-byte chunks per row
    static constexpr int kABytes = BM * kRowBytes, kBBytes = BN * kRowBytes;
    static constexpr int kStage = kABytes + kBBytes;
    static constexpr int kBiasBytes = BN * 2;                      // one tile's bias entries
    static constexpr int kBiasOffset = STAGES * kStage;            // two bias slots behind the stage ring
    static constexpr int kSmemBytes = STAGES * kStage + 2 * kBiasBytes;
    static constexpr int LA = BM / (kRowsPerLoad * kWaves), LB = BN / (kRowsPerLoad * kWaves);
    static constexpr int kLoadsPerSlice = LA + LB;                 // per wavefront
    static constexpr int kSliceK = BK;                             // values of K per slice
    static constexpr int kSteps = BK / KI;                         // K steps per slice
    // 16-row tiles, wavefront tiles of four of them in height: a wavefront leaves out the blocks of 16
    // rows that hold no rows of the tile (64-expert shape with skewed routing: the experts' 13 039 rows
    // take the matrix instructions of 13 424 rows that way, of 14 656 with whole wavefronts left out only)
    static constexpr bool kBlockSkip = MI == 16 && TM == 4;
    static constexpr int kReleaseAt = 4;                  // matrix instructions of the third quarter in front of the barrier that frees the stage
    static_assert(!AHEAD2 || (MI == 16 && kSteps == 2));
    static constexpr int kQuarters = 4;                            // a slice's matrix instructions in four equal runs
    static constexpr int kPerQuarter = TN * TM * kSteps / kQuarters;
    static constexpr int kPanelRows = kEpiloguePanelRows;          // epilogue staging: 32 rows x 64 columns per wavefront
    static_assert(BK == 32 || BK == 64);
    static_assert(MI == 32 || MI == 16);
    static_assert(kQuarters % kSteps == 0 && (TN * TM * kSteps) % kQuarters == 0);
    static_assert(!AHEAD2 || STAGES == 2);
    static_assert(STAGES >= 2 && STAGES <= 4);
    static_assert(WM % 32 == 0 && WN % 64 == 0);
    static_assert(BM % (kRowsPerLoad * kWaves) == 0 && BN % (kRowsPerLoad * kWaves) == 0);
    static_assert(kWaves * kPanelRows * 128 <= kStage, "epilogue staging must fit one stage");
    static_assert((STAGES - 1) * kLoadsPerSlice < 64);
    static_assert(kBiasBytes <= 1024, "one direct load brings the bias");

    static __device__ __forceinline__ int swizzle(int r) {
        if constexpr (BK == 64) return ((r >> 1) & 7) ^ ((r & 1) << 2);
        else return (r >> 2) & 3;
    }

    struct Tile {
        const elem16_t* pa[LA];
        const elem16_t* pb[LB];
        elem16_t* c_base;
        uint32_t ldc, m_valid, n_valid, k_tiles, act;
        uint32_t k_first;           // the kt-th slice the tile works on is slice (k_first + kt) % k_tiles of K
        int stage0;                 // stage of the tile's first slice; its kt-th slice uses (stage0 + kt) % STAGES
        int bias_slot;              // which of the two LDS bias slots holds this tile's bias
    };

    typedef std::conditional_t<MI == 32, f32x16, f32x4> AccTile;
    typedef AccTile Acc[TN][TM];

    static __device__ __forceinline__ int stage_of(const Tile& t, uint32_t kt) { return (t.stage0 + kt) % STAGES; }

    // the direct loads that bring K slice kt of the tile into its stage: activation rows first (they
    // come from L2 and return early), then the weight rows
    static __device__ __forceinline__ void issue_slice(const Tile& t, char* smem, uint32_t kt) {
        const uint32_t sa = lds_address(smem) + stage_of(t, kt) * kStage + 1024 * scalar_wave();   // this wavefront's first KB of the stage
        const uint32_t sb = sa + kABytes;
        uint32_t slice = kt + t.k_first;
        slice = slice >= t.k_tiles ? slice - t.k_tiles : slice;
        const uint32_t k0 = slice * BK;
#pragma unroll
        for (int i = 0; i < LA; ++i)
            direct_load16<false>(t.pa[i] + k0, sa + 1024 * kWaves * i);
#pragma unroll
        for (int i = 0; i < LB; ++i)
            direct_load16<STREAM_B>(t.pb[i] + k0, sb + 1024 * kWaves * i);
    }

    // Load number j (0 <= j < LA + LB) of a K slice: activation rows first (they come from L2 and return
    // early), then the weight rows.
    // (sa, sb: the LDS addresses of this wavefront's first KB of the stage's activation and weight rows)
    static __device__ __forceinline__ void issue_one(const Tile& t, uint32_t sa, uint32_t sb, uint32_t k0, int j) {
        if (j >= LA)
            direct_load16<STREAM_B>(t.pb[j - LA] + k0, sb + 1024 * kWaves * (j - LA));
        else
            direct_load16<false>(t.pa[j] + k0, sa + 1024 * kWaves * j);
    }
    // Loads first .. first + count - 1 of K slice kt.
    template <int FIRST, int COUNT>
    static __device__ __forceinline__ void issue_range(const Tile& t, char* smem, uint32_t kt) {
        const uint32_t sa = lds_address(smem) + stage_of(t, kt) * kStage + 1024 * scalar_wave();
        const uint32_t sb = sa + kABytes;
        uint32_t slice = kt + t.k_first;
        slice = slice >= t.k_tiles ? slice - t.k_tiles : slice;
        const uint32_t k0 = slice * BK;
#pragma unroll
        for (int j = 0; j < COUNT; ++j) issue_one(t, sa, sb, k0, FIRST + j);
    }

    // begin() in parts. The load of the bias, by the first wavefront:
    static __device__ __forceinline__ void load_bias(const GemmTileArgs<elem16_t>& g, int bias_slot, char* smem, uint32_t wave, uint32_t lane) {
        if (wave == 0 && lane < uint32_t(kBiasBytes / 16)) {
            const uint32_t n = lane * 8 < g.n_valid ? lane * 8 : 0u;
            direct_load16<false>(g.bias + n, lds_address(smem) + kBiasOffset + bias_slot * kBiasBytes);
        }
    }
    // Where the lane's 16 bytes of the tile's activation rows `row` come from. The slot->token table was written earlier in the
    // same launch, possibly on another XCD: device-coherent loads, all in flight together (an index is clamped
    // to the table it points into, so that no value it could ever hold turns into an address
    // outside the caller's buffer).
    static __device__ __forceinline__ void source_rows(const elem16_t* (&pa)[LA], const GemmTileArgs<elem16_t>& g, const uint32_t (&row)[LA], uint32_t ld_p) {
        uint32_t src[LA];
#pragma unroll
        for (int i = 0; i < LA; ++i) src[i] = row[i] < g.m_valid ? row[i] : g.m_valid - 1;
        if (g.a_row_index) {
#pragma unroll
            for (int i = 0; i < LA; ++i) src[i] = uint32_t(load_coherent(g.a_row_index + src[i]));
#pragma unroll
            for (int i = 0; i < LA; ++i) src[i] = src[i] < g.a_rows ? src[i] : g.a_rows - 1;
        }
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const elem16_t* from = g.a_base + size_t(src[i]) * g.lda;
            if (g.a_pad && row[i] >= g.m_valid) from = g.a_pad;
            pa[i] = from + ((ld_p ^ swizzle(row[i])) << 3);
        }
    }
    static __device__ __forceinline__ void weight_rows(const elem16_t* (&pb)[LB], const GemmTileArgs<elem16_t>& g, const uint32_t (&row)[LB], uint32_t ld_p) {
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const uint32_t r = row[i] < g.n_valid ? row[i] : g.n_valid - 1;
            pb[i] = g.b_base + size_t(r) * g.ldb + ((ld_p ^ swizzle(row[i])) << 3);
        }
    }
    static __device__ __forceinline__ void describe(Tile& t, const GemmTileArgs<elem16_t>& g, int stage0, int bias_slot) {
        t.c_base = g.c_base; t.ldc = g.ldc;
        t.m_valid = g.m_valid; t.n_valid = g.n_valid; t.k_tiles = g.K / BK;
        t.k_first = g.k_first < t.k_tiles ? g.k_first : 0u;
        t.act = g.act; t.stage0 = stage0; t.bias_slot = bias_slot;
    }

    // Per-lane source addresses, the load of the bias into LDS slot `bias_slot`, then the loads of
    // the first STAGES-1 slices. Activation rows past the valid range read zeros (a_pad; the last valid
    // row without it) and weight rows past it re-read the last valid row: their products land in
    // accumulator rows / columns that are never stored, and a matrix core that multiplies zeros draws
    // less power than one that multiplies data. The stages stage0 ..
    // stage0+STAGES-2 and the bias slot must not be in use by any wavefront. The bias load is the
    // oldest of the tile's loads, so the first wait of mainloop() covers it.
    static __device__ __forceinline__ void begin(Tile& t, const GemmTileArgs<elem16_t>& g, int stage0, int bias_slot, char* smem) {
        const uint32_t tid = local_tid();
        const int wave = group_wave(__builtin_amdgcn_readfirstlane(tid >> 6)), lane = tid & 63;
        const int ld_r = lane / kChunks, ld_p = lane % kChunks;
        load_bias(g, bias_slot, smem, wave, lane);
        uint32_t arow[LA], brow[LB];
#pragma unroll
        for (int i = 0; i < LA; ++i) arow[i] = kRowsPerLoad * (wave + kWaves * i) + ld_r;
#pragma unroll
        for (int i = 0; i < LB; ++i) brow[i] = kRowsPerLoad * (wave + kWaves * i) + ld_r;
        source_rows(t.pa, g, arow, ld_p);
        weight_rows(t.pb, g, brow, ld_p);
        describe(t, g, stage0, bias_slot);
#pragma unroll
        for (int st = 0; st < STAGES - 1; ++st)
            if (uint32_t(st) < t.k_tiles) issue_slice(t, smem, st);
    }

    // `after_first_barrier()` is called by every thread once, right behind the workgroup barrier that
    // follows the wait for the tile's first slice. Every vector-memory operation a wavefront issued
    // before begin() of this tile has completed by then, in every wavefront: what a persistent
    // workgroup stored in the epilogue of its previous tile may be announced to other workgroups from
    // there without a wait of its own. (begin() must follow the previous tile's finish().)
    static __device__ __forceinline__ void mainloop(const Tile& t, Acc& acc, char* smem) {
        mainloop(t, acc, smem, [] {});
    }
    template <typename Hook>
    static __device__ __forceinline__ void mainloop(const Tile& t, Acc& acc, char* smem, Hook&& after_first_barrier) {
        const int wave = group_wave(threadIdx.x >> 6), lane = threadIdx.x & 63;
        const int wm = wave / WAVES_N, wn = wave % WAVES_N;
        // a lane's share of an operand fragment: 16 bytes of row fr_row, the fr_part-th 8 values of the K step
        const int fr_row = lane & (MI - 1), fr_part = lane / MI;
        if (rows_absent(t, __builtin_amdgcn_readfirstlane(wave) / WAVES_N)) {   // (a scalar condition: the branch holds barriers)
            // None of this wavefront's rows exist (an expert with few rows): it brings its share of
            // every slice into LDS at the same points of the same sequence of barriers as the others,
            // and leaves the fragment reads and the matrix instructions out.
            if constexpr (AHEAD2) {
                constexpr int L = LA + LB;
                asm volatile("s_barrier" ::: "memory");
                if (t.k_tiles > 1) issue_range<0, L>(t, smem, 1);
                for (uint32_t kt = 0; kt < t.k_tiles; ++kt) {
                    if (kt + 1 < t.k_tiles) wait_vmcnt<L>();
                    else wait_vmcnt<0>();
                    asm volatile("s_barrier" ::: "memory");
                    if (kt == 0) after_first_barrier();
                    if (kt + 2 < t.k_tiles) {
                        asm volatile("s_barrier" ::: "memory");
                        issue_range<0, L>(t, smem, kt + 2);
                    }
                }
            } else {
                for (uint32_t kt = 0; kt < t.k_tiles; ++kt) {
                    const uint32_t later = t.k_tiles - 1 - kt;
                    if (STAGES >= 4 && later >= 2) wait_vmcnt<(STAGES >= 4 ? 2 : 0) * kLoadsPerSlice>();
                    else if (STAGES >= 3 && later >= 1) wait_vmcnt<kLoadsPerSlice>();
                    else wait_vmcnt<0>();
                    asm volatile("s_barrier" ::: "memory");
                    if (kt == 0) after_first_barrier();
                    if (kt + (STAGES - 1) < t.k_tiles) issue_slice(t, smem, kt + STAGES - 1);
                }
            }
            return;
        }
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int mi = 0; mi < TM; ++mi)
#pragma unroll
                for (int v = 0; v < int(sizeof(AccTile) / sizeof(float)); ++v) acc[ni][mi][v] = 0.f;
        // Fragment addresses inside a stage. Rows MI apart share their swizzle, and K step ks only
        // flips the upper bits of the chunk position (a step spans 2 chunks of 16 bytes with the
        // 32-row tiles, 4 with the 16-row tiles), so one base per operand is enough: the address of
        // block i at step ks is (base ^ (ks << kStepShift)) + i * MI rows.
        constexpr int kStepShift = MI == 32 ? 5 : 6;
        const int rx = wm * WM + fr_row, rw = wn * WN + fr_row;
        const int base_x = rx * kRowBytes + ((fr_part ^ swizzle(rx)) << 4);
        const int base_w = kABytes + rw * kRowBytes + ((fr_part ^ swizzle(rw)) << 4);
        // The operand fragments of K step ks+1 are read from LDS while the matrix core works on step ks.
        // 32-row tiles: two sets of fragments, fw[ks & 1] and fx[ks & 1]. 16-row tiles have twice as many
        // fragments per step: the larger set (the `outer` one: x with tall wavefront tiles, w with wide
        // ones) is walked in the outer loop of a step, each of its fragments serving NI instructions in
        // a row and making way for its successor of the next step right behind them (one set of
        // registers, fo); only the smaller set is kept twice (fi[ks & 1]).
        constexpr bool kOuterX = TM >= TN;
        constexpr int NO = kOuterX ? TM : TN, NI = kOuterX ? TN : TM;
        static_assert(MI == 32 || (NI >= 2 && NO >= NI));
        // XB: how many of the wavefront's TM blocks of MI rows hold rows of the tile. The blocks behind
        // them are left out of the fragment reads and the matrix instructions (with the 16-row tiles, in
        // the configurations that take the trouble: kBlockSkip); their accumulators are never stored.
        auto body = [&](auto xb_tag) {
            constexpr int XB = decltype(xb_tag)::value;
            auto x_block_used = [](int mi) { return mi < XB; };
            vec8 fw[2][MI == 32 ? TN : 1], fx[2][MI == 32 ? TM : 1];
            vec8 fo[MI == 16 ? NO : 1], fi[2][MI == 16 ? NI : 1];
            const int base_o = kOuterX ? base_x : base_w, base_i = kOuterX ? base_w : base_x;
            auto read_fragments = [&](const char* st, int ks) {
                if constexpr (MI == 32) {
#pragma unroll
                    for (int ni = 0; ni < TN; ++ni) fw[ks & 1][ni] = __builtin_bit_cast(vec8, load16(st + (base_w ^ (ks << kStepShift)) + ni * MI * kRowBytes));
#pragma unroll
                    for (int mi = 0; mi < TM; ++mi) fx[ks & 1][mi] = __builtin_bit_cast(vec8, load16(st + (base_x ^ (ks << kStepShift)) + mi * MI * kRowBytes));
                } else {
#pragma unroll
                    for (int k = 0; k < NI; ++k)
                        if (kOuterX || x_block_used(k)) fi[ks & 1][k] = __builtin_bit_cast(vec8, load16(st + (base_i ^ (ks << kStepShift)) + k * MI * kRowBytes));
#pragma unroll
                    for (int o = 0; o < NO; ++o)
                        if (!kOuterX || x_block_used(o)) fo[o] = __builtin_bit_cast(vec8, load16(st + (base_o ^ (ks << kStepShift)) + o * MI * kRowBytes));
                }
            };
            // Where one load of slice kn comes from and goes to (load li < LA: activation rows, else weight rows).
            struct SliceLoads { uint32_t sa, sb, k0; };
            const uint32_t lds_wave = lds_address(smem) + 1024 * scalar_wave();
            auto loads_of = [&](uint32_t kn) {
                SliceLoads l;
                l.sa = lds_wave + stage_of(t, kn) * kStage;
                l.sb = l.sa + kABytes;
                uint32_t slice = kn + t.k_first;
                slice = slice >= t.k_tiles ? slice - t.k_tiles : slice;
                l.k0 = slice * BK;
                return l;
            };
            // A quarter of a slice's matrix instructions (one K step with the 32-row tiles, half a K step
            // with the 16-row tiles) in a pinned order: one matrix instruction, behind it one LDS read of the
            // next K step's fragments (behind the first TN + TM instructions of a step) and, with LOADS, one
            // global load of a later slice, and again. Issued as blocks - all reads, then all
            // matrix instructions - the two wavefronts of a SIMD took turns instead of overlapping, and a
            // slice's loads in a block in front of a K step held the matrix cores up (8 experts x 2560
            // rows, hidden size 4096, both projections: 3.80 ms in blocks, 3.49 with the reads interleaved,
            // 3.47 with the loads interleaved too; with operands resident in L2 3.49, 2.96 and 2.72).
            // The loads are a compile-time switch: a branch around matrix instructions makes the compiler keep
            // two copies of the accumulators.
            // `first_tag`, `count_tag`: the quarter carries the loads first .. first + count - 1 of the slice `l`
            // describes, evenly spaced behind its matrix instructions (count 0: none).
            // `sync_tag` (S >= 0): in front of the quarter's S-th matrix instruction the wavefront waits for its LDS
            // reads and for the workgroup; the quarter's loads come behind that point.
            auto quarter = [&](const char* st, auto q_tag, const SliceLoads& l, auto first_tag, auto count_tag, auto sync_tag) {
                constexpr int Q = decltype(q_tag)::value, FIRST = decltype(first_tag)::value, COUNT = decltype(count_tag)::value;
                constexpr int S = decltype(sync_tag)::value, J0 = S > 0 ? S : 0;
                constexpr int kParts = kQuarters / kSteps;                 // quarters per K step
                constexpr int ks = Q / kParts, part = Q % kParts;
                static_assert(COUNT <= kPerQuarter - J0);
                constexpr int kEvery = (kPerQuarter - J0) / (COUNT > 0 ? COUNT : 1);
#pragma unroll
                for (int j = 0; j < kPerQuarter; ++j) {
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (S >= 0) {
                        if (j == S) {
                            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
                            asm volatile("s_barrier" ::: "memory");
                        }
                    }
                    const int i = part * kPerQuarter + j;                  // the step's i-th matrix instruction
                    if constexpr (MI == 32) {
                        const int ni = i / TM, mi = i % TM;
                        acc[ni][mi] = Elem16<E>::mfma32(fw[ks & 1][ni], fx[ks & 1][mi], acc[ni][mi]);
                        if (ks + 1 < kSteps) {
                            const int nb = (ks + 1) & 1;
                            if (i < TN) fw[nb][i] = __builtin_bit_cast(vec8, load16(st + (base_w ^ ((ks + 1) << kStepShift)) + i * MI * kRowBytes));
                            else if (i < TN + TM) fx[nb][i - TN] = __builtin_bit_cast(vec8, load16(st + (base_x ^ ((ks + 1) << kStepShift)) + (i - TN) * MI * kRowBytes));
                        }
                    } else {
                        const int o = i / NI, k = i % NI;
                        if (x_block_used(kOuterX ? o : k)) {   // (folds at compile time: o and k are unrolled)
                            if constexpr (kOuterX) acc[k][o] = Elem16<E>::mfma16(fi[ks & 1][k], fo[o], acc[k][o]);
                            else acc[o][k] = Elem16<E>::mfma16(fo[o], fi[ks & 1][k], acc[o][k]);
                        }
                        if (ks + 1 < kSteps) {
                            // behind the last instruction that uses fo[o]: its successor; behind the first
                            // instructions of the first NI outer rounds: the inner set of the next step
                            if (k == NI - 1) {
                                if (!kOuterX || x_block_used(o)) fo[o] = __builtin_bit_cast(vec8, load16(st + (base_o ^ ((ks + 1) << kStepShift)) + o * MI * kRowBytes));
                            } else if (k == 0 && o < NI) {
                                if (kOuterX || x_block_used(o)) fi[(ks + 1) & 1][o] = __builtin_bit_cast(vec8, load16(st + (base_i ^ ((ks + 1) << kStepShift)) + o * MI * kRowBytes));
                            }
                        }
                    }
                    if constexpr (COUNT > 0) {
                        if (j >= J0 && (j - J0) % kEvery == 0 && (j - J0) / kEvery < COUNT) issue_one(t, l.sa, l.sb, l.k0, FIRST + (j - J0) / kEvery);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            using Q0 = std::integral_constant<int, 0>; using Q1 = std::integral_constant<int, 1>;
            using Q2 = std::integral_constant<int, 2>; using Q3 = std::integral_constant<int, 3>;
            using NoSync = std::integral_constant<int, -1>;
            static_assert(MI == 16 || TN + TM <= kPerQuarter, "the first quarter of a K step has a matrix instruction for every fragment read");
            if constexpr (AHEAD2) {
                // The barrier that frees the stage sits kReleaseAt matrix instructions into the second K step, and
                // all loads of the slice after the next go out behind it, half in each quarter.
                constexpr int L = LA + LB;
                constexpr int AT = kReleaseAt;
                constexpr int M2 = L / 2;
                static_assert(M2 <= kPerQuarter - AT && L - M2 <= kPerQuarter);
                using None = std::integral_constant<int, 0>;
                asm volatile("s_barrier" ::: "memory");   // every wavefront has left the previous tile's epilogue, staged where slice 1 goes
                if (t.k_tiles > 1) issue_range<0, L>(t, smem, 1);
                auto slice = [&](uint32_t kt, auto next_tag, auto next2_tag) {
                    constexpr bool NEXT = decltype(next_tag)::value, NEXT2 = decltype(next2_tag)::value;
                    // this wavefront's loads of slice kt are complete once only those of slice kt+1 are outstanding
                    if constexpr (NEXT) wait_vmcnt<L>();
                    else wait_vmcnt<0>();
                    asm volatile("s_barrier" ::: "memory");   // every wavefront's share of slice kt is in LDS
                    if (kt == 0) after_first_barrier();
                    const char* st = smem + stage_of(t, kt) * kStage;
                    read_fragments(st, 0);
                    quarter(st, Q0{}, SliceLoads{}, None{}, None{}, NoSync{});
                    quarter(st, Q1{}, SliceLoads{}, None{}, None{}, NoSync{});
                    const SliceLoads l2 = NEXT2 ? loads_of(kt + 2) : SliceLoads{};
                    quarter(st, Q2{}, l2, None{}, std::integral_constant<int, NEXT2 ? M2 : 0>{}, std::integral_constant<int, NEXT2 ? AT : -1>{});
                    quarter(st, Q3{}, l2, std::integral_constant<int, M2>{}, std::integral_constant<int, NEXT2 ? L - M2 : 0>{}, NoSync{});
                };
                const uint32_t ahead = t.k_tiles >= 2 ? t.k_tiles - 2 : 0u;   // slices that request slice kt+2
                for (uint32_t kt = 0; kt < ahead; ++kt) slice(kt, std::true_type{}, std::true_type{});
                if (t.k_tiles >= 2) slice(t.k_tiles - 2, std::true_type{}, std::false_type{});
                slice(t.k_tiles - 1, std::false_type{}, std::false_type{});
            } else {
                static_assert(LA + LB <= kQuarters * kPerQuarter, "the loads of a slice fit behind the matrix instructions of a slice");
                auto top = [&](uint32_t kt) {
                    // This wavefront's loads of slice kt are complete once only those of the later slices
                    // already issued (STAGES-2 of them, fewer at the end of the tile) are outstanding.
                    const uint32_t later = t.k_tiles - 1 - kt;
                    if (STAGES >= 4 && later >= 2) wait_vmcnt<(STAGES >= 4 ? 2 : 0) * kLoadsPerSlice>();
                    else if (STAGES >= 3 && later >= 1) wait_vmcnt<kLoadsPerSlice>();
                    else wait_vmcnt<0>();
                    // every wavefront's share of slice kt is in LDS, and everyone has finished with the stage
                    // the next loads overwrite (slice kt-1, or the previous tile's epilogue staging)
                    asm volatile("s_barrier" ::: "memory");
                    if (kt == 0) after_first_barrier();
                };
                // Quarter q carries the loads q * kPerQuarter ... of the slice STAGES-1 ahead, one behind each
                // matrix instruction, until they run out (sharing them out evenly over the four K steps,
                // which three stages would allow, changes nothing where it was measured: 2.93 against
                // 2.92 ms per forward at the 256-expert top-8 shape, which is bound by HBM)
                auto ksteps = [&](const char* st, const SliceLoads& l, auto loads_tag) {
                    static_for<kQuarters>([&](auto q_tag) {
                        constexpr int q = decltype(q_tag)::value;
                        constexpr int left = LA + LB - q * kPerQuarter;
                        constexpr int count = !decltype(loads_tag)::value || left <= 0 ? 0 : (left < kPerQuarter ? left : kPerQuarter);
                        quarter(st, q_tag, l, std::integral_constant<int, q * kPerQuarter>{}, std::integral_constant<int, count>{}, NoSync{});
                    });
                };
                const uint32_t ahead = t.k_tiles >= uint32_t(STAGES - 1) ? t.k_tiles - (STAGES - 1) : 0u;   // slices that request a later one
                for (uint32_t kt = 0; kt < ahead; ++kt) {
                    top(kt);
                    const char* st = smem + stage_of(t, kt) * kStage;
                    read_fragments(st, 0);
                    ksteps(st, loads_of(kt + STAGES - 1), std::true_type{});
                }
                for (uint32_t kt = ahead; kt < t.k_tiles; ++kt) {
                    top(kt);
                    const char* st = smem + stage_of(t, kt) * kStage;
                    read_fragments(st, 0);
                    ksteps(st, SliceLoads{}, std::false_type{});
                }
            }
        };   // body
        if constexpr (kBlockSkip) {
            // (the same in all lanes of a wavefront; every version goes through the same barriers)
            const int rows_here = int(t.m_valid) - __builtin_amdgcn_readfirstlane(wave) / WAVES_N * WM;
            const int used = rows_here >= WM ? TM : (rows_here <= MI ? 1 : (rows_here + MI - 1) / MI);
            static_assert(TM == 4);
            switch (used) {
                case 1: body(std::integral_constant<int, 1>{}); break;
                case 2: body(std::integral_constant<int, 2>{}); break;
                case 3: body(std::integral_constant<int, 3>{}); break;
                default: body(std::integral_constant<int, 4>{}); break;
            }
        } else {
            body(std::integral_constant<int, TM>{});
        }
    }

    // Whether none of the rows of the wavefronts in row wm of the wavefront grid exist in this tile
    // (the same for all lanes of a wavefront), for the configurations that treat such wavefronts
    // apart: the one with the loads two slices ahead, which runs where experts hold few rows and
    // the loads bound the tile (64-expert shape with skewed routing: 301 against 304 us per forward);
    // where the matrix work bounds it the extra branch costs more than the few such tiles bring
    // (8-expert shape with hidden size 4096: 3.57 against 3.53 ms).
    static __device__ __forceinline__ bool rows_absent(const Tile& t, int wm) {
        if constexpr (AHEAD2) return uint32_t(wm * WM) >= t.m_valid;
        else return false;
    }

    // The stage the tile's last K slice was read from (free once every wavefront has left mainloop()).
    static __device__ __forceinline__ int last_stage(const Tile& t) { return (t.stage0 + t.k_tiles - 1) % STAGES; }
    // The stage the next tile's first slice must go to.
    static __device__ __forceinline__ int next_stage0(const Tile& t) { return (t.stage0 + t.k_tiles) % STAGES; }

    // Epilogue that keeps the fp32 sums as they are (no bias, no activation, no rounding): the
    // tile goes to out[m * ldo + n] as floats, for a caller that sums several K ranges of one product.
    // Every wavefront must have left mainloop(). Each wavefront transposes its 32 x 32 blocks through
    // 4 KB of its own in the stage of the last slice (rows of 128 bytes, chunk c of row r at position
    // c ^ ((r >> 1) & 7)) and stores whole 128-byte lines.
    static __device__ __forceinline__ void finish_partial(const Tile& t, Acc& acc, char* smem, float* out, uint32_t ldo) {
        static_assert(MI == 32, "written for the accumulator layout of the 32 x 32 tiles");
        const uint32_t tid = local_tid();
        const int wave = group_wave(__builtin_amdgcn_readfirstlane(tid >> 6)), lane = tid & 63;
        const int wm = wave / WAVES_N, wn = wave % WAVES_N;
        const int fr_row = lane & 31, fr_half = lane >> 5;
        char* stg = smem + last_stage(t) * kStage + wave * (kPanelRows * 128);
#pragma unroll
        for (int mi = 0; mi < TM; ++mi)
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 v{acc[ni][mi][4 * q], acc[ni][mi][4 * q + 1], acc[ni][mi][4 * q + 2], acc[ni][mi][4 * q + 3]};
                    *reinterpret_cast<f32x4*>(stg + fr_row * 128 + (((2 * q + fr_half) ^ ((fr_row >> 1) & 7)) << 4)) = v;
                }
#pragma unroll
                for (int it = 0; it < kPanelRows * 8 / kWave; ++it) {
                    const int id = it * kWave + lane;
                    const int r = id >> 3, c = id & 7;
                    const u32x4 v = load16(stg + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
                    const uint32_t m = wm * WM + mi * 32 + r, n = wn * WN + ni * 32 + c * 4;
                    // the sums are read by other workgroups after a grid-wide barrier
                    if (m < t.m_valid && n < t.n_valid) store16_through(out + size_t(m) * ldo + n, v);
                }
            }
    }

    // Epilogue. Every wavefront must have left mainloop().
    static __device__ __forceinline__ void finish(const Tile& t, Acc& acc, char* smem) {
        if (rows_absent(t, __builtin_amdgcn_readfirstlane(int(local_tid() >> 6)) / WAVES_N)) return;   // nothing of this wavefront's is stored
        const TileOut out{t.c_base, t.ldc, t.m_valid, t.n_valid, t.act};
        epilogue16<E, WM, WN, WAVES_N, STREAM_OUT>(out, acc, smem + last_stage(t) * kStage, smem + kBiasOffset + t.bias_slot * kBiasBytes);
    }
};

// ------------------------------------------------------------------------------------------------
// The 256 x 256 tile, 2 x 4 wavefronts of 128 x 64, in which the two wavefronts of a SIMD take turns: while one
// multiplies, the other reads its next fragments from LDS and requests loads. A slice of 64 values of K is two
// sections of 32 matrix instructions, the upper and the lower half of the wavefront's rows against all of its
// columns, each behind the LDS reads it needs; wavefronts 4 to 7 run one half section behind wavefronts 0 to 3,
// which sit on the same SIMDs, and a workgroup barrier ends every half section:
//
//     wavefronts 0-3   read 0 | multiply 0 | read 1     | multiply 1 | read 0 of the next slice ...
//     wavefronts 4-7          | read 0     | multiply 0 | read 1     | multiply 1 ...
//
// (Both wavefronts of a SIMD in step, the reads between the matrix instructions, is the main loop of Gemm16 with AHEAD2:
// its slices begin with reads that nothing covers and its matrix cores are busy 66 % of an 8-expert forward.)
// Every accumulator takes the two K steps of a section one right behind the other: the second reads the sum where
// the first leaves it, which takes 5 % less energy (register operands, whole device, both 32 instructions a run: 2 160 against
// 2 055 TFLOP/s). K is added in the order of Gemm16, so that a row's bits do not depend on the tile that computes it.
//
// Two stages. The rows a section reads are free once both groups of wavefronts have read them, and take the slice
// after the next: the weights and the upper halves' activations behind section 0, the lower halves' behind section 1.
// Of the 8 loads of a wavefront and slice, 6 go out in section 1 and 2 in section 0 of the next slice, and a wait
// always leaves the 8 youngest outstanding: every load has a whole slice to land.
//
// What bounds it: power, and where it is not reached the ends of a tile. In a loop over the tiles of 8 experts of 2 048 rows (random data) a slice takes 2 240 to
// 2 400 clocks of which the matrix cores need 2 048, against 2 700 to 2 830 in step; they run at 1.65 GHz instead of 1.8, and
// the projections of 4 096 x 14 336 take 1 289 + 1 264 us (1 490 + 1 520 TFLOP/s) instead of 1 437 + 1 392, of 2 048 x 2 048 98 instead of 112 each. Four sections
// of 16 instructions a slice: 1 382 + 1 328, 107. Us per forward: 8 192 tokens, 8 experts top-2, 4 096 x 14 336:
// 3 085 -> 2 806; 4 608 tokens, 16 experts, 2 048 x 4 096: 371 -> 344; 4 096, 2 048 x 2 048: 146.5 -> 139.5; 8 192, 64 experts,
// skewed: 281 -> 276.5; 1 280, 8 experts top-1, 4 096 x 7 168: 262 -> 254.
// ------------------------------------------------------------------------------------------------
template <typename E, bool STREAM_B>
struct GemmPingPong : Gemm16<E, 256, 256, 2, 4, 64, 2, STREAM_B, true> {
    typedef Gemm16<E, 256, 256, 2, 4, 64, 2, STREAM_B, true> Base;
    typedef typename Base::Tile Tile;
    typedef typename Base::Acc Acc;
    typedef typename Base::vec8 vec8;
    using Base::kStage; using Base::kABytes; using Base::kRowBytes; using Base::kSteps; using Base::WM; using Base::WN; using Base::TM; using Base::TN;
    static constexpr int kLive = TM / 2;                 // blocks of 16 rows in a section
    static constexpr int kLoads = 4;                     // loads of a wavefront and slice: as many for the activations as for the weights
    static_assert(Base::LA == kLoads && Base::LB == kLoads && kSteps == 2 && Base::kWaves == 8 && WM == 128);

    // The first row of the tile that load j of wavefront w covers, 8 rows each: loads 0 and 1 bring the upper halves of the
    // two wavefront rows, 2 and 3 the lower ones. (Weight rows: as in Gemm16.)
    static __device__ __forceinline__ uint32_t x_row(uint32_t w, int j) { return uint32_t(j & 1) * WM + uint32_t(j >> 1) * (WM / 2) + 8 * w; }
    static __device__ __forceinline__ uint32_t w_row(uint32_t w, int j) { return 64 * uint32_t(j) + 8 * w; }

    struct SliceLoads { uint32_t lds, k0; };   // the LDS address of the wavefront's rows in the stage, the first value of K
    static __device__ __forceinline__ SliceLoads loads_of(const Tile& t, char* smem, uint32_t kt) {
        uint32_t slice = kt + t.k_first;
        slice = slice >= t.k_tiles ? slice - t.k_tiles : slice;
        return SliceLoads{lds_address(smem) + Base::stage_of(t, kt) * kStage + 1024 * wave_index(), slice * Base::kSliceK};
    }
    // The loads of a slice that replace what section 0 reads, and those that replace what only section 1 reads.
    static __device__ __forceinline__ void load_x(const Tile& t, const SliceLoads& l, int j) { direct_load16<false>(t.pa[j] + l.k0, l.lds + x_row(0, j) * kRowBytes); }
    static __device__ __forceinline__ void load_first(const Tile& t, const SliceLoads& l) {
        load_x(t, l, 0); load_x(t, l, 1);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) direct_load16<STREAM_B>(t.pb[j] + l.k0, l.lds + kABytes + w_row(0, j) * kRowBytes);
    }
    static __device__ __forceinline__ void load_second(const Tile& t, const SliceLoads& l) { load_x(t, l, 2); load_x(t, l, 3); }
    static constexpr int kFirst = 2 + kLoads, kSecond = 2;   // how many they are

    static __device__ __forceinline__ void begin(Tile& t, const GemmTileArgs<elem16_t>& g, int stage0, int bias_slot, char* smem) {
        const uint32_t lane = local_tid() & 63, wave = __builtin_amdgcn_readfirstlane(local_tid() >> 6);
        const uint32_t ld_r = lane / Base::kChunks, ld_p = lane % Base::kChunks;
        Base::load_bias(g, bias_slot, smem, wave, lane);
        uint32_t row[kLoads];
#pragma unroll
        for (int j = 0; j < kLoads; ++j) row[j] = x_row(wave, j) + ld_r;
        Base::source_rows(t.pa, g, row, ld_p);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) row[j] = w_row(wave, j) + ld_r;
        Base::weight_rows(t.pb, g, row, ld_p);
        Base::describe(t, g, stage0, bias_slot);
        const SliceLoads l = loads_of(t, smem, 0);
        load_first(t, l);
        load_second(t, l);
    }

    // (`after_first_barrier`: as in Gemm16)
    template <typename Hook>
    static __device__ __forceinline__ void mainloop(const Tile& t, Acc& acc, char* smem, Hook&& after_first_barrier) {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
        const int wm = wave / Base::kWavesN, wn = wave % Base::kWavesN;
        const bool behind = wave >= Base::kWaves / 2;   // (a scalar condition: the branches on it hold barriers)
        auto barrier = [] { asm volatile("s_barrier" ::: "memory"); };

        barrier();   // every wavefront has left the previous tile's epilogue, staged where slice 1 goes
        if (t.k_tiles > 1) {
            load_first(t, loads_of(t, smem, 1));
            wait_vmcnt<kSecond + kFirst>();
        } else {
            wait_vmcnt<kSecond>();
        }
        barrier();   // what section 0 of slice 0 reads is in LDS
        after_first_barrier();
        if (behind) barrier();

        const int fr_row = lane & 15, fr_part = lane >> 4;
        const int rx = wm * WM + fr_row, rw = wn * WN + fr_row;
        const int base_x = rx * kRowBytes + ((fr_part ^ Base::swizzle(rx)) << 4);
        const int base_w = kABytes + rw * kRowBytes + ((fr_part ^ Base::swizzle(rw)) << 4);
        // Blocks of 16 of the wavefront's rows that the tile has rows in. Only they are multiplied, and a section without any
        // reads no fragments. A branch around the matrix instructions of a block costs a full tile 8 % of its loop, so that
        // wavefronts with all their rows run a version without (the same in all lanes, and the same barriers in both).
        const int rows_here = int(t.m_valid) - wm * WM;
        const int blocks = rows_here <= 0 ? 0 : (rows_here + 15) / 16;
        auto body = [&](auto full_tag) {
            constexpr bool FULL = decltype(full_tag)::value;
            auto used = [&](int block) { return FULL || block < blocks; };
#pragma unroll
            for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                for (int mi = 0; mi < TM; ++mi) acc[ni][mi] = f32x4{0.f, 0.f, 0.f, 0.f};
            vec8 fx[kSteps][kLive], fw[kSteps][TN];
            auto read_x = [&](const char* st, int section) {
                if (!used(section * kLive)) return;
#pragma unroll
                for (int ks = 0; ks < kSteps; ++ks)
#pragma unroll
                    for (int i = 0; i < kLive; ++i)
                        fx[ks][i] = __builtin_bit_cast(vec8, load16(st + (base_x ^ (ks << 6)) + (section * kLive + i) * 16 * kRowBytes));
            };
            auto read_w = [&](const char* st) {
                if (!used(0)) return;
#pragma unroll
                for (int ks = 0; ks < kSteps; ++ks)
#pragma unroll
                    for (int i = 0; i < TN; ++i) fw[ks][i] = __builtin_bit_cast(vec8, load16(st + (base_w ^ (ks << 6)) + i * 16 * kRowBytes));
            };
            auto product = [&](int ni, int i, int section) {
#pragma unroll
                for (int ks = 0; ks < kSteps; ++ks) {
                    acc[ni][section * kLive + i] = Elem16<E>::mfma16(fw[ks][ni], fx[ks][i], acc[ni][section * kLive + i]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            // The half section that multiplies, and the barriers around it. The reads have returned in front of the first of
            // them: behind it, loads may replace what they read.
            auto multiply = [&](int section) {
                __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
                __builtin_amdgcn_sched_barrier(0);
                barrier();
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_setprio(1);        // ahead of the reads and loads of the SIMD's other wavefront
                if constexpr (FULL) {
#pragma unroll
                    for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                        for (int i = 0; i < kLive; ++i) product(ni, i, section);
                } else {
#pragma unroll
                    for (int i = 0; i < kLive; ++i)
                        if (used(section * kLive + i)) {
#pragma unroll
                            for (int ni = 0; ni < TN; ++ni) product(ni, i, section);
                        }
                }
                __builtin_amdgcn_s_setprio(0);
                __builtin_amdgcn_sched_barrier(0);
                barrier();
                __builtin_amdgcn_sched_barrier(0);
            };
            // LATER: slices behind this one, 2 standing for any number from there on. Its wait leaves outstanding what the
            // next section does not read.
            auto slice = [&](uint32_t kt, auto later_tag) {
                constexpr int LATER = decltype(later_tag)::value;
                const char* st = smem + Base::stage_of(t, kt) * kStage;
                read_w(st);
                read_x(st, 0);
                if constexpr (LATER >= 1) load_second(t, loads_of(t, smem, kt + 1));
                wait_vmcnt<(LATER >= 1 ? kFirst + kSecond : 0)>();
                multiply(0);
                read_x(st, 1);
                if constexpr (LATER >= 2) load_first(t, loads_of(t, smem, kt + 2));
                if constexpr (LATER >= 1) wait_vmcnt<(LATER >= 2 ? kSecond + kFirst : kSecond)>();
                multiply(1);
            };
            const uint32_t ahead = t.k_tiles >= 2 ? t.k_tiles - 2 : 0u;
            for (uint32_t kt = 0; kt < ahead; ++kt) slice(kt, std::integral_constant<int, 2>{});
            if (t.k_tiles >= 2) slice(t.k_tiles - 2, std::integral_constant<int, 1>{});
            slice(t.k_tiles - 1, std::integral_constant<int, 0>{});
        };
        if (blocks >= TM) body(std::true_type{});
        else body(std::false_type{});
        if (!behind) barrier();
    }
};

// ------------------------------------------------------------------------------------------------
// The same turns for tiles of half the size, 128 x 256 or 256 x 128: wavefronts of 64 x 64, so that a slice is one section of 32
// matrix instructions. Three stages: a slice's loads go out two slices ahead, in the half section that reads, where the stage of
// the slice before is free of both groups' reads; the wait behind them is for the next slice.
//
// What bounds it: its loads, 48 KB a slice. In a loop over the tiles of one expert (2 048 rows, 4 096 x 4 096, random data) a slice takes
// 1 290 clocks of which the matrix cores need 1 024, against 1 720 in step (Gemm16 with three stages); with the wait of the wavefronts in front
// moved behind their matrix instructions (a scalar branch) 1 430. As the smaller tile of 256-row layers, us per forward: 2 944 tokens, 6 experts top-4,
// 448 x 1 088: 89.7 -> 86.0; 2 560, 16 experts top-3, 1 472 x 11 200: 580 -> 571.5; 8 192, 8 experts top-2, 4 096 x 14 336: 2 851 -> 2 837.
// Where weights stream from HBM and are read once the loads of Gemm16, half a slice earlier, are the better ones (variant 1: 1 280 tokens, 256
// experts, 2 304 x 576: 280.5 -> 283).
// ------------------------------------------------------------------------------------------------
// HALVES: the sums of the two halves of K are formed apart and added at the end, as GemmKSplit's are, in whose place such a tile runs (relative
// error against 64 bits, 2 048 tokens, one expert, 1 024 x 4 096, GELU: K in one run 1.66323e-3 in bf16 and 2.0794e-4 in fp16, in halves 1.66308e-3 and
// 2.0783e-4, as on 128 x 128 tiles; 50.8 -> 51.8 us per forward).
template <typename E, int BM, int BN, int WAVES_M, int WAVES_N, bool HALVES>
struct GemmTurns : Gemm16<E, BM, BN, WAVES_M, WAVES_N, 64, 3, false, false> {
    typedef Gemm16<E, BM, BN, WAVES_M, WAVES_N, 64, 3, false, false> Base;
    typedef typename Base::Tile Tile;
    typedef typename Base::Acc Acc;
    typedef typename Base::vec8 vec8;
    using Base::kStage; using Base::kABytes; using Base::kRowBytes; using Base::kSteps; using Base::WM; using Base::WN; using Base::TM; using Base::TN;
    static constexpr int L = Base::kLoadsPerSlice;
    static_assert(WM == 64 && WN == 64 && Base::kWaves == 8 && kSteps == 2);

    // (`after_first_barrier`, the blocks of rows, the barriers: as in GemmPingPong)
    template <typename Hook>
    static __device__ __forceinline__ void mainloop(const Tile& t, Acc& acc, char* smem, Hook&& after_first_barrier) {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
        const int wm = wave / WAVES_N, wn = wave % WAVES_N;
        const bool behind = wave >= Base::kWaves / 2;
        auto barrier = [] { asm volatile("s_barrier" ::: "memory"); };
        if (t.k_tiles > 1) wait_vmcnt<L>();
        else wait_vmcnt<0>();
        barrier();   // slice 0 is in LDS, and every wavefront has left the previous tile's epilogue
        after_first_barrier();
        if (behind) barrier();

        const int fr_row = lane & 15, fr_part = lane >> 4;
        const int rx = wm * WM + fr_row, rw = wn * WN + fr_row;
        const int base_x = rx * kRowBytes + ((fr_part ^ Base::swizzle(rx)) << 4);
        const int base_w = kABytes + rw * kRowBytes + ((fr_part ^ Base::swizzle(rw)) << 4);
        const int rows_here = int(t.m_valid) - wm * WM;
        const int blocks = rows_here <= 0 ? 0 : (rows_here + 15) / 16;
        auto body = [&](auto full_tag) {
            constexpr bool FULL = decltype(full_tag)::value;
            auto used = [&](int block) { return FULL || block < blocks; };
#pragma unroll
            for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                for (int mi = 0; mi < TM; ++mi) acc[ni][mi] = f32x4{0.f, 0.f, 0.f, 0.f};
            vec8 fx[kSteps][TM], fw[kSteps][TN];
            auto product = [&](int ni, int i) {
#pragma unroll
                for (int ks = 0; ks < kSteps; ++ks) {
                    acc[ni][i] = Elem16<E>::mfma16(fw[ks][ni], fx[ks][i], acc[ni][i]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            auto slice = [&](uint32_t kt, auto later_tag) {
                constexpr int LATER = decltype(later_tag)::value;
                const char* st = smem + Base::stage_of(t, kt) * kStage;
                if (used(0)) {
#pragma unroll
                    for (int ks = 0; ks < kSteps; ++ks) {
#pragma unroll
                        for (int i = 0; i < TN; ++i) fw[ks][i] = __builtin_bit_cast(vec8, load16(st + (base_w ^ (ks << 6)) + i * 16 * kRowBytes));
#pragma unroll
                        for (int i = 0; i < TM; ++i) fx[ks][i] = __builtin_bit_cast(vec8, load16(st + (base_x ^ (ks << 6)) + i * 16 * kRowBytes));
                    }
                }
                if constexpr (LATER >= 2) Base::issue_slice(t, smem, kt + 2);
                if constexpr (LATER >= 1) wait_vmcnt<(LATER >= 2 ? L : 0)>();
                __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
                __builtin_amdgcn_sched_barrier(0);
                barrier();
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_setprio(1);
                if constexpr (FULL) {
#pragma unroll
                    for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                        for (int i = 0; i < TM; ++i) product(ni, i);
                } else {
#pragma unroll
                    for (int i = 0; i < TM; ++i)
                        if (used(i)) {
#pragma unroll
                            for (int ni = 0; ni < TN; ++ni) product(ni, i);
                        }
                }
                __builtin_amdgcn_s_setprio(0);
                __builtin_amdgcn_sched_barrier(0);
                barrier();
                __builtin_amdgcn_sched_barrier(0);
            };
            const uint32_t ahead = t.k_tiles >= 2 ? t.k_tiles - 2 : 0u;
            uint32_t kt = 0;
            f32x4 saved[HALVES ? TN : 1][HALVES ? TM : 1];
            auto halfway = [&] {
#pragma unroll
                for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                    for (int mi = 0; mi < TM; ++mi) {
                        saved[ni][mi] = acc[ni][mi];
                        acc[ni][mi] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
            };
            if constexpr (HALVES) {
                const uint32_t half = t.k_tiles >= 4 ? (t.k_tiles + 1) / 2 : 0u;   // (at most `ahead`)
                for (; kt < half; ++kt) slice(kt, std::integral_constant<int, 2>{});
                halfway();
            }
            for (; kt < ahead; ++kt) slice(kt, std::integral_constant<int, 2>{});
            if (t.k_tiles >= 2) slice(t.k_tiles - 2, std::integral_constant<int, 1>{});
            if constexpr (HALVES) {
                if (t.k_tiles == 2 || t.k_tiles == 3) halfway();   // (what it saved above was zero)
            }
            slice(t.k_tiles - 1, std::integral_constant<int, 0>{});
            if constexpr (HALVES) {
#pragma unroll
                for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                    for (int mi = 0; mi < TM; ++mi) acc[ni][mi] = saved[ni][mi] + acc[ni][mi];
            }
        };
        if (blocks >= TM) body(std::true_type{});
        else body(std::false_type{});
        if (!behind) barrier();
    }
    static __device__ __forceinline__ void finish(const Tile& t, Acc& acc, char* smem) {
        const TileOut out{t.c_base, t.ldc, t.m_valid, t.n_valid, t.act};
        epilogue16<E, WM, WN, WAVES_N, false>(out, acc, smem + Base::last_stage(t) * kStage, smem + Base::kBiasOffset + t.bias_slot * Base::kBiasBytes);
    }
};

// ------------------------------------------------------------------------------------------------
// A tile small enough for four wavefronts, worked on by eight: two groups of four each run the main loop
// of G over one half of K, on LDS of their own, and the halves are added at the end. For layers whose
// tiles would otherwise leave CUs without one. Four wavefronts of 64 x 64 read half as much LDS per
// matrix instruction as eight of 32 x 64 would, and two rings of stages keep twice the bytes in flight,
// which is what a CU with a single small tile is short of.
//
// What bounds it is the CU's load path (47 KB a microsecond): a 64 x 128 tile moves 24 KB per 64 values of K. Measured
// against the 128 x 256 tile at layers that have few: 128 tokens, 8 experts top-2, 4 096 x 14 336: 389 -> 341 us per
// forward; 640 tokens, 8 experts, 704 x 512: 50 -> 37; one expert, 384 tokens, 512 x 13 376: 218 -> 105.
//
// The groups share the workgroup's barriers: a barrier of one is a barrier of the other, whichever slice
// each is at, so all that has to match is how many they pass (barriers_of). The sum of the halves is one fp32
// addition per element, in the same order in every launch mode.
// ------------------------------------------------------------------------------------------------
template <typename G>
struct GemmKSplit {
    typedef typename G::Element E;
    static constexpr int BM = G::kBM, BN = G::kBN;
    static constexpr int kGroups = 2, kThreads = kGroups * G::kThreads, kSliceK = G::kSliceK;
    static constexpr int kSmemBytes = kGroups * G::kSmemBytes;
    static_assert(G::kMI == 16, "the accumulator layout finish() expects");
    static_assert(BM * BN * 4 <= G::kStages * G::kStage, "a group's sums fit its stages");
    static_assert(BN % 64 == 0 && kThreads % (BN / 8) == 0 && BM % (kThreads / (BN / 8)) == 0);

    struct Tile {
        typename G::Tile half;     // this group's half of K
        uint32_t missing;          // barriers the other group passes beyond this one's
    };
    typedef typename G::Acc Acc;

    static __device__ __forceinline__ uint32_t group() { return wave_index() / uint32_t(G::kWaves); }
    // Workgroup barriers in G's main loop over n slices.
    static __device__ __forceinline__ uint32_t barriers_of(uint32_t n) {
        if (!G::kAhead2 || n == 0) return n;
        return 1 + n + (n > 2 ? n - 2 : 0);
    }
    static __device__ __forceinline__ int next_stage0(const Tile& t) { return G::next_stage0(t.half); }

    static __device__ __forceinline__ void begin(Tile& t, const GemmTileArgs<elem16_t>& args, int stage0, int bias_slot, char* smem) {
        GemmTileArgs<elem16_t> g = args;
        const uint32_t n = args.K / kSliceK, first = (n + 1) / 2, mine = group() == 0 ? first : n - first;
        if (group() != 0) {
            g.a_base += size_t(first) * kSliceK;
            g.b_base += size_t(first) * kSliceK;
        }
        g.K = mine * kSliceK;
        if (g.k_first >= mine) g.k_first = mine ? g.k_first % mine : 0u;
        t.missing = barriers_of(first) - barriers_of(mine);
        G::begin(t.half, g, stage0, bias_slot, smem + group() * G::kSmemBytes);
    }

    // Brings the weight rows of a tile's first slices, two of either half of K, into the L2: called between the main loop of a tile and its
    // finish(), for the next one. Its own loads go out behind that and behind the look-up of its rows, and the memory has nothing to do meanwhile
    // where all CUs are between two tiles at the same time and a weight row is read by nobody else. `scratch`: kTouchBytes of LDS.
    // Us per forward: 512 tokens, 16 experts top-2, 2 048 x 2 048: 84.4 -> 83.5; 128 tokens, 8 experts, 4 096 x 14 336: 332.4 -> 327.6. Tiles that
    // share weights lose (256 x 256 ones 2 %, 128-row ones that stream their weights between +2.5 and -1 %), as do 64-row ones of several row blocks.
    static constexpr int kTouchBytes = kGroups * G::kWaves * 256;
    static __device__ __forceinline__ void touch(const GemmTileArgs<elem16_t>& args, char* scratch) {
        static_assert(kThreads == 4 * BN);
        const uint32_t tid = local_tid(), row = tid % BN, half = (tid / BN) & 1u, n = args.K / kSliceK, first = (n + 1) / 2;
        const uint32_t mine = half ? n - first : first, slice = mine ? (args.k_first + tid / (2 * BN)) % mine + half * first : 0u;
        const elem16_t* from = args.b_base + size_t(row < args.n_valid ? row : args.n_valid - 1) * args.ldb + size_t(slice) * kSliceK;
        touch_lines(from, lds_address(scratch) + 256 * wave_index());
    }

    template <typename Hook>
    static __device__ __forceinline__ void mainloop(const Tile& t, Acc& acc, char* smem, Hook&& after_first_barrier) {
        if (t.half.k_tiles != 0) {
            G::mainloop(t.half, acc, smem + group() * G::kSmemBytes, after_first_barrier);
        } else {
            // K is a single slice, the other group's (whose first barrier announces this group's stores too)
#pragma unroll
            for (auto& row : acc)
#pragma unroll
                for (auto& a : row) a = f32x4{0.f, 0.f, 0.f, 0.f};
            wait_vmcnt<0>();
        }
        for (uint32_t i = 0; i < t.missing; ++i) asm volatile("s_barrier" ::: "memory");
    }

    // Both groups leave their fp32 sums in their stages (rows of BN values, 16-byte chunk c of row r at
    // position c ^ (r & 15)); then every thread adds, biases, activates and stores runs of eight columns.
    // Every wavefront must have left mainloop(), and takes part in the two barriers.
    static __device__ __forceinline__ void finish(const Tile& t, Acc& acc, char* smem) {
        if (t.half.act == 0) finish_act<0>(t, acc, smem);
        else if (t.half.act == 1) finish_act<1>(t, acc, smem);
        else finish_act<2>(t, acc, smem);
    }
    template <int ACT>
    static __device__ __forceinline__ void finish_act(const Tile& t, Acc& acc, char* smem) {
        const uint32_t tid = local_tid();
        const int wave = G::group_wave(__builtin_amdgcn_readfirstlane(tid >> 6)), lane = tid & 63;
        const int wm = wave / G::kWavesN, wn = wave % G::kWavesN;
        char* sums = smem + group() * G::kSmemBytes;
        if (uint32_t(wm * G::WM) < t.half.m_valid) {
#pragma unroll
            for (int mi = 0; mi < G::TM; ++mi)
#pragma unroll
                for (int ni = 0; ni < G::TN; ++ni) {
                    const int r = wm * G::WM + mi * 16 + (lane & 15), c = (wn * G::WN + ni * 16) / 4 + (lane >> 4);
                    *reinterpret_cast<f32x4*>(sums + r * (BN * 4) + ((c ^ (r & 15)) << 4)) = acc[ni][mi];
                }
        }
        __syncthreads();
        constexpr int kPerRow = BN / 8, kRows = kThreads / kPerRow;   // threads a row, rows a pass
        const int c = int(tid) % kPerRow;
        typename Elem16<E>::vec8 bias = __builtin_bit_cast(typename Elem16<E>::vec8, load16(smem + G::kBiasOffset + t.half.bias_slot * G::kBiasBytes + c * 16));
#pragma unroll
        for (int pass = 0; pass < BM / kRows; ++pass) {
            const int r = pass * kRows + int(tid) / kPerRow;
            if (uint32_t(r) < t.half.m_valid && uint32_t(c * 8) < t.half.n_valid) {
                typename Elem16<E>::vec8 o;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const char* at = smem + r * (BN * 4) + (((2 * c + h) ^ (r & 15)) << 4);
                    const f32x4 a = *reinterpret_cast<const f32x4*>(at), b = *reinterpret_cast<const f32x4*>(at + G::kSmemBytes);
#pragma unroll
                    for (int j = 0; j < 4; ++j) o[4 * h + j] = static_cast<E>(activate<ACT, E>(a[j] + b[j] + float(bias[4 * h + j])));
                }
                constexpr int kAgentScope = 16;   // sc1: written through the L2, like every output row
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), coherent_rows(t.half.c_base),
                                                       int((size_t(r) * t.half.ldc + c * 8) * sizeof(E)), 0, kAgentScope);
            }
        }
        __syncthreads();   // the next tile's loads land in these stages
    }
};

// ------------------------------------------------------------------------------------------------
// 32-bit Elements (fp32, tf32), fp32 matrix cores: the tile of Gemm16 with 4-byte Elements. K is walked
// in slices of 32 values (128-byte rows, the same swizzle) through a ring of STAGES stages that direct
// loads fill STAGES-1 slices ahead, and the tile is split into begin() / mainloop() / finish() for the
// same persistent loop. One matrix instruction (32x32x2) takes two values of K, one from either half of
// the wavefront; a lane reads four consecutive values of its row at once and feeds them to four
// instructions, so instruction j of a group of eight values adds K values 8 g + j and 8 g + 4 + j.
//
// What bounds it: the fp32 matrix rate (157 TFLOP/s nominal, 256 operations a clock and CU), sixteen
// times below the bf16 rate. A 64 x 64 tile then needs only 16 bytes a clock through the CU's load
// path and leaves the path half idle, so the tile is kept small for the sake of the tile counts: two
// workgroups of four wavefronts on a CU, each in its own phase, cover each other's barriers.
// Measured against the tile before it (slices of 16 values through registers, one at a time, one
// workgroup on a CU): 1 024 tokens, 8 experts top-2, 1 024 x 4 096, fp32: 567 -> 347 us per forward (316 with all
// that has changed since, the matrix cores busy 70 % of the whole launch at 2.26 GHz); 8 192 tokens, 64 experts top-2, 2 048 x 2 048, tf32:
// 4 177 -> 2 729 us; 128 tokens, 8 experts, 256 x 512: 57 -> 44 us.
// With barrier and first reads of a slice inside the last group of the slice before, and its first loads there too, against all of them in
// front of it: that fp32 layer 342.6 -> 333.4; 9 984 tokens, 16 experts top-1, 704 x 7 808, fp32: 2 195 -> 2 115; 1 920, 128 experts top-3, 1 472 x
// 640, tf32: 478 -> 457; 16 layers between 0 and 10 % faster. (Loads a group later: 340, and 415 us where 256 tokens, one expert, 832 x 11 200, tf32
// take 380: a CU that has one workgroup waits for its loads, 412 before.)
// T: float, or tf32_t - then the operands lose their lower 13 mantissa bits on the way into the matrix
// cores and the results are rounded to tf32 Elements.
// ------------------------------------------------------------------------------------------------
template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int STAGES>
struct Gemm32 {
    static_assert(sizeof(T) == 4);
    static constexpr bool kTf32 = std::is_same<T, tf32_t>::value;
    static constexpr int kWaves = WAVES_M * WAVES_N;
    static constexpr int kThreads = kWaves * kWave;
    static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
    static constexpr int TM = WM / 32, TN = WN / 32;
    static constexpr int kSliceK = 32, kGroups = 4;                // values of K per slice; groups of eight of them
    static constexpr int kRowBytes = kSliceK * 4, kRowsPerLoad = 8, kChunks = 8;
    static constexpr int kABytes = BM * kRowBytes, kBBytes = BN * kRowBytes, kStage = kABytes + kBBytes;
    static constexpr int kBiasBytes = BN * 4, kBiasOffset = STAGES * kStage;
    static constexpr int kSmemBytes = STAGES * kStage + 2 * kBiasBytes;
    static constexpr int LA = BM / (kRowsPerLoad * kWaves), LB = BN / (kRowsPerLoad * kWaves);
    static constexpr int kLoadsPerSlice = LA + LB;
    static_assert(WM % 32 == 0 && WN % 32 == 0 && BM % (kRowsPerLoad * kWaves) == 0 && BN % (kRowsPerLoad * kWaves) == 0);
    static_assert(STAGES >= 3 && STAGES <= 5 && (STAGES - 1) * kLoadsPerSlice < 64);
    static_assert(kWaves * 4096 <= kStage, "the epilogue's 32 x 32 blocks must fit one stage");
    static_assert(kBiasBytes <= 1024, "one direct load brings the bias");

    struct Tile {
        const float* pa[LA];
        const float* pb[LB];
        float* c_base;
        uint32_t ldc, m_valid, n_valid, k_tiles, act, k_first;
        int stage0, bias_slot;
    };
    typedef f32x16 Acc[TN][TM];

    static __device__ __forceinline__ int swizzle(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }
    static __device__ __forceinline__ int stage_of(const Tile& t, uint32_t kt) { return (t.stage0 + kt) % STAGES; }
    static __device__ __forceinline__ int last_stage(const Tile& t) { return (t.stage0 + t.k_tiles - 1) % STAGES; }
    static __device__ __forceinline__ int next_stage0(const Tile& t) { return (t.stage0 + t.k_tiles) % STAGES; }

    static __device__ __forceinline__ void issue_slice(const Tile& t, char* smem, uint32_t kt) {
        const uint32_t sa = lds_address(smem) + stage_of(t, kt) * kStage + 1024 * wave_index();
        uint32_t slice = kt + t.k_first;
        slice = slice >= t.k_tiles ? slice - t.k_tiles : slice;
        const uint32_t k0 = slice * kSliceK;
#pragma unroll
        for (int i = 0; i < LA; ++i) direct_load16<false>(t.pa[i] + k0, sa + 1024 * kWaves * i);
#pragma unroll
        for (int i = 0; i < LB; ++i) direct_load16<false>(t.pb[i] + k0, sa + kABytes + 1024 * kWaves * i);
    }

    // As Gemm16::begin: addresses, the bias, the first STAGES-1 slices.
    static __device__ __forceinline__ void begin(Tile& t, const GemmTileArgs<float>& g, int stage0, int bias_slot, char* smem) {
        const uint32_t tid = local_tid();
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const int ld_r = lane / kChunks, ld_p = lane % kChunks;
        if (wave == 0 && lane < kBiasBytes / 16) {
            const uint32_t n = uint32_t(lane) * 4 < g.n_valid ? uint32_t(lane) * 4 : 0u;
            direct_load16<false>(g.bias + n, lds_address(smem) + kBiasOffset + bias_slot * kBiasBytes);
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
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int row = kRowsPerLoad * (wave + kWaves * i) + ld_r;
            const uint32_t r = row < int(g.n_valid) ? row : g.n_valid - 1;
            t.pb[i] = g.b_base + size_t(r) * g.ldb + ((ld_p ^ swizzle(row)) << 2);
        }
        t.c_base = g.c_base; t.ldc = g.ldc;
        t.m_valid = g.m_valid; t.n_valid = g.n_valid; t.k_tiles = g.K / kSliceK;
        t.k_first = g.k_first < t.k_tiles ? g.k_first : 0u;
        t.act = g.act; t.stage0 = stage0; t.bias_slot = bias_slot;
#pragma unroll
        for (int st = 0; st < STAGES - 1; ++st)
            if (uint32_t(st) < t.k_tiles) issue_slice(t, smem, st);
    }

    // This wavefront's loads of slice kt have landed once only those of the slices behind it that are
    // already on their way (STAGES-2, fewer at the end of the tile) are outstanding; behind the barrier
    // that holds for every wavefront, and the stage of slice kt-1 is free.
    static __device__ __forceinline__ void wait_slice(uint32_t later) {
        if (STAGES >= 5 && later >= 3) wait_vmcnt<(STAGES >= 5 ? 3 : 0) * kLoadsPerSlice>();
        else if (STAGES >= 4 && later >= 2) wait_vmcnt<(STAGES >= 4 ? 2 : 0) * kLoadsPerSlice>();
        else if (later >= 1) wait_vmcnt<kLoadsPerSlice>();
        else wait_vmcnt<0>();
        asm volatile("s_barrier" ::: "memory");
    }

    template <typename Hook>
    static __device__ __forceinline__ void mainloop(const Tile& t, Acc& acc, char* smem, Hook&& after_first_barrier) {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        const int wm = wave / WAVES_N, wn = wave % WAVES_N;
        if (rows_absent(t, __builtin_amdgcn_readfirstlane(wave) / WAVES_N)) {
            // none of this wavefront's rows exist: it brings its share of the slices and nothing else
            for (uint32_t kt = 0; kt < t.k_tiles; ++kt) {
                wait_slice(t.k_tiles - 1 - kt);
                if (kt == 0) after_first_barrier();
                if (kt + STAGES - 1 < t.k_tiles) issue_slice(t, smem, kt + STAGES - 1);
            }
            return;
        }
#pragma unroll
        for (int ni = 0; ni < TN; ++ni)
#pragma unroll
            for (int mi = 0; mi < TM; ++mi)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[ni][mi][v] = 0.f;
        const int fr_row = lane & 31, fr_half = lane >> 5;
        const int rx = wm * WM + fr_row, rw = wn * WN + fr_row;
        const int base_x = rx * kRowBytes + ((fr_half ^ swizzle(rx)) << 4);
        const int base_w = kABytes + rw * kRowBytes + ((fr_half ^ swizzle(rw)) << 4);
        f32x4 fw[2][TN], fx[2][TM];
        auto read = [&](const char* st, int g) {
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) fw[g & 1][ni] = __builtin_bit_cast(f32x4, load16(st + (base_w ^ (g << 5)) + ni * 32 * kRowBytes));
#pragma unroll
            for (int mi = 0; mi < TM; ++mi) fx[g & 1][mi] = __builtin_bit_cast(f32x4, load16(st + (base_x ^ (g << 5)) + mi * 32 * kRowBytes));
        };
        // share `part` of this wavefront's loads of slice kt
        constexpr int kShare = (kLoadsPerSlice + kGroups - 1) / kGroups;
        auto request = [&](uint32_t kt, int part) {
            const uint32_t to = lds_address(smem) + stage_of(t, kt) * kStage + 1024 * wave_index();
            uint32_t src = kt + t.k_first;
            src = src >= t.k_tiles ? src - t.k_tiles : src;
            const uint32_t k0 = src * kSliceK;
#pragma unroll
            for (int i = part * kShare; i < (part + 1) * kShare && i < kLoadsPerSlice; ++i) {
                if (i < LA) direct_load16<false>(t.pa[i < LA ? i : 0] + k0, to + 1024 * kWaves * i);
                else direct_load16<false>(t.pb[i < LA ? 0 : i - LA] + k0, to + kABytes + 1024 * kWaves * (i - LA));
            }
        };
        // A slice: behind the first instruction of every group a share of the loads of a later slice, behind
        // them the reads of the next group's fragments, all pinned. (Left alone the compiler reads a group where
        // it is used and waits for it there; and a slice's loads in one run hold up the instructions behind them.)
        // The last group does so for the next slice: its barrier lies behind that group's first instruction and a wait for
        // this slice's last reads, so that the stage is free from there on and takes the first share of slice kt+STAGES. (In front of a
        // slice, barrier and first reads lay open.) LOADS: 2 this slice requests the rest of slice kt+STAGES-1 and the first share of the one behind it,
        // 1 there is none behind it, 0 neither. NEXT: there is a slice kt+1.
        auto slice = [&](uint32_t kt, auto loads_tag, auto next_tag) {
            constexpr int LOADS = decltype(loads_tag)::value;
            constexpr bool NEXT = decltype(next_tag)::value;
            const char* st = smem + stage_of(t, kt) * kStage;
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
#pragma unroll
                    for (int ni = 0; ni < TN; ++ni)
#pragma unroll
                        for (int mi = 0; mi < TM; ++mi)
                            acc[ni][mi] = __builtin_amdgcn_mfma_f32_32x32x2f32(operand(fw[g & 1][ni][j]), operand(fx[g & 1][mi][j]), acc[ni][mi], 0, 0, 0);
                    if (j == 0) {
                        __builtin_amdgcn_sched_barrier(0);
                        if (g + 1 < kGroups) {
                            read(st, g + 1);
                            if constexpr (LOADS > 0) request(kt + STAGES - 1, g + 1);
                        } else if constexpr (NEXT) {
                            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the whole of this slice's last fragments, of which the instruction above took one value each
                            wait_slice(t.k_tiles - 2 - kt);
                            read(smem + stage_of(t, kt + 1) * kStage, 0);
                            if constexpr (LOADS > 1) request(kt + STAGES, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        };
        static_assert(kGroups % 2 == 0 && STAGES > 2);
        using Zero = std::integral_constant<int, 0>;
        wait_slice(t.k_tiles - 1);
        after_first_barrier();
        read(smem + stage_of(t, 0) * kStage, 0);
        const uint32_t ahead = t.k_tiles >= uint32_t(STAGES) ? t.k_tiles - STAGES : 0u;   // slices with LOADS 2
        uint32_t kt = 0;
        if (t.k_tiles >= uint32_t(STAGES)) {
            request(STAGES - 1, 0);
            for (; kt < ahead; ++kt) slice(kt, std::integral_constant<int, 2>{}, std::true_type{});
            slice(kt++, std::integral_constant<int, 1>{}, std::true_type{});
        }
        for (; kt + 1 < t.k_tiles; ++kt) slice(kt, Zero{}, std::true_type{});
        slice(kt, Zero{}, std::false_type{});
    }

    // (one value where an instruction takes it: a whole fragment where it is read would wait for the read there)
    static __device__ __forceinline__ float operand(float v) {
        if constexpr (kTf32) v = __uint_as_float(__float_as_uint(v) & 0xffffe000u);
        return v;
    }
    static __device__ __forceinline__ f32x4 operand(u32x4 v) {
        if constexpr (kTf32) v &= u32x4{0xffffe000u, 0xffffe000u, 0xffffe000u, 0xffffe000u};
        return __builtin_bit_cast(f32x4, v);
    }
    static __device__ __forceinline__ bool rows_absent(const Tile& t, int wm) { return uint32_t(wm * WM) >= t.m_valid; }

    // Bias, activation, the rounding of tf32, and the rows written through the L2. A wavefront transposes
    // its 32 x 32 blocks through 4 KB of its own in the stage of the last slice, so that the stores cover
    // whole 128-byte lines. Every wavefront must have left mainloop().
    static __device__ __forceinline__ void finish(const Tile& t, Acc& acc, char* smem) {
        if (rows_absent(t, __builtin_amdgcn_readfirstlane(int(local_tid() >> 6)) / WAVES_N)) return;
        if (t.act == 0) finish_act<0>(t, acc, smem);
        else if (t.act == 1) finish_act<1>(t, acc, smem);
        else finish_act<2>(t, acc, smem);
    }
    template <int ACT>
    static __device__ __forceinline__ void finish_act(const Tile& t, Acc& acc, char* smem) {
        const uint32_t tid = local_tid();
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const int wm = wave / WAVES_N, wn = wave % WAVES_N;
        const int fr_row = lane & 31, fr_half = lane >> 5;
        char* stg = smem + last_stage(t) * kStage + wave * 4096;
        const char* bias = smem + kBiasOffset + t.bias_slot * kBiasBytes + (wn * WN + 4 * fr_half) * 4;
#pragma unroll
        for (int mi = 0; mi < TM; ++mi)
#pragma unroll
            for (int ni = 0; ni < TN; ++ni) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 b4 = *reinterpret_cast<const f32x4*>(bias + (ni * 32 + 8 * q) * 4);
                    f32x4 v;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        v[j] = activate<ACT, T>(acc[ni][mi][4 * q + j] + b4[j]);
                        if constexpr (kTf32) v[j] = tf32_round(v[j]);
                    }
                    *reinterpret_cast<f32x4*>(stg + fr_row * 128 + (((2 * q + fr_half) ^ ((fr_row >> 1) & 7)) << 4)) = v;
                }
                // (the wavefront that wrote the block reads it: its LDS operations complete in order)
#pragma unroll
                for (int it = 0; it < 4; ++it) {
                    const int id = it * kWave + lane, r = id >> 3, c = id & 7;
                    const u32x4 v = load16(stg + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
                    const uint32_t m = wm * WM + mi * 32 + r, n = wn * WN + ni * 32 + c * 4;
                    constexpr int kAgentScope = 16;   // sc1
                    if (m < t.m_valid && n < t.n_valid)
                        __builtin_amdgcn_raw_buffer_store_b128(v, coherent_rows(t.c_base), int((size_t(m) * t.ldc + n) * 4), 0, kAgentScope);
                }
            }
    }
};

// ------------------------------------------------------------------------------------------------
// 32-bit Elements, layers too small for 64 x 64 tiles: a 32 x 32 tile of which each of the four wavefronts works
// on every fourth K slice, on two stages of LDS of its own, without a barrier in between; the four sums are added
// in the epilogue, in order. What bounds such a layer is the chain of one tile: with 64 x 64 the 512 values of K of a
// down-projection take 7.5 us of matrix instructions on a quarter of the CUs, here 1.9 on four times as many. A CU
// that is kept busy loads more than it multiplies (256 bytes a value of K against 8 clocks), which is why larger
// layers keep the larger tile. (128 tokens, 8 experts top-2, 256 x 512, fp32: 41 -> 33 us per forward.)
// ------------------------------------------------------------------------------------------------
template <typename T>
struct Gemm32Wave {
    typedef Gemm32<T, 64, 64, 2, 2, 4> Base;   // operand conversion, swizzle
    static constexpr int BM = 32, BN = 32, kWaves = 4, kThreads = kWaves * kWave;
    static constexpr int kSliceK = 32, kGroups = 4, kRowBytes = 128;
    static constexpr int kOperand = 32 * kRowBytes, kStage = 2 * kOperand, kLoads = 4;   // direct loads per operand and slice
    static constexpr int kBiasBytes = BN * 4, kBiasOffset = kWaves * 2 * kStage;
    static constexpr int kSmemBytes = kBiasOffset + 2 * kBiasBytes;

    struct Tile {
        const float* pa[kLoads];
        const float* pb[kLoads];
        float* c_base;
        uint32_t ldc, m_valid, n_valid, slices, act;   // slices: this wavefront's
        int bias_slot;
    };
    typedef f32x16 Acc;

    static __device__ __forceinline__ int next_stage0(const Tile&) { return 0; }
    // this wavefront's i-th slice: slice 4 i + wavefront of K, into its stage i % 2
    static __device__ __forceinline__ void issue_slice(const Tile& t, char* smem, uint32_t i) {
        const uint32_t at = lds_address(smem) + (2 * wave_index() + (i & 1u)) * kStage;
        const uint32_t k0 = (i * kWaves + wave_index()) * kSliceK;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) direct_load16<false>(t.pa[j] + k0, at + 1024 * j);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) direct_load16<false>(t.pb[j] + k0, at + kOperand + 1024 * j);
    }

    static __device__ __forceinline__ void begin(Tile& t, const GemmTileArgs<float>& g, int, int bias_slot, char* smem) {
        const uint32_t tid = local_tid();
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const int ld_r = lane >> 3, ld_p = lane & 7;
        if (wave == 0 && lane < kBiasBytes / 16) {
            const uint32_t n = uint32_t(lane) * 4 < g.n_valid ? uint32_t(lane) * 4 : 0u;
            direct_load16<false>(g.bias + n, lds_address(smem) + kBiasOffset + bias_slot * kBiasBytes);
        }
        uint32_t src[kLoads];
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const uint32_t row = 8 * i + ld_r;
            src[i] = row < g.m_valid ? row : g.m_valid - 1;
        }
        if (g.a_row_index) {
#pragma unroll
            for (int i = 0; i < kLoads; ++i) src[i] = uint32_t(load_coherent(g.a_row_index + src[i]));
#pragma unroll
            for (int i = 0; i < kLoads; ++i) src[i] = src[i] < g.a_rows ? src[i] : g.a_rows - 1;
        }
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const uint32_t row = 8 * i + ld_r, n = row < g.n_valid ? row : g.n_valid - 1;
            const float* from = g.a_base + size_t(src[i]) * g.lda;
            if (g.a_pad && row >= g.m_valid) from = g.a_pad;
            t.pa[i] = from + ((ld_p ^ Base::swizzle(row)) << 2);
            t.pb[i] = g.b_base + size_t(n) * g.ldb + ((ld_p ^ Base::swizzle(row)) << 2);
        }
        const uint32_t k_tiles = g.K / kSliceK;
        t.c_base = g.c_base; t.ldc = g.ldc; t.m_valid = g.m_valid; t.n_valid = g.n_valid; t.act = g.act; t.bias_slot = bias_slot;
        t.slices = k_tiles > uint32_t(wave) ? (k_tiles - wave + kWaves - 1) / kWaves : 0u;
        if (t.slices > 0) issue_slice(t, smem, 0);
        if (t.slices > 1) issue_slice(t, smem, 1);
    }

    template <typename Hook>
    static __device__ __forceinline__ void mainloop(const Tile& t, Acc& acc, char* smem, Hook&& after_first_barrier) {
        const int lane = threadIdx.x & 63;
        const int fr_row = lane & 31, fr_half = lane >> 5;
        const int base = fr_row * kRowBytes + ((fr_half ^ Base::swizzle(fr_row)) << 4);
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.f;
        auto landed = [&](uint32_t i) {   // slice i, and everything this wavefront issued before it
            if (i + 1 < t.slices) wait_vmcnt<2 * kLoads>();
            else wait_vmcnt<0>();
        };
        landed(0);
        asm volatile("s_barrier" ::: "memory");
        after_first_barrier();
        for (uint32_t i = 0; i < t.slices; ++i) {
            if (i != 0) {
                landed(i);
                asm volatile("" ::: "memory");
            }
            const char* st = smem + (2 * wave_index() + (i & 1u)) * kStage;
            f32x4 fx[kGroups], fw[kGroups];
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
                fx[g] = Base::operand(load16(st + (base ^ (g << 5))));
                fw[g] = Base::operand(load16(st + kOperand + (base ^ (g << 5))));
            }
            // the fragments are in registers: the stage is free for the slice after the next
            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
            if (i + 2 < t.slices) issue_slice(t, smem, i + 2);
#pragma unroll
            for (int g = 0; g < kGroups; ++g)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fw[g][j], fx[g][j], acc, 0, 0, 0);
        }
    }

    // Every wavefront must have left mainloop(), and takes part in the two barriers.
    static __device__ __forceinline__ void finish(const Tile& t, Acc& acc, char* smem) {
        if (t.act == 0) finish_act<0>(t, acc, smem);
        else if (t.act == 1) finish_act<1>(t, acc, smem);
        else finish_act<2>(t, acc, smem);
    }
    template <int ACT>
    static __device__ __forceinline__ void finish_act(const Tile& t, Acc& acc, char* smem) {
        const uint32_t tid = local_tid();
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const int fr_row = lane & 31, fr_half = lane >> 5;
        char* sums = smem + 2 * wave * kStage;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(sums + fr_row * 128 + (((2 * q + fr_half) ^ ((fr_row >> 1) & 7)) << 4)) =
                f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
        __syncthreads();
        const uint32_t r = tid >> 3, c = tid & 7;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kWaves; ++w) v += *reinterpret_cast<const f32x4*>(smem + 2 * w * kStage + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
        v += *reinterpret_cast<const f32x4*>(smem + kBiasOffset + t.bias_slot * kBiasBytes + c * 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = activate<ACT, T>(v[j]);
            if constexpr (Base::kTf32) v[j] = tf32_round(v[j]);
        }
        constexpr int kAgentScope = 16;   // sc1
        if (r < t.m_valid && c * 4 < t.n_valid)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), coherent_rows(t.c_base), int((size_t(r) * t.ldc + c * 4) * 4), 0, kAgentScope);
        __syncthreads();   // the next tile's loads land in these stages
    }
};

}  // namespace kleos_amd
