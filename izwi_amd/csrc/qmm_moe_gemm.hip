// Expert MLP of many sorted pairs per expert, Q4_K stacks: matrix products whose k runs through the
// 6-bit scales inside the int8 matrix instruction.
//
// A sub-block's dot needs its scale, so a kernel that multiplies nibbles has to multiply every result
// of every matrix instruction by a scale: eight integer multiply-adds per output value and 256 k (the
// 16-row-tile kernels of qmm_gemv_mfma.hip, bound by exactly that).  Here the scale goes into the
// weight operand before the product: sc = 8 hi + lo with three bits each, quant * lo and quant * hi are
// at most 105 and fit the int8 operand, four bytes take one packed 16-bit multiply.  A unit of 256 k is
// then two running integer sums (lo, hi) over eight v_mfma_i32_32x32x32_i8 each; per output value and
// unit there remain one shift-add, one conversion and three multiply-adds.  Twice the matrix
// instructions, a fourth of the vector instructions.  The min term is one v_mfma_f32_32x32x16_f16 per unit:
// mins (m, 32 m) against the sub-block sums split in two (sum = 32 hi + lo), exact in f16 and
// below 2^24 in its f32 sum.  The same integers and the same f32 operations in the same order as
// q4k_panel_dot: the same bits.
//
// A work item is up to 64 sorted pairs (two blocks of 32) of one expert and, of every one of eight waves, two blocks of 32
// weight rows: gate and up of the same 32 columns, or two blocks of down.  A workgroup per compute unit takes its items in turn.
// The pairs' activation records pass through a ring of four units in LDS, requested two steps (units) ahead and on into the next
// item, the weights of a wave one unit ahead in its registers, so that between items only the finish of the sums stands still.  No
// barrier in between: the waves of a SIMD run half a phase apart, and a barrier would bring them together; counters in LDS say which
// steps have landed and which slots are free.  One wave of eight requests all of a step's records in its turn.
//
// gate | up: the 256 columns of a workgroup are one unit of the down projection's input, so
// silu(gate) * up is quantized here, in LDS, and leaves as records: 9.5 bytes instead of 64 per eight
// values, no launch in between.
//
// Bound by the issue of vector instructions, 640 per unit and wave (320 of them the finish of the sums, 300 the unpacking, which two
// blocks of pairs share) beside 68 matrix instructions: a SIMD with two waves issues one in 4.4 to 4.9 cycles, which makes 6900 of the
// 7250 cycles that a unit takes; and by the clock, which falls to 1.45 to 1.75 GHz under it.  (A start of the items with the long ones
// first at every size, 3 % fewer cycles at the end of a launch, was therefore no faster.)
// 128 experts, top-8, 2048 x 768, layer: items as workgroups of their own, each with its records over all of k, 7 to 8 of 42 us of
// a gate | up item and 7 of 18 of a down item before the first unit was done / now: 108 / 102 us at 256 tokens, 133 / 124 at 512,
// 185 / 169 at 1024, 281 / 265 at 2048, 498 / 471 at 4096, where 32 % of gate | up's cycles and 39 % of down's still pass outside the units
// (finish, exchange of silu(gate) * up, stores, the last round).  Each wave requesting its share of every step's records instead of
// one in turn: 8200 cycles a unit, 486 us at 4096 when the one in turn took 471.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>

#include "qmm_internal.h"
#include "qmm_moe_route.h"
#include "qmm_records.h"
#include "qmm_tile.h"

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr uint32_t kNib = 0x0f0f0f0fu;
constexpr int kWaves = 8, kRows = QMM_MOE_CHUNK_ROWS;
constexpr int kMaxUnits = 8;
// LDS image of a unit: [2 halves][64 rows][128 B of quants] | [64 rows][32 B of sums] | [64] scales.
// Chunk c of a row's 128 bytes sits at position c ^ ((row >> 1) & 7), half h of its sums at
// h ^ ((row >> 3) & 1): sixteen lanes that read one chunk of sixteen rows touch every bank once.
constexpr int kSumsAt = 2 * kRows * 128, kScalesAt = kSumsAt + kRows * 32, kUnitLds = kScalesAt + kRows * 4;
static_assert(kUnitLds % 128 == 0);
constexpr int kHStride = 264; // floats per row of silu(gate) * up in LDS
constexpr int kRing = 4, kAhead = 2; // units of records in LDS, and how many steps ahead of its use one is requested
// Items whose rows are known, and how many items ahead.  A wave that enters item i writes the table of item i + kTablesAhead; with one
// unit per item the slowest wave may then still store item i - kRing - 1 (it has counted that step as done), so the tables reach
// further than from there to here: eight of them did not (an item's rows could go where a later item's belong).
constexpr int kTables = 16, kTablesAhead = 4;
static_assert(kTables >= kTablesAhead + kRing + 2 && (kTables & (kTables - 1)) == 0);
// s_waitcnt vmcnt(n), n < 16, the other counters left alone
constexpr int wait_vector(int n) { return 0x0f70 | n; }

struct MoeGemmParams {
    const uint8_t *w0, *w1;   // gate, up; down: the stack twice
    const uint8_t* records;   // wide row records, `row_bytes` per source row
    void* out;                // gate | up: wide row records by sorted position; down: f32 [pair][n]
    const int32_t* perm;      // sorted position -> pair
    const int32_t* offsets;   // sorted positions of expert e: [offsets[e], offsets[e + 1])
    const int32_t* chunks;    // its chunks of 64 positions: [chunks[e], chunks[e + 1])
    const int32_t* chunk_expert;
    int64_t matrix_bytes;
    uint32_t row_bytes;
    uint32_t row_magic;       // source row of a pair = pair / row_div by multiplication; row_div 0: the position itself
    int row_div;
    uint32_t zero_row;        // a source row of zeros
    int n_experts, parts, n, row_tiles, k_units, k_groups, s, slots, panel_bytes;
    int out_units;
    int fill2; // long items first: twice the short items asked for per place of the last round
};

__device__ __forceinline__ void barrier_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// Counters in LDS between the waves of a workgroup.  A wave's LDS instructions run in their order, so what it read or wrote
// before it counts is read or written; the asm keeps the compiler to that order.
// (One lane adds, without a branch: a block that ends between a unit's products and its sums costs registers.)
__device__ __forceinline__ void count_up(uint32_t* counter) {
    uint64_t all;
    asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, 1\n\tds_add_u32 %1, %2\n\ts_mov_b64 exec, %0"
                 : "=&s"(all)
                 : "v"((uint32_t)(uintptr_t)counter), "v"(1u)
                 : "memory");
}
__device__ __forceinline__ void wait_for(const uint32_t* counter, uint32_t at_least) {
    while (__builtin_amdgcn_readfirstlane(__hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) < at_least)
        __builtin_amdgcn_s_sleep(1);
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ i32x4 lds_i32x4(uint32_t at) { return *reinterpret_cast<const __attribute__((address_space(3))) i32x4*>(at); }
// The lane's number, worked out anew: what depends on it is not kept in registers over the loops.
__device__ __forceinline__ int lane_here(int lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}

// What a lane holds of its weight row's unit: the header and, of every chunk pair b, chunk 2b + h.
struct UnitRegs {
    u32x4 hdr, q[4];
};

// bytes of w (at most 15 each) times the 16-bit half `I` of `digits` (at most 7)
template <int I>
__device__ __forceinline__ uint32_t times(uint32_t w, uint32_t digits) {
    const u16x2 d = __builtin_bit_cast(u16x2, digits);
    const u16x2 dd = {d[I], d[I]};
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, w) * dd));
}

// Two bytes of `m` as the f16 pair c * byte (1024 + byte as bits, then one exact fma; c is 1 or 32).
template <int SEL>
__device__ __forceinline__ f16x2 mins_pair(uint32_t m, f16x2 c, f16x2 minus_1024_c) {
    constexpr uint32_t sel = SEL ? 0x04030402u : 0x04010400u; // bytes: 0x64, m[hi], 0x64, m[lo]
    const f16x2 v = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, m, sel));
    return __builtin_elementwise_fma(v, c, minus_1024_c);
}

constexpr int kCusPerXcd = 32;
constexpr int kOrderedItems = 4 * kCusPerXcd; // the longest run of an XCD's items that is put in order

struct WorkItem {
    int e, part, pos_begin, pos_end;
};

// What the waves of a workgroup share beside the records: counters that only grow, and the tables of the items.
struct Shared {
    uint32_t ready[kRing];  // steps whose records have landed in a slot
    uint32_t done[kRing];   // waves that have read them
    uint32_t h_written, h_read; // gate | up: waves that have written (read) silu(gate) * up of an item
    uint32_t pad[2];
    uint32_t known[kTables]; // 1 + the item whose table stands there
    WorkItem items[kTables];
    uint32_t src_off[kTables][kRows]; // byte offsets of the rows' records
    uint32_t out_off[kTables][kRows]; // down: of the output rows
    uint8_t order[kOrderedItems];     // ORDERED: this run's items, long ones first
};

// A wave's place in the stream of (item, unit) steps
struct Stream {
    int n_items;              // of this workgroup
    int step;                 // being multiplied
    int l_step, l_item, l_unit; // whose records are requested next
    const uint8_t* wp[2];     // the panels of the wave's first row tile: gate and up, or two blocks of down
    uint32_t unit_off;        // of the unit to request: panel, then unit in the panel
    int in_panel;
};

__device__ __forceinline__ WorkItem uniform_item(const Shared& S, int j) {
    const WorkItem& it = S.items[j & (kTables - 1)];
    return {__builtin_amdgcn_readfirstlane(it.e), __builtin_amdgcn_readfirstlane(it.part), __builtin_amdgcn_readfirstlane(it.pos_begin),
            __builtin_amdgcn_readfirstlane(it.pos_end)};
}

template <bool GATE_UP>
__device__ __forceinline__ void first_panels(const MoeGemmParams& P, const WorkItem& it, int wave, const uint8_t* (&wp)[2]) {
    const int64_t matrix = (int64_t)it.e * P.matrix_bytes;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int rt = (GATE_UP ? it.part * 16 : it.part * 32 + c * 16) + wave * 2; // (a block past the end: multiplied, not stored)
        wp[c] = (c ? P.w1 : P.w0) + matrix + (uint32_t)(min(rt, P.row_tiles - 2) * P.k_groups) * (uint32_t)P.panel_bytes;
    }
}

__device__ __forceinline__ void request_unit(UnitRegs& w, const uint8_t* unit, uint32_t lane_off, uint32_t half_off, uint32_t slots16) {
    w.hdr = *reinterpret_cast<const u32x4*>(unit + lane_off);
#pragma unroll
    for (int b = 0; b < 4; b++) w.q[b] = *reinterpret_cast<const u32x4*>(unit + (uint32_t)(1 + 2 * b) * slots16 + half_off);
}

// The next step's records into their LDS image, all of them by the wave whose turn it is (shared out, the instructions around the
// loads are issued eight times).
__device__ __forceinline__ void request_records(const MoeGemmParams& P, Stream& t, Shared& S, uint8_t* smem, int wave, int lane) {
    if (t.l_item >= t.n_items) return; // uniform
    if ((t.l_step & (kWaves - 1)) == wave) {
        lane = lane_here(lane);
        const int slot = t.l_step & (kRing - 1), table = t.l_item & (kTables - 1);
        wait_for(&S.known[table], (uint32_t)t.l_item + 1);
        wait_for(&S.done[slot], (uint32_t)(t.l_step / kRing) * kWaves);
        const int groups = __builtin_amdgcn_readfirstlane(S.items[table].pos_end - S.items[table].pos_begin) > 32 ? 8 : 4;
        const uint32_t unit_lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem + (uint32_t)slot * kUnitLds);
        const uint8_t* base = P.records + t.l_unit * kWideRowUnitBytes;
        const uint32_t* src = S.src_off[table];
#pragma unroll 1
        for (int g = 0; g < groups; g++) { // eight rows: both halves of the quants
            const int r = g * 8 + (lane >> 3);
            const uint32_t from = src[r] + (uint32_t)((lane & 7) ^ ((r >> 1) & 7)) * 16u;
            load_to_lds(base, from, unit_lds + g * 1024);
            load_to_lds(base, from + 128u, unit_lds + kRows * 128 + g * 1024);
        }
#pragma unroll 1
        for (int q = 0; q < groups / 4; q++) { // 32 rows: their sums
            const int r = q * 32 + (lane >> 1);
            load_to_lds(base, src[r] + 256u + (uint32_t)((lane & 1) ^ ((r >> 3) & 1)) * 16u, unit_lds + kSumsAt + q * 1024);
        }
        load_to_lds4(base, src[lane] + 288u, unit_lds + kScalesAt);
    }
    t.l_step++;
    if (++t.l_unit == P.k_units) t.l_unit = 0, t.l_item++;
}

template <bool GATE_UP, int NRB>
__device__ __forceinline__ void chunk_body(const MoeGemmParams& P, Shared& S, Stream& t, uint8_t* smem, UnitRegs (&raw)[2], int item,
                                           const WorkItem& it, int wave, int lane) {
    const int row = lane & 31, h = lane >> 5;
    // byte offsets of the lane's A chunks, of its sums, and of its four runs of scales
    // (the four chunks' differ in bits that the swizzle leaves apart, and images start on 128 bytes)
    const uint32_t a_off = (uint32_t)row * 128u + (((uint32_t)(2 * h)) ^ ((uint32_t)(row >> 1) & 7u)) * 16u;
    const uint32_t sum_off = (uint32_t)kSumsAt + (uint32_t)row * 32u + (((uint32_t)h ^ ((uint32_t)(row >> 3) & 1u)) * 16u);
    const uint32_t scale_off = (uint32_t)kScalesAt + (uint32_t)h * 16u;
    const _Float16 cf = h ? (_Float16)32.0f : (_Float16)1.0f, kf = h ? (_Float16)-32768.0f : (_Float16)-1024.0f;
    const f16x2 c2 = {cf, cf}, k2 = {kf, kf};
    const uint32_t slots16 = (uint32_t)P.slots * 16u;
    const uint32_t lane_off = (uint32_t)((lane >> 4) & 1) * (uint32_t)P.k_groups * (uint32_t)P.panel_bytes + (uint32_t)(lane & 15) * 16u;
    const uint32_t half_off = lane_off + (uint32_t)h * slots16;

    f32x16 acc[2][NRB];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int rb = 0; rb < NRB; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[c][rb][r] = 0.0f;

    for (int u = 0; u < P.k_units; u++) {
        // (known to be the same in all lanes)
        t.step = __builtin_amdgcn_readfirstlane(t.step);
        t.l_step = __builtin_amdgcn_readfirstlane(t.l_step), t.l_item = __builtin_amdgcn_readfirstlane(t.l_item);
        t.l_unit = __builtin_amdgcn_readfirstlane(t.l_unit);
        t.unit_off = __builtin_amdgcn_readfirstlane(t.unit_off), t.in_panel = __builtin_amdgcn_readfirstlane(t.in_panel);
        // Behind the records that this wave requested at the last step came ten loads of weights, so with five left open they have
        // landed.  (The builtin also tells the compiler, which otherwise waited for all of the weights here.)
        __builtin_amdgcn_s_waitcnt(wait_vector(5));
        if (((t.step + kAhead - 1) & (kWaves - 1)) == wave) count_up(&S.ready[(t.step + kAhead - 1) & (kRing - 1)]);
        // the weights to request next: the following unit's, or the first of the next item (of the last: the same again)
        if (u + 1 < P.k_units) {
            if (++t.in_panel == P.s) t.in_panel = 0, t.unit_off += (uint32_t)P.panel_bytes - (uint32_t)(P.s - 1) * 256u;
            else t.unit_off += 256u;
        } else if (item + 1 < t.n_items) {
            wait_for(&S.known[(item + 1) & (kTables - 1)], (uint32_t)item + 2);
            first_panels<GATE_UP>(P, uniform_item(S, item + 1), wave, t.wp);
            t.unit_off = 0, t.in_panel = 0;
        }
        request_records(P, t, S, smem, wave, lane);
        const int slot = t.step & (kRing - 1);
        const uint8_t* lds = smem + slot * kUnitLds;
        const uint32_t a_at = (uint32_t)(uintptr_t)lds + a_off;
        wait_for(&S.ready[slot], (uint32_t)(t.step / kRing + 1));
#pragma unroll
        for (int c = 0; c < 2; c++) {
            // (a wave in its matrix instructions goes before the other one of its SIMD in its finish)
            __builtin_amdgcn_s_setprio(1);
            UnitRegs& w = raw[c];
            const u32x4 hdr = w.hdr;
            const uint32_t sc[2] = {hdr.y & 0x3f3f3f3fu, (hdr.w & 0x0f0f0f0fu) | (((hdr.y >> 6) & 0x03030303u) << 4)};
            // digits of the scales as 16-bit pairs: [dword][sub-block parity], sub-blocks 4 d + {0, 2} + parity
            uint32_t lo_d[2][2], hi_d[2][2];
#pragma unroll
            for (int d = 0; d < 2; d++) {
                lo_d[d][0] = sc[d] & 0x00070007u, lo_d[d][1] = (sc[d] >> 8) & 0x00070007u;
                hi_d[d][0] = (sc[d] >> 3) & 0x00070007u, hi_d[d][1] = (sc[d] >> 11) & 0x00070007u;
            }
            i32x16 lo[NRB], hi[NRB];
#pragma unroll
            for (int b = 0; b < 4; b++) {
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t w0 = w.q[b][2 * i], w1 = w.q[b][2 * i + 1];
                    const uint32_t n0 = w0 & kNib, n1 = w1 & kNib, m0 = (w0 >> 4) & kNib, m1 = (w1 >> 4) & kNib;
                    const uint32_t le = lo_d[b >> 1][0], lod = lo_d[b >> 1][1], he = hi_d[b >> 1][0], ho = hi_d[b >> 1][1];
                    u32x4 wl, wh;
                    if (b & 1) {
                        wl = u32x4{times<1>(n0, le), times<1>(n1, le), times<1>(m0, lod), times<1>(m1, lod)};
                        wh = u32x4{times<1>(n0, he), times<1>(n1, he), times<1>(m0, ho), times<1>(m1, ho)};
                    } else {
                        wl = u32x4{times<0>(n0, le), times<0>(n1, le), times<0>(m0, lod), times<0>(m1, lod)};
                        wh = u32x4{times<0>(n0, he), times<0>(n1, he), times<0>(m0, ho), times<0>(m1, ho)};
                    }
#pragma unroll
                    for (int rb = 0; rb < NRB; rb++) {
                        const i32x4 a = lds_i32x4((a_at ^ (uint32_t)(64 * (b & 1) + 16 * i)) + (b >> 1) * (kRows * 128) + rb * 4096);
                        if (b == 0 && i == 0) {
                            lo[rb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, __builtin_bit_cast(i32x4, wl), i32x16{}, 0, 0, 0);
                            hi[rb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, __builtin_bit_cast(i32x4, wh), i32x16{}, 0, 0, 0);
                        } else {
                            lo[rb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, __builtin_bit_cast(i32x4, wl), lo[rb], 0, 0, 0);
                            hi[rb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, __builtin_bit_cast(i32x4, wh), hi[rb], 0, 0, 0);
                        }
                    }
                }
            }
            float d = qmm_f16_bits_to_f32((uint16_t)(hdr.x & 0xffffu));
            float dmin = qmm_f16_bits_to_f32((uint16_t)(hdr.x >> 16));
            const uint32_t mn_lo = hdr.z & 0x3f3f3f3fu;
            const uint32_t mn_hi = ((hdr.w >> 4) & 0x0f0f0f0fu) | (((hdr.z >> 6) & 0x03030303u) << 4);
            const f16x2 mm[4] = {mins_pair<0>(mn_lo, c2, k2), mins_pair<1>(mn_lo, c2, k2), mins_pair<0>(mn_hi, c2, k2), mins_pair<1>(mn_hi, c2, k2)};
            const f16x8 mins = {mm[0][0], mm[0][1], mm[1][0], mm[1][1], mm[2][0], mm[2][1], mm[3][0], mm[3][1]};
            // What the finish reads from LDS, and the min term, behind the last products: their latencies run under those.
            f32x16 msum[NRB];
            f32x4 dx[4];
#pragma unroll
            for (int rb = 0; rb < NRB; rb++) {
                const f16x8 sums = *reinterpret_cast<const f16x8*>(lds + sum_off + rb * 1024);
                msum[rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, mins, f32x16{}, 0, 0, 0);
            }
#pragma unroll
            for (int g = 0; g < 4; g++) dx[g] = *reinterpret_cast<const f32x4*>(lds + scale_off + g * 32);
            asm volatile("" : "+v"(d), "+v"(dmin)); // (computed here, so that the header's registers are free)
            __builtin_amdgcn_s_setprio(0);
            // the unit is consumed: the next one into its registers (the fences keep the scheduler from
            // gathering the loads of both columns at the loop's end, where nothing is left to cover them)
            __builtin_amdgcn_sched_barrier(0);
            request_unit(w, t.wp[c] + t.unit_off, lane_off, half_off, slots16);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rb = 0; rb < NRB; rb++) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int isum = (hi[rb][r] << 3) + lo[rb][r];
                    acc[c][rb][r] = fmaf(fmaf(-dmin, msum[rb][r], d * (float)isum), dx[r >> 2][r & 3], acc[c][rb][r]);
                    if (rb + 1 < NRB && (r & 3) == 3) dx[r >> 2] = *reinterpret_cast<const f32x4*>(lds + scale_off + (rb + 1) * 128 + (r >> 2) * 32);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        count_up(&S.done[slot]);
        t.step++;
    }

    lane = lane_here(lane);
    const int h_ = lane >> 5, col = wave * 32 + (lane & 31);
    if constexpr (GATE_UP) {
        float* hbuf = reinterpret_cast<float*>(smem + kRing * kUnitLds);
#pragma unroll
        for (int rb = 0; rb < NRB; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[0][rb][r] = qmm_silu(acc[0][rb][r]) * acc[1][rb][r];
        // (the next item's weights have landed; the compiler, told so, does not wait for the stores behind at the top of the loop)
        __builtin_amdgcn_s_waitcnt(wait_vector(0));
        wait_for(&S.h_read, (uint32_t)item * kWaves); // the last item's
#pragma unroll
        for (int rb = 0; rb < NRB; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                hbuf[(rb * 32 + (r & 3) + 8 * (r >> 2) + 4 * h_) * kHStride + col] = acc[0][rb][r];
        count_up(&S.h_written);
        wait_for(&S.h_written, (uint32_t)(item + 1) * kWaves);
        const int j = lane & 15;
#pragma unroll
        for (int pass = 0; pass < NRB; pass++) {
            const int m = pass * 32 + wave * 4 + (lane >> 4);
            float v[16];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const f32x4 f = *reinterpret_cast<const f32x4*>(hbuf + m * kHStride + 16 * j + 4 * i);
                v[4 * i] = f.x, v[4 * i + 1] = f.y, v[4 * i + 2] = f.z, v[4 * i + 3] = f.w;
            }
            if (pass == NRB - 1) count_up(&S.h_read);
            if (it.pos_begin + m < it.pos_end) // (whole 16-lane groups)
                quantize_into_record<QMM_Q4_K, kWideRowRecord>(
                    v, j, 0, static_cast<uint8_t*>(P.out) + ((int64_t)(it.pos_begin + m) * P.out_units + it.part) * kWideRowUnitBytes);
        }
    } else {
        __builtin_amdgcn_s_waitcnt(wait_vector(0)); // (as above)
        // 32-bit byte offsets from one uniform base; only an expert's last chunk has rows that do not exist
        uint8_t* y = static_cast<uint8_t*>(P.out);
        const uint32_t* out_off = S.out_off[item & (kTables - 1)];
        const bool whole = it.pos_end - it.pos_begin == NRB * 32;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int n = it.part * 512 + c * 256 + col;
            if (n >= P.n) continue; // (uniform: n is a multiple of 256)
#pragma unroll
            for (int rb = 0; rb < NRB; rb++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const u32x4 rows = *reinterpret_cast<const u32x4*>(out_off + rb * 32 + 8 * g + 4 * h_);
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (whole || rb * 32 + 8 * g + 4 * h_ + r < it.pos_end - it.pos_begin)
                            *reinterpret_cast<float*>(y + (rows[r] + (uint32_t)n * 4u)) = acc[c][rb][4 * g + r];
                }
        }
    }
}

__device__ __forceinline__ WorkItem work_item(const MoeGemmParams& P, int item) {
    const int e = P.chunk_expert[item / P.parts]; // (an expert's items begin at parts * its first chunk)
    const int chunk0 = P.chunks[e], n_chunks = P.chunks[e + 1] - chunk0;
    const int local = item - chunk0 * P.parts, part = local / n_chunks, chunk = local - part * n_chunks;
    const int begin = P.offsets[e] + chunk * kRows;
    return {e, part, begin, min(P.offsets[e + 1], begin + kRows)};
}

// A wave leaves the table of this workgroup's item j.
__device__ __forceinline__ void prepare_item(const MoeGemmParams& P, Shared& S, const WorkItem& it, int j, int lane) {
    const int at = j & (kTables - 1);
    lane = lane_here(lane);
    // (A row past the end is one of zeros, its sums are never stored: the matrix instructions take the less power the fewer bits change.
    // With the chunk's first row there instead 108.1 / 105.1 us a layer at 256 tokens, 143.2 / 138.3 at 600, 177.4 / 176.2 at 1024.)
    const bool exists = it.pos_begin + lane < it.pos_end;
    const int pos = exists ? it.pos_begin + lane : it.pos_begin;
    const uint32_t pair = (uint32_t)P.perm[pos];
    const uint32_t src = !exists ? P.zero_row : P.row_div == 0 ? (uint32_t)pos : P.row_div == 1 ? pair : __umulhi(pair, P.row_magic);
    S.src_off[at][lane] = src * P.row_bytes;
    S.out_off[at][lane] = pair * (uint32_t)P.n * 4u;
    if (lane == 0) S.items[at] = it;
    asm volatile("" ::: "memory");
    if (lane == 0) __hip_atomic_store(&S.known[at], (uint32_t)j + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Where the last of an XCD's rounds can hold short items alone, those of more than 32 pairs go first (a lane per item)
// and the short ones fill in behind them.  Leaves the run's order in S.order; one wave.
__device__ __forceinline__ void order_items(const MoeGemmParams& P, Shared& S, int first, int run, int lane) {
    constexpr int kPerLane = (kOrderedItems + 63) / 64;
    uint64_t heavy[kPerLane], exist[kPerLane];
    int heavies = 0;
#pragma unroll
    for (int j = 0; j < kPerLane; j++) {
        const bool exists = 64 * j + lane < run;
        const WorkItem mine = work_item(P, first + (exists ? 64 * j + lane : 0));
        heavy[j] = __ballot(exists && mine.pos_end - mine.pos_begin > 32), exist[j] = __ballot(exists);
        heavies += __popcll(heavy[j]);
    }
    const int lights = run - heavies, last_round = (run - 1) % kCusPerXcd + 1;
    const bool sorted = heavies > 0 && 2 * lights >= P.fill2 * last_round; // uniform, the same in all workgroups of the run
    int at_heavy = 0, at_light = heavies;
#pragma unroll
    for (int j = 0; j < kPerLane; j++) {
        const bool is_heavy = heavy[j] >> lane & 1;
        const uint64_t light = exist[j] & ~heavy[j], set = is_heavy ? heavy[j] : light;
        const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(set >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)set, 0));
        const int rank = sorted ? (is_heavy ? at_heavy : at_light) + below : 64 * j + lane;
        if (exist[j] >> lane & 1) S.order[rank] = (uint8_t)(64 * j + lane);
        at_heavy += __popcll(heavy[j]), at_light += __popcll(light);
    }
}

// A run of two rounds: the second item of a workgroup, -1 if it has none.  Those whose first item is short are done first and are
// first to take one, long ones first.  Places that heed no lengths gave some a long item behind a long one while their neighbours
// were done: layer of 64 experts of 2048 x 1024 at 384 tokens with uneven counts (logits and N(0, 0.4) per expert) 125 us, and 119 with a
// workgroup of its own for every item, which the hardware starts as others end; this way 112.  Even counts 82 / 83 / 82.  With more
// rounds the differences even out.  A lane per item, while the first records are on their way (ahead of them a launch took 1 us more).
__device__ __forceinline__ int second_item(const MoeGemmParams& P, int first, int run, int slot, int lane) {
    const WorkItem mine = work_item(P, first + min(lane, run - 1));
    const uint64_t heavy = __ballot(lane < run && mine.pos_end - mine.pos_begin > 32);
    const uint32_t before = (1u << slot) - 1, long0 = (uint32_t)heavy, long1 = (uint32_t)(heavy >> kCusPerXcd);
    const uint32_t short1 = ~(uint32_t)0 >> (2 * kCusPerXcd - run) & ~long1; // (run > kCusPerXcd)
    const int rank = long0 >> slot & 1 ? __popc(~long0) + __popc(long0 & before) : __popc(~long0 & before), longs = __popc(long1);
    const uint32_t set = rank < longs ? long1 : short1;
    const int nth = rank < longs ? rank : rank - longs;
    const uint64_t at = __ballot(lane < kCusPerXcd && (set >> (lane & 31) & 1) && (int)__builtin_amdgcn_mbcnt_lo(set, 0) == nth);
    return at ? kCusPerXcd + __ffsll((unsigned long long)at) - 1 : -1;
}

template <bool GATE_UP, bool ORDERED>
__global__ __launch_bounds__(64 * kWaves) void moe_gemm_q4k_kernel(MoeGemmParams P) {
    extern __shared__ __attribute__((aligned(128))) uint8_t smem[];
    __shared__ __attribute__((aligned(16))) Shared S;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // Work items in the order (expert, part of the weight rows, chunk of the pairs), cut into eight equal
    // runs: workgroups go to the XCDs round-robin, so a run is one XCD's, and the chunks that read the same weights
    // follow one another there and find them in its L2.  A workgroup takes its items from every round of the run, in turn from
    // its front and its back, of two rounds by their lengths.
    const int items = P.chunks[P.n_experts] * P.parts, per_xcd = (items + 7) >> 3;
    const int slot = (int)(blockIdx.x >> 3), slots = (int)(gridDim.x >> 3), first = (int)(blockIdx.x & 7) * per_xcd;
    const int run = min(per_xcd, items - first); // items of this XCD
    if (slot >= run) return; // uniform
    const auto place = [&](int j) { return j * slots + (j & 1 ? slots - 1 - slot : slot); };
    const bool ordered = ORDERED && run > kCusPerXcd && run <= kOrderedItems; // uniform
    const bool two_rounds = !ORDERED && run > kCusPerXcd && run <= 2 * kCusPerXcd; // uniform
    int second = -1;
    const auto local_item = [&](int j) {
        return ordered ? (int)__builtin_amdgcn_readfirstlane(S.order[place(j)]) : two_rounds && j == 1 ? second : place(j);
    };
    Stream t{};
    t.n_items = __builtin_amdgcn_readfirstlane(run / slots + (place(run / slots) < run));
    if (threadIdx.x < (int)(offsetof(Shared, items) / 4)) reinterpret_cast<uint32_t*>(&S)[threadIdx.x] = 0;
    if (ordered && wave == 0) order_items(P, S, first, run, lane);
    barrier_lds();

    // The first item's weights, the first items' tables, the first steps' records
    const uint32_t slots16 = (uint32_t)P.slots * 16u;
    const uint32_t lane_off = (uint32_t)((lane >> 4) & 1) * (uint32_t)P.k_groups * (uint32_t)P.panel_bytes + (uint32_t)(lane & 15) * 16u;
    first_panels<GATE_UP>(P, work_item(P, first + local_item(0)), wave, t.wp);
    UnitRegs raw[2];
#pragma unroll
    for (int c = 0; c < 2; c++) request_unit(raw[c], t.wp[c], lane_off, lane_off + (uint32_t)(lane >> 5) * slots16, slots16);
    if (wave == 0) prepare_item(P, S, work_item(P, first + local_item(0)), 0, lane);
    static_assert(kAhead == 2);
    request_records(P, t, S, smem, wave, lane);
    if (two_rounds) second = second_item(P, first, run, slot, lane), t.n_items = second < 0 ? 1 : 2;
    if (wave > 0 && wave < kTablesAhead && wave < t.n_items) prepare_item(P, S, work_item(P, first + local_item(wave)), wave, lane);
    request_records(P, t, S, smem, wave, lane);
    __builtin_amdgcn_s_waitcnt(wait_vector(0));
    if (wave == 0) count_up(&S.ready[0]); // (the second step's: at the top of the loop)
    if (wave >= kWaves / 2) __builtin_amdgcn_s_sleep(10); // the two waves of a SIMD half a phase apart
    for (int i = 0; i < t.n_items; i++) {
        if ((i & (kWaves - 1)) == wave && i + kTablesAhead < t.n_items)
            prepare_item(P, S, work_item(P, first + local_item(i + kTablesAhead)), i + kTablesAhead, lane);
        wait_for(&S.known[i & (kTables - 1)], (uint32_t)i + 1);
        const WorkItem it = uniform_item(S, i);
        if (it.pos_end - it.pos_begin > 32) chunk_body<GATE_UP, 2>(P, S, t, smem, raw, i, it, wave, lane);
        else chunk_body<GATE_UP, 1>(P, S, t, smem, raw, i, it, wave, lane);
    }
}

// ---- the activation rows' records, 16 lanes per (row, unit) ----------------------------------
__device__ __forceinline__ void load16(const float* __restrict__ src, float (&v)[16]) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float4 f = reinterpret_cast<const float4*>(src)[i];
        v[4 * i] = f.x, v[4 * i + 1] = f.y, v[4 * i + 2] = f.z, v[4 * i + 3] = f.w;
    }
}
// The rows of zeros behind the records of x and of silu(gate) * up, by one workgroup
struct ZeroRows {
    u32x4* at[2];
    int pieces[2];
};
__device__ __forceinline__ void write_zero_rows(const ZeroRows& Z) {
#pragma unroll
    for (int i = 0; i < 2; i++)
        for (int q = threadIdx.x; q < Z.pieces[i]; q += blockDim.x) Z.at[i][q] = u32x4{0, 0, 0, 0};
}
__global__ void wide_rows_kernel(const float* __restrict__ x, int64_t groups, uint8_t* __restrict__ out, ZeroRows Z) {
    if (blockIdx.x == gridDim.x - 1) return write_zero_rows(Z);
    const int64_t group = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4;
    const int j = threadIdx.x & 15;
    if (group >= groups) return; // whole 16-lane groups leave together
    float v[16];
    load16(x + group * 256 + 16 * j, v);
    quantize_into_record<QMM_Q4_K, kWideRowRecord>(v, j, 0, out + group * kWideRowUnitBytes);
}

// Routing and records of the tokens' rows side by side, as route_rows_kernel in qmm_gemv_mfma.hip.
template <int PER_LANE>
__global__ void route_wide_rows_kernel(const float* __restrict__ logits, int64_t t, int n_experts, int top_k,
                                       int32_t* __restrict__ ids, float* __restrict__ weights,
                                       const float* __restrict__ x, int k_units, uint8_t* __restrict__ out, ZeroRows Z) {
    if (blockIdx.x == gridDim.x - 1) return write_zero_rows(Z);
    const int lane = threadIdx.x & 63, j = lane & 15;
    const int wave = threadIdx.x >> 6, tokens_per_block = blockDim.x >> 7;
    const bool quantizes = wave >= tokens_per_block; // (uniform per wave)
    const int64_t tok = (int64_t)blockIdx.x * tokens_per_block + (quantizes ? wave - tokens_per_block : wave);
    if (tok >= t) return; // whole waves leave together
    if (!quantizes) {
        int id;
        float w;
        moe_route::route_token<PER_LANE>(logits + tok * n_experts, n_experts, top_k, lane, id, w);
        if (lane < top_k) {
            ids[tok * top_k + lane] = id;
            weights[tok * top_k + lane] = w;
        }
        return;
    }
    for (int unit = lane >> 4; unit < k_units; unit += 4) {
        float v[16];
        load16(x + (tok * k_units + unit) * 256 + 16 * j, v);
        quantize_into_record<QMM_Q4_K, kWideRowRecord>(v, j, 0, out + (tok * k_units + unit) * kWideRowUnitBytes);
    }
}

template <bool GATE_UP, bool ORDERED>
hipError_t launch(const MoeGemmParams& P, int64_t max_chunks, hipStream_t stream) {
    constexpr size_t lds = kRing * kUnitLds + (GATE_UP ? (size_t)kRows * kHStride * 4 : 0);
    auto fn = &moe_gemm_q4k_kernel<GATE_UP, ORDERED>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    const unsigned grid = (unsigned)std::min<int64_t>((max_chunks * P.parts + 7) / 8 * 8, 8 * kCusPerXcd);
    fn<<<grid, 64 * kWaves, lds, stream>>>(P);
    return hipGetLastError();
}

// An item of up to 32 pairs is done in two thirds of the time of a longer one, and at one to four items per compute
// unit a launch ends with whoever has the most of them.  Long ones first pays where short items fill the last round: the kernel
// sees the counts and decides per XCD.  Here only where such counts are likely, because looking costs half a microsecond: around the 22 to
// 32 pairs per expert at which a few to half of the experts have more than 32, and at 61 to 72, where many spill a short second chunk.
// Set apart from the first that chunk reads its weights again, so there half as many short items again as the last round has places are
// asked for (29 for 29 cost 3 % when items were workgroups of their own; from 80 pairs on it never paid there).  us a layer (k = 2048), places that
// heed lengths in two rounds alone / this, even counts: 128 experts x 768 at 24, 28, 61, 64, 68 and 72 pairs 126 / 119, 127 / 119, 188 / 179,
// 198 / 191, 208 / 215, 211 / 215; 192 x 512 131 / 127, 135 / 133, 184 / 184, 215 / 207, 217 / 219, 224 / 229; 256 x 512 161 / 155, 163 / 158, then the
// same within 1 %; 160 x 768 148 / 145, then the same; 32 x 1536 78 / 78, 79 / 79, 102 / 99, 116 / 116, 115 / 118, 115 / 121.  Uneven counts (logits
// and N(0, 0.5) per expert) 0.92 to 1.02, where the last two columns of 32 x 1536 are 118 / 119 and 123 / 122.  Over 144 such layers 0.987.  Not for down,
// whose items are short already: 3 less to 3 us more when it was drawn, 5 at 256 experts.
// Returns twice the short items per place that the last round asks for, 0: the order of the experts.
int long_items_first(const MoeGemmParams& P, int64_t pairs) {
    const int64_t per_expert = pairs / P.n_experts;
    return per_expert >= 22 && per_expert <= 32 ? 2 : per_expert >= 61 && per_expert <= 72 ? 3 : 0;
}

MoeGemmParams base_params(const QmmLayout& L, const int32_t* perm, const int32_t* offsets, const int32_t* chunks,
                          const int32_t* chunk_expert, int n_experts) {
    MoeGemmParams P{};
    P.perm = perm, P.offsets = offsets, P.chunks = chunks, P.chunk_expert = chunk_expert, P.n_experts = n_experts;
    P.matrix_bytes = L.matrix_bytes, P.n = (int)L.n, P.row_tiles = (int)L.row_tiles;
    P.k_units = (int)L.k_units, P.k_groups = (int)L.k_groups, P.s = L.s, P.slots = L.slots, P.panel_bytes = (int)L.panel_bytes;
    P.row_bytes = (uint32_t)L.k_units * kWideRowUnitBytes;
    return P;
}

} // namespace

// (with the row of zeros behind them)
size_t qmm_wide_records_bytes(int64_t rows, int64_t k) { return (size_t)(rows + 1) * (size_t)(k / 256) * kWideRowUnitBytes; }

bool qmm_moe_gemm_supported(const QmmLayout& G, const QmmLayout& D, int64_t t, int top_k) {
    const int64_t pairs = t * top_k;
    if (G.dtype != QMM_Q4_K || D.dtype != QMM_Q4_K || G.k_units > kMaxUnits || D.k_units > kMaxUnits) return false;
    if (G.n < 256 || D.n < 256 || G.n % 256 || G.n != D.k) return false;
    // 32-bit offsets into a matrix and into the records, pair / top_k by multiplication, the grid
    if (G.matrix_bytes >= ((int64_t)1 << 31) || D.matrix_bytes >= ((int64_t)1 << 31)) return false;
    if ((t + 1) * G.k_units * kWideRowUnitBytes >= ((int64_t)1 << 32) || (pairs + 1) * D.k_units * kWideRowUnitBytes >= ((int64_t)1 << 32)) return false;
    if (pairs * D.n * 4 >= ((int64_t)1 << 32)) return false;
    const int64_t parts = G.n / 256 > (D.n + 511) / 512 ? G.n / 256 : (D.n + 511) / 512;
    return pairs * top_k < ((int64_t)1 << 32) && (pairs / kRows + G.n_stacked) * parts < 0x7ffffff0;
}

static ZeroRows zero_rows(void* records, int64_t rows, int64_t k, void* h_records, int64_t h_rows, int64_t h_k) {
    const int64_t row = k / 256 * kWideRowUnitBytes, h_row = h_k / 256 * kWideRowUnitBytes;
    static_assert(kWideRowUnitBytes % 16 == 0);
    return {{reinterpret_cast<u32x4*>((uint8_t*)records + rows * row), reinterpret_cast<u32x4*>((uint8_t*)h_records + h_rows * h_row)},
            {(int)(row / 16), (int)(h_row / 16)}};
}

hipError_t qmm_launch_wide_rows(const float* x, int64_t rows, int64_t k, void* records, void* h_records, int64_t h_rows, int64_t h_k,
                                hipStream_t stream) {
    const int64_t groups = rows * (k / 256);
    wide_rows_kernel<<<(unsigned)((groups * 16 + 255) / 256 + 1), 256, 0, stream>>>(x, groups, (uint8_t*)records,
                                                                                    zero_rows(records, rows, k, h_records, h_rows, h_k));
    return hipGetLastError();
}

hipError_t qmm_launch_moe_route_wide_rows(const float* logits, int64_t t, int n_experts, int top_k, int32_t* ids, float* weights,
                                          const float* x, int64_t k, void* records, void* h_records, int64_t h_rows, int64_t h_k,
                                          hipStream_t stream) {
    if (n_experts < 1 || n_experts > 1024 || top_k < 1 || top_k > 64 || top_k > n_experts) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)((t + 3) / 4 + 1); // four tokens per workgroup: four routing waves, four quantizing; the zeros
    const ZeroRows Z = zero_rows(records, t, k, h_records, h_rows, h_k);
    const int per_lane = (n_experts + 63) / 64, k_units = (int)(k / 256);
    auto go = [&](auto kernel) { kernel<<<grid, 512, 0, stream>>>(logits, t, n_experts, top_k, ids, weights, x, k_units, (uint8_t*)records, Z); };
    if (per_lane <= 2) go(route_wide_rows_kernel<2>);
    else if (per_lane <= 4) go(route_wide_rows_kernel<4>);
    else go(route_wide_rows_kernel<16>);
    return hipGetLastError();
}

hipError_t qmm_launch_moe_gemm_gate_up(const QmmLayout& G, const void* gate, const void* up, const void* records, int top_k,
                                       const int32_t* perm, const int32_t* offsets, const int32_t* chunks,
                                       const int32_t* chunk_expert, int n_experts, int64_t pairs, int64_t max_chunks, void* out_records,
                                       hipStream_t stream) {
    MoeGemmParams P = base_params(G, perm, offsets, chunks, chunk_expert, n_experts);
    P.w0 = (const uint8_t*)gate, P.w1 = (const uint8_t*)up;
    P.records = (const uint8_t*)records, P.out = out_records;
    P.row_div = top_k;
    P.row_magic = top_k > 1 ? (uint32_t)((((uint64_t)1 << 32) / (uint32_t)top_k) + 1) : 0;
    P.zero_row = (uint32_t)(pairs / top_k);
    P.parts = (int)(G.n / 256), P.out_units = P.parts;
    P.fill2 = long_items_first(P, pairs);
    return P.fill2 ? launch<true, true>(P, max_chunks, stream) : launch<true, false>(P, max_chunks, stream);
}

hipError_t qmm_launch_moe_gemm_down(const QmmLayout& D, const void* down, const void* records, const int32_t* perm,
                                    const int32_t* offsets, const int32_t* chunks, const int32_t* chunk_expert, int n_experts,
                                    int64_t pairs, int64_t max_chunks, float* y, hipStream_t stream) {
    MoeGemmParams P = base_params(D, perm, offsets, chunks, chunk_expert, n_experts);
    P.w0 = P.w1 = (const uint8_t*)down;
    P.records = (const uint8_t*)records, P.out = y;
    P.row_div = 0;
    P.zero_row = (uint32_t)pairs;
    P.parts = (int)((D.n + 511) / 512);
    return launch<false, false>(P, max_chunks, stream);
}
