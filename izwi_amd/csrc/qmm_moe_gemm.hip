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
// A workgroup of eight waves owns up to 64 sorted pairs (two blocks of 32) of one expert and, of every
// wave, two blocks of 32 weight rows: gate and up of the same 32 columns, or two blocks of down.  The
// pairs' activation records stay in LDS over all of k (up to eight units), so that after one barrier the
// waves walk k on their own; a lane's weight chunks are requested one unit ahead.
//
// gate | up: the 256 columns of a workgroup are one unit of the down projection's input, so
// silu(gate) * up is quantized here, in LDS, and leaves as records: 9.5 bytes instead of 64 per eight
// values, no launch in between.
//
// Bound by vector instructions (about 160 per block of 32 x 32 outputs and unit in the loop, half of them the
// unpacking that two blocks of pairs share, 640 cycles; 209 and 191 with everything around it) beside 17 matrix
// instructions (544 cycles), which two waves per SIMD overlap in part: at 4096 tokens the vector ALU is busy
// 56 % of the cycles of gate | up and the matrix pipe 36 %.
// 128 experts, top-8, 2048 x 768: gate | up 282 us and down 164 at 4096 tokens (730 and 630 TOP/s), where the
// 16-row-tile kernels took 480 and 260 and the quantizer between them 40; 80 and 41 at 512 tokens (70 with the long
// items first), before 92, 48 and 8 (a workgroup's life is 40 us there, 1.5 per compute unit).  The layer 823 -> 497 us and 156 -> 136.  Of that,
// starting on the first unit's records while the others land, stores at 32-bit offsets and the two waves
// of a SIMD half a phase apart with the one in its matrix instructions preferred: 556 -> 497 and 150 -> 136.
#include <hip/hip_runtime.h>

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
constexpr int kHStride = 264; // floats per row of silu(gate) * up in LDS

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
    int n_experts, parts, n, row_tiles, k_units, k_groups, s, slots, panel_bytes;
    int out_units;
    int fill2; // long items first: twice the short items asked for per place of the last round
};

__device__ __forceinline__ void barrier_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ float silu(float v) { return v / (1.0f + expf(-v)); }

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

template <bool GATE_UP, int NRB>
__device__ __forceinline__ void chunk_body(const MoeGemmParams& P, const uint8_t* wbase0, const uint8_t* wbase1, uint8_t* smem,
                                           UnitRegs (&raw)[2], const uint32_t (&lane_off)[2], const uint32_t* out_off, int part,
                                           int pos_begin, int pos_end, int wave, int lane) {
    const int row = lane & 31, h = lane >> 5;
    // byte offsets of the lane's A chunks: [b & 1][i], of its sums, and of its four runs of scales
    const uint32_t sw = (uint32_t)(row >> 1) & 7u;
    uint32_t a_off[2][2];
#pragma unroll
    for (int bb = 0; bb < 2; bb++)
#pragma unroll
        for (int i = 0; i < 2; i++) a_off[bb][i] = (uint32_t)row * 128u + (((uint32_t)(4 * bb + 2 * h + i)) ^ sw) * 16u;
    const uint32_t sum_off = (uint32_t)kSumsAt + (uint32_t)row * 32u + (((uint32_t)h ^ ((uint32_t)(row >> 3) & 1u)) * 16u);
    const uint32_t scale_off = (uint32_t)kScalesAt + (uint32_t)h * 16u;
    const _Float16 cf = h ? (_Float16)32.0f : (_Float16)1.0f, kf = h ? (_Float16)-32768.0f : (_Float16)-1024.0f;
    const f16x2 c2 = {cf, cf}, k2 = {kf, kf};
    const uint32_t slots16 = (uint32_t)P.slots * 16u;

    f32x16 acc[2][NRB];
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
        for (int rb = 0; rb < NRB; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[c][rb][r] = 0.0f;

    uint32_t unit_off = 0;                    // of the next unit to request: panel, then unit in the panel
    int in_panel = 0;
    const uint8_t* lds = smem;
    if (wave >= kWaves / 2) __builtin_amdgcn_s_sleep(10); // the two waves of a SIMD half a phase apart
    for (int u = 0; u < P.k_units; u++, lds += kUnitLds) {
        if (u == 1) { // the other units' records have landed
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            barrier_lds();
        }
        // (past the last unit the same one is requested again: no branch around the loads)
        if (u + 1 < P.k_units) {
            if (++in_panel == P.s) in_panel = 0, unit_off += (uint32_t)P.panel_bytes - (uint32_t)(P.s - 1) * 256u;
            else unit_off += 256u;
        }
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
                        const i32x4 a = *reinterpret_cast<const i32x4*>(lds + (b >> 1) * (kRows * 128) + rb * 4096 + a_off[b & 1][i]);
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
            // the unit is consumed: the next one into its registers (the fences keep the scheduler from
            // gathering the loads of both columns at the loop's end, where nothing is left to cover them)
            asm volatile("" : "+v"(d), "+v"(dmin)); // (computed here, so that the header's registers are free)
            __builtin_amdgcn_s_setprio(0);
            if (NRB > 1) __builtin_amdgcn_sched_barrier(0);
            const uint8_t* wu = (c ? wbase1 : wbase0) + unit_off;
            w.hdr = *reinterpret_cast<const u32x4*>(wu + lane_off[c]);
#pragma unroll
            for (int b = 0; b < 4; b++)
                w.q[b] = *reinterpret_cast<const u32x4*>(wu + (uint32_t)(1 + 2 * b) * slots16 + (lane_off[c] + (uint32_t)h * slots16));
            if (NRB > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rb = 0; rb < NRB; rb++) {
                const f16x8 sums = *reinterpret_cast<const f16x8*>(lds + sum_off + rb * 1024);
                const f32x16 msum = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, mins, f32x16{}, 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const f32x4 dx = *reinterpret_cast<const f32x4*>(lds + scale_off + rb * 128 + g * 32);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int isum = (hi[rb][4 * g + r] << 3) + lo[rb][4 * g + r];
                        acc[c][rb][4 * g + r] =
                            fmaf(fmaf(-dmin, msum[4 * g + r], d * (float)isum), dx[r], acc[c][rb][4 * g + r]);
                    }
                }
                if (NRB > 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    const int col = wave * 32 + row;
    if constexpr (GATE_UP) {
        barrier_lds(); // every wave has read its last activations
        float* hbuf = reinterpret_cast<float*>(smem);
#pragma unroll
        for (int rb = 0; rb < NRB; rb++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                hbuf[(rb * 32 + (r & 3) + 8 * (r >> 2) + 4 * h) * kHStride + col] = silu(acc[0][rb][r]) * acc[1][rb][r];
        barrier_lds();
        const int j = lane & 15;
#pragma unroll
        for (int pass = 0; pass < NRB; pass++) {
            const int m = pass * 32 + (int)(threadIdx.x >> 4);
            float v[16];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const f32x4 f = *reinterpret_cast<const f32x4*>(hbuf + m * kHStride + 16 * j + 4 * i);
                v[4 * i] = f.x, v[4 * i + 1] = f.y, v[4 * i + 2] = f.z, v[4 * i + 3] = f.w;
            }
            if (pos_begin + m < pos_end) // (whole 16-lane groups)
                quantize_into_record<QMM_Q4_K, kWideRowRecord>(
                    v, j, 0, static_cast<uint8_t*>(P.out) + ((int64_t)(pos_begin + m) * P.out_units + part) * kWideRowUnitBytes);
        }
    } else {
        // 32-bit byte offsets from one uniform base; only an expert's last chunk has rows that do not exist
        uint8_t* y = static_cast<uint8_t*>(P.out);
        const bool whole = pos_end - pos_begin == NRB * 32;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int n = part * 512 + c * 256 + col;
            if (n >= P.n) continue; // (uniform: n is a multiple of 256)
#pragma unroll
            for (int rb = 0; rb < NRB; rb++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const u32x4 rows = *reinterpret_cast<const u32x4*>(out_off + rb * 32 + 8 * g + 4 * h);
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (whole || rb * 32 + 8 * g + 4 * h + r < pos_end - pos_begin)
                            *reinterpret_cast<float*>(y + (rows[r] + (uint32_t)n * 4u)) = acc[c][rb][4 * g + r];
                }
        }
    }
}

// The records of units [u0, u1) of the chunk's rows into their LDS images
__device__ __forceinline__ void issue_records(const MoeGemmParams& P, const uint32_t* src_off, uint8_t* smem, int nrb, int u0, int u1,
                                              int wave, int lane) {
    const uint32_t lds_base = (uint32_t)(uintptr_t)smem;
    const int groups = nrb * 4, per_unit = 2 * groups + nrb + 1; // pieces of quants (two halves), sums, scales
    for (int piece = u0 * per_unit + wave; piece < u1 * per_unit; piece += kWaves) {
        const int u = piece / per_unit, sub = piece - u * per_unit;
        const uint32_t unit_lds = lds_base + (uint32_t)u * kUnitLds;
        const uint8_t* base = P.records + u * kWideRowUnitBytes;
        if (sub < 2 * groups) {
            const int p = sub / groups, g = sub - p * groups;
            const int r = g * 8 + (lane >> 3);
            const uint32_t to = __builtin_amdgcn_readfirstlane(unit_lds + p * (kRows * 128) + g * 1024);
            load_to_lds(base, src_off[r] + (uint32_t)p * 128u + (uint32_t)((lane & 7) ^ ((r >> 1) & 7)) * 16u, to);
        } else if (sub < 2 * groups + nrb) {
            const int q = sub - 2 * groups, r = q * 32 + (lane >> 1);
            const uint32_t to = __builtin_amdgcn_readfirstlane(unit_lds + kSumsAt + q * 1024);
            load_to_lds(base, src_off[r] + 256u + (uint32_t)((lane & 1) ^ ((r >> 3) & 1)) * 16u, to);
        } else {
            const uint32_t to = __builtin_amdgcn_readfirstlane(unit_lds + kScalesAt);
            load_to_lds4(base, src_off[lane] + 288u, to);
        }
    }
}

struct WorkItem {
    int e, part, pos_begin, pos_end;
};
constexpr int kCusPerXcd = 32;
constexpr int kOrderedItems = 4 * kCusPerXcd; // the longest run of an XCD's items that is put in order
constexpr int kOrderedPerLane = (kOrderedItems + 63) / 64;

__device__ __forceinline__ WorkItem work_item(const MoeGemmParams& P, int item) {
    const int e = P.chunk_expert[item / P.parts]; // (an expert's items begin at parts * its first chunk)
    const int chunk0 = P.chunks[e], n_chunks = P.chunks[e + 1] - chunk0;
    const int local = item - chunk0 * P.parts, part = local / n_chunks, chunk = local - part * n_chunks;
    const int begin = P.offsets[e] + chunk * kRows;
    return {e, part, begin, min(P.offsets[e + 1], begin + kRows)};
}

template <bool GATE_UP, bool ORDERED>
__global__ __launch_bounds__(64 * kWaves) void moe_gemm_q4k_kernel(MoeGemmParams P) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ __attribute__((aligned(16))) uint32_t out_off[kRows]; // down: byte offsets of the output rows
    __shared__ uint32_t src_off[kRows];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // Work items in the order (expert, part of the weight rows, chunk of the pairs), cut into eight equal
    // runs: workgroups go to the XCDs round-robin, so a run is one XCD's, and the chunks that read the same weights
    // follow one another there and find them in its L2.
    const int items = P.chunks[P.n_experts] * P.parts, per_xcd = (items + 7) >> 3;
    const int slot = (int)(blockIdx.x >> 3), first = (int)(blockIdx.x & 7) * per_xcd;
    const int run = min(per_xcd, items - first); // items of this XCD
    if (slot >= run) return; // uniform
    // Where the last of an XCD's rounds can hold short items alone, those of more than 32 pairs go first (every wave looks at
    // the whole run, a lane per item) and the short ones fill in behind them.
    WorkItem it = work_item(P, first + slot);
    if (ORDERED && run > kCusPerXcd && run <= kOrderedItems) {
        WorkItem mine[kOrderedPerLane];
        uint64_t heavy[kOrderedPerLane], light[kOrderedPerLane];
        int heavies = 0;
#pragma unroll
        for (int j = 0; j < kOrderedPerLane; j++) {
            heavy[j] = light[j] = 0;
            if (64 * j >= run) continue; // uniform
            const bool exists = 64 * j + lane < run;
            mine[j] = work_item(P, first + (exists ? 64 * j + lane : 0));
            heavy[j] = __ballot(exists && mine[j].pos_end - mine[j].pos_begin > 32);
            light[j] = __ballot(exists && mine[j].pos_end - mine[j].pos_begin <= 32);
            heavies += __popcll(heavy[j]);
        }
        const int lights = run - heavies, last_round = (run - 1) % kCusPerXcd + 1;
        if (heavies > 0 && 2 * lights >= P.fill2 * last_round) { // uniform, the same in all workgroups of the run
            int rank = slot < heavies ? slot : slot - heavies;
            bool found = false;
#pragma unroll
            for (int j = 0; j < kOrderedPerLane; j++) {
                const uint64_t set = slot < heavies ? heavy[j] : light[j];
                const int in_set = __popcll(set);
                if (!found && rank < in_set) { // uniform
                    const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(set >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)set, 0));
                    const int at = __ffsll((unsigned long long)__ballot((set >> lane & 1) && below == rank)) - 1;
                    it.e = __builtin_amdgcn_readlane(mine[j].e, at), it.part = __builtin_amdgcn_readlane(mine[j].part, at);
                    it.pos_begin = __builtin_amdgcn_readlane(mine[j].pos_begin, at), it.pos_end = __builtin_amdgcn_readlane(mine[j].pos_end, at);
                    found = true;
                }
                rank -= in_set;
            }
        }
    }
    const int e = it.e, part = it.part, pos_begin = it.pos_begin, pos_end = it.pos_end;
    const int nrb = pos_end - pos_begin > 32 ? 2 : 1;

    const uint8_t* wbase0 = P.w0 + (int64_t)e * P.matrix_bytes;
    const uint8_t* wbase1 = P.w1 + (int64_t)e * P.matrix_bytes;
    const int h = lane >> 5;
    uint32_t lane_off[2];
    UnitRegs raw[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int rt = (GATE_UP ? part * 16 : part * 32 + c * 16) + wave * 2 + ((lane >> 4) & 1);
        lane_off[c] = (uint32_t)(min(rt, P.row_tiles - 1) * P.k_groups) * (uint32_t)P.panel_bytes + (uint32_t)(lane & 15) * 16u;
        const uint8_t* wu = c ? wbase1 : wbase0;
        const uint32_t slots16 = (uint32_t)P.slots * 16u;
        raw[c].hdr = *reinterpret_cast<const u32x4*>(wu + lane_off[c]);
#pragma unroll
        for (int b = 0; b < 4; b++)
            raw[c].q[b] = *reinterpret_cast<const u32x4*>(wu + (uint32_t)(1 + 2 * b) * slots16 + (lane_off[c] + (uint32_t)h * slots16));
    }
    if (threadIdx.x < kRows) {
        // (a row past the end reads the chunk's first row; its sums are never stored)
        const int pos = pos_begin + (int)threadIdx.x;
        const int at = pos < pos_end ? pos : pos_begin;
        const uint32_t pair = (uint32_t)P.perm[at];
        const uint32_t src = P.row_div == 0 ? (uint32_t)at : P.row_div == 1 ? pair : __umulhi(pair, P.row_magic);
        src_off[threadIdx.x] = src * P.row_bytes;
        out_off[threadIdx.x] = pair * (uint32_t)P.n * 4u;
    }
    barrier_lds();
    // The first unit's records, then, under the arithmetic of the first unit, the others'
    issue_records(P, src_off, smem, nrb, 0, 1, wave, lane);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // (a use of the loaded registers: the compiler's own wait for them stands here, not in the loop)
#pragma unroll
    for (int c = 0; c < 2; c++) {
        asm volatile("" : "+v"(raw[c].hdr));
#pragma unroll
        for (int b = 0; b < 4; b++) asm volatile("" : "+v"(raw[c].q[b]));
    }
    barrier_lds();
    issue_records(P, src_off, smem, nrb, 1, P.k_units, wave, lane);
    if (nrb == 2)
        chunk_body<GATE_UP, 2>(P, wbase0, wbase1, smem, raw, lane_off, out_off, part, pos_begin, pos_end, wave, lane);
    else
        chunk_body<GATE_UP, 1>(P, wbase0, wbase1, smem, raw, lane_off, out_off, part, pos_begin, pos_end, wave, lane);
}

// ---- the activation rows' records, 16 lanes per (row, unit) ----------------------------------
__device__ __forceinline__ void load16(const float* __restrict__ src, float (&v)[16]) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float4 f = reinterpret_cast<const float4*>(src)[i];
        v[4 * i] = f.x, v[4 * i + 1] = f.y, v[4 * i + 2] = f.z, v[4 * i + 3] = f.w;
    }
}
__global__ void wide_rows_kernel(const float* __restrict__ x, int64_t groups, uint8_t* __restrict__ out) {
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
                                       const float* __restrict__ x, int k_units, uint8_t* __restrict__ out) {
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
    const size_t window = (size_t)P.k_units * kUnitLds, hbuf = GATE_UP ? (size_t)kRows * kHStride * 4 : 0;
    const size_t lds = window > hbuf ? window : hbuf;
    auto fn = &moe_gemm_q4k_kernel<GATE_UP, ORDERED>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxUnits * kUnitLds);
    if (e != hipSuccess) return e;
    const unsigned grid = (unsigned)((max_chunks * P.parts + 7) / 8 * 8);
    fn<<<grid, 64 * kWaves, lds, stream>>>(P);
    return hipGetLastError();
}

// An item of up to 32 pairs is done in two thirds of the time of a longer one, and at one to four items per compute
// unit a launch ends with whoever started a long one last.  Long ones first pays where short items fill the last round: the kernel
// sees the counts and decides per XCD.  Here only where such counts are likely, because looking costs half a microsecond: around the 22 to
// 32 pairs per expert at which a few to half of the experts have more than 32, and at 61 to 72, where many spill a short second chunk.
// Set apart from the first that chunk reads its weights again, so there half as many short items again as the last round has places are
// asked for (29 for 29 cost 3 %); from 80 pairs on it never pays (1500 tokens 250 / 263, 4096 521 / 542).  us of gate | up (top-8, k =
// 2048) over the order of the experts, by pairs per expert: 128 experts x 768 -10 at 24 to 30, -21 at 64, -7 at 72; 192 x 512 -10 and
// -20; 256 x 512 -9 at 24 to 28, +5 to +7 at 61 and 64, -13 at 72; 160 x 768 -9 at 28, +4 at 64, -16 at 72.  Not for down, whose items
// are short already: 3 less to 3 us more, 5 at 256 experts.
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

size_t qmm_wide_records_bytes(int64_t rows, int64_t k) { return (size_t)rows * (size_t)(k / 256) * kWideRowUnitBytes; }

bool qmm_moe_gemm_supported(const QmmLayout& G, const QmmLayout& D, int64_t t, int top_k) {
    const int64_t pairs = t * top_k;
    if (G.dtype != QMM_Q4_K || D.dtype != QMM_Q4_K || G.k_units > kMaxUnits || D.k_units > kMaxUnits) return false;
    if (G.n < 256 || D.n < 256 || G.n % 256 || G.n != D.k) return false;
    // 32-bit offsets into a matrix and into the records, pair / top_k by multiplication, the grid
    if (G.matrix_bytes >= ((int64_t)1 << 31) || D.matrix_bytes >= ((int64_t)1 << 31)) return false;
    if (t * G.k_units * kWideRowUnitBytes >= ((int64_t)1 << 32) || pairs * D.k_units * kWideRowUnitBytes >= ((int64_t)1 << 32)) return false;
    if (pairs * D.n * 4 >= ((int64_t)1 << 32)) return false;
    const int64_t parts = G.n / 256 > (D.n + 511) / 512 ? G.n / 256 : (D.n + 511) / 512;
    return pairs * top_k < ((int64_t)1 << 32) && (pairs / kRows + G.n_stacked) * parts < 0x7ffffff0;
}

hipError_t qmm_launch_wide_rows(const float* x, int64_t rows, int64_t k, void* records, hipStream_t stream) {
    const int64_t groups = rows * (k / 256);
    wide_rows_kernel<<<(unsigned)((groups * 16 + 255) / 256), 256, 0, stream>>>(x, groups, (uint8_t*)records);
    return hipGetLastError();
}

hipError_t qmm_launch_moe_route_wide_rows(const float* logits, int64_t t, int n_experts, int top_k, int32_t* ids, float* weights,
                                          const float* x, int64_t k, void* records, hipStream_t stream) {
    if (n_experts < 1 || n_experts > 1024 || top_k < 1 || top_k > 64 || top_k > n_experts) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)((t + 3) / 4); // four tokens per workgroup: four routing waves, four quantizing
    const int per_lane = (n_experts + 63) / 64, k_units = (int)(k / 256);
    auto go = [&](auto kernel) { kernel<<<grid, 512, 0, stream>>>(logits, t, n_experts, top_k, ids, weights, x, k_units, (uint8_t*)records); };
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
    P.parts = (int)(G.n / 256), P.out_units = P.parts;
    P.fill2 = long_items_first(P, pairs);
    return P.fill2 ? launch<true, true>(P, max_chunks, stream) : launch<true, false>(P, max_chunks, stream);
}

hipError_t qmm_launch_moe_gemm_down(const QmmLayout& D, const void* down, const void* records, const int32_t* perm,
                                    const int32_t* offsets, const int32_t* chunks, const int32_t* chunk_expert, int n_experts,
                                    int64_t max_chunks, float* y, hipStream_t stream) {
    MoeGemmParams P = base_params(D, perm, offsets, chunks, chunk_expert, n_experts);
    P.w0 = P.w1 = (const uint8_t*)down;
    P.records = (const uint8_t*)records, P.out = y;
    P.row_div = 0;
    P.parts = (int)((D.n + 511) / 512);
    return launch<false, false>(P, max_chunks, stream);
}
