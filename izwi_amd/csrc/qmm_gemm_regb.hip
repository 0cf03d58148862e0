// Prefill kernel for few activation rows: y[m, n] = x[m, k] * dequant(W)[n, k]^T with bf16 MFMA,
// weights dequantized straight into the matrix instruction's operand registers.
//
// From 65 to a few hundred rows what counts is that every weight byte is requested early, is
// dequantized once and needs no trip through LDS.  A workgroup of eight waves owns 32 * MT
// activation rows x 128 weight rows; wave (c, p) owns 32 of the weight rows and, of every unit of
// 256 k-elements, half p.  A lane's 16-byte quant chunk holds k-elements of one weight row only,
// which is what a lane supplies to v_mfma_f32_32x32x16_bf16: the chunk is unpacked into weight operands (the
// instruction's first) in registers, in the k order the chunk has, and the activation operand (staged in LDS by
// LDS-direct loads) is picked in the same order.  No weight tile in LDS, no LDS writes, one barrier per
// unit.  The two halves' sums meet in LDS at the end.  Where the tiles alone leave compute units idle, k is
// split over workgroups and the row tiles get lower.
//
// The loads run ahead of the units: weights four units in registers, activations two in LDS, and the
// first unit waits for its own loads alone.  The workgroups of an XCD begin at different units of k: beginning
// together they read the same 512 bytes of every activation row at once, and rows lie a power of two apart.
// One unit ahead and all at the same unit / four ahead / six and three (bf16 rows, us in a graph, cold weights): 2048 + 1024 + 1024
// at k = 2048, Q6_K, 80 rows 13.7 / 13.4 / 14.2, Q8_0 97 rows 14.5 / 14.1 / 14.8; 4096 x 4096 Q6_K 97 rows 17.9 / 16.9 / 17.5; 4096 + 1024 +
// 1024 Q8_0 66 rows 20.9 / 19.6 / 20.8, 128 rows 24.2 / 23.0 / 22.5; 3 x 1024 at k = 1024, Q8_0, 10.2 / 8.6 / 9.4: slices of four to
// eight units request deeper than they are long, in front of the second unit's activations.
//
// Bound by the life of a workgroup: at 2 x 12288 x 4096 (Q4_K, cold weights; time stamps) it has its arguments after 1.0 us
// and its first operands 4.2 later, takes 30 in sixteen units (1.95 a unit at 101 rows, 1.65 at 65; 2.1 and 1.8 with the
// loads one unit ahead and all workgroups at the same unit) and 2.2 for the exchange of the sums and stores (of a value a lane; since in 16-byte pieces).  Of a
// unit's 1.95 us 1.57 remain without its loads and 1.3 without unpacking and activations: matrix instructions (1.0),
// unpacking (1.0), LDS reads (0.9 to 1.2) and the loads share the compute unit, and two waves per SIMD overlap them in
// part.  An unpacking of a fifth fewer vector instructions (mixed-precision fma on f16 denormals) gave nothing.
// Splitting a unit four ways over the waves (64 x 128 wave tiles, fewer LDS reads) cost
// 14 us per workgroup instead: the exchange of the sums is 512 KB of LDS traffic there, 128 KB here.  us per
// call on f32 rows in a graph, one call per weight on 128 x 256 / 64 x 128 tiles with the weights through
// LDS / here with the loads one unit ahead.  Q4_K, 101 rows: q|k|v 81 / 27, 4096 x 4096 28 / 19, gate|up 82 / 47, down 47 / 32; Q6_K down
// 201 / 35; 512 rows: q|k|v 54 / 45; 0.6B shapes at 512: q|k|v 27 / 15.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "qmm_internal.h"
#include "qmm_tile.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kCols = 4, kSplits = 2; // waves of a workgroup: column groups x halves of a unit
constexpr int kWaves = kCols * kSplits;
constexpr int kBN = 32 * kCols;
constexpr int kUnitBytes = QMM_UNIT_ELEMS * 2; // one activation row of one unit, bf16

// fma(scale, byte, bias) of the eight bytes of (lo, hi) as one bf16 operand
__device__ __forceinline__ bf16x8 scaled_bytes(uint32_t lo, uint32_t hi, float scale, float bias) {
    u32x4 o;
    o.x = pack_bf16(__builtin_fmaf(scale, ubyte_f32<0>(lo), bias), __builtin_fmaf(scale, ubyte_f32<1>(lo), bias));
    o.y = pack_bf16(__builtin_fmaf(scale, ubyte_f32<2>(lo), bias), __builtin_fmaf(scale, ubyte_f32<3>(lo), bias));
    o.z = pack_bf16(__builtin_fmaf(scale, ubyte_f32<0>(hi), bias), __builtin_fmaf(scale, ubyte_f32<1>(hi), bias));
    o.w = pack_bf16(__builtin_fmaf(scale, ubyte_f32<2>(hi), bias), __builtin_fmaf(scale, ubyte_f32<3>(hi), bias));
    return __builtin_bit_cast(bf16x8, o);
}

struct RegbParams {
    const uint16_t* x; // bf16 [m, k], k a multiple of 32
    int64_t m, k;
    int k_units;
    int s, slots;
    int64_t panel_bytes, row_bytes; // row_bytes: all panels of a row tile
    int tiles_m, cols;              // cols: the members' column tiles times their slices
    uint32_t nibble_mask;           // 0x0f0f0f0f as data: one AND per four weights, v_cvt_f32_ubyteN for each
    int out_bf16;
    const void* residual; // single weight only
    int col_end[QMM_MAX_GROUP]; // one past each member's last (unused entries: past every column)
    int slices_v[QMM_MAX_GROUP], slice_units_v[QMM_MAX_GROUP];
    const uint8_t* wv[QMM_MAX_GROUP];
    void* yv[QMM_MAX_GROUP];
    float* partial_v[QMM_MAX_GROUP]; // [slice][m][n] where k is split
    int64_t nv[QMM_MAX_GROUP], row_tiles_v[QMM_MAX_GROUP];
};

// What a lane holds of its weight row's half unit (two steps of 64 k-elements).
template <int QT>
struct HalfRegs {
    static constexpr int NQ = QT == QMM_Q8_0 ? 4 : 2;
    static constexpr int kLoads = 1 + NQ + (QT == QMM_Q6_K ? 2 : 0); // load instructions of load_half
    using Header = std::conditional_t<QT == QMM_Q4_K, u32x4, u32x2>; // Q8_0, Q6_K: the two steps' scale dwords
    Header hdr;
    u32x4 q[NQ];
    u32x4 qh;   // Q6_K: the high bit pairs
    uint32_t d; // Q6_K
};

// Byte offsets of those pieces from the unit's address (a lane's row included).
struct HalfOffsets {
    uint32_t hdr, q, qh, d, q_stride;
};

template <int QT>
__device__ __forceinline__ void load_half(HalfRegs<QT>& r, const uint8_t* unit, const HalfOffsets& o) {
    r.hdr = *reinterpret_cast<const typename HalfRegs<QT>::Header*>(unit + o.hdr);
#pragma unroll
    for (int c = 0; c < HalfRegs<QT>::NQ; c++) r.q[c] = *reinterpret_cast<const u32x4*>(unit + o.q + c * o.q_stride);
    if (QT == QMM_Q6_K) {
        r.qh = *reinterpret_cast<const u32x4*>(unit + o.qh);
        r.d = *reinterpret_cast<const uint32_t*>(unit + o.d);
    }
}

// A use of the loaded registers: the compiler's own wait for them stands here and not behind the next unit's requests.  The
// counted wait in front covers the activations alone; up to two units' weights are in flight behind these, and the compiler,
// which counts the register loads only, waits until no more than those of the units behind are.
template <int QT>
__device__ __forceinline__ void arrived(HalfRegs<QT>& r) {
    asm volatile("" : "+v"(r.hdr));
#pragma unroll
    for (int c = 0; c < HalfRegs<QT>::NQ; c++) asm volatile("" : "+v"(r.q[c]));
    if (QT == QMM_Q6_K) asm volatile("" : "+v"(r.qh), "+v"(r.d));
}

// The factors of a step's two 32-element blocks: w = scale * byte + bias.
struct StepScales {
    float scale[2], bias[2];
};
template <int QT, int ST>
__device__ __forceinline__ StepScales step_scales(const HalfRegs<QT>& r, int half, int h) {
    StepScales s;
    if constexpr (QT == QMM_Q4_K) {
        const float d = qmm_f16_bits_to_f32((uint16_t)(r.hdr.x & 0xffffu)), dmin = qmm_f16_bits_to_f32((uint16_t)(r.hdr.x >> 16));
        uint32_t sc_lo, sc_hi, mn_lo, mn_hi;
        qmm_unpack_q4k_scales(r.hdr.y, r.hdr.z, r.hdr.w, sc_lo, sc_hi, mn_lo, mn_hi);
        const uint32_t sc = (half ? sc_hi : sc_lo) >> (16 * ST), mn = (half ? mn_hi : mn_lo) >> (16 * ST); // half is uniform
        s.scale[0] = d * (float)(sc & 0xffu), s.scale[1] = d * (float)((sc >> 8) & 0xffu);
        s.bias[0] = -(dmin * (float)(mn & 0xffu)), s.bias[1] = -(dmin * (float)((mn >> 8) & 0xffu));
    } else if constexpr (QT == QMM_Q8_0) {
        const uint32_t dd = r.hdr[ST];
        s.scale[0] = qmm_f16_bits_to_f32((uint16_t)(dd & 0xffffu)), s.scale[1] = qmm_f16_bits_to_f32((uint16_t)(dd >> 16));
        s.bias[0] = -128.0f * s.scale[0], s.bias[1] = -128.0f * s.scale[1]; // int8 q as unsigned byte u = q + 128
    } else {
        const float d = qmm_f16_bits_to_f32((uint16_t)(r.d & 0xffffu));
        const uint32_t sw = r.hdr[ST] >> (8 * h); // a scale per 16 elements: h, 2 + h of the step's four
        s.scale[0] = d * (float)(int8_t)(sw & 0xffu), s.scale[1] = d * (float)(int8_t)((sw >> 16) & 0xffu);
        s.bias[0] = -32.0f * s.scale[0], s.bias[1] = -32.0f * s.scale[1];
    }
    return s;
}

// Weight operand of matrix instruction SS (of eight): k-elements 64 (SS / 4) + 32 (SS / 2 % 2) + 16 h + 8 (SS % 2) .. + 7
// of the half unit.
template <int QT, int SS>
__device__ __forceinline__ bf16x8 half_operand(const HalfRegs<QT>& r, const StepScales& s, uint32_t nibble_mask) {
    constexpr int st = SS >> 2, q = (SS >> 1) & 1, e = SS & 1;
    uint32_t lo, hi;
    if constexpr (QT == QMM_Q4_K) {
        lo = (q ? r.q[st][2 * e] >> 4 : r.q[st][2 * e]) & nibble_mask;
        hi = (q ? r.q[st][2 * e + 1] >> 4 : r.q[st][2 * e + 1]) & nibble_mask;
    } else if constexpr (QT == QMM_Q8_0) {
        lo = r.q[2 * st + q][2 * e] ^ 0x80808080u;
        hi = r.q[2 * st + q][2 * e + 1] ^ 0x80808080u;
    } else {
        lo = ((r.q[q][2 * e] >> (4 * st)) & nibble_mask) | (((r.qh[2 * e] >> (4 * st + 2 * q)) & 0x03030303u) << 4);
        hi = ((r.q[q][2 * e + 1] >> (4 * st)) & nibble_mask) | (((r.qh[2 * e + 1] >> (4 * st + 2 * q)) & 0x03030303u) << 4);
    }
    return scaled_bytes(lo, hi, s.scale[q], s.bias[q]);
}

// Stages of activations in LDS and units of weights in registers
constexpr int kStages = 2, kBuffers = 4;

// f(I, false); if there is more, f(I, true) and the same from I + 1 on (nested, not a loop with exits: every
// step is reached from one place, so the compiler's waits there are for what was requested on that path)
template <int I, int N, class F, class M>
__device__ __forceinline__ void chain(F&& f, M&& more) {
    f(std::integral_constant<int, I>{}, std::false_type{});
    if constexpr (I + 1 < N)
        if (more()) {
            f(std::integral_constant<int, I>{}, std::true_type{});
            chain<I + 1, N>(f, more);
        }
}

// GATED: members 0 and 1 are gate and up of one shape, k is not split, and y = silu(gate) * up: a workgroup owns 64 columns of
// both (two of its four column groups each), whose sums meet in LDS; no launch behind it and no f32 products in memory.
template <int QT, int MT, bool GATED>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_regb_kernel(RegbParams P) {
    constexpr int BM = 32 * MT;
    constexpr int kStage = BM * kUnitBytes;
    constexpr int XL = BM / 2 / kWaves; // LDS-direct loads per wave and unit (1 KiB = two rows each)
    constexpr int NS = kStages, DW = kBuffers, WL = HalfRegs<QT>::kLoads;
    static_assert(NS == 2 && DW % NS == 0 && DW >= 3); // (the waits below)
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    // Workgroups go to the eight XCDs round-robin by their index; the row tiles of one (column tile,
    // slice) follow each other on one XCD, so its weights come from memory once.
    const int xcd = blockIdx.x & 7, pos = blockIdx.x >> 3;
    const int tm = pos % P.tiles_m;
    const int col = (pos / P.tiles_m) * 8 + xcd;
    if (col >= P.cols) return; // uniform
    // this workgroup's member, by selects: every table entry is loaded at once, none waits for another
    int slices = P.slices_v[0], slice_units = P.slice_units_v[0], first_col = 0;
    int64_t n = P.nv[0], row_tiles = P.row_tiles_v[0];
    const uint8_t* weights = P.wv[0];
    void* y = P.yv[0];
    float* partial = P.partial_v[0];
#pragma unroll
    for (int i = 1; i < QMM_MAX_GROUP; i++)
        if (!GATED && col >= P.col_end[i - 1]) {
            slices = P.slices_v[i], slice_units = P.slice_units_v[i], first_col = P.col_end[i - 1];
            n = P.nv[i], row_tiles = P.row_tiles_v[i];
            weights = P.wv[i], y = P.yv[i], partial = P.partial_v[i];
        }
    const int tn = (col - first_col) / slices, slice = col - first_col - tn * slices;
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * (GATED ? kBN / 2 : kBN);
    // A workgroup's units u0 .. u1 - 1 of k in turn, from `first` on: those that share an XCD begin at different
    // ones (see above).
    const int u0 = slice * slice_units, u1 = min(P.k_units, u0 + slice_units);
    const int first = (tn >> (GATED ? 4 : 3)) % (u1 - u0); // (GATED: as the same columns' own product)
    auto unit_of = [&](int u) { return u + first < u1 ? u + first : u + first - (u1 - u0); };

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wc = wave >> 1, half = wave & 1;
    const int h = lane >> 5;

    // ---- activations: instruction q of a unit moves rows 2 q, 2 q + 1; the 16-byte chunk c of a row
    // sits at chunk position c ^ (row & 15), so that 16 consecutive rows of one chunk touch every bank once
    const uint8_t* x_tile = reinterpret_cast<const uint8_t*>(P.x) + m0 * P.k * 2;
    uint32_t x_off[XL];
    {
        const int r0 = 2 * wave + h, c = (lane & 31) ^ (r0 & 15); // (row & 15 is the same for every i)
#pragma unroll
        for (int i = 0; i < XL; i++)
            x_off[i] = (uint32_t)((min(m0 + r0 + 2 * kWaves * i, P.m - 1) - m0) * P.k * 2 + c * 16);
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    // k ends inside the last unit (Q8_0 only): chunks at or past its end read the unit's first chunk
    // and are zeroed when they have landed
    const int x_tail = QT == QMM_Q8_0 ? (int)(P.k % QMM_UNIT_ELEMS) / 8 : 0;
    const int x_chunk = (lane & 31) ^ ((2 * wave + h) & 15);
    auto issue_x = [&](int at, int stage) {
        const int u = unit_of(at);
        const uint8_t* src = x_tile + (size_t)u * kUnitBytes;
        const uint32_t dst = lds0 + stage * kStage + wave * 1024;
        const uint32_t back = x_tail && u == P.k_units - 1 && x_chunk >= x_tail ? x_chunk * 16 : 0;
#pragma unroll
        for (int i = 0; i < XL; i++) load_to_lds(src, x_off[i] - back, dst + i * kWaves * 1024);
    };
    auto zero_tail = [&](int at, int stage) { // behind this wave's loads of the unit, in front of a barrier
        if (x_tail && unit_of(at) == P.k_units - 1 && x_chunk >= x_tail)
#pragma unroll
            for (int i = 0; i < XL; i++)
                *reinterpret_cast<u32x4*>(smem + stage * kStage + (wave + i * kWaves) * 1024 + lane * 16) = u32x4{0, 0, 0, 0};
    };

    // ---- weights: uniform unit address + 32-bit offsets
    const int64_t rt0 = n0 >> 4;
    const uint8_t* w_tile = (GATED && wc >= kCols / 2 ? P.wv[1] : weights) + rt0 * P.row_bytes;
    const int col32 = GATED ? wc & (kCols / 2 - 1) : wc; // the wave's 32 columns of the tile
    HalfOffsets off;
    {
        const int row = col32 * 32 + (lane & 31);
        const int64_t rt = min(rt0 + (row >> 4), row_tiles - 1);
        const uint32_t base = (uint32_t)((rt - rt0) * P.row_bytes) + (row & 15) * 16, chunk = (uint32_t)P.slots * 16;
        off.hdr = base + (QT == QMM_Q4_K ? 0 : 8 * half);
        off.q = base + (1 + (QT == QMM_Q8_0 ? 8 : 4) * half + h) * chunk;
        off.q_stride = 2 * chunk;
        off.qh = base + (9 + 2 * half + h) * chunk;
        off.d = base + 13 * chunk;
    }
    auto load_w = [&](HalfRegs<QT>& r, int at) {
        const int u = unit_of(at);
        const int kg = u / P.s, us = u - kg * P.s;
        load_half<QT>(r, w_tile + (int64_t)kg * P.panel_bytes + us * 256, off);
    };

    f32x16 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;

    // Activation operand of matrix instruction ss: row l & 31 of each 32-row block, chunk 16 half + 8 (ss / 4) + 4 (ss / 2 % 2)
    // + 2 h + ss % 2 of the unit
    const int frag_x = (lane & 31) * kUnitBytes + (((16 * half + 2 * h) ^ (lane & 15)) << 4);

    // Software pipeline: the operands of instruction ss + 1 are read / unpacked behind instruction ss;
    // the unit's only barrier sits in front of its last one, where every activation of the unit is in
    // registers and the next unit has landed; behind it the activations NS units on and the weights DW units
    // on are requested, in this order.  Loads land in order: what may still be in flight at a barrier is
    // what was requested behind the next unit's activations, one unit's weights.  (The compiler's own waits count the weights
    // alone; with three units of them or more they ask for no more.)
    HalfRegs<QT> w[DW];
    StepScales sc[2];
    bf16x8 a[2][MT], b[2];
    auto read_a = [&](int stage, auto SS) {
        constexpr int ss = decltype(SS)::value;
        const uint8_t* src = smem + stage * kStage + (frag_x ^ ((8 * (ss >> 2) + 4 * ((ss >> 1) & 1) + (ss & 1)) << 4));
#pragma unroll
        for (int i = 0; i < MT; i++) a[ss & 1][i] = *reinterpret_cast<const bf16x8*>(src + i * 32 * kUnitBytes);
    };
    const int last = u1 - 1;
    // (past the end: the last unit's weights again, never used)
    auto request_w = [&](auto I) {
        load_w(w[decltype(I)::value], min(u0 + decltype(I)::value, last));
        asm volatile("" ::: "memory"); // the requests stay here, in this order
    };
    issue_x(u0, 0);
    static_for<DW - 1>(request_w);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DW - 2) * WL) : "memory");
    zero_tail(u0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    arrived<QT>(w[0]);
    if (u0 + 1 <= last) issue_x(u0 + 1, 1); // only now: the first unit does not wait for them
    request_w(std::integral_constant<int, DW - 1>{});
    read_a(0, std::integral_constant<int, 0>{});
    sc[0] = step_scales<QT, 0>(w[0], half, h);
    b[0] = half_operand<QT, 0>(w[0], sc[0], P.nibble_mask);
    int u = u0;
    auto multiply = [&](auto SS) {
        constexpr int ss = decltype(SS)::value;
#pragma unroll
        for (int j = 0; j < MT; j++) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[ss & 1], a[ss & 1][j], acc[j], 0, 0, 0);
#pragma unroll
        for (int q = 0; q < MT; q++) { // one matrix instruction, then a share of the next one's operands
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 32 / MT, 0);
        }
    };
    auto front = [&](auto I) { // matrix instructions 0 .. 6 of the unit in stage I % NS, buffer I
        constexpr int i = decltype(I)::value;
        static_for<7>([&](auto SS) {
            constexpr int ss = decltype(SS)::value;
            if constexpr (ss == 3) sc[1] = step_scales<QT, 1>(w[i], half, h);
            read_a(i % NS, std::integral_constant<int, ss + 1>{});
            b[(ss + 1) & 1] = half_operand<QT, ss + 1>(w[i], sc[(ss + 1) >> 2], P.nibble_mask);
            multiply(SS);
        });
    };
    // The turn to the next unit around the last matrix instruction.  Behind the next unit's activations may still
    // fly: the weights requested with them (BEHIND).
    auto turn = [&](auto I, auto REQUESTS, auto BEHIND) {
        constexpr int i = decltype(I)::value, next = (i + 1) % DW;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(BEHIND)::value) : "memory");
        zero_tail(u + 1, (i + 1) % NS);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        arrived<QT>(w[next]);
        if (u + NS <= last) issue_x(u + NS, i % NS);
        asm volatile("" ::: "memory");
        if constexpr (decltype(REQUESTS)::value) load_w(w[i], min(u + DW, last));
        asm volatile("" ::: "memory"); // the requests stay here
        read_a((i + 1) % NS, std::integral_constant<int, 0>{});
        sc[0] = step_scales<QT, 0>(w[next], half, h);
        b[0] = half_operand<QT, 0>(w[next], sc[0], P.nibble_mask);
        multiply(std::integral_constant<int, 7>{});
        u++;
    };
    while (u + DW <= last)
        static_for<DW>([&](auto I) {
            front(I);
            turn(I, std::true_type{}, std::integral_constant<int, WL>{});
        });
    // the last 1 .. DW units, whose weights have all been requested
    chain<0, DW>([&](auto I, auto MORE) {
        if constexpr (!decltype(MORE)::value) front(I);
        else turn(I, std::false_type{}, std::integral_constant<int, decltype(I)::value == 0 ? WL : 0>{});
    }, [&] { return u < last; });
    multiply(std::integral_constant<int, 7>{});

    // ---- epilogue.  The weights are the matrix instruction's first operand: a lane holds four consecutive columns at a time of
    // one activation row.  32 x 32 blocks of sums leave through LDS in whole 16-byte pieces; the residual is requested
    // in front of the halves' exchange.  (Stored from the accumulators, two bytes a lane, the residual read in front of each:
    // 4096 x 4096 with a bf16 residual, Q4_K, 32 us at 400 rows and 33 at 500 in two slices, which were the faster; so in
    // one slice 27 and 29.)
    constexpr int kOwn = (MT + 1) / 2; // the wave of half p finishes the blocks i with i % 2 = p
    const bool split = slices > 1, f32_out = split || !P.out_bf16;
    RowsOut R;
    R.out = split ? partial + (int64_t)slice * P.m * n : y, R.residual = split ? nullptr : P.residual;
    R.m = P.m, R.n = n, R.n_end = n, R.col0 = n0 + col32 * 32;
    const bool is_up = GATED && wc >= kCols / 2, whole = whole_pieces(R); // uniform
    auto rows_of = [&](auto I) {
        RowsOut own = R;
        own.row0 = m0 + (2 * decltype(I)::value + half) * 32;
        return own;
    };
    auto own = [&](auto&& f) { // (GATED: of a wave pair (gate, up) of the same columns the one finishes block 0, the other block 1)
        static_for<kOwn>([&](auto I) {
            if (2 * decltype(I)::value + half < MT && (!GATED || decltype(I)::value == (int)is_up)) f(I);
        });
    };
    RowPieces<32, 4, 0, 4> pieces_f32[kOwn];
    RowPieces<32, 8, 0, 2> pieces_bf16[kOwn];
    if (whole) own([&](auto I) {
        if (f32_out) pieces_f32[decltype(I)::value].request(rows_of(I), lane);
        else pieces_bf16[decltype(I)::value].request(rows_of(I), lane);
    });
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); // (every activation request has been waited for)

    // ---- the two halves' sums
    f32x16 sum[kOwn];
    {
        uint8_t* dst = smem + wc * (MT * 4096) + lane * 16;
        auto send = [&](auto PAIR) { // the blocks of the other half
            static_for<MT>([&](auto I) {
                constexpr int i = decltype(I)::value;
                if constexpr (i % 2 == decltype(PAIR)::value)
                    for (int r = 0; r < 4; r++)
                        *reinterpret_cast<f32x4*>(dst + i * 4096 + r * 1024) =
                            f32x4{acc[i][4 * r], acc[i][4 * r + 1], acc[i][4 * r + 2], acc[i][4 * r + 3]};
            });
        };
        if (half) send(std::integral_constant<int, 0>{}); // uniform
        else send(std::integral_constant<int, 1>{});
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        auto take = [&](auto PAIR) {
            static_for<MT>([&](auto I) {
                constexpr int i = decltype(I)::value;
                if constexpr (i % 2 == decltype(PAIR)::value)
                    for (int r = 0; r < 4; r++) {
                        const f32x4 v = *reinterpret_cast<const f32x4*>(dst + i * 4096 + r * 1024);
                        for (int e = 0; e < 4; e++) sum[i / 2][4 * r + e] = acc[i][4 * r + e] + v[e];
                    }
            });
        };
        if (half) take(std::integral_constant<int, 1>{});
        else take(std::integral_constant<int, 0>{});
    }
    if constexpr (GATED) {
        uint8_t* at = smem + kCols * MT * 4096 + (2 * col32 + half) * 8192 + lane * 16; // (behind the halves' sums)
        auto put = [&](const f32x16& v, int slot) {
            for (int r = 0; r < 4; r++)
                *reinterpret_cast<f32x4*>(at + slot * 4096 + r * 1024) = f32x4{v[4 * r], v[4 * r + 1], v[4 * r + 2], v[4 * r + 3]};
        };
        if (is_up) put(sum[0], 0);
        else if constexpr (kOwn > 1) put(sum[1], 1);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (!is_up)
            for (int r = 0; r < 4; r++) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(at + r * 1024);
                for (int e = 0; e < 4; e++) sum[0][4 * r + e] = qmm_silu(sum[0][4 * r + e]) * v[e];
            }
        else if constexpr (kOwn > 1)
            for (int r = 0; r < 4; r++) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(at + 4096 + r * 1024);
                for (int e = 0; e < 4; e++) sum[1][4 * r + e] = qmm_silu(v[e]) * sum[1][4 * r + e];
            }
    }
    // A block goes where the wave has read the other half's sums of it: chunk c (four columns) of row r at chunk c ^ (r / 2 % 8)
    auto block_at = [&](int i, int row, int col) {
        return smem + wc * (MT * 4096) + (2 * i + half) * 4096 + row * 128 + (((col >> 2) ^ ((row >> 1) & 7)) << 4) + (col & 3) * 4;
    };
    auto keep = [&](auto I) {
        constexpr int i = decltype(I)::value;
        static_for<4>([&](auto G) {
            constexpr int g = decltype(G)::value;
            *reinterpret_cast<f32x4*>(block_at(i, lane & 31, 8 * g + 4 * h)) =
                f32x4{sum[i][4 * g], sum[i][4 * g + 1], sum[i][4 * g + 2], sum[i][4 * g + 3]};
        });
    };
    lanes_exchange(); // (the other half's sums have been read)
    auto finish = [&](auto& pieces) {
        own(keep);
        lanes_exchange();
        own([&](auto I) {
            pieces[decltype(I)::value].store(rows_of(I), lane, [&](int row, int col) {
                return *reinterpret_cast<const f32x4*>(block_at(decltype(I)::value, row, col));
            });
        });
    };
    if (whole) {
        if (f32_out) finish(pieces_f32);
        else finish(pieces_bf16);
    } else {
        own([&](auto I) {
            auto one = [&](int row, int col) { return *reinterpret_cast<const float*>(block_at(decltype(I)::value, row, col)); };
            keep(I);
            lanes_exchange();
            if (f32_out) store_values<32, true>(rows_of(I), lane, one);
            else store_values<32, false>(rows_of(I), lane, one);
        });
    }
}

// y = sum over slices (in order) of partial[slice] (+ residual), four consecutive values per thread, all
// split members of a group in one launch (blocks of member i: block_end[i - 1] .. block_end[i])
struct RegbReduceParams {
    const float* partial[QMM_MAX_GROUP];
    void* y[QMM_MAX_GROUP];
    int64_t count[QMM_MAX_GROUP];
    int block_end[QMM_MAX_GROUP], slices[QMM_MAX_GROUP];
    int out_bf16;
    const void* residual;
};
__global__ __launch_bounds__(256) void regb_reduce_kernel(RegbReduceParams P) {
    int slices = P.slices[0], first_block = 0;
    int64_t count = P.count[0];
    const float* partial = P.partial[0];
    void* y = P.y[0];
#pragma unroll
    for (int i = 1; i < QMM_MAX_GROUP; i++)
        if ((int)blockIdx.x >= P.block_end[i - 1])
            slices = P.slices[i], first_block = P.block_end[i - 1], count = P.count[i], partial = P.partial[i], y = P.y[i];
    const int64_t i = ((int64_t)(blockIdx.x - first_block) * 256 + threadIdx.x) * 4;
    partial += i;
    if (i + 4 <= count && (count & 3) == 0 && ((reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(P.residual)) & 15) == 0) {
        f32x4 res = {0.0f, 0.0f, 0.0f, 0.0f};
        if (P.residual && P.out_bf16) {
            const u32x2 v = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(P.residual) + i);
            res = f32x4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u)};
        } else if (P.residual) {
            res = *reinterpret_cast<const f32x4*>(static_cast<const float*>(P.residual) + i);
        }
        f32x4 sum = *reinterpret_cast<const f32x4*>(partial);
        for (int s = 1; s < slices; s++) sum += *reinterpret_cast<const f32x4*>(partial + s * count);
        if (P.residual) sum += res;
        if (P.out_bf16) *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(y) + i) = u32x2{pack_bf16(sum.x, sum.y), pack_bf16(sum.z, sum.w)};
        else *reinterpret_cast<f32x4*>(static_cast<float*>(y) + i) = sum;
    } else {
        for (int e = 0; e < 4 && i + e < count; e++) {
            float sum = partial[e];
            for (int s = 1; s < slices; s++) sum += partial[s * count + e];
            qmm_store(y, QmmEpilogue{P.residual, P.out_bf16}, i + e, sum);
        }
    }
}

struct RegbPlan {
    int mt, slices[QMM_MAX_GROUP], slice_units[QMM_MAX_GROUP];
};

// Slices of k for n columns in `tiles` full-height tiles, in microseconds: a unit costs 1.2 where the row tiles are as
// low as the compute units allow; the slices' sums a launch (4.2) and their bytes twice.
int slices_of(int64_t tiles, int64_t n, int64_t m, int k_units, int64_t limit, int min_units) {
    double best = 1.2 * k_units;
    int slices = 1;
    for (int s = 2; s <= 8 && tiles * s <= limit; s++) {
        const int su = (k_units + s - 1) / s;
        if (su < min_units || (k_units + su - 1) / su != s) continue;
        const double cost = 1.2 * su + 4.2 + s * (double)m * (double)n * 4.0 / 2.2e6;
        if (cost < 0.98 * best) best = cost, slices = s;
    }
    return slices;
}

// Up to 128 rows a matrix is split by its own shape and m, whatever group it is in, so that a group's sums are
// those of its members' separate calls bit for bit.  The split that is best for a wide matrix alone fills the chip once and
// is a second round in a group (gate|up of 2 x 12288 at k = 4096, 101 rows: 47 us in one slice, 61 in two; one of the
// two alone 41 and 34): so a split stops at half of the compute units (two such members fill the chip) and at four units
// per slice.  What that leaves idle the row tiles take: their height is no matter of the sums, so it is chosen for the
// launch as a whole, the lowest whose workgroups still run in one round (of each XCD, which holds whole
// column tiles): the 12288 alone 31 us in 64-row tiles, 2 x 6144 at k = 2048 24.6 -> 19.4, 2 x 3072 at k = 1024
// 16.1 -> 12.2, 1024 x 2048 15.2 -> 12.1.  (It costs a wide matrix alone at 65 to 96 rows, of which the second
// 64-row tile is half empty: 12288 x 4096 at 65, Q4_K 29.2 -> 31.4, Q8_0 32.7 -> 36.3.)  Matrices more
// than twice as long as wide (the MLP's last) and up to 64 rows, where groups run the integer arithmetic, come
// alone: they are split over the whole chip.
// Beyond 128 rows a group is planned as one matrix (4096 -> 4096 + 1024 + 1024 at 512 rows: 45 us, member by member 52).
RegbPlan plan_regb(const QmmLayout* const* layouts, int n_weights, int64_t m, int n_cus) {
    RegbPlan p;
    const int k_units = (int)layouts[0]->k_units, min_units = m <= 32 ? 2 : std::clamp(k_units / 4, 2, 4);
    const int64_t full_tiles = (m + 127) / 128;
    int64_t tiles[QMM_MAX_GROUP] = {}, all_tiles = 0, n_total = 0, cols = 0;
    for (int i = 0; i < n_weights; i++) {
        tiles[i] = (layouts[i]->n + kBN - 1) / kBN * full_tiles;
        all_tiles += tiles[i], n_total += layouts[i]->n;
    }
    for (int i = 0; i < QMM_MAX_GROUP; i++) {
        p.slices[i] = 1, p.slice_units[i] = k_units;
        if (i >= n_weights) continue;
        const bool alone = m <= 64 || layouts[i]->k > 2 * layouts[i]->n;
        p.slices[i] = m <= 128 ? slices_of(tiles[i], layouts[i]->n, m, k_units, alone ? n_cus : n_cus / 2, min_units)
                               : slices_of(all_tiles, n_total, m, k_units, n_cus, min_units);
        p.slice_units[i] = (k_units + p.slices[i] - 1) / p.slices[i];
        cols += tiles[i] / full_tiles * p.slices[i];
    }
    const int64_t blocks = (m + 31) / 32, cols_xcd = (cols + 7) / 8;
    p.mt = (int)((blocks + full_tiles - 1) / full_tiles);
    for (int mt = p.mt - 1; mt >= 1; mt--)
        if (cols_xcd * ((blocks + mt - 1) / mt) <= n_cus / 8) p.mt = mt;
    return p;
}

// bytes of member i's partial sums
size_t partial_bytes(const RegbPlan& p, const QmmLayout& L, int i, int64_t m) {
    return p.slices[i] <= 1 ? 0 : (((size_t)p.slices[i] * (size_t)m * (size_t)L.n * sizeof(float)) + 255) & ~(size_t)255;
}

template <int QT, int MT, bool GATED>
hipError_t launch_regb(const RegbParams& P, int64_t grid, hipStream_t stream) {
    constexpr size_t stages = std::max((size_t)kStages * 32 * MT * kUnitBytes, (size_t)kCols * MT * 4096 + (GATED ? kWaves * 4096 : 0)); // (the sums' exchange)
    static_assert(stages <= 160 * 1024, "LDS of a CU");
    auto fn = &gemm_regb_kernel<QT, MT, GATED>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)stages);
    if (e != hipSuccess) return e;
    fn<<<dim3((unsigned)grid), dim3(64 * kWaves), stages, stream>>>(P);
    return hipGetLastError();
}

template <int QT, bool GATED>
hipError_t launch_regb_qt(const RegbParams& P, const RegbPlan& p, int64_t grid, hipStream_t stream) {
    switch (p.mt) {
        case 1: return launch_regb<QT, 1, GATED>(P, grid, stream);
        case 2: return launch_regb<QT, 2, GATED>(P, grid, stream);
        case 3: return launch_regb<QT, 3, GATED>(P, grid, stream);
        default: return launch_regb<QT, 4, GATED>(P, grid, stream);
    }
}
template <bool GATED>
hipError_t launch_regb_type(int dtype, const RegbParams& P, const RegbPlan& p, int64_t grid, hipStream_t stream) {
    return dtype == QMM_Q6_K   ? launch_regb_qt<QMM_Q6_K, GATED>(P, p, grid, stream)
           : dtype == QMM_Q4_K ? launch_regb_qt<QMM_Q4_K, GATED>(P, p, grid, stream)
                               : launch_regb_qt<QMM_Q8_0, GATED>(P, p, grid, stream);
}
// what every member shares
RegbParams base_params(const QmmLayout& L0, const RegbPlan& plan, const uint16_t* x_bf16, int64_t m, int out_bf16) {
    RegbParams P;
    P.x = x_bf16;
    P.m = m, P.k = L0.k;
    P.k_units = (int)L0.k_units;
    P.s = L0.s, P.slots = L0.slots;
    P.panel_bytes = L0.panel_bytes, P.row_bytes = L0.k_groups * L0.panel_bytes;
    P.nibble_mask = 0x0f0f0f0fu;
    P.out_bf16 = out_bf16;
    P.residual = nullptr;
    P.tiles_m = (int)((m + 32 * plan.mt - 1) / (32 * plan.mt));
    return P;
}

} // namespace

// Up to 128 rows always, beyond where the 128 x 128 tiles are at most one per compute unit: measured against
// the 256-row tiles of qmm_gemm.hip (Q4_K, us per call in a graph, here / there): q|k|v 4096 -> 6144 39.0 / 50.9
// at 512 rows (192 tiles), 71.9 / 64.9 at 768 (288); 4096 x 4096 42.1 / 54.8 at 1024 (256), 93.1 / 80.6 at
// 2048 (512); gate|up of 2 x 3072 at k = 1024 14.7 / 25.6 at 512 (192), 26.9 / 26.4 at 768 (288); gate|up of
// 2 x 12288 at 129, 150 and 192 rows (384) 78 / 83, 75 / 75 and 75 / 71 (Q8_0 at 192: 80 / 74); 65536 x 1024 at
// 129 rows (1024) 54 / 44, 151936 x 4096 (2374) 363 / 333 and at 193 rows 422 / 316.
bool qmm_gemm_regb_applies(const QmmLayout* const* layouts, int n_weights, int64_t m, int n_cus) {
    if (m <= 0 || n_weights < 1 || qmm_gemm_tile_forced()) return false;
    int64_t tiles = 0;
    const int64_t tiles_m = (m + 127) / 128;
    for (int i = 0; i < n_weights; i++) {
        const QmmLayout& L = *layouts[i];
        if (L.n_stacked != 1 || L.n == 0 || L.dtype != layouts[0]->dtype || L.k != layouts[0]->k) return false;
        tiles += tiles_m * ((L.n + kBN - 1) / kBN);
    }
    if (m <= 128) return true;
    if (qmm_get_prefill_form() >= 0) return false; // one of the other forms was asked for
    return tiles <= n_cus;
}

size_t qmm_gemm_regb_workspace_bytes(const QmmLayout* const* layouts, int n_weights, int64_t m, int n_cus) {
    const RegbPlan p = plan_regb(layouts, n_weights, m, n_cus);
    size_t total = 0;
    for (int i = 0; i < n_weights; i++) total += partial_bytes(p, *layouts[i], i, m);
    return total;
}

hipError_t qmm_launch_gemm_regb(const QmmLayout* const* layouts, const void* const* tiled, int n_weights, const uint16_t* x_bf16,
                                int64_t m, void* const* ys, int out_bf16, void* workspace, int n_cus, hipStream_t stream,
                                const void* residual) {
    if (n_weights < 1 || n_weights > QMM_MAX_GROUP || (residual && n_weights != 1)) return hipErrorInvalidValue;
    const QmmLayout& L0 = *layouts[0];
    const RegbPlan plan = plan_regb(layouts, n_weights, m, n_cus);
    RegbParams P = base_params(L0, plan, x_bf16, m, out_bf16);
    P.residual = plan.slices[0] > 1 ? nullptr : residual;
    RegbReduceParams R;
    uint8_t* next = static_cast<uint8_t*>(workspace);
    int64_t cols = 0, blocks = 0;
    for (int i = 0; i < QMM_MAX_GROUP; i++) {
        P.col_end[i] = 0x7fffffff, P.slices_v[i] = 1, P.slice_units_v[i] = 0, P.wv[i] = nullptr, P.yv[i] = nullptr, P.partial_v[i] = nullptr;
        P.nv[i] = 0, P.row_tiles_v[i] = 0;
        R.partial[i] = nullptr, R.y[i] = nullptr, R.count[i] = 0, R.slices[i] = 1, R.block_end[i] = (int)blocks;
        if (i >= n_weights) continue;
        const QmmLayout& L = *layouts[i];
        if (L.dtype != L0.dtype || L.k != L0.k || L.n_stacked != 1 || L.n == 0) return hipErrorInvalidValue;
        cols += (L.n + kBN - 1) / kBN * plan.slices[i];
        if (cols > 0x7ffffff0) return hipErrorInvalidValue;
        P.col_end[i] = (int)cols;
        P.slices_v[i] = plan.slices[i], P.slice_units_v[i] = plan.slice_units[i];
        P.wv[i] = static_cast<const uint8_t*>(tiled[i]), P.yv[i] = ys[i];
        P.nv[i] = L.n, P.row_tiles_v[i] = L.row_tiles;
        if (plan.slices[i] <= 1) continue;
        if (workspace == nullptr) return hipErrorInvalidValue;
        P.partial_v[i] = reinterpret_cast<float*>(next);
        next += partial_bytes(plan, L, i, m);
        R.partial[i] = P.partial_v[i], R.y[i] = ys[i], R.count[i] = m * L.n, R.slices[i] = plan.slices[i];
        blocks += (R.count[i] + 1023) / 1024;
        if (blocks > 0x7fffffff) return hipErrorInvalidValue;
        R.block_end[i] = (int)blocks;
    }
    const int64_t grid = (cols + 7) / 8 * 8 * P.tiles_m;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    P.cols = (int)cols;
    hipError_t e = launch_regb_type<false>(L0.dtype, P, plan, grid, stream);
    if (e != hipSuccess || blocks == 0) return e;
    R.out_bf16 = out_bf16, R.residual = residual;
    regb_reduce_kernel<<<(unsigned)blocks, 256, 0, stream>>>(R);
    return hipGetLastError();
}

bool qmm_gemm_regb_gated_applies(const QmmLayout& L, int64_t m, int n_cus) {
    const QmmLayout* const pair[2] = {&L, &L};
    if (!qmm_gemm_regb_applies(pair, 2, m, n_cus)) return false;
    const RegbPlan plan = plan_regb(pair, 2, m, n_cus);
    return plan.slices[0] == 1 && plan.slices[1] == 1;
}

hipError_t qmm_launch_gemm_regb_gated(const QmmLayout& L, const void* gate, const void* up, const uint16_t* x_bf16, int64_t m, void* h,
                                      int h_bf16, int n_cus, hipStream_t stream) {
    if (!qmm_gemm_regb_gated_applies(L, m, n_cus)) return hipErrorNotSupported;
    const QmmLayout* const pair[2] = {&L, &L};
    const RegbPlan plan = plan_regb(pair, 2, m, n_cus);
    RegbParams P = base_params(L, plan, x_bf16, m, h_bf16);
    const int64_t cols = (L.n + kBN / 2 - 1) / (kBN / 2), grid = (cols + 7) / 8 * 8 * P.tiles_m;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    P.cols = (int)cols;
    for (int i = 0; i < QMM_MAX_GROUP; i++) {
        P.col_end[i] = 0x7fffffff, P.slices_v[i] = 1, P.slice_units_v[i] = (int)L.k_units, P.partial_v[i] = nullptr;
        P.wv[i] = static_cast<const uint8_t*>(i ? up : gate), P.yv[i] = h, P.nv[i] = L.n, P.row_tiles_v[i] = L.row_tiles;
    }
    return launch_regb_type<true>(L.dtype, P, plan, grid, stream);
}
