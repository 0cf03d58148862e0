// Prefill kernel: y[m, n] = x[m, k] * dequant(W)[n, k]^T with bf16 MFMA.
//
// A workgroup (8 waves, 4 x 2) owns a BM x BN output tile (256 x 256 when the
// problem fills the chip with such tiles, 256 x 192 or 256 x 128 otherwise; few rows and small
// products take qmm_gemm_regb.hip); each wave a (BM/4) x (BN/2) sub-tile held in
// v_mfma_f32_32x32x16_bf16 accumulators.
// Per 64-wide k step the workgroup
//   * copies the BM x 64 bf16 activation tile to LDS,
//   * reads the matching 64 k-elements of BN weight rows straight from the
//     panel layout (header + nibble / int8 chunks), dequantizes them in
//     registers and writes bf16 to LDS,
//   * runs 4 k16 steps of MFMAs per wave, operands read from LDS as one
//     16-byte load per lane (row stride padded to 144 B: conflict free).
// LDS holds two such stages: while the MFMAs of step i run out of one, the
// tile of step i+1 (loaded to registers during step i-1) is dequantized into
// the other and the global loads of step i+2 are issued, with one barrier per
// step.
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
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int BK = 64;
constexpr int kRowStride = 144; // bytes per LDS tile row: 64 bf16 + 16 B pad
#ifndef QMM_GEMM_VALU_PER_MFMA
#define QMM_GEMM_VALU_PER_MFMA 4
#endif

struct GemmParams {
    const uint8_t* w;
    const uint16_t* x; // bf16 [m, k]
    void* y;
    int64_t m, n, k;
    int64_t n_begin, n_end; // output columns (weight rows) of this launch, n_begin a multiple of 256
    int k_units, k_groups, s, slots;
    int64_t row_tiles, panel_bytes;
    int out_bf16;
    int tiles_m, tiles_n;
    // split-k form (blockIdx.y = slice): slice s covers units [s * slice_units, ..) of 256
    // k-elements and writes its f32 tile to partial[s][m][n]; a second kernel adds the slices
    // in order
    int slice_units;
    // 0x0f0f0f0f, passed as data: with the constant in the code the compiler folds mask and
    // byte select into one bit-field extract per weight, followed by a convert; with an unknown
    // mask it emits one AND per four weights and v_cvt_f32_ubyteN for each
    uint32_t nibble_mask;
    float* partial;
    const void* residual; // of y's type, added to the sums before they are stored (may alias y)
    // several weights of equal k and type on the same activations in one launch (pipelined tiles
    // only): column tile t of the grid belongs to weight i with tn_end[i - 1] <= t < tn_end[i];
    // w / y / n / n_end / row_tiles / partial above are replaced by the member's at kernel entry
    int n_weights; // 0 or 1: a single weight
    int tn_end[QMM_MAX_GROUP];
    const uint8_t* wv[QMM_MAX_GROUP];
    void* yv[QMM_MAX_GROUP];
    int64_t nv[QMM_MAX_GROUP], row_tiles_v[QMM_MAX_GROUP];
    float* partial_v[QMM_MAX_GROUP];
};

// Pipelined 256-column tile.  The k loop runs over units of 256 k-elements with the four
// 64-wide steps of a unit unrolled, so that the sub-block index, the LDS stage and the
// chunk offsets inside the panel are compile-time constants; whatever depends on the
// step otherwise (unit offset inside the panel row, activation column) is uniform and
// stays in scalar registers, the per-lane part of every address is a 32-bit offset
// computed once.  XTAIL: k is not a multiple of 64 (Q8_0 only), activation chunks at or
// past k are zeroed on their way to LDS.
template <int QT, int BM, int BN, bool XTAIL, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_pipe_kernel(GemmParams P_in) {
    GemmParams P = P_in;
    int tn_local = (int)(blockIdx.x / P_in.tiles_m);
    if (P_in.n_weights > 1) { // a projection group: this workgroup's member (uniform)
        int i = 0;
        while (i + 1 < P_in.n_weights && tn_local >= P_in.tn_end[i]) i++;
        tn_local -= i ? P_in.tn_end[i - 1] : 0;
        P.w = P_in.wv[i];
        P.y = P_in.yv[i];
        P.n = P.n_end = P_in.nv[i];
        P.row_tiles = P_in.row_tiles_v[i];
        P.partial = P_in.partial ? P_in.partial_v[i] : nullptr;
    }
    // NW waves as a (NW / 2) x 2 grid of wave tiles; with eight waves two share a SIMD, each with
    // half the accumulators, and one issues while the other waits
    constexpr int THREADS = 64 * NW, WM = NW / 2;
    constexpr int MT = BM / WM / 32, NT = BN / 64;       // 32 x 32 accumulator tiles per wave
    // 192 weight rows among 512 threads: at every k step one half of the waves stages rows 0 .. 127, two threads a row,
    // and the other rows 128 .. 191, four threads a row; the halves change places with the parity of the staged step, so
    // that each has its one and a half shares in the mean.  The two parities' rows are two sets of staging state, and
    // the k loop exists twice, once for either half (H).
    constexpr bool MIXED = BN == 192;
    constexpr int NSET = MIXED ? 2 : 1;
    constexpr int XC = BM * 8 / THREADS;                 // 16-byte activation chunks per thread and k step
    constexpr int TPR = MIXED ? 2 : THREADS / BN;        // threads that share a weight row: 1, 2 or 4 (the fewest)
    constexpr bool Q6 = QT == QMM_Q6_K;
    static_assert(!MIXED || (NW == 8 && BM == 256 && !Q6));
    static_assert(!Q6 || TPR == 2 || TPR == 4, "Q6_K is staged by two or four threads per weight row");
    constexpr int NCR = QT == QMM_Q4_K ? 2 : 4;          // 16-byte quant chunks per row and k step
    // Q6_K: a half unit (two k steps) shares its 64 bytes of low nibbles and 32 bytes of bit pairs.
    // A thread takes 16 of the 32 byte positions (the half `lh` = part & 1) in both 32-element groups
    // of a step (two parts per row) or in one of them (four parts): NQL dwords of nibbles, NQH of
    // bit pairs, held for both steps
    constexpr int NGG = 4 / TPR, NQL = 4 * NGG, NQH = 4;
    constexpr int ND = Q6 ? NQL + NQH : 4 * NCR / TPR;   // the thread's run of quant dwords: 2 .. 16
    // of the thread at a step with tpr threads per row
    auto nd_of = [](int tpr) constexpr { return Q6 ? NQL + NQH : 4 * NCR / tpr; };
    auto nc_of = [](int tpr) constexpr { return Q6 ? NGG : 4 * NCR / tpr >= 4 ? NCR / tpr : 1; }; // loads per k step (16 bytes; 8 for two dwords)
    constexpr int GS = NT == 3 ? 3 : 4; // MFMAs of a group
    constexpr int GPK = MT * NT / GS;   // groups per k16 step
    constexpr int NG = 4 * GPK;         // groups per k step: 16 (64 x 128 wave tiles) or 8
    constexpr int kStage = (BM + BN) * kRowStride;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    const int tm = blockIdx.x % P.tiles_m;
    const int tn = tn_local;
    const int64_t m0 = (int64_t)tm * BM, n0 = P.n_begin + (int64_t)tn * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int u0 = P.partial ? (int)blockIdx.y * P.slice_units : 0;             // first unit of this workgroup
    const int u1 = P.partial ? min(P.k_units, u0 + P.slice_units) : P.k_units;  // one past its last
    const int last_step = P.k_units * 4 - 1;

    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    // ---- staging state: tile kt+1 sits in xr / wr while step kt runs
    // activation chunks in flight: tile kt+1 (written to LDS during step kt) and, where the
    // register file allows, tile kt+2 behind it, so that a chunk is requested XD k steps
    // before it is needed
    constexpr int XD = BN == 128 ? 2 : 1;
    u32x4 xr[XD][XC];
    u32x4 w_hdr[NSET]; // header of the unit fetched last (Q6_K: its 16 signed scales)
    uint32_t w_d = 0; // Q6_K: the dword with d of that unit
    // quant dwords of tile kt+1 (being dequantized) and tile kt+2 (in flight), by parity of the k step
    // (Q6_K: of the half unit; low nibbles first, bit pairs behind them)
    uint32_t wq[2][ND];
    // activations: uniform tile base + uniform column + per-lane (row, chunk) offset
    const uint8_t* x_tile = reinterpret_cast<const uint8_t*>(P.x) + m0 * P.k * 2;
    uint32_t x_off[XC];
    int x_lds[XC];
#pragma unroll
    for (int i = 0; i < XC; i++) {
        const int c = tid + THREADS * i;
        const int row = c >> 3, kc = c & 7;
        x_off[i] = (uint32_t)((min(m0 + row, P.m - 1) - m0) * P.k * 2 + kc * 16);
        x_lds[i] = row * kRowStride + kc * 16;
    }
    // weights: thread t stages part t / BN of row n0 + t % BN (the lanes of a wave write 64
    // different rows of the padded LDS tile: no bank conflicts, and the part is wave-uniform);
    // rows past the matrix read the last row-tile (their output columns are never stored)
    const int64_t rt0 = n0 >> 4;
    const int64_t rowtile_bytes = (int64_t)P.k_groups * P.panel_bytes;
    const uint8_t* w_tile = P.w + rt0 * rowtile_bytes;
    const uint32_t slot_bytes = (uint32_t)P.slots * 16u;
    // part p holds dwords p ND .. p ND + ND - 1 of the row's quant dwords of a step (Q4_K: 8
    // dwords of nibbles, dword D = elements 4 D .. (low) and 32 + 4 D .. (high); Q8_0: 16 dwords of
    // int8): its first chunk (and, for half a chunk, the offset inside it) and its LDS position
    const int w_part = tid / BN; // (not MIXED)
    uint32_t w_off[NSET], w_off_q[NSET];
    int w_lds[NSET], w_block[NSET]; // (w_block: the block of 32 elements, Q8_0)
#pragma unroll
    for (int p = 0; p < NSET; p++) {
        const bool two = !MIXED || p == tid >> 8;
        const int t = tid & 255;
        const int row = !MIXED ? tid % BN : two ? t & 127 : 128 + (t & 63);
        const int part = !MIXED ? w_part : two ? t >> 7 : t >> 6;
        const int d0 = Q6 ? 0 : part * (two ? ND : ND / 2);
        w_off[p] = (uint32_t)((min(rt0 + (row >> 4), P.row_tiles - 1) - rt0) * rowtile_bytes) + (uint32_t)(row & 15) * 16u;
        w_off_q[p] = w_off[p] + (uint32_t)(d0 / 4) * slot_bytes + (uint32_t)(d0 % 4) * 4u;
        w_lds[p] = (BM + row) * kRowStride + (Q6 ? 32 * part : d0 * 8);
        w_block[p] = d0 / 8;
    }
    // Q6_K: element 32 gg + l of the k step with nibble `nib` of half unit h is nibble `nib` of
    // ql[64 h + 32 gg + l] with bit pair 2 nib + gg of qh[32 h + l]; its 16-element group is
    // 4 (2 h + nib) + 2 gg + l / 16.  Part p: l = 16 lh .., lh = p & 1; gg = 0 and 1 (two parts)
    // or p / 2 (four parts)
    const int q6_lh = w_part & 1, q6_gg = TPR == 4 ? w_part >> 1 : 0;
    const uint32_t w_off_ql = w_off[0] + (uint32_t)(2 * q6_gg + q6_lh) * slot_bytes;
    const uint32_t w_off_qh = w_off[0] + (uint32_t)q6_lh * slot_bytes;
    const int q6_pair_shift = 2 * q6_gg;
    const int q6_scale_shift = 8 * (2 * q6_gg + q6_lh); // of the step's four scale bytes
    // load cursor: the unit whose chunks are fetched next (clamped to the last unit)
    int cur_us = u0 < P.k_units ? u0 % P.s : 0;
    uint32_t cur_kg_off = (uint32_t)((u0 < P.k_units ? u0 / P.s : 0) * P.panel_bytes);
    int cur_unit = min(u0, P.k_units - 1);
    auto advance_cursor = [&]() {
        if (cur_unit + 1 < P.k_units) {
            cur_unit++;
            cur_us++;
            if (cur_us == P.s) cur_us = 0, cur_kg_off += (uint32_t)P.panel_bytes;
        }
    };

    auto x_load = [&](int kt, int buf, int i) {
        if (XTAIL) {
            // chunks at or past k read chunk 0 of the row; x_write turns them into zeros
            const bool ok = (int64_t)kt * BK + (tid & 7) * 8 < P.k;
            xr[buf][i] = *reinterpret_cast<const u32x4*>(x_tile + (ok ? (int64_t)kt * (BK * 2) : -(int64_t)((tid & 7) * 16)) + x_off[i]);
        } else {
            xr[buf][i] = *reinterpret_cast<const u32x4*>(x_tile + (size_t)min(kt, last_step) * (BK * 2) + x_off[i]);
        }
    };
    auto x_write = [&](int kt, int buf, int i, uint8_t* stage) {
        if (XTAIL) {
            const bool ok = (int64_t)kt * BK + (tid & 7) * 8 < P.k;
            *reinterpret_cast<u32x4*>(stage + x_lds[i]) = ok ? xr[buf][i] : u32x4{0, 0, 0, 0};
        } else {
            *reinterpret_cast<u32x4*>(stage + x_lds[i]) = xr[buf][i];
        }
    };
    auto w_load_hdr = [&]() {
#pragma unroll
        for (int p = 0; p < NSET; p++)
            w_hdr[p] = *reinterpret_cast<const u32x4*>(w_tile + (cur_kg_off + (uint32_t)cur_us * 256u) + w_off[p]);
        if constexpr (Q6)
            w_d = *reinterpret_cast<const uint32_t*>(w_tile + (cur_kg_off + (uint32_t)cur_us * 256u + 13u * slot_bytes) + w_off[0]);
    };
    // Q6_K: the low nibbles of the thread's group c (HI = 0) or its bit pairs (HI = 1, c = 0) of half
    // unit HALF of the cursor's unit
    auto w_load_q6 = [&](auto HALF, auto HI, int c) {
        constexpr int half = decltype(HALF)::value, hi = decltype(HI)::value;
        const uint8_t* src = w_tile +
                             (cur_kg_off + (uint32_t)cur_us * 256u + (uint32_t)(hi ? 9 + 2 * half : 1 + 4 * half + 2 * c) * slot_bytes) +
                             (hi ? w_off_qh : w_off_ql);
        const u32x4 v = *reinterpret_cast<const u32x4*>(src);
        constexpr int o = hi ? NQL : 0;
        wq[half][o + 4 * c] = v.x, wq[half][o + 4 * c + 1] = v.y, wq[half][o + 4 * c + 2] = v.z, wq[half][o + 4 * c + 3] = v.w;
    };
    auto w_load_q = [&](auto SUB, auto TPRS, int c) {
        constexpr int sub = decltype(SUB)::value, par = sub & 1, set = MIXED ? par : 0;
        const uint8_t* src =
            w_tile + (cur_kg_off + (uint32_t)cur_us * 256u + (uint32_t)(1 + sub * NCR + c) * slot_bytes) + w_off_q[set];
        if constexpr (nd_of(decltype(TPRS)::value) >= 4) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(src);
            wq[par][4 * c] = v.x, wq[par][4 * c + 1] = v.y, wq[par][4 * c + 2] = v.z, wq[par][4 * c + 3] = v.w;
        } else {
            const uint2 v = *reinterpret_cast<const uint2*>(src);
            wq[par][0] = v.x, wq[par][1] = v.y;
        }
    };
    // header of the unit being staged, unpacked once per unit
    struct Unpacked {
        float hd = 0, hdmin = 0;                             // Q4_K: d, dmin
        uint32_t sc_lo = 0, sc_hi = 0, mn_lo = 0, mn_hi = 0; // Q4_K: 8 scale bytes, 8 min bytes; Q8_0: 8 f16 scales
    } hu[NSET];
    auto w_unpack = [&]() {
#pragma unroll
        for (int p = 0; p < NSET; p++) {
            Unpacked& u = hu[p];
            const u32x4 h = w_hdr[p];
            if (QT == QMM_Q4_K) {
                u.hd = qmm_f16_bits_to_f32((uint16_t)(h.x & 0xffffu));
                u.hdmin = -qmm_f16_bits_to_f32((uint16_t)(h.x >> 16));
                qmm_unpack_q4k_scales(h.y, h.z, h.w, u.sc_lo, u.sc_hi, u.mn_lo, u.mn_hi);
            } else {
                if (Q6) u.hd = qmm_f16_bits_to_f32((uint16_t)(w_d & 0xffffu));
                u.sc_lo = h.x, u.sc_hi = h.y, u.mn_lo = h.z, u.mn_hi = h.w; // (Q6_K: scales 4 sub .. 4 sub + 3 in dword sub)
            }
        }
    };
    // scales of the tile being staged
    float sa = 0, ba = 0, sb = 0, bb = 0; // Q4_K: (d1, -m1, d2, -m2); Q8_0: (dA, -128 dA, dB, -128 dB)
    float sw = 0, bw = 0;                 // Q8_0, two threads per row: the scale of this thread's block
    auto w_scales = [&](auto SUB) {
        constexpr int g = decltype(SUB)::value, set = MIXED ? g & 1 : 0;
        const float hd = hu[set].hd, hdmin = hu[set].hdmin;
        const uint32_t sc_lo = hu[set].sc_lo, sc_hi = hu[set].sc_hi, mn_lo = hu[set].mn_lo, mn_hi = hu[set].mn_hi;
        if (QT == QMM_Q4_K) {
            const uint32_t sc = g < 2 ? sc_lo : sc_hi, mn = g < 2 ? mn_lo : mn_hi;
            sa = hd * ubyte_f32<(2 * g) & 3>(sc);
            ba = hdmin * ubyte_f32<(2 * g) & 3>(mn);
            sb = hd * ubyte_f32<(2 * g + 1) & 3>(sc);
            bb = hdmin * ubyte_f32<(2 * g + 1) & 3>(mn);
        } else if (Q6) {
            // the thread's 16-element group(s) of the step: w = d scale (q - 32)
            const uint32_t four = g == 0 ? sc_lo : g == 1 ? sc_hi : g == 2 ? mn_lo : mn_hi;
            sa = hd * (float)(int8_t)(four >> q6_scale_shift);
            ba = -32.0f * sa;
            if (TPR == 2) { // the same byte positions of the step's second 32-element group
                sb = hd * (float)(int8_t)(four >> (q6_scale_shift + 16));
                bb = -32.0f * sb;
            }
        } else {
            const uint32_t pair = g == 0 ? sc_lo : g == 1 ? sc_hi : g == 2 ? mn_lo : mn_hi; // blocks 2g, 2g + 1
            sa = qmm_f16_bits_to_f32((uint16_t)(pair & 0xffffu));
            sb = qmm_f16_bits_to_f32((uint16_t)(pair >> 16));
            ba = -128.0f * sa;
            bb = -128.0f * sb;
            sw = w_block[set] ? sb : sa; // the thread's dwords lie in one block of 8 dwords
            bw = -128.0f * sw;
        }
    };
    const uint32_t nibble_mask = P.nibble_mask;
    uint32_t stash[4]; // finished bf16 pairs waiting for their 16-byte LDS write
    // piece H of NP of the tile with sub-block parity PAR: four of the thread's weights (Q4_K: the
    // low or the high nibbles of one dword; Q8_0: one dword), converted and, every other piece,
    // written as 16 bytes
    auto w_piece = [&](auto NSUB, auto HH, uint8_t* stage) {
        constexpr int par = decltype(NSUB)::value & 1, h = decltype(HH)::value;
        uint8_t* row = stage + w_lds[MIXED ? par : 0];
        if constexpr (Q6) {
            // dword h % 4 of the thread's 16 byte positions in its group h / 4: four elements
            constexpr int half = decltype(NSUB)::value >> 1, nib = par, gi = h / 4, dw = h % 4;
            const uint32_t v = wq[half][h], vh = wq[half][NQL + dw];
            const uint32_t q4 = (nib ? v >> 4 : v) & nibble_mask;
            const uint32_t two = (vh >> (4 * nib + 2 * gi + q6_pair_shift)) & 0x03030303u;
            const uint32_t q6 = q4 | (two << 4);
            const float sc = gi ? sb : sa, bi = gi ? bb : ba;
            constexpr int o = (h % 2) * 2;
            stash[o] = pack_bf16(__builtin_fmaf(sc, ubyte_f32<0>(q6), bi), __builtin_fmaf(sc, ubyte_f32<1>(q6), bi));
            stash[o + 1] = pack_bf16(__builtin_fmaf(sc, ubyte_f32<2>(q6), bi), __builtin_fmaf(sc, ubyte_f32<3>(q6), bi));
            if (h % 2) *reinterpret_cast<uint4*>(row + 64 * gi + 16 * (dw / 2)) = make_uint4(stash[0], stash[1], stash[2], stash[3]);
        } else if constexpr (QT == QMM_Q4_K) {
            // the thread's dword pair pp: low nibbles of both dwords, then high nibbles of both
            constexpr int pp = h / 4, hi = (h % 4) / 2;
            const uint32_t v = wq[par][2 * pp + (h % 2)];
            const uint32_t q4 = (hi ? v >> 4 : v) & nibble_mask;
            const float sc = hi ? sb : sa, bi = hi ? bb : ba;
            constexpr int o = (h % 2) * 2;
            stash[o] = pack_bf16(__builtin_fmaf(sc, ubyte_f32<0>(q4), bi), __builtin_fmaf(sc, ubyte_f32<1>(q4), bi));
            stash[o + 1] = pack_bf16(__builtin_fmaf(sc, ubyte_f32<2>(q4), bi), __builtin_fmaf(sc, ubyte_f32<3>(q4), bi));
            if (h % 2) // low nibbles: k 8 (d0 / 2 + pp) .., high nibbles: 32 elements further
                *reinterpret_cast<uint4*>(row + 64 * hi + 16 * pp) = make_uint4(stash[0], stash[1], stash[2], stash[3]);
        } else {
            // the thread's dword h: block (d0 + h) / 8 of the step
            float d, bias;
            if (TPR == 1) d = (h >> 3) ? sb : sa, bias = (h >> 3) ? bb : ba;
            else d = sw, bias = bw;
            const uint32_t u = wq[par][h] ^ 0x80808080u;
            constexpr int o = (h % 2) * 2;
            stash[o] = pack_bf16(__builtin_fmaf(d, ubyte_f32<0>(u), bias), __builtin_fmaf(d, ubyte_f32<1>(u), bias));
            stash[o + 1] = pack_bf16(__builtin_fmaf(d, ubyte_f32<2>(u), bias), __builtin_fmaf(d, ubyte_f32<3>(u), bias));
            if (h % 2) *reinterpret_cast<uint4*>(row + 16 * (h / 2)) = make_uint4(stash[0], stash[1], stash[2], stash[3]);
        }
    };

    // Operand fragments of one k16 step, two sets: the MFMAs of step kk read set kk & 1 while
    // the other set is filled.  A group of four MFMAs uses one row fragment and all column
    // fragments, so the column fragments are fetched first.
    bf16x8 fa[2][MT], fb[2][NT];
    const int frag_x = (wm * (BM / WM) + (lane & 31)) * kRowStride + (lane >> 5) * 16;
    const int frag_w = (BM + wn * (BN / 2) + (lane & 31)) * kRowStride + (lane >> 5) * 16;
    // part gi of GPK: read while group gi runs, used from group gi of the next k16 step on
    auto read_frags = [&](const uint8_t* stage, int kk, int set, auto PART) {
        constexpr int part = decltype(PART)::value;
        constexpr int jb = GPK == 1 ? 0 : NT == 3 ? (part == 0 ? 0 : NT) : NT == 4 ? (part < GPK / 2 ? part * 2 * NT / GPK : NT) : (part == 0 ? 0 : NT);
        constexpr int je = GPK == 1 ? NT : NT == 3 ? NT : NT == 4 ? (part < GPK / 2 ? (part + 1) * 2 * NT / GPK : NT) : NT;
        constexpr int ib = GPK == 1 ? 0 : NT == 3 ? 0 : NT == 4 ? (part < GPK / 2 ? 0 : (part - GPK / 2) * 2 * MT / GPK) : (part == 0 ? 0 : MT / 2);
        constexpr int ie = GPK == 1 ? MT : NT == 3 ? (part == 0 ? 0 : MT) : NT == 4 ? (part < GPK / 2 ? 0 : (part - GPK / 2 + 1) * 2 * MT / GPK) : (part == 0 ? MT / 2 : MT);
#pragma unroll
        for (int j = jb; j < je; j++)
            fb[set][j] = *reinterpret_cast<const bf16x8*>(stage + frag_w + j * 32 * kRowStride + kk * 32);
#pragma unroll
        for (int i = ib; i < ie; i++)
            fa[set][i] = *reinterpret_cast<const bf16x8*>(stage + frag_x + i * 32 * kRowStride + kk * 32);
    };

    // One k step: MFMAs out of stage SUB & 1; between them tile kt+1 goes from registers to the
    // other stage (first three quarters of the step), tile kt+2 is fetched, and after the
    // step's only barrier, which follows the last fragment reads of this stage and the last
    // writes to the other one, the first fragments of step kt+1 are read while the last quarter
    // of the MFMAs runs.  Steps past the workgroup's last one stage and fetch the (clamped) last
    // tile again: nobody uses it.
    // H: the thread's half of the waves (MIXED); threads per row of the tile staged (s) and fetched (l) meanwhile
    auto k_step = [&](int unit, auto SUB, auto H) {
        constexpr int sub = decltype(SUB)::value;
        constexpr int tprs = !MIXED || ((sub + 1) & 1) == decltype(H)::value ? TPR : 2 * TPR;
        constexpr int tprl = !MIXED || (sub & 1) == decltype(H)::value ? TPR : 2 * TPR;
        constexpr int NP = 16 / tprs, NC = nc_of(tprl); // pieces of four weights and loads per thread
        constexpr int nsub = (sub + 1) & 3, lsub = (sub + 2) & 3; // sub-block staged / fetched meanwhile
        const int kt = unit * 4 + sub;
        const uint8_t* cur = smem + (sub & 1) * kStage;
        uint8_t* next = smem + ((sub + 1) & 1) * kStage;
        static_for<4>([&](auto KK) {
            constexpr int kk = decltype(KK)::value;
            static_for<GPK>([&](auto GI) {
                constexpr int gi = decltype(GI)::value;
                constexpr int g = kk * GPK + gi;
                // the operands of the next k16 step (of the next k step in the last quarter)
                read_frags(kk < 3 ? cur : next, (kk + 1) & 3, (kk + 1) & 1, GI);
#pragma unroll
                for (int q = 0; q < GS; q++) {
                    const int t = gi * GS + q, i = t / NT, j = t % NT;
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[kk & 1][j], fa[kk & 1][i], acc[i][j], 0, 0, 0);
                }
                // group g's share of staging tile kt+1 (the thread's NP weight pieces and XC
                // activation chunks over the first 3 NG / 4 groups) and of fetching tile kt+2
                constexpr int NGS = 3 * NG / 4;
                constexpr int p0 = (NP * g + NGS - 1) / NGS, p1 = g < NGS ? (NP * (g + 1) + NGS - 1) / NGS : p0;
                constexpr int c0 = (XC * g + NGS - 1) / NGS, c1 = g < NGS ? (XC * (g + 1) + NGS - 1) / NGS : c0;
                constexpr int l0 = g == 0 ? 0 : (XC * (g - 1) + NGS - 1) / NGS, l1 = g == 0 ? 0 : c0; // chunks written a group ago
                if (g == 0) {
                    if (sub == 3) w_unpack(); // tile kt+1 opens the next unit: its header arrived a step ago
                    w_scales(std::integral_constant<int, nsub>{});
                }
                static_for<p1 - p0>([&](auto PI) {
                    w_piece(std::integral_constant<int, nsub>{},
                            std::integral_constant<int, (p0 + decltype(PI)::value) % NP>{}, next);
                });
                constexpr int xbuf = (sub + 1) % XD; // registers of tile kt+1, refilled with tile kt+1+XD
#pragma unroll
                for (int i = c0; i < c1; i++) x_write(kt + 1, xbuf, i, next);
#pragma unroll
                for (int i = l0; i < (g <= NGS ? l1 : l0); i++) x_load(kt + 1 + XD, xbuf, i);
                // Q6_K fetches by half units, a step earlier: step 1 requests the low nibbles of the
                // next unit's first half, step 2 its bit pairs, step 3 the low nibbles of the second
                // half and step 0 (of that unit) its bit pairs; each half is complete one step before
                // its first tile is dequantized
                if (g == 1 && sub == (Q6 ? 1 : 2)) advance_cursor();
                if (g == 1 && sub == 2) w_load_hdr();
                if (g >= 2 && g < 2 + NC) {
                    if constexpr (!Q6) w_load_q(std::integral_constant<int, lsub>{}, std::integral_constant<int, tprl>{}, g - 2);
                    else if constexpr (sub % 2 == 1 || g == 2)
                        w_load_q6(std::integral_constant<int, (sub == 0 || sub == 3) ? 1 : 0>{},
                                  std::integral_constant<int, (sub % 2 == 0) ? 1 : 0>{}, g - 2);
                }
                // inside the group: one MFMA, then its share of the other instructions, so
                // the matrix pipe is fed while they issue
                constexpr int valu = (Q6 || GS == 3 ? 4 : 3) * (p1 - p0) + (g == 0 ? 4 : 1);
                constexpr int reads = GPK == 1 ? NT + MT : NT == 3 ? (gi == 0 ? NT : MT) : NT == 4 ? (gi < GPK / 2 ? 2 * NT / GPK : 2 * MT / GPK) : (gi == 0 ? NT + MT / 2 : MT / 2);
#pragma unroll
                for (int q = 0; q < GS; q++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, valu, 0);
                    if (q == 0) __builtin_amdgcn_sched_group_barrier(0x100, (reads + 1) / 2, 0);
                    if (q == 1) __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
                    if (q == 2) __builtin_amdgcn_sched_group_barrier(0x100, reads / 2, 0);
                    if (q == GS - 1) __builtin_amdgcn_sched_group_barrier(0x200, 3, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if (kk == 2) {
                // this stage's fragments are all in registers, the other stage is complete
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };

    if (u0 < u1) {
        // ---- prologue: tile (u0, 0) -> stage 0, tile (u0, 1) -> registers
        auto run = [&](auto H) {
            constexpr int tpr0 = !MIXED || decltype(H)::value == 0 ? TPR : 2 * TPR, tpr1 = !MIXED || decltype(H)::value == 1 ? TPR : 2 * TPR;
#pragma unroll
            for (int i = 0; i < XC; i++) x_load(u0 * 4, 0, i);
            w_load_hdr();
#pragma unroll
            for (int c = 0; c < nc_of(tpr0); c++) {
                if constexpr (Q6) {
                    w_load_q6(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, c);
                    if (c == 0) w_load_q6(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{}, 0);
                } else {
                    w_load_q(std::integral_constant<int, 0>{}, std::integral_constant<int, tpr0>{}, c);
                }
            }
#pragma unroll
            for (int i = 0; i < XC; i++) x_write(u0 * 4, 0, i, smem);
            w_unpack();
            w_scales(std::integral_constant<int, 0>{});
            static_for<16 / tpr0>([&](auto HH) { w_piece(std::integral_constant<int, 0>{}, HH, smem); });
#pragma unroll
            for (int d = 1; d <= XD; d++)
#pragma unroll
                for (int i = 0; i < XC; i++) x_load(u0 * 4 + d, d % XD, i);
#pragma unroll
            for (int c = 0; c < nc_of(tpr1); c++) {
                if constexpr (Q6) w_load_q6(std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{}, c);
                else w_load_q(std::integral_constant<int, 1>{}, std::integral_constant<int, tpr1>{}, c);
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            static_for<GPK>([&](auto PART) { read_frags(smem, 0, 0, PART); });

            for (int unit = u0; unit < u1; unit++) static_for<4>([&](auto SUB) { k_step(unit, SUB, H); });
        };
        if constexpr (MIXED) {
            if (__builtin_amdgcn_readfirstlane(wave) < NW / 2) run(std::integral_constant<int, 0>{});
            else run(std::integral_constant<int, 1>{});
        } else {
            run(std::integral_constant<int, 0>{});
        }
    }

    // ---- epilogue.  The weights are the matrix instruction's first operand, so a lane holds four consecutive columns at a time
    // of one activation row: 32 rows of the wave's columns go through the wave's own LDS (f32) and leave in whole 16-byte
    // pieces of a row, the residual comes in as such.  (Stored from the accumulators, two bytes a lane, a 2048 x 4096 product
    // with a bf16 residual took 92 us, 75 without.)
    constexpr int COLS = BN / 2, kOutStride = COLS * 4 + 16;
    static_assert(NW * 32 * kOutStride <= 2 * kStage);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); // every wave has read its last fragments
    uint8_t* out_lds = smem + wave * (32 * kOutStride);
    const bool f32_out = P.partial || !P.out_bf16;
    RowsOut R; // a split-k slice: its own f32 [m, n] plane, which the second kernel finishes
    R.out = P.partial ? P.partial + (int64_t)blockIdx.y * P.m * P.n : P.y, R.residual = P.partial ? nullptr : P.residual;
    R.m = P.m, R.n = P.n, R.n_end = P.n_end, R.col0 = n0 + wn * COLS;
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    auto four = [&](int row, int col) { return *reinterpret_cast<const f32x4*>(out_lds + row * kOutStride + col * 4); };
    auto one = [&](int row, int col) { return *reinterpret_cast<const float*>(out_lds + row * kOutStride + col * 4); };
    auto rows_out = [&](auto W) {
        constexpr int w = decltype(W)::value, PASSES = COLS / w / 2, CH = PASSES > 8 ? PASSES / 2 : PASSES;
        static_for<PASSES / CH>([&](auto C) {
            RowPieces<COLS, w, decltype(C)::value * CH, CH> pieces;
            pieces.request(R, lane);
            pieces.store(R, lane, four);
        });
    };
    const bool whole = whole_pieces(R);
    static_for<MT>([&](auto I) {
        constexpr int i = decltype(I)::value;
        lanes_exchange(); // (the rows before these have been read)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *reinterpret_cast<f32x4*>(out_lds + (lane & 31) * kOutStride + (j * 32 + 8 * g + 4 * (lane >> 5)) * 4) =
                    f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        lanes_exchange();
        R.row0 = m0 + wm * (BM / WM) + i * 32;
        if (!whole && f32_out) store_values<COLS, true>(R, lane, one); // uniform
        else if (!whole) store_values<COLS, false>(R, lane, one);
        else if (f32_out) rows_out(std::integral_constant<int, 4>{});
        else rows_out(std::integral_constant<int, 8>{});
    });
}

// out[i] = sum over slices (in order) of partial[s][i], as f32 or bf16; i runs over the
// columns [n_begin, n_end) of all rows
// EIGHT: whole planes, eight values per thread in 16-byte pieces (m n a multiple of eight, everything aligned to 16 bytes).
// Bound by memory: the product 2048 x 4096, k = 12288, in two slices with a bf16 residual (100 MB here), 205 us with the reduction
// value by value, 194 by pieces; Q8_0 217 / 200.
template <bool EIGHT>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial, int slices, int64_t m, int64_t n,
                                                            int64_t n_begin, int64_t n_end, void* y, int out_bf16, const void* residual) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if constexpr (!EIGHT) {
        const int64_t width = n_end - n_begin;
        if (idx >= m * width) return;
        const int64_t row = idx / width, col = n_begin + (idx - row * width);
        float sum = 0.0f;
        for (int s = 0; s < slices; s++) sum += partial[((int64_t)s * m + row) * n + col];
        qmm_store(y, QmmEpilogue{residual, out_bf16}, row * n + col, sum);
        return;
    }
    const int64_t i = idx * 8, count = m * n;
    if (i >= count) return;
    f32x4 res[2] = {};
    if (residual && out_bf16) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(residual) + i);
#pragma unroll
        for (int e = 0; e < 4; e++)
            res[e >> 1][2 * (e & 1)] = __uint_as_float(v[e] << 16), res[e >> 1][2 * (e & 1) + 1] = __uint_as_float(v[e] & 0xffff0000u);
    } else if (residual) {
        res[0] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(residual) + i);
        res[1] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(residual) + i + 4);
    }
    f32x4 sum[2] = {};
    for (int s = 0; s < slices; s++) {
        const f32x4* p = reinterpret_cast<const f32x4*>(partial + s * count + i);
        sum[0] += p[0], sum[1] += p[1];
    }
    if (residual) sum[0] += res[0], sum[1] += res[1];
    if (out_bf16) {
        *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(y) + i) = u32x4{pack_bf16(sum[0].x, sum[0].y), pack_bf16(sum[0].z, sum[0].w),
                                                                         pack_bf16(sum[1].x, sum[1].y), pack_bf16(sum[1].z, sum[1].w)};
    } else {
        *reinterpret_cast<f32x4*>(static_cast<float*>(y) + i) = sum[0];
        *reinterpret_cast<f32x4*>(static_cast<float*>(y) + i + 4) = sum[1];
    }
}
hipError_t launch_splitk_reduce(const float* partial, int slices, int64_t m, int64_t n, int64_t n_begin, int64_t n_end, void* y, int out_bf16,
                                const void* residual, hipStream_t stream) {
    const int64_t count = m * (n_end - n_begin);
    const uintptr_t at = reinterpret_cast<uintptr_t>(partial) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(residual);
    if (n_begin == 0 && n_end == n && count % 8 == 0 && at % 16 == 0)
        splitk_reduce_kernel<true><<<(unsigned)((count / 8 + 255) / 256), 256, 0, stream>>>(partial, slices, m, n, 0, n, y, out_bf16, residual);
    else
        splitk_reduce_kernel<false><<<(unsigned)((count + 255) / 256), 256, 0, stream>>>(partial, slices, m, n, n_begin, n_end, y, out_bf16, residual);
    return hipGetLastError();
}

__global__ void f32_to_bf16_kernel(const float* __restrict__ x, uint16_t* __restrict__ out,
                                   int64_t count) {
    int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i + 4 <= count) {
        float4 f = *reinterpret_cast<const float4*>(x + i);
        uint2 o;
        o.x = pack_bf16(f.x, f.y);
        o.y = pack_bf16(f.z, f.w);
        *reinterpret_cast<uint2*>(out + i) = o;
    } else {
        for (; i < count; i++) out[i] = qmm_f32_to_bf16_bits(x[i]);
    }
}

__global__ void epilogue_kernel(const float* __restrict__ t, const void* residual, void* y, int y_bf16,
                                int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) qmm_store(y, QmmEpilogue{residual, y_bf16}, i, t[i]);
}

__global__ void bf16_to_f32_kernel(const uint16_t* __restrict__ x, float* __restrict__ out, int64_t count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) out[i] = qmm_bf16_bits_to_f32(x[i]);
}

template <int QT, int BM, int BN>
hipError_t launch_tile(GemmParams P, int slices, hipStream_t stream) {
    constexpr int NW = 8;
    P.tiles_m = (int)((P.m + BM - 1) / BM);
    P.tiles_n = (int)((P.n_end - P.n_begin + BN - 1) / BN);
    if (P.n_weights > 1) { // a projection group: the members' column tiles one after the other
        int64_t t = 0;
        for (int i = 0; i < P.n_weights; i++) P.tn_end[i] = (int)(t += (P.nv[i] + BN - 1) / BN);
        P.tiles_n = (int)t;
    }
    const int64_t grid = (int64_t)P.tiles_m * P.tiles_n;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    constexpr size_t lds = (size_t)2 * (BM + BN) * kRowStride;
    const bool x_tail = QT == QMM_Q8_0 && (P.k & 63) != 0; // the K-quant types have k a multiple of 256
    auto fn = x_tail ? &gemm_pipe_kernel<QT, BM, BN, QT == QMM_Q8_0, NW> : &gemm_pipe_kernel<QT, BM, BN, false, NW>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    float* partial = P.partial;
    if (slices > 1) P.slice_units = (P.k_units + slices - 1) / slices;
    else P.partial = nullptr;
    fn<<<dim3((unsigned)grid, (unsigned)slices), dim3(64 * NW), lds, stream>>>(P);
    if (slices > 1 && P.n_weights > 1) {
        for (int i = 0; i < P.n_weights; i++)
            if ((e = launch_splitk_reduce(P.partial_v[i], slices, P.m, P.nv[i], 0, P.nv[i], P.yv[i], P.out_bf16, nullptr, stream)) != hipSuccess)
                return e;
    } else if (slices > 1) {
        return launch_splitk_reduce(partial, slices, P.m, P.n, P.n_begin, P.n_end, P.y, P.out_bf16, P.residual, stream);
    }
    return hipGetLastError();
}

// How a [m, n] x k product is cut into launches.  Big tiles reuse each LDS byte most, but
// the grid runs in rounds of one workgroup per CU and a partly filled last round idles
// CUs; a product with few tiles can be split along k (each slice writes an f32 tile, a
// second kernel adds the slices in order).  Costs are in k steps of a 256 x 256 tile
// (relative tile efficiencies measured on the 8B shapes).
struct GemmPlan {
    int bm, bn;          // tile of the only / the second launch: 256 x 256, 256 x 192 (Q4_K, Q8_0) or 256 x 128
    int slices;          // split along k
    int64_t full_cols;   // > 0: first a launch of 256 x 256 tiles over this many 256-column strips
};

// IZWI_QMM_GEMM_TILE="bm,bn,slices,strips" (tuning aid; the last two 1 and 0 if left out) replaces the plan, at every number of
// rows, and the choice of the few-row kernel: bm = 256, bn in {128, 192, 256}.
bool forced_plan(GemmPlan& plan) {
    static const GemmPlan forced = [] {
        GemmPlan p{0, 0, 1, 0};
        const char* e = getenv("IZWI_QMM_GEMM_TILE");
        int strips = 0;
        if (e && sscanf(e, "%d,%d,%d,%d", &p.bm, &p.bn, &p.slices, &strips) >= 2) {
            const bool ok = p.bm == 256 && (p.bn == 128 || p.bn == 192 || p.bn == 256) && p.slices >= 1 && p.slices <= 8 && strips >= 0;
            if (!ok) p.bm = p.bn = 0, p.slices = 1;
            else p.full_cols = strips;
        }
        return p;
    }();
    if (forced.bm == 0) return false;
    plan = forced;
    return true;
}

// 192-column tiles of the members; 0 for the types that have no such tile
int64_t tiles_of_192(const QmmLayout* const* layouts, int n_weights) {
    int64_t t = 0;
    for (int i = 0; i < n_weights; i++) t += (layouts[i]->n + 191) / 192;
    return n_weights > 0 && layouts[0]->dtype == QMM_Q6_K ? 0 : t;
}

// `n_weights` members planned as one matrix of n columns (a group: more than one, or a split's sums per member)
GemmPlan plan_gemm(int64_t m, int64_t n, int k_steps, int n_cus, int64_t tiles_n192, int n_weights = 1) {
    const double kQ128 = 0.76; // relative rate of a half-size tile
    // A 256 x 192 tile takes 0.82 of the time of a whole one.  Where whole tiles would fill the last round badly, us per call (2 x
    // 12288 x 4096, Q4_K): 112 -> 105 at 500 rows (192 whole tiles, 256 of these), 212 -> 182 at 640 (288, 384), 217 ->
    // 197 at 1000 (384, 512), 330 -> 290 at 1400 (576, 768); 2 x 3072 x 1024 42 -> 37 at 2048 rows (192, 256).
    const double kCost192 = 0.82;
    const int hm = 256, hn = 128;
    {
        GemmPlan forced;
        if (forced_plan(forced)) {
            while (forced.slices > 1 && k_steps / 4 < forced.slices) forced.slices /= 2;
            if (forced.bn == 192 && tiles_n192 == 0) forced.bn = 256;
            if (n_weights > 1 || forced.full_cols * 256 >= n) forced.full_cols = 0;
            return forced;
        }
    }
    auto tiles = [&](int bm, int bn, int64_t cols) { return ((m + bm - 1) / bm) * ((cols + bn - 1) / bn); };
    auto rounds = [&](int64_t t) { return (double)((t + n_cus - 1) / n_cus); };
    GemmPlan best{256, 256, 1, 0};
    double best_cost = rounds(tiles(256, 256, n)) * k_steps;
    auto consider = [&](GemmPlan p, double cost) {
        if (cost < 0.98 * best_cost) best = p, best_cost = cost;
    };
    consider({hm, hn, 1, 0}, rounds(tiles(hm, hn, n)) * k_steps * 0.5 / kQ128);
    if (tiles_n192 > 0) consider({256, 192, 1, 0}, rounds((m + 255) / 256 * tiles_n192) * k_steps * kCost192);
    // whole rounds of 256 x 256 tiles first, the remaining columns as half-size tiles
    const int64_t tiles_m256 = (m + 255) / 256, cols256 = (n + 255) / 256;
    const int64_t full_cols = (tiles_m256 * cols256 / n_cus) * n_cus / tiles_m256;
    if (n_weights == 1 && full_cols > 0 && full_cols < cols256)
        consider({hm, hn, 1, full_cols},
                 (double)(tiles_m256 * full_cols / n_cus) * k_steps +
                     rounds(tiles(hm, hn, n - full_cols * 256)) * k_steps * 0.5 / kQ128);
    // split along k: the slices' f32 tiles are written in the launch and read by a second one per member (4.5 us, and 2 TB/s for
    // both ways; a 256 x 256 k step takes 1.9 us).  Constants from every form of 249 products (15 shapes, three types, 129 to 3000
    // rows): the plan's form takes 1.001 of the best one's time in the mean, 1.045 at worst.  Priced at one launch and the
    // reads alone (3 us, 4.5 TB/s), splits were taken where they cost 5 to 20 %: 2 x 6144 x 2048 at 400 rows 37.9 / 44.9 in two slices of
    // 192 columns, 4096 x 12288 at 1400 rows 163 in two slices / 196 in eight, 8192 x 8192 at 1400 rows 203 / 237 in four.
    // Where a split pays (bf16 residual): 4096 x 12288 at 1400 rows, 256 x 256 whole 252, in two slices 163.
    for (int slices = 2; slices <= 8; slices *= 2) {
        if (k_steps / slices < 8) break;
        const double reduce_cost = (slices * (double)m * (double)n * 4.0 / 2e6 + 4.5 * n_weights) / 1.9;
        const double steps = 4.0 * (double)((k_steps / 4 + slices - 1) / slices); // slices are whole units
        consider({256, 256, slices, 0}, rounds(tiles(256, 256, n) * slices) * steps + reduce_cost);
        if (tiles_n192 > 0)
            consider({256, 192, slices, 0}, rounds((m + 255) / 256 * tiles_n192 * slices) * steps * kCost192 + reduce_cost);
        consider({hm, hn, slices, 0}, rounds(tiles(hm, hn, n) * slices) * steps * 0.5 / kQ128 + reduce_cost);
    }
    return best;
}

template <int QT>
hipError_t launch_qt(const GemmParams& P0, int n_cus, hipStream_t stream) {
    const GemmPlan plan = plan_gemm(P0.m, P0.n, P0.k_units * 4, n_cus, QT == QMM_Q6_K ? 0 : (P0.n + 191) / 192);
    GemmParams P = P0;
    P.n_begin = 0;
    P.n_end = P0.n;
    if (plan.slices > 1 && P0.partial == nullptr) return hipErrorInvalidValue;
    if (plan.full_cols > 0) {
        P.n_end = plan.full_cols * 256;
        hipError_t e = launch_tile<QT, 256, 256>(P, 1, stream);
        if (e != hipSuccess) return e;
        P.n_begin = P.n_end;
        P.n_end = P0.n;
    }
    if constexpr (QT != QMM_Q6_K) {
        if (plan.bn == 192) return launch_tile<QT, 256, 192>(P, plan.slices, stream);
    }
    return plan.bn == 256 ? launch_tile<QT, 256, 256>(P, plan.slices, stream) : launch_tile<QT, 256, 128>(P, plan.slices, stream);
}

// n of the single matrix a group is planned as: the members' columns, each rounded up to whole
// 256-column strips
int64_t group_columns(const QmmLayout* const* layouts, int n_weights) {
    int64_t n = 0;
    for (int i = 0; i < n_weights; i++) n += (layouts[i]->n + 255) / 256 * 256;
    return n;
}

template <int QT>
hipError_t launch_group_qt(GemmParams P, int64_t n_planned, int64_t tiles_n192, int n_cus, hipStream_t stream) {
    const GemmPlan plan = plan_gemm(P.m, n_planned, P.k_units * 4, n_cus, tiles_n192, P.n_weights);
    if (plan.slices > 1) {
        if (P.partial == nullptr) return hipErrorInvalidValue;
        float* base = P.partial;
        for (int i = 0; i < P.n_weights; i++) {
            P.partial_v[i] = base;
            base += (size_t)plan.slices * (size_t)P.m * (size_t)P.nv[i];
        }
    }
    if constexpr (QT != QMM_Q6_K) {
        if (plan.bn == 192) return launch_tile<QT, 256, 192>(P, plan.slices, stream);
    }
    return plan.bn == 256 ? launch_tile<QT, 256, 256>(P, plan.slices, stream) : launch_tile<QT, 256, 128>(P, plan.slices, stream);
}

} // namespace

bool qmm_gemm_tile_forced() {
    GemmPlan plan;
    return forced_plan(plan);
}

// a group takes the plane form when every member can
static bool group_plane_applies(const QmmLayout* const* layouts, int n_weights, int64_t m) {
    for (int i = 0; i < n_weights; i++)
        if (!qmm_gemm_plane_applies(*layouts[i], m) || layouts[i]->k != layouts[0]->k) return false;
    return n_weights >= 1;
}

size_t qmm_gemm_group_workspace_bytes(const QmmLayout* const* layouts, int n_weights, int64_t m, int n_cus) {
    if (n_weights < 2) return 0;
    if (n_cus <= 0) n_cus = 1;
    if (qmm_gemm_regb_applies(layouts, n_weights, m, n_cus)) return qmm_gemm_regb_workspace_bytes(layouts, n_weights, m, n_cus);
    if (group_plane_applies(layouts, n_weights, m)) {
        size_t total = 0;
        for (int i = 0; i < n_weights; i++) total += qmm_gemm_plane_bytes(*layouts[i]);
        return total;
    }
    const GemmPlan plan = plan_gemm(m, group_columns(layouts, n_weights), (int)layouts[0]->k_units * 4, n_cus,
                                    tiles_of_192(layouts, n_weights), n_weights);
    if (plan.slices <= 1) return 0;
    size_t total = 0;
    for (int i = 0; i < n_weights; i++) total += (size_t)plan.slices * (size_t)m * (size_t)layouts[i]->n * sizeof(float);
    return total;
}

hipError_t qmm_launch_gemm_bf16_multi(const QmmLayout* const* layouts, const void* const* tiled, int n_weights,
                                      const uint16_t* x_bf16, int64_t m, void* const* ys, int out_bf16,
                                      void* workspace, int n_cus, hipStream_t stream) {
    if (n_weights < 2 || n_weights > QMM_MAX_GROUP) return hipErrorInvalidValue;
    if (n_cus <= 0) n_cus = 1;
    if (qmm_gemm_regb_applies(layouts, n_weights, m, n_cus))
        return qmm_launch_gemm_regb(layouts, tiled, n_weights, x_bf16, m, ys, out_bf16, workspace, n_cus, stream);
    if (group_plane_applies(layouts, n_weights, m)) {
        if (workspace == nullptr) return hipErrorInvalidValue;
        return qmm_launch_gemm_plane(layouts, tiled, n_weights, x_bf16, m, ys, out_bf16, workspace, n_cus, stream);
    }
    const QmmLayout& L0 = *layouts[0];
    GemmParams P;
    P.w = (const uint8_t*)tiled[0];
    P.x = x_bf16;
    P.y = ys[0];
    P.m = m;
    P.n = L0.n;
    P.n_begin = 0;
    P.n_end = L0.n;
    P.k = L0.k;
    P.k_units = (int)L0.k_units;
    P.k_groups = (int)L0.k_groups;
    P.s = L0.s;
    P.slots = L0.slots;
    P.row_tiles = L0.row_tiles;
    P.panel_bytes = L0.panel_bytes;
    P.out_bf16 = out_bf16;
    P.tiles_m = P.tiles_n = 0;
    P.slice_units = 0;
    P.nibble_mask = 0x0f0f0f0fu;
    P.partial = (float*)workspace;
    P.residual = nullptr;
    P.n_weights = n_weights;
    for (int i = 0; i < n_weights; i++) {
        const QmmLayout& L = *layouts[i];
        if (L.dtype != L0.dtype || L.k != L0.k || L.n_stacked != 1 || L.n == 0) return hipErrorInvalidValue;
        P.wv[i] = (const uint8_t*)tiled[i];
        P.yv[i] = ys[i];
        P.nv[i] = L.n;
        P.row_tiles_v[i] = L.row_tiles;
        P.partial_v[i] = nullptr;
        P.tn_end[i] = 0;
    }
    const int64_t n_planned = group_columns(layouts, n_weights), n192 = tiles_of_192(layouts, n_weights);
    if (L0.dtype == QMM_Q6_K) return launch_group_qt<QMM_Q6_K>(P, n_planned, n192, n_cus, stream);
    return L0.dtype == QMM_Q4_K ? launch_group_qt<QMM_Q4_K>(P, n_planned, n192, n_cus, stream)
                                : launch_group_qt<QMM_Q8_0>(P, n_planned, n192, n_cus, stream);
}

size_t qmm_gemm_workspace_bytes(const QmmLayout& L, int64_t m, int n_cus) {
    if (m <= 0 || L.n == 0) return 0;
    if (n_cus <= 0) n_cus = 1;
    const QmmLayout* lp = &L;
    if (qmm_gemm_regb_applies(&lp, 1, m, n_cus)) return qmm_gemm_regb_workspace_bytes(&lp, 1, m, n_cus);
    if (qmm_gemm_plane_applies(L, m)) return qmm_gemm_plane_bytes(L);
    const GemmPlan plan = plan_gemm(m, L.n, (int)L.k_units * 4, n_cus, tiles_of_192(&lp, 1));
    return plan.slices > 1 ? (size_t)plan.slices * (size_t)m * (size_t)L.n * sizeof(float) : 0;
}

hipError_t qmm_launch_gemm_bf16(const QmmLayout& L, const void* tiled, const uint16_t* x_bf16,
                                int64_t m, void* y, int out_bf16, void* workspace, int n_cus,
                                hipStream_t stream, const void* residual) {
    if (m <= 0 || L.n == 0) return hipSuccess;
    if (n_cus <= 0) n_cus = 1;
    const QmmLayout* lp = &L;
    if (qmm_gemm_regb_applies(&lp, 1, m, n_cus))
        return qmm_launch_gemm_regb(&lp, &tiled, 1, x_bf16, m, &y, out_bf16, workspace, n_cus, stream, residual);
    if (qmm_gemm_plane_applies(L, m)) {
        if (workspace == nullptr) return hipErrorInvalidValue;
        return qmm_launch_gemm_plane(&lp, &tiled, 1, x_bf16, m, &y, out_bf16, workspace, n_cus, stream, residual);
    }
    GemmParams P;
    P.w = (const uint8_t*)tiled;
    P.x = x_bf16;
    P.y = y;
    P.m = m;
    P.n = L.n;
    P.n_begin = 0;
    P.n_end = L.n;
    P.k = L.k;
    P.k_units = (int)L.k_units;
    P.k_groups = (int)L.k_groups;
    P.s = L.s;
    P.slots = L.slots;
    P.row_tiles = L.row_tiles;
    P.panel_bytes = L.panel_bytes;
    P.out_bf16 = out_bf16;
    P.tiles_m = P.tiles_n = 0;
    P.slice_units = 0;
    P.nibble_mask = 0x0f0f0f0fu;
    P.partial = (float*)workspace;
    P.residual = residual;
    P.n_weights = 0;
    if (L.dtype == QMM_Q6_K) return launch_qt<QMM_Q6_K>(P, n_cus, stream);
    return L.dtype == QMM_Q4_K ? launch_qt<QMM_Q4_K>(P, n_cus, stream)
                               : launch_qt<QMM_Q8_0>(P, n_cus, stream);
}

hipError_t qmm_launch_f32_to_bf16(const float* x, uint16_t* out, int64_t count,
                                  hipStream_t stream) {
    if (count <= 0) return hipSuccess;
    int64_t threads = (count + 3) / 4;
    f32_to_bf16_kernel<<<(unsigned)((threads + 255) / 256), 256, 0, stream>>>(x, out, count);
    return hipGetLastError();
}

hipError_t qmm_launch_epilogue(const float* t, const void* residual, void* y, int y_bf16, int64_t count,
                               hipStream_t stream) {
    if (count <= 0) return hipSuccess;
    if ((count + 255) / 256 > 0x7fffffff) return hipErrorInvalidValue;
    epilogue_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>(t, residual, y, y_bf16, count);
    return hipGetLastError();
}

hipError_t qmm_launch_bf16_to_f32(const uint16_t* x, float* out, int64_t count, hipStream_t stream) {
    if (count <= 0) return hipSuccess;
    if ((count + 255) / 256 > 0x7fffffff) return hipErrorInvalidValue;
    bf16_to_f32_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>(x, out, count);
    return hipGetLastError();
}
