// Device helpers of the matrix-core tile kernels (prefill and expert products).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

namespace {

template <int N, class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
// f(0), f(1), .. f(N - 1) with compile-time indexes
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    bf16x2 v = {(__bf16)a, (__bf16)b}; // v_cvt_pk_bf16_f32: round to nearest even
    return __builtin_bit_cast(uint32_t, v);
}

// byte N of v as float (v_cvt_f32_ubyteN)
template <int N>
__device__ __forceinline__ float ubyte_f32(uint32_t v) {
    return (float)((v >> (8 * N)) & 0xffu);
}

// 16 (4) bytes per lane from global memory straight into LDS: lane l's bytes land at lds + 16 l (4 l).
__device__ __forceinline__ void load_to_lds(const uint8_t* base, uint32_t lane_off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(lane_off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void load_to_lds4(const uint8_t* base, uint32_t lane_off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(lane_off), "s"(base) : "memory", "m0");
}

// Between a wave's writes to LDS and its reads of what other lanes wrote, or the other way round: its LDS instructions run in
// their order, this keeps the compiler from changing it (it sees one lane's addresses).  No instruction.
__device__ __forceinline__ void lanes_exchange() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// A wave's 32 rows of results from (row0, col0) on, which stand as f32 in its own LDS, on their way to memory.
struct RowsOut {
    void* out;            // the matrix of m x n values; columns from n_end on are not written
    const void* residual; // null: none.  It may be the output: a lane reads what it writes
    int64_t m, n, n_end, row0, col0;
};
// whole pieces of 16 bytes: rows of a multiple of eight values that start on 16 bytes
__device__ __forceinline__ bool whole_pieces(const RowsOut& R) {
    return R.n % 8 == 0 && ((reinterpret_cast<uintptr_t>(R.out) | reinterpret_cast<uintptr_t>(R.residual)) & 15) == 0;
}
// Pieces FIRST .. FIRST + COUNT - 1 of each lane, W columns each (4 of f32, 8 of bf16: 16 bytes of the output), consecutive lanes
// on consecutive pieces of the COLS columns.  request: the residual's loads, all at once; store: sums from value(row, column of
// four), and out.
template <int COLS, int W, int FIRST, int COUNT>
struct RowPieces {
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    static_assert(32 * COLS / W % 64 == 0);
    int64_t at[COUNT]; // index of the piece, negative: outside
    u32x4 res[COUNT];
    static __device__ __forceinline__ int row(int q, int lane) { return ((FIRST + q) * 64 + lane) / (COLS / W); }
    static __device__ __forceinline__ int col(int q, int lane) { return ((FIRST + q) * 64 + lane) % (COLS / W) * W; }
    __device__ __forceinline__ void request(const RowsOut& R, int lane) {
#pragma unroll
        for (int q = 0; q < COUNT; q++) {
            const int64_t gm = R.row0 + row(q, lane), gn = R.col0 + col(q, lane);
            at[q] = gm < R.m && gn < R.n_end ? gm * R.n + gn : -1;
            res[q] = u32x4{0, 0, 0, 0};
            if (R.residual && at[q] >= 0) res[q] = *reinterpret_cast<const u32x4*>(static_cast<const uint8_t*>(R.residual) + at[q] * (16 / W));
        }
    }
    template <class F>
    __device__ __forceinline__ void store(const RowsOut& R, int lane, F&& value) const {
#pragma unroll
        for (int q = 0; q < COUNT; q++) {
            f32x4 v[W / 4];
#pragma unroll
            for (int e = 0; e < W / 4; e++) v[e] = value(row(q, lane), col(q, lane) + 4 * e);
            if (R.residual) // uniform
#pragma unroll
                for (int e = 0; e < W; e++)
                    v[e >> 2][e & 3] += __uint_as_float(W == 4 ? res[q][e & 3] : e & 1 ? res[q][e >> 1] & 0xffff0000u : res[q][e >> 1] << 16);
            u32x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++)
                o[e] = W == 4 ? __float_as_uint(v[0][e]) : pack_bf16(v[e * W / 16][2 * e & 3], v[e * W / 16][(2 * e & 3) + 1]);
            if (at[q] >= 0) *reinterpret_cast<u32x4*>(static_cast<uint8_t*>(R.out) + at[q] * (16 / W)) = o;
        }
    }
};
// The same value by value, where pieces are not whole: 16 rows of 32 columns at a time, their residuals together.
// (Kept short: it is not in the instruction cache when a workgroup gets here, 600 instructions of it took 4 us.)
template <int COLS, bool F32, class F>
__device__ __forceinline__ void store_values(const RowsOut& R, int lane, F&& value) {
    typedef std::conditional_t<F32, float, uint16_t> T;
#pragma unroll 1
    for (int part = 0; part < COLS / 16; part++) {
        const int col = part / 2 * 32 + (lane & 31), row = part % 2 * 16 + (lane >> 5); // the lane's: row, row + 2, .. + 14
        const int rows = (int)min((int64_t)16, R.m - R.row0 - row);
        const int64_t at = (R.row0 + row) * R.n + R.col0 + col;
        if (R.col0 + col >= R.n_end || rows <= 0) continue;
        float v[8];
        if (R.residual) { // uniform
            const T* from = static_cast<const T*>(R.residual) + at;
            T res[8];
#pragma unroll
            for (int q = 0; q < 8; q++) res[q] = from[min(2 * q, (rows - 1) & ~1) * R.n];
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = F32 ? (float)res[q] : __uint_as_float((uint32_t)res[q] << 16);
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = value(row + 2 * q, col) + v[q];
        } else {
#pragma unroll
            for (int q = 0; q < 8; q++) v[q] = value(row + 2 * q, col);
        }
        T* to = static_cast<T*>(R.out) + at;
#pragma unroll
        for (int q = 0; q < 8; q++, to += 2 * R.n)
            if (2 * q < rows) {
                if constexpr (F32) *to = v[q];
                else *to = (uint16_t)pack_bf16(v[q], v[q]);
            }
    }
}

} // namespace
