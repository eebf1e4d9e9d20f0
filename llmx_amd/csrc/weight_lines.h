// How the weight-streaming products (bf16 and float32) ask memory for a strip of 16 weight rows.
//
// A step of the matrix instruction takes 64 bytes of each row, lane (r, kg) the 16 bytes kg of row r; memory gives and the caches keep lines
// of 128.  So two steps come together as whole lines, eight rows' each, and the halves that belong to another lane are exchanged between
// lanes 8 apart in a row of 16: lane (r, kg) asks for chunk kg + 4 (r / 8) (of 8 of 16 bytes) of rows r % 8 and 8 + r % 8.  Whole lines can
// be asked for as bytes that are read once (LINES), which the caches then do not keep: a kernel that only reads gets 7.1 TB/s that way and
// 6.3 without, and what a step's other kernels read stays near; half lines asked for so arrive twice (5.6 TB/s).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint32_t line_u32x4_t __attribute__((ext_vector_type(4)));

struct WeightLines {
    line_u32x4_t lo, hi;     // of rows r % 8 and 8 + r % 8
};
// A strip's rows as the loads see them: 32-bit byte offsets from a base the wave shares; what lies past the strip's bytes reads as 0.
typedef __amdgpu_buffer_rsrc_t strip_t;
__device__ __forceinline__ strip_t strip_of(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ uint32_t line_chunk(int r, int kg) { return 16 * kg + 64 * (r >> 3); }     // the lane's byte of a line
// at: the lane's byte of row r % 8 (its row and line_chunk); next: bytes from a row to the eighth after it; step: the wave's bytes into the rows
template <bool LINES>
__device__ __forceinline__ WeightLines two_lines(strip_t strip, uint32_t at, uint32_t next, uint32_t step) {
    constexpr int ONCE = LINES ? 2 : 0;
    return WeightLines{__builtin_bit_cast(line_u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(strip, (int)at, (int)step, ONCE)),
                       __builtin_bit_cast(line_u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(strip, (int)(at + next), (int)step, ONCE))};
}
// The operands of the two steps, 16 bytes a lane each.
template <typename Operand>
__device__ __forceinline__ void two_steps(const WeightLines& l, Operand& first, Operand& second) {
    line_u32x4_t a, b;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        a[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)l.lo[i], (int)l.hi[i], 0x128, 0xf, 0xc, false);
        b[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)l.hi[i], (int)l.lo[i], 0x128, 0xf, 0x3, false);
    }
    first = __builtin_bit_cast(Operand, a);
    second = __builtin_bit_cast(Operand, b);
}
