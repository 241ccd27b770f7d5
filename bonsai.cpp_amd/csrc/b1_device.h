// Device helpers shared by the gfx950 kernel files: operand types, the
// weight-bit expansion, LDS-DMA and buffer accesses, waits, and the fp32
// elementwise functions of the epilogues and producers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace b1 {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kSignPair = 0x80008000u;

// Bits of m: ~(x ^ y); other bits: y.  One v_bitop3_b32, whose 8-bit table
// is indexed by (x_bit << 2) | (m_bit << 1) | y_bit: 0xa6 = {0,1,1,0,0,1,0,1}
// for indices 0..7.  Through the compiler builtin, not inline asm: the
// compiler must see the VALU write, or it cannot insert the wait states an
// MFMA reading the result as a source operand needs (an MFMA issued too
// soon after an asm-hidden write read stale operands here).
__device__ __forceinline__ uint32_t xnor_sel(uint32_t m, uint32_t x, uint32_t y) {
    return __builtin_amdgcn_bitop3_b32(x, m, y, 0xa6);
}

// (lo, hi) -> packed fp16 pair, round to nearest even (v_cvt_pk_f16_f32).
__device__ __forceinline__ uint32_t pack_f16(float lo, float hi) {
    float2v v = {lo, hi};
    half2v h = __builtin_convertvector(v, half2v);
    return __builtin_bit_cast(uint32_t, h);
}

// fp32 -> fp16 bits of one value, rounded once from the fp32 value: the
// empty asm keeps the compiler from folding the multiply that produced x
// into the conversion (v_fma_mixlo_f16 rounds the exact product to fp16
// once, which differs from the producer passes' fp32-then-fp16 rounding in
// the rare products an fp32 rounding puts on an fp16 midpoint).
__device__ __forceinline__ uint16_t half_bits(float x) {
    asm("" : "+v"(x));
    return (uint16_t)pack_f16(x, 0.0f);
}

// (lo, hi) -> packed fp16 pair, each rounded once from its fp32 value (the
// fold half_bits keeps out, for two values).
__device__ __forceinline__ uint32_t pack_f16_rounded(float lo, float hi) {
    asm("" : "+v"(lo), "+v"(hi));
    return pack_f16(lo, hi);
}

// max(m, |a|, |b|) in one v_max3_f32: the running largest magnitude of the
// activations a lane converts, against fp16's range (a quiet NaN operand is
// passed over, as IEEE maxNum does: a NaN does not count as out of range).
__device__ __forceinline__ float absmax3(float m, float a, float b) {
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}
// fp32 magnitudes from this on round to fp16 infinity
constexpr float kF16Overflow = 65520.0f;

// s_waitcnt vmcnt(N) leaving expcnt and lgkmcnt alone (gfx9 encoding:
// vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// Waits for this wave's LDS operations only (vmcnt and expcnt left open).
__device__ __forceinline__ void wait_lgkmcnt0() {
    __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4) | (0x0 << 8));
}

// Work-group barrier that does not drain outstanding global->LDS loads
// (__syncthreads() would add s_waitcnt vmcnt(0) while LDS-DMA is pending).
// Each wave waits for its own loads with wait_vmcnt<> before arriving.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

typedef __attribute__((address_space(3))) void lds_void_t;

// Global -> LDS copies without VGPR staging.  `lds` must be wave-uniform
// (it goes through M0).  Lane i's 16 bytes land at lds + 16 i; 12-byte
// loads also land at lds + 16 i (a 16-byte lane stride, measured on gfx950
// for the global and the buffer forms), leaving 4 bytes untouched per lane.
// Kept as plain device functions: a kernel template that calls these
// builtins directly loses its host-side launch stub.
// global_load_lds_dword: lane i's 4 bytes land at lds + 4 i.  The compiler
// treats this global form as a FLAT access that may touch LDS, and with one
// in a kernel it makes every LDS wait of that kernel a full lgkmcnt(0).  In
// the GEMM (its row-scale copy) the buffer form instead gives waits that
// count only the reads a step needs, and it measured no faster (252.9-253.4
// vs 253.1 us at M=4096 K=3072 N=12288, 0.3-0.6 % slower on four other
// shapes, bit-identical): the fragment reads' latency is already covered.
__device__ __forceinline__ void dma_lds4(const void *src, void *lds) {
    __builtin_amdgcn_global_load_lds(src, (lds_void_t *)lds, 4, 0, 0);
}

// Raw buffer loads with range checking (offsets at or past num_records read
// zeros); word 3 of the resource for gfx9-family raw buffers.
constexpr int kBufferFlags = 0x00020000;
// Cache policy of the GEMM's full-tile output stores: the default.  Each
// 16-byte store covers 32 rows x 32 bytes, a quarter of each 128-byte line,
// and L2 merges the four quarters before the line goes to memory; the
// non-temporal policy sends each quarter on its own (355 vs ~267 us at
// M=4096 K=3072 N=12288).
#ifndef B1_STORE_AUX
#define B1_STORE_AUX 0
#endif
constexpr int kStoreNT = B1_STORE_AUX;
// A 16-byte buffer store followed by 5 wait states before any instruction
// may rewrite its data registers.  A store of more than 8 bytes reads its
// data in the cycles after it issues; the compiler inserts that gap only
// for stores whose soffset is not a register, and the epilogue stores carry
// their row offset in an SGPR.  Without it, a VALU write issued right after
// such a store changed the stored values of some lanes (the SwiGLU
// epilogue: 2272 of 786,432 outputs, different on every launch).  The asm
// takes the data as an input, so its registers stay live until the nops
// have issued, and its memory clobber keeps it after the store.
template <int AUX>
__device__ __forceinline__ void store16_guarded(u32x4 v, __amdgpu_buffer_rsrc_t rsrc, int voff, int soff) {
    __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, voff, soff, AUX);
    asm volatile("s_nop 4" ::"v"(v) : "memory");
}

// 16 bytes per lane from the buffer at byte offset voff, landing at
// lds + 16 * lane (wave-uniform lds, through M0).
__device__ __forceinline__ void dma_buf_lds16(__amdgpu_buffer_rsrc_t rsrc, void *lds, uint32_t voff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t *)lds, 16, voff, 0, 0, 0);
}
// The same, 16 or 12 bytes per lane (12-byte lanes also land 16 bytes
// apart), with a wave-uniform byte offset soff (an SGPR) added to voff.  A
// constant offset goes into soff, not the instruction's offset field: for
// these loads the instruction offset moves the LDS destination as well.
__device__ __forceinline__ void dma_buf_lds16s(__amdgpu_buffer_rsrc_t rsrc, void *lds, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t *)lds, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void dma_buf_lds12s(__amdgpu_buffer_rsrc_t rsrc, void *lds, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t *)lds, 12, voff, soff, 0, 0);
}
// 4 bytes per lane, landing at lds + 4 * lane.
__device__ __forceinline__ void dma_buf_lds4(__amdgpu_buffer_rsrc_t rsrc, void *lds, uint32_t voff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t *)lds, 4, voff, 0, 0, 0);
}

__device__ __forceinline__ uint32_t dup_lo16(uint32_t d) {
    return __builtin_amdgcn_perm(d, d, 0x01000100u);
}
__device__ __forceinline__ uint32_t dup_hi16(uint32_t d) {
    return __builtin_amdgcn_perm(d, d, 0x03020302u);
}

// Weight dword for fp16 pair slot (bits p and p+16 of `w`, p = 15 - sh):
// each half is the fp16 scale with its sign flipped where the bit is 0.
__device__ __forceinline__ uint32_t wpair(uint32_t w, int sh, uint32_t scale2) {
    return xnor_sel(kSignPair, w << sh, scale2);
}

// One v_lshlrev_b64 of the pair (w, w >> 8): its low dword is w << SH and
// its high dword carries bits d + 8 and d + 24 of w at 15 and 31 (d = 15 -
// SH < 8), so that one shift serves the weight dwords of pairs d and d + 8.
// A 64-bit shift costs what a 32-bit one does on gfx950 (measured: both
// about 2 ns per wave instruction per SIMD with the SIMDs saturated, a
// v_bitop3 1.2 ns); the compiler splits a constant 64-bit shift into two
// 32-bit ops, hence the asm.  Its result only feeds VALU bit ops (no MFMA
// operand hazard).
template <int SH>
__device__ __forceinline__ uint64_t shl64(uint64_t v) {
    static_assert(SH >= 0 && SH <= 15, "a 16-bit half");
    uint64_t r;
    asm("v_lshlrev_b64 %0, %1, %2" : "=v"(r) : "I"(SH), "v"(v));
    return r;
}
// The weight dwords of pairs 4T + j (lo) and 4T + j + 8 (hi), j = 0..3,
// T = 0 or 1, from the sign word w and w8 = w >> 8: the same values as
// wpair(w, 15 - 4T - j, scale2) and wpair(w, 7 - 4T - j, scale2).
template <int T>
__device__ __forceinline__ void wpair_quads(uint32_t w, uint32_t w8, uint32_t scale2, u32x4 &lo, u32x4 &hi) {
    const uint64_t v = (uint64_t)w8 << 32 | w;
    const uint64_t v0 = shl64<15 - 4 * T>(v), v1 = shl64<14 - 4 * T>(v), v2 = shl64<13 - 4 * T>(v),
                   v3 = shl64<12 - 4 * T>(v);
    lo[0] = xnor_sel(kSignPair, (uint32_t)v0, scale2);
    lo[1] = xnor_sel(kSignPair, (uint32_t)v1, scale2);
    lo[2] = xnor_sel(kSignPair, (uint32_t)v2, scale2);
    lo[3] = xnor_sel(kSignPair, (uint32_t)v3, scale2);
    hi[0] = xnor_sel(kSignPair, (uint32_t)(v0 >> 32), scale2);
    hi[1] = xnor_sel(kSignPair, (uint32_t)(v1 >> 32), scale2);
    hi[2] = xnor_sel(kSignPair, (uint32_t)(v2 >> 32), scale2);
    hi[3] = xnor_sel(kSignPair, (uint32_t)(v3 >> 32), scale2);
}

// The weight dwords of pairs d .. d + 3 from the sign word shifted so that
// pair d + 3's bits are at 15 and 31: one 32-bit and one 64-bit shift (the
// bit the latter carries into its high dword is not a sign) instead of a
// shift a pair.
__device__ __forceinline__ u32x4 wpair4(uint32_t w, uint32_t scale2) {
    const uint32_t w2 = w << 2;
    const uint64_t v = shl64<1>((uint64_t)w2 << 32 | w);
    return u32x4{xnor_sel(kSignPair, (uint32_t)(v >> 32), scale2), xnor_sel(kSignPair, w2, scale2),
                 xnor_sel(kSignPair, (uint32_t)v, scale2), xnor_sel(kSignPair, w, scale2)};
}

__device__ __forceinline__ void count_nonfinite(int32_t *ctr, int bad) {
    if (bad && ctr) atomicAdd(ctr, bad);
}

// Work-groups are dispatched round-robin over the 8 XCDs (bid % 8).  Give
// each XCD a contiguous run of tiles (N-fastest) so the work-groups resident
// on one XCD share activation rows in that XCD's L2.
__device__ __forceinline__ int xcd_tile(int bid, int nblk) {
    const int xcd = bid & 7, loc = bid >> 3;
    const int q = nblk >> 3, r = nblk & 7;
    return xcd * q + min(xcd, r) + loc;
}

// GELU-tanh, 0.5 x (1 + tanh(u)), u = sqrt(2/pi) (x + 0.044715 x^3).
// Evaluated as x / (1 + e^(-2u)), the same function (1 + tanh(u) =
// 2 / (1 + e^(-2u))), with e^(-2u) = 2^(x (c1 + c2 x^2)), c1 = -2
// sqrt(2/pi) / ln 2 and c2 = 0.044715 c1: one hardware exp2 and one
// reciprocal instead of a library tanh, which matters in the GEMM epilogue
// where no MFMA work overlaps it.  Within 3e-7 max(1, |x|) of the float64
// function (1-ulp exp2 and reciprocal included).  Large negative x: the
// exponential overflows to inf and the result is -0; NaN stays NaN.
__device__ __forceinline__ float gelu_tanh(float x) {
    const float c1 = -2.30220819f;  // -2 sqrt(2/pi) log2(e)
    const float c2 = -0.102943242f; // 0.044715 c1
    const float t = x * __builtin_fmaf(c2, x * x, c1);
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t));
}

// silu(x) = x / (1 + e^-x), in fp32 with the device library's expf.
__device__ __forceinline__ float silu_f32(float x) {
#pragma clang fp contract(off)
    return x / (1.0f + expf(-x));
}

// r + g y as the reference's two ggml ops (a multiply, then an add), each
// rounded to fp32: never contracted into one FMA.
__device__ __forceinline__ float gate_residual(float r, float g, float y) {
#pragma clang fp contract(off)
    const float t = g * y;
    return r + t;
}

__device__ __forceinline__ float mul_f32(float a, float b) {
#pragma clang fp contract(off)
    return a * b;
}

} // namespace
} // namespace b1
