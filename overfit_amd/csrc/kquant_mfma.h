// kquant_mfma.h — Q4_K / Q6_K weight operands of the int8-MFMA kernels (v_mfma_i32_16x16x64_i8), built in registers
// from the GGUF bytes. The regrouping they rest on, and why it is exact, is described in mfma.hip.
#pragma once

#include "kquant_blocks.h"
#include "ovfq_device.h"

namespace ovfq {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ i32x4 mfma16(i32x4 a, i32x4 b, i32x4 c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// Two dwords of 16-bit lanes (pe: K bytes 0 and 2, po: K bytes 1 and 3), each holding u = v + 128 for a value v in
// [-4064, 4224) (two's complement): lo = the low byte of v as int8 (v mod 256, signed), hi = u >> 8 (the high byte of
// u), so that v = 256*hi + lo, as packed bytes in K order. v_perm_b32 gathers bytes 0 and 2 of each source (selector
// 0x06020400 = [pe.b0, po.b0, pe.b2, po.b2]) or bytes 1 and 3 (0x07030501); the low byte of v is the low byte of u
// with its top bit flipped.
__device__ __forceinline__ void split_lo_hi(uint32_t pe, uint32_t po, uint32_t& lo, uint32_t& hi) {
    lo = __builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u;
    hi = __builtin_amdgcn_perm(po, pe, 0x07030501u);
}

// K permutation. The four MFMAs t = 0..3 of a super-block each cover 64 of its 256 elements; lane-group g of
// MFMA t holds 16 consecutive elements starting at base(t, g), in both operands. The activation row is staged in
// LDS as 16-byte pieces in (t, g) order (logical slot 4t + g), so a lane reads its A operand with one
// ds_read_b128. The bases are chosen so that every nibble/bit-field shift on the weight side is a compile-time
// constant. Rows are 256 bytes with the slot XOR-swizzled by (row % 16): the 16 lanes of an A read (16 rows, one
// logical slot) then hit 16 distinct 16-byte bank groups.

// ------------------------------------------------------------------------------------------ Q4_K weight operands
struct Q4KMfma {
    static constexpr int kBytes = kQ4KBytes;
    static constexpr int kNumMfma = 3;  // lo, hi, min
    // MFMA t: nibble (t >> 1) of qs[64(t & 1) + 16g + j]  ->  element 128(t&1) + 64(g>>1) + 32(t>>1) + 16(g&1) + j
    // (qs byte b holds elements 64(b/32) + b%32 in its low nibble and +32 in its high nibble).
    // LDS slot 4t + g holds source piece (element / 16) s with bits [t&1, g>>1, t>>1, g&1].
    __device__ __forceinline__ static uint32_t src_piece(uint32_t slot) {
        const uint32_t t = slot >> 2, g = slot & 3u;
        return 8u * (t & 1u) + 4u * (g >> 1) + 2u * (t >> 1) + (g & 1u);
    }
    struct W {
        u32x4 h;      // d, dmin, 12 packed scale/min bytes
        u32x4 q[2];   // qs[16g .. +16], qs[64 + 16g .. +16]
    };
    __device__ __forceinline__ static W load(__amdgpu_buffer_rsrc_t r, uint32_t off, int g) {
        W w;
        w.h = ld4(r, off);
        w.q[0] = ld4(r, off + 16 + 16 * g);
        w.q[1] = ld4(r, off + 16 + 64 + 16 * g);
        return w;
    }
    // The min MFMA's B operand for lane group g: m_{2g}, m_{2g}, m_{2g+1}, m_{2g+1} in fp16, from the eight 6-bit
    // mins (LD/GgmlDequant.cs:64-79 unpacking; lane group g takes sub-blocks 2g and 2g + 1).
    __device__ __forceinline__ static u32x2 min_operand(const W& w, int g) {
        const uint32_t m_lo = w.h.z & 0x3f3f3f3fu;
        const uint32_t m_hi = ((w.h.w >> 4) & 0x0f0f0f0fu) | ((w.h.z >> 2) & 0x30303030u);
        const uint32_t mg = (g < 2 ? m_lo : m_hi) >> (16 * (g & 1));
        const uint32_t m0 = __builtin_bit_cast(uint16_t, (_Float16)(mg & 0xffu));
        const uint32_t m1 = __builtin_bit_cast(uint16_t, (_Float16)((mg >> 8) & 0xffu));
        return u32x2{m0 * 0x00010001u, m1 * 0x00010001u};
    }
    // Sub-block of MFMA t, lane-group g: js = 4(t&1) + 2(g>>1) + (t>>1) (LD/GgmlDequant.cs:64-79 unpacking).
    template <int T>
    __device__ __forceinline__ static void operands(const W& w, int g, i32x4 (&op)[kNumMfma]) {
        const uint32_t jj = (uint32_t)(2 * (g >> 1) + (T >> 1)) * 8;  // byte index js & 3
        uint32_t sc, m;
        if ((T & 1) == 0) {  // js < 4
            sc = (w.h.y >> jj) & 63u;
            m = (w.h.z >> jj) & 63u;
        } else {
            const uint32_t A = w.h.y >> jj, B = w.h.z >> jj, C = (w.h.w >> jj) & 0xffu;
            sc = (C & 0x0fu) | ((A >> 2) & 0x30u);
            m = (C >> 4) | ((B >> 2) & 0x30u);
        }
        const u32x4 src = w.q[T & 1];
        const uint32_t qv[4] = {src.x, src.y, src.z, src.w};
        constexpr uint32_t kShift = (T >> 1) * 4;
        // sc = 8*sc_hi + sc_lo with both parts in [0, 7]: sc_lo*nib and sc_hi*nib are <= 105, so one packed 16-bit
        // multiply of the four nibble bytes gives the four byte products with no carry between bytes.
        const unsigned short sl = (unsigned short)(sc & 7u), sh = (unsigned short)(sc >> 3);
        const u16x2 sl2 = {sl, sl}, sh2 = {sh, sh};
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const u16x2 nib = __builtin_bit_cast(u16x2, (qv[k] >> kShift) & 0x0f0f0f0fu);
            lo[k] = __builtin_bit_cast(uint32_t, nib * sl2);
            hi[k] = __builtin_bit_cast(uint32_t, nib * sh2);
        }
        op[0] = i32x4{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3]};
        op[1] = i32x4{(int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
        const int mm = (int)__builtin_amdgcn_perm(0u, m, 0u);  // m in all four bytes
        op[2] = i32x4{mm, mm, mm, mm};
    }
    __device__ __forceinline__ static float d_of(const W& w) { return half_lo(w.h.x); }
    __device__ __forceinline__ static float dmin_of(const W& w) { return half_hi(w.h.x); }
    __device__ __forceinline__ static uint32_t raw_scales(const W& w) { return w.h.x; }  // fp16 d | fp16 dmin << 16
    // q8Scale * (d * mainAcc - dmin * minAcc)   (RT/Q4KDotKernel.cs:944)
    __device__ __forceinline__ static float tail(const i32x4 (&acc)[kNumMfma], int i, float d, float dmin,
                                                 float q8s) {
        const int main_acc = acc[0][i] + (acc[1][i] << 3);
        return q8s * (d * (float)main_acc - dmin * (float)acc[2][i]);
    }
};

// ------------------------------------------------------------------------------------------ Q6_K weight operands
struct Q6KMfma {
    static constexpr int kBytes = kQ6KBytes;
    static constexpr int kNumMfma = 2;  // lo, hi
    // MFMA t = qh bit pair p: element 128h + 32p + l with h = g >> 1, l = 16(g&1) + j: nibble (p >> 1) of
    // ql[64h + 32(p&1) + l], bits 2p of qh[32h + l], scale sc[8h + 2p + (g&1)] (RT/Q6KDotKernel.cs:189-213).
    // LDS slot 4p + g holds source piece s with bits [g>>1, p, p, g&1].
    __device__ __forceinline__ static uint32_t src_piece(uint32_t slot) {
        const uint32_t p = slot >> 2, g = slot & 3u;
        return 8u * (g >> 1) + 2u * p + (g & 1u);
    }
    struct W {
        uint32_t ql[2][4];  // ql[64h + 16(g&1) .. +16], ql[64h + 32 + 16(g&1) .. +16]
        uint32_t qh[4];     // qh[32h + 16(g&1) .. +16]
        uint32_t sc;        // byte p = sc[8h + 2p + (g&1)]
        uint32_t d;
    };
    // Run by run. With all the runs' loads ahead of their shifts the kernels that read the GGUF bytes here lost up to 10 %
    // (MI355X, us, loads first / run by run: small-M 15371x2560 at 6 rows 19.7 / 17.7, from a caller's quantised activation
    // 10331x2304 at 5 rows 12.1 / 11.0, 17194x7168 at 4 rows 49.8 / 45.7).
    __device__ __forceinline__ static W load(__amdgpu_buffer_rsrc_t r, uint32_t off, int g) {
        W w;
        const uint32_t h = (uint32_t)g >> 1, l0 = 16u * (uint32_t)(g & 1);
        Q6K::run16(r, off + 64 * h + l0, w.ql[0]);
        Q6K::run16(r, off + 64 * h + 32 + l0, w.ql[1]);
        Q6K::run16(r, off + 128 + 32 * h + l0, w.qh);
        const uint32_t so = off + 192 + 8 * h, sh = so & 3u;
        const u32x3 sv = ld3(r, so & ~3u);
        const uint32_t s0 = __builtin_amdgcn_alignbyte(sv.y, sv.x, sh), s1 = __builtin_amdgcn_alignbyte(sv.z, sv.y, sh);
        w.sc = __builtin_amdgcn_perm(s1, s0, (g & 1) ? 0x07050301u : 0x06040200u);
        w.d = __builtin_amdgcn_raw_buffer_load_b16(r, (int)(off + 208), 0, 0);
        return w;
    }
    __device__ __forceinline__ static u32x2 min_operand(const W&, int) { return u32x2{0u, 0u}; }
    template <int P>
    __device__ __forceinline__ static void operands(const W& w, int, i32x4 (&op)[kNumMfma]) {
        // W + 128 = sc * q - 32 * sc + 128 (W = sc * (q - 32) in [-4064, 4096]), computed per 16-bit lane modulo
        // 2^16 (two's complement).
        const uint32_t scp = (uint32_t)(int)(int8_t)((w.sc >> (8 * P)) & 0xffu);
        const uint32_t sc16 = scp & 0xffffu, bias16 = (128u - 32u * scp) & 0xffffu;
        const u16x2 sc2 = {(unsigned short)sc16, (unsigned short)sc16};
        const u16x2 bias2 = {(unsigned short)bias16, (unsigned short)bias16};
        constexpr uint32_t kNib = (P >> 1) * 4, kBits = 2 * P;
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t qhb = kBits <= 4 ? (w.qh[k] << (4 - kBits)) : (w.qh[k] >> (kBits - 4));
            const uint32_t q = ((w.ql[P & 1][k] >> kNib) & 0x0f0f0f0fu) | (qhb & 0x30303030u);
            const uint32_t qe = __builtin_amdgcn_perm(0u, q, 0x0c020c00u);  // K bytes 0, 2 as 16-bit lanes
            const uint32_t qo = __builtin_amdgcn_perm(0u, q, 0x0c030c01u);  // K bytes 1, 3
            const u16x2 we = __builtin_bit_cast(u16x2, qe) * sc2 + bias2;
            const u16x2 wo = __builtin_bit_cast(u16x2, qo) * sc2 + bias2;
            split_lo_hi(__builtin_bit_cast(uint32_t, we), __builtin_bit_cast(uint32_t, wo), lo[k], hi[k]);
        }
        op[0] = i32x4{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3]};
        op[1] = i32x4{(int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
    }
    __device__ __forceinline__ static float d_of(const W& w) { return half_lo(w.d); }
    __device__ __forceinline__ static float dmin_of(const W&) { return 0.0f; }
    __device__ __forceinline__ static uint32_t raw_scales(const W& w) { return w.d; }  // fp16 d
    // d * q8Scale * mainAcc   (RT/Q6KDotKernel.cs:114-115)
    __device__ __forceinline__ static float tail(const i32x4 (&acc)[kNumMfma], int i, float d, float, float q8s) {
        const int main_acc = acc[0][i] + (acc[1][i] << 8);
        return d * q8s * (float)main_acc;
    }
};

}  // namespace ovfq
