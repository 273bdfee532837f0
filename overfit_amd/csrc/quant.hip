// quant.hip — on-device quantisers: the Q8_K / Q8_0 activation quantisers every projection starts with,
// the Q4_K / Q6_K weight encoders, and the row decoders.
//
// All of them are bit-exact restatements of the reference's scalar code: per-operation IEEE binary32
// (the library is built with -ffp-contract=off, and fp32 division / reciprocal are the correctly rounded
// ones), rintf for MathF.Round (round half to even), integer fp32 -> fp16 conversion with ties to even.
#include "ovfq_device.h"
#include "ovfq_launch.h"

namespace ovfq {

// ------------------------------------------------------------------------------------------ Q8_K activation
// Q4KDotKernel.QuantizeActivationQ8K (RT/Q4KDotKernel.cs:71-136): absMax is a max (exact in any order); scale =
// absMax / 127f; inverse = scale > 0 ? 1f / scale : 0f; q = clamp(rint(x * inverse), -127, 127); bsums[g] = sum
// of the 16 quants of group g. Four super-blocks per wave, one per 16-lane DPP row, sixteen consecutive elements (one
// bsum group) per lane: four 16-byte loads and one 16-byte store of quants per lane, the block's absMax by a 4-step
// DPP row max (a wave per block spent most of its time in the 6 cross-lane exchanges of its max).
__global__ __launch_bounds__(256) void quantize_q8k_kernel(const float* __restrict__ x, int64_t n_blocks,
                                                            int8_t* __restrict__ q, float* __restrict__ s,
                                                            int16_t* __restrict__ bs, uint16_t* __restrict__ bh) {
    // wave_id() is a readfirstlane value, so the buffer resource below is provably wave-uniform (SGPRs).
    const int64_t blk0 = ((int64_t)blockIdx.x * 4 + wave_id()) * 4;
    if (blk0 >= n_blocks) return;
    const int lane = threadIdx.x & 63, row = lane >> 4, l16 = lane & 15;
    const int64_t blk = blk0 + row;
    // blocks past the end read zeros (the resource ends with the last block) and store nothing
    const __amdgpu_buffer_rsrc_t xr =
        make_rsrc(x + blk0 * kQK, rsrc_bytes((uint64_t)n_blocks * kQK * 4, (uint64_t)blk0 * kQK * 4));
    float v[16];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const u32x4 t = ld4(xr, (uint32_t)row * 1024u + (uint32_t)l16 * 64u + (uint32_t)i * 16u);
        v[4 * i] = as_float(t.x);
        v[4 * i + 1] = as_float(t.y);
        v[4 * i + 2] = as_float(t.z);
        v[4 * i + 3] = as_float(t.w);
    }
    const Q8KRow r = q8k_quantize_row16(v);
    if (blk < n_blocks) {
        *reinterpret_cast<u32x4*>(q + blk * kQK + l16 * 16) = r.packed;
        bs[blk * 16 + l16] = (int16_t)r.group_sum;
        if (bh) bh[blk * 16 + l16] = __builtin_bit_cast(uint16_t, (_Float16)r.group_sum);
        if (l16 == 0) s[blk] = r.scale;
    }
}

// The same quantisation into operand-ordered planes (launch_quantize_q8k_tiled): the 16-byte piece that lane (g, r16) of
// MFMA t reads goes to byte 1024 t + 256 g + 16 r16 of its (16 rows, super-block) record, so that a wave loads an A operand
// as one contiguous KiB. Piece p of a super-block (elements 16 p ..) belongs to the (t, g) with src_piece(4 t + g) == p of
// the weight format's operand order (Q4KMfma / Q6KMfma). Lane (g, r16) of the min MFMA reads bsums 4 g .. 4 g + 3.
__global__ __launch_bounds__(256) void quantize_q8k_tiled_kernel(const float* __restrict__ x, int64_t n_blocks, int spr,
                                                                 int q6, uint8_t* __restrict__ q,
                                                                 uint8_t* __restrict__ s, uint8_t* __restrict__ bh) {
    const int64_t blk0 = ((int64_t)blockIdx.x * 4 + wave_id()) * 4;
    if (blk0 >= n_blocks) return;
    const int lane = threadIdx.x & 63, p = lane & 15;
    const int64_t blk = blk0 + (lane >> 4);
    const __amdgpu_buffer_rsrc_t xr =
        make_rsrc(x + blk0 * kQK, rsrc_bytes((uint64_t)n_blocks * kQK * 4, (uint64_t)blk0 * kQK * 4));
    float v[16];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const u32x4 t = ld4(xr, (uint32_t)lane * 64u + (uint32_t)i * 16u);
        v[4 * i] = as_float(t.x);
        v[4 * i + 1] = as_float(t.y);
        v[4 * i + 2] = as_float(t.z);
        v[4 * i + 3] = as_float(t.w);
    }
    const Q8KRow r = q8k_quantize_row16(v);
    if (blk < n_blocks) {
        const int64_t row = blk / spr;
        const size_t rec = (size_t)(row >> 4) * spr + (size_t)(blk - row * spr);
        const int r16 = (int)(row & 15);
        const int slot = tiled_slot(p, q6 != 0);  // 4 t + g
        *reinterpret_cast<u32x4*>(q + rec * kTiledQ + slot * 256 + r16 * 16) = r.packed;
        if (bh)
            *reinterpret_cast<_Float16*>(bh + rec * kTiledB + (p >> 2) * 128 + r16 * 8 + (p & 3) * 2) =
                (_Float16)r.group_sum;
        if (p == 0) *reinterpret_cast<float*>(s + rec * kTiledS + r16 * 4) = r.scale;
    }
}

// ------------------------------------------------------------------------------------------ Q8_0 activation
// Q8DotKernel.Quantize (RT/Q8DotKernel.cs:42-91): 32-element blocks, eight lanes per block.
__global__ __launch_bounds__(256) void quantize_q8_0_kernel(const float* __restrict__ x, int64_t n_blocks,
                                                             int8_t* __restrict__ q, float* __restrict__ s) {
    // One wave covers 8 consecutive blocks; the resource starts at the wave's first block (wave-uniform).
    const int64_t wblk = ((int64_t)blockIdx.x * 4 + wave_id()) * 8;
    const int lane = threadIdx.x & 63;
    const int64_t blk = wblk + (lane >> 3);
    if (wblk >= n_blocks) return;
    const int sub = lane & 7;
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(x + wblk * 32, rsrc_bytes((uint64_t)n_blocks * 128, (uint64_t)wblk * 128));
    const Q80Lane r = q8_0_quantize_lane(ld4(xr, lane * 16));
    if (blk < n_blocks) {
        reinterpret_cast<uint32_t*>(q + blk * 32)[sub] = r.packed;
        if (sub == 0) s[blk] = r.scale;
    }
}

// ------------------------------------------------------------------------------------------ weight encoders
// Both encoders spread a 256-element super-block over a 16-lane DPP row, sixteen consecutive elements a lane (four 16-byte
// loads), so a wave covers four; per-block values are exchanged inside the row. They are bound by the source's stream: a
// thread per super-block (1024 waves in all for 4096x4096, every load instruction touching 64 lines) was bound by those loads.
// us before / after: Q4_K 4096x4096 118 / 18.0 (4.2 TB/s), 8192x8192 1287 / 73; Q6_K 242 / 20.4 and 1487 / 67.
template <int kCtrl>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xf, 0xf, false);
}
// The value of the lane whose number in the 16-lane row differs in bit 1, 2, 4 or 8.
__device__ __forceinline__ uint32_t row_xor1(uint32_t v) { return dpp_u32<0xb1>(v); }
__device__ __forceinline__ uint32_t row_xor2(uint32_t v) { return dpp_u32<0x4e>(v); }
__device__ __forceinline__ uint32_t row_xor4(uint32_t v) { return dpp_u32<0x1b>(dpp_u32<0x141>(v)); }  // 7 - i, then i ^ 3
__device__ __forceinline__ uint32_t row_xor8(uint32_t v) { return dpp_u32<0x128>(v); }
__device__ __forceinline__ uint32_t f_bits(float f) { return __builtin_bit_cast(uint32_t, f); }

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// Lane `l16` of row `lane >> 4` loads its sixteen elements of super-block blk0 + row (zeros past n_blocks).
__device__ __forceinline__ void load_row16(const float* __restrict__ w, int64_t blk0, int64_t n_blocks, float (&v)[16]) {
    const __amdgpu_buffer_rsrc_t xr =
        make_rsrc(w + blk0 * kQK, rsrc_bytes((uint64_t)n_blocks * kQK * 4, (uint64_t)blk0 * kQK * 4));
    const uint32_t off = (threadIdx.x & 63) * 64u;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const u32x4 t = ld4(xr, off + 16u * i);
        v[4 * i] = as_float(t.x);
        v[4 * i + 1] = as_float(t.y);
        v[4 * i + 2] = as_float(t.z);
        v[4 * i + 3] = as_float(t.w);
    }
}

// GgmlQuant.EncodeQ4_KBlock (LD/GgmlQuant.cs:31-126). Lane i holds half of sub-block i >> 1.
__global__ __launch_bounds__(256) void encode_q4k_kernel(const float* __restrict__ w, int64_t n_blocks,
                                                          uint8_t* __restrict__ dst) {
    const int64_t blk0 = ((int64_t)blockIdx.x * 4 + wave_id()) * 4;
    if (blk0 >= n_blocks) return;
    const int lane = threadIdx.x & 63, l16 = lane & 15;
    const int64_t blk = blk0 + (lane >> 4);
    float v[16];
    load_row16(w, blk0, n_blocks, v);
    float lo = __builtin_inff(), hi = -__builtin_inff();
#pragma unroll
    for (int e = 0; e < 16; e++) {
        if (v[e] < lo) lo = v[e];
        if (v[e] > hi) hi = v[e];
    }
    const float lo1 = as_float(row_xor1(f_bits(lo))), hi1 = as_float(row_xor1(f_bits(hi)));
    if (lo1 < lo) lo = lo1;
    if (hi1 > hi) hi = hi1;
    if (lo > 0.0f) lo = 0.0f;
    const float sub_scale = (hi - lo) / 15.0f, sub_min = -lo;
    float max_scale = 0.0f, max_min = 0.0f;  // over the row's eight sub-blocks
    if (sub_scale > max_scale) max_scale = sub_scale;
    if (sub_min > max_min) max_min = sub_min;
    auto max_with = [&](uint32_t s, uint32_t m) {
        if (as_float(s) > max_scale) max_scale = as_float(s);
        if (as_float(m) > max_min) max_min = as_float(m);
    };
    max_with(row_xor2(f_bits(max_scale)), row_xor2(f_bits(max_min)));
    max_with(row_xor4(f_bits(max_scale)), row_xor4(f_bits(max_min)));
    max_with(row_xor8(f_bits(max_scale)), row_xor8(f_bits(max_min)));
    const float inv_scale = max_scale > 0.0f ? 63.0f / max_scale : 0.0f;
    const float inv_min = max_min > 0.0f ? 63.0f / max_min : 0.0f;
    const int sa = (int)rintf(inv_scale * sub_scale), ma = (int)rintf(inv_min * sub_min);
    const uint32_t sc = (uint32_t)(sa < 63 ? sa : 63), m = (uint32_t)(ma < 63 ? ma : 63);
    const float d = max_scale / 63.0f;
    const float dmin = max_min / 63.0f;
    // Nibbles from the float d / dmin (LD/GgmlQuant.cs:108-116): qs[32p+e] = q[64p+e] | q[64p+32+e] << 4, a byte of four
    // dwords each; the odd sub-blocks' go to the lanes of the even ones.
    const float es = d * (float)sc, em = dmin * (float)m;
    uint32_t q[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 16; e++) {
        int l = es > 0.0f ? (int)rintf((v[e] + em) / es) : 0;
        l = l < 0 ? 0 : (l > 15 ? 15 : l);
        q[e >> 2] |= (uint32_t)l << (8 * (e & 3));
    }
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] |= row_xor2(q[i]) << 4;
    // PackScalesMins (LD/GgmlQuant.cs:164-172), four bytes per 32-bit word: sub-block j < 4 (lane 2j) with j + 4.
    const uint32_t sc4 = row_xor8(sc), m4 = row_xor8(m);
    const bool packs = l16 < 8 && (l16 & 1) == 0;
    const uint32_t at = 4u * (uint32_t)l16;  // 8 j
    uint32_t p0 = packs ? ((sc & 0x3f) | ((sc4 >> 4) << 6)) << at : 0;
    uint32_t p1 = packs ? ((m & 0x3f) | ((m4 >> 4) << 6)) << at : 0;
    uint32_t p2 = packs ? ((sc4 & 0x0f) | ((m4 & 0x0f) << 4)) << at : 0;
    p0 |= row_xor2(p0);
    p1 |= row_xor2(p1);
    p2 |= row_xor2(p2);
    p0 |= row_xor4(p0);
    p1 |= row_xor4(p1);
    p2 |= row_xor4(p2);
    if (blk >= n_blocks) return;
    uint8_t* out = dst + blk * kQ4KBytes;  // any 4-byte-aligned address
    if ((l16 & 2) == 0) *reinterpret_cast<u32x4_a4*>(out + 16 + 32 * (l16 >> 2) + 16 * (l16 & 1)) = u32x4{q[0], q[1], q[2], q[3]};
    if (l16 == 0)
        *reinterpret_cast<u32x4_a4*>(out) =
            u32x4{(uint32_t)float_to_half_rne(d) | ((uint32_t)float_to_half_rne(dmin) << 16), p0, p1, p2};
}

// The build's own Q6_K encoder (the reference has none): the signed value of largest magnitude in each
// 16-element sub-block maps to q = -32; one fp16 super-scale d = 1 / (-128 / largest sub-scale) carries 16
// int8 sub-scales; quants are rint(x / (fp16(d) * sc)) clamped to [-32, 31], stored +32. The byte layout is
// the inverse of GgmlDequant.DecodeQ6_KBlock (LD/GgmlDequant.cs:143-209). Lane s holds sub-block s = 8 h + 2 p + l: the
// elements 32 p + 16 l .. of half h. A wave's four 210-byte blocks are put together in LDS and stored as 210 dwords.
__global__ __launch_bounds__(256) void encode_q6k_kernel(const float* __restrict__ w, int64_t n_blocks,
                                                          uint8_t* __restrict__ dst) {
    __shared__ __align__(16) uint16_t stage[4][4 * kQ6KBytes / 2];
    const int wave = wave_id();
    const int64_t blk0 = ((int64_t)blockIdx.x * 4 + wave) * 4;
    if (blk0 >= n_blocks) return;
    const int lane = threadIdx.x & 63, l16 = lane & 15;
    float v[16];
    load_row16(w, blk0, n_blocks, v);
    float amax = 0.0f, vmax = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const float a = fabsf(v[e]);
        if (a > amax) {
            amax = a;
            vmax = v[e];
        }
    }
    const float sub_scale = amax > 0.0f ? vmax / -32.0f : 0.0f;
    // the first sub-scale of the largest magnitude
    float max_scale = sub_scale;
    uint32_t first = (uint32_t)l16;
    auto larger = [&](uint32_t s, uint32_t i) {
        const float o = fabsf(as_float(s)), mine = fabsf(max_scale);
        if (o > mine || (o == mine && i < first)) {
            max_scale = as_float(s);
            first = i;
        }
    };
    larger(row_xor1(f_bits(max_scale)), row_xor1(first));
    larger(row_xor2(f_bits(max_scale)), row_xor2(first));
    larger(row_xor4(f_bits(max_scale)), row_xor4(first));
    larger(row_xor8(f_bits(max_scale)), row_xor8(first));
    const bool zero = fabsf(max_scale) == 0.0f;  // the whole block: all bytes 0
    const float iscale = -128.0f / max_scale;
    const float d = 1.0f / iscale;
    const uint16_t dh = float_to_half_rne(d);
    const int sv = (int)rintf(iscale * sub_scale);
    const int sc = sv < 127 ? sv : 127;
    const float ds = half_bits_to_float(dh) * (float)sc;
    uint32_t nib[4] = {0, 0, 0, 0}, top[4] = {0, 0, 0, 0};
    const int p = (l16 >> 1) & 3;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        int l = 0;
        if (ds != 0.0f) {
            l = (int)rintf(v[e] / ds);
            l = l < -32 ? -32 : (l > 31 ? 31 : l);
        }
        const uint32_t qv = zero ? 0u : (uint32_t)(l + 32);
        nib[e >> 2] |= (qv & 0x0f) << (8 * (e & 3));
        top[e >> 2] |= (qv >> 4) << (8 * (e & 3));
    }
    // ql[64h + 32 (p & 1) + 16 l + i] = q of p & 1 | q of (p & 1) + 2 << 4; qh[32h + 16 l + i] = the four p's top bits
#pragma unroll
    for (int i = 0; i < 4; i++) {
        nib[i] |= row_xor4(nib[i]) << 4;
        top[i] <<= 2 * p;
        top[i] |= row_xor2(top[i]);
        top[i] |= row_xor4(top[i]);
    }
    uint16_t* out = &stage[wave][(lane >> 4) * (kQ6KBytes / 2)];
    const int h = l16 >> 3, l = l16 & 1;
    if (p < 3) {  // p = 0, 1: ql; 2: qh
        const int at = p < 2 ? 64 * h + 32 * p + 16 * l : 128 + 32 * h + 16 * l;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t word = p < 2 ? nib[i] : top[i];
            out[at / 2 + 2 * i] = (uint16_t)word;
            out[at / 2 + 2 * i + 1] = (uint16_t)(word >> 16);
        }
    }
    reinterpret_cast<uint8_t*>(out)[192 + l16] = zero ? 0 : (uint8_t)sc;
    if (l16 == 0) out[104] = zero ? 0 : dh;
    wave_sync();
    // four blocks are 210 dwords from a 4-byte-aligned address on; the last wave's may be fewer
    const int64_t blocks = n_blocks - blk0 < 4 ? n_blocks - blk0 : 4;
    uint8_t* base = dst + blk0 * kQ6KBytes;
    if (blocks == 4) {
        for (int i = lane; i < 4 * kQ6KBytes / 4; i += 64)
            reinterpret_cast<uint32_t*>(base)[i] = reinterpret_cast<const uint32_t*>(stage[wave])[i];
    } else {
        for (int i = lane; i < (int)blocks * (kQ6KBytes / 2); i += 64)
            reinterpret_cast<uint16_t*>(base)[i] = stage[wave][i];
    }
}

// ------------------------------------------------------------------------------------------ row decode
// GgmlDequant.DecodeQ4_KBlock (LD/GgmlDequant.cs:95-141) over one output row: one thread per element.
__global__ __launch_bounds__(256) void decode_row_q4k_kernel(const uint8_t* __restrict__ row, float* __restrict__ dst) {
    const uint8_t* b = row + (size_t)blockIdx.x * kQ4KBytes;
    const int i = threadIdx.x;
    const int p = i >> 6, hi = (i >> 5) & 1, e = i & 31;
    const float d = half_bits_to_float((uint16_t)(b[0] | (b[1] << 8)));
    const float dmin = half_bits_to_float((uint16_t)(b[2] | (b[3] << 8)));
    const uint8_t* q = b + 4;
    const int j = 2 * p + hi;
    int sc, m;
    if (j < 4) {
        sc = q[j] & 63;
        m = q[j + 4] & 63;
    } else {
        sc = (q[j + 4] & 0x0f) | ((q[j - 4] >> 6) << 4);
        m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
    }
    const int packed = b[16 + 32 * p + e];
    const int nib = hi ? (packed >> 4) : (packed & 0x0f);
    const float scale = d * (float)sc;
    const float mn = dmin * (float)m;
    dst[(size_t)blockIdx.x * kQK + i] = scale * (float)nib - mn;
}

// GgmlDequant.DecodeQ6_KBlock (LD/GgmlDequant.cs:143-209): dst = d * s * (q - 32).
__global__ __launch_bounds__(256) void decode_row_q6k_kernel(const uint8_t* __restrict__ row, float* __restrict__ dst) {
    const uint8_t* b = row + (size_t)blockIdx.x * kQ6KBytes;
    const int i = threadIdx.x;
    const int h = i >> 7, r = i & 127, grp = r >> 5, l = r & 31;
    const int qlb = b[64 * h + l + ((grp & 1) ? 32 : 0)];
    const int nib = (grp >= 2) ? (qlb >> 4) : (qlb & 0x0f);
    const int hb = (b[128 + 32 * h + l] >> (2 * grp)) & 3;
    const int q = nib | (hb << 4);
    const int s = (int8_t)b[192 + 8 * h + (l >> 4) + 2 * grp];
    const float d = half_bits_to_float((uint16_t)(b[208] | (b[209] << 8)));
    dst[(size_t)blockIdx.x * kQK + i] = d * (float)s * (float)(q - 32);
}

// Q8Weight.DecodeRow (RT/Q8Weight.cs:81-106): dst[i] = scale[block] * quant[i].
__global__ __launch_bounds__(256) void decode_row_q8_0_kernel(const int8_t* __restrict__ q, const float* __restrict__ s,
                                                              int n, float* __restrict__ dst) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    dst[i] = s[i >> 5] * (float)q[i];
}

// ------------------------------------------------------------------------------------------ launchers

// ------------------------------------------------------------------------------------------ GGUF Q8_0 upload
// GgufReader.LoadTensorQ8_0Raw (LD/GgufReader.cs:198-266): the file's 34-byte blocks (fp16 d, 32 int8) become the
// resident planes — quants copied, d widened exactly to f32. One thread per block; blocks are 2-byte aligned, so
// the block is read as 17 halfwords.
__global__ __launch_bounds__(256) void q8_0_deinterleave_kernel(const uint16_t* __restrict__ src, int64_t n_blocks,
                                                                uint32_t* __restrict__ q, float* __restrict__ s) {
    const int64_t blk = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (blk >= n_blocks) return;
    const uint16_t* b = src + blk * 17;
    s[blk] = half_bits_to_float(b[0]);
#pragma unroll
    for (int i = 0; i < 8; i++) q[blk * 8 + i] = (uint32_t)b[1 + 2 * i] | ((uint32_t)b[2 + 2 * i] << 16);
}

// ------------------------------------------------------------------------------------------ GGUF Q5_0 / Q5_K upload
// The loader keeps 5-bit tensors as Q8_0 (LD/GgufLlamaLoader.cs:665-680 for experts, the F32 fallback of the
// per-layer tensors): every block decoded to F32 as GgmlDequant.DecodeQ5_0Block / DecodeQ5_KBlock do
// (LD/GgmlDequant.cs:222-320), then requantised with Q8Weight.QuantizeRows (RT/Q8Weight.cs:115-175). Here both
// happen in registers: eight lanes per 32-element Q8_0 block, four elements per lane, the block's absmax by three
// lane exchanges. Rows are whole numbers of blocks, so the flat 32-element block index of the tensor is also the
// block index of the resident planes. Source blocks are 2-byte aligned (22 bytes) or 16-byte aligned (176 bytes);
// they are read byte by byte (load time only).
__global__ __launch_bounds__(256) void q5_to_q8_0_kernel(const uint8_t* __restrict__ src, int kquant, int64_t n_blocks,
                                                         int8_t* __restrict__ q, float* __restrict__ s) {
    const int64_t wblk = ((int64_t)blockIdx.x * 4 + wave_id()) * 8;
    if (wblk >= n_blocks) return;
    const int lane = threadIdx.x & 63;
    const int64_t blk = wblk + (lane >> 3);
    const int sub = lane & 7;
    const bool live = blk < n_blocks;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (live && !kquant) {
        // Q5_0: d fp16 @0, qh @2 (bit i = the 5th bit of element i), qs @6 (element i < 16: low nibble of qs[i],
        // element i >= 16: high nibble of qs[i - 16]); value (q - 16) * d.
        const uint8_t* b = src + blk * 22;
        const float d = half_bits_to_float((uint16_t)(b[0] | (b[1] << 8)));
        const uint32_t qh = (uint32_t)b[2] | ((uint32_t)b[3] << 8) | ((uint32_t)b[4] << 16) | ((uint32_t)b[5] << 24);
        for (int k = 0; k < 4; k++) {
            const int i = 4 * sub + k;
            const int packed = b[6 + (i & 15)];
            const int nib = i < 16 ? (packed & 0x0f) : (packed >> 4);
            const int x = (nib | (int)(((qh >> i) & 1u) << 4)) - 16;
            v[k] = (float)x * d;
        }
    } else if (live) {
        // Q5_K: the Q4_K header (d, dmin, 12 packed scale/min bytes), qh @16, qs @48. Sub-block j = 2g + h of the
        // super-block takes the low (h = 0) or high (h = 1) nibbles of qs[32g ..] and qh bit 2g + h of qh[l].
        const uint8_t* b = src + (blk >> 3) * 176;
        const int j = (int)(blk & 7), g = j >> 1, h = j & 1;
        const float d = half_bits_to_float((uint16_t)(b[0] | (b[1] << 8)));
        const float dmin = half_bits_to_float((uint16_t)(b[2] | (b[3] << 8)));
        const uint8_t* pk = b + 4;
        int sc, m;
        if (j < 4) {
            sc = pk[j] & 63;
            m = pk[j + 4] & 63;
        } else {
            sc = (pk[j + 4] & 0x0f) | ((pk[j - 4] >> 6) << 4);
            m = (pk[j + 4] >> 4) | ((pk[j] >> 6) << 4);
        }
        const float scale = d * (float)sc;
        const float mn = dmin * (float)m;
        for (int k = 0; k < 4; k++) {
            const int l = 4 * sub + k;
            const int packed = b[48 + 32 * g + l];
            const int nib = h ? (packed >> 4) : (packed & 0x0f);
            const int hi = ((b[16 + l] >> (2 * g + h)) & 1) ? 16 : 0;
            v[k] = scale * (float)(nib + hi) - mn;
        }
    }
    u32x4 raw;
    raw.x = __builtin_bit_cast(uint32_t, v[0]);
    raw.y = __builtin_bit_cast(uint32_t, v[1]);
    raw.z = __builtin_bit_cast(uint32_t, v[2]);
    raw.w = __builtin_bit_cast(uint32_t, v[3]);
    const Q80Lane r = q8_0_quantize_lane(raw);  // every lane of the block takes part in the exchanges
    if (live) {
        reinterpret_cast<uint32_t*>(q + blk * 32)[sub] = r.packed;
        if (sub == 0) s[blk] = r.scale;
    }
}

hipError_t launch_q5_to_q8_0(const void* gguf, bool q5k, int64_t n_blocks, int8_t* q, float* s, hipStream_t st) {
    if (n_blocks <= 0) return hipSuccess;
    const int64_t grid = (n_blocks * 8 + 255) / 256;
    hipLaunchKernelGGL(q5_to_q8_0_kernel, dim3((unsigned)grid), dim3(256), 0, st, static_cast<const uint8_t*>(gguf),
                       q5k ? 1 : 0, n_blocks, q, s);
    return hipGetLastError();
}

hipError_t launch_quantize_q8k(const float* x, int64_t n_blocks, int8_t* q, float* s, int16_t* b, hipStream_t st,
                               uint16_t* bh) {
    if (n_blocks <= 0) return hipSuccess;
    const int64_t grid = (n_blocks + 15) / 16;
    hipLaunchKernelGGL(quantize_q8k_kernel, dim3((unsigned)grid), dim3(256), 0, st, x, n_blocks, q, s, b, bh);
    return hipGetLastError();
}

hipError_t launch_quantize_q8k_tiled(int type, const float* x, int rows, int in, int8_t* q, float* s, uint16_t* bh,
                                     hipStream_t st) {
    const int64_t n_blocks = (int64_t)rows * (in / kQK);
    hipLaunchKernelGGL(quantize_q8k_tiled_kernel, dim3((unsigned)((n_blocks + 15) / 16)), dim3(256), 0, st, x, n_blocks,
                       in / kQK, type == 14 ? 1 : 0, reinterpret_cast<uint8_t*>(q), reinterpret_cast<uint8_t*>(s),
                       type == 12 ? reinterpret_cast<uint8_t*>(bh) : nullptr);
    return hipGetLastError();
}

hipError_t launch_quantize_q8_0(const float* x, int64_t n_blocks, int8_t* q, float* s, hipStream_t st) {
    if (n_blocks <= 0) return hipSuccess;
    const int64_t grid = (n_blocks * 8 + 255) / 256;
    hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((unsigned)grid), dim3(256), 0, st, x, n_blocks, q, s);
    return hipGetLastError();
}

hipError_t launch_q8_0_deinterleave(const void* gguf, int64_t n_blocks, int8_t* q, float* s, hipStream_t st) {
    if (n_blocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(q8_0_deinterleave_kernel, dim3((unsigned)((n_blocks + 255) / 256)), dim3(256), 0, st,
                       static_cast<const uint16_t*>(gguf), n_blocks, reinterpret_cast<uint32_t*>(q), s);
    return hipGetLastError();
}

hipError_t launch_encode_q4k(const float* w, int64_t n_blocks, uint8_t* dst, hipStream_t st) {
    if (n_blocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(encode_q4k_kernel, dim3((unsigned)((n_blocks + 15) / 16)), dim3(256), 0, st, w, n_blocks, dst);
    return hipGetLastError();
}

hipError_t launch_encode_q6k(const float* w, int64_t n_blocks, uint8_t* dst, hipStream_t st) {
    if (n_blocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(encode_q6k_kernel, dim3((unsigned)((n_blocks + 15) / 16)), dim3(256), 0, st, w, n_blocks, dst);
    return hipGetLastError();
}

hipError_t launch_decode_row(int type, const void* blocks, const float* scales, int in, int row, float* dst,
                             hipStream_t st) {
    if (type == 12) {
        const uint8_t* r = static_cast<const uint8_t*>(blocks) + (size_t)row * (in / kQK) * kQ4KBytes;
        hipLaunchKernelGGL(decode_row_q4k_kernel, dim3(in / kQK), dim3(256), 0, st, r, dst);
    } else if (type == 14) {
        const uint8_t* r = static_cast<const uint8_t*>(blocks) + (size_t)row * (in / kQK) * kQ6KBytes;
        hipLaunchKernelGGL(decode_row_q6k_kernel, dim3(in / kQK), dim3(256), 0, st, r, dst);
    } else {
        const int8_t* q = static_cast<const int8_t*>(blocks) + (size_t)row * in;
        const float* s = scales + (size_t)row * (in / 32);
        hipLaunchKernelGGL(decode_row_q8_0_kernel, dim3((in + 255) / 256), dim3(256), 0, st, q, s, in, dst);
    }
    return hipGetLastError();
}

}  // namespace ovfq
