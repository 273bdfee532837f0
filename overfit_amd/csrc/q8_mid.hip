// q8_mid.hip — Q8_0 projections (and the per-head attention output) of a few to some hundred activation rows on int8 MFMA,
// from an activation quantised in operand order.
//
// Q8DotKernel.ProjectBatched (RT/Q8DotKernel.cs:352-445): per 32-element block the exact int32 dot, the reference's
// (wScale * aScale) * dot, and the block values added in ascending order from +0 (Dot, :127-137); per-head Wo
// (RT/CachedMultiHeadAttention.cs:600-614, :689-710): each head's sum added to the running output in ascending order.
//
// A block is one v_mfma_i32_16x16x32_i8 per 16 x 16 tile. The scale products of four blocks come from one
// v_mfma_f32_16x16x1_4b_f32 (sixteen products a lane, each a single multiplication added to zero, subnormal and non-finite
// factors and products included: test_gpu_q8_mid.py compares a million pairs of any exponent), which leaves the
// vector units a conversion, a multiplication and an addition per block value instead of those, the product and the loads of
// its factors. A sum never is -0, so that blocks past a plane's end can be added as zeros.
//
// The contraction goes in groups of up to four blocks (128 elements) that never cross a weight plane (a head's); the
// activation lies as one 2 KiB record of quants and 256 bytes of scales per group and 16 rows (launch_quantize_q8_0_tiled):
// lane (g, r) of a wave holds bytes 8 g .. 8 g + 7 of row r's blocks, two blocks to each of two 16-byte loads, and the scale of
// block g. A wave's 16 weight rows of a group come by LDS DMA, 128 bytes a row whose 16-byte pieces are XOR-swizzled by the
// row, with the rows' scales beside them.
//
// MI355X, graph replay, us with the quantise launch, before (one-wave workgroups of 16 outputs up to 16 rows, then the 64 x 64
// tile; heads in launches of eight rows below 32) / now: 4096x4096 at 12 / 32 / 64 / 128 / 300 / 512 rows 27.8 / 30.8 / 31.2 /
// 31.7 / 42.7 / 45.4 -> 11.5 / 14.5 / 19.3 / 20.3 / 34.2 / 42.8; 4096x14336 at 4 / 16 / 32 / 300 rows 51.2 / 81.7 / 95.3 / 131
// -> 22.7 / 22.9 / 33.7 / 99.7; 14336x4096 at 16 / 64 / 512 rows 31.4 / 33.2 / 132 -> 20.7 / 30.1 / 122; per-head Wo of 32 x
// 4096x128 at 8 / 16 / 64 / 300 rows 18.1 / 26.9 / 35.3 / 46.1 -> 11.8 / 12.0 / 22.0 / 36.3.
#include "ovfq_device.h"
#include "ovfq_launch.h"

namespace ovfq {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct Q8Args {
    const int8_t* wq[kHeadsMax];  // weight planes: one, or a head's each
    const float* ws[kHeadsMax];
    const float* bias;
    float* y;
    int n_out;
    int planes;
    int in;       // elements of a plane's row
    int rows;
    int subs;     // 16-row activation tiles
    int n_tiles;  // activation tiles of a workgroup's height
    int o_tiles;  // weight tiles of a workgroup's width
    const int8_t* q;
    const float* s;
};

// One weight group of a wave in LDS.
constexpr int kQ8Slot = 16 * 128 + 256;
constexpr int kQ8Fetch = 3;  // memory operations of fetch()

// What a lane needs to bring in and read back its wave's 16 weight rows of a group.
struct Q8Weights {
    uint32_t row_src[2];  // byte offset of the lane's two pieces in group 0 of a plane
    uint32_t scale_src;
    uint32_t piece;  // LDS offset of the lane's bytes of block 0 in its row; block j: piece ^ (32 j)
    uint32_t row;    // LDS offset of the lane's row
};

__device__ __forceinline__ Q8Weights q8_weights(uint32_t wk, uint32_t wnb, int lane) {
    Q8Weights w;
    const uint32_t g = (uint32_t)lane >> 4, r16 = (uint32_t)lane & 15u;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t row = 8u * i + ((uint32_t)lane >> 3);
        w.row_src[i] = row * wk + 16u * (((uint32_t)lane & 7u) ^ ((row >> 1) & 7u));
    }
    w.scale_src = (r16 * wnb + g) * 4u;
    w.row = r16 * 128u;
    w.piece = 16u * ((g >> 1) ^ ((r16 >> 1) & 7u)) + 8u * (g & 1u);
    return w;
}

// Group lb0 / 4 of a plane into `slot`; rows past n_out and bytes past the plane read zeros or other rows' bytes, unused.
__device__ __forceinline__ void q8_fetch(const Q8Weights& w, const int8_t* plane, const float* scales, uint32_t o0,
                                         uint32_t wk, uint32_t wnb, uint32_t rows, uint32_t lb0, uint8_t* slot) {
    const __amdgpu_buffer_rsrc_t wr = make_rsrc(plane + (uint64_t)o0 * wk, rows * wk);
    const __amdgpu_buffer_rsrc_t sr = make_rsrc(scales + (uint64_t)o0 * wnb, rows * wnb * 4u);
#pragma unroll
    for (int i = 0; i < 2; i++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void*)(slot + 1024 * i), 16,
                                                 (int)(w.row_src[i] + lb0 * 32u), 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(sr, (__attribute__((address_space(3))) void*)(slot + 2048), 4,
                                             (int)(w.scale_src + lb0 * 4u), 0, 0, 0);
}

struct Q8Group {
    u32x2 b[4];   // the lane's bytes of the four blocks of its weight row
    float scale;  // of block g
};
// Reads a slot back once all but the last kLeft memory operations of the wave are done (one asm block: the compiler cannot
// tell which DMAs a read of its own depends on).
template <int kLeft>
__device__ __forceinline__ Q8Group q8_read(const Q8Weights& w, uint32_t slot, int lane) {
    Q8Group r;
    uint32_t sc;
    const uint32_t a = slot + w.row;
    asm volatile("s_waitcnt vmcnt(%10)\n\t"
                 "ds_read_b64 %0, %5\n\t"
                 "ds_read_b64 %1, %6\n\t"
                 "ds_read_b64 %2, %7\n\t"
                 "ds_read_b64 %3, %8\n\t"
                 "ds_read_b32 %4, %9 offset:2048\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(r.b[0]), "=&v"(r.b[1]), "=&v"(r.b[2]), "=&v"(r.b[3]), "=&v"(sc)
                 : "v"(a + w.piece), "v"(a + (w.piece ^ 32u)), "v"(a + (w.piece ^ 64u)), "v"(a + (w.piece ^ 96u)),
                   "v"(slot + 4u * (uint32_t)lane), "n"(kLeft)
                 : "memory");
    r.scale = as_float(sc);
    return r;
}

__device__ __forceinline__ i32x4 q8_mfma(uint32_t a0, uint32_t a1, u32x2 b) {
    const long av = (long)(((uint64_t)a1 << 32) | a0), bv = __builtin_bit_cast(long, b);
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(av, bv, i32x4{0, 0, 0, 0}, 0, 0, 0);
}
// Products of the activation scales (lane (g, r): row r, block g) and the weight scales (column r, block g): element
// 4 j + i is block j's at (row 4 g + i, the lane's column).
__device__ __forceinline__ f32x16 q8_scales(float xs, float ws) {
    f32x16 zero;
#pragma unroll
    for (int i = 0; i < 16; i++) zero[i] = 0.0f;
    return __builtin_amdgcn_mfma_f32_16x16x1f32(xs, ws, zero, 0, 0, 0);
}

// Walks a wave's groups plane by plane; the plane's pointers are loaded one advance ahead of their use.
template <bool kHeads>
struct Q8Cursor {
    const int8_t* q;
    const float* s;
    int h, g;
    __device__ __forceinline__ void start(const Q8Args& a, int gph, int gi) {
        h = kHeads ? gi / gph : 0;
        g = gi - h * gph;
        load(a);
    }
    // by `step` groups, step = sq * gph + sr
    __device__ __forceinline__ void advance(const Q8Args& a, int gph, int step, int sq, int sr) {
        if constexpr (kHeads) {
            g += sr;
            h += sq;
            if (g >= gph) {
                g -= gph;
                h++;
            }
            load(a);
        } else {
            g += step;
        }
    }
    __device__ __forceinline__ void load(const Q8Args& a) {
        const int p = kHeads ? min(h, a.planes - 1) : 0;  // past the last group: read, unused
        q = a.wq[p];
        s = a.ws[p];
    }
};

// ------------------------------------------------------------------------------------------ panel kernel
// 64 outputs (16 a wave) x 16 T rows a workgroup, the groups in ascending order, the sums in registers. The activation
// (shared by the four waves) and each wave's weights are DMA'd two steps ahead; the one wait of a step leaves the next step's in
// flight. Bound by the block values' three vector operations beside the matrix work: with heads of 32 x 4096x128 at 300 rows (33.8
// us, T = 3) vector instructions issue 65 % of the time and the matrix units work 23 %, a third of it beside them, with 1.6 waves a
// SIMD (a conversion takes twice the issue of a multiplication or addition: 60 against 111 lanes a clock and CU). 4096x4096 at 512
// rows, 40.3 us: 30 were left with the DMAs taken out. Eight waves a workgroup, each with half the rows, were no faster (512 rows
// 43.4; 64 rows 20.6 instead of 19.5), nor were more groups in flight.
// J: blocks of a group that are computed (planes of fewer than four blocks).
template <int T, bool kHeads, int J = 4>
__global__ __launch_bounds__(256, 2) void q8_0_panel_kernel(const Q8Args a) {
    __shared__ __align__(16) uint8_t ring[3][4][kQ8Slot];
    __shared__ __align__(16) uint8_t act0[T * 2048], act1[T * 2048], act2[T * 2048];
    __shared__ __align__(16) uint32_t sc0[4 * 64], sc1[4 * 64], sc2[4 * 64];
    constexpr int kStage = (T + 1) / 2 + 1;  // memory operations of stage()
    const int wave = wave_id();
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    // XCD-aware: the activation tiles of one weight tile run on one XCD (blockIdx % 8) and share its L2
    const int local = blockIdx.x >> 3;
    const int o_tile = (blockIdx.x & 7) + 8 * (local / a.n_tiles);
    if (o_tile >= a.o_tiles) return;  // uniform over the workgroup
    const int o0 = o_tile * 64 + wave * 16, n0 = local % a.n_tiles * 16 * T;
    const uint32_t wk = (uint32_t)a.in, wnb = wk / 32;
    const int gph = (int)(wnb + 3) / 4, ng = kHeads ? a.planes * gph : gph;
    const uint32_t w_rows = (uint32_t)__builtin_amdgcn_readfirstlane(max(0, min(16, a.n_out - o0)));
    const uint32_t w_o0 = w_rows ? (uint32_t)o0 : 0u;
    const Q8Weights w = q8_weights(wk, wnb, lane);
    Q8Cursor<kHeads> next;
    next.start(a, gph, 0);
    auto fetch = [&](int k) {
        q8_fetch(w, next.q, next.s, w_o0, wk, wnb, w_rows, (uint32_t)next.g * 4u, ring[k][wave]);
        next.advance(a, gph, 1, gph == 1, gph > 1);
    };
    // wave w moves a quarter of the tiles' quants, and tile w's scales
    const uint64_t recs = (uint64_t)a.subs * (uint64_t)ng, rec0 = (uint64_t)(n0 / 16) * (uint64_t)ng;
    const __amdgpu_buffer_rsrc_t qr = make_rsrc(a.q + rec0 * 2048, rsrc_bytes(recs * 2048, rec0 * 2048));
    const __amdgpu_buffer_rsrc_t sr = make_rsrc(a.s + rec0 * 64, rsrc_bytes(recs * 256, rec0 * 256));
    constexpr int kQuarter = T * 512;  // bytes
    auto stage = [&](int gi, uint8_t* act, uint32_t* sc) {
#pragma unroll
        for (int i = 0; i < (T + 1) / 2; i++) {
            const uint32_t at = (uint32_t)(wave * kQuarter + 1024 * i) + 16u * (uint32_t)lane;  // in the tiles
            if (1024 * i + 1024 <= kQuarter || lane < (kQuarter - 1024 * i) / 16)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    qr, (__attribute__((address_space(3))) void*)(act + wave * kQuarter + 1024 * i), 16,
                    (int)((at / 2048u * (uint32_t)ng + (uint32_t)gi) * 2048u + at % 2048u), 0, 0, 0);
        }
        // every wave, so that all count alike: a wave past T brings in scales that nothing reads
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            sr, (__attribute__((address_space(3))) void*)(sc + wave * 64), 4,
            (int)((uint32_t)(wave * ng + gi) * 256u + 4u * (uint32_t)lane), 0, 0, 0);
    };
    const uint32_t slot = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)&ring[0][wave][0];
    float acc[T][4], tot[kHeads ? T : 1][4];
    const int o = o0 + r16;
    const float bias_o = a.bias && o < a.n_out ? a.bias[o] : 0.0f;
#pragma unroll
    for (int s = 0; s < T; s++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            acc[s][i] = 0.0f;
            if (kHeads) tot[s][i] = bias_o;
        }
    uint32_t left = wnb;  // blocks of the plane not yet added
    auto step = [&](int gi, int k, const uint8_t* act, const uint32_t* sc, uint8_t* act_n, uint32_t* sc_n) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0x0070 | (kStage + kQ8Fetch));  // vmcnt(..) lgkmcnt(0): all but the next step's data
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        stage(gi + 2, act_n, sc_n);
        asm volatile("" ::: "memory");
        fetch(k == 0 ? 2 : k - 1);
        Q8Group b = q8_read<63>(w, slot + (uint32_t)(k * 4 * kQ8Slot), lane);
        // blocks past the plane's end add a zero (the scales read there are other rows' or leftovers)
        const uint32_t in = (uint32_t)g < left ? 0xffffffffu : 0u;
        b.scale = as_float(__builtin_bit_cast(uint32_t, b.scale) & in);
#pragma unroll
        for (int s = 0; s < T; s++) {
            const u32x4 q0 = *reinterpret_cast<const u32x4*>(act + s * 2048 + 16 * lane);
            const u32x4 q1 = *reinterpret_cast<const u32x4*>(act + s * 2048 + 1024 + 16 * lane);
            const f32x16 sp = q8_scales(as_float(sc[s * 64 + lane] & in), b.scale);
            const i32x4 d[4] = {q8_mfma(q0.x, q0.y, b.b[0]), q8_mfma(q0.z, q0.w, b.b[1]), q8_mfma(q1.x, q1.y, b.b[2]),
                                q8_mfma(q1.z, q1.w, b.b[3])};  // those past J are dropped by the compiler
#pragma unroll
            for (int j = 0; j < J; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[s][i] += sp[4 * j + i] * (float)d[j][i];
        }
        // keeps the step's additions here: the compiler else leaves those of three steps to the third, their inputs in registers
#pragma unroll
        for (int s = 0; s < T; s++) asm volatile("" : "+v"(acc[s][0]), "+v"(acc[s][1]), "+v"(acc[s][2]), "+v"(acc[s][3]));
        left -= 4;
        if (kHeads && (int)left <= 0) {  // the head's last group
            left = wnb;
#pragma unroll
            for (int s = 0; s < T; s++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    tot[s][i] += acc[s][i];
                    acc[s][i] = 0.0f;
                }
        }
    };
    fetch(0);
    asm volatile("" ::: "memory");
    stage(0, act0, sc0);
    asm volatile("" ::: "memory");
    stage(1, act1, sc1);
    asm volatile("" ::: "memory");
    fetch(1);
    int gi = 0;
    for (; gi + 2 < ng; gi += 3) {
        step(gi, 0, act0, sc0, act2, sc2);
        step(gi + 1, 1, act1, sc1, act0, sc0);
        step(gi + 2, 2, act2, sc2, act1, sc1);
    }
    if (gi < ng) step(gi, 0, act0, sc0, act2, sc2);
    if (gi + 1 < ng) step(gi + 1, 1, act1, sc1, act0, sc0);
#pragma unroll
    for (int s = 0; s < T; s++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n = n0 + s * 16 + 4 * g + i;
            if (n >= a.rows || o >= a.n_out) continue;
            a.y[(size_t)n * a.n_out + o] = kHeads ? tot[s][i] : a.bias ? bias_o + acc[s][i] : acc[s][i];
        }
    __builtin_amdgcn_s_waitcnt(0);  // no DMA lands in LDS that another workgroup may have by then
}

// ------------------------------------------------------------------------------------------ split kernel
// 16 outputs x 16 T rows (T = 1, 2) a workgroup, wave w taking groups w, w + W, ... (W = 4, 8 waves): a matrix gives as many
// workgroups as it has 16-row tiles, and W times the loads in flight of one that walks its groups in order. A round leaves
// 4 W block values per output in LDS, which the workgroup's threads add up in order between two barriers. Bound by the
// latency of a round (about 1.3 us, four rounds of 4096 inputs with eight waves), then by the LDS traffic of the values.
template <int T, int W, bool kHeads>
__global__ __launch_bounds__(64 * W, 2) void q8_0_split_kernel(const Q8Args a) {
    constexpr int kOuts = 256 * T, kThreads = 64 * W, kPer = kOuts > kThreads ? kOuts / kThreads : 1;
    __shared__ __align__(16) uint8_t ring[3][W][kQ8Slot];
    __shared__ __align__(16) float vals[W][4][kOuts];
    const int wave = wave_id();
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    const int local = blockIdx.x >> 3;
    const int o_tile = (blockIdx.x & 7) + 8 * (local / a.n_tiles);
    if (o_tile >= a.o_tiles) return;  // uniform over the workgroup
    const int o0 = o_tile * 16, n0 = local % a.n_tiles * 16 * T;
    const uint32_t wk = (uint32_t)a.in, wnb = wk / 32;
    const int gph = (int)(wnb + 3) / 4, ng = kHeads ? a.planes * gph : gph;
    const uint32_t w_rows = (uint32_t)min(16, a.n_out - o0);
    const Q8Weights w = q8_weights(wk, wnb, lane);
    const int adv_q = kHeads ? W / gph : 0, adv_r = kHeads ? W % gph : 0;
    Q8Cursor<kHeads> next;
    next.start(a, gph, wave);
    auto fetch = [&](int k) {
        q8_fetch(w, next.q, next.s, (uint32_t)o0, wk, wnb, w_rows, (uint32_t)next.g * 4u, ring[k][wave]);
        next.advance(a, gph, W, adv_q, adv_r);
    };
    const uint64_t recs = (uint64_t)a.subs * (uint64_t)ng, rec0 = (uint64_t)(n0 / 16) * (uint64_t)ng;
    const __amdgpu_buffer_rsrc_t qr = make_rsrc(a.q + rec0 * 2048, rsrc_bytes(recs * 2048, rec0 * 2048));
    const __amdgpu_buffer_rsrc_t sr = make_rsrc(a.s + rec0 * 64, rsrc_bytes(recs * 256, rec0 * 256));
    struct Act {
        u32x4 q[T][2];
        uint32_t s[T];
    };
    auto load_act = [&](int gi, Act& v) {
#pragma unroll
        for (int s = 0; s < T; s++) {
            const uint32_t rec = (uint32_t)(s * ng + gi);
            v.q[s][0] = ld4(qr, rec * 2048u + 16u * (uint32_t)lane);
            v.q[s][1] = ld4(qr, rec * 2048u + 1024u + 16u * (uint32_t)lane);
            v.s[s] = ld1(sr, rec * 256u + 4u * (uint32_t)lane);
        }
    };
    // a round's weights are read with at least one round's activation and two rounds' weights in flight
    constexpr int kLeft = 3 * T + 2 * kQ8Fetch;
    const uint32_t slot = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)&ring[0][wave][0];
    // output idx: column (idx >> 4) & 15, row (idx >> 8) * 16 + (idx & 15)
    float sum[kPer], tot[kPer];
#pragma unroll
    for (int p = 0; p < kPer; p++) {
        const int o = o0 + ((((int)threadIdx.x + p * kThreads) >> 4) & 15);
        sum[p] = 0.0f;
        tot[p] = kHeads && a.bias && o < a.n_out ? a.bias[o] : 0.0f;
    }
    auto barrier = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): a plain __syncthreads would also wait for the DMAs in flight
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    int my_g = kHeads ? wave % gph : wave;  // the wave's group in its plane
    int sum_g = 0;                          // the round's first group in its plane
    auto step = [&](int r, int k, const Act& cur, Act& nxt) {
        const int gi = r * W + wave;
        Q8Group b = q8_read<kLeft>(w, slot + (uint32_t)(k * W * kQ8Slot), lane);
        load_act(gi + W, nxt);
        asm volatile("" ::: "memory");
        fetch(k);  // the slot has been read above
        // blocks past the plane's end and groups past the last leave zeros (the scales read there are other rows' or
        // leftovers)
        const uint32_t in = gi < ng && (uint32_t)(4 * my_g + g) < wnb ? 0xffffffffu : 0u;
        b.scale = as_float(__builtin_bit_cast(uint32_t, b.scale) & in);
        if constexpr (kHeads) {
            my_g += adv_r;
            if (my_g >= gph) my_g -= gph;
        } else {
            my_g += W;
        }
#pragma unroll
        for (int s = 0; s < T; s++) {
            const f32x16 sp = q8_scales(as_float(cur.s[s] & in), b.scale);
            const u32x4 q0 = cur.q[s][0], q1 = cur.q[s][1];
            const i32x4 d[4] = {q8_mfma(q0.x, q0.y, b.b[0]), q8_mfma(q0.z, q0.w, b.b[1]), q8_mfma(q1.x, q1.y, b.b[2]),
                                q8_mfma(q1.z, q1.w, b.b[3])};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                f32x4 v;
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = sp[4 * j + i] * (float)d[j][i];
                *reinterpret_cast<f32x4*>(&vals[wave][j][s * 256 + r16 * 16 + 4 * g]) = v;
            }
        }
        barrier();
#pragma unroll
        for (int p = 0; p < kPer; p++) {
            const int idx = (int)threadIdx.x + p * kThreads;
            if (kOuts < kThreads && idx >= kOuts) continue;
            float v[W][4];
#pragma unroll
            for (int i = 0; i < W; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) v[i][j] = vals[i][j][idx];
            int in_plane = sum_g;
#pragma unroll
            for (int i = 0; i < W; i++) {
#pragma unroll
                for (int j = 0; j < 4; j++) sum[p] += v[i][j];
                if (kHeads && ++in_plane == gph) {
                    in_plane = 0;
                    tot[p] += sum[p];
                    sum[p] = 0.0f;
                }
            }
        }
        if constexpr (kHeads) {
            sum_g += adv_r;
            if (sum_g >= gph) sum_g -= gph;
        }
        barrier();  // the values are read: the next round may write
    };
    Act a0, a1;
    fetch(0);
    asm volatile("" ::: "memory");  // kLeft counts on this order
    load_act(wave, a0);
    asm volatile("" ::: "memory");
    fetch(1);
    fetch(2);
    const int rounds = (ng + W - 1) / W;
    int k = 0;
    auto next_slot = [](int i) { return i == 2 ? 0 : i + 1; };
    int r = 0;
    for (; r + 1 < rounds; r += 2) {
        step(r, k, a0, a1);
        k = next_slot(k);
        step(r + 1, k, a1, a0);
        k = next_slot(k);
    }
    if (r < rounds) step(r, k, a0, a1);
#pragma unroll
    for (int p = 0; p < kPer; p++) {
        const int idx = (int)threadIdx.x + p * kThreads;
        const int o = o0 + ((idx >> 4) & 15), n = n0 + (idx >> 8) * 16 + (idx & 15);
        if (idx < kOuts && o < a.n_out && n < a.rows)
            a.y[(size_t)n * a.n_out + o] = kHeads ? tot[p] : a.bias ? a.bias[o] + sum[p] : sum[p];
    }
    __builtin_amdgcn_s_waitcnt(0);  // no DMA lands in LDS that another workgroup may have by then
}

// ------------------------------------------------------------------------------------------ quantiser
// Q8DotKernel.Quantize (RT/Q8DotKernel.cs:42-91) of rows x (planes * plane_in) into the records above: eight lanes a block.
__global__ __launch_bounds__(256) void quantize_q8_0_tiled_kernel(const float* __restrict__ x, int64_t n_blocks, int nb,
                                                                  int wnb, int gph, uint8_t* __restrict__ q,
                                                                  float* __restrict__ s) {
    const int64_t wblk = ((int64_t)blockIdx.x * 4 + wave_id()) * 8;
    const int lane = threadIdx.x & 63;
    const int64_t blk = wblk + (lane >> 3);
    if (wblk >= n_blocks) return;
    const int sub = lane & 7;  // elements 4 sub .. 4 sub + 3
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(x + wblk * 32, rsrc_bytes((uint64_t)n_blocks * 128, (uint64_t)wblk * 128));
    const Q80Lane r = q8_0_quantize_lane(ld4(xr, lane * 16));
    if (blk >= n_blocks) return;
    const int64_t row = blk / nb;
    const int b = (int)(blk - row * nb), plane = b / wnb, bp = b - plane * wnb;
    const int64_t rec = (row >> 4) * ((int64_t)(nb / wnb) * gph) + plane * gph + bp / 4;
    const int j = bp & 3, r16 = (int)(row & 15), g = sub >> 1;
    uint8_t* dst = q + rec * 2048 + (j >> 1) * 1024 + (g * 16 + r16) * 16 + (j & 1) * 8 + (sub & 1) * 4;
    *reinterpret_cast<uint32_t*>(dst) = r.packed;
    if (sub == 0) s[rec * 64 + j * 16 + r16] = r.scale;
}

hipError_t launch_quantize_q8_0_tiled(const float* x, int rows, int planes, int plane_in, int8_t* q, float* s,
                                      hipStream_t st) {
    const int wnb = plane_in / 32, nb = planes * wnb;
    const int64_t n_blocks = (int64_t)rows * nb;
    hipLaunchKernelGGL(quantize_q8_0_tiled_kernel, dim3((unsigned)((n_blocks + 31) / 32)), dim3(256), 0, st, x, n_blocks, nb,
                       wnb, (wnb + 3) / 4, reinterpret_cast<uint8_t*>(q), s);
    return hipGetLastError();
}

template <bool kHeads, int J>
static hipError_t launch_panel_t(const Q8Args& a, int T, dim3 grid, hipStream_t st) {
    if (T == 2)
        hipLaunchKernelGGL((q8_0_panel_kernel<2, kHeads, J>), grid, dim3(256), 0, st, a);
    else if (T == 3)
        hipLaunchKernelGGL((q8_0_panel_kernel<3, kHeads, J>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((q8_0_panel_kernel<4, kHeads, J>), grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

template <bool kHeads>
static hipError_t launch_panel(Q8Args& a, hipStream_t st) {
    a.o_tiles = (a.n_out + 63) / 64;
    // Rows of a workgroup: a CU's step takes about T + 0.84 (in 0.125 us) for each of its workgroups, and one unit more where
    // it has only one, whose waits nothing hides (4096x4096, us at T = 2 / 3 / 4: 128 rows 20.3 / 25.0 / 29.1, 160 rows 28.5 /
    // 25.5 / 29.6, 300 rows 39.0 / 34.4 / 41.3, 512 rows 52.6 / 47.0 / 43.6).
    int T = 2;
    double best = 1e30;
    for (int t = 2; t <= 4; t++) {
        const double n = (double)(((long)((a.o_tiles + 7) / 8) * ((a.subs + t - 1) / t) + 31) / 32);  // of the busiest XCD
        const double cost = n * (t + 0.84) + (n == 1 ? 1.0 : 0.0);
        if (cost < best) {
            best = cost;
            T = t;
        }
    }
    a.n_tiles = (a.subs + T - 1) / T;
    const dim3 grid((a.o_tiles + 7) / 8 * 8 * a.n_tiles);
    const int wnb = a.in / 32;
    if constexpr (kHeads)
        if (wnb < 4) return wnb < 3 ? launch_panel_t<true, 2>(a, T, grid, st) : launch_panel_t<true, 3>(a, T, grid, st);
    return launch_panel_t<kHeads, 4>(a, T, grid, st);
}

template <bool kHeads>
static hipError_t launch_mid(Q8Args& a, hipStream_t st) {
    const int wnb = a.in / 32, ng = (kHeads ? a.planes : 1) * ((wnb + 3) / 4);
    // The split kernel while its workgroups fit the CUs at one each (eight waves; four where there are no more groups than
    // that), and up to 16 rows with four waves up to two each; then the panel kernel (MI355X, us, split of 8 / of 4 / panel:
    // 4096x4096 at 16 rows 11.6 / 11.8 / 19.0, 32 rows 14.5 / 15.6 / 19.4, 64 rows 23.6 / 20.6 / 19.5; 5120x5120 at 16 rows
    // 20.4 / 17.2 / 22.7, 32 rows 27.3 / 24.6 / 23.3; 8192x8192 at 16 rows 27.2 / 25.2 / 33.3; 11264x4096 at 16 rows 25.8 /
    // 20.7 / 20.2; 896x4864 at 128 rows 16.2 / - / 22.7, 200 rows 27.3 / - / 23.4).
    a.o_tiles = (a.n_out + 15) / 16;
    const int T = a.subs == 1 ? 1 : 2;
    a.n_tiles = (a.subs + T - 1) / T;
    const long wgs = (long)((a.o_tiles + 7) / 8) * a.n_tiles * 8;  // as the busiest XCD has them (293x1088 at 370 rows, 228
                                                                   // workgroups, 36 on three XCDs: 14.5, panel 9.8)
    if (wgs > 256 && (T == 2 || wgs > 512)) return launch_panel<kHeads>(a, st);
    const dim3 grid((a.o_tiles + 7) / 8 * 8 * a.n_tiles);
    if (wgs > 256 || ng <= 4) {
        if (T == 1)
            hipLaunchKernelGGL((q8_0_split_kernel<1, 4, kHeads>), grid, dim3(256), 0, st, a);
        else
            hipLaunchKernelGGL((q8_0_split_kernel<2, 4, kHeads>), grid, dim3(256), 0, st, a);
    } else {
        if (T == 1)
            hipLaunchKernelGGL((q8_0_split_kernel<1, 8, kHeads>), grid, dim3(512), 0, st, a);
        else
            hipLaunchKernelGGL((q8_0_split_kernel<2, 8, kHeads>), grid, dim3(512), 0, st, a);
    }
    return hipGetLastError();
}

bool q8_0_mid_supported(int planes, int plane_in, int rows) {
    // 32-bit offsets: 64 activation rows and 16 weight rows; from 513 rows on the quantise launch's scattered stores cost
    // what the kernel gains (4096x4096 at 1024 / 2048 rows, us, 64 x 64 tile kernel / panel: 79.7 / 77.8, 145.5 / 150.3)
    return plane_in >= 32 && plane_in % 32 == 0 && rows >= 2 && rows <= 512 &&
           (uint64_t)planes * (uint64_t)((plane_in + 127) / 128 * 128) * 64 < (1ull << 31);
}

hipError_t launch_q8_0_mid(const int8_t* const* wq, const float* const* ws, int planes, bool heads, int plane_in, int n_out,
                           int rows, const float* bias, const int8_t* q, const float* s, float* y, hipStream_t st) {
    if (planes < 1 || planes > kHeadsMax || (planes > 1 && !heads) || !q8_0_mid_supported(planes, plane_in, rows))
        return hipErrorInvalidValue;
    Q8Args a{};
    for (int i = 0; i < planes; i++) {
        a.wq[i] = wq[i];
        a.ws[i] = ws[i];
    }
    a.bias = bias;
    a.y = y;
    a.n_out = n_out;
    a.planes = planes;
    a.in = plane_in;
    a.rows = rows;
    a.subs = (rows + 15) / 16;
    a.q = q;
    a.s = s;
    return heads ? launch_mid<true>(a, st) : launch_mid<false>(a, st);
}

}  // namespace ovfq
