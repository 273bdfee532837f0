// mfma_split.hip — Q4_K / Q6_K projections of a few to some hundred activation rows on int8 MFMA, the contraction split
// over the waves of a workgroup.
//
// Between the decode kernels (1 to 4 rows) and prefill a launch has few outputs: a 4096-row matrix and 24 rows make 64
// workgroups of the tiled kernel, each of which walks the whole row, so the launch lasts as long as one such walk (Q6_K
// 4096x14336: 92 us from 32 to 256 rows) and the small-M kernel builds its weight operands again for every 16 rows (23 us a
// pass). Here a workgroup owns 16 weight rows x 16 T activation rows (T = 1 .. 4) and its W waves (4 or 8) take super-blocks
// w, w + W, ...: every weight byte is read and every operand built once for up to 64 rows, and a 4096-row matrix gives 256
// workgroups at any row count. Each round leaves W block values per output in LDS; after the round's barrier the
// workgroup's threads add them in ascending super-block order (the reference's sequential sum), while the waves compute
// the next round into a second buffer.
//
// Both operands stream. A wave's 16 weight rows of a super-block come by LDS DMA in 16-byte pieces, three rounds ahead (a
// lane's own loads would touch 16 rows x 2 cache lines an instruction: 8 us more for every 16 activation rows when the
// activation was read that way). The activation is quantised in operand order (launch_quantize_q8k_tiled), so an A operand
// is one contiguous KiB; it is loaded a round ahead into registers.
//
// What bounds it: the latency of the rounds. Of a 24-row launch of Q6_K 4096x14336 (18.6 us beside a 4.8 us quantise launch)
// the vector units issue 42 % of the time and the matrix units 9 %, with two waves a SIMD; the same launch without operand
// build, MFMAs and activation loads took 11 us at 6 rows (4.4 TB/s), the operand build adds 2.5, the rest is rounds that wait for
// each other. Every further 16 rows add 3 us: the activation from L2 (0.9 MB a workgroup and 64 rows) and the exchange. With
// the quantise launch, before / after: 24 rows 41.4 / 25.1 us, 64 rows 76.8 / 31.9; Q4_K 4096x4096 at 64 rows 23.5 / 14.1.
#include <cstdlib>

#include "kquant_mfma.h"
#include "ovfq_launch.h"

namespace ovfq {

struct PJob {
    const uint8_t* w;
    const float* bias;
    float* y;
    int n_out;
    int tile0;  // first 16-row weight tile of this job in the launch
};

struct PArgs {
    PJob job[kMaxJobs];
    int njobs;
    int o_tiles;   // 16-row weight tiles over all jobs
    int n_tiles;   // 16T-row activation tiles
    int m_rows;    // activation rows
    int subs;      // 16-row activation tiles of the operand-ordered planes
    int spr;
    const int8_t* q;
    const float* s;
    const uint16_t* b;  // Q4_K: the bsums as fp16
};

// The weight side of a format: 16 rows' super-blocks per wave and step, DMA'd as 16-byte pieces into one LDS slot.
struct SplitQ4K {
    using F = Q4KMfma;
    static constexpr int kPieces = 9;  // 144 bytes a row
    // byte offset of a row's pieces for a block that starts `o` bytes into the resource
    __device__ __forceinline__ static uint32_t start(uint32_t o) { return o; }
    // The lane's part of the block whose row starts at LDS byte address `row`, once all but the last kLeft memory
    // operations of the wave are done. (The reads and both waits are one asm block: the compiler cannot tell which DMAs a
    // read of its own depends on, and would wait for all of them.)
    template <int kLeft>
    __device__ __forceinline__ static F::W read(uint32_t row, uint32_t, int g) {
        F::W w;
        asm volatile("s_waitcnt vmcnt(%5)\n\t"
                     "ds_read_b128 %0, %3\n\t"
                     "ds_read_b128 %1, %4 offset:16\n\t"
                     "ds_read_b128 %2, %4 offset:80\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(w.h), "=&v"(w.q[0]), "=&v"(w.q[1])
                     : "v"(row), "v"(row + 16u * (uint32_t)g), "n"(kLeft)
                     : "memory");
        return w;
    }
};

// A 210-byte block starts an even number of bytes past a 16-byte boundary: its pieces are the 14 aligned ones from that
// boundary on (14 + 210 bytes at the most), and the lane reads it back `o % 16` bytes into them as aligned dwords shifted by
// 0 or 2 bytes.
struct SplitQ6K {
    using F = Q6KMfma;
    static constexpr int kPieces = 14;
    __device__ __forceinline__ static uint32_t start(uint32_t o) { return o & ~15u; }
    template <int kLeft>
    __device__ __forceinline__ static F::W read(uint32_t row, uint32_t o, int g) {
        // the block starts at row + o % 16, and every run that the lane reads a multiple of 4 bytes after it
        const uint32_t sh = o & 3u, h = (uint32_t)g >> 1, l0 = 16u * ((uint32_t)g & 1u);
        const uint32_t blk = row + (o & 12u);
        u32x2 a01, a23, b01, b23, h01, h23, s01;
        uint32_t a4, b4, h4, s2, dw;
        asm volatile("s_waitcnt vmcnt(%16)\n\t"
                     "ds_read2_b32 %0, %12 offset1:1\n\t"
                     "ds_read2_b32 %1, %12 offset0:2 offset1:3\n\t"
                     "ds_read_b32 %2, %12 offset:16\n\t"
                     "ds_read2_b32 %3, %12 offset0:8 offset1:9\n\t"
                     "ds_read2_b32 %4, %12 offset0:10 offset1:11\n\t"
                     "ds_read_b32 %5, %12 offset:48\n\t"
                     "ds_read2_b32 %6, %13 offset1:1\n\t"
                     "ds_read2_b32 %7, %13 offset0:2 offset1:3\n\t"
                     "ds_read_b32 %8, %13 offset:16\n\t"
                     "ds_read2_b32 %9, %14 offset1:1\n\t"
                     "ds_read_b32 %10, %14 offset:8\n\t"
                     "ds_read_b32 %11, %15 offset:208\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(a01), "=&v"(a23), "=&v"(a4), "=&v"(b01), "=&v"(b23), "=&v"(b4), "=&v"(h01), "=&v"(h23),
                       "=&v"(h4), "=&v"(s01), "=&v"(s2), "=&v"(dw)
                     : "v"(blk + 64u * h + l0), "v"(blk + 128u + 32u * h + l0), "v"(blk + 192u + 8u * h), "v"(blk),
                       "n"(kLeft)
                     : "memory");
        const uint32_t ra[5] = {a01.x, a01.y, a23.x, a23.y, a4}, rb[5] = {b01.x, b01.y, b23.x, b23.y, b4};
        const uint32_t rh[5] = {h01.x, h01.y, h23.x, h23.y, h4};
        F::W w;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            w.ql[0][i] = __builtin_amdgcn_alignbyte(ra[i + 1], ra[i], sh);
            w.ql[1][i] = __builtin_amdgcn_alignbyte(rb[i + 1], rb[i], sh);
            w.qh[i] = __builtin_amdgcn_alignbyte(rh[i + 1], rh[i], sh);
        }
        const uint32_t s0 = __builtin_amdgcn_alignbyte(s01.y, s01.x, sh), s1 = __builtin_amdgcn_alignbyte(s2, s01.y, sh);
        w.sc = __builtin_amdgcn_perm(s1, s0, (g & 1) ? 0x07050301u : 0x06040200u);
        w.d = (dw >> (8u * sh)) & 0xffffu;
        return w;
    }
};

template <class FS, int T, int W>
__global__ __launch_bounds__(64 * W, 2) void kquant_mfma_split_kernel(const PArgs a) {
    using F = typename FS::F;
    constexpr bool kMin = F::kNumMfma == 3;
    constexpr int kOuts = T * 256;                         // outputs of the workgroup's tile
    constexpr int kPer = (kOuts + 64 * W - 1) / (64 * W);  // per thread in the ordered sum
    constexpr int kSlot = 16 * 16 * FS::kPieces;
    constexpr int kInstr = (FS::kPieces + 3) / 4;  // 64 pieces each
    __shared__ __align__(16) uint8_t ring[3][W][kSlot];
    __shared__ __align__(16) float vals0[W][kOuts], vals1[W][kOuts];
    __shared__ __align__(16) float scl[W][64];

    const int wave = wave_id();
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    // XCD-aware: the activation tiles of one weight tile run on one XCD (blockIdx % 8) and share its L2
    const int local = blockIdx.x >> 3;
    const int o_tile = (blockIdx.x & 7) + 8 * (local / a.n_tiles);
    if (o_tile >= a.o_tiles) return;  // uniform over the workgroup
    int j = 0;
#pragma unroll
    for (int t = 1; t < kMaxJobs; t++)
        if (t < a.njobs && o_tile >= a.job[t].tile0) j = t;
    const int n_out = a.job[j].n_out;
    const int o0 = (o_tile - a.job[j].tile0) * 16;
    const int n0 = local % a.n_tiles * 16 * T;
    const int spr = a.spr;
    const uint32_t row_bytes = (uint32_t)spr * F::kBytes;
    const uint64_t wbase = (uint64_t)o0 * row_bytes;
    const uint64_t wbase16 = wbase & ~15ull;
    // up to the end of the last block, in whole 16-byte pieces (weight allocations are a multiple of 256 bytes)
    const __amdgpu_buffer_rsrc_t wr =
        make_rsrc(a.job[j].w + wbase16, rsrc_bytes(((uint64_t)n_out * row_bytes + 15) & ~15ull, wbase16));
    const uint32_t woff = (uint32_t)(wbase - wbase16) + (uint32_t)r16 * row_bytes;  // the lane's row
    uint32_t dma_row[kInstr], dma_col[kInstr];
#pragma unroll
    for (int i = 0; i < kInstr; i++) {
        const uint32_t p = 64u * i + (uint32_t)lane;
        dma_row[i] = (uint32_t)(wbase - wbase16) + p / FS::kPieces * row_bytes;
        dma_col[i] = 16u * (p % FS::kPieces);
    }
    auto fetch = [&](uint8_t* slot, int sb) {
#pragma unroll
        for (int i = 0; i < kInstr; i++)
            if (64 * i + 64 <= 16 * FS::kPieces || lane < 16 * FS::kPieces - 64 * i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    wr, (__attribute__((address_space(3))) void*)(slot + 1024 * i), 16,
                    (int)(FS::start(dma_row[i] + (uint32_t)sb * F::kBytes) + dma_col[i]), 0, 0, 0);
    };
    // the activation from this workgroup's first tile on; tiles past the last read zeros
    const uint64_t recs = (uint64_t)a.subs * (uint64_t)spr, rec0 = (uint64_t)(n0 / 16) * (uint64_t)spr;
    const __amdgpu_buffer_rsrc_t qr = make_rsrc(a.q + rec0 * kTiledQ, rsrc_bytes(recs * kTiledQ, rec0 * kTiledQ));
    const __amdgpu_buffer_rsrc_t br =
        make_rsrc(a.b + (kMin ? rec0 * (kTiledB / 2) : 0), kMin ? rsrc_bytes(recs * kTiledB, rec0 * kTiledB) : 0u);
    const __amdgpu_buffer_rsrc_t sr = make_rsrc(a.s + rec0 * (kTiledS / 4), rsrc_bytes(recs * kTiledS, rec0 * kTiledS));

    struct Act {
        u32x4 q[T][4];
        u32x2 b[kMin ? T : 1];
        uint32_t s;
    };

    auto load_act = [&](int sb, Act& v) {
#pragma unroll
        for (int s = 0; s < T; s++) {
            const uint32_t rec = (uint32_t)(s * spr + sb);
#pragma unroll
            for (int t = 0; t < 4; t++) v.q[s][t] = ld4(qr, rec * 4096u + 1024u * t + 16u * (uint32_t)lane);
            if constexpr (kMin) v.b[s] = ld2(br, rec * 512u + 8u * (uint32_t)lane);
        }
        v.s = ld1(sr, (uint32_t)(g * spr + sb) * 64u + 4u * (uint32_t)r16);
    };

    // Memory operations of the wave that may be in flight when a round's weights are read: all those issued after the
    // weights', at the least one round's activations and two rounds' weights.
    constexpr int kLeft = T * (kMin ? 5 : 4) + 1 + 2 * kInstr;
    const uint32_t slot_adr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)&ring[0][wave][0] +
                              (uint32_t)(16 * FS::kPieces * r16);
    float sum[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++) sum[i] = 0.0f;

    // Adds one round's block values, n of them, to the running sums in ascending super-block order.
    auto add_round = [&](const float (&vals)[W][kOuts], int n) {
#pragma unroll
        for (int i = 0; i < kPer; i++) {
            const int idx = (int)threadIdx.x + 64 * W * i;
            if (kOuts % (64 * W) == 0 || idx < kOuts) {
                const float* p = &vals[0][idx];
                if (n == W) {
#pragma unroll
                    for (int j = 0; j < W; j++) sum[i] += p[j * kOuts];
                } else {
                    for (int j = 0; j < n; j++) sum[i] += p[j * kOuts];
                }
            }
        }
    };
    // One round: the wave's super-block into `vals`; the round before it, whose values every wave has written by now
    // (`prev`), is added up meanwhile.
    auto step = [&](int r, int k, float (&vals)[W][kOuts], const float (&prev)[W][kOuts], const Act& cur, Act& nxt) {
        const int sb = r * W + wave;
        const uint32_t o = woff + (uint32_t)sb * F::kBytes;
        const typename F::W w = FS::template read<kLeft>(slot_adr + (uint32_t)(k * W * kSlot), o, g);
        load_act(sb + W, nxt);
        asm volatile("" ::: "memory");
        fetch(ring[k][wave], sb + 3 * W);  // the slot has been read above
        add_round(prev, W);
        i32x4 op[4][F::kNumMfma];
        F::template operands<0>(w, g, op[0]);
        F::template operands<1>(w, g, op[1]);
        F::template operands<2>(w, g, op[2]);
        F::template operands<3>(w, g, op[3]);
        const float d = F::d_of(w), dmin = F::dmin_of(w);
        const u32x2 mb = F::min_operand(w, g);
        __builtin_amdgcn_sched_barrier(0);  // the activations are waited for after the operand build, not before
        scl[wave][lane] = as_float(cur.s);
        wave_sync();
        float* out = vals[wave];
#pragma unroll
        for (int s = 0; s < T; s++) {
            i32x4 lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const u32x4 av = cur.q[s][t];
                const i32x4 aop = i32x4{(int)av.x, (int)av.y, (int)av.z, (int)av.w};
                lo = mfma16(aop, op[t][0], lo);
                hi = mfma16(aop, op[t][1], hi);
            }
            const f32x4 q8s = *reinterpret_cast<const f32x4*>(&scl[wave][16 * s + 4 * g]);
            f32x4 v;
            if constexpr (kMin) {
                const f32x4 mn = __builtin_amdgcn_mfma_f32_16x16x16f16(
                    __builtin_bit_cast(f16x4, cur.b[s]), __builtin_bit_cast(f16x4, mb),
                    f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = q8s[i] * (d * (float)(lo[i] + (hi[i] << 3)) - dmin * mn[i]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = d * q8s[i] * (float)(lo[i] + (hi[i] << 8));
            }
            *reinterpret_cast<f32x4*>(out + s * 256 + r16 * 16 + 4 * g) = v;
        }
        // The workgroup's block values become visible to all its waves. A plain __syncthreads would also wait for the
        // DMAs in flight (they write LDS).
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    // Each wave's super-blocks: wave, wave + W, ...; weights three rounds ahead, activations one.
    Act a0, a1;
    fetch(ring[0][wave], wave);
    asm volatile("" ::: "memory");  // kLeft counts on this order
    load_act(wave, a0);
    asm volatile("" ::: "memory");
    fetch(ring[1][wave], wave + W);
    fetch(ring[2][wave], wave + 2 * W);
    const int rounds = (spr + W - 1) / W;
    // round 0 adds up zeros (a thread reads the places it writes here)
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const int idx = (int)threadIdx.x + 64 * W * i;
        if (kOuts % (64 * W) == 0 || idx < kOuts)
#pragma unroll
            for (int j = 0; j < W; j++) vals1[j][idx] = 0.0f;
    }
    int k = 0;
    auto next_slot = [](int i) { return i == 2 ? 0 : i + 1; };
    int r = 0;
    for (; r + 1 < rounds; r += 2) {
        step(r, k, vals0, vals1, a0, a1);
        k = next_slot(k);
        step(r + 1, k, vals1, vals0, a1, a0);
        k = next_slot(k);
    }
    if (r < rounds) step(r, k, vals0, vals1, a0, a1);
    add_round(rounds & 1 ? vals0 : vals1, spr - (rounds - 1) * W);
    // y[n][o] = biasO + sum   (RT/Q4KDotKernel.cs:951, RT/Q6KDotKernel.cs:507)
    const float* bias = a.job[j].bias;
    float* y = a.job[j].y;
#pragma unroll
    for (int i = 0; i < kPer; i++) {
        const int idx = (int)threadIdx.x + 64 * W * i;
        const int o = o0 + ((idx >> 4) & 15), n = n0 + (idx >> 8) * 16 + (idx & 15);
        if (idx < kOuts && n < a.m_rows && o < n_out) y[(size_t)n * n_out + o] = bias ? bias[o] + sum[i] : sum[i];
    }
    __builtin_amdgcn_s_waitcnt(0);  // no DMA lands in LDS that another workgroup may have by then
}

template <class F, int W>
static hipError_t launch_split_t(const PArgs& pa, int T, hipStream_t st) {
    const dim3 grid((pa.o_tiles + 7) / 8 * 8 * pa.n_tiles), wg(64 * W);
    if (T == 1)
        hipLaunchKernelGGL((kquant_mfma_split_kernel<F, 1, W>), grid, wg, 0, st, pa);
    else if (T == 2)
        hipLaunchKernelGGL((kquant_mfma_split_kernel<F, 2, W>), grid, wg, 0, st, pa);
    else if (T == 3)
        hipLaunchKernelGGL((kquant_mfma_split_kernel<F, 3, W>), grid, wg, 0, st, pa);
    else
        hipLaunchKernelGGL((kquant_mfma_split_kernel<F, 4, W>), grid, wg, 0, st, pa);
    return hipGetLastError();
}

template <int W>
static hipError_t launch_split_w(int type, const PArgs& pa, int T, hipStream_t st) {
    return type == 12 ? launch_split_t<SplitQ4K, W>(pa, T, st) : launch_split_t<SplitQ6K, W>(pa, T, st);
}

// ------------------------------------------------------------------------------------------ panel kernel
// Tall matrices and expert groups, 16 to 80 rows a workgroup (64 in groups): there are workgroups enough without splitting
// the contraction, but the 64-row-tiled kernel of mfma.hip waited for every load of the next super-block before the barrier
// of each one, so a super-block took a memory latency (1.8 us a step, whatever the rows). Here a workgroup's four waves own
// 16 weight rows each against the same 16 T activation rows and walk the super-blocks in order, the sums in registers. A
// step's activation tile is DMA'd into LDS one step ahead, each wave's weights two steps ahead into a ring of its own
// (mfma_split's slots), and the one wait of a step leaves the weights of the next in flight. Rows are taken 16 at a time: 45
// rows cost three tiles, not 64 or 128 rows.
// At 16 rows of gate/up (2 x 14336x4096, 66 MB) it is near the weights' stream (17 us beside the quantise launch); every 16
// rows more add 4 us. Past that it waits as much as it computes: at 45 rows (T = 3, 25.2 us) vector instructions issue 50 %
// of the time and the matrix units work 23 %, a third of it beside them, with 1.5 waves a SIMD; q/k/v of 4096 at 331 rows (T
// = 5, 36.8 us) 53 and 30 %; gathered expert groups of 40 pairs 54 and 24 %. us with the quantise launch, before / after: 32
// rows 33.8 / 26.0, 64 rows 36.8 / 34.3; Q6_K 14336x4096 at 64 rows 37.9 / 30.0; 8 experts of 48 pairs on average, 4096x7168,
// Q6_K, gate/up 156 / 138, down 115 / 71, Q4_K 106 / 118 and 75 / 55.
struct PanelGroup {
    const uint8_t* w0[kMaxExperts];
    const uint8_t* w1[kMaxExperts];
    const int* expert_off;
    const int* pair_row;  // Src::kGather: activation row of each pair
    const int* tiles;  // expert e | (tile i << 8): pairs expert_off[e] + [64 i, 64 i + 64)
    const int* tile_count;
    float* y0;
    float* y1;
    int n_rows;    // outputs per matrix
    int o_tiles1;  // 64-row weight tiles of one matrix
};

struct PanelArgs {
    PArgs p;  // job tiles, o_tiles: 64 weight rows
    PanelGroup grp;
};

// Where the activation comes from: operand-ordered planes, those of expert groups, or the row-major planes of the tokens (with
// fp16 bsums), gathered through the pairs' rows into the same order in LDS.
enum class Src { kDense, kGroups, kGather };

template <class FS, int T, Src SRC>
__global__ __launch_bounds__(256, 2) void kquant_mfma_panel_kernel(const PanelArgs args) {
    using F = typename FS::F;
    constexpr bool kMin = F::kNumMfma == 3;
    constexpr bool GRP = SRC != Src::kDense;
    constexpr int W = 4;
    constexpr int kSlot = 16 * 16 * FS::kPieces;
    constexpr int kInstr = (FS::kPieces + 3) / 4;
    __shared__ __align__(16) uint8_t ring[3][W][kSlot];
    __shared__ __align__(16) uint8_t act0[T * 4096], act1[T * 4096];
    constexpr int kPerW = (T + W - 1) / W;  // tiles whose bsums and scales a wave brings in: wave, wave + W, ..
    __shared__ __align__(16) uint8_t bs0[kMin ? kPerW * W * 512 : 16], bs1[kMin ? kPerW * W * 512 : 16];
    __shared__ __align__(16) float sc0[kPerW * W * 16], sc1[kPerW * W * 16];

    const PArgs& a = args.p;
    const int wave = wave_id();
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    const int local = blockIdx.x >> 3;
    const int o_tile = (blockIdx.x & 7) + 8 * (local / a.n_tiles);
    const int n_tile = local % a.n_tiles;
    if (o_tile >= a.o_tiles) return;  // uniform over the workgroup
    const uint8_t* wptr;
    const float* bias = nullptr;
    float* y;
    int n_out, o0, n0, m_end, sub0;  // output rows n0 .. m_end, activation tiles sub0 ..
    if constexpr (GRP) {
        if (n_tile >= args.grp.tile_count[0]) return;
        const int te = args.grp.tiles[n_tile];
        const int e = te & 0xff;
        const int mat = o_tile >= args.grp.o_tiles1 ? 1 : 0;
        wptr = mat ? args.grp.w1[e] : args.grp.w0[e];
        y = mat ? args.grp.y1 : args.grp.y0;
        n_out = args.grp.n_rows;
        o0 = (o_tile - mat * args.grp.o_tiles1) * 64 + wave * 16;
        const int pbeg = args.grp.expert_off[e];
        n0 = pbeg + (te >> 8) * 64;
        m_end = min(n0 + 64, args.grp.expert_off[e + 1]);
        sub0 = pbeg / 16 + e + (te >> 8) * 4;
    } else {
        int j = 0;
#pragma unroll
        for (int t = 1; t < kMaxJobs; t++)
            if (t < a.njobs && o_tile >= a.job[t].tile0) j = t;
        wptr = a.job[j].w;
        bias = a.job[j].bias;
        y = a.job[j].y;
        n_out = a.job[j].n_out;
        o0 = (o_tile - a.job[j].tile0) * 64 + wave * 16;
        n0 = n_tile * 16 * T;
        m_end = min(n0 + 16 * T, a.m_rows);
        sub0 = n_tile * T;
    }
    const int live = (m_end - n0 + 15) >> 4;  // 16-row tiles that hold rows
    const int spr = a.spr;
    const uint32_t row_bytes = (uint32_t)spr * F::kBytes;
    const uint64_t wbase = (uint64_t)o0 * row_bytes;
    const uint64_t wbase16 = wbase & ~15ull;
    const __amdgpu_buffer_rsrc_t wr =
        make_rsrc(wptr + wbase16, rsrc_bytes(((uint64_t)n_out * row_bytes + 15) & ~15ull, wbase16));
    const uint32_t woff = (uint32_t)(wbase - wbase16) + (uint32_t)r16 * row_bytes;
    uint32_t dma_row[kInstr], dma_col[kInstr];
#pragma unroll
    for (int i = 0; i < kInstr; i++) {
        const uint32_t p = 64u * i + (uint32_t)lane;
        dma_row[i] = (uint32_t)(wbase - wbase16) + p / FS::kPieces * row_bytes;
        dma_col[i] = 16u * (p % FS::kPieces);
    }
    auto fetch = [&](int k, int sb) {
#pragma unroll
        for (int i = 0; i < kInstr; i++)
            if (64 * i + 64 <= 16 * FS::kPieces || lane < 16 * FS::kPieces - 64 * i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    wr, (__attribute__((address_space(3))) void*)(&ring[k][wave][0] + 1024 * i), 16,
                    (int)(FS::start(dma_row[i] + (uint32_t)sb * F::kBytes) + dma_col[i]), 0, 0, 0);
    };
    // Activation: wave w moves a quarter of every tile, and tile w's bsums and scales. Offsets of the lane's pieces in
    // super-block 0 and from one super-block to the next; tiles and rows past the launch's read zeros.
    const bool gather = SRC == Src::kGather;
    const uint64_t rec0 = gather ? 0 : (uint64_t)sub0 * (uint64_t)spr;
    const uint64_t recs = gather ? 0 : (uint64_t)a.subs * (uint64_t)spr;
    const uint64_t blocks = (uint64_t)a.m_rows * (uint64_t)spr;
    const __amdgpu_buffer_rsrc_t qr = make_rsrc(
        a.q + rec0 * kTiledQ, gather ? rsrc_bytes(blocks * kQK, 0) : rsrc_bytes(recs * kTiledQ, rec0 * kTiledQ));
    const __amdgpu_buffer_rsrc_t br =
        make_rsrc(a.b + (kMin ? rec0 * (kTiledB / 2) : 0),
                  !kMin ? 0u : gather ? rsrc_bytes(blocks * 32, 0) : rsrc_bytes(recs * kTiledB, rec0 * kTiledB));
    const __amdgpu_buffer_rsrc_t sr =
        make_rsrc(a.s + rec0 * (kTiledS / 4),
                  gather ? rsrc_bytes(blocks * 4, 0) : rsrc_bytes(recs * kTiledS, rec0 * kTiledS));
    constexpr uint32_t kStepQ = SRC == Src::kGather ? kQK : kTiledQ, kStepB = SRC == Src::kGather ? 32 : kTiledB,
                       kStepS = SRC == Src::kGather ? 4 : kTiledS;
    uint32_t q_src[T], b_src[2], s_src;
    if constexpr (SRC == Src::kGather) {
        // Row by row, so that an instruction reads four rows' 256 contiguous bytes: in LDS, rows of 16 pieces XOR-swizzled by
        // the row, so that the 16 lanes of one A read hit distinct banks. Bsums: 32 bytes a row, two lanes each.
        constexpr uint32_t kAbsent = 0x80000000u;  // past every resource
        auto act_row = [&](uint32_t i) -> uint32_t {  // activation row of the tile's row i
            return n0 + (int)i < m_end ? (uint32_t)args.grp.pair_row[n0 + (int)i] : ~0u;
        };
#pragma unroll
        for (int s = 0; s < T; s++) {
            const uint32_t i = 4u * wave + (uint32_t)g, r = act_row(16u * s + i);
            q_src[s] = r == ~0u ? kAbsent : r * (uint32_t)spr * kQK + 16u * F::src_piece((uint32_t)r16 ^ i);
        }
        const uint32_t rb = act_row(16u * wave + (((uint32_t)lane >> 1) & 15u)), rs = act_row(16u * wave + (uint32_t)r16);
        b_src[0] = rb == ~0u ? kAbsent : rb * (uint32_t)spr * 32u + 16u * ((uint32_t)lane & 1u);
        s_src = rs == ~0u ? kAbsent : rs * (uint32_t)spr * 4u;
    } else {
#pragma unroll
        for (int s = 0; s < T; s++)
            q_src[s] = (uint32_t)(s * spr) * (uint32_t)kTiledQ + 1024u * wave + 16u * (uint32_t)lane;
#pragma unroll
        for (int i = 0; i < 2; i++)
            b_src[i] = (uint32_t)(wave * spr) * (uint32_t)kTiledB + 256u * i + 4u * (uint32_t)lane;
        s_src = (uint32_t)(wave * spr) * (uint32_t)kTiledS + 4u * (uint32_t)r16;
    }
    auto stage = [&](int sb, uint8_t* act, uint8_t* bs, float* sc) {
#pragma unroll
        for (int s = 0; s < T; s++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                qr, (__attribute__((address_space(3))) void*)(act + s * 4096 + wave * 1024), 16,
                (int)(q_src[s] + (uint32_t)sb * kStepQ), 0, 0, 0);
        if constexpr (kMin && SRC == Src::kGather) {
            if (lane < 32)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(br, (__attribute__((address_space(3))) void*)(bs + wave * 512), 16,
                                                         (int)(b_src[0] + (uint32_t)sb * kStepB), 0, 0, 0);
        } else if constexpr (kMin) {
#pragma unroll
            for (int i = 0; i < 2 * kPerW; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    br, (__attribute__((address_space(3))) void*)(bs + (wave + i / 2 * W) * 512 + i % 2 * 256), 4,
                    (int)(b_src[i % 2] + (uint32_t)(i / 2 * W * spr + sb) * kStepB), 0, 0, 0);
        }
        if (lane < 16)
#pragma unroll
            for (int i = 0; i < kPerW; i++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(sr, (__attribute__((address_space(3))) void*)(sc + (wave + i * W) * 16),
                                                         4, (int)(s_src + (uint32_t)(i * W * spr + sb) * kStepS), 0, 0, 0);
    };
    const uint32_t slot_adr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)&ring[0][wave][0] +
                              (uint32_t)(16 * FS::kPieces * r16);

    uint32_t a_off[4];  // the lane's A operand of MFMA t, and its bsums, in a tile's slot
#pragma unroll
    for (int t = 0; t < 4; t++)
        a_off[t] = SRC == Src::kGather ? 256u * r16 + 16u * ((4u * t + (uint32_t)g) ^ (uint32_t)r16)
                                       : 1024u * t + 16u * (uint32_t)lane;
    const uint32_t b_off = SRC == Src::kGather ? 32u * r16 + 8u * g : 8u * (uint32_t)lane;
    float out[T][4];
#pragma unroll
    for (int s = 0; s < T; s++)
#pragma unroll
        for (int i = 0; i < 4; i++) out[s][i] = 0.0f;

    auto step = [&](int sb, int k, const uint8_t* act, const uint8_t* bs, const float* sc, uint8_t* act_n, uint8_t* bs_n,
                    float* sc_n) {
        // This step's activation and weights have landed (only the next step's weights may be in flight), in every wave,
        // and every wave is done with the slots that are filled next.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0x0070 | kInstr);  // vmcnt(kInstr) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        stage(sb + 1, act_n, bs_n, sc_n);
        asm volatile("" ::: "memory");
        fetch(k == 0 ? 2 : k - 1, sb + 2);
        const typename F::W w = FS::template read<63>(slot_adr + (uint32_t)(k * W * kSlot), woff + (uint32_t)sb * F::kBytes, g);
        i32x4 op[4][F::kNumMfma];
        F::template operands<0>(w, g, op[0]);
        F::template operands<1>(w, g, op[1]);
        F::template operands<2>(w, g, op[2]);
        F::template operands<3>(w, g, op[3]);
        const float d = F::d_of(w), dmin = F::dmin_of(w);
        const u32x2 mb = F::min_operand(w, g);
#pragma unroll
        for (int s = 0; s < T; s++) {
            if (GRP && s >= live) break;
            i32x4 lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const u32x4 av = *reinterpret_cast<const u32x4*>(act + s * 4096 + a_off[t]);
                const i32x4 aop = i32x4{(int)av.x, (int)av.y, (int)av.z, (int)av.w};
                lo = mfma16(aop, op[t][0], lo);
                hi = mfma16(aop, op[t][1], hi);
            }
            const f32x4 q8s = *reinterpret_cast<const f32x4*>(sc + s * 16 + 4 * g);
            if constexpr (kMin) {
                const f16x4 bq = *reinterpret_cast<const f16x4*>(bs + s * 512 + b_off);
                const f32x4 mn = __builtin_amdgcn_mfma_f32_16x16x16f16(bq, __builtin_bit_cast(f16x4, mb),
                                                                      f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) out[s][i] += q8s[i] * (d * (float)(lo[i] + (hi[i] << 3)) - dmin * mn[i]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; i++) out[s][i] += d * q8s[i] * (float)(lo[i] + (hi[i] << 8));
            }
        }
    };
    fetch(0, 0);
    asm volatile("" ::: "memory");
    stage(0, act0, bs0, sc0);
    asm volatile("" ::: "memory");
    fetch(1, 1);
    int k = 0;
    auto next_slot = [](int i) { return i == 2 ? 0 : i + 1; };
    int sb = 0;
    for (; sb + 1 < spr; sb += 2) {
        step(sb, k, act0, bs0, sc0, act1, bs1, sc1);
        k = next_slot(k);
        step(sb + 1, k, act1, bs1, sc1, act0, bs0, sc0);
        k = next_slot(k);
    }
    if (sb < spr) step(sb, k, act0, bs0, sc0, act1, bs1, sc1);

    // y[n][o] = biasO + sum   (RT/Q4KDotKernel.cs:951, RT/Q6KDotKernel.cs:507)
    const int o = o0 + r16;
    const float bias_o = bias && o < n_out ? bias[o] : 0.0f;
#pragma unroll
    for (int s = 0; s < T; s++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n = n0 + s * 16 + 4 * g + i;
            if (n < m_end && o < n_out) y[(size_t)n * n_out + o] = bias ? bias_o + out[s][i] : out[s][i];
        }
    __builtin_amdgcn_s_waitcnt(0);  // no DMA lands in LDS that another workgroup may have by then
}

template <class FS>
static hipError_t launch_panel_t(const PanelArgs& pa, int T, hipStream_t st) {
    const dim3 grid((pa.p.o_tiles + 7) / 8 * 8 * pa.p.n_tiles), wg(256);
    if (T == 1)
        hipLaunchKernelGGL((kquant_mfma_panel_kernel<FS, 1, Src::kDense>), grid, wg, 0, st, pa);
    else if (T == 2)
        hipLaunchKernelGGL((kquant_mfma_panel_kernel<FS, 2, Src::kDense>), grid, wg, 0, st, pa);
    else if (T == 3)
        hipLaunchKernelGGL((kquant_mfma_panel_kernel<FS, 3, Src::kDense>), grid, wg, 0, st, pa);
    else if (T == 4)
        hipLaunchKernelGGL((kquant_mfma_panel_kernel<FS, 4, Src::kDense>), grid, wg, 0, st, pa);
    else if constexpr (FS::F::kNumMfma == 3)  // Q4_K: two workgroups' LDS still fit a CU
        hipLaunchKernelGGL((kquant_mfma_panel_kernel<FS, 5, Src::kDense>), grid, wg, 0, st, pa);
    return hipGetLastError();
}

hipError_t launch_project_panel(int type, const ProjJob* jobs, int njobs, int in, int rows, ActQ act,
                                hipStream_t st) {
    PanelArgs pa{};
    int tiles = 0;
    for (int i = 0; i < njobs; i++) {
        pa.p.job[i] = PJob{jobs[i].w, jobs[i].bias, jobs[i].y, jobs[i].n_rows, tiles};
        tiles += (jobs[i].n_rows + 63) / 64;
    }
    pa.p.njobs = njobs;
    pa.p.o_tiles = tiles;
    pa.p.m_rows = rows;
    pa.p.subs = (rows + 15) / 16;
    pa.p.spr = in / kQK;
    pa.p.q = act.q;
    pa.p.s = act.s;
    pa.p.b = act.bh;
    if (type == 12 && !pa.p.b) return hipErrorInvalidValue;  // the Q4_K kernel reads the bsums
    int T;
    panel_cost(type, tiles, pa.p.subs, &T);
    pa.p.n_tiles = (pa.p.subs + T - 1) / T;
    return type == 12 ? launch_panel_t<SplitQ4K>(pa, T, st) : launch_panel_t<SplitQ6K>(pa, T, st);
}

hipError_t launch_mfma_grouped(int type, const GroupLaunch& L, const int* tiles, const int* tile_count,
                               int max_tiles, hipStream_t st) {
    PanelArgs pa{};
    const int o1 = (L.n_rows + 63) / 64;
    pa.p.o_tiles = o1 * (L.w1 ? 2 : 1);
    pa.p.n_tiles = max_tiles;
    pa.p.subs = grouped_subs(L.pairs, L.experts);
    pa.p.m_rows = L.rows;
    pa.p.spr = L.in / kQK;
    pa.p.q = L.act.q;
    pa.p.s = L.act.s;
    pa.p.b = L.act.bh;
    if (L.act.tiled == (L.pair_row != nullptr) || (type == 12 && !pa.p.b)) return hipErrorInvalidValue;
    if (L.comb) return hipErrorInvalidValue;  // the combine has its own launch
    for (int e = 0; e < L.experts; e++) {
        pa.grp.w0[e] = L.w0[e];
        pa.grp.w1[e] = L.w1 ? L.w1[e] : nullptr;
    }
    pa.grp.expert_off = L.expert_off;
    pa.grp.pair_row = L.pair_row;
    pa.grp.tiles = tiles;
    pa.grp.tile_count = tile_count;
    pa.grp.y0 = L.y0;
    pa.grp.y1 = L.y1;
    pa.grp.n_rows = L.n_rows;
    pa.grp.o_tiles1 = o1;
    const dim3 grid((pa.p.o_tiles + 7) / 8 * 8 * max_tiles);
    if (type == 12 && L.pair_row)
        hipLaunchKernelGGL((kquant_mfma_panel_kernel<SplitQ4K, 4, Src::kGather>), grid, dim3(256), 0, st, pa);
    else if (type == 12)
        hipLaunchKernelGGL((kquant_mfma_panel_kernel<SplitQ4K, 4, Src::kGroups>), grid, dim3(256), 0, st, pa);
    else if (L.pair_row)
        hipLaunchKernelGGL((kquant_mfma_panel_kernel<SplitQ6K, 4, Src::kGather>), grid, dim3(256), 0, st, pa);
    else
        hipLaunchKernelGGL((kquant_mfma_panel_kernel<SplitQ6K, 4, Src::kGroups>), grid, dim3(256), 0, st, pa);
    return hipGetLastError();
}

bool mid_enabled() {
    static const bool on = [] {
        const char* v = getenv("OVFQ_SPLIT");
        return !(v && *v == '0');
    }();
    return on;
}

MidKernel mid_kernel(int type, int in, int rows, long tiles, int count, bool prepared) {
    if (!mid_enabled() || (type != 12 && type != 14) || in % kQK) return MidKernel::kNone;
    return mid_choice(type, in, rows, tiles, count, prepared);
}

hipError_t launch_project_split(int type, const ProjJob* jobs, int njobs, int in, int rows, ActQ act,
                                hipStream_t st) {
    PArgs pa{};
    int tiles = 0;
    for (int i = 0; i < njobs; i++) {
        pa.job[i] = PJob{jobs[i].w, jobs[i].bias, jobs[i].y, jobs[i].n_rows, tiles};
        tiles += (jobs[i].n_rows + 15) / 16;
    }
    pa.njobs = njobs;
    pa.o_tiles = tiles;
    pa.m_rows = rows;
    pa.subs = (rows + 15) / 16;
    pa.spr = in / kQK;
    pa.q = act.q;
    pa.s = act.s;
    pa.b = act.bh;
    if (type == 12 && !pa.b) return hipErrorInvalidValue;  // the Q4_K kernel reads the bsums
    pa.n_tiles = (pa.subs + 3) / 4;  // at most four 16-row tiles a workgroup, spread evenly
    const int T = (pa.subs + pa.n_tiles - 1) / pa.n_tiles;
    // Eight waves where that leaves at most a workgroup per CU and there are eight super-blocks to share (MI355X, us, eight /
    // four waves: Q6_K 4096x14336 at 64 rows, 256 workgroups, 30.2 / 34.0 and at 96 rows, 512 workgroups, 47.5 / 40.6; Q4_K
    // 1024x14336 at 128 rows 25.9 / 30.7, 1024x1024 at 64 rows 8.5 / 7.1).
    const int w8 = pa.spr >= 8 && (long)tiles * pa.n_tiles <= 256;
    return w8 ? launch_split_w<8>(type, pa, T, st) : launch_split_w<4>(type, pa, T, st);
}

}  // namespace ovfq
