// Large-tile f16 MFMA contraction with block-quantized int4 weights (W4A16 with more than a
// decode batch of rows, and every scale block width that is a multiple of 32).
//
// A workgroup owns a 32 MI x 32 WGN tile of D (activation rows x output channels) and walks k in
// stages of 128 through a ring of NS LDS stages filled by direct global -> LDS loads. Every wave
// owns 32 channels and all 32 MI rows of the tile, so each weight is decoded by one wave only; KS
// wave groups split every stage's four 32-k sub-steps between them, and their f32 partial tiles
// are added in LDS at the end in a fixed order.
//
// What bounds it. A sub-step of a wave is 2 MI v_mfma_f32_32x32x16_f16 of 32 cycles; beside them the
// VALU decodes the wave's 32 x 32 weights (24 instructions) and, once per scale block, multiplies
// the block's f32 partial sums by its scale into the accumulators (16 MI fused multiply-adds of 4
// cycles: with 32-wide blocks as many cycles as the MFMAs themselves). MI = 4 spreads the decode
// over four fragments, and a k-step's multiply-adds, MFMAs and operand reads are issued fragment by
// fragment (fragment i's multiply-adds of the finished block, its MFMAs of the next one, the reads
// of the one after), so that both pipes and LDS run together.
//
// Numerics: (q - 8) is exact in f16, products are exact in f32, one block's products are summed by
// the MFMA in f32, and the block sum times the f32 value of its f16 scale is accumulated in f32
// (one rounding) - the per-block scaling of the reference test's oracle. With 32-wide blocks the
// accumulators are compensated and meet in f64 wherever the kernel that the shape had before sums in
// f64 or in shorter chains.
//
// LDS layout (conflict-free): activation row r's 16-byte chunk c at c ^ (r & 15) of its 256 bytes;
// a weight row's 16 bytes of sub-step T at T ^ ((r >> 2) & 3) of its 64; scales as whole dwords (the
// aligned dword that holds the f16 scale; a lane picks its half), channel by channel. A lane of
// half h feeds 8 consecutive k per MFMA: chunks 4 T + 2 h + t of sub-step T, t = 0, 1.
//
// Loads past k and stages past the last are range-checked to zeros by the buffer resources (zero
// activations, and zero scales past the last block), so the loop has no tail and every wait is a
// constant vmcnt. The barrier of a stage sits where its last fragments are in registers.
//
// Measured: 1024 x 4096 x 11008, 128-wide blocks, f32 results 114 us (318 ms on the per-output
// kernel, the only one for blocks other than 32 wide); 32-wide blocks, compensated, f16 results, 128 x
// 4096 x 4096 22 us (45 on the chunk-stream kernel, one pass over the weights per 32 rows) and 1024 x
// 4096 x 4096 70 us (337); f32 results 78 (337) and 300 x 4096 x 4096 51 (107).
// A stage of a plain 128 x 128 tile with 32-wide blocks takes 1.65 us against 0.43 of MFMAs at 2.4 GHz:
// the multiply-adds and the decode are 0.7 us of VALU a SIMD, and the activation reads (1 KiB of LDS
// per MFMA, as each wave has one 32-channel column) slow the MFMAs further.
#pragma once

#include <type_traits>

#include "int8_tile.hpp"

namespace tqt {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct F16TileArgs
{
    int M, N, K;
    const _Float16 *A;
    long long lda;
    const uint8_t *B;
    long long bstride;  // bytes between weight rows
    const _Float16 *scale_b;
    long long ldsb;
    const void *C;
    long long ldc;
    void *D;
    long long ldd;
    const void *bias;
    float cmin, cmax;
    int bl, nblocks;
    int nan_to_min;  // a NaN sum becomes cmin (the clamp of the 32-wide-block kernels) or stays
    int tiles_m, tiles_n, per_xcd;
};

// Nibbles 2 b and 2 b + 1 of x -> two exact f16 values q - 8. A byte permute puts byte b into both
// halves of a dword, where the low half keeps the low nibble as 1024 + q and the high half the high
// nibble as 1024 + 16 q, and one packed fma (times 1 and 1/16) leaves both q - 8.
__device__ __forceinline__ uint32_t tile_decode_pair(uint32_t x, int b)
{
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 mul = h2{static_cast<_Float16>(1.0f), static_cast<_Float16>(0.0625f)};
    const h2 add = h2{static_cast<_Float16>(-1032.0f), static_cast<_Float16>(-72.0f)};
    const uint32_t t =
        __builtin_amdgcn_perm(x, x, 0x0c000c00u | static_cast<uint32_t>(b | (b << 16)));
    return __builtin_bit_cast(
        uint32_t, __builtin_elementwise_fma(
                      __builtin_bit_cast(h2, (t & 0x00f0000fu) | 0x64006400u), mul, add));
}

// SPB: 32-k sub-steps per scaling (1, 2 or 4: the scale block width is a multiple of 32 SPB).
// COMP > 0: the accumulators are compensated. A plain f32 accumulator adds k / 32 terms, a chain whose
// rounding would exceed that of the chunk-stream kernel, whose waves sum every sixteenth block and meet
// in f64 (route.hpp: the errors of both and which COMP is taken). So acc holds the sum of COMP blocks
// plus the error of the last addition to hi, the running sum (four operations every COMP blocks), and
// both meet in f64.
template <int MI, int WGN, int KS, int NSMAX, int SPB, int COMP, int OUT>
__global__ __launch_bounds__(64 * WGN * KS, 2) void w4a16_tile_kernel(F16TileArgs a)
{
    constexpr int WAVES = WGN * KS;
    constexpr int BM = 32 * MI;
    constexpr int BN = 32 * WGN;
    constexpr int SUW = 4 / KS;   // sub-steps per wave and stage
    static_assert(SUW >= SPB && SUW % SPB == 0, "a scaling unit stays in one wave");
    constexpr int NSC = 4 / SPB;  // scales per channel and stage
    constexpr int SX = BM * 256;
    constexpr int SW = BN * 64;
    constexpr int SS = BN * NSC * 4;
    constexpr int STAGE = SX + SW + SS;
    constexpr int NS = tile_stages(STAGE, NSMAX);
    static_assert(NS >= 2, "ring");
    constexpr int XPW = SX / 1024 >= WAVES ? SX / 1024 / WAVES : 1;
    constexpr int WPW = SW / 1024 >= WAVES ? SW / 1024 / WAVES : 1;
    constexpr int SPW = SS / 256 >= WAVES ? SS / 256 / WAVES : 1;
    static_assert(XPW * WAVES * 1024 >= SX && WPW * WAVES * 1024 >= SW && SPW * WAVES * 256 >= SS,
                  "the loads cover a stage");
    constexpr int PER_STAGE = XPW + WPW + SPW;
    static_assert((NS - 1) * PER_STAGE < 64, "vmcnt");
    static_assert(BM * BN * 4 * (KS - 1) <= NS * STAGE, "partial tiles fit the ring");

    __shared__ __attribute__((aligned(1024))) int8_t ring[NS * STAGE];

    int tm, tn;
    if (!tile_coords(a.tiles_m, a.tiles_n, a.per_xcd, tm, tn)) {
        return;
    }
    const int m0 = tm * BM;
    const int n0 = tn * BN;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = wave % KS;
    const int wn = wave / KS;
    const int r32 = lane & 31;
    const int h = lane >> 5;
    const int gch = n0 + wn * 32 + r32;  // this lane's channel

    // an absent bias adds -0, which leaves every value as it is
    const float pre_bias = a.bias ? load_out<OUT>(a.bias, min(gch, a.N - 1)) : -0.f;

    // load roles, 32-bit offsets from the tile's first rows (the launcher bounds the strides)
    i32x4 x_rsrc = raw_rsrc(a.A + static_cast<long long>(m0) * a.lda, kTileRecords);
    i32x4 w_rsrc = raw_rsrc(a.B + static_cast<long long>(n0) * a.bstride, kTileRecords);
    const uintptr_t s_addr =
        reinterpret_cast<uintptr_t>(a.scale_b + static_cast<long long>(n0) * a.ldsb);
    const uint32_t s_mis = static_cast<uint32_t>(s_addr & 3);
    const i32x4 s_rsrc = raw_rsrc(reinterpret_cast<const void *>(s_addr - s_mis), kTileRecords);
    auto x_blk = [&](int j) { return (wave * XPW + j) % (SX / 1024); };
    auto w_blk = [&](int j) { return (wave * WPW + j) % (SW / 1024); };
    auto x_chunk = [&](int j) {  // of this lane's row of load block j
        return static_cast<uint32_t>((lane & 15) ^ ((4 * x_blk(j) + (lane >> 4)) & 15));
    };
    auto w_chunk = [&](int) { return static_cast<uint32_t>((lane & 3) ^ ((lane >> 4) & 3)); };
    uint32_t x_off[XPW];
#pragma unroll
    for (int j = 0; j < XPW; ++j) {
        const int row = 4 * x_blk(j) + (lane >> 4);
        x_off[j] = static_cast<uint32_t>(min(row, a.M - 1 - m0)) *
                       static_cast<uint32_t>(2 * a.lda) + x_chunk(j) * 16;
    }
    uint32_t w_off[WPW];
#pragma unroll
    for (int j = 0; j < WPW; ++j) {
        const int row = 16 * w_blk(j) + (lane >> 2);
        w_off[j] = static_cast<uint32_t>(min(row, a.N - 1 - n0)) *
                       static_cast<uint32_t>(a.bstride) + w_chunk(j) * 16;
    }
    // scales: dword s of a stage is channel s / NSC, unit s % NSC; this lane's unit advances by 128
    // k per stage: its scale index and the k left behind in its block
    uint32_t s_off[SPW], s_idx, s_rem;
    {
        const uint32_t unit_k = static_cast<uint32_t>(lane % NSC) * (32 * SPB);
        s_idx = unit_k / static_cast<uint32_t>(a.bl);
        s_rem = unit_k - s_idx * static_cast<uint32_t>(a.bl);
    }
#pragma unroll
    for (int j = 0; j < SPW; ++j) {
        const int dw = ((wave * SPW + j) % (SS / 256)) * 64 + lane;
        s_off[j] = static_cast<uint32_t>(min(dw / NSC, a.N - 1 - n0)) *
                       static_cast<uint32_t>(2 * a.ldsb) + s_mis;
    }
    const uint32_t s_q = 128u / static_cast<uint32_t>(a.bl);
    const uint32_t s_r = 128u - s_q * static_cast<uint32_t>(a.bl);
    const uint32_t K = static_cast<uint32_t>(a.K);
    const int nst = (a.K + 127) / 128;
    auto issue = [&](int st, int off) {  // called for st = 0, 1, 2, ... in order
        const uint32_t k0 = static_cast<uint32_t>(st) * 128u;
        x_rsrc[2] = w_rsrc[2] = st < nst ? kTileRecords : 0;  // stages past the last: all zeros
        if (st == nst - 1 && (K & 127) != 0) {
            // k ends inside this stage: the chunks past it out of range (once per launch)
#pragma unroll
            for (int j = 0; j < XPW; ++j) {
                x_off[j] = 8 * x_chunk(j) + k0 < K ? x_off[j] : kTileOob;
            }
#pragma unroll
            for (int j = 0; j < WPW; ++j) {
                w_off[j] = 32 * w_chunk(j) + k0 < K ? w_off[j] : kTileOob;
            }
        }
#pragma unroll
        for (int j = 0; j < XPW; ++j) {
            dma_lds16_buf_s(x_rsrc, static_cast<int>(x_off[j]), static_cast<int>(2 * k0),
                            ring + off + x_blk(j) * 1024);
        }
#pragma unroll
        for (int j = 0; j < WPW; ++j) {
            dma_lds16_buf_s(w_rsrc, static_cast<int>(w_off[j]), static_cast<int>(k0 / 2),
                            ring + off + SX + w_blk(j) * 1024);
        }
#pragma unroll
        for (int j = 0; j < SPW; ++j) {
            dma_lds4_buf(s_rsrc,
                         static_cast<int>(s_idx < static_cast<uint32_t>(a.nblocks)
                                              ? ((s_off[j] + 2 * s_idx) & ~3u) : kTileOob),
                         ring + off + SX + SW + ((wave * SPW + j) % (SS / 256)) * 256);
        }
        s_idx += s_q;
        s_rem += s_r;
        if (s_rem >= static_cast<uint32_t>(a.bl)) {
            s_rem -= static_cast<uint32_t>(a.bl);
            ++s_idx;
        }
    };

    static_assert(COMP == 0 || (SPB == 1 && (SUW % COMP == 0 || COMP % SUW == 0)),
                  "whole compensation steps per stage, or stages per step");
    f32x16 acc[MI], part[MI];
    f32x16 hi[COMP > 0 ? MI : 1];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[i][r] = 0.f;
            part[i][r] = 0.f;
            hi[COMP > 0 ? i : 0][r] = 0.f;
        }
    }
    // hi += acc, acc = what the addition lost. Where hi leaves the finite range the loss is no
    // number; any finite value then keeps an infinite sum infinite (fmed3 of a NaN is the minimum
    // of the other two).
    auto compensate = [&](int i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float t = hi[COMP > 0 ? i : 0][r] + acc[i][r];
            acc[i][r] = __builtin_amdgcn_fmed3f(acc[i][r] - (t - hi[COMP > 0 ? i : 0][r]),
                                                -3.40282347e38f, 3.40282347e38f);
            hi[COMP > 0 ? i : 0][r] = t;
        }
    };

    // LDS offsets of this lane's operands of its sub-step q (fragment i adds 32 rows)
    int x_lane[SUW][2], w_lane[SUW];
#pragma unroll
    for (int q = 0; q < SUW; ++q) {
        const int T = ks * SUW + q;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            x_lane[q][t] = r32 * 256 + (((4 * T + 2 * h + t) ^ (r32 & 15)) << 4);
        }
        w_lane[q] = SX + (wn * 32 + r32) * 64 + ((T ^ ((r32 >> 2) & 3)) << 4) + 8 * h;
    }
    // the wave's scale dwords of a stage, and which half of its dword a scale is: the parity of
    // its f16 index from an aligned address, i.e. of (row base) + (scale index)
    constexpr int NSW = NSC / KS;
    const int s_lane = SX + SW + ((wn * 32 + r32) * NSC + ks * NSW) * 4;
    const uint32_t s_par = (s_mis >> 1) + static_cast<uint32_t>(min(wn * 32 + r32, a.N - 1 - n0)) *
                                              static_cast<uint32_t>(a.ldsb & 1);
    // scale index of the wave's unit 0 .. NSW - 1 of the stage being computed (wave-uniform)
    uint32_t c_idx[NSW], c_rem[NSW];
#pragma unroll
    for (int u = 0; u < NSW; ++u) {
        const uint32_t unit_k = static_cast<uint32_t>(ks * NSW + u) * (32 * SPB);
        c_idx[u] = unit_k / static_cast<uint32_t>(a.bl);
        c_rem[u] = unit_k - c_idx[u] * static_cast<uint32_t>(a.bl);
    }

    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    // Activation fragments are read DIST fragments ahead of their MFMAs into two alternating sets:
    // the registers of a whole sub-step ahead would push the 4-fragment tile past 256.
    constexpr int DIST = MI >= 2 ? 2 : 1;
    u32x4 x[2][2];
    u32x2 raw[SUW];      // weight nibbles of a stage's sub-steps
    uint32_t w[2][2][4]; // decoded weights of this sub-step and the next
    uint32_t sraw[NSW];
    float s_cur = 0.f;   // scale of the block being summed in part
    auto read_stage = [&](int off) {
#pragma unroll
        for (int q = 0; q < SUW; ++q) {
            raw[q] = *reinterpret_cast<const u32x2 *>(ring + off + w_lane[q]);
        }
#pragma unroll
        for (int u = 0; u < NSW; ++u) {
            sraw[u] = *reinterpret_cast<const uint32_t *>(ring + off + s_lane + 4 * u);
        }
    };
    auto read_x = [&](int s, int off, int q, int i) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            x[s][t] = *reinterpret_cast<const u32x4 *>(ring + off + x_lane[q][t] + i * 32 * 256);
        }
    };
    // pair e of 8 of sub-step q's decoded operands, into set p
    auto decode = [&](int p, int q, int e) {
        w[p][e >> 2][e & 3] = tile_decode_pair(raw[q][e >> 2], e & 3);
    };
    auto operand = [&](int p, int t) {
        return __builtin_bit_cast(f16x8, u32x4{w[p][t][0], w[p][t][1], w[p][t][2], w[p][t][3]});
    };

#pragma unroll
    for (int s = 0; s < NS; ++s) {
        issue(s, s * STAGE);
    }
    __builtin_amdgcn_s_waitcnt(tile_waitcnt((NS - 1) * PER_STAGE));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_stage(0);
#pragma unroll
    for (int i = 0; i < DIST; ++i) {
        read_x(i, 0, 0, i);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        decode(0, 0, e);
    }

    int cur = 0;
    // stages per iteration: the operand sets alternate statically
    constexpr int SPI = SUW == 1 ? 2 : 1;
    for (int st0 = 0; st0 < nst; st0 += SPI) {
#pragma unroll
        for (int v = 0; v < SPI * SUW; ++v) {
            const int q = v % SUW;
            const int st = st0 + v / SUW;
            if (SPI > 1 && st >= nst) {
                break;
            }
            const int p = v & 1;
            const int nq = (q + 1) % SUW;
            const float s_done = s_cur;  // scale of the finished block
            if (q % SPB == 0) {
                const uint32_t u = q / SPB;
                const uint32_t sh = ((s_par + c_idx[u]) & 1) * 16;
                const uint16_t hb = static_cast<uint16_t>(sraw[u] >> sh);
                s_cur = static_cast<float>(__builtin_bit_cast(_Float16, hb));
                asm volatile("" : "+v"(s_cur));  // converted once, not inside every multiply-add
                c_idx[u] += s_q;
                c_rem[u] += s_r;
                if (c_rem[u] >= static_cast<uint32_t>(a.bl)) {
                    c_rem[u] -= static_cast<uint32_t>(a.bl);
                    ++c_idx[u];
                }
            }
            // fragment by fragment: the finished block's multiply-adds, this sub-step's MFMAs, the
            // reads of the fragment DIST ahead, a share of the next weights' decode
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int f = v * MI + i;
                if (q + 1 == SUW && i == MI - DIST) {
                    // the stage is read: refill its buffer; the next stage has landed
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_s_waitcnt(tile_waitcnt((NS - 2) * PER_STAGE));
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    issue(st + NS, cur);
                    cur = cur == (NS - 1) * STAGE ? 0 : cur + STAGE;
                    read_stage(cur);
                }
                f32x16 c0 = part[i];
                if (q % SPB == 0) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        acc[i][r] = __builtin_fmaf(part[i][r], s_done, acc[i][r]);
                        c0[r] = 0.f;
                    }
                    // (this adds the block before the sub-step's own)
                    if (COMP > 0 && COMP <= SUW && q % (COMP > 0 ? COMP : 1) == 0) {
                        compensate(i);
                    } else if (COMP > SUW && q == 0 && st % (COMP > SUW ? COMP / SUW : 1) == 0) {
                        compensate(i);
                    }
                    // here and not later: sunk towards the end of the loop, as the compiler would,
                    // they keep several sub-steps' partial sums in registers
                    asm volatile("" : "+v"(acc[i]));
                }
                part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                    __builtin_bit_cast(f16x8, x[f & 1][0]), operand(p, 0), c0, 0, 0, 0);
                part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                    __builtin_bit_cast(f16x8, x[f & 1][1]), operand(p, 1), part[i], 0, 0, 0);
                read_x((f + DIST) & 1, cur, i + DIST < MI ? q : nq, (i + DIST) % MI);
                // a stage's last sub-step has the next nibbles only now: all in its last fragment
                constexpr int kEach = 8 / MI;
                const int e0 = q + 1 < SUW ? i * kEach : (i + 1 == MI ? 0 : 8);
                const int e1 = q + 1 < SUW ? (i + 1) * kEach : 8;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if (e >= e0 && e < e1) {
                        decode(p ^ 1, nq, e);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[i][r] = __builtin_fmaf(part[i][r], s_cur, acc[i][r]);
        }
    }
    // a compensated tile as one f32 per output, for KS == 1 (below otherwise)
    if constexpr (COMP > 0 && KS == 1) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][r] = static_cast<float>(static_cast<double>(hi[i][r]) +
                                               static_cast<double>(acc[i][r]));
            }
        }
    }

    // every load landed, every wave past its last LDS read: the ring is free
    __builtin_amdgcn_s_waitcnt(tile_waitcnt(0));
    if constexpr (KS > 1) {
        __syncthreads();
        // group g > 0 hands its partial tile over; group 0 adds them in group order (compensated
        // tiles: both parts, in f64)
        constexpr int PARTS = COMP > 0 ? 2 : 1;
        static_assert(BM * BN * 4 * (KS - 1) * PARTS <= NS * STAGE, "partial tiles fit the ring");
        f32x4 *slot = reinterpret_cast<f32x4 *>(ring) + static_cast<size_t>(wn) * (MI * PARTS * 256);
        constexpr size_t kGroup = static_cast<size_t>(WGN) * (MI * PARTS * 256);
        if (ks > 0) {
            f32x4 *mine = slot + static_cast<size_t>(ks - 1) * kGroup;
#pragma unroll
            for (int i = 0; i < MI; ++i) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    mine[(i * 4 + g) * 64 + lane] = f32x4{acc[i][4 * g], acc[i][4 * g + 1],
                                                          acc[i][4 * g + 2], acc[i][4 * g + 3]};
                    if constexpr (COMP > 0) {
                        mine[(MI * 4 + i * 4 + g) * 64 + lane] =
                            f32x4{hi[i][4 * g], hi[i][4 * g + 1], hi[i][4 * g + 2],
                                  hi[i][4 * g + 3]};
                    }
                }
            }
        }
        __syncthreads();
        if (ks > 0) {
            return;
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if constexpr (COMP > 0) {
                    double sum[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        sum[e] = static_cast<double>(hi[i][4 * g + e]) +
                                 static_cast<double>(acc[i][4 * g + e]);
                    }
#pragma unroll
                    for (int o = 0; o < KS - 1; ++o) {
                        const f32x4 lo = slot[o * kGroup + (i * 4 + g) * 64 + lane];
                        const f32x4 up = slot[o * kGroup + (MI * 4 + i * 4 + g) * 64 + lane];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            sum[e] += static_cast<double>(up[e]) + static_cast<double>(lo[e]);
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        acc[i][4 * g + e] = static_cast<float>(sum[e]);
                    }
                } else {
#pragma unroll
                    for (int o = 0; o < KS - 1; ++o) {
                        const f32x4 v = slot[o * kGroup + (i * 4 + g) * 64 + lane];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            acc[i][4 * g + e] += v[e];
                        }
                    }
                }
            }
        }
    }

    // Epilogue: lane (channel r32 of the wave) holds rows 8 (r / 4) + 4 h + r % 4 of every fragment;
    // a store covers 32 consecutive channels of two rows. Rows past M and channels past N are
    // dropped by the resources' range checks.
    constexpr uint32_t ES = OUT == OUT_F32 ? 4 : 2;
    const uint32_t rows = static_cast<uint32_t>(min(BM, a.M - m0));
    auto out_rsrc = [&](const void *p, long long ld) {
        const int8_t *base = static_cast<const int8_t *>(p) +
                             (static_cast<long long>(m0) * ld + n0) * ES;
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<int8_t *>(base), static_cast<short>(0),
            static_cast<int>(rows * static_cast<uint32_t>(ld) * ES), 0x00020000);
    };
    const uint32_t lane_col = gch < a.N ? static_cast<uint32_t>(wn * 32 + r32) * ES : kTileOob;
    if (a.C) {
        const __amdgpu_buffer_rsrc_t c_rsrc = out_rsrc(a.C, a.ldc);
        const uint32_t ldc = static_cast<uint32_t>(a.ldc) * ES;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = static_cast<uint32_t>(32 * i + 8 * (r >> 2) + (r & 3) + 4 * h);
                acc[i][r] += load_out_buf<OUT>(c_rsrc, row < rows ? row * ldc + lane_col : kTileOob,
                                               0);
            }
        }
    }
    const __amdgpu_buffer_rsrc_t d_rsrc = out_rsrc(a.D, a.ldd);
    const uint32_t ldd = static_cast<uint32_t>(a.ldd) * ES;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t row = static_cast<uint32_t>(32 * i + 8 * (r >> 2) + (r & 3) + 4 * h);
            const float sum = acc[i][r] + pre_bias;
            float v = fminf(fmaxf(sum, a.cmin), a.cmax);
            v = sum != sum && !a.nan_to_min ? sum : v;
            store_out_buf<OUT>(d_rsrc, row < rows ? row * ldd + lane_col : kTileOob, 0, v);
        }
    }
}

}  // namespace
}  // namespace tqt
