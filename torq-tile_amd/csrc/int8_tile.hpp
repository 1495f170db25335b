// Large-tile int8 MFMA contraction with int4 weights (W4A8 with more than a few rows).
//
// A workgroup of 8 wave64s owns a BM x BN tile of D (activation rows x output channels) and walks
// k in stages of 128 through a ring of NS LDS stages filled by direct global -> LDS loads. The
// waves form a WGM x WGN grid over the tile, each with MI x NI fragments of
// v_mfma_i32_32x32x32_i8 (32 MI rows x 32 NI channels), times KS groups that split every stage's
// four k-steps between them; the KS int32 partial tiles are added in LDS at the end (exact), each
// wave finishing its share of the fragments.
//
// What bounds it. A k-step of a wave reads (MI + NI) fragments from LDS for MI * NI MFMAs of 32
// cycles. The int8 matrix cores of a CU retire 8192 operations a clock against 128 bytes a clock of
// LDS reads, so the fragments a wave reads per MFMA decide the rate: 64 x 64 per wave reads 1 KiB
// per MFMA (at most the LDS rate), 128 x 64 0.75 KiB. Weights stay packed in LDS (half a byte each)
// and are decoded in registers as they are read, which halves their share of that traffic.
//
// Weight decode (natural k order, so the activations need no permutation): w ^ 0x88888888 makes
// each nibble the two's complement of q - 8; masked into the high half of a byte it is the signed
// byte 16 (q - 8), and two byte permutes interleave the even and odd k. The MFMA then accumulates
// 16 sum a (q - 8) exactly (|.| < 2^31 for k <= 65536) and one shift recovers the sum. The
// zero-point correction's sum (q - 8) is one v_dot8_i32_i4 per weight dword on the same registers.
//
// Operand roles: the weights are the 32-row operand and the activations the 32-column operand, so
// a lane's accumulators are one activation row by runs of four consecutive channels, which the
// epilogue stores as one vector.
//
// LDS layout (conflict-free ds_read_b128 / b64): an activation row is 128 bytes, its 16-byte chunk
// c at c ^ ((row >> 1) & 7); a weight row is 64 bytes, its chunk c at c ^ ((row >> 2) & 3). The k
// values a lane feeds to k-step t are chunk 4 (t >> 1) + 2 h + (t & 1) of 16 (h = lane / 32), the
// same for both operands, so that a lane's weight nibbles of two k-steps are contiguous.
//
// Pipeline: the barrier of a stage sits before its last k-step, whose fragments are in registers
// by then: every wave has then read the whole stage, its buffer is refilled NS stages ahead, and
// the first fragments of the next stage are read behind that k-step's MFMAs. Loads past k, and the
// stages past the last, are range-checked to zeros by the buffer resource (no memory traffic), so
// the loop has no tail and every wait is a constant vmcnt.
//
// Measured (f32 out): 1000 x 11008 x 4096 with its quantization 66 us (one pass over the weights
// per 15 rows before: 373 us), 200 x 4096 x 4096 12.8 us (27.1), 2000 x 4096 x 1024 f16 19.7 us
// (107). At 4096^3 one 256 x 256 tile a CU takes 82 us (1.67 POP/s): the MFMAs alone 44 us (the
// clock falls under that load), the loads 12, the decode 10, the operand reads 5, and the launch,
// first loads and the 64 MB of results 14.
#pragma once

#include <type_traits>

#include "route.hpp"
#include "tqt_hip_common.hpp"

namespace tqt {
namespace {

// s_waitcnt immediate (gfx9: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] << 14):
// vmcnt <= vm and lgkmcnt == 0.
__host__ __device__ constexpr int tile_waitcnt(int vm)
{
    return (vm & 15) | (7 << 4) | ((vm >> 4) << 14);
}

constexpr int kTileK = 128;                  // k per stage
constexpr int kTileRingBytes = 150 * 1024;   // LDS for the ring, at most
constexpr uint32_t kTileOob = 0x80000000u;   // a buffer offset past every resource below
constexpr int kTileRecords = 0x7fffffff;

struct TileArgs
{
    int M, N, K;
    const int8_t *A;
    long long lda;
    const uint8_t *B;
    long long bstride;  // bytes between weight rows
    const void *C;
    long long ldc;
    void *D;
    long long ldd;
    const void *bias;
    float cmin, cmax;
    const float *scale_a;
    const int32_t *zp_a;
    const float *scale_b;
    int tiles_m, tiles_n, per_xcd;
    int vec_d;  // four channels of D may be stored as one vector (rows and base aligned)
};

// Tile order: block b runs on XCD b % 8 and each XCD takes a contiguous range; inside it tiles
// advance M first within groups of 8 tile rows, so the workgroups that run together on an XCD
// cover a near-square block of D and share its rows of A and B in that XCD's L2.
__device__ __forceinline__ bool tile_coords(int tiles_m, int tiles_n, int per_xcd, int &tm, int &tn)
{
    const int t = static_cast<int>((blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3));
    if (t >= tiles_m * tiles_n) {
        return false;
    }
    constexpr int kGroup = 8;
    const int per_group = kGroup * tiles_n;
    const int g = t / per_group;
    const int first = g * kGroup;
    const int rows = min(kGroup, tiles_m - first);
    const int r = t - g * per_group;
    tn = r / rows;
    tm = first + (r - tn * rows);
    return true;
}

// One int8 operand of 16 natural-order k from 8 bytes of nibbles, and the running sum (q - 8).
__device__ __forceinline__ i32x4 tile_decode_w4(uint32_t x0, uint32_t x1, int32_t &rs)
{
    i32x4 o;
    const uint32_t x[2] = {x0 ^ 0x88888888u, x1 ^ 0x88888888u};
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        rs = __builtin_amdgcn_sdot8(static_cast<int>(x[d]), 0x11111111, rs, false);
        const uint32_t hi = x[d] & 0xf0f0f0f0u;
        const uint32_t lo = (x[d] << 4) & 0xf0f0f0f0u;
        o[2 * d] = static_cast<int32_t>(__builtin_amdgcn_perm(hi, lo, 0x05010400u));
        o[2 * d + 1] = static_cast<int32_t>(__builtin_amdgcn_perm(hi, lo, 0x07030602u));
    }
    return o;
}

__host__ __device__ constexpr int tile_stages(int stage_bytes, int cap)
{
    return kTileRingBytes / stage_bytes < cap ? kTileRingBytes / stage_bytes : cap;
}

template <int MI, int NI, int WGM, int WGN, int KS, int NSMAX, int OUT>
__global__ __launch_bounds__(64 * WGM * WGN * KS, 2) void w4a8_tile_kernel(TileArgs a)
{
    static_assert(KS == 1 || KS == 2 || KS == 4, "k groups");
    constexpr int WAVES = WGM * WGN * KS;
    constexpr int THREADS = 64 * WAVES;
    constexpr int BM = 32 * MI * WGM;
    constexpr int BN = 32 * NI * WGN;
    constexpr int SX = BM * kTileK;      // activation bytes of a stage
    constexpr int SW = BN * kTileK / 2;  // weight bytes of a stage
    constexpr int STAGE = SX + SW;
    constexpr int NS = tile_stages(STAGE, NSMAX);
    static_assert(NS >= 2, "ring");
    // 1 KiB load blocks per wave (tiles with fewer blocks than waves: several waves load the same one)
    constexpr int XPW = SX / 1024 >= WAVES ? SX / 1024 / WAVES : 1;
    constexpr int WPW = SW / 1024 >= WAVES ? SW / 1024 / WAVES : 1;
    constexpr int PER_STAGE = XPW + WPW;
    constexpr int KPW = 4 / KS;  // k-steps per wave and stage
    static_assert((NS - 1) * PER_STAGE < 64, "vmcnt");
    static_assert(BM * BN * 4 * (KS - 1) <= NS * STAGE, "partial tiles fit the ring");

    __shared__ __attribute__((aligned(1024))) int8_t ring[NS * STAGE];
    __shared__ __attribute__((aligned(16))) float s_sb[BN];
    __shared__ __attribute__((aligned(16))) float s_bias[BN];
    __shared__ __attribute__((aligned(16))) int32_t s_rs[BN];
    __shared__ float s_sa[BM];
    __shared__ int32_t s_za[BM];

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
    const int wn = (wave / KS) % WGN;
    const int wm = wave / (KS * WGN);
    const int r32 = lane & 31;
    const int h = lane >> 5;

    // Epilogue operands, requested ahead of the stream (their wait is the first stage's): the
    // channels' scales and biases (threads < BN), the rows' scales and zero points (threads < BM).
    static_assert(BM <= THREADS && BN <= THREADS, "one row and channel per thread");
    const int pre_n = min(n0 + tid, a.N - 1), pre_m = min(m0 + tid, a.M - 1);
    const float pre_sb = a.scale_b[pre_n];
    // an absent bias adds -0, which leaves every value as it is
    const float pre_bias = a.bias ? load_out<OUT>(a.bias, pre_n) : -0.f;
    const float pre_sa = a.scale_a[pre_m];
    const int32_t pre_za = a.zp_a[pre_m];

    // Load roles: activation block b holds rows 8 b .. 8 b + 7 (lane: row lane / 8, slot lane % 8),
    // weight block b rows 16 b .. 16 b + 15 (row lane / 4, slot lane % 4). Offsets are 32-bit from
    // the tile's first row (the launcher bounds the strides).
    const i32x4 x_rsrc = raw_rsrc(a.A + static_cast<long long>(m0) * a.lda, kTileRecords);
    const i32x4 w_rsrc = raw_rsrc(a.B + static_cast<long long>(n0) * a.bstride, kTileRecords);
    uint32_t x_off[XPW], x_k[XPW];
    int x_lds[XPW];
#pragma unroll
    for (int j = 0; j < XPW; ++j) {
        const int blk = (wave * XPW + j) % (SX / 1024);
        const int row = 8 * blk + (lane >> 3);
        x_k[j] = static_cast<uint32_t>(((lane & 7) ^ ((row >> 1) & 7)) * 16);
        x_off[j] = static_cast<uint32_t>(min(row, a.M - 1 - m0)) * static_cast<uint32_t>(a.lda) +
                   x_k[j];
        x_lds[j] = blk * 1024;
    }
    uint32_t w_off[WPW], w_k[WPW];
    int w_lds[WPW];
#pragma unroll
    for (int j = 0; j < WPW; ++j) {
        const int blk = (wave * WPW + j) % (SW / 1024);
        const int row = 16 * blk + (lane >> 2);
        const int chunk = (lane & 3) ^ ((row >> 2) & 3);
        w_k[j] = static_cast<uint32_t>(chunk * 32);
        w_off[j] = static_cast<uint32_t>(min(row, a.N - 1 - n0)) *
                       static_cast<uint32_t>(a.bstride) + chunk * 16;
        w_lds[j] = SX + blk * 1024;
    }
    const uint32_t K = static_cast<uint32_t>(a.K);
    auto issue = [&](int st, int off) {
        const uint32_t k0 = static_cast<uint32_t>(st) * kTileK;
#pragma unroll
        for (int j = 0; j < XPW; ++j) {
            dma_lds16_buf(x_rsrc, static_cast<int>(x_k[j] + k0 < K ? x_off[j] + k0 : kTileOob),
                          ring + off + x_lds[j]);
        }
#pragma unroll
        for (int j = 0; j < WPW; ++j) {
            dma_lds16_buf(w_rsrc, static_cast<int>(w_k[j] + k0 < K ? w_off[j] + k0 / 2 : kTileOob),
                          ring + off + w_lds[j]);
        }
    };

    i32x16 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = 0;
            }
        }
    }
    int32_t rs[NI] = {};

    // LDS offsets of this lane's operands of its k-step q (fragment i / j adds 32 rows)
    int x_lane[KPW], w_lane[KPW];
#pragma unroll
    for (int q = 0; q < KPW; ++q) {
        const int t = ks * KPW + q;
        const int c = 4 * (t >> 1) + 2 * h + (t & 1);
        x_lane[q] = (wm * MI * 32 + r32) * kTileK + ((c ^ ((r32 >> 1) & 7)) << 4);
        w_lane[q] = SX + (wn * NI * 32 + r32) * (kTileK / 2) +
                    (((c >> 1) ^ ((r32 >> 2) & 3)) << 4) + 8 * (c & 1);
    }

    // Operand registers: the fragments of the current and the next k-step, and the raw weight
    // nibbles, which are read for two k-steps at once (one when a wave has one per stage) and
    // decoded one k-step ahead, between the MFMAs of the current one.
    constexpr int RD = KPW == 1 ? 2 : 4;  // dwords of a raw read
    typedef uint32_t RawT __attribute__((ext_vector_type(RD)));
    i32x4 fx[2][MI], fw[2][NI];
    RawT raw[2][NI];
    auto read_x = [&](int p, int off, int q) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            fx[p][i] = *reinterpret_cast<const i32x4 *>(ring + off + x_lane[q] + i * 32 * kTileK);
        }
    };
    auto read_w = [&](int p, int off, int q) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            raw[p][j] = *reinterpret_cast<const RawT *>(ring + off + w_lane[q] +
                                                        j * 32 * (kTileK / 2));
        }
    };
    auto decode = [&](int p, int rp, int d) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            fw[p][j] = tile_decode_w4(raw[rp][j][2 * d], raw[rp][j][2 * d + 1], rs[j]);
        }
    };
    auto mfma = [&](int p) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fw[p][j], fx[p][i], acc[i][j], 0,
                                                                  0, 0);
            }
        }
    };
    // Instruction order of a k-step: its LDS reads, then each MFMA with a share of the decode
    // behind it (a decode after the MFMAs leaves the matrix core idle: the two waves of a SIMD run
    // in step). `late`: the nibbles arrive with this k-step's reads, so the decode starts halfway.
    auto order = [&](auto late) {
        constexpr int kM = MI * NI;
        constexpr int kLead = decltype(late)::value ? kM / 2 : 0;
        constexpr int kVal = (NI * 14 + (kM - kLead) - 1) / (kM - kLead);
        __builtin_amdgcn_sched_group_barrier(0x100, MI + NI, 0);
        if constexpr (kLead > 0) {
            __builtin_amdgcn_sched_group_barrier(0x008, kLead, 0);
        }
#pragma unroll
        for (int m = 0; m < kM - kLead; ++m) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, kVal, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Stage st is read by every wave after this: refill its buffer, stage st + 1 has landed.
    auto sync = [&](int st, int off) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(tile_waitcnt((NS - 2) * PER_STAGE));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(st + NS, off);
    };

    const int nst = (a.K + kTileK - 1) / kTileK;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        issue(s, s * STAGE);
    }
    __builtin_amdgcn_s_waitcnt(tile_waitcnt((NS - 1) * PER_STAGE));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_w(0, 0, 0);
    read_x(0, 0, 0);
    decode(0, 0, 0);

    int cur = 0;
    // two stages per iteration when a wave has one k-step per stage, so that the register sets
    // alternate statically
    constexpr int SPI = KPW == 1 ? 2 : 1;
    for (int st0 = 0; st0 < nst; st0 += SPI) {
#pragma unroll
        for (int u = 0; u < SPI; ++u) {
            const int st = st0 + u;
            if (SPI == 1 || st < nst) {
#pragma unroll
                for (int q = 0; q < KPW; ++q) {
                    const int p = (u * KPW + q) & 1;
                    if (q + 1 < KPW) {
                        // raw set q / 2 holds k-steps 2 (q / 2) and the one after
                        if (q % 2 == 0 && q + 2 < KPW) {
                            read_w((q / 2 + 1) & 1, cur, q + 2);
                        }
                        read_x(p ^ 1, cur, q + 1);
                        mfma(p);
                        decode(p ^ 1, ((q + 1) / 2) & 1, (q + 1) & 1);
                        order(std::false_type{});
                    } else {
                        sync(st, cur);
                        cur = cur == (NS - 1) * STAGE ? 0 : cur + STAGE;
                        read_w(0, cur, 0);
                        read_x(p ^ 1, cur, 0);
                        mfma(p);
                        decode(p ^ 1, 0, 0);
                        order(std::true_type{});
                    }
                }
            }
        }
    }

    // every load landed, every wave past its last LDS read: the ring is free
    __builtin_amdgcn_s_waitcnt(tile_waitcnt(0));
    if (tid < BN) {
        s_sb[tid] = pre_sb;
        s_bias[tid] = pre_bias;
        // zero bytes past k decode as q - 8 = -8
        s_rs[tid] = 8 * (nst * kTileK - a.K);
    }
    if (tid < BM) {
        s_sa[tid] = pre_sa;
        s_za[tid] = pre_za;
    }
    __syncthreads();
    if (wm == 0) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            // less the 16 zero nibbles of the stage past the last that the pipeline decoded
            atomicAdd(&s_rs[(wn * NI + j) * 32 + r32], rs[j] + 8 * 16);
        }
    }
    if constexpr (KS > 1) {
        // fragments of the waves that do not finish them: [group][fragment][distance of the
        // wave's k group from the finishing one - 1][register / 4][lane] of 16 bytes
        i32x4 *part = reinterpret_cast<i32x4 *>(ring) +
                      static_cast<size_t>(wm * WGN + wn) * (MI * NI * (KS - 1) * 256);
#pragma unroll
        for (int f = 0; f < MI * NI; ++f) {
            if (f % KS != ks) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    part[(f * (KS - 1) + (ks - f % KS - 1 + KS) % KS) * 256 + g * 64 + lane] =
                        i32x4{acc[f / NI][f % NI][4 * g], acc[f / NI][f % NI][4 * g + 1],
                              acc[f / NI][f % NI][4 * g + 2], acc[f / NI][f % NI][4 * g + 3]};
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int f = 0; f < MI * NI; ++f) {
            if (f % KS == ks) {
#pragma unroll
                for (int o = 1; o < KS; ++o) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const i32x4 v = part[(f * (KS - 1) + o - 1) * 256 + g * 64 + lane];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            acc[f / NI][f % NI][4 * g + e] = static_cast<int32_t>(
                                static_cast<uint32_t>(acc[f / NI][f % NI][4 * g + e]) +
                                static_cast<uint32_t>(v[e]));
                        }
                    }
                }
            }
        }
    } else {
        __syncthreads();
    }

    // Epilogue. Lane (r32, h) holds row r32 of a fragment's activation rows and its channels
    // 8 g + 4 h + e: stored as they lie, one store instruction would touch 32 rows of D. The sums
    // are turned through the wave's own LDS buffer instead, up to MI fragments at a time, and read back
    // four channels per lane and eight rows per instruction: a lane then keeps its channels'
    // constants for the whole pass and a store writes whole 32-channel rows. The read side is a
    // rolled loop: unrolled over all fragments the epilogue is 30 KB of code that every CU fetches
    // once per launch.
    constexpr int PITCH = 32 * 4 + 16;  // conflict-free for the writes of four channels
    constexpr int TI = WAVES * MI * 32 * PITCH <= NS * STAGE ? MI : (MI + 1) / 2;
    static_assert(MI % TI == 0 && WAVES * TI * 32 * PITCH <= NS * STAGE, "the buffers fit the ring");
    __syncthreads();  // the partial tiles are read
    int8_t *turn = ring + wave * (TI * 32 * PITCH);
#pragma unroll
    for (int ji = 0; ji < NI * (MI / TI); ++ji) {
        const int j = ji % NI, i0 = ji / NI * TI;
        asm volatile("" ::: "memory");
#pragma unroll
        for (int t = 0; t < TI; ++t) {
            const int i = i0 + t;
            if (KS == 1 || (i * NI + j) % KS == ks) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    *reinterpret_cast<i32x4 *>(turn + (t * 32 + r32) * PITCH + (8 * g + 4 * h) * 4) =
                        i32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2],
                              acc[i][j][4 * g + 3]};
                }
            }
        }
        asm volatile("" ::: "memory");
        const int lc = (wn * NI + j) * 32 + (lane & 7) * 4;
        const int gn = n0 + lc;
        const f32x4 sb = *reinterpret_cast<const f32x4 *>(&s_sb[lc]);
        const f32x4 fb = *reinterpret_cast<const f32x4 *>(&s_bias[lc]);
        const i32x4 rv = *reinterpret_cast<const i32x4 *>(&s_rs[lc]);
        if (gn >= a.N) {
            continue;
        }
#pragma unroll 1
        for (int r = 0; r < TI * 32; r += 8) {
            if (KS > 1 && ((i0 + (r >> 5)) * NI + j) % KS != ks) {
                continue;
            }
            const int row = r + (lane >> 3);
            const int lr = (wm * MI + i0) * 32 + row;
            const int gm = m0 + lr;
            const i32x4 s = *reinterpret_cast<const i32x4 *>(turn + row * PITCH + (lane & 7) * 16);
            const float sa = s_sa[lr];
            const int32_t za = s_za[lr];
            if (gm >= a.M) {
                continue;
            }
            // an absent C adds -0, which leaves every value as it is
            f32x4 c = f32x4{-0.f, -0.f, -0.f, -0.f};
            if (a.C) {
                const long long e0 = static_cast<long long>(gm) * a.ldc + gn;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    c[e] = gn + e < a.N ? load_out<OUT>(a.C, e0 + e) : 0.f;
                }
            }
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = w4a8_value(s[e] >> 4, rv[e], za, sa, sb[e], c[e], fb[e], a.cmin, a.cmax);
            }
            const long long d0 = static_cast<long long>(gm) * a.ldd + gn;
            if (a.vec_d && gn + 4 <= a.N) {
                store_out4<OUT>(a.D, d0, v);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (gn + e < a.N) {
                        store_out<OUT>(a.D, d0 + e, v[e]);
                    }
                }
            }
        }
    }
}

}  // namespace
}  // namespace tqt
