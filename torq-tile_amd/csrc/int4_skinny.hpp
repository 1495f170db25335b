// Few-row int8 contraction with int4 weights (W4A8 decode batches: up to 32 rows, k a multiple of 32).
//
// A workgroup of WV wave64s owns 16 output channels over all of k; wave w takes the 256-k blocks w,
// w + WV, ... A block - 16 weight rows of 128 bytes (whole cache lines) and the activation rows -
// lands in a ring of the wave's own in LDS by direct global -> LDS loads, is read into registers, and
// its slot refilled before the math. Lane (r, g) reads 16 bytes of weights, 32 k of channel r, and
// decodes them into the two operands of v_mfma_i32_16x16x64_i8 whose activations are the matching 16
// byte chunks. The waves meet once, at the end, where their exact int32 partial tiles are added.
//
// What bounds it: the weight stream, with one or two 2 KiB weight blocks in flight per wave (32 KiB a CU
// at one strip each), behind a fixed 2 to 3 us (launch and the first loads' latency); 8 x 28672 x 8192
// runs at 5.1 TB/s, 8 x 4096 x 11008 at 3.1. Before (k-split kernel, or 32 x 128 tiles where k is no
// multiple of 256) -> now, each layer's weights from HBM: 8 x 4096 x 11008 7.9 -> 7.6 us, 9 x 5120 x
// 13824 15.8 -> 14.6, 16 x 11008 x 4096 13.2 -> 8.8, 4 x 896 x 13824 7.0 -> 5.5, at k 13792 30.8 -> 5.9.
#pragma once

#include "int8_tile.hpp"

namespace tqt {
namespace {

constexpr int kIsK = 256;  // k per block

// XB: 1 KiB load blocks of activations per 256 k (four rows each); NS: blocks in flight per wave.
template <int WV, int XB, int NS, int OUT>
__global__ __launch_bounds__(WV * 64) void w4a8_skinny_kernel(TileArgs a)
{
    constexpr int MT = XB > 4 ? 2 : 1;  // 16-row MFMA tiles
    constexpr int PER = 2 + XB;
    constexpr int SLOT = PER * 1024;
    constexpr int RING = NS * SLOT;
    static_assert(MT * 1024 + 64 <= RING, "a wave's partial tile fits its ring");
    static_assert(MT * 256 <= WV * 64, "an output per thread");
    static_assert((NS - 1) * PER < 64, "vmcnt");
    __shared__ __attribute__((aligned(1024))) int8_t ring[WV * RING];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * 16;
    const int fr = lane & 15;  // activation row / channel of the MFMA operands
    const int fg = lane >> 4;  // 32-k group

    // epilogue operands of this thread's output (row tid / 16, channel tid % 16)
    const int orow = tid >> 4, gn = n0 + (tid & 15);
    const int cn = min(gn, a.N - 1), cm = min(orow, a.M - 1);
    const float p_sb = a.scale_b[cn];
    const float p_sa = a.scale_a[cm];
    const int32_t p_za = a.zp_a[cm];
    const float p_bias = a.bias ? load_out<OUT>(a.bias, cn) : -0.f;
    const float p_c = a.C ? load_out<OUT>(a.C, static_cast<long long>(cm) * a.ldc + cn) : -0.f;

    const i32x4 x_rsrc = raw_rsrc(a.A, kTileRecords);
    const i32x4 w_rsrc = raw_rsrc(a.B + static_cast<long long>(n0) * a.bstride, kTileRecords);
    // weights: load j holds rows 8 j .. 8 j + 7 (lane: row lane / 8, slot lane % 8, chunk slot ^
    // ((row >> 1) & 7)); activations: rows 4 j .. 4 j + 3 (row lane / 16, slot lane % 16, chunk slot
    // ^ (row & 15))
    uint32_t off[PER], kc[PER];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = 8 * j + (lane >> 3);
        const uint32_t chunk = static_cast<uint32_t>((lane & 7) ^ ((row >> 1) & 7));
        kc[j] = chunk * 32;
        off[j] = static_cast<uint32_t>(min(row, a.N - 1 - n0)) * static_cast<uint32_t>(a.bstride) +
                 chunk * 16;
    }
#pragma unroll
    for (int j = 0; j < XB; ++j) {
        const int row = 4 * j + (lane >> 4);
        const uint32_t chunk = static_cast<uint32_t>((lane & 15) ^ (row & 15));
        kc[2 + j] = chunk * 16;
        off[2 + j] = static_cast<uint32_t>(min(row, a.M - 1)) * static_cast<uint32_t>(a.lda) +
                     chunk * 16;
    }
    int8_t *mine = ring + wave * RING;
    const uint32_t K = static_cast<uint32_t>(a.K);
    auto issue = [&](int it, int slot) {
        const uint32_t k0 = static_cast<uint32_t>(it * WV + wave) * kIsK;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const uint32_t o = off[j] + (j < 2 ? k0 / 2 : k0);
            dma_lds16_buf(j < 2 ? w_rsrc : x_rsrc,
                          static_cast<int>(kc[j] + k0 < K ? o : kTileOob),
                          mine + slot * SLOT + j * 1024);
        }
    };

    const int nit = (a.K + WV * kIsK - 1) / (WV * kIsK);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        issue(s, s);
    }

    i32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        acc[i] = i32x4{0, 0, 0, 0};
    }
    int32_t rs = 0;  // this lane's share of sum_k (q - 8) of its channel
    for (int it0 = 0; it0 < nit; it0 += NS) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (it0 + s >= nit) {
                break;
            }
            __builtin_amdgcn_s_waitcnt(tile_waitcnt((NS - 1) * PER));
            asm volatile("" ::: "memory");
            const int8_t *blk = mine + s * SLOT;
            u32x4 w[2];
            i32x4 x[MT][4];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                w[u] = *reinterpret_cast<const u32x4 *>(blk + fr * 128 +
                                                        (((4 * u + fg) ^ ((fr >> 1) & 7)) << 4));
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    // rows past the loaded ones repeat the last (not stored)
                    const int row = XB < 4 ? min(fr, 4 * XB - 1) : 16 * i + fr;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        x[i][2 * u + h] = *reinterpret_cast<const i32x4 *>(
                            blk + 2048 + row * 256 + (((2 * (4 * u + fg) + h) ^ (row & 15)) << 4));
                    }
                }
            }
            // the block is in registers before its slot is refilled
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(tile_waitcnt(63));
            asm volatile("" ::: "memory");
            issue(it0 + s + NS, s);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const i32x4 q = tile_decode_w4(w[u][2 * h], w[u][2 * h + 1], rs);
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[i][2 * u + h], q, acc[i],
                                                                       0, 0, 0);
                    }
                }
            }
        }
    }

    // partial tiles (row, channel) of every wave, each in its own ring once its last loads have landed
    __builtin_amdgcn_s_waitcnt(tile_waitcnt(0));
    asm volatile("" ::: "memory");
    int32_t *part = reinterpret_cast<int32_t *>(mine);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            part[(16 * i + 4 * fg + r) * 16 + fr] = acc[i][r];
        }
    }
    int32_t t = rs + __shfl_xor(rs, 16);
    t += __shfl_xor(t, 32);
    if (lane < 16) {
        part[MT * 256 + lane] = t;
    }
    __syncthreads();
    if (orow >= min(a.M, 16 * MT) || gn >= a.N) {
        return;
    }
    // zero bytes past k decoded as q - 8 = -8
    int32_t sum = 0, rsum = 8 * (nit * WV * kIsK - a.K);
#pragma unroll
    for (int v = 0; v < WV; ++v) {
        const int32_t *pw = reinterpret_cast<const int32_t *>(ring + v * RING);
        sum += pw[tid];
        rsum += pw[MT * 256 + (tid & 15)];
    }
    // the operands hold 16 (q - 8)
    store_out<OUT>(a.D, static_cast<long long>(orow) * a.ldd + gn,
                   w4a8_value(sum >> 4, rsum, p_za, p_sa, p_sb, p_c, p_bias, a.cmin, a.cmax));
}

}  // namespace
}  // namespace tqt
