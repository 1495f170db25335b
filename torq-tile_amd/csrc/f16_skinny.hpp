// Few-row f16 contraction with block-quantized int4 weights (W4A16 decode and small prefill chunks:
// groups of up to 16 rows, every scale block width that is a multiple of 32).
//
// A workgroup of WV wave64s owns 16 output channels of one row group over all of k; wave w takes the 256-k blocks w,
// w + WV, ... A block - 16 weight rows of 128 bytes (whole cache lines), the activation rows and the
// scales of its eight 32-k sub-blocks - lands in a ring of the wave's own in LDS by direct global ->
// LDS loads, is read into registers, and its slot refilled before the math. The waves meet once, at
// the end.
//
// Per sub-block: one weight dword per lane (8 k of one channel), decoded to exact f16 q - 8, one
// v_mfma_f32_16x16x32_f16, and the four partial sums of the lane times the sub-block's scale into
// f32 accumulators - eight of them, one per sub-block of a block, so that a chain holds k / (256 WV)
// terms; they and the waves' sums are added in f64 and rounded once.
//
// What bounds it: the weight stream behind a fixed 4 us (launch and the first loads' latency): 1 x
// 28672 x 8192 (132 MB with the scales) runs at 4.2 TB/s, 32 us; at 1 x 14336 x 4096 the decode and the
// scaling issue for over half of all cycles beside it. The other kernels' fixed share is larger (they pad
// to 32 rows and meet all waves at each chunk of k), or they have too few workgroups. Before -> now:
// 1 x 4096 x 4096 12.0 -> 6.5 us, 1 x 4096 x 14336 31.6 -> 12.0, 1 x 4096 x 11008 in 128-wide blocks
// 37.3 -> 10.8, 8 x 4096 x 11008 41.7 -> 11.1, 16 x 4096 x 4096 12.3 -> 7.4.
#pragma once

#include "f16_tile.hpp"

namespace tqt {
namespace {

constexpr int kFsK = 256;  // k per block

struct F16SkinnyArgs
{
    F16TileArgs t;
    uint32_t bdiv;  // 32-k blocks per scale block
};

// XB: 1 KiB load blocks of activations per 256 k (two rows each); NS: blocks in flight per wave.
// The register bound of the four-wave, two-row form lets four workgroups share a CU instead of three
// (1 x 14336 x 4096, 3.5 workgroups a CU: 13.5 -> 12.1 us).
template <int WV, int XB, int NS, int OUT>
__global__ __launch_bounds__(WV * 64, WV == 4 && XB == 1 ? 4 : 2) void w4a16_skinny_kernel(F16SkinnyArgs fa)
{
    const F16TileArgs &a = fa.t;
    constexpr int SW = 2048, SX = XB * 1024, SS = 512;
    constexpr int SLOT = SW + SX + SS;
    constexpr int RING = NS * SLOT;
    constexpr int PER = 2 + XB + 2;
    static_assert(RING >= 16 * 16 * 8, "a wave's f64 partial tile fits its ring");
    static_assert((NS - 1) * PER < 64, "vmcnt");
    __shared__ __attribute__((aligned(1024))) int8_t ring[WV * RING];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * 16;
    const int m0 = blockIdx.y * 16;
    const int rows = min(16, a.M - m0);
    const int fr = lane & 15;  // activation row / channel of the MFMA operands
    const int fg = lane >> 4;  // 8-k group

    // epilogue operands of this thread's output (the first 256: row tid / 16, channel tid % 16)
    const int orow = (tid >> 4) & 15, gm = m0 + orow, gn = n0 + (tid & 15);
    const int cn = min(gn, a.N - 1), cm = min(gm, a.M - 1);
    const uint32_t p_bias = a.bias ? load_out_bits<OUT>(a.bias, cn) : 0u;
    const uint32_t p_c = a.C ? load_out_bits<OUT>(a.C, static_cast<long long>(cm) * a.ldc + cn) : 0u;

    const i32x4 x_rsrc = raw_rsrc(a.A + static_cast<long long>(m0) * a.lda, kTileRecords);
    const i32x4 w_rsrc = raw_rsrc(a.B + static_cast<long long>(n0) * a.bstride, kTileRecords);
    const uintptr_t s_addr =
        reinterpret_cast<uintptr_t>(a.scale_b + static_cast<long long>(n0) * a.ldsb);
    const uint32_t s_mis = static_cast<uint32_t>(s_addr & 3);
    const i32x4 s_rsrc = raw_rsrc(reinterpret_cast<const void *>(s_addr - s_mis), kTileRecords);
    // weights: load j holds rows 8 j .. 8 j + 7 (lane: row lane / 8, slot lane % 8, chunk slot ^
    // ((row >> 1) & 7)); activations: rows 2 j, 2 j + 1 (row lane / 32, slot lane % 32, chunk slot ^
    // (row & 15)); scales: dword (channel 8 j + lane / 8, sub-block lane % 8)
    uint32_t w_off[2], x_off[XB], s_off[2], x_k[XB];
    const uint32_t w_k = static_cast<uint32_t>(((lane & 7) ^ ((lane >> 4) & 3)) * 32);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = 8 * j + (lane >> 3);
        const uint32_t chunk = static_cast<uint32_t>((lane & 7) ^ ((row >> 1) & 7));
        w_off[j] = static_cast<uint32_t>(min(row, a.N - 1 - n0)) *
                       static_cast<uint32_t>(a.bstride) + chunk * 16;
        s_off[j] = static_cast<uint32_t>(min(row, a.N - 1 - n0)) *
                       static_cast<uint32_t>(2 * a.ldsb) + s_mis;
    }
#pragma unroll
    for (int j = 0; j < XB; ++j) {
        const int row = 2 * j + (lane >> 5);
        const uint32_t chunk = static_cast<uint32_t>((lane & 31) ^ (row & 15));
        x_k[j] = chunk * 8;
        x_off[j] = static_cast<uint32_t>(min(row, rows - 1)) * static_cast<uint32_t>(2 * a.lda) +
                   chunk * 16;
    }
    // scale index of 32-k block kb (the launcher keeps k and the block width where it is exact; past
    // the last block it may only read high, and is refused by its count all the same)
    const uint32_t inv = scale_block_inverse(fa.bdiv);
    auto scale_idx = [&](uint32_t kb) { return scale_block_of(kb, fa.bdiv, inv); };
    int8_t *mine = ring + wave * RING;
    const uint32_t K = static_cast<uint32_t>(a.K);
    auto issue = [&](int it, int slot) {
        const uint32_t k0 = static_cast<uint32_t>(it * WV + wave) * kFsK;
        int8_t *base = mine + slot * SLOT;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            // chunk's first k: the swizzle of rows 8 j + lane / 8 takes their bits 1 .. 3
            const uint32_t kc = j == 0 ? w_k : (w_k ^ 128u);
            dma_lds16_buf(w_rsrc, static_cast<int>(kc + k0 < K ? w_off[j] + k0 / 2 : kTileOob),
                          base + j * 1024);
        }
#pragma unroll
        for (int j = 0; j < XB; ++j) {
            dma_lds16_buf(x_rsrc, static_cast<int>(x_k[j] + k0 < K ? x_off[j] + 2 * k0 : kTileOob),
                          base + SW + j * 1024);
        }
        const uint32_t idx = scale_idx(k0 / 32 + static_cast<uint32_t>(lane & 7));
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            dma_lds4_buf(s_rsrc,
                         static_cast<int>(idx < static_cast<uint32_t>(a.nblocks)
                                              ? ((s_off[j] + 2 * idx) & ~3u) : kTileOob),
                         base + SW + SX + j * 256);
        }
    };

    const int nit = (a.K + WV * kFsK - 1) / (WV * kFsK);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        issue(s, s);
    }

    f32x4 acc[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // which half of its dword a scale is: the parity of its f16 index from an aligned address
    const uint32_t s_sh = 16 * (((s_mis >> 1) + static_cast<uint32_t>(min(fr, a.N - 1 - n0)) *
                                                    static_cast<uint32_t>(a.ldsb & 1)) & 1);
    const int xrow = min(fr, 2 * XB - 1);  // rows past the loaded ones repeat the last (not stored)
    for (int it0 = 0; it0 < nit; it0 += NS) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (it0 + s >= nit) {
                break;
            }
            __builtin_amdgcn_s_waitcnt(tile_waitcnt((NS - 1) * PER));
            asm volatile("" ::: "memory");
            const int8_t *blk = mine + s * SLOT;
            uint32_t w[8];
            u32x4 x[8], sc[2];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                w[t] = *reinterpret_cast<const uint32_t *>(blk + fr * 128 +
                                                           ((t ^ ((fr >> 1) & 7)) << 4) + 4 * fg);
                x[t] = *reinterpret_cast<const u32x4 *>(blk + SW + xrow * 512 +
                                                        (((4 * t + fg) ^ (xrow & 15)) << 4));
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                sc[j] = *reinterpret_cast<const u32x4 *>(blk + SW + SX + fr * 32 + 16 * j);
            }
            // the block is in registers before its slot is refilled
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(tile_waitcnt(63));
            asm volatile("" ::: "memory");
            issue(it0 + s + NS, s);
            const uint32_t kb = static_cast<uint32_t>((it0 + s) * WV + wave) * (kFsK / 32);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                u32x4 q;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    q[b] = tile_decode_pair(w[t], b);
                }
                const uint32_t sh = s_sh ^ (16 * (scale_idx(kb + t) & 1));
                const uint16_t hb = static_cast<uint16_t>(sc[t >> 2][t & 3] >> sh);
                const float sf = static_cast<float>(__builtin_bit_cast(_Float16, hb));
                const f32x4 part = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    __builtin_bit_cast(f16x8, x[t]), __builtin_bit_cast(f16x8, q),
                    f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    acc[t][r] = __builtin_fmaf(part[r], sf, acc[t][r]);
                }
            }
        }
    }

    // the waves' f64 sums (row, channel), each in its own ring once its last loads have landed
    __builtin_amdgcn_s_waitcnt(tile_waitcnt(0));
    asm volatile("" ::: "memory");
    double *part = reinterpret_cast<double *>(mine);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        double v = 0.0;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            v += static_cast<double>(acc[t][r]);
        }
        part[(4 * fg + r) * 16 + fr] = v;
    }
    __syncthreads();
    if (tid >= 256 || gm >= a.M || gn >= a.N) {
        return;
    }
    double sum = 0.0;
#pragma unroll
    for (int v = 0; v < WV; ++v) {
        sum += reinterpret_cast<const double *>(ring + v * RING)[tid];
    }
    float v = static_cast<float>(sum);
    if (a.C) {
        v += out_from_bits<OUT>(p_c);
    }
    if (a.bias) {
        v += out_from_bits<OUT>(p_bias);
    }
    const float cl = fminf(fmaxf(v, a.cmin), a.cmax);
    store_out<OUT>(a.D, static_cast<long long>(gm) * a.ldd + gn,
                   v != v && !a.nan_to_min ? v : cl);
}

}  // namespace
}  // namespace tqt
