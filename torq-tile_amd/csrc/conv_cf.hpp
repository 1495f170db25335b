// Channel-first implicit convolution (igemmcf, plain weights): KH x KW taps in one depth plane, any
// stride, dilation and padding in h and w, group channels a multiple of 16. Included by
// int8_mfma.hip, whose argument struct and epilogue steps it uses.
//
// The NCDHW input has consecutive pixels of one channel next to each other, and the weights (ic, kh,
// kw) per output channel: gathered as they lie, every byte of the contraction is a load and address
// arithmetic of its own (int8_mfma_kernel's channel-first mode: 69 us for 8 x 28 x 28, 64 -> 128
// channels). This kernel turns both operands once per workgroup into channel-last LDS tiles, where
// a tap of a pixel is 16 contiguous channels, and contracts tap by tap:
//   * a workgroup of 4 wave64s owns 64 output pixels x 64 output channels; output pixels are
//     numbered row by row through the depth (batch) axis, so the input rows they need are one
//     contiguous run of every channel's plane (the halo), loaded once for all taps;
//   * a thread turns 4 pixels x 16 channels: 16 dword loads (consecutive lanes read consecutive
//     dwords of a plane), four 4 x 4 byte transposes (8 byte permutes each), 4 ds_write_b128;
//   * a thread turns the taps of one (output channel, 16 input channels): the 16 T bytes are T
//     16-byte loads; output dword q of tap t collects bytes t + T (4 q .. 4 q + 3) with three
//     permutes, all compile-time;
//   * v_mfma_i32_32x32x32_i8 per wave (32 pixels x 32 channels) and 32 channels of a tap; a padding
//     tap reads a zero line. Channels go in blocks of 64; a block's missing 16-channel chunks are
//     zero weights.
// A lane's accumulators are one output channel by runs of 4 pixels: its multiplier, shift and bias
// are lane constants, and the requantized tile is stored through LDS in 16-byte runs of pixels.
// What bounds it: at these sizes the chain of loads, turns and barriers of a workgroup, not a rate
// (2 workgroups share a CU to overlap it). Measured, with the double-buffered kernel's channel-first
// mode before: 8 x 28 x 28, 64 -> 128, 3 x 3 6.6 us (69); 8 x 56 x 56, 128 -> 128, 3 x 3 20 (146); 4 x
// 15 x 15, 512 -> 32, 3 x 3 25 (409: a serial gather of k 4608); 8 x 84 x 84, 64 -> 256, 1 x 1 stride
// 2 9.1.
#pragma once

namespace tqt {
namespace {

constexpr int kCfPix = 64;
constexpr int kCfCh = 64;
constexpr int kCfIc = 64;  // input channels per block

struct CfPlan
{
    int tiles_c;
    int tiles;
    int per_xcd;
    int px_rows;  // halo rows at most
};

template <int T, int PX>
__global__ __launch_bounds__(256) void conv_cf_kernel(Int8Args a, CfPlan hp)
{
    __shared__ __attribute__((aligned(128))) int8_t s_w[T * kCfCh * kCfIc];
    __shared__ __attribute__((aligned(128))) int8_t s_x[(PX + 4) * kCfIc];  // row PX: zeros
    const int t_id = static_cast<int>((blockIdx.x & 7) * hp.per_xcd + (blockIdx.x >> 3));
    if (t_id >= hp.tiles) {
        return;
    }
    const ConvGeom &g = a.cv;
    const int oc0 = (t_id % hp.tiles_c) * kCfCh;
    const int n0 = (t_id / hp.tiles_c) * kCfPix;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wp = wave >> 1;  // 32-pixel half
    const int wc = wave & 1;   // 32-channel half
    const int r32 = lane & 31;
    const int h = lane >> 5;

    // this lane's output channel (MFMA column): requantization constants
    const int oc = oc0 + wc * 32 + r32;
    const int coc = min(oc, a.M - 1);
    const float p_sb = a.scale_b[a.quant_channel_b == 1 ? 0 : coc];
    const int32_t p_bias = a.bias ? a.bias[coc] : 0;

    // the tile's halo: stacked input rows [lo, hi) (row id * IH + ih)
    auto coords = [&](uint32_t p, int &od, int &oh, int &ow) {
        const uint32_t q1 = p / static_cast<uint32_t>(g.OW);
        ow = static_cast<int>(p - q1 * static_cast<uint32_t>(g.OW));
        const uint32_t q2 = q1 / static_cast<uint32_t>(g.OH);
        oh = static_cast<int>(q1 - q2 * static_cast<uint32_t>(g.OH));
        od = static_cast<int>(q2);
    };
    const uint32_t p0 = static_cast<uint32_t>(a.p0);
    int od, oh, ow;
    coords(p0 + static_cast<uint32_t>(n0), od, oh, ow);
    const int lo = od * g.IH + cf_clamp_row(oh * g.SH - g.PH, g.IH);
    coords(p0 + static_cast<uint32_t>(min(n0 + kCfPix, a.N) - 1), od, oh, ow);
    const int hi = od * g.IH + cf_clamp_row(oh * g.SH - g.PH + (g.KH - 1) * g.DH + 1, g.IH);
    const int px = max(0, min(hi - lo, hp.px_rows)) * g.IW;  // <= PX (the launcher's bound)
    const int ngrp = (px + 3) >> 2;
    // this lane's pixel (MFMA row): halo index of its window's first tap and its coordinates
    coords(p0 + static_cast<uint32_t>(min(n0 + wp * 32 + r32, a.N - 1)), od, oh, ow);
    const int ihb = oh * g.SH - g.PH;
    const int iwb = ow * g.SW - g.PW;
    const int base_px = (od * g.IH + ihb - lo) * g.IW + iwb;

    if (tid < 16) {
        reinterpret_cast<uint32_t *>(s_x + PX * kCfIc)[tid] = 0u;
    }

    i32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        acc[r] = 0;
    }
    const long long plane = static_cast<long long>(g.ID) * g.IH * g.IW;
    const int nchunk = g.ICg / 16;
    // the group's input ends here: a dword load that would pass it is moved back and shifted
    const int8_t *in_end = a.B + plane * g.ICg;

    for (int c0 = 0; c0 < nchunk; c0 += kCfIc / 16) {
        const int nc = min(kCfIc / 16, nchunk - c0);
        if (c0 > 0) {
            __syncthreads();  // the previous block is read
        }
        // weights: item (channel, 16-channel chunk)
        for (int it = tid; it < kCfCh * (kCfIc / 16); it += 256) {
            const int ch = it >> 2;
            const int c = it & 3;
            uint32_t w[4 * T];
            const bool ok = c < nc;
            const int8_t *src = a.A + static_cast<long long>(min(oc0 + ch, a.M - 1)) * a.lda +
                                static_cast<long long>(c0 + (ok ? c : 0)) * (16 * T);
#pragma unroll
            for (int q = 0; q < T; ++q) {
                const u32x4 v = reinterpret_cast<const u32x4 *>(src)[q];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    w[4 * q + e] = ok ? v[e] : 0u;
                }
            }
#pragma unroll
            for (int t = 0; t < T; ++t) {
                u32x4 o;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // bytes b0 .. b3 of the item: compile-time positions
                    const int b0 = t + T * (4 * q), b1 = b0 + T, b2 = b1 + T, b3 = b2 + T;
                    const uint32_t l = __builtin_amdgcn_perm(
                        w[b1 >> 2], w[b0 >> 2],
                        0x0c0c0000u | static_cast<uint32_t>((b0 & 3) | ((4 + (b1 & 3)) << 8)));
                    const uint32_t u = __builtin_amdgcn_perm(
                        w[b3 >> 2], w[b2 >> 2],
                        0x0c0c0000u | static_cast<uint32_t>((b2 & 3) | ((4 + (b3 & 3)) << 8)));
                    o[q] = l | (u << 16);
                }
                *reinterpret_cast<u32x4 *>(s_w + (t * kCfCh + ch) * kCfIc +
                                           ((c ^ ((ch >> 2) & 3)) << 4)) = o;
            }
        }
        // input: item (4 consecutive halo pixels, 16-channel chunk)
        for (int it = tid; it < ngrp * nc; it += 256) {
            const int c = it / ngrp;
            const int grp = it - c * ngrp;
            const int8_t *src = a.B + static_cast<long long>(16 * (c0 + c)) * plane +
                                static_cast<long long>(lo) * g.IW + 4 * grp;
            uint32_t d[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int8_t *p = src + k * plane;
                const long long over = p + 4 - in_end;
                const uint32_t back = over > 0 ? static_cast<uint32_t>(over) : 0u;
                __builtin_memcpy(&d[k], p - back, 4);
                d[k] >>= 8 * back;
            }
            u32x4 o[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                // 4 x 4 byte transpose of channels 4 q .. 4 q + 3
                const uint32_t a0 = __builtin_amdgcn_perm(d[4 * q + 1], d[4 * q], 0x05010400u);
                const uint32_t a1 = __builtin_amdgcn_perm(d[4 * q + 1], d[4 * q], 0x07030602u);
                const uint32_t b0 = __builtin_amdgcn_perm(d[4 * q + 3], d[4 * q + 2], 0x05010400u);
                const uint32_t b1 = __builtin_amdgcn_perm(d[4 * q + 3], d[4 * q + 2], 0x07030602u);
                o[0][q] = __builtin_amdgcn_perm(b0, a0, 0x05040100u);
                o[1][q] = __builtin_amdgcn_perm(b0, a0, 0x07060302u);
                o[2][q] = __builtin_amdgcn_perm(b1, a1, 0x05040100u);
                o[3][q] = __builtin_amdgcn_perm(b1, a1, 0x07060302u);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                *reinterpret_cast<u32x4 *>(s_x + (4 * grp + e) * kCfIc +
                                           ((c ^ (grp & 3)) << 4)) = o[e];
            }
        }
        __syncthreads();
        const int ksteps = (nc + 1) >> 1;
        int kh = 0, kw = 0;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int ih = ihb + kh * g.DH, iw = iwb + kw * g.DW;
            const bool ok = ih >= 0 && ih < g.IH && iw >= 0 && iw < g.IW;
            const int idx = ok ? base_px + kh * g.DH * g.IW + kw * g.DW : PX;
            for (int k = 0; k < ksteps; ++k) {
                const int c = 2 * k + h;
                const i32x4 fx = *reinterpret_cast<const i32x4 *>(
                    s_x + idx * kCfIc + ((c ^ ((idx >> 2) & 3)) << 4));
                const i32x4 fw = *reinterpret_cast<const i32x4 *>(
                    s_w + (t * kCfCh + wc * 32 + r32) * kCfIc + ((c ^ ((r32 >> 2) & 3)) << 4));
                acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fx, fw, acc, 0, 0, 0);
            }
            if (++kw == g.KW) {
                kw = 0;
                ++kh;
            }
        }
    }
    __syncthreads();  // the tiles are read: the results are turned in s_w's place

    int32_t mult, shift;
    column_multiplier_val(a.scale_a, p_sb, a.scale_d, mult, shift);
    constexpr int PITCH = kCfPix + 16;
    static_assert(kCfCh * PITCH <= (T * kCfCh * kCfIc > (PX + 4) * kCfIc ? T * kCfCh * kCfIc
                                                                        : (PX + 4) * kCfIc),
                  "the result tile fits");
    int8_t *s_o = T * kCfCh * kCfIc >= kCfCh * PITCH ? s_w : s_x;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t v = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int8_t y = requant_dev(static_cast<int32_t>(static_cast<uint32_t>(acc[4 * q + e]) +
                                                              static_cast<uint32_t>(p_bias)),
                                         mult, shift, a.zp_d, a.cmin, a.cmax);
            v |= static_cast<uint32_t>(static_cast<uint8_t>(y)) << (8 * e);
        }
        *reinterpret_cast<uint32_t *>(s_o + (wc * 32 + r32) * PITCH + wp * 32 + 8 * q + 4 * h) = v;
    }
    __syncthreads();
    // 64 channels x 4 runs of 16 pixels: one per thread
    const int ch = tid >> 2;
    const int run = (tid & 3) * 16;
    if (oc0 + ch < a.M && n0 + run < a.N) {
        const u32x4 v = *reinterpret_cast<const u32x4 *>(s_o + ch * PITCH + run);
        int8_t *d = static_cast<int8_t *>(a.D) + static_cast<long long>(oc0 + ch) * a.ldd + n0 + run;
        if (n0 + run + 16 <= a.N && (reinterpret_cast<uintptr_t>(d) & 15u) == 0) {
            *reinterpret_cast<u32x4 *>(d) = v;
        } else if (n0 + run + 16 <= a.N && (reinterpret_cast<uintptr_t>(d) & 3u) == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                reinterpret_cast<uint32_t *>(d)[e] = v[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                if (n0 + run + e < a.N) {
                    d[e] = static_cast<int8_t>(v[e >> 2] >> (8 * (e & 3)));
                }
            }
        }
    }
}

// Launches the channel-first kernel when the geometry suits it; false otherwise.
inline bool launch_conv_cf(const Int8Args &a, hipStream_t stream)
{
    const ConvGeom &g = a.cv;
    const int taps = g.KH * g.KW;
    if (g.KD != 1 || g.SD != 1 || g.PD != 0 || g.ICg % 16 != 0 || g.KH <= 0 || g.KW <= 0 ||
        (taps != 1 && taps != 9 && taps != 25) || a.C != nullptr || a.d_row0 != 0 ||
        a.p0 + a.N >= (1ll << 31) || static_cast<long long>(g.ID) * g.IH * g.IW >= (1ll << 30) ||
        g.OH > 4096 || static_cast<long long>(g.OH) * g.SH >= (1ll << 30) ||
        static_cast<long long>(g.ID) * g.IH * g.IW * g.ICg < 4) {
        return false;
    }
    // the output pixels must lie in the input's depth planes (the runs of the reference do)
    if (a.p0 + a.N > static_cast<long long>(g.ID) * g.OH * g.OW) {
        return false;
    }
    const long long rows =
        cf_halo_rows(g.OH, g.OW, g.IH, g.SH, g.PH, (g.KH - 1) * g.DH + 1, kCfPix);
    const long long px = rows * g.IW;
    if (rows <= 0 || px > 1024 || (taps == 25 && px > 512)) {
        return false;
    }
    CfPlan hp;
    hp.px_rows = static_cast<int>(rows);
    hp.tiles_c = (a.M + kCfCh - 1) / kCfCh;
    const long long tiles = static_cast<long long>((a.N + kCfPix - 1) / kCfPix) * hp.tiles_c;
    if (!grid_fits(tiles + 8, 256)) {
        return false;
    }
    hp.tiles = static_cast<int>(tiles);
    hp.per_xcd = static_cast<int>((tiles + 7) / 8);
    const dim3 grid(8 * static_cast<unsigned>(hp.per_xcd)), block(256);
    if (taps == 1) {
        if (px <= 512) {
            hipLaunchKernelGGL((conv_cf_kernel<1, 512>), grid, block, 0, stream, a, hp);
        } else {
            hipLaunchKernelGGL((conv_cf_kernel<1, 1024>), grid, block, 0, stream, a, hp);
        }
    } else if (taps == 9) {
        if (px <= 512) {
            hipLaunchKernelGGL((conv_cf_kernel<9, 512>), grid, block, 0, stream, a, hp);
        } else {
            hipLaunchKernelGGL((conv_cf_kernel<9, 1024>), grid, block, 0, stream, a, hp);
        }
    } else {
        hipLaunchKernelGGL((conv_cf_kernel<25, 512>), grid, block, 0, stream, a, hp);
    }
    return true;
}

}  // namespace
}  // namespace tqt
