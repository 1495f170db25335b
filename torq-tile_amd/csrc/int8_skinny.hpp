// Few-row int8 contraction (W8A8 decode: static and per-row quantized activations, plain or packed
// operands, up to 32 rows per workgroup). Included by int8_mfma.hip, whose argument struct and
// epilogue steps it uses.
//
// A workgroup of 8 wave64s owns 16 output channels over all of k; wave w takes the 128-k blocks w,
// w + 8, w + 16, ... Every wave streams its blocks of 16 weight rows and the activation rows
// through a ring of its own in LDS by direct global -> LDS loads (8 rows x 128 bytes, whole cache
// lines, per instruction; no registers, no staging stores), NS blocks ahead, and meets the others
// only at the end, where the eight exact int32 partial tiles are added and one output per thread
// runs the epilogue.
//
// What bounds it: the weight stream from HBM. The large tiles give N 4096 only 32 workgroups, each
// walking k in serial stages (17 us per 8 x 4096 x 4096 launch, 16.8 MB); here every CU has a
// workgroup whose eight waves stream independently (6.4 us; 8 x 16384 x 8192 24 us, 5.6 TB/s).
// Sixteen channels a workgroup (and not 32 or 64) because a decode layer has a few thousand
// channels for 256 CUs; the activation rows are re-read from L2 by every workgroup.
#pragma once

namespace tqt {
namespace {

constexpr int kSkinnyWaves = 8;
constexpr int kSkinnyN = 16;  // channels per workgroup
constexpr int kSkinnyK = 128;  // k per block

// XB: 8-row blocks of activations (1, 2 or 4: up to 8, 16 or 32 rows); NS: blocks in flight.
template <int XB, int NS, int EPI, int PK>
__global__ __launch_bounds__(kSkinnyWaves * 64) void int8_skinny_kernel(Int8Args a)
{
    constexpr int MT = (XB + 1) / 2;  // 16-row MFMA tiles
    constexpr int PER = 2 + XB;       // loads per block
    constexpr int SLOT = PER * 1024;
    constexpr int RING = NS * SLOT;   // bytes per wave
    constexpr bool kAP = (PK & PK_A) != 0;
    constexpr bool kBP = (PK & PK_B) != 0;
    static_assert(MT * 1024 + 64 <= RING, "a wave's partial tile fits its ring");
    static_assert((NS - 1) * PER < 64, "vmcnt");
    __shared__ __attribute__((aligned(1024))) int8_t ring[kSkinnyWaves * RING];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * kSkinnyN;
    const int m0 = blockIdx.y * (8 * XB);

    // Epilogue operands of this thread's output (row tid / 16, channel tid % 16), requested ahead
    // of the stream.
    const int orow = tid >> 4;
    const int ocol = tid & 15;
    const int gm = m0 + orow;
    const int gn = n0 + ocol;
    const bool out_ok = orow < 8 * XB && gm < a.M && gn < a.N;
    const int cm = min(gm, a.M - 1), cn = min(gn, a.N - 1);
    const float p_sb = a.scale_b[EPI == EPI_REQUANT_I8 && a.quant_channel_b == 1 ? 0 : cn];
    float p_sa = 0.f, p_fb = 0.f;
    int32_t p_za = 0;
    uint32_t p_add = 0;
    if constexpr (is_dyn(EPI)) {
        p_sa = a.dyn_sa[cm];
        p_za = a.dyn_za[cm];
        p_fb = dyn_bias<EPI>(a, cn);
    } else {
        if (a.bias) {
            p_add = static_cast<uint32_t>(a.bias[cn]);
        }
        if (a.C) {
            p_add += static_cast<uint32_t>(a.C[static_cast<long long>(cm) * a.ldc + cn]);
        }
    }

    // Load roles of an 8-row block (1 KiB): plain rows, lane = 8 * row + slot, the slot holding
    // 16-byte chunk slot ^ ((row >> 1) & 7); packed rows (16-byte chunks stored chunk-major), lane =
    // 8 * slot + row, the slot holding chunk slot ^ (block & 1) - 8 consecutive lanes read 128
    // contiguous bytes either way. Offsets are 32-bit from a uniform base (the launcher bounds the
    // strides); rows past the last reload it, k past the end is out of range (zeros).
    auto chunk_of = [&](bool packed, int blk) {
        const int row = 8 * blk + (lane >> 3);
        return packed ? ((lane >> 3) ^ (blk & 1)) : ((lane & 7) ^ ((row >> 1) & 7));
    };
    long long abase, bbase;
    if constexpr (kAP) {
        int w;
        abase = pack_row_fixed<kPackI8MStep>(a.pa, m0 & ~static_cast<int>(kPackI8MStep - 1), w);
    } else {
        abase = static_cast<long long>(m0) * a.lda;
    }
    if constexpr (kBP) {
        int w;
        bbase = pack_row_fixed<kPackI8NStep>(a.pb, n0 & ~static_cast<int>(kPackI8NStep - 1), w);
    } else {
        bbase = static_cast<long long>(n0) * a.ldb;
    }
    const i32x4 a_rsrc = raw_rsrc(a.A + abase, 0x7fffffff);
    const i32x4 b_rsrc = raw_rsrc(a.B + bbase, 0x7fffffff);
    uint32_t off[PER];  // weights, then activations
    uint32_t kc[PER];   // first k of this lane's chunk
    int mul[PER];       // k multiplier of a packed row (its panel width)
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const bool is_b = j < 2;
        const int blk = is_b ? j : j - 2;
        const bool packed = is_b ? kBP : kAP;
        const int row = 8 * blk + (packed ? (lane & 7) : (lane >> 3));
        kc[j] = static_cast<uint32_t>(chunk_of(packed, blk)) * 16u;
        mul[j] = 1;
        if (is_b) {
            const int r = min(n0 + row, a.N - 1);
            if constexpr (kBP) {
                off[j] = static_cast<uint32_t>(pack_row_fixed<kPackI8NStep>(a.pb, r, mul[j]) - bbase);
            } else {
                off[j] = static_cast<uint32_t>(r - n0) * static_cast<uint32_t>(a.ldb);
            }
        } else {
            const int r = min(m0 + row, a.M - 1);
            if constexpr (kAP) {
                off[j] = static_cast<uint32_t>(pack_row_fixed<kPackI8MStep>(a.pa, r, mul[j]) - abase);
            } else {
                off[j] = static_cast<uint32_t>(r - m0) * static_cast<uint32_t>(a.lda);
            }
        }
    }
    int8_t *mine = ring + wave * RING;
    const uint32_t K = static_cast<uint32_t>(a.K);
    auto issue = [&](int it, int slot) {
        const uint32_t k0 = static_cast<uint32_t>(it * kSkinnyWaves + wave) * kSkinnyK;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const uint32_t k = kc[j] + k0;
            const bool packed = j < 2 ? kBP : kAP;
            const uint32_t o = off[j] + (packed ? __umul24(k, static_cast<uint32_t>(mul[j])) : k);
            dma_lds16_buf(j < 2 ? b_rsrc : a_rsrc, static_cast<int>(k < K ? o : 0x80000000u),
                          mine + slot * SLOT + j * 1024);
        }
    };

    const int nit = (a.K + kSkinnyWaves * kSkinnyK - 1) / (kSkinnyWaves * kSkinnyK);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        issue(s, s);
    }

    // MFMA operands: lane (r = lane % 16, g = lane / 16) takes chunk 4 t + g of row r for step t
    const int fr = lane & 15;
    const int fg = lane >> 4;
    auto lds_pos = [](bool packed, int row, int c) {
        return packed ? (row >> 3) * 1024 + ((((c ^ ((row >> 3) & 1)) << 3) + (row & 7)) << 4)
                      : row * kSkinnyK + ((c ^ ((row >> 1) & 7)) << 4);
    };
    i32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        acc[i] = i32x4{0, 0, 0, 0};
    }
    int32_t rs = 0;  // this lane's share of sum_k q_b of its channel
    for (int it0 = 0; it0 < nit; it0 += NS) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (it0 + s >= nit) {
                break;
            }
            __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0((NS - 1) * PER));
            asm volatile("" ::: "memory");
            const int8_t *blk = mine + s * SLOT;
            i32x4 fb[2], fa[MT][2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                fb[t] = *reinterpret_cast<const i32x4 *>(blk + lds_pos(kBP, fr, 4 * t + fg));
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    // with one 8-row block the tile's upper rows repeat the lower (not stored)
                    const int row = XB == 1 ? (fr & 7) : 16 * i + fr;
                    fa[i][t] = *reinterpret_cast<const i32x4 *>(blk + 2048 +
                                                                lds_pos(kAP, row, 4 * t + fg));
                }
            }
            // the block is in registers before its slot is refilled
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(63));
            asm volatile("" ::: "memory");
            issue(it0 + s + NS, s);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[i][t], fb[t], acc[i], 0, 0, 0);
                }
                if constexpr (is_dyn(EPI)) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        rs = __builtin_amdgcn_sdot4(fb[t][q], 0x01010101, rs, false);
                    }
                }
            }
        }
    }

    // partial tiles (row, channel) of every wave, each in its own ring; the loads still in flight
    // into it (blocks past k, zeros) land first
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
    asm volatile("" ::: "memory");
    int32_t *part = reinterpret_cast<int32_t *>(mine);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            part[(16 * i + 4 * fg + r) * 16 + fr] = acc[i][r];
        }
    }
    if constexpr (is_dyn(EPI)) {
        int32_t t = rs + __shfl_xor(rs, 16);
        t += __shfl_xor(t, 32);
        if (lane < 16) {
            part[MT * 256 + lane] = t;
        }
    }
    __syncthreads();
    if (!out_ok) {
        return;
    }
    uint32_t sum = 0, rsum = 0;
#pragma unroll
    for (int w = 0; w < kSkinnyWaves; ++w) {
        const int32_t *pw = reinterpret_cast<const int32_t *>(ring + w * RING);
        sum += static_cast<uint32_t>(pw[orow * 16 + ocol]);
        if constexpr (is_dyn(EPI)) {
            rsum += static_cast<uint32_t>(pw[MT * 256 + ocol]);
        }
    }
    if constexpr (is_dyn(EPI)) {
        if (dyn_zp_in_range(p_za)) {
            dyn_finish_v<EPI>(a, gn, gm, sum - static_cast<uint32_t>(p_za) * rsum, p_sb, p_sa, p_fb);
        } else {
            dyn_finish_v<EPI>(a, gn, gm, dyn_exact_acc<PK>(a, gm, gn, p_za), p_sb, p_sa, p_fb);
        }
    } else {
        int32_t mult, shift;
        column_multiplier_val(a.scale_a, p_sb, a.scale_d, mult, shift);
        static_cast<int8_t *>(a.D)[static_cast<long long>(gm) * a.ldd + gn] = requant_dev(
            static_cast<int32_t>(sum + p_add), mult, shift, a.zp_d, a.cmin, a.cmax);
    }
}

// The few-row kernel where it is the faster one (route.hpp) and the strides fit its 32-bit offsets.
// Ring depth: 2 blocks (1 from 17 rows on) measured as fast as 3 or 4 at 4096 channels and faster at
// 11008 (11.8 against 12.4 and 15.8 us at 8 rows), where the smaller ring lets two or three
// workgroups share a CU.
template <int EPI, int PK>
bool launch_skinny(const Int8Args &a, hipStream_t stream)
{
    if (a.lda >= (1 << 22) || a.ldb >= (1 << 22) ||
        !w8a8_few_row(a.M, a.N, a.K, is_dyn(EPI), PK != PK_NONE)) {
        return false;
    }
    const int passes = (a.M + 31) / 32;
    const unsigned gx = static_cast<unsigned>((a.N + kSkinnyN - 1) / kSkinnyN);
    const dim3 block(kSkinnyWaves * 64);
    if (a.M <= 8) {
        hipLaunchKernelGGL((int8_skinny_kernel<1, 2, EPI, PK>), dim3(gx, 1), block, 0, stream, a);
    } else if (a.M <= 16) {
        hipLaunchKernelGGL((int8_skinny_kernel<2, 2, EPI, PK>), dim3(gx, 1), block, 0, stream, a);
    } else {
        hipLaunchKernelGGL((int8_skinny_kernel<4, 1, EPI, PK>),
                           dim3(gx, static_cast<unsigned>(passes)), block, 0, stream, a);
    }
    return true;
}

}  // namespace
}  // namespace tqt
