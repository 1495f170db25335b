// Large-tile int8 MFMA contraction of W8A8 (static and per-row quantized activations, plain or
// packed operands) for outputs that fill the chip with tiles of 128 x 128 and more. Included by
// int8_mfma.hip, whose argument struct and epilogue steps it uses; the tiling, the pipeline, the k
// groups and the turned epilogue are those of int8_tile.hpp.
//
// What bounds it: int8_stream_kernel's waves own 64 x 32 of a 128 x 128 tile and read 1.5 KiB of
// LDS per v_mfma_i32_32x32x32_i8 - three times what LDS delivers in the MFMA's 32 cycles beside it
// on the other SIMDs. A wave here owns 128 x 64 (0.75 KiB per MFMA).
#pragma once

namespace tqt {
namespace {

template <int MI, int NI, int WGM, int WGN, int KS, int NSMAX, int EPI, int PK>
__global__ __launch_bounds__(64 * WGM * WGN * KS, 2) void w8a8_tile_kernel(Int8Args a, int tiles_m,
                                                                          int tiles_n, int per_xcd,
                                                                          int vec_d)
{
    static_assert(KS == 1 || KS == 2, "k groups");
    static_assert(KS == 1 || NI == KS, "a k group finishes one 32-channel column of each wave tile");
    constexpr int WAVES = WGM * WGN * KS;
    constexpr int THREADS = 64 * WAVES;
    constexpr int BM = 32 * MI * WGM;
    constexpr int BN = 32 * NI * WGN;
    constexpr int SX = BM * kTileK;
    constexpr int SW = BN * kTileK;
    constexpr int STAGE = SX + SW;
    constexpr int NS = tile_stages(STAGE, NSMAX);
    static_assert(NS >= 2, "ring");
    constexpr int XPW = SX / 1024 / WAVES;  // 1 KiB load blocks per wave
    constexpr int WPW = SW / 1024 / WAVES;
    static_assert(XPW * WAVES * 1024 == SX && WPW * WAVES * 1024 == SW, "whole blocks per wave");
    constexpr int PER_STAGE = XPW + WPW;
    constexpr int KPW = 4 / KS;  // k-steps per wave and stage (even)
    static_assert((NS - 1) * PER_STAGE < 64, "vmcnt");
    static_assert(BM * BN * 4 * (KS - 1) <= NS * STAGE, "partial tiles fit the ring");
    constexpr bool kAP = (PK & PK_A) != 0;
    constexpr bool kBP = (PK & PK_B) != 0;
    constexpr bool kDyn = is_dyn(EPI);

    __shared__ __attribute__((aligned(1024))) int8_t ring[NS * STAGE];
    __shared__ __attribute__((aligned(16))) int32_t s_c0[BN];  // multiplier, or channel scale bits
    __shared__ __attribute__((aligned(16))) int32_t s_c1[BN];  // shift, or bias bits
    __shared__ __attribute__((aligned(16))) int32_t s_c2[BN];  // int32 bias, or channel sum
    __shared__ float s_sa[kDyn ? BM : 1];
    __shared__ int32_t s_za[kDyn ? BM : 1];

    int tm, tn;
    if (!tile_coords(tiles_m, tiles_n, per_xcd, tm, tn)) {
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

    // epilogue operands, requested ahead of the stream (their wait is the first stage's)
    static_assert(BM <= THREADS && BN <= THREADS, "one row and channel per thread");
    const int pre_n = min(n0 + tid, a.N - 1);
    const float pre_sb = a.scale_b[!kDyn && a.quant_channel_b == 1 ? 0 : pre_n];
    float pre_fb = 0.f, pre_sa = 0.f;
    int32_t pre_za = 0, pre_bias = 0;
    if constexpr (kDyn) {
        const int pre_m = min(m0 + tid, a.M - 1);
        pre_fb = dyn_bias<EPI>(a, pre_n);
        pre_sa = a.dyn_sa[pre_m];
        pre_za = a.dyn_za[pre_m];
    } else if (a.bias) {
        pre_bias = a.bias[pre_n];
    }

    // Load roles of an 8-row block: plain rows, lane = 8 * row + slot with chunk slot ^ ((row >> 1)
    // & 7); packed rows, lane = 8 * slot + row with chunk slot ^ (block & 1). Offsets are 32-bit
    // from the tile's first row or panel (the launcher bounds the strides).
    auto chunk_of = [&](bool packed, int blk) {
        return static_cast<uint32_t>(packed ? ((lane >> 3) ^ (blk & 1))
                                            : ((lane & 7) ^ ((4 * blk + (lane >> 4)) & 7)));
    };
    long long xbase, wbase;
    if constexpr (kAP) {
        int w;
        xbase = pack_row_fixed<kPackI8MStep>(a.pa, m0 & ~static_cast<int>(kPackI8MStep - 1), w);
    } else {
        xbase = static_cast<long long>(m0) * a.lda;
    }
    if constexpr (kBP) {
        int w;
        wbase = pack_row_fixed<kPackI8NStep>(a.pb, n0 & ~static_cast<int>(kPackI8NStep - 1), w);
    } else {
        wbase = static_cast<long long>(n0) * a.ldb;
    }
    const i32x4 x_rsrc = raw_rsrc(a.A + xbase, kTileRecords);
    const i32x4 w_rsrc = raw_rsrc(a.B + wbase, kTileRecords);
    uint32_t off[PER_STAGE];  // activations, then weights
    [[maybe_unused]] uint32_t mul[PER_STAGE];
#pragma unroll
    for (int j = 0; j < PER_STAGE; ++j) {
        const bool is_x = j < XPW;
        const int blk = is_x ? wave * XPW + j : wave * WPW + j - XPW;
        const bool packed = is_x ? kAP : kBP;
        const int row = 8 * blk + (packed ? (lane & 7) : (lane >> 3));
        int w = 1;
        if (is_x) {
            const int r = min(m0 + row, a.M - 1);
            if constexpr (kAP) {
                off[j] = static_cast<uint32_t>(pack_row_fixed<kPackI8MStep>(a.pa, r, w) - xbase);
            } else {
                off[j] = static_cast<uint32_t>(r - m0) * static_cast<uint32_t>(a.lda);
            }
        } else {
            const int r = min(n0 + row, a.N - 1);
            if constexpr (kBP) {
                off[j] = static_cast<uint32_t>(pack_row_fixed<kPackI8NStep>(a.pb, r, w) - wbase);
            } else {
                off[j] = static_cast<uint32_t>(r - n0) * static_cast<uint32_t>(a.ldb);
            }
        }
        mul[j] = static_cast<uint32_t>(w);
        off[j] += 16u * chunk_of(packed, blk) * mul[j];
    }
    const uint32_t K = static_cast<uint32_t>(a.K);
    auto issue = [&](int st, int base) {
        const uint32_t k0 = static_cast<uint32_t>(st) * kTileK;
#pragma unroll
        for (int j = 0; j < PER_STAGE; ++j) {
            const bool is_x = j < XPW;
            const int blk = is_x ? wave * XPW + j : wave * WPW + j - XPW;
            const bool packed = is_x ? kAP : kBP;
            const uint32_t k = 16u * chunk_of(packed, blk) + k0;
            const uint32_t o = off[j] + (packed ? __umul24(k0, mul[j]) : k0);
            dma_lds16_buf(is_x ? x_rsrc : w_rsrc, static_cast<int>(k < K ? o : kTileOob),
                          ring + base + (is_x ? 0 : SX) + blk * 1024);
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
    [[maybe_unused]] int32_t rs[NI] = {};

    auto lds_pos = [](bool packed, int row, int c) {
        return packed ? (row >> 3) * 1024 + ((((c ^ ((row >> 3) & 1)) << 3) + (row & 7)) << 4)
                      : row * kTileK + ((c ^ ((row >> 1) & 7)) << 4);
    };
    int x_lane[KPW], w_lane[KPW];
#pragma unroll
    for (int q = 0; q < KPW; ++q) {
        const int c = 2 * (ks * KPW + q) + h;
        x_lane[q] = wm * MI * 32 * kTileK + lds_pos(kAP, r32, c);
        w_lane[q] = SX + wn * NI * 32 * kTileK + lds_pos(kBP, r32, c);
    }
    i32x4 fx[2][MI], fw[2][NI];
    auto read = [&](int p, int base, int q) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            fw[p][j] = *reinterpret_cast<const i32x4 *>(ring + base + w_lane[q] + j * 32 * kTileK);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            fx[p][i] = *reinterpret_cast<const i32x4 *>(ring + base + x_lane[q] + i * 32 * kTileK);
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
            if constexpr (kDyn) {
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    rs[j] = __builtin_amdgcn_sdot4(fw[p][j][d], 0x01010101, rs[j], false);
                }
            }
        }
    };
    // the next k-step's reads one by one behind the MFMAs of the current one
    auto order = [&]() {
#pragma unroll
        for (int m = 0; m < MI + NI; ++m) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, MI * NI, 0);
        __builtin_amdgcn_sched_barrier(0);
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
    read(0, 0, 0);
    int cur = 0;
    for (int st = 0; st < nst; ++st) {
#pragma unroll
        for (int q = 0; q < KPW; ++q) {
            if (q + 1 == KPW) {
                // the stage is read (its last operands are in registers): refill its buffer; the
                // next stage has landed
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(tile_waitcnt((NS - 2) * PER_STAGE));
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                issue(st + NS, cur);
                cur = cur == (NS - 1) * STAGE ? 0 : cur + STAGE;
            }
            read((q & 1) ^ 1, cur, (q + 1) % KPW);
            mfma(q & 1);
            order();
        }
    }

    // every load landed, every wave past its last LDS read: the ring is free
    __builtin_amdgcn_s_waitcnt(tile_waitcnt(0));
    if (tid < BN) {
        if constexpr (kDyn) {
            s_c0[tid] = __builtin_bit_cast(int32_t, pre_sb);
            s_c1[tid] = __builtin_bit_cast(int32_t, pre_fb);
            s_c2[tid] = 0;
        } else {
            column_multiplier_val(a.scale_a, pre_sb, a.scale_d, s_c0[tid], s_c1[tid]);
            s_c2[tid] = pre_bias;
        }
    }
    if (kDyn && tid < BM) {
        s_sa[tid] = pre_sa;
        s_za[tid] = pre_za;
    }
    __syncthreads();
    if constexpr (kDyn) {
        if (wm == 0) {
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                atomicAdd(&s_c2[(wn * NI + j) * 32 + r32], rs[j]);
            }
        }
    }
    if constexpr (KS > 1) {
        // column j is finished by k group j: the other group hands its fragments over
        i32x4 *part = reinterpret_cast<i32x4 *>(ring) +
                      static_cast<size_t>(wm * WGN + wn) * (MI * NI * 256);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                if (j != ks) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        part[(i * NI + j) * 256 + g * 64 + lane] =
                            i32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2],
                                  acc[i][j][4 * g + 3]};
                    }
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                if (j == ks) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const i32x4 v = part[(i * NI + j) * 256 + g * 64 + lane];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            acc[i][j][4 * g + e] = static_cast<int32_t>(
                                static_cast<uint32_t>(acc[i][j][4 * g + e]) +
                                static_cast<uint32_t>(v[e]));
                        }
                    }
                }
            }
        }
    }
    __syncthreads();

    // Epilogue: each 32-row slice of the wave's finished columns (CW channels) is turned through
    // the wave's own LDS buffer, so that a lane reads runs of one row and keeps its channels'
    // constants: 16 channels per lane for int8 results (16-byte stores), four for float ones.
    constexpr int CW = KS > 1 ? 32 : 32 * NI;
    constexpr int PITCH = CW * 4 + 16;
    static_assert(WAVES * 32 * PITCH <= NS * STAGE, "the turning buffers fit the ring");
    int8_t *turn = ring + wave * (32 * PITCH);
    constexpr int CPL = kDyn ? 4 : 16;  // channels per lane
    constexpr int LPR = CW / CPL;       // lanes per row
    constexpr int RPI = 64 / LPR;       // rows per instruction
    const int lc = wn * NI * 32 + (KS > 1 ? ks * 32 : 0) + (lane % LPR) * CPL;
    const int gn = n0 + lc;
    i32x4 c0[CPL / 4], c1[CPL / 4], c2[CPL / 4];
#pragma unroll
    for (int q = 0; q < CPL / 4; ++q) {
        c0[q] = *reinterpret_cast<const i32x4 *>(&s_c0[lc + 4 * q]);
        c1[q] = *reinterpret_cast<const i32x4 *>(&s_c1[lc + 4 * q]);
        c2[q] = *reinterpret_cast<const i32x4 *>(&s_c2[lc + 4 * q]);
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            if (KS == 1 || j == ks) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    *reinterpret_cast<i32x4 *>(turn + r32 * PITCH + (KS > 1 ? 0 : j * 128) +
                                               (8 * g + 4 * h) * 4) =
                        i32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2],
                              acc[i][j][4 * g + 3]};
                }
            }
        }
        asm volatile("" ::: "memory");
#pragma unroll 1
        for (int r = 0; r < 32; r += RPI) {
            const int row = r + lane / LPR;
            const int lr = (wm * MI + i) * 32 + row;
            const int gm = m0 + lr;
            if (gm >= a.M || gn >= a.N) {
                continue;
            }
            const i32x4 *src = reinterpret_cast<const i32x4 *>(turn + row * PITCH +
                                                               (lane % LPR) * CPL * 4);
            if constexpr (kDyn) {
                const i32x4 s = src[0];
                const f32x4 sb = __builtin_bit_cast(f32x4, c0[0]);
                const f32x4 fb = __builtin_bit_cast(f32x4, c1[0]);
                const float sa = s_sa[lr];
                const int32_t za = s_za[lr];
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t x = static_cast<uint32_t>(s[e]) -
                                 static_cast<uint32_t>(za) * static_cast<uint32_t>(c2[0][e]);
                    if (!dyn_zp_in_range(za)) {
                        x = gn + e < a.N ? dyn_exact_acc<PK>(a, gm, gn + e, za) : 0u;
                    }
                    v[e] = dyn_value<EPI>(a, x, sb[e], sa, fb[e]);
                }
                constexpr int kOut = EPI == EPI_DYN_F32 ? OUT_F32 : OUT_F16;
                const long long d0 = static_cast<long long>(gm) * a.ldd + gn;
                if (vec_d && gn + 4 <= a.N) {
                    store_out4<kOut>(a.D, d0, v);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (gn + e < a.N) {
                            store_out<kOut>(a.D, d0 + e, v[e]);
                        }
                    }
                }
            } else {
                u32x4 out;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const i32x4 s = src[q];
                    uint32_t b[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        uint32_t v = static_cast<uint32_t>(s[e]) + static_cast<uint32_t>(c2[q][e]);
                        if (a.C && gn + 4 * q + e < a.N) {
                            v += static_cast<uint32_t>(
                                a.C[static_cast<long long>(gm) * a.ldc + gn + 4 * q + e]);
                        }
                        b[e] = static_cast<uint8_t>(requant_dev(static_cast<int32_t>(v), c0[q][e],
                                                                c1[q][e], a.zp_d, a.cmin, a.cmax));
                    }
                    out[q] = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
                }
                int8_t *d = static_cast<int8_t *>(a.D) + static_cast<long long>(gm) * a.ldd + gn;
                if (vec_d && gn + 16 <= a.N) {
                    *reinterpret_cast<u32x4 *>(d) = out;
                } else {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        if (gn + e < a.N) {
                            d[e] = static_cast<int8_t>(out[e >> 2] >> (8 * (e & 3)));
                        }
                    }
                }
            }
        }
    }
}

template <int MI, int NI, int WGM, int WGN, int KS, int NS, int EPI, int PK>
void launch_w8_tile(const Int8Args &a, hipStream_t stream)
{
    constexpr int BM = 32 * MI * WGM, BN = 32 * NI * WGN;
    const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
    const long long tiles = static_cast<long long>(tiles_m) * tiles_n;
    const int per_xcd = static_cast<int>((tiles + 7) / 8);
    constexpr int kVec = EPI == EPI_REQUANT_I8 ? 16 : 4;
    constexpr int kElem = EPI == EPI_REQUANT_I8 ? 1 : (EPI == EPI_DYN_F32 ? 4 : 2);
    const int vec_d = a.ldd % kVec == 0 && reinterpret_cast<uintptr_t>(a.D) % (kVec * kElem) == 0;
    hipLaunchKernelGGL((w8a8_tile_kernel<MI, NI, WGM, WGN, KS, NS, EPI, PK>),
                       dim3(8 * static_cast<unsigned>(per_xcd)), dim3(64 * WGM * WGN * KS), 0,
                       stream, a, tiles_m, tiles_n, per_xcd, vec_d);
}

// The large tiles where they are the faster ones (route.hpp) and the strides fit their 32-bit offsets.
template <int EPI, int PK>
bool launch_w8a8_tile(const Int8Args &a, hipStream_t stream)
{
    if (a.lda >= (1 << 22) || a.ldb >= (1 << 22)) {
        return false;
    }
    constexpr bool kDyn = is_dyn(EPI);
    const W8A8Tile tile = w8a8_tile(a.M, a.N, a.K, kDyn);
    if (tile == W8A8_NO_TILE) {
        return false;
    }
    if (tile == W8A8_TILE_256X256) {
        launch_w8_tile<4, 2, 2, 4, 1, 2, EPI, PK>(a, stream);
    } else if constexpr (kDyn) {
        // two k groups: 128 x 64 per wave, the channel sums' dot products over half the k-steps
        launch_w8_tile<4, 2, 1, 2, 2, 2, EPI, PK>(a, stream);
    } else {
        launch_w8_tile<2, 2, 2, 2, 1, 2, EPI, PK>(a, stream);
    }
    return true;
}

}  // namespace
}  // namespace tqt
