// Int8 contraction for the layouts the 16-byte-aligned kernels refuse (plain operands; odd strides,
// pointers, k or channel counts; the implicit convolution of a first layer's three channels).
// Included by int8_mfma.hip, whose argument struct and epilogue steps it uses.
//
// 64 x 64 outputs per 4 wave64s, k in stages of 128 bytes: the stage's operands are fetched into
// registers during the previous stage's v_mfma_i32_32x32x32_i8, 16 bytes of a row per load at any
// alignment (byte by byte only at the end of k; the convolution's taps byte by byte always, their
// bytes packed when the stage is stored), and stored to LDS as [row][k], rows padded to 144 bytes so
// that 16 lanes' operand reads touch every bank once. The [k, n] B is turned 4 x 4 bytes at a time.
//
// What bounds it: the fetch instructions (per tap byte its bounds and carries), and for a [k, n] B the
// turned dword stores (LDS busy 0.42 of the time at 2032 x 5169 x 1152, 0.6 of it bank conflicts). One
// thread per output, reading both operands byte by byte, took 5430 us for a 2032 x 5169 x 1152
// clamp_i32, 110 ms for a 2000 x 4096 x 4100 requantized product and 514 us for a 7 x 7 stride 2
// convolution of 3 x 221 x 221 pixels to 96 channels; here 62, 88 and 35 us.
#pragma once

namespace tqt {
namespace {

constexpr int kEdgeT = 64;                  // output tile edge
constexpr int kEdgeK = 128;                 // k per stage
constexpr int kEdgePitch = kEdgeK + 16;     // bytes between LDS rows

// Bytes k .. k + 15 of a row of K, zeros past its end.
__device__ __forceinline__ i32x4 edge_load16(const int8_t *row, int k, int K)
{
    i32x4 v = {0, 0, 0, 0};
    if (k + 16 <= K) {
        __builtin_memcpy(&v, row + k, 16);
    } else {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            if (k + j < K) {
                v[j >> 2] |= static_cast<int32_t>(static_cast<uint32_t>(static_cast<uint8_t>(
                                 row[k + j])) << (8 * (j & 3)));
            }
        }
    }
    return v;
}

// Columns n .. n + 3 of row k of a [k, n] matrix, zeros outside it.
__device__ __forceinline__ uint32_t edge_load4(const int8_t *B, long long ldb, int k, int n, int K,
                                               int N)
{
    uint32_t v = 0;
    if (k < K) {
        const int8_t *p = B + static_cast<long long>(k) * ldb + n;
        if (n + 4 <= N) {
            __builtin_memcpy(&v, p, 4);
        } else {
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                if (n + j < N) {
                    v |= static_cast<uint32_t>(static_cast<uint8_t>(p[j])) << (8 * j);
                }
            }
        }
    }
    return v;
}

template <int AM, int BMd, int EPI>
__global__ __launch_bounds__(256) void int8_edge_kernel(Int8Args a)
{
    __shared__ __attribute__((aligned(16))) int8_t lds[2 * kEdgeT * kEdgePitch];
    static_assert(sizeof(lds) >= kEdgeT * kEdgeT * 4, "the output tile fits the stage");
    int8_t *sa = lds, *sb = lds + kEdgeT * kEdgePitch;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wm = (tid >> 6) & 1, wn = tid >> 7;
    const int r32 = lane & 31, h = lane >> 5;
    const int tiles_n = (a.N + kEdgeT - 1) / kEdgeT;
    const int m0 = static_cast<int>(blockIdx.x / tiles_n) * kEdgeT;
    const int n0 = static_cast<int>(blockIdx.x % tiles_n) * kEdgeT;

    // fetch roles: rows tid / 8 and tid / 8 + 32 (past the last: the last again, not stored), 16
    // bytes at 16 (tid % 8)
    const int frow = tid >> 3, fk = 16 * (tid & 7);
    const int8_t *arow[2], *brow[2];
    int px[2][3];  // convolution: first tap's input coordinates of the row's pixel
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int m = min(m0 + frow + 32 * i, a.M - 1);
        if constexpr (AM == A_MATRIX) {
            arow[i] = a.A + static_cast<long long>(m) * a.lda;
        } else {
            const ConvGeom &g = a.cv;
            const long long p = a.p0 + m;
            const long long ohw = static_cast<long long>(g.OH) * g.OW;
            px[i][0] = static_cast<int>(p / ohw) * g.SD - g.PD;
            px[i][1] = static_cast<int>((p / g.OW) % g.OH) * g.SH - g.PH;
            px[i][2] = static_cast<int>(p % g.OW) * g.SW - g.PW;
        }
        if constexpr (BMd == B_NK) {
            brow[i] = a.B + static_cast<long long>(min(n0 + frow + 32 * i, a.N - 1)) * a.ldb;
        }
    }
    // [k, n] B: columns 4 (tid % 16), k groups of four tid / 16 and tid / 16 + 16
    const int qn = 4 * (tid & 15), qk = 4 * (tid >> 4);

    i32x4 ra[2], rb[2];
    uint32_t tap[2][16];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if constexpr (AM == A_MATRIX) {
                ra[i] = edge_load16(arow[i], k0 + fk, a.K);
            } else {
                const ConvGeom &g = a.cv;
                const int k = k0 + fk;
                int t = k / g.ICg;
                int ic = k - t * g.ICg;
                int kw = t % g.KW;
                t /= g.KW;
                int kh = t % g.KH;
                int kd = t / g.KH;
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int id = px[i][0] + kd * g.DD;
                    const int ih = px[i][1] + kh * g.DH;
                    const int iw = px[i][2] + kw * g.DW;
                    tap[i][j] = 0;
                    if (k + j < a.K && static_cast<unsigned>(id) < static_cast<unsigned>(g.ID) &&
                        static_cast<unsigned>(ih) < static_cast<unsigned>(g.IH) &&
                        static_cast<unsigned>(iw) < static_cast<unsigned>(g.IW)) {
                        tap[i][j] = static_cast<uint8_t>(
                            a.A[((static_cast<long long>(id) * g.IH + ih) * g.IW + iw) * g.IC + ic]);
                    }
                    if (++ic == g.ICg) {
                        ic = 0;
                        if (++kw == g.KW) {
                            kw = 0;
                            if (++kh == g.KH) {
                                kh = 0;
                                ++kd;
                            }
                        }
                    }
                }
            }
            if constexpr (BMd == B_NK) {
                rb[i] = edge_load16(brow[i], k0 + fk, a.K);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    rb[i][j] = static_cast<int32_t>(
                        edge_load4(a.B, a.ldb, k0 + qk + 64 * i + j, n0 + qn, a.K, a.N));
                }
            }
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if constexpr (AM == A_CONV_CL) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    ra[i][j] = static_cast<int32_t>(tap[i][4 * j] | tap[i][4 * j + 1] << 8 |
                                                    tap[i][4 * j + 2] << 16 | tap[i][4 * j + 3] << 24);
                }
            }
            *reinterpret_cast<i32x4 *>(sa + (frow + 32 * i) * kEdgePitch + fk) = ra[i];
            if constexpr (BMd == B_NK) {
                *reinterpret_cast<i32x4 *>(sb + (frow + 32 * i) * kEdgePitch + fk) = rb[i];
            } else {
                const uint32_t r0 = static_cast<uint32_t>(rb[i][0]);
                const uint32_t r1 = static_cast<uint32_t>(rb[i][1]);
                const uint32_t r2 = static_cast<uint32_t>(rb[i][2]);
                const uint32_t r3 = static_cast<uint32_t>(rb[i][3]);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t v = ((r0 >> (8 * j)) & 0xffu) | ((r1 >> (8 * j)) & 0xffu) << 8 |
                                       ((r2 >> (8 * j)) & 0xffu) << 16 | (r3 >> (8 * j)) << 24;
                    *reinterpret_cast<uint32_t *>(sb + (qn + j) * kEdgePitch + qk + 64 * i) = v;
                }
            }
        }
    };

    i32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        acc[r] = 0;
    }
    if (a.K > 0) {
        fetch(0);
    }
    for (int k0 = 0; k0 < a.K; k0 += kEdgeK) {
        __syncthreads();  // every wave has read the previous stage
        store();
        __syncthreads();
        if (k0 + kEdgeK < a.K) {
            fetch(k0 + kEdgeK);
        }
#pragma unroll
        for (int s = 0; s < kEdgeK / 32; ++s) {
            const i32x4 fa = *reinterpret_cast<const i32x4 *>(sa + (32 * wm + r32) * kEdgePitch +
                                                              32 * s + 16 * h);
            const i32x4 fb = *reinterpret_cast<const i32x4 *>(sb + (32 * wn + r32) * kEdgePitch +
                                                              32 * s + 16 * h);
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb, acc, 0, 0, 0);
        }
    }
    // the output tile through LDS: lane (column r32, half h) holds rows 8 g + 4 h + e of its column
    __syncthreads();
    int32_t *so = reinterpret_cast<int32_t *>(lds);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        so[(32 * wm + 8 * (i >> 2) + 4 * h + (i & 3)) * kEdgeT + 32 * wn + r32] = acc[i];
    }
    __syncthreads();
    const int gn = n0 + lane;
    if (gn >= a.N) {
        return;
    }
    int32_t mult = 0, shift = 0;
    if constexpr (EPI == EPI_REQUANT_I8) {
        column_multiplier_dev(a.scale_a, a.scale_b, a.quant_channel_b, a.scale_d, gn, mult, shift);
    }
#pragma unroll 1
    for (int row = tid >> 6; row < kEdgeT; row += 4) {
        const int gm = m0 + row;
        if (gm >= a.M) {
            break;
        }
        uint32_t v = static_cast<uint32_t>(so[row * kEdgeT + lane]);
        if (a.C) {
            v += static_cast<uint32_t>(a.C[static_cast<long long>(gm) * a.ldc + gn]);
        }
        if (a.bias) {
            v += static_cast<uint32_t>(a.bias[EPI == EPI_REQUANT_ROW ? gm : gn]);
        }
        const long long d = (a.d_row0 + gm) * a.ldd + gn;
        if constexpr (EPI == EPI_CLAMP_I32) {
            int32_t x = static_cast<int32_t>(v);
            x = x < a.cmin ? a.cmin : x;
            x = x > a.cmax ? a.cmax : x;
            static_cast<int32_t *>(a.D)[d] = x;
        } else {
            if constexpr (EPI == EPI_REQUANT_ROW) {
                column_multiplier_dev(a.scale_a, a.scale_b, a.quant_channel_b, a.scale_d, gm, mult,
                                      shift);
            }
            static_cast<int8_t *>(a.D)[d] =
                requant_dev(static_cast<int32_t>(v), mult, shift, a.zp_d, a.cmin, a.cmax);
        }
    }
}

template <int AM, int BMd, int EPI>
bool launch_edge(const Int8Args &a, hipStream_t stream)
{
    constexpr EdgeForm form = AM == A_CONV_CL       ? EDGE_CONV
                              : BMd == B_NK         ? EDGE_NK
                              : EPI == EPI_CLAMP_I32 ? EDGE_KN_CLAMP
                                                     : EDGE_KN_REQUANT;
    const long long taps = AM == A_CONV_CL
                               ? static_cast<long long>(a.cv.KD) * a.cv.KH * a.cv.KW : 0;
    if (!int8_edge_faster(form, a.M, a.N, a.K, taps)) {
        return false;
    }
    const long long blocks = static_cast<long long>((a.M + kEdgeT - 1) / kEdgeT) *
                             ((a.N + kEdgeT - 1) / kEdgeT);
    if (!grid_fits(blocks, 256)) {
        return false;
    }
    hipLaunchKernelGGL((int8_edge_kernel<AM, BMd, EPI>), dim3(static_cast<unsigned>(blocks)),
                       dim3(256), 0, stream, a);
    return true;
}

}  // namespace
}  // namespace tqt
