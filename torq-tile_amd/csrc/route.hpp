// Rules that say which kernel may take a call, and the index arithmetic whose range they depend on.
// Plain C++ without HIP, so that a host program can evaluate them as the launchers do.
#pragma once

#include <cstdint>
#include <initializer_list>

namespace tqt {

// Compute units of an MI355X, which the estimates below are for (a device with fewer runs the same
// kernels, by estimates that fit it less).
constexpr int kTileCUs = 256;

// Whether `blocks` workgroups of `threads` fit one grid dimension: a launch counts its work-items along
// a dimension in 32 bits.
constexpr bool grid_fits(long long blocks, int threads)
{
    return blocks * threads < 0x100000000ll;
}

constexpr long long ceil_div(long long a, long long b)
{
    return (a + b - 1) / b;
}

// ---------------------------------------------------------------------------------------------
// W4A8: the few-row kernel (int4_skinny.hpp), the tiles of int8_tile.hpp, or neither - the k-split
// kernel where it applies (k a multiple of 256) and one thread per output otherwise.
// ---------------------------------------------------------------------------------------------

enum W4A8Route
{
    W4A8_OTHER,
    W4A8_FEW_ROW,
    W4A8_TILE_256X256,
    W4A8_TILE_128X128,
    W4A8_TILE_64X128,
    W4A8_TILE_32X128
};

// Every tile is one pass of a CU over k, so a launch costs ceil(tiles / 256) times (fixed + stages *
// rate) of its tile; the rates are microseconds measured on MI355X at k 864 and 4096 (M x N tiles:
// 256 x 256 82 us for one round of 256 at k 4096, 128 x 128 23, 64 x 128 14.7, 32 x 128 11.7), and the
// cheapest wins: 1000 x 11008 x 4096 takes 128 x 128 tiles (69 us; 74 with 256 x 256, 79 with 64 x
// 128, 108 with 32 x 128), 512 x 4096 x 4096 64 x 128 (18.3; 25.7, 21.6 with 32 x 128), 4096^3 256 x
// 256 (82; 97).
struct W4A8Tile
{
    W4A8Route route;
    int bm, bn, threads;
    float fixed, stage;  // us per round: fixed + stage * ceil(k / 128)
};
constexpr W4A8Tile kW4A8Tiles[] = {{W4A8_TILE_256X256, 256, 256, 512, 18.0f, 2.0f},
                                   {W4A8_TILE_128X128, 128, 128, 256, 5.0f, 0.57f},
                                   {W4A8_TILE_64X128, 64, 128, 256, 4.5f, 0.32f},
                                   {W4A8_TILE_32X128, 32, 128, 256, 4.0f, 0.24f}};

// Microseconds of the cheapest tile, and which it is; 0 where no tile's grid fits.
inline float w4a8_tile_us(long long M, long long N, long long K, W4A8Route &best)
{
    const float stages = static_cast<float>(ceil_div(K, 128));
    float best_us = 0.f;
    for (const W4A8Tile &p : kW4A8Tiles) {
        const long long tiles = ceil_div(M, p.bm) * ceil_div(N, p.bn);
        if (!grid_fits(tiles + 8, p.threads)) {
            continue;
        }
        const float us = static_cast<float>(ceil_div(tiles, kTileCUs)) * (p.fixed + p.stage * stages);
        if (best_us == 0.f || us < best_us) {
            best = p.route;
            best_us = us;
        }
    }
    return best_us;
}

// Whether the few-row kernel is faster than the k-split kernel (k a multiple of 256, up to 32 rows).
// Both give 16 channels (a strip) to a workgroup of eight waves that split k. The k-split kernel
// requests all of a wave's weights at once, one pass per 15 rows, and stages up to 15 rows of all of
// k in LDS; the few-row kernel keeps one or two blocks of 256 k in flight per wave and reads the
// weights once for 32 rows. Measured on MI355X with each layer's weights from HBM, 110 shapes of 4 to
// 1813 strips and k 256 to 16128 (few-row, k-split, us):
//   up to 8 rows
//     k to 1024: few-row (2 x 16384 x 512 3.8, 4.5; 4 x 1024 x 1024 2.5, 2.6)
//     k to 2048: few-row, but k-split to four rows and two strips a CU (2 x 2048 x 2048 3.4, 3.1; 2 x
//       18720 x 1792 1.12 times faster in few rows)
//     k to 4096: k-split, whose one or two loads a wave are all in flight (8 x 4096 x 4096 4.6, 4.3; 2 x
//       11008 x 4096 6.4, 6.1; 2 x 6272 x 2816 5.2, 4.4), but few-row over three strips a CU to k 3072
//       (8 x 15712 x 3072 7.5, 8.2)
//     longer k, strips that leave CUs idle: few-row (2 x 896 x 13824 5.5, 6.6; 8 rows 5.9, 8.8), but
//       k-split for one row to k 8192 (1 x 272 x 4608 3.5, 3.3)
//     longer k, more strips: the k-split kernel while two of its workgroups share a CU (1 x 8192 x 8192
//       9.8, 7.8; 8 rows 9.9, 9.1; 2 x 5120 x 13824 11.2, 10.0), the few-row kernel where its staged
//       rows no longer let them (8 x 5120 x 13824 12.9, 15.3; 8 x 17648 x 9472 1.4 times faster; 4 x
//       9008 x 11264 12.5, 14.0) or it runs over two strips a CU with five rows and more (8 x 12080 x
//       4608 1.2 times)
//   9 to 16 rows: few-row (12 x 6352 x 4608 7.1, 8.5), but 9 x 8192 x 8192 11.3, 10.2
//   17 to 32 rows, where the k-split kernel makes two or three passes: few-row (32 x 11008 x 4096 13.1,
//     19.2), but k-split where its passes fit a workgroup a CU (17 x 1280 x 3840 4.7, 4.2) and for
//     short k (24 x 2048 x 2048 4.2, 3.6; 17 x 16384 x 512 8.9, 7.2), three passes over more than a
//     strip a CU aside (32 x 7616 x 1280 5.9, 7.4)
inline bool w4a8_few_row_beats_ksplit(long long M, long long N, long long K)
{
    const long long strips = ceil_div(N, 16);
    if (M <= 8) {
        if (K <= 2048) {
            return K <= 1024 || M > 4 || strips > 2 * kTileCUs;
        }
        if (K <= 4096) {
            return K <= 3072 && strips > 3 * kTileCUs;
        }
        if (strips <= 224) {
            return M > 1 || K > 8192;
        }
        if (K > 8192) {
            return strips <= 256 || M >= 5 || (M == 4 && strips > 512);
        }
        return M >= 5 && strips > 512;
    }
    if (M <= 16) {
        return !(M <= 10 && K > 6144 && K <= 8192 && strips > 224 && strips <= 512);
    }
    const long long passes = ceil_div(M, 15);
    if (K > 4096) {
        return true;
    }
    if (K > 2048) {
        return strips * passes > 256;
    }
    return passes == 3 && K >= 1024 && strips > 224 && strips <= 512;
}

// Plain operands in the tile kernels' layout. ksplit: the k-split kernel applies (else one thread per
// output is the alternative, which both others beat but for more than 32 rows of one 32-k group: 33 x
// 700 x 32 4.1 us, in tiles 4.8).
// The few-row kernel against the tiles, past 8 rows: the activations weigh as much as the weights and
// each strip reloads them (16 x 28672 x 8192 26.7 us, 24 in tiles; 32 x 28672 x 8192 35, 24).
// The k-split kernel against the tiles: one pass over the weights per 15 rows, 3.2 us + 0.115 us per
// 10^6 weights and pass (11008 x 4096: 12.6 us at 16 rows, 18.5 at 32, 23.0 at 48, against 12.2-12.8
// in tiles; 4096 x 4096: 9.7 at 48 and 27.1 at 200, against 12.5 and 12.8).
inline W4A8Route w4a8_route(long long M, long long N, long long K, bool ksplit)
{
    W4A8Route tile = W4A8_OTHER;
    const float tile_us = w4a8_tile_us(M, N, K, tile);
    const long long strips = ceil_div(N, 16);
    if (M <= 32 && grid_fits(strips, 512) && (!ksplit || w4a8_few_row_beats_ksplit(M, N, K))) {
        const float rate = (M > 16 ? 2.3f : 1.5f) / 4096.f;
        const float us = 3.4f + rate * static_cast<float>(ceil_div(strips, kTileCUs)) *
                                    static_cast<float>(K);
        if (M <= 8 || us <= tile_us) {
            return W4A8_FEW_ROW;
        }
    }
    // (up to 8 rows a pass costs the k-split kernel 0.08 us per 10^6 weights: never in tiles)
    if (tile_us == 0.f || (ksplit && M <= 8) || (M > 32 && K <= 32 && M * N <= 65536) ||
        (ksplit && 3.2f + 0.115e-6f * static_cast<float>(N) * static_cast<float>(K) *
                              static_cast<float>(ceil_div(M, 15)) <= tile_us)) {
        return W4A8_OTHER;
    }
    return tile;
}

// ---------------------------------------------------------------------------------------------
// W8A8 with B = [n, k], static and per-row quantized ("dynamic") activations, plain or packed operands.
// ---------------------------------------------------------------------------------------------

// Whether the few-row kernel (int8_skinny.hpp; 16 channels and 32 rows a workgroup) is faster than what
// takes the shape otherwise: the stream kernel (k a multiple of 128), or the double-buffered one. Both
// sides in microseconds, fitted on MI355X with each layer's weights from HBM over 45 shapes of 128 to
// 2048 strips of 16 channels, k 64 to 14336, and 9 row counts to 32 (the pick is within 6% of the
// better one but for a few points, at most 18%; always the few-row kernel was up to 97% slower):
//   few-row: a workgroup's fixed part and its share of k, by rounds of 256 of them, more with the
//     activation rows that every strip loads too (f32 results: 8 x 4096 x 4096 6.4 us, 16.8 in the
//     stream kernel; static: 1 x 11008 x 4096 11.6, 15.6; 32 x 11008 x 4096 15.9, 17.5)
//   stream kernel: a serial walk over k of 128-channel tiles, then their number and the bytes of the
//     weights (static: 9 x 16384 x 512 5.0, few-row 6.7; 16 x 23232 x 128 4.6, 8.4; 32 x 28672 x 8192 51, 63)
// Past 32 rows every 32 rows are a pass over the weights, about 4 us + 0.29 us per 10^6 weights and
// pass and no less than a workgroup's fixed part, against 3 us + 0.5 us per 128 of k for each round of
// the stream kernel's 64-row tiles (64 x 4096 x 4096 11.5 us, 19.5; 65 x 23232 x 128 20.6, 5.8).
inline bool w8a8_few_row(long long M, long long N, long long K, bool dyn, bool packed)
{
    const long long strips = ceil_div(N, 16);
    const long long passes = ceil_div(M, 32);
    if (passes > 4 || K <= 0 || !grid_fits(strips, 512)) {
        return false;
    }
    const float rounds = strips < kTileCUs ? 1.f : static_cast<float>(strips) / kTileCUs;
    const float mw = 1e-6f * static_cast<float>(N) * static_cast<float>(K);
    if (passes > 1) {
        const float by_bytes = 4.0f + 0.29f * mw * static_cast<float>(passes);
        const float by_count = 2.2f + rounds * static_cast<float>(passes);
        const float stream = static_cast<float>(ceil_div(ceil_div(M, 64) * ceil_div(N, 128), kTileCUs)) *
                             (3.0f + 0.5f * static_cast<float>(K) / 128.0f);
        return (by_bytes > by_count ? by_bytes : by_count) <= stream;
    }
    const float rows = static_cast<float>(M);
    const float fixed = (M <= 8 ? 0.66f : 1.0f) + (dyn ? 0.2f : 0.f);
    const float rate = (M <= 8 ? 2.55f : (M <= 16 ? 2.95f : 3.6f)) * (packed ? 1.05f : 1.f);
    const float few = 2.2f + rounds * (fixed + rate * static_cast<float>(K) / 4096.f);
    const float tiles = static_cast<float>(ceil_div(N, 128)) / kTileCUs;
    const float stages = static_cast<float>(ceil_div(K, 128));
    float other;
    if (K % 128 == 0) {
        other = dyn ? 2.95f + 0.36f * stages + 2.6f * tiles + 0.067f * mw + 0.075f * rows
                    : 2.9f + 0.28f * stages + 1.5f * tiles + 0.078f * mw + 0.02f * rows;
    } else {
        other = dyn ? 3.9f + 0.8f * stages + 2.6f * tiles + 0.0124f * mw + 0.14f * rows
                    : 4.1f + (packed ? 0.6f : 0.75f) * stages + 1.6f * tiles + 0.025f * mw + 0.12f * rows;
    }
    const float by_bytes = 2.f + mw / (dyn ? 4.3f : 4.9f);
    return few < (other > by_bytes ? other : by_bytes);
}

// Which large tile (w8a8_tile.hpp) takes a shape, if any. Rounds of 256 tiles, one per CU (the 128 x 128
// tiles also two: a pair of rounds), in microseconds of fixed + rate * ceil(k / 128), measured on MI355X
// at k 512, 4096 and 11008 with requantized (per-row dynamic, f32) results:
//   stream kernel 128 x 128   3 + 0.67 n (3 + 1.0 n)
//   128 x 128                 4 + 0.7 n (6 + 0.9 n), a pair 5 + 1.2 n (6 + 1.5 n)
//   256 x 256                 14 + 1.5 n (20 + 1.8 n); the MFMAs alone are 1.37 n at the clock the
//                             chip holds under them, the fixed part is the launch, the first loads
//                             and 6 us of requantization that nothing overlaps
// 4000 x 11008 x 4096 runs 256 x 256 tiles in 179 us (218 with 128 x 128, 255 on the stream kernel),
// 2048 x 4096 x 11008 128 x 128 tiles in 95 (114), 2000 x 4096 x 4096 dynamic f32 in 53 (66); one
// round, as 1000 x 4096 x 4096, stays on the stream kernel (24.5 us, 27 with 128 x 128 tiles).
// Requantized results of a short k stay there too: the epilogue is most of such a launch, and the
// stream kernel's overlaps better (2048 x 4096 x 1024 15.1 us, 15.8 in tiles; 551 x 30304 x 128 16.9,
// 20.2; 1201 x 15968 x 128 17.7, 20.0; from k 1280 the tiles win, 313 x 13616 x 1280 14.9, 16.5).
// k not a multiple of 128 has the double-buffered kernel instead of the stream kernel, which one nearly
// full round of large tiles beats too (1000 x 4096 x 4112: 32.1 us, 41.2 there) and a half full one does
// not (512 x 4096 x 4112: 30 us, 27 there), nor tiles half of whose rows are past the last (64 x 32544
// x 3104: 27.9 us, 24.0 there, on 64-row tiles).
enum W8A8Tile
{
    W8A8_NO_TILE,
    W8A8_TILE_128X128,
    W8A8_TILE_256X256
};

inline W8A8Tile w8a8_tile(long long M, long long N, long long K, bool dyn)
{
    const bool other = K % 128 != 0;
    if (K <= 0 || (!dyn && !other && K <= 1024) || (other && M <= 64)) {
        return W8A8_NO_TILE;
    }
    const float n = static_cast<float>(ceil_div(K, 128));
    const long long t128 = ceil_div(M, 128) * ceil_div(N, 128);
    const long long t256 = ceil_div(M, 256) * ceil_div(N, 256);
    const long long r128 = ceil_div(t128, kTileCUs);
    const float stream_us = static_cast<float>(r128) *
                            (other ? 3.f + 1.2f * n : (dyn ? 3.f + 1.0f * n : 3.f + 0.67f * n));
    const float mid_us = static_cast<float>(r128 / 2) * (dyn ? 6.f + 1.5f * n : 5.f + 1.2f * n) +
                         static_cast<float>(r128 % 2) * (dyn ? 6.f + 0.9f * n : 4.f + 0.7f * n);
    const float big_us =
        static_cast<float>(ceil_div(t256, kTileCUs)) * (dyn ? 20.f + 1.8f * n : 14.f + 1.5f * n);
    if (!grid_fits(t256 + 8, 512) || !grid_fits(t128 + 8, 256) ||
        t128 <= (other ? 3 * kTileCUs / 4 : kTileCUs) || (stream_us <= mid_us && stream_us <= big_us)) {
        return W8A8_NO_TILE;
    }
    return big_us < mid_us ? W8A8_TILE_256X256 : W8A8_TILE_128X128;
}

// ---------------------------------------------------------------------------------------------
// Int8 products and convolutions off the 16-byte grid: 64 x 64 MFMA tiles (int8_edge.hpp) or one thread
// per output, which finishes a short k before a stage is staged.
// ---------------------------------------------------------------------------------------------

enum EdgeForm
{
    EDGE_NK,          // B = [n, k], requantized
    EDGE_KN_CLAMP,    // B = [k, n], int32 results
    EDGE_KN_REQUANT,  // B = [k, n], requantized
    EDGE_CONV         // channel-last implicit convolution (M pixels, N channels)
};

// Whether the tiles are faster. Microseconds of both on MI355X, fitted over M 1 to 512, N 15 to 4097, k
// 1 to 200 and 273 convolutions of 1 to 40 channels and 1 to 49 taps, the pick never over 26% from the
// better one:
//   a thread per output: a launch and k steps of one thread, more once the outputs fill the chip (64 x
//     64 x 44 5.5 us, in tiles 9.9; 200 x 4097 x 33 requantized 31.9, in tiles 8.5)
//   tiles: a launch, the epilogue of up to 64 rows and, for a k that ends inside a 16-byte load, its last
//     bytes one by one (64 x 255 requantized: k 33 8.2, k 41 9.7); more where every row has a multiplier
//     of its own (64 x 255 x 81 12.8, a thread per output 10.8); a convolution's taps byte by byte
//     (28 x 28 x 3 to 32, 3 x 3, 12.9, a thread per output 7.5; 112 x 112 x 3 to 96 14.3, 31.8)
inline bool int8_edge_faster(EdgeForm form, long long M, long long N, long long K, long long taps)
{
    const float outs = static_cast<float>(M) * static_cast<float>(N);
    const float tiles = static_cast<float>(ceil_div(M, 64)) * static_cast<float>(ceil_div(N, 64));
    const float k = static_cast<float>(K);
    const float rows = M < 64 ? static_cast<float>(M) : 64.f;
    const float tail = static_cast<float>(K % 16);
    auto larger = [](float a, float b) { return a > b ? a : b; };
    float thread_us, tile_us;
    switch (form) {
    case EDGE_NK:
        thread_us = 2.7f + k * larger(0.066f, (K <= 32 ? 0.75e-6f : 1.15e-6f) * outs);
        tile_us = 4.9f + 0.05f * rows + 0.16f * tail + 0.003f * tiles;
        break;
    case EDGE_CONV:
        thread_us = 4.f + 0.065f * k + 0.2f * static_cast<float>(taps) +
                    1e-6f * outs * (3.f + 0.5f * k + 0.5f * static_cast<float>(taps));
        tile_us = 12.f + tiles * (0.009f + 0.00013f * k);
        break;
    default:
        thread_us = 2.3f + k * larger(N < 64 ? 0.07f : 0.1f, 0.28e-6f * outs);
        tile_us = (form == EDGE_KN_CLAMP ? 4.6f + 0.028f * rows : 4.9f + 0.105f * rows) + 0.02f * k +
                  0.1f * tail + 0.003f * tiles;
    }
    return tile_us < thread_us;
}

// ---------------------------------------------------------------------------------------------
// Channel-first implicit convolution (conv_cf.hpp).
// ---------------------------------------------------------------------------------------------

// An input row position inside its plane: 0 .. IH.
constexpr int cf_clamp_row(int row, int IH)
{
    return row < 0 ? 0 : (row > IH ? IH : row);
}

// Input rows that a tile of `pix` consecutive output pixels needs at most: it touches d + 1 output rows,
// starting at any row oh of a plane. `ext`: input rows between a window's first and one past its last.
// Rows whose last one lies in the same plane: the difference of two clamped positions, c rows apart, is
// a trapezoid over the first position oh * SH - PH, so its largest value lies at a row beside an end of
// the flat part. Rows that reach the next plane: at most d, one by one. (A walk over all output rows
// took 11 us of host time per call at 4096 of them, also where the call was then refused.)
inline long long cf_halo_rows(int OH, int OW, int IH, int SH, int PH, int ext, int pix)
{
    const int d = (pix - 1 + OW - 1) / OW;
    long long most = 0;
    auto take = [&](int oh) {
        const int last = oh + d;
        const long long rows = static_cast<long long>(last / OH) * IH +
                               cf_clamp_row((last % OH) * SH - PH + ext, IH) -
                               cf_clamp_row(oh * SH - PH, IH);
        most = rows > most ? rows : most;
    };
    const int same = OH - d;  // rows 0 .. same - 1 end in their own plane
    if (same > 0 && SH > 0) {
        const long long c = static_cast<long long>(d) * SH + ext;
        for (long long x : {0ll, IH - c}) {
            const long long oh = (x + PH) / SH - (x + PH < 0 ? 1 : 0);
            for (long long r : {oh, oh + 1}) {
                take(static_cast<int>(r < 0 ? 0 : (r > same - 1 ? same - 1 : r)));
            }
        }
    } else if (same > 0) {
        take(0);  // every row reads the same input rows
    }
    for (int oh = same > 0 ? same : 0; oh < OH; ++oh) {
        take(oh);
    }
    return most;
}

// ---------------------------------------------------------------------------------------------
// W4A16
// ---------------------------------------------------------------------------------------------

// Scale block of the 32-k block kb, bdiv 32-k blocks to a scale block: kb / bdiv by the rounded-up
// reciprocal inv = ceil(2^32 / bdiv). With inv * bdiv = 2^32 + e, 0 <= e < bdiv, the product kb * inv
// exceeds kb * 2^32 / bdiv by kb * e / bdiv, so the quotient is exact while kb * bdiv <= 2^32. bdiv
// 65537, kb 65536 is the first pair past that line that is wrong.
constexpr uint32_t scale_block_inverse(uint32_t bdiv)
{
    return static_cast<uint32_t>((0x100000000ull + bdiv - 1) / bdiv);
}

constexpr uint32_t scale_block_of(uint32_t kb, uint32_t bdiv, uint32_t inv)
{
    return bdiv == 1 ? kb : static_cast<uint32_t>((static_cast<uint64_t>(kb) * inv) >> 32);
}

// Whether the few-row kernel's scale indexes are exact over k (bl and k multiples of 32).
constexpr bool w4a16_skinny_scales_exact(long long k, long long bl)
{
    return (k / 32) * (bl / 32) <= 0x100000000ll;
}

enum W4A16Other  // what takes a shape beside the few-row and the tile kernels
{
    W4A16_GENERIC,   // one thread per output
    W4A16_REGISTER,  // w4a16_mfma_kernel: 32-wide blocks, k % 128 == 0, k <= 4096
    W4A16_CHUNK      // w4a16_chunk_kernel: 32-wide blocks, k % 512 == 0
};

enum W4A16Kernel
{
    W4A16_OTHER,
    W4A16_FEW_ROW,
    W4A16_TILE_128X256,
    W4A16_TILE_128X128,
    W4A16_TILE_64X128,
    W4A16_TILE_32X64
};

struct W4A16Route
{
    W4A16Kernel kernel;
    int comp;  // tiles: blocks per compensation of the f32 accumulators, 0 for plain ones
};

// A tile launch is rounds of 256 tiles, one per CU, of fixed + rate * ceil(k / 128) microseconds; the
// 4-wave tiles also run two to a CU (a pair of rounds at a cost of its own). Measured on MI355X at
// k 4096 (32 stages), per round of 256 tiles; pair in parentheses:
//                     32-wide blocks   64-wide    compensated every two 32-wide blocks
//   128 x 256         110              80
//   128 x 128         58               50
//   64 x 128          35 (64)          33 (51)    49 (78)
//   32 x 64           18 (25)          16 (24)    24 (31)
struct W4A16Tile
{
    W4A16Kernel kernel;
    int bm, bn, threads;
    float fixed, stage;            // us of one round
    float pair_fixed, pair_stage;  // us of two
};
constexpr W4A16Tile kW4A16Tiles32[] = {{W4A16_TILE_128X256, 128, 256, 512, 9.f, 3.1f, 18.f, 6.2f},
                                       {W4A16_TILE_128X128, 128, 128, 512, 6.f, 1.6f, 12.f, 3.2f},
                                       {W4A16_TILE_64X128, 64, 128, 256, 4.5f, .95f, 5.f, 1.85f},
                                       {W4A16_TILE_32X64, 32, 64, 256, 4.2f, .44f, 5.f, .61f}};
constexpr W4A16Tile kW4A16Tiles64[] = {{W4A16_TILE_128X256, 128, 256, 512, 9.f, 2.2f, 18.f, 4.4f},
                                       {W4A16_TILE_128X128, 128, 128, 512, 6.f, 1.4f, 12.f, 2.8f},
                                       {W4A16_TILE_64X128, 64, 128, 256, 4.5f, .9f, 5.f, 1.45f},
                                       {W4A16_TILE_32X64, 32, 64, 256, 4.2f, .38f, 5.f, .58f}};
// (the registers of the two larger tiles do not suffice for compensated accumulators)
constexpr W4A16Tile kW4A16TilesComp[] = {{W4A16_TILE_64X128, 64, 128, 256, 4.5f, 1.4f, 5.f, 2.4f},
                                         {W4A16_TILE_32X64, 32, 64, 256, 4.2f, .6f, 5.f, .8f}};

// Blocks per compensation of the tiles' f32 accumulators with 32-wide blocks. A plain accumulator adds
// k / 32 terms; the chunk-stream kernel's sixteen waves add k / 512 each and meet in f64, the register
// kernel's eight k / 256. Relative error against 64 bits, in 1e-8, and microseconds at 1024 x 4096
// rows and channels:
//   k                      640    1024   2048   3968   4096   8192   11264
//   chunk / register       6.6    4.8    5.4    9.6    6.5    8.2    9.3
//   plain                  8.6   10.6   14.7   20.2   20.5   28.8   33.7    (k 4096: 60 us)
//   every block            4.5 at every k
//   every 2 blocks         5.1    5.0    5.0    4.9    4.9    4.9    4.9    (78)
//   every 4                5.7    5.7    5.6    5.6    5.6    5.5    5.5    (70)
//   every 8                6.5    6.7    6.7    6.6    6.7    6.6    6.6    (65)
// f32 results keep within every one or two blocks; f16 results take the widest step whose sums are no
// further off than those of the kernel that takes the shape otherwise (where that is one thread per
// output, whose chain is longer than a tile's, plain accumulators).
constexpr int w4a16_compensation(long long K, bool f32, W4A16Other other)
{
    if (f32) {
        return K < 1536 ? 1 : 2;
    }
    if (other == W4A16_CHUNK) {
        return K < 1536 ? 1 : (K < 3072 ? 2 : (K < 5120 ? 4 : 8));
    }
    return other == W4A16_REGISTER ? (K < 640 ? 4 : 8) : 0;
}

// Microseconds of the chunk-stream and register kernels: every 32 rows are a pass of their own over the
// weights. The register kernel's, with 16 rows: 4096 x 640 8.2, 1280 x 3840 11.2, 14784 x 256 10.4,
// 19472 x 896 14.5.
inline float w4a16_other_us(long long M, long long N, long long K, W4A16Other other)
{
    const long long ntiles = ceil_div(N, 16);
    const long long row_groups = ceil_div(M, 32);
    const float k = static_cast<float>(K);
    if (other == W4A16_CHUNK) {
        const long long wgs = ntiles <= kTileCUs ? ntiles : ceil_div(ntiles, 4);
        const long long nwg = ntiles > kTileCUs && wgs < kTileCUs ? kTileCUs : wgs;
        return static_cast<float>(ceil_div(row_groups * nwg, kTileCUs)) *
               (3.5f + 0.97f * static_cast<float>(K / 512));
    }
    const long long gx = ntiles < kTileCUs ? ntiles : kTileCUs;
    const float tiles = static_cast<float>(ntiles) / static_cast<float>(gx);  // per workgroup
    return static_cast<float>(ceil_div(row_groups * gx, kTileCUs)) *
           (3.5f + 1.4f * tiles + k * (0.0008f + 0.0006f * tiles));
}

// Microseconds of the few-row kernel, 0 where it does not apply: a fixed part and the 16-channel strips
// that one CU streams, more slowly with the activation rows that each strip loads too (load blocks for
// 2, 8 or 16 rows). At k 4096 and one row: 256 strips 6.3, 512 8.7, 688 10.1, 896 12.6; 1792 strips at
// k 8192 32; with 8 rows 6.3, 688 strips 11.8, 1792 at k 8192 36; with 12 rows 6.9, 14.2 and 41. More
// than 16 rows, a group of 16 each, only where one thread per output is the alternative (26 x 1152 x
// 11008 in 128-wide blocks 11.7, 36.8 in tiles): the 32-row kernels read the weights once.
inline float w4a16_few_row_us(long long M, long long N, long long K, long long bl, W4A16Other other)
{
    const long long ntiles = ceil_div(N, 16);
    if (M > (other == W4A16_GENERIC ? 64 : 16) || K < 128 || !w4a16_skinny_scales_exact(K, bl) ||
        !grid_fits(ntiles, 512)) {
        return 0.f;
    }
    const float rounds = static_cast<float>(ceil_div(ntiles * ceil_div(M, 16), kTileCUs));
    const float rows = static_cast<float>(M < 16 ? M : 16);
    const float by_rows = M <= 2 ? 1.f : (M <= 8 ? 1.1f + 0.015f * rows : 1.27f + 0.02f * rows);
    const float round_us = 1.95f / 4096.f * static_cast<float>(K) * by_rows;
    return 4.2f + rounds * (M > 8 && round_us < 0.95f ? 0.95f : round_us);
}

// Plain layouts that the tile kernels take (16-byte aligned rows, whole 32-k groups per block).
inline W4A16Route w4a16_route(long long M, long long N, long long K, long long bl, bool f32,
                              W4A16Other other)
{
    const bool other_kernel = other != W4A16_GENERIC;  // a 32-row kernel has the shape otherwise
    const float other_us = other_kernel ? w4a16_other_us(M, N, K, other) : 0.f;
    W4A16Route tile = {W4A16_OTHER, bl % 64 == 0 ? 0 : w4a16_compensation(K, f32, other)};
    float tile_us = 0.f;
    // Under a stage of k and few outputs one thread each takes a few microseconds and sums in the
    // oracle's order; one chunk of k with f32 results: the chunk-stream kernel's sixteen f64-summed
    // blocks are the more exact (4.5e-8 against 4.7e-8).
    if (!(K < 128 && M * N <= 65536) && !(f32 && K == 512 && other_kernel)) {
        const float stages = static_cast<float>(ceil_div(K, 128));
        // microseconds a stage against those of a compensation every two blocks
        const float scale = tile.comp == 0 || tile.comp == 2
                                ? 1.f : (tile.comp == 1 ? 1.4f : (tile.comp == 4 ? 0.89f : 0.82f));
        auto consider = [&](const W4A16Tile &p) {
            const long long tiles = ceil_div(M, p.bm) * ceil_div(N, p.bn);
            if (!grid_fits(tiles + 8, p.threads)) {
                return;
            }
            const long long rounds = ceil_div(tiles, kTileCUs);
            const float us =
                static_cast<float>(rounds / 2) * (p.pair_fixed + p.pair_stage * scale * stages) +
                static_cast<float>(rounds % 2) * (p.fixed + p.stage * scale * stages);
            if (tile_us == 0.f || us < tile_us) {
                tile.kernel = p.kernel;
                tile_us = us;
            }
        };
        if (tile.comp > 0) {
            for (const W4A16Tile &p : kW4A16TilesComp) {
                consider(p);
            }
        } else {
            for (int i = 0; i < 4; ++i) {
                consider(bl % 64 == 0 ? kW4A16Tiles64[i] : kW4A16Tiles32[i]);
            }
        }
    }
    const float few_us = w4a16_few_row_us(M, N, K, bl, other);
    // other_us reads low with up to 32 rows, where the weights' stream is most of it (8192 x 8192 19.0,
    // measured 21; 4096 x 11264 24.8, 25.8; 11008 x 4096 11.3, 13.0). Measured with each layer's weights
    // from HBM, few rows and the 32-row kernel: 1 x 4096 x 4096 6.3, 11.9; 1 x 14336 x 4096 12.6, 13.8;
    // 8 x 11008 x 4096 11.8, 13.1; 16 x 8192 x 8192 19.9, 21.1; but 12 x 11008 x 4096 14.2, 13.1; 4 x
    // 14336 x 4096 14.3, 13.7; 9 x 23200 x 512 10.1, 9.2
    if (few_us > 0.f && (!other_kernel || few_us < 1.09f * other_us) &&
        (tile_us == 0.f || few_us < tile_us)) {
        return {W4A16_FEW_ROW, 0};
    }
    if (tile_us > 0.f && (!other_kernel || tile_us < (f32 || M <= 32 ? 1.f : 1.08f) * other_us)) {
        return tile;
    }
    return {W4A16_OTHER, 0};
}

}  // namespace tqt
