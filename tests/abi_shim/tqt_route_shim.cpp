// The dispatch rules of torq-tile_amd/csrc/route.hpp behind C symbols, for the host tests.
#include "route.hpp"

using namespace tqt;

extern "C" {

int tqtr_grid_fits(long long blocks, int threads)
{
    return grid_fits(blocks, threads);
}

int tqtr_w4a8_route(long long m, long long n, long long k, int ksplit)
{
    return w4a8_route(m, n, k, ksplit != 0);
}

int tqtr_w8a8_few_row(long long m, long long n, long long k, int dyn, int packed)
{
    return w8a8_few_row(m, n, k, dyn != 0, packed != 0);
}

int tqtr_w8a8_tile(long long m, long long n, long long k, int dyn)
{
    return w8a8_tile(m, n, k, dyn != 0);
}

int tqtr_int8_edge_faster(int form, long long m, long long n, long long k, long long taps)
{
    return int8_edge_faster(static_cast<EdgeForm>(form), m, n, k, taps);
}

// the kernel, and in hundreds its blocks per compensation
int tqtr_w4a16_route(long long m, long long n, long long k, long long bl, int f32, int other)
{
    const W4A16Route r = w4a16_route(m, n, k, bl, f32 != 0, static_cast<W4A16Other>(other));
    return r.kernel + 100 * r.comp;
}

long long tqtr_cf_halo_rows(int OH, int OW, int IH, int SH, int PH, int ext, int pix)
{
    return cf_halo_rows(OH, OW, IH, SH, PH, ext, pix);
}

// The same by a walk over every output row.
long long tqtr_cf_halo_rows_walk(int OH, int OW, int IH, int SH, int PH, int ext, int pix)
{
    const int d = (pix - 1 + OW - 1) / OW;
    long long most = 0;
    for (int oh = 0; oh < OH; ++oh) {
        const int last = oh + d;
        const long long rows = static_cast<long long>(last / OH) * IH +
                               cf_clamp_row((last % OH) * SH - PH + ext, IH) -
                               cf_clamp_row(oh * SH - PH, IH);
        most = rows > most ? rows : most;
    }
    return most;
}

uint32_t tqtr_scale_block_of(uint32_t kb, uint32_t bdiv)
{
    return scale_block_of(kb, bdiv, scale_block_inverse(bdiv));
}

int tqtr_w4a16_skinny_scales_exact(long long k, long long bl)
{
    return w4a16_skinny_scales_exact(k, bl);
}

// The first 32-k block of k whose scale block the reciprocal gets wrong, or -1.
long long tqtr_first_wrong_scale_block(long long k, long long bl)
{
    const uint32_t bdiv = static_cast<uint32_t>(bl / 32);
    const uint32_t inv = scale_block_inverse(bdiv);
    for (long long kb = 0; kb < k / 32; ++kb) {
        if (scale_block_of(static_cast<uint32_t>(kb), bdiv, inv) != kb / bdiv) {
            return kb;
        }
    }
    return -1;
}

}  // extern "C"
