// The prompt GEMM's weight and scale loads over whole grids: how many lie outside the copy, or
// differ from the column and block they stand for where those exist.  The schedule is the
// kernel's: a step's blocks, then at each step the next one's, past the last one too.
#include <cstddef>

#include "jy_gemm_offsets.h"

using namespace jy;

extern "C" long long gemm_offsets_bad(int rows, int cols, int nt_n, int slices) {
    constexpr int KB = 4, WAVES = 4;
    const int tiles = (rows + 15) / 16, nb = cols / 32, nb4 = (nb + 3) / 4;
    const long long qbytes = (long long)tiles * nb * 512, dbytes = (long long)tiles * nb4 * 256;
    const int nbz = (nb + slices - 1) / slices, nct = (tiles + 8 * nt_n - 1) / (8 * nt_n);
    long long bad = 0;
    for (int ct = 0; ct < nct; ct++)
        for (int wave = 0; wave < WAVES; wave++) {
            const int tilet = ct * 8 * nt_n + wave * 2 * nt_n, t0 = gm_base_tile(tilet, tiles);
            for (int z = 0; z * nbz < nb; z++) {
                const int b0 = z * nbz, b1 = b0 + nbz < nb ? b0 + nbz : nb;
                for (int b = b0 / KB * KB; b < b1 + KB; b += KB)  // (each step's blocks, and the next one's)
                    for (int nt = 0; nt < nt_n; nt++)
                        for (int l = 0; l < 64; l++) {
                            const int tile = tilet + 2 * nt + (l & 31) / 16;
                            for (int kb = 0; kb < KB; kb++) {
                                const long long o = (long long)t0 * nb * 512 + gm_q_lane(tilet, nt, l, tiles, nb) +
                                                    gm_q_block(b + kb, nb);
                                bad += o < 0 || o + 16 > qbytes;
                                if (tile < tiles && b + kb < nb)
                                    bad += o != ((long long)tile * nb + b + kb) * 512 + (l % 16) * 16 + 256 * (l / 32);
                            }
                            const long long o = (long long)t0 * nb4 * 256 + gm_d_lane(tilet, nt, l, tiles, nb4) +
                                                gm_d_block(b, nb4);
                            bad += o < 0 || o + 16 > dbytes;
                            if (tile < tiles && b < nb) bad += o != ((long long)tile * nb4 + b / 4) * 256 + (l % 16) * 16;
                        }
            }
        }
    return bad;
}
