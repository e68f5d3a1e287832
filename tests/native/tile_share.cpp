// Walks TileShare (wide_layout.h): every super-block of every tile in exactly one part, no workgroup with more than `longest` of them, the two parts of a
// shared tile on one die and at one place there, no place taken twice, row units a permutation.
#include <cstdio>
#include <vector>

#include "wide_layout.h"

using namespace slai::wide;

extern "C" int share_walk(uint32_t units, uint32_t blocks, uint32_t ncb, uint32_t *longest, char *msg, size_t cap) {
    const TileShare share(units, blocks, ncb);
    struct Seen { uint32_t parts = 0, blocks = 0, die = 0, place = 0; };
    std::vector<Seen> tiles(units * blocks);
    *longest = share.longest();
    for (uint32_t die = 0; die < SHARE_DIES; ++die) {
        std::vector<int> places(SHARE_RUNS, -1);
        for (uint32_t run = 0; run < SHARE_RUNS; ++run) {
            uint32_t mine = 0;
            for (uint32_t i = 0; i < share.rounds + share.mains; ++i) {
                const TileShare::Part p = share.part(die, run, i);
                if (!p.any) continue;
                if (p.tile >= tiles.size() || p.c1 > ncb || p.c0 >= p.c1) { snprintf(msg, cap, "die %u run %u part %u: tile %u, %u .. %u", die, run, i, p.tile, p.c0, p.c1); return 1; }
                mine += p.c1 - p.c0;
                Seen &t = tiles[p.tile];
                if (t.parts++ && (t.die != die || t.place != p.place)) { snprintf(msg, cap, "tile %u at two places", p.tile); return 2; }
                t.blocks += p.c1 - p.c0; t.die = die; t.place = p.place;
                if (p.c1 - p.c0 < ncb) {
                    if (p.place >= SHARE_RUNS || (places[p.place] >= 0 && places[p.place] != (int)p.tile)) { snprintf(msg, cap, "die %u: place %u", die, p.place); return 3; }
                    places[p.place] = (int)p.tile;
                }
            }
            if (share.part(die, run, share.rounds + share.mains).any) { snprintf(msg, cap, "die %u run %u: a part past the last", die, run); return 4; }
            if (mine > share.longest()) { snprintf(msg, cap, "die %u run %u: %u super-blocks", die, run, mine); return 5; }
        }
    }
    for (uint32_t t = 0; t < tiles.size(); ++t)
        if (tiles[t].blocks != ncb || tiles[t].parts > 2) { snprintf(msg, cap, "tile %u: %u parts, %u super-blocks", t, tiles[t].parts, tiles[t].blocks); return 6; }
    std::vector<uint32_t> count(units * blocks);
    for (uint32_t t = 0; t < tiles.size(); ++t) {
        const uint32_t u = share.unit(t), b = share.token_block(t);
        if (u >= units || b >= blocks || count[u * blocks + b]++) { snprintf(msg, cap, "tile %u is unit %u, block %u", t, u, b); return 7; }
    }
    return 0;
}
