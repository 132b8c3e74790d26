// Asks the rules that choose a kernel's form (csrc/*_forms.h) on the host.  One question a line of the standard input:
//   gemm M N K batch trans_b dma_applies  ->  small | tile TMW TNW NBUF ragged | none
//   lines M N K  ->  TMW TNW NBUF of a ragged problem whose rows begin off a 128-byte line
//   wide S nbh  ->  keys of a block (heads of more than 224)
//   mha HD compact S nbh causal plain lengths z16  ->  in the launcher's order: tiles WAVES SPLIT STEPS (the 32 x 32 kernel) | waves WAVES TILES | turns ragged
#include <cstdio>
#include <cstring>

#include "attention_forms.h"
#include "gemm_forms.h"

int main() {
    char line[256];
    while (fgets(line, sizeof line, stdin)) {
        int m, n, k, batch, trans, dma, padded, z16;  // the numbers, by their names in the first question
        if (sscanf(line, "gemm %d %d %d %d %d %d", &m, &n, &k, &batch, &trans, &dma) == 6) {
            et::DmaTile t{};
            const bool tile = dma && et::pick_dma_tile(m, n, k, batch, trans != 0, &t);
            if (et::takes_small_result(m, n, k, batch, tile)) puts("small");
            else if (tile) printf("tile %d %d %d %d\n", t.tmw, t.tnw, t.nbuf, (int)t.ragged);
            else puts("none");
        } else if (sscanf(line, "lines %d %d %d", &m, &n, &k) == 3) {
            et::DmaTile t{};
            if (et::pick_dma_tile(m, n, k, 1, true, &t) && t.ragged) t = et::dma_lines_tile(t, m, n, k);
            printf("%d %d %d\n", t.tmw, t.tnw, t.nbuf);
        } else if (sscanf(line, "mha %d %d %d %d %d %d %d %d", &m, &n, &k, &batch, &trans, &dma, &padded, &z16) == 8) {
            const bool applies = n == 0 && et::mha_tiles_apply(m, dma != 0, z16 != 0, 0, batch, 1);
            const et::MhaTiles tiles = applies ? et::mha_tiles(m, k, batch, trans != 0, padded) : et::MhaTiles{};
            if (tiles.waves) {
                printf("tiles %d %d %d\n", tiles.waves, tiles.split, tiles.steps);
                continue;
            }
            const et::MhaForm f = et::mha_form(m, n != 0, k, batch, trans != 0, dma != 0, padded != 0);
            if (f.in_turn) printf("turns %d\n", (int)f.ragged);
            else printf("waves %d %d\n", f.waves, f.tiles);
        } else if (sscanf(line, "wide %d %d", &m, &n) == 2) {
            puts(et::mha_wide_blocks(m, n) ? "128" : "64");
        } else {
            fprintf(stderr, "not understood: %s", line);
            return 1;
        }
    }
    return 0;
}
