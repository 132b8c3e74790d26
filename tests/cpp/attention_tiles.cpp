// Asks the rule of the 32 x 32 attention (csrc/attention_forms.h) on the host: HD S nbh causal lengths -> waves split steps a line.
#include <cstdio>

#include "attention_forms.h"

int main() {
    int hd, s, nbh, causal, lengths;
    while (scanf("%d %d %d %d %d", &hd, &s, &nbh, &causal, &lengths) == 5) {
        const et::MhaTiles f = et::mha_tiles(hd, s, nbh, causal != 0, lengths);
        printf("%d %d %d\n", f.waves, f.split, f.steps);
    }
}
