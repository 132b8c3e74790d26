// Which kernel, and which of its tiles, a dense product of M x N results and K inputs takes.  Plain C++: a test on the host
// asks the same rules.
#pragma once

namespace et {

// Tile choice: the form with the least time by what each was measured to take, in ns: `start` and `depth` per 64 of depth once,
// `round` and `stage` per 64 of depth for every workgroup a compute unit gets (256 units).  Fitted to 123 Linears of 16..8192
// rows, 208..4096 wide, multiples of 16 and of 64, with and without GELU, eight sets of buffers in turn: each
// form within 9-15 % of its time, the choice 1.1 % slower than the best form in the mean (19 % at worst, 8192 x 256 -> 1024).
// Against forms with one slice of fragments ahead, activations chosen per value and loads past the end (us, mean of no
// activation and GELU): 2048 x 768 -> 3072 20.7 -> 16.0 (128 x 192 tiles), 768 8.8 -> 7.5 and 2048 x 3072 -> 768 22.3 -> 18.2 (128 x 64),
// 4096 x 3072 -> 768 40.6 -> 32.0 (64 x 192), 8192 x 3072 -> 768 62.6 -> 47.6, 2048^3 27.9 -> 22.8 (128 x 128), 528 x 768 -> 3072 11.1 -> 7.9,
// 1024 x 4096^2 62.2 -> 42.0.  Two buffers, several workgroups to a unit, where a short depth leaves mostly epilogues: 6448 x 1568 ->
// 1040 54.9 -> 35.6 (41.1 with four).  128 x 192 tiles with a fourth buffer, which take all of the LDS, and 128 x 256 with eight waves were up
// to 40 % slower on operands out of the caches than in them (2048 x 384 -> 3072 10.2 and 14.8, this form 10.8).
struct DmaTile { int tmw, tnw, nbuf; bool ragged; };
struct DmaForm { int tmw, tnw, nbuf, start, depth, round, stage; };  // tiles of 64 tmw x 64 tnw
constexpr int kDmaK = 64;  // K per stage: one 128-byte line of every row
constexpr DmaForm kDmaForms[] = {
    {1, 1, 4, 2000, 30, 1150, 209}, {2, 1, 4, 250, 0, 3250, 330}, {1, 2, 4, 200, 0, 3300, 336}, {2, 2, 4, 0, 0, 4800, 490},
    {1, 3, 4, 0, 0, 4400, 430},     {2, 3, 3, 0, 0, 6100, 605},   {2, 2, 2, 900, 300, 2600, 440}, {2, 1, 2, 1500, 340, 1300, 275},
    {4, 4, 4, 0, 0, 8200, 1220},
};
inline bool pick_dma_tile(int M, int N, int K, int batch, bool trans_b, DmaTile *out) {
    if (M % 16 || N % 16 || K % 16) return false;
    if (batch != 1 || !trans_b) {
        // Batched problems and B stored k-major run on 64 x 64 tiles where they are
        // bound by the latency of a long K loop in few workgroups (the stacked VO product of the
        // pre-computed-VO attention: 32 -> 22 us); gathering the k-major fragments with 2-byte LDS
        // reads costs more than it saves elsewhere (Linear_VO 28 -> 78 us), those stay on the
        // register-staged kernel.
        const long long w = (long long)((M + 63) / 64) * ((N + 63) / 64) * batch;
        if (w > 256 || K / kDmaK < 16) return false;
        *out = {1, 1, trans_b ? 4 : K / kDmaK < 24 ? 2 : 3, true};
        return true;
    }
    // So many tiles of 256 x 256 that their last round hardly counts, but not all of them whole (the form of whole ones is among those
    // below): four waves of 128 x 128 (16368 x 8192^2 1980 us against 2380 in tiles of 128 x 192, 8176^3 1134 / 1400; 512 such
    // tiles, 8176 x 4080^2, 330 / 325).  Edges of 64 are whole in the smaller tiles, which a short depth then leaves ahead: 16320 x 8192^2 1850 /
    // 2300, 8128 x 4096 -> 8192 484 / 592, 16320 x 256 -> 4096 60 / 64, of 64 inputs 38.5 / 36.8.
    const bool ragged64 = M % 64 || N % 64 || K % kDmaK, ragged256 = M % 256 || N % 256;
    if ((ragged64 || (ragged256 && K >= 256)) && (long long)((M + 255) / 256) * ((N + 255) / 256) >= 1024) {
        *out = {4, 4, 2, true};
        return true;
    }
    long long best = -1;
    const long long stages = (K + kDmaK - 1) / kDmaK;
    for (const DmaForm &f : kDmaForms) {
        const int bm = 64 * f.tmw, bn = 64 * f.tnw;
        const bool whole = M % bm == 0 && N % bn == 0 && K % kDmaK == 0;
        if (f.tmw == 4 && !whole) continue;  // (written for whole tiles)
        const long long wgs = (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn), rounds = (wgs + 255) / 256;
        const long long ns = f.start + stages * f.depth + rounds * (f.round + stages * f.stage);
        if (best < 0 || ns < best) {
            best = ns;
            *out = {f.tmw, f.tnw, f.nbuf, !whole};
        }
    }
    return true;
}

// The small-result kernel applies when 64 x 64 tiles would leave most of the chip idle: up to 1024 tiles of 16 x 16, from a depth of
// 784 on up to 640 (us, this kernel / the direct-to-LDS kernel: 672 tiles of 704 4.5 / 5.6, 990 of 528 5.4 / 6.0, 513 of 1056 6.5 / 7.7, 558
// of 2096 10.2 / 12.3, 384 of 3072 8.5 / 13.8; 1043 of 864 9.3 / 7.3, 860 of 1632 12.9 / 9.7, 1536 of 768 6.8 / 6.1, 1760 of 320
// 4.9 / 4.6).  Operands that kernel does not take (a result off its alignment, as
// a row-pruned Linear may be given) would fall to the register-staged kernel, so there the line lies at 2048: 512 x 3072 -> 528 scattered
// 20.0 / 37.4, 1024 x 1536 -> 448 14.3 / 23.1, 1024 x 4096 -> 448 29.2 / 46.7.  (Batched problems do not come near it:
// with more than 640 tiles each, four of them have more than 128 of 64 x 64.)
inline bool takes_small_result(int M, int N, int K, int batch, bool dma_applies) {
    const long long tiles64 = (long long)((M + 63) / 64) * ((N + 63) / 64) * batch;
    const long long tiles16 = (long long)(M / 16) * (N / 16);
    return K >= 256 && tiles64 < 128 && tiles16 <= (!dma_applies ? 2048 : K > 768 ? 640 : 1024);
}

}  // namespace et
