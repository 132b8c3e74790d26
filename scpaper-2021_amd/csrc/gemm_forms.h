// Which kernel, and which of its tiles, a dense product of M x N results and K inputs takes.  Plain C++: a test on the host
// asks the same rules.
#pragma once

namespace et {

// Tile choice: the form with the least time by what each was measured to take, in ns: `start` and `depth` per 64 of depth once,
// `round` and `stage` per 64 of depth for every workgroup a compute unit gets (256 units).  Fitted to 123 Linears of 16..8192
// rows, 208..4096 wide, multiples of 16 and of 64, with and without GELU, eight sets of buffers in turn: each
// form within 9-15 % of its time, the choice 1.1 % slower than the best form in the mean (19 % at worst, 8192 x 256 -> 1024).  The stage
// of 128 x 192 tiles is that of operands too large for the caches: 600 ns within them, 700 to 790 over 3 and more rounds.  At 605 they were taken
// where two workgroups of 128 x 128 to a unit are ahead (us, 128 x 192 and that form: 6000 x 3216 -> 2448 135 and 125, 7104 x 2688 -> 2160 112 and
// 93, 4736 x 2368 -> 3072 92 and 78; 520 Linears of more than 2048 tiles of 16 x 16, 2.3 % slower than the best form in the mean, 1.8 % at 650).
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
    {1, 3, 4, 0, 0, 4400, 430},     {2, 3, 3, 0, 0, 6100, 650},   {2, 2, 2, 900, 300, 2600, 440}, {2, 1, 2, 1500, 340, 1300, 275},
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

// The tile where rows begin off a 128-byte line, whose requests fetch whole lines through four buffers: one workgroup of 128 x 128 or more to a
// compute unit, where the forms above hold two or three.  Time of this over the form above, 220 ragged Linears of 208 to 4080 inputs: forms of four
// buffers 0.79 to 0.98, 128 x 192 0.78 to 0.89.  128 x 128 on two buffers: a tile a unit 0.82 to 0.88 (beyond, with fewer inputs, what two to a
// unit hide weighs more: 0.90 to 1.19 below 944), from 1024 inputs on 0.78 to 1.02, from 944 where the last round is four fifths full 0.88 to 0.98;
// 128 x 192 instead where it saves a round, to three rounds from 448 inputs on 0.78 to 0.81 (304 0.97), more rounds from 880 on 0.83 to 1.00.
// 128 x 64 on two buffers: from 880 inputs on 0.86 to 0.90, below 1.10 to 1.44.
inline DmaTile dma_lines_tile(DmaTile t, int M, int N, int K) {
    if (t.tmw > 2 || t.nbuf == 4) return t;
    auto tiles = [&](int wide) { return (long long)((M + 127) / 128) * ((N + wide - 1) / wide); };
    auto rounds = [&](int wide) { return (tiles(wide) + 255) / 256; };
    if (t.tnw == 3 || (t.tnw == 1 && K >= 880)) t.nbuf = 4;
    if (t.tnw == 2) {
        const long long r2 = rounds(128), r3 = rounds(192);
        if (r2 > 1 && 13 * r3 < 10 * r2 && K >= (r2 <= 3 ? 448 : 880)) t.tnw = 3, t.nbuf = 4;
        else if (r2 == 1 || K >= 1024 || (K >= 944 && 5 * tiles(128) >= 4 * 256 * r2)) t.nbuf = 4;
    }
    return t;
}

// The small-result kernel (one tile of 16 x 16 a workgroup, K in pieces of 64 over its four waves) applies when 64 x 64 tiles would
// leave most of the chip idle: up to 768 tiles of 16 x 16, three workgroups to a compute unit; up to 1024 of at most 768 inputs, three
// pieces a wave, and where the pieces of a wave fill two or more of its rounds of six loads (2817 to 3072 inputs).
// us, this kernel / the direct-to-LDS kernel, operands in turn: 672 tiles of 3072 inputs 10.7 / 15.3, 704 of 1024 5.9 / 6.9, 726 of 1648
// 8.5 / 9.6, 864 of 768 5.4 / 6.0, of 3072 12.9 / 14.4; in the mean of Linears with 640 to 768 tiles 0.96 up to 1536 inputs, 1.01 up to 2560, 0.84
// up to 3072, 0.93 up to 4096; with 768 to 1024 tiles 0.96 of 512 to 768 inputs, 1.08, 1.12 and 1.05 up to 1024, 1280 and 1536, 1.19 up to 2560, 0.96
// of 2817 to 3072, 1.05 beyond; with 1024 to 1280 tiles 1.07 up to 768, 1.15 to 1.5 beyond.
// Several problems: 640 tiles each and more than 768 inputs (2 of 480 x 2048 -> 368 15.7 / 10.6, 3 of 736 x 1248 -> 176 12.0 / 7.9, 2 of
// 192 x 1312 -> 672 7.3 / 7.9; fewer than 1024 inputs the direct-to-LDS kernel does not take).
// The two add in another order (four partial sums, one chain): 0.5 to 1.4e-5 apart in binary16 results, both 2.07e-4 from binary64.
// Operands that kernel does not take (a result off its alignment, as
// a row-pruned Linear may be given) would fall to the register-staged kernel, so there the line lies at 2048: 512 x 3072 -> 528 scattered
// 20.0 / 37.4, 1024 x 1536 -> 448 14.3 / 23.1, 1024 x 4096 -> 448 29.2 / 46.7.
inline bool takes_small_result(int M, int N, int K, int batch, bool dma_applies) {
    const long long tiles64 = (long long)((M + 63) / 64) * ((N + 63) / 64) * batch;
    const long long tiles16 = (long long)(M / 16) * (N / 16);
    const int pieces = ((K + 63) / 64 + 3) / 4;  // of a wave
    const bool full_rounds = K <= 768 || (pieces >= 12 && pieces % 6 == 0);
    const int most = !dma_applies ? 2048 : batch > 1 && K > 768 ? 640 : full_rounds ? 1024 : 768;
    return K >= 256 && tiles64 < 128 && tiles16 <= most;
}

}  // namespace et
