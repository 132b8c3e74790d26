// Which form of the fused attention a problem takes: waves of a workgroup, 16-query tiles of a wave, the two groups of waves in turn.
// Plain C++: a test on the host asks the same rule.
#pragma once

namespace et {

struct MhaForm {
    int waves, tiles;       // queries of a workgroup: 16 * waves * tiles
    bool in_turn, ragged;   // the two groups of waves in turn (8 waves of two tiles); strips that a sequence ends in
};

// What comes here: few short sequences, additive masks, scales that are not positive, results off 16 bytes, a compact V, heads of more than 224; mha_tiles (below) is asked
// first and takes the others.  The figures of this rule are of problems without a mask.
//
// 4 waves per workgroup and one 16-query tile per wave, whatever the last strip holds: a wave without queries still stages
// its share of every key block.  (Strips of 2 or 1 waves where 4 leave one half-empty, 12 heads of 64, against 4: 16 x 80 keys 6.8
// and 5.8 us, 3 x 176 9.0 and 6.1, 16 x 176 25.4 and 10.1, 16 x 528 126 and 38, 16 x 720 193 and 57; one sequence of 16 to 112 keys 5.6-5.9
// and 4.6-4.8.)
//
// Many short sequences: 2 waves (1 for heads of 32 and 16 keys) where the chip then holds them in fewer rounds.  A compute unit holds
// three workgroups of 4 waves (two with a compact V), four of 2 by the LDS (six for heads of 32 by the registers, four with a compact V), eight of 1.
// us, 4 and fewer: 16 keys, 920 heads of 64 7.5 and 5.9, 1840 13.1 and 11.2, 1536 9.7 and 10.4 (two rounds either way), 1800 heads of 32 6.7 and 4.0;
// 96 keys, 456 heads of 32 7.7 and 6.8; compact, 16 keys, 896 heads of 64 11.8 and 8.0, 96 keys, 300 11.6 and 8.8, 160 keys, 192 0.76 of the time.
// Longer than 32 keys only strips that 4 waves leave half empty, and only where all are there at once (96 keys: up to three rounds of 4, heads of 32 with a
// full V any): 1.05 to 1.2 of the time beyond.  32 keys keep 2 from 512 heads on (768 heads of 40 6.8 and 7.5; 512 to 768 of 64 level), heads of
// 32 with a compact V always (5.6 and 5.7).
//
// Larger workgroups stage each key block for more queries: 8 waves (128 queries) from 256 such workgroups on.  Without a causal mask by
// the workgroups that the fullest compute unit gets: one of 8 waves takes as long as 1.84 of 4 (heads of 64), 1.94 (96), 1.75 (128), and
// a unit works through its own one after the other.  (us, 4 and 8 waves: 8 x 12 heads of 64, 704 keys 26.6 and 29.0 with 3 and 2 a unit, 16 x 16, 128 keys
// 5.7 and 5.1 with 2 and 1, 16 heads, 2048 keys 37.3 and 34.3, 14 x 8 of 128, 1088 keys 120 and 135, 17 x 8 of 128, 640 keys 76 and 68.  Over 700
// problems of 64 to 2048 keys the choice is 0.2 % (64), 0.4 % (96, 128) behind the better one in the mean and 3 to 8 % at worst.  Up to 96 keys, where two
// or three of the 8 waves have no queries, 1.6 for heads of 64: 54 x 16, 96 keys 13.4 and 15.2, 4 a unit and 7; 3 and 5, 66 x 8, 11.5 and 11.8.  128-wide heads with
// one block of keys have no next one to fetch ahead: 8 waves there only where they are one to a unit, 61 x 8 heads, 128 keys 0.94 of their time with 4.
// One workgroup of 8 waves a unit cannot even out sequences of unequal length, two of 4 can: from 449 keys on padded heads of 64 keep 4 there (3 x 12 heads,
// 640 keys 13.6 and 14.5, 24 layers of 4 x 16, 512 keys 1163 and 1172; on operands that stay in the caches 8 are 0 to 9 % ahead).  Padded 128-wide
// heads, which even out over the rounds too: 8 by the strips of a sequence alone (38 x 8, 448 keys 79.5 and 83.0, 39 x 8, 320 keys 52.4 and
// 55.6, 3 x 16, 928 keys 54.0 and 47.5; 134 problems of 80 to 1024 keys 0.3 % behind the better one in the mean, 1.0 % by the fullest unit).)
// Under a causal mask strips differ in length and even out, so what counts is the last strip, the longest one: 8 waves for
// whole strips only, always for 128-wide heads (as against 4: 16 x 8 heads, 256 keys 12.8 and 13.7, 14 x 16, 1216 keys, not whole, 253 and 233), which
// take them also where the last is no emptier than two of 4 and two thirds of the places are taken (10 x 8, 1392 keys 116 and 124),
// never for 96 (25 x 10 heads of 80, 448 keys 51 and 57; whole strips level), for 64 up to two strips a sequence (64 x 12 heads, 128 keys 15.8
// -> 15.3) and where they give a unit one and a half to two and a half (1152 keys, 48 heads 0.88 of the time of 4, 896, 72 heads 0.86, 1280, 64
// heads 0.93; below 1.12 of it, 1152 keys, 36 heads 1.19; above level, 1024, 88 heads 1.18).
//
// 8 waves with two query tiles each (256 queries; every K and V^T fragment read from LDS feeds two
// MFMAs) from 512 on (2048 keys, 16 x 16 heads 516 -> 464 us; 214 registers, two waves per SIMD), unless a causal sequence is one such strip:
// both of its blocks are multiplied for all of its queries (256 causal keys, heads of 64: 24 to 512 heads 1.26 to 1.9 of the time in smaller strips).
// Heads of 65 to 96 gain from it throughout (80 x 10: 1792 keys 0.77 of the time of the better of 4 and 8, 256 keys 0.90; causal 0.9 to 1.0, one and
// two strips a sequence 1.05 to 1.15).  128-wide heads never: the 8-wave
// form prefetches the next block through registers (565 -> 532 us at 2048 keys, 16 x 8 heads), and with two tiles it took all
// 256 registers and spilled 49 (two and one, additive mask: 32 x 8 heads, 1024 keys 526 and 428, causal 517 and 337, 16 x 8, 2048 keys 1003 and 829).
// Two tiles on 4 waves lose more to the missing third wave than they save (735 us).
// HD: head size of the template; nbh: sequences times heads; plain: no additive mask and a positive scale; padded: sequences of their own lengths.
inline MhaForm mha_form(int HD, bool compact, int S, int nbh, bool causal, bool plain, bool padded) {
    constexpr int kDies = 8;  // accelerator dies, of 32 compute units; the strips of a (sequence, head) share one
    const int qblocks = S / 16;
    if (!compact) {
        const int strips8 = (qblocks + 7) / 8, strips4 = (qblocks + 3) / 4;
        // The two groups of waves in turn: 256-query strips like the next form, but from 192 of them on (2 x 16 heads, 2048
        // keys, 256 strips: 58.7 -> 45.2 us; 4 x 12 heads, 1024 keys, 192: 30.3 -> 24.0; with 128 strips 35 -> 41) and from
        // 512 keys on (512 strips of 512 keys 32.4 either way, of 256 keys 32.3 -> 34): a sequence of one or two blocks
        // has nothing to take turns with.
        if (HD == 64 && qblocks % 16 == 0 && S >= 512 && (long)nbh * (qblocks / 16) >= 192 && plain) return {8, 2, true, false};
        // The same for other lengths, where the strips of 256 leave no more than a tenth more places empty
        // than strips of 128 and fill the last round of every die (32 units) to 85 % (16 x 12 heads: 912 keys 98.3 -> 83.5 us, 1872 302 -> 252,
        // 2032 332 -> 271; 8 x 16 heads, 1296 keys 115 -> 96; but 8 x 12 heads, 912 keys, three quarters full, 45.8 -> 51.3; causal level or
        // slower, and the form has no code for it, which is 4 % of its time).
        const int strips16 = (qblocks + 15) / 16, units = (nbh + kDies - 1) / kDies;
        const long u16 = (long)units * strips16;
        if (HD == 64 && qblocks % 16 != 0 && S >= 768 && !causal && plain && 20 * strips16 <= 11 * strips8 &&
            100 * u16 >= 85 * 32 * ((u16 + 31) / 32))
            return {8, 2, true, true};
        const bool one_causal_strip = HD == 64 && causal && qblocks == 16;
        if (HD >= 64 && HD != 128 && qblocks % 16 == 0 && (long)nbh * (qblocks / 16) >= 512 && !one_causal_strip) return {8, 2, false, false};
        const long u8 = (long)units * strips8, u4 = (long)units * strips4;  // workgroups of a die
        bool takes8;
        if (causal) {
            const bool whole = qblocks % 8 == 0, as_full = 2 * strips8 == strips4 && 10 * u8 >= 7 * (64 * ((u8 + 63) / 64));
            takes8 = HD == 128 ? whole || as_full : HD == 64 && whole && (qblocks <= 16 || (u8 > 48 && u8 <= 80));
        } else {
            const int cost8 = HD == 64 ? (qblocks <= 6 ? 160 : 184) : HD == 96 ? 194 : 175;  // of 8 waves, in hundredths of 4
            const bool uneven = HD == 64 && padded && S > 448 && u8 <= 32;
            takes8 = uneven ? false : HD == 128 && S <= 128 ? u8 <= 32
                     : HD == 128 && padded ? 182 * strips8 <= 100 * strips4 : cost8 * ((u8 + 31) / 32) <= 100 * ((u4 + 31) / 32);
        }
        if (HD >= 64 && (long)nbh * strips8 >= 256 && takes8) return {8, 1, false, false};
    }
    if (HD <= 64 && (qblocks == 1 || qblocks % 4 == 2)) {
        const auto rounds = [&](int waves, int held) {  // of the chip's 256 units, each holding `held` workgroups
            return ((long)nbh * ((qblocks + waves - 1) / waves) + 256 * held - 1) / (256 * held);
        };
        const long in4 = rounds(4, compact ? 2 : 3), in2 = rounds(2, HD == 32 && !compact ? 6 : 4), in1 = rounds(1, 8);
        const bool fits = qblocks <= 2 || in2 == 1 || (qblocks == 6 && (in4 <= 3 || (HD == 32 && !compact)));
        if (HD == 32 && qblocks == 1 && in1 < in4 && (in1 < in2 || (in1 == in2 && in1 > 1))) return {1, 1, false, false};
        if ((in2 < in4 && fits) || (qblocks == 2 && (compact ? HD == 32 : nbh >= 512))) return {2, 1, false, false};
    } else if (qblocks == 2 && nbh >= 512 && !compact) {
        return {2, 1, false, false};
    }
    return {4, 1, false, false};
}

// Heads of more than 224 columns in blocks of 128 keys instead of 64, which leaves a compute unit room for one workgroup: where it gets
// no more than one, and the sequence is long enough to fill the blocks.  us, 6 heads of 256, blocks of 64 and 128: 640 keys 34.4 and 32.0, 1824 causal
// 90.2 and 84.1, 2 x 336 22.0 and 21.2, 2 x 928 50.0 and 48.6; 176 keys 13.1 and 15.5; more workgroups than units, 4 x 1040 1.40 the other way.
// Heads of up to 224 are level or ahead in blocks of 64 throughout (4 of 200: 2048 keys 88.8 and 89.7).
inline bool mha_wide_blocks(int S, int nbh) {
    return S > 192 && (long)((nbh + 7) / 8) * ((S + 63) / 64) <= 32;  // units of a die
}

// ---- products of 32 x 32 x 16 (mha_tiles32_kernel) -------------------------------------------------------
// `waves` of a workgroup, `split` of which share a tile of 32 queries (each with its part of every staged block of keys), and
// 32-key steps of a wave a block; 0 waves: none, the forms above.
struct MhaTiles {
    int waves, split, steps;
    constexpr int queries() const { return 32 * (waves / split); }  // of a workgroup
    constexpr int keys() const { return 32 * steps * split; }       // staged at a time
};
// What a form was measured to take, in units of 10 ns: `start` once; a block of keys `chain` where the workgroup is alone on its compute unit, and
// `block` for every workgroup the fullest unit gets where they fill it; `wg` for each of those once.  Fitted to 400 problems of 80 to 2048 keys, 1 to
// 64 sequences, causal and padded ones among them, three sets of operands in turn: each form within 5 to 11 % of its time, the
// choice 0.8 % (heads of 64), 0.3 % (32) to 1 % (128) behind the best form in the mean, and 0.81 (64), 0.85 (32), 0.72 (96), 0.68 (128) and
// 0.86 (200) times the forms above.  us, the forms above and the choice: 12 heads of 64, 1 x 512 keys 8.7 and 6.2 (a tile's keys
// over four waves), 16 heads, 4 x 512 12.6 and 10.0 (over two), 16 x 2048 351 and 326 (tiles of one wave; 372 and 346 on another board: the power it is allowed), causal 274 and 218;
// 8 heads of 128, 8 x 1024 68 and 46.
// `again`: under a causal mask the fullest unit's second workgroup is the 32nd after its first in the die's list of strips (the longest of a (sequence, head) first), as long as that
// where the strips of a sequence divide 32, and booked as the mean the form was chosen where it is slower than the forms above (16 heads of 64, 4 x 1024 keys 28.5 us for 25.2,
// now 25.1 in another, 2 x 2048 43.0, 42.0 and 36.6; 10 of 80, 7 x 448 19.7 for 17.2, now 15.5).  Only for two a unit, up to 2048 keys and the forms that were chosen wrongly for it: 21 of 1070 causal problems change, 0.89 of
// their time; booked for all forms and lengths it would choose worse ones as often.
struct MhaTilesCost { MhaTiles form; int start, chain, block, wg; bool again = false; };
constexpr MhaTilesCost kMhaTiles32[] = {{{4, 1, 2}, 192, 85, 54, 81}, {{4, 2, 2}, 231, 74, 48, 91}, {{4, 4, 1}, 225, 59, 30, 73}};
constexpr MhaTilesCost kMhaTiles64[] = {{{4, 1, 2}, 108, 88, 54, 221}, {{8, 1, 2}, 120, 127, 111, 154}, {{4, 2, 2}, 157, 106, 64, 177},
                                        {{8, 2, 2}, 0, 123, 116, 412, true}, {{4, 4, 1}, 192, 80, 48, 137}};
constexpr MhaTilesCost kMhaTiles96[] = {{{4, 1, 2}, 0, 124, 76, 377}, {{8, 1, 2}, 0, 147, 156, 376}, {{4, 2, 2}, 48, 155, 134, 362, true}, {{8, 2, 2}, 0, 154, 160, 547}};
constexpr MhaTilesCost kMhaTiles128[] = {{{4, 1, 2}, 19, 145, 97, 364}, {{8, 1, 2}, 0, 173, 200, 364}, {{4, 2, 2}, 21, 165, 151, 422}, {{4, 4, 1}, 96, 0, 118, 341}};
// 129 to 224 columns, where the forms above (64 queries a workgroup, blocks of 64 keys) stay ahead for some: 4 heads of 200, 12 x 48
// keys 6.3 and 6.7 us.  (Eight waves of a tile each: problems without a mask show what a block costs a full unit alone; the chain is that of the longest causal
// strip, 4 heads of 200, 2048 keys 94.8 us, the forms above 89.3, two waves a tile, which are chosen, 58; over 540 causal problems of 80 to 4096 keys the choice is
// 2.7 % behind the best form in the mean, 0.94 of the time of the chain of 112 that fits the others, and slower than that for none.)
constexpr MhaTilesCost kMhaTiles224[] = {{{0, 1, 2}, 0, 274, 182, 330}, {{4, 1, 1}, 0, 158, 109, 393}, {{4, 2, 1}, 0, 201, 190, 500},
                                         {{4, 1, 2}, 0, 250, 279, 412}, {{8, 1, 2}, 0, 240, 354, 359}};

template <int N> inline MhaTiles mha_tiles_least(const MhaTilesCost (&costs)[N], int S, int nbh, bool causal) {
    long long best = -1;
    MhaTiles form{};
    for (const MhaTilesCost &c : costs) {
        const int q = c.form.waves ? c.form.queries() : 64, keys = c.form.waves ? c.form.keys() : 64, strips = (S + q - 1) / q;
        long long sum = 0, longest = (S + keys - 1) / keys;  // blocks of all strips, of the longest
        if (causal)
            for (int i = 1; i <= strips; i++) sum += ((i * q < S ? i * q : S) + keys - 1) / keys;
        else
            sum = longest * strips;
        const long long units = ((long long)((nbh + 7) / 8) * strips + 31) / 32;  // workgroups of the fullest of a die's 32
        long long blocks = sum * units;  // of the fullest unit, times the strips
        if (causal && c.again && units == 2 && S <= 2048) {
            const int before = 32 % strips, limit = (strips - before) * q;  // strips that end later, keys that the second one sees
            const long long two = (longest + ((limit < S ? limit : S) + keys - 1) / keys) * strips;
            if (two > blocks) blocks = two;
        }
        const long long alone = c.chain * longest * strips, full = c.block * blocks;
        const long long t = (long long)(c.start + c.wg * units) * strips * 1000 + (alone > full ? alone : full) * 1000;
        const long long per = t / strips;
        if (best < 0 || per < best) {
            best = per;
            form = c.form;
        }
    }
    return form;
}
// What mha_tiles32_kernel can do at all: nothing added to the scores and a positive scale, heads of up to 224, rows of the result at multiples of 16
// bytes; rows of a block are addressed with 32-bit offsets; the reciprocal of the number of heads is exact up to 2^32 over it; the rows of its grid.
inline bool mha_tiles_apply(int hd, bool plain, bool z16, int widest, int nbh, int nh) {
    return plain && hd <= 224 && z16 && widest <= 1 << 21 && (unsigned long long)nbh * (unsigned)nh < 1ull << 32 && nbh <= 8 * 32768 && nh < 1 << 24;
}

// Few short sequences keep the forms above: the one launch of attention and output projection (mha_fuseo_kernel) is made of those, and where it
// is used the two launches it replaces give the same bits.  (us, the forms above and this kernel: 12 heads of 64, 1 x 128 keys 4.2 and 3.9, 8 x 128 4.5
// and 4.4, 3 x 176 5.9 and 4.9.)  Otherwise up to 64 keys, one block of them, there is nothing to share (1.0 to 1.3 of the time); a tile of its own for
// every wave against the strips of 4, 2 and 1 waves above, 16 to 64 keys, 408 to 4800 tiles: 0.64 to 0.88 of the time (84 x 16 keys, 12 heads of 64 6.1 and 4.8,
// 128 x 32, 12 of 32 7.7 and 6.5, 300 x 32, 8 of 128 32 and 21).
// Sequences of their own lengths (padded): the costs know none, and one long sequence among short ones keeps a unit's only workgroup of eight waves
// to its end.  Heads of 33 to 96 take four there (tiles of 65 to 96 columns that waves share gain nothing, nor do sequences of one strip): us, the 16 x 16 kernel, eight and four, lengths of a quarter
// to the whole, 16 heads of 64, 4 x 640 keys 14.3, 16.0 and 14.1, 4 x 512 12.6, 9.1 and 8.4, 12 heads, 3 x 784 17.4, 19.3 and 15.5, 10 of 80, 4 x 1024 27.4, 29.7 and 25.4.
// Where all are nearly whole it costs 5 to 8 % (4 x 12, 448 keys 9.0 and 9.7); two a unit gain as often as they lose (8 x 16, 1024 keys 40.8 and 35.4 or 32.1 and 35.1 by
// the lengths, 16 x 16, 512 keys 23.7 and 25.3), and so do heads of 128 alone on theirs (3 x 1536 keys 37.7 and 31.0, 12 x 512 20.9 and 22.4).  One sequence has nothing to
// even out: it keeps eight (12 heads, 1 x 2048 keys 17.7, four 19.1; 10 of 80, 1 x 3584 62.1 and 67.9).
// lengths: sequences that have lengths of their own, 0 if they do not.
inline MhaTiles mha_tiles(int HD, int S, int nbh, bool causal, int lengths = 0) {
    const bool padded = lengths > 0;
    const auto evened = [&](MhaTiles f) {
        const int units = ((nbh + 7) / 8 * ((S + f.queries() - 1) / f.queries()) + 31) / 32;  // workgroups of the fullest of a die's 32
        if (lengths > 1 && f.waves == 8 && (HD == 64 || f.split == 1) && units == 1 && S > f.queries()) f.waves = 4;
        return f;
    };
    if (HD <= 128 && S <= 384 && (long long)nbh * ((S + 31) / 32) <= 400) return {};
    if (HD <= 128 && S <= 64) return {4, 1, 2};
    // Wide heads, few of them (us, the forms above and tiles): 65 to 96 causal keys, 1 x 4 heads of 200, 80 keys 7.3 and 7.8, 8 x 6 of 136 7.4 and 8.1, 24 x 5 of 160 8.4
    // and 8.7, 96 keys, 8 x 6 7.7 and 8.1; more, 80 keys, 16 x 8 of 224 9.4 and 9.3, 24 x 6 10.1 and 8.9, 96 keys, 16 x 4 8.7 and 8.6.  65 to 80 keys of sequences of their own
    // lengths, 1 x 4 of 200 6.6 and 7.0, 6 of 136 6.1 and 7.0, 5 x 6 7.1 and 7.6, 6 x 6 7.8 and 8.0; more, 8 x 4 of 200 9.0 and 8.5, 10 x 6 of 136 level.
    if (HD == 224 && S > 64 && ((causal && S <= 96 && nbh <= (S <= 80 ? 120 : 48)) || (!causal && padded && S <= 80 && nbh <= 30))) return {};
    // Heads of 33 to 64 without a causal mask, where workgroups of eight waves are one to a unit: two of four, which the cost of one alone and of a full unit put ahead, take longer.
    // From 2560 keys on whole strips of 256 keep the waves in turn there, and from 6144 keys on eight waves are ahead of four wherever they are half as many, the longer the launch the lower the
    // clock.  us, waves in turn, four and eight: 12 heads, 4 x 1280 keys 30.4, 33.1 and 30.1, 1 x 4096 80, 89 and 84, 1 x 8192 305, 326 and 307, 16 heads, 4 x 1024 26.5, 27.5 and 26.2,
    // 2 x 2048 46, 49 and 46, 1 x 3584 69, 75 and 72.  70 of 1530 problems of up to 8192 keys change, 0.95 of their time; 45 were slower than waves in turn by 1.5 to 13 %, now one by 3 %.
    if (HD == 64 && !causal) {
        const auto fullest = [&](int queries) { return ((nbh + 7) / 8 * ((S + queries - 1) / queries) + 31) / 32; };
        const bool one = fullest(256) == 1;
        if (one && S >= 2560 && S % 256 == 0 && mha_form(HD, false, S, nbh, causal, true, padded).in_turn) return {};
        const MhaTiles f = mha_tiles_least(kMhaTiles64, S, nbh, causal);
        return evened(f.waves == 4 && f.split == 1 && (one || S >= 6144) && fullest(128) == 2 * fullest(256) ? MhaTiles{8, 1, 2} : f);
    }
    switch (HD) {
        case 32: {  // (four waves a tile: a unit holds three such workgroups, and the fourth of four waits; 12 x 12 heads, 208 keys 8.0 us in the forms above, 8.7 so, 7.4 with two)
            const MhaTiles f = mha_tiles_least(kMhaTiles32, S, nbh, causal);
            return f.split == 4 && S <= 256 && ((nbh + 7) / 8 * ((S + 31) / 32) + 31) / 32 == 4 ? MhaTiles{4, 2, 2} : f;
        }
        case 64: return evened(mha_tiles_least(kMhaTiles64, S, nbh, causal));
        case 96: return evened(mha_tiles_least(kMhaTiles96, S, nbh, causal));
        case 128: return mha_tiles_least(kMhaTiles128, S, nbh, causal);
        case 224: return mha_tiles_least(kMhaTiles224, S, nbh, causal);
        default: return {};
    }
}

}  // namespace et
