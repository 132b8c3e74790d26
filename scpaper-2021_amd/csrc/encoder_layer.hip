// Everything of a tile-sparse encoder layer that is local to a token, in one launch:
//
//   V1 = Z Wo^T + bo + x;  y = LN1(V1);  V2 = act(y W1^T + b1) W2^T + b2 + y;  x' = LN2(V2);  QKV' = x' Wq^T + bq
//
// (Encoder/Encoder.h:81-96 from the output projection on, and the next layer's projection, Attention/Attention.h:246-265;
// all weights in 16x16 tiles, the mathematics of Linear/SPMM_tile.cu:249-324).
//
// A workgroup of 16 waves owns 16 MT token rows and takes them through all five steps: the token strip, the hidden
// activations and the vectors stay in LDS, the sums in registers, and what passes through memory is Z, x and QKV'.
// What it has to take in is the weight: every workgroup streams all kept tiles once, 1 KiB (two tiles, one
// v_mfma_f32_16x16x32_f16 per 16 tokens) at a time.  All workgroups of an XCD stream the same bytes at about the same
// time, so the stream comes out of its L2: measured 115-125 GB/s per compute unit with 8 slots of every wave in
// flight, first touch included (2.9 MB, BERT-base at 80 %: 25 us, whether 8 or 256 workgroups read it), which bounds a
// launch with one token tile (53 000 of 65 000 cycles at 4096 rows).  With two (from 4097 rows on, half the workgroups a
// row) the waves' own instructions do, vector and scalar together: the products without any load or LDS read still take
// two thirds of the time.
//
// Against separate launches per matrix (five to seven a layer) this removes the intermediate activations (at 8192 rows
// and BERT-base sizes about 300 MB of reads and writes per layer) and the launch boundaries (1.6 us each), and the weight
// requests never drain: the ring of a wave is filled across barriers, since no weight depends on an activation.
// 12 layers of BERT-base at 80 %, three models in turn: 64 x 128 tokens 2101 -> 889 us, 8 x 128 540 -> 369; BERT-large 4 x 512 at
// 90 % 1842 -> 1185.  On the way: the residual and the shares in tile order instead of rows (lines written in halves by two waves),
// QKV' through LDS as whole rows instead of 32 bytes a token, and the parts of a strip on one XCD: 1150 -> 1060 at 64 x
// 128, 562 -> 480 at 8 x 128; accumulating in place of a zeroed sum and a later addition: 2 %.
//
// Few rows leave most compute units without a strip.  Then PARTS workgroups share a strip.  In two launches the first
// repeats the output projection and LN1, and each part runs its share of the hidden features, leaving its share of
// the second product in binary32; the second adds the shares in a fixed order, applies LN2 and runs its share of
// the QKV block-rows.  That projection can be had alone, of x' as it was rounded for it (et_encoder_layer_project_f16), so
// that a stack whose layers hand binary16 to each other gives the same bits layer by layer.
// The joined launch does both: behind the second product the parts of a strip meet at a word in their XCD's L2 (meet_wait), and
// the shares come back out of that L2, where behind a launch boundary they come from the memory-side cache, as do table, offsets
// and first slots, which here are on their way while the parts meet; 2 us of boundary go besides.  8 x 128 tokens at 80 %
// 382 -> 361 us (12 layers, weights in the memory-side cache), 12 x 128 241 -> 220 (6 layers), BERT-large 4 x 512 at 90 % 1175 ->
// 1124.  (The first form of it, with requests only behind the meeting: 387.)  What the parts do between the products is bound by
// scalar round trips and by vector instructions, not by bytes (of 52 000 cycles at 8 x 128 the LayerNorms are 6 600, the shares 3 800, the way
// out of the projection 2 100): the others' shares requested in one go at addresses worked out once, the chunks of the projection in
// the table instead of divisions, binary16 values added by v_fma_mix: 375.7 -> 368.1 us there, one sequence 320.4 -> 311.8.
//
// Streams (built on the host, et_encoder_layer_pack_create; those of the second launch, or of the projection alone, behind
// those of the first): per (part, wave) the slots in the order they are multiplied, the byte offsets of their two column
// tiles in the strip, and a descriptor per block-row: slots, kind, where the result goes, where its bias lies.  A segment is what lies between two
// workgroup barriers: Wo; the first chunk of hidden features; (chunk c + 1 of W1, the columns of chunk c of W2)...; the
// last columns of W2; Wq.  Hidden chunks alternate between two LDS buffers, so one barrier per chunk is enough.
// Block-rows are dealt to the waves longest first, within a segment.
#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <type_traits>
#include <vector>

#include "common.hip.h"
#include "strip_meeting.h"

namespace et {

constexpr int kElWaves = 16;
constexpr int kElRing = 8;     // weight slots of a wave in flight
constexpr int kElMaxSeg = 24;  // segments of a launch
constexpr size_t kElLds = 160 * 1024;
// table of a (part, wave), 64 words, a lane holds one: block-rows of every segment, sums of every wave, slots, and of every chunk of
// the projection its first block-row (bits 0-15) and their number (worked out in the kernel, four divisions a chunk); and the descriptors
// of its block-rows behind it, in the same way: one request each at the start, read with v_readlane
constexpr int kElTabSeg = 0, kElTabCount = kElTabSeg + kElMaxSeg, kElTabSlots = kElTabCount + kElWaves, kElTabOut = kElTabSlots + 1, kElTabWords = 64, kElRowRegs = 2, kElTab = kElTabWords * (1 + kElRowRegs);
// descriptor: slots (bits 0-7), kind (8-9), operand in the hidden chunk (10), target (11-20), bias over 16 (21-31)
constexpr int kElBufferWord = 0x00020000;  // of a raw buffer resource
constexpr int kElKindSum = 0, kElKindHidden = 1, kElKindQkv = 2, kElMaxSlots = 255;

typedef int i4 __attribute__((ext_vector_type(4)));

struct LayerArgs {
    // joined launch: the streams behind the join, and a word per strip
    const char *slots2, *offs2;
    const int32_t *tab2;
    uint32_t *join;
    int cap2, spin;
    const char *slots;
    float *x32_out;       // x' in tile order (may be null)
    _Float16 *out16;      // x' rounded (may be null)
    _Float16 *qkv;
    float *partial;       // [parts], each T x H in tile order
    int T, H, FF, Q;
    // Tile order: the 16 x 16 values of 16 tokens and a block-row are 1 KiB, a lane's four together, so that a wave reads
    // and writes whole lines of what only these launches exchange
    int hs;               // bytes of a hidden row in LDS, a multiple of 256
    int nseg_ff, nseg_q;  // segments of the hidden features, of the projection
    int hbuf;             // bytes between the two hidden buffers (0: one is enough)
    int parts, nshare, act;  // parts of this launch, shares of the second product
    float eps1, eps2, inv_h;
    uint32_t sums[kElWaves];  // block-rows of the model width a wave holds the sums of, 8 bits each (255: none)
};

// What the first requests need, in front of the other arguments and one by one: preloaded into scalar registers.  Read from memory, and with
// divisions for a workgroup's place and its pieces of the strip, a wave had asked for everything 3 400 cycles after it started, of 48 000 (us, before
// and now, three models in turn: one sequence of 128 tokens 316 and 311, 8 x 128 362 and 357, BERT-large 4 x 512 1109 and 1091, 528 rows 228 and 223).
struct LayerFirst {
    const _Float16 *Z;
    const void *x;       // residual: binary32 in tile order, or binary16 row by row
    const char *offs;    // per wave and eight slots: 8 x 16 bits of the first tiles' offsets, 8 of the second
    const int32_t *tab;  // per (part, wave) the table and its descriptors
    const _Float16 *vec;  // bo, g1, be1, b1, b2, g2, be2, bq
    int T, H;
    int cap;             // slots from one (part, wave) to the next
    unsigned form;       // bytes of a strip row in LDS over 256 (bits 0-7), the residual is binary16 (8), vectors over 8 (16-31)
};
#define ET_EL_FIRST const _Float16 *Z, const void *x, const char *offs, const int32_t *tab, const _Float16 *vec, int T, int H, int cap, unsigned form
constexpr size_t kElFirstBytes = 56;  // of them among the arguments
static_assert(sizeof(LayerFirst) == kElFirstBytes, "the other arguments follow them");

// The weight ring lives in registers the compiler does not have: v[96:127] hold the next eight slots of the wave,
// v[88:91] the column offsets of the current eight slots (16 bits each, those of this half of the wave), v[92:95] those of
// the eight after them.  The kernel is compiled for 88 registers, and only the assembly below touches the others, so a
// request can stay in flight across anything the compiler puts between two block-rows (left to the compiler, the
// ring was copied between registers at every block-row, in flight or not).  vmcnt counts in order: behind the request of
// a slot lie seven of later slots and one of offsets (the slot at position 7: seven), so a slot has arrived at vmcnt(8)
// (7); whatever else the compiler issues in between only makes the wait longer.  The compiler warns that it does not
// expect assembly to touch registers it was told to leave; what it makes of this file is held to these rules, instruction
// by instruction, by a test.
#define ET_EL_CLOBBERS                                                                                                   \
    "v88", "v89", "v90", "v91", "v92", "v93", "v94", "v95", "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103", \
        "v104", "v105", "v106", "v107", "v108", "v109", "v110", "v111", "v112", "v113", "v114", "v115", "v116", "v117",  \
        "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125", "v126", "v127", "memory"
// (registers the compiler may use; the attribute counts them in pairs on this architecture)
constexpr int kElOwnVgprs = 88 / 2;

// The column offsets of the wave's first eight slots, the first request of a wave: its first block-row reads them before it
// waits for anything, so they have to be there when the prologue ends (requested with the ring, a wait for them costs
// another round trip: 8 x 128 tokens, 12 layers, 481 us against 475).
__device__ __forceinline__ void el_ask_offsets(unsigned offs_off, const char *offs) {
    asm volatile("global_load_dwordx4 v[88:91], %0, %1" ::"v"(offs_off), "s"(offs) : "v88", "v89", "v90", "v91", "memory");
}
// fills the ring behind it: `slots` + lane_off and `offs` + offs_off point at the wave's first slot and offsets; both are
// left behind what was requested
constexpr int kElRingAsks = kElRing + 1;  // requests of a ring filled
__device__ __forceinline__ void el_ring_start(unsigned &lane_off, unsigned &offs_off, i4 slots, const char *offs) {
    asm volatile(
        "buffer_load_dwordx4 v[96:99], %0, %2, 0 offen\n\t"
        "buffer_load_dwordx4 v[100:103], %0, %2, 0 offen offset:1024\n\t"
        "buffer_load_dwordx4 v[104:107], %0, %2, 0 offen offset:2048\n\t"
        "buffer_load_dwordx4 v[108:111], %0, %2, 0 offen offset:3072\n\t"
        "v_add_u32 %0, 0x1000, %0\n\t"
        "buffer_load_dwordx4 v[112:115], %0, %2, 0 offen\n\t"
        "buffer_load_dwordx4 v[116:119], %0, %2, 0 offen offset:1024\n\t"
        "buffer_load_dwordx4 v[120:123], %0, %2, 0 offen offset:2048\n\t"
        "global_load_dwordx4 v[92:95], %1, %3 offset:32\n\t"
        "buffer_load_dwordx4 v[124:127], %0, %2, 0 offen offset:3072\n\t"
        "v_add_u32 %0, 0x1000, %0\n\t"
        "v_add_u32 %1, 64, %1"
        : "+v"(lane_off), "+v"(offs_off)
        : "s"(slots), "s"(offs)
        : ET_EL_CLOBBERS);
}

// A block-row of n >= 1 slots from ring position `pos` on (compiled once per set of accumulators): acc[m] += tiles x (16 tokens at LDS byte `base` + m `step`).
// The operand fragments of a slot (one read of 16 tokens x 32 values per token tile, at the slot's column offset XORed
// with the row's swizzle) are requested a slot ahead, into the two sets in turn; behind its products the slot's registers
// take the request of the slot eight further on.  At position 7 the offsets of the next eight slots move up.
#define ET_EL_FRAG1(U, SH, X) "v_bfe_u32 %[t], v" #U ", " #SH ", 16\n\tv_xad_u32 %[t], %[t], %[kx], %[base]\n\tds_read_b128 %[" X "0], %[t]\n\t"
#define ET_EL_FRAG2(U, SH, X) ET_EL_FRAG1(U, SH, X) "v_add_u32 %[t], %[t], %[step]\n\tds_read_b128 %[" X "1], %[t]\n\t"
#define ET_EL_MUL1(W, X, VM, LG) "s_waitcnt vmcnt(" VM ") lgkmcnt(" LG ")\n\tv_mfma_f32_16x16x32_f16 %[a0], v[" W "], %[" X "0], %[a0]\n\t"
#define ET_EL_MUL2(W, X, VM, LG) ET_EL_MUL1(W, X, VM, LG) "v_mfma_f32_16x16x32_f16 %[a1], v[" W "], %[" X "1], %[a1]\n\t"
#define ET_EL_REQ(W, OFF, ADV) "buffer_load_dwordx4 v[" W "], %[lo], %[slots], 0 offen" OFF "\n\t" ADV
#define ET_EL_ADV "v_add_u32 %[lo], 0x1000, %[lo]\n\t"
#define ET_EL_NEXT                                                                                       \
    "s_waitcnt vmcnt(7)\n\t"                                                                             \
    "v_mov_b32 v88, v92\n\tv_mov_b32 v89, v93\n\tv_mov_b32 v90, v94\n\tv_mov_b32 v91, v95\n\t"         \
    "global_load_dwordx4 v[92:95], %[oo], %[offs]\n\tv_add_u32 %[oo], 32, %[oo]\n\t"
// OFF, ADV: the slot's offset in its four, and the step to the next four; NI, NU, NSH, NX: the next position, its offset
// register and shift, its fragment set
#define ET_EL_SLOT(I, W, X, OFF, ADV, PRE, NI, NU, NSH, NX, FRAG, MUL, LG)               \
    "el_slot%=_" #I ":\n\ts_add_i32 %[n], %[n], -1\n\ts_cmp_eq_u32 %[n], 0\n\ts_cbranch_scc1 el_last%=_" #I "\n\t" \
    PRE FRAG(NU, NSH, NX) MUL(W, X, "8", LG) ET_EL_REQ(W, OFF, ADV)
#define ET_EL_LAST(I, W, X, OFF, ADV, PRE, NI, MUL)                                      \
    "el_last%=_" #I ":\n\t" PRE MUL(W, X, "8", "0") ET_EL_REQ(W, OFF, ADV) "s_mov_b32 %[pos], " #NI "\n\ts_branch el_done%=\n\t"
#define ET_EL_ENTER(I, U, SH, X, FRAG) "el_enter%=_" #I ":\n\t" FRAG(U, SH, X) "s_branch el_slot%=_" #I "\n\t"
#define ET_EL_BODY(FRAG, MUL, LG)                                                          \
    "s_cmp_lt_u32 %[pos], 4\n\ts_cbranch_scc0 el_hi%=\n\t"                                 \
    "s_cmp_lt_u32 %[pos], 2\n\ts_cbranch_scc0 el_23%=\n\t"                                 \
    "s_cmp_eq_u32 %[pos], 0\n\ts_cbranch_scc0 el_enter%=_1\n\t"                           \
    ET_EL_ENTER(0, 88, 0, "x", FRAG) ET_EL_ENTER(1, 88, 16, "y", FRAG)                     \
    "el_23%=:\n\ts_cmp_eq_u32 %[pos], 2\n\ts_cbranch_scc0 el_enter%=_3\n\t"               \
    ET_EL_ENTER(2, 89, 0, "x", FRAG) ET_EL_ENTER(3, 89, 16, "y", FRAG)                     \
    "el_hi%=:\n\ts_cmp_lt_u32 %[pos], 6\n\ts_cbranch_scc0 el_67%=\n\t"                     \
    "s_cmp_eq_u32 %[pos], 4\n\ts_cbranch_scc0 el_enter%=_5\n\t"                           \
    ET_EL_ENTER(4, 90, 0, "x", FRAG) ET_EL_ENTER(5, 90, 16, "y", FRAG)                     \
    "el_67%=:\n\ts_cmp_eq_u32 %[pos], 6\n\ts_cbranch_scc0 el_enter%=_7\n\t"               \
    ET_EL_ENTER(6, 91, 0, "x", FRAG) ET_EL_ENTER(7, 91, 16, "y", FRAG)                     \
    ET_EL_SLOT(0, "96:99", "x", "", "", "", 1, 88, 16, "y", FRAG, MUL, LG) \
    ET_EL_SLOT(1, "100:103", "y", " offset:1024", "", "", 2, 89, 0, "x", FRAG, MUL, LG) \
    ET_EL_SLOT(2, "104:107", "x", " offset:2048", "", "", 3, 89, 16, "y", FRAG, MUL, LG) \
    ET_EL_SLOT(3, "108:111", "y", " offset:3072", ET_EL_ADV, "", 4, 90, 0, "x", FRAG, MUL, LG) \
    ET_EL_SLOT(4, "112:115", "x", "", "", "", 5, 90, 16, "y", FRAG, MUL, LG) \
    ET_EL_SLOT(5, "116:119", "y", " offset:1024", "", "", 6, 91, 0, "x", FRAG, MUL, LG) \
    ET_EL_SLOT(6, "120:123", "x", " offset:2048", "", "", 7, 91, 16, "y", FRAG, MUL, LG) \
    ET_EL_SLOT(7, "124:127", "y", " offset:3072", ET_EL_ADV, ET_EL_NEXT, 0, 88, 0, "x", FRAG, MUL, LG) \
    "s_branch el_slot%=_0\n\t" \
    ET_EL_LAST(0, "96:99", "x", "", "", "", 1, MUL) \
    ET_EL_LAST(1, "100:103", "y", " offset:1024", "", "", 2, MUL) \
    ET_EL_LAST(2, "104:107", "x", " offset:2048", "", "", 3, MUL) \
    ET_EL_LAST(3, "108:111", "y", " offset:3072", ET_EL_ADV, "", 4, MUL) \
    ET_EL_LAST(4, "112:115", "x", "", "", "", 5, MUL) \
    ET_EL_LAST(5, "116:119", "y", " offset:1024", "", "", 6, MUL) \
    ET_EL_LAST(6, "120:123", "x", " offset:2048", "", "", 7, MUL) \
    ET_EL_LAST(7, "124:127", "y", " offset:3072", ET_EL_ADV, ET_EL_NEXT, 0, MUL) \
    "el_done%=:\n\ts_nop 15\n\ts_nop 7"  /* the products have left the matrix pipe */
template <int MT>
__device__ __forceinline__ void el_row(f4 (&acc)[MT], int n, int &pos, unsigned base, unsigned step, unsigned kx, unsigned &lane_off,
                                       unsigned &offs_off, i4 slots, const char *offs) {
    pos = __builtin_amdgcn_readfirstlane(pos);
    unsigned t;
    h8 x0, x1, y0, y1;
    if constexpr (MT == 1)
        asm volatile(ET_EL_BODY(ET_EL_FRAG1, ET_EL_MUL1, "1")
                     : [a0] "+v"(acc[0]), [n] "+s"(n), [pos] "+s"(pos), [lo] "+v"(lane_off), [oo] "+v"(offs_off), [t] "=&v"(t),
                       [x0] "=&v"(x0), [y0] "=&v"(y0)
                     : [base] "v"(base), [kx] "v"(kx), [slots] "s"(slots), [offs] "s"(offs)
                     : ET_EL_CLOBBERS, "scc");
    else
        asm volatile(ET_EL_BODY(ET_EL_FRAG2, ET_EL_MUL2, "2")
                     : [a0] "+v"(acc[0]), [a1] "+v"(acc[MT - 1]), [n] "+s"(n), [pos] "+s"(pos), [lo] "+v"(lane_off), [oo] "+v"(offs_off),
                       [t] "=&v"(t), [x0] "=&v"(x0), [x1] "=&v"(x1), [y0] "=&v"(y0), [y1] "=&v"(y1)
                     : [base] "v"(base), [step] "v"(step), [kx] "v"(kx), [slots] "s"(slots), [offs] "s"(offs)
                     : ET_EL_CLOBBERS, "scc");
    pos = __builtin_amdgcn_readfirstlane(pos);
}

__device__ __forceinline__ void el_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void el_load_to_lds(const void *base, unsigned lane_off, unsigned lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_off), "s"(base), "s"(lds_base)
                 : "memory", "m0");
}

// Requests of the prologue, in assembly for the same reason: the compiler, which does not know of the ring, would wait for
// all of it with the first value it uses.  The caller waits by count and ties the values through el_tie.
__device__ __forceinline__ void el_ask(h8 &v, unsigned off, const void *base) {
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(v) : "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void el_ask(f4 &v, unsigned off, const void *base) {
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(v) : "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void el_ask(int &v, unsigned off, const void *base) {
    asm volatile("global_load_dword %0, %1, %2" : "=v"(v) : "v"(off), "s"(base) : "memory");
}
template <typename T> __device__ __forceinline__ void el_tie(T &v) { asm volatile("" : "+v"(v)); }

// the value, as something the compiler cannot compute ahead: keeps the addresses of what happens once or twice a launch from
// being held in registers through the multiplying loop
__device__ __forceinline__ int el_here(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

__device__ __forceinline__ int el_here_s(int v) {  // the same for a uniform value
    asm volatile("" : "+s"(v));
    return v;
}

// The word in the L2 of their XCD at which the parts of a strip meet (strip_meeting.h).  One wave, its first lane.  (In assembly:
// the arrival is in flight while the ring goes out, and an addition of nothing, which a part that waits reads the word with, would
// become a load that the L1 answers.)
#define ET_EL_ADD "s_mov_b64 exec, 1\n\tglobal_atomic_add %0, %1, %2, off sc0\n\ts_mov_b64 exec, -1"
struct ElWord {
    uint32_t *at;
    __device__ __forceinline__ uint32_t add(uint32_t v) {
        uint32_t was;
        asm volatile(ET_EL_ADD "\n\ts_waitcnt vmcnt(0)" : "=&v"(was) : "v"(at), "v"(v) : "memory");
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)was);
    }
    __device__ __forceinline__ void clear() { __hip_atomic_store(at, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
    __device__ __forceinline__ void pause() { __builtin_amdgcn_s_sleep(1); }
};

// MODE 0: all steps.  1: up to the second product, binary32 share to `partial`.  2: from the sum of the shares on.  3: the
// projection alone, of x' as 2 rounds it, given in `Z`: the same products in the same order.
// 4: 1 and 2 in one launch; behind the second product the parts of a strip meet.
template <int MT, int NR, int MODE> __device__ __forceinline__ void encoder_layer(const LayerFirst &f, const LayerArgs &a) {
    extern __shared__ __align__(256) unsigned char el_smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g = lane >> 4, gbit = g & 1;
    // The parts of a strip on one XCD (workgroups go to the 8 XCDs round-robin by id, x first): what they share comes from HBM once.
    const int group = MODE == 0 ? 0 : (int)(blockIdx.z ? blockIdx.y + gridDim.y * blockIdx.z : blockIdx.y);
    const int strip = MODE == 0 ? blockIdx.x : blockIdx.x % 8 + 8 * group, part = MODE == 0 ? 0 : blockIdx.x / 8;
    if (MODE != 0 && strip * MT * 16 >= f.T) return;  // padding of the grid (the whole workgroup)
    const int tok0 = strip * (MT * 16);
    const int H = f.H, xs = (f.form & 255) << 8;
    // The joined launch reads what it needs behind the join when it needs it: held from the start it would not fit the scalar
    // registers, and a scalar register that comes back from a vector lane must not be read by a request within five
    // instructions, which the compiler cannot see in the assembly here.
    auto late = [] {
        auto *p = (const __attribute__((address_space(4))) LayerArgs *)((const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr() + kElFirstBytes);
        asm volatile("" : "+s"(p));
        return p;
    };
    constexpr bool kLate = MODE == 4;
#define ET_EL_ARG(F) (kLate ? late()->F : a.F)
#define ET_EL_ONCE(F) (kLate || MODE == 0 ? late()->F : a.F)
    auto here = [](int v) { return kLate ? el_here_s(v) : v; };

    unsigned char *X = el_smem;                            // [MT * 16][xs], 16-byte units XORed with the row
    unsigned char *Hb = X + MT * 16 * xs;                // [1 or 2 chunks][MT * 16][hs], the same
    float *red = reinterpret_cast<float *>(Hb + a.hbuf + MT * 16 * a.hs);  // [2][16 waves][MT * 16]
    _Float16 *vec = reinterpret_cast<_Float16 *>(red + 2 * kElWaves * MT * 16);
    // (bo, g1, be1, b1, b2, g2, be2, bq)

    // ---- requests: the strip, the vectors, the residual or the shares, all at addresses the arguments give
    constexpr bool kFirst = MODE < 2 || MODE == 4, kParts = MODE == 1 || MODE == 4;  // begins with Z; has parts of the hidden features
    const int stream = part * kElWaves + wave;
    // A buffer that ends with the wave's last slot: the ring's requests past it go nowhere.  Answered, they were 128 KiB of the
    // 0.9 MiB a workgroup of the first launch took in at 8 x 128 tokens, and of the 0.6 of the second.
    const uint64_t slots_at = (uint64_t)(a.slots + (size_t)stream * f.cap * 1024);
    i4 slots = {(int)(unsigned)slots_at, (int)(unsigned)(slots_at >> 32), f.cap * 1024, kElBufferWord};
    const char *offs = f.offs + (size_t)stream * f.cap * 4;  // uniform
    unsigned lane_off = lane * 16, offs_off = (g >> 1) * 16;
    el_ask_offsets(offs_off, offs);
    if constexpr (MODE != 2) {
        // Z -> X, straight into LDS, a wave a row: the lane that fills unit pu of a row fetches the row's unit pu ^ (row % 16); units
        // past H repeat the last one (nothing names them)
        const int upr = xs >> 4, last = (H >> 3) - 1;
        const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) void *)X);
#pragma unroll
        for (int m = 0; m < MT; m++) {
            const int row = wave + m * kElWaves;
            const char *zb = reinterpret_cast<const char *>(f.Z + (size_t)min(tok0 + row, f.T - 1) * H);
            for (int u = 0; u < upr; u += 64)  // (at least 16 lanes of each)
                if (u + lane < upr) el_load_to_lds(zb, (unsigned)(min((u + lane) ^ (row & 15), last) << 4), lds0 + (unsigned)(row * xs + u * 16));
        }
    }
    // the table of the wave and its descriptors
    int tab, desc[kElRowRegs];
    el_ask(tab, lane * 4, f.tab + (size_t)stream * kElTab);
#pragma unroll
    for (int i = 0; i < kElRowRegs; i++) el_ask(desc[i], lane * 4, f.tab + (size_t)stream * kElTab + (1 + i) * kElTabWords);

    const uint32_t own = a.sums[wave];
    int rb[NR];
#pragma unroll
    for (int j = 0; j < NR; j++) rb[j] = (own >> (8 * j) & 255) == 255 ? -1 : (int)(own >> (8 * j) & 255);
    // bytes from the strip's first value to a tile in tile order (uniform); a second tile past the end: the first
    const int tiles_here = min(MT, (f.T - tok0) >> 4);
    auto tile_at = [&](int m, int j) { return (unsigned)((MT == 1 ? 0 : min(m, tiles_here - 1) * H) + max(here(rb[j]), 0) * 16) * 64; };

    auto ask_vectors = [&] {  // straight into LDS, 512 values an instruction
        const int nvec = f.form >> 16;
        const unsigned lds0 = (unsigned)(size_t)((__attribute__((address_space(3))) void *)vec);
        for (int i = wave * 64; i < nvec; i += kElWaves * 64)
            if (i + lane < nvec) el_load_to_lds(f.vec, (unsigned)(i + lane) * 16u, lds0 + (unsigned)i * 16u);
    };
    const bool half_in = MODE != 2 && (f.form >> 8 & 1);  // uniform
    f4 V[NR][MT];
    unsigned long long r16v[NR][MT];
    auto ask_residual = [&](f4 (&to)[NR][MT]) {
        if (half_in) {
            const char *src = reinterpret_cast<const char *>(static_cast<const _Float16 *>(f.x) + (size_t)tok0 * H);
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    const unsigned row_at = (unsigned)(min(tok0 + m * 16 + r16, f.T - 1) - tok0) * H * 2;
                    asm volatile("global_load_dwordx2 %0, %1, %2" : "=v"(r16v[j][m]) : "v"(row_at + max(rb[j], 0) * 32 + g * 8), "s"(src) : "memory");
                }
        } else {
            const char *src = reinterpret_cast<const char *>(static_cast<const float *>(f.x) + (size_t)tok0 * H);
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int m = 0; m < MT; m++) el_ask(to[j][m], tile_at(m, j) + lane * 16, src);
        }
    };
    auto keep_residual = [&](f4 (&to)[NR][MT]) {
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int m = 0; m < MT; m++) {
                if (half_in) {
                    el_tie(r16v[j][m]);
                    const h4 r = __builtin_bit_cast(h4, r16v[j][m]);
                    to[j][m] = f4{(float)r[0], (float)r[1], (float)r[2], (float)r[3]};
                } else {
                    el_tie(to[j][m]);
                }
            }
    };
    // The ring goes out behind what every wave needs to begin with: 128 KiB of it ahead of a later wave's strip, vectors and
    // residual would hold up all, since a compute unit takes in 64 bytes a cycle (8 x 128 tokens, 12 layers, weights in the
    // memory-side cache: 390 -> 382 us).  Ends with everything but the ring there.
    auto ring_start = [&] {
        asm volatile("s_barrier" ::: "memory");
        el_ring_start(lane_off, offs_off, slots, offs);
        asm volatile("s_waitcnt vmcnt(%0)" ::"i"(kElRingAsks) : "memory");
    };
    // The shares of a strip, added in the order of the parts, into V.  The ring goes out behind the last of them.
    auto sum_shares = [&] {
        constexpr int kTogether = NR > 3 ? 2 : 4;  // shares requested together
        f4 u[kTogether][NR][MT], sum[NR][MT];
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int m = 0; m < MT; m++) sum[j][m] = f4{0.f, 0.f, 0.f, 0.f};
        const int nshare = a.nshare;
        auto ask_shares = [&](int p) {
#pragma unroll
            for (int q = 0; q < kTogether; q++) {
                const char *src = reinterpret_cast<const char *>(a.partial + ((size_t)min(p + q, nshare - 1) * a.T + tok0) * a.H);
#pragma unroll
                for (int j = 0; j < NR; j++)
#pragma unroll
                    for (int m = 0; m < MT; m++) el_ask(u[q][j][m], tile_at(m, j) + lane * 16, src);
            }
        };
        auto add_shares = [&](int p) {
#pragma unroll
            for (int q = 0; q < kTogether; q++)
#pragma unroll
                for (int j = 0; j < NR; j++)
#pragma unroll
                    for (int m = 0; m < MT; m++) el_tie(u[q][j][m]);
#pragma unroll
            for (int q = 0; q < kTogether; q++)
                if (p + q < nshare) {  // uniform
#pragma unroll
                    for (int j = 0; j < NR; j++)
#pragma unroll
                        for (int m = 0; m < MT; m++) sum[j][m] += u[q][j][m];
                }
        };
        int p = 0;
        for (; p + kTogether < nshare; p += kTogether) {
            ask_shares(p);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            add_shares(p);
        }
        ask_shares(p);
        ring_start();
        add_shares(p);
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int m = 0; m < MT; m++) V[j][m] = sum[j][m];
    };
    // The same in the joined launch, where V holds the share of part `mine` and the ring went out while the parts met: the others'
    // shares are requested together, as many as there are registers for (with four parts all three), at addresses worked
    // out once.  The order of the additions is that of the parts.
    auto sum_others = [&](int mine) {
        constexpr int kTogether = NR > 3 ? 2 : 3;
        const auto *l = late();
        const int last = l->nshare - 1;
        const size_t stride = (size_t)l->T * (size_t)l->H * 4;
        const char *const base = reinterpret_cast<const char *>(l->partial) + (size_t)tok0 * (size_t)l->H * 4;
        f4 u[kTogether][NR][MT], sum[NR][MT];
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int m = 0; m < MT; m++) sum[j][m] = f4{0.f, 0.f, 0.f, 0.f};
        auto add = [&](f4 (&v)[NR][MT]) {
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int m = 0; m < MT; m++) sum[j][m] += v[j][m];
        };
        for (int o = 0; o < last; o += kTogether) {  // o + q: the others, counted without `mine`
#pragma unroll
            for (int q = 0; q < kTogether; q++) {
                const int p = min(o + q, last - 1);
                const char *src = base + (size_t)(p + (p >= mine ? 1 : 0)) * stride;
#pragma unroll
                for (int j = 0; j < NR; j++)
#pragma unroll
                    for (int m = 0; m < MT; m++) el_ask(u[q][j][m], tile_at(m, j) + lane * 16, src);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int q = 0; q < kTogether; q++)
#pragma unroll
                for (int j = 0; j < NR; j++)
#pragma unroll
                    for (int m = 0; m < MT; m++) el_tie(u[q][j][m]);
#pragma unroll
            for (int q = 0; q < kTogether; q++) {
                if (o + q >= last) continue;  // uniform
                if (o + q == mine) add(V);
                add(u[q]);
            }
        }
        if (mine == last) add(V);
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int m = 0; m < MT; m++) V[j][m] = sum[j][m];
    };
    if constexpr (MODE == 3) {
        ask_vectors();
        ring_start();
    } else if constexpr (MODE == 2) {
        ask_vectors();
        sum_shares();
    } else {
        ask_vectors();
        ask_residual(V);
        ring_start();
    }
    if constexpr (kFirst) keep_residual(V);
    el_tie(tab);
#pragma unroll
    for (int i = 0; i < kElRowRegs; i++) el_tie(desc[i]);
    slots[2] = __builtin_amdgcn_readlane(tab, kElTabSlots) * 1024;
    el_barrier();

    const unsigned kx = (unsigned)((gbit ^ r16) & 15) << 4;
    const unsigned hbuf = a.hbuf;
    // the lane's token row in the strip and in a hidden chunk, held: worked out for every block-row, the two products took as
    // long as eight other vector instructions
    unsigned row_x = (unsigned)r16 * xs, row_h = (unsigned)r16 * a.hs;
    asm volatile("" : "+v"(row_x), "+v"(row_h));

    // LayerNorm of V (+ add) in place; the result is also rounded into X.  A wave sums its features of a token and their
    // squared distances from its own mean; the waves exchange both through LDS once, and the second moment about the
    // common mean is the sum of theirs and of the distances of their means.  A wave with fewer than NR block-rows repeats
    // its first one with weight zero, so that nothing here is under a branch and all reads go out together.
    auto vec_of = [&](h4 (&v)[NR], const _Float16 *src) {
        const int g = el_here(lane >> 4);
#pragma unroll
        for (int j = 0; j < NR; j++) v[j] = *reinterpret_cast<const h4 *>(src + max(rb[j], 0) * 16 + g * 4);
    };
    // features of this wave, and of the four waves whose sums this lane adds (one over them; 0 for a wave without any)
    const int own_rows = __builtin_amdgcn_readlane(tab, kElTabCount + wave);
    // A binary16 value added to a binary32 one in one instruction (v_fma_mix: converted, times one, plus; the same bits as a
    // conversion and an addition).  Four waves share a SIMD's vector unit, and a LayerNorm is bound by its instructions.
    auto add_half = [&](f4 &v, h4 b, float one) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = __builtin_fmaf((float)b[e], one, v[e]);
    };
    auto opaque_one = [] {
        float one = 1.0f;
        asm volatile("" : "+v"(one));
        return one;
    };
    auto norm = [&](const _Float16 *add, const _Float16 *gam, const _Float16 *bet, float eps) {
        const int r16 = el_here(lane & 15), g = el_here(lane >> 4), gbit = g & 1;
        float mean[MT], rstd[MT], n_of[4], inv_of[4], live[NR];
#pragma unroll
        for (int j = 0; j < NR; j++) live[j] = here(rb[j]) >= 0 ? 1.0f : 0.0f;
        float inv_own;
        if (H == kElWaves * 16 * NR) {  // uniform: every wave holds NR
#pragma unroll
            for (int k = 0; k < 4; k++) {
                n_of[k] = (float)(NR * 16);
                inv_of[k] = 1.0f / (float)(NR * 16);
            }
            inv_own = 1.0f / (float)(NR * 16);
        } else {
            const int own_here = here(own_rows);
            inv_own = own_here ? 1.0f / (float)(own_here * 16) : 0.0f;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int rows_of = __shfl(tab, kElTabCount + g * 4 + k, 64);
                n_of[k] = (float)(rows_of * 16);
                inv_of[k] = rows_of ? __builtin_amdgcn_rcpf(n_of[k]) : 0.0f;
            }
        }
        if (add) {  // uniform
            h4 bv[NR];
            vec_of(bv, add);
            const float one = opaque_one();
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int m = 0; m < MT; m++) add_half(V[j][m], bv[j], one);
        }
        float2 *rd = reinterpret_cast<float2 *>(red);
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float s = 0.0f, q = 0.0f;
#pragma unroll
            for (int j = 0; j < NR; j++) s = __builtin_fmaf((V[j][m][0] + V[j][m][1]) + (V[j][m][2] + V[j][m][3]), live[j], s);
            s = rows_sum(s);
            const float own = s * inv_own;
#pragma unroll
            for (int j = 0; j < NR; j++) {
                float t = 0.0f;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float d = V[j][m][e] - own;
                    t = __builtin_fmaf(d, d, t);
                }
                q = __builtin_fmaf(t, live[j], q);
            }
            q = rows_sum(q);
            if (g == 0) rd[(wave * MT + m) * 16 + r16] = float2{s, q};
        }
        el_barrier();
        const float inv_h = ET_EL_ARG(inv_h);
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float2 part_of[4];
            float s = 0.0f, q = 0.0f;
#pragma unroll
            for (int k = 0; k < 4; k++) part_of[k] = rd[((g * 4 + k) * MT + m) * 16 + r16];
#pragma unroll
            for (int k = 0; k < 4; k++) s += part_of[k].x;
            mean[m] = rows_sum(s) * inv_h;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float d = __builtin_fmaf(part_of[k].x, inv_of[k], -mean[m]);
                q += __builtin_fmaf(d * d, n_of[k], part_of[k].y);
            }
            rstd[m] = rsqrtf(rows_sum(q) * inv_h + eps);
        }
        h4 gm[NR], bt[NR];
        vec_of(gm, gam);
        vec_of(bt, bet);
        unsigned xrow = r16 * xs + gbit * 8;  // (once; sunk under the branches it is a product for each)
        asm volatile("" : "+v"(xrow));
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int m = 0; m < MT; m++) {
                h4 o;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    V[j][m][e] = norm_value(V[j][m][e], mean[m], rstd[m], (float)gm[j][e], (float)bt[j][e]);
                    o[e] = (_Float16)V[j][m][e];
                }
                const int u = rb[j] * 2 + (g >> 1);
                if (rb[j] >= 0) *reinterpret_cast<h4 *>(X + (xrow + m * 16 * xs + ((u ^ r16) << 4))) = o;
            }
    };

    // MODE 4, behind the second product: this part's share goes to memory, the parts meet, the shares come back.  False:
    // the rest is left to another part.  `others`: parts whose projection is run here besides this one's.
    unsigned others = 0;
    int who = part;
    auto ask_stream = [&](int s) {  // of the second launch's streams: table, descriptors and first offsets
        const auto *l = late();
        const int cap2 = l->cap2;
        const char *at = l->offs2 + (size_t)s * cap2 * 4;
        offs = at;
        offs_off = (g >> 1) * 16;
        lane_off = lane * 16;
        el_ask_offsets(offs_off, offs);
        el_ask(tab, lane * 4, l->tab2 + (size_t)s * kElTab);
#pragma unroll
        for (int i = 0; i < kElRowRegs; i++) el_ask(desc[i], lane * 4, l->tab2 + (size_t)s * kElTab + (1 + i) * kElTabWords);
        const uint64_t slots_at = (uint64_t)(l->slots2 + (size_t)s * cap2 * 1024);
        slots = i4{(int)(unsigned)slots_at, (int)(unsigned)(slots_at >> 32), cap2 * 1024, kElBufferWord};
    };
    auto have_stream = [&] {
        el_tie(tab);
#pragma unroll
        for (int i = 0; i < kElRowRegs; i++) el_tie(desc[i]);
        slots[2] = __builtin_amdgcn_readlane(tab, kElTabSlots) * 1024;
    };
    auto store_share = [&] {
        const auto *l = late();
        char *dst = reinterpret_cast<char *>(l->partial + ((size_t)part * l->T + tok0) * l->H);
        const unsigned at16 = el_here(lane) * 16;
#pragma unroll
        for (int j = 0; j < NR; j++)
#pragma unroll
            for (int m = 0; m < MT; m++)
                if (here(rb[j]) >= 0 && m < tiles_here) *reinterpret_cast<f4 *>(dst + (tile_at(m, j) + at16)) = V[j][m];
    };
    auto join = [&]() -> bool {
        ask_stream((ET_EL_ARG(Q) ? part : 0) * kElWaves + wave);
        store_share();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // in the L2
        el_barrier();
        int *got = reinterpret_cast<int *>(red);
        if (wave == 0) {
            const auto *l = late();
            uint32_t *const word = l->join + strip, was;
            asm volatile(ET_EL_ADD : "=&v"(was) : "v"(word), "v"(kMeetArrived) : "memory");
            el_ring_start(lane_off, offs_off, slots, offs);
            asm volatile("s_waitcnt vmcnt(%0)" ::"i"(kElRingAsks) : "memory");
            el_tie(was);
            *got = meet_wait(ElWord{word}, (uint32_t)__builtin_amdgcn_readfirstlane((int)was), part, l->parts, l->Q > 0, l->spin);
        } else {
            el_ring_start(lane_off, offs_off, slots, offs);
        }
        el_barrier();
        const int mask = __builtin_amdgcn_readfirstlane(*got);
        if (mask < 0) return false;
        others = (unsigned)mask;
        el_barrier();  // (`red` is written again)
        sum_others(part);
        have_stream();
        return true;
    };

    const int act = a.act;
    auto write_out = [&] {  // x', once for a strip
        const int H = ET_EL_ONCE(H);
        if (float *const to = ET_EL_ONCE(x32_out)) {
            char *dst = reinterpret_cast<char *>(to + (size_t)tok0 * H);
            const unsigned at16 = el_here(lane) * 16;
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int m = 0; m < MT; m++)
                    if (here(rb[j]) >= 0 && m < tiles_here) *reinterpret_cast<f4 *>(dst + (tile_at(m, j) + at16)) = V[j][m];
        }
        if (_Float16 *const to = ET_EL_ONCE(out16)) {
            const int r16 = el_here(lane & 15), g = el_here(lane >> 4);
            char *dst = reinterpret_cast<char *>(to + (size_t)tok0 * H);
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int m = 0; m < MT; m++)
                    if (here(rb[j]) >= 0 && m < tiles_here)
                        *reinterpret_cast<h4 *>(dst + ((unsigned)(m * 16 + r16) * H * 2 + here(rb[j]) * 32 + g * 8)) =
                            h4{(_Float16)V[j][m][0], (_Float16)V[j][m][1], (_Float16)V[j][m][2], (_Float16)V[j][m][3]};
        }
    };
    auto norm_k = [&](bool first) {
        const int H = ET_EL_ONCE(H);
        const _Float16 *const b2 = vec + 3 * H + ET_EL_ONCE(FF), *const gam = first ? vec + H : b2 + H;
        norm(first ? vec : nullptr, gam, gam + H, first ? ET_EL_ONCE(eps1) : ET_EL_ONCE(eps2));
        if (first && !(kParts && part != 0)) {  // the second product is added to y + b2
            h4 bv[NR];
            vec_of(bv, b2);
            const float one = opaque_one();
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int m = 0; m < MT; m++) add_half(V[j][m], bv[j], one);
        } else if (first) {
#pragma unroll
            for (int j = 0; j < NR; j++)
#pragma unroll
                for (int m = 0; m < MT; m++) V[j][m] = f4{0.f, 0.f, 0.f, 0.f};
        }
    };
    // The segments of a launch (PHASE 0), or of a joined one up to the second product (1) and of the projection (2).
    auto run = [&](auto phase) {
        constexpr int PHASE = decltype(phase)::value;
        int pos = 0, row_no = 0;
        const int first_seg = MODE == 3 || PHASE == 2 ? a.nseg_ff + 1 : MODE == 2 ? a.nseg_ff : 0;
        const int last_seg = a.nseg_ff + (MODE == 1 || PHASE == 1 ? 0 : a.nseg_q);
        for (int seg = first_seg;; seg++) {  // (the shares' sum enters behind the last hidden segment, which holds no rows there)
            const int nrows = __builtin_amdgcn_readlane(tab, kElTabSeg + seg);
            // hidden chunk c is written in segment c + 1 and read in the next; projection chunk c is written in nseg_ff + 1 + c
            const unsigned odd = (seg > a.nseg_ff ? seg - a.nseg_ff : seg) & 1, hb_up = odd ? 0u : hbuf, hb_dn = odd ? hbuf : 0u;
            for (int r = 0; r < nrows; r++) {
                const uint32_t d = (uint32_t)__builtin_amdgcn_readlane(row_no < 64 ? desc[0] : desc[1], row_no & 63);
                row_no++;
                // A SIMD's oldest wave is served first by the memory pipe, which bounds a segment, and the youngest ones end it
                // a third later: more rows left go first (390 -> 382 us at 8 x 128, 1026 -> 1003 at 64 x 128).
                if (nrows - r >= 3) __builtin_amdgcn_s_setprio(3);
                else if (nrows - r == 2) __builtin_amdgcn_s_setprio(2);
                else __builtin_amdgcn_s_setprio(1);
                const int n = d & 255, kind = (d >> 8) & 3, target = (d >> 11) & 1023, bias_at = (d >> 21) * 16;
                const bool hid = (d >> 10) & 1;
                const unsigned base = hid ? row_h + (MT * 16 * xs + hb_dn) : row_x, step = 16 * (hid ? a.hs : xs);
                if constexpr (MODE != 3 && PHASE != 2) {
                    if (kind == kElKindSum) {
#pragma unroll
                        for (int j = 0; j < NR; j++)
                            if (target == j) el_row<MT>(V[j], n, pos, base, step, kx, lane_off, offs_off, slots, offs);
                        continue;
                    }
                }
                const h4 bv = *reinterpret_cast<const h4 *>(vec + bias_at + el_here(lane >> 4) * 4);
                f4 acc[MT];
#pragma unroll
                for (int m = 0; m < MT; m++) acc[m] = f4{(float)bv[0], (float)bv[1], (float)bv[2], (float)bv[3]};
                if (n) el_row<MT>(acc, n, pos, base, step, kx, lane_off, offs_off, slots, offs);
                if (PHASE != 2 && kind == kElKindHidden) {
                    if (act == ET_ACT_GELU) {
#pragma unroll
                        for (int m = 0; m < MT; m++)
#pragma unroll
                            for (int e = 0; e < 4; e++) acc[m][e] = gelu_tanh(acc[m][e]);
                    } else if (act == ET_ACT_RELU) {
#pragma unroll
                        for (int m = 0; m < MT; m++)
#pragma unroll
                            for (int e = 0; e < 4; e++) acc[m][e] = fmaxf(acc[m][e], 0.0f);
                    }
                }
                const int r16 = el_here(lane & 15);
                const unsigned u = (unsigned)target * 2 + (g >> 1);
#pragma unroll
                for (int m = 0; m < MT; m++)
                    *reinterpret_cast<h4 *>(Hb + (row_h + (hb_up + m * 16 * a.hs + ((u ^ r16) << 4) + gbit * 8))) =
                        h4{(_Float16)acc[m][0], (_Float16)acc[m][1], (_Float16)acc[m][2], (_Float16)acc[m][3]};
            }
            const bool first = kFirst && PHASE != 2 && seg == 0;
            if (first || (PHASE == 0 && (MODE == 0 || MODE == 2) && seg == ET_EL_ARG(nseg_ff))) {
                norm_k(first);
                if (!first && part == 0) write_out();
            }
            if (MODE != 1 && PHASE != 1 && seg > ET_EL_ARG(nseg_ff)) {  // the projection's chunk leaves the LDS, whole rows of it at a time
                el_barrier();
                const auto *l = late();
                const int Q = l->Q, hs = l->hs, c = seg - l->nseg_ff - 1, nq = l->nseg_q;
                const uint32_t chunk = (uint32_t)__builtin_amdgcn_readlane(tab, kElTabOut + c);
                const int first_rb = chunk & 0xffff, units = (chunk >> 16) * 2;
                const unsigned char *src = Hb + ((c & 1) ? hbuf : 0u);
                char *const qkv = reinterpret_cast<char *>(l->qkv + (size_t)tok0 * Q + first_rb * 16);
                // both halves of a wave's rows are read ahead of the first store
                for (int t = wave; t < tiles_here * 16; t += kElWaves) {
                    char *dst = qkv + (size_t)(t * Q * 2);
                    for (int u = el_here(lane); u < units; u += 128) {
                        const h8 v = *reinterpret_cast<const h8 *>(src + t * hs + ((u ^ (t & 15)) << 4));
                        const int u2 = u + 64;
                        if (u2 < units) {
                            const h8 v2 = *reinterpret_cast<const h8 *>(src + t * hs + ((u2 ^ (t & 15)) << 4));
                            *reinterpret_cast<h8 *>(dst + u2 * 16) = v2;
                        }
                        *reinterpret_cast<h8 *>(dst + u * 16) = v;
                    }
                }
                if (c == nq - 1) break;
                continue;
            }
            if (seg == last_seg) break;
            el_barrier();
        }
    };
    if constexpr (MODE != 4) {
        run(std::integral_constant<int, 0>{});
        if constexpr (MODE == 1) store_share();
    } else {
        run(std::integral_constant<int, 1>{});
        if (!join()) return;
        norm_k(false);
        if (part == 0 || (others & 1) || ET_EL_ARG(Q) == 0) write_out();
        if (ET_EL_ARG(Q) > 0) {
            el_barrier();
            for (;;) {
                run(std::integral_constant<int, 2>{});
                if (others == 0) break;
                // the projection of a part whose workgroup did not wait
                who = __builtin_ctz(others);
                others &= others - 1;
                el_barrier();  // this one's has left the LDS
                ask_stream(who * kElWaves + wave);
                ring_start();
                have_stream();
            }
        }
        if (wave == 0) {
            const auto *l = late();
            meet_through(ElWord{l->join + strip}, l->parts);
        }
    }
}

template <int MT, int NR, int MODE>
__global__ __launch_bounds__(kElWaves * 64) __attribute__((amdgpu_num_vgpr(kElOwnVgprs))) void encoder_layer_kernel(ET_EL_FIRST, const LayerArgs a) {
    encoder_layer<MT, NR, MODE>(LayerFirst{Z, x, offs, tab, vec, T, H, cap, form}, a);
}
template <int NR> __global__ __launch_bounds__(kElWaves * 64) __attribute__((amdgpu_num_vgpr(kElOwnVgprs))) void encoder_layer_joined_kernel(ET_EL_FIRST, const LayerArgs a) {
    encoder_layer<1, NR, 4>(LayerFirst{Z, x, offs, tab, vec, T, H, cap, form}, a);
}

// slot s = tiles order[2s], order[2s + 1] (bits 28-29: which weight; negative: a zero tile) in lane order: the 16-byte
// piece of lane (r, g) is row r, values 8 (g & 1) .. + 7 of tile g >> 1
struct LayerTiles {
    const _Float16 *t[4];
};
__global__ void layer_gather_kernel(_Float16 *__restrict__ dst, LayerTiles tl, const int32_t *__restrict__ order, int nslots) {
    const int s = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (s >= nslots) return;
    const int src = order[2 * s + (lane >> 5)];
    const int piece = (lane & 15) * 2 + ((lane >> 4) & 1);
    h8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (src >= 0) v = reinterpret_cast<const h8 *>(tl.t[(src >> 28) & 3] + (size_t)(src & 0x0fffffff) * 256)[piece];
    reinterpret_cast<h8 *>(dst + (size_t)s * 512)[lane] = v;
}

}  // namespace et

// The streams of a layer and the geometry they were built for.
struct et_layer_pack_s {
    int T = 0, H = 0, FF = 0, Q = 0;
    int mt = 1, nr = 1, parts = 1, nseg_ff = 0, nseg_q = 0, hbuf = 0, xs = 0, hs = 0;
    size_t lds = 0;
    uint32_t sums[et::kElWaves] = {};
    int second = 0, nstream = 0;  // first stream of the second launch (or of the projection alone), all streams
    int cap = 0, cap2 = 0;        // slots from one stream to the next, before and from there on
    void *slots = nullptr, *offs = nullptr, *tab = nullptr, *vec = nullptr;
    ~et_layer_pack_s() {
        for (void *p : {slots, offs, tab, vec}) (void)et_free(p);
    }
};

using namespace et;

namespace et {

struct HostBsr {
    std::vector<int32_t> rp, ci;
};

static int el_fetch(HostBsr &m, const int32_t *row_ptr, const int32_t *col_idx, int nbr, int nbc, const char *what) {
    m.rp.resize((size_t)nbr + 1);
    ET_HIP(hipMemcpy(m.rp.data(), row_ptr, m.rp.size() * 4, hipMemcpyDeviceToHost));
    ET_REQUIRE(m.rp[0] == 0, ET_ERR_INVALID_ARG, "et_encoder_layer_pack_create: %s: row_ptr must start at 0", what);
    for (int r = 0; r < nbr; r++)
        ET_REQUIRE(m.rp[(size_t)r + 1] >= m.rp[(size_t)r], ET_ERR_INVALID_ARG, "et_encoder_layer_pack_create: %s: row_ptr decreases", what);
    m.ci.resize((size_t)m.rp.back());
    if (!m.ci.empty()) ET_HIP(hipMemcpy(m.ci.data(), col_idx, m.ci.size() * 4, hipMemcpyDeviceToHost));
    for (int32_t c : m.ci)
        ET_REQUIRE(c >= 0 && c < nbc, ET_ERR_INVALID_ARG, "et_encoder_layer_pack_create: %s: column-tile index %d outside [0, %d)", what, c, nbc);
    return ET_OK;
}

static size_t el_lds(int mt, int xs, int hs, int nbuf, int H, int FF, int Q) {
    return (size_t)mt * 16 * (xs + nbuf * hs) + (size_t)2 * kElWaves * mt * 16 * 4 + (size_t)2 * (6 * H + FF + Q);
}

struct ElRow {
    int kind, target, bias, hidden, row;
    std::vector<std::pair<int32_t, int32_t>> tiles;  // (tile with its weight in bits 28-29, byte offset of its column)
    int slots() const { return ((int)tiles.size() + 1) / 2; }
};

}  // namespace et

extern "C" {

int et_encoder_layer_supported(int T, int emdim, int dimFF, int qkv_out) {
    return T > 0 && T % 16 == 0 && emdim >= 16 && emdim % 16 == 0 && emdim <= 1024 && dimFF > 0 && dimFF % 16 == 0 && dimFF <= 4096 &&
           qkv_out >= 0 && qkv_out % 16 == 0 && qkv_out <= 3072;
}

static int el_pack_create(const et_layer_weights *w, int T, int emdim, int dimFF, int qkv_out, int mt, int parts, bool projecting,
                          struct et_layer_pack_s **pack) {
    ET_REQUIRE(pack != nullptr && w != nullptr, ET_ERR_INVALID_ARG, "et_encoder_layer_pack_create: NULL pointer");
    *pack = nullptr;
    ET_REQUIRE(et_encoder_layer_supported(T, emdim, dimFF, qkv_out) == 1, ET_ERR_UNSUPPORTED,
               "et_encoder_layer_pack_create: T=%d emdim=%d dimFF=%d qkv_out=%d outside the kernel's range", T, emdim, dimFF, qkv_out);
    ET_REQUIRE((mt == 1 || mt == 2) && parts >= 1 && parts <= 32 && (parts == 1 || mt == 1), ET_ERR_INVALID_ARG,
               "et_encoder_layer_pack_create: mt=%d parts=%d", mt, parts);
    const int nmat = qkv_out ? 4 : 3;
    for (int i = 0; i < nmat; i++) {
        ET_REQUIRE(w->row_ptr[i] && w->col_idx[i] && w->tiles[i] && w->bias[i], ET_ERR_INVALID_ARG,
                   "et_encoder_layer_pack_create: NULL weight %d", i);
        ET_REQUIRE((reinterpret_cast<uintptr_t>(w->tiles[i]) & 15) == 0, ET_ERR_UNSUPPORTED,
                   "et_encoder_layer_pack_create: the tiles of weight %d must be 16-byte aligned", i);
    }
    for (int i = 0; i < 2; i++)
        ET_REQUIRE(w->gamma[i] && w->beta[i], ET_ERR_INVALID_ARG, "et_encoder_layer_pack_create: NULL norm %d", i);
    const int H = emdim, FF = dimFF, Q = qkv_out, nbH = H / 16, nbF = FF / 16, nbQ = Q / 16;
    parts = std::min(parts, nbF);
    HostBsr mo, mu, md, mq;
    int s = el_fetch(mo, w->row_ptr[0], w->col_idx[0], nbH, nbH, "output projection");
    if (s == ET_OK) s = el_fetch(mu, w->row_ptr[1], w->col_idx[1], nbF, nbH, "first FFN weight");
    if (s == ET_OK) s = el_fetch(md, w->row_ptr[2], w->col_idx[2], nbH, nbF, "second FFN weight");
    if (s == ET_OK && Q) s = el_fetch(mq, w->row_ptr[3], w->col_idx[3], nbQ, nbH, "QKV projection");
    if (s != ET_OK) return s;

    // chunks of hidden features and of the projection, which passes through the same buffers: as few as the LDS allows, of
    // about equal size
    const int xs = (H * 2 + 255) / 256 * 256;
    const int part_rows = (nbF + parts - 1) / parts, part_q = (nbQ + parts - 1) / parts;
    int nchunk = 1, nchunk_q = Q ? 1 : 0, hs = 0, nbuf = 1;
    for (;;) {
        const int cf = (part_rows + nchunk - 1) / nchunk, cq = Q ? (part_q + nchunk_q - 1) / nchunk_q : 0;
        nbuf = nchunk > 1 || nchunk_q > 1 ? 2 : 1;
        hs = (std::max(cf, cq) * 32 + 255) / 256 * 256;
        if (el_lds(mt, xs, hs, nbuf, H, FF, Q) <= kElLds) break;
        ET_REQUIRE(std::max(cf, cq) > 1 && nchunk + nchunk_q + 3 < kElMaxSeg, ET_ERR_UNSUPPORTED,
                   "et_encoder_layer_pack_create: the strip does not fit the LDS");
        (cf >= cq ? nchunk : nchunk_q)++;
    }
    const int nseg_ff = nchunk + 1, nseg = nseg_ff + 1 + nchunk_q;

    // the block-rows of the model width: wave -> rows, balanced over the tiles of both products that sum into them
    const int nr = std::max(1, (nbH + kElWaves - 1) / kElWaves);
    std::vector<std::vector<int>> sums(kElWaves);
    {
        std::vector<int> order((size_t)nbH), load(kElWaves, 0);
        auto cost = [&](int r) { return mo.rp[(size_t)r + 1] - mo.rp[(size_t)r] + (md.rp[(size_t)r + 1] - md.rp[(size_t)r]) / parts; };
        for (int r = 0; r < nbH; r++) order[(size_t)r] = r;
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return cost(x) > cost(y); });
        for (int r : order) {
            int best = -1;
            for (int v = 0; v < kElWaves; v++)
                if ((int)sums[(size_t)v].size() < nr && (best < 0 || load[(size_t)v] < load[(size_t)best])) best = v;
            sums[(size_t)best].push_back(r);
            load[(size_t)best] += cost(r);
        }
    }
    struct Stream {
        std::vector<int32_t> order, tab;
        std::vector<uint32_t> rows;
        std::vector<std::pair<int, int>> offs;
    };
    std::vector<Stream> streams;
    int most_slots = 0;  // of a block-row in a segment (a column may occur in it more than once)
    auto tiles_of = [](const HostBsr &m, int mat, int r) {
        std::vector<std::pair<int32_t, int32_t>> v;
        for (int t = m.rp[(size_t)r]; t < m.rp[(size_t)r + 1]; t++) v.push_back({t | mat << 28, m.ci[(size_t)t] * 32});
        return v;
    };
    // deals `free` to the waves, longest first, on top of what they have in the segment
    auto deal = [](std::vector<std::vector<ElRow>> &seg, std::vector<ElRow> &free) {
        std::vector<int> load(kElWaves, 0);
        for (int v = 0; v < kElWaves; v++)
            for (const ElRow &r : seg[(size_t)v]) load[(size_t)v] += r.slots() + 1;
        std::stable_sort(free.begin(), free.end(), [](const ElRow &x, const ElRow &y) { return x.tiles.size() > y.tiles.size(); });
        for (ElRow &r : free) {
            const int v = (int)(std::min_element(load.begin(), load.end()) - load.begin());
            load[(size_t)v] += r.slots() + 1;  // a block-row costs about a slot besides its slots
            seg[(size_t)v].push_back(std::move(r));
        }
    };
    // vectors in LDS: bo g1 be1 | b1 | b2 g2 be2 | bq
    const int at_b1 = 3 * H, at_bq = 6 * H + FF;
    std::vector<int32_t> chunks_of_q;  // of the streams that are emitted next
    auto emit = [&](const std::vector<std::vector<std::vector<ElRow>>> &segs) {  // [segment][wave]
        for (int v = 0; v < kElWaves; v++) {
            Stream st;
            st.tab.assign(kElTabWords, 0);
            std::copy(chunks_of_q.begin(), chunks_of_q.end(), st.tab.begin() + kElTabOut);
            for (int o = 0; o < kElWaves; o++) st.tab[(size_t)(kElTabCount + o)] = (int)sums[(size_t)o].size();
            for (size_t sg = 0; sg < segs.size(); sg++) {
                st.tab[kElTabSeg + sg] = (int32_t)segs[sg][(size_t)v].size();
                for (const ElRow &r : segs[sg][(size_t)v]) {
                    most_slots = std::max(most_slots, r.slots());
                    st.rows.push_back((uint32_t)r.slots() | (uint32_t)r.kind << 8 | (uint32_t)r.hidden << 10 | (uint32_t)r.target << 11 |
                                      (uint32_t)(r.bias / 16) << 21);
                    for (size_t t = 0; t < r.tiles.size(); t += 2) {
                        const bool two = t + 1 < r.tiles.size();  // else a zero tile on the column of the first
                        st.order.push_back(r.tiles[t].first);
                        st.order.push_back(two ? r.tiles[t + 1].first : -1);
                        st.offs.push_back({r.tiles[t].second, r.tiles[two ? t + 1 : t].second});
                    }
                }
            }
            st.tab[kElTabSlots] = (int32_t)(st.order.size() / 2);
            streams.push_back(std::move(st));
        }
    };
    const auto empty = [] { return std::vector<std::vector<ElRow>>(kElWaves); };
    auto qkv_segments = [&](std::vector<std::vector<std::vector<ElRow>>> &segs, int q, int nq) {
        const int q0 = nbQ * q / nq, n = nbQ * (q + 1) / nq - q0;
        chunks_of_q.clear();
        for (int c = 0; c < nchunk_q; c++) {
            std::vector<ElRow> free;
            const int cb = q0 + n * c / nchunk_q, ce = q0 + n * (c + 1) / nchunk_q;
            chunks_of_q.push_back(cb | (ce - cb) << 16);
            for (int r = cb; r < ce; r++) free.push_back({kElKindQkv, r - cb, at_bq + r * 16, 0, r, tiles_of(mq, 3, r)});
            deal(segs[(size_t)(nseg_ff + 1 + c)], free);
        }
    };
    for (int p = 0; p < parts; p++) {
        std::vector<std::vector<std::vector<ElRow>>> segs((size_t)nseg, empty());
        for (int v = 0; v < kElWaves; v++)
            for (size_t j = 0; j < sums[(size_t)v].size(); j++) {
                const int r = sums[(size_t)v][j];
                ElRow row{kElKindSum, (int)j, 0, 0, r, tiles_of(mo, 0, r)};
                if (!row.tiles.empty()) segs[0][(size_t)v].push_back(std::move(row));
            }
        const int f0 = nbF * p / parts, f1 = nbF * (p + 1) / parts;
        for (int c = 0; c <= nchunk; c++) {
            auto &seg = segs[(size_t)c + 1];
            if (c > 0) {  // the columns of chunk c - 1 of the second product
                const int cb = f0 + (f1 - f0) * (c - 1) / nchunk, ce = f0 + (f1 - f0) * c / nchunk;
                for (int v = 0; v < kElWaves; v++)
                    for (size_t j = 0; j < sums[(size_t)v].size(); j++) {
                        const int r = sums[(size_t)v][j];
                        ElRow row{kElKindSum, (int)j, 0, 1, r, {}};
                        for (int t = md.rp[(size_t)r]; t < md.rp[(size_t)r + 1]; t++) {
                            const int col = md.ci[(size_t)t];
                            if (col >= cb && col < ce) row.tiles.push_back({t | 2 << 28, (col - cb) * 32});
                        }
                        if (!row.tiles.empty()) seg[(size_t)v].push_back(std::move(row));
                    }
            }
            if (c < nchunk) {
                const int cb = f0 + (f1 - f0) * c / nchunk, ce = f0 + (f1 - f0) * (c + 1) / nchunk;
                std::vector<ElRow> free;
                for (int r = cb; r < ce; r++) free.push_back({kElKindHidden, r - cb, at_b1 + r * 16, 0, r, tiles_of(mu, 1, r)});
                deal(seg, free);
            }
        }
        if (parts == 1 && Q) qkv_segments(segs, 0, 1);
        emit(segs);
    }
    const int second = (int)streams.size();
    if (parts > 1 || (projecting && Q))
        for (int p = 0; p < (Q ? parts : 1); p++) {
            std::vector<std::vector<std::vector<ElRow>>> segs((size_t)nseg, empty());
            if (Q) qkv_segments(segs, p, parts);
            emit(segs);
        }
    // the streams of a launch at one distance from each other, so that a wave finds its own without reading anything; a
    // wave requests a ring of slots, and two of offsets, past its own
    size_t cap_of[2] = {0, 0}, most_rows = 0;
    for (size_t i = 0; i < streams.size(); i++) {
        size_t &cap = cap_of[(int)i >= second];
        cap = std::max(cap, streams[i].order.size() / 2);
        most_rows = std::max(most_rows, streams[i].rows.size());
    }
    for (size_t &cap : cap_of) cap = (cap + kElRing - 1) / kElRing * kElRing + kElRing;
    const auto first_slot = [&](size_t i) {
        const size_t ahead = std::min(i, (size_t)second);
        return ahead * cap_of[0] + (i - ahead) * cap_of[1];
    };
    const size_t all_slots = first_slot(streams.size());
    ET_REQUIRE(most_slots <= kElMaxSlots, ET_ERR_UNSUPPORTED,
               "et_encoder_layer_pack_create: %d slots in one block-row, at most %d fit its descriptor", most_slots, kElMaxSlots);
    ET_REQUIRE(most_rows <= 64 * kElRowRegs, ET_ERR_UNSUPPORTED, "et_encoder_layer_pack_create: %zu block-rows in one wave", most_rows);
    std::vector<int32_t> tab(streams.size() * kElTab, 0), order(all_slots * 2, -1);
    std::vector<uint16_t> offs((all_slots + 2 * kElRing) * 2, 0);
    for (size_t i = 0; i < streams.size(); i++) {
        const Stream &st = streams[i];
        std::copy(st.tab.begin(), st.tab.end(), tab.begin() + (long)(i * kElTab));
        std::copy(st.rows.begin(), st.rows.end(), tab.begin() + (long)(i * kElTab + kElTabWords));
        std::copy(st.order.begin(), st.order.end(), order.begin() + (long)(first_slot(i) * 2));
        for (size_t k = 0; k < st.offs.size(); k++) {
            const size_t at = (first_slot(i) + k / kElRing * kElRing) * 2 + k % kElRing;
            offs[at] = (uint16_t)st.offs[k].first;
            offs[at + kElRing] = (uint16_t)st.offs[k].second;
        }
    }

    std::unique_ptr<et_layer_pack_s> p(new (std::nothrow) et_layer_pack_s);
    ET_REQUIRE(p != nullptr, ET_ERR_ALLOC, "et_encoder_layer_pack_create: out of host memory");
    p->T = T, p->H = H, p->FF = FF, p->Q = Q, p->mt = mt, p->nr = nr, p->parts = parts;
    for (int v = 0; v < kElWaves; v++) {
        p->sums[v] = 0xffffffffu;
        for (size_t j = 0; j < sums[(size_t)v].size(); j++)
            p->sums[v] = (p->sums[v] & ~(255u << (8 * j))) | (uint32_t)sums[(size_t)v][j] << (8 * j);
    }
    p->nseg_ff = nseg_ff, p->nseg_q = nchunk_q, p->hbuf = nbuf == 2 ? mt * 16 * hs : 0, p->xs = xs, p->hs = hs;
    p->second = second, p->nstream = (int)streams.size();
    p->cap = (int)cap_of[0], p->cap2 = (int)cap_of[1];
    p->lds = el_lds(mt, xs, hs, nbuf, H, FF, Q);
    auto upload = [](void **dst, const void *src, size_t bytes) -> int {
        const int st = et_malloc(dst, bytes);
        if (st != ET_OK) return st;
        ET_HIP(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
        return ET_OK;
    };
    void *d_order = nullptr;
    const int nslots = (int)(order.size() / 2);
    s = upload(&p->offs, offs.data(), offs.size() * 2);
    if (s == ET_OK) s = upload(&p->tab, tab.data(), tab.size() * 4);
    if (s == ET_OK) s = upload(&d_order, order.data(), order.size() * 4);
    if (s == ET_OK) s = et_malloc(&p->slots, (size_t)nslots * 1024);
    if (s == ET_OK) s = et_malloc(&p->vec, (size_t)2 * (6 * H + FF + Q));
    if (s == ET_OK) {
        const LayerTiles tl{{reinterpret_cast<const _Float16 *>(w->tiles[0]), reinterpret_cast<const _Float16 *>(w->tiles[1]),
                             reinterpret_cast<const _Float16 *>(w->tiles[2]), reinterpret_cast<const _Float16 *>(Q ? w->tiles[3] : nullptr)}};
        layer_gather_kernel<<<(unsigned)((nslots + 3) / 4), 256>>>(static_cast<_Float16 *>(p->slots), tl, static_cast<const int32_t *>(d_order), nslots);
        s = check_launch("layer_gather_kernel");
        const struct { const et_f16 *src; int n; } parts_of[8] = {{w->bias[0], H}, {w->gamma[0], H}, {w->beta[0], H}, {w->bias[1], FF},
                                                                {w->bias[2], H}, {w->gamma[1], H}, {w->beta[1], H}, {Q ? w->bias[3] : nullptr, Q}};
        size_t at = 0;
        for (const auto &v : parts_of) {
            if (s == ET_OK && v.n)
                s = check_hip(hipMemcpyAsync(static_cast<char *>(p->vec) + at, v.src, (size_t)v.n * 2, hipMemcpyDeviceToDevice, nullptr), "hipMemcpyAsync");
            at += (size_t)v.n * 2;
        }
        if (s == ET_OK) s = check_hip(hipDeviceSynchronize(), "hipDeviceSynchronize");
    }
    (void)et_free(d_order);
    if (s != ET_OK) return s;
    *pack = p.release();
    return ET_OK;
}

int et_encoder_layer_pack_create(const et_layer_weights *w, int T, int emdim, int dimFF, int qkv_out, int mt, int parts,
                                 struct et_layer_pack_s **pack) {
    return el_pack_create(w, T, emdim, dimFF, qkv_out, mt, parts, false, pack);
}

int et_encoder_layer_pack_create_projecting(const et_layer_weights *w, int T, int emdim, int dimFF, int qkv_out, int mt, int parts,
                                            struct et_layer_pack_s **pack) {
    return el_pack_create(w, T, emdim, dimFF, qkv_out, mt, parts, true, pack);
}

int et_encoder_layer_pack_destroy(struct et_layer_pack_s *pack) {
    delete pack;
    return ET_OK;
}

}  // extern "C"

namespace et {
template <int MT, int NR, int MODE> static int el_launch(const LayerFirst &f, const LayerArgs &a, size_t lds, hipStream_t stream) {
    auto kernel = [] {
        if constexpr (MODE == 4) return encoder_layer_joined_kernel<NR>;
        else return encoder_layer_kernel<MT, NR, MODE>;
    }();
    static bool raised = false;  // per instantiation
    if (!raised) {
        ET_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kElLds));
        raised = true;
    }
    const unsigned strips = (unsigned)((f.T + MT * 16 - 1) / (MT * 16)), groups = (strips + 7) / 8, rows = std::min(groups, 32768u);
    const dim3 grid = MODE == 0 ? dim3(strips) : dim3(8 * (unsigned)a.parts, rows, (groups + rows - 1) / rows);
    kernel<<<grid, kElWaves * 64, lds, stream>>>(f.Z, f.x, f.offs, f.tab, f.vec, f.T, f.H, f.cap, f.form, a);
    return check_launch("encoder_layer_kernel");
}
template <int MT, int MODE> static int el_dispatch(const LayerFirst &f, const LayerArgs &a, const et_layer_pack_s &p, hipStream_t stream) {
    switch (p.nr) {
        case 1:
        case 2: return el_launch<MT, 2, MODE>(f, a, p.lds, stream);
        case 3: return el_launch<MT, 3, MODE>(f, a, p.lds, stream);
        default: return el_launch<MT, 4, MODE>(f, a, p.lds, stream);
    }
}
}  // namespace et

// the arguments a pack gives, and those of its second launch (or of the projection alone)
static LayerArgs el_args(const et_layer_pack_s &p) {
    LayerArgs a{};
    a.slots = static_cast<const char *>(p.slots);
    std::copy(p.sums, p.sums + kElWaves, a.sums);
    a.inv_h = 1.0f / (float)p.H;
    a.T = p.T, a.H = p.H, a.FF = p.FF, a.Q = p.Q;
    a.hs = p.hs, a.nseg_ff = p.nseg_ff, a.nseg_q = p.nseg_q, a.hbuf = p.hbuf, a.parts = a.nshare = p.parts;
    return a;
}
static LayerFirst el_first(const et_layer_pack_s &p) {
    return {nullptr, nullptr, static_cast<const char *>(p.offs), static_cast<const int32_t *>(p.tab), static_cast<const _Float16 *>(p.vec),
            p.T,     p.H,     p.cap, (unsigned)(p.xs >> 8) | (unsigned)((6 * p.H + p.FF + p.Q) >> 3) << 16};
}
static void el_second(LayerFirst &f, LayerArgs &a, const et_layer_pack_s &p) {
    f.tab += (size_t)p.second * kElTab;
    a.slots += (size_t)p.second * p.cap * 1024;
    f.offs += (size_t)p.second * p.cap * 4;
    f.cap = p.cap2;
    a.parts = p.Q ? p.parts : 1;  // without a projection only the normalisation is left
}

extern "C" int et_encoder_layer_pack_streams(const struct et_layer_pack_s *p, et_span *streams) {
    ET_REQUIRE(p && streams, ET_ERR_INVALID_ARG, "et_encoder_layer_pack_streams: NULL pointer");
    *streams = {p->slots, ((size_t)p->second * p->cap + (size_t)(p->nstream - p->second) * p->cap2) * 1024};
    return ET_OK;
}

extern "C" int et_encoder_layer_project_f16(const struct et_layer_pack_s *p, const et_f16 *x16, et_f16 *QKV, et_stream stream) {
    ET_REQUIRE(p && x16 && QKV, ET_ERR_INVALID_ARG, "et_encoder_layer_project_f16: NULL pointer");
    ET_REQUIRE(p->Q > 0 && p->nstream > p->second, ET_ERR_UNSUPPORTED,
               "et_encoder_layer_project_f16: the pack has no projection of its own (parts=%d qkv_out=%d)", p->parts, p->Q);
    ET_REQUIRE(((reinterpret_cast<uintptr_t>(x16) | reinterpret_cast<uintptr_t>(QKV)) & 15) == 0, ET_ERR_UNSUPPORTED,
               "et_encoder_layer_project_f16: x16 and QKV must be 16-byte aligned");
    LayerArgs a = el_args(*p);
    LayerFirst f = el_first(*p);
    f.Z = reinterpret_cast<const _Float16 *>(x16);
    a.qkv = reinterpret_cast<_Float16 *>(QKV);
    el_second(f, a, *p);
    return el_launch<1, 2, 3>(f, a, p->lds, as_stream(stream));  // one token tile a workgroup, whatever the pack's strips are: the sums are the same
}

// Workgroups of equal id modulo 8 share an XCD, as they are dealt out: looked at once per device.
namespace et {
__global__ void el_xcc_kernel(uint32_t *xcc) {
    if (threadIdx.x == 0) xcc[blockIdx.x] = __builtin_amdgcn_s_getreg((3 << 11) | 20) & 15u;  // XCC_ID
}
static int el_xcd_by_id(bool *by_id) {
    static std::mutex lock;
    static int known[64] = {};  // 1: yes, 2: no
    int dev = 0;
    ET_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> hold(lock);
    int &k = known[std::min(dev, 63)];
    if (!k) {
        constexpr int n = 512;
        void *d = nullptr;
        int s = et_malloc(&d, n * sizeof(uint32_t));
        uint32_t h[n];
        if (s == ET_OK) {
            el_xcc_kernel<<<n, 64>>>(static_cast<uint32_t *>(d));
            s = check_launch("el_xcc_kernel");
            if (s == ET_OK) s = check_hip(hipMemcpy(h, d, sizeof h, hipMemcpyDeviceToHost), "hipMemcpy");
        }
        (void)et_free(d);
        if (s != ET_OK) return s;
        k = 1;
        for (int i = 8; i < n; i++)
            if (h[i] != h[i % 8]) k = 2;
    }
    *by_id = k == 1;
    return ET_OK;
}
}  // namespace et

extern "C" int et_encoder_layer_joins(const struct et_layer_pack_s *p, int *joins) {
    ET_REQUIRE(p && joins, ET_ERR_INVALID_ARG, "et_encoder_layer_joins: NULL pointer");
    bool by_id = false;
    const int s = p->parts > 1 && p->parts <= kMeetMaxParts ? el_xcd_by_id(&by_id) : ET_OK;
    *joins = by_id;
    return s;
}

static int el_run(const struct et_layer_pack_s *p, const et_f16 *Z, const float *x32, const et_f16 *x16, float *x32_out,
                  et_f16 *out16, et_f16 *QKV, float *partial, uint32_t *join, int spin, int act, float eps1, float eps2, et_stream stream) {
    ET_REQUIRE(p && Z && (x32 || x16) && (p->Q == 0 || QKV) && (p->parts == 1 || partial), ET_ERR_INVALID_ARG,
               "et_encoder_layer_f32: NULL pointer");
    ET_REQUIRE(act >= ET_ACT_NONE && act <= ET_ACT_GELU, ET_ERR_INVALID_ARG, "et_encoder_layer_f32: act=%d", act);
    const auto at = [](const void *q) { return reinterpret_cast<uintptr_t>(q); };
    ET_REQUIRE(((at(Z) | at(x32) | at(x32_out) | at(QKV) | at(partial)) & 15) == 0, ET_ERR_UNSUPPORTED,
               "et_encoder_layer_f32: Z, x32, x32_out, QKV and partial must be 16-byte aligned");
    ET_REQUIRE(((at(x16) | at(out16)) & 7) == 0, ET_ERR_UNSUPPORTED, "et_encoder_layer_f32: x16 and out16 must be 8-byte aligned");
    const size_t x32_bytes = (size_t)p->T * p->H * 4;
    ET_REQUIRE(!x32 || !x32_out || at(x32_out) >= at(x32) + x32_bytes || at(x32) >= at(x32_out) + x32_bytes, ET_ERR_INVALID_ARG,
               "et_encoder_layer_f32: x32_out overlaps x32");
    LayerArgs a = el_args(*p);
    LayerFirst f = el_first(*p);
    f.Z = reinterpret_cast<const _Float16 *>(Z);
    f.x = x32 ? static_cast<const void *>(x32) : x16;
    f.form |= x32 ? 0u : 1u << 8;
    a.x32_out = x32_out;
    a.out16 = reinterpret_cast<_Float16 *>(out16);
    a.qkv = reinterpret_cast<_Float16 *>(QKV);
    a.partial = partial;
    a.act = act;
    a.eps1 = eps1, a.eps2 = eps2;
    hipStream_t st = as_stream(stream);
    if (join) {
        LayerArgs second = a;
        LayerFirst first = f;
        el_second(first, second, *p);
        a.slots2 = second.slots, a.offs2 = first.offs, a.tab2 = first.tab, a.cap2 = first.cap;
        a.join = join, a.spin = spin;
        return el_dispatch<1, 4>(f, a, *p, st);
    }
    if (p->parts == 1) return p->mt == 2 ? el_dispatch<2, 0>(f, a, *p, st) : el_dispatch<1, 0>(f, a, *p, st);
    LayerFirst shares = f;
    shares.form = (f.form & 0xffffu) | (unsigned)((6 * p->H + p->FF) >> 3) << 16;  // (the projection's bias is the second launch's)
    const int s = el_dispatch<1, 1>(shares, a, *p, st);
    if (s != ET_OK) return s;
    el_second(f, a, *p);
    return el_dispatch<1, 2>(f, a, *p, st);
}

extern "C" int et_encoder_layer_f32(const struct et_layer_pack_s *p, const et_f16 *Z, const float *x32, const et_f16 *x16, float *x32_out,
                                    et_f16 *out16, et_f16 *QKV, float *partial, int act, float eps1, float eps2, et_stream stream) {
    return el_run(p, Z, x32, x16, x32_out, out16, QKV, partial, nullptr, 0, act, eps1, eps2, stream);
}

extern "C" int et_encoder_layer_joined_f32(const struct et_layer_pack_s *p, const et_f16 *Z, const float *x32, const et_f16 *x16, float *x32_out,
                                           et_f16 *out16, et_f16 *QKV, float *partial, uint32_t *join, int spin, int act, float eps1, float eps2,
                                           et_stream stream) {
    int joins = 0;
    ET_REQUIRE(join && (reinterpret_cast<uintptr_t>(join) & 3) == 0 && spin >= 0, ET_ERR_INVALID_ARG, "et_encoder_layer_joined_f32: join=%p spin=%d",
               static_cast<void *>(join), spin);
    const int s = et_encoder_layer_joins(p, &joins);
    if (s != ET_OK) return s;
    ET_REQUIRE(joins, ET_ERR_UNSUPPORTED, "et_encoder_layer_joined_f32: one part, more than %d, or a device that deals workgroups otherwise", kMeetMaxParts);
    return el_run(p, Z, x32, x16, x32_out, out16, QKV, partial, join, spin, act, eps1, eps2, stream);
}
