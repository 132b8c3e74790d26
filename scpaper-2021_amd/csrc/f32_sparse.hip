// binary32 twins of the Linear layers over the tile-sparse, 1x16 vector-sparse and CSR
// weight containers: values are stored, multiplied and accumulated in binary32
// (MFMA 16x16x4 f32 for the tile and vector forms, vector FMA for CSR).  They are the
// verification path of pruned fp32 models, as the dense twins are for dense ones; the
// reference's kernels are binary16 only (Linear/Linear.h:9).
//
// Operand feed shared by the tile and vector forms: v_mfma_f32_16x16x4_f32 contracts 4
// values of k per instruction, lane (r = lane % 16, q = lane / 16) supplying A[r][k_q] and
// B[k_q][r].  A sum over k does not care which k a lane brings as long as A and B bring the
// same one, so lane q holds k = 4q .. 4q+3 of a 16-wide cell (one 16-byte load per operand)
// and the cell takes four instructions, the j-th contracting k = {j, 4+j, 8+j, 12+j}.
#include <algorithm>

#include "common.hip.h"

#define ET_LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))

namespace et {

struct Bsr32Args {
    const float *X;
    const int32_t *row_ptr, *col_idx;
    const float *tiles, *bias;
    int T, in, out;
    int die_bits;  // 0 to 3: see strip_of
    float *Y;
    int act;
};
// one by one, those that the requests need in front: preloaded into scalar registers (six layers of 256 rows, seven launches
// each, 247 -> 242 us)
#define ET_BSR32_PARAMS const float *X, const int32_t *row_ptr, const int32_t *col_idx, const float *tiles, const float *bias_of, int T, int in, int out, int die_bits, float *Y, int act
#define ET_BSR32_ARGS(A) (A).X, (A).row_ptr, (A).col_idx, (A).tiles, (A).bias, (A).T, (A).in, (A).out, (A).die_bits, (A).Y, (A).act
#define ET_BSR32_TAKE const Bsr32Args a{X, row_ptr, col_idx, tiles, bias_of, T, in, out, die_bits, Y, act}

// row of the grid (its size, which only more than 32768 rows need, would be read from memory)
__device__ __forceinline__ unsigned grid_row() { return blockIdx.z ? blockIdx.y + blockIdx.z * gridDim.y : blockIdx.y; }

__device__ __forceinline__ f4 mfma_cell_f32(const float4 w, const float4 x, f4 acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, x.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, x.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.z, x.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.w, x.w, acc, 0, 0, 0);
    return acc;
}

__device__ __forceinline__ f4 bias_cell_f32(const float *bias, int f0) {
    return bias ? f4{bias[f0], bias[f0 + 1], bias[f0 + 2], bias[f0 + 3]} : f4{0.f, 0.f, 0.f, 0.f};
}

// lane (r, q) holds features f0 + 4q .. 4q+3 of token `tok`: bias, activation, one 16-byte store
__device__ __forceinline__ void store_cell_f32(float *Y, f4 bias, f4 acc, int tok, int T, int out, int f0, int act) {
    if (tok >= T) return;
    float4 o;
    float *po = reinterpret_cast<float *>(&o);
#pragma unroll
    for (int e = 0; e < 4; e++) po[e] = apply_act(acc[e] + bias[e], act);
    *reinterpret_cast<float4 *>(Y + (size_t)tok * out + f0) = o;
}

// ---- 16x16 tiles ----------------------------------------------------------------
// Tile t of a block-row: A = its 16 x 16 weights (row = feature), B = X[16 tokens][16 col_idx[t] ..], four products of 32
// cycles.  A verification batch has few (block-row, 16 tokens) pairs with a chain of loads and products each, so what
// bounds it is the length of that chain; with many pairs it is the reads of X and of the weights.  Three forms: one that
// keeps pairs short, one for many pairs with the tokens' rows in LDS, and one for many pairs of an input too wide for
// that, in which a wave multiplies a tile with several blocks of 16 tokens.
//
// The wide form: a wave has one block-row and MT blocks of 16 tokens; the four waves of a workgroup take neighbouring
// block-rows over the same tokens and meet in the cache.
template <int MT> __global__ __launch_bounds__(256) void bsr16_linear_wide_f32_kernel(ET_BSR32_PARAMS) {
    ET_BSR32_TAKE;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, q = lane >> 4;
    const int br = blockIdx.x * 4 + wave, tok0 = (int)grid_row() * (MT * 16);
    if (br >= (a.out >> 4) || tok0 >= a.T) return;  // no barrier below
    const float *xrow[MT];
    f4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {  // rows past the end: the last one, not stored
        xrow[m] = a.X + (size_t)min(tok0 + m * 16 + r16, a.T - 1) * a.in + 4 * q;
        acc[m] = f4{0.f, 0.f, 0.f, 0.f};
    }
    const int ts = a.row_ptr[br], te = a.row_ptr[br + 1];
    const float *wp = a.tiles + (size_t)ts * 256 + r16 * 16 + 4 * q;
#pragma unroll 2
    for (int t = ts; t < te; t++, wp += 256) {
        const int c = a.col_idx[t];
        const float4 w = *reinterpret_cast<const float4 *>(wp);
#pragma unroll
        for (int m = 0; m < MT; m++) acc[m] = mfma_cell_f32(w, *reinterpret_cast<const float4 *>(xrow[m] + c * 16), acc[m]);
    }
#pragma unroll
    for (int m = 0; m < MT; m++) store_cell_f32(a.Y, bias_cell_f32(a.bias, br * 16 + 4 * q), acc[m], tok0 + m * 16 + r16, a.T, a.out, br * 16 + 4 * q, a.act);
}

// The short form, for few pairs.  Against the wide one, us, at 80 %: 256 tokens 768 -> 2304 8.0 / 10.4, 768 -> 3072 8.4 / 11.0,
// 3072 -> 768 8.9 / 21.5; 16 tokens 4.0 / 6.2 and 4.8 / 14.7.
//
// The waves of a workgroup share one (block-row, 16 tokens), each every WAVES-th tile; the sums meet in LDS and are added
// in the order of the waves.  A lane reads the column index of one of its wave's tiles, 64 at a time, so no operand waits
// for an index from memory, and kAhead tiles are requested ahead of the products.  The requests are straight-line and go
// through buffer resources that end with the tiles: one past the last moves nothing.  (Its whole offset is in the vector
// operand, which the bounds check is documented to look at.  Asking for the last tile again, as before, cost 16 tokens of a 6-layer stack of 768 at 80 % 13 us of 175).  8 ahead are slower, 300 us against 292 for 256
// tokens of that stack: it is no longer the latency of a load that bounds a pair.
//
// The workgroups of one die (blockIdx.x % 8) keep to a part of the strips and a part of the columns of the grid, so that what an L2
// has to fetch is a part of X and a part of the weights: 2^die_bits parts of the strips, 8 / 2^die_bits of the columns.  (By shifts:
// two divisions by the number of parts cost every wave 0.3 us.)
__device__ __forceinline__ int strip_of(int die_bits) {
    return (int)(blockIdx.x & ((1u << die_bits) - 1)) + ((int)grid_row() << die_bits);
}
__device__ __forceinline__ int column_of(int die_bits) { return (int)((blockIdx.x & 7) >> die_bits) + ((int)(blockIdx.x >> 3) << (3 - die_bits)); }

constexpr int kAhead = 4;
constexpr int kRawBuffer = 0x00020000;   // word 3 of a resource: raw, 32-bit data
constexpr unsigned kPastEnd = 0x7fffff00;  // an offset past the end of any resource here, also with a row's added to it (below 2^32)
constexpr int kSplitMaxIn = 1 << 24;     // 16 rows of X lie within the offsets of a resource, and below kPastEnd
template <int WAVES>
__global__ __launch_bounds__(WAVES * 64) void bsr16_linear_split_f32_kernel(ET_BSR32_PARAMS) {
    ET_BSR32_TAKE;
    __shared__ f4 part[WAVES][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, q = lane >> 4;
    const int strip = strip_of(a.die_bits), br = column_of(a.die_bits);
    if (strip * 16 >= a.T || br >= (a.out >> 4)) return;  // padding of the grid (whole workgroup)
    const int tok = strip * 16 + r16;
    const f4 bias = bias_cell_f32(a.bias, br * 16 + 4 * q);
    const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.X) + (size_t)strip * 16 * a.in, 0, 16 * a.in * 4, kRawBuffer);
    const unsigned xo = (unsigned)(min(r16, a.T - 1 - strip * 16) * a.in + 4 * q) * 4;  // rows past the end: the last one, not stored
    const int wo = (r16 * 16 + 4 * q) * 4;
    f4 acc = f4{0.f, 0.f, 0.f, 0.f};
    const int ts = a.row_ptr[br] + wave, te = a.row_ptr[br + 1];
    const int n = ts < te ? (te - ts + WAVES - 1) / WAVES : 0;  // tiles of this wave
    for (int base = 0; base < n; base += 64) {
        const int here = min(n - base, 64), t0 = ts + base * WAVES;
        const int cols = a.col_idx[t0 + min(lane, here - 1) * WAVES];
        const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.tiles) + (size_t)t0 * 256, 0, ((here - 1) * WAVES + 1) * 1024, kRawBuffer);
        float4 w[kAhead], x[kAhead];
        auto ask = [&](int slot, int i) {
            const unsigned xat = i < here ? (unsigned)__builtin_amdgcn_readlane(cols, i & 63) * 64 : kPastEnd;
            w[slot] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(wr, wo + i * WAVES * 1024, 0, 0));
            x[slot] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(xo + xat), 0, 0));
        };
#pragma unroll
        for (int s = 0; s < kAhead; s++) ask(s, s);
        for (int i = 0; i < here; i += kAhead) {
#pragma unroll
            for (int s = 0; s < kAhead; s++) {
                if (i + s < here) acc = mfma_cell_f32(w[s], x[s], acc);  // uniform
                ask(s, i + s + kAhead);
            }
        }
    }
    if constexpr (WAVES > 1) {
        part[wave][lane] = acc;
        __syncthreads();
        if (wave) return;
#pragma unroll
        for (int v = 1; v < WAVES; v++) acc += part[v][lane];
    }
    store_cell_f32(a.Y, bias, acc, tok, a.T, a.out, br * 16 + 4 * q, a.act);
}

// Eight waves, eight neighbouring block-rows, 16 tokens, whose rows of X lie in LDS (kStripPad floats between two rows:
// the 16 cells of a fragment read lie in different banks).  Read from memory, the fragment of a tile is 16 rows x 64 bytes,
// and 16 neighbouring lanes touch 16 lines: with many tiles that is what the kernels above wait for.  The rows go straight
// to LDS, all of them requested before anything is waited for, with the first weights behind them, which stay in flight
// across the barrier (waited for with the rows, 256 tokens 768 -> 2304 at 80 % 8.05 us, now 6.7; 2048 768 -> 3072 35.8 / 29.1).
// Against the wide form: 4096 tokens 768 -> 3072 at 50 / 80 / 90 / 95 % 111 / 172, 55 / 79, 41 / 49, 34 / 33; ten shapes of 1024 to 8192
// tokens 0.46 - 0.69 of its time at 50 %, 0.55 - 0.77 at 80, 0.65 - 0.89 at 90, 0.78 - 1.11 at 95.
constexpr int kStripPad = 4, kStripWaves = 8;
__global__ __launch_bounds__(kStripWaves * 64) void bsr16_linear_strip_f32_kernel(ET_BSR32_PARAMS) {
    ET_BSR32_TAKE;
    extern __shared__ __align__(16) unsigned char strip_smem[];
    float *xs = reinterpret_cast<float *>(strip_smem);  // [16][in + kStripPad]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, q = lane >> 4;
    const int strip = strip_of(a.die_bits), br = column_of(a.die_bits) * kStripWaves + wave;
    if (strip * 16 >= a.T || br - wave >= (a.out >> 4)) return;  // padding of the grid (whole workgroup)
    const int ld = a.in + kStripPad, tok0 = strip * 16, quads = a.in >> 2;
    const bool mine = br < (a.out >> 4);  // uniform
    const int at = mine ? br : 0, ts = a.row_ptr[at], te = a.row_ptr[at + 1];  // (used behind the rows' requests)
    for (int row = wave; row < 16; row += kStripWaves) {  // past the end: the last row, not stored
        const float *src = a.X + (size_t)min(tok0 + row, a.T - 1) * a.in;
        for (int i = 0; i < quads; i += 64)
            if (i + lane < quads) {
                // (behind the compiler's back: it would wait for every request, the weights among them, before the LDS is read)
                const unsigned to = (unsigned)(uintptr_t)ET_LDS_PTR(xs + row * ld + i * 4);
                asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane * 16), "s"(src + i * 4), "s"(to) : "memory", "m0");
            }
    }
    const int n = mine ? te - ts : 0;
    const f4 bias = bias_cell_f32(mine ? a.bias : nullptr, br * 16 + 4 * q);
    const float *xp = xs + r16 * ld + 4 * q;
    const int wo = (r16 * 16 + 4 * q) * 4;
    f4 acc = f4{0.f, 0.f, 0.f, 0.f};
    // the strip is complete (every wave passes one of the two once): behind the requests for weights, at most 4 of which
    // may be outstanding, or behind the rows alone
    if (n == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
    for (int base = 0; base < n; base += 64) {
        const int here = min(n - base, 64), t0 = ts + base;
        const int cols = a.col_idx[t0 + min(lane, here - 1)];
        const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.tiles) + (size_t)t0 * 256, 0, here * 1024, kRawBuffer);
        float4 w[kAhead];
        auto ask = [&](int slot, int i) {
            w[slot] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(wr, wo + i * 1024, 0, 0));
        };
#pragma unroll
        for (int s = 0; s < kAhead; s++) ask(s, s);
        if (base == 0) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAhead) : "memory");
            __syncthreads();
        }
        for (int i = 0; i < here; i += kAhead) {
#pragma unroll
            for (int s = 0; s < kAhead; s++) {
                if (i + s < here)  // uniform
                    acc = mfma_cell_f32(w[s], *reinterpret_cast<const float4 *>(xp + __builtin_amdgcn_readlane(cols, i + s) * 16), acc);
                ask(s, i + s + kAhead);
            }
        }
    }
    if (mine) store_cell_f32(a.Y, bias, acc, tok0 + r16, a.T, a.out, br * 16 + 4 * q, a.act);
}

// ---- 1x16 vectors ---------------------------------------------------------------
struct V16F32Args {
    const int32_t *tile_idx, *row_idx;
    const float *data, *bias, *X;
    float *Y;
    int T, in, out, act;
};

constexpr int kV16F32Ld = 20;  // floats per row of the per-wave 16 x 16 weight cell (16-byte aligned rows)

// A wave owns one row-set and MT blocks of 16 tokens.  For each part that holds vectors it
// clears its private 16 x 16 cell in LDS, drops the vectors into the rows they name
// (row_idx % 16, at most 16 of them) and multiplies with the cell as the A operand.  LDS
// operations of one wave execute in issue order: clear, fill and read need no barrier.
template <int MT>
__global__ __launch_bounds__(256) void vec1x16_linear_f32_kernel(const V16F32Args a) {
    __shared__ __align__(16) float cells[4][16 * kV16F32Ld];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, q = lane >> 4;
    const int npart = a.in >> 4;
    const int rset = blockIdx.x * 4 + wave;
    if (rset >= (a.out >> 4)) return;  // no workgroup barrier below
    const int tok0 = blockIdx.y * (MT * 16);
    float *cell = cells[wave];
    const int32_t *cellp = a.tile_idx + (size_t)rset * (npart + 1);
    const float *xrow[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const int tok = tok0 + m * 16 + r16;
        xrow[m] = a.X + (size_t)(tok < a.T ? tok : a.T - 1) * a.in + 4 * q;
    }
    f4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) acc[m] = f4{0.f, 0.f, 0.f, 0.f};
    const float4 zero4 = float4{0.f, 0.f, 0.f, 0.f};
    const int fill_vec = lane >> 2, fill_q = lane & 3;  // four lanes copy one vector
    for (int p = 0; p < npart; p++) {
        const int s = cellp[p], e = cellp[p + 1];
        if (e == s) continue;  // wave-uniform
        *reinterpret_cast<float4 *>(cell + fill_vec * kV16F32Ld + fill_q * 4) = zero4;
        const int idx = s + fill_vec;
        if (idx < e) {
            const int row = a.row_idx[idx] & 15;
            *reinterpret_cast<float4 *>(cell + row * kV16F32Ld + fill_q * 4) =
                *reinterpret_cast<const float4 *>(a.data + (size_t)idx * 16 + fill_q * 4);
        }
        const float4 w = *reinterpret_cast<const float4 *>(cell + r16 * kV16F32Ld + 4 * q);
#pragma unroll
        for (int m = 0; m < MT; m++)
            acc[m] = mfma_cell_f32(w, *reinterpret_cast<const float4 *>(xrow[m] + p * 16), acc[m]);
    }
#pragma unroll
    for (int m = 0; m < MT; m++)
        store_cell_f32(a.Y, bias_cell_f32(a.bias, rset * 16 + 4 * q), acc[m], tok0 + m * 16 + r16, a.T, a.out, rset * 16 + 4 * q, a.act);
}

// ---- CSR ------------------------------------------------------------------------
struct Csr32Args {
    const int32_t *indptr, *indices;
    const float *data, *bias, *X;
    float *Y;
    int T, in, out, act;
};

// A wave takes 16 tokens and four output features at a time: lane (tok = lane % 16,
// g = lane / 16) accumulates feature o0 + g of its token over that feature's non-zeros
// (index and value are the same for the 16 lanes of a feature; the rows of X come from
// the cache), then lane g == 0 collects the four results of its token into one 16-byte
// store.  Workgroup = 4 waves over the same tokens, 16 features a trip.
__global__ __launch_bounds__(256) void csr_linear_f32_kernel(const Csr32Args a, int rows_per_wg) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int tokl = lane & 15, g = lane >> 4;
    const int tok = blockIdx.y * 16 + tokl;
    const bool tok_ok = tok < a.T;
    const float *xrow = a.X + (size_t)(tok_ok ? tok : 0) * a.in;
    const int o_begin = blockIdx.x * rows_per_wg;
    const int o_end = min(o_begin + rows_per_wg, a.out);
    for (int o0 = o_begin + wave * 4; o0 < o_end; o0 += 16) {  // out % 4 == 0: a group of four is whole
        const int o = o0 + g;
        const int ks = a.indptr[o], ke = a.indptr[o + 1];
        float acc = 0.0f;
        int k = ks;
        for (; k + 4 <= ke; k += 4) {  // four non-zeros a trip: their loads are issued together
            int idx[4];
            float val[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                idx[u] = a.indices[k + u];
                val[u] = a.data[k + u];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) acc = fmaf(val[u], xrow[idx[u]], acc);
        }
        for (; k < ke; k++) acc = fmaf(a.data[k], xrow[a.indices[k]], acc);
        acc = apply_act(acc + (a.bias ? a.bias[o] : 0.0f), a.act);
        const float v1 = __shfl(acc, tokl + 16, kWave);
        const float v2 = __shfl(acc, tokl + 32, kWave);
        const float v3 = __shfl(acc, tokl + 48, kWave);
        if (g == 0 && tok_ok) *reinterpret_cast<float4 *>(a.Y + (size_t)tok * a.out + o0) = float4{acc, v1, v2, v3};
    }
}

static inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// token blocks of 16 per wave: more of them reuse a weight cell more often, fewer give a
// small problem more workgroups
static inline int token_blocks(int T) { return T >= 2048 ? 4 : T >= 64 ? 2 : 1; }

}  // namespace et

using namespace et;

extern "C" {

int et_linear_bsr16_f32(const int32_t *row_ptr, const int32_t *col_idx, const float *tiles, const float *bias,
                        const float *X, float *Y, int T, int in, int out, int act, et_stream stream) {
    ET_REQUIRE(row_ptr && col_idx && tiles && X && Y, ET_ERR_INVALID_ARG, "et_linear_bsr16_f32: NULL pointer");
    ET_REQUIRE(T >= 0 && in > 0 && out > 0, ET_ERR_INVALID_ARG, "et_linear_bsr16_f32: T=%d in=%d out=%d", T, in, out);
    ET_REQUIRE(act >= ET_ACT_NONE && act <= ET_ACT_GELU, ET_ERR_INVALID_ARG, "et_linear_bsr16_f32: act=%d", act);
    ET_REQUIRE(in % 16 == 0 && out % 16 == 0, ET_ERR_UNSUPPORTED,
               "et_linear_bsr16_f32: in=%d out=%d must be multiples of 16", in, out);
    ET_REQUIRE(aligned16(tiles) && aligned16(X) && aligned16(Y), ET_ERR_UNSUPPORTED,
               "et_linear_bsr16_f32: tiles, X and Y must be 16-byte aligned");
    if (T == 0) return ET_OK;
    Bsr32Args a{X, row_ptr, col_idx, tiles, bias, T, in, out, 0, Y, act};
    hipStream_t st = as_stream(stream);
    const int strips = (T + 15) / 16;
    // The parts of the strips and of the columns the dies keep to: of the splits that leave the busiest die the fewest
    // (strip, column) pairs, or up to 3 % more, the one that leaves a die the fewest bytes, taking a fifth of the tiles as kept
    // (their number is not known here).  Against the best of the four splits, 23 shapes of 16 to 4096 rows: 1.00 - 1.03 of its
    // time at 50 % sparsity, 1.00 - 1.04 at 80 %, 1.00 - 1.05 at 95 %.  (By bytes alone the dies were loaded unevenly: 160 rows
    // 3072 -> 768 at 50 % 15.2 us, now 10.7.)
    auto place = [&](int columns) {
        auto parts = [](int n, int d) { return (n + d - 1) / d; };
        auto load = [&](int k) { return (double)parts(strips, 1 << k) * parts(columns, 8 >> k); };
        auto bytes = [&](int k) { return (double)T / (1 << k) + 0.2 * out * (1 << k) / 8; };  // in units of a row of X
        double least = load(0);
        for (int k = 1; k <= 3; k++) least = std::min(least, load(k));
        int best = -1;
        for (int k = 0; k <= 3; k++)
            if (load(k) <= 1.03 * least && (best < 0 || bytes(k) < bytes(best))) best = k;
        a.die_bits = best;
        const int rows = parts(strips, 1 << best), gy = std::min(rows, 32768);
        return dim3(8 * parts(columns, 8 >> best), gy, parts(rows, gy));
    };
    const long long pairs = (long long)(out / 16) * strips;
    const size_t lds = (size_t)16 * (in + kStripPad) * sizeof(float);
    // The strip form where two workgroups fit a compute unit and there are six pairs or more for each: 80 %, us, strip
    // against not: 2304 pairs of 768 values 6.7 / 7.2, 3072 7.0 / 9.7, 1536 5.2 / 5.8, 768 5.1 / 4.0 (95 %: 2304 4.8 / 4.3, 3072 5.0 / 5.9).
    if (pairs >= 1536 && lds <= 80 * 1024) {
        if (lds > 64 * 1024)
            ET_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(bsr16_linear_strip_f32_kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        const dim3 grid = place((out / 16 + kStripWaves - 1) / kStripWaves);
        bsr16_linear_strip_f32_kernel<<<grid, kStripWaves * 64, lds, st>>>(ET_BSR32_ARGS(a));
        return check_launch("bsr16_linear_strip_f32_kernel");
    }
    // Wider than that, the wide form from two of its workgroups a compute unit on: 80 %, us, wide against short: 512 workgroups
    // 1024 x 4096 -> 1024 38 / 43, 512 x 2048 -> 2048 21 / 25; 768 1024 x 1536 -> 1536 22 / 27; 384 2048 x 3072 -> 768 52 / 46,
    // 512 x 1536 -> 1536 15.4 / 14.3.  (Many rows of a narrow result 1.04 the other way: 768 4096 x 3072 -> 768 93 / 89.)
    const int mt = token_blocks(T), wide_strips = (T + 16 * mt - 1) / (16 * mt), wide_x = (out / 16 + 3) / 4;
    if (in > kSplitMaxIn || (mt > 1 && lds > 80 * 1024 && (long long)wide_x * wide_strips >= 512)) {
        const int wide_y = std::min(wide_strips, 32768);
        const dim3 grid(wide_x, wide_y, (wide_strips + wide_y - 1) / wide_y);
        if (mt == 4) bsr16_linear_wide_f32_kernel<4><<<grid, 256, 0, st>>>(ET_BSR32_ARGS(a));
        else bsr16_linear_wide_f32_kernel<2><<<grid, 256, 0, st>>>(ET_BSR32_ARGS(a));
        return check_launch("bsr16_linear_wide_f32_kernel");
    }
    // Two waves a pair below two pairs a compute unit: 192 pairs of 38 tiles 5.2 us against 7.3, 576 pairs of 10 tiles 4.9
    // against 4.7; four waves are no faster.
    const dim3 grid = place(out / 16);
    if (pairs < 512) bsr16_linear_split_f32_kernel<2><<<grid, 128, 0, st>>>(ET_BSR32_ARGS(a));
    else bsr16_linear_split_f32_kernel<1><<<grid, 64, 0, st>>>(ET_BSR32_ARGS(a));
    return check_launch("bsr16_linear_split_f32_kernel");
}

int et_linear_vec1x16_f32(const int32_t *tile_idx, const int32_t *row_idx, const float *data, const float *bias,
                          const float *X, float *Y, int T, int in, int out, int act, et_stream stream) {
    ET_REQUIRE(tile_idx && row_idx && data && X && Y, ET_ERR_INVALID_ARG, "et_linear_vec1x16_f32: NULL pointer");
    ET_REQUIRE(T >= 0 && in > 0 && out > 0, ET_ERR_INVALID_ARG, "et_linear_vec1x16_f32: T=%d in=%d out=%d", T, in, out);
    ET_REQUIRE(act >= ET_ACT_NONE && act <= ET_ACT_GELU, ET_ERR_INVALID_ARG, "et_linear_vec1x16_f32: act=%d", act);
    ET_REQUIRE(in % 16 == 0 && out % 16 == 0, ET_ERR_UNSUPPORTED,
               "et_linear_vec1x16_f32: in=%d out=%d must be multiples of 16", in, out);
    ET_REQUIRE(aligned16(data) && aligned16(X) && aligned16(Y), ET_ERR_UNSUPPORTED,
               "et_linear_vec1x16_f32: data, X and Y must be 16-byte aligned");
    if (T == 0) return ET_OK;
    const V16F32Args a{tile_idx, row_idx, data, bias, X, Y, T, in, out, act};
    const int mt = token_blocks(T);
    const dim3 grid((out / 16 + 3) / 4, (T + 16 * mt - 1) / (16 * mt));
    hipStream_t st = as_stream(stream);
    if (mt == 4) vec1x16_linear_f32_kernel<4><<<grid, 256, 0, st>>>(a);
    else if (mt == 2) vec1x16_linear_f32_kernel<2><<<grid, 256, 0, st>>>(a);
    else vec1x16_linear_f32_kernel<1><<<grid, 256, 0, st>>>(a);
    return check_launch("vec1x16_linear_f32_kernel");
}

int et_linear_csr_f32(const int32_t *indptr, const int32_t *indices, const float *data, const float *bias,
                      const float *X, float *Y, int T, int in, int out, int act, et_stream stream) {
    ET_REQUIRE(indptr && indices && data && X && Y, ET_ERR_INVALID_ARG, "et_linear_csr_f32: NULL pointer");
    ET_REQUIRE(T >= 0 && in > 0 && out > 0, ET_ERR_INVALID_ARG, "et_linear_csr_f32: T=%d in=%d out=%d", T, in, out);
    ET_REQUIRE(act >= ET_ACT_NONE && act <= ET_ACT_GELU, ET_ERR_INVALID_ARG, "et_linear_csr_f32: act=%d", act);
    ET_REQUIRE(out % 4 == 0, ET_ERR_UNSUPPORTED, "et_linear_csr_f32: out=%d must be a multiple of 4", out);
    ET_REQUIRE(aligned16(Y), ET_ERR_UNSUPPORTED, "et_linear_csr_f32: Y must be 16-byte aligned");
    if (T == 0) return ET_OK;
    const Csr32Args a{indptr, indices, data, bias, X, Y, T, in, out, act};
    const int strips = (T + 15) / 16;
    int groups = (1024 + strips - 1) / strips;  // about 1024 workgroups, whole 16-feature groups each
    int rpw = (out + groups - 1) / groups;
    rpw = ((rpw + 15) / 16) * 16;
    const dim3 grid((out + rpw - 1) / rpw, strips);
    csr_linear_f32_kernel<<<grid, 256, 0, as_stream(stream)>>>(a, rpw);
    return check_launch("csr_linear_f32_kernel");
}

}  // extern "C"
