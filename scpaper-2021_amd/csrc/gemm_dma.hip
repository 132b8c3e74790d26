// Dense GEMM for gfx950 on direct-to-LDS loads: C[M x N] = act(A[M x K] * B^T + bias), A and B
// both K-contiguous (B stored [N x K]), M, N and K multiples of 16; whole tiles and stages of 64, or ragged edges.
//
// The 64x64-per-wave kernel in gemm.hip reads 1 byte of LDS per 32 flops, which at the
// MFMA peak is the whole bandwidth of the LDS port, and stages through registers; it tops
// out near a third of the matrix peak.  Here a workgroup of 4 waves (2 x 2) computes a tile of
// 64 TMW x 64 TNW and each wave a block of TMW x TNW v_mfma_f32_32x32x16_f16 tiles.  What bounds a stage
// of 64 of depth is the LDS port (a 128 x 192 tile: 960 cycles of reads and direct loads against 774 of products), so a
// tile is as large as leaves every compute unit one; what is added once is 3 us of launch, first stage and epilogue.
// Latencies are covered inside the wave: K advances in stages of 64 through four LDS buffers, a later stage is
// loaded straight from global memory into an idle buffer while the current one is multiplied (staging through registers and
// ds_write costs a third of the rate: the LDS port is then the bound), fragments are read two K slices ahead, and
// reads and loads are issued between the MFMAs that hide them, in an order fixed in the source.  With two or three buffers
// (several workgroups to a compute unit, or the 128 x 192 tile) and with eight waves (256 x 256, whole tiles; four waves of 128 x 128 where
// edges are ragged) fragments are read one slice ahead: another wave, or a slice of 16 MFMAs, covers for it.  So does the 64 x 64 tile with
// ragged edges, where the deep order lost.
//
// The MFMA A operand is the B matrix (output features) and vice versa, so a lane ends with
// 4 consecutive features of one row of C per 8-row group of a tile; the epilogue transposes
// through LDS to store whole row segments.
#include "gemm.hip.h"
#include "gemm_forms.h"

namespace et {

constexpr int kDmaXcds = 8;
constexpr int kSbM = 4, kSbN = 8;        // tile block one XCD works on at a time
constexpr size_t dma_lds_bytes(int tmw, int tnw, int nbuf, int ks = kDmaK, int nwn = 2) {  // buffers of (BM + BN) rows of ks k-values
    return (size_t)nbuf * (64 * tmw + 32 * nwn * tnw) * ks * sizeof(_Float16);
}
// s_waitcnt immediate for vmcnt(n) alone on gfx9: vmcnt in bits 3:0 and 15:14, expcnt 6:4 and
// lgkmcnt 11:8 left at their maxima
constexpr int wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }
#define ET_GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void *)(p))
#define ET_LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))

typedef float f16v __attribute__((ext_vector_type(16)));

// TMW x TNW: 32 x 32 MFMA tiles per wave.  IDX: the result columns are scattered (c_scatter) or
// their bias is gathered (bias_idx).  RAGGED: M, N and K are multiples of 16 only; rows past the
// end of an operand are loaded from its last row and never stored, the chunks of the last K
// stage past the end of K are zeroed in LDS before they are read.
// BT: B is stored [K x N] (N contiguous) instead of [N x K]; its stage lies in LDS as loaded, k-major,
// and a lane gathers the 8 k-values of a fragment with 2-byte reads (64 x 64 tiles only).
// Problem z = blockIdx.y of a batch uses the operand offsets of GemmArgs.
// KS: k-values per stage, 64 or (whole tiles only) 32: half the stage, twice the buffers in the same LDS, so the
// loads of a stage are issued three stages ahead and spread over two K slices.
// NWN: waves along N, 2 (four waves, one per SIMD) or (whole tiles only) 4: eight waves, two per SIMD, so that a wave
// held up at a load or at the barrier leaves the matrix pipe to the other.
// The arguments in front are what the first requests need: preloaded into scalar registers (us, before and now, with the tile found without divisions: 2048 x 768 ->
// 768 7.65 and 7.30, 2304 13.9 and 13.5, 3072 with GELU 17.1 and 16.5, 1024^3 7.2 and 6.8, 512 x 768 -> 3072 8.35 and 7.95).
#define ET_DMA_FIRST const _Float16 *A, const _Float16 *B, const _Float16 *bias, int M, int N, int K, int lda, int ldb, int group_rows, unsigned per_row
// LINES (ragged tiles through four buffers): rows that begin off a 128-byte line.
template <int TMW, int TNW, int NBUF, bool IDX, bool RAGGED = false, bool BT = false, int KS = kDmaK, int NWN = 2, bool LINES = false>
__global__ __launch_bounds__(128 * NWN) void gemm_f16_dma_kernel(ET_DMA_FIRST, const GemmArgs ga) {
    static_assert(NWN == 2 || (NWN == 4 && !RAGGED && !BT), "eight waves are written for whole tiles");
    constexpr int kWaves = 2 * NWN;
    static_assert(NBUF >= 2 && NBUF <= 4 && (NBUF - 1) * (2 * TMW + 2 * TNW) * KS / kDmaK <= 63, "vmcnt holds 63 loads");
    static_assert(KS == kDmaK || (KS == 32 && !RAGGED && !BT), "half stages are written for whole tiles");
    static_assert(!BT || (TMW == 1 && TNW == 1 && RAGGED), "the k-major B stage is written for the 64 x 64 tile");
    static_assert(!LINES || (RAGGED && !BT && NBUF == 4 && KS == 64), "rows by lines are written for four buffers of 64");
    GemmArgs g = ga;
    g.A = A, g.B = B, g.bias = bias, g.M = M, g.N = N, g.K = K, g.lda = lda, g.ldb = ldb;
    if (TMW == 1 && TNW == 1 && blockIdx.y) {  // (several problems run on 64 x 64 tiles)
        const long long zo = blockIdx.y / g.batch_inner, zi = blockIdx.y % g.batch_inner;
        g.A += zo * g.sAo + zi * g.sAi;
        g.B += zo * g.sBo + zi * g.sBi;
        g.C += zo * g.sCo + zi * g.sCi;
        if (g.bias) g.bias += zo * g.sBias_o + zi * g.sBias_i;
    }
    constexpr int BM = 64 * TMW, BN = 32 * NWN * TNW;  // workgroup tile: 2 x NWN waves
    constexpr int WM = 32 * TMW, WN = 32 * TNW;  // wave block
    extern __shared__ __align__(16) unsigned char dma_smem[];
    _Float16 *As = reinterpret_cast<_Float16 *>(dma_smem);  // [NBUF][BM][KS], chunks swizzled
    _Float16 *Bs = As + NBUF * BM * KS;                      // [NBUF][BN][KS]

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: LDS targets of the loads stay scalar
    const int wm = wave / NWN, wn = wave % NWN;
    const int l32 = lane & 31, kg = lane >> 5;
    // Workgroup id -> tile, XCD-aware.  Workgroups go to the 8 XCDs round-robin by id and each XCD runs them in
    // order; consecutive workgroups of an XCD are given consecutive tiles of an order that walks the result in
    // blocks of group_rows x 8 tiles (4 x 8: 4 panels of A, 8 of B), so the XCD's L2 serves about 12 panels to 32
    // workgroups instead of up to 64.  The order counts existing tiles only (a block at the right or lower edge
    // is narrower or shorter) and the groups are dealt to the XCDs in turn, so every XCD gets the same number of
    // tiles to within one group; dealing whole 4 x 8 blocks instead gave the XCDs with odd numbers only the
    // half-empty blocks of a result 12 tiles wide.
    const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
    const int sbm = group_rows, gsh = sbm == 4 ? 5 : sbm == 2 ? 4 : 3;  // a group: sbm x 8 = 1 << gsh tiles
    const int xcd = blockIdx.x % kDmaXcds, j = blockIdx.x / kDmaXcds;
    const int t = ((((j >> gsh) * kDmaXcds + xcd)) << gsh) + (j & ((1 << gsh) - 1));
    if (t >= tiles_m * tiles_n) return;  // padding of the grid (whole workgroup)
    int ty, tx;
    {
        // (no division that the scalar unit would spend 150 cycles on: `per_row` is 2^32 over the tiles of a block row, rounded up, or 0
        // where that would not be exact; a block is 1 to 4 tiles high and 1 to 8 wide)
        const int per_br = sbm * tiles_n, full_br = tiles_m >> (gsh - 3);  // tiles of a full block row; such rows
        const int br = min(per_row ? (int)(((unsigned long long)(unsigned)t * per_row) >> 32) : t / per_br, full_br);
        const int rem = t - br * per_br;
        if (br < full_br && (tiles_n & (kSbN - 1)) == 0) {  // whole blocks only: shifts
            const int q = rem & ((1 << gsh) - 1);
            ty = br * sbm + (q >> 3);
            tx = (rem >> gsh) * kSbN + (q & 7);
        } else {
            static_assert(kSbM == 4 && kSbN == 8, "the divisions below");
            const int rows = br < full_br ? sbm : tiles_m - full_br * sbm;  // tile rows of this block row
            const int per_bc = rows * kSbN, full_bc = tiles_n / kSbN;
            const unsigned eights = (unsigned)rem >> 3;
            const int bc = min((int)(rows == 3 ? (unsigned)(((unsigned long long)eights * 0x55555556u) >> 32) : eights >> (rows >> 1)), full_bc);
            const int q = rem - bc * per_bc;
            const int w = bc < full_bc ? kSbN : tiles_n - full_bc * kSbN;  // tile columns of this block
            const int over = w == 1 ? q : (q * (int)(0x00805640342b2520ull >> (64 - 8 * w) & 255)) >> 8;  // q / w, q < 32
            ty = br * sbm + over;
            tx = bc * kSbN + q - over * w;
        }
    }
    const int m0 = ty * BM, n0 = tx * BN;

    const int nbase = n0 + wn * WN;
    // The bias: a lane of kScLanes holds that of one feature in kScCols, an epilogue hands them round through LDS.  Two-byte loads of
    // all the features a lane's accumulators belong to (32 of them with two feature tiles, ahead of the first stage in the
    // order loads are answered in) held every workgroup up by 1 us.  Unconditional (from B when there is no bias) and selected.
    // IDX: the same lanes store the scattered columns, so the index of a lane's bias is also where its column goes.
    constexpr int kScLanes = WN % 64 == 0 ? 64 : 32;  // lanes to a row of scattered columns
    constexpr int kScCols = WN / kScLanes;            // column groups
    const bool has_bias = g.bias != nullptr;
    const int32_t *col_idx = g.c_scatter ? g.c_scatter : g.bias_idx;  // bias index of result column n
    int bias_at[kScCols];
    _Float16 bias_of[kScCols];
#pragma unroll
    for (int e = 0; e < kScCols; e++) {
        const int n = nbase + e * kScLanes + lane % kScLanes;
        bias_at[e] = RAGGED ? min(n, g.N - 1) : n;
        if (IDX && col_idx) bias_at[e] = col_idx[bias_at[e]];
    }
    auto load_bias = [&] {
#pragma unroll
        for (int e = 0; e < kScCols; e++) bias_of[e] = (has_bias ? g.bias : g.B)[has_bias ? bias_at[e] : 0];
    };
    if constexpr (!IDX) load_bias();  // (behind an index: once the first stage is there, and the index with it)

    f16v acc[TMW][TNW];  // [token tile][feature tile]
#pragma unroll
    for (int i = 0; i < TMW; i++)
#pragma unroll
        for (int j = 0; j < TNW; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    // Stage loads go straight from global memory to LDS (global_load_lds_dwordx4): a wave
    // instruction fills 1 KB of consecutive LDS, 16 bytes per lane, from addresses the lanes
    // choose.  Here that is 8 rows of 128 bytes, 8 lanes a row (whole lines of the operand);
    // within the row the lane at position p fetches chunk p ^ swz(row), so that the fragment
    // reads below, 16 rows apart by one chunk column, spread over all banks with no padding.
    const int lrow = lane >> 3, lpos = lane & 7;
    // K-contiguous operands (kWhole; all but BT): a lane's loads differ between stages only by the stage's k0, so a
    // load is a buffer resource at the tile's first row, the stage's k0 as scalar offset and a 32-bit lane offset computed once; every stage
    // issues its loads (past the last stage through a resource without records: they touch no memory),
    // which keeps the loads in the block of the multiplications, where they can be placed between them, and the
    // number of outstanding loads the same in every stage.  RAGGED: rows past the end of an operand take the offset
    // of its last row, and the last stage, when K ends inside it, has offsets of its own: chunks past the end of K
    // fetch the last chunk of the row instead (and are zeroed in LDS once they have landed).
    constexpr bool kWhole = !BT;
    constexpr bool kImm = !RAGGED;  // (a clamped row may have a smaller offset than the immediate it would have to undo)
    // A stage row holds KS k-values = kLpr 16-byte chunks; one load instruction fills kRpi rows.  The chunk at
    // position p of row r is chunk p ^ swz(r) of the operand: rows that share their banks (2 rows of 128 bytes,
    // 4 rows of 64 bytes span all banks) get different chunks at one position.
    constexpr int kLpr = KS / 8, kRpi = 64 / kLpr;
    constexpr int kLA = BM / kWaves / kRpi, kLB = BN / kWaves / kRpi;  // loads per wave and stage
    auto swz_of = [](int r) { return KS == 64 ? (r >> 1) & 7 : (r >> 2) & 3; };
    // The instruction's immediate offset is added to the global address and to the LDS address alike: loads
    // 4j .. 4j + 3 of an operand share one LDS base (M0) and differ in the immediate, 1024 (v % 4), which the
    // lane's global offset has subtracted again.  One write of M0 per four loads instead of one per load.
    unsigned offA[kLA], offB[kLB];  // bytes from the tile's first row at k = 0, minus the immediate
    // what a last stage that K ends in adds to them: rows 16 apart have the same chunk at a position, so loads of even and of odd number
    // have one each (held for every load they were up to 32 registers)
    unsigned tail_by[2] = {0, 0};
    // The 64 x 64 tile has four loads a stage and holds theirs, chosen instead of added: us, added and so, 304 x 4096 -> 3072 20.1 and 19.2, 224 x 4096 -> 4096 20.1 and 19.2, 864 x 5120 ->
    // 240 22.8 and 22.0; 276 problems of 1024 to 5120 inputs 0.975 of their time.  (Added to the offsets once, ahead of the last stage, which costs no stage an instruction: 1.03.)
    constexpr bool kHoldTail = RAGGED && !LINES && TMW == 1 && TNW == 1;
    unsigned tail_a[kHoldTail ? kLA : 1], tail_b[kHoldTail ? kLB : 1];
    const int k_tail0 = (g.K - 1) / KS * KS;   // first k of the last stage
    const int k_tail = g.K - k_tail0;          // k-values of the last stage, 16 .. KS
    // LINES: a stage's 128 bytes of a row that begins off a line lie in two lines, and the L1 does not hold the other part until the
    // next stage asks for it: 1.25 to 1.3 times the time (2048 x 3056 -> 768 22.7 us, 3072 17.6).  So a request fetches whole lines: line l
    // of a row are its chunks 8 l - shift .. + 7, `shift` the row's chunks off a line, and stage s reads lines s and s + 1 (a fragment's chunk lies
    // shift further, in the next buffer past 8).  A lane's rows are multiples of 8 apart and so have one shift, in the requests as in the fragments.
    // Chunks ahead of a row or past its end are its first or last one instead, which no product takes.  us, before and now: 2048 x 3056 -> 768 22.7 and 18.9,
    // 4096 x 2032 -> 2048 51.4 and 42.2, 1104 x 1040 -> 3072 14.4 and 12.3, 8192 x 4080 -> 4096 369 and 323, 110 Linears of 256 to 8192 rows 0.94 of their
    // time in the mean; the same bits.
    int line_a[2] = {0, 0}, line_b[2] = {0, 0};              // chunk of line 0 that the lane's loads of even and of odd number fetch
    unsigned by_a[2] = {0, 0}, by_b[2] = {0, 0};             // bytes to that of the line asked for
    auto shift_of = [](const _Float16 *first, int row, int ld) { return (int)(((unsigned)(reinterpret_cast<uintptr_t>(first) >> 4) + (unsigned)row * (unsigned)(ld >> 3)) & 7); };
    const int chunks = g.K >> 3;
    auto at_line = [&](int line) {
#pragma unroll
        for (int e = 0; e < 2; e++) {
            by_a[e] = (unsigned)min(max(line_a[e] + line * 8, 0), chunks - 1) * 16;
            by_b[e] = (unsigned)min(max(line_b[e] + line * 8, 0), chunks - 1) * 16;
        }
    };
    if (kWhole) {
        const int lr = lane / kLpr, lp = lane % kLpr;
#pragma unroll
        for (int v = 0; v < kLA; v++) {
            const int r = wave * (BM / kWaves) + v * kRpi + lr;
            const int row = RAGGED ? min(m0 + r, g.M - 1) - m0 : r;
            const int c8 = (lp ^ swz_of(r)) * 8;
            offA[v] = (unsigned)((row * g.lda + c8) * 2 - (kImm ? (v % 4) * 1024 : 0));
            if (RAGGED && v < 2) tail_by[v] = (unsigned)((min(c8, k_tail - 8) - c8) * 2);
            if (kHoldTail) tail_a[kHoldTail ? v : 0] = (unsigned)((row * g.lda + min(c8, k_tail - 8)) * 2);
            if (LINES) offA[v] = (unsigned)(row * g.lda * 2);
            if (LINES && v < 2) line_a[v] = (c8 >> 3) - shift_of(g.A, m0 + lr, g.lda);
        }
#pragma unroll
        for (int v = 0; v < kLB; v++) {
            const int r = wave * (BN / kWaves) + v * kRpi + lr;
            const int row = RAGGED ? min(n0 + r, g.N - 1) - n0 : r;
            const int c8 = (lp ^ swz_of(r)) * 8;
            offB[v] = (unsigned)((row * g.ldb + c8) * 2 - (kImm ? (v % 4) * 1024 : 0));
            if (kHoldTail) tail_b[kHoldTail ? v : 0] = (unsigned)((row * g.ldb + min(c8, k_tail - 8)) * 2);
            if (LINES) offB[v] = (unsigned)(row * g.ldb * 2);
            if (LINES && v < 2) line_b[v] = (c8 >> 3) - shift_of(g.B, n0 + lr, g.ldb);
        }
    }
    // Requests past the last stage are needed for the count of those outstanding, not for their data: through a buffer without
    // records they touch no memory (fetching the last stage again was a quarter of what a workgroup took in at 12 stages, and
    // the epilogue waited for it).  Everything about the buffer is made scalar here; a resource in vector registers would put
    // a loop around every request.
    auto scalar = [](const void *p) {
        const uint64_t v = reinterpret_cast<uint64_t>(p);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        return reinterpret_cast<char *>((uint64_t)hi << 32 | lo);
    };
    char *const a_tile = scalar(g.A + (size_t)m0 * g.lda);
    char *const b_tile = scalar(g.B + (size_t)n0 * g.ldb);
    int records = 0;  // of both buffers: 1 GiB (256 rows of the widest operand taken) or none
    auto aim = [&](int stages_left) { records = __builtin_amdgcn_readfirstlane(min(max(stages_left, 0), 1) << 30); };
    // loads [first, first + count) of a stage's kLA + kLB (whole tiles)
    auto load_part = [&](int buf, int k0, int first, int count) {
        auto four = [&](__amdgpu_buffer_rsrc_t rsrc, unsigned off, _Float16 *dst, int sub) {  // sub = v % 4 (a constant once unrolled)
            if (sub == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, ET_LDS_PTR(dst), 16, off, k0 * 2, 0, 0);
            else if (sub == 1) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, ET_LDS_PTR(dst), 16, off, k0 * 2, 1024, 0);
            else if (sub == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, ET_LDS_PTR(dst), 16, off, k0 * 2, 2048, 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, ET_LDS_PTR(dst), 16, off, k0 * 2, 3072, 0);
        };
        auto ra = __builtin_amdgcn_make_buffer_rsrc(a_tile, 0, records, 0x00020000);
        auto rb = __builtin_amdgcn_make_buffer_rsrc(b_tile, 0, records, 0x00020000);
        static_assert(!RAGGED || (kRpi == 8 && BM / kWaves % 16 == 0 && BN / kWaves % 16 == 0 && kLA >= 2), "the chunks of a last stage");
        const bool tail = RAGGED && !LINES && k0 == k_tail0 && k_tail < KS;  // uniform
        const unsigned by[2] = {tail ? tail_by[0] : 0u, tail ? tail_by[1] : 0u};
#pragma unroll
        for (int v = 0; v < kLA; v++)
            if (v >= first && v < first + count) {
                const unsigned off = kHoldTail ? (tail ? tail_a[kHoldTail ? v : 0] : offA[v]) : RAGGED ? offA[v] + (LINES ? by_a[v & 1] : by[v & 1]) : offA[v];
                four(ra, off, As + (buf * BM + wave * (BM / kWaves) + (kImm ? (v / 4) * 4 : v) * kRpi) * KS, kImm ? v % 4 : 0);
            }
#pragma unroll
        for (int v = 0; v < kLB; v++)
            if (kLA + v >= first && kLA + v < first + count) {
                const unsigned off = kHoldTail ? (tail ? tail_b[kHoldTail ? v : 0] : offB[v]) : RAGGED ? offB[v] + (LINES ? by_b[v & 1] : by[v & 1]) : offB[v];
                four(rb, off, Bs + (buf * BN + wave * (BN / kWaves) + (kImm ? (v / 4) * 4 : v) * kRpi) * KS, kImm ? v % 4 : 0);
            }
    };
    auto load_stage = [&](int buf, int k0) {  // BT
#pragma unroll
        for (int v = 0; v < 2 * TMW; v++) {  // a wave loads a quarter of the rows of each operand
            const int r0 = wave * (BM / 4) + v * 8, r = r0 + lrow;
            const int c = lpos ^ ((r >> 1) & 7);
            const int row = RAGGED ? min(m0 + r, g.M - 1) : m0 + r;
            const int k = RAGGED ? min(k0 + c * 8, g.K - 8) : k0 + c * 8;
            __builtin_amdgcn_global_load_lds(ET_GLOBAL_PTR(g.A + (size_t)row * g.lda + k),
                                             ET_LDS_PTR(As + (buf * BM + r0) * kDmaK), 16, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 2 * TNW; v++) {
            const int r0 = wave * (BN / 4) + v * 8, r = r0 + lrow;
            // LDS row r = k-value k0 + r of the stage, 64 columns of B from n0
            const int krow = min(k0 + r, g.K - 1), n = min(n0 + lpos * 8, g.N - 8);
            __builtin_amdgcn_global_load_lds(ET_GLOBAL_PTR(g.B + (size_t)krow * g.ldb + n),
                                             ET_LDS_PTR(Bs + (buf * kDmaK + r0) * BN), 16, 0, 0);
        }
    };
    // RAGGED: zeros over the chunks of the last stage that lie past the end of K, in the rows
    // this wave loaded (after its loads have landed, before the barrier that releases the buffer)
    const int ktail = g.K - (g.K - 1) / kDmaK * kDmaK;  // k-values of the last stage, 16..64
    auto zero_tail = [&](int buf) {
        const h8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int v = 0; v < 2 * TMW; v++) {
            const int r = wave * (BM / 4) + v * 8 + lrow;
            if ((lpos ^ ((r >> 1) & 7)) * 8 >= ktail)
                *reinterpret_cast<h8 *>(As + (buf * BM + r) * kDmaK + lpos * 8) = zero8;
        }
#pragma unroll
        for (int v = 0; v < 2 * TNW; v++) {
            const int r = wave * (BN / 4) + v * 8 + lrow;
            if (BT) {  // whole k-rows past the end of K
                if (r >= ktail) *reinterpret_cast<h8 *>(Bs + (buf * kDmaK + r) * BN + lpos * 8) = zero8;
            } else if ((lpos ^ ((r >> 1) & 7)) * 8 >= ktail) {
                *reinterpret_cast<h8 *>(Bs + (buf * BN + r) * kDmaK + lpos * 8) = zero8;
            }
        }
    };
    // fragments of one 16-wide K slice: the token tiles and feature tiles of the wave's block.
    // Rows WM wm + 32 i + l32: the swizzle term (row >> 1) & 7 depends on the lane only.
    struct Frag { h8 x[TMW], w[TNW]; };
    const int swz = swz_of(l32);
    const _Float16 *a_rows = As + (wm * WM + l32) * KS, *b_rows = Bs + (wn * WN + l32) * KS;
    auto read_frag = [&](Frag &f, int buf, int ks) {
        const int chunk = ((ks * 2 + kg) ^ swz) * 8;
#pragma unroll
        for (int i = 0; i < TMW; i++)
            f.x[i] = *reinterpret_cast<const h8 *>(a_rows + buf * BM * KS + chunk + i * 32 * KS);
#pragma unroll
        for (int j = 0; j < TNW; j++) {
            if (BT) {
                const _Float16 *col = Bs + (buf * kDmaK + ks * 16 + kg * 8) * BN + wn * WN + l32;
#pragma unroll
                for (int e = 0; e < 8; e++) f.w[j][e] = col[e * BN];
            } else {
                f.w[j] = *reinterpret_cast<const h8 *>(b_rows + buf * BN * KS + chunk + j * 32 * KS);
            }
        }
    };
    auto multiply = [&](const Frag &f) {
#pragma unroll
        for (int i = 0; i < TMW; i++)
#pragma unroll
            for (int j = 0; j < TNW; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.w[j], f.x[i], acc[i][j], 0, 0, 0);
    };

    const int nstage = RAGGED ? (g.K + kDmaK - 1) / kDmaK : g.K / KS;
    // Stage s is multiplied from LDS buffer s % NBUF; the loads of kAhead later stages are in
    // flight meanwhile.  A direct-to-LDS load has landed when vmcnt says so, and vmcnt counts
    // in issue order: "stage s + 1 has landed" is "at most the loads of the stages after it
    // are outstanding".
    constexpr int kAhead = NBUF - 1;
    // Fragments two slices ahead: four waves and four buffers.  The 64 x 64 tile with ragged edges keeps to one slice: its one
    // MFMA a slice hides little either way, and the deep form asks for a stage half a stage later (719 of 728 ragged Linears of 16..2048
    // rows slower, by 1 to 9 %: 784 x 3072 -> 768 15.9 us deep, 14.6 so, 400 x 4096 -> 1024 19.0 and 18.0; whole tiles are 8 % slower
    // the other way, 1024 x 4096 -> 1024 18.0 and 19.4).
    constexpr bool kDeep = kWhole && NBUF == 4 && NWN == 2 && (LINES || !(RAGGED && TMW * TNW == 1));
    constexpr int kStageLoads = kWhole ? kLA + kLB : 2 * TMW + 2 * TNW;  // per wave
    auto wait_stages = [&](int later) {  // wait until at most `later` whole stages are outstanding
        if (later <= 0) __builtin_amdgcn_s_waitcnt(wait_vm(0));
        else if (later == 1) __builtin_amdgcn_s_waitcnt(wait_vm(kStageLoads));
        else __builtin_amdgcn_s_waitcnt(wait_vm(2 * kStageLoads));
    };
    // Workgroup barrier that orders LDS accesses only.  __syncthreads() carries a fence that
    // waits for every outstanding global access, the direct-to-LDS loads of the later stages
    // included, which is exactly what a deeper pipeline must not do; here this wave's LDS reads
    // are waited for, the barrier is passed, and the compiler moves no memory access across.
    auto lds_barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    // Order of issue inside one K slice (K-contiguous operands).  The wave's instruction stream is the only thing that feeds
    // the matrix pipe of its SIMD, so the slice is written out in the order it is to be issued in, one MFMA at a time
    // with a fence for the scheduler behind it: the fragments of a later slice are read, and `nload` loads of a later
    // stage (from number `first`) issued, evenly between the MFMAs (left alone the scheduler puts every read directly in
    // front of its first use, and the pipe drains while it returns).
    constexpr int kNM = TMW * TNW, kND = TMW + TNW;
    constexpr int kSlices = KS / 16;                  // K slices (steps) of a stage
    constexpr int kLoadSteps = KS == 32 ? 2 : 1;      // steps of a stage that issue a share of a later stage's loads
    constexpr int kStepLoads = (kStageLoads + kLoadSteps - 1) / kLoadSteps;  // in the first such step; the rest in the second
    constexpr int kStepLoads2 = kStageLoads - kStepLoads;
    // LINES: where in the buffers, from a stage's own on, a lane finds its chunk of a slice; round the end of the ring
    unsigned line_x[kSlices], line_w[kSlices];
    if constexpr (LINES) {
        const int sx = kg + shift_of(g.A, m0 + l32, g.lda), sw = kg + shift_of(g.B, n0 + l32, g.ldb);
#pragma unroll
        for (int ks = 0; ks < kSlices; ks++) {
            line_x[ks] = (unsigned)((((2 * ks + sx) & 7) ^ swz) * 8 + ((2 * ks + sx) >> 3) * (BM * KS));
            line_w[ks] = (unsigned)((((2 * ks + sw) & 7) ^ swz) * 8 + ((2 * ks + sw) >> 3) * (BN * KS));
        }
    }
    auto ring = [](unsigned at, unsigned whole) { return min(at, at - whole); };
    auto read_x = [&](Frag &f, int i, int buf, int ks) {
        if constexpr (LINES) f.x[i] = *reinterpret_cast<const h8 *>(a_rows + ring(buf * BM * KS + line_x[ks], NBUF * BM * KS) + i * 32 * KS);
        else f.x[i] = *reinterpret_cast<const h8 *>(a_rows + buf * BM * KS + ((ks * 2 + kg) ^ swz) * 8 + i * 32 * KS);
    };
    auto read_w = [&](Frag &f, int j, int buf, int ks) {
        if constexpr (LINES) f.w[j] = *reinterpret_cast<const h8 *>(b_rows + ring(buf * BN * KS + line_w[ks], NBUF * BN * KS) + j * 32 * KS);
        else f.w[j] = *reinterpret_cast<const h8 *>(b_rows + buf * BN * KS + ((ks * 2 + kg) ^ swz) * 8 + j * 32 * KS);
    };
    auto read_slice = [&](Frag &f, int buf, int ks) {
#pragma unroll
        for (int i = 0; i < TMW; i++) read_x(f, i, buf, ks);
#pragma unroll
        for (int j = 0; j < TNW; j++) read_w(f, j, buf, ks);
    };
    auto step = [&](const Frag &fm, Frag &fr, int rbuf, int rks, int nload, int lbuf, int k_later, int first) {
#pragma unroll
        for (int m = 0; m < kNM; m++) {
            const int i = m / TNW, j = m % TNW;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fm.w[j], fm.x[i], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int idx = m * kND / kNM; idx < (m + 1) * kND / kNM; idx++) {
                if (idx < TMW) read_x(fr, idx, rbuf, rks);
                else read_w(fr, idx - TMW, rbuf, rks);
            }
            if (nload > 0) load_part(lbuf, k_later, first + m * nload / kNM, (m + 1) * nload / kNM - m * nload / kNM);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    Frag f0, f1;
    if constexpr (LINES) {
#pragma unroll
        for (int p = 0; p < NBUF; p++) {
            aim(nstage + 1 - p);
            at_line(p);
            load_part(p, 0, 0, kStageLoads);
        }
        __builtin_amdgcn_s_waitcnt(wait_vm(2 * kStageLoads));  // lines 0 and 1 have landed
    } else if constexpr (kWhole) {
#pragma unroll
        for (int p = 0; p < kAhead; p++) {
            aim(nstage - p);
            load_part(p, min(p, nstage - 1) * KS, 0, kStageLoads);
        }
        __builtin_amdgcn_s_waitcnt(wait_vm((kAhead - 1) * kStageLoads));  // stage 0 has landed
    } else {
#pragma unroll
        for (int p = 0; p < kAhead; p++)
            if (p < nstage) load_stage(p, p * kDmaK);
        wait_stages(min(kAhead, nstage) - 1);
    }
    if constexpr (IDX) load_bias();
    if (RAGGED && !LINES && nstage == 1 && ktail < kDmaK) zero_tail(0);
    lds_barrier();
    if constexpr (LINES) read_slice(f0, 0, 0);
    else read_frag(f0, 0, 0);
    int cur = 0;
    if constexpr (LINES) {
        // As the deep form below, but the barrier in the middle of a stage waits for the stage's reads too: its own buffer, whose line no
        // later stage reads, takes line s + 4.
        Frag f2, f3;
        read_slice(f1, 0, 1);
        for (int s = 0; s < nstage - 1; s++) {
            const int nxt = (cur + 1) & 3;
            aim(nstage + 1 - s - NBUF);
            at_line(s + NBUF);
            step(f0, f2, cur, 2, 0, cur, 0, 0);
            step(f1, f3, cur, 3, 0, cur, 0, 0);
            __builtin_amdgcn_s_waitcnt(wait_vm(kStageLoads));  // lines up to s + 2 have landed, s + 3 may be on its way
            lds_barrier();
            step(f2, f0, nxt, 0, kStageLoads / 2, cur, 0, 0);
            step(f3, f1, nxt, 1, kStageLoads - kStageLoads / 2, cur, 0, kStageLoads / 2);
            cur = nxt;
        }
        // the slices of the last stage that K has
        if (k_tail > 32) read_slice(f2, cur, 2);
        if (k_tail > 48) read_slice(f3, cur, 3);
        multiply(f0);
        if (k_tail > 16) multiply(f1);
        if (k_tail > 32) multiply(f2);
        if (k_tail > 48) multiply(f3);
    } else if constexpr (kDeep) {
        // One stage of the deep form.  A slice's fragments are read two slices ahead: with one wave on the SIMD, a slice of
        // TMW x TNW MFMAs (32 cycles each) is shorter than the return of the reads dealt between them, and each slice
        // waited for the last of its own (128 x 128 tile: 1170 cycles a stage, 850 with this order, of which the LDS port
        // needs 768).  So slices 0 and 1 of the next stage are read in the second half of this one, and the barrier, which
        // lets them, sits in the middle.  It waits for no LDS read: the buffer that loads go to behind it is that of the
        // stage before, whose fragments every wave has multiplied by then.
        Frag f2, f3;
        read_frag(f1, 0, 1);
        for (int s = 0; s < nstage; s++) {
            const int nxt = (cur + 1) & 3, prev = (cur + 3) & 3;
            const int k_later = min(s + kAhead, nstage - 1) * KS;
            aim(nstage - s - kAhead);
            step(f0, f2, cur, 2, 0, prev, k_later, 0);
            step(f1, f3, cur, 3, 0, prev, k_later, 0);
            __builtin_amdgcn_s_waitcnt(wait_vm(kStageLoads));  // stage s + 1 has landed, s + 2 may be on its way
            if (RAGGED && s + 2 == nstage && ktail < kDmaK) {
                zero_tail(nxt);
                lds_barrier();
            } else {
                asm volatile("s_barrier" ::: "memory");
            }
            step(f2, f0, nxt, 0, kStageLoads / 2, prev, k_later, 0);
            step(f3, f1, nxt, 1, kStageLoads - kStageLoads / 2, prev, k_later, kStageLoads / 2);
            cur = nxt;
        }
    } else {
        // One stage of the others, with the matrix pipe fed across the barrier: every K slice is read from LDS
        // while the one before it is multiplied, the first slice of the next stage included, so the
        // barrier of the stage sits before its last slice.  The loads of stage s + kAhead are issued
        // in stage s into the buffer stage s - 1 was read from (its last readers passed
        // the previous barrier); stage s + 1 is waited for just before the barrier.  The fragment
        // read after the barrier of the last stage touches valid LDS and is never used; the loop
        // has a single exit (a second one in the middle makes the register allocator copy the
        // accumulators).
        for (int s = 0; s < nstage; s++) {
            const int nxt = cur + 1 == NBUF ? 0 : cur + 1;
            const int prev = cur == 0 ? NBUF - 1 : cur - 1;
            const int k_later = min(s + kAhead, nstage - 1) * KS;
            if constexpr (kWhole) {
                aim(nstage - s - kAhead);
                step(f0, f1, cur, 1, kStepLoads, prev, k_later, 0);
                if constexpr (kSlices == 4) {
                    step(f1, f0, cur, 2, 0, prev, k_later, 0);
                    step(f0, f1, cur, 3, 0, prev, k_later, 0);
                }
                // outstanding at most: the stages after s + 1 as far as they have been issued
                __builtin_amdgcn_s_waitcnt(wait_vm((kAhead - 2) * kStageLoads + kStepLoads));
                if (RAGGED && s + 2 == nstage && ktail < kDmaK) zero_tail(nxt);
                lds_barrier();
                step(f1, f0, nxt, 0, kLoadSteps == 2 ? kStepLoads2 : 0, prev, k_later, kStepLoads);
            } else {
                if (s + kAhead < nstage) load_stage(prev, (s + kAhead) * kDmaK);
                read_frag(f1, cur, 1);
                multiply(f0);
                __builtin_amdgcn_sched_barrier(0);
                read_frag(f0, cur, 2);
                multiply(f1);
                __builtin_amdgcn_sched_barrier(0);
                read_frag(f1, cur, 3);
                multiply(f0);
                __builtin_amdgcn_sched_barrier(0);
                wait_stages(min(kAhead - 1, nstage - 2 - s));
                if (RAGGED && s + 2 == nstage && ktail < kDmaK) zero_tail(nxt);
                lds_barrier();
                read_frag(f0, nxt, 0);
                multiply(f1);
                __builtin_amdgcn_sched_barrier(0);
            }
            cur = nxt;
        }
    }
    // the loads issued past the last stage have landed before the staging LDS is written again
    if constexpr (kWhole) __builtin_amdgcn_s_waitcnt(wait_vm(0));
    __syncthreads();  // the staging LDS becomes the transposition buffer of the epilogue

    // Epilogue.  acc[i][j][e] is token WM wm + 32 i + l32, feature WN wn + 32 j + 8 (e / 4) +
    // 4 kg + e % 4 of the tile: a lane holds 4 consecutive features of one row, 32 rows per
    // instruction.  Each wave passes its 32 x WN strips through its own LDS region and stores
    // rows of 2 WN contiguous bytes.
    constexpr int kEpLd = WN + 8;
    constexpr int kRowChunks = WN / 8;  // 16-byte chunks of a stored row: 4, 8, 12 or 16
    _Float16 *ep = reinterpret_cast<_Float16 *>(dma_smem) + wave * 32 * kEpLd;
    // Scattered columns are stored one 2-byte element per lane, kScLanes consecutive result
    // columns of one row per group of lanes: ascending c_scatter keeps those stores within a
    // few neighbouring sectors of the row of C.
    constexpr int kScRows = 64 / kScLanes;       // rows per instruction
    const bool scatter = IDX && g.c_scatter != nullptr;  // a gathered bias alone keeps the vector stores
    // (a strip is written and read by one wave, whose LDS accesses execute in order: only the compiler has to keep it.  A
    // workgroup barrier here waits for every store to memory besides.)
    auto wave_order = [] { asm volatile("" ::: "memory"); };
    const int act = g.act;
#pragma unroll
    for (int e = 0; e < kScCols; e++)
        if (lane < kScLanes) ep[e * kScLanes + lane] = has_bias ? bias_of[e] : (_Float16)0.0f;
    wave_order();
    h4 bias4[TNW][4];
#pragma unroll
    for (int j = 0; j < TNW; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) bias4[j][q] = *reinterpret_cast<const h4 *>(ep + j * 32 + q * 8 + kg * 4);
    wave_order();
#pragma unroll
    for (int i = 0; i < TMW; i++) {
        float v[TNW][16];  // (the activation is chosen once for a strip: chosen per value, each took its own branches, one after the other)
#pragma unroll
        for (int j = 0; j < TNW; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) v[j][e] = acc[i][j][e] + (float)bias4[j][e / 4][e % 4];
        if (act == ET_ACT_GELU) {
#pragma unroll
            for (int j = 0; j < TNW; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) v[j][e] = gelu_tanh(v[j][e]);
        } else if (act == ET_ACT_RELU) {
#pragma unroll
            for (int j = 0; j < TNW; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) v[j][e] = v[j][e] > 0.0f ? v[j][e] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < TNW; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                *reinterpret_cast<h4 *>(ep + l32 * kEpLd + j * 32 + q * 8 + kg * 4) =
                    h4{(_Float16)v[j][q * 4], (_Float16)v[j][q * 4 + 1], (_Float16)v[j][q * 4 + 2], (_Float16)v[j][q * 4 + 3]};
        wave_order();
        if (scatter) {
#pragma unroll
            for (int v = 0; v < 32 / kScRows; v++) {
                const int r = v * kScRows + lane / kScLanes;
                const int m = m0 + wm * WM + i * 32 + r;
                _Float16 *crow = g.C + (size_t)m * g.ldc;
#pragma unroll
                for (int e = 0; e < kScCols; e++) {
                    const bool inside = !RAGGED || (m < g.M && nbase + e * kScLanes + lane % kScLanes < g.N);
                    if (inside) crow[bias_at[e]] = ep[r * kEpLd + e * kScLanes + lane % kScLanes];
                }
            }
        } else {
#pragma unroll
            for (int v = 0; v < 32 * kRowChunks / 64; v++) {
                const int idx = lane + v * 64, r = idx / kRowChunks, c = idx % kRowChunks;
                const h8 val = *reinterpret_cast<const h8 *>(ep + r * kEpLd + c * 8);
                const int m = m0 + wm * WM + i * 32 + r;
                // N is a multiple of 16: a chunk of 8 columns is inside or outside as a whole
                if (!RAGGED || (m < g.M && nbase + c * 8 < g.N))
                    *reinterpret_cast<h8 *>(g.C + (size_t)m * g.ldc + nbase + c * 8) = val;
            }
        }
        wave_order();
    }
}

// The kernel moves 16 bytes at a time: operands and result 16-byte aligned, leading dimensions
// multiples of 8.
bool gemm_dma_applies(const GemmArgs &g, int batch, bool trans_b) {
    DmaTile t;
    const auto misaligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; };
    if (batch < 1 || batch > 65535 || g.a_gather || g.M <= 0) return false;
    if (g.lda % 8 || g.ldb % 8 || g.ldc % 8 || misaligned(g.A) || misaligned(g.B) || misaligned(g.C)) return false;
    if (g.lda > (1 << 21) || g.ldb > (1 << 21)) return false;  // a tile's rows are addressed with 32-bit byte offsets
    if (batch > 1 && ((g.sAo | g.sAi | g.sBo | g.sBi | g.sCo | g.sCi) & 7)) return false;  // every problem aligned
    return pick_dma_tile(g.M, g.N, g.K, batch, trans_b, &t);
}

template <int TMW, int TNW, int NBUF, bool IDX, bool RAGGED, bool BT = false, int KS = kDmaK, int NWN = 2, bool LINES = false>
static int launch_dma_variant(const GemmArgs &g, int batch, hipStream_t stream) {
    constexpr int BM = 64 * TMW, BN = 32 * NWN * TNW;
    constexpr size_t lds = dma_lds_bytes(TMW, TNW, NBUF, KS, NWN);
    const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
    // groups of group_rows x 8 tiles are dealt to the XCDs in turn: the size (32, 16 or 8 tiles) that leaves the
    // fullest XCD the fewest tiles, the larger on a tie
    const long long total = (long long)tiles_m * tiles_n;
    int sbm = kSbM;
    long long best = -1;
    for (int cand = kSbM; cand >= 1; cand /= 2) {
        const long long gsz = (long long)cand * kSbN, ngr = (total + gsz - 1) / gsz;
        const long long most = (ngr + kDmaXcds - 1) / kDmaXcds * gsz;
        if (best < 0 || most < best) { best = most; sbm = cand; }
    }
    const long long groups = (total + sbm * kSbN - 1) / (sbm * kSbN);
    const long long rounds = (groups + kDmaXcds - 1) / kDmaXcds;
    const dim3 grid((unsigned)(rounds * kDmaXcds * sbm * kSbN), (unsigned)batch);
    const unsigned long long per_br = (unsigned long long)sbm * tiles_n, most = (unsigned long long)grid.x * per_br;
    const unsigned per_row = per_br > 1 && most < 1ull << 32 ? (unsigned)(((1ull << 32) + per_br - 1) / per_br) : 0;
    auto kernel = gemm_f16_dma_kernel<TMW, TNW, NBUF, IDX, RAGGED, BT, KS, NWN, LINES>;
    static bool raised = false;  // more than 64 KB of dynamic LDS needs the attribute, once per kernel
    if (!raised) {
        ET_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        raised = true;
    }
    return launch_kernel("gemm_f16_dma_kernel", kernel, grid, 128 * NWN, lds, stream, g.A, g.B, g.bias, g.M, g.N, g.K, g.lda, g.ldb, sbm, per_row, g);
}

// rows that do not all begin on a 128-byte line
static bool off_lines(const _Float16 *p, int ld) { return ld % 64 || (reinterpret_cast<uintptr_t>(p) & 127); }

template <int TMW, int TNW, int NBUF, bool RAGGED = false, bool BT = false, int KS = kDmaK, int NWN = 2, bool LINES = false>
static int launch_dma_tile(const GemmArgs &g, int batch, hipStream_t stream) {
    if constexpr (RAGGED && !BT && NBUF == 4 && !LINES) {
        if (off_lines(g.A, g.lda) || off_lines(g.B, g.ldb)) return launch_dma_tile<TMW, TNW, NBUF, true, false, KS, NWN, true>(g, batch, stream);
    }
    return (g.c_scatter || g.bias_idx) ? launch_dma_variant<TMW, TNW, NBUF, true, RAGGED, BT, KS, NWN, LINES>(g, batch, stream)
                                       : launch_dma_variant<TMW, TNW, NBUF, false, RAGGED, BT, KS, NWN, LINES>(g, batch, stream);
}

int launch_gemm_dma(const GemmArgs &g, int batch, bool trans_b, hipStream_t stream) {
    DmaTile t{};
    if (!pick_dma_tile(g.M, g.N, g.K, batch, trans_b, &t)) return ET_ERR_UNSUPPORTED;
    if (!trans_b)
        return t.nbuf == 3 ? launch_dma_tile<1, 1, 3, true, true>(g, batch, stream)
                           : launch_dma_tile<1, 1, 2, true, true>(g, batch, stream);
    if (t.ragged && (off_lines(g.A, g.lda) || off_lines(g.B, g.ldb))) t = dma_lines_tile(t, g.M, g.N, g.K);
    switch (t.tmw * 100 + t.tnw * 10 + t.nbuf + (t.ragged ? 1000 : 0)) {
        case 114: return launch_dma_tile<1, 1, 4>(g, 1, stream);
        case 124: return launch_dma_tile<1, 2, 4>(g, 1, stream);
        case 134: return launch_dma_tile<1, 3, 4>(g, 1, stream);
        case 212: return launch_dma_tile<2, 1, 2>(g, 1, stream);
        case 214: return launch_dma_tile<2, 1, 4>(g, 1, stream);
        case 222: return launch_dma_tile<2, 2, 2>(g, 1, stream);
        case 224: return launch_dma_tile<2, 2, 4>(g, 1, stream);
        case 233: return launch_dma_tile<2, 3, 3>(g, 1, stream);
        // 256 x 256: eight waves of 128 x 64, half stages through four buffers (four waves of 128 x 128 in the same
        // LDS: 0.5-2 % slower)
        case 444: return launch_dma_tile<4, 2, 4, false, false, 32, 4>(g, 1, stream);
        case 1114: return launch_dma_tile<1, 1, 4, true>(g, batch, stream);
        case 1124: return launch_dma_tile<1, 2, 4, true>(g, 1, stream);
        case 1134: return launch_dma_tile<1, 3, 4, true>(g, 1, stream);
        case 1212: return launch_dma_tile<2, 1, 2, true>(g, 1, stream);
        case 1214: return launch_dma_tile<2, 1, 4, true>(g, 1, stream);
        case 1222: return launch_dma_tile<2, 2, 2, true>(g, 1, stream);
        case 1224: return launch_dma_tile<2, 2, 4, true>(g, 1, stream);
        case 1234: return launch_dma_tile<2, 3, 4, true, false, kDmaK, 2, true>(g, 1, stream);  // (by lines only)
        case 1233: return launch_dma_tile<2, 3, 3, true>(g, 1, stream);
        case 1442: return launch_dma_tile<4, 4, 2, true>(g, 1, stream);
        default: return ET_ERR_UNSUPPORTED;
    }
}

}  // namespace et
