// fp32 twins of the dense Linear and the fused attention: every value is stored,
// multiplied and accumulated in binary32 (MFMA 16x16x4 f32 for the Linear, vector
// FMA for the attention core), so an encoder layer built from them agrees with a
// CPU fp32 forward to ~1e-5.  This is the verification path for dense fp32 models
// (the reference is fp16-only, Linear/Linear.h:9); the production path is fp16.
#include "common.hip.h"

namespace et {

// ---- dense Linear ---------------------------------------------------------------
// Y[T x out] = act(X[T x in] * W^T + b), W [out x in] row-major.  One workgroup of
// 4 waves computes a 64-token x 64-feature block; wave (wr, wc) owns tokens
// 32*wr.. and features 32*wc.. as 2x2 MFMA tiles.  The MFMA A operand is W and the B
// operand is X, so a lane ends with 4 consecutive output features of one token
// (one 16-byte store).
constexpr int kF32K = 64;       // k-values staged per step
constexpr int kF32Ld = kF32K + 1;  // LDS row stride in floats (odd: conflict-free column reads)

// TILE x TILE outputs per workgroup (64 or 32), a wave TILE/2 x TILE/2 of them.  The small
// tile is for problems that would leave compute units idle with the large one: the fp32 MFMA
// rate of the waves that run is what bounds a small problem.
// The pruned forms run the same kernel.  GATHER (column-pruned weight): W is [out x in] over the
// surviving input features and feature k of W multiplies X[:, in_id[k]].  OUT (row-pruned weight,
// W = its surviving rows): kOutScatter stores feature f in column out_id[f] of Y with bias[out_id[f]];
// kOutCompact stores it in column f with that same bias.  ldx and ldy are the row strides of X and Y.
constexpr int kOutPlain = 0, kOutScatter = 1, kOutCompact = 2;
struct LinearF32Args {
    const float *W, *bias, *X;
    float *Y;
    const int32_t *in_id, *out_id;
    int T, in, out, ldx, ldy;
};
template <int ACT, int TILE, bool GATHER, int OUT>
__global__ __launch_bounds__(256) void linear_dense_f32_kernel(const float *__restrict__ W, const float *__restrict__ X, const float *__restrict__ bias, int T, int in,
                                                               int out, int ldx, const LinearF32Args rest) {
    LinearF32Args a = rest;  // (those in front are preloaded into scalar registers)
    a.ldx = ldx;
    float *__restrict__ Y = a.Y;
    constexpr int WB = TILE / 2;          // wave block
    constexpr int MI = WB / 16;           // 16 x 16 MFMA tiles per wave and dimension
    constexpr int TPR = 256 / TILE;       // staging threads per row
    constexpr int VPT = kF32K / 4 / TPR;  // float4 per thread, operand and step
    __shared__ float xs[TILE * kF32Ld];
    __shared__ float ws[TILE * kF32Ld];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = wave >> 1, wc = wave & 1;
    const int tok0 = blockIdx.y * TILE, f0 = blockIdx.x * TILE;
    const int r16 = lane & 15, kq = lane >> 4;

    // staging: thread -> (row, 4 consecutive k at sk, sk + 4 TPR, ...)
    const int srow = threadIdx.x / TPR, sk = (threadIdx.x % TPR) << 2;
    const bool x_ok = tok0 + srow < T, w_ok = f0 + srow < out;
    const float *xp = X + (size_t)(tok0 + (x_ok ? srow : 0)) * a.ldx;
    const float *wp = W + (size_t)(f0 + (w_ok ? srow : 0)) * in;
    const float4 zero4 = float4{0.0f, 0.0f, 0.0f, 0.0f};
    float4 xv[VPT], wv[VPT];
    // unconditional loads from clamped addresses and a select (a load under a branch is waited
    // for on the spot); `in` is a multiple of 16, so a group of 4 is inside or outside
    auto load_step = [&](int k0) {
#pragma unroll
        for (int j = 0; j < VPT; j++) {
            const int k = k0 + sk + 4 * TPR * j;
            const bool k_ok = k < in;
            if (GATHER) {
                const int4 id = *reinterpret_cast<const int4 *>(a.in_id + (k_ok ? k : 0));
                xv[j] = float4{xp[id.x], xp[id.y], xp[id.z], xp[id.w]};
            } else {
                xv[j] = *reinterpret_cast<const float4 *>(xp + (k_ok ? k : 0));
            }
            wv[j] = *reinterpret_cast<const float4 *>(wp + (k_ok ? k : 0));
            if (!(x_ok && k_ok)) xv[j] = zero4;
            if (!(w_ok && k_ok)) wv[j] = zero4;
        }
    };

    f4 acc[MI][MI];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < MI; j++) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};

    load_step(0);
    for (int k0 = 0; k0 < in; k0 += kF32K) {
        __syncthreads();  // the previous step's reads are done
#pragma unroll
        for (int j = 0; j < VPT; j++) {
            float *xd = xs + srow * kF32Ld + sk + 4 * TPR * j, *wd = ws + srow * kF32Ld + sk + 4 * TPR * j;
            xd[0] = xv[j].x; xd[1] = xv[j].y; xd[2] = xv[j].z; xd[3] = xv[j].w;
            wd[0] = wv[j].x; wd[1] = wv[j].y; wd[2] = wv[j].z; wd[3] = wv[j].w;
        }
        __syncthreads();
        load_step(k0 + kF32K);  // the next step travels while this one is multiplied (past the end: zeros)
#pragma unroll
        for (int kk = 0; kk < kF32K; kk += 4) {
            float a[MI], b[MI];
#pragma unroll
            for (int i = 0; i < MI; i++) {
                a[i] = ws[(wc * WB + i * 16 + r16) * kF32Ld + kk + kq];  // A[m = feature][k]
                b[i] = xs[(wr * WB + i * 16 + r16) * kF32Ld + kk + kq];  // B[k][n = token]
            }
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < MI; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[i], acc[i][j], 0, 0, 0);
        }
    }
    // acc[i][j]: token tok0 + WB*wr + 16*i + r16, features f0 + WB*wc + 16*j + 4*kq .. +3
#pragma unroll
    for (int i = 0; i < MI; i++) {
        const int t = tok0 + wr * WB + i * 16 + r16;
        if (t >= T) continue;
#pragma unroll
        for (int j = 0; j < MI; j++) {
            const int f = f0 + wc * WB + j * 16 + kq * 4;
            if (f >= out) continue;  // out % 4 == 0: a group of 4 is inside or outside
            float4 o;
            float *po = reinterpret_cast<float *>(&o);
            int col[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                col[e] = OUT == kOutPlain ? f + e : a.out_id[f + e];
                float v = acc[i][j][e] + (bias ? bias[col[e]] : 0.0f);
                if (ACT == ET_ACT_RELU) v = v > 0.0f ? v : 0.0f;
                if (ACT == ET_ACT_GELU) v = gelu_tanh(v);
                po[e] = v;
            }
            if (OUT == kOutScatter) {
#pragma unroll
                for (int e = 0; e < 4; e++) Y[(size_t)t * a.ldy + col[e]] = po[e];
            } else {
                *reinterpret_cast<float4 *>(Y + (size_t)t * a.ldy + f) = o;
            }
        }
    }
}

// ---- fused attention ------------------------------------------------------------
// One workgroup of 4 waves = 16 queries of one head of one sequence.  The 16 x S strip of scores lives in LDS; Q, K and V
// go from memory straight into the operands of v_mfma_f32_16x16x4_f32, with a lane's four k-values a 16-wide cell's
// 4q .. 4q+3 (a sum over k does not care which k a lane brings as long as both operands bring the same one).
//   scores: waves take 16 keys in turn; A = K (row = key), B = Q, so lane (r, q) ends with keys 4q .. 4q+3 of query r
//   softmax: 16 threads a query
//   Z: waves take 16 features in turn; A = V transposed (row = feature), B = P: features 4q .. 4q+3 of query r
// A few hundred workgroups is all a verification batch has, so the length of one workgroup's chain is its time: HD / 4
// products a key block and S / 4 a feature block, 32 cycles each.  2 x 128 tokens, 12 heads of 64: 20.3 -> 7.1 us, 1 x 512 tokens 85 -> 26 (the
// former kernel staged K and V element by element and multiplied on the vector unit).
// So the query and the first keys are requested together at the start, the next keys ahead of the products, and the first
// values before the softmax: 12 heads of 64, 16 tokens 3.9 us, 1 x 64 4.9, 2 x 128 6.6, 1 x 256 9.8.  With neither ahead 3.9, 5.1,
// 7.2 and 11.0; with the first values at the start, a branch around each cell and four blocks of values at once 4.2, 5.4, 7.6
// and 11.5 (6 layers of 256 tokens 286 us, now 276).
constexpr int kAttQ = 16;
constexpr int kAttKeys = 64;  // (of the LDS limit of et_mha_fused_f32)
constexpr int kAttAhead = 2;  // blocks of 16 keys whose values are asked for at once
constexpr int kAttPad = 4;    // floats between the rows of the strip: 16 rows' cells in different banks, 16-byte aligned

struct MhaF32Args {
    const float *Q, *K, *V;
    float *Z;
    const float *mask;
    const int32_t *lens;
    int ldq, ldk, ldv, ldz;
    int B, S, nh, hd;
    float scale;
    int causal;
};

template <bool VEC> __device__ __forceinline__ f4 load_quad_f32(const float *p) {
    if constexpr (VEC) return *reinterpret_cast<const f4 *>(p);
    else return f4{p[0], p[1], p[2], p[3]};
}

// VEC: rows of Q and K start at multiples of 16 bytes.  MAXC: cells of 16 features of a head, at most.
template <int MAXC, bool VEC>
__global__ __launch_bounds__(256) void mha_fused_f32_kernel(const float *Q, const float *K, const float *V, const int32_t *lens, int ldq, int ldk, int ldv, int S,
                                                            int hd_, int causal, const MhaF32Args rest) {
    MhaF32Args a = rest;  // (those in front are preloaded into scalar registers)
    a.Q = Q, a.K = K, a.V = V, a.lens = lens, a.ldq = ldq, a.ldk = ldk, a.ldv = ldv, a.S = S, a.hd = hd_, a.causal = causal;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float *sc = reinterpret_cast<float *>(smem_raw);  // [16][S + kAttPad]
    __shared__ float inv_sum[kAttQ];
    const int q0 = blockIdx.x * kAttQ, h = blockIdx.y, b = blockIdx.z;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int len = a.lens ? min(max(a.lens[b], 0), a.S) : a.S;
    const size_t row0 = (size_t)b * a.S;
    const int hd = a.hd, ncell = hd >> 4, ld = a.S + kAttPad;
    float *zrow = a.Z + (row0 + q0 + r16) * a.ldz + h * hd + 4 * g;
    if (len == 0) {  // a sequence without keys: zeros
        for (int c = wave; c < ncell; c += 4)
#pragma unroll
            for (int e = 0; e < 4; e++) zrow[c * 16 + e] = 0.0f;
        return;
    }
    // keys this block of queries can see
    int kend = len;
    if (a.causal) kend = min(kend, q0 + kAttQ);
    const int nkb = (kend + 15) >> 4;
    const float ninf = -__builtin_inff();

    // (Cells past the head: its last one again, not multiplied.  With a branch around each, a wave waited for every cell of its
    // query.)
    f4 qv[MAXC], kv[MAXC], v[kAttAhead];
    auto ask_row = [&](f4 (&to)[MAXC], const float *row) {
#pragma unroll
        for (int c = 0; c < MAXC; c++) to[c] = load_quad_f32<VEC>(row + 16 * min(c, ncell - 1));
    };
    auto ask_keys = [&](f4 (&k)[MAXC], int kb) {  // (keys past kend: the last one again, not used below)
        ask_row(k, a.K + (row0 + min(kb * 16 + r16, kend - 1)) * a.ldk + h * hd + 4 * g);
    };
    auto ask_values = [&](int c, int kb) {  // of kAttAhead blocks of keys
        const float *vp = a.V + row0 * a.ldv + h * hd + c * 16 + r16;
#pragma unroll
        for (int s = 0; s < kAttAhead; s++)
            if (s == 0 || kb + s < nkb)  // uniform
#pragma unroll
                for (int j = 0; j < 4; j++) v[s][j] = vp[(size_t)min((kb + s) * 16 + 4 * g + j, kend - 1) * a.ldv];
    };
    ask_row(qv, a.Q + (row0 + q0 + r16) * a.ldq + h * hd + 4 * g);
    ask_keys(kv, wave);
#pragma unroll
    for (int c = 0; c < MAXC; c++) qv[c] *= a.scale;

    // ---- scores
    for (int kb = wave; kb < nkb; kb += 4) {
        f4 next[MAXC];
        ask_keys(next, kb + 4);
        f4 s = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < MAXC; c++)
            if (c < ncell)
#pragma unroll
                for (int j = 0; j < 4; j++) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[c][j], qv[c][j], s, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int key = kb * 16 + 4 * g + e;
            if (a.mask && key < kend) s[e] += a.mask[(size_t)(q0 + r16) * a.S + key];
            if (key >= kend || (a.causal && key > q0 + r16)) s[e] = ninf;
        }
        *reinterpret_cast<f4 *>(sc + r16 * ld + kb * 16 + 4 * g) = s;
#pragma unroll
        for (int c = 0; c < MAXC; c++) kv[c] = next[c];
    }
    if (wave < ncell) ask_values(wave, 0);
    __syncthreads();
    // ---- softmax over the keys of row q: 16 threads per row (keys past kend become zeros)
    {
        const int q = threadIdx.x >> 4, c = threadIdx.x & 15;
        float m = ninf;
        for (int k = c; k < nkb * 16; k += 16) m = fmaxf(m, sc[q * ld + k]);
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 16));
        float l = 0.0f;
        for (int k = c; k < nkb * 16; k += 16) {
            const float p = m == ninf || k >= kend ? 0.0f : __expf(sc[q * ld + k] - m);
            sc[q * ld + k] = p;
            l += p;
        }
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) l += __shfl_xor(l, off, 16);
        if (c == 0) inv_sum[q] = l > 0.0f ? 1.0f / l : 0.0f;
    }
    __syncthreads();
    // ---- Z = P V (rows of V past kend are not multiplied, whatever they hold)
    const float inv = inv_sum[r16];
    for (int c = wave; c < ncell; c += 4) {
        f4 acc = f4{0.f, 0.f, 0.f, 0.f};
        if (c != wave) ask_values(c, 0);
        for (int kb = 0; kb < nkb; kb += kAttAhead) {
            f4 now[kAttAhead];
#pragma unroll
            for (int s = 0; s < kAttAhead; s++) {
                now[s] = v[s];
                if ((kb + s + 1) * 16 > kend)  // uniform
#pragma unroll
                    for (int j = 0; j < 4; j++) now[s][j] = (kb + s) * 16 + 4 * g + j < kend ? v[s][j] : 0.0f;
            }
            if (kb + kAttAhead < nkb) ask_values(c, kb + kAttAhead);
#pragma unroll
            for (int s = 0; s < kAttAhead; s++) {
                if (kb + s >= nkb) break;  // uniform
                const f4 p = *reinterpret_cast<const f4 *>(sc + r16 * ld + (kb + s) * 16 + 4 * g);
#pragma unroll
                for (int j = 0; j < 4; j++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(now[s][j], p[j], acc, 0, 0, 0);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) zrow[c * 16 + e] = acc[e] * inv;
    }
}

template <int OP>
__global__ __launch_bounds__(256) void unary_f32_kernel(float *__restrict__ out, const float *__restrict__ in,
                                                        size_t n) {
    const size_t step = (size_t)gridDim.x * blockDim.x;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += step) {
        const float x = in[i];
        out[i] = OP == 0 ? gelu_tanh(x) : (x > 0.0f ? x : 0.0f);
    }
}

// Y[r][c] = act(bias[c]) (act(0) without a bias): the value of a pruned output feature.
__global__ __launch_bounds__(256) void fill_rows_bias_act_f32_kernel(float *__restrict__ Y,
                                                                     const float *__restrict__ bias, size_t n,
                                                                     int cols, int act) {
    const size_t step = (size_t)gridDim.x * blockDim.x;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += step)
        Y[i] = apply_act(bias ? bias[i % cols] : 0.0f, act);
}

}  // namespace et

using namespace et;

extern "C" {

// One launch of the Linear kernel in the form (gather, out mode, activation) names.
static int launch_linear_f32(const LinearF32Args &a, int act, bool gather, int out_mode, hipStream_t st) {
    // 64 x 64 tiles once they give every compute unit a workgroup, 32 x 32 below that
    const bool small = (long long)((a.out + 63) / 64) * ((a.T + 63) / 64) < 256;
    const int tile = small ? 32 : 64;
    const dim3 grid((a.out + tile - 1) / tile, (a.T + tile - 1) / tile);
#define ET_F32_FORM(ACTV, G, O)                                                       \
    {                                                                                 \
        if (small) linear_dense_f32_kernel<ACTV, 32, G, O><<<grid, 256, 0, st>>>(a.W, a.X, a.bias, a.T, a.in, a.out, a.ldx, a);  \
        else linear_dense_f32_kernel<ACTV, 64, G, O><<<grid, 256, 0, st>>>(a.W, a.X, a.bias, a.T, a.in, a.out, a.ldx, a);        \
    }
#define ET_F32_LINEAR(ACTV)                                                \
    {                                                                      \
        if (gather) ET_F32_FORM(ACTV, true, kOutPlain)                     \
        else if (out_mode == kOutScatter) ET_F32_FORM(ACTV, false, kOutScatter)  \
        else if (out_mode == kOutCompact) ET_F32_FORM(ACTV, false, kOutCompact)  \
        else ET_F32_FORM(ACTV, false, kOutPlain)                           \
    }
    switch (act) {
        case ET_ACT_RELU: ET_F32_LINEAR(ET_ACT_RELU) break;
        case ET_ACT_GELU: ET_F32_LINEAR(ET_ACT_GELU) break;
        default: ET_F32_LINEAR(ET_ACT_NONE) break;
    }
#undef ET_F32_LINEAR
#undef ET_F32_FORM
    return check_launch("linear_dense_f32_kernel");
}

static inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int et_linear_dense_f32(const float *W, const float *bias, const float *X, float *Y, int T, int in, int out,
                        int act, et_stream stream) {
    ET_REQUIRE(W && X && Y, ET_ERR_INVALID_ARG, "et_linear_dense_f32: NULL pointer");
    ET_REQUIRE(T >= 0 && in > 0 && out > 0, ET_ERR_INVALID_ARG, "et_linear_dense_f32: T=%d in=%d out=%d", T, in, out);
    ET_REQUIRE(act >= ET_ACT_NONE && act <= ET_ACT_GELU, ET_ERR_INVALID_ARG, "et_linear_dense_f32: act=%d", act);
    ET_REQUIRE(in % 16 == 0 && out % 4 == 0, ET_ERR_UNSUPPORTED,
               "et_linear_dense_f32: in=%d must be a multiple of 16, out=%d of 4", in, out);
    ET_REQUIRE(aligned16(W) && aligned16(X) && aligned16(Y), ET_ERR_UNSUPPORTED,
               "et_linear_dense_f32: W, X and Y must be 16-byte aligned");
    if (T == 0) return ET_OK;
    const LinearF32Args a{W, bias, X, Y, nullptr, nullptr, T, in, out, in, out};
    return launch_linear_f32(a, act, false, kOutPlain, as_stream(stream));
}

int et_linear_rowpruned_f32(const float *rows, const int32_t *row_id, int nnz_row, const float *bias,
                            const float *X, float *Y, int T, int in, int out, int act, et_stream stream) {
    ET_REQUIRE(X && Y && (nnz_row == 0 || (rows && row_id)), ET_ERR_INVALID_ARG, "et_linear_rowpruned_f32: NULL pointer");
    ET_REQUIRE(T >= 0 && in > 0 && out > 0 && nnz_row >= 0 && nnz_row <= out, ET_ERR_INVALID_ARG,
               "et_linear_rowpruned_f32: T=%d in=%d out=%d nnz_row=%d", T, in, out, nnz_row);
    ET_REQUIRE(act >= ET_ACT_NONE && act <= ET_ACT_GELU, ET_ERR_INVALID_ARG, "et_linear_rowpruned_f32: act=%d", act);
    ET_REQUIRE(in % 16 == 0 && nnz_row % 4 == 0, ET_ERR_UNSUPPORTED,
               "et_linear_rowpruned_f32: in=%d must be a multiple of 16, nnz_row=%d of 4", in, nnz_row);
    ET_REQUIRE(aligned16(rows) && aligned16(X), ET_ERR_UNSUPPORTED,
               "et_linear_rowpruned_f32: rows and X must be 16-byte aligned");
    if (T == 0) return ET_OK;
    hipStream_t st = as_stream(stream);
    // pruned features: act(bias) — every column is written first, the surviving ones again below
    const size_t n = (size_t)T * out;
    fill_rows_bias_act_f32_kernel<<<(unsigned)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536), 256, 0, st>>>(
        Y, bias, n, out, act);
    const int s = check_launch("fill_rows_bias_act_f32_kernel");
    if (s != ET_OK || nnz_row == 0) return s;
    const LinearF32Args a{rows, bias, X, Y, nullptr, row_id, T, in, nnz_row, in, out};
    return launch_linear_f32(a, act, false, kOutScatter, st);
}

int et_linear_rowpruned_compact_f32(const float *rows, const int32_t *row_id, int nnz_row, const float *bias,
                                    const float *X, float *Yc, int T, int in, et_stream stream) {
    ET_REQUIRE(rows && row_id && X && Yc, ET_ERR_INVALID_ARG, "et_linear_rowpruned_compact_f32: NULL pointer");
    ET_REQUIRE(T >= 0 && in > 0 && nnz_row > 0, ET_ERR_INVALID_ARG,
               "et_linear_rowpruned_compact_f32: T=%d in=%d nnz_row=%d", T, in, nnz_row);
    ET_REQUIRE(in % 16 == 0 && nnz_row % 4 == 0, ET_ERR_UNSUPPORTED,
               "et_linear_rowpruned_compact_f32: in=%d must be a multiple of 16, nnz_row=%d of 4", in, nnz_row);
    ET_REQUIRE(aligned16(rows) && aligned16(X) && aligned16(Yc), ET_ERR_UNSUPPORTED,
               "et_linear_rowpruned_compact_f32: rows, X and Yc must be 16-byte aligned");
    if (T == 0) return ET_OK;
    const LinearF32Args a{rows, bias, X, Yc, nullptr, row_id, T, in, nnz_row, in, nnz_row};
    return launch_linear_f32(a, ET_ACT_NONE, false, bias ? kOutCompact : kOutPlain, as_stream(stream));
}

int et_linear_colpruned_f32(const float *cols, const int32_t *col_id, int nnz_col, const float *bias,
                            const float *X, float *Y, int T, int in, int out, int act, et_stream stream) {
    ET_REQUIRE(cols && col_id && X && Y, ET_ERR_INVALID_ARG, "et_linear_colpruned_f32: NULL pointer");
    ET_REQUIRE(T >= 0 && in > 0 && out > 0 && nnz_col > 0 && nnz_col <= in, ET_ERR_INVALID_ARG,
               "et_linear_colpruned_f32: T=%d in=%d out=%d nnz_col=%d", T, in, out, nnz_col);
    ET_REQUIRE(act >= ET_ACT_NONE && act <= ET_ACT_GELU, ET_ERR_INVALID_ARG, "et_linear_colpruned_f32: act=%d", act);
    ET_REQUIRE(nnz_col % 16 == 0 && out % 4 == 0, ET_ERR_UNSUPPORTED,
               "et_linear_colpruned_f32: nnz_col=%d must be a multiple of 16, out=%d of 4", nnz_col, out);
    ET_REQUIRE(aligned16(cols) && aligned16(col_id) && aligned16(Y), ET_ERR_UNSUPPORTED,
               "et_linear_colpruned_f32: cols, col_id and Y must be 16-byte aligned");
    if (T == 0) return ET_OK;
    const LinearF32Args a{cols, bias, X, Y, col_id, nullptr, T, nnz_col, out, in, out};
    return launch_linear_f32(a, act, true, kOutPlain, as_stream(stream));
}

int et_mha_fused_f32(const float *Q, const float *K, const float *V, int ldq, int ldk, int ldv, float *Z, int ldz,
                     const float *mask, const int32_t *lens, int B, int S, int nh, int hd, float scale, int flags,
                     et_stream stream) {
    ET_REQUIRE(Q && K && V && Z, ET_ERR_INVALID_ARG, "et_mha_fused_f32: NULL pointer");
    ET_REQUIRE(B >= 0 && S > 0 && nh > 0, ET_ERR_INVALID_ARG, "et_mha_fused_f32: B=%d S=%d nh=%d", B, S, nh);
    ET_REQUIRE((flags & ~ET_MHA_CAUSAL) == 0, ET_ERR_INVALID_ARG, "et_mha_fused_f32: flags=%d", flags);
    ET_REQUIRE(S % 16 == 0 && hd > 0 && hd % 16 == 0 && hd <= 128, ET_ERR_UNSUPPORTED,
               "et_mha_fused_f32: S=%d and hd=%d must be multiples of 16, hd at most 128", S, hd);
    const int width = nh * hd;
    ET_REQUIRE(ldq >= width && ldk >= width && ldv >= width && ldz >= width, ET_ERR_INVALID_ARG,
               "et_mha_fused_f32: row strides must cover nh*hd=%d", width);
    // (as large as with K and V staged in blocks of 64 rows, the form of the kernel that set the limit)
    const int hdt = hd <= 32 ? 32 : hd <= 64 ? 64 : 128;
    const size_t lds = sizeof(float) * ((size_t)kAttQ * hdt + (size_t)kAttKeys * (hdt + 1) + (size_t)kAttQ * S);
    ET_REQUIRE(lds <= 160 * 1024, ET_ERR_UNSUPPORTED, "et_mha_fused_f32: S=%d does not fit the on-chip score strip", S);
    if (B == 0) return ET_OK;
    MhaF32Args a{Q, K, V, Z, mask, lens, ldq, ldk, ldv, ldz, B, S, nh, hd, scale, (flags & ET_MHA_CAUSAL) ? 1 : 0};
    const dim3 grid(S / kAttQ, nh, B);
    const size_t strip = sizeof(float) * kAttQ * (size_t)(S + kAttPad);  // (less than the limit above is for)
    hipStream_t st = as_stream(stream);
#define ET_MHA32(MAXC, VEC)                                                                                  \
    {                                                                                                        \
        auto kern = mha_fused_f32_kernel<MAXC, VEC>;                                                         \
        if (strip > 64 * 1024)                                                                               \
            ET_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),                                 \
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)strip));             \
        kern<<<grid, 256, strip, st>>>(a.Q, a.K, a.V, a.lens, a.ldq, a.ldk, a.ldv, a.S, a.hd, a.causal, a);  \
    }
    // 16-byte loads of Q and K where every row starts at a multiple of 16 bytes
    const bool vec = aligned16(Q) && aligned16(K) && ldq % 4 == 0 && ldk % 4 == 0;
    if (hd <= 64) {
        if (vec) ET_MHA32(4, true) else ET_MHA32(4, false)
    } else {
        if (vec) ET_MHA32(8, true) else ET_MHA32(8, false)
    }
#undef ET_MHA32
    return check_launch("mha_fused_f32_kernel");
}

int et_gelu_f32(float *out, const float *in, size_t n, et_stream stream) {
    ET_REQUIRE((out && in) || n == 0, ET_ERR_INVALID_ARG, "et_gelu_f32: NULL pointer");
    if (n == 0) return ET_OK;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    unary_f32_kernel<0><<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(out, in, n);
    return check_launch("unary_f32_kernel<gelu>");
}

int et_relu_f32(float *out, const float *in, size_t n, et_stream stream) {
    ET_REQUIRE((out && in) || n == 0, ET_ERR_INVALID_ARG, "et_relu_f32: NULL pointer");
    if (n == 0) return ET_OK;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    unary_f32_kernel<1><<<(unsigned)blocks, 256, 0, as_stream(stream)>>>(out, in, n);
    return check_launch("unary_f32_kernel<relu>");
}

}  // extern "C"
