// MLP surrogate of a feature map: trained and evaluated with hand-written
// BF16 matrix-core (MFMA) kernels accumulating in FP32, for gfx950.
//
// No counterpart in the reference.  The network maps 2 normalised parameters
// to feature predictions:
//   encode   x (2) -> 16 fixed Fourier features, sin and cos    -> 32
//   layer 1  32  -> 256, SiLU
//   layer 2  256 -> 256, SiLU
//   layer 3  256 -> 256, SiLU
//   layer 4  256 -> 256, SiLU
//   heads    256 -> 4 heads x (log-period, amplitude, 16 class logits) = 72,
//            padded to 128 output columns (the padding stays exactly zero)
// Weights are kept transposed, Wt[out][in], as FP32 master copies (Adam) and
// BF16 copies (MFMA operands).  Activations are BF16, pre-activations FP32.
//
// The 4 heads share the trunk and are trained on different bootstrap subsets
// of every minibatch (a sample is seen by a head unless a hash of
// (sample, head) is 0 mod 4), so their disagreement measures the network's
// uncertainty.  Screening flags a grid cell for re-solving by the integrator
// when the heads disagree, when the predicted class differs from a
// neighbour's, and within a dilation radius of such cells.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <random>
#include <string>
#include <vector>

#include "../../../include/clode_mlp.h"
#include "../runtime/staged_copy.h"
#include "normals.h"

// Staging memory of clode_mlp_screen_grid_noalloc: one byte per grid cell for
// the dilation's second flag buffer.  Each device holds its own copy of the
// array; host code reaches it only through the address that
// hipGetSymbolAddress returns on that device (clode_mlp_create records it).
static __device__ __align__(256) unsigned char scratch[CLODE_MLP_NOALLOC_MAX_CELLS];

namespace {

constexpr int NFF = 16;         // Fourier frequencies
constexpr int D0 = 2 * NFF;     // encoded input width
constexpr int H = 256;          // hidden width
constexpr int NHID = 4;         // hidden layers
constexpr int NHEAD = 4;        // heads
constexpr int NCLS = 16;        // classes
constexpr int HW = 2 + NCLS;    // outputs per head
constexpr int NOUT = NHEAD * HW;  // 72 used output columns
constexpr int NOUTP = 128;      // padded output columns
constexpr int NLAYER = NHID + 1;

typedef uint16_t bf16_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

// round to nearest even (NaN kept quiet), identical on host and device
__host__ __device__ inline bf16_t f2bf(float f)
{
    uint32_t u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x007fffffu))
        return (bf16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}
__host__ __device__ inline float bf2f(bf16_t h)
{
    uint32_t u = (uint32_t)h << 16;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

// logistic sigmoid with the hardware exponential and reciprocal (v_exp_f32,
// v_rcp_f32; about 1 ulp each): the GEMM epilogues evaluate it once per
// output element, and an IEEE division there cost more than the products
__device__ inline float sigm(float z) { return __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }
__device__ inline float silu(float z) { return z * sigm(z); }
__device__ inline float dsilu(float z)
{
    const float s = sigm(z);
    return s * (1.0f + z * (1.0f - s));
}
// float -> BF16 on the device, round to nearest even: the gfx950 conversion
// instruction, which agrees with f2bf for every finite input
__device__ inline bf16_t f2bf_dev(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }

// ---------------------------------------------------------------- GEMM
// C[M x N] = A[M x K] * B[K x N] with arbitrary strides on both operands,
// BF16 operands, FP32 accumulation on v_mfma_f32_16x16x32_bf16, and a fused
// epilogue.  Workgroup tile 64 x 64 (4 waves of 32 x 32, each 2 x 2 MFMA
// blocks), MFMA K step 32.  K is staged through LDS in chunks of 128 with k
// contiguous (each lane's 8-element operand is one 16-byte LDS read; the row
// pitch of 136 elements puts the 16 rows a read instruction touches on
// disjoint banks), and the global loads of the next chunk are issued before
// the MFMAs of the current one, so a 256-deep product waits on memory about
// once rather than once per K step.
enum Epi { EPI_FWD_SILU = 0, EPI_FWD_LINEAR = 1, EPI_BWD_DSILU = 2, EPI_WGRAD = 3 };

struct GemmArgs {
    int M, N, K;
    const bf16_t *A;
    long long lda_m, lda_k;
    const bf16_t *B;
    long long ldb_k, ldb_n;
    const float *bias;  // [N]                      (forward)
    const float *Zin;   // [M][ldz] pre-activation  (EPI_BWD_DSILU)
    float *Zout;        // [M][ldz] pre-activation  (forward; optional with SiLU)
    bf16_t *Yout;       // [M][ldy]                 (forward SiLU, dsilu)
    float *Cout;        // [M][ldc]                 (EPI_WGRAD)
    bf16_t *YTout;      // [N][ldt] transposed copy of Yout (optional)
    int ldz, ldy, ldc, ldt;
    int ksplit;         // K range of split z (blockIdx.z): [z * ksplit, (z + 1) * ksplit); 0 = all of K
    long long cstride;  // Cout offset between splits (EPI_WGRAD)
};

constexpr int TK = 32, KPAD = 8;

// Workgroup tiles: 64 x 64 (each of the 4 waves 32 x 32 = 2 x 2 MFMA blocks,
// K staged 128 deep) for the training products of a few thousand rows, where
// the number of workgroups matters; 128 x 128 (each wave 64 x 64 = 4 x 4
// blocks, K staged 64 deep) for the screening products, where every 16-byte
// LDS operand read then feeds four MFMAs instead of two.  The row pitch of
// KC + 8 elements keeps the 16 rows an operand read touches on disjoint banks.
template <int T>
struct Tile;
template <>
struct Tile<32> {
    static constexpr int TM = 32, TN = 32, KC = 128, WB = 1;
};
template <>
struct Tile<64> {
    static constexpr int TM = 64, TN = 64, KC = 128, WB = 2;
};
template <>
struct Tile<128> {
    static constexpr int TM = 128, TN = 128, KC = 64, WB = 4;
};

// rows [r0, r0 + TM) x k [k, k + KC) of a strided BF16 operand into registers
// (zero outside [0, rows) x [k, kend)); slot j of thread t is row
// (t + 256 j) / KG, group (t + 256 j) % KG, so consecutive threads read one
// contiguous row segment
template <int TM, int KC>
__device__ inline void gemm_load(const bf16_t *X, long long ld_r, long long ld_k, bool vec, int rows, int r0,
                                 int k, int kend, u16x8 (&v)[TM * (KC / 8) / 256])
{
    constexpr int KG = KC / 8;
#pragma unroll
    for (int j = 0; j < TM * KG / 256; ++j) {
        const int slot = (int)threadIdx.x + 256 * j;
        const int r = r0 + slot / KG, kk = k + (slot % KG) * 8;
        if (vec && r < rows && kk + 8 <= kend) {
            v[j] = *(const u16x8 *)(X + (long long)r * ld_r + kk);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[j][e] = (r < rows && kk + e < kend) ? X[(long long)r * ld_r + (long long)(kk + e) * ld_k] : 0;
        }
    }
}

template <int TM, int KC>
__device__ inline void gemm_stage(bf16_t *S, const u16x8 (&v)[TM * (KC / 8) / 256])
{
    constexpr int KG = KC / 8, KCP = KC + KPAD;
#pragma unroll
    for (int j = 0; j < TM * KG / 256; ++j) {
        const int slot = (int)threadIdx.x + 256 * j;
        *(u16x8 *)&S[(slot / KG) * KCP + (slot % KG) * 8] = v[j];
    }
}

// workgroup-tile product of one block (bx, by, bz) of the grid
// (ceil(N / TN), ceil(M / TM), splits); smem holds (TM + TN) x (KC + KPAD)
// BF16 elements
template <int EPI, int T>
__device__ __attribute__((always_inline)) inline void gemm_block(const GemmArgs &g, int bx, int by, int bz,
                                                                 bf16_t *smem)
{
    constexpr int TM = Tile<T>::TM, TN = Tile<T>::TN, KC = Tile<T>::KC, WB = Tile<T>::WB;
    constexpr int KCP = KC + KPAD, LDT = TM * (KC / 8) / 256;
    bf16_t *As = smem, *Bs = smem + TM * KCP;
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = by * TM, n0 = bx * TN;
    const int kbeg = g.ksplit > 0 ? bz * g.ksplit : 0;
    const int kend = g.ksplit > 0 ? min(g.K, kbeg + g.ksplit) : g.K;
    f32x4 acc[WB][WB];
#pragma unroll
    for (int i = 0; i < WB; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j)
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const bool a_vec = g.lda_k == 1 && (g.lda_m % 8) == 0 && ((uintptr_t)g.A & 15) == 0;
    const bool b_vec = g.ldb_k == 1 && (g.ldb_n % 8) == 0 && ((uintptr_t)g.B & 15) == 0;
    u16x8 va[LDT], vb[LDT];
    if (kbeg < kend) {
        gemm_load<TM, KC>(g.A, g.lda_m, g.lda_k, a_vec, g.M, m0, kbeg, kend, va);
        gemm_load<TN, KC>(g.B, g.ldb_n, g.ldb_k, b_vec, g.N, n0, kbeg, kend, vb);
    }
    for (int kc = kbeg; kc < kend; kc += KC) {
        gemm_stage<TM, KC>(As, va);
        gemm_stage<TN, KC>(Bs, vb);
        __syncthreads();
        if (kc + KC < kend) {  // next chunk in flight during this chunk's MFMAs
            gemm_load<TM, KC>(g.A, g.lda_m, g.lda_k, a_vec, g.M, m0, kc + KC, kend, va);
            gemm_load<TN, KC>(g.B, g.ldb_n, g.ldb_k, b_vec, g.N, n0, kc + KC, kend, vb);
        }
        const int nks = (min(KC, kend - kc) + TK - 1) / TK;
        const int r = lane & 15;
        for (int ks = 0; ks < nks; ++ks) {
            const int kk = ks * TK + (lane >> 4) * 8;
            bf16x8 bfr[WB];
#pragma unroll
            for (int j = 0; j < WB; ++j)
                bfr[j] = *(const bf16x8 *)&Bs[(wn * (TN / 2) + j * 16 + r) * KCP + kk];
#pragma unroll
            for (int i = 0; i < WB; ++i) {
                const bf16x8 a = *(const bf16x8 *)&As[(wm * (TM / 2) + i * 16 + r) * KCP + kk];
#pragma unroll
                for (int j = 0; j < WB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bfr[j], acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();  // before the next chunk overwrites the tiles
    }
    // epilogue: lane holds rows (lane >> 4) * 4 + q, column lane & 15 of each
    // block.  The transposed copy (YTout) is first gathered in LDS (the
    // tiles are free once the K loop's last barrier has passed) and then
    // written a row of YT at a time with 16-byte stores, instead of one
    // scattered 2-byte store per element.
    constexpr int TP = TM + 8;  // pitch of the transposed tile
    static_assert(TN * TP <= (TM + TN) * KCP, "the transposed tile fits in the staging LDS");
    bf16_t *Tt = smem;
    const bool stage_t = (EPI == EPI_FWD_SILU || EPI == EPI_BWD_DSILU) && g.YTout != nullptr;
#pragma unroll
    for (int i = 0; i < WB; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int ml = wm * (TM / 2) + i * 16 + (lane >> 4) * 4 + q;
                const int nl = wn * (TN / 2) + j * 16 + (lane & 15);
                const int m = m0 + ml;
                const int n = n0 + nl;
                if (m >= g.M || n >= g.N)
                    continue;
                float v = acc[i][j][q];
                if (EPI == EPI_FWD_SILU || EPI == EPI_FWD_LINEAR) {
                    v += g.bias[n];
                    if (EPI == EPI_FWD_LINEAR || g.Zout)
                        g.Zout[(long long)m * g.ldz + n] = v;
                    if (EPI == EPI_FWD_SILU) {
                        const bf16_t y = f2bf_dev(silu(v));
                        g.Yout[(long long)m * g.ldy + n] = y;
                        if (stage_t)
                            Tt[nl * TP + ml] = y;
                    }
                } else if (EPI == EPI_BWD_DSILU) {
                    const bf16_t y = f2bf_dev(v * dsilu(g.Zin[(long long)m * g.ldz + n]));
                    g.Yout[(long long)m * g.ldy + n] = y;
                    if (stage_t)
                        Tt[nl * TP + ml] = y;
                } else {
                    g.Cout[(long long)bz * g.cstride + (long long)m * g.ldc + n] = v;
                }
            }
    if (stage_t) {  // uniform across the workgroup
        __syncthreads();
        const bool vec = (g.ldt % 8) == 0 && ((uintptr_t)g.YTout & 15) == 0;
#pragma unroll
        for (int slot = (int)threadIdx.x; slot < TN * TM / 8; slot += 256) {
            const int nl = slot / (TM / 8), ml = (slot % (TM / 8)) * 8;
            const int n = n0 + nl, m = m0 + ml;
            if (n >= g.N)
                continue;
            bf16_t *dst = g.YTout + (long long)n * g.ldt + m;
            if (vec && m + 8 <= g.M) {
                *(u16x8 *)dst = *(const u16x8 *)&Tt[nl * TP + ml];
            } else {
                for (int e = 0; e < 8 && m + e < g.M; ++e)
                    dst[e] = Tt[nl * TP + ml + e];
            }
        }
    }
}

template <int EPI, int T>
__global__ void __launch_bounds__(256) mlp_gemm(const GemmArgs g)
{
    __shared__ __attribute__((aligned(16))) bf16_t smem[(Tile<T>::TM + Tile<T>::TN) * (Tile<T>::KC + KPAD)];
    gemm_block<EPI, T>(g, (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, smem);
}

// ---------------------------------------------------------------- encode
// Fourier feature f of the input (x0, x1): sin and cos of
// 2 pi (B[0][f] x0 + B[1][f] x1), rounded to BF16
__device__ __attribute__((always_inline)) inline void encode_pair(float x0, float x1, int f, const float *Bff, bf16_t &s, bf16_t &c)
{
    const float p = 6.283185307179586f * (Bff[f] * x0 + Bff[NFF + f] * x1);
    float sp, cp;
    sincosf(p, &sp, &cp);  // one argument reduction for both
    s = f2bf_dev(sp);
    c = f2bf_dev(cp);
}

// row i of the encoded inputs; A0t (optional): transposed copy [32][ldt]
__device__ inline void encode_row(float x0, float x1, int i, const float *Bff, bf16_t *A0, bf16_t *A0t, int ldt)
{
    for (int f = 0; f < NFF; ++f) {
        bf16_t s, c;
        encode_pair(x0, x1, f, Bff, s, c);
        A0[(long long)i * D0 + 2 * f] = s;
        A0[(long long)i * D0 + 2 * f + 1] = c;
        if (A0t) {
            A0t[(long long)(2 * f) * ldt + i] = s;
            A0t[(long long)(2 * f + 1) * ldt + i] = c;
        }
    }
}

__global__ void __launch_bounds__(256) mlp_encode(const float *X, int n, const float *Bff, bf16_t *A0, bf16_t *A0t,
                                                  int ldt)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    encode_row(X[2 * i], X[2 * i + 1], i, Bff, A0, A0t, ldt);
}

// grid inputs (c < nx * ny <= 2^26): cell c = ix * ny + iy at (lo + (hi - lo) * i / (n - 1)), normalised to [0, 1]
__device__ __attribute__((always_inline)) inline void grid_point(long long c, int nx, int ny, float &x0, float &x1)
{
    const unsigned int k = (unsigned int)c, n = (unsigned int)ny;
    const int ix = (int)(k / n), iy = (int)(k - k / n * n);
    x0 = nx > 1 ? (float)ix / (float)(nx - 1) : 0.f;
    x1 = ny > 1 ? (float)iy / (float)(ny - 1) : 0.f;
}

__global__ void __launch_bounds__(256) mlp_grid_inputs(long long c0, int n, int nx, int ny, float *X)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    grid_point(c0 + i, nx, ny, X[2 * i], X[2 * i + 1]);
}

// ---------------------------------------------------------------- loss
__host__ __device__ inline bool head_keeps(unsigned long long sample, int head)
{
    unsigned long long z = sample * 4ull + (unsigned long long)head + 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z ^= z >> 31;
    return (z & 3ull) != 0ull;
}

// Per sample and head: squared error of the two normalised regression
// targets plus the softmax cross-entropy of the class, over the samples the
// head keeps; the loss is the mean over the batch of the sum over heads.
// dOut (BF16, [n][128]) is the gradient of that loss w.r.t. the head outputs,
// dOutT ([128][ldt]) its transpose.  One thread per (sample, head), sample
// fastest, so the transposed rows are written coalesced; the columns past the
// heads stay zero in dOut (cleared when the buffer is allocated) and are
// cleared here in dOutT, whose row pitch follows the batch size.
constexpr int PADROWS = (NOUTP - NOUT) / NHEAD;  // transposed padding rows each head thread clears
static_assert(PADROWS * NHEAD == NOUTP - NOUT, "padding rows split evenly over the heads");

// one (row, head): its loss into l, the gradient of its 18 outputs into d
__device__ __attribute__((always_inline)) inline void loss_row(const float *zh, bool kept, float t0, float t1, int y,
                                                               float inv_n, bf16_t (&d)[HW], float &l)
{
    if (!kept) {
#pragma unroll
        for (int c = 0; c < HW; ++c)
            d[c] = 0;
        return;
    }
    const float e0 = zh[0] - t0, e1 = zh[1] - t1;
    l += e0 * e0 + e1 * e1;
    d[0] = f2bf(2.f * e0 * inv_n);
    d[1] = f2bf(2.f * e1 * inv_n);
    float mx = zh[2];
#pragma unroll
    for (int c = 1; c < NCLS; ++c)
        mx = fmaxf(mx, zh[2 + c]);
    // each class's exponential once, for the sum and the gradient
    float ex[NCLS];
    float se = 0.f, zy = zh[2];
#pragma unroll
    for (int c = 0; c < NCLS; ++c) {
        ex[c] = __expf(zh[2 + c] - mx);
        se += ex[c];
        zy = c == y ? zh[2 + c] : zy;
    }
    l += (mx + __logf(se)) - zy;
#pragma unroll
    for (int c = 0; c < NCLS; ++c) {
        const float p = ex[c] / se;
        d[2 + c] = f2bf((p - (c == y ? 1.f : 0.f)) * inv_n);
    }
}

__global__ void __launch_bounds__(256) mlp_loss(const float *Zh, int n, const float *T, const int *cls,
                                                const unsigned long long *ids, float inv_n, bf16_t *dOut,
                                                bf16_t *dOutT, int ldt, float *loss)
{
    __shared__ float red[256];
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.f;
    if (t < (long long)NHEAD * n) {
        const int h = (int)(t / n), i = (int)(t % n);
        bf16_t d[HW];
        const unsigned long long id = ids ? ids[i] : (unsigned long long)i;
        loss_row(Zh + (long long)i * NOUTP + h * HW, head_keeps(id, h), T[2 * i], T[2 * i + 1], cls[i], inv_n, d, l);
        bf16_t *dh = dOut + (long long)i * NOUTP + h * HW;
        for (int c = 0; c < HW; ++c) {
            dh[c] = d[c];
            dOutT[(long long)(h * HW + c) * ldt + i] = d[c];
        }
        for (int c = NOUT + h * PADROWS; c < NOUT + (h + 1) * PADROWS; ++c)
            dOutT[(long long)c * ldt + i] = 0;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        atomicAdd(loss, red[0] * inv_n);
}

// one launch for both per-layer reductions of the backward pass: blocks
// [0, sum_blocks) sum the split-K partial weight gradients in a fixed order
// (gw[e] = sum_z part[z * count + e]); the remaining ncol blocks form the bias
// gradient db[c] = sum_m dZ[m][c] from the transposed copy dZt[c][m] (row
// stride ld), each block reading one contiguous row
__global__ void __launch_bounds__(256) mlp_layer_grads(const float *part, int splits, long long count, float *gw,
                                                       int sum_blocks, const bf16_t *dZt, int n, int ncol, int ld,
                                                       float *db)
{
    __shared__ float red[256];
    if ((int)blockIdx.x < sum_blocks) {
        const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
        if (e >= count)
            return;
        float s = 0.f;
        for (int z = 0; z < splits; ++z)
            s += part[(long long)z * count + e];
        gw[e] = s;
        return;
    }
    const int c = (int)blockIdx.x - sum_blocks;
    float s = 0.f;
    for (int m = threadIdx.x; m < n; m += blockDim.x)
        s += bf2f(dZt[(long long)c * ld + m]);
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k)
            red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0 && c < ncol)
        db[c] = red[0];
}

// layer table for the Adam kernels: weights of layer l occupy
// [woff, woff + in * out) as Wt[out][in], its biases the out entries after
// them
struct LayerTable {
    long long woff[NLAYER];
    int in[NLAYER], out[NLAYER];
};

// The BF16 copies of the weights that the products read, all at the layer's
// weight offset: Wt[out][in], W[in][out], and both again in fragment order.
struct WeightCopies {
    bf16_t *w, *wT, *f, *fT;
};

// Fragment order of a product's B operand, rows n of K entries: the 16 x 32
// block of rows 16 nb .. and entries 32 kb .. is 512 consecutive values, the 8
// of lane (k / 8 % 4) * 16 + n % 16 together, so that a wave's load of one
// fragment is 1 KB in a row.  From Wt[out][in] the same load touches 16 rows, a
// different one in every consecutive lane.
__device__ inline int frag_at(int n, int k, int K)
{
    return ((n >> 4) * (K >> 5) + (k >> 5)) * 512 + (((k >> 3) & 3) * 16 + (n & 15)) * 8 + (k & 7);
}

// parameter i in the copies (a bias only at its place in the first)
__device__ __forceinline__ void put_weight(const WeightCopies &c, const LayerTable &lt, long long i, float v)
{
    const bf16_t b16 = f2bf(v);
    c.w[i] = b16;
    int l = 0;
    while (l < NLAYER - 1 && i >= lt.woff[l + 1])
        ++l;
    const int r = (int)(i - lt.woff[l]), in = lt.in[l], out = lt.out[l];
    if (r >= in * out)
        return;
    const int o = r / in, k = r % in;
    c.wT[lt.woff[l] + k * out + o] = b16;
    c.f[lt.woff[l] + frag_at(o, k, in)] = b16;
    c.fT[lt.woff[l] + frag_at(k, o, out)] = b16;
}

__global__ void __launch_bounds__(256) mlp_put_weights(const float *p, const WeightCopies c, const LayerTable lt,
                                                       long long n)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        put_weight(c, lt, i, p[i]);
}

struct AdamStep {
    float lr, b1, b2, eps, c1, c2;
};

// Adam (Kingma & Ba 2015) on one FP32 master parameter, refreshing the BF16
// copies of the weights
__device__ __forceinline__ void adam_update(long long i, float gi, float *p, float *m1, float *m2,
                                            const WeightCopies &wc, const LayerTable &lt, const AdamStep &as)
{
    const float a = as.b1 * m1[i] + (1.f - as.b1) * gi;
    const float b = as.b2 * m2[i] + (1.f - as.b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    const float v = p[i] - as.lr * (a * as.c1) / (sqrtf(b * as.c2) + as.eps);
    p[i] = v;
    put_weight(wc, lt, i, v);
}

// Adam from a finished gradient vector g; frozen entries (mask 0: head
// padding) stay put
__global__ void __launch_bounds__(256) mlp_adam(float *p, const float *g, float *m1, float *m2, const uint8_t *mask,
                                                const WeightCopies wc, const LayerTable lt, long long n,
                                                const AdamStep as)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !mask[i])
        return;
    adam_update(i, g[i], p, m1, m2, wc, lt, as);
}

// Adam that also finishes the gradient, in place of the per-layer reduction
// launches of the backward pass (the training loop's optimizer step).
// Blocks [0, wblocks): one thread per parameter; a weight's gradient is the
// sum of its split-K partial products part[z * pstride + i], z = 0 .. splits-1
// in order (the sum mlp_layer_grads forms).  The following blocks take one
// bias each, layer by layer: db[c] = sum_m dZt_l[c][m] over the minibatch by
// the same strided sums and tree as mlp_layer_grads, then thread 0 updates it.
// The updated parameters equal those of the separate launches bit for bit.
struct GradSources {
    const float *part;
    long long pstride;
    int splits;
    const bf16_t *dzt[NLAYER];  // transposed output gradient of each layer, [out][ld]
    int n, ld;
};

__global__ void __launch_bounds__(256) mlp_adam_sum(float *p, float *m1, float *m2, const uint8_t *mask,
                                                    const WeightCopies wc, const LayerTable lt, long long n, int wblocks,
                                                    const GradSources gs, const AdamStep as)
{
    if ((int)blockIdx.x < wblocks) {
        const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
        if (i >= n || !mask[i])
            return;
        int l = 0;
        while (l < NLAYER - 1 && i >= lt.woff[l + 1])
            ++l;
        if (i - lt.woff[l] >= (long long)lt.in[l] * lt.out[l])
            return;  // a bias: the blocks below
        float s = 0.f;
        for (int z = 0; z < gs.splits; ++z)
            s += gs.part[(long long)z * gs.pstride + i];
        adam_update(i, s, p, m1, m2, wc, lt, as);
        return;
    }
    __shared__ float red[256];
    int c = (int)blockIdx.x - wblocks, l = 0;
    while (l < NLAYER - 1 && c >= lt.out[l]) {
        c -= lt.out[l];
        ++l;
    }
    const long long i = lt.woff[l] + (long long)lt.in[l] * lt.out[l] + c;
    if (!mask[i])
        return;  // head padding: its gradient rows are not formed
    const bf16_t *dzt = gs.dzt[l];
    float s = 0.f;
    for (int m = threadIdx.x; m < gs.n; m += blockDim.x)
        s += bf2f(dzt[(long long)c * gs.ld + m]);
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k)
            red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        adam_update(i, red[0], p, m1, m2, wc, lt, as);
}

// minibatch gather: row r of the batch is sample perm[r] of the training
// set; its inputs are encoded (with the transposed copy) in the same pass.
// One thread per (row, frequency), row fastest, so that a minibatch of a
// few thousand rows spreads its sin/cos over 16x more lanes and the
// transposed rows are written coalesced.
__global__ void __launch_bounds__(256) mlp_gather(const unsigned int *perm, int nb, const float *Xa, const float *Ta,
                                                  const int *Ca, float *T, int *C, unsigned long long *ids,
                                                  const float *Bff, bf16_t *A0, bf16_t *A0t, int ldt)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nb * NFF)
        return;
    const int r = idx % nb, f = idx / nb;
    const unsigned int j = perm[r];
    if (f == 0) {
        T[2 * r] = Ta[2 * j];
        T[2 * r + 1] = Ta[2 * j + 1];
        C[r] = Ca[j];
        ids[r] = j;
    }
    bf16_t sv, cv;
    encode_pair(Xa[2 * j], Xa[2 * j + 1], f, Bff, sv, cv);
    A0[(long long)r * D0 + 2 * f] = sv;
    A0[(long long)r * D0 + 2 * f + 1] = cv;
    A0t[(long long)(2 * f) * ldt + r] = sv;
    A0t[(long long)(2 * f + 1) * ldt + r] = cv;
}

// ---------------------------------------------------------------- screening
// Per cell: each head's (log-period, amplitude) back to feature units and
// class argmax; the ensemble prediction is the head mean (softmax mean for the
// class).  flags bit 0: the heads disagree (relative spread above tol, or a
// head's class differs from the ensemble class).
// z: the 72 head outputs of one cell
__device__ __attribute__((always_inline)) inline void predict_row(const float *z, const float *tmean,
                                                                  const float *tstd, float tol, float &period,
                                                                  float &amp, int &cls, uint8_t &flags)
{
    // every loop has a constant trip count and is unrolled, so the arrays
    // live in registers (the first-occurrence argmax keeps its best value
    // instead of indexing prob[] at a run-time index)
    float P[NHEAD], A[NHEAD], prob[NCLS];
    int hc[NHEAD];
#pragma unroll
    for (int c = 0; c < NCLS; ++c)
        prob[c] = 0.f;
    float pm = 0.f, am = 0.f;
#pragma unroll
    for (int h = 0; h < NHEAD; ++h) {
        const float *zh = z + h * HW;
        P[h] = expf(zh[0] * tstd[0] + tmean[0]);
        A[h] = zh[1] * tstd[1] + tmean[1];
        pm += P[h];
        am += A[h];
        float mx = zh[2];
        int am_i = 0;
#pragma unroll
        for (int c = 1; c < NCLS; ++c)
            if (zh[2 + c] > mx) {
                mx = zh[2 + c];
                am_i = c;
            }
        hc[h] = am_i;
        float se = 0.f;
#pragma unroll
        for (int c = 0; c < NCLS; ++c)
            se += __expf(zh[2 + c] - mx);
#pragma unroll
        for (int c = 0; c < NCLS; ++c)
            prob[c] += __expf(zh[2 + c] - mx) / se;
    }
    pm *= 1.f / NHEAD;
    am *= 1.f / NHEAD;
    int best = 0;
    float pbest = prob[0];
#pragma unroll
    for (int c = 1; c < NCLS; ++c)
        if (prob[c] > pbest) {
            pbest = prob[c];
            best = c;
        }
    bool dis = false;
#pragma unroll
    for (int h = 0; h < NHEAD; ++h) {
        dis |= fabsf(P[h] - pm) > tol * fabsf(pm);
        dis |= fabsf(A[h] - am) > tol * fabsf(am);
        dis |= hc[h] != best;
    }
    period = pm;
    amp = am;
    cls = best;
    flags = dis ? 1 : 0;
}

__global__ void __launch_bounds__(256) mlp_predict_cells(const float *Zh, int n, const float *tmean,
                                                         const float *tstd, float tol, float *period, float *amp,
                                                         int *cls, uint8_t *flags)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    predict_row(Zh + (long long)i * NOUTP, tmean, tstd, tol, period[i], amp[i], cls[i], flags[i]);
}

// flags bit 1: a 4-neighbour on the nx x ny grid has another class
__global__ void __launch_bounds__(256) mlp_boundary(const int *cls, int nx, int ny, uint8_t *flags)
{
    const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= (long long)nx * ny)
        return;
    const int ix = (int)(c / ny), iy = (int)(c % ny);
    const int k = cls[c];
    bool b = (ix > 0 && cls[c - ny] != k) || (ix + 1 < nx && cls[c + ny] != k) || (iy > 0 && cls[c - 1] != k) ||
             (iy + 1 < ny && cls[c + 1] != k);
    if (b)
        flags[c] |= 2;
}

// one step of 3 x 3 dilation of "any flag" into bit 2 (out must not alias in)
__global__ void __launch_bounds__(256) mlp_dilate(const uint8_t *in, int nx, int ny, uint8_t *out)
{
    const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= (long long)nx * ny)
        return;
    const int ix = (int)(c / ny), iy = (int)(c % ny);
    uint8_t f = in[c];
    bool any = false;
    for (int dx = -1; dx <= 1; ++dx)
        for (int dy = -1; dy <= 1; ++dy) {
            const int jx = ix + dx, jy = iy + dy;
            if (jx >= 0 && jx < nx && jy >= 0 && jy < ny && in[(long long)jx * ny + jy])
                any = true;
        }
    out[c] = (uint8_t)(f | (any && !f ? 4 : 0));
}

// ---------------------------------------------------------------- host
thread_local std::string g_err;

// ---------------------------------------------------------------- fused screening
// One workgroup per block of SROWS grid cells runs the whole network:
// encode, the four hidden layers, the heads and the per-cell prediction.
// The activations stay in LDS between layers; only the weights (0.4 MB,
// L2-resident) and the four per-cell results touch memory, where the
// layer-by-layer path writes and re-reads 0.5 KB of activations per cell and
// layer.  Each wave owns 64 output columns of a hidden layer (8 x 4 blocks of
// 16 x 16) or 32 rows of the heads (2 x 5 blocks), takes its weight fragments
// straight from global memory with the next K step's in flight, and reads the
// activations from LDS.  K order (32-deep steps, ascending) and epilogue
// arithmetic are those of mlp_gemm, so every output equals the layer-by-layer
// path bit for bit.
// What bounds it is the vector ALU's issue: busy 70 % of the time at 2.5 ms, the
// matrix cores 36 %, and every instruction taken out shows (SiLU of 1024 values
// per cell is 60 % of them).  2048 x 2048 cells: 3.45 ms with weights read row
// by row and scalar LDS stores; 3.25 with weights in fragment order, 2.80 with
// the weights as first operand (one 8-byte LDS store for four values), 2.5 with
// biases in LDS and the next layer's weights on their way during the epilogue,
// 2.30 with the prediction spread over the four waves.  Two groups of four
// waves kept half a layer apart by shared barriers, so that one's products
// overlap the other's epilogues, took 2.78: two workgroups that drift do better.
//
// LDS: the activations [SROWS][H] BF16, 64 KiB, two workgroups per CU.  The
// 16-byte chunk kc of row m is stored at chunk kc ^ (m & 15) of that row, so
// the 16 rows an operand read touches fall on 16 different chunk positions
// (no padding, which would not fit two workgroups).  After the last hidden
// layer the same bytes hold the FP32 head outputs [SROWS][ZPITCH].
constexpr int SROWS = 128;         // cells per workgroup
constexpr int ZPITCH = NOUT + 1;   // row pitch of the head outputs (floats)
static_assert(SROWS * ZPITCH * 4 <= SROWS * H * 2, "head outputs fit in the activation buffer");
constexpr int HBLK = (NOUT + 15) / 16;  // column blocks of the heads that hold used columns
static_assert(SROWS == 8 * 16 && SROWS == 4 * 32 && H == 4 * 64 && NOUT % 4 == 0 && HBLK * 16 <= NOUTP, "wave tiling");

struct ScreenArgs {
    long long ncell;
    int nx, ny;
    const float *Bff;
    const bf16_t *W[NLAYER];  // Wt[out][in] in fragment order
    const float *bias[NLAYER];
    const float *tm;  // tmean[2], tstd[2]
    float tol;
    float *period, *amp;
    int *cls;
    uint8_t *flags;
};

// The lane index, recomputed where it is used: an opaque value keeps the
// compiler from computing every layer's epilogue LDS addresses once at the
// top of the kernel, where they would stay live across all the K loops and
// spill (two v_mbcnt instructions per epilogue instead).
__device__ __attribute__((always_inline)) inline int lane_here()
{
    int v;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(v));
    return v;
}

// element (m, k) of the swizzled activation tile
__device__ __attribute__((always_inline)) inline int sw(int m, int k) { return m * H + ((((k >> 3) ^ (m & 15))) << 3) + (k & 7); }

// Weight fragments in flight: K step ks of a product is in b[ks % PF], loaded
// PF - 1 steps ahead, the first ones during the layer before.
constexpr int PF = 2;

template <int K, int NB>
__device__ __attribute__((always_inline)) inline void screen_load(const bf16_t *__restrict__ W, int n0, int ks, int lane,
                                                                  bf16x8 (&b)[PF][NB])
{
    if (ks < K / TK) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
            b[ks % PF][j] = *(const bf16x8 *)(W + ((n0 / 16 + j) * (K / TK) + ks) * 512 + lane * 8);
    }
}

template <int K, int NB>
__device__ __attribute__((always_inline)) inline void screen_first(const bf16_t *__restrict__ W, int n0, int lane,
                                                                   bf16x8 (&b)[PF][NB])
{
#pragma unroll
    for (int ks = 0; ks < PF - 1; ++ks)
        screen_load<K, NB>(W, n0, ks, lane, b);
}

// acc[i][j] = W[columns of block j][0, K) * act[rows of block i][0, K)^T for
// the NB column blocks starting at column n0 and the RB row blocks starting at
// row m0.  The weights are the first MFMA operand, so a lane holds four
// consecutive columns (lane >> 4) * 4 .. + 3 of one row lane & 15: four
// neighbouring elements of the activation tile (the sums are those of the
// other operand order, element by element).
template <int K, int RB, int NB>
__device__ __attribute__((always_inline)) inline void screen_product(const bf16_t *act, const bf16_t *__restrict__ W, int m0, int n0,
                                      int lane, bf16x8 (&b)[PF][NB], f32x4 (&acc)[RB][NB])
{
    constexpr int NKS = K / TK;
    const int r = lane & 15, kq = (lane >> 4) * 8;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int HR = RB / 2;
    bf16x8 a[2][HR];
#pragma unroll
    for (int i = 0; i < HR; ++i)
        a[0][i] = *(const bf16x8 *)&act[sw(m0 + i * 16 + r, kq)];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        screen_load<K, NB>(W, n0, ks + PF - 1, lane, b);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (h == 0 || ks + 1 < NKS) {
#pragma unroll
                for (int i = 0; i < HR; ++i)
                    a[1 - h][i] = *(const bf16x8 *)&act[sw(m0 + ((1 - h) * HR + i) * 16 + r, (ks + h) * TK + kq)];
            }
#pragma unroll
            for (int i = 0; i < HR; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    acc[h * HR + i][j] =
                        __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[ks % PF][j], a[h][i], acc[h * HR + i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);  // keep the loads where they are
        }
    }
}

// hidden layer's epilogue in place: act <- SiLU(acc + bias), BF16, four elements
// to a conversion pair and one 8-byte LDS store
__device__ __attribute__((always_inline)) inline void screen_hidden(bf16_t *act, const f32x4 (&acc)[8][4], const float *bias, int wave)
{
    __syncthreads();  // every wave has read the layer's input
    const int lane = lane_here();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = wave * 64 + j * 16 + (lane >> 4) * 4;
        const f32x4 bj = *(const f32x4 *)(bias + n);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const f32x4 v = acc[i][j] + bj;
            const bf16x4 y = {(__bf16)silu(v[0]), (__bf16)silu(v[1]), (__bf16)silu(v[2]), (__bf16)silu(v[3])};
            *(bf16x4 *)&act[sw(i * 16 + (lane & 15), n)] = y;
        }
    }
    __syncthreads();
}

// One head's outputs zh in place: to feature units, and its class scores to
// softmax values; returns its class.  The quotients by the sum take three
// instructions instead of ten: its reciprocal is refined once and every quotient
// corrected by its remainder.  They are those of a division (80 million random
// pairs, with a reciprocal off by one unit either way) but where the quotient is
// so near to underflow that its remainder is not exact; only the sums of a class
// over the heads read them, and the largest class of a head is at least 1/16.
__device__ __attribute__((always_inline)) inline uint8_t predict_head(float *zh, const float *tmean, const float *tstd)
{
    float ex[NCLS];
#pragma unroll
    for (int c = 0; c < NCLS; ++c)
        ex[c] = zh[2 + c];
    float mx = ex[0];
    int best = 0;
#pragma unroll
    for (int c = 1; c < NCLS; ++c) {
        best = ex[c] > mx ? c : best;
        mx = ex[c] > mx ? ex[c] : mx;
    }
    float se = 0.f;
#pragma unroll
    for (int c = 0; c < NCLS; ++c) {
        ex[c] = __expf(ex[c] - mx);
        se += ex[c];
    }
    float r = __builtin_amdgcn_rcpf(se);
    r = fmaf(fmaf(-se, r, 1.f), r, r);
#pragma unroll
    for (int c = 0; c < NCLS; ++c) {
        const float q = ex[c] * r;
        zh[2 + c] = fmaf(fmaf(-q, se, ex[c]), r, q);
    }
    zh[0] = expf(zh[0] * tstd[0] + tmean[0]);
    zh[1] = zh[1] * tstd[1] + tmean[1];
    return (uint8_t)best;
}

// The heads of one row (z, hc: what predict_head left) in two neighbouring
// lanes: the mean period (half 0) or amplitude (half 1), and in both the class
// and whether the heads disagree.  A half takes eight of the classes.
__device__ __attribute__((always_inline)) inline bool predict_pair(const float *z, const uint8_t *hc, int half, float tol,
                                                                   float &mean, int &cls)
{
    float v[NHEAD];
    mean = 0.f;
#pragma unroll
    for (int h = 0; h < NHEAD; ++h) {
        v[h] = z[h * HW + half];
        mean += v[h];
    }
    mean *= 1.f / NHEAD;
    bool dis = false;
#pragma unroll
    for (int h = 0; h < NHEAD; ++h)
        dis |= fabsf(v[h] - mean) > tol * fabsf(mean);
    const int c0 = half * (NCLS / 2);
    float pbest = 0.f;
    int best = c0;
#pragma unroll
    for (int c = 0; c < NCLS / 2; ++c) {
        float p = 0.f;
#pragma unroll
        for (int h = 0; h < NHEAD; ++h)
            p += z[h * HW + 2 + c0 + c];
        if (c == 0) {
            pbest = p;
        } else {
            best = p > pbest ? c0 + c : best;
            pbest = p > pbest ? p : pbest;
        }
    }
    const float po = __shfl_xor(pbest, 1);
    const int bo = __shfl_xor(best, 1);
    cls = half ? (pbest > po ? best : bo) : (po > pbest ? bo : best);
#pragma unroll
    for (int k = 0; k < NHEAD / 2; ++k)
        dis |= hc[half * (NHEAD / 2) + k] != cls;
    return __shfl_xor((int)dis, 1) | (int)dis;
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) mlp_screen_fused(const ScreenArgs s)
{
    __shared__ __attribute__((aligned(16))) bf16_t act[SROWS * H];
    __shared__ __attribute__((aligned(16))) float bias[NHID * H + NOUT];
    __shared__ uint8_t hc[SROWS * NHEAD];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const long long c0 = (long long)blockIdx.x * SROWS;
#pragma unroll
    for (int l = 0; l < NHID; ++l)
        bias[l * H + t] = s.bias[l][t];
    if (t < NOUT)
        bias[NHID * H + t] = s.bias[NHID][t];
    {  // encode: thread t -> cell row t / 2, frequencies (t % 2) * 8 .. + 8
        const int m = t >> 1, f0 = (t & 1) * (NFF / 2);
        const long long c = c0 + m < s.ncell ? c0 + m : s.ncell - 1;
        float x0, x1;
        grid_point(c, s.nx, s.ny, x0, x1);
        for (int f = f0; f < f0 + NFF / 2; ++f) {
            bf16_t sv, cv;
            encode_pair(x0, x1, f, s.Bff, sv, cv);
            act[sw(m, 2 * f)] = sv;
            act[sw(m, 2 * f + 1)] = cv;
        }
    }
    __syncthreads();
    f32x4 acc[8][4];
    bf16x8 bw[PF][4];
    screen_first<D0, 4>(s.W[0], wave * 64, lane, bw);
    screen_product<D0, 8, 4>(act, s.W[0], 0, wave * 64, lane, bw, acc);
    screen_first<H, 4>(s.W[1], wave * 64, lane, bw);
    screen_hidden(act, acc, bias, wave);
#pragma unroll
    for (int l = 1; l < NHID - 1; ++l) {
        screen_product<H, 8, 4>(act, s.W[l], 0, wave * 64, lane, bw, acc);
        screen_first<H, 4>(s.W[l + 1], wave * 64, lane, bw);
        screen_hidden(act, acc, bias + l * H, wave);
    }
    bf16x8 bh[PF][HBLK];
    screen_product<H, 8, 4>(act, s.W[NHID - 1], 0, wave * 64, lane, bw, acc);
    screen_first<H, HBLK>(s.W[NHID], 0, lane, bh);
    screen_hidden(act, acc, bias + (NHID - 1) * H, wave);
    // heads: every wave takes 32 rows and the five column blocks that hold the
    // 72 used columns; they go to LDS in FP32
    f32x4 az[2][HBLK];
    screen_product<H, 2, HBLK>(act, s.W[NHID], wave * 32, 0, lane, bh, az);
    __syncthreads();  // the activations are no longer needed: z overlays them
    float *z = reinterpret_cast<float *>(act);
    const int hl = lane_here();
#pragma unroll
    for (int j = 0; j < HBLK; ++j) {
        const int n = j * 16 + (hl >> 4) * 4;
        if (n < NOUT) {
            const f32x4 bj = *(const f32x4 *)(bias + NHID * H + n);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const f32x4 v = az[i][j] + bj;
                float *zr = z + (wave * 32 + i * 16 + (hl & 15)) * ZPITCH + n;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    zr[q] = v[q];
            }
        }
    }
    __syncthreads();
    // predict_row's steps and results, over all four waves: two heads of a row
    // to a thread, then the row's heads together in a pair of threads
    {
        float *zr = z + (t & 127) * ZPITCH;
#pragma unroll
        for (int k = 0; k < NHEAD / 2; ++k) {
            const int h = (t >> 7) * (NHEAD / 2) + k;
            hc[(t & 127) * NHEAD + h] = predict_head(zr + h * HW, s.tm, s.tm + 2);
        }
    }
    __syncthreads();
    {
        const int m = t >> 1, half = t & 1;
        const long long c = c0 + m;
        int best;
        float mean;
        const bool dis = predict_pair(z + m * ZPITCH, hc + m * NHEAD, half, s.tol, mean, best);
        if (c < s.ncell) {
            if (half) {
                s.amp[c] = mean;
                s.flags[c] = dis ? 1 : 0;
            } else {
                s.period[c] = mean;
                s.cls[c] = best;
            }
        }
    }
}

// ---------------------------------------------------------------- fused training pass
// One launch for everything of an optimizer step that runs row by row: gather
// and encode, the four hidden layers, the heads, the loss, and the input
// gradients back to the first layer.  A workgroup of 8 waves takes 16 rows of
// the minibatch; activations and gradients stay in LDS (two 8 KiB tiles, one
// barrier per layer), SiLU' stays in the registers of the lane that needs it
// again (a lane forms the same elements of a layer forward and backward), and
// each wave's weight fragments of the next product are loaded while the current
// one runs.  Only the transposed operands of the weight-gradient products leave
// the CU.
// What bounds it is the chain of nine products, each waiting for the one
// before: 17 us with 4 workgroups, 21 us with 128 (2048 rows), 23 us with 256;
// past one workgroup per CU the weights' way from L2, 1 MB per workgroup at
// 64 B per cycle, 17 us per 256 workgroups.  An optimizer step's three launches
// take 40 us at 2048 rows and 29 us at 64; the thirteen that this replaces
// (gather, five forward products, loss, five backward ones, optimizer) took
// 79 us and 58 us, each waiting for a few hundred workgroups to start and drain.
// K order and epilogue arithmetic are those of gemm_block, so the weights
// after training are the same bits.
constexpr int FROWS = 16;    // rows per workgroup
constexpr int FWAVES = 8;    // waves per workgroup, 32 columns each
constexpr int FKH = 96;      // head gradient columns that can be nonzero, in whole K steps
static_assert(FWAVES * 32 == H && HBLK <= FWAVES && NOUT <= FKH && FKH % TK == 0, "fused training tiling");

struct FusedStep {
    const unsigned int *perm;  // this minibatch's samples
    int nb, ldt;
    const float *Xa, *Ta;
    const int *Ca;
    const float *Bff;
    const bf16_t *W[NLAYER];   // Wt[out][in] and
    const bf16_t *WT[NLAYER];  // W[in][out], in fragment order
    const float *bias[NLAYER];
    bf16_t *A0t, *Yt[NHID], *dYt[NHID], *dOutT;  // [width][ldt]
    float inv_n;
    float *loss;
};

// weight fragments of NB column blocks from block nb0 for the first K of KW entries
template <int K, int NB, int KW = K>
__device__ __attribute__((always_inline)) inline void fused_load(const bf16_t *__restrict__ W, int nb0, int lane,
                                                                 bf16x8 (&b)[K / TK][NB])
{
#pragma unroll
    for (int ks = 0; ks < K / TK; ++ks)
#pragma unroll
        for (int j = 0; j < NB; ++j)
            b[ks][j] = *(const bf16x8 *)(W + ((nb0 + j) * (KW / TK) + ks) * 512 + lane * 8);
}

template <int K, int NB>
__device__ __attribute__((always_inline)) inline void fused_product(const bf16_t *act, const bf16x8 (&b)[K / TK][NB],
                                                                    int lane, f32x4 (&acc)[NB])
{
#pragma unroll
    for (int j = 0; j < NB; ++j)
        acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < K / TK; ++ks) {
        const bf16x8 a = *(const bf16x8 *)&act[sw(lane & 15, ks * TK + (lane >> 4) * 8)];
#pragma unroll
        for (int j = 0; j < NB; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[ks][j], acc[j], 0, 0, 0);
    }
}

// four rows ml .. ml + 3 of column n: into the activation tile, and at dst in
// the transposed copy, whose rows past the minibatch are padding
__device__ __attribute__((always_inline)) inline void fused_put(bf16_t *act, int ml, int n, const bf16x4 &y, bf16_t *dst)
{
    union {
        bf16x4 v;
        bf16_t e[4];
    } u = {y};
#pragma unroll
    for (int q = 0; q < 4; ++q)
        act[sw(ml + q, n)] = u.e[q];
    *(bf16x4 *)dst = y;
}

__global__ void __launch_bounds__(FWAVES * 64) mlp_fused_step(const FusedStep s)
{
    __shared__ __attribute__((aligned(16))) bf16_t act[2][FROWS * H];
    __shared__ float zh[FROWS * ZPITCH];
    __shared__ float bias[NHID * H + NOUT];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    // 8 consecutive workgroups are on 8 XCDs: each XCD takes consecutive rows,
    // which share the lines of the transposed copies
    const int per = (int)(gridDim.x >> 3);
    const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    const int r0 = tile * FROWS;                       // the workgroup's rows of the minibatch
    if (r0 >= s.nb)
        return;
    const int ml = (lane >> 4) * 4, m = r0 + ml;       // the lane's four output rows
    const int n0 = wave * 32, c0 = n0 + (lane & 15);   // the wave's columns, the lane's first
    // everything that is read from memory apart from weights comes first: a
    // later load would wait for the prefetched weights and the stores before it
    const int rr = t & 15, row = r0 + rr;
    const unsigned int id = s.perm[row < s.nb ? row : s.nb - 1];
    const float x0 = s.Xa[2 * (size_t)id], x1 = s.Xa[2 * (size_t)id + 1];
    const float t0 = s.Ta[2 * (size_t)id], t1 = s.Ta[2 * (size_t)id + 1];
    const int cls = s.Ca[id];
#pragma unroll
    for (int l = 0; l < NHID; l += 2) {
        const int l1 = l + (t >> 8), n = t & 255;
        bias[l1 * H + n] = s.bias[l1][n];
    }
    if (t < NOUT)
        bias[NHID * H + t] = s.bias[NHID][t];
    bf16x8 b0[1][2], ba[H / TK][2], bb[H / TK][2];
    fused_load<D0, 2>(s.W[0], n0 / 16, lane, b0);
    fused_load<H, 2>(s.W[1], n0 / 16, lane, ba);
    if (t < FROWS * NFF) {
        const int f = t >> 4;
        bf16_t sv, cv;
        encode_pair(x0, x1, f, s.Bff, sv, cv);
        act[0][sw(rr, 2 * f)] = sv;
        act[0][sw(rr, 2 * f + 1)] = cv;
        s.A0t[(long long)(2 * f) * s.ldt + row] = sv;
        s.A0t[(long long)(2 * f + 1) * s.ldt + row] = cv;
    }
    __syncthreads();
    f32x4 D[NHID][2];  // SiLU'(z), for the way back
    auto hidden = [&](int l, f32x4 (&acc)[2], bf16_t *out) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = c0 + j * 16;
            const float bj = bias[l * H + n];
            bf16x4 y;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v = acc[j][q];
                v += bj;
                const float sg = sigm(v);
                D[l][j][q] = sg * (1.0f + v * (1.0f - sg));
                y[q] = (__bf16)(v * sg);
            }
            fused_put(out, ml, n, y, s.Yt[l] + (long long)n * s.ldt + m);
        }
        __syncthreads();
    };
    f32x4 acc[2];
    fused_product<D0, 2>(act[0], b0, lane, acc);
    hidden(0, acc, act[1]);
    fused_load<H, 2>(s.W[2], n0 / 16, lane, bb);
    fused_product<H, 2>(act[1], ba, lane, acc);
    hidden(1, acc, act[0]);
    fused_load<H, 2>(s.W[3], n0 / 16, lane, ba);
    fused_product<H, 2>(act[0], bb, lane, acc);
    hidden(2, acc, act[1]);
    // heads: one 16-column block on each of the first waves
    bf16x8 bh[H / TK][1];
    const int hb = wave < HBLK ? wave : 0;
    fused_load<H, 1>(s.W[NHID], hb, lane, bh);
    fused_product<H, 2>(act[1], ba, lane, acc);
    hidden(3, acc, act[0]);
    bf16x8 bg[FKH / TK][2];
    fused_load<FKH, 2, NOUTP>(s.WT[NHID], n0 / 16, lane, bg);
    fused_load<H, 2>(s.WT[3], n0 / 16, lane, bb);
    {
        f32x4 az[1];
        fused_product<H, 1>(act[0], bh, lane, az);
        const int n = hb * 16 + (lane & 15);
        if (wave < HBLK && n < NOUT) {
            const float bj = bias[NHID * H + n];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v = az[0][q];
                v += bj;
                zh[(ml + q) * ZPITCH + n] = v;
            }
        }
    }
    __syncthreads();
    // loss and head gradient, one lane per (row, head), by the first wave; the
    // others clear the gradient tile's columns past the heads
    if (wave == 0) {
        const int h = lane >> 4;
        float l = 0.f;
        bf16_t d[HW];
        loss_row(zh + rr * ZPITCH + h * HW, row < s.nb && head_keeps(id, h), t0, t1, cls, s.inv_n, d, l);
#pragma unroll
        for (int c = 0; c < HW; ++c) {
            act[1][sw(rr, h * HW + c)] = d[c];
            s.dOutT[(long long)(h * HW + c) * s.ldt + row] = d[c];
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            l += __shfl_xor(l, o);
        if (lane == 0)
            atomicAdd(s.loss, l * s.inv_n);
    } else if (t < 64 + FROWS * (FKH - NOUT)) {
        const int e = t - 64;
        act[1][sw(e & 15, NOUT + (e >> 4))] = 0;
    }
    __syncthreads();
    auto back = [&](int l, f32x4 (&g)[2], bf16_t *out) __attribute__((always_inline)) {  // into layer l's output gradient
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = c0 + j * 16;
            bf16x4 y;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                y[q] = (__bf16)(g[j][q] * D[l][j][q]);
            fused_put(out, ml, n, y, s.dYt[l] + (long long)n * s.ldt + m);
        }
        __syncthreads();
    };
    fused_product<FKH, 2>(act[1], bg, lane, acc);
    back(3, acc, act[0]);
    fused_load<H, 2>(s.WT[2], n0 / 16, lane, ba);
    fused_product<H, 2>(act[0], bb, lane, acc);
    back(2, acc, act[1]);
    fused_load<H, 2>(s.WT[1], n0 / 16, lane, bb);
    fused_product<H, 2>(act[1], ba, lane, acc);
    back(1, acc, act[0]);
    fused_product<H, 2>(act[0], bb, lane, acc);
    back(0, acc, act[1]);
}

// every layer's weight-gradient product in one launch: blocks [first[l],
// first[l + 1]) are layer l's grid, x fastest
struct WgradAll {
    GemmArgs g[NLAYER];
    int gx[NLAYER], gy[NLAYER], first[NLAYER + 1];
};

template <int T>
__global__ void __launch_bounds__(256) mlp_wgrad_all(const WgradAll a)
{
    __shared__ __attribute__((aligned(16))) bf16_t smem[(Tile<T>::TM + Tile<T>::TN) * (Tile<T>::KC + KPAD)];
    const int b = (int)blockIdx.x;
    int l = 0;
    while (b >= a.first[l + 1])
        ++l;
    const int k = b - a.first[l];
    gemm_block<EPI_WGRAD, T>(a.g[l], k % a.gx[l], k / a.gx[l] % a.gy[l], k / (a.gx[l] * a.gy[l]), smem);
}

struct MlpError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

void check(hipError_t e, const char *what)
{
    if (e != hipSuccess)
        throw MlpError(std::string(what) + ": " + hipGetErrorString(e));
}

// Device address of the static `scratch` array, per device: looked up once
// per device, with that device current, by the first clode_mlp_create on it.
std::mutex g_scratch_mu;
std::vector<unsigned char *> g_scratch_addr;

unsigned char *scratch_address(int device)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if ((size_t)device >= g_scratch_addr.size())
        g_scratch_addr.resize((size_t)device + 1, nullptr);
    if (!g_scratch_addr[device]) {
        void *p = nullptr;
        check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        g_scratch_addr[device] = static_cast<unsigned char *>(p);
    }
    return g_scratch_addr[device];
}

template <class T>
struct Dev {
    T *p = nullptr;
    size_t n = 0;
    void alloc(size_t k)
    {
        if (k <= n && p)
            return;
        free();
        check(hipMalloc((void **)&p, std::max<size_t>(k, 1) * sizeof(T)), "hipMalloc");
        n = k;
    }
    void free()
    {
        if (p)
            (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    ~Dev() { free(); }
};

struct Layer {
    int in, out;        // out x in weights, stored transposed Wt[out][in]
    size_t woff, boff;  // offsets in the flat parameter vector
};

}  // namespace

struct clode_mlp {
    int device = 0;
    int cus = 256;  // compute units of the device (tile-size choice)
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    Layer L[NLAYER];
    size_t nparam = 0;
    std::vector<float> Bff;       // [2][16] Fourier frequencies
    float tmean[2] = {0, 0}, tstd[2] = {1, 1};
    Dev<float> p, g, m1, m2, dBff, dT, dtm;
    Dev<uint8_t> mask;
    Dev<bf16_t> pbf, pbfT, pbfF, pbfTF;  // the WeightCopies
    // activations for a chunk of rows, and transposed copies [width][ldt]
    // (ldt = rows rounded up to 16) for the weight-gradient products
    Dev<bf16_t> A0, Y[NHID], dY[NHID], dOut;
    Dev<bf16_t> A0t, Yt[NHID], dYt[NHID], dOutT;
    Dev<float> Z[NHID], Zh, X, T, loss, wsp;
    Dev<float> wall;  // split-K partial weight gradients of all layers (training), KSPLIT_MAX x nparam
    Dev<int> C;
    Dev<unsigned long long> ids;
    long long adamStep = 0;
    double lastMs = 0;
    size_t rows = 0;
    unsigned char *stage = nullptr;  // this device's static scratch (no-allocation screening)
    // outputs of the last screening, kept for the next up to GRID_KEEP cells;
    // one screening of a network uses them at a time
    std::mutex gridMu;
    Dev<float> gP, gA;
    Dev<int> gC;
    Dev<uint8_t> gF, gF2;
    const std::shared_ptr<clode::StagedCopy> staging = clode::StagedCopy::get();

    WeightCopies copies() const { return {pbf.p, pbfT.p, pbfF.p, pbfTF.p}; }
    LayerTable table() const
    {
        LayerTable lt;
        for (int l = 0; l < NLAYER; ++l) {
            lt.woff[l] = (long long)L[l].woff;
            lt.in[l] = L[l].in;
            lt.out[l] = L[l].out;
        }
        return lt;
    }

    // the transposed operands of the weight gradients (all that a fused
    // training pass leaves in memory)
    void ensureTransposed(size_t n)
    {
        const size_t nt = (n + FROWS - 1) / FROWS * FROWS;
        A0t.alloc(nt * D0);
        for (int l = 0; l < NHID; ++l) {
            Yt[l].alloc(nt * H);
            dYt[l].alloc(nt * H);
        }
        dOutT.alloc(nt * NOUTP);
    }

    void ensureRows(size_t n)
    {
        if (n <= rows)
            return;
        ensureTransposed(n);
        A0.alloc(n * D0);
        for (int l = 0; l < NHID; ++l) {
            Y[l].alloc(n * H);
            dY[l].alloc(n * H);
            Z[l].alloc(n * H);
        }
        dOut.alloc(n * NOUTP);
        // the loss kernel never writes the padding columns: they stay zero
        check(hipMemsetAsync(dOut.p, 0, n * NOUTP * sizeof(bf16_t), stream), "hipMemsetAsync");
        Zh.alloc(n * NOUTP);
        X.alloc(n * 2);
        T.alloc(n * 2);
        C.alloc(n);
        ids.alloc(n);
        rows = n;
    }
};

namespace {

template <int T>
void gemm_tiled(clode_mlp *h, int epi, const GemmArgs &a)
{
    constexpr int TM = Tile<T>::TM, TN = Tile<T>::TN;
    const int splits = a.ksplit > 0 ? (a.K + a.ksplit - 1) / a.ksplit : 1;
    dim3 grid((a.N + TN - 1) / TN, (a.M + TM - 1) / TM, splits);
    switch (epi) {
    case EPI_FWD_SILU: hipLaunchKernelGGL((mlp_gemm<EPI_FWD_SILU, T>), grid, dim3(256), 0, h->stream, a); break;
    case EPI_FWD_LINEAR: hipLaunchKernelGGL((mlp_gemm<EPI_FWD_LINEAR, T>), grid, dim3(256), 0, h->stream, a); break;
    case EPI_BWD_DSILU: hipLaunchKernelGGL((mlp_gemm<EPI_BWD_DSILU, T>), grid, dim3(256), 0, h->stream, a); break;
    default: hipLaunchKernelGGL((mlp_gemm<EPI_WGRAD, T>), grid, dim3(256), 0, h->stream, a); break;
    }
    check(hipGetLastError(), "mlp_gemm launch");
}

// 128 x 128 tiles once the product has enough rows to keep every CU busy
// with them (screening chunks); 64 x 64 below that; 32 x 32 when 64 x 64
// tiles would leave CUs idle (the training minibatch products: 2048 x 256
// is 128 tiles of 64 x 64 on 256 CUs).  Every tile size accumulates each
// output element over the same K chunks in the same order, so the results
// are identical.
int tile_for(const clode_mlp *h, const GemmArgs &a)
{
    const long long splits = a.ksplit > 0 ? (a.K + a.ksplit - 1) / a.ksplit : 1;
    const long long tiles64 = (long long)((a.M + 63) / 64) * ((a.N + 63) / 64) * splits;
    if (a.ksplit == 0 && a.M >= 32768)
        return 128;
    return tiles64 < h->cus ? 32 : 64;
}

void gemm(clode_mlp *h, int epi, const GemmArgs &a)
{
    switch (tile_for(h, a)) {
    case 128: gemm_tiled<128>(h, epi, a); break;
    case 32: gemm_tiled<32>(h, epi, a); break;
    default: gemm_tiled<64>(h, epi, a); break;
    }
}

GemmArgs ga() { GemmArgs a; std::memset(&a, 0, sizeof(a)); return a; }

inline int ldT(int n) { return (n + FROWS - 1) / FROWS * FROWS; }

constexpr long long GRID_KEEP = 1ll << 23;  // screening outputs kept between calls: 14 bytes per cell, 117 MB
constexpr int KSPLIT_MAX = 32;    // partial products per weight gradient
constexpr int KSPLIT_ROWS = 256;  // rows per partial product (at least)

// forward over n rows already encoded in h->A0; with train, the activations'
// transposed copies are written for backward
void forward(clode_mlp *h, int n, bool train = false)
{
    const bf16_t *in = h->A0.p;
    int kin = D0;
    for (int l = 0; l < NHID; ++l) {
        GemmArgs a = ga();
        a.M = n; a.N = H; a.K = kin;
        a.A = in; a.lda_m = kin; a.lda_k = 1;
        a.B = h->pbf.p + h->L[l].woff; a.ldb_k = 1; a.ldb_n = kin;
        a.bias = h->p.p + h->L[l].boff;
        a.ldz = H;
        a.Yout = h->Y[l].p; a.ldy = H;
        if (train) {  // backward needs the pre-activations and the transposed activations
            a.Zout = h->Z[l].p;
            a.YTout = h->Yt[l].p;
            a.ldt = ldT(n);
        }
        gemm(h, EPI_FWD_SILU, a);
        in = h->Y[l].p;
        kin = H;
    }
    GemmArgs a = ga();
    a.M = n; a.N = NOUTP; a.K = H;
    a.A = in; a.lda_m = H; a.lda_k = 1;
    a.B = h->pbf.p + h->L[NHID].woff; a.ldb_k = 1; a.ldb_n = H;
    a.bias = h->p.p + h->L[NHID].boff;
    a.Zout = h->Zh.p; a.ldz = NOUTP;
    gemm(h, EPI_FWD_LINEAR, a);
}

// layer l's weight gradient from the transposed operands of n rows, as split-K
// partial products cstride apart: dWt[o][i] = sum_m dz[m][o] x[m][i] =
// sum_m dzt[o][m] xt[i][m], the batch (the reduction) split so that the product
// has enough workgroups
GemmArgs wgrad_args(clode_mlp *h, int l, int n, const bf16_t *dzt, float *Cout, long long cstride, int *splits_used)
{
    const Layer &Ly = h->L[l];
    const int lt = ldT(n);
    GemmArgs w = ga();
    w.M = Ly.out; w.N = Ly.in; w.K = n;
    w.A = dzt; w.lda_m = lt; w.lda_k = 1;
    w.B = l > 0 ? h->Yt[l - 1].p : h->A0t.p; w.ldb_k = 1; w.ldb_n = lt;
    const int splits = std::max(1, std::min(KSPLIT_MAX, n / KSPLIT_ROWS));
    w.ksplit = ((n + splits - 1) / splits + TK - 1) / TK * TK;
    *splits_used = (n + w.ksplit - 1) / w.ksplit;
    w.Cout = Cout; w.ldc = Ly.in; w.cstride = cstride;
    return w;
}

// backward from h->dOut / h->dOutT (BF16) into h->g; every product reads
// operands that are contiguous along its reduction index
void backward(clode_mlp *h, int n)
{
    const int lt = ldT(n);
    const bf16_t *dz = h->dOut.p, *dzt = h->dOutT.p;
    int nout = NOUTP;
    for (int l = NHID; l >= 0; --l) {
        const Layer &Ly = h->L[l];
        // the partial products are summed in a fixed order
        int used = 0;
        const long long count = (long long)Ly.out * Ly.in;
        gemm(h, EPI_WGRAD, wgrad_args(h, l, n, dzt, h->wsp.p, count, &used));
        const int sum_blocks = (int)((count + 255) / 256);
        hipLaunchKernelGGL(mlp_layer_grads, dim3((unsigned int)(sum_blocks + Ly.out)), dim3(256), 0, h->stream,
                           h->wsp.p, used, count, h->g.p + Ly.woff, sum_blocks, dzt, n, Ly.out, lt, h->g.p + Ly.boff);
        check(hipGetLastError(), "mlp_layer_grads launch");
        if (l == 0)
            break;
        // dY[l-1][m][i] = (sum_o dz[m][o] W[i][o]) * silu'(Z[l-1][m][i])
        GemmArgs d = ga();
        d.M = n; d.N = Ly.in; d.K = Ly.out;
        d.A = dz; d.lda_m = nout; d.lda_k = 1;
        d.B = h->pbfT.p + Ly.woff; d.ldb_k = 1; d.ldb_n = Ly.out;
        d.Zin = h->Z[l - 1].p; d.ldz = H;
        d.Yout = h->dY[l - 1].p; d.ldy = H;
        d.YTout = h->dYt[l - 1].p; d.ldt = lt;
        gemm(h, EPI_BWD_DSILU, d);
        dz = h->dY[l - 1].p;
        dzt = h->dYt[l - 1].p;
        nout = H;
    }
}

// One training step's row-wise pass and weight-gradient products, two launches.
// The partial weight gradients of every layer stay in h->wall (split z of
// parameter i at z * nparam + i); gs receives where they and the transposed
// output gradients are, for mlp_adam_sum.
void fused_step(clode_mlp *h, const FusedStep &f, GradSources &gs)
{
    const unsigned int groups = (unsigned int)((f.nb + 8 * FROWS - 1) / (8 * FROWS) * 8);  // as many for each XCD
    hipLaunchKernelGGL(mlp_fused_step, dim3(groups), dim3(FWAVES * 64), 0, h->stream, f);
    check(hipGetLastError(), "mlp_fused_step launch");
    WgradAll a;
    int blocks = 0, tiles64 = 0;
    gs.part = h->wall.p;
    gs.pstride = (long long)h->nparam;
    gs.n = f.nb;
    gs.ld = f.ldt;
    for (int l = 0; l < NLAYER; ++l) {
        gs.dzt[l] = l < NHID ? h->dYt[l].p : h->dOutT.p;
        a.g[l] = wgrad_args(h, l, f.nb, gs.dzt[l], h->wall.p + h->L[l].woff, gs.pstride, &gs.splits);
        if (l == NHID)
            a.g[l].M = NOUT;  // the padding's gradients are not used
        tiles64 += ((a.g[l].N + 63) / 64) * ((a.g[l].M + 63) / 64) * gs.splits;
    }
    // 32 x 32 tiles until 64 x 64 ones fill every CU twice.  A step took, with
    // 32 and with 64: 35.4 and 37.7 us at 1000 rows (180 tiles of 64 x 64), the
    // same at 2048 (480), 53.0 and 51.1 at 4096 (960), 175 and 168 at 16384
    const int tile = tiles64 < 2 * h->cus ? 32 : 64;
    for (int l = 0; l < NLAYER; ++l) {
        a.first[l] = blocks;
        a.gx[l] = (a.g[l].N + tile - 1) / tile;
        a.gy[l] = (a.g[l].M + tile - 1) / tile;
        blocks += a.gx[l] * a.gy[l] * gs.splits;
    }
    a.first[NLAYER] = blocks;
    if (tile == 32)
        hipLaunchKernelGGL((mlp_wgrad_all<32>), dim3((unsigned int)blocks), dim3(256), 0, h->stream, a);
    else
        hipLaunchKernelGGL((mlp_wgrad_all<64>), dim3((unsigned int)blocks), dim3(256), 0, h->stream, a);
    check(hipGetLastError(), "mlp_wgrad_all launch");
}

void encode(clode_mlp *h, const float *Xdev, int n, bool train = false)
{
    hipLaunchKernelGGL(mlp_encode, dim3((n + 255) / 256), dim3(256), 0, h->stream, Xdev, n, h->dBff.p, h->A0.p,
                       train ? h->A0t.p : nullptr, ldT(n));
    check(hipGetLastError(), "mlp_encode launch");
}

void upload(clode_mlp *h, void *dst, const void *src, size_t bytes)
{
    check(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, h->stream), "hipMemcpy H2D");
}
void download(clode_mlp *h, void *dst, const void *src, size_t bytes)
{
    check(h->staging->toHost(h->device, dst, src, bytes, h->stream), "hipMemcpy D2H");
}

void refresh_bf16(clode_mlp *h)
{
    hipLaunchKernelGGL(mlp_put_weights, dim3((unsigned int)((h->nparam + 255) / 256)), dim3(256), 0, h->stream, h->p.p,
                       h->copies(), h->table(), (long long)h->nparam);
    check(hipGetLastError(), "mlp_put_weights launch");
    check(hipStreamSynchronize(h->stream), "hipStreamSynchronize");
}

// loss and gradient over n rows (inputs X, targets T, classes C already on the device)
float loss_grad(clode_mlp *h, int n)
{
    encode(h, h->X.p, n, true);
    forward(h, n, true);
    check(hipMemsetAsync(h->loss.p, 0, 4, h->stream), "hipMemset");
    hipLaunchKernelGGL(mlp_loss, dim3((NHEAD * n + 255) / 256), dim3(256), 0, h->stream, h->Zh.p, n, h->T.p, h->C.p, h->ids.p,
                       1.0f / (float)n, h->dOut.p, h->dOutT.p, ldT(n), h->loss.p);
    check(hipGetLastError(), "mlp_loss launch");
    backward(h, n);
    float l = 0;
    download(h, &l, h->loss.p, 4);
    return l;
}

// a caller's pointer that must not be null
template <class T>
T *need(T *p, const char *what)
{
    if (!p)
        throw std::invalid_argument(std::string("null ") + what);
    return p;
}

#define MLP_TRY try {
#define MLP_CATCH                        \
    }                                    \
    catch (const std::invalid_argument &e) \
    {                                    \
        g_err = e.what();                \
        return CLODE_MLP_ERR_INVALID;    \
    }                                    \
    catch (const std::exception &e)      \
    {                                    \
        g_err = e.what();                \
        return CLODE_MLP_ERR_RUNTIME;    \
    }                                    \
    return CLODE_MLP_OK;

#define CHECK_H(h)                        \
    if (!(h)) {                           \
        g_err = "null surrogate handle";  \
        return CLODE_MLP_ERR_INVALID;     \
    }

// ---- screening steps shared by the allocating and the no-allocation entry points

void upload_target_scaling(clode_mlp *h)
{
    float tm[4] = {h->tmean[0], h->tmean[1], h->tstd[0], h->tstd[1]};
    upload(h, h->dtm.p, tm, 16);
}

// the fused screening kernel over the nx x ny grid into device outputs
void screen_fused(clode_mlp *h, int nx, int ny, float tol, float *P, float *A, int *C, uint8_t *F)
{
    const long long ncell = (long long)nx * ny;
    ScreenArgs a;
    std::memset(&a, 0, sizeof(a));
    a.ncell = ncell;
    a.nx = nx;
    a.ny = ny;
    a.Bff = h->dBff.p;
    for (int l = 0; l < NLAYER; ++l) {
        a.W[l] = h->pbfF.p + h->L[l].woff;
        a.bias[l] = h->p.p + h->L[l].boff;
        if (((uintptr_t)a.W[l] & 15) != 0)  // the kernel reads 16-byte weight fragments
            throw MlpError("screening weights are not 16-byte aligned");
    }
    a.tm = h->dtm.p;
    a.tol = tol;
    a.period = P;
    a.amp = A;
    a.cls = C;
    a.flags = F;
    const unsigned int nblk = (unsigned int)((ncell + SROWS - 1) / SROWS);
    hipLaunchKernelGGL(mlp_screen_fused, dim3(nblk), dim3(256), 0, h->stream, a);
    check(hipGetLastError(), "mlp_screen_fused launch");
}

// flags bit 1 (class boundary) into F, then `dilate` rounds of dilation
// between F and F2 (two buffers of nx * ny bytes); returns the buffer that
// holds the final flags
const uint8_t *screen_flags(clode_mlp *h, int nx, int ny, int dilate, const int *C, uint8_t *F, uint8_t *F2)
{
    const long long ncell = (long long)nx * ny;
    const unsigned int gb = (unsigned int)((ncell + 255) / 256);
    hipLaunchKernelGGL(mlp_boundary, dim3(gb), dim3(256), 0, h->stream, C, nx, ny, F);
    check(hipGetLastError(), "mlp_boundary launch");
    for (int r = 0; r < dilate; ++r) {
        hipLaunchKernelGGL(mlp_dilate, dim3(gb), dim3(256), 0, h->stream, F, nx, ny, F2);
        check(hipGetLastError(), "mlp_dilate launch");
        std::swap(F, F2);
    }
    return F;
}

// a caller's output pointer that must be device memory of the handle's device
template <class T>
void need_device(clode_mlp *h, T *p, const char *what)
{
    need(p, what);
    hipPointerAttribute_t at;
    std::memset(&at, 0, sizeof(at));
    const hipError_t e = hipPointerGetAttributes(&at, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();  // leave no error behind for the next HIP call
        throw std::invalid_argument(std::string(what) + " is not device memory");
    }
    if ((at.type != hipMemoryTypeDevice && at.type != hipMemoryTypeManaged) || at.device != h->device)
        throw std::invalid_argument(std::string(what) + " is not device memory of device " +
                                    std::to_string(h->device));
}

}  // namespace

extern "C" {

const char *clode_mlp_last_error(void) { return g_err.c_str(); }

int clode_mlp_create(clode_mlp **out, int device, unsigned long long seed)
{
    if (!out) {
        g_err = "null output handle";
        return CLODE_MLP_ERR_INVALID;
    }
    *out = nullptr;
    MLP_TRY
    int nd = 0;
    if (hipGetDeviceCount(&nd) != hipSuccess || nd <= 0)
        throw MlpError("no HIP device is available");
    if (device < 0 || device >= nd)
        throw std::invalid_argument("device ordinal out of range");
    check(hipSetDevice(device), "hipSetDevice");
    auto *h = new clode_mlp;
    try {
        h->device = device;
        check(hipDeviceGetAttribute(&h->cus, hipDeviceAttributeMultiprocessorCount, device), "hipDeviceGetAttribute");
        check(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking), "hipStreamCreate");
        check(hipEventCreate(&h->ev0), "hipEventCreate");
        check(hipEventCreate(&h->ev1), "hipEventCreate");
        size_t off = 0;
        int in = D0;
        for (int l = 0; l < NLAYER; ++l) {
            int o = l < NHID ? H : NOUTP;
            h->L[l] = Layer{in, o, off, off + (size_t)in * o};
            off += (size_t)in * o + o;
            in = o;
        }
        h->nparam = off;
        // He-style initialisation for SiLU layers, small heads; Fourier frequencies ~ N(0, 3^2)
        clode::Normals nd01(seed);
        std::vector<float> p(h->nparam, 0.f);
        std::vector<uint8_t> mask(h->nparam, 1);
        for (int l = 0; l < NLAYER; ++l) {
            const Layer &Ly = h->L[l];
            float sd = l < NHID ? std::sqrt(2.f / Ly.in) : std::sqrt(1.f / Ly.in);
            for (int o = 0; o < Ly.out; ++o)
                for (int i = 0; i < Ly.in; ++i) {
                    size_t k = Ly.woff + (size_t)o * Ly.in + i;
                    if (l == NHID && o >= NOUT) {
                        mask[k] = 0;  // padding columns stay zero
                        continue;
                    }
                    p[k] = sd * nd01();
                }
            if (l == NHID)
                for (int o = NOUT; o < NOUTP; ++o)
                    mask[Ly.boff + o] = 0;
        }
        h->Bff.resize(2 * NFF);
        for (auto &b : h->Bff)
            b = 3.f * nd01();
        h->p.alloc(h->nparam);
        h->g.alloc(h->nparam);
        h->m1.alloc(h->nparam);
        h->m2.alloc(h->nparam);
        h->mask.alloc(h->nparam);
        h->pbf.alloc(h->nparam);
        h->pbfT.alloc(h->nparam);
        h->pbfF.alloc(h->nparam);
        h->pbfTF.alloc(h->nparam);
        h->wsp.alloc((size_t)KSPLIT_MAX * H * H);  // the largest weight gradient, per split
        h->wall.alloc((size_t)KSPLIT_MAX * h->nparam);  // every layer's, per split (30 MB)
        h->dBff.alloc(2 * NFF);
        h->dtm.alloc(4);
        h->loss.alloc(1);
        h->stage = scratch_address(device);  // device is current (hipSetDevice above)
        upload(h, h->p.p, p.data(), p.size() * 4);
        upload(h, h->mask.p, mask.data(), mask.size());
        upload(h, h->dBff.p, h->Bff.data(), h->Bff.size() * 4);
        check(hipMemsetAsync(h->g.p, 0, h->nparam * 4, h->stream), "hipMemset");
        check(hipMemsetAsync(h->m1.p, 0, h->nparam * 4, h->stream), "hipMemset");
        check(hipMemsetAsync(h->m2.p, 0, h->nparam * 4, h->stream), "hipMemset");
        refresh_bf16(h);
    } catch (...) {
        clode_mlp_destroy(h);
        throw;
    }
    *out = h;
    MLP_CATCH
}

int clode_mlp_destroy(clode_mlp *h)
{
    if (!h)
        return CLODE_MLP_OK;
    (void)hipSetDevice(h->device);
    if (h->stream) {
        (void)hipStreamSynchronize(h->stream);
        (void)hipStreamDestroy(h->stream);
    }
    if (h->ev0)
        (void)hipEventDestroy(h->ev0);
    if (h->ev1)
        (void)hipEventDestroy(h->ev1);
    delete h;
    return CLODE_MLP_OK;
}

int clode_mlp_n_params(clode_mlp *h, size_t *n)
{
    CHECK_H(h) MLP_TRY *need(n, "n") = h->nparam;
    MLP_CATCH
}

int clode_mlp_get_params(clode_mlp *h, float *out, size_t n)
{
    CHECK_H(h) MLP_TRY
    if (n != h->nparam)
        throw std::invalid_argument("parameter vector has the wrong length");
    need(out, "output buffer");
    check(hipSetDevice(h->device), "hipSetDevice");
    download(h, out, h->p.p, n * 4);
    MLP_CATCH
}

int clode_mlp_set_params(clode_mlp *h, const float *in, size_t n)
{
    CHECK_H(h) MLP_TRY
    if (n != h->nparam)
        throw std::invalid_argument("parameter vector has the wrong length");
    need(in, "parameter vector");
    check(hipSetDevice(h->device), "hipSetDevice");
    upload(h, h->p.p, in, n * 4);
    refresh_bf16(h);
    MLP_CATCH
}

int clode_mlp_get_fourier(clode_mlp *h, float *out, size_t n)
{
    CHECK_H(h) MLP_TRY
    if (n != 2 * NFF)
        throw std::invalid_argument("Fourier matrix has 32 entries");
    std::copy(h->Bff.begin(), h->Bff.end(), need(out, "output buffer"));
    MLP_CATCH
}

int clode_mlp_set_target_scaling(clode_mlp *h, const float *mean2, const float *std2)
{
    CHECK_H(h) MLP_TRY
    need(mean2, "mean2");
    need(std2, "std2");
    for (int k = 0; k < 2; ++k) {
        if (!(std2[k] > 0))
            throw std::invalid_argument("target scales must be positive");
        h->tmean[k] = mean2[k];
        h->tstd[k] = std2[k];
    }
    MLP_CATCH
}

int clode_mlp_forward(clode_mlp *h, const float *X, size_t n, float *out, unsigned short *encoded)
{
    CHECK_H(h) MLP_TRY
    if (n == 0 || n > (1u << 18))
        throw std::invalid_argument("forward takes 1 to 262144 rows");
    need(X, "input rows");
    need(out, "output buffer");
    check(hipSetDevice(h->device), "hipSetDevice");
    h->ensureRows(n);
    upload(h, h->X.p, X, n * 8);
    encode(h, h->X.p, (int)n);
    forward(h, (int)n);
    std::vector<float> z(n * NOUTP);
    download(h, z.data(), h->Zh.p, z.size() * 4);
    for (size_t i = 0; i < n; ++i)
        std::copy(z.begin() + i * NOUTP, z.begin() + i * NOUTP + NOUT, out + i * NOUT);
    if (encoded)
        download(h, encoded, h->A0.p, n * D0 * 2);
    MLP_CATCH
}

int clode_mlp_loss_grad(clode_mlp *h, const float *X, const float *T, const int *cls, size_t n, float *loss,
                        float *grad)
{
    CHECK_H(h) MLP_TRY
    if (n == 0 || n > (1u << 16))
        throw std::invalid_argument("loss_grad takes 1 to 65536 rows");
    need(X, "input rows");
    need(T, "targets");
    need(cls, "class labels");
    need(loss, "loss output");
    for (size_t i = 0; i < n; ++i)
        if (cls[i] < 0 || cls[i] >= NCLS)
            throw std::invalid_argument("class labels must be in 0..15");
    check(hipSetDevice(h->device), "hipSetDevice");
    h->ensureRows(n);
    upload(h, h->X.p, X, n * 8);
    upload(h, h->T.p, T, n * 8);
    upload(h, h->C.p, cls, n * 4);
    std::vector<unsigned long long> ids(n);
    for (size_t i = 0; i < n; ++i)
        ids[i] = i;
    upload(h, h->ids.p, ids.data(), n * 8);
    *loss = loss_grad(h, (int)n);
    if (grad)
        download(h, grad, h->g.p, h->nparam * 4);
    MLP_CATCH
}

int clode_mlp_train(clode_mlp *h, const float *X, const float *T, const int *cls, size_t n, int epochs, int batch,
                    float lr, unsigned long long seed, float *epoch_loss)
{
    CHECK_H(h) MLP_TRY
    if (n < 1 || n > (1u << 24) || epochs < 1 || batch < 64 || batch > 65536)
        throw std::invalid_argument("train: 1..16777216 samples, epochs >= 1, batch 64..65536");
    need(X, "input rows");
    need(T, "targets");
    need(cls, "class labels");
    for (size_t i = 0; i < n; ++i)
        if (cls[i] < 0 || cls[i] >= NCLS)
            throw std::invalid_argument("class labels must be in 0..15");
    check(hipSetDevice(h->device), "hipSetDevice");
    // the training set stays on the device; each step gathers a shuffled
    // minibatch into the activation buffers
    Dev<float> Xall, Tall, eloss;
    Dev<int> Call;
    Dev<unsigned int> dperm;
    Xall.alloc(n * 2);
    Tall.alloc(n * 2);
    Call.alloc(n);
    dperm.alloc(n);
    eloss.alloc((size_t)epochs);
    upload(h, Xall.p, X, n * 8);
    upload(h, Tall.p, T, n * 8);
    upload(h, Call.p, cls, n * 4);
    std::mt19937_64 rng(seed);
    // epoch e's order is a shuffle of epoch e-1's; the next epoch's shuffle
    // runs on the host while the GPU trains on the current one.  Every
    // epoch's order has its own host buffer, untouched after its upload
    // is queued, and the epoch losses stay on the device until the end, so
    // the host waits between epochs only for an upload two epochs back.
    std::vector<unsigned int> perms[2] = {std::vector<unsigned int>(n), std::vector<unsigned int>(n)};
    hipEvent_t uploaded[2];
    for (int b = 0; b < 2; ++b)
        check(hipEventCreateWithFlags(&uploaded[b], hipEventDisableTiming), "hipEventCreate");
    for (size_t i = 0; i < n; ++i)
        perms[0][i] = (unsigned int)i;
    std::shuffle(perms[0].begin(), perms[0].end(), rng);
    const size_t steps_per_epoch = (n + batch - 1) / batch;
    const double total = (double)steps_per_epoch * epochs;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const LayerTable lt = h->table();
    // by default a step is three launches: the fused row-wise pass, every
    // layer's weight-gradient products, and the optimizer with the gradient
    // sums; CLODE_MLP_FUSED_TRAIN=0 launches every product on its own and sums
    // in the backward pass (22 launches, same parameters bit for bit)
    const char *fa = std::getenv("CLODE_MLP_FUSED_TRAIN");
    const bool fused = !(fa && std::strcmp(fa, "0") == 0);
    if (fused)
        h->ensureTransposed((size_t)batch);
    else
        h->ensureRows((size_t)batch);
    int nbias = 0;
    for (int l = 0; l < NLAYER; ++l)
        nbias += h->L[l].out;
    long long step = 0;
    check(hipMemsetAsync(eloss.p, 0, (size_t)epochs * 4, h->stream), "hipMemset");
    check(hipEventRecord(h->ev0, h->stream), "hipEventRecord");
    for (int e = 0; e < epochs; ++e) {
        upload(h, dperm.p, perms[e % 2].data(), n * 4);
        check(hipEventRecord(uploaded[e % 2], h->stream), "hipEventRecord");
        for (size_t s = 0; s < steps_per_epoch; ++s, ++step) {
            const size_t b0 = s * (size_t)batch;
            const int nb = (int)std::min<size_t>((size_t)batch, n - b0);
            GradSources gs;
            std::memset(&gs, 0, sizeof(gs));
            if (fused) {
                FusedStep f;
                std::memset(&f, 0, sizeof(f));
                f.perm = dperm.p + b0;
                f.nb = nb;
                f.ldt = ldT(nb);
                f.Xa = Xall.p;
                f.Ta = Tall.p;
                f.Ca = Call.p;
                f.Bff = h->dBff.p;
                for (int l = 0; l < NLAYER; ++l) {
                    f.W[l] = h->pbfF.p + h->L[l].woff;
                    f.WT[l] = h->pbfTF.p + h->L[l].woff;
                    f.bias[l] = h->p.p + h->L[l].boff;
                }
                f.A0t = h->A0t.p;
                for (int l = 0; l < NHID; ++l) {
                    f.Yt[l] = h->Yt[l].p;
                    f.dYt[l] = h->dYt[l].p;
                }
                f.dOutT = h->dOutT.p;
                f.inv_n = 1.0f / (float)nb;
                f.loss = eloss.p + e;
                fused_step(h, f, gs);
            } else {
                hipLaunchKernelGGL(mlp_gather, dim3((nb * NFF + 255) / 256), dim3(256), 0, h->stream, dperm.p + b0, nb,
                                   Xall.p, Tall.p, Call.p, h->T.p, h->C.p, h->ids.p, h->dBff.p, h->A0.p, h->A0t.p,
                                   ldT(nb));
                check(hipGetLastError(), "mlp_gather launch");
                forward(h, nb, true);
                hipLaunchKernelGGL(mlp_loss, dim3((NHEAD * nb + 255) / 256), dim3(256), 0, h->stream, h->Zh.p, nb,
                                   h->T.p, h->C.p, h->ids.p, 1.0f / (float)nb, h->dOut.p, h->dOutT.p, ldT(nb),
                                   eloss.p + e);
                check(hipGetLastError(), "mlp_loss launch");
                backward(h, nb);
            }
            // cosine decay to 5 % of the initial rate
            const double frac = (double)step / total;
            AdamStep as;
            as.lr = (float)(lr * (0.05 + 0.95 * 0.5 * (1.0 + std::cos(3.141592653589793 * frac))));
            as.b1 = b1;
            as.b2 = b2;
            as.eps = eps;
            ++h->adamStep;
            as.c1 = (float)(1.0 / (1.0 - std::pow((double)b1, (double)h->adamStep)));
            as.c2 = (float)(1.0 / (1.0 - std::pow((double)b2, (double)h->adamStep)));
            const int wblocks = (int)((h->nparam + 255) / 256);
            if (fused)
                hipLaunchKernelGGL(mlp_adam_sum, dim3((unsigned int)(wblocks + nbias)), dim3(256), 0, h->stream,
                                   h->p.p, h->m1.p, h->m2.p, h->mask.p, h->copies(), lt,
                                   (long long)h->nparam, wblocks, gs, as);
            else
                hipLaunchKernelGGL(mlp_adam, dim3((unsigned int)wblocks), dim3(256), 0, h->stream, h->p.p, h->g.p,
                                   h->m1.p, h->m2.p, h->mask.p, h->copies(), lt, (long long)h->nparam, as);
            check(hipGetLastError(), "mlp_adam launch");
        }
        if (e + 1 < epochs) {
            std::vector<unsigned int> &nx = perms[(e + 1) % 2];
            if (e >= 1)  // epoch e-1's upload read this buffer
                check(hipEventSynchronize(uploaded[(e + 1) % 2]), "hipEventSynchronize");
            nx = perms[e % 2];
            std::shuffle(nx.begin(), nx.end(), rng);
        }
    }
    for (int b = 0; b < 2; ++b)
        (void)hipEventDestroy(uploaded[b]);
    std::vector<float> el((size_t)epochs);
    download(h, el.data(), eloss.p, (size_t)epochs * 4);
    if (epoch_loss)
        for (int e = 0; e < epochs; ++e)
            epoch_loss[e] = el[(size_t)e] / (float)steps_per_epoch;
    check(hipEventRecord(h->ev1, h->stream), "hipEventRecord");
    check(hipStreamSynchronize(h->stream), "hipStreamSynchronize");
    float ms = 0;
    (void)hipEventElapsedTime(&ms, h->ev0, h->ev1);
    h->lastMs = ms;
    MLP_CATCH
}

int clode_mlp_screen_grid(clode_mlp *h, int nx, int ny, float tol, int dilate, float *period, float *amp, int *cls,
                          unsigned char *flags)
{
    CHECK_H(h) MLP_TRY
    if (nx < 1 || ny < 1 || (long long)nx * ny > (1ll << 26))
        throw std::invalid_argument("grid must have 1 to 2^26 cells");
    if (dilate < 0 || dilate > 64)
        throw std::invalid_argument("dilation radius must be 0..64");
    need(period, "period output");
    need(amp, "amplitude output");
    need(cls, "class output");
    need(flags, "flags output");
    check(hipSetDevice(h->device), "hipSetDevice");
    const long long ncell = (long long)nx * ny;
    std::lock_guard<std::mutex> lk(h->gridMu);
    // the fused kernel by default; CLODE_MLP_FUSED_SCREEN=0 runs the network
    // layer by layer over chunks of 2^18 cells (same results, bit for bit)
    const char *fe = std::getenv("CLODE_MLP_FUSED_SCREEN");
    const bool fused = !(fe && std::strcmp(fe, "0") == 0);
    const int chunk = (int)std::min<long long>(ncell, 1 << 18);
    if (!fused)
        h->ensureRows((size_t)chunk);
    Dev<float> &dP = h->gP, &dA = h->gA;
    Dev<int> &dC = h->gC;
    Dev<uint8_t> &dF = h->gF, &dF2 = h->gF2;
    struct GiveBack {  // a grid past GRID_KEEP leaves nothing behind, nor does a call that fails
        clode_mlp *h;
        bool keep;
        ~GiveBack()
        {
            if (keep)
                return;
            h->gP.free();
            h->gA.free();
            h->gC.free();
            h->gF.free();
            h->gF2.free();
        }
    } back{h, false};
    dP.alloc(ncell);
    dA.alloc(ncell);
    dC.alloc(ncell);
    dF.alloc(ncell);
    dF2.alloc(ncell);
    upload_target_scaling(h);
    check(hipEventRecord(h->ev0, h->stream), "hipEventRecord");
    if (fused)
        screen_fused(h, nx, ny, tol, dP.p, dA.p, dC.p, dF.p);
    for (long long c0 = 0; !fused && c0 < ncell; c0 += chunk) {
        const int nb = (int)std::min<long long>(chunk, ncell - c0);
        hipLaunchKernelGGL(mlp_grid_inputs, dim3((nb + 255) / 256), dim3(256), 0, h->stream, c0, nb, nx, ny, h->X.p);
        check(hipGetLastError(), "mlp_grid_inputs launch");
        encode(h, h->X.p, nb);
        forward(h, nb);
        hipLaunchKernelGGL(mlp_predict_cells, dim3((nb + 255) / 256), dim3(256), 0, h->stream, h->Zh.p, nb, h->dtm.p,
                           h->dtm.p + 2, tol, dP.p + c0, dA.p + c0, dC.p + c0, dF.p + c0);
        check(hipGetLastError(), "mlp_predict_cells launch");
    }
    const uint8_t *res = screen_flags(h, nx, ny, dilate, dC.p, dF.p, dF2.p);
    check(hipEventRecord(h->ev1, h->stream), "hipEventRecord");
    download(h, period, dP.p, ncell * 4);
    download(h, amp, dA.p, ncell * 4);
    download(h, cls, dC.p, ncell * 4);
    download(h, flags, res, ncell);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, h->ev0, h->ev1);
    h->lastMs = ms;
    back.keep = ncell <= GRID_KEEP;
    MLP_CATCH
}

int clode_mlp_screen_grid_noalloc(clode_mlp *h, int nx, int ny, float tol, int dilate, float *d_period, float *d_amp,
                                  int *d_cls, unsigned char *d_flags)
{
    CHECK_H(h) MLP_TRY
    if (nx < 1 || ny < 1)
        throw std::invalid_argument("grid must have at least one cell");
    const long long ncell = (long long)nx * ny;
    if (ncell > CLODE_MLP_NOALLOC_MAX_CELLS)
        throw std::invalid_argument("grid of " + std::to_string(ncell) + " cells exceeds the " +
                                    std::to_string(CLODE_MLP_NOALLOC_MAX_CELLS) +
                                    "-cell limit of the no-allocation screening (its static staging buffer)");
    if (dilate < 0 || dilate > 64)
        throw std::invalid_argument("dilation radius must be 0..64");
    check(hipSetDevice(h->device), "hipSetDevice");
    need_device(h, d_period, "period output");
    need_device(h, d_amp, "amplitude output");
    need_device(h, d_cls, "class output");
    need_device(h, d_flags, "flags output");
    if (!h->stage)
        throw MlpError("the static scratch of this device has no address");
    upload_target_scaling(h);
    check(hipEventRecord(h->ev0, h->stream), "hipEventRecord");
    screen_fused(h, nx, ny, tol, d_period, d_amp, d_cls, d_flags);
    const uint8_t *res = screen_flags(h, nx, ny, dilate, d_cls, d_flags, h->stage);
    if (res != d_flags)  // an odd number of dilation rounds ends in the staging buffer
        check(hipMemcpyAsync(d_flags, res, (size_t)ncell, hipMemcpyDeviceToDevice, h->stream), "hipMemcpy D2D");
    check(hipEventRecord(h->ev1, h->stream), "hipEventRecord");
    check(hipStreamSynchronize(h->stream), "hipStreamSynchronize");
    float ms = 0;
    (void)hipEventElapsedTime(&ms, h->ev0, h->ev1);
    h->lastMs = ms;
    MLP_CATCH
}

int clode_mlp_last_ms(clode_mlp *h, double *ms)
{
    CHECK_H(h) MLP_TRY *need(ms, "ms") = h->lastMs;
    MLP_CATCH
}

}  // extern "C"
