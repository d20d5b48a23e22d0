// hx_block.hip — the full Mamba block forward on gfx950:
//   xz = x . W_in^T           (matrix-core GEMM, split into x | z)
//   xc = SiLU(conv1d_causal(x) + conv_b)   (depthwise, kernel d_conv)
//   dt_lo | B | C = xc . W_x^T  (GEMM, three outputs)
//   dt = dt_lo . W_dt^T       (GEMM)
//   y  = selective_scan(xc, dt, A, B, C, D, z, dt_bias, softplus)
//   out = y . W_out^T         (GEMM)
// The reference's exported MambaBlock::forward_mamba is Linear -> SiLU -> Linear
// (crates/nn/src/lib.rs:888-906) and allocates A/B/C/D/delta_proj/B_proj/C_proj it never uses
// (lib.rs:851-867); this is the block those parameters describe. bf16 storage, fp32 arithmetic.
#include "hx_common.h"
#include "hx_wave.h"

extern "C" int hx_gemm_bf16(int64_t M, int64_t N, int64_t K, const void* X, int64_t ldx,
                            const void* W, int64_t ldw, const float* bias, int act, int out_dtype,
                            void* Y0, int64_t ld0, int64_t split1, void* Y1, int64_t ld1,
                            int64_t split2, void* Y2, int64_t ld2, void* stream);

namespace hx {
namespace {

// Causal depthwise conv over time + bias + SiLU. A thread owns CPT adjacent channels (16 bytes
// of a row when VEC) and TT consecutive steps; it keeps the last KW input rows in registers, so
// each input row is read once plus a KW-1 row halo per run of TT steps. Block = 256 threads
// across channels; grid.x = batch x step-runs, grid.y = channel blocks.
// y[b,t,d] = silu(bias[d] + sum_j w[d,j] * x[b, t-(KW-1)+j, d]), zero before t = 0.
template <typename T, int CPT, bool VEC>
struct ConvRow {
    __device__ static inline void load(const T* p, float (&v)[CPT]) {
        if constexpr (VEC && sizeof(T) == 2 && CPT == 8) {
            const uint4 q = *reinterpret_cast<const uint4*>(p);
            const uint32_t wds[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[2 * i] = __uint_as_float(wds[i] << 16);
                v[2 * i + 1] = __uint_as_float(wds[i] & 0xffff0000u);
            }
        } else if constexpr (VEC && sizeof(T) == 4 && CPT == 4) {
            const float4 q = *reinterpret_cast<const float4*>(p);
            v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        } else {
#pragma unroll
            for (int i = 0; i < CPT; ++i) v[i] = Storage<T>::load(p + i);
        }
    }
    __device__ static inline void store(T* p, const float (&v)[CPT]) {
        if constexpr (VEC && sizeof(T) == 2 && CPT == 8) {
            uint32_t wds[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                wds[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
            *reinterpret_cast<uint4*>(p) = make_uint4(wds[0], wds[1], wds[2], wds[3]);
        } else if constexpr (VEC && sizeof(T) == 4 && CPT == 4) {
            *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int i = 0; i < CPT; ++i) Storage<T>::store(p + i, v[i]);
        }
    }
};

template <typename T, int KW, int CPT, bool VEC, int TT>
__global__ __launch_bounds__(256) void conv1d_silu_kernel(int L, int Dm, int nruns,
                                                          const T* __restrict__ x, int64_t ldx,
                                                          const float* __restrict__ w,
                                                          const float* __restrict__ bias,
                                                          T* __restrict__ y) {
    const int d0 = (blockIdx.y * blockDim.x + threadIdx.x) * CPT;
    if (d0 >= Dm) return;
    const int b = blockIdx.x / nruns;
    const int t0 = (blockIdx.x - b * nruns) * TT;
    float wk[KW][CPT], bv[CPT];
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
        bv[i] = bias ? bias[d0 + i] : 0.0f;
#pragma unroll
        for (int j = 0; j < KW; ++j) wk[j][i] = w[(d0 + i) * KW + j];
    }
    const T* xb = x + (int64_t)b * L * ldx + d0;
    T* yb = y + (int64_t)b * L * Dm + d0;
    if constexpr (VEC && sizeof(T) == 2 && CPT == 8) {
        if (t0 + TT <= L) {
            // a whole run: every input row of it (and the halo) is loaded up front, raw, so the
            // thread has all its loads in flight at once; then the same arithmetic as below
            uint4 raw[TT + KW - 1];
#pragma unroll
            for (int j = 0; j < TT + KW - 1; ++j) {
                const int tt = t0 - (KW - 1) + j;
                raw[j] = tt >= 0 ? *reinterpret_cast<const uint4*>(xb + (int64_t)tt * ldx) : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int s = 0; s < TT; ++s) {
                float o[CPT];
#pragma unroll
                for (int i = 0; i < CPT; ++i) {
                    float acc = bv[i];
#pragma unroll
                    for (int j = 0; j < KW; ++j) {
                        const uint4 q = raw[s + j];
                        const uint32_t wd = (i >> 1) == 0 ? q.x : (i >> 1) == 1 ? q.y : (i >> 1) == 2 ? q.z : q.w;
                        const float xv = __uint_as_float((i & 1) ? (wd & 0xffff0000u) : (wd << 16));
                        acc = fmaf(wk[j][i], xv, acc);
                    }
                    o[i] = silu(acc);
                }
                ConvRow<T, CPT, VEC>::store(yb + (int64_t)(t0 + s) * Dm, o);
            }
            return;
        }
    }
    float win[KW][CPT];  // win[KW-1] = row t, win[KW-2] = row t-1, ...
#pragma unroll
    for (int j = 0; j < KW - 1; ++j) {
        const int tt = t0 - (KW - 1) + j;
        if (tt >= 0) {
            ConvRow<T, CPT, VEC>::load(xb + (int64_t)tt * ldx, win[j + 1]);
        } else {
#pragma unroll
            for (int i = 0; i < CPT; ++i) win[j + 1][i] = 0.0f;
        }
    }
#pragma unroll
    for (int s = 0; s < TT; ++s) {
        const int t = t0 + s;
        if (t >= L) break;
#pragma unroll
        for (int j = 0; j < KW - 1; ++j)
#pragma unroll
            for (int i = 0; i < CPT; ++i) win[j][i] = win[j + 1][i];
        ConvRow<T, CPT, VEC>::load(xb + (int64_t)t * ldx, win[KW - 1]);
        float o[CPT];
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            float acc = bv[i];
#pragma unroll
            for (int j = 0; j < KW; ++j) acc = fmaf(wk[j][i], win[j][i], acc);
            o[i] = silu(acc);
        }
        ConvRow<T, CPT, VEC>::store(yb + (int64_t)t * Dm, o);
    }
}

template <typename T, int KW, int CPT, bool VEC, int TT>
void launch_conv_tt(int64_t Bt, int64_t L, int64_t Dm, int64_t groups, int nthr, const void* x,
                    int64_t ldx, const float* w, const float* b, void* y, hipStream_t s) {
    const int nruns = (int)((L + TT - 1) / TT);
    dim3 grid((unsigned)(Bt * nruns), (unsigned)((groups + nthr - 1) / nthr));
    hipLaunchKernelGGL((conv1d_silu_kernel<T, KW, CPT, VEC, TT>), grid, dim3(nthr), 0, s, (int)L,
                       (int)Dm, nruns, (const T*)x, ldx, w, b, (T*)y);
}

template <typename T, int KW, int CPT, bool VEC>
void launch_conv_k(int64_t Bt, int64_t L, int64_t Dm, const void* x, int64_t ldx, const float* w,
                   const float* b, void* y, hipStream_t s) {
    // threads per block: the row's channel groups rounded up to whole waves, at most 256
    const int64_t groups = (Dm + CPT - 1) / CPT;
    const int nthr = groups >= 256 ? 256 : (int)((groups + 63) / 64 * 64);
    // runs of 32 steps (half the halo re-reads of 16) where they still give every SIMD 8 waves;
    // measured: config 5 (16 x 8192 x 1024) 32-step runs faster, config 3 (4 x 4096 x 4096) 16
    const int64_t waves32 = Bt * ((L + 31) / 32) * ((groups + nthr - 1) / nthr) * (nthr / 64);
    if (waves32 >= 32 * (int64_t)device_cus())
        launch_conv_tt<T, KW, CPT, VEC, 32>(Bt, L, Dm, groups, nthr, x, ldx, w, b, y, s);
    else
        launch_conv_tt<T, KW, CPT, VEC, 16>(Bt, L, Dm, groups, nthr, x, ldx, w, b, y, s);
}

template <typename T, int CPT, bool VEC>
void launch_conv_w(int64_t Bt, int64_t L, int64_t Dm, int64_t KW, const void* x, int64_t ldx,
                   const float* w, const float* b, void* y, hipStream_t s) {
    switch (KW) {
        case 1: launch_conv_k<T, 1, CPT, VEC>(Bt, L, Dm, x, ldx, w, b, y, s); break;
        case 2: launch_conv_k<T, 2, CPT, VEC>(Bt, L, Dm, x, ldx, w, b, y, s); break;
        case 3: launch_conv_k<T, 3, CPT, VEC>(Bt, L, Dm, x, ldx, w, b, y, s); break;
        default: launch_conv_k<T, 4, CPT, VEC>(Bt, L, Dm, x, ldx, w, b, y, s); break;
    }
}

template <typename T>
int launch_conv(int64_t Bt, int64_t L, int64_t Dm, int64_t KW, const void* x, int64_t ldx,
                const float* w, const float* b, void* y, hipStream_t s) {
    constexpr int CV = 16 / sizeof(T);  // channels in 16 bytes
    const bool vec = Dm % CV == 0 && ldx % CV == 0 && aligned(x, 16) && aligned(y, 16);
    if (vec)
        launch_conv_w<T, CV, true>(Bt, L, Dm, KW, x, ldx, w, b, y, s);
    else
        launch_conv_w<T, 4, false>(Bt, L, Dm, KW, x, ldx, w, b, y, s);
    HX_LAUNCH_CHECK();
    return HX_OK;
}

}  // namespace
}  // namespace hx

extern "C" int hx_conv1d_silu(int64_t batch, int64_t seqlen, int64_t dim, int64_t width,
                              int dtype, const void* x, int64_t ldx, const float* weight,
                              const float* bias, void* y, void* stream) {
    using namespace hx;
    HX_REQUIRE(batch >= 0 && seqlen >= 0 && dim >= 0, HX_ERR_INVALID_DIMENSION,
               "conv1d_silu: negative size");
    HX_REQUIRE(width >= 1 && width <= 4, HX_ERR_UNSUPPORTED, "conv1d_silu: width %lld (1..4)",
               (long long)width);
    HX_REQUIRE(dim % 4 == 0, HX_ERR_UNSUPPORTED, "conv1d_silu: dim %lld not a multiple of 4",
               (long long)dim);
    HX_REQUIRE(dtype == HX_F32 || dtype == HX_BF16, HX_ERR_DTYPE_MISMATCH, "conv1d_silu: dtype %d",
               dtype);
    if (batch == 0 || seqlen == 0 || dim == 0) return HX_OK;
    HX_REQUIRE(x && weight && y && ldx >= dim, HX_ERR_INVALID_INPUT,
               "conv1d_silu: x, weight, y required and ldx >= dim");
    HX_REQUIRE(seqlen < (1LL << 31) && dim <= 65535LL * 1024 && batch * ((seqlen + 15) / 16) < (1LL << 31),
               HX_ERR_UNSUPPORTED, "conv1d_silu: sizes beyond the launch grid");
    return dtype == HX_F32
               ? launch_conv<float>(batch, seqlen, dim, width, x, ldx, weight, bias, y, as_stream(stream))
               : launch_conv<uint16_t>(batch, seqlen, dim, width, x, ldx, weight, bias, y, as_stream(stream));
}

// Workspace layout (bf16 elements, M = batch*seqlen): xpart | z | xconv | dt | y  [M, d_inner]
// each, dt_lo [M, dt_rank], B [M, N], C [M, N]; every region 256-byte aligned. The layer entry
// points add a normalised-input region [M, d_model] in front.
namespace {
inline size_t align256(size_t b) { return (b + 255) / 256 * 256; }
}  // namespace

extern "C" size_t hx_mamba_block_workspace_size(int64_t batch, int64_t seqlen, int64_t d_inner,
                                                int64_t dt_rank, int64_t dstate) {
    const size_t M = (size_t)batch * seqlen;
    return 5 * align256(M * d_inner * 2) + align256(M * dt_rank * 2) + 2 * align256(M * dstate * 2);
}

extern "C" size_t hx_mamba_layer_workspace_size(int64_t batch, int64_t seqlen, int64_t d_model,
                                                int64_t d_inner, int64_t dt_rank, int64_t dstate) {
    return align256((size_t)batch * seqlen * d_model * 2) +
           hx_mamba_block_workspace_size(batch, seqlen, d_inner, dt_rank, dstate);
}

namespace hx {
int conv_state_capture(int64_t Bt, int64_t L, int64_t Dm, int K, const uint16_t* x, int64_t ldx,
                       float* state, hipStream_t s);
}  // namespace hx

extern "C" int hx_conv1d_step(int64_t batch, int64_t dim, int64_t width, int dtype, const void* x,
                              int64_t ldx, const float* weight, const float* bias, float* state,
                              void* y, void* stream);
extern "C" int hx_rmsnorm_fwd(int64_t rows, int64_t dim, const float* x, const float* weight,
                              float eps, int out_dtype, void* y, void* stream);

namespace {

struct BlockWeights {
    const void *w_in, *w_x, *w_dt, *w_out;
    const float *conv_w, *conv_b, *dt_bias, *A, *D;
};

// ----------------------------------------------------------------------------- fused decode
using namespace ::hx;

// The SSM half of one recurrent decode step of a layer, one block per sequence:
// the conv window step, x_proj (dt_lo | B | C), dt_proj, the state update with the D skip and
// the SiLU(z) gate — four launches of the unfused step in one, with every intermediate in LDS or
// registers instead of HBM. Rounding points are the unfused path's (xc, dt_lo, B, C and dt are
// rounded to bf16 where that path stores them), so the two differ only in the order of the
// x_proj and dt_proj sums.
//   pass 1: xc = silu(conv_b + sum_j conv_w[c][j] * window[j]) -> LDS; window advanced
//   x_proj: dt_lo | B | C = W_x . xc (J = dt_rank + 32 outputs)
//   pass 2: dt[c] = sum_r w_dt[c][r] * dt_lo[r]; dl = softplus(dt + dt_bias); per state n:
//           h = exp(dl * A[c][n]) * h + dl * xc * B[n]; y = (sum_n C[n] * h + D * xc) * silu(z)
// State [batch][d_inner][16] fp32 and conv window [batch][d_conv-1][d_inner] fp32 in place.
constexpr int kDecThreads = 512;   // the general kernel's block
constexpr int kRowThreads = 1024;  // the row kernel's block (16 waves)
// The state is read and written once per step: non-temporal (streaming) accesses keep its 16.8 MB
// per layer at config 5 from evicting the data the step reuses (the layer's weights, the
// activations the next launch reads) from the caches; the config-5 decode step 0.391 -> 0.348
// ms. (The conv window, 3 MB per layer, measured 2 us per step slower streamed so.)
typedef float hx_f32x4 __attribute__((ext_vector_type(4)));

__device__ inline float bf16r(float v) { return bf16_bits_to_f32(Storage<uint16_t>::round(v)); }

// Pass 2 of both decode kernels for one channel ch of the sequence b: k4 = lane % 4 holds states
// 4 k4 .. 4 k4 + 3 (hq, aq), dt_proj partial d over ranks 8 k4 .. 8 k4 + 7 (and beyond, looping)
// summed across the 4 lanes; the state is stored, and the lane with k4 = 0 stores y.
__device__ __attribute__((always_inline)) inline void decode_state_step(
    int64_t b, int d_inner, int ch, int k4, float d, float4 hq, float4 aq, const float (&bk)[4],
    const float (&ck)[4], const float* s_xc, const float* s_aux, const float* Dv,
    float* __restrict__ ssm_state, uint16_t* __restrict__ y) {
    d += __shfl_xor(d, 1, 64);
    d += __shfl_xor(d, 2, 64);
    if (ch >= d_inner) return;  // uniform per lane group
    float dl = bf16r(d) + s_aux[ch];
    dl = softplus(dl);
    const float uv = s_xc[ch];
    const float du = dl * uv;
    float h4[4] = {hq.x, hq.y, hq.z, hq.w};
    const float a4[4] = {aq.x, aq.y, aq.z, aq.w};
    float yy = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float ab = fast_exp2(dl * (a4[i] * kLog2e));
        h4[i] = fmaf(ab, h4[i], du * bk[i]);
        yy = fmaf(ck[i], h4[i], yy);
    }
    __builtin_nontemporal_store(hx_f32x4{h4[0], h4[1], h4[2], h4[3]},
                                reinterpret_cast<hx_f32x4*>(ssm_state + (b * (int64_t)d_inner + ch) * 16) + k4);
    yy += __shfl_xor(yy, 1, 64);
    yy += __shfl_xor(yy, 2, 64);
    if (k4 == 0) {
        if (Dv) yy = fmaf(s_aux[d_inner + ch], uv, yy);
        y[b * (int64_t)d_inner + ch] = Storage<uint16_t>::round(yy * silu(s_aux[2 * d_inner + ch]));
    }
}

// Row kernel, for d_inner <= 1024 and dt_rank <= 32: 16 waves (1024 threads), one conv channel
// per thread in pass 1, 4 x_proj outputs per wave, 4 pass-2 channels per thread, straight-line
// code. The step is a chain of dependent phases whose time is load latency, the CU's load port
// (every block reads all of W_x, A and W_dt, 256 KB at config 5) and the state's 16.8 MB read
// and write, so:
//   * x_proj: wave w owns outputs 4w .. 4w+3 over every channel; lane l sums channel chunks
//     8l + 512q (XV4: 16-byte loads, d_inner % 8 == 0) or 4l + 256q (8-byte loads), so each load
//     instruction reads 1 KB or 512 B of a W_x row contiguously; the 4 per-lane sums meet by a
//     register reduce-scatter (lane halves swapped, then 16-lane rows: lane bits 5, 4 pick the
//     output 2 b5 + b4) and a DPP sum over the 16 lanes of a row, with no LDS round trip;
//   * the loads are issued in the order the phases use them: pass-1 operands, W_x, then, once
//     the pass-1 operands are in (they would otherwise queue behind 16 MB of state reads), this
//     thread's state; A and the dt_proj rows (L2-hot) after the x_proj products; the conv-window
//     stores come last (stores under a branch would make the compiler's waits for W_x also wait
//     for the state).
// 16 waves instead of 8 (each loading half the W_x rows and half the state): config 5 decode
// 0.347 -> 0.332 ms per step.
template <int KC, bool XV4>
__global__ __launch_bounds__(kRowThreads) void ssm_decode_row_kernel(
    int d_inner, int dt_rank, const uint16_t* __restrict__ xpart, const uint16_t* __restrict__ z,
    const float* __restrict__ conv_w, const float* __restrict__ conv_b,
    float* __restrict__ conv_state, const uint16_t* __restrict__ w_x,
    const uint16_t* __restrict__ w_dt, const float* __restrict__ dt_bias,
    const float* __restrict__ A, const float* __restrict__ Dv, float* __restrict__ ssm_state,
    uint16_t* __restrict__ y) {
    extern __shared__ __attribute__((aligned(16))) float s_dec[];
    const int J = dt_rank + 32;
    float* s_xc = s_dec;
    float* s_aux = s_xc + d_inner;
    float* s_dbc = s_aux + 3 * d_inner;
    const int64_t b = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float* cst = conv_state + b * (int64_t)(KC - 1) * d_inner;

    const int c = tid < d_inner ? tid : d_inner - 1;
    const float p_x = bf16_bits_to_f32(xpart[b * (int64_t)d_inner + c]);
    const float p_z = bf16_bits_to_f32(z[b * (int64_t)d_inner + c]);
    float p_prev[KC > 1 ? KC - 1 : 1];
#pragma unroll
    for (int j = 0; j < KC - 1; ++j) p_prev[j] = cst[(int64_t)j * d_inner + c];
    float p_wk[KC];
    if constexpr (KC == 4) {
        const float4 w4 = reinterpret_cast<const float4*>(conv_w)[c];
        p_wk[0] = w4.x; p_wk[1] = w4.y; p_wk[2] = w4.z; p_wk[3] = w4.w;
    } else {
#pragma unroll
        for (int j = 0; j < KC; ++j) p_wk[j] = conv_w[c * KC + j];
    }
    const float p_cb = conv_b ? conv_b[c] : 0.0f;
    const float p_dtb = dt_bias ? dt_bias[c] : 0.0f;
    const float p_dv = Dv ? Dv[c] : 0.0f;
    constexpr int CW = XV4 ? 8 : 4;
    constexpr int NQ = 1024 / (64 * CW);
    using WChunk = std::conditional_t<XV4, uint4, uint2>;
    WChunk wx[4][NQ];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int jr = 4 * wave + r < J ? 4 * wave + r : J - 1;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int ch = CW * lane + 64 * CW * q < d_inner ? CW * lane + 64 * CW * q : 0;
            wx[r][q] = *reinterpret_cast<const WChunk*>(w_x + (int64_t)jr * d_inner + ch);
        }
    }
    float acc0 = p_cb;
#pragma unroll
    for (int j = 0; j < KC - 1; ++j) acc0 = fmaf(p_wk[j], p_prev[j], acc0);
    acc0 = fmaf(p_wk[KC - 1], p_x, acc0);
    const float xcv = bf16r(silu(acc0));
    asm volatile("" ::"v"(xcv) : "memory");
    constexpr int UC = 4;
    constexpr int CSTEP = kRowThreads / 4;
    const int k4 = tid & 3;
    float4 hq[UC];
#pragma unroll
    for (int u = 0; u < UC; ++u) {
        const int ch = (tid >> 2) + u * CSTEP < d_inner ? (tid >> 2) + u * CSTEP : d_inner - 1;
        const hx_f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const hx_f32x4*>(ssm_state + (b * (int64_t)d_inner + ch) * 16) + k4);
        hq[u] = make_float4(v[0], v[1], v[2], v[3]);
    }
    if (tid < d_inner) {
        s_xc[c] = xcv;
        s_aux[c] = p_dtb;
        s_aux[d_inner + c] = p_dv;
        s_aux[2 * d_inner + c] = p_z;
    }
    __syncthreads();

    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int c0 = CW * lane + 64 * CW * q;
        if (c0 < d_inner) {
            float xs[CW];
#pragma unroll
            for (int i = 0; i < CW; i += 4) {
                const float4 x4 = *reinterpret_cast<const float4*>(s_xc + c0 + i);
                xs[i] = x4.x; xs[i + 1] = x4.y; xs[i + 2] = x4.z; xs[i + 3] = x4.w;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                uint32_t wv[CW / 2];
                if constexpr (XV4) {
                    wv[0] = wx[r][q].x; wv[1] = wx[r][q].y; wv[2] = wx[r][q].z; wv[3] = wx[r][q].w;
                } else {
                    wv[0] = wx[r][q].x; wv[1] = wx[r][q].y;
                }
#pragma unroll
                for (int i = 0; i < CW / 2; ++i) {
                    acc[r] = fmaf(__uint_as_float(wv[i] << 16), xs[2 * i], acc[r]);
                    acc[r] = fmaf(__uint_as_float(wv[i] & 0xffff0000u), xs[2 * i + 1], acc[r]);
                }
            }
        }
    }
    const bool vec_dt = (dt_rank & 31) == 0;
    float4 aq[UC];
    uint4 wq[UC];
#pragma unroll
    for (int u = 0; u < UC; ++u) {
        const int ch = (tid >> 2) + u * CSTEP < d_inner ? (tid >> 2) + u * CSTEP : d_inner - 1;
        aq[u] = reinterpret_cast<const float4*>(A + (int64_t)ch * 16)[k4];
        if (vec_dt) wq[u] = *reinterpret_cast<const uint4*>(w_dt + (int64_t)ch * dt_rank + 8 * k4);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) { swap32(acc[i], acc[i + 2]); acc[i] += acc[i + 2]; }
    swap16(acc[0], acc[1]);
    acc[0] += acc[1];
    acc[0] += dpp<kDppXor1>(acc[0]);
    acc[0] += dpp<kDppXor2>(acc[0]);
    acc[0] += dpp<kDppHalfMirror>(acc[0]);
    acc[0] += dpp<kDppRor8>(acc[0]);
    {
        const int jrow = 4 * wave + 2 * ((lane >> 5) & 1) + ((lane >> 4) & 1);
        if ((lane & 15) == 0 && jrow < J) s_dbc[jrow] = bf16r(acc[0]);
    }
    __syncthreads();

    const float* dtlo = s_dbc;
    const float* Bn = s_dbc + dt_rank;
    const float* Cn = Bn + 16;
    float bk[4], ck[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { bk[i] = Bn[4 * k4 + i]; ck[i] = Cn[4 * k4 + i]; }
#pragma unroll
    for (int u = 0; u < UC; ++u) {
        const int ch = (tid >> 2) + u * CSTEP;
        float d = 0.0f;
        if (vec_dt) {
            const uint32_t ws[4] = {wq[u].x, wq[u].y, wq[u].z, wq[u].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                d = fmaf(__uint_as_float(ws[i] << 16), dtlo[8 * k4 + 2 * i], d);
                d = fmaf(__uint_as_float(ws[i] & 0xffff0000u), dtlo[8 * k4 + 2 * i + 1], d);
            }
        } else {
            const uint16_t* wr = w_dt + (int64_t)(ch < d_inner ? ch : d_inner - 1) * dt_rank;
            for (int r = k4; r < dt_rank; r += 4) d = fmaf(bf16_bits_to_f32(wr[r]), dtlo[r], d);
        }
        decode_state_step(b, d_inner, ch, k4, d, hq[u], aq[u], bk, ck, s_xc, s_aux, Dv, ssm_state, y);
    }
    if (tid < d_inner) {
#pragma unroll
        for (int j = 0; j + 1 < KC - 1; ++j) cst[(int64_t)j * d_inner + c] = p_prev[j + 1];
        if (KC > 1) cst[(int64_t)(KC - 2) * d_inner + c] = p_x;
    }
}

// General kernel (any d_inner % 4 == 0, any dt_rank): the same phases in loops.
//   pass 1: a thread owns channel pairs c = 2 tid + 1024 i
//   x_proj: 64 outputs at a time; thread (quad q = tid % 256, group g = tid / 256) sums
//           w_x[j][4q..4q+3] * xc over its channels for 32 outputs j, a butterfly reduce-scatter
//           leaves one output per lane pair, the 4 waves of a group add through LDS
//   pass 2: rounds of 8 channels per group of four lanes, each round's operands loaded at its
//           start
// One level of a butterfly reduce-scatter across the wave: K values in acc[0..K) become K / 2,
// the lanes with bit K set keeping the upper half of the pairwise sums (K a template argument so
// every index is a constant and acc stays in registers).
template <int K>
__device__ inline void rs_level(float* acc, int lane) {
    const bool up = (lane & K) != 0;
#pragma unroll
    for (int i = 0; i < K / 2; ++i) {
        const float send = up ? acc[i] : acc[i + K / 2];
        const float keep = up ? acc[i + K / 2] : acc[i];
        acc[i] = keep + __shfl_xor(send, K, 64);
    }
}

template <int KC>
__global__ __launch_bounds__(kDecThreads) void ssm_decode_kernel(
    int d_inner, int dt_rank, const uint16_t* __restrict__ xpart, const uint16_t* __restrict__ z,
    const float* __restrict__ conv_w, const float* __restrict__ conv_b,
    float* __restrict__ conv_state, const uint16_t* __restrict__ w_x,
    const uint16_t* __restrict__ w_dt, const float* __restrict__ dt_bias,
    const float* __restrict__ A, const float* __restrict__ Dv, float* __restrict__ ssm_state,
    uint16_t* __restrict__ y) {
    extern __shared__ __attribute__((aligned(16))) float s_dec[];
    const int J = dt_rank + 32;
    const int Jp = (J + 63) / 64 * 64;
    float* s_xc = s_dec;                 // [d_inner]
    float* s_aux = s_xc + d_inner;       // [3][d_inner]: dt_bias, D, z (staged in pass 1)
    float* s_dbc = s_aux + 3 * d_inner;  // [Jp]: dt_lo | B | C, bf16-rounded
    float* s_red = s_dbc + Jp;           // [8][32]: x_proj wave sums
    const int64_t b = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint16_t* xr = xpart + b * (int64_t)d_inner;
    const uint16_t* zr = z + b * (int64_t)d_inner;
    float* cst = conv_state + b * (int64_t)(KC - 1) * d_inner;

    // pass 1: conv window step
    for (int c = 2 * tid; c < d_inner; c += 2 * kDecThreads) {
        const uint32_t p_xw = *reinterpret_cast<const uint32_t*>(xr + c);
        const uint32_t p_zw = *reinterpret_cast<const uint32_t*>(zr + c);
        const float xv[2] = {__uint_as_float(p_xw << 16), __uint_as_float(p_xw & 0xffff0000u)};
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            float acc = conv_b ? conv_b[c + e] : 0.0f;
#pragma unroll
            for (int j = 0; j < KC - 1; ++j) acc = fmaf(conv_w[(c + e) * KC + j], cst[(int64_t)j * d_inner + c + e], acc);
            acc = fmaf(conv_w[(c + e) * KC + KC - 1], xv[e], acc);
#pragma unroll
            for (int j = 0; j + 1 < KC - 1; ++j) cst[(int64_t)j * d_inner + c + e] = cst[(int64_t)(j + 1) * d_inner + c + e];
            if (KC > 1) cst[(int64_t)(KC - 2) * d_inner + c + e] = xv[e];
            s_xc[c + e] = bf16r(silu(acc));
            s_aux[c + e] = dt_bias ? dt_bias[c + e] : 0.0f;
            s_aux[d_inner + c + e] = Dv ? Dv[c + e] : 0.0f;
        }
        s_aux[2 * d_inner + c] = __uint_as_float(p_zw << 16);
        s_aux[2 * d_inner + c + 1] = __uint_as_float(p_zw & 0xffff0000u);
    }
    __syncthreads();

    // x_proj: 64 outputs at a time
    const int xq = tid & 255, xg = tid >> 8;
    const int jj_lane = (((lane >> 5) & 1) << 4) | (((lane >> 4) & 1) << 3) | (((lane >> 3) & 1) << 2) |
                        (((lane >> 2) & 1) << 1) | ((lane >> 1) & 1);
    for (int j0 = 0; j0 < J; j0 += 64) {
        float acc[32];
#pragma unroll
        for (int jj = 0; jj < 32; ++jj) acc[jj] = 0.0f;
        for (int cb = 0; cb < d_inner; cb += 1024) {
            const int c = cb + 4 * xq;
            if (c < d_inner) {
                const float4 x4 = *reinterpret_cast<const float4*>(s_xc + c);
#pragma unroll
                for (int jj = 0; jj < 32; ++jj) {
                    const int jr = j0 + 32 * xg + jj < J ? j0 + 32 * xg + jj : J - 1;  // clamped: never stored
                    const uint2 w = *reinterpret_cast<const uint2*>(w_x + (int64_t)jr * d_inner + c);
                    acc[jj] = fmaf(__uint_as_float(w.x << 16), x4.x, acc[jj]);
                    acc[jj] = fmaf(__uint_as_float(w.x & 0xffff0000u), x4.y, acc[jj]);
                    acc[jj] = fmaf(__uint_as_float(w.y << 16), x4.z, acc[jj]);
                    acc[jj] = fmaf(__uint_as_float(w.y & 0xffff0000u), x4.w, acc[jj]);
                }
            }
        }
        // butterfly reduce-scatter across the wave: the lane pair (2i, 2i + 1) ends with the
        // wave's sum for output jj_lane
        rs_level<32>(acc, lane);
        rs_level<16>(acc, lane);
        rs_level<8>(acc, lane);
        rs_level<4>(acc, lane);
        rs_level<2>(acc, lane);
        acc[0] += __shfl_xor(acc[0], 1, 64);
        if ((lane & 1) == 0) s_red[wave * 32 + jj_lane] = acc[0];
        __syncthreads();
        if (tid < 64 && j0 + tid < J) {
            const int g = tid >> 5, jj = tid & 31;
            float t = s_red[(4 * g) * 32 + jj];
#pragma unroll
            for (int w = 1; w < 4; ++w) t += s_red[(4 * g + w) * 32 + jj];
            s_dbc[j0 + tid] = bf16r(t);
        }
        __syncthreads();
    }

    // pass 2: dt_proj, state update, skip and gate, in rounds of UC channels per lane group
    constexpr int UC = 8;
    constexpr int CSTEP = kDecThreads / 4;
    const int k4 = tid & 3;
    const bool vec_dt = (dt_rank & 31) == 0;
    const float* dtlo = s_dbc;
    const float* Bn = s_dbc + dt_rank;
    const float* Cn = Bn + 16;
    float bk[4], ck[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) { bk[i] = Bn[4 * k4 + i]; ck[i] = Cn[4 * k4 + i]; }
    for (int ch0 = tid >> 2; ch0 < d_inner; ch0 += UC * CSTEP) {
        float4 hq[UC], aq[UC];
#pragma unroll
        for (int u = 0; u < UC; ++u) {
            const int ch = ch0 + u * CSTEP < d_inner ? ch0 + u * CSTEP : d_inner - 1;  // clamped: unused
            const hx_f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const hx_f32x4*>(ssm_state + (b * (int64_t)d_inner + ch) * 16) + k4);
            hq[u] = make_float4(v[0], v[1], v[2], v[3]);
            aq[u] = reinterpret_cast<const float4*>(A + (int64_t)ch * 16)[k4];
        }
#pragma unroll
        for (int u = 0; u < UC; ++u) {
            const int ch = ch0 + u * CSTEP;
            const int chc = ch < d_inner ? ch : d_inner - 1;
            const uint16_t* wr = w_dt + (int64_t)chc * dt_rank;
            float d = 0.0f;
            if (vec_dt) {
                for (int r0 = 8 * k4; r0 < dt_rank; r0 += 32) {
                    const uint4 wv = *reinterpret_cast<const uint4*>(wr + r0);
                    const uint32_t w4[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        d = fmaf(__uint_as_float(w4[i] << 16), dtlo[r0 + 2 * i], d);
                        d = fmaf(__uint_as_float(w4[i] & 0xffff0000u), dtlo[r0 + 2 * i + 1], d);
                    }
                }
            } else {
                for (int r = k4; r < dt_rank; r += 4) d = fmaf(bf16_bits_to_f32(wr[r]), dtlo[r], d);
            }
            decode_state_step(b, d_inner, ch, k4, d, hq[u], aq[u], bk, ck, s_xc, s_aux, Dv, ssm_state, y);
        }
    }
}

size_t ssm_decode_lds(int64_t d_inner, int64_t dt_rank) {
    const int64_t J = dt_rank + 32, Jp = (J + 63) / 64 * 64;
    return (size_t)(4 * d_inner + Jp + 8 * 32) * sizeof(float);
}

int launch_ssm_decode(int64_t batch, int64_t d_inner, int64_t dt_rank, int64_t d_conv,
                      const void* xpart, const void* z, const float* conv_w, const float* conv_b,
                      float* conv_state, const void* w_x, const void* w_dt, const float* dt_bias,
                      const float* A, const float* D, float* ssm_state, void* y, void* stream) {
    HX_REQUIRE(batch <= 0x7fffffff, HX_ERR_UNSUPPORTED, "mamba_layer_decode: batch %lld too large",
               (long long)batch);
    const bool row = d_inner <= kRowThreads && dt_rank <= 32;
    const bool xv4 = d_inner % 8 == 0 && aligned(w_x, 16);  // 16-byte W_x chunks
    const size_t lds = row ? (size_t)(4 * d_inner + 64) * sizeof(float) : ssm_decode_lds(d_inner, dt_rank);
    auto go = [&](auto kern, int threads) {
        if (lds > 64 * 1024 &&
            hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return set_error(HX_ERR_UNSUPPORTED, "mamba_layer_decode: %zu bytes of LDS unavailable", lds);
        hipLaunchKernelGGL(kern, dim3((unsigned)batch), dim3(threads), lds, as_stream(stream),
                           (int)d_inner, (int)dt_rank, (const uint16_t*)xpart, (const uint16_t*)z,
                           conv_w, conv_b, conv_state, (const uint16_t*)w_x, (const uint16_t*)w_dt,
                           dt_bias, A, D, ssm_state, (uint16_t*)y);
        HX_LAUNCH_CHECK();
        return (int)HX_OK;
    };
    if (row && xv4) {
        switch (d_conv) {
            case 1: return go(ssm_decode_row_kernel<1, true>, kRowThreads);
            case 2: return go(ssm_decode_row_kernel<2, true>, kRowThreads);
            case 3: return go(ssm_decode_row_kernel<3, true>, kRowThreads);
            default: return go(ssm_decode_row_kernel<4, true>, kRowThreads);
        }
    }
    if (row) {
        switch (d_conv) {
            case 1: return go(ssm_decode_row_kernel<1, false>, kRowThreads);
            case 2: return go(ssm_decode_row_kernel<2, false>, kRowThreads);
            case 3: return go(ssm_decode_row_kernel<3, false>, kRowThreads);
            default: return go(ssm_decode_row_kernel<4, false>, kRowThreads);
        }
    }
    switch (d_conv) {
        case 1: return go(ssm_decode_kernel<1>, kDecThreads);
        case 2: return go(ssm_decode_kernel<2>, kDecThreads);
        case 3: return go(ssm_decode_kernel<3>, kDecThreads);
        default: return go(ssm_decode_kernel<4>, kDecThreads);
    }
}

struct BlockBufs {
    void *xpart, *z, *xconv, *dt, *y, *dtlo, *B, *C;
};

BlockBufs carve(char* p, int64_t M, int64_t d_inner, int64_t dt_rank, int64_t dstate) {
    auto take = [&](size_t bytes) { void* r = p; p += align256(bytes); return r; };
    BlockBufs b;
    b.xpart = take(M * d_inner * 2);
    b.z = take(M * d_inner * 2);
    b.xconv = take(M * d_inner * 2);
    b.dt = take(M * d_inner * 2);
    b.y = take(M * d_inner * 2);
    b.dtlo = take(M * dt_rank * 2);
    b.B = take(M * dstate * 2);
    b.C = take(M * dstate * 2);
    return b;
}

int check_block_args(int64_t batch, int64_t seqlen, int64_t d_model, int64_t d_inner,
                     int64_t dstate, int64_t dt_rank, int64_t d_conv, const BlockWeights& w) {
    using namespace hx;
    HX_REQUIRE(batch >= 0 && seqlen >= 0 && d_model > 0 && d_inner > 0 && dt_rank > 0,
               HX_ERR_INVALID_DIMENSION, "mamba_block: bad sizes");
    HX_REQUIRE(dstate == 16, HX_ERR_UNSUPPORTED, "mamba_block: dstate %lld (16 supported)",
               (long long)dstate);
    HX_REQUIRE(d_inner % 4 == 0, HX_ERR_UNSUPPORTED, "mamba_block: d_inner %lld not a multiple of 4",
               (long long)d_inner);
    HX_REQUIRE(d_conv >= 1 && d_conv <= 4, HX_ERR_UNSUPPORTED, "mamba_block: d_conv %lld (1..4)",
               (long long)d_conv);
    HX_REQUIRE(w.w_in && w.conv_w && w.w_x && w.w_dt && w.A && w.w_out, HX_ERR_INVALID_INPUT,
               "mamba_block: a required weight pointer is NULL");
    return HX_OK;
}

// The block on bf16 input x [M, d_model]: writes out (bf16, or fp32 accumulated into when
// accumulate) and optionally the scan's last state and the conv window for decode.
int block_core(int64_t batch, int64_t seqlen, int64_t d_model, int64_t d_inner, int64_t dstate,
               int64_t dt_rank, int64_t d_conv, const void* x, const BlockWeights& w, void* out,
               int out_dtype, bool accumulate, float* last_state, float* conv_state,
               const BlockBufs& b, void* stream) {
    const int64_t M = batch * seqlen;
    int rc;
    // in_proj: [M, d_model] x [2*d_inner, d_model]^T -> xpart | z
    if ((rc = hx_gemm_bf16(M, 2 * d_inner, d_model, x, d_model, w.w_in, d_model, nullptr, 0,
                           HX_BF16, b.xpart, d_inner, d_inner, b.z, d_inner, 2 * d_inner, nullptr,
                           0, stream)))
        return rc;
    if (conv_state &&
        (rc = hx::conv_state_capture(batch, seqlen, d_inner, (int)d_conv, (const uint16_t*)b.xpart,
                                     d_inner, conv_state, hx::as_stream(stream))))
        return rc;
    if ((rc = hx_conv1d_silu(batch, seqlen, d_inner, d_conv, HX_BF16, b.xpart, d_inner, w.conv_w,
                             w.conv_b, b.xconv, stream)))
        return rc;
    // x_proj: [M, d_inner] x [dt_rank + 2N, d_inner]^T -> dt_lo | B | C. Narrow and long (config 3:
    // N 160, K 4096): hx_gemm_bf16's narrow kernel streams xconv once with every column in the
    // block. Where that kernel does not apply, a long K is split four ways with the fp32 partials
    // in the in_proj x region, which the conv has consumed by now. Either choice depends on the
    // weight shape only, so every batch size and sequence length gets the same arithmetic per token.
    const int64_t nx = dt_rank + 2 * dstate;
    const int splits = (!hx::gemm_narrow_auto(nx, d_inner) && d_inner >= 2048 && d_inner % 256 == 0 &&
                        nx <= 256 && 4 * nx * 2 <= d_inner) ? 4 : 1;
    rc = splits > 1 ? hx_gemm_bf16_splitk(M, nx, d_inner, b.xconv, d_inner, w.w_x, d_inner, nullptr, 0,
                                          HX_BF16, b.dtlo, dt_rank, dt_rank, b.B, dstate, dt_rank + dstate,
                                          b.C, dstate, splits, b.xpart, (size_t)M * d_inner * 2, stream)
                    : hx_gemm_bf16(M, nx, d_inner, b.xconv, d_inner, w.w_x, d_inner, nullptr, 0, HX_BF16,
                                   b.dtlo, dt_rank, dt_rank, b.B, dstate, dt_rank + dstate, b.C, dstate,
                                   stream);
    if (rc) return rc;
    // the in_proj x region, consumed by the conv, holds the end states of a sequence cut into segments
    if (hx::scan_variant_is_auto() && hx::scan_dtproj_ok(batch, seqlen, d_inner, dt_rank)) {
        // dt_proj inside the scan: each 16-step chunk's dt tile is dt_lo . w_dt^T on the matrix
        // core, rounded to bf16 as the separate product stores it (dt_bias is added after)
        rc = hx::scan_fwd_dtproj(batch, seqlen, d_inner, (const uint16_t*)b.xconv, (const uint16_t*)b.dtlo,
                                 dt_rank, (const uint16_t*)w.w_dt, w.A, (const uint16_t*)b.B,
                                 (const uint16_t*)b.C, w.D, (const uint16_t*)b.z, w.dt_bias,
                                 (uint16_t*)b.y, last_state, b.xpart, (size_t)M * d_inner * 2,
                                 hx::as_stream(stream));
        if (rc) return rc;
    } else {
        // dt_proj: [M, dt_rank] x [d_inner, dt_rank]^T -> dt (dt_bias is added inside the scan)
        if ((rc = hx_gemm_bf16(M, d_inner, dt_rank, b.dtlo, dt_rank, w.w_dt, dt_rank, nullptr, 0,
                               HX_BF16, b.dt, d_inner, d_inner, nullptr, 0, d_inner, nullptr, 0, stream)))
            return rc;
        if ((rc = hx::scan_fwd_scratch(batch, seqlen, d_inner, (const uint16_t*)b.xconv, (const uint16_t*)b.dt,
                                       w.A, (const uint16_t*)b.B, (const uint16_t*)b.C, w.D,
                                       (const uint16_t*)b.z, w.dt_bias, (uint16_t*)b.y, last_state, b.xpart,
                                       (size_t)M * d_inner * 2, hx::as_stream(stream))))
            return rc;
    }
    // out_proj: [M, d_inner] x [d_model, d_inner]^T -> out (+= out when accumulating)
    return hx_gemm_bf16(M, d_model, d_inner, b.y, d_inner, w.w_out, d_inner, nullptr,
                        accumulate ? 2 : 0, out_dtype, out, d_model, d_model, nullptr, 0, d_model,
                        nullptr, 0, stream);
}

}  // namespace

extern "C" int hx_mamba_block_fwd(int64_t batch, int64_t seqlen, int64_t d_model, int64_t d_inner,
                                  int64_t dstate, int64_t dt_rank, int64_t d_conv,
                                  const void* x, const void* w_in, const float* conv_w,
                                  const float* conv_b, const void* w_x, const void* w_dt,
                                  const float* dt_bias, const float* A, const float* D,
                                  const void* w_out, void* out, void* workspace,
                                  size_t workspace_bytes, void* stream) {
    using namespace hx;
    const BlockWeights w{w_in, w_x, w_dt, w_out, conv_w, conv_b, dt_bias, A, D};
    int rc;
    if ((rc = check_block_args(batch, seqlen, d_model, d_inner, dstate, dt_rank, d_conv, w))) return rc;
    if (batch == 0 || seqlen == 0) return HX_OK;
    HX_REQUIRE(x && out && workspace, HX_ERR_INVALID_INPUT, "mamba_block: x, out, workspace required");
    const size_t need = hx_mamba_block_workspace_size(batch, seqlen, d_inner, dt_rank, dstate);
    HX_REQUIRE(workspace_bytes >= need, HX_ERR_INVALID_INPUT,
               "mamba_block: workspace %zu bytes < %zu required", workspace_bytes, need);
    const BlockBufs b = carve((char*)workspace, batch * seqlen, d_inner, dt_rank, dstate);
    return block_core(batch, seqlen, d_model, d_inner, dstate, dt_rank, d_conv, x, w, out, HX_BF16,
                      false, nullptr, nullptr, b, stream);
}

extern "C" int hx_mamba_layer_fwd(int64_t batch, int64_t seqlen, int64_t d_model, int64_t d_inner,
                                  int64_t dstate, int64_t dt_rank, int64_t d_conv, float* resid,
                                  const float* norm_w, float eps, const void* w_in,
                                  const float* conv_w, const float* conv_b, const void* w_x,
                                  const void* w_dt, const float* dt_bias, const float* A,
                                  const float* D, const void* w_out, float* ssm_state,
                                  float* conv_state, void* workspace, size_t workspace_bytes,
                                  void* stream) {
    using namespace hx;
    const BlockWeights w{w_in, w_x, w_dt, w_out, conv_w, conv_b, dt_bias, A, D};
    int rc;
    if ((rc = check_block_args(batch, seqlen, d_model, d_inner, dstate, dt_rank, d_conv, w))) return rc;
    if (batch == 0 || seqlen == 0) return HX_OK;
    HX_REQUIRE(resid && norm_w && workspace, HX_ERR_INVALID_INPUT,
               "mamba_layer: resid, norm_w, workspace required");
    const int64_t M = batch * seqlen;
    const size_t need = hx_mamba_layer_workspace_size(batch, seqlen, d_model, d_inner, dt_rank, dstate);
    HX_REQUIRE(workspace_bytes >= need, HX_ERR_INVALID_INPUT,
               "mamba_layer: workspace %zu bytes < %zu required", workspace_bytes, need);
    char* p = (char*)workspace;
    void* xn = p;
    const BlockBufs b = carve(p + align256((size_t)M * d_model * 2), M, d_inner, dt_rank, dstate);
    if ((rc = hx_rmsnorm_fwd(M, d_model, resid, norm_w, eps, HX_BF16, xn, stream))) return rc;
    return block_core(batch, seqlen, d_model, d_inner, dstate, dt_rank, d_conv, xn, w, resid, HX_F32,
                      true, ssm_state, conv_state, b, stream);
}

extern "C" int hx_mamba_layer_decode(int64_t batch, int64_t d_model, int64_t d_inner,
                                     int64_t dstate, int64_t dt_rank, int64_t d_conv, float* resid,
                                     const float* norm_w, float eps, const void* w_in,
                                     const float* conv_w, const float* conv_b, const void* w_x,
                                     const void* w_dt, const float* dt_bias, const float* A,
                                     const float* D, const void* w_out, float* ssm_state,
                                     float* conv_state, void* workspace, size_t workspace_bytes,
                                     void* stream) {
    using namespace hx;
    const BlockWeights w{w_in, w_x, w_dt, w_out, conv_w, conv_b, dt_bias, A, D};
    int rc;
    if ((rc = check_block_args(batch, 1, d_model, d_inner, dstate, dt_rank, d_conv, w))) return rc;
    if (batch == 0) return HX_OK;
    HX_REQUIRE(resid && norm_w && ssm_state && workspace && (d_conv == 1 || conv_state),
               HX_ERR_INVALID_INPUT, "mamba_layer_decode: resid, norm_w, ssm_state, conv_state, "
                                     "workspace required");
    const size_t need = hx_mamba_layer_workspace_size(batch, 1, d_model, d_inner, dt_rank, dstate);
    HX_REQUIRE(workspace_bytes >= need, HX_ERR_INVALID_INPUT,
               "mamba_layer_decode: workspace %zu bytes < %zu required", workspace_bytes, need);
    char* p = (char*)workspace;
    void* xn = p;
    const BlockBufs b = carve(p + align256((size_t)batch * d_model * 2), batch, d_inner, dt_rank, dstate);
    // the pre-norm inside in_proj's operand load where the small-M GEMM holds whole rows
    // (d_model <= 512: config 5's decode), else RMSNorm to bf16 then in_proj
    if (gemm_rmsnorm_small_ok(batch, 2 * d_inner, d_model, resid, d_model, norm_w, w.w_in, d_model)) {
        if ((rc = gemm_rmsnorm_small(batch, 2 * d_inner, d_model, resid, d_model, norm_w, eps, w.w_in,
                                     d_model, HX_BF16, b.xpart, d_inner, d_inner, b.z, d_inner,
                                     2 * d_inner, nullptr, 0, as_stream(stream))))
            return rc;
    } else {
        if ((rc = hx_rmsnorm_fwd(batch, d_model, resid, norm_w, eps, HX_BF16, xn, stream))) return rc;
        if ((rc = hx_gemm_bf16(batch, 2 * d_inner, d_model, xn, d_model, w.w_in, d_model, nullptr, 0,
                               HX_BF16, b.xpart, d_inner, d_inner, b.z, d_inner, 2 * d_inner,
                               nullptr, 0, stream)))
            return rc;
    }
    // conv step, x_proj, dt_proj, state update and gate in one launch (ssm_decode_kernel)
    HX_REQUIRE(aligned(ssm_state, 16) && aligned(w.A, 16) && aligned(w.w_x, 8) &&
                   aligned(w.w_dt, 16) && aligned(w.conv_w, 16),
               HX_ERR_INVALID_INPUT,
               "mamba_layer_decode: ssm_state, A, w_dt and conv_w must be 16-byte aligned, w_x 8-byte");
    if ((rc = launch_ssm_decode(batch, d_inner, dt_rank, d_conv, b.xpart, b.z, w.conv_w, w.conv_b,
                                conv_state, w.w_x, w.w_dt, w.dt_bias, w.A, w.D, ssm_state, b.y,
                                stream)))
        return rc;
    return hx_gemm_bf16(batch, d_model, d_inner, b.y, d_inner, w.w_out, d_inner, nullptr, 2, HX_F32,
                        resid, d_model, d_model, nullptr, 0, d_model, nullptr, 0, stream);
}
