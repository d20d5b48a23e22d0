// hx_scan_ps.h — the selective scan with paired state and element waves (included by hx_scan.hip).
#pragma once
#include "hx_common.h"
#include "hx_wave.h"

namespace hx {
namespace {

constexpr int kBufRsrcWord3 = 0x00020000;  // gfx9 raw buffer: 32-bit data format, no swizzle

struct PsArgs {
    int64_t L, Dm;
    int ntiles, Bt, nseg;
    int seg_len;                 // a multiple of 16; the last segment may be shorter
    int drop;                    // END_ONLY: stop at kDecayDrop
    const float *A, *D, *bias, *init;
    float* last;
    float4 *hend, *decay;        // [nseg - 1][Bt][ntiles][4][64], nseg > 1
    const uint16_t *dtlo, *wdt;  // fused dt projection
};

__device__ inline float row_load(__amdgpu_buffer_rsrc_t rs, uint32_t lane_off, uint32_t row_off, const float*) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, lane_off, row_off, 0));
}
__device__ inline uint16_t row_load(__amdgpu_buffer_rsrc_t rs, uint32_t lane_off, uint32_t row_off, const uint16_t*) {
    return __builtin_amdgcn_raw_buffer_load_b16(rs, lane_off, row_off, 0);
}
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ inline float4 row_load4(__amdgpu_buffer_rsrc_t rs, uint32_t off, const float*) {
    return __builtin_bit_cast(float4, (u32x4_t)__builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
}
__device__ inline uint2 row_load4(__amdgpu_buffer_rsrc_t rs, uint32_t off, const uint16_t*) {
    return __builtin_bit_cast(uint2, (u32x2_t)__builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
}
__device__ inline void row_store(float v, __amdgpu_buffer_rsrc_t rs, uint32_t lane_off, uint32_t row_off, float*) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rs, lane_off, row_off, 0);
}
__device__ inline void row_store(float v, __amdgpu_buffer_rsrc_t rs, uint32_t lane_off, uint32_t row_off, uint16_t*) {
    __builtin_amdgcn_raw_buffer_store_b16(Storage<uint16_t>::round(v), rs, lane_off, row_off, 0);
}
__device__ inline float to_f32(float v) { return v; }
__device__ inline float to_f32(uint16_t v) { return bf16_bits_to_f32(v); }

// Selective scan, dstate 16: a block of 8 waves owns 64 channels of one batch row (or of one time
// segment of it) and its waves work in pairs on one SIMD each (waves w and w + 4):
//   * state wave w runs the recurrence and readout of 16 channels x 16 states in the layout of
//     scan_wave3_kernel (lane (c, r): channel c, states 4r..4r+3). Its inputs B[t][n] * (dt*u)[t][d]
//     are outer products over (state, channel), so they come from the matrix core, 4 steps x 16
//     states x 16 channels per v_mfma_f32_16x16x1_4b_f32, whose result layout is the lane layout;
//     K is 1, so each is one exactly rounded product as a multiply would give. C reaches the readout
//     multiplies by DPP row_newbcast. That leaves 4 VALU instructions per state and step: dt*A, exp2,
//     the recurrence's FMA and the readout's.
//   * element wave w does the per-(step, channel) work of steps 4w..4w+3 of every 16-step chunk for
//     the 64 channels, lane = channel: whole-row loads three chunks ahead, softplus, dt*u, SiLU(z),
//     and after the recurrence the sum of the four lane rows' readouts, D*u, the gate and the store.
//     The dt tile of a fused dt projection (DTPK > 0: rank 32 DTPK, bf16) is formed here too, by
//     v_mfma_f32_16x16x32_bf16, and rounded to bf16 as a stored dt would be.
// They hand over through LDS, one barrier per chunk: in iteration i the state waves run chunk i and
// read ahead into i + 1, the element waves finish i - 1 and prepare i + 2.
// Every operation is scan_wave3_kernel's in its order, so results match it bit for bit.
//
// Bound: instruction issue. The state wave is the critical path, 18 instructions a step at the 5-6
// cycles (10 for exp2) that one wave takes for each; the SIMD's VALU is 73-77% busy over both waves with one
// block per CU (88% with two), 25% fewer VALU cycles than scan_ws2_kernel at the same shape. Measured (gfx950):
// 16 x 8192 x 1024 bf16 with rank 32 666 -> 540 us, 4 x 4096 x 4096 with rank 128 338 -> 285 us (scan_wave3_kernel,
// one wave a SIMD); 1 x 65536 x 2048 fp32, segmented, 695 -> 603 us. Splitting the states over two waves (three waves
// a SIMD) was slower, 600 us at the first shape: readouts and hand-over double. The state waves'
// priority gives 2-3%.
//
// END_ONLY: a segment's end state from a zero entry state and its decay, for the segments that follow;
// it walks backwards from the end, adding exp2(S) * B*dt*u with S the sum of A*dt from there to the end
// (a sum per state, one FMA each: A = -inf gives S = -inf, where A times a sum of dt would be NaN at the last
// step, whose sum is 0), and stops at the first 48-step round at which every state of the block's channels has decayed
// below 2^-32 (kDecayDrop): what is left out is 2^-8 of the fp32 rounding of the state there. Such a
// segment publishes decay 0. Below 4096 steps, in segments below 1024, in the Mamba block, and for dims that are no
// multiple of 4 or rows that are not 16-byte aligned (drop = 0) it walks its whole segment instead: a NaN, an infinity or
// an outlier reaches everything after it, as in the uncut scan, and segments of a few hundred steps hardly
// ever decay that far. The output pass chains the segments before its own itself.
// Sizes: byte offsets inside a segment below 2^31, in B and C (16 wide) too.
template <typename T, bool HAS_Z, bool SOFTPLUS, bool END_ONLY, int DTPK>
__global__ __launch_bounds__(512, 4) void scan_ps_kernel(
    const PsArgs a, const T* __restrict__ u, const T* __restrict__ delta, const T* __restrict__ Bm,
    const T* __restrict__ Cm, const T* __restrict__ z, T* __restrict__ out) {
    constexpr int NS = 16, TCH = 16, NB = 3;
    constexpr bool USE_Z = HAS_Z && !END_ONLY;
    constexpr bool DTP = DTPK > 0;
    constexpr int NKB = DTP ? DTPK : 1;
    typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
    typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
    typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
    // chunk buffers: [step / 4][channel] float4 of 4 steps for dt and dt*u; readouts per DPP row;
    // the dt tile of the fused projection (bf16); END_ONLY: stop votes
    using Row = float4[4][64];
    using Part = float4[4][4][64];
    using Raw = uint2[4][64];
    using Vote = int[4];
    constexpr size_t kRow = NB * sizeof(Row), kPart = END_ONLY ? 0 : NB * sizeof(Part), kRaw = DTP ? NB * sizeof(Raw) : 0;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * kRow + kPart + kRaw + (END_ONLY ? sizeof(Vote) : 0)];
    Row* const s_dt = reinterpret_cast<Row*>(smem);
    Row* const s_du = reinterpret_cast<Row*>(smem + kRow);
    Part* const s_part = reinterpret_cast<Part*>(smem + 2 * kRow);
    Raw* const s_raw = reinterpret_cast<Raw*>(smem + 2 * kRow + kPart);
    Vote* const s_vote = reinterpret_cast<Vote*>(smem + 2 * kRow + kPart + kRaw);

    const int nblk = gridDim.x;
    int id = blockIdx.x;
    if ((nblk & 7) == 0) id = (id & 7) * (nblk >> 3) + (id >> 3);  // XCD-aware order
    const int tile = id % a.ntiles;
    const int b = (id / a.ntiles) % a.Bt;
    const int seg = id / a.ntiles / a.Bt;
    const int L = (int)a.L;
    const int tbeg = seg * a.seg_len;
    const int len = L - tbeg < a.seg_len ? L - tbeg : a.seg_len;
    const int nch = (len + TCH - 1) / TCH;  // END_ONLY segments are whole chunks
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w = wave & 3;
    const int r = lane >> 4, c = lane & 15;  // DPP row, lane of the row
    const int64_t Dm = a.Dm;
    const int64_t seq0 = (int64_t)b * L + tbeg;  // the segment's first row
    // first step (inside the segment) of the i-th chunk walked: forwards, or (END_ONLY) backwards;
    // past the last one it repeats (prefetches run past the end)
    auto chunk_t = [&](int i) {
        const int ii = i < nch ? i : nch - 1;
        return (END_ONLY ? nch - 1 - ii : ii) * TCH;
    };
    auto stop_vote = [&]() {
        int any = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) any |= s_vote[0][i];
        return __builtin_amdgcn_readfirstlane(any) == 0;
    };

    // Walks the chunks: whole rounds of NB, so that nothing in a round depends on a branch (a skipped
    // chunk would merge the load rings' registers, and the copies would wait for loads in flight),
    // then the remainder, whose length it returns. END_ONLY stops after a round at whose end the
    // state waves voted to.
    auto walk = [&](auto& body, auto stopped) __attribute__((always_inline)) {
        int i = 0;
        for (; i + NB <= nch; i += NB) {
            StepLoop<NB>::run([&](auto kc) __attribute__((always_inline)) { body(kc, i + decltype(kc)::value); });
            if constexpr (END_ONLY) {
                if (a.drop && stop_vote()) {
                    stopped(i + NB);
                    return 0;
                }
            }
        }
        if (i < nch) {
            body(std::integral_constant<int, 0>{}, i);
            if (i + 1 < nch) {
                body(std::integral_constant<int, 1>{}, i + 1);
                return 2;
            }
            return 1;
        }
        return 0;
    };

    if (wave < 4) {
        // ------------------------------------------------------------- state wave: 16 channels
        __builtin_amdgcn_s_setprio(2);  // the serial chain first
        const int64_t d = (int64_t)tile * 64 + 16 * w + c;
        const bool dvalid = d < Dm;
        const int64_t dc = dvalid ? d : Dm - 1;
        float A2[4], h[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < 4; ++k) A2[k] = a.A[dc * NS + 4 * r + k] * kLog2e;
        const int64_t sidx = ((int64_t)b * Dm + dc) * NS + 4 * r;
        const int64_t slot = (((int64_t)b * a.ntiles + tile) * 4 + w) * 64 + lane;
        const int64_t sper = (int64_t)a.Bt * a.ntiles * 256;
        // B: lane (c, r) holds state c of step 4 g + r (the outer product's rows); C: lane (c, r)
        // holds states 4 r..4 r + 3 of step c (read by DPP row_newbcast)
        // (buffer loads whose lane offset runs with the chunks: rows outside the segment give zeros)
        const uint32_t nbc = (uint32_t)len * NS * sizeof(T);
        const __amdgpu_buffer_rsrc_t brs =
            __builtin_amdgcn_make_buffer_rsrc((void*)(Bm + seq0 * NS), (short)0, (int)nbc, kBufRsrcWord3);
        const __amdgpu_buffer_rsrc_t crs = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(END_ONLY ? nullptr : Cm + seq0 * NS), (short)0, (int)nbc, kBufRsrcWord3);
        constexpr uint32_t kBcStep = TCH * NS * sizeof(T);
        uint32_t bo = (uint32_t)((chunk_t(0) + r) * NS + c) * sizeof(T), co = (uint32_t)((chunk_t(0) + c) * NS + 4 * r) * sizeof(T);
        T rb[NB][4];
        typename Vec4<T>::raw rc[NB];
        auto fetch = [&](int k) __attribute__((always_inline)) {  // the next chunk
#pragma unroll
            for (int g = 0; g < 4; ++g) rb[k][g] = row_load(brs, bo + g * (4 * NS * (uint32_t)sizeof(T)), 0, (const T*)nullptr);
            bo = END_ONLY ? bo - kBcStep : bo + kBcStep;
            if constexpr (!END_ONLY) {
                rc[k] = row_load4(crs, co, (const T*)nullptr);
                co += kBcStep;
            }
        };
        auto raw4 = [](const typename Vec4<T>::raw& v) -> float4 {
            if constexpr (sizeof(T) == 4) return v;
            else return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u),
                                    __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u));
        };
#pragma unroll
        for (int k = 0; k < NB; ++k) fetch(k);
        if constexpr (!END_ONLY) {
            if (a.init)
#pragma unroll
                for (int k = 0; k < 4; ++k) h[k] = a.init[sidx + k];
            // entry state: the segments before this one, chained
#pragma unroll 8
            for (int s = 0; s < seg; ++s) {
                const float4 de = a.decay[s * sper + slot], he = a.hend[s * sper + slot];
                h[0] = fmaf(de.x, h[0], he.x);
                h[1] = fmaf(de.y, h[1], he.y);
                h[2] = fmaf(de.z, h[2], he.z);
                h[3] = fmaf(de.w, h[3], he.w);
            }
        }
        if constexpr (DTP) lds_barrier();
        lds_barrier();
        float ex[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // END_ONLY: log2 of each state's decay from the step reached to the segment's end
        bool dropped = false;
        constexpr int G0 = END_ONLY ? 3 : 0;  // first group of 4 steps walked
        float du[4];
        const float* dup = reinterpret_cast<const float*>(smem + kRow) + (16 * w + c) * 4 + r;  // component r of s_du[buf][g][16 w + c]
        auto read_du = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < 4; ++g) du[g] = dup[(buf * 4 + g) * 256];
        };
        const f32x16_t zero = {};
        read_du(0);
        float4 dt = s_dt[0][G0][16 * w + c];
        f32x16_t x = __builtin_amdgcn_mfma_f32_16x16x1f32(to_f32(rb[0][G0]), du[G0], zero, 0, 0, 0);
        auto body = [&](auto kc, int i) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value, kn = (k + 1) % NB;
            float4 C4 = {};
            if constexpr (!END_ONLY) {
                C4 = raw4(rc[k]);
                // a DPP source needs two wait states after the instruction that wrote it, which the
                // compiler does not see for fmac_bcast's
                asm volatile("s_nop 1" : "+v"(C4.x), "+v"(C4.y), "+v"(C4.z), "+v"(C4.w));
            }
            const float ck[4] = {C4.x, C4.y, C4.z, C4.w};
            StepLoop<4>::run([&](auto gc) __attribute__((always_inline)) {
                constexpr int gi = decltype(gc)::value, g = END_ONLY ? 3 - gi : gi;
                // the next group's dt and inputs B * dt*u while this group computes
                constexpr int gn = END_ONLY ? (g + 3) % 4 : (g + 1) % 4;
                const float4 q = dt;
                const f32x16_t xc = x;
                if constexpr (gi < 3) {
                    dt = s_dt[k][gn][16 * w + c];
                    x = __builtin_amdgcn_mfma_f32_16x16x1f32(to_f32(rb[k][gn]), du[gn], zero, 0, 0, 0);
                    if constexpr (gi == 2) read_du(kn);
                } else {
                    dt = s_dt[kn][gn][16 * w + c];
                    x = __builtin_amdgcn_mfma_f32_16x16x1f32(to_f32(rb[kn][gn]), du[gn], zero, 0, 0, 0);
                }
                const float qd[4] = {q.x, q.y, q.z, q.w};
                if constexpr (END_ONLY) {
#pragma unroll
                    for (int e = 3; e >= 0; --e) {
#pragma unroll
                        for (int n = 0; n < 4; ++n) {
                            h[n] = fmaf(fast_exp2(ex[n]), xc[4 * e + n], h[n]);
                            ex[n] = fmaf(A2[n], qd[e], ex[n]);
                        }
                    }
                    // nothing here has a side effect: pins the group's work to its place
                    asm volatile("" : "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]), "+v"(ex[0]), "+v"(ex[1]), "+v"(ex[2]), "+v"(ex[3]));
                } else {
                    float ab[4][4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int n = 0; n < 4; ++n) ab[e][n] = fast_exp2(qd[e] * A2[n]);
                    float y[4];
                    StepLoop<4>::run([&](auto ec) __attribute__((always_inline)) {
                        constexpr int e = decltype(ec)::value, s = 4 * g + e;
#pragma unroll
                        for (int n = 0; n < 4; ++n) h[n] = fmaf(ab[e][n], h[n], xc[4 * e + n]);
                        float acc = dpp<kDppBcast<s>>(ck[0]) * h[0];
                        acc = fmac_bcast<s>(acc, ck[1], h[1]);
                        acc = fmac_bcast<s>(acc, ck[2], h[2]);
                        y[e] = fmac_bcast<s>(acc, ck[3], h[3]);
                    });
                    s_part[k][g][r][16 * w + c] = make_float4(y[0], y[1], y[2], y[3]);
                }
                // keeps the scheduler from collecting the groups' independent work (and spilling it)
                __builtin_amdgcn_sched_barrier(0);
            });
            fetch(k);
            if constexpr (END_ONLY && k == NB - 1) {
                // stop once every state of the block's channels has decayed below 2^-32 on its way
                // to the segment's end (a NaN or growing decay never stops it)
                float m = fast_exp2(ex[0]);
#pragma unroll
                for (int n = 1; n < 4; ++n) m = fmaxf(m, fast_exp2(ex[n]));
                const int go = __ballot(dvalid && !(m < kDecayDrop)) != 0;
                if (lane == 0) s_vote[0][w] = go;
            }
            lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
        walk(body, [&](int i) { dropped = i < nch; });
        if constexpr (END_ONLY) {
            const int64_t o = seg * sper + slot;
            a.hend[o] = make_float4(h[0], h[1], h[2], h[3]);
            float q[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) q[n] = dropped ? 0.0f : fast_exp2(ex[n]);
            a.decay[o] = make_float4(q[0], q[1], q[2], q[3]);
        } else if (a.last && dvalid && seg == a.nseg - 1) {
#pragma unroll
            for (int k = 0; k < 4; ++k) a.last[sidx + k] = h[k];
        }
    } else {
        // ------------------------------------------------ element wave: steps 4 w..4 w + 3 of every
        // chunk for the block's 64 channels, lane = channel
        const int64_t d = (int64_t)tile * 64 + lane;
        const bool dvalid = d < Dm;
        const uint32_t dc = (uint32_t)(dvalid ? d : Dm - 1);
        const uint32_t loff = dc * sizeof(T);
        // stores of channels past dim (and of steps past the end) go to an offset past the resource, which
        // the hardware drops: a branch around them would make the loads' wait counts conservative.
        // Segments stay below 2^31 bytes, so neither it nor its sum with a row offset wraps into range.
        constexpr uint32_t kDrop = 0x80000000u;
        const uint32_t soff = dvalid ? loff : kDrop;
        // buffer resources of the segment's rows: lane offsets stay fixed, a row's byte offset is the
        // scalar operand; every access is inside (rows are clamped)
        const uint32_t rowb = (uint32_t)(Dm * sizeof(T));
        const uint32_t nrec = (uint32_t)len * rowb;
        auto rsrc = [&](const T* p) {
            return __builtin_amdgcn_make_buffer_rsrc((void*)(p ? p + seq0 * Dm : p), (short)0, (int)nrec, kBufRsrcWord3);
        };
        const __amdgpu_buffer_rsrc_t urs = rsrc(u), drs = rsrc(DTP ? nullptr : delta), zrs = rsrc(USE_Z ? z : nullptr),
                                     ors = rsrc(END_ONLY ? nullptr : out);
        const float Dd = !END_ONLY && a.D ? a.D[dc] : 0.0f;
        const float bias = a.bias ? a.bias[dc] : 0.0f;
        T ru[NB][4], rd[NB][4], rz[NB][4];
        auto fetch = [&](int k, int i) __attribute__((always_inline)) {
            const int t0 = chunk_t(i) + 4 * w;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t ro = (uint32_t)(t0 + e < len ? t0 + e : len - 1) * rowb;
                ru[k][e] = row_load(urs, loff, ro, (const T*)nullptr);
                if constexpr (!DTP) rd[k][e] = row_load(drs, loff, ro, (const T*)nullptr);
                if constexpr (USE_Z) rz[k][e] = row_load(zrs, loff, ro, (const T*)nullptr);
            }
        };
        // fused dt projection: this wave forms the 16 channels' tile w of each chunk
        bf16x8_t wdtf[NKB], rdl[NKB];
        auto fetch_dl = [&](int i) __attribute__((always_inline)) {
            if constexpr (DTP) {
                const int t = chunk_t(i) + c;
                const uint16_t* p = a.dtlo + (seq0 + (t < len ? t : len - 1)) * (32 * DTPK) + 8 * r;
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb) rdl[kb] = *reinterpret_cast<const bf16x8_t*>(p + 32 * kb);
            }
        };
        auto dt_tile = [&](int buf) __attribute__((always_inline)) {  // lane (c, r): steps 4 r..4 r + 3 of channel 16 w + c
            if constexpr (DTP) {
                f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int kb = 0; kb < NKB; ++kb) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(rdl[kb], wdtf[kb], acc, 0, 0, 0);
                // rounded to bf16 (nearest even) as a stored dt would be
                s_raw[buf][r][16 * w + c] = make_uint2(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]));
            }
        };
        float pu[NB][4], pg[NB][4];  // u and SiLU(z) of the chunks prepared and not yet finished
        auto prepare = [&](int k, int i) __attribute__((always_inline)) {
            float x[4], q[4];
            if constexpr (DTP) {
                const uint2 v = s_raw[k][w][lane];
                x[0] = __uint_as_float(v.x << 16);
                x[1] = __uint_as_float(v.x & 0xffff0000u);
                x[2] = __uint_as_float(v.y << 16);
                x[3] = __uint_as_float(v.y & 0xffff0000u);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pu[k][e] = to_f32(ru[k][e]);
                asm("" : "+v"(pu[k][e]));  // a register of its own: the ring's keeps its place
                if constexpr (!DTP) x[e] = to_f32(rd[k][e]);
                x[e] += bias;
                if (SOFTPLUS) x[e] = softplus(x[e]);
                q[e] = x[e] * pu[k][e];
                if constexpr (USE_Z) pg[k][e] = silu(to_f32(rz[k][e]));
            }
            const int n = len - chunk_t(i) - 4 * w;  // steps past the end change nothing
            if (n < 4) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (e >= n) x[e] = q[e] = 0.0f;
            }
            s_dt[k][w][lane] = make_float4(x[0], x[1], x[2], x[3]);
            s_du[k][w][lane] = make_float4(q[0], q[1], q[2], q[3]);
        };
        auto finish = [&](int k, int i, auto lastc) __attribute__((always_inline)) {
            const float4 p0 = s_part[k][w][0][lane], p1 = s_part[k][w][1][lane], p2 = s_part[k][w][2][lane],
                         p3 = s_part[k][w][3][lane];
            const int t = i * TCH + 4 * w;
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[e] = (f4get(p0, e) + f4get(p2, e)) + (f4get(p1, e) + f4get(p3, e));
                y[e] = fmaf(Dd, pu[k][e], y[e]);
                if (HAS_Z) y[e] *= pg[k][e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // only the last chunk may be ragged; iteration 0's call (chunk -1) stores nothing
                const bool in = lastc() ? t + e < len : i >= 0;
                row_store(y[e], ors, in ? soff : kDrop, in ? (uint32_t)(t + e) * rowb : 0u, (T*)nullptr);
            }
        };
#pragma unroll
        for (int k = 0; k < NB; ++k) fetch(k, k);
        if constexpr (DTP) {
            int64_t ch = (int64_t)tile * 64 + 16 * w + c;
            ch = ch < Dm ? ch : Dm - 1;
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb)
                wdtf[kb] = *reinterpret_cast<const bf16x8_t*>(a.wdt + ch * (32 * DTPK) + 32 * kb + 8 * r);
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                fetch_dl(k);
                dt_tile(k);
            }
            fetch_dl(NB);
            lds_barrier();
        }
        prepare(0, 0);
        fetch(0, NB);
        prepare(1, 1);
        fetch(1, NB + 1);
        lds_barrier();
        // iteration i: finish chunk i - 1, prepare chunk i + 2 (the state waves run chunk i and read
        // ahead into i + 1), form the dt tile of chunk i + 3
        auto body = [&](auto kc, int i) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value, k2 = (k + 2) % NB;
            if constexpr (!END_ONLY) {
                finish(k2, i - 1, std::false_type{});
            }
            prepare(k2, i + 2);
            fetch(k2, i + 2 + NB);
            if constexpr (DTP) {
                dt_tile(k);
                fetch_dl(i + 4);
            }
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
        const int rem = walk(body, [](int) {});
        if constexpr (!END_ONLY) {
            if (rem == 1) finish(0, nch - 1, std::true_type{});
            else if (rem == 2) finish(1, nch - 1, std::true_type{});
            else finish(2, nch - 1, std::true_type{});
        }
    }
}

}  // namespace
}  // namespace hx
