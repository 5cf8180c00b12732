// Narrow conv layers (at most 16 outputs) with at most 160 elements in a field:
// one pixel per lane, or per four lanes, with all its outputs in registers
// (LeNet-5's convolutions, T1V:83-162).
//
// A lane loads its elements of the field and packs every event into one key,
// {bin, element, decay index}, so that the smallest key above the last one is
// the next event in the reference's order: bins ascending, within a bin (kh,
// kw, cin).  Finding it takes a subtract per element and a three-way minimum
// per two; the event then adds its weight row (LDS) to the open bin's sums of
// all outputs.  Where a bin closes, the carry stands until the pixel's next
// event, and with thresholds that fall over the window a neuron fires in that
// run iff its carry reaches the run's last threshold; the step itself is
// searched once per neuron at the end.
//
// Bound by instruction issue: 1.5 instructions per element and event for the
// search and about 12 per output.  Up to 32 elements a lane has a pixel to
// itself (25 elements, 6 outputs, 590K pixels, T = 64: 34 us; one output per
// lane, every element compared with every occupied bin, took 145).  Past that
// four lanes share the elements and the outputs of a pixel: a lane alone needs
// all registers and leaves one wave per SIMD (150 elements, 16 outputs, 66K
// pixels: 160 us against 136; eight lanes 163).
#include "common.h"
#include "wave.h"

namespace vdttfs {
namespace {

constexpr int kPxMaxEl = 160;  // a key holds an element in 8 bits
constexpr int kPxMaxOut = 16;

// N: elements that the tables hold, 32 or kPxMaxEl (a launch of a few
// microseconds feels a kilobyte of arguments).
template <int N>
struct PxArgs {
    const float* in;     // [n_cols][C_in] spike times (NHWC map)
    const float* alpha;  // decay LUT, T + 1 entries
    const float* W;      // [nel][C_out]
    const float* bias;
    const float* theta;  // T entries
    float* out;          // [n_pix][C_out]
    int n_pix, T, t_min, alpha_by_time;
    float tfs;
    int H_in, W_in, C_in, H_out, W_out, C_out, pad_h, pad_w, nel;
    int in_bytes;        // bytes of `in`, below 2^31
    int inside;          // every tap of every pixel lies inside the map
    FastDiv div_w, div_h;
    // element e: its offset from the field's first element, and its tap's row
    // << 16 | column
    int dk[N], tap[N];
};

// The smallest value of a group of G lanes.
template <int G>
__device__ __forceinline__ unsigned group_min(unsigned v) {
    auto with = [&](unsigned x) { v = x < v ? x : v; };
    if constexpr (G > 1) with((unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true));  // lane ^ 1
    if constexpr (G > 2) with((unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true));  // lane ^ 2
    return v;
}

// G lanes share a pixel: each holds CO outputs and NEL elements, e = G i + g.
template <int G, int CO, int NEL>
__global__ __launch_bounds__(256) void k_conv_px(PxArgs<(G > 1 ? kPxMaxEl : 32)> a) {
    constexpr int COP = G * ((CO + 3) & ~3);
    constexpr unsigned kNone = ~0u;
    __shared__ __attribute__((aligned(16))) float w_lds[G * NEL * COP];
    __shared__ float lut[256], th[256];  // th: the threshold where a spike may occur, else NaN
    const int T = a.T;
    for (int i = threadIdx.x; i < a.nel * COP; i += blockDim.x) {
        const int e = i / COP, c = i - e * COP;
        w_lds[i] = c < a.C_out ? a.W[e * a.C_out + c] : 0.0f;
    }
    for (int t = threadIdx.x; t < 256; t += blockDim.x) {
        lut[t] = t <= T ? a.alpha[t] : 0.0f;
        const float x = t < T ? a.theta[t] : 0.0f;
        th[t] = (t < T && t >= a.t_min && x >= 1e-5f) ? x : __builtin_nanf("");
    }
    // the lane's field
    const int g = threadIdx.x & (G - 1), c0 = g * CO;
    const int idx = (blockIdx.x * blockDim.x + threadIdx.x) / G;
    const bool ok = idx < a.n_pix;
    const int px = ok ? idx : a.n_pix - 1;
    const int qd = fdiv(px, a.div_w);
    const int w_out = px - qd * a.W_out;
    const int img = fdiv(qd, a.div_h);
    const int h0 = qd - img * a.H_out - a.pad_h, w0 = w_out - a.pad_w;
    const int base = ((img * a.H_in + h0) * a.W_in + w0) * a.C_in;
    const __amdgpu_buffer_rsrc_t rin =
        __builtin_amdgcn_make_buffer_rsrc((void*)a.in, (short)0, a.in_bytes, 0x00020000);
    float time[NEL];
    if constexpr (G > 1) {
#pragma unroll
        for (int i = 0; i < NEL; ++i) {
            const int e = G * i + g < a.nel ? G * i + g : 0;
            const int tap = a.tap[e];
            const bool inb = (unsigned)(h0 + (tap >> 16)) < (unsigned)a.H_in &&
                             (unsigned)(w0 + (tap & 0xFFFF)) < (unsigned)a.W_in;
            const float t =
                __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rin, inb ? (base + a.dk[e]) * 4 : 0, 0, 0));
            time[i] = inb ? t : kInfTime;
        }
    } else if (a.inside) {  // uniform
#pragma unroll
        for (int e = 0; e < NEL; ++e)  // past nel: element 0 (dk 0)
            time[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rin, base * 4, a.dk[e] * 4, 0));
    } else {
#pragma unroll
        for (int e = 0; e < NEL; ++e) {
            const bool inb = (unsigned)(h0 + (a.tap[e] >> 16)) < (unsigned)a.H_in &&
                             (unsigned)(w0 + (a.tap[e] & 0xFFFF)) < (unsigned)a.W_in;
            const float t =
                __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rin, inb ? (base + a.dk[e]) * 4 : 0, 0, 0));
            time[e] = inb ? t : kInfTime;
        }
    }
    __syncthreads();
    // the bins that may fire, [lo, hi), and whether they are one run with
    // thresholds that fall or stay (a NaN inside fails)
    const int lane = lane_id();
    int lo = 256, hi = 0;
    bool fall = true;
    for (int k = 0; k < T; k += 64) {
        const uint64_t v = __ballot(th[k + lane] == th[k + lane]);
        if (v != 0) {
            const int f = k + __ffsll((unsigned long long)v) - 1;
            lo = f < lo ? f : lo;
            hi = k + 64 - __clzll((long long)v);
        }
    }
    for (int k = 0; k < T; k += 64) {
        const int t = k + lane;
        if (t >= lo && t < hi - 1) fall = fall && th[t] >= th[t + 1];
    }
    const bool mono = __ballot(!fall) == 0;
    // keys: bin << 16 | element << 8 | decay index (arrival_bin and
    // alpha_index without branches)
    unsigned key[NEL];
#pragma unroll
    for (int i = 0; i < NEL; ++i) {
        const int e = G * i + g;
        const float t = time[i];
        const int tb = (int)floorf(fmaxf(t - a.tfs, 0.0f));
        const bool ev = e < a.nel && t < kInfTime && tb < T;
        const int ai = a.alpha_by_time ? (int)__builtin_amdgcn_fmed3f(t, 0.0f, (float)T) : tb;
        key[i] = ev ? (unsigned)(tb << 16 | e << 8 | ai) : kNone;
    }
    float acc[CO], carry[CO], at_fire[CO];
    int from[CO];  // a neuron that fires: its run's first bin that may (its step, where not mono), else -1
#pragma unroll
    for (int c = 0; c < CO; ++c) {
        acc[c] = 0.0f;
        carry[c] = c0 + c < a.C_out ? a.bias[c0 + c] : 0.0f;
        at_fire[c] = 0.0f;
        from[c] = -1;
    }
    // the standing carries against bins [b0, b2); a neuron that fires goes on
    // with a NaN carry, which fires no more
    auto test = [&](int b0, int b2) __attribute__((always_inline)) {
        const int s = b0 > lo ? b0 : lo, e = b2 < hi ? b2 : hi;
        if (mono) {  // uniform
            const float x = th[e > 0 ? e - 1 : 0];
            const float last = s < e ? x : __builtin_nanf("");
#pragma unroll
            for (int c = 0; c < CO; ++c) {
                const bool f = carry[c] >= last;
                at_fire[c] = f ? carry[c] : at_fire[c];
                from[c] = f ? s : from[c];
                carry[c] = f ? __builtin_nanf("") : carry[c];
            }
        } else {
            for (int t = s; t < e; ++t) {
                const float x = th[t];
#pragma unroll
                for (int c = 0; c < CO; ++c) {
                    const bool f = carry[c] >= x;
                    from[c] = f ? t : from[c];
                    carry[c] = f ? __builtin_nanf("") : carry[c];
                }
            }
        }
    };
    unsigned m = key[0];
#pragma unroll
    for (int e = 1; e < NEL; ++e) m = key[e] < m ? key[e] : m;
    m = group_min<G>(m);
    test(0, m == kNone ? T : (int)(m >> 16));
    while (m != kNone) {
        const int b = (int)(m >> 16);
        const float al = lut[m & 0xFF];
        const float* const w = w_lds + ((m >> 8) & 0xFF) * COP + c0;
        float wv[(CO + 3) & ~3];
#pragma unroll
        for (int c = 0; c < CO; c += 4) *reinterpret_cast<float4*>(wv + c) = *reinterpret_cast<const float4*>(w + c);
#pragma unroll
        for (int c = 0; c < CO; ++c) acc[c] = __builtin_fmaf(wv[c], al, acc[c]);
        // the smallest key above m: those at or below it, and kNone, stay past
        // 24 bits
        const unsigned m1 = m + 1;
        unsigned d = key[0] - m1;
#pragma unroll
        for (int e = 1; e < NEL; ++e) {
            const unsigned x = key[e] - m1;
            d = x < d ? x : d;
        }
        d = group_min<G>(d);
        m = d < (1u << 24) ? d + m1 : kNone;
        const int b2 = m == kNone ? T : (int)(m >> 16);
        if (b2 != b) {
#pragma unroll
            for (int c = 0; c < CO; ++c) {
                carry[c] = carry[c] + acc[c];
                acc[c] = 0.0f;
            }
            test(b, b2);
        }
    }
    if (!ok) return;
    float* const po = a.out + (int64_t)px * a.C_out;
    if (mono) {
        // the first bin from `from` on whose threshold the carry reaches
        int r0[CO], r1[CO];
#pragma unroll
        for (int c = 0; c < CO; ++c) {
            r1[c] = hi > 0 ? hi - 1 : 0;
            r0[c] = from[c] < 0 ? r1[c] : from[c];
        }
        for (int span = hi - lo; span > 0; span >>= 1) {  // uniform
#pragma unroll
            for (int c = 0; c < CO; ++c) {
                const int mid = (r0[c] + r1[c]) >> 1;
                const bool le = th[mid] <= at_fire[c] || mid == r1[c];
                r1[c] = le ? mid : r1[c];
                r0[c] = le ? r0[c] : mid + 1;
            }
        }
#pragma unroll
        for (int c = 0; c < CO; ++c) from[c] = from[c] < 0 ? -1 : r1[c];
    }
#pragma unroll
    for (int c = 0; c < CO; ++c)
        if (c0 + c < a.C_out) po[c0 + c] = from[c] < 0 ? kInfTime : (float)from[c];
}

}  // namespace

// Up to 32 elements, past 64 steps: against lists in memory, at every size
// (LeNet-5's conv1 at T = 80, batch 128: 78 -> 13 us).  Up to 64 steps
// k_conv_small spreads a pixel's outputs over lanes and finishes first where
// outputs are many and pixels leave the chip idle (us a call, k_conv_small
// against this; a fifth of the inputs active):
//   25 elements, 16 outputs:  4,096 pixels 12.9 / 15.3, 12,544 17.8 / 16.2
//   27 elements, 16 outputs:  4,096 pixels 15.8 / 17.5, 12,544 23.4 / 18.2
//   25 elements, 8 outputs:   784 pixels 12.5 / 11.3;  16 and 16: 12.5 / 12.8
// Past 32 elements the search costs more than a list, which finds its order
// once, unless the pixels are many: k_merge_dense + k_stream_narrow against
// this, T = 64: 108 elements, 16K pixels 50 -> 39 us (density 0.5) and 40 ->
// 23 (0.1), at 8K 0.8 to 1.3 times the speed; 150 elements, LeNet-5's conv2:
// 66K pixels 168 -> 136.  The line for those lies where a workgroup has four
// waves (launch_conv_px): with one, each wave loads the weights for itself, and
// LeNet-5 takes 7 to 13% longer a pass at 45K to 64K pixels (batches 700 to
// 1000, T = 64; with three passes in flight they are even).
bool conv_px_ok(int T, const IntegShape& s) {
    const int64_t in = (int64_t)s.B * s.H_in * s.W_in * s.C_in * 4, pix = (int64_t)s.B * s.H_out * s.W_out;
    const int64_t nel = (int64_t)s.K_h * s.K_w * s.C_in;
    if (s.is_fc || s.C_out > kPxMaxOut || nel > kPxMaxEl) return false;
    if (in >= (INT64_C(1) << 31) || 4 * pix >= (INT64_C(1) << 31) - 256) return false;
    if (nel > 32) return pix >= (nel <= 112 ? 8192 : 65536);
    return T > 64 || s.C_out <= 8 || nel <= 16 || pix >= 12288;
}

namespace {

template <int N>
PxArgs<N> px_args(const vdttfs_ctx* ctx, float* out, const float* in, const float* alpha, const float* W,
                  const float* bias, const float* theta, int t_min, const IntegShape& s) {
    PxArgs<N> a{};
    a.in = in;
    a.alpha = alpha;
    a.W = W;
    a.bias = bias;
    a.theta = theta;
    a.out = out;
    a.n_pix = s.B * s.H_out * s.W_out;
    a.T = ctx->c.T;
    a.t_min = t_min;
    a.alpha_by_time = ctx->c.alpha_by_time;
    a.tfs = ctx->c.tfs;
    a.H_in = s.H_in;
    a.W_in = s.W_in;
    a.C_in = s.C_in;
    a.H_out = s.H_out;
    a.W_out = s.W_out;
    a.C_out = s.C_out;
    a.pad_h = s.pad_h;
    a.pad_w = s.pad_w;
    a.nel = s.K_h * s.K_w * s.C_in;  // at most N
    a.in_bytes = s.B * s.H_in * s.W_in * s.C_in * 4;
    a.inside = s.pad_h == 0 && s.pad_w == 0 && s.H_out <= s.H_in - s.K_h + 1 && s.W_out <= s.W_in - s.K_w + 1;
    a.div_w = make_fastdiv(s.W_out);
    a.div_h = make_fastdiv(s.H_out);
    for (int kh = 0, e = 0; kh < s.K_h; ++kh)
        for (int kw = 0; kw < s.K_w; ++kw)
            for (int ci = 0; ci < s.C_in; ++ci, ++e) {
                a.dk[e] = (kh * s.W_in + kw) * s.C_in + ci;
                a.tap[e] = kh << 16 | kw;
            }
    return a;
}

}  // namespace

int launch_conv_px(vdttfs_ctx* ctx, float* out, const float* in, const float* alpha, const float* W, const float* bias,
                   const float* theta, int t_min, const IntegShape& s) {
    if (!conv_px_ok(ctx->c.T, s) || ctx->c.T > 255) return set_error(VDTTFS_E_UNSUPPORTED, "conv_px: layer outside its limits");
    const int n_pix = s.B * s.H_out * s.W_out, nel = s.K_h * s.K_w * s.C_in;
    if (n_pix <= 0) return VDTTFS_OK;
    // few pixels: one wave per workgroup, so that they spread over the CUs
    const int threads = n_pix >= 256 * 256 ? 256 : 64;
    const int G = nel > 32 ? 4 : 1;
    const dim3 grid((unsigned)(((int64_t)n_pix * G + threads - 1) / threads)), block(threads);
#define VD_PX(G_, C, N)                                                              \
    hipLaunchKernelGGL((k_conv_px<G_, C, N>), grid, block, 0, ctx->stream,           \
                       px_args<(G_ > 1 ? kPxMaxEl : 32)>(ctx, out, in, alpha, W, bias, theta, t_min, s))
#define VD_PX_N(C)            \
    do {                      \
        if (nel <= 9)         \
            VD_PX(1, C, 9);   \
        else if (nel <= 16)   \
            VD_PX(1, C, 16);  \
        else if (nel <= 25)   \
            VD_PX(1, C, 25);  \
        else                  \
            VD_PX(1, C, 32);  \
    } while (0)
    if (G > 1) {
        if (nel <= 64)
            VD_PX(4, 4, 16);
        else if (nel <= 112)
            VD_PX(4, 4, 28);
        else
            VD_PX(4, 4, 40);
    } else if (s.C_out <= 4)
        VD_PX_N(4);
    else if (s.C_out <= 6)
        VD_PX_N(6);
    else if (s.C_out <= 8)
        VD_PX_N(8);
    else if (s.C_out <= 12)
        VD_PX_N(12);
    else
        VD_PX_N(16);
#undef VD_PX_N
#undef VD_PX
    VD_HIP(hipGetLastError());
    return VDTTFS_OK;
}

}  // namespace vdttfs
