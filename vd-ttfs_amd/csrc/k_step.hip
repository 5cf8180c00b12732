// Step-by-step (time-driven) baseline kernels: the reference's own GPU
// denominator (T1S = task1_lenet_mnist/stepbystep_cuda/snn_mnist_stepbystep.cu,
// T2S = task2_vgg16_cifar10/stepbystep_cuda/bench_vgg_timedriven_baseline.cu):
// every neuron takes every step of its windows, scans its whole receptive
// field (no event lists), and fires once on the decaying threshold.  The
// programs scan the field at every step; k_step_layer scans it once for all of
// them, so its time is no measure of theirs.
//   k_step_layer  conv / FC layer, all its steps (T1S:47-103, T2S:53-108 and
//                 141-200);
//   k_step_pool   spiking 2x2 pool (T1S:107-127, T2S:110-139);
//   k_s3_*        the CuLIF network of T3S (below), a launch per layer and step.
// T1S and T2S launch every layer at every step; their neurons spike at most
// once and feed forward only, so a layer's spikes of all steps are its
// first-spike steps, and the layers run one after the other, each over all
// steps, with the state of a neuron in registers in between.
// The step's decay kv(t) and threshold th(t) are the same for every neuron of
// a layer; the host evaluates them once per (layer, step) with the same expf
// expressions and passes them in.
#include "common.h"
#include "wave.h"

namespace vdttfs {
namespace {

// One thread per neuron (numbered c_out fastest, so a wave's threads read the
// same inputs and consecutive weights), one wave per workgroup.  A thread scans
// its field once, in (kh, kw, c_in) order, and adds each input that spikes to
// the sum of its step, one LDS column of n_int steps per thread: a step's sum
// is the same chain, in the same order, as a scan of the field at that step.
// Then the thread runs the steps.  Bound by latency: the read-modify-write of
// the LDS column per spike and the loads of the scan, with ten waves on a CU
// (16 KB of LDS each at 64 steps); 16 inputs and weights are loaded ahead of
// the chain, and a wave's place in the field is kept in scalar registers.
// LeNet-5, T = 64, batch 256: 520 launches that read the field and the state
// of every neuron T times took 3126 us, these nine take 124 (conv1 71 us,
// conv2 64, the FC layers 78 when each runs alone).
constexpr int kStepAhead = 16;

struct StepArgs {
    const float* in;   // first-spike steps of the inputs (no step: does not spike)
    float* out;        // first-spike steps, else +inf (T1S output: 9999); T2S output layer: max(V + b)
    const float* W;
    const float* bias;
    int64_t n, n0;     // neurons, and the first of this launch
    int H_in, W_in, C_in, H_out, W_out, C_out, K_h, K_w, pad_h, pad_w;
    StepWindows w;
};

// PAD: taps may fall outside the map.
template <int MODE, bool PAD>  // 1: T1S (psp = sum w; V = fma(psp, kv, V)); 2: T2S (psp = fma chain of w*kv; V += psp)
__global__ __launch_bounds__(64) void k_step_layer(StepArgs a) {
    extern __shared__ float lds[];
    const int lane = threadIdx.x;
    const int n_int = a.w.n_int, n_pad = (n_int + 7) & ~7;
    float* const psp = lds + lane;  // step t0 + s at psp[64 s]; read and written by this thread alone
    for (int s = 0; s < n_pad; s += 8)
#pragma unroll
        for (int k = 0; k < 8; ++k) psp[64 * (s + k)] = 0.0f;
    float kvr[kStepMaxWin / 64];  // T2S: kv of step 64 k + lane
#pragma unroll
    for (int k = 0; k < kStepMaxWin / 64; ++k) kvr[k] = MODE == 2 ? a.w.kv[64 * k + lane] : 0.0f;
    const int64_t nid_raw = a.n0 + (int64_t)blockIdx.x * 64 + lane;
    const bool real = nid_raw < a.n;
    const int64_t nid = real ? nid_raw : a.n - 1;
    const int64_t q = nid / a.C_out;
    const int co = (int)(nid - q * a.C_out);
    const int wo = (int)(q % a.W_out);
    const int ho = (int)((q / a.W_out) % a.H_out);
    const int64_t img = q / ((int64_t)a.W_out * a.H_out);
    const int h0 = ho - a.pad_h, w0 = wo - a.pad_w;
    const float* const src = a.in + img * a.H_in * a.W_in * a.C_in;
    const float* const tap0 = src + ((int64_t)h0 * a.W_in + w0) * a.C_in;  // tap (0, 0); read inside the map only
    const int K = a.K_h * a.K_w * a.C_in;
    const int64_t row = (int64_t)(a.W_in - a.K_w) * a.C_in;  // from a row's last tap to the next row's first
    // the next element, the same in every lane: its place, its distance from
    // tap (0, 0) and its weights
    int kh = 0, kw = 0, ci = 0;
    int64_t off = 0;
    const float* wt = a.W;
    for (int e0 = 0; e0 < K; e0 += kStepAhead) {
        float x[kStepAhead], w[kStepAhead];
#pragma unroll
        for (int u = 0; u < kStepAhead; ++u) {
            const bool in_field = e0 + u < K;  // past the last element: the last one again, as no input
            bool ok = in_field;
            if constexpr (PAD) {
                ok = ok && (unsigned)(h0 + kh) < (unsigned)a.H_in && (unsigned)(w0 + kw) < (unsigned)a.W_in;
                x[u] = *(ok ? tap0 + off : src);
            } else {
                x[u] = tap0[off];
            }
            if (!ok) x[u] = -1.0f;
            w[u] = wt[co];
            if (e0 + u + 1 < K) {
                ++off;
                wt += a.C_out;
                if (++ci == a.C_in) {
                    ci = 0;
                    if (++kw == a.K_w) {
                        kw = 0;
                        ++kh;
                        off += row;
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kStepAhead; ++u) {
            // an input spikes at step t where its time equals t
            const float d = x[u] - a.w.t0;
            const bool ev = d >= 0.0f && d < (float)n_int && x[u] == floorf(x[u]);
            const int s = ev ? (int)d : 0;
            float kv = 0.0f;
            if constexpr (MODE == 2) {
                kv = __shfl(kvr[0], s & 63, 64);
#pragma unroll
                for (int k = 1; k < kStepMaxWin / 64; ++k)
                    if (64 * k < n_int) {  // uniform
                        const float y = __shfl(kvr[k], s & 63, 64);
                        kv = (s >> 6) == k ? y : kv;
                    }
            }
            if (ev) psp[64 * s] = MODE == 1 ? psp[64 * s] + w[u] : __builtin_fmaf(w[u], kv, psp[64 * s]);
        }
    }
    const float b = a.bias[co];
    float V = 0.0f;
    // the steps, 8 sums and their constants loaded at a time (those past the
    // last add nothing and cannot fire)
    float first = __builtin_inff(), best = -1e9f;
    for (int s0 = 0; s0 < n_pad; s0 += 8) {
        float p[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) p[k] = psp[64 * (s0 + k)];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            // a neuron that has fired integrates on: nothing reads its V then
            V = MODE == 1 ? __builtin_fmaf(p[k], a.w.kv[s0 + k], V) : V + p[k];
            const float v = V + b;
            if (MODE == 2 && a.w.out_layer)
                best = v > best ? v : best;
            else if (first == __builtin_inff() && v >= a.w.th[s0 + k])
                first = a.w.t0 + (float)(s0 + k);
        }
    }
    if (MODE == 2 && a.w.out_layer) {
        if (real) a.out[nid] = best;
        return;
    }
    for (int s = 0; s < a.w.n_after; ++s)
        if (first == __builtin_inff() && V + b >= a.w.th_after[s]) first = a.w.t_after + (float)s;
    if (a.w.out_layer && first == __builtin_inff()) first = kInfTime;
    if (real) a.out[nid] = first;
}

// A pool neuron spikes with the first spike of its window.
__global__ __launch_bounds__(256) void k_step_pool(const float* __restrict__ in, float* __restrict__ out, int64_t n,
                                                   int H_in, int W_in, int C, float steps) {
    const int Ho = H_in / 2, Wo = W_in / 2;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int c = (int)(idx % C), w = (int)((idx / C) % Wo), h = (int)((idx / C / Wo) % Ho);
        const int64_t b = idx / ((int64_t)C * Wo * Ho);
        float m = __builtin_inff();
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float x = in[((b * H_in + 2 * h + k / 2) * W_in + 2 * w + k % 2) * C + c];
            if (x >= 0.0f && x < steps && x == floorf(x)) m = fminf(m, x);
        }
        out[idx] = m;
    }
}

__global__ __launch_bounds__(256) void k_step_fill(float* __restrict__ p, int64_t n, float v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

unsigned step_grid(int64_t n) {
    int64_t b = (n + 255) / 256;
    if (b > (1 << 20)) b = 1 << 20;
    return (unsigned)(b < 1 ? 1 : b);
}

}  // namespace

int launch_step_layer(vdttfs_ctx* ctx, const StepLayer& L, const float* in, float* out, int mode,
                      const StepWindows& w) {
    if (L.n <= 0) return VDTTFS_OK;
    if (w.n_int < 0 || w.n_int > kStepMaxWin || w.n_after < 0 || w.n_after > kStepMaxWin)
        return set_error(VDTTFS_E_UNSUPPORTED, "step layer: windows of %d and %d steps", w.n_int, w.n_after);
    StepArgs a{};
    a.in = in;
    a.out = out;
    a.W = L.W;
    a.bias = L.bias;
    a.n = L.n;
    a.H_in = L.is_fc ? 1 : L.H_in;
    a.W_in = L.is_fc ? 1 : L.W_in;
    a.C_in = L.is_fc ? L.H_in * L.W_in * L.C_in : L.C_in;
    a.H_out = L.is_fc ? 1 : L.H_out;
    a.W_out = L.is_fc ? 1 : L.W_out;
    a.C_out = L.C_out;
    a.K_h = L.is_fc ? 1 : L.K_h;
    a.K_w = L.is_fc ? 1 : L.K_w;
    a.pad_h = L.is_fc ? 0 : L.pad_h;
    a.pad_w = L.is_fc ? 0 : L.pad_w;
    a.w = w;
    const size_t lds = (size_t)64 * ((w.n_int + 7) & ~7) * 4;
    const bool pad = a.pad_h != 0 || a.pad_w != 0;
    constexpr int64_t kMost = INT64_C(1) << 30;  // a launch's neurons: a grid holds below 2^32 threads
    for (a.n0 = 0; a.n0 < L.n; a.n0 += kMost) {
        const int64_t left = L.n - a.n0;
        const dim3 blocks((unsigned)(((left < kMost ? left : kMost) + 63) / 64));
        if (mode == 1 && pad)
            hipLaunchKernelGGL((k_step_layer<1, true>), blocks, dim3(64), lds, ctx->stream, a);
        else if (mode == 1)
            hipLaunchKernelGGL((k_step_layer<1, false>), blocks, dim3(64), lds, ctx->stream, a);
        else if (pad)
            hipLaunchKernelGGL((k_step_layer<2, true>), blocks, dim3(64), lds, ctx->stream, a);
        else
            hipLaunchKernelGGL((k_step_layer<2, false>), blocks, dim3(64), lds, ctx->stream, a);
        VD_HIP(hipGetLastError());
    }
    return VDTTFS_OK;
}

int launch_step_pool(vdttfs_ctx* ctx, const float* in, float* out, int64_t n, int H_in, int W_in, int C, int steps) {
    hipLaunchKernelGGL(k_step_pool, dim3(step_grid(n)), dim3(256), 0, ctx->stream, in, out, n, H_in, W_in, C,
                       (float)steps);
    VD_HIP(hipGetLastError());
    return VDTTFS_OK;
}

int launch_step_fill(vdttfs_ctx* ctx, float* p, int64_t n, float v) {
    hipLaunchKernelGGL(k_step_fill, dim3(step_grid(n)), dim3(256), 0, ctx->stream, p, n, v);
    VD_HIP(hipGetLastError());
    return VDTTFS_OK;
}

// ---------------------------------------------------------------------------
// T3S = task3_dvsgesture/stepbystep_cuda/snn_dvs_stepbystep.cu: the CuLIF
// network stepped densely.  Every step, every layer computes every neuron's
// input current from that step's 0/1 spike map (the raw event values for the
// first layer) in the reference's order -- conv over c_in, ky, kx
// (T3S:53-64), FC over i ascending (T3S:104-106), all as fma(in, w, sum) --
// and runs the CuIF neuron I = fma(I, decay, cur); V = V + I; spike once at
// V >= th (T3S:119-140).  Maps are NCHW, threads numbered like the
// reference's (x fastest, FC: output fastest).  The current and the neuron
// share one kernel (the reference's separate current buffer changes
// nothing), except for the recurrent FC, whose current reads the layer's own
// spikes of step t-1 and so must complete before any of them is replaced.
namespace {

struct Step3Args {
    const float* in;
    const float* weight;
    const float* weight_rec;
    float* I;
    float* V;
    float* s;
    uint8_t* fired;
    float* ft;
    float* cur;
    int64_t n;
    int C_in, H, Wd, C_out, T, t;
    float decay, th;
};

__device__ __forceinline__ void s3_neuron(const Step3Args& a, int64_t i, float cur) {
    const float ci = __builtin_fmaf(a.I[i], a.decay, cur);
    const float cv = a.V[i] + ci;
    a.I[i] = ci;
    a.V[i] = cv;
    if (!a.fired[i] && cv >= a.th) {
        a.s[i] = 1.0f;
        a.fired[i] = 1;
        a.ft[i] = (float)a.t;
    } else {
        a.s[i] = 0.0f;
    }
}

// extract_input_step (T3S:33-39): the raw events of step t, NCHW
__global__ __launch_bounds__(256) void k_s3_extract(const float* __restrict__ data, float* __restrict__ out,
                                                    int64_t n, int T, int t) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = data[i * T + t];
}

// conv2d_kernel (T3S:41-68) + neuron.  Taps outside the map are skipped as
// in the reference (a select keeps sum unchanged, whatever the weight).
// A thread computes COB consecutive c_out of one pixel (threads numbered
// x fastest, then y, c_out block, n), so each input load feeds COB
// independent fma chains, each in the reference's c_in, ky, kx order.
// UNI: H*W is a multiple of 64, so a wave's threads share (n, c_out block)
// and read each weight as one scalar load.
template <bool UNI, int COB>
__global__ __launch_bounds__(256) void k_s3_conv(Step3Args a) {
    const int H = a.H, W = a.Wd, C_in = a.C_in, n_cb = a.C_out / COB;
    const int64_t HW = (int64_t)H * W;
    const int64_t n_thr = a.n / COB;
    for (int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; tid < n_thr;
         tid += (int64_t)gridDim.x * blockDim.x) {
        const int x = (int)(tid % W), y = (int)((tid / W) % H);
        int cb = (int)((tid / HW) % n_cb);
        int64_t nb = tid / (HW * n_cb);
        if (UNI) {
            cb = __builtin_amdgcn_readfirstlane(cb);
            nb = ((int64_t)__builtin_amdgcn_readfirstlane((int)(nb >> 32)) << 32) |
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)nb);
        }
        bool ok[9];
        int off[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const int iy = y + k / 3 - 1, ix = x + k % 3 - 1;
            ok[k] = iy >= 0 && iy < H && ix >= 0 && ix < W;
            off[k] = ok[k] ? iy * W + ix : 0;
        }
        const int co0 = cb * COB;
        const float* ip = a.in + nb * C_in * HW;
        float sum[COB];
#pragma unroll
        for (int o = 0; o < COB; ++o) sum[o] = 0.0f;
        for (int c = 0; c < C_in; ++c) {
            float v[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) v[k] = ip[off[k]];
#pragma unroll
            for (int o = 0; o < COB; ++o) {
                const float* wk = a.weight + ((int64_t)(co0 + o) * C_in + c) * 9;
#pragma unroll
                for (int k = 0; k < 9; ++k) sum[o] = ok[k] ? __builtin_fmaf(v[k], wk[k], sum[o]) : sum[o];
            }
            ip += HW;
        }
#pragma unroll
        for (int o = 0; o < COB; ++o) s3_neuron(a, ((nb * a.C_out + co0 + o) * H + y) * (int64_t)W + x, sum[o]);
    }
}

// maxpool2d_kernel (T3S:70-94) + neuron
__global__ __launch_bounds__(256) void k_s3_pool(Step3Args a) {
    const int H_in = a.H, W_in = a.Wd, H_out = H_in / 2, W_out = W_in / 2, C = a.C_in;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < a.n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int xo = (int)(idx % W_out), yo = (int)((idx / W_out) % H_out);
        const int c = (int)((idx / ((int64_t)W_out * H_out)) % C);
        const int64_t nb = idx / ((int64_t)C * H_out * W_out);
        const float* p = a.in + ((nb * C + c) * H_in + yo * 2) * (int64_t)W_in + xo * 2;
        float m = -1e9f;
        m = fmaxf(m, p[0]);
        m = fmaxf(m, p[1]);
        m = fmaxf(m, p[W_in]);
        m = fmaxf(m, p[W_in + 1]);
        s3_neuron(a, idx, m);
    }
}

// sum over i ascending of x[i] * w[i * stride] (FC weights are stored
// [in][out], stride = out)
__device__ __forceinline__ float s3_dot(const float* __restrict__ x, const float* __restrict__ w, int n,
                                        int stride) {
    float sum = 0.0f;
    int i = 0;
    // 16 loads in flight per thread; the fma chain keeps the i-ascending order
    for (; i + 16 <= n; i += 16) {
        float xv[16], wv[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            xv[k] = x[i + k];
            wv[k] = w[(int64_t)(i + k) * stride];
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) sum = __builtin_fmaf(xv[k], wv[k], sum);
    }
    for (; i < n; ++i) sum = __builtin_fmaf(x[i], w[(int64_t)i * stride], sum);
    return sum;
}

// fc_kernel (T3S:96-109) + neuron
__global__ __launch_bounds__(256) void k_s3_fc(Step3Args a) {
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < a.n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = idx / a.C_out;
        const int col = (int)(idx % a.C_out);
        s3_neuron(a, idx, s3_dot(a.in + row * a.C_in, a.weight + col, a.C_in, a.C_out));
    }
}

// recurrent FC current (T3S:244-246): the FC of the input plus, added after,
// the FC of the layer's own spikes of step t-1
__global__ __launch_bounds__(256) void k_s3_fcrec_current(Step3Args a) {
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < a.n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = idx / a.C_out;
        const int col = (int)(idx % a.C_out);
        const float f = s3_dot(a.in + row * a.C_in, a.weight + col, a.C_in, a.C_out);
        const float r = s3_dot(a.s + row * a.C_out, a.weight_rec + col, a.C_out, a.C_out);
        a.cur[idx] = f + r;
    }
}

__global__ __launch_bounds__(256) void k_s3_neuron(Step3Args a) {
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < a.n;
         idx += (int64_t)gridDim.x * blockDim.x)
        s3_neuron(a, idx, a.cur[idx]);
}

}  // namespace

int launch_step3_layer(vdttfs_ctx* ctx, const Step3Layer& L, const float* in, int N, int T, int t) {
    Step3Args a{};
    a.in = in;
    a.weight = L.weight;
    a.weight_rec = L.weight_rec;
    a.I = L.I;
    a.V = L.V;
    a.s = L.s;
    a.fired = L.fired;
    a.ft = L.ft;
    a.cur = L.cur;
    a.n = L.n;
    a.C_in = L.C_in;
    a.H = L.H;
    a.Wd = L.W;
    a.C_out = L.C_out;
    a.T = T;
    a.t = t;
    a.decay = L.decay;
    a.th = L.th;
    const dim3 grid(step_grid(L.n)), block(256);
    const bool uni = ((int64_t)L.H * L.W) % 64 == 0;
    switch (L.kind) {
        case VDTTFS_CULIF_RAW_CONV: {
            // the step's events first, as the reference does
            if (!L.cur) return set_error(VDTTFS_E_INVALID, "step3: raw conv without a step-input buffer");
            const int64_t n_in = (int64_t)N * L.C_in * L.H * L.W;
            hipLaunchKernelGGL(k_s3_extract, dim3(step_grid(n_in)), block, 0, ctx->stream, in, L.cur, n_in, T, t);
            VD_HIP(hipGetLastError());
            a.in = L.cur;
        }
            [[fallthrough]];
        case VDTTFS_CULIF_CONV: {
            const bool cob4 = L.C_out % 4 == 0;
            const dim3 cgrid(step_grid(cob4 ? L.n / 4 : L.n));
            if (uni && cob4)
                hipLaunchKernelGGL((k_s3_conv<true, 4>), cgrid, block, 0, ctx->stream, a);
            else if (cob4)
                hipLaunchKernelGGL((k_s3_conv<false, 4>), cgrid, block, 0, ctx->stream, a);
            else if (uni)
                hipLaunchKernelGGL((k_s3_conv<true, 1>), cgrid, block, 0, ctx->stream, a);
            else
                hipLaunchKernelGGL((k_s3_conv<false, 1>), cgrid, block, 0, ctx->stream, a);
            break;
        }
        case VDTTFS_CULIF_POOL: hipLaunchKernelGGL(k_s3_pool, grid, block, 0, ctx->stream, a); break;
        case VDTTFS_CULIF_FC: hipLaunchKernelGGL(k_s3_fc, grid, block, 0, ctx->stream, a); break;
        case VDTTFS_CULIF_FC_REC:
            if (!L.cur) return set_error(VDTTFS_E_INVALID, "step3: recurrent layer without a current buffer");
            hipLaunchKernelGGL(k_s3_fcrec_current, grid, block, 0, ctx->stream, a);
            VD_HIP(hipGetLastError());
            hipLaunchKernelGGL(k_s3_neuron, grid, block, 0, ctx->stream, a);
            break;
        default: return set_error(VDTTFS_E_INVALID, "step3: layer kind %d", L.kind);
    }
    VD_HIP(hipGetLastError());
    return VDTTFS_OK;
}

}  // namespace vdttfs
