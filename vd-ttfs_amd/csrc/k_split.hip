// The split integrator of layers with a fire start (T2V:59-60): every spike
// up to the fire start arrives in bin 0, which so holds most of a layer's
// events, and that bin's sums are a dense contraction.  Three kernels per
// layer:
//  k_split - one pass over the spike map: per input element the bin-0 factor
//            (alpha of its spike, 0 where it has no bin-0 event), and per
//            input column the list of its later events in cin order;
//  k_gemm0 - bin 0 of every neuron on the matrix cores, written to `out`;
//  k_late  - one workgroup per output pixel: sorts the pixel's later events
//            by bin in LDS and streams them as k_stream_quad does, the bin-0
//            sums read from `out` in place of bin 0's events.
//
// The arithmetic stays the reference's.  A bin's sum is the fma chain over its
// events in (kh, kw, cin) order from +0; v_mfma_f32_32x32x2_f32 adds its two
// products as two fmas in k order with one rounding each (checked bit for bit
// against fmaf chains, denormals and wide exponents included), and an element
// without an event contributes fma(w, 0, acc) = acc.  Two cases differ from
// skipping it: a non-finite weight (0 * inf = NaN), where k_late sees the NaN
// and adds the pixel's bin-0 events one by one instead; and the sign of a zero
// sum, which no threshold test sees.
#include <type_traits>

#include "common.h"
#include "wave.h"

namespace vdttfs {
namespace {

typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

constexpr int kSplitMaxT = 256;   // four blocks of 64 bins
constexpr int kSplitMaxTaps = 25;
constexpr int kLatePad = 32;      // zeroed entries after the list (k_late reads up to four quads ahead)
constexpr int kLateMaxWaves = 4;
constexpr int kLateKeep = 2;      // chunks per wave kept in registers between the two passes

// ---------------------------------------------------------------------------
// What k_late needs of a layer's thresholds, prepared once per call by the
// kernel that writes its lists (k_split or k_ref_lists).
struct LateThr {
    float th[kSplitMaxT];  // theta where a spike may occur (t >= t_min, theta >= 1e-5), else NaN
    // Where those bins are one run [lo, hi) with non-increasing thresholds
    // (mono), a neuron whose carry stands at c from bin b on fires at the
    // first bin t >= b with th[t] <= c, near lo + (lg0 - log2 c) * inv for the
    // exponential thresholds of the LUTs.
    float lg0, inv;
    int lo, hi, mono;
};

// A workgroup of 256 threads fills *thr.
__device__ inline void prepare_thresholds(const float* theta, int T, int t_min, LateThr* thr) {
    const int lane = lane_id();
    __shared__ float ths[kSplitMaxT + 1];
    for (int t = threadIdx.x; t <= kSplitMaxT; t += 256) {
        const float th = theta && t < T ? theta[t] : 0.0f;
        ths[t] = (t < T && t >= t_min && th >= 1e-5f) ? th : __builtin_nanf("");
        if (t < kSplitMaxT) thr->th[t] = ths[t];
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        int lo = kSplitMaxT, hi = 0;
#pragma unroll
        for (int k = 0; k < kSplitMaxT / 64; ++k) {
            const float x = ths[64 * k + lane];
            const uint64_t v = __ballot(x == x);
            if (v != 0) {
                const int f = 64 * k + __ffsll((unsigned long long)v) - 1;
                lo = f < lo ? f : lo;
                hi = 64 * k + 64 - __clzll((long long)v);
            }
        }
        lo = lo < hi ? lo : hi;
        // every step within [lo, hi) down or level (a NaN inside fails)
        bool down = true;
#pragma unroll
        for (int k = 0; k < kSplitMaxT / 64; ++k) {
            const int t = 64 * k + lane;
            if (t >= lo && t < hi - 1) down = down && ths[t] >= ths[t + 1];
        }
        const bool mono = __ballot(!down) == 0;
        if (lane == 0) {
            const float l0 = hi > lo ? log2f(ths[lo]) : 0.0f, l1 = hi > lo ? log2f(ths[hi - 1]) : 0.0f;
            thr->lg0 = l0;
            thr->inv = l0 > l1 ? (float)(hi - 1 - lo) / (l0 - l1) : 0.0f;
            thr->lo = lo;
            thr->hi = hi;
            thr->mono = mono;
        }
    }
}

struct SplitArgs {
    const float* in;     // [cols][C_in] spike times
    float* a0;           // null: no bin-0 factors, and the lists hold bin 0's events too; else [cols][Cp] bin-0 factors, C_in padded with zeros to whole groups of 4 HL; element
                         // HL s + h of a group at 4 h + s (k_gemm0's lane h takes its four steps s in one load)
    int2* late;          // [cols][C_in] later events {cin | bin << 16, alpha bits}
    int32_t* cnt;        // [cols] later events
    const float* alpha;  // decay LUT, T + 1 entries
    const float* theta;  // T thresholds
    LateThr* thr;
    int64_t cols;
    int C_in, Cp, T, alpha_by_time, t_min;
    int hl;  // log2 HL: 1 or 2
    float tfs;
};

// Arrival bin (-1: no event) and decay-LUT index of a spike time.
__device__ __forceinline__ int split_bin(float t, float tfs, int T) {
    const int tb = (int)floorf(fmaxf(t - tfs, 0.0f));
    return (t < kInfTime && tb < T) ? tb : -1;
}
__device__ __forceinline__ int split_alpha(float t, int tb, int alpha_by_time, int T) {
    return alpha_by_time ? (int)fminf(fmaxf(t, 0.0f), (float)T) : tb;
}

// One column per segment of 1 << seg lanes (a power of two of at least Cp
// lanes, 64 where Cp is larger: then the wave walks the column).  Bound by
// HBM: 4 bytes read and 4 written per element, and 8 per later event.
__global__ __launch_bounds__(256) void k_split(SplitArgs a, int seg) {
    __shared__ float lut[kSplitMaxT + 1];
    for (int i = threadIdx.x; i <= a.T; i += 256) lut[i] = a.alpha[i];
    const int lane = lane_id(), wave = uniform(threadIdx.x >> 6);
    if (blockIdx.x == 0) prepare_thresholds(a.theta, a.T, a.t_min, a.thr);
    __syncthreads();
    const int S = 1 << seg, P = 64 >> seg;
    const int sub = lane >> seg, r = lane & (S - 1);
    const uint64_t segm = S == 64 ? ~0ull : ((1ull << S) - 1) << (sub * S);
    const uint64_t lt = lanemask_lt() & segm;
    const int64_t step = (int64_t)gridDim.x * 4 * P;
    for (int64_t c0 = ((int64_t)blockIdx.x * 4 + wave) * P; c0 < a.cols; c0 += step) {
        const int64_t col = c0 + sub;
        const bool cok = col < a.cols;
        int base = 0;
        for (int c = 0; c < a.Cp; c += S) {  // S < 64: one round
            const int ci = c + r;
            float t = kInfTime;
            if (cok && ci < a.C_in) t = a.in[col * a.C_in + ci];
            const int tb = split_bin(t, a.tfs, a.T);
            const float al = tb >= 0 ? lut[split_alpha(t, tb, a.alpha_by_time, a.T)] : 0.0f;
            const int g = (4 << a.hl) - 1;
            const int at = (ci & ~g) | ((ci & ((1 << a.hl) - 1)) << 2) | ((ci & g) >> a.hl);
            if (a.a0 && cok && ci < a.Cp) a.a0[col * a.Cp + at] = tb == 0 ? al : 0.0f;
            const bool listed = tb > 0 || (tb == 0 && !a.a0);
            const uint64_t m = __ballot(listed) & segm;
            if (listed) a.late[col * a.C_in + base + __popcll(m & lt)] = make_int2(ci | (tb << 16), __float_as_int(al));
            base += __popcll(m);
        }
        if (cok && r == 0) a.cnt[col] = base;
    }
}

// The lists of k_late from the reference's buckets: per column the events of
// its bucket entries in entry order.  An entry counts where the loop nest over
// the chunks (k_integrate_generic) would take it: its own chunk's offsets,
// clamped to the column, hold its position, and its step and input are in
// range.  A step's events all come from one chunk, so entry order is that
// loop's order within every step.
struct RefListArgs {
    const int32_t* cin;  // [cols][C_in]
    const float* tin;
    const int32_t* off;  // [cols][n_chunks + 1]
    int2* late;
    int32_t* cnt;
    const float* alpha;
    const float* theta;
    LateThr* thr;
    int64_t cols;
    int C_in, T, D, alpha_by_time, t_min;
    float tfs;
};

__global__ __launch_bounds__(256) void k_ref_lists(RefListArgs a) {
    const int lane = lane_id(), wave = uniform(threadIdx.x >> 6);
    if (blockIdx.x == 0) prepare_thresholds(a.theta, a.T, a.t_min, a.thr);
    const int NC = (a.T + a.D - 1) / a.D;
    const uint64_t lt = lanemask_lt();
    for (int64_t col = (int64_t)blockIdx.x * 4 + wave; col < a.cols; col += (int64_t)gridDim.x * 4) {
        const int32_t* const off = a.off + col * (NC + 1);
        auto clamped = [&](int c, int* s, int* e) {
            const int s0 = off[c], e0 = off[c + 1];
            *s = s0 < 0 ? 0 : (s0 > a.C_in ? a.C_in : s0);
            *e = e0 < *s ? *s : (e0 > a.C_in ? a.C_in : e0);
        };
        // entries past every chunk's end are not read
        int last = 0;
        for (int c = lane; c < NC; c += 64) {
            int s, e;
            clamped(c, &s, &e);
            last = e > s && e > last ? e : last;
        }
        for (int o = 32; o > 0; o >>= 1) {
            const int x = __shfl_xor(last, o, 64);
            last = x > last ? x : last;
        }
        int base = 0;
        for (int p0 = 0; p0 < last; p0 += 64) {
            const int p = p0 + lane;
            bool ev = p < last;
            int ci = 0, tb = 0;
            float t = 0.0f;
            if (ev) {
                ci = a.cin[col * a.C_in + p];
                t = a.tin[col * a.C_in + p];
                tb = (int)floorf(t - a.tfs);
                if (tb < 0) tb = 0;
                ev = tb < a.T && (unsigned)ci < (unsigned)a.C_in;
            }
            if (ev) {
                int s, e;
                clamped(tb / a.D, &s, &e);
                ev = p >= s && p < e;
            }
            const uint64_t m = __ballot(ev);
            if (ev)
                a.late[col * a.C_in + base + __popcll(m & lt)] =
                    make_int2(ci | (tb << 16), __float_as_int(a.alpha[alpha_index(t, tb, a.alpha_by_time, a.T)]));
            base += __popcll(m);
        }
        if (lane == 0) a.cnt[col] = base;
    }
}

// ---------------------------------------------------------------------------
// Bin 0 as an implicit GEMM: out[pixel][c_out] = sum over (tap, cin) in order
// of a0[column of the tap][cin] * W[tap * C_in + cin][c_out], one fma per
// element in that order (v_mfma_f32_32x32x2 adds its two products, and
// v_mfma_f32_16x16x4 its four, in k order).  A wave owns RT x CT tiles of
// MF x MF (pixels x c_out); four waves of a workgroup take consecutive pixels
// of one c_out block, so its weight rows meet in L1.  Operands come straight
// from the caches to registers, NS groups of KG elements ahead, without LDS
// staging or barriers.
//
// The sums cannot be split along the elements, so a wave's time is its chain:
// 32 cycles an element for a 32x32 tile, 8 for a 16x16 tile.  Where the tiles
// fill the chip the large ones need the fewest loads per product; where they
// do not, the small ones finish first (gemm0_config).
struct Gemm0Args {
    const float* a0;
    const float* W;
    float* out;
    int n_pix, B, H_in, W_in, C_in, Cp, H_out, W_out, C_out, K_h, K_w, pad_h, pad_w;
    int pos_major;  // rows in (position, image) order: a wave's pixels share their out-of-map taps
    int a_bytes, w_bytes, rowbytes, n_mt, n_nt;
    FastDiv div_w, div_h, div_b;
};

constexpr int kOob = 0x7fffff00;  // past every buffer: the load returns 0

template <int MF, int RT, int CT, int NS, bool EVEN>
__global__ __launch_bounds__(256) void k_gemm0(Gemm0Args a) {
    constexpr int HL = 64 / MF;  // elements per instruction
    constexpr int KG = 4 * HL;   // elements per group: four instructions of each tile
    constexpr int NR = MF == 32 ? 16 : 4;
    typedef typename std::conditional<MF == 32, f16v, f4>::type Acc;
    const int lane = lane_id(), wave = uniform(threadIdx.x >> 6);
    const int h = lane / MF, l = lane % MF;
    // c_out block and pixel block: block b takes c_out block b % n_nt, and
    // where that leaves several XCDs per c_out block each takes a contiguous
    // range of the pixels
    const int bi = blockIdx.x;
    const int j = bi / a.n_nt;
    const int S = (8 % a.n_nt == 0) ? 8 / a.n_nt : 1;
    const int mbr = j % S, per = a.n_mt / S, rem = a.n_mt - per * S;
    const int mt = mbr * per + (mbr < rem ? mbr : rem) + j / S;
    const int n0 = (bi - j * a.n_nt) * (MF * CT);
    const int m0 = (mt * 4 + wave) * MF * RT;
    if (m0 >= a.n_pix) return;  // uniform; no barriers below
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)a.a0, (short)0, a.a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)a.W, (short)0, a.w_bytes, 0x00020000);
    int hi0[RT], wi0[RT], base[RT];  // input row and column of tap (0, 0), and its column index
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int m = m0 + MF * i + l;
        int img, ho, wo;
        if (a.pos_major) {
            const int pos = fdiv(m, a.div_b);
            img = m - pos * a.B;
            ho = fdiv(pos, a.div_w);
            wo = pos - ho * a.W_out;
        } else {
            const int q = fdiv(m, a.div_w);
            wo = m - q * a.W_out;
            img = fdiv(q, a.div_h);
            ho = q - img * a.H_out;
        }
        hi0[i] = m < a.n_pix ? ho - a.pad_h : -(1 << 20);  // no tap of a row past the end is in the map
        wi0[i] = wo - a.pad_w;
        base[i] = (img * a.H_in + ho - a.pad_h) * a.W_in + wi0[i];
    }
    const int taps = a.K_h * a.K_w;
    auto in_map = [&](int i, int kh, int kw) {
        return hi0[i] + kh >= 0 && hi0[i] + kh < a.H_in && wi0[i] + kw >= 0 && wi0[i] + kw < a.W_in;
    };
    unsigned mask = 0;  // taps that some pixel of the wave has in its map
    for (int t = 0, kh = 0, kw = 0; t < taps; ++t) {
        bool any = false;
#pragma unroll
        for (int i = 0; i < RT; ++i) any |= in_map(i, kh, kw);
        if (__ballot(any) != 0) mask |= 1u << t;
        if (++kw == a.K_w) {
            kw = 0;
            ++kh;
        }
    }
    const int n_grp = __popc(mask) * (a.Cp / KG);
    int va[RT], sa = 0, sb = 0;
    const int a_end = a.Cp * 4;
    const int vb = h * a.rowbytes + n0 * 4 + (EVEN ? 4 * CT : 4) * l;
    auto next_tap = [&]() __attribute__((always_inline)) {
        if (mask == 0) {  // past the last group: zeros
#pragma unroll
            for (int i = 0; i < RT; ++i) va[i] = kOob;
            sa = 0;
            sb = 0;
            return;
        }
        const int t = __ffs(mask) - 1;
        mask &= mask - 1;
        const int kh = t / a.K_w, kw = t - kh * a.K_w;
#pragma unroll
        for (int i = 0; i < RT; ++i)
            va[i] = in_map(i, kh, kw) ? (base[i] + kh * a.W_in + kw) * a_end + 16 * h : kOob;
        sa = 0;
        sb = t * a.C_in * a.rowbytes;
    };
    struct Set {
        f4 a[RT];
        float b[4][CT];
    };
    // Scalar offsets sa and sb stay inside the buffers; rows past the weights
    // (the padding of C_in) are out of range by the vector offset and load 0.
    int vq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) vq[q] = vb + HL * q * a.rowbytes;
    auto load_a = [&](Set& s) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const u4 x = __builtin_amdgcn_raw_buffer_load_b128(ra, va[i], sa, 0);
            s.a[i] = f4{__uint_as_float(x.x), __uint_as_float(x.y), __uint_as_float(x.z), __uint_as_float(x.w)};
        }
    };
    auto load_b = [&](Set& s, int q) __attribute__((always_inline)) {
        if constexpr (EVEN && CT == 2) {
            const auto x = __builtin_amdgcn_raw_buffer_load_b64(rw, vq[q], sb, 0);
            s.b[q][0] = __uint_as_float(x[0]);
            s.b[q][CT - 1] = __uint_as_float(x[1]);
        } else {
#pragma unroll
            for (int v = 0; v < CT; ++v)
                s.b[q][v] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rw, vq[q] + 4 * MF * v, sb, 0));
        }
    };
    auto advance = [&]() __attribute__((always_inline)) {
        sa += 4 * KG;
        sb += KG * a.rowbytes;
        if (sa == a_end) next_tap();
    };
    Acc acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int v = 0; v < CT; ++v)
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[i][v][r] = 0.0f;
    next_tap();
    Set s[NS];
#pragma unroll
    for (int u = 0; u < NS; ++u) {
#pragma unroll
        for (int q = 0; q < 4; ++q) load_b(s[u], q);
        load_a(s[u]);
        advance();
    }
    // The loads go between the matrix instructions (a wave issues in order,
    // and with one wave per SIMD all of them behind a group's last one would
    // leave the matrix unit idle: VGG-16 512 -> 512 on 4x4 at B=1, one 32x32 tile
    // a wave, 135 -> 110 us with its other kernels).
    for (int n = 0; n < n_grp; n += NS) {  // groups past n_grp hold zeros
#pragma unroll
        for (int u = 0; u < NS; ++u) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int i = 0; i < RT; ++i)
#pragma unroll
                    for (int v = 0; v < CT; ++v) {
                        if constexpr (MF == 32)
                            acc[i][v] = __builtin_amdgcn_mfma_f32_32x32x2f32(s[u].a[i][q], s[u].b[q][v], acc[i][v], 0, 0, 0);
                        else
                            acc[i][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[u].a[i][q], s[u].b[q][v], acc[i][v], 0, 0, 0);
                    }
                __builtin_amdgcn_sched_barrier(0);
                load_b(s[u], q);
                if (q == 3) {
                    load_a(s[u]);
                    advance();
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // lane (h, l) holds rows 8 (r / 4) + 4 h + r % 4 of column l
    const int co = n0 + (EVEN ? CT : 1) * l;
    const int hw = a.H_out * a.W_out;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int m = m0 + MF * i + 8 * (r >> 2) + 4 * h + (r & 3);
            if (m >= a.n_pix) continue;
            int pix = m;
            if (a.pos_major) {
                const int pos = fdiv(m, a.div_b);
                pix = (m - pos * a.B) * hw + pos;
            }
            float* o = a.out + (int64_t)pix * a.C_out + co;
            if constexpr (EVEN && CT == 2) {
                if (co < a.C_out) *reinterpret_cast<f2*>(o) = f2{acc[i][0][r], acc[i][CT - 1][r]};
            } else {
#pragma unroll
                for (int v = 0; v < CT; ++v)
                    if (co + MF * v < a.C_out) o[MF * v] = acc[i][v][r];
            }
        }
}

// ---------------------------------------------------------------------------
// The later bins: one workgroup per output pixel and group of c_out blocks.
// Its waves collect the pixel's later events from the columns' lists (a prefix
// sum over the taps' counts maps list positions to columns), sort them by bin
// in LDS (counts, scan, placement with LDS bit masks as ranks, each bin in
// element order), and stream them as k_stream_quad does, for 64 (GEO 4) or
// 128 (GEO 2) c_out each.  TB blocks of 64 bins.  A list past `cap`
// entries comes in windows.
struct LateArgs {
    const int2* late;
    const int32_t* cnt;
    const float* in;
    const float* alpha;
    const float* theta;
    const LateThr* thr;
    const float* bias;
    const float* W;
    float* out;
    int n_pix, T, t_min, alpha_by_time;
    float tfs;
    int H_in, W_in, C_in, H_out, W_out, C_out, K_h, K_w, pad_h, pad_w;
    int rowbytes, w_bytes, cap, n_cblk, n_grp;
    float decay, th;  // CuLIF
    FastDiv div_w, div_h;
};

// What k_late integrates: the later bins after k_gemm0's bin 0, or every bin
// from the lists (k_split without bin-0 factors), with the LUT-threshold or the
// CuLIF neuron.
enum LateMode { kLateBins, kLateAll, kLateCulif };

__host__ __device__ inline int late_entries(int cap) { return cap + kLatePad; }  // a multiple of 16
// counts, cursors (64 TB each) and rank masks (128 TB) of one wave
__host__ __device__ inline int late_wave_words(int tb) { return tb * (64 + 64 + 128); }
__host__ __device__ inline int late_words(int cap, int waves, int tb) {
    return late_entries(cap) / 2 + late_entries(cap) + waves * late_wave_words(tb) + 64 * tb + 4;
}

// Keeps the compiler from moving LDS accesses across this point without
// making the wave wait: a wave's LDS instructions execute in program order.
__device__ __forceinline__ void lds_fence() { asm volatile("" ::: "memory"); }

// Inclusive prefix sum over the lanes, in DPP adds.
__device__ __forceinline__ int dpp_incl_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}

// One pixel's neurons c_out co .. co + OWN - 1 by the reference's loop: bin
// by bin, the bin's events in element order, straight from the spike map.
template <int OWN>
__device__ __forceinline__ void slow_pixel(const LateArgs& a, int pix, int co) {
    const int lane = lane_id();
    const int taps = a.K_h * a.K_w;
    const int qd = fdiv(pix, a.div_w);
    const int w_out = pix - qd * a.W_out;
    const int img = fdiv(qd, a.div_h);
    const int h_out = qd - img * a.H_out;
    float carry[OWN], res[OWN];
    bool ok[OWN];
#pragma unroll
    for (int v = 0; v < OWN; ++v) {
        ok[v] = co + v < a.C_out;
        carry[v] = ok[v] ? a.bias[co + v] : 0.0f;
        res[v] = kInfTime;
    }
    for (int b = 0; b < a.T; ++b) {
        float acc[OWN];
#pragma unroll
        for (int v = 0; v < OWN; ++v) acc[v] = 0.0f;
        for (int s = 0; s < taps; ++s) {
            const int kh = s / a.K_w, kw = s - kh * a.K_w;
            const int hi = h_out - a.pad_h + kh, wi = w_out - a.pad_w + kw;
            if (hi < 0 || hi >= a.H_in || wi < 0 || wi >= a.W_in) continue;
            const float* src = a.in + (int64_t)((img * a.H_in + hi) * a.W_in + wi) * a.C_in;
            for (int c0 = 0; c0 < a.C_in; c0 += 64) {
                const float t = c0 + lane < a.C_in ? src[c0 + lane] : kInfTime;
                const int tb = split_bin(t, a.tfs, a.T);
                const float al = tb == b ? a.alpha[split_alpha(t, tb, a.alpha_by_time, a.T)] : 0.0f;
                for (uint64_t m = __ballot(tb == b); m != 0; m &= m - 1) {
                    const int i = __ffsll((unsigned long long)m) - 1;
                    const float f = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(al), i));
                    const float* w = a.W + (int64_t)(s * a.C_in + c0 + i) * a.C_out + co;
#pragma unroll
                    for (int v = 0; v < OWN; ++v)
                        if (ok[v]) acc[v] = __builtin_fmaf(w[v], f, acc[v]);
                }
            }
        }
        const float th = a.theta[b];
#pragma unroll
        for (int v = 0; v < OWN; ++v) {
            carry[v] = carry[v] + acc[v];
            if (res[v] == kInfTime && b >= a.t_min && carry[v] >= th && th >= 1e-5f) res[v] = (float)b;
        }
    }
#pragma unroll
    for (int v = 0; v < OWN; ++v)
        if (ok[v]) a.out[(int64_t)pix * a.C_out + co + v] = res[v];
}

template <int GEO, int TB, bool TAPS9, bool W1, LateMode MODE>
__global__ __launch_bounds__(W1 ? 64 : 64 * kLateMaxWaves) void k_late(LateArgs a) {
    constexpr int OWN = 4 / GEO;  // c_out per lane
    constexpr int LPG = 8 / GEO;  // loads per group of 8 events
    extern __shared__ __align__(16) int lds_words[];
    const int W = W1 ? 1 : blockDim.x >> 6;
    const int wave = W1 ? 0 : uniform(threadIdx.x >> 6);
    const int lane = lane_id();
    const int T = a.T;
    const int E = late_entries(a.cap);
    unsigned short* rows = reinterpret_cast<unsigned short*>(lds_words);
    int* alph = lds_words + E / 2;
    int* tables = lds_words + E / 2 + E;
    int* mine = tables + late_wave_words(TB) * wave;
    int* cur = mine + 64 * TB;
    unsigned* msk = reinterpret_cast<unsigned*>(mine + 128 * TB);
    const int q = GEO == 4 ? lane >> 4 : lane >> 5;
    const int r = GEO == 4 ? (lane & 15) : (lane & 31);
    // workgroup b: c_out group b % n_grp (an XCD integrates few groups, so its
    // L2 holds their weights); the XCDs of a group take contiguous pixels
    const int grp = blockIdx.x % a.n_grp, jb = blockIdx.x / a.n_grp;
    const int S = (8 % a.n_grp == 0) ? 8 / a.n_grp : 1;
    const int mbr = jb % S, per = a.n_pix / S, rem = a.n_pix - per * S;
    const int pix = mbr * per + (mbr < rem ? mbr : rem) + jb / S;
    const int cb = grp * W + wave;
    const int co = (GEO == 4 ? 4 * r + q : 4 * r + 2 * q) + cb * (64 * OWN);
    const int voff = 16 * r + cb * (256 * OWN);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a.W, (short)0, a.w_bytes, 0x00020000);
    // the taps: lane s < K_h K_w holds tap s's column and first list position
    const int taps = a.K_h * a.K_w;
    const int qd = fdiv(pix, a.div_w);
    const int w_out = pix - qd * a.W_out;
    const int img = fdiv(qd, a.div_h);
    const int h_out = qd - img * a.H_out;
    int col, n_ev = 0;
    {
        const int kh = lane / a.K_w, kw = lane - kh * a.K_w;
        const int hi = h_out - a.pad_h + kh, wi = w_out - a.pad_w + kw;
        col = (img * a.H_in + hi) * a.W_in + wi;
        if (lane < taps && hi >= 0 && hi < a.H_in && wi >= 0 && wi < a.W_in) n_ev = a.cnt[col];
    }
    float* const po = a.out + (int64_t)pix * a.C_out + co;
    bool ok[OWN];
    float carry[OWN], acc[OWN];  // acc starts as bin 0's sum
#pragma unroll
    for (int v = 0; v < OWN; ++v) {
        ok[v] = co + v < a.C_out;
        carry[v] = MODE != kLateCulif && ok[v] ? a.bias[co + v] : 0.0f;
        acc[v] = MODE == kLateBins && ok[v] ? po[v] : 0.0f;
    }
    float v_th[TB];
    float* const tht = reinterpret_cast<float*>(tables + late_wave_words(TB) * W) + 2;  // thresholds, two NaN each side
#pragma unroll
    for (int k = 0; k < TB; ++k) v_th[k] = MODE != kLateCulif ? a.thr->th[64 * k + lane] : 0.0f;
    {
        const int z = vzero();
#pragma unroll
        for (int i = 0; i < TB; ++i)  // counts, cursors, masks
            reinterpret_cast<int4*>(mine)[64 * i + lane] = make_int4(z, z, z, z);
    }
    if (MODE != kLateCulif && (W1 || wave == 0)) {
#pragma unroll
        for (int k = 0; k < TB; ++k) tht[64 * k + lane] = v_th[k];
        if (lane < 4) tht[lane < 2 ? lane - 2 : 64 * TB + lane - 2] = __builtin_nanf("");
    }
    const int incl_t = dpp_incl_scan(n_ev);
    const int total = __builtin_amdgcn_readlane(incl_t, 63);
    const int start = lane < taps ? incl_t - n_ev : INT_MAX;
    const int delta = col * a.C_in - (incl_t - n_ev);  // list position to index in `late` (in the map)
    // event at list position f (element order; past the end the last one):
    // {row | bin << 16, alpha}; its tap is the last one that starts at or
    // before f
    auto element = [&](int f) __attribute__((always_inline)) -> int2 {
        f = f < total ? f : total - 1;
        int k = 0;
        if constexpr (TAPS9) {
#pragma unroll
            for (int s = 1; s < 9; ++s) k += f >= __builtin_amdgcn_readlane(start, s) ? 1 : 0;
        } else {
            for (int s = 1; s < taps; ++s) k += f >= __builtin_amdgcn_readlane(start, s) ? 1 : 0;
        }
        int2 e = a.late[(int64_t)(__shfl(delta, k, 64) + f)];
        e.x += k * a.C_in;  // row below 2^16 (host check)
        return e;
    };
    if (MODE == kLateCulif && total == 0) {  // uniform over the workgroup
        // no input: I and V stay 0, so a neuron fires at step 0 when 0 >= th
        // (T3V:50-62) and never otherwise
#pragma unroll
        for (int v = 0; v < OWN; ++v)
            if (cb < a.n_cblk && ok[v]) po[v] = 0.0f >= a.th ? 0.0f : kInfTime;
        return;
    }
    const int n_chunks = (total + 63) >> 6;
    const int c_lo = W1 ? 0 : (int)((unsigned)(n_chunks * wave) / (unsigned)W);
    const int c_hi = W1 ? n_chunks : (int)((unsigned)(n_chunks * (wave + 1)) / (unsigned)W);
    lds_fence();
    // pass 1: events per bin; the first kLateKeep chunks stay in registers
    int2 keep[kLateKeep];
#pragma unroll
    for (int i = 0; i < kLateKeep; ++i) {
        keep[i] = make_int2(0, 0);
        if (c_lo + i < c_hi) keep[i] = element((c_lo + i) * 64 + lane);  // uniform
    }
#pragma unroll
    for (int i = 0; i < kLateKeep; ++i)
        if (c_lo + i < c_hi && (c_lo + i) * 64 + lane < total) atomicAdd(&mine[keep[i].x >> 16], 1);
    for (int c = c_lo + kLateKeep; c < c_hi; ++c) {
        const int2 e = element(c * 64 + lane);
        if (c * 64 + lane < total) atomicAdd(&mine[e.x >> 16], 1);
    }
    auto sync = [&]() __attribute__((always_inline)) {
        if constexpr (W1)
            wave_sync();
        else
            __syncthreads();
    };
    sync();
    // bin ends and this wave's cursors
    int v_end[TB], start_b[TB];
    {
        int run = 0;
#pragma unroll
        for (int k = 0; k < TB; ++k) {
            int tot = 0, below = 0;
            if constexpr (W1) {
                tot = mine[64 * k + lane];
            } else {
                for (int w2 = 0; w2 < W; ++w2) {
                    const int x = tables[late_wave_words(TB) * w2 + 64 * k + lane];
                    tot += x;
                    below += w2 < wave ? x : 0;
                }
            }
            const int incl = dpp_incl_scan(tot) + run;
            // the last event's bin and those after it stay open to the tail
            v_end[k] = incl < total ? incl : INT_MAX;
            start_b[k] = incl - tot + below;
            cur[64 * k + lane] = start_b[k];
            run = __builtin_amdgcn_readlane(incl, 63);
        }
    }
    const uint64_t lt = lanemask_lt();
    const unsigned bit = 1u << (lane & 31);
    // places a chunk's events whose position falls in [P0, P0 + cap)
    auto place_chunk = [&](int2 e, bool ev, int P0) __attribute__((always_inline)) {
        if (ev) {
            const int b = e.x >> 16;
            atomicOr(&msk[2 * b + (lane >> 5)], bit);
            lds_fence();
            const uint64_t mm = *reinterpret_cast<const uint64_t*>(&msk[2 * b]);
            const int at = cur[b];
            lds_fence();
            if ((mm >> lane) == 1ull) {  // the bin's last lane in this chunk
                atomicAdd(&cur[b], __popcll(mm));
                const int z = vzero();
                *reinterpret_cast<int2*>(&msk[2 * b]) = make_int2(z, z);
            }
            lds_fence();
            const int p = at + __popcll(mm & lt) - P0;
            if (p >= 0 && p < a.cap) {
                rows[p] = (unsigned short)e.x;
                alph[p] = e.y;
            }
        }
    };
    auto pad = [&](int P0) __attribute__((always_inline)) {
        const int n_w = total - P0 < a.cap ? total - P0 : a.cap;
        if ((W1 || wave == 0) && lane < kLatePad) {
            // a row past the weights (host check): its load returns 0
            rows[n_w + lane] = 0xFFFF;
            alph[n_w + lane] = vzero();
        }
    };
    lds_fence();
    pad(0);
#pragma unroll
    for (int i = 0; i < kLateKeep; ++i)
        if (c_lo + i < c_hi) place_chunk(keep[i], (c_lo + i) * 64 + lane < total, 0);  // uniform
    for (int c = c_lo + kLateKeep; c < c_hi; ++c) place_chunk(element(c * 64 + lane), c * 64 + lane < total, 0);
    sync();
    bool live = cb < a.n_cblk;  // waves past the last c_out block only help build
    int res[OWN];
    uint64_t alive[OWN];
#pragma unroll
    for (int v = 0; v < OWN; ++v) {
        res[v] = 0;
        alive[v] = __ballot(ok[v]);
    }
    int blk = 0, b = 0;  // open bin: b within block blk of 64
    float cur_i[OWN];     // the CuLIF current I
#pragma unroll
    for (int v = 0; v < OWN; ++v) cur_i[v] = 0.0f;
    float c_th = v_th[0];
    int c_end = v_end[0];
    int bend = __builtin_amdgcn_readlane(c_end, 0);
    constexpr bool AL_AHEAD = GEO == 4;
    struct Raw {
        u4 x[LPG];
        f4 al[AL_AHEAD ? 2 : 1];
    };
    auto load = [&](int j, Raw& g) __attribute__((always_inline)) {
        {
#pragma unroll
            for (int k = 0; k < LPG; ++k) {
                const int off = (int)__umul24((unsigned)rows[j + GEO * k + q], (unsigned)a.rowbytes) + voff;
                g.x[k] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0);
            }
        }
        if constexpr (AL_AHEAD) {
            g.al[0] = *reinterpret_cast<const f4*>(alph + j);
            g.al[1] = *reinterpret_cast<const f4*>(alph + j + 4);
        }
    };
    auto next_block = [&]() __attribute__((always_inline)) {
        ++blk;
        b = 0;
#pragma unroll
        for (int k = 1; k < TB; ++k)
            if (blk == k) {
                c_th = v_th[k];
                c_end = v_end[k];
            }
    };
    // closes one bin: against the standing carries, or one CuLIF step with the
    // bin's sum as its input (I = fma(I, decay, in); V += I)
    auto close_bin = [&]() __attribute__((always_inline)) {
        const float th = MODE == kLateCulif ? a.th : __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c_th), b));
#pragma unroll
        for (int v = 0; v < OWN; ++v) {
            if constexpr (MODE == kLateCulif) {
                cur_i[v] = __builtin_fmaf(cur_i[v], a.decay, acc[v]);
                acc[v] = 0.0f;
                carry[v] = carry[v] + cur_i[v];
            }
            alive[v] &= ~__ballot(carry[v] >= th);
            res[v] = add_lane_bit(res[v], alive[v]);
        }
        ++b;
    };
    // closes the bins before the one of the event at position p
    auto close_to = [&](int p) __attribute__((always_inline)) {
        if constexpr (MODE != kLateCulif) {
#pragma unroll
            for (int v = 0; v < OWN; ++v) {
                carry[v] = carry[v] + acc[v];
                acc[v] = 0.0f;
            }
        }
        if constexpr (TB > 1) {
            for (;;) {
                const int stop = __popcll(__builtin_amdgcn_ballot_w64(c_end <= p));
                while (b < stop) close_bin();
                if (b < 64) break;
                next_block();
            }
        } else {
            const int stop = __popcll(__builtin_amdgcn_ballot_w64(c_end <= p));
            do close_bin();
            while (b < stop);
        }
        bend = __builtin_amdgcn_readlane(c_end, b);
    };
    // integrates the events at positions j .. j + 7 (the list's padding adds
    // 0 * 0 to the last bin)
    auto consume = [&](int j, Raw& g) __attribute__((always_inline)) {
        float w[8][OWN], al[8];
#pragma unroll
        for (int k = 0; k < LPG; ++k) {
            unsigned c0 = g.x[k].x, c1 = g.x[k].y, c2 = g.x[k].z, c3 = g.x[k].w;
            auto p = __builtin_amdgcn_permlane32_swap(c0, c2, false, false);
            c0 = p[0];
            c2 = p[1];
            p = __builtin_amdgcn_permlane32_swap(c1, c3, false, false);
            c1 = p[0];
            c3 = p[1];
            if constexpr (GEO == 4) {
                p = __builtin_amdgcn_permlane16_swap(c0, c1, false, false);
                c0 = p[0];
                c1 = p[1];
                p = __builtin_amdgcn_permlane16_swap(c2, c3, false, false);
                c2 = p[0];
                c3 = p[1];
                w[4 * k + 0][0] = __uint_as_float(c0);
                w[4 * k + 1][0] = __uint_as_float(c1);
                w[4 * k + 2][0] = __uint_as_float(c2);
                w[4 * k + 3][0] = __uint_as_float(c3);
            } else {
                w[2 * k + 0][0] = __uint_as_float(c0);
                w[2 * k + 0][OWN - 1] = __uint_as_float(c1);
                w[2 * k + 1][0] = __uint_as_float(c2);
                w[2 * k + 1][OWN - 1] = __uint_as_float(c3);
            }
        }
        f4 a0, a1;
        if constexpr (AL_AHEAD) {
            a0 = g.al[0];
            a1 = g.al[AL_AHEAD ? 1 : 0];
        } else {
            a0 = *reinterpret_cast<const f4*>(alph + j);
            a1 = *reinterpret_cast<const f4*>(alph + j + 4);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            al[i] = a0[i];
            al[4 + i] = a1[i];
        }
        auto integ = [&](int i) __attribute__((always_inline)) {
#pragma unroll
            for (int v = 0; v < OWN; ++v) acc[v] = __builtin_fmaf(w[i][v], al[i], acc[v]);
        };
        if (bend >= j + 8) {  // all in the open bin
#pragma unroll
            for (int i = 0; i < 8; ++i) integ(i);
            return;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if (bend <= j + i) close_to(j + i);
            integ(i);
        }
    };
    // a NaN bin-0 sum: redone below
    bool redo = false;
    {
        bool nan = false;
#pragma unroll
        for (int v = 0; v < OWN; ++v) nan |= acc[v] != acc[v];
        redo = MODE == kLateBins && live && __ballot(nan) != 0;
    }
    Raw g0, g1;
    int P0 = 0;
    for (;;) {
        const bool more = total - P0 > a.cap;  // a window follows
        const int n_w = more ? a.cap : total - P0;
        if (live && n_w > 0) {
            load(0, g0);
            for (int j = 0;; j += 16) {
                load(j + 8, g1);
                __builtin_amdgcn_sched_barrier(0);
                consume(j, g0);
                if (j + 8 >= n_w) break;
                load(j + 16, g0);
                __builtin_amdgcn_sched_barrier(0);
                consume(j + 8, g1);
                uint64_t any = alive[0];
#pragma unroll
                for (int v = 1; v < OWN; ++v) any |= alive[v];
                live = any != 0;
                if (j + 16 >= n_w || !live) break;
            }
        }
        if (!more) break;  // uniform over the workgroup
        // the next window: cursors from the bins' starts again
        __syncthreads();  // every wave is done with this window
        P0 += a.cap;
#pragma unroll
        for (int k = 0; k < TB; ++k) {
            cur[64 * k + lane] = start_b[k];
            v_end[k] = v_end[k] != INT_MAX ? v_end[k] - a.cap : INT_MAX;
        }
        lds_fence();
        pad(P0);
        for (int c = c_lo; c < c_hi; ++c) place_chunk(element(c * 64 + lane), c * 64 + lane < total, P0);
        __syncthreads();
        c_end = v_end[0];
#pragma unroll
        for (int k = 1; k < TB; ++k)
            if (blk == k) c_end = v_end[k];
        bend = __builtin_amdgcn_readlane(c_end, b);
    }
    auto close_rest = [&]() __attribute__((always_inline)) {
        for (;;) {
            const int end = T - 64 * blk < 64 ? T - 64 * blk : 64;
            while (b < end) {
                close_bin();
                if constexpr (MODE == kLateCulif) {
                    uint64_t any = alive[0];
#pragma unroll
                    for (int v = 1; v < OWN; ++v) any |= alive[v];
                    if (any == 0) return;
                }
            }
            if (TB == 1 || 64 * blk + 64 >= T) return;
            next_block();
        }
    };
    if (MODE == kLateCulif) {
        if (live) close_rest();  // every step without input steps the neuron too
    } else if (live) {
        // The carries stand from the open bin on.  The first bin whose
        // threshold a carry reaches is guessed from the thresholds' slope and
        // taken where the thresholds around it bracket the carry; where one
        // does not (or the thresholds are not monotone) the bins close one by
        // one.  All bins one by one: 32 bins of a VGG-16 pixel's tail cost 96
        // vector and 220 scalar instructions.
#pragma unroll
        for (int v = 0; v < OWN; ++v) carry[v] = carry[v] + acc[v];
        const int b0 = 64 * blk + b;
        const int lo = a.thr->lo, hi = a.thr->hi;
        const float lg0 = a.thr->lg0, inv = a.thr->inv;
        bool bad = a.thr->mono == 0;
        const int lim = b0 > lo ? b0 : lo;
        int first[OWN];
        uint64_t fires[OWN];
#pragma unroll
        for (int v = 0; v < OWN; ++v) {
            const float c = carry[v];
            const float x = (lg0 - __builtin_amdgcn_logf(fmaxf(c, 1e-6f))) * inv + (float)lo;
            const int g = (int)ceilf(fminf(fmaxf(x, (float)lim), (float)hi));  // within [0, 64 TB]
            const bool f_2 = tht[g - 2] <= c && g - 2 >= lim, f_1 = tht[g - 1] <= c && g - 1 >= lim;
            const bool f0 = tht[g] <= c, f1 = tht[g + 1] <= c;
            first[v] = f_1 ? g - 1 : (f0 ? g : g + 1);
            const bool f = f_1 || f0 || f1;
            fires[v] = __ballot(f) & alive[v];
            bad |= __builtin_amdgcn_inverse_ballot_w64(alive[v]) && (f_2 || (!f && g + 2 < hi));
        }
        if (__ballot(bad) == 0) {
#pragma unroll
            for (int v = 0; v < OWN; ++v) {
                res[v] = __builtin_amdgcn_inverse_ballot_w64(fires[v]) ? first[v] : res[v];
                alive[v] &= ~fires[v];
            }
        } else {
            close_rest();
        }
    }
    if (cb < a.n_cblk) {
        if (redo) {
            slow_pixel<OWN>(a, pix, co);
        } else {
#pragma unroll
            for (int v = 0; v < OWN; ++v)
                if (ok[v]) po[v] = __builtin_amdgcn_inverse_ballot_w64(alive[v]) ? kInfTime : (float)res[v];
        }
    }
}

int ceil16(int c) { return (c + 15) & ~15; }
int64_t split_cols(const IntegShape& s) { return s.is_fc ? s.B : (int64_t)s.B * s.H_in * s.W_in; }
int64_t split_pix(const IntegShape& s) { return s.is_fc ? s.B : (int64_t)s.B * s.H_out * s.W_out; }

// k_gemm0's tiles: 0: 64 x 64 a wave (2 x 2 of 32x32), 1: 32 x 64, 2: 32 x 32, 3: 16 x 16, by the 32x32 tiles of
// the layer.
int64_t tiles32(int64_t pix, int c_out) { return ((pix + 31) / 32) * ((c_out + 31) / 32); }
int gemm0_config(int64_t pix, int c_out) {
    const int64_t tiles = tiles32(pix, c_out);
    return tiles >= 16384 ? 0 : (tiles >= 2048 ? 1 : (tiles >= 768 ? 2 : 3));
}
size_t align256(size_t n) { return (n + 255) & ~size_t(255); }

}  // namespace

// k_late's grid: a wave per pixel and 64 outputs, up to three idle ones in a
// group; a launch holds below 2^32 threads.
static bool late_grid_ok(int64_t pix, int C_out) {
    return pix < (INT64_C(1) << 31) - 1024 && pix * 64 * ((C_out + 63) / 64 + 3) < (INT64_C(1) << 32);
}

size_t split_scratch_bytes(const IntegShape& s) {
    const size_t cols = (size_t)split_cols(s);
    return align256(cols * ceil16(s.C_in) * 4) + align256(cols * s.C_in * 8) + align256(cols * 4) +
           align256(sizeof(LateThr));
}

bool split_ok(const vdttfs_ctx* ctx, const IntegShape& s, bool net) {
    const int T = ctx->c.T;
    const int taps = s.is_fc ? 1 : s.K_h * s.K_w;
    const int64_t cols = split_cols(s), pix = split_pix(s), K = (int64_t)taps * s.C_in;
    if (T > 128 || taps > kSplitMaxTaps || s.C_out < 32 || s.C_out > 16384) return false;
    // 16-bit weight rows in a list entry, row 0xFFFF past the weights; 32-bit buffer offsets
    if (K > 0xFFFF || K * s.C_out * 4 >= kOob) return false;
    if (cols * ceil16(s.C_in) * 4 >= kOob) return false;
    if (!late_grid_ok(pix, s.C_out)) return false;
    // Bin 0 collects the spikes up to the fire start: from a quarter of the
    // window on it holds enough of them that the dense sum beats the gather
    // (VGG-16's layers hold 70-85% there at half the window).
    if (!(ctx->c.tfs * 4.0f >= (float)T)) return false;
    // Three launches and the element chain of k_gemm0 (32 cycles an element,
    // 8 in 16x16 tiles) need work to hide under.  Where the fused kernels do
    // not serve (T > 64, or more than 9 taps: bucketize or dense merge and a
    // stream) that is any layer of a few inputs past nine taps, until the list
    // comes in many windows, each of which reads it from its start (times as
    // fast as merged lists at densities 0.1 / 0.3 / 0.7, T = 80: 64 outputs, 64
    // pixels, 2,750 elements 1.36 / 1.45 / 1.28, 3,750 1.08 / 1.08 / 0.93, 6,400
    // 0.93 / 0.98 / 0.61; two waves a list: 200 outputs, 512 pixels, 6,400 1.31 /
    // 1.56 / 1.48, but 4,096 pixels 5,000 0.89 / 1.13 and 3,750 1.00 / 1.19 / 1.34).
    if (taps > 9 && K > (s.C_out > 128 && pix <= 512 ? 6400 : 3750)) return false;
    if (T <= 64 && taps > 9) return K >= 4;
    // Past 64 steps the lists of every bin (two launches) are there as well and
    // finish first in short fields, where the split even lost to the kernels
    // before it (3x3, C_in 3, 64 outputs, T = 80, 1,024 pixels, us at densities
    // 0.1 / 0.7: dense merge and stream 11.9 / 16.0, split 14.9 / 15.4, lists
    // 8.4 / 9.2; times as fast as the split: 72 elements 1.75 / 1.6, 171 1.7 /
    // 1.35, 300 1.9 / 1.2, 576 1.7 / 1.06 there and 1.5 / 0.8 at 16K pixels), and
    // at one tap outside networks (1,500 elements, 128 outputs, 1,024 pixels:
    // split 0.92 / 1.61 times the speed of merged lists, lists 1.59 / 1.38).
    if (T > 64) return K > 300 && (net || (taps > 1 && (K > 576 || pix > 1024)));
    // Against the fused kernels: FC layers keep them (VGG-16's 512 -> 512 at
    // B=256: 28 against 34 us), and so do maps of up to 2x2 below 1,024
    // pixels, whose taps mostly fall outside (512 -> 512 at B=128: 54 against
    // 57 us; B=256: 98 -> 91).
    if (s.is_fc || (s.H_out * s.W_out <= 4 && pix < 1024)) return false;
    // The dense sum costs the same at any density, so the line depends on what
    // arrives, which the host does not see.
    const int64_t products = K * pix * s.C_out;
    if (net) {
        // Layers of a network: most of their inputs spike before the fire
        // start.  Past 10^8 products, or with long fields, which the fused
        // kernels stream one event after the other (VGG-16 at B=1: 128 -> 256
        // on 8x8 38 -> 29 us, 512 -> 512 on 4x4 1.2 to 1.4 times as fast).
        // Weights past an XCD's L2 (4 MB) come from the Infinity Cache once per
        // row of 16-pixel tiles, which costs more than the events where
        // neither pixels nor chains hide it (VGG-16 with its 4x4 layers split
        // against fused, us a pass alone and of three in flight: B=3 544 / 575,
        // 237 / 232; B=4 570 / 576, 258 / 237; B=8 585 / 584, 288 / 261; B=16
        // 645 / 645, 359 / 354; B=24 744 / 772, 469 / 485).
        if (K * s.C_out > (1 << 20) && pix > 48 && pix < 384) return false;
        return products >= 100000000 || (K >= 1024 && s.C_out > 64);
    }
    // Single layers, spikes spread over the window (half of them in bin 0):
    // from 768 tiles of 32x32 on, where k_gemm0 takes those (split against
    // fused, times as fast at densities 0.1 / 0.3 / 0.7, alone: 64 -> 64 at 16K
    // pixels 1.0 / 1.16 / 1.22, 128 -> 256 at 4K 0.83 / 1.06 / 1.27, 72 -> 100
    // at 8K 0.92 / 1.08 / 1.17, 64 -> 128 at 64K 1.07 / 1.25 / 1.32).  Below, with
    // 16x16 tiles, it loses at most densities (128 -> 128 at 4K 0.65 / 0.83 /
    // 1.02, at 1K 0.77 / 0.88 / 0.92; 190 -> 239 at 1K 0.72 / 0.94 / 1.14), more
    // with several passes in flight, and so do short chains (1x1, 128 -> 128 at
    // 8K 0.71 / 0.79 / 0.90) and, on fewer than 4,096 tiles, fire starts in the
    // window's first half (a quarter: 128 -> 256 at 8K 0.86 / 0.94 / 1.05).
    const int64_t tiles = tiles32(pix, s.C_out);
    if (tiles < 768 || products < 100000000) return false;
    if (K < 144 && products < 1000000000) return false;
    return ctx->c.tfs * 2.0f >= (float)T || tiles >= 4096;
}

namespace {

// Sizes k_late takes every bin of.
bool lists_fit(const vdttfs_ctx* ctx, const IntegShape& s) {
    const int T = ctx->c.T;
    const int taps = s.is_fc ? 1 : s.K_h * s.K_w;
    const int64_t cols = split_cols(s), pix = split_pix(s), K = (int64_t)taps * s.C_in;
    if (T > kSplitMaxT || taps > kSplitMaxTaps || s.C_out > 1024) return false;
    if (K > 0xFFFF || K * s.C_out * 4 >= kOob) return false;
    return cols * s.C_in * 4 < kOob && late_grid_ok(pix, s.C_out);
}

}  // namespace

// Layers the list form takes (k_split's lists with bin 0's events, then k_late
// over every bin) in place of bucketize or dense merge, k_merge and k_stream:
// windows past 64 steps, whose bins the fused kernels' lanes do not hold.
// Measured, three launches to two: CuLIF 64->128 at 32x32, T = 160, batch 33:
// 387 -> 190 us, 128->128 at 16x16: 321 -> 132; LeNet-5's FC layers at T = 80,
// batch 128: 113 -> 51.  At T = 64 the fused kernels win: CuLIF 64->128 at
// 128x128 2248 against 2460 us, LeNet-5's FC layers at batch 1024 45 against
// 51.  Layers narrower than a wave leave most of its lanes idle and still win
// past 64 steps (LeNet-5's conv2 at T = 80, 16 outputs: 37 -> 20 us for one
// image, 48 -> 37 for 128); at T = 64
// the register and narrow kernels do (batch 1024: conv1 145 against 567 us,
// conv2 169 against 169).  Each group of four c_out blocks rebuilds a pixel's
// list, so layers past 1024 outputs keep the merged lists.
//
// So do long lists: one past `cap` entries is read from its start for every
// window of it, where the merged lists are read once.  Times as fast as those,
// T = 80: FC to 64 outputs, 30 images, densities 0.05 / 0.2 / 0.5: 2,500 inputs
// 1.32 / 1.42 / 1.39, 4,096 1.17 / 1.35 / 0.97; one image to 10 outputs 2,500 1.23 /
// 1.15 / 0.97, 4,096 1.04 / 0.98 / 0.77; 128 outputs, 32 images, densities 0.05 /
// 0.3 / 1: 8,192 1.01 / 0.91 / 0.67, 16,384 0.83 / 0.86 / 0.42; 1,000 outputs, 32
// images, 8,192 0.96 / 1.45 / 1.34, 256 images 0.81 at 0.05.  3x3, 512 channels,
// 1,024 pixels, densities 0.1 / 0.7: 128 outputs 1.84 / 1.11, 512 outputs 1.20 /
// 0.65.  5x5 (each entry's tap is found among 25), 512 pixels, densities 0.1 / 0.3 /
// 0.7: 64 outputs 2,750 elements 2.41 / 1.42 / 0.71, 3,750 2.15 / 1.08 / 0.48; 200
// outputs 3,750 2.53 / 1.68 / 0.93, 5,000 2.42 / 1.43 / 0.80, 6,400 2.00 / 1.18 / 0.68.
bool lists_ok(const vdttfs_ctx* ctx, const IntegShape& s) {
    if (ctx->c.T <= 64 || !lists_fit(ctx, s)) return false;
    const int taps = s.is_fc ? 1 : s.K_h * s.K_w, K = taps * s.C_in;
    if (taps > 9) return K <= (s.C_out > 128 ? 5000 : 3200);
    if (taps > 1) return K <= (s.C_out > 128 ? 2304 : 4096);
    return K <= (s.C_out > 128 && split_pix(s) <= 64 ? 8192 : 4096);
}

int split_choice(const vdttfs_ctx* ctx, const IntegShape& s, bool net) {
    // (up to 64 steps fields of at most 32 elements have a plan of their own)
    if (conv_px_ok(ctx->c.T, s) && s.K_h * s.K_w <= kSplitMaxTaps && (ctx->c.T > 64 || s.K_h * s.K_w * s.C_in > 32))
        return kSplitPixel;
    if (split_ok(ctx, s, net)) return kSplitDense;
    return lists_ok(ctx, s) ? kSplitLists : 0;
}

// Over the reference's buckets the other way is the loop nest, which the lists
// beat up to 16,384 elements whatever arrives (all inputs active, 32 columns, 10
// outputs: 8,192 3.2 times as fast, 16,384 1.9, 32,768 1.0; one column 1.3, 0.7).
bool ref_lists_ok(const vdttfs_ctx* ctx, const IntegShape& s) {
    return lists_fit(ctx, s) && (s.is_fc ? 1 : s.K_h * s.K_w) * s.C_in <= 16384;
}

namespace {

// k_late's launch over the lists in `late` and `cnt`.
struct LateScratch {
    int2* late;
    int32_t* cnt;
    LateThr* thr;
};

void carve(void* scratch, int64_t cols, int C_in, LateScratch* sc) {
    unsigned char* sp = static_cast<unsigned char*>(scratch);
    sc->late = reinterpret_cast<int2*>(sp);
    sp += align256((size_t)cols * C_in * 8);
    sc->cnt = reinterpret_cast<int32_t*>(sp);
    sp += align256((size_t)cols * 4);
    sc->thr = reinterpret_cast<LateThr*>(sp);
}

template <LateMode MODE>
int launch_late(vdttfs_ctx* ctx, float* out, const float* in, const float* alpha, const LateScratch& sc, const float* W,
                const float* bias, const float* theta, int t_min, const IntegShape& s, const CulifNeuron* culif) {
    const int taps = s.is_fc ? 1 : s.K_h * s.K_w;
    const int64_t pix = split_pix(s);
    LateArgs l{};
    l.late = sc.late;
    l.cnt = sc.cnt;
    l.thr = sc.thr;
    l.in = in;
    l.alpha = alpha;
    l.theta = theta;
    l.bias = bias;
    l.W = W;
    l.out = out;
    l.n_pix = (int)pix;
    l.T = ctx->c.T;
    l.t_min = t_min;
    l.alpha_by_time = ctx->c.alpha_by_time;
    l.tfs = ctx->c.tfs;
    l.H_in = s.H_in;
    l.W_in = s.W_in;
    l.C_in = s.C_in;
    l.H_out = s.H_out;
    l.W_out = s.W_out;
    l.C_out = s.C_out;
    l.K_h = s.is_fc ? 1 : s.K_h;
    l.K_w = s.is_fc ? 1 : s.K_w;
    l.pad_h = s.pad_h;
    l.pad_w = s.pad_w;
    l.rowbytes = s.C_out * 4;
    l.w_bytes = taps * s.C_in * s.C_out * 4;
    l.div_w = make_fastdiv(s.W_out);
    l.div_h = make_fastdiv(s.H_out);
    if (culif) {
        l.decay = culif->decay;
        l.th = culif->th;
    }
    const int geo = s.C_out % 4 != 0 || s.C_out <= 64 ? 4 : 2;
    const int cw = 256 / geo;
    l.n_cblk = (s.C_out + cw - 1) / cw;
    // waves that share a list: two keep an XCD's c_out group, and so the
    // weights in its L2, small (VGG-16's 512-wide layers, four waves: 294 ->
    // 311 us); the list form's longer lists are built by four
    const int most = MODE == kLateBins ? 2 : kLateMaxWaves;
    const int waves = l.n_cblk < most ? l.n_cblk : most;
    l.n_grp = (l.n_cblk + waves - 1) / waves;
    // list entries of a window: past the events of a usual field (later bins:
    // a ninth of its elements in VGG-16), and LDS for 32 waves per CU
    const int nel = taps * s.C_in;
    const int nel_pad = (nel + 15) & ~15;
    int cap = waves > 1 ? 640 : (nel > 1152 ? 512 : (MODE == kLateBins ? 192 : 320));
    if (cap > nel_pad) cap = nel_pad;
    l.cap = cap;
    const int tb = l.T > 128 ? 4 : (l.T > 64 ? 2 : 1);
    const size_t lds = (size_t)late_words(cap, waves, tb) * 4;
    const int64_t lb = pix * l.n_grp;
    if (lb > 0x7fffffff) return set_error(VDTTFS_E_UNSUPPORTED, "integrate: grid too large");
#define VD_LATE(G, TBK, T9)                                                                                          \
    do {                                                                                                             \
        if (waves == 1)                                                                                              \
            hipLaunchKernelGGL((k_late<G, TBK, T9, true, MODE>), dim3((unsigned)lb), dim3(64), lds, ctx->stream, l); \
        else                                                                                                         \
            hipLaunchKernelGGL((k_late<G, TBK, T9, false, MODE>), dim3((unsigned)lb), dim3(64 * waves), lds,         \
                               ctx->stream, l);                                                                      \
    } while (0)
#define VD_LATE_T(G, TBK)           \
    do {                            \
        if (taps <= 9)              \
            VD_LATE(G, TBK, true);  \
        else                        \
            VD_LATE(G, TBK, false); \
    } while (0)
#define VD_LATE_G(G)         \
    do {                     \
        if (tb == 1)         \
            VD_LATE_T(G, 1); \
        else if (tb == 2)    \
            VD_LATE_T(G, 2); \
        else if constexpr (MODE != kLateBins) \
            VD_LATE_T(G, 4); \
    } while (0)
    if (geo == 4)
        VD_LATE_G(4);
    else
        VD_LATE_G(2);
#undef VD_LATE_G
#undef VD_LATE_T
#undef VD_LATE
    VD_HIP(hipGetLastError());
    return VDTTFS_OK;
}

int launch_split(vdttfs_ctx* ctx, const SplitArgs& k) {
    int seg = 3;
    while ((1 << seg) < k.Cp && seg < 6) ++seg;
    const int64_t per_block = 4 * (64 >> seg);
    int64_t blocks = (k.cols + per_block - 1) / per_block;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_split, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, k, seg);
    VD_HIP(hipGetLastError());
    return VDTTFS_OK;
}

}  // namespace

int launch_integrate_ref_lists(vdttfs_ctx* ctx, float* out, const int32_t* cin, const float* tin, const int32_t* off,
                               void* scratch, const float* W, const float* bias, const float* alpha,
                               const float* theta, int t_min, const IntegShape& s) {
    const int64_t cols = split_cols(s);
    if (cols == 0 || split_pix(s) == 0) return VDTTFS_OK;
    LateScratch sc;
    carve(scratch, cols, s.C_in, &sc);
    RefListArgs a{cin, tin, off, sc.late, sc.cnt, alpha, theta, sc.thr, cols, s.C_in, ctx->c.T, ctx->c.delta,
                  ctx->c.alpha_by_time, t_min, ctx->c.tfs};
    int64_t blocks = (cols + 3) / 4;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_ref_lists, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, a);
    VD_HIP(hipGetLastError());
    return launch_late<kLateAll>(ctx, out, nullptr, alpha, sc, W, bias, theta, t_min, s, nullptr);
}

int launch_integrate_lists(vdttfs_ctx* ctx, float* out, const float* in, const float* alpha, void* scratch,
                           const float* W, const float* bias, const float* theta, int t_min, const IntegShape& s,
                           const CulifNeuron* culif) {
    const int64_t cols = split_cols(s);
    if (cols == 0 || split_pix(s) == 0) return VDTTFS_OK;
    LateScratch sc;
    carve(scratch, cols, s.C_in, &sc);
    VD_TRY(launch_split(ctx, SplitArgs{in, nullptr, sc.late, sc.cnt, alpha, theta, sc.thr, cols, s.C_in, s.C_in,
                                       ctx->c.T, ctx->c.alpha_by_time, t_min, 1, ctx->c.tfs}));
    if (culif) return launch_late<kLateCulif>(ctx, out, in, alpha, sc, W, bias, theta, t_min, s, culif);
    return launch_late<kLateAll>(ctx, out, in, alpha, sc, W, bias, theta, t_min, s, nullptr);
}

int launch_integrate_split(vdttfs_ctx* ctx, float* out, const float* in, const float* alpha, void* scratch,
                           const float* W, const float* bias, const float* theta, int t_min, const IntegShape& s) {
    const int64_t cols = split_cols(s), pix = split_pix(s);
    const int taps = s.is_fc ? 1 : s.K_h * s.K_w;
    if (cols == 0 || pix == 0) return VDTTFS_OK;
    const int cfg = gemm0_config(pix, s.C_out);
    const int mf = cfg == 3 ? 16 : 32, rt = cfg == 0 ? 2 : 1, ct = cfg < 2 ? 2 : 1;
    const int Cp = mf == 16 ? ceil16(s.C_in) : (s.C_in + 7) & ~7;
    unsigned char* sp = static_cast<unsigned char*>(scratch);
    float* a0 = reinterpret_cast<float*>(sp);
    LateScratch sc;
    carve(sp + align256((size_t)cols * ceil16(s.C_in) * 4), cols, s.C_in, &sc);
    VD_TRY(launch_split(ctx, SplitArgs{in, a0, sc.late, sc.cnt, alpha, theta, sc.thr, cols, s.C_in, Cp, ctx->c.T,
                                       ctx->c.alpha_by_time, t_min, mf == 16 ? 2 : 1, ctx->c.tfs}));

    Gemm0Args g{};
    g.a0 = a0;
    g.W = W;
    g.out = out;
    g.n_pix = (int)pix;
    g.B = s.B;
    g.H_in = s.H_in;
    g.W_in = s.W_in;
    g.C_in = s.C_in;
    g.Cp = Cp;
    g.H_out = s.H_out;
    g.W_out = s.W_out;
    g.C_out = s.C_out;
    g.K_h = s.is_fc ? 1 : s.K_h;
    g.K_w = s.is_fc ? 1 : s.K_w;
    g.pad_h = s.pad_h;
    g.pad_w = s.pad_w;
    g.a_bytes = (int)(cols * Cp * 4);
    g.rowbytes = s.C_out * 4;
    g.w_bytes = taps * s.C_in * s.C_out * 4;
    g.div_w = make_fastdiv(s.W_out);
    g.div_h = make_fastdiv(s.H_out);
    g.div_b = make_fastdiv(s.B);
    g.pos_major = taps > 1 && s.H_out * s.W_out <= 64 && s.B >= mf;
    g.n_nt = (s.C_out + mf * ct - 1) / (mf * ct);
    const int rows = 4 * mf * rt;
    g.n_mt = (int)((pix + rows - 1) / rows);
    const int64_t gb = (int64_t)g.n_mt * g.n_nt;
    if (gb > 0x7fffffff) return set_error(VDTTFS_E_UNSUPPORTED, "integrate: grid too large");
    const bool even = s.C_out % 2 == 0;
#define VD_GEMM0(MF, RT, CT, NS)                                                                                  \
    do {                                                                                                          \
        if (even)                                                                                                 \
            hipLaunchKernelGGL((k_gemm0<MF, RT, CT, NS, true>), dim3((unsigned)gb), dim3(256), 0, ctx->stream, g);  \
        else                                                                                                      \
            hipLaunchKernelGGL((k_gemm0<MF, RT, CT, NS, false>), dim3((unsigned)gb), dim3(256), 0, ctx->stream, g); \
    } while (0)
    if (cfg == 0)
        VD_GEMM0(32, 2, 2, 2);
    else if (cfg == 1)
        VD_GEMM0(32, 1, 2, 4);
    else if (cfg == 2)
        VD_GEMM0(32, 1, 1, 6);
    else
        VD_GEMM0(16, 1, 1, 8);
#undef VD_GEMM0
    VD_HIP(hipGetLastError());

    return launch_late<kLateBins>(ctx, out, in, alpha, sc, W, bias, theta, t_min, s, nullptr);
}

}  // namespace vdttfs
