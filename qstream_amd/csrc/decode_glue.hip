// decode_glue.hip - the per-layer work around the matvecs of a batch-1
// decode step, on gfx950, so a device-resident engine needs no host round
// trip between its projections (src/engine.c:709-1187):
//   RMS / layer norm          src/kernels_scalar.c:148-185 (engine.c:805-815)
//   RoPE                      apply_rope, src/engine.c:204-235
//   int8 KV-cache store       kv_cache_store, src/engine.c:240-300
//   attention over the cache  src/engine.c:879-923
//   activation x up           src/engine.c:1128-1140
//   residual add + NaN check  src/engine.c:1172-1187
//   embedding row             src/engine.c:709-765
// Where the reference's result is integer (int8 KV codes) or follows one
// fixed sequence of fp32 roundings (KV scales, embedding values, the
// residual add) the kernels use the same operations in the same order with
// explicitly rounded multiplies and adds, so they match bit for bit; sums
// the kernels spread over lanes differ only in fp32 rounding order.
#include "qsf_device.h"
#include "qsf_hip_internal.h"

namespace {

constexpr int NORM_THREADS = 1024;

__device__ __forceinline__ float block_sum(float v, float* red) { return qsf::wg_sum(v, red); }

// RMS norm (LAYER = false) or layer norm over one vector of `dim` floats,
// one workgroup.  Output rounding order as src/kernels_scalar.c:148-185:
// (x * inv) * w, and (x - mean) * inv_std * w + b.
template <bool LAYER>
__global__ __launch_bounds__(NORM_THREADS) void norm_kernel(const float* __restrict__ in, float* out,
                                                            const float* __restrict__ w,
                                                            const float* __restrict__ b, int dim,
                                                            float eps) {
    __shared__ float red[NORM_THREADS / 64];
    if (!LAYER) {
        float ss = 0.f;
        for (int i = threadIdx.x; i < dim; i += blockDim.x) ss = fmaf(in[i], in[i], ss);
        ss = block_sum(ss, red);
        const float inv = __fdiv_rn(1.0f, __fsqrt_rn(qsf::add_rn(__fdiv_rn(ss, (float)dim), eps)));
        for (int i = threadIdx.x; i < dim; i += blockDim.x) out[i] = qsf::mul_rn(qsf::mul_rn(in[i], inv), w[i]);
    } else {
        float s = 0.f;
        for (int i = threadIdx.x; i < dim; i += blockDim.x) s += in[i];
        const float mean = __fdiv_rn(block_sum(s, red), (float)dim);
        float v = 0.f;
        for (int i = threadIdx.x; i < dim; i += blockDim.x) {
            const float d = in[i] - mean;
            v = fmaf(d, d, v);
        }
        const float var = __fdiv_rn(block_sum(v, red), (float)dim);
        const float inv = __fdiv_rn(1.0f, __fsqrt_rn(qsf::add_rn(var, eps)));
        for (int i = threadIdx.x; i < dim; i += blockDim.x) {
            float o = qsf::mul_rn(qsf::mul_rn(qsf::sub_rn(in[i], mean), inv), w[i]);
            if (b) o = qsf::add_rn(o, b[i]);
            out[i] = o;
        }
    }
}

// RoPE: one thread per (head, pair).  freq[j] = 1 / powf(theta, 2j/hd) is
// computed by the host C library once (qsf_hip_rope_create), so every
// angle position * freq matches the reference's; the angle is reduced in
// double as there, then rotated in fp32.
__global__ __launch_bounds__(256) void rope_kernel(float* q, float* k, const float* __restrict__ freq,
                                                   int head_dim, int nq_pairs, int nk_pairs,
                                                   int position) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nq_pairs + nk_pairs) return;
    float* v = t < nq_pairs ? q + 2 * t : k + 2 * (t - nq_pairs);
    const int j = (t < nq_pairs ? t : t - nq_pairs) % (head_dim / 2);
    double ang = (double)position * (double)freq[j];
    ang = fmod(ang, 2.0 * 3.14159265358979323846);
    const float c = cosf((float)ang), s = sinf((float)ang);
    const float a0 = v[0], a1 = v[1];
    v[0] = qsf::sub_rn(qsf::mul_rn(a0, c), qsf::mul_rn(a1, s));
    v[1] = qsf::add_rn(qsf::mul_rn(a0, s), qsf::mul_rn(a1, c));
}

// int8 KV store: one wave per (kv head, K or V).  absmax, scale =
// amax / 127, codes = trunc(clamp(x * (127 / amax)) +- 0.5) with every
// operation rounded as in src/engine.c:252-296: bit-exact.
__global__ __launch_bounds__(64) void kv_store_kernel(int8_t* kc, int8_t* vc, float* ks, float* vs,
                                                      const float* __restrict__ k,
                                                      const float* __restrict__ v, int max_seq,
                                                      int head_dim, int position) {
    const int h = blockIdx.x >> 1, isv = blockIdx.x & 1, lane = threadIdx.x;
    const float* src = (isv ? v : k) + (size_t)h * head_dim;
    const size_t row = (size_t)h * max_seq + position;
    int8_t* dst = (isv ? vc : kc) + row * head_dim;
    float amax = 0.f;
    for (int i = lane; i < head_dim; i += 64) {
        const float a = src[i] < 0 ? -src[i] : src[i];
        amax = a > amax ? a : amax;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float o = __shfl_xor(amax, off, 64);
        amax = o > amax ? o : amax;
    }
    if (lane == 0) (isv ? vs : ks)[row] = __fdiv_rn(amax, 127.0f);
    if (amax > 1e-30f) {
        const float inv = __fdiv_rn(127.0f, amax);
        for (int i = lane; i < head_dim; i += 64) {
            float x = qsf::mul_rn(src[i], inv);
            if (x > 127.0f) x = 127.0f;
            if (x < -127.0f) x = -127.0f;
            dst[i] = (int8_t)(int)qsf::add_rn(x, x >= 0 ? 0.5f : -0.5f);
        }
    } else {
        for (int i = lane; i < head_dim; i += 64) dst[i] = 0;
    }
}

// Attention over positions 0..position, split over positions so a short
// decode step still fills the chip: workgroup (head, chunk) handles
// ATT_CHUNK positions and leaves its local max m, its sum l of
// exp(score - m) and its unnormalised output o[d] = sum exp(score - m) *
// v_scale * v[d] in the workspace; attention_combine_kernel rescales the
// chunks to the global max and normalises.  This is the reference's
// softmax(q . k * scale / sqrt(hd)) . v (src/engine.c:879-923), regrouped:
// the fp32 sums run in a different order.
constexpr int ATT_THREADS = 256;
constexpr int ATT_CHUNK = 128;
constexpr int ATT_MAX_SEQ = QK_ATT_MAX_SEQ;
constexpr int ATT_FILL = 256;                            // workgroups that fill the CUs
typedef uint32_t att_u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float sbyte(uint32_t w, int i) {
    return (float)(int8_t)(uint8_t)(w >> (8 * i));
}

__global__ __launch_bounds__(ATT_THREADS) void attention_part_kernel(
    const float* __restrict__ q, const int8_t* __restrict__ kc, const int8_t* __restrict__ vc,
    const float* __restrict__ ks, const float* __restrict__ vs, int max_seq, int groups,
    int head_dim, int seq, int nsplit, float* __restrict__ ws) {
    __shared__ float qs[256];
    __shared__ float ew[ATT_CHUNK];                      // exp(score - m) * v_scale per position
    __shared__ float parts[ATT_THREADS];
    __shared__ float red[ATT_THREADS / 64];
    const int h = blockIdx.x, chunk = blockIdx.y, kvh = h / groups, t = threadIdx.x;
    const int p0 = chunk * ATT_CHUNK, np = min(ATT_CHUNK, seq - p0);
    for (int d = t; d < head_dim; d += ATT_THREADS) qs[d] = q[(size_t)h * head_dim + d];
    __syncthreads();
    // scores: one thread per position; the row's int8 codes 16 at a time
    const float inv_sqrt_d = __fdiv_rn(1.0f, __fsqrt_rn((float)head_dim));
    float sc = -INFINITY;
    if (t < np) {
        const size_t row = (size_t)kvh * max_seq + p0 + t;
        const att_u32x4* kr = reinterpret_cast<const att_u32x4*>(kc + row * head_dim);
        const float kscale = ks[row];
        float dot = 0.f;
        for (int c = 0; c < head_dim / 16; c++) {
            const att_u32x4 w = kr[c];
#pragma unroll
            for (int j = 0; j < 16; j++)
                dot = fmaf(qs[16 * c + j], qsf::mul_rn(sbyte(w[j >> 2], j & 3), kscale), dot);
        }
        sc = qsf::mul_rn(dot, inv_sqrt_d);
    }
    float m = sc;
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float e = t < np ? expf(sc - m) : 0.f;
    if (t < np) ew[t] = qsf::mul_rn(e, vs[(size_t)kvh * max_seq + p0 + t]);
    const float l = block_sum(e, red);                   // also orders the ew writes
    // weighted V: thread (d, part) over positions part, part + P, ...
    const int P = ATT_THREADS / head_dim, d = t % head_dim, part = t / head_dim;
    float acc = 0.f;
    if (part < P) {
        const int8_t* vr = vc + ((size_t)kvh * max_seq + p0) * head_dim + d;
        for (int p = part; p < np; p += P) acc = fmaf(ew[p], (float)vr[(size_t)p * head_dim], acc);
    }
    parts[t] = acc;
    __syncthreads();
    float* rec = ws + ((size_t)h * nsplit + chunk) * (head_dim + 2);
    if (t < head_dim) {
        float o = 0.f;
        for (int i = 0; i < P; i++) o += parts[i * head_dim + t];
        rec[2 + t] = o;
    }
    if (t == 0) {
        rec[0] = m;
        rec[1] = l;
    }
}

// gate = act(gate) * up (QSFActivation: 2 SiLU, 0/1 GELU tanh form, else
// ReLU), src/kernels_scalar.c:129-147 and src/engine.c:1128-1140.
__global__ __launch_bounds__(256) void act_mul_kernel(float* gate, const float* __restrict__ up,
                                                      int n, int act) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    gate[i] = qsf::act_mul(act, gate[i], up[i]);
}

// res += x, then the first index whose value is NaN or beyond +-1e30 (or
// -1) into *bad when bad is given.  One workgroup: the minimum is reduced
// in LDS, so nothing has to be cleared before the launch.
__global__ __launch_bounds__(1024) void residual_kernel(float* res, const float* __restrict__ x, int n,
                                                        int* bad) {
    __shared__ int red[1024 / 64];
    int first = n;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float r = qsf::add_rn(res[i], x[i]);
        res[i] = r;
        if ((r != r || r > 1e30f || r < -1e30f) && i < first) first = i;
    }
    if (!bad) return;
    for (int off = 32; off > 0; off >>= 1) first = min(first, __shfl_xor(first, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = first;
    __syncthreads();
    if (threadIdx.x == 0) {
        int f = n;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) f = min(f, red[w]);
        *bad = f < n ? f : -1;
    }
}

// Residual add + NaN check, then the next norm of the updated residual, in
// one workgroup: the engine's sequence res += x (src/engine.c:937 / 1174),
// check (1176-1187), norm (940-948 / 805-815).  Each thread walks the same
// elements as residual_kernel and norm_kernel, so the results equal those
// two launches bit for bit.
template <bool LAYER>
__global__ __launch_bounds__(NORM_THREADS) void residual_norm_kernel(
    float* res, const float* __restrict__ x, int n, int* bad, const float* __restrict__ w,
    const float* __restrict__ b, float eps, float* out) {
    __shared__ int ired[NORM_THREADS / 64];
    __shared__ float red[NORM_THREADS / 64];
    int first = n;
    float acc = 0.f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float r = qsf::add_rn(res[i], x[i]);
        res[i] = r;
        if ((r != r || r > 1e30f || r < -1e30f) && i < first) first = i;
        acc = LAYER ? acc + r : fmaf(r, r, acc);
    }
    if (bad) {
        for (int off = 32; off > 0; off >>= 1) first = min(first, __shfl_xor(first, off, 64));
        if ((threadIdx.x & 63) == 0) ired[threadIdx.x >> 6] = first;
        __syncthreads();
        if (threadIdx.x == 0) {
            int f = n;
            for (int wv = 0; wv < (int)(blockDim.x >> 6); wv++) f = min(f, ired[wv]);
            *bad = f < n ? f : -1;
        }
    }
    if (!LAYER) {
        const float ss = block_sum(acc, red);
        const float inv = __fdiv_rn(1.0f, __fsqrt_rn(qsf::add_rn(__fdiv_rn(ss, (float)n), eps)));
        for (int i = threadIdx.x; i < n; i += blockDim.x) out[i] = qsf::mul_rn(qsf::mul_rn(res[i], inv), w[i]);
    } else {
        const float mean = __fdiv_rn(block_sum(acc, red), (float)n);
        float v = 0.f;
        for (int i = threadIdx.x; i < n; i += blockDim.x) {
            const float d = res[i] - mean;
            v = fmaf(d, d, v);
        }
        const float var = __fdiv_rn(block_sum(v, red), (float)n);
        const float inv = __fdiv_rn(1.0f, __fsqrt_rn(qsf::add_rn(var, eps)));
        for (int i = threadIdx.x; i < n; i += blockDim.x) {
            float o = qsf::mul_rn(qsf::mul_rn(qsf::sub_rn(res[i], mean), inv), w[i]);
            if (b) o = qsf::add_rn(o, b[i]);
            out[i] = o;
        }
    }
}

// RoPE of q and k and the int8 KV store of k (rotated) and v in one launch:
// one wave per q head (rotate), per kv head's k (rotate, then store) and
// per kv head's v (store).  The rotation is rope_kernel's arithmetic and the
// store kv_store_kernel's, so q, k and the cache rows equal the two
// launches bit for bit (absmax and the per-element codes do not depend on
// the order elements are visited).  head_dim <= 256: two pairs a lane.
__device__ __forceinline__ void rope_pair(float& a0, float& a1, const float* __restrict__ freq, int j,
                                          int position) {
    double ang = (double)position * (double)freq[j];
    ang = fmod(ang, 2.0 * 3.14159265358979323846);
    const float c = cosf((float)ang), sn = sinf((float)ang);
    const float x0 = a0, x1 = a1;
    a0 = qsf::sub_rn(qsf::mul_rn(x0, c), qsf::mul_rn(x1, sn));
    a1 = qsf::add_rn(qsf::mul_rn(x0, sn), qsf::mul_rn(x1, c));
}

__device__ __forceinline__ int8_t kv_code(float x, float inv) {
    x = qsf::mul_rn(x, inv);
    if (x > 127.0f) x = 127.0f;
    if (x < -127.0f) x = -127.0f;
    return (int8_t)(int)qsf::add_rn(x, x >= 0 ? 0.5f : -0.5f);
}

__global__ __launch_bounds__(64) void rope_kv_kernel(float* q, float* k, const float* __restrict__ v,
                                                     const float* __restrict__ freq, int head_dim,
                                                     int n_heads, int position, int8_t* kc, int8_t* vc,
                                                     float* ks, float* vs, int max_seq) {
    const int lane = threadIdx.x, hp = head_dim / 2;
    if ((int)blockIdx.x < n_heads) {
        float* qh = q + (size_t)blockIdx.x * head_dim;
        for (int j = lane; j < hp; j += 64) rope_pair(qh[2 * j], qh[2 * j + 1], freq, j, position);
        return;
    }
    const int idx = (int)blockIdx.x - n_heads, h = idx >> 1, isv = idx & 1;
    const size_t row = (size_t)h * max_seq + position;
    float val[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
    const float* src = (isv ? v : k) + (size_t)h * head_dim;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int j = lane + 64 * u;
        if (j < hp) {
            val[u][0] = src[2 * j];
            val[u][1] = src[2 * j + 1];
            if (!isv) {
                rope_pair(val[u][0], val[u][1], freq, j, position);
                float* kh = k + (size_t)h * head_dim;
                kh[2 * j] = val[u][0];
                kh[2 * j + 1] = val[u][1];
            }
        }
    }
    float amax = 0.f;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const float a = val[u][e] < 0 ? -val[u][e] : val[u][e];
            amax = a > amax ? a : amax;
        }
    for (int off = 32; off > 0; off >>= 1) {
        const float o = __shfl_xor(amax, off, 64);
        amax = o > amax ? o : amax;
    }
    if (lane == 0) (isv ? vs : ks)[row] = __fdiv_rn(amax, 127.0f);
    int8_t* dst = (isv ? vc : kc) + row * head_dim;
    const bool live = amax > 1e-30f;
    const float inv = live ? __fdiv_rn(127.0f, amax) : 0.f;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int j = lane + 64 * u;
        if (j < hp) {
            dst[2 * j] = live ? kv_code(val[u][0], inv) : (int8_t)0;
            dst[2 * j + 1] = live ? kv_code(val[u][1], inv) : (int8_t)0;
        }
    }
}

// The same chunk result for head_dim = 16 HC in {64, 128, 256}, for G query
// heads of one KV head at a time: a K or V code is loaded and converted once
// for the G heads instead of once a head.  FUSED: the RoPE of q and k and
// the int8 KV store of the new row in the same launch.
//
// Bound by the cache bytes (2 (hd + 4) a position and KV head) and, short of
// a few thousand positions, by its chain of one load and three barriers.
// Every byte of the chunk (and its scales) is requested before any is used, as
// 16-byte pieces; thread t holds pieces t, t + 256, ..., i.e. dims
// 16 (t % HC) .. + 15 of positions (t + 256 j) / HC, for K and V alike, so a
// wave's load covers 1 KB of consecutive rows.
//  * Scores: the thread's 16 dims of every head's q sit in registers; a
//    position's HC partial dots are summed with DPP into LDS.
//  * Softmax terms: wave g takes head g, two positions a lane.
//  * Weighted V: 16 dims x G heads a thread, summed over the wave's 64 / HC
//    position groups by halving (each step exchanges half of the values with
//    the lanes 32, 16, 8 or 4 away and adds), then over the waves in LDS.
// Measured with the merge below (32 heads on 8 KV heads of 128, 12345 positions, graph
// replay, 26 MB of cache): 68.2 -> 19.4 us a step against one workgroup a
// (head, chunk), an LDS pass over 32 partial rows an output and the serial
// merge; a 7B layer step (1024 positions, MHA, G = 1) 49.3 -> 48.2 us.
// The arithmetic of a head does not depend on G, nor on FUSED: the cache
// rows, scales and chunk records of the fused launch equal those of
// rope_kv_kernel followed by the plain one bit for bit.
//
// FUSED: every workgroup rotates its heads' q itself, into LDS.  The
// position being decoded lies in the last chunk: its workgroups rotate the
// new k and quantise k and v with the KV store's arithmetic, and use those
// codes for that row instead of reading the cache; the first workgroup of
// each KV head also stores them, with the scales.  No other workgroup needs
// that row, so the store orders with nothing.  q and k stay as they were:
// several workgroups read each of them, so none may rotate them in place.
struct AttArgs {
    const float *q, *k, *v, *freq;
    int8_t *kc, *vc;
    float *ks, *vs;
    int max_seq, groups, seq, nsplit;
    float* ws;
};

__device__ __forceinline__ float wave_max64(float v) {
#define QSF_DPPM(x, ctrl, rmask) \
    __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, -__builtin_inff()), \
                                                          __builtin_bit_cast(int, (x)), (ctrl), (rmask), 0xF, false))
    v = fmaxf(v, QSF_DPPM(v, 0xB1, 0xF));     // quad_perm [1,0,3,2]
    v = fmaxf(v, QSF_DPPM(v, 0x4E, 0xF));     // quad_perm [2,3,0,1]
    v = fmaxf(v, QSF_DPPM(v, 0x141, 0xF));    // row_half_mirror
    v = fmaxf(v, QSF_DPPM(v, 0x140, 0xF));    // row_mirror
    v = fmaxf(v, QSF_DPPM(v, 0x142, 0xA));    // row_bcast15
    v = fmaxf(v, QSF_DPPM(v, 0x143, 0xC));    // row_bcast31
#undef QSF_DPPM
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ float wave_sum64(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(
                                         __builtin_bit_cast(int, qsf::group_sum_last(v, 64)), 63));
}

// a[0 .. N): each value summed over the lanes `lane ^ D` pairs; the lanes
// with bit D clear keep the sums of a[0 .. N/2), the others those of
// a[N/2 .. N), in a[0 .. N/2) either way.
template <int D, int N>
__device__ __forceinline__ void halve(float* a) {
#pragma unroll
    for (int i = 0; i < N / 2; i++) {
        const uint32_t lo = __builtin_bit_cast(uint32_t, a[i]), hi = __builtin_bit_cast(uint32_t, a[i + N / 2]);
        if constexpr (D == 32 || D == 16) {
            const auto r = D == 32 ? __builtin_amdgcn_permlane32_swap(lo, hi, false, false)
                                   : __builtin_amdgcn_permlane16_swap(lo, hi, false, false);
            a[i] = __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
        } else {
            const bool up = (threadIdx.x & D) != 0;
            const uint32_t keep = up ? hi : lo, send = up ? lo : hi;
            const uint32_t got = D == 8 ? (uint32_t)__builtin_amdgcn_update_dpp(0, (int)send, 0x128, 0xF, 0xF, false)
                                        : (uint32_t)__shfl_xor((int)send, D, 64);   // 0x128: row_ror:8
            a[i] = __builtin_bit_cast(float, keep) + __builtin_bit_cast(float, got);
        }
    }
}

template <int HC, int G, bool FUSED>
__global__ __launch_bounds__(ATT_THREADS) void attention_chunk_kernel(AttArgs a) {
    constexpr int HD = 16 * HC, HP = HD / 2, NJ = ATT_CHUNK * HC / ATT_THREADS, NW = ATT_THREADS / 64;
    static_assert(ATT_THREADS % HC == 0 && HP <= 128 && G <= NW, "one wave a head's softmax, one k pair a thread");
    __shared__ __align__(16) float qs[G * HD];
    __shared__ float dots[G][ATT_CHUNK];                 // q . k codes, then exp(score - m) * v_scale
    __shared__ float red[4];
    __shared__ __align__(16) float part[NW][G * HD];
    __shared__ __align__(16) int8_t newc[2][HD];         // the new row's K and V codes
    __shared__ float news[2];                            // and their scales
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int h0 = blockIdx.x * G, chunk = blockIdx.y, kvh = h0 / a.groups;
    const int p0 = chunk * ATT_CHUNK, np = min(ATT_CHUNK, a.seq - p0);
    const bool last = FUSED && chunk == a.nsplit - 1;    // holds the new row, np - 1
    const size_t row0 = (size_t)kvh * a.max_seq + p0;
    // 1. all loads.  Positions past the chunk end load the last valid row and
    //    are masked.  FUSED, last chunk: only the rows before the new one
    //    (none when the new row starts the chunk: no workgroup reads the row
    //    that is being stored).
    const int nold = last ? np - 1 : np;                 // rows already in the cache
    att_u32x4 kk[NJ], vv[NJ];
    float kscale[2] = {0.f, 0.f}, vscale[2] = {0.f, 0.f};
    if (nold > 0) {                                      // (uniform)
        const att_u32x4* kr = reinterpret_cast<const att_u32x4*>(a.kc + row0 * HD);
        const att_u32x4* vr = reinterpret_cast<const att_u32x4*>(a.vc + row0 * HD);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int i = t + ATT_THREADS * j;
            kk[j] = kr[min(i / HC, nold - 1) * HC + i % HC];
        }
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int i = t + ATT_THREADS * j;
            vv[j] = vr[min(i / HC, nold - 1) * HC + i % HC];
        }
        if (wave < G) {
#pragma unroll
            for (int e = 0; e < 2; e++) {
                kscale[e] = a.ks[row0 + min(lane + 64 * e, nold - 1)];
                vscale[e] = a.vs[row0 + min(lane + 64 * e, nold - 1)];
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < NJ; j++) kk[j] = vv[j] = att_u32x4{0u, 0u, 0u, 0u};
    }
    if constexpr (FUSED) {
        float nk[2] = {0.f, 0.f}, nv[2] = {0.f, 0.f};
        if (last && t < HP) {
            nk[0] = a.k[(size_t)kvh * HD + 2 * t];
            nk[1] = a.k[(size_t)kvh * HD + 2 * t + 1];
            nv[0] = a.v[(size_t)kvh * HD + 2 * t];
            nv[1] = a.v[(size_t)kvh * HD + 2 * t + 1];
        }
#pragma unroll
        for (int i0 = 0; i0 < G * HP; i0 += ATT_THREADS) {
            const int i = i0 + t;
            if (G * HP % ATT_THREADS == 0 || i < G * HP) {
                float q0 = a.q[(size_t)h0 * HD + 2 * i], q1 = a.q[(size_t)h0 * HD + 2 * i + 1];
                rope_pair(q0, q1, a.freq, i % HP, a.seq - 1);
                qs[2 * i] = q0;
                qs[2 * i + 1] = q1;
            }
        }
        if (last) {
            if (t < HP) rope_pair(nk[0], nk[1], a.freq, t, a.seq - 1);
            // absmax as the KV store takes it (NaN compares false and drops out)
            float ak = 0.f, av = 0.f;
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const float x = nk[e] < 0 ? -nk[e] : nk[e], y = nv[e] < 0 ? -nv[e] : nv[e];
                ak = x > ak ? x : ak;
                av = y > av ? y : av;
            }
            for (int off = 32; off > 0; off >>= 1) {
                const float ok = __shfl_xor(ak, off, 64), ov = __shfl_xor(av, off, 64);
                ak = ok > ak ? ok : ak;
                av = ov > av ? ov : av;
            }
            if (HP > 64) {                               // pairs in waves 0 and 1
                if (t == 0 || t == 64) {
                    red[t >> 5] = ak;
                    red[(t >> 5) + 1] = av;
                }
                __syncthreads();
                ak = red[2] > red[0] ? red[2] : red[0];
                av = red[3] > red[1] ? red[3] : red[1];
            }
            const bool lk = ak > 1e-30f, lv = av > 1e-30f;
            const float ik = lk ? __fdiv_rn(127.0f, ak) : 0.f, iv = lv ? __fdiv_rn(127.0f, av) : 0.f;
            const bool store = h0 % a.groups == 0;
            const size_t row = (size_t)kvh * a.max_seq + a.seq - 1;
            if (t < HP) {
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int8_t ck = lk ? kv_code(nk[e], ik) : (int8_t)0, cv = lv ? kv_code(nv[e], iv) : (int8_t)0;
                    newc[0][2 * t + e] = ck;
                    newc[1][2 * t + e] = cv;
                    if (store) {
                        a.kc[row * HD + 2 * t + e] = ck;
                        a.vc[row * HD + 2 * t + e] = cv;
                    }
                }
            }
            if (t == 0) {
                news[0] = __fdiv_rn(ak, 127.0f);
                news[1] = __fdiv_rn(av, 127.0f);
                if (store) {
                    a.ks[row] = news[0];
                    a.vs[row] = news[1];
                }
            }
        }
    } else {
        for (int i = t; i < G * HD; i += ATT_THREADS) qs[i] = a.q[(size_t)h0 * HD + i];
    }
    __syncthreads();
    if (last) {                                          // the new row in place of the loaded one
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int i = t + ATT_THREADS * j;
            if (i / HC == np - 1) {
                kk[j] = reinterpret_cast<const att_u32x4*>(newc[0])[i % HC];
                vv[j] = reinterpret_cast<const att_u32x4*>(newc[1])[i % HC];
            }
        }
#pragma unroll
        for (int e = 0; e < 2; e++)
            if (lane + 64 * e == np - 1) {
                kscale[e] = news[0];
                vscale[e] = news[1];
            }
    }
    // 2. dots of the chunk's K codes with every head's q
    {
        float qr[G][16];
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float4 x = *reinterpret_cast<const float4*>(&qs[g * HD + 16 * (t % HC) + 4 * c]);
                qr[g][4 * c] = x.x; qr[g][4 * c + 1] = x.y; qr[g][4 * c + 2] = x.z; qr[g][4 * c + 3] = x.w;
            }
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            float d[G];
#pragma unroll
            for (int g = 0; g < G; g++) d[g] = 0.f;
#pragma unroll
            for (int b = 0; b < 16; b++) {
                const float c = sbyte(kk[j][b >> 2], b & 3);
#pragma unroll
                for (int g = 0; g < G; g++) d[g] = fmaf(qr[g][b], c, d[g]);
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                d[g] = qsf::group_sum_last(d[g], HC);
                if (t % HC == HC - 1) dots[g][(t + ATT_THREADS * j) / HC] = d[g];
            }
        }
    }
    __syncthreads();
    // 3. wave g: head g's scores, the chunk's max and softmax terms
    if (wave < G) {
        const float inv_sqrt_d = __fdiv_rn(1.0f, __fsqrt_rn((float)HD));
        float sc[2];
        bool wide = false;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            sc[e] = qsf::mul_rn(dots[wave][lane + 64 * e], kscale[e]);
            wide |= !(__builtin_fabsf(sc[e]) < INFINITY);
        }
        // The codes' sum can pass fp32's range (q from 2^113 on) where the
        // dequantised row's does not, and an Inf scale times a zero code is
        // NaN: such positions take their rows element by element.
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(wide) != 0, 0)) {
#pragma unroll 1
            for (int e = 0; e < 2; e++) {
                const int p = lane + 64 * e;
                const float scale = e ? kscale[1] : kscale[0], d = e ? sc[1] : sc[0];
                if (p >= np || __builtin_fabsf(d) < INFINITY) continue;
                const int8_t* row = last && p == np - 1 ? newc[0] : a.kc + (row0 + p) * HD;
                float x = 0.f;
#pragma unroll 1
                for (int c = 0; c < HD; c++) x = fmaf(qs[wave * HD + c], qsf::mul_rn((float)row[c], scale), x);
                if (e) sc[1] = x;
                else sc[0] = x;
            }
        }
#pragma unroll
        for (int e = 0; e < 2; e++) sc[e] = lane + 64 * e < np ? qsf::mul_rn(sc[e], inv_sqrt_d) : -INFINITY;
        const float m = wave_max64(fmaxf(sc[0], sc[1]));
        float l = 0.f;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const float x = lane + 64 * e < np ? expf(sc[e] - m) : 0.f;
            dots[wave][lane + 64 * e] = lane + 64 * e < np ? qsf::mul_rn(x, vscale[e]) : 0.f;
            l += x;
        }
        l = wave_sum64(l);
        if (lane == 0) {
            float* rec = a.ws + ((size_t)(h0 + wave) * a.nsplit + chunk) * (HD + 2);
            rec[0] = m;
            rec[1] = l;
        }
    }
    __syncthreads();
    // 4. weighted V: dims 16 (t % HC) .. + 15 of the thread's positions
    float acc[16 * G];
#pragma unroll
    for (int i = 0; i < 16 * G; i++) acc[i] = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        float w[G];
#pragma unroll
        for (int g = 0; g < G; g++) w[g] = dots[g][(t + ATT_THREADS * j) / HC];
#pragma unroll
        for (int b = 0; b < 16; b++) {
            const float c = sbyte(vv[j][b >> 2], b & 3);
#pragma unroll
            for (int g = 0; g < G; g++) acc[16 * g + b] = fmaf(w[g], c, acc[16 * g + b]);
        }
    }
    halve<32, 16 * G>(acc);
    halve<16, 8 * G>(acc);
    int at = (lane & 32 ? 8 * G : 0) + (lane & 16 ? 4 * G : 0);
    if constexpr (HC <= 8) {
        halve<8, 4 * G>(acc);
        at += lane & 8 ? 2 * G : 0;
    }
    if constexpr (HC <= 4) {
        halve<4, 2 * G>(acc);
        at += lane & 4 ? G : 0;
    }
#pragma unroll
    for (int i = 0; i < 16 * G * HC / 64; i++)           // value at + i: head / 16, dim % 16 of the thread's 16
        part[wave][((at + i) >> 4) * HD + 16 * (t % HC) + ((at + i) & 15)] = acc[i];
    __syncthreads();
    for (int i = t; i < G * HD; i += ATT_THREADS) {
        float o = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) o += part[w][i];
        a.ws[((size_t)(h0 + i / HD) * a.nsplit + chunk) * (HD + 2) + 2 + i % HD] = o;
    }
}

// Merge of a head's chunk records: rescale to the largest chunk maximum, add,
// normalise.  A workgroup a head, 1024 threads: thread (dim, part) adds the
// chunks part, part + P, ... of its dim, the P parts meet in LDS.  (One
// thread a dim walking every record twice, each step a memory latency, took
// 45 us at 97 chunks.)
constexpr int CMB_THREADS = 1024;
__global__ __launch_bounds__(CMB_THREADS) void attention_combine_kernel(const float* __restrict__ ws,
                                                                        int head_dim, int nsplit,
                                                                        float* __restrict__ out) {
    constexpr int MAXS = ATT_MAX_SEQ / ATT_CHUNK;
    static_assert(MAXS == 128, "two chunks a lane");
    __shared__ float f[MAXS];                            // exp(chunk max - max)
    __shared__ float parts[CMB_THREADS];
    __shared__ float Ls;
    const int h = blockIdx.x, t = threadIdx.x, stride = head_dim + 2;
    const int P = CMB_THREADS / head_dim, d = t % head_dim, part = t / head_dim;
    const float* base = ws + (size_t)h * nsplit * stride;
    if (t < 64) {
        const bool on0 = t < nsplit, on1 = t + 64 < nsplit;
        const float* r0 = base + (size_t)min(t, nsplit - 1) * stride;
        const float* r1 = base + (size_t)min(t + 64, nsplit - 1) * stride;
        const float m0 = r0[0], l0 = r0[1], m1 = r1[0], l1 = r1[1];
        const float M = wave_max64(fmaxf(m0, m1));       // (lanes past nsplit repeat the last record)
        const float f0 = expf(m0 - M), f1 = expf(m1 - M);
        if (on0) f[t] = f0;
        if (on1) f[t + 64] = f1;
        const float L = wave_sum64(fmaf(on1 ? f1 : 0.f, l1, on0 ? f0 * l0 : 0.f));
        if (t == 0) Ls = L;
    }
    __syncthreads();
    float O = 0.f;
    if (part < P) {
#pragma unroll 8
        for (int c = part; c < nsplit; c += P) O = fmaf(f[c], base[(size_t)c * stride + 2 + d], O);
    }
    parts[t] = O;
    __syncthreads();
    if (t < head_dim) {
        float o = 0.f;
        for (int i = 0; i < P; i++) o += parts[i * head_dim + t];
        out[(size_t)h * head_dim + t] = __fdiv_rn(o, Ls);
    }
}

// One row of a blockwise table: value i = scale * q + zero (4-bit sym:
// scale * q), each product and sum rounded as in src/quant.c:95-177.
__global__ __launch_bounds__(256) void embed_row_kernel(const uint8_t* __restrict__ blocks, int fmt,
                                                        int bs, int bb, int hd, float* out,
                                                        int frag_row, int nq, int plane, int nb) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= hd) return;
    // byte j of the value's block: on-disk or row-plane order (`blocks` is
    // the row), or fragment order (`blocks` is the tensor, frag_row the row)
    const int b = i / bs;
    auto byte_at = [&](int j) -> unsigned {
        return frag_row >= 0 ? blocks[qsf::frag_off((size_t)frag_row, b, j, nq, bb)]
               : plane       ? blocks[qsf::plane_off(b, j, nb, bb, bs)]
                             : blocks[(size_t)b * bb + j];
    };
    const uint32_t meta = byte_at(0) | (byte_at(1) << 8) | (byte_at(2) << 16) | (byte_at(3) << 24);
    const int k = i % bs;
    unsigned c;
    if (fmt == QK_FMT_2) {
        c = (byte_at(4 + (k >> 2)) >> ((k & 3) * 2)) & 3u;
    } else if (fmt == QK_FMT_3) {
        const int bit = 3 * k, byte = bit >> 3, off = bit & 7;
        unsigned v = byte_at(4 + byte) >> off;
        if (off > 5) v |= byte_at(4 + byte + 1) << (8 - off);
        c = v & 7u;
    } else {
        c = (byte_at(4 + (k >> 1)) >> ((k & 1) * 4)) & 15u;
    }
    const float s = qsf::f16_lo(meta);
    if (fmt == QK_FMT_4SYM) {
        out[i] = qsf::mul_rn(s, (float)(c >= 8u ? (int)c - 16 : (int)c));
    } else {
        out[i] = qsf::add_rn(qsf::mul_rn(s, (float)c), qsf::f16_hi(meta));
    }
}

__global__ __launch_bounds__(256) void embed_row_fp16_kernel(const uint16_t* __restrict__ row, int hd,
                                                             float* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < hd) out[i] = qsf::f16_bits(row[i]);
}

// Heads of one KV head a workgroup takes together: as many of 4, 2, 1 as
// divide the group while the launch still has a workgroup for each CU.
// (More heads convert and load each code fewer times; fewer workgroups than
// CUs leave CUs idle.)
template <bool FUSED>
bool launch_chunks(const AttArgs& a, int head_dim, int n_heads, hipStream_t s) {
    int G = a.groups % 4 == 0 ? 4 : a.groups % 2 == 0 ? 2 : 1;
    while (G > 1 && (long)(n_heads / G) * a.nsplit < ATT_FILL) G >>= 1;
    const dim3 grid(n_heads / G, a.nsplit), block(ATT_THREADS);
#define QSF_ATT_G(HC)                                                                                     \
    if (G == 4) hipLaunchKernelGGL((attention_chunk_kernel<HC, 4, FUSED>), grid, block, 0, s, a);         \
    else if (G == 2) hipLaunchKernelGGL((attention_chunk_kernel<HC, 2, FUSED>), grid, block, 0, s, a);    \
    else hipLaunchKernelGGL((attention_chunk_kernel<HC, 1, FUSED>), grid, block, 0, s, a);                \
    return true;
    switch (head_dim) {
    case 64: QSF_ATT_G(4)
    case 128: QSF_ATT_G(8)
    case 256: QSF_ATT_G(16)
    default: return false;
    }
#undef QSF_ATT_G
}

}  // namespace

extern "C" int qk_norm(const float* in, float* out, const float* w, const float* b, int dim,
                       float eps, int layer, hipStream_t s) {
    if (dim <= 0) return 0;
    if (layer)
        hipLaunchKernelGGL(norm_kernel<true>, dim3(1), dim3(NORM_THREADS), 0, s, in, out, w, b, dim, eps);
    else
        hipLaunchKernelGGL(norm_kernel<false>, dim3(1), dim3(NORM_THREADS), 0, s, in, out, w, b, dim, eps);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int qk_rope(float* q, float* k, const float* freq, int head_dim, int n_heads,
                       int n_kv, int position, hipStream_t s) {
    const int nq = n_heads * head_dim / 2, nk = n_kv * head_dim / 2;
    if (nq + nk == 0) return 0;
    hipLaunchKernelGGL(rope_kernel, dim3((nq + nk + 255) / 256), dim3(256), 0, s, q, k, freq, head_dim,
                       nq, nk, position);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int qk_kv_store(int8_t* kc, int8_t* vc, float* ks, float* vs, int max_seq, int n_kv,
                           int head_dim, int position, const float* k, const float* v,
                           hipStream_t s) {
    if (n_kv <= 0) return 0;
    hipLaunchKernelGGL(kv_store_kernel, dim3(2 * n_kv), dim3(64), 0, s, kc, vc, ks, vs, k, v, max_seq,
                       head_dim, position);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" size_t qk_attention_ws_bytes(int n_heads, int head_dim, int position) {
    const int nsplit = (position + 1 + ATT_CHUNK - 1) / ATT_CHUNK;
    return sizeof(float) * (size_t)n_heads * nsplit * (head_dim + 2);
}

extern "C" int qk_attention(const float* q, const int8_t* kc, const int8_t* vc, const float* ks,
                            const float* vs, int max_seq, int n_heads, int n_kv, int head_dim,
                            int position, float* out, void* ws, hipStream_t s) {
    const int seq = position + 1;
    if (head_dim > ATT_THREADS || head_dim % 16 || seq > ATT_MAX_SEQ || n_kv <= 0 ||
        n_heads % n_kv)
        return -2;
    const int nsplit = (seq + ATT_CHUNK - 1) / ATT_CHUNK, groups = n_heads / n_kv;
    const AttArgs a = {q, nullptr, nullptr, nullptr, const_cast<int8_t*>(kc), const_cast<int8_t*>(vc),
                       const_cast<float*>(ks), const_cast<float*>(vs), max_seq, groups, seq, nsplit, (float*)ws};
    if (!launch_chunks<false>(a, head_dim, n_heads, s))
        hipLaunchKernelGGL(attention_part_kernel, dim3(n_heads, nsplit), dim3(ATT_THREADS), 0, s, q, kc, vc, ks,
                           vs, max_seq, groups, head_dim, seq, nsplit, (float*)ws);
    hipLaunchKernelGGL(attention_combine_kernel, dim3(n_heads), dim3(CMB_THREADS), 0, s, (const float*)ws,
                       head_dim, nsplit, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int qk_act_mul(float* gate, const float* up, int n, int act, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(act_mul_kernel, dim3((n + 255) / 256), dim3(256), 0, s, gate, up, n, act);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int qk_residual(float* res, const float* x, int n, int* bad, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(residual_kernel, dim3(1), dim3(1024), 0, s, res, x, n, bad);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int qk_residual_norm(float* res, const float* x, int n, int* bad, const float* w,
                                const float* b, float eps, int layer, float* out, hipStream_t s) {
    if (n <= 0) return 0;
    if (layer)
        hipLaunchKernelGGL(residual_norm_kernel<true>, dim3(1), dim3(NORM_THREADS), 0, s, res, x, n, bad, w,
                           b, eps, out);
    else
        hipLaunchKernelGGL(residual_norm_kernel<false>, dim3(1), dim3(NORM_THREADS), 0, s, res, x, n, bad,
                           w, b, eps, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int qk_rope_kv_store(float* q, float* k, const float* v, const float* freq, int head_dim,
                                int n_heads, int n_kv, int position, int8_t* kc, int8_t* vc, float* ks,
                                float* vs, int max_seq, hipStream_t s) {
    if (head_dim <= 0 || head_dim > 256 || (head_dim & 1) || n_kv <= 0 || position < 0 ||
        position >= max_seq)
        return -2;
    hipLaunchKernelGGL(rope_kv_kernel, dim3(n_heads + 2 * n_kv), dim3(64), 0, s, q, k, v, freq, head_dim,
                       n_heads, position, kc, vc, ks, vs, max_seq);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int qk_rope_kv_attention(float* q, float* k, const float* v, const float* freq, int head_dim,
                                    int n_heads, int n_kv, int position, int8_t* kc, int8_t* vc, float* ks,
                                    float* vs, int max_seq, float* out, void* ws, hipStream_t s) {
    const int seq = position + 1;
    if (head_dim <= 0 || head_dim > 256 || head_dim % 16 || n_heads <= 0 || n_kv <= 0 || n_heads % n_kv ||
        position < 0 || position >= max_seq || seq > ATT_MAX_SEQ)
        return -2;
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) {
        const int rc = qk_rope_kv_store(q, k, v, freq, head_dim, n_heads, n_kv, position, kc, vc, ks, vs,
                                        max_seq, s);
        return rc ? rc : qk_attention(q, kc, vc, ks, vs, max_seq, n_heads, n_kv, head_dim, position, out, ws, s);
    }
    const int nsplit = (seq + ATT_CHUNK - 1) / ATT_CHUNK;
    const AttArgs a = {q, k, v, freq, kc, vc, ks, vs, max_seq, n_heads / n_kv, seq, nsplit, (float*)ws};
    launch_chunks<true>(a, head_dim, n_heads, s);
    hipLaunchKernelGGL(attention_combine_kernel, dim3(n_heads), dim3(CMB_THREADS), 0, s, (const float*)ws, head_dim,
                       nsplit, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int qk_embed_row(const qsf_hip_tensor* t, int token, float* out, hipStream_t s) {
    if (t->fmt < 0 || token < 0 || token >= t->rows) return -2;
    if (t->cols <= 0) return 0;
    const uint8_t* row = t->frag ? t->d_blocks : t->d_blocks + (size_t)token * t->nb * t->block_bytes;
    hipLaunchKernelGGL(embed_row_kernel, dim3((t->cols + 255) / 256), dim3(256), 0, s, row, t->fmt, t->bs,
                       t->block_bytes, t->cols, out, t->frag ? token : -1, t->frag_nq, t->plane, t->nb);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int qk_embed_row_fp16(const uint16_t* table, int hd, int token, float* out,
                                 hipStream_t s) {
    if (hd <= 0) return 0;
    hipLaunchKernelGGL(embed_row_fp16_kernel, dim3((hd + 255) / 256), dim3(256), 0, s,
                       table + (size_t)token * hd, hd, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
