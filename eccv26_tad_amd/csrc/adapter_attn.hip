// The adapter's attention of the visual tokens to a few key tokens
// (reference vit_sparse_adapter_poguise.py:598-620): LayerNorm of the token
// rows, per-head LayerNorm of queries and keys, softmax over the key tokens,
// and their gradients (gfx950).
//
// All of it is row work on [M, a] and [M, h] matrices with a handful of keys
// per sample: a wave holds 64 channels of a row, one per lane (64 / HD heads),
// keys and values of those channels sit in registers, and every dot product of
// a head is a sum over its HD lanes. It is bound by each row's chain of load
// and lane sums, not by its bytes: at 17254 rows k_key_attn moves 9 MB in 15.1
// us (0.6 TB/s), its backward 13 MB in 23.3, k_ln_fwd 26 MB in 12.1 (2.2 TB/s).
// PyTorch's chain of per-head LayerNorms, transposed copies, batched products
// with 3 columns and their gradients took 1.1 ms of a 1.7 ms step (B2 x 8628
// tokens, a = 128, 3 keys).
#include <algorithm>

#include "sv_common.h"
#include "sv_conv.h"
#include "sv_internal.h"
#include "sv_mfma.h"

namespace svtad {

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
    const int t = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true);
    return v + __builtin_bit_cast(float, t);
}

// Sum over the N consecutive lanes of a lane's group (16, 32 or 64), in every
// lane of it, in a fixed order.
template <int N>
__device__ __forceinline__ float lane_sum(float v) {
    v = dpp_add<0xB1>(v);   // quad_perm: lane ^ 1
    v = dpp_add<0x4E>(v);   // quad_perm: lane ^ 2
    v = dpp_add<0x141>(v);  // row_half_mirror: the other quad of 8
    v = dpp_add<0x140>(v);  // row_mirror: the other half of 16
    if constexpr (N >= 32) v += __shfl_xor(v, 16, 64);
    if constexpr (N >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

template <typename T>
__device__ __forceinline__ float load_param(const void* p, int i, bool f32) {
    return f32 ? ((const float*)p)[i] : (float)((const T*)p)[i];
}

// ---------------------------------------------------------------------------
// LayerNorm of [rows, C] rows, C = 64 VPL: one wave per row, VPL consecutive
// channels per lane; mean and 1 / std of each row are kept for the gradient.
// ---------------------------------------------------------------------------
// Rows per workgroup, a wave's rows one dependent chain of loads and lane sums
// after another: forward 13 us with 64 rows at 17254 x 256, 7.8 with 32, 7.3
// with 16.
constexpr int kLnRows = 16;

template <typename T, int VPL>
struct RowVec {
    T e[VPL];
};

// Row m of [batch, n_tokens, C] kept as special rows [batch, n_special, C] and
// patch rows: its address in one of them (n_special 0: in `patch`).
template <typename T>
__device__ __forceinline__ T* split_row(T* special, T* patch, int64_t m, uint32_t n_tokens, uint32_t n_special, int c) {
    if (n_special == 0) return patch + m * c;
    const uint32_t b = (uint32_t)m / n_tokens, r = (uint32_t)m - b * n_tokens;
    return r < n_special ? special + ((int64_t)b * n_special + r) * c
                         : patch + ((int64_t)b * (n_tokens - n_special) + (r - n_special)) * c;
}

template <typename T, int VPL>
__global__ __launch_bounds__(256) void k_ln_fwd(const T* __restrict__ special, const T* __restrict__ x,
                                                T* __restrict__ copy, uint32_t n_tokens, uint32_t n_special,
                                                const void* __restrict__ w, const void* __restrict__ b,
                                                T* __restrict__ y, float* __restrict__ stats, int64_t rows, float eps,
                                                bool p32) {
    constexpr int C = 64 * VPL;
    typedef RowVec<T, VPL> V;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float gw[VPL], gb[VPL];
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
        gw[j] = load_param<T>(w, lane * VPL + j, p32);
        gb[j] = load_param<T>(b, lane * VPL + j, p32);
    }
    const int64_t r1 = min<int64_t>(rows, (int64_t)(blockIdx.x + 1) * kLnRows);
    for (int64_t r = (int64_t)blockIdx.x * kLnRows + wave; r < r1; r += 4) {
        const V v = *(const V*)(split_row(special, x, r, n_tokens, n_special, C) + lane * VPL);
        if (copy) *(V*)(copy + r * C + lane * VPL) = v;
        float f[VPL], s = 0.f;
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            f[j] = (float)v.e[j];
            s += f[j];
        }
        const float mean = lane_sum<64>(s) * (1.f / C);
        s = 0.f;
#pragma unroll
        for (int j = 0; j < VPL; ++j) s += (f[j] - mean) * (f[j] - mean);
        const float rstd = rsqrtf(lane_sum<64>(s) * (1.f / C) + eps);
        V o;
#pragma unroll
        for (int j = 0; j < VPL; ++j) o.e[j] = (T)((f[j] - mean) * rstd * gw[j] + gb[j]);
        *(V*)(y + r * C + lane * VPL) = o;
        if (lane == 0) {
            stats[r * 2] = mean;
            stats[r * 2 + 1] = rstd;
        }
    }
}

// dx (+ add, the gradient of x by another way; stored by token kind), and
// part[workgroup][0 / 1][C]: the workgroup's sums of dy xhat and dy
template <typename T, int VPL>
__global__ __launch_bounds__(256) void k_ln_bwd(const T* __restrict__ dy, const T* __restrict__ x,
                                                const T* __restrict__ add, const float* __restrict__ stats,
                                                const void* __restrict__ w, T* __restrict__ dx_special,
                                                T* __restrict__ dx, uint32_t n_tokens, uint32_t n_special,
                                                float* __restrict__ part, int64_t rows, bool p32) {
    constexpr int C = 64 * VPL;
    typedef RowVec<T, VPL> V;
    __shared__ float red[4][2][C];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float gw[VPL], sw[VPL], sb[VPL];
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
        gw[j] = load_param<T>(w, lane * VPL + j, p32);
        sw[j] = sb[j] = 0.f;
    }
    const int64_t r1 = min<int64_t>(rows, (int64_t)(blockIdx.x + 1) * kLnRows);
    for (int64_t r = (int64_t)blockIdx.x * kLnRows + wave; r < r1; r += 4) {
        const V v = *(const V*)(x + r * C + lane * VPL), d = *(const V*)(dy + r * C + lane * VPL);
        const float mean = stats[r * 2], rstd = stats[r * 2 + 1];
        float xh[VPL], g[VPL], s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const float t = (float)d.e[j];
            xh[j] = ((float)v.e[j] - mean) * rstd;
            g[j] = t * gw[j];
            s1 += g[j];
            s2 += g[j] * xh[j];
            sw[j] += t * xh[j];
            sb[j] += t;
        }
        s1 = lane_sum<64>(s1) * (1.f / C);
        s2 = lane_sum<64>(s2) * (1.f / C);
        V o, ad;
        if (add) ad = *(const V*)(add + r * C + lane * VPL);
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const float t = rstd * (g[j] - s1 - xh[j] * s2);
            o.e[j] = (T)(add ? t + (float)ad.e[j] : t);
        }
        *(V*)(split_row(dx_special, dx, r, n_tokens, n_special, C) + lane * VPL) = o;
    }
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
        red[wave][0][lane * VPL + j] = sw[j];
        red[wave][1][lane * VPL + j] = sb[j];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 2 * C; e += 256) {
        const float* p = &red[0][0][0] + e;
        part[(int64_t)blockIdx.x * 2 * C + e] = p[0] + p[2 * C] + p[4 * C] + p[6 * C];
    }
}

// ---------------------------------------------------------------------------
// attention
// ---------------------------------------------------------------------------
struct KeyAttnArgs {
    const void* q;      // [B, N, a]
    const void* kv;     // [B, nk, 2 a]
    const void* dout;   // [B, N, a] (backward)
    const void *qn_w, *qn_b, *kn_w, *kn_b;  // [HD]
    void* out;          // [B, N, a]: the output, or dq
    float* part;        // backward: [B][workgroups][2 nk + 2][a]
    int64_t n;          // N
    int nk;
    float eps, scale;
    bool p32;
};
// Token rows per workgroup, as kLnRows: at 2 x 8627 rows of 128 channels and 3
// keys forward / backward 28 / 47 us with 64, 14.9 / 33 with 32, 11.3 / 29 with
// 16 (backward with its two small launches). With the chain's roundings
// (16 rows, kernel trace) the forward 15.3 us; the backward kernel alone 23.3.
constexpr int kAttnRows = 16;

// A = 4 HD channels in WPR = A / 64 waves per row; 4 / WPR rows at a time. A
// head's channels are HD consecutive lanes. NKT bounds the key count (register
// arrays; keys past nk have probability 0).
template <typename T, int HD, int NKT, bool BWD>
__global__ __launch_bounds__(256) void k_key_attn(KeyAttnArgs p) {
    constexpr int A = 4 * HD, WPR = A / 64, RPI = 4 / WPR;
    __shared__ float red[BWD ? 4 : 1][BWD ? 2 * NKT + 2 : 1][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = (wave % WPR) * 64 + lane, j = c % HD;
    const int64_t b = blockIdx.y;
    const T* const q = (const T*)p.q + b * p.n * A;
    const T* const kv = (const T*)p.kv + b * p.nk * 2 * A;
    T* const out = (T*)p.out + b * p.n * A;
    auto norm = [&](float v, float& xh, float& rstd) {  // the head's LayerNorm: xhat
        const float mean = lane_sum<HD>(v) * (1.f / HD);
        const float d = v - mean;
        rstd = rsqrtf(lane_sum<HD>(d * d) * (1.f / HD) + p.eps);
        xh = d * rstd;
    };
    // The reference's roundings: queries and keys enter the score product in
    // T; with float32 parameters (autocast) the scores, their scaling and the
    // probabilities of the weighted sum are rounded to T as well.
    auto round_amp = [&](float v) { return p.p32 ? (float)(T)v : v; };
    const float qw = load_param<T>(p.qn_w, j, p.p32), qb = load_param<T>(p.qn_b, j, p.p32);
    const float kw = load_param<T>(p.kn_w, j, p.p32), kb = load_param<T>(p.kn_b, j, p.p32);
    float kh[NKT], vv[NKT];
#pragma unroll
    for (int t = 0; t < NKT; ++t) {
        kh[t] = vv[t] = 0.f;
        if (t < p.nk) {  // uniform
            float xh, rstd;
            norm((float)kv[t * 2 * A + c], xh, rstd);
            kh[t] = (float)(T)(xh * kw + kb);
            vv[t] = (float)kv[t * 2 * A + A + c];
        }
    }
    float dk[BWD ? NKT : 1], dv[BWD ? NKT : 1], dqw = 0.f, dqb = 0.f;
#pragma unroll
    for (int t = 0; t < (BWD ? NKT : 1); ++t) dk[t] = dv[t] = 0.f;
    const int64_t r1 = min<int64_t>(p.n, (int64_t)(blockIdx.x + 1) * kAttnRows);
    for (int64_t r = (int64_t)blockIdx.x * kAttnRows + wave / WPR; r < r1; r += RPI) {
        if (r < p.nk) {  // a key token: no query (uniform)
            out[r * A + c] = (T)0.f;
            continue;
        }
        float xh, rstd;
        norm((float)q[r * A + c], xh, rstd);
        const float qh = (float)(T)(xh * qw + qb);
        float s[NKT], pr[NKT], mx = -__builtin_huge_valf();
#pragma unroll
        for (int t = 0; t < NKT; ++t) {
            s[t] = t < p.nk ? round_amp(round_amp(lane_sum<HD>(qh * kh[t])) * p.scale) : -__builtin_huge_valf();
            mx = fmaxf(mx, s[t]);
        }
        float z = 0.f;
#pragma unroll
        for (int t = 0; t < NKT; ++t) {
            s[t] = __expf(s[t] - mx);
            z += s[t];
        }
        const float iz = 1.f / z;
#pragma unroll
        for (int t = 0; t < NKT; ++t) {
            s[t] *= iz;
            pr[t] = round_amp(s[t]);
        }
        if constexpr (!BWD) {
            float o = 0.f;
#pragma unroll
            for (int t = 0; t < NKT; ++t) o += pr[t] * vv[t];
            out[r * A + c] = (T)o;
        } else {
            const float d = (float)((const T*)p.dout + b * p.n * A)[r * A + c];
            float dp[NKT], dot = 0.f;
#pragma unroll
            for (int t = 0; t < NKT; ++t) {
                dp[t] = t < p.nk ? lane_sum<HD>(d * vv[t]) : 0.f;
                dot += s[t] * dp[t];
                dv[t] += pr[t] * d;
            }
            float g = 0.f;  // gradient of the normalised query
#pragma unroll
            for (int t = 0; t < NKT; ++t) {
                const float ds = s[t] * (dp[t] - dot) * p.scale;
                g += ds * kh[t];
                dk[t] += ds * qh;
            }
            dqw += g * xh;
            dqb += g;
            const float w = g * qw;
            const float m1 = lane_sum<HD>(w) * (1.f / HD), m2 = lane_sum<HD>(w * xh) * (1.f / HD);
            out[r * A + c] = (T)(rstd * (w - m1 - xh * m2));
        }
    }
    if constexpr (BWD) {
#pragma unroll
        for (int t = 0; t < NKT; ++t) {
            red[wave][t][lane] = dk[t];
            red[wave][NKT + t][lane] = dv[t];
        }
        red[wave][2 * NKT][lane] = dqw;
        red[wave][2 * NKT + 1][lane] = dqb;
        __syncthreads();
        // waves with the same channels in order; rows dk 0 .. nk - 1, dv, dqw, dqb
        const int nr = 2 * p.nk + 2;
        float* const dst = p.part + (b * gridDim.x + blockIdx.x) * (int64_t)nr * A;
        for (int e = threadIdx.x; e < nr * A; e += 256) {
            const int row = e / A, ch = e - row * A;
            const int src = row < p.nk ? row : row < 2 * p.nk ? NKT + row - p.nk : 2 * NKT + row - 2 * p.nk;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < RPI; ++w) v += red[w * WPR + ch / 64][src][ch % 64];
            dst[e] = v;
        }
    }
}

// sums[b][e] = sum of part[b][g][e] over the sample's G workgroups in order;
// 8 thread groups take an eighth of them each
__global__ __launch_bounds__(256) void k_key_attn_sum(const float* __restrict__ part, float* __restrict__ sums, int groups,
                                                      int count) {
    __shared__ float red[8][32];
    const int lane = threadIdx.x & 31, g = threadIdx.x >> 5;
    const int e = blockIdx.x * 32 + lane;
    const int per = (groups + 7) / 8, g0 = min(groups, g * per), g1 = min(groups, g0 + per);
    const float* const p = part + (int64_t)blockIdx.y * groups * count;
    float s = 0.f;
    if (e < count) {
        for (int q = g0; q < g1; q += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = p[(int64_t)min(q + u, g1 - 1) * count + e];
#pragma unroll
            for (int u = 0; u < 8; ++u) s += q + u < g1 ? v[u] : 0.f;
        }
    }
    red[g][lane] = s;
    __syncthreads();
    if (g != 0 || e >= count) return;
    s = red[0][lane];
#pragma unroll
    for (int q = 1; q < 8; ++q) s += red[q][lane];
    sums[(int64_t)blockIdx.y * count + e] = s;
}

// The keys' LayerNorm backward and the small sums: dkv [B, nk, 2 A] and, per
// workgroup of A threads and `per` samples, dn [4][HD] (qn_w, qn_b, kn_w, kn_b
// gradients). A key is a chain of loads and lane sums, 0.53 us: up to
// kKeysInOne keys run in one workgroup (6 keys 4.7 us, 16 keys 10.1), more in
// up to kKeyGroups, whose sums a reduction adds (20 keys 11.8 -> 3.9 + 2.1 us,
// 256 samples of 16 keys 2162 -> 10.6 + 4.4).
constexpr int kKeysInOne = 8, kKeyGroups = 256;
template <typename T, int HD>
__global__ __launch_bounds__(4 * HD) void k_key_attn_keys(KeyAttnArgs p, const float* __restrict__ sums, int batch,
                                                          int per, T* __restrict__ dkv, float* __restrict__ dn) {
    constexpr int A = 4 * HD;
    __shared__ float red[4][A];
    const int c = threadIdx.x, j = c % HD;
    const int nr = 2 * p.nk + 2;
    const float kw = load_param<T>(p.kn_w, j, p.p32);
    float dqw = 0.f, dqb = 0.f, dkw = 0.f, dkb = 0.f;
    const int b1 = min(batch, ((int)blockIdx.x + 1) * per);
    for (int b = (int)blockIdx.x * per; b < b1; ++b) {
        const float* const s = sums + (int64_t)b * nr * A;
        const T* const kv = (const T*)p.kv + (int64_t)b * p.nk * 2 * A;
        for (int t = 0; t < p.nk; ++t) {
            const float v = (float)kv[t * 2 * A + c];
            const float mean = lane_sum<HD>(v) * (1.f / HD);
            const float d = v - mean;
            const float rstd = rsqrtf(lane_sum<HD>(d * d) * (1.f / HD) + p.eps);
            const float xh = d * rstd, g = s[t * A + c], w = g * kw;
            dkw += g * xh;
            dkb += g;
            const float m1 = lane_sum<HD>(w) * (1.f / HD), m2 = lane_sum<HD>(w * xh) * (1.f / HD);
            T* const o = dkv + ((int64_t)b * p.nk + t) * 2 * A;
            o[c] = (T)(rstd * (w - m1 - xh * m2));
            o[A + c] = (T)s[(p.nk + t) * A + c];
        }
        dqw += s[2 * p.nk * A + c];
        dqb += s[(2 * p.nk + 1) * A + c];
    }
    red[0][c] = dqw;
    red[1][c] = dqb;
    red[2][c] = dkw;
    red[3][c] = dkb;
    __syncthreads();
    for (int e = c; e < 4 * HD; e += A) {
        const float* r = red[e / HD] + e % HD;
        dn[blockIdx.x * 4 * HD + e] = r[0] + r[HD] + r[2 * HD] + r[3 * HD];
    }
}

static bool al16a(const void* p) { return ((uintptr_t)p & 15) == 0; }
// ---------------------------------------------------------------------------
// projection of the few key rows (a library product costs the host 40 us for
// these 6 x 256 x 128 values; the launches here take 4.3 us and, backward, 12.5:
// a key row of dxa is one chain of 2 A products per thread)
// ---------------------------------------------------------------------------
constexpr int kKeyRowsMax = 64;

// one workgroup of 2 A threads per key row, one output column per thread
template <typename T, int A>
__global__ __launch_bounds__(2 * A) void k_key_proj(const T* __restrict__ xa, const T* __restrict__ w,
                                                    const T* __restrict__ b, T* __restrict__ kv, int64_t n, int nk) {
    __shared__ float x[A];
    const int row = blockIdx.x, c = threadIdx.x;
    if (c < A) x[c] = (float)xa[((int64_t)(row / nk) * n + row % nk) * A + c];
    __syncthreads();
    float s = 0.f;
#pragma unroll 4
    for (int k = 0; k < A; k += 8) {
        const RowVec<T, 8> v = *(const RowVec<T, 8>*)(w + (int64_t)c * A + k);
#pragma unroll
        for (int e = 0; e < 8; ++e) s += x[k + e] * (float)v.e[e];
    }
    kv[(int64_t)row * 2 * A + c] = (T)(s + (float)b[c]);
}

// workgroups of A threads: [0, 2 A) one row of dw (and its db), then one key
// row of dxa each
template <typename T, int A>
__global__ __launch_bounds__(A) void k_key_proj_bwd(const T* __restrict__ dkv, const T* __restrict__ xa,
                                                    const T* __restrict__ w, T* __restrict__ dxa, void* __restrict__ dw,
                                                    void* __restrict__ db, int64_t n, int nk, int rows, bool w32, bool b32) {
    __shared__ float g[2 * A > kKeyRowsMax ? 2 * A : kKeyRowsMax];
    const int c = threadIdx.x;
    if ((int)blockIdx.x < 2 * A) {
        const int o = blockIdx.x;
        for (int r = c; r < rows; r += A) g[r] = (float)dkv[(int64_t)r * 2 * A + o];
        __syncthreads();
        float s = 0.f, t = 0.f;
        for (int r = 0; r < rows; ++r) {
            s += g[r] * (float)xa[((int64_t)(r / nk) * n + r % nk) * A + c];
            t += g[r];
        }
        if (w32) ((float*)dw)[o * A + c] = s;
        else ((T*)dw)[o * A + c] = (T)s;
        if (c == 0) {
            if (b32) ((float*)db)[o] = t;
            else ((T*)db)[o] = (T)t;
        }
        return;
    }
    const int row = blockIdx.x - 2 * A;
    for (int e = c; e < 2 * A; e += A) g[e] = (float)dkv[(int64_t)row * 2 * A + e];
    __syncthreads();
    float s = 0.f;
#pragma unroll 8
    for (int e = 0; e < 2 * A; ++e) s += g[e] * (float)w[(int64_t)e * A + c];
    dxa[((int64_t)(row / nk) * n + row % nk) * A + c] = (T)s;
}

static bool half_type(int d) { return d == SVTAD_F16 || d == SVTAD_BF16; }

}  // namespace svtad

using namespace svtad;

// the split of svtad_layer_norm / _bwd: whole samples, 32-bit row numbers
static bool split_ok(int64_t rows, int64_t n_tokens, int64_t n_special) {
    return n_special == 0 || (n_special > 0 && n_special <= n_tokens && n_tokens < (int64_t)INT32_MAX &&
                              rows < (int64_t)INT32_MAX && rows % n_tokens == 0);
}

extern "C" int svtad_layer_norm(const void* special, const void* x, void* copy, int64_t n_tokens, int64_t n_special,
                                const void* w, const void* b, void* y, float* stats, int64_t rows, int c, float eps,
                                int dtype, int param_f32, void* stream) {
    if (!half_type(dtype) || (c != 128 && c != 256))
        return set_error(SVTAD_ERR_UNSUPPORTED, "layer_norm: f16 / bf16 rows of 128 or 256 channels");
    if (rows < 0 || !split_ok(rows, n_tokens, n_special) ||
        (rows > 0 && ((!x && (n_special == 0 || n_tokens > n_special)) || (n_special > 0 && !special) || !w || !b || !y || !stats)) ||
        !al16a(x) || !al16a(special) || !al16a(copy) || !al16a(y))
        return set_error(SVTAD_ERR_INVALID, "layer_norm: bad arguments");
    if (rows == 0) return SVTAD_OK;
    const dim3 g((unsigned)cdiv(rows, kLnRows));
#define SVTAD_LN(T, V) \
    hipLaunchKernelGGL((k_ln_fwd<T, V>), g, dim3(256), 0, (hipStream_t)stream, (const T*)special, (const T*)x, (T*)copy, (uint32_t)n_tokens, (uint32_t)n_special, w, b, (T*)y, stats, rows, eps, param_f32 != 0)
    if (dtype == SVTAD_F16) {
        if (c == 128) SVTAD_LN(f16, 2);
        else SVTAD_LN(f16, 4);
    } else {
        if (c == 128) SVTAD_LN(bf16, 2);
        else SVTAD_LN(bf16, 4);
    }
#undef SVTAD_LN
    return launch_status();
}

extern "C" size_t svtad_layer_norm_bwd_workspace_bytes(int64_t rows, int c) {
    return rows <= 0 || c <= 0 ? 0 : (size_t)cdiv(rows, kLnRows) * 2 * c * 4;
}

extern "C" int svtad_layer_norm_bwd(const void* dy, const void* x, const void* add, const float* stats, const void* w,
                                    void* dx_special, void* dx, int64_t n_tokens, int64_t n_special, float* dwb,
                                    void* workspace, size_t workspace_bytes, int64_t rows, int c, int dtype,
                                    int param_f32, void* stream) {
    if (!half_type(dtype) || (c != 128 && c != 256))
        return set_error(SVTAD_ERR_UNSUPPORTED, "layer_norm_bwd: f16 / bf16 rows of 128 or 256 channels");
    if (rows < 1 || !split_ok(rows, n_tokens, n_special) || !dy || !x || !stats || !w || (!dx && (n_special == 0 || n_tokens > n_special)) ||
        (n_special > 0 && !dx_special) || !dwb || !workspace || !al16a(dy) || !al16a(x) || !al16a(add) || !al16a(dx_special) ||
        !al16a(dx))
        return set_error(SVTAD_ERR_INVALID, "layer_norm_bwd: bad arguments");
    if (workspace_bytes < svtad_layer_norm_bwd_workspace_bytes(rows, c))
        return set_error(SVTAD_ERR_WORKSPACE, "layer_norm_bwd: workspace too small");
    const int64_t wgs = cdiv(rows, kLnRows);
#define SVTAD_LN(T, V)                                                                                             \
    hipLaunchKernelGGL((k_ln_bwd<T, V>), dim3((unsigned)wgs), dim3(256), 0, (hipStream_t)stream, (const T*)dy, (const T*)x, \
                       (const T*)add, stats, w, (T*)dx_special, (T*)dx, (uint32_t)n_tokens, (uint32_t)n_special, (float*)workspace, rows, param_f32 != 0)
    if (dtype == SVTAD_F16) {
        if (c == 128) SVTAD_LN(f16, 2);
        else SVTAD_LN(f16, 4);
    } else {
        if (c == 128) SVTAD_LN(bf16, 2);
        else SVTAD_LN(bf16, 4);
    }
#undef SVTAD_LN
    split_reduce(SVTAD_F32, workspace, 2 * c, (int)wgs, dwb, (hipStream_t)stream);
    return launch_status();
}

extern "C" int svtad_key_attention_ok(int heads, int head_dim, int64_t n, int nk) {
    return heads == 4 && (head_dim == 16 || head_dim == 32) && nk >= 1 && nk <= 16 && n > nk;
}

static int key_attn_check(const char* what, int64_t batch, int64_t n, int nk, int hd, int dtype) {
    if (!half_type(dtype) || !svtad_key_attention_ok(4, hd, n, nk)) return set_error(SVTAD_ERR_UNSUPPORTED, what);
    if (batch < 1 || batch > 65535) return set_error(SVTAD_ERR_INVALID, what);
    return SVTAD_OK;
}

template <bool BWD>
static void launch_key_attn(const KeyAttnArgs& p, int64_t batch, int hd, int dtype, hipStream_t s) {
    const dim3 g((unsigned)cdiv(p.n, kAttnRows), (unsigned)batch);
#define SVTAD_KA(T, H)                                                                                 \
    if (p.nk <= 4) hipLaunchKernelGGL((k_key_attn<T, H, 4, BWD>), g, dim3(256), 0, s, p);              \
    else hipLaunchKernelGGL((k_key_attn<T, H, 16, BWD>), g, dim3(256), 0, s, p)
    if (dtype == SVTAD_F16) {
        if (hd == 16) { SVTAD_KA(f16, 16); } else { SVTAD_KA(f16, 32); }
    } else {
        if (hd == 16) { SVTAD_KA(bf16, 16); } else { SVTAD_KA(bf16, 32); }
    }
#undef SVTAD_KA
}

extern "C" int svtad_key_attention(const void* q, const void* kv, const void* qn_w, const void* qn_b, const void* kn_w,
                                   const void* kn_b, void* out, int64_t batch, int64_t n, int nk, int head_dim, float eps,
                                   int dtype, int param_f32, void* stream) {
    const int st = key_attn_check("key_attention: 4 heads of 16 or 32 channels, 1 to 16 keys, f16 / bf16", batch, n, nk,
                                  head_dim, dtype);
    if (st) return st;
    if (!q || !kv || !qn_w || !qn_b || !kn_w || !kn_b || !out) return set_error(SVTAD_ERR_INVALID, "key_attention: null pointer");
    const KeyAttnArgs p{q, kv, nullptr, qn_w, qn_b, kn_w, kn_b, out, nullptr, n, nk, eps, 1.f / sqrtf((float)head_dim),
                        param_f32 != 0};
    launch_key_attn<false>(p, batch, head_dim, dtype, (hipStream_t)stream);
    return launch_status();
}

static int64_t key_attn_part(int64_t batch, int64_t n, int nk, int hd) {
    return batch * cdiv(n, kAttnRows) * (2 * nk + 2) * 4 * hd;
}

// Samples per workgroup of k_key_attn_keys.
static int key_samples(int64_t batch, int nk) {
    return (int)(batch * nk <= kKeysInOne ? batch : cdiv(batch, std::min<int64_t>(batch, kKeyGroups)));
}

extern "C" size_t svtad_key_attention_bwd_workspace_bytes(int64_t batch, int64_t n, int nk, int head_dim) {
    if (batch < 1 || n < 1 || nk < 1 || head_dim < 1) return 0;
    const int64_t groups = cdiv(batch, key_samples(batch, nk));
    return (size_t)(key_attn_part(batch, n, nk, head_dim) + batch * (2 * nk + 2) * 4 * head_dim +
                    (groups > 1 ? groups * 4 * head_dim : 0)) * 4;
}

extern "C" int svtad_key_attention_bwd(const void* dout, const void* q, const void* kv, const void* qn_w, const void* qn_b,
                                       const void* kn_w, const void* kn_b, void* dq, void* dkv, float* dnorm,
                                       void* workspace, size_t workspace_bytes, int64_t batch, int64_t n, int nk,
                                       int head_dim, float eps, int dtype, int param_f32, void* stream) {
    const int st = key_attn_check("key_attention_bwd: 4 heads of 16 or 32 channels, 1 to 16 keys, f16 / bf16", batch, n, nk,
                                  head_dim, dtype);
    if (st) return st;
    if (!dout || !q || !kv || !qn_w || !qn_b || !kn_w || !kn_b || !dq || !dkv || !dnorm || !workspace)
        return set_error(SVTAD_ERR_INVALID, "key_attention_bwd: null pointer");
    if (workspace_bytes < svtad_key_attention_bwd_workspace_bytes(batch, n, nk, head_dim))
        return set_error(SVTAD_ERR_WORKSPACE, "key_attention_bwd: workspace too small");
    float* const part = (float*)workspace;
    float* const sums = part + key_attn_part(batch, n, nk, head_dim);
    const KeyAttnArgs p{q, kv, dout, qn_w, qn_b, kn_w, kn_b, dq, part, n, nk, eps, 1.f / sqrtf((float)head_dim),
                        param_f32 != 0};
    hipStream_t s = (hipStream_t)stream;
    launch_key_attn<true>(p, batch, head_dim, dtype, s);
    const int count = (2 * nk + 2) * 4 * head_dim;
    hipLaunchKernelGGL(k_key_attn_sum, dim3((unsigned)cdiv(count, 32), (unsigned)batch), dim3(256), 0, s, part, sums,
                       (int)cdiv(n, kAttnRows), count);
    const int per = key_samples(batch, nk), groups = (int)cdiv(batch, per);
    float* const dn = groups > 1 ? sums + batch * count : dnorm;
#define SVTAD_KK(T, H) \
    hipLaunchKernelGGL((k_key_attn_keys<T, H>), dim3((unsigned)groups), dim3(4 * H), 0, s, p, (const float*)sums, (int)batch, per, (T*)dkv, dn)
    if (dtype == SVTAD_F16) {
        if (head_dim == 16) SVTAD_KK(f16, 16);
        else SVTAD_KK(f16, 32);
    } else {
        if (head_dim == 16) SVTAD_KK(bf16, 16);
        else SVTAD_KK(bf16, 32);
    }
#undef SVTAD_KK
    if (groups > 1) split_reduce(SVTAD_F32, dn, 4 * head_dim, groups, dnorm, s);
    return launch_status();
}

static int key_proj_check(const char* what, int64_t batch, int64_t n, int nk, int a, int dtype) {
    if (!half_type(dtype) || (a != 64 && a != 128)) return set_error(SVTAD_ERR_UNSUPPORTED, what);
    if (batch < 1 || nk < 1 || n < nk || batch * nk > kKeyRowsMax) return set_error(SVTAD_ERR_UNSUPPORTED, what);
    return SVTAD_OK;
}

#define SVTAD_KP(K, ...)                                                            \
    if (dtype == SVTAD_F16) {                                                       \
        if (a == 64) { K(f16, 64); } else { K(f16, 128); }                          \
    } else {                                                                        \
        if (a == 64) { K(bf16, 64); } else { K(bf16, 128); }                        \
    }

extern "C" int svtad_key_proj(const void* xa, const void* w, const void* b, void* kv, int64_t batch, int64_t n, int nk, int a,
                              int dtype, void* stream) {
    const int st = key_proj_check("key_proj: f16 / bf16, a 64 or 128, at most 64 key rows", batch, n, nk, a, dtype);
    if (st) return st;
    if (!xa || !w || !b || !kv || !al16a(w)) return set_error(SVTAD_ERR_INVALID, "key_proj: bad pointer");
#define SVTAD_KP1(T, A)                                                                                            \
    hipLaunchKernelGGL((k_key_proj<T, A>), dim3((unsigned)(batch * nk)), dim3(2 * A), 0, (hipStream_t)stream, (const T*)xa, \
                       (const T*)w, (const T*)b, (T*)kv, n, nk)
    SVTAD_KP(SVTAD_KP1)
#undef SVTAD_KP1
    return launch_status();
}

extern "C" int svtad_key_proj_bwd(const void* dkv, const void* xa, const void* w, void* dxa, void* dw, void* db, int64_t batch,
                                  int64_t n, int nk, int a, int dtype, int dw_f32, int db_f32, void* stream) {
    const int st = key_proj_check("key_proj_bwd: f16 / bf16, a 64 or 128, at most 64 key rows", batch, n, nk, a, dtype);
    if (st) return st;
    if (!dkv || !xa || !w || !dxa || !dw || !db) return set_error(SVTAD_ERR_INVALID, "key_proj_bwd: null pointer");
#define SVTAD_KP1(T, A)                                                                                                \
    hipLaunchKernelGGL((k_key_proj_bwd<T, A>), dim3((unsigned)(2 * A + batch * nk)), dim3(A), 0, (hipStream_t)stream,  \
                       (const T*)dkv, (const T*)xa, (const T*)w, (T*)dxa, dw, db, n, nk, (int)(batch * nk), dw_f32 != 0, \
                       db_f32 != 0)
    SVTAD_KP(SVTAD_KP1)
#undef SVTAD_KP1
    return launch_status();
}
#undef SVTAD_KP
