// GEMMs of the sparse-conv adapter that keep a whole token tile in LDS
// (gfx950 MFMA): out = epilogue(A W^T) for the widths the adapters use, with
// the weight in fragment order (k_adapter_prep).
//
// All four products of the adapter's training step stream token rows whose
// bytes bound them (down projection and its mirror in the up projection's
// backward: [M, E] in; up projection and the input gradient: [M, E] in and
// out), so a workgroup issues every load of its tile at once: the token rows
// (converted to the compute type on the way into LDS when they are fp32, and
// stored once for the weight gradients), the first weight fragments and the
// residual. There is one barrier, between the LDS writes and the products;
// the waves of a workgroup own different columns and run apart after it.
#include <algorithm>

#include "sv_common.h"
#include "sv_conv.h"
#include "sv_internal.h"
#include "sv_mfma.h"

namespace svtad {

// Column of the 16-row weight fragment f, fragment row rr (0 .. 15), within
// the tile of a wave: a lane of the MFMA result holds fragment rows 4 g .. 4 g
// + 3. Natural order: 16 consecutive columns per fragment. Pair order
// (outputs stored from the MFMA layout): fragments 2 p and 2 p + 1 interleave
// in groups of 4 columns, so a lane's 8 values of a pair are 16 bytes.
__host__ __device__ __forceinline__ int frag_col(bool pair, int f, int rr) {
    return pair ? (f >> 1) * 32 + (rr >> 2) * 8 + (f & 1) * 4 + (rr & 3) : f * 16 + rr;
}

// ---------------------------------------------------------------------------
// preparation: casts and fragment layouts of the adapter's parameters, one launch
// ---------------------------------------------------------------------------
struct PrepJobs {
    svtad_prep_job j[kMaxPrepJobs];
    int first[kMaxPrepJobs + 1];  // first workgroup of each job
    int count;
};

// Outputs of a job.
__host__ __device__ __forceinline__ int64_t prep_outputs(const svtad_prep_job& j) {
    return j.kind == SVTAD_PREP_TOKEN_ROWS ? (int64_t)j.off * (j.pair ? j.n - j.k : j.n) : (int64_t)j.off * j.n * j.k;
}

// One thread per 8 output values. The values go through T first (autocast's
// cast) and, with gamma, through T again after the product, as the separate
// casts and multiply round them.
template <typename T>
__global__ __launch_bounds__(256) void k_adapter_prep(PrepJobs jobs) {
    int q = 0;
    while (q + 1 < jobs.count && (int)blockIdx.x >= jobs.first[q + 1]) ++q;
    const svtad_prep_job j = jobs.j[q];
    const int64_t slot = (int64_t)((int)blockIdx.x - jobs.first[q]) * 256 + threadIdx.x;
    const int64_t total = prep_outputs(j);
    if (j.kind == SVTAD_PREP_CONV_BWD && slot == 0) *(uint32_t*)((T*)j.dst + total) = 0u;  // orphan flag after the layout
    if (slot * 8 >= total) return;
    if (j.kind == SVTAD_PREP_TOKEN_ROWS) {
        // written by the training forward's one launch: a list kept between
        // calls would have to follow streams and graph captures
        const uint32_t S = (uint32_t)j.k, P = (uint32_t)(j.n - j.k), head = j.pair ? 0u : (uint32_t)j.off * S;
        for (int64_t e = slot * 8; e < total && e < slot * 8 + 8; ++e) {
            const uint32_t t = (uint32_t)e;
            const uint32_t b = t < head ? t / S : (t - head) / P;
            ((int32_t*)j.dst)[e] = (int32_t)(b * (uint32_t)j.n + (t < head ? t - b * S : S + (t - head) - b * P));
        }
        return;
    }
    if (j.kind == SVTAD_PREP_WIDEN) {
        const u32x4 v = *(const u32x4*)((const T*)j.src + slot * 8);
        f32x4 o[2];
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e >> 2][e & 3] = (float)__builtin_bit_cast(T, (u16)((e & 1) ? v[e >> 1] >> 16 : v[e >> 1] & 0xffffu));
        *(f32x4*)((float*)j.dst + slot * 8) = o[0];
        *(f32x4*)((float*)j.dst + slot * 8 + 4) = o[1];
        return;
    }
    const float gm = !j.gamma ? 1.f : j.gamma_f32 ? *(const float*)j.gamma : (float)*(const T*)j.gamma;
    auto at = [&](int64_t i) -> T {
        const T v = j.src_f32 ? (T)f32_rounded(((const float*)j.src)[i]) : ((const T*)j.src)[i];
        return j.gamma ? (T)f32_rounded((float)v * gm) : v;
    };
    // element e of the slot is src[base + e * step]
    int64_t base, step = 1;
    const int lane = (int)(slot & 63), g = lane >> 4, rr = lane & 15;
    if (j.kind == SVTAD_PREP_CAST) {
        base = slot * 8;
    } else {
        // fragments of the [n, k] operand: (offset, step of 32 k values, block of 16 n), 64 lanes each
        const int nb = j.n / 16, ncs = j.k / 32;
        int64_t f = slot >> 6;
        const int b = (int)(f % nb);
        f /= nb;
        const int cs = (int)(f % ncs), off = (int)(f / ncs);
        const int c = cs * 32 + g * 8;
        int n = b * 16 + rr;
        if (j.kind == SVTAD_PREP_ROWS || j.kind == SVTAD_PREP_COLS) n = (b & ~1) * 16 + frag_col(j.pair, b & 1, rr);
        const int64_t o = (int64_t)off * j.n * j.k;
        if (j.kind == SVTAD_PREP_ROWS || j.kind == SVTAD_PREP_CONV_BWD) {
            base = o + (int64_t)n * j.k + c;  // src [n, k]
        } else {
            base = o + (int64_t)c * j.n + n;  // src [k, n]
            step = j.n;
        }
    }
    u16 v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = __builtin_bit_cast(u16, at(base + e * step));
    u32x4 o;
#pragma unroll
    for (int h = 0; h < 4; ++h) o[h] = (unsigned)v[2 * h] | ((unsigned)v[2 * h + 1] << 16);
    *(u32x4*)((T*)j.dst + slot * 8) = o;
}

// ---------------------------------------------------------------------------
// the GEMM
// ---------------------------------------------------------------------------
struct RowsArgs {
    const void* a0;   // A rows: [M, K], or the special-token rows
    const void* a1;   // with the split source, the patch rows
    const void* w;    // fragment order
    const void* bias; // T [N] or NULL
    const void* gamma;
    const void* res;  // [M, N]
    void* a_copy;     // T [M, K]: the converted A rows (NULL: not stored)
    void* out0;
    void* out1;
    void* out2;
    int64_t m_rows;
    int n_out;
    uint32_t n_tokens, n_special;  // split of a sample's tokens
    int n_col_groups;
    int64_t n_tiles;
};

enum { ROWS_GELU = 0, ROWS_SPLIT = 1, ROWS_RES = 2, ROWS_PLAIN = 3 };

__device__ __forceinline__ float gelu_erf_rows(float u) { return 0.5f * u * (1.0f + erff(u * 0.70710678118654752f)); }

// Measured at 17250 rows, E = 768, h = 256 (calls back to back; the copy rate
// of this card gives 20, 18, 24 and 24 us for their bytes): fp32 rows in, down
// projection 32 us (cast 16 + GEMM on 64 x 64 tiles 24.5 before), its mirror
// 27 us (cast 16, library GEMM 24 and slice copy 7), up projection with fp32
// residual 27 us (36), input gradient 25 us (library GEMM 20, conversion 13,
// addition 24). Non-temporal loads and stores made the fp32 ones 36, 30, 41 and
// 40 us, 128 columns x 64 rows beat 256 x 32 (32 us) and 128 x 32 (45 us).
//
// EPI: ROWS_GELU   out0 = z = T(acc + bias); GELU(z) split into out1 (special)
//                  and out2 (patch rows)
//      ROWS_SPLIT  T(acc) split into out1 and out2
//      ROWS_PLAIN  out0 = T(acc + bias)
//      ROWS_RES    with gamma: out0 = T?(z) gamma + res, else out0 = acc + res
// AF32: A rows are fp32. ASPLIT: A rows come from a0 / a1 by token kind.
// GF32 / RF32 / OF32: gamma, residual, output in fp32 (else T); a fp32 gamma
// makes the product and the sum fp32, as in the reference under autocast.
template <typename T, int EPI, int K, int FM, int FN, int D, bool AF32, bool ASPLIT, bool GF32, bool RF32, bool OF32>
__global__ __launch_bounds__(256, K > 768 && FM == 2 ? 2 : 3) void k_adapter_rows(RowsArgs p) {
    constexpr int BM = 16 * FM, NC = K / KS;
    constexpr int CPR = K / 8;  // 16-byte chunks of an LDS row, chunk q of row m at q ^ (m & 7)
    constexpr bool PAIR = EPI != ROWS_RES;
    constexpr int BN = 64 * FN;  // columns of the workgroup
    constexpr int OP = BN + 4;   // pitch (floats) of the output tile in LDS (ROWS_RES)
    static_assert(K % 64 == 0 && NC % D == 0 && FN % 2 == 0, "shape");
    __shared__ __align__(16) u16 As[EPI == ROWS_RES && BM * OP * 2 > BM * K ? BM * OP * 2 : BM * K];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, r16 = lane & 15;
    const int64_t tile = xcd_tile(blockIdx.x, p.n_tiles);
    const int64_t row0 = (tile / p.n_col_groups) * BM;
    const int col0 = ((int)(tile % p.n_col_groups) * 4 + wave) * FN * 16;
    const uint32_t n_patch = p.n_tokens - p.n_special;
    auto split = [&](int64_t m, bool& sp) -> int64_t {
        const uint32_t b = (uint32_t)m / p.n_tokens, r = (uint32_t)m - b * p.n_tokens;
        sp = r < p.n_special;
        return sp ? (int64_t)b * p.n_special + r : (int64_t)b * n_patch + (r - p.n_special);
    };

    // Rows past the end are out-of-range loads (zeros) and stores (dropped):
    // no branches, and 32-bit offsets from a scalar base.
    const int rows = (int)min<int64_t>(BM, p.m_rows - row0);
    auto tile_rsrc = [&](const void* base, int width, int size) {
        return make_rsrc((const char*)base + row0 * width * size, (uint32_t)rows * (uint32_t)(width * size));
    };
    // every load of the tile: the A rows (contiguous unless split), ...
    constexpr int EPT = AF32 ? 4 : 8;                    // A elements per load
    constexpr int LPR = K / EPT;                         // loads per row
    constexpr int A_PER = BM * LPR / 256;
    static_assert(A_PER * 256 == BM * LPR, "loads per thread");
    u32x4 ra[A_PER];
    if constexpr (ASPLIT) {
#pragma unroll
        for (int q = 0; q < A_PER; ++q) {
            const int e = tid + q * 256;
            bool sp;
            const int64_t r = split(min<int64_t>(row0 + e / LPR, p.m_rows - 1), sp);
            ra[q] = *(const u32x4*)((const T*)(sp ? p.a0 : p.a1) + r * K + (e % LPR) * EPT);
        }
    } else {
        const rsrc_t rsa = tile_rsrc(p.a0, K, AF32 ? 4 : 2);
#pragma unroll
        for (int q = 0; q < A_PER; ++q)
            ra[q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsa, (uint32_t)(tid * 16 + q * 4096), 0, 0));
    }
    // ... the residual, in the pieces of whole rows that the epilogue stores, ...
    constexpr int PW = OF32 ? 4 : 8;  // columns per 16-byte piece of the output
    constexpr int PPR = BN / PW;      // pieces per tile row
    constexpr int R_PER = BM * PPR / 256;
    constexpr int R4 = RF32 ? PW / 4 : 1;
    static_assert(EPI != ROWS_RES || R_PER * 256 == BM * PPR, "pieces per thread");
    const int wgcol0 = (int)(tile % p.n_col_groups) * BN;
    u32x4 rres[EPI == ROWS_RES ? R_PER : 1][R4];
    if constexpr (EPI == ROWS_RES) {
        constexpr int RS = RF32 ? 4 : 2;
        const rsrc_t rsr = tile_rsrc(p.res, p.n_out, RS);
#pragma unroll
        for (int q = 0; q < R_PER; ++q) {
            const int e = tid + q * 256;
            const uint32_t o = (uint32_t)((e / PPR) * p.n_out + wgcol0 + (e % PPR) * PW) * RS;
            if constexpr (RF32 || !OF32) {
#pragma unroll
                for (int h = 0; h < R4; ++h)
                    rres[q][h] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsr, o + h * 16, 0, 0));
            } else {
                typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
                const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rsr, o, 0, 0));
                rres[q][0] = u32x4{t[0], t[1], 0u, 0u};
            }
        }
    }
    // ... and the first D steps of the wave's weight fragments
    const rsrc_t rw = make_rsrc(p.w, (uint32_t)p.n_out * (uint32_t)K * 2u);
    const uint32_t wo = (uint32_t)(col0 / 16) * 1024u + (uint32_t)lane * 16u;
    const uint32_t step_bytes = (uint32_t)(p.n_out / 16) * 1024u;
    u32x4 ring[D][FN];
    auto load_w = [&](int cs, int d) {
#pragma unroll
        for (int f = 0; f < FN; ++f)
            ring[d][f] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, wo + (uint32_t)f * 1024u, (uint32_t)cs * step_bytes, 0));
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load_w(d, d);

    // A rows into LDS in the compute type
    const rsrc_t rsc = AF32 && p.a_copy ? tile_rsrc(p.a_copy, K, 2) : make_rsrc(p.a0, 0u);
#pragma unroll
    for (int q = 0; q < A_PER; ++q) {
        const int e = tid + q * 256;
        const int m = e / LPR, c = (e % LPR) * EPT;
        u16* const dst = &As[m * K + (((c >> 3) ^ (m & 7)) << 3) + (c & 7)];
        if constexpr (AF32) {
            u16 h[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) h[j] = __builtin_bit_cast(u16, (T)__uint_as_float(ra[q][j]));
            const uint2 t = {(unsigned)h[0] | ((unsigned)h[1] << 16), (unsigned)h[2] | ((unsigned)h[3] << 16)};
            *(uint2*)dst = t;
            if (p.a_copy) {  // uniform
                typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
                __builtin_amdgcn_raw_buffer_store_b64(u32x2{t.x, t.y}, rsc, (uint32_t)(tid * 8 + q * 2048), 0, 0);
            }
        } else {
            *(u32x4*)dst = ra[q];
        }
    }
    __syncthreads();

    f32x4 acc[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int f = 0; f < FN; ++f) acc[a][f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int cs = 0; cs < NC; ++cs) {
        u32x4 fa[FM];
#pragma unroll
        for (int a = 0; a < FM; ++a) fa[a] = *(const u32x4*)&As[(a * 16 + r16) * K + (((cs * 4 + g) ^ (r16 & 7)) << 3)];
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int f = 0; f < FN; ++f) acc[a][f] = MfmaOp<T>::run(ring[cs % D][f], fa[a], acc[a][f]);
        if (cs + D < NC) load_w(cs + D, cs % D);
    }

    // epilogue: lane (g, r) holds, of row r of each fragment, columns
    // frag_col(PAIR, f, 4 g) .. + 3
    float gm = 1.f;
    if (EPI == ROWS_RES && p.gamma) gm = GF32 ? *(const float*)p.gamma : (float)*(const T*)p.gamma;  // uniform
    float bv[FN][4];
#pragma unroll
    for (int f = 0; f < FN; ++f)
#pragma unroll
        for (int j = 0; j < 4; ++j) bv[f][j] = 0.f;
    if (EPI != ROWS_SPLIT && p.bias) {  // uniform
#pragma unroll
        for (int f = 0; f < FN; ++f) {
            const uint2 t = *(const uint2*)((const T*)p.bias + col0 + frag_col(PAIR, f, g * 4));
            bv[f][0] = (float)__builtin_bit_cast(T, (u16)(t.x & 0xffffu));
            bv[f][1] = (float)__builtin_bit_cast(T, (u16)(t.x >> 16));
            bv[f][2] = (float)__builtin_bit_cast(T, (u16)(t.y & 0xffffu));
            bv[f][3] = (float)__builtin_bit_cast(T, (u16)(t.y >> 16));
        }
    }
    if constexpr (EPI == ROWS_RES) {
        // (c W^T + b) rounded to T, times gamma (fp32, or rounded to T), as
        // fp32 through LDS, so that whole rows meet the residual and leave in
        // 16-byte pieces of consecutive lanes (16 rows of 64-byte segments per
        // load and store, straight in the MFMA layout: 34 us against 27)
        float* const ot = (float*)As;
        __syncthreads();  // every wave has read its A fragments
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int f = 0; f < FN; ++f) {
                f32x4 t;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float z = acc[a][f][j] + bv[f][j];
                    t[j] = z;
                    if (p.gamma) {
                        const float y = f32_rounded((float)(T)z * gm);
                        t[j] = GF32 ? y : (float)(T)y;
                    }
                }
                *(f32x4*)&ot[(a * 16 + r16) * OP + wave * FN * 16 + f * 16 + g * 4] = t;
            }
        __syncthreads();
        constexpr int OS = OF32 ? 4 : 2;
        const rsrc_t rso = tile_rsrc(p.out0, p.n_out, OS);
#pragma unroll
        for (int q = 0; q < R_PER; ++q) {
            const int e = tid + q * 256;
            const int m = e / PPR, c = (e % PPR) * PW;
            float y[PW];
#pragma unroll
            for (int h = 0; h < PW / 4; ++h) {
                const f32x4 t = *(const f32x4*)&ot[m * OP + c + h * 4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float r;
                    if constexpr (RF32) {
                        const unsigned u = rres[q][h][j];
                        r = __uint_as_float(u);
                    } else {
                        const unsigned u = rres[q][0][(h * 4 + j) >> 1];
                        r = (float)__builtin_bit_cast(T, (u16)((j & 1) ? u >> 16 : u & 0xffffu));
                    }
                    y[h * 4 + j] = f32_rounded(t[j] + r);
                }
            }
            u32x4 o;
            if constexpr (OF32) {
                o = u32x4{__float_as_uint(y[0]), __float_as_uint(y[1]), __float_as_uint(y[2]), __float_as_uint(y[3])};
            } else {
#pragma unroll
                for (int h = 0; h < 4; ++h)
                    o[h] = (unsigned)__builtin_bit_cast(u16, (T)y[2 * h]) |
                           ((unsigned)__builtin_bit_cast(u16, (T)y[2 * h + 1]) << 16);
            }
            __builtin_amdgcn_raw_buffer_store_b128(o, rso, (uint32_t)(m * p.n_out + wgcol0 + c) * OS, 0, 0);
        }
        return;
    }
    // 16-bit outputs from the MFMA layout, 16 bytes per pair of fragments
    const uint32_t oel = (uint32_t)(r16 * p.n_out + col0 + g * 8);  // first output element of the lane in the tile
    const rsrc_t rso = EPI != ROWS_SPLIT ? tile_rsrc(p.out0, p.n_out, 2) : make_rsrc(p.a0, 0u);
#pragma unroll
    for (int a = 0; a < FM; ++a) {
        const int64_t m = row0 + a * 16 + r16;
        const bool ok = m < p.m_rows;
        bool sp = false;
        const int64_t rs = EPI == ROWS_PLAIN ? 0 : split(ok ? m : 0, sp);
#pragma unroll
        for (int v = 0; v < FN / 2; ++v) {
            u32x4 o, ge;
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                const int f = 2 * v + (h >> 1), j = (h & 1) * 2;
                const T lo = (T)(acc[a][f][j] + bv[f][j]), hi = (T)(acc[a][f][j + 1] + bv[f][j + 1]);
                o[h] = (unsigned)__builtin_bit_cast(u16, lo) | ((unsigned)__builtin_bit_cast(u16, hi) << 16);
                if constexpr (EPI == ROWS_GELU)
                    ge[h] = (unsigned)__builtin_bit_cast(u16, (T)gelu_erf_rows((float)lo)) |
                            ((unsigned)__builtin_bit_cast(u16, (T)gelu_erf_rows((float)hi)) << 16);
            }
            if constexpr (EPI != ROWS_SPLIT)
                __builtin_amdgcn_raw_buffer_store_b128(o, rso, (oel + (uint32_t)(a * 16 * p.n_out + v * 32)) * 2u, 0, 0);
            if (EPI != ROWS_PLAIN && ok) *(u32x4*)((T*)(sp ? p.out1 : p.out2) + rs * p.n_out + col0 + v * 32 + g * 8) = EPI == ROWS_GELU ? ge : o;
        }
    }
}

template <typename T, int EPI, int K, int FM, int FN, int D, bool AF32, bool ASPLIT, bool GF32, bool RF32, bool OF32>
static void launch_rows(RowsArgs p, hipStream_t s) {
    p.n_col_groups = p.n_out / (64 * FN);
    p.n_tiles = cdiv(p.m_rows, 16 * FM) * p.n_col_groups;
    hipLaunchKernelGGL((k_adapter_rows<T, EPI, K, FM, FN, D, AF32, ASPLIT, GF32, RF32, OF32>), dim3((unsigned)p.n_tiles),
                       dim3(256), 0, s, p);
}

// Rows per workgroup: 32 (16 where that leaves CUs without a workgroup) where
// the tile's K is the embedding width (16 at 17250 rows: 33.4 us against 31.9,
// 16-bit rows 27.8 against 23.5), 64 (32) where it is the hidden width.
template <typename T, int EPI, int K, bool AF32>
static void rows_in(const RowsArgs& p, hipStream_t s) {
    const bool few = cdiv(p.m_rows, 32) < cu_count();
    if (p.n_out == 256) {
        if (few) launch_rows<T, EPI, K, 1, 4, 4, AF32, false, false, false, false>(p, s);
        else launch_rows<T, EPI, K, 2, 4, 4, AF32, false, false, false, false>(p, s);
    } else {
        if (few) launch_rows<T, EPI, K, 1, 2, 4, AF32, false, false, false, false>(p, s);
        else launch_rows<T, EPI, K, 2, 2, 4, AF32, false, false, false, false>(p, s);
    }
}

template <typename T, int K, bool ASPLIT, bool GF32, bool RF32, bool OF32>
static void rows_out(const RowsArgs& p, hipStream_t s) {
    constexpr int D = K / KS < 8 ? K / KS : 8;
    if (cdiv(p.m_rows, 64) * (p.n_out / 128) < 2 * cu_count())
        launch_rows<T, ROWS_RES, K, 2, 2, D, false, ASPLIT, GF32, RF32, OF32>(p, s);
    else
        launch_rows<T, ROWS_RES, K, 4, 2, D, false, ASPLIT, GF32, RF32, OF32>(p, s);
}

template <typename T, int EPI>
static bool rows_in_k(const RowsArgs& p, int k, bool f32, hipStream_t s) {
#define SVTAD_K(KK)                                                    \
    if (k == KK) {                                                     \
        if (f32) rows_in<T, EPI, KK, true>(p, s);                      \
        else rows_in<T, EPI, KK, false>(p, s);                         \
        return true;                                                   \
    }
    SVTAD_K(384)
    SVTAD_K(768)
    SVTAD_K(1024)
#undef SVTAD_K
    return false;
}

template <typename T>
static bool rows_gemm(const RowsArgs& p, int epi, int k, bool af32, bool asplit, bool g32, bool r32, bool o32, hipStream_t s) {
    if (epi == ROWS_GELU) return rows_in_k<T, ROWS_GELU>(p, k, af32, s);
    if (epi == ROWS_SPLIT) return rows_in_k<T, ROWS_SPLIT>(p, k, af32, s);
    if (epi == ROWS_PLAIN) {  // 17250 rows, 256 -> 128, 128 -> 128, 128 -> 256: 6.3, 5.4, 6.6 us
        if (af32) return false;
        if (k == 128) launch_rows<T, ROWS_PLAIN, 128, 2, 2, 4, false, false, false, false, false>(p, s);
        else launch_rows<T, ROWS_PLAIN, 256, 2, 2, 8, false, false, false, false, false>(p, s);
        return true;
    }
#define SVTAD_O(KK, SP, G, R, O)                                                              \
    if (k == KK && asplit == SP && g32 == G && r32 == R && o32 == O) {                        \
        rows_out<T, KK, SP, G, R, O>(p, s);                                                   \
        return true;                                                                          \
    }
#define SVTAD_OK(KK, SP)              \
    SVTAD_O(KK, SP, false, false, false) \
    SVTAD_O(KK, SP, true, true, true)    \
    SVTAD_O(KK, SP, true, false, true)   \
    SVTAD_O(KK, SP, true, true, false)   \
    SVTAD_O(KK, SP, true, false, false)
    SVTAD_OK(128, true)
    SVTAD_OK(256, true)
    SVTAD_OK(128, false)
    SVTAD_OK(256, false)
    SVTAD_O(128, false, false, true, true)  // no gamma: the input gradient under autocast
    SVTAD_O(256, false, false, true, true)
    SVTAD_O(64, false, false, false, false)
    SVTAD_O(64, false, true, false, false)
#undef SVTAD_OK
#undef SVTAD_O
    return false;
}

static bool al16r(const void* p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace svtad

using namespace svtad;

extern "C" int svtad_adapter_prep(const svtad_prep_job* jobs, int count, int dtype, void* stream) {
    if (dtype != SVTAD_F16 && dtype != SVTAD_BF16)
        return set_error(SVTAD_ERR_UNSUPPORTED, "adapter_prep: needs f16/bf16");
    if (count < 0 || count > kMaxPrepJobs || (count > 0 && !jobs))
        return set_error(SVTAD_ERR_INVALID, "adapter_prep: bad job list");
    PrepJobs pj;
    pj.count = count;
    int64_t blocks = 0;
    for (int q = 0; q < count; ++q) {
        const svtad_prep_job& j = jobs[q];
        const bool list = j.kind == SVTAD_PREP_TOKEN_ROWS;
        if ((!j.src && !list) || !j.dst || !al16r(j.dst) || j.kind < SVTAD_PREP_CAST || j.kind > SVTAD_PREP_TOKEN_ROWS ||
            j.off < 1 || j.n < 1 || j.k < (list ? 0 : 1) || (list && (j.k > j.n || (int64_t)j.off * j.n >= (int64_t)INT32_MAX)))
            return set_error(SVTAD_ERR_INVALID, "adapter_prep: bad job");
        if (j.kind == SVTAD_PREP_WIDEN && (!al16r(j.src) || j.src_f32 || j.gamma))
            return set_error(SVTAD_ERR_INVALID, "adapter_prep: bad job");
        if (!list && (j.kind == SVTAD_PREP_CAST || j.kind == SVTAD_PREP_WIDEN ? (int64_t)j.off * j.n * j.k % 8 != 0 : (j.k % 32 != 0 || j.n % 32 != 0)))
            return set_error(SVTAD_ERR_UNSUPPORTED, "adapter_prep: shape without a layout");
        if (prep_outputs(j) >= (int64_t)INT32_MAX)
            return set_error(SVTAD_ERR_UNSUPPORTED, "adapter_prep: 2^31 values or more");
        pj.j[q] = j;
        pj.first[q] = (int)blocks;
        blocks += cdiv(prep_outputs(j), 2048);
    }
    pj.first[count] = (int)blocks;
    if (blocks == 0) return SVTAD_OK;
    if (dtype == SVTAD_F16)
        hipLaunchKernelGGL(k_adapter_prep<f16>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, pj);
    else
        hipLaunchKernelGGL(k_adapter_prep<bf16>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, pj);
    return launch_status();
}

extern "C" int svtad_adapter_rows_ok(int kind, int k, int n) {
    if (kind == SVTAD_ROWS_PLAIN) return (k == 128 || k == 256) && n > 0 && n % 128 == 0;
    if (kind == SVTAD_ROWS_RES) return (k == 64 || k == 128 || k == 256) && n > 0 && n % 128 == 0;
    return (kind == SVTAD_ROWS_GELU || kind == SVTAD_ROWS_SPLIT) && (k == 384 || k == 768 || k == 1024) &&
           (n == 128 || n == 256);
}

extern "C" int svtad_adapter_rows(const svtad_rows_args* a, int dtype, void* stream) {
    if (dtype != SVTAD_F16 && dtype != SVTAD_BF16)
        return set_error(SVTAD_ERR_UNSUPPORTED, "adapter_rows: needs f16/bf16");
    if (!a || a->batch < 0 || a->n_tokens < 0 || a->n_special < 0 || a->n_special > a->n_tokens)
        return set_error(SVTAD_ERR_INVALID, "adapter_rows: bad sizes");
    const int64_t rows = a->batch * a->n_tokens;
    if (!svtad_adapter_rows_ok(a->kind, a->k, a->n) || rows >= (int64_t)INT32_MAX)
        return set_error(SVTAD_ERR_UNSUPPORTED, "adapter_rows: shape without a kernel");
    if (rows == 0) return SVTAD_OK;
    const bool res = a->kind == SVTAD_ROWS_RES;
    const bool any_sp = a->n_special > 0, any_pa = a->n_tokens > a->n_special;
    const bool split_src = res && a->a_patch_split;
    if (!a->w || (split_src ? (any_sp && !a->a0) || (any_pa && !a->a1) : !a->a0) ||
        (res ? !a->res || !a->out0 : a->kind != SVTAD_ROWS_PLAIN && ((any_sp && !a->out1) || (any_pa && !a->out2))) ||
        ((a->kind == SVTAD_ROWS_GELU || a->kind == SVTAD_ROWS_PLAIN) && !a->out0))
        return set_error(SVTAD_ERR_INVALID, "adapter_rows: null pointer");
    for (const void* q : {a->a0, a->a1, a->w, a->bias, a->res, (const void*)a->a_copy, (const void*)a->out0,
                          (const void*)a->out1, (const void*)a->out2})
        if (!al16r(q)) return set_error(SVTAD_ERR_INVALID, "adapter_rows: buffers need 16-byte alignment");
    RowsArgs p;
    p.a0 = a->a0;
    p.a1 = a->a1;
    p.w = a->w;
    p.bias = a->bias;
    p.gamma = a->gamma;
    p.res = a->res;
    p.a_copy = a->a_copy;
    p.out0 = a->out0;
    p.out1 = a->out1;
    p.out2 = a->out2;
    p.m_rows = rows;
    p.n_out = a->n;
    p.n_tokens = (uint32_t)a->n_tokens;
    p.n_special = (uint32_t)a->n_special;
    const int epi = a->kind;  // the public kinds are ROWS_*
    const bool done = dtype == SVTAD_F16
                          ? rows_gemm<f16>(p, epi, a->k, a->a_f32, split_src, a->gamma_f32, a->res_f32, a->out_f32, (hipStream_t)stream)
                          : rows_gemm<bf16>(p, epi, a->k, a->a_f32, split_src, a->gamma_f32, a->res_f32, a->out_f32, (hipStream_t)stream);
    if (!done) return set_error(SVTAD_ERR_UNSUPPORTED, "adapter_rows: combination of types without a kernel");
    return launch_status();
}
