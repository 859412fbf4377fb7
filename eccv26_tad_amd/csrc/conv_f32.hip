// float32 SparseConv2D kernels on the matrix cores (v_mfma_f32_16x16x4_f32:
// fp32 products and fp32 accumulation, 256 flop per clock and CU, twice the
// vector rate). The fp32 MFMA is slow enough against the L2 that no operand
// goes through LDS: each wave loads its fragments from global memory, D steps
// ahead in registers, and waves share no state but an optional split of the
// offsets.
#include <algorithm>

#include "sv_common.h"
#include "sv_conv.h"
#include "sv_internal.h"
#include "sv_mfma.h"

namespace svtad {

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// N consecutive floats at byte offset off (dword aligned), zeros out of range.
template <int N>
__device__ __forceinline__ void bload_f32(rsrc_t r, uint32_t off, float* v) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x3 __attribute__((ext_vector_type(3)));
    if constexpr (N == 4) {
        const u32x4 t = bload16(r, off);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __uint_as_float(t[j]);
    } else if constexpr (N == 3) {
        const u32x3 t = __builtin_bit_cast(u32x3, __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, 0));
#pragma unroll
        for (int j = 0; j < 3; ++j) v[j] = __uint_as_float(t[j]);
    } else {
        static_assert(N == 2, "2, 3 or 4 floats");
        const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
#pragma unroll
        for (int j = 0; j < 2; ++j) v[j] = __uint_as_float(t[j]);
    }
}

template <int N>
__device__ __forceinline__ void bstore_f32(rsrc_t r, uint32_t off, const float* v) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x3 __attribute__((ext_vector_type(3)));
    auto b = [&](int j) { return __float_as_uint(v[j]); };
    if constexpr (N == 4) __builtin_amdgcn_raw_buffer_store_b128(u32x4{b(0), b(1), b(2), b(3)}, r, off, 0, 0);
    else if constexpr (N == 3) __builtin_amdgcn_raw_buffer_store_b96(u32x3{b(0), b(1), b(2)}, r, off, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b64(u32x2{b(0), b(1)}, r, off, 0, 0);
}

// Gathered GEMM (forward / backward-input): a wave owns 16 FM rows and 16 FN
// columns. The four waves of a workgroup are wgn column tiles x wgk offset
// sets x row tiles; offset set h takes every wgk-th of the offsets that a row
// of the tile uses, and the sets' sums are added in order through LDS.
//
// A step is 16 reduction values, four MFMA steps: lane (g = lane / 16,
// r = lane % 16) holds values 4 g .. 4 g + 3 of row r as one 16-byte load, and
// MFMA step s takes value 4 g + s of every group, for both operands. Column r
// of fragment f is column FN r + f of the tile, so the forward reads FN
// consecutive weights per reduction value and stores FN consecutive outputs;
// backward-input reads four consecutive weights per column. The weight is the
// MFMA's first operand: lane (g, r) then holds columns FN (4 g + j) + f of row
// r. Missing neighbors and reduction values past c_red are out-of-range
// loads (zeros); columns past n_out are not stored.
//
// Bound by the matrix cores and the load path together at large row counts
// (21952 x 128 at 70 % keep: forward 203 us with 64 x 64 tiles through LDS on
// the vector units, 65 us here, 100 TFLOP/s of the dense products;
// backward-input 181 -> 76 us) and by a wave's chain of load latencies at
// small ones (784 rows of 48 channels: 67 -> 7.8 us and 62 -> 7.7 us), which
// the offset sets shorten.
template <int MODE, int FM, int FN, int D>
__global__ __launch_bounds__(256) void k_gg_f32(const float* __restrict__ src, const int32_t* __restrict__ nbr,
                                                const float* __restrict__ w, const float* __restrict__ bias,
                                                float* __restrict__ out, int64_t n, int c_red, int n_out,
                                                int64_t tpb, int wgn, int wgk, int n_col_groups, int64_t n_tiles,
                                                bool sym) {
    constexpr int BM = 16 * FM;
    __shared__ int32_t sidx[4][9][BM];
    __shared__ __align__(16) f32x4 red[3][FM * FN][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, r16 = lane & 15;
    const int wn = wave % wgn, set = (wave / wgn) % wgk, wm = wave / (wgn * wgk);
    const int wgm = 4 / (wgn * wgk);
    const int64_t tile = xcd_tile(blockIdx.x, n_tiles);
    const int64_t row0 = ((tile / n_col_groups) * wgm + wm) * BM;
    const int col0 = ((int)(tile % n_col_groups) * wgn + wn) * 16 * FN;

    // source rows of the wave's tile, by offset
    for (int e = lane; e < 9 * BM; e += 64) {
        const int m = e / 9, kk = e - m * 9;
        const int64_t i = row0 + m;
        const int k = MODE == MODE_FWD ? kk : 8 - kk;
        int64_t r = -1;
        if (i < n) {
            r = src_row(nbr, i, kk, n, tpb);
            // transposed source of offset k: entry (i, 8 - k), accepted when
            // its partner points back (src_row_t)
            if (MODE != MODE_FWD && !sym && r >= 0 && src_row(nbr, r, k, n, tpb) != i) r = -1;
        }
        sidx[wave][k][m] = (int32_t)r;
    }
    __syncthreads();
    // this set's offsets
    unsigned mine = 0;
    int count = 0;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const bool any = __ballot(lane < BM && sidx[wave][k][lane < BM ? lane : 0] >= 0) != 0;
        if (any) {
            if (count % wgk == set) mine |= 1u << k;
            ++count;
        }
    }
    mine = __builtin_amdgcn_readfirstlane(mine);
    const int nc = (c_red + 15) / 16;
    const int steps = col0 < n_out ? __popc(mine) * nc : 0;  // a column tile past n_out: nothing

    const rsrc_t rs = make_rsrc(src, (uint32_t)(n * c_red * 4));
    const rsrc_t rw = make_rsrc(w, 9u * (uint32_t)c_red * (uint32_t)n_out * 4u);
    float fa[D][FM][4], fb[D][FN][4];
    uint32_t voff[FM];  // byte offset of the lane's row in src for the offset being loaded
    uint32_t wk = 0;    // byte offset of that offset's weight
    int cl = nc * 16;   // reduction value of the next load
    unsigned rest = mine;
    auto load = [&](int d) {
        if (cl >= nc * 16) {  // uniform: the next offset
            const int k = rest ? __builtin_ctz(rest) : 0;
#pragma unroll
            for (int a = 0; a < FM; ++a) {
                const int32_t r = sidx[wave][k][a * 16 + r16];
                voff[a] = rest && r >= 0 ? (uint32_t)r * (uint32_t)(c_red * 4) : kOOB;
            }
            wk = rest ? (uint32_t)k * (uint32_t)c_red * (uint32_t)n_out * 4u : kOOB;
            rest &= rest - 1;
            cl = 0;
        }
        const int c = cl + g * 4;
        // out of range past c_red (a multiple of 4); a select would become a
        // branch around the loads
        const uint32_t oob = c < c_red ? 0u : kOOB;
#pragma unroll
        for (int a = 0; a < FM; ++a) bload_f32<4>(rs, (voff[a] + (uint32_t)c * 4u) | oob, fa[d][a]);
        if constexpr (MODE == MODE_FWD) {
            const uint32_t o = wk + ((uint32_t)c * (uint32_t)n_out + (uint32_t)(col0 + FN * r16)) * 4u;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                float t[FN];
                bload_f32<FN>(rw, (o + (uint32_t)s * (uint32_t)n_out * 4u) | oob, t);
#pragma unroll
                for (int f = 0; f < FN; ++f) fb[d][f][s] = t[f];
            }
        } else {
            const uint32_t o = wk + ((uint32_t)(col0 + FN * r16) * (uint32_t)c_red + (uint32_t)c) * 4u;
#pragma unroll
            for (int f = 0; f < FN; ++f) bload_f32<4>(rw, (o + (uint32_t)(f * c_red) * 4u) | oob, fb[d][f]);
        }
        cl += 16;
    };
    f32x4 acc[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int f = 0; f < FN; ++f) acc[a][f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < D; ++d) load(d);
    for (int t = 0; t < steps; t += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            // past the last step the registers hold zeros
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int a = 0; a < FM; ++a)
#pragma unroll
                    for (int f = 0; f < FN; ++f) acc[a][f] = mfma_f32(fb[d][f][s], fa[d][a][s], acc[a][f]);
            load(d);
        }
    }
    if (wgk > 1) {  // uniform
        const int slot = (wm * wgn + wn) * (wgk - 1);  // at most 3 slots: wgm wgn (wgk - 1) <= 3
        if (set > 0) {
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int f = 0; f < FN; ++f) red[slot + set - 1][a * FN + f][lane] = acc[a][f];
        }
        __syncthreads();
        if (set > 0) return;
        for (int h = 0; h < wgk - 1; ++h)
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int f = 0; f < FN; ++f) acc[a][f] += red[slot + h][a * FN + f][lane];
    }
    // lane (g, r): columns FN (4 g + j) .. + FN - 1 of row r; whole groups of
    // FN lie inside n_out or outside it (f32_frags), rows and columns outside
    // are out-of-range stores (dropped)
    const rsrc_t ro = make_rsrc(out, (uint32_t)(n * n_out * 4));
    const rsrc_t rb = make_rsrc(bias, bias ? (uint32_t)n_out * 4u : 0u);
    float bv[4][FN];
#pragma unroll
    for (int j = 0; j < 4; ++j) bload_f32<FN>(rb, (uint32_t)(col0 + FN * (g * 4 + j)) * 4u, bv[j]);
#pragma unroll
    for (int a = 0; a < FM; ++a) {
        const int64_t i = row0 + a * 16 + r16;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int col = col0 + FN * (g * 4 + j);
            float v[FN];
#pragma unroll
            for (int f = 0; f < FN; ++f) v[f] = acc[a][f][j] + bv[j][f];
            bstore_f32<FN>(ro, i < n && col < n_out ? ((uint32_t)i * (uint32_t)n_out + (uint32_t)col) * 4u : kOOB, v);
        }
    }
}

// Column fragments per wave: the count whose tiles cover n columns (a multiple
// of 4) with the fewest to spare, the larger of equals; 3 only for whole
// groups of 3.
static int f32_frags(int n) {
    int best = 4, waste = (int)cdiv(n, 64) * 64 - n;
    for (int fn = 3; fn >= 2; --fn) {
        const int wst = (int)cdiv(n, 16 * fn) * 16 * fn - n;
        if (wst < waste && n % fn == 0) {
            best = fn;
            waste = wst;
        }
    }
    return best;
}

bool gg_f32_supported(int64_t n, int c_red, int n_out) {
    // 32-bit byte offsets; 16-byte rows on the reduction and the output side
    return c_red % 4 == 0 && n_out % 4 == 0 && n * std::max(c_red, n_out) * 4 < (int64_t)INT32_MAX &&
           9LL * c_red * n_out * 4 < (int64_t)INT32_MAX;
}

template <int MODE, int FM, int FN, int D>
static void launch_gg_f32(const float* src, const int32_t* nbr, const float* w, const float* bias, float* out,
                          int64_t n, int c_red, int n_out, int64_t tpb, int wgn, int wgk, bool sym,
                          hipStream_t s) {
    const int ncg = (int)cdiv(cdiv(n_out, 16 * FN), wgn);
    const int64_t tiles = cdiv(n, 16 * FM * (4 / (wgn * wgk))) * ncg;
    hipLaunchKernelGGL((k_gg_f32<MODE, FM, FN, D>), dim3((unsigned)tiles), dim3(256), 0, s, src, nbr, w, bias, out,
                       n, c_red, n_out, tpb, wgn, wgk, ncg, tiles, sym);
}

// Row fragments and the split of a workgroup's waves: the smallest of these
// estimates, in clocks (every constant fitted to the 15 shapes timed at nine
// sizes from 784 x 48 to 21952 x 128):
// * a step costs a CU 1.27 times its MFMA clocks (32 per MFMA, one wave per
//   SIMD and workgroup), or, where that is more, its four waves' loads: 64
//   clocks for a load whose neighboring lanes read different rows (gathered
//   rows; the weight of backward-input) and 29 for one that reads along rows
//   (the forward's weight);
// * a step takes at least 500 clocks (load latency over the ring), a
//   workgroup 6000 besides, and 1500 for the sum over offset sets.
// Few rows then take 16-row tiles with the offsets over four waves (941 rows
// of 128 channels: forward 11.8 us against 25.5 with one set and 42.8 with 32
// rows), backward-input 32 rows (21952 x 128: 76.5 us against 117 with 16).
struct F32Shape { int fm, wgn, wgk; };
static F32Shape pick_f32(int mode, int64_t n, int c_red, int n_out, int fn) {
    const int nct = (int)cdiv(n_out, 16 * fn), nc = (int)cdiv(c_red, 16);
    const int64_t cu = cu_count();
    F32Shape best{1, 1, 1};
    double best_cost = 0;
    for (int fm = 1; fm <= 4; fm <<= 1)
        for (int wgk = 1; wgk <= 4; wgk <<= 1) {
            const int room = 4 / wgk;
            const int wgn = nct >= room ? room : (nct >= 2 && room >= 2 ? 2 : 1);
            const int64_t wgs = cdiv(n, 16 * fm * (room / wgn)) * cdiv(nct, wgn);
            const double steps = (double)cdiv(9, wgk) * nc;
            const double step = std::max(1.27 * 128.0 * fm * fn, 4.0 * (64 * fm + (mode == MODE_FWD ? 29 : 64) * fn));
            const double held = (double)cdiv(wgs, cu * (fm == 4 ? 2 : 3));  // rounds of what the CUs hold
            const double cost = std::max((double)cdiv(wgs, cu) * steps * step, held * steps * 500) +
                                held * (6000 + (wgk > 1 ? 1500 : 0));
            if (best_cost == 0 || cost < best_cost) {
                best_cost = cost;
                best = F32Shape{fm, wgn, wgk};
            }
        }
    return best;
}

template <int MODE, int FN>
static void gg_f32_fn(const F32Shape& p, const float* src, const int32_t* nbr, const float* w, const float* bias,
                      float* out, int64_t n, int c_red, int n_out, int64_t tpb, bool sym, hipStream_t s) {
    switch (p.fm) {
        case 1: launch_gg_f32<MODE, 1, FN, 4>(src, nbr, w, bias, out, n, c_red, n_out, tpb, p.wgn, p.wgk, sym, s); break;
        case 2: launch_gg_f32<MODE, 2, FN, 3>(src, nbr, w, bias, out, n, c_red, n_out, tpb, p.wgn, p.wgk, sym, s); break;
        default: launch_gg_f32<MODE, 4, FN, 2>(src, nbr, w, bias, out, n, c_red, n_out, tpb, p.wgn, p.wgk, sym, s); break;
    }
}

void gg_f32(int mode, const void* src, const int32_t* nbr, const void* w, const void* bias, void* out, int64_t n,
            int c_red, int n_out, int64_t tpb, bool sym, hipStream_t s) {
    const int fn = f32_frags(n_out);
    const F32Shape p = pick_f32(mode, n, c_red, n_out, fn);
#define SVTAD_F32_CASE(M, FN)                                                                                   \
    if (mode == M && fn == FN) {                                                                                 \
        gg_f32_fn<M, FN>(p, (const float*)src, nbr, (const float*)w, (const float*)bias, (float*)out, n, c_red, n_out, \
                         tpb, sym, s);                                                                           \
        return;                                                                                                  \
    }
    SVTAD_F32_CASE(MODE_FWD, 2)
    SVTAD_F32_CASE(MODE_FWD, 3)
    SVTAD_F32_CASE(MODE_FWD, 4)
    SVTAD_F32_CASE(MODE_BWDIN, 2)
    SVTAD_F32_CASE(MODE_BWDIN, 3)
    SVTAD_F32_CASE(MODE_BWDIN, 4)
#undef SVTAD_F32_CASE
}

}  // namespace svtad
