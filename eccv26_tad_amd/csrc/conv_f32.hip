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

// Backward-weight partials: part[s][k][ci][co] = sum over the rows i of split s
// of x[src(i, k), ci] go[i, co], part_b[s][co] = sum of go[i, co]. A workgroup
// takes one offset of one split: it lists the rows whose neighbor exists (in
// row order) in LDS, kF32List rows of the split at a time, and its four waves
// are wgt tiles of 16 FM x 16 FN weights x (4 / wgt) row sets, set h taking
// every (4 / wgt)-th block of 16 listed rows; the sets' sums are added in
// order through LDS. An MFMA step takes 4 rows (lane group g row 4 g + t of
// the block), each lane FM channels of x and FN of go at once: channel FM r +
// a is row r of fragment a, so that one 16-byte load feeds four fragments.
// The last n_bias workgroups sum go for the bias, 64 columns each.
//
// Bound by the matrix cores, each wave holding 16 fragments against two loads
// per step: 21952 x 128 at 70 % keep 49 us, 57 with the reduction (320 + 21 us
// on the vector units), 784 x 48 6 + 3 us (35 + 9).
constexpr int kF32List = 1024;
template <int FM, int FN>
__global__ __launch_bounds__(256) void k_bw_f32(const float* __restrict__ go, const float* __restrict__ x,
                                                const int32_t* __restrict__ nbr, float* __restrict__ part,
                                                float* __restrict__ part_b, int64_t n, int c_in, int c_out,
                                                int64_t tpb, int64_t rows_per_split, int n_co_tiles, int n_tiles,
                                                int wgt, int64_t n_main) {
    __shared__ __align__(16) uint32_t list[2][kF32List];  // byte offsets of the rows in x and in go
    __shared__ int wcnt[4];
    __shared__ __align__(16) f32x4 red[3][FM * FN][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r16 = lane & 15;
    const rsrc_t rg = make_rsrc(go, (uint32_t)(n * c_out * 4));
    if ((int64_t)blockIdx.x >= n_main) {  // bias: 16 row lanes x 16 column groups of 4
        const int ncb = (c_out + 63) / 64;
        const int64_t b = blockIdx.x - n_main;
        const int64_t s = b / ncb;
        const int c = (int)(b - s * ncb) * 64 + r16 * 4, rl = tid >> 4;
        const int64_t r1 = min(n, (s + 1) * rows_per_split);
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        for (int64_t r0 = s * rows_per_split; r0 < r1; r0 += 128) {
            float v[8][4];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t r = r0 + u * 16 + rl;
                bload_f32<4>(rg, r < r1 && c < c_out ? ((uint32_t)r * (uint32_t)c_out + (uint32_t)c) * 4u : kOOB, v[u]);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) sum += f32x4{v[u][0], v[u][1], v[u][2], v[u][3]};
        }
        f32x4* const rr = &red[0][0][0];  // [row lane][column group]
        rr[rl * 16 + r16] = sum;
        __syncthreads();
        if (tid < 16 && c < c_out) {
            f32x4 t = rr[r16];
            for (int q = 1; q < 16; ++q) t += rr[q * 16 + r16];
            *(f32x4*)(part_b + s * c_out + c) = t;
        }
        return;
    }
    const int64_t lin = xcd_tile(blockIdx.x, n_main);
    const int groups = (n_tiles + wgt - 1) / wgt;  // workgroups per split and offset
    const int64_t s = lin / (9 * groups);
    const int rem = (int)(lin - s * 9 * groups);
    const int k = rem / groups;
    const int tile = (rem - k * groups) * wgt + wave % wgt;
    const int sets = 4 / wgt, set = wave / wgt;
    const bool live = tile < n_tiles;  // wave-uniform
    const int ci0 = (tile / n_co_tiles) * 16 * FM, co0 = (tile % n_co_tiles) * 16 * FN;
    const int64_t r_begin = s * rows_per_split;
    const int64_t r_end = min(n, r_begin + rows_per_split);
    const rsrc_t rx = make_rsrc(x, (uint32_t)(n * c_in * 4));
    // past the last tile: out of range (the waves still list rows and meet the barriers)
    const uint32_t xc = live ? (uint32_t)(ci0 + FM * r16) * 4u : kOOB, gc = live ? (uint32_t)(co0 + FN * r16) * 4u : kOOB;

    f32x4 acc[FM][FN];
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int64_t c0 = r_begin; c0 < r_end; c0 += kF32List) {
        const int rows = (int)min<int64_t>(kF32List, r_end - c0);
        int total = 0;
        for (int q0 = 0; q0 < rows; q0 += 256) {
            const int q = q0 + tid;
            const int64_t sr = q < rows ? src_row(nbr, c0 + q, k, n, tpb) : -1;
            const uint64_t bal = __ballot(sr >= 0);
            if (lane == 0) wcnt[wave] = __popcll(bal);
            __syncthreads();
            int at = total;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int c = wcnt[w];
                if (w < wave) at += c;
                total += c;
            }
            at += __popcll(bal & ((1ull << lane) - 1ull));
            if (sr >= 0) {
                list[0][at] = (uint32_t)sr * (uint32_t)(c_in * 4);
                list[1][at] = (uint32_t)(c0 + q) * (uint32_t)(c_out * 4);
            }
            __syncthreads();
        }
        const int blocks = (total + 15) / 16;
        if (tid < blocks * 16 - total) list[0][total + tid] = list[1][total + tid] = kOOB;  // at most 15, inside the list
        __syncthreads();
        // 4 steps of 4 rows per block; the next block's loads are in flight
        // (out of range past the end)
        u32x4 ox, og;
        auto offs = [&](int blk) {
            const int q = blk < blocks ? blk * 16 + g * 4 : 0;
            ox = *(const u32x4*)&list[0][q];
            og = *(const u32x4*)&list[1][q];
            const uint32_t oob = blk < blocks ? 0u : kOOB;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                ox[t] |= oob;
                og[t] |= oob;
            }
        };
        float fa[2][4][FM], fb[2][4][FN];
        auto load = [&](int buf) {
            // both kOOB (a row past the list, a wave past the tiles): their sum would wrap
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                bload_f32<FM>(rx, (ox[t] + (xc & ~kOOB)) | (xc & kOOB), fa[buf][t]);
                bload_f32<FN>(rg, (og[t] + (gc & ~kOOB)) | (gc & kOOB), fb[buf][t]);
            }
        };
        auto compute = [&](int buf) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int a = 0; a < FM; ++a)
#pragma unroll
                    for (int b = 0; b < FN; ++b) acc[a][b] = mfma_f32(fa[buf][t][a], fb[buf][t][b], acc[a][b]);
        };
        offs(set);
        load(0);
        offs(set + sets);
        // (without the scheduling barriers the compiler sinks a block's loads
        // below the MFMAs of the block before it, next to their uses)
        for (int blk = set; blk < blocks; blk += 2 * sets) {
            load(1);
            offs(blk + 2 * sets);
            __builtin_amdgcn_sched_barrier(0);
            compute(0);
            __builtin_amdgcn_sched_barrier(0);
            load(0);
            offs(blk + 3 * sets);
            __builtin_amdgcn_sched_barrier(0);
            compute(1);  // zeros past the end (under a condition, the loads would move under it too)
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();  // the next rows' list overwrites this one
    }
    if (sets > 1) {  // uniform
        const int slot = (wave % wgt) * (sets - 1);  // at most 3 slots
        if (set > 0) {
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) red[slot + set - 1][a * FN + b][lane] = acc[a][b];
        }
        __syncthreads();
        if (set > 0) return;
        for (int h = 0; h < sets - 1; ++h)
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) acc[a][b] += red[slot + h][a * FN + b][lane];
    }
    // lane (g, r): weights (FM (4 g + j) + a, FN r + b), FN of a row at once
    float* const dst = part + (s * 9 + k) * c_in * c_out;
    const rsrc_t ro = make_rsrc(dst, (uint32_t)c_in * (uint32_t)c_out * 4u);
    const int co = co0 + FN * r16;
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int ci = ci0 + FM * (g * 4 + j) + a;
            float v[FN];
#pragma unroll
            for (int b = 0; b < FN; ++b) v[b] = acc[a][b][j];
            bstore_f32<FN>(ro, live && ci < c_in && co < c_out ? ((uint32_t)ci * (uint32_t)c_out + (uint32_t)co) * 4u : kOOB, v);
        }
}

// gw[e] = sum_s part[s][e] (quads of 4 weights; then gb from part_b): four
// thread groups of a workgroup sum a quarter of the splits each, eight loads
// in flight, and the quarters are added in order through LDS.
__global__ __launch_bounds__(256) void k_bw_f32_reduce(const float* __restrict__ part, const float* __restrict__ part_b,
                                                       int splits, int64_t quads, int64_t quads_b,
                                                       float* __restrict__ gw, float* __restrict__ gb) {
    __shared__ f32x4 qsum[4][64];
    const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int64_t blocks_w = (quads + 63) / 64;
    const bool bias = (int64_t)blockIdx.x >= blocks_w;  // uniform
    const int64_t e = (bias ? blockIdx.x - blocks_w : blockIdx.x) * 64 + lane;
    const int64_t per = bias ? quads_b : quads;
    const f32x4* const p = (const f32x4*)(bias ? part_b : part);
    const int spt = (splits + 3) / 4;
    const int s0 = min(splits, g * spt), s1 = min(splits, s0 + spt);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (e < per) {
        for (int q = s0; q < s1; q += 8) {
            f32x4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = __builtin_nontemporal_load(p + (int64_t)min(q + u, s1 - 1) * per + e);
#pragma unroll
            for (int u = 0; u < 8; ++u) acc += q + u < s1 ? v[u] : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    qsum[g][lane] = acc;
    __syncthreads();
    if (g != 0 || e >= per) return;
    acc = qsum[0][lane] + qsum[1][lane];
    acc += qsum[2][lane];
    acc += qsum[3][lane];
    ((f32x4*)(bias ? gb : gw))[e] = acc;
}

bool bw_f32_supported(int64_t n, int c_in, int c_out) {
    return gg_f32_supported(n, c_in, c_out) && (int64_t)c_in * c_out * 4 < (int64_t)INT32_MAX;
}

// Weight tiles of a split and offset, and how many of them share a workgroup.
static void bw_f32_tiles(int c_in, int c_out, int* n_tiles, int* wgt) {
    *n_tiles = (int)(cdiv(c_in, 16 * f32_frags(c_in)) * cdiv(c_out, 16 * f32_frags(c_out)));
    *wgt = *n_tiles >= 4 ? 4 : *n_tiles >= 2 ? 2 : 1;
}

// Two workgroups for every CU (an offset's length follows its hit rate, which
// the host does not know, and two in one place even that out; 21952 x 128:
// partials and reduction 64.7 / 57.2 / 70.7 / 64.9 us with 1 / 2 / 3 / 4 for
// every CU), splits of at least 128 rows (shorter ones are mostly partial
// traffic: 3764 x 64 14.0 us with 28 splits, 16.7 with 56).
int64_t bw_f32_rows_per_split(int64_t n, int c_in, int c_out) {
    int n_tiles, wgt;
    bw_f32_tiles(c_in, c_out, &n_tiles, &wgt);
    const int64_t splits = std::max<int64_t>(1, 2 * cu_count() / (9 * cdiv(n_tiles, wgt)));
    return std::max<int64_t>(128, cdiv(cdiv(std::max<int64_t>(n, 1), splits), 16) * 16);
}

void bw_f32(const BwPlan& p, const void* go, const void* x, const int32_t* nbr, void* gw, void* gb, void* ws, int64_t n,
            int c_in, int c_out, int64_t tpb, hipStream_t s) {
    float* const part = (float*)ws;
    float* const part_b = gb ? part + (int64_t)p.splits * 9 * c_in * c_out : nullptr;
    int n_tiles, wgt;
    bw_f32_tiles(c_in, c_out, &n_tiles, &wgt);
    const int fm = f32_frags(c_in), fn = f32_frags(c_out);
    const int64_t n_main = (int64_t)p.splits * 9 * cdiv(n_tiles, wgt);
    const int64_t n_bias = gb ? (int64_t)p.splits * cdiv(c_out, 64) : 0;
#define SVTAD_F32_CASE(M, N)                                                                                     \
    if (fm == M && fn == N)                                                                                      \
        hipLaunchKernelGGL((k_bw_f32<M, N>), dim3((unsigned)(n_main + n_bias)), dim3(256), 0, s, (const float*)go, \
                           (const float*)x, nbr, part, part_b, n, c_in, c_out, tpb, p.rows_per_split,           \
                           (int)cdiv(c_out, 16 * N), n_tiles, wgt, n_main);
    SVTAD_F32_CASE(2, 2)
    SVTAD_F32_CASE(2, 3)
    SVTAD_F32_CASE(2, 4)
    SVTAD_F32_CASE(3, 2)
    SVTAD_F32_CASE(3, 3)
    SVTAD_F32_CASE(3, 4)
    SVTAD_F32_CASE(4, 2)
    SVTAD_F32_CASE(4, 3)
    SVTAD_F32_CASE(4, 4)
#undef SVTAD_F32_CASE
    if (!gw) return;  // partials only
    const int64_t quads = 9LL * c_in * c_out / 4, quads_b = gb ? c_out / 4 : 0;
    hipLaunchKernelGGL(k_bw_f32_reduce, dim3((unsigned)(cdiv(quads, 64) + cdiv(quads_b, 64))), dim3(256), 0, s, part,
                       part_b, p.splits, quads, quads_b, (float*)gw, (float*)gb);
}

}  // namespace svtad
