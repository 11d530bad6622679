// q4.hip - the q4 format on gfx950: the pack layout -> device layout permutation, dequantization, the RTN packer,
// int8 activation quantization (optionally fused with RMSNorm) and the dequant-in-register skinny GEMM.
//
// Reference arithmetic restated here (paths relative to the reference's engine/src):
//   dequant_row            kernels.cpp:1214-1228   level x (E4M3 x global), bit for bit
//   q4_block / e4m3_byte   yue2_q4.cpp:72-114       the packer's candidates and choice, bit for bit
//   quantize_activation    kernels.cpp:1254-1295   amax / 127 per 16 values, lrint, clamp +-127, bit for bit
//   rmsnorm                kernels.cpp:1520-1529   double sum of squares, 1 / sqrt(float(ss / n) + eps), x inv (1 + w)
//   matvec_rows_q_ref      kernels.cpp:1304-1322   the int8 path's products: exact weights x (q x act scale) on the
//                                                  matrix cores, fp32 sums (mfma_gemv.hpp)
#include "common.hpp"
#include "kernels.hpp"
#include "mfma_gemv.hpp"

namespace gv {

// ---------------------------------------------------------------- layout
namespace {
// pack code c -> affine c' (level 2c' - 15): 0..7 (levels 1..15) -> 8..15, 8..15 (levels -1..-15) -> 7..0
__device__ inline uint32_t affine_nibbles(uint32_t w) {
    // per nibble: c < 8 ? c + 8 : 15 - c, i.e. c ^ 8 or c ^ 15, on all 8 nibbles at once
    const uint32_t neg = ((w & 0x88888888u) >> 3) * 0xFu;   // 0xF where c >= 8
    return w ^ (neg | 0x88888888u);
}
}  // namespace

// one thread per (row, 8-value code word): the pack's word w of row r into the tile layout (mfma_gemv.hpp)
__global__ void q4_from_pack_kernel(const uint8_t *__restrict__ pack, int64_t rows, int64_t cols,
                                    uint8_t *__restrict__ codes, uint8_t *__restrict__ scales) {
    const int64_t nw = cols / 8;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= rows * nw) return;
    const int64_t r = i / nw, wi = i % nw;
    const size_t rb = static_cast<size_t>(cols / 16) * 9;
    const uint8_t *row = pack + static_cast<size_t>(r) * rb;
    const uint32_t w = *reinterpret_cast<const uint32_t *>(row + wi * 4);
    const int64_t T = r / kTileR, rr = r % kTileR, nsc = cols / kSuperK;
    const int64_t sc = wi / 16, j = (wi % 16) / 4, g = wi % 4;   // word 16 sc + 4 j + g
    const int64_t blk = T * nsc + sc;
    *reinterpret_cast<uint32_t *>(codes + blk * 1024 + (rr + 16 * g) * 16 + j * 4) = tile_word(affine_nibbles(w));
    if (g % 2 == 0)   // the block of (chunk j, k-groups g, g + 1): pack scale 8 sc + 2 j + g / 2
        scales[tq4_scale_off(T, (nsc + 3) / 4, sc, rr, g, j)] = row[cols / 2 + 8 * sc + 2 * j + g / 2];
}

int q4_from_pack(const uint8_t *pack_dev, int64_t rows, int64_t cols, float global, uint8_t *codes, uint8_t *scales,
                 Q4 &out, hipStream_t st) {
    GV_REQUIRE(rows > 0 && cols > 0 && cols % kSuperK == 0, "q4: cols must be a positive multiple of 128");
    const int64_t nsc = cols / kSuperK, nsq = (nsc + 3) / 4;
    if (rows % kTileR != 0) {   // the last tile's missing rows: zero codes and scales (their sums are discarded)
        const int64_t T = rows / kTileR;
        GV_CHECK_HIP(hipMemsetAsync(codes + T * nsc * 1024, 0, nsc * 1024, st));
        GV_CHECK_HIP(hipMemsetAsync(scales + T * nsq * 512, 0, nsq * 512, st));
    }
    if (nsc % 4 != 0)   // the last quad's unused super-chunks: zero scales (never read, kept defined)
        GV_CHECK_HIP(hipMemsetAsync(scales, 0, static_cast<size_t>(tiles_rows(rows)) * nsq * 512, st));
    const int64_t n = rows * (cols / 8);
    hipLaunchKernelGGL(q4_from_pack_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, pack_dev,
                       rows, cols, codes, scales);
    GV_CHECK_HIP(hipGetLastError());
    out.codes = codes;
    out.scales = scales;
    out.rows = rows;
    out.cols = cols;
    out.S = 0;
    out.steps = 0;
    out.global = global;
    return 0;
}

// ---------------------------------------------------------------- dequant (kernels.cpp:1214-1228)
__global__ void q4_dequant_kernel(Q4 w, float *__restrict__ out) {
    const int64_t nw = w.cols / 8;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= w.rows * nw) return;
    const int64_t r = i / nw, wi = i % nw;
    uint32_t word, sb;
    tq4_word(w, r, wi, word, sb);
    const float s = __fmul_rn(e4m3_to_f32(sb), w.global);   // E4M3 x global, then level x that
    float *o = out + r * w.cols + wi * 8;
    for (int b = 0; b < 8; ++b) {
        const int cp = static_cast<int>((word >> (4 * b)) & 15u);
        o[b] = __fmul_rn(static_cast<float>(2 * cp - 15), s);
    }
}

int q4_dequant(const Q4 &w, float *out, hipStream_t st) {
    const int64_t n = w.rows * (w.cols / 8);
    hipLaunchKernelGGL(q4_dequant_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, w, out);
    GV_CHECK_HIP(hipGetLastError());
    return 0;
}

// ---------------------------------------------------------------- the RTN packer (yue2_q4.cpp:72-114, :332-358)
__constant__ float c_e4m3_pos[127];   // E4M3's finite non-negative values, codes 0x00..0x7E

__device__ inline int e4m3_byte_dev(float x) {
    if (!(x > 0.0f)) return 0;
    if (x >= c_e4m3_pos[126]) return 126;
    int lo = 0, hi = 126;   // invariant: v[lo] <= x < v[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (c_e4m3_pos[mid] <= x) lo = mid;
        else hi = mid;
    }
    const float dl = __fsub_rn(x, c_e4m3_pos[lo]), dh = __fsub_rn(c_e4m3_pos[hi], x);
    if (dl < dh) return lo;
    if (dh < dl) return hi;
    return lo % 2 == 0 ? lo : hi;
}

__global__ void absmax_kernel(const float *__restrict__ w, int64_t n, unsigned int *__restrict__ out) {
    float m = 0.0f;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x)
        m = fmaxf(m, fabsf(w[i]));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) atomicMax(out, __float_as_uint(m));   // non-negative floats order as their bits
}

__global__ void q4_pack_kernel(const float *__restrict__ w, int64_t rows, int64_t cols,
                               const unsigned int *__restrict__ wmax_bits, uint8_t *__restrict__ out,
                               float *__restrict__ global_out) {
    const int64_t nb = cols / 16;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    // s2 = max|w| x 1.25 / (15 x 448)
    const float s2 = __fdiv_rn(__fmul_rn(__uint_as_float(*wmax_bits), 1.25f), 6720.0f);
    if (i == 0 && global_out) *global_out = s2;
    if (i >= rows * nb) return;
    const int64_t r = i / nb, blk = i % nb;
    const float *x = w + r * cols + blk * 16;
    float xv[16];
    float amax = 0.0f;
    for (int j = 0; j < 16; ++j) {
        xv[j] = x[j];
        amax = fmaxf(amax, fabsf(xv[j]));
    }
    int cand[10], nc = 0;
    const float ts[2] = {15.0f, 13.0f};
    for (int ti = 0; ti < 2; ++ti) {
        const int b0 = e4m3_byte_dev(__fdiv_rn(amax, __fmul_rn(ts[ti], s2)));
        for (int k = -2; k <= 2; ++k) cand[nc++] = min(max(b0 + k, 0), 0x7E);
    }
    float best = __builtin_inff();
    uint32_t best_codes[2] = {0, 0};
    int best_sb = 0;
    for (int c = 0; c < nc; ++c) {
        const float scale = __fmul_rn(c_e4m3_pos[cand[c]], s2), safe = scale == 0.0f ? 1.0f : scale;
        float err = 0.0f;
        uint32_t codes[2] = {0, 0};
        for (int j = 0; j < 16; ++j) {
            const float y = __fdiv_rn(xv[j], safe), a = fminf(fabsf(y), 15.0f);
            const int idx = min(max(static_cast<int>(rintf(__fmul_rn(__fsub_rn(a, 1.0f), 0.5f))), 0), 7);
            const bool neg = y < 0.0f;
            const float q = __fmul_rn(static_cast<float>(neg ? -(2 * idx + 1) : 2 * idx + 1), scale);
            const float d = __fsub_rn(q, xv[j]);
            err = __fadd_rn(err, __fmul_rn(d, d));
            codes[j / 8] |= static_cast<uint32_t>(idx + (neg ? 8 : 0)) << (4 * (j % 8));
        }
        if (err < best) {
            best = err;
            best_sb = cand[c];
            best_codes[0] = codes[0];
            best_codes[1] = codes[1];
        }
    }
    uint8_t *o = out + static_cast<size_t>(r) * (nb * 9);
    *reinterpret_cast<uint2 *>(o + blk * 8) = make_uint2(best_codes[0], best_codes[1]);
    o[nb * 8 + blk] = static_cast<uint8_t>(best_sb);
}

int q4_init_constants() {
    static bool done = false;
    if (done) return 0;
    float v[127];
    for (int b = 0; b < 127; ++b) {
        const int ex = (b >> 3) & 15, man = b & 7;
        v[b] = ex == 0 ? static_cast<float>(man) / 8.0f / 64.0f : (1.0f + static_cast<float>(man) / 8.0f) *
                                                                        static_cast<float>(1 << ex) / 128.0f;
    }
    GV_CHECK_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_e4m3_pos), v, sizeof v));
    done = true;
    return 0;
}

int q4_pack(const float *w, int64_t rows, int64_t cols, unsigned int *scratch_u32, uint8_t *out, float *global_out,
            hipStream_t st) {
    GV_REQUIRE(cols % 16 == 0 && rows > 0, "q4_pack: cols must be a multiple of 16");
    if (q4_init_constants() != 0) return -1;
    GV_CHECK_HIP(hipMemsetAsync(scratch_u32, 0, 4, st));
    const int64_t n = rows * cols;
    hipLaunchKernelGGL(absmax_kernel, dim3(static_cast<unsigned>(std::min<int64_t>(4096, (n + 255) / 256))), dim3(256),
                       0, st, w, n, scratch_u32);
    const int64_t nb = rows * (cols / 16);
    hipLaunchKernelGGL(q4_pack_kernel, dim3(static_cast<unsigned>((nb + 255) / 256)), dim3(256), 0, st, w, rows, cols,
                       scratch_u32, out, global_out);
    GV_CHECK_HIP(hipGetLastError());
    return 0;
}

// Rows of activations into the products' operands (mfma_gemv.hpp: act16 layout, the int8 path's values), optionally
// RMSNorm first and the normalized fp32 rows out; a workgroup per row.
__global__ __launch_bounds__(256) void quantize_act_kernel(const float *__restrict__ x, int64_t ldx, int cols,
                                                           const float *__restrict__ norm_w, float eps,
                                                           _Float16 *__restrict__ act, int64_t act_stride,
                                                           float *__restrict__ h_out, int64_t ldh) {
    __shared__ double red[16];
    const int t = blockIdx.x;
    norm_quant_row(x + t * ldx, cols, norm_w, eps, act + t * act_stride, h_out ? h_out + t * ldh : nullptr, red);
}

int quantize_act(const float *x, int64_t ldx, int M, int cols, const float *norm_w, float eps, _Float16 *act,
                 int64_t act_stride, float *h_out, int64_t ldh, hipStream_t st) {
    GV_REQUIRE(cols % 16 == 0 && cols <= 8192 && M > 0, "quantize_act: cols must be a multiple of 16, at most 8192");
    GV_REQUIRE(ldx % 4 == 0 && (!h_out || ldh % 4 == 0), "quantize_act: row strides must keep 16-byte alignment");
    hipLaunchKernelGGL(quantize_act_kernel, dim3(M), dim3(256), 0, st, x, ldx, cols, norm_w, eps, act, act_stride,
                       h_out, ldh);
    GV_CHECK_HIP(hipGetLastError());
    return 0;
}

// ---------------------------------------------------------------- the skinny GEMM (mfma_gemv.hpp)
// WMAX: the most waves a launch of the instance takes (8: a budget of 256 VGPRs a lane)
// PACK: at most 8 rows, their hi and lo halves in the MFMA's two column halves (mfma_tiles)
// NT > 0 (a launch of at most NT tiles a workgroup): the tile loop straight-line, every tile's loads issued before
// the first tile is computed (NT <= the ring's depth); 0: the ring of three over any number of tiles
// RSPLIT: the M rows in gridDim.y groups of ceil(M / gridDim.y), group blockIdx.y's rows by this workgroup (each row's
// sums as in a launch of its group alone)
template <int KW, int NTT, int WMAX, bool PACK, int NT = 0, bool RSPLIT = false>
__global__ __launch_bounds__(64 * WMAX) void gemv_q4_kernel(Q4 w, const _Float16 *__restrict__ act,
                                                            int64_t act_stride, int M, int sc0, int tiles_per_wg,
                                                            GemvOut out) {
    extern __shared__ f4 part_lds[];
    __shared__ uint2 tab[256];
    int r0 = 0;   // the first row of the workgroup's group (its outputs' row index offset; out itself is left as
                  // passed: a copy of it would go to scratch, its segment arrays being indexed at run time)
    if constexpr (RSPLIT) {
        const int mh = (M + static_cast<int>(gridDim.y) - 1) / static_cast<int>(gridDim.y);
        r0 = static_cast<int>(blockIdx.y) * mh;
        if (r0 >= M) return;   // (uniform)
        act += static_cast<int64_t>(r0) * act_stride;
        M = min(mh, M - r0);
    }
    const int tc = out.trace_cls;
    if (tc >= 0) trace(tc, 0);
    const int64_t ntiles = tiles_rows(w.rows);
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * tiles_per_wg;
    const int64_t t1 = t0 + tiles_per_wg < ntiles ? t0 + tiles_per_wg : ntiles;
    if (t0 >= ntiles) return;
    const int nt = static_cast<int>(t1 - t0);
    // The outputs are written as mfma_tiles' split-K epilogue writes them (output o = (tile, column, 4 rows) by
    // thread o mod blockDim), here so that an accumulating product's earlier values for the thread's first output
    // are loaded with the weights (in the hook) rather than one round trip a row at the end.
    const int o0 = threadIdx.x;
    auto item = [&](int o, int64_t &row0, int &j) {
        const int i = o / (NTT * 64), tt = (o / 64) % NTT, ll = o % 64;
        row0 = (t0 + i) * kTileR + 4 * (ll / 16);
        j = tt * 16 + ll % 16;
    };
    float old[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto prefetch = [&] {
        if (!out.accumulate) return;   // uniform
        int64_t row0;
        int j;
        item(min(o0, nt * NTT * 64 - 1), row0, j);
        const float *p = out.y + (r0 + min(j, M - 1)) * out.ldy;
#pragma unroll
        for (int r = 0; r < 4; ++r) old[r] = p[min(row0 + r, w.rows - 1)];   // (clamped: always a valid address)
    };
    mfma_tiles<KW, NTT, kKeepParts, NT, (NT == 0 ? 3 : NT == 1 ? 2 : NT), PACK>(
        w.codes, w.scales, w.rows, static_cast<int>(w.cols / kSuperK), sc0, nt, M,
        [&](int j) { return act + j * act_stride; }, [](int64_t, int, float) {}, part_lds, tab, TileRun{t0}, prefetch,
        [&] { if (tc >= 0) trace(tc, 5); });
    if (tc >= 0) trace(tc, 6);
    const int W = blockDim.x / 64;
    for (int o = o0; o < nt * NTT * 64; o += blockDim.x) {   // the waves' partial sums added in wave order
        const int i = o / (NTT * 64), tt = (o / 64) % NTT, ll = o % 64;
        f4 sum = part_lds[((i * W + 0) * NTT + tt) * 64 + ll];
        for (int w2 = 1; w2 < W; ++w2) sum += part_lds[((i * W + w2) * NTT + tt) * 64 + ll];
        int64_t row0;
        int j;
        item(o, row0, j);
        if (j >= M) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = row0 + r;
            if (row >= w.rows) break;
            if (o == o0 && out.accumulate) out.y[(r0 + j) * out.ldy + row] = old[r] + out.scaled(row, sum[r]);
            else out.put(row, r0 + j, sum[r]);
        }
    }
    if (tc >= 0) trace(tc, 3);
}

// The skinny product at 17..32 rows over two K ranges in one launch (each range's activations fill the waves'
// registers, as in two gemv_q4_kernel launches, the second accumulating): the workgroup runs the first range's tiles,
// keeps their partial sums in LDS, runs the second's, then writes (y + s0 x global) + s1 x global (accumulate), or
// s0 x global + s1 x global: the two launches' sums in their order.
template <int KW, int WMAX>
__global__ __launch_bounds__(64 * WMAX) void gemv_q4_2pass_kernel(Q4 w, const _Float16 *__restrict__ act,
                                                                  int64_t act_stride, int M, int sc_step,
                                                                  int tiles_per_wg, GemvOut out) {
    extern __shared__ f4 part_lds[];
    __shared__ uint2 tab[256];
    const int64_t ntiles = tiles_rows(w.rows);
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * tiles_per_wg;
    if (t0 >= ntiles) return;
    const int nt = static_cast<int>(std::min<int64_t>(tiles_per_wg, ntiles - t0));
    const int W = blockDim.x / 64, o0 = threadIdx.x;
    f4 *part1 = part_lds + static_cast<size_t>(tiles_per_wg) * W * 2 * 64;
    auto item = [&](int o, int64_t &row0, int &j) {
        const int i = o / 128, tt = (o / 64) % 2, ll = o % 64;
        row0 = (t0 + i) * kTileR + 4 * (ll / 16);
        j = tt * 16 + ll % 16;
    };
    float old[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto prefetch = [&] {
        if (!out.accumulate) return;   // uniform
        int64_t row0;
        int j;
        item(min(o0, nt * 128 - 1), row0, j);
        const float *p = out.y + min(j, M - 1) * out.ldy;
#pragma unroll
        for (int r = 0; r < 4; ++r) old[r] = p[min(row0 + r, w.rows - 1)];   // (clamped: always a valid address)
    };
    const int nsc = static_cast<int>(w.cols / kSuperK);
    mfma_tiles<KW, 2, kKeepParts, 0, 3, false>(w.codes, w.scales, w.rows, nsc, 0, nt, M,
                                                [&](int j) { return act + j * act_stride; },
                                                [](int64_t, int, float) {}, part_lds, tab, TileRun{t0}, prefetch);
    mfma_tiles<KW, 2, kKeepParts, 0, 3, false>(w.codes, w.scales, w.rows, nsc, sc_step, nt, M,
                                                [&](int j) { return act + j * act_stride; },
                                                [](int64_t, int, float) {}, part1, tab, TileRun{t0});
    for (int o = o0; o < nt * 128; o += blockDim.x) {   // each range's waves' partial sums in wave order
        const int i = o / 128, tt = (o / 64) % 2, ll = o % 64;
        f4 s0 = part_lds[((i * W + 0) * 2 + tt) * 64 + ll], s1 = part1[((i * W + 0) * 2 + tt) * 64 + ll];
        for (int w2 = 1; w2 < W; ++w2) {
            s0 += part_lds[((i * W + w2) * 2 + tt) * 64 + ll];
            s1 += part1[((i * W + w2) * 2 + tt) * 64 + ll];
        }
        int64_t row0;
        int j;
        item(o, row0, j);
        if (j >= M) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t row = row0 + r;
            if (row >= w.rows) break;
            float *p = out.y + j * out.ldy + row;
            const float first = out.scaled(row, s0[r]);
            const float v = out.accumulate ? (o == o0 ? old[r] : *p) + first : first;
            *p = v + out.scaled(row, s1[r]);
        }
    }
}

// The skinny product over many row tiles a workgroup (a vocabulary head): a round of the chip's workgroups takes every
// tile, a stride of the grid apart (all of them read adjacent tiles at a time, at most one tile more than the others),
// and the waves' sums are put every few tiles (mfma_tiles FLUSH) with the loads of the next ones in flight: the same
// sums in the same order as gemv_q4_kernel, the activations loaded once a CU and the partial sums' LDS small. The waves
// wait for one another at a flush only: two halves of the partial sums in turn, one barrier each; a lane's four rows go
// out in one store. NTT 2 (17..32 rows): a K range's activations take half the registers; PACK 2: at most 24 rows, the
// second column tile's hi and lo halves in one MFMA.
// The 151,936 x 2048 head with its norm's launch, 17 rows: 62.9 us with four tiles a flush in one buffer over two
// rounds of workgroups; one store a lane 4 rows, packed, two buffers 56.2; one round of workgroups 49.2; two tiles a
// flush 47.7 (one: 52.5); strided tiles 46.6 (its weights and logits at a copy's rate: 36). Sixteen waves of half the
// K range each: 58. Up to 16 rows against gemv_q4_kernel's contiguous tiles, every tile's sums kept to the end: 1 row
// 37.9 -> 33.5 us, 5 rows 38.8 -> 35.4, 16 rows 46.7 -> 44.2, 248,320 x 2048 at 5 rows 64.2 -> 54.7, 32,000 x 2048 at 8
// rows 14.3 -> 13.4; four tiles a flush (eight: the same; two: 2 us more at 16 rows), the ring of three (four: 16 rows
// spill).
constexpr int gemv_flush(int ntt) { return ntt == 1 ? 4 : 2; }   // tiles a flush
template <int KW, int WMAX, int NTT, int PACK>
__global__ __launch_bounds__(64 * WMAX) void gemv_q4_flush_kernel(Q4 w, const _Float16 *__restrict__ act,
                                                                  int64_t act_stride, int M, int sc0, GemvOut out) {
    extern __shared__ f4 part_lds[];
    __shared__ uint2 tab[256];
    const int ntiles = static_cast<int>(tiles_rows(w.rows));
    const int wg = static_cast<int>(blockIdx.x), nwg = static_cast<int>(gridDim.x);   // (at most ntiles workgroups)
    const int nt = (ntiles - wg + nwg - 1) / nwg;
    // a lane's four rows of a column in one store: one segment, whole row tiles, 16-byte rows of y
    const bool whole = !out.accumulate && out.nseg == 1 && w.rows % kTileR == 0 &&
                       (reinterpret_cast<uintptr_t>(out.y) | static_cast<uintptr_t>(out.ldy) * 4) % 16 == 0;
    auto tile_of = [&](int i) -> int64_t { return wg + static_cast<int64_t>(i) * nwg; };
    mfma_tiles<KW, NTT, kSplitK, 0, NTT == 1 ? 3 : 4, PACK, gemv_flush(NTT), 2>(
        w.codes, w.scales, w.rows, static_cast<int>(w.cols / kSuperK), sc0, nt, M,
        [&](int j) { return act + j * act_stride; }, [](int64_t, int, float) {}, part_lds, tab, tile_of, NoHook{},
        NoHook{}, flush_with([&](int i0, int i1, const f4 *part, int W) {   // a tile and column tile a lane: wave order
            for (int o = threadIdx.x; o < (i1 - i0) * NTT * 64; o += blockDim.x) {
                const int i = o / (NTT * 64), tt = (o / 64) % NTT, ll = o % 64, j = tt * 16 + ll % 16;
                if (j >= M) continue;
                f4 sum = part[(i * W * NTT + tt) * 64 + ll];
                for (int w2 = 1; w2 < W; ++w2) sum += part[((i * W + w2) * NTT + tt) * 64 + ll];
                const int64_t row0 = tile_of(i0 + i) * kTileR + 4 * (ll / 16);
                if (whole) {
                    *reinterpret_cast<f4 *>(out.y + j * out.ldy + row0) = sum * out.seg_global[0];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (row0 + r < w.rows) out.put(row0 + r, j, sum[r]);
                }
            }
        }));
}

GV_ACT_MODE_SETTER(act_mode_set_q4)
// ---------------------------------------------------------------- the dense SwiGLU FFN (C1) in three launches
// x fp16 rows to the products' operands (the int8 path's quantization of the fp32 values, which fp16 converts to
// exactly): a workgroup a row
__global__ __launch_bounds__(256) void quantize_f16_kernel(const uint16_t *__restrict__ x, int cols,
                                                           _Float16 *__restrict__ act, int64_t act_stride) {
    __shared__ double red[16];
    const int t = blockIdx.x, ng = cols / 8;
    float v[4][8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int g = threadIdx.x + q * blockDim.x;
        uint4 w = make_uint4(0, 0, 0, 0);
        if (g < ng) w = *reinterpret_cast<const uint4 *>(x + static_cast<int64_t>(t) * cols + g * 8);
        const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[q][2 * i] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(u[i] & 0xFFFFu)));
            v[q][2 * i + 1] = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(u[i] >> 16)));
        }
    }
    norm_quant_regs(v, cols, nullptr, 0.0f, act + static_cast<int64_t>(t) * act_stride, nullptr, red);
}

// The gate and up products with the SwiGLU and its quantization in one launch, up to 32 rows: a workgroup per 16-row
// tile pair (gate tile p, up tile p), its waves splitting K; the 16 values m = silu(g) x u of a row and tile are one
// quantization block, so the down product's operands are the workgroup's own (swiglu_pair_out). Both tiles' loads are
// in flight at once (a matrix pair as one call's two tiles): bound by the latency of that one round of loads, which
// eight waves (half the K range each, three waves a SIMD at 384 workgroups) wait for together.
// 2048 -> 6144, 5 rows: 10.9 us with the two products one after the other on four waves, 8.4 so.
// (NP pairs a workgroup: at 17..32 rows its operands are several times its weights)
template <int KW, int NTT, bool PACK, int NP>
__global__ __launch_bounds__(512) void ffn_up_kernel(Q4 gate, Q4 up, const _Float16 *__restrict__ act,
                                                     int64_t act_stride, int M, _Float16 *__restrict__ act_m,
                                                     int64_t act_m_stride) {
    extern __shared__ f4 part_lds[];
    __shared__ uint2 tab[256];
    const int W = blockDim.x / 64, npair = static_cast<int>(gate.rows / kTileR);
    const int p0 = static_cast<int>(blockIdx.x) * NP, np = min(NP, npair - p0);
    mfma_tiles_of<KW, NTT, kKeepParts, 2 * NP, 2 * NP < 3 ? 2 * NP : 3, PACK>(
        MatrixPair{gate.codes, gate.scales, up.codes, up.scales}, gate.rows, static_cast<int>(gate.cols / kSuperK), 0,
        2 * np, M, [&](int j) { return act + static_cast<int64_t>(j) * act_stride; }, [](int64_t, int, float) {},
        part_lds, tab, [&](int i) -> int64_t { return p0 + (i >> 1); });
    for (int o = threadIdx.x; o < np * NTT * 64; o += blockDim.x) {   // a wave a pair and 16-column tile of rows
        const int q = o / (NTT * 64), tt = (o / 64) % NTT, lane = o % 64, j = tt * 16 + lane % 16;
        const f4 *gp = part_lds + (2 * q * W * NTT + tt) * 64 + lane, *up_ = gp + W * NTT * 64;
        f4 gs = gp[0], us = up_[0];
        for (int w2 = 1; w2 < W; ++w2) {   // the waves' sums in wave order
            gs += gp[w2 * NTT * 64];
            us += up_[w2 * NTT * 64];
        }
        swiglu_pair_out(gs, us, gate.global, up.global, p0 + q, j < M, act_m + j * act_m_stride);
    }
}

int quantize_f16(const uint16_t *x, int M, int cols, _Float16 *act, int64_t act_stride, hipStream_t st) {
    GV_REQUIRE(cols % 16 == 0 && cols <= 8192 && M > 0, "quantize_f16: cols must be a multiple of 16, at most 8192");
    hipLaunchKernelGGL(quantize_f16_kernel, dim3(M), dim3(256), 0, st, x, cols, act, act_stride);
    GV_CHECK_HIP(hipGetLastError());
    return 0;
}

// K split over eight waves where it can be (half the decode chain of four), whole 16-row tiles
static bool ffn_up_split(const Q4 &gate, int M, int &waves, int &kw) {
    const int ntt = M <= 16 ? 1 : 2;
    if (gate.rows % kTileR != 0 || !mfma_split(gate.cols, ntt, waves, kw)) return false;
    if (waves <= 4 && kw == 16) kw = 8, waves *= 2;
    return M <= 8 || kw <= 8;   // (unpacked: the hi and lo operands of 16 chunks do not fit a wave's registers twice)
}
bool ffn_up_fits(const Q4 &gate, const Q4 &up, int M) {
    int waves = 0, kw = 0;
    return M >= 1 && M <= kMaxRows && gate.rows == up.rows && gate.cols == up.cols && ffn_up_split(gate, M, waves, kw);
}

template <int KW, int NTT, bool PACK, int NP>
static int launch_ffn_up(const Q4 &gate, const Q4 &up, const _Float16 *act, int64_t act_stride, int M, int waves,
                         _Float16 *act_m, int64_t act_m_stride, hipStream_t st) {
    const int64_t npair = gate.rows / kTileR;
    const size_t lds = static_cast<size_t>(2 * NP * waves * NTT) * 1024;   // at most 64 KB
    hipLaunchKernelGGL((ffn_up_kernel<KW, NTT, PACK, NP>), dim3(static_cast<unsigned>((npair + NP - 1) / NP)),
                       dim3(static_cast<unsigned>(64 * waves)), lds, st, gate, up, act, act_stride, M, act_m,
                       act_m_stride);
    GV_CHECK_HIP(hipGetLastError());
    return 0;
}

int ffn_up(const Q4 &gate, const Q4 &up, const _Float16 *act, int64_t act_stride, int M, _Float16 *act_m,
           int64_t act_m_stride, hipStream_t st) {
    int waves = 0, kw = 0;
    GV_REQUIRE(ffn_up_fits(gate, up, M) && ffn_up_split(gate, M, waves, kw),
               "ffn_up: 1 <= M <= 32, gate and up alike, whole row tiles, K split over at most 8 waves");
#define GV_FFN_UP(KW, NTT, PACK, NP) \
    return launch_ffn_up<KW, NTT, PACK, NP>(gate, up, act, act_stride, M, waves, act_m, act_m_stride, st)
    if (M <= 8) {
        if (kw == 16) GV_FFN_UP(16, 1, true, 1);
        if (kw == 8) GV_FFN_UP(8, 1, true, 1);
        GV_FFN_UP(4, 1, true, 1);
    }
    if (M <= 16) {
        if (kw == 8) GV_FFN_UP(8, 1, false, 1);
        GV_FFN_UP(4, 1, false, 1);
    }
    if (kw == 8) GV_FFN_UP(8, 2, false, 2);
    GV_FFN_UP(4, 2, false, 2);
#undef GV_FFN_UP
}

int trace_set_q4(uint64_t *p) {
    GV_CHECK_HIP(hipMemcpyToSymbol(HIP_SYMBOL(g_trace), &p, sizeof p));
    return 0;
}

int mfma_split(int64_t K, int ntt, int &waves, int &kw) {
    const int chunks = static_cast<int>(K / 32);
    kw = ntt == 1 ? 16 : 8;
    while (kw > 4 && (chunks % kw || chunks / kw < 2)) kw /= 2;
    waves = chunks / kw;
    return K % kSuperK == 0 && waves >= 1 && waves <= 8;
}

// tiles a workgroup: about as many workgroups as the chip holds at once (2 waves a SIMD at these kernels' register
// use: 512 / waves workgroups), the waves' partial sums within 76 KB of LDS (two workgroups a CU)
int64_t tiles_per_wg(int64_t ntiles, int waves, int ntt) {
    const int64_t resident = 256 * std::max(1, 8 / waves);
    const int64_t cap = waves > 1 ? std::max(1, 76 / (waves * ntt)) : 64;
    return std::min<int64_t>(cap, std::max<int64_t>(1, (ntiles + resident - 1) / resident));
}

template <int KW, int NTT, int WMAX, bool PACK>
static int launch_gemv(const Q4 &w, const _Float16 *act, int64_t act_stride, int M, int sc0, int waves,
                       const GemvOut &out, hipStream_t st) {
    const int64_t ntiles = tiles_rows(w.rows);
    const int64_t per = tiles_per_wg(ntiles, waves, NTT);
    // a matrix whose tiles outnumber 4 a workgroup of the chip's resident ones (a vocabulary head): the flushed form, the
    // resident workgroups over all the tiles (up to 16 rows, a range that adds to earlier sums keeps gemv_q4_kernel, which
    // has those loaded ahead, and so does a traced launch)
    const int64_t resident = 256 * std::max(1, 8 / waves);
    const bool flushed = NTT == 1 ? ntiles > 4 * resident && !out.accumulate && out.trace_cls < 0 : ntiles > per * resident;
    if (flushed) {
        const dim3 grid(static_cast<unsigned>(std::min(ntiles, resident))), block(static_cast<unsigned>(64 * waves));
        const size_t lds = static_cast<size_t>(2 * gemv_flush(NTT)) * waves * NTT * 1024;   // at most 64 KB
        constexpr int P = PACK ? 1 : NTT == 1 ? 0 : 2;
        if (NTT == 1 || M <= 24)
            hipLaunchKernelGGL((gemv_q4_flush_kernel<KW, WMAX, NTT, P>), grid, block, lds, st, w, act, act_stride, M, sc0,
                               out);
        else
            hipLaunchKernelGGL((gemv_q4_flush_kernel<KW, WMAX, NTT, NTT == 1 ? P : 0>), grid, block, lds, st, w, act,
                               act_stride, M, sc0, out);
        return 0;
    }
    const int64_t wg = (ntiles + per - 1) / per;
    const size_t lds = static_cast<size_t>(per) * waves * NTT * 1024;   // the waves' partial sums
    if (per <= 3 && per > 1) {   // a few tiles a workgroup (q|k|v): all of them in flight at once
        static int granted3 = 0;
        if (lds_grant(reinterpret_cast<const void *>(&gemv_q4_kernel<KW, NTT, WMAX, PACK, 3>), 76 * 1024, granted3) != 0)
            return -1;
        hipLaunchKernelGGL((gemv_q4_kernel<KW, NTT, WMAX, PACK, 3>), dim3(static_cast<unsigned>(wg)), dim3(64 * waves),
                           static_cast<size_t>(3) * waves * NTT * 1024, st, w, act, act_stride, M, sc0,
                           static_cast<int>(per), out);
        return 0;
    }
    static int granted = 0;
    if (lds_grant(reinterpret_cast<const void *>(&gemv_q4_kernel<KW, NTT, WMAX, PACK>), 76 * 1024, granted) != 0)
        return -1;
    hipLaunchKernelGGL((gemv_q4_kernel<KW, NTT, WMAX, PACK>), dim3(static_cast<unsigned>(wg)), dim3(64 * waves), lds,
                       st, w, act, act_stride, M, sc0, static_cast<int>(per), out);
    return 0;
}

// one launch over super-chunks [sc0, sc0 + n) of every row
static int gemv_range(const Q4 &w, const _Float16 *act, int64_t act_stride, int M, int ntt, int sc0, int n,
                      const GemvOut &out, hipStream_t st) {
    int waves, kw;
    if (!mfma_split(static_cast<int64_t>(n) * kSuperK, ntt, waves, kw)) {
        set_error("gemv_q4: no split of this K range");
        return -1;
    }
    // a short launch (a few tiles a workgroup): eight waves, each half the decode chain (measured: the 9216-row
    // q|k|v product 9.6 -> 8.3 us; the 151,936-row lm_head keeps four, 36.8 against 39.9 us)
    if (ntt == 1 && waves <= 4 && kw == 16 && tiles_rows(w.rows) < 2048) kw = 8, waves *= 2;
    if (ntt == 1 && M <= 8) {
        if (kw == 16) return launch_gemv<16, 1, 8, true>(w, act, act_stride, M, sc0, waves, out, st);
        if (kw == 8) return launch_gemv<8, 1, 8, true>(w, act, act_stride, M, sc0, waves, out, st);
        return launch_gemv<4, 1, 8, true>(w, act, act_stride, M, sc0, waves, out, st);
    }
    if (ntt == 1) {
        if (kw == 16) return launch_gemv<16, 1, 8, false>(w, act, act_stride, M, sc0, waves, out, st);
        if (kw == 8) return launch_gemv<8, 1, 8, false>(w, act, act_stride, M, sc0, waves, out, st);
        return launch_gemv<4, 1, 8, false>(w, act, act_stride, M, sc0, waves, out, st);
    }
    if (kw == 8) return launch_gemv<8, 2, 8, false>(w, act, act_stride, M, sc0, waves, out, st);
    return launch_gemv<4, 2, 8, false>(w, act, act_stride, M, sc0, waves, out, st);
}

int gemv_q4(const Q4 &w, const _Float16 *act, int64_t act_stride, int M, const GemvOut &out, hipStream_t st) {
    GV_REQUIRE(M >= 1 && M <= kMaxRows, "gemv_q4: 1 <= M <= 32 rows");
    GV_REQUIRE(w.cols % kSuperK == 0 && w.cols <= kMaxActCols, "gemv_q4: cols must be a multiple of 128, at most 16384");
    const int ntt = M <= 16 ? 1 : 2;
    const int nsc = static_cast<int>(w.cols / kSuperK);
    const int64_t ntiles = tiles_rows(w.rows);
    if (ntt == 2 && ntiles <= (nsc > 16 ? 256 : 128)) {
        // 17..32 rows over few tiles (a tree's output projection, a dense MLP's down product): the rows in two groups of
        // at most 16, both in one launch: twice the workgroups, each loading half the rows' operands (the sums of an
        // M <= 16 launch). K in ranges of at most 4096; with the rows in one group the ranges are half that. Few: both
        // groups' workgroups fit a round of the chip, or K needs the larger ranges. 2048 x 4096, 17 rows: 16.0 us in
        // one group, 10.6 so; 2048 x 6144 in two ranges instead of three, 17 and 32 rows: the whole MLP 41 -> 30 and
        // 51 -> 37 us; 4096 x 2048 at 17 rows the other way, 9.1 us against 10.6.
        // (A matrix of more tiles than CUs streams many a workgroup and loses more by loading each twice: the 9216-row
        // q|k|v product took the 40-layer step from 5.58 to 5.93 ms.)
        GemvOut o = out;
        for (int sc0 = 0; sc0 < nsc;) {
            int n = std::min(nsc - sc0, 32), waves, kw;
            while (n > 1 && !mfma_split(static_cast<int64_t>(n) * kSuperK, 1, waves, kw)) --n;
            GV_REQUIRE(sc0 % 4 == 0 && mfma_split(static_cast<int64_t>(n) * kSuperK, 1, waves, kw),
                       "gemv_q4: a K range must start on a quad of super-chunks");
            if (kw == 16 && waves <= 4) kw = 8, waves *= 2;   // (half the decode chain, as gemv_range)
            const dim3 grid(static_cast<unsigned>(ntiles), 2), block(static_cast<unsigned>(64 * waves));
            const size_t lds = static_cast<size_t>(waves) * 1024;
            if (kw == 16)
                hipLaunchKernelGGL((gemv_q4_kernel<16, 1, 8, false, 0, true>), grid, block, lds, st, w, act, act_stride, M, sc0, 1, o);
            else if (kw == 8)
                hipLaunchKernelGGL((gemv_q4_kernel<8, 1, 8, false, 0, true>), grid, block, lds, st, w, act, act_stride, M, sc0, 1, o);
            else
                hipLaunchKernelGGL((gemv_q4_kernel<4, 1, 8, false, 0, true>), grid, block, lds, st, w, act, act_stride, M, sc0, 1, o);
            GV_CHECK_HIP(hipGetLastError());
            o.accumulate = 1;
            sc0 += n;
        }
        return 0;
    }
    if (M <= 8 && nsc > 32 && nsc <= 48 && nsc % 4 == 0 && ntiles <= 256) {
        // K of 4096 .. 6144 over at most a tile a CU (a dense MLP's down product): one launch of up to twelve waves,
        // 512 values each, instead of two K ranges one after the other - with a tile a workgroup a launch is one
        // round of loads, so the second range's launch costs about as much as the first's. 2048 rows, 5 rows of x: K =
        // 4608 6.7 us (4352, in ranges: 7.2 + 3.7), 6144 7.8 us (5888, in ranges: 7.1 + 4.7). A wave takes 512 values, so
        // K in multiples of it; 9..16 rows (unpacked: twice the operand registers, which twelve waves do not have; 9 rows
        // at 6144: 9.4 + 6.1), more tiles (each CU streaming many) or wider K: the ranges below.
        const int waves = nsc / 4;
        hipLaunchKernelGGL((gemv_q4_kernel<16, 1, 12, true, 1>), dim3(static_cast<unsigned>(ntiles)),
                           dim3(64 * waves), static_cast<size_t>(waves) * 1024, st, w, act, act_stride, M, 0, 1, out);
        GV_CHECK_HIP(hipGetLastError());
        return 0;
    }
    // K ranges whose activations fit the waves' registers: one launch up to 4096 (2048 for 17..32 rows) values,
    // later ranges adding to the first's sums
    if (ntt == 2 && nsc == 32) {   // two ranges of 2048 in one launch (kept parts, up to two tiles a workgroup)
        int waves, kw;
        if (mfma_split(16 * kSuperK, 2, waves, kw) && kw == 8 && waves == 8 && tiles_per_wg(ntiles, waves, 2) <= 2) {
            const int64_t per = tiles_per_wg(ntiles, waves, 2), wg = (ntiles + per - 1) / per;
            const size_t lds = static_cast<size_t>(2 * per) * waves * 2 * 1024;
            static int granted = 0;
            if (lds_grant(reinterpret_cast<const void *>(&gemv_q4_2pass_kernel<8, 8>), lds, granted) != 0) return -1;
            hipLaunchKernelGGL((gemv_q4_2pass_kernel<8, 8>), dim3(static_cast<unsigned>(wg)), dim3(64 * waves), lds, st,
                               w, act, act_stride, M, 16, static_cast<int>(per), out);
            GV_CHECK_HIP(hipGetLastError());
            return 0;
        }
    }
    for (int sc0 = 0, part = 0; sc0 < nsc; ++part) {
        int n = std::min(nsc - sc0, ntt == 1 ? 32 : 16);
        int waves, kw;
        while (n > 1 && !mfma_split(static_cast<int64_t>(n) * kSuperK, ntt, waves, kw)) --n;
        GV_REQUIRE(sc0 % 4 == 0, "gemv_q4: a K range must start on a quad of super-chunks");
        GemvOut o = out;
        if (part > 0) o.accumulate = 1;
        if (gemv_range(w, act, act_stride, M, ntt, sc0, n, o, st) != 0) return -1;
        sc0 += n;
    }
    GV_CHECK_HIP(hipGetLastError());
    return 0;
}

}  // namespace gv
