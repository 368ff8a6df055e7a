// float32 linear layer and its gradients on the fp16 matrix cores:
//   y = x w^T + bias,   gx = gy w,   gw = gy^T x
// (F.linear of the quantization-aware training forward on the float32 A_q,
// RPFQ-ViT-main/quant_models/quant_i.py:554, and its backward).
//
// gfx950 has no matrix instruction between float32 (1/16 of the fp16 rate)
// and 16 bits, so each float32 operand is split into two fp16 terms,
// v s = h + l with s a power of two: h = fp16(v s), l = fp16(v s - h), and a
// product is the three MFMAs h h' + h l' + l h' in one float32 accumulator.
// h + l keeps v to 2^-22 relative (2^-39 of the scaled row's largest value
// once l is subnormal), and the dropped l l' is below 2^-22 of h h'; the
// accumulator takes 3 K / 16 roundings where a float32 GEMM takes K.
//
// A value more than 2^15 below the largest of its scale keeps fewer bits than
// a float32's.  Next to sums that hold the largest values that is lost in
// their rounding; it shows where a weight, or another row, takes those out.
// Such rows are summed in plain float32 instead: f32_wide_row (y, gx),
// gw_listed (gw), and all rows of a w whose parts differ that much.
//
// Scales: y and gx scale each row of x / gy by its own largest magnitude and
// w by one bound (the sum of its quantizer's scales), undone exactly on the
// output.  gw contracts over the rows, so a row's scale cannot be undone
// after the sum: gy keeps its row scales r[m], and row m of x is taken times
// 1 / r[m] times one power of two for the whole tensor.
#include <algorithm>

#include "rpfq_device.h"

namespace rpfq {

// Split rows ("planes"): row m, 32-column step ks at byte m ld + 128 ks:
// the step's 32 h values, then its 32 l values, so a step's tile row is one
// 128-byte line.  Rows and columns past the matrix are zero.
constexpr int kF32NoRow = -100000;
// What the passes of a call leave for the ones behind them, in its workspace.
struct F32Words {
    int emax;   // gw: largest exponent of a row's product of maxima, or kF32NoRow
    int gw;     // gw has rows that f32_exact_grad_kernel adds
    int rows;   // rows of y / gx that f32_exact_rows writes
};
// Most blocks of the gy pass where it also sums columns: 4 a CU.
constexpr int kColBlocks = 1024;

__device__ __forceinline__ int f32_scale_exp(float s) {  // s = 2^e
    return (int)((__float_as_uint(s) >> 23) & 0xffu) - 127;
}

// Rows of gw that f32_exact_grad_kernel sums, by the scales of gy's and x's row:
// inf or NaN (0), a wide row (negative), or a product of maxima more than 2^14
// below the largest such product.
__device__ __forceinline__ bool gw_listed(float r, float sx, int emax) {
    if (r <= 0.0f || sx <= 0.0f) return true;
    return r < __builtin_inff() && sx < __builtin_inff() && emax + f32_scale_exp(r) + f32_scale_exp(sx) > 14;
}

// Whether a row (mx: its largest magnitude, finite and not 0) holds values
// that the split loses beside the others and a sum may still depend on: in one
// half of its columns (a complex layer's weight can be 0 on one) fewer than 32
// values reach mx / 16, and the rest average below 2^-15 mx -- split operands
// keep 2^-39 mx, float32 2^-24 of the rest.  Also rows that row_prescale cannot
// lift to the top of fp16's range.  Ordinary rows are told by the count alone.
template <int NC>
__device__ __forceinline__ bool f32_wide_row(const f32x4 (&v)[NC][2], float mx, int K, int lane) {
    if (mx < 0x1p-112f) return true;
    const float thr = mx * 0.0625f;
    const int cut = (K / 2 + 7) / 8;  // of the 8-column pieces, those of the first half
    uint32_t count = 0;               // first half, second half << 16
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        uint32_t c = 0;
#pragma unroll
        for (int t = 0; t < 8; ++t) c += fabsf(v[i][t >> 2][t & 3]) >= thr;
        count += lane + 64 * i < cut ? c : c << 16;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) count += __shfl_xor((int)count, o, 64);
    const uint32_t big[2] = {count & 0xffffu, count >> 16};
    if (big[0] >= 32 && big[1] >= 32) return false;
    bool wide = false;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float sum = 0.0f, n = 0.0f;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            if ((lane + 64 * i < cut) != (h == 0)) continue;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const float a = fabsf(v[i][t >> 2][t & 3]);
                sum += a < thr ? a : 0.0f;
                n += a < thr && a > 0.0f ? 1.0f : 0.0f;
            }
        }
        sum = group_sum<64>(sum);
        n = group_sum<64>(n);
        wide |= big[h] < 32 && sum < 0x1p-15f * mx * n;
    }
    return wide;
}

// One wave per row, the row in registers (K <= 4096).  MODE 0: the row's own
// scale 2^e (largest magnitude in [2^14, 2^15)), written to scale[m]; +inf
// for a zero row, 0 for one with inf or NaN (its planes are zeroed), negative
// for a wide one; these two go to the list of exact rows.
// MODE 1 (gy): also collects the largest exponent of x's rows over r (emax).
// MODE 2 (x of gw): times 1 / r[m], r = gscale, and 2^-emax; rows that are not
// part of the split sum (gw_listed) are zero.
// COLS (gy): also the column sums of the block's rows, colsum[block][K], for
// the bias gradient: each lane adds the values it holds anyway (a separate
// reduction over 12,608 x 3,072 reads 155 MB again, 40.6 us; here 7.5 us and
// 8.2 of f32_colsum_kernel).
// HBM bound: 8 bytes per element.
template <int NC, int MODE, bool COLS = false>
__global__ void __launch_bounds__(256) f32_split_rows_kernel(const float* x, int64_t M, int64_t Mp, int K, int Kp,
                                                            const float* xscale, const float* gscale, F32Words* word,
                                                            int* list, char* planes, float* scale, float* colsum) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int emax = kF32NoRow, listed = 0;
    const int e2 = MODE == 2 ? word->emax : 0;
    f32x4 cs[NC][2];
    if (COLS) {
#pragma unroll
        for (int i = 0; i < NC; ++i) cs[i][0] = cs[i][1] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (int64_t m = (int64_t)blockIdx.x * 4 + wave; m < Mp; m += (int64_t)gridDim.x * 4) {
        f32x4 v[NC][2];
        const bool in = m < M;
        const float* row = x + (in ? m : 0) * (int64_t)K;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int c = lane + 64 * i;
            const bool ok = in && 8 * c < K;
            const f32x4* p = reinterpret_cast<const f32x4*>(row + (ok ? 8 * c : 0));
            v[i][0] = p[0];
            v[i][1] = p[1];
            if (!ok) v[i][0] = v[i][1] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
            if (COLS) {
                cs[i][0] += v[i][0];
                cs[i][1] += v[i][1];
            }
        }
        int k = 0;        // the row's scale is 2^k
        bool zero = !in;  // write zeros
        if (MODE != 2) {
            uint32_t mx = 0;
#pragma unroll
            for (int i = 0; i < NC; ++i)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    mx = max(mx, max(__float_as_uint(v[i][0][t]) & 0x7fffffffu, __float_as_uint(v[i][1][t]) & 0x7fffffffu));
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, o, 64));
            const bool fin = mx < 0x7f800000u;
            zero = !in || mx == 0 || !fin;
            const float s = !fin ? 0.0f : mx == 0 ? __builtin_inff() : row_prescale(__uint_as_float(mx));
            k = zero ? 0 : f32_scale_exp(s);
            const bool wide = !zero && f32_wide_row<NC>(v, __uint_as_float(mx), K, lane);
            if (in && lane == 0) {
                scale[m] = wide ? -s : s;
                if (!fin || wide) list[atomicAdd(&word->rows, 1)] = (int)m;
            }
            if (MODE == 1 && in) {
                const float sx = xscale[m];
                if (!zero && !wide && sx > 0.0f && sx < __builtin_inff()) emax = max(emax, -k - f32_scale_exp(sx));
            }
        } else if (in) {
            const float r = gscale[m], sx = xscale[m];
            const bool apart = gw_listed(r, sx, e2);
            if (apart) listed = 1;
            zero = apart || r == __builtin_inff() || sx == __builtin_inff();
            k = zero ? 0 : -f32_scale_exp(r) - e2;
        }
        char* dst = planes + m * (int64_t)Kp * 4;
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int c = lane + 64 * i;
            if (8 * c >= Kp) continue;
            uint4 h, l;
            uint32_t hw[4], lw[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float a = __builtin_amdgcn_ldexpf(v[i][t >> 1][2 * (t & 1)], k);
                const float b = __builtin_amdgcn_ldexpf(v[i][t >> 1][2 * (t & 1) + 1], k);
                split2(a, b, hw[t], lw[t]);
                if (zero) hw[t] = lw[t] = 0;
            }
            h = make_uint4(hw[0], hw[1], hw[2], hw[3]);
            l = make_uint4(lw[0], lw[1], lw[2], lw[3]);
            char* d = dst + (c >> 2) * 128 + (c & 3) * 16;
            *reinterpret_cast<uint4*>(d) = h;
            *reinterpret_cast<uint4*>(d + 64) = l;
        }
    }
    if (MODE == 1) {
        __shared__ int sm[4];
        if (lane == 0) sm[wave] = emax;
        __syncthreads();
        if (threadIdx.x == 0) atomicMax(&word->emax, max(max(sm[0], sm[1]), max(sm[2], sm[3])));
    }
    if (MODE == 2 && listed && lane == 0) atomicOr(&word->gw, 1);
    if (COLS) {  // the four waves one after another, then one coalesced row
        __shared__ __align__(16) float sum[NC * 512];
        for (int w = 0; w < 4; ++w) {
            if (wave == w) {
#pragma unroll
                for (int i = 0; i < NC; ++i) {
                    f32x4* d = reinterpret_cast<f32x4*>(sum + 8 * (lane + 64 * i));
                    d[0] = w == 0 ? cs[i][0] : d[0] + cs[i][0];
                    d[1] = w == 0 ? cs[i][1] : d[1] + cs[i][1];
                }
            }
            __syncthreads();
        }
        for (int c = threadIdx.x; c < K; c += 256) colsum[(int64_t)blockIdx.x * K + c] = sum[c];
    }
}

// out[c] = sum of parts[p][c], p < P, in a fixed order: 16 columns a block,
// 64 threads a column.
__global__ void __launch_bounds__(1024) f32_colsum_kernel(const float* parts, int P, int N, float* out) {
    __shared__ float sm[64][17];
    const int c = threadIdx.x & 15, q = threadIdx.x >> 4, n = blockIdx.x * 16 + c;
    float v = 0.0f;
    if (n < N)
        for (int p = q; p < P; p += 64) v += parts[(int64_t)p * N + n];
    sm[q][c] = v;
    __syncthreads();
    for (int h = 32; h > 0; h >>= 1) {
        if (q < h) sm[q][c] += sm[q + h][c];
        __syncthreads();
    }
    if (q == 0 && n < N) out[n] = sm[0][c];
}

// w [N, K] as the GEMM's A fragments of v_mfma_f32_32x32x16_f16, h and l:
// wf[rows / 32][contraction / 16][h, l][lane][8 fp16], lane (r, g) holding
// row r, contraction 8 g .. 8 g + 7.  TRANS = 0: rows = N, contraction = K;
// 1: rows = K, contraction = N.  One thread per 16 bytes of h and l; zero
// past the matrix.  The scale 2^e of w from the bound sum |parts| >= |w|
// goes to wscale[0] (0 if that is not finite, below 2^-112 or 2^15 times the
// smallest part: every row is then an exact one);
// block 0 also initialises the words.
template <int TRANS>
__global__ void __launch_bounds__(256) f32_split_w_kernel(const float* w, int N, int K, int rows32, int kt,
                                                         const float* parts, int nparts, char* wf, float* wscale,
                                                         F32Words* word) {
    float bound = 0.0f, least = __builtin_inff();
    for (int i = 0; i < nparts; ++i) {
        bound += fabsf(parts[i]);
        if (parts[i] != 0.0f) least = fminf(least, fabsf(parts[i]));
    }
    const bool fin = bound <= 3.40282347e38f && !(least < 0x1p-15f * bound) && !(bound > 0.0f && bound < 0x1p-112f);
    const float s = bound > 0.0f ? row_prescale(bound) : 1.0f;
    const int k = f32_scale_exp(s);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        wscale[0] = fin ? s : 0.0f;
        *word = {kF32NoRow, 0, 0};
    }
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= (int64_t)rows32 * kt * 64) return;
    const int lane = (int)(id & 63), r = lane & 31, g = lane >> 5;
    // TRANS: neighbouring threads take neighbouring rows (= columns of w)
    const int64_t f = id >> 6;
    const int t = (int)(f % kt);
    const int64_t row = (f / kt) * 32 + r;
    const int c0 = t * 16 + 8 * g;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int c = c0 + e;
        const bool ok = TRANS ? (row < K && c < N) : (row < N && c < K);
        const int64_t off = ok ? (TRANS ? (int64_t)c * K + row : row * K + c) : 0;
        v[e] = ok ? w[off] : 0.0f;
    }
    uint32_t h[4], l[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        split2(__builtin_amdgcn_ldexpf(v[2 * e], k), __builtin_amdgcn_ldexpf(v[2 * e + 1], k), h[e], l[e]);
    uint4* d = reinterpret_cast<uint4*>(wf) + f * 128 + lane;
    d[0] = make_uint4(h[0], h[1], h[2], h[3]);
    d[64] = make_uint4(l[0], l[1], l[2], l[3]);
}

struct F32Args {
    const char* xp;       // planes of the row operand
    const char* wf;       // fragments of w
    const float* scale;   // row scales [M]
    const float* wscale;  // scale of w
    const float* bias;    // [N] or NULL
    float* y;             // [M, N]
    int64_t M;
    int N, KS;            // outputs, 32-column steps
    int wf_bytes;
    int tiles_m, tiles_n, group;
};

// Workgroup = 4 waves, tile = BM rows x 256 outputs, wave w the outputs
// 64 w .. 64 w + 63 (two 32-row fragments of wf) of every row.  Rows go
// global -> LDS by DMA (3 stages of one 32-column step, swizzled as the
// packed DMA kernel's); w's fragments are private to the wave and go
// straight from L2 to registers, three 16-column substeps ahead, so LDS
// carries only the rows.  24 MFMAs (BM = 128) per substep on 8 LDS reads and
// 4 fragment loads.  Two workgroups per CU; the product is transposed (w is
// the A operand), so a lane holds 4 consecutive outputs of one row and the
// tile leaves through a swizzled LDS transpose of its own as whole 256-byte
// row pieces.  MFMA bound: 12,608 x 3072 x 768 in 165 us, 1.08 PFLOP/s of
// fp16 products (the float32 library GEMM: 541 us).
constexpr int kF32Epi = 8192;  // epilogue bytes of one wave: 32 rows x 64 outputs
template <int MB> constexpr int f32_stage() { return MB * 32 * 128; }
template <int MB> constexpr int f32_lds() { return 3 * f32_stage<MB>() + 4 * kF32Epi; }
static_assert(2 * f32_lds<4>() <= 160 * 1024, "two workgroups per CU");

__device__ __forceinline__ floatx16 mfma_h(half8 a, half8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// One wave's 32 x 64 block (acc0, acc1: outputs 0..31, 32..63 of lane rows
// r) through its LDS to y: rows m0 .. m0 + 31 below M, outputs n0 .. n0 + 63
// below N (a multiple of 4, y 16-byte aligned), times 2^e (e per lane row).
__device__ __forceinline__ void f32_store_block(char* epi, const floatx16& acc0, const floatx16& acc1, int e,
                                                const float* bias, float* y, int64_t m0, int64_t M, int64_t n0,
                                                int64_t N, int lane) {
    const int r = lane & 31, g = lane >> 5;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        *reinterpret_cast<f32x4*>(epi + r * 256 + (((2 * q + g) ^ (r & 15)) * 16)) =
            (f32x4){__builtin_amdgcn_ldexpf(acc0[4 * q], e), __builtin_amdgcn_ldexpf(acc0[4 * q + 1], e),
                    __builtin_amdgcn_ldexpf(acc0[4 * q + 2], e), __builtin_amdgcn_ldexpf(acc0[4 * q + 3], e)};
        *reinterpret_cast<f32x4*>(epi + r * 256 + (((8 + 2 * q + g) ^ (r & 15)) * 16)) =
            (f32x4){__builtin_amdgcn_ldexpf(acc1[4 * q], e), __builtin_amdgcn_ldexpf(acc1[4 * q + 1], e),
                    __builtin_amdgcn_ldexpf(acc1[4 * q + 2], e), __builtin_amdgcn_ldexpf(acc1[4 * q + 3], e)};
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    const int c = lane & 15;
    const int64_t n = n0 + 4 * c;
    f32x4 b = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    if (bias && n < N) b = (f32x4){bias[n], bias[n + 1], bias[n + 2], bias[n + 3]};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int row = 4 * j + (lane >> 4);
        const f32x4 v = *reinterpret_cast<const f32x4*>(epi + row * 256 + ((c ^ (row & 15)) * 16));
        if (m0 + row < M && n < N)
            __builtin_nontemporal_store(v + b, reinterpret_cast<f32x4*>(y + (m0 + row) * N + n));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

template <int MB>
__global__ void __launch_bounds__(256, 2) f32_gemm_kernel(F32Args a) {
    if (a.wscale[0] == 0.0f) return;  // every row is an exact one
    extern __shared__ __align__(16) char smem[];
    constexpr int BM = 32 * MB, RPW = BM / 4, XL = RPW / 8;  // rows and DMA loads per wave and step
    constexpr int STAGE = f32_stage<MB>();
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    char* epi = smem + 3 * STAGE + wave * kF32Epi;
    const int64_t ld = (int64_t)a.KS * 128;
    const int kt = 2 * a.KS;
    // wave w fills rows RPW w .. of a stage with 1-KB loads of 8 rows: lane l
    // writes row l >> 3, slot l & 7, which holds chunk (l & 7) ^ ((row >> 1) & 7)
    uint32_t voff[2];
#pragma unroll
    for (int p = 0; p < 2; ++p)
        voff[p] = (uint32_t)((lane >> 3) * ld + (((lane & 7) ^ ((4 * p + (lane >> 4)) & 7)) * 16));
    const int par = (XL * wave) & 1;
    const uint32_t v0 = par ? voff[1] : voff[0], v1 = par ? voff[0] : voff[1];
    const uint32_t lds_x = lds_addr(smem) + RPW * wave * 128;
    const char* xw = nullptr;
    // buffer loads: one resource and a scalar offset per load
    const __amdgpu_buffer_rsrc_t wf = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.wf), 0, a.wf_bytes, 0x00027000);
    const uint32_t wv = lane * 16;
    uint32_t wo[2] = {0, 0};
    auto issue_x = [&](int ks, int st) {
        const char* src = xw + ks * 128;
#pragma unroll
        for (int j = 0; j < XL; ++j) dma_dwordx4(src + 8 * j * ld, j & 1 ? v1 : v0, lds_x + st * STAGE + j * 1024);
    };
    // fragments of substep t: [j][h, l]
    auto load_w = [&](int t, uint4 (&f)[2][2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            f[j][0] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wf, wv, wo[j] + t * 2048, 0));
            f[j][1] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wf, wv, wo[j] + t * 2048 + 1024, 0));
        }
    };
    uint32_t aoff[2][2];  // [h, l][substep]: chunk 4 p + 2 s + g of row r
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int s = 0; s < 2; ++s) aoff[p][s] = lds_addr(smem) + r * 128 + (((4 * p + 2 * s + g) ^ ((r >> 1) & 7)) * 16);

    const int total = a.tiles_m * a.tiles_n;
    int mt = 0, ntl = 0;
    auto set_tile = [&](int vb) {
        group_tile(xcd_tile(vb, total), a.tiles_m, a.tiles_n, a.group, mt, ntl);
        xw = a.xp + ((int64_t)mt * BM + RPW * wave) * ld;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            wo[j] = (uint32_t)__builtin_amdgcn_readfirstlane(((ntl * 4 + wave) * 2 + j) * kt * 2048);
    };
    uint4 w0[2][2], w1[2][2], w2[2][2];
    const int we = f32_scale_exp(a.wscale[0]);
    if ((int)blockIdx.x < total) {
        set_tile(blockIdx.x);
        issue_x(0, 0);
        if (a.KS > 1) issue_x(1, 1);
        load_w(0, w0);
        load_w(1, w1);
        load_w(kt > 2 ? 2 : 1, w2);
    }
    for (int vb = blockIdx.x; vb < total; vb += gridDim.x) {
        const int64_t mrow = (int64_t)mt * BM, n0 = (int64_t)ntl * 256 + 64 * wave;
        floatx16 acc[2][MB];
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[0][i] = acc[1][i] = floatx16{0};
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        auto substep = [&](int t, int s, int st, uint4 (&f)[2][2], bool issue, int ks) {
            half8 xh[MB], xl[MB];
#pragma unroll
            for (int i = 0; i < MB; ++i) xh[i] = *((lds_h8_t)aoff[0][s] + (st * STAGE + i * 4096) / 16);
#pragma unroll
            for (int i = 0; i < MB; ++i) xl[i] = *((lds_h8_t)aoff[1][s] + (st * STAGE + i * 4096) / 16);
            const half8 h0 = as_half8(f[0][0]), h1 = as_half8(f[1][0]);
            const half8 l0 = as_half8(f[0][1]), l1 = as_half8(f[1][1]);
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                acc[0][i] = mfma_h(h0, xh[i], acc[0][i]);
                acc[1][i] = mfma_h(h1, xh[i], acc[1][i]);
            }
            if (issue) issue_x(ks + 2, (st + 2) % 3);
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                acc[0][i] = mfma_h(l0, xh[i], acc[0][i]);
                acc[1][i] = mfma_h(l1, xh[i], acc[1][i]);
            }
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                acc[0][i] = mfma_h(h0, xl[i], acc[0][i]);
                acc[1][i] = mfma_h(h1, xl[i], acc[1][i]);
            }
            load_w(t + 3 < kt ? t + 3 : kt - 1, f);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto kstep = [&](int ks, int st, uint4 (&fa)[2][2], uint4 (&fb)[2][2]) {
            const bool more = ks + 2 < a.KS;
            substep(2 * ks, 0, st, fa, more, ks);
            substep(2 * ks + 1, 1, st, fb, false, ks);
            // the rows of ks + 1 landed: younger are 8 fragment loads of the
            // step before, this step's 8 and the XL of ks + 2
            if (more)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(16 + XL) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        int ks = 0;
        for (; ks + 3 <= a.KS; ks += 3) {
            kstep(ks, 0, w0, w1);
            kstep(ks + 1, 1, w2, w0);
            kstep(ks + 2, 2, w1, w2);
        }
        if (ks < a.KS) kstep(ks, 0, w0, w1);
        if (ks + 1 < a.KS) kstep(ks + 1, 1, w2, w0);
        if (vb + (int)gridDim.x < total) {  // the next tile's first loads land beside the epilogue
            set_tile(vb + (int)gridDim.x);
            issue_x(0, 0);
            if (a.KS > 1) issue_x(1, 1);
            load_w(0, w0);
            load_w(1, w1);
            load_w(kt > 2 ? 2 : 1, w2);
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const int64_t m = mrow + 32 * i;
            const float s = a.scale[m + r < a.M ? m + r : a.M - 1];
            f32_store_block(epi, acc[0][i], acc[1][i], -f32_scale_exp(s) - we, a.bias, a.y, m, a.M, n0, a.N, lane);
        }
    }
}

// gw tile: 128 columns of gy x 256 columns of x over 16-row steps of the two
// planes, both contracted down their rows: the tiles lie in LDS as in memory
// and ds_read_b64_tr_b16 gathers 4 rows of a column per lane.  Wave w takes
// 64 of x's columns against all 128 of gy's.  A stage row is 512 B of gy and
// 1 KB of x, chunk c of 16 B stored at c ^ ((row & 3) << 2): the 4 rows one
// read touches fall on distinct banks.  part: [split][N][K] partial sums
// (or gw itself for one split).  gw [3072, 768] over 12,608 rows: 168 us,
// 1.06 PFLOP/s of fp16 products (the float32 library GEMM: 515 us); a
// transposed copy of both operands for f32_gemm_kernel would move 0.4 GB more.
struct F32GwArgs {
    const char* gp;   // planes of gy
    const char* xp;   // planes of x
    const F32Words* word;
    float* part;
    int64_t ldg, ldx;  // plane row bytes
    int N, K;
    int steps, per;    // 16-row steps in all, and per split
    int tiles_n, tiles_k, splits;
};
constexpr int kGwG = 16 * 512, kGwStage = kGwG + 16 * 1024;
constexpr int kGwLds = 3 * kGwStage + 256;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s4_t;

__global__ void __launch_bounds__(256, 2) f32_gw_kernel(F32GwArgs a) {
    extern __shared__ __align__(16) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 5, i16 = lane & 15, hf = (lane >> 4) & 1;
    const int tiles = a.tiles_n * a.tiles_k;
    const int unit = xcd_tile(blockIdx.x, tiles * a.splits);
    const int sp = unit / tiles, tile = unit - sp * tiles;
    const int tn = tile / a.tiles_k, tk = tile - tn * a.tiles_k;
    const int s0 = sp * a.per, s1 = min(a.steps, s0 + a.per);
    // DMA: gy 2 loads of 2 rows, x 4 loads of 1 row per wave
    uint32_t gv[2], xv[4];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int row = 4 * wave + 2 * e + (lane >> 5);
        gv[e] = (uint32_t)(row * a.ldg + (((lane & 31) ^ ((row & 3) << 2)) * 16));
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) xv[e] = (uint32_t)((4 * wave + e) * a.ldx + ((lane ^ (e << 2)) * 16));
    const char* gsrc = a.gp + (int64_t)tn * 512;
    const char* xsrc = a.xp + (int64_t)tk * 1024;
    const uint32_t lds0 = lds_addr(smem);
    auto issue = [&](int step, int st) {
        const char* gs = gsrc + (int64_t)step * 16 * a.ldg;
        const char* xs = xsrc + (int64_t)step * 16 * a.ldx;
        const uint32_t d = lds0 + st * kGwStage;
#pragma unroll
        for (int e = 0; e < 2; ++e) dma_dwordx4(gs, gv[e], d + (4 * wave + 2 * e) * 512);
#pragma unroll
        for (int e = 0; e < 4; ++e) dma_dwordx4(xs, xv[e], d + kGwG + (4 * wave + e) * 1024);
    };
    // lane l of a transposed read: row 8 g + i16 / 4 (+ 4 for the second
    // half), columns 16 hf + 4 (i16 & 3) .. + 3 of the 32-column block
    const int row = 8 * g + (i16 >> 2), sw = (i16 >> 2) << 2;
    uint32_t ga[2][2], xa[2][2];  // [h, l][block parity]
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int cg = j * 8 + p * 4 + 2 * hf + ((i16 & 3) >> 1);
            const int cx = (2 * wave + j) * 8 + p * 4 + 2 * hf + ((i16 & 3) >> 1);
            ga[p][j] = lds0 + row * 512 + ((cg ^ sw) * 16) + (i16 & 1) * 8;
            xa[p][j] = lds0 + kGwG + row * 1024 + ((cx ^ sw) * 16) + (i16 & 1) * 8;
        }
    auto frag = [&](uint32_t at, int half) -> half8 {  // 8 rows of a column
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)at);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)(at + half));
        return __builtin_bit_cast(half8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    floatx16 acc[2][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[0][i] = acc[1][i] = floatx16{0};
    if (s0 < s1) issue(s0, 0);
    if (s0 + 1 < s1) issue(s0 + 1, 1);
    int st = 0;
    for (int s = s0; s < s1; ++s) {
        if (s + 1 < s1)
            asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int nst = st == 0 ? 2 : st - 1;  // (st + 2) % 3: read a step ago
        if (s + 2 < s1) issue(s + 2, nst);
        const uint32_t so = st * kGwStage;
        half8 xh[2], xl[2], gf[4];
#pragma unroll
        for (int j = 0; j < 2; ++j) xh[j] = frag(xa[0][j] + so, 4096);
#pragma unroll
        for (int i = 0; i < 4; ++i) gf[i] = frag(ga[0][i & 1] + so + (i >> 1) * 256, 2048);
#pragma unroll
        for (int j = 0; j < 2; ++j) xl[j] = frag(xa[1][j] + so, 4096);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[0][i] = mfma_h(xh[0], gf[i], acc[0][i]);
            acc[1][i] = mfma_h(xh[1], gf[i], acc[1][i]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[0][i] = mfma_h(xl[0], gf[i], acc[0][i]);
            acc[1][i] = mfma_h(xl[1], gf[i], acc[1][i]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) gf[i] = frag(ga[1][i & 1] + so + (i >> 1) * 256, 2048);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[0][i] = mfma_h(xh[0], gf[i], acc[0][i]);
            acc[1][i] = mfma_h(xh[1], gf[i], acc[1][i]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        st = st == 2 ? 0 : st + 1;
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int e = a.splits == 1 && a.word->emax != kF32NoRow ? a.word->emax : 0;
    const int64_t k0 = (int64_t)tk * 256 + 64 * wave;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f32_store_block(smem + wave * kF32Epi, acc[0][i], acc[1][i], e, nullptr,
                        a.part + (int64_t)sp * a.N * a.K, (int64_t)tn * 128 + 32 * i, a.N, k0, a.K, lane);
    }
}

// gw = 2^emax (1 after f32_exact_grad_kernel) times the sum of the splits'
// partials, in their order.
__global__ void __launch_bounds__(256) f32_gw_reduce_kernel(const float* part, int64_t n4, int splits, const F32Words* word,
                                                           float* gw) {
    const int e = word->emax == kF32NoRow || word->gw ? 0 : word->emax;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) {
        f32x4 v = reinterpret_cast<const f32x4*>(part)[i];
        for (int s = 1; s < splits; ++s) v += reinterpret_cast<const f32x4*>(part)[i + s * n4];
        f32x4 o;
#pragma unroll
        for (int t = 0; t < 4; ++t) o[t] = __builtin_amdgcn_ldexpf(v[t], e);
        reinterpret_cast<f32x4*>(gw)[i] = o;
    }
}

// ---------------------------------------------------------------------------
// exact rows: plain float32 sums
// ---------------------------------------------------------------------------
// Where split operands do not stand for their values the products
// run on v_mfma_f32_32x32x2_f32, so that special values come out as a float32
// GEMM's: the listed rows of y and gx, and the listed rows' share of gw.  1/16
// of the fp16 rate; with every row listed 12,608 x 3,072 x 768 takes 640 us a
// product (the float32 library GEMM: 541), and an empty list one short launch.
//
// Tile: 128 rows i x 128 outputs j, 4 waves of 64 x 64, 16 of the contraction
// c a step through two LDS buffers of odd row stride (17 floats: 32 rows of a
// column on distinct banks), the next step's loads in registers meanwhile.
// AC / BC: operand a / b lies with c contiguous (rows of lda), else with i / j
// contiguous.  Sums of 512 products, then the sum of those.
struct F32Exact {
    const float* a;
    const float* b;
    const float* bias;  // of the outputs j, or NULL
    float* out;         // [.., J]
    const int* list;    // rows i of a and out, or NULL: as they are
    int64_t lda, ldb;
    int64_t I;
    int J;
};
constexpr int kExLd = 17, kExHalf = 128 * kExLd;
struct F32ExactSum {
    floatx16 acc[2][2], sum[2][2];  // [j block][i block]
    int steps;
    __device__ __forceinline__ void zero() {
        steps = 0;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[j][i] = sum[j][i] = floatx16{0};
    }
};

// Adds c0 .. c1 - 1 of the contraction to the tile at (i0, j0); rows: where c
// is a row number of a and b, these (in LDS) instead of c itself.
template <bool AC, bool BC>
__device__ __forceinline__ void f32_exact_add(const F32Exact& x, float* lds, int64_t i0, int j0, int64_t c0, int64_t c1,
                                              const int* rows, F32ExactSum& s) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, g = lane >> 5, wi = (wave & 1) * 64, wj = (wave >> 1) * 64;
    // two 4-float loads of each operand: (row q4, columns 4 qc ..) of the tile,
    // or (contraction q, rows 4 qr ..)
    const int q4 = tid >> 2, qc = 4 * (tid & 3), q = tid >> 5, qr = 4 * (tid & 31);
    const float* ap[2];
    const float* bp[2];
    bool aok[2], bok[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int64_t i = AC ? i0 + q4 + 64 * p : i0 + qr;
        aok[p] = i < x.I;
        const int64_t row = !aok[p] ? 0 : AC && x.list ? x.list[i] : i;
        ap[p] = AC ? x.a + row * x.lda + qc : x.a + row;
        const int j = BC ? j0 + q4 + 64 * p : j0 + qr;
        bok[p] = j < x.J;
        bp[p] = BC ? x.b + (int64_t)(bok[p] ? j : 0) * x.ldb + qc : x.b + (bok[p] ? j : 0);
    }
    f32x4 ra[2], rb[2];
    auto load = [&](int64_t c) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            ra[p] = rb[p] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
            const int64_t ca = AC ? c + qc : c + q + 8 * p, cb = BC ? c + qc : c + q + 8 * p;
            const int64_t at = !AC && rows && ca < c1 ? rows[ca] : ca, bt = !BC && rows && cb < c1 ? rows[cb] : cb;
            if (aok[p] && ca < c1) ra[p] = *reinterpret_cast<const f32x4*>(AC ? ap[p] + c : ap[p] + at * x.lda);
            if (bok[p] && cb < c1) rb[p] = *reinterpret_cast<const f32x4*>(BC ? bp[p] + c : bp[p] + bt * x.ldb);
        }
    };
    auto store = [&](float* d) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                d[AC ? (q4 + 64 * p) * kExLd + qc + e : (qr + e) * kExLd + q + 8 * p] = ra[p][e];
                d[kExHalf + (BC ? (q4 + 64 * p) * kExLd + qc + e : (qr + e) * kExLd + q + 8 * p)] = rb[p][e];
            }
    };
    __syncthreads();  // rows is written, the step before this one is read
    load(c0);
    store(lds);
    __syncthreads();
    int buf = 0;
    for (int64_t c = c0; c < c1; c += 16) {
        const bool more = c + 16 < c1;
        if (more) load(c + 16);
        const float* la = lds + buf * 2 * kExHalf + (wi + r) * kExLd + g;
        const float* lb = lds + buf * 2 * kExHalf + kExHalf + (wj + r) * kExLd + g;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float a0 = la[2 * k], a1 = la[32 * kExLd + 2 * k], b0 = lb[2 * k], b1 = lb[32 * kExLd + 2 * k];
            s.acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(b0, a0, s.acc[0][0], 0, 0, 0);
            s.acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(b0, a1, s.acc[0][1], 0, 0, 0);
            s.acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(b1, a0, s.acc[1][0], 0, 0, 0);
            s.acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(b1, a1, s.acc[1][1], 0, 0, 0);
        }
        if (++s.steps % 32 == 0) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    s.sum[j][i] += s.acc[j][i];
                    s.acc[j][i] = floatx16{0};
                }
        }
        if (more) store(lds + (buf ^ 1) * 2 * kExHalf);
        __syncthreads();
        buf ^= 1;
    }
}

// out = the tile plus bias, or (ADD) out times 2^e plus the tile.
template <bool ADD>
__device__ __forceinline__ void f32_exact_store(const F32Exact& x, int64_t i0, int j0, const F32ExactSum& s, int e) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 31, g = lane >> 5, wi = (wave & 1) * 64, wj = (wave >> 1) * 64;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int64_t at = i0 + wi + 32 * i + r;
        if (at >= x.I) continue;
        float* out = x.out + (x.list ? (int64_t)x.list[at] : at) * x.J;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) {  // a lane holds 4 consecutive outputs
                const int n = j0 + wj + 32 * j + 8 * t + 4 * g;
                if (n >= x.J) continue;
                f32x4* o = reinterpret_cast<f32x4*>(out + n);
                f32x4 v, b = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
                if (ADD) v = *o;
                else if (x.bias) b = (f32x4){x.bias[n], x.bias[n + 1], x.bias[n + 2], x.bias[n + 3]};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float w = s.sum[j][i][4 * t + k] + s.acc[j][i][4 * t + k];
                    v[k] = ADD ? __builtin_amdgcn_ldexpf(v[k], e) + w : w + b[k];
                }
                *o = v;
            }
    }
}

// The listed rows of y = x w^T + bias (BC) or gx = gy w, or every row where w
// has no scale: block `first` of `blocks`.  C: the contraction.
template <bool BC>
__device__ __forceinline__ void f32_exact_rows(F32Exact x, float* lds, int C, const F32Words* word, const float* wscale,
                                               int first, int blocks) {
    if (wscale[0] == 0.0f)
        x.list = nullptr;
    else
        x.I = word->rows;
    const int tj = (x.J + 127) / 128;
    const int64_t tiles = (x.I + 127) / 128 * tj;
    for (int64_t t = first; t < tiles; t += blocks) {
        F32ExactSum s;
        s.zero();
        f32_exact_add<true, BC>(x, lds, t / tj * 128, (int)(t % tj) * 128, 0, C, nullptr, s);
        f32_exact_store<false>(x, t / tj * 128, (int)(t % tj) * 128, s, 0);
    }
}

__global__ void __launch_bounds__(256, 2) f32_exact_y_kernel(F32Exact x, int C, const F32Words* word, const float* wscale) {
    __shared__ float lds[4 * kExHalf];
    f32_exact_rows<true>(x, lds, C, word, wscale, blockIdx.x, gridDim.x);
}

// Both gradients' share in one launch: the first gx_blocks blocks the listed
// rows of gx; the others, one per tile of gw and row split of f32_gw_kernel,
// add the listed rows' share to gw (splits = 1) or to the partial sums, which
// leave their unit 2^emax with it (the listed rows may lie far above), in the
// rows' order, 1,024 rows at a time through LDS.
struct F32ExactGrad {
    F32Exact gx, gw;
    int gx_blocks, N;
    int64_t M, per;
    int splits;
    const float *gscale, *xscale, *wscale;
    const F32Words* word;
};
__global__ void __launch_bounds__(256, 2) f32_exact_grad_kernel(F32ExactGrad a) {
    __shared__ float lds[4 * kExHalf];
    __shared__ int rows[1024], total[4];
    if ((int)blockIdx.x < a.gx_blocks) {
        f32_exact_rows<false>(a.gx, lds, a.N, a.word, a.wscale, blockIdx.x, a.gx_blocks);
        return;
    }
    if (a.word->gw == 0) return;
    F32Exact x = a.gw;
    const int emax = a.word->emax, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int tj = (x.J + 127) / 128, tiles = (int)((x.I + 127) / 128) * tj;
    const int unit = blockIdx.x - a.gx_blocks, sp = unit / tiles, tile = unit - sp * tiles;
    const int j0 = tile % tj * 128;
    const int64_t i0 = (int64_t)(tile / tj) * 128;
    const int64_t m1 = min(a.M, ((int64_t)sp + 1) * a.per);
    x.out += (int64_t)sp * x.I * x.J;
    F32ExactSum s;
    s.zero();
    for (int64_t m0 = (int64_t)sp * a.per; m0 < m1; m0 += 1024) {
        bool on[4];
        int n = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int64_t m = m0 + 4 * threadIdx.x + t;
            on[t] = m < m1 && gw_listed(a.gscale[m], a.xscale[m], emax);
            n += on[t];
        }
        int before = n;  // of the lanes up to this one
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(before, o, 64);
            if (lane >= o) before += v;
        }
        if (lane == 63) total[wave] = before;
        __syncthreads();
        int at = before - n, count = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            if (w < wave) at += total[w];
            count += total[w];
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (on[t]) rows[at++] = (int)(m0 + 4 * threadIdx.x + t);
        if (count) f32_exact_add<false, false>(x, lds, i0, j0, 0, count, rows, s);
        __syncthreads();  // total and rows are read
    }
    f32_exact_store<true>(x, i0, j0, s, a.splits > 1 && emax != kF32NoRow ? emax : 0);
}

// ---------------------------------------------------------------------------
// workspaces and launches
// ---------------------------------------------------------------------------
static int64_t up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

static int f32_splits(int64_t N, int64_t K, int64_t steps) {
    const int64_t tiles = ((N + 127) / 128) * ((K + 255) / 256), slots = 2 * (int64_t)device_cus();
    int best = 1;
    double cost = 1e30;
    for (int s = 1; s <= 64 && (s == 1 || steps / s >= 16); ++s) {
        const int64_t per = (steps + s - 1) / s;
        // ~1 us per step and round of slots; partials leave and return at ~4 bytes a picosecond
        const double c = (double)((tiles * s + slots - 1) / slots) * (double)(per + 8) * 0.9 +
                         (s > 1 ? (double)s * N * K * 8.0 / 4.0e6 + 3.0 : 0.0);
        if (c < cost) {
            cost = c;
            best = s;
        }
    }
    return best;
}

F32Plan f32_plan(int64_t M, int64_t N, int64_t K) {
    F32Plan p = {};
    p.Mp = up(M, 384);  // whole tiles of 128, 96 and 64 rows
    p.Kp = up(K, 32);
    p.Np = up(N, 32);
    const size_t slack = 2048;  // a gw tile's last rows read past a ragged plane row
    size_t at = 256;
    p.x_at = at;
    at += (size_t)up(p.Mp * p.Kp * 4 + slack, 256);
    p.w_at = at;
    at += (size_t)(up(N, 256) / 32 * (p.Kp / 16) * 2048);
    p.wf_bytes = at - p.w_at;
    p.list_at = at;
    at += (size_t)up(M * 4, 256);
    p.fwd_bytes = at;
    at = 256;
    // x's planes; before they are written, the column sums of gy's blocks
    p.bx_at = at;
    const int64_t xb = p.Mp * p.Kp * 4 + slack, cb = std::min<int64_t>(p.Mp / 4, kColBlocks) * N * 4;
    at += (size_t)up(xb > cb ? xb : cb, 256);
    p.g_at = at;
    at += (size_t)up(p.Mp * p.Np * 4 + slack, 256);
    p.bw_at = at;
    at += (size_t)(up(K, 256) / 32 * (p.Np / 16) * 2048);
    p.bwf_bytes = at - p.bw_at;
    p.gs_at = at;
    at += (size_t)up(p.Mp * 4, 256);
    p.blist_at = at;
    at += (size_t)up(M * 4, 256);
    p.steps = (int)(up(M, 16) / 16);
    p.splits = f32_splits(N, K, p.steps);
    p.part_at = at;
    if (p.splits > 1) at += (size_t)p.splits * N * K * 4;
    p.bwd_bytes = at;
    return p;
}

template <int MODE, bool COLS = false>
static hipError_t split_rows(const float* x, int64_t M, int64_t Mp, int64_t K, int64_t Kp, const float* xscale,
                             const float* gscale, F32Words* word, int* list, char* planes, float* scale, hipStream_t s,
                             float* colsum = nullptr, float* colout = nullptr) {
    const int nc = (int)((Kp + 511) / 512);
    const int64_t rows4 = (Mp + 3) / 4, most = COLS ? kColBlocks : 2048;
    const int grid = (int)(rows4 < most ? rows4 : most);
#define RPFQ_SPLIT(NC)                                                                                              \
    hipLaunchKernelGGL((f32_split_rows_kernel<NC, MODE, COLS>), dim3(grid), dim3(256), 0, s, x, M, Mp, (int)K,    \
                       (int)Kp, xscale, gscale, word, list, planes, scale, colsum)
    if (nc <= 1) RPFQ_SPLIT(1);
    else if (nc <= 2) RPFQ_SPLIT(2);
    else if (nc <= 4) RPFQ_SPLIT(4);
    else if (nc <= 6) RPFQ_SPLIT(6);
    else RPFQ_SPLIT(8);
#undef RPFQ_SPLIT
    if (COLS)
        hipLaunchKernelGGL(f32_colsum_kernel, dim3((unsigned)((K + 15) / 16)), dim3(1024), 0, s, (const float*)colsum, grid,
                           (int)K, colout);
    return hipGetLastError();
}

template <int TRANS>
static hipError_t split_w(const float* w, int64_t N, int64_t K, const float* parts, int nparts, char* wf,
                          float* wscale, F32Words* word, hipStream_t s) {
    const int64_t rows = TRANS ? K : N, con = TRANS ? N : K;
    const int rows32 = (int)(up(rows, 256) / 32), kt = (int)(up(con, 32) / 16);
    hipLaunchKernelGGL((f32_split_w_kernel<TRANS>), dim3((rows32 * kt + 3) / 4), dim3(256), 0, s, w, (int)N, (int)K,
                       rows32, kt, parts, nparts, wf, wscale, word);
    return hipGetLastError();
}

template <int MB>
static hipError_t f32_gemm_go(F32Args& a, hipStream_t s) {
    static std::atomic<uint64_t> attr_done{0};
    const hipError_t e = set_lds_attr_once(reinterpret_cast<const void*>(&f32_gemm_kernel<MB>), f32_lds<MB>(), attr_done);
    if (e != hipSuccess) return e;
    a.tiles_m = (int)((a.M + 32 * MB - 1) / (32 * MB));
    a.tiles_n = (a.N + 255) / 256;
    a.group = tile_group(a.tiles_n, (int64_t)a.KS * 32768);
    const int total = a.tiles_m * a.tiles_n, slots = 2 * device_cus();
    hipLaunchKernelGGL((f32_gemm_kernel<MB>), dim3(total < slots ? total : slots), dim3(256), f32_lds<MB>(), s, a);
    return hipGetLastError();
}

static hipError_t f32_gemm(F32Args& a, hipStream_t s) {
    const int mb = rows_per_tile(a.M, a.N);
    if (mb == 2) return f32_gemm_go<2>(a, s);
    if (mb == 3) return f32_gemm_go<3>(a, s);
    return f32_gemm_go<4>(a, s);
}

// Blocks of f32_exact_rows for rows x J outputs.
static int exact_blocks(int64_t rows, int64_t J) {
    return (int)std::min<int64_t>((rows + 127) / 128 * ((J + 127) / 128), 2 * (int64_t)device_cus());
}

#define RPFQ_TRY(e)                           \
    do {                                      \
        const hipError_t e_ = (e);            \
        if (e_ != hipSuccess) return e_;      \
    } while (0)

hipError_t launch_linear_f32(const float* x, const float* w, const float* bias, int64_t M, int64_t N, int64_t K,
                             const float* parts, int nparts, float* y, float* xscale, void* work, hipStream_t s) {
    const F32Plan p = f32_plan(M, N, K);
    char* base = reinterpret_cast<char*>(work);
    float* wscale = reinterpret_cast<float*>(base);
    F32Words* word = reinterpret_cast<F32Words*>(base + 64);
    int* list = reinterpret_cast<int*>(base + p.list_at);
    RPFQ_TRY(split_w<0>(w, N, K, parts, nparts, base + p.w_at, wscale, word, s));
    RPFQ_TRY(split_rows<0>(x, M, p.Mp, K, p.Kp, nullptr, nullptr, word, list, base + p.x_at, xscale, s));
    F32Args a = {};
    a.xp = base + p.x_at;
    a.wf = base + p.w_at;
    a.scale = xscale;
    a.wscale = wscale;
    a.bias = bias;
    a.y = y;
    a.M = M;
    a.N = (int)N;
    a.KS = (int)(p.Kp / 32);
    a.wf_bytes = (int)p.wf_bytes;
    RPFQ_TRY(f32_gemm(a, s));
    F32Exact e = {};
    e.a = x;
    e.b = w;
    e.bias = bias;
    e.out = y;
    e.list = list;
    e.lda = e.ldb = K;
    e.I = M;
    e.J = (int)N;
    hipLaunchKernelGGL(f32_exact_y_kernel, dim3(exact_blocks(M, N)), dim3(256), 0, s, e, (int)K, (const F32Words*)word,
                       (const float*)wscale);
    return hipGetLastError();
}

hipError_t launch_linear_f32_grad(const float* gy, const float* x, const float* w, int64_t M, int64_t N, int64_t K,
                                  const float* parts, int nparts, const float* xscale, float* gx, float* gw,
                                  float* gb, void* work, hipStream_t s) {
    const F32Plan p = f32_plan(M, N, K);
    char* base = reinterpret_cast<char*>(work);
    float* wscale = reinterpret_cast<float*>(base);
    F32Words* word = reinterpret_cast<F32Words*>(base + 64);
    int* list = reinterpret_cast<int*>(base + p.blist_at);
    float* gscale = reinterpret_cast<float*>(base + p.gs_at);
    F32ExactGrad e = {};
    e.M = M;
    e.N = (int)N;
    e.splits = p.splits;
    e.gscale = gscale;
    e.xscale = xscale;
    e.wscale = wscale;
    e.word = word;
    int exact = 0;  // blocks
    RPFQ_TRY(split_w<1>(w, N, K, parts, nparts, base + p.bw_at, wscale, word, s));
    if (gb)
        RPFQ_TRY((split_rows<1, true>(gy, M, p.Mp, N, p.Np, xscale, nullptr, word, list, base + p.g_at, gscale, s,
                                      reinterpret_cast<float*>(base + p.bx_at), gb)));
    else
        RPFQ_TRY(split_rows<1>(gy, M, p.Mp, N, p.Np, xscale, nullptr, word, list, base + p.g_at, gscale, s));
    if (gx) {
        F32Args a = {};
        a.xp = base + p.g_at;
        a.wf = base + p.bw_at;
        a.scale = gscale;
        a.wscale = wscale;
        a.y = gx;
        a.M = M;
        a.N = (int)K;
        a.KS = (int)(p.Np / 32);
        a.wf_bytes = (int)p.bwf_bytes;
        RPFQ_TRY(f32_gemm(a, s));
        e.gx.a = gy;
        e.gx.b = w;
        e.gx.out = gx;
        e.gx.list = list;
        e.gx.lda = N;
        e.gx.ldb = K;
        e.gx.I = M;
        e.gx.J = (int)K;
        exact = e.gx_blocks = exact_blocks(M, K);
    }
    if (gw) {
        RPFQ_TRY(split_rows<2>(x, M, p.Mp, K, p.Kp, xscale, gscale, word, nullptr, base + p.bx_at, nullptr, s));
        static std::atomic<uint64_t> attr_done{0};
        RPFQ_TRY(set_lds_attr_once(reinterpret_cast<const void*>(&f32_gw_kernel), kGwLds, attr_done));
        F32GwArgs g = {};
        g.gp = base + p.g_at;
        g.xp = base + p.bx_at;
        g.word = word;
        g.part = p.splits > 1 ? reinterpret_cast<float*>(base + p.part_at) : gw;
        g.ldg = p.Np * 4;
        g.ldx = p.Kp * 4;
        g.N = (int)N;
        g.K = (int)K;
        g.steps = p.steps;
        g.per = (p.steps + p.splits - 1) / p.splits;
        g.tiles_n = (int)((N + 127) / 128);
        g.tiles_k = (int)((K + 255) / 256);
        g.splits = p.splits;
        hipLaunchKernelGGL(f32_gw_kernel, dim3(g.tiles_n * g.tiles_k * g.splits), dim3(256), kGwLds, s, g);
        RPFQ_TRY(hipGetLastError());
        e.gw.a = gy;
        e.gw.b = x;
        e.gw.out = g.part;
        e.gw.lda = N;
        e.gw.ldb = K;
        e.gw.I = N;
        e.gw.J = (int)K;
        e.per = (int64_t)g.per * 16;
        exact += (int)(((N + 127) / 128) * ((K + 127) / 128)) * p.splits;
    }
    hipLaunchKernelGGL(f32_exact_grad_kernel, dim3((unsigned)exact), dim3(256), 0, s, e);
    RPFQ_TRY(hipGetLastError());
    if (gw && p.splits > 1) {
        const int64_t n4 = N * K / 4;
        const int grid = (int)((n4 + 255) / 256 < 2048 ? (n4 + 255) / 256 : 2048);
        hipLaunchKernelGGL(f32_gw_reduce_kernel, dim3(grid), dim3(256), 0, s,
                           (const float*)reinterpret_cast<float*>(base + p.part_at), n4, p.splits, (const F32Words*)word, gw);
        RPFQ_TRY(hipGetLastError());
    }
    return hipSuccess;
}

}  // namespace rpfq
