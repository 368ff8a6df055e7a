// Widely-linear layer and its input gradient for many rows of fp16: the
// packed weight is decoded once per call into the matrix cores' operand
// fragments, and a GEMM without a decode runs on them.
#include <type_traits>

#include "rpfq_device.h"

namespace rpfq {

// ---------------------------------------------------------------------------
// decode: packed blob -> fragments
// ---------------------------------------------------------------------------
// frag[rows / 32][t][lane][8 fp16], t = 8 columns of the contraction's complex
// index: lane (r, g) of a 32-row tile holds row r, columns 8 t .. 8 t + 7 of
// the re (g = 0) or im (g = 1) half -- the A operand of
// v_mfma_f32_32x32x16_f16 in the packed DMA kernel's k order, so both kernels
// give the same bits.  TRANS = 0: rows are the 2N' outputs (re, then im),
// contraction K'; 1: rows the 2K' inputs, contraction N'.  Half a workgroup
// decodes one 1-KB code block (32 rows x 32 columns) with its LUT in LDS;
// every coefficient is fuse_h of the fp16 U and W entries, as everywhere.
// Writes 8 bytes per byte of codes; ~4 us for ViT-B fc1's 590 KB.
template <int CB, int TRANS>
__global__ void __launch_bounds__(256) dense_decode_kernel(const uint32_t* codes, const float4* params, RotParams rot,
                                                          int N, int K, int NT, int KS, int nblk, int block_ks,
                                                          uint4* frag) {
    __shared__ uint32_t lut[2][32][33];   // [half][row][16 U, 16 W] fp16 (re, im)
    __shared__ uint32_t blk[2][32][9];    // the code block, a row's 8 dwords
    const int tid = threadIdx.x, h = tid >> 7, t = tid & 127;
    const int nt = blockIdx.y, ks = blockIdx.x * 2 + h;
    const bool on = ks < KS;
    if (on) {
        const int r = t & 31, q = t >> 5;  // entries 8 q .. 8 q + 7 of row r
        const int64_t n = (int64_t)nt * 32 + r;
        float4 p = make_float4(0, 0, 0, 0);
        if constexpr (CB != RPFQ_CB_TABLE) p = params[(n * nblk + ks / block_ks) * 2 + (q >> 1)];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int idx = (8 * q + e) & 15;
            float2 v;
            if constexpr (CB == RPFQ_CB_TABLE)
                v = reinterpret_cast<const float2*>(params)[n * 32 + 8 * q + e];
            else
                v = lut_entry<CB>((uint32_t)idx, p);
            if (rot.rotate) v = q < 2 ? derotate(v, rot.cu, rot.su) : derotate(v, rot.cw, rot.sw);
            lut[h][r][8 * q + e] = cvt_pk(v.x, v.y);
        }
        const uint32_t* src = codes + ((int64_t)nt * KS + ks) * 256;
        blk[h][t >> 3][t & 7] = src[t];
        blk[h][16 + (t >> 3)][t & 7] = src[128 + t];
    }
    __syncthreads();
    if (!on) return;
    const int r = t & 31, s = t >> 5;
    uint32_t p1[8], p2[8];  // (A11, A12), (A21, A22) of 8 complex elements
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        // byte 16 g + 4 s' + e' of a row is column 8 s' + 4 g + e'
        const int row = TRANS ? 8 * s + e : r, col = TRANS ? r : 8 * s + e;
        const uint32_t word = blk[h][row][4 * ((col >> 2) & 1) + (col >> 3)];
        const uint32_t c = (word >> (8 * (col & 3))) & 0xffu;
        fuse_h(lut[h][row][c & 15u], lut[h][row][16u + (c >> 4)], p1[e], p2[e]);
    }
    auto half = [&](const uint32_t (&p)[8], bool hi) {
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            o[e] = __builtin_amdgcn_perm(p[2 * e + 1], p[2 * e], hi ? 0x07060302u : 0x05040100u);
        return make_uint4(o[0], o[1], o[2], o[3]);
    };
    const uint4 a11 = half(p1, false), a12 = half(p1, true), a21 = half(p2, false), a22 = half(p2, true);
    const int rows = TRANS ? K : N, i = (TRANS ? ks : nt) * 32 + r, kt = 4 * (TRANS ? NT : KS);
    const int at = 4 * (TRANS ? nt : ks) + s;
    if (i >= rows) return;
    auto put = [&](int row, const uint4 re, const uint4 im) {
        uint4* d = frag + ((int64_t)(row >> 5) * kt + at) * 64 + (row & 31);
        d[0] = re;
        d[32] = im;
    };
    put(i, a11, TRANS ? a21 : a12);
    put(rows + i, TRANS ? a12 : a21, a22);
}

// ---------------------------------------------------------------------------
// GEMM
// ---------------------------------------------------------------------------
struct DenseArgs {
    const char* x;       // [M, 64 KS] fp16: re half, im half
    const void* frag;
    const float* xs;     // row scales to undo, or NULL
    const float* bias;   // [N] or NULL
    const void* res;     // [M, N] of y's dtype or NULL (may be y)
    void* y;             // [M, N]
    int64_t M;
    int N, KS;           // outputs, 32-column steps
    int frag_bytes;
    int tiles_m, tiles_n, group;
};

// Workgroup = 4 waves, tile = BM rows x 256 outputs, wave w the outputs
// 64 w .. 64 w + 63.  As in the packed DMA kernel the rows go global -> LDS by
// DMA (3 stages, two steps ahead, same swizzle and k order) and two
// workgroups share a CU; here the wave's fragments go straight from L2 to
// registers, 4 substeps ahead, and the tile leaves wave by wave through LDS
// as float32 (32 rows x 64 outputs at a time), so no barrier holds the other
// waves in the epilogue and the GELU of one workgroup runs beside the other's
// MFMAs.  Tiles go in groups of `group` column tiles, whose fragments stay in
// each XCD's L2 (fc1's 4.7 MB in one sweep do not: 270 against 248 us).
// 50,432 rows fp16, packed DMA kernel -> decode + this, us: fc1 + GELU 360 ->
// 330, qkv 212 -> 207, proj 80 -> 81, fc1 281 -> 273, fc2 264 -> 262; float32
// proj + residual 263 -> 157.  Input gradient, adjoint kernel -> this: fp16
// fc1 308 -> 235, fc2 338 -> 249, float32 fc1 516 -> 401.  Power bounds the
// large launches: with zero operands the same qkv launch takes 158 of 205 us.
constexpr int kDenseEpi = 8192;
template <int MB> constexpr int dense_lds() { return 3 * MB * 4096 + 4 * kDenseEpi; }
static_assert(2 * dense_lds<4>() <= 160 * 1024, "two workgroups per CU");
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

template <int MB, int YDT, int ACT>
__global__ void __launch_bounds__(256, 2) wide_dense_kernel(DenseArgs a) {
    extern __shared__ __align__(16) char smem[];
    constexpr int BM = 32 * MB, RPW = BM / 4, XL = RPW / 8;
    constexpr int STAGE = BM * 128;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    char* epi = smem + 3 * STAGE + wave * kDenseEpi;
    const int64_t ld = (int64_t)a.KS * 128;
    const int kt = 4 * a.KS;
    // wave w fills rows RPW w .. of a stage, 8 rows a load: lane l writes row
    // l >> 3, slot l & 7, which holds chunk (l & 7) ^ ((row >> 1) & 7)
    uint32_t v0, v1;
    {
        const int par = (XL * wave) & 1;
        const int c0 = (lane & 7) ^ ((4 * par + (lane >> 4)) & 7), c1 = (lane & 7) ^ ((4 * (par ^ 1) + (lane >> 4)) & 7);
        v0 = (uint32_t)((lane >> 3) * ld + (c0 >> 2) * (ld / 2) + (c0 & 3) * 16);
        v1 = (uint32_t)((lane >> 3) * ld + (c1 >> 2) * (ld / 2) + (c1 & 3) * 16);
    }
    const uint32_t lds_x = lds_addr(smem) + RPW * wave * 128;
    const char* xw = nullptr;
    auto issue_x = [&](int ks, int st) {
        const char* src = xw + ks * 64;
#pragma unroll
        for (int j = 0; j < XL; ++j) dma_dwordx4(src + 8 * j * ld, j & 1 ? v1 : v0, lds_x + st * STAGE + j * 1024);
    };
    // buffer loads: one resource and a scalar offset per load (pointers per
    // load would hold ~50 registers through the loop)
    const __amdgpu_buffer_rsrc_t frag = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.frag), 0, a.frag_bytes, 0x00027000);
    const uint32_t fv = lane * 16;
    uint32_t fo[2] = {0, 0};
    auto load_w = [&](int t, uint4 (&f)[2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            f[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(frag, fv, fo[j] + t * 1024, 0));
    };
    uint32_t aoff[4];  // chunk 4 g + s of row r
#pragma unroll
    for (int s = 0; s < 4; ++s) aoff[s] = lds_addr(smem) + r * 128 + (((4 * g + s) ^ ((r >> 1) & 7)) * 16);
    const int total = a.tiles_m * a.tiles_n;
    auto set_tile = [&](int vb, int& mt, int& ntl) {
        group_tile(xcd_tile(vb, total), a.tiles_m, a.tiles_n, a.group, mt, ntl);
        xw = a.x + (min((int64_t)mt * BM, a.M - BM) + RPW * wave) * ld;
#pragma unroll
        for (int j = 0; j < 2; ++j) fo[j] = (uint32_t)__builtin_amdgcn_readfirstlane(((ntl * 4 + wave) * 2 + j) * kt * 1024);
    };
    uint4 w[4][2];
    auto start = [&]() {
        issue_x(0, 0);
        if (a.KS > 1) issue_x(1, 1);
#pragma unroll
        for (int s = 0; s < 4; ++s) load_w(s, w[s]);
    };
    int mt, ntl;
    set_tile(blockIdx.x, mt, ntl);
    start();
    for (int vb = blockIdx.x; vb < total; vb += gridDim.x) {
        // the last row tile ends at row M; rows below m_own are the tile's before it
        const int64_t m0 = min((int64_t)mt * BM, a.M - BM), m_own = (int64_t)mt * BM;
        const int64_t n0 = (int64_t)ntl * 256 + 64 * wave;
        float inv[MB];
#pragma unroll
        for (int i = 0; i < MB; ++i) inv[i] = a.xs ? a.xs[m0 + 32 * i + r] : 1.0f;
        floatx16 acc[2][MB];
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[0][i] = acc[1][i] = floatx16{0};
        // this tile's first loads landed (the first tile: here; later ones: before the stores below)
        if (vb == (int)blockIdx.x) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        auto kstep = [&](int ks, int st) {
            const bool more = ks + 2 < a.KS;
            half8 xc[MB];
#pragma unroll
            for (int i = 0; i < MB; ++i) xc[i] = *((lds_h8_t)aoff[0] + (st * STAGE + i * 4096) / 16);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                half8 xn[MB];
                if (s < 3) {
#pragma unroll
                    for (int i = 0; i < MB; ++i) xn[i] = *((lds_h8_t)aoff[s + 1] + (st * STAGE + i * 4096) / 16);
                }
                const half8 h0 = as_half8(w[s][0]), h1 = as_half8(w[s][1]);
#pragma unroll
                for (int i = 0; i < MB; ++i) {
                    acc[0][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(h0, xc[i], acc[0][i], 0, 0, 0);
                    acc[1][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(h1, xc[i], acc[1][i], 0, 0, 0);
                }
                if (s == 0 && more) issue_x(ks + 2, (st + 2) % 3);
                load_w(ks + 1 < a.KS ? 4 * (ks + 1) + s : s, w[s]);
                if (s < 3) {
#pragma unroll
                    for (int i = 0; i < MB; ++i) xc[i] = xn[i];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
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
            kstep(ks, 0);
            kstep(ks + 1, 1);
            kstep(ks + 2, 2);
        }
        if (ks < a.KS) kstep(ks, 0);
        if (ks + 1 < a.KS) kstep(ks + 1, 1);
        if (vb + (int)gridDim.x < total) {  // the next tile's first loads
            set_tile(vb + (int)gridDim.x, mt, ntl);
            start();
        }
        // opaque lane: the epilogue's addresses are formed here and not held through the loop
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int er = ln & 31, eg = ln >> 5, c = ln & 15, row4 = ln >> 4;
        const int64_t n = n0 + 4 * c;
        const bool n_ok = n < a.N;
        f32x4 b = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        if (a.bias && n_ok) b = (f32x4){a.bias[n], a.bias[n + 1], a.bias[n + 2], a.bias[n + 3]};
        using chunk = typename std::conditional<YDT == RPFQ_F32, f32x4, u32x2>::type;  // 4 outputs
        const chunk* res = reinterpret_cast<const chunk*>(a.res);
        chunk* y = reinterpret_cast<chunk*>(a.y);
        const int64_t n4 = n >> 2, ld4 = a.N >> 2;
        // residual chunks are requested a block of rows ahead of the stores
        // (float32: with the block, two blocks of 32 registers would spill)
        constexpr bool AHEAD = YDT != RPFQ_F32;
        chunk rc[8] = {}, rn[8] = {};
        auto load_res = [&](int i, chunk (&d)[8]) {
            if (ACT != 0 || !res) return;
#pragma unroll
            for (int j = 0; j < 8; ++j) d[j] = n_ok ? res[(m0 + 32 * i + 4 * j + row4) * ld4 + n4] : chunk{};
        };
        if (AHEAD) load_res(0, rc);
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            if (!AHEAD) load_res(i, rc);
            if (AHEAD && i + 1 < MB) load_res(i + 1, rn);
            const float f = a.xs ? row_unscale(inv[i]) : 1.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                *reinterpret_cast<f32x4*>(epi + er * 256 + (((2 * q + eg) ^ (er & 15)) * 16)) =
                    (f32x4){acc[0][i][4 * q] * f, acc[0][i][4 * q + 1] * f, acc[0][i][4 * q + 2] * f, acc[0][i][4 * q + 3] * f};
                *reinterpret_cast<f32x4*>(epi + er * 256 + (((8 + 2 * q + eg) ^ (er & 15)) * 16)) =
                    (f32x4){acc[1][i][4 * q] * f, acc[1][i][4 * q + 1] * f, acc[1][i][4 * q + 2] * f, acc[1][i][4 * q + 3] * f};
            }
            if (i == 0)
                asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            else
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int row = 4 * j + row4;
                f32x4 v = *reinterpret_cast<const f32x4*>(epi + row * 256 + ((c ^ (row & 15)) * 16)) + b;
                const int64_t m = m0 + 32 * i + row;
                chunk o;
                if constexpr (YDT == RPFQ_F32) {
                    if constexpr (ACT != 0) {
#pragma unroll
                        for (int t = 0; t < 4; ++t) v[t] = gelu_fast(v[t]);
                    }
                    o = ACT == 0 && res ? rc[j] + v : v;
                } else {
                    constexpr bool f16 = YDT == RPFQ_F16;
                    o[0] = f16 ? cvt_pk(v[0], v[1]) : pack_bf2(v[0], v[1]);
                    o[1] = f16 ? cvt_pk(v[2], v[3]) : pack_bf2(v[2], v[3]);
                    if constexpr (ACT != 0) {
                        o[0] = gelu2_y(o[0], f16);
                        o[1] = gelu2_y(o[1], f16);
                    } else if (res) {
                        o[0] = add2_y(o[0], rc[j][0], f16);
                        o[1] = add2_y(o[1], rc[j][1], f16);
                    }
                }
                if (m >= m_own && n_ok) y[m * ld4 + n4] = o;
            }
            if (AHEAD && i + 1 < MB) {
#pragma unroll
                for (int j = 0; j < 8; ++j) rc[j] = rn[j];
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// ---------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------
size_t wide_dense_bytes(const WideGeom& g, int trans) {
    const int64_t rows = 2 * (trans ? g.K : g.N), con = trans ? g.NT : g.KS;
    return (size_t)((rows + 255) / 256 * 8) * (size_t)con * 4096;
}

template <int CB>
static hipError_t decode_cb(const rpfq_wide_desc& d, const WideGeom& g, const void* packed, int trans, void* frag,
                            hipStream_t s) {
    const dim3 grid((unsigned)((g.KS + 1) / 2), (unsigned)g.NT);
    const uint32_t* codes = reinterpret_cast<const uint32_t*>(packed);
    const float4* params = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(packed) + g.codes_bytes);
    if (trans)
        hipLaunchKernelGGL((dense_decode_kernel<CB, 1>), grid, dim3(256), 0, s, codes, params, rot_of(d), (int)g.N, (int)g.K,
                           (int)g.NT, (int)g.KS, (int)g.nblk, (int)g.block_ks, reinterpret_cast<uint4*>(frag));
    else
        hipLaunchKernelGGL((dense_decode_kernel<CB, 0>), grid, dim3(256), 0, s, codes, params, rot_of(d), (int)g.N, (int)g.K,
                           (int)g.NT, (int)g.KS, (int)g.nblk, (int)g.block_ks, reinterpret_cast<uint4*>(frag));
    return hipGetLastError();
}

template <int MB, int YDT, int ACT>
static hipError_t dense_go(DenseArgs& a, hipStream_t s) {
    static std::atomic<uint64_t> attr_done{0};
    const hipError_t e = set_lds_attr_once(reinterpret_cast<const void*>(&wide_dense_kernel<MB, YDT, ACT>), dense_lds<MB>(),
                                           attr_done);
    if (e != hipSuccess) return e;
    a.tiles_m = (int)((a.M + 32 * MB - 1) / (32 * MB));
    a.tiles_n = (a.N + 255) / 256;
    a.group = tile_group(a.tiles_n, (int64_t)a.KS * 32768);
    const int total = a.tiles_m * a.tiles_n, slots = 2 * device_cus();
    hipLaunchKernelGGL((wide_dense_kernel<MB, YDT, ACT>), dim3(total < slots ? total : slots), dim3(256), dense_lds<MB>(), s, a);
    return hipGetLastError();
}

template <int YDT, int ACT>
static hipError_t dense_mb(DenseArgs& a, hipStream_t s) {
    const int mb = rows_per_tile(a.M, a.N);
    if (mb == 2) return dense_go<2, YDT, ACT>(a, s);
    if (mb == 3) return dense_go<3, YDT, ACT>(a, s);
    return dense_go<4, YDT, ACT>(a, s);
}

template <int YDT>
static hipError_t dense_y(DenseArgs& a, int act, hipStream_t s) {
    return act ? dense_mb<YDT, 1>(a, s) : dense_mb<YDT, 0>(a, s);
}

hipError_t launch_wide_dense(const rpfq_wide_desc& d, const WideGeom& g, const void* packed, int trans, const void* x,
                             int64_t M, const float* xs, const float* bias, const void* res, void* y, int ydt, int act,
                             void* work, hipStream_t s) {
    hipError_t e;
    switch (d.codebook) {
        case RPFQ_CB_SIGN: e = decode_cb<RPFQ_CB_SIGN>(d, g, packed, trans, work, s); break;
        case RPFQ_CB_PSK16: e = decode_cb<RPFQ_CB_PSK16>(d, g, packed, trans, work, s); break;
        case RPFQ_CB_TABLE: e = decode_cb<RPFQ_CB_TABLE>(d, g, packed, trans, work, s); break;
        default: e = decode_cb<RPFQ_CB_AXIS>(d, g, packed, trans, work, s); break;
    }
    if (e != hipSuccess) return e;
    DenseArgs a = {};
    a.x = reinterpret_cast<const char*>(x);
    a.frag = work;
    a.xs = xs;
    a.bias = bias;
    a.res = res;
    a.y = y;
    a.M = M;
    a.N = (int)(2 * (trans ? g.K : g.N));
    a.KS = (int)(trans ? g.NT : g.KS);
    a.frag_bytes = (int)wide_dense_bytes(g, trans);
    switch (ydt) {
        case RPFQ_F32: return dense_y<RPFQ_F32>(a, act, s);
        case RPFQ_F16: return dense_y<RPFQ_F16>(a, act, s);
        default: return dense_y<RPFQ_BF16>(a, act, s);
    }
}

}  // namespace rpfq
