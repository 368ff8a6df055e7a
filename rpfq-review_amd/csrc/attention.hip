// Attention over short token sequences, straight from the qkv layer's output:
// out = softmax(q k^T scale) v per (image, head), the SDPA between the packed
// qkv and proj layers of a ViT block
// (RPFQ-ViTApple/scripts/audit_rpfq_vit_ios_parity.py:523-545).
#include "rpfq_device.h"

namespace rpfq {

// One workgroup of 4 waves per (image, head, part of the queries).  All K and
// V rows of the head (N <= 288 tokens of 64 values) go to LDS by DMA from the
// [B, N, 3, H, 64] tensor as it lies; each wave then takes blocks of 32
// queries.  S^T = K Q^T (v_mfma_f32_32x32x16: keys as rows), so a lane holds
// one query's scores (half of them; the other half 32 lanes away): the
// softmax is in-lane but for one exchange, and the probabilities, rounded to
// 16 bits, are already the B operand of O^T = V^T P^T: of each 16 keys lane
// half g holds keys 4 g .. 4 g + 3 and 8 + 4 g .. 8 + 4 g + 3, and
// ds_read_b64_tr_b16 gathers V's rows in that order.  Scores, maxima, sums
// and outputs are float32.
// Bound by HBM (q, k, v once, out once) and, next to it, the exponentials:
// 256 x 12 heads, 197 tokens 85 us (310 MB, 3.6 TB/s; torch's library kernel
// 172), 64 x 3 heads, 198 tokens 9 us (17).  Without the fences around each
// key block the compiler read every fragment first and spilled (141 us).
struct AttnArgs {
    const char* qkv;
    char* out;
    int N, H, parts;
    float scale2;  // scale * log2(e)
};

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s4_t;

template <bool BF>
__device__ __forceinline__ floatx16 mfma16(uint4 a, uint4 b, floatx16 c) {
    if constexpr (BF)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(as_half8(a), as_half8(b), c, 0, 0, 0);
}
template <bool BF>
__device__ __forceinline__ uint32_t pack16(float lo, float hi) {
    if constexpr (BF) return pack_bf2(lo, hi);
    return cvt_pk(lo, hi);
}

// c + lo + hi of a 16-bit pair
template <bool BF>
__device__ __forceinline__ float sum2(uint32_t v, float c) {
    if constexpr (BF) {
        typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2, v), __builtin_bit_cast(bf2, 0x3f803f80u), c, false);
    } else {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2v, v), __builtin_bit_cast(half2v, 0x3c003c00u), c, false);
    }
}

// NB: 32-key blocks (N <= 32 NB).  One block of keys is one block of queries
// too: a workgroup of one wave, so that no wave waits beside it.  49,152 heads
// of 5 tokens 39 us and of 32 tokens 189 us (on two blocks and four waves: 104
// and 225; torch's: 60 bf16, 176 fp16, and 215).
constexpr int attn_waves(int nb) { return nb == 1 ? 1 : 4; }
template <int NB, bool BF>
__global__ void __launch_bounds__(64 * attn_waves(NB), 2) attention_kernel(AttnArgs a) {
    extern __shared__ __align__(16) char smem[];
    constexpr int KV = NB * 32 * 128;  // bytes of K, then of V
    constexpr int W = attn_waves(NB);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int part = blockIdx.x % a.parts, bh = blockIdx.x / a.parts;
    const int b = bh / a.H, h = bh - b * a.H;
    const int64_t row = (int64_t)a.H * 384;  // bytes of a token: 3 H 64 values
    const char* base = a.qkv + (int64_t)b * a.N * row + h * 128;

    // DMA of 8 rows per load: lane l fills row l >> 3, slot l & 7.  K: chunk c
    // at slot c ^ ((row >> 1) & 7); V: c ^ (((row >> 1) & 1) << 2).
    // Rows past N repeat row N - 1 (K: masked below; V: zeroed below).
    for (int i = wave; i < 4 * NB; i += W) {
        const int t = 8 * i + (lane >> 3);
        const int64_t at = (int64_t)min(t, a.N - 1) * row;
        const uint32_t kc = (uint32_t)((lane & 7) ^ ((t >> 1) & 7)) * 16, vc = (uint32_t)((lane & 7) ^ (((t >> 1) & 1) << 2)) * 16;
        dma_dwordx4(base + a.H * 128, (uint32_t)at + kc, lds_addr(smem) + i * 1024);
        dma_dwordx4(base + a.H * 256, (uint32_t)at + vc, lds_addr(smem) + KV + i * 1024);
    }
    const int blocks = (a.N + 31) / 32;
    int qb = part * W + wave;
    auto load_q = [&](int blk, uint4 (&q)[4]) {  // lane (r, g): d 16 s + 8 g .. + 7 of query 32 blk + r
        const char* src = base + (int64_t)min(32 * blk + r, a.N - 1) * row + 16 * g;
#pragma unroll
        for (int s = 0; s < 4; ++s) q[s] = *reinterpret_cast<const uint4*>(src + 32 * s);
    };
    uint4 q[4];
    load_q(qb < blocks ? qb : 0, q);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // V rows past N (up to 63 of them: 65 tokens on 4 blocks): a probability of 0
    // must meet a finite value
    for (int t = a.N + (tid >> 3); t < 32 * NB; t += 8 * W)
        *reinterpret_cast<uint4*>(smem + KV + t * 128 + (tid & 7) * 16) = make_uint4(0, 0, 0, 0);
    __syncthreads();

    const int sw = (r >> 1) & 7, i16 = lane & 15, hf = (lane >> 4) & 1;
    uint32_t koff[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) koff[s] = lds_addr(smem) + r * 128 + (((2 * s + g) ^ sw) * 16);
    // V^T fragment of 16 keys, d block j: rows 4 g + i16 / 4 (+ 8), columns
    // 32 j + 16 hf + 4 (i16 & 3) .. + 3
    const int vr = 4 * g + (i16 >> 2);
    uint32_t voff[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
        voff[j] = lds_addr(smem) + KV + vr * 128 + (((4 * j + 2 * hf + ((i16 & 3) >> 1)) ^ (((vr >> 1) & 1) << 2)) * 16) + (i16 & 1) * 8;

    for (; qb < blocks; qb += W * a.parts) {
        floatx16 s[NB];
        auto read_k = [&](int kb, u32x4 (&f)[4]) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                f[t] = *reinterpret_cast<__attribute__((address_space(3))) const u32x4*>(koff[t] + kb * 4096);
        };
        u32x4 kf[4];
        read_k(0, kf);
#pragma unroll
        for (int kb = 0; kb < NB; ++kb) {  // one block's fragments ahead, and no further (registers)
            u32x4 kn[4];
            if (kb + 1 < NB) read_k(kb + 1, kn);
            s[kb] = floatx16{0};
#pragma unroll
            for (int t = 0; t < 4; ++t) s[kb] = mfma16<BF>(__builtin_bit_cast(uint4, kf[t]), q[t], s[kb]);
            if (kb + 1 < NB) {
#pragma unroll
                for (int t = 0; t < 4; ++t) kf[t] = kn[t];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // keys past N: in the last block, or the last two where NB = 4 also
        // serves N = 65 .. 96
#pragma unroll
        for (int kb = NB == 4 ? NB - 2 : NB - 1; kb < NB; ++kb) {
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (32 * kb + acc_row(v, g) >= a.N) s[kb][v] = -__builtin_inff();
        }
        float mx = s[0][0];
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
#pragma unroll
            for (int v = 0; v < 16; ++v) mx = fmaxf(mx, s[kb][v]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        // Scores far from 0: the product of the largest with scale2 is rounded,
        // and past 2^20 by enough to carry a probability out of fp16's range
        // (an inf, and NaN with it).  There the largest is subtracted first.
        const bool far = fabsf(mx) * a.scale2 > 0x1p20f;
        if (__any(far)) {
            const float sub = far ? mx : 0.0f;
#pragma unroll
            for (int kb = 0; kb < NB; ++kb)
#pragma unroll
                for (int v = 0; v < 16; ++v) s[kb][v] -= sub;
            mx -= sub;
        }
        const int next = qb + W * a.parts;
        load_q(next < blocks ? next : 0, q);
        // fp16: probabilities times 2^15, normal down to 2^-29 of the row's
        // largest, in sums below 2^39.  bf16 has float32's range and so have
        // its values: times 2^-9, so that the sum of 288 of them stays within
        // the largest value.  Undone by l, which carries the same factor.
        const float mc = mx * a.scale2 + (BF ? 9.0f : -15.0f);
        float l = 0.0f;
        floatx16 o[2];
        o[0] = o[1] = floatx16{0};
        auto read_v = [&](int k16, s16x4 (&f)[4]) {  // 16 keys: [d block][half]
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                f[2 * j] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)(voff[j] + k16 * 2048));
                f[2 * j + 1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)(voff[j] + k16 * 2048 + 1024));
            }
        };
        s16x4 vf[4];
        read_v(0, vf);
#pragma unroll
        for (int k16 = 0; k16 < 2 * NB; ++k16) {
            const int kb = k16 >> 1, u = k16 & 1;
            s16x4 vn[4];
            if (k16 + 1 < 2 * NB) read_v(k16 + 1, vn);
#pragma unroll
            for (int v = 8 * u; v < 8 * u + 8; ++v) s[kb][v] = __builtin_amdgcn_exp2f(fmaf(s[kb][v], a.scale2, -mc));
            const uint4 p = make_uint4(pack16<BF>(s[kb][8 * u], s[kb][8 * u + 1]), pack16<BF>(s[kb][8 * u + 2], s[kb][8 * u + 3]),
                                       pack16<BF>(s[kb][8 * u + 4], s[kb][8 * u + 5]), pack16<BF>(s[kb][8 * u + 6], s[kb][8 * u + 7]));
            // the sum of the rounded probabilities: their rounding errors then
            // weigh the values' distance to the output, not the values
            l = sum2<BF>(p.x, sum2<BF>(p.y, sum2<BF>(p.z, sum2<BF>(p.w, l))));
#pragma unroll
            for (int j = 0; j < 2; ++j)
                o[j] = mfma16<BF>(__builtin_bit_cast(uint4, __builtin_shufflevector(vf[2 * j], vf[2 * j + 1], 0, 1, 2, 3, 4, 5, 6, 7)), p, o[j]);
            if (k16 + 1 < 2 * NB) {
#pragma unroll
                for (int t = 0; t < 4; ++t) vf[t] = vn[t];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        l += __shfl_xor(l, 32, 64);
        const float inv = 1.0f / l;
        const int query = 32 * qb + r;
        char* dst = a.out + ((int64_t)b * a.N + query) * a.H * 128 + h * 128;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int p = 0; p < 2; ++p) {  // 8 consecutive outputs per lane: trade halves across the 32 lanes
                uint32_t x[2], y[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    x[e] = pack16<BF>(o[j][8 * p + 2 * e] * inv, o[j][8 * p + 2 * e + 1] * inv);
                    y[e] = pack16<BF>(o[j][8 * p + 4 + 2 * e] * inv, o[j][8 * p + 5 + 2 * e] * inv);
                }
                const auto s0 = __builtin_amdgcn_permlane32_swap(x[0], y[0], false, false);
                const auto s1 = __builtin_amdgcn_permlane32_swap(x[1], y[1], false, false);
                if (query < a.N)
                    *reinterpret_cast<uint4*>(dst + 64 * j + 32 * p + 16 * g) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
            }
    }
}

template <int NB, bool BF>
static hipError_t attention_go(const AttnArgs& a, int64_t heads, hipStream_t s) {
    static std::atomic<uint64_t> attr_done{0};
    constexpr int lds = 2 * NB * 32 * 128;
    const hipError_t e = set_lds_attr_once(reinterpret_cast<const void*>(&attention_kernel<NB, BF>), lds, attr_done);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((attention_kernel<NB, BF>), dim3((unsigned)(heads * a.parts)), dim3(64 * attn_waves(NB)),
                       lds, s, a);
    return hipGetLastError();
}

template <bool BF>
static hipError_t attention_nb(const AttnArgs& a, int64_t heads, hipStream_t s) {
    switch ((a.N + 31) / 32) {
        case 1: return attention_go<1, BF>(a, heads, s);
        case 2: return attention_go<2, BF>(a, heads, s);
        case 3: case 4: return attention_go<4, BF>(a, heads, s);
        case 5: return attention_go<5, BF>(a, heads, s);
        case 6: return attention_go<6, BF>(a, heads, s);
        case 7: return attention_go<7, BF>(a, heads, s);
        case 8: return attention_go<8, BF>(a, heads, s);
        default: return attention_go<9, BF>(a, heads, s);
    }
}

hipError_t launch_attention(const void* qkv, int dt, int64_t B, int64_t N, int64_t H, float scale, void* out,
                            hipStream_t s) {
    AttnArgs a = {};
    a.qkv = reinterpret_cast<const char*>(qkv);
    a.out = reinterpret_cast<char*>(out);
    a.N = (int)N;
    a.H = (int)H;
    a.scale2 = scale * 1.44269504088896340736f;
    // few heads: spread the query blocks, a block per wave, over more workgroups
    const int blocks = (int)(N + 31) / 32, most = (blocks + 3) / 4;
    a.parts = B * H * most <= 2 * device_cus() ? most : 1;
    return dt == RPFQ_BF16 ? attention_nb<true>(a, B * H, s) : attention_nb<false>(a, B * H, s);
}

}  // namespace rpfq
