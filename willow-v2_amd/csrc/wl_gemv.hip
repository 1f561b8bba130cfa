// Quantized matrix times a few tokens: y[t, r] = W[r, :] . x[t, :] (wl_gemv, wl_gemv_dtype). Replaces the Metal kernel
// gemv_<T> (gguf/metal.py:189-215).
#include <hip/hip_runtime.h>

#include "wl_common.h"
#include "wl_host.h"

namespace wl {

// A lane's two 16-value runs of a block as exact f16 pairs (values 0 and 2 of each packed word in e, 1 and 3 in o),
// which v_fma_mix_f32 reads directly. A pair is one byte permute (each byte under 0x64: 1024 + q) and one packed
// subtraction, made once per block and used for every token, in half the registers that fp32 values take. The values
// are q itself, not q 2^-24 (the raw field as an f16 subnormal, one instruction less): products with |x| < 2^-102
// would be fp32 subnormals and lose bits (|x| near 1e-36: error 6e-4).
template <int TYPE>
struct HalfRuns {
    wl_f16x2 e_lo[4], o_lo[4], e_hi[4], o_hi[4];
    float a_lo, a_hi, b_lo, b_hi;
    template <int FIRST>
    static __device__ __forceinline__ wl_f16x2 pair(uint32_t w) {  // bytes FIRST and FIRST + 2
        const uint32_t v = __builtin_amdgcn_perm(0x64646464u, w, FIRST == 0 ? 0x04020400u : 0x04030401u);
        return __builtin_bit_cast(wl_f16x2, v) - static_cast<_Float16>(1024.0f);
    }
    __device__ __forceinline__ void set(const RawLane<TYPE>& raw, int c) {
        Lane32 l;
        raw.unpack(c, l);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            e_lo[i] = pair<0>(l.lo[i]);
            o_lo[i] = pair<1>(l.lo[i]);
            e_hi[i] = pair<0>(l.hi[i]);
            o_hi[i] = pair<1>(l.hi[i]);
        }
        a_lo = l.a_lo;
        a_hi = l.a_hi;
        b_lo = l.b_lo;
        b_hi = l.b_hi;
    }
    static __device__ __forceinline__ float dot(const wl_f16x2 (&e)[4], const wl_f16x2 (&o)[4], const float4 (&x)[4]) {
        float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            s0 = __builtin_fmaf(static_cast<float>(e[i].x), x[i].x, s0);
            s1 = __builtin_fmaf(static_cast<float>(o[i].x), x[i].y, s1);
            s0 = __builtin_fmaf(static_cast<float>(e[i].y), x[i].z, s0);
            s1 = __builtin_fmaf(static_cast<float>(o[i].y), x[i].w, s1);
        }
        return s0 + s1;
    }
    // the lane's share of the block's product with x (its two runs, their sums known)
    __device__ __forceinline__ float run(const float4 (&xl)[4], const float4 (&xh)[4], float sxl, float sxh) const {
        return a_lo * dot(e_lo, o_lo, xl) + b_lo * sxl + a_hi * dot(e_hi, o_hi, xh) + b_hi * sxh;
    }
};

__device__ __forceinline__ void load_run16(const float* __restrict__ p, float4 (&x)[4]) { load_run(p, x); }
__device__ __forceinline__ void load_run16(const uint16_t* __restrict__ p, float4 (&x)[4]) {
    const uint4* q = reinterpret_cast<const uint4*>(p);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint4 v = q[i];
        x[2 * i] = make_float4(__builtin_bit_cast(float, v.x << 16), __builtin_bit_cast(float, v.x & 0xFFFF0000u),
                               __builtin_bit_cast(float, v.y << 16), __builtin_bit_cast(float, v.y & 0xFFFF0000u));
        x[2 * i + 1] = make_float4(__builtin_bit_cast(float, v.z << 16), __builtin_bit_cast(float, v.z & 0xFFFF0000u),
                                   __builtin_bit_cast(float, v.w << 16), __builtin_bit_cast(float, v.w & 0xFFFF0000u));
    }
}

// a summed over lanes l and l ^ 32 in the low half of the wavefront, b in the high half: one swap and one add for
// two values (swap_add spends them on one)
__device__ __forceinline__ float pair_add32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    return __builtin_bit_cast(float, static_cast<uint32_t>(r[0])) +
           __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}
// the same over lanes l and l ^ 16: a in the even rows of 16 lanes, b in the odd ones
__device__ __forceinline__ float pair_add16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    return __builtin_bit_cast(float, static_cast<uint32_t>(r[0])) +
           __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}

// v[0 .. 3] each summed over the wavefront: row i of 16 lanes returns v[i]'s sum. Every level adds as group_sum<64>
// does (addition commutes exactly), so the bits are its; the last two levels take one swap and one add for two values.
__device__ __forceinline__ float quad_sum(const float (&v)[4]) {
    float u[4];
#pragma unroll
    for (int i = 0; i < 4; i++) u[i] = group_sum<16>(v[i]);
    return pair_add32(pair_add16(u[0], u[1]), pair_add16(u[2], u[3]));
}

// The matrix times TT tokens (1 .. 8). A block belongs to 8 lanes (wl_common.h), 2^ks blocks of a row to a
// wavefront pass; a wavefront holds R rows in each of its 8 >> ks lane groups, and kw of the workgroup's 4
// wavefronts split the blocks of longer rows, 8 kw to a round (MORE: more than one round, more than 32 blocks a
// row; apart, because its loop costs every shorter row registers). The lane's x runs come straight from global
// memory (L2 and L1 hold them) and serve R rows each.
// Every sum is added as k_gemv_batch adds it (wl_quant.hip): a lane its blocks slot, slot + 8, ... in order, then
// the lanes, so a matrix gives the same bits alone and among batched experts, however its blocks are split. With kw
// > 1 a round's products meet in LDS, lane by lane, in quads of values, Q of them, and each wavefront adds up and
// reduces its share: with kw = 2 a wavefront hands over the quads that it does not finish itself ([2][Q][64] of
// LDS), with kw = 4 all of them ([4][Q][64], and [Q][64] running sums when MORE). Both that way with kw = 2 took
// 12.0 us where this takes 10.9, as sums reduced before they meet, in another order, did (Q4_K 4096 x 2560, 8
// tokens of bf16).
// What bounds it: at 8 tokens the x reads (a lane's 64-byte runs, 64 bytes apart) and the rows they are read for,
// which is why a lane group holds several; at one token the launch and one trip to memory.
// Measured per call in a graph (bf16 in and out; before: a row per wavefront, its x read again for every row, and a
// converting launch on each side): Q4_K 4096 x 2048 at 1 token 8.5 -> 4.2 us, 8 tokens 21.8 -> 7.6; Q6_K 2048 x
// 4096 9.6 -> 4.4 and 22.2 -> 8.2, 8 tokens of fp32 18.1 -> 8.5; Q4_K 2048 x 512 6.5 -> 3.0 and 10.6 -> 5.1.
template <int TYPE, int TT, int R, typename XT, bool MORE>
__global__ __launch_bounds__(256) void k_gemv(const uint8_t* __restrict__ w, int rows, int nb, int64_t row_stride,
                                              const XT* __restrict__ x, int64_t ldx, void* __restrict__ y,
                                              int64_t ldy, int y_bf16, int ks, int kw) {
    constexpr int N = TT * R, Q = (N + 3) / 4;  // a lane's values, t R + r, and quads of them
    extern __shared__ __attribute__((aligned(16))) float4 lds[];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int g = lane >> 3, c = lane & 7;
    const int slot = g & ((1 << ks) - 1), sub = g >> ks, subs = 8 >> ks;
    const int kwi = wv % kw, rset = wv / kw;
    const int row0 = (static_cast<int>(blockIdx.x) * (4 / kw) + rset) * subs * R + sub * R;
    const int lo_start = BlockInfo<TYPE>::lo_start(c);
    const uint8_t* rp[R];
#pragma unroll
    for (int r = 0; r < R; r++) rp[r] = w + static_cast<int64_t>(min(row0 + r, rows - 1)) * row_stride;
    float d[N];
#pragma unroll
    for (int n = 0; n < N; n++) d[n] = 0.0f;
    auto add_block = [&](int kb) {  // the lane's products of block kb
        RawLane<TYPE> raw[R];
#pragma unroll
        for (int r = 0; r < R; r++) raw[r].fetch(rp[r] + static_cast<int64_t>(kb) * BlockInfo<TYPE>::bytes, c);
        const XT* xk = x + kb * kQK + lo_start;
        HalfRuns<TYPE> h[R];
#pragma unroll
        for (int r = 0; r < R; r++) h[r].set(raw[r], c);
#pragma unroll
        for (int t = 0; t < TT; t++) {
            float4 xl[4], xh[4];
            load_run16(xk + t * ldx, xl);
            load_run16(xk + t * ldx + BlockInfo<TYPE>::hi_offset, xh);
            const float sxl = sum16(xl), sxh = sum16(xh);
#pragma unroll
            for (int r = 0; r < R; r++) d[t * R + r] += h[r].run(xl, xh, sxl, sxh);
        }
    };
    auto store = [&](int n, float v) {
        const int row = row0 + n % R;
        if (row >= rows) return;
        const int64_t at = (n / R) * ldy + row;
        if (y_bf16)
            static_cast<uint16_t*>(y)[at] = static_cast<uint16_t>(f32_to_bf16_bits(v));
        else
            static_cast<float*>(y)[at] = v;
    };
    auto quad = [&](int i) {
        return make_float4(d[4 * i], 4 * i + 1 < N ? d[4 * i + 1] : 0.0f, 4 * i + 2 < N ? d[4 * i + 2] : 0.0f,
                           4 * i + 3 < N ? d[4 * i + 3] : 0.0f);
    };
    auto finish = [&](int i, const float4& s) {  // quad i's lanes added and stored
        const float v[4] = {s.x, s.y, s.z, s.w};
        const float sum = quad_sum(v);
        const int n = 4 * i + (lane >> 4);
        if ((lane & 15) == 0 && n < N) store(n, sum);
    };
    if (8 * kwi + slot < nb) add_block(8 * kwi + slot);
    if (kw == 1) {
        if (ks == 3) {
#pragma unroll
            for (int i = 0; i < Q; i++) finish(i, quad(i));
        } else {
#pragma unroll
            for (int n = 0; n < N; n++) {
                float s = group_sum<8>(d[n]);
                if (ks >= 1) s += dpp<0x140>(s);
                if (ks >= 2) s = swap_add<16>(s);
                if ((lane & ((8 << ks) - 1)) == 0) store(n, s);
            }
        }
    } else if (kw == 2) {
        constexpr int Q0 = (Q + 1) / 2;  // wavefront 0 finishes quads 0 .. Q0 - 1
        float4* area = lds + rset * Q * 64 + lane;
        if (kwi == 0) {
#pragma unroll
            for (int i = Q0; i < Q; i++) area[i * 64] = quad(i);
        } else {
#pragma unroll
            for (int i = 0; i < Q0; i++) area[i * 64] = quad(i);
        }
        __syncthreads();
        auto finish_both = [&](int i) {
            const float4 a = quad(i), b = area[i * 64];
            finish(i, make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w));  // neither is -0: d starts from 0
        };
        if (kwi == 0) {
#pragma unroll
            for (int i = 0; i < Q0; i++) finish_both(i);
        } else {
#pragma unroll
            for (int i = Q0; i < Q; i++) finish_both(i);
        }
    } else {
        const float4* part = lds + lane;
        float4* mine = lds + wv * Q * 64 + lane;
        float4* run = lds + 4 * Q * 64 + lane;
        for (int kb0 = 32;; kb0 += 32) {
#pragma unroll
            for (int i = 0; i < Q; i++) mine[i * 64] = quad(i);
            __syncthreads();
            const bool last = !MORE || kb0 >= nb;
            for (int i = wv; i < Q; i += 4) {
                float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (MORE && kb0 > 32) s = run[i * 64];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float4 p = part[(j * Q + i) * 64];
                    s = make_float4(s.x + p.x, s.y + p.y, s.z + p.z, s.w + p.w);
                }
                if (last)
                    finish(i, s);
                else
                    run[i * 64] = s;
            }
            if (last) return;
#pragma unroll
            for (int n = 0; n < N; n++) d[n] = 0.0f;
            const int kb = kb0 + 8 * wv + slot;
            if (kb < nb) add_block(kb);
            __syncthreads();  // the round's products are read
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// Host side

struct GemvCall {
    const uint8_t* w;
    int rows, nb;
    int64_t row_stride;
    int64_t k;
    int y_bf16;
    hipStream_t s;
};

template <int TYPE, int TT, int R, typename XT>
static void launch_gemv_r(const GemvCall& g, const XT* x, void* y, int ks, int kw) {
    const int rows_wg = 4 / kw * (8 >> ks) * R;
    const unsigned grid = static_cast<unsigned>((g.rows + rows_wg - 1) / rows_wg);
    constexpr int Q = (TT * R + 3) / 4;
    const bool more = g.nb > 32;
    const size_t lds = kw == 1 ? 0 : static_cast<size_t>(kw == 2 ? 2 : more ? 5 : 4) * Q * 64 * sizeof(float4);
    auto kernel = more ? k_gemv<TYPE, TT, R, XT, true> : k_gemv<TYPE, TT, R, XT, false>;
    kernel<<<grid, 256, lds, g.s>>>(g.w, g.rows, g.nb, g.row_stride, x, g.k, y, g.rows, g.y_bf16, ks, kw);
}

template <int TYPE, int TT, typename XT>
static void launch_gemv_t(const GemvCall& g, const XT* x, void* y) {
    const int ks = g.nb > 4 ? 3 : g.nb > 2 ? 2 : g.nb > 1 ? 1 : 0;
    const int kw = g.nb <= 8 ? 1 : g.nb <= 16 ? 2 : 4;
    // Rows per lane group, by the workgroups that one row each would make: more rows reuse each x read, fewer leave
    // more workgroups (us with 1 / 2 / 4 rows below; workgroups in brackets). fp32 x: one workgroup to a CU, so two
    // rows above 256 and four above 512 (Q4_K, 8 tokens, 1500 x 2048 [375] 9.7 / 6.7 / 7.7, 3000 x 1536 [750] 12.1
    // / 9.5 / 7.6); one token reads x least, four above 1536 (4096 x 2048 [1024] 4.85 / 4.18 / 4.14, 6000 x 2048
    // [1500] 5.9 / 4.9 / 5.3, 151936 x 2048 84 / 52 / 48). bf16 x, half the reads: two above 256 and four above
    // 1536 (3 tokens, 2048 x 2048 [512] 4.4 / 4.0 / 4.5, 6000 x 2048 7.9 / 6.3 / 6.6, 8192 x 2048 [2048] 9.4 / 7.4
    // / 6.8), with 7 and 8 tokens four above 512 (3000 x 1536 8.1 / 8.1 / 7.2), and for one token two above 1024,
    // four above 3072 (4096 x 2048 4.21 / 4.10 / 4.13, 6000 x 2048 4.8 / 4.7 / 5.2, 151936 x 2048 68 / 50 / 43).
    const int64_t wgs = g.rows / (4 / kw * (8 >> ks));
    constexpr bool kBf16 = sizeof(XT) == 2;
    constexpr int kTwo = kBf16 ? (TT == 1 ? 1024 : TT < 7 ? 256 : 512) : 256;
    constexpr int kFour = kBf16 ? (TT == 1 ? 3072 : TT < 7 ? 1536 : 512) : TT == 1 ? 1536 : 512;
    const int want = wgs > kFour ? 4 : wgs > kTwo ? 2 : 1;
    if (want == 4)
        launch_gemv_r<TYPE, TT, 4>(g, x, y, ks, kw);
    else if (want == 2)
        launch_gemv_r<TYPE, TT, 2>(g, x, y, ks, kw);
    else
        launch_gemv_r<TYPE, TT, 1>(g, x, y, ks, kw);
}

template <int TYPE, typename XT>
static void launch_gemv(const GemvCall& g, const XT* x, int64_t tokens, void* y) {
    for (int64_t t0 = 0; t0 < tokens; t0 += 8) {
        const XT* xt = x + t0 * g.k;
        void* yt = static_cast<char*>(y) + t0 * g.rows * (g.y_bf16 ? 2 : 4);
        switch (tokens - t0 < 8 ? tokens - t0 : 8) {
            case 1: launch_gemv_t<TYPE, 1>(g, xt, yt); break;
            case 2: launch_gemv_t<TYPE, 2>(g, xt, yt); break;
            case 3: launch_gemv_t<TYPE, 3>(g, xt, yt); break;
            case 4: launch_gemv_t<TYPE, 4>(g, xt, yt); break;
            case 5: launch_gemv_t<TYPE, 5>(g, xt, yt); break;
            case 6: launch_gemv_t<TYPE, 6>(g, xt, yt); break;
            case 7: launch_gemv_t<TYPE, 7>(g, xt, yt); break;
            default: launch_gemv_t<TYPE, 8>(g, xt, yt); break;
        }
    }
}

}  // namespace wl

using namespace wl;

extern "C" {

int wl_gemv_dtype(int type, const void* w, int64_t rows, int64_t k, int64_t row_stride, const void* x, int x_dtype,
                  int64_t tokens, void* y, int y_dtype, void* stream) {
    const int rc = check_matrix(type, w, rows, k, row_stride);
    if (rc) return rc;
    if (!x || !y) return WL_EINVAL_NULL;
    if (tokens <= 0) return WL_EINVAL_SHAPE;
    if ((x_dtype != WL_DTYPE_F32 && x_dtype != WL_DTYPE_BF16) || (y_dtype != WL_DTYPE_F32 && y_dtype != WL_DTYPE_BF16))
        return WL_EINVAL_DTYPE;
    if (reinterpret_cast<uintptr_t>(x) % 16 != 0) return WL_EINVAL_ALIGN;
    const GemvCall g{static_cast<const uint8_t*>(w), static_cast<int>(rows), static_cast<int>(k / kQK), row_stride, k,
                     y_dtype == WL_DTYPE_BF16 ? 1 : 0, static_cast<hipStream_t>(stream)};
    if (x_dtype == WL_DTYPE_BF16) {
        const uint16_t* xb = static_cast<const uint16_t*>(x);
        type == WL_TYPE_Q4_K ? launch_gemv<WL_TYPE_Q4_K>(g, xb, tokens, y)
                             : launch_gemv<WL_TYPE_Q6_K>(g, xb, tokens, y);
    } else {
        const float* xf = static_cast<const float*>(x);
        type == WL_TYPE_Q4_K ? launch_gemv<WL_TYPE_Q4_K>(g, xf, tokens, y)
                             : launch_gemv<WL_TYPE_Q6_K>(g, xf, tokens, y);
    }
    return launch_status();
}

int wl_gemv(int type, const void* w, int64_t rows, int64_t k, int64_t row_stride, const float* x, int64_t tokens,
            float* y, void* stream) {
    return wl_gemv_dtype(type, w, rows, k, row_stride, x, WL_DTYPE_F32, tokens, y, WL_DTYPE_F32, stream);
}

}  // extern "C"
