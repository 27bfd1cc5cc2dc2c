// zz_matmul.hip -- the gpu.h matmul contract on gfx950: y[S,O] = W[O,I] x[S,I]
// with f32 activations and the weights in the reference's own byte layout
// (gpu.h:71-84). Numerically this is the *_dot_f32 path (q40.h:290-305,
// 443-455; tq2.h:235-252, 405-427): partial sums of small-integer x f32 products in
// fp32, scaled by the block's d, accumulated in fp32; the contract (gemma4.c:2361,
// maple.c:1813-1815) is relative error < 1e-4 against the double reference. Q4A's affine
// term m * sum(x) is a second partial.
//
// A workgroup owns MV_R weight rows and T tokens. Its 256 threads split the row by units
// of 8 weights (4 lanes a 32-weight block), so a wave's loads of weights and of x are
// contiguous and each x value loaded serves MV_R rows, each weight T tokens; the
// partial sums meet by a transposing wave reduction and LDS. Bound by latency at an
// engine's sizes. Against one wave per (row, token) whose lanes read whole blocks byte by
// byte and every token's wave the weights again, q4_0, kernel trace with other work between
// the calls: 2112 x 2816, 1 token 8.0 -> 4.9 us, 5 tokens 22.6 -> 7.2, 4096 x 2816, 16
// tokens 111.5 -> 18.0 (q8_0 9.7 -> 5.4, 25.8 -> 8.1, 127 -> 20.8). It rests on the sums
// staying in registers: in scratch they made 17.9, 17.9 and 49.9 us.
#include "zz_common.h"
#include "zz_kernels.h"

#define MV_R 4           // weight rows per workgroup
#define MV_T 8           // most tokens per workgroup

// The tensors start wherever the caller's mapping holds them and rows are 18-, 34- or
// 36-byte blocks: loads of any alignment (one instruction each on gfx950).
template <typename V>
__device__ __forceinline__ V ld_any(const uint8_t *p) {
    V v;
    __builtin_memcpy(&v, p, sizeof v);
    return v;
}

// Unit u of a row: 8 weights as floats, two runs of four that multiply x[xo..xo+3] and
// x[xo + XD..xo + XD + 3], and their scale d (tq2: 1; the row's alpha comes at the end)
// and q4a's offset m.
template <int FMT>
struct MvUnit {
    static constexpr int XD = FMT == ZZ_FMT_Q80 ? 4 : 16;
    static __device__ __forceinline__ int xo(int u) { return ZZ_BLK * (u >> 2) + (FMT == ZZ_FMT_Q80 ? 8 : 4) * (u & 3); }
    uint32_t a, b, s;
    __device__ __forceinline__ void load(const uint8_t *r, int u) {
        const int k = u >> 2, q = u & 3;
        b = 0;
        s = 0;
        if constexpr (FMT == ZZ_FMT_TQ2) {
            a = ld_any<uint32_t>(r + 16 * (u >> 3) + 4 * q);
        } else if constexpr (FMT == ZZ_FMT_Q4A) {
            // 64 weights in 36 bytes: fp16 d, fp16 m, then two halves of 16 bytes whose
            // low nibbles are w[j] and high nibbles w[j + 16] (tq2.h:269-282)
            const uint8_t *g = r + 36 * (size_t)(u >> 3);
            s = ld_any<uint32_t>(g);
            a = ld_any<uint32_t>(g + 4 + 16 * (k & 1) + 4 * q);
        } else if constexpr (FMT == ZZ_FMT_Q80) {
            const uint8_t *g = r + 34 * (size_t)k;
            s = ld_any<uint16_t>(g);
            a = ld_any<uint32_t>(g + 2 + 8 * q);
            b = ld_any<uint32_t>(g + 6 + 8 * q);
        } else {
            const uint8_t *g = r + 18 * (size_t)k;
            s = ld_any<uint16_t>(g);
            a = ld_any<uint32_t>(g + 2 + 4 * q);
        }
    }
    __device__ __forceinline__ void unpack(int u, float (&w)[8], float &d, float &m) const {
        d = 1.0f;
        m = 0.0f;
        if constexpr (FMT != ZZ_FMT_TQ2) d = zz_h2f((uint16_t)(s & 0xffff));
        if constexpr (FMT == ZZ_FMT_Q4A) m = zz_h2f((uint16_t)(s >> 16));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (FMT == ZZ_FMT_TQ2) {
                const int sh = 4 * ((u >> 2) & 1);         // bit planes 2h and 2h + 1 of half h
                w[i] = (float)((int)((a >> (8 * i + sh)) & 3) - 1);
                w[4 + i] = (float)((int)((a >> (8 * i + sh + 2)) & 3) - 1);
            } else if constexpr (FMT == ZZ_FMT_Q80) {
                w[i] = (float)(int8_t)(a >> (8 * i));
                w[4 + i] = (float)(int8_t)(b >> (8 * i));
            } else {
                const float z = FMT == ZZ_FMT_Q40 ? 8.0f : 0.0f;
                w[i] = (float)((a >> (8 * i)) & 15) - z;
                w[4 + i] = (float)((a >> (8 * i + 4)) & 15) - z;
            }
        }
    }
};

// v summed over the four lanes of each quad (one 32-weight block), the same bits in all
__device__ __forceinline__ float mv_quad_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));    // lane ^ 1
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));   // lane ^ 2
}

// V sums over the wave into acc[0]: at step k a lane keeps the half of its values that bit
// k of its number names and hands the other half to its partner, V - 1 exchanges instead of
// 6 V (none at all in the first two steps where a quad's lanes hold equal sums); lane l < V
// ends with the value of l's bits reversed, the lanes beyond V are added in the usual way.
// A template, so that every index is a constant: as a loop the compiler kept it dynamic,
// 2,000 selects a thread.
template <bool QUAD, int V, int N, int K = 0>
__device__ __forceinline__ void mv_reduce(float (&acc)[N], int l) {
    if constexpr (V > 1) {
        constexpr int h = V / 2;
        const bool up = (l >> K) & 1;
#pragma unroll
        for (int v = 0; v < h; v++) {
            // both read first: a choice between two elements is a choice of addresses to
            // the compiler, and the array then lives in scratch or LDS
            const float lo = acc[v], hi = acc[v + h], keep = up ? hi : lo;
            if constexpr (QUAD && K < 2) acc[v] = keep;
            else acc[v] = keep + __shfl_xor(up ? lo : hi, 1 << K);
        }
        mv_reduce<QUAD, h, N, K + 1>(acc, l);
    } else if constexpr ((1 << K) < 64) {
        acc[0] += __shfl_xor(acc[0], 1 << K);
        mv_reduce<QUAD, 1, N, K + 1>(acc, l);
    }
}

template <int FMT, int T>
__global__ __launch_bounds__(256) void zz_matmul_f32_kernel(float *y, const uint8_t *W, const float *x, int O, int I,
                                                            int S) {
    constexpr int N = T <= 1 ? 1 : T <= 2 ? 2 : T <= 4 ? 4 : 8, V = MV_R * N;
    // a block's partial is whole before its d scales it, as in the reference: an
    // infinite d then gives the reference's infinities and NaNs. tq2 has no block scale.
    constexpr bool QUAD = FMT != ZZ_FMT_TQ2;
    const int row0 = blockIdx.x * MV_R, s0 = blockIdx.y * T, tid = threadIdx.x, w = tid >> 6, l = tid & 63;
    const uint8_t *data = W + (FMT == ZZ_FMT_TQ2 ? (size_t)O * 4 : 0);
    const size_t rb = FMT == ZZ_FMT_TQ2 ? (size_t)I / 4 : FMT == ZZ_FMT_Q4A ? (size_t)(I / 64) * 36
                    : (size_t)(I / ZZ_BLK) * (FMT == ZZ_FMT_Q80 ? 34 : 18);
    const uint8_t *rp[MV_R];
    const float *xp[T];
#pragma unroll
    for (int r = 0; r < MV_R; r++) rp[r] = data + (size_t)min(row0 + r, O - 1) * rb;    // clamped: not stored
#pragma unroll
    for (int t = 0; t < T; t++) xp[t] = x + (size_t)min(s0 + t, S - 1) * I;
    float acc[V];                                // [row][token]
#pragma unroll
    for (int v = 0; v < V; v++) acc[v] = 0.0f;
    for (int u = tid; u < I / 8; u += 256) {
        MvUnit<FMT> k[MV_R];
#pragma unroll
        for (int r = 0; r < MV_R; r++) k[r].load(rp[r], u);
        const int xo = MvUnit<FMT>::xo(u);
        float4 xa[T], xb[T];
#pragma unroll
        for (int t = 0; t < T; t++) {
            xa[t] = *(const float4 *)(xp[t] + xo);
            xb[t] = *(const float4 *)(xp[t] + xo + MvUnit<FMT>::XD);
        }
        float sx[T];                             // q4a: the block's sum of x
        if constexpr (FMT == ZZ_FMT_Q4A)
#pragma unroll
            for (int t = 0; t < T; t++)
                sx[t] = mv_quad_sum(((xa[t].x + xa[t].y) + (xa[t].z + xa[t].w)) + ((xb[t].x + xb[t].y) + (xb[t].z + xb[t].w)));
#pragma unroll
        for (int r = 0; r < MV_R; r++) {
            float f[8], d, m;
            k[r].unpack(u, f, d, m);
#pragma unroll
            for (int t = 0; t < T; t++) {
                float p = f[0] * xa[t].x;
                p = fmaf(f[1], xa[t].y, p);
                p = fmaf(f[2], xa[t].z, p);
                p = fmaf(f[3], xa[t].w, p);
                p = fmaf(f[4], xb[t].x, p);
                p = fmaf(f[5], xb[t].y, p);
                p = fmaf(f[6], xb[t].z, p);
                p = fmaf(f[7], xb[t].w, p);
                if (QUAD) p = mv_quad_sum(p);
                float &A = acc[r * N + t];
                if constexpr (FMT == ZZ_FMT_Q4A) {
                    A = fmaf(d, p, fmaf(m, sx[t], A));
                } else if constexpr (FMT == ZZ_FMT_TQ2) {
                    A += p;
                } else {
                    A = fmaf(d, p, A);
                }
            }
        }
    }
    mv_reduce<QUAD, V>(acc, l);
    __shared__ float part[4][V];
    if (l < V) part[w][__brev((unsigned)l) / (0xFFFFFFFFu / V + 1)] = acc[0];
    __syncthreads();
    const int r = row0 + tid / N, t = tid % N;
    if (tid < V && t < T && r < O && s0 + t < S) {
        float v = (part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]);
        if (FMT == ZZ_FMT_TQ2) v *= ld_any<float>(W + 4 * (size_t)r);
        y[(size_t)(s0 + t) * O + r] = v;
    }
}

template <int FMT>
static void zz_matmul_fmt(int T, dim3 g, float *y, const uint8_t *W, const float *x, int O, int I, int S, hipStream_t st) {
    switch (T) {
#define MV(N) case N: hipLaunchKernelGGL((zz_matmul_f32_kernel<FMT, N>), g, dim3(256), 0, st, y, W, x, O, I, S); break
        MV(1); MV(2); MV(3); MV(4); MV(5); MV(6); MV(7);
    default: MV(8);
#undef MV
    }
}

int zz_launch_matmul_f32(int fmt, float *y, const uint8_t *W, const float *x, int O, int I,
                         int S, hipStream_t st) {
    // the tokens in equal shares of at most MV_T, so that no workgroup works on padding
    const int ny = (S + MV_T - 1) / MV_T, T = (S + ny - 1) / ny;
    const dim3 g((O + MV_R - 1) / MV_R, ny);
    switch (fmt) {
    case ZZ_FMT_Q40: zz_matmul_fmt<ZZ_FMT_Q40>(T, g, y, W, x, O, I, S, st); break;
    case ZZ_FMT_Q80: zz_matmul_fmt<ZZ_FMT_Q80>(T, g, y, W, x, O, I, S, st); break;
    case ZZ_FMT_TQ2: zz_matmul_fmt<ZZ_FMT_TQ2>(T, g, y, W, x, O, I, S, st); break;
    default: zz_matmul_fmt<ZZ_FMT_Q4A>(T, g, y, W, x, O, I, S, st); break;
    }
    return hipGetLastError() == hipSuccess;
}

__global__ __launch_bounds__(256) void zz_copy_f32_kernel(float4 *dst, const float4 *src, unsigned n4) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i < n4) dst[i] = src[i];
}

int zz_launch_copy_f32(float *dst, const float *src, size_t n, hipStream_t st) {
    const unsigned n4 = (unsigned)((n + 3) / 4);
    hipLaunchKernelGGL(zz_copy_f32_kernel, dim3((n4 + 255) / 256), dim3(256), 0, st, (float4 *)dst, (const float4 *)src, n4);
    return hipGetLastError() == hipSuccess;
}
