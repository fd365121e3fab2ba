// Rotary positions of the decoder shell's attention (rotate-half form), bfloat16, fused with taking the projection apart:
//
//   forward   qkv [B, S, 3, H, d]  ->  q, k [B, S, H, d]:   y1 = x1 cos1 - x2 sin1,  y2 = x2 cos2 + x1 sin2     (halves of d)
//   backward  dq, dk, dv (any strides) -> dqkv:             dx1 = d1 cos1 + d2 sin2,  dx2 = d2 cos2 - d1 sin1,  dv as it is
//
// Every product and every sum is rounded to bfloat16, as the element-wise operations it stands for round them, so results are
// those of x * cos + rotate_half(x) * sin bit for bit.  Bound by HBM and launches: one launch each way instead of ten
// forward and over twenty backward (slices, negations, concatenations, fills and their sums).
#include "mhffn_common.hpp"

namespace mhffn {

namespace {

struct RopeArgs {
    const bf16_t* qkv;
    const bf16_t *cos, *sin;      // [S, d]
    bf16_t *q, *k, *dqkv;
    const bf16_t* d[3];           // dq, dk, dv: element (b, h, s, c) at b * stride[0] + h * stride[1] + s * stride[2] + c
    long stride[3][3];
    unsigned n;                   // threads: B * S * H * d / 16
    int S, H, dh;
    FastDiv by_vec, by_h, by_s;   // d / 16, H, S
};

// (contraction is off in the kernels: with it the compiler takes a product's own rounding away and fuses it with the sum)
__device__ __forceinline__ float rnd(float x) { return (float)(bf16_t)x; }

struct RopeAt {
    unsigned b, h;
    int c;                        // first column of this thread's eight of each half
    long row, s;                  // b * S + s
    __device__ RopeAt(const RopeArgs& p, unsigned i)
    {
        const unsigned r = p.by_vec.div(i), t = p.by_h.div(r);
        c = (i - r * (p.dh / 16)) * 8;
        h = r - t * p.H;
        b = p.by_s.div(t);
        row = t;
        s = t - b * (unsigned)p.S;
    }
};

__global__ __launch_bounds__(256) void rope_fwd_kernel(RopeArgs p)
{
#pragma clang fp contract(off)
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= p.n) return;
    const RopeAt a(p, i);
    const int half = p.dh / 2;
    const long tab = a.s * p.dh + a.c;
    const bf16x8 c1 = *reinterpret_cast<const bf16x8*>(p.cos + tab), c2 = *reinterpret_cast<const bf16x8*>(p.cos + tab + half);
    const bf16x8 s1 = *reinterpret_cast<const bf16x8*>(p.sin + tab), s2 = *reinterpret_cast<const bf16x8*>(p.sin + tab + half);
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const bf16_t* src = p.qkv + ((a.row * 3 + w) * p.H + a.h) * p.dh + a.c;
        bf16_t* dst = (w ? p.k : p.q) + (a.row * p.H + a.h) * p.dh + a.c;
        const bf16x8 x1 = *reinterpret_cast<const bf16x8*>(src), x2 = *reinterpret_cast<const bf16x8*>(src + half);
        bf16x8 y1, y2;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            y1[j] = (bf16_t)(rnd((float)x1[j] * (float)c1[j]) + rnd(-(float)x2[j] * (float)s1[j]));
            y2[j] = (bf16_t)(rnd((float)x2[j] * (float)c2[j]) + rnd((float)x1[j] * (float)s2[j]));
        }
        *reinterpret_cast<bf16x8*>(dst) = y1;
        *reinterpret_cast<bf16x8*>(dst + half) = y2;
    }
}

__global__ __launch_bounds__(256) void rope_bwd_kernel(RopeArgs p)
{
#pragma clang fp contract(off)
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= p.n) return;
    const RopeAt a(p, i);
    const int half = p.dh / 2;
    const long tab = a.s * p.dh + a.c;
    const bf16x8 c1 = *reinterpret_cast<const bf16x8*>(p.cos + tab), c2 = *reinterpret_cast<const bf16x8*>(p.cos + tab + half);
    const bf16x8 s1 = *reinterpret_cast<const bf16x8*>(p.sin + tab), s2 = *reinterpret_cast<const bf16x8*>(p.sin + tab + half);
#pragma unroll
    for (int w = 0; w < 3; ++w) {
        const bf16_t* src = p.d[w] + a.b * p.stride[w][0] + a.h * p.stride[w][1] + a.s * p.stride[w][2] + a.c;
        bf16_t* dst = p.dqkv + ((a.row * 3 + w) * p.H + a.h) * p.dh + a.c;
        bf16x8 d1, d2;
#pragma unroll
        for (int j = 0; j < 8; ++j) { d1[j] = src[j]; d2[j] = src[half + j]; }      // (rows may start at any element)
        if (w < 2) {
            bf16x8 x1, x2;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                x1[j] = (bf16_t)(rnd((float)d1[j] * (float)c1[j]) + rnd((float)d2[j] * (float)s2[j]));
                x2[j] = (bf16_t)(rnd((float)d2[j] * (float)c2[j]) - rnd((float)d1[j] * (float)s1[j]));
            }
            d1 = x1;
            d2 = x2;
        }
        *reinterpret_cast<bf16x8*>(dst) = d1;
        *reinterpret_cast<bf16x8*>(dst + half) = d2;
    }
}

RopeArgs rope_args(const void* cos, const void* sin, int B, int S, int H, int dh)
{
    RopeArgs a{};
    a.cos = (const bf16_t*)cos;
    a.sin = (const bf16_t*)sin;
    a.n = (unsigned)((long)B * S * H * (dh / 16));
    a.S = S;
    a.H = H;
    a.dh = dh;
    a.by_vec = FastDiv(dh / 16);
    a.by_h = FastDiv(H);
    a.by_s = FastDiv(S);
    return a;
}

}  // namespace

hipError_t launch_rope_fwd(const void* qkv, const void* cos, const void* sin, void* q, void* k, int B, int S, int H, int dh,
                           hipStream_t st)
{
    RopeArgs a = rope_args(cos, sin, B, S, H, dh);
    a.qkv = (const bf16_t*)qkv;
    a.q = (bf16_t*)q;
    a.k = (bf16_t*)k;
    hipLaunchKernelGGL(rope_fwd_kernel, dim3((a.n + 255) / 256), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_rope_bwd(const void* const d[3], const long (*stride)[3], const void* cos, const void* sin, void* dqkv, int B, int S,
                           int H, int dh, hipStream_t st)
{
    RopeArgs a = rope_args(cos, sin, B, S, H, dh);
    a.dqkv = (bf16_t*)dqkv;
    for (int w = 0; w < 3; ++w) {
        a.d[w] = (const bf16_t*)d[w];
        for (int i = 0; i < 3; ++i) a.stride[w][i] = stride[w][i];
    }
    hipLaunchKernelGGL(rope_bwd_kernel, dim3((a.n + 255) / 256), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace mhffn
