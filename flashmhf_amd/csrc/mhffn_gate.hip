// Head prologue of the multi-head FFN block for gfx950: per-head RMSNorm of the projected heads and the expert gate, in
// one pass over the [B, S, H, d_h] activations, forward and backward.
//
//   u = x * rsqrt(mean(x^2) + eps)            fp32, per (token, head) row          (modeling_mhffnmoe.py:124-129)
//   y = bf16(u * w[h])                        the Q the fused operator reads       (:130-133)
//   z = y . router[h]      (fp32, d_h x E)    s = sigmoid(z)    R = s / max(sum_e s, 1e-20)   (:384-386)
//
// Both kernels are bound by HBM traffic, not by arithmetic: a wave owns tiles of 32 tokens of one head, loads each row
// once with 16-byte accesses (a lane holds half a row: the 8-element chunks 2ks + g), keeps everything between the load
// and the stores in registers, and takes the router products on the matrix cores:
//   * logits^T [E x 32 tokens] = router^T (A, staged once per workgroup in LDS as bf16 hi + lo parts of the fp32
//     values, so a float32 router is honoured to 2^-17) x y^T (B = the lane's own packed row chunks);
//     the sum over experts is then a sum over a lane's registers plus one exchange between the two lane halves;
//   * backward: dy += dz router^T (B = dz straight from the logits' registers: the router rows are fed in row_perm32
//     order, exactly as the main kernels chain their products) and d_router += y^T dz (contraction over tokens = lanes:
//     y and dz go through a wave-private LDS tile and come back with transposing reads).
// d_router and d_norm_weight are summed over all tokens: partial sums per wave, added up per workgroup, then either one atomic
// add per workgroup and element (mhffn_gate_bwd: the caller passes zero-filled or to-be-accumulated buffers) or a partial
// sum in memory that a second pass adds in order and writes in the parameters' type (mhffn_gate_bwd_into).
#include "mhffn_common.hpp"

namespace mhffn {

struct GateArgs {
    const bf16_t* X;     // [B, S, H, DH]
    const void* Wn;      // [H, DH] (NORM only), float or bfloat16 (wn_bf16)
    const void* Wr;      // [H, DH, E], float or bfloat16 (wr_bf16)
    bf16_t* Qn;          // [B, S, H, DH] (NORM only)
    float* R;            // [B, H, S, E]
    const bf16_t* dQ;    // gradient of y, rows addressed through dq_tokmaj
    const float* dR;     // [B, H, S, E]
    bf16_t* dX;          // [B, S, H, DH]
    float* dWn;          // [H, DH] and
    float* dWr;          // [H, DH, E], accumulated by atomic adds, or (part != null) not used:
    float* part;         // [H][workgroups of a head][DH * E + DH] sums of d_router, d_norm_weight over a workgroup's tokens
    int B, H, S, E, tpw, dq_tokmaj, wn_bf16, wr_bf16;
    float eps;
    int wgs, heads_first;      // backward: workgroups of a head and batch; the head runs fastest over the workgroups
    FastDiv by_fast;           // heads if heads_first, else wgs
};

__device__ __forceinline__ float param(const void* p, long i, int bf16)
{
    return bf16 ? (float)static_cast<const bf16_t*>(p)[i] : static_cast<const float*>(p)[i];
}
__device__ __forceinline__ float bf_even(unsigned w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf_odd(unsigned w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
__device__ __forceinline__ float bf_at(const u32x4& v, int j) { return (j & 1) ? bf_odd(v[j >> 1]) : bf_even(v[j >> 1]); }

template <int DH, int NT, typename T>
__device__ void stage_router_rows(const T* Wr, int E, unsigned char* dst);
template <int DH, int NT, typename T>
__device__ void stage_router_cols(const T* Wr, int E, unsigned char* dst);

// Router slice of head h as MFMA A operands in LDS.
//   part 0/1 (hi/lo), expert tile nt, k-step ks, lane (rho, g): router[(2ks+g)*8 + j][nt*32 + row_perm32(rho)], j = 0..7
// so that register 8s + kk of lane half g of the product holds expert nt*32 + 16s + 8g + kk.
template <int DH, int NT>
__device__ __forceinline__ void stage_router_rows(const void* Wr, long w0, int bf16, int E, unsigned char* dst)
{
    if (bf16) stage_router_rows<DH, NT>(static_cast<const bf16_t*>(Wr) + w0, E, dst);
    else stage_router_rows<DH, NT>(static_cast<const float*>(Wr) + w0, E, dst);
}
template <int DH, int NT, typename T>
__device__ __forceinline__ void stage_router_rows(const T* Wr, int E, unsigned char* dst)
{
    constexpr int KS = DH / 16;
    for (int idx = threadIdx.x; idx < NT * KS * 64; idx += blockDim.x) {
        const int ln = idx & 63, ks = (idx >> 6) % KS, nt = idx / (KS * 64);
        const int e = nt * 32 + row_perm32(ln & 31), k0 = (2 * ks + (ln >> 5)) * 8;
        bf16x8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float x = (float)Wr[(long)(k0 + j) * E + (e < E ? e : 0)], v = e < E ? x : 0.0f;
            hi[j] = (bf16_t)v;
            lo[j] = (bf16_t)(v - (float)hi[j]);
        }
        *reinterpret_cast<bf16x8*>(dst + idx * 16) = hi;
        *reinterpret_cast<bf16x8*>(dst + (NT * KS * 64 + idx) * 16) = lo;
    }
}

// Router slice as A operands of dy^T [d_h x tokens] = router [d_h x E] dz^T: column tile ct, k-step q = 2nt + s,
// lane (rho, g): router[ct*32 + row_perm32(rho)][nt*32 + 16s + 8g + j]  (bf16, high part only: dy is rounded to bf16).
template <int DH, int NT>
__device__ __forceinline__ void stage_router_cols(const void* Wr, long w0, int bf16, int E, unsigned char* dst)
{
    if (bf16) stage_router_cols<DH, NT>(static_cast<const bf16_t*>(Wr) + w0, E, dst);
    else stage_router_cols<DH, NT>(static_cast<const float*>(Wr) + w0, E, dst);
}
template <int DH, int NT, typename T>
__device__ __forceinline__ void stage_router_cols(const T* Wr, int E, unsigned char* dst)
{
    constexpr int CT = DH / 32;
    for (int idx = threadIdx.x; idx < CT * 2 * NT * 64; idx += blockDim.x) {
        const int ln = idx & 63, q = (idx >> 6) % (2 * NT), ct = idx / (2 * NT * 64);
        const int col = ct * 32 + row_perm32(ln & 31), e0 = q * 16 + 8 * (ln >> 5);
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float x = (float)Wr[(long)col * E + (e0 + j < E ? e0 + j : 0)];
            v[j] = (bf16_t)(e0 + j < E ? x : 0.0f);
        }
        *reinterpret_cast<bf16x8*>(dst + idx * 16) = v;
    }
}

// 32 rows of DH values as whole rows between memory and registers or LDS, and as half rows (the 16-byte chunks 2 ks + g of row
// l32) between LDS and the lanes that compute.  Whole rows: a wave-instruction moves the 64 chunks from 64 i on, counted along
// the rows; chunk c of row r sits at c ^ swz(r) in LDS, which keeps 16 rows' reads of one chunk in different banks.
struct WholeRows {};      // (mode of the kernels below)
template <int DH>
struct RowTile {
    static constexpr int CH = DH / 8, INS = DH / 16;
    __device__ static int swz(int r)
    {
        return DH == 128 ? swz16(r) : DH == 96 ? (r >> 2) & 3 : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
    }
    __device__ static int row(int i, int lane) { return (i * 64 + lane) / CH; }
    __device__ static int chunk(int i, int lane) { return (i * 64 + lane) % CH ^ swz(row(i, lane)); }
    __device__ static int half(int ks, int l32, int g) { return l32 * (2 * DH) + (((2 * ks + g) ^ swz(l32)) << 4); }
};

// Whole rows leave past the caches, room in which they would take from the rows that are being read.  us through them / past, four inputs in turn: 8,192 tokens of 8 heads of 128
// forward 12.1 / 10.5, backward 22.9 / 21.2, 16,384 18.3 / 17.0 and 36.3 / 33.5, 32,768 of 16 heads 62.4 / 62.2 and 109.6 / 105.7.  Where x is in the memory-side cache already, it
// stays there: the last on one input again and again 66.6 / 54.3 forward; both passes behind each other 169 / 161.  Not so R, whose blocks begin and end inside a line (16,384 of
// 8 heads 16.0 instead of 14.8, one input), nor x on its way in (32,768 of 16 61 instead of 50).
__device__ __forceinline__ void store_past(bf16_t* to, u32x4 v) { __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(to)); }

// Everything the forward computes for one tile, shared by both kernels.
template <int DH, int NT, bool NORM>
struct GateTile {
    static constexpr int KS = DH / 16;
    u32x4 xr[KS];       // the lane's half row of x
    bf16x8 y[KS];       // normalised, rounded
    float rstd;
    float s[NT][16];    // sigmoid(z), 0 for experts >= E
    float inv;          // 1 / max(sum s, 1e-20)
    float sum;

    __device__ __forceinline__ void load(const bf16_t* xrow, int g)
    {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) xr[ks] = *reinterpret_cast<const u32x4*>(xrow + (2 * ks + g) * 8);
    }
    // FENCED: one k-step's LDS reads at a time (the backward has no registers for all of them at once)
    template <bool FENCED>
    __device__ __forceinline__ void normalise(const float* sW, int g)
    {
        if constexpr (NORM) {
            float ss = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float v = bf_at(xr[ks], j);
                    ss = fmaf(v, v, ss);
                }
            ss += __shfl_xor(ss, 32);
            rstd = 1.0f / sqrtf(ss / (float)DH + eps_);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const f32x4 w0 = *reinterpret_cast<const f32x4*>(sW + (2 * ks + g) * 8);
                const f32x4 w1 = *reinterpret_cast<const f32x4*>(sW + (2 * ks + g) * 8 + 4);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    y[ks][j] = (bf16_t)((bf_at(xr[ks], j) * rstd) * (j < 4 ? w0[j & 3] : w1[j & 3]));
                if constexpr (FENCED) __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            rstd = 1.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) y[ks] = __builtin_bit_cast(bf16x8, xr[ks]);
        }
    }
    template <bool FENCED>
    __device__ __forceinline__ void gate(const unsigned char* sA, int lane, int g, int E)
    {
        f32x16 acc[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[nt][i] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const unsigned char* a = sA + ((nt * KS + ks) * 64 + lane) * 16;
                acc[nt] = mfma32(*reinterpret_cast<const bf16x8*>(a), y[ks], acc[nt]);
                acc[nt] = mfma32(*reinterpret_cast<const bf16x8*>(a + NT * KS * 1024), y[ks], acc[nt]);
            }
            if constexpr (FENCED) {
                if (ks % 2 == 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
        sum = 0.0f;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int e = nt * 32 + 16 * (i >> 3) + 8 * g + (i & 7);
                s[nt][i] = e < E ? fast_sigmoid(acc[nt][i]) : 0.0f;
                sum += s[nt][i];
            }
        sum += __shfl_xor(sum, 32);
        inv = 1.0f / fmaxf(sum, 1e-20f);
    }
    float eps_;
};

// router operands | norm weight | per wave: a [32 tokens][E] float tile of R, so that the 32 x E block (contiguous in
// memory) leaves the wave as whole cache lines instead of one scattered dword per lane and expert
constexpr size_t gate_fwd_smem(int DH, int NT) { return (size_t)2 * NT * (DH / 16) * 1024 + DH * 4 + 4 * TILE_B; }

// With WholeRows the rows move between memory and the wave as whole rows, by way of its LDS; else each lane loads and stores its half row,
// in 32-byte pieces of 32 rows per instruction.  Pieces keep the path from L2 busy four times as long: 32,768 tokens of 16 heads of
// 128 take 71.5 us with them and 62.8 with whole rows (loads alone in pieces 65.3), 16,384 of
// 8 heads 18.3 and 16.9 (those past the caches: store_past; 5.1 TB/s for the former, what a large copy reaches).
// Few tokens wait for one tile's chain, which the way through LDS makes longer: 512 of 8 heads 6.0 and 6.3.
template <int DH, int NT, bool NORM, class... Mode>
__global__ __launch_bounds__(256) void mhffn_gate_fwd_kernel(GateArgs p)
{
    constexpr bool WHOLE = sizeof...(Mode) > 0;
    constexpr int KS = DH / 16;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    float* sW = reinterpret_cast<float*>(smem + 2 * NT * KS * 1024);
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* rtile = sW + DH + wave * (TILE_B / 4);
    const int h = blockIdx.y, b = blockIdx.z;

    stage_router_rows<DH, NT>(p.Wr, (long)h * DH * p.E, p.wr_bf16, p.E, smem);
    if constexpr (NORM)
        for (int i = threadIdx.x; i < DH; i += blockDim.x) sW[i] = param(p.Wn, h * DH + i, p.wn_bf16);
    __syncthreads();

    const int ntiles = (p.S + 31) / 32;
    const int tile0 = (blockIdx.x * 4 + wave) * p.tpw;
    const int tile1 = min(tile0 + p.tpw, ntiles);
    for (int tile = tile0; tile < tile1; ++tile) {
        const int t = tile * 32 + l32;
        const bool valid = t < p.S;
        const long row = (((long)b * p.S + (valid ? t : p.S - 1)) * p.H + h) * DH;
        GateTile<DH, NT, NORM> T;
        T.eps_ = p.eps;
        using Rows = RowTile<DH>;
        unsigned char* xt = reinterpret_cast<unsigned char*>(rtile);      // the wave's rows of x, then of y, then of R
        const long row0 = (((long)b * p.S + tile * 32) * p.H + h) * DH, stride = (long)p.H * DH;
        const int nrow = min(32, p.S - tile * 32);
        if constexpr (WHOLE) {
#pragma unroll
            for (int i = 0; i < Rows::INS; ++i)
                __builtin_amdgcn_global_load_lds((gptr_t)(p.X + row0 + min(Rows::row(i, lane), nrow - 1) * stride + Rows::chunk(i, lane) * 8),
                                                 (lptr_t)(xt + i * 1024), 16, 0, 0);
            wait_vmcnt<0>();
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) T.xr[ks] = *reinterpret_cast<const u32x4*>(xt + Rows::half(ks, l32, g));
        } else {
            T.load(p.X + row, g);
        }
        T.template normalise<false>(sW, g);
        if constexpr (NORM && WHOLE) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) *reinterpret_cast<bf16x8*>(xt + Rows::half(ks, l32, g)) = T.y[ks];
#pragma unroll
            for (int i = 0; i < Rows::INS; ++i) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(xt + i * 1024 + lane * 16);
                if (Rows::row(i, lane) < nrow)
                    store_past(p.Qn + row0 + Rows::row(i, lane) * stride + Rows::chunk(i, lane) * 8, v);
            }
        } else if constexpr (NORM) {
            if (valid) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    *reinterpret_cast<bf16x8*>(p.Qn + row + (2 * ks + g) * 8) = T.y[ks];
            }
        }
        T.template gate<false>(smem, lane, g, p.E);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int e = nt * 32 + 16 * (i >> 3) + 8 * g + (i & 7);
                if (e < p.E) rtile[l32 * p.E + e] = T.s[nt][i] * T.inv;
            }
        float* rblock = p.R + (((long)b * p.H + h) * p.S + tile * 32) * p.E;
        const int lim = min(32, p.S - tile * 32) * p.E;
        for (int idx = lane; idx < lim; idx += 64) rblock[idx] = rtile[idx];
    }
}

// ---- backward -------------------------------------------------------------------------------------------------------
// LDS: router rows (hi, lo) | router columns | norm weight | per wave: y tile (8 KB, the swizzled 32 x 256-byte layout of the
// main kernels so the transposing reads can be shared) + dz tile (NT = 2: the same; NT = 1: 4 KB) | [waves][128] floats for
// the sums across waves.  A wave takes enough consecutive tiles that the launch fills the chip once, which also bounds
// the number of partial sums.
//
// Up to 32 experts (NT = 1) eight waves, two per SIMD (with few tokens four: gate_bwd_waves), and nothing but sums in few
// registers lives across tiles: the waves' y and dz tiles are contracted together, each wave keeping one column tile of d_router (16 registers) over the tokens
// of several waves, two barriers per tile; the products d * u of d_norm_weight pass through the wave's LDS region a half at a
// time and are added up down the columns (4 values per 64 columns).  What that frees holds the next tile's rows of x, requested
// behind the contraction, while dR and dQ of a tile are requested at its top and used half a trip later.  One wave per SIMD
// with all sums in registers, ~2,400 instructions per tile, a quarter of them register moves, took 150 us on 32,768 tokens of
// 16 heads of 128 with 22 experts; two waves with the d_router sums in registers and no rows ahead 145; this 109 us, 101
// with dX stored as whole rows; past the caches 105.7 with its sums where it was 109.6, four inputs in turn (4.2 TB/s).  What is left is latency inside a tile (LDS operands, the chains over a row) at two waves per SIMD.
// More experts (NT = 2) have twice the d_router operands: four waves, one per SIMD, all sums in registers, and the next
// tile's rows requested before the current tile's arithmetic starts.
constexpr int GATE_Z_ROW_B = 64;                           // NT = 1: row of the dz tile
constexpr int GATE_WAVE_REGION_B = 2 * TILE_B + 1024;      // NT = 2: also a 64 x 65 float transpose
template <int NT>
constexpr int gate_bwd_region() { return NT == 1 ? TILE_B + 32 * 32 * 4 : GATE_WAVE_REGION_B; }      // (dR passes through the dz tile as fp32)
template <int NT>
constexpr size_t gate_bwd_smem(int DH, int waves)
{
    return (size_t)2 * NT * (DH / 16) * 1024 + (size_t)(DH / 32) * 2 * NT * 1024 + DH * 4 +
           waves * (gate_bwd_region<NT>() + 128 * 4);
}

// Transposed operand (column tile ct, k-half s) of a swizzled tile.  Only column tile 0's two lane offsets are kept in
// registers: the swizzle XORs the chunk index, and a column tile is 4 chunks = 64 bytes, so tile ct's offset is tile
// 0's with bits 6..7 XORed by ct (one VALU instruction per read instead of two more registers per column tile).
__device__ __forceinline__ bf16x8 tile_cols(const unsigned char* tile, const TrLane<1>& tl, int ct, int s)
{
    typedef __attribute__((address_space(3))) v4bf16_t* lds_v4;
    const v4bf16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4)(tile + (tl.off[0][0] ^ (ct << 6)) + 4096 * s));
    const v4bf16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4)(tile + (tl.off[0][1] ^ (ct << 6)) + 4096 * s));
    bf16x8 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        r[j] = lo[j];
        r[4 + j] = hi[j];
    }
    return r;
}

// The same of the dz tile of NT = 1: rows of 32 experts, chunk c of row r at c ^ (r / 4 % 4).
__device__ __forceinline__ bf16x8 z_cols(const unsigned char* tile, int lane, int s)
{
    typedef __attribute__((address_space(3))) v4bf16_t* lds_v4;
    const int lam = lane & 15, l32 = lane & 31, g = lane >> 5, r = 8 * g + (lam >> 2), c = 2 * (l32 >> 4) + ((lam & 3) >> 1);
    const int at = r * GATE_Z_ROW_B + ((c ^ (r >> 2 & 3)) << 4) + (lam & 1) * 8;
    const v4bf16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4)(tile + at + 16 * GATE_Z_ROW_B * s));
    const v4bf16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4)(tile + (at ^ 16) + (16 * s + 4) * GATE_Z_ROW_B));
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        v[j] = lo[j];
        v[4 + j] = hi[j];
    }
    return v;
}

// With WholeRows, workgroups of eight waves, dX leaves as whole rows, by way of the y tile, past the caches (store_past) as Q does in the forward.
// Both kernels, us, whole rows / half rows' pieces, one input again and again: 32,768 tokens of 16 heads of 128 98 / 112 (104 as whole rows through the caches),
// 16,384 of 8 30.1 / 31.2, 8,192 18.5 / 20.3, 5,000 17.1 / 18.2, 7,001 of 64 12.9 / 13.3, 4,096 of 96 15.5 / 15.6.  Workgroups of four, one tile a wave, wait for the
// way through LDS: 3,000 of 8 heads of 128 14.7 / 14.0.  (x and dQ as whole rows, too, take registers: 108 us with a spill, 111 for x alone.)
template <int DH, int NT, bool NORM, class... Mode>
__global__ __launch_bounds__(sizeof...(Mode) > 0 ? 512 : 256, NT == 1 ? 2 : 1) void mhffn_gate_bwd_kernel(GateArgs p)      // (two waves per SIMD up to 32 experts)
{
    constexpr bool WHOLE = sizeof...(Mode) > 0;
    constexpr int NW = WHOLE ? 8 : 4;
    constexpr int KS = DH / 16, CT = DH / 32, REGION_B = gate_bwd_region<NT>();
    constexpr bool AHEAD = NT > 1;                              // rows requested one tile ahead; d_norm_weight in registers
    constexpr int NHALF = (DH + 63) / 64;
    // NT = 1: wave w sums column tile w % CT of d_router over the TPG token tiles of its group w / CT of the workgroup's
    // waves (waves beyond GROUPS * CT none); NT = 2: a wave sums all of it over its own tiles
    constexpr int TPG = CT == 2 ? 2 : 4, WCT = AHEAD ? CT : 1;
    constexpr int GROUPS = NW / TPG;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char* sA = smem;                                   // logits operands
    unsigned char* sC = sA + 2 * NT * KS * 1024;                // dy operands
    float* sW = reinterpret_cast<float*>(sC + CT * 2 * NT * 1024);
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave-uniform: tile counters and tile bases stay scalar
    unsigned char* regions = reinterpret_cast<unsigned char*>(sW + DH);
    unsigned char* ytile = regions + wave * REGION_B;
    unsigned char* ztile = ytile + TILE_B;
    const unsigned slow = p.by_fast.div(blockIdx.x), fast = blockIdx.x - slow * (p.heads_first ? p.H : p.wgs);
    const int wg = p.heads_first ? slow : fast, h = p.heads_first ? fast : slow, b = blockIdx.y;

    stage_router_rows<DH, NT>(p.Wr, (long)h * DH * p.E, p.wr_bf16, p.E, sA);
    stage_router_cols<DH, NT>(p.Wr, (long)h * DH * p.E, p.wr_bf16, p.E, sC);
    if constexpr (NORM)
        for (int i = threadIdx.x; i < DH; i += blockDim.x) sW[i] = param(p.Wn, h * DH + i, p.wn_bf16);
    // the dz tile's chunks beyond the experts in use are read by nobody, but columns e >= E inside a used chunk are:
    // they are written as zeros every tile, so nothing needs clearing here
    __syncthreads();

    const TokRows dqrows = tok_rows(p.dq_tokmaj, b, h, p.H, p.S);
    f32x16 wacc[WCT][NT];           // d_router partial: rows = columns of y, cols = experts
#pragma unroll
    for (int ct = 0; ct < WCT; ++ct)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 16; ++i) wacc[ct][nt][i] = 0.0f;
    // d_norm_weight partial: for the lane's own columns, or columns 64 h + 4 (lane % 16) .. +3 over rows lane / 16 + 4k
    [[maybe_unused]] float dwacc[KS][8];
    [[maybe_unused]] f32x4 dwcol[NHALF];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int j = 0; j < 8; ++j) dwacc[ks][j] = 0.0f;
#pragma unroll
    for (int i = 0; i < NHALF; ++i) dwcol[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const int ntiles = (p.S + 31) / 32;
    const int tile0 = (wg * NW + wave) * p.tpw;
    const int tile1 = min(tile0 + p.tpw, ntiles);
    u32x4 nx[KS], ndq[KS];
    float ngr[NT * 16];
    auto request_x = [&](int tile, int lane) {
        const int l32 = lane & 31, g = lane >> 5, t = tile * 32 + l32;
        const bf16_t* xrow = p.X + (((long)b * p.S + (t < p.S ? t : p.S - 1)) * p.H + h) * DH;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) nx[ks] = *reinterpret_cast<const u32x4*>(xrow + (2 * ks + g) * 8);
    };
    auto request = [&](int tile, int lane) {
        const int l32 = lane & 31, g = lane >> 5, t = tile * 32 + l32;
        const bool valid = t < p.S;
        const int tc = valid ? t : p.S - 1;
        const bf16_t* dqrow = p.dQ + (dqrows.base + (long)tc * dqrows.stride) * DH;
        const float* dblock = p.dR + (((long)b * p.H + h) * p.S + tile * 32) * p.E;
        // the tile's [32][E] block of dR is contiguous: dword k*64 + lane of it, zero past the last token
        const int lim = min(32, p.S - tile * 32) * p.E;
#pragma unroll
        for (int k = 0; k < NT * 16; ++k) {
            const float v = dblock[min(k * 64 + lane, lim - 1)];
            ngr[k] = k * 64 + lane < lim ? v : 0.0f;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) ndq[ks] = *reinterpret_cast<const u32x4*>(dqrow + (2 * ks + g) * 8);
    };
    if (tile0 < tile1) {
        request_x(tile0, lane);
        if (AHEAD) request(tile0, lane);
    }
    for (int tile = tile0; tile < (AHEAD ? tile1 : tile0 + p.tpw); ++tile) {
        // (The lane number of this trip is hidden from the compiler, or it keeps the dozens of addresses below, which cost
        // an instruction or two each, in registers across the loop: with two waves per SIMD there are none to spare.)
        int lane = threadIdx.x & 63;
        if constexpr (!AHEAD) asm volatile("" : "+v"(lane));
        const int l32 = lane & 31, g = lane >> 5;
        const TrLane<1> trl = make_tr_lane<1, 8, 4>(lane);
        // Lane parts of the LDS addresses: row l32 of the y and dz tiles, of the product tile, and this lane's reads of the
        // latter (16 bytes of row lane / 16); the rest of an address is a constant that the swizzle's exclusive-or and the
        // row pitch leave alone.
        const int yrow = l32 * TILE_ROW_B + ((g ^ swz16(l32)) << 4), prow = l32 * TILE_ROW_B + (((2 * g) ^ (l32 & 15)) << 4);
        const int zrow = AHEAD ? yrow : l32 * GATE_Z_ROW_B + ((g ^ (l32 >> 2 & 3)) << 4);
        const int pread = (lane >> 4) * TILE_ROW_B + (((lane & 15) ^ (lane >> 4)) << 4);
        // NT = 1: this tile's token contraction, two barriers around it (every wave of the workgroup passes them p.tpw times)
        auto contract = [&]() {
            __syncthreads();
            const int grp = wave / CT, ct = wave - grp * CT;
            if (grp < GROUPS) {
                for (int k = 0; k < TPG; ++k) {
                    const unsigned char* yt = regions + (grp * TPG + k) * REGION_B;
#pragma unroll
                    for (int s = 0; s < 2; ++s)
                        wacc[0][0] = mfma32(tile_cols(yt, trl, ct, s), z_cols(yt + TILE_B, lane, s), wacc[0][0]);
                }
            }
            __syncthreads();
        };
        if (!AHEAD && tile >= tile1) {      // no tile left for this wave: it adds zeros
            const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) *reinterpret_cast<u32x4*>(ytile + (yrow ^ (ks << 5))) = zero;
#pragma unroll
            for (int s = 0; s < 2; ++s) *reinterpret_cast<u32x4*>(ztile + (zrow ^ (s << 5))) = zero;
            contract();
            continue;
        }
        const int t = tile * 32 + l32;
        const bool valid = t < p.S;
        const long row = (((long)b * p.S + (valid ? t : p.S - 1)) * p.H + h) * DH;
        if (!AHEAD) request(tile, lane);
        GateTile<DH, NT, NORM> T;
        T.eps_ = p.eps;
        u32x4 dqr[KS];
        float gr[NT][16];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            T.xr[ks] = nx[ks];
            dqr[ks] = ndq[ks];
        }
        // dR goes lane-major -> token-major through the (currently idle) dz tile
        auto exchange_dr = [&]() {
            float* rt = reinterpret_cast<float*>(ztile);
#pragma unroll
            for (int k = 0; k < NT * 16; ++k) rt[k * 64 + lane] = ngr[k];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int e = nt * 32 + 16 * (i >> 3) + 8 * g + (i & 7);
                    const float v = rt[min(l32 * p.E + e, 1024 * NT - 1)];
                    gr[nt][i] = e < p.E ? v : 0.0f;
                }
        };
        if (AHEAD) exchange_dr();
        if (AHEAD && tile + 1 < tile1) {
            request_x(tile + 1, lane);
            request(tile + 1, lane);
        }
        if constexpr (!AHEAD) __builtin_amdgcn_sched_barrier(0);
        T.template normalise<!AHEAD>(sW, g);
        if (!valid) {   // rows past the end contribute nothing to the sums over tokens
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) T.y[ks] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            *reinterpret_cast<bf16x8*>(ytile + (yrow ^ (ks << 5))) = T.y[ks];
        T.template gate<!AHEAD>(sA, lane, g, p.E);
        if (!AHEAD) exchange_dr();      // (requested at the top of the trip)

        // R = s * inv; d s = (dR - [sum >= 1e-20] sum_e dR R) * inv; d z = d s * s (1 - s)
        float dot = 0.0f;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 16; ++i) dot = fmaf(gr[nt][i], T.s[nt][i] * T.inv, dot);
        dot += __shfl_xor(dot, 32);
        if (T.sum < 1e-20f) dot = 0.0f;
        bf16x8 dzb[NT][2];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float sv = T.s[nt][i];
                dzb[nt][i >> 3][i & 7] = (bf16_t)((gr[nt][i] - dot) * T.inv * (sv * (1.0f - sv)));
            }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int s = 0; s < 2; ++s)
                *reinterpret_cast<bf16x8*>(ztile + (zrow ^ ((4 * nt + 2 * s) << 4))) = dzb[nt][s];

        // The phases of a tile are fenced, and each unpacks the rows of x anew: left to itself the compiler keeps the 64
        // unpacked values (and their products with rstd) from one phase to the next, which two waves per SIMD have no
        // registers for.
        auto next_phase = [&]() {
            if constexpr (!AHEAD) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(T.xr[ks]));
            }
        };
        next_phase();
        // d_router += y^T dz over this tile's tokens
        if constexpr (!AHEAD) {
            contract();
            request_x(min(tile + 1, ntiles - 1), lane);     // (always: behind a branch the waits for dq below would be for x too)
        } else
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            bf16x8 bz[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) bz[nt] = tile_cols(ztile, trl, nt, s);
#pragma unroll
            for (int ct = 0; ct < WCT; ++ct) {
                const bf16x8 ay = tile_cols(ytile, trl, ct, s);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) wacc[ct][nt] = mfma32(ay, bz[nt], wacc[ct][nt]);
            }
        }

        next_phase();
        // dy^T = router dz^T, then the RMSNorm backward on the lane's own half row
        // (one column tile of dy at a time)
        f32x16 dy;
        float du[KS][8];
        float cpart = 0.0f;
        static_for<KS>([&](auto kc) {
            constexpr int ks = decltype(kc)::value, ct = ks / 2;
            if constexpr (ks % 2 == 0) {
#pragma unroll
                for (int i = 0; i < 16; ++i) dy[i] = 0.0f;
#pragma unroll
                for (int q = 0; q < 2 * NT; ++q)
                    dy = mfma32(*reinterpret_cast<const bf16x8*>(sC + ((ct * 2 * NT + q) * 64 + lane) * 16), dzb[q >> 1][q & 1], dy);
            }
            [[maybe_unused]] f32x4 w0, w1, prod[2];
            if constexpr (NORM) {
                w0 = *reinterpret_cast<const f32x4*>(sW + (2 * ks + g) * 8);
                w1 = *reinterpret_cast<const f32x4*>(sW + (2 * ks + g) * 8 + 4);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                float d = dy[8 * (ks & 1) + j] + bf_at(dqr[ks], j);
                if constexpr (NORM) {
                    const float u = bf_at(T.xr[ks], j) * T.rstd;
                    if constexpr (AHEAD) {
                        if (valid) dwacc[ks][j] = fmaf(d, u, dwacc[ks][j]);
                    } else {
                        prod[j >> 2][j & 3] = valid ? d * u : 0.0f;
                    }
                    d *= (j < 4 ? w0[j & 3] : w1[j & 3]);
                    cpart = fmaf(d, u, cpart);
                }
                du[ks][j] = d;
            }
            if constexpr (NORM && !AHEAD) {
                // 64 columns of the products at a time (chunk c of row r at c ^ (r % 16)) into the y tile, which has been
                // read, and down the columns
                constexpr int half = ks / 4, c0 = 4 * (ks % 4);
                unsigned char* ptile = ytile;
#pragma unroll
                for (int q = 0; q < 2; ++q) *reinterpret_cast<f32x4*>(ptile + (prow ^ ((c0 + q) << 4))) = prod[q];
                if constexpr (ks % 4 == 3 || ks == KS - 1) {
#pragma unroll
                    for (int k = 0; k < 8; ++k)      // (lanes of columns beyond d_h add up what nobody reads)
                        dwcol[half] += *reinterpret_cast<const f32x4*>(ptile + k * 1024 + (pread ^ ((k & 3) << 6)));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        next_phase();
        if constexpr (NORM) {
            cpart += __shfl_xor(cpart, 32);
            const float c = cpart / (float)DH;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    du[ks][j] = T.rstd * (du[ks][j] - bf_at(T.xr[ks], j) * T.rstd * c);
        }
        auto out = [&](int ks) {
            bf16x8 o;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = (bf16_t)du[ks][j];
            return o;
        };
        if constexpr (WHOLE) {
            using Rows = RowTile<DH>;
            bf16_t* d0 = p.dX + (((long)b * p.S + tile * 32) * p.H + h) * DH;
            const int nrow = min(32, p.S - tile * 32);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) *reinterpret_cast<bf16x8*>(ytile + Rows::half(ks, l32, g)) = out(ks);
#pragma unroll
            for (int i = 0; i < Rows::INS; ++i) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(ytile + i * 1024 + lane * 16);
                if (Rows::row(i, lane) < nrow)
                    store_past(d0 + (long)Rows::row(i, lane) * (p.H * DH) + Rows::chunk(i, lane) * 8, v);
            }
        } else if (valid) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) *reinterpret_cast<bf16x8*>(p.dX + row + (2 * ks + g) * 8) = out(ks);
        }
    }

    // ---- sums over tokens: the waves' partials meet in LDS, then leave as one atomic add or one partial sum per workgroup
    // and element --------------------------------------------------------------------------------------------------------
    __syncthreads();   // every wave is past its last tile: the per-wave regions are free
    float* mine = reinterpret_cast<float*>(ytile);
    float* part = p.part ? p.part + (((long)h * gridDim.y + b) * p.wgs + wg) * (DH * p.E + DH) : nullptr;
    float* dWr = p.dWr + (long)h * DH * p.E;
    auto put = [&](int nt, int idx, float v) {      // value idx of expert tile nt: lane idx % 64, register idx / 64 % 16, column tile
        const int ln = idx & 63, i = (idx >> 6) & 15, ct = idx >> 10;
        const int e = nt * 32 + (ln & 31), col = ct * 32 + 8 * (i >> 2) + 4 * (ln >> 5) + (i & 3);
        if (e >= p.E) return;
        if (part) part[col * p.E + e] = v;
        else unsafeAtomicAdd(dWr + (long)col * p.E + e, v);
    };
    {
        if constexpr (!AHEAD) {
            if constexpr (GROUPS == 1) {      // (a wave's sums are those of the workgroup)
                if (wave < CT)
#pragma unroll
                    for (int i = 0; i < 16; ++i) put(0, (wave * 16 + i) * 64 + lane, wacc[0][0][i]);
            } else {
                float* sums = reinterpret_cast<float*>(regions);      // [GROUPS][CT][16][64]
                if (wave < GROUPS * CT)
#pragma unroll
                    for (int i = 0; i < 16; ++i) sums[(wave * 16 + i) * 64 + lane] = wacc[0][0][i];
                __syncthreads();
                for (int idx = threadIdx.x; idx < CT * 16 * 64; idx += 64 * NW) {
                    float v = 0.0f;
#pragma unroll
                    for (int q = 0; q < GROUPS; ++q) v += sums[q * CT * 1024 + idx];
                    put(0, idx, v);
                }
                __syncthreads();
            }
        } else {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
                for (int ct = 0; ct < WCT; ++ct)
#pragma unroll
                    for (int i = 0; i < 16; ++i) mine[(ct * 16 + i) * 64 + lane] = wacc[ct][nt][i];
                __syncthreads();
                for (int idx = threadIdx.x; idx < CT * 16 * 64; idx += 64 * NW) {
                    float v = 0.0f;
#pragma unroll
                    for (int w = 0; w < NW; ++w) v += reinterpret_cast<const float*>(regions + w * REGION_B)[idx];
                    put(nt, idx, v);
                }
                __syncthreads();
            }
        }
        if constexpr (NORM) {
            float* cross = reinterpret_cast<float*>(regions + NW * REGION_B);   // [NW waves][128 columns]
            if constexpr (AHEAD) {
                // transpose inside the wave: value v = 8 ks + j of every lane goes to row v (row stride 65 floats keeps both
                // the writes and the row-wise reads conflict-free), then lane v adds up each lane half of its row
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int j = 0; j < 8; ++j) mine[(ks * 8 + j) * 65 + lane] = dwacc[ks][j];
                if (lane < KS * 8) {
                    float s0 = 0.0f, s1 = 0.0f;
                    for (int i = 0; i < 32; ++i) {
                        s0 += mine[lane * 65 + i];
                        s1 += mine[lane * 65 + 32 + i];
                    }
                    const int ks = lane >> 3, j = lane & 7;
                    cross[wave * 128 + (2 * ks) * 8 + j] = s0;
                    cross[wave * 128 + (2 * ks + 1) * 8 + j] = s1;
                }
            } else {
#pragma unroll
                for (int i = 0; i < NHALF; ++i) {
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        float v = dwcol[i][x];
                        v += __shfl_xor(v, 16);
                        v += __shfl_xor(v, 32);
                        if (lane < 16 && 64 * i + 4 * lane < DH) cross[wave * 128 + 64 * i + 4 * lane + x] = v;
                    }
                }
            }
            __syncthreads();
            if (threadIdx.x < DH) {
                float v = 0.0f;
#pragma unroll
                for (int w = 0; w < NW; ++w) v += cross[w * 128 + threadIdx.x];
                if (part) part[DH * p.E + threadIdx.x] = v;
                else unsafeAtomicAdd(p.dWn + h * DH + threadIdx.x, v);
            }
        }
    }
}

// Adds the workgroups' sums of a head (in order) and writes d_router and d_norm_weight in the parameters' types.  The head runs fastest over
// the workgroups, as it does there for few tokens.
__global__ __launch_bounds__(256) void mhffn_gate_sum_kernel(const float* part, void* dWn, int wn_bf16, void* dWr, int wr_bf16, int dh,
                                                             int E, int wgs)
{
    const int i = blockIdx.y * 256 + threadIdx.x, h = blockIdx.x, nr = dh * E, n = nr + dh;
    if (i >= n || (i >= nr && !dWn)) return;
    const float* src = part + (long)h * wgs * n + i;
    const float v = sum_in_order(0.0f, 0, wgs, [&](int w) { return src[(long)w * n]; });
    const bool r = i < nr;
    void* dst = r ? dWr : dWn;
    const long at = r ? (long)h * nr + i : (long)h * dh + i - nr;
    if (r ? wr_bf16 : wn_bf16) static_cast<bf16_t*>(dst)[at] = (bf16_t)v;
    else static_cast<float*>(dst)[at] = v;
}

// ---- launch ---------------------------------------------------------------------------------------------------------
namespace {

// Tiles a wave takes.  Forward: several waves per SIMD hide the latency, so a wave only takes several tiles once there
// are at least 8 waves per SIMD; backward: as many waves (and partial sums) as fill the chip once, but for what is left over in a
// second round of workgroups.  A compute unit holds one of eight waves, and one of four with more than 32 experts; with up to
// 32 it holds two of four (LDS and registers), and those, fewer than 1,024 tiles, never need a second round.  A round is priced at
// 6 us and 8.5 for each of its waves' tiles (heads of 128, 11 experts).
// 12,288 tokens of 8 heads of 128: 34.1 us in 384 workgroups of eight waves and one tile per wave, 28.4 in 192 of two; of 64 24.0, 20.5;
// 9,000 of 16 heads of 96 44.0, 33.0; 8,500 of 8 heads of 128 with 40 experts 129, 102.  Two workgroups per compute unit: 3 x 1,300 tokens of
// 8 heads of 128 19.6 in 264 workgroups of four waves, 20.8 in 144 of two tiles per wave; of 64 15.1, 15.9.
int tiles_per_wave(int B, int H, int S, int waves, long cap)
{
    const long total = (long)B * H * ((S + 31) / 32);
    const long tpw = total / waves;
    return (int)(tpw < 1 ? 1 : tpw > cap ? cap : tpw);
}
// Waves of a backward workgroup.  Few tokens run with four also where up to 32 experts leave room for eight: with eight they fill
// less than half the chip, and a workgroup's tiles share its barriers and its LDS.  The backward's two kernels, us, with eight and with
// four waves: 16 tiles of 8 heads of 128 (11 experts) 16.3, 13.1; 64 tiles of 8 heads 17.2, 13.9; 20 tiles of 8 heads of 96 15.1, 12.6;
// 63 of 16 heads of 128 (22 experts) 18.9, 16.6; one tile 12.1, 11.9.  With more the second set of partial sums costs more than it
// gives: 122 tiles of 16 heads 21.3, 22.9.
int gate_bwd_waves(const Dims& d) { return d.E > 32 || (long)d.B * d.H * ((d.S + 31) / 32) < 4 * CUS ? 4 : 8; }
dim3 gate_bwd_grid(const Dims& d, int& tpw)
{
    const int nw = gate_bwd_waves(d), ntiles = (d.S + 31) / 32;
    auto workgroups = [&](int t) { return (ntiles + nw * t - 1) / (nw * t); };
    const int at_once = (nw == 4 && d.E <= 32 ? 2 : 1) * CUS;
    auto rounds = [&](int t) { return ((long)d.B * d.H * workgroups(t) + at_once - 1) / at_once; };
    tpw = tiles_per_wave(d.B, d.H, d.S, nw * CUS, 64);
    for (int t = tpw + 1; t <= 64 && rounds(t - 1) > 1 && workgroups(t - 1) > 1; ++t)
        if (rounds(t) * (6 + 8.5 * t) < rounds(tpw) * (6 + 8.5 * tpw)) tpw = t;
    return dim3(workgroups(tpw), d.H, d.B);
}

}  // namespace

// whole rows from four tiles per compute unit on (us in pieces / whole: 752 tiles of 8 heads of 128 6.7 / 7.2, 1,256 8.7 / 7.4, 2,000 of 16 9.9 / 8.1;
// 1,024 of 8 heads of 96 6.4 / 6.2)
// Not with more than 32 experts, whose arithmetic hides the pieces (4,096 tiles of 4 heads of 64 with 40 16.3 / 17.4, of 8 of 128 25.2 / 26.0),
// nor with 32 or, below d_h 128, 16: their rows of R share LDS banks, and the way through LDS waits for their writes (16,384 tiles of
// 12 heads of 128 with 32 + 9 %, of 96 + 9 %; 12,288 of 96 with 16 35.3 / 36.0).
bool gate_fwd_whole_rows(const Dims& d)
{
    return d.E <= 32 && (d.E % 16 != 0 || (d.d_h == 128 && d.E == 16)) && (long)d.B * d.H * ((d.S + 31) / 32) >= 4 * CUS;
}
bool gate_bwd_whole_rows(const Dims& d) { return gate_bwd_waves(d) == 8; }

namespace {

template <int DH, int NT, bool NORM>
hipError_t launch_gate(GateArgs a, const Dims& d, bool backward, hipStream_t st)
{
    static LdsOptIn optin_fwd[2], optin_bwd[2];
    if (backward) {
        const int waves = gate_bwd_waves(d), smem = (int)gate_bwd_smem<NT>(DH, waves);
        const dim3 grid = gate_bwd_grid(d, a.tpw);      // (workgroups of a head and batch, heads, batches)
        a.wgs = grid.x;
        a.heads_first = NT > 1 || a.tpw < 4;
        a.by_fast = FastDiv(a.heads_first ? a.H : a.wgs);
        const bool whole = gate_bwd_whole_rows(d);
        auto* fn = whole ? mhffn_gate_bwd_kernel<DH, 1, NORM, WholeRows> : mhffn_gate_bwd_kernel<DH, NT, NORM>;
        const hipError_t e = ensure_dynamic_lds(optin_bwd[whole], (const void*)fn, smem);
        if (e != hipSuccess) return e;
        // Up to three tiles per wave (and with more than 32 experts) the workgroups of a head run on one XCD, if heads are a multiple of eight: its sums are still in that L2 when the
        // pass behind reads them, and dQ, dR where the operator left them.  Both kernels, us, head by head / so: 16 tokens of 16 heads of 128
        // 13.6 / 12.4, 512 of 8 13.0 / 12.8, 3,000 14.7 / 14.0, 5,000 17.8 / 17.1, 7,001 of 64 13.6 / 12.9, 16,384 20.2 / 19.8, of 128 30.0 / 30.1.  Of many rows
        // a head's workgroups in turn read faster: 32,768 tokens of 16 heads 103.3, in that order 107.2.
        hipLaunchKernelGGL(fn, dim3(grid.x * d.H, d.B), dim3(64 * waves), smem, st, a);
    } else {
        const size_t smem = gate_fwd_smem(DH, NT);
        const bool whole = gate_fwd_whole_rows(d);
        auto* fn = whole ? mhffn_gate_fwd_kernel<DH, 1, NORM, WholeRows> : mhffn_gate_fwd_kernel<DH, NT, NORM>;
        const hipError_t e = ensure_dynamic_lds(optin_fwd[whole], (const void*)fn, (int)smem);
        if (e != hipSuccess) return e;
        a.tpw = tiles_per_wave(a.B, a.H, a.S, 8192, 16);
        const dim3 grid(((a.S + 31) / 32 + 4 * a.tpw - 1) / (4 * a.tpw), a.H, a.B);
        hipLaunchKernelGGL(fn, grid, dim3(256), smem, st, a);
    }
    return hipGetLastError();
}

template <int DH>
hipError_t launch_gate_dh(const GateArgs& a, const Dims& d, bool backward, hipStream_t st)
{
    const bool norm = a.Wn != nullptr;
    if (a.E <= 32) return norm ? launch_gate<DH, 1, true>(a, d, backward, st) : launch_gate<DH, 1, false>(a, d, backward, st);
    return norm ? launch_gate<DH, 2, true>(a, d, backward, st) : launch_gate<DH, 2, false>(a, d, backward, st);
}

hipError_t launch_gate_any(const GateArgs& a, const Dims& d, bool backward, hipStream_t st)
{
    switch (d.d_h) {
        case 64: return launch_gate_dh<64>(a, d, backward, st);
        case 96: return launch_gate_dh<96>(a, d, backward, st);
        case 128: return launch_gate_dh<128>(a, d, backward, st);
    }
    return hipErrorInvalidValue;
}

int gate_bwd_workgroups(const Dims& d)      // of one head
{
    int tpw;
    const dim3 g = gate_bwd_grid(d, tpw);
    return (int)(g.x * g.z);
}

}  // namespace

hipError_t launch_gate_fwd(const void* X, const void* Wn, int wn_bf16, float eps, const void* Wr, int wr_bf16, void* Qn, float* R,
                           const Dims& d, hipStream_t st)
{
    GateArgs a{};
    a.X = (const bf16_t*)X;
    a.Wn = Wn;
    a.Wr = Wr;
    a.wn_bf16 = wn_bf16;
    a.wr_bf16 = wr_bf16;
    a.Qn = (bf16_t*)Qn;
    a.R = R;
    a.B = d.B, a.H = d.H, a.S = d.S, a.E = d.E, a.eps = eps;
    return launch_gate_any(a, d, false, st);
}

size_t gate_bwd_workspace_bytes(const Dims& d)
{
    return (size_t)d.H * gate_bwd_workgroups(d) * (d.d_h * d.E + d.d_h) * sizeof(float);
}

hipError_t launch_gate_bwd(const void* X, const void* Wn, int wn_bf16, float eps, const void* Wr, int wr_bf16, const void* dQ,
                           int dq_tokmaj, const float* dR, void* dX, void* dWn, void* dWr, void* ws, const Dims& d, hipStream_t st)
{
    GateArgs a{};
    a.X = (const bf16_t*)X;
    a.Wn = Wn;
    a.Wr = Wr;
    a.wn_bf16 = wn_bf16;
    a.wr_bf16 = wr_bf16;
    a.dQ = (const bf16_t*)dQ;
    a.dR = dR;
    a.dX = (bf16_t*)dX;
    a.part = (float*)ws;
    if (!ws) {
        a.dWn = (float*)dWn;
        a.dWr = (float*)dWr;
    }
    a.dq_tokmaj = dq_tokmaj;
    a.B = d.B, a.H = d.H, a.S = d.S, a.E = d.E, a.eps = eps;
    hipError_t err = launch_gate_any(a, d, true, st);
    if (err != hipSuccess || !ws) return err;
    const dim3 grid(d.H, (d.d_h * d.E + d.d_h + 255) / 256);
    const int wgs = gate_bwd_workgroups(d);
    hipLaunchKernelGGL(mhffn_gate_sum_kernel, grid, dim3(256), 0, st, a.part, Wn ? dWn : nullptr, wn_bf16, dWr, wr_bf16, d.d_h, d.E, wgs);
    return hipGetLastError();
}

}  // namespace mhffn
