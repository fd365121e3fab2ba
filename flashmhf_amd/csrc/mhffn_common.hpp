// Shared device/host definitions for the gfx950 fused multi-head FFN kernels.
//
// Tile vocabulary used by every kernel in this directory
// -------------------------------------------------------
// * "j" indexes rows of K/U/V inside one expert (the d_e axis), "c" indexes the head dim (d_h), "t" a token.
// * The d_e axis is processed in blocks of JB = 32 rows; blocks never straddle experts (d_e % 32 == 0).
// * All matrix products use v_mfma_f32_32x32x16_bf16.  For one instruction D = A(32x16) * B(16x32) + C:
//       A: lane l holds row (l % 32), k = 8*(l / 32) .. +7        (8 bf16 = 4 VGPRs)
//       B: lane l holds col (l % 32), k = 8*(l / 32) .. +7
//       C/D: lane l holds col (l % 32), register i (0..15) holds row 8*(i/4) + 4*(l/32) + (i%4)
// * Chained products keep the first product's C registers as the second product's B operand without a trip
//   through LDS: with the first product written "transposed" (rows = j, cols = t) registers 8s..8s+7 of lane
//   (t, g = l/32) are exactly the 8 k-slots the second product's B operand wants, provided slot (s, g, kk)
//   means j = 16s + 8g + kk.  That holds when output row rho of the first product was fed K row
//   PI(rho) (see row_perm32): the permutation is applied in the LDS read address of the K/U/V tiles.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <atomic>
#include <type_traits>

namespace mhffn {

typedef __bf16 bf16_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));   // 16-byte copy unit (native vector: stays in registers)

constexpr int JB = 32;          // rows of K/U/V per block
// Experts whose gate values the forward and the dQ/dR kernel keep in LDS at a time ([GATE_WIN][256 tokens] fp32 = 64 KB,
// next to the 96 KB weight ring); a power of two.  With more experts the forward restages the tile every GATE_WIN experts
// (a multiple of four blocks whatever d_e is, so every window starts on its LDS stage 0) and the dQ/dR kernel refills it
// as a ring, expert e in slot e % GATE_WIN.
constexpr int GATE_WIN = 64;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float FLT_MAX_F = 3.402823466e+38f;

// MFMA output row rho (0..31) -> which row of the 32-row weight block must be fed as A-row rho so that
// C registers 8s..8s+7 of lane group g hold j = 16s + 8g + kk.  rho = 8a + 4g + b  ->  16(a/2) + 8g + 4(a%2) + b.
__host__ __device__ constexpr int row_perm32(int rho)
{
    return 16 * ((rho >> 3) >> 1) + 8 * ((rho >> 2) & 1) + 4 * ((rho >> 3) & 1) + (rho & 3);
}

// Position p (0..31) inside a transposed token tile -> token it holds, so that B-operand k-slot (s, g, kk) of a
// [t, j] product's C registers (token 16s + 8(kk/4) + 4g + kk%4) lines up with 8 contiguous positions 16s + 8g + kk.
__host__ __device__ constexpr int tok_perm32(int p)
{
    return (p & 16) + 8 * ((p >> 2) & 1) + 4 * ((p >> 3) & 1) + (p & 3);
}

// Compile-time loop: f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>).  Arrays indexed through it are
// indexed by constants from the first optimisation pass on, so they are promoted to registers (never scratch).
template <int I, int N>
struct StaticFor {
    template <class F>
    __device__ __forceinline__ static void run(F&& f)
    {
        f(std::integral_constant<int, I>{});
        StaticFor<I + 1, N>::run(f);
    }
};
template <int N>
struct StaticFor<N, N> {
    template <class F>
    __device__ __forceinline__ static void run(F&&) {}
};
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    StaticFor<0, N>::run(f);
}

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// The same instruction with its accumulator forced into architectural VGPRs (the compiler picks one register file for
// the accumulators of all builtin MFMAs of a kernel; a one-wave-per-SIMD kernel gets AGPRs, from which every value the
// VALU needs costs a v_accvgpr_read).  Used for products whose result feeds element-wise VALU work directly.
// The compiler cannot see that this is an MFMA, so the caller must leave the required wait states between the last of
// these and the first VALU read of the result (mfma_result_fence).  A/B operand waits (LDS loads) are still inserted
// by the compiler, back-to-back accumulation into the same registers is interlocked by hardware.
__device__ __forceinline__ void mfma32_vgpr_first(f32x16& d, bf16x8 a, bf16x8 b)
{
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma32_vgpr_acc(f32x16& d, bf16x8 a, bf16x8 b)
{
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
}
// Same, with the B operand held in an accumulation register (AGPRs are legal MFMA A/B sources): used for operands that
// stay resident for a whole kernel, so they do not compete with the VALU's working set for architectural VGPRs.
__device__ __forceinline__ void mfma32_vgpr_first_bacc(f32x16& d, bf16x8 a, bf16x8 b)
{
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma32_vgpr_acc_bacc(f32x16& d, bf16x8 a, bf16x8 b)
{
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma_result_fence(f32x16& a, f32x16& b, f32x16& c)
{
    // 8-pass MFMA result -> VALU read needs at most 18 wait states on gfx940-class hardware; leave 32.  The results
    // are operands of the statement, so no read of them can be scheduled above it.
    asm volatile("s_nop 15\n\ts_nop 15" : "+v"(a), "+v"(b), "+v"(c));
}
__device__ __forceinline__ void mfma_result_fence(f32x16& a, f32x16& b)
{
    asm volatile("s_nop 15\n\ts_nop 15" : "+v"(a), "+v"(b));
}
// Never pass the same object twice to one fence: the compiler would materialise the extra operands as register copies
// of the result, and those copies are VALU reads issued before the wait states have passed.
__device__ __forceinline__ void mfma_result_fence(f32x16& a)
{
    asm volatile("s_nop 15\n\ts_nop 15" : "+v"(a));
}

__device__ __forceinline__ float fast_sigmoid(float x)
{
    // 1 / (1 + 2^(-x log2 e)): v_mul, v_exp_f32, v_add, v_rcp_f32.  x -> -inf gives rcp(inf) = 0, x -> +inf gives 1.
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-LOG2E * x));
}

// ---- LDS tile layout shared by the main kernels -------------------------------------------------------------------
// A staged tile is 32 rows (weight rows j, or tokens) of 256 bytes: 16 chunks of 8 bf16, d_h/8 of them used.  The chunk
// holding columns [8c, 8c+8) of row r sits at chunk position c ^ swz16(r).  With this XOR swizzle both access patterns
// -- 16-byte row reads (16 lanes = 16 different rows, same column chunk) and transposing 8-byte reads (a 16-lane group
// reads 4 consecutive rows x 32 contiguous bytes) -- are bank-conflict free without padding, so tiles can be filled
// by global_load_lds_dwordx4, whose LDS destination is (wave-uniform base) + lane * 16.
constexpr int TILE_ROW_B = 256;
constexpr int TILE_B = JB * TILE_ROW_B;   // 8 KB

__device__ __forceinline__ int swz16(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 v4bf16_t;

// One wave-instruction of an asynchronous tile fill: 4 rows (ins*4 .. ins*4+3) of a row-major [32][DH] bf16 source
// tile whose row `r` starts at src_row0 + r * row_stride (elements).  Counts as one vmcnt event.  PAST: the caches need not keep the rows.
template <int DH, bool PAST = false>
__device__ __forceinline__ void tile_fill_ins(const bf16_t* src_row0, long row_stride, unsigned char* lds_tile, int ins,
                                              int lane)
{
    const int r = 4 * ins + (lane >> 4);
    int c = (lane & 15) ^ swz16(r);
    c = c < DH / 8 ? c : 0;   // chunk positions a narrow row does not use receive a dummy chunk
    __builtin_amdgcn_global_load_lds((gptr_t)(src_row0 + r * row_stride + c * 8), (lptr_t)(lds_tile + ins * 1024), 16, 0,
                                     PAST ? 2 : 0);      // (the instruction's nt bit)
}

// A operand (32 rows x 16 k) for k-step ks from a swizzled tile, row-major use: lane holds row `row`, columns
// 16ks + 8g .. +7.
__device__ __forceinline__ bf16x8 tile_read_rows(const unsigned char* tile, int row, int ks, int g)
{
    return *reinterpret_cast<const bf16x8*>(tile + row * TILE_ROW_B + (((2 * ks + g) ^ swz16(row)) << 4));
}

// A operand (32 rows = tile columns 32ct + l32, 16 k = tile rows) from a swizzled tile, transposed use:
// lane holds column 32ct + l32; its 8 k values are tile rows rlo + {0..3} then rhi + {0..3}.  rlo/rhi must be uniform
// within each 16-lane group (they may depend on lane / 32).
//
// The two ds_read_b64_tr_b16 are issued from inline assembly, not through the compiler builtin: behind the builtin the
// compiler cannot tell that the read does not touch the LDS stage an asynchronous LDS-direct load is filling, and puts
// a full s_waitcnt vmcnt(0) in front of it, which stalls every loop iteration for the whole global-memory latency.
// The price is that the compiler does not know these reads are in flight either: the consumer must call
// lds_tr_wait() on the operands before their first use.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
struct TrOperand {
    u32x2 lo, hi;
};
__device__ __forceinline__ unsigned lds_addr(const void* p)
{
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
// Per-lane byte offsets (inside a tile, for s = 0) of the two reads of a transposed operand, for every column tile ct.
// The tile rows a lane group reads are  16 s + RG * (lane / 32) + RH * hi + (lane % 16) / 4,  hi = 0, 1
//   (RG, RH) = (8, 4): k-slot (s, g, kk) is row 16 s + 8 g + kk            (weights: second products of fwd, dQ)
//   (RG, RH) = (4, 8): k-slot (s, g, kk) is row 16 s + 8 (kk / 4) + 4 g + kk % 4   (tokens: dK/dU/dV contraction)
// s only adds 16 rows = 4096 bytes (the swizzle has period 16 rows), which goes into the instruction's immediate offset.
template <int CT>
struct TrLane {
    unsigned off[CT][2];
};
template <int CT, int RG, int RH>
__device__ __forceinline__ TrLane<CT> make_tr_lane(int lane)
{
    TrLane<CT> t;
    const int lam = lane & 15, l32 = lane & 31, g = lane >> 5;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
            const int r = RG * g + RH * hi + (lam >> 2);
            const int chunk = 4 * ct + 2 * (l32 >> 4) + ((lam & 3) >> 1);
            t.off[ct][hi] = r * TILE_ROW_B + ((chunk ^ swz16(r)) << 4) + (lam & 1) * 8;
        }
    return t;
}
// Requests operand (ct, s) of the tile at LDS byte address `tile_addr` (wave-uniform); IMM = 4096 * s + any
// compile-time displacement (must stay below 65536 together).
template <int IMM, int CT>
__device__ __forceinline__ TrOperand tile_read_cols_async(unsigned tile_addr, const TrLane<CT>& tl, int ct)
{
    const unsigned a0 = tile_addr + tl.off[ct][0], a1 = tile_addr + tl.off[ct][1];
    TrOperand t;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(t.lo) : "v"(a0), "n"(IMM));
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(t.hi) : "v"(a1), "n"(IMM));
    return t;
}
// Waits for every LDS operation of this wave (lgkmcnt(0)); the operands are inputs and outputs of the statement, so no
// use of them can be scheduled above it.
__device__ __forceinline__ void lds_tr_wait(TrOperand& a)
{
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a.lo), "+v"(a.hi));
}
__device__ __forceinline__ void lds_tr_wait(TrOperand& a, TrOperand& b)
{
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a.lo), "+v"(a.hi), "+v"(b.lo), "+v"(b.hi));
}
__device__ __forceinline__ void lds_tr_wait(TrOperand& a, TrOperand& b, TrOperand& c, TrOperand& d)
{
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(a.lo), "+v"(a.hi), "+v"(b.lo), "+v"(b.hi), "+v"(c.lo), "+v"(c.hi), "+v"(d.lo), "+v"(d.hi));
}
// Partial wait: at most N LDS operations of this wave still outstanding.  Only exact inside a region that the caller
// has fenced with sched_barrier(0) and that contains no other LDS instruction than the asynchronous reads above
// (LDS operations complete in order; each TrOperand is two of them).
template <int N>
__device__ __forceinline__ void lds_tr_wait_n(TrOperand& a, TrOperand& b)
{
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(a.lo), "+v"(a.hi), "+v"(b.lo), "+v"(b.hi) : "n"(N));
}
// The same for 16 contiguous bytes per lane (a row-major A operand as in tile_read_rows, four gate values): issued from
// inline assembly so that the waits in front of the uses can be partial -- the compiler's own bookkeeping puts a full
// lgkmcnt(0) in front of the first use of any read of a group in flight.  IMM: compile-time displacement.
template <int IMM>
__device__ __forceinline__ u32x4 lds_read16_async(unsigned addr)
{
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(IMM));
    return v;
}
// N 4-byte values per lane, 128 bytes apart (one instruction, one LDS operation); for N = 1 the same one twice, so that the read fills
// both registers of the result: put together from a single one, the compiler copied that one before the read had returned.
template <int N>
__device__ __forceinline__ u32x2 lds_read_apart_async(unsigned addr)
{
    u32x2 v;
    asm volatile("ds_read2_b32 %0, %1 offset1:%2" : "=v"(v) : "v"(addr), "n"(32 * (N - 1)));
    return v;
}
// At most N LDS operations of this wave still outstanding; the operands cannot be used above it.  Same conditions as
// lds_tr_wait_n.
template <int N>
__device__ __forceinline__ void lds_wait_n(u32x4& a, u32x4& b, u32x2& c)
{
    asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(a), "+v"(b), "+v"(c) : "n"(N));
}
// The same without operands, for reads whose only consumers are matrix instructions issued from inline assembly (volatile
// statements keep their order): with the operands tied to the wait the compiler assumes the statement wrote them and puts
// a hazard s_nop in front of the matrix instruction.
template <int N>
__device__ __forceinline__ void lds_wait_n()
{
    asm volatile("s_waitcnt lgkmcnt(%0)" :: "n"(N));
}
template <int N>
__device__ __forceinline__ void lds_wait_n(u32x4& a, u32x4& b, u32x4& c, u32x4& d, u32x4& e, u32x4& f)
{
    asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(a), "+v"(b), "+v"(c), "+v"(d), "+v"(e), "+v"(f) : "n"(N));
}
__device__ __forceinline__ bf16x8 tr_value(const TrOperand& t)
{
    u32x4 v = {t.lo[0], t.lo[1], t.hi[0], t.hi[1]};
    return __builtin_bit_cast(bf16x8, v);
}

// Stores 32 rows of DH fp32 values held as accumulator tiles of a transposed product (acc(i), row tile i: register 4a + x of
// lane (l32, g) is column 32i + 8a + 4g + x of row l32) to dst[row][DH], rows below nrows.  Stored straight from the registers
// these would be 32-byte pieces of 32 rows per instruction (23 MB of partial sums of the forward took 10 us longer that
// way); they go 64 columns at a time through 8 KB of LDS private to the wave (256-byte rows, 16-byte chunk c of row r at
// c ^ (r & 15)) and leave as 256-byte runs, 4 rows per instruction.  LDS operations of one wave complete in order.
template <int DH, class Acc>
__device__ __forceinline__ void store_rows_f32(unsigned char* region, float* dst, int nrows, int lane, Acc&& acc)
{
    constexpr int CT = DH / 32;
    const int l32 = lane & 31, g = lane >> 5, c16 = lane & 15;
    if (nrows <= 0) return;
    static_for<(CT + 1) / 2>([&](auto hc) {
        constexpr int h = decltype(hc)::value, NT = 2 * h + 1 < CT ? 2 : 1;
        static_for<NT>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const f32x16& v16 = acc(std::integral_constant<int, 2 * h + i>{});
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                f32x4 v;
#pragma unroll
                for (int x = 0; x < 4; ++x) v[x] = v16[4 * a + x];
                *reinterpret_cast<f32x4*>(region + l32 * 256 + (((8 * i + 2 * a + g) ^ (l32 & 15)) << 4)) = v;
            }
        });
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int row = 4 * k + (lane >> 4);
            if (c16 < 8 * NT && row < nrows)
                *reinterpret_cast<f32x4*>(dst + row * DH + 64 * h + 4 * c16) =
                    *reinterpret_cast<const f32x4*>(region + row * 256 + ((c16 ^ (row & 15)) << 4));
        }
    });
}

// ---- tiles of 32 rows, a wave per block -----------------------------------------------------------------------------
// With few rows the tiles of 128 and 256 rows leave most of the chip idle, and a workgroup walks a head's blocks one after
// the other.  The rows32 kernels put four waves of a workgroup on four consecutive blocks of the same 32 rows instead:
// a wave takes the first products and the element-wise work of its own block, hands the rounded result to the others
// through LDS, and all blocks are added, in their order, by a wave for each 32 output columns (the forward of short parts: the same
// waves, four blocks at a time; the others: four more waves, one block at a time): the sums are those of the kernels with larger
// tiles bit for bit.
// Every LDS access of their loops is inline assembly and every wait counted by hand: the compiler would put a wait for all
// outstanding LDS-direct loads in front of each access.
constexpr int QUAD = 4;                      // waves of a workgroup of the forward = blocks of a trip

// Asynchronous fill of one 32-row tile by one wave: eight vmcnt events.
template <int DH, bool PAST>
__device__ __forceinline__ void quad_fill(const bf16_t* src, unsigned char* tile, int lane)
{
#pragma unroll
    for (int i = 0; i < 8; ++i) tile_fill_ins<DH, PAST>(src, DH, tile, i, lane);
}
// Asynchronous fills of a block's K, U and V tiles by four waves, each a quarter of every tile: two vmcnt events a tile.  A lane's
// place in a tile is a 32-bit offset to a uniform base (a narrow row's unused chunks take chunk 0).  The tiles go round in KU sets
// of K | U and in NV sets of V; ku and v are the sets of the block behind the last one aimed at.
template <int DH, int KU, int NV>
struct QuadFill {
    const bf16_t* K;
    long offU, offV;          // U - K, V - K in bytes
    unsigned char *ku0, *v0, *to_ku, *to_v;
    const char* from;
    unsigned place[2];
    int nblk, ku, v;
    __device__ __forceinline__ QuadFill(const bf16_t* K_, long offU_, long offV_, int nblk_, unsigned char* ku0_, unsigned char* v0_, int quarter,
                                        int lane)
        : K(K_), offU(2 * offU_), offV(2 * offV_), ku0(ku0_ + 2 * quarter * 1024), v0(v0_ + 2 * quarter * 1024), nblk(nblk_), ku(0), v(0)
    {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = 4 * (2 * quarter + i) + (lane >> 4), c = (lane & 15) ^ swz16(row);
            place[i] = (row * DH + (c < DH / 8 ? c : 0) * 8) * 2;
        }
    }
    __device__ __forceinline__ void aim(int b)      // (behind the last block: the last one again)
    {
        from = reinterpret_cast<const char*>(K + (long)(b < nblk ? b : nblk - 1) * JB * DH);
        asm("" : "+s"(from));           // (kept apart from the lane's offset: one scalar addition per tile)
        to_ku = ku0 + ku * 2 * TILE_B;
        to_v = v0 + v * TILE_B;
        ku = ku + 1 == KU ? 0 : ku + 1;
        v = v + 1 == NV ? 0 : v + 1;
    }
    template <class T_, class I_>
    __device__ __forceinline__ void request(T_, I_)     // half I of this wave's part of K, U or V (T = 0, 1, 2)
    {
        constexpr int T = T_::value, I = I_::value;
        const char* src = from + (T == 0 ? 0 : T == 1 ? offU : offV);
        unsigned char* dst = (T == 2 ? to_v : to_ku + T * TILE_B) + I * 1024;
        __builtin_amdgcn_global_load_lds((gptr_t)(src + place[I]), (lptr_t)dst, 16, 0, 0);
    }
};
// The transposed operands' places for one column tile.
template <int CT>
__device__ __forceinline__ TrLane<1> quad_tr_lane(int lane, int col)
{
    const TrLane<CT> all = make_tr_lane<CT, 8, 4>(lane);
    TrLane<1> t{};
#pragma unroll
    for (int i = 0; i < CT; ++i)
        if (i == col) { t.off[0][0] = all.off[i][0]; t.off[0][1] = all.off[i][1]; }
    return t;
}
template <int IMM, class T>
__device__ __forceinline__ void lds_write16(unsigned addr, const T& v)
{
    asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(addr), "v"(__builtin_bit_cast(u32x4, v)), "n"(IMM));
}
__device__ __forceinline__ void lds_write4(unsigned addr, float v) { asm volatile("ds_write_b32 %0, %1" ::"v"(addr), "v"(v)); }
// This wave's LDS operations are done, then the workgroup's; loads in flight stay in flight.
__device__ __forceinline__ void quad_barrier()
{
    __builtin_amdgcn_sched_barrier(0);
    lds_wait_n<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}
// Row-major operands of every k-step of up to three tiles (16-byte LDS reads, all requested before the first is used: the
// wave is alone on its SIMD), and the wait for k-step KSI of the N tiles.
template <int KS, int N>
struct QuadRows {
    u32x4 v[N][KS];
    template <int T, int KSI, int IMM = 0>
    __device__ __forceinline__ void request(unsigned rowaddr)      // address of the row's k-step 0 chunk position
    {
        v[T][KSI] = lds_read16_async<IMM>(rowaddr);
    }
    template <int KSI>
    __device__ __forceinline__ void wait()
    {
        constexpr int younger = (KS - 1 - KSI) * N < 15 ? (KS - 1 - KSI) * N : 15;
        lds_wait_n<younger>();
#pragma unroll
        for (int t = 0; t < N; ++t) asm volatile("" : "+v"(v[t][KSI]));
    }
    __device__ __forceinline__ bf16x8 get(int t, int ks) const { return __builtin_bit_cast(bf16x8, v[t][ks]); }
};
// Gate values of 32 rows, expert-major [nex][32]: R row address(t) of every row t (clamped by the caller), eight lanes per row.
template <class Row>
__device__ __forceinline__ void quad_stage_gates(float* sR, const float* R, int nex, int tid, Row&& address)
{
    const int t = tid >> 3;
    const float* src = R + address(t);
    for (int e = tid & 7; e < nex; e += 8) sR[e * 32 + t] = src[e];
}
// Stores a 32 x 32 tile held as an accumulator of a transposed product (register 4a + x of lane (l32, g): column 8a + 4g + x of
// row l32) through 4 KB of LDS private to the wave, rows below nrows: fp32 to dst(row), or rounded to bf16.
template <class Dst>
__device__ __forceinline__ void quad_store_f32(unsigned char* region, const f32x16& acc, int nrows, int lane, Dst&& dst)
{
    const int l32 = lane & 31, g = lane >> 5;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        f32x4 v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = acc[4 * a + x];
        *reinterpret_cast<f32x4*>(region + l32 * 128 + (((2 * a + g) ^ (l32 & 7)) << 4)) = v;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int row = 8 * k + (lane >> 3), c = lane & 7;
        if (row < nrows) *reinterpret_cast<f32x4*>(dst(row) + 4 * c) = *reinterpret_cast<const f32x4*>(region + row * 128 + ((c ^ (row & 7)) << 4));
    }
}
template <class Dst>
__device__ __forceinline__ void quad_store_bf16(unsigned char* region, const f32x16& acc, int nrows, int lane, Dst&& dst)
{
    const int l32 = lane & 31, g = lane >> 5;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        bf16x4 v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = (bf16_t)acc[4 * a + x];
        *reinterpret_cast<bf16x4*>(region + l32 * 64 + ((a ^ (l32 & 3)) << 4) + 8 * g) = v;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int row = 16 * k + (lane >> 2), c = lane & 3;
        if (row < nrows) *reinterpret_cast<u32x4*>(dst(row) + 8 * c) = *reinterpret_cast<const u32x4*>(region + row * 64 + ((c ^ (row & 3)) << 4));
    }
}

// s_waitcnt vmcnt(N) only (gfx9 encoding: vmcnt[3:0] at bits 3:0, vmcnt[5:4] at bits 15:14; other counters unconstrained).
template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// Dynamic LDS above 64 KB must be opted into per kernel function and per device.  One LdsOptIn per kernel function (static
// storage, zero-initialised) remembers the largest size already granted on each device, so the attribute call is made
// once per (kernel, device) whichever host thread launches first; a repeated call is harmless.
constexpr int LDS_OPTIN_MAX_DEVICES = 64;
struct LdsOptIn {
    std::atomic<int> granted[LDS_OPTIN_MAX_DEVICES];
};
inline hipError_t ensure_dynamic_lds(LdsOptIn& c, const void* fn, int bytes)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const bool tracked = dev >= 0 && dev < LDS_OPTIN_MAX_DEVICES;
    if (tracked && bytes <= c.granted[dev].load(std::memory_order_acquire)) return hipSuccess;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess && tracked) c.granted[dev].store(bytes, std::memory_order_release);
    return e;
}

// Host-side launch entry points (defined in the per-kernel .hip files).
struct Dims {
    int B, H, Hkuv, S, d_h, E, d_e;
    int tokmaj;   // layout of Q, O, dO, dQ: 0 = [B, H, S, d_h], 1 = [B, S, H, d_h] (token-major, heads interleaved)
};

// Rows (units of d_h elements) of Q/O/dO/dQ: token t of (batch b, q-head h) is row base + t * stride.
struct TokRows {
    long base;
    int stride;
};
__host__ __device__ inline TokRows tok_rows(int tokmaj, int b, int h, int H, int S)
{
    return tokmaj ? TokRows{(long)b * S * H + h, H} : TokRows{((long)b * H + h) * S, 1};
}

// Unsigned division by a fixed divisor, exact for dividends below 2^31 (the round-up method of Granlund and Montgomery,
// "Division by invariant integers using multiplication", 1994): q = (mulhi(n, m) + n) >> l with l = ceil(log2 d).
struct FastDiv {
    unsigned m, l;
    FastDiv() = default;
    explicit FastDiv(unsigned d)
    {
        l = 0;
        while ((1ull << l) < d) ++l;
        m = (unsigned)(((1ull << 32) * ((1ull << l) - d)) / d + 1);
    }
    __device__ __forceinline__ unsigned div(unsigned n) const { return (__umulhi(n, m) + n) >> l; }
};

// The rows that meet one K/U/V head: the B * S tokens of its G q-heads, numbered so that a tile of consecutive rows is as
// contiguous in memory as the layout allows ([B, H, S]: batch, then head of the group, then token; [B, S, H]: token,
// then head of the group).  The forward and the dQ/dR kernel tile this list instead of the tokens of one (batch, q-head):
// short sequences, decoded tokens and the heads of a group then share a tile and one pass over the weights.
struct RowMap {
    int tokmaj, H, Hkuv, G, S;
    int n;            // rows of the list: G * B * S
    FastDiv by_g, by_s, by_gs, by_hkuv;
    RowMap() = default;
    explicit RowMap(const Dims& d)
        : tokmaj(d.tokmaj), H(d.H), Hkuv(d.Hkuv), G(d.H / d.Hkuv), S(d.S), n(d.H / d.Hkuv * d.B * d.S), by_g(d.H / d.Hkuv), by_s(d.S),
          by_gs((unsigned)(d.H / d.Hkuv) * d.S), by_hkuv(d.Hkuv)
    {
    }
    // row of Q, O, dO, dQ (units of d_h elements)
    __device__ __forceinline__ long tok(int hk, unsigned r) const
    {
        if (tokmaj) {
            const unsigned t = by_g.div(r);
            return (long)t * H + hk * G + (r - t * G);
        }
        return head_major(hk, r);
    }
    // row of R, dR (units of E elements; always [B, H, S])
    __device__ __forceinline__ long gate(int hk, unsigned r) const
    {
        if (tokmaj) {
            const unsigned t = by_g.div(r), b = by_s.div(t);
            return ((long)b * H + hk * G + (r - t * G)) * S + (t - b * S);
        }
        return head_major(hk, r);
    }
    // The rows first .. first + count - 1 (those of the list; first < n) as base + i * stride where they are such a run of
    // Q, O, dO, dQ (tok) and of R, dR (gate); stride 0 where they are not.  Wave-uniform arguments: the kernels take the
    // addresses of a run without a division per lane and stored row, which a tile needs only where it mixes batches
    // (always divided, the twenty divisions of a wave cost the forward 1 % at 16,384 tokens).
    struct Run {
        TokRows tok, gate;
    };
    __device__ __forceinline__ Run run(int hk, unsigned first, unsigned count) const
    {
        const unsigned last = first + count <= (unsigned)n ? first + count - 1 : n - 1;
        const FastDiv& d = tokmaj ? by_s : by_gs;
        const bool one_batch = d.div(first) == d.div(last), ungrouped = !tokmaj || G == 1;
        return Run{TokRows{tok(hk, first), tokmaj ? (ungrouped ? H : 0) : one_batch},
                   TokRows{gate(hk, first), one_batch && ungrouped}};
    }
    __device__ __forceinline__ long tok(const Run& u, int hk, unsigned first, unsigned r) const
    {
        return u.tok.stride ? u.tok.base + (long)(r - first) * u.tok.stride : tok(hk, r);
    }
    __device__ __forceinline__ long gate(const Run& u, int hk, unsigned first, unsigned r) const
    {
        return u.gate.stride ? u.gate.base + (r - first) : gate(hk, r);
    }
    // The same rows in [B, H, S] order whatever the layout (sums over rows then have one order): row of Q, dO; the row of R
    // is head_major(hk, r).
    __device__ __forceinline__ long tok_head_major(int hk, unsigned r) const
    {
        if (!tokmaj) return head_major(hk, r);
        const unsigned b = by_gs.div(r), rem = r - b * (unsigned)(G * S), gi = by_s.div(rem);
        return ((long)b * S + (rem - gi * S)) * H + hk * G + gi;
    }
    __device__ __forceinline__ long head_major(int hk, unsigned r) const
    {
        const unsigned b = by_gs.div(r);
        return ((long)b * Hkuv + hk) * ((long)G * S) + (r - b * (unsigned)(G * S));
    }
};

// The E * nbe blocks of a head (nbe = d_e / 32 per expert) in nsplit parts of consecutive blocks.
struct Parts {
    int E, nbe, nsplit;
    FastDiv by_nbe, by_nsplit;
    Parts() = default;
    Parts(int E_, int nbe_, int nsplit_) : E(E_), nbe(nbe_), nsplit(nsplit_), by_nbe(nbe_), by_nsplit(nsplit_) {}
    // first block of part z (z = nsplit: the end); E * nbe * nsplit < 2^31
    __device__ __forceinline__ int first(int z) const { return by_nsplit.div(E * nbe * z); }
    // the parts that hold blocks of expert e: part_lo(e) .. part_hi(e) - 1 (every part has a block: nsplit <= E * nbe)
    __host__ __device__ __forceinline__ int part_lo(int e) const
    {
        const unsigned t = (unsigned)E * nbe;
        return (((unsigned)e * nbe + 1u) * nsplit + t - 1) / t - 1;
    }
    __host__ __device__ __forceinline__ int part_hi(int e) const { return ((e + 1u) * nsplit + E - 1) / E; }
};

// acc + load(z0) + load(z0 + 1) + .. + load(z1 - 1), added in this order, with up to sixteen loads in flight: a summing pass
// has few lanes and a load of partial sums takes half a microsecond, so one load per addition made such a pass a chain of
// latencies.  A last batch of more than four is filled up with loads of the last element, which are not added (31 parts: two
// latencies instead of the five of batches of 8, 8, 8, 4, 2).
template <int N, class T, class Load>
__device__ __forceinline__ void add_batch(T& acc, int z, int z1, Load&& load)
{
    T x[N];
#pragma unroll
    for (int k = 0; k < N; ++k) x[k] = load(z + k < z1 ? z + k : z1 - 1);
#pragma unroll
    for (int k = 0; k < N; ++k)
        if (z + k < z1) acc += x[k];
}
template <class T, class Load>
__device__ __forceinline__ T sum_in_order(T acc, int z0, int z1, Load&& load)
{
    int z = z0;
    for (; z + 8 < z1; z += 16) add_batch<16>(acc, z, z1, load);
    switch (z1 - z) {
        case 8: case 7: case 6: case 5: add_batch<8>(acc, z, z1, load); break;
        case 4: add_batch<4>(acc, z, z1, load); break;
        case 3: add_batch<3>(acc, z, z1, load); break;
        case 2: add_batch<2>(acc, z, z1, load); break;
        case 1: add_batch<1>(acc, z, z1, load); break;
    }
    return acc;
}

// Asks for a kernel's arguments (FwdArgs, DqArgs) in front of the return of a workgroup without rows (whole_xcds).  Behind it the compiler loads all but the two that the return
// needs, a second latency in front of a launch's first load.  176 tokens of 8 heads of 128 with 121 blocks, under the profiler, asked for behind / in front: forward 15.1 / 14.3 us,
// dQ/dR 18.0 / 17.7.
template <class Args>
__device__ __forceinline__ void arguments_first(const Args& p)
{
    asm volatile("" ::"s"(p.Q), "s"(p.K), "s"(p.U), "s"(p.V), "s"(p.R), "s"(p.part), "s"(p.rows.tokmaj), "s"(p.rows.H), "s"(p.rows.G), "s"(p.rows.S), "s"(p.rows.n),
                 "s"(p.rows.by_g.m), "s"(p.rows.by_s.m), "s"(p.rows.by_gs.m), "s"(p.rows.by_hkuv.m), "s"(p.parts.E), "s"(p.parts.nbe), "s"(p.parts.nsplit),
                 "s"(p.parts.by_nbe.m), "s"(p.parts.by_nsplit.m), "s"(p.parts.by_nsplit.l));
}

// Into how many parts the forward and the dQ/dR kernel cut the blocks of a head, and which of a kernel's tile heights runs.
// The steps are times of each kernel on half a chip, one of them of an earlier form of it (at each kernel's variants); a step of the
// rows32 forward is a trip of four blocks.
// One part needs no partial sums and is what runs where the row tiles alone fill the chip.  With fewer tiles than compute
// units a part per idle unit shortens the serial walk over the blocks (one token of the 370M layer, 8 tiles of 121 blocks: 46 us
// in one part, 7.8 in 31), and every part costs a set of fp32 sums that is written and read back.  Time of a launch in us:
// rounds of CUS workgroups x (blocks of a part x step + 3 for prologue and epilogue), + 2 for the summing pass (dQ/dR: none where
// the weights' gradients have one, which adds up both) + 0.6 per MB of sums; a step slows by up to `full` as the chip fills
// (power).  The prices are those of d_h = 128 for every d_h: with it the
// variants of a kernel get cheaper nearly together, and that of the 32-row forward is its trips' for its pipeline, too.  Against tile heights and numbers of
// parts around the pick, on 300 bfloat16 calls of the forward drawn from layers of 4 to 16 heads and 1 to 16,384 tokens (profiles/pick_parts_sweep.csv), it is
// 1.8 % slower than the fastest on average and 21 % at worst.  The prices stay above what sums cost since they are added up where they are (whole_xcds):
// 1.5 us and 0.5 per MB, with steps fitted to them on other calls, come to 1.6 % there, but six of the 300 calls take 3 to 17 % longer with them than with these
// (47 tokens of 16 heads of 128 on eight 17.4 / 20.4 us, 8 x 449 of 8 heads of 128 91.9 / 101.2; of 520 rows of 6 heads of 128 with 88 blocks 19.5 / 22.1).
// dQ/dR: at its variants.
// Not cut: more experts than one LDS window of gate values holds (bfloat16); and 16,384 rows per head or more, where a head
// fills a quarter of the chip alone and its results do not depend on how many other heads run beside it.
constexpr int CUS = 256;                     // compute units of an MI355X
constexpr int XCDS = 8;
constexpr long SPLIT_ROWS_BELOW = 16384;
struct Variant {
    int tile_rows;
    double step, full;
    int unit;             // blocks of a step
    int ahead = 0;        // steps that a pipeline takes beyond those of its blocks
    int rows_from = 0;    // rows of a head from which on it is a choice
};
struct Pick {
    int tile_rows, nsplit;
};
// Workgroup i of a launch runs on XCD i % 8, and what it writes stays in that XCD's L2 for the next kernel.  A pass that adds up what several
// workgroups left therefore runs where they did: launches that leave parts are padded (workgroups with nothing to do return
// at once), so that the parts of a tile are written on one XCD, and the pass counts its workgroups the same way.  Only time depends on it.
// 733 tokens of the 128M layer, forward, us: sums by rows on any XCD 19.4, here 16.0; 2,048 33.2, 29.0; 512 of the 370M layer 26.2, 24.1.
// Padding puts more workgroups on some XCDs than an even share, and where those work longer for it than the sums save, the grid stays as it is.  150 forwards and 100 training
// calls drawn from layers of 4 to 16 heads, us, as it is / padded:
// * more workgroups than the launch's rounds hold on an XCD: never padded;
// * tiles of 256 rows of weights above PAD_WEIGHTS (their steps are bound by the tile fills of the XCD's workgroups): 2 x 3,200 rows of 6 heads of 128 with 26 MB 105.8 / 107.7,
//   4 x 346 tokens of 8 heads of 128 on four, backward, 149.3 / 152.7; below it the sums count for more (8 x 459 of 4 heads of 64 on two with 3 MB 36.7 / 33.6,
//   8 x 348 of 4 of 96, backward, 53.8 / 49.5; 5 to 9 MB go either way by 2 %: 8 x 171 tokens of 8 heads of 128 on two 193 / 198 forward and backward);
// * smaller tiles, which are few where it matters and read all weights once: an XCD reads more of them, a microsecond for every MB.  One to eight tokens of 8 heads of 128 on
//   two, whose 31 parts would all run on two XCDs, 8.3 / 8.9 to 9.5 / 10.4, 39 of 6 heads of 128 with 26 MB 14.6 / 15.6; with less than PAD_MORE
//   more (270 of 8 of 96 on two 14.8 / 12.9, one of 6 of 64 on three 7.2 / 6.6) the sums save half a microsecond and more.
// Padded by this rule, 2 of the 150 forwards and 2 of the 100 training calls are slower than as they are by 1.5 to 3 %; always padded 17 and 7, by up to 10 %.
constexpr double PAD_WEIGHTS = 5e6, PAD_MORE = 0.6e6;      // bytes
inline unsigned tiles_of(const Dims& d, const Pick& pick)
{
    return (unsigned)(((long)(d.H / d.Hkuv) * d.B * d.S + pick.tile_rows - 1) / pick.tile_rows * d.Hkuv);
}
// the workgroups of a part
inline unsigned whole_xcds(const Dims& d, const Pick& pick, size_t element)
{
    const unsigned tiles = tiles_of(d, pick), parts = pick.nsplit, padded = (tiles + XCDS - 1) / XCDS * XCDS;
    const unsigned most = padded / XCDS * parts, share = (unsigned)(((long)tiles * parts + XCDS - 1) / XCDS);
    const unsigned rounds = (unsigned)(((long)tiles * parts + CUS - 1) / CUS);
    const double weights = 3.0 * d.Hkuv * d.E * d.d_e * d.d_h * element;
    if (parts < 2 || most > rounds * (CUS / XCDS)) return tiles;
    return (pick.tile_rows == 256 ? weights <= PAD_WEIGHTS : weights / XCDS * (most - share) <= PAD_MORE * share) ? padded : tiles;
}
template <int N>
inline Pick pick_parts(const Variant (&variants)[N], const Dims& d, int blocks, bool may_cut, size_t part_bytes, size_t ws_bytes, double sum_us = 2)
{
    const long rows = (long)(d.H / d.Hkuv) * d.B * d.S;
    const int most = may_cut && rows < SPLIT_ROWS_BELOW && blocks < (1 << 24) ? (blocks < 64 ? blocks : 64) : 1;
    const double part_us = part_bytes * 0.6e-6;
    Pick best{variants[0].tile_rows, 1};
    double best_us = 0;
    for (const Variant& v : variants) {
        if (v.tile_rows == 32 ? !may_cut : may_cut && rows < v.rows_from) continue;      // (32-row tiles hold all gate values of a tile in LDS)
        const long tiles = (rows + v.tile_rows - 1) / v.tile_rows * d.Hkuv;
        for (int ns = 1; ns <= most; ++ns) {
            if (ns > 1 && (ns * part_bytes > ws_bytes || tiles * (ns - 1) >= 2 * CUS)) break;
            const long wgs = tiles * ns;
            const double load = wgs <= CUS / 2 ? 0 : wgs >= CUS ? 1 : (wgs - CUS / 2) / (double)(CUS / 2);
            const double us = (double)((wgs + CUS - 1) / CUS) * ((((blocks + ns - 1) / ns + v.unit - 1) / v.unit + v.ahead) * v.step * (1 + v.full * load) + 3) +
                              (ns > 1 ? sum_us + ns * part_us : 0);
            if (best_us == 0 || us < best_us) { best_us = us; best = Pick{v.tile_rows, ns}; }
        }
    }
    return best;
}

// What a launch with this workspace (0: none) and these phases runs.
Pick fwd_pick_bf16(const Dims& d, size_t ws_bytes, int phases);
Pick dq_pick_bf16(const Dims& d, size_t ws_bytes, int phases);
int dw_slices_bf16(const Dims& d, size_t ws_bytes);
bool dw_token_halves(const Dims& d, size_t ws_bytes);      // two waves for a block of rows
bool fwd_reads_past(const Dims& d, const Pick& pick);      // the weights, past the caches
unsigned grid_of_part_f32(const Dims& d, const Pick& pick);      // workgroups (whole_xcds)
Pick fwd_pick_f32(const Dims& d, size_t ws_bytes, int phases);
Pick dq_pick_f32(const Dims& d, size_t ws_bytes, int phases);
int dw_slices_f32(const Dims& d);

size_t fwd_workspace_bytes_bf16(const Dims& d);       // what the launch uses when it may choose freely (0: one part);
                                                      // with less it runs fewer parts
size_t bwd_workspace_bytes_bf16(const Dims& d);       // what the launch uses when it may choose freely: the token slices of
                                                      // dK, dU, dV and the parts of dQ, dR (0: one of each); with less it
                                                      // runs fewer
size_t bwd_min_workspace_bytes_bf16(const Dims& d);   // those of the token slices alone
hipError_t launch_fwd_bf16(const void* Q, const void* K, const void* U, const void* V, const float* R, void* O,
                           void* ws, size_t ws_bytes, const Dims& d, hipStream_t st, int phases);
hipError_t launch_bwd_bf16(const void* Q, const void* K, const void* U, const void* V, const float* R, const void* dO,
                           void* dQ, void* dK, void* dU, void* dV, float* dR, int grad_w_f32,
                           void* ws, size_t ws_bytes, const Dims& d, hipStream_t st, int phases);

// fp32 instantiation (mhffn_f32.hip): d_h a multiple of 8 up to 128, any d_e, any E.
size_t fwd_workspace_bytes_f32(const Dims& d);        // as fwd_workspace_bytes_bf16
size_t bwd_workspace_bytes_f32(const Dims& d);        // as bwd_workspace_bytes_bf16, but the token slices are fixed:
size_t bwd_min_workspace_bytes_f32(const Dims& d);    // the launch needs these
hipError_t launch_fwd_f32(const void* Q, const void* K, const void* U, const void* V, const float* R, void* O,
                          void* ws, size_t ws_bytes, const Dims& d, hipStream_t st, int phases);
hipError_t launch_bwd_f32(const void* Q, const void* K, const void* U, const void* V, const float* R, const void* dO,
                          void* dQ, void* dK, void* dU, void* dV, float* dR, int grad_w_f32, void* ws, size_t ws_bytes,
                          const Dims& d, hipStream_t st, int phases);

// Head prologue (mhffn_gate.hip): per-head RMSNorm + expert gate over [B, S, H, d_h] bf16 rows; d_h 64/96/128, E <= 64.
// Wn, Wr (and dWn, dWr where there is a workspace) are float or, with wn_bf16, wr_bf16, bfloat16.  Without a workspace the backward adds
// to float dWn, dWr; with one (gate_bwd_workspace_bytes) it overwrites them.
hipError_t launch_gate_fwd(const void* X, const void* Wn, int wn_bf16, float eps, const void* Wr, int wr_bf16, void* Qn, float* R,
                           const Dims& d, hipStream_t st);
size_t gate_bwd_workspace_bytes(const Dims& d);
bool gate_fwd_whole_rows(const Dims& d), gate_bwd_whole_rows(const Dims& d);      // whether whole rows move (WholeRows)
hipError_t launch_gate_bwd(const void* X, const void* Wn, int wn_bf16, float eps, const void* Wr, int wr_bf16, const void* dQ,
                           int dq_tokmaj, const float* dR, void* dX, void* dWn, void* dWr, void* ws, const Dims& d, hipStream_t st);

// Rotary positions of the decoder's attention (mhffn_rope.hip); d a multiple of 16, B * S * H * d / 16 below 2^31.
hipError_t launch_rope_fwd(const void* qkv, const void* cos, const void* sin, void* q, void* k, int B, int S, int H, int dh,
                           hipStream_t st);
hipError_t launch_rope_bwd(const void* const d[3], const long (*stride)[3], const void* cos, const void* sin, void* dqkv, int B, int S,
                           int H, int dh, hipStream_t st);

// Bits of the `phases` argument of the launch functions (the values of MHFFN_FWD_*, MHFFN_BWD_*, MHFFN_ONE_PART in
// include/mhffn.h).
constexpr int PH_FWD_MAIN = 1, PH_BWD_DQDR = 1, PH_BWD_DKDUDV = 2, PH_BWD_REDUCE = 4, PH_ONE_PART = 256;

}  // namespace mhffn
