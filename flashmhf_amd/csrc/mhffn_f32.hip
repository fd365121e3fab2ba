// fp32 instantiation of the fused multi-head FFN (forward, dQ/dR, dK/dU/dV): operands, sums and everything between the products are
// float32, products are off by 2^-24 at most and the sigmoid by a rounding or two, so results track an fp32 eager evaluation to
// ~1e-6.  Same fusion as the bf16 kernels -- the
// [tokens, E*d_e] intermediate exists only in registers.  Generic in d_h (multiple of 8, at most 128; CT = 32-column tiles of
// it), d_e and E.
// Formulas: models/flashmhf/modeling_mhffnmoe.py:418-427 (forward), kernels/triton/flash_mlp_moe.py:401-414, 527-542,
// 720-729 (backward).
//
// The products run on v_mfma_f32_32x32x16_bf16 with every operand taken apart into three bfloat16 values ("planes", below);
// operand layouts are those of mhffn_common.hpp.  dK/dU/dV for d_h > 96, whose planes do not fit a wave's registers, parts of one
// block and rows whose results are not finite run on v_mfma_f32_32x32x2_f32, D = A(32x2) * B(2x32) + C, 64 cycles each:
//       A: lane l holds row (l % 32), k = l / 32         B: lane l holds col (l % 32), k = l / 32
//       C/D: lane l holds col (l % 32), register i holds row 8*(i/4) + 4*(l/32) + (i%4)
// * First products contract over the head dim.  The order of the k index is free as long as A and B agree: with lane group
//   g = l / 32 holding columns 8m + 4g .. +3, one 16-byte read of each operand row feeds four instructions.
// * They are written with rows = tokens, columns = j, so that register i of the result is, as it stands, the B operand of the
//   second products' step i: k slot g is row 8*(i/4) + 4g + i%4.  The A operand of that step is one row of Q (dO) per lane
//   group, read along its columns.
//
// What bounds them.  256 tokens of the 128M layer took 30 (forward), 45 (dQ/dR) and 61 us (dK/dU/dV) on the fp32 matrix
// instructions, whose time a kernel's four waves could not go below (15, 26 and 31 us, 153 TFLOP/s over the chip) and under which
// they issue next to nothing else.  The planes take 2.7 times less matrix time and some VALU instructions per operand and
// element, put between the matrix instructions where registers allow: 25, 34 and 46 us; per 32 rows of weights (forward, dQ/dR;
// 128 rows, a part of 64 in one) 5.2 -> 2.3 and 8.2 -> 4.0 us, per 32 tokens (dK/dU/dV, two tiles) 11.2 -> 6.6, the rest is prologue
// and epilogue.
#include "mhffn_common.hpp"

#include <utility>

namespace mhffn {

namespace {

struct F32Args {
    const float *Q, *K, *U, *V, *R, *dO;
    float *O, *dQ, *dR;
    float* part;        // fp32 partial sums: parts of O, or of dQ and dR, or token slices of dK, dU, dV
    void* out[3];       // dK, dU, dV
    int out_f32;        // their element type: 1 = float32, 0 = bfloat16
    RowMap rows;        // rows of Q, O, dO, dQ, R, dR that meet one K/U/V head
    Parts parts;        // blocks of 32 weight rows of that head, the last of an expert with de % 32 rows if that is not 0
    int DH, de, nslice;
    int heads_first;    // dK/dU/dV: the head runs fastest over the workgroups
};

__device__ __forceinline__ f32x16 mfma2(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float sigmoid_exact(float x) { return 1.0f / (1.0f + __expf(-x)); }
// Sixteen times that of x = 2^-48 xs, in the kernels that have VALU time to lose: the reciprocal with one Newton step (an IEEE division
// takes three times the instructions), a normal number up to the largest finite e^-x; 0 beyond that, where the step would make
// NaN of an infinite one.
__device__ __forceinline__ float sigmoid16(float xs)
{
    const float t = -LOG2E * 0x1p-48f * xs, d = fmaf(__builtin_amdgcn_exp2f(t), 0.0625f, 0.0625f), y = __builtin_amdgcn_rcpf(d);
    const float s = fmaf(fmaf(-d, y, 1.0f), y, y);
    return t >= 128.0f ? 0.0f : s;
}
__device__ __forceinline__ f32x16 zero16()
{
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.0f;
    return z;
}
// row of register i of a result tile
__device__ __forceinline__ int reg_row(int i, int g) { return 8 * (i >> 2) + 4 * g + (i & 3); }

// LDS tile: 32 rows of CH 16-byte chunks (a power of two, d_h / 4 of them used), chunk c of row r at c ^ (r % 16): 16-byte reads
// of 16 different rows, and 4-byte reads along a row, spread over the banks; filled by LDS-direct loads of 1 KB.
template <int CT>
struct Tile {
    static constexpr int CH = CT == 1 ? 8 : CT == 2 ? 16 : 32, ROW_B = 16 * CH, BYTES = 32 * ROW_B, INS = BYTES / 1024;
    static constexpr int SWZ = (CH < 16 ? CH : 16) - 1;
    // Wave-instruction `ins` of the fill: row(r) gives the source row; chunk positions beyond d_h receive chunk 0.
    template <class Row>
    __device__ static void fill(unsigned char* tile, int ins, int lane, int DH, Row&& row)
    {
        const int pos = ins * 64 + lane, r = pos / CH;
        int c = (pos % CH) ^ (r & SWZ);
        c = 4 * c < DH ? c : 0;
        __builtin_amdgcn_global_load_lds((gptr_t)(row(r) + 4 * c), (lptr_t)(tile + ins * 1024), 16, 0, 0);
    }
    // Per-lane parts of the two kinds of reads; everything else of an address is a compile-time constant (the exclusive-or of
    // the swizzle acts on chunk bits that the constants do not carry into).
    struct Lane {
        int k0, e0;
        __device__ Lane(int l32, int g)
            : k0(l32 * ROW_B + ((g ^ (l32 & SWZ)) << 4)), e0(4 * g * ROW_B + (((l32 >> 2) ^ (4 * g)) << 4) + 4 * (l32 & 3))
        {
            asm volatile("" : "+v"(k0), "+v"(e0));      // (kept out of the compiler's sight, or it hoists every sum with
        }                                               // a constant out of the loop into a register of its own)
    };
    // columns 8m + 4g .. +3 of row l32
    template <int M>
    __device__ static f32x4 along_k(const unsigned char* tile, const Lane& l)
    {
        return *reinterpret_cast<const f32x4*>(tile + (l.k0 ^ ((2 * M & SWZ) << 4)) + (((2 * M) & ~SWZ) << 4));
    }
    // column 32 ct + l32 of the row that is register I of a result, 8a + 4g + b
    template <int I>
    __device__ static float element(const unsigned char* tile, const Lane& l, int ct)
    {
        constexpr int a = I >> 2, b = I & 3;
        return *reinterpret_cast<const float*>(tile + (l.e0 ^ (b << 4)) + (8 * a + b) * ROW_B + (((8 * ct) ^ (8 * a & SWZ)) << 4));
    }
};

// This lane's half of a row as first-product operand: columns 8m + 4g .. +3 for every m, zero beyond d_h.
template <int CT>
__device__ __forceinline__ void load_row(f32x4 (&v)[4 * CT], const float* row, int g, int DH)
{
#pragma unroll
    for (int m = 0; m < 4 * CT; ++m) {
        v[m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (8 * m < DH) v[m] = *reinterpret_cast<const f32x4*>(row + 8 * m + 4 * g);
    }
}

// acc[ct] += (rows of `tile` as columns 32 ct + l32) * b: one second product, b a result of the first products.  Here and in
// first_products the operands are read one step ahead, and a fence per step keeps the compiler from gathering reads at
// the front, which costs more registers than a wave has.
template <int CT>
__device__ __forceinline__ void second_product(f32x16 (&acc)[CT], const unsigned char* tile, const f32x16& b,
                                               const typename Tile<CT>::Lane& l)
{
    float a[2][CT];
    auto read = [&](auto ic) {
        constexpr int i = decltype(ic)::value;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) a[i & 1][ct] = Tile<CT>::template element<i>(tile, l, ct);
    };
    read(std::integral_constant<int, 0>{});
    static_for<16>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (i < 15) read(std::integral_constant<int, i + 1>{});
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[ct] = mfma2(a[i & 1][ct], b[i], acc[ct]);
        __builtin_amdgcn_sched_barrier(0);
    });
}

// d[k] = product of the rows of tile t[k] (A operand) with this lane's row v[k] (B operand) over the head dim
template <int CT, int N>
__device__ __forceinline__ void first_products(f32x16 (&d)[N], const unsigned char* const (&tile)[N], const f32x4* const (&v)[N],
                                               const typename Tile<CT>::Lane& l)
{
    f32x4 a[2][N];
    auto read = [&](auto cc) {
        constexpr int c = decltype(cc)::value;
#pragma unroll
        for (int k = 0; k < N; ++k)
            a[c & 1][k] = k > 0 && tile[k] == tile[k - 1] ? a[c & 1][k - 1] : Tile<CT>::template along_k<c>(tile[k], l);
    };
    read(std::integral_constant<int, 0>{});
#pragma unroll
    for (int k = 0; k < N; ++k) d[k] = zero16();
    static_for<4 * CT>([&](auto cc) {
        constexpr int c = decltype(cc)::value;
        if constexpr (c + 1 < 4 * CT) read(std::integral_constant<int, c + 1>{});
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int k = 0; k < N; ++k) d[k] = mfma2(a[c & 1][k][x], v[k][c][x], d[k]);
        __builtin_amdgcn_sched_barrier(0);
    });
}

// Transposed accumulators (register 4a + x of tile ct: column 32 ct + 8a + 4g + x of this lane's row) to dst, this lane's row.
template <int CT>
__device__ __forceinline__ void store_row(const f32x16 (&acc)[CT], float* dst, int g, int DH)
{
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int a = 0; a < 4; ++a)
            if (32 * ct + 8 * a < DH) {
                f32x4 v;
#pragma unroll
                for (int x = 0; x < 4; ++x) v[x] = acc[ct][4 * a + x];
                *reinterpret_cast<f32x4*>(dst + 32 * ct + 8 * a + 4 * g) = v;
            }
}

// ---- float32 operands on the bf16 matrix instructions -----------------------------------------------------------------
// A float32 value is the exact sum of three bfloat16 values: it rounded to one, the rest rounded, and what is left.  With units of the
// value's binade these are at most 2, 2^-8 and 2^-17.  Of the nine products of two such sums the six of the largest terms run on
// v_mfma_f32_32x32x16_bf16, which has sixteen times the rate of v_mfma_f32_32x32x2_f32; the three left out are at most 2^-24
// of the product (2^-24.06 found by trying), no more than one float32 addition rounds away, and of either sign over mantissas.  (With
// the largest plane cut off instead of rounded they reach 2^-22.)  A sum over k then rounds once
// per sixteen terms and plane instead of once per two: against 64 bits the results are 10 to 30 % closer than those of the fp32
// instructions (32 to 1,024 tokens, d_h 24 to 128; O 3.5e-7 -> 2.7e-7, dQ 4.0 -> 3.4, dK, dU, dV 3.4 -> 2.8, dR 3.6 -> 3.0
// for 256 tokens of the 128M layer).
// The matrix instructions take a plane below 2^-126 for zero, and the last plane is 2^-23 of a value: operands are taken apart 2^24
// times as large, which holds every float32 to its last bit.  First products are 2^48 times as large, and so are dM, dN and P (without a
// multiplication more); the sums of the second products are 2^72 times as large.
// What is too large for that (products beyond 2^79, P, dM and dN beyond 2^79, results beyond 2^55) overflows.  An infinity or NaN in an operand, or a value that rounds to an infinite
// bfloat16, makes every sum that it enters NaN: such rows are taken again (below, "the same on the fp32 matrix instructions").
constexpr float UP = 0x1p24f;                   // of an operand of the first products and of weights
constexpr float DOWN1 = 0x1p-48f, DOWN2 = 0x1p-72f;      // results of the first and of the second products
constexpr int PLANE_B = TILE_B;                 // one plane of a 32-row tile, in the layout of the bf16 kernels' tiles
constexpr int PLANES_B = 3 * PLANE_B;

// the pair (x0, x1) as three packed pairs of bfloat16, largest first
__device__ __forceinline__ void split2(float x0, float x1, unsigned& h, unsigned& m, unsigned& l)
{
    typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
    auto round = [](float a, float b) {
        unsigned v = __builtin_bit_cast(unsigned, bf16x2{(bf16_t)a, (bf16_t)b});
        asm("" : "+v"(v));      // (or the compiler rounds a second time instead of shifting the pair)
        return v;
    };
    h = round(x0, x1);
    const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
    m = round(r0, r1);
    l = __builtin_bit_cast(unsigned, bf16x2{(bf16_t)(r0 - __uint_as_float(m << 16)), (bf16_t)(r1 - __uint_as_float(m & 0xffff0000u))});
}
struct Split8 {
    bf16x8 p[3];
};
// 16 bytes per lane from src to dst + 16 lane, asynchronously and without the compiler's knowledge, which would put a wait for it in
// front of every LDS read behind it.
template <int IMM>
__device__ __forceinline__ void lds_direct16(const float* src, unsigned char* dst)
{
    // (the instruction's offset counts at both ends; m0, where the compiler keeps the base of its own such loads and which a clobber
    // list cannot name, is left as it was)
    unsigned m0;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:%3\n\ts_mov_b32 m0, %0"
                 : "=&s"(m0) : "v"(src), "s"(lds_addr(dst) - IMM), "n"(IMM) : "memory");
}
// pair I of eight values: the planes' registers I
template <int I, class V>
__device__ __forceinline__ void split8_pair(u32x4 (&v)[3], V&& x)
{
    unsigned h, m, l;
    split2(x(2 * I), x(2 * I + 1), h, m, l);
    v[0][I] = h; v[1][I] = m; v[2][I] = l;
}
__device__ __forceinline__ Split8 split8_of(const u32x4 (&v)[3])
{
    return Split8{{__builtin_bit_cast(bf16x8, v[0]), __builtin_bit_cast(bf16x8, v[1]), __builtin_bit_cast(bf16x8, v[2])}};
}
template <class V>
__device__ __forceinline__ Split8 split8(V&& x)      // x(0) .. x(7)
{
    u32x4 v[3];
    static_for<4>([&](auto ic) { split8_pair<decltype(ic)::value>(v, x); });
    return split8_of(v);
}
// the planes of the six products, smallest terms first
constexpr int SPLIT_A[6] = {2, 0, 1, 1, 0, 0}, SPLIT_B[6] = {0, 2, 1, 0, 1, 0};

// four weights taken apart, two at a time
struct CutPiece {
    u32x2 h, m, l;
    template <int I>
    __device__ __forceinline__ void half(const f32x4& x)
    {
        unsigned a, b, c;
        split2(UP * x[2 * I], UP * x[2 * I + 1], a, b, c);
        h[I] = a; m[I] = b; l[I] = c;
    }
};
// A thread of a team of 256 that takes 32 rows x 32 CT columns of weights apart: row t / 8, columns 32 k + 4 (t % 8) .. + 3.
template <int CT>
struct Cut {
    int row, col, at;                      // at: byte in a plane, column group 0 (column group k: at ^ (k << 6))
    __device__ explicit Cut(int t) : row(t >> 3), col(4 * (t & 7)), at((t >> 3) * TILE_ROW_B + ((((t & 7) >> 1) ^ swz16(t >> 3)) << 4) + 8 * (t & 1)) {}
    // W: first row of the tile, of which `rows` exist; the columns beyond d_h are zero
    __device__ void load(f32x4 (&x)[CT], const float* W, int rows, int DH) const
    {
        const float* src = W + (row < rows ? row : rows - 1) * DH + col;
#pragma unroll
        for (int k = 0; k < CT; ++k) {
            x[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (32 * k + col < DH) x[k] = *reinterpret_cast<const f32x4*>(src + 32 * k);
        }
    }
    __device__ void store(unsigned char* planes, int k, const f32x4& x) const
    {
        CutPiece c;
        c.half<0>(x);
        c.half<1>(x);
        store(planes, k, c);
    }
    __device__ void store(unsigned char* planes, int k, const CutPiece& c) const
    {
        unsigned char* d = planes + (at ^ (k << 6));
        *reinterpret_cast<u32x2*>(d) = c.h;
        *reinterpret_cast<u32x2*>(d + PLANE_B) = c.m;
        *reinterpret_cast<u32x2*>(d + 2 * PLANE_B) = c.l;
    }
};
// Per-lane byte offsets of the reads of a plane: by rows (k-step ks: row ^ (ks << 5)) and by columns (column tile ct, 16 rows s:
// (col ^ (ct << 6)) + 4096 s).
struct PlaneLane {
    int row, col[2];
    __device__ explicit PlaneLane(int lane)
    {
        const int r = row_perm32(lane & 31);
        const TrLane<1> t = make_tr_lane<1, 8, 4>(lane);
        row = r * TILE_ROW_B + (((lane >> 5) ^ swz16(r)) << 4);
        col[0] = t.off[0][0]; col[1] = t.off[0][1];
    }
};
// row of the weight tile that register i of a first product holds
__device__ __forceinline__ int split_row(int i, int g) { return 16 * (i >> 3) + 8 * g + (i & 7); }

struct Operand {
    bf16x8 p[3];
};
__device__ __forceinline__ Operand read_rows(const unsigned char* planes, const PlaneLane& l, int ks)
{
    Operand a;
#pragma unroll
    for (int x = 0; x < 3; ++x) a.p[x] = *reinterpret_cast<const bf16x8*>(planes + (l.row ^ (ks << 5)) + x * PLANE_B);
    return a;
}
__device__ __forceinline__ Operand read_cols(const unsigned char* planes, const PlaneLane& l, int ct, int s)
{
    typedef __attribute__((address_space(3))) v4bf16_t* lds_v4;
    Operand a;
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const v4bf16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4)(planes + (l.col[0] ^ (ct << 6)) + 4096 * s + x * PLANE_B));
        const v4bf16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_v4)(planes + (l.col[1] ^ (ct << 6)) + 4096 * s + x * PLANE_B));
        a.p[x] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    return a;
}
// d[k] = rows of the planes of a tile times this lane's row v[k].  The first SHARED products take the first tile (planes), every
// further one the next.  ACC(k, plane): that plane of v[k] is kept in accumulation registers.  slot(i) runs behind the i-th of the
// 12 CT N matrix instructions.  The results are architectural registers and need mfma_result_fence before the VALU reads them.
template <int CT, int N, int SHARED, class Acc, class Slot>
__device__ __forceinline__ void first_split(f32x16 (&d)[N], const unsigned char* planes, const Split8* const (&v)[N], const PlaneLane& l,
                                            Acc, Slot&& slot)
{
    constexpr int T = N - SHARED + 1;
    Operand a[2];
    a[0] = read_rows(planes, l, 0);
    static_for<2 * CT * T>([&](auto uc) {
        constexpr int u = decltype(uc)::value, n = u + 1, ks = u / T, k0 = u % T ? u % T + SHARED - 1 : 0, kn = u % T ? 1 : SHARED;
        if constexpr (n < 2 * CT * T) a[n & 1] = read_rows(planes + (n % T) * PLANES_B, l, n / T);
        static_for<6 * kn>([&](auto xc) {
            constexpr int x = decltype(xc)::value / kn, k = k0 + decltype(xc)::value % kn;
            const bf16x8 w = a[u & 1].p[SPLIT_A[x]], q = v[k][ks].p[SPLIT_B[x]];
            if constexpr (Acc{}(k, SPLIT_B[x])) {
                if constexpr (ks == 0 && x == 0) mfma32_vgpr_first_bacc(d[k], w, q);
                else mfma32_vgpr_acc_bacc(d[k], w, q);
            } else {
                if constexpr (ks == 0 && x == 0) mfma32_vgpr_first(d[k], w, q);
                else mfma32_vgpr_acc(d[k], w, q);
            }
            slot(std::integral_constant<int, 6 * (N * ks + k0) + decltype(xc)::value>{});
        });
        __builtin_amdgcn_sched_barrier(0);
    });
}
struct NoAcc {
    constexpr bool operator()(int, int) const { return false; }
};
struct AllAcc {
    constexpr bool operator()(int, int) const { return true; }
};
// dK/dU/dV: K and the last plane of U beside the accumulators of the gradients
struct WeightAcc {
    constexpr bool operator()(int k, int plane) const { return k == 0 || (k == 1 && plane == 2); }
};
// acc[ct] += columns 32 ct + l32 of the planes' rows 16 s .. + 15 times b.  slot(i) runs behind the i-th of the 6 CT matrix
// instructions.
template <int CT, class Slot>
__device__ __forceinline__ void second_split(f32x16 (&acc)[CT], const unsigned char* planes, int s, const Split8& b, const PlaneLane& l,
                                             Slot&& slot)
{
    Operand a[2];
    a[0] = read_cols(planes, l, 0, s);
    static_for<CT>([&](auto cc) {
        constexpr int ct = decltype(cc)::value;
        if constexpr (ct + 1 < CT) a[(ct + 1) & 1] = read_cols(planes, l, ct + 1, s);
        static_for<6>([&](auto xc) {
            constexpr int x = decltype(xc)::value;
            acc[ct] = mfma32(a[ct & 1].p[SPLIT_A[x]], b.p[SPLIT_B[x]], acc[ct]);
            slot(std::integral_constant<int, 6 * ct + x>{});
        });
        __builtin_amdgcn_sched_barrier(0);
    });
}
// This lane's row as B operands of the first products, zero beyond d_h: its values, then their planes.
template <int CT>
__device__ __forceinline__ void load_row_operand(f32x4 (&x)[4 * CT], const float* row, int g, int DH)
{
#pragma unroll
    for (int i = 0; i < 4 * CT; ++i) {
        const int c = 16 * (i >> 1) + 8 * g;
        x[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (c < DH) x[i] = *reinterpret_cast<const f32x4*>(row + c + 4 * (i & 1));
    }
}
template <int CT>
__device__ __forceinline__ void split_row_operand(Split8 (&v)[2 * CT], const f32x4 (&x)[4 * CT])
{
#pragma unroll
    for (int ks = 0; ks < 2 * CT; ++ks) v[ks] = split8([&](int i) { return UP * x[2 * ks + (i >> 2)][i & 3]; });
}

// Workgroup of the forward and of dQ/dR: 4 waves of 32 rows of one K/U/V head, one part of the head's blocks.
constexpr int F32_ROWS = 128;
struct Place {
    int hk, z, row0, row, blk0, nblk;      // row0: this wave's first row of the list, row: this lane's (clamped into the list)
    bool valid;                            // this lane's row exists
    bool none;                             // no row of the workgroup does (whole_xcds)
    __device__ explicit Place(const F32Args& p, int wave, int l32)
    {
        const int tile = p.rows.by_hkuv.div(blockIdx.x);
        hk = blockIdx.x - tile * p.rows.Hkuv;
        z = blockIdx.y;
        none = tile * F32_ROWS >= p.rows.n;
        row0 = tile * F32_ROWS + wave * 32;
        valid = row0 + l32 < p.rows.n;
        row = valid ? row0 + l32 : p.rows.n - 1;
        blk0 = p.parts.first(z);
        nblk = p.parts.first(z + 1) - blk0;
    }
};
// First weight row of block blk of kv-head hk, the block's expert and its rows.
struct Block {
    long wrow;
    int e, rows;
    __device__ Block(const F32Args& p, int hk, int blk)
    {
        e = p.parts.by_nbe.div(blk);
        const int j0 = (blk - e * p.parts.nbe) * JB;
        wrow = ((long)hk * p.parts.E + e) * p.de + j0;
        rows = p.de - j0 < JB ? p.de - j0 : JB;
    }
};

// ---- the same on the fp32 matrix instructions -------------------------------------------------------------------------------
// What the planes cannot carry comes out as NaN: an infinity in an operand, or a value beyond the largest float32 between the products
// (infinity minus infinity, in split2).  A row of results that is not finite is therefore taken again on
// v_mfma_f32_32x32x2_f32, which knows infinities, by the waves of its workgroup together; the workgroup's other rows keep theirs.
// 256 tokens of the 128M layer: looking for such rows takes 0.1 (forward), 0.4 (dQ/dR) and 0.9 us (dK/dU/dV) of 24.5, 34.3 and 45.1;
// with one in every workgroup the kernels take 47, 67 and 95 us, alone on these instructions 30, 46 and 61.
__device__ __forceinline__ bool finite(float x) { return (__float_as_uint(x) & 0x7f800000u) != 0x7f800000u; }
template <int CT>
__device__ __forceinline__ bool finite(const f32x16 (&acc)[CT])
{
    unsigned most = 0;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 16; ++i) most = max(most, __float_as_uint(acc[ct][i]) & 0x7fffffffu);
    return most < 0x7f800000u;
}
template <int CT>
__device__ __forceinline__ void scale(f32x16 (&acc)[CT], float by)
{
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[ct][i] *= by;
}
// Whether it holds in this lane or in the one with the other half of its row.
__device__ __forceinline__ bool in_row(bool here)
{
    const int other = __shfl_xor((int)here, 32);      // (read by every lane)
    return here || other != 0;
}
// Whether `here` holds in a lane of the workgroup, which is done with its LDS; word: four bytes of it per wave (of four).
__device__ __forceinline__ bool anywhere(bool here, unsigned char* words, int wave)
{
    volatile unsigned* word = reinterpret_cast<volatile unsigned*>(words);
    const bool own = __ballot(here) != 0;
    quad_barrier();      // (__syncthreads would wait for the results' stores)
    if ((threadIdx.x & 63) == 0) word[wave] = own;
    quad_barrier();
    return __builtin_amdgcn_readfirstlane(word[0] | word[1] | word[2] | word[3]) != 0;
}
// K, U and V tiles of block b by four waves, waited for.
template <int CT>
__device__ __forceinline__ void fill_block(const F32Args& p, const Block& b, unsigned char* lds, int wave)
{
    using T = Tile<CT>;
    constexpr int FI = T::INS / 4 > 0 ? T::INS / 4 : 1;      // fill instructions per wave and tile
    __syncthreads();      // every wave is done with the block before
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));      // (the fills' addresses are not worth a register each)
    auto row = [&](const float* W) {
        return [&, W](int r) { return W + (b.wrow + (r < b.rows ? r : b.rows - 1)) * p.DH; };
    };
#pragma unroll
    for (int k = 0; k < FI; ++k) {
        T::fill(lds, wave * FI + k, lane, p.DH, row(p.K));
        T::fill(lds + T::BYTES, wave * FI + k, lane, p.DH, row(p.U));
        T::fill(lds + 2 * T::BYTES, wave * FI + k, lane, p.DH, row(p.V));
    }
    wait_vmcnt<0>();
    __syncthreads();
}
// O of this wave's rows over the part's blocks.
template <int CT>
__device__ __forceinline__ void fwd_fp32(const F32Args& p, const Place& w, unsigned char* lds, int wave, f32x16 (&o)[CT])
{
    using T = Tile<CT>;
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    f32x4 q[4 * CT];
    load_row<CT>(q, p.Q + p.rows.tok(w.hk, w.row) * p.DH, g, p.DH);
    const float* rrow = p.R + p.rows.gate(w.hk, w.row) * p.parts.E;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) o[ct] = zero16();
    for (int blk = 0; blk < w.nblk; ++blk) {
        const Block b(p, w.hk, w.blk0 + blk);
        const float r = rrow[b.e];
        fill_block<CT>(p, b, lds, wave);
        f32x16 mn[2];
        const typename T::Lane l(l32, g);
        first_products<CT, 2>(mn, {lds, lds + T::BYTES}, {q, q}, l);
        f32x16 &m = mn[0], &n = mn[1];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float v = m[i] * sigmoid_exact(m[i]) * n[i] * r;
            asm volatile("" : "+v"(v));      // (or the compiler makes a branch of each element)
            m[i] = reg_row(i, g) < b.rows ? v : 0.0f;
        }
        second_product<CT>(o, lds + 2 * T::BYTES, m, l);
    }
}
// dQ of this wave's rows over the part's blocks, and their dR to drow where `store` holds.
template <int CT>
__device__ __forceinline__ void dqdr_fp32(const F32Args& p, const Place& w, unsigned char* lds, int wave, float* drow, bool store, f32x16 (&dq)[CT])
{
    using T = Tile<CT>;
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const long tok = p.rows.tok(w.hk, w.row) * p.DH;
    f32x4 q[4 * CT], go[4 * CT];
    load_row<CT>(q, p.Q + tok, g, p.DH);
    load_row<CT>(go, p.dO + tok, g, p.DH);
    const float* rrow = p.R + p.rows.gate(w.hk, w.row) * p.parts.E;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) dq[ct] = zero16();
    float dr = 0.0f;
    for (int blk = 0; blk < w.nblk; ++blk) {
        const Block b(p, w.hk, w.blk0 + blk);
        const float r = rrow[b.e];
        fill_block<CT>(p, b, lds, wave);
        f32x16 mna[3];
        const typename T::Lane l(l32, g);
        first_products<CT, 3>(mna, {lds, lds + T::BYTES, lds + 2 * T::BYTES}, {q, q, go}, l);
        f32x16 &m = mna[0], &n = mna[1], &da = mna[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float sg = sigmoid_exact(m[i]), sl = m[i] * sg;
            const float a = reg_row(i, g) < b.rows ? da[i] : 0.0f;
            dr = fmaf(a * sl, n[i], dr);
            m[i] = r * a * n[i] * (sg + sl * (1.0f - sg));      // dM
            n[i] = r * a * sl;                                  // dN
        }
        second_product<CT>(dq, lds, m, l);
        second_product<CT>(dq, lds + T::BYTES, n, l);
        if (blk + 1 == w.nblk || Block(p, w.hk, w.blk0 + blk + 1).e != b.e) {
            const float tot = dr + __shfl_xor(dr, 32);
            if (g == 0 && store) drow[b.e] = tot;
            dr = 0.0f;
        }
    }
}

// Parts of one block: taking operands apart, a second team and the longer way to the results do not pay there.  Forward of 64 rows of 4
// heads of 96 in 64 parts 22.5 us, 27.6 with the kernels below; of 32 rows of 4 heads of 64 in 16 parts 10.2, 13.2; of one block of 8 x 8 4.8,
// 6.9.  dQ/dR: level for d_h > 64, 4 % less time for 64, 7 % below.  From two blocks on the kernels below are level (forward, 266 calls,
// 0.98 on average) or faster (dQ/dR, 0.86).
template <int CT>
__global__ __launch_bounds__(256, 2) void fwd_fp32_kernel(F32Args p)
{
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const Place w(p, wave, lane & 31);
    if (w.none) return;
    f32x16 o[CT];
    fwd_fp32<CT>(p, w, lds, wave, o);
    if (w.valid)
        store_row<CT>(o, p.parts.nsplit > 1 ? p.part + (((long)w.z * p.rows.Hkuv + w.hk) * p.rows.n + w.row) * p.DH
                                            : p.O + p.rows.tok(w.hk, w.row) * p.DH, lane >> 5, p.DH);
}
// Where a part leaves the sums of dR of this lane's row.
__device__ __forceinline__ float* dr_row(const F32Args& p, const Place& w)
{
    const long hrows = (long)p.rows.Hkuv * p.rows.n;
    return p.parts.nsplit > 1 ? p.part + p.parts.nsplit * hrows * p.DH + (w.z * hrows + (long)w.hk * p.rows.n + w.row) * p.parts.E
                              : p.dR + p.rows.gate(w.hk, w.row) * p.parts.E;
}
template <int CT>
__global__ __launch_bounds__(256, CT > 3 ? 1 : 2) void dqdr_fp32_kernel(F32Args p)
{
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const Place w(p, wave, lane & 31);
    if (w.none) return;
    f32x16 dq[CT];
    dqdr_fp32<CT>(p, w, lds, wave, dr_row(p, w), w.valid, dq);
    if (w.valid)
        store_row<CT>(dq, p.parts.nsplit > 1 ? p.part + (((long)w.z * p.rows.Hkuv + w.hk) * p.rows.n + w.row) * p.DH
                                             : p.dQ + p.rows.tok(w.hk, w.row) * p.DH, lane >> 5, p.DH);
}

// Forward: 128 rows, GROUPS teams of four waves that take the blocks of the part in turn, their sums added at the end.  A team's
// threads take the next block's weights apart on their way from memory to LDS, K and U under the second products, V under the first.
template <int CT, int GROUPS>
__global__ __launch_bounds__(256 * GROUPS, GROUPS) void fwd_f32_kernel(F32Args p)
{
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), group = wave >> 2;
    const Place w(p, wave & 3, l32);
    if (w.none) return;
    const int DH = p.DH;
    const Cut<CT> cut(threadIdx.x & 255);
    const PlaneLane pl(lane);
    unsigned char* planes = lds + group * 3 * PLANES_B;      // K, U, V

    auto block = [&](int it) { return Block(p, w.hk, w.blk0 + (it * GROUPS + group < w.nblk ? it * GROUPS + group : w.nblk - 1)); };
    f32x4 xk[CT], xu[CT], xv[CT];
    {
        const Block b = block(0);
        cut.load(xk, p.K + b.wrow * DH, b.rows, DH);
        cut.load(xu, p.U + b.wrow * DH, b.rows, DH);
        cut.load(xv, p.V + b.wrow * DH, b.rows, DH);
    }
    f32x4 qx[4 * CT];
    load_row_operand<CT>(qx, p.Q + p.rows.tok(w.hk, w.row) * DH, g, DH);
    Split8 q[2 * CT];
    split_row_operand<CT>(q, qx);
    const float* rrow = p.R + p.rows.gate(w.hk, w.row) * p.parts.E;
    f32x16 o[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) o[ct] = zero16();
#pragma unroll
    for (int k = 0; k < CT; ++k) {
        cut.store(planes, k, xk[k]);
        cut.store(planes + PLANES_B, k, xu[k]);
    }
    const int iters = (w.nblk + GROUPS - 1) / GROUPS;
    Block b = block(0);
    float r = group < w.nblk ? rrow[b.e] : 0.0f;      // (0 removes the block that a team lacks in the last turn)
    if (group == 1) {
        __syncthreads();
        __builtin_amdgcn_s_setprio(2);
    }
    for (int it = 0; it < iters; ++it) {
        const Block next = block(it + 1);
        __syncthreads();      // K and U are there, and V has been read
        const float rnext = (it + 1) * GROUPS + group < w.nblk ? rrow[next.e] : 0.0f;
        cut.load(xk, p.K + next.wrow * DH, next.rows, DH);
        cut.load(xu, p.U + next.wrow * DH, next.rows, DH);
        f32x16 mn[2];
        first_split<CT, 2, 1>(mn, planes, {q, q}, pl, NoAcc{}, [&](auto ic) {
            constexpr int i = decltype(ic)::value, k = i / 24;      // 24 CT instructions, CT pieces
            if constexpr (i % 24 == 11) cut.store(planes + 2 * PLANES_B, k, xv[k]);
        });
        __syncthreads();      // V is there, and K and U have been read
        cut.load(xv, p.V + next.wrow * DH, next.rows, DH);
        f32x16 &m = mn[0], &n = mn[1];
        mfma_result_fence(m, n);
#pragma unroll
        for (int i = 0; i < 16; ++i) m[i] = m[i] * sigmoid16(m[i]) * (0.0625f * DOWN1) * n[i] * r;
        if (b.rows < JB) {
#pragma unroll
            for (int i = 0; i < 16; ++i) m[i] = split_row(i, g) < b.rows ? m[i] : 0.0f;
        }
        static_for<2>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            const Split8 ps = split8([&](int i) { return m[8 * s + i]; });
            second_split<CT>(o, planes + 2 * PLANES_B, s, ps, pl, [&](auto ic) {
                constexpr int i = decltype(ic)::value, k = i / 6;
                if constexpr (i % 6 == 5) cut.store(planes + s * PLANES_B, k, s ? xu[k] : xk[k]);
            });
        });
        b = next;
        r = rnext;
    }
    if (GROUPS > 1 && group == 0) __syncthreads();
    if (GROUPS > 1) {
        __syncthreads();
        float* xch = reinterpret_cast<float*>(lds) + (wave & 3) * (CT * 16 * 64) + lane;
        if (group == 1) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int i = 0; i < 16; ++i) xch[(ct * 16 + i) * 64] = o[ct][i];
        }
        __syncthreads();
        if (group == 1) return;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[ct][i] += xch[(ct * 16 + i) * 64];
    }
    // (the place of a lane's row is worked out anew, out of the compiler's sight, instead of kept)
    int l32b = l32;
    asm volatile("" : "+v"(l32b));
    const Place w2(p, wave, l32b);
    const bool again = in_row(!finite(o)) && w2.valid;
    scale(o, DOWN2);
    float* dst = p.parts.nsplit > 1 ? p.part + (((long)w2.z * p.rows.Hkuv + w2.hk) * p.rows.n + w2.row) * DH : p.O + p.rows.tok(w2.hk, w2.row) * DH;
    if (w2.valid && !again) store_row<CT>(o, dst, g, DH);
    if (!anywhere(again, lds + GROUPS * 3 * PLANES_B - 16, wave)) return;
    fwd_fp32<CT>(p, w2, lds, wave, o);
    if (again) store_row<CT>(o, dst, g, DH);
}

// dQ and dR: four waves of 32 rows, alone on their SIMDs.  LDS: the planes of two blocks; the next block's weights are taken apart
// between the matrix instructions of this block's first products, and the element-wise code of its second half of rows between
// those of the second products of the first.
template <int CT>
__global__ __launch_bounds__(256, 1) void dqdr_f32_kernel(F32Args p)
{
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Place w(p, wave, l32);
    if (w.none) return;
    const int DH = p.DH, E = p.parts.E;
    const Cut<CT> cut(threadIdx.x);
    const PlaneLane pl(lane);

    f32x4 x[3][CT];
    auto load = [&](int blk) {
        const Block b(p, w.hk, w.blk0 + (blk < w.nblk ? blk : w.nblk - 1));
        cut.load(x[0], p.K + b.wrow * DH, b.rows, DH);
        cut.load(x[1], p.U + b.wrow * DH, b.rows, DH);
        cut.load(x[2], p.V + b.wrow * DH, b.rows, DH);
    };
    load(0);
    const long tok = p.rows.tok(w.hk, w.row) * DH;
    Split8 q[2 * CT], go[2 * CT];
    {
        f32x4 qx[4 * CT], gx[4 * CT];
        load_row_operand<CT>(qx, p.Q + tok, g, DH);
        load_row_operand<CT>(gx, p.dO + tok, g, DH);
        split_row_operand<CT>(q, qx);
        split_row_operand<CT>(go, gx);
    }
    if (CT < 4) {      // (held there over the loop; with 64 registers more the compiler does better by itself)
#pragma unroll
        for (int ks = 0; ks < 2 * CT; ++ks)
#pragma unroll
            for (int x = 0; x < 3; ++x) asm volatile("" : "+a"(q[ks].p[x]), "+a"(go[ks].p[x]));
    }
    const float* rrow = p.R + p.rows.gate(w.hk, w.row) * E;
    float* drow = dr_row(p, w);
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int k = 0; k < CT; ++k) cut.store(lds + t * PLANES_B, k, x[t][k]);
    load(1);

    f32x16 dq[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) dq[ct] = zero16();
    float dr = 0.0f;
    bool again = false;      // a result of this row is not finite
    Block b(p, w.hk, w.blk0);
    float r = rrow[b.e];
    for (int blk = 0; blk < w.nblk; ++blk) {
        const Block next(p, w.hk, w.blk0 + (blk + 1 < w.nblk ? blk + 1 : blk));
        const float rnext = rrow[next.e];
        const unsigned char* planes = lds + (blk & 1) * 3 * PLANES_B;
        unsigned char* other = lds + (~blk & 1) * 3 * PLANES_B;
        __syncthreads();      // this block's planes are there, and the other ones have been read
        f32x16 mna[3];
        CutPiece c;
        first_split<CT, 3, 1>(mna, planes, {q, q, go}, pl, AllAcc{}, [&](auto ic) {
            constexpr int i = decltype(ic)::value, t = i / 12 / CT, k = i / 12 % CT;      // 36 CT instructions, 3 CT pieces
            if constexpr (i % 12 == 3) c.half<0>(x[t][k]);
            if constexpr (i % 12 == 6) c.half<1>(x[t][k]);
            if constexpr (i % 12 == 9) cut.store(other + t * PLANES_B, k, c);
        });
        load(blk + 2);
        f32x16 &m = mna[0], &n = mna[1], &da = mna[2];
        mfma_result_fence(m, n, da);
        if (b.rows < JB) {
#pragma unroll
            for (int i = 0; i < 16; ++i) da[i] = split_row(i, g) < b.rows ? da[i] : 0.0f;
        }
        float sg16;
        auto sigma = [&](int i) { sg16 = sigmoid16(m[i]); };
        auto element = [&](int i) {      // (sl and nn as they are; da, dM, dN and dR times 2^48)
            const float sl = m[i] * sg16 * (0.0625f * DOWN1), sg = 0.0625f * sg16, nn = DOWN1 * n[i], a = da[i] * sl, ra = r * da[i];
            dr = fmaf(a, nn, dr);
            m[i] = ra * nn * fmaf(sl, 1.0f - sg, sg);           // dM
            n[i] = r * a;                                       // dN
        };
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            sigma(i);
            element(i);
        }
        // The second products of the first eight rows; behind their matrix instructions the rest of the element-wise code.
        u32x4 dm[3], dn[3], dm1[3];
        static_for<4>([&](auto ic) { split8_pair<decltype(ic)::value>(dm, [&](int i) { return m[i]; }); });
        second_split<CT>(dq, planes, 0, split8_of(dm), pl, [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i < 4) split8_pair<i>(dn, [&](int j) { return n[j]; });
            else if constexpr (i < 8 || (i < 16 && CT > 2)) {
                if constexpr (i & 1) element(8 + (i - 4) / 2);
                else sigma(8 + (i - 4) / 2);
            }
        });
        constexpr int DONE = CT == 1 ? 9 : CT == 2 ? 10 : 14;      // (6, 12 or 18 instructions and more)
        second_split<CT>(dq, planes + PLANES_B, 0, split8_of(dn), pl, [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i < 2 * (16 - DONE)) {
                if constexpr (i & 1) element(DONE + i / 2);
                else sigma(DONE + i / 2);
            } else if constexpr (i < 2 * (16 - DONE) + 4) split8_pair<i - 2 * (16 - DONE)>(dm1, [&](int j) { return m[8 + j]; });
        });
        static_for<16>([&](auto ic) {      // (what d_h < 96 leaves)
            constexpr int i = decltype(ic)::value;
            if constexpr (i >= DONE + 3 * CT) {
                sigma(i);
                element(i);
            }
        });
        if constexpr (6 * CT < 2 * (16 - DONE) + 4) static_for<4>([&](auto ic) { split8_pair<decltype(ic)::value>(dm1, [&](int j) { return m[8 + j]; }); });
        second_split<CT>(dq, planes, 1, split8_of(dm1), pl, [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i < 4) split8_pair<i>(dn, [&](int j) { return n[8 + j]; });
        });
        second_split<CT>(dq, planes + PLANES_B, 1, split8_of(dn), pl, [](auto) {});
        if (blk + 1 == w.nblk || next.e != b.e) {
            const float tot = dr + __shfl_xor(dr, 32);      // the two lane halves hold different rows j of the same token
            if (g == 0 && w.valid) drow[b.e] = DOWN1 * tot;
            again |= !finite(tot);
            dr = 0.0f;
        }
        b = next;
        r = rnext;
    }
    again |= !finite(dq);
    again = in_row(again) && w.valid;
    scale(dq, DOWN2);
    float* dst = p.parts.nsplit > 1 ? p.part + (((long)w.z * p.rows.Hkuv + w.hk) * p.rows.n + w.row) * DH : p.dQ + tok;
    if (w.valid && !again) store_row<CT>(dq, dst, g, DH);
    if (!anywhere(again, lds + 6 * PLANES_B - 16, wave)) return;
    dqdr_fp32<CT>(p, w, lds, wave, drow, again, dq);
    if (again) store_row<CT>(dq, dst, g, DH);
}

// Head and pair of blocks of a workgroup of dK/dU/dV.  The head runs fastest, so that a head's weights, which dQ/dR has read, are in the L2 of
// the XCD (both kernels, 256 tokens of the 128M layer 79.2 us in the other order, 77.4; 32 tokens 43.5, 41.5); several slices run in the other
// order, in which their sums are read faster (500 tokens on four K/U/V heads 131.8, 133.8).
__device__ __forceinline__ int head_of(const F32Args& p) { return p.heads_first ? blockIdx.x : blockIdx.y; }
__device__ __forceinline__ int pair_of(const F32Args& p) { return p.heads_first ? blockIdx.y : blockIdx.x; }

// End of a dK/dU/dV kernel: the odd tiles' sums to the wave with the even ones (64 lanes x 48 CT floats, lane-private), then the
// rows that `take` picks to memory: take(finite) says whether a row goes, given whether all of it is finite.  (This lane's row and
// the bounds of its columns are worked out again, out of the compiler's sight: kept over the loop they are the few registers too many
// that made it spill for d_h > 96.)
template <int CT, class Take>
__device__ __forceinline__ void add_halves_and_store(const F32Args& p, unsigned char* lds, f32x16 (&dk)[CT], f32x16 (&du)[CT], f32x16 (&dv)[CT],
                                                     Take&& take)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wave >> 1, bw = wave & 1;
    const int hk = head_of(p), z = blockIdx.z, E = p.parts.E, nblk = E * p.parts.nbe;
    const int blk = pair_of(p) * 2 + bw;
    const Block b(p, hk, blk < nblk ? blk : nblk - 1);
    __syncthreads();
    int lane = threadIdx.x & 63, DH = p.DH;
    asm volatile("" : "+v"(lane), "+s"(DH));
    const int l32 = lane & 31, g = lane >> 5;
    float* xch = reinterpret_cast<float*>(lds) + bw * (3 * CT * 16 * 64) + lane;
    if (half == 1) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                xch[(ct * 16 + i) * 64] = dk[ct][i];
                xch[((CT + ct) * 16 + i) * 64] = du[ct][i];
                xch[((2 * CT + ct) * 16 + i) * 64] = dv[ct][i];
            }
    }
    __syncthreads();
    if (half == 1 || blk >= nblk) return;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            dk[ct][i] += xch[(ct * 16 + i) * 64];
            du[ct][i] += xch[((CT + ct) * 16 + i) * 64];
            dv[ct][i] += xch[((2 * CT + ct) * 16 + i) * 64];
        }
    if (!take([&] { return !in_row(!finite(dk) || !finite(du) || !finite(dv)); }) || l32 >= b.rows) return;
    const long wrow = b.wrow + l32, wsz = (long)p.rows.Hkuv * E * p.de * DH;
    auto store_bf16 = [&](const f32x16(&acc)[CT], void* out) {
        bf16_t* dst = static_cast<bf16_t*>(out) + wrow * DH;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int a = 0; a < 4; ++a)
                if (32 * ct + 8 * a < DH) {
                    bf16x4 v;
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[x] = (bf16_t)acc[ct][4 * a + x];
                    *reinterpret_cast<bf16x4*>(dst + 32 * ct + 8 * a + 4 * g) = v;
                }
    };
    if (p.nslice > 1) {
        float* dst = p.part + (long)z * 3 * wsz + wrow * DH;
        store_row<CT>(dk, dst, g, DH);
        store_row<CT>(du, dst + wsz, g, DH);
        store_row<CT>(dv, dst + 2 * wsz, g, DH);
    } else if (p.out_f32) {
        store_row<CT>(dk, static_cast<float*>(p.out[0]) + wrow * DH, g, DH);
        store_row<CT>(du, static_cast<float*>(p.out[1]) + wrow * DH, g, DH);
        store_row<CT>(dv, static_cast<float*>(p.out[2]) + wrow * DH, g, DH);
    } else {
        store_bf16(dk, p.out[0]);
        store_bf16(du, p.out[1]);
        store_bf16(dv, p.out[2]);
    }
}

// dK, dU, dV.  A wave owns one block of weight rows (B operands and accumulators stay in registers) and every other
// 32-row tile of its slice of the head's rows: waves 0, 1 take the even tiles of two blocks, waves 2, 3 the odd ones, and their
// sums meet in LDS at the end.  (Halving the tiles inside the workgroup doubles the workgroups of a layer whose blocks are
// few, without partial sums in memory; LDS is idle, so that each pair of waves has tiles of its own costs nothing.)
template <int CT>
__device__ __forceinline__ void dkdudv_fp32(const F32Args& p, unsigned char* lds, f32x16 (&dk)[CT], f32x16 (&du)[CT], f32x16 (&dv)[CT])
{
    using T = Tile<CT>;
    constexpr int FI = T::INS / 2 > 0 ? T::INS / 2 : 1;
    constexpr int STAGE_B = 2 * T::BYTES;      // Q and dO tile
    float* sR = reinterpret_cast<float*>(lds + 4 * STAGE_B);      // [stage][wave][32] gate values
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wave >> 1, bw = wave & 1;
    const int hk = head_of(p), z = blockIdx.z, E = p.parts.E, nblk = E * p.parts.nbe;
    const int blk = pair_of(p) * 2 + bw;
    const Block b(p, hk, blk < nblk ? blk : nblk - 1);

    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5, DH = p.DH;
    const int ntile = (p.rows.n + 31) / 32;
    const int t0 = (int)((long)ntile * z / p.nslice), t1 = (int)((long)ntile * (z + 1) / p.nslice);
    const int steps = (t1 - t0 + 1) / 2;
    auto fill = [&](int s) {
        const int t = t0 + 2 * s + half;
        const int row0 = 32 * (t < ntile ? t : ntile - 1);
        unsigned char* stage = lds + (half * 2 + (s & 1)) * STAGE_B;
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));      // (the fills' addresses are not worth a register each)
        auto row = [&](const float* W) {
            return [&, W](int r) { return W + p.rows.tok_head_major(hk, row0 + r < p.rows.n ? row0 + r : p.rows.n - 1) * DH; };
        };
#pragma unroll
        for (int k = 0; k < FI; ++k) {
            T::fill(stage, bw * FI + k, lane, DH, row(p.Q));
            T::fill(stage + T::BYTES, bw * FI + k, lane, DH, row(p.dO));
        }
        // gate values of this wave's expert; 0 for the rows that a tile lacks, which removes them from every product
        if (g == 0) {
            const bool ok = t < t1 && row0 + l32 < p.rows.n;
            sR[((s & 1) * 4 + wave) * 32 + l32] = ok ? p.R[p.rows.head_major(hk, ok ? row0 + l32 : 0) * E + b.e] : 0.0f;
        }
    };
    fill(0);
    f32x4 kB[4 * CT], uB[4 * CT], vB[4 * CT];
    const long wrow = b.wrow + (l32 < b.rows ? l32 : b.rows - 1);
    load_row<CT>(kB, p.K + wrow * DH, g, DH);
    load_row<CT>(uB, p.U + wrow * DH, g, DH);
    load_row<CT>(vB, p.V + wrow * DH, g, DH);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) { dk[ct] = zero16(); du[ct] = zero16(); dv[ct] = zero16(); }

    for (int s = 0; s < steps; ++s) {
        const unsigned char *sQ = lds + (half * 2 + (s & 1)) * STAGE_B, *sG = sQ + T::BYTES;
        wait_vmcnt<0>();
        __syncthreads();
        if (s + 1 < steps) fill(s + 1);
        f32x16 mna[3];
        const typename T::Lane l(l32, g);
        first_products<CT, 3>(mna, {sQ, sQ, sG}, {kB, uB, vB}, l);
        f32x16 &m = mna[0], &n = mna[1], &da = mna[2];
        const float* rw = sR + ((s & 1) * 4 + wave) * 32;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float r = rw[reg_row(i, g)], sg = sigmoid_exact(m[i]), sl = m[i] * sg, a = da[i], nn = n[i];
            m[i] = r * a * nn * (sg + sl * (1.0f - sg));      // dM
            n[i] = r * a * sl;                                // dN
            da[i] = r * sl * nn;                              // P
        }
        second_product<CT>(dk, sQ, m, l);
        second_product<CT>(du, sQ, n, l);
        second_product<CT>(dv, sG, da, l);
    }
}

// dK, dU, dV for d_h <= 96.  A wave owns one block of weight rows (the planes of its rows and the accumulators stay in registers)
// and every other 32-row tile of its slice of the head's rows: waves 0, 1 take the even tiles of two blocks, waves 2, 3 the odd
// ones, and their sums meet in LDS at the end.  The two waves of a tile take it apart; its float32 values, requested a step
// ahead, wait in LDS where the lane that needs them put them (there are no registers for them).
template <int CT>
__global__ __launch_bounds__(256, 1) void dkdudv_split_kernel(F32Args p)
{
    static_assert(CT <= 3, "");
    constexpr int RAW = 4 * CT;                // 16-byte loads of a lane and step: Q and dO, two halves of the rows, CT column groups
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wave >> 1, bw = wave & 1;
    unsigned char* planes = lds + half * 2 * PLANES_B;                            // Q, dO
    unsigned char* raw = lds + 4 * PLANES_B + wave * RAW * 1024;
    float* sR = reinterpret_cast<float*>(lds + 4 * PLANES_B + 4 * RAW * 1024) + wave * 32;      // gate values of the wave's expert
    const int hk = head_of(p), z = blockIdx.z, E = p.parts.E, nblk = E * p.parts.nbe, DH = p.DH;
    const int blk = pair_of(p) * 2 + bw;
    const Block b(p, hk, blk < nblk ? blk : nblk - 1);
    const int ntile = (p.rows.n + 31) / 32;
    const int t0 = (int)((long)ntile * z / p.nslice), t1 = (int)((long)ntile * (z + 1) / p.nslice);
    const int steps = (t1 - t0 + 1) / 2;

    const Cut<CT> cut(threadIdx.x & 127);      // rows 0 .. 15 of a tile; the same columns of rows 16 .. 31
    auto request = [&](int s) {
        const int t = t0 + 2 * s + half, row0 = 32 * (t < ntile ? t : ntile - 1);
        int col = cut.col;
        asm volatile("" : "+v"(col));      // (the addresses are not worth a register each)
        const int last = 32 * (CT - 1) + col < DH ? 32 * (CT - 1) : -col;      // (columns beyond d_h: any; they are replaced by zero below)
        static_for<4>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int r = row0 + 16 * (i & 1) + cut.row;
            const float* src = (i < 2 ? p.Q : p.dO) + p.rows.tok_head_major(hk, r < p.rows.n ? r : p.rows.n - 1) * DH + col;
            static_for<CT - 1>([&](auto kc) { lds_direct16<128 * decltype(kc)::value>(src, raw + (i * CT + decltype(kc)::value) * 1024); });
            lds_direct16<0>(src + last, raw + (i * CT + CT - 1) * 1024);
        });
    };
    // gate value of row l32 of this wave's next tile; 0 for the rows that a tile lacks, which removes them from every product
    auto gate = [&](int s) {
        const int t = t0 + 2 * s + half, r = 32 * t + l32;
        const bool ok = t < t1 && r < p.rows.n;
        return ok ? p.R[p.rows.head_major(hk, ok ? r : 0) * E + b.e] : 0.0f;
    };
    request(0);
    float rg = gate(0);
    Split8 kB[2 * CT], uB[2 * CT], vB[2 * CT];
    const long wrow = b.wrow + (l32 < b.rows ? l32 : b.rows - 1);
    {
        f32x4 x[2][4 * CT];
        load_row_operand<CT>(x[0], p.K + wrow * DH, g, DH);
        load_row_operand<CT>(x[1], p.U + wrow * DH, g, DH);
        __builtin_amdgcn_sched_barrier(0);
        split_row_operand<CT>(kB, x[0]);
#pragma unroll
        for (int ks = 0; ks < 2 * CT; ++ks)
#pragma unroll
            for (int i = 0; i < 3; ++i) asm volatile("" : "+a"(kB[ks].p[i]));
        load_row_operand<CT>(x[0], p.V + wrow * DH, g, DH);
        __builtin_amdgcn_sched_barrier(0);
        split_row_operand<CT>(uB, x[1]);
#pragma unroll
        for (int ks = 0; ks < 2 * CT; ++ks) asm volatile("" : "+v"(uB[ks].p[0]), "+v"(uB[ks].p[1]), "+a"(uB[ks].p[2]));
        __builtin_amdgcn_sched_barrier(0);
        split_row_operand<CT>(vB, x[0]);
    }
    const PlaneLane pl(lane);
    f32x16 dk[CT], du[CT], dv[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) { dk[ct] = zero16(); du[ct] = zero16(); dv[ct] = zero16(); }

    for (int s = 0; s < steps; ++s) {
        wait_vmcnt<0>();      // this lane's values have landed
        __builtin_amdgcn_sched_barrier(0);
        static_for<RAW>([&](auto ic) {
            constexpr int i = decltype(ic)::value, k = i % CT, h = i / CT % 2;
            f32x4 x = *reinterpret_cast<const f32x4*>(raw + i * 1024 + lane * 16);
            if (32 * k + cut.col >= DH) x = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            cut.store(planes + (i < 2 * CT ? 0 : PLANES_B) + h * 16 * TILE_ROW_B, k, x);
        });
        if (g == 0) sR[l32] = rg;
        __syncthreads();      // the planes are there, and this lane's values have been read
        request(s + 1 < steps ? s + 1 : s);
        rg = gate(s + 1);
        f32x16 mna[3];
        first_split<CT, 3, 2>(mna, planes, {kB, uB, vB}, pl, WeightAcc{}, [](auto) {});
        f32x16 &m = mna[0], &n = mna[1], &da = mna[2];
        f32x4 r4[2];
        auto gates = [&](int h) {
            r4[0] = *reinterpret_cast<const f32x4*>(sR + split_row(8 * h, g));
            r4[1] = *reinterpret_cast<const f32x4*>(sR + split_row(8 * h + 4, g));
        };
        gates(0);
        mfma_result_fence(m, n, da);
        float sg16;
        auto sigma = [&](int i) { sg16 = sigmoid16(m[i]); };
        auto element = [&](int i) {      // (sl and nn as they are; da, dM, dN and P times 2^48)
            const float r = r4[(i >> 2) & 1][i & 3], sl = m[i] * sg16 * (0.0625f * DOWN1), sg = 0.0625f * sg16, ra = r * da[i], ns = n[i], nn = DOWN1 * ns;
            m[i] = ra * nn * fmaf(sl, 1.0f - sg, sg);      // dM
            n[i] = ra * sl;                                // dN
            da[i] = r * sl * ns;                           // P
        };
        static_for<8>([&](auto ic) {
            sigma(decltype(ic)::value);
            element(decltype(ic)::value);
            __builtin_amdgcn_sched_barrier(0);
        });
        gates(1);
        // The second products of the first eight rows; behind their 18 CT matrix instructions the rest of the element-wise code.
        u32x4 dm[3], dn[3], pp[3];
        auto pair = [&](auto ic, u32x4(&v)[3], const f32x16& x, int first) {
            split8_pair<decltype(ic)::value>(v, [&](int j) { return x[first + j]; });
        };
        auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
        static_for<4>([&](auto ic) { pair(ic, dm, m, 0); });
        second_split<CT>(dk, planes, 0, split8_of(dm), pl, [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i < 4) pair(ic, dn, n, 0);
            fence();
        });
        second_split<CT>(du, planes, 0, split8_of(dn), pl, [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i < 4) pair(ic, pp, da, 0);
            fence();
        });
        second_split<CT>(dv, planes + PLANES_B, 0, split8_of(pp), pl, [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i < 16) {
                if constexpr (i & 1) element(8 + i / 2);
                else sigma(8 + i / 2);
            }
            fence();
        });
        static_for<16>([&](auto ic) {      // (what d_h < 96 leaves)
            constexpr int i = decltype(ic)::value;
            if constexpr (i >= 8 + 3 * CT) {
                sigma(i);
                element(i);
                fence();
            }
        });
        static_for<4>([&](auto ic) { pair(ic, dm, m, 8); });
        second_split<CT>(dk, planes, 1, split8_of(dm), pl, [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i < 4) pair(ic, dn, n, 8);
            fence();
        });
        second_split<CT>(du, planes, 1, split8_of(dn), pl, [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i < 4) pair(ic, pp, da, 8);
            fence();
        });
        second_split<CT>(dv, planes + PLANES_B, 1, split8_of(pp), pl, [](auto) {});
        __syncthreads();      // the planes have been read
    }
    wait_vmcnt<0>();         // what the last step has requested is not used, but lands in LDS
    scale(dk, DOWN2);
    scale(du, DOWN2);
    scale(dv, DOWN2);
    bool again = false;      // this lane's row is not finite
    add_halves_and_store<CT>(p, lds, dk, du, dv, [&](auto all_finite) { return !(again = !all_finite()); });
    if (!anywhere(again, lds + 4 * PLANES_B + 16 * CT * 1024, wave)) return;
    dkdudv_fp32<CT>(p, lds, dk, du, dv);
    add_halves_and_store<CT>(p, lds, dk, du, dv, [&](auto) { return again; });
}

template <int CT>
__global__ __launch_bounds__(256, 1) void dkdudv_f32_kernel(F32Args p)
{
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    f32x16 dk[CT], du[CT], dv[CT];
    dkdudv_fp32<CT>(p, lds, dk, du, dv);
    add_halves_and_store<CT>(p, lds, dk, du, dv, [](auto) { return true; });
}

// Adds the parts' sums in order: the rows of O or dQ (dst, four columns per lane) and, behind a tile's row_blocks, the values of dR over
// the parts that hold blocks of the expert.  Workgroups count tiles and heads as the kernel that left the parts did (whole_xcds).
__global__ __launch_bounds__(256) void sum_f32_kernel(F32Args p, float* dst, unsigned row_blocks, unsigned tiles, FastDiv by_tiles)
{
    const unsigned block = by_tiles.div(blockIdx.x), x = blockIdx.x - block * tiles;
    const int tile = p.rows.by_hkuv.div(x), hk = x - tile * p.rows.Hkuv, DH = p.DH, E = p.parts.E;
    const long hrows = (long)p.rows.Hkuv * p.rows.n;
    if (block < row_blocks) {
        const unsigned i = block * 256 + threadIdx.x, row = i / (unsigned)(DH / 4), r = tile * F32_ROWS + row;
        const int c = (i - row * (DH / 4)) * 4;
        if (row >= (unsigned)F32_ROWS || r >= (unsigned)p.rows.n) return;
        const float* src = p.part + ((long)hk * p.rows.n + r) * DH + c;
        auto load = [&](int z) { return *reinterpret_cast<const f32x4*>(src + z * hrows * DH); };
        *reinterpret_cast<f32x4*>(dst + p.rows.tok(hk, r) * DH + c) = sum_in_order(load(0), 1, p.parts.nsplit, load);
    } else {
        const unsigned i = (block - row_blocks) * 256 + threadIdx.x, row = i / (unsigned)E, r = tile * F32_ROWS + row;
        const int e = i - row * E;
        if (row >= (unsigned)F32_ROWS || r >= (unsigned)p.rows.n) return;
        const float* src = p.part + p.parts.nsplit * hrows * DH + ((long)hk * p.rows.n + r) * E + e;
        p.dR[p.rows.gate(hk, r) * E + e] =
            sum_in_order(0.0f, p.parts.part_lo(e), p.parts.part_hi(e), [&](int z) { return src[z * hrows * E]; });
    }
}

template <typename OutT>
__global__ __launch_bounds__(256) void reduce_f32_kernel(const float* __restrict__ part, OutT* dK, OutT* dU, OutT* dV,
                                                         long wsz, int nslice)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= wsz) return;
    OutT* outs[3] = {dK, dU, dV};
    for (int w = 0; w < 3; ++w) {
        outs[w][i] = (OutT)sum_in_order(0.0f, 0, nslice, [&](int z) { return part[((long)z * 3 + w) * wsz + i]; });
    }
}

// Parts of the blocks for the forward and dQ/dR as for bfloat16 (pick_parts).  A block took 5 us on the fp32 instructions and takes half of it;
// the choice does not depend on it: with any step from 2 to 5 us it loses 1.7 to 2.1 (forward) and 1.2 to 2.1 % (dQ/dR) to the best number
// of parts, 28 and 20 % at worst, over 165 calls (twelve layers of d_h 8 to 128; 1 to 1,500 tokens).
constexpr Variant F32_VARIANTS[] = {{128, 5.0, 0.0, 1}};
int nbe_of(const Dims& d) { return (d.d_e + JB - 1) / JB; }
size_t o_part_bytes(const Dims& d) { return (size_t)d.B * d.H * d.S * d.d_h * sizeof(float); }
size_t dq_part_bytes(const Dims& d) { return (size_t)d.B * d.H * d.S * (d.d_h + d.E) * sizeof(float); }
Pick pick_f32(const Dims& d, size_t part_bytes, size_t ws_bytes, int phases)
{
    return pick_parts(F32_VARIANTS, d, d.E * nbe_of(d), true, part_bytes, phases & PH_ONE_PART ? 0 : ws_bytes);
}

F32Args f32_args(const void* Q, const void* K, const void* U, const void* V, const float* R, const Dims& d, int nsplit)
{
    F32Args a{};
    a.Q = (const float*)Q; a.K = (const float*)K; a.U = (const float*)U; a.V = (const float*)V; a.R = R;
    a.rows = RowMap(d);
    a.parts = Parts(d.E, nbe_of(d), nsplit);
    a.DH = d.d_h; a.de = d.d_e;
    return a;
}

// Workgroups of the summing pass for a tile's rows of `width` lanes.
unsigned blocks_of_tile(const F32Args& a, int width)
{
    return (unsigned)(((long)(a.rows.n < F32_ROWS ? a.rows.n : F32_ROWS) * width + 255) / 256);
}

template <int CT>
hipError_t launch_fwd_f32_t(const F32Args& a, const Dims& d, hipStream_t st)
{
    constexpr int GROUPS = CT > 3 ? 1 : 2;
    const bool one_block = a.parts.nsplit == a.parts.E * a.parts.nbe;
    const int smem = one_block ? 3 * Tile<CT>::BYTES : GROUPS * 3 * PLANES_B;
    static_assert(GROUPS == 1 || 4 * CT * 16 * 64 * 4 <= GROUPS * 3 * PLANES_B, "the teams' exchange fits the planes");
    static LdsOptIn optin[2];
    auto* fn = one_block ? fwd_fp32_kernel<CT> : fwd_f32_kernel<CT, GROUPS>;
    const hipError_t e = ensure_dynamic_lds(optin[one_block], (const void*)fn, smem);
    if (e != hipSuccess) return e;
    const unsigned tiles = grid_of_part_f32(d, Pick{F32_ROWS, a.parts.nsplit});
    hipLaunchKernelGGL(fn, dim3(tiles, (unsigned)a.parts.nsplit), dim3(one_block ? 256 : 256 * GROUPS), smem, st, a);
    if (a.parts.nsplit > 1) {
        const unsigned rb = blocks_of_tile(a, d.d_h / 4);
        hipLaunchKernelGGL(sum_f32_kernel, dim3(tiles * rb), dim3(256), 0, st, a, a.O, rb, tiles, FastDiv(tiles));
    }
    return hipGetLastError();
}

template <int CT>
hipError_t launch_bwd_f32_t(F32Args a, const Dims& d, hipStream_t st, int phases)
{
    hipError_t err = hipSuccess;
    if (phases & PH_BWD_DQDR) {
        const bool one_block = a.parts.nsplit == a.parts.E * a.parts.nbe;
        const int smem = one_block ? 3 * Tile<CT>::BYTES : 6 * PLANES_B;
        static LdsOptIn optin[2];
        auto* fn = one_block ? dqdr_fp32_kernel<CT> : dqdr_f32_kernel<CT>;
        err = ensure_dynamic_lds(optin[one_block], (const void*)fn, smem);
        if (err != hipSuccess) return err;
        const unsigned tiles = grid_of_part_f32(d, Pick{F32_ROWS, a.parts.nsplit});
        hipLaunchKernelGGL(fn, dim3(tiles, (unsigned)a.parts.nsplit), dim3(256), smem, st, a);
        if (a.parts.nsplit > 1) {
            const unsigned rb = blocks_of_tile(a, d.d_h / 4), eb = blocks_of_tile(a, d.E);
            hipLaunchKernelGGL(sum_f32_kernel, dim3(tiles * (rb + eb)), dim3(256), 0, st, a, a.dQ, rb, tiles, FastDiv(tiles));
        }
        err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    if (phases & PH_BWD_DKDUDV) {
        dim3 grid((unsigned)((d.E * nbe_of(d) + 1) / 2), (unsigned)d.Hkuv, (unsigned)a.nslice);
        a.heads_first = a.nslice == 1 && grid.x <= 65535;
        if (a.heads_first) std::swap(grid.x, grid.y);
        // on the fp32 instructions: d_h > 96, and one step of d_h <= 32 (7.8 of 8.2 us; of d_h 33 to 96 5 % more, two steps 8 to 20 %)
        constexpr bool EVER = CT == 1 || CT > 3, ALWAYS = CT > 3;
        const bool plain = ALWAYS || (EVER && (a.rows.n + 31) / 32 <= 2 * a.nslice);
        auto* kernel = plain ? dkdudv_f32_kernel<EVER ? CT : 1> : dkdudv_split_kernel<ALWAYS ? 1 : CT>;
        const int smem = plain ? 8 * Tile<CT>::BYTES + 2 * 4 * 32 * (int)sizeof(float) : 4 * PLANES_B + 16 * CT * 1024 + 4 * 32 * (int)sizeof(float);
        static_assert(!EVER || 2 * 3 * CT * 16 * 64 * 4 <= 8 * Tile<CT>::BYTES, "the waves' exchange fits the tile stages");
        static_assert(ALWAYS || 2 * 3 * CT * 16 * 64 * 4 <= 4 * PLANES_B, "the waves' exchange fits the planes");
        static LdsOptIn optin[2];
        err = ensure_dynamic_lds(optin[plain], (const void*)kernel, smem);
        if (err != hipSuccess) return err;
        hipLaunchKernelGGL(kernel, grid, dim3(256), smem, st, a);
        err = hipGetLastError();
    }
    return err;
}

}  // namespace

Pick fwd_pick_f32(const Dims& d, size_t ws_bytes, int phases) { return pick_f32(d, o_part_bytes(d), ws_bytes, phases); }
Pick dq_pick_f32(const Dims& d, size_t ws_bytes, int phases) { return pick_f32(d, dq_part_bytes(d), ws_bytes, phases); }

// Token slices of dK/dU/dV: only where the workgroups (two blocks of weight rows each) leave compute units idle.
int dw_slices_f32(const Dims& d)
{
    const long groups = ((long)d.E * nbe_of(d) + 1) / 2 * d.Hkuv;
    const long ntile = ((long)(d.H / d.Hkuv) * d.B * d.S + 31) / 32;
    long ns = CUS / groups;
    if (ns > ntile / 2) ns = ntile / 2;
    if (ns > 64) ns = 64;
    return ns < 1 ? 1 : (int)ns;
}

size_t fwd_workspace_bytes_f32(const Dims& d)
{
    const int ns = fwd_pick_f32(d, ~(size_t)0, 0).nsplit;
    return ns > 1 ? ns * o_part_bytes(d) : 0;
}

// (at least one copy of dK, dU, dV, which the launch needs only where it slices the tokens: what callers of earlier versions
// reserve)
// Float32 kernels work longer for a row, so that an XCD's even share counts for more beside the sums: padded up to three tiles an XCD (us, as it is / padded: 268 tokens of the
// 128M layer on four heads 98.7 / 97.7 with gradients), not above (44 tiles 48.8 / 49.1 forward, 28 153.7 / 156.9 and 60 261.2 / 264.0 with gradients).
unsigned grid_of_part_f32(const Dims& d, const Pick& pick)
{
    return tiles_of(d, pick) <= 3 * XCDS ? whole_xcds(d, pick, sizeof(float)) : tiles_of(d, pick);
}

size_t bwd_min_workspace_bytes_f32(const Dims& d)
{
    return (size_t)dw_slices_f32(d) * 3 * d.Hkuv * d.E * d.d_e * d.d_h * sizeof(float);
}

// ... and room for the parts of dQ, dR
size_t bwd_workspace_bytes_f32(const Dims& d)
{
    const size_t dw = bwd_min_workspace_bytes_f32(d);
    const int nq = dq_pick_f32(d, ~(size_t)0, 0).nsplit;
    const size_t dq = nq > 1 ? nq * dq_part_bytes(d) : 0;
    return dw > dq ? dw : dq;
}

hipError_t launch_fwd_f32(const void* Q, const void* K, const void* U, const void* V, const float* R, void* O, void* ws,
                          size_t ws_bytes, const Dims& d, hipStream_t st, int phases)
{
    F32Args a = f32_args(Q, K, U, V, R, d, fwd_pick_f32(d, ws ? ws_bytes : 0, phases).nsplit);
    a.O = (float*)O;
    a.part = (float*)ws;
    switch ((d.d_h + 31) / 32) {
        case 1: return launch_fwd_f32_t<1>(a, d, st);
        case 2: return launch_fwd_f32_t<2>(a, d, st);
        case 3: return launch_fwd_f32_t<3>(a, d, st);
        default: return launch_fwd_f32_t<4>(a, d, st);
    }
}

hipError_t launch_bwd_f32(const void* Q, const void* K, const void* U, const void* V, const float* R, const void* dO,
                          void* dQ, void* dK, void* dU, void* dV, float* dR, int grad_w_f32, void* ws, size_t ws_bytes,
                          const Dims& d, hipStream_t st, int phases)
{
    F32Args a = f32_args(Q, K, U, V, R, d, dq_pick_f32(d, ws_bytes, phases).nsplit);
    a.dO = (const float*)dO; a.dQ = (float*)dQ; a.dR = dR; a.part = (float*)ws;
    a.out[0] = dK; a.out[1] = dU; a.out[2] = dV; a.out_f32 = grad_w_f32;
    a.nslice = dw_slices_f32(d);
    hipError_t err;
    switch ((d.d_h + 31) / 32) {
        case 1: err = launch_bwd_f32_t<1>(a, d, st, phases); break;
        case 2: err = launch_bwd_f32_t<2>(a, d, st, phases); break;
        case 3: err = launch_bwd_f32_t<3>(a, d, st, phases); break;
        default: err = launch_bwd_f32_t<4>(a, d, st, phases); break;
    }
    if (err == hipSuccess && (phases & PH_BWD_REDUCE) && a.nslice > 1) {
        const long wsz = (long)d.Hkuv * d.E * d.d_e * d.d_h;
        const unsigned rblocks = (unsigned)((wsz + 255) / 256);
        if (grad_w_f32)
            hipLaunchKernelGGL((reduce_f32_kernel<float>), dim3(rblocks), dim3(256), 0, st, a.part, (float*)dK, (float*)dU,
                               (float*)dV, wsz, a.nslice);
        else
            hipLaunchKernelGGL((reduce_f32_kernel<bf16_t>), dim3(rblocks), dim3(256), 0, st, a.part, (bf16_t*)dK,
                               (bf16_t*)dU, (bf16_t*)dV, wsz, a.nslice);
        err = hipGetLastError();
    }
    return err;
}

}  // namespace mhffn
