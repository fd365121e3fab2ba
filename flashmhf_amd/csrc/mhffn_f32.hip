// fp32 instantiation of the fused multi-head FFN (forward, dQ/dR, dK/dU/dV), on the fp32 matrix instructions: operands,
// products and sums are float32 and the sigmoid is exact, so results track an fp32 eager evaluation to ~1e-6.  Same fusion
// as the bf16 kernels -- the [tokens, E*d_e] intermediate exists only in registers.  Generic in d_h (multiple of 8, at most
// 128; CT = 32-column tiles of it), d_e and E.
// Formulas: models/flashmhf/modeling_mhffnmoe.py:418-427 (forward), kernels/triton/flash_mlp_moe.py:401-414, 527-542,
// 720-729 (backward).
//
// All products are v_mfma_f32_32x32x2_f32, D = A(32x2) * B(2x32) + C, 64 cycles each:
//       A: lane l holds row (l % 32), k = l / 32         B: lane l holds col (l % 32), k = l / 32
//       C/D: lane l holds col (l % 32), register i holds row 8*(i/4) + 4*(l/32) + (i%4)
// * First products contract over the head dim.  The order of the k index is free as long as A and B agree: with lane group
//   g = l / 32 holding columns 8m + 4g .. +3, one 16-byte read of each operand row feeds four instructions.
// * They are written with rows = j (weight rows) and columns = tokens (in dK/dU/dV: rows = tokens, columns = j), so that
//   register i of the result is, as it stands, the B operand of the second products' step i: k slot g is row
//   8*(i/4) + 4g + i%4.  The A operand of that step is one row of V (K, U; Q, dO) per lane group, read along its columns.
//
// What bounds them: the matrix pipe (an instruction moves 2 operand rows per 64 cycles, so LDS and L2 are idle most of the
// time; 153 TFLOP/s is what a large library product reaches on the card).  256 tokens of the 128M layer, forward + backward:
// 6.0 ms with plain FMAs on 32-token tiles of one workgroup each, the whole E * d_e axis in series; see the launchers for
// how the work is spread over the chip now.
#include "mhffn_common.hpp"

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
};

__device__ __forceinline__ f32x16 mfma2(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float sigmoid_exact(float x) { return 1.0f / (1.0f + __expf(-x)); }
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

// Workgroup of the forward and of dQ/dR: 4 waves of 32 rows of one K/U/V head, one part of the head's blocks.
struct Place {
    int hk, z, row0, row, blk0, nblk;      // row0: this wave's first row of the list, row: this lane's (clamped into the list)
    bool valid;                            // this lane's row exists
    __device__ explicit Place(const F32Args& p, int wave, int l32)
    {
        const int tile = p.rows.by_hkuv.div(blockIdx.x);
        hk = blockIdx.x - tile * p.rows.Hkuv;
        z = blockIdx.y;
        row0 = tile * 128 + wave * 32;
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

// Forward.  LDS: K and U tiles of two blocks, V tile of one (80 KB for d_h > 64, so that two workgroups share a CU and one's
// element-wise code and barriers lie under the other's matrix instructions).
template <int CT>
__global__ __launch_bounds__(256, 2) void fwd_f32_kernel(F32Args p)
{
    using T = Tile<CT>;
    constexpr int FI = T::INS / 4 > 0 ? T::INS / 4 : 1;      // fill instructions per wave and tile
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Place w(p, wave, l32);
    const int DH = p.DH;

    auto fill = [&](const float* W, int blk, unsigned char* tile) {
        const Block b(p, w.hk, w.blk0 + (blk < w.nblk ? blk : w.nblk - 1));
#pragma unroll
        for (int k = 0; k < FI; ++k)
            T::fill(tile, wave * FI + k, lane, DH, [&](int r) { return W + (b.wrow + (r < b.rows ? r : b.rows - 1)) * DH; });
    };
    unsigned char* sV = lds + 4 * T::BYTES;
    fill(p.K, 0, lds);
    fill(p.U, 0, lds + T::BYTES);
    f32x4 q[4 * CT];
    load_row<CT>(q, p.Q + p.rows.tok(w.hk, w.row) * DH, g, DH);
    const float* rrow = p.R + p.rows.gate(w.hk, w.row) * p.parts.E;

    f32x16 o[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) o[ct] = zero16();
    for (int blk = 0; blk < w.nblk; ++blk) {
        const Block b(p, w.hk, w.blk0 + blk);
        const unsigned char *sK = lds + (blk & 1) * 2 * T::BYTES, *sU = sK + T::BYTES;
        const float r = rrow[b.e];
        wait_vmcnt<0>();      // K and U of this block have landed
        __syncthreads();      // ... for every wave, and every wave is done with the block before
        fill(p.V, blk, sV);
        fill(p.K, blk + 1, lds + (~blk & 1) * 2 * T::BYTES);
        fill(p.U, blk + 1, lds + (~blk & 1) * 2 * T::BYTES + T::BYTES);
        f32x16 mn[2];
        const typename T::Lane l(l32, g);
        first_products<CT, 2>(mn, {sK, sU}, {q, q}, l);
        f32x16 &m = mn[0], &n = mn[1];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            // (computed for the rows that a short block lacks too: hidden from the compiler, or it makes a branch of each element,
            // and fp32 matrix instructions leave no time under them: 1,024 rows of 8 heads of 128 224 us, now 216)
            float v = m[i] * sigmoid_exact(m[i]) * n[i] * r;
            asm volatile("" : "+v"(v));
            m[i] = reg_row(i, g) < b.rows ? v : 0.0f;
        }
        wait_vmcnt<2 * FI>();      // V has landed (the next block's K and U may be in flight)
        __syncthreads();
        second_product<CT>(o, sV, m, l);
    }
    wait_vmcnt<0>();
    if (w.valid)
        store_row<CT>(o, p.parts.nsplit > 1 ? p.part + (((long)w.z * p.rows.Hkuv + w.hk) * p.rows.n + w.row) * DH
                                            : p.O + p.rows.tok(w.hk, w.row) * DH, g, DH);
}

// dQ and dR.  LDS: K, U and V tiles of one block; the second workgroup of the CU covers the wait for the next.  (d_h > 96
// takes more than half the register file: one workgroup.)
template <int CT>
__global__ __launch_bounds__(256, CT > 3 ? 1 : 2) void dqdr_f32_kernel(F32Args p)
{
    using T = Tile<CT>;
    constexpr int FI = T::INS / 4 > 0 ? T::INS / 4 : 1;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Place w(p, wave, l32);
    const int DH = p.DH, E = p.parts.E;
    const unsigned char *sK = lds, *sU = lds + T::BYTES, *sV = lds + 2 * T::BYTES;

    const long tok = p.rows.tok(w.hk, w.row) * DH;
    f32x4 q[4 * CT], go[4 * CT];
    load_row<CT>(q, p.Q + tok, g, DH);
    load_row<CT>(go, p.dO + tok, g, DH);
    const float* rrow = p.R + p.rows.gate(w.hk, w.row) * E;
    const long hrows = (long)p.rows.Hkuv * p.rows.n;
    float* drow = p.parts.nsplit > 1 ? p.part + p.parts.nsplit * hrows * DH + (w.z * hrows + (long)w.hk * p.rows.n + w.row) * E
                                     : p.dR + p.rows.gate(w.hk, w.row) * E;

    f32x16 dq[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) dq[ct] = zero16();
    float dr = 0.0f;
    for (int blk = 0; blk < w.nblk; ++blk) {
        const Block b(p, w.hk, w.blk0 + blk);
        const float r = rrow[b.e];
        __syncthreads();      // every wave is done with the block before
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));      // (the fills' addresses are not worth a register each)
#pragma unroll
        for (int k = 0; k < FI; ++k) {
            auto row = [&](const float* W) {
                return [&, W](int rr) { return W + (b.wrow + (rr < b.rows ? rr : b.rows - 1)) * DH; };
            };
            T::fill(lds, wave * FI + k, lane, DH, row(p.K));
            T::fill(lds + T::BYTES, wave * FI + k, lane, DH, row(p.U));
            T::fill(lds + 2 * T::BYTES, wave * FI + k, lane, DH, row(p.V));
        }
        wait_vmcnt<0>();
        __syncthreads();
        f32x16 mna[3];
        const typename T::Lane l(l32, g);
        first_products<CT, 3>(mna, {sK, sU, sV}, {q, q, go}, l);
        f32x16 &m = mna[0], &n = mna[1], &da = mna[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float sg = sigmoid_exact(m[i]), sl = m[i] * sg;
            const float a = reg_row(i, g) < b.rows ? da[i] : 0.0f;
            dr = fmaf(a * sl, n[i], dr);
            m[i] = r * a * n[i] * (sg + sl * (1.0f - sg));      // dM
            n[i] = r * a * sl;                                  // dN
        }
        second_product<CT>(dq, sK, m, l);
        second_product<CT>(dq, sU, n, l);
        if (blk + 1 == w.nblk || Block(p, w.hk, w.blk0 + blk + 1).e != b.e) {
            const float tot = dr + __shfl_xor(dr, 32);      // the two lane halves hold different rows j of the same token
            if (g == 0 && w.valid) drow[b.e] = tot;
            dr = 0.0f;
        }
    }
    if (w.valid)
        store_row<CT>(dq, p.parts.nsplit > 1 ? p.part + (((long)w.z * p.rows.Hkuv + w.hk) * p.rows.n + w.row) * DH : p.dQ + tok, g, DH);
}

// dK, dU, dV.  A wave owns one block of weight rows (B operands and accumulators stay in registers) and every other
// 32-row tile of its slice of the head's rows: waves 0, 1 take the even tiles of two blocks, waves 2, 3 the odd ones, and their
// sums meet in LDS at the end.  (Halving the tiles inside the workgroup doubles the workgroups of a layer whose blocks are
// few, without partial sums in memory; LDS is idle, so that each pair of waves has tiles of its own costs nothing.)
template <int CT>
__global__ __launch_bounds__(256, 1) void dkdudv_f32_kernel(F32Args p)
{
    using T = Tile<CT>;
    constexpr int FI = T::INS / 2 > 0 ? T::INS / 2 : 1;
    constexpr int STAGE_B = 2 * T::BYTES;      // Q and dO tile
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    float* sR = reinterpret_cast<float*>(lds + 4 * STAGE_B);      // [stage][wave][32] gate values
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = wave >> 1, bw = wave & 1;
    const int hk = blockIdx.y, z = blockIdx.z, E = p.parts.E, nblk = E * p.parts.nbe;
    const int blk = blockIdx.x * 2 + bw;
    const Block b(p, hk, blk < nblk ? blk : nblk - 1);

    f32x16 dk[CT], du[CT], dv[CT];
    {
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
    // The odd tiles' sums to the wave with the even ones, one gradient at a time (64 lanes x 16 CT floats, lane-private).
    // (This lane's row and the bounds of its columns are worked out again, out of the compiler's sight: kept over the loop they
    // are the few registers too many that made it spill for d_h > 96.)
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
    if (half == 1 || blk >= nblk || l32 >= b.rows) return;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            dk[ct][i] += xch[(ct * 16 + i) * 64];
            du[ct][i] += xch[((CT + ct) * 16 + i) * 64];
            dv[ct][i] += xch[((2 * CT + ct) * 16 + i) * 64];
        }
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

// Adds the parts' sums in order: the rows of O or dQ (dst, four columns per lane) and, for blockIdx.x >= row_blocks, the
// values of dR over the parts that hold blocks of the expert.
__global__ __launch_bounds__(256) void sum_f32_kernel(F32Args p, float* dst, unsigned row_blocks)
{
    const int hk = blockIdx.y, DH = p.DH, E = p.parts.E;
    const long hrows = (long)p.rows.Hkuv * p.rows.n;
    if (blockIdx.x < row_blocks) {
        const unsigned i = blockIdx.x * 256 + threadIdx.x, r = i / (unsigned)(DH / 4);
        const int c = (i - r * (DH / 4)) * 4;
        if (r >= (unsigned)p.rows.n) return;
        const float* src = p.part + ((long)hk * p.rows.n + r) * DH + c;
        auto load = [&](int z) { return *reinterpret_cast<const f32x4*>(src + z * hrows * DH); };
        *reinterpret_cast<f32x4*>(dst + p.rows.tok(hk, r) * DH + c) = sum_in_order(load(0), 1, p.parts.nsplit, load);
    } else {
        const unsigned i = (blockIdx.x - row_blocks) * 256 + threadIdx.x, r = i / (unsigned)E;
        const int e = i - r * E;
        if (r >= (unsigned)p.rows.n) return;
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

// Parts of the blocks for the forward and dQ/dR as for bfloat16 (pick_parts).
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

template <int CT>
hipError_t launch_fwd_f32_t(const F32Args& a, const Dims& d, hipStream_t st)
{
    const int smem = 5 * Tile<CT>::BYTES;
    static LdsOptIn optin;
    const hipError_t e = ensure_dynamic_lds(optin, (const void*)fwd_f32_kernel<CT>, smem);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(fwd_f32_kernel<CT>, dim3((unsigned)(((a.rows.n + 127) / 128) * d.Hkuv), (unsigned)a.parts.nsplit), dim3(256),
                       smem, st, a);
    if (a.parts.nsplit > 1) {
        const unsigned rb = (unsigned)(((long)a.rows.n * (d.d_h / 4) + 255) / 256);
        hipLaunchKernelGGL(sum_f32_kernel, dim3(rb, (unsigned)d.Hkuv), dim3(256), 0, st, a, a.O, rb);
    }
    return hipGetLastError();
}

template <int CT>
hipError_t launch_bwd_f32_t(F32Args a, const Dims& d, hipStream_t st, int phases)
{
    hipError_t err = hipSuccess;
    if (phases & PH_BWD_DQDR) {
        const int smem = 3 * Tile<CT>::BYTES;
        static LdsOptIn optin;
        err = ensure_dynamic_lds(optin, (const void*)dqdr_f32_kernel<CT>, smem);
        if (err != hipSuccess) return err;
        hipLaunchKernelGGL(dqdr_f32_kernel<CT>, dim3((unsigned)(((a.rows.n + 127) / 128) * d.Hkuv), (unsigned)a.parts.nsplit),
                           dim3(256), smem, st, a);
        if (a.parts.nsplit > 1) {
            const unsigned rb = (unsigned)(((long)a.rows.n * (d.d_h / 4) + 255) / 256);
            const unsigned eb = (unsigned)(((long)a.rows.n * d.E + 255) / 256);
            hipLaunchKernelGGL(sum_f32_kernel, dim3(rb + eb, (unsigned)d.Hkuv), dim3(256), 0, st, a, a.dQ, rb);
        }
        err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    if (phases & PH_BWD_DKDUDV) {
        const int smem = 8 * Tile<CT>::BYTES + 2 * 4 * 32 * (int)sizeof(float);
        static_assert(2 * 3 * CT * 16 * 64 * 4 <= 8 * Tile<CT>::BYTES, "the waves' exchange fits the tile stages");
        static LdsOptIn optin;
        err = ensure_dynamic_lds(optin, (const void*)dkdudv_f32_kernel<CT>, smem);
        if (err != hipSuccess) return err;
        dim3 grid((unsigned)((d.E * nbe_of(d) + 1) / 2), (unsigned)d.Hkuv, (unsigned)a.nslice);
        hipLaunchKernelGGL(dkdudv_f32_kernel<CT>, grid, dim3(256), smem, st, a);
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
