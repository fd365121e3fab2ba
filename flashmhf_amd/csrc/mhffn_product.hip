// The block's projections: C = A B over bfloat16 matrices, fp32 sums rounded once, in the three forms that a linear layer and
// its backward need.
//
//     NT   C[M,N] = A[M,K]   B[N,K]^T    x w^T       both operands have the summed index running fastest ("rows")
//     NN   C[M,N] = A[M,K]   B[K,N]      dy w        A rows, B the summed index slowest ("cols")
//     TN   C[M,N] = A[K,M]^T B[K,N]      dy^T x      both cols
//
// They stand beside the library's products, which are made for matrices large enough to fill the chip with tiles of 256: at one
// round of smaller tiles these are faster but for the exceptions at product_faster.  us per product in a captured graph of 20, library / here:
//     hidden 1024, tokens    64         512        1,024       2,048       4,096
//         NT             6.6 / 3.9   6.5 / 5.1   8.0 / 7.5  10.3 / 9.1  13.5 / 12.5
//         NN             8.7 / 6.8   8.0 / 6.9   9.3 / 7.2  11.2 / 8.8  14.3 / 12.7
//         TN             4.7 / 3.8   8.5 / 5.2  11.3 / 6.8  16.1 / 10.1 27.5 / 17.6
//     hidden 2048, 16 tokens: NT 5.3 / 4.8.
// About 3 us of each are the launch, the first loads and the last stores; the rest is the rate at which a compute unit's LDS is
// filled from L2 (65 to 80 GB/s in these kernels; 115 in a loop of nothing but fills), not the matrix pipe (a third busy).
//
// The tile kernels add the terms of an element in the order of the summed index, one accumulator from the first to the last (a tile
// whose k-steps two groups of waves shared took 6.3 instead of 6.9 us for 64 x 64 of K = 1,024, as long or longer in larger ones).
// The library's do, too, wherever it does not split the summed index: the same bits.  Only the split kernel (NT, few tiles) does not.
//
// LDS units are 32 rows of 128 bytes: 32 rows of C x 64 of the summed index (rows), or 32 of the summed index x 64 rows of C
// (cols), filled by global_load_lds_dwordx4, read by 16-byte row reads or transposing 8-byte reads.  Chunk c (16 bytes) of row r
// sits at c ^ prod_swz(r), which makes both kinds of read free of bank conflicts (16 consecutive rows at one chunk, and 4
// consecutive rows at 4 aligned chunks, each cover 256 bytes once).
#include "mhffn_common.hpp"
#include "mhffn_product.hpp"

#include <utility>

namespace mhffn {

constexpr int PROD_UNIT_B = 4096;
constexpr int FILLERS = 4;          // waves of a tile kernel's workgroup that do nothing but fill
__device__ __forceinline__ int prod_swz(int r) { return (((r >> 1) & 1) << 2) | ((r >> 2) & 3); }

struct ProductArgs {
    const bf16_t* A;
    const bf16_t* B;
    bf16_t* C;
    int M, N, K;
    int mtiles, ntiles;
};

// (what lanes of a fill read where the summed index or the columns end)
static __device__ __align__(16) const unsigned prod_zeros[4] = {0u, 0u, 0u, 0u};

// Workgroup i runs on XCD i % 8: each XCD takes a run of consecutive tiles, counted in columns four tiles of rows high, so that what
// it reads fits its L2.
__device__ __forceinline__ void prod_tile(const ProductArgs& p, unsigned block, int& mt, int& nt)
{
    const unsigned total = p.mtiles * p.ntiles, xcd = block & 7, q = total >> 3, rem = total & 7;
    const unsigned t = (block >> 3) + xcd * q + (xcd < rem ? xcd : rem);
    const unsigned band = t / (4u * p.ntiles), in = t - band * 4u * p.ntiles;
    const unsigned high = min(4u, p.mtiles - 4u * band);
    mt = 4 * band + in % high;
    nt = in / high;
}

// One operand's share of a stage: BR rows of C, KU units of 64 of the summed index, filled by WAVES waves: COUNT instructions each
// per stage, at a uniform base plus a lane offset that does not change from stage to stage.  Rows of C that are not there are
// the last one again (nothing stores what they give); where the summed index ends, zeros.
template <bool COLS, int BR, int KU, int WAVES>
struct ProductFill {
    static constexpr int COUNT = BR * KU / (8 * WAVES), REGION_B = BR * KU * 128;
    const unsigned char* base;     // wave-uniform
    unsigned off[COUNT];
    int lim[COUNT];                // the lane has something to read while stage * KU * 64 < lim
    long inc;
    __device__ __forceinline__ void init(const bf16_t* X, int row0, int rows, int K, int wave, int lane)
    {
        const long ld = COLS ? rows : K;
        base = reinterpret_cast<const unsigned char*>(X + (COLS ? row0 : row0 * ld));
        inc = 2 * (COLS ? KU * 64 * ld : KU * 64);
#pragma unroll
        for (int i = 0; i < COUNT; ++i) {
            const int id = wave * COUNT + i, unit = id >> 2, r = 8 * (id & 3) + (lane >> 3), c = (lane & 7) ^ prod_swz(r);
            if constexpr (COLS) {
                const int kr = unit / (BR / 64), cu = unit % (BR / 64);
                const int k = 32 * kr + r, col = 64 * cu + 8 * c;
                off[i] = 2 * (unsigned)(k * ld + col);
                lim[i] = row0 + col < rows ? K - k : 0;
            } else {
                const int ku = unit / (BR / 32), rg = unit % (BR / 32);
                const int k = 64 * ku + 8 * c, row = 32 * rg + r;
                off[i] = 2 * (unsigned)((row0 + row < rows ? row : rows - 1 - row0) * ld + k);
                lim[i] = K - k;
            }
        }
    }
    // CHECK: a stage that reaches beyond the end of the summed index or a tile that reaches beyond the last column
    template <int I, bool CHECK>
    __device__ __forceinline__ void issue(unsigned char* region, int k0, int wave) const
    {
        const unsigned char* p = base + off[I];
        if constexpr (CHECK) p = k0 < lim[I] ? p : reinterpret_cast<const unsigned char*>(prod_zeros);
        __builtin_amdgcn_global_load_lds((gptr_t)p, (lptr_t)(region + (wave * COUNT + I) * 1024), 16, 0, 0);
    }
    __device__ __forceinline__ void skip(int stages) { base += stages * inc; }
};

template <int IMM>
__device__ __forceinline__ TrOperand prod_read_cols(unsigned lo, unsigned hi)
{
    TrOperand t;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(t.lo) : "v"(lo), "n"(IMM));
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(t.hi) : "v"(hi), "n"(IMM));
    return t;
}

// One operand's reads of a wave: TR tiles of TH rows of C from tile t0 on, the steps of a stage: 16 of the summed index each for the
// 32-row instruction, 32 for the 16-row one.  (The reads are inline assembly and in flight only inside one basic block: nothing
// can copy their registers before they arrive.)
template <bool COLS, int BR, int KU, int TH, int TR>
struct ProductRead {
    static constexpr int STEPS = KU * (TH == 32 ? 4 : 2), ACROSS = (BR + 63) / 64;
    unsigned off[COLS ? 2 * TR : STEPS];
    struct Set {
        u32x4 row[COLS ? 1 : TR][COLS ? 1 : STEPS];
        TrOperand col[COLS ? TR : 1][COLS ? STEPS : 1];
    };
    __device__ __forceinline__ void init(int t0, int lane)
    {
        if constexpr (COLS) {
            const int lam = lane & 15;
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int hi = 0; hi < 2; ++hi) {
                    const int r = 8 * (lane / TH) + 4 * hi + (lam >> 2), col = (t0 + i) * TH + (lane % TH & 16);      // 16 columns from `col` on
                    const int chunk = ((col & 63) >> 3) + ((lam & 3) >> 1);
                    off[2 * i + hi] = (col >> 6) * PROD_UNIT_B + r * 128 + ((chunk ^ prod_swz(r)) << 4) + (lam & 1) * 8;
                }
        } else {
            const int r = t0 * TH + lane % TH;
#pragma unroll
            for (int j = 0; j < STEPS; ++j) {
                constexpr int PER = TH == 32 ? 4 : 2;      // steps of a unit
                const int chunk = 8 / PER * (j % PER) + lane / TH;
                off[j] = (j / PER * (BR / 32) + (r >> 5)) * PROD_UNIT_B + (r & 31) * 128 + ((chunk ^ prod_swz(r & 31)) << 4);
            }
        }
    }
    template <int J, int I>
    __device__ __forceinline__ void request(unsigned base, Set& s) const      // step J of tile I
    {
        if constexpr (COLS) {
            constexpr int IMM = TH == 32 ? (J >> 1) * ACROSS * PROD_UNIT_B + (J & 1) * 2048 : J * ACROSS * PROD_UNIT_B;
            s.col[I][J] = prod_read_cols<IMM>(base + off[2 * I], base + off[2 * I + 1]);
        } else {
            s.row[I][J] = lds_read16_async<I * (TH == 32 ? PROD_UNIT_B : 2048)>(base + off[J]);
        }
    }
    // behind a wait: no use of the operands above it
    static __device__ __forceinline__ void arrived(Set& s, int j)
    {
#pragma unroll
        for (int i = 0; i < TR; ++i) {
            if constexpr (COLS) asm volatile("" : "+v"(s.col[i][j].lo), "+v"(s.col[i][j].hi));
            else asm volatile("" : "+v"(s.row[i][j]));
        }
    }
    static __device__ __forceinline__ bf16x8 get(const Set& s, int i, int j)
    {
        if constexpr (COLS) return tr_value(s.col[i][j]);
        else return __builtin_bit_cast(bf16x8, s.row[i][j]);
    }
};
__device__ __forceinline__ f32x16 prod_mfma(bf16x8 a, bf16x8 b, f32x16 c) { return mfma32(a, b, c); }
__device__ __forceinline__ f32x4 prod_mfma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// BM x BN of C per workgroup.  Four waves fill a ring of NST stages of KU * 64 of the summed index.  Eight multiply, WM of them side by
// side along the rows of the tile, with instructions of TH x TH; four of them (one per SIMD) run half a stage behind the other
// four: one wave of a SIMD reads its operands while the other multiplies.
// The waves that multiply do not fill: a fill instruction holds its wave for 30 ns and more, and in the same wave it held up the
// products behind it (TN of 1,024 x 1,024 x 2,048: 11.1 us with every wave filling, 12.2 with the fills between the products, 9.5
// with waves of their own for them; all eight waves reading and then multiplying together were between these).
template <bool ACOLS, bool BCOLS, int BM, int BN, int TH, int WM, int KU, int NST>
__device__ __forceinline__ void product_tile_of(const ProductArgs& p, unsigned block)
{
    constexpr int TM = BM / WM / TH, TN = BN / (8 / WM) / TH;      // tiles of a wave
    using FA = ProductFill<ACOLS, BM, KU, FILLERS>;
    using FB = ProductFill<BCOLS, BN, KU, FILLERS>;
    constexpr int FILLS = FA::COUNT + FB::COUNT, STAGE_B = FA::REGION_B + FB::REGION_B;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int late = wave >> 2, wm = wave % WM, wn = wave / WM;

    int mt, nt;
    prod_tile(p, block, mt, nt);
    const int m0 = mt * BM, n0 = nt * BN;
    const int nst = (p.K + 64 * KU - 1) / (64 * KU);
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    // Barriers 2st + 1 and 2st + 2 of a stage, counted from the first as 0: the early waves read stage st before 2st + 1 and multiply
    // before 2st + 2, the late ones one barrier later; fillers refill the slot of stage st - 1 behind barrier 2st, when both have read it,
    // and have seen stage st + 1 land before barrier 2st + 2.
    if (wave >= 8) {
        const int pw = wave - 8;
        FA fa;
        FB fb;
        fa.init(p.A, m0, p.M, p.K, pw, lane);
        fb.init(p.B, n0, p.N, p.K, pw, lane);
        const bool inside = (!ACOLS || m0 + BM <= p.M) && (!BCOLS || n0 + BN <= p.N);
        auto issue = [&](int st, int slot) {
            unsigned char* s = smem + slot * STAGE_B;
            auto all = [&](auto check_) {
                constexpr bool CHECK = decltype(check_)::value;
                static_for<FA::COUNT>([&](auto ic) { fa.template issue<decltype(ic)::value, CHECK>(s, st * KU * 64, pw); });
                static_for<FB::COUNT>([&](auto ic) { fb.template issue<decltype(ic)::value, CHECK>(s + FA::REGION_B, st * KU * 64, pw); });
            };
            if (inside && (st + 1) * KU * 64 <= p.K) all(std::false_type{});
            else all(std::true_type{});
            fa.skip(1);
            fb.skip(1);
        };
        // this wave's fills of all stages up to `st` have landed, those of younger ones (up to NST - 2) may be in flight
        auto landed = [&](int st, int issued) {
            const int younger = issued - 1 - st;
            static_assert((NST - 2) * FILLS < 64, "the counter has six bits");
            static_for<NST - 1>([&](auto yc) {
                constexpr int y = decltype(yc)::value;
                if (younger == y) wait_vmcnt<y * FILLS>();
            });
        };
#pragma unroll
        for (int s = 0; s < NST - 1; ++s)
            if (s < nst) issue(s, s);
        landed(0, NST - 1 < nst ? NST - 1 : nst);
        barrier();
        int prev = NST - 1;
        for (int st = 0; st < nst; ++st) {
            if (st + NST - 1 < nst) issue(st + NST - 1, prev);
            barrier();
            if (st + 1 < nst) landed(st + 1, st + NST < nst ? st + NST : nst);
            barrier();
            prev = prev + 1 == NST ? 0 : prev + 1;
        }
        barrier();
        __syncthreads();
        __syncthreads();
        return;
    }
    using RA = ProductRead<ACOLS, BM, KU, TH, TM>;
    using RB = ProductRead<BCOLS, BN, KU, TH, TN>;
    using Acc = std::conditional_t<TH == 32, f32x16, f32x4>;
    constexpr int STEPS = RA::STEPS, QUADS = TH == 32 ? 4 : 1;
    Acc acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int x = 0; x < 4 * QUADS; ++x) acc[i][j][x] = 0.0f;
    RA ra;
    RB rb;
    ra.init(wm * TM, lane);
    rb.init(wn * TN, lane);
    const unsigned smem0 = lds_addr(smem);
    barrier();
    if (late) barrier();
    int slot = 0;
    for (int st = 0; st < nst; ++st) {
        const unsigned sa = smem0 + slot * STAGE_B, sb = sa + FA::REGION_B;
        typename RA::Set a;
        typename RB::Set b;
        static_for<STEPS>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            static_for<TM>([&](auto ic) { ra.template request<j, decltype(ic)::value>(sa, a); });
            static_for<TN>([&](auto ic) { rb.template request<j, decltype(ic)::value>(sb, b); });
        });
        __builtin_amdgcn_sched_barrier(0);
        lds_wait_n<0>();
        static_for<STEPS>([&](auto jc) {
            RA::arrived(a, decltype(jc)::value);
            RB::arrived(b, decltype(jc)::value);
        });
        barrier();
#pragma unroll
        for (int j = 0; j < STEPS; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int n = 0; n < TN; ++n) acc[i][n] = prod_mfma(RB::get(b, n, j), RA::get(a, i, j), acc[i][n]);   // (lanes: rows of C)
        barrier();
        slot = slot + 1 == NST ? 0 : slot + 1;
    }
    if (!late) barrier();
    __syncthreads();
    // the tile leaves as whole rows, by way of LDS: rows of BN * 2 bytes, 16-byte chunk c of row r at c ^ (r % 8)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int a = 0; a < QUADS; ++a) {
                bf16x4 v;
#pragma unroll
                for (int x = 0; x < 4; ++x) v[x] = (bf16_t)acc[i][n][4 * a + x];
                const int r = (wm * TM + i) * TH + lane % TH, col = (wn * TN + n) * TH + (TH == 32 ? 8 * a : 0) + 4 * (lane / TH);
                *reinterpret_cast<bf16x4*>(smem + r * (BN * 2) + (((col >> 3) ^ (r & 7)) << 4) + (col & 4) * 2) = v;
            }
    __syncthreads();
    constexpr int CH = BN / 8;
#pragma unroll
    for (int id = threadIdx.x; id < BM * CH; id += 512) {
        const int r = id / CH, c = id % CH;
        if (m0 + r < p.M && n0 + 8 * c < p.N)
            *reinterpret_cast<u32x4*>(p.C + (long)(m0 + r) * p.N + n0 + 8 * c) =
                *reinterpret_cast<const u32x4*>(smem + r * (BN * 2) + ((c ^ (r & 7)) << 4));
    }
}

template <bool ACOLS, bool BCOLS, int BM, int BN, int TH, int WM, int KU, int NST>
__global__ __launch_bounds__(512 + 64 * FILLERS) void mhffn_product_kernel(ProductArgs p)
{
    product_tile_of<ACOLS, BCOLS, BM, BN, TH, WM, KU, NST>(p, blockIdx.x);
}

// The tiles that every form has, by their place in PRODUCT_VARIANTS.
template <int V>
struct Tiles {
    static constexpr int BM = V ? 128 : 64, BN = V == 2 ? 128 : 64, TH = V ? 32 : 16, WM = 4, KU = V == 2 ? 1 : 2, NST = V == 1 ? 3 : 4;
    static constexpr int SMEM = (BM + BN) * KU * 128 * NST;      // (holds the tile of C, too)
    static_assert(BM * BN * 2 <= SMEM && SMEM <= 160 * 1024, "LDS of a compute unit");
};

// Both products of a linear layer's backward in one launch: dx = dy w (NN, tiles VN) in the workgroups from nn0 on, dw = dy^T x (TN,
// tiles VT) in those from tn0 on.  Each alone leaves compute units idle, most of them with few tokens, and the second waits for a
// launch; us for both, two launches / one, in a graph of ten:
//     hidden 768, 512 tokens 11.0 / 6.6, 2,048 17.5 / 11.3; hidden 1024, 64 tokens 10.3 / 7.3, 512 12.0 / 7.8, 1,024 13.6 / 9.1, 2,048 19.7 / 15.8,
//     4,096 30.2 / 27.8; 512 of 1024 -> 3072 23.1 / 15.1; hidden 2048, 512 20.0 / 15.5, 2,048 42.4 / 41.5.
template <int VN, int VT>
__global__ __launch_bounds__(512 + 64 * FILLERS) void mhffn_product_pair_kernel(ProductArgs nn, unsigned nn0, ProductArgs tn, unsigned tn0)
{
    using N = Tiles<VN>;
    using T = Tiles<VT>;
    if (blockIdx.x - nn0 < (unsigned)(nn.mtiles * nn.ntiles)) product_tile_of<false, true, N::BM, N::BN, N::TH, N::WM, N::KU, N::NST>(nn, blockIdx.x - nn0);
    else product_tile_of<true, true, T::BM, T::BN, T::TH, T::WM, T::KU, T::NST>(tn, blockIdx.x - tn0);
}

// NT with few tiles: 32 TM x 32 TN of C per workgroup.  Its eight waves take every eighth chunk of 64 of the summed index each, through
// LDS of their own (Q chunks in flight, no barrier before the end), and their sums are added at the end, in the waves' order.
// (512 x 1,024 x 1,024: 5.1 us with 64 x 32 against 6.0 with 32 x 64 above; 64 x 64 this way 6.7.)
template <int TM, int TN, int Q>
__global__ __launch_bounds__(512) void mhffn_product_split_kernel(ProductArgs p)
{
    constexpr int BM = 32 * TM, BN = 32 * TN;
    using FA = ProductFill<false, BM, 1, 1>;
    using FB = ProductFill<false, BN, 1, 1>;
    using RA = ProductRead<false, BM, 1, 32, TM>;
    using RB = ProductRead<false, BN, 1, 32, TN>;
    constexpr int FILLS = FA::COUNT + FB::COUNT, CHUNK_B = FA::REGION_B + FB::REGION_B;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int mt, nt;
    prod_tile(p, blockIdx.x, mt, nt);
    const int m0 = mt * BM, n0 = nt * BN;
    unsigned char* own = smem + wave * Q * CHUNK_B;
    FA fa;
    FB fb;
    fa.init(p.A, m0, p.M, p.K, 0, lane);
    fb.init(p.B, n0, p.N, p.K, 0, lane);
    fa.skip(wave);
    fb.skip(wave);
    const int chunks = (p.K + 63) / 64;
    auto fill = [&](int ch, int buf) {
        unsigned char* s = own + buf * CHUNK_B;
        auto all = [&](auto check_) {
            constexpr bool CHECK = decltype(check_)::value;
            static_for<FA::COUNT>([&](auto ic) { fa.template issue<decltype(ic)::value, CHECK>(s, 64 * ch, 0); });
            static_for<FB::COUNT>([&](auto ic) { fb.template issue<decltype(ic)::value, CHECK>(s + FA::REGION_B, 64 * ch, 0); });
        };
        if (64 * ch + 64 <= p.K) all(std::false_type{});
        else all(std::true_type{});
        fa.skip(8);
        fb.skip(8);
    };
#pragma unroll
    for (int q = 0; q < Q; ++q)
        if (wave + 8 * q < chunks) fill(wave + 8 * q, q);
    RA ra;
    RB rb;
    ra.init(0, lane);
    rb.init(0, lane);
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int x = 0; x < 16; ++x) acc[i][j][x] = 0.0f;
    int buf = 0;
    for (int ch = wave; ch < chunks; ch += 8) {
        if (Q > 1 && ch + 8 < chunks) wait_vmcnt<(Q - 1) * FILLS>();
        else wait_vmcnt<0>();
        static_assert(Q <= 2, "the wait above");
        __builtin_amdgcn_sched_barrier(0);
        const unsigned t = lds_addr(own) + buf * CHUNK_B;
        typename RA::Set a;
        typename RB::Set b;
        static_for<4>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            static_for<TM>([&](auto ic) { ra.template request<j, decltype(ic)::value>(t, a); });
            static_for<TN>([&](auto ic) { rb.template request<j, decltype(ic)::value>(t + FA::REGION_B, b); });
        });
        lds_wait_n<0>();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            RA::arrived(a, j);
            RB::arrived(b, j);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (ch + 8 * Q < chunks) fill(ch + 8 * Q, buf);      // (this wave alone reads what it fills)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int n = 0; n < TN; ++n) acc[i][n] = mfma32(RB::get(b, n, j), RA::get(a, i, j), acc[i][n]);   // (lanes: rows of C)
        buf = buf + 1 == Q ? 0 : buf + 1;
    }
    __syncthreads();
    f32x4* sums = reinterpret_cast<f32x4*>(smem);
    constexpr int QUADS = TM * TN * 4;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                f32x4 v;
#pragma unroll
                for (int x = 0; x < 4; ++x) v[x] = acc[i][n][4 * q + x];
                sums[(wave * QUADS + (i * TN + n) * 4 + q) * 64 + lane] = v;
            }
    __syncthreads();
    for (int k = wave; k < QUADS; k += 8) {
        f32x4 s = sums[k * 64 + lane];
#pragma unroll
        for (int v = 1; v < 8; ++v) s += sums[(v * QUADS + k) * 64 + lane];
        bf16x4 o;
#pragma unroll
        for (int x = 0; x < 4; ++x) o[x] = (bf16_t)s[x];
        const int m = m0 + 32 * (k / (4 * TN)) + l32, n = n0 + 32 * (k / 4 % TN) + 8 * (k % 4) + 4 * g;
        if (m < p.M && n < p.N) *reinterpret_cast<bf16x4*>(p.C + (long)m * p.N + n) = o;
    }
}

template <bool ACOLS, bool BCOLS, int BM, int BN, int TH, int WM, int KU, int NST>
static hipError_t launch_tiles(ProductArgs a, hipStream_t st)
{
    constexpr int smem = (BM + BN) * KU * 128 * NST;
    static_assert(BM * BN * 2 <= smem && smem <= 160 * 1024, "LDS of a compute unit");
    static LdsOptIn optin;
    auto* fn = mhffn_product_kernel<ACOLS, BCOLS, BM, BN, TH, WM, KU, NST>;
    const hipError_t e = ensure_dynamic_lds(optin, (const void*)fn, smem);
    if (e != hipSuccess) return e;
    a.mtiles = (a.M + BM - 1) / BM;
    a.ntiles = (a.N + BN - 1) / BN;
    hipLaunchKernelGGL(fn, dim3((unsigned)a.mtiles * a.ntiles), dim3(512 + 64 * FILLERS), smem, st, a);
    return hipGetLastError();
}
template <int TM, int TN, int Q>
static hipError_t launch_split(ProductArgs a, hipStream_t st)
{
    constexpr int smem = 8 * PROD_UNIT_B * (TM + TN) * Q;      // (holds the sums, 8 * TM * TN units, too)
    static_assert(TM * TN <= (TM + TN) * Q && smem <= 160 * 1024, "LDS of a compute unit");
    static LdsOptIn optin;
    auto* fn = mhffn_product_split_kernel<TM, TN, Q>;
    const hipError_t e = ensure_dynamic_lds(optin, (const void*)fn, smem);
    if (e != hipSuccess) return e;
    a.mtiles = (a.M + 32 * TM - 1) / (32 * TM);
    a.ntiles = (a.N + 32 * TN - 1) / (32 * TN);
    hipLaunchKernelGGL(fn, dim3((unsigned)a.mtiles * a.ntiles), dim3(512), smem, st, a);
    return hipGetLastError();
}

// Time of a launch in us: base + rounds of CUS workgroups x (stages of 64 of the summed index x step, slower by up to `full` as the
// chip fills) + again for every round after the first.  Fitted to the three forms at hidden 768, 1024 and 2048 with 16 to 8,192
// tokens; the pick is the fastest or within 0.4 us of it at each of these where one round suffices.
struct ProductVariant {
    int bm, bn;
    double base, step, full, again;
};
constexpr ProductVariant PRODUCT_VARIANTS[] = {{64, 64, 3.2, 0.23, 0.0, 2.8}, {128, 64, 3.4, 0.285, 0.12, 2.9}, {128, 128, 3.6, 0.4, 0.3, 1.0},
                                               {32, 64, 2.8, 0.18, 0.1, 1.6},                                       // NT in order
                                               {32, 32, 2.4, 0.08, 0.2, 1.3}, {64, 32, 3.0, 0.115, 0.1, 1.6}};      // NT in any order
constexpr int FIRST_SPLIT = 4;
static long product_tiles(const ProductVariant& p, int M, int N) { return (long)((M + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn); }
static int product_variant(int form, bool in_order, int M, int N, int K)
{
    int best = 0;
    double best_us = 0;
    for (int v = 0; v < (form != PRODUCT_NT ? 3 : in_order ? 4 : 6); ++v) {
        const ProductVariant& p = PRODUCT_VARIANTS[v];
        const long tiles = product_tiles(p, M, N), rounds = (tiles + CUS - 1) / CUS;
        const double load = tiles <= CUS / 2 ? 0 : tiles >= CUS ? 1 : (tiles - CUS / 2) / (double)(CUS / 2);
        const double us = p.base + (rounds - 1) * p.again + rounds * ((K + 63) / 64) * p.step * (1 + p.full * load);
        if (best_us == 0 || us < best_us) { best_us = us; best = v; }
    }
    return best;
}
int product_tile(int form, bool in_order, int M, int N, int K)
{
    const ProductVariant& p = PRODUCT_VARIANTS[product_variant(form, in_order, M, N, K)];
    return 65536 * p.bm + p.bn;
}
// Time of a pair's launch in tiles vn and vt, by the same prices: n + t workgroups, those that take longer first, each to the compute unit
// that is free first.  Over 35 pairs (hidden 512 to 2048, 1 to 8,192 tokens) the fastest by this is the fastest of the nine measured or
// 2.4 % slower, 0.2 % on average; the tiles that each product alone would take are up to 49 % slower (both then run to a second
// round, which larger tiles do without: 1,024 tokens of hidden 768 11.4 us, in 128 x 64 and 64 x 64 7.7).
static double product_pair_us(int vn, int vt, int M, int N, int K, bool& nn_first)
{
    const ProductVariant &pn = PRODUCT_VARIANTS[vn], &pt = PRODUCT_VARIANTS[vt];
    long n = product_tiles(pn, M, K), t = product_tiles(pt, N, K);
    const long all = n + t;
    const double load = all <= CUS / 2 ? 0 : all >= CUS ? 1 : (all - CUS / 2) / (double)(CUS / 2);
    double dn = pn.again + (N + 63) / 64 * pn.step * (1 + pn.full * load), dt = pt.again + (M + 63) / 64 * pt.step * (1 + pt.full * load);
    nn_first = dn >= dt;
    const double launch = pn.base - pn.again > pt.base - pt.again ? pn.base - pn.again : pt.base - pt.again;
    if (all > 16 * CUS) return launch + (n * dn + t * dt) / CUS;
    if (!nn_first) {
        std::swap(n, t);
        std::swap(dn, dt);
    }
    // compute units with n / CUS of the longer ones and with one more; the shorter ones to whichever is free first
    const long more = n % CUS, less = CUS - more;
    double a = (double)(n / CUS) * dn, b = a + dn, end = more ? b : a;
    while (t > 0) {
        double& free = a <= b || !more ? a : b;
        t -= &free == &a ? less : more;
        free += dt;
        if (free > end) end = free;
    }
    return launch + end;
}

// One round of the largest tiles: there these kernels are as fast as the library's or faster (NT of 3,000 x 1,024 x 1,024 11.3 us
// against 11.7, of 2,048^3 20.3 against 20.4; TN of the latter 21.2 against 25.3); with more its larger tiles win in NT and NN
// (8,192 x 1,024 x 1,024: 25 against 22).
bool product_preferred(int M, int N) { return (long)((M + 127) / 128) * ((N + 127) / 128) <= CUS; }

// ... but for what the form and the length of the sum add to that.  us here / library, in a graph of ten:
//   TN  faster at every length of the sum: hidden 1024 with 2,048 tokens 10.9 / 16.8, 16,384 59.6 / 101.6, 32,768 128 / 198; hidden 2048
//       23 / 28, 151 / 168 and 292 / 292; 1,024 x 3,072 of 16,384 tokens 127 / 148.
//   NN  for few rows the library splits the sum, and here it is one wave's chain: 8 rows of hidden 320 5.0 / 5.8, 384 5.0 / 4.6, 768
//       6.4 / 5.2, 2048 11.0 / 7.0; 24 rows of hidden 1024 7.3 / 8.2, 1280 8.2 / 6.0, 2048 11.0 / 7.6; 64 rows of hidden 2048 11.0 / 13.1.
//   NT  a long sum in the tile kernels takes longer than in the library's deeper tiles: 733 rows of hidden 2048 14.4 / 13.5, but 1,024 rows
//       15.4 / 16.5; of 2560 19.2 / 18.1 and 22.4 / 21.9; of 4096 33.6 / 28.9 and 38.0 / 35.7.  One round of the split kernel is faster
//       at any length: 64 rows of hidden 4096 9.2 / 12.5.
bool product_faster(int form, bool in_order, int M, int N, int K)
{
    if (!product_preferred(M, N)) return false;
    if (form == PRODUCT_NN) return M > 16 ? K <= 1024 || M >= 64 : K < 384;
    if (form == PRODUCT_NT && K > 2048) {
        const int v = product_variant(form, in_order, M, N, K);
        return v >= FIRST_SPLIT && product_tiles(PRODUCT_VARIANTS[v], M, N) <= CUS;
    }
    return true;
}

// Both products of a backward in one launch: wherever each is taken here, and where dw is two rounds of the largest tiles, which the
// library's product beats, but not by the launch and the idle compute units that the pair saves (two launches with the library's dw /
// one: 512 rows of 1024 -> 8192 48.8 / 34.5, 2,048 84.8 / 79.6; of 768 -> 8192 48.0 / 33.3, 77.0 / 66.7, 4,096 127.2 / 115.6).  Where dx
// leaves few of them idle, or the sums of dw are long, it does (4,096 rows of 1024 -> 8192 142.4 / 147.9, of 1024 -> 5632 111.6 / 119.0; 2,048 of
// 2048 -> 3072 64.0 / 66.1; 5,400 of 512 -> 16384 214 / 230).
bool product_pair_faster(bool in_order, int M, int N, int K)
{
    if (!product_faster(PRODUCT_NN, in_order, M, K, N)) return false;
    if (product_faster(PRODUCT_TN, in_order, N, K, M)) return true;
    return product_tiles(PRODUCT_VARIANTS[2], N, K) <= 2 * CUS && product_tiles(PRODUCT_VARIANTS[2], M, K) <= 3 * CUS / 4 && M <= 4096;
}

template <bool ACOLS, bool BCOLS>
static hipError_t launch_form(const ProductArgs& a, int variant, hipStream_t st)
{
    auto tiles = [&](auto t) {
        using T = decltype(t);
        return launch_tiles<ACOLS, BCOLS, T::BM, T::BN, T::TH, T::WM, T::KU, T::NST>(a, st);
    };
    switch (variant) {
        case 0: return tiles(Tiles<0>{});
        case 1: return tiles(Tiles<1>{});
        case 2: return tiles(Tiles<2>{});
    }
    if constexpr (!ACOLS && !BCOLS) switch (variant) {
        case 3: return launch_tiles<ACOLS, BCOLS, 32, 64, 16, 2, 2, 4>(a, st);
        case 4: return launch_split<1, 1, 2>(a, st);
        case 5: return launch_split<2, 1, 1>(a, st);
    }
    return hipErrorInvalidValue;
}

template <int VN, int VT>
static hipError_t launch_pair_of(ProductArgs nn, ProductArgs tn, bool nn_first, hipStream_t st)
{
    constexpr int smem = Tiles<VN>::SMEM > Tiles<VT>::SMEM ? Tiles<VN>::SMEM : Tiles<VT>::SMEM;
    static LdsOptIn optin;
    auto* fn = mhffn_product_pair_kernel<VN, VT>;
    const hipError_t e = ensure_dynamic_lds(optin, (const void*)fn, smem);
    if (e != hipSuccess) return e;
    nn.mtiles = (nn.M + Tiles<VN>::BM - 1) / Tiles<VN>::BM;
    nn.ntiles = (nn.N + Tiles<VN>::BN - 1) / Tiles<VN>::BN;
    tn.mtiles = (tn.M + Tiles<VT>::BM - 1) / Tiles<VT>::BM;
    tn.ntiles = (tn.N + Tiles<VT>::BN - 1) / Tiles<VT>::BN;
    const unsigned n = nn.mtiles * nn.ntiles, t = tn.mtiles * tn.ntiles;
    hipLaunchKernelGGL(fn, dim3(n + t), dim3(512 + 64 * FILLERS), smem, st, nn, nn_first ? 0u : t, tn, nn_first ? n : 0u);
    return hipGetLastError();
}
hipError_t launch_product_pair(const void* dy, const void* w, const void* x, void* dx, void* dw, int M, int N, int K, hipStream_t st)
{
    const ProductArgs nn{(const bf16_t*)dy, (const bf16_t*)w, (bf16_t*)dx, M, K, N, 0, 0};
    const ProductArgs tn{(const bf16_t*)dy, (const bf16_t*)x, (bf16_t*)dw, N, K, M, 0, 0};
    using Launch = hipError_t (*)(ProductArgs, ProductArgs, bool, hipStream_t);
    static constexpr Launch of[3][3] = {{launch_pair_of<0, 0>, launch_pair_of<0, 1>, launch_pair_of<0, 2>},
                                        {launch_pair_of<1, 0>, launch_pair_of<1, 1>, launch_pair_of<1, 2>},
                                        {launch_pair_of<2, 0>, launch_pair_of<2, 1>, launch_pair_of<2, 2>}};
    int best = 0;
    double best_us = 0;
    bool best_first = true;
    for (int v = 0; v < 9; ++v) {
        bool first;
        const double us = product_pair_us(v / 3, v % 3, M, N, K, first);
        if (v == 0 || us < best_us) { best = v; best_us = us; best_first = first; }
    }
    return of[best / 3][best % 3](nn, tn, best_first, st);
}

hipError_t launch_product(int form, bool in_order, const void* A, const void* B, void* C, int M, int N, int K, hipStream_t st)
{
    const ProductArgs a{(const bf16_t*)A, (const bf16_t*)B, (bf16_t*)C, M, N, K, 0, 0};
    const int v = product_variant(form, in_order, M, N, K);
    switch (form) {
        case PRODUCT_NT: return launch_form<false, false>(a, v, st);
        case PRODUCT_NN: return launch_form<false, true>(a, v, st);
        case PRODUCT_TN: return launch_form<true, true>(a, v, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace mhffn
