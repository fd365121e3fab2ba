// Fused multi-head FFN backward for gfx950 (bf16 MFMA, fp32 accumulation), two kernels:
//
//  (1) dQ/dR kernel -- a workgroup of 8 waves (two per SIMD) owns 256 rows of one K/U/V head (tokens of any batch and
//      q-head of its group: RowMap), 32 per wave, and all the head's blocks or one part of them (pick_parts); it
//      streams the K, U, V blocks (32 rows at a time) through a ring of LDS stages with LDS-direct loads.  Per block:
//          M^T = K Q^T, N^T = U Q^T, dA^T = V dO^T            (recomputed, registers only)
//          dR_e += sum_j dA * silu(M) * N                      (fp32, before any rounding)
//          dN^T = r_e dA^T silu(M^T),  dM^T = r_e dA^T N^T silu'(M^T)      (rounded once to bf16)
//          dQ^T += K^T dM^T + U^T dN^T                         (K^T, U^T: transposing reads of the same K, U tiles)
//      The two waves of a SIMD work half a block apart (one's element-wise phase under the other's matrix phases),
//      the later one at a higher wave priority.
//      Formulas: kernels/triton/flash_mlp_moe.py:401-414, :527-542.
//
//  (2) dK/dU/dV kernel -- a wave owns one 32-row block of K/U/V (held in registers as MFMA B operands) and loops
//      over token tiles of 32 staged in LDS by its workgroup; dK^T, dU^T, dV^T (d_h x 32, fp32) stay in registers
//      for the whole token loop.  Products are written [t, j] here (M = Q K^T) so that the recomputed tile is the
//      B operand of the token contraction; the A operands Q^T / dO^T come from the natural LDS tiles through
//      ds_read_b64_tr_b16.  Token slices (grid.z) write fp32 partials that a small epilogue sums and converts.
//      Formulas: kernels/triton/flash_mlp_moe.py:683-729.
#include "mhffn_common.hpp"

namespace mhffn {

// ------------------------------------------------------------------------------------------------ dQ / dR
struct DqArgs {
    const bf16_t* Q;
    const bf16_t* dO;
    const bf16_t* K;
    const bf16_t* U;
    const bf16_t* V;
    const float* R;
    bf16_t* dQ;
    float* dR;
    float* part;          // [nsplit][Hkuv][rows.n][DH] dQ, then [nsplit][Hkuv][rows.n][E] dR: fp32 partial sums
    RowMap rows;          // rows of Q, dO, dQ, R, dR that meet one K/U/V head
    Parts parts;          // ... and the blocks of that head
    int tile_rows;
};

constexpr int DQ_NST = 4;                  // LDS stages (K | U | V tiles each)
constexpr int DQ_STAGE_B = 3 * TILE_B;

template <int DH>
__global__ __launch_bounds__(512) void mhffn_bwd_dqdr_kernel(DqArgs p)
{
    constexpr int KS = DH / 16, CT = DH / 32, NW = 8;
    constexpr int BT = NW * 32;
    constexpr int FILL = 24 / NW;          // tile-fill wave-instructions per wave and block (3 tiles x 8 / NW waves)
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    float* sR = reinterpret_cast<float*>(smem + DQ_NST * DQ_STAGE_B);   // [min(E, 64)][BT]: expert e in slot e % 64

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // blockIdx.x = tile * Hkuv + kv-head: the head index runs fastest, so each head's weights stay in one XCD's L2
    arguments_first(p);
    const int tile = p.rows.by_hkuv.div(blockIdx.x), hk = blockIdx.x - tile * p.rows.Hkuv, z = blockIdx.y;
    if (tile * BT >= p.rows.n) return;                       // (whole_xcds)
    const int tok0 = tile * BT + wave * 32;                  // this wave's rows of the list (RowMap)
    const int nbe = p.parts.nbe, E = p.parts.E, nsplit = p.parts.nsplit;
    const int blk0 = p.parts.first(z), nblk = p.parts.first(z + 1) - blk0;   // blocks of this workgroup, counted from blk0
    const int ex0 = p.parts.by_nbe.div(blk0), jb0 = blk0 - ex0 * nbe;        // expert of the first, its place in the expert
    const int nex = p.parts.by_nbe.div(jb0 + nblk + nbe - 1);                // experts they belong to, counted from ex0
    const bf16_t* Kh = p.K + ((long)hk * E * nbe + blk0) * JB * DH;
    const long offU = p.U - p.K, offV = p.V - p.K;

    auto issue_block = [&](int blk) {
        const int bc = blk < nblk ? blk : nblk - 1;
        unsigned char* st = smem + (blk % DQ_NST) * DQ_STAGE_B;
        const long roff = (long)bc * JB * DH;
#pragma unroll
        for (int k = 0; k < FILL; ++k) {
            const int id = wave + NW * k;            // 0..23: tile id/8 (K, U, V), 4-row group id%8
            const int which = id >> 3;
            const long toff = which == 0 ? 0 : (which == 1 ? offU : offV);
            tile_fill_ins<DH>(Kh + toff + roff, DH, st + which * TILE_B, id & 7, lane);
        }
    };
    const int first = tok0 < p.rows.n ? tok0 : p.rows.n - 1;
    const RowMap::Run run = p.rows.run(hk, first, 32);
    // The Q and dO rows come from HBM and are the longest wait of the prologue: request them before anything else.
    bf16x8 q[KS], go[KS];
    {
        int t = tok0 + l32;
        t = t < p.rows.n ? t : p.rows.n - 1;
        const long row = p.rows.tok(run, hk, first, t) * DH + 8 * g;
        const bf16_t* qr = p.Q + row;
        const bf16_t* gr = p.dO + row;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            q[ks] = *reinterpret_cast<const bf16x8*>(qr + ks * 16);
            go[ks] = *reinterpret_cast<const bf16x8*>(gr + ks * 16);
        }
    }
    issue_block(0);
    // Gate values of the workgroup's 256 tokens, expert-major [E][BT]: asynchronous 4-byte LDS-direct loads, lane = token;
    // a pair of waves shares a group of 64 tokens and takes the even and the odd experts.  LDS holds 64 experts, expert e
    // in slot e % 64; the first 64 are issued between block 0 and block 1, so that the first wait for block 0 covers
    // them too, and a layer with more experts refills the slots 32 at a time as the block loop leaves them behind.
    const float* rrow;
    {
        int t = tile * BT + (wave >> 1) * 64 + lane;
        t = t < p.rows.n ? t : p.rows.n - 1;
        rrow = p.R + p.rows.gate(hk, t) * E + ex0;
    }
    auto stage_gates = [&](int e0, int e1) {
        e1 = e1 < nex ? e1 : nex;
        for (int e = e0 + (wave & 1); e < e1; e += 2)
            __builtin_amdgcn_global_load_lds((gptr_t)(rrow + e), (lptr_t)(sR + (e & 63) * BT + (wave >> 1) * 64), 4, 0, 0);
    };
    stage_gates(0, 64);
    issue_block(1);

    f32x16 dq[CT];
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int x = 0; x < 16; ++x) dq[i][x] = 0.0f;

    const int krow = row_perm32(l32);
    const TrLane<CT> trl = make_tr_lane<CT, 8, 4>(lane);
    // One block takes three phases per wave: first products (24 matrix instructions for d_h = 128), element-wise work
    // (VALU only), second products (16 matrix instructions).  The two waves that share a SIMD run them in opposite phase
    // between two barriers -- waves 0..3: first(b), element-wise(b), second(b); waves 4..7: element-wise(b-1),
    // second(b-1), first(b) -- so that one wave's VALU phase lies under the other's matrix phases.  Left to the
    // hardware's oldest-first arbitration the early waves win every conflict and then idle at the barrier while the late
    // waves catch up alone; the late waves therefore run at a higher wave priority, which evens the two out.  The late
    // waves carry M, N, dA of block b across the barrier and need one more trip at the end; the ring keeps block b-1
    // alive that long (the refill behind barrier b targets the stage of block b-2).
    f32x16 m, n, da;
    bf16x8 dmt[2], dnt[2];
    float dr = 0.0f;
    auto first_products = [&](int blk) {
        const unsigned char* sK = smem + (blk % DQ_NST) * DQ_STAGE_B;
        const unsigned char* sU = sK + TILE_B;
        const unsigned char* sV = sU + TILE_B;
#pragma unroll
        for (int x = 0; x < 16; ++x) { m[x] = 0.0f; n[x] = 0.0f; da[x] = 0.0f; }
        // The K/U/V operands come from LDS through a ring of three register sets, read two k-steps ahead of the
        // matrix instructions that use them; the fence after each k-step keeps the compiler from gathering the
        // reads back to the front (which costs their whole latency once per block).
        bf16x8 ak[3], au[3], av[3];
#pragma unroll
        for (int k0 = 0; k0 < 2; ++k0) {
            ak[k0] = tile_read_rows(sK, krow, k0, g);
            au[k0] = tile_read_rows(sU, krow, k0, g);
            av[k0] = tile_read_rows(sV, krow, k0, g);
        }
        static_for<KS>([&](auto kc) {
            constexpr int ks = decltype(kc)::value;
            if constexpr (ks + 2 < KS) {
                ak[(ks + 2) % 3] = tile_read_rows(sK, krow, ks + 2, g);
                au[(ks + 2) % 3] = tile_read_rows(sU, krow, ks + 2, g);
                av[(ks + 2) % 3] = tile_read_rows(sV, krow, ks + 2, g);
            }
            m = mfma32(ak[ks % 3], q[ks], m);
            n = mfma32(au[ks % 3], q[ks], n);
            da = mfma32(av[ks % 3], go[ks], da);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto element_wise = [&](float r) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
                const int i = 8 * s + kk;
                const float x = m[i], nn = n[i], a = da[i];
                const float sg = fast_sigmoid(x);
                const float sl = x * sg;                 // silu(m)
                const float as = a * sl;
                dr = __builtin_fmaf(as, nn, dr);
                const float w = __builtin_fmaf(sl, 1.0f - sg, sg);    // silu'(m)
                dnt[s][kk] = (bf16_t)(r * as);
                dmt[s][kk] = (bf16_t)((r * a) * (nn * w));
            }
    };
    // second products: operand pairs (Kt, Ut) are requested two steps ahead of the MFMAs that consume them; the region is
    // fenced so that the partial LDS waits count exactly these reads
    auto second_products = [&](int blk) {
        const unsigned sK = lds_addr(smem + (blk % DQ_NST) * DQ_STAGE_B);
        __builtin_amdgcn_sched_barrier(0);
        {
            constexpr int NSET = 2 * CT;          // (s, i) in s-major order
            TrOperand tk[3], tu[3];
            auto request = [&](auto ic) {
                constexpr int idx = decltype(ic)::value;
                constexpr int s = idx / CT, i = idx % CT;
                tk[idx % 3] = tile_read_cols_async<4096 * s>(sK, trl, i);
                tu[idx % 3] = tile_read_cols_async<4096 * s + TILE_B>(sK, trl, i);
            };
            request(std::integral_constant<int, 0>{});
            request(std::integral_constant<int, 1>{});
            static_for<NSET>([&](auto ic) {
                constexpr int idx = decltype(ic)::value;
                constexpr int s = idx / CT, i = idx % CT;
                if constexpr (idx + 2 < NSET) request(std::integral_constant<int, idx + 2>{});
                constexpr int ahead = (NSET - 1 - idx) < 2 ? (NSET - 1 - idx) : 2;
                lds_tr_wait_n<4 * ahead>(tk[idx % 3], tu[idx % 3]);
                dq[i] = mfma32(tr_value(tk[idx % 3]), dmt[s], dq[i]);
                dq[i] = mfma32(tr_value(tu[idx % 3]), dnt[s], dq[i]);
            });
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // where this lane's dR values go: the row of dR itself, or of this part's sums
    float* drow;
    {
        const int t = tok0 + l32 < p.rows.n ? tok0 + l32 : p.rows.n - 1;
        const long hrows = (long)p.rows.Hkuv * p.rows.n;
        drow = nsplit == 1 ? p.dR + p.rows.gate(run, hk, first, t) * E
                           : p.part + nsplit * hrows * DH + (z * hrows + (long)hk * p.rows.n + t) * E + ex0;
    }
    int e = 0, jb = jb0;        // expert and block-in-expert of the block whose element-wise work comes next
    auto finish_block = [&](int blk) {
        element_wise(sR[(e & 63) * BT + wave * 32 + l32]);
        second_products(blk);
        if (++jb == nbe || blk == nblk - 1) {
            // dR[t, e]: the two lane halves hold disjoint j rows of the same token column.
            const float tot = dr + __shfl_xor(dr, 32);
            if (g == 0 && tok0 + l32 < p.rows.n) drow[e] = tot;
            dr = 0.0f;
            jb = 0;
            ++e;
            // More than 64 experts: with expert 32k behind it (k >= 1), this pair of waves refills the slots of experts
            // 32k-32 .. 32k-1 with experts 32k+32 .. 32k+63 of its own 64 tokens.  Its partner is in the same interval
            // between two barriers, so at a block of expert 32k or later; the values are first read 31 experts on, and
            // every barrier's wait on the way leaves at most three of this wave's loads outstanding.
            if (e > 1 && (e & 31) == 1 && e + 31 < nex) stage_gates(e + 31, e + 63);
        }
    };
    // Barrier b: block b has landed for every wave, and every wave is done with block b - 2, whose stage the fill of
    // block b + 2 takes.
    auto next_interval = [&](int b) {
        wait_vmcnt<FILL>();       // block b has landed (block b+1 may be in flight)
        __syncthreads();
        issue_block(b + 2);
    };
    if (wave < NW / 2) {
        for (int b = 0; b < nblk; ++b) {
            next_interval(b);
            first_products(b);
            finish_block(b);
        }
        next_interval(nblk);      // the barrier of the late waves' extra trip
    } else {
        __builtin_amdgcn_s_setprio(2);
        next_interval(0);
        first_products(0);
        for (int b = 1; b < nblk; ++b) {
            next_interval(b);
            finish_block(b - 1);
            first_products(b);
        }
        next_interval(nblk);
        finish_block(nblk - 1);
        __builtin_amdgcn_s_setprio(0);
    }
    wait_vmcnt<0>();   // drain the phantom prefetches: they write the ring, which the epilogue reuses
    __syncthreads();   // every wave is done reading the ring

    if (nsplit > 1) {     // a part of the blocks leaves its sums as they are, fp32, for the pass that adds the parts
        store_rows_f32<DH>(smem + wave * TILE_B, p.part + (((long)z * p.rows.Hkuv + hk) * p.rows.n + tok0) * DH,
                           p.rows.n - tok0, lane, [&](auto ic) -> const f32x16& { return dq[decltype(ic)::value]; });
        return;
    }
    // dQ^T registers -> dQ[t][c] through a private 8 KB region of the ring per wave (rows of 256 bytes, 16-byte chunk c16
    // of row r at chunk c16 ^ (r & 15)), so that the stores are whole rows (16 lanes x 16 bytes, 4 rows per instruction)
    // instead of 8-byte pieces scattered over 32 rows.  Register 4a+x of row tile i is c = 32i + 8a + 4g + x.
    {
        unsigned char* otile = smem + wave * (32 * TILE_ROW_B);
#pragma unroll
        for (int i = 0; i < CT; ++i)
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                bf16x4 v;
#pragma unroll
                for (int x = 0; x < 4; ++x) v[x] = (bf16_t)dq[i][4 * a + x];
                *reinterpret_cast<bf16x4*>(otile + l32 * TILE_ROW_B + (((4 * i + a) ^ (l32 & 15)) << 4) + 8 * g) = v;
            }
        const int c16 = lane & 15;
        auto store = [&](auto&& address_row) {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int row = 4 * k + (lane >> 4);
                if (c16 < DH / 8 && tok0 + row < p.rows.n) {
                    const u32x4 v = *reinterpret_cast<const u32x4*>(otile + row * TILE_ROW_B + ((c16 ^ (row & 15)) << 4));
                    *reinterpret_cast<u32x4*>(p.dQ + address_row(row) * DH + c16 * 8) = v;
                }
            }
        };
        if (run.tok.stride) store([&](int row) { return run.tok.base + (long)row * run.tok.stride; });
        else store([&](int row) { return p.rows.tok(hk, tok0 + row); });
    }
}

// 32 rows, the blocks in a pipeline: the same products, element-wise formulas and order of sums as the kernel above.  Four waves
// take the first products and the element-wise work, each of every fourth block, in four phases of about equal length and a
// phase apart from each other; four more request the tiles, 24 KB a phase, and add one block a phase to dQ, a column tile
// each.  A SIMD has one wave of either kind.  (Four waves that did all of it for four blocks at a time, products, element-wise code,
// barrier, sums, barrier, took 0.60 us a block, most of it the chain of these; a phase takes 0.42 us at half a chip, 0.53 where
// every compute unit has a workgroup.  By s_memtime, of the 870 cycles of a phase a wave works 560 to 720, and none of the four
// phases and neither kind of wave stands out; without the fills 0.41.  First products in one phase: 0.56.  512 rows of the
// 370M heads in one part 78.9 -> 52.5 us, of 8 heads of 96 40.1 -> 27.7, of 64 37.5 -> 28.3.)
// What a phase reads was there before the barrier in front of it wherever it can be: V's and the transposed K and U operands are
// requested a phase ahead.  dR is one running sum over the elements of an expert's blocks, which the wave of a block hands to the
// wave of the next through LDS.  Loads go out three phases ahead of their block.
constexpr int DQ32_A = 4, DQ32_W = DQ32_A + 4;        // waves of the first kind, and all; also a block's phases up to its sums
constexpr int DQ32_AHEAD = 7 - DQ32_A;                 // phases between the request of a block's tiles and its first products
constexpr int DQ32_KU = 7, DQ32_V = DQ32_AHEAD + 1;    // tile sets: a block's K and U from the request to its sums, V to its first products
constexpr int DQ32_V0 = DQ32_KU * 2 * TILE_B, DQ32_D0 = DQ32_V0 + DQ32_V * TILE_B, DQ32_E0 = DQ32_D0 + 2 * 4096, DQ32_SMEM = DQ32_E0 + 256;
template <int DH>
__global__ __launch_bounds__(DQ32_W * 64) void mhffn_bwd_dqdr_rows32_kernel(DqArgs p)
{
    constexpr int KS = DH / 16, CT = DH / 32;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    arguments_first(p);
    const int tile = p.rows.by_hkuv.div(blockIdx.x), hk = blockIdx.x - tile * p.rows.Hkuv, z = blockIdx.y;
    const int tok0 = tile * 32, nbe = p.parts.nbe, E = p.parts.E, nsplit = p.parts.nsplit;
    if (tok0 >= p.rows.n) return;                            // (whole_xcds)
    const int blk0 = p.parts.first(z), nblk = p.parts.first(z + 1) - blk0;
    const int ex0 = p.parts.by_nbe.div(blk0), jb0 = blk0 - ex0 * nbe;
    const bf16_t* Kh = p.K + ((long)hk * E * nbe + blk0) * JB * DH;
    const unsigned smem0 = lds_addr(smem);
    const int nphase = nblk + DQ32_A;      // block b: first products in phase b, its sums in phase b + DQ32_A; every phase ends with a barrier

    if (wave < DQ32_A) {
        const int t = tok0 + l32 < p.rows.n ? tok0 + l32 : p.rows.n - 1;
        const long grow = p.rows.gate(hk, t) * E;
        bf16x8 q[KS], go[KS];
        {
            const long row = p.rows.tok(hk, t) * DH + 8 * g;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                q[ks] = *reinterpret_cast<const bf16x8*>(p.Q + row + ks * 16);
                go[ks] = *reinterpret_cast<const bf16x8*>(p.dO + row + ks * 16);
            }
        }
        const float* rrow = p.R + grow + ex0;
        const long hrows = (long)p.rows.Hkuv * p.rows.n;
        float* drow = nsplit == 1 ? p.dR + grow : p.part + nsplit * hrows * DH + (z * hrows + (long)hk * p.rows.n + t) * E + ex0;
        auto gate = [&](int b) { return rrow[p.parts.by_nbe.div(jb0 + (b < nblk ? b : nblk - 1))]; };
        float r = 0.0f, rnext = gate(wave);
        // (these loads end here: waited for in the loop, each trip would also wait for the next gate value)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(q[ks]), "+v"(go[ks]));
        asm volatile("" : "+v"(rnext));
        const int krow = row_perm32(l32), sw = swz16(krow);
        unsigned at[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) at[ks] = smem0 + krow * TILE_ROW_B + (((2 * ks + g) ^ sw) << 4);
        const unsigned sD = smem0 + DQ32_D0 + lane * 16, sE = smem0 + DQ32_E0 + lane * 4;

        f32x16 m, n, da, sg;
        f32x16 as;                // as, n: the factors of dR's terms
        bf16x8 dmt[2], dnt[2];
        QuadRows<KS, 2> a;
        QuadRows<KS, 1> av;
        // Phase 1: K1 k-steps of M and N, with the reads of the others and of V between the matrix instructions.
        constexpr int K1 = KS / 2, FIRST = KS - K1;
        auto phase1 = [&](int b) {
            r = rnext;
            rnext = gate(b + DQ32_A);      // a round ahead of its use
            const unsigned ku = (b % DQ32_KU) * 2 * TILE_B, v = DQ32_V0 + (b % DQ32_V) * TILE_B;
            auto request = [&](auto kc) {
                constexpr int ks = decltype(kc)::value;
                const unsigned x = at[ks] + ku;
                a.template request<0, ks>(x);
                a.template request<1, ks, TILE_B>(x);
            };
            __builtin_amdgcn_sched_barrier(0);
            static_for<FIRST>([&](auto kc) { request(kc); });
#pragma unroll
            for (int x = 0; x < 16; ++x) { m[x] = 0.0f; n[x] = 0.0f; }
            // behind k-step ks: the reads of k-step FIRST + ks and as many of V as leaves none for the last one
            constexpr int VN = (KS + K1 - 1) / K1;
            static_for<K1>([&](auto kc) {
                constexpr int ks = decltype(kc)::value;
                constexpr int kus = (FIRST + ks < KS ? FIRST + ks : KS) - (ks + 1), vs = ks * VN < KS ? ks * VN : KS;
                lds_wait_n<(2 * kus + vs < 15 ? 2 * kus + vs : 15)>();
                asm volatile("" : "+v"(a.v[0][ks]), "+v"(a.v[1][ks]));
                m = mfma32(a.get(0, ks), q[ks], m);
                n = mfma32(a.get(1, ks), q[ks], n);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (FIRST + ks < KS) request(std::integral_constant<int, FIRST + ks>{});
                static_for<VN>([&](auto vc) {
                    constexpr int k = ks * VN + decltype(vc)::value;
                    if constexpr (k < KS) av.template request<0, k>(at[k] + v);
                });
                __builtin_amdgcn_sched_barrier(0);
            });
            static_assert(FIRST + K1 >= KS, "every k-step's operands are requested in phase 1");
        };
        // Phase 2: the other k-steps, then dA with the sigmoids of the first elements under its matrix instructions.
        constexpr int SIG = 6;
        auto phase2 = [&]() {
            static_for<KS - K1>([&](auto kc) {
                constexpr int ks = K1 + decltype(kc)::value;
                asm volatile("" : "+v"(a.v[0][ks]), "+v"(a.v[1][ks]));       // (returned before the barrier, as V's)
                m = mfma32(a.get(0, ks), q[ks], m);
                n = mfma32(a.get(1, ks), q[ks], n);
            });
#pragma unroll
            for (int x = 0; x < 16; ++x) da[x] = 0.0f;
            __builtin_amdgcn_sched_barrier(0);
            static_for<KS>([&](auto kc) {
                constexpr int ks = decltype(kc)::value;
                asm volatile("" : "+v"(av.v[0][ks]));
                da = mfma32(av.get(0, ks), go[ks], da);
#pragma unroll
                for (int i = ks * SIG / KS; i < (ks + 1) * SIG / KS; ++i) sg[i] = fast_sigmoid(m[i]);
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        auto elements = [&](auto i0_, auto i1_) {
            constexpr int i0 = decltype(i0_)::value, i1 = decltype(i1_)::value;
#pragma unroll
            for (int i = i0 < SIG ? SIG : i0; i < i1; ++i) sg[i] = fast_sigmoid(m[i]);
#pragma unroll
            for (int i = i0; i < i1; ++i) {
                const float x = m[i], nn = n[i], a = da[i];
                const float sl = x * sg[i];              // silu(m)
                as[i] = a * sl;
                const float w = __builtin_fmaf(sl, 1.0f - sg[i], sg[i]);    // silu'(m)
                dnt[i >> 3][i & 7] = (bf16_t)(r * as[i]);
                dmt[i >> 3][i & 7] = (bf16_t)((r * a) * (nn * w));
            }
        };
        // The running sum of dR goes from block to block through LDS: the block before has left it a phase ago.
        auto gate_gradient = [&](int b, const u32x2& in) {
            const int j = jb0 + b, e = p.parts.by_nbe.div(j), jb = j - e * nbe;
            const unsigned bits = in[0];
            float dr = jb == 0 || b == 0 ? 0.0f : __builtin_bit_cast(float, bits);
#pragma unroll
            for (int i = 0; i < 16; ++i) dr = __builtin_fmaf(as[i], n[i], dr);
            lds_write4(sE, dr);
            if (jb == nbe - 1 || b == nblk - 1) {
                const float tot = dr + __shfl_xor(dr, 32);      // the lane halves hold disjoint j rows of one token column
                if (g == 0 && tok0 + l32 < p.rows.n) drow[e] = tot;
            }
        };
        using I0 = std::integral_constant<int, 0>;
        using I12 = std::integral_constant<int, 12>;
        using I16 = std::integral_constant<int, 16>;
        for (int i = 0; i <= wave; ++i) quad_barrier();      // (the first: block 0 has landed)
        int phase = wave;
        for (int b = wave; b < nblk; b += DQ32_A, phase += DQ32_A) {
            phase1(b);
            quad_barrier();
            phase2();
            quad_barrier();
            elements(I0{}, I12{});
            asm volatile("" : "+v"(dmt[0]), "+v"(dnt[0]), "+v"(dmt[1]), "+v"(dnt[1]), "+v"(as));     // (here, not behind the barrier)
            const unsigned d = sD + (b & 1) * 4096;
            quad_barrier();
            u32x2 in = lds_read_apart_async<1>(sE);
            lds_write16<0>(d, dmt[0]);
            lds_write16<2048>(d, dnt[0]);
            elements(I12{}, I16{});
            lds_write16<1024>(d, dmt[1]);
            lds_write16<3072>(d, dnt[1]);
            asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(in));
            gate_gradient(b, in);
            quad_barrier();
        }
        for (; phase <= nphase; ++phase) quad_barrier();     // (and the one in front of the epilogue)
        return;
    }

    // Fills and sums.  Each of these waves requests a quarter of every tile: six vmcnt events a block.
    const int col = wave - DQ32_A;
    QuadFill<DH, DQ32_KU, DQ32_V> fill(Kh, p.U - p.K, p.V - p.K, nblk, smem, smem + DQ32_V0, col, lane);
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    const TrLane<1> tr = quad_tr_lane<CT>(lane, col);
    f32x16 dq;
#pragma unroll
    for (int x = 0; x < 16; ++x) dq[x] = 0.0f;
    for (int b = 0; b < DQ32_AHEAD; ++b) {
        fill.aim(b);
        static_for<3>([&](auto t) {
            fill.request(t, I0{});
            fill.request(t, I1{});
        });
    }
    wait_vmcnt<6 * (DQ32_AHEAD - 1)>();
    quad_barrier();                           // block 0 has landed
    TrOperand tk[2], tu[2];
    auto phase_of = [&](auto sums_, int phase) {
        constexpr bool SUMS = decltype(sums_)::value;
        __builtin_amdgcn_sched_barrier(0);
        u32x4 d[4];                           // dM s 0, 1, dN s 0, 1
        if constexpr (SUMS) {
            const unsigned sD = smem0 + DQ32_D0 + ((phase - DQ32_A) & 1) * 4096 + lane * 16;
            d[0] = lds_read16_async<0>(sD);
            d[2] = lds_read16_async<2048>(sD);
            d[1] = lds_read16_async<1024>(sD);
            d[3] = lds_read16_async<3072>(sD);
        }
        fill.aim(phase + DQ32_AHEAD);
        fill.request(I0{}, I0{});
        fill.request(I0{}, I1{});
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SUMS) {
            lds_wait_n<0>();
            asm volatile("" : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]));
        }
        // this block's sums, each operand followed by the next block's (from the tile set that the next phase requests into)
        const unsigned aK = smem0 + fill.ku * 2 * TILE_B;
        static_for<4>([&](auto kc) {
            constexpr int k = decltype(kc)::value, half = k >> 1;
            TrOperand& t = k & 1 ? tu[half] : tk[half];
            if constexpr (SUMS) dq = mfma32(tr_value(t), __builtin_bit_cast(bf16x8, d[(k & 1) * 2 + half]), dq);
            __builtin_amdgcn_sched_barrier(0);
            t = tile_read_cols_async<(k & 1) * TILE_B + half * 4096>(aK, tr, 0);
            fill.request(std::integral_constant<int, (k + 2) / 2>{}, std::integral_constant<int, (k & 1)>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        wait_vmcnt<6 * (DQ32_AHEAD - 1)>();   // the next phase's first products have their tiles
        quad_barrier();
#pragma unroll
        for (int s = 0; s < 2; ++s) asm volatile("" : "+v"(tk[s].lo), "+v"(tk[s].hi), "+v"(tu[s].lo), "+v"(tu[s].hi));
    };
    int phase = 0;
    for (const int idle = col < CT ? DQ32_A : nphase; phase < idle; ++phase) phase_of(std::false_type{}, phase);
    for (; phase < nphase; ++phase) phase_of(std::true_type{}, phase);
    wait_vmcnt<0>();          // the fills of blocks that are not there write the tiles, which the epilogue reuses
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (col >= CT) return;
    unsigned char* own = smem + col * TILE_B;
    const int nrows = p.rows.n - tok0;
    if (nsplit > 1) {
        float* prow = p.part + (((long)z * p.rows.Hkuv + hk) * p.rows.n + tok0) * DH + 32 * col;
        quad_store_f32(own, dq, nrows, lane, [&](int row) { return prow + row * DH; });
    } else {
        quad_store_bf16(own, dq, nrows, lane, [&](int row) { return p.dQ + p.rows.tok(hk, tok0 + row) * DH + 32 * col; });
    }
}

// Adds the parts' sums of dQ (in the order of the parts) and rounds once, four columns per lane; adds the sums of dR over the
// parts that hold blocks of the expert, one value per lane.  Workgroup `block` of tile x, counted with the heads as the kernel that left the
// parts did: below dq_blocks dQ, otherwise dR.
template <int DH>
__device__ __forceinline__ void dqdr_sum(const DqArgs& p, unsigned x, unsigned block, unsigned dq_blocks)
{
    const int tile = p.rows.by_hkuv.div(x), hk = x - tile * p.rows.Hkuv;
    const long hrows = (long)p.rows.Hkuv * p.rows.n;
    if (block < dq_blocks) {
        const unsigned i = block * 256 + threadIdx.x;
        const unsigned r = tile * p.tile_rows + i / (DH / 4), c = (i % (DH / 4)) * 4;
        if (r >= (unsigned)p.rows.n) return;
        const float* src = p.part + ((long)hk * p.rows.n + r) * DH + c;
        auto load = [&](int z) { return *reinterpret_cast<const f32x4*>(src + z * hrows * DH); };
        const f32x4 sum = sum_in_order(load(0), 1, p.parts.nsplit, load);
        bf16x4 v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = (bf16_t)sum[x];
        *reinterpret_cast<bf16x4*>(p.dQ + p.rows.tok(hk, r) * DH + c) = v;
    } else {
        const unsigned i = (block - dq_blocks) * 256 + threadIdx.x;
        const int E = p.parts.E;
        const unsigned row = i / (unsigned)E, r = tile * p.tile_rows + row;
        const int e = i - row * E;
        if (row >= (unsigned)p.tile_rows || r >= (unsigned)p.rows.n) return;
        const float* src = p.part + p.parts.nsplit * hrows * DH + ((long)hk * p.rows.n + r) * E + e;
        p.dR[p.rows.gate(hk, r) * E + e] =
            sum_in_order(0.0f, p.parts.part_lo(e), p.parts.part_hi(e), [&](int z) { return src[z * hrows * E]; });
    }
}
template <int DH>
__global__ __launch_bounds__(256) void mhffn_bwd_dqdr_sum_kernel(DqArgs p, unsigned dq_blocks)
{
    dqdr_sum<DH>(p, blockIdx.x, blockIdx.y, dq_blocks);
}

// ------------------------------------------------------------------------------------------------ dK / dU / dV
struct DwArgs {
    const bf16_t* Q;
    const bf16_t* dO;
    const bf16_t* K;
    const bf16_t* U;
    const bf16_t* V;
    const float* R;
    float* part;        // [nslice][3][Hkuv][E*d_e][DH] fp32 partial sums (nslice > 1)
    void* out[3];       // dK, dU, dV: written directly when there is one token slice
    int out_f32;        // element type of out: 1 = float32, 0 = bfloat16
    int B, H, G, S, E, nbe, nslice;
    int tokmaj;         // Q, dO token-major ([B, S, H, d_h]) instead of [B, H, S, d_h]
};

constexpr int DW_NST = 4;                              // LDS stages of the token-tile ring
constexpr int DW_RTILE_B = 1024;                       // staged gate values: [4 waves][64 lanes] fp32 (each wave: its expert)
constexpr int DW_STAGE_B = 2 * TILE_B + DW_RTILE_B;    // Q tile | dO tile | gate values
constexpr int DW_PAIR_STAGE_B = 2 * TILE_B + DW_RTILE_B / 2;

// With TokenHalves (PAIR): two blocks of rows a workgroup, and two waves for each of them: waves 0 and 1 take the first half of the slice's tokens, waves
// 2 and 3 the second, through a ring of their own, and a block's sums meet in LDS at the end.  Twice the workgroups with half the
// token tiles each, where the other form leaves compute units idle or takes twice the slices, every one of which is a set of float32
// sums in memory.  (Four waves on one block would need four rings, 264 KB.)
struct TokenHalves {};
template <int DH, bool TAIL, class... Mode>
__global__ __launch_bounds__(256) void mhffn_bwd_dkdudv_kernel(DwArgs p)
{
    constexpr bool PAIR = sizeof...(Mode) > 0;
    constexpr int KS = DH / 16, CT = DH / 32;
    constexpr int NCHUNK = DH / 8;                    // 16-byte chunks per token row
    constexpr int NB = PAIR ? 2 : 4;                  // blocks of the workgroup; waves of a ring
    constexpr int STAGE_B = PAIR ? DW_PAIR_STAGE_B : DW_STAGE_B, RING_B = DW_NST * STAGE_B;
    constexpr int FILLS = 8 / NB;                     // a wave's fill instructions per tile
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hk = blockIdx.x, z = blockIdx.z;   // head index fastest: all columns of a head run on one XCD and share its L2
    const int nblk = p.E * p.nbe;
    const int half = PAIR ? wave >> 1 : 0, wv = PAIR ? wave & 1 : wave;      // which ring, and which block of the workgroup
    unsigned char* ring = smem_raw + half * RING_B;
    const int jblk = blockIdx.y * NB + wv;
    const bool active = jblk < nblk;
    const int jb_c = active ? jblk : nblk - 1;        // waves of the last column without a block: addresses stay valid
    const int e_w = jb_c / p.nbe;
    const long wrow = ((long)hk * nblk + jb_c) * JB + l32;      // this lane's row of K/U/V (column j of the products)

    float* sZero = reinterpret_cast<float*>(smem_raw + (PAIR ? 2 : 1) * RING_B);   // 32 zero gate values
    if (tid < 32) sZero[tid] = 0.0f;
    // The first step contracts a tile that does not exist (zero gate values) out of the last stage, which no load has
    // filled yet: clear its Q and dO tiles, or whatever bit patterns the previous kernel left there (possibly NaN or
    // Inf as bf16) would be multiplied by those zeros.
    {
        u32x4 z = {0u, 0u, 0u, 0u};
        u32x4* last_stage = reinterpret_cast<u32x4*>(ring + (DW_NST - 1) * STAGE_B);
        for (int i = tid & (64 * NB - 1); i < 2 * TILE_B / 16; i += 64 * NB) last_stage[i] = z;
    }
    // These clears are ordinary LDS stores that other waves read in step 0, and the barriers of the token loop are bare
    // (no wait on this wave's own LDS stores): one fenced barrier here publishes them, once per workgroup.
    __syncthreads();
    const int nS = (p.S + 31) / 32;
    const int ntile = p.G * p.B * nS;
    int t_begin = (int)((long)ntile * z / p.nslice), t_end = (int)((long)ntile * (z + 1) / p.nslice);
    bool one_less = false;                            // the other waves have a tile, and a barrier, more
    if constexpr (PAIR) {                             // (the launcher gives every slice two tiles or more)
        const int mid = t_begin + (t_end - t_begin + 1) / 2;
        one_less = half && t_end - mid < mid - t_begin;
        if (half) t_begin = mid;
        else t_end = mid;
    }
    const int nt = t_end - t_begin;

    // Tile cursor of the prefetcher: tile index -> (q-head of the group, batch, 32-token tile).  It is kept as a running
    // token-row index that advances by one of three precomputed strides (next tile of the sequence, next
    // batch, next q-head of the group), so a step spends a handful of scalar instructions on it.
    int pf_st = t_begin % nS, pf_bb = (t_begin / nS) % p.B;
    int pf_left = nt;                                 // tiles not yet requested
    // (token rows are counted in 32 bits: B * H * S < 2^31 is checked on the host)
    const int pf_h0 = hk * p.G + t_begin / (nS * p.B);                        // q-head of the first tile
    int pf_row = (pf_bb * p.H + pf_h0) * p.S + pf_st * 32;                     // row of R ([B, H, S, E])
    const int drow_s = p.H * p.S - (nS - 1) * 32;                              // last tile of a sequence -> next batch
    const int drow_b = p.S - (p.B - 1) * p.H * p.S - (nS - 1) * 32;            // ... of the last batch -> next q-head
    // The same walk in rows of Q/dO, whose token stride is qs rows (1, or H when token-major).
    const int qs = p.tokmaj ? p.H : 1;
    int pf_qrow = p.tokmaj ? (pf_bb * p.S + pf_st * 32) * p.H + pf_h0 : pf_row;
    const int dqrow_s = p.H * p.S - (nS - 1) * 32 * qs;
    const int dqrow_b = (p.tokmaj ? 1 : p.S) - (p.B - 1) * p.H * p.S - (nS - 1) * 32 * qs;

    // per-lane constants of the tile fill: this wave's two 4-row groups of the Q/dO tiles (swizzled source chunk); of the four of PAIR
    // the first two, the others being 16 rows on, where the swizzle comes round
    int fill_row[2], fill_coff[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int ins = wv + NB * k;
        const int r = 4 * ins + (lane >> 4);
        int c = (lane & 15) ^ swz16(r);
        c = c < NCHUNK ? c : 0;                       // unused chunk positions of narrow rows load a dummy chunk
        fill_row[k] = r;
        fill_coff[k] = c * 16;                        // bytes
    }

    // Asynchronous fill of a stage with the tile under the cursor (the last tile again once all are requested); every wave
    // issues its share of LDS-direct loads (no staging registers).  Addresses are a wave-uniform 64-bit base plus a
    // 32-bit lane offset.  Rows past the end of a sequence are clamped to its last row and their gate value is zeroed
    // afterwards (zero_tail), which removes them from all three products.
    // The work is split: prepare_tile computes the uniform bases of the tile under the cursor and advances the cursor
    // (some forty scalar instructions; called under the last matrix instructions of a step, where the wave has issue
    // slots to spare), fire_tile issues the loads (right behind the barrier) and returns the tile's valid rows.
    const char* nx_qb = nullptr;
    const char* nx_gb = nullptr;
    const char* nx_rbp = nullptr;
    int nx_last = 31;
    auto prepare_tile = [&]() {
        nx_last = p.S - pf_st * 32 - 1;                                       // last valid row of the tile (>= 0)
        nx_qb = reinterpret_cast<const char*>(p.Q) + (long)pf_qrow * (DH * 2);
        nx_gb = reinterpret_cast<const char*>(p.dO) + (long)pf_qrow * (DH * 2);
        nx_rbp = reinterpret_cast<const char*>(p.R) + (long)pf_row * (p.E * 4);
        // advance unless this was the last tile of the slice (then later requests reload it, harmlessly)
        // (0/1 flags and multiplies: selects here were turned into branches inside the hot loop)
        const int more = pf_left > 1 ? 1 : 0;
        const int ws = (pf_st + 1 == nS ? 1 : 0) * more;
        const int wb = (pf_bb + 1 == p.B ? 1 : 0) * ws;
        pf_left -= more;
        pf_row += more * 32 + ws * (drow_s - 32) + wb * (drow_b - drow_s);
        pf_qrow += more * 32 * qs + ws * (dqrow_s - 32 * qs) + wb * (dqrow_b - dqrow_s);
        pf_st = (pf_st + more) * (1 - ws);
        pf_bb = (pf_bb + ws) * (1 - wb);
    };
    auto fire_tile = [&](int sidx) -> int {
        const int last = nx_last;
        unsigned char* sbase = ring + sidx * STAGE_B;
#pragma unroll
        for (int k = 0; k < FILLS; ++k) {
            const int on = 16 * (k >> 1), r = fill_row[k & 1] + (TAIL ? on : 0);
            const int row = TAIL ? (r < last ? r : last) : r;
            const unsigned off = (unsigned)(row * qs * (DH * 2) + fill_coff[k & 1]) + (TAIL ? 0u : (unsigned)(on * qs * (DH * 2)));
            const int ins = wv + NB * k;
            __builtin_amdgcn_global_load_lds((gptr_t)(nx_qb + off), (lptr_t)(sbase + ins * 1024), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((gptr_t)(nx_gb + off), (lptr_t)(sbase + TILE_B + ins * 1024), 16, 0, 0);
        }
        // gate values of this wave's expert for the 32 token rows (lanes 32..63 repeat them): one 4-byte element per lane
        const int trow = TAIL ? (l32 < last ? l32 : last) : l32;
        __builtin_amdgcn_global_load_lds((gptr_t)(nx_rbp + (unsigned)((trow * p.E + e_w) * 4)),
                                         (lptr_t)(sbase + 2 * TILE_B + wv * 256), 4, 0, 0);
        return last + 1;
    };
    // Called by every wave after its own loads of stage `sidx` have landed and before the barrier that publishes
    // the stage: zeroes the gate values of the rows a tail tile does not have.
    auto zero_tail = [&](int sidx, int nvalid) {
        float* sR = reinterpret_cast<float*>(ring + sidx * STAGE_B + 2 * TILE_B);
        if (l32 >= nvalid) sR[wv * 64 + lane] = 0.0f;
    };

    // First two tiles of the slice; the third is fired behind the first barrier of the loop.
    prepare_tile();
    int nv0 = fire_tile(0);
    prepare_tile();
    int nv1 = fire_tile(1), nv2 = 32, nv3 = 32;        // valid rows of the tile in each stage
    if constexpr (!TAIL) prepare_tile();

    if (!active) {
        // A wave of a head's last column that has no block: it keeps up its share of the tile fills and the barriers
        // (as many as the working waves pass, nt + 1) and issues no matrix instruction.
        for (int k = 0; k <= nt; ++k) {
            const int st = k & 3;
            wait_vmcnt<0>();
            if constexpr (TAIL) {
                const int nvalid = st == 0 ? nv0 : (st == 1 ? nv1 : (st == 2 ? nv2 : nv3));
                if (nvalid < 32) zero_tail(st, nvalid);
            }
            __builtin_amdgcn_s_barrier();
            if constexpr (TAIL) prepare_tile();
            const int nvn = fire_tile((st + 2) & 3);
            if constexpr (!TAIL) prepare_tile();
            if constexpr (TAIL) {
                if (st == 0) nv2 = nvn; else if (st == 1) nv3 = nvn; else if (st == 2) nv0 = nvn; else nv1 = nvn;
            }
        }
        wait_vmcnt<0>();
        if (PAIR && one_less) __builtin_amdgcn_s_barrier();
        __syncthreads();   // the barrier the working waves pass before their epilogue reuses the ring
        if constexpr (PAIR) __syncthreads();      // ... and the one between its halves
        return;
    }

    // The K, U and V blocks stay in registers as MFMA B operands for the whole kernel (K, U in accumulation registers).
    bf16x8 kB[KS], uB[KS];
    bf16x8 vR[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        kB[ks] = *reinterpret_cast<const bf16x8*>(p.K + wrow * DH + ks * 16 + 8 * g);
        uB[ks] = *reinterpret_cast<const bf16x8*>(p.U + wrow * DH + ks * 16 + 8 * g);
        vR[ks] = *reinterpret_cast<const bf16x8*>(p.V + wrow * DH + ks * 16 + 8 * g);
    }

    f32x16 dk[CT], du[CT], dv[CT];
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int x = 0; x < 16; ++x) { dk[i][x] = 0.0f; du[i][x] = 0.0f; dv[i][x] = 0.0f; }

    const int fr = swz16(l32);
    TrLane<CT> trl = make_tr_lane<CT, 4, 8>(lane);
    if constexpr (PAIR) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) { trl.off[ct][0] += half * RING_B; trl.off[ct][1] += half * RING_B; }
    }
    // LDS address of this lane's 16 bytes of k-step 0 in the Q tile of stage 0 (row l32, chunk g ^ swizzle); k-step ks is
    // this address ^ (ks << 5): the ring starts on a 1 KB boundary, so the exclusive-or commutes with the sum
    static_assert(RING_B % 1024 == 0, "the exclusive-or of qaddr");
    const unsigned qaddr = lds_addr(ring) + l32 * 256 + ((g ^ fr) << 4);
    const unsigned raddr = lds_addr(ring) + wv * 256;       // the wave's gate values, but for their place in a stage (wave-uniform)

    // B operands of the token contraction (P, dM, dN of one tile, bf16).  They live across steps: the element pairs 0 and 1
    // of a tile are converted under the last matrix instructions of the step that computed its first products, the other
    // six under the next step's first 36.  Zero for the tile that does not exist before the first one.
    bf16x8 pB[2], dmB[2], dnB[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) { pB[s][kk] = (bf16_t)0.0f; dmB[s][kk] = (bf16_t)0.0f; dnB[s][kk] = (bf16_t)0.0f; }

    // first products of the tile in stage ST -> (m, n, da) in architectural VGPRs, element-wise work of the PREVIOUS
    // tile (registers pm, pn, pda; gate values from stage SP) dealt out between the matrix instructions so that the VALU
    // works under them; then the token contraction of the previous tile, with the first element pairs of THIS tile's
    // element-wise work under its last matrix instructions.
    //   registers 4a+b of m/n/da: token 8a + 4g + b (rows), column j = l32.
    auto step = [&](auto st_c, auto sp_c, f32x16& m, f32x16& n, f32x16& da, const f32x16& pm, const f32x16& pn,
                    const f32x16& pda, bool live, int& nv_next) {
        constexpr int ST = decltype(st_c)::value, SP = decltype(sp_c)::value;
        const unsigned char* pQ = smem_raw + SP * STAGE_B;       // (trl holds the ring's place)
        // the previous tile's gate values, or zeros when there is no previous tile to contract (first step of a slice,
        // phantom steps that pad the loop): a zero gate makes P, dM and dN exactly zero
        const unsigned rp = live ? raddr + (SP * STAGE_B + 2 * TILE_B) : lds_addr(sZero);

        // LDS reads of the first products: the gate values of this tile's first four token rows (for the element pairs
        // converted at the end of this step) and of the previous tile for this lane's 16 token rows (4
        // consecutive rows per 16-byte read), then the operand ring (k-step ks + 2 is requested while ks is consumed).
        // All are issued from inline assembly and waited for by count; the element-wise slices in between are VALU only.
        __builtin_amdgcn_sched_barrier(0);
        u32x4 rvn = lds_read16_async<0>(raddr + (ST * STAGE_B + 2 * TILE_B) + 16 * g);
        u32x4 rvu[4];
        {
            const unsigned ra = rp + 16 * g;
            rvu[0] = lds_read16_async<0>(ra);
            rvu[1] = lds_read16_async<32>(ra);
            rvu[2] = lds_read16_async<64>(ra);
            rvu[3] = lds_read16_async<96>(ra);
        }
        u32x4 aq[3], ag[3];
        auto request = [&](auto kc) {
            constexpr int ks = decltype(kc)::value;
            const unsigned a = qaddr ^ (ks << 5);     // the stage goes into the instruction's immediate offset
            aq[ks % 3] = lds_read16_async<ST * STAGE_B>(a);
            ag[ks % 3] = lds_read16_async<ST * STAGE_B + TILE_B>(a);
        };
        request(std::integral_constant<int, 0>{});
        request(std::integral_constant<int, 1>{});
        // The fill of the stage that came free at the barrier (tile k + 2) is issued behind the first reads: its five
        // instructions (nine with TokenHalves) and their address arithmetic pass while those reads are on their way.
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (TAIL) prepare_tile();     // (the tail instantiation has no registers to spare for the early call)
        nv_next = fire_tile((ST + 2) % DW_NST);
        f32x4 rv[4];
        // Transposed operands of the token contraction (phases 2 and 3 below), in (s, ct) order.  They come from the
        // previous tile, so the first two sets are requested under the last two k-steps of the first products, in the
        // ring slots those no longer need, and have arrived when the contraction starts.
        constexpr int NSET = 2 * CT;
        TrOperand tq[3], tg[3];
        auto request_tr = [&](auto ic) {
            constexpr int idx = decltype(ic)::value;
            constexpr int s = idx / CT, ct = idx % CT;
            tq[idx % 3] = tile_read_cols_async<4096 * s>(lds_addr(pQ), trl, ct);
            tg[idx % 3] = tile_read_cols_async<4096 * s + TILE_B>(lds_addr(pQ), trl, ct);
        };

        // Element-wise work of the previous tile, two elements (register indices 2pr, 2pr+1 of pm/pn/pda) at a time so
        // that no instruction waits on the one just before it, in five slices of at most six VALU instructions; one slice
        // fits under one MFMA (32 cycles).  With sigma = 1/(1+2^(-m log2 e)), B = r sigma, A = m B (= r silu(m)):
        //     P = A n,   dN = A dA,   dM = (B + A (1 - sigma)) (n dA)         [silu'(m) = sigma + silu(m) (1 - sigma)]
        float ex[8][2], sg[8][2], nda[8][2], Av[8][2], Bv[8][2], s1[8][2];
        f32x4 rvn4;                                   // gate values of THIS tile's token rows 4g .. 4g+3 (elements 0..3)
        auto slice_on = [&](auto pc, auto kc, const f32x16& sm, const f32x16& sn, const f32x16& sda, auto gate) {
            constexpr int pr = decltype(pc)::value, k = decltype(kc)::value;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int i = 2 * pr + u;
                if constexpr (k == 0) {
                    ex[pr][u] = __builtin_amdgcn_exp2f(-LOG2E * sm[i]);
                } else if constexpr (k == 1) {
                    sg[pr][u] = __builtin_amdgcn_rcpf(1.0f + ex[pr][u]);
                    nda[pr][u] = sn[i] * sda[i];
                } else if constexpr (k == 2) {
                    Bv[pr][u] = gate(i) * sg[pr][u];
                    Av[pr][u] = sm[i] * Bv[pr][u];
                    s1[pr][u] = 1.0f - sg[pr][u];
                } else if constexpr (k == 3) {
                    pB[i >> 3][i & 7] = (bf16_t)(Av[pr][u] * sn[i]);
                    dnB[i >> 3][i & 7] = (bf16_t)(Av[pr][u] * sda[i]);
                } else {
                    dmB[i >> 3][i & 7] = (bf16_t)(__builtin_fmaf(Av[pr][u], s1[pr][u], Bv[pr][u]) * nda[pr][u]);
                }
            }
        };
        // The 40 slices of a tile (8 element pairs x 5) are spread over 48 consecutive matrix instructions for d_h = 128
        // (NSL in general): pairs 0 and 1 of THIS tile behind the last 3 CT of this step (the s = 1 half of the
        // contraction, which reads only the operand halves of elements 8..15), pairs 2..7 of the PREVIOUS tile behind
        // this step's first NSL - 3 CT.  Pairs 2 and 3 are done long before the s = 0 half starts, pairs 4..7 before the
        // s = 1 half.  Each matrix instruction so has about one slice behind it; two slices behind one cost the wave
        // more issue time than the instruction's 32 cycles, none leaves the matrix pipe's shadow unused.
        constexpr int NS1 = 3 * KS, NSL = NS1 + 6 * CT, NLATE = 3 * CT, NEARLY = NSL - NLATE;
        static_assert(9 * NEARLY / 30 < NS1, "pairs 2 and 3 must be converted before the s = 0 half of the contraction");
        auto ew_slot = [&](auto kc) {
            constexpr int k = decltype(kc)::value;
            if constexpr (k < NEARLY) {
                static_for<30>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    if constexpr (q * NEARLY / 30 == k)
                        slice_on(std::integral_constant<int, 2 + q / 5>{}, std::integral_constant<int, q % 5>{}, pm, pn, pda,
                                 [&](int i) { return rv[i >> 2][i & 3]; });
                });
            } else {
                static_for<10>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    if constexpr (NEARLY + q * NLATE / 10 == k)
                        slice_on(std::integral_constant<int, q / 5>{}, std::integral_constant<int, q % 5>{}, m, n, da,
                                 [&](int i) { return rvn4[i & 3]; });
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto after_slot1 = [&](auto kc) { ew_slot(kc); };

        static_for<KS>([&](auto kc) {
            constexpr int ks = decltype(kc)::value;
            if constexpr (ks + 2 < KS) request(std::integral_constant<int, ks + 2>{});
            if constexpr (ks == KS - 2) request_tr(std::integral_constant<int, 0>{});
            if constexpr (ks == KS - 1) request_tr(std::integral_constant<int, 1>{});
            // reads younger than this k-step's operands: two per later k-step of the ring, four per transposed set
            constexpr int younger = ks + 2 < KS ? 4 : (ks == KS - 2 ? 2 + 4 : 4 + 4);
            if constexpr (ks == 0) {
                lds_wait_n<younger>(aq[0], ag[0], rvu[0], rvu[1], rvu[2], rvu[3]);       // (the gate values are older)
#pragma unroll
                for (int a = 0; a < 4; ++a) rv[a] = __builtin_bit_cast(f32x4, rvu[a]);
                asm volatile("" : "+v"(rvn));     // (older than the reads just waited for; no use of it may move above)
                rvn4 = __builtin_bit_cast(f32x4, rvn);
            } else {
                lds_wait_n<younger>();        // (consumed by asm matrix instructions only)
            }
            const bf16x8 aqv = __builtin_bit_cast(bf16x8, aq[ks % 3]), agv = __builtin_bit_cast(bf16x8, ag[ks % 3]);
            if constexpr (ks == 0) mfma32_vgpr_first_bacc(m, aqv, kB[0]);
            else mfma32_vgpr_acc_bacc(m, aqv, kB[ks]);
            after_slot1(std::integral_constant<int, 3 * ks>{});
            if constexpr (ks == 0) mfma32_vgpr_first_bacc(n, aqv, uB[0]);
            else mfma32_vgpr_acc_bacc(n, aqv, uB[ks]);
            after_slot1(std::integral_constant<int, 3 * ks + 1>{});
            if constexpr (ks == 0) mfma32_vgpr_first(da, agv, vR[0]);
            else mfma32_vgpr_acc(da, agv, vR[ks]);
            after_slot1(std::integral_constant<int, 3 * ks + 2>{});
        });

        // Phases 2 and 3: token contraction of the previous tile, s-major.  A = Q^T / dO^T gathered from the row-major
        // tiles with transposing LDS reads (k-slot (s, g, kk) of the B operands is token 16s + 8(kk/4) + 4g + kk%4; a
        // 16-lane group covers 16 columns c), requested two operand sets ahead.  The s = 0 MFMAs only need the operands
        // phase 1 produced, so elements 8..15 are converted between them.  The region is fenced and contains no other
        // LDS instruction, so the partial LDS waits count exactly the asynchronous reads.
        __builtin_amdgcn_sched_barrier(0);
        {
            static_for<NSET>([&](auto ic) {
                constexpr int idx = decltype(ic)::value;
                constexpr int s = idx / CT, ct = idx % CT;
                if constexpr (idx + 2 < NSET) request_tr(std::integral_constant<int, idx + 2>{});
                constexpr int ahead = (NSET - 1 - idx) < 2 ? (NSET - 1 - idx) : 2;
                lds_tr_wait_n<4 * ahead>(tq[idx % 3], tg[idx % 3]);
                // (element-wise slices behind each matrix instruction: see ew_slot)
                auto after_slot2 = [&](auto kc) {
                    ew_slot(std::integral_constant<int, NS1 + 3 * idx + decltype(kc)::value>{});
                };
                dk[ct] = mfma32(tr_value(tq[idx % 3]), dmB[s], dk[ct]);
                if constexpr (idx == NSET - 1 && !TAIL) prepare_tile();     // scalar work of the next fill, under this MFMA
                after_slot2(std::integral_constant<int, 0>{});
                du[ct] = mfma32(tr_value(tq[idx % 3]), dnB[s], du[ct]);
                after_slot2(std::integral_constant<int, 1>{});
                dv[ct] = mfma32(tr_value(tg[idx % 3]), pB[s], dv[ct]);
                after_slot2(std::integral_constant<int, 2>{});
            });
        }
        __builtin_amdgcn_sched_barrier(0);
        // The first products were written by inline-assembly MFMAs the compiler cannot see.  The 6 CT contraction MFMAs
        // issued since then cover the wait states before the next step's element-wise code reads them; what is still
        // needed is that their registers stay allocated to the end of the step even when nothing reads them (the
        // phantom steps), or the compiler hands them to other values that the late write would overwrite.
        static_assert(KS >= 2 && NSET >= 2 && 6 * CT >= 8, "the contraction MFMAs of a step must cover the hazard window of its first products");
        asm volatile("" :: "v"(m), "v"(n), "v"(da));
    };

    // Pipeline over tiles k = 0 .. nt (step k: first products of tile k, element-wise + contraction of tile k-1).
    // Stage of tile k is k % 4; the two (m, n, da) register sets alternate with the parity of k.  Before step k every
    // wave waits for its own outstanding loads (tiles <= k), then the barrier publishes tile k and retires the stage
    // that tile k+2 is about to overwrite (last read by the contraction of tile k-2 in step k-1).
    f32x16 mA, nA, dA_, mB, nB, dB_;
#pragma unroll
    for (int x = 0; x < 16; ++x) { mA[x] = 0.0f; nA[x] = 0.0f; dA_[x] = 0.0f; mB[x] = 0.0f; nB[x] = 0.0f; dB_[x] = 0.0f; }
    auto sync_step = [&](auto st_c, int nvalid) {
        constexpr int ST = decltype(st_c)::value;
        // All of this wave's loads, not only the older tile's: a partial count (the next tile's loads still in flight)
        // measured no faster.
        wait_vmcnt<0>();
        if constexpr (TAIL) {
            if (nvalid < 32) zero_tail(ST, nvalid);
        }
        // (a bare barrier: the LDS-direct loads were waited for just above, and this wave's LDS reads of the stage that
        // is refilled next were consumed by the matrix instructions of the step before)
        __builtin_amdgcn_s_barrier();
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    // nt + 1 steps (step k contracts tile k-1), in trips of four (one per LDS stage) and a remainder of up to three.
    {
        int k = 0;
        for (; k + 3 <= nt; k += 4) {
            sync_step(I0{}, nv0);
            step(I0{}, I3{}, mA, nA, dA_, mB, nB, dB_, k > 0, nv2);
            sync_step(I1{}, nv1);
            step(I1{}, I0{}, mB, nB, dB_, mA, nA, dA_, true, nv3);
            sync_step(I2{}, nv2);
            step(I2{}, I1{}, mA, nA, dA_, mB, nB, dB_, true, nv0);
            sync_step(I3{}, nv3);
            step(I3{}, I2{}, mB, nB, dB_, mA, nA, dA_, true, nv1);
        }
        if (k <= nt) {
            sync_step(I0{}, nv0);
            step(I0{}, I3{}, mA, nA, dA_, mB, nB, dB_, k > 0, nv2);
            if (k + 1 <= nt) {
                sync_step(I1{}, nv1);
                step(I1{}, I0{}, mB, nB, dB_, mA, nA, dA_, true, nv3);
                if (k + 2 <= nt) {
                    sync_step(I2{}, nv2);
                    step(I2{}, I1{}, mA, nA, dA_, mB, nB, dB_, true, nv0);
                }
            }
        }
    }
    wait_vmcnt<0>();
    if (PAIR && one_less) __builtin_amdgcn_s_barrier();
    __syncthreads();      // every wave is done reading the tile ring, which the epilogue reuses

    // PAIR: the first wave of a block takes over the other's sums of dK and dU, the other the first's of dV, each through 16 KB a
    // gradient that the taker alone reads, and which then serve its stores.
    unsigned char* region = smem_raw + (PAIR ? wv * 49152 + half * 32768 : wave * 16384);
    if constexpr (PAIR) {
        auto leave = [&](const f32x16 (&acc)[CT], unsigned char* to) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    f32x4 v;
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[x] = acc[ct][4 * a + x];
                    *reinterpret_cast<f32x4*>(to + (ct * 4 + a) * 1024 + lane * 16) = v;
                }
        };
        auto take = [&](f32x16 (&acc)[CT], const unsigned char* from) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(from + (ct * 4 + a) * 1024 + lane * 16);
#pragma unroll
                    for (int x = 0; x < 4; ++x) acc[ct][4 * a + x] += v[x];
                }
        };
        unsigned char* block = smem_raw + wv * 49152;
        if (half) {
            leave(dk, block);
            leave(du, block + 16384);
        } else {
            leave(dv, block + 32768);
        }
        __syncthreads();
        if (half) {
            take(dv, block + 32768);
        } else {
            take(dk, block);
            take(du, block + 16384);
        }
    }

    // dK^T registers 4a+x of row tile ct: c = 32ct + 8a + 4g + x, column j = l32, i.e. a lane owns runs of 4 c of weight row
    // j.  Stored directly these are 8- or 16-byte pieces scattered over 32 rows per instruction; instead each wave passes
    // one gradient block at a time through a private 16 KB region of the ring (16-byte chunk c16 of row r at chunk
    // c16 ^ r), reads it back row-wise and stores whole rows.  Only this wave touches the region, and LDS operations of
    // one wave complete in order, so no barrier is needed between the three blocks.
    {
        const long wsz = (long)gridDim.x * nblk * JB * DH;   // elements of one weight tensor
        const long row0 = (wrow - l32) * DH;                 // first element of this wave's block of rows
        // (The addresses are made here, and for PAIR by each store anew: there are no registers to keep them, or parts of them from
        // before the loop, beside all the sums.)
        int here = lane;
        asm volatile("" : "+v"(here));
        auto own_lane = [&]() {
            int l = here;
            if constexpr (PAIR) asm volatile("" : "+v"(l));
            return l;
        };
        auto store_f32 = [&](const f32x16 (&acc)[CT], float* dst) {      // rows of DH floats, 512-byte rows in LDS
            const int lane = own_lane(), l32 = lane & 31, g = lane >> 5;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    f32x4 v;
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[x] = acc[ct][4 * a + x];
                    *reinterpret_cast<f32x4*>(region + l32 * 512 + (((8 * ct + 2 * a + g) ^ l32) << 4)) = v;
                }
            const int c16 = lane & 31;
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const int row = 2 * k + (lane >> 5);
                if (c16 < DH / 4) {
                    const u32x4 v = *reinterpret_cast<const u32x4*>(region + row * 512 + ((c16 ^ row) << 4));
                    *reinterpret_cast<u32x4*>(dst + row0 + row * DH + c16 * 4) = v;
                }
            }
        };
        auto store_bf16 = [&](const f32x16 (&acc)[CT], bf16_t* dst) {    // rows of DH bf16, 256-byte rows in LDS
            const int lane = own_lane(), l32 = lane & 31, g = lane >> 5;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    bf16x4 v;
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[x] = (bf16_t)acc[ct][4 * a + x];
                    *reinterpret_cast<bf16x4*>(region + l32 * 256 + (((4 * ct + a) ^ (l32 & 15)) << 4) + 8 * g) = v;
                }
            const int c16 = lane & 15;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int row = 4 * k + (lane >> 4);
                if (c16 < DH / 8) {
                    const u32x4 v = *reinterpret_cast<const u32x4*>(region + row * 256 + ((c16 ^ (row & 15)) << 4));
                    *reinterpret_cast<u32x4*>(dst + row0 + row * DH + c16 * 8) = v;
                }
            }
        };
        const bool ku = !PAIR || !half, v = !PAIR || half;   // the gradients whose sums this wave has
        if (p.nslice > 1) {                                  // fp32 partial sums of this token slice
            float* base = p.part + (long)z * 3 * wsz;
            if (ku) { store_f32(dk, base); store_f32(du, base + wsz); }
            if (v) store_f32(dv, base + 2 * wsz);
        } else if (p.out_f32) {                              // one slice: the sums are the gradients
            if (ku) { store_f32(dk, static_cast<float*>(p.out[0])); store_f32(du, static_cast<float*>(p.out[1])); }
            if (v) store_f32(dv, static_cast<float*>(p.out[2]));
        } else {
            if (ku) { store_bf16(dk, static_cast<bf16_t*>(p.out[0])); store_bf16(du, static_cast<bf16_t*>(p.out[1])); }
            if (v) store_bf16(dv, static_cast<bf16_t*>(p.out[2]));
        }
    }
}

// Sums the token-slice partials of dK, dU and dV and converts to the output dtype, four values per lane.  Workgroups count the columns of
// the kernel that left them (rows of weights of a head's workgroup) as it did, then 1,024 values of such a column at a time, then the
// gradients.  (That kernel's grid is not padded: where its columns are no multiple of eight, a column's slices are on several XCDs, and behind a number of
// tiles that is none, this pass begins on another one.  62 columns in four slices behind 44 tiles in five parts, 8 x 171 tokens of 8 heads of 128 on two: 14.1 us, 13.8 in the
// order of rows.)
struct WeightSums {
    const float* part;
    void* out[3];
    long size;            // values of a gradient
    unsigned head;        // ... of a head
    int nslice, Hkuv, column;      // values of a column
    unsigned columns, steps;       // workgroups that the kernel's grid has for a slice; workgroups of this pass for a column
    FastDiv by_columns, by_steps, by_hkuv;
};
template <typename OutT>
__device__ __forceinline__ void slice_sum(const WeightSums& p, unsigned block)
{
    typedef OutT OutT4 __attribute__((ext_vector_type(4)));
    const unsigned k = p.by_columns.div(block), u = block - k * p.columns, w = p.by_steps.div(k), step = k - w * p.steps;
    const unsigned col = p.by_hkuv.div(u), hk = u - col * p.Hkuv, in = col * p.column + step * 1024 + threadIdx.x * 4;
    if (in >= p.head) return;
    const long i4 = (long)hk * p.head + in;
    const float* src = p.part + w * p.size + i4;
    auto load = [&](int z) { return *reinterpret_cast<const f32x4*>(src + 3 * z * p.size); };
    const f32x4 sum = sum_in_order(load(0), 1, p.nslice, load);
    OutT4 v;
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = (OutT)sum[x];
    *reinterpret_cast<OutT4*>(static_cast<OutT*>(w == 0 ? p.out[0] : w == 1 ? p.out[1] : p.out[2]) + i4) = v;
}
template <typename OutT>
__global__ __launch_bounds__(256) void reduce_partials_kernel(WeightSums p)
{
    slice_sum<OutT>(p, blockIdx.x);
}

// Both sums of a backward in one launch, behind both its kernels: a launch less, and one pass fills the chip where two were
// latency (2 x 300 tokens of 8 heads of 96, two K/U/V heads: 4.9 + 7.0 us under the profiler, 10.0 in one; the call, bound by the host there, 99 -> 92).  Workgroups: dq_blocks of dQ and
// r_blocks of dR per tile, then the gradients'.
template <int DH, typename OutT>
__global__ __launch_bounds__(256) void mhffn_bwd_sums_kernel(DqArgs p, unsigned dq_blocks, unsigned tile_blocks, unsigned tiles, FastDiv by_tiles,
                                                             WeightSums w)
{
    const unsigned of_tiles = tile_blocks * tiles;
    if (blockIdx.x < of_tiles) {
        const unsigned block = by_tiles.div(blockIdx.x);
        dqdr_sum<DH>(p, blockIdx.x - block * tiles, block, dq_blocks);
    } else {
        slice_sum<OutT>(w, blockIdx.x - of_tiles);
    }
}

// ------------------------------------------------------------------------------------------------ host side
static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Token slices of the dK/dU/dV kernel for a workspace of `ws_bytes`.  One workgroup fits a CU at a time, so a launch
// runs in rounds of CUs workgroups; a workgroup costs its share of the token tiles plus a fixed prologue and epilogue
// (loading its K/U/V blocks, storing 3 x 64 accumulator registers per lane: about 9 tiles' worth).  More slices than
// one are worth it only where one slice leaves CUs idle; with one slice the kernel writes dK, dU, dV itself and neither
// partial sums nor the summing pass exist.  Every further slice adds a set of fp32 partial sums that is written and
// read back once (priced at the time of a token tile per 2.5 MB: about 4 TB/s against 1.25 us per tile).
constexpr long DW_FIXED_TILES = 9;      // prologue + epilogue of a workgroup, in token tiles
// Two blocks a workgroup (PAIR) are the choice between: half the tiles for a wave, in steps that are 8 to 14 % longer (twice the fills a
// wave) and with two tiles' worth more at the end.  Whole backward, us, before / with it: 512 tokens of 8 heads of 96 with 8 experts of 256 40.8 / 36.2,
// 1,000 67.8 / 54.0 (two slices / none), 2,048 95.4 / 92.3, 8,192 282.3 / 284.5 (not taken); 600 of 4 heads of 128 with the same experts 47.5 / 40.6, of
// 12 with 4 of 128 41.9 / 34.9; 2 x 300 of 8 heads of 96 on two, eight slices / four, 54.3 / 51.6; 128 of 8 of 96 22.6 / 22.8 (not taken).
// In two slices they run instead of one, or of the other form's two or three, but not of its four and more, with which they are level.  The whole backward in two such
// slices over what the price takes without them, 100 calls drawn from layers of 4 to 16 heads that it would send there: instead of two 0.86 to 0.93 (136 tokens twice of 4 heads
// of 96 on two with 12 blocks 26.9 / 23.2), of three 0.94 to 0.96, of one 0.90 to 1.00 (409 of 8 of 128 on two with 121 82.6 / 74.0); instead of four or five 0.95 to 1.03,
// 0.99 on average (2 x 716 of 8 of 96 on four with 64 87.5 / 90.1, 2 x 376 64.7 / 61.9).
constexpr double DW_PAIR_FIXED_TILES = 10.8, DW_PAIR_STEP = 1.14;
constexpr long DW_BYTES_PER_TILE_TIME = 2500000;
struct DwPick {
    bool pair;
    int nslice;
};
static DwPick dw_pick(const Dims& d, size_t ws_bytes)
{
    const int nblk = d.E * (d.d_e / JB);
    const long ntile = (long)(d.H / d.Hkuv) * d.B * ((d.S + 31) / 32);
    const size_t slice_b = (size_t)3 * d.Hkuv * d.E * d.d_e * d.d_h * sizeof(float);
    DwPick best{false, 1};
    double best_cost = -1;
    for (int pair = 0; pair < 2; ++pair) {
        const long cols = (long)((nblk + (pair ? 1 : 3)) / (pair ? 2 : 4)) * d.Hkuv;
        if (pair && ntile < 2) break;      // (a tile for either half; slices have eight)
        for (long ns = 1; ns <= 64 && (ns == 1 || ns <= ntile / 8); ++ns) {
            if (ns > 1 && align256((size_t)ns * slice_b) > ws_bytes) break;
            if (pair && ns == 2 && !best.pair && best.nslice >= 4) continue;
            const long rounds = (cols * ns + CUS - 1) / CUS, tiles = (ntile + ns - 1) / ns;
            const double cost = rounds * (pair ? (tiles + 1) / 2 * DW_PAIR_STEP + DW_PAIR_FIXED_TILES : tiles + DW_FIXED_TILES) +
                                (ns > 1 ? ns * (double)slice_b / DW_BYTES_PER_TILE_TIME : 0);
            if (best_cost < 0 || cost < best_cost) { best = DwPick{pair != 0, (int)ns}; best_cost = cost; }
        }
    }
    return best;
}
int dw_slices_bf16(const Dims& d, size_t ws_bytes) { return dw_pick(d, ws_bytes).nslice; }
bool dw_token_halves(const Dims& d, size_t ws_bytes) { return dw_pick(d, ws_bytes).pair; }

static size_t dq_part_bytes(const Dims& d) { return (size_t)d.B * d.H * d.S * (d.d_h + d.E) * sizeof(float); }

// Tiles of 256 rows where they fill the chip, of 32 below that: a block of theirs takes a quarter of the time, with an eighth of
// the rows.  One part of 121 blocks of the 370M heads, 512 rows: 199 us with 256 rows, 48 with 32; 2,048 rows: 200 and (two
// rounds) 108.  At their best numbers of parts 512 rows take 34.5 us with 32 rows, 36.1 with 256, 733 rows 49.7 and 45.0.  The prices lose
// 0.7 % on average and 10 % at worst over 160 training calls drawn from layers of 4 to 16 heads and 128 to 16,384 tokens (the whole backward with tile
// heights and numbers of parts around the pick; profiles/pick_parts_sweep.csv).  Steps of 1.9 and 0.36 with sums at 0.5 us per MB lose 0.6 %, but make parts of more sums
// (4 x 471 tokens of 8 heads of 96 with 9 blocks 45.4 -> 48.7 us) and with them workspaces larger (2 x 2,568 of 8 of 128 with 90 blocks none -> 67.5 MB).
// Where dK, dU, dV have slices to add up, the parts go along in that launch: whole backward of 2 x 300 tokens of 8 heads of 96 on
// two 61.7 us with a pass of their own in the price (32 rows, one part), 58.6 without (256 rows, eight parts); 900 of 8 of 128 on four 117.0, 114.6.
// (With no room behind the slices, too, where the pass is there: the choice does not cost more than 1 % then, over 30 calls.)
// Tiles of 256 rows that are half empty are no choice, whatever the prices of a part of one block say: 64 rows of 6 heads of 64 with 25 blocks
// 12.1 us in 25 parts, 8.8 in 5 of 32-row tiles; 50 of 4 heads of 128 with 24 blocks 12.5, 10.5; 128 of 2 heads of 128 with 9 blocks 13.2, 8.9.
constexpr Variant DQ_VARIANTS[] = {{256, 1.7, 0.15, 1, 0, 129}, {32, 0.36, 0.15, 1, DQ32_A + 1}};
Pick dq_pick_bf16(const Dims& d, size_t ws_bytes, int phases)
{
    return pick_parts(DQ_VARIANTS, d, d.E * (d.d_e / JB), d.E <= GATE_WIN, dq_part_bytes(d), phases & PH_ONE_PART ? 0 : ws_bytes,
                      dw_slices_bf16(d, ws_bytes) > 1 ? 0 : 2);
}

static size_t dw_slice_bytes(const Dims& d, int nslice) { return align256((size_t)nslice * 3 * d.Hkuv * d.E * d.d_e * d.d_h * sizeof(float)); }
size_t bwd_min_workspace_bytes_bf16(const Dims& d)
{
    const int ns = dw_slices_bf16(d, ~(size_t)0);
    return ns > 1 ? dw_slice_bytes(d, ns) : 0;
}

// The parts of dQ, dR lie behind the token slices of dK, dU, dV, so that one launch can add up both.  Where they do not fit there
// they share the workspace, and are added up before the slices are written.  So they do where both are most of what the memory-side
// cache holds: the parts are still in it then right behind their kernel, and gone behind the next one (training steps in two passes / in
// one: 84 MB 437.5 us / 435.6, 126 MB 668 / 667, 155 MB 493.8 / 491.6, 168 MB 931 / 934, 196 MB 1,094 / 1,098).
constexpr size_t SUMS_TOGETHER_B = (size_t)160 << 20;
static bool sums_together(const Dims& d, int nslice, int nsplit)
{
    return nslice > 1 && nsplit > 1 && dw_slice_bytes(d, nslice) + nsplit * dq_part_bytes(d) <= SUMS_TOGETHER_B;
}
size_t bwd_workspace_bytes_bf16(const Dims& d)
{
    const int nq = dq_pick_bf16(d, ~(size_t)0, 0).nsplit;
    const size_t dw = bwd_min_workspace_bytes_bf16(d), dq = nq > 1 ? align256(nq * dq_part_bytes(d)) : 0;
    return sums_together(d, dw_slices_bf16(d, ~(size_t)0), nq) ? dw + dq : dw > dq ? dw : dq;
}

template <int DH>
static hipError_t launch_bwd_t(const void* Q, const void* K, const void* U, const void* V, const float* R,
                               const void* dO, void* dQ, void* dK, void* dU, void* dV, float* dR, int grad_w_f32,
                               void* ws, size_t ws_bytes, const Dims& d, hipStream_t st, int phases)
{
    hipError_t err = hipSuccess;
    float* part = reinterpret_cast<float*>(ws);
    const int nbe = d.d_e / JB, G = d.H / d.Hkuv, nslice = dw_slices_bf16(d, ws_bytes);
    const long wsz = (long)d.Hkuv * d.E * d.d_e * d.d_h;
    const Pick pick = dq_pick_bf16(d, ws ? ws_bytes : 0, phases);
    const size_t slices_b = dw_slice_bytes(d, nslice);
    constexpr int ALL = PH_BWD_DQDR | PH_BWD_DKDUDV | PH_BWD_REDUCE;
    const bool together = (phases & ALL) == ALL && sums_together(d, nslice, pick.nsplit) && slices_b + pick.nsplit * dq_part_bytes(d) <= ws_bytes;
    DqArgs dq{(const bf16_t*)Q, (const bf16_t*)dO, (const bf16_t*)K, (const bf16_t*)U, (const bf16_t*)V, R, (bf16_t*)dQ, dR,
              together ? reinterpret_cast<float*>(reinterpret_cast<char*>(ws) + slices_b) : part, RowMap(d), Parts(d.E, nbe, pick.nsplit), pick.tile_rows};
    // the summing pass's workgroups of a tile for dQ and dR, and the tiles of the grid of dQ/dR
    const int in_tile = dq.rows.n < pick.tile_rows ? dq.rows.n : pick.tile_rows;
    const unsigned qb = (unsigned)((in_tile * (DH / 4) + 255) / 256), rb = (unsigned)(((long)in_tile * d.E + 255) / 256);
    const unsigned tiles = whole_xcds(d, pick, sizeof(bf16_t));
    static_assert(32 * (DH / 4) % 256 == 0, "a workgroup's rows are of one tile");

    const bool pair = dw_pick(d, ws_bytes).pair;
    const int nb = pair ? 2 : 4;            // blocks of a workgroup of dK/dU/dV
    const unsigned columns = (unsigned)((d.E * nbe + nb - 1) / nb * d.Hkuv);

    if (phases & PH_BWD_DQDR) {
        const DqArgs& a = dq;
        const int tokw = pick.tile_rows;
        const int smem = tokw == 32 ? DQ32_SMEM : DQ_NST * DQ_STAGE_B + (d.E < GATE_WIN ? d.E : GATE_WIN) * tokw * (int)sizeof(float);
        if (smem > 160 * 1024) return hipErrorInvalidValue;
        static LdsOptIn optin, optin32;
        err = tokw == 32 ? ensure_dynamic_lds(optin32, (const void*)mhffn_bwd_dqdr_rows32_kernel<DH>, smem)
                         : ensure_dynamic_lds(optin, (const void*)mhffn_bwd_dqdr_kernel<DH>, smem);
        if (err != hipSuccess) return err;
        dim3 grid(tiles, (unsigned)a.parts.nsplit);
        if (tokw == 32) hipLaunchKernelGGL((mhffn_bwd_dqdr_rows32_kernel<DH>), grid, dim3(DQ32_W * 64), smem, st, a);
        else hipLaunchKernelGGL((mhffn_bwd_dqdr_kernel<DH>), grid, dim3(512), smem, st, a);
        if (a.parts.nsplit > 1 && !together)
            hipLaunchKernelGGL((mhffn_bwd_dqdr_sum_kernel<DH>), dim3(tiles, qb + rb), dim3(256), 0, st, a, qb);
        err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    if (phases & PH_BWD_DKDUDV) {
        DwArgs a{(const bf16_t*)Q, (const bf16_t*)dO, (const bf16_t*)K, (const bf16_t*)U, (const bf16_t*)V, R, part,
                 {dK, dU, dV}, grad_w_f32, d.B, d.H, G, d.S, d.E, nbe, nslice, d.tokmaj};
        const bool tail = d.S % 32 != 0;
        const int smem = (pair ? 2 * DW_NST * DW_PAIR_STAGE_B : DW_NST * DW_STAGE_B) + 128;
        static LdsOptIn optin[4];
        auto* fn = pair ? tail ? mhffn_bwd_dkdudv_kernel<DH, true, TokenHalves> : mhffn_bwd_dkdudv_kernel<DH, false, TokenHalves>
                        : tail ? mhffn_bwd_dkdudv_kernel<DH, true> : mhffn_bwd_dkdudv_kernel<DH, false>;
        err = ensure_dynamic_lds(optin[2 * pair + tail], (const void*)fn, smem);
        if (err != hipSuccess) return err;
        hipLaunchKernelGGL(fn, dim3((unsigned)d.Hkuv, columns / d.Hkuv, (unsigned)nslice), dim3(256), smem, st, a);
        err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    if ((phases & PH_BWD_REDUCE) && nslice > 1) {
        const int column = nb * JB * DH;
        static_assert(2 * JB * DH % 1024 == 0, "a workgroup's values are of one column");
        const WeightSums w{part, {dK, dU, dV}, wsz, (unsigned)(wsz / d.Hkuv), nslice, d.Hkuv, column, columns, (unsigned)column / 1024,
                           FastDiv(columns), FastDiv(column / 1024), FastDiv(d.Hkuv)};
        const unsigned wb = 3 * columns * w.steps, tb = together ? (qb + rb) * tiles : 0;
        if (together && grad_w_f32)
            hipLaunchKernelGGL((mhffn_bwd_sums_kernel<DH, float>), dim3(tb + wb), dim3(256), 0, st, dq, qb, qb + rb, tiles, FastDiv(tiles), w);
        else if (together)
            hipLaunchKernelGGL((mhffn_bwd_sums_kernel<DH, bf16_t>), dim3(tb + wb), dim3(256), 0, st, dq, qb, qb + rb, tiles, FastDiv(tiles), w);
        else if (grad_w_f32)
            hipLaunchKernelGGL((reduce_partials_kernel<float>), dim3(wb), dim3(256), 0, st, w);
        else
            hipLaunchKernelGGL((reduce_partials_kernel<bf16_t>), dim3(wb), dim3(256), 0, st, w);
        err = hipGetLastError();
    }
    return err;
}

hipError_t launch_bwd_bf16(const void* Q, const void* K, const void* U, const void* V, const float* R, const void* dO,
                           void* dQ, void* dK, void* dU, void* dV, float* dR, int grad_w_f32, void* ws, size_t ws_bytes,
                           const Dims& d, hipStream_t st, int phases)
{
    switch (d.d_h) {
        case 64: return launch_bwd_t<64>(Q, K, U, V, R, dO, dQ, dK, dU, dV, dR, grad_w_f32, ws, ws_bytes, d, st, phases);
        case 96: return launch_bwd_t<96>(Q, K, U, V, R, dO, dQ, dK, dU, dV, dR, grad_w_f32, ws, ws_bytes, d, st, phases);
        case 128: return launch_bwd_t<128>(Q, K, U, V, R, dO, dQ, dK, dU, dV, dR, grad_w_f32, ws, ws_bytes, d, st, phases);
    }
    return hipErrorInvalidValue;
}

}  // namespace mhffn
