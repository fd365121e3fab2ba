// Fused multi-head FFN forward for gfx950 (bf16 MFMA, fp32 accumulation).
//
// One workgroup (4 waves, one per SIMD, 512 registers each) owns 256 rows of one K/U/V head (tokens of any batch and q-head
// of its group: RowMap) and all the head's blocks or one part of them (pick_parts); a wave owns 64 rows (NT = 2 column tiles
// of 32), "tokens" below.  With few rows the same code runs on 128 of them, one column tile per wave, and four more waves do the
// filling (FWD_VARIANTS, fwd_body).  The workgroup streams the K, U, V blocks (32 rows of the E*d_e axis at a time) straight
// from the weight tensors into a ring of LDS stages with asynchronous LDS-direct loads.  Per block and wave:
//     M^T = K Q^T, N^T = U Q^T               (A = rows of the K/U tiles, B = Q^T held in AGPRs for the whole kernel)
//     P^T = silu(M^T) * N^T * r_e             (fp32 in the accumulator registers, rounded once to bf16)
//     O^T += V^T P^T                          (A = columns of the V tile via transposing LDS reads, B = P^T registers)
// so the [tokens, E*d_e] intermediate lives only in registers.  Reference semantics:
// kernels/triton/flash_mlp_moe.py:243-266.
//
// Why this shape.  A wave that is alone on its SIMD issues about one instruction every five cycles whatever its type,
// and a 32x32x16 MFMA occupies the matrix pipe for 32 cycles: the kernel runs at MFMA speed only if every MFMA is
// followed by about five other instructions that do not depend on it.  With 64 tokens per wave every K/U/V operand
// read from LDS feeds two MFMAs (32 tokens per wave and two waves per SIMD needs the full LDS bandwidth to feed the
// matrix pipe), and the loop is software-pipelined by hand: the first-product MFMAs of block i+1 and the
// second-product MFMAs of block i form the slots of one step; the element-wise work of block i (16 element pairs per
// lane) is cut into 48 chunks of five VALU instructions that are spread over the slots, as are the LDS operand reads.
// First products use the VGPR form of the instruction (inline assembly) so the element-wise code reads them without
// v_accvgpr_read; the O^T accumulators live in AGPRs.
#include "mhffn_common.hpp"

namespace mhffn {

struct FwdArgs {
    const bf16_t* Q;
    const bf16_t* K;
    const bf16_t* U;
    const bf16_t* V;
    const float* R;
    bf16_t* O;
    float* part;          // [nsplit][Hkuv][rows.n][DH] fp32 partial sums (more parts than one)
    RowMap rows;          // rows of Q, O, R that meet one K/U/V head
    Parts parts;          // ... and the blocks of that head
    int tile_rows;
};

// LDS ring of FWD_NST stages, laid out as three regions (all V tiles, all K tiles, all U tiles).  The block loop is
// unrolled over the four stages, so the stage of every LDS access is a compile-time constant and goes into the
// instruction's 16-bit offset field: the per-lane parts of the addresses (row, swizzled chunk) are computed once before the
// loop and no step spends VALU instructions on addresses.  V and K regions lie below 64 KB; the U reads use a second set
// of per-lane bases that already contains the U region's start.
constexpr int FWD_NST = 4;
constexpr int FWD_REGION_B = FWD_NST * TILE_B;   // 32 KB
constexpr int FWD_V0 = 0, FWD_K0 = FWD_REGION_B, FWD_U0 = 2 * FWD_REGION_B;
constexpr int FWD_RING_B = 3 * FWD_REGION_B;     // 96 KB

// LDS operations issued behind the K/U reads of k-step ks up to the wait in front of that k-step's matrix instructions,
// for the issue order of the block step (K/U of k-steps 0 and 1 up front; in k-step j first the four V^T reads of row
// tile j - 1 while 1 <= j <= CT, then the two K/U reads of k-step j + 2).
__host__ __device__ constexpr int fwd_younger_reads(int ks, int KS, int CT)
{
    int n = ks == 0 ? 2 : 0;                       // k-step 1's reads follow k-step 0's up front
    for (int j = ks < 2 ? 0 : ks - 1; j <= ks; ++j) n += (j >= 1 && j <= CT ? 4 : 0) + (j + 2 < KS ? 2 : 0);
    return n;
}

// One matrix instruction of the first products, Q^T in accumulation registers or (QV) in ordinary ones: with two waves per SIMD a wave
// has 256 of both together, and the compiler would split them in half.
template <bool QV, bool FIRST>
__device__ __forceinline__ void first_product(f32x16& d, bf16x8 a, bf16x8 q)
{
    if constexpr (QV) {
        if constexpr (FIRST) mfma32_vgpr_first(d, a, q);
        else mfma32_vgpr_acc(d, a, q);
    } else {
        if constexpr (FIRST) mfma32_vgpr_first_bacc(d, a, q);
        else mfma32_vgpr_acc_bacc(d, a, q);
    }
}

// FILLERS: waves 4 to 7 do nothing but fill the ring, for waves 0 to 3.  A fill instruction holds its wave for 30 ns and more, six of
// them a third of a step of one column tile: a block takes 0.53 us instead of 0.60 (d_h 96; 0.60 instead of 0.67 with 128), 733 tokens of the
// 128M layer 19.5 us instead of 21.2.  With two column tiles a wave needs more than the 256 registers that two waves per SIMD leave it.
template <int DH, int NT, bool FILLERS>
__device__ __forceinline__ void fwd_body(const FwdArgs& p)
{
    constexpr int KS = DH / 16, CT = DH / 32, NW = 4, WT = 32 * NT, BT = NW * WT;
    constexpr int FILL = 24 / NW;
    constexpr int NG1 = 2 * NT * KS, NG2 = 2 * NT * CT, NSLOT = NG1 + NG2;   // MFMAs per step
    // The first products of a step are written by inline-assembly MFMAs whose results the next step's element-wise code
    // reads without a fence of its own: the NG2 second-product MFMAs issued in between (32 matrix-pipe cycles each) are
    // what covers the 18 wait states an MFMA result needs before a VALU read.
    static_assert(NG2 >= 4, "the second-product MFMAs of a step must cover the hazard window of its first products");
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    // gate values of one expert window: [min(E, GATE_WIN)][NW][64], a wave's WT rows (repeated where that is 32)
    float* sR = reinterpret_cast<float*>(smem + FWD_RING_B);

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // blockIdx.x = tile * Hkuv + kv-head: the head index runs fastest, so each head's weights stay in one XCD's L2
    arguments_first(p);
    const int tile = p.rows.by_hkuv.div(blockIdx.x), hk = blockIdx.x - tile * p.rows.Hkuv, z = blockIdx.y;
    if (tile * BT >= p.rows.n) return;                       // (whole_xcds)
    const int tok0 = tile * BT + wave * WT;                  // this wave's rows of the list (RowMap)
    const int nbe = p.parts.nbe, E = p.parts.E;
    const int blk0 = p.parts.first(z), nblk = p.parts.first(z + 1) - blk0;   // blocks of this workgroup, counted from blk0
    const int ex0 = p.parts.by_nbe.div(blk0), jb0 = blk0 - ex0 * nbe;        // expert of the first, its place in the expert
    const int nex = p.parts.by_nbe.div(jb0 + nblk + nbe - 1);                // experts they belong to, counted from ex0
    const long wbase = ((long)hk * E * nbe + blk0) * JB * DH;
    const bf16_t* Kh = p.K + wbase;
    const long offU = p.U - p.K, offV = p.V - p.K;

    auto issue_block = [&](int blk, int stage) {
        const int bc = blk < nblk ? blk : nblk - 1;
        const long roff = (long)bc * JB * DH;
#pragma unroll
        for (int k = 0; k < FILL; ++k) {
            const int id = (FILLERS ? wave & (NW - 1) : wave) + NW * k;      // (the filling waves are numbered from NW on)
            const int which = id >> 3;
            const long toff = which == 0 ? 0 : (which == 1 ? offU : offV);
            const int region = which == 0 ? FWD_K0 : (which == 1 ? FWD_U0 : FWD_V0);
            tile_fill_ins<DH>(Kh + toff + roff, DH, smem + region + stage * TILE_B, id & 7, lane);
        }
    };
    if (FILLERS && wave >= NW) {
        // One barrier of the workgroup for each of the others': behind the landing of blocks 0, and of b + 1 before step b.
        auto barrier = [&]() {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
        issue_block(0, 0);
        issue_block(1, 1);
        issue_block(2, 2);
        __builtin_amdgcn_sched_barrier(0);
        wait_vmcnt<2 * FILL>();
        barrier();
        const int window = GATE_WIN * nbe;
        for (int b = 0; b < nblk; ++b) {
            if (b > 0 && b % window == 0) {      // (the others restage the gate values)
                barrier();
                barrier();
            }
            wait_vmcnt<FILL>();
            barrier();
            issue_block(b + 3, (b + 3) % FWD_NST);
            __builtin_amdgcn_sched_barrier(0);
        }
        wait_vmcnt<0>();
        barrier();
        return;
    }
    const int first = tok0 < p.rows.n ? tok0 : p.rows.n - 1;
    const RowMap::Run run = p.rows.run(hk, first, WT);
    // The Q rows come from HBM and are the longest wait of the prologue: request them before anything else.
    bf16x8 q[NT][KS];
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
        int t = tok0 + ct * 32 + l32;
        t = t < p.rows.n ? t : p.rows.n - 1;
        const bf16_t* qr = p.Q + p.rows.tok(run, hk, first, t) * DH + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) q[ct][ks] = *reinterpret_cast<const bf16x8*>(qr + ks * 16);
    }
    if (!FILLERS) issue_block(0, 0);
    // Gate values of the workgroup's tokens, expert-major: one asynchronous 4-byte LDS-direct load per expert
    // and wave (lane = token, so the 64 values of an instruction are contiguous in LDS).  LDS holds a window of GATE_WIN
    // experts at a time; the first window is issued between block 0 and block 1, so that the wait for block 0 below
    // covers it too, and a layer with more experts restages the tile between two steps of the block loop.
    const float* rrow;
    {
        int t = tok0 + lane % WT;
        t = t < p.rows.n ? t : p.rows.n - 1;
        rrow = p.R + p.rows.gate(run, hk, first, t) * E + ex0;
    }
    auto stage_gates = [&](int e0) {
        const int e1 = e0 + GATE_WIN < nex ? e0 + GATE_WIN : nex;
        for (int e = e0; e < e1; ++e)
            __builtin_amdgcn_global_load_lds((gptr_t)(rrow + e), (lptr_t)(sR + ((e - e0) * NW + wave) * 64), 4, 0, 0);
    };
    stage_gates(0);
    if (!FILLERS) {
        issue_block(1, 1);
        issue_block(2, 2);
    }

    f32x16 oacc[CT][NT];
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int ct = 0; ct < NT; ++ct)
#pragma unroll
            for (int x = 0; x < 16; ++x) oacc[i][ct][x] = 0.0f;

    const int krow = row_perm32(l32);
    const TrLane<CT> trl = make_tr_lane<CT, 8, 4>(lane);
    // per-lane LDS addresses of the K row reads for every k-step (stage 0); the stage, and the distance to the U region,
    // go into the instruction's immediate offset
    unsigned kaddr[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
        kaddr[ks] = lds_addr(smem) + FWD_K0 + krow * TILE_ROW_B + (((2 * ks + g) ^ swz16(krow)) << 4);
    const unsigned smem0 = lds_addr(smem);

    // consumes M/N of block blk (mc, nc), produces M/N of block blk+1 (mn, nn); ST = blk % FWD_NST
    auto step = [&](auto st_, int blk, int e, f32x16 (&mc)[NT], f32x16 (&nc)[NT], f32x16 (&mn)[NT], f32x16 (&nn)[NT]) {
        constexpr int ST = decltype(st_)::value, STN = (ST + 1) % FWD_NST;
        if (!FILLERS) wait_vmcnt<FILL>();   // blocks <= blk+1 have landed (only block blk+2's loads may be in flight)
        __syncthreads();      // ... for every wave; and every wave is done with the stage about to be refilled

        // LDS reads of the step, all issued from inline assembly and waited for by count (the compiler's own waits are
        // full ones: behind a group of reads in flight it waits for the youngest along with the one it needs).  Issue
        // order: the two gate values, the K/U operands of k-steps 0 and 1, then per k-step ks the V^T operands of row tile
        // ks - 1 (for the second product, long after) and the K/U operands of k-step ks + 2.  LDS operations complete in
        // order, so "at most younger(ks) outstanding" means the operands of k-step ks have arrived; the V^T operands
        // have a full wait of their own in front of the second product, by when they have long landed.
        u32x2 rvu = lds_read_apart_async<NT>(lds_addr(sR + ((e & (GATE_WIN - 1)) * NW + wave) * 64 + l32));
        TrOperand av[CT][2];
        u32x4 ak[3], au[3];   // K/U operand ring, two k-steps ahead
        auto request = [&](auto kc) {
            constexpr int ks = decltype(kc)::value;
            ak[ks % 3] = lds_read16_async<STN * TILE_B>(kaddr[ks]);
            au[ks % 3] = lds_read16_async<FWD_U0 - FWD_K0 + STN * TILE_B>(kaddr[ks]);
        };
        auto request_v = [&](auto ic) {
            constexpr int i = decltype(ic)::value;
            av[i][0] = tile_read_cols_async<FWD_V0 + ST * TILE_B>(smem0, trl, i);
            av[i][1] = tile_read_cols_async<FWD_V0 + ST * TILE_B + 4096>(smem0, trl, i);
        };
        request(std::integral_constant<int, 0>{});
        request(std::integral_constant<int, 1>{});
        // the fill of the stage that has just come free is issued behind the first reads: its address arithmetic and six
        // instructions pass while those reads are on their way
        __builtin_amdgcn_sched_barrier(0);
        if (!FILLERS) issue_block(blk + 3, (ST + 3) % FWD_NST);
        float rinv[NT];
        bf16x8 pt[NT][2];
        float e0 = 0, e1 = 0, xn0 = 0, xn1 = 0;   // carried between the chunks of one element pair
        __builtin_amdgcn_sched_barrier(0);

        // chunk c: third c%3 of element pair c/3; pairs ordered s-major ((tile 0, s 0), (tile 1, s 0), (tile 0, s 1), ...)
        // so that each second-product operand P^T[ct][s] is complete well before the slot that consumes it.  The thirds
        // are cut so that their issue times are about equal (a transcendental instruction costs a lone wave about 10
        // cycles, a plain one about 6): 3 plain + 1 transcendental, 2 + 2, 4 + 1.
        float t1 = 0, s0 = 0;
        auto chunk = [&](auto c_) {
            constexpr int c = decltype(c_)::value;
            constexpr int pi = c / 3, third = c % 3;
            constexpr int ct = (pi / 4) % NT, pp = (pi % 4) + 4 * (pi / (4 * NT)), i0 = 2 * pp, i1 = i0 + 1;
            if constexpr (third == 0) {
                const float t0 = -LOG2E * mc[ct][i0];
                t1 = -LOG2E * mc[ct][i1];
                e0 = __builtin_amdgcn_exp2f(t0);
                xn0 = mc[ct][i0] * nc[ct][i0];
            } else if constexpr (third == 1) {
                e1 = __builtin_amdgcn_exp2f(t1);
                s0 = __builtin_amdgcn_rcpf(__builtin_fmaf(e0, rinv[ct], rinv[ct]));
                xn1 = mc[ct][i1] * nc[ct][i1];
            } else {
                const float s1 = __builtin_amdgcn_rcpf(__builtin_fmaf(e1, rinv[ct], rinv[ct]));
                pt[ct][i0 >> 3][i0 & 7] = (bf16_t)(xn0 * s0);
                pt[ct][i0 >> 3][i1 & 7] = (bf16_t)(xn1 * s1);
            }
        };

        static_for<NSLOT>([&](auto k_) {
            constexpr int k = decltype(k_)::value;
            if constexpr (k < NG1) {
                constexpr int ks = k / (2 * NT), w = k % (2 * NT), ct = w >> 1;
                if constexpr (w == 0) {
                    if constexpr (ks >= 1 && ks <= CT) request_v(std::integral_constant<int, ks - 1>{});
                    if constexpr (ks + 2 < KS) request(std::integral_constant<int, ks + 2>{});
                    if constexpr (ks == 0) {
                        lds_wait_n<fwd_younger_reads(0, KS, CT)>(ak[0], au[0], rvu);     // (the gate values are older)
                        // The gate value enters through its reciprocal: r / (1 + e) = 1 / fma(e, 1/r, 1/r), one multiply
                        // fewer per element.  1/r is clamped to the largest finite float, so a zero gate makes the
                        // denominator at least FLT_MAX, whose reciprocal the hardware flushes to exactly 0.
#pragma unroll
                        for (int c2 = 0; c2 < NT; ++c2) {
                            const unsigned bits = rvu[c2];    // (a scalar copy: the cast below must not see a vector element)
                            rinv[c2] = __builtin_amdgcn_fmed3f(__builtin_amdgcn_rcpf(__builtin_bit_cast(float, bits)),
                                                               -FLT_MAX_F, FLT_MAX_F);
                        }
                    } else {
                        lds_wait_n<fwd_younger_reads(ks, KS, CT)>();     // (consumed by asm matrix instructions only)
                    }
                }
                const bf16x8 a = __builtin_bit_cast(bf16x8, (w & 1) == 0 ? ak[ks % 3] : au[ks % 3]);
                first_product<FILLERS, ks == 0>((w & 1) == 0 ? mn[ct] : nn[ct], a, q[ct][ks]);
            } else {
                constexpr int g2 = k - NG1, s = g2 / (NT * CT), ct = (g2 / CT) % NT, i = g2 % CT;
                if constexpr (g2 == 0) {
#pragma unroll
                    for (int ii = 0; ii < CT; ++ii) lds_tr_wait(av[ii][0], av[ii][1]);
                }
                oacc[i][ct] = mfma32(tr_value(av[i][s]), pt[ct][s], oacc[i][ct]);
            }
            // element-wise chunks: chunk c goes behind slot c * (NSLOT - CT) / NCHUNK, so the last one is done before the
            // CT slots that consume P^T of the last tile's s = 1
            constexpr int NCHUNK = 24 * NT;
            static_for<NCHUNK>([&](auto c_) {
                if constexpr (decltype(c_)::value * (NSLOT - CT) / NCHUNK == k) chunk(c_);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        // The first products are written by the matrix pipe long after their instruction has issued.  Keep their
        // registers allocated to the end of the step even when nothing reads them (the phantom block behind an odd
        // count): otherwise the compiler hands them to other values, which the late write then overwrites.
        if constexpr (NT == 2) asm volatile("" :: "v"(mn[0]), "v"(mn[NT - 1]), "v"(nn[0]), "v"(nn[NT - 1]));
        else asm volatile("" :: "v"(mn[0]), "v"(nn[0]));
    };

    f32x16 mA[NT], nA[NT], mB[NT], nB[NT];
    if (FILLERS) wait_vmcnt<0>();
    else wait_vmcnt<2 * FILL>();   // all but the fills of blocks 1 and 2: block 0 and the gate values have landed
    __syncthreads();
    {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const bf16x8 a = tile_read_rows(smem + FWD_K0, krow, ks, g), u = tile_read_rows(smem + FWD_U0, krow, ks, g);
#pragma unroll
            for (int ct = 0; ct < NT; ++ct) {
                if (ks == 0) { first_product<FILLERS, true>(mA[ct], a, q[ct][0]); first_product<FILLERS, true>(nA[ct], u, q[ct][0]); }
                else { first_product<FILLERS, false>(mA[ct], a, q[ct][ks]); first_product<FILLERS, false>(nA[ct], u, q[ct][ks]); }
            }
        }
        // the element-wise code of step 0 reads these results
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) mfma_result_fence(mA[ct], nA[ct]);
    }
    // Four blocks per trip (one per LDS stage; the two M/N register sets alternate), then the last one to three.  (The
    // step of the last block still computes first products, of the block its prefetch clamped to; nothing reads them.)
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    using S3 = std::integral_constant<int, 3>;
    int e = 0, jb = jb0, blk = 0;
    auto advance = [&]() {
        if (++jb == nbe) { jb = 0; ++e; }
    };
    // (A window of GATE_WIN experts is a multiple of four blocks, so every window starts on stage 0 and register set A.
    // The launcher cuts the blocks only where one window holds all experts: a part then has just this first window.)
    for (int e0 = 0; e0 < nex; e0 += GATE_WIN) {
        if (e0 > 0) {
            __syncthreads();      // every wave has read its gate values of the window before
            stage_gates(e0);
            wait_vmcnt<0>();      // (also lands the two blocks in flight; the next step's wait then passes at once)
            __syncthreads();
        }
        const int wend = (e0 + GATE_WIN) * nbe < nblk ? (e0 + GATE_WIN) * nbe : nblk;
        for (; blk + 4 <= wend; blk += 4) {
            step(S0{}, blk, e, mA, nA, mB, nB);
            advance();
            step(S1{}, blk + 1, e, mB, nB, mA, nA);
            advance();
            step(S2{}, blk + 2, e, mA, nA, mB, nB);
            advance();
            step(S3{}, blk + 3, e, mB, nB, mA, nA);
            advance();
        }
    }
    if (blk < nblk) {
        step(S0{}, blk, e, mA, nA, mB, nB);
        advance();
        if (blk + 1 < nblk) {
            step(S1{}, blk + 1, e, mB, nB, mA, nA);
            advance();
            if (blk + 2 < nblk) step(S2{}, blk + 2, e, mA, nA, mB, nB);
        }
    }
    wait_vmcnt<0>();      // drain the phantom prefetches: they write the ring, which the epilogue reuses
    __syncthreads();      // every wave is done reading the ring

    if (p.parts.nsplit > 1) {     // a part of the blocks leaves its sums as they are, fp32, for the pass that adds the parts
        float* prow = p.part + (((long)z * p.rows.Hkuv + hk) * p.rows.n + tok0) * DH;
#pragma unroll
        for (int ct = 0; ct < NT; ++ct)
            store_rows_f32<DH>(smem + wave * TILE_B, prow + ct * 32 * DH, p.rows.n - tok0 - ct * 32, lane,
                               [&](auto ic) -> const f32x16& { return oacc[decltype(ic)::value][ct]; });
        return;
    }
    // O^T registers -> O[t][c].  Register 4a+b of row tile i is c = 32i + 8a + 4g + b: a lane owns runs of 4 c of one
    // token, which stored directly would be 8-byte pieces scattered over 32 rows per instruction.  Instead each wave
    // writes its rows x d_h tile into a private region of the ring (rows of 256 bytes, 16-byte chunk c16 of row r at
    // chunk c16 ^ (r & 15)), reads it back row-wise and stores whole rows: 16 lanes x 16 bytes per row, 4 rows per
    // instruction.  Only this wave touches the region, and LDS operations of one wave complete in order.
    {
        unsigned char* otile = smem + wave * (WT * TILE_ROW_B);
#pragma unroll
        for (int ct = 0; ct < NT; ++ct)
#pragma unroll
            for (int i = 0; i < CT; ++i)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    bf16x4 v;
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[x] = (bf16_t)oacc[i][ct][4 * a + x];
                    *reinterpret_cast<bf16x4*>(otile + (ct * 32 + l32) * TILE_ROW_B + (((4 * i + a) ^ (l32 & 15)) << 4) + 8 * g) = v;
                }
        const int c16 = lane & 15;
        auto store = [&](auto&& address_row) {
#pragma unroll
            for (int k = 0; k < 8 * NT; ++k) {
                const int row = 4 * k + (lane >> 4);
                if (c16 < DH / 8 && tok0 + row < p.rows.n) {
                    const u32x4 v = *reinterpret_cast<const u32x4*>(otile + row * TILE_ROW_B + ((c16 ^ (row & 15)) << 4));
                    *reinterpret_cast<u32x4*>(p.O + address_row(row) * DH + c16 * 8) = v;
                }
            }
        };
        if (run.tok.stride) store([&](int row) { return run.tok.base + (long)row * run.tok.stride; });
        else store([&](int row) { return p.rows.tok(hk, tok0 + row); });
    }
}

template <int DH>
__global__ __launch_bounds__(256) void mhffn_fwd_kernel(FwdArgs p) { fwd_body<DH, 2, false>(p); }
template <int DH>
__global__ __launch_bounds__(512) void mhffn_fwd_rows128_kernel(FwdArgs p) { fwd_body<DH, 1, true>(p); }

// 32 rows, four blocks a trip: the same products, element-wise formula and order of sums as fwd_body.  One barrier a trip: P^T
// operands and V tiles (which all waves read) have two sets, K and U tiles (which only their wave reads) are refilled as
// soon as the first products have read them.  A trip is 1.43 us, bound by the issue of a lone wave and LDS; with the tiles loaded
// to registers and written to LDS it was 2.15 (0.58 us of it the writes, 0.45 waiting for the loads).  With StreamedWeights the tiles are
// read past the caches (fwd_reads_past).
struct StreamedWeights {};
constexpr int FWD32_V0 = QUAD * 2 * TILE_B, FWD32_P0 = FWD32_V0 + 2 * QUAD * TILE_B, FWD32_R0 = FWD32_P0 + 2 * QUAD * 2048;
template <int DH, class... Mode>
__global__ __launch_bounds__(256) void mhffn_fwd_rows32_kernel(FwdArgs p)
{
    constexpr bool PAST = sizeof...(Mode) > 0;
    constexpr int KS = DH / 16, CT = DH / 32;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    float* sR = reinterpret_cast<float*>(smem + FWD32_R0);                       // [E][32]
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    arguments_first(p);
    const int tile = p.rows.by_hkuv.div(blockIdx.x), hk = blockIdx.x - tile * p.rows.Hkuv, z = blockIdx.y;
    const int tok0 = tile * 32, nbe = p.parts.nbe, E = p.parts.E, nsplit = p.parts.nsplit;
    if (tok0 >= p.rows.n) return;                            // (whole_xcds)
    const int blk0 = p.parts.first(z), nblk = p.parts.first(z + 1) - blk0;
    const int ex0 = p.parts.by_nbe.div(blk0), jb0 = blk0 - ex0 * nbe;
    const int nex = p.parts.by_nbe.div(jb0 + nblk + nbe - 1);
    const bf16_t* Kh = p.K + ((long)hk * E * nbe + blk0) * JB * DH;
    const long offU = p.U - p.K, offV = p.V - p.K;
    unsigned char* own = smem + wave * 2 * TILE_B;      // K | U of this wave's block
    auto row_of = [&](int t) { return tok0 + t < p.rows.n ? tok0 + t : p.rows.n - 1; };
    auto block = [&](int b0) { return Kh + (long)(b0 + wave < nblk ? b0 + wave : nblk - 1) * JB * DH; };
    auto fill_v = [&](int b0, int set) { quad_fill<DH, PAST>(block(b0) + offV, smem + FWD32_V0 + (set * QUAD + wave) * TILE_B, lane); };
    auto fill_ku = [&](int b0) {
        quad_fill<DH, PAST>(block(b0), own, lane);
        quad_fill<DH, PAST>(block(b0) + offU, own + TILE_B, lane);
    };

    bf16x8 q[KS];
    {
        const bf16_t* qr = p.Q + p.rows.tok(hk, row_of(l32)) * DH + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) q[ks] = *reinterpret_cast<const bf16x8*>(qr + ks * 16);
    }
    quad_stage_gates(sR, p.R + ex0, nex, tid, [&](int t) { return p.rows.gate(hk, row_of(t)) * E; });
    // (the compiler's own loads and stores end here; from the next line on the vmcnt events are the fills)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(q[ks]));
    __syncthreads();          // the gate values
    fill_ku(0);
    fill_v(0, 0);
    f32x16 o;
#pragma unroll
    for (int x = 0; x < 16; ++x) o[x] = 0.0f;
    const int krow = row_perm32(l32);
    const TrLane<CT> trl = make_tr_lane<CT, 8, 4>(lane);
    TrLane<1> tr{};                           // this wave's column tile
#pragma unroll
    for (int i = 0; i < CT; ++i)
        if (i == wave) { tr.off[0][0] = trl.off[i][0]; tr.off[0][1] = trl.off[i][1]; }
    const unsigned own_row = lds_addr(own) + krow * TILE_ROW_B, sw = swz16(krow);
    const unsigned smem0 = lds_addr(smem), ra = lds_addr(sR) + 4 * l32;

    auto trip = [&](auto set_, int b0) {
        constexpr int SET = decltype(set_)::value;
        bf16x8 pt[2];
        wait_vmcnt<8>();      // this wave's K and U of the trip have landed, its V (issued behind them) may be in flight
        __builtin_amdgcn_sched_barrier(0);
        u32x2 rv = lds_read_apart_async<1>(ra + 128 * p.parts.by_nbe.div(jb0 + (b0 + wave < nblk ? b0 + wave : nblk - 1)));
        QuadRows<KS, 2> a;
        static_for<KS>([&](auto kc) {
            constexpr int ks = decltype(kc)::value;
            const unsigned at = own_row + (((2 * ks + g) ^ sw) << 4);
            a.template request<0, ks>(at);
            a.template request<1, ks>(at + TILE_B);
        });
        f32x16 m, n;
#pragma unroll
        for (int x = 0; x < 16; ++x) { m[x] = 0.0f; n[x] = 0.0f; }
        static_for<KS>([&](auto kc) {
            constexpr int ks = decltype(kc)::value;
            a.template wait<ks>();
            m = mfma32(a.get(0, ks), q[ks], m);
            n = mfma32(a.get(1, ks), q[ks], n);
        });
        asm volatile("" : "+v"(rv));
        __builtin_amdgcn_sched_barrier(0);
        fill_ku(b0 + QUAD);   // (every read of the two tiles has returned)
        const unsigned rbits = rv[0];
        const float rinv = __builtin_amdgcn_fmed3f(__builtin_amdgcn_rcpf(__builtin_bit_cast(float, rbits)), -FLT_MAX_F, FLT_MAX_F);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float ex = __builtin_amdgcn_exp2f(-LOG2E * m[i]);
            const float xn = m[i] * n[i];
            pt[i >> 3][i & 7] = (bf16_t)(xn * __builtin_amdgcn_rcpf(__builtin_fmaf(ex, rinv, rinv)));
        }
        const unsigned sP = smem0 + FWD32_P0 + SET * QUAD * 2048 + lane * 16;
        lds_write16<0>(sP + wave * 2048, pt[0]);
        lds_write16<1024>(sP + wave * 2048, pt[1]);
        wait_vmcnt<16>();     // this wave's V has landed, the next K and U may be in flight
        quad_barrier();       // the four blocks' P^T and V tiles; and every wave is done with the trip before
        fill_v(b0 + QUAD, 1 - SET);
        if (wave < CT) {
            // (a block that is not there is the last one again, and not used)
            const int nb = nblk - b0 < QUAD ? nblk - b0 : QUAD;
            u32x4 pv[QUAD][2];
            TrOperand v[QUAD][2];
            static_for<QUAD>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const unsigned sV = smem0 + FWD32_V0 + (SET * QUAD + k) * TILE_B;
                pv[k][0] = lds_read16_async<k * 2048>(sP);
                pv[k][1] = lds_read16_async<k * 2048 + 1024>(sP);
                v[k][0] = tile_read_cols_async<0>(sV, tr, 0);
                v[k][1] = tile_read_cols_async<4096>(sV, tr, 0);
            });
            static_for<QUAD>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                lds_tr_wait_n<(QUAD - 1 - k) * 6 < 15 ? (QUAD - 1 - k) * 6 : 15>(v[k][0], v[k][1]);
                asm volatile("" : "+v"(pv[k][0]), "+v"(pv[k][1]));
                if (k < nb) {
                    o = mfma32(tr_value(v[k][0]), __builtin_bit_cast(bf16x8, pv[k][0]), o);
                    o = mfma32(tr_value(v[k][1]), __builtin_bit_cast(bf16x8, pv[k][1]), o);
                }
            });
        }
    };
    for (int b0 = 0; b0 < nblk; b0 += 2 * QUAD) {
        trip(std::integral_constant<int, 0>{}, b0);
        if (b0 + QUAD < nblk) trip(std::integral_constant<int, 1>{}, b0 + QUAD);
    }
    wait_vmcnt<0>();          // the fills of blocks that are not there write this wave's tiles, which the epilogue reuses
    __builtin_amdgcn_sched_barrier(0);
    if (wave >= CT) return;
    const int nrows = p.rows.n - tok0;
    if (nsplit > 1) {
        float* prow = p.part + (((long)z * p.rows.Hkuv + hk) * p.rows.n + tok0) * DH + 32 * wave;
        quad_store_f32(own, o, nrows, lane, [&](int row) { return prow + row * DH; });
    } else {
        quad_store_bf16(own, o, nrows, lane, [&](int row) { return p.O + p.rows.tok(hk, tok0 + row) * DH + 32 * wave; });
    }
}

// 32 rows and many blocks: the same products, element-wise formula and order of sums, the blocks in a pipeline as in the 32-row dQ/dR
// kernel.  Four waves take the first products and the element-wise work, each of every fourth block, in four phases, a phase apart
// from each other; four more request the tiles, 24 KB a phase, and add one block a phase to O, a column tile each.  A phase takes
// 0.34 us against the 0.40 of a quarter of a trip above (1,024 rows of 8 heads of 128, 8 experts of 256: 30.0 -> 27.4 us; one part
// of 512 rows of the 370M heads 48.9 -> 42.0, of 1,024 54.8 -> 47.6, of 512 of 8 heads of 96 24.0 -> 22.7, of 64 21.3 -> 20.8; 100 rows of
// the 1.3B heads 91.3 -> 75.2).  What bounds it is the issue of the loads to LDS, 65 cycles of a wave each (none of them: 37.1 us for
// the 512 rows), and the first phase, 570 of 690 cycles.  Three
// waves in three phases with operands read a phase ahead and a fifth wave for a third of the loads: 44.2.  Its four phases in front of
// the first sum cost short parts more than it gives: the kernel above takes those.
constexpr int FWDL_A = 4, FWDL_W = FWDL_A + 4;          // waves of the first kind, and all; also a block's phases up to its sums
constexpr int FWDL_AHEAD = 4;                             // phases between the request of a block's tiles and its first products
constexpr int FWDL_KU = FWDL_AHEAD + 1, FWDL_V = FWDL_AHEAD + FWDL_A;      // tile sets: K and U to a block's first phase, V to its sums
constexpr int FWDL_V0 = FWDL_KU * 2 * TILE_B, FWDL_P0 = FWDL_V0 + FWDL_V * TILE_B, FWDL_SMEM = FWDL_P0 + 2 * 2048;
template <int DH>
__global__ __launch_bounds__(FWDL_W * 64) void mhffn_fwd_rows32_long_kernel(FwdArgs p)
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
    const unsigned smem0 = lds_addr(smem);
    const int nphase = nblk + FWDL_A;     // block b: first products in phase b, its sums in phase b + FWDL_A; every phase ends with a barrier
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;

    if (wave < FWDL_A) {
        const int t = tok0 + l32 < p.rows.n ? tok0 + l32 : p.rows.n - 1;
        bf16x8 q[KS];
        {
            const bf16_t* qr = p.Q + p.rows.tok(hk, t) * DH + 8 * g;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) q[ks] = *reinterpret_cast<const bf16x8*>(qr + ks * 16);
        }
        const float* rrow = p.R + p.rows.gate(hk, t) * E + ex0;
        auto gate = [&](int b) { return rrow[p.parts.by_nbe.div(jb0 + (b < nblk ? b : nblk - 1))]; };
        float rnext = gate(wave), rinv = 0.0f;
        // (these loads end here: waited for in the loop, each trip would also wait for the next gate value)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(q[ks]));
        asm volatile("" : "+v"(rnext));
        const int krow = row_perm32(l32), sw = swz16(krow);
        unsigned at[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) at[ks] = smem0 + krow * TILE_ROW_B + (((2 * ks + g) ^ sw) << 4);
        const unsigned sP = smem0 + FWDL_P0 + lane * 16;

        f32x16 m, n;
        bf16x8 pt[2];
        QuadRows<KS, 2> a;
        // Phase 1: half the k-steps of M and N, with the reads of the others between the matrix instructions.
        constexpr int K1 = KS / 2;
        auto phase1 = [&](int b) {
            rinv = __builtin_amdgcn_fmed3f(__builtin_amdgcn_rcpf(rnext), -FLT_MAX_F, FLT_MAX_F);
            rnext = gate(b + FWDL_A);     // a round ahead of its use
            const unsigned ku = (b % FWDL_KU) * 2 * TILE_B;
            auto request = [&](auto kc) {
                constexpr int ks = decltype(kc)::value;
                const unsigned x = at[ks] + ku;
                a.template request<0, ks>(x);
                a.template request<1, ks, TILE_B>(x);
            };
            __builtin_amdgcn_sched_barrier(0);
            static_for<KS - K1>([&](auto kc) { request(kc); });
#pragma unroll
            for (int x = 0; x < 16; ++x) { m[x] = 0.0f; n[x] = 0.0f; }
            static_for<K1>([&](auto kc) {
                constexpr int ks = decltype(kc)::value;
                lds_wait_n<2 * (KS - K1 - 1)>();      // (as many k-steps are requested behind this one)
                asm volatile("" : "+v"(a.v[0][ks]), "+v"(a.v[1][ks]));
                m = mfma32(a.get(0, ks), q[ks], m);
                n = mfma32(a.get(1, ks), q[ks], n);
                __builtin_amdgcn_sched_barrier(0);
                request(std::integral_constant<int, KS - K1 + ks>{});
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        auto phase2 = [&]() {
            static_for<KS - K1>([&](auto kc) {
                constexpr int ks = K1 + decltype(kc)::value;
                asm volatile("" : "+v"(a.v[0][ks]), "+v"(a.v[1][ks]));       // (returned before the barrier)
                m = mfma32(a.get(0, ks), q[ks], m);
                n = mfma32(a.get(1, ks), q[ks], n);
            });
        };
        auto elements = [&](auto i0_, auto i1_) {
#pragma unroll
            for (int i = decltype(i0_)::value; i < decltype(i1_)::value; ++i) {
                const float ex = __builtin_amdgcn_exp2f(-LOG2E * m[i]);
                const float xn = m[i] * n[i];
                pt[i >> 3][i & 7] = (bf16_t)(xn * __builtin_amdgcn_rcpf(__builtin_fmaf(ex, rinv, rinv)));
            }
            asm volatile("" : "+v"(pt[0]), "+v"(pt[1]));     // (here, not behind the barrier)
        };
        using I4 = std::integral_constant<int, 4>;
        using I10 = std::integral_constant<int, 10>;
        using I16 = std::integral_constant<int, 16>;
        for (int i = 0; i <= wave; ++i) quad_barrier();      // (the first: block 0 has landed)
        int phase = wave;
        for (int b = wave; b < nblk; b += FWDL_A, phase += FWDL_A) {
            phase1(b);
            quad_barrier();
            phase2();
            elements(I0{}, I4{});
            quad_barrier();
            elements(I4{}, I10{});
            quad_barrier();
            elements(I10{}, I16{});
            const unsigned d = sP + (b & 1) * 2048;
            lds_write16<0>(d, pt[0]);
            lds_write16<1024>(d, pt[1]);
            quad_barrier();
        }
        for (; phase <= nphase; ++phase) quad_barrier();     // (and the one in front of the epilogue)
        return;
    }

    // Fills and sums.  Each of these waves requests a quarter of every tile: six vmcnt events a block.
    const int col = wave - FWDL_A;
    QuadFill<DH, FWDL_KU, FWDL_V> fill(p.K + ((long)hk * E * nbe + blk0) * JB * DH, p.U - p.K, p.V - p.K, nblk, smem, smem + FWDL_V0, col, lane);
    const TrLane<1> tr = quad_tr_lane<CT>(lane, col);
    f32x16 o;
#pragma unroll
    for (int x = 0; x < 16; ++x) o[x] = 0.0f;
    for (int b = 0; b < FWDL_AHEAD; ++b) {
        fill.aim(b);
        static_for<3>([&](auto t) {
            fill.request(t, I0{});
            fill.request(t, I1{});
        });
    }
    wait_vmcnt<6 * (FWDL_AHEAD - 1)>();
    quad_barrier();                           // block 0 has landed
    TrOperand v[2];
    auto phase_of = [&](auto sums_, int phase) {
        constexpr bool SUMS = decltype(sums_)::value;
        __builtin_amdgcn_sched_barrier(0);
        u32x4 pv[2];
        if constexpr (SUMS) {
            const unsigned sP = smem0 + FWDL_P0 + ((phase - FWDL_A) & 1) * 2048 + lane * 16;
            pv[0] = lds_read16_async<0>(sP);
            pv[1] = lds_read16_async<1024>(sP);
        }
        fill.aim(phase + FWDL_AHEAD);
        fill.request(I0{}, I0{});
        fill.request(I0{}, I1{});
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SUMS) {
            lds_wait_n<0>();
            asm volatile("" : "+v"(pv[0]), "+v"(pv[1]));
        }
        // this block's sums, each operand followed by the next block's (from the tile set that the next phase requests into)
        const unsigned aV = smem0 + FWDL_V0 + fill.v * TILE_B;
        static_for<2>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if constexpr (SUMS) o = mfma32(tr_value(v[s]), __builtin_bit_cast(bf16x8, pv[s]), o);
            __builtin_amdgcn_sched_barrier(0);
            v[s] = tile_read_cols_async<s * 4096>(aV, tr, 0);
            fill.request(std::integral_constant<int, 1 + s>{}, I0{});
            fill.request(std::integral_constant<int, 1 + s>{}, I1{});
            __builtin_amdgcn_sched_barrier(0);
        });
        wait_vmcnt<6 * (FWDL_AHEAD - 1)>();  // the next phase's first products have their tiles
        quad_barrier();
#pragma unroll
        for (int s = 0; s < 2; ++s) asm volatile("" : "+v"(v[s].lo), "+v"(v[s].hi));
    };
    int phase = 0;
    for (const int idle = col < CT ? FWDL_A : nphase; phase < idle; ++phase) phase_of(std::false_type{}, phase);
    for (; phase < nphase; ++phase) phase_of(std::true_type{}, phase);
    wait_vmcnt<0>();          // the fills of blocks that are not there write the tiles, which the epilogue reuses
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (col >= CT) return;
    unsigned char* own = smem + col * TILE_B;
    const int nrows = p.rows.n - tok0;
    if (nsplit > 1) {
        float* prow = p.part + (((long)z * p.rows.Hkuv + hk) * p.rows.n + tok0) * DH + 32 * col;
        quad_store_f32(own, o, nrows, lane, [&](int row) { return prow + row * DH; });
    } else {
        quad_store_bf16(own, o, nrows, lane, [&](int row) { return p.O + p.rows.tok(hk, tok0 + row) * DH + 32 * col; });
    }
}

// Adds the parts' sums (in the order of the parts) and rounds once: O row r of kv-head hk, four columns per lane.  blockIdx.x counts tiles
// and heads as the kernel that left the parts did.
template <int DH>
__global__ __launch_bounds__(256) void mhffn_fwd_sum_kernel(FwdArgs p)
{
    const int tile = p.rows.by_hkuv.div(blockIdx.x), hk = blockIdx.x - tile * p.rows.Hkuv;
    const unsigned i = blockIdx.y * 256 + threadIdx.x;
    const unsigned r = tile * p.tile_rows + i / (DH / 4), c = (i % (DH / 4)) * 4;
    if (r >= (unsigned)p.rows.n) return;
    const long step = (long)p.rows.Hkuv * p.rows.n * DH;
    const float* src = p.part + ((long)hk * p.rows.n + r) * DH + c;
    auto load = [&](int z) { return *reinterpret_cast<const f32x4*>(src + z * step); };
    const f32x4 sum = sum_in_order(load(0), 1, p.parts.nsplit, load);
    bf16x4 v;
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = (bf16_t)sum[x];
    *reinterpret_cast<bf16x4*>(p.O + p.rows.tok(hk, r) * DH + c) = v;
}

// Tiles of 256 rows (64 per wave) where they fill the chip; of 128 (32 per wave) below that: a step then takes 0.53 to 0.6 us
// instead of 1.0 (1,500 tokens of the 370M layer in one part: 130 us with 256 rows, 74 with 128; 733 tokens at each one's best number of
// parts 32.6 and 29.8, of the 128M layer 25.2 and 20.6), and the two are level where every compute unit has one.  Of 32, four blocks a trip of 1.43 us, below that, where 128-row tiles take, at each one's best
// number of parts: one token of the 370M layer 7.8 us against 10.0, 16 tokens of the 1.3B layer 20.3 against 22.5 (95 MB of
// weights); 400 rows in one part 46 against 82.  Rows have the same sums, bit for bit, in all three.  (Priced at 0.6 for 128 rows, as
// before its filling waves: the line between the two kernels lies where it did.)  Up to 32 rows the larger tiles are no choice, whatever the prices say of
// parts of one or two blocks: two tokens of 8 heads of 96 on four with 64 blocks 10.3 us in 64 parts of 128-row tiles, 7.2 in 16 of 32-row ones; one of 4 heads of 64
// with 42 7.9, 6.6; 40 such calls 15 % on average, the worst, of 16 blocks or fewer, 3 to 6 % the other way (6.1 / 6.5).
// A part of FWDL_FROM blocks or more goes through the pipeline.  Trips / pipeline, us in one part, 512 rows of 8 heads of 128: 4 blocks 6.1 / 6.6,
// 12 9.0 / 8.9, 20 11.7 / 11.1, 28 14.5 / 13.3, 32 15.9 / 14.5, 64 27.1 / 23.9; of 96: 16 blocks 9.3 / 9.4, 24 11.6 / 11.4, 32 13.7 / 13.3, 64 23.7 / 22.0;
// of 64: 16 8.6 / 8.7, 24 10.8 / 10.6, 32 12.9 / 12.7, 64 21.8 / 20.6.  (They meet at 12 to 20 blocks; the line above that is a cautious one, drawn
// when 16 and 64 were measured.)
constexpr int FWDL_FROM = 32;
constexpr Variant FWD_VARIANTS[] = {{256, 1.0, 0.2, 1, 0, 33}, {128, 0.6, 0.33, 1, 0, 33}, {32, 1.45, 0.05, QUAD}};
// A call in one part has its tile height by a step of 256 rows that is 8 % dearer on a full chip: three rounds of 128-row tiles are faster than two of 256-row ones, and rows have the same
// sums in both.  120 calls of 16,384 to 65,000 rows per head drawn from layers of 4 to 16 heads, us, 256 rows / 128: 37 of them with one and a half rounds or less of the larger 0.88 to 0.95
// (20,664 rows of 4 heads of 128 with 121 blocks 292 / 266, 41,160 of 2 of 96 with 64 142 / 125, 21,936 of 3 of 64 with 65 117 / 103); over all of them 3.0 % over the faster one on average with
// the step above, 0.03 % with this.  Calls that might be cut keep the step above beside their parts (2 x 1,571 tokens of 8 heads of 128 with 140 blocks in two parts of 256-row tiles 106,
// in one of 128 114).
constexpr Variant FWD_ONE_PART[] = {{256, 1.0, 0.3, 1, 0, 33}, FWD_VARIANTS[1], FWD_VARIANTS[2]};
static size_t fwd_part_bytes(const Dims& d) { return (size_t)d.B * d.H * d.S * d.d_h * sizeof(float); }
Pick fwd_pick_bf16(const Dims& d, size_t ws_bytes, int phases)
{
    const int blocks = d.E * (d.d_e / JB);
    const Pick pick = pick_parts(FWD_VARIANTS, d, blocks, d.E <= GATE_WIN, fwd_part_bytes(d), phases & PH_ONE_PART ? 0 : ws_bytes);
    return pick.nsplit > 1 ? pick : pick_parts(FWD_ONE_PART, d, blocks, d.E <= GATE_WIN, fwd_part_bytes(d), 0);
}

// Large weights are read past the caches by the trips of the 32-row kernel: each is read by one workgroup or a few at about the same time, and keeping it only pushes out
// what comes next.  Forward with its sums, us, kept / past, twelve sets of weights in turn: one token of 16 heads of 128 with 95 MB 23.1 / 21.3, with 74 MB 19.1 / 17.8,
// 32 tokens 24.2 / 23.0 and 20.5 / 19.7; the block 40.5 / 38.2 and 36.9 / 35.5 for one token.  Three sets in turn stay in the memory-side cache of 256 MB where they are
// smaller, and then the caches do help: the block with 48 MB (16 heads of 128 on eight) of 9 tokens 30.0 / 31.4, of 21 30.7 / 33.1, with 53 MB (12 heads of 96) of 16
// 27.8 / 29.1; twelve such sets 34.7 / 33.4, 36.8 / 35.5, 31.4 / 30.8.  The line lies where neither way loses: with 74 MB three sets in turn 33.4 / 33.7 to 36.9 / 35.7,
// with 95 MB 39.7 / 36.7.
constexpr size_t PAST_FROM_B = (size_t)64 << 20;
static bool fwd_pipeline(const Dims& d, const Pick& pick) { return pick.tile_rows == 32 && d.E * (d.d_e / JB) / pick.nsplit >= FWDL_FROM; }
bool fwd_reads_past(const Dims& d, const Pick& pick)
{
    return pick.tile_rows == 32 && !fwd_pipeline(d, pick) && (size_t)3 * d.Hkuv * d.E * d.d_e * d.d_h * sizeof(bf16_t) > PAST_FROM_B;
}

template <int DH>
static hipError_t launch_fwd_t(const FwdArgs& a, const Dims& d, const Pick& pick, hipStream_t st)
{
    const int tile_rows = pick.tile_rows;
    const int gates = d.E < GATE_WIN ? d.E : GATE_WIN;
    const bool pipeline = fwd_pipeline(d, pick), past = fwd_reads_past(d, pick);
    const int smem = pipeline          ? FWDL_SMEM
                     : tile_rows == 32 ? FWD32_R0 + gates * 32 * (int)sizeof(float)
                                     : FWD_RING_B + gates * 256 * (int)sizeof(float);
    if (smem > 160 * 1024) return hipErrorInvalidValue;
    auto* rows32 = past ? mhffn_fwd_rows32_kernel<DH, StreamedWeights> : mhffn_fwd_rows32_kernel<DH>;
    static LdsOptIn optin, optin128, optin32[2], optinl;
    const hipError_t e = pipeline           ? ensure_dynamic_lds(optinl, (const void*)mhffn_fwd_rows32_long_kernel<DH>, smem)
                         : tile_rows == 256 ? ensure_dynamic_lds(optin, (const void*)mhffn_fwd_kernel<DH>, smem)
                         : tile_rows == 128 ? ensure_dynamic_lds(optin128, (const void*)mhffn_fwd_rows128_kernel<DH>, smem)
                                            : ensure_dynamic_lds(optin32[past], (const void*)rows32, smem);
    if (e != hipSuccess) return e;
    dim3 grid(whole_xcds(d, pick, sizeof(bf16_t)), (unsigned)pick.nsplit);
    if (tile_rows == 256) hipLaunchKernelGGL((mhffn_fwd_kernel<DH>), grid, dim3(256), smem, st, a);
    else if (tile_rows == 128) hipLaunchKernelGGL((mhffn_fwd_rows128_kernel<DH>), grid, dim3(512), smem, st, a);
    else if (pipeline) hipLaunchKernelGGL((mhffn_fwd_rows32_long_kernel<DH>), grid, dim3(FWDL_W * 64), smem, st, a);
    else hipLaunchKernelGGL(rows32, grid, dim3(256), smem, st, a);
    if (a.parts.nsplit > 1) {
        static_assert(32 * (DH / 4) % 256 == 0, "a workgroup's rows are of one tile");
        dim3 sgrid(grid.x, (unsigned)(((a.rows.n < tile_rows ? a.rows.n : tile_rows) * (DH / 4) + 255) / 256));
        hipLaunchKernelGGL((mhffn_fwd_sum_kernel<DH>), sgrid, dim3(256), 0, st, a);
    }
    return hipGetLastError();
}

size_t fwd_workspace_bytes_bf16(const Dims& d)
{
    const int ns = fwd_pick_bf16(d, ~(size_t)0, 0).nsplit;
    return ns > 1 ? ns * fwd_part_bytes(d) : 0;
}

hipError_t launch_fwd_bf16(const void* Q, const void* K, const void* U, const void* V, const float* R, void* O,
                           void* ws, size_t ws_bytes, const Dims& d, hipStream_t st, int phases)
{
    if (!(phases & PH_FWD_MAIN)) return hipSuccess;
    const Pick pick = fwd_pick_bf16(d, ws ? ws_bytes : 0, phases);
    FwdArgs a{(const bf16_t*)Q, (const bf16_t*)K, (const bf16_t*)U, (const bf16_t*)V,           R,
              (bf16_t*)O,       (float*)ws,       RowMap(d),        Parts(d.E, d.d_e / JB, pick.nsplit), pick.tile_rows};
    switch (d.d_h) {
        case 64: return launch_fwd_t<64>(a, d, pick, st);
        case 96: return launch_fwd_t<96>(a, d, pick, st);
        case 128: return launch_fwd_t<128>(a, d, pick, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace mhffn
