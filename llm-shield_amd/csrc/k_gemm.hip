// Prefill GEMM against GGUF-quantized weights: y = x . W^T on the MFMA cores.
//
// Replaces PanelGemm (PanelGemm.cs:87-318) for calls of two or more tokens.
//
// Numerics.  The weight quants are small integers (Q8_0 q in [-127,127],
// Q4_0 q-8 in [-8,7], Q5_1 q in [0,31]) and therefore exact in fp16; only the
// per-32 block scale d (and Q5_1's min m) is not.  One MFMA of 16x16x32 covers
// exactly one quant block, so each block's dot of x with the integer quants
// comes out of the matrix core unscaled and the fp32 scale is applied on the
// vector ALU:  acc += d * (x . q)  (+ m * sum(x) for Q5_1).  The activation x
// enters as an fp16 pair hi + lo (two MFMAs into the same partial), ~22
// significant bits; a single fp16 or bf16 operand measured 4e-3 / 2e-2
// relative error on the 26-layer logits, the pair 3e-5.
//
// Determinism.  Each output is the same sequence of MFMAs and FMAs over its K
// blocks whatever M is and whichever tile shape or position its row lands in,
// so a token's result does not depend on the batch around it (the reference's
// batch invariance, PanelGemm.cs:28-31); that is what keeps a tree pass
// bit-identical to running its branches one at a time.  Tile shapes may
// therefore be chosen by M without changing a single bit.
//
// Pipeline.  K advances 64 (two quant blocks) per stage.  The waves of a
// workgroup sit side by side along N; each streams its own weight tiles from
// HBM as raw quant bytes into registers two stages ahead and decodes them
// there (a tile slot is the lane's B fragment), while the stage's activation
// tile goes to LDS once per workgroup, double buffered, and serves every wave.
// One barrier per stage.
//
// Outputs.  Store-mode results (and K-split partials) are written with
// nontemporal stores: their consumer runs on whichever XCD its workgroup lands
// on, so they must reach memory anyway.  Streamed out during the kernel rather
// than written back from L2 after it, the 256-row projections launched back
// to back took 1-6 % less time (QKV 25.4 -> 24.8 us, O 18.7 -> 17.8, down
// 34.9 -> 34.3); in the model, between other kernels, under 0.5 %.
//
// Tiles.  16 TM x 16 TN per wave, four to sixteen waves per workgroup, chosen
// by the shape (launch_mode).  Workgroup ids are remapped so each XCD (ids
// round-robin over 8) works on a contiguous run of a grouped tile order:
// neighbouring tiles on one XCD share weight and activation tiles in its L2.
#include "jev_dev.h"

#include <algorithm>
#include <type_traits>

namespace jev {

namespace {

constexpr int kCUs = 256;

// One loader chunk: a lane slot of a weight tile -- the quants of one row
// at k = 8g .. 8g + 7 of both blocks of the stage -- and that row's scales.
struct BChunk {
    uint4 q;       // bytes (Q8_0, Q5_1's byte copy): 16; nibbles (Q4_0): 8 in .x, .y
    uint32_t d, m; // two fp16 each (block 0 low half)
};

// Loads are unconditional with clamped addresses: a row past the weight's end
// or a block past K only feeds outputs that are never stored, and keeping the
// loop free of divergent loads lets the compiler count outstanding loads
// exactly instead of draining the queue every stage.

// Quants as these kernels read them: whole bytes, 1 KiB per tile -- Q8_0's
// (QWeight::qs, stored biased as q + 128) or Q5_1's byte copy (QWeight::qb, q
// itself: one byte permute and one packed subtraction per two weights instead
// of the nibble and fifth-bit assembly) -- or Q4_0's nibbles, 512 B per tile.
template <int TYPE>
constexpr bool kByteQuants = TYPE != kQ4_0;

template <int TYPE>
__device__ __forceinline__ rsrc_t quant_rsrc(const QWeight &w, uint32_t tiles)
{
    return make_rsrc(TYPE == kQ5_1 ? w.qb : w.qs, tiles * (kByteQuants<TYPE> ? 1024u : 512u));
}

// Four quants of a block as two fp16 pairs of exact integers: a byte b placed
// under the exponent byte is 1024 + b; the bias subtracts 1024 and, for Q8_0's
// biased bytes or Q4_0's offset 8, that too.
template <int TYPE>
__device__ __forceinline__ void decode4(const BChunk &c, int bb, int half, uint32_t &pa, uint32_t &pb)
{
    if (kByteQuants<TYPE>) {
        const uint32_t w = bb ? (half ? c.q.w : c.q.z) : (half ? c.q.y : c.q.x);
        bytes_to_f16(w, TYPE == kQ8_0 ? (_Float16)1152.0f : (_Float16)1024.0f, pa, pb);
    } else {
        // byte i = element i (low nibble) | element i + 4 (high nibble)
        const uint32_t w = bb ? c.q.y : c.q.x;
        const uint32_t n = half ? (w >> 4) & 0x0f0f0f0fu : w & 0x0f0f0f0fu;
        bytes_to_f16(n, (_Float16)1032.0f, pa, pb);
    }
}

// B fragment of block bb of a loaded chunk: 8 fp16 integers for the lane's
// row at k = 8g .. 8g + 7.
template <int TYPE>
__device__ __forceinline__ half8_t decode_b_frag(const BChunk &c, int bb)
{
    uint32_t o0, o1, o2, o3;
    decode4<TYPE>(c, bb, 0, o0, o1);
    decode4<TYPE>(c, bb, 1, o2, o3);
    return __builtin_bit_cast(half8_t, make_uint4(o0, o1, o2, o3));
}

} // namespace

// ---------------------------------------------------------------------------
// B-direct: the waves sit side by side along N, each owning TN weight tiles
// (16 rows each) that it streams from HBM straight into registers and decodes
// there -- a tile slot is exactly the lane's B fragment -- while the BM x 64
// activation tile of a stage is loaded once per workgroup into LDS and read by
// all of them.
//
// FOLD: the workgroup walks every K-split range of its tile in order (the
// grid has no split dimension), each range's chain from zero as a split
// workgroup would run it, and keeps the ranges' sum in split order in a
// second accumulator set; it stores that sum once instead of ksplit partials.
//
// NW: waves per workgroup, side by side along N (BN = 16 TN NW).  All of them
// share one activation tile: the wider the workgroup, the fewer activation
// loads and LDS stores per MFMA.
// Tile pairs by which a tile's scale FMAs trail its MFMA pair (0: right after
// it, where they wait for the matrix core unless other waves fill in), and
// whether the scale is converted once instead of inside every FMA
// (v_fma_mix_f32 takes the fp16 scale as it is but issues slower than a plain
// FMA).  Both are settled per tile by timing, cold weights, 3B projections, us:
//   4 x 2 and 4 x 4 tiles: two pairs; 4 x 2 with plain FMAs but for Q4_0 (Q5_1
//     QKV 1500 rows 160 -> 149, down 236 -> 219, SwiGLU 640 193 -> 178; SwiGLU
//     256 rows Q8_0 81 -> 72, Q5_1 100 -> 84)
//   5 x 2 and 6 x 2 of Q4_0 and Q5_1: one pair.  With two they need 4 to 14
//     registers past the 128 of two workgroups per CU, and the scratch they took
//     cost more than the lag gives (Q5_1 SwiGLU 520 rows 165 -> 145 us; Q4_0 calls
//     of 768 rows: down 106 -> 97, QKV 75 -> 68)
//   2 x 1: two pairs and plain FMAs (Q8_0 QKV 96 rows 14.9 -> 13.9, Q4_0 down
//     20.6 -> 18.6)
//   1 x 1, 1 x 2: one pair (Q8_0 down 32 rows 12.6 -> 11.8, Q5_1 16.3 -> 15.0)
//   2 x 2: neither (two to four waves per SIMD fill in: 160 rows 16.9 -> 17.4
//     with two pairs), except Q5_1 at four waves per SIMD, where they leave
//     room in its 128 registers (SwiGLU 200 rows 97 -> 68)
constexpr int bd_lag(int type, int tm, int tn, int nw)
{
    if (tm >= 5 && type != kQ8_0) return 1;
    return tm * tn >= 8 || (tm == 2 && tn == 1) || (type == kQ5_1 && nw >= 14) ? 2 : tm == 1 ? 1 : 0;
}
constexpr bool bd_plain_scale(int type, int tm, int tn, int nw)
{
    return (tm == 2 && tn == 1) || (tm * tn == 8 && type != kQ4_0) || (type == kQ5_1 && nw >= 14);
}

template <int TYPE, int MODE, int TM, int TN, int PD, int OCC, bool FOLD = false, int NW = 4>
__global__ __launch_bounds__(64 * NW, OCC) void gemm_bd_kernel(GemmArgs a, int mt, int nt, int gm)
{
    constexpr int BM = 16 * TM, BN = 16 * TN * NW;
    constexpr int U = PD + 1; // weight register ring
    static_assert(!FOLD || MODE == kGemmStore, "folded K splits are a store-mode form");
    __shared__ __attribute__((aligned(16))) uint16_t As[2][TM * 4 * 512]; // [mi][block][part] operand tiles

    // ---- tile of this workgroup (per-XCD runs of a grouped order; K split z = whole runs of it)
    const int total = gridDim.x;
    const int per_xcd = total >> 3;
    const int L = blockIdx.x;
    int Lp = (L & 7) * per_xcd + (L >> 3);
    const int tiles8 = FOLD ? total : total / a.ksplit;
    const int z = FOLD ? 0 : Lp / tiles8;
    Lp -= z * tiles8;
    const int group = gm * nt;
    const int first_m = (Lp / group) * gm;
    const int gsz = min(mt - first_m, gm);
    if (gsz <= 0) return;
    const int tile_m = first_m + (Lp % group) % gsz;
    const int tile_n = (Lp % group) / gsz;
    if (tile_m >= mt || tile_n >= nt) return;

    // wave-uniform in a scalar register: the activation loads' scalar offset
    // depends on it, and a vector one would make the compiler wrap each load in
    // a one-pass loop that drains every outstanding load at the next wait
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = a.M, K = a.K, nblk = K >> 5;
    const int nb_per = gemm_split_blocks(nblk, a.ksplit);
    const int kb_begin = z * nb_per;
    const int nb = FOLD ? nblk : min(nblk - kb_begin, nb_per); // blocks this workgroup walks
    const int nstage = (nb + 1) >> 1;
    const int m0 = tile_m * BM;

    // ---- activation loader: the stage's TM * 4 fragments (row group mi,
    // block f >> 1, part f & 1 for fragment 4 mi + f) of 1 KiB go to the waves
    // round robin, wave w taking fragments w, w + NW, ...; each lane loads its
    // 16-byte slot.  With four waves, wave w takes fragment f = w of every row
    // group.  Past the last fragment a wave repeats it (the same bytes to the
    // same LDS slot).
    const int rg_last = (M - 1) >> 4; // groups past M feed unstored rows
    const rsrc_t ra = make_rsrc(a.xt, (uint32_t)(rg_last + 1) * nblk * 2048);
    constexpr int NCH = TM * 4, AL = (NCH + NW - 1) / NW;
    int ach[AL], abb[AL];
    uint32_t va[AL];
#pragma unroll
    for (int j = 0; j < AL; j++) {
        // four waves: fragment `wave` of row group j (block and part are the wave's for every j)
        const int ch = NW == 4 ? 4 * j + wave : min(wave + NW * j, NCH - 1);
        const int mi = NW == 4 ? j : ch >> 2, part = NW == 4 ? wave & 1 : ch & 1;
        ach[j] = ch;
        abb[j] = NW == 4 ? wave >> 1 : (ch >> 1) & 1;
        va[j] = (((uint32_t)min((m0 >> 4) + mi, rg_last) * nblk * 2 + part) * 512 + lane * 8) * 2;
    }
    // Q5_1 block sums of the stage's BM rows x 2 blocks, one per thread of the
    // first 2 * BM, staged through LDS with the activations.  The block index
    // rides in the per-thread offset so the scalar offset stays uniform; the
    // other threads read past the buffer (zeros).  A missing odd last block
    // reads a finite neighbour that its zero min cancels.
    __shared__ __attribute__((aligned(16))) float Xs[2][TYPE == kQ5_1 ? 64 * NW : 4]; // [bb * BM + row], the rest unused
    rsrc_t rs;
    uint32_t vx = 0;
    if (TYPE == kQ5_1) {
        rs = make_rsrc(a.xsum, (uint32_t)M * nblk * 4);
        vx = tid < 2 * BM ? ((uint32_t)(m0 + tid % BM) * nblk + tid / BM) * 4 : 0x40000000u;
    }
    struct AStage {
        uint4 v[AL];
        float xs;
    };
    auto load_a = [&](int st, AStage &r) __attribute__((always_inline)) {
        st = min(st, nstage - 1);
#pragma unroll
        for (int j = 0; j < AL; j++) {
            const int kblk = kb_begin + min(2 * st + (NW == 4 ? abb[0] : abb[j]), nb - 1);
            r.v[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ra, va[j], kblk * 2048, 0));
        }
        if (TYPE == kQ5_1) r.xs = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, vx, (kb_begin + 2 * st) * 4, 0));
    };
    auto store_a = [&](int buf, const AStage &r) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < AL; j++) *(uint4 *)&As[buf][(NW == 4 ? j * 4 + wave : ach[j]) * 512 + lane * 8] = r.v[j];
        if (TYPE == kQ5_1) Xs[buf][tid] = r.xs;
    };

    // ---- weight loader: tile n of this wave is tile row wave * TN + n of the workgroup
    constexpr bool BQ = kByteQuants<TYPE>;
    rsrc_t rq[TN], rd[TN];
    int btile0[TN];
    const uint32_t vq = (uint32_t)lane * (BQ ? 16 : 8), vd = 4 * (lane & 15);
#pragma unroll
    for (int n = 0; n < TN; n++) {
        const int t = wave * TN + n;
        int seg, rgw;
        if (MODE == kGemmSwiGlu) {
            seg = t & 1; // 16-row groups alternate gate and up
            rgw = tile_n * (BN / 32) + (t >> 1);
        } else {
            // the segment of the workgroup's tile (four waves: a tile never
            // straddles two) or of this wave's 16 TN rows (which never do)
            int s0 = 0, start = 0;
            const int r0 = tile_n * BN + (NW == 4 ? 0 : 16 * t);
            while (s0 + 1 < a.nseg && r0 >= start + a.seg[s0].rows) {
                start += a.seg[s0].rows;
                s0++;
            }
            seg = s0;
            rgw = (r0 - start) / 16 + (NW == 4 ? t : 0);
        }
        seg = __builtin_amdgcn_readfirstlane(seg);
        const QWeight &w = a.seg[seg];
        const int KP = tile_kpairs(w.cols), RG = tile_rows(w.rows);
        const uint32_t tiles = (uint32_t)RG * KP;
        rq[n] = quant_rsrc<TYPE>(w, tiles);
        rd[n] = make_rsrc(w.d, tiles * tile_d_bytes(TYPE));
        btile0[n] = __builtin_amdgcn_readfirstlane(min(rgw, RG - 1) * KP + (kb_begin >> 1));
    }
    auto load_b = [&](int st, BChunk (&br)[TN]) __attribute__((always_inline)) {
        st = min(st, nstage - 1);
#pragma unroll
        for (int n = 0; n < TN; n++) {
            const int tile = btile0[n] + st;
            if (BQ) {
                br[n].q = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rq[n], vq, tile * 1024, 0));
            } else {
                uint2 v = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rq[n], vq, tile * 512, 0));
                br[n].q = make_uint4(v.x, v.y, 0u, 0u);
            }
            if (TYPE == kQ5_1) {
                const uint2 dm = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rd[n], 2 * vd, tile * 128, 0));
                br[n].d = dm.x;
                br[n].m = dm.y;
            } else {
                br[n].d = __builtin_amdgcn_raw_buffer_load_b32(rd[n], vd, tile * 64, 0);
            }
        }
    };

    floatx4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    // FOLD: the finished ranges' sum in split order; a range of spr stages ends
    // after stage done - 1 when done is a multiple of spr
    floatx4 tot[FOLD ? TM : 1][FOLD ? TN : 1];
    const int spr = nb_per >> 1;
    auto fold_range = [&](int done) __attribute__((always_inline)) {
        if constexpr (FOLD) {
            if (done % spr != 0 || done >= nstage) return;
            const bool first = done == spr;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
#pragma unroll
                    for (int r = 0; r < 4; r++) tot[i][j][r] = first ? acc[i][j][r] : tot[i][j][r] + acc[i][j][r];
                    acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                }
        }
    };

    // Each accumulator takes its blocks' FMAs in block order whatever the lag
    // is, so the arithmetic is that of the plain order.
    auto compute = [&](int st, int buf, const BChunk (&br)[TN]) __attribute__((always_inline)) {
        const bool second = 2 * st + 1 < nb;
        constexpr int LAG = bd_lag(TYPE, TM, TN, NW), NQ = 2 * TM * TN;
        floatx4 pq[LAG > 0 ? LAG : 1], xq[LAG > 0 ? LAG : 1];
        float dq[LAG > 0 ? LAG : 1], mq[LAG > 0 ? LAG : 1];
        auto apply = [&](int t) __attribute__((always_inline)) {
            const int mt_ = (t / TN) % TM, nt_ = t % TN, k = LAG > 0 ? t % LAG : 0;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float v = fmaf(dq[k], pq[k][r], acc[mt_][nt_][r]);
                if (TYPE == kQ5_1) v = fmaf(mq[k], xq[k][r], v);
                acc[mt_][nt_][r] = v;
            }
        };
#pragma unroll
        for (int bb = 0; bb < 2; bb++) {
            // an odd block count's missing second block adds 0 * p (p is finite)
            // (a mask rather than a select: the compiler turns a select on a
            // uniform condition into branches around the conversions)
            const uint32_t live = bb == 0 || second ? ~0u : 0u;
            half8_t bf[TN];
            float dv[TN], mv[TN];
#pragma unroll
            for (int n = 0; n < TN; n++) {
                bf[n] = decode_b_frag<TYPE>(br[n], bb);
                dv[n] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, h2f((uint16_t)(bb ? br[n].d >> 16 : br[n].d))) & live);
                if (TYPE == kQ5_1)
                    mv[n] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, h2f((uint16_t)(bb ? br[n].m >> 16 : br[n].m))) & live);
                if constexpr (bd_plain_scale(TYPE, TM, TN, NW)) {
                    asm("" : "+v"(dv[n])); // not foldable into the FMAs
                    if (TYPE == kQ5_1) asm("" : "+v"(mv[n]));
                }
            }
#pragma unroll
            for (int mi = 0; mi < TM; mi++) {
                const half8_t ah = *(const half8_t *)&As[buf][(mi * 4 + bb * 2 + 0) * 512 + lane * 8];
                const half8_t al = *(const half8_t *)&As[buf][(mi * 4 + bb * 2 + 1) * 512 + lane * 8];
                floatx4 xs4; // block sums of the lane's four C rows
                if (TYPE == kQ5_1) xs4 = *(const floatx4 *)&Xs[buf][bb * BM + mi * 16 + 4 * (lane >> 4)];
#pragma unroll
                for (int n = 0; n < TN; n++) {
                    floatx4 p = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bf[n], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    p = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bf[n], p, 0, 0, 0);
                    if constexpr (LAG == 0) {
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            float v = fmaf(dv[n], p[r], acc[mi][n][r]);
                            if (TYPE == kQ5_1) v = fmaf(mv[n], xs4[r], v);
                            acc[mi][n][r] = v;
                        }
                    } else {
                        const int q = (bb * TM + mi) * TN + n;
                        if (q >= LAG) apply(q - LAG);
                        pq[q % LAG] = p;
                        dq[q % LAG] = dv[n];
                        if (TYPE == kQ5_1) {
                            xq[q % LAG] = xs4;
                            mq[q % LAG] = mv[n];
                        }
                        __builtin_amdgcn_sched_group_barrier(0x008, 2, 0); // the pair's MFMAs
                        __builtin_amdgcn_sched_group_barrier(0x002, 6, 0); // then vector work
                    }
                }
            }
        }
        if constexpr (LAG > 0) {
#pragma unroll
            for (int t = NQ - LAG; t < NQ; t++) apply(t);
        }
    };

    // ---- pipeline: weights U stages ahead in a register ring; activations
    // loaded UA stages ahead into a register ring (stage t in slot t % UA)
    // and copied to LDS (double buffered) by the stage before their own.
    // Whole groups of U stages in the loop, the remainder after it: a loop
    // with exits inside its body would merge a half-advanced ring into the
    // loop header, where the compiler would then drain every outstanding load.
    // The prologue issues its loads in the loop's order
    // (activations of stage t + 1, then weights of stage t) so the compiler's
    // wait counts at the loop head, merged over entry and back edge, stay
    // those of the loop.
    // Tall tiles (TM = 4) keep one activation slot: a second would cost the
    // registers of a third resident workgroup.
    constexpr int UA = TM >= 4 ? 1 : U;
    BChunk br[U][TN];
    AStage araw[UA], a0;
    load_a(0, a0);
#pragma unroll
    for (int t = 0; t < U; t++) {
        if (t < UA) load_a(t + 1, araw[(t + 1) % UA]);
        load_b(t, br[t]);
        __builtin_amdgcn_sched_barrier(0);
    }
    store_a(0, a0);
    __syncthreads();
    auto stage = [&](auto jc, int s) __attribute__((always_inline)) {
        constexpr int j = decltype(jc)::value;
        compute(s, s & 1, br[j]);
        fold_range(s + 1);
        store_a((s + 1) & 1, araw[(j + 1) % UA]);
        load_a(s + 1 + UA, araw[(j + 1) % UA]);
        load_b(s + U, br[j]);
        __syncthreads();
        // keep the next stage's decode below the barrier: hoisted above it,
        // it would wait on the weights loaded one stage ago
        __builtin_amdgcn_sched_barrier(0);
    };
    const int ngroups = nstage / U;
    int s0 = 0;
    for (int g = 0; g < ngroups; g++, s0 += U) {
        stage(std::integral_constant<int, 0>{}, s0);
        if constexpr (U > 1) stage(std::integral_constant<int, 1 % U>{}, s0 + 1);
        if constexpr (U > 2) stage(std::integral_constant<int, 2 % U>{}, s0 + 2);
        if constexpr (U > 3) stage(std::integral_constant<int, 3 % U>{}, s0 + 3);
        static_assert(U <= 4, "ring deeper than the unrolled group");
    }
    {
        const int rem = nstage - s0;
        if constexpr (U > 1) if (rem > 0) stage(std::integral_constant<int, 0>{}, s0);
        if constexpr (U > 2) if (rem > 1) stage(std::integral_constant<int, 1 % U>{}, s0 + 1);
        if constexpr (U > 3) if (rem > 2) stage(std::integral_constant<int, 2 % U>{}, s0 + 2);
    }

    if constexpr (FOLD) {
        if (nstage > spr) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][j][r] = tot[i][j][r] + acc[i][j][r];
        }
    }

    // ---- epilogue.  Lane holds C[4*(lane/16) + r][lane % 16] of each 16x16 tile.
    const int row_base = m0 + 4 * (lane >> 4);
    if (MODE == kGemmStore) {
        // columns are the segments' rows concatenated; only the last segment
        // may end inside a tile
        float *y = a.y + (size_t)z * M * a.ldy;
        const int n0 = tile_n * BN;
        int seg = 0, start = 0, end = 0;
        if constexpr (NW == 4) {
            // a four-wave tile lies in one segment
            while (seg + 1 < a.nseg && n0 >= start + a.seg[seg].rows) {
                start += a.seg[seg].rows;
                seg++;
            }
            end = start + a.seg[seg].rows;
        } else {
            for (int i = 0; i < a.nseg; i++) end += a.seg[i].rows;
        }
#pragma unroll
        for (int n = 0; n < TN; n++) {
            const int col = n0 + (wave * TN + n) * 16 + (lane & 15);
            if (col >= end) continue;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int row = row_base + 16 * i + r;
                    if (row < M) __builtin_nontemporal_store(acc[i][n][r], &y[(size_t)row * a.ldy + col]);
                }
        }
    } else {
        const int ld = a.seg[0].rows;
#pragma unroll
        for (int pp = 0; pp < TN / 2; pp++) {
            // tiles 2pp (gate) and 2pp+1 (up) of this wave cover the same outputs
            const int col = tile_n * (BN / 2) + ((wave * TN + 2 * pp) >> 1) * 16 + (lane & 15);
            if (col >= ld) continue;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int row = row_base + 16 * i + r;
                    if (row >= M) continue;
                    // Kernels.SwiGlu (Kernels.cs:82-89): (g*u) * sigmoid(g).
                    const float g = acc[i][2 * pp][r], u = acc[i][2 * pp + 1][r];
                    const float gu = g * u;
                    const float e = expf(-g);
                    const float sg = 1.0f / (1.0f + e);
                    const float v = sg * gu;
                    uint16_t hi, lo;
                    split_f16(v, hi, lo);
                    a.ot[xt_index(row, col, ld >> 5, 0)] = hi;
                    a.ot[xt_index(row, col, ld >> 5, 1)] = lo;
                }
        }
    }
}

// Skinny variant for M <= 16 (one row group: the reasoning decider's rows,
// short branches).  The B-direct grid at such M is N / 128 x splits
// workgroups -- 96 for a 3072-row projection split 4 -- and leaves most of the
// chip's load bandwidth idle.  Here each wave owns TN 16-row weight groups over
// one K split and streams them through its own register ring of CH stages,
// while the activation fragments (and Q5_1 block sums), the same for all waves
// of the workgroup, go through LDS in chunks of CH stages, double buffered,
// one barrier per chunk.
//
// Bound by the chain of one wave's stages (the 3B projections give 0.75 waves
// per SIMD) and, for the vocabulary head, by the weight bytes.  So:
//  * A ring slot holds a stage's weights and this wave's share of the
//    activations CH stages further on, loaded and retired together.  Loads
//    retire in order, so nothing ever waits for a load younger than its own
//    stage; with the activations loaded once per chunk, the wait for them at
//    the chunk's end also drained the weight ring.
//  * Loads stay at the end of their stage (the sched_barriers): left alone, the
//    compiler sinks them to their use.
//  * LDS reads run one block ahead; for one Q5_1 group per wave the scale FMAs
//    trail their MFMA pair by one block with the scales converted once.  (The
//    other types issue too few vector instructions for that to hide the pair.)
//  * SwiGLU: gate and up in neighbouring waves (GU), twice the waves, the
//    up sums handed over through LDS at the end.
//  * One round of at most 256 workgroups, each as wide as that needs
//    (launch_skinny), since a CU with a second workgroup finishes last.
// 12 rows, cold weights, 3B projections, us, before -> now: Q5_1 QKV 9.3 ->
// 8.3, O 7.4 -> 6.6, gate/up 21.7 -> 19.7, down 12.3 -> 10.4, head 97 -> 72;
// Q8_0 QKV 7.8 -> 6.8, gate/up 19.1 -> 16.0, down 10.0 -> 8.2, head 88 -> 76;
// Q4_0 gate/up 17.1 -> 13.0, head 73 -> 49.
//
// Per output it issues exactly gemm_bd_kernel's sequence: per block p =
// mfma(x_hi, q); p = mfma(x_lo, q, p); acc = fma(d, p, acc) (+ fma(m, sum x,
// acc)), blocks ascending within the split -- so its results are the same bits.
// The missing second block of an odd K reads a finite neighbour's activations
// against the layout's zero scales.
// F5: Q5_1 quants from the 5-bit fields (two thirds of the byte copy's bytes,
// more decode) instead of the byte copy.
template <int TYPE, int MODE, int TN, int NW, bool F5>
__global__ __launch_bounds__(64 * NW, 2) void gemm_skinny_kernel(GemmArgs a, int ngroups, int nq)
{
    constexpr bool GU = MODE == kGemmSwiGlu;
    constexpr int CH = 4;                                    // stages per chunk and ring turn
    constexpr int LAG = TYPE == kQ5_1 && TN == 1 ? 1 : 0;    // blocks the scale FMAs trail
    constexpr int GW = GU ? NW / 2 : NW * TN;                // row groups per workgroup
    static_assert(!GU || (TN == 1 && NW % 2 == 0), "gate and up in neighbouring waves");
    static_assert(CH * 32 <= 64 * NW, "one block sum per thread");
    __shared__ __attribute__((aligned(16))) uint4 As[2][CH * 4 * 64]; // [stage][block][part][lane]
    __shared__ __attribute__((aligned(16))) float Xs[2][TYPE == kQ5_1 ? CH * 2 * 16 : 4]; // [block][row]

    // Every index below is wave-uniform and kept in scalar registers: the
    // integer divisions are vector-ALU sequences, and left as vector values
    // their results would drag all the per-stage address arithmetic onto the
    // vector ALU with the decode and the scale FMAs.
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int z = __builtin_amdgcn_readfirstlane((int)blockIdx.x / nq), q = blockIdx.x - z * nq;
    const int g0 = q * GW + (GU ? wave >> 1 : wave * TN);    // this wave's first row group; past ngroups: loads only
    const int M = a.M, K = a.K, nblk = K >> 5;
    const int nb_per = __builtin_amdgcn_readfirstlane(gemm_split_blocks(nblk, a.ksplit));
    const int kb_begin = z * nb_per;
    const int nb = min(nblk - kb_begin, nb_per);
    const int nstage = __builtin_amdgcn_readfirstlane((nb + 1) >> 1);

    const rsrc_t ra = make_rsrc(a.xt, (uint32_t)nblk * 2048); // row group 0 of the operand tiles
    rsrc_t rs;
    if (TYPE == kQ5_1) rs = make_rsrc(a.xsum, (uint32_t)M * nblk * 4);

    // weights: group n of this wave
    constexpr bool BQ = kByteQuants<TYPE> && !F5;
    rsrc_t rq[TN], rd[TN], rh[TN];
    int btile0[TN];
    const uint32_t vq = (uint32_t)lane * (BQ ? 16 : 8), vd = 4 * (lane & 15), vh = 2 * lane;
#pragma unroll
    for (int n = 0; n < TN; n++) {
        const int gl = min(g0 + n, ngroups - 1);
        int seg, rgw;
        if (GU) {
            seg = wave & 1;
            rgw = gl;
        } else {
            int s0 = 0, start = 0;
            while (s0 + 1 < a.nseg && gl * 16 >= start + a.seg[s0].rows) {
                start += a.seg[s0].rows;
                s0++;
            }
            seg = s0;
            rgw = (gl * 16 - start) / 16;
        }
        seg = __builtin_amdgcn_readfirstlane(seg);
        const QWeight &wt = a.seg[seg];
        const int KP = tile_kpairs(wt.cols), RG = tile_rows(wt.rows);
        const uint32_t tiles = (uint32_t)RG * KP;
        rq[n] = F5 ? make_rsrc(wt.qs, tiles * 512u) : quant_rsrc<TYPE>(wt, tiles);
        rd[n] = make_rsrc(wt.d, tiles * tile_d_bytes(TYPE));
        if (F5) rh[n] = make_rsrc(wt.qh, tiles * 128u);
        btile0[n] = __builtin_amdgcn_readfirstlane(min(rgw, RG - 1) * KP + (kb_begin >> 1));
    }

    // Activation fragment f = block * 2 + part of a stage, one KiB each: wave f
    // takes it (waves past the fourth repeat the last: the same bytes to the
    // same slot); eight waves take half a fragment each.
    auto load_a = [&](int st) __attribute__((always_inline)) -> uint4 {
        st = min(st, nstage - 1);
        const int f = NW == 8 ? wave >> 1 : min(wave, 3);
        const int kblk = kb_begin + min(2 * st + (f >> 1), nb - 1);
        // the offset is wave-uniform; as a vector value it would cost a one-pass loop per load
        const int soff = __builtin_amdgcn_readfirstlane((kblk * 2 + (f & 1)) * 1024);
        if (NW != 8) return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(ra, lane * 16, soff, 0));
        const uint2 v = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(ra, (wave & 1) * 512 + lane * 8, soff, 0));
        return make_uint4(v.x, v.y, 0u, 0u);
    };
    auto store_a = [&](int buf, int j, const uint4 &v) __attribute__((always_inline)) {
        if (NW != 8)
            As[buf][(j * 4 + min(wave, 3)) * 64 + lane] = v;
        else
            ((uint2 *)&As[buf][(j * 4 + (wave >> 1)) * 64])[(wave & 1) * 64 + lane] = make_uint2(v.x, v.y);
    };
    // Chunk c's block sums, thread t: block t / 16 of the chunk, row t % 16
    // (the address gemm_bd_kernel reads for that row and block).
    auto load_xs = [&](int c) __attribute__((always_inline)) -> float {
        if (TYPE != kQ5_1) return 0.f;
        // every thread loads (threads past CH * 32 a clamped entry nobody
        // stores): a branch around the load would cost the compiler its count
        // of the loads in flight, and a full drain at each chunk's first stage
        const int e = min(tid, CH * 32 - 1);
        const int bl = e >> 4, st = min(c * CH + (bl >> 1), nstage - 1);
        const uint32_t off = ((uint32_t)(e & 15) * nblk + kb_begin + 2 * st + (bl & 1)) * 4;
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
    };
    auto store_xs = [&](int buf, float v) __attribute__((always_inline)) {
        if (TYPE == kQ5_1 && tid < CH * 32) Xs[buf][tid] = v;
    };
    struct Slot {
        BChunk b[TN];
        uint32_t qh[TN];
        uint4 a;  // of stage st + CH
        float xs; // of the next chunk, in a chunk's first slot
    };
    // Slot of stage s0 + j (s0 a chunk's first stage).  Past the last stage
    // everything repeats it, into slots and buffers nobody reads, so every
    // chunk issues the same loads and the compiler's wait counts hold.
    auto load = [&](int s0, int j, Slot &s) __attribute__((always_inline)) {
        const int st = min(s0 + j, nstage - 1);
#pragma unroll
        for (int n = 0; n < TN; n++) {
            const int tile = __builtin_amdgcn_readfirstlane(btile0[n] + st);
            if (BQ) {
                s.b[n].q = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rq[n], vq, tile * 1024, 0));
            } else {
                uint2 v = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rq[n], vq, tile * 512, 0));
                s.b[n].q = make_uint4(v.x, v.y, 0u, 0u);
            }
            if (TYPE == kQ5_1) {
                const uint2 dm = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rd[n], 2 * vd, tile * 128, 0));
                s.b[n].d = dm.x;
                s.b[n].m = dm.y;
                if (F5) s.qh[n] = __builtin_amdgcn_raw_buffer_load_b16(rh[n], vh, tile * 128, 0);
            } else {
                s.b[n].d = __builtin_amdgcn_raw_buffer_load_b32(rd[n], vd, tile * 64, 0);
            }
        }
        s.a = load_a(s0 + j + CH);
        if (TYPE == kQ5_1 && j == 0) s.xs = load_xs(s0 / CH + 1);
    };

    floatx4 acc[TN];
#pragma unroll
    for (int n = 0; n < TN; n++) acc[n] = floatx4{0.f, 0.f, 0.f, 0.f};
    struct Frag {
        half8_t ah, al;
        floatx4 xs; // block sums of the lane's four C rows
    };
    struct Pair { // a block's unscaled products and what scales them
        floatx4 p, xs;
        float d, m;
    };
    auto read = [&](int buf, int i, Frag &f) __attribute__((always_inline)) {
        f.ah = __builtin_bit_cast(half8_t, As[buf][(i * 2 + 0) * 64 + lane]);
        f.al = __builtin_bit_cast(half8_t, As[buf][(i * 2 + 1) * 64 + lane]);
        if (TYPE == kQ5_1) f.xs = *(const floatx4 *)&Xs[buf][i * 16 + 4 * (lane >> 4)];
    };
    auto apply = [&](int n, const Pair &t) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float v = fmaf(t.d, t.p[r], acc[n][r]);
            if (TYPE == kQ5_1) v = fmaf(t.m, t.xs[r], v);
            acc[n][r] = v;
        }
    };
    Pair late;
    // block bb of the slot's stage; first: nothing trails it yet
    auto block = [&](const Frag &f, const Slot &s, int bb, bool first) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < TN; n++) {
            half8_t bf;
            if constexpr (F5)
                bf = decode_q5_frag(bb ? s.b[n].q.y : s.b[n].q.x, s.qh[n], bb);
            else
                bf = decode_b_frag<TYPE>(s.b[n], bb);
            Pair t;
            t.d = h2f((uint16_t)(bb ? s.b[n].d >> 16 : s.b[n].d));
            if (TYPE == kQ5_1) {
                t.m = h2f((uint16_t)(bb ? s.b[n].m >> 16 : s.b[n].m));
                t.xs = f.xs;
            }
            if constexpr (LAG > 0) {
                asm("" : "+v"(t.d)); // not foldable into the FMAs
                asm("" : "+v"(t.m));
            }
            t.p = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.ah, bf, floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            t.p = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.al, bf, t.p, 0, 0, 0);
            if constexpr (LAG > 0) {
                if (!first) apply(n, late);
                late = t;
            } else {
                apply(n, t);
            }
        }
    };

    // ---- pipeline
    Slot ring[CH];
    {
        uint4 a0[CH];
        const float x0 = load_xs(0);
#pragma unroll
        for (int j = 0; j < CH; j++) a0[j] = load_a(j);
#pragma unroll
        for (int j = 0; j < CH; j++) {
            load(0, j, ring[j]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < CH; j++) store_a(0, j, a0[j]);
        store_xs(0, x0);
    }
    const int nfull = nstage / CH;
    for (int c = 0; c < nfull; c++) {
        const int buf = c & 1;
        __syncthreads(); // chunk c staged by everyone; chunk c - 1's buffer is free
        __builtin_amdgcn_sched_barrier(0);
        Frag fr[2];
        read(buf, 0, fr[0]);
#pragma unroll
        for (int j = 0; j < CH; j++) {
#pragma unroll
            for (int bb = 0; bb < 2; bb++) {
                const int i = 2 * j + bb;
                if (i + 1 < 2 * CH) read(buf, i + 1, fr[(i + 1) & 1]);
                block(fr[i & 1], ring[j], bb, i == 0);
            }
            store_a(buf ^ 1, j, ring[j].a);
            if (j == 0) store_xs(buf ^ 1, ring[j].xs);
            load((c + 1) * CH, j, ring[j]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (LAG > 0) apply(0, late);
    }
    {
        const int rem = nstage - nfull * CH, buf = nfull & 1; // the last stages
        if (rem > 0) {
            __syncthreads();
#pragma unroll
            for (int j = 0; j < CH - 1; j++) {
                if (j < rem) {
                    Frag f0, f1;
                    read(buf, 2 * j, f0);
                    read(buf, 2 * j + 1, f1);
                    block(f0, ring[j], 0, true);
                    block(f1, ring[j], 1, false);
                    if constexpr (LAG > 0) apply(0, late);
                }
            }
        }
    }

    // ---- epilogue.  Lane holds C[4*(lane/16) + r][lane % 16].
    const int row_base = 4 * (lane >> 4);
    if (MODE == kGemmStore) {
#pragma unroll
        for (int n = 0; n < TN; n++) {
            // columns are the segments' rows concatenated; only the last
            // segment may end inside a group
            const int col = (g0 + n) * 16 + (lane & 15);
            int end = 0;
            for (int i = 0; i < a.nseg; i++) end += a.seg[i].rows;
            if (col >= end) continue;
            float *y = a.y + (size_t)z * M * a.ldy + col;
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (row_base + r < M) __builtin_nontemporal_store(acc[n][r], &y[(size_t)(row_base + r) * a.ldy]);
        }
    } else {
        constexpr int NG = NW / 2; // row groups of the workgroup
        const int ld = a.seg[0].rows;
        floatx4 *up = (floatx4 *)&As[0][0];   // [group][lane]
        float *es = (float *)&As[1][0];       // [row][column of the workgroup's]: hi + lo of each output
        static_assert(NG * 64 <= CH * 4 * 64 && 16 * NG * 16 <= CH * 4 * 64 * 4, "the exchange fits the staging buffers");
        __syncthreads(); // everyone is done with the staging buffers
        if (wave & 1) up[(wave >> 1) * 64 + lane] = acc[0];
        __syncthreads();
        if (!(wave & 1)) {
            const floatx4 u4 = up[(wave >> 1) * 64 + lane];
            const int col = g0 * 16 + (lane & 15);
            const bool live = g0 < ngroups && col < ld;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = row_base + r;
                // Kernels.SwiGlu (Kernels.cs:82-89): (g*u) * sigmoid(g).
                const float gv = acc[0][r], u = u4[r];
                const float gu = gv * u;
                const float e = expf(-gv);
                const float sg = 1.0f / (1.0f + e);
                const float v = sg * gu;
                uint16_t hi, lo;
                split_f16(v, hi, lo);
                if (live && row < M) {
                    a.ot[xt_index(row, col, ld >> 5, 0)] = hi;
                    a.ot[xt_index(row, col, ld >> 5, 1)] = lo;
                }
                if (a.osum) es[row * 16 * NG + (wave >> 1) * 16 + (lane & 15)] = h2f(hi) + h2f(lo);
            }
        }
        if (NG % 2 == 0 && a.osum) {
            // the Q5_1 block sums of these outputs for the down projection: an
            // even number of row groups is whole blocks of consecutive columns
            // (ld is a multiple of 32), each summed in ascending column order
            // as the block-sum kernel sums an operand tile
            __syncthreads();
            const int row = tid & 15, blk = tid >> 4, c0 = q * 16 * NG + 32 * blk;
            if (tid < 8 * NG && row < M && c0 < ld) {
                float sum = 0.f;
                for (int j = 0; j < 32; j++) sum += es[row * 16 * NG + 32 * blk + j];
                a.osum[(size_t)row * (ld >> 5) + (c0 >> 5)] = sum;
            }
        }
    }
}

template <int TYPE, int MODE, int TN, int NW, bool F5 = false>
static hipError_t launch_skinny_cfg(const GemmArgs &a, int ngroups, hipStream_t s)
{
    constexpr int GW = MODE == kGemmSwiGlu ? NW / 2 : NW * TN;
    const int nq = (ngroups + GW - 1) / GW;
    launch_stamped(a.ev_start, a.ev_stop, gemm_skinny_kernel<TYPE, MODE, TN, NW, F5>, dim3(nq * a.ksplit), dim3(64 * NW), 0,
                   s, a, ngroups, nq);
    return hipGetLastError();
}

// As many waves per workgroup as one round of workgroups needs (12 rows, us,
// 4 / 6 / 8 waves): Q8_0 store 16384 columns 12.8 / 14.1 / 16.4, 24576 20.5 /
// 16.5 / 17.4, 32768 23.4 / 27.0 / 21.4; SwiGLU of 4096 outputs 10.0 / 12.1 /
// 12.3, of 9216 19.2 / 16.0 / 18.2 (with the block sums, which take whole
// blocks of columns, four or eight).  Past eight waves' one round, two groups
// per wave share their activation reads (40960 columns: 28.4, one group 31.3
// at best); from a full round of those on, Q5_1 is short of bytes rather than
// of vector issue and reads the 5-bit fields (65536 columns 37.9 against 42.4
// for the byte copy, 49152 39.0 against 34.4).
template <int TYPE, int MODE>
static hipError_t launch_skinny(const GemmArgs &a, hipStream_t s)
{
    if (MODE == kGemmSwiGlu) {
        const int ngroups = a.seg[0].rows / 16;
        if (ngroups <= 2 * kCUs) return launch_skinny_cfg<TYPE, MODE, 1, 4>(a, ngroups, s);
        if (ngroups <= 3 * kCUs && !a.osum) return launch_skinny_cfg<TYPE, MODE, 1, 6>(a, ngroups, s);
        return launch_skinny_cfg<TYPE, MODE, 1, 8>(a, ngroups, s);
    }
    // every segment but the last is a whole number of 16-row groups
    int ntot = 0;
    for (int i = 0; i < a.nseg; i++) ntot += a.seg[i].rows;
    const int ngroups = (ntot + 15) / 16;
    auto fits = [&](int gw) { return (ngroups + gw - 1) / gw * a.ksplit <= kCUs; };
    if (fits(4)) return launch_skinny_cfg<TYPE, kGemmStore, 1, 4>(a, ngroups, s);
    if (fits(6)) return launch_skinny_cfg<TYPE, kGemmStore, 1, 6>(a, ngroups, s);
    if (fits(8)) return launch_skinny_cfg<TYPE, kGemmStore, 1, 8>(a, ngroups, s);
    if constexpr (TYPE == kQ5_1)
        if ((ngroups + 15) / 16 * a.ksplit >= kCUs) return launch_skinny_cfg<TYPE, kGemmStore, 2, 8, true>(a, ngroups, s);
    return launch_skinny_cfg<TYPE, kGemmStore, 2, 8>(a, ngroups, s);
}

// gm_cap: M tiles per group of the tile order (the tiles of a group that share
// an N column run on one XCD, so its L2 serves their common weight tile).
template <int TYPE, int MODE, int TM, int TN, int PD, int OCC, bool FOLD = false, int NW = 4>
static hipError_t launch_bd(const GemmArgs &a, hipStream_t s, int gm_cap = 8)
{
    constexpr int BM = 16 * TM, BN = 16 * TN * NW;
    static_assert(MODE != kGemmSwiGlu || TN % 2 == 0, "SwiGLU pairs tiles within a wave");
    int mt = (a.M + BM - 1) / BM;
    int ncols;
    if (MODE == kGemmSwiGlu) {
        ncols = (a.seg[0].rows + BN / 2 - 1) / (BN / 2);
    } else {
        int ntot = 0;
        for (int i = 0; i < a.nseg; i++) ntot += a.seg[i].rows;
        ncols = (ntot + BN - 1) / BN;
    }
    int gm = mt <= gm_cap ? mt : gm_cap;
    int tiles = mt * ncols;
    int grid = ((tiles + 7) & ~7) * (FOLD ? 1 : a.ksplit);
    launch_stamped(a.ev_start, a.ev_stop, gemm_bd_kernel<TYPE, MODE, TM, TN, PD, OCC, FOLD, NW>, dim3(grid), dim3(64 * NW), 0, s,
                   a, mt, ncols, gm);
    return hipGetLastError();
}

// Tile choice.  It only changes which rows and columns share a workgroup,
// never a result bit.  What bounds these grids below ~700 rows is the busiest
// compute unit: each wave's K stage costs about the same whatever runs beside
// it (its MFMAs, the scale FMAs and the decode share one issue port), every
// workgroup stages its own copy of the activation tile, and a second workgroup
// on a few of the 256 compute units doubles the launch.  So the workgroup is
// made just wide enough that the grid is one round -- one workgroup per
// compute unit, all of its waves sharing one activation tile -- and no wider
// (a wave's share grows with the width).  Cold weights, 3B projections, in us,
// four-wave 32 x 128 tiles (225..256 rows: twelve-wave) against these:
//   Q8_0 QKV     32 rows 13.1 -> 9.4    64 13.3 -> 11.8   96 17.1 -> 14.6
//               160 rows 18.0 -> 16.9  224 23.7 -> 21.6  320 33.3 -> 29.4
//               512 rows 46.9 -> 44.0  640 (64 x 256) 55.5 -> 52.2
//   Q5_1 down    32 rows 23.5 -> 15.8  128 33.5 -> 26.1  320 57.6 -> 52.2
//               640 rows 111.9 -> 95.3, 1500 266 -> 232, 4528 665 -> 634
//   Q8_0 SwiGLU  32 rows 29.2 -> 24.7   48 35.0 -> 25.0   96 35.8 -> 29.4
//               128 rows 46.6 -> 35.9  192 62.1 -> 51.8  256 74.2 -> 69.7
//               320 rows 89.5 -> 83.4  448 117 -> 101

template <int TYPE, int MODE>
static hipError_t launch_mode(const GemmArgs &a, hipStream_t s)
{
    // One row group (the reasoning decider's rows, short branches): one wave
    // per weight row group, 1.5-2x the B-direct kernel there (12 rows of the
    // Q5_1 3B shape: 2.1 against 3.6 ms of GEMM per step)
    if (a.M <= 16) return launch_skinny<TYPE, MODE>(a, s);
    int tcols;           // 16-wide tile columns of the output (gate and up both count)
    bool one_seg = true; // a four-wave tile of 128 or 256 columns lies in one segment
    if (MODE == kGemmSwiGlu) {
        tcols = 2 * (a.seg[0].rows / 16);
    } else {
        int ntot = 0;
        for (int i = 0; i < a.nseg; i++) ntot += a.seg[i].rows;
        for (int i = 0; i + 1 < a.nseg; i++) one_seg = one_seg && a.seg[i].rows % 256 == 0;
        tcols = (ntot + 15) / 16;
    }
    // workgroups of a grid of 16 tm x 16 tn nw tiles
    auto wgs = [&](int tm, int tn, int nw) {
        return (long)((a.M + 16 * tm - 1) / (16 * tm)) * ((tcols + tn * nw - 1) / (tn * nw)) * a.ksplit;
    };
    if constexpr (MODE == kGemmSwiGlu) {
        if (a.M <= 512) {
            if (wgs(1, 2, 8) <= kCUs) return launch_bd<TYPE, MODE, 1, 2, 1, 1, false, 8>(a, s, 4);
            if (wgs(2, 2, 8) <= kCUs) return launch_bd<TYPE, MODE, 2, 2, 1, 1, false, 8>(a, s, 4);
            if (wgs(2, 2, 10) <= kCUs) return launch_bd<TYPE, MODE, 2, 2, 1, 1, false, 10>(a, s, 4);
            if (wgs(2, 2, 12) <= kCUs) return launch_bd<TYPE, MODE, 2, 2, 1, 1, false, 12>(a, s, 4);
            if (wgs(2, 2, 14) <= kCUs) return launch_bd<TYPE, MODE, 2, 2, 1, 1, false, 14>(a, s, 4);
            if (wgs(2, 2, 16) <= kCUs) return launch_bd<TYPE, MODE, 2, 2, 1, 1, false, 16>(a, s, 4);
            // 64-row tiles (half the decode per MFMA) where their grid nearly
            // fills the round; nine waves only when the last tile is more than
            // half full (208 rows of Q5_1: 76 -> 86 us)
            long g = wgs(4, 2, 9);
            if (g <= kCUs && g > kCUs * 7 / 8 && (a.M - 1) % 64 >= 32) return launch_bd<TYPE, MODE, 4, 2, 1, 1, false, 9>(a, s);
            g = wgs(4, 2, 12);
            if (g <= kCUs && g > kCUs * 7 / 8) return launch_bd<TYPE, MODE, 4, 2, 1, 1, false, 12>(a, s);
            g = wgs(4, 2, 8);
            if (g <= 2 * kCUs && g > kCUs * 3 / 2) return launch_bd<TYPE, MODE, 4, 2, 1, 1, false, 8>(a, s); // two per CU
            // no width fits: four-wave tiles built for five resident
            // workgroups per CU (80 VGPRs), in groups of 4 M tiles
            return launch_bd<TYPE, MODE, 2, 2, 1, 5>(a, s, 4);
        }
    } else if (a.M <= 512) {
        // (up to 2.25 of these short workgroups per CU beat wider ones: 48 rows of QKV, Q8_0 11.7 -> 10.8 us, Q4_0 12.4 -> 11.3)
        if (wgs(1, 1, 4) <= kCUs * 9 / 4) return launch_bd<TYPE, MODE, 1, 1, 1, 4>(a, s);
        if (wgs(2, 1, 8) <= kCUs) return launch_bd<TYPE, MODE, 2, 1, 1, 1, false, 8>(a, s);
        if (wgs(2, 1, 12) <= kCUs) return launch_bd<TYPE, MODE, 2, 1, 1, 1, false, 12>(a, s);
        if (wgs(2, 2, 8) <= kCUs) return launch_bd<TYPE, MODE, 2, 2, 1, 1, false, 8>(a, s);
        if (wgs(2, 2, 12) <= kCUs) return launch_bd<TYPE, MODE, 2, 2, 1, 1, false, 12>(a, s);
        // two or three per CU, eight waves of 32 rows (Q5_1, whose second FMA per
        // output favours fewer columns: 64 rows of half the width) unless
        // four-wave workgroups leave the busiest CU fewer waves (400 rows of
        // Q4_0 QKV 43.6 -> 41.1 us; equal counts go to the wider one, 457
        // rows 47.3 -> 44.7)
        const long wide = TYPE == kQ5_1 ? wgs(4, 1, 8) : wgs(2, 2, 8);
        if ((wgs(2, 2, 4) + kCUs - 1) / kCUs < 2 * ((wide + kCUs - 1) / kCUs)) return launch_bd<TYPE, MODE, 2, 2, 1, 4, false, 4>(a, s);
        if constexpr (TYPE == kQ5_1) return launch_bd<TYPE, MODE, 4, 1, 1, 1, false, 8>(a, s);
        return launch_bd<TYPE, MODE, 2, 2, 1, 1, false, 8>(a, s);
    }
    // Large batches, tiles of 256 columns.
    if constexpr (MODE == kGemmStore && TYPE != kQ5_1)
        if (a.fold) return launch_bd<TYPE, MODE, 4, 4, 1, 2, true>(a, s);
    // The height of the tile by the rounds its grid takes.  Eight waves of 64,
    // 80 or 96 rows x 32 columns (two such workgroups fit a CU) finish when the
    // busiest CU does, so their time is whole workgroups per CU times a
    // workgroup's; four waves of 64 x 64, up to three workgroups at a time, run on
    // through a partial round, and among many rounds, where the power limit sets
    // the clock, are the cheapest per row.  The relative times per workgroup are
    // of kernels between others (us, four waves / 64 rows / 80 / 96): Q8_0 O, 700
    // rows 46.0 / 47.3 / 41.2 / 45.2, 900 49.6 / 50.0 / 59.8 / 48.8, 3000 139.9 /
    // 144.1 / 149.8 / 145.5; Q4_0 O, 700 rows 45.5 / 46.0 / 39.0 / 42.6, 1500 77.0 /
    // 76.2 / 75.3 / 73.6; SwiGLU, 520 rows of Q8_0 133 / 135 / 119 / 131, 900 of Q4_0
    // 214 / 210 / 209 / 187; Q5_1 SwiGLU 700 rows 64 / 80: 212 / 202.  In a
    // single matmul, between a pair split and a sum of partials, a store of 80 rows
    // can be up to 5 % behind the four waves that it is ahead of in a prompt (Q4_0
    // at 1150 rows: QKV 102 against 97, the prompt's four layers 2598 against 2687).
    // Against four waves throughout, four 3B layers take, 700 / 900 / 1500 / 2400
    // rows: Q4_0 1828 -> 1683, 2164 -> 1992, 3176 -> 3120, 5061 -> 5005; Q8_0 1839 ->
    // 1738, 2173 -> 2114, 3228 -> 3212, 5169 -> 5124.  Q5_1 has no registers for 96
    // rows, nor for its byte quants in the four-wave tile.
    constexpr double k80 = MODE == kGemmStore ? 1.28 : 1.24, k96 = 1.41;
    auto rounds = [&](int tm) { return (double)((wgs(tm, 2, 8) + kCUs - 1) / kCUs); };
    double best = rounds(4);
    int tall = 4;
    if (rounds(5) * k80 < best) {
        best = rounds(5) * k80;
        tall = 5;
    }
    if constexpr (TYPE != kQ5_1) {
        if (rounds(6) * k96 < best) {
            best = rounds(6) * k96;
            tall = 6;
        }
        constexpr double k64 = TYPE == kQ4_0 ? 0.96 : MODE == kGemmStore ? 0.90 : 0.95; // four waves
        const double share = (double)wgs(4, 4, 4) / kCUs, r4 = rounds(4);
        const double four = std::min(r4, share + 0.88) * k64;
        if (one_seg && (four < best || (tall == 4 && share > 4)) && (MODE == kGemmSwiGlu || r4 > 2))
            return launch_bd<TYPE, MODE, 4, 4, 1, 2>(a, s);
        if (tall == 6) return launch_bd<TYPE, MODE, 6, 2, 1, 4, false, 8>(a, s);
    }
    if (tall == 5) return launch_bd<TYPE, MODE, 5, 2, 1, 4, false, 8>(a, s);
    return launch_bd<TYPE, MODE, 4, 2, 1, 1, false, 8>(a, s);
}

template <int TYPE>
static hipError_t launch_typed(const GemmArgs &a, hipStream_t s)
{
    if (a.mode == kGemmSwiGlu) return launch_mode<TYPE, kGemmSwiGlu>(a, s);
    return launch_mode<TYPE, kGemmStore>(a, s);
}

hipError_t launch_gemm(const GemmArgs &a, hipStream_t s)
{
    if (a.M <= 0) return hipSuccess;
    if (a.K % 32 != 0 || a.ksplit < 1 || a.ksplit > 8) return hipErrorInvalidValue;
    if (a.ksplit > 1 && (a.mode != kGemmStore || gemm_split_blocks(a.K >> 5, a.ksplit) * (a.ksplit - 1) >= (a.K >> 5)))
        return hipErrorInvalidValue; // every split non-empty; SwiGLU needs whole sums
    for (int i = 0; i < a.nseg; i++) {
        if (a.seg[i].type != a.seg[0].type || a.seg[i].cols != a.K) return hipErrorInvalidValue;
        // every segment but the last is whole four-wave tiles of 64 or 128 columns
        // and whole wave shares of the wider workgroups (256-column four-wave
        // tiles ask for more: one_seg, and the check of the fold below)
        if (a.mode == kGemmStore && i + 1 < a.nseg && a.seg[i].rows % 128 != 0) return hipErrorInvalidValue;
    }
    if (a.mode == kGemmSwiGlu && (a.nseg != 2 || a.seg[0].rows != a.seg[1].rows || a.seg[0].rows % 32 != 0))
        return hipErrorInvalidValue;
    if (a.osum && (a.mode != kGemmSwiGlu || a.M > 16)) return hipErrorInvalidValue; // written by the skinny kernel only
    // the folded form exists for the large-batch store tiles (the caller asks
    // for it exactly when gemm_fold says so)
    if (a.fold && (a.mode != kGemmStore || !gemm_fold(a.seg[0].type, a.M, a.ksplit))) return hipErrorInvalidValue;
    for (int i = 0; a.fold && i + 1 < a.nseg; i++)
        if (a.seg[i].rows % 256 != 0) return hipErrorInvalidValue;
    switch (a.seg[0].type) {
    case kQ8_0: return launch_typed<kQ8_0>(a, s);
    case kQ4_0: return launch_typed<kQ4_0>(a, s);
    case kQ5_1: return launch_typed<kQ5_1>(a, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace jev
