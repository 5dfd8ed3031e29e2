// The direct-to-LDS tile of the int8 matmuls, shared by the plain (matmul_w8a8_dma.hip) and the grouped matmul
// (matmul_w8a8_group.hip).
//
// Built on the two CDNA4 data-movement instructions that remove all register staging:
//
//   * global_load_lds_dwordx4: every lane names a 16-byte global source, the data lands in LDS at
//     (uniform base + lane * 16) without passing through registers and is tracked by vmcnt.  Because the global
//     address is free per lane, the bank-conflict swizzles are applied on the *source* side: the lane that owns LDS
//     slot s fetches the 16 bytes that belong in that slot.
//   * ds_read_b64_tr_b8: a transposing LDS read.  Within 16 lanes, lane l receives byte (l & 7) of the eight 8-byte
//     rows addressed by lanes 2b + (l >> 3), b = 0..7.  Pointing even lanes at columns [c, c+8) and odd lanes at
//     [c+8, c+16) of eight consecutive k rows gives every lane the 8 consecutive k values of column c + l: exactly
//     the MFMA B operand, read from a B tile that is stored in LDS as it is in memory ([k][n], n contiguous).
//
// So the main loop is: DMA loads for the next K step, LDS reads, MFMAs - no VALU work, no LDS writes, no staging
// registers.  A workgroup is 512 lanes (8 wavefronts, two per SIMD, so that one wavefront's LDS / address
// instructions issue under the other's MFMAs) and owns a 256 x 256 tile; a wavefront owns 128 x 64 (4 x 2 MFMA
// blocks of 32x32x32 or 8 x 4 of 16x16x64, 128 accumulator registers).  Two LDS stages of 64 KiB (A 256 x 128 B, B 128 x 256 B) are
// separate arrays so that the compiler can tell that LDS reads of one stage do not depend on DMA writes to the
// other.
//
// LDS layouts (all reads and writes conflict-free, measured at ~220-250 B/clk/CU):
//   A stage: row r = 128 bytes = 8 pieces of 16; piece c is stored at position c ^ ((r >> 1) & 7).
//   B stage: row k = 256 bytes = 16 pieces of 16; piece q is stored at position q ^ (2 * (k & 7)), in the 16x16x64 form
//   also ^ ((k >> 4) & 1).
#pragma once
#include <type_traits>
#include <utility>

#include "matmul_w8a8.h"

namespace ascq {
namespace {

constexpr int kThreads = 512;
constexpr int BK = 128;

// The forms of a tile: its matrix instruction (gemm_dma_form says which one runs where), and whether k may end inside a
// step.  Looking for that step costs about 1 % (600 x 4096 x 4096 43.5 -> 43.9 us), so it is a form of its own.
// kRing: small tiles with a ring of stages (matmul_w8a8_ring.hip), every output; kRingHalf: those to half or bfloat16, one value per
// column and no quant words (a tile is short enough to notice what else its kernel holds: 729 x 4304 x 1152 20.0 us with every output's code).
constexpr int k16 = 16, k32 = 32, k32Ragged = 33, kRing = 64, kRingHalf = 65;
constexpr bool ring_form(int form) { return form == kRing || form == kRingHalf; }

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) const void* gptr_t;
typedef i32x2_t __attribute__((address_space(3)))* lds_v2_t;

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): a loop whose index is a constant expression.
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// 16-bit output of two adjacent columns packed into one dword store.
template <int kOut>
__device__ __forceinline__ uint32_t to_bits16(float v)
{
    if constexpr (kOut == ASCQ_BF16) {
        return f32_to_bf16_bits(v);
    } else {
        return f32_to_half_bits_sat(v);
    }
}

template <bool kBiasPost, bool kGelu>
__device__ __forceinline__ float epi_value(int32_t acc, float chan, float tok, float bias_post)
{
    float v = static_cast<float>(acc) * chan;
    v = v * tok;  // tok is 1.0f without a token scale: an exact identity
    if constexpr (kBiasPost) {
        v = v + bias_post;
    }
    if constexpr (kGelu) {
        v = faster_gelu(v);
    }
    return v;
}

// 256 x 256: wavefronts 2 (M) x 4 (N), 128 x 64 each.  256 x 128: wavefronts 4 (M) x 2 (N), 64 x 64 each (used for the
// last, partially filled round of tiles: half-width tiles finish it in half the time).  128 x 128: 32 x 64 per
// wavefront, 64 KiB of LDS so that two workgroups share a CU; with kSplitK the K range is divided over blockIdx.y and
// the int32 partial tiles go to a workspace [split][m][n] that a second kernel sums (small M: the weights are read
// once, by enough workgroups to fill the chip).
// The body of a workgroup: tile number `bid` (before the XCD remapping) of the launch, K split `bidy`.  The LDS arrays
// are declared by the kernels and handed in, so that one kernel can run tiles of two shapes.
// kBT: B is given as [n][k] (transposed operand): its tile is staged and read exactly like A's, with plain 16-byte
// LDS reads instead of the transposing ones.
// Where a tile lies: rows [row0, row_end) of A and C (row_end clips the tile), columns from n0, the weight matrix it
// multiplies with and the offset of that matrix's per-channel parameters (grouped: those of the tile's group).
struct TilePlace {
    uint32_t row0, row_end, n0;
    const int8_t* b;
    size_t chan_off;
};

// One of the two LDS stages of a tile.  a[0] holds all rows of A, or in the 16x16x64 form those of every wavefront's first
// half (a[1]: its second half): distinct arrays, like the stages themselves.
struct Stage {
    char* a[2];
    char* b;
};

constexpr uint32_t kPastEnd = 0x7FFFFFF0u;  // an offset the buffer range check rejects: zeros arrive, nothing is fetched

// The main loop of a tile.  first(A, B): the first operands of a step into registers; head(A, B): everything of a step
// but its last part, whose operands are in registers when it returns; tail(An, Bn): the last part, while the first
// operands of the next step arrive; last(): the last part of the last step.
// Per K step: head, wait for the next stage's DMA, barrier (every wavefront has the last operands of this stage in
// registers, so the stage is free), DMA of the step after next into this stage, tail: the matrix pipe has work during the
// burst of LDS reads that follows every barrier.  The loop body never branches between two ways of updating the
// accumulators (that would make the compiler shuffle all of them): the steady state always has a next step, the last one
// or two steps are peeled.
// active: not a wavefront whose rows all lie past the end of the tile's group.
template <class Issue, class First, class Head, class Tail, class Last>
__device__ __forceinline__ void gemm_dma_loop(uint32_t steps, bool active, char* A0, char* B0, char* A1, char* B1, Issue&& issue,
                                              First&& first, Head&& head, Tail&& tail, Last&& last)
{
    if (steps != 0) {
        issue(0, A0, B0);
    }
    asm volatile("s_waitcnt vmcnt(0)");
    __syncthreads();
    if (steps > 1) {
        issue(1, A1, B1);
    }
    if (active && steps != 0) {
        first(A0, B0);
    }
    uint32_t s = 0;
    for (; s + 2 < steps; s += 2) {
        if (active) head(A0, B0);
        asm volatile("s_waitcnt vmcnt(0)");
        __syncthreads();
        issue(s + 2, A0, B0);
        if (active) tail(A1, B1);
        if (active) head(A1, B1);
        asm volatile("s_waitcnt vmcnt(0)");
        __syncthreads();
        if (s + 3 < steps) {
            issue(s + 3, A1, B1);
        }
        if (active) tail(A0, B0);
    }
    if (s + 1 < steps) {  // two steps left: this one in stage 0, the last one on its way into stage 1
        if (active) head(A0, B0);
        asm volatile("s_waitcnt vmcnt(0)");
        __syncthreads();
        if (active) tail(A1, B1);
        ++s;
    }
    if (s < steps) {  // the last step: stage 0 for an odd number of steps, stage 1 for an even one
        if (active) {
            head((steps & 1u) ? A0 : A1, (steps & 1u) ? B0 : B1);
            last();
        }
    }
}

// Where piece q of row kb of a [k][BN] B tile lies: at q ^ b_swizzle(kb).  It spreads the 8 rows of a transposing read over half of
// the banks and, in the 16 x 16 forms, the rows 16 further, which are read beside them, over the other half.
template <int BN, bool k16x16>
__device__ __forceinline__ uint32_t b_swizzle(uint32_t kb)
{
    const uint32_t rows = BN == 256 ? 2u * (kb & 7u) : BN == 128 ? 2u * ((kb >> 1) & 3u) : 2u * ((kb >> 2) & 1u);
    return rows ^ (k16x16 ? (kb >> 4) & 1u : 0u);
}

// The body of a tile on v_mfma_i32_16x16x64_i8, 16-bit outputs only.
// wave, lane: of the workgroup; n0: first column; bases(step): where a K step's loads start; load(bases, u, stage): load u
// of the wavefront's kBLoads + kALoads of a step (B, first half of A's rows, second half).
template <int BM, int BN, bool kGrouped, int kB, int kALoads, int kBLoads, class Bases, class Load>
__device__ __forceinline__ void gemm_dma_body16(const GemmParams& p, const TilePlace& at, uint32_t n0, uint32_t steps, uint32_t wave,
                                                uint32_t lane, Bases&& bases, Load&& load, const Stage& S0, const Stage& S1, float* TS)
{
    constexpr bool kBT = kB == 1, kBP = kB == 2;
    constexpr int kWN = BN / 64;            // wavefronts along N
    constexpr int kWM = 8 / kWN;            // wavefronts along M
    constexpr int NA = BM / 16 / kWM;       // 16 x 16 blocks per wavefront along M
    constexpr int NH = NA / 2;              // of which a quarter of a K step multiplies
    constexpr int TJ = 4;                   // and along N
    static_assert(NH >= 1 && NH * 32 * kWM == BM, "tile shape does not fit eight wavefronts");
    const uint32_t wm = wave / kWN, wn = wave % kWN;
    const uint32_t N = p.n, row0 = at.row0, row_end = at.row_end;
    const size_t chan_off = at.chan_off;

    i32x4 acc[NA][TJ];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            acc[i][j] = i32x4{0, 0, 0, 0};
            asm volatile("" : "+v"(acc[i][j]));
        }
    }

    // ---- operands of v_mfma_i32_16x16x64_i8: lane l holds row (column) l % 16 of a block of 16 and 16 consecutive k,
    // 64 ks + 16 (l / 16) .. + 15.  A step is four quarters: quarter q multiplies half q / 2 of the wavefront's rows
    // with the 64 k of sub-step ks = q % 2.  (This form moves half the sums per product that the 32 x 32 x 32 one
    // moves: on random operands, where the power limit sets the clock, a loop of nothing but matrix instructions reaches
    // 4.0 instead of 3.3 POP/s.)
    const uint32_t lc = lane & 15u, lq = lane >> 4;
    uint32_t foff[2], b_base[TJ];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) foff[ks] = lc * 128u + (((4u * ks + lq) ^ (lc >> 1)) << 4);
    if constexpr (kBP) {
        b_base[0] = wn * 8192u + lane * 16u;  // block j of the wavefront is slab 4 wn + j: two tiles of 1 KiB
    } else if constexpr (!kBT) {
        // transposing reads: in 16 lanes, rows bsub of 8 and halves psub of the block's 16 columns
        const uint32_t bsub = lc >> 1, psub = lc & 1u;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            b_base[j] = (16u * lq + bsub) * BN + (((4u * wn + j) ^ b_swizzle<BN, true>(16u * lq + bsub)) << 4) + 8u * psub;
        }
    }
    i32x4 af[2][NH], bf[2][TJ];
    i32x2_t blo;
    constexpr int kBReads = (kBT || kBP) ? TJ : 2 * TJ;  // LDS reads of a sub-step's columns
    auto load_a = [&](const Stage& S, int q, int i) __attribute__((always_inline)) {
        af[q & 1][i] = *reinterpret_cast<const i32x4*>(S.a[q >> 1] + (wm * NH + i) * 2048u + foff[q & 1]);
    };
    auto load_b = [&](const Stage& S, int ks, int r) __attribute__((always_inline)) {
        if constexpr (kBT) {
            bf[ks][r] = *reinterpret_cast<const i32x4*>(S.b + wn * 8192u + r * 2048u + foff[ks]);
        } else if constexpr (kBP) {
            bf[ks][r] = *reinterpret_cast<const i32x4*>(S.b + b_base[0] + r * 2048u + ks * 1024u);
        } else {
            const i32x2_t v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2_t)(S.b + b_base[r >> 1] + ks * (64 * BN) + (r & 1) * (8 * BN)));
            if (r & 1) {
                bf[ks][r >> 1] = i32x4{blo[0], blo[1], v[0], v[1]};
            } else {
                blo = v;
            }
        }
    };
    // Matrix instruction number n of quarter q, written as an instruction that accumulates in place (the compiler's own
    // choice of another destination moves accumulators about).  Its operands come from LDS reads, which the compiler
    // waits for; no vector instruction touches them or the sums inside the loop.
    auto mfma = [&](int q, int n) __attribute__((always_inline)) {
        i32x4& c = acc[(q >> 1) * NH + n / TJ][n % TJ];
        asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(c) : "v"(af[q & 1][n / TJ]), "v"(bf[q & 1][n % TJ]));
    };
    // One quarter: its NH * TJ matrix instructions.  The LDS reads `read(r)`, r < kReads, are spread behind the first ones,
    // so that the others run while the last reads are on their way; the loads `fetch(u)`, u in [kFrom, kTo), behind all.
    // The order is the one written.
    constexpr int kM = NH * TJ;
    auto quarter = [&](auto qq, auto reads, auto&& read, auto from, auto to, auto&& fetch) __attribute__((always_inline)) {
        constexpr int q = decltype(qq)::value, kReads = decltype(reads)::value, kFrom = decltype(from)::value, kCount = decltype(to)::value - kFrom;
        constexpr int kFront = kM >= 8 ? kM / 2 : kM, kPer = (kReads + kFront - 1) / kFront;
        constexpr int kAtOnce = kCount > kM ? (kCount + kM - 1) / kM : 1, kTimes = kCount > 0 ? (kCount + kAtOnce - 1) / kAtOnce : 1;
        constexpr int kEvery = kM / kTimes;
        static_for<kM>([&](auto nn) {
            constexpr int n = decltype(nn)::value;
            mfma(q, n);
            static_for<kPer>([&](auto r) {
                constexpr int i = n * kPer + decltype(r)::value;
                if constexpr (i < kReads) read(i);
            });
            if constexpr (n % kEvery == kEvery - 1) {
                static_for<kAtOnce>([&](auto r) {
                    constexpr int u = n / kEvery * kAtOnce + decltype(r)::value;
                    if constexpr (u < kCount) fetch(kFrom + u);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // Behind it all but the newest kLeft loads of every wavefront have landed, and every wavefront has the operands it asked
    // for in registers.  (Not __syncthreads(): its fence waits for every load.)
    auto arrive = [&](auto left) __attribute__((always_inline)) {
        constexpr int kLeft = decltype(left)::value;
        __builtin_amdgcn_s_waitcnt(0x0070 | (kLeft & 15) | ((kLeft >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // the operands that quarter 0 of a K step and quarter 1 read first
    auto first_operands = [&](const Stage& S, int i) __attribute__((always_inline)) {
        constexpr int kFirst = kBReads / TJ;  // reads of the first block of columns
        if (i < kFirst || i >= kFirst + NH) {
            load_b(S, 0, i < kFirst ? i : i - NH);
        } else {
            load_a(S, 0, i - kFirst);
        }
    };
    auto second_operands = [&](const Stage& S, int i) __attribute__((always_inline)) {
        if (i < kBReads) {
            load_b(S, 1, i);
        } else {
            load_a(S, 1, i - kBReads);
        }
    };
    // A K step in stage X, the next one in Y, the one after it on its way into X where `fetches`.  B and the first half of
    // A's rows have been read when quarter 1 begins, the second half when quarter 3 begins: a barrier there, and the loads
    // of the step after next go out behind it.  So a load has one and a half K steps to arrive, and is issued behind a
    // matrix instruction of its own (all of a step's loads behind one barrier per step: 2048 x 4096 x 11008 with the quantiser 94.7 us, 88.2
    // like this; 2048 x 8192 x 28672 378 and 361; 256 x 256 tiles on operands of zeros, where the power limit is not met,
    // 8192 x 4096 x 11008 256 and 238).  The counts are the loads issued behind the one that is waited for.
    constexpr int kLoads = kBLoads + kALoads, kMid = kBLoads + kALoads / 2;
    static_assert(kALoads % 2 == 0, "the halves of A's rows are whole loads");
    auto step = [&](const Stage& X, const Stage& Y, uint32_t fetched, auto fetches, auto more, auto works) __attribute__((always_inline)) {
        constexpr bool kFetch = decltype(fetches)::value, kMore = decltype(more)::value, kWorks = decltype(works)::value;
        constexpr std::integral_constant<int, 0> zero{};
        constexpr std::integral_constant<int, kFetch ? kMid : 0> mid{};
        constexpr std::integral_constant<int, kFetch ? kLoads : 0> end{};
        auto work = [&](auto q, auto reads, auto&& read, auto from, auto to, auto&& fetch) __attribute__((always_inline)) {
            if constexpr (kWorks) {
                quarter(q, reads, read, from, to, fetch);
            } else {
                static_for<decltype(to)::value - decltype(from)::value>([&](auto u) { fetch(decltype(from)::value + decltype(u)::value); });
            }
        };
        // Re-materialise the bases inside the loop body: the constant parts of every address then fold into the
        // 16-bit offset field of the DS instructions instead of being hoisted into dozens of registers.
#pragma unroll
        for (int q = 0; q < 2; ++q) asm volatile("" : "+v"(foff[q]));
        if constexpr (!kBT) {
#pragma unroll
            for (int j = 0; j < (kBP ? 1 : TJ); ++j) asm volatile("" : "+v"(b_base[j]));
        }
        constexpr std::integral_constant<int, NH> half{};
        constexpr std::integral_constant<int, NH + kBReads> whole{};
        work(zero, whole, [&](int i) __attribute__((always_inline)) { second_operands(X, i); }, zero, zero, [](int) {});
        arrive(std::integral_constant<int, kMore ? kLoads : 0>{});
        const auto from = bases(fetched);
        auto fetch = [&](int u) __attribute__((always_inline)) { load(from, u, X); };
        work(std::integral_constant<int, 1>{}, half, [&](int i) __attribute__((always_inline)) { load_a(X, 2, i); }, zero, mid, fetch);
        work(std::integral_constant<int, 2>{}, half, [&](int i) __attribute__((always_inline)) { load_a(X, 3, i); }, zero, zero, [](int) {});
        if constexpr (kMore) {
            arrive(std::integral_constant<int, kFetch ? kLoads : kLoads - kMid>{});
            work(std::integral_constant<int, 3>{}, whole, [&](int i) __attribute__((always_inline)) { first_operands(Y, i); }, mid, end, fetch);
        }
    };
    // The loop body never branches between two ways of updating the accumulators (that would make the compiler shuffle all
    // of them): the steady state always has a next step, the last one or two steps are peeled.  A fetch past the end repeats
    // the last step into a stage that nobody reads again.
    const uint32_t last = steps - 1u;
    auto run_steps = [&](auto works) __attribute__((always_inline)) {
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        uint32_t s = 0;
        for (; s + 2 < steps; s += 2) {
            step(S0, S1, s + 2, yes, yes, works);
            step(S1, S0, s + 3 < last ? s + 3 : last, yes, yes, works);
        }
        if (s + 1 < steps) {  // two steps left: this one in stage 0, the last one on its way into stage 1
            step(S0, S1, last, no, yes, works);
        }
        const bool odd = (steps & 1u) != 0;
        const Stage X{{odd ? S0.a[0] : S1.a[0], odd ? S0.a[1] : S1.a[1]}, odd ? S0.b : S1.b};
        step(X, X, last, no, no, works);
    };
    {
        const auto from0 = bases(0u), from1 = bases(last < 1u ? last : 1u);
        // (in this order: the waits count the loads behind the ones they are for)
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            load(from0, u, S0);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            load(from1, u, S1);
            __builtin_amdgcn_sched_barrier(0);
        }
        arrive(std::integral_constant<int, 2 * kLoads - kMid>{});
    }
    // a wavefront whose rows all lie past the end of the tile's group skips the matrix work and only keeps the loads and
    // barriers going: its SIMD then runs one wavefront's matrix instructions per K step instead of two
    if (!kGrouped || row0 + wm * (NA * 16u) < row_end) {
#pragma unroll
        for (int i = 0; i < NH + kBReads; ++i) first_operands(S0, i);
        run_steps(std::true_type{});
        static_for<kM>([&](auto n) { mfma(3, decltype(n)::value); });
    } else {
        run_steps(std::false_type{});
    }
    // The last sums are on their way through the matrix pipe, which the compiler does not know: it sees them
    // changed behind the wait, so that nothing that reads them can move ahead of it.  (check_matrix_asm.py looks
    // through the machine code for what this cannot rule out, a copy inside the loop.)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < NA; ++i) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) asm volatile("" : "+v"(acc[i][j]));
    }

    // ---- epilogue: register r of lane l in a 16 x 16 block is row 4 (l / 16) + r, column l % 16
    const uint32_t colw = n0 + wn * 64u;  // first column of this wavefront
    const EpiParams& e = p.epi;
    ChannelQ q[TJ];
    float bias_post[TJ];
    int32_t bias_pre[TJ];
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        const uint32_t col = colw + j * 16u + lc;
        q[j] = ChannelQ{1.0f, 0, 1};
        bias_post[j] = 0.0f;
        bias_pre[j] = 0;
        if (col < N) {
            q[j] = load_channel_q(e, chan_off + col);
            bias_post[j] = load_bias_post(e, chan_off + col);
            if (e.bias_kind == ASCQ_MM_BIAS_I32_PRE) {
                bias_pre[j] = static_cast<const int32_t*>(e.bias)[chan_off + col];
            }
        }
    }
    // Quant words that shift the accumulator first (mode-control bit) are rare: when any column of the wavefront carries one,
    // it goes element by element with every choice made at run time.  The sums pass through the wavefront's part of a stage,
    // 16 rows by 32 columns at a time, so that one loop with one copy of the epilogue serves all of them and neighbouring
    // lanes hold neighbouring columns.
    bool by_element = false;
    if (e.scale_format == ASCQ_MM_SCALE_U64) {  // (the same for the whole workgroup)
        by_element = __builtin_amdgcn_ballot_w64(((q[0].ctl | q[1].ctl | q[2].ctl | q[3].ctl) & 2) != 0) != 0;
        __syncthreads();  // everyone has left the last stage
    }
    if (by_element) {
        int32_t* const mine = reinterpret_cast<int32_t*>(S0.b) + wave * 512u;
        auto cell = [](uint32_t row, uint32_t c) __attribute__((always_inline)) { return row * 32u + (c ^ ((row << 2) & 16u)); };
#pragma unroll 1
        for (uint32_t part = 0; part < NA * 2u; ++part) {
            static_for<NA * 2>([&](auto c) {
                constexpr int i = decltype(c)::value / 2, j0 = decltype(c)::value % 2 * 2;
                if (part == static_cast<uint32_t>(decltype(c)::value)) {  // uniform
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) mine[cell(4u * lq + r, j * 16u + lc)] = acc[i][j0 + j][r];
                    }
                }
            });
            const uint32_t col = colw + (part & 1u) * 32u + (lane & 31u);
            const bool live = col < N;
            const ChannelQ cq = live ? load_channel_q(e, chan_off + col) : ChannelQ{1.0f, 0, 1};
            const float post = live ? load_bias_post(e, chan_off + col) : 0.0f;
            const int32_t pre = live && e.bias_kind == ASCQ_MM_BIAS_I32_PRE ? static_cast<const int32_t*>(e.bias)[chan_off + col] : 0;
#pragma unroll 1
            for (uint32_t r = lane >> 5; r < 16u; r += 2u) {
                const uint32_t lrow = (wm * NA + part / 2u) * 16u + r;
                if (live && row0 + lrow < row_end) {
                    epilogue_store_lanes(e, row0 + lrow, col, mine[cell(r, lane & 31u)] + pre, cq, TS[lrow], post);
                }
            }
        }
        return;
    }
    auto run = [&](auto tag) {
        constexpr int kOut = decltype(tag)::value;
        const bool b0 = (lane & 1u) != 0, b1 = (lane & 2u) != 0;
        // SwiGLU of the four de-quantised values of a row: adjacent lanes hold the two columns of a pair.  After one lane
        // swap the even lane owns the pairs of blocks 0 and 2 (src0 its own value, src1 its neighbour's), the odd lane
        // those of blocks 1 and 3 (src0 its neighbour's).
        auto swiglu_row = [&](const float (&v)[TJ], uint32_t row) __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float recv = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(b0 ? v[2 * h] : v[2 * h + 1]), 0xB1, 0xF, 0xF, true));  // lane ^ 1
                const float o = swiglu(b0 ? recv : v[2 * h], b0 ? v[2 * h + 1] : recv, e.act_beta);
                const uint32_t col = colw + 32u * h + (b0 ? 16u + lc - 1u : lc);  // first column of the pair
                if (row < row_end && col < N) {
                    __builtin_nontemporal_store(static_cast<uint16_t>(to_bits16<kOut>(o)),
                                                static_cast<uint16_t*>(e.c) + static_cast<size_t>(row) * e.ldc + (col >> 1));
                }
            }
        };
        // The uniform choices (post-dequant bias, activation) are made once, outside the element loops, so that each
        // wavefront runs one compact straight-line epilogue.
        auto store_all = [&](auto bias_tag, auto gelu_tag, auto swiglu_tag) {
            constexpr bool kBiasPost = decltype(bias_tag)::value;
            constexpr bool kGelu = decltype(gelu_tag)::value;
            constexpr bool kSwiGlu = decltype(swiglu_tag)::value;
            // A 4 x 4 transposition inside each four neighbouring lanes (two exchanges of packed pairs) leaves lane b of
            // the four with columns 4 (l / 4) .. + 3 of block b: one 8-byte store per lane and row, and the 16 lanes of
            // a row write one full 128-byte line.
            const uint32_t col = colw + 16u * (lane & 3u) + (lc & 12u);
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                const uint32_t lbase = (wm * NA + i) * 16u + 4u * lq;
                const f32x4 tok4 = *reinterpret_cast<const f32x4*>(&TS[lbase]);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t row = row0 + lbase + r;
                    float v[TJ];
#pragma unroll
                    for (int j = 0; j < TJ; ++j) {
                        v[j] = epi_value<kBiasPost, kGelu>(acc[i][j][r] + bias_pre[j], q[j].s, tok4[r], bias_post[j]);
                    }
                    if constexpr (kSwiGlu) {
                        swiglu_row(v, row);
                        continue;
                    }
                    uint32_t h[TJ];
#pragma unroll
                    for (int j = 0; j < TJ; ++j) h[j] = to_bits16<kOut>(v[j]);
                    const uint32_t give = b0 ? h[0] | (h[2] << 16) : h[1] | (h[3] << 16);
                    const uint32_t got = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(give), 0xB1, 0xF, 0xF, true));  // lane ^ 1
                    const uint32_t lo = b0 ? (got & 0xFFFFu) | (h[1] << 16) : h[0] | (got << 16);
                    const uint32_t hi = b0 ? (got >> 16) | (h[3] << 16) : h[2] | (got & 0xFFFF0000u);
                    const uint32_t got2 = static_cast<uint32_t>(
                        __builtin_amdgcn_mov_dpp(static_cast<int>(b1 ? lo : hi), 0x4E, 0xF, 0xF, true));  // lane ^ 2
                    if (row < row_end && col < N) {
                        __builtin_nontemporal_store(b1 ? u32x2{got2, hi} : u32x2{lo, got2},
                                                    reinterpret_cast<u32x2*>(static_cast<uint16_t*>(e.c) +
                                                                             static_cast<size_t>(row) * e.ldc + col));
                    }
                }
            }
        };
        const bool bias_post_on = e.bias_kind >= ASCQ_MM_BIAS_F32_POST;
        const bool gelu_on = e.activation == ASCQ_MM_ACT_FASTER_GELU;
        if (e.activation == ASCQ_MM_ACT_SWIGLU) {
            if (bias_post_on) {
                store_all(std::true_type{}, std::false_type{}, std::true_type{});
            } else {
                store_all(std::false_type{}, std::false_type{}, std::true_type{});
            }
        } else if (gelu_on) {
            if (bias_post_on) {
                store_all(std::true_type{}, std::true_type{}, std::false_type{});
            } else {
                store_all(std::false_type{}, std::true_type{}, std::false_type{});
            }
        } else if (bias_post_on) {
            store_all(std::true_type{}, std::false_type{}, std::false_type{});
        } else {
            store_all(std::false_type{}, std::false_type{}, std::false_type{});
        }
    };
    if (e.out_dtype == ASCQ_BF16) {
        run(OutTag<ASCQ_BF16>{});
    } else {
        run(OutTag<ASCQ_F16>{});
    }
}

// The body of a small tile: a ring of kStages LDS stages of a K step each, loads that are issued kStages - 1/2 steps ahead
// (see matmul_w8a8_ring.hip).  load(step, u, stage): load u of the wavefront's kLoads of a step; past the end it brings zeros.
// kHalf: see kRingHalf.
template <int BM, int BN, int kB, int kStages, int kLoads, bool kHalf, class Load>
__device__ __forceinline__ void gemm_ring_body(const GemmParams& p, const TilePlace& at, uint32_t n0, uint32_t steps, uint32_t wave,
                                               uint32_t lane, Load&& load, char* const (&L)[kStages], float* TS)
{
    constexpr bool kBT = kB == 1, kBP = kB == 2;
    constexpr int TJ = BN == 64 ? 2 : 4;                       // 16 x 16 blocks per wavefront along N
    constexpr int kWN = BN / 16 / TJ, kWM = 8 / kWN;           // wavefronts along N and M
    constexpr int NA = BM / 16 / kWM;                          // blocks along M
    static_assert(NA >= 1 && NA * 16 * kWM == BM && kWM * kWN == 8, "tile shape does not fit eight wavefronts");
    const uint32_t wm = wave / kWN, wn = wave % kWN;
    const uint32_t lc = lane & 15u, lq = lane >> 4;

    i32x4 acc[NA][TJ];
    static_for<NA * TJ>([&](auto c) {
        i32x4& v = acc[decltype(c)::value / TJ][decltype(c)::value % TJ];
        v = i32x4{0, 0, 0, 0};
        asm volatile("" : "+v"(v));
    });
    uint32_t foff[2], b_base[TJ];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) foff[ks] = lc * 128u + (((4u * ks + lq) ^ (lc >> 1)) << 4);
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        // transposing reads: in 16 lanes, rows bsub of 8 and halves psub of the block's 16 columns
        const uint32_t bsub = lc >> 1, psub = lc & 1u, row = 16u * lq + bsub;
        b_base[j] = kBP ? wn * (TJ * 2048u) + lane * 16u : row * BN + (((static_cast<uint32_t>(TJ) * wn + j) ^ b_swizzle<BN, true>(row)) << 4) + 8u * psub;
    }
    i32x4 af[2][2][NA], bf[2][2][TJ];  // [set][half of the step]: a step's operands arrive while those of the one before are in use
    i32x2_t blo;
    constexpr int kBReads = (kBT || kBP) ? TJ : 2 * TJ, kReads = NA + kBReads;  // LDS reads of 64 k
    auto read = [&](const char* S, int set, int r) __attribute__((always_inline)) {
        const char* const Bs = S + BM * BK;
        const int ks = r / kReads;
        r %= kReads;
        if (r < NA) {
            af[set][ks][r] = *reinterpret_cast<const i32x4*>(S + (wm * NA + r) * 2048u + foff[ks]);
            return;
        }
        r -= NA;
        if constexpr (kBT) {
            bf[set][ks][r] = *reinterpret_cast<const i32x4*>(Bs + (wn * TJ + r) * 2048u + foff[ks]);
        } else if constexpr (kBP) {
            bf[set][ks][r] = *reinterpret_cast<const i32x4*>(Bs + b_base[0] + r * 2048u + ks * 1024u);
        } else {
            const i32x2_t v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2_t)(Bs + b_base[r >> 1] + ks * (64 * BN) + (r & 1) * (8 * BN)));
            if (r & 1) {
                bf[set][ks][r >> 1] = i32x4{blo[0], blo[1], v[0], v[1]};
            } else {
                blo = v;
            }
        }
    };
    auto arrive = [&](auto left) __attribute__((always_inline)) {
        constexpr int kLeft = decltype(left)::value;
        __builtin_amdgcn_s_waitcnt(0x0070 | (kLeft & 15) | ((kLeft >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();  // (not __syncthreads(): its fence waits for every load)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // A step in stage X, the next one in Y.  Its operands are in registers or on their way there: behind the wait (they are there,
    // the next step has landed, those behind it are on their way) and the barrier every wavefront has read the stage, which
    // takes the step kStages ahead, and the next step's operands are read behind this one's matrix instructions, in the order written.
    constexpr int kM = 2 * NA * TJ, kPer = (2 * kReads + kM - 1) / kM, kLoadPer = (kLoads + kM - 1) / kM;
    auto step = [&](uint32_t s, char* X, const char* Y, auto set) __attribute__((always_inline)) {
        constexpr int x = decltype(set)::value;
#pragma unroll
        for (int q = 0; q < 2; ++q) asm volatile("" : "+v"(foff[q]));
#pragma unroll
        for (int j = 0; j < (kBP ? 1 : TJ); ++j) asm volatile("" : "+v"(b_base[j]));
        arrive(std::integral_constant<int, (kStages - 2) * kLoads>{});
        static_for<kM>([&](auto nn) {
            constexpr int n = decltype(nn)::value, ks = n / (NA * TJ), i = n / TJ % NA, j = n % TJ;
            i32x4& c = acc[i][j];
            asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(c) : "v"(af[x][ks][i]), "v"(bf[x][ks][j]));
            static_for<kPer>([&](auto r) {
                constexpr int m = n * kPer + decltype(r)::value;
                if constexpr (m < 2 * kReads) read(Y, 1 - x, m);
            });
            static_for<kLoadPer>([&](auto r) {
                constexpr int u = n * kLoadPer + decltype(r)::value;
                if constexpr (u < kLoads) load(s + kStages, u, X);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    static_for<kStages>([&](auto st) {  // (in this order: the waits count the loads behind the ones they are for)
#pragma unroll
        for (int u = 0; u < kLoads; ++u) load(decltype(st)::value, u, L[decltype(st)::value]);
        __builtin_amdgcn_sched_barrier(0);
    });
    arrive(std::integral_constant<int, (kStages - 1) * kLoads>{});
#pragma unroll
    for (int r = 0; r < 2 * kReads; ++r) read(L[0], 0, r);
    constexpr int kGroup = kStages % 2 ? 2 * kStages : kStages;  // stages and sets
    uint32_t s = 0;
    for (; s + kGroup <= steps; s += kGroup) {
        static_for<kGroup>([&](auto st) {
            constexpr int i = decltype(st)::value;
            step(s + i, L[i % kStages], L[(i + 1) % kStages], std::integral_constant<int, i % 2>{});
        });
    }
    bool more = true;  // what is left of the last group (a step without a next one reads what nobody uses)
    static_for<kGroup - 1>([&](auto st) {
        constexpr int i = decltype(st)::value;
        more = more && s + i < steps;
        if (more) step(s + i, L[i % kStages], L[(i + 1) % kStages], std::integral_constant<int, i % 2>{});
    });
    // The last sums are on their way through the matrix pipe, which the compiler does not know; the loads past the end land
    // before the LDS is given back.
    asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
    static_for<NA * TJ>([&](auto c) {
        i32x4& v = acc[decltype(c)::value / TJ][decltype(c)::value % TJ];
        asm volatile("" : "+v"(v));
    });

    // ---- epilogue: register r of lane l in a 16 x 16 block is row 4 (l / 16) + r, column l % 16
    const EpiParams& e = p.epi;
    const uint32_t N = p.n, colw = n0 + wn * (TJ * 16u);
    ChannelQ q[TJ];
    float bias_post[TJ];
    int32_t bias_pre[TJ];
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        const uint32_t col = colw + j * 16u + lc;
        q[j] = ChannelQ{1.0f, 0, 1};
        bias_post[j] = 0.0f;
        bias_pre[j] = 0;
        if (col < N) {
            q[j] = load_channel_q(e, at.chan_off + col);
            bias_post[j] = load_bias_post(e, at.chan_off + col);
            if (e.bias_kind == ASCQ_MM_BIAS_I32_PRE) {
                bias_pre[j] = static_cast<const int32_t*>(e.bias)[at.chan_off + col];
            }
        }
        asm volatile("" : "+v"(q[j].s), "+v"(bias_post[j]), "+v"(bias_pre[j]));  // (waited for once, not at every store)
    }
    bool shifts = false;  // quant words that shift the accumulator first (rare): element by element
    if (!kHalf && e.scale_format == ASCQ_MM_SCALE_U64) {
        int any = 0;
#pragma unroll
        for (int j = 0; j < TJ; ++j) any |= q[j].ctl;
        shifts = __builtin_amdgcn_ballot_w64((any & 2) != 0) != 0;
    }
    const bool quantised = kHalf || e.quant_mode != ASCQ_MM_QUANT_NONE, half_out = kHalf || (quantised && (e.out_dtype == ASCQ_BF16 || e.out_dtype == ASCQ_F16));
    const bool wide_out = !quantised || e.out_dtype == ASCQ_F32;  // four bytes: raw sums or floats
    if (kHalf || (!shifts && (half_out || wide_out))) {
        // (Element by element, a lane's choices made at run time, 364 x 1024 x 7000 with SwiGLU to float took 21.0 us and 829 x 592 x
        // 5120 to float 31.9; 14.0 and 18.4 like this.)
        const bool b0 = (lane & 1u) != 0, b1 = (lane & 2u) != 0, post = e.bias_kind >= ASCQ_MM_BIAS_F32_POST;
        const bool gelu = e.activation == ASCQ_MM_ACT_FASTER_GELU, bf16 = e.out_dtype == ASCQ_BF16;
        const bool pairs = !kHalf && quantised && e.activation == ASCQ_MM_ACT_SWIGLU;
        auto value = [&](int i, int j, int r, float tok) __attribute__((always_inline)) {
            float v = static_cast<float>(acc[i][j][r] + bias_pre[j]) * q[j].s;
            v = v * tok;  // 1.0f without a token scale: an exact identity
            return post ? v + bias_post[j] : v;
        };
        auto bits16 = [&](float v) __attribute__((always_inline)) { return bf16 ? to_bits16<ASCQ_BF16>(v) : to_bits16<ASCQ_F16>(v); };
        auto swap1 = [](uint32_t v) __attribute__((always_inline)) { return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0xB1, 0xF, 0xF, true)); };  // lane ^ 1
        auto swap2 = [](uint32_t v) __attribute__((always_inline)) { return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x4E, 0xF, 0xF, true)); };  // lane ^ 2
        // every 4 rows of the wavefront's blocks: block row i, register r, its row of the matrix, its token scale
        auto rows = [&](auto&& each) __attribute__((always_inline)) {
            static_for<NA>([&](auto ii) {
                constexpr int i = decltype(ii)::value;
                const uint32_t lbase = (wm * NA + i) * 16u + 4u * lq;
                each(ii, at.row0 + lbase, *reinterpret_cast<const f32x4*>(&TS[lbase]));
            });
        };
        if (half_out && !pairs) {
            rows([&](auto ii, uint32_t row0, const f32x4& tok4) __attribute__((always_inline)) {
                constexpr int i = decltype(ii)::value;
                static_for<4>([&](auto rr) {
                    constexpr int r = decltype(rr)::value;
                    const uint32_t row = row0 + r;
                    uint32_t h[TJ];
                    static_for<TJ>([&](auto jj) {
                        constexpr int j = decltype(jj)::value;
                        const float v = value(i, j, r, tok4[r]);
                        h[j] = bits16(gelu ? faster_gelu(v) : v);
                    });
                    uint16_t* const out = static_cast<uint16_t*>(e.c) + static_cast<size_t>(row) * e.ldc;
                    if constexpr (TJ == 4) {
                        // a 4 x 4 transposition inside each four neighbouring lanes (see gemm_dma_body16): 8-byte stores, whole lines
                        const uint32_t col = colw + 16u * (lane & 3u) + (lc & 12u);
                        const uint32_t got = swap1(b0 ? h[0] | (h[2] << 16) : h[1] | (h[3] << 16));
                        const uint32_t lo = b0 ? (got & 0xFFFFu) | (h[1] << 16) : h[0] | (got << 16);
                        const uint32_t hi = b0 ? (got >> 16) | (h[3] << 16) : h[2] | (got & 0xFFFF0000u);
                        const uint32_t got2 = swap2(b1 ? lo : hi);
                        if (row < at.row_end && col < N) {
                            __builtin_nontemporal_store(b1 ? u32x2{got2, hi} : u32x2{lo, got2}, reinterpret_cast<u32x2*>(out + col));
                        }
                    } else {
                        // after one swap the even lane holds two adjacent columns of the first block, the odd lane two of the second
                        const uint32_t col = b0 ? colw + 16u + lc - 1u : colw + lc;
                        const uint32_t got = swap1(b0 ? h[0] : h[1]);
                        if (row < at.row_end && col < N) {
                            __builtin_nontemporal_store(b0 ? got | (h[1] << 16) : h[0] | (got << 16), reinterpret_cast<uint32_t*>(out + col));
                        }
                    }
                });
            });
            return;
        }
        if (pairs) {
            // Adjacent lanes hold the two columns of a pair.  After one swap the even lane owns the pair of the first of two blocks, the
            // odd lane that of the second; after another one, of two rows, lanes l and l ^ 2 hold two adjacent outputs of a row each.
            rows([&](auto ii, uint32_t row0, const f32x4& tok4) __attribute__((always_inline)) {
                static_for<TJ>([&](auto cc) {
                    constexpr int i = decltype(ii)::value, j = decltype(cc)::value / 2 * 2, r = decltype(cc)::value % 2 * 2;
                    float o[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const float v0 = value(i, j, r + t, tok4[r + t]), v1 = value(i, j + 1, r + t, tok4[r + t]);
                        const float got = __int_as_float(static_cast<int>(swap1(static_cast<uint32_t>(__float_as_int(b0 ? v0 : v1)))));
                        o[t] = swiglu(b0 ? got : v0, b0 ? v1 : got, e.act_beta);
                    }
                    const uint32_t row = row0 + r + (b1 ? 1u : 0u), col = colw + 16u * j + (b0 ? 16u : 0u) + (lc & 12u);
                    const size_t to = static_cast<size_t>(row) * e.ldc + (col >> 1);
                    if (half_out) {
                        const uint32_t h0 = bits16(o[0]), h1 = bits16(o[1]), got = swap2(b1 ? h0 : h1);
                        if (row < at.row_end && col < N) {
                            __builtin_nontemporal_store(b1 ? got | (h1 << 16) : h0 | (got << 16), reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(e.c) + to));
                        }
                    } else {
                        const uint32_t h0 = static_cast<uint32_t>(__float_as_int(o[0])), h1 = static_cast<uint32_t>(__float_as_int(o[1]));
                        const uint32_t got = swap2(b1 ? h0 : h1);
                        if (row < at.row_end && col < N) {
                            __builtin_nontemporal_store(b1 ? u32x2{got, h1} : u32x2{h0, got}, reinterpret_cast<u32x2*>(static_cast<uint32_t*>(e.c) + to));
                        }
                    }
                });
            });
            return;
        }
        rows([&](auto ii, uint32_t row0, const f32x4& tok4) __attribute__((always_inline)) {
            static_for<2 * TJ>([&](auto cc) {
                // two blocks of a row: after one swap the even lane holds two adjacent columns of the first, the odd lane two of the second
                constexpr int i = decltype(ii)::value, r = decltype(cc)::value % 4, j = decltype(cc)::value / 4 * 2;
                uint32_t h[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    float v = value(i, j + t, r, tok4[r]);
                    v = gelu ? faster_gelu(v) : v;
                    h[t] = quantised ? static_cast<uint32_t>(__float_as_int(v)) : static_cast<uint32_t>(acc[i][j + t][r] + bias_pre[j + t]);
                }
                const uint32_t row = row0 + r, col = b0 ? colw + 16u * j + 16u + lc - 1u : colw + 16u * j + lc, got = swap1(b0 ? h[0] : h[1]);
                if (row < at.row_end && col < N) {
                    __builtin_nontemporal_store(b0 ? u32x2{got, h[1]} : u32x2{h[0], got},
                                                reinterpret_cast<u32x2*>(static_cast<uint32_t*>(e.c) + static_cast<size_t>(row) * e.ldc + col));
                }
            });
        });
        return;
    }
    static_for<NA * TJ>([&](auto c) {
        constexpr int i = decltype(c)::value / TJ, j = decltype(c)::value % TJ;
        const uint32_t lbase = (wm * NA + i) * 16u + 4u * lq, col = colw + j * 16u + lc;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (at.row0 + lbase + r < at.row_end && col < N) {
                epilogue_store_lanes(e, at.row0 + lbase + r, col, acc[i][j][r] + bias_pre[j], q[j], TS[lbase + r], bias_post[j]);
            }
        }
    });
}

// The body of a tile on v_mfma_i32_32x32x32_i8, every output.
template <int BM, int BN, bool kSplitK, bool kGrouped, int kB, class Issue>
__device__ __forceinline__ void gemm_dma_body32(const GemmParams& p, const TilePlace& at, uint32_t n0, uint32_t steps, uint32_t bidy,
                                                uint32_t wave, uint32_t lane, Issue&& issue, char* A0, char* B0, char* A1, char* B1,
                                                float* TS)
{
    constexpr bool kBT = kB == 1, kBP = kB == 2;
    constexpr int kWN = BN / 64;            // wavefronts along N
    constexpr int kWM = 8 / kWN;            // wavefronts along M
    constexpr int TI = BM / 32 / kWM;       // 32x32 blocks per wavefront along M
    constexpr int TJ = 2;                   // and along N
    constexpr int kKsB = 32 * BN;           // bytes of B per K sub-step of 32 rows
    static_assert(TI >= 1 && TI * 32 * kWM == BM, "tile shape does not fit eight wavefronts");
    const uint32_t wm = wave / kWN, wn = wave % kWN;
    const uint32_t N = p.n, row0 = at.row0, row_end = at.row_end;
    const size_t chan_off = at.chan_off;

    i32x16 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
        }
    }

    // ---- fragment addresses: one base per K sub-step (A) / per column block (B), everything else is an immediate
    const uint32_t lrow = lane & 31u, g = lane >> 5;
    const uint32_t grp16 = (lane >> 4) & 1u, bsub = (lane & 15u) >> 1, psub = lane & 1u;
    uint32_t a_base[4], b_base[2], bt_base[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        a_base[ks] = (wm * (TI * 32) + lrow) * 128 + (((2 * ks + g) ^ ((lrow >> 1) & 7u)) << 4);
        bt_base[ks] = (wn * (TJ * 32) + lrow) * 128 + (((2 * ks + g) ^ ((lrow >> 1) & 7u)) << 4);
        if constexpr (kBP) {
            // column block j of the wavefront: slabs 4 wn + 2 j + lrow / 16 (2 KiB each: the step's two k tiles); sub-step
            // ks is k tile ks / 2, its 16-byte groups 2 (ks % 2) + g; inside a group the 16 columns lie side by side
            bt_base[ks] = wn * 8192u + (lrow >> 4) * 2048u + (ks >> 1) * 1024u + ((ks & 1) * 2u + g) * 256u + (lrow & 15u) * 16u;
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint32_t swz = BN == 256 ? 2u * bsub : 2u * ((bsub >> 1) & 3u);
        b_base[j] = (16 * g + bsub) * BN + (((4 * wn + 2 * j + grp16) ^ swz) << 4) + 8 * psub;
    }
    // In the order the MFMAs of a sub-step want them (they run row block by row block): B0, A0, B1, A1, A2, ...
    auto load_frags = [&](const char* As, const char* Bs, int ks, i32x4 (&af)[TI], i32x4 (&bf)[TJ]) {
        auto load_b = [&](int j) {
            if constexpr (kBT || kBP) {
                bf[j] = *reinterpret_cast<const i32x4*>(Bs + bt_base[ks] + j * 4096);
            } else {
                const i32x2_t lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2_t)(Bs + b_base[j] + ks * kKsB));
                const i32x2_t hi =
                    __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2_t)(Bs + b_base[j] + ks * kKsB + 8 * BN));
                bf[j] = i32x4{lo[0], lo[1], hi[0], hi[1]};
            }
        };
        load_b(0);
        af[0] = *reinterpret_cast<const i32x4*>(As + a_base[ks]);
        load_b(1);
#pragma unroll
        for (int i = 1; i < TI; ++i) {
            af[i] = *reinterpret_cast<const i32x4*>(As + a_base[ks] + i * 4096);
        }
    };
    // Fragment registers live across K steps: buffer 0 holds sub-steps 0 and 2, buffer 1 sub-steps 1 and 3.
    i32x4 af[2][TI], bf[2][TJ];
    auto mfma_block = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TI; ++i) {
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[buf][i], bf[buf][j], acc[i][j], 0, 0, 0);
            }
        }
    };
    // The LDS reads of a sub-step go out behind its first MFMAs (kReadsPerMfma behind each), so that the matrix
    // instructions of its second half run while the last reads are still on their way: the next sub-step starts by
    // waiting for all of them.
    auto interleave = [&]() __attribute__((always_inline)) {
        constexpr int kReads = TI + ((kBT || kBP) ? TJ : 2 * TJ);
        constexpr int kMfmas = TI * TJ;
        constexpr int kFront = (kMfmas + 1) / 2;
        constexpr int kPer = (kReads + kFront - 1) / kFront;
        static_for<kMfmas>([&](auto n) {
            constexpr int kLeft = kReads - decltype(n)::value * kPer;
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if constexpr (kLeft > 0) {
                __builtin_amdgcn_sched_group_barrier(0x100, kLeft < kPer ? kLeft : kPer, 0);
            }
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    // Sub-steps 0-2 of a K step whose sub-step-0 fragments are already in buffer 0; on return the fragments of
    // sub-step 3 are on their way into buffer 1 and nothing else of the stage will be read.
    auto head = [&](const char* As, const char* Bs) __attribute__((always_inline)) {
        // Re-materialise the bases inside the loop body: the constant parts of every address then fold into the
        // 16-bit offset field of the DS instructions instead of being hoisted into dozens of registers.
#pragma unroll
        for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(a_base[q]));
#pragma unroll
        for (int q = 0; q < 2; ++q) asm volatile("" : "+v"(b_base[q]));
        if constexpr (kBT || kBP) {
#pragma unroll
            for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(bt_base[q]));
        }
#pragma unroll
        for (int ks = 0; ks < 3; ++ks) {
            load_frags(As, Bs, ks + 1, af[(ks + 1) & 1], bf[(ks + 1) & 1]);
            mfma_block(ks & 1);
            interleave();
        }
    };
    // sub-step 3, and the first fragments of the next K step (stage An, Bn)
    auto tail = [&](const char* An, const char* Bn) __attribute__((always_inline)) {
        load_frags(An, Bn, 0, af[0], bf[0]);
        mfma_block(1);
        interleave();
    };

    gemm_dma_loop(
        steps, !kGrouped || row0 + wm * (TI * 32u) < row_end, A0, B0, A1, B1, issue,
        [&](const char* As, const char* Bs) __attribute__((always_inline)) { load_frags(As, Bs, 0, af[0], bf[0]); }, head, tail,
        [&]() __attribute__((always_inline)) { mfma_block(1); });

    // ---- epilogue: register r of lane l in a 32x32 block is row 8*(r/4) + 4*(l/32) + r%4, column l%32
    if constexpr (kSplitK) {
        int32_t* part = p.partial + static_cast<size_t>(bidy) * p.m * N;
#pragma unroll
        for (int i = 0; i < TI; ++i) {
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                const uint32_t col = n0 + (wn * TJ + j) * 32u + lrow;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t row = row0 + (wm * TI + i) * 32u + 8u * (r >> 2) + 4u * g + (r & 3);
                    if (row < row_end && col < N) {
                        part[static_cast<size_t>(row) * N + col] = acc[i][j][r];
                    }
                }
            }
        }
        return;
    }
    const EpiParams& e = p.epi;
    auto run = [&](auto tag) {
        constexpr int kOut = decltype(tag)::value;
        const uint32_t colw = n0 + wn * (TJ * 32u);  // first column of this wavefront
        ChannelQ q[TJ];
        float bias_post[TJ];
        int32_t bias_pre[TJ];
        bool cvalid[TJ];
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const uint32_t col = colw + j * 32u + lrow;
            cvalid[j] = col < N;
            q[j] = ChannelQ{1.0f, 0, 1};
            bias_post[j] = 0.0f;
            bias_pre[j] = 0;
            if (cvalid[j]) {
                q[j] = load_channel_q(e, chan_off + col);
                bias_post[j] = load_bias_post(e, chan_off + col);
                if (e.bias_kind == ASCQ_MM_BIAS_I32_PRE) {
                    bias_pre[j] = static_cast<const int32_t*>(e.bias)[chan_off + col];
                }
            }
            // Wait for the conditional loads here: left to itself the compiler waits at each use, and each such wait is one
            // for the stores before it (2048 x 4096 x 11008, int32 98 -> 105 us).
            asm volatile("" : "+v"(q[j].s), "+v"(bias_post[j]), "+v"(bias_pre[j]));
        }
        // The uniform choices (post-dequant bias, activation) are made once, outside the element loops, so that each
        // wavefront runs one compact straight-line epilogue.
        auto store_all = [&](auto bias_tag, auto gelu_tag, auto swiglu_tag) {
            constexpr bool kBiasPost = decltype(bias_tag)::value;
            constexpr bool kGelu = decltype(gelu_tag)::value;
            constexpr bool kSwiGlu = decltype(swiglu_tag)::value;
            (void)kBiasPost;
            (void)kGelu;
            (void)kSwiGlu;
    #pragma unroll
            for (int i = 0; i < TI; ++i) {
                const uint32_t lbase = (wm * TI + i) * 32u + 4u * g;  // row inside the tile of register 0
    #pragma unroll
                for (int rq = 0; rq < 4; ++rq) {
                    const f32x4 tok4 = *reinterpret_cast<const f32x4*>(&TS[lbase + 8u * rq]);
    #pragma unroll
                    for (int rr = 0; rr < 4; ++rr) {
                        const int r = 4 * rq + rr;
                        const uint32_t row = row0 + lbase + 8u * rq + rr;
                        if constexpr (kOut == ASCQ_BF16 || kOut == ASCQ_F16) {
                            // One dword store per lane covers a full 128-byte line per row: even lanes write columns
                            // (l, l+1) of the first 32-column block, odd lanes columns (l-1, l) of the second one.
                            static_assert(TJ == 2, "the paired store assumes two column blocks per wavefront");
                            const bool odd = (lane & 1u) != 0;
                            if constexpr (kSwiGlu) {
                                // Adjacent lanes hold the two columns of a pair.  After one lane swap the even lane
                                // owns the pair of the first 32-column block (src0 its own value, src1 its
                                // neighbour's), the odd lane the pair of the second block (src0 its neighbour's).
                                const float v0 = epi_value<kBiasPost, false>(acc[i][0][r] + bias_pre[0], q[0].s, tok4[rr],
                                                                             bias_post[0]);
                                const float v1 = epi_value<kBiasPost, false>(acc[i][1][r] + bias_pre[1], q[1].s, tok4[rr],
                                                                             bias_post[1]);
                                const float recv = __int_as_float(__builtin_amdgcn_mov_dpp(
                                    __float_as_int(odd ? v0 : v1), 0xB1, 0xF, 0xF, true));  // lane ^ 1
                                const float o = swiglu(odd ? recv : v0, odd ? v1 : recv, e.act_beta);
                                const uint32_t col = odd ? colw + 32u + (lrow - 1u) : colw + lrow;  // first column of the pair
                                if (row < row_end && col < N) {
                                    __builtin_nontemporal_store(
                                        static_cast<uint16_t>(to_bits16<kOut>(o)),
                                        static_cast<uint16_t*>(e.c) + static_cast<size_t>(row) * e.ldc + (col >> 1));
                                }
                                continue;
                            }
                            const uint32_t h0 =
                                to_bits16<kOut>(
                                    epi_value<kBiasPost, kGelu>(acc[i][0][r] + bias_pre[0], q[0].s, tok4[rr], bias_post[0]));
                            const uint32_t h1 =
                                to_bits16<kOut>(
                                    epi_value<kBiasPost, kGelu>(acc[i][1][r] + bias_pre[1], q[1].s, tok4[rr], bias_post[1]));
                            const uint32_t send = odd ? h0 : h1;
                            const uint32_t recv = static_cast<uint32_t>(
                                __builtin_amdgcn_mov_dpp(static_cast<int>(send), 0xB1, 0xF, 0xF, true));  // lane ^ 1
                            const uint32_t word = odd ? (recv | (h1 << 16)) : (h0 | (recv << 16));
                            const uint32_t col = odd ? colw + 32u + (lrow - 1u) : colw + lrow;
                            if (row < row_end && col < N) {
                                __builtin_nontemporal_store(
                                    word, reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(e.c) +
                                                                      static_cast<size_t>(row) * e.ldc + col));
                            }
                        } else {
    #pragma unroll
                            for (int j = 0; j < TJ; ++j) {
                                if (cvalid[j] && row < row_end) {
                                    epilogue_store<kOut>(e, row, colw + j * 32u + lrow, acc[i][j][r] + bias_pre[j], q[j],
                                                         tok4[rr], bias_post[j]);
                                }
                            }
                        }
                    }
                }
            }
        };
        if constexpr (kOut == ASCQ_BF16 || kOut == ASCQ_F16) {
            // Quant words that shift the accumulator first (mode-control bit) are rare: when any column of the
            // wavefront carries one, a compact epilogue that reads every choice at run time serves the whole
            // wavefront, element by element, and the specialised ones below stay as they are.
            if (e.scale_format == ASCQ_MM_SCALE_U64 && e.quant_mode != ASCQ_MM_QUANT_NONE &&
                __builtin_amdgcn_ballot_w64(((q[0].ctl | q[TJ - 1].ctl) & 2) != 0) != 0) {
                const bool odd = (lane & 1u) != 0;
#pragma unroll  // (a run-time index into the accumulators would move them to scratch memory)
                for (int i = 0; i < TI; ++i) {
                    const uint32_t lbase = (wm * TI + i) * 32u + 4u * g;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const uint32_t lrow_t = lbase + 8u * (r >> 2) + (r & 3);
                        const uint32_t row = row0 + lrow_t;
                        const float tok = TS[lrow_t];
                        float v[TJ];
#pragma unroll
                        for (int j = 0; j < TJ; ++j) {
                            v[j] = epilogue_value(e, acc[i][j][r] + bias_pre[j], q[j], tok, bias_post[j]);
                        }
                        if (e.activation == ASCQ_MM_ACT_SWIGLU) {
                            const float recv = __int_as_float(__builtin_amdgcn_mov_dpp(
                                __float_as_int(odd ? v[0] : v[TJ - 1]), 0xB1, 0xF, 0xF, true));  // lane ^ 1
                            const float o = swiglu(odd ? recv : v[0], odd ? v[TJ - 1] : recv, e.act_beta);
                            const uint32_t col = odd ? colw + 32u + (lrow - 1u) : colw + lrow;
                            if (row < row_end && col < N) {
                                static_cast<uint16_t*>(e.c)[static_cast<size_t>(row) * e.ldc + (col >> 1)] =
                                    static_cast<uint16_t>(to_bits16<kOut>(o));
                            }
                            continue;
                        }
#pragma unroll
                        for (int j = 0; j < TJ; ++j) {
                            if (cvalid[j] && row < row_end) {
                                const float o = e.activation == ASCQ_MM_ACT_FASTER_GELU ? faster_gelu(v[j]) : v[j];
                                static_cast<uint16_t*>(e.c)[static_cast<size_t>(row) * e.ldc + colw + j * 32u + lrow] =
                                    static_cast<uint16_t>(to_bits16<kOut>(o));
                            }
                        }
                    }
                }
                return;
            }
            const bool bias_post_on = e.bias_kind >= ASCQ_MM_BIAS_F32_POST;
            const bool gelu_on = e.activation == ASCQ_MM_ACT_FASTER_GELU;
            if (e.activation == ASCQ_MM_ACT_SWIGLU) {
                if (bias_post_on) {
                    store_all(std::true_type{}, std::false_type{}, std::true_type{});
                } else {
                    store_all(std::false_type{}, std::false_type{}, std::true_type{});
                }
            } else if (gelu_on) {
                if (bias_post_on) {
                    store_all(std::true_type{}, std::true_type{}, std::false_type{});
                } else {
                    store_all(std::false_type{}, std::true_type{}, std::false_type{});
                }
            } else if (bias_post_on) {
                store_all(std::true_type{}, std::false_type{}, std::false_type{});
            } else {
                store_all(std::false_type{}, std::false_type{}, std::false_type{});
            }
        } else {
            // the generic store reads both choices at run time (the host sends SwiGLU with these outputs elsewhere)
            store_all(std::false_type{}, std::false_type{}, std::false_type{});
        }
    };
    dispatch_out(e, run);
}

// kB: how B lies in memory.  0: [k, n] (or the fractal panels); 1: [n, k]; 2: the layout of ascq_pack_weight_w8
// (slabs of 16 columns, each a run of 1 KiB tiles of 64 k: lane l of a tile owns column l % 16, k 16 (l / 16) .. + 15).
// k is a multiple of BK, with k32Ragged of 16 (the pieces of a last, partial step that lie past k arrive as zeros).  With kB = 0 and an n
// that is no multiple of 16 the last tile is moved left until it ends at n (n >= BN then): the columns it shares with
// its neighbour are computed twice, with the same values.
// stages: S0, S1 (kRing: the array of the ring's stages)
template <int BM, int BN, bool kSplitK, bool kGrouped, int kB, int kForm, class... Stages>
__device__ __forceinline__ void gemm_dma_tile_at(const GemmParams& p, const TilePlace& at, uint32_t bidy, float* TS, const Stages&... stages)
{
    constexpr bool kBT = kB == 1, kBP = kB == 2;
    constexpr int kPieces = BN / 16;        // 16-byte pieces per B row
    constexpr int kAInstr = BM * BK / 1024 / 8;  // A DMA instructions per wavefront and K step
    constexpr int kBInstr = BK * BN / 1024 / 8;  // B DMA instructions per wavefront and K step
    static_assert(kAInstr >= 1 && kBInstr >= 1, "tile shape does not fit eight wavefronts");

    const uint32_t K = p.k, N = p.n, lda = ring_form(kForm) && p.lda != 0u ? p.lda : K;
    const uint32_t row0 = at.row0, row_end = at.row_end;
    const uint32_t n0 = kB == 0 && N % 16u != 0 && at.n0 + BN > N ? N - BN : at.n0;
    const int8_t* Bmat = at.b;
    uint32_t tid = threadIdx.x;
    if constexpr (kGrouped) {
        // The grouped kernel runs tiles in a loop: without this the compiler computes everything that depends only on
        // the lane once, ahead of the loop, and those registers are missing in the tile's main loop.
        asm volatile("" : "+v"(tid));
    }
    const uint32_t lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (tid < BM) {
        // read by the epilogue only; the barriers of the main loop order this store before those reads
        const uint32_t row = row0 + tid;
        TS[tid] = (p.epi.has_tok && row < row_end) ? p.epi.tok_scale[row] : 1.0f;
    }

    // ---- DMA sources: 4 A and 4 B instructions per wavefront and K step; lane owns LDS slot (instr * 64 + lane)
    auto a_slot = [&](int u) __attribute__((always_inline)) { return (wave * kAInstr + u) * 64u + lane; };
    auto b_slot = [&](int u) __attribute__((always_inline)) { return (wave * kBInstr + u) * 64u + lane; };
    auto line_piece = [](uint32_t s) __attribute__((always_inline)) { return (s & 7u) ^ ((s >> 4) & 7u); };  // of slot s of a [line][128] tile
    // 16x16x64 form: instructions of a half of A's rows, per wavefront (64 rows: four in all, issued by two wavefronts each,
    // so that every wavefront counts the same loads)
    constexpr int kHalfAll = BM * BK / 2048, kHalfInstr = kHalfAll >= 8 ? kHalfAll / 8 : 1;
    constexpr int kALoads = kForm == k16 ? 2 * kHalfInstr : kAInstr;
    uint32_t aoff[kALoads], boff[kBInstr];
#pragma unroll
    for (int u = 0; u < kALoads; ++u) {
        uint32_t s = a_slot(u), line = s >> 3;
        if constexpr (kForm == k16) {
            // loads of half h of every wavefront's rows: line r of its LDS array is row r % kRows of that half of wavefront
            // row r / kRows
            constexpr uint32_t kRows = BM * (BN / 64) / 16;
            s = (wave * kHalfInstr + u % kHalfInstr) % kHalfAll * 64u + lane;
            line = ((s >> 3) / kRows * 2u + u / kHalfInstr) * kRows + (s >> 3) % kRows;
        }
        uint32_t row = row0 + line;
        row = row < row_end ? row : row_end - 1;  // rows past the end are never stored: any valid row will do
        aoff[u] = (row - row0) * lda + 16u * line_piece(s);
    }
#pragma unroll
    for (int u = 0; u < kBInstr; ++u) {
        const uint32_t s = b_slot(u);
        if constexpr (kBP) {
            // one instruction = one packed tile: piece (slab j of the tile's BN / 16, k tile h of the step's two)
            // lands in LDS as it lies in memory; slabs past the last one are never stored
            const uint32_t piece = wave * kBInstr + u, j = piece >> 1, h = piece & 1u;
            const uint32_t slab0 = n0 >> 4, last = (N + 15u) / 16u - 1u;
            const uint32_t slab = slab0 + j < last ? slab0 + j : last;
            boff[u] = (slab - slab0) * (K * 16u) + h * 1024u + lane * 16u;
            continue;
        }
        if constexpr (kBT) {
            uint32_t col = n0 + (s >> 3);
            col = col < N ? col : N - 1u;  // columns past the end are never stored
            boff[u] = (col - n0) * K + 16u * line_piece(s);
            continue;
        }
        const uint32_t kb = s / kPieces, q = (s % kPieces) ^ b_swizzle<BN, kForm == k16 || ring_form(kForm)>(kb);
        uint32_t col = n0 + 16u * q;
        col = col + 16u <= N ? col : N - 16u;      // columns past the end are never stored
        // fractal B: panels of 32 columns, each a contiguous row-major [K][32] block
        boff[u] = p.b_nz ? ((col >> 5) * K + kb) * 32u + (col & 31u) : kb * N + (col - n0);
    }
    const uint32_t ldb = kBT ? 1u : kBP ? 16u : p.b_nz ? 32u : N;  // bytes from one k to the next
    // K range of this workgroup, in steps of BK
    const uint32_t all_steps = kForm == k32Ragged || ring_form(kForm) ? (K + BK - 1u) / BK : K / BK;
    uint32_t s_begin = 0, steps = all_steps;
    if constexpr (kSplitK) {
        s_begin = steps * bidy / p.k_splits;
        steps = steps * (bidy + 1u) / p.k_splits - s_begin;
    }
    const uint32_t partial = K % BK != 0 ? all_steps - 1u - s_begin : 0xFFFFFFFFu;  // the step with less than BK of k
    const int8_t* Abase = p.a + static_cast<size_t>(row0) * lda + static_cast<size_t>(s_begin) * BK;
    const int8_t* Bbase = Bmat + (kBT ? static_cast<size_t>(n0) * K : kBP ? static_cast<size_t>(n0 >> 4) * K * 16u : p.b_nz ? 0u : n0) +
                          static_cast<size_t>(s_begin) * BK * ldb;
    // A wavefront-uniform address, pinned to scalar registers: a load's address is then this base plus the lane's
    // 32-bit offset, which the load instruction adds itself (otherwise the compiler widens the offsets to 64 bits
    // ahead of the loop and adds the base per load: twice the registers and an addition per load).
    auto uniform = [](const int8_t* q) __attribute__((always_inline)) {
        const uint64_t v = reinterpret_cast<uint64_t>(q);
        uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
        uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
        asm volatile("" : "+s"(lo), "+s"(hi));
        return reinterpret_cast<const int8_t*>((static_cast<uint64_t>(hi) << 32) | lo);
    };
    auto issue = [&](uint32_t step, char* As, char* Bs) __attribute__((always_inline)) {
        const int8_t* ab = uniform(Abase + step * BK);
        const int8_t* bb = uniform(Bbase + static_cast<size_t>(step) * BK * ldb);
#pragma unroll
        for (int u = 0; u < kAInstr; ++u) asm volatile("" : "+v"(aoff[u]));
#pragma unroll
        for (int u = 0; u < kBInstr; ++u) asm volatile("" : "+v"(boff[u]));
        if (kForm == k32Ragged && step == partial) {  // uniform, once per tile at most
            const uint32_t left = K - (s_begin + step) * BK;
            const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(ab), 0, 0x7FFFFF00, 0x00020000);
            const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(bb), 0, 0x7FFFFF00, 0x00020000);
#pragma unroll
            for (int u = 0; u < kAInstr; ++u) {
                const uint32_t off = 16u * line_piece(a_slot(u)) < left ? aoff[u] : kPastEnd;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(As + (wave * kAInstr + u) * 1024), 16, off, 0, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < kBInstr; ++u) {
                const uint32_t at_k = kBT ? 16u * line_piece(b_slot(u)) : kBP ? ((wave * kBInstr + u) & 1u) * 64u : b_slot(u) / kPieces;
                const uint32_t off = at_k < left ? boff[u] : kPastEnd;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(Bs + (wave * kBInstr + u) * 1024), 16, off, 0, 0, 0);
            }
            return;
        }
#pragma unroll
        for (int u = 0; u < kAInstr; ++u) {
            __builtin_amdgcn_global_load_lds((gptr_t)(ab + aoff[u]), (lds_ptr_t)(As + (wave * kAInstr + u) * 1024), 16,
                                             0, 0);
        }
#pragma unroll
        for (int u = 0; u < kBInstr; ++u) {
            // split-K (few rows): the weights are read once, or by a handful of row tiles at the same time
            __builtin_amdgcn_global_load_lds((gptr_t)(bb + boff[u]), (lds_ptr_t)(Bs + (wave * kBInstr + u) * 1024), 16, 0,
                                             kSplitK ? 2 : 0);
        }
    };

    if constexpr (kForm == k16) {
        static_assert(!kSplitK, "K splits run the other form");
        struct Bases {
            const int8_t *a, *b;
        };
        auto bases = [&](uint32_t step) __attribute__((always_inline)) {
            return Bases{uniform(Abase + step * BK), uniform(Bbase + static_cast<size_t>(step) * BK * ldb)};
        };
        auto load = [&](const Bases& from, int u, const Stage& S) __attribute__((always_inline)) {
            if (u < kBInstr) {
                asm volatile("" : "+v"(boff[u]));
                __builtin_amdgcn_global_load_lds((gptr_t)(from.b + boff[u]), (lds_ptr_t)(S.b + (wave * kBInstr + u) * 1024), 16, 0, 0);
            } else {
                const int v = u - kBInstr;
                asm volatile("" : "+v"(aoff[v]));
                __builtin_amdgcn_global_load_lds((gptr_t)(from.a + aoff[v]),
                                                 (lds_ptr_t)(S.a[v / kHalfInstr] + (wave * kHalfInstr + v % kHalfInstr) % kHalfAll * 1024), 16, 0, 0);
            }
        };
        gemm_dma_body16<BM, BN, kGrouped, kB, kALoads, kBInstr>(p, at, n0, steps, wave, lane, bases, load, stages..., TS);
    } else if constexpr (ring_form(kForm)) {
        auto load = [&](uint32_t step, int u, char* S) __attribute__((always_inline)) {
            // how much of the row's k is left from here on, nothing past the last step; a piece past it brings zeros
            const uint32_t at_k = step < steps ? step : 0u, left = step < steps ? K - step * BK : 0u;
            if (u < kAInstr) {
                const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(uniform(Abase + at_k * BK)), 0, 0x7FFFFF00, 0x00020000);
                const uint32_t off = 16u * line_piece(a_slot(u)) < left ? aoff[u] : kPastEnd;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(S + (wave * kAInstr + u) * 1024), 16, off, 0, 0, 0);
            } else {
                const int v = u - kAInstr;
                const __amdgpu_buffer_rsrc_t r =
                    __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(uniform(Bbase + static_cast<size_t>(at_k) * BK * ldb)), 0, 0x7FFFFF00, 0x00020000);
                const uint32_t k0 = kBT ? 16u * line_piece(b_slot(v)) : kBP ? ((wave * kBInstr + v) & 1u) * 64u : b_slot(v) / kPieces;
                const uint32_t off = k0 < left ? boff[v] : kPastEnd;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(S + BM * BK + (wave * kBInstr + v) * 1024), 16, off, 0, 0, 0);
            }
        };
        gemm_ring_body<BM, BN, kB, (sizeof(Stages) + ...) / sizeof(char*), kAInstr + kBInstr, kForm == kRingHalf>(p, at, n0, steps, wave, lane, load, stages..., TS);
    } else {
        auto run = [&](const Stage& S0, const Stage& S1) __attribute__((always_inline)) {
            gemm_dma_body32<BM, BN, kSplitK, kGrouped, kB>(p, at, n0, steps, bidy, wave, lane, issue, S0.a[0], S0.b, S1.a[0], S1.b, TS);
        };
        run(stages...);
    }
}

inline bool gemm_half_output(const GemmParams& p)
{
    return p.epi.quant_mode != ASCQ_MM_QUANT_NONE && (p.epi.out_dtype == ASCQ_F16 || p.epi.out_dtype == ASCQ_BF16);
}

// The matrix instruction of the plain matmul's 256-row tiles (its smaller ones run the 32 x 32 x 32 one, the ring tiles the other; grouped
// tiles: launch_gemm_dma_group).  The 16 x 16 x 64 form moves half the sums, which is what counts where the power limit sets the
// clock, and its loads have longer to arrive; but a tile starts with two stages of loads where the other form waits for one, and
// its epilogue holds more code.  Time of the 16 x 16 x 64 form over the other's, geometric means of random calls of 513 to 8192 rows with
// up to 64 / 65 to 512 / more tiles: k = 128 1.06 / 1.05 / 1.08, 512 1.03 / 1.00 / 1.03, 768 1.01 / 1.00 / 1.05, 896 1.01 / 0.98 /
// 0.98, 1024 1.00 / 0.98 / 1.01, 1280 1.00 / 0.97 / 1.00, 1536 0.99 / 0.98 / 0.94, 2048 1.00 / 0.95, 4096 0.99 / 0.93 / 0.89.  In us
// with the quantiser: 2048 x 4096 x 11008 98.1 and 88.3; 1024 x 11008 x 4096 (64 tiles) 107.8 and 103.9.  Outputs other than half and
// bfloat16 are what the 32 x 32 x 32 form writes from registers.
inline int gemm_dma_form(const GemmParams& p)
{
    if (p.k % BK != 0) {
        return k32Ragged;
    }
    const uint64_t tiles = static_cast<uint64_t>((p.m + 255u) / 256u) * ((p.n + 255u) / 256u), cus = device_compute_units();
    const bool middle = 4u * tiles > cus && tiles <= 2u * cus;
    return gemm_half_output(p) && p.k >= (middle ? 896u : 1536u) ? k16 : k32;
}

// The plain matmul: tile number `bid` of the launch (before the XCD remapping), column tiles counted from col_begin,
// row tiles innermost so that the tiles an XCD runs side by side share their B columns.
template <int BM, int BN, bool kSplitK, int kB, int kForm>
__device__ __forceinline__ void gemm_dma_tile(const GemmParams& p, uint32_t col_begin, uint32_t bid, uint32_t bidy,
                                              const Stage& S0, const Stage& S1, float* TS)
{
    const uint32_t total = p.tiles_m * p.tiles_n;
    const uint32_t t = xcd_remap(bid, total);
    if (t >= total) {
        return;
    }
    // bands of 8 row tiles, inside a band column by column (band_order): an XCD's share stays a block of a few columns
    // by 8 rows whose rows of A and columns of B it reuses from its L2, however many rows the matrix has
    uint32_t ms, tn;
    band_order(t, p.tiles_m, p.tiles_n, ms, tn);
    const TilePlace at{ms * BM, p.m, col_begin + tn * BN, p.b, 0};
    gemm_dma_tile_at<BM, BN, kSplitK, false, kB, kForm>(p, at, bidy, TS, S0, S1);
}

// The LDS stages S0 and S1 of a kernel (an array that nothing reads takes no space).
#define ASCQ_DMA_STAGES(kForm, BM, BN)                                                                       \
    __shared__ __attribute__((aligned(1024))) char A0[BM * BK / (kForm == k16 ? 2 : 1)], A1[sizeof(A0)];      \
    __shared__ __attribute__((aligned(1024))) char A0h[sizeof(A0)], A1h[sizeof(A0)], B0[BK * BN], B1[BK * BN]; \
    const Stage S0{{A0, A0h}, B0}, S1{{A1, A1h}, B1}

template <int BM, int BN, bool kSplitK, int kB, int kForm>
__global__ __launch_bounds__(kThreads, (BM * BK + BK * BN) * 2 <= 65536 ? 2 : 1) void gemm_dma_kernel(
    GemmParams p, uint32_t col_begin)
{
    ASCQ_DMA_STAGES(kForm, BM, BN);
    __shared__ __attribute__((aligned(16))) float TS[BM];  // token scales of the tile's rows (1.0f when there are none)
    gemm_dma_tile<BM, BN, kSplitK, kB, kForm>(p, col_begin, blockIdx.x, blockIdx.y, S0, S1, TS);
}

// One launch for a matrix whose last round of 256 x 256 tiles would be mostly empty: workgroups [0, wide_wgs) run the
// 256 x 256 tiles of the first `p.tiles_n` tile columns, the rest 256 x 128 tiles of the remaining columns.  A compute
// unit that has finished its wide tile takes a narrow one at once, without the drain between two launches.
template <int kB, int kForm>
__global__ __launch_bounds__(kThreads, 1) void gemm_dma_dual_kernel(GemmParams p, uint32_t wide_wgs,
                                                                    uint32_t narrow_tiles_n, uint32_t col_begin)
{
    ASCQ_DMA_STAGES(kForm, 256, 256);
    __shared__ __attribute__((aligned(16))) float TS[256];
    if (blockIdx.x < wide_wgs) {
        gemm_dma_tile<256, 256, false, kB, kForm>(p, 0u, blockIdx.x, 0u, S0, S1, TS);
    } else {
        GemmParams q = p;
        q.tiles_n = narrow_tiles_n;
        gemm_dma_tile<256, 128, false, kB, kForm>(q, col_begin, blockIdx.x - wide_wgs, 0u, S0, S1, TS);
    }
}

}  // namespace

// One launch of the plain matmul's kernels.
struct DmaLaunch {
    enum Shape { kWide, kNarrow, kBoth, kSmall, kSplit } shape;  // 256 x 256, 256 x 128, both, 128 x 128, those with K split
    dim3 grid;
    uint32_t col_begin, wide_wgs, narrow_tiles_n;
};

namespace {

template <int kB, int kForm>
void run_dma_layout(const GemmParams& p, const DmaLaunch& l, hipStream_t st)
{
    if (l.shape == DmaLaunch::kBoth) {
        gemm_dma_dual_kernel<kB, kForm><<<l.grid, kThreads, 0, st>>>(p, l.wide_wgs, l.narrow_tiles_n, l.col_begin);
    } else if (l.shape == DmaLaunch::kWide) {
        gemm_dma_kernel<256, 256, false, kB, kForm><<<l.grid, kThreads, 0, st>>>(p, l.col_begin);
    } else if constexpr (kForm != k16) {
        if (l.shape == DmaLaunch::kNarrow) {
            gemm_dma_kernel<256, 128, false, kB, kForm><<<l.grid, kThreads, 0, st>>>(p, l.col_begin);
        } else if (l.shape == DmaLaunch::kSmall) {
            gemm_dma_kernel<128, 128, false, kB, kForm><<<l.grid, kThreads, 0, st>>>(p, l.col_begin);
        } else {
            gemm_dma_kernel<128, 128, true, kB, kForm><<<l.grid, kThreads, 0, st>>>(p, l.col_begin);
        }
    }
}

// b_layout: 0 [k, n], 1 [n, k], 2 packed by ascq_pack_weight_w8
template <int kForm>
void run_dma(const GemmParams& p, const DmaLaunch& l, int b_layout, hipStream_t st)
{
    if (b_layout == 2) {
        run_dma_layout<2, kForm>(p, l, st);
    } else if (b_layout == 1) {
        run_dma_layout<1, kForm>(p, l, st);
    } else {
        run_dma_layout<0, kForm>(p, l, st);
    }
}

}  // namespace

// matmul_w8a8_ragged.hip (k32Ragged) and matmul_w8a8_long.hip (k16): translation units of their own, the kernels take
// minutes to compile
void run_dma_ragged(const GemmParams& p, const DmaLaunch& l, int b_layout, hipStream_t st);
void run_dma_long(const GemmParams& p, const DmaLaunch& l, int b_layout, hipStream_t st);

}  // namespace ascq
