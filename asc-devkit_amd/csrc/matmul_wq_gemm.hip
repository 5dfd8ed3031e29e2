// Half x quantised weights with many activation rows: a half GEMM whose B-tile loader de-quantises int8 weights kept as
// [n, k] (W8A16) or int4 weights packed by ascq_pack_weight_w4 (W4A16).
//
// What bounds it is the matrix pipe, and with it the power limit: every weight becomes a half once per row tile, which
// at 256 rows costs the vector ALU about a quarter of the clocks the matrix instructions take, and the two run side by
// side.  v_mfma_f32_16x16x32_f16 instead of the 32 x 32 x 16 form: on random operands a loop of nothing but matrix
// instructions reaches 1880 against 1640 TFLOP/s (it moves half the sums per product, and the clock is set by the power),
// which is 4 to 6 % of this kernel.  k = 8192, n = 28672, before (one pass over the weights per 16 rows; 128 x 128 tiles)
// and now: int4 512 rows 1035 -> 207 us (1160 TFLOP/s), int8 2048 rows 1120 -> 810 us (1190), 512 rows 310 -> 216 us.  A workgroup is 8
// wavefronts on a BM x BN tile, K step 64, two LDS stages.  x goes from memory to LDS without registers
// (global_load_lds_dwordx4); the raw bytes of B take the way through registers (16 or 32 per thread and step, fetched
// two steps ahead), are de-quantised with the operators' own roundings and written to LDS as halves, one 16-byte piece
// behind the matrix instructions of each quarter of a step.  Both tiles lie in LDS as lines of 64 halves (128 bytes), one
// 16-byte piece of which is the operand of v_mfma_f32_16x16x32_f16 as it lies; neither reads nor writes meet a bank twice
// (wq_swizzle; with pieces swizzled by half the line number alone every write of the B tile cost 9 cycles more, 21 % of the
// LDS cycles: 2048 x 8192 x 28672 813 -> 809 us, 300 x 4096 x 11008 64 -> 62).  The barriers stand before a step's second and last quarter, whose operands are in registers by
// then: behind them the matrix pipe has work while loads are issued and operands read.  At 2048 rows of int8 the matrix
// pipe works in 69 % of the clocks, which the power limit holds at 1.64 GHz.
#include <type_traits>
#include <utility>

#include "ascq_common.h"
#include "ascq_device.h"
#include "matmul_wq_gemm.h"

namespace ascq {
namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) const void* gptr_t;

constexpr uint32_t kBK = 64;  // halves of a K step
constexpr int kThreads = 512;

template <class F, int... I>
__device__ __forceinline__ void wq_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void wq_for(F&& f)
{
    wq_for_impl(f, std::make_integer_sequence<int, N>{});
}

// One of the two LDS stages of a tile.
struct WqStage {
    char* a[2];  // the first and the second half of every wavefront's rows: distinct arrays, like the stages
    char* b;
};

// One BM x BN tile of rows from row0 and columns from n0.  BN = 256: wavefronts 2 (M) x 4 (N); BN = 128: 4 x 2.  A
// wavefront owns BM / kWM rows by 64 columns.  kOnce: a step's loads go out at once (BN = 128, see launch_wq_gemm).
template <int BM, int BN, bool kInt4, bool kOff, bool kOnce>
__device__ __forceinline__ void wq_tile(const WqParams& p, uint32_t row0, uint32_t n0, const WqStage& S0, const WqStage& S1)
{
    constexpr int kWN = BN / 64, kWM = 8 / kWN, NA = BM / 16 / kWM, NH = NA / 2, TJ = 4;
    constexpr int kAInstr = BM * 128 / 1024 / 8;           // direct-to-LDS instructions per wavefront and step
    constexpr int kParts = BN / 64;                        // 16-byte pieces of the B tile per thread and step
    static_assert(NH >= 1 && NH * 32 * kWM == BM && kAInstr >= 1 && (kParts == 4 || kParts == 2), "tile shape");
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave / kWN, wn = wave % kWN;

    // ---- A: lane owns LDS slot (instr * 64 + lane) of 16 bytes of a half's array: line slot / 8, piece position ^ wq_swizzle(line);
    // line r is row r % kRows of that half of wavefront row r / kRows
    constexpr int kHalf = kAInstr / 2;                     // instructions per half
    constexpr uint32_t kRows = NH * 16u;
    static_assert(kAInstr % 2 == 0, "the halves are whole instructions");
    const uint32_t row_bytes = p.k * 2u;
    uint32_t aoff[kAInstr];
#pragma unroll
    for (int u = 0; u < kAInstr; ++u) {
        const uint32_t s = (wave * kHalf + u % kHalf) * 64u + lane, line = s >> 3;
        const uint32_t r = (line / kRows * 2u + u / kHalf) * kRows + line % kRows;
        const uint32_t row = row0 + r < p.m ? r : p.m - 1u - row0;  // rows past the end are never stored
        aoff[u] = row * row_bytes + (((s & 7u) ^ wq_swizzle(line)) << 4);
    }
    const char* Abase = reinterpret_cast<const char*>(p.x) + static_cast<size_t>(row0) * row_bytes;
    const uint32_t last = p.k / kBK - 1u;
    // a scalar base plus the lane's 32-bit offset, which the load instruction adds itself; past the end the last step's, into
    // a stage nobody reads
    auto a_base = [&](uint32_t step) __attribute__((always_inline)) {
        const uint64_t v = reinterpret_cast<uint64_t>(Abase + (step < last ? step : last) * 128u);
        uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
        uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
        asm volatile("" : "+s"(lo), "+s"(hi));
        return reinterpret_cast<const char*>((static_cast<uint64_t>(hi) << 32) | lo);
    };
    auto load_rows = [&](const char* base, int u, const WqStage& S) __attribute__((always_inline)) {
        asm volatile("" : "+v"(aoff[u]));
        __builtin_amdgcn_global_load_lds((gptr_t)(base + aoff[u]), (lds_ptr_t)(S.a[u / kHalf] + (wave * kHalf + u % kHalf) * 1024u), 16, 0, 0);
    };

    // ---- B: the thread's column of the tile and its first piece (of 8 weights) in the column's line
    uint32_t bcol, bpiece, boff;
    if constexpr (kInt4) {
        // a K step is half a packed tile: 32 lanes of 16 bytes, lane column l % 16, k 32 (l / 16) .. + 31
        constexpr uint32_t kPer = 4u / kParts;             // threads that share such a lane's 16 bytes
        // (neighbouring threads take both halves of a column's 64 k, so that eight of them write eight pieces apart)
        const uint32_t s = tid / kPer, l = kParts == 4 ? ((s >> 1) & 15u) | (s & 1u) << 4 : s & 31u;
        bcol = (s >> 5) * 16u + (l & 15u);
        bpiece = 4u * (l >> 4) + (tid % kPer) * kParts;
        boff = (s >> 5) * (p.k * 8u) + l * 16u + (tid % kPer) * 8u;
    } else {
        constexpr uint32_t kPer = 8u / kParts;             // threads that share a column's 64 bytes
        bcol = tid / kPer;
        bpiece = (tid % kPer) * kParts;
        boff = bcol * p.k + bpiece * 8u;
    }
    // columns past n fall outside the buffer: zeros arrive (their results are never stored)
    const uint32_t left = p.n - n0 < BN ? p.n - n0 : BN;
    const uint64_t wbase = kInt4 ? static_cast<uint64_t>(n0 / 16u) * (p.k * 8u) : static_cast<uint64_t>(n0) * p.k;
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.w) + wbase, 0, static_cast<int>(kInt4 ? (left + 15u) / 16u * (p.k * 8u) : left * p.k), 0x00020000);
    const uint32_t gcol = n0 + (bcol < left ? bcol : left - 1u);
    f16x2 csc = both(0.0f), cof = both(0.0f);              // int8: scale and offset belong to the column
    if constexpr (!kInt4) {
        const uint32_t sb = p.scale ? p.scale[gcol] : p.scale_bits;
        const uint32_t ob = kOff ? (p.scale ? p.offset[gcol] : p.offset_bits) : 0u;
        csc = as_h2(sb * 0x10001u);
        cof = as_h2(ob * 0x10001u);
    }
    __amdgpu_buffer_rsrc_t rs = rw, ro = rw;               // int4: scale and offset of a group of k and a column
    uint32_t poff = 0;
    if constexpr (kInt4) {
        const int bytes = static_cast<int>((p.k >> (5u + p.gs_shift)) * p.n * 2u);
        rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.scale), 0, bytes, 0x00020000);
        ro = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kOff ? p.offset : p.scale), 0, bytes, 0x00020000);
        poff = gcol * 2u + (p.gs_shift == 0 ? (bpiece >> 2) * p.n * 2u : 0u);
    }
    // Raw bytes of a step: two parts of two pieces each, fetched apart (BN = 128: one part).
    constexpr int kFetches = kParts / 2;
    struct Raw {
        u32x4 b[kInt4 ? 1 : kFetches];
        uint32_t sc, of;
    };
    // part `which`: its weights, with the last part the parameters
    constexpr int kPartLoads = 1, kParamLoads = kInt4 ? (kOff ? 2 : 1) : 0;
    auto fetch = [&](Raw& raw, uint32_t step, int which) __attribute__((always_inline)) {
        step = step < last ? step : last;                  // past the end: the last step's, into a stage nobody reads
        const uint32_t at = kInt4 ? step * 512u : step * kBK;
        if constexpr (kInt4) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(rw, boff + 8u * which, at, 0);
            raw.b[0][2 * which] = v[0];
            raw.b[0][2 * which + 1] = v[1];
        } else {
            raw.b[which] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, boff + 16u * which, at, 0));
        }
        if constexpr (kInt4) {
            if (which == kFetches - 1) {
                // the group of 32 k 2 step + (0 or 1); the lane's half matters for groups of 32 only
                const uint32_t pat = ((2u * step) >> p.gs_shift) * p.n * 2u;
                raw.sc = __builtin_amdgcn_raw_buffer_load_b16(rs, poff, pat, 0);
                raw.of = kOff ? __builtin_amdgcn_raw_buffer_load_b16(ro, poff, pat, 0) : 0u;
            }
        }
    };
    const uint32_t bline = bcol * 128u, bswz = wq_swizzle(bcol);
    WqMasks mk = p.mk;
    asm volatile("" : "+v"(mk.exp_even), "+v"(mk.exp_odd));  // (an instruction takes one scalar operand)
    // pair c of piece q of the thread's share of a step; the finished piece goes to LDS
    u32x4 piece;
    auto dequant_pair = [&](const Raw& raw, int q, int c) __attribute__((always_inline)) {
        if constexpr (kInt4) {
            piece[c] = pair_of_i4<kOff>(raw.b[0][q], c, as_h2(raw.sc * 0x10001u), as_h2(raw.of * 0x10001u), mk);
        } else {
            piece[c] = pair_of_i8<kOff>(raw.b[q >> 1][2 * (q & 1) + (c >> 1)], c & 1, csc, cof);
        }
    };
    auto write_piece = [&](char* Bs, int q) __attribute__((always_inline)) {
        *reinterpret_cast<u32x4*>(Bs + bline + (((bpiece + q) ^ bswz) << 4)) = piece;
    };

    f32x4 acc[NA][TJ];
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            asm volatile("" : "+v"(acc[i][j]));
        }

    // ---- operands: lane l holds line l % 16 of a block of 16 and the 8 k of piece 4 ks + l / 16.  A step is four
    // quarters: quarter q multiplies half q / 2 of the wavefront's rows with the 32 k of sub-step ks = q % 2.
    const uint32_t lc = lane & 15u, lq = lane >> 4;
    uint32_t foff[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) foff[ks] = lc * 128u + (((4u * ks + lq) ^ wq_swizzle(lc)) << 4);
    f16x8 af[2][NH], bf[2][TJ];
    auto load_a = [&](const WqStage& S, int q, int i) __attribute__((always_inline)) {
        af[q & 1][i] = *reinterpret_cast<const f16x8*>(S.a[q >> 1] + (wm * NH + i) * 2048u + foff[q & 1]);
    };
    auto load_b = [&](const WqStage& S, int ks, int j) __attribute__((always_inline)) {
        bf[ks][j] = *reinterpret_cast<const f16x8*>(S.b + wn * 8192u + j * 2048u + foff[ks]);
    };
    // Matrix instruction number n of quarter q.  Written as an instruction that accumulates in place: left to itself the
    // compiler gave it another destination than its addend and moved accumulators about, spilling some.  (Its operands
    // come from LDS reads, which the compiler waits for; no vector instruction touches them or the sums in the loop.)
    auto mfma = [&](int q, int n) __attribute__((always_inline)) {
        f32x4& c = acc[(q >> 1) * NH + n / TJ][n % TJ];
        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(af[q & 1][n / TJ]), "v"(bf[q & 1][n % TJ]));
    };
    // One quarter: its NH * TJ matrix instructions, the LDS reads `read(r)`, r < kReads, one behind each of the first, loads
    // `load(u)`, u < kLoads, behind the odd ones, and a piece of weights de-quantised pair by pair behind four later ones.
    // The order is the one written.
    constexpr int kM = NH * TJ;
    auto quarter = [&](auto qq, auto reads, auto&& read, auto part, const Raw& raw, char* Bs, auto loads, auto&& load) __attribute__((always_inline)) {
        constexpr int q = decltype(qq)::value, kReads = decltype(reads)::value, kPart = decltype(part)::value, kLoads = decltype(loads)::value;
        constexpr int kPer = (kReads + kM - 1) / kM, kLoadPer = (2 * kLoads + kM - 1) / kM;
        wq_for<kM>([&](auto nn) {
            constexpr int n = decltype(nn)::value;
            mfma(q, n);
            wq_for<kPer>([&](auto r) {
                constexpr int i = n * kPer + decltype(r)::value;
                if constexpr (i < kReads) read(std::integral_constant<int, i>{});
            });
            if constexpr (n % 2 == 1) {
                wq_for<kLoadPer>([&](auto r) {
                    constexpr int u = n / 2 * kLoadPer + decltype(r)::value;
                    if constexpr (u < kLoads) load(u);
                });
            }
            if constexpr (kPart >= 0) {
                // pairs behind instructions kM - 5 .. kM - 2 (of at least 4)
                constexpr int first = kM >= 8 ? kM - 5 : 0;
                if constexpr (n >= first && n < first + 4) dequant_pair(raw, kPart, n - first);
                if constexpr (n == first + 3) write_piece(Bs, kPart);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto first_operands = [&](const WqStage& S, int i) __attribute__((always_inline)) {
        if (i == 0 || i > NH) {
            load_b(S, 0, i == 0 ? 0 : i - NH);
        } else {
            load_a(S, 0, i - 1);
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
    // Step s in stage X, step s + 1 in Y; `next` holds the raw bytes of step s + 1, `next2` those of s + 2.  When quarter 1
    // begins, every wavefront has read X's weights and the first half of its rows, when quarter 3 begins, the second half,
    // and Y's weights are written: a barrier there, and what was freed takes the loads of step s + 2, what was used up of
    // the raw bytes those of step s + 3.  So the loads have one and a half steps to arrive (int4's parameters one), where one wait for all of
    // them at a step's end left them one.  The waits count the loads behind the ones that are needed: before quarter 1 the second
    // half of this step's rows and the last raw bytes of step s + 1 (behind them all of a step's loads), before quarter 3 the
    // first half of the next step's rows and the first raw bytes of step s + 2, with int4 its parameters.  (Without a count of its own
    // for the raw bytes the compiler waits for everything where they cross the loop's end.)
    // `ahead`: how many steps follow, 2 for two or more.  The last step but one issues no loads: nobody would use what they bring, so the
    // compiler may leave those into registers out, and a count that includes them would no longer hold the waits back.
    // (BN = 128, two small workgroups on a unit: a quarter is four matrix instructions, and one barrier, before quarter 3, is better: 100 x
    // 4096 x 4096 int4 40.0 us, 42.4 with two.)
    constexpr bool kMid = kFetches == 2;
    constexpr int kPartAll = kFetches * kPartLoads + kParamLoads, kLate = kPartLoads + kParamLoads;  // fetches of a step; behind quarter 3
    constexpr int kEarly = kPartAll - kLate, kRowsLate = kMid ? kHalf : kAInstr;                      // fetches, rows behind quarter 1 / 3
    auto step = [&](uint32_t s, const WqStage& X, const WqStage& Y, Raw& next, Raw& next2, auto ahead) __attribute__((always_inline)) {
        constexpr bool kSteady = decltype(ahead)::value == 2, kMore = decltype(ahead)::value != 0;
        constexpr std::integral_constant<int, kSteady && kMid ? kHalf + kEarly : 0> early{};
        constexpr std::integral_constant<int, kSteady ? kRowsLate + 1 : 0> late{};
#pragma unroll
        for (int q = 0; q < 2; ++q) asm volatile("" : "+v"(foff[q]));
        const char* const base = a_base(s + 2u);
        quarter(std::integral_constant<int, 0>{}, std::integral_constant<int, TJ + NH>{}, [&](auto r) __attribute__((always_inline)) {
            constexpr int i = decltype(r)::value;
            if constexpr (i < TJ) {
                load_b(X, 1, i);
            } else {
                load_a(X, 1, i - TJ);
            }
        }, std::integral_constant<int, kMore && kParts == 4 ? 1 : -1>{}, next, Y.b, std::integral_constant<int, 0>{}, [](int) {});
        if constexpr (kMid) arrive(std::integral_constant<int, kMore ? kAInstr + kPartAll : 0>{});
        quarter(std::integral_constant<int, 1>{}, std::integral_constant<int, NH>{}, [&](auto r) __attribute__((always_inline)) {
            load_a(X, 2, decltype(r)::value);
        }, std::integral_constant<int, !kMore ? -1 : kParts == 4 ? 2 : 1>{}, next, Y.b, early, [&](int u) __attribute__((always_inline)) {
            if (u < kHalf) {
                load_rows(base, u, X);
            } else {
                fetch(next, s + 3u, 0);  // (its first part was used up by quarter 0)
            }
        });
        quarter(std::integral_constant<int, 2>{}, std::integral_constant<int, NH>{}, [&](auto r) __attribute__((always_inline)) {
            load_a(X, 3, decltype(r)::value);
        }, std::integral_constant<int, kMore && kParts == 4 ? 3 : -1>{}, next, Y.b, std::integral_constant<int, 0>{}, [](int) {});
        if constexpr (kMore) {
            arrive(std::integral_constant<int, !kMid ? 0 : !kSteady ? kHalf + kPartAll : kInt4 ? kHalf + kEarly : kAInstr + kPartAll>{});
            auto late_load = [&](int u) __attribute__((always_inline)) {
                if (u < kRowsLate) {
                    load_rows(base, kAInstr - kRowsLate + u, X);
                } else {
                    fetch(next, s + 3u, kFetches - 1);
                }
            };
            static_assert(!kOnce || !kMid, "one barrier per step");
            constexpr int kAtOnce = kOnce ? decltype(late)::value : 0;
#pragma unroll
            for (int u = 0; u < kAtOnce; ++u) late_load(u);
            __builtin_amdgcn_sched_barrier(0);
            quarter(std::integral_constant<int, 3>{}, std::integral_constant<int, NH + TJ>{}, [&](auto r) __attribute__((always_inline)) {
                first_operands(Y, decltype(r)::value);
            }, std::integral_constant<int, kSteady ? 0 : -1>{}, next2, X.b, std::integral_constant<int, decltype(late)::value - kAtOnce>{}, late_load);
        } else {
            wq_for<kM>([&](auto n) { mfma(3, decltype(n)::value); });
        }
    };

    // The loads in the order in which the loop would have issued them.
    Raw r0, r1;
#pragma unroll
    for (int w = 0; w < kFetches; ++w) fetch(r0, 0, w);
    auto prologue_rows = [&](uint32_t st, int h, const WqStage& S) __attribute__((always_inline)) {
        const char* const base = a_base(st);
#pragma unroll
        for (int u = 0; u < kHalf; ++u) load_rows(base, h * kHalf + u, S);
    };
    auto in_order = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };  // the waits count them
    in_order();
    prologue_rows(0, 0, S0);
    in_order();
    if constexpr (kEarly != 0) fetch(r1, 1, 0);
    in_order();
    prologue_rows(0, 1, S0);
    in_order();
    fetch(r1, 1, kFetches - 1);
    in_order();
    wq_for<kParts>([&](auto q) {
#pragma unroll
        for (int c = 0; c < 4; ++c) dequant_pair(r0, decltype(q)::value, c);
        write_piece(S0.b, decltype(q)::value);
    });
    in_order();
    prologue_rows(1, 0, S1);
    in_order();
    if constexpr (kEarly != 0) fetch(r0, 2, 0);
    arrive(std::integral_constant<int, kMid ? kEarly + kHalf + kLate + kHalf + kEarly : kHalf>{});
    prologue_rows(1, 1, S1);
    in_order();
    fetch(r0, 2, kFetches - 1);
    in_order();
#pragma unroll
    for (int c = 0; c < 4; ++c) dequant_pair(r1, 0, c);
    write_piece(S1.b, 0);
#pragma unroll
    for (int i = 0; i < NH + TJ; ++i) first_operands(S0, i);
    // At the top of step s (stage X, other stage Y): its first operands are in registers, piece 0 of step s + 1 is in Y, the
    // rest of it in raw set (s + 1) % 2, step s + 2's raw bytes are on their way into set s % 2.
    const uint32_t steps = last + 1u;
    constexpr std::integral_constant<int, 2> two{};
    uint32_t s = 0;
    for (; s + 2u < steps; s += 2u) {
        step(s, S0, S1, r1, r0, two);
        step(s + 1u, S1, S0, r0, r1, two);
    }
    if (s + 1u < steps) {
        step(s, S0, S1, r1, r0, std::integral_constant<int, 1>{});
    }
    {
        const bool odd = (steps & 1u) != 0;
        const WqStage X{{odd ? S0.a[0] : S1.a[0], odd ? S0.a[1] : S1.a[1]}, odd ? S0.b : S1.b};
        step(last, X, X, r1, r0, std::integral_constant<int, 0>{});
    }
    // The last sums are on their way through the matrix pipe, which the compiler does not know: it sees them changed behind
    // the wait, so that nothing that reads them can move ahead of it.  (check_matrix_asm.py looks through the machine code
    // for what this cannot rule out, a copy inside the loop.)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < NA; ++i) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) asm volatile("" : "+v"(acc[i][j]));
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the end

    // ---- register r of lane l in a 16 x 16 block: row 4 (l / 16) + r, column l % 16
    const uint32_t colw = n0 + wn * 64u, roww = row0 + wm * (NA * 16u) + 4u * lq;
    if (!p.out_f32 && p.n % 4u == 0) {
        // half output: a 4 x 4 transposition inside each four neighbouring lanes (two exchanges of packed pairs) leaves
        // lane b of the four with columns 4 (l / 4) .. + 3 of block b: one 8-byte store per lane and row, and the 16
        // lanes of a row write one full 128-byte line
        const bool b0 = (lane & 1u) != 0, b1 = (lane & 2u) != 0;
        const uint32_t col = colw + 16u * (lane & 3u) + (lc & 12u);
#pragma unroll
        for (int i = 0; i < NA; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t row = roww + i * 16u + r;
                uint32_t h[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) h[j] = f32_to_half_bits(acc[i][j][r]);
                const uint32_t give = b0 ? h[0] | (h[2] << 16) : h[1] | (h[3] << 16);
                const uint32_t got = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(give), 0xB1, 0xF, 0xF, true));  // lane ^ 1
                const uint32_t lo = b0 ? (got & 0xFFFFu) | (h[1] << 16) : h[0] | (got << 16);
                const uint32_t hi = b0 ? (got >> 16) | (h[3] << 16) : h[2] | (got & 0xFFFF0000u);
                const uint32_t got2 = static_cast<uint32_t>(
                    __builtin_amdgcn_mov_dpp(static_cast<int>(b1 ? lo : hi), 0x4E, 0xF, 0xF, true));  // lane ^ 2
                if (row < p.m && col < p.n) {
                    __builtin_nontemporal_store(b1 ? u32x2{got2, hi} : u32x2{lo, got2},
                                                reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p.y) + static_cast<size_t>(row) * p.n + col));
                }
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const uint32_t col = colw + j * 16u + lc;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t row = roww + i * 16u + r;
                if (row < p.m && col < p.n) {
                    const size_t idx = static_cast<size_t>(row) * p.n + col;
                    if (p.out_f32) {
                        static_cast<float*>(p.y)[idx] = acc[i][j][r];
                    } else {
                        static_cast<uint16_t*>(p.y)[idx] = static_cast<uint16_t>(f32_to_half_bits(acc[i][j][r]));
                    }
                }
            }
        }
    }
}

// 256 x 256: the first p.full tiles are run as they are; each of the others, which would leave part of the last
// round of the chip idle, is run by two workgroups with 128 x 256 tiles.
template <int BM, int BN, bool kInt4, bool kOff, bool kOnce>
__global__ __launch_bounds__(kThreads) void wq_gemm_kernel(WqParams p)
{
    __shared__ __attribute__((aligned(1024))) char A0[BM * 64], A0h[BM * 64], A1[BM * 64], A1h[BM * 64], B0[BN * 128], B1[BN * 128];
    const WqStage S0{{A0, A0h}, B0}, S1{{A1, A1h}, B1};
    const uint32_t tiles = p.tiles_m * p.tiles_n;
    uint32_t tm, tn;
    if (BM == 128 || blockIdx.x < p.full) {
        const uint32_t t = xcd_remap(blockIdx.x, BM == 128 ? tiles : p.full);
        if (t == 0xFFFFFFFFu) {
            return;  // whole workgroup (the launch is rounded up to a multiple of 8)
        }
        band_order(t, p.tiles_m, p.tiles_n, tm, tn);
        wq_tile<BM, BN, kInt4, kOff, kOnce>(p, tm * BM, tn * BN, S0, S1);
    } else if constexpr (BM == 256) {
        const uint32_t t = xcd_remap(blockIdx.x - p.full, 2u * (tiles - p.full));
        if (t == 0xFFFFFFFFu) {
            return;
        }
        band_order(p.full + t / 2u, p.tiles_m, p.tiles_n, tm, tn);
        const uint32_t row0 = tm * 256u + (t & 1u) * 128u;
        if (row0 < p.m) {
            wq_tile<128, BN, kInt4, kOff, kOnce>(p, row0, tn * BN, S0, S1);
        }
    }
}

template <int BM, int BN, bool kOnce = false>
void wq_launch(WqParams p, bool int4, bool has_offset, hipStream_t st)
{
    p.tiles_m = (p.m + BM - 1u) / BM;
    p.tiles_n = (p.n + BN - 1u) / BN;
    const uint32_t tiles = p.tiles_m * p.tiles_n;
    const uint32_t blocks = BM == 256 ? p.full + 2u * (tiles - p.full) : tiles;
    const uint32_t grid = (blocks + 7u) / 8u * 8u;
    if (int4) {
        has_offset ? wq_gemm_kernel<BM, BN, true, true, kOnce><<<grid, kThreads, 0, st>>>(p)
                   : wq_gemm_kernel<BM, BN, true, false, kOnce><<<grid, kThreads, 0, st>>>(p);
    } else {
        has_offset ? wq_gemm_kernel<BM, BN, false, true, kOnce><<<grid, kThreads, 0, st>>>(p)
                   : wq_gemm_kernel<BM, BN, false, false, kOnce><<<grid, kThreads, 0, st>>>(p);
    }
}

}  // namespace

// The tile shape: the one with the smallest estimate of rounds of the chip times a round's time per K step, measured at
// k = 8192, n = 28672 with every compute unit busy (us): 256 x 256 1.62, 128 x 256 1.11, 128 x 128 1.2 for the two tiles
// that share a unit and 0.62 for one alone; since then the loads of all three are spread better and take 3 to 8 % less, which
// leaves the choice where it was.  256 x 256 tiles that would fill less than about two thirds of the last round
// are cut in half there (k = 4096, n = 11008, 2048 rows: 204 -> 187 us; where the power limit and not
// the rounds sets the time it makes no difference, k = 8192, n = 28672, 2048 rows).
struct WqShape {
    double c256, c128, csmall;  // us per K step of each tile shape
    uint32_t t256, t128, tsmall, rounds;
    bool halve;
};
static WqShape wq_shape(uint32_t m, uint32_t n)
{
    const uint32_t cus = device_compute_units();
    auto up = [](uint32_t a, uint32_t b) { return (a + b - 1u) / b; };
    WqShape s{};
    s.t256 = up(m, 256u) * up(n, 256u);
    s.tsmall = up(m, 128u) * up(n, 128u);
    s.t128 = up(m, 128u) * up(n, 256u);
    const uint32_t rest = s.t256 % cus;
    s.rounds = s.t256 / cus;
    const double tail = up(2u * rest, cus) * 1.11;
    s.halve = rest != 0 && tail < 1.62;
    s.c256 = s.rounds * 1.62 + (rest == 0 ? 0.0 : s.halve ? tail : 1.62);
    s.c128 = up(s.t128, cus) * 1.11;
    s.csmall = s.tsmall <= cus ? 0.62 : up(s.tsmall, 2u * cus) * 1.2;
    return s;
}

// 3.5 us and 0.91 of the estimate above (214 random calls of 33 rows and more that leave the chip partly idle, half of them within 5 %,
// nine tenths within 20 %).  One round of 128 x 256 tiles on at most three quarters of the compute units has their share of the way to
// memory as well, and takes 0.77 of it: int4 641 x 6272 x 6656 79 us (102 without that factor, and the whole-k tiles that were then
// taken needed 88), 403 x 8064 x 12032 102 (131), 493 x 4096 x 12160 55 (68); at 236 tiles of 256 the estimate holds.
double wq_gemm_estimate(uint32_t m, uint32_t n, uint32_t k)
{
    const WqShape s = wq_shape(m, n);
    double c = s.c256 < s.c128 ? s.c256 : s.c128;
    if (s.t128 <= device_compute_units() * 3u / 4u) {
        c *= 0.77;
    }
    return 3.5 + 0.91 * (s.csmall < c ? s.csmall : c) * (k / kBK);
}

int launch_wq_gemm(const WqParams& p, bool int4, bool has_offset, hipStream_t st)
{
    WqParams q = p;
    q.mk = WqMasks{0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
    const WqShape s = wq_shape(p.m, p.n);
    const double c256 = s.c256, c128 = s.c128, csmall = s.csmall;
    if (csmall <= c128 && csmall <= c256) {
        // From half a million on (tiles times k): a step is as long as its loads' way from memory, and they all go out at once
        // behind its barrier.  Less: each goes out behind a matrix instruction of its own.  In us, one behind every other
        // instruction and at once: w8a16 108 x 8064 x 18496 106.8 and 98.1, 1509 x 10752 x 1664 121.1 and 106.7, int4 49 x 6272 x
        // 20480 76.7 and 70.7; w8a16 54 x 5888 x 1440 52.1 and 55.7, int4 68 x 2176 x 2304 21.6 and 23.5.
        if (static_cast<uint64_t>(s.tsmall) * p.k >= 500000u) {
            wq_launch<128, 128, true>(q, int4, has_offset, st);
        } else {
            wq_launch<128, 128>(q, int4, has_offset, st);
        }
    } else if (c128 < c256) {
        wq_launch<128, 256>(q, int4, has_offset, st);
    } else {
        q.full = s.halve ? s.rounds * device_compute_units() : s.t256;
        wq_launch<256, 256>(q, int4, has_offset, st);
    }
    return launch_status("half x quantised weights (tile GEMM)");
}

}  // namespace ascq
