// Block-scaled (MX) matmul of two e1m2 operands: 256 x 256 tiles on 6-bit e2m3 codes, which the matrix core runs at the
// 4-bit rate.
//
// mx_widen_e1m2_kernel rewrites codes and scale bytes into the order in which the tile kernel's lanes want them:
//   codes   [block of 32 rows][step of 128 k][3072 bytes]: two units of 16 rows; lane l of a unit owns row l % 16,
//           k = 32 (l / 16) .. + 31 as 32 little-endian 6-bit fields, 24 bytes: 16 bytes of every lane of unit 0, of unit 1, then
//           the other 8 of unit 0, of unit 1.  So a step's codes of a block are one contiguous run, every LDS read is linear
//           and free of bank conflicts, and 96 bytes of a row travel per 128 k.
//   scales  a: [128 rows][step][lane][8 units], b: [64 rows][step][lane][4 units]: a wavefront's bytes of a step are one LDS
//           read for a and one for b, and the unit is the byte selector of the instruction, a constant.
// An e1m2 value is +-(code / 4), code 0 .. 7, which is the e2m3 value with magnitude bits 2 * code (its subnormals run 0,
// 1/8 .. 7/8 and its first binade 1, 9/8 .. 15/8).
//
// The tile kernel: 8 wavefronts as 2 x 4, each 128 x 64 of the tile: 8 x 4 blocks of v_mfma_scale_f32_16x16x128_f8f6f4, which
// on random operands, where the power limit sets the clock, reaches 6.2 PFLOP/s against 5.6 of the 32x32x64 form.  Three LDS stages of a step
// each (48 KiB), filled by direct-to-LDS loads that are issued two steps ahead, one behind every fourth matrix instruction or so, so that the way
// from the L2 is never idle: with two stages and all loads waited for at every step the loads arrived at 11 TB/s over
// the chip, a loop of nothing but loads with a stage always on its way reaches 26.  m = n = k = 8192: tiles 330 -> 264 us, the call
// with the widening launch 365 -> 290 (operands of zeros, where the power limit is not met: 301 -> 215); 512 x 8192 x 8192 88 -> 69;
// 4096 x 4096 x 4096 66 -> 56.  What is left: 24 + 2 LDS reads for 32 matrix instructions of a wavefront, the power limit.
#include <type_traits>
#include <utility>

#include "matmul_mx.h"

namespace ascq {
namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) const void* gptr_t;
typedef int v6i __attribute__((ext_vector_type(6)));

constexpr uint32_t kUnit = 1536u, kBlock = 2u * kUnit;  // bytes of a step's codes of 16 and of 32 rows
constexpr uint32_t kOperand = 8u * kBlock;              // of the 256 rows of a tile
constexpr uint32_t kScaleA = 512u, kScaleB = 256u;      // bytes of a step's scales of 128 rows of a, of 64 of b

struct MxWidenParams {
    const uint8_t* src[2];
    const uint8_t* scale[2];
    uint8_t* dst[2];
    uint8_t* scale_dst[2];
    uint32_t rows[2];
    uint32_t a_scale_blocks, scale_blocks;  // workgroups of the scale bytes: of the first operand, of both
    uint32_t a_blocks, k_blocks, k, sk;     // workgroups of the first operand's codes; workgroups per block of 32 rows
};

constexpr uint32_t kScaleSteps = 8u, kScaleRow = 4u * kScaleSteps + 4u;  // K steps of a workgroup, bytes of its LDS rows

// The scale bytes of 128 rows and 8 steps: in as 32 bytes of a row, out as whole lines (as 16-bit stores beside the
// codes, one line gathered from four workgroups, m = n = k = 8192 took 31 us instead of 28).
__device__ __forceinline__ void mx_order_scales(const MxWidenParams& p, uint32_t which, uint32_t id, uint8_t* rows)
{
    const uint32_t steps = p.k / 128u, chunks = (steps + kScaleSteps - 1u) / kScaleSteps;
    const uint32_t row0 = id / chunks * 128u, step0 = id % chunks * kScaleSteps;
    const uint32_t here = steps - step0 < kScaleSteps ? steps - step0 : kScaleSteps, last_row = p.rows[which] - 1u;
    constexpr uint32_t kEach = 128u * kScaleSteps / 256u;
    const uint32_t sl = threadIdx.x % kScaleSteps, rl = threadIdx.x / kScaleSteps, sr = sl < here ? sl : here - 1u;
    uint32_t in[kEach];
#pragma unroll
    for (uint32_t e = 0; e < kEach; ++e) {
        const uint32_t r = row0 + rl + e * (256u / kScaleSteps), row = r < last_row ? r : last_row;
        in[e] = *reinterpret_cast<const uint32_t*>(p.scale[which] + static_cast<size_t>(row) * p.sk + (step0 + sr) * 4u);
    }
#pragma unroll
    for (uint32_t e = 0; e < kEach; ++e) {
        *reinterpret_cast<uint32_t*>(rows + (rl + e * (256u / kScaleSteps)) * kScaleRow + 4u * sl) = in[e];
    }
    __syncthreads();
    const uint32_t units = which ? 4u : 8u, words = units / 4u;  // units of 16 rows of a group; dwords of a lane
#pragma unroll
    for (uint32_t e = 0; e < kEach; ++e) {
        const uint32_t i = threadIdx.x + e * 256u, s = i / 128u, at = i % 128u;  // dword `at` of the step's 512 bytes of these rows
        const uint32_t group = which ? at / 64u : 0u, l = which ? at % 64u : at / 2u, first = which ? group * 4u : at % 2u * 4u;
        if (s >= here || (which && row0 + group * 64u > last_row)) {
            continue;  // past the last step; a group that does not exist
        }
        uint32_t v = 0;
#pragma unroll
        for (uint32_t b = 0; b < 4u; ++b) {
            v |= static_cast<uint32_t>(rows[((first + b) * 16u + (l & 15u)) * kScaleRow + 4u * s + (l >> 4)]) << (8u * b);
        }
        const size_t to = static_cast<size_t>(row0 / (16u * units) + group) * steps + step0 + s;
        reinterpret_cast<uint32_t*>(p.scale_dst[which])[(to * 64u + l) * words + (which ? 0u : at % 2u)] = v;
    }
}

// Both operands in one launch: a workgroup takes 32 rows x 256 k, whole 128-byte lines of the source.
__global__ __launch_bounds__(256) void mx_widen_e1m2_kernel(MxWidenParams p)
{
    __shared__ __attribute__((aligned(16))) uint8_t rows[128u * kScaleRow];
    if (blockIdx.x < p.scale_blocks) {
        const bool of_b = blockIdx.x >= p.a_scale_blocks;
        mx_order_scales(p, of_b ? 1u : 0u, blockIdx.x - (of_b ? p.a_scale_blocks : 0u), rows);
        return;
    }
    const uint32_t block_id = blockIdx.x - p.scale_blocks, which = block_id < p.a_blocks ? 0u : 1u;
    const uint32_t id = block_id - (which ? p.a_blocks : 0u);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, half = wave & 1u;
    const uint32_t block = id / p.k_blocks, step = id % p.k_blocks * 2u + (wave >> 1), steps = p.k / 128u;
    const uint32_t last_row = p.rows[which] - 1u;  // (rows past the end are never stored by the matmul: any one will do)
    if (step < steps) {
        uint32_t row = block * 32u + half * 16u + (lane & 15u);
        row = row < last_row ? row : last_row;
        const u32x4 q = *reinterpret_cast<const u32x4*>(p.src[which] + static_cast<size_t>(row) * (p.k / 2u) + step * 64u + (lane >> 4) * 16u);
        uint64_t c[4];  // 32 values, value v of a dword in bits 4 v .. 4 v + 3
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            uint64_t t = q[d];
            t = (t & 0xFFFFull) | ((t & 0xFFFF0000ull) << 8);                              // values 0-3 | 4-7, 24 bits each
            t = (t & 0x00000000FF0000FFull) | ((t & 0x000000FF0000FF00ull) << 4);          // pairs, 12 bits each
            t = (t & 0x00000F00F00F00Full) | ((t & 0x0000F00F00F00F0ull) << 2);            // value v in bits 6 v .. 6 v + 3
            c[d] = ((t & 0x0000208208208208ull) << 2) | ((t & 0x00001C71C71C71C7ull) << 1);  // sign to bit 5, magnitude doubled
        }
        uint8_t* const out = p.dst[which] + (static_cast<size_t>(block) * steps + step) * kBlock;
        *reinterpret_cast<u32x4*>(out + half * 1024u + lane * 16u) =
            u32x4{static_cast<uint32_t>(c[0]), static_cast<uint32_t>(c[0] >> 32) | (static_cast<uint32_t>(c[1]) << 16),
                  static_cast<uint32_t>(c[1] >> 16), static_cast<uint32_t>(c[2])};
        *reinterpret_cast<u32x2*>(out + 2048u + half * 512u + lane * 8u) =
            u32x2{static_cast<uint32_t>(c[2] >> 32) | (static_cast<uint32_t>(c[3]) << 16), static_cast<uint32_t>(c[3] >> 16)};
    }
}

// How a tile is stored: 16-bit or float rows of a multiple of 4 values, anything else.  A kernel each, and a loop for each 16-bit type: the
// epilogue runs once per tile, so the way of its instructions from memory is part of its time.  (One kernel, both 16-bit
// conversions in one loop: 2048 x 2048 x 512 to bfloat16 15.4 us, 14.2 like this, to half 18.7 and 16.3.)
constexpr int kStoreHalf = 0, kStoreFloat = 1, kStoreAny = 2;

struct MxSixParams {
    const uint8_t *a, *b, *sa, *sb;  // as written by mx_widen_e1m2_kernel
    MxParams out;                    // c, bias, m, n, k, tiles, output type
};

template <class F, int... I>
__device__ __forceinline__ void six_static_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void six_static_for(F&& f)
{
    six_static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// d += a x b, 16 x 16 x 128 of e2m3 codes, in place (an instruction that the compiler is free to give another destination
// moves sums about); unit i of a's scale bytes, unit j of b's
template <int i, int j>
__device__ __forceinline__ void six_mfma(f32x4& d, const v6i& a, const v6i& b, uint32_t sa, uint32_t sb)
{
    constexpr int al = i & 1, ah = (i >> 1) & 1, bl = j & 1, bh = j >> 1;
    asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel:[%5,%6,0] op_sel_hi:[%7,%8,0] cbsz:2 blgp:2"
                 : "+v"(d)
                 : "v"(a), "v"(b), "v"(sa), "v"(sb), "n"(al), "n"(bl), "n"(ah), "n"(bh));
}

template <int kStore>
__global__ __launch_bounds__(512, 1) void mx_six_kernel(MxSixParams q)
{
    const MxParams& p = q.out;
    // one array per stage (the compiler tells at most eight targets of such loads apart); scales of a (2 x 512), of b (4 x 256)
    __shared__ __attribute__((aligned(1024))) char L0[2 * kOperand], L1[2 * kOperand], L2[2 * kOperand];
    __shared__ __attribute__((aligned(1024))) char C0[2048], C1[2048], C2[2048];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave >> 2, wn = wave & 3u;
    const uint32_t total = p.tiles_m * p.tiles_n;
    const uint32_t t = xcd_remap(blockIdx.x, total);  // every XCD takes a contiguous share
    if (t >= total) {
        return;
    }
    uint32_t tm, tn;
    band_order(t, p.tiles_m, p.tiles_n, tm, tn);
    const uint32_t row0 = tm * 256u, n0 = tn * 256u;
    const uint32_t steps = p.k / 128u, last = steps - 1u;

    // ---- loads: wavefront w brings block w of a and of b (three instructions each, one contiguous run) and 256 of the 2048
    // scale bytes; blocks past the end are never stored, the last one will do
    auto clamp = [](uint32_t v, uint32_t rows, uint32_t per) __attribute__((always_inline)) {
        const uint32_t most = (rows + per - 1u) / per - 1u;
        return v < most ? v : most;
    };
    auto uniform = [](const uint8_t* ptr) __attribute__((always_inline)) {  // pinned to scalar registers
        const uint64_t v = reinterpret_cast<uint64_t>(ptr);
        uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
        uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
        asm volatile("" : "+s"(lo), "+s"(hi));
        return reinterpret_cast<const uint8_t*>((static_cast<uint64_t>(hi) << 32) | lo);
    };
    const uint8_t* const a_src = uniform(q.a + static_cast<size_t>(clamp(row0 / 32u + wave, p.m, 32u)) * steps * kBlock);
    const uint8_t* const b_src = uniform(q.b + static_cast<size_t>(clamp(n0 / 32u + wave, p.n, 32u)) * steps * kBlock);
    const bool of_a = wave < 4u;
    const uint8_t* const s_src =
        uniform(of_a ? q.sa + static_cast<size_t>(clamp(row0 / 128u + (wave >> 1), p.m, 128u)) * steps * kScaleA + (wave & 1u) * 256u
                     : q.sb + static_cast<size_t>(clamp(n0 / 64u + (wave - 4u), p.n, 64u)) * steps * kScaleB);
    const uint32_t s_step = of_a ? kScaleA : kScaleB;
    uint32_t lane16 = lane * 16u, lane8 = lane * 8u, lane4 = lane * 4u;
    constexpr int kLoads = 7;
    struct Stage {
        char *a, *b, *s;
    };
    struct Sources {
        const uint8_t *a, *b, *s;
    };
    auto sources = [&](uint32_t step) __attribute__((always_inline)) {
        const uint32_t at = step < last ? step : last;  // past the end: the last step again, into a stage that nobody uses
        return Sources{uniform(a_src + static_cast<size_t>(at) * kBlock), uniform(b_src + static_cast<size_t>(at) * kBlock),
                       uniform(s_src + static_cast<size_t>(at) * s_step)};
    };
    auto load = [&](const Sources& from, int u, const Stage& S) __attribute__((always_inline)) {
        asm volatile("" : "+v"(lane16), "+v"(lane4));
        const gptr_t a = (gptr_t)(from.a + lane16), b = (gptr_t)(from.b + lane16);
        const lds_ptr_t la = (lds_ptr_t)(S.a + wave * kBlock), lb = (lds_ptr_t)(S.b + wave * kBlock);
        // (the offset counts for both addresses)
        switch (u) {
        case 0: __builtin_amdgcn_global_load_lds(b, lb, 16, 0, 0); break;
        case 1: __builtin_amdgcn_global_load_lds(b, lb, 16, 1024, 0); break;
        case 2: __builtin_amdgcn_global_load_lds(b, lb, 16, 2048, 0); break;
        case 3: __builtin_amdgcn_global_load_lds(a, la, 16, 0, 0); break;
        case 4: __builtin_amdgcn_global_load_lds(a, la, 16, 1024, 0); break;
        case 5: __builtin_amdgcn_global_load_lds(a, la, 16, 2048, 0); break;
        default: __builtin_amdgcn_global_load_lds((gptr_t)(from.s + lane4), (lds_ptr_t)(S.s + wave * 256u), 4, 0, 0); break;
        }
    };

    f32x4 acc[8][4];
    six_static_for<32>([&](auto c) {
        f32x4& v = acc[decltype(c)::value / 4][decltype(c)::value % 4];
        v = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        asm volatile("" : "+v"(v));
    });
    // ---- operands of a step: units 0-3 and 4-7 of the wavefront's rows, units 0-3 of its columns (two sets: those of the
    // next step arrive while this one's are in use), the scale bytes
    v6i af[8], bf[2][4];
    u32x2 sa[2];
    uint32_t sb[2];
    auto unit = [&](const char* S, uint32_t w, int u, auto piece, v6i& v) __attribute__((always_inline)) {
        const char* block = S + w * kBlock + (u >> 1) * kBlock;
        if constexpr (decltype(piece)::value == 0) {
            const i32x4 lo = *reinterpret_cast<const i32x4*>(block + (u & 1) * 1024 + lane16);
            v[0] = lo[0];
            v[1] = lo[1];
            v[2] = lo[2];
            v[3] = lo[3];
        } else {
            const i32x2_t hi = *reinterpret_cast<const i32x2_t*>(block + 2048 + (u & 1) * 512 + lane8);
            v[4] = hi[0];
            v[5] = hi[1];
        }
    };
    // read r of the operands that a step needs first: scale bytes, b, units 0 and 1 of a; then units 2-7 of a
    auto first_read = [&](const Stage& S, auto set, auto r) __attribute__((always_inline)) {
        constexpr int n = decltype(r)::value, x = decltype(set)::value;
        if constexpr (n == 0) {
            sa[x] = *reinterpret_cast<const u32x2*>(S.s + wm * kScaleA + lane8);
        } else if constexpr (n == 1) {
            sb[x] = *reinterpret_cast<const uint32_t*>(S.s + 2u * kScaleA + wn * kScaleB + lane4);
        } else if constexpr (n < 10) {
            unit(S.b, wn * 2u, (n - 2) / 2, std::integral_constant<int, n % 2>{}, bf[x][(n - 2) / 2]);
        } else {
            unit(S.a, wm * 4u, (n - 10) / 2, std::integral_constant<int, n % 2>{}, af[(n - 10) / 2]);
        }
    };
    auto second_read = [&](const Stage& S, auto r) __attribute__((always_inline)) {
        constexpr int n = decltype(r)::value + 4;
        unit(S.a, wm * 4u, n / 2, std::integral_constant<int, n % 2>{}, af[n / 2]);
    };
    constexpr int kFirst = 14, kSecond = 12;

    // ---- one step, in stage X with operand set `set`; the next one is in Y, the one behind it on its way into Z.
    // The first half of its matrix instructions takes units 0-3 of a and reads the rest of the step's operands behind them; then the wait
    // (the next step's stage has landed, only the seven loads of the step behind it are on their way; every
    // wavefront has read this stage) and the barrier; the second half reads the next step's first operands.  The loads of the step
    // three ahead go into this stage: four of them in this step's second half, the others in the next one's first, each
    // behind a fourth matrix instruction (all in the second half, behind every other one: m = n = k = 8192 300 us, so 292).
    constexpr int kNow = 4, kEvery = 4;
    auto half = [&](auto hh, auto set, auto&& behind) __attribute__((always_inline)) {
        constexpr int h = decltype(hh)::value, x = decltype(set)::value;
        six_static_for<16>([&](auto nn) {
            constexpr int n = decltype(nn)::value, i = 4 * h + n / 4, j = n % 4;
            six_mfma<i & 3, j>(acc[i][j], af[i], bf[x][j], sa[x][h], sb[x]);
            behind(nn);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto arrive = [&](auto left) __attribute__((always_inline)) {
        constexpr int kLeft = decltype(left)::value;
        __builtin_amdgcn_s_waitcnt(0x0070 | (kLeft & 15) | ((kLeft >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();  // (not __syncthreads(): its fence waits for every load)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](uint32_t s, const Stage& X, const Stage& Y, const Stage& Z, auto set) __attribute__((always_inline)) {
        auto due = [](int n, int count) { return n % kEvery == kEvery - 1 && n / kEvery < count; };
        const Sources behind = sources(s + 2u);
        asm volatile("" : "+v"(lane16), "+v"(lane8), "+v"(lane4));
        half(std::integral_constant<int, 0>{}, set, [&](auto n) __attribute__((always_inline)) {
            if constexpr (decltype(n)::value < kSecond) second_read(X, n);
            if (due(decltype(n)::value, kLoads - kNow)) load(behind, kNow + decltype(n)::value / kEvery, Z);
        });
        arrive(std::integral_constant<int, kLoads>{});
        const Sources ahead = sources(s + 3u);
        half(std::integral_constant<int, 1>{}, set, [&](auto n) __attribute__((always_inline)) {
            if constexpr (decltype(n)::value < kFirst) first_read(Y, std::integral_constant<int, 1 - decltype(set)::value>{}, n);
            if (due(decltype(n)::value, kNow)) load(ahead, decltype(n)::value / kEvery, X);
        });
    };
    const Stage T0{L0, L0 + kOperand, C0}, T1{L1, L1 + kOperand, C1}, T2{L2, L2 + kOperand, C2};
    {
        const Sources f0 = sources(0), f1 = sources(1), f2 = sources(2);
        // (stage by stage: the waits count the loads behind the ones they are for)
#pragma unroll
        for (int u = 0; u < kLoads; ++u) load(f0, u, T0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kLoads; ++u) load(f1, u, T1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kNow; ++u) load(f2, u, T2);
    }
    arrive(std::integral_constant<int, kLoads + kNow>{});
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    six_static_for<kFirst>([&](auto r) { first_read(T0, even, r); });
    // Three stages and two operand sets: steps in groups of six, then what is left.  (A step that has no next one reads a
    // stage that holds the last step again, or still an older one; nobody uses what it read.)
    uint32_t s = 0;
    for (; s + 6u <= steps; s += 6u) {
        step(s, T0, T1, T2, even);
        step(s + 1u, T1, T2, T0, odd);
        step(s + 2u, T2, T0, T1, even);
        step(s + 3u, T0, T1, T2, odd);
        step(s + 4u, T1, T2, T0, even);
        step(s + 5u, T2, T0, T1, odd);
    }
    if (s < steps) {
        step(s, T0, T1, T2, even);
        if (s + 1u < steps) {
            step(s + 1u, T1, T2, T0, odd);
            if (s + 2u < steps) {
                step(s + 2u, T2, T0, T1, even);
                if (s + 3u < steps) {
                    step(s + 3u, T0, T1, T2, odd);
                    if (s + 4u < steps) {
                        step(s + 4u, T1, T2, T0, even);
                    }
                }
            }
        }
    }
    // The last sums are on their way through the matrix pipe, which the compiler does not know: it sees them changed behind the
    // wait.  (check_matrix_asm.py looks for what this cannot rule out.)  The repeated loads land before the LDS is given back.
    asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
    six_static_for<32>([&](auto c) {
        f32x4& v = acc[decltype(c)::value / 4][decltype(c)::value % 4];
        asm volatile("" : "+v"(v));
    });

    // ---- register r of lane l in a 16 x 16 block: row 4 (l / 16) + r, column l % 16
    const uint32_t lc = lane & 15u, lq = lane >> 4, colw = n0 + wn * 64u;
    float bias[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t col = colw + j * 16u + lc;
        bias[j] = (p.bias != nullptr && col < p.n) ? p.bias[col] : 0.0f;
    }
    // Rows of an even number of values: transpositions inside neighbouring lanes.  After one exchange a lane has two adjacent columns
    // of blocks l % 2 (`lo`) and 2 + l % 2 (`hi`) each, after a second one, n a multiple of 4, lane b of four has columns 4 (l / 4)
    // .. + 3 of block b, and the 16 lanes of a row store whole lines of its 64 columns.  (A wavefront's 128 stores of single elements take
    // 13 us: 2048 x 2050 x 512 to bfloat16 32.3 -> 16.4 us, 636 x 3728 x 1024 to float 31.8 -> 17.0.)
    const bool b0 = (lane & 1u) != 0, b1 = (lane & 2u) != 0, bf16 = p.out_dtype == ASCQ_BF16;
    const uint32_t col4 = colw + 16u * (lane & 3u) + (lc & 12u), col2 = colw + 16u * (lane & 1u) + (lc & 14u);
    auto exchange = [](uint32_t give, auto by) __attribute__((always_inline)) {  // with lane ^ by
        return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(give), decltype(by)::value == 1 ? 0xB1 : 0x4E, 0xF, 0xF, true));
    };
    constexpr std::integral_constant<int, 1> by1{};
    constexpr std::integral_constant<int, 2> by2{};
    auto each_row = [&](auto&& store) __attribute__((always_inline)) {  // store(row, the row's sum in block j, j = 0 .. 3)
        six_static_for<32>([&](auto c) {
            constexpr int i = decltype(c)::value / 4, r = decltype(c)::value % 4;
            store(row0 + (wm * 8u + i) * 16u + 4u * lq + r, [&](int j) __attribute__((always_inline)) { return acc[i][j][r] + bias[j]; });
        });
    };
    auto half_pairs = [&](auto to_bf16, auto&& value, uint32_t& lo, uint32_t& hi) __attribute__((always_inline)) {
        uint32_t h[4];
        six_static_for<4>([&](auto jj) {
            constexpr int j = decltype(jj)::value;
            const float v = value(j);
            h[j] = decltype(to_bf16)::value ? f32_to_bf16_bits(v) : f32_to_half_bits_sat(v);
        });
        const uint32_t got = exchange(b0 ? h[0] | (h[2] << 16) : h[1] | (h[3] << 16), by1);
        lo = b0 ? (got & 0xFFFFu) | (h[1] << 16) : h[0] | (got << 16);
        hi = b0 ? (got >> 16) | (h[3] << 16) : h[2] | (got & 0xFFFF0000u);
    };
    auto float_pairs = [&](auto&& value, u32x2& lo, u32x2& hi) __attribute__((always_inline)) {
        uint32_t w[4];
        six_static_for<4>([&](auto jj) { w[decltype(jj)::value] = __builtin_bit_cast(uint32_t, value(decltype(jj)::value)); });
        const uint32_t got0 = exchange(b0 ? w[0] : w[1], by1), got1 = exchange(b0 ? w[2] : w[3], by1);
        lo = b0 ? u32x2{got0, w[1]} : u32x2{w[0], got0};
        hi = b0 ? u32x2{got1, w[3]} : u32x2{w[2], got1};
    };
    uint16_t* const half_out = static_cast<uint16_t*>(p.c);
    float* const float_out = static_cast<float*>(p.c);
    if constexpr (kStore == kStoreHalf) {
        auto store_all = [&](auto to_bf16) __attribute__((always_inline)) {
            each_row([&](uint32_t row, auto&& value) __attribute__((always_inline)) {
                uint32_t lo, hi;
                half_pairs(to_bf16, value, lo, hi);
                const uint32_t got = exchange(b1 ? lo : hi, by2);
                if (row < p.m && col4 < p.n) {
                    __builtin_nontemporal_store(b1 ? u32x2{got, hi} : u32x2{lo, got},
                                                reinterpret_cast<u32x2*>(half_out + static_cast<size_t>(row) * p.n + col4));
                }
            });
        };
        if (bf16) {
            store_all(std::true_type{});
        } else {
            store_all(std::false_type{});
        }
        return;
    }
    if constexpr (kStore == kStoreFloat) {
        each_row([&](uint32_t row, auto&& value) __attribute__((always_inline)) {
            u32x2 lo, hi;
            float_pairs(value, lo, hi);
            const uint32_t got0 = exchange(b1 ? lo[0] : hi[0], by2), got1 = exchange(b1 ? lo[1] : hi[1], by2);
            if (row < p.m && col4 < p.n) {
                __builtin_nontemporal_store(b1 ? u32x4{got0, got1, hi[0], hi[1]} : u32x4{lo[0], lo[1], got0, got1},
                                            reinterpret_cast<u32x4*>(float_out + static_cast<size_t>(row) * p.n + col4));
            }
        });
        return;
    }
    if (p.n % 2u == 0) {
        auto store = [&](uint32_t row, auto* out, auto lo, auto hi) __attribute__((always_inline)) {
            auto* const at = out + static_cast<size_t>(row) * p.n + col2;
            if (row < p.m && col2 < p.n) __builtin_nontemporal_store(lo, reinterpret_cast<decltype(lo)*>(at));
            if (row < p.m && col2 + 32u < p.n) __builtin_nontemporal_store(hi, reinterpret_cast<decltype(hi)*>(at + 32));
        };
        if (p.out_dtype == ASCQ_F32) {
            each_row([&](uint32_t row, auto&& value) __attribute__((always_inline)) {
                u32x2 lo, hi;
                float_pairs(value, lo, hi);
                store(row, float_out, lo, hi);
            });
        } else {
            each_row([&](uint32_t row, auto&& value) __attribute__((always_inline)) {
                uint32_t lo, hi;
                if (bf16) {
                    half_pairs(std::true_type{}, value, lo, hi);
                } else {
                    half_pairs(std::false_type{}, value, lo, hi);
                }
                store(row, half_out, lo, hi);
            });
        }
        return;
    }
    six_static_for<128>([&](auto c) {
        constexpr int i = decltype(c)::value / 16, j = decltype(c)::value / 4 % 4, r = decltype(c)::value % 4;
        const uint32_t row = row0 + (wm * 8u + i) * 16u + 4u * lq + r, col = colw + j * 16u + lc;
        if (row < p.m && col < p.n) {
            mx_store(p, static_cast<size_t>(row) * p.n + col, acc[i][j][r] + bias[j]);
        }
    });
}

struct SixLayout {
    size_t codes[2], scales[2];
};

// rows of both operands rounded up to the blocks and groups of the widened form
inline SixLayout six_layout(uint64_t m, uint64_t n, uint64_t k)
{
    return SixLayout{{(m + 31u) / 32u * (k / 128u) * kBlock, (n + 31u) / 32u * (k / 128u) * kBlock},
                     {(m + 127u) / 128u * (k / 128u) * kScaleA, (n + 63u) / 64u * (k / 128u) * kScaleB}};
}

}  // namespace

size_t mx_six_bytes(uint32_t m, uint32_t n, uint32_t k)
{
    const SixLayout l = six_layout(m, n, k);
    return l.codes[0] + l.codes[1] + l.scales[0] + l.scales[1];
}

int launch_mx_six(const MxParams& p, void* workspace, hipStream_t st)
{
    const SixLayout l = six_layout(p.m, p.n, p.k);
    uint8_t* const ws = static_cast<uint8_t*>(workspace);
    MxWidenParams w{{p.a, p.b}, {p.sa, p.sb}, {ws, ws + l.codes[0]}, {}, {p.m, p.n}, 0, 0, 0, (p.k + 255u) / 256u, p.k, p.sk};
    w.scale_dst[0] = w.dst[1] + l.codes[1];
    w.scale_dst[1] = w.scale_dst[0] + l.scales[0];
    w.a_blocks = (p.m + 31u) / 32u * w.k_blocks;
    const uint32_t chunks = (p.k / 128u + kScaleSteps - 1u) / kScaleSteps;
    w.a_scale_blocks = (p.m + 127u) / 128u * chunks;
    w.scale_blocks = w.a_scale_blocks + (p.n + 127u) / 128u * chunks;
    mx_widen_e1m2_kernel<<<w.scale_blocks + w.a_blocks + (p.n + 31u) / 32u * w.k_blocks, 256, 0, st>>>(w);
    MxSixParams q{w.dst[0], w.dst[1], w.scale_dst[0], w.scale_dst[1], p};
    q.out.tiles_m = (p.m + 255u) / 256u;
    q.out.tiles_n = (p.n + 255u) / 256u;
    const uint32_t grid = (q.out.tiles_m * q.out.tiles_n + 7u) / 8u * 8u;
    if (p.n % 4u != 0) {
        mx_six_kernel<kStoreAny><<<grid, 512, 0, st>>>(q);
    } else if (p.out_dtype == ASCQ_F32) {
        mx_six_kernel<kStoreFloat><<<grid, 512, 0, st>>>(q);
    } else {
        mx_six_kernel<kStoreHalf><<<grid, 512, 0, st>>>(q);
    }
    return launch_status("ascq_matmul_mx (e1m2)");
}

}  // namespace ascq
