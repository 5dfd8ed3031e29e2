// Block-scaled (MX) matmul for few activation rows (decode), and for the shapes the 256 x 256 tile kernel of
// matmul_mx.hip does not take: c[m, n] = sum_k a 2^(sa - 127) * b 2^(sb - 127) (+ bias), operands as described there.
//
// What bounds it is the weights' trip from memory: at 16 rows, n = k = 8192 and e2m1 operands they are 33.5 of the
// 36 MB the call touches, and their 0.5 us of matrix work disappears behind it.  So a workgroup owns whole columns
// (16 S of them, nothing is added across workgroups: one launch, no workspace, the same bits from call to call), its
// wavefronts split k, and each streams 128-byte runs of its columns - whole cache lines - and the matching pieces of up
// to 16 RT activation rows through a two-slot LDS ring of its own: direct-to-LDS loads, one batch in flight while the
// other is computed, no barrier before the final sum.  The activations travel in the same queue: they are re-read by
// every workgroup from the L2, m / (16 S) of the weights' bytes, which is why more rows are cut into blocks of 64
// only up to a few hundred rows (mx_plan).  n = k = 8192, 16 rows, with one lane per output element before:
// e2m1 4830 -> 8.8 us a call (4.1 TB/s: a wavefront's share is four batches and two are on their way, so a third is asked
// for when the first has landed; 3 us less host time per call left it where it was), e4m3 3870 -> 16.3 us, fp8
// activations on e2m1 weights 4415 -> 14.8 us; 64 rows on the 256 x 256 tiles before: e2m1 42.4 -> 13.0 us, e4m3 77 ->
// 19.5 us.  32 columns per workgroup (S = 2) give every compute unit one at n = 8192; narrower matrices take 16 (a unit then
// streams half the bytes: n = 1024, k = 14336, e4m3, 9 against 14 us).
//
// v_mfma_scale_f32_16x16x128_f8f6f4 takes one scale byte per lane: lane l holds the scale of row l % 16 and block of 32 k
// number l / 16; a 4-bit operand's four registers hold the lane's own block, an 8-bit operand's registers 0-3 hold k =
// 16 (l / 16) .. + 15 and 4-7 k = 64 + 16 (l / 16) .. + 15; e1m2, which the instruction does not know, is widened to e4m3 in
// registers (exact).  The products of two 4-bit operands lie less than 2^8 apart, and the instruction drops none; those
// of fp8 operands it aligns to the largest and drops what lies 2^13 below it.  The tiles live with that, so fp8 at the
// tiles' shapes may run it here too.
// Elsewhere fp8 runs v_mfma_f32_16x16x32_bf16 on operands converted in registers (every fp8 and fp4 value is a bfloat16
// value, every product of two exact in fp32), one instruction per block of 32 k from zero, whose sums the vector ALU
// scales and adds: the arithmetic of the kernel with one lane per output element, which took these calls before.
// Against 64 bits (2-norm, k = 8192, 16 rows, normally distributed e4m3): scaled instruction 1.3e-5, one lane per output
// 2.2e-7, this 9.2e-8; e2m1 x e4m3 3.0e-7, 1.2e-7 and 6.8e-8.  That arithmetic is also what bounds these pairs from 16
// rows on: per block of 32 k and 16 x 16 results a multiplication and an addition per sum beside the conversions (e4m3,
// 16 rows: 16.3 us a call where the scaled instruction took 12.3).
#include <type_traits>
#include <utility>

#include "matmul_w8a8.h"
#include "matmul_mx.h"

namespace ascq {
namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) const void* gptr_t;
typedef int v8i __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// operand formats: the instruction's codes, and e1m2
enum { kE4M3 = 0, kE5M2 = 1, kE2M1 = 4, kE1M2 = 5 };
constexpr bool fmt_is_8bit(int f) { return f == kE4M3 || f == kE5M2; }
// the pairs whose products the scaled matrix instruction adds up without dropping any
constexpr bool fmt_lossless(int fa, int fb) { return !fmt_is_8bit(fa) && !fmt_is_8bit(fb); }
constexpr uint32_t kPastEnd = 0x7FFFFFF0u;  // an offset every buffer's range check rejects: the load moves no data

// A batch is 128 bytes of a weight column: KB values of k.
template <int FA, int FB, int RT, int S>
struct MxdShape {
    static constexpr uint32_t KB = fmt_is_8bit(FB) ? 128u : 256u;
    static constexpr uint32_t tiles = KB / 128u;                           // matrix instructions per block pair
    static constexpr uint32_t arb = fmt_is_8bit(FA) ? KB : KB / 2u, brb = 128u;  // bytes of a row of the batch
    static constexpr uint32_t a_bytes = RT * 16u * arb, b_bytes = S * 16u * brb;
    static constexpr uint32_t srows = (RT + S) * 16u, sdw = KB / 128u;     // scale rows and dwords per row
    static constexpr uint32_t a_instr = a_bytes / 1024u, b_instr = b_bytes / 1024u, s_instr = (srows * sdw + 63u) / 64u;
    static constexpr uint32_t sc_bytes = s_instr * 256u;
    static constexpr uint32_t slot = a_bytes + b_bytes + sc_bytes;
    static constexpr uint32_t waves = slot * 16u <= 150u * 1024u ? 8u : 4u;
    static constexpr uint32_t red_bytes = waves * RT * S * 1024u;
    static constexpr uint32_t lds = slot * 2u * waves > red_bytes ? slot * 2u * waves : red_bytes;
    static constexpr uint32_t loads = a_instr + b_instr + s_instr;
    static_assert(lds <= 158u * 1024u && loads * 2u < 63u, "the ring must fit the LDS and the load counter");
};

// 8 e1m2 values (a dword, the even one of a byte in the low nibble) -> 8 e4m3 codes in order.  A magnitude code c is the
// value c / 4; the eight e4m3 codes are a byte table in two registers that a byte permute looks up.
__device__ __forceinline__ i32x2_t widen_e1m2(uint32_t q)
{
    constexpr uint32_t lut_hi = 0x3E3C3A38u, lut_lo = 0x34302800u;
    const uint32_t ve = __builtin_amdgcn_perm(lut_hi, lut_lo, q & 0x07070707u) | ((q << 4) & 0x80808080u);
    const uint32_t vo = __builtin_amdgcn_perm(lut_hi, lut_lo, (q >> 4) & 0x07070707u) | (q & 0x80808080u);
    return i32x2_t{static_cast<int>(__builtin_amdgcn_perm(vo, ve, 0x05010400u)),
                   static_cast<int>(__builtin_amdgcn_perm(vo, ve, 0x07030602u))};
}

// 8 values of a format as bfloat16, every one exact (the scale operand of the conversions is 1)
template <int F>
__device__ __forceinline__ bf16x8_t to_bf16(const typename std::conditional<fmt_is_8bit(F), i32x2_t, uint32_t>::type raw)
{
    u32x4 out;
    auto put = [&](int i, bf16x2_t v) __attribute__((always_inline)) { out[i] = __builtin_bit_cast(uint32_t, v); };
    if constexpr (F == kE2M1) {
        put(0, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(raw, 1.0f, 0));
        put(1, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(raw, 1.0f, 1));
        put(2, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(raw, 1.0f, 2));
        put(3, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(raw, 1.0f, 3));
    } else {
        i32x2_t d;
        if constexpr (F == kE1M2) {
            d = widen_e1m2(raw);
        } else {
            d = raw;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t v = static_cast<uint32_t>(d[i]);
            if constexpr (F == kE5M2) {
                put(2 * i, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(v, 1.0f, false));
                put(2 * i + 1, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(v, 1.0f, true));
            } else {
                put(2 * i, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, false));
                put(2 * i + 1, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, true));
            }
        }
    }
    return __builtin_bit_cast(bf16x8_t, out);
}

// 2^(e - 127) of byte `blk` of a dword of scales, but for e = 0 (the subnormal 2^-127, 0 here) and e = 255 (NaN, infinity
// here): exact_scale puts those right where a batch has any.
__device__ __forceinline__ float plain_scale(uint32_t dword, int blk)
{
    return __uint_as_float((blk == 3 ? dword >> 1 : dword << (23 - 8 * blk)) & 0x7F800000u);
}
__device__ __forceinline__ float exact_scale(float plain)
{
    const uint32_t u = __float_as_uint(plain);
    return __uint_as_float(u == 0u ? 0x00400000u : u == 0x7F800000u ? 0x7FC00000u : u);
}

// LDS reads are instructions in an asm: one that the compiler knows of makes it wait for every load on its way into LDS.
template <uint32_t kOff>
__device__ __forceinline__ i32x4 lds_b128(uint32_t addr)
{
    i32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(kOff) : "memory");
    return v;
}
template <uint32_t kOff>
__device__ __forceinline__ i32x2_t lds_b64(uint32_t addr)
{
    i32x2_t v;
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(kOff) : "memory");
    return v;
}
template <uint32_t kOff>
__device__ __forceinline__ uint32_t lds_b32(uint32_t addr)
{
    uint32_t v;
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(kOff) : "memory");
    return v;
}
template <uint32_t kOff>
__device__ __forceinline__ uint32_t lds_u8(uint32_t addr)
{
    uint32_t v;
    asm volatile("ds_read_u8 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "i"(kOff) : "memory");
    return v;
}

template <int... I, class F>
__device__ __forceinline__ void mxd_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void mxd_for(F&& f)
{
    mxd_for_impl(f, std::make_integer_sequence<int, N>{});
}

struct MxdParams {
    MxParams p;
    uint32_t a_row_bytes, b_row_bytes;
    uint32_t blocks;       // blocks of 32 k (the last may be partial)
    uint32_t tiles_k;      // tiles of 128 k
    uint32_t tpw;          // tiles of k per wavefront, a multiple of the batch's
    uint32_t row_blocks, col_blocks;
};

// kScaled: on the scaled matrix instruction; otherwise in bfloat16
template <int FA, int FB, int RT, int S, bool kScaled>
__global__ __launch_bounds__((MxdShape<FA, FB, RT, S>::waves * 64)) void mx_decode_kernel(MxdParams q)
{
    typedef MxdShape<FA, FB, RT, S> T;
    __shared__ __attribute__((aligned(1024))) char LDS[T::lds];
    const MxParams& p = q.p;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lc = lane & 15u, lq = lane >> 4;
    // an XCD takes neighbouring column blocks, and the row blocks of a column block next to each other
    const uint32_t t = xcd_remap(blockIdx.x, q.row_blocks * q.col_blocks);
    if (t >= q.row_blocks * q.col_blocks) {
        return;
    }
    const uint32_t row0 = (t % q.row_blocks) * (RT * 16u), n0 = (t / q.row_blocks) * (S * 16u);
    const uint32_t ta = min(wave * q.tpw, q.tiles_k), tb = min(ta + q.tpw, q.tiles_k);
    const uint32_t batches = (tb - ta + T::tiles - 1u) / T::tiles;
    char* const ring = LDS + wave * (2u * T::slot);

    // ---- sources.  An operand's batch lies in LDS as rows of arb / brb bytes whose 16-byte pieces are XOR-ed with the
    // row number so that 16 lanes reading one piece of 16 rows meet all 64 banks; lane i of a load owns LDS bytes
    // 16 i .. + 15 and fetches the piece that belongs there.  Rows past the end and pieces past the end of k are given
    // an offset outside the buffer: zeros arrive, nothing is fetched.
    auto piece_of = [](uint32_t row_bytes, uint32_t slot_piece, uint32_t& row) __attribute__((always_inline)) {
        const uint32_t per = row_bytes / 16u;
        row = slot_piece / per;
        return (slot_piece % per) ^ ((row / (16u / per)) & (per - 1u));
    };
    uint32_t a_off[T::a_instr], a_pc[T::a_instr], b_off[T::b_instr], b_pc[T::b_instr];
#pragma unroll
    for (uint32_t u = 0; u < T::a_instr; ++u) {
        uint32_t r;
        a_pc[u] = piece_of(T::arb, u * 64u + lane, r) * 16u;
        a_off[u] = row0 + r < p.m ? (row0 + r) * q.a_row_bytes + a_pc[u] : kPastEnd;
    }
#pragma unroll
    for (uint32_t u = 0; u < T::b_instr; ++u) {
        uint32_t r;
        b_pc[u] = piece_of(T::brb, u * 64u + lane, r) * 16u;
        b_off[u] = n0 + r < p.n ? (n0 + r) * q.b_row_bytes + b_pc[u] : kPastEnd;
    }
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.a), 0,
                                                                       static_cast<int>(p.m * q.a_row_bytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.b), 0,
                                                                       static_cast<int>(p.n * q.b_row_bytes), 0x00020000);
    // scale bytes: one dword per lane, rows of a first, then columns of b (rows past the end read the last one's)
    const uint8_t* s_src[T::s_instr];
    uint32_t s_dw[T::s_instr];
#pragma unroll
    for (uint32_t u = 0; u < T::s_instr; ++u) {
        uint32_t i = u * 64u + lane;
        i = i < T::srows * T::sdw ? i : T::srows * T::sdw - 1u;
        const uint32_t r = i / T::sdw;
        s_dw[u] = i % T::sdw;
        if (r < RT * 16u) {
            s_src[u] = p.sa + static_cast<size_t>(min(row0 + r, p.m - 1u)) * p.sk;
        } else {
            s_src[u] = p.sb + static_cast<size_t>(min(n0 + r - RT * 16u, p.n - 1u)) * p.sk;
        }
    }
    const uint32_t last_dw = p.sk / 4u - 1u;
    auto load = [&](uint32_t b, char* slot) __attribute__((always_inline)) {
        const uint32_t tile = ta + b * T::tiles;
        const bool live = b < batches;  // past the end the loads are issued all the same (the waits count) and move nothing
        const uint32_t a_at = tile * (T::arb / T::tiles), b_at = tile * (T::brb / T::tiles);
#pragma unroll
        for (uint32_t u = 0; u < T::b_instr; ++u) {
            const uint32_t off = live && b_at + b_pc[u] < q.b_row_bytes ? b_off[u] : kPastEnd;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(slot + T::a_bytes + u * 1024u), 16, off, b_at, 0, 0);
        }
#pragma unroll
        for (uint32_t u = 0; u < T::a_instr; ++u) {
            const uint32_t off = live && a_at + a_pc[u] < q.a_row_bytes ? a_off[u] : kPastEnd;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(slot + u * 1024u), 16, off, a_at, 0, 0);
        }
#pragma unroll
        for (uint32_t u = 0; u < T::s_instr; ++u) {
            const uint32_t dw = min(tile + s_dw[u], last_dw);
            __builtin_amdgcn_global_load_lds((gptr_t)(s_src[u] + dw * 4u), (lds_ptr_t)(slot + T::a_bytes + T::b_bytes + u * 256u), 4, 0, 0);
        }
    };

    f32x4 acc[RT][S];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
#pragma unroll
        for (int j = 0; j < S; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const uint32_t ring_addr = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)ring));
    // LDS bytes of the lane's 16-byte piece `piece` of row lc of an operand (rows 16 apart share the swizzle)
    auto at = [&](uint32_t row_bytes, uint32_t piece) __attribute__((always_inline)) {
        const uint32_t per = row_bytes / 16u;
        return lc * row_bytes + ((piece ^ ((lc / (16u / per)) & (per - 1u))) << 4);
    };
    constexpr std::integral_constant<int, FA> fa{};
    constexpr std::integral_constant<int, FB> fb{};
    constexpr std::integral_constant<uint32_t, T::arb> arb{};
    constexpr std::integral_constant<uint32_t, T::brb> brb{};
    // loads return in order: everything but the newest batch has landed
    auto wait_batch = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt((T::loads & 15) | ((T::loads >> 4) << 14) | (7 << 4) | (15 << 8));
        asm volatile("" ::: "memory");
    };

    // The scaled instruction.  e2m1: a lane's 16 bytes of a tile are its operand as they lie; fp8: two times 16 bytes; e1m2,
    // which the instruction does not know: the two times 8 bytes that widened to e4m3 are the lane's operand of 8 bits.
    auto step_scaled = [&](uint32_t b, uint32_t slot_off) __attribute__((always_inline)) {
        const uint32_t abase = ring_addr + slot_off, bbase = abase + T::a_bytes, sbase = bbase + T::b_bytes;
        const uint32_t slane = sbase + lc * (4u * T::sdw) + lq;
        struct Raw {
            i32x4 v, w;        // e2m1 (v), fp8
            i32x2_t h0, h1;    // e1m2
        };
        auto read = [&](auto fmt, auto line, auto row_bytes, auto tt, uint32_t base) __attribute__((always_inline)) {
            constexpr uint32_t bytes = decltype(row_bytes)::value, off = decltype(line)::value * 16u * bytes, tl = decltype(tt)::value;
            Raw r;
            if constexpr (fmt_is_8bit(decltype(fmt)::value)) {
                r.v = lds_b128<off>(base + at(bytes, 8u * tl + lq));
                r.w = lds_b128<off>(base + at(bytes, 8u * tl + 4u + lq));
            } else if constexpr (decltype(fmt)::value == kE2M1) {
                r.v = lds_b128<off>(base + at(bytes, 4u * tl + lq));
            } else {
                r.h0 = lds_b64<off>(base + at(bytes, 4u * tl + (lq >> 1)) + 8u * (lq & 1u));
                r.h1 = lds_b64<off>(base + at(bytes, 4u * tl + 2u + (lq >> 1)) + 8u * (lq & 1u));
            }
            return r;
        };
        auto landed = [](auto fmt, Raw& r, uint32_t& scale) __attribute__((always_inline)) {  // usable from here on
            if constexpr (fmt_is_8bit(decltype(fmt)::value)) {
                asm volatile("" : "+v"(r.v), "+v"(r.w), "+v"(scale));
            } else if constexpr (decltype(fmt)::value == kE2M1) {
                asm volatile("" : "+v"(r.v), "+v"(scale));
            } else {
                asm volatile("" : "+v"(r.h0), "+v"(r.h1), "+v"(scale));
            }
        };
        auto operand = [](auto fmt, const Raw& r) __attribute__((always_inline)) {
            if constexpr (fmt_is_8bit(decltype(fmt)::value)) {
                return v8i{r.v[0], r.v[1], r.v[2], r.v[3], r.w[0], r.w[1], r.w[2], r.w[3]};
            } else if constexpr (decltype(fmt)::value == kE2M1) {
                return __builtin_shufflevector(r.v, r.v, 0, 1, 2, 3, -1, -1, -1, -1);
            } else {
                const i32x2_t a = widen_e1m2(static_cast<uint32_t>(r.h0[0])), b = widen_e1m2(static_cast<uint32_t>(r.h0[1]));
                const i32x2_t c = widen_e1m2(static_cast<uint32_t>(r.h1[0])), d = widen_e1m2(static_cast<uint32_t>(r.h1[1]));
                return v8i{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
            }
        };
        constexpr int kCodeA = FA == kE1M2 ? kE4M3 : FA, kCodeB = FB == kE1M2 ? kE4M3 : FB;
        Raw ar[T::tiles][RT], br[T::tiles][S];
        uint32_t asc[T::tiles][RT], bsc[T::tiles][S];
        mxd_for<static_cast<int>(T::tiles)>([&](auto tt) {
            constexpr uint32_t tl = decltype(tt)::value;
            mxd_for<S>([&](auto j) {
                br[tl][j] = read(fb, j, brb, tt, bbase);
                bsc[tl][j] = lds_u8<(RT + decltype(j)::value) * 64u * T::sdw + 4u * tl>(slane);
            });
            mxd_for<RT>([&](auto i) {
                ar[tl][i] = read(fa, i, arb, tt, abase);
                asc[tl][i] = lds_u8<decltype(i)::value * 64u * T::sdw + 4u * tl>(slane);
            });
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        mxd_for<static_cast<int>(T::tiles)>([&](auto tt) {
            mxd_for<S>([&](auto j) { landed(fb, br[tt][j], bsc[tt][j]); });
            mxd_for<RT>([&](auto i) { landed(fa, ar[tt][i], asc[tt][i]); });
        });
        load(b + 2u, ring + slot_off);  // the slot is free again
        mxd_for<static_cast<int>(T::tiles)>([&](auto tt) {
            constexpr uint32_t tl = decltype(tt)::value;
            const uint32_t tile = ta + b * T::tiles + tl;
            if (tile < tb) {  // uniform
                // blocks past the end of k hold zeros; their scale bytes may be anything, a NaN too
                const bool in_k = tile * 4u + lq < q.blocks;
                v8i bo[S];
                int bs[S];
#pragma unroll
                for (int j = 0; j < S; ++j) {
                    bo[j] = operand(fb, br[tl][j]);
                    bs[j] = in_k ? static_cast<int>(bsc[tl][j]) : 127;
                }
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const v8i ao = operand(fa, ar[tl][i]);
                    const int as = in_k ? static_cast<int>(asc[tl][i]) : 127;
#pragma unroll
                    for (int j = 0; j < S; ++j) {
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(ao, bo[j], acc[i][j], kCodeA, kCodeB, 0, as, 0, bs[j]);
                    }
                }
            }
        });
    };

    // In bfloat16: lane l holds k = 32 blk + 8 (l / 16) .. + 7 of row l % 16 for each of a tile's four blocks blk, and
    // the scale bytes of its four rows of the result (rows 4 (l / 16) .. + 3) and of its column.
    typedef typename std::conditional<fmt_is_8bit(FA), i32x2_t, uint32_t>::type RawA;
    typedef typename std::conditional<fmt_is_8bit(FB), i32x2_t, uint32_t>::type RawB;
    auto step_exact = [&](uint32_t b, uint32_t slot_off) __attribute__((always_inline)) {
        const uint32_t abase = ring_addr + slot_off, bbase = abase + T::a_bytes, sbase = bbase + T::b_bytes;
        RawA ar[T::tiles][4][RT];
        RawB br[T::tiles][4][S];
        i32x4 asc[RT][T::sdw];  // dword r of the four rows' T::sdw dwords each, in order
        typename std::conditional<T::sdw == 2, i32x2_t, uint32_t>::type bsc[S];
        uint32_t staged[T::s_instr];
        auto read = [](auto fmt, auto line, auto row_bytes, uint32_t addr) __attribute__((always_inline)) {
            constexpr uint32_t off = decltype(line)::value * 16u * decltype(row_bytes)::value;
            if constexpr (fmt_is_8bit(decltype(fmt)::value)) {
                return lds_b64<off>(addr);
            } else {
                return lds_b32<off>(addr);
            }
        };
        // bytes of the lane's 8 values of block blk of tile tl, from the operand's start
        auto place = [&](auto fmt, auto row_bytes, uint32_t tl, uint32_t blk) __attribute__((always_inline)) {
            if constexpr (fmt_is_8bit(decltype(fmt)::value)) {
                return at(row_bytes, 8u * tl + 2u * blk + (lq >> 1)) + 8u * (lq & 1u);
            } else {
                return at(row_bytes, 4u * tl + blk) + 4u * lq;
            }
        };
        mxd_for<S>([&](auto j) {
            constexpr uint32_t off = (RT + decltype(j)::value) * 64u * T::sdw;
            if constexpr (T::sdw == 2) {
                bsc[j] = lds_b64<off>(sbase + lc * 8u);
            } else {
                bsc[j] = lds_b32<off>(sbase + lc * 4u);
            }
        });
        mxd_for<RT>([&](auto i) {
            mxd_for<static_cast<int>(T::sdw)>([&](auto h) {
                asc[i][h] = lds_b128<decltype(i)::value * 64u * T::sdw + decltype(h)::value * 16u>(sbase + lq * (16u * T::sdw));
            });
        });
        mxd_for<static_cast<int>(T::s_instr)>([&](auto u) { staged[u] = lds_b32<decltype(u)::value * 256u>(sbase + lane * 4u); });
        mxd_for<static_cast<int>(T::tiles) * 4>([&](auto n) {
            constexpr uint32_t tl = decltype(n)::value / 4, blk = decltype(n)::value % 4;
            const uint32_t bat = bbase + place(fb, brb, tl, blk), aat = abase + place(fa, arb, tl, blk);
            mxd_for<S>([&](auto j) { br[tl][blk][j] = read(fb, j, brb, bat); });
            mxd_for<RT>([&](auto i) { ar[tl][blk][i] = read(fa, i, arb, aat); });
        });
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        auto landed = [](auto& r) __attribute__((always_inline)) { asm volatile("" : "+v"(r)); };  // usable from here on
        mxd_for<S>([&](auto j) { landed(bsc[j]); });
        mxd_for<RT>([&](auto i) {
            mxd_for<static_cast<int>(T::sdw)>([&](auto h) { landed(asc[i][h]); });
        });
        mxd_for<static_cast<int>(T::s_instr)>([&](auto u) { landed(staged[u]); });
        mxd_for<static_cast<int>(T::tiles) * 4>([&](auto n) {
            mxd_for<S>([&](auto j) { landed(br[n / 4][n % 4][j]); });
            mxd_for<RT>([&](auto i) { landed(ar[n / 4][n % 4][i]); });
        });
        load(b + 2u, ring + slot_off);  // the slot is free again
        // a byte 0 or 255 among the batch's scales?  (x - 0x01..01 borrows into the top bit of a zero byte)
        bool odd = false;
#pragma unroll
        for (uint32_t u = 0; u < T::s_instr; ++u) {
            const uint32_t x = staged[u], y = ~x;
            odd = odd || ((((x - 0x01010101u) & y) | ((y - 0x01010101u) & x)) & 0x80808080u) != 0u;
        }
        const bool special = __builtin_amdgcn_ballot_w64(odd) != 0;
        mxd_for<static_cast<int>(T::tiles) * 4>([&](auto n) {
            constexpr uint32_t tl = decltype(n)::value / 4, blk = decltype(n)::value % 4;
            const uint32_t block = (ta + b * T::tiles + tl) * 4u + blk;
            if (block < tb * 4u && block < q.blocks) {  // uniform; blocks past the end of k may have any scale bytes
                float sa[RT][4], sb[S];
#pragma unroll
                for (int j = 0; j < S; ++j) {
                    if constexpr (T::sdw == 2) {
                        sb[j] = plain_scale(static_cast<uint32_t>(bsc[j][tl]), blk);
                    } else {
                        sb[j] = plain_scale(bsc[j], blk);
                    }
                }
#pragma unroll
                for (int i = 0; i < RT; ++i) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const uint32_t d = r * T::sdw + tl;
                        sa[i][r] = plain_scale(static_cast<uint32_t>(asc[i][d / 4u][d % 4u]), blk);
                    }
                }
                if (special) {  // uniform
#pragma unroll
                    for (int j = 0; j < S; ++j) sb[j] = exact_scale(sb[j]);
#pragma unroll
                    for (int i = 0; i < RT; ++i) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) sa[i][r] = exact_scale(sa[i][r]);
                    }
                }
                bf16x8_t bo[S];
#pragma unroll
                for (int j = 0; j < S; ++j) bo[j] = to_bf16<FB>(br[tl][blk][j]);
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const bf16x8_t ao = to_bf16<FA>(ar[tl][blk][i]);
#pragma unroll
                    for (int j = 0; j < S; ++j) {
                        const f32x4 part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ao, bo[j], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[i][j][r] = __builtin_fmaf(part[r], sa[i][r] * sb[j], acc[i][j][r]);
                    }
                }
            }
        });
    };
    auto step = [&](uint32_t b, uint32_t slot_off) __attribute__((always_inline)) {
        if (b >= batches) {
            return;  // uniform
        }
        wait_batch();
        if constexpr (kScaled) {
            step_scaled(b, slot_off);
        } else {
            step_exact(b, slot_off);
        }
    };
    load(0, ring);
    load(1, ring + T::slot);
    for (uint32_t b = 0; b < batches; b += 2u) {
        step(b, 0u);
        step(b + 1u, T::slot);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the requests past the last batch
    __syncthreads();

    // ---- the wavefronts' sums, added in wavefront order: [wavefront][block][register][lane]
    float* const red = reinterpret_cast<float*>(LDS);
#pragma unroll
    for (int i = 0; i < RT; ++i) {
#pragma unroll
        for (int j = 0; j < S; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) red[((wave * RT + i) * S + j) * 256u + r * 64u + lane] = acc[i][j][r];
        }
    }
    __syncthreads();
    for (uint32_t v = wave; v < RT * S * 4u; v += T::waves) {
        const uint32_t blk = v >> 2, row = row0 + (blk / S) * 16u + 4u * lq + (v & 3u), col = n0 + (blk % S) * 16u + lc;
        if (row >= p.m || col >= p.n) {
            continue;
        }
        const float* part = red + v * 64u + lane;
        float sum = part[0];
#pragma unroll
        for (uint32_t w = 1; w < T::waves; ++w) sum += part[w * (RT * S * 256u)];
        if (p.bias != nullptr) {
            sum += p.bias[col];
        }
        mx_store(p, static_cast<size_t>(row) * p.n + col, sum);
    }
}

template <int FA, int FB, int RT, int S, bool kScaled>
void mxd_launch(MxdParams q, hipStream_t st)
{
    typedef MxdShape<FA, FB, RT, S> T;
    q.row_blocks = (q.p.m + RT * 16u - 1u) / (RT * 16u);
    q.col_blocks = (q.p.n + S * 16u - 1u) / (S * 16u);
    const uint32_t per = (q.tiles_k + T::waves - 1u) / T::waves;
    q.tpw = (per + T::tiles - 1u) / T::tiles * T::tiles;
    mx_decode_kernel<FA, FB, RT, S, kScaled><<<(q.row_blocks * q.col_blocks + 7u) / 8u * 8u, T::waves * 64u, 0, st>>>(q);
}

template <int FA, int FB>
void mxd_pick(const MxdParams& q, bool tile_shape, hipStream_t st)
{
    constexpr bool kLossless = fmt_lossless(FA, FB);
    constexpr int kMost = fmt_is_8bit(FA) && !fmt_is_8bit(FB) ? 2 : 4;  // (twice the bytes per row of a: 64 rows do not fit the ring)
    const uint32_t m = q.p.m;
    const bool few_columns = (q.p.n + 31u) / 32u < device_compute_units() / 2u;
    if (!kLossless && tile_shape) {
        mxd_launch<FA, FB, kMost, 2, true>(q, st);
    } else if (m <= 16u) {
        few_columns ? mxd_launch<FA, FB, 1, 1, kLossless>(q, st) : mxd_launch<FA, FB, 1, 2, kLossless>(q, st);
    } else if (m <= 32u || kMost == 2) {
        mxd_launch<FA, FB, 2, 2, kLossless>(q, st);
    } else {
        mxd_launch<FA, FB, kMost, 2, kLossless>(q, st);
    }
}

inline int code_of(int f)
{
    return f == ASCQ_QDST_FP8_E4M3FN ? kE4M3 : f == ASCQ_QDST_FP8_E5M2 ? kE5M2 : f == ASCQ_QDST_FP4_E2M1 ? kE2M1 : kE1M2;
}

}  // namespace

bool mx_decode_supported(const MxParams& p)
{
    const bool a8 = p.a_format == ASCQ_QDST_FP8_E4M3FN || p.a_format == ASCQ_QDST_FP8_E5M2;
    const bool b8 = p.b_format == ASCQ_QDST_FP8_E4M3FN || p.b_format == ASCQ_QDST_FP8_E5M2;
    const uint64_t arb = a8 ? p.k : p.k / 2u, brb = b8 ? p.k : p.k / 2u;
    // 16-byte pieces that never straddle two rows, dwords of scale bytes, 31-bit buffer offsets
    return arb % 16u == 0 && brb % 16u == 0 && aligned16(p.a) && aligned16(p.b) && p.sk % 4u == 0 &&
           (reinterpret_cast<uintptr_t>(p.sa) & 3u) == 0 && (reinterpret_cast<uintptr_t>(p.sb) & 3u) == 0 &&
           p.m * arb < kPastEnd && p.n * brb < kPastEnd &&
           static_cast<uint64_t>((p.m + 15u) / 16u) * ((p.n + 15u) / 16u) < (1ull << 31);
}

int launch_mx_decode(const MxParams& p, bool tile_shape, hipStream_t st)
{
    MxdParams q{};
    q.p = p;
    const int fa = code_of(p.a_format), fb = code_of(p.b_format);
    q.a_row_bytes = fmt_is_8bit(fa) ? p.k : p.k / 2u;
    q.b_row_bytes = fmt_is_8bit(fb) ? p.k : p.k / 2u;
    q.blocks = (p.k + 31u) / 32u;
    q.tiles_k = (p.k + 127u) / 128u;
#define ASCQ_MXD(A, B)                     \
    if (fa == (A) && fb == (B)) {          \
        mxd_pick<(A), (B)>(q, tile_shape, st); \
    }
    ASCQ_MXD(kE4M3, kE4M3)
    ASCQ_MXD(kE4M3, kE5M2)
    ASCQ_MXD(kE4M3, kE2M1)
    ASCQ_MXD(kE4M3, kE1M2)
    ASCQ_MXD(kE5M2, kE4M3)
    ASCQ_MXD(kE5M2, kE5M2)
    ASCQ_MXD(kE5M2, kE2M1)
    ASCQ_MXD(kE5M2, kE1M2)
    ASCQ_MXD(kE2M1, kE4M3)
    ASCQ_MXD(kE2M1, kE5M2)
    ASCQ_MXD(kE2M1, kE2M1)
    ASCQ_MXD(kE2M1, kE1M2)
    ASCQ_MXD(kE1M2, kE4M3)
    ASCQ_MXD(kE1M2, kE5M2)
    ASCQ_MXD(kE1M2, kE2M1)
    ASCQ_MXD(kE1M2, kE1M2)
#undef ASCQ_MXD
    return launch_status("ascq_matmul_mx (few rows)");
}

}  // namespace ascq
