// Block-scaled (MX) matmul of medium size: small tiles with a ring of LDS stages (operands and scales as described in matmul_mx.hip).
//
// 256 x 256 tiles leave most of the chip idle where there are few of them, and their loop waits for all of its loads at every
// K step, 1.1 to 1.4 us whatever the loads' size.  Here a workgroup of 8 wavefronts owns 64 x 64 to 128 x 128 results, and its LDS holds
// 3 to 8 K steps: a load has kStages - 1 steps to arrive, a step waits only for the next one's, and its operands are read
// from the LDS behind the matrix instructions (v_mfma_scale_f32_16x16x128_f8f6f4) of the step before.  A K step is 128 values of a pair of 8-bit
// operands and 256 of pairs with a 4-bit one; an e2m1 operand beside an 8-bit one stays as it is (the tiles widen it in a launch of its own).
// Scale bytes come 16 per row and load, those of four or two steps, ahead of the first of these steps' tiles.
//
// The direct-to-LDS loads are inline assembly without results: the compiler, which knows such loads by the array they fill, would
// wait for all of them wherever it cannot tell the stages apart.  Every wait for them is written out (arrive).
//
// In us, 256 x 256 tiles or the few-row kernel and this: e4m3 441 x 4032 x 1792 24.7 and 9.1, 1370 x 2800 x 8448 89 and 39; e2m1 999 x 1856 x 3328 26.0 and
// 9.7, 470 x 5888 x 11520 63 and 32; e4m3 x e2m1 507 x 6896 x 7936 104 and 31.  The sums are the tiles' bit for bit, but for an e2m1 operand taken as it is
// beside an 8-bit one, whose products the instruction adds in another order than those of its widened form (2-norm error the same to three
// digits on normally distributed values, 4.60e-5 and 4.58e-5 where the e4m3 codes are uniform).  What is left: a step of 64 x 64
// takes 0.23 us (the barrier, the LDS reads of eight wavefronts), one of 128 x 128 0.36 on a nearly idle chip and 0.51 on a full one (0.67 of 256 k), and a
// second round of the chip starts 2 to 4 us after the first has ended: there is room for one workgroup on a compute unit.
#include <type_traits>
#include <utility>

#include "matmul_mx.h"

namespace ascq {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));

constexpr int kThreads = 512;
constexpr uint32_t kLine = 128;               // bytes of an LDS line: of a row's K step, or of half of it

template <class F, int... I>
__device__ __forceinline__ void ring_for_impl(F&& f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void ring_for(F&& f)
{
    ring_for_impl(f, std::make_integer_sequence<int, N>{});
}

constexpr bool is_8bit(int code) { return code < 2; }  // the instruction's codes: 0 e4m3, 1 e5m2, 4 e2m1

// the chunk of scale bytes that a load replaces was last read a step before
constexpr uint32_t mx_ring_chunks(uint32_t stages, uint32_t spc)
{
    return stages + spc - 1u <= 2u * spc ? 2u : stages + spc - 1u <= 4u * spc ? 4u : 8u;
}
// as many stages as fit, up to 8
constexpr uint32_t mx_ring_stages(uint32_t stage, uint32_t chunk, uint32_t spc)
{
    uint32_t n = 8u;
    while (n * stage + mx_ring_chunks(n, spc) * chunk > 158u * 1024u) --n;
    return n;
}

// BM x BN results, formats of a and b
template <int BM, int BN, int kCa, int kCb>
struct RingShape {
    static constexpr uint32_t kb = is_8bit(kCa) && is_8bit(kCb) ? 128u : 256u;  // values of k per step
    static constexpr uint32_t subs = kb / 128u;                                   // matrix instructions per block pair
    static constexpr uint32_t pa = is_8bit(kCa) ? subs : 1u, pb = is_8bit(kCb) ? subs : 1u;  // lines per row and step
    static constexpr uint32_t stage = (BM * pa + BN * pb) * kLine;
    static constexpr uint32_t spc = 4u / subs;                                    // steps of a chunk of 16 scale bytes
    static constexpr uint32_t chunk = (BM + BN) * 16u;
    static constexpr uint32_t stages = mx_ring_stages(stage, chunk, spc), chunks = mx_ring_chunks(stages, spc);
    static constexpr uint32_t lds = stages * stage + chunks * chunk;
    static_assert(stages >= 3u && lds <= 160u * 1024u && chunks * spc >= stages + spc - 1u, "ring");
};

template <int BM, int BN, int kCa, int kCb>
__global__ __launch_bounds__(kThreads, 1) void mx_ring_kernel(MxParams p)
{
    using S = RingShape<BM, BN, kCa, kCb>;
    constexpr int kStages = S::stages, kSubs = S::subs;
    constexpr int TJ = BN / 32, NA = BM / 64;                  // blocks of 16 x 16 per wavefront: 4 wavefronts along m, 2 along n
    constexpr int kALoads = BM * S::pa / 64, kBLoads = BN * S::pb / 64, kLoads = kALoads + kBLoads;
    __shared__ __attribute__((aligned(1024))) char L[S::lds];

    const uint32_t t = xcd_remap(blockIdx.x, p.tiles_m * p.tiles_n);
    if (t >= p.tiles_m * p.tiles_n) {
        return;  // whole workgroup (the launch is rounded up to a multiple of 8)
    }
    uint32_t tm, tn;
    band_order(t, p.tiles_m, p.tiles_n, tm, tn);
    const uint32_t row0 = tm * BM, n0 = tn * BN;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, lc = lane & 15u, lq = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave >> 1, wn = wave & 1u;
    const uint32_t steps = p.k / S::kb, last = steps - 1u;
    const uint32_t arb = is_8bit(kCa) ? p.k : p.k / 2u, brb = is_8bit(kCb) ? p.k : p.k / 2u;  // bytes of a row
    const uint32_t rows_a = p.m - row0 < BM ? p.m - row0 : BM, rows_b = p.n - n0 < BN ? p.n - n0 : BN;

    // ---- loads.  Instruction i of a tile fills lines 8 i .. + 7, lane l piece l % 8 of line l / 8; piece q of line r lies at q ^ (r / 2 % 8), which
    // the source address takes into account.  Lines run plane by plane (8-bit operand, step of 256: two planes of 128 k).  Rows
    // past the end are never stored: the last one will do.
    auto buffer = [](const uint8_t* base, uint64_t bytes) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), 0, static_cast<int>(bytes), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t ra = buffer(p.a + static_cast<uint64_t>(row0) * arb, static_cast<uint64_t>(rows_a) * arb);
    const __amdgpu_buffer_rsrc_t rb = buffer(p.b + static_cast<uint64_t>(n0) * brb, static_cast<uint64_t>(rows_b) * brb);
    auto source = [&](uint32_t instr, uint32_t rows, uint32_t valid, uint32_t row_bytes) __attribute__((always_inline)) {
        const uint32_t line = instr * 8u + (lane >> 3), plane = line / rows, r = line % rows, row = r < valid ? r : valid - 1u;
        return row * row_bytes + plane * kLine + (((lane & 7u) ^ ((r >> 1) & 7u)) << 4);
    };
    uint32_t aoff[kALoads], boff[kBLoads];
#pragma unroll
    for (int u = 0; u < kALoads; ++u) aoff[u] = source(wave * kALoads + u, BM, rows_a, arb);
#pragma unroll
    for (int u = 0; u < kBLoads; ++u) boff[u] = source(wave * kBLoads + u, BN, rows_b, brb);
    // scale bytes: wavefront w brings those of rows 64 w .. + 63 of the tile's BM + BN
    const bool has_scales = wave < (BM + BN) / 64u, sc_is_a = wave < BM / 64u;
    const uint32_t sc_first = (sc_is_a ? wave : wave - BM / 64u) * 64u, sc_valid = sc_is_a ? rows_a : rows_b;
    const __amdgpu_buffer_rsrc_t rs = buffer(sc_is_a ? p.sa + static_cast<uint64_t>(row0) * p.sk : p.sb + static_cast<uint64_t>(n0) * p.sk,
                                             static_cast<uint64_t>(sc_valid) * p.sk);
    const uint32_t sc_off = (sc_first + lane < sc_valid ? sc_first + lane : sc_valid - 1u) * p.sk;
    const uint32_t chunk_last = last / S::spc;
    auto chunk_at = [&](uint32_t c) __attribute__((always_inline)) {  // its first byte in a row: moved back to stay inside the row
        const uint32_t at = (c < chunk_last ? c : chunk_last) * 16u, cap = p.sk - 16u;
        return at < cap ? at : cap;
    };
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)L));
    auto dma = [](uint32_t to, uint32_t off, const __amdgpu_buffer_rsrc_t& r, uint32_t at) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" : : "s"(to), "v"(off), "s"(r), "s"(at) : "memory");
    };
    auto load_tile = [&](uint32_t step, uint32_t stage_at, int u) __attribute__((always_inline)) {
        const uint32_t at = step < last ? step : last;          // past the end: the last step again, into a stage that nobody uses
        if (u < kALoads) {
            dma(lds0 + stage_at + (wave * kALoads + u) * 1024u, aoff[u < kALoads ? u : 0], ra, at * (S::pa * kLine));
        } else {
            dma(lds0 + stage_at + BM * S::pa * kLine + (wave * kBLoads + u - kALoads) * 1024u, boff[u < kALoads ? 0 : u - kALoads], rb, at * (S::pb * kLine));
        }
    };
    auto load_scales = [&](uint32_t step) __attribute__((always_inline)) {
        if (has_scales && step % S::spc == 0) {                 // (uniform; a wavefront that waits for one load more waits a little early)
            const uint32_t c = step / S::spc;
            dma(lds0 + S::stages * S::stage + c % S::chunks * S::chunk + wave * 1024u, sc_off, rs, chunk_at(c));
        }
    };

    f32x4 acc[NA][TJ];
    ring_for<NA * TJ>([&](auto c) { acc[decltype(c)::value / TJ][decltype(c)::value % TJ] = f32x4{0.0f, 0.0f, 0.0f, 0.0f}; });

    // ---- operands of a step, two sets: those of the next step arrive while this one's are in use.  8-bit: registers 0-3 and 4-7 of a lane
    // are pieces l / 16 and 4 + l / 16 of its row's 128 k; 4-bit: piece 4 s + l / 16 is the lane's block of sub-step s
    v8i af[2][kSubs][NA], bf[2][kSubs][TJ];
    uint32_t sca[2][kSubs][NA], scb[2][kSubs][TJ];
    uint32_t foff[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) foff[h] = lc * kLine + (((4u * h + lq) ^ (lc >> 1)) << 4);
    const uint32_t sca_off = (wm * NA * 16u + lc) * 16u, scb_off = (BM + wn * TJ * 16u + lc) * 16u;
    auto operand = [&](auto code, const char* T, uint32_t rows, uint32_t line0, int s) __attribute__((always_inline)) {
        v8i v = {};
        if constexpr (is_8bit(decltype(code)::value)) {
            const char* at = T + (s * rows + line0) * kLine;
            const i32x4 lo = *reinterpret_cast<const i32x4*>(at + foff[0]), hi = *reinterpret_cast<const i32x4*>(at + foff[1]);
            v = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        } else {
            const i32x4 lo = *reinterpret_cast<const i32x4*>(T + line0 * kLine + foff[s & 1]);
            v = __builtin_shufflevector(lo, lo, 0, 1, 2, 3, -1, -1, -1, -1);  // the instruction reads 4 registers of a 4-bit operand
        }
        return v;
    };
    constexpr int kReads = kSubs * (NA + TJ) + NA + TJ;        // the scale bytes of a row and its operands, row block by row block
    auto read = [&](uint32_t step, uint32_t stage_at, auto set, int r) __attribute__((always_inline)) {
        constexpr int x = decltype(set)::value;
        const char* const T = L + stage_at;
        if (r < NA + TJ) {
            const uint32_t s1 = step < last ? step : last, c = step / S::spc;
            const char* const C = L + S::stages * S::stage + c % S::chunks * S::chunk + (s1 * (4u * kSubs) - chunk_at(c));
            const char* const at = C + (r < NA ? sca_off + r * 256u : scb_off + (r - NA) * 256u);
            uint32_t v[2];
            if constexpr (kSubs == 2) {
                const u32x2 w = *reinterpret_cast<const u32x2*>(at);
                v[0] = w[0];
                v[1] = w[1];
            } else {
                v[0] = *reinterpret_cast<const uint32_t*>(at);
            }
#pragma unroll
            for (int s = 0; s < kSubs; ++s) (r < NA ? sca[x][s][r < NA ? r : 0] : scb[x][s][r < NA ? 0 : r - NA]) = v[s];
            return;
        }
        r -= NA + TJ;
        const int s = r / (NA + TJ);
        r %= NA + TJ;
        if (r < NA) {
            af[x][s][r] = operand(std::integral_constant<int, kCa>{}, T, BM, (wm * NA + r) * 16u, s);
        } else {
            bf[x][s][r - NA] = operand(std::integral_constant<int, kCb>{}, T + BM * S::pa * kLine, BN, (wn * TJ + r - NA) * 16u, s);
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
    // A step whose operands are in registers or on their way there.  Behind the wait (they are there, the next step has landed,
    // those behind it are on their way) and the barrier every wavefront has read its stage, which takes the step kStages ahead.
    constexpr int kM = kSubs * NA * TJ, kPer = (kReads + kM - 1) / kM, kLoadPer = (kLoads + kM - 1) / kM;
    auto step = [&](uint32_t s, uint32_t here, uint32_t next, auto set) __attribute__((always_inline)) {
        constexpr int x = decltype(set)::value;
#pragma unroll
        for (int h = 0; h < 2; ++h) asm volatile("" : "+v"(foff[h]));
        arrive(std::integral_constant<int, (kStages - 2) * kLoads>{});
        load_scales(s + kStages);
        __builtin_amdgcn_sched_barrier(0);
        ring_for<kM>([&](auto nn) {
            constexpr int n = decltype(nn)::value, u = n / (NA * TJ), i = n / TJ % NA, j = n % TJ;
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(af[x][u][i], bf[x][u][j], acc[i][j], kCa, kCb, 0,
                                                                         static_cast<int>(sca[x][u][i] >> (8u * lq)), 0,
                                                                         static_cast<int>(scb[x][u][j] >> (8u * lq)));
            ring_for<kPer>([&](auto r) {
                constexpr int m = n * kPer + decltype(r)::value;
                if constexpr (m < kReads) read(s + 1u, next, std::integral_constant<int, 1 - x>{}, m);
            });
            ring_for<kLoadPer>([&](auto r) {
                constexpr int m = n * kLoadPer + decltype(r)::value;
                if constexpr (m < kLoads) load_tile(s + kStages, here, m);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    for (uint32_t st = 0; st < S::stages; ++st) {  // (scale bytes ahead of the tiles: the waits count the tiles' loads)
        load_scales(st);
#pragma unroll
        for (int u = 0; u < kLoads; ++u) load_tile(st, st * S::stage, u);
    }
    arrive(std::integral_constant<int, (kStages - 1) * kLoads>{});
#pragma unroll
    for (int r = 0; r < kReads; ++r) read(0, 0, std::integral_constant<int, 0>{}, r);
    constexpr uint32_t kEnd = S::stages * S::stage;
    uint32_t here = 0;
    auto after = [](uint32_t at) __attribute__((always_inline)) { return at + S::stage == kEnd ? 0u : at + S::stage; };
    uint32_t s = 0;
    for (; s + 2u <= steps; s += 2u) {  // (a step without a next one reads a stage that nobody uses)
        const uint32_t next = after(here), then = after(next);
        step(s, here, next, std::integral_constant<int, 0>{});
        step(s + 1u, next, then, std::integral_constant<int, 1>{});
        here = then;
    }
    if (s < steps) {
        step(s, here, after(here), std::integral_constant<int, 0>{});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the end land before the LDS is given back

    // ---- register r of lane l in a 16 x 16 block: row 4 (l / 16) + r, column l % 16.  Stores through a buffer that ends with the tile's last
    // row, columns past the end lie past it too
    constexpr uint32_t kNoColumn = 0x7FFFFFF0u;
    const bool f32 = p.out_dtype == ASCQ_F32, bf16 = p.out_dtype == ASCQ_BF16;
    const uint32_t row_size = p.n * (f32 ? 4u : 2u), colw = n0 + wn * (TJ * 16u);
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(static_cast<char*>(p.c) + static_cast<size_t>(row0) * row_size, 0,
                                                                        static_cast<int>(rows_a * row_size), 0x00020000);
    uint32_t row_lo = wm * (NA * 16u) * row_size;
    asm volatile("" : "+s"(row_lo));
    auto row_at = [&](int i, int r) __attribute__((always_inline)) { return row_lo + (i * 16u + r) * row_size; };
    float bias[TJ];
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        const uint32_t col = colw + j * 16u + lc;
        bias[j] = (p.bias != nullptr && col < p.n) ? p.bias[col] : 0.0f;
    }
    if (!f32 && p.n % 2u == 0 && (reinterpret_cast<uintptr_t>(p.c) & 3u) == 0) {
        // after one swap the even lane holds two adjacent columns of the first of two blocks, the odd lane two of the second
        const bool odd = (lane & 1u) != 0;
        auto store_all = [&](auto to_bf16) __attribute__((always_inline)) {
            ring_for<NA * TJ / 2 * 4>([&](auto cc) {
                constexpr int r = decltype(cc)::value % 4, j = decltype(cc)::value / 4 % (TJ / 2) * 2, i = decltype(cc)::value / 4 / (TJ / 2);
                const uint32_t col = odd ? colw + (j + 1) * 16u + lc - 1u : colw + j * 16u + lc;
                uint32_t h[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const float v = acc[i][j + t][r] + bias[j + t];
                    h[t] = decltype(to_bf16)::value ? f32_to_bf16_bits(v) : f32_to_half_bits_sat(v);
                }
                const uint32_t got = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(odd ? h[0] : h[1]), 0xB1, 0xF, 0xF, true));  // lane ^ 1
                __builtin_amdgcn_raw_buffer_store_b32(odd ? got | (h[1] << 16) : h[0] | (got << 16), rc,
                                                      col < p.n ? 4u * lq * row_size + col * 2u : kNoColumn, row_at(i, r), 0);
            });
        };
        if (bf16) {
            store_all(std::true_type{});
        } else {
            store_all(std::false_type{});
        }
        return;
    }
    ring_for<NA * TJ * 4>([&](auto cc) {
        constexpr int r = decltype(cc)::value % 4, j = decltype(cc)::value / 4 % TJ, i = decltype(cc)::value / 4 / TJ;
        const uint32_t col = colw + j * 16u + lc;
        const float v = acc[i][j][r] + bias[j];
        if (f32) {
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rc, col < p.n ? 4u * lq * row_size + col * 4u : kNoColumn, row_at(i, r), 0);
        } else {
            const uint16_t bits = static_cast<uint16_t>(bf16 ? f32_to_bf16_bits(v) : f32_to_half_bits_sat(v));
            __builtin_amdgcn_raw_buffer_store_b16(bits, rc, col < p.n ? 4u * lq * row_size + col * 2u : kNoColumn, row_at(i, r), 0);
        }
    });
}

template <int kCa, int kCb>
void ring_launch(MxParams p, int shape, hipStream_t st)
{
    const uint32_t bm = shape == 0 ? 64u : 128u, bn = shape == 2 ? 128u : 64u;
    p.tiles_m = (p.m + bm - 1u) / bm;
    p.tiles_n = (p.n + bn - 1u) / bn;
    const uint32_t grid = (p.tiles_m * p.tiles_n + 7u) / 8u * 8u;
    switch (shape) {
        case 0: mx_ring_kernel<64, 64, kCa, kCb><<<grid, kThreads, 0, st>>>(p); break;
        case 1: mx_ring_kernel<128, 64, kCa, kCb><<<grid, kThreads, 0, st>>>(p); break;
        default: mx_ring_kernel<128, 128, kCa, kCb><<<grid, kThreads, 0, st>>>(p); break;
    }
}

}  // namespace

int launch_mx_ring(const MxParams& p, int shape, int code_a, int code_b, hipStream_t st)
{
    switch (code_a * 8 + code_b) {
        case 0: ring_launch<0, 0>(p, shape, st); break;
        case 1: ring_launch<0, 1>(p, shape, st); break;
        case 4: ring_launch<0, 4>(p, shape, st); break;
        case 8: ring_launch<1, 0>(p, shape, st); break;
        case 9: ring_launch<1, 1>(p, shape, st); break;
        case 12: ring_launch<1, 4>(p, shape, st); break;
        default: ring_launch<4, 4>(p, shape, st); break;
    }
    return launch_status("ascq_matmul_mx (ring)");
}

}  // namespace ascq
