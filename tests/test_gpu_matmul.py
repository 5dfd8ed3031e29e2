"""GPU parity of the int8 matmul quant path, the quantized grouped matmul and W4A16 against the CPU oracle, through
the C ABI.  int32 accumulators and every epilogue without a transcendental are compared bit for bit (each epilogue
step rounds once in fp32, in the reference's order); FasterGelu outputs within 1 ulp of the output type; W4A16
(free summation order) within the stated tolerance."""
import ctypes as C

import numpy as np
import pytest
import torch

import orc
from ascq import _abi as abi
from ascq import ops
import gpu_util
from gpu_util import DEV, announce, bits, max_ulp, pack_int4, to_dev

pytestmark = pytest.mark.gpu


def rand_i8(rng, shape, lo=-127, hi=127):
    return rng.integers(lo, hi + 1, shape).astype(np.int8)


def run_mm(m, n, k, a, b, *, out, bias=None, quant=None, tok=None, trans_a=False, trans_b=False, act=abi.MM_ACT_NONE,
           scalar=None):
    mm = ops.Matmul(m, n, k, trans_a, trans_b)
    mm.set_tensor_a(to_dev(a))
    mm.set_tensor_b(to_dev(b))
    if bias is not None:
        mm.set_bias(to_dev(bias[0], bias[1]))
    if quant is not None:
        mm.set_quant_vector(to_dev(quant))
    if scalar is not None:
        mm.set_quant_scalar(scalar)
    if tok is not None:
        mm.set_token_scale(to_dev(tok))
    mm.set_activation(act)
    c = torch.zeros((m, n), dtype=out, device=DEV)
    mm.iterate_all(c)
    torch.cuda.synchronize()
    return c, mm.desc


def oracle_mm(desc, a, b, bias=None, quant=None, tok=None):
    orc.set_threads(16)
    return orc.matmul_w8a8(desc, a, b, None if bias is None else bias[0], quant, tok)


# shapes chosen to hit: the 32-row split-K tile, the 128-row tile with a row tail, the 256-row tile with row and
# column tails, K tails (K not a multiple of 128), and the generic kernel (odd sizes)
SHAPES = [(1, 256, 512), (16, 1024, 4096), (32, 264, 1040), (33, 256, 256), (128, 512, 384), (300, 520, 272),
          (1100, 776, 400), (2048, 512, 128), (19, 23, 77), (40, 100, 48),
          # the weight-stream kernel (m <= 32, k % 64 == 0): one chunk, column tails, runs that cross column blocks
          (1, 16, 64), (7, 144, 192), (32, 400, 64), (32, 1040, 2048), (5, 2064, 8192),
          # 128 x 128 tiles with and without a K split, row / column tails
          (33, 144, 128), (200, 528, 384), (512, 272, 256), (130, 2064, 1024),
          # 256-row tiles: a partial last round (narrow tiles), K steps odd and even
          (513, 528, 256), (2048, 2832, 384),
          # four and five K steps: the steady-state loop runs once, then two steps / one step are peeled
          (600, 528, 512), (600, 528, 640), (300, 272, 512), (300, 272, 640),
          # 344 tiles of 256 x 256: wide and narrow tiles in one launch, for B as [k, n] and as [n, k]
          (2048, 11008, 128),
          # more than 8 row tiles: bands of 8 row tiles and a last band of 2 (with a partial last row tile)
          (2500, 784, 128)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("trans_b", [False, True])
def test_int32_accumulators_bit_exact(m, n, k, trans_b):
    announce("matmul int32", m, n, k, trans_b)
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a = rand_i8(rng, (m, k), -128, 127)
    b = rand_i8(rng, (k, n), -128, 127)
    bias = rng.integers(-10000, 10000, n).astype(np.int32)
    b_in = np.ascontiguousarray(b.T) if trans_b else b
    c, desc = run_mm(m, n, k, a, b_in, out=torch.int32, bias=(bias, None), trans_b=trans_b)
    want = a.astype(np.int64) @ b.astype(np.int64) + bias
    assert np.array_equal(c.cpu().numpy().astype(np.int64), want)
    assert np.array_equal(oracle_mm(desc, a, b_in, (bias, None)).astype(np.int64), want)


def test_trans_a_generic_path():
    announce("matmul trans_a")
    rng = np.random.default_rng(3)
    m, n, k = 48, 64, 96
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    c, _ = run_mm(m, n, k, np.ascontiguousarray(a.T), b, out=torch.int32, trans_a=True)
    assert np.array_equal(c.cpu().numpy().astype(np.int64), a.astype(np.int64) @ b.astype(np.int64))


def test_config1_small_w8a8_bf16_with_bias():
    """A int8 [256,1024], B int8 [1024,1024], per-channel fp32 deqScale in [1e-4,1e-3], fp32 bias N(0,1) -> bf16."""
    announce("config 1")
    rng = np.random.default_rng(0xC1)
    m, n, k = 256, 1024, 1024
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    sc = rng.uniform(1e-4, 1e-3, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c, desc = run_mm(m, n, k, a, b, out=torch.bfloat16, bias=(bias, None), quant=sc)
    assert np.array_equal(bits(c), oracle_mm(desc, a, b, (bias, None), sc))


@pytest.mark.parametrize("m", [1, 16, 128, 2048])
def test_config3_w8a8_linear(m):
    """bf16 activations quantised per token on the GPU, int8 weights [4096,11008], fused dequant to bf16."""
    announce("config 3", m)
    rng = np.random.default_rng(0xC3 + m)
    k, n = 4096, 11008
    x = orc.f32_to_bf16_bits(rng.standard_normal((m, k)).astype(np.float32))
    w = rand_i8(rng, (k, n))
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    q, ts = ops.dynamic_quant_per_token(to_dev(x, "bf16"))
    wq, wts = orc.dynamic_quant_per_token(abi.BF16, x)
    assert np.array_equal(q.cpu().numpy(), wq) and np.array_equal(ts.cpu().numpy(), wts)
    c, desc = run_mm(m, n, k, wq, w, out=torch.bfloat16, quant=cs, tok=wts)
    want = oracle_mm(desc, wq, w, None, cs, wts)
    got = bits(c)
    assert max_ulp(got, want) <= 1
    assert np.array_equal(got, want)


@pytest.mark.parametrize("m", [1, 16, 17, 32])
def test_config3_w8a8_linear_weights_as_n_k(m):
    """Config 3's decode sizes on weights kept as [n, k] (isTransposeB): the whole-column kernel, one launch, no
    workspace; bf16 output with channel and token scales, bit-exact against the oracle on the same weights."""
    announce("config 3 [n, k]", m)
    rng = np.random.default_rng(0xC3 + 100 + m)
    k, n = 4096, 11008
    a = rand_i8(rng, (m, k))
    wt = rand_i8(rng, (n, k))
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    ts = rng.uniform(1e-2, 1e-1, m).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c, desc = run_mm(m, n, k, a, wt, out=torch.bfloat16, bias=(bias, None), quant=cs, tok=ts, trans_b=True)
    orc.set_threads(16)
    assert np.array_equal(bits(c), oracle_mm(desc, a, wt, (bias, None), cs, ts))
    wsz = C.c_size_t(1)
    assert abi.load_library().ascq_matmul_w8a8_workspace_size(C.byref(desc), C.byref(wsz)) == abi.OK and wsz.value == 0
    # int8 requantised output and SwiGLU through the same kernel
    words = (cs * 50).astype(np.float32).view(np.uint32).astype(np.uint64) | (np.uint64(1) << np.uint64(46))
    c8, d8 = run_mm(m, n, k, a, wt, out=torch.int8, quant=words, trans_b=True)
    assert np.array_equal(bits(c8), oracle_mm(d8, a, wt, None, words))


def run_mm_packed(m, n, k, a, b, *, out, bias=None, quant=None, tok=None, trans_b=False, act=abi.MM_ACT_NONE,
                  scalar=None):
    """run_mm on weights packed by ops.pack_weight_w8 (from [k, n], or from [n, k] with trans_b); the descriptor it
    returns describes the same matmul on the unpacked [k, n] weights, for the oracle."""
    mm = ops.Matmul(m, n, k)
    mm.set_tensor_a(to_dev(a))
    mm.set_tensor_b_packed(ops.pack_weight_w8(to_dev(b), k, n, trans_b))
    if bias is not None:
        mm.set_bias(to_dev(bias[0], bias[1]))
    if quant is not None:
        mm.set_quant_vector(to_dev(quant))
    if scalar is not None:
        mm.set_quant_scalar(scalar)
    if tok is not None:
        mm.set_token_scale(to_dev(tok))
    mm.set_activation(act)
    c = torch.zeros((m, n), dtype=out, device=DEV)
    mm.iterate_all(c)
    torch.cuda.synchronize()
    return c, mm.desc


def w8_packed_reference(w, k, n):
    """The packed int8 layout restated in numpy: slabs of 16 columns, tiles of 64 k, lane l of a tile owns column
    l % 16 and the 16 bytes k 16 (l / 16) .. + 15; zeros past n and k, 16 tiles of zeros behind the last slab."""
    slabs, ktiles = (n + 15) // 16, (k + 63) // 64
    full = np.zeros((ktiles * 64, slabs * 16), dtype=np.int8)
    full[:k, :n] = w
    t = full.reshape(ktiles, 4, 16, slabs, 16)            # tile, k quarter, byte, slab, column
    body = np.ascontiguousarray(t.transpose(3, 0, 1, 4, 2)).reshape(-1)   # slab, tile, k quarter, column, byte
    return np.concatenate([body, np.zeros(16 * 1024, dtype=np.int8)]).view(np.uint8)


@pytest.mark.parametrize("k,n", [(64, 16), (128, 40), (200, 1040), (1024, 272)])
def test_pack_weight_w8_layout(k, n):
    announce("pack w8", k, n)
    rng = np.random.default_rng(k + n)
    w = rand_i8(rng, (k, n))
    want = w8_packed_reference(w, k, n)
    assert np.array_equal(ops.pack_weight_w8(to_dev(w), k, n).cpu().numpy(), want)
    assert np.array_equal(ops.pack_weight_w8(to_dev(np.ascontiguousarray(w.T)), k, n, trans_b=True).cpu().numpy(), want)


@pytest.mark.parametrize("m", [1, 2, 3, 5, 8, 16, 17, 20, 31, 32, 33, 50])
@pytest.mark.parametrize("n,k", [(16, 64), (48, 128), (1040, 512), (272, 4096), (96, 8192), (32, 16384), (2064, 192)])
def test_w8a8_packed_small(m, n, k):
    """The one-launch kernel on packed weights computes what ascq_matmul_w8a8 computes: int32 accumulators and the
    dequantising epilogues bit for bit against the oracle on the unpacked weights.  k of one tile (seven wavefronts
    without work), column tails, more rows than a pass, k long enough for several batches per slab; more rows than a
    pass holds with the weights held in registers (k up to 16384)."""
    announce("w8a8 packed", m, n, k)
    rng = np.random.default_rng(m * 31 + n + k)
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    c, desc = run_mm_packed(m, n, k, a, b, out=torch.int32)
    assert np.array_equal(c.cpu().numpy(), a.astype(np.int64) @ b.astype(np.int64))
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    ts = rng.uniform(1e-2, 1e-1, m).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c, desc = run_mm_packed(m, n, k, a, np.ascontiguousarray(b.T), out=torch.bfloat16, bias=(bias, None), quant=cs, tok=ts,
                            trans_b=True)
    assert np.array_equal(bits(c), oracle_mm(desc, a, b, (bias, None), cs, ts))
    # requantised int8 output from uint64 words, int32 bias ahead of the dequantisation, FasterGelu to half
    words = (cs * 50).astype(np.float32).view(np.uint32).astype(np.uint64) | (np.uint64(1) << np.uint64(46))
    bias_i = rng.integers(-1000, 1000, n).astype(np.int32)
    c8, d8 = run_mm_packed(m, n, k, a, b, out=torch.int8, bias=(bias_i, None), quant=words)
    assert np.array_equal(bits(c8), oracle_mm(d8, a, b, (bias_i, None), words))
    cg, dg = run_mm_packed(m, n, k, a, b, out=torch.float16, scalar=1e-3, act=abi.MM_ACT_FASTER_GELU)
    assert max_ulp(bits(cg), oracle_mm(dg, a, b).view(np.uint16), "f16") <= 1


@pytest.mark.parametrize("m", [1, 2, 3, 5, 8, 13, 16])
@pytest.mark.parametrize("n,k", [(16, 64), (48, 128), (1040, 512), (272, 4096), (2064, 192), (100, 5632), (96, 8192),
                                 (40, 11008), (4100, 256)])
def test_w8a8_decode_on_n_k_weights_through_lds(m, n, k):
    """Up to 16 rows on weights kept as [n, k]: where the staged activations leave 64 KiB of LDS free the weights go
    through a ring there (four columns' 256 bytes per load, XOR-swizzled pieces), otherwise straight into registers
    (long k with many rows).  k of one tile (seven wavefronts without work), column counts that are no multiple of 16
    (the last slab's columns past n read as zeros), several slabs per workgroup, batches that end inside a wavefront's
    range.  int32 accumulators exactly, the dequantising and the requantising epilogue against the oracle."""
    announce("w8a8 [n, k] decode", m, n, k)
    rng = np.random.default_rng(m * 47 + n + k)
    a, b = rand_i8(rng, (m, k), -128, 127), rand_i8(rng, (k, n), -128, 127)
    bt = np.ascontiguousarray(b.T)
    c, _ = run_mm(m, n, k, a, bt, out=torch.int32, trans_b=True)
    assert np.array_equal(c.cpu().numpy(), a.astype(np.int64) @ b.astype(np.int64))
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    ts = rng.uniform(1e-2, 1e-1, m).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c, desc = run_mm(m, n, k, a, bt, out=torch.bfloat16, bias=(bias, None), quant=cs, tok=ts, trans_b=True)
    assert np.array_equal(bits(c), oracle_mm(desc, a, bt, (bias, None), cs, ts))  # (the descriptor says [n, k])
    words = (cs * 50).astype(np.float32).view(np.uint32).astype(np.uint64) | (np.uint64(1) << np.uint64(46))
    bias_i = rng.integers(-1000, 1000, n).astype(np.int32)
    c8, d8 = run_mm(m, n, k, a, bt, out=torch.int8, bias=(bias_i, None), quant=words, trans_b=True)
    assert np.array_equal(bits(c8), oracle_mm(d8, a, bt, (bias_i, None), words))


@pytest.mark.parametrize("m", [17, 33, 47, 64, 100, 128, 129, 224, 225, 300])
@pytest.mark.parametrize("n,k", [(16, 64), (48, 128), (1040, 512), (272, 4096), (2064, 192), (13000, 256), (96, 4160)])
def test_w8a8_weights_held_in_registers(m, n, k):
    """More than 16 rows on packed weights (17 to 224 on [n, k] weights): the weights of a workgroup's columns stay in
    registers and the activations stream past them, the sums and the epilogue in blocks of 128 rows (on [n, k]
    weights, more rows take the other kernels).  int32 accumulators against int64
    arithmetic, the dequantising epilogue bit for bit against the oracle, both forms."""
    announce("w8a8 weights in registers", m, n, k)
    rng = np.random.default_rng(m * 37 + n + k)
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    bt = np.ascontiguousarray(b.T)
    want = a.astype(np.int64) @ b.astype(np.int64)
    c, _ = run_mm_packed(m, n, k, a, b, out=torch.int32)
    assert np.array_equal(c.cpu().numpy(), want)
    c, _ = run_mm(m, n, k, a, bt, out=torch.int32, trans_b=True)
    assert np.array_equal(c.cpu().numpy(), want)
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    ts = rng.uniform(1e-2, 1e-1, m).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c, desc = run_mm_packed(m, n, k, a, b, out=torch.bfloat16, bias=(bias, None), quant=cs, tok=ts)
    gold = oracle_mm(desc, a, b, (bias, None), cs, ts)
    assert np.array_equal(bits(c), gold)
    c, desc = run_mm(m, n, k, a, bt, out=torch.bfloat16, bias=(bias, None), quant=cs, tok=ts, trans_b=True)
    assert np.array_equal(bits(c), gold)
    if n > 2064 or k > 4096:
        return
    # requantised int8 output from uint64 words (one of them with the pre-shift), int32 bias ahead of the
    # dequantisation; FasterGelu to half from a scalar scale
    words = (cs * 50).astype(np.float32).view(np.uint32).astype(np.uint64) | (np.uint64(1) << np.uint64(46))
    words[n // 2] |= (np.uint64(1) << np.uint64(36)) | (np.uint64(3) << np.uint64(32))
    bias_i = rng.integers(-1000, 1000, n).astype(np.int32)
    c8, d8 = run_mm_packed(m, n, k, a, b, out=torch.int8, bias=(bias_i, None), quant=words)
    gold8 = oracle_mm(d8, a, b, (bias_i, None), words)
    assert np.array_equal(bits(c8), gold8)
    c8, _ = run_mm(m, n, k, a, bt, out=torch.int8, bias=(bias_i, None), quant=words, trans_b=True)
    assert np.array_equal(bits(c8), gold8)
    cg, dg = run_mm_packed(m, n, k, a, b, out=torch.float16, scalar=1e-3, act=abi.MM_ACT_FASTER_GELU)
    assert max_ulp(bits(cg), oracle_mm(dg, a, b).view(np.uint16), "f16") <= 1


@pytest.mark.parametrize("m", [13, 16, 17, 64, 129, 300])
@pytest.mark.parametrize("n,k", [(48, 11008), (272, 8192), (4112, 4160), (1040, 5632), (40, 16384), (96, 14336),
                                 (528, 12352)])
def test_w8a8_weights_held_in_registers_long_k(m, n, k):
    """k beyond 4096 (up to 16384): a wavefront's k range of its slabs is held in chunks of 8 tiles, two slabs by two
    chunks (k up to 8192; n = 4112 gives workgroups two slabs) or one slab by four, and the activations stream past
    them a chunk at a time.  Also the calls of 13 to 16 rows whose staged activations no longer fit the LDS in one
    pass.  int32 accumulators against exact double arithmetic, the dequantising epilogue bit for bit against the
    oracle, packed and [n, k] weights."""
    announce("w8a8 weights in registers, long k", m, n, k)
    rng = np.random.default_rng(m * 41 + n + k)
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    bt = np.ascontiguousarray(b.T)
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.int64)  # sums below 2^53: exact
    c, _ = run_mm_packed(m, n, k, a, b, out=torch.int32)
    assert np.array_equal(c.cpu().numpy(), want)
    c, _ = run_mm(m, n, k, a, bt, out=torch.int32, trans_b=True)
    assert np.array_equal(c.cpu().numpy(), want)
    if n > 2064:
        return
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    ts = rng.uniform(1e-2, 1e-1, m).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c, desc = run_mm_packed(m, n, k, a, b, out=torch.bfloat16, bias=(bias, None), quant=cs, tok=ts)
    gold = oracle_mm(desc, a, b, (bias, None), cs, ts)
    assert np.array_equal(bits(c), gold)
    c, desc = run_mm(m, n, k, a, bt, out=torch.bfloat16, bias=(bias, None), quant=cs, tok=ts, trans_b=True)
    assert np.array_equal(bits(c), gold)


@pytest.mark.parametrize("m", [129, 200, 256, 300, 513, 700, 1100])
@pytest.mark.parametrize("n,k", [(256, 128), (1040, 512), (272, 4096), (2064, 384), (4112 + 16, 256), (96, 1152)])
def test_w8a8_packed_many_rows_on_the_tile_kernels(m, n, k):
    """Many rows on packed weights (n a multiple of 16, k of 128): the direct-to-LDS tile kernels (128 x 128 tiles up to
    512 rows, 256-row tiles beyond, with the narrow tiles of a partly filled last round) read the packed tiles as they
    lie.  int32 accumulators against exact double arithmetic; the dequantising epilogue, the requantising one and
    SwiGLU against the oracle."""
    announce("w8a8 packed, tile kernels", m, n, k)
    rng = np.random.default_rng(m * 43 + n + k)
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.int64)
    c, _ = run_mm_packed(m, n, k, a, b, out=torch.int32)
    assert np.array_equal(c.cpu().numpy(), want)
    if n > 2064:
        return
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    ts = rng.uniform(1e-2, 1e-1, m).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c, desc = run_mm_packed(m, n, k, a, np.ascontiguousarray(b.T), out=torch.bfloat16, bias=(bias, None), quant=cs, tok=ts,
                            trans_b=True)
    assert np.array_equal(bits(c), oracle_mm(desc, a, b, (bias, None), cs, ts))
    words = (cs * 50).astype(np.float32).view(np.uint32).astype(np.uint64) | (np.uint64(1) << np.uint64(46))
    words[n // 2] |= (np.uint64(1) << np.uint64(36)) | (np.uint64(3) << np.uint64(32))
    bias_i = rng.integers(-1000, 1000, n).astype(np.int32)
    c8, d8 = run_mm_packed(m, n, k, a, b, out=torch.int8, bias=(bias_i, None), quant=words)
    assert np.array_equal(bits(c8), oracle_mm(d8, a, b, (bias_i, None), words))
    # SwiGLU of the column pairs in the tile kernels' epilogue (16-bit outputs)
    css = rng.uniform(1e-4, 4e-4, n).astype(np.float32)
    tss = rng.uniform(0.5, 2.0, m).astype(np.float32)
    mm = ops.Matmul(m, n, k, False, False)
    mm.set_tensor_a(to_dev(a))
    mm.set_tensor_b_packed(ops.pack_weight_w8(to_dev(b), k, n))
    mm.set_quant_vector(to_dev(css))
    mm.set_token_scale(to_dev(tss))
    mm.set_activation(abi.MM_ACT_SWIGLU, 1.702)
    cg = torch.zeros((m, n // 2), dtype=torch.bfloat16, device=DEV)
    mm.iterate_all(cg)
    d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32,
                       has_tok_scale=1, activation=abi.MM_ACT_SWIGLU, act_beta=1.702)
    swiglu_close(bits(cg), oracle_mm(d, a, b, None, css, tss).view(np.uint16), "bf16")


@pytest.mark.parametrize("m", [1, 16, 32])
def test_config3_w8a8_linear_packed(m):
    """Config 3's decode sizes on packed weights: per-token quantisation on the GPU, one launch for the matmul, bf16
    output bit-exact against the oracle."""
    announce("config 3 packed", m)
    rng = np.random.default_rng(0xC3 + m)
    k, n = 4096, 11008
    x = orc.f32_to_bf16_bits(rng.standard_normal((m, k)).astype(np.float32))
    w = rand_i8(rng, (k, n))
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    q, ts = ops.dynamic_quant_per_token(to_dev(x, "bf16"))
    wq, wts = orc.dynamic_quant_per_token(abi.BF16, x)
    assert np.array_equal(q.cpu().numpy(), wq) and np.array_equal(ts.cpu().numpy(), wts)
    c, desc = run_mm_packed(m, n, k, wq, w, out=torch.bfloat16, quant=cs, tok=wts)
    assert np.array_equal(bits(c), oracle_mm(desc, wq, w, None, cs, wts))


def test_w8a8_packed_rejects():
    lib = abi.load_library()
    t = torch.zeros(1 << 16, dtype=torch.int8, device=DEV)
    c = torch.zeros(1 << 12, dtype=torch.int32, device=DEV)

    def call(**kw):
        d = abi.MatmulDesc(m=1, n=64, k=128, out_dtype=abi.I32, quant_mode=abi.MM_QUANT_NONE, scale_format=abi.MM_SCALE_U64)
        for key, v in kw.items():
            setattr(d, key, v)
        return lib.ascq_matmul_w8a8_packed(C.byref(d), C.c_void_p(c.data_ptr()), C.c_void_p(t.data_ptr()),
                                           C.c_void_p(t.data_ptr()), None, None, None, None)

    assert call() == abi.OK
    assert call(k=100) == abi.EUNSUPPORTED          # k % 64
    assert call(trans_a=1) == abi.EUNSUPPORTED
    assert call(b_format=abi.MM_B_NZ) != abi.OK
    torch.cuda.synchronize()


@pytest.mark.parametrize("m", [48, 128, 300, 512])
def test_config3_w8a8_mid_m_both_weight_layouts(m):
    """Config 3 between the decode sizes and the large tiles: 128 x 128 direct-to-LDS tiles, K split four ways for one
    row tile and not at all for more, on weights as [k, n]; on [n, k] weights the same tiles from 225 rows on and the
    weights-in-registers kernel below; bit-exact against the oracle."""
    announce("config 3 mid m", m)
    rng = np.random.default_rng(0xC3 + 200 + m)
    k, n = 4096, 11008
    a = rand_i8(rng, (m, k))
    w = rand_i8(rng, (k, n))
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    ts = rng.uniform(1e-2, 1e-1, m).astype(np.float32)
    c, desc = run_mm(m, n, k, a, w, out=torch.bfloat16, quant=cs, tok=ts)
    want = oracle_mm(desc, a, w, None, cs, ts)
    assert np.array_equal(bits(c), want)
    ct, _ = run_mm(m, n, k, a, np.ascontiguousarray(w.T), out=torch.bfloat16, quant=cs, tok=ts, trans_b=True)
    assert np.array_equal(bits(ct), want)
    # [k, n]: one row tile splits K four ways through the workspace; [n, k]: up to 224 rows need none
    wsz = C.c_size_t(0)
    assert abi.load_library().ascq_matmul_w8a8_workspace_size(C.byref(desc), C.byref(wsz)) == abi.OK
    assert wsz.value == (4 * m * n * 4 if m <= 128 else 0)
    desc.trans_b = 1
    assert abi.load_library().ascq_matmul_w8a8_workspace_size(C.byref(desc), C.byref(wsz)) == abi.OK
    assert wsz.value == 0


def test_fixpipe_modes_uint64_words():
    announce("matmul fixpipe words: VDEQF16, DEQF16 scalar, VREQ8, bf16")
    rng = np.random.default_rng(21)
    m, n, k = 64, 256, 256
    a, b = rand_i8(rng, (m, k), -10, 10), rand_i8(rng, (k, n), -10, 10)
    bias = rng.integers(-2, 2, n).astype(np.int32)
    qf = rng.uniform(0.1, 2.0, n).astype(np.float32)
    qf[0], qf[1] = 3000.0, -3000.0
    words = qf.view(np.uint32).astype(np.uint64) | (np.uint64(7) << np.uint64(37)) | (np.uint64(1) << np.uint64(46))
    for out in (torch.float16, torch.bfloat16, torch.int8):
        c, desc = run_mm(m, n, k, a, b, out=out, bias=(bias, None), quant=words)
        want = oracle_mm(desc, a, b, (bias, None), words)
        assert np.array_equal(bits(c), want.view(np.uint16) if out == torch.float16 else want)
    assert (np.abs(bits(run_mm(m, n, k, a, b, out=torch.float16, quant=words)[0]).view(np.float16)
                   .astype(np.float32)) == 65504).any()            # the fp16 output saturates instead of overflowing
    c, desc = run_mm(m, n, k, a, b, out=torch.float16, bias=(bias, None),
                     scalar=ops.pack_quant_param(0.1))
    assert np.array_equal(bits(c), oracle_mm(desc, a, b, (bias, None)).view(np.uint16))
    c, desc = run_mm(m, n, k, a, b, out=torch.float32, scalar=0.1)
    assert np.array_equal(bits(c), oracle_mm(desc, a, b))


@pytest.mark.parametrize("m,n,k,trans_b", [(7, 144, 192, False), (64, 256, 256, False), (12, 272, 256, True),
                                           (200, 528, 384, False), (600, 528, 640, False), (19, 23, 77, False)])
def test_fixpipe_pre_shift_words(m, n, k, trans_b):
    """Quant words with the mode-control bit 36: the accumulator is shifted right by bits [35:32] and saturated before
    the multiply.  Every column draws its own bit and shift; all four output types, and a scalar word."""
    announce(f"matmul fixpipe pre-shift words m={m} n={n} k={k} trans_b={trans_b}")
    rng = np.random.default_rng(1000 + m)
    a = rand_i8(rng, (m, k), -127, 128)
    b = rand_i8(rng, (n, k) if trans_b else (k, n), -127, 128)
    bias = rng.integers(-3000000, 3000000, n).astype(np.int32)
    qf = rng.uniform(0.01, 1.5, n).astype(np.float32)
    sh = rng.integers(0, 16, n).astype(np.uint64)
    on = rng.integers(0, 2, n).astype(np.uint64)
    on[:4], sh[:4] = 1, (0, 1, 4, 15)
    words = (qf.view(np.uint32).astype(np.uint64) | (sh << np.uint64(32)) | (on << np.uint64(36)) |
             (rng.integers(0, 512, n).astype(np.uint64) << np.uint64(37)) |
             (rng.integers(0, 2, n).astype(np.uint64) << np.uint64(46)))
    for out in (torch.float16, torch.int8, torch.bfloat16, torch.float32):
        c, desc = run_mm(m, n, k, a, b, out=out, bias=(bias, None), quant=words, trans_b=trans_b)
        want = oracle_mm(desc, a, b, (bias, None), words)
        assert np.array_equal(bits(c), want.view(np.uint16) if out == torch.float16 else want), out
    plain = words & ~(np.uint64(1) << np.uint64(36))
    c0, _ = run_mm(m, n, k, a, b, out=torch.float16, bias=(bias, None), quant=plain, trans_b=trans_b)
    c1, _ = run_mm(m, n, k, a, b, out=torch.float16, bias=(bias, None), quant=words, trans_b=trans_b)
    assert not np.array_equal(bits(c0), bits(c1)), "bit 36 had no effect"
    if n % 2 == 0 and not trans_b:      # SwiGLU over column pairs that shift differently (small scales keep exp in range)
        sw = words & ~np.uint64(0xFFFFFFFF) | (qf * np.float32(1e-4)).view(np.uint32).astype(np.uint64)
        mm = ops.Matmul(m, n, k)
        mm.set_tensor_a(to_dev(a))
        mm.set_tensor_b(to_dev(b))
        mm.set_quant_vector(to_dev(sw))
        mm.set_bias(to_dev(bias))
        mm.set_activation(abi.MM_ACT_SWIGLU, 1.0)
        c = torch.zeros((m, n // 2), dtype=torch.float16, device=DEV)
        mm.iterate_all(c)
        swiglu_close(bits(c), oracle_mm(mm.desc, a, b, (bias, None), sw).view(np.uint16), "f16")
    scalar = int(np.float32(0.37).view(np.uint32)) | (3 << 32) | (1 << 36) | (9 << 37) | (1 << 46)
    for out in (torch.float16, torch.int8):
        c, desc = run_mm(m, n, k, a, b, out=out, bias=(bias, None), scalar=scalar, trans_b=trans_b)
        want = oracle_mm(desc, a, b, (bias, None))
        assert np.array_equal(bits(c), want.view(np.uint16) if out == torch.float16 else want), out


def gpu_mm(m, n, k, a, b, layout, kind, out, quant, tok, bias):
    mm = ops.Matmul(m, n, k, trans_b=layout == "nk")
    mm.set_tensor_a(a)
    if layout == "packed":
        mm.set_tensor_b_packed(b)
    else:
        mm.set_tensor_b(b)
    mm.set_quant_vector(quant)
    mm.set_token_scale(tok)
    mm.set_bias(bias)
    mm.set_activation({"gelu": abi.MM_ACT_FASTER_GELU, "swiglu": abi.MM_ACT_SWIGLU}.get(kind, abi.MM_ACT_NONE), 1.0)
    c = torch.zeros((m, n // 2 if kind == "swiglu" else n), dtype=out, device=DEV)
    mm.iterate_all(c)
    return c


@pytest.mark.parametrize("k,n,layout", [(3072, 10240, "kn"), (3088, 10008, "kn"), (3200, 10000, "nk"), (3088, 10008, "nk"),
                                        (3136, 10000, "packed")])
@pytest.mark.parametrize("kind", ["plain", "gelu", "swiglu", "words", "shifts"])
def test_w8a8_both_matrix_instructions_agree(k, n, layout, kind):
    """Sums long enough for the 16 x 16 x 64 instruction in 256 x 256 tiles (5 x 40 of them, the last of 3 rows) to a 16-bit type,
    against a float output, which the 32 x 32 x 32 instruction writes, rounded to that type: equal bits, whole and partial last
    steps, every weight layout, the activations, quant words (those with the bit that shifts the accumulator: only against the
    same rows in two calls).  The plain form also against the sums in 64 bits."""
    announce("w8a8 both instructions", k, n, layout, kind)
    g = torch.Generator(device=DEV)
    g.manual_seed(k + n)
    m, cut = 1027, 514
    a = torch.randint(-127, 128, (m, k), dtype=torch.int8, device=DEV, generator=g)
    b = torch.randint(-127, 128, (n, k) if layout == "nk" else (k, n), dtype=torch.int8, device=DEV, generator=g)
    w = ops.pack_weight_w8(b, k, n) if layout == "packed" else b
    tok = torch.rand(m, device=DEV, generator=g) * 0.1 + 1e-3
    cs = torch.rand(n, device=DEV, generator=g) * 1e-4 + 1e-5
    bias = torch.randn(n, device=DEV, generator=g)
    quant, out = cs, torch.bfloat16
    if kind in ("words", "shifts"):
        quant = cs.view(torch.int32).to(torch.int64) & 0xFFFFFFFF
        bias, out = torch.randint(-3000, 3000, (n,), dtype=torch.int32, device=DEV, generator=g), torch.float16
        if kind == "shifts":
            pick = torch.randint(0, 32, (n,), device=DEV, generator=g)
            quant = quant | ((pick & 15) << 32) | ((pick >> 4) << 36)
    elif kind == "gelu":
        bias = bias.to(torch.bfloat16)
    got = gpu_mm(m, n, k, a, w, layout, kind, out, quant, tok, bias)
    parts = [gpu_mm(hi - lo, n, k, a[lo:hi].clone(), w, layout, kind, out, quant, tok[lo:hi].clone(), bias) for lo, hi in ((0, cut), (cut, m))]
    assert torch.equal(got.view(torch.int16), torch.cat(parts).view(torch.int16))
    if kind != "shifts":                     # (a half output rounds a shifted sum once more)
        wide = gpu_mm(m, n, k, a, w, layout, kind, torch.float32, quant, tok, bias)
        assert torch.equal(got.view(torch.int16), wide.to(out).view(torch.int16))
    if kind == "plain":
        acc = a.double() @ (b.double().t().contiguous() if layout == "nk" else b.double())      # exact: below 2^53
        want = (acc.float() * cs * tok[:, None] + bias).to(out)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("layout", ["kn", "nk", "packed"])
@pytest.mark.parametrize("m,n,k", [(520, 528, 128), (600, 264, 256), (513, 528, 384), (1000, 272, 512), (520, 1040, 640), (769, 528, 768),
                                   (2048, 11008, 256)])
def test_w8a8_large_tiles_with_half_outputs(m, n, k, layout):
    """256-row tiles whose loads have one and a half K steps to arrive: one to six K steps (prologue, steady state and both
    peeled ends), row and column remainders; the last size runs 256 x 256 and 256 x 128 tiles in one launch."""
    announce("half outputs", m, n, k, layout)
    rng = np.random.default_rng(m + n + k)
    a, b = rand_i8(rng, (m, k), -128, 127), rand_i8(rng, (k, n), -128, 127)
    sc, tok = rng.uniform(1e-4, 1e-3, n).astype(np.float32), rng.uniform(5e-3, 2e-2, m).astype(np.float32)
    mm = ops.Matmul(m, n, k, False, layout == "nk")
    mm.set_tensor_a(to_dev(a))
    if layout == "packed":
        mm.set_tensor_b_packed(ops.pack_weight_w8(to_dev(b), k, n))
    else:
        mm.set_tensor_b(to_dev(np.ascontiguousarray(b.T) if layout == "nk" else b))
    mm.set_quant_vector(to_dev(sc))
    mm.set_token_scale(to_dev(tok))
    want = None
    for out in (torch.bfloat16, torch.float16):
        c = torch.zeros((m, n), dtype=out, device=DEV)
        mm.iterate_all(c)
        # fp32 with one rounding per step, then one to the output (float32 holds every sum of up to 768 products exactly)
        if want is None:
            want = (a.astype(np.float32) @ b.astype(np.float32)) * sc * tok[:, None]
        assert torch.equal(c.cpu(), torch.from_numpy(want).to(out))


@pytest.mark.parametrize("layout", ["kn", "nk", "packed"])
@pytest.mark.parametrize("m,n,k", [(1030, 3344, 768), (1030, 3344, 896), (1030, 3344, 1024), (520, 528, 1408), (520, 528, 1536), (600, 264, 1664),
                                   (2304, 14600, 1408), (2304, 14600, 1536)])
def test_w8a8_half_outputs_on_both_sides_of_the_instruction_rule(m, n, k, layout):
    """256-row tiles to half: 70 of them change to the 16 x 16 x 64 instruction at seven K steps, few (6) and many (more than
    two rounds of the chip) at twelve; even and odd numbers of steps of both, against the sums in 64 bits."""
    announce("instruction rule", m, n, k, layout)
    g = torch.Generator(device=DEV)
    g.manual_seed(m + n + k)
    a = torch.randint(-127, 128, (m, k), dtype=torch.int8, device=DEV, generator=g)
    b = torch.randint(-127, 128, (n, k) if layout == "nk" else (k, n), dtype=torch.int8, device=DEV, generator=g)
    w = ops.pack_weight_w8(b, k, n) if layout == "packed" else b
    tok = torch.rand(m, device=DEV, generator=g) * 0.1 + 1e-3
    cs = torch.rand(n, device=DEV, generator=g) * 1e-4 + 1e-5
    bias = torch.randn(n, device=DEV, generator=g)
    acc = a.double() @ (b.double().t().contiguous() if layout == "nk" else b.double())      # exact: below 2^53
    want = acc.float() * cs * tok[:, None] + bias                                           # one rounding per step
    for out in (torch.bfloat16, torch.float16):
        got = gpu_mm(m, n, k, a, w, layout, "plain", out, cs, tok, bias)
        assert torch.equal(got.view(torch.int16), want.to(out).view(torch.int16))


@pytest.mark.parametrize("kind", ["plain", "gelu", "swiglu"])
def test_group_matmul_both_matrix_instructions_agree(kind):
    """The grouped matmul at a size for the 16 x 16 x 64 instruction against the plain matmul of each group's rows to a float
    output, which the 32 x 32 x 32 instruction writes, rounded to the grouped one's type."""
    announce("grouped matmul, both instructions", kind)
    g = torch.Generator(device=DEV)
    g.manual_seed(3)
    counts, k, n = [513, 0, 300, 260], 3072, 10240
    m = sum(counts)
    x = torch.randint(-127, 128, (m, k), dtype=torch.int8, device=DEV, generator=g)
    w = torch.randint(-127, 128, (len(counts), k, n), dtype=torch.int8, device=DEV, generator=g)
    tok = torch.rand(m, device=DEV, generator=g) * 0.1 + 1e-3
    cs = torch.rand((len(counts), n), device=DEV, generator=g) * 1e-4 + 1e-5
    bias = torch.randn((len(counts), n), device=DEV, generator=g).to(torch.bfloat16)
    y = torch.zeros((m, n // 2 if kind == "swiglu" else n), dtype=torch.bfloat16, device=DEV)
    ops.quant_group_matmul(y, x, w, torch.tensor(counts, dtype=torch.int64, device=DEV), cs, tok, bias,
                           activation={"gelu": abi.MM_ACT_FASTER_GELU, "swiglu": abi.MM_ACT_SWIGLU}.get(kind, abi.MM_ACT_NONE))
    first = 0
    for i, c in enumerate(counts):
        if c:
            rows = slice(first, first + c)
            want = gpu_mm(c, n, k, x[rows].clone(), w[i], "kn", kind, torch.float32, cs[i].clone(), tok[rows].clone(), bias[i].clone())
            assert torch.equal(y[rows].view(torch.int16), want.to(torch.bfloat16).view(torch.int16)), i
        first += c


@pytest.mark.parametrize("k", [128, 384, 1408, 2560])
@pytest.mark.parametrize("nz", [False, True])
@pytest.mark.parametrize("n", [544, 1632, 2080, 2720])
@pytest.mark.parametrize("counts", [[300, 64, 1, 130, 0, 96, 65, 17], [33, 128, 0, 16, 480, 5], [1] * 7 + [0] * 57, [3] * 70])
@pytest.mark.parametrize("act", ["none", "swiglu"])
def test_group_matmul_tile_shapes_by_width(counts, n, nz, k, act):
    """The widths on both sides of the rule that names the tiles (64 x 64, 64 x 128, 128 x 128 with a ring of stages, and those of 256 rows): fewer K
    steps than stages and more, groups without rows, one to 300 rows, 64 groups and more than the ring's kernel scans; counts
    and prefix sums of more rows than there are give the same."""
    announce("grouped, shapes by width", counts[:8], n, nz, k, act)
    g = torch.Generator(device=DEV)
    g.manual_seed(k + n)
    gr, m = len(counts), sum(counts)
    x = torch.randint(-127, 128, (m, k), dtype=torch.int8, device=DEV, generator=g)
    w = torch.randint(-127, 128, (gr, k, n), dtype=torch.int8, device=DEV, generator=g)
    tok = torch.rand(m, device=DEV, generator=g) * 0.02 + 5e-3
    cs = torch.rand((gr, n), device=DEV, generator=g) * 1e-3 + 1e-4
    wd = ops.pack_weight_nz(w) if nz else w
    code = abi.MM_ACT_SWIGLU if act == "swiglu" else abi.MM_ACT_NONE
    out = n // 2 if act == "swiglu" else n
    room = torch.zeros((m + 1) * out, dtype=torch.float16, device=DEV)
    y = room[:m * out].view(m, out)
    ops.quant_group_matmul(y, x, wd, torch.tensor(counts, dtype=torch.int64, device=DEV), cs, tok, activation=code, weight_nz=nz)
    assert not room[m * out:].any()
    r = 0
    for i, c in enumerate(counts):       # (float64 holds the sums exactly; one fp32 rounding per step of the epilogue)
        if c and (gr < 20 or i % 9 == 0):
            v = (x[r:r + c].double() @ w[i].double()).float() * cs[i] * tok[r:r + c, None]
            if act == "swiglu":
                a, b = v[:, 0::2].double(), v[:, 1::2].double()
                want = a * (b / (1.0 + torch.exp(-b)))
                assert ((y[r:r + c].double() - want).abs() <= 2.0 ** -10 * want.abs() + 1e-4).all(), i
            else:
                assert torch.equal(y[r:r + c], v.half()), i
        r += c
    y2 = torch.zeros_like(y)
    big = torch.tensor(counts, dtype=torch.int64, device=DEV).cumsum(0)
    big[-1] += 1000
    ops.quant_group_matmul(y2, x, wd, big, cs, tok, activation=code, weight_nz=nz, group_list_kind=abi.GROUP_LIST_PREFIX_SUM)
    assert torch.equal(y2.view(torch.int16), y.view(torch.int16))


# counts, and the k from which on they run the form whose loads are spread over a step and a half
GROUP_REMAINDERS = [([300, 64, 1, 130, 0, 96, 65, 17], 2560), ([33, 128, 256, 16, 480, 385], 1408), ([257, 512, 64, 384], 1280)]
GROUP_WIDE = 2592      # columns, wide enough for tiles of 256 rows (544: tiles of 64 x 64 with a ring of stages)


@pytest.mark.parametrize("k", [256, 384, 1280, 1408, 2432, 2560, 3072, 3200])
@pytest.mark.parametrize("nz", [False, True])
@pytest.mark.parametrize("counts", [counts for counts, _ in GROUP_REMAINDERS])
@pytest.mark.parametrize("n", [544, GROUP_WIDE])
def test_group_matmul_remainders_in_both_forms(counts, nz, k, n):
    """Remainders of 64 and of 128 rows, and big tiles whose second wavefront row is empty, partly filled or full, on both
    sides of the rule that names the instruction: from k = 2560, 1408 and 1280 on (84, 216 and 304 rows per group) the form
    whose loads are spread over a step and a half; even and odd numbers of K steps.  The narrow width runs the ring's tiles."""
    announce("group remainders", counts, nz, k, n)
    rng = np.random.default_rng(k + len(counts) + nz)
    g, m = len(counts), sum(counts)
    x, w = rand_i8(rng, (m, k)), rand_i8(rng, (g, k, n))
    sc, tok = rng.uniform(1e-4, 1e-3, (g, n)).astype(np.float32), rng.uniform(5e-3, 2e-2, m).astype(np.float32)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    wd = to_dev(w)
    ops.quant_group_matmul(y, to_dev(x), ops.pack_weight_nz(wd) if nz else wd, torch.tensor(counts, dtype=torch.int64, device=DEV),
                           to_dev(sc), to_dev(tok), weight_nz=nz)
    want, r = np.zeros((m, n), np.float32), 0
    for i, c in enumerate(counts):      # (float64 holds the sums exactly; one fp32 rounding per step of the epilogue)
        sums = (x[r:r + c].astype(np.float64) @ w[i].astype(np.float64)).astype(np.float32)
        want[r:r + c] = sums * sc[i] * tok[r:r + c, None]
        r += c
    assert torch.equal(y.cpu(), torch.from_numpy(want).to(torch.float16))


def test_post_bias_bf16_and_gelu():
    announce("matmul bf16 bias + token scale + FasterGelu")
    rng = np.random.default_rng(22)
    m, n, k = 96, 512, 384
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    cs = rng.uniform(1e-4, 1e-3, n).astype(np.float32)
    ts = rng.uniform(1e-2, 1e-1, m).astype(np.float32)
    bias = orc.f32_to_bf16_bits(rng.standard_normal(n).astype(np.float32))
    c, desc = run_mm(m, n, k, a, b, out=torch.bfloat16, bias=(bias, "bf16"), quant=cs, tok=ts)
    assert np.array_equal(bits(c), oracle_mm(desc, a, b, (bias, None), cs, ts))
    c, desc = run_mm(m, n, k, a, b, out=torch.float16, quant=cs, tok=ts, act=abi.MM_ACT_FASTER_GELU)
    want = oracle_mm(desc, a, b, None, cs, ts)
    assert max_ulp(bits(c), want.view(np.uint16)) <= 1             # expf differs by at most an ulp of fp32


# ------------------------------------------------------------------ grouped matmul
def run_group(m, k, n, counts, kind, out, rng, with_bias, act, rows_cap=None):
    G = len(counts)
    x, w = rand_i8(rng, (m, k)), rand_i8(rng, (G, k, n))
    cs = rng.uniform(1e-4, 1e-2, (G, n)).astype(np.float32)
    ts = rng.uniform(1e-3, 1e-1, m).astype(np.float32)
    bias = orc.f32_to_bf16_bits(rng.standard_normal((G, n)).astype(np.float32)) if with_bias else None
    gl = np.asarray(counts, dtype=np.int64) if kind == abi.GROUP_LIST_COUNTS else np.cumsum(counts).astype(np.int64)
    y = torch.zeros((m, n), dtype=out, device=DEV)
    y.view(torch.int16).fill_(0x7E7E)
    ops.quant_group_matmul(y, to_dev(x), to_dev(w), to_dev(gl), to_dev(cs), to_dev(ts),
                           None if bias is None else to_dev(bias, "bf16"), kind, act)
    torch.cuda.synchronize()
    mm = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16 if out == torch.bfloat16 else abi.F16,
                        quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32, has_tok_scale=1,
                        bias_kind=abi.MM_BIAS_BF16_POST if with_bias else abi.MM_BIAS_NONE, activation=act)
    d = abi.GroupMatmulDesc(mm=mm, groups=G, group_list_kind=kind)
    orc.set_threads(16)
    want = orc.group_matmul_w8a8(d, x, w, bias, cs, ts, gl, fill=0x7E7E)
    return bits(y), (want.view(np.uint16) if want.dtype == np.float16 else want)


GROUP_EDGES = [[30, 0, 1, 45, 12], [256, 256], [0, 0, 700, 0], [1, 1, 1, 1, 1, 1, 1, 1], [513, 255, 0, 256]]
GROUP_EDGES_WIDE = 6664      # columns, wide enough for tiles of 256 rows (520: the ring's tiles)


@pytest.mark.parametrize("kind", [abi.GROUP_LIST_COUNTS, abi.GROUP_LIST_PREFIX_SUM])
@pytest.mark.parametrize("counts", GROUP_EDGES)
@pytest.mark.parametrize("n", [520, GROUP_EDGES_WIDE])
def test_group_matmul_edge_cases(kind, counts, n):
    announce("grouped matmul", kind, counts, n)
    rng = np.random.default_rng(sum(counts) + len(counts))
    m = sum(counts) + 8                                         # 8 rows belong to no group and stay untouched
    got, want = run_group(m, 256, n, counts, kind, torch.bfloat16, rng, True, abi.MM_ACT_NONE)
    assert np.array_equal(got, want)
    assert np.all(got[sum(counts):] == 0x7E7E)


def test_group_matmul_reference_example_form():
    """The reference example's form: counts group list, no bias, FasterGelu, fp16 output."""
    announce("grouped matmul, example form")
    rng = np.random.default_rng(77)
    got, want = run_group(512, 256, 512, [128] * 4, abi.GROUP_LIST_COUNTS, torch.float16, rng, False,
                          abi.MM_ACT_FASTER_GELU)
    assert max_ulp(got, want) <= 1


def test_config5_moe_up_projection():
    """8 experts, 4096 tokens from a seeded multinomial, K=4096, N=14336, bf16 bias, prefix-sum group list."""
    announce("config 5")
    rng = np.random.default_rng(0xC5)
    counts = rng.multinomial(4096, [1 / 8] * 8).tolist()
    got, want = run_group(4096, 4096, 14336, counts, abi.GROUP_LIST_PREFIX_SUM, torch.bfloat16, rng, True,
                          abi.MM_ACT_NONE)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("counts,act", [([600, 40, 560], abi.MM_ACT_NONE), ([200, 0, 513, 129, 128, 1], abi.MM_ACT_FASTER_GELU),
                                        ([300, 300, 300, 300], abi.MM_ACT_SWIGLU)])
def test_group_matmul_all_tile_shapes(counts, act):
    """Enough 256-row tiles and tile columns that the launch holds a whole round of 256 x 256 tiles, a partial round
    of 256 x 128 tiles (the last of them 80 columns wide) and 128-row tiles for the groups' short remainders; groups
    with 128, 129 and 200 remainder rows sit on either side of the rule that picks the row-tile height."""
    announce("grouped matmul, every tile shape", counts, act)
    rng = np.random.default_rng(len(counts))
    m, k, n = sum(counts) + 3, 128, 16976
    out = torch.float16 if act == abi.MM_ACT_FASTER_GELU else torch.bfloat16
    if act == abi.MM_ACT_SWIGLU:
        x, w = rand_i8(rng, (m, k)), rand_i8(rng, (len(counts), k, n))
        cs = rng.uniform(1e-4, 1e-3, (len(counts), n)).astype(np.float32)
        ts = rng.uniform(1e-2, 1e-1, m).astype(np.float32)
        gl = np.asarray(counts, dtype=np.int64)
        y = torch.zeros((m, n // 2), dtype=out, device=DEV)
        y.view(torch.int16).fill_(0x7E7E)
        ops.quant_group_matmul(y, to_dev(x), to_dev(w), to_dev(gl), to_dev(cs), to_dev(ts), None, abi.GROUP_LIST_COUNTS,
                               act, act_beta=1.0)
        torch.cuda.synchronize()
        mm = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR,
                            scale_format=abi.MM_SCALE_F32, has_tok_scale=1, activation=act, act_beta=1.0)
        orc.set_threads(16)
        want = orc.group_matmul_w8a8(abi.GroupMatmulDesc(mm=mm, groups=len(counts), group_list_kind=abi.GROUP_LIST_COUNTS),
                                     x, w, None, cs, ts, gl, fill=0x7E7E)
        got = bits(y)
        assert np.all(got[sum(counts):] == 0x7E7E)
        rows = sum(counts)
        assert max_ulp(got[:rows], want.view(np.uint16)[:rows], "bf16") <= 1  # expf differs by at most an ulp of fp32
        assert np.mean(got[:rows] == want.view(np.uint16)[:rows]) > 0.98
        return
    got, want = run_group(m, k, n, counts, abi.GROUP_LIST_COUNTS, out, rng, act == abi.MM_ACT_NONE, act)
    if act == abi.MM_ACT_NONE:
        assert np.array_equal(got, want)
    else:
        assert np.all(got[sum(counts):] == 0x7E7E)
        assert max_ulp(got[:sum(counts)], want[:sum(counts)]) <= 1


# ------------------------------------------------------------------ W4A16
def w4_case(rng, m, k, n, gs, has_offset):
    x = rng.standard_normal((m, k)).astype(np.float16)
    w = rng.integers(-8, 8, (k, n)).astype(np.int8)
    sc = rng.uniform(1e-3, 1e-2, (k // gs, n)).astype(np.float16)
    of = rng.integers(-8, 8, (k // gs, n)).astype(np.float16) if has_offset else None
    return x, pack_int4(w), sc, of


@pytest.mark.parametrize("m", [1, 2, 3, 4, 7, 9, 16, 19, 32, 33, 37, 70])
@pytest.mark.parametrize("k,n,gs", [(512, 1024, 128), (1024, 544, 64), (256, 66, 128), (384, 512, 384)])
@pytest.mark.parametrize("has_offset", [True, False])
def test_w4a16_small(m, k, n, gs, has_offset):
    announce("w4a16", m, k, n, gs, has_offset)
    rng = np.random.default_rng(m + k + n)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, has_offset)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.matmul_w4a16(y, to_dev(x), to_dev(wp), to_dev(sc), None if of is None else to_dev(of), gs)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=int(has_offset))
    want = orc.matmul_w4a16(d, x, wp, sc, of)
    got = y.cpu().numpy()
    # fp32 accumulation in a different order than the oracle's: rel-err <= 1e-3 of the row scale, and <= 1 fp16 ulp
    # wherever the result is not close to a cancellation
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    ref = np.abs(x.astype(np.float64)).sum(axis=1, keepdims=True) * 8 * 1e-2      # bound on sum |x||w|
    assert np.all(err <= 1e-3 * ref + 1e-6)
    assert np.mean(got.view(np.uint16) == want.view(np.uint16)) > 0.9


def w4_packed_reference(w_bytes, k, n):
    """The packed int4 layout restated in numpy: slabs of 16 columns, tiles of 128 k, lane l of a tile owns column l % 16
    and k 32 (l / 16) .. + 31, dword d holds k + 8 d .. + 7 with k offsets 0..7 in nibbles 0 4 1 5 2 6 3 7, nibbles stored as
    w + 8; 16 tiles of w = 0 behind the last slab."""
    slabs, ktiles = (n + 15) // 16, (k + 127) // 128
    u = np.full((ktiles * 128, slabs * 16), 8, dtype=np.uint32)                    # w = 0 where there is no weight
    lo, hi = w_bytes & 15, w_bytes >> 4
    nib = np.empty((k, n), dtype=np.uint32)
    nib[:, 0::2], nib[:, 1::2] = lo, hi
    u[:k, :n] = nib ^ 8
    u = u.reshape(ktiles, 4, 4, 8, slabs, 16)                                      # tile, g, d, e, slab, j
    pos = np.array([0, 4, 1, 5, 2, 6, 3, 7], dtype=np.uint32)                      # nibble of k offset e
    words = (u << (4 * pos)[None, None, None, :, None, None]).sum(axis=3, dtype=np.uint64).astype(np.uint32)
    words = words.transpose(3, 0, 1, 4, 2)                                         # slab, tile, g, j, d
    body = np.ascontiguousarray(words).reshape(-1)
    pad = np.full(16 * 256, 0x88888888, dtype=np.uint32)
    return np.concatenate([body, pad]).view(np.uint8)


@pytest.mark.parametrize("k,n", [(128, 16), (256, 40), (384, 1040), (1024, 272)])
def test_pack_weight_w4_layout(k, n):
    announce("pack w4", k, n)
    rng = np.random.default_rng(k + n)
    wp = pack_int4(rng.integers(-8, 8, (k, n)).astype(np.int8))
    got = ops.pack_weight_w4(to_dev(wp), k, n).cpu().numpy()
    assert np.array_equal(got, w4_packed_reference(wp, k, n))


def w4_check(got, want, x):
    # fp32 accumulation in a different order than the oracle's: rel-err <= 1e-3 of the row scale, and bit-identical
    # halves nearly everywhere (<= 1 fp16 ulp wherever the result is not close to a cancellation)
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    ref = np.abs(x.astype(np.float64)).sum(axis=1, keepdims=True) * 8 * 1e-2      # bound on sum |x||w|
    assert np.all(err <= 1e-3 * ref + 1e-6)
    assert np.mean(got.view(np.uint16) == want.view(np.uint16)) > 0.9


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 9, 16, 17, 33])
@pytest.mark.parametrize("k,n,gs", [(512, 1024, 128), (1024, 544, 64), (256, 40, 32), (384, 512, 128), (2048, 272, 256),
                                     (2048, 64, 512), (128, 4112, 128)])
@pytest.mark.parametrize("offset", ["int", "frac", None])
def test_w4a16_packed_small(m, k, n, gs, offset):
    """The pre-packed weight path computes what the [k, n / 2] path computes (same oracle)."""
    announce("w4a16 packed", m, k, n, gs, offset)
    rng = np.random.default_rng(m + k + n)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, offset is not None)
    if offset == "frac":
        of = (rng.standard_normal((k // gs, n)) * 3).astype(np.float16)
    w_gpu = ops.pack_weight_w4(to_dev(wp), k, n)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.matmul_w4a16_packed(y, to_dev(x), w_gpu, to_dev(sc), None if of is None else to_dev(of), gs)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=int(of is not None))
    w4_check(y.cpu().numpy(), orc.matmul_w4a16(d, x, wp, sc, of), x)


@pytest.mark.parametrize("m,k,n,gs", [(5, 1024, 1152, 64), (16, 1408, 264, 128), (17, 1792, 1440, 32), (33, 2304, 1152, 128), (64, 1152, 2976, 64),
                                       (96, 1280, 96, 128), (48, 4224, 32, 32)])
@pytest.mark.parametrize("offset", [True, False])
def test_w4a16_few_rows_repacked_or_in_passes(m, k, n, gs, offset):
    """[k, n / 2] weights of which some are repacked into the workspace first and some run as passes (5 rows; (48, 4224, 32, 32) has
    more groups than the repacked form is taken for): the oracle's values; a workspace too small for the passes is refused where
    the repacked weights do not fit it either.  (A workspace for the passes and not for the repacked weights: a test below.)"""
    import ctypes as C
    announce("w4a16 few rows", m, k, n, gs, offset)
    rng = np.random.default_rng(m + k + n)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, offset)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=int(offset))
    want = orc.matmul_w4a16(d, x, wp, sc, of)
    need, packed = C.c_size_t(0), C.c_size_t(0)
    lib = ops.load_library()
    assert lib.ascq_matmul_w4a16_workspace_size(C.byref(d), C.byref(need)) == abi.OK
    assert lib.ascq_pack_weight_w4_size(k, n, C.byref(packed)) == abi.OK
    for room in [need.value] + ([packed.value - 16] if n % 32 == 0 else []):
        y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
        ws = torch.zeros(room, dtype=torch.uint8, device=DEV)
        xd, wd, sd, od = to_dev(x), to_dev(wp), to_dev(sc), to_dev(of) if offset else None
        rc = lib.ascq_matmul_w4a16(C.byref(d), ops._ptr(y), ops._ptr(xd), ops._ptr(wd), ops._ptr(sd), ops._ptr(od), ops._ptr(ws), room, ops._stream())
        if rc == abi.EINVAL and room < need.value:
            continue      # too small for the passes as well: refused
        assert rc == abi.OK
        w4_check(y.cpu().numpy(), want, x)


def test_w4a16_packed_multi_pass_and_repeatable():
    """k too long for one pass of staged activations (several passes per wavefront), and two calls give identical bits."""
    m, k, n, gs = 4, 24576, 256, 128
    announce("w4a16 packed long k", m, k, n)
    rng = np.random.default_rng(5)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, True)
    w_gpu = ops.pack_weight_w4(to_dev(wp), k, n)
    xs, scs, ofs = to_dev(x), to_dev(sc), to_dev(of)
    y1 = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    y2 = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.matmul_w4a16_packed(y1, xs, w_gpu, scs, ofs, gs)
    ops.matmul_w4a16_packed(y2, xs, w_gpu, scs, ofs, gs)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=1)
    w4_check(y1.cpu().numpy(), orc.matmul_w4a16(d, x, wp, sc, of), x)
    assert torch.equal(y1, y2)


@pytest.mark.parametrize("m,k,n,gs", [(7, 3200, 144, 64), (16, 5248, 48, 128), (12, 1024, 2320, 1024),
                                      (8, 8192, 64, 32)])
def test_w4a16_packed_more_than_four_rows(m, k, n, gs):
    """5 to 16 rows on packed weights: one wavefront per slab over all of k, activations shared chunk by chunk.  k of
    several chunks with a short last one, a last workgroup with idle wavefronts, one group per chunk; the last case has
    more quantisation groups than that kernel stages and runs the kernel of the few-row case in several passes.  Two
    calls give identical bits."""
    announce("w4a16 packed rows", m, k, n, gs)
    rng = np.random.default_rng(m * 131 + k + n)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, True)
    w_gpu = ops.pack_weight_w4(to_dev(wp), k, n)
    xs, scs, ofs = to_dev(x), to_dev(sc), to_dev(of)
    y1 = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    y2 = torch.full((m, n), 7.0, dtype=torch.float16, device=DEV)
    ops.matmul_w4a16_packed(y1, xs, w_gpu, scs, ofs, gs)
    ops.matmul_w4a16_packed(y2, xs, w_gpu, scs, ofs, gs)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=1)
    w4_check(y1.cpu().numpy(), orc.matmul_w4a16(d, x, wp, sc, of), x)
    assert torch.equal(y1, y2)


W4_MANY_ROWS = {"wq_rows_kernel": [(49, 128, 8, 32), (128, 256, 248, 64), (129, 384, 264, 128), (257, 640, 520, 128)],
                "wq_gemm_kernel<128, 128, ": [(300, 128, 1032, 32), (69, 128, 2312, 32), (129, 384, 5128, 64), (257, 640, 6152, 32), (1030, 1152, 2056, 128)],
                "wq_gemm_kernel<256, 256, ": [(1300, 256, 14600, 256)]}


@pytest.mark.parametrize("m,k,n,gs", [s for sizes in W4_MANY_ROWS.values() for s in sizes])
@pytest.mark.parametrize("offset", ["int", "frac", None])
def test_w4a16_packed_many_rows(m, k, n, gs, offset):
    """More rows than a few passes: the half GEMM whose B-tile loader de-quantises the packed tiles.  Two steps of k and more, row
    and column tails, groups of half a step, on tiles of 128 x 128; the last case runs 256 x 256 ones, those beyond a whole
    round cut in half (wide ones are checked on their first, a middle and the last columns); few rows or columns run whole-k tiles."""
    announce("w4a16 packed many rows", m, k, n, gs, offset)
    rng = np.random.default_rng(m + 3 * k + n)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, offset is not None)
    if offset == "frac":
        of = (rng.standard_normal((k // gs, n)) * 3).astype(np.float16)
    w_gpu = ops.pack_weight_w4(to_dev(wp), k, n)
    y = torch.full((m, n), 7.0, dtype=torch.float16, device=DEV)
    ops.matmul_w4a16_packed(y, to_dev(x), w_gpu, to_dev(sc), None if of is None else to_dev(of), gs)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=int(of is not None))
    orc.set_threads(16)
    for c0, c1 in [(0, n)] if n < 2000 else [(0, 80), (n // 2, n // 2 + 80), (n - 80, n)]:
        want = orc.matmul_w4a16(d, x, wp, sc, of, cols=(c0, c1))[:, c0:c1]
        w4_check(np.ascontiguousarray(y.cpu().numpy()[:, c0:c1]), np.ascontiguousarray(want), x)


W4_WHOLE_K = {(16, 16): [(36, 4096, 1032, 64), (12, 4224, 1032, 128)], (32, 16): [(21, 1152, 3336, 128), (5, 128, 8, 128), (17, 384, 24, 32)],
              (32, 32): [(129, 1152, 1544, 32), (30, 1920, 5320, 128)], (64, 16): [(40, 1280, 3336, 128)],
              (64, 32): [(60, 2176, 5128, 64), (40, 1280, 6504, 128)], (64, 64): [(100, 1152, 7208, 32), (85, 1152, 6920, 64), (80, 1152, 7400, 128)],
              (): [(85, 1408, 13320, 128)]}  # (per weight 128 x 128, as group sums 64 x 64)


@pytest.mark.parametrize("m,k,n,gs", [s for sizes in W4_WHOLE_K.values() for s in sizes])
@pytest.mark.parametrize("offset", ["frac", None])
@pytest.mark.parametrize("mode", [abi.W4A16_PER_WEIGHT, abi.W4A16_GROUP_SUM])
def test_w4a16_packed_whole_k_tiles(m, k, n, gs, offset, mode):
    """Rows and columns that leave the large tiles' chip idle: every tile of 16 x 16 to 64 x 64 in both forms (row and column tails, k that the
    eight wavefronts cannot share evenly, a half-filled last stage), and calls shorter than the wavefronts' smallest share.
    (Groups that are no multiple of 128 run the per-weight form.)  Two calls give identical bits, past the last row nothing is written."""
    announce("w4a16 packed whole-k tiles", m, k, n, gs, offset, mode)
    rng = np.random.default_rng(m + 5 * k + n)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, offset is not None)
    if offset == "frac":
        of = (rng.standard_normal((k // gs, n)) * 3).astype(np.float16)
    w_gpu = ops.pack_weight_w4(to_dev(wp), k, n)
    xd, sd, od = to_dev(x), to_dev(sc), None if of is None else to_dev(of)
    # (the outputs begin 2 bytes off an 8-byte line: no wide stores)
    buf = [torch.full(((m + 1) * n + 1,), 7.0, dtype=torch.float16, device=DEV) for _ in range(2)]
    ys = [b[j:j + m * n].view(m, n) for j, b in enumerate(buf)]
    for y in ys:
        ops.matmul_w4a16_packed(y, xd, w_gpu, sd, od, gs, mode=mode)
    assert torch.equal(ys[0].reshape(-1).view(torch.int16), ys[1].reshape(-1).view(torch.int16))
    assert all(bool((b[j + m * n:] == 7.0).all()) for j, b in enumerate(buf))
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=int(of is not None))
    orc.set_threads(16)
    for c0, c1 in [(0, n)] if n < 4000 else [(0, 80), (n // 2, n // 2 + 80), (n - 80, n)]:
        want = np.ascontiguousarray(orc.matmul_w4a16(d, x, wp, sc, of, cols=(c0, c1))[:, c0:c1])
        got = np.ascontiguousarray(ys[0].cpu().numpy()[:, c0:c1])
        if mode == abi.W4A16_GROUP_SUM:
            w4_group_sum_gate(got, want)
        else:
            w4_check(got, want, x)


@pytest.mark.parametrize("m", [36, 140, 700])
def test_w4a16_group_sum_whole_k_tiles_are_the_real_number_value(m):
    """The group-sum form with more rows than a pass: on inputs whose products and sums are exact in fp32 (as above, at most
    2^23 in units of 2^-6 with k = 1024) it gives the exact value."""
    k, n, gs = 1024, 1032, 256
    announce("w4a16 packed group sum, many rows, exact", m, k, n)
    rng = np.random.default_rng(78 + m)
    x = rng.integers(-4, 5, (m, k)).astype(np.float16)
    w = rng.integers(-8, 8, (k, n)).astype(np.int8)
    sc = (2.0 ** rng.integers(-6, -2, (k // gs, n))).astype(np.float16)
    of = rng.integers(-8, 8, (k // gs, n)).astype(np.float16)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.matmul_w4a16_packed(y, to_dev(x), ops.pack_weight_w4(to_dev(pack_int4(w)), k, n), to_dev(sc), to_dev(of), gs,
                            mode=abi.W4A16_GROUP_SUM)
    xg = x.astype(np.float64).reshape(m, k // gs, gs)
    wg = w.astype(np.float64).reshape(k // gs, gs, n)
    want = sum((xg[:, g] @ wg[g] + xg[:, g].sum(axis=1)[:, None] * of[g].astype(np.float64)[None]) * sc[g].astype(np.float64)[None]
               for g in range(k // gs))
    assert np.array_equal(y.cpu().numpy(), want.astype(np.float16))


@pytest.mark.parametrize("m,k,n,gs", [(8, 1152, 18064, 128), (12, 640, 26400, 64), (6, 5248, 28720, 128)])
@pytest.mark.parametrize("mode", [abi.W4A16_PER_WEIGHT, abi.W4A16_GROUP_SUM])
def test_w4a16_packed_rows_kernel_wide(m, k, n, gs, mode):
    """5 to 16 rows and as many columns as give every compute unit a full workgroup: the kernel with one wavefront per slab (chunks of
    1024 k with a short last one, a last workgroup with idle wavefronts)."""
    announce("w4a16 packed rows, wide", m, k, n, gs, mode)
    rng = np.random.default_rng(m * 131 + k + n)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, True)
    y = torch.full((m, n), 7.0, dtype=torch.float16, device=DEV)
    ops.matmul_w4a16_packed(y, to_dev(x), ops.pack_weight_w4(to_dev(wp), k, n), to_dev(sc), to_dev(of), gs, mode=mode)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=1)
    orc.set_threads(16)
    for c0, c1 in [(0, 80), (n // 2, n // 2 + 80), (n - 80, n)]:
        want = np.ascontiguousarray(orc.matmul_w4a16(d, x, wp, sc, of, cols=(c0, c1))[:, c0:c1])
        got = np.ascontiguousarray(y.cpu().numpy()[:, c0:c1])
        w4_group_sum_gate(got, want) if mode == abi.W4A16_GROUP_SUM else w4_check(got, want, x)


W4_PACKED_FIRST = {"wq_rows_kernel": [(97, 128, 8, 32), (98, 384, 40, 128), (130, 256, 528, 64), (200, 640, 1032, 128)],
                   "wq_gemm_kernel<128, 128, ": [(140, 256, 4104, 32), (300, 640, 5000, 128)]}


@pytest.mark.parametrize("m,k,n,gs", [s for sizes in W4_PACKED_FIRST.values() for s in sizes])
@pytest.mark.parametrize("offset", [True, False])
def test_w4a16_many_rows_packs_the_weights_first(m, k, n, gs, offset):
    """More than 96 rows on [k, n] weights: the call packs them into its workspace and runs the packed form (whole-k tiles or tiles
    of 128 x 128), whose bits it has; the workspace that a call of 32 rows asks for is accepted."""
    announce("w4a16 many rows", m, k, n, gs, offset)
    rng = np.random.default_rng(m + k + n)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, offset)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=int(offset))
    want = orc.matmul_w4a16(d, x, wp, sc, of)
    xd, wd, sd, od = to_dev(x), to_dev(wp), to_dev(sc), None if of is None else to_dev(of)
    y, yp = (torch.zeros((m, n), dtype=torch.float16, device=DEV) for _ in range(2))
    ops.matmul_w4a16(y, xd, wd, sd, od, gs)
    w4_check(y.cpu().numpy(), want, x)
    ops.matmul_w4a16_packed(yp, xd, ops.pack_weight_w4(wd, k, n), sd, od, gs)
    assert torch.equal(y.view(torch.int16), yp.view(torch.int16))
    d.m = 32
    need = C.c_size_t(0)
    abi.check(abi.load_library().ascq_matmul_w4a16_workspace_size(C.byref(d), C.byref(need)))
    ops.matmul_w4a16(y, xd, wd, sd, od, gs, workspace=torch.zeros(max(need.value // 4, 4), dtype=torch.float32, device=DEV))
    w4_check(y.cpu().numpy(), want, x)


# calls whose weights would be packed or turned round first, in a workspace that holds the passes' pieces (128 MiB) and not the weights
SMALL_WORKSPACE = [("w4a16", 33, 8960, 32576), ("w4a16", 97, 3328, 80672), ("w8a16", 48, 8704, 15584), ("w8a16", 136, 8576, 15680)]


def passes_workspace(kind, m, k, n):
    """(bytes that the passes need, bytes that the call asks for)"""
    lib, need = abi.load_library(), []
    for rows in (4, m):                  # (4 rows run in passes)
        size = C.c_size_t(0)
        if kind == "w4a16":
            abi.check(lib.ascq_matmul_w4a16_workspace_size(C.byref(abi.W4A16Desc(m=rows, n=n, k=k, group_size=128, has_offset=1)), C.byref(size)))
        else:
            abi.check(lib.ascq_matmul_w8a16_workspace_size(C.byref(abi.W8A16Desc(m=rows, n=n, k=k, has_offset=1, out_dtype=abi.F16)), C.byref(size)))
        need.append(size.value)
    return need


@pytest.mark.parametrize("kind,m,k,n", SMALL_WORKSPACE)
def test_half_matmul_in_a_workspace_too_small_for_the_weights(kind, m, k, n):
    """Weights that are brought into another form first and, where the workspace has no room for that, passes over them as they are:
    whole numbers (exact halves, exact fp32 sums), so both give the value itself."""
    announce("small workspace", kind, m, k, n)
    g = torch.Generator(device=DEV)
    g.manual_seed(m + k)
    x = torch.randint(-4, 5, (m, k), device=DEV, generator=g).to(torch.float16)
    w = torch.randint(-8, 8, (k, n), dtype=torch.int8, device=DEV, generator=g)
    of = torch.randint(-3, 4, (n,), device=DEV, generator=g).to(torch.float16)
    sc = torch.randint(1, 3, (n,), device=DEV, generator=g).to(torch.float16) * 0.5
    want = torch.cat([x.double() @ ((w[:, c:c + 8192].double() + of[c:c + 8192].double()) * sc[c:c + 8192].double()) for c in range(0, n, 8192)], 1)
    small, whole = passes_workspace(kind, m, k, n)
    assert small < whole                 # sums of at most 2^23 halves: exact in fp32
    for room in (whole, small):
        y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
        ws = torch.empty(room // 4, dtype=torch.float32, device=DEV)
        if kind == "w4a16":
            nibbles = (w & 15).to(torch.uint8).view(k, n // 2, 2)
            ops.matmul_w4a16(y, x, (nibbles[..., 0] | (nibbles[..., 1] << 4)).contiguous(), sc.expand(k // 128, n).contiguous(),
                             of.expand(k // 128, n).contiguous(), 128, workspace=ws)
        else:
            ops.matmul_w8a16(y, x, w, of, sc, workspace=ws)
        assert torch.equal(y, want.clamp(-65504, 65504).half()), room


def config4_columns(m, n):
    """The oracle covers every column at M=1 (about 6 s on 16 threads); for more rows three slabs: the first and the last
    512 columns (the kernels' first and last column blocks) and one from the middle."""
    return [(0, n)] if m == 1 else [(0, 512), (n // 2 - 256, n // 2 + 256), (n - 512, n)]


def config4_check(got, x, wp, sc, of, d, cols):
    orc.set_threads(16)
    for c0, c1 in cols:
        want = orc.matmul_w4a16(d, x, wp, sc, of, cols=(c0, c1))[:, c0:c1]
        g = got[:, c0:c1]
        err = np.abs(g.astype(np.float64) - want.astype(np.float64))
        tol = 1e-3 * np.maximum(np.abs(want.astype(np.float64)), 1.0)          # fp32 epilogue rel-err <= 1e-3
        assert np.all(err <= tol + 2e-3)
        assert np.mean(g.view(np.uint16) == want.view(np.uint16)) > 0.99


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("m", [1, 4, 16])
def test_config4_w4a16_decode(m, packed):
    """fp16 [M,8192] x int4 [8192,28672], group 128, fp16 scale and offset; both weight layouts."""
    announce("config 4", m, "packed" if packed else "nd")
    rng = np.random.default_rng(0xC4 + m)
    k, n, gs = 8192, 28672, 128
    x, wp, sc, of = w4_case(rng, m, k, n, gs, True)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    if packed:
        ops.matmul_w4a16_packed(y, to_dev(x), ops.pack_weight_w4(to_dev(wp), k, n), to_dev(sc), to_dev(of), gs)
    else:
        ops.matmul_w4a16(y, to_dev(x), to_dev(wp), to_dev(sc), to_dev(of), gs)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=1)
    config4_check(y.cpu().numpy(), x, wp, sc, of, d, config4_columns(m, n))


def w4_group_sum_gate(got, want):
    """The bar of a half output whose accumulation order is free, against the oracle's per-weight arithmetic: every
    element within one bfloat16 ulp of the expected value - where the expected value is small against its row (a
    cancellation), one bfloat16 ulp of the row's root mean square - and the error of a row as a whole within 1e-3 of the
    row.  No share of bit-identical elements is asked for: the group-sum form leaves out the per-weight roundings."""
    g, w = got.astype(np.float64), want.astype(np.float64)
    rms = np.sqrt(np.mean(w * w, axis=1, keepdims=True))
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(w), rms) + 1e-300)) - 7)
    assert np.all(np.abs(g - w) <= ulp)
    assert np.all(np.linalg.norm(g - w, axis=1) <= 1e-3 * np.linalg.norm(w, axis=1))


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 9, 16, 17, 33])
@pytest.mark.parametrize("k,n,gs", [(512, 1024, 128), (1024, 544, 64), (384, 512, 128), (2048, 272, 256), (2048, 64, 512),
                                     (128, 4112, 128), (3200, 144, 128)])
@pytest.mark.parametrize("offset", ["int", "frac", None])
def test_w4a16_packed_group_sum_small(m, k, n, gs, offset):
    """ASCQ_W4A16_GROUP_SUM: scale and offset applied once per quantisation group to fp32 sums.  Same oracle (the
    per-weight arithmetic), the tolerance of a half output; a group size that is no multiple of 128 runs the per-weight
    form and must pass the same gate.  Two calls give identical bits."""
    announce("w4a16 packed group sum", m, k, n, gs, offset)
    rng = np.random.default_rng(m * 7 + k + n)
    x, wp, sc, of = w4_case(rng, m, k, n, gs, offset is not None)
    if offset == "frac":
        of = (rng.standard_normal((k // gs, n)) * 3).astype(np.float16)
    w_gpu = ops.pack_weight_w4(to_dev(wp), k, n)
    xs, scs, ofs = to_dev(x), to_dev(sc), None if of is None else to_dev(of)
    y1 = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    y2 = torch.full((m, n), 7.0, dtype=torch.float16, device=DEV)
    ops.matmul_w4a16_packed(y1, xs, w_gpu, scs, ofs, gs, mode=abi.W4A16_GROUP_SUM)
    ops.matmul_w4a16_packed(y2, xs, w_gpu, scs, ofs, gs, mode=abi.W4A16_GROUP_SUM)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=int(of is not None))
    w4_group_sum_gate(y1.cpu().numpy(), orc.matmul_w4a16(d, x, wp, sc, of))
    assert torch.equal(y1, y2)


def test_w4a16_packed_group_sum_is_the_real_number_value():
    """What the group-sum form computes, pinned without the oracle: on inputs whose products and sums are exact in
    fp32 (integer activations, power-of-two scales, integer offsets) it must give the exact value of
    sum_g scale_g (sum_k x_k w_k + offset_g sum_k x_k), computed here in Python integers."""
    m, k, n, gs = 3, 1024, 96, 128
    announce("w4a16 packed group sum exact", m, k, n)
    rng = np.random.default_rng(77)
    x = rng.integers(-4, 5, (m, k)).astype(np.float16)
    w = rng.integers(-8, 8, (k, n)).astype(np.int8)
    sc = (2.0 ** rng.integers(-6, -2, (k // gs, n))).astype(np.float16)
    of = rng.integers(-8, 8, (k // gs, n)).astype(np.float16)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.matmul_w4a16_packed(y, to_dev(x), ops.pack_weight_w4(to_dev(pack_int4(w)), k, n), to_dev(sc), to_dev(of), gs,
                            mode=abi.W4A16_GROUP_SUM)
    xg = x.astype(np.int64).reshape(m, k // gs, gs)
    wg = w.astype(np.int64).reshape(k // gs, gs, n)
    dots = np.einsum("mgk,gkn->mgn", xg, wg) + xg.sum(axis=2)[:, :, None] * of.astype(np.int64)[None]
    want = (dots.astype(np.float64) * sc.astype(np.float64)[None]).sum(axis=1)      # exact: multiples of 2^-6 below 2^24
    assert np.array_equal(y.cpu().numpy(), want.astype(np.float16))


@pytest.mark.parametrize("offset", ["int", "frac"])
@pytest.mark.parametrize("m", [1, 4, 16])
def test_config4_w4a16_decode_group_sum(m, offset):
    """Config 4 in the group-sum form: every column at M=1, three slabs of 512 columns at M=4 / 16, integer and
    fractional offsets, against the unchanged oracle."""
    announce("config 4 group sum", m, offset)
    rng = np.random.default_rng(0xC4 + m)
    k, n, gs = 8192, 28672, 128
    x, wp, sc, of = w4_case(rng, m, k, n, gs, True)
    if offset == "frac":
        of = (rng.standard_normal((k // gs, n)) * 3).astype(np.float16)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.matmul_w4a16_packed(y, to_dev(x), ops.pack_weight_w4(to_dev(wp), k, n), to_dev(sc), to_dev(of), gs,
                            mode=abi.W4A16_GROUP_SUM)
    d = abi.W4A16Desc(m=m, n=n, k=k, group_size=gs, has_offset=1)
    got = y.cpu().numpy()
    orc.set_threads(16)
    for c0, c1 in config4_columns(m, n):
        want = orc.matmul_w4a16(d, x, wp, sc, of, cols=(c0, c1))[:, c0:c1]
        w4_group_sum_gate(got[:, c0:c1], want)


# ------------------------------------------------------------------ W8A16 (Matmul anti-quant path)
def w8a16_check(got, want, x, out_f32):
    # fp32 accumulation in a different order than the oracle's wide one: error bounded relative to sum |x| |w| (w up
    # to 137 * 1e-2 in these cases), and bit-identical halves nearly everywhere
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    ref = np.abs(x.astype(np.float64)).sum(axis=1, keepdims=True) * 1.4
    assert np.all(err <= 1e-5 * ref + 1e-6) if out_f32 else np.all(err <= 1e-3 * ref + 1e-6)
    if not out_f32:
        assert np.mean(got.view(np.uint16) == want.view(np.uint16)) > 0.9


@pytest.mark.parametrize("m", [1, 3, 16, 17, 32, 33, 40, 70, 97, 300])   # above 96 rows: transposed copy + tile GEMM
@pytest.mark.parametrize("k,n", [(256, 256), (512, 1040), (96, 48), (100, 30), (2048, 512), (192, 30)])
@pytest.mark.parametrize("mode", ["vector+offset", "vector", "scalar+offset", "scalar", "vector+intoffset"])
def test_w8a16_small(m, k, n, mode):
    announce("w8a16", m, k, n, mode)
    rng = np.random.default_rng(m * 7 + k + n)
    x = rng.standard_normal((m, k)).astype(np.float16)
    w = rng.integers(-128, 128, (k, n)).astype(np.int8)
    per_tensor = mode.startswith("scalar")
    has_offset = "offset" in mode
    out_f32 = (m + k) % 2 == 1
    if per_tensor:
        sc, of = 0.0077, (2.5 if has_offset else None)
    else:
        sc = rng.uniform(1e-3, 1e-2, n).astype(np.float16)
        of = None
        if has_offset:
            of = (rng.integers(-9, 10, n) if "int" in mode else rng.uniform(-9, 9, n)).astype(np.float16)
    y = torch.zeros((m, n), dtype=torch.float32 if out_f32 else torch.float16, device=DEV)
    ops.matmul_w8a16(y, to_dev(x), to_dev(w), of if per_tensor else (None if of is None else to_dev(of)),
                     sc if per_tensor else to_dev(sc))
    d = abi.W8A16Desc(m=m, n=n, k=k, per_tensor=int(per_tensor), has_offset=int(has_offset),
                      scale=sc if per_tensor else 0.0, offset=of if per_tensor and has_offset else 0.0,
                      out_dtype=abi.F32 if out_f32 else abi.F16)
    want = orc.matmul_w8a16(d, x, w, None if per_tensor else of, None if per_tensor else sc)
    w8a16_check(y.cpu().numpy(), want, x, out_f32)


@pytest.mark.parametrize("m", [1, 16])
def test_w8a16_decode_shape(m):
    """fp16 [M,4096] x int8 [4096,11008], per-channel scale and offset (the W8A8 headline weight shape)."""
    announce("w8a16 decode", m)
    rng = np.random.default_rng(0xA16 + m)
    k, n = 4096, 11008
    x = rng.standard_normal((m, k)).astype(np.float16)
    w = rng.integers(-128, 128, (k, n)).astype(np.int8)
    sc = rng.uniform(1e-3, 1e-2, n).astype(np.float16)
    of = rng.uniform(-9, 9, n).astype(np.float16)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.matmul_w8a16(y, to_dev(x), to_dev(w), to_dev(of), to_dev(sc))
    d = abi.W8A16Desc(m=m, n=n, k=k, per_tensor=0, has_offset=1, out_dtype=abi.F16)
    orc.set_threads(16)
    want = orc.matmul_w8a16(d, x, w, of, sc)
    w8a16_check(y.cpu().numpy(), want, x, False)


@pytest.mark.parametrize("m", [1, 4])
@pytest.mark.parametrize("mode", [abi.W8A16_PER_WEIGHT, abi.W8A16_CHANNEL_SUM])
def test_w8a16_decode_shape_weights_as_n_k(m, mode):
    """fp16 [M, 8192] x int8 [28672, 8192] kept as [n, k] (the benchmark's decode shape), per-channel scale and offset,
    on the stream kernel with the activations resident in LDS: the per-weight mode within the usual tolerance of a free
    accumulation order, the channel-sum mode within one bfloat16 ulp per element and 1e-3 per row."""
    announce("w8a16 decode [n, k]", m, mode)
    rng = np.random.default_rng(0xB16 + m)
    k, n = 8192, 28672
    x = rng.standard_normal((m, k)).astype(np.float16)
    wt = rng.integers(-128, 128, (n, k)).astype(np.int8)
    sc = rng.uniform(1e-3, 1e-2, n).astype(np.float16)
    of = rng.uniform(-9, 9, n).astype(np.float16)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.matmul_w8a16(y, to_dev(x), to_dev(wt), to_dev(of), to_dev(sc), workspace=torch.empty(4, device=DEV), trans_b=True,
                     mode=mode)
    d = abi.W8A16Desc(m=m, n=n, k=k, per_tensor=0, has_offset=1, out_dtype=abi.F16, trans_b=1)
    orc.set_threads(16)
    want = orc.matmul_w8a16(d, x, wt, of, sc)
    if mode == abi.W8A16_PER_WEIGHT:
        w8a16_check(y.cpu().numpy(), want, x, False)
    else:
        w4_group_sum_gate(y.cpu().numpy(), np.asarray(want))


@pytest.mark.parametrize("m", [2, 16])
def test_w8a16_exact_integers_full_size(m):
    """Small integer activations, power-of-two scales and integer offsets make every product and partial sum exact in
    fp32, so the result is independent of the accumulation order: bit-equal to plain integer arithmetic at full size."""
    announce("w8a16 exact", m)
    rng = np.random.default_rng(0xE8 + m)
    k, n = 4096, 11008
    xi = rng.integers(-2, 3, (m, k))
    w = rng.integers(-128, 128, (k, n)).astype(np.int8)
    sc = rng.choice([0.25, 0.5, 1.0], n)
    of = rng.integers(-9, 10, n)
    y = torch.zeros((m, n), dtype=torch.float32, device=DEV)
    ops.matmul_w8a16(y, to_dev(xi.astype(np.float16)), to_dev(w), to_dev(of.astype(np.float16)),
                     to_dev(sc.astype(np.float16)))
    want = (xi.astype(np.float64) @ (w.astype(np.float64) + of[None, :])) * sc[None, :]
    assert np.array_equal(y.cpu().numpy().astype(np.float64), want)

@pytest.mark.parametrize("m", [1, 3, 16, 17, 40, 49, 130, 300])
@pytest.mark.parametrize("k,n", [(128, 16), (256, 256), (512, 1040), (384, 30), (2048, 520), (8192, 144), (192, 40),
                                 (77, 23)])
@pytest.mark.parametrize("mode", ["vector+offset", "vector", "scalar+offset", "scalar"])
def test_w8a16_trans_b(m, k, n, mode):
    """B given as [n, k] (isTransposeB): one launch, no workspace; the whole-column kernel up to 48 rows, the
    de-quantising tile GEMM above, one lane per output element when k is no multiple of 128.  Against the oracle on
    the same transposed weights, and bit-equal between two calls (the summation order is fixed)."""
    announce("w8a16 [n, k]", m, k, n, mode)
    rng = np.random.default_rng(m * 5 + k + n)
    x = rng.standard_normal((m, k)).astype(np.float16)
    wt = rng.integers(-128, 128, (n, k)).astype(np.int8)
    per_tensor = mode.startswith("scalar")
    has_offset = "offset" in mode
    out_f32 = (m + k // 128) % 2 == 1
    if per_tensor:
        sc, of = 0.0077, (2.5 if has_offset else None)
    else:
        sc = rng.uniform(1e-3, 1e-2, n).astype(np.float16)
        of = rng.uniform(-9, 9, n).astype(np.float16) if has_offset else None
    ys = []
    for _ in range(2):
        y = torch.zeros((m, n), dtype=torch.float32 if out_f32 else torch.float16, device=DEV)
        y.view(torch.int16).fill_(0x7E7E)
        ops.matmul_w8a16(y, to_dev(x), to_dev(wt), of if per_tensor else (None if of is None else to_dev(of)),
                         sc if per_tensor else to_dev(sc), workspace=torch.empty(4, device=DEV), trans_b=True)
        ys.append(y.cpu().numpy())
    assert np.array_equal(ys[0].view(np.uint16), ys[1].view(np.uint16))
    d = abi.W8A16Desc(m=m, n=n, k=k, per_tensor=int(per_tensor), has_offset=int(has_offset),
                      scale=sc if per_tensor else 0.0, offset=of if per_tensor and has_offset else 0.0,
                      out_dtype=abi.F32 if out_f32 else abi.F16, trans_b=1)
    want = orc.matmul_w8a16(d, x, wt, None if per_tensor else of, None if per_tensor else sc)
    w8a16_check(ys[0], want, x, out_f32)
    # the oracle's own transposed indexing: the same answer from the [k, n] form
    d.trans_b = 0
    assert np.array_equal(np.asarray(want).view(np.uint8),
                          np.asarray(orc.matmul_w8a16(d, x, np.ascontiguousarray(wt.T), None if per_tensor else of,
                                                      None if per_tensor else sc)).view(np.uint8))


W8_WHOLE_K = {(16, 16): [(14, 8448, 1379)], (32, 16): [(28, 2176, 2573), (20, 768, 11)], (32, 32): [(30, 1920, 5317)],
              (64, 16): [(70, 3072, 1551), (22, 128, 51)], (64, 32): [(100, 1152, 2055), (40, 2048, 5000)], (64, 64): [(300, 1152, 2059), (85, 1152, 6913)],
              (): [(9, 8448, 1280), (5, 128, 3), (16, 1664, 23264)]}  # passes of 16 rows


@pytest.mark.parametrize("m,k,n", [s for sizes in W8_WHOLE_K.values() for s in sizes])
@pytest.mark.parametrize("mode", ["vector+offset", "scalar"])
@pytest.mark.parametrize("out_f32", [True, False])
def test_w8a16_trans_b_whole_k_tiles(m, k, n, mode, out_f32):
    """Rows and columns that leave the large tiles' chip idle: every tile of 16 x 16 to 64 x 64, row and column tails (odd widths), k
    that the eight wavefronts cannot share evenly or at all; the last three stay with the passes of 16 rows."""
    announce("w8a16 [n, k] whole-k tiles", m, k, n, mode, out_f32)
    rng = np.random.default_rng(m * 7 + k + n)
    x = rng.standard_normal((m, k)).astype(np.float16)
    wt = rng.integers(-128, 128, (n, k)).astype(np.int8)
    per_tensor, has_offset = mode == "scalar", mode.endswith("offset")
    sc, of = (0.0077, None) if per_tensor else (rng.uniform(1e-3, 1e-2, n).astype(np.float16), rng.uniform(-9, 9, n).astype(np.float16))
    y = torch.full((m + 1, n), 7.0, dtype=torch.float32 if out_f32 else torch.float16, device=DEV)
    ops.matmul_w8a16(y[:m], to_dev(x), to_dev(wt), of if per_tensor else to_dev(of), sc if per_tensor else to_dev(sc), trans_b=True)
    assert bool((y[m] == 7.0).all())
    d = abi.W8A16Desc(m=m, n=n, k=k, per_tensor=int(per_tensor), has_offset=int(has_offset), scale=sc if per_tensor else 0.0, offset=0.0,
                      out_dtype=abi.F32 if out_f32 else abi.F16, trans_b=1)
    orc.set_threads(16)
    w8a16_check(y[:m].cpu().numpy(), orc.matmul_w8a16(d, x, wt, None if per_tensor else of, None if per_tensor else sc), x, out_f32)


def test_w8a16_rows_beyond_thirty_two_bit_offsets():
    """128 rows of x of 32.5 MiB each: the last rows of a tile of 128 lie more than 4 GiB behind its first, where a lane's
    32-bit offset would wrap round to another row.  x is zero but for a few halves, so every result is an exact integer."""
    m, n, k = 128, 16, (1 << 24) + (1 << 18)
    announce("w8a16 long rows", m, n, k)
    g = torch.Generator(device=DEV)
    g.manual_seed(1)
    x = torch.zeros((m, k), dtype=torch.float16, device=DEV)
    w = torch.randint(-8, 9, (n, k), dtype=torch.int8, device=DEV, generator=g)
    want = torch.zeros((m, n), dtype=torch.float32, device=DEV)
    for row, col in ((0, 0), (3, 64), (64, 5), (124, 70), (125, 3), (126, k - 1), (127, 0), (127, 9)):
        x[row, col] = row % 7 + 1
        want[row] += (row % 7 + 1) * w[:, col].float()
    y = torch.full((m, n), -1.0, dtype=torch.float32, device=DEV)
    ops.matmul_w8a16(y, x, w, None, 1.0, trans_b=True)
    assert torch.equal(y, want)


@pytest.mark.parametrize("m,k,n", [(17, 1280, 1040), (24, 1408, 36), (33, 2304, 1152), (65, 1024, 2688), (96, 128, 7)])
@pytest.mark.parametrize("offset", [True, False])
def test_w8a16_few_rows_transposed_first(m, k, n, offset):
    """[k, n] weights that are transposed into the workspace first: the value in 64 bits, and the call on [n, k] weights; columns
    that are no multiple of 16 among them."""
    announce("w8a16 few rows on [k, n]", m, k, n, offset)
    g = torch.Generator(device=DEV)
    g.manual_seed(m + k + n)
    x = torch.randn((m, k), device=DEV, generator=g).half()
    w = torch.randint(-128, 128, (k, n), device=DEV, dtype=torch.int8, generator=g)
    sc = (torch.rand(n, device=DEV, generator=g) * 0.01 + 0.001).half()
    of = (torch.rand(n, device=DEV, generator=g) * 16 - 8).half() if offset else None
    y0, y1 = torch.zeros((m, n), dtype=torch.float16, device=DEV), torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.matmul_w8a16(y0, x, w, of, sc)
    ops.matmul_w8a16(y1, x, w.t().contiguous(), of, sc, trans_b=True)
    wf = w.half() + of if offset else w.half()
    want = x.double().cpu() @ (wf * sc).double().cpu()
    # two roundings of a result in half, fp32 sums: 2^-11 of the value and 1e-6 of the sum of magnitudes
    room = 2.0 ** -11 * want.abs() + 1e-6 * (x.double().abs().cpu() @ (wf * sc).double().abs().cpu()) + 1e-7
    assert ((y0.double().cpu() - want).abs() <= room).all()
    assert torch.allclose(y0.float(), y1.float(), rtol=2.0 ** -10, atol=1e-3)


W8_MANY_ROWS = {"wq_rows_kernel": [(33, 128, 7), (128, 256, 248), (129, 384, 264), (257, 640, 521)],
                "wq_gemm_kernel<128, 128, ": [(300, 128, 1034), (69, 128, 2307), (700, 384, 3001), (640, 640, 3080), (1030, 640, 2056)]}


@pytest.mark.parametrize("m,k,n", [s for sizes in W8_MANY_ROWS.values() for s in sizes])
@pytest.mark.parametrize("mode", ["vector+offset", "vector", "scalar+offset"])
@pytest.mark.parametrize("out_f32", [False, True])
def test_w8a16_trans_b_many_rows(m, k, n, mode, out_f32):
    """The half GEMM whose B-tile loader de-quantises [n, k] weights, on tiles of 128 x 128: two steps of k and more, row and
    column tails, column counts that are no multiple of 4 (stored element by element) and of 2; few rows or columns run whole-k tiles."""
    announce("w8a16 [n, k] many rows", m, k, n, mode, out_f32)
    rng = np.random.default_rng(m + k + n)
    x = rng.standard_normal((m, k)).astype(np.float16)
    wt = rng.integers(-128, 128, (n, k)).astype(np.int8)
    per_tensor, has_offset = mode.startswith("scalar"), "offset" in mode
    sc = 0.0077 if per_tensor else rng.uniform(1e-3, 1e-2, n).astype(np.float16)
    of = None if not has_offset else 2.5 if per_tensor else rng.uniform(-9, 9, n).astype(np.float16)
    y = torch.full((m, n), 7.0, dtype=torch.float32 if out_f32 else torch.float16, device=DEV)
    ops.matmul_w8a16(y, to_dev(x), to_dev(wt), of if per_tensor or of is None else to_dev(of), sc if per_tensor else to_dev(sc),
                     workspace=torch.empty(4, device=DEV), trans_b=True)
    d = abi.W8A16Desc(m=m, n=n, k=k, per_tensor=int(per_tensor), has_offset=int(has_offset), scale=sc if per_tensor else 0.0,
                      offset=of if per_tensor and has_offset else 0.0, out_dtype=abi.F32 if out_f32 else abi.F16, trans_b=1)
    orc.set_threads(16)
    want = orc.matmul_w8a16(d, x, wt, None if per_tensor else of, None if per_tensor else sc)
    w8a16_check(y.cpu().numpy(), want, x, out_f32)


@pytest.mark.parametrize("m,n", [(300, 24600), (384, 20480), (1300, 14600)])
@pytest.mark.parametrize("kind,k", [("int8", k) for k in (64, 128, 192, 256, 320, 448)] + [("int4", k) for k in (128, 256, 384, 512)])
@pytest.mark.parametrize("offset", [True, False])
def test_half_gemm_on_tiles_of_256_columns(m, n, kind, k, offset):
    """The half GEMM's tiles of 256 columns, whose loads go out in halves behind two counted waits a step: 256 x 256, 128 x 256, and
    256 x 256 with the tiles beyond a whole round cut in half; one to eight K steps of 64 (prologue, steady state, the last step but one
    and the last); row and column tails.  Whole numbers: the de-quantised weights are exact halves and every sum an exact float, so
    the order of the sums does not matter and every element is compared, float and half outputs."""
    announce("half GEMM, 256 columns", m, n, kind, k, offset)
    g = torch.Generator(device=DEV)
    g.manual_seed(m + k)
    x = torch.randint(-4, 5, (m, k), device=DEV, generator=g).to(torch.float16)
    lo, hi = (-8, 7) if kind == "int4" else (-100, 100)
    w = torch.randint(lo, hi + 1, (k, n), dtype=torch.int8, device=DEV, generator=g)
    of = torch.randint(-3, 4, (n,), device=DEV, generator=g).to(torch.float16)
    sc = torch.randint(1, 3, (n,), device=DEV, generator=g).to(torch.float16) * 0.5
    # at most 512 * 4 * 103 in magnitude, in halves: exact in fp32
    want = (x.double() @ ((w.double() + (of.double() if offset else 0.0)) * sc.double())).float()
    outs = (torch.float16,) if kind == "int4" else (torch.float16, torch.float32)
    for out in outs:
        y = torch.full((m, n), 7.0, dtype=out, device=DEV)
        if kind == "int4":
            nibbles = (w & 15).to(torch.uint8).view(k, n // 2, 2)
            packed = ops.pack_weight_w4((nibbles[..., 0] | (nibbles[..., 1] << 4)).contiguous(), k, n)
            groups = k // 128
            ops.matmul_w4a16_packed(y, x, packed, sc.expand(groups, n).contiguous(), of.expand(groups, n).contiguous() if offset else None, 128)
        elif k % 128 == 0:
            ops.matmul_w8a16(y, x, w.t().contiguous(), of if offset else None, sc, trans_b=True)
        else:                        # ([n, k] weights take steps of 128; [k, n] ones are turned round and run the same tiles)
            ops.matmul_w8a16(y, x, w, of if offset else None, sc)
        assert torch.equal(y, want.clamp(-65504, 65504).to(out) if out == torch.float16 else want)


# m, n, kind, k: whether all loads of a step go out at once
LOAD_RULE = {False: [(200, 8440, "int8", 3648), (200, 8440, "int8", 3712), (200, 8440, "int8", 3776), (200, 8440, "int4", 3712)],
             True: [(200, 8440, "int8", 3840), (200, 8440, "int8", 3904), (200, 8440, "int8", 3968), (200, 8440, "int4", 3840)],
             None: [(100, 14600, "int8", k) for k in (4224, 4352, 4416, 4480)] + [(100, 14600, "int4", k) for k in (4224, 4352, 4480)]}


@pytest.mark.parametrize("m,n,kind,k", [s for sizes in LOAD_RULE.values() for s in sizes])
@pytest.mark.parametrize("offset", [True, False])
def test_half_gemm_on_both_sides_of_the_load_rule(m, n, kind, k, offset):
    """132 tiles of 128 x 128: below 3788 of k each load of a step goes out behind a matrix instruction, from there on all at once; even
    and odd numbers of K steps, exact sums as above.  (100 rows run whole-k tiles of 64 x 64.)"""
    test_half_gemm_on_tiles_of_256_columns(m, n, kind, k, offset)


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("k,n", [(128, 16), (256, 256), (512, 1040), (384, 30), (2048, 520), (8192, 144)])
@pytest.mark.parametrize("mode", ["vector+offset", "vector", "scalar+offset", "scalar"])
def test_w8a16_trans_b_channel_sum(m, k, n, mode):
    """ASCQ_W8A16_CHANNEL_SUM on [n, k] weights: scale and offset applied once per output to fp32 sums.  Same oracle
    (the per-weight arithmetic), the tolerance of a half output: every element within one bfloat16 ulp, the row error
    within 1e-3; 5 rows run the per-weight kernel and pass the same gate.  Two calls give identical bits."""
    announce("w8a16 [n, k] channel sum", m, k, n, mode)
    rng = np.random.default_rng(m * 11 + k + n)
    x = rng.standard_normal((m, k)).astype(np.float16)
    wt = rng.integers(-128, 128, (n, k)).astype(np.int8)
    per_tensor = mode.startswith("scalar")
    has_offset = "offset" in mode
    if per_tensor:
        sc, of = 0.0077, (2.5 if has_offset else None)
    else:
        sc = rng.uniform(1e-3, 1e-2, n).astype(np.float16)
        of = rng.uniform(-9, 9, n).astype(np.float16) if has_offset else None
    ys = []
    for _ in range(2):
        y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
        y.view(torch.int16).fill_(0x7E7E)
        ops.matmul_w8a16(y, to_dev(x), to_dev(wt), of if per_tensor else (None if of is None else to_dev(of)),
                         sc if per_tensor else to_dev(sc), workspace=torch.empty(4, device=DEV), trans_b=True,
                         mode=abi.W8A16_CHANNEL_SUM)
        ys.append(y.cpu().numpy())
    assert np.array_equal(ys[0].view(np.uint16), ys[1].view(np.uint16))
    d = abi.W8A16Desc(m=m, n=n, k=k, per_tensor=int(per_tensor), has_offset=int(has_offset),
                      scale=sc if per_tensor else 0.0, offset=of if per_tensor and has_offset else 0.0,
                      out_dtype=abi.F16, trans_b=1)
    want = orc.matmul_w8a16(d, x, wt, None if per_tensor else of, None if per_tensor else sc)
    w4_group_sum_gate(ys[0], np.asarray(want))


def test_w8a16_channel_sum_is_the_real_number_value():
    """The channel-sum form rounds the exact value of the quantised product once; the per-weight form carries two
    roundings per weight.  Against float64 arithmetic on the same quantised inputs the channel-sum result is at least
    as close, on average, as the per-weight one."""
    announce("w8a16 channel sum against float64")
    rng = np.random.default_rng(91)
    m, k, n = 4, 4096, 1024
    x = rng.standard_normal((m, k)).astype(np.float16)
    wt = rng.integers(-128, 128, (n, k)).astype(np.int8)
    sc = rng.uniform(1e-3, 1e-2, n).astype(np.float16)
    of = rng.uniform(-9, 9, n).astype(np.float16)
    exact = (x.astype(np.float64) @ (wt.astype(np.float64).T + of.astype(np.float64)[None, :])) * sc.astype(np.float64)[None, :]
    errs = []
    for mode in (abi.W8A16_PER_WEIGHT, abi.W8A16_CHANNEL_SUM):
        y = torch.zeros((m, n), dtype=torch.float32, device=DEV)
        ops.matmul_w8a16(y, to_dev(x), to_dev(wt), to_dev(of), to_dev(sc), workspace=torch.empty(4, device=DEV), trans_b=True,
                         mode=mode)
        errs.append(np.abs(y.cpu().numpy().astype(np.float64) - exact).mean())
    assert errs[1] <= errs[0]
    assert errs[1] <= 1e-5 * np.abs(exact).mean()


@pytest.mark.parametrize("m", [1, 16])
def test_w8a16_trans_b_exact_integers_full_size(m):
    """K=8192, N=28672 as [n, k]: small integer activations, power-of-two scales and integer offsets make every partial
    sum exact in fp32, so the result must equal plain integer arithmetic bit for bit on every column."""
    announce("w8a16 [n, k] exact", m)
    rng = np.random.default_rng(0xE9 + m)
    k, n = 8192, 28672
    xi = rng.integers(-2, 3, (m, k))
    wt = rng.integers(-128, 128, (n, k)).astype(np.int8)
    sc = rng.choice([0.25, 0.5, 1.0], n)
    of = rng.integers(-9, 10, n)
    y = torch.zeros((m, n), dtype=torch.float32, device=DEV)
    ops.matmul_w8a16(y, to_dev(xi.astype(np.float16)), to_dev(wt), to_dev(of.astype(np.float16)),
                     to_dev(sc.astype(np.float16)), trans_b=True)
    want = ((wt.astype(np.float32) + of[:, None].astype(np.float32)) @ xi.T.astype(np.float32)).T * sc[None, :]
    assert np.array_equal(y.cpu().numpy().astype(np.float64), want.astype(np.float64))


# ------------------------------------------------------------------ fractal (NZ) weights
def to_nz(w):
    """[.., k, n] -> [.., n/32, k/16, 16, 32], as the reference example packs its weights
    (quant_group_matmul_high_performance/scripts/gen_data.py:62-65)."""
    *lead, k, n = w.shape
    nd = len(lead)
    perm = list(range(nd)) + [nd + 2, nd + 0, nd + 1, nd + 3]
    return np.ascontiguousarray(w.reshape(*lead, k // 16, 16, n // 32, 32).transpose(perm))


@pytest.mark.parametrize("m,n,k", [(1, 64, 128), (48, 160, 256), (200, 544, 384), (513, 288, 128), (2048, 2848, 256)])
@pytest.mark.parametrize("out", [torch.int32, torch.bfloat16])
def test_matmul_nz_weights(m, n, k, out):
    """The same product from fractal weights: bit-equal to the oracle on the row-major weights."""
    announce("nz weights", m, n, k, out)
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    w = rng.integers(-127, 128, (k, n)).astype(np.int8)
    c = torch.zeros((m, n), dtype=out, device=DEV)
    mm = ops.Matmul(m, n, k)
    mm.set_tensor_a(to_dev(a))
    mm.set_tensor_b(to_dev(to_nz(w)), nz=True)
    d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.I32)
    cs = ts = None
    if out != torch.int32:
        cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
        ts = rng.uniform(1e-3, 1e-1, m).astype(np.float32)
        mm.set_quant_vector(to_dev(cs))
        mm.set_token_scale(to_dev(ts))
        d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR,
                           scale_format=abi.MM_SCALE_F32, has_tok_scale=1)
    mm.iterate_all(c)
    orc.set_threads(16)
    want = orc.matmul_w8a8(d, a, w, None, cs, ts)
    assert np.array_equal(bits(c), want)


@pytest.mark.parametrize("m", [9, 200, 513, 729])
@pytest.mark.parametrize("k,n", [(16, 256), (112, 264), (144, 1152), (1040, 280), (4304, 1160)])
def test_w8a8_ragged_sizes_on_the_tile_kernels(m, k, n):
    """The direct-to-LDS tiles with a last, partial K step and with columns that are no multiple of 16 (the last tile of
    [k, n] weights moves left), K split or not, in all weight layouts; SwiGLU; a grouped matmul of the same sizes.
    Integer sums are exact, the de-quantised outputs have the oracle's bits."""
    announce("w8a8 ragged tiles", m, k, n)
    rng = np.random.default_rng(m + 3 * k + n)
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.int64)
    bt = np.ascontiguousarray(b.T)
    for trans in (False, True):
        c, _ = run_mm(m, n, k, a, bt if trans else b, out=torch.int32, trans_b=trans)
        assert np.array_equal(c.cpu().numpy(), want)
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(DEV).to(torch.bfloat16)
    q, ts = orc.dynamic_quant_per_token(abi.BF16, bits(x))
    d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32,
                       has_tok_scale=1, bias_kind=abi.MM_BIAS_F32_POST)
    gold = orc.matmul_w8a8(d, q, b, bias, cs, ts)
    d.activation, d.act_beta = abi.MM_ACT_SWIGLU, 1.0
    gold_swiglu = orc.matmul_w8a8(d, q, b, bias, cs, ts).view(np.uint16)
    for trans in (False, True):
        w = to_dev(bt if trans else b)
        c = torch.zeros((m, n), dtype=torch.bfloat16, device=DEV)
        ops.linear_w8a8_dynamic(c, x, w, to_dev(cs), to_dev(bias), abi.MM_ACT_NONE, trans)
        assert np.array_equal(bits(c), gold)
        cg = torch.zeros((m, n // 2), dtype=torch.bfloat16, device=DEV)
        ops.linear_w8a8_dynamic(cg, x, w, to_dev(cs), to_dev(bias), abi.MM_ACT_SWIGLU, trans)
        swiglu_close(bits(cg), gold_swiglu, "bf16")
    counts = [m // 3, 0, m - m // 3 - 1]
    got, ref = run_group(m, k, n, counts, abi.GROUP_LIST_COUNTS, torch.bfloat16, rng, True, abi.MM_ACT_NONE)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("k", [16, 48, 112, 144])
@pytest.mark.parametrize("m,n,layout", [(33, 1376, "nk"), (300, 640, "nk"), (16, 1376, "nk"), (40, 248, "kn"), (600, 24, "kn"), (17, 136, "kn"), (24, 40, "group")])
def test_staged_kernel_reads_nothing_past_its_operands(m, n, k, layout):
    """The register-staged kernel with a k below, or just above, its K step of 128: both operands end where their allocation
    ends (whole multiples of 2 MiB), so a piece past k must not be fetched from behind the last row."""
    announce("staged, short k", m, n, k, layout)
    def at_the_end(t):
        room = torch.zeros(32 << 20, dtype=torch.int8, device=DEV)
        tail = room[room.numel() - t.numel():].view(t.shape)
        tail.copy_(t)
        return tail
    rng = np.random.default_rng(m + n + k)
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    if a.size % 16 or b.size % 16:
        pytest.skip("the operands would not be 16-byte aligned")
    want = (a.astype(np.int64) @ b.astype(np.int64)).astype(np.int32)
    if layout == "group":
        w = at_the_end(torch.from_numpy(b).view(1, k, n))
        y = torch.zeros((m, n), dtype=torch.float32, device=DEV)
        ops.quant_group_matmul(y, at_the_end(torch.from_numpy(a)), w, torch.tensor([m], dtype=torch.int64, device=DEV), torch.ones((1, n), device=DEV))
        assert np.array_equal(y.cpu().numpy(), want.astype(np.float32))
        return
    mm = ops.Matmul(m, n, k, trans_b=layout == "nk")
    mm.set_tensor_a(at_the_end(torch.from_numpy(a)))
    mm.set_tensor_b(at_the_end(torch.from_numpy(np.ascontiguousarray(b.T) if layout == "nk" else b)))
    c = torch.zeros((m, n), dtype=torch.int32, device=DEV)
    mm.iterate_all(c)
    assert np.array_equal(c.cpu().numpy(), want)


@pytest.mark.parametrize("m", [1, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("k,n", [(128, 65), (132, 257), (1000, 1023), (6784, 515), (512, 2050)])
def test_w8a8_few_rows_on_unaligned_columns(m, k, n):
    """[k, n] weights whose rows start at any byte: int32 sums, and the linear's bits against the oracle."""
    announce("w8a8 unaligned columns", m, k, n)
    rng = np.random.default_rng(m + 5 * k + n)
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    c, _ = run_mm(m, n, k, a, b, out=torch.int32)
    assert np.array_equal(c.cpu().numpy(), a.astype(np.int64) @ b.astype(np.int64))
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(DEV).to(torch.bfloat16)
    c = torch.zeros((m, n), dtype=torch.bfloat16, device=DEV)
    ops.linear_w8a8_dynamic(c, x, to_dev(b), to_dev(cs), to_dev(bias))
    q, ts = orc.dynamic_quant_per_token(abi.BF16, bits(x))
    d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32,
                       has_tok_scale=1, bias_kind=abi.MM_BIAS_F32_POST)
    assert np.array_equal(bits(c), orc.matmul_w8a8(d, q, b, bias, cs, ts))


@pytest.mark.parametrize("m", [129, 300, 480, 600])
@pytest.mark.parametrize("k,n", [(64, 40), (1472, 512), (5888, 520), (4096, 1024), (1024, 2048)])
def test_linear_w8a8_dynamic_packed_split_over_k(m, k, n):
    """Packed weights with too few tiles for the chip: K split over workgroups, the pieces in the call's workspace, or,
    where that costs more than it gives (the last shape, up to 512 rows), the tiles as they are."""
    announce("linear dynamic packed, K split", m, k, n)
    rng = np.random.default_rng(m + k + n)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(DEV).to(torch.float16)
    w = rand_i8(rng, (k, n))
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c = torch.zeros((m, n), dtype=torch.bfloat16, device=DEV)
    ops.linear_w8a8_dynamic_packed(c, x, ops.pack_weight_w8(to_dev(w), k, n), n, to_dev(cs), to_dev(bias))
    q, ts = orc.dynamic_quant_per_token(abi.F16, bits(x))
    d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32,
                       has_tok_scale=1, bias_kind=abi.MM_BIAS_F32_POST)
    assert np.array_equal(bits(c), orc.matmul_w8a8(d, q, w, bias, cs, ts))


@pytest.mark.parametrize("m,k,n", [(33, 16, 264), (65, 144, 520), (130, 400, 1032), (200, 1040, 264), (100, 1152, 1000), (97, 1664, 256), (130, 2192, 272),
                                   (300, 640, 4400), (290, 1136, 4408), (600, 384, 6400), (520, 1744, 6008)])
@pytest.mark.parametrize("act", [abi.MM_ACT_NONE, abi.MM_ACT_FASTER_GELU, abi.MM_ACT_SWIGLU])
def test_linear_w8a8_small_tiles_with_a_ring_of_stages(m, k, n, act):
    """The linears of medium size, all weight layouts: tiles of 64 x 64, 128 x 64 (from 300 x 640 x 4400 on) and 128 x 128
    (from 600 x 384 x 6400 on), one K step to eighteen (fewer and more than the ring has stages, whole groups of them and
    every remainder), a last K step of 16 to 112, rows and columns that end inside a tile, a last [k, n] tile moved left."""
    announce("ring", m, k, n, act)
    rng = np.random.default_rng(m + k + n)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(DEV).to(torch.bfloat16)
    w = rand_i8(rng, (k, n))
    cs = rng.uniform(1e-4, 1e-3, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    q, ts = orc.dynamic_quant_per_token(abi.BF16, bits(x))
    sums = (q.astype(np.float64) @ w.astype(np.float64)).astype(np.int32)      # exact
    v = sums.astype(np.float32) * cs * ts[:, None] + bias                      # one rounding per step, like the epilogue
    forms = [("kn", to_dev(w)), ("nk", to_dev(np.ascontiguousarray(w.T)))]
    if k % 64 == 0:
        forms.append(("packed", ops.pack_weight_w8(to_dev(w), k, n)))
    for out in (torch.bfloat16, torch.float16, torch.float32):
        for layout, wd in forms:
            c = torch.zeros((m, n // 2 if act == abi.MM_ACT_SWIGLU else n), dtype=out, device=DEV)
            if layout == "packed":
                ops.linear_w8a8_dynamic_packed(c, x, wd, n, to_dev(cs), to_dev(bias), act)
            else:
                ops.linear_w8a8_dynamic(c, x, wd, to_dev(cs), to_dev(bias), act, layout == "nk")
            if act == abi.MM_ACT_NONE:
                assert torch.equal(c.cpu(), torch.from_numpy(v).to(out)), layout
                continue
            # the activations' exponentials (of arguments up to 2^5) and quotients are approximations of about one fp32 ulp
            t = v.astype(np.float64)
            want = t / (1.0 + np.exp(-1.702 * t)) if act == abi.MM_ACT_FASTER_GELU else t[:, 0::2] * t[:, 1::2] / (1.0 + np.exp(-t[:, 1::2]))
            ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}[out]
            got = c.double().cpu().numpy()
            assert np.all(np.abs(got - want) <= (ulp + 2.0 ** -18) * np.abs(want) + 1e-6), layout


def ring_tiles(call):
    """The tiles of the ring kernel that `call` launches, by the kernel names that the profiler saw: {(rows, columns)}."""
    import re
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        call()
        torch.cuda.synchronize()
    found = [re.search(r"gemm_ring_kernel(?:ILi(\d+)ELi(\d+)|<(\d+), (\d+))", e.key) for e in prof.key_averages()]
    return {tuple(int(g) for g in f.groups() if g) for f in found if f}


@pytest.mark.parametrize("m,k,n,tile", [(65, 144, 520, (64, 64)), (200, 1040, 264, (64, 64)), (130, 2192, 272, (64, 64)), (300, 640, 4400, (128, 64)),
                                        (290, 1136, 4408, (128, 64)), (600, 384, 6400, (128, 128)), (520, 1744, 6008, (128, 128))])
def test_linears_reach_every_tile_of_the_ring(m, k, n, tile):
    """The sizes of the test above that stand for a tile shape run it, with and without SwiGLU: its comparisons are of that kernel."""
    announce("ring tiles", m, k, n, tile)
    x = torch.zeros((m, k), dtype=torch.bfloat16, device=DEV)
    cs = torch.ones(n, device=DEV)
    for trans_b in (False, True):
        w = torch.zeros((n, k) if trans_b else (k, n), dtype=torch.int8, device=DEV)
        for act in (abi.MM_ACT_NONE, abi.MM_ACT_SWIGLU):
            c = torch.zeros((m, n // 2 if act == abi.MM_ACT_SWIGLU else n), dtype=torch.bfloat16, device=DEV)
            assert ring_tiles(lambda: ops.linear_w8a8_dynamic(c, x, w, cs, None, act, trans_b)) == {tile}, (trans_b, act)


@pytest.mark.parametrize("m,k,n", [(300, 4112, 11008), (434, 2192, 18688), (131, 9136, 18048)])
def test_linears_of_ragged_k_leave_the_register_staged_tiles(m, k, n):
    """[n, k] weights with a k off 128 and tiles enough for the chip: the plain matmul runs register-staged tiles, which the ring is
    twice as fast as, so the linear takes the ring; sampled columns against exact sums."""
    announce("ring or staged", m, k, n)
    g = torch.Generator(device=DEV)
    g.manual_seed(m + k)
    x = torch.randn((m, k), device=DEV, generator=g).to(torch.bfloat16)
    w = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=DEV, generator=g)
    cs = torch.rand(n, device=DEV, generator=g) * 1e-3 + 1e-4
    c = torch.zeros((m, n), dtype=torch.bfloat16, device=DEV)
    assert ring_tiles(lambda: ops.linear_w8a8_dynamic(c, x, w, cs, trans_b=True)) != set()
    q, ts = ops.dynamic_quant_per_token(x)
    cols = torch.tensor([0, 1, 63, 64, 127, 128, n // 2, n - 9, n - 1], device=DEV)
    want = (q.double() @ w[cols].double().t().contiguous()).float() * cs[cols] * ts[:, None]      # exact sums, one rounding per step
    assert torch.equal(c[:, cols], want.to(torch.bfloat16))


@pytest.mark.parametrize("m,n,k", [(100, 272, 1040), (130, 528, 1152), (257, 1000, 1280)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_matmul_outputs_of_the_ring_tiles(m, n, k, trans_b):
    """The plain matmul where 64 x 64 tiles with a ring of stages are one round of the chip: raw int32 sums, and quant words
    with and without the pre-shift to every output type."""
    mm = ops.Matmul(m, n, k, trans_b=trans_b)
    mm.set_tensor_a(torch.zeros((m, k), dtype=torch.int8, device=DEV))
    mm.set_tensor_b(torch.zeros((n, k) if trans_b else (k, n), dtype=torch.int8, device=DEV))
    plan = mm.plan(torch.zeros((m, n), dtype=torch.int32, device=DEV))
    assert (plan.tile_m, plan.tile_n) == (64, 64)
    test_int32_accumulators_bit_exact(m, n, k, trans_b)
    test_fixpipe_pre_shift_words(m, n, k, trans_b)


@pytest.mark.parametrize("m,kernel", [(1, abi.MM_KERNEL_STREAM), (100, abi.MM_KERNEL_DMA_128),
                                      (700, abi.MM_KERNEL_DMA_256)])
def test_matmul_plan_then_call(m, kernel):
    """The plan query names the kernel family and launches nothing; the call that follows is unaffected."""
    announce("plan", m)
    rng = np.random.default_rng(m)
    n, k = 544, 384
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    w = rng.integers(-127, 128, (k, n)).astype(np.int8)
    c = torch.full((m, n), -7, dtype=torch.int32, device=DEV)
    mm = ops.Matmul(m, n, k)
    mm.set_tensor_a(to_dev(a))
    mm.set_tensor_b(to_dev(w))
    plan = mm.plan(c)
    torch.cuda.synchronize()
    assert plan.kernel == kernel and plan.launches >= 1 and plan.workgroups >= 1
    assert bool((c == -7).all())                      # nothing ran
    mm.iterate_all(c)
    assert np.array_equal(c.cpu().numpy(), a.astype(np.int32) @ w.astype(np.int32))


@pytest.mark.parametrize("g,k,n", [(1, 16, 32), (1, 128, 160), (3, 208, 544), (2, 4096, 1024), (1, 80, 11008)])
def test_pack_weight_nz(g, k, n):
    """The device-side packer against the reference script's reshape / transpose, and its error paths."""
    announce("pack nz", g, k, n)
    rng = np.random.default_rng(g + k + n)
    w = rng.integers(-128, 128, (g, k, n)).astype(np.int8)
    got = ops.pack_weight_nz(to_dev(w)).cpu().numpy()
    assert np.array_equal(got, to_nz(w))
    if g == 1:
        got2 = ops.pack_weight_nz(to_dev(w[0])).cpu().numpy()
        assert got2.shape == (n // 32, k // 16, 16, 32) and np.array_equal(got2, to_nz(w[0]))


def test_pack_weight_nz_feeds_the_matmul():
    """ND weights packed on the device give the product of the ND weights, bit for bit."""
    announce("pack nz + matmul")
    rng = np.random.default_rng(0x4E5A)
    m, n, k = 300, 544, 384
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    w = rng.integers(-127, 128, (k, n)).astype(np.int8)
    c = torch.zeros((m, n), dtype=torch.int32, device=DEV)
    mm = ops.Matmul(m, n, k)
    mm.set_tensor_a(to_dev(a))
    mm.set_tensor_b(ops.pack_weight_nz(to_dev(w)), nz=True)
    mm.iterate_all(c)
    assert np.array_equal(c.cpu().numpy(), a.astype(np.int32) @ w.astype(np.int32))


def test_pack_weight_nz_rejects():
    announce("pack nz rejects")
    w = torch.zeros((24, 32), dtype=torch.int8, device=DEV)
    with pytest.raises(ops.AscqError, match="k % 16"):
        ops.pack_weight_nz(w)
    w = torch.zeros((16, 48), dtype=torch.int8, device=DEV)
    with pytest.raises(ops.AscqError, match="n % 32"):
        ops.pack_weight_nz(w)
    w = torch.zeros((16, 32), dtype=torch.int8, device=DEV)
    with pytest.raises(ops.AscqError, match="same buffer"):
        ops.pack_weight_nz(w, out=w)


def test_group_matmul_nz_weights_as_the_reference_example_packs_them():
    """The example's configuration in small: counts group list, fractal weights, FasterGelu, fp16 out."""
    announce("group nz")
    rng = np.random.default_rng(0x6E7A)
    groups, k, n = 4, 256, 320
    counts = [100, 0, 257, 31]
    m = sum(counts)
    x = rng.integers(-10, 10, (m, k)).astype(np.int8)
    w = rng.integers(-10, 10, (groups, k, n)).astype(np.int8)
    sc = rng.normal(0, 0.01, (groups, n)).astype(np.float32)
    ts = rng.normal(0, 0.01, m).astype(np.float32)
    y = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    gl = torch.tensor(counts, dtype=torch.int64, device=DEV)
    ops.quant_group_matmul(y, to_dev(x), to_dev(to_nz(w)), gl, to_dev(sc), to_dev(ts),
                           activation=abi.MM_ACT_FASTER_GELU, weight_nz=True)
    mmd = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.F16, quant_mode=abi.MM_QUANT_VECTOR,
                         scale_format=abi.MM_SCALE_F32, has_tok_scale=1, activation=abi.MM_ACT_FASTER_GELU)
    gd = abi.GroupMatmulDesc(mm=mmd, groups=groups, group_list_kind=abi.GROUP_LIST_COUNTS)
    want = orc.group_matmul_w8a8(gd, x, w, None, sc, ts, np.array(counts, dtype=np.int64))
    got = bits(y)
    assert max_ulp(got, want.view(np.uint16), "f16") <= 1


def test_group_matmul_example_full_size_nz_equals_nd():
    """The reference example's own size (8 groups x 1024 tokens, k=1024, n=8192, FasterGelu, fp16): the result from
    the fractal weights is bit-equal to the one from row-major weights (which the other tests tie to the oracle), and
    a sample of rows is checked against the example's golden formula in float64."""
    announce("group example full size")
    rng = np.random.default_rng(0xE8A)
    groups, m, k, n = 8, 8192, 1024, 8192
    counts = [1024] * groups
    x = rng.integers(-10, 10, (m, k)).astype(np.int8)
    w = rng.integers(-10, 10, (groups, k, n)).astype(np.int8)
    sc = rng.normal(0, 0.01, (groups, n)).astype(np.float32)
    ts = rng.normal(0, 0.01, m).astype(np.float32)
    gl = torch.tensor(counts, dtype=torch.int64, device=DEV)
    xd, scd, tsd = to_dev(x), to_dev(sc), to_dev(ts)
    y_nd = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    y_nz = torch.zeros((m, n), dtype=torch.float16, device=DEV)
    ops.quant_group_matmul(y_nd, xd, to_dev(w), gl, scd, tsd, activation=abi.MM_ACT_FASTER_GELU)
    ops.quant_group_matmul(y_nz, xd, to_dev(to_nz(w)), gl, scd, tsd, activation=abi.MM_ACT_FASTER_GELU, weight_nz=True)
    assert torch.equal(y_nd.view(torch.int16), y_nz.view(torch.int16))
    rows = rng.choice(m, 64, replace=False)
    got = y_nz[torch.from_numpy(rows).to(DEV)].float().cpu().numpy().astype(np.float64)
    for i, r in enumerate(rows):
        g = r // 1024
        v = (x[r].astype(np.float64) @ w[g].astype(np.float64)) * sc[g].astype(np.float64) * float(ts[r])
        gold = v / (1.0 + np.exp(-1.702 * v))                       # the example's FastGelu, in closed form
        assert np.all(np.abs(got[i] - gold) <= 2e-3 * np.abs(gold) + 1e-6)

# ------------------------------------------------------------------ SwiGLU epilogue
def swiglu_close(got_bits, want_bits, fmt):
    # expf of the device library against libm: the activation may differ by an ulp of the output type
    assert max_ulp(got_bits, want_bits, fmt) <= 1
    assert np.mean(got_bits == want_bits) > 0.98


@pytest.mark.parametrize("m,n,k", [(1, 64, 128), (16, 1040, 2048), (33, 144, 128), (200, 528, 384), (600, 528, 640),
                                   (1100, 784, 384), (19, 22, 77), (2048, 2832, 384)])
@pytest.mark.parametrize("out,bias", [(torch.bfloat16, None), (torch.float16, "f32"), (torch.float32, "bf16")])
def test_matmul_swiglu_epilogue(m, n, k, out, bias):
    """Columns 2j / 2j + 1 -> output column j; every kernel family (weight streams, K-split tiles, large tiles with the
    in-register form, generic) against the oracle."""
    announce("swiglu", m, n, k, out, bias)
    rng = np.random.default_rng(m * 3 + n + k)
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    cs = rng.uniform(1e-4, 4e-4, n).astype(np.float32)
    ts = rng.uniform(0.5, 2.0, m).astype(np.float32)
    bv = None
    if bias == "f32":
        bv = (rng.standard_normal(n).astype(np.float32), None)
    elif bias == "bf16":
        bv = (orc.f32_to_bf16_bits(rng.standard_normal(n).astype(np.float32)), "bf16")
    mm = ops.Matmul(m, n, k)
    mm.set_tensor_a(to_dev(a))
    mm.set_tensor_b(to_dev(b))
    mm.set_quant_vector(to_dev(cs))
    mm.set_token_scale(to_dev(ts))
    if bv is not None:
        mm.set_bias(to_dev(bv[0], bv[1]))
    mm.set_activation(abi.MM_ACT_SWIGLU, 1.0 if m % 2 else 1.702)
    c = torch.zeros((m, n // 2), dtype=out, device=DEV)
    mm.iterate_all(c)
    want = oracle_mm(mm.desc, a, b, bv, cs, ts)
    if out == torch.float32:
        got = c.cpu().numpy()
        assert np.all(np.abs(got - want) <= 4 * np.spacing(np.abs(want)) + 1e-30)
    else:
        fmt = "bf16" if out == torch.bfloat16 else "f16"
        swiglu_close(bits(c), want.view(np.uint16), fmt)


def test_group_matmul_swiglu_and_dynamic_linear():
    """The grouped matmul (MoE gate / up projection with interleaved columns) and the fused quantise + linear call."""
    announce("group swiglu")
    rng = np.random.default_rng(0x51)
    groups, m, k, n = 4, 700, 256, 544
    counts = np.array([300, 0, 1, 399], dtype=np.int64)
    x, w = rand_i8(rng, (m, k)), rand_i8(rng, (groups, k, n))
    sc = rng.uniform(1e-4, 4e-4, (groups, n)).astype(np.float32)
    ts = rng.uniform(0.5, 2.0, m).astype(np.float32)
    y = torch.zeros((m, n // 2), dtype=torch.bfloat16, device=DEV)
    ops.quant_group_matmul(y, to_dev(x), to_dev(w), to_dev(counts), to_dev(sc), to_dev(ts),
                           activation=abi.MM_ACT_SWIGLU, act_beta=1.0)
    mmd = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32,
                         has_tok_scale=1, activation=abi.MM_ACT_SWIGLU, act_beta=1.0)
    gd = abi.GroupMatmulDesc(mm=mmd, groups=groups, group_list_kind=abi.GROUP_LIST_COUNTS)
    want = orc.group_matmul_w8a8(gd, x, w, None, sc, ts, counts)
    swiglu_close(bits(y), want.view(np.uint16), "bf16")
    # dynamic quantisation + linear + SwiGLU in one call, decode and prefill sizes
    for mm_rows in (3, 640):
        xa = orc.f32_to_bf16_bits(rng.standard_normal((mm_rows, k)).astype(np.float32))
        wl = rand_i8(rng, (k, n))
        cs = rng.uniform(1e-4, 4e-4, n).astype(np.float32)
        c = torch.zeros((mm_rows, n // 2), dtype=torch.bfloat16, device=DEV)
        ops.linear_w8a8_dynamic(c, to_dev(xa, "bf16"), to_dev(wl), to_dev(cs), activation=abi.MM_ACT_SWIGLU)
        q, tsn = orc.dynamic_quant_per_token(abi.BF16, xa)
        d = abi.MatmulDesc(m=mm_rows, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR,
                           scale_format=abi.MM_SCALE_F32, has_tok_scale=1, activation=abi.MM_ACT_SWIGLU, act_beta=1.0)
        swiglu_close(bits(c), orc.matmul_w8a8(d, q, wl, None, cs, tsn).view(np.uint16), "bf16")


@pytest.mark.parametrize("m", [1, 5, 16, 17, 64, 130, 300])
@pytest.mark.parametrize("n,k", [(22, 128), (1040, 2048), (528, 384), (96, 4096), (64, 8192), (48, 11008)])
@pytest.mark.parametrize("out,bias", [(torch.bfloat16, None), (torch.float16, "f32"), (torch.float32, "bf16")])
def test_matmul_swiglu_in_the_decode_kernels(m, n, k, out, bias):
    """SwiGLU on [n, k] and on packed weights: the decode kernels (activations resident in LDS up to 16 rows, weights
    held in registers beyond, also in chunks of a longer k) pair the columns of a row through neighbouring lanes in
    their own epilogue - one launch, no raw accumulators; [n, k] weights past 224 rows (64 or 48 at k above 4096) take the
    tile kernels.  Against the oracle."""
    announce("swiglu decode", m, n, k, out, bias)
    rng = np.random.default_rng(m * 5 + n + k)
    a, b = rand_i8(rng, (m, k)), rand_i8(rng, (k, n))
    cs = rng.uniform(1e-4, 4e-4, n).astype(np.float32)
    ts = rng.uniform(0.5, 2.0, m).astype(np.float32)
    bv = None
    if bias == "f32":
        bv = (rng.standard_normal(n).astype(np.float32), None)
    elif bias == "bf16":
        bv = (orc.f32_to_bf16_bits(rng.standard_normal(n).astype(np.float32)), "bf16")
    beta = 1.0 if m % 2 else 1.702
    want = None
    for packed in (False, True):
        mm = ops.Matmul(m, n, k, False, not packed)
        mm.set_tensor_a(to_dev(a))
        if packed:
            mm.set_tensor_b_packed(ops.pack_weight_w8(to_dev(b), k, n))
        else:
            mm.set_tensor_b(to_dev(np.ascontiguousarray(b.T)))
        mm.set_quant_vector(to_dev(cs))
        mm.set_token_scale(to_dev(ts))
        if bv is not None:
            mm.set_bias(to_dev(bv[0], bv[1]))
        mm.set_activation(abi.MM_ACT_SWIGLU, beta)
        c = torch.zeros((m, n // 2), dtype=out, device=DEV)
        mm.iterate_all(c)
        if want is None:
            d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=mm.desc.out_dtype, quant_mode=abi.MM_QUANT_VECTOR,
                               scale_format=abi.MM_SCALE_F32, has_tok_scale=1, bias_kind=mm.desc.bias_kind,
                               activation=abi.MM_ACT_SWIGLU, act_beta=beta)
            want = oracle_mm(d, a, b, bv, cs, ts)
        if out == torch.float32:
            assert np.all(np.abs(c.cpu().numpy() - want) <= 4 * np.spacing(np.abs(want)) + 1e-30)
        else:
            swiglu_close(bits(c), want.view(np.uint16), "bf16" if out == torch.bfloat16 else "f16")


@pytest.mark.parametrize("m", [1, 3, 8, 12, 40])
def test_linear_dynamic_swiglu_in_one_launch(m):
    """The gate / up projection of a decode step in one call: per-token quantisation, int8 matmul on [n, k] or packed
    weights, SwiGLU of the column pairs (up to 8 rows inside one kernel).  Against the oracle of the steps."""
    announce("linear dynamic swiglu", m)
    rng = np.random.default_rng(0x5E + m)
    k, n = 512, 736
    xa = orc.f32_to_bf16_bits(rng.standard_normal((m, k)).astype(np.float32))
    w = rand_i8(rng, (k, n))
    cs = rng.uniform(1e-4, 4e-4, n).astype(np.float32)
    q, tsn = orc.dynamic_quant_per_token(abi.BF16, xa)
    d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32,
                       has_tok_scale=1, activation=abi.MM_ACT_SWIGLU, act_beta=1.0)
    want = orc.matmul_w8a8(d, q, w, None, cs, tsn).view(np.uint16)
    c = torch.zeros((m, n // 2), dtype=torch.bfloat16, device=DEV)
    ops.linear_w8a8_dynamic(c, to_dev(xa, "bf16"), to_dev(np.ascontiguousarray(w.T)), to_dev(cs), trans_b=True,
                            activation=abi.MM_ACT_SWIGLU)
    swiglu_close(bits(c), want, "bf16")
    c2 = torch.zeros((m, n // 2), dtype=torch.bfloat16, device=DEV)
    ops.linear_w8a8_dynamic_packed(c2, to_dev(xa, "bf16"), ops.pack_weight_w8(to_dev(w), k, n), n, to_dev(cs),
                                   activation=abi.MM_ACT_SWIGLU)
    swiglu_close(bits(c2), want, "bf16")
    assert torch.equal(c, c2)


# ------------------------------------------------------------------ workspace contract, determinism
@pytest.mark.parametrize("m", [1, 5, 16, 19, 130])
def test_workspaces_need_no_initialisation_and_results_repeat(m):
    """The scratch of the weight-stream and split-K paths may hold anything (here: all-ones bytes = NaN / -1) and two
    calls give the same bits."""
    announce("workspace garbage", m)
    rng = np.random.default_rng(0x5C + m)
    k, n = 1024, 1056
    # W8A8 (stream kernel for m <= 32, split-K tiles above)
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    w = rng.integers(-127, 128, (k, n)).astype(np.int8)
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    mm = ops.Matmul(m, n, k)
    mm.set_tensor_a(to_dev(a))
    mm.set_tensor_b(to_dev(w))
    mm.set_quant_vector(to_dev(cs))
    c1 = torch.zeros((m, n), dtype=torch.bfloat16, device=DEV)
    mm.iterate_all(c1)
    if mm._ws is not None:
        mm._ws.fill_(-1)
    c2 = torch.zeros((m, n), dtype=torch.bfloat16, device=DEV)
    mm.iterate_all(c2)
    d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32)
    want = orc.matmul_w8a8(d, a, w, None, cs, None)
    assert np.array_equal(bits(c1), want) and np.array_equal(bits(c2), want)
    # W4A16 and W8A16
    x = rng.standard_normal((m, k)).astype(np.float16)
    xw, wp, sc, of = w4_case(rng, m, k, n, 128, True)
    garbage = torch.full((1 << 22,), float("nan"), dtype=torch.float32, device=DEV)
    outs = []
    for ws in (None, garbage, garbage):
        y4 = torch.zeros((m, n), dtype=torch.float16, device=DEV)
        ops.matmul_w4a16(y4, to_dev(xw), to_dev(wp), to_dev(sc), to_dev(of), 128, workspace=ws)
        y8 = torch.zeros((m, n), dtype=torch.float16, device=DEV)
        ops.matmul_w8a16(y8, to_dev(x), to_dev(w), to_dev(of[0]), to_dev(sc[0]), workspace=ws)
        outs.append((bits(y4), bits(y8)))
        garbage.fill_(float("nan"))
    for y4, y8 in outs[1:]:
        assert np.array_equal(y4, outs[0][0]) and np.array_equal(y8, outs[0][1])
    assert not np.isnan(outs[0][0].view(np.float16)).any() and not np.isnan(outs[0][1].view(np.float16)).any()

# ------------------------------------------------------------------ fused dynamic quantisation + matmul
@pytest.mark.parametrize("m", [1, 2, 5, 8, 9, 40])
@pytest.mark.parametrize("k,n", [(256, 128), (1024, 1056), (4096, 2064), (320, 48)])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float16, torch.float32])
def test_linear_w8a8_dynamic_equals_quantise_then_matmul(m, k, n, xdt):
    """One call = per-token quantisation followed by the matmul, bit for bit (oracle of the two steps)."""
    announce("linear dynamic", m, k, n, xdt)
    rng = np.random.default_rng(m * 3 + k + n)
    xf = rng.standard_normal((m, k)).astype(np.float32) * rng.uniform(0.1, 30.0, (m, 1)).astype(np.float32)
    if m > 2:
        xf[1] = 0.0                                       # an all-zero row: scale 1, zeros
    x = torch.from_numpy(xf).to(DEV).to(xdt)
    w = rng.integers(-127, 128, (k, n)).astype(np.int8)
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c = torch.zeros((m, n), dtype=torch.bfloat16, device=DEV)
    ops.linear_w8a8_dynamic(c, x, to_dev(w), to_dev(cs), to_dev(bias))
    xdt_abi = {torch.bfloat16: abi.BF16, torch.float16: abi.F16, torch.float32: abi.F32}[xdt]
    q, ts = orc.dynamic_quant_per_token(xdt_abi, bits(x))
    d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32,
                       has_tok_scale=1, bias_kind=abi.MM_BIAS_F32_POST)
    want = orc.matmul_w8a8(d, q, w, bias, cs, ts)
    assert np.array_equal(bits(c), want)


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 7, 8, 9, 17])
@pytest.mark.parametrize("k,n", [(64, 16), (192, 40), (256, 128), (1024, 1056), (4096, 2064), (320, 48), (5632, 100),
                                 (8192, 100), (11008, 272), (12288, 16)])
@pytest.mark.parametrize("xdt,odt", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                     (torch.bfloat16, torch.float32)])
def test_linear_w8a8_dynamic_on_n_k_weights(m, k, n, xdt, odt):
    """Weights kept as [n, k] (isTransposeB): up to 8 rows are quantised inside the weight-streaming kernel, more rows
    by the two kernels; either way the bits of quantise-then-matmul (oracle of the two steps)."""
    announce("linear dynamic [n, k]", m, k, n, xdt, odt)
    rng = np.random.default_rng(m * 7 + k + n)
    xf = rng.standard_normal((m, k)).astype(np.float32) * rng.uniform(0.1, 30.0, (m, 1)).astype(np.float32)
    if m > 2:
        xf[1] = 0.0
        xf[2, : k // 2] = 0.0                              # the row's maximum lies in the upper half of k only
    x = torch.from_numpy(xf).to(DEV).to(xdt)
    w = rng.integers(-127, 128, (n, k)).astype(np.int8)
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c = torch.zeros((m, n), dtype=odt, device=DEV)
    ops.linear_w8a8_dynamic(c, x, to_dev(w), to_dev(cs), to_dev(bias), trans_b=True)
    xdt_abi = {torch.bfloat16: abi.BF16, torch.float16: abi.F16}[xdt]
    odt_abi = {torch.bfloat16: abi.BF16, torch.float16: abi.F16, torch.float32: abi.F32}[odt]
    q, ts = orc.dynamic_quant_per_token(xdt_abi, bits(x))
    d = abi.MatmulDesc(m=m, n=n, k=k, trans_b=1, out_dtype=odt_abi, quant_mode=abi.MM_QUANT_VECTOR,
                       scale_format=abi.MM_SCALE_F32, has_tok_scale=1, bias_kind=abi.MM_BIAS_F32_POST)
    want = orc.matmul_w8a8(d, q, w, bias, cs, ts)
    assert np.array_equal(bits(c), gpu_util.as_bits(want))


@pytest.mark.parametrize("m", [1, 3, 4, 5, 8, 9, 33])
@pytest.mark.parametrize("k,n", [(64, 16), (192, 40), (1024, 1056), (4096, 2064), (11008, 272)])
@pytest.mark.parametrize("xdt,src_nk", [(torch.bfloat16, False), (torch.float16, True), (torch.float32, False)])
def test_linear_w8a8_dynamic_on_packed_weights(m, k, n, xdt, src_nk):
    """ascq_linear_w8a8_dynamic_packed: up to 8 rows of half / bfloat16 x in one launch, anything else quantiser +
    packed matmul; either way the bits of quantise-then-matmul (oracle of the two steps)."""
    announce("linear dynamic packed", m, k, n, xdt, src_nk)
    rng = np.random.default_rng(m * 11 + k + n)
    xf = rng.standard_normal((m, k)).astype(np.float32) * rng.uniform(0.1, 30.0, (m, 1)).astype(np.float32)
    if m > 2:
        xf[1] = 0.0
    x = torch.from_numpy(xf).to(DEV).to(xdt)
    w = rng.integers(-127, 128, (k, n)).astype(np.int8)
    wp = ops.pack_weight_w8(to_dev(np.ascontiguousarray(w.T)) if src_nk else to_dev(w), k, n, src_nk)
    cs = rng.uniform(1e-4, 1e-2, n).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    c = torch.zeros((m, n), dtype=torch.bfloat16, device=DEV)
    ops.linear_w8a8_dynamic_packed(c, x, wp, n, to_dev(cs), to_dev(bias))
    xdt_abi = {torch.bfloat16: abi.BF16, torch.float16: abi.F16, torch.float32: abi.F32}[xdt]
    q, ts = orc.dynamic_quant_per_token(xdt_abi, bits(x))
    d = abi.MatmulDesc(m=m, n=n, k=k, out_dtype=abi.BF16, quant_mode=abi.MM_QUANT_VECTOR, scale_format=abi.MM_SCALE_F32,
                       has_tok_scale=1, bias_kind=abi.MM_BIAS_F32_POST)
    want = orc.matmul_w8a8(d, q, w, bias, cs, ts)
    assert np.array_equal(bits(c), want)


@pytest.mark.parametrize("m", [2, 9])
def test_prepared_linear_object_equals_the_function(m):
    """ops.DynamicLinear (descriptor and scratch prepared once) gives what ops.linear_w8a8_dynamic gives, on [k, n],
    [n, k] and packed weights."""
    k, n = 512, 208
    rng = np.random.default_rng(m)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(DEV).to(torch.bfloat16)
    w = to_dev(rng.integers(-127, 128, (k, n)).astype(np.int8))
    wt = w.t().contiguous()
    cs, bias = to_dev(rng.uniform(1e-4, 1e-2, n).astype(np.float32)), to_dev(rng.standard_normal(n).astype(np.float32))
    want = ops.linear_w8a8_dynamic(torch.zeros((m, n), dtype=torch.bfloat16, device=DEV), x, w, cs, bias)
    for lin in (ops.DynamicLinear(m, k, w, cs, bias), ops.DynamicLinear(m, k, wt, cs, bias, trans_b=True),
                ops.DynamicLinear(m, k, ops.pack_weight_w8(w, k, n), cs, bias, packed_n=n)):
        for _ in range(2):
            got = lin(torch.zeros((m, n), dtype=torch.bfloat16, device=DEV), x)
            assert torch.equal(got, want)


# ------------------------------------------------------------------ Matmul<int4b_t, int4b_t, C>
def ref_pack_int4(x):
    """The packing of the reference example's script (matmul_int4/scripts/gen_data.py:32-42): byte j of a row is
    (x[2j+1] << 4) + (x[2j] & 0x0F), kept in int8."""
    return ((x[..., 1::2].astype(np.int32) << 4) + (x[..., 0::2].astype(np.int32) & 0x0F)).astype(np.int8)


def test_matmul_int4_reference_example():
    """The example at its own size and with its own data recipe: M=256, N=7680, K=128, values from
    uniform(-5, 5) cast to int8, int32 bias, int32 out (matmul_int4/scripts/gen_data.py:20-31)."""
    announce("int4 example")
    rng = np.random.default_rng(0x14)
    m, n, k = 256, 7680, 128
    x1 = rng.uniform(-5, 5, (m, k)).astype(np.int8)
    x2 = rng.uniform(-5, 5, (k, n)).astype(np.int8)
    bias = rng.uniform(-5, 5, n).astype(np.int32)
    golden = x1.astype(np.int32) @ x2.astype(np.int32) + bias
    c = torch.zeros((m, n), dtype=torch.int32, device=DEV)
    mm = ops.MatmulInt4(m, n, k)
    mm.set_tensor_a(to_dev(ref_pack_int4(x1)))
    mm.set_tensor_b(to_dev(ref_pack_int4(x2)))
    mm.set_bias(to_dev(bias))
    mm.iterate_all(c)
    assert np.array_equal(c.cpu().numpy(), golden)


@pytest.mark.parametrize("m,n,k,trans_b", [(1, 64, 128, False), (33, 160, 96, False), (200, 544, 384, True),
                                           (513, 34, 130, False), (70, 33, 64, True)])
@pytest.mark.parametrize("out", [torch.int32, torch.float16])
def test_matmul_int4_full_range(m, n, k, trans_b, out):
    """Every nibble value, both B orientations, int32 and the half output the reference allows (through the
    fixpipe scale words), bit-equal to the int8 oracle on the widened operands."""
    announce("int4", m, n, k, trans_b, out)
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-8, 8, (m, k)).astype(np.int8)
    b = rng.integers(-8, 8, (n, k) if trans_b else (k, n)).astype(np.int8)
    c = torch.zeros((m, n), dtype=out, device=DEV)
    mm = ops.MatmulInt4(m, n, k, trans_b=trans_b)
    mm.set_tensor_a(to_dev(pack_int4(a)))
    mm.set_tensor_b(to_dev(pack_int4(b)))
    d = abi.MatmulDesc(m=m, n=n, k=k, trans_b=int(trans_b), out_dtype=abi.I32)
    qv = None
    if out != torch.int32:
        qv = np.array([ops.pack_quant_param(s) for s in rng.uniform(1e-3, 1e-1, n)], dtype=np.uint64)
        mm.set_quant_vector(to_dev(qv.view(np.int64)))
        d = abi.MatmulDesc(m=m, n=n, k=k, trans_b=int(trans_b), out_dtype=abi.F16, quant_mode=abi.MM_QUANT_VECTOR,
                           scale_format=abi.MM_SCALE_U64)
    mm.iterate_all(c)
    want = orc.matmul_w8a8(d, a, b, None, qv, None)
    assert np.array_equal(bits(c), want if out == torch.int32 else want.view(np.uint16))


@pytest.mark.parametrize("count", [2, 30, 32, 4096 + 34, 1 << 20])
def test_unpack_int4(count):
    announce("unpack int4", count)
    rng = np.random.default_rng(count)
    v = rng.integers(-8, 8, count).astype(np.int8)
    got = ops.unpack_int4(to_dev(pack_int4(v))).cpu().numpy()
    assert got.dtype == np.int8 and np.array_equal(got, v)
    assert np.array_equal(ops.unpack_int4(to_dev(ref_pack_int4(v))).cpu().numpy(), v)


def test_matmul_int4_rejects():
    announce("int4 rejects")
    z = torch.zeros(64, dtype=torch.int8, device=DEV)
    c = torch.zeros((4, 4), dtype=torch.int32, device=DEV)
    for kw, msg in [(dict(m=4, n=4, k=3), "k 3 must be even"), (dict(m=4, n=3, k=4), "n 3 must be even"),
                    (dict(m=4, n=4, k=4, trans_a=True), "cannot be transposed")]:
        mm = ops.MatmulInt4(**kw)
        mm.set_tensor_a(z)
        mm.set_tensor_b(z)
        with pytest.raises(ops.AscqError, match=msg):
            mm.iterate_all(c)
