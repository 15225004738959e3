"""Dense projections of a token batch on the GPU against the CPU oracle, bit for
bit: strata_bf16_project and strata_quant_project at the edges of the batch
kernel's tiles (4 weight rows a wave and 16 a block, one, two and four groups of
4 tokens a wave and what is left of them, chunks of 4 x 64 columns and what is
left of them) and of the general kernels (few outputs, and one column count that
is no multiple of 64)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [  # cols, rows, tokens
    # the general kernel for bf16 (few outputs), the first and the last for quantized weights too (few outputs, ragged columns)
    (64, 1, 2), (64, 1281, 2), (64, 97, 33), (128, 863, 3), (192, 640, 4), (320, 515, 5), (704, 337, 8), (640, 289, 9),
    (3072, 161, 17), (100, 600, 6),
    # one group of tokens a wave
    (64, 2305, 2), (64, 141, 33), (128, 1537, 3), (192, 1153, 4), (320, 923, 5), (640, 513, 9), (5120, 700, 7),
    # two: 7, 13 of 16, 27 of 32 and all tokens; 1, 1, 2 and no steps past the last whole chunk
    (64, 10240, 7), (320, 4100, 13), (128, 4100, 27), (2560, 4100, 16),
    # four: 61 of 64, 30 of 32 and all; 3, 2 and 3 steps
    (704, 2570, 61), (384, 6000, 30), (1216, 8200, 32)]


def same(a, b):
    nan = np.isnan(b)
    assert np.array_equal(np.isnan(a), nan)
    assert np.array_equal(a.view(np.uint32)[~nan], b.view(np.uint32)[~nan])


def inputs(cols, rows, tokens):
    """Rows of ordinary, tiny (their products are subnormal or underflow) and huge values, and a few zeros and infinities."""
    rng = np.random.default_rng(cols + rows + tokens)
    x = rng.normal(0, 1, (tokens, cols)).astype(np.float32)
    x[tokens // 2] *= np.float32(1e-38)
    x[-1] *= np.float32(1e30)
    x[0, :: max(cols // 7, 1)] = -0.0
    if tokens > 2:
        x[1, cols - 1] = np.inf
    return rng, x.reshape(-1)


@pytest.mark.parametrize("cols,rows,tokens", SHAPES)
def test_bf16_batch(backend, oracle, cols, rows, tokens):
    rng, x = inputs(cols, rows, tokens)
    w = rng.normal(0, 0.05, rows * cols).astype(np.float32)
    w[rows * cols // 2] = np.inf
    w[rows * cols // 3] = -1e-39
    half = (w.view(np.uint32) >> 16).astype(np.uint32)
    codes = half[0::2] | half[1::2] << 16
    stride, off = rows + 3, 2
    y = backend.alloc(np.full(tokens * stride, -7, np.float32))
    backend.run("strata_bf16_project", {"X": backend.alloc(x), "Codes": backend.alloc(codes, "u32"), "Y": y, "cols": cols,
                                        "rows": rows, "tokens": tokens, "outputStride": stride, "outputOffset": off},
                [rows, tokens, 1])
    want = oracle.bf16_project(x, codes, cols, rows, tokens, stride, off, Y=np.full(tokens * stride, -7, np.float32))
    same(backend.read(y), want)


@pytest.mark.parametrize("cols,rows,tokens", SHAPES)
@pytest.mark.parametrize("nbits,group,codebook,offset", [(4, 32, 0, 1), (8, 32, 0, 1), (4, 64, 1, 0), (2, 4, 0, 0),
                                                         (8, 20, 0, 1)])
def test_quant_batch(backend, oracle, cols, rows, tokens, nbits, group, codebook, offset):
    if cols % group:
        group = 4
    rng, x = inputs(cols, rows, tokens)
    codes = rng.integers(0, 1 << 32, (rows * cols * nbits + 31) // 32, dtype=np.uint32)
    scales = rng.normal(0, 0.02, rows * cols // group).astype(np.float32)
    offsets = rng.normal(0, 0.01, scales.size).astype(np.float32)
    stride, off, bias = rows + 3, 2, -(1 << (nbits - 1))
    y = backend.alloc(np.full(tokens * stride, -7, np.float32))
    backend.run("strata_quant_project",
                {"X": backend.alloc(x), "Codes": backend.alloc(codes, "u32"), "Scales": backend.alloc(scales),
                 "Offsets": backend.alloc(offsets), "Y": y, "cols": cols, "rows": rows, "tokens": tokens,
                 "outputStride": stride, "outputOffset": off, "bits": nbits, "groupSize": group, "bias": bias,
                 "codebook": codebook, "hasOffset": offset}, [rows, tokens, 1])
    want = oracle.quant_project(x, codes, scales, offsets, np.full(tokens * stride, -7, np.float32), cols, rows, tokens,
                                stride, off, nbits, group, bias, codebook, offset)
    same(backend.read(y), want)


ONE_TOKEN = [(cols, rows, *form) for cols, rows in ((64, 1), (128, 3), (320, 17), (2560, 4100), (4096, 66), (3072, 301), (100, 7))
             for form in ((4, 32, 0, 1), (8, 32, 0, 1), (4, 64, 1, 0), (2, 4, 0, 0), (8, 64, 0, 0), (2, 32, 0, 1), (4, 2, 0, 1))]
# groups of one and two weights, by the general kernel and (more than 2,048 rows, up to 256 groups each) from LDS;
# rows in pieces of 2,048 columns (groups of 16 and 4, a group of two pieces, a short last piece of one group) and 1,024
ONE_TOKEN += [(256, 35, 8, 1, 0, 1), (576, 2050, 8, 2, 0, 1), (256, 2051, 8, 1, 0, 1), (192, 2054, 2, 1, 0, 0), (512, 2049, 4, 2, 1, 1),
              (4096, 3101, 8, 16, 0, 1), (4096, 2051, 4, 4, 1, 1), (8192, 3074, 4, 4096, 0, 1), (6208, 3079, 8, 64, 0, 0), (4096, 8195, 8, 16, 0, 1)]


@pytest.mark.parametrize("cols,rows,nbits,group,codebook,offset", ONE_TOKEN)
def test_quant_one_token(backend, oracle, cols, rows, nbits, group, codebook, offset):
    """One token: blocks of four, three and fewer waves (the rows' bytes in LDS), waves of four rows and fewer."""
    if cols % group:
        group = 4
    rng, x = inputs(cols, rows, 2)
    x = x[:cols] if rows % 2 else x[cols:]
    codes = rng.integers(0, 1 << 32, (rows * cols * nbits + 31) // 32, dtype=np.uint32)
    scales = rng.normal(0, 0.02, rows * cols // group).astype(np.float32)
    offsets = rng.normal(0, 0.01, scales.size).astype(np.float32)
    bias = -(1 << (nbits - 1))
    y = backend.alloc(np.full(rows + 1, -7, np.float32))
    backend.run("strata_quant_gemv",
                {"X": backend.alloc(x), "Codes": backend.alloc(codes, "u32"), "Scales": backend.alloc(scales),
                 "Offsets": backend.alloc(offsets), "Y": y, "cols": cols, "rows": rows, "bits": nbits, "groupSize": group,
                 "bias": bias, "codebook": codebook, "hasOffset": offset}, [rows, 1, 1])
    want = oracle.quant_gemv(x, codes, scales, offsets, cols, rows, nbits, group, bias, codebook, offset)
    got = backend.read(y)
    same(got[:rows], np.asarray(want, np.float32).reshape(-1)[:rows])
    assert got[rows] == -7


@pytest.mark.parametrize("W,E,tokens", [(320, 64, 300), (384, 40, 129), (192, 256, 253), (192, 256, 257), (2560, 8, 131)])
def test_route_batch(backend, oracle, W, E, tokens):
    """The router by the batched projection: one group of tokens a wave (131 and
    129 tokens), two with 4 and 5 of 8 tokens left, and past its last size the tiles."""
    rng = np.random.default_rng(W + tokens)
    x, wr = rng.normal(0, 1, tokens * W).astype(np.float32), rng.normal(0, 0.05, E * W).astype(np.float32)
    bias, K = rng.normal(0, 1, E).astype(np.float32), 5
    logits, ids, w = backend.alloc(tokens * E), backend.alloc(tokens * K, "i32"), backend.alloc(tokens * K)
    backend.moe_route(backend.alloc(x), tokens, W, backend.alloc(wr), E, K, ids, w, logits=logits, bias=backend.alloc(bias))
    want = (oracle.project(x, wr, W, E, tokens).reshape(tokens, E) + bias).reshape(-1)
    same(backend.read(logits), want)
    rids, rw = oracle.router(want, E, K, tokens)
    assert np.array_equal(backend.read(ids), rids)
    same(backend.read(w), rw)
