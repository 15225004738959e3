"""The prompt chunk's sequence mixers on the GPU against the CPU oracle, bit for
bit, at the edges of their kernels: attention with one and two heads a wave
(more than 1,024 waves), odd head groups, counts around 64 cells, grids of
fewer heads, tiles or tokens than the layout holds, and values that are not
finite in cells a token must not see; the gated delta rule with grids that end
inside a block of 32 columns and chunks longer than its 16-token stage."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def same(a, b):
    nan = np.isnan(b)
    assert np.array_equal(np.isnan(a), nan)
    assert np.array_equal(a.view(np.uint32)[~nan], b.view(np.uint32)[~nan])


@pytest.mark.parametrize("dim,heads,kvh,position,tokens", [(256, 15, 3, 61, 20), (256, 24, 2, 1000, 11),
                                                           (128, 6, 2, 0, 1), (64, 5, 1, 63, 2), (128, 40, 2, 127, 25),
                                                           (64, 34, 2, 190, 30), (256, 24, 2, 2047, 1),
                                                           # one, two and three launches, and both kernels of scores
                                                           (64, 32, 1, 60, 8), (64, 32, 1, 61, 8), (128, 17, 1, 8, 8), (128, 32, 1, 9, 8),
                                                           (64, 8, 2, 632, 8), (64, 8, 2, 633, 8), (64, 32, 8, 700, 24), (64, 12, 1, 3, 5),
                                                           (64, 32, 2, 40, 3), (128, 8, 2, 376, 8), (128, 8, 2, 377, 8), (128, 5, 1, 100, 7),
                                                           (256, 3, 3, 381, 3), (256, 8, 2, 382, 3), (256, 24, 2, 58, 16), (256, 24, 2, 59, 16)])
def test_attention_batch_edges(backend, oracle, dim, heads, kvh, position, tokens):
    rng = np.random.default_rng(dim + position)
    cells = position + tokens
    keys = rng.normal(0, 1, (cells, kvh * dim)).astype(np.float32)
    values = rng.normal(0, 1, (cells, kvh * dim)).astype(np.float32)
    if tokens > 1:  # seen by the last token only
        keys[-1, 0] = np.inf
        values[-1, ::3] = np.nan
        values[-1, 1] = np.inf
    q = rng.normal(0, 1, tokens * heads * dim).astype(np.float32)
    scale = 1 / np.sqrt(dim)
    want = oracle.attention_batch(q, keys.reshape(-1), values.reshape(-1), dim, heads, kvh, position, scale, tokens)
    bufs = [backend.alloc(v) for v in (q, keys.reshape(-1), values.reshape(-1))]
    tiles = (dim + 63) // 64
    for grid in ([heads, tiles, tokens], [heads - 1, tiles, max(tokens - 1, 1)], [heads, max(tiles - 1, 1), tokens]):
        y = backend.alloc(np.full(q.size, -7, np.float32))
        backend.run("strata_attention_batch", {"Q": bufs[0], "Keys": bufs[1], "Values": bufs[2], "Y": y, "dim": dim,
                                               "heads": heads, "kvHeads": kvh, "position": position, "scale": scale}, grid)
        got, full = backend.read(y).reshape(tokens, heads, dim), np.full((tokens, heads, dim), -7, np.float32)
        part = (slice(0, grid[2]), slice(0, grid[0]), slice(0, 64 * grid[1]))
        full[part] = want.reshape(tokens, heads, dim)[part]
        same(got, full)


@pytest.mark.parametrize("dim,kh,vh,tokens,groups", [(128, 2, 4, 17, 8), (128, 2, 4, 33, 5), (64, 2, 6, 1, 6), (64, 1, 3, 16, 2)])
def test_gdn_batch_edges(backend, oracle, dim, kh, vh, tokens, groups):
    rng = np.random.default_rng(dim + tokens)
    state = rng.normal(0, 0.1, dim * vh * dim).astype(np.float32)
    q, k = (rng.normal(0, dim ** -0.5, tokens * kh * dim).astype(np.float32) for _ in range(2))
    v = rng.normal(0, 1, tokens * vh * dim).astype(np.float32)
    v[5] = -0.0
    decay, beta = (rng.random(tokens * vh).astype(np.float32) for _ in range(2))
    sb, y = backend.alloc(state), backend.alloc(np.full(v.size, -7, np.float32))
    backend.run("strata_gdn_batch", {"State": sb, "Q": backend.alloc(q), "K": backend.alloc(k), "V": backend.alloc(v),
                                     "Decay": backend.alloc(decay), "Beta": backend.alloc(beta), "Y": y, "dim": dim,
                                     "keyHeads": kh, "valueHeads": vh, "tokens": tokens}, [groups, 1, 1])
    after = state.copy()
    want = oracle.gdn_batch(after, q, k, v, decay, beta, dim, kh, vh, tokens).reshape(tokens, -1)
    cols = min(64 * groups, vh * dim)
    want[:, cols:] = -7
    after = after.reshape(dim, -1)
    after[:, cols:] = state.reshape(dim, -1)[:, cols:]
    same(backend.read(y).reshape(tokens, -1), want)
    same(backend.read(sb).reshape(dim, -1), after)
