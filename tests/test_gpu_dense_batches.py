"""The Q8_0 product at the edges of its shapes: every count of tokens where the
columns held or the column tiles change, widths that leave partial steps and
slices or whose rows start off the cache lines, matrices of few and of many
tiles, non-finite and tiny inputs.

Tolerance: an output sums exact products in f32: within 1e-6 of the sum of
magnitudes of the f64 product (at most 8 + 8 + 4 sums, two roundings a block
and the scale's, each of 2^-24 of a partial sum: 1.4e-6 of it if every partial
sum were the whole).  Wide rows of random signs hold to 1e-7: their partial
sums stay below 5 sqrt(n) of n terms, a ninth of the magnitudes at 2,560
inputs, and some 20 independent roundings of that add to 1.5e-8 rms; a lost
low part would give 6e-7 at 8,192 inputs."""
import numpy as np
import pytest

import fg_hip
import oracle_ffi as O
from test_gpu_dense import check_f64, fused, packed_random, plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 2, 5, 6, 8, 9, 16, 17, 32, 33, 48, 49, 64, 65, 130])
@pytest.mark.parametrize("width,rows", [(32, 16), (96, 40), (160, 300), (192, 33), (2560, 300),
                                        (6944, 50), (8192, 17)])
def test_tokens_widths(dev, tokens, width, rows):
    rng = np.random.default_rng(tokens * 31 + width)
    packed = packed_random(rng, width, rows)
    cooked = fg_hip.cook_q8_0(packed, width, rows)
    x = rng.normal(0, 1, (tokens, width)).astype(np.float32)
    y = plain(dev, cooked, x, width, rows, 0.75)
    worst = check_f64(y, packed, x, width, rows, 0.75)
    assert width < 2560 or worst <= 1e-7
    sl = fg_hip.OutputSlice(rows, 1, 0, rows, tokens)
    ref = plain(dev, cooked, x, width, rows, 1.0)
    v, i, s, _ = fused(dev, sl, cooked, x, width, logits=False)
    wv, wi, ws = O.slice_finalists(ref, 0)
    assert np.array_equal(i, wi) and np.array_equal(v.view(np.uint32), wv.view(np.uint32))
    assert np.array_equal(s, ws)
    # A token's logits have the same bits beside any others of its form.
    for n in (m for m in (1, 3, 6, 8, 9, 16, 17, 50) if m < tokens and (m <= 8) == (tokens <= 8)):
        assert np.array_equal(plain(dev, cooked, x[:n], width, rows, 1.0).view(np.uint32),
                              ref[:n].view(np.uint32)), n


@pytest.mark.parametrize("tokens", [1, 4, 7, 16, 30, 40, 64])
@pytest.mark.parametrize("width,rows", [(32, 29_001), (64, 57_345), (160, 127_990), (256, 70_001),
                                        (256, 127_990), (288, 131_073), (2_176, 28_672)])
def test_many_tiles(dev, tokens, width, rows):
    rng = np.random.default_rng(tokens + width)
    packed = packed_random(rng, width, rows)
    cooked = fg_hip.cook_q8_0(packed, width, rows)
    x = rng.normal(0, 1, (tokens, width)).astype(np.float32)
    y = plain(dev, cooked, x, width, rows, 1.0)
    sample = np.unique(np.concatenate([rng.choice(rows, 500), np.arange(40), rows - 1 - np.arange(40)]))
    check_f64(y, packed, x, width, rows, 1.0, sample=sample)
    sl = fg_hip.OutputSlice(rows, 1, 0, rows, tokens)
    v, i, s, _ = fused(dev, sl, cooked, x, width, logits=False)
    wv, wi, ws = O.slice_finalists(y, 0)
    assert np.array_equal(i, wi) and np.array_equal(v.view(np.uint32), wv.view(np.uint32))
    # The bits of the form's fewest tokens (another shape).
    n = 1 if tokens <= 8 else 9
    assert np.array_equal(plain(dev, cooked, x[:n], width, rows, 1.0).view(np.uint32),
                          y[:n].view(np.uint32))


@pytest.mark.parametrize("tokens", [1, 5, 8, 9, 16, 33, 64])
@pytest.mark.parametrize("width,rows", [(96, 40), (2560, 64), (6944, 20), (8192, 17)])
def test_low_parts_decide(dev, tokens, width, rows):
    """Inputs in pairs that differ in their lowest 8 bits alone, against weights
    that cancel the rest, in one block at a time: what is left is the low parts'
    sum, about 4e-6 of the magnitudes, so that one lost in any slice shows."""
    rng = np.random.default_rng(tokens * 7 + width)
    blocks = width // 32
    b = packed_random(rng, width, rows).reshape(rows, blocks, 34)
    q = rng.integers(1, 128, (rows, blocks, 16), dtype=np.int8)
    b[:, :, 2::2] = q.view(np.uint8)
    b[:, :, 3::2] = (-q).view(np.uint8)
    packed = b.reshape(-1)
    cooked = fg_hip.cook_q8_0(packed, width, rows)
    for at in np.unique([0, blocks // 3, blocks // 2, blocks - 2, blocks - 1]):
        base = np.uint32(0x3f800000) | rng.integers(0, 1 << 15, (tokens, 16), dtype=np.uint32) << 8
        x = np.zeros((tokens, width), dtype=np.float32)
        x[:, 32 * at + 1:32 * at + 32:2] = base.view(np.float32)
        x[:, 32 * at:32 * at + 32:2] = (
            base | rng.integers(64, 256, (tokens, 16), dtype=np.uint32)).view(np.float32)
        y = plain(dev, cooked, x, width, rows, 1.0)
        want, mag = O.dense_q8_0_f64(packed, x, width, rows, 1.0)
        assert np.all(want > 3e-6 * mag)
        assert np.all(np.abs(y - want) <= 1e-7 * mag), (at, np.max(np.abs(y - want) / mag))


@pytest.mark.parametrize("width,rows", [(32, 3), (96, 700), (160, 131_073), (6944, 33)])
def test_weights_off_the_lines(dev, width, rows):
    """Weights 16-byte aligned but not on a cache line: the same bits."""
    import torch
    rng = np.random.default_rng(width)
    packed = packed_random(rng, width, rows)
    cooked = fg_hip.cook_q8_0(packed, width, rows)
    x = rng.normal(0, 1, (3, width)).astype(np.float32)
    want = plain(dev, cooked, x, width, rows, 1.0)
    for at in (16, 80):
        buf = torch.zeros(len(cooked) + 128, dtype=torch.uint8, device=dev)
        w = buf[at:at + len(cooked)]
        w.copy_(torch.from_numpy(cooked))
        y = torch.empty(3 * rows, dtype=torch.float32, device=dev)
        fg_hip.dense_q8_0_cooked(y, w, torch.from_numpy(x).to(dev), width, rows, 3, 1.0)
        assert np.array_equal(y.cpu().numpy().view(np.uint32).reshape(3, rows), want.view(np.uint32))


@pytest.mark.parametrize("tokens", [2, 8, 12, 64])
def test_extreme_inputs(dev, tokens):
    """Non-finite inputs reach only their own token, with IEEE results; inputs
    from 1e-30 to 1e30 keep the f32 product's accuracy."""
    rng = np.random.default_rng(tokens)
    width, rows = 320, 100
    packed = packed_random(rng, width, rows)
    cooked = fg_hip.cook_q8_0(packed, width, rows)
    x = (rng.normal(0, 1, (tokens, width)) * 10.0 ** rng.uniform(-30, 30, (tokens, width))).astype(np.float32)
    check_f64(plain(dev, cooked, x, width, rows, 1.0), packed, x, width, rows, 1.0)
    x = rng.normal(0, 1, (tokens, width)).astype(np.float32)
    clean = plain(dev, cooked, x, width, rows, 1.0)
    bad = x.copy()
    bad[1, 7] = np.inf
    bad[-1, 40] = np.uint32(0x7f800001).view(np.float32)  # a NaN with a low payload
    y = plain(dev, cooked, bad, width, rows, 1.0)
    q = packed.reshape(rows, width // 32, 34)[:, 0, 2 + 7].view(np.int8)
    if tokens > 2:
        assert np.array_equal(y[0].view(np.uint32), clean[0].view(np.uint32))
        want = np.where(q > 0, np.inf, np.where(q < 0, -np.inf, np.nan)).astype(np.float32)
        assert np.array_equal(np.isnan(y[1]), np.isnan(want))
        assert np.array_equal(y[1][~np.isnan(want)], want[~np.isnan(want)])
    assert np.all(np.isnan(y[-1]))


@pytest.mark.parametrize("tokens", [1, 2, 8, 9, 17, 33, 64, 66])
@pytest.mark.parametrize("width,rows", [(96, 40), (2560, 150), (8192, 17)])
def test_tiny_inputs(dev, tokens, width, rows):
    """Inputs whose bits reach below the smallest subnormal bf16 (from about
    1e-33 down to f32's subnormals) keep the f32 product's accuracy: within the
    tolerance above of the token's own sum of magnitudes, besides the rounding
    of a subnormal result (2^-150, below 1e-45).  One tiny input, in the last
    block, is enough; the tokens beside such ones keep their bits, the fused
    finalist carries the plain values."""
    rng = np.random.default_rng(tokens + width)
    packed = packed_random(rng, width, rows, 0.25, 1.0)
    cooked = fg_hip.cook_q8_0(packed, width, rows)
    for first in (0, 1):
        x = rng.normal(0, 1, (tokens, width)).astype(np.float32)
        clean = plain(dev, cooked, x, width, rows, 0.75)
        tiny = np.arange(first, tokens, 2)
        for j, t in enumerate(tiny):
            x[t] *= np.float32(10.0 ** -[33, 34, 36, 38, 39, 41][j % 6])
            if j % 4 == 3:  # all zero but the last block
                x[t, :-32] = 0
        y = plain(dev, cooked, x, width, rows, 0.75)
        check_f64(y, packed, x, width, rows, 0.75, floor=1e-45)
        others = np.arange(1 - first, tokens, 2)
        assert np.array_equal(y[others].view(np.uint32), clean[others].view(np.uint32))
        if len(others):  # a normal token with one tiny input
            x[others[0], -1] = np.float32(1.1e-38)
            y = plain(dev, cooked, x, width, rows, 1.0)
            check_f64(y, packed, x, width, rows, 1.0, floor=1e-45)
        else:
            y = plain(dev, cooked, x, width, rows, 1.0)
        sl = fg_hip.OutputSlice(rows, 1, 0, rows, tokens)
        v, i, s, _ = fused(dev, sl, cooked, x, width, logits=False)
        wv, wi, ws = O.slice_finalists(y, 0)
        assert np.array_equal(i, wi) and np.array_equal(v.view(np.uint32), wv.view(np.uint32))
        assert np.array_equal(s, ws)


@pytest.mark.parametrize("tokens", [1, 8, 64])
def test_captured_calls_replay(dev, tokens):
    """The three forms captured in a graph and replayed over new inputs, with
    eager calls between the replays."""
    import torch
    rng = np.random.default_rng(tokens)
    width, vocab = 256, 5_000
    cooked = torch.from_numpy(fg_hip.cook_q8_0(packed_random(rng, width, vocab), width, vocab)).to(dev)
    x = torch.zeros((tokens, width), device=dev)
    u = torch.full((tokens,), 0.4, device=dev)
    cfg = [fg_hip.make_config(0.8, 0.9, 20)] * tokens
    sl = fg_hip.OutputSlice(vocab, 1, 0, vocab, tokens)

    def outputs():
        return (torch.empty((tokens, vocab), device=dev),
                *(torch.empty(tokens, dtype=d, device=dev)
                  for d in (torch.float32, torch.int32, torch.int32) * 2))

    def run(o):
        stream = torch.cuda.current_stream().cuda_stream
        fg_hip.dense_q8_0_cooked(o[0], cooked, x, width, vocab, tokens, scale=0.02, stream=stream)
        sl.run_dense(cooked, x, width, tokens, o[1], o[2], o[3], scale=0.02, stream=stream)
        sl.run_dense_sampled(cooked, x, width, tokens, cfg, u, o[5], o[4], o[6], scale=0.02,
                             stream=stream)

    kept, eager = outputs(), outputs()
    run(eager)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(kept)
    for replay in range(4):
        x.copy_(torch.from_numpy(rng.normal(0, 1, (tokens, width)).astype(np.float32)))
        graph.replay()
        run(eager)
        torch.cuda.synchronize()
        for a, b in zip(kept, eager):
            assert torch.equal(a.view(torch.int32), b.view(torch.int32)), replay
