"""GPU parity of the encoder forward (manta_rocm_encoder_pooled) against the
CPU oracle's restatement of examples/encoder_trainable_q8.manta
(embed_pooled_batch).  Bar: per-row cosine >= 0.9999 with the oracle's f32
embedding and max abs error below 2e-3 (the device output is f16; the
device's reductions run in tree order)."""
import numpy as np
import pytest

from manta_amd._lib import MantaRocmError
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _pack_cols(w):
    """q8 with an f32 scale per column: code = round(w / s), s = maxabs / 127."""
    s = (np.abs(w).max(0) / 127.0).astype(np.float32)
    s[s == 0] = 1.0
    codes = np.clip(np.round(w / s), -127, 127).astype(np.int8)
    return codes, s


def _case(seed, b, t, vocab, d, h, empty_row=True):
    rng = np.random.default_rng(seed)
    tokens = rng.integers(0, vocab, size=(b, t), dtype=np.int32)
    lengths = rng.integers(1, t + 1, size=b)
    if empty_row:
        lengths[0] = 0  # a fully masked sequence pools to zeros
    mask = (np.arange(t)[None, :] < lengths[:, None]).astype(np.int32)
    table = (rng.standard_normal((vocab, d)) * 0.5).astype(np.float32)
    tcodes, tscales = orc.pack_q8_rows(table)
    ws = [(rng.standard_normal(s) / np.sqrt(s[0])).astype(np.float32)
          for s in [(d, d), (d, d), (d, d), (d, d), (d, h), (h, d)]]
    packed = [_pack_cols(w) for w in ws]
    return tokens, mask, tcodes, tscales, packed


def _run(rt, tokens, mask, tcodes, tscales, packed):
    dev = [(rt.to_device(c), rt.to_device(s)) for c, s in packed]
    out = rt.encoder_pooled(rt.to_device(tokens), rt.to_device(mask), rt.to_device(tcodes), rt.to_device(tscales),
                            dev)
    return out.download().view(np.float16).astype(np.float32)


def _want(tokens, mask, tcodes, tscales, packed):
    table = (tcodes.astype(np.float32) * tscales[:, None]).astype(np.float32)
    ws = [(c.astype(np.float32) * s[None, :]).astype(np.float32) for c, s in packed]
    return orc.encoder_pooled(tokens, mask, table, *ws)


@pytest.mark.parametrize("b,t,vocab,d,h", [(6, 16, 50, 64, 128), (5, 24, 70, 96, 160), (3, 1, 9, 32, 64),
                                           # d and h multiples of 128: the weight GEMMs on f16 MFMA (the
                                           # second with 120 rows, not a multiple of the 64-row tiles)
                                           (8, 64, 300, 384, 1536), (3, 40, 100, 128, 384),
                                           # d, h and t not multiples of 16: the scalar staging path of the
                                           # q8-weight and transposed-K GEMMs, with their bounds-checked K tails
                                           (4, 24, 40, 40, 72)])
def test_encoder_matches_oracle(rt, b, t, vocab, d, h):
    case = _case(b * 100 + t, b, t, vocab, d, h)
    got = _run(rt, *case)
    want = _want(*case)
    assert np.all(got[0] == 0.0) and np.all(want[0] == 0.0)  # the fully masked row
    live = np.linalg.norm(want, axis=1) > 0
    cos = (got[live] * want[live]).sum(1) / (np.linalg.norm(got[live], axis=1) * np.linalg.norm(want[live], axis=1))
    assert cos.min() >= 0.9999, cos.min()
    assert np.abs(got - want).max() < 2e-3


def test_encoder_token_out_of_range_is_reported(rt):
    tokens, mask, tcodes, tscales, packed = _case(7, 2, 8, 10, 32, 64, empty_row=False)
    tokens[1, 3] = 10
    dev = [(rt.to_device(c), rt.to_device(s)) for c, s in packed]
    rt.encoder_pooled(rt.to_device(tokens), rt.to_device(mask), rt.to_device(tcodes), rt.to_device(tscales), dev)
    with pytest.raises(MantaRocmError, match="gather index 10 out of range"):
        rt.synchronize()


def _run_layers(rt, layers, tokens, mask, tcodes, tscales, packed):
    dev = [(rt.to_device(c), rt.to_device(s)) for c, s in packed]
    out = rt.encoder_pooled(rt.to_device(tokens), rt.to_device(mask), rt.to_device(tcodes), rt.to_device(tscales),
                            dev, layers=layers)
    return out


def _want_layers(layers, tokens, mask, tcodes, tscales, packed):
    table = (tcodes.astype(np.float32) * tscales[:, None]).astype(np.float32)
    ws = [(c.astype(np.float32) * s[None, :]).astype(np.float32) for c, s in packed]
    return orc.encoder_pooled(tokens, mask, table, *ws, layers=layers)


@pytest.mark.parametrize("b,t,vocab,d,h", [(6, 16, 50, 64, 128), (8, 64, 300, 384, 1536), (4, 24, 40, 40, 72)])
def test_two_layer_encoder_matches_oracle(rt, b, t, vocab, d, h):
    """encoder_trainable_q8x2 (the block twice, shared weights) at the same
    bar as one layer."""
    case = _case(b * 77 + t, b, t, vocab, d, h)
    got = _run_layers(rt, 2, *case).download().view(np.float16).astype(np.float32)
    want = _want_layers(2, *case)
    assert np.all(got[0] == 0.0) and np.all(want[0] == 0.0)
    live = np.linalg.norm(want, axis=1) > 0
    cos = (got[live] * want[live]).sum(1) / (np.linalg.norm(got[live], axis=1) * np.linalg.norm(want[live], axis=1))
    assert cos.min() >= 0.9999, cos.min()
    assert np.abs(got - want).max() < 2e-3
    one = _run_layers(rt, 1, *case).download().view(np.float16).astype(np.float32)
    assert np.abs(one - got).max() > 1e-2  # the second block ran


@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("b,t,vocab,d,h", [
    # 256-row tiles with several sequences' shares in a 64-row slab, and a
    # last tile that is not full
    (4100, 8, 60, 128, 128),
    # 64-row tiles: one row, sequences that cross slabs, one to five blocks of
    # 64 positions (the last past the fused attention), d past the fused layernorm
    (1, 1, 9, 128, 128), (3, 31, 50, 256, 384), (2, 70, 50, 256, 128), (3, 130, 80, 128, 256), (2, 200, 60, 384, 128),
    (2, 257, 40, 128, 128), (2, 33, 40, 512, 128), (1, 20, 30, 640, 256)])
def test_encoder_f16_tile_edges(rt, b, t, vocab, d, h, layers):
    """The f16 weight path at the edges of its tiles, slabs and fused forms,
    at the bar above."""
    if b * t > 10000 and layers > 1:
        layers = 1  # the oracle's time
    case = _case(b * 31 + t, b, t, vocab, d, h, empty_row=b > 1)
    got = _run_layers(rt, layers, *case).download().view(np.float16).astype(np.float32)
    want = _want_layers(layers, *case)
    live = np.linalg.norm(want, axis=1) > 0
    assert np.all(got[~live] == 0.0)
    cos = (got[live] * want[live]).sum(1) / (np.linalg.norm(got[live], axis=1) * np.linalg.norm(want[live], axis=1))
    assert cos.min() >= 0.9999, cos.min()
    assert np.abs(got - want).max() < 2e-3


def test_encoder_output_feeds_score_topk(rt):
    """The encoder's device output is the query matrix of the fused score +
    top-k with no host round trip; the result equals the reference scoring
    of those embeddings (cosineRows on the dequantized candidates)."""
    from manta_amd import synth
    b, t, vocab, d, h = 16, 32, 200, 128, 256
    case = _case(91, b, t, vocab, d, h, empty_row=False)
    emb = _run_layers(rt, 2, *case)  # f16 [b, d] on device
    codes, scales = synth.q8_rows(91, 5, 20000, d, normalize=True)
    cands = rt.bind_q8(codes, scales)
    ids, scores, _ = rt.score_topk(cands, "cosine", emb, 25)
    q = emb.download()
    ref = orc.cosine_rows(orc.f16_to_f32(q), orc.dequant_q8(codes, scales))
    want = orc.topk(ref, 25)
    np.testing.assert_array_equal(ids.download(), want)
    np.testing.assert_array_equal(scores.download(), np.take_along_axis(ref, want, 1))


def _exact_layers(layers, tokens, mask, tcodes, tscales, packed, r=lambda x: x):
    """The forward in 64 bits; r: what the operands of the weight products and
    the output are rounded by."""
    y = tcodes[tokens].astype(np.float64) * tscales[tokens].astype(np.float64)[..., None]
    w = [c.astype(np.float64) * s.astype(np.float64)[None, :] for c, s in packed]

    def layernorm(x):
        x = x - x.mean(-1, keepdims=True)
        return x / np.sqrt((x * x).mean(-1, keepdims=True) + 1e-5)

    for _ in range(layers):
        q, k, v = (r(y) @ w[i] for i in range(3))
        s = q @ k.transpose(0, 2, 1)
        p = np.exp(s - s.max(-1, keepdims=True))
        hid = layernorm(r((p / p.sum(-1, keepdims=True)) @ v) @ w[3] + y)
        up = r(hid) @ w[4]
        up = 0.5 * up * (1.0 + np.tanh(0.7978845608 * (up + 0.044715 * up ** 3)))
        y = layernorm(r(up) @ w[5] + hid)
    y /= np.linalg.norm(y, axis=-1, keepdims=True)
    m = mask[..., None].astype(np.float64)
    return r((y * m).sum(1) / np.maximum(m.sum(1), 1.0))


@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("b,t,d,h", [(9, 33, 384, 1536), (40, 64, 256, 512), (3, 200, 128, 512), (512, 64, 384, 256),
                                     (7, 40, 512, 256)])
def test_encoder_repeats_and_stays_near_64_bits(rt, b, t, d, h, layers):
    """The same call gives the same bits among calls on other inputs, and its
    error against 64 bits stays that of its roundings to f16 (the products'
    left operands and the output): at most 1.5 times what the same roundings
    leave of a forward that is otherwise in 64 bits.  The f32 steps round 2^13
    times finer; what they add is to move a few of those roundings."""
    case, other = _case(b + t, b, t, 500, d, h), _case(b + t + 1, b, t, 500, d, h)
    got = [_run_layers(rt, layers, *c).download() for c in (case, other, case, case, other, case)]
    for i in (2, 3, 5):
        np.testing.assert_array_equal(got[i], got[0])
    np.testing.assert_array_equal(got[4], got[1])
    want = _exact_layers(layers, *case)
    rounded = _exact_layers(layers, *case, r=lambda x: x.astype(np.float16).astype(np.float64))
    off = np.linalg.norm(got[0].view(np.float16).astype(np.float64) - want)
    assert off <= 1.5 * np.linalg.norm(rounded - want), off / np.linalg.norm(want)


class _At:
    """A device array's memory at an odd address."""

    def __init__(self, array, shape, dtype, offset):
        self.array, self.shape, self.dtype = array, shape, dtype
        self.addr = array.addr + offset


@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("d,h,t", [(384, 256, 33), (128, 128, 64), (512, 128, 20), (96, 64, 20)])
def test_encoder_unaligned_table(rt, d, h, t, layers):
    """Token rows that do not begin on 16 bytes: the same bits (the fused
    gather and residual take aligned rows only)."""
    tokens, mask, tcodes, tscales, packed = _case(d + t, 5, t, 60, d, h)
    want = _run_layers(rt, layers, tokens, mask, tcodes, tscales, packed).download()
    dev = [(rt.to_device(c), rt.to_device(s)) for c, s in packed]
    tok, msk, sc = rt.to_device(tokens), rt.to_device(mask), rt.to_device(tscales)
    for offset in (1, 8):
        padded = np.concatenate([np.zeros(offset, np.int8), tcodes.reshape(-1)])
        table = _At(rt.to_device(padded), tcodes.shape, tcodes.dtype, offset)
        got = rt.encoder_pooled(tok, msk, table, sc, dev, layers=layers).download()
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("b,t,d,h", [(5, 40, 384, 256), (4100, 8, 128, 128), (3, 20, 512, 128), (3, 20, 96, 64)])
def test_encoder_overflowing_variance(rt, b, t, d, h, layers):
    """Rows whose layernorm variance overflows in f32 are zero after it, and
    stay zero through the normalize and the pool (finite deviations)."""
    tokens, mask, tcodes, tscales, packed = _case(b + t + d, b, t, 50, d, h)
    packed[5] = (packed[5][0], packed[5][1] * np.float32(1e22))
    got = _run_layers(rt, layers, tokens, mask, tcodes, tscales, packed).download().view(np.float16)
    n = min(b, 5)  # (the oracle's time)
    want = _want_layers(layers, tokens[:n], mask[:n], tcodes, tscales, packed)
    assert np.all(want == 0.0)
    assert np.all(got == 0.0)
