"""Top-p rows without a top-k or min-p: chunk candidates with their mass
certificate, and the whole-row finish behind them, against the oracle
(nucleus_mask, crates/app/cli/src/qwen_forward.rs:474-549).  Statuses, kept
sets, adjusted logits and tokens are bit-exact."""
import numpy as np
import pytest

from helpers import compare, run_gpu

pytestmark = pytest.mark.gpu

LARGE = 11   # MXS_PATH_LARGE


@pytest.fixture(scope="module")
def torch_mod():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def text_row(rng, V, fall, spread=2.5):
    x = (spread * rng.standard_normal(V)).astype(np.float32)
    n = min(4096, max(1, V // 2))
    ids = rng.choice(V, n, replace=False)
    x[ids] = np.maximum(x[ids], 20.0 - fall * np.log(np.arange(1, n + 1))).astype(np.float32)
    return x


def rows_of(kind, rng, R, V):
    if kind == "text":       # nuclei of a few to thousands of tokens
        return np.stack([text_row(rng, V, 1.1 + 0.4 * (r % 8)) for r in range(R)])
    if kind == "flat":       # nuclei of most of the row
        return (0.5 + 0.5 * (np.arange(R)[:, None] % 4)).astype(np.float32) * rng.standard_normal((R, V)).astype(np.float32)
    if kind == "steps":      # crowded bins: a few values, each thousands of times
        v = rng.standard_normal((R, 7)).astype(np.float32)
        return v[np.arange(R)[:, None], rng.integers(0, 7, (R, V))]
    if kind == "one_head":   # all head mass in one chunk, the others flat
        x = rng.standard_normal((R, V)).astype(np.float32)
        x[:, : max(1, V // 40)] += 9.0
        return x
    if kind == "lowest":     # most tokens at the lowest finite value
        x = np.full((R, V), np.finfo(np.float32).min, dtype=np.float32)
        n = min(V, 300)
        for r in range(R):
            x[r, rng.choice(V, n, replace=False)] = rng.standard_normal(n)
        return x
    raise ValueError(kind)


def batch(kind, R, V, bf16=False, history=0, bias=0, mask=False, seed=0):
    from metallix_amd.synth import Batch, bf16_bits_to_f32, to_bf16_bits

    rng = np.random.default_rng([R, V, seed])
    x = rows_of(kind, rng, R, V)
    bits = None
    if bf16:
        bits = to_bf16_bits(x)
        x = bf16_bits_to_f32(bits)
    b = Batch(name=f"nucleus-{kind}", logits=x, temperature=rng.uniform(0.5, 1.5, R), uniform=rng.random(R),
              top_p=np.array([0.05, 0.5, 0.9, 0.95, 0.99, 0.9999, 1.0 - 1e-9, 0.8])[np.arange(R) % 8], bf16_bits=bits,
              tokenizer_vocab=V)
    if history:
        b.history_offsets = (np.arange(R + 1) * history).astype(np.uint32)
        b.history_ids = rng.integers(0, V, R * history).astype(np.uint32)
        b.repetition = np.where(np.arange(R) % 2, 1.2, 0.9).astype(np.float32)
        b.presence = np.full(R, 0.4, dtype=np.float32)
        b.frequency = np.full(R, 0.1, dtype=np.float32)
    if bias:
        b.bias_offsets = (np.arange(R + 1) * bias).astype(np.uint32)
        b.bias_ids = np.concatenate([np.sort(rng.choice(V, bias, replace=False)) for _ in range(R)]).astype(np.uint32)
        vals = rng.uniform(-3, 3, R * bias).astype(np.float32)
        vals[::5] = -np.inf
        b.bias_values = vals
    if mask:
        words = (V + 31) // 32
        m = rng.integers(0, 2 ** 32, (R, words), dtype=np.uint64).astype(np.uint32)
        m[::2] &= rng.integers(0, 2 ** 32, (len(m[::2]), words), dtype=np.uint64).astype(np.uint32)
        m[:, 0] |= 1
        b.mask_words = m
        b.tokenizer_vocab = max(1, V - 5)
    return b


CASES = [
    # (kind, rows, vocab, options): the chunk and segment edges of the layout
    ("text", 8, 1, {}), ("text", 8, 5, {}), ("text", 8, 4097, {}), ("text", 8, 40963, {}),
    ("text", 16, 151936, {}), ("text", 72, 50257, dict(bf16=True)), ("text", 8, 262144, {}),
    ("text", 8, 100003, dict(history=700)), ("text", 8, 100003, dict(history=300, bias=40)),
    ("text", 16, 151936, dict(mask=True)), ("text", 8, 70001, dict(bf16=True, mask=True, history=50)),
    ("flat", 8, 151936, {}), ("flat", 8, 50257, dict(bf16=True)), ("flat", 8, 262144, {}),
    ("flat", 8, 99999, dict(history=3000, bias=7)), ("flat", 8, 151936, dict(mask=True, bf16=True)),
    ("one_head", 8, 151936, {}), ("one_head", 8, 65541, dict(bias=3)),
    ("lowest", 8, 151936, {}), ("lowest", 8, 30011, dict(bias=25)),
]


@pytest.mark.parametrize("kind,R,V,opt", CASES, ids=lambda v: str(v))
def test_nucleus_rows(torch_mod, orc, kind, R, V, opt):
    from metallix_amd import Sampler

    b = batch(kind, R, V, **opt)
    print(f"case nucleus {kind} rows {R} vocab {V} {opt}", flush=True)
    s = Sampler(max_rows=R, max_vocab=V)
    gpu = run_gpu(torch_mod, s, b)
    s.close()
    # top_p = 1 - 1e-9 cuts among weights near the f64 sums' error bound: only
    # such a row may report status 1
    unc = np.nonzero(gpu["status"] == 1)[0]
    assert (b.top_p[unc] > 0.99999).all(), (unc, b.top_p[unc])
    compare(b, gpu, orc.sample_batch(b, debug=True), allow_uncertified=len(unc))


@pytest.mark.parametrize("V,bf16", [(20000, False), (151936, True)])
def test_crowded_bins(torch_mod, orc, V, bf16):
    """Seven values per row, thousands of tokens each: the cut lies among
    equal keys (cut by their count and ID).  A prefix sum that equals theta
    to within the bound is the only uncertified case, and these have none."""
    from metallix_amd import Sampler

    b = batch("steps", 8, V, bf16=bf16, seed=3)
    s = Sampler(max_rows=8, max_vocab=V)
    print(f"case nucleus steps vocab {V} bf16 {bf16}", flush=True)
    gpu = run_gpu(torch_mod, s, b)
    s.close()
    compare(b, gpu, orc.sample_batch(b, debug=True))


def test_paths(torch_mod, orc):
    """A peaked batch is decided from its candidates, a flat one over the
    whole row; results are the same through either (the two above)."""
    from helpers import to_device
    from metallix_amd import Sampler

    torch, V = torch_mod, 151936
    s = Sampler(max_rows=8, max_vocab=V)
    buf = torch.zeros(8, dtype=torch.int32, device="cuda")
    s.lib.mxs_debug_set_paths(s.ctx, buf.data_ptr())
    for kind, large in (("text", False), ("flat", True)):
        b = batch(kind, 8, V)
        b.top_p, b.temperature = np.full(8, 0.9), np.full(8, 0.6)
        if kind == "text":
            b.logits = np.stack([text_row(np.random.default_rng(r), V, 2.5) for r in range(8)])
        logits, kw = to_device(torch, b)
        s.sample(logits, **kw)
        torch.cuda.synchronize()
        got = buf.cpu().numpy()
        assert ((got == LARGE) == large).all(), (kind, got)
    s.lib.mxs_debug_set_paths(s.ctx, None)
    s.close()


def clustered(rng, R, V, total, share):
    """Mask words with `total` legal tokens per row, `share` of them in one run."""
    legal = np.zeros((R, (V + 31) // 32 * 32), dtype=bool)
    run = int(total * share)
    for r in range(R):
        legal[r, rng.choice(V, total - run, replace=False)] = True
        s = int(rng.integers(0, V - run + 1))
        legal[r, s:s + run] = True
    return np.packbits(legal.reshape(R, -1, 32), axis=-1, bitorder="little").view(np.uint32).reshape(R, -1)


# Legal tokens that lie in few of a row's chunks: up to 8192 of them (the
# finisher's cache) every chunk lists its own whatever its share, beyond that
# every chunk thins its list and sums its mass.
@pytest.mark.parametrize("kind", ["text", "flat"])
@pytest.mark.parametrize("V,total,share", [(151936, 1000, 1.0), (151936, 3000, 0.55), (151936, 4000, 1.0), (151936, 8192, 0.9),
                                           (151936, 9000, 0.5), (40000, 12000, 1.0), (262144, 3000, 0.55), (20011, 3500, 0.7), (20011, 10000, 0.5)])
def test_clustered_masks(torch_mod, orc, kind, V, total, share):
    from helpers import to_device
    from metallix_amd import Sampler

    R = 8
    b = batch(kind, R, V, bf16=kind == "flat", seed=7)
    b.top_p = np.array([0.05, 0.5, 0.8, 0.9, 0.95, 0.95, 0.99, 0.999])
    b.mask_words, b.tokenizer_vocab = clustered(np.random.default_rng(total), R, V, total, share), V - 3
    print(f"case nucleus clustered {kind} vocab {V} legal {total} share {share}", flush=True)
    s = Sampler(max_rows=R, max_vocab=V)
    compare(b, run_gpu(torch_mod, s, b), orc.sample_batch(b, debug=True))
    if total <= 4000:   # ... and such rows stay within the finisher's LDS working set
        buf = torch_mod.zeros(R, dtype=torch_mod.int32, device="cuda")
        s.lib.mxs_debug_set_paths(s.ctx, buf.data_ptr())
        logits, kw = to_device(torch_mod, b)
        s.sample(logits, **kw)
        torch_mod.cuda.synchronize()
        assert (buf.cpu().numpy() != LARGE).all(), buf.cpu().numpy()
        s.lib.mxs_debug_set_paths(s.ctx, None)
    s.close()


@pytest.mark.parametrize("opt", [{}, dict(bf16=True, mask=True), dict(history=300, bias=5), dict(history=40, mask=True)],
                         ids=lambda v: "-".join(v) or "plain")
def test_export_of_top_p_rows(torch_mod, orc, opt):
    """What a top-p row exports: a list that holds its nucleus where the chunks'
    candidates decided it, none where the whole row did, and every legal token
    (or the top `width` of them, ties by ID) of an uncertified row.  Rows 2 and 3
    are flat; row 3's top_p puts the cut among weights below the f64 sums'
    error bound, so it is uncertified."""
    from metallix_amd import Sampler

    R, V = 4, 40003
    b = batch("text", R, V, seed=11, **opt)
    flat = batch("flat", R, V, seed=11, **opt)
    b.logits[2:] = flat.logits[2:]
    if b.bf16_bits is not None:
        b.bf16_bits[2:] = flat.bf16_bits[2:]
    b.temperature, b.top_p = np.full(R, 0.8), np.array([0.5, 0.6, 0.999, 1.0 - 1e-15])
    ref = orc.sample_batch(b, debug=True)
    legal = np.ones((R, V), dtype=bool)
    if b.mask_words is not None:
        legal = np.unpackbits(b.mask_words.view(np.uint8), axis=1, bitorder="little")[:, :V].astype(bool)
        legal[:, b.tokenizer_vocab:] = False
    print(f"case export vocab {V} {opt}", flush=True)
    s = Sampler(max_rows=R, max_vocab=V)
    gpu = run_gpu(torch_mod, s, b)
    assert list(gpu["status"]) == [0, 0, 0, 1], gpu["status"]
    compare(b, gpu, ref, allow_uncertified=1)
    for width in (V, 3000):
        cnt, ids, lg = (t.cpu().numpy() for t in s.export_candidates(R, width))
        assert cnt[2] == -1
        for r in (0, 1, 3):
            i, l = ids[r, :cnt[r]], lg[r, :cnt[r]]
            assert np.array_equal(l.view(np.uint32), ref["adjusted"][r][i].view(np.uint32)) and legal[r, i].all()
            assert (np.diff(i) > 0).all()
            if r == 3:
                all_ids = np.nonzero(legal[r])[0]
                order = np.lexsort((all_ids, -ref["adjusted"][r][all_ids].astype(np.float64)))[:width]
                assert np.array_equal(i, np.sort(all_ids[order])), (width, len(i))
            elif width == V:
                assert np.isin(np.nonzero(ref["kept"][r])[0], i).all()
    s.close()


def crowded(rng, R, V, levels):
    """N(0, 0.3^2), or two levels whose second is spread over a few thousand ulps."""
    if not levels:
        return (0.3 * rng.standard_normal((R, V))).astype(np.float32)
    x = (np.float32(1.0) + rng.integers(0, 4000, (R, V)).astype(np.float32) * np.float32(2.0 ** -23)).astype(np.float32)
    top = rng.random((R, V)) < 0.02
    return np.where(top, np.float32(4.0) + rng.standard_normal((R, V)).astype(np.float32) * np.float32(0.1), x).astype(np.float32)


# Cuts inside a mass bin (1/64 octave) that holds more than the 4096 tokens the
# whole-row finish sorts, at distinct keys: N(0, 0.3^2) at T 4 to 20 puts V / 100
# tokens and more in a bin; the second level of the two-level rows is one bin.
# top_p cuts far from the f64 sums' error bound (1e-11 of the row): status 0, the
# exact kept set.
@pytest.mark.parametrize("levels,bf16,history", [(False, False, 0), (False, True, 0), (False, False, 300), (True, False, 0),
                                                 (True, False, 300)])
@pytest.mark.parametrize("V", [151936, 262144])
def test_crowded_distinct_keys(torch_mod, orc, V, levels, bf16, history):
    from metallix_amd import Sampler
    from metallix_amd.synth import bf16_bits_to_f32, to_bf16_bits

    R = 4
    b = batch("flat", R, V, bf16=bf16, history=history, seed=13)
    b.logits = crowded(np.random.default_rng([V, levels, bf16]), R, V, levels)
    if bf16:
        b.bf16_bits = to_bf16_bits(b.logits)
        b.logits = bf16_bits_to_f32(b.bf16_bits)
    b.temperature, b.top_p = np.array([4.0, 8.0, 20.0, 5.0]), np.array([0.3, 0.5, 0.9, 0.7])
    print(f"case nucleus crowded vocab {V} levels {levels} bf16 {bf16} history {history}", flush=True)
    s = Sampler(max_rows=R, max_vocab=V)
    gpu = run_gpu(torch_mod, s, b)
    assert (gpu["status"] == 0).all(), gpu["status"]
    compare(b, gpu, orc.sample_batch(b, debug=True))
    s.close()
