"""Device sampling step (rwkv_sample_logits through chatrwkv_amd.sampling) against the oracle's restatement of
rwkv/utils.py:55-88, 103-123."""
import os
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
from oracle import sampling as osamp  # noqa: E402

pytestmark = pytest.mark.gpu
G = os.path.join(ROOT, "tests", "golden")
DEV = "cuda:0"


def logits_for(case_index, vocab, scale):
    rng = np.random.Generator(np.random.PCG64([case_index, 0x5A11]))
    return (rng.standard_normal(vocab) * scale).astype(np.float32)


def _boundary_margin(x, top_p, temperature):
    """Distance of top_p from the nearest cumulative sum of the sorted probabilities: a cut closer than fp32
    summation noise may legitimately land one entry to either side."""
    if temperature == 0 or top_p <= 0:
        return 1.0
    p = np.sort(osamp.softmax32(x).astype(np.float64))[::-1]
    return float(np.abs(np.cumsum(p) - top_p).min())


def _check_probs(got, ref, margin):
    kept_g, kept_r = got > 0, ref > 0
    if margin > 1e-5:
        assert np.array_equal(kept_g, kept_r), (kept_g.sum(), kept_r.sum())
    else:
        assert abs(int(kept_g.sum()) - int(kept_r.sum())) <= 1
    both = kept_g & kept_r
    np.testing.assert_allclose(got[both], ref[both], rtol=2e-4, atol=1e-12)


def test_filter_matches_oracle_on_golden_cases():
    from chatrwkv_amd.sampling import Sampler
    g = np.load(os.path.join(G, "sampler.npz"))
    for ci, (V, scale, temp, top_p, top_k) in enumerate(g["cases"]):
        V = int(V)
        x = logits_for(ci, V, float(scale))
        s = Sampler(V, device=DEV)
        xt = torch.from_numpy(x).to(DEV)
        ref = osamp.filter_probs(x, temperature=float(temp), top_p=float(top_p), top_k=int(top_k)).astype(np.float64)
        margin = _boundary_margin(x, float(top_p), float(temp))
        for u in (0.0, 0.137, 0.5, 0.731, 0.9999):
            tok = int(s.sample(xt, float(temp), float(top_p), int(top_k), u=u, penalties=False))
            got = s.probs.cpu().numpy().astype(np.float64)
            _check_probs(got, ref, margin)
            # the draw: inverse CDF of the device's own filtered vector, recomputed on the host in fp64
            cdf = np.cumsum(got)
            want = osamp.choose(got, u)
            if tok != want:  # fp32 running sums on the device: only an entry adjacent in the CDF may differ
                t = u * cdf[-1]
                assert got[tok] > 0 and abs(cdf[tok] - got[tok] - t) <= 1e-5 * cdf[-1] + 1e-12 or abs(cdf[want] - t) <= 1e-5 * cdf[-1], \
                    (ci, u, tok, want)
            assert ref[tok] > 0 or margin <= 1e-5


def test_temperature_zero_is_argmax_and_top_p_zero():
    from chatrwkv_amd.sampling import Sampler, sample_logits
    x = logits_for(77, 50277, 4.0)
    xt = torch.from_numpy(x).to(DEV)
    s = Sampler(50277, device=DEV)
    for u in (0.0, 0.3, 0.99):
        assert int(s.sample(xt, 0.0, 0.85, 0, u=u, penalties=False)) == int(x.argmax())
        assert int(s.sample(xt, 1.0, 0.0, 0, u=u, penalties=False)) == int(x.argmax())
    assert sample_logits(xt, temperature=0) == int(x.argmax())
    # top_p = 1 within rounding of the total: the reference then keeps everything or, if the fp32 cumulative sum
    # stops short of 1, only the largest entry; the kernel follows the same rule on its own total
    s.sample(xt, 1.0, 1.0, 0, u=0.5, penalties=False)
    kept = int((s.probs > 0).sum())
    assert kept in (1, int((osamp.softmax32(x) > 0).sum()))


def test_ban_penalties_and_occurrence_tables():
    from chatrwkv_amd.sampling import Sampler
    V = 1000
    x = logits_for(5, V, 3.0)
    xt = torch.from_numpy(x).to(DEV)
    ban = [int(np.argmax(x)), 3, 999]
    rng = np.random.Generator(np.random.PCG64(9))
    weight = (rng.random(V) > 0.3).astype(np.float32)      # some ids count for nothing, as blanks / digits do
    s = Sampler(V, device=DEV, token_ban=ban, token_weight=torch.from_numpy(weight), seed=1)
    occ = {}
    pres, freq, decay = 0.2, 0.3, 0.9
    for step in range(40):
        u = float(rng.random())
        adj = osamp.apply_penalties(x, ban, occ, pres, freq)
        ref = osamp.filter_probs(adj, temperature=1.1, top_p=0.9, top_k=50).astype(np.float64)
        tok = int(s.sample(xt, 1.1, 0.9, 50, pres, freq, decay, u=u))
        got = s.probs.cpu().numpy().astype(np.float64)
        _check_probs(got, ref, _boundary_margin(adj, 0.9, 1.1))
        assert tok not in ban and got[tok] > 0
        osamp.update_occurrence(occ, tok, float(weight[tok]), decay)
        seen = s.seen.cpu().numpy()
        assert set(np.nonzero(seen)[0]) == set(occ)
        o = s.occurrence.cpu().numpy()
        np.testing.assert_allclose([o[k] for k in occ], [occ[k] for k in occ], rtol=1e-5, atol=1e-6)
    assert len(occ) > 3


def test_generate_ids_on_tiny_model():
    from chatrwkv_amd import synth
    from chatrwkv_amd.model import RWKV
    from chatrwkv_amd.sampling import PIPELINE_ARGS, generate_ids
    ck = synth.make_checkpoint(version=4, n_layer=2, n_embd=128, n_ffn=512, vocab=211, seed=3)
    m = RWKV(ck, "cuda fp16i8", verbose=False)
    ctx = synth.random_tokens(300, 211, seed=1)              # longer than chunk_len: fed in two calls
    args = PIPELINE_ARGS(temperature=1.0, top_p=0.8, token_ban=[0], chunk_len=256)
    a, _ = generate_ids(m, ctx, 24, args, seed=5)
    b, _ = generate_ids(m, ctx, 24, args, seed=5)
    c, _ = generate_ids(m, ctx, 24, args, seed=6)
    assert a == b and len(a) == 24 and all(0 < t < 211 for t in a)
    assert a != c
    # greedy: temperature 0 equals the argmax loop through forward()
    g, _ = generate_ids(m, ctx, 8, PIPELINE_ARGS(temperature=0, alpha_presence=0, alpha_frequency=0), seed=1)
    out, st = None, None
    for i in range(0, len(ctx), 256):
        out, st = m.forward(ctx[i:i + 256], st)
    want = []
    for _ in range(8):
        t = int(out.argmax())
        want.append(t)
        out, st = m.forward([t], st)
    assert g == want
    # stop token: the output ends before it
    stop = a[5]
    cut, _ = generate_ids(m, ctx, 24, PIPELINE_ARGS(temperature=1.0, top_p=0.8, token_ban=[0], token_stop=[stop]), seed=5)
    assert cut == a[:a.index(stop)]


@pytest.mark.parametrize("vocab", [1, 7, 1000, 8192, 50277, 65536, 70001])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_greedy_token(vocab, dtype):
    """rwkv_greedy_token, the temperature-0 draw without penalties (utils.py:56-58), against numpy's argmax (first
    index of the maximum): random logits, the maximum repeated at several indices, NaN and -inf entries, all entries
    equal; fp32 logits and the fp16 logits RWKV-7 returns; the id is written to the tensor given."""
    from chatrwkv_amd import lib, sampling
    x = logits_for(vocab, vocab, 3.0)
    cases = [x.copy()]
    if vocab >= 7:
        y = x.copy(); y[[vocab - 1, vocab // 2, 3]] = 50.0; cases.append(y)            # ties: the lowest index
        y = x.copy(); y[::3] = np.nan; y[1] = -np.inf; cases.append(y)                    # NaN is never chosen
        y = x.copy(); y[vocab - 1] = 60.0; cases.append(y)                                # the last entry
    cases.append(np.full(vocab, -1.25, np.float32))                                       # all equal: index 0
    out = torch.full((1,), -7, dtype=torch.int32, device=DEV)
    for c in cases:
        t = torch.from_numpy(c).to(DEV).to(dtype)
        ref = c.astype(np.float16 if dtype == torch.float16 else np.float32)
        want = int(np.argmax(np.where(np.isnan(ref), -np.inf, ref)))
        got = sampling.greedy_token(t, out)
        assert got is out and int(out) == want, (vocab, int(out), want)
        assert int(sampling.greedy_token(t)) == want
    L = lib.load()
    assert L.rwkv_greedy_token(None, lib.RWKV_DT_F32, 8, out.data_ptr(), None) == -3
    assert L.rwkv_greedy_token(out.data_ptr(), lib.RWKV_DT_F32, 0, out.data_ptr(), None) == -1
    assert L.rwkv_greedy_token(out.data_ptr(), 7, 8, out.data_ptr(), None) == -5


@pytest.mark.parametrize("vocab", [1, 5, 255, 1023, 4096, 4099, 50277, 65536])
@pytest.mark.parametrize("kind", ["flat", "peaked", "equal", "banned"])
def test_sample_edges(vocab, kind):
    """The register groups of four, the last partial group row and both stages of the cut's search: vocabularies around
    4, 256 and 4096 entries, logits nearly flat (tens of thousands of entries between the first bounds), peaked, all
    equal, and all but one banned; pointers that are not 16-byte aligned take the scalar loads."""
    from chatrwkv_amd.sampling import Sampler
    x = logits_for(vocab, vocab, 0.05 if kind == "flat" else 4.0)
    ban = ()
    if kind == "equal":
        x[:] = 0.75
    if kind == "banned":
        ban = [i for i in range(vocab) if i != vocab // 2][:4000]
        x[vocab // 2] = 30.0
    buf = torch.zeros(vocab + 1, dtype=torch.float32, device=DEV)
    buf[1:] = torch.from_numpy(x).to(DEV)
    adj = osamp.apply_penalties(x, ban)
    for top_p, top_k in ((0.5, 0), (0.9, 0), (0.9, 20), (0.0, 0)):
        if kind == "equal" and top_k:
            continue                       # ties at the k-th place are kept here and cut arbitrarily in the reference
        ref = osamp.filter_probs(adj, 1.0, top_p, top_k).astype(np.float64)
        margin = _boundary_margin(adj, top_p, 1.0) if kind != "equal" else 1.0
        probs = []
        for logits in (torch.from_numpy(x).to(DEV), buf[1:]):
            s = Sampler(vocab, device=DEV, token_ban=ban, seed=1)
            for u in (0.0, 0.4321, 0.99999):
                tok = int(s.sample(logits, 1.0, top_p, top_k, u=u))
                got = s.probs.cpu().numpy().astype(np.float64)
                _check_probs(got, ref, margin)
                cdf = np.cumsum(got)
                # fp32 running sums: off by at most the rounding of ~25 additions in a chain, 25 * 2^-24 of the total
                slack = 25 * 2.0 ** -24 * cdf[-1]
                assert got[tok] > 0 and cdf[tok] >= u * cdf[-1] - slack and cdf[tok] - got[tok] <= u * cdf[-1] + slack
                assert int(s.seen[tok]) == 1
            probs.append(got)
        assert np.array_equal(probs[0], probs[1])


@pytest.mark.parametrize("vocab", [211, 50277, 65536])
@pytest.mark.parametrize("mask", [float(np.finfo(np.float32).min), -2.5e38, -1e30, -np.inf])
def test_masked_logits(vocab, mask):
    """Logits masked with the lowest value of the type, with other values below -2.36e38 (whose product with log2 e is no
    finite fp32 number) and with -inf, one entry or all but three: probability 0, and everything else as it is."""
    from chatrwkv_amd.sampling import Sampler
    x = logits_for(vocab, vocab, 3.0)
    one, most = x.copy(), np.full(vocab, mask, np.float32)
    one[int(x.argmax())] = mask
    most[[1, vocab // 2, vocab - 1]] = [1.0, 1.5, 0.5]
    for y in (one, most):
        t = torch.from_numpy(y).to(DEV)
        for temperature in (1.0, 0.7, 0.0):
            ref = osamp.filter_probs(y, temperature, 0.8, 0).astype(np.float64)
            s = Sampler(vocab, device=DEV, seed=1)
            tok = int(s.sample(t, temperature, 0.8, 0, u=0.6))
            got = s.probs.cpu().numpy().astype(np.float64)
            _check_probs(got, ref, _boundary_margin(y, 0.8, temperature))
            assert ref[tok] > 0 and y[tok] != mask and set(np.nonzero(s.seen.cpu().numpy())[0]) == {tok}


@pytest.mark.parametrize("vocab", [50277, 65536])
@pytest.mark.parametrize("temperature", [0.7, 1.6])
def test_temperature_with_bans_and_penalties(vocab, temperature):
    """Temperatures other than 1 at 13 and 16 group rows, with banned ids, penalties that decay and a weight of 0 for some ids:
    every draw of a short reply against the oracle's filter."""
    from chatrwkv_amd.sampling import Sampler
    x = logits_for(vocab, vocab, 3.0)
    xt = torch.from_numpy(x).to(DEV)
    ban = [int(np.argmax(x)), 0, vocab - 1]
    rng = np.random.Generator(np.random.PCG64(vocab))
    weight = (rng.random(vocab) > 0.3).astype(np.float32)
    s = Sampler(vocab, device=DEV, token_ban=ban, token_weight=torch.from_numpy(weight), seed=1)
    occ = {}
    for step in range(12):
        adj = osamp.apply_penalties(x, ban, occ, 0.3, 0.4)
        top_k = 0 if step % 2 else 60
        ref = osamp.filter_probs(adj, temperature, 0.8, top_k).astype(np.float64)
        tok = int(s.sample(xt, temperature, 0.8, top_k, 0.3, 0.4, 0.9, u=float(rng.random())))
        got = s.probs.cpu().numpy().astype(np.float64)
        _check_probs(got, ref, _boundary_margin(adj, 0.8, temperature))
        assert tok not in ban and got[tok] > 0
        osamp.update_occurrence(occ, tok, float(weight[tok]), 0.9)
        o = s.occurrence.cpu().numpy()
        np.testing.assert_allclose([o[k] for k in occ], [occ[k] for k in occ], rtol=1e-5, atol=1e-6)


def test_uniform_number_from_a_device_tensor():
    """A one-element fp32 tensor on the GPU is read where it is, whatever its shape and place in a larger one, and not
    changed; other types and a tensor on the CPU are converted: all draw the id that the same number as a float draws."""
    from chatrwkv_amd.sampling import Sampler
    xt = torch.from_numpy(logits_for(3, 5003, 3.0)).to(DEV)
    draws = lambda u: int(Sampler(5003, device=DEV, seed=1).sample(xt, 1.0, 0.95, 0, u=u))
    grid = torch.rand(6, 5, generator=torch.Generator().manual_seed(4)).to(DEV)
    before = grid.clone()
    for i, j in ((0, 0), (2, 3), (5, 4)):
        want = draws(float(grid[i, j]))
        for u in (grid[i, j], grid[i:i + 1, j:j + 1], grid[i, j].double(), grid[i, j].cpu()):
            assert draws(u) == want, (i, j, u)
    assert len({draws(v) for v in grid.flatten()}) > 5 and torch.equal(grid, before)


@pytest.mark.parametrize("V", [16388, 20001, 50277, 65536])
@pytest.mark.parametrize("scale", [0.3, 3.0, 30.0])
def test_draw_over_the_chip_against_one_workgroup(V, scale):
    """Vocabularies of more than 16384 entries: the three launches against the one-workgroup kernel on the same operands --
    ragged segments, flat logits (lists too long for LDS), peaked ones (every bound above the cut), masks of -inf and of the
    type's lowest value, bans, penalties, ties, cuts by sum and by count, temperatures.  The probabilities differ by the
    order of the sum they are divided by and two roundings (2^-23 each; a power by up to 1 / T times that), the rest is equal
    where no running sum lies within that of the cut or of the drawn number."""
    from chatrwkv_amd import lib
    from chatrwkv_amd.sampling import Sampler
    L = lib.load()
    rng = np.random.Generator(np.random.PCG64([V, int(10 * scale)]))
    x = (rng.standard_normal(V) * scale).astype(np.float32)
    x[rng.integers(0, V, 50)] = -np.inf
    x[rng.integers(0, V, 50)] = np.finfo(np.float32).min
    x[rng.integers(0, V, 200)] = np.float32(x.max() - 1)          # ties
    xt = torch.from_numpy(x).to(DEV)
    for top_p, top_k, temp in [(0.7, 0, 1.0), (0.05, 0, 1.0), (0.95, 0, 0.7), (0.999, 0, 1.0), (0.9, 40, 1.0), (0.95, 2000, 1.3),
                               (0.85, 1, 1.0), (0.85, 0, 0.0), (0.0, 3, 1.0), (1.0, 100, 1.0), (0.5, 150, 1.0)]:
        s = Sampler(V, device=DEV, token_ban=[0, V - 1, 777])
        seen = rng.integers(0, V, 40)
        s.seen[torch.from_numpy(seen).to(DEV)] = 1
        s.occurrence[torch.from_numpy(seen).to(DEV)] = 2.5
        probs, token = torch.empty_like(s.probs), torch.zeros_like(s.token)
        tables = s.seen.clone(), s.occurrence.clone()
        u = torch.tensor([float(rng.random())], device=DEV)
        s.sample(xt, temp, top_p, top_k, 0.2, 0.3, 0.996, u=u)
        lib.check(L.rwkv_sample_logits(xt.data_ptr(), V, temp, top_p, top_k, s.ban.data_ptr(), 3, tables[0].data_ptr(), tables[1].data_ptr(),
                                       None, 0.2, 0.3, 0.996, u.data_ptr(), probs.data_ptr(), token.data_ptr(),
                                       torch.cuda.current_stream().cuda_stream), "rwkv_sample_logits")
        got, ref = s.probs.cpu().numpy().astype(np.float64), probs.cpu().numpy().astype(np.float64)
        # a running sum near 1 over up to 16 terms in turn and 16 levels of pairs is within 32 * 2^-24 = 2e-6 of the exact one in
        # either order: entries at the cut that add up to twice that may fall to either side
        least = min(v[v > 0].min() ** temp if temp else 1.0 for v in (got, ref))
        assert abs(int((got > 0).sum()) - int((ref > 0).sum())) <= (0 if top_k or top_p in (0.0, 1.0) else 1 + 4e-6 / least), (top_p, top_k, temp)
        both = (got > 0) & (ref > 0)
        np.testing.assert_allclose(got[both], ref[both], rtol=4e-6, atol=1e-30)
        cdf = np.cumsum(ref)
        near = np.abs(cdf / cdf[-1] - float(u)).min()
        if near > 1e-5 and np.array_equal(got > 0, ref > 0):
            assert int(s.token) == int(token), (top_p, top_k, temp)
            assert torch.equal(s.seen, tables[0]) and torch.equal(s.occurrence, tables[1])


def test_draw_without_a_finite_total():
    """Logits that are NaN, infinite or all masked: the three launches leave these to the one-workgroup kernel."""
    from chatrwkv_amd.sampling import Sampler
    V = 50277
    for fill in (float("nan"), float("inf"), float("-inf")):
        x = torch.zeros(V, device=DEV) if fill != float("-inf") else torch.full((V,), fill, device=DEV)
        x[5] = fill
        s = Sampler(V, device=DEV)
        assert 0 <= int(s.sample(x, 1.0, 0.7, 0, 0.2, 0.2, 0.996, u=0.5)) < V


@pytest.mark.parametrize("V", [16388, 50277, 65536])
@pytest.mark.parametrize("temp", [1.0, 0.7, 0.0])
@pytest.mark.parametrize("kind", ["nan", "inf", "masked", "nan among masks"])
def test_draw_without_a_total_as_one_workgroup_makes_it(V, temp, kind):
    """Logits whose exponentials have no positive finite sum: token, probabilities and both tables as the one-workgroup kernel
    leaves them, bit for bit, from buffers that held something else."""
    from chatrwkv_amd import lib
    from chatrwkv_amd.sampling import Sampler
    L = lib.load()
    rng = np.random.Generator(np.random.PCG64([V, 7]))
    x = torch.from_numpy((rng.standard_normal(V) * 3).astype(np.float32)).to(DEV)
    if kind == "nan":
        x[V // 2] = float("nan")
    elif kind == "inf":
        x[V // 2] = float("inf")
    elif kind == "masked":
        x[:] = float("-inf")
    else:                                   # the 1024 entries around the one that is no number are masked
        x[8192:9216] = float("-inf")
        x[8200] = float("nan")
    s = Sampler(V, device=DEV, token_ban=[3])
    seen = torch.from_numpy(rng.integers(0, V, 40)).to(DEV)
    s.seen[seen] = 1
    s.occurrence[seen] = 2.5
    tables = s.seen.clone(), s.occurrence.clone()
    s.token.fill_(-1)
    s.probs.fill_(7.0)
    probs, token = s.probs.clone(), s.token.clone()
    u = torch.tensor([0.4], device=DEV)
    s.sample(x, temp, 0.7, 0, 0.2, 0.3, 0.996, u=u)
    lib.check(L.rwkv_sample_logits(x.data_ptr(), V, temp, 0.7, 0, s.ban.data_ptr(), 1, tables[0].data_ptr(), tables[1].data_ptr(),
                                   None, 0.2, 0.3, 0.996, u.data_ptr(), probs.data_ptr(), token.data_ptr(),
                                   torch.cuda.current_stream().cuda_stream), "rwkv_sample_logits")
    assert int(s.token) == int(token) and torch.equal(s.seen, tables[0]) and torch.equal(s.occurrence, tables[1])
    np.testing.assert_array_equal(s.probs.cpu().numpy(), probs.cpu().numpy())


def _wide(kind, V, rng):
    """Logits of which thousands lie in half an octave: equal ones, two levels, a slope, close ones (an untrained model's), all
    with masks and all but equal and close ones with a few outliers"""
    if kind == "equal":
        x = np.zeros(V)
    elif kind == "levels":
        x = np.where(rng.random(V) < 0.4, 0.0, -0.25)
    elif kind == "slope":
        x = rng.permutation(V) * (0.3 / V)
    elif kind == "close":
        x = rng.standard_normal(V) * 0.003
    else:
        x = rng.standard_normal(V) * 3
    x = x.astype(np.float32)
    if kind not in ("equal", "close"):
        x[rng.integers(0, V, 3)] += 2
    x[rng.integers(0, V, 20)] = -np.inf
    return torch.from_numpy(x).to(DEV)


def _one_workgroup(L, x, temp, top_p, top_k, u, probs, token):
    from chatrwkv_amd import lib
    lib.check(L.rwkv_sample_logits(x.data_ptr(), x.numel(), temp, top_p, top_k, None, 0, None, None, None, 0.0, 0.0, 1.0, u.data_ptr(),
                                   probs.data_ptr(), token.data_ptr(), torch.cuda.current_stream().cuda_stream), "rwkv_sample_logits")


@pytest.mark.parametrize("V", [16388, 50277, 65536])
@pytest.mark.parametrize("kind", ["equal", "levels", "slope", "close", "normal"])
def test_draw_from_logits_close_to_each_other(V, kind):
    """Thousands of entries around the cut, ties among them: kept sets and probabilities as the one-workgroup kernel has them;
    bounds as in test_draw_over_the_chip_against_one_workgroup (equal entries stand or fall together)."""
    from chatrwkv_amd import lib
    from chatrwkv_amd.sampling import Sampler
    L = lib.load()
    rng = np.random.Generator(np.random.PCG64([V, 11]))
    x = _wide(kind, V, rng)
    s = Sampler(V, device=DEV)
    for top_p, top_k, temp in [(0.3, 0, 1.0), (0.7, 0, 1.0), (0.97, 0, 0.8), (0.999, 0, 1.0), (0.9, 50, 1.0), (0.9, 7000, 1.0), (0.8, 3, 1.2)]:
        u = torch.tensor([float(rng.random())], device=DEV)
        probs, token = torch.empty_like(s.probs), torch.full_like(s.token, -1)
        s.sample(x, temp, top_p, top_k, u=u)
        _one_workgroup(L, x, temp, top_p, top_k, u, probs, token)
        got, ref = s.probs.cpu().numpy().astype(np.float64), probs.cpu().numpy().astype(np.float64)
        least = min(v[v > 0].min() ** temp for v in (got, ref))
        loose = 0 if top_k or kind in ("equal", "levels") else 1 + 4e-6 / least
        assert abs(int((got > 0).sum()) - int((ref > 0).sum())) <= loose, (top_p, top_k, temp)
        both = (got > 0) & (ref > 0)
        np.testing.assert_allclose(got[both], ref[both], rtol=4e-6, atol=1e-30)
        cdf = np.cumsum(ref)
        if np.abs(cdf / cdf[-1] - float(u)).min() > 1e-5 and np.array_equal(got > 0, ref > 0):
            assert int(s.token) == int(token), (top_p, top_k, temp)


@pytest.mark.parametrize("V", [16388, 50277, 65536])
@pytest.mark.parametrize("temp,top_k", [(1.0, 0), (0.8, 0), (1.0, 30)])
def test_draw_whose_cut_is_at_the_end_of_the_short_list(V, temp, top_k):
    """Cuts in ties at 2^-12.4 to 2^-13.6 of the largest probability, around the 2^-13 that the short list of candidates ends at: the
    same entries, ids and (up to two roundings and the order of the sum) probabilities as with one workgroup."""
    from chatrwkv_amd import lib
    from chatrwkv_amd.sampling import Sampler
    L = lib.load()
    rng = np.random.Generator(np.random.PCG64([V, 13]))
    levels = [0.0, 12.4, 12.9, 13.0, 13.1, 13.6]
    sizes = [40, 600, 600, 600, 600, 600]
    x = np.full(V, -30.0, np.float32)
    at = rng.permutation(V)
    for d, n in zip(levels, sizes):
        x[at[:n]] = -d * np.log(2.0)
        at = at[n:]
    mass = np.array([n * 2.0 ** -d for d, n in zip(levels, sizes)])
    s, xt = Sampler(V, device=DEV), torch.from_numpy(x).to(DEV)
    probs, token = torch.empty_like(s.probs), torch.zeros_like(s.token)
    for i in range(len(levels)):
        top_p = float((mass[:i].sum() + 0.5 * mass[i]) / mass.sum())   # half a level is 1e-3: far from any rounding
        u = torch.tensor([float(rng.random())], device=DEV)
        s.sample(xt, temp, top_p, top_k, u=u, penalties=False)
        _one_workgroup(L, xt, temp, top_p, top_k, u, probs, token)
        got, ref = s.probs.cpu().numpy().astype(np.float64), probs.cpu().numpy().astype(np.float64)
        kept = sum(sizes[:1 if top_k else i + 1])
        assert (got > 0).sum() == kept and np.array_equal(got > 0, ref > 0), (i, temp, top_k)
        assert np.abs(got - ref).max() <= 2e-6 * ref.max()
        cdf = np.cumsum(ref)
        if np.abs(cdf / cdf[-1] - float(u)).min() > 1e-5:
            assert int(s.token) == int(token), (i, temp, top_k)


@pytest.mark.parametrize("V", [16388, 50277, 65536])
@pytest.mark.parametrize("kind,top_p,temp", [("equal", 0.7, 1.0), ("close", 0.7, 1.0), ("slope", 0.85, 0.8), ("normal", 0.999, 1.0), ("normal", 0.999, 0.8)])
def test_draws_over_the_chip_are_not_slower(V, kind, top_p, temp):
    """Draws that keep or search thousands of entries: the three launches take no longer than the one-workgroup kernel on the
    same operands, by the best of several runs (a tenth is left for the clock)."""
    from chatrwkv_amd import lib
    from chatrwkv_amd.sampling import Sampler
    L = lib.load()
    x = _wide(kind, V, np.random.Generator(np.random.PCG64([V, 11])))
    s = Sampler(V, device=DEV)
    u = torch.tensor([0.4], device=DEV)
    token, probs = torch.zeros_like(s.token), torch.empty_like(s.probs)

    def best(draw):
        ms = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(50):
                draw()
            b.record()
            torch.cuda.synchronize()
            ms.append(a.elapsed_time(b))
        return min(ms)

    stream = torch.cuda.current_stream().cuda_stream
    chip = best(lambda: lib.check(L.rwkv_sample_logits_ws(x.data_ptr(), V, temp, top_p, 0, None, 0, None, None, None, 0.0, 0.0, 1.0, u.data_ptr(),
                                                          probs.data_ptr(), token.data_ptr(), s.ws.data_ptr(), s.ws.numel(), stream), "ws"))
    one = best(lambda: _one_workgroup(L, x, temp, top_p, 0, u, probs, token))
    assert chip <= 1.1 * one, (chip, one)
