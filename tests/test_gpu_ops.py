"""GPU parity tests of the operator-level entry points (through the C ABI via ctypes)
against the numpy oracle on the same seeded inputs."""
import numpy as np
import pytest
import torch

from oracle import ops as oops
from oracle import quant as oquant

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _ops():
    from chatrwkv_amd import ops
    return ops


def _rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _quantized(N, M, seed, atype=np.float16):
    w = (_rng(seed).standard_normal((N, M)) * 0.02).astype(np.float32)
    return w, oquant.quantize_u8(w, atype=atype)


def _to_dev_ic(q):
    """uint8/fp16 [N, M] numpy -> GPU tensor of the same shape in the input-contiguous layout."""
    return torch.from_numpy(np.ascontiguousarray(q.T)).to(DEV).t()


# ------------------------------------------------------------------------------ quantizer
@pytest.mark.parametrize("N,M", [(96, 200), (200, 96), (128, 128), (768, 3072), (3072, 768), (333, 77),
                                 (4096, 4096), (4096, 16384), (16384, 4096)])
@pytest.mark.parametrize("scale_dtype", [torch.float16, torch.float32])
def test_quantize_bit_exact(N, M, scale_dtype):
    """uint8 weights and mx/rx/my/ry equal the oracle's (which is pinned bit-exact to the
    reference's routine) for both branches, both input layouts and both output layouts."""
    ops = _ops()
    w = (_rng(N * 7 + M).standard_normal((N, M)) * 0.02).astype(np.float32)
    nat = np.float16 if scale_dtype == torch.float16 else np.float32
    q, mx, rx, my, ry = oquant.quantize_u8(w, atype=nat)
    big = N * M > 4_000_000
    for in_ic in ((True,) if big else (True, False)):
        wt = torch.from_numpy(np.ascontiguousarray(w.T)).to(DEV).t() if in_ic else torch.from_numpy(w).to(DEV)
        for out_ic in ((True,) if big else (True, False)):
            gq, gmx, grx, gmy, gry = ops.quantize_u8(wt, scale_dtype=scale_dtype, input_contiguous=out_ic)
            assert gq.shape == (N, M) and gmy.shape == (N, 1) and gmx.shape == (M,)
            assert gq.stride() == ((1, N) if out_ic else (M, 1))
            assert np.array_equal(gq.cpu().numpy(), q)
            for a, b in ((gmx, mx), (grx, rx), (gmy, my), (gry, ry)):
                assert np.array_equal(a.cpu().numpy().view(np.uint8), b.view(np.uint8))


def test_repack_round_trip():
    ops = _ops()
    q = _rng(5).integers(0, 256, size=(200, 333), dtype=np.uint8)
    t = torch.from_numpy(q).to(DEV)
    ic = ops.to_input_contiguous(t)
    assert ic.stride() == (1, 200) and np.array_equal(ic.cpu().numpy(), q)
    h = torch.from_numpy(_rng(6).standard_normal((130, 70)).astype(np.float16)).to(DEV)
    hic = ops.to_input_contiguous(h)
    assert hic.stride() == (1, 130) and torch.equal(hic, h)


# ------------------------------------------------------------------------------ mm8_one / mm8_seq
MM8_SHAPES = [(768, 768), (768, 3072), (3072, 768), (768, 50277), (2560, 2560), (4096, 4096), (4096, 16384),
              (16384, 4096), (5120, 20480), (4096, 65536)]


def _mm8_case(N, M, B, seed):
    w, (q, mx, rx, my, ry) = _quantized(N, M, seed)
    x = _rng(seed + 1).standard_normal((B, N)).astype(np.float16)
    ref = x.astype(np.float64) @ oquant.dequant_f64(q, mx, rx, my, ry)
    dev = [_to_dev_ic(q)] + [torch.from_numpy(a).to(DEV) for a in (mx, rx, my, ry)]
    return x, ref, dev


@pytest.mark.parametrize("N,M", MM8_SHAPES)
def test_mm8_one(N, M):
    """fp32 result against the fp64 evaluation of x @ W'; tolerance: 1e-3 of the output scale
    (fp16 rounding of x * ry is ~2.4e-4 relative per term), and the fp16 result within one
    fp16 ulp of the rounded fp64 value."""
    ops = _ops()
    x, ref, (q, mx, rx, my, ry) = _mm8_case(N, M, 1, N + M)
    xt = torch.from_numpy(x[0]).to(DEV)
    y32 = ops.mm8_one_f32(N, M, xt, q, mx, rx, my, ry).cpu().numpy().astype(np.float64)
    scale = np.sqrt(np.mean(ref ** 2))
    err = np.abs(y32 - ref[0]).max()
    assert err <= 1e-3 * scale, (err, scale)
    y16 = ops.cuda_mm8_one(N, M, xt, q, mx, rx, my, ry)
    assert y16.dtype == torch.float16 and y16.shape == (M,)
    d = np.abs(y16.cpu().numpy().astype(np.float64) - ref[0])
    assert d.max() <= 1e-3 * scale + np.abs(ref).max() * 2 ** -10


@pytest.mark.parametrize("N,M,B", [(768, 768, 2), (768, 3072, 5), (3072, 768, 128), (768, 50277, 3),
                                   (2560, 2560, 200), (4096, 4096, 1024), (4096, 16384, 256), (16384, 4096, 130), (4096, 16384, 1024),
                                   # long calls: 256 x 256 tiles loaded straight into LDS; whole, ragged and split-K
                                   (4096, 8192, 1000), (16384, 4096, 520), (2560, 10240, 768),
                                   # ragged tiles of the direct-to-LDS kernel: widths and row counts that end inside a tile
                                   (128, 200, 37), (192, 1000, 300), (64, 8, 2), (1024, 136, 129),
                                   # 2 .. 16 rows: every weight row streamed once, K split over the 16 waves of a workgroup
                                   (768, 768, 3), (768, 50277, 9), (4096, 4096, 2), (4096, 16384, 16), (16384, 4096, 7),
                                   (2560, 2560, 13), (5120, 20480, 16), (128, 211, 4), (64, 24, 16), (2048, 512, 6)])
def test_mm8_seq(N, M, B):
    ops = _ops()
    x, ref, (q, mx, rx, my, ry) = _mm8_case(N, M, B, N + M + B)
    xt = torch.from_numpy(x).to(DEV)
    y = ops.cuda_mm8_seq(B, N, M, xt, q, mx, rx, my, ry)
    assert y.dtype == torch.float16 and y.shape == (B, M)
    scale = np.sqrt(np.mean(ref ** 2))
    d = np.abs(y.cpu().numpy().astype(np.float64) - ref)
    assert d.max() <= 1e-3 * scale + np.abs(ref).max() * 2 ** -10, (d.max(), scale)
    # one-token mode and sequence mode agree on the same row (up to fp16 rounding)
    y1 = ops.cuda_mm8_one(N, M, xt[B - 1].contiguous(), q, mx, rx, my, ry)
    assert np.abs(y1.cpu().numpy().astype(np.float64) - y[B - 1].cpu().numpy()).max() <= np.abs(ref).max() * 2 ** -9


@pytest.mark.parametrize("N,M,B", [(64, 4100, 16), (1088, 12304, 2), (2048, 24, 9), (3136, 8200, 8), (4096, 12304, 15), (5120, 8208, 9),
                                   (8192, 4112, 3), (8256, 200, 16), (8320, 4128, 5), (16384, 4112, 13)])
def test_products_of_short_calls(N, M, B):
    """2 .. 16 rows: every number of units a wave holds and the form for longer rows, units that only some waves have, more
    row groups than CUs and fewer, a last one of 4 or 8 rows.  fp16 weights: sums of small whole numbers, so exact, with one
    infinite weight, which stays in its own output.  uint8: bounds as in test_mm8_seq."""
    ops = _ops()
    r = _rng(N + M + B)
    x = r.integers(-2, 3, (B, N)).astype(np.float16)
    w = r.integers(-3, 4, (N, M)).astype(np.float16)
    ref = (x.astype(np.float32) @ w.astype(np.float32)).astype(np.float16)
    wt, xt = _to_dev_ic(w), torch.from_numpy(x).to(DEV)
    y = ops.matmul_float(xt, wt, output_dtype=torch.float16)
    assert np.array_equal(y.cpu().numpy(), ref)
    wt[0, 0] = float("inf")
    y = ops.matmul_float(xt, wt, output_dtype=torch.float32).cpu().numpy()
    assert np.array_equal(y[:, 1:], ref[:, 1:].astype(np.float32)) and not np.isfinite(y[:, 0]).any()
    x, ref, (q, mx, rx, my, ry) = _mm8_case(N, M, B, N + M + B)
    y = ops.cuda_mm8_seq(B, N, M, torch.from_numpy(x).to(DEV), q, mx, rx, my, ry)
    d = np.abs(y.cpu().numpy().astype(np.float64) - ref)
    assert d.max() <= 1e-3 * np.sqrt(np.mean(ref ** 2)) + np.abs(ref).max() * 2 ** -10, d.max()


@pytest.mark.parametrize("N,M,B", [(512, 4, 700), (544, 20, 17), (1056, 100, 300), (2592, 64, 1024), (4096, 192, 651), (8192, 36, 45)])
def test_narrow_outputs(N, M, B):
    """Products of few outputs that one or two rounds of 16 x 16 blocks cover: a last chunk that only some waves have, rows
    that take two rounds of chunks, ragged blocks in both directions.  Sums of small whole numbers, so exact."""
    r = _rng(N + M + B)
    x = r.integers(-2, 3, (B, N)).astype(np.float16)
    w = r.integers(-3, 4, (N, M)).astype(np.float16)
    y = _ops().matmul_float(torch.from_numpy(x).to(DEV), _to_dev_ic(w), output_dtype=torch.float16)
    assert np.array_equal(y.cpu().numpy(), (x.astype(np.float32) @ w.astype(np.float32)).astype(np.float16))


@pytest.mark.parametrize("N,M,B", [(64, 128, 33), (128, 8, 20), (1024, 1000, 17), (1024, 136, 63), (2048, 264, 64), (4096, 4096, 40),
                                   (4096, 2056, 65), (4096, 4096, 129), (1024, 8192, 192), (16384, 512, 256)])
def test_mm8_seq_tile_edges(N, M, B):
    """The 64 x 128 tile (17 .. 64 rows) and the four-stage 128 x 128 tile: fewer k-tiles than stages, ragged rows and
    columns, full depth and K split; bounds as in test_mm8_seq."""
    ops = _ops()
    x, ref, (q, mx, rx, my, ry) = _mm8_case(N, M, B, N + M + B)
    y = ops.cuda_mm8_seq(B, N, M, torch.from_numpy(x).to(DEV), q, mx, rx, my, ry)
    d = np.abs(y.cpu().numpy().astype(np.float64) - ref)
    assert d.max() <= 1e-3 * np.sqrt(np.mean(ref ** 2)) + np.abs(ref).max() * 2 ** -10, d.max()


@pytest.mark.parametrize("N,M,B", [(64, 64, 65), (128, 8, 100), (320, 72, 129), (768, 768, 513), (1024, 1000, 70), (2048, 2048, 333),
                                   (4096, 1032, 256)])
def test_64x64_tile_edges(N, M, B):
    """Products of a few tiles, both weight types: few k-tiles, ragged rows and columns; bounds as in test_mm8_seq and
    test_gemm_f16."""
    ops = _ops()
    x, ref, (q, mx, rx, my, ry) = _mm8_case(N, M, B, N + M + B)
    xt = torch.from_numpy(x).to(DEV)
    d = np.abs(ops.cuda_mm8_seq(B, N, M, xt, q, mx, rx, my, ry).cpu().numpy().astype(np.float64) - ref)
    assert d.max() <= 1e-3 * np.sqrt(np.mean(ref ** 2)) + np.abs(ref).max() * 2 ** -10, d.max()
    w = (_rng(N + M).standard_normal((N, M)) * 0.02).astype(np.float16)
    ref = x.astype(np.float64) @ w.astype(np.float64)
    y = ops.matmul_float(xt, _to_dev_ic(w), output_dtype=torch.float32)
    assert np.abs(y.cpu().numpy() - ref).max() <= 1e-4 * np.sqrt(np.mean(ref ** 2))


def _affine_case(N, M, B, seed):
    """Operands whose sums are exact in fp32 in any order, and (twice) what the uint8 product then has to return bit for
    bit: rounded to fp32 and from there to fp16, and rounded to fp16 at once."""
    r = _rng(seed)
    m = 3 if N <= 4096 else 1
    x = r.integers(-m, m + 1, (B, N)).astype(np.float16)
    q = r.integers(0, 256, (N, M), dtype=np.uint8)
    ry = r.choice(np.array([0.5, 1, 2], np.float16), (N, 1))
    my = (r.integers(-64, 65, (N, 1)) / 1024).astype(np.float16)
    rx, mx = ((r.standard_normal(M) * 2.0 ** -10).astype(np.float16) for _ in range(2))
    xs = x.astype(np.float64) * ry.astype(np.float64).T
    assert (np.abs(xs).sum(1).max() * 256) < 2 ** 22              # quarters: every partial sum has at most 24 bits
    xt, qt = torch.from_numpy(xs), torch.from_numpy(q.astype(np.float64) + 0.5)
    acc = (xt @ qt).numpy()
    s0, s2 = x.astype(np.float64).sum(1), x.astype(np.float64) @ my.astype(np.float64)[:, 0]
    # fp64 holds both fused multiply-adds exactly (46 bits)
    t = (mx.astype(np.float64)[None] * s0[:, None] + s2[:, None]).astype(np.float32).astype(np.float64)
    v = rx.astype(np.float64)[None] * acc + t
    return x, (q, mx, rx, my, ry), v.astype(np.float32).astype(np.float16), v.astype(np.float16)


@pytest.mark.parametrize("N,M,B", [(4096, 4096, 16), (4096, 4096, 45), (768, 3072, 513), (4096, 4096, 256), (4096, 4096, 1024),
                                   (4096, 16384, 1024), (2048, 4096, 65),
                                   # K split of a width that is a multiple of four only: the four-wide second pass
                                   (16384, 1004, 100), (4096, 204, 64), (16384, 36, 300)])
def test_mm8_epilogue_rounding(N, M, B):
    """Every kernel that ends in the uint8 format's rank-1 corrections rounds them to fp32 first and then to fp16, whatever
    its tile and with and without K split: with sums that are exact the results are equal bit for bit."""
    x, (q, mx, rx, my, ry), want, at_once = _affine_case(N, M, B, N + M + B)
    if B >= 256:
        assert (want != at_once).any()                            # the two ways of rounding can be told apart here
    y = _ops().cuda_mm8_seq(B, N, M, torch.from_numpy(x).to(DEV), _to_dev_ic(q), *(torch.from_numpy(a).to(DEV) for a in (mx, rx, my, ry)))
    assert np.array_equal(y.cpu().numpy(), want)


@pytest.mark.parametrize("cfg", ["20", "21"])
@pytest.mark.parametrize("N,M,B", [(64, 64, 17), (128, 8, 100), (192, 136, 45), (320, 1000, 64), (448, 520, 65), (1088, 264, 130),
                                   (4096, 768, 100), (4160, 260, 33), (16384, 1004, 100)])
def test_wave_group_tiles(N, M, B, cfg, monkeypatch):
    """The 64 x 64 and 64 x 128 tiles whose wave groups share K, both weight types: K shorter than a stage, a last stage that
    is there in part, an odd number of stages, ragged rows and columns, K splits (the last three).  The sums are exact, so
    the results are equal bit for bit."""
    ops = _ops()
    x, (q, mx, rx, my, ry), want, _ = _affine_case(N, M, B, N + M + B)
    xt = torch.from_numpy(x).to(DEV)
    monkeypatch.setenv("RWKV_GEMM_CFG", cfg)
    y = ops.cuda_mm8_seq(B, N, M, xt, _to_dev_ic(q), *(torch.from_numpy(a).to(DEV) for a in (mx, rx, my, ry)))
    assert np.array_equal(y.cpu().numpy(), want)
    w = (_rng(N).integers(-64, 65, (N, M)) / 64).astype(np.float16)
    y = ops.matmul_float(xt, _to_dev_ic(w), output_dtype=torch.float32)
    assert np.array_equal(y.cpu().numpy(), x.astype(np.float64) @ w.astype(np.float64))


@pytest.mark.parametrize("cfg", ["14"] + [str(c) for c in (18, *range(22, 31))])
@pytest.mark.parametrize("N,M,B", [(64, 200, 17), (192, 1000, 257), (448, 264, 600), (4096, 520, 225), (128, 1003, 160)])
def test_tiles_with_sides_of_128_to_256(N, M, B, cfg, monkeypatch):
    """128 x 128 with K over two groups and all tiles with a side of 160 to 256, both weight types: fewer k-tiles than stages, odd
    numbers of them, ragged rows and columns, K splits (4096 inputs), and outputs that leave four at a time (fp32, and 1003 of them).
    The sums are exact, so the results are equal bit for bit."""
    ops = _ops()
    x, (q, mx, rx, my, ry), want, _ = _affine_case(N, M, B, N + M + B)
    xt = torch.from_numpy(x).to(DEV)
    monkeypatch.setenv("RWKV_GEMM_CFG", cfg)
    y = ops.cuda_mm8_seq(B, N, M, xt, _to_dev_ic(q), *(torch.from_numpy(a).to(DEV) for a in (mx, rx, my, ry)))
    assert np.array_equal(y.cpu().numpy(), want)
    w = (_rng(N).integers(-64, 65, (N, M)) / 64).astype(np.float16)
    exact = x.astype(np.float64) @ w.astype(np.float64)
    for dtype, np_dtype in ((torch.float32, np.float64), (torch.float16, np.float16)):
        assert np.array_equal(ops.matmul_float(xt, _to_dev_ic(w), output_dtype=dtype).cpu().numpy(), exact.astype(np_dtype))


@pytest.mark.parametrize("cfg", [str(c) for c in range(31, 46)])
@pytest.mark.parametrize("N,M,B", [(64, 200, 17), (192, 1000, 50), (320, 264, 97), (4096, 520, 33), (8192, 96, 64), (1088, 1003, 65)])
def test_tiles_of_few_rows(N, M, B, cfg, monkeypatch):
    """The tiles of 32, 48 and 64 rows and 16 to 96 columns, both weight types: K shorter than a stage, a last stage that is there in
    part, odd and even numbers of stages, ragged rows and columns, K splits (4096 and 8192 inputs), outputs that leave four at a time
    (fp32, and 1003 of them).  The sums are exact, so the results are equal bit for bit."""
    ops = _ops()
    x, (q, mx, rx, my, ry), want, _ = _affine_case(N, M, B, N + M + B)
    xt = torch.from_numpy(x).to(DEV)
    monkeypatch.setenv("RWKV_GEMM_CFG", cfg)
    y = ops.cuda_mm8_seq(B, N, M, xt, _to_dev_ic(q), *(torch.from_numpy(a).to(DEV) for a in (mx, rx, my, ry)))
    assert np.array_equal(y.cpu().numpy(), want)
    w = (_rng(N).integers(-64, 65, (N, M)) / 64).astype(np.float16)
    exact = x.astype(np.float64) @ w.astype(np.float64)
    for dtype, np_dtype in ((torch.float32, np.float64), (torch.float16, np.float16)):
        assert np.array_equal(ops.matmul_float(xt, _to_dev_ic(w), output_dtype=dtype).cpu().numpy(), exact.astype(np_dtype))


@pytest.mark.parametrize("cfg", [str(c) for c in range(46, 49)])
@pytest.mark.parametrize("N,M,B", [(64, 200, 17), (192, 1000, 257), (448, 264, 600), (4096, 520, 97), (128, 1003, 160), (320, 97, 96)])
def test_tiles_with_a_side_of_96(N, M, B, cfg, monkeypatch):
    """As above for 96 x 128, 128 x 96 and 96 x 96: rows of outputs that are no power of two, and the last column tile one wide."""
    test_tiles_with_sides_of_128_to_256(N, M, B, cfg, monkeypatch)


@pytest.mark.parametrize("u8,N,M,B", [(False, 16384, 1000, 48), (False, 8192, 66, 100), (False, 11520, 78, 29), (False, 4096, 512, 64),
                                      (True, 3904, 2880, 1922), (True, 3584, 7042, 663)])
def test_tile_that_the_cost_model_puts_first(u8, N, M, B, monkeypatch):
    """Within 1.1 of the best tile, full depth: fp16 operators, which have no scratch to split K over, with long rows and few tiles
    (a price fitted to split launches made it 1.4 to 1.6), and uint8 products of several rounds of tiles (1.15 and 1.24)."""
    ops = _ops()
    x = torch.randn(B, N, device=DEV).half()
    if u8:
        w = torch.randint(0, 256, (M, N), dtype=torch.uint8, device=DEV).t()
        v = [torch.rand(n, device=DEV).half() for n in ((M,), (M,), (N, 1), (N, 1))]
        call = lambda: ops.mm8(x, w, *v)
    else:
        w = torch.randn(M, N, device=DEV).half().t()
        call = lambda: ops.matmul_float(x, w)

    def best(cfg):
        monkeypatch.setenv("RWKV_GEMM_CFG", cfg)
        ms = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(30):
                call()
            b.record()
            torch.cuda.synchronize()
            ms.append(a.elapsed_time(b))
        return min(ms)

    times = {cfg: best(cfg) for cfg in ("", "15", "20", "21")}
    assert times[""] <= 1.1 * min(times.values()), times


@pytest.mark.parametrize("u8,N,M,B", [(True, 16384, 4096, 45), (True, 4096, 20480, 80), (True, 4096, 16384, 160), (True, 4096, 12288, 333),
                                      (False, 4096, 20480, 80), (False, 16384, 4096, 160), (False, 4096, 8192, 300)])
def test_choice_among_all_tiles(u8, N, M, B, monkeypatch):
    """Within 1.15 of the best of all tiles, each with its K split of least price, in a chain of products with weights of their own (from
    memory, not from a cache): the prices' error there is 1 to 3 % on average and under 10 % for these."""
    ops = _ops()
    x = torch.randn(B, N, device=DEV).half()
    copies = 10
    if u8:
        ws = [torch.randint(0, 256, (M, N), dtype=torch.uint8, device=DEV).t() for _ in range(copies)]
        v = [torch.rand(n, device=DEV).half() for n in ((M,), (M,), (N, 1), (N, 1))]
        call = lambda w: ops.mm8(x, w, *v)
    else:
        ws = [torch.randn(M, N, device=DEV).half().t() for _ in range(copies)]
        call = lambda w: ops.matmul_float(x, w)

    def best(cfg):
        monkeypatch.setenv("RWKV_GEMM_CFG", cfg)
        ms = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(3):
                for w in ws:
                    call(w)
            b.record()
            torch.cuda.synchronize()
            ms.append(a.elapsed_time(b))
        return min(ms)

    cfgs = ["", "14", "15", "18"] + [str(c) for c in range(20, 49)]
    times = {cfg: best(cfg) for cfg in cfgs}
    print(f"chosen {times['']:.3f}, best {min(times, key=times.get)} {min(times.values()):.3f}")
    assert times[""] <= 1.15 * min(times.values()), times


@pytest.mark.parametrize("N,M,B", [(4096, 4096, 100), (768, 3072, 513)])
def test_forced_tile_configurations(N, M, B, monkeypatch):
    """RWKV_GEMM_CFG (tuning): each tile configuration of the uint8 product, with sums that are exact, gives the bits of the
    default; a number that is no configuration, and the one that fp16 weights do not have, are refused."""
    from chatrwkv_amd import lib
    ops = _ops()
    x, (q, mx, rx, my, ry), want, _ = _affine_case(N, M, B, N + M + B)
    args = (torch.from_numpy(x).to(DEV), _to_dev_ic(q), *(torch.from_numpy(a).to(DEV) for a in (mx, rx, my, ry)))
    for cfg in ("3", "9", "14", "15"):
        monkeypatch.setenv("RWKV_GEMM_CFG", cfg)
        assert np.array_equal(ops.cuda_mm8_seq(B, N, M, *args).cpu().numpy(), want), cfg
    w = torch.zeros((M, N), dtype=torch.float16, device=DEV).t()
    for cfg, call in (("17", lambda: ops.cuda_mm8_seq(B, N, M, *args)), ("9", lambda: ops.matmul_float(args[0], w))):
        monkeypatch.setenv("RWKV_GEMM_CFG", cfg)
        with pytest.raises(lib.RwkvHipError):
            call()


# configurations that add the products of a row in one order at full depth
SAME_ORDER = [(3, 9), (14, 15, *range(22, 31)), (18, 46, 47, 48), (31, 33, 36, 38, 41, 43), (32, 34, 35, 37, 39, 40, 42, 44, 45)]


@pytest.mark.parametrize("order", SAME_ORDER, ids=lambda o: str(o[0]))
@pytest.mark.parametrize("N,M,B", [(960, 1088, 90), (448, 1003, 129)])
def test_configurations_that_agree_bit_for_bit(N, M, B, order, monkeypatch):
    """Rows do not depend on the tile's sides, on sums that round: neither with uint8 nor with fp16 weights, nor where outputs leave
    four at a time (1003 of them, fp32).  960 inputs are too few for a K split."""
    ops = _ops()
    x = torch.from_numpy(_rng(N).standard_normal((B, N)).astype(np.float16)).to(DEV)
    w = torch.from_numpy((_rng(M).standard_normal((M, N)) * 0.02).astype(np.float32)).to(DEV)
    q, h = ops.quantize_u8(w.t(), scale_dtype=torch.float16, input_contiguous=True), w.half().t()
    calls = [lambda: ops.mm8(x, *q)]
    if order != (3, 9):   # 9 is uint8 alone
        calls += [lambda: ops.matmul_float(x, h), lambda: ops.matmul_float(x, h, output_dtype=torch.float32)]
    for call in calls:
        want = None
        for cfg in order:
            monkeypatch.setenv("RWKV_GEMM_CFG", str(cfg))
            y = call()
            assert want is None or torch.equal(y, want), cfg
            want = y


@pytest.mark.parametrize("cfg", ["", "14", "15", "20", "21"])
@pytest.mark.parametrize("N,M,B", [(1088, 1000, 2176), (8192, 200, 520), (8192, 516, 600)])
def test_tiles_that_walk_along_the_outputs(N, M, B, cfg, monkeypatch):
    """More activations than weights and more than an XCD's L2 holds: consecutive tiles go along the outputs.  Several columns
    of tiles, the last one ragged, at full depth (the first) and in K splits (the others), every tile size, both weight types;
    the sums are exact, so the results are equal bit for bit."""
    ops = _ops()
    x, (q, mx, rx, my, ry), want, _ = _affine_case(N, M, B, N + M + B)
    xt = torch.from_numpy(x).to(DEV)
    monkeypatch.setenv("RWKV_GEMM_CFG", cfg)
    y = ops.cuda_mm8_seq(B, N, M, xt, _to_dev_ic(q), *(torch.from_numpy(a).to(DEV) for a in (mx, rx, my, ry)))
    assert np.array_equal(y.cpu().numpy(), want)
    w = (_rng(N).integers(-64, 65, (N, M)) / 64).astype(np.float16)
    y = ops.matmul_float(xt, _to_dev_ic(w), output_dtype=torch.float32)
    assert np.array_equal(y.cpu().numpy(), x.astype(np.float64) @ w.astype(np.float64))


@pytest.mark.parametrize("cfg", ["14", "15", "20", "21"])
def test_forced_direct_to_lds_tiles_refuse_other_layouts(cfg, monkeypatch):
    """RWKV_GEMM_CFG (tuning): operands that the direct-to-LDS kernels do not take -- here mx on no 16-byte boundary -- are
    refused by every one of their tiles, before anything is launched on them."""
    from chatrwkv_amd import lib
    N, M, B = 128, 72, 40
    x, (q, mx, rx, my, ry), want, _ = _affine_case(N, M, B, 7)
    odd = torch.empty(M + 1, dtype=torch.float16, device=DEV)[1:]
    odd.copy_(torch.from_numpy(mx))
    args = (torch.from_numpy(x).to(DEV), _to_dev_ic(q), odd, *(torch.from_numpy(a).to(DEV) for a in (rx, my, ry)))
    assert np.array_equal(_ops().cuda_mm8_seq(B, N, M, *args).cpu().numpy(), want)
    monkeypatch.setenv("RWKV_GEMM_CFG", cfg)
    with pytest.raises(lib.RwkvHipError):
        _ops().cuda_mm8_seq(B, N, M, *args)


@pytest.mark.parametrize("N,M,B", [(4096, 4096, 100), (768, 3072, 513), (64, 130, 17), (1024, 16384, 1024)])
@pytest.mark.parametrize("which", ["mx", "rx"])
def test_mm8_scales_on_any_boundary(N, M, B, which):
    """mx or rx on no 16-byte boundary: the register-staged tiles (128 x 128 with and without K split, 256 x 256) return the
    bits that the others do."""
    x, (q, mx, rx, my, ry), want, _ = _affine_case(N, M, B, N + M + B)
    v = {"mx": mx, "rx": rx}
    odd = torch.empty(M + 1, dtype=torch.float16, device=DEV)[1:]
    odd.copy_(torch.from_numpy(v[which]))
    dev = {k: odd if k == which else torch.from_numpy(a).to(DEV) for k, a in v.items()}
    y = _ops().cuda_mm8_seq(B, N, M, torch.from_numpy(x).to(DEV), _to_dev_ic(q), dev["mx"], dev["rx"], *(torch.from_numpy(a).to(DEV) for a in (my, ry)))
    assert np.array_equal(y.cpu().numpy(), want)


@pytest.mark.parametrize("N,M,B", [(768, 768, 300), (4096, 4096, 40), (4096, 4096, 256), (2048, 8192, 600)])
@pytest.mark.parametrize("pad,shift", [(0, 1), (3, 0), (8, 0), (5, 1)])
@pytest.mark.parametrize("kind", ["u8", "f16", "f32"])
def test_output_strides_and_boundaries(N, M, B, pad, shift, kind):
    """Output rows that are padded, by whole 16-byte pieces or not, and that start on no 16-byte boundary, through the C ABI:
    the dense results bit for bit (uint8: sums that are exact; fp16 weights: the same tile and K split, which a stride does
    not decide), and nothing written between the rows."""
    from chatrwkv_amd import lib
    L = lib.load()
    x, (q, mx, rx, my, ry), want, _ = _affine_case(N, M, B, N + M + B)
    st = torch.cuda.current_stream().cuda_stream
    xt = torch.from_numpy(x).to(DEV)
    dt = torch.float32 if kind == "f32" else torch.float16
    buf = torch.full((shift + B * (M + pad),), float("nan"), dtype=dt, device=DEV)
    y = buf[shift:].view(B, M + pad)
    if kind == "u8":
        w = _to_dev_ic(q)
        v = [torch.from_numpy(a).to(DEV) for a in (mx, rx, my, ry)]
        ws = torch.empty(L.rwkv_mm8_seq_workspace(B, N), dtype=torch.uint8, device=DEV)
        rc = L.rwkv_mm8_seq_f16(B, N, M, xt.data_ptr(), N, w.data_ptr(), 1, N, *(t.data_ptr() for t in v), y.data_ptr(), M + pad,
                                ws.data_ptr(), ws.numel(), st)
    else:
        # integers: exact in any order, fp32 results exact and fp16 ones rounded once
        w16 = _rng(7).integers(-3, 4, (M, N)).astype(np.float16)
        w = torch.from_numpy(w16).to(DEV)
        rc = L.rwkv_gemm_f16(B, N, M, xt.data_ptr(), N, w.data_ptr(), 1, N, y.data_ptr(), M + pad,
                             lib.RWKV_DT_F32 if kind == "f32" else lib.RWKV_DT_F16, st)
        want = (torch.from_numpy(x.astype(np.float32)) @ torch.from_numpy(w16.astype(np.float32)).t()).numpy()
        if kind == "f16":
            want = want.astype(np.float16)
    assert rc == 0, rc
    assert np.array_equal(y[:, :M].cpu().numpy(), want)
    assert bool(torch.isnan(y[:, M:]).all()) and bool(torch.isnan(buf[:shift]).all())


@pytest.mark.parametrize("N,M,B", [(64, 33, 40), (128, 203, 70), (192, 1001, 300), (2048, 257, 129), (768, 50277, 130), (256, 4099, 1025)])
def test_odd_output_widths(N, M, B):
    """Output rows that start on no 16-byte boundary and end inside a group of eight, both weight types and output types, in
    calls of every tile; bounds as in test_mm8_seq and test_gemm_f16."""
    ops = _ops()
    x, ref, (q, mx, rx, my, ry) = _mm8_case(N, M, B, N + M + B)
    xt = torch.from_numpy(x).to(DEV)
    d = np.abs(ops.cuda_mm8_seq(B, N, M, xt, q, mx, rx, my, ry).cpu().numpy().astype(np.float64) - ref)
    assert d.max() <= 1e-3 * np.sqrt(np.mean(ref ** 2)) + np.abs(ref).max() * 2 ** -10, d.max()
    w = (_rng(N + M).standard_normal((N, M)) * 0.02).astype(np.float16)
    ref = x.astype(np.float64) @ w.astype(np.float64)
    wt = _to_dev_ic(w)
    for dt, tol in ((torch.float32, 0.0), (torch.float16, np.abs(ref).max() * 2 ** -10)):
        y = ops.matmul_float(xt, wt, output_dtype=dt).cpu().numpy().astype(np.float64)
        assert np.abs(y - ref).max() <= 1e-4 * np.sqrt(np.mean(ref ** 2)) + tol


@pytest.mark.parametrize("N,M", [(5120, 20480), (20480, 5120), (5120, 5120)])
def test_mm8_seq_14b_call_length(N, M):
    """The launches of the 14B configuration at its own call length (1024 rows): 320 large
    tiles = 1.25 rounds over the chip for the wide product, K split for the deep one.  Checked against the fp64
    evaluation on 40 rows that include both ends of every 128- and 256-row tile boundary, all columns."""
    ops = _ops()
    B = 1024
    w, (q, mx, rx, my, ry) = _quantized(N, M, N + M + B)
    x = _rng(N + M + B + 1).standard_normal((B, N)).astype(np.float16)
    rows = sorted({0, 1, 63, 64, 127, 128, 129, 255, 256, 257, 383, 384, 511, 512, 513, 639, 640, 767, 768, 769, 895,
                   896, 1000, 1022, 1023} | {int(r) for r in _rng(7).integers(0, B, 15)})
    ref = x[rows].astype(np.float64) @ oquant.dequant_f64(q, mx, rx, my, ry)
    dev = [_to_dev_ic(q)] + [torch.from_numpy(a).to(DEV) for a in (mx, rx, my, ry)]
    y = ops.cuda_mm8_seq(B, N, M, torch.from_numpy(x).to(DEV), *dev)
    assert y.dtype == torch.float16 and y.shape == (B, M)
    scale = np.sqrt(np.mean(ref ** 2))
    d = np.abs(y[rows].cpu().numpy().astype(np.float64) - ref)
    assert d.max() <= 1e-3 * scale + np.abs(ref).max() * 2 ** -10, (d.max(), scale)


def test_mm8_seq_timing_aid_leaves_the_product():
    """rwkv_mm8_seq_time_kernel (the kernel-only timer of the bench) runs the same two launches as
    rwkv_mm8_seq_f16: the output is bit-equal and the mean launch time is positive; whole, ragged and split-K."""
    import ctypes
    from chatrwkv_amd import lib
    ops = _ops()
    L = lib.load()
    for N, M, B in ((4096, 4096, 256), (1024, 136, 129), (16384, 4096, 520)):
        x, ref, (q, mx, rx, my, ry) = _mm8_case(N, M, B, N + M + B)
        xt = torch.from_numpy(x).to(DEV)
        want = ops.cuda_mm8_seq(B, N, M, xt, q, mx, rx, my, ry)
        y = torch.zeros((B, M), device=DEV, dtype=torch.float16)
        nbytes = L.rwkv_mm8_seq_workspace(B, N)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
        ms = ctypes.c_float(-1.0)
        rc = L.rwkv_mm8_seq_time_kernel(B, N, M, xt.data_ptr(), N, q.data_ptr(), q.stride(0), q.stride(1),
                                        mx.data_ptr(), rx.data_ptr(), my.data_ptr(), ry.data_ptr(), y.data_ptr(), M,
                                        ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream, 3,
                                        ctypes.byref(ms))
        lib.check(rc, "rwkv_mm8_seq_time_kernel")
        assert torch.equal(y, want) and 0.0 < ms.value < 100.0
        assert L.rwkv_mm8_seq_time_kernel(B, N, M, xt.data_ptr(), N, q.data_ptr(), q.stride(0), q.stride(1),
                                          mx.data_ptr(), rx.data_ptr(), my.data_ptr(), ry.data_ptr(), y.data_ptr(),
                                          M, ws.data_ptr(), nbytes, None, 0, ctypes.byref(ms)) == -1  # RWKV_E_SHAPE


def test_mm8_linearity_full_size():
    """Size-independent property at the 7B shape: mm8(a + b) == mm8(a) + mm8(b) in fp32 up to rounding."""
    ops = _ops()
    N, M = 4096, 16384
    x, ref, (q, mx, rx, my, ry) = _mm8_case(N, M, 2, 99)
    a, b = torch.from_numpy(x[0]).to(DEV), torch.from_numpy(x[1]).to(DEV)
    s = (a.float() + b.float()).half()
    ya, yb, ys = (ops.mm8_one_f32(N, M, t, q, mx, rx, my, ry) for t in (a, b, s))
    exact_s = s.float().cpu().numpy().astype(np.float64) @ oquant.dequant_f64(
        q.cpu().numpy(), *(t.cpu().numpy() for t in (mx, rx, my, ry)))
    assert np.abs(ys.cpu().numpy() - exact_s).max() <= 1e-3 * np.sqrt(np.mean(exact_s ** 2))
    lin = (ya + yb - ys).abs().max().item()
    assert lin <= 2e-2 * float(np.sqrt(np.mean(exact_s ** 2)))  # s is rounded to fp16


# ------------------------------------------------------------------------------ fp16 gemm / gemv
@pytest.mark.parametrize("N,M,B", [(768, 768, 1), (768, 3072, 1), (4096, 4096, 1), (16384, 4096, 1), (768, 50277, 1),
                                   (768, 768, 7), (3072, 768, 128), (4096, 4096, 300), (768, 50277, 4),
                                   # long calls (256 x 256 tiles loaded straight into LDS): split-K, ragged, shallow
                                   (4096, 4096, 1024), (4096, 8192, 520), (128, 4096, 1024),
                                   (128, 200, 37), (192, 1000, 300), (64, 8, 2),
                                   # 2 .. 16 rows: the streaming kernel
                                   (768, 768, 3), (4096, 4096, 16), (16384, 4096, 5), (2560, 10240, 11), (128, 211, 2), (2048, 512, 6),
                                   # narrow outputs of a LoRA's first stage (17 .. 512 rows, up to 192 outputs, fp16 out):
                                   # ragged rows, an output count that is no multiple of 16, a row length that is no
                                   # multiple of the 512 values one round of the eight waves covers, the row limit
                                   (4096, 160, 256), (4096, 64, 37), (5120, 100, 300), (1056, 192, 512), (4096, 128, 17)])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.float32])
def test_gemm_f16(N, M, B, out_dtype):
    ops = _ops()
    w = (_rng(N + 3 * M).standard_normal((N, M)) * 0.02).astype(np.float16)
    x = _rng(B).standard_normal((B, N)).astype(np.float16)
    ref = x.astype(np.float64) @ w.astype(np.float64)
    wt = _to_dev_ic(w)
    xt = torch.from_numpy(x).to(DEV)
    y = ops.matmul_float(xt[0] if B == 1 else xt, wt, output_dtype=out_dtype)
    assert y.dtype == out_dtype and tuple(y.shape) == ((M,) if B == 1 else (B, M))
    d = np.abs(y.cpu().numpy().astype(np.float64).reshape(B, M) - ref).max()
    tol = 1e-4 * np.sqrt(np.mean(ref ** 2)) + (np.abs(ref).max() * 2 ** -10 if out_dtype == torch.float16 else 0)
    assert d <= tol, (d, tol)


def test_gemm_f16_batched_and_row_major():
    """3-D operands are a batch of products (the RWKV-6 LoRA use, model.py:1269: [5, T, 32] x [5, 32, C]), and a
    plain row-major weight tensor is accepted (converted to the streamed layout)."""
    ops = _ops()
    r = _rng(99)
    a = (r.standard_normal((5, 9, 32))).astype(np.float16)
    b = (r.standard_normal((5, 32, 256)) * 0.1).astype(np.float16)
    ref = np.einsum("bij,bjk->bik", a.astype(np.float64), b.astype(np.float64))
    y = ops.matmul_float(torch.from_numpy(a).to(DEV), torch.from_numpy(b).to(DEV))
    assert y.dtype == torch.float16 and tuple(y.shape) == (5, 9, 256)
    assert np.abs(y.cpu().numpy().astype(np.float64) - ref).max() <= np.abs(ref).max() * 2 ** -10 + 1e-4
    y32 = ops.matmul_float(torch.from_numpy(a[0]).to(DEV), torch.from_numpy(b[0]).to(DEV), output_dtype=torch.float32)
    assert y32.dtype == torch.float32
    assert np.abs(y32.cpu().numpy().astype(np.float64) - ref[0]).max() <= 1e-4 * max(np.abs(ref[0]).max(), 1.0)


def test_gemm_f16_batched_entry_strides():
    """rwkv_gemm_f16_batched through the C ABI with batch strides that are not the dense ones: operands and results
    of the five products lie in larger buffers; long enough (300 rows, K = 64) for the MFMA kernel, and one-row
    products for the streaming one."""
    from chatrwkv_amd import lib
    L = lib.load()
    r = _rng(17)
    nb, N, M = 5, 64, 136
    for B in (300, 1):
        a = torch.from_numpy(r.standard_normal((nb, B + 3, N)).astype(np.float16)).to(DEV)      # 3 unused rows per item
        bt = torch.from_numpy((r.standard_normal((nb, M + 2, N)) * 0.1).astype(np.float16)).to(DEV)  # [batch, M + 2, N]
        c = torch.full((nb, B + 1, M), float("nan"), dtype=torch.float32, device=DEV)
        rc = L.rwkv_gemm_f16_batched(nb, B, N, M, a.data_ptr(), a.stride(1), a.stride(0), bt.data_ptr(), 1, bt.stride(1),
                                     bt.stride(0), c.data_ptr(), c.stride(1), c.stride(0), lib.RWKV_DT_F32,
                                     torch.cuda.current_stream().cuda_stream)
        assert rc == 0, rc
        torch.cuda.synchronize()
        ref = np.einsum("bij,bkj->bik", a[:, :B].cpu().numpy().astype(np.float64), bt[:, :M].cpu().numpy().astype(np.float64))
        got = c[:, :B].cpu().numpy().astype(np.float64)
        assert np.abs(got - ref).max() <= 1e-4 * max(np.abs(ref).max(), 1.0)
        assert bool(torch.isnan(c[:, B]).all())                                               # the spare row is untouched
    assert L.rwkv_gemm_f16_batched(0, 4, 64, 8, a.data_ptr(), 64, 0, bt.data_ptr(), 1, 64, 0, c.data_ptr(), 8, 0, 0, None) == -1
    assert L.rwkv_gemm_f16_batched(2, 4, 64, 8, a.data_ptr(), 64, 4, bt.data_ptr(), 1, 64, 0, c.data_ptr(), 8, 0, 0, None) == -2


def test_mm8_accepts_the_reference_device_layout():
    """A uint8 matrix as the reference's loader leaves it on the GPU (``.contiguous()`` [N, M], output index
    contiguous; model.py:860): the operator functions repack it once per tensor and reuse the copy; results equal the
    ones from the kernel layout bit for bit, and an in-place change of the tensor is seen."""
    ops = _ops()
    N, M, B = 768, 3072, 37
    x, ref, (q_ic, mx, rx, my, ry) = _mm8_case(N, M, B, 4321)
    q_ref = q_ic.contiguous()                                  # strides (M, 1): the reference's layout
    assert q_ref.stride() == (M, 1) and q_ic.stride() == (1, N)
    xt = torch.from_numpy(x).to(DEV)
    y_ic = ops.cuda_mm8_seq(B, N, M, xt, q_ic, mx, rx, my, ry)
    y_ref = ops.cuda_mm8_seq(B, N, M, xt, q_ref, mx, rx, my, ry)
    assert torch.equal(y_ic, y_ref)
    n_cached = len(ops._repacked)
    y1 = ops.cuda_mm8_one(N, M, xt[0].contiguous(), q_ref, mx, rx, my, ry)
    assert len(ops._repacked) == n_cached                      # the second call reused the repacked copy
    assert torch.equal(y1, ops.cuda_mm8_one(N, M, xt[0].contiguous(), q_ic, mx, rx, my, ry))
    q_ref[5].add_(1)                                           # in place: the version counter moves, the copy is redone
    q_ic2 = q_ic.clone()
    q_ic2[5].add_(1)
    assert torch.equal(ops.cuda_mm8_seq(B, N, M, xt, q_ref, mx, rx, my, ry), ops.cuda_mm8_seq(B, N, M, xt, q_ic2, mx, rx, my, ry))
    del q_ref
    import gc
    gc.collect()
    assert len(ops._repacked) == n_cached - 1                  # the copy goes with the tensor


# ------------------------------------------------------------------------------ LayerNorm and mix
@pytest.mark.parametrize("C", [2112, 2560, 4096, 5120, 8192])
@pytest.mark.parametrize("nj", [1, 2, 3, 4, 6])
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("maa", [0, 1])
def test_lnmix_rows_do_not_depend_on_the_call_length(C, nj, scaled, maa):
    """The launch that normalises, shifts, mixes and (uint8) scales a call's rows and sums them, under its C++ name: calls of 2,
    16 and 300 rows (512 threads per row) and of 600 (256 threads) give the same outputs and sums for the same rows, bit
    for bit."""
    import ctypes
    from chatrwkv_amd import lib
    vp = ctypes.c_void_p

    class Args(ctypes.Structure):    # SeqMixArgs
        _fields_ = [("T", ctypes.c_int), ("C", ctypes.c_int)] + [(n, vp) for n in ("x", "ln_w", "ln_b", "sx", "xx_last", "state_out")] + \
                   [(n, vp * 6) for n in ("mix", "ry", "my", "xs", "s0", "s2")] + [("maa_form", ctypes.c_int)]

    launch = getattr(lib.load(), "_Z16lnmix_seq_launchRK10SeqMixArgsiP12ihipStream_t")
    launch.argtypes, launch.restype = [ctypes.POINTER(Args), ctypes.c_int, vp], ctypes.c_int
    g = torch.Generator(device=DEV)
    g.manual_seed(C + nj)
    half = lambda *shape, scale=1.0, mean=0.0: (torch.randn(*shape, generator=g, device=DEV) * scale + mean).half()
    x, w, b, sx = half(600, C, scale=2.0), half(C, scale=0.1, mean=1.0), half(C, scale=0.1), half(C)
    mix, ry, my = ([half(C, scale=s, mean=m) for _ in range(nj)] for s, m in ((0.2, 0.5), (0.01, 0.0), (0.01, 0.0)))
    runs = {}
    for T in (600, 300, 16, 2):
        xs = [torch.zeros(T, C, dtype=torch.float16, device=DEV) for _ in range(nj)]
        s0, s2 = ([torch.zeros(T, device=DEV) for _ in range(nj)] for _ in range(2))
        a = Args(T=T, C=C, x=x.data_ptr(), ln_w=w.data_ptr(), ln_b=b.data_ptr(), sx=sx.data_ptr(), maa_form=maa)
        for j in range(nj):
            a.mix[j], a.xs[j], a.s0[j], a.s2[j] = mix[j].data_ptr(), xs[j].data_ptr(), s0[j].data_ptr(), s2[j].data_ptr()
            if scaled:
                a.ry[j], a.my[j] = ry[j].data_ptr(), my[j].data_ptr()
        assert launch(ctypes.byref(a), nj, torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        runs[T] = xs + s0 + s2
        for got, want in zip(runs[T], runs[600]):
            assert torch.equal(got, want[:T]), T


# ------------------------------------------------------------------------------ WKV
@pytest.mark.parametrize("T,C", [(1, 768), (7, 768), (64, 1000), (300, 768), (1024, 4096)])
def test_wkv4(T, C):
    ops = _ops()
    r = _rng(T * C)
    k = r.standard_normal((T, C)).astype(np.float32)
    v = r.standard_normal((T, C)).astype(np.float32)
    w = -np.exp(r.uniform(-6, -1, C)).astype(np.float32)
    u = r.uniform(-1, 1, C).astype(np.float32)
    aa = r.standard_normal(C).astype(np.float32)
    bb = np.abs(r.standard_normal(C)).astype(np.float32) + 0.1
    pp = r.standard_normal(C).astype(np.float32)
    for zero_state in (True, False):
        if zero_state:
            a0, b0, p0 = np.zeros(C, np.float32), np.zeros(C, np.float32), np.full(C, -1e30, np.float32)
        else:
            a0, b0, p0 = aa, bb, pp
        y_ref, a_ref, b_ref, p_ref = oops.wkv4(k, v, u, w, a0, b0, p0)
        ta, tb, tp = (torch.from_numpy(t.copy()).to(DEV) for t in (a0, b0, p0))
        y, ta2, tb2, tp2 = ops.cuda_wkv(T, C, torch.from_numpy(w).to(DEV), torch.from_numpy(u).to(DEV),
                                        torch.from_numpy(k).to(DEV), torch.from_numpy(v).to(DEV), ta, tb, tp)
        assert ta2 is ta  # state is updated in place, as the reference's kernel does
        np.testing.assert_allclose(y.cpu().numpy(), y_ref, rtol=2e-4, atol=2e-4)
        np.testing.assert_allclose(ta.cpu().numpy(), a_ref, rtol=2e-4, atol=2e-4)
        np.testing.assert_allclose(tb.cpu().numpy(), b_ref, rtol=2e-4, atol=2e-4)
        np.testing.assert_allclose(tp.cpu().numpy(), p_ref, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("T", [2, 8, 37, 63])
def test_wkv4_bits_do_not_depend_on_a_tokens_place(T):
    """One call, and the same tokens one call each: the recurrence of a call that is not cut into chunks rounds every token
    alike, wherever in the kernel's batches of eight it stands, so outputs and state agree bit for bit."""
    ops = _ops()
    C = 768
    r = _rng(T)
    k, v = (torch.from_numpy(r.standard_normal((T, C)).astype(np.float32)).to(DEV) for _ in range(2))
    w = torch.from_numpy(-np.exp(r.uniform(-6, -1, C)).astype(np.float32)).to(DEV)
    u = torch.from_numpy(r.uniform(-1, 1, C).astype(np.float32)).to(DEV)
    one, each = ([torch.zeros(C, device=DEV), torch.zeros(C, device=DEV), torch.full((C,), -1e30, device=DEV)] for _ in range(2))
    y = ops.cuda_wkv(T, C, w, u, k, v, *one)[0]
    for t in range(T):
        yt = ops.cuda_wkv(1, C, w, u, k[t:t + 1].contiguous(), v[t:t + 1].contiguous(), *each)[0]
        assert torch.equal(yt[0], y[t]), t
    assert all(torch.equal(a, b) for a, b in zip(one, each))


@pytest.mark.parametrize("C", [1 << 24, (1 << 24) + 5])
def test_wkv4_rows_on_both_sides_of_the_offsets_range(C):
    """Rows as long as 32-bit offsets allow, and longer ones, which go one at a time: the channels at both ends come out as in calls
    of their own."""
    ops = _ops()
    T = 3
    k, v = (torch.randn(T, C, device=DEV) for _ in range(2))
    w, u = -torch.rand(C, device=DEV), torch.randn(C, device=DEV)
    st = [torch.zeros(C, device=DEV), torch.zeros(C, device=DEV), torch.full((C,), -1e30, device=DEV)]
    y = ops.cuda_wkv(T, C, w, u, k, v, *st)[0]
    for part in (slice(0, 100), slice(C - 100, C)):
        own = [torch.zeros(100, device=DEV), torch.zeros(100, device=DEV), torch.full((100,), -1e30, device=DEV)]
        want = ops.cuda_wkv(T, 100, w[part], u[part], k[:, part], v[:, part], *own)[0]
        assert torch.equal(y[:, part], want) and all(torch.equal(a[part], b) for a, b in zip(st, own))


@pytest.mark.parametrize("T,H", [(1, 2), (5, 3), (16, 2), (17, 2), (50, 4), (256, 64)])
@pytest.mark.parametrize("v6", [False, True])
@pytest.mark.parametrize("layout", [0, 1])
def test_wkv56(T, H, v6, layout):
    ops = _ops()
    N = 64
    C = H * N
    g = _rng(T * H + 10 * layout + int(v6))
    r, k, v = (g.standard_normal((T, H, N)).astype(np.float32) * 0.5 for _ in range(3))
    u = g.uniform(-1, 1, (H, N)).astype(np.float32)
    S0 = g.standard_normal((H, N, N)).astype(np.float32)  # [h][key j][value i], deliberately non-symmetric
    if v6:
        wlogit = g.uniform(-6, 1, (T, H, N)).astype(np.float32)
        dec = np.exp(-np.exp(wlogit)).astype(np.float32)
    else:
        dec = np.exp(-np.exp(g.uniform(-6, 1, (H, N)))).astype(np.float32)
    out_ref, S_ref = oops.wkv56(r, k, v, dec, u, S0)
    st = S0 if layout == 1 else np.ascontiguousarray(S0.transpose(0, 2, 1))
    st_t = torch.from_numpy(st.copy()).to(DEV)
    args = [torch.from_numpy(a.reshape(1, T, C).copy()).to(DEV) for a in (r, k, v)]
    ut = torch.from_numpy(u.reshape(-1)).to(DEV)
    if v6:
        y, st2 = ops.RUN_RWKV_6(1, T, C, H, st_t, *args, torch.from_numpy(wlogit.reshape(1, T, C)).to(DEV), ut,
                                state_layout=layout)
    else:
        y, st2 = ops.RUN_RWKV_5(1, T, C, H, st_t, *args, torch.from_numpy(dec.reshape(-1)).to(DEV), ut,
                                state_layout=layout)
    assert st2 is st_t and y.shape == (1, T, C)
    np.testing.assert_allclose(y.cpu().numpy().reshape(T, H, N), out_ref, rtol=1e-4, atol=1e-4)
    got = st_t.cpu().numpy()
    if layout == 0:
        got = got.transpose(0, 2, 1)
    np.testing.assert_allclose(got, S_ref, rtol=1e-4, atol=1e-4)
