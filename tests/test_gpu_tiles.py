"""The GEMM tiles of the larger shapes (from 256 rows): the single-bf16 tiles
give the bits of the 64 x 64 ones that small shapes take, forwards of every
precision give a position the same bits on all tiles that a batch may take,
and forwards at batches where the choice of tile, a row split or the LayerNorm
fold changes agree with small batches."""

import dataclasses

import numpy as np
import pytest

from metalfish_amd import backend, synth

pytestmark = pytest.mark.gpu


def _bits(rng, shape, scale=1.0):
    x = (rng.standard_normal(shape) * scale).astype(np.float32)
    u = x.view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


# Rows and widths around the edges of 64-, 128- and 256-wide tiles, K of one
# 64-wide stage, fewer and more stages than any ring holds.
@pytest.mark.parametrize("m,n,k", [(1536, 128, 64), (1537, 130, 128), (1600, 1024, 320),
                                   (2047, 1024, 1024), (4096, 1024, 1024), (4100, 1536, 1024),
                                   (6400, 1024, 1536), (12800, 256, 192), (16385, 256, 64),
                                   (16640, 1024, 256), (1536, 1056, 96), (2048, 2048, 256),
                                   (1601, 2304, 128), (16384, 1024, 224), (256, 1536, 1024), (511, 3136, 1024),
                                   (700, 1538, 512), (1030, 3136, 1024), (1535, 1536, 640)])
@pytest.mark.parametrize("act", ["none", "mish"])
def test_large_tiles_equal_small_ones(m, n, k, act):
    """Single bf16 with fp32 output: the MFMAs of an output accumulate over
    K in one order on every tile, so a row's bits do not depend on how many
    rows the call has (the small call's 64 x 64 tiles run over the whole K); float64 bounds the product:
    at most K * 2^-24 of the summed magnitudes, with a factor 2 for the
    products' own rounding, and mish's slope is below 1.1."""
    rng = np.random.default_rng(m * 7 + n + k)
    a, w = _bits(rng, (m, k)), _bits(rng, (n, k), 1 / np.sqrt(k))
    bias = rng.standard_normal(n).astype(np.float32)
    out = backend.gemm_bf16(a, w, bias, act)
    for lo in {0, m // 2, m - 70}:
        rows = slice(lo, lo + 70)
        small = backend.gemm_bf16(a[rows], w, bias, act)
        assert np.array_equal(out[rows].view(np.uint32), small.view(np.uint32)), (lo, act)
        x = (a[rows].astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        y = (w.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        z = x @ y.T + bias
        bound = 1.1 * k * 2.0 ** -23 * (np.abs(x) @ np.abs(y).T + np.abs(bias)) + 1e-6
        if act == "mish":
            z = z * np.tanh(np.logaddexp(0.0, z))
            bound = bound + 1e-5 * np.abs(z)
        assert (np.abs(small - z) <= bound).all()


@pytest.mark.parametrize("m,n,k", [(2_200_000, 64, 1024), (1_060_000, 128, 1024),
                                   (64, 2_200_000, 1024), (1536, 700_032, 1600),
                                   (300, 66, 1 << 22)])
def test_operands_past_2_and_4_gib(m, n, k):
    """Operands of more than 2 and 4 GiB, which the pipelined tiles' 32-bit
    offsets do not reach (activations: taken in ranges of rows; weights, or
    rows too long for a range: lock-step tiles): rows on both sides of the
    limits equal those of a small call, to the bit.  (Zeros elsewhere, which
    a wrapped or range-checked address would read.)"""
    rng = np.random.default_rng(m + n)

    def picked(count):
        if count <= 70:
            return list(range(count))
        near = [limit // (2 * k) + i for limit in (1 << 31, 1 << 32) for i in (-1, 0, 1)]
        return sorted({i for i in near + [0, 1, count // 2, count - 66, count - 1] if i < count})

    rows, cols = picked(m), picked(n)
    a, w = np.zeros((m, k), np.uint16), np.zeros((n, k), np.uint16)
    at = slice(k - 1024, k)
    a[rows, at] = _bits(rng, (len(rows), 1024))
    w[cols, at] = _bits(rng, (len(cols), 1024), 1 / 32)
    out = backend.gemm_bf16(a, w)
    small = backend.gemm_bf16(a[rows][:, at], w[cols][:, at])
    assert np.count_nonzero(small) == small.size
    assert np.array_equal(out[np.ix_(rows, cols)].view(np.uint32), small.view(np.uint32))


def test_lo8_rows_past_2_gib():
    """The same for activations with e4m3 lo codes, bf16 output and codes."""
    m, n, k = 1_100_000, 64, 1024
    rng = np.random.default_rng(3)
    rows = [0, 1, m // 2, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, m - 66, m - 1]
    a, a8 = np.zeros((m, k), np.uint16), np.zeros((m, k), np.uint8)
    a[rows] = _bits(rng, (len(rows), k))
    a8[rows] = rng.integers(0, 0x40, (len(rows), k))
    w, w8 = _bits(rng, (n, k), 1 / 32), rng.integers(0, 0x40, (n, k)).astype(np.uint8)
    scale = np.full(n, 0.5, np.float32)
    out = backend.gemm_lo8(a, a8, w, w8, scale, bf16_out=True)
    small = backend.gemm_lo8(a[rows], a8[rows], w, w8, scale, bf16_out=True)
    for got, want in zip(out, small):
        assert np.array_equal(got[rows], want)


@pytest.mark.parametrize("precision,weights_dtype", [("bf16x2", "bf16"), ("bf16x2", "fp8"),
                                                     ("bf16", "bf16")])
def test_net_with_hidden_rows_past_2_gib(precision, weights_dtype):
    """4200 positions with an FFN of width 4096: FFN2 reads 2.2 GB of hidden
    rows (each plane), with the residual; every position has the bits of
    batch 321."""
    spec = dataclasses.replace(synth.SPECS["bt4"], name="wide", layers=1, ffn=4096)
    weights = synth.make_weights(spec, seed=1)
    planes, _ = synth.playout_positions(8, seed=2)
    masks, values = backend.pack_planes(planes)
    net = backend.create_network(spec, weights, max_batch=4200, device=0, precision=precision,
                                 weights_dtype=weights_dtype)
    idx = np.arange(4200) % 8
    policy, wdl = net.eval_packed(masks[idx], values[idx])
    small_policy, small_wdl = net.eval_packed(masks[idx[:321]], values[idx[:321]])
    net.close()
    assert np.isfinite(policy).all() and np.ptp(policy) > 0
    assert np.array_equal(policy, small_policy[:8][idx])
    assert np.array_equal(wdl, small_wdl[:8][idx])


# Batches of one group take different tiles, row splits and edges, but the same
# K order everywhere else (below 24 some products are split over K; the policy
# map and the smolgen compression change theirs at 65, the compression at 48).
_BIT_GROUPS = {
    ("plain", "0"): [[24, 25, 33, 43, 48, 63, 64], [65, 86, 100, 129, 200, 255, 256, 257, 300, 321,
                                                    513]],
    ("smolgen", "0"): [[48, 62, 63, 64], [65, 66, 86, 100, 129, 200, 255, 256, 257, 300, 321, 513]],
    ("plain", "1"): [[24, 25, 33, 43, 48, 62], [63, 64], [65, 100, 257, 300], [255, 256, 512]],
    ("smolgen", "1"): [[48, 62], [255, 256, 512]],
}
# K of one, two, three and eight 64-wide stages: fewer, as many and more than a
# ring holds.  (No e4m3 net of width 256, which takes the row panel at 128.)
_BIT_GROUPS["narrow", "0"] = _BIT_GROUPS["middle", "0"] = _BIT_GROUPS["plain", "0"]
_BIT_KINDS = {
    "smolgen": {},
    "plain": dict(smolgen_compress=0, smolgen_hidden=0, smolgen_gen=0),
    "narrow": dict(smolgen_compress=0, smolgen_hidden=0, smolgen_gen=0, embedding=128, heads=4,
                   ffn=64, input_ffn=64, policy_dim=128),
    "middle": dict(smolgen_compress=0, smolgen_hidden=0, smolgen_gen=0, embedding=512, heads=16,
                   ffn=192, input_ffn=192, policy_dim=64),
}


@pytest.mark.parametrize("kind,precision,weights_dtype,fold", [
    (kind, precision, dtype, fold) for kind, fold in _BIT_GROUPS for precision, dtype in (
        ("bf16x2", "bf16"), ("bf16x2_gemm", "bf16"), ("bf16x2", "fp8"), ("bf16", "bf16"),
        ("bf16", "fp8")) if fold == "0" or (precision != "bf16" and dtype == "bf16")])
def test_a_position_has_the_same_bits_on_every_tile(kind, precision, weights_dtype, fold,
                                                    monkeypatch):
    """Two layers of the BT4 width and narrower, the split, e4m3, residual and
    folded epilogues and the row splits among them: each position of a batch
    has the bits that the other batches of its group give it."""
    monkeypatch.setenv("METALFISH_HIP_FOLD_LN", fold)
    spec = dataclasses.replace(synth.SPECS["bt4"], name="bits", layers=2, **_BIT_KINDS[kind])
    weights = synth.make_weights(spec, seed=3)
    planes, _ = synth.playout_positions(8, seed=4)
    net = backend.create_network(spec, weights, max_batch=513, device=0, precision=precision,
                                 weights_dtype=weights_dtype)
    for group in _BIT_GROUPS[kind, fold]:
        want = None
        for batch in group:
            idx = (np.arange(batch) * 5 + batch) % 8
            out = net.evaluate_batch(planes[idx])
            got = {k: np.ascontiguousarray(out[k]).view(np.uint32) for k in ("policy", "wdl")}
            if want is None:
                want = {k: np.stack([got[k][np.flatnonzero(idx == i)[0]] for i in range(8)])
                        for k in got}
            for k in got:
                bad = np.flatnonzero((got[k] != want[k][idx]).any(axis=1))
                print(f"{kind} {precision}/{weights_dtype} fold {fold} batch {batch} {k}: "
                      f"{bad.size} positions differ", flush=True)
                assert bad.size == 0, (batch, k, bad[:8])
    net.close()


@pytest.mark.parametrize("weights_dtype", ["bf16", "fp8"])
@pytest.mark.parametrize("precision", ["bf16x2", "bf16x2_gemm", "bf16"])
def test_batches_across_tile_rules_agree(precision, weights_dtype):
    """Two BT4-width layers: batches below the fold whose tiles differ (8 to
    20), the first folded one (24), odd ones,
    one past a tile's whole rounds (65, 129, 257: the rows split over two
    launches) and others agree with batch 4 position by position.  In bf16x2
    to summation-order noise, 1e-4, as between any two batch sizes; the
    other precisions round activations to bf16 (2^-9), so a last-bit
    difference in a sum can move a logit by what the precision itself is off
    by: 5e-3 and 3e-2 (their errors against the oracle)."""
    tol = {"bf16x2": 1e-4, "bf16x2_gemm": 5e-3, "bf16": 3e-2}[precision]
    spec = dataclasses.replace(synth.SPECS["bt4"], name="two", layers=2)
    weights = synth.make_weights(spec, seed=2)
    planes, _ = synth.playout_positions(4, seed=9)
    net = backend.create_network(spec, weights, max_batch=321, device=0, precision=precision,
                                 weights_dtype=weights_dtype)
    small = net.evaluate_batch(planes)
    assert weights_dtype == "bf16" or "e4m3" in net.info()
    for batch in (8, 12, 16, 20, 24, 25, 33, 43, 64, 65, 100, 129, 200, 257, 300, 321):
        idx = np.arange(batch) % 4
        out = net.evaluate_batch(planes[idx])
        err = np.abs(out["policy"] - small["policy"][idx]).max()
        werr = np.abs(out["wdl"] - small["wdl"][idx]).max()
        print(f"{precision}/{weights_dtype} batch {batch}: policy {err:.2e} wdl {werr:.2e}", flush=True)
        assert err <= tol and werr <= tol
    net.close()


@pytest.mark.parametrize("compress", [8, 40, 104])
@pytest.mark.parametrize("precision,weights_dtype", [("bf16x2", "bf16"), ("bf16x2", "fp8"),
                                                     ("bf16", "bf16"), ("bf16", "fp8")])
@pytest.mark.parametrize("embedding", [256, 768])
def test_narrow_products_agree(precision, weights_dtype, compress, embedding):
    """The compression as a launch of its own on narrow tiles (17 to 47
    positions; columns of a part of a tile, of two and of four; folded
    LayerNorm from 24; an eighth of K of 32 and of 96) against batch 4, where
    it is part of Q|K|V.  Tolerances as between any two batch sizes."""
    tol = {"bf16x2": 1e-4, "bf16": 3e-2}[precision]
    spec = dataclasses.replace(synth.SPECS["bt4"], name="narrow", layers=2, embedding=embedding,
                               heads=embedding // 32, ffn=512, input_ffn=512,
                               smolgen_compress=compress, smolgen_hidden=64, smolgen_gen=64)
    weights = synth.make_weights(spec, seed=6, fp8=weights_dtype == "fp8")
    planes, _ = synth.playout_positions(4, seed=5)
    net = backend.create_network(spec, weights, max_batch=48, device=0, precision=precision,
                                 weights_dtype=weights_dtype)
    small = net.evaluate_batch(planes)
    for batch in (17, 23, 24, 47, 48):
        idx = np.arange(batch) % 4
        out = net.evaluate_batch(planes[idx])
        err = max(np.abs(out[k] - small[k][idx]).max() for k in ("policy", "wdl"))
        print(f"{precision}/{weights_dtype} {embedding} x {compress} batch {batch}: {err:.2e}",
              flush=True)
        assert err <= tol
    net.close()
