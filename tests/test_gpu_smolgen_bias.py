"""The smolgen chain's last LayerNorm with the global projection in one launch
(smolgen_bias.hip) against the attention kernel that generates the bias itself
from separately normalised gen vectors."""

import dataclasses

import numpy as np
import pytest

import oracle
from metalfish_amd import backend, synth

pytestmark = pytest.mark.gpu


# Positions per workgroup of 32 rows: 8, 4, 2 with rows left over and one (with
# and without); gen widths of one, two and four K stages.  Batches: one
# position, a part of a workgroup, whole ones, one and several column tiles per
# workgroup, the last below 3072 rows.
@pytest.mark.parametrize("heads,gen", [(4, 64), (4, 256), (8, 128), (12, 128), (24, 64), (32, 256),
                                       (28, 256), (32, 64)])
@pytest.mark.parametrize("precision,weights_dtype", [("bf16x2", "bf16"), ("bf16x2", "fp8"),
                                                     ("bf16x2_gemm", "bf16"), ("bf16", "bf16"),
                                                     ("bf16", "fp8")])
def test_bias_agrees_with_attention_kernel(heads, gen, precision, weights_dtype, monkeypatch):
    """bf16x2: the two compute the same sums in another order, 1e-4 as between
    two batch sizes.  The single-precision modes hold the gen vectors, and
    here the bias, in bf16 (2^-9 of it), which moves an output by at most
    what their activations' rounding does: 5e-3 and 3e-2."""
    tol = {"bf16x2": 1e-4, "bf16x2_gemm": 5e-3, "bf16": 3e-2}[precision]
    spec = dataclasses.replace(synth.SPECS["bt4"], name="bias", layers=2, embedding=heads * 32,
                               heads=heads, ffn=256, smolgen_gen=gen, smolgen_hidden=64,
                               smolgen_compress=8, input_ffn=256)
    weights = synth.make_weights(spec, seed=4, fp8=weights_dtype == "fp8")
    planes, _ = synth.playout_positions(5, seed=3)
    kw = dict(max_batch=47, device=0, precision=precision, weights_dtype=weights_dtype)
    monkeypatch.setenv("METALFISH_HIP_SKINNY", "0")
    net = backend.create_network(spec, weights, **kw)
    monkeypatch.setenv("METALFISH_HIP_SMOLGEN_BIAS", "attention")
    ref = backend.create_network(spec, weights, **kw)
    assert "bias tensor" in net.info() and "bias in attention" in ref.info()
    for batch in (1, 2, 5, 17, 33, 47):
        idx = np.arange(batch) % 5
        out, want = net.evaluate_batch(planes[idx]), ref.evaluate_batch(planes[idx])
        err = max(np.abs(out[k] - want[k]).max() for k in ("policy", "wdl"))
        print(f"{heads} x {gen} {precision}/{weights_dtype} batch {batch}: {err:.2e}", flush=True)
        assert err <= tol
    net.close()
    ref.close()


@pytest.mark.parametrize("heads,gen", [(40, 64), (8, 192)])
@pytest.mark.parametrize("precision", ["bf16x2", "bf16x2_gemm", "bf16"])
def test_shapes_without_the_one_launch(heads, gen, precision, monkeypatch):
    """More than 32 heads, or a gen width other than 64, 128 and 256: at one
    position the chain is three few-row launches, each LayerNorm applied by
    the GEMM that reads its rows (2L LayerNorm launches fewer than the split-K
    chain, METALFISH_HIP_SKINNY=0); at two, dense1's LayerNorm alone (L
    fewer), then dense2's and the projection GEMM; at 24, all separate.
    Against the oracle and that chain, with the bounds of those precisions
    (bf16x2: summation order, 1e-4; the others round activations to bf16)."""
    layers = 2
    spec = dataclasses.replace(synth.SPECS["bt4"], name="other", layers=layers,
                               embedding=heads * 32, heads=heads, ffn=512, input_ffn=512,
                               smolgen_gen=gen, smolgen_hidden=64, smolgen_compress=8,
                               policy_dim=256)
    weights = synth.make_weights(spec, seed=8)
    planes, _ = synth.playout_positions(4, seed=8)
    ref = oracle.OracleNet(oracle.NetFormat(body_heads=heads), weights).evaluate_batch(planes)
    outs, lns = {}, {}
    for skinny in ("1", "0"):
        monkeypatch.setenv("METALFISH_HIP_SKINNY", skinny)
        net = backend.create_network(spec, weights, max_batch=24, device=0, precision=precision)
        net.set_profiling(True)
        for batch in (1, 2, 24):
            net.profile_reset()
            outs[skinny, batch] = net.evaluate_batch(planes[np.arange(batch) % 4])
            lns[skinny, batch] = net.profile()["layernorm"]["launches"]
        net.close()
    ptol, wtol, dtol = {"bf16x2": (1e-3, 1e-4, 1e-4), "bf16x2_gemm": (2e-2, 5e-3, 2e-2),
                        "bf16": (3e-2, 5e-3, 2e-2)}[precision]
    for (skinny, batch), out in outs.items():
        idx = np.arange(batch) % 4
        perr = np.abs(out["policy"] - ref["policy"][idx]).max()
        werr = np.abs(out["wdl"] - ref["wdl"][idx]).max()
        diff = np.abs(out["policy"] - outs["0", batch]["policy"]).max()
        print(f"{heads} x {gen} {precision} batch {batch} skinny {skinny}: policy {perr:.2e} "
              f"wdl {werr:.2e}, from the split-K chain {diff:.2e}, "
              f"{lns[skinny, batch]} LayerNorms", flush=True)
        assert perr <= ptol and werr <= wtol and diff <= dtol
    for batch, fewer in ((1, 2 * layers), (2, layers), (24, 0)):
        assert lns["1", batch] == lns["0", batch] - fewer, batch
