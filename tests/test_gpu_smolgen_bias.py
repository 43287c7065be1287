"""The smolgen chain's last LayerNorm with the global projection in one launch
(smolgen_bias.hip) against the attention kernel that generates the bias itself
from separately normalised gen vectors."""

import dataclasses

import numpy as np
import pytest

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
