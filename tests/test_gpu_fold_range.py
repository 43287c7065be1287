"""The forwards that fold the body's residual LayerNorms into the GEMMs around
them, and those that keep the LayerNorm kernels."""

import dataclasses

import numpy as np
import pytest

from metalfish_amd import backend, synth

pytestmark = pytest.mark.gpu


def _off_centre(spec, seed):
    """Weights whose residual rows have a mean of about three times their
    spread, where the fold's stored rows round coarser than LN(x)."""
    weights = synth.make_weights(spec, seed=seed)
    for i in range(spec.layers):
        for ln in ("ln1", "ln2"):
            weights[f"body.encoder.{i}.{ln}_betas"] = (
                weights[f"body.encoder.{i}.{ln}_betas"] + np.float32(3.0))
    return weights


@pytest.mark.parametrize("precision", ["bf16x2", "bf16x2_gemm", "bf16x2_fp8lo"])
def test_fold_range(precision, monkeypatch):
    """At width 1024 the residual GEMMs have 256 tiles of 128 x 128 from 63
    positions on and whole rounds of 256 x 256 ones at 256 (and at 255, the
    last row tile partial).  24 to 62, 255 and 256 positions fold: 2L - 1 = 3
    LayerNorm launches fewer than with METALFISH_HIP_FOLD_LN=0.  All others
    run the LayerNorm kernels, to the bit."""
    spec = dataclasses.replace(synth.SPECS["bt4"], name="two", layers=2)
    weights = _off_centre(spec, 4)
    planes, _ = synth.playout_positions(4, seed=6)
    batches = {23: 0, 24: 3, 62: 3, 63: 0, 64: 0, 100: 0, 200: 0, 255: 3, 256: 3, 257: 0, 300: 0}
    outs = {}
    for env in ("1", "0"):
        monkeypatch.setenv("METALFISH_HIP_FOLD_LN", env)
        net = backend.create_network(spec, weights, max_batch=300, device=0, precision=precision)
        net.set_profiling(True)
        for b in batches:
            net.profile_reset()
            out = net.evaluate_batch(planes[np.arange(b) % 4])
            outs[env, b] = out, net.profile()["layernorm"]["launches"]
        net.close()
    for b, fewer in batches.items():
        (got, launches), (want, kernels) = outs["1", b], outs["0", b]
        print(f"{precision} batch {b}: {launches} / {kernels} LayerNorm launches, policy max-abs "
              f"{np.abs(got['policy'] - want['policy']).max():.2e}", flush=True)
        assert launches == kernels - fewer, b
        if not fewer:
            assert np.array_equal(got["policy"], want["policy"]), b
            assert np.array_equal(got["wdl"], want["wdl"]), b


@pytest.mark.parametrize("precision", ["bf16x2", "bf16x2_gemm"])
def test_e4m3_weights_do_not_fold(precision, monkeypatch):
    """Nets on e4m3 weights keep the LayerNorm kernels at every batch: the
    bits and launches of METALFISH_HIP_FOLD_LN=0."""
    spec = dataclasses.replace(synth.SPECS["bt4"], name="two", layers=2)
    weights = _off_centre(spec, 5)
    planes, _ = synth.playout_positions(4, seed=7)
    outs = {}
    for env in ("1", "0"):
        monkeypatch.setenv("METALFISH_HIP_FOLD_LN", env)
        net = backend.create_network(spec, weights, max_batch=256, device=0, precision=precision,
                                     weights_dtype="fp8")
        assert "e4m3" in net.info()
        net.set_profiling(True)
        for b in (24, 47, 62, 100, 256):
            net.profile_reset()
            out = net.evaluate_batch(planes[np.arange(b) % 4])
            outs[env, b] = out, net.profile()["layernorm"]["launches"]
        net.close()
    for (env, b), (got, launches) in outs.items():
        want, kernels = outs["0", b]
        assert launches == kernels, b
        assert np.array_equal(got["policy"], want["policy"]), b
        assert np.array_equal(got["wdl"], want["wdl"]), b


def test_e4m3_weights_of_width_256_take_the_row_panel():
    """From 128 positions (8192 rows) nets of width 256 on e4m3 weights run
    their residual GEMMs with the LayerNorm in one row-panel launch without
    being asked to (2L + 1 = 5 LayerNorm launches fewer than at 127), wider
    ones do not."""
    planes, _ = synth.playout_positions(4, seed=7)
    wide = dataclasses.replace(synth.SPECS["cpu_plumbing"], name="wide", embedding=512, heads=16)
    for spec, fewer in ((synth.SPECS["cpu_plumbing"], 5), (wide, 0)):
        weights = synth.make_weights(spec, seed=1, fp8=True)
        outs = []
        for fused in (False, True):
            net = backend.create_network(spec, weights, max_batch=128, device=0,
                                         weights_dtype="fp8", fused_layernorm=fused)
            net.set_profiling(True)
            launches = []
            for b in (127, 128):
                net.profile_reset()
                out = net.evaluate_batch(planes[np.arange(b) % 4])
                launches.append(net.profile()["layernorm"]["launches"])
            net.close()
            outs.append(out)
            assert launches[1] == launches[0] - (5 if fused else fewer), (spec.name, launches)
        if fewer:
            assert np.array_equal(outs[0]["policy"], outs[1]["policy"])
        assert np.abs(outs[0]["policy"] - outs[1]["policy"]).max() <= 1e-4
