"""The evaluation calls whose speed is measured.

A search engine holds one network on the GPU for its whole run and hands it
batches of leaf positions: a single leaf, the few leaves of a narrow search,
odd-sized batches as the tree allows, the full batches of a wide search, and
the large batches of self-play.  A case is one such call: a network, its
activation precision and weight storage, an entry point and a batch size.

Networks (``metalfish_amd.synth.SPECS``): ``bt4`` (15 layers of width 1024,
smolgen), ``layer`` (the same with one encoder layer, the layer benchmark's
shape) and ``cpu_plumbing`` (2 layers of width 256, no smolgen).  Weights are
random, as no trained network is at hand; positions come from seeded random
playouts.  A network is built once per process and kept, as an engine keeps
it; the positions and the output buffers belong to the state.

Entry points: ``device`` (packed positions and outputs in device memory),
``packed`` (packed positions in host arrays, logits back), ``priors`` (packed
positions and move lists in host arrays, move priors back) and ``planes``
(float planes in host arrays, every output field back).
"""

import dataclasses
import math

import numpy as np
import torch

from metalfish_amd import backend, synth

MAX_BATCH = 1024
SQUARES = 64
POLICY = 1858
MAX_MOVES = 256

SPECS = {
    "bt4": synth.SPECS["bt4"],
    "layer": dataclasses.replace(synth.SPECS["bt4"], name="layer", layers=1),
    "cpu_plumbing": synth.SPECS["cpu_plumbing"],
}
# (activation precision, weight storage) pairs an engine may ask for.
MODES = (("bf16x2", "bf16"), ("bf16x2_fp8lo", "bf16"), ("bf16x2_gemm", "bf16"), ("bf16", "bf16"),
         ("bf16x2", "fp8"), ("bf16x2_fp8lo", "fp8"))


def _case(net, entry, batch, precision="bf16x2", weights="bf16", name=None):
    case = {"net": net, "entry": entry, "batch": batch, "precision": precision,
            "weights": weights}
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # One leaf at a time: analysis, the last moments of a game.
        _case("bt4", "device", 1, name="leaf-1"),
        # A narrow search's few leaves, from the engine's host arrays.
        _case("bt4", "packed", 8, name="leaves-8-host"),
        # A default mini-batch.
        _case("bt4", "device", 32, name="batch-32"),
        # What a tree of that size really gives, with the move priors formed
        # on the device.
        _case("bt4", "priors", 45, name="batch-45-priors"),
        # The fastest precision, a middle batch.
        _case("bt4", "device", 64, precision="bf16", name="batch-64-bf16"),
        # Pairs for the dense layers only, an odd batch.
        _case("bt4", "device", 100, precision="bf16x2_gemm", name="batch-100-gemm"),
        # The benchmark's batch, positions and outputs on the device.
        _case("bt4", "device", 256, name="batch-256"),
        # The same through the call an engine's plain evaluator makes.
        _case("bt4", "planes", 256, name="batch-256-planes"),
        # A large odd batch with the fp8 correction term.
        _case("bt4", "device", 300, precision="bf16x2_fp8lo", name="batch-300-fp8lo"),
        # Self-play on e4m3 weights.
        _case("bt4", "device", 1024, weights="fp8", name="batch-1024-fp8w"),
        # One encoder layer (with the embedding and the heads) in bf16.
        _case("layer", "device", 256, precision="bf16", name="layer-256-bf16"),
        # The small network of tests and CPU-sized engines.
        _case("cpu_plumbing", "packed", 16, name="plumbing-16-host"),
    ]


def draw(rng):
    net = rng.choice(("bt4", "bt4", "bt4", "bt4", "layer", "cpu_plumbing"))
    entry = rng.choice(("device", "device", "packed", "priors", "planes"))
    modes = MODES
    if net == "cpu_plumbing":
        modes = MODES[:1] + MODES[2:5]
    precision, weights = rng.choice(modes)
    batch = int(round(math.exp(rng.uniform(0.0, math.log(MAX_BATCH)))))
    return _case(net, entry, batch, precision, weights)


_weights = {}
_nets = {}


def _host_weights(net):
    if net not in _weights:
        _weights[net] = synth.make_weights(SPECS[net], seed=0)
    return _weights[net]


def _network(case):
    key = (case["net"], case["precision"], case["weights"])
    if key not in _nets:
        _nets[key] = backend.create_network(SPECS[case["net"]], _host_weights(case["net"]),
                                            max_batch=MAX_BATCH, device=0,
                                            precision=case["precision"],
                                            weights_dtype=case["weights"])
    return _nets[key]


def _positions(case, seed):
    """Planes [batch, 112, 64] and the policy indices of the legal moves."""
    planes, legal = synth.playout_positions(case["batch"], seed=seed)
    return planes, [m[m >= 0] for m in legal]


def _move_arrays(moves):
    offsets = np.zeros(len(moves) + 1, np.int32)
    offsets[1:] = np.cumsum([m.size for m in moves])
    return offsets, np.ascontiguousarray(np.concatenate(moves), dtype=np.int16)


def prepare(case, seed):
    net = _network(case)
    planes, moves = _positions(case, seed)
    state = {"net": net, "entry": case["entry"], "batch": case["batch"]}
    if case["entry"] == "planes":
        state["planes"] = planes
        return state
    masks, values = backend.pack_planes(planes)
    if case["entry"] == "device":
        state["masks"] = torch.from_numpy(masks.view(np.int64)).cuda()
        state["values"] = torch.from_numpy(values).cuda()
        state["policy"] = torch.empty((case["batch"], POLICY), dtype=torch.float32, device="cuda")
        state["wdl"] = torch.empty((case["batch"], 3), dtype=torch.float32, device="cuda")
        return state
    state["masks"], state["values"] = masks, values
    if case["entry"] == "priors":
        state["offsets"], state["indices"] = _move_arrays(moves)
        # The engine's edges, as many as a position can have.
        state["edges"] = np.zeros(case["batch"] * MAX_MOVES, np.float32)
    return state


def run(state):
    net = state["net"]
    if state["entry"] == "device":
        net.eval_device(state["batch"], state["masks"].data_ptr(), state["values"].data_ptr(),
                        state["policy"].data_ptr(), state["wdl"].data_ptr(),
                        stream=torch.cuda.current_stream().cuda_stream)
        return {"policy": state["policy"], "wdl": state["wdl"]}
    if state["entry"] == "packed":
        policy, wdl = net.eval_packed(state["masks"], state["values"])
        return {"policy": policy, "wdl": wdl}
    if state["entry"] == "priors":
        priors, wdl = net.eval_priors_flat(state["masks"], state["values"], state["offsets"],
                                           state["indices"], 1.0)
        state["edges"][:priors.size] = priors
        return {"priors": state["edges"], "wdl": wdl}
    out = net.evaluate_batch(state["planes"])
    return {"policy": out["policy"], "wdl": out["wdl"], "value": out["value"]}


def work(case):
    """Weights, inputs and outputs once; the products of the dense layers,
    smolgen, attention and the policy map (one multiply-add is two
    operations, whatever the precision spends on it)."""
    spec = SPECS[case["net"]]
    B, E, S = case["batch"], spec.embedding, SQUARES
    per_weight = 1 if case["weights"] == "fp8" else 2
    weight_bytes = 0
    for _, shape, _, _, dense in synth.tensor_layout(spec):
        weight_bytes += int(np.prod(shape)) * (per_weight if dense else 4)
    macs = S * spec.pe_channels * S * 12 + S * E * (112 + spec.pe_channels)
    macs += 2 * S * E * spec.input_ffn
    layer = S * 4 * E * E + 2 * S * E * spec.ffn + 2 * S * S * E
    if spec.smolgen_compress:
        c, h, g = spec.smolgen_compress, spec.smolgen_hidden, spec.smolgen_gen
        layer += S * E * c + S * c * h + h * spec.heads * g + spec.heads * g * S * S
    macs += spec.layers * layer
    dp = spec.policy_dim
    macs += S * E * dp + 2 * S * dp * dp + S * S * dp
    macs += S * E * spec.value_dim + S * spec.value_dim * spec.value_hidden
    planes_in = 112 * S * 4 if case["entry"] == "planes" else 112 * 12
    # Priors: about 35 moves a position, an index in and a prior out each.
    out = 35 * 6 + 12 if case["entry"] == "priors" else (POLICY + 3) * 4
    return {"bytes": float(weight_bytes + B * (planes_in + out)), "flops": 2.0 * macs * B}


# Errors against 64 bits measured over the listed cases and batches 1 to 1024
# (2-norm; largest over the root mean square): bf16x2 1.4e-5 and 9.5e-5,
# bf16x2_fp8lo 8.7e-5 and 4.6e-4, bf16x2_gemm 7.3e-4 and 4.1e-3, bf16 5.8e-3
# and 2.9e-2.  About four times those.
_TOLERANCE = {
    "bf16x2": {"rel": 6e-5, "max": 4e-4},
    "bf16x2_fp8lo": {"rel": 4e-4, "max": 2e-3},
    "bf16x2_gemm": {"rel": 3e-3, "max": 1.6e-2},
    "bf16": {"rel": 2.4e-2, "max": 1.2e-1},
}


def tolerance(case):
    return dict(_TOLERANCE[case["precision"]])


# ---- The same in 64 bits ------------------------------------------------------


def _weights64(case, device):
    """Weights in float64 as the network computes with them: bf16 values as
    they are, or each dense row as e4m3 codes over max|row| / 448."""
    spec = SPECS[case["net"]]
    host = _host_weights(case["net"])
    out = {}
    for name, shape, _, _, dense in synth.tensor_layout(spec):
        w = torch.from_numpy(host[name])
        if dense and case["weights"] == "fp8":
            # (On the host, whose fp32 division rounds correctly.)
            w = w.reshape(shape[0], -1)
            top = w.abs().amax(dim=1, keepdim=True)
            scale = torch.where(top > 0, top / 448.0, torch.ones_like(top))
            codes = (w / scale).to(torch.float8_e4m3fn)
            w = codes.to(device, torch.float64) * scale.to(device, torch.float64)
        out[name] = w.to(device, torch.float64).reshape(shape)
    return out


def _mish(x):
    return x * torch.tanh(torch.nn.functional.softplus(x))


def _swish(x):
    return x * torch.sigmoid(x)


def _norm(x, g, b):
    mean = x.mean(-1, keepdim=True)
    var = (x - mean).square().mean(-1, keepdim=True)
    return (x - mean) / torch.sqrt(var + 1e-3) * g + b


def _forward64(spec, w, planes):
    """Logits [B, 1858] and win / draw / loss [B, 3] of planes [B, 112, 64]."""
    E, H, S, dp = spec.embedding, spec.heads, SQUARES, spec.policy_dim

    def dense(x, name, part):
        y = x @ w[f"{name}{part}_w"].T.contiguous()
        return y + w[f"{name}{part}_b"]

    x = planes.transpose(1, 2).contiguous()
    B = x.shape[0]
    pe = dense(x[:, :, :12].reshape(B, S * 12), "body.", "ip_emb_preproc")
    x = torch.cat([x, pe.reshape(B, S, spec.pe_channels)], dim=-1)
    x = _norm(_mish(dense(x, "body.", "ip_emb")), w["body.ip_emb_ln_gammas"],
              w["body.ip_emb_ln_betas"])
    x = (x * w["body.ip_mult_gate"].reshape(E, S).T + w["body.ip_add_gate"].reshape(E, S).T)
    alpha = (2.0 * spec.layers) ** -0.25
    f = dense(_mish(dense(x, "body.ip_emb_ffn.", "dense1")), "body.ip_emb_ffn.", "dense2")
    x = _norm(x + alpha * f, w["body.ip_emb_ffn_ln_gammas"], w["body.ip_emb_ffn_ln_betas"])
    for i in range(spec.layers):
        p = f"body.encoder.{i}"
        q, k, v = (dense(x, f"{p}.mha.", t).reshape(B, S, H, E // H).transpose(1, 2).contiguous()
                   for t in "qkv")
        scores = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(E // H)
        if spec.smolgen_compress:
            sg = f"{p}.mha.smolgen."
            c = (x @ w[sg + "compress"].T.contiguous()).reshape(B, -1)
            h = _norm(_swish(dense(c, sg, "dense1")), w[sg + "ln1_gammas"], w[sg + "ln1_betas"])
            h = _norm(_swish(dense(h, sg, "dense2")), w[sg + "ln2_gammas"], w[sg + "ln2_betas"])
            gen = h.reshape(B * H, -1) @ w["body.smolgen_w"].T.contiguous()
            scores = scores + gen.reshape(B, H, S, S)
        ctx = torch.matmul(torch.softmax(scores, dim=-1), v)
        ctx = ctx.transpose(1, 2).reshape(B, S, E)
        x = _norm(x + alpha * dense(ctx, f"{p}.mha.", "dense"), w[p + ".ln1_gammas"],
                  w[p + ".ln1_betas"])
        f = dense(_mish(dense(x, f"{p}.ffn.", "dense1")), f"{p}.ffn.", "dense2")
        x = _norm(x + alpha * f, w[p + ".ln2_gammas"], w[p + ".ln2_betas"])
    pol, val = "policy.vanilla.", "value.winner."
    emb = _mish(dense(x, pol, "ip_pol"))
    q, k = dense(emb, pol, "ip2_pol"), dense(emb, pol, "ip3_pol")
    raw = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(dp)
    # Promotions: the move from rank 7 to rank 8 (64 square pairs), three
    # pieces; the piece's term depends on the target file.
    promo = w[pol + "ip4_pol_w"]
    at = torch.arange(192, device=x.device)
    pair = at % 64
    piece = torch.matmul(k[:, 56:], (promo[:3] + promo[3:]).T.contiguous())  # [B, 8, 3]
    moves = raw[:, 48 + pair // 8, 56 + pair % 8] + piece[:, (at % 24) // 3, at % 3]
    table = torch.cat([raw.reshape(B, S * S), moves], dim=1)
    # The order of the 1858 moves among the table's 4288 (a format table).
    gather = torch.from_numpy(synth.policy_tables()[1].astype(np.int64)).to(x.device)
    v = _mish(dense(x, val, "ip_val")).reshape(B, -1)
    v = dense(_mish(dense(v, val, "ip1_val")), val, "ip2_val")
    return table[:, gather], torch.softmax(v, dim=-1)


def _fast_exp(x):
    """Schraudolph's exponential, the definition of a move's prior: the
    binary32 pattern int(x * 12102203) + 1065353216, without the rounding of
    the pattern."""
    bits = np.clip(x, -88.0, 88.0) * 12102203.0 / 2.0 ** 23 + 127.0
    whole = np.floor(bits)
    return np.ldexp(1.0 + (bits - whole), (whole - 127.0).astype(np.int64))


def exact(case, seed):
    spec = SPECS[case["net"]]
    device = "cuda" if torch.cuda.is_available() else "cpu"
    w = _weights64(case, device)
    planes, moves = _positions(case, seed)
    policy, wdl = [], []
    for at in range(0, case["batch"], 256):
        x = torch.from_numpy(planes[at:at + 256]).to(device, torch.float64)
        p, v = _forward64(spec, w, x)
        policy.append(p.cpu())
        wdl.append(v.cpu())
    policy, wdl = torch.cat(policy).numpy(), torch.cat(wdl).numpy()
    if case["entry"] == "priors":
        edges, at = np.zeros(case["batch"] * MAX_MOVES), 0
        for logits, m in zip(policy, moves):
            if m.size:
                e = _fast_exp(logits[m] - logits[m].max())
                edges[at:at + m.size] = e / e.sum()
                at += m.size
        return {"priors": edges, "wdl": wdl}
    if case["entry"] == "planes":
        return {"policy": policy, "wdl": wdl, "value": wdl[:, 0] - wdl[:, 2]}
    return {"policy": policy, "wdl": wdl}
