"""The work this framework is used for, as cases that can be timed: prompts, greedy decoding,
follow-up turns over a cached conversation, and the single blocks a program can call.

Every case goes through qxg.Context, on the seeded random-init models of qxg.MemModel.
The model of a case is fixed (a program loads one model and meets many inputs); token ids,
residual rows and cached KV rows come from the seed."""
import base64
import functools
import os
import sys
import zlib

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "qx-mini-c_amd"))
import qxg  # noqa: E402

HIDDEN, VOCAB, EXPERTS, MAX_CTX = 2048, 151936, 128, 4096
Q_ROWS, KV_ROWS, FF = 4096, 512, 768
BLOCK_BYTES = {"q4k": 144, "q5k": 176, "q6k": 210, "iq2xs": 74, "iq2s": 82, "iq3xxs": 98, "iq3s": 110, "iq4xs": 136}


def listed():
    return [
        # one attention block of a program that steps layer by layer (the smallest call)
        {"name": "attention", "kind": "attention", "mix": 0, "pos": 1500},
        # one routed expert block for one token
        {"name": "moe", "kind": "moe", "mix": 0, "experts": 128, "act": "f32"},
        # the same with the ggml-compatible Q8_K activations, on the real checkpoint's formats
        {"name": "moe_q8_mix", "kind": "moe", "mix": 1, "experts": 128, "act": "q8_k_compat"},
        # the output head on one residual, logits back to the host
        {"name": "head", "kind": "head", "vocab": VOCAB},
        # one layer over a full prompt chunk, the benchmark formats
        {"name": "layer_512", "kind": "layer", "mix": 0, "layer": 0, "experts": 128, "n": 512, "pos": 0},
        # one layer of the real checkpoint's formats (Q5_K, IQ2_S, IQ3_S), a ragged chunk after earlier turns
        {"name": "layer_mix_ragged", "kind": "layer", "mix": 1, "layer": 3, "experts": 128, "n": 149, "pos": 333},
        # the benchmark prompt: 512 tokens through the whole model, logits of the last
        {"name": "prompt_512", "kind": "prompt", "mix": 0, "layers": 48, "n": 512, "pos": 0},
        # a long document, the real checkpoint's formats
        {"name": "prompt_long_mix", "kind": "prompt", "mix": 1, "layers": 16, "n": 1900, "pos": 0},
        # a short follow-up turn in a long conversation
        {"name": "prompt_turn", "kind": "prompt", "mix": 0, "layers": 16, "n": 37, "pos": 2100},
        # greedy decoding in the middle of a conversation (the headline benchmark's path)
        {"name": "greedy", "kind": "greedy", "mix": 0, "layers": 16, "pos": 450, "steps": 12},
        # greedy decoding at the end of the context
        {"name": "greedy_long", "kind": "greedy", "mix": 0, "layers": 16, "pos": 4000, "steps": 12},
        # greedy decoding of the real checkpoint's formats
        {"name": "greedy_mix", "kind": "greedy", "mix": 1, "layers": 16, "pos": 300, "steps": 12},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["attention", "moe", "head", "layer", "layer", "prompt", "prompt", "prompt", "greedy", "greedy", "greedy"])
    mix = rng.randrange(2)
    if kind == "attention":
        return {"kind": kind, "mix": mix, "pos": _log_int(rng, 1, MAX_CTX - 1)}
    if kind == "moe":
        return {"kind": kind, "mix": mix, "experts": rng.choice([8, 24, 64, 100, 128]),
                "act": rng.choice(["f32", "f32", "q8_k_compat"])}
    if kind == "head":
        return {"kind": kind, "vocab": _log_int(rng, 16000, VOCAB)}
    if kind == "layer":
        return {"kind": kind, "mix": mix, "layer": rng.randrange(4) if mix else 0, "experts": rng.choice([16, 60, 128, 128, 128]),
                "n": _log_int(rng, 1, 512), "pos": rng.choice([0, rng.randrange(1, MAX_CTX - 512)])}
    # (a random model of the benchmark formats multiplies a rounding from layer to layer while its
    # cache is short, so those have fewer layers and greedy tokens come after some positions)
    layers = rng.choice([4, 8, 16] if mix else [4, 6, 8])
    if kind == "prompt":
        return {"kind": kind, "mix": mix, "layers": layers, "n": _log_int(rng, 2, 1900), "pos": rng.choice([0, rng.randrange(1, 2000)])}
    return {"kind": kind, "mix": mix, "layers": layers, "pos": _log_int(rng, 8 if mix else 300, MAX_CTX - 32),
            "steps": _log_int(rng, 1, 12)}


def _shape(case):
    """(layers, vocab, experts, with embedding and head) of the case's model."""
    kind = case["kind"]
    if kind == "head":
        return 0, case["vocab"], 8, False, True
    if kind in ("prompt", "greedy"):
        return case["layers"], VOCAB, EXPERTS, True, True
    return (4 if case["mix"] else 1), 256, case.get("experts", EXPERTS), False, False


@functools.lru_cache(maxsize=None)
def _model(layers, vocab, experts, ends, head, mix):
    return qxg.MemModel(layers, vocab, experts, ends, head, seed=1, mix=mix)


def _model_of(case):
    layers, vocab, experts, ends, head = _shape(case)
    return _model(layers, vocab, experts, ends, head, case.get("mix", 0))


class _Loaded:
    """A context with the model on the GPU, given back with its last user."""

    def __init__(self, path):
        self.ctx = qxg.Context(0)
        self.ctx.load(path, verify=False)

    def __del__(self):
        self.ctx.close()


def _cached_rows(rng, positions):
    """INT8 K and V rows and their scales, as earlier turns leave them."""
    k = rng.integers(-127, 128, size=(positions, KV_ROWS), dtype=np.int8)
    v = rng.integers(-127, 128, size=(positions, KV_ROWS), dtype=np.int8)
    ks, vs = ((rng.uniform(0.5, 2.0, size=positions) / 127.0).astype(np.float32) for _ in range(2))
    return k, v, ks, vs


def _residual_rows(rng, n):
    """Residual rows as they stand between layers (measured there: about 6 in root mean square)."""
    return (6.0 * rng.standard_normal((n, HIDDEN))).astype(np.float32)


def _block_layer(case):
    """The layer that a block's case calls: of a mixed model one with Q5_K, IQ2_S and IQ4_XS."""
    return case["layer"] if "layer" in case else case["mix"]


def _block_inputs(case, seed):
    """(residual rows, cached rows or None) of a block's case."""
    rng = np.random.default_rng(seed)
    x = _residual_rows(rng, case.get("n", 1))
    return x, _cached_rows(rng, case["pos"]) if case.get("pos") else None


def prepare(case, seed):
    kind, held = case["kind"], _Loaded(_model_of(case).path)
    ctx, state = held.ctx, {"kind": case["kind"], "held": held}
    if kind in ("prompt", "greedy"):
        rng = np.random.default_rng(seed)
        layers, pos, more = case["layers"], case["pos"], case.get("n", 0) + case.get("steps", 0)
        ctx.kv_create(layers, pos + more + 1)
        for layer in range(layers if pos else 0):
            ctx.kv_write(layer, 0, *_cached_rows(rng, pos))
        state.update(pos=pos, tokens=rng.integers(0, VOCAB, size=max(case.get("n", 0), 1)).astype(np.uint32))
        if kind == "greedy":
            state.update(steps=case["steps"])
        return state
    x, rows = _block_inputs(case, seed)
    state.update(x=x)
    if kind in ("attention", "layer"):
        layer, pos = _block_layer(case), case["pos"]
        ctx.kv_create(4 if case["mix"] else 1, pos + len(x))
        if rows:
            ctx.kv_write(layer, 0, *rows)
        state.update(layer=layer, pos=pos)
    elif kind == "moe":
        ctx.set_activation(case["act"])
        state.update(layer=_block_layer(case))
    return state


def run(state):
    kind, ctx = state["kind"], state["held"].ctx
    if kind == "attention":
        out, context, values = ctx.attention_layer(state["layer"], state["pos"], state["x"][0])
        return {"out": out, "context": context, "values": values}
    if kind == "moe":
        out, moe, ids, weights = ctx.moe_layer(state["layer"], state["x"][0])
        return {"out": out, "moe": moe, "ids": ids, "weights": weights}
    if kind == "head":
        norm, logits, _, _ = ctx.final_head(state["x"][0])
        return {"norm": norm, "logits": logits}
    if kind == "layer":
        ffn_in, moe, out = ctx.prefill_layer(state["layer"], state["pos"], state["x"])
        return {"ffn_in": ffn_in, "moe": moe, "out": out}
    if kind == "prompt":
        _, logits, _, _, _ = ctx.prefill(state["tokens"], state["pos"], want_logits=True)
        return {"logits": logits}
    tokens, _ = ctx.generate(state["tokens"], state["steps"], state["pos"])
    last, _, logits, _, _ = ctx.decode_token(int(tokens[-1]), state["pos"] + state["steps"], want_logits=True)
    return {"tokens": tokens, "residual": last, "logits": logits}


def _layer_formats(mix, layer):
    """(V and O, gate and up, down) of a layer; Q and K are IQ4_XS throughout."""
    kind = layer % 4 if mix else 0
    return ("q5k" if kind in (1, 3) else "iq4xs", "iq2s" if kind in (1, 3) else "iq2xs",
            {0: "iq3xxs", 1: "iq4xs"}.get(kind, "iq3s"))


def _mat_bytes(fmt, rows, cols):
    return rows * cols // 256 * BLOCK_BYTES[fmt]


def _attention_work(mix, layer, n, pos):
    vo, _, _ = _layer_formats(mix, layer)
    bytes_ = (_mat_bytes("iq4xs", Q_ROWS + KV_ROWS, HIDDEN) + _mat_bytes(vo, KV_ROWS, HIDDEN) + _mat_bytes(vo, HIDDEN, Q_ROWS)
              + (pos + n) * (2 * KV_ROWS + 8) + 4 * HIDDEN)
    flops = 2.0 * n * HIDDEN * (2 * Q_ROWS + 2 * KV_ROWS) + 4.0 * Q_ROWS * n * (pos + (n + 1) / 2)
    return bytes_, flops


def _moe_work(mix, layer, n, experts):
    _, gate_up, down = _layer_formats(mix, layer)
    used = experts * (1.0 - (1.0 - 8.0 / experts) ** n)   # experts that n tokens reach, picked evenly
    bytes_ = used * (2 * _mat_bytes(gate_up, FF, HIDDEN) + _mat_bytes(down, HIDDEN, FF)) + 4 * HIDDEN * (experts + 1)
    return bytes_, 2.0 * n * (8 * 3 * FF * HIDDEN + experts * HIDDEN)


def _head_work(vocab):
    return _mat_bytes("q6k", vocab, HIDDEN) + 4 * HIDDEN + 4 * vocab, 2.0 * vocab * HIDDEN


def work(case):
    kind, mix = case["kind"], case.get("mix", 0)
    if kind == "head":
        b, f = _head_work(case["vocab"])
        return {"bytes": b + 8 * HIDDEN, "flops": f}
    if kind == "attention":
        b, f = _attention_work(mix, _block_layer(case), 1, case["pos"])
        return {"bytes": b + 4 * (2 * HIDDEN + Q_ROWS + KV_ROWS), "flops": f}
    if kind == "moe":
        b, f = _moe_work(mix, _block_layer(case), 1, case["experts"])
        return {"bytes": b + 4 * 3 * HIDDEN, "flops": f}
    if kind == "layer":
        n = case["n"]
        parts = [_attention_work(mix, case["layer"], n, case["pos"]), _moe_work(mix, case["layer"], n, case["experts"])]
        return {"bytes": sum(p[0] for p in parts) + 4 * 4 * n * HIDDEN, "flops": sum(p[1] for p in parts)}
    # a prompt reads the weights once for all its tokens, greedy decoding once for each
    passes = [(case["n"], case["pos"])] if kind == "prompt" else [(1, case["pos"] + i) for i in range(case["steps"] + 1)]
    total_b, total_f = 0.0, 0.0
    for n, pos in passes:
        parts = [_head_work(VOCAB)]
        for layer in range(case["layers"]):
            parts += [_attention_work(mix, layer, n, pos), _moe_work(mix, layer, n, EXPERTS)]
        total_b += sum(p[0] for p in parts)
        total_f += sum(p[1] for p in parts)
    return {"bytes": total_b, "flops": total_f}


def tolerance(case):
    """Measured: single blocks against `exact`, whole calls against token steps or the one-kernel-per-phase
    path, about four times the largest difference seen.  One INT8 code of a cache row that rounds the other
    way shows as 1e-6 to 7e-6 of a layer; carried through the layers that follow it is up to 7e-4 of the
    logits (4e-3 over a short cache; 3e-5 in the mixed formats, whose residuals are larger).  A Q8_K code
    that does is 5e-4 of the block."""
    kind = case["kind"]
    if case.get("act") == "q8_k_compat":
        return {"rel": 2e-3, "max": 2e-2}
    if kind == "layer":
        return {"rel": 3e-5, "max": 5e-4}
    if kind in ("prompt", "greedy"):
        if case["mix"]:
            return {"rel": 2e-4, "max": 2e-3}
        short = case["pos"] + case.get("n", 0) < 400
        return {"rel": 1.6e-2, "max": 1e-1} if short else {"rel": 3e-3, "max": 2e-2}
    return {"rel": 2.5e-6, "max": 1e-5}


# ---- the same in 64 bits, in plain torch, from the model file's own bytes ----

# the ggml codebooks (fixed data, MIT licence): 16-bit entries of 2-bit (iq2) or 3-bit (iq3) level numbers
_CODEBOOKS = {
    "iq2xs": (
        "eNoFwVFP6jwYAOC3TbsUrtqlmOlVIWCQX9EunRledWYQPFeTyBcPv6Ij00yu0KBRrybxmMmv/J4HAAMFBl0QIOEETkHBAEYwBgMW"
        "LmEKDq5hBgu4hTvwsIEHqOEZ9vABDSBEUIA6iKMQ9VCEzlAfDZFGMUpQijKUowLdoxJVaIcAY0wxwwJLrLDBFjs8wx5vMSKEBKRD"
        "OAlJj0SkT4ZEk5gkJCUZycmcFKQkFdkRoJhSyqigkipqqKWO3lJPUUACHpwHOoiDKgCGGWWMdZlgkik2YoZZ5tiCedawI0Md0uEd"
        "3Sk7Tx3oqu64+9ZtuogTHvAO5zzkPR7xPh9yzWOe8JRnPOcFX/OSV3zHQWBBBRNCSKGEEVY44cVevAkUkjAIeajDIgSJJZVMCiml"
        "kkZaOZVO3kkvUY/0eE/34ESeTE9QRCIehZGO8ugxglN6+t9pdvZ7BgorqpjqKqGkUsooq5zyqlGoT/q8r/tpf9WHwWDgB+0ADcmQ"
        "Dy+GeggjM7oefYzQ+dn5zzmM2bg7VuPZuB4fxvcXuws2UZPNpJ5sJ0gTHeiO5jrUPR3pvh5qrWOd6FRf6UznutArXepK7zQYbKhh"
        "RhhplDHGGme8eTAHg2IS8ziML2Idg8WWWmaFlfbUKmustc56u7coIQlPholOPhO47F7aS3eJUpLyVKdJmqfLFKZiaqdu+ndKrsBh"
        "Rx1zwkmn3NgZZ51z3qGMZDzrZTqLM7i218drlJOc5/1c50Ve5l85zNjMz+pZf34//5rDQi7Mwi0+Fmc3+ia+efiDClLwQhd5sSwe"
        "i98CbofLq+XLEu5O7vhKr5LV9wrdr+9Hf4N1vl6uwWNPPfPCS6/8xBtvvfPeb3zrjx6VpAxKXuoyK29K2KiN32w2zabdoIpUvAqr"
        "XqWronqq4ME+/HuIHtePULN6VP+pfb2p2zp4Gmz9tt6+bdst2pEd3+ndfFft4HnwfPc8f3l6gT3d273bL/YXr7vXl1fzlr3/vE8/"
        "ep/FJzS4YU23Uc2kaZrs6+br5wsO+MAOk4M/NAf9/fq9+nn/6baqHbTjtmnblvxWv4+/4+Pk+Hw8Hv8HtxDu+w=="
    ),
    "iq3xxs": (
        "eNoFwUtIVFEYAOD//Oc/z3vvuY4TpZKIMuSUCzcGMSLMA81czYiaukoKF5KLaNEELnwUqAhOQmBJjZughChIWgwEPggnMakoMAYi"
        "Ctu0sU24aNH3ASAQGPAghCqohlpognbogBRkoBt6IAf9MAjDMALXIQ+TMA13YA4KsAQPYAWK8AxewBvYhB0owy58gWPwWAOLsVbW"
        "zjpYil1kw2yMPWLrrMz22D77yf4whhw1WoxgFGuwDk9jM8YxiWm8hFnsxSmcwVmcx3u4jCXcwC38gF/xF/5FxgWP8yzv46P8Nr/L"
        "P/HvHAjJkEdVVE0nqZaaKEUZ6qRu6qEcDdJNukV5mqRpmqNFKtASFWmVntMmlWmPjukf1YsWkRGXxYiYEJtiW+yLQ8GkllZGZFTG"
        "5XmZkEmZllk5JK/JUTklZ+SsvC/XZEm+kxVZo5pVQiVVl+pV42pBPVavVEUdKdKhrtcNukW36gld0EW9ql/q13pHH2oyZ02b6TdX"
        "Td68NWWzaw6MtY32gk3aLjtgx+2CfWhLdsv+ttqLeqe8hJf2hryn3mfvh3fCj/ln/DY/59/wF/11/8D/5seCzmAsWAm2g48Bd8Ip"
        "p12dO+cG3BU37564Nbfh3ruKO3KRsDFMhumwL1wO/wOVTW9x"
    ),
    "iq2s": (
        "eNoFwUFvokwDAOAZMkMGTzNkMLCnwWBj/RUzZCDY02CwsT1ho5vu/gow0FhP2GDjfidr3Dddf+X3PABYAAMCBoABDoYgAAKMwBhM"
        "gAIapGAGDJiDBViCFViDn+AXqMAWtGAHDqAHZ/AX3ACECNrQgRS60IM+DGEEJYxhAjOYwwI+widYwg18hTVsYAc/4BF+wSsElmVh"
        "i1jM4pawppaytJVaM8tYC6uyWmtv9dbFggghGzmIIhd5yEchitAdukcSxShBGXpAOSrQI3pCJXpBG1SjBr2hd9ShIzqhL3RFAFsY"
        "Y4IHmGGOhzjAAo/xBCuscYpn2OA5XuAlXuE1rvAWt3iHD7jHZwxtZNu2Y1Pbs6Wd2Jmd24Vd2rXd2J0NiEUwIYQRToYkIIKMyZQo"
        "oklKZsSQOVmQJVmRNalIS3pyI9BBDnVcx3N8J3SkkziZkzuFUzq10zlgwAZ8MBpMBtOBGfwZQIqoTR1KqUs96tOQRvSOShrThGY0"
        "pwV9pE+0pC90Q19pTRv6Rjt6pCf6Ra8UMIthRtiAMcbZkAVMsBEbswlTTLOUzZhhc7ZgS7Zia1axLWvZjh1Yz6CLXMelrueGbuRK"
        "N3Fzt3Brt3E7F3CLY04445wPecAFH/MJV1zzlM+44XO+4Eu+4mte8S1v+Y4feM/PHHrIsz3Ho57reZ7vhV7kSS/2Ei/zcq/wSq/2"
        "Gq/zwBAPyZAN+VAM1VAPzbAa3obQR77tOz71Pd/3Q1/6sZ/4mZ/7hV/6td/4ILACHJCABTwQgQp0YIJfwSVAP+gP+ePxBxCWwIII"
        "JrgYikAIMRZToYQWRszFQqxFJfaiFzcBQxTS0A29MAxlGIdJmIdFWIZ12IRdCEaD0Wg0GU1HemRGu9F+9D2CEYrsyIlo5EV+FEZR"
        "JKM4SqIsyqMiKqM6aqIuAmM8JmM25mMxVmM9NuOf42oM79AdvZN3T3dggidswidqoidmsp/cJvAe3dP74/1gOpqup7vpfgolkrZ0"
        "JJWu9KQvf8hQRvJOShnLRGbyQeaykI/ySZbyRW5kLRvZyaM8yS95lUBZCiuimOJqqAIl1EiNlVJapWqmjJqrhVqqlVqrSm1Vq3bq"
        "oHp1VjBGMY3d2Iv9OIplnMRZnMdFXMZ13MRAWxprogeaaa6HOtBCj/RYT7TSWqd6po2e64Ve6pVe60pvdat3+qB7fdYwQYmdOAlN"
        "3MRL/CRMokQmcZIkWZInRVImv5M6aZIuAamV4pSkLOWpSFWqU5NW6d8UZihzMpq5mZf5WZhFmcziLMmyLM+KrMyarMvAzJrhGZmx"
        "GZ+JmZrpmZlVs88ZfEAP9EE+AGMZbIhhhpuhCYwwIzM2E6OMNqmZGWPmZmGWZmXWpjJb05qdOZjewBzldu7kNHdzL/fzMI9ymcd5"
        "kmd5nhd5mdd5k3c5mOM5mbM5n4u5muu5mf+aV3NYoMIunIIWbuEVfhEWUSGLuEiKrMiLoiiLumiKrgALa4EXZMEWfCEWaqEXZlEt"
        "4CN6pI93j/IRLK0lXpIlW/KlWKqlXprl87Jawif0RJ/kE3gOntvn72dYotIuaemWXumXYRmVskzKrMzLoizLpuxKsLJWeEVWbMVX"
        "YqVWemVW1erPCr3QF/ny+PL1AtZ4TdZszddirdZ6bdbVGm7Qhm7k5mHzuvnYgJ/9T/iKXunr5vX0Cn5Nf8W/v36DyqpwRSpW8Sqo"
        "RDWuVKUrU82rRbWsVlVVtdWh6itYo9qpae3WXu3XYR3Vso7rpM7qvC7qum7qrv5Xgy3eDrZsy7dqq7dmCxvU2I3T0MZtvMZvwkY2"
        "cZM0WZM3RVM2ddM0XQNaq8UtaVnLW9GqVremrdp9C9/QG327f5NvYId3bMd3aqd3ZnfZwXf0Lt8376P9cv+83+4ve9ihzulo53Ze"
        "53dRJ7u4S7qsy7uiK7u6a7quAwd8YAd+UAd9MIfnA/xAH/RDfvz3AXqrxz3pWc970ate96av+s8eHtGRHuXxdPw6gs/0c/0JT+hE"
        "T3cnefp3An9mf+Z/uv+BMz4Pzvw8Ok/P6qzP5nw5387ya/NlXQaX0WVymV62l91lf/m+wCu60qu8vl+vV/A3+Jv/N/iefF++i39v"
        "/8htcBO30W1y291ut/8Dvmbuvw=="
    ),
    "iq3s": (
        "eNoN0utPl1UcAPDv+Z7vuTznOc95fiDOgDQuKpdYI2oFpotrcrEFmIqoy+uKXM1aNYebA9NAmARTFxorpKsxpvkKqxfcnBC6wa8m"
        "ENEi3MIub9wqm2uLP+GzfQAYIAhQoMEDAxYcRCAGlkMiJEEKrIE0yICHIRtyIA/Ww9OQDwVQCMVQCmXwLFTCZtgG22EX7IfX4E2o"
        "hwZohBPQBM3QCm3QAWehE7qgBz6Bz+Ai9EI/fA3DMAY3YQKiMAOz8BPchkX4Df6Bf+E/AOazkMWwOJbAklgqy2C5rJAVs0pWzbay"
        "HWwPO8BeZG+xI+wddpK1snPsC3aVDbAhNsImWJTdYrNskf2xxGKISKjRQx8DDDGCsRiPD+IqzMJH8FFch/lYgEX4DJbiJqzCGtyB"
        "e/AlfBkP41FswBY8he9iO57B89iNH2EfXsavcBBH8DqO4jhO4hRO4484j3fxHnIuuOGWx/NEnsLX8nSexQt4Ka/gVbyG1/I63s7P"
        "8Pf4x/xTPsiH+Sj/lk/yOT7P7/J7HIgRJ0GKNBmy5CiGltEKeoASKJlSaQ2lUyY9Sbn0FG2gfCqkUqqg56iattB22kl7qY4a6Tg1"
        "UQedpk76kC5QL12iq/QNDdAQXaMxitL3NEOz9Ast0t/EhBIRsUwkiJUiWawTG0SxKBPV4gWxWxwUh0WDOCaaRIfoE1+Ka2JM3BLT"
        "YkEsCpSe9GUgQxkr42WiXClT5GqZJjPkYzJPFsgiWSI3ySq5We6Wh2S9PCobZItsl+dll/xcDspReUNOyu/klJyW83JB/ir/lPcl"
        "V55yKlbFq0yVrR5XBapUlastqlbtV6+qI6pNXVCDalhNqKiaW8pK2uiIjtMrdIJO1uk6VxfqjbpMV+hqXaN36X26Tr+iG/Xbulmf"
        "0h36fd2tL+krul+P6DE9rid0VM/ouaX06MV5D3lJXp5X4m30qrzXvVavy7vsjXo3vWlvwbvjodHGmliTZFabNJNpnjDrTYEpMiWm"
        "3FSZWlNvGsxJc9p0mg9Mrxky182omTK3zR3zl7lvmE9+xE/w1/rl/la/zj/o9/hD/ogf9T3r28DG20SbbfNtpd1m37Attsv22D57"
        "xfbbAXvDTtqf7fIgNcgJ8oOiYGdwKDgRdAdjwXgAjpxyERfrVrkkl+VyXKErc8+7fe6Aa3THXbNrcx2u0110Q+4HN+d+dywUoR9G"
        "wvSwOtwbHgvPhQPh/4QW4Xo="
    ),
}
_LEVELS = {"iq2xs": (2, 8, [8, 25, 43, 0]), "iq2s": (2, 8, [8, 25, 43, 0]), "iq3xxs": (3, 4, [4, 12, 20, 28, 36, 44, 52, 62]),
           "iq3s": (3, 4, [1, 3, 5, 7, 9, 11, 13, 15])}
_IQ4_VALUES = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]
_FORMAT_OF = {12: "q4k", 13: "q5k", 14: "q6k", 17: "iq2xs", 18: "iq3xxs", 21: "iq3s", 22: "iq2s", 23: "iq4xs"}


@functools.lru_cache(maxsize=None)
def _codebook(fmt):
    bits, per, levels = _LEVELS[fmt]
    packed = np.frombuffer(zlib.decompress(base64.b64decode(_CODEBOOKS[fmt])), np.uint16).astype(np.int64)
    at = (packed[:, None] >> (bits * np.arange(per))) & ((1 << bits) - 1)
    return torch.tensor(np.array(levels)[at], dtype=torch.float64, device="cuda")


def _signs(bytes_):
    """+1 or -1 for the 8 bits of each value."""
    bits = (bytes_.unsqueeze(-1) >> torch.arange(8, device="cuda")) & 1
    return 1.0 - 2.0 * bits.double()


def _parity_signs(index):
    """The sign byte of a 7-bit index: its bits, and their parity as bit 7."""
    odd = ((index.unsqueeze(-1) >> torch.arange(7, device="cuda")) & 1).sum(-1) & 1
    return _signs(index | (odd << 7))


def _half(raw, at):
    return raw[:, at:at + 2].contiguous().view(torch.float16).double()


def _nibbles(b):
    return torch.stack([b & 15, b >> 4], -1)


def _scale_min(raw, at):
    """The eight 6-bit scales and minima of a Q5_K block."""
    b = raw[:, at:at + 12].long()
    low, mid, high = b[:, :4], b[:, 4:8], b[:, 8:]
    scale = torch.cat([low & 63, (high & 15) | ((low >> 6) << 4)], 1)
    return scale.double(), torch.cat([mid & 63, (high >> 4) | ((mid >> 6) << 4)], 1).double()


def _dequant(fmt, raw):
    """[blocks, bytes] of one format as [blocks, 256] in 64 bits."""
    nb, d = len(raw), _half(raw, 208 if fmt == "q6k" else 0)
    if fmt == "iq4xs":
        high = (raw[:, 2].long() | (raw[:, 3].long() << 8)).unsqueeze(1) >> (2 * torch.arange(8, device="cuda"))
        scale = (_nibbles(raw[:, 4:8].long()).reshape(nb, 8) | ((high & 3) << 4)) - 32
        q = raw[:, 8:].long().reshape(nb, 8, 16)
        values = torch.tensor(_IQ4_VALUES, dtype=torch.float64, device="cuda")[torch.cat([q & 15, q >> 4], -1)]
        return ((d * scale).unsqueeze(-1) * values).reshape(nb, 256)
    if fmt == "iq2xs":
        q = raw[:, 2:66].contiguous().view(torch.int16).long() & 0xffff
        scale = _nibbles(raw[:, 66:74].long()).reshape(nb, 16).repeat_interleave(2, 1)
        return ((d * (0.5 + scale) * 0.25).unsqueeze(-1) * _codebook(fmt)[q & 511] * _parity_signs(q >> 9)).reshape(nb, 256)
    if fmt == "iq2s":
        high = raw[:, 66:74].long().unsqueeze(-1) >> (2 * torch.arange(4, device="cuda"))
        index = raw[:, 2:34].long() | ((high & 3).reshape(nb, 32) << 8)
        scale = _nibbles(raw[:, 74:82].long()).reshape(nb, 16).repeat_interleave(2, 1)
        return ((d * (0.5 + scale) * 0.25).unsqueeze(-1) * _codebook(fmt)[index] * _signs(raw[:, 34:66].long())).reshape(nb, 256)
    if fmt == "iq3xxs":
        aux = raw[:, 66:98].contiguous().view(torch.int32).long() & 0xffffffff
        signs = _parity_signs((aux.unsqueeze(-1) >> (7 * torch.arange(4, device="cuda"))) & 127)
        values = _codebook(fmt)[raw[:, 2:66].long()].reshape(nb, 8, 32) * signs.reshape(nb, 8, 32)
        return ((d * (0.5 + (aux >> 28)) * 0.5).unsqueeze(-1) * values).reshape(nb, 256)
    if fmt == "iq3s":
        high = (raw[:, 66:74].long().unsqueeze(-1) >> torch.arange(8, device="cuda")) & 1
        values = _codebook(fmt)[raw[:, 2:66].long() | (high.reshape(nb, 64) << 8)].reshape(nb, 8, 32)
        values = values * _signs(raw[:, 74:106].long()).reshape(nb, 8, 32)
        scale = d * (1 + 2 * _nibbles(raw[:, 106:110].long()).reshape(nb, 8))
        return (scale.unsqueeze(-1) * values).reshape(nb, 256)
    if fmt == "q5k":
        scale, low = _scale_min(raw, 4)
        q = raw[:, 48:].long().reshape(nb, 4, 32)
        high = (raw[:, 16:48].long().unsqueeze(1) >> torch.arange(8, device="cuda").reshape(1, 8, 1)) & 1
        code = torch.stack([q & 15, q >> 4], 2).reshape(nb, 8, 32) | (high << 4)
        return ((d * scale).unsqueeze(-1) * code - (_half(raw, 2) * low).unsqueeze(-1)).reshape(nb, 256)
    assert fmt == "q6k", fmt
    ql, qh = raw[:, :128].long().reshape(nb, 2, 2, 32), raw[:, 128:192].long().reshape(nb, 2, 1, 32)
    low = torch.stack([ql & 15, ql >> 4], 2).reshape(nb, 2, 4, 32)
    code = (low | (((qh >> (2 * torch.arange(4, device="cuda").reshape(1, 1, 4, 1))) & 3) << 4)) - 32
    scale = raw[:, 192:208].contiguous().view(torch.int8).double() * d
    return (scale.unsqueeze(-1) * code.reshape(nb, 16, 16)).reshape(nb, 256)


@functools.lru_cache(maxsize=4)
def _tensors(path):
    """{name: (ggml type, dims, bytes)} of a QXF1 file."""
    data = np.memmap(path, np.uint8, "r")
    count, at = int(data[16:20].view(np.uint32)[0]), int(data[24:32].view(np.uint64)[0])
    found = {}
    for i in range(count):
        e = data[at + 208 * i:at + 208 * (i + 1)]
        dims, (offset, size) = e[112:144].view(np.uint64), e[144:160].view(np.uint64)
        found[bytes(e[:96]).split(b"\0")[0].decode()] = (int(e[164:168].view(np.uint32)[0]), [int(v) for v in dims],
                                                         data[int(offset):int(offset + size)])
    return found


def _weights(path, name, part=None, parts=1):
    """A matrix, or its part'th of `parts` equal runs of rows, in 64 bits."""
    kind, dims, data = _tensors(path)[name]
    size = len(data) // parts
    data = torch.from_numpy(np.array(data if part is None else data[part * size:(part + 1) * size])).cuda()
    if kind == 0:
        return data.view(torch.float32).double().reshape(-1, dims[0])
    fmt = _FORMAT_OF[kind]
    return _dequant(fmt, data.reshape(-1, BLOCK_BYTES[fmt])).reshape(-1, dims[0])


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w


def _rope(x, positions):
    """[n, heads, 128] rotated by position, halves paired."""
    angle = positions.double().reshape(-1, 1, 1) * 1e6 ** (-torch.arange(64, device="cuda").double() / 64)
    a, b, c, s = x[..., :64], x[..., 64:], torch.cos(angle), torch.sin(angle)
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _int8_rows(x):
    """Rows as the INT8 cache holds them, and how near a value comes to the boundary of two codes."""
    scale = x.abs().amax(-1, keepdim=True) / 127.0
    codes = torch.round(x / scale)
    return codes * scale, float((0.5 - (x / scale - codes).abs()).min())


def _attention(path, layer, x, pos, rows):
    """(output, context, V, margin of the cache rows' codes) of the attention block on x [n, 2048] at positions pos..."""
    w = functools.partial(_weights, path)
    n, name = len(x), "blk.%d." % layer
    at = torch.arange(pos, pos + n, device="cuda")
    xn = _norm(x, w(name + "attn_norm.weight"))
    values = xn @ w(name + "attn_v.weight").T
    k = _norm((xn @ w(name + "attn_k.weight").T).reshape(n, 4, 128), w(name + "attn_k_norm.weight"))
    q = _norm((xn @ w(name + "attn_q.weight").T).reshape(n, 32, 128), w(name + "attn_q_norm.weight"))
    (k, near_k), (v, near_v), q = _int8_rows(_rope(k, at).reshape(n, 512)), _int8_rows(values), _rope(q, at)
    if rows:
        rk, rv, ks, vs = (torch.from_numpy(r).cuda().double() for r in rows)
        k, v = torch.cat([rk * ks.unsqueeze(1), k]), torch.cat([rv * vs.unsqueeze(1), v])
    unseen = torch.arange(pos + n, device="cuda") > at.unsqueeze(1)
    context = torch.empty(n, 32, 128, dtype=torch.float64, device="cuda")
    for head in range(32):
        g = slice(head // 8 * 128, head // 8 * 128 + 128)
        scores = (q[:, head] @ k[:, g].T / 128 ** 0.5).masked_fill(unseen, float("-inf"))
        context[:, head] = torch.softmax(scores, -1) @ v[:, g]
    context = context.reshape(n, 4096)
    return context @ w(name + "attn_output.weight").T, context, values, min(near_k, near_v)


def _moe(path, layer, x):
    """(weighted expert sum, ids, weights) of the expert block on x [n, 2048]."""
    w = functools.partial(_weights, path)
    name = "blk.%d." % layer
    xn = _norm(x, w(name + "ffn_norm.weight"))
    router = w(name + "ffn_gate_inp.weight")
    probs, ids = torch.softmax(xn @ router.T, -1).topk(8)
    probs, out = probs / probs.sum(-1, keepdim=True), torch.zeros_like(x)
    for e in ids.unique().tolist():
        token, rank = torch.where(ids == e)
        gate, up, down = (w(name + "ffn_%s_exps.weight" % m, e, len(router)) for m in ("gate", "up", "down"))
        g = xn[token] @ gate.T
        out.index_add_(0, token, probs[token, rank].unsqueeze(1) * ((torch.nn.functional.silu(g) * (xn[token] @ up.T)) @ down.T))
    return out, ids, probs


def exact(case, seed):
    """Single blocks only: in a whole call each layer works on INT8 cache rows that the layers
    before it decide, and a value near a rounding boundary has no one 64-bit result."""
    kind = case["kind"]
    if kind in ("prompt", "greedy") or case.get("act") == "q8_k_compat":
        return None
    path, (x, rows) = _model_of(case).path, _block_inputs(case, seed)
    x = torch.from_numpy(x).cuda().double()
    if kind == "head":
        xn = _norm(x, _weights(path, "output_norm.weight"))
        parts = next(p for p in (16, 8, 4, 2, 1) if case["vocab"] % p == 0)
        return {"norm": xn[0], "logits": torch.cat([xn @ _weights(path, "output.weight", i, parts).T for i in range(parts)], 1)[0]}
    if kind == "moe":
        moe, ids, weights = _moe(path, _block_layer(case), x)
        return {"out": (x + moe)[0], "moe": moe[0], "ids": ids[0], "weights": weights[0]}
    out, context, values, margin = _attention(path, _block_layer(case), x, case["pos"], rows)
    if kind == "attention":
        return {"out": out[0], "context": context[0], "values": values[0]}
    if margin < 2e-5 and case["pos"] < 2000:   # one code of a short cache's row shows in the outputs
        return None
    moe, _, _ = _moe(path, case["layer"], x + out)
    return {"ffn_in": x + out, "moe": moe, "out": x + out + moe}
