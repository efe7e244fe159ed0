"""The workloads a user of this library has it run, as cases to time and to
compare: products of Q8_0 weights, the whisper decoder, the pocket-TTS flow
LM with its flow head, the Mimi decoder, the FastConformer encoder (offline
and streaming) and the TDT / RNN-T greedy decoder.

Model widths are those of gorelaxor_amd/synth.py.  A case is a dict of plain
values; `prepare` makes weights and inputs from a seed (on the GPU, so that
it is quick), `run` is one pass through the public entry points, and `exact`
is the same result in 64 bits with plain torch.  `exact` rounds activations
to Q8_0 where the products do (that rounding is part of what they compute)
and keeps everything else in float64.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from gorelaxor_amd import kern
from gorelaxor_amd.conformer import ConformerEncoder, ConformerStream, frames_out, stream_geom
from gorelaxor_amd.mimi import MimiDecoder
from gorelaxor_amd.pocket import PocketLM
from gorelaxor_amd.rnnt import TransducerDecoder
from gorelaxor_amd.synth import (MIMI, NEMOTRON_STREAMING, PARAKEET_TDT_06B, POCKET_FLOW, POCKET_TTS_LM, RNNT_TDT,
                                 WHISPER_BASE_EN, WHISPER_LARGE_V3_TURBO, mimi_steps)
from gorelaxor_amd.whisper import Rules, WhisperDecoder, special_tokens

DEV = "cuda"
WHISPER = {"base": WHISPER_BASE_EN, "turbo": WHISPER_LARGE_V3_TURBO}


# ---------------------------------------------------------------- cases

def listed():
    return [
        # the smallest call: one activation row through one 1024 x 1024 matrix
        dict(name="linear_1x1024x1024", kind="linear", m=1, n=1024, k=1024, bias=False),
        # one row through 512 such matrices stacked: every weight from HBM
        dict(name="linear_1x524288x1024", kind="linear", m=1, n=524288, k=1024, bias=False),
        # an encoder's feed-forward product over 300 frames
        dict(name="linear_300x1024x4096", kind="linear", m=300, n=1024, k=4096, bias=True),
        # a 30 s window decoded greedily with the small model
        dict(name="whisper_base_window", kind="whisper", model="base", audio=1500, streams=1, prompt=4, steps=96,
             rules=False),
        # a window conditioned on the text before it: the prompt is the work
        dict(name="whisper_base_prompt", kind="whisper", model="base", audio=1500, streams=1, prompt=187, steps=0,
             rules=False),
        # eight windows served together with the large model
        dict(name="whisper_turbo_8_streams", kind="whisper", model="turbo", audio=1500, streams=8, prompt=4, steps=96,
             rules=False),
        # a sentence spoken: its text as a prefix, then 4 s of frames
        dict(name="pocket_speak", kind="pocket", prefix=37, frames=50, flow=True),
        # those frames' latents to audio as they come, one a call
        dict(name="mimi_16_latents", kind="mimi", latents=16, per_call=1),
        # one 10 s utterance through the whole encoder
        dict(name="conformer_1x1001", kind="conformer", layers=24, batch=1, frames=1001),
        # sixteen of unequal length through a few of its blocks
        dict(name="conformer_16x1001", kind="conformer", layers=4, batch=16, frames=1001),
        # a live transcription's next chunk (1.12 s), the caches full
        dict(name="conformer_stream_right13", kind="stream", layers=24, right=13, batch=1),
        # an utterance's tokens from its encoder output
        dict(name="tdt_125_frames", kind="rnnt", frames=125, head="tdt"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "whisper", "whisper", "pocket", "mimi", "conformer", "conformer", "stream",
                       "rnnt"])
    if kind == "linear":
        m = rng.choice([1, _log(rng, 2, 32), _log(rng, 16, 1000)])
        return dict(kind=kind, m=m, n=_log(rng, 64, 16384), k=32 * _log(rng, 2, 160), bias=rng.random() < 0.5)
    if kind == "whisper":
        streams = rng.choice([1, 1, 1, 2, 4, 8])
        return dict(kind=kind, model=rng.choice(["base", "turbo"]), audio=rng.choice([1500, rng.randint(97, 1500)]),
                    streams=streams, prompt=_log(rng, 1, 223) if streams == 1 else _log(rng, 1, 24),
                    steps=_log(rng, 1, 64), rules=streams == 1 and rng.random() < 0.4)
    if kind == "pocket":
        return dict(kind=kind, prefix=_log(rng, 1, 180), frames=_log(rng, 2, 100), flow=rng.random() < 0.6)
    if kind == "mimi":
        return dict(kind=kind, latents=_log(rng, 1, 40), per_call=rng.choice([1, 1, 2, 3, 4]))
    if kind == "conformer":
        batch = _log(rng, 1, 16)
        return dict(kind=kind, layers=rng.randint(2, 6), batch=batch, frames=_log(rng, 60, min(3001, 16016 // batch)))
    if kind == "stream":
        return dict(kind=kind, layers=rng.randint(3, 8), right=rng.choice([13, 6, 1, 0]), batch=_log(rng, 1, 16))
    return dict(kind=kind, frames=_log(rng, 16, 400), head=rng.choice(["tdt", "tdt", "rnnt"]))


# ---------------------------------------------------------------- weights and inputs

class _Gen:
    """Tensors drawn on the GPU from one seed, in the order asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, *shape, scale=1.0, base=0.0):
        return torch.randn(*shape, generator=self.g, device=DEV) * scale + base

    def ints(self, n, lo, hi):
        return torch.randint(lo, hi, (n,), generator=self.g, device=DEV)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def q8(self, rows, cols, gain=1.0):
        """A trained-like Q8_0 matrix: normal values, rounded block by block."""
        return _to_q8(self.normal(rows, cols, scale=gain / math.sqrt(cols)))


class _Q8:
    """A Q8_0 matrix as ggml bytes on the GPU."""

    def __init__(self, data, rows, cols):
        self.data, self.rows, self.cols = data, rows, cols

    def numpy(self):
        return self.data.reshape(-1).cpu().numpy()

    def f64(self):
        d = self.data[:, :2].contiguous().view(torch.float16).double()
        return (self.data[:, 2:].contiguous().view(torch.int8).double() * d).reshape(self.rows, self.cols)


def _to_q8(w):
    """Weight.ToQ8: the scale amax/127 stored as float16, values rounded with
    the float32 scale, halves away from zero."""
    rows, cols = w.shape
    b = w.reshape(-1, 32).float()
    d = b.abs().amax(1, keepdim=True) / 127.0
    p = b * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    q = (torch.sign(p) * torch.floor(p.abs() + 0.5)).to(torch.int8)
    return _Q8(torch.cat([d.half().view(torch.uint8).reshape(-1, 2), q.view(torch.uint8)], 1), rows, cols)


def _host(t):
    return t.numpy() if isinstance(t, _Q8) else t.cpu().numpy()


def _bind(model, tensors):
    for name, t in tensors.items():
        model.set_tensor(name, _host(t))


def _whisper_hp(c):
    return dict(WHISPER[c["model"]], n_audio_ctx=c["audio"])


def _whisper_tensors(c, g):
    hp = _whisper_hp(c)
    st, t = hp["n_state"], {}
    t["decoder.token_embedding.weight"] = g.q8(hp["n_vocab"], st, gain=0.3 * math.sqrt(st))
    t["decoder.positional_embedding"] = g.normal(hp["n_text_ctx"] * st, scale=0.1)
    lns = ["decoder.ln"]
    for i in range(hp["n_layer"]):
        p = f"decoder.blocks.{i}."
        lns += [p + "attn_ln", p + "cross_attn_ln", p + "mlp_ln"]
        for a in ("attn", "cross_attn"):
            for w in ("query", "key", "value", "out"):
                t[p + f"{a}.{w}.weight"] = g.q8(st, st, gain=1.5)
            for b in ("query", "value", "out"):
                t[p + f"{a}.{b}.bias"] = g.normal(st, scale=0.1)
        t[p + "mlp.0.weight"], t[p + "mlp.0.bias"] = g.q8(4 * st, st, gain=1.2), g.normal(4 * st, scale=0.1)
        t[p + "mlp.2.weight"], t[p + "mlp.2.bias"] = g.q8(st, 4 * st, gain=1.2), g.normal(st, scale=0.1)
    for n in lns:
        t[n + ".weight"], t[n + ".bias"] = g.normal(st, scale=0.1, base=1.0), g.normal(st, scale=0.1)
    return t


def _whisper_inputs(c, g):
    hp = _whisper_hp(c)
    enc = g.normal(c["streams"], c["audio"], hp["n_state"])
    prompts = g.ints(c["streams"] * c["prompt"], 0, 50256).reshape(c["streams"], -1)
    return enc, prompts


def _pocket_hp(c):
    return dict(POCKET_TTS_LM, max_pos=max(POCKET_TTS_LM["max_pos"], c["prefix"] + c["frames"]))


def _pocket_tensors(c, g):
    hp, fhp, t = _pocket_hp(c), POCKET_FLOW, {}
    d, ff, ld, D = hp["d"], hp["ff"], hp["ldim"], fhp["dim"]
    for i in range(hp["n_layer"]):
        p = f"lm.blk.{i}."
        for n in ("norm1", "norm2"):
            t[p + n + ".weight"], t[p + n + ".bias"] = g.normal(d, scale=0.1, base=1.0), g.normal(d, scale=0.02)
        t[p + "attn_qkv.weight"], t[p + "attn_out.weight"] = g.q8(3 * d, d, gain=1.5), g.q8(d, d, gain=1.5)
        t[p + "ff1.weight"], t[p + "ff2.weight"] = g.q8(ff, d, gain=1.5), g.q8(d, ff, gain=1.5)
    t["lm.input.weight"], t["lm.bos"] = g.normal(d, ld, scale=0.2), g.normal(ld)
    t["lm.out_norm.weight"], t["lm.out_norm.bias"] = g.normal(d, scale=0.1, base=1.0), g.normal(d, scale=0.1)
    t["lm.eos.weight"], t["lm.eos.bias"] = g.normal(d, scale=0.05), g.normal(1, scale=0.1)
    f = {}
    if c["flow"]:
        f["flow.cond.weight"], f["flow.cond.bias"] = g.q8(D, d), g.normal(D, scale=0.1)
        f["flow.input.weight"], f["flow.input.bias"] = g.normal(D, ld, scale=1 / math.sqrt(ld)), g.normal(D, scale=0.1)
        for i in range(2):
            p = f"flow.time.{i}."
            f[p + "freqs"] = torch.exp(-math.log(1e4) * torch.arange(128, dtype=torch.float64, device=DEV) / 128).float()
            f[p + "fc1.weight"], f[p + "fc1.bias"] = g.q8(D, 256), g.normal(D, scale=0.1)
            f[p + "fc2.weight"], f[p + "fc2.bias"] = g.q8(D, D), g.normal(D, scale=0.1)
            f[p + "norm.alpha"] = g.normal(D, scale=0.1, base=1.0)
        for i in range(fhp["depth"]):
            p = f"flow.res.{i}."
            f[p + "norm.weight"], f[p + "norm.bias"] = g.normal(D, scale=0.1, base=1.0), g.normal(D, scale=0.1)
            f[p + "fc1.weight"], f[p + "fc1.bias"] = g.q8(D, D), g.normal(D, scale=0.1)
            f[p + "fc2.weight"], f[p + "fc2.bias"] = g.q8(D, D, gain=0.5), g.normal(D, scale=0.1)
            f[p + "ada.weight"], f[p + "ada.bias"] = g.q8(3 * D, D, gain=0.5), g.normal(3 * D, scale=0.1)
        f["flow.final.ada.weight"], f["flow.final.ada.bias"] = g.q8(2 * D, D, gain=0.5), g.normal(2 * D, scale=0.1)
        f["flow.final.out.weight"] = g.normal(ld, D, scale=1 / math.sqrt(D))
        f["flow.final.out.bias"] = g.normal(ld, scale=0.1)
    return t, f


def _pocket_inputs(c, g):
    hp = _pocket_hp(c)
    return g.normal(c["prefix"], hp["d"]), g.normal(c["frames"], hp["ldim"])


def _mimi_tensors(g):
    hp, t = MIMI, {}
    d, ff = hp["d"], hp["ff"]

    def mat(rows, cols, gain=1.0):  # the converter's typing: Q8_0 from 64 x 64 on, else float32
        if rows >= 64 and cols >= 64 and cols % 32 == 0:
            return g.q8(rows, cols, gain)
        return g.normal(rows, cols, scale=gain / math.sqrt(cols))

    t["mimi.quant"], t["mimi.up"] = mat(d, hp["ldim"]), g.normal(d, 2 * hp["up_s"], scale=0.3)
    for i in range(hp["n_layer"]):
        p = f"mimi.dec_tf.{i}."
        for n in ("norm1", "norm2"):
            t[p + n + ".weight"], t[p + n + ".bias"] = g.normal(d, scale=0.1, base=1.0), g.normal(d, scale=0.1)
        t[p + "attn_qkv.weight"], t[p + "attn_out.weight"] = mat(3 * d, d), mat(d, d)
        t[p + "ff1.weight"], t[p + "ff2.weight"] = mat(ff, d), mat(d, ff, 0.5)
        t[p + "ls1"], t[p + "ls2"] = g.normal(d, scale=0.05, base=0.2), g.normal(d, scale=0.05, base=0.2)
    for kind, name, _, cin, cout, k, _, _ in mimi_steps(hp):
        if kind == "conv":
            t[name + ".weight"], t[name + ".bias"] = mat(cout, k * cin), g.normal(cout, scale=0.1)
        elif kind == "convtr":
            t[name + ".weight"], t[name + ".bias"] = mat(k * cout, cin), g.normal(cout, scale=0.1)
        else:
            t[name + ".1.weight"], t[name + ".1.bias"] = mat(cout, k * cin), g.normal(cout, scale=0.1)
            t[name + ".3.weight"], t[name + ".3.bias"] = mat(cin, cout, 0.5), g.normal(cin, scale=0.1)
    return t


def _conf_hp(c):
    return dict(NEMOTRON_STREAMING if c["kind"] == "stream" else PARAKEET_TDT_06B, layers=c["layers"])


def _causal(hp):
    return hp.get("att_style", "regular") == "chunked_limited"


def _sub_out(n, causal):
    return n // 2 + 1 if causal else (n - 1) // 2 + 1


def _conf_tensors(c, g):
    """As converted files hold them: linears Q8_0, pointwise convolutions
    float16 (rounded to Q8_0 at load), the pre-encoder's 1x1s float32."""
    hp, t = _conf_hp(c), {}
    d, ch, ff, K, F = hp["d"], hp["sub_channels"], hp["dff"], hp["conv_kernel"], hp["n_mels"]
    for _ in range(3):
        F = _sub_out(F, _causal(hp))
    pe = "enc.pre_encode."
    for n in ("conv.0", "conv.2", "conv.5"):
        t[pe + n + ".weight"], t[pe + n + ".bias"] = g.normal(ch * 9, scale=0.3), g.normal(ch, scale=0.1)
    for n in ("conv.3", "conv.6"):
        t[pe + n + ".weight"], t[pe + n + ".bias"] = g.normal(ch, ch, scale=1 / math.sqrt(ch)), g.normal(ch, scale=0.1)
    t[pe + "out.weight"], t[pe + "out.bias"] = g.q8(d, ch * F), g.normal(d, scale=0.1)
    for i in range(hp["layers"]):
        p = f"enc.blocks.{i}."
        for f in ("ff1", "ff2"):
            t[p + f + ".linear1.weight"], t[p + f + ".linear1.bias"] = g.q8(ff, d), g.normal(ff, scale=0.1)
            t[p + f + ".linear2.weight"], t[p + f + ".linear2.bias"] = g.q8(d, ff), g.normal(d, scale=0.1)
        for n in ("norm_ff1", "norm_ff2", "norm_attn", "norm_conv", "norm_out"):
            t[p + n + ".weight"], t[p + n + ".bias"] = g.normal(d, scale=0.1, base=1.0), g.normal(d, scale=0.1)
        for n in ("linear_q", "linear_k", "linear_v", "linear_out"):
            t[p + f"attn.{n}.weight"], t[p + f"attn.{n}.bias"] = g.q8(d, d), g.normal(d, scale=0.1)
        t[p + "attn.linear_pos.weight"] = g.q8(d, d)
        t[p + "attn.pos_bias_u"], t[p + "attn.pos_bias_v"] = g.normal(d, scale=0.1), g.normal(d, scale=0.1)
        for n, rows in (("pointwise1", 2 * d), ("pointwise2", d)):
            t[p + f"conv.{n}.weight"] = g.normal(rows, d, scale=1 / math.sqrt(d)).half()
            t[p + f"conv.{n}.bias"] = g.normal(rows, scale=0.1)
        t[p + "conv.depthwise.weight"], t[p + "conv.depthwise.bias"] = g.normal(d * K, scale=0.3), g.normal(d, scale=0.1)
        t[p + "conv.bn.weight"], t[p + "conv.bn.bias"] = g.normal(d, scale=0.1, base=1.0), g.normal(d, scale=0.1)
        t[p + "conv.bn.running_mean"] = g.normal(d, scale=0.1)
        t[p + "conv.bn.running_var"] = g.uniform(d, lo=0.5, hi=1.5)
    return t


def _mel(c, g):
    """Per-feature normalized log-mel frames and the valid ones of each
    utterance (a batch's are of unequal length)."""
    mel = g.normal(c["batch"], PARAKEET_TDT_06B["n_mels"], c["frames"])
    short = g.uniform(c["batch"]).tolist()
    valid = [max(1, c["frames"] - 1 - (int(0.4 * s * c["frames"]) if c["batch"] > 1 else 0)) for s in short]
    return mel, valid


def _stream_chunks(c, g):
    """Chunk mels [batch][mels][frames] of a session: the first, enough to
    fill the left context, and the one that `run` takes; every frame real."""
    geo = stream_geom(_conf_hp(c), c["right"])
    before = 2 + geo["left"] // geo["chunk"]
    out = []
    for j in range(before + 1):
        nf = geo["mel_first"] if j == 0 else geo["mel_cache"] + geo["mel_next"]
        out.append(g.normal(c["batch"], PARAKEET_TDT_06B["n_mels"], nf))
    return geo, out


def _rnnt_hp(c):
    return dict(RNNT_TDT) if c["head"] == "tdt" else dict(RNNT_TDT, head_kind="rnnt", durations=[])


def _rnnt_tensors(c, g):
    hp, t = _rnnt_hp(c), {}
    H, V, J, nd = hp["pred_hidden"], hp["pred_vocab"], hp["joint_hidden"], len(hp["durations"])
    t["pred.embed.weight"] = g.normal(V, H, scale=0.5)
    for i in range(hp["pred_layers"]):
        p = f"pred.lstm.{i}."
        t[p + "Wx"], t[p + "Wh"], t[p + "bias"] = g.q8(4 * H, H), g.q8(4 * H, H), g.normal(4 * H, scale=0.1)
    t["joint.enc.weight"], t["joint.enc.bias"] = g.q8(J, hp["d"]), g.normal(J, scale=0.1)
    t["joint.pred.weight"], t["joint.pred.bias"] = g.q8(J, H, gain=4.0), g.normal(J, scale=0.1)
    t["joint.out.weight"], t["joint.out.bias"] = g.q8(V + nd, J), g.normal(V + nd, scale=0.1)
    t["joint.out.bias"][V - 1] += 3.0  # frames advance as well as emit: about a token in two or three frames
    return t


# ---------------------------------------------------------------- prepare and run

def prepare(case, seed):
    c, g = case, _Gen(seed)
    if c["kind"] == "linear":
        w = kern.NewQ8(c["n"], c["k"], g.q8(c["n"], c["k"]).numpy())
        s = dict(w=w, x=g.normal(c["m"], c["k"]), bias=g.normal(c["n"], scale=0.1) if c["bias"] else None,
                 dst=torch.empty(c["m"], c["n"], device=DEV))
    elif c["kind"] == "whisper":
        dec = WhisperDecoder(_whisper_hp(c), streams=c["streams"])
        _bind(dec, _whisper_tensors(c, g))
        enc, prompts = _whisper_inputs(c, g)
        sp = special_tokens(_whisper_hp(c)["n_vocab"])
        s = dict(dec=dec, enc=_host(enc), prompts=_host(prompts).astype(np.int32),
                 rules=Rules(sp, (1, 2, 7, 8, 9, 10, 220), space=220, n_audio_ctx=c["audio"]))
    elif c["kind"] == "pocket":
        lm = PocketLM(_pocket_hp(c))
        t, f = _pocket_tensors(c, g)
        _bind(lm, t)
        if c["flow"]:
            lm.flow_init(POCKET_FLOW["dim"], POCKET_FLOW["depth"], POCKET_FLOW["steps"])
            _bind(lm, f)
        text, rows = _pocket_inputs(c, g)
        s = dict(lm=lm, text=_host(text), rows=_host(rows))
    elif c["kind"] == "mimi":
        dec = MimiDecoder(MIMI, max_latents=c["per_call"])
        _bind(dec, _mimi_tensors(g))
        s = dict(dec=dec, lat=_host(g.normal(c["latents"], MIMI["ldim"])))
    elif c["kind"] == "conformer":
        enc = ConformerEncoder(_conf_hp(c))
        _bind(enc, _conf_tensors(c, g))
        mel, valid = _mel(c, g)
        s = dict(enc=enc, mel=mel, valid=valid,
                 out=torch.empty(c["batch"], frames_out(c["frames"]), enc.hp["d"], device=DEV))
    elif c["kind"] == "stream":
        enc = ConformerEncoder(_conf_hp(c))
        _bind(enc, _conf_tensors(c, g))
        geo, chunks = _stream_chunks(c, g)
        stream = ConformerStream(enc, c["right"], batch=c["batch"])
        out = torch.empty(c["batch"], geo["chunk"], enc.hp["d"], device=DEV)
        torch.cuda.synchronize()
        for ch in chunks[:-1]:
            stream.step_dev(ch.data_ptr(), ch.shape[2], ch.shape[2], out.data_ptr())
        s = dict(stream=stream, mel=chunks[-1], out=out)
    else:
        dec = TransducerDecoder(_rnnt_hp(c))
        _bind(dec, _rnnt_tensors(c, g))
        s = dict(dec=dec, enc=g.normal(c["frames"], dec.hp["d"]))
    torch.cuda.synchronize()  # inputs come from torch's stream, the library has its own
    return dict(case=c, **s)


def _column(values, n, dtype):
    """The tokens' values, as many of them as there are, in n places."""
    out = np.zeros(n, dtype)
    out[:min(n, len(values))] = values[:n]
    return out


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "linear":
        kern.matmul_dev(s["dst"], s["x"], c["m"], s["w"], s["bias"])
        return s["dst"]
    if c["kind"] == "whisper":
        dec = s["dec"]
        dec.reset()
        if c["streams"] > 1:
            for i in range(c["streams"]):
                dec.set_encoder_output_stream(i, s["enc"][i])
            first = dec.greedy_streams(s["prompts"], 0)
            begun = np.stack([dec.logits(i) for i in range(c["streams"])])
            toks = dec.steps(c["steps"])
            return dict(prompt_logits=begun, first=first, tokens=toks,
                        logits=np.stack([dec.logits(i) for i in range(c["streams"])]))
        dec.set_encoder_output(s["enc"][0])
        logits, tok = dec.decode(s["prompts"][0])
        out = dict(prompt_logits=logits, first=tok)
        if c["rules"]:
            toks, end = dec.rules_loop(s["rules"], 0, 3000, c["steps"])
            n = c["steps"]
            out.update(ids=_column([t["id"] for t in toks], n, np.int64), tids=_column([t["tid"] for t in toks], n, np.int64),
                       p=_column([t["p"] for t in toks], n, np.float32),
                       plog=_column([t["plog"] for t in toks], n, np.float32), end=end)
        elif c["steps"]:
            out.update(tokens=dec.steps(c["steps"]), logits=dec.logits())
        return out
    if c["kind"] == "pocket":
        lm = s["lm"]
        lm.reset()
        text = lm.run(s["text"])
        rows, eos = lm.speak(s["rows"]) if c["flow"] else lm.frames(s["rows"])
        return dict(text=text, rows=rows, eos=eos)
    if c["kind"] == "mimi":
        s["dec"].reset()
        step = c["per_call"]
        return np.concatenate([s["dec"].decode(s["lat"][i:i + step]) for i in range(0, c["latents"], step)])
    if c["kind"] == "conformer":
        s["enc"].encode_dev(s["mel"].data_ptr(), c["batch"], c["frames"], s["valid"], s["out"].data_ptr())
        return s["out"]
    if c["kind"] == "stream":
        nf = s["mel"].shape[2]
        rows = s["stream"].step_dev(s["mel"].data_ptr(), nf, nf, s["out"].data_ptr())
        return dict(rows=rows, out=s["out"])
    st = s["dec"].new_state()
    toks = s["dec"].decode_dev(s["enc"].data_ptr(), c["frames"], st)
    h, cc, last = st.read()
    n = 10 * c["frames"]
    return dict(ids=_column([t.ID for t in toks], n, np.int64), frames=_column([t.Frame for t in toks], n, np.int64),
                durations=_column([t.Duration for t in toks], n, np.int64), p=_column([t.P for t in toks], n, np.float32),
                h=h, c=cc, last=last)


# ---------------------------------------------------------------- work

def _q8_bytes(vals):
    return vals * 34 / 32


def work(case):
    """Bytes: weights once for each step that needs the one before it, inputs
    and outputs once, keys and values once a step.  Operations: 2 for each
    multiply-add of the products and the attention."""
    c = case
    if c["kind"] == "linear":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=_q8_bytes(n * k) + 4 * (m * k + m * n + (n if c["bias"] else 0)), flops=2 * m * n * k)
    if c["kind"] == "whisper":
        hp, S = _whisper_hp(c), c["streams"]
        d, L, V, A = hp["n_state"], hp["n_layer"], hp["n_vocab"], c["audio"]
        mats, P, N = L * (6 * d * d + 8 * d * d), c["prompt"], c["steps"]
        cross, keys = 2 * L * A * d, 2 * L * d * sum(P + i + 1 for i in range(N))
        rows = S * (P + N)
        return dict(bytes=S * 4 * A * d + _q8_bytes(2 * L * d * d) + (1 + N) * (_q8_bytes(mats + V * d) + S * 4 * cross)
                    + S * 4 * (keys + 2 * V),
                    flops=2 * (S * A * 2 * L * d * d + rows * (mats + cross) + S * (1 + N) * V * d + S * keys))
    if c["kind"] == "pocket":
        hp, D, ld = _pocket_hp(c), POCKET_FLOW["dim"], POCKET_TTS_LM["ldim"]
        d, L, T, N = hp["d"], hp["n_layer"], c["prefix"], c["frames"]
        mats = L * (4 * d * d + 2 * d * hp["ff"])
        flow = D * d + POCKET_FLOW["depth"] * 5 * D * D + 2 * D * D if c["flow"] else 0
        kv = 2 * L * d * sum(T + i + 1 for i in range(N))
        return dict(bytes=(N + 1) * _q8_bytes(mats) + N * (_q8_bytes(flow) + 4 * ld * d) + 4 * (kv + T * d),
                    flops=2 * ((T + N) * mats + N * (flow + ld * d) + kv + L * d * T * (T + 1)))
    if c["kind"] == "mimi":
        hp, n, calls = MIMI, c["latents"], -(-c["latents"] // c["per_call"])
        d, rows = hp["d"], hp["up_s"]
        w, f = hp["n_layer"] * (4 * d * d + 2 * d * hp["ff"]), 0
        f = w * rows + 2 * d * hp["n_layer"] * rows * hp["context"]
        for kind, _, _, cin, cout, k, stride, _ in mimi_steps(hp):
            per = cin * cout * (k + 1) if kind == "res" else cin * cout * k
            w, f = w + per, f + per * rows
            rows *= stride if kind == "convtr" else 1
        return dict(bytes=calls * _q8_bytes(w) + n * 4 * rows, flops=2 * n * f)
    if c["kind"] in ("conformer", "stream"):
        hp, B = _conf_hp(c), c["batch"]
        d, ff, L, ch = hp["d"], hp["dff"], c["layers"], hp["sub_channels"]
        F, cs = hp["n_mels"], _causal(hp)
        for _ in range(3):
            F = _sub_out(F, cs)
        if c["kind"] == "stream":
            geo = stream_geom(hp, c["right"])
            T, frames = geo["chunk"], geo["mel_cache"] + geo["mel_next"]
            keys, pos = geo["left"] + T, geo["left"] + 2 * T
            ring = 4 * B * L * (2 * keys * d + hp["conv_left"] * d)
        else:
            T, frames = frames_out(c["frames"]), c["frames"]
            keys, pos, ring = T, 2 * T - 1, 0
        lin = 4 * d * ff + 7 * d * d
        pre = 2 * ch * ch + d * ch * F
        return dict(bytes=_q8_bytes(L * (lin + d * d) + d * ch * F) + 8 * ch * ch + ring
                    + 4 * B * (frames * hp["n_mels"] + T * d),
                    flops=2 * (B * T * L * (lin + 3 * keys * d + d * hp["conv_kernel"]) + L * pos * d * d
                               + B * T * (pre + 8 * F * ch * ch)))
    hp = _rnnt_hp(c)
    H, V, J, T = hp["pred_hidden"], hp["pred_vocab"] + len(hp["durations"]), hp["joint_hidden"], c["frames"]
    lstm, joint = hp["pred_layers"] * 8 * H * H + J * H, V * J
    steps = T * 0.4  # emissions; every frame's joint besides
    return dict(bytes=_q8_bytes(J * hp["d"]) + 4 * T * hp["d"] + steps * _q8_bytes(lstm) + T * _q8_bytes(joint),
                flops=2 * (T * J * hp["d"] + steps * lstm + T * joint))


def tolerance(case):
    """A product against 64 bits is off by 1e-7 to 2e-7, whatever the order of
    its sums within that.  A model is off by 0.7 to 1.9 %: one activation on
    the edge between two int8 values falls the other way after any other
    rounding before it, and the blocks that follow turn that into as much
    difference as the rounding to Q8_0 itself makes."""
    if case["kind"] == "linear":
        return dict(rel=1e-6, max=3e-5, differ=0.0)
    return dict(rel=0.03, max=0.9, differ=0.01)


# ---------------------------------------------------------------- the same in 64 bits

def _f64(t):
    return t.f64() if isinstance(t, _Q8) else t.double()


def _round(x):
    """x with each 32 values of a row rounded to Q8_0, as the int8 products
    take their activations (in x's own precision), as float64."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    inv = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
    sc = amax * torch.tensor(1 / 127, dtype=torch.float32 if x.dtype == torch.float32 else torch.float64, device=x.device)
    return (torch.round(b * inv).double() * sc.double()).reshape(x.shape)


def _lin(x, w, b=None):
    """The int8 route of a Q8_0 weight, the float route of a float32 one."""
    y = (_round(x) if isinstance(w, _Q8) else x.double()) @ _f64(w).T
    return y if b is None else y + b.double()


def _flin(x, w, b=None):
    """The float route whatever the weight's type."""
    y = x @ _f64(w).T
    return y if b is None else y + b.double()


def _ln(x, w=None, b=None, eps=1e-5):
    y = (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + eps)
    return y if w is None else y * w.double() + b.double()


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * x * (1 + 0.044715 * x * x)))


def _silu(x):
    return x * torch.sigmoid(x)


def _elu(x):
    return torch.where(x > 0, x, torch.expm1(torch.clamp(x, max=0)))


def _heads(x, h):
    return x.reshape(x.shape[0], h, -1).transpose(0, 1).contiguous()


def _attend(q, k, v, mask=None):
    """[heads][rows][width] each; mask [rows][keys] True where seen."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[2])
    if mask is not None:
        s = s.masked_fill(~mask, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v).transpose(0, 1).reshape(q.shape[1], -1)


def _rope(x, heads, pos, period):
    hd = x.shape[1] // heads
    f = period ** (-2.0 * torch.arange(hd // 2, dtype=torch.float64, device=DEV) / hd)
    a = (pos.double()[:, None] * f)[:, None, :]
    y = x.reshape(x.shape[0], heads, hd // 2, 2)
    r, i = y[..., 0], y[..., 1]
    return torch.stack([r * a.cos() - i * a.sin(), r * a.sin() + i * a.cos()], -1).reshape(x.shape)


def _exact_whisper(c, seed):
    g = _Gen(seed)
    t = _whisper_tensors(c, g)
    enc, prompts = _whisper_inputs(c, g)
    hp = _whisper_hp(c)
    H, emb, out = hp["n_head"], t["decoder.token_embedding.weight"], []
    embf = emb.f64()
    for s in range(c["streams"]):
        x = embf[prompts[s]] + t["decoder.positional_embedding"].double().reshape(-1, hp["n_state"])[:c["prompt"]]
        mask = torch.ones(c["prompt"], c["prompt"], dtype=torch.bool, device=DEV).tril()
        for i in range(hp["n_layer"]):
            p = f"decoder.blocks.{i}."
            n = lambda z, ln: _ln(z, t[p + ln + ".weight"], t[p + ln + ".bias"])  # noqa: E731
            W = lambda z, w: _lin(z, t[p + w + ".weight"], t.get(p + w + ".bias"))  # noqa: E731
            h = n(x, "attn_ln")
            a = _attend(*(_heads(W(h, "attn." + w), H) for w in ("query", "key", "value")), mask)
            x = x + W(a, "attn.out")
            q = _heads(W(n(x, "cross_attn_ln"), "cross_attn.query"), H)
            a = _attend(q, _heads(W(enc[s], "cross_attn.key"), H), _heads(W(enc[s], "cross_attn.value"), H))
            x = x + W(a, "cross_attn.out")
            x = x + W(_gelu(W(n(x, "mlp_ln"), "mlp.0")), "mlp.2")
        out.append(_lin(_ln(x[-1:], t["decoder.ln.weight"], t["decoder.ln.bias"]), emb)[0])
    # the tokens after the prompt hang on near ties of a random model's logits
    return dict(prompt_logits=torch.stack(out) if c["streams"] > 1 else out[0])


def _pocket_rows(hp, t, x, cache):
    """Rows x after the cached positions, through the transformer."""
    H, d = hp["heads"], hp["d"]
    pos0 = cache[0][0].shape[0] if cache[0] is not None else 0
    T = x.shape[0]
    pos = torch.arange(pos0, pos0 + T, device=DEV)
    mask = torch.arange(pos0 + T, device=DEV)[None, :] <= pos[:, None]
    for i in range(hp["n_layer"]):
        p = f"lm.blk.{i}."
        qkv = _lin(_ln(x, t[p + "norm1.weight"], t[p + "norm1.bias"]), t[p + "attn_qkv.weight"])
        q, k, v = (_rope(qkv[:, :d], H, pos, hp["period"]), _rope(qkv[:, d:2 * d], H, pos, hp["period"]), qkv[:, 2 * d:])
        if cache[i] is not None:
            k, v = torch.cat([cache[i][0], k]), torch.cat([cache[i][1], v])
        cache[i] = (k, v)
        x = x + _lin(_attend(_heads(q, H), _heads(k, H), _heads(v, H), mask), t[p + "attn_out.weight"])
        h = _gelu(_lin(_ln(x, t[p + "norm2.weight"], t[p + "norm2.bias"]), t[p + "ff1.weight"]))
        x = x + _lin(h, t[p + "ff2.weight"])
    return _ln(x[-1:], t["lm.out_norm.weight"], t["lm.out_norm.bias"])


def _exact_pocket(c, seed):
    g = _Gen(seed)
    t, f = _pocket_tensors(c, g)
    text, rows = _pocket_inputs(c, g)
    hp, fhp = _pocket_hp(c), POCKET_FLOW
    W = {k: _f64(v) for k, v in f.items()}
    cache = [None] * hp["n_layer"]
    first = _pocket_rows(hp, t, text.double(), cache)
    fl = lambda z, n: z @ W[n + ".weight"].T + W[n + ".bias"]  # noqa: E731

    def embed(e, time):
        p = f"flow.time.{e}"
        a = time * W[p + ".freqs"]
        y = fl(_silu(fl(torch.cat([a.cos(), a.sin()]), p + ".fc1")), p + ".fc2")
        return y * W[p + ".norm.alpha"] / torch.sqrt(y.var(unbiased=True) + 1e-5)

    conds = [(embed(0, i / fhp["steps"]) + embed(1, (i + 1) / fhp["steps"])) / 2
             for i in range(fhp["steps"])] if c["flow"] else []

    def flow(out, x):
        y0 = fl(out, "flow.cond")
        for cond in conds:
            sy, h = _silu(y0 + cond), fl(x, "flow.input")
            for i in range(fhp["depth"]):
                p = f"flow.res.{i}"
                shift, scale, gate = fl(sy, p + ".ada").chunk(3, -1)
                n = _ln(h, W[p + ".norm.weight"], W[p + ".norm.bias"], 1e-6) * (1 + scale) + shift
                h = h + gate * fl(_silu(fl(n, p + ".fc1")), p + ".fc2")
            shift, scale = fl(sy, "flow.final.ada").chunk(2, -1)
            x = x + fl(_ln(h, eps=1e-6) * (1 + scale) + shift, "flow.final.out") / len(conds)
        return x

    lat, outs, eos = t["lm.bos"].double(), [], []
    for i in range(c["frames"]):
        feed = lat if c["flow"] else rows[i].double()
        out = _pocket_rows(hp, t, feed[None] @ t["lm.input.weight"].double().T, cache)[0]
        eos.append(out @ t["lm.eos.weight"].double() + t["lm.eos.bias"].double()[0])
        if c["flow"]:
            lat = flow(out, rows[i].double())
        outs.append(lat if c["flow"] else out)
    return dict(text=first[0], rows=torch.stack(outs), eos=torch.stack(eos))


def _exact_mimi(c, seed):
    g = _Gen(seed)
    t, hp = _mimi_tensors(g), MIMI
    lat = g.normal(c["latents"], hp["ldim"]).double()
    d, H, S, n = hp["d"], hp["heads"], hp["up_s"], c["latents"]
    z, up = _lin(lat, t["mimi.quant"]), t["mimi.up"].double()
    full = torch.zeros((n + 1) * S, d, dtype=torch.float64, device=DEV)
    for j in range(2 * S):
        full[j:j + n * S:S] += z * up[:, j]
    x, T = full[:n * S], n * S
    pos = torch.arange(T, device=DEV)
    mask = (pos[None, :] <= pos[:, None]) & (pos[None, :] > pos[:, None] - hp["context"])
    for i in range(hp["n_layer"]):
        p = f"mimi.dec_tf.{i}."
        qkv = _lin(_ln(x, t[p + "norm1.weight"], t[p + "norm1.bias"]), t[p + "attn_qkv.weight"])
        q, k = (_rope(qkv[:, o:o + d], H, pos, hp["period"]) for o in (0, d))
        a = _attend(_heads(q, H), _heads(k, H), _heads(qkv[:, 2 * d:], H), mask)
        x = x + t[p + "ls1"].double() * _lin(a, t[p + "attn_out.weight"])
        h = _gelu(_lin(_ln(x, t[p + "norm2.weight"], t[p + "norm2.bias"]), t[p + "ff1.weight"]))
        x = x + t[p + "ls2"].double() * _lin(h, t[p + "ff2.weight"])

    def conv(name, x, cin, k, stride, dil):
        w, past = t[name + ".weight"], (k - 1) * dil + 1 - stride
        xp = torch.cat([torch.zeros(past, cin, dtype=torch.float64, device=DEV), x])
        xp = _round(xp) if isinstance(w, _Q8) else xp
        w = _f64(w).reshape(w.rows if isinstance(w, _Q8) else w.shape[0], k, cin)
        rows = x.shape[0] // stride
        y = t[name + ".bias"].double().expand(rows, -1).clone()
        for j in range(k):
            y += xp[j * dil:j * dil + (rows - 1) * stride + 1:stride] @ w[:, j].T.contiguous()
        return y

    for kind, name, el, cin, cout, k, stride, dil in mimi_steps(hp):
        x = _elu(x) if el else x
        if kind == "conv":
            x = conv(name, x, cin, k, stride, dil)
        elif kind == "convtr":
            zz = _lin(x, t[name + ".weight"]).reshape(-1, k, cout)
            T = x.shape[0]
            full = t[name + ".bias"].double().expand((T - 1) * stride + k, -1).clone()
            for j in range(k):
                full[j:j + (T - 1) * stride + 1:stride] += zz[:, j]
            x = full[:T * stride]
        else:
            x = x + conv(name + ".3", _elu(conv(name + ".1", _elu(x), cin, k, 1, dil)), cout, 1, 1, 1)
    return x[:, 0]


def _subsample(hp, t, mel, valid):
    """The pre-encoder: mel [mels][frames] -> (rows, valid rows)."""
    cs, ch = _causal(hp), hp["sub_channels"]
    pl, pe = (2 if cs else 1), "enc.pre_encode."
    x = mel.double().T.clone()
    x[valid:] = 0

    def conv(x, name, depthwise):
        T, F = x.shape[:2]
        T1, F1 = _sub_out(T, cs), _sub_out(F, cs)
        pad = torch.zeros(2 * T1 + 2, 2 * F1 + 2, *x.shape[2:], dtype=torch.float64, device=DEV)
        pad[pl:pl + T, pl:pl + F] = x
        w = t[pe + name + ".weight"].double().reshape(ch, 3, 3)
        y = t[pe + name + ".bias"].double().expand(T1, F1, -1).clone()
        for i in range(3):
            for j in range(3):
                tap = pad[i:i + 2 * T1:2, j:j + 2 * F1:2]
                y += (tap if depthwise else tap[..., None]) * w[:, i, j]
        return y

    L = _sub_out(valid, cs)
    x = conv(x, "conv.0", False)
    x[L:] = 0
    x = torch.relu(x)
    for dw, pw in (("conv.2", "conv.3"), ("conv.5", "conv.6")):
        x, L = conv(x, dw, True), _sub_out(L, cs)
        x[L:] = 0
        x = _lin(x, t[pe + pw + ".weight"], t[pe + pw + ".bias"])
        x[L:] = 0
        x = torch.relu(x)
    x = x.transpose(1, 2).reshape(x.shape[0], -1)
    return _lin(x, t[pe + "out.weight"], t[pe + "out.bias"]), max(0, min(L, x.shape[0]))


def _conf_block(hp, t, i, x, L, mask, before=None, conv_before=None):
    """One block over rows x (L of them valid): mask [rows][keys] over the
    normalized rows `before` and these; returns (x, those rows, gated frames)."""
    d, H, K, T = hp["d"], hp["heads"], hp["conv_kernel"], x.shape[0]
    p = f"enc.blocks.{i}."
    n = lambda z, ln: _ln(z, t[p + ln + ".weight"], t[p + ln + ".bias"])  # noqa: E731
    W = lambda z, w: _lin(z, t[p + w + ".weight"], t.get(p + w + ".bias"))  # noqa: E731
    ff = lambda z, f: z + 0.5 * W(_silu(W(n(z, "norm_" + f), f + ".linear1")), f + ".linear2")  # noqa: E731
    x = ff(x, "ff1")
    h = n(x, "norm_attn")
    kv = h if before is None else torch.cat([before, h])
    c, Tk = kv.shape[0] - T, kv.shape[0]
    q = W(h, "attn.linear_q")
    k, v = _heads(W(kv, "attn.linear_k"), H), _heads(W(kv, "attn.linear_v"), H)
    rel = torch.arange(-(T - 1), Tk, dtype=torch.float64, device=DEV)  # query minus key
    ang = rel[:, None] * 10000.0 ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEV) / d)
    pos = _heads(W(torch.stack([ang.sin(), ang.cos()], -1).reshape(len(rel), d), "attn.linear_pos"), H)
    u, w = t[p + "attn.pos_bias_u"].double(), t[p + "attn.pos_bias_v"].double()
    bd = torch.matmul(_heads(q + w, H), pos.transpose(1, 2).contiguous())
    at = torch.arange(T, device=DEV)[:, None] + c - torch.arange(Tk, device=DEV)[None, :] + T - 1
    s = torch.matmul(_heads(q + u, H), k.transpose(1, 2).contiguous()) + bd.gather(2, at.expand(H, -1, -1))
    s = (s / math.sqrt(d // H)).masked_fill(~mask, -math.inf)
    a = torch.nan_to_num(torch.softmax(s, -1))  # a row that sees nothing gives zeros
    x = x + W(torch.matmul(a, v).transpose(0, 1).reshape(T, d), "attn.linear_out")
    z = W(n(x, "norm_conv"), "conv.pointwise1")
    gl = z[:, :d] * torch.sigmoid(z[:, d:])
    gl[L:] = 0
    chunked = hp.get("conv_left", -1) >= 0 and hp.get("conv_right", -1) >= 0
    pl = hp["conv_left"] if chunked else (K - 1) // 2
    pad = torch.zeros(T + K - 1, d, dtype=torch.float64, device=DEV)
    if conv_before is not None:
        pad[:pl] = conv_before
    pad[pl:pl + T] = gl
    dw = t[p + "conv.depthwise.weight"].double().reshape(d, K)
    y = t[p + "conv.depthwise.bias"].double().expand(T, -1).clone()
    for j in range(K):
        y += dw[:, j] * pad[j:j + T]
    gw, gb = t[p + "conv.bn.weight"].double(), t[p + "conv.bn.bias"].double()
    if hp.get("conv_norm", "batch_norm") == "layer_norm":
        y = _ln(y, gw, gb)
    else:
        y = (y - t[p + "conv.bn.running_mean"].double()) / torch.sqrt(t[p + "conv.bn.running_var"].double() + 1e-5) * gw + gb
    x = ff(x + W(_silu(y), "conv.pointwise2"), "ff2")
    return n(x, "norm_out"), kv, gl


def _loaded(t):
    """The tensors as the encoder holds them: float16 matrices rounded to Q8_0."""
    return {k: _to_q8(v) if getattr(v, "dtype", None) == torch.float16 else v for k, v in t.items()}


def _exact_conformer(c, seed):
    g = _Gen(seed)
    t = _loaded(_conf_tensors(c, g))
    mel, valid = _mel(c, g)
    hp, out = _conf_hp(c), []
    for b in range(c["batch"]):
        x, L = _subsample(hp, t, mel[b], valid[b])
        x = x * math.sqrt(hp["d"])
        seen = torch.arange(x.shape[0], device=DEV) < L
        mask = seen[:, None] & seen[None, :]
        for i in range(hp["layers"]):
            x = _conf_block(hp, t, i, x, L, mask)[0]
        out.append(x)
    return torch.stack(out)


def _exact_stream(c, seed):
    g = _Gen(seed)
    t = _loaded(_conf_tensors(c, g))
    geo, chunks = _stream_chunks(c, g)
    hp, out = _conf_hp(c), []
    for b in range(c["batch"]):
        kv, conv, n = [None] * hp["layers"], [None] * hp["layers"], 0
        for j, ch in enumerate(chunks):
            x, L = _subsample(hp, t, ch[b], ch.shape[2])
            if j:
                x, L = x[geo["drop"]:], L - geo["drop"]
            x = x * math.sqrt(hp["d"])
            T = x.shape[0]
            slot0 = geo["left"] - n
            qc = (slot0 + n + torch.arange(T, device=DEV))[:, None] // geo["chunk"]
            key = torch.arange(n + T, device=DEV)[None, :]
            mask = (key >= (qc - geo["left_chunks"]) * geo["chunk"] - slot0) & (key < (qc + 1) * geo["chunk"] - slot0)
            for i in range(hp["layers"]):
                x, rows, gl = _conf_block(hp, t, i, x, L, mask, kv[i], conv[i])
                kv[i] = rows[-geo["left"]:]
                prev = conv[i] if conv[i] is not None else torch.zeros(hp["conv_left"], hp["d"], dtype=torch.float64,
                                                                       device=DEV)
                conv[i] = torch.cat([prev, gl])[-hp["conv_left"]:]
            n = kv[0].shape[0]
        out.append(x)
    return dict(out=torch.stack(out))


def _exact_rnnt(c, seed):
    g = _Gen(seed)
    t, hp = _rnnt_tensors(c, g), _rnnt_hp(c)
    enc = g.normal(c["frames"], hp["d"])
    V, Ln, blank, durs = hp["pred_vocab"], hp["pred_layers"], hp["pred_vocab"] - 1, hp["durations"]
    ep = (_lin if c["frames"] > 1 else _flin)(enc.double(), t["joint.enc.weight"], t["joint.enc.bias"])
    W = {k: _f64(v) for k, v in t.items()}
    H = hp["pred_hidden"]
    h = [torch.zeros(H, dtype=torch.float64, device=DEV)] * Ln
    cc, last, pred, new, step, syms, p, gap = list(h), -1, None, None, 0, 0, [], math.inf

    def top(z):
        nonlocal gap
        v, i = z.topk(2)
        gap = min(gap, float(v[0] - v[1]))
        return int(i[0])

    while step < c["frames"]:
        if pred is None:
            x = W["pred.embed.weight"][last] if 0 <= last != blank else torch.zeros(H, dtype=torch.float64, device=DEV)
            nh, nc = [], []
            for i in range(Ln):
                q = f"pred.lstm.{i}."
                a, f, z, o = (W[q + "Wx"] @ x + W[q + "bias"] + W[q + "Wh"] @ h[i]).chunk(4)
                nc.append(torch.sigmoid(f) * cc[i] + torch.sigmoid(a) * torch.tanh(z))
                nh.append(torch.sigmoid(o) * torch.tanh(nc[-1]))
                x = nh[-1]
            new, pred = (nh, nc), W["joint.pred.weight"] @ x + W["joint.pred.bias"]
        z = W["joint.out.weight"] @ torch.relu(ep[step] + pred) + W["joint.out.bias"]
        tok, dur = top(z[:V]), durs[top(z[V:])] if durs else 1
        if tok != blank:
            p.append(float(torch.softmax(z[:V], 0)[tok]))
            (h, cc), last, pred = new, tok, None
        if durs:
            syms += 1
            step += dur
            if dur:
                syms = 0
            elif syms >= hp["max_symbols"]:
                step, syms = step + 1, 0
        elif tok == blank:
            step, syms = step + 1, 0
        else:
            syms += 1
            if syms >= 10:
                step, syms = step + 1, 0
    if gap < 2e-2:  # a near tie: another path would be as right
        return None
    return dict(p=_column(p, 10 * c["frames"], np.float64), h=torch.stack(h), c=torch.stack(cc))


def exact(case, seed):
    c = case
    if c["kind"] == "linear":
        g = _Gen(seed)
        w, x = g.q8(c["n"], c["k"]), g.normal(c["m"], c["k"])
        b = g.normal(c["n"], scale=0.1) if c["bias"] else None
        return _lin(x, w, b)
    return {"whisper": _exact_whisper, "pocket": _exact_pocket, "mimi": _exact_mimi, "conformer": _exact_conformer,
            "stream": _exact_stream, "rnnt": _exact_rnnt}[c["kind"]](c, seed)
