"""Performance cases of the serving hot path: the calls a Qwen3-TTS engine makes of this package.

Each case is one captured call (or one eager call where the engine makes it eagerly) with the
shapes of the serving configurations in ``bench.py``: the talker decode step over a paged KV pool,
the talker prefill step, one layer of mixed prefill + decode attention, the code predictor's whole
frame and the incremental codec step.  ``exact`` restates each in float64 torch.
"""

from __future__ import annotations

import math
from dataclasses import dataclass, field
from types import SimpleNamespace

import numpy as np
import torch
import torch.nn.functional as F

PAGE = 16
EPS = 1e-6
THETA = 1_000_000.0
# talker: hidden 2048, 16 query / 8 kv heads of 128, SwiGLU 6144, codec vocabulary 3072
HID, HQ, HKV, HD, FFN, VOCAB, TEXT = 2048, 16, 8, 128, 6144, 3072, 4096
# code predictor: 5 layers, hidden 1024, 16 / 8 heads of 64, SwiGLU 3072, 15 heads of 2048 codes
C_LAYERS, C_HID, C_HQ, C_HKV, C_HD, C_FFN, C_VOCAB, GROUPS = 5, 1024, 16, 8, 64, 3072, 2048, 15


def listed():
    return [
        # one listener's stream: the smallest decode bucket, where launches and latency count
        {"name": "decode-1", "kind": "decode", "rows": 1, "low": 64, "high": 512, "layers": 4, "whole": False,
         "batch": 1},
        # a lightly loaded server: 8 rows of short histories
        {"name": "decode-8", "kind": "decode", "rows": 8, "low": 16, "high": 512, "layers": 4, "whole": False,
         "batch": 2},
        # between the two: half the largest bucket
        {"name": "decode-32", "kind": "decode", "rows": 32, "low": 64, "high": 1024, "layers": 4, "whole": False,
         "batch": 3},
        # the headline step: 64 rows, 28 layers, planned, replayed and its pages returned
        {"name": "decode-64", "kind": "decode", "rows": 64, "low": 64, "high": 2048, "layers": 28, "whole": True,
         "batch": 4},
        # a new request's prompt alone, the time to its first audio (a 64-token bucket, ragged)
        {"name": "prefill-1", "kind": "prefill", "rows": 1, "tokens": 64, "fill": 45, "prior": 0, "layers": 4,
         "batch": 5},
        # a few prompts admitted together in the 192-token bucket
        {"name": "prefill-4", "kind": "prefill", "rows": 4, "tokens": 192, "fill": 183, "prior": 0, "layers": 4,
         "batch": 6},
        # the largest prefill bucket, chunks of long prompts over what they have in the cache
        {"name": "prefill-8", "kind": "prefill", "rows": 8, "tokens": 640, "fill": 631, "prior": 512, "layers": 4,
         "batch": 7},
        # one layer's attention of a batch that mixes prompt chunks and decode rows
        {"name": "mixed", "kind": "mixed", "chunks": 16, "rows": 112, "chunk": 256, "prior": 512, "high": 2048,
         "batch": 8},
        # the code predictor's frame for one stream and for a full batch
        {"name": "frame-1", "kind": "frame", "rows": 1, "top_k": 50},
        {"name": "frame-128", "kind": "frame", "rows": 128, "top_k": 50},
        # the codec step of one stream's short chunk (the reference's captured call) ...
        {"name": "codec-1", "kind": "codec", "streams": 1, "low": 4, "high": 4, "ragged": False, "batch": 11},
        # ... and of 32 streams with ragged chunks (the decoder's own state slots)
        {"name": "codec-32", "kind": "codec", "streams": 32, "low": 12, "high": 48, "ragged": True, "batch": 12},
    ]


def _log(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49))))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "mixed", "frame", "frame", "codec", "codec"))
    if kind == "decode":
        high = _log(rng, 32, 2048)
        return {"kind": kind, "rows": _log(rng, 1, 64), "low": max(1, high // rng.choice((2, 8, 32))), "high": high,
                "layers": 4, "whole": False, "batch": rng.randrange(1000)}
    if kind == "prefill":
        rows = rng.randint(1, 8)
        tokens = max(_log(rng, 10, 640), rows)
        return {"kind": kind, "rows": rows, "tokens": tokens, "fill": rng.randint(max(rows, tokens * 3 // 4), tokens),
                "prior": rng.choice((0, 0, _log(rng, 16, 512))), "layers": 4, "batch": rng.randrange(1000)}
    if kind == "mixed":
        return {"kind": kind, "chunks": rng.randint(1, 16), "rows": _log(rng, 8, 112), "chunk": _log(rng, 32, 256),
                "prior": _log(rng, 16, 512), "high": _log(rng, 128, 2048), "batch": rng.randrange(1000)}
    if kind == "frame":
        return {"kind": kind, "rows": _log(rng, 1, 128), "top_k": rng.randint(5, 50)}
    low = _log(rng, 1, 24)
    streams = _log(rng, 1, 32)
    ragged = rng.random() < 0.6
    return {"kind": kind, "streams": streams, "low": low, "high": min(48, low * rng.choice((1, 2))) if ragged else low,
            "ragged": ragged, "batch": rng.randrange(1000)}


# -- the package -------------------------------------------------------------------------------------


def _package(*names):
    from __graft_entry__ import load_package

    load_package()
    import importlib

    return [importlib.import_module(f"nari_qwen3_tts_amd.{n}") for n in names]


def _generator(seed, salt, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed((int(seed) * 1_000_003 + salt) % (1 << 62))
    return g


def _split(rng, total, parts):
    """``total`` tokens over ``parts`` rows, each at least one, uneven."""

    cuts = np.sort(rng.choice(np.arange(1, total), size=parts - 1, replace=False)) if parts > 1 else np.empty(0, int)
    return np.diff(np.concatenate(([0], cuts, [total]))).astype(int)


# -- inputs of the talker cases ------------------------------------------------------------------------


def _talker_weights(seed, layers):
    """N(0, 0.02) projections, those that write to the residual stream scaled by the model's depth of 28
    layers as such models are initialised, norm weights near 1, N(0, 1) embeddings; bf16 on the GPU."""

    g = _generator(seed, 1)

    def randn(*shape, std=0.02, mean=0.0):
        return torch.empty(*shape, device="cuda").normal_(mean, std, generator=g).to(torch.bfloat16)

    out = 0.02 / math.sqrt(2 * 28)
    return SimpleNamespace(
        layers=[SimpleNamespace(input_norm=randn(HID, std=0.1, mean=1.0), qkv=randn((HQ + 2 * HKV) * HD, HID),
                                q_norm=randn(HD, std=0.1, mean=1.0), k_norm=randn(HD, std=0.1, mean=1.0),
                                o=randn(HID, HQ * HD, std=out), post_norm=randn(HID, std=0.1, mean=1.0),
                                gate_up=randn(2 * FFN, HID), down=randn(HID, FFN, std=out)) for _ in range(layers)],
        norm=randn(HID, std=0.1, mean=1.0), head=randn(VOCAB, HID), text=randn(TEXT, HID, std=1.0),
        codec=randn(VOCAB, HID, std=1.0))


def _norm_module(w):
    return SimpleNamespace(weight=w, variance_epsilon=EPS)


def _linear_module(w, b=None):
    return SimpleNamespace(weight=w, bias=b)


def _layer_module(L):
    return SimpleNamespace(
        input_layernorm=_norm_module(L.input_norm), post_attention_layernorm=_norm_module(L.post_norm),
        self_attn=SimpleNamespace(qkv_proj=_linear_module(L.qkv), o_proj=_linear_module(L.o),
                                  q_norm=_norm_module(L.q_norm), k_norm=_norm_module(L.k_norm), rope_theta=THETA),
        mlp=SimpleNamespace(gate_up_proj=_linear_module(L.gate_up), down_proj=_linear_module(L.down)))


def _config(layers):
    predictor = SimpleNamespace(num_hidden_layers=C_LAYERS, hidden_size=C_HID, num_attention_heads=C_HQ,
                                num_key_value_heads=C_HKV, head_dim=C_HD, intermediate_size=C_FFN, vocab_size=C_VOCAB,
                                rms_norm_eps=EPS, rope_theta=THETA)
    return SimpleNamespace(talker=SimpleNamespace(
        num_hidden_layers=layers, hidden_size=HID, num_attention_heads=HQ, num_key_value_heads=HKV, head_dim=HD,
        intermediate_size=FFN, vocab_size=VOCAB, text_vocab_size=TEXT, codec_eos_token_id=2150, rms_norm_eps=EPS,
        rope_theta=THETA, num_code_groups=GROUPS + 1, code_predictor=predictor))


def _load_talker(w):
    (talker,) = _package("talker")
    model = SimpleNamespace(
        model=SimpleNamespace(layers=[_layer_module(L) for L in w.layers], norm=_norm_module(w.norm),
                              codec_embedding=_linear_module(w.codec)),
        codec_head=_linear_module(w.head), get_projected_text_embedding_cache=lambda: w.text)
    return talker.TalkerWeights.from_reference_model(model, _config(len(w.layers)))


def _pages(priors, advances, seed, scratch):
    """The pool: the first pages are the executor's scratch, the next ones are free (a step's new pages
    come from there, lowest first, in row order), the rows' own pages are scattered over the rest."""

    have = -(-priors // PAGE)
    new = -(-(priors + advances) // PAGE) - have
    spare = scratch + int(new.sum()) + 64
    owned = np.random.default_rng(seed).permutation(int(have.sum())) + spare
    old = np.split(owned, np.cumsum(have)[:-1])
    fresh = np.split(scratch + np.arange(int(new.sum())), np.cumsum(new)[:-1])
    return SimpleNamespace(total=spare + int(have.sum()), scratch=scratch, old=old, fresh=fresh, new=int(new.sum()))


def _fill(storage, seed):
    g = _generator(seed, 2)
    for layer in range(storage.shape[0]):
        storage[layer].normal_(generator=g)


def _kv(layers, pages, priors, seed):
    (talker_kv,) = _package("talker_kv")
    kv = talker_kv.PagedTalkerKV(num_layers=layers, num_kv_heads=HKV, num_qo_heads=HQ, head_dim=HD,
                                 total_pages=pages.total, page_size=PAGE, scratch_page_count=pages.scratch,
                                 workspace_bytes=0, device=torch.device("cuda:0"), dtype=torch.bfloat16)
    _fill(kv.storage, seed)
    names = tuple(f"r{i}" for i in range(len(priors)))
    for name, own, length in zip(names, pages.old, priors):
        kv.add_request(name)
        if length:
            kv.adopt_request(name, own.tolist(), int(length))
    return kv, names


def _talker_shape(case, seed):
    """Rows' lengths in the cache before the call, and their new tokens: the case's own (outputs keep
    their shapes); which pages hold them is the seed's."""

    rng = np.random.default_rng(case["batch"])
    if case["kind"] == "decode":
        priors = rng.integers(case["low"], case["high"] + 1, size=case["rows"])
        advances = np.ones(case["rows"], dtype=int)
        tokens = scratch = case["rows"]
    elif case["kind"] == "prefill":
        priors = rng.integers(0, case["prior"] + 1, size=case["rows"])
        advances = _split(rng, case["fill"], case["rows"])
        tokens, scratch = case["tokens"], max(case["rows"], -(-case["tokens"] // PAGE))
    else:
        chunks = rng.integers(min(32, case["chunk"]), case["chunk"] + 1, size=case["chunks"])
        priors = np.concatenate([rng.integers(0, case["prior"] + 1, size=case["chunks"]),
                                 rng.integers(64, case["high"] + 1, size=case["rows"])])
        advances = np.concatenate([chunks, np.ones(case["rows"], dtype=int)])
        tokens = int(advances.sum())
        scratch = max(len(priors), -(-tokens // PAGE) + 8)
    return SimpleNamespace(priors=priors, advances=advances, tokens=tokens,
                           pages=_pages(priors, advances, seed, scratch))


def _decode_inputs(case, seed):
    g = _generator(seed, 3)
    rows = case["rows"]
    return SimpleNamespace(
        embed=torch.empty(rows, HID, device="cuda").normal_(generator=g).to(torch.bfloat16),
        text=torch.randint(0, TEXT, (rows,), device="cuda", generator=g),
        history=torch.randint(0, 2048, (rows, 64), device="cuda", generator=g))


def _prefill_inputs(case, seed):
    g = _generator(seed, 4)
    n = case["tokens"]
    return SimpleNamespace(text=torch.randint(0, TEXT, (n,), device="cuda", generator=g),
                           codec=torch.randint(0, VOCAB, (n,), device="cuda", generator=g),
                           mask=torch.rand(n, device="cuda", generator=g) < 0.5)


def _sampling(step, rows, seed):
    """The serving defaults: T 0.9, top-k 50, top-p 0.95."""

    step.temperature.fill_(0.9)
    step.top_k.fill_(50)
    step.top_p.fill_(0.95)
    step.penalty.fill_(1.05)
    step.seed.copy_(torch.arange(rows, device="cuda") * 7919 + seed % 65536)
    step.offsets.fill_(512)


class _Key:
    def __init__(self, rows, tokens=None):
        self.capture_batch_size = rows
        if tokens is not None:
            self.token_capacity = tokens


def _prepare_decode(case, seed):
    graphs, talker = _package("graphs", "talker")
    s, x = _talker_shape(case, seed), _decode_inputs(case, seed)
    rows = case["rows"]
    kv, names = _kv(case["layers"], s.pages, s.priors, seed)
    key = _Key(rows)
    context = kv.create_decode(key, slot=0)
    step = talker.TalkerDecodeStep(_load_talker(_talker_weights(seed, case["layers"])), context, rows,
                                   use_counter_rng=True)
    _sampling(step, rows, seed)
    step.step_embed.copy_(x.embed)
    step.text_ids.copy_(x.text)
    held = kv.prepare_decode(context, key, names)
    call = graphs.HipGraphCaptureDriver(device=kv.device, warmups=1).capture(step.forward)
    if case["whole"]:
        kv.abort(held)
    step.seen.zero_().scatter_(1, x.history, True)
    fresh = kv.storage[:, s.pages.scratch:s.pages.scratch + s.pages.new]
    out = {"logits": step.logits, "hidden": step.hidden, "kv": fresh}
    # the graph reads the step's buffers and weights: the program keeps the step as long as the graph
    return SimpleNamespace(run=_run_whole_decode if case["whole"] else _run_replay, call=call, out=out, step=step,
                           kv=kv, context=context, key=key, names=names, held=held)


def _run_replay(state):
    state.call.replay()
    return state.out


def _run_whole_decode(state):
    # one decision: the GPU planner, the captured step, then the pages go back (the next pass is the
    # same decision again)
    taken = state.kv.prepare_decode(state.context, state.key, state.names)
    state.call.replay()
    state.kv.abort(taken)
    return state.out


def _prepare_prefill(case, seed):
    graphs, talker = _package("graphs", "talker")
    s, x = _talker_shape(case, seed), _prefill_inputs(case, seed)
    rows, tokens = case["rows"], case["tokens"]
    kv, names = _kv(case["layers"], s.pages, s.priors, seed)
    key = _Key(rows, tokens)
    context = kv.create_prefill(key, slot=0)
    step = talker.TalkerPrefillStep(_load_talker(_talker_weights(seed, case["layers"])), context, rows, tokens)
    _sampling(step, rows, seed)
    step.text_ids.copy_(x.text)
    step.codec_ids.copy_(x.codec)
    step.codec_mask.copy_(x.mask)
    held = kv.prepare_prefill(context, key, names, tuple(int(n) for n in s.advances))
    call = graphs.HipGraphCaptureDriver(device=kv.device, warmups=1).capture(step.forward)
    step.seen.zero_()
    fresh = kv.storage[:, s.pages.scratch:s.pages.scratch + s.pages.new]
    out = {"logits": step.logits, "last": step.last_hidden, "hidden": step.hidden[:case["fill"]], "kv": fresh}
    return SimpleNamespace(run=_run_replay, call=call, out=out, step=step, kv=kv, held=held, context=context)


def _queries(tokens, seed):
    return torch.empty(tokens, HQ, HD, device="cuda").normal_(generator=_generator(seed, 5)).to(torch.bfloat16)


def _prepare_mixed(case, seed):
    s = _talker_shape(case, seed)
    kv, names = _kv(1, s.pages, s.priors, seed)
    key = _Key(len(s.priors), s.tokens)
    context = kv.create_prefill(key, slot=0, decode_rows=True)
    held = kv.prepare_prefill(context, key, names, tuple(int(n) for n in s.advances))
    q = _queries(s.tokens, seed)
    return SimpleNamespace(run=lambda state: context.run_attention(q, 0), kv=kv, held=held)


# -- the code predictor --------------------------------------------------------------------------------


def _frame_weights(seed):
    """Random layers under heads that, as trained ones do, know the next code well: each group's head
    scores the code whose embedding (permuted) it was given far above the rest, so that a frame's codes
    do not hang on the last bits of a logit."""

    g = _generator(seed, 6)

    def randn(*shape, std=0.02, mean=0.0):
        return torch.empty(*shape, device="cuda").normal_(mean, std, generator=g).to(torch.bfloat16)

    w = SimpleNamespace(
        layers=[SimpleNamespace(input_norm=randn(C_HID, std=0.1, mean=1.0), qkv=randn((C_HQ + 2 * C_HKV) * C_HD, C_HID),
                                q_norm=randn(C_HD, std=0.1, mean=1.0), k_norm=randn(C_HD, std=0.1, mean=1.0),
                                o=randn(C_HID, C_HQ * C_HD), post_norm=randn(C_HID, std=0.1, mean=1.0),
                                gate_up=randn(2 * C_FFN, C_HID), down=randn(C_HID, C_FFN)) for _ in range(C_LAYERS)],
        norm=randn(C_HID, std=0.1, mean=1.0), proj_w=randn(C_HID, HID), proj_b=randn(C_HID),
        layer0=randn(VOCAB, HID, std=1.0), codec=randn(GROUPS, C_VOCAB, HID, std=1.0))
    heads = []
    for group in range(GROUPS):
        table = (w.layer0[:C_VOCAB] if group == 0 else w.codec[group - 1]).float()
        given = table @ w.proj_w.float().t() + w.proj_b.float()
        order = torch.randperm(C_VOCAB, device="cuda", generator=g)
        heads.append((1.3 * given / given.square().mean(1, keepdim=True).sqrt())[order].to(torch.bfloat16))
    w.heads = torch.stack(heads)
    return w


def _frame_inputs(case, seed):
    g = _generator(seed, 7)
    rows = case["rows"]
    return SimpleNamespace(token=torch.randint(0, C_VOCAB, (rows,), device="cuda", generator=g),
                           hidden=torch.empty(rows, HID, device="cuda").normal_(generator=g).to(torch.bfloat16))


def _prepare_frame(case, seed):
    graphs, code_predictor = _package("graphs", "code_predictor")
    w, x, rows = _frame_weights(seed), _frame_inputs(case, seed), case["rows"]
    model = SimpleNamespace(
        model=SimpleNamespace(layers=[_layer_module(L) for L in w.layers], norm=_norm_module(w.norm),
                              codec_embedding=[_linear_module(e) for e in w.codec]),
        lm_head=[_linear_module(h) for h in w.heads], small_to_mtp_projection=_linear_module(w.proj_w, w.proj_b))
    weights = code_predictor.CodePredictorWeights.from_reference_model(model, _linear_module(w.layer0), _config(0))
    frame = code_predictor.CodePredictorFrame(weights, rows, use_counter_rng=True)
    frame.layer0_token.copy_(x.token)
    frame.past_hidden.copy_(x.hidden)
    frame.temperature.fill_(0.9)
    frame.top_k.fill_(case["top_k"])
    frame.seed.copy_(torch.arange(rows, device="cuda") * 7919 + seed % 65536)
    frame.offsets.copy_(torch.arange(rows * GROUPS, device="cuda").view(rows, GROUPS))
    call = graphs.HipGraphCaptureDriver(device=torch.device("cuda:0"), warmups=1).capture(frame.forward)
    out = {"frames": frame.frames, "codec_sum": frame.codec_sum, "logits": frame.logits}
    return SimpleNamespace(run=_run_replay, call=call, out=out, frame=frame)


# -- the codec -----------------------------------------------------------------------------------------

WARM = 25  # frames of history every stream comes with: one full window of retained context


@dataclass
class CodecState:
    """The engine's record of one stream (the decoder's reference call reads and replaces its tensors)."""

    frame_position: int = 0
    transformer_context_length: int = 0
    transformer_keys: dict = field(default_factory=dict)
    transformer_values: dict = field(default_factory=dict)
    conv_histories: dict = field(default_factory=dict)
    transconv_overlaps: dict = field(default_factory=dict)


def _codec_inputs(case, seed):
    frames = np.random.default_rng(case["batch"]).integers(case["low"], case["high"] + 1, size=case["streams"])
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(rng.integers(0, 2048, size=(16, WARM + int(f)))) for f in frames]


def _prepare_codec(case, seed):
    graphs, codec = _package("graphs", "codec")
    device = torch.device("cuda:0")
    weights = codec.CodecWeights(codec.CodecConfig(), device, seed=seed % (1 << 31))
    decoder = codec.IncrementalCodecDecoder(weights, max_streams=case["streams"])
    codes = _codec_inputs(case, seed)
    warm, fresh = [c[:, :WARM] for c in codes], [c[:, WARM:].contiguous() for c in codes]
    if case["ragged"]:
        states = [decoder.new_state() for _ in codes]
        decoder.decode_ragged(warm, states)
        return SimpleNamespace(run=lambda state: {"wav": decoder.decode_ragged(fresh, states)[0]})
    rows, frames = len(codes), fresh[0].shape[1]
    states = [CodecState() for _ in codes]
    decoder(torch.stack(warm).to(device), states)
    held = torch.stack(fresh).to(device)
    position = torch.arange(frames, device=device).unsqueeze(0).expand(rows, -1) + WARM
    context = torch.full((rows,), WARM, dtype=torch.long, device=device)
    new = []

    def operation():
        new[:] = [CodecState(s.frame_position, s.transformer_context_length, dict(s.transformer_keys),
                             dict(s.transformer_values), dict(s.conv_histories), dict(s.transconv_overlaps))
                  for s in states]
        return decoder(held, new, position_ids=position, context_lengths=context)

    call = graphs.HipGraphCaptureDriver(device=device, warmups=1).capture(operation)
    out = {"wav": call.output, "keys": [s.transformer_keys[7] for s in new],
           "histories": [s.conv_histories["decoder.0"] for s in new]}
    return SimpleNamespace(run=_run_replay, call=call, out=out, operation=operation)


def prepare(case, seed):
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "mixed": _prepare_mixed, "frame": _prepare_frame,
            "codec": _prepare_codec}[case["kind"]](case, seed)


def run(state):
    return state.run(state)


# -- what a call cannot do without -----------------------------------------------------------------------

_ATTENTION = (HQ + 2 * HKV) * HD * HID + HID * HQ * HD  # QKV and o weights of a talker layer
_C_LAYER = (C_HQ + 2 * C_HKV) * C_HD * C_HID + C_HID * C_HQ * C_HD + 3 * C_FFN * C_HID


def _codec_work(frames):
    d, f, u, parameters = 512, 0.0, 1, 0
    for n in (d * d * 3, 2 * d * d, 8 * (4 * d * d + 2 * d * 1536)):
        f += 2.0 * frames * n
        parameters += n
    f += 2.0 * frames * 8 * 8 * 26 * 64 * 2
    for s in (2, 2):
        f += 2.0 * frames * u * d * d * 2 * s
        u *= s
        f += 2.0 * frames * u * (d * 7 + 2 * d * 1024)
        parameters += d * d * 2 * s + 2 * d * 1024
    channels = (128, 64, 32, 16, 8)
    f += 2.0 * frames * u * d * 128 * 7
    parameters += d * 128 * 7
    for i, s in enumerate((5, 5, 4, 5)):
        f += 2.0 * frames * u * channels[i] * channels[i + 1] * 2 * s
        u *= s
        f += 2.0 * frames * u * 3 * channels[i + 1] ** 2 * 8
        parameters += channels[i] * channels[i + 1] * 2 * s + 24 * channels[i + 1] ** 2
    f += 2.0 * frames * u * 8 * 7
    return f, parameters, u


def work(case):
    kind = case["kind"]
    if kind == "frame":
        rows = case["rows"]
        parameters = C_LAYERS * _C_LAYER
        flops = 2.0 * rows * ((GROUPS + 1) * parameters + GROUPS * C_VOCAB * C_HID + C_HID * HID)
        out = rows * (GROUPS * C_VOCAB * 2 + HID * 4 + (GROUPS + 1) * 8)
        return {"bytes": 2.0 * (parameters + GROUPS * C_VOCAB * C_HID + C_HID * HID) + out, "flops": flops}
    if kind == "codec":
        frames = case["streams"] * (case["low"] + case["high"]) / 2
        flops, parameters, up = _codec_work(frames)
        state = case["streams"] * (8 * 2 * WARM * 512 + 7000) * 4
        return {"bytes": 4.0 * (parameters + frames * (16 * 512 + up)) + 2 * state, "flops": flops}
    if kind == "decode":
        rows, layers, tokens = case["rows"], case["layers"], case["rows"]
        read = rows * ((case["low"] + case["high"]) / 2 + 1)
        pairs = read
    elif kind == "prefill":
        rows, layers, tokens = case["rows"], case["layers"], case["fill"]
        prior = case["prior"] / 2
        read = rows * prior + tokens
        pairs = tokens * (prior + tokens / rows / 2)
    else:
        chunk, prior = (min(32, case["chunk"]) + case["chunk"]) / 2, case["prior"] / 2
        tokens = case["chunks"] * chunk + case["rows"]
        decode = case["rows"] * ((64 + case["high"]) / 2 + 1)
        read = case["chunks"] * (prior + chunk) + decode
        pairs = case["chunks"] * chunk * (prior + chunk / 2) + decode
        return {"bytes": read * HKV * HD * 4 + 2 * tokens * HQ * HD * 2, "flops": 4.0 * HQ * HD * pairs}
    attention = {"bytes": layers * read * HKV * HD * 4, "flops": layers * 4.0 * HQ * HD * pairs}
    weights = layers * (2 * (_ATTENTION + HID * FFN) + 2 * FFN * HID) + 2 * VOCAB * HID
    flops = layers * 2.0 * tokens * (_ATTENTION + 3 * HID * FFN) + 2.0 * rows * VOCAB * HID
    return {"bytes": attention["bytes"] + weights + tokens * HID * 4 + rows * VOCAB * 2,
            "flops": attention["flops"] + flops}


def tolerance(case):
    # against float64 the present kernels are 0.00024 off for the codec (products of split bf16 halves, fp32
    # sums), 0.002 for attention alone (bf16 outputs), 0.006 for a frame, 0.007 for a stack of four FP8 layers
    # and 0.02 for 28 (an FP8 code that falls to the other side moves a value by a tenth); sums in another
    # order end as far from these as either is from float64
    if case["kind"] == "codec":
        return {"rel": 1e-3, "max": 0.05}
    if case["kind"] == "mixed":
        return {"rel": 8e-3, "max": 0.1}
    if case["kind"] == "frame":
        return {"rel": 0.02, "max": 0.3}
    return {"rel": 0.03 if case["layers"] > 4 else 0.02, "max": 0.3}


# -- the same in 64 bits -----------------------------------------------------------------------------------


def _rms(x, w, eps=EPS):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope(x, positions, theta):
    """Rotate-half RoPE of x [T, H, D]."""

    d = x.shape[-1]
    inv = theta ** (-torch.arange(0, d, 2, device=x.device, dtype=torch.float64) / d)
    angle = positions.double()[:, None] * inv
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)


def _attend(q, k, v, mask=None):
    """q [T, Hq, D] over k, v [S, Hkv, D], query heads grouped; mask [T, S] True where seen."""

    group = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(group, 1).transpose(0, 1), v.repeat_interleave(group, 1).transpose(0, 1)
    scores = q.transpose(0, 1) @ k.transpose(1, 2).contiguous() / math.sqrt(q.shape[2])
    if mask is not None:
        scores = scores.masked_fill(~mask, -math.inf)
    return (scores.softmax(-1) @ v).transpose(0, 1)


def _fp8(x):
    return x.float().to(torch.float8_e4m3fn).double()


def _fp8_blocks(w):
    """The reference build's gate/up weights: 128 x 128 FP8 blocks under power-of-two scales."""

    n, k = w.shape
    blocks = w.float().view(n // 128, 128, k // 128, 128)
    top = blocks.abs().amax((1, 3), keepdim=True).clamp_min(1e-4)
    scale = torch.exp2(torch.ceil(torch.log2(top / 448.0)))
    return (_fp8(blocks / scale) * scale.double()).view(n, k)


def _fp8_rows(x):
    groups = x.view(x.shape[0], -1, 128)
    top = groups.abs().amax(-1, keepdim=True)
    scale = torch.where(top > 0, top / 448.0, torch.ones_like(top))
    return (_fp8(groups / scale) * scale).view_as(x)


def _swiglu(x, gate_up):
    gate, up = (x @ gate_up.t()).chunk(2, -1)
    return F.silu(gate) * up


def _mask(prior, new, device):
    return torch.arange(prior + new, device=device) <= prior + torch.arange(new, device=device)[:, None]


def _past(cache, pages, prior):
    """The first ``prior`` cached keys and values of a row."""

    got = cache[torch.as_tensor(pages, device=cache.device)].double()
    return (got[:, i].reshape(-1, HKV, HD)[:prior] for i in (0, 1))


def _exact_talker(case, seed):
    s, w = _talker_shape(case, seed), _talker_weights(seed, case["layers"])
    storage = torch.empty(case["layers"], s.pages.total, 2, PAGE, HKV, HD, dtype=torch.bfloat16, device="cuda")
    _fill(storage, seed)
    total = int(s.advances.sum())
    if case["kind"] == "decode":
        x = _decode_inputs(case, seed)
        h = x.embed.double() + w.text[x.text].double()
    else:
        x = _prefill_inputs(case, seed)
        h = (w.text[x.text].double() + w.codec[x.codec].double() * x.mask[:, None])[:total]
    starts = np.concatenate(([0], np.cumsum(s.advances)))
    positions = torch.cat([torch.arange(p, p + n) for p, n in zip(s.priors, s.advances)]).cuda()
    written = []
    for layer, L in enumerate(w.layers):
        qkv = (_rms(h, L.input_norm) @ L.qkv.double().t()).view(total, HQ + 2 * HKV, HD)
        q = _rope(_rms(qkv[:, :HQ], L.q_norm), positions, THETA)
        k = _rope(_rms(qkv[:, HQ:HQ + HKV], L.k_norm), positions, THETA)
        v = qkv[:, HQ + HKV:]
        attended = torch.empty_like(q)
        fresh = storage[layer, s.pages.scratch:s.pages.scratch + s.pages.new].double()
        for row, (prior, new) in enumerate(zip(s.priors, s.advances)):
            a, b, prior, new = int(starts[row]), int(starts[row + 1]), int(prior), int(new)
            pages = np.concatenate([s.pages.old[row], s.pages.fresh[row]]).astype(np.int64)
            past_k, past_v = _past(storage[layer], pages, prior)
            attended[a:b] = _attend(q[a:b], torch.cat((past_k, k[a:b])), torch.cat((past_v, v[a:b])),
                                    _mask(prior, new, "cuda"))
            slots = prior + np.arange(new)
            page = pages[slots // PAGE] - s.pages.scratch
            keep = (page >= 0) & (page < s.pages.new)
            at = torch.from_numpy(page[keep]).cuda(), torch.from_numpy(slots[keep] % PAGE).cuda()
            fresh[at[0], 0, at[1]] = k[a:b][torch.from_numpy(keep).cuda()]
            fresh[at[0], 1, at[1]] = v[a:b][torch.from_numpy(keep).cuda()]
        written.append(fresh)
        h = h + attended.reshape(total, HQ * HD) @ L.o.double().t()
        h = h + _swiglu(_fp8_rows(_rms(h, L.post_norm)), _fp8_blocks(L.gate_up)) @ L.down.double().t()
    hidden = _rms(h, w.norm)
    last = hidden if case["kind"] == "decode" else hidden[torch.from_numpy(starts[1:] - 1).cuda()]
    out = {"logits": last @ w.head.double().t(), "hidden": hidden, "kv": torch.stack(written)}
    return out if case["kind"] == "decode" else {**out, "last": last}


def _exact_mixed(case, seed):
    s, q = _talker_shape(case, seed), _queries(_talker_shape(case, seed).tokens, seed).double()
    storage = torch.empty(1, s.pages.total, 2, PAGE, HKV, HD, dtype=torch.bfloat16, device="cuda")
    _fill(storage, seed)
    out, at = torch.empty_like(q), 0
    for row, (prior, new) in enumerate(zip(s.priors, s.advances)):
        prior, new = int(prior), int(new)
        k, v = _past(storage[0], np.concatenate([s.pages.old[row], s.pages.fresh[row]]).astype(np.int64), prior + new)
        out[at:at + new] = _attend(q[at:at + new], k, v, _mask(prior, new, "cuda"))
        at += new
    return out


def _exact_frame(case, seed):
    w, x, rows = _frame_weights(seed), _frame_inputs(case, seed), case["rows"]
    cache = [([], []) for _ in w.layers]

    def layers(h, position):
        at = torch.full((rows,), position, device="cuda")
        for L, (keys, values) in zip(w.layers, cache):
            qkv = (_rms(h, L.input_norm) @ L.qkv.double().t()).view(rows, C_HQ + 2 * C_HKV, C_HD)
            q = _rope(_rms(qkv[:, :C_HQ], L.q_norm), at, THETA)
            keys.append(_rope(_rms(qkv[:, C_HQ:C_HQ + C_HKV], L.k_norm), at, THETA))
            values.append(qkv[:, C_HQ + C_HKV:])
            k, v = (torch.stack(t, 1).repeat_interleave(C_HQ // C_HKV, 2) for t in (keys, values))
            p = ((q[:, None] * k).sum(-1) / math.sqrt(C_HD)).softmax(1)
            h = h + (p[..., None] * v).sum(1).reshape(rows, -1) @ L.o.double().t()
            h = h + _swiglu(_rms(h, L.post_norm), L.gate_up.double()) @ L.down.double().t()
        return _rms(h, w.norm)

    def project(e):
        return e.double() @ w.proj_w.double().t() + w.proj_b.double()

    layers(project(x.hidden), 0)
    token, total, h, logits, frames = x.token, w.layer0[x.token].double(), project(w.layer0[x.token]), [], [x.token]
    for group in range(GROUPS):
        logits.append(layers(h, group + 1) @ w.heads[group].double().t())
        token = logits[-1].argmax(-1)
        frames.append(token)
        total = total + w.codec[group][token].double()
        h = project(w.codec[group][token])
    return {"frames": torch.stack(frames, 1), "codec_sum": total, "logits": torch.stack(logits)}


def _exact_codec(case, seed):
    """The whole causal pass of each stream from its first frame; the fresh frames' samples are the last."""

    (codec,) = _package("codec")
    w = codec.CodecWeights(codec.CodecConfig(), torch.device("cuda:0"), seed=seed % (1 << 31))

    def conv(x, weight, bias, dilation=1):
        """Causal convolution of x [C, T], dense or depthwise, a product per tap."""

        weight, taps, t = weight.double(), weight.shape[2], x.shape[1]
        x = F.pad(x, ((taps - 1) * dilation, 0))
        y = bias.double()[:, None]
        for j in range(taps):
            part = x[:, j * dilation:j * dilation + t]
            y = y + (weight[:, 0, j, None] * part if weight.shape[1] == 1 < x.shape[0] else weight[:, :, j] @ part)
        return y

    def up(x, weight, bias, stride):
        """Causal transposed convolution of x [C, T] whose kernel spans two strides."""

        y = torch.einsum("ct,cok->otk", x, weight.double())
        y = y[..., :stride] + F.pad(y[..., stride:], (0, 0, 1, 0))[:, :-1]
        return y.reshape(y.shape[0], -1) + bias.double()[:, None]

    def snake(x, alpha, beta):
        a, b = alpha.double().exp()[:, None], beta.double().exp()[:, None]
        return x + (x * a).sin().square() / (b + 1e-9)

    def linear(x, weight, bias=None):
        return F.linear(x, weight.double(), None if bias is None else bias.double())

    wavs = []
    for codes in _codec_inputs(case, seed):
        t = codes.shape[1]
        x = sum(w.codebooks[i].double()[codes[i].cuda()] for i in range(16))
        h = linear(conv(x.t(), w.pre_conv_w, w.pre_conv_b).t(), w.in_w, w.in_b)
        at = torch.arange(t, device="cuda")
        seen = (at <= at[:, None]) & (at > at[:, None] - 26)
        for L in w.tf:
            q, k, v = linear(_rms(h, L.ln1), L.wqkv).view(t, 3, 8, 64).unbind(1)
            q, k = _rope(_rms(q, L.qn), at, 1e4), _rope(_rms(k, L.kn), at, 1e4)
            h = h + linear(_attend(q, k, v, seen).reshape(t, 512), L.wo) * L.ls1.double()
            h = h + linear(F.gelu(linear(_rms(h, L.ln2), L.w1)), L.w2) * L.ls2.double()
        x = linear(_rms(h, w.out_norm), w.out_w, w.out_b).t()
        for U in w.up:
            x = up(x, U.tc_w, U.tc_b, 2)
            y = conv(x, U.dw_w, U.dw_b).t()
            y = F.layer_norm(y, (512,), U.ln_w.double(), U.ln_b.double(), 1e-6)
            y = linear(F.gelu(linear(y, U.pw1_w, U.pw1_b)), U.pw2_w, U.pw2_b)
            x = x + (U.gamma.double() * y).t()
        x = conv(x, w.dec0_w, w.dec0_b)
        for stride, B in zip((5, 5, 4, 5), w.blocks):
            x = up(snake(x, B.alpha, B.beta), B.tc_w, B.tc_b, stride)
            for dilation, R in zip((1, 3, 9), B.res):
                y = conv(snake(x, R.a1, R.b1), R.c1_w, R.c1_b, dilation)
                x = x + conv(snake(y, R.a2, R.b2), R.c2_w, R.c2_b)
        x = conv(snake(x, w.final_alpha, w.final_beta), w.final_w, w.final_b)
        wavs.append(x[0, WARM * 2000:].clamp(-1, 1))
    if case["ragged"]:
        return {"wav": wavs}
    none = [None] * len(wavs)
    return {"wav": torch.stack(wavs)[:, None], "keys": none, "histories": none}


def exact(case, seed):
    return {"decode": _exact_talker, "prefill": _exact_talker, "mixed": _exact_mixed, "frame": _exact_frame,
            "codec": _exact_codec}[case["kind"]](case, seed)
