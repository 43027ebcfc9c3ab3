"""The work a program gives this library, as cases that can be timed and compared.

Everything goes through the entry points such a program calls (`guffin_amd.model`, `guffin_amd.hip`) on the two models
the library is configured for: the 12B-shaped K-quant target and the 270M-shaped Q8_0 drafter, with seeded random
weights and filled KV rings.  A case is a dict of plain values; its `kind` says which part of a conversation it is:

  prefill   a run of prompt tokens through one model: a long document, an ordinary question, a short chat turn on top of
            a conversation, the drafter's own pass over a prompt
  step      one speculative cycle (draft, verify two rows, accept, publish) at a given context
  session   consecutive cycles of a conversation, the host reading each cycle's tokens
  decode    plain decoding of one token by the target (no speculation): forward, head, argmax, publish
  draft     the drafter's side of a chain of proposals: ingest what was accepted, propose, drop the transaction
  tree      a verify pass over a small token tree as a transaction: submit, complete, commit a path, keep part of it
  sample    logits to a decision: candidates of two verify rows, the proposal law, accept or residual
  gemv      one quantised matrix times one or two rows (receipt and product), the smallest call
  repack    one weight matrix into the device layout, as the loader of a model file does for each
"""
import ctypes as C
import math
import random
from dataclasses import replace

import torch

from guffin_amd import hip, model, synth

TARGET, DRAFTER = model.GEMMA3_12B, model.GEMMA3_270M
SHAPES = {"12b": TARGET, "270m": DRAFTER}
CONTEXT = 8192            # tokens the models' global rings hold
OPTIONS = dict(temperature=1.0, top_k=64, top_p=0.95, min_p=0.0)


def listed():
    return [
        # the largest: a long document ahead of a conversation
        {"name": "prefill_document", "kind": "prefill", "model": "12b", "mixed": False, "rows": 2048, "position": 0},
        # a question with some context, on a file that keeps half of its blocks' v and down matrices in four bits
        {"name": "prefill_question", "kind": "prefill", "model": "12b", "mixed": True, "rows": 333, "position": 0},
        # a short turn of a running conversation, ragged, behind wrapped local rings
        {"name": "prefill_turn", "kind": "prefill", "model": "12b", "mixed": False, "rows": 37, "position": 1500},
        # the drafter ingests the same kind of prompt
        {"name": "prefill_drafter", "kind": "prefill", "model": "270m", "mixed": False, "rows": 1000, "position": 0},
        # one cycle at the longest context, the library's own benchmark workload
        {"name": "step_long_context", "kind": "step", "position": 8190, "draft_position": 4096},
        # two cycles of a chat with the host in the loop, the second one also ingesting the accepted proposal
        {"name": "session_chat", "kind": "session", "position": 611, "cycles": 2},
        # decoding without a drafter
        {"name": "decode_plain", "kind": "decode", "mixed": True, "position": 1733},
        # what the drafter does between two verify passes of a chain of four
        {"name": "draft_chain", "kind": "draft", "prefix": 150, "append": 3, "horizon": 4},
        # a four-row tree: two continuations of the root, one of them two tokens deep
        {"name": "verify_tree", "kind": "tree", "position": 900, "parents": "-,0,0,1", "keep": 2},
        # sampling alone
        {"name": "sample_rows", "kind": "sample", "top_k": 64},
        # one matrix-vector product, the smallest call
        {"name": "gemv_gate", "kind": "gemv", "dtype": synth.Q4_K, "k": 3840, "n": 15360, "rows": 1},
        # loading: one of the large matrices
        {"name": "repack_down", "kind": "repack", "dtype": synth.Q6_K, "k": 15360, "n": 3840},
    ]


TREES = {"-,0": 2, "-,0,0": 2, "-,0,1": 3, "-,0,0,1": 3, "-,0,1,2": 4, "-,0,0,0": 2}   # parents of each row : longest path


def _matrices():
    """(dtype, K, N) of every kind of projection of the two models."""
    seen = []
    for sh in (TARGET, DRAFTER):
        for dt, (k, n) in zip(sh.dtypes, sh.proj_shapes()):
            if (dt, k, n) not in seen:
                seen.append((dt, k, n))
    return seen


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "prefill", "step", "session", "decode", "draft", "tree", "sample", "gemv", "repack"])
    if kind == "prefill":
        rows = _spread(rng, 2, 2048)
        start = rng.choice([0, 1]) * _spread(rng, 1, CONTEXT // 4)
        if rng.random() < 0.3:
            return {"kind": kind, "model": "270m", "mixed": False, "rows": rows, "position": start}
        # the longest run starts a conversation; what follows one is shorter
        return {"kind": kind, "model": "12b", "mixed": rng.random() < 0.5, "rows": min(rows, 2048 if start == 0 else 1024),
                "position": start}
    if kind == "step":
        at = _spread(rng, 16, CONTEXT - 2)
        return {"kind": kind, "position": at, "draft_position": min(at, rng.choice([512, 4096, CONTEXT - 2]))}
    if kind == "session":
        return {"kind": kind, "position": _spread(rng, 16, CONTEXT // 2), "cycles": rng.randint(1, 3)}
    if kind == "decode":
        return {"kind": kind, "mixed": rng.random() < 0.5, "position": _spread(rng, 16, CONTEXT - 1)}
    if kind == "draft":
        return {"kind": kind, "prefix": _spread(rng, 8, 250), "append": rng.randint(1, 6), "horizon": rng.randint(1, 8)}
    if kind == "tree":
        parents = rng.choice(sorted(TREES))
        return {"kind": kind, "position": _spread(rng, 16, CONTEXT - 8), "parents": parents, "keep": rng.randint(1, TREES[parents])}
    if kind == "sample":
        return {"kind": kind, "top_k": rng.randint(1, 64)}
    dtype, k, n = rng.choice(_matrices())
    if kind == "gemv":
        return {"kind": kind, "dtype": dtype, "k": k, "n": n, "rows": rng.randint(1, 2)}
    if rng.random() < 0.2:   # a head: the vocabulary's rows, or part of a larger one's
        dtype, k = rng.choice([(TARGET.embed_dtype, TARGET.hidden), (DRAFTER.embed_dtype, DRAFTER.hidden)])
        n = 64 * _spread(rng, 500, TARGET.vocab // 64)
    return {"kind": kind, "dtype": dtype, "k": k, "n": n}


# ---- models -----------------------------------------------------------------------------------------------

def _shape(case):
    sh = SHAPES[case.get("model", "12b")]
    if case.get("mixed"):
        # the usual four-bit mix: every other block keeps attn_v and ffn_down in four bits as well
        four = tuple(synth.Q4_K for _ in sh.dtypes)
        sh = replace(sh, layer_dtypes=tuple(sh.dtypes if l % 2 == 0 else four for l in range(sh.layers)))
    return sh


def _model(shape, seed, position):
    """A device model whose rings lie in two allocations (windowed and global layers), so that they can be looked at whole."""
    m = model.DeviceModel.random(shape, seed=seed, position=position)
    arenas = []
    for local in (True, False):
        layers = [l for l in range(shape.layers) if shape.is_local(l) == local]
        arena = torch.stack([torch.stack([m.ring_k[l], m.ring_v[l]]) for l in layers])
        for i, l in enumerate(layers):
            m.ring_k[l], m.ring_v[l] = arena[i, 0], arena[i, 1]
            m.layers[l].ring_k, m.layers[l].ring_v = m.ring_k[l].data_ptr(), m.ring_v[l].data_ptr()
        arenas.append(arena)
    m.ring_k_table.copy_(torch.tensor([t.data_ptr() for t in m.ring_k], dtype=torch.int64))
    m.ring_v_table.copy_(torch.tensor([t.data_ptr() for t in m.ring_v], dtype=torch.int64))
    return m, arenas


def _tokens(seed, count):
    rng = random.Random(seed)
    return [rng.randrange(2, TARGET.vocab) for _ in range(count)]


def _device_tokens(seed, count):
    return torch.tensor(_tokens(seed, count), dtype=torch.int32, device="cuda")


def _candidates(blob):
    """Candidate records as tensors: counts and status, token ids, logits."""
    words = blob.view(torch.int32).view(-1, hip.candidates_dtype.itemsize // 4)
    return {"count": words[:, :2], "tokens": words[:, 2::2], "logits": words.view(torch.float32)[:, 3::2]}


def _decision(blob):
    """A cycle's decision: accepted, token, next root, status; acceptance probability and residual mass; residual count, proposal."""
    return {"head": blob.view(torch.int32)[:4], "mass": blob[16:32].view(torch.float64), "tail": blob.view(torch.int32)[8:10]}


# ---- one pass ---------------------------------------------------------------------------------------------

def prepare(case, seed):
    hip.init(0)
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "prefill":
        s["model"], s["rings"] = _model(_shape(case), seed, case["position"])
        s["tokens"], s["position"] = _device_tokens(seed, case["rows"]), case["position"]
    elif kind == "step":
        s["target"], s["rings"] = _model(_shape(case), 2 * seed, case["position"])
        s["drafter"], _ = _model(DRAFTER, 2 * seed + 1, case["draft_position"])
        s["plan"] = model.H1Plan(s["target"], s["drafter"], case["position"], case["draft_position"], seed=seed, **OPTIONS)
        s["plan"].root.fill_(_tokens(seed, 1)[0])
    elif kind == "session":
        s["target"], s["rings"] = _model(_shape(case), 2 * seed, case["position"])
        s["drafter"], _ = _model(DRAFTER, 2 * seed + 1, case["position"])
        s["root"], s["position"], s["cycles"] = _tokens(seed, 1)[0], case["position"], case["cycles"]
        s["session"] = model.Session(s["target"], s["drafter"], s["root"], s["position"], s["position"], s["cycles"], seed=seed, **OPTIONS)
    elif kind == "decode":
        s["model"], s["rings"] = _model(_shape(case), seed, case["position"])
        s["tokens"], s["position"] = _device_tokens(seed, 1), case["position"]
    elif kind == "draft":
        s["drafter"], s["rings"] = _model(DRAFTER, seed, 0)
        tokens = _tokens(seed, case["prefix"] + case["append"])
        s["plan"] = model.DraftPlan(s["drafter"])
        s["plan"].append(tokens[:case["prefix"]])
        s["append"] = tokens[case["prefix"]:]
        s["words"] = [random.Random(seed + i).getrandbits(32) for i in range(case["horizon"])]
        s["options"] = hip.SamplerOptions(OPTIONS["temperature"], OPTIONS["top_k"], OPTIONS["top_p"], OPTIONS["min_p"], 1.0)
    elif kind == "tree":
        s["target"], s["rings"] = _model(_shape(case), seed, case["position"])
        s["ticket"] = model.VerifyTicket(s["target"], case["position"] + 4)
        s["parents"] = [None if p == "-" else int(p) for p in case["parents"].split(",")]
        s["tokens"], s["position"], s["keep"] = _tokens(seed, len(s["parents"])), case["position"], case["keep"]
        # the deepest path of the tree, ending in its last deepest row
        depth = [0] * len(s["parents"])
        for r, p in enumerate(s["parents"]):
            depth[r] = 0 if p is None else depth[p] + 1
        node, path = max(range(len(depth)), key=lambda r: (depth[r], r)), []
        while node is not None:
            path.insert(0, node)
            node = s["parents"][node]
        s["path"] = path
    elif kind == "sample":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        s["p"] = 2.0 * torch.randn((2, TARGET.vocab), device="cuda", generator=gen)
        s["q"] = s["p"][0] + 0.5 * torch.randn(TARGET.vocab, device="cuda", generator=gen)
        s["options"] = hip.SamplerOptions(OPTIONS["temperature"], case["top_k"], OPTIONS["top_p"], OPTIONS["min_p"], 1.0)
        s["seed"], s["top_k"] = seed, case["top_k"]
    else:
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        dtype, k, n = case["dtype"], case["k"], case["n"]
        blocks = n * (k // synth.BLOCK_ELEMS[dtype])
        raw = torch.randint(0, 256, (blocks, synth.BLOCK_BYTES[dtype]), dtype=torch.uint8, device="cuda", generator=gen)
        for at in {synth.Q4_K: (0, 2), synth.Q6_K: (208,), synth.Q8_0: (0,)}[dtype]:   # the blocks' fp16 scales
            scale = torch.randn(blocks, device="cuda", generator=gen).mul_(0.02).abs_().to(torch.float16)
            raw[:, at:at + 2] = scale.view(torch.uint8).view(blocks, 2)
        s.update(dtype=dtype, k=k, n=n, canonical=raw.view(-1))
        if kind == "gemv":
            s["tiles"] = hip.repack(dtype, s["canonical"], k, n)
            s["x"] = torch.randn((case["rows"], k), device="cuda", generator=gen)
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "prefill":
        hidden, status = s["model"].prefill(s["tokens"], s["position"])
        return {"hidden": hidden, "status": status, "rings": s["rings"]}
    if kind == "step":
        plan = s["plan"]
        plan.step(0)
        b = plan.buffers()
        return {"decision": _decision(plan.result), "status": plan.status, "hidden": b["target_hidden"], "p_logits": b["p_logits"],
                "q_logits": b["q_logits"], "candidates": _candidates(b["candidates"]), "rows": [plan.t_pk, plan.t_pv, plan.d_pk, plan.d_pv],
                "rings": s["rings"]}
    if kind == "session":
        sess = s["session"]
        hip.check(hip.lib().guffin_hip_session_start(C.byref(sess.s), s["root"], s["position"], s["position"]))
        emitted = []
        for _ in range(s["cycles"]):
            sess.submit()
            emitted += sess.complete()
        b = sess.buffers()
        return {"emitted": torch.tensor(emitted), "decision": _decision(sess.result), "hidden": b["target_hidden"], "p_logits": b["p_logits"],
                "q_logits": b["q_logits"], "rings": s["rings"]}
    if kind == "decode":
        m = s["model"]
        hidden, sums, pk, pv, status = m.forward(s["tokens"], s["position"])
        logits = hip.gemv_packed(m.shape.embed_dtype, m.head_tiles, hidden, sums, m.shape.vocab)
        token, logit = hip.argmax(logits, status)
        hip.check(hip.lib().guffin_hip_commit_rows(hip._stream(), C.byref(m.desc), hip._p(pk), hip._p(pv), hip._p(m.ring_k_table),
                                                   hip._p(m.ring_v_table), None, s["position"], 1))
        return {"token": token, "logit": logit, "status": status, "logits": logits, "hidden": hidden, "rings": s["rings"]}
    if kind == "draft":
        plan = s["plan"]
        plan.begin_transaction()
        plan.append(s["append"])
        proposed = plan.propose(s["words"], s["options"])
        plan.abort_transaction()
        return {"proposed": torch.tensor(proposed), "rings": s["rings"]}
    if kind == "tree":
        ticket = s["ticket"]
        ticket.encode_tree(s["tokens"], s["parents"], s["position"])
        ticket.submit()
        raised = ticket.complete()
        ticket.provisional_commit(s["path"])
        ticket.finalize(s["keep"])
        rows = len(s["tokens"])   # of the four rows a ticket has room for
        return {"raised": raised, "candidates": _candidates(ticket.candidates[:rows * hip.candidates_dtype.itemsize]), "rings": s["rings"]}
    if kind == "sample":
        cands, status = hip.select_candidates(s["p"], s["top_k"])
        law, proposal, _ = hip.draft_law(s["q"], s["options"], seed=s["seed"], step=0)
        result = hip.spec_accept(cands, law, proposal, s["options"], seed=s["seed"], step=0, status=status)
        return {"candidates": _candidates(cands), "law": law.view(torch.int32), "proposal": proposal, "decision": _decision(result),
                "status": status}
    if kind == "gemv":
        receipt = hip.group_sums(s["x"])
        return hip.gemv_packed(s["dtype"], s["tiles"], s["x"], receipt, s["n"])
    return hip.repack(s["dtype"], s["canonical"], s["k"], s["n"])


# ---- what a pass cannot do without ------------------------------------------------------------------------

def _kv_bytes(sh, position, rows):
    """The ring rows a run at `position` sees, once, and its own rows written."""
    seen = sum(min(position, sh.sliding_window) if sh.is_local(l) else position for l in range(sh.layers))
    return 2 * 2 * sh.kv_width * (seen + rows * sh.layers)


def _attention_flops(sh, position, rows):
    """Scores and values of every (row, visible token) pair."""
    pairs = 0
    for l in range(sh.layers):
        for r in range(rows):
            t = position + r + 1
            pairs += min(t, sh.sliding_window) if sh.is_local(l) else t
    return 4 * sh.q_width * pairs


def _pass_work(sh, position, rows, head_rows):
    weights = sh.body_weight_bytes() + (sh.head_bytes() if head_rows else 0)
    macs = rows * sum(k * n for k, n in sh.proj_shapes()) * sh.layers + head_rows * sh.hidden * sh.vocab
    return (weights + _kv_bytes(sh, position, rows) + 8 * rows * sh.hidden + 4 * head_rows * sh.vocab,
            2 * macs + _attention_flops(sh, position, rows))


def work(case):
    kind, parts = case["kind"], []
    if kind == "prefill":
        parts = [_pass_work(_shape(case), case["position"], case["rows"], 0)]
    elif kind == "step":
        parts = [_pass_work(TARGET, case["position"], 2, 2), _pass_work(DRAFTER, case["draft_position"], 1, 1)]
    elif kind == "session":
        parts = case["cycles"] * [_pass_work(TARGET, case["position"], 2, 2), _pass_work(DRAFTER, case["position"], 1, 1)]
    elif kind == "decode":
        parts = [_pass_work(_shape(case), case["position"], 1, 1)]
    elif kind == "draft":
        # the accepted tokens could go through together; the proposals depend on each other
        parts = [_pass_work(DRAFTER, case["prefix"], case["append"], 1)]
        parts += [_pass_work(DRAFTER, case["prefix"] + case["append"] + i, 1, 1) for i in range(case["horizon"] - 1)]
    elif kind == "tree":
        rows = len(case["parents"].split(","))
        parts = [_pass_work(TARGET, case["position"], rows, rows)]
    elif kind == "sample":
        parts = [(3 * 4 * TARGET.vocab, 3 * TARGET.vocab)]
    elif kind == "gemv":
        parts = [(synth.weight_bytes(case["dtype"], case["k"], case["n"]) + 4 * case["rows"] * (case["k"] + case["n"]),
                  2 * case["rows"] * case["k"] * case["n"])]
    else:
        parts = [(2 * synth.weight_bytes(case["dtype"], case["k"], case["n"]), 0)]
    return {"bytes": float(sum(b for b, _ in parts)), "flops": float(sum(f for _, f in parts))}


def tolerance(case):
    kind = case["kind"]
    if kind == "repack":
        return "exact"
    if kind == "gemv":       # exact products, 32-bit sums of them
        return {"rel": 1e-5}
    if kind == "sample":     # whole numbers and double-precision masses of given 32-bit logits
        return {"rel": 1e-6}
    # Sums are 32-bit over exact products.  Keys and values are kept in 16 bits between a layer and the next: where two
    # such sums fall on either side of a rounding, an element is off by one or two units of its last place (1e-3 of it)
    # and the pass goes on with that; few elements are, so the whole stays far closer.  Candidates that tie up to that
    # may change places.
    return {"rel": 1e-4, "max": 4e-3, "differ": 0.01}
