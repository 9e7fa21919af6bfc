"""The Timopel decoder through the engine against the plain implementation, float32 and bfloat16:
whole prompts and first tokens; prompt then token by token; portions down to two tokens; unequal requests
in one batch against each alone, with pages and slots that are freed and used again; a far key among
hundreds, at page borders, in prompts and in decoding; positions just before and at a temperature step; a
sink that outweighs the keys; long decoding; greedy generation through the scheduler; the trace runner as a
program; and the kernels alone."""
from __future__ import annotations

import math
import random

import pytest
import torch

from tests import timopel_models as tm
from tests.plain import timopel_plain as tp

pytestmark = pytest.mark.gpu

DTYPES = ["float32", "bfloat16"]
NAMES = ["TA", "TB", "TC", "TD", "TE"]


def tokens_for(n, seed, vocab, folder=None, dtype="float32"):
    """Random tokens; for a comparison in bfloat16 of a model with routers (`folder` given), tokens whose routing
    decisions are all clear in the plain model, so that the comparison does not rest on a close call."""
    if folder is not None and dtype == "bfloat16":
        return tm.clear_tokens(folder, n, seed, vocab)
    rng = random.Random(seed)
    return [rng.randrange(vocab) for _ in range(n)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_whole_prompts_and_first_tokens(tmp_path, name, dtype):
    folder = tm.make_folder(tmp_path, name)
    engine = tm.engine_for(folder, dtype)
    vocab = tm.MODELS[name][0].vocab
    for n in (1, 2, 3, 5, 61):
        tokens = tokens_for(n, 100 + n, vocab, folder, dtype)
        got = tm.run_portions(engine, f"r{n}", tokens, [n])
        tm.assert_matches_plain(got, folder, tokens, dtype, f"{name} whole {n}")
    engine.runner.cache.check_invariants()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_prompt_then_token_by_token(tmp_path, name, dtype):
    folder = tm.make_folder(tmp_path, name)
    engine = tm.engine_for(folder, dtype)
    vocab = tm.MODELS[name][0].vocab
    tokens = tokens_for(84, 7, vocab, folder, dtype)
    got = tm.run_portions(engine, "r", tokens, [84 - 45] + [1] * 45)     # temperature steps pass under decoded tokens
    tm.assert_matches_plain(got, folder, tokens, dtype, f"{name} prompt + 45 single tokens")
    got = tm.run_portions(engine, "s", tokens[:30], [1] * 30)             # from the very first token on
    tm.assert_matches_plain(got, folder, tokens, dtype, f"{name} token by token from the start", rows=slice(0, 30))
    if dtype == "float32":
        whole = tm.run_portions(engine, "w", tokens, [84])
        assert tm.row_distance(got, whole[:30]).max().item() <= 2e-5


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_portions_of_changing_size(tmp_path, name, dtype):
    folder = tm.make_folder(tmp_path, name)
    engine = tm.engine_for(folder, dtype)
    vocab = tm.MODELS[name][0].vocab
    tokens = tokens_for(73, 8, vocab, folder, dtype)
    for portions in ([7, 2, 16, 3, 2, 9, 2, 11, 5, 4, 1, 1, 2, 8], [2] * 10 + [53], [1, 3, 69], [40, 33]):
        got = tm.run_portions(engine, "r", tokens, portions)
        tm.assert_matches_plain(got, folder, tokens, dtype, f"{name} portions {portions}")


def mixed_trace(rng, reqs, max_live=4):
    """Up to `max_live` live requests; portions of some beside single tokens of others; staggered."""
    fed = {k: 0 for k in reqs}
    order, live, steps, nxt = list(reqs), [], [], 0
    while nxt < len(order) or live:
        while len(live) < max_live and nxt < len(order) and (not live or rng.random() < 0.6):
            live.append(order[nxt])
            nxt += 1
        entries, ended = [], []
        for k in list(live):
            if rng.random() < 0.2 and len(live) > 1:
                continue                         # left out of this step, goes on later
            n = min(len(reqs[k]) - fed[k], rng.choice([1, 1, 1, 2, 3, 5, 8, 13]))
            entries.append((k, reqs[k][fed[k]: fed[k] + n]))
            fed[k] += n
            if fed[k] == len(reqs[k]):
                ended.append(k)
                live.remove(k)
        if entries:
            steps.append((entries, ended))
    return steps


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_unequal_requests_together_with_pages_and_slots_used_again(tmp_path, name, dtype):
    from serve_amd.engine.batch import Segment
    folder = tm.make_folder(tmp_path, name)
    lengths = [23, 41, 9, 30, 17, 2, 36, 1, 40, 28, 33, 5]
    # four live requests of at most 41 tokens: pool and slots are far fewer than the requests need together
    engine = tm.engine_for(folder, dtype, num_pages=4 * 11 + 1, page_size=4, max_requests=4)
    vocab = tm.MODELS[name][0].vocab
    reqs = {f"q{i}": tokens_for(n, 300 + i, vocab, folder, dtype) for i, n in enumerate(lengths)}
    steps = mixed_trace(random.Random(13), reqs)
    rows = {k: [] for k in reqs}
    slots_seen, pages_seen = {}, {}
    for entries, ended in steps:
        segs = []
        for k, toks in entries:
            if k not in engine.runner.cache:
                assert engine.runner.admit(k)
                slots_seen.setdefault(engine.runner.cache.slot_of(k), []).append(k)
            segs.append(Segment(k, toks, list(range(len(toks)))))
        logits = engine.step(segs)
        at = 0
        for k, toks in entries:
            rows[k].append(logits[at: at + len(toks)])
            at += len(toks)
            for page in engine.runner.cache.block_table(k, 0):
                pages_seen.setdefault(page, set()).add(k)
        for k in ended:
            engine.runner.release(k)
        engine.runner.cache.check_invariants()
    assert any(len(v) > 1 for v in slots_seen.values()), "no slot was used twice"
    assert any(len(v) > 1 for v in pages_seen.values()), "no page went from one request to another"
    for k, toks in reqs.items():
        tm.assert_matches_plain(torch.cat(rows[k]), folder, toks, dtype, f"{name} request {k} in the mix")


def one_layer_model(tmp_path, name, heads=2, kv_heads=1, dim=16, vdim=16, scale=1.0, temp=None, seed=11, vocab=90):
    from serve_amd.config.timopel import TimopelConfig, TimopelLayerConfig
    cfg = TimopelConfig(vocab=vocab, width=64, eps=1e-5, residual_mult=1.0, embedding_scale=1.0, layers=(
        TimopelLayerConfig(tm._att(heads, kv_heads, dim, vdim, scale, temp), None),))
    return tm.make_folder(tmp_path, name, config=cfg, seed=seed)


def far_key_model(tmp_path):
    """One attention layer and an embedding table made so that one score stands out: the row of token 1 is set
    so that, behind the layer's first norm and its query matrix, the queries of both heads point along the
    normed key of token 0.  A sequence that ends in token 1 and holds token 0 once, far back, then reads that
    one key with nearly all of its weight (its score is about 16 times the scale, the others' are spread by 4 times
    the scale around zero)."""
    import os
    from safetensors.torch import save_file
    folder = one_layer_model(tmp_path, "far", scale=2.5)
    W = {k: v.double() for k, v in tm.plain_weights(folder).items()}
    h0 = tp.rms_norm(W["embed"][0:1], W["l0.norm1"], 1e-5)
    k0 = tp.rms_norm((h0 @ W["l0.mix.k"].T).view(1, 1, 16), W["l0.mix.k.norm"], 1e-5)[0, 0]
    # h1 with W_q h1 = [k0 | k0] (per head), then the table's row as the normed stream's pre-image
    want_q = torch.cat([k0 / W["l0.mix.q.norm"]] * 2)
    h1 = torch.linalg.pinv(W["l0.mix.q"]) @ want_q
    row = h1 / W["l0.norm1"]
    out = tm.plain_weights(folder)
    out["embed"][1] = (row / row.pow(2).mean().sqrt()).to(out["embed"].dtype)
    save_file({k: v.contiguous() for k, v in out.items()}, os.path.join(folder, "model.safetensors"))
    return folder


@pytest.mark.parametrize("dtype", DTYPES)
def test_a_far_key_among_hundreds(tmp_path, dtype):
    folder = far_key_model(tmp_path)
    rng = random.Random(5)
    n = 420
    for far in (3, 37, 203):                  # in the first page, further on, and the last key of a page (page size 4)
        with_key = [rng.randrange(2, 90) for _ in range(n - 1)] + [1]
        with_key[far] = 0
        without = list(with_key)
        without[far] = 2
        want = tm.plain_logits(folder, with_key)[-1:]
        # losing that one key would move the last row by far more than the tolerance
        assert tm.row_distance(tm.plain_logits(folder, without)[-1:], want).item() > 2 * tm.TOLERANCE["bfloat16"]
        engine = tm.engine_for(folder, dtype, num_pages=120, page_size=4)
        got = tm.run_portions(engine, "r", with_key, [n - 3, 1, 1, 1])[-1:]
        tm.assert_rows_close(got, want, dtype, f"key {far} of {n}, read by a token decoded alone")
        got = tm.run_portions(engine, "r", with_key, [200, 220])[-1:]
        tm.assert_rows_close(got, want, dtype, f"key {far} of {n}, read from a portion")


@pytest.mark.parametrize("dtype", DTYPES)
def test_a_sink_that_outweighs_the_keys(tmp_path, dtype):
    """Sinks of +8 and -6 in the two heads of one layer: the first head's output nearly vanishes, the second
    head's does not feel its sink; without the sinks the logits are far away (the plain model says so)."""
    import os
    from safetensors.torch import save_file
    folder = one_layer_model(tmp_path, "sink", scale=0.3, temp=(0.1, 4))
    W = tm.plain_weights(folder)
    W["l0.mix.sink"] = torch.tensor([8.0, -6.0]).to(W["l0.mix.sink"].dtype)
    save_file({k: v.contiguous() for k, v in W.items()}, os.path.join(folder, "model.safetensors"))
    tokens = tokens_for(150, 3, 90)
    want = tm.plain_logits(folder, tokens)
    none = dict(W)
    none["l0.mix.sink"] = torch.tensor([-1e4, -1e4])
    moved = tm.row_distance(tm.plain_logits(folder, tokens, weights=none), want) > 2 * tm.TOLERANCE["bfloat16"]
    assert moved[:20].all() and moved.float().mean() > 0.8
    engine = tm.engine_for(folder, dtype, num_pages=80, page_size=4)
    for portions in ([150], [100] + [1] * 50, [3, 2, 60, 85]):
        tm.assert_rows_close(tm.run_portions(engine, "r", tokens, portions), want, dtype, f"sinks, portions {portions[:4]}")


@pytest.mark.parametrize("dtype", DTYPES)
def test_temperature_steps_in_prompts_and_in_decoding(tmp_path, dtype):
    """A strong temperature (coef 3) that steps every 6 positions: portions that end just before, at and just
    behind a step, and single tokens across steps.  A step that came one position late would show."""
    import copy
    folder = one_layer_model(tmp_path, "temp", scale=0.5, temp=(3.0, 6), seed=12)
    tokens = tokens_for(40, 9, 90)
    want = tm.plain_logits(folder, tokens)
    late = copy.deepcopy(tm.plain_config(folder))
    late["layers"][0]["mixer"]["q_temp"]["every"] = 7
    moved = tm.row_distance(tm.plain_logits(folder, tokens, late), want)
    # (positions 5 and 11 are the first whose count of steps differs between the two)
    assert moved[:5].max().item() == 0.0 and moved[5] > 2 * tm.TOLERANCE["bfloat16"] and moved[11] > 100 * tm.TOLERANCE["float32"]
    engine = tm.engine_for(folder, dtype, page_size=4)
    for portions in ([40], [4, 1, 1, 1, 4, 1, 1, 1, 26], [5, 6, 6, 7] + [1] * 16, [1] * 40):
        tm.assert_rows_close(tm.run_portions(engine, "r", tokens, portions), want, dtype, f"temperature, portions {portions[:5]}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["TA", "TB"])
def test_long_decoding(tmp_path, name, dtype):
    folder = tm.make_folder(tmp_path, name)
    engine = tm.engine_for(folder, dtype, num_pages=80)
    vocab = tm.MODELS[name][0].vocab
    tokens = tokens_for(260, 31, vocab, folder, dtype)
    got = tm.run_portions(engine, "r", tokens, [4] + [1] * 256)
    tm.assert_matches_plain(got, folder, tokens, dtype, f"{name} 256 single tokens")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["TA", "TB"])
def test_greedy_generation_through_the_scheduler(tmp_path, name, dtype):
    """`generate` (scheduler, mixed steps, graphs, steps launched ahead of the host) picks the tokens the
    plain model picks, as long as the plain model's choice is clear."""
    from serve_amd.engine.engine import Request
    folder = tm.make_folder(tmp_path, name)
    engine = tm.engine_for(folder, dtype, num_pages=128, page_size=8, max_requests=3)
    vocab = tm.MODELS[name][0].vocab
    prompts = [tokens_for(n, 50 + n, vocab, folder, dtype) for n in (5, 19, 1, 33, 8)]
    new = 12
    reqs = [Request(torch.tensor(p), len(p), new) for p in prompts]
    out = engine.generate(reqs, temperature=0.0, return_logits="all")
    compared = 0
    for p, o in zip(prompts, out):
        assert o.error is None and len(o.generated_tokens) == new
        seq = list(p)
        for i, tok in enumerate(o.generated_tokens.tolist()):
            row = tm.plain_logits(folder, seq)[-1]
            top2 = row.topk(2).values
            if (top2[0] - top2[1]).item() < (1e-3 if dtype == "float32" else 0.15):
                break                            # the plain model's own choice is a close call: stop comparing
            assert tok == int(row.argmax()), f"{name}: token {i} after a prompt of {len(p)}"
            if dtype == "float32":
                tm.assert_rows_close(o.logits[i: i + 1], row[None], dtype, f"{name} logits of generated token {i}")
            seq.append(tok)
            compared += 1
    assert compared >= new
    engine.runner.cache.check_invariants()
    assert engine.runner.cache.free_slots() == 3
    # without the logits the scheduler samples on the device and replays decode steps from graphs: the same tokens
    again = engine.generate([Request(torch.tensor(p), len(p), new) for p in prompts], temperature=0.0)
    if dtype == "float32":
        assert [o.generated_tokens.tolist() for o in again] == [o.generated_tokens.tolist() for o in out]


# ---------------------------------------------------------------------------------------------
# the kernels alone
# ---------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("pad", [5, 8])      # rows that do not keep 16-byte alignment (the general kernel), and rows that do
@pytest.mark.parametrize("H,G,D,Dv,Dp", [(4, 2, 16, 16, 16), (6, 1, 24, 40, 48), (3, 3, 10, 7, 16), (2, 1, 136, 24, 144),
                                         (5, 5, 128, 64, 128)])
def test_qk_norm_kv_write(dtype, H, G, D, Dv, Dp, pad):
    from serve_amd import ops
    torch.manual_seed(D)
    T, page, P = 11, 4, 9
    width = H * D + G * (D + Dv)
    wide = torch.randn(T, width + pad, device="cuda").to(dtype)             # rows inside wider rows
    qkv = wide[:, :width]
    first = torch.randn(T, G * Dv + pad, device="cuda").to(dtype)[:, : G * Dv]
    wq, wk = torch.rand(D, device="cuda") + 0.5, torch.rand(D, device="cuda") + 0.5
    positions = torch.tensor([0, 1, 2, 3, 4, 5, 6, 7, 30, 31, 32], dtype=torch.int32, device="cuda")
    slots = torch.tensor([5, 6, 7, 8, 20, 21, 22, 23, -1, 1, 35], dtype=torch.int32, device="cuda")
    k_pages = torch.full((P, G, page, Dp), 7.0, device="cuda").to(dtype)
    v_pages = torch.full((P, G, Dp, page), 7.0, device="cuda").to(dtype)
    q = torch.full((T, H * Dp), 7.0, device="cuda").to(dtype)
    eps, coef, every, lam = 1e-5, 0.6, 4, 0.3
    ops.qk_norm_kv_write(qkv, q, positions, slots, k_pages, v_pages, wq, wk, eps, H, G, D, Dv, coef, every, first, lam)
    x = qkv.double().cpu()
    temp = tp.query_temperature(positions.cpu().long(), coef, every)
    want_q = tp.rms_norm(x[:, : H * D].view(T, H, D), wq.double().cpu(), eps) * temp[:, None, None]
    want_k = tp.rms_norm(x[:, H * D: (H + G) * D].view(T, G, D), wk.double().cpu(), eps)
    want_v = (1 - lam) * x[:, (H + G) * D:].view(T, G, Dv) + lam * first.double().cpu().view(T, G, Dv)
    tol = dict(atol=1e-5, rtol=1e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=1e-2)
    got_q = q.double().cpu().view(T, H, Dp)
    assert torch.allclose(got_q[:, :, :D], want_q, **tol) and (got_q[:, :, D:] == 0).all()
    kp, vp = k_pages.double().cpu(), v_pages.double().cpu()
    written = set()
    for t, s in enumerate(slots.tolist()):
        if s < 0:
            continue
        pg, off = divmod(s, page)
        written.add((pg, off))
        assert torch.allclose(kp[pg, :, off, :D], want_k[t], **tol) and (kp[pg, :, off, D:] == 0).all()
        assert torch.allclose(vp[pg, :, :Dv, off], want_v[t], **tol) and (vp[pg, :, Dv:, off] == 0).all()
    for pg in range(P):
        for off in range(page):
            if (pg, off) not in written:
                assert (kp[pg, :, off] == 7.0).all() and (vp[pg, :, :, off] == 7.0).all(), "a slot that no token named was written"
    # queries alone (no slots), no temperature, no blending
    q2 = torch.empty_like(q)
    ops.qk_norm_kv_write(qkv, q2, positions, None, None, None, wq, wk, eps, H, G, D, Dv)
    assert torch.allclose(q2.double().cpu().view(T, H, Dp)[:, :, :D], want_q / temp[:, None, None], **tol)


def _attention_case(dtype, H, G, D, page, lens, ctxs, seed=0):
    """Random pages and block tables for segments of `lens` tokens that end contexts of `ctxs` tokens."""
    from serve_amd.ops import AttentionStep
    torch.manual_seed(seed)
    B, T = len(lens), sum(lens)
    per = [-(-c // page) for c in ctxs]
    P = sum(per) + 3
    order = torch.randperm(P - 1)[: sum(per)] + 1          # (page 0 stays unused)
    bt = torch.zeros(B, max(per), dtype=torch.int32)
    at = 0
    for b in range(B):
        bt[b, : per[b]] = order[at: at + per[b]].int()
        at += per[b]
    k_pages = torch.randn(P, G, page, D)
    v_pages = torch.randn(P, G, D, page)
    q = torch.randn(T, H * D)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    seg = [b for b, n in enumerate(lens) for _ in range(n)]
    dev = lambda t, dt=None: (t.to(dt) if dt else t).cuda().contiguous()   # noqa: E731
    step = AttentionStep(num_segments=B, num_tokens=T, cu_q=dev(torch.tensor(cu, dtype=torch.int32)),
                         ctx_len=dev(torch.tensor(ctxs, dtype=torch.int32)), seg_of_token=dev(torch.tensor(seg, dtype=torch.int32)),
                         q_lens=list(lens), ctx_lens=list(ctxs), max_q_len=max(lens), max_ctx_len=max(ctxs),
                         decode_only=all(n == 1 for n in lens))
    q, k_pages, v_pages = q.to(dtype), k_pages.to(dtype), v_pages.to(dtype)       # (the reference reads the rounded values)
    return step, dev(q), dev(k_pages), dev(v_pages), dev(bt), (q.double(), k_pages.double(), v_pages.double(), bt, cu)


def _attention_reference(host, lens, ctxs, H, G, D, page, scale, sinks):
    q, kp, vp, bt, cu = host
    out = torch.zeros(q.shape[0], H, D, dtype=torch.float64)
    for b, (n, c) in enumerate(zip(lens, ctxs)):
        pages = bt[b, : -(-c // page)].long()
        for h in range(H):
            g = h // (H // G)
            keys = kp[pages, g].reshape(-1, D)[:c]
            vals = vp[pages, g].permute(0, 2, 1).reshape(-1, D)[:c]
            for j in range(n):
                pos = c - n + j
                s = (keys[: pos + 1] @ q[cu[b] + j].view(H, D)[h]) * scale
                sink = torch.tensor(-math.inf if sinks is None else float(sinks[h]), dtype=torch.float64)
                out[cu[b] + j, h] = tp.sink_softmax(s[None], sink[None])[0] @ vals[: pos + 1]
    return out.view(q.shape[0], H * D)


ATTENTION_CASES = [
    # (heads, kv heads, head size, page size, portion lengths, contexts)
    (4, 2, 32, 8, [1, 1, 1], [5, 300, 64]),                    # single tokens, short contexts: keys cut inside a workgroup
    (8, 1, 64, 16, [1] * 5, [1500, 900, 2200, 33, 700]),       # single tokens over long contexts: keys cut over the grid
    (6, 3, 48, 4, [40, 7, 130], [40, 90, 130]),                # prompt portions, whole prompts among them
    (2, 1, 16, 16, [20], [2100]),                              # a short portion of a long context: its keys cut over the grid
    (4, 1, 128, 8, [1, 1, 1, 1, 33, 2], [9, 70, 200, 64, 33, 58]),   # single tokens first, then portions: two launches
    (3, 3, 144, 4, [1, 9], [37, 9]),                           # a head size only the general kernel takes
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", range(len(ATTENTION_CASES)))
def test_attention_kernels_with_sinks(dtype, case):
    """Every family of attention kernels with a sink in each head's softmax, against the plain softmax with one
    more term in its denominator; sinks far below the scores change nothing; no sinks: the kernels as before."""
    from serve_amd import ops
    H, G, D, page, lens, ctxs = ATTENTION_CASES[case]
    step, q, k_pages, v_pages, bt, host = _attention_case(dtype, H, G, D, page, lens, ctxs, seed=case)
    scale = 0.5 / math.sqrt(D)
    sinks = torch.linspace(-2.0, 3.0, H)
    tol = dict(atol=2e-5, rtol=1e-4) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    for s in (sinks, None, torch.full((H,), -80.0)):
        out = torch.empty(q.shape[0], H * D, dtype=dtype, device="cuda")
        ops.paged_attention(q, H * D, out, k_pages, v_pages, bt, step, H, scale, None,
                            None if s is None else s.float().cuda())
        want = _attention_reference(host, lens, ctxs, H, G, D, page, scale, None if s is None or s[0] < -50 else s)
        got = out.double().cpu()
        assert torch.allclose(got, want, **tol), f"sinks {None if s is None else s.tolist()}: max diff {(got - want).abs().max():.3g}"


@pytest.mark.parametrize("experts,top", [(5, 1), (16, 2), (70, 3), (130, 8), (4, 4)])
def test_route_over_all_experts(experts, top):
    from serve_amd import ops
    torch.manual_seed(experts)
    T = 37
    logits = (torch.randn(T, experts + 1, device="cuda") * 3).contiguous()
    ids = torch.empty(T, top, dtype=torch.int32, device="cuda")
    w = torch.empty(T, top, dtype=torch.float32, device="cuda")
    ops.moe_route(logits, experts, top, ids, w, over_all=True, scale=2.5)
    want_ids, want_w = tp.route(logits[:, :experts].double().cpu(), top, 2.5)
    assert torch.equal(ids.long().cpu(), want_ids)
    assert torch.allclose(w.double().cpu(), want_w, atol=1e-6, rtol=1e-5)
    # the experts' call routes by itself for few tokens: the same ids and weights
    d, F = 32, 16
    h = torch.randn(9, d, device="cuda")
    wg, wu, wd = torch.randn(experts, F, d, device="cuda"), torch.randn(experts, F, d, device="cuda"), torch.randn(experts, d, F, device="cuda")
    ids2, w2 = torch.empty(9, top, dtype=torch.int32, device="cuda"), torch.empty(9, top, device="cuda")
    ops.moe_experts(h, ids2, wg, wu, wd, torch.empty(9 * top, d, device="cuda"), logits[:9].contiguous(), w2,
                    over_all=True, scale=2.5, gate="clamped_swish", limit=1.0)
    assert torch.equal(ids2, ids[:9]) and torch.equal(w2, w[:9])


@pytest.mark.parametrize("T,d,F", [(45, 72, 40), (45, 75, 42), (400, 64, 48)])   # few rows; sizes the matrix cores do not take; many rows
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_experts_with_clamped_gates(dtype, T, d, F):
    from serve_amd import ops
    torch.manual_seed(3)
    E, top, limit = 7, 3, 0.8
    h = torch.randn(T, d, device="cuda").to(dtype)
    wg, wu = (torch.randn(E, F, d, device="cuda") * 0.2).to(dtype), (torch.randn(E, F, d, device="cuda") * 0.2).to(dtype)
    wd = (torch.randn(E, d, F, device="cuda") * 0.2).to(dtype)
    ids = torch.stack([torch.randperm(E, device="cuda")[:top] for _ in range(T)]).int().contiguous()
    yk = torch.empty(T * top, d, dtype=torch.float32, device="cuda")
    ops.moe_experts(h, ids, wg, wu, wd, yk, gate="clamped_swish", limit=limit)
    hd = h.double().cpu()
    clipped = 0
    for t in list(range(0, T, 7)) + [T - 1]:
        for k in range(top):
            e = int(ids[t, k])
            g, u = hd[t] @ wg[e].double().cpu().t(), hd[t] @ wu[e].double().cpu().t()
            clipped += int((g > limit).sum() + (u.abs() > limit).sum())
            a = tp.clamped_swish_gate(g, u, limit)
            if dtype == torch.bfloat16:
                a = a.to(dtype).double()
            want = a @ wd[e].double().cpu().t()
            assert torch.allclose(yk[t * top + k].double().cpu(), want, atol=2e-4 if dtype == torch.float32 else 2e-2, rtol=1e-3)
    assert clipped > 20, "the limit was hardly reached: the test shows nothing"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind,limit", [("silu", 0.0), ("gelu_tanh", 0.0), ("clamped_swish", 0.7)])
def test_gates(dtype, kind, limit):
    from serve_amd import ops
    torch.manual_seed(1)
    for T, I in ((5, 24), (3, 37)):                  # whole groups of eight, and not
        gu = (torch.randn(T, 2 * I, device="cuda") * 2).to(dtype)
        out = torch.empty(T, I, device="cuda", dtype=dtype)
        ops.gate_mul(gu, out, kind, limit)
        g, u = gu.double().cpu()[:, :I], gu.double().cpu()[:, I:]
        want = {"silu": lambda: g * torch.sigmoid(g) * u, "gelu_tanh": lambda: tp.gelu_tanh(g) * u,
                "clamped_swish": lambda: tp.clamped_swish_gate(g, u, limit)}[kind]()
        assert torch.allclose(out.double().cpu(), want, atol=1e-5 if dtype == torch.float32 else 3e-2, rtol=1e-5 if dtype == torch.float32 else 1e-2)


def test_scaled_embedding_rows():
    from serve_amd import ops
    torch.manual_seed(2)
    for d, dt in ((64, torch.bfloat16), (50, torch.bfloat16), (50, torch.float32)):
        table = torch.randn(20, d, device="cuda").to(dt)
        ids = torch.tensor([3, 19, 0, 3], dtype=torch.int32, device="cuda")
        x = torch.empty(4, d, dtype=torch.float32, device="cuda")
        ops.embed(table, ids, x, scale=2.75)
        assert torch.equal(x, table[ids.long()].float() * 2.75)


# ---------------------------------------------------------------------------------------------
# the trace runner as a user runs it
# ---------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
def test_traces_through_the_program(tmp_path, dtype):
    """`bin/trace_run` as a child process on a model folder: whole prompts, prompt then single tokens, portions, and
    a mix of four live requests (pages for 256 tokens, so pages go from request to request), against the plain model."""
    import json
    import os
    import subprocess
    import numpy as np
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    name = "TA"
    folder = tm.make_folder(tmp_path, name)
    vocab = tm.MODELS[name][0].vocab
    reqs, steps = {}, []

    def feed(key, n, portions, seed):
        reqs[key] = tokens_for(n, seed, vocab, folder, dtype)
        at = 0
        for j, m in enumerate(portions):
            steps.append(([(key, reqs[key][at: at + m])], [key] if j == len(portions) - 1 else []))
            at += m
        assert at == n
    feed("whole", 50, [50], 1)
    feed("tail", 70, [30] + [1] * 40, 2)
    feed("cut", 61, [7, 2, 16, 3, 2, 9, 2, 11, 5, 4], 3)
    mixed = {f"m{i}": tokens_for(n, 40 + i, vocab, folder, dtype) for i, n in enumerate([23, 41, 9, 30, 17, 2, 36, 12, 40])}
    reqs.update(mixed)
    steps.extend(mixed_trace(random.Random(5), mixed))
    lines = [json.dumps({"step": i, "entries": [{"id": k, "tokens": t, "want": list(range(len(t)))} for k, t in entries],
                         "end": ended}) for i, (entries, ended) in enumerate(steps)]
    out = tmp_path / "out"
    proc = subprocess.run([os.path.join(root, "bin", "trace_run"), "--model", folder, "--dtype", dtype, "--out", str(out),
                           "--max-tokens", "256"], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stderr[-3000:]
    assert [l for l in proc.stdout.splitlines() if l.startswith("done")] == [f"done {i}" for i in range(len(steps))]
    rows = {k: [] for k in reqs}
    for i, (entries, _) in enumerate(steps):
        arr = torch.from_numpy(np.fromfile(out / f"{i}.f32", dtype="<f4").reshape(sum(len(t) for _, t in entries), vocab))
        at = 0
        for k, t in entries:
            rows[k].append(arr[at: at + len(t)])
            at += len(t)
    assert sum(len(t) for t in reqs.values()) > 256          # pages went from request to request
    for k, t in reqs.items():
        tm.assert_matches_plain(torch.cat(rows[k]), folder, t, dtype, f"trace request {k}")


def test_generate_from_the_command_line():
    """`python -m serve_amd generate` with the named shape: as many token lists as prompts, of the asked length."""
    import json
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    proc = subprocess.run([sys.executable, "-m", "serve_amd", "generate", "--shape", "timopel-tiny", "--random-prompts", "3:20",
                           "--max-new-tokens", "6", "--temperature", "0"], cwd=root, capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stderr[-3000:]
    lines = [json.loads(l) for l in proc.stdout.splitlines() if l.startswith("[")]
    assert len(lines) == 3 and all(len(l) == 6 and all(0 <= t < 512 for t in l) for l in lines)


@pytest.mark.parametrize("dtype", DTYPES)
def test_steps_with_prompt_portions_replayed_from_graphs(tmp_path, dtype):
    """Six slots and portions of eight tokens: steps of a few decoding requests in front of prompt portions come
    again and again, are padded with inert segments (no pages, no slot: nothing of them is stored) and replayed from
    graphs; the greedy tokens are those of the same schedule launched kernel by kernel, and the plain model's where
    its choice is clear."""
    from serve_amd.engine.engine import Request
    name = "TA"
    folder = tm.make_folder(tmp_path, name)
    vocab = tm.MODELS[name][0].vocab
    rng = random.Random(46)
    count = 30
    prompts = [tokens_for(rng.randrange(9, 30), 700 + i, vocab, folder, dtype) for i in range(count)]
    new = [rng.randrange(4, 12) for _ in range(count)]
    kw = dict(num_pages=64, page_size=8, max_requests=6)
    outs = []
    for mixed in (True, False):
        from serve_amd.config.engine import EngineConfig
        from serve_amd.engine.engine import Engine
        engine = Engine.from_folder(folder, EngineConfig(dtype=dtype, max_context=256, max_tokens_per_step=24, prefill_chunk=8,
                                                         graph_mixed_steps=mixed, **kw))
        out = engine.generate([Request(torch.tensor(p), len(p), n) for p, n in zip(prompts, new)], temperature=0.0)
        assert all(r.error is None and len(r.generated_tokens) == n for r, n in zip(out, new))
        graphs = [k for k, e in engine.runner._graphs.items() if k[0] == "mixed" and e.graph is not None and e.launches > 2]
        assert bool(graphs) == mixed, f"mixed graphs {mixed}: replayed shapes {graphs}"
        engine.runner.cache.check_invariants()
        outs.append([r.generated_tokens.tolist() for r in out])
    if dtype == "float32":
        assert outs[0] == outs[1]
    compared = 0
    for p, got in zip(prompts, outs[0]):
        seq = list(p)
        for tok in got:
            row = tm.plain_logits(folder, seq)[-1]
            top2 = row.topk(2).values
            if (top2[0] - top2[1]).item() < (1e-3 if dtype == "float32" else 0.15):
                break
            assert tok == int(row.argmax())
            seq.append(tok)
            compared += 1
    assert compared > 3 * count


@pytest.mark.parametrize("T,N,K,E,top", [(1, 1, 8, 1, 1), (15, 17, 40, 17, 2), (16, 16, 256, 16, 1), (17, 33, 2048, 32, 4), (33, 48, 1000, 40, 4),
                                         (100, 65, 4096, 64, 6), (47, 80, 2056, 80, 4), (1000, 96, 264, 90, 8)])
@pytest.mark.parametrize("mode", ["chosen", "all", "sigmoid"])
def test_router_product_with_the_routing(T, N, K, E, top, mode):
    """One kernel for the router's logits and what is chosen by them: the logits against 64 bits, the choice as the routing kernel
    makes it from the same logits; rows of the matrix, tokens and columns that are no whole tiles or steps."""
    from serve_amd import ops
    g = torch.Generator("cuda").manual_seed(T + N + K)
    h = torch.randn((T, K), device="cuda", generator=g).bfloat16()
    w = (torch.randn((N, K), device="cuda", generator=g) * K ** -0.5).bfloat16()
    corr = torch.randn((E,), device="cuda", generator=g) * 0.02 if mode == "all" else None
    assert ops.moe_router_available(h, w)
    logits = torch.full((T, N), float("nan"), dtype=torch.float32, device="cuda")
    ids, weights = torch.full((T, top), -1, dtype=torch.int32, device="cuda"), torch.full((T, top), float("nan"), device="cuda")
    ops.moe_router(h, w, E, logits, ids, weights, mode, 1.5, corr)
    size = h.double().abs() @ w.double().abs().T
    # a rounding of a running sum, at most `size`, for every 32 columns and the eight sums that are joined (and the truncation inside
    # a step: counted as another)
    assert ((logits.double() - h.double() @ w.double().T).abs() <= size * (2 * (K / 32 + 1) + 8) * 2.0 ** -24).all()
    want_ids, want = torch.empty_like(ids), torch.empty_like(weights)
    ops.moe_route(logits, E, top, want_ids, want, mode, 1.5, corr)
    assert torch.equal(ids, want_ids) and torch.allclose(weights, want, rtol=1e-6, atol=0)


@pytest.mark.parametrize("mode", ["chosen", "all", "sigmoid", "corrected"])
@pytest.mark.parametrize("E,top", [(1, 1), (2, 2), (63, 5), (64, 8), (65, 8), (130, 3)])        # an output a lane, and more than a wave has
def test_routing_of_ties_and_of_what_is_no_number(E, top, mode):
    """Of equal logits the first is chosen (zeros of either sign are equal), infinities are logits like others, and what is no number
    is not chosen: where nothing else is left the place is given to no expert."""
    from serve_amd import ops
    inf, nan = float("inf"), float("nan")
    g = torch.Generator().manual_seed(E)
    rows = [torch.zeros(E), torch.randint(-2, 3, (E,), generator=g).float(), torch.randint(0, 2, (E,), generator=g).float() * -0.0,
            torch.full((E,), -inf), torch.where(torch.rand(E, generator=g) < 0.9, -inf, 1.0), torch.full((E,), -1e4)]
    ends = torch.randn(E, generator=g)
    ends[0] = ends[-1] = 9.0                                             # first and last equal, above the others
    rows.append(ends)
    if mode != "corrected":                                              # (there a share of NaN makes all of them NaN)
        rows += [torch.full((E,), nan), torch.where(torch.arange(E) % 7 == 3, 2.0, nan), torch.where(torch.arange(E) == E // 2, nan, 1.0)]
    z = torch.stack(rows).cuda()
    T = z.shape[0]
    corr = torch.randint(0, 3, (E,), generator=g).float() / 4 if mode == "corrected" else None
    over = "all" if mode == "corrected" else mode
    ids, w = torch.full((T, top), -1, dtype=torch.int32, device="cuda"), torch.zeros((T, top), device="cuda")
    ops.moe_route(z, E, top, ids, w, over, 1.5, None if corr is None else corr.cuda())
    ids, w = ids.cpu(), w.cpu().double()
    for t, row in enumerate(z.double().cpu()):
        numbers = [e for e in range(E) if row[e] == row[e]]
        if corr is not None:
            shares = torch.softmax(row, 0)
            if not torch.isfinite(shares).all():
                assert ((ids[t] >= 0) & (ids[t] < E)).all()             # stays within the table
                continue
            score = (torch.softmax(row.float(), 0) + corr).tolist()
            chosen = ids[t].tolist()
            assert len(set(chosen)) == top
            # (shares are rounded: scores as near as that are in either order, equal logits with equal corrections in theirs)
            left = min((score[e] for e in chosen))
            assert all(score[e] <= left + 1e-6 for e in range(E) if e not in chosen)
            for a, b in zip(chosen, chosen[1:]):
                assert score[a] >= score[b] - 1e-6 and (row[a] != row[b] or corr[a] != corr[b] or a < b)
            want = shares[ids[t].long()]
            assert torch.allclose(w[t], 1.5 * want / (want.sum() + 1e-20), rtol=1e-5, atol=1e-7)
            continue
        order = sorted(numbers, key=lambda e: (-row[e].item(), e))[:top]
        assert ids[t, : len(order)].tolist() == order
        assert ((ids[t, len(order):] < 0) | (ids[t, len(order):] >= E)).all()
        value = torch.cat([row[order], torch.full((top - len(order),), -inf, dtype=torch.float64)])
        if mode == "sigmoid":
            want = torch.sigmoid(value) * 1.5
        else:
            want = torch.softmax(value, 0) * 1.5                         # (of the chosen: the sum over all cancels)
            if mode == "all" and not torch.isfinite(row).all() and torch.isnan(row).any():
                want = torch.full_like(want, nan)                        # (the sum over all is none)
        assert torch.allclose(w[t], want, rtol=1e-5, atol=1e-7, equal_nan=True), (t, w[t], want)


@pytest.mark.parametrize("T,d,E,fused", [(63, 2048, 8, False), (64, 2048, 8, True), (64, 4096, 8, True), (64, 3072, 8, False), (95, 1024, 32, False),
                                         (96, 1024, 32, True), (64, 2048, 32, True), (256, 1024, 63, True), (255, 1024, 64, False),
                                         (300, 1088, 64, False), (300, 256, 65, False), (4096, 64, 8, True), (4097, 64, 8, False)])
def test_when_the_router_takes_product_and_routing_together(monkeypatch, T, d, E, fused):
    """Both ways of the rule, at its edges: the same feed-forward."""
    from serve_amd import ops
    from serve_amd.parts.base import Runtime
    from serve_amd.registry import get_part
    part = get_part("feed_forward", "routed_experts")(hidden_size=d, experts=E, top=2, expert_size=64, shared_size=64)
    g = torch.Generator("cuda").manual_seed(T + d)
    part.load({r.name: (torch.randn(tuple(r.shape), device="cuda", generator=g) * 0.05).bfloat16() for r in part.param_requests()},
              Runtime(torch.device("cuda:0"), torch.bfloat16, max_context=64))
    h = torch.randn((T, d), device="cuda", generator=g).bfloat16()
    calls = []
    router = ops.moe_router
    monkeypatch.setattr(ops, "moe_router", lambda *a: (calls.append(1), router(*a)))
    y = part.forward(h, None)
    assert bool(calls) == fused
    monkeypatch.setattr(ops, "moe_router_pays", lambda *a: not fused)
    want = part.forward(h, None)
    assert len(calls) == 1
    # The logits are float32 sums in another order, so the weights of the rows differ by float32 roundings and the bf16 rows not at
    # all; a token whose second and third logits are as near as that may choose another expert
    same = ((y - want).norm(dim=1) <= 1e-4 * want.norm(dim=1))
    assert same.float().mean() > 0.995


@pytest.mark.parametrize("K", [8, 264, 1000, 2048, 2056, 4104])     # parts of steps, of a wave's share and of what is loaded at once
def test_router_logits_of_numbers_without_bounds(K):
    """An infinity in a row of the router's matrix makes that row's logits infinite, and no NaN comes of columns that were read and
    do not count; infinities and NaN in a token stay with the token."""
    from serve_amd import ops
    g = torch.Generator("cuda").manual_seed(K)
    h = torch.randn((40, K), device="cuda", generator=g).bfloat16()
    w = (torch.randn((33, K), device="cuda", generator=g) * K ** -0.5).bfloat16()
    inf = float("inf")
    h[h == 0] = 1
    for n, k in ((0, K - 1), (3, K // 2), (5, 0), (9, K - 8), (17, (3 * K) // 4), (32, K - 1)):
        w[n, k] = inf if n % 2 else -inf
    h[11, K - 1], h[12, 0], h[30, K // 2] = inf, -inf, float("nan")
    w[w == 0] = 1e-3
    logits = torch.zeros((40, 33), dtype=torch.float32, device="cuda")
    ids, weights = torch.zeros((40, 2), dtype=torch.int32, device="cuda"), torch.zeros((40, 2), device="cuda")
    ops.moe_router(h, w, 32, logits, ids, weights)
    want = (h.double().cpu()[:, None] * w.double().cpu()[None]).sum(-1)        # (a product and a sum of its own for each: no library)
    got = logits.double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.isinf(want).sum() > 100
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
    ok = torch.isfinite(want)
    size = (h.double().cpu()[:, None] * w.double().cpu()[None]).abs().sum(-1)
    assert torch.isfinite(got[ok]).all() and ((got - want).abs() <= size * (2 * (K / 32 + 1) + 8) * 2.0 ** -24)[ok].all()   # (as above)


# (256 compute units)  both sides of each line of the rule: the smallest number of rows, half of the chip, two rows an expert, a
# second round of workgroups that is nearly empty
@pytest.mark.parametrize("T,top,E,d,F,tiles", [(16, 4, 32, 128, 256, False), (17, 4, 32, 128, 256, True), (65, 1, 32, 64, 256, True),
                                               (40, 4, 32, 192, 256, True), (256, 4, 32, 128, 256, True), (159, 1, 8, 64, 512, False),
                                               (160, 1, 8, 64, 512, True), (127, 1, 64, 64, 128, False), (128, 1, 64, 64, 128, True),
                                               (119, 2, 36, 64, 512, False), (121, 2, 36, 64, 512, True), (1024, 1, 4, 64, 192, False)])
@pytest.mark.parametrize("identity", [0, 3])
def test_experts_of_65_to_1024_rows(T, top, E, d, F, tiles, identity):
    """Which kernels a step of few rows takes, and what they give: experts with many rows, with one and with none, and identity
    outputs, whose rows are left alone."""
    from serve_amd import ops
    assert ops.moe_wide_pays(T * top, E, F) == tiles
    gc = torch.Generator("cuda").manual_seed(T + E + identity)
    # (the last expert without rows, the one before with one, the first with more than its share)
    order = torch.rand((T, E + identity), device="cuda", generator=gc)
    order[:, 0] += 0.3
    order[:, E - 2: E] = -1
    order[0, E - 2] = 2
    ids = order.topk(top, -1).indices.int().contiguous()
    h = torch.randn((T, d), device="cuda", generator=gc).bfloat16()
    wgu = (torch.randn((2, E, F, d), device="cuda", generator=gc) * d ** -0.5).bfloat16()
    wd = (torch.randn((E, d, F), device="cuda", generator=gc) * F ** -0.5).bfloat16()
    assert ops.moe_wide_available(h, wgu[0], wgu[1], wd)
    yk = torch.full((T * top, d), float("nan"), dtype=torch.float32, device="cuda")
    ops.moe_experts(h, ids, wgu[0], wgu[1], wd, yk, outputs=E + identity)
    flat = ids.view(-1)
    assert torch.isnan(yk[flat >= E]).all() and not (flat == E - 1).any() and (flat == E - 2).sum() == 1
    for e in range(E):
        r = (flat == e).nonzero()[:, 0]
        x = h[r // top].double()
        z = x @ wgu[0, e].double().T
        act = z * torch.sigmoid(z) * (x @ wgu[1, e].double().T)
        # (as below: the gated values are rounded to bf16's eight bits)
        bound = 1.1 * 2.0 ** -8 * (act.abs() @ wd[e].double().abs().T)
        assert torch.isfinite(yk[r]).all() and ((yk[r].double() - act @ wd[e].double().T).abs() <= bound).all(), e


# (256 compute units)  128 weight rows a workgroup in both products; 256 in the first, in both, and in the second, over one stage and more
@pytest.mark.parametrize("d,F,E", [(64, 64, 14), (128, 2048, 14), (1152, 3264, 15), (3392, 192, 14)])
def test_experts_products_at_the_edges_of_tiles(d, F, E):
    """Experts with as many rows as a tile of every size takes and with one more, two and three tiles of equal size, none; widths
    that are no whole share of a workgroup."""
    from serve_amd import ops
    counts = ([1, 32, 33, 64, 65, 128, 129, 160, 161, 192, 193, 256, 0, 257, 545] * 2)[:E]
    T = sum(counts)
    g = torch.Generator().manual_seed(d + F)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)].int()[:, None].cuda()
    gc = torch.Generator("cuda").manual_seed(d + F)
    h = torch.randn((T, d), device="cuda", generator=gc).bfloat16()
    wgu = (torch.randn((2, E, F, d), device="cuda", generator=gc) * d ** -0.5).bfloat16()
    wd = (torch.randn((E, d, F), device="cuda", generator=gc) * F ** -0.5).bfloat16()
    w = torch.rand((T, 1), device="cuda", generator=gc) + 0.5
    assert T > ops.MOE_WIDE_MIN_ROWS and ops.moe_wide_available(h, wgu[0], wgu[1], wd)
    for weights in (None, w):
        yk = torch.full((T, d), float("nan"), dtype=torch.float32, device="cuda")
        ops.moe_experts(h, ids, wgu[0], wgu[1], wd, yk, weights=weights, weight_inputs=weights is not None)
        for e in range(E):
            t = (ids[:, 0] == e).nonzero()[:, 0]
            x = h[t].double() * (1.0 if weights is None else weights[t].double())
            z = x @ wgu[0, e].double().T
            act = z * torch.sigmoid(z) * (x @ wgu[1, e].double().T)
            # the gated values are rounded to bf16's eight bits, by 2^-8 of each at most; the rest is float32 (a tenth of that is far more)
            bound = 1.1 * 2.0 ** -8 * (act.abs() @ wd[e].double().abs().T)
            assert torch.isfinite(yk[t]).all() and ((yk[t].double() - act @ wd[e].double().T).abs() <= bound).all(), (e, counts[e])


@pytest.mark.parametrize("rows,E,F,tile", [(8000, 32, 1024, 192), (7360, 32, 1024, 256), (7361, 32, 1024, 192), (9600, 32, 1024, 256),
                                           (5640, 24, 1024, 256), (6600, 24, 1024, 192), (3760, 16, 1536, 256), (4400, 16, 1536, 192),
                                           (16000, 64, 1536, 256), (17600, 64, 1536, 192), (1400, 8, 1024, 128)])
def test_the_rows_of_experts_tiles(rows, E, F, tile):
    """(256 compute units)  192 rows near 256 an expert, where second tiles have no room in the last round of workgroups."""
    from ctypes import c_int

    from serve_amd.csrc.build import load_library
    assert load_library("gemm_experts").sa_expert_tile_rows(c_int(rows), c_int(E), c_int(F)) == tile


def test_experts_products_with_tiles_of_192_rows():
    """Experts with as many rows as one, two and three of these tiles take, with one more, with few and with none."""
    from ctypes import c_int

    from serve_amd import ops
    from serve_amd.csrc.build import load_library
    d, F, E = 64, 512, 32
    counts = [192, 193, 385, 0, 576, 577, 1, 17] * 4
    T = sum(counts)
    assert load_library("gemm_experts").sa_expert_tile_rows(c_int(T), c_int(E), c_int(F)) == 192
    g = torch.Generator().manual_seed(T)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)].int()[:, None].cuda()
    gc = torch.Generator("cuda").manual_seed(T)
    h = torch.randn((T, d), device="cuda", generator=gc).bfloat16()
    wgu = (torch.randn((2, E, F, d), device="cuda", generator=gc) * d ** -0.5).bfloat16()
    wd = (torch.randn((E, d, F), device="cuda", generator=gc) * F ** -0.5).bfloat16()
    assert ops.moe_wide_pays(T, E, F) and ops.moe_wide_available(h, wgu[0], wgu[1], wd)
    yk = torch.full((T, d), float("nan"), dtype=torch.float32, device="cuda")
    ops.moe_experts(h, ids, wgu[0], wgu[1], wd, yk)
    for e in range(E):
        t = (ids[:, 0] == e).nonzero()[:, 0]
        x = h[t].double()
        z = x @ wgu[0, e].double().T
        act = z * torch.sigmoid(z) * (x @ wgu[1, e].double().T)
        bound = 1.1 * 2.0 ** -8 * (act.abs() @ wd[e].double().abs().T)       # (as above)
        assert torch.isfinite(yk[t]).all() and ((yk[t].double() - act @ wd[e].double().T).abs() <= bound).all(), (e, counts[e])


# tiles of 16 rows and more, one and several of them; fewer weight rows than a workgroup takes and no whole share; ahead and behind
@pytest.mark.parametrize("gate,limit,shared_limit", [("silu", 0.0, 0.0), ("clamped_swish", 0.8, 1.7)])
@pytest.mark.parametrize("T,d,S", [(65, 64, 64), (96, 192, 320), (129, 128, 192), (257, 64, 2048), (640, 320, 192), (641, 64, 64), (1153, 192, 576)])
def test_a_shared_expert_in_the_experts_launches(T, d, S, gate, limit, shared_limit):
    from serve_amd import ops
    E, F, top = 64, 128, 2
    g = torch.Generator("cuda").manual_seed(T + d + S)
    h = torch.randn((T, d), device="cuda", generator=g).bfloat16()
    wgu = (torch.randn((2, E, F, d), device="cuda", generator=g) * d ** -0.5).bfloat16()
    wd = (torch.randn((E, d, F), device="cuda", generator=g) * F ** -0.5).bfloat16()
    sgu = (torch.randn((2 * S, d), device="cuda", generator=g) * d ** -0.5).bfloat16()
    sd = (torch.randn((d, S), device="cuda", generator=g) * S ** -0.5).bfloat16()
    ids = torch.stack([torch.randperm(E, device="cuda", generator=g)[:top] for _ in range(T)]).int().contiguous()
    assert ops.moe_wide_pays(T * top, E, F) and ops.moe_shared_available(h, sgu, sd)
    alone, both = (torch.full((T * top, d), float("nan"), device="cuda") for _ in range(2))
    ops.moe_experts(h, ids, wgu[0], wgu[1], wd, alone, gate=gate, limit=limit)
    shared = ops.SharedExpert(sgu, sd, shared_limit)
    ops.moe_experts(h, ids, wgu[0], wgu[1], wd, both, gate=gate, limit=limit, shared=shared)
    assert torch.equal(alone, both), "the experts' own rows have changed"
    z, u = h.double() @ sgu[:S].double().T, h.double() @ sgu[S:].double().T
    if gate == "silu":
        act = z * torch.sigmoid(z) * u
    else:
        z, u = z.clamp(max=shared_limit), u.clamp(-shared_limit, shared_limit)
        act = z * torch.sigmoid(1.702 * z) * (u + 1.0)
    want = act @ sd.double().T
    # the gated values and the result are rounded to bf16's eight bits; the rest is float32
    bound = 1.1 * 2.0 ** -8 * (act.abs() @ sd.double().abs().T + want.abs())
    assert shared.out.shape == (T, d) and ((shared.out.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("T,d,S", [(65, 64, 64), (100, 320, 128), (129, 128, 64), (700, 64, 192)])
def test_a_shared_expert_in_the_experts_launches_stays_in_32_bits_behind_its_gate(T, d, S):
    """One column of the last matrix: a result is one product of two bf16 numbers, which has more bits than bf16."""
    from serve_amd import ops
    E, F, top = 64, 128, 2
    g = torch.Generator("cuda").manual_seed(T + d + S)
    h = torch.randn((T, d), device="cuda", generator=g).bfloat16()
    wgu, wd = torch.zeros((2, E, F, d), device="cuda").bfloat16(), torch.zeros((E, d, F), device="cuda").bfloat16()
    sgu = (torch.randn((2 * S, d), device="cuda", generator=g) * d ** -0.5).bfloat16()
    sd = torch.zeros((d, S), device="cuda").bfloat16()
    sd[:, S - 3] = torch.randn((d,), device="cuda", generator=g).bfloat16()
    sd[0, S - 3] = 1.0
    ids = torch.stack([torch.randperm(E, device="cuda", generator=g)[:top] for _ in range(T)]).int().contiguous()
    shared = ops.SharedExpert(sgu, sd)
    ops.moe_experts(h, ids, wgu[0], wgu[1], wd, torch.empty((T * top, d), device="cuda"), shared=shared)
    act = shared.out[:, 0].float()
    assert torch.equal(act, act.bfloat16().float()) and (act != 0).float().mean() > 0.9
    assert torch.equal(shared.out.float(), act[:, None] * sd[:, S - 3].float())


def _gated(z, u, gate, limit):
    if gate == "silu":
        return z * torch.sigmoid(z) * u
    if gate == "gelu_tanh":
        return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3))) * u
    z, u = z.clamp(max=limit), u.clamp(-limit, limit)
    return z * torch.sigmoid(1.702 * z) * (u + 1.0)


# (256 compute units) 256 weight rows a workgroup in both products of the experts, the last ones ragged; ahead and behind
@pytest.mark.parametrize("gate", ["silu", "gelu_tanh", "clamped_swish"])
@pytest.mark.parametrize("weight_inputs", [False, True])
@pytest.mark.parametrize("T,S", [(129, 64), (200, 448), (640, 192), (641, 192), (1030, 320)])
def test_a_shared_expert_beside_experts_of_wide_columns(T, S, weight_inputs, gate):
    """... which takes no part in the weights on the experts' inputs and has a limit of its own."""
    from serve_amd import ops
    E, F, d, top, limit, shared_limit = 64, 320, 704, 2, 0.8, 1.7
    g = torch.Generator("cuda").manual_seed(T + S)
    h = torch.randn((T, d), device="cuda", generator=g).bfloat16()
    wgu = (torch.randn((2, E, F, d), device="cuda", generator=g) * d ** -0.5).bfloat16()
    wd = (torch.randn((E, d, F), device="cuda", generator=g) * F ** -0.5).bfloat16()
    sgu = (torch.randn((2 * S, d), device="cuda", generator=g) * d ** -0.5).bfloat16()
    sd = (torch.randn((d, S), device="cuda", generator=g) * S ** -0.5).bfloat16()
    ids = torch.rand((T, E), device="cuda", generator=g).topk(top, dim=1).indices.int().contiguous()
    weights = 0.25 + torch.rand((T, top), device="cuda", generator=g)
    assert ops.moe_wide_pays(T * top, E, F) and 4 * E * -(-F // 128) >= 3 * ops.compute_units() and 4 * E * -(-d // 256) >= 3 * ops.compute_units()
    alone, both = (torch.full((T * top, d), float("nan"), device="cuda") for _ in range(2))
    more = dict(weights=weights, gate=gate, limit=limit, weight_inputs=weight_inputs)
    ops.moe_experts(h, ids, wgu[0], wgu[1], wd, alone, **more)
    shared = ops.SharedExpert(sgu, sd, shared_limit)
    ops.moe_experts(h, ids, wgu[0], wgu[1], wd, both, shared=shared, **more)
    assert torch.equal(alone, both), "the experts' own rows have changed"
    x = h.double()
    act = _gated(x @ sgu[:S].double().T, x @ sgu[S:].double().T, gate, shared_limit)
    want = act @ sd.double().T
    # the gated values are rounded to eight bits, by at most 2^-8 of each; the rest is float32
    assert ((shared.out.double() - want).abs() <= 1.1 * 2.0 ** -8 * (act.abs() @ sd.double().abs().T)).all()
    w_in = weights.double() if weight_inputs else torch.ones_like(weights, dtype=torch.float64)
    rows = both.view(T, top, d).double()
    for e in (0, 31, E - 1):
        t, k = (ids == e).nonzero(as_tuple=True)
        xe = x[t] * w_in[t, k][:, None]
        act = _gated(xe @ wgu[0, e].double().T, xe @ wgu[1, e].double().T, gate, limit)
        assert ((rows[t, k] - act @ wd[e].double().T).abs() <= 1.1 * 2.0 ** -8 * (act.abs() @ wd[e].double().abs().T)).all(), e


# T, d, E, F, top, S: both sides of each line of the rule
@pytest.mark.parametrize("T,d,E,F,top,S,inside", [
    (16, 128, 64, 128, 8, 64, False), (17, 128, 64, 128, 8, 64, True),                  # the routing in a call of its own
    (128, 128, 64, 256, 4, 128, True), (128, 128, 64, 320, 4, 128, False), (129, 128, 64, 320, 4, 128, True),
    (300, 64, 64, 128, 4, 2048, True), (300, 64, 64, 128, 4, 2112, False),
    (300, 1088, 64, 128, 4, 2176, True), (300, 1088, 64, 128, 4, 2240, False), (128, 1088, 64, 128, 4, 2176, False),
    (640, 1088, 64, 128, 2, 2176, True), (641, 1088, 64, 128, 2, 2176, False), (128, 2112, 64, 64, 4, 2112, True),
    (2145, 2048, 8, 64, 1, 2048, True), (2146, 2048, 8, 64, 1, 2048, False)])
@pytest.mark.parametrize("gate,limit,shared_limit", [("silu", 0.0, None), ("clamped_swish", 0.8, 1.7)])
def test_when_the_shared_expert_goes_with_the_experts(monkeypatch, T, d, E, F, top, S, inside, gate, limit, shared_limit):
    """The whole feed-forward with its shared expert's gate: which way it takes, its result, and no further from 64 bits than with the
    shared expert in products of its own."""
    from serve_amd import ops
    from serve_amd.parts.base import Runtime
    from serve_amd.registry import get_part
    part = get_part("feed_forward", "routed_experts")(hidden_size=d, experts=E, top=top, expert_size=F, shared_size=S, activation=gate,
                                                      limit=limit, shared_limit=shared_limit)
    g = torch.Generator("cuda").manual_seed(T + d + S)
    tensors = {r.name: (torch.randn(tuple(r.shape), device="cuda", generator=g) * r.shape[1] ** -0.5).bfloat16() for r in part.param_requests()}
    part.load(tensors, Runtime(torch.device("cuda:0"), torch.bfloat16, max_context=64))
    h = torch.randn((T, d), device="cuda", generator=g).bfloat16()
    calls, experts = [], ops.moe_experts

    def spy(h, ids, *args, **more):
        out = experts(h, ids, *args, **more)
        calls.append((more.get("shared"), ids, more.get("weights", args[5] if len(args) > 5 else None)))
        return out
    monkeypatch.setattr(ops, "moe_experts", spy)
    y = part.forward(h, None)
    shared, ids, weights = calls[0]
    assert (shared is not None) == inside
    w = {n: t.double() for n, t in tensors.items()}
    x = h.double()
    act = _gated(x @ w["shared.gate"].T, x @ w["shared.up"].T, gate, limit if shared_limit is None else shared_limit)
    share = torch.sigmoid(x @ w["shared.sg"].T)
    want, size = share * (act @ w["shared.down"].T), share * (act.abs() @ w["shared.down"].abs().T)
    for e in range(E):
        t, k = (ids == e).nonzero(as_tuple=True)
        act = _gated(x[t] @ w[f"e{e}.gate"].T, x[t] @ w[f"e{e}.up"].T, gate, limit)
        want.index_add_(0, t, weights[t, k].double()[:, None] * (act @ w[f"e{e}.down"].T))
        size.index_add_(0, t, weights[t, k].double()[:, None] * (act.abs() @ w[f"e{e}.down"].abs().T))
    off = (y.double() - want).abs()
    # inside, the gated values are rounded to eight bits, by at most 2^-8 of each, and the rest is float32; in products of its own the
    # shared expert's gates, ups and rows may be rounded too (0.003 of the result, and four times that)
    if inside:
        assert (off <= 1.1 * 2.0 ** -8 * size + 1e-5).all()
    assert off.norm() <= 0.012 * want.norm()
    monkeypatch.setattr(ops, "moe_shared_inside", lambda *a: False)
    alone = part.forward(h, None)
    if inside:
        assert off.norm() <= 1.02 * (alone.double() - want).norm()
    else:
        assert torch.equal(alone, y)


@pytest.mark.parametrize("gate,limit", [("silu", 0.0), ("clamped_swish", 0.8)])
@pytest.mark.parametrize("T,d,F,E,top", [(700, 128, 192, 5, 2), (300, 64, 64, 9, 4), (2048, 256, 128, 6, 1)])
def test_experts_of_many_rows_with_both_operands_through_lds(T, d, F, E, top, gate, limit):
    """More than 1,024 (token, k) rows in bf16 with widths that are multiples of 64 and the gates' and ups' matrices in
    one tensor: tiles of up to 256 grouped rows; experts with no row, with a few, and with several tiles of rows."""
    from serve_amd import ops
    torch.manual_seed(T + E)
    h = torch.randn(T, d, device="cuda").bfloat16()
    wgu = (torch.randn(2, E, F, d, device="cuda") * 0.1).bfloat16()
    wd = (torch.randn(E, d, F, device="cuda") * 0.1).bfloat16()
    assert T * top > ops.MOE_WIDE_MIN_ROWS and ops.moe_wide_available(h, wgu[0], wgu[1], wd)
    ids = torch.stack([torch.randperm(E, device="cuda")[:top] for _ in range(T)]).int().contiguous()
    if top < E:
        ids[ids == E - 1] = 0 if top == 1 else ids[ids == E - 1]          # (top 1: the last expert gets no row at all)
    ids[: T // 2, 0] = ids[0, 0]                                          # one expert with many tiles of rows
    if top > 1:
        ids[: T // 2, 1:] = ids[0, 1:]
    yk = torch.full((T * top, d), float("nan"), dtype=torch.float32, device="cuda")
    ops.moe_experts(h, ids, wgu[0], wgu[1], wd, yk, gate=gate, limit=limit)
    assert torch.isfinite(yk).all(), "a row was not written"
    # the same through the kernels for few rows, slice by slice
    ref = torch.empty_like(yk)
    for t0 in range(0, T, 200):
        n = min(200, T - t0)
        ops.moe_experts(h[t0: t0 + n].contiguous(), ids[t0: t0 + n].contiguous(), wgu[0], wgu[1], wd,
                        ref[t0 * top: (t0 + n) * top], gate=gate, limit=limit)
    assert torch.allclose(yk, ref, atol=2e-2, rtol=2e-2), f"max diff {(yk - ref).abs().max().item():.3g}"
    hd = h.double().cpu()
    for t in (0, 1, T // 2 - 1, T // 2, T - 1):
        for k in range(top):
            e = int(ids[t, k])
            g, u = hd[t] @ wgu[0, e].double().cpu().t(), hd[t] @ wgu[1, e].double().cpu().t()
            a = (tp.clamped_swish_gate(g, u, limit) if gate == "clamped_swish" else g * torch.sigmoid(g) * u).bfloat16().double()
            want = a @ wd[e].double().cpu().t()
            assert torch.allclose(yk[t * top + k].double().cpu(), want, atol=2e-2, rtol=1e-2)
