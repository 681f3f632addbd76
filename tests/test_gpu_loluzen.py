"""Loluzen on the GPU against the plain implementation (tests/plain/loluzen_plain.py): every mechanism
alone, whole prompts against token-by-token decoding, portions down to two tokens, batches of unequal
requests, pages and slots used again, far keys and page borders, first tokens, long decoding, sizes
nobody tuned the kernels for, and greedy generation through the scheduler and the command line."""
import functools
import json
import math
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import loluzen_util as lu
import util
from plain import loluzen_plain as plain

pytestmark = pytest.mark.gpu

DTYPES = ["float32", "bfloat16"]
WHOLE = ["mixed", "wide", "odd", "plain"]


@functools.lru_cache(maxsize=None)
def model(name: str, seed: int = 0, peaky: float = 1.0):
    raw = lu.CONFIGS[name]
    w = lu.make_weights(raw, seed, peaky)
    folder = os.path.join(util._TMP.name, f"loluzen_{name}_{seed}_{peaky}")
    return lu.write_folder(raw, w, folder), raw, w


@functools.lru_cache(maxsize=512)
def _plain(name, seed, peaky, tokens, scale):
    _, raw, w = model(name, seed, peaky)
    if scale is None:
        return plain.forward(raw, w, list(tokens))
    return plain.forward(raw, w, list(tokens), rnd=lambda t: plain.bf16_round(t * scale) / scale)


def expected(name, tokens, seed=0, peaky=1.0) -> util.Expected:
    """Exact logits, and three realizations of the logits of a model that rounds its activations to bfloat16."""
    tokens = tuple(tokens)
    return util.Expected(_plain(name, seed, peaky, tokens, None),
                         [_plain(name, seed, peaky, tokens, s) for s in util.REALIZATION_SCALES])


def engine(name, dtype, seed=0, peaky=1.0, **kw):
    from tuff_amd.engine.engine import Engine
    folder, _, _ = model(name, seed, peaky)
    kw.setdefault("page_size", 16)
    kw.setdefault("max_tokens", 1024)
    kw.setdefault("max_requests", 4)
    return Engine.from_folder(folder, dtype=dtype, poison_cache=True, **kw)


def requests(name, lengths, seed=0):
    V = lu.CONFIGS[name]["vocab"]
    return {f"r{i}": util.rand_tokens(n, V, seed * 100 + i) for i, n in enumerate(lengths)}


def compare(name, dtype, got, reqs, seed=0, peaky=1.0, what=""):
    """float32: every request against the exact logits.  bfloat16: the rows of all requests together against the
    rounding model's error (a request of one or two rows alone scatters too much for a bound on a mean)."""
    exp = {rid: expected(name, toks, seed, peaky) for rid, toks in reqs.items()}
    if dtype == "float32":
        for rid in reqs:
            util.assert_close_f32(got[rid], exp[rid], f"{what} {name} {rid}")
        return
    rids = list(reqs)
    for r in rids:
        assert torch.isfinite(got[r]).all(), f"{what} {name} {r}: non-finite logits"
    if sum(len(reqs[r]) for r in rids) < 8:
        return
    want = util.Expected(torch.cat([exp[r].want for r in rids]),
                         [torch.cat([exp[r].rounded[i] for r in rids]) for i in range(len(util.REALIZATION_SCALES))])
    util.assert_close_bf16(torch.cat([got[r] for r in rids]), want, f"{what} {name} bfloat16")


def check(name, dtype, plan, reqs, seed=0, peaky=1.0, **kw):
    eng = engine(name, dtype, seed, peaky, **kw)
    got = util.run_plan(eng, plan)
    eng.manager.check()
    assert not eng.manager.live()
    compare(name, dtype, got, reqs, seed, peaky)
    return eng, got


def all_single(reqs):
    return util.plan_tail(reqs, tail=10 ** 6)


# ------------------------------------------------------------------------ mechanisms alone
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", [n for n in lu.CONFIGS if n.startswith("only_")])
def test_each_mechanism_alone(gpu, name, dtype):
    reqs = requests(name, [37, 1, 9])
    check(name, dtype, util.plan_whole(reqs), reqs)
    check(name, dtype, util.plan_chunks(reqs, sizes=(2, 5, 1, 3, 16, 2)), reqs)


# -------------------------------------------------------------- whole models under every plan
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", WHOLE)
def test_whole_prompts(gpu, name, dtype):
    reqs = requests(name, [90, 1, 2, 33])
    check(name, dtype, util.plan_whole(reqs), reqs)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", WHOLE)
def test_prompt_then_single_tokens_and_single_tokens_from_the_start(gpu, name, dtype):
    reqs = requests(name, [70, 40], seed=1)
    check(name, dtype, util.plan_tail(reqs, tail=32), reqs, seed=1)
    first = requests(name, [24], seed=2)        # the first tokens one by one: states start at zero, taps reach before the start
    check(name, dtype, all_single(first), first, seed=1)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", WHOLE)
def test_portions_of_changing_size(gpu, name, dtype):
    reqs = requests(name, [150, 61], seed=3)
    check(name, dtype, util.plan_chunks(reqs), reqs)
    small = {"r1": reqs["r1"]}                  # portions shorter than the convolutions' taps
    check(name, dtype, util.plan_chunks(small, sizes=(2, 2, 3, 2, 1, 2)), small)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", WHOLE)
def test_batches_of_unequal_requests_with_pages_and_slots_used_again(gpu, name, dtype):
    reqs = requests(name, [5, 77, 130, 2, 40, 64, 19, 95, 33], seed=4)
    plan = util.plan_mixed(reqs, seed=4, max_live=3)
    peak = util.live_tokens_peak(plan)
    eng, got = check(name, dtype, plan, reqs, max_tokens=peak, max_requests=3)
    assert eng.manager.groups[0].pool.allocations > eng.manager.groups[0].pool.num_pages       # pages came back and went out again
    # once more on the same engine: every page and slot has been used before, and holds NaN or another request's state
    again = util.run_plan(eng, plan)
    if dtype == "float32":
        for rid in reqs:
            assert torch.equal(again[rid], got[rid]), rid
    else:
        compare(name, dtype, again, reqs, what="second run")


@pytest.mark.parametrize("name", ["mixed", "wide", "odd"])
def test_float32_logits_do_not_depend_on_the_plan(gpu, name):
    """The same bits whether a prompt comes whole, in portions, token by token or beside other requests, with
    recorded steps or without."""
    reqs = requests(name, [83, 30, 47], seed=5)
    plans = [util.plan_whole(reqs), util.plan_chunks(reqs), all_single(reqs), util.plan_mixed(reqs, seed=1)]
    base = util.run_plan(engine(name, "float32"), plans[0])
    for i, plan in enumerate(plans[1:]):
        for graphs in (True, False):
            got = util.run_plan(engine(name, "float32", use_graphs=graphs), plan)
            for rid in reqs:
                assert torch.equal(got[rid], base[rid]), f"plan {i + 1}, graphs {graphs}, {rid}"


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding(gpu, dtype):
    reqs = requests("mixed", [330], seed=6)
    check("mixed", dtype, util.plan_tail(reqs, tail=325), reqs)


# --------------------------------------------------------------- far keys and page borders
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["only_attention", "only_attention_equal", "only_attention_bare", "only_pair", "only_pair_wide"])
def test_peaky_attention_far_keys_in_prompts_and_in_decoding(gpu, name, dtype):
    """W_q and W_k scaled up: a few keys hold the weight, anywhere in hundreds; a key lost, taken twice or read
    from a neighbour's page moves the logits."""
    reqs = requests(name, [420, 300], seed=8)
    check(name, dtype, util.plan_tail(reqs, tail=70), reqs, peaky=4.0)
    check(name, dtype, util.plan_chunks(reqs, sizes=(15, 1, 16, 17, 2, 31, 33, 64, 63, 65)), reqs, peaky=4.0)


def _mixed_heads(q, k, v, r1, r2, talk, scale):
    """The last query of q [n, H, dk] over k [n, G, dk], v [n, G, dv], float64 -> [H, dv]: a logarithmic distance penalty
    off the scaled scores, softmax, the heads' weights mixed by talk, each head on its own kv head's values."""
    n, H, G = q.shape[0], q.shape[1], k.shape[1]
    dist = torch.arange(n - 1, -1, -1, dtype=torch.float64)
    p = torch.stack([torch.softmax((k[:, h // (H // G)] @ q[-1, h]) * scale - r1[h] * torch.log1p(r2[h] * dist), 0) for h in range(H)])
    mixed = talk @ p
    return torch.stack([mixed[h] @ v[:, h // (H // G)] for h in range(H)])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dk, dv, H, G", [(16, 16, 4, 2), (64, 64, 8, 2), (24, 40, 3, 1), (128, 128, 2, 2), (80, 48, 4, 4),
                                          (64, 128, 6, 3), (256, 256, 2, 1), (32, 32, 12, 1), (40, 8, 1, 1)])
def test_attention_with_mixed_heads_one_key_stands_out(gpu, dk, dv, H, G, dtype):
    """The pair's attention mixer alone, its projections identities: one key, at the start, far back, at a page's border
    or the last, lines up with the last query so that it holds most of the weight against the distance penalty; the
    mixing matrix has negative and large entries.  The step's queries see it from a prompt's portion and from single
    tokens.  Pages are scattered and everything else in the pool is NaN."""
    from tuff_amd.cache.manager import CacheLayout, CacheManager
    from tuff_amd.cache.storage import CacheStorage
    from tuff_amd.engine.batch import StepEntry, build_context
    from tuff_amd.parts.attention import AttentionMixer
    from tuff_amd.parts.base import Runtime
    ps = 16
    gen = torch.Generator().manual_seed(dk + dv + H)
    width = H * dk + G * dk + G * dv
    names = {k: k for k in ("q", "k", "v", "o", "q.b", "k.b", "v.b", "r1", "r2", "talk")}
    mixer = AttentionMixer(width, H, G, dk, value_dim=dv, scale=0.4, names=names)
    eye = torch.eye(width)
    r1, r2 = 0.2 + torch.rand(H, generator=gen), 0.1 + 2.0 * torch.rand(H, generator=gen)
    talk = torch.randn(H, H, generator=gen)
    weights = {"q": eye[:H * dk], "k": eye[H * dk:H * dk + G * dk], "v": eye[H * dk + G * dk:], "o": torch.eye(H * dv),
               "q.b": torch.zeros(H * dk), "k.b": torch.zeros(G * dk), "v.b": torch.zeros(G * dv), "r1": r1, "r2": r2, "talk": talk}
    weights = {n: t.to(dtype).to(gpu) for n, t in weights.items()}
    mixer.bind(weights, Runtime(gpu, dtype))
    r1, r2, talk = (weights[n].double().cpu() for n in ("r1", "r2", "talk"))
    layout = CacheLayout.from_specs({0: mixer.cache_spec()})
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    for n, special in [(1, 0), (17, 0), (257, 15), (257, 16), (300, 255), (300, 256), (700, 3), (129, 128), (200, 136)]:
        mgr = CacheManager(layout, ps, 64, 2)
        store = CacheStorage(mgr, dtype, gpu, poison=True)
        mgr.admit("pad")
        mgr.extend("pad", 40)                               # the request's pages do not start at page 0
        mgr.admit("a")
        x = torch.randn(n, width, generator=gen) * 0.5
        qrows = x[:, :H * dk].view(n, H, dk)
        krows = x[:, H * dk:H * dk + G * dk].view(n, G, dk)
        for g in range(G):                                   # the special key lines up with the last query's heads
            krows[special, g] = qrows[n - 1, g * (H // G)] * (6.0 + 1.5 * math.log1p(n))
        x = x.to(dtype)
        xf = x.double()
        qf = xf[:, :H * dk].view(n, H, dk)
        kf = xf[:, H * dk:H * dk + G * dk].view(n, G, dk)
        vf = xf[:, H * dk + G * dk:].view(n, G, dv)
        tail = min(3, n - 1)
        steps = [list(range(0, n - tail))] + [[i] for i in range(n - tail, n)] if n > tail else [[0]]
        for rows in steps:
            if not rows:
                continue
            mgr.extend("a", len(rows))
            ctx = build_context([StepEntry("a", [0] * len(rows), [])], mgr, gpu, 10)
            res = torch.zeros(len(rows), H * dv, dtype=torch.float32, device=gpu)
            mixer.forward(x[rows].to(gpu).contiguous(), ctx, store.views[0], res)
            for at in {len(rows) - 1, len(rows) // 2}:       # the last query of the step, and one in a portion's middle
                i = rows[at]
                want = _mixed_heads(qf[:i + 1], kf[:i + 1], vf[:i + 1], r1, r2, talk, 0.4).reshape(-1)
                err = (res[at].double().cpu() - want).abs().max()
                assert err <= tol * max(1.0, float(want.abs().max())), (n, special, i, float(err))


def _paged_case(gpu, H, Hkv, hd, vd, reqs, opts, ps=16, seed=0):
    """Scattered pages of random bfloat16 keys and values for requests (tokens before the step, tokens of the step), queries,
    and the options' tensors; everything a kernel's launch takes."""
    gen = torch.Generator().manual_seed(seed)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)
    R, T = len(reqs), sum(n for _, n in reqs)
    longest = max(c + n for c, n in reqs)
    nblk = -(-longest // ps)
    P = R * nblk + 3
    table = torch.randperm(P, generator=gen)[:R * nblk].view(R, nblk).int().to(gpu)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=gpu)
    req_of, pos, info, t = [], [], [], 0
    for r, (c, n) in enumerate(reqs):
        info.append((t, n, c, 0)); req_of += [r] * n; pos += list(range(c, c + n)); t += n
    window, sinks, slopes, logd, talk, gate = opts
    case = dict(q=(rnd(T, H * hd) * 1.5).bfloat16().to(gpu), k=rnd(P, Hkv, ps, hd).bfloat16().to(gpu), v=rnd(P, Hkv, vd, ps).bfloat16().to(gpu),
                table=table, req_of=i32(req_of), pos=i32(pos), info=i32(info), longest=longest, T=T, window=window,
                sinks=(rnd(H) + 1).to(gpu) if sinks else None, slopes=(torch.rand(H, generator=gen) * 0.1).to(gpu) if slopes else None,
                logd=((torch.rand(H, generator=gen) + 0.2).to(gpu), (torch.rand(H, generator=gen) * 2 + 0.1).to(gpu)) if logd else None,
                talk=rnd(H, H).to(gpu) if talk else None, gates=rnd(T, H).to(gpu) if gate else None)
    return case


def _general(c, H, Hkv, hd, vd, ps=16):
    """The one-wave-a-head kernel (float32 weights; held to the plain functions by the float32 tests above), then the
    heads' mixing and gates: [T, H * vd] float32."""
    from tuff_amd.csrc import ops
    mixed = c["talk"] is not None
    o = torch.zeros((c["T"], H * Hkv * vd) if mixed else (c["T"], H * vd), dtype=torch.float32 if mixed else torch.bfloat16, device=c["q"].device)
    ops.attention_general(c["q"], c["k"], c["v"], o, block_table=c["table"], req_of_token=c["req_of"], positions=c["pos"], H=H, Hkv=Hkv,
                          hd=hd, page_size=ps, window=c["window"], scale=0.2, vd=vd, sinks=c["sinks"], slopes=c["slopes"],
                          log_distance=c["logd"], all_values=mixed)
    if not mixed and c["gates"] is None:
        return o.float()
    out = torch.zeros(c["T"], H * vd, dtype=o.dtype, device=o.device)
    ops.head_mix_gate(o, out, H=H, Hkv=Hkv, vd=vd, talk=c["talk"], gates=c["gates"])
    return out.float()


SHAPES = [(4, 2, 64, 64), (4, 4, 80, 48), (6, 3, 24, 40), (2, 1, 128, 128), (8, 2, 40, 16), (2, 2, 256, 64), (40, 2, 16, 8), (3, 3, 8, 256)]
# (window, sinks, slopes, logarithmic penalty, mixed heads, gates)
OPTIONS = [(0, 0, 0, 0, 0, 0), (48, 0, 0, 0, 0, 0), (0, 1, 0, 0, 0, 1), (300, 1, 0, 0, 0, 0), (0, 0, 1, 0, 0, 0), (0, 0, 0, 1, 0, 0),
           (0, 0, 0, 1, 1, 1), (100, 1, 0, 1, 1, 0)]


@pytest.mark.parametrize("H, Hkv, hd, vd", SHAPES)
def test_prompt_kernel_in_its_wide_form_against_the_general_kernel(gpu, H, Hkv, hd, vd):
    """Portions at the start, far into a request and across page and step borders, a single token among them; float32
    sums where the heads are mixed agree to float32's rounding: the weights keep their precision through the matrix cores."""
    from tuff_amd.csrc import ops
    reqs = [(0, 70), (130, 5), (300, 1), (17, 200)]
    for opts in OPTIONS:
        c = _paged_case(gpu, H, Hkv, hd, vd, reqs, opts, seed=H + hd)
        c["gates"] = None
        want = _general(c, H, Hkv, hd, vd)
        mixed = c["talk"] is not None
        o = torch.zeros((c["T"], H * Hkv * vd) if mixed else (c["T"], H * vd), dtype=torch.float32 if mixed else torch.bfloat16, device=gpu)
        blocks = torch.from_numpy(ops.query_blocks(np.array([n for _, n in reqs]), H // Hkv, 8, np.array([a + n for a, n in reqs]))).to(gpu)
        ops.attention_prefill_wide(c["q"], c["k"], c["v"], o, block_table=c["table"], blocks=blocks, req_info=c["info"], H=H, Hkv=Hkv, hd=hd,
                                   vd=vd, page_size=16, max_ctx_len=c["longest"], window=c["window"], scale=0.2, sinks=c["sinks"],
                                   slopes=c["slopes"], log_distance=c["logd"], all_values=mixed)
        if mixed:
            got = torch.zeros(c["T"], H * vd, dtype=torch.float32, device=gpu)
            ops.head_mix_gate(o, got, H=H, Hkv=Hkv, vd=vd, talk=c["talk"], gates=None)
        else:
            got = o.float()
        tol = 3e-5 if mixed else 0.01
        assert (got - want).abs().max() <= tol * max(1.0, float(want.abs().max())), opts


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("ps", [16, 48])
@pytest.mark.parametrize("H, Hkv, hd, vd", [(8, 8, 64, 64), (10, 5, 64, 24), (9, 9, 16, 32), (12, 3, 40, 64), (4, 4, 32, 32), (6, 6, 8, 8)])
def test_prompt_kernel_with_the_values_of_several_kv_heads_a_workgroup(gpu, H, Hkv, hd, vd, ps, many):
    """Heads of up to 64 channels and more than two kv heads: launches of few workgroups, which take two kv heads each, and of many,
    which take four, numbers of kv heads that fill those and that do not, every kind of penalty, page sizes that are and
    are not a power of two; to float32's rounding, as above."""
    from tuff_amd.csrc import ops
    reqs = [(i % 70, 1 + i % 9) for i in range(64)] if many else [(0, 70), (1090, 5), (300, 1), (17, 200)]
    for opts in [(0, 0, 0, 0, 1, 0), (0, 0, 1, 0, 1, 0), (0, 1, 0, 1, 1, 0), (0, 0, 1, 1, 1, 0), (100, 1, 0, 1, 1, 0)]:
        c = _paged_case(gpu, H, Hkv, hd, vd, reqs, opts, ps=ps, seed=H + hd)
        want = _general({**c, "gates": None}, H, Hkv, hd, vd, ps=ps)
        o = torch.zeros((c["T"], H * Hkv * vd), dtype=torch.float32, device=gpu)
        blocks = torch.from_numpy(ops.query_blocks(np.array([n for _, n in reqs]), H // Hkv, 8, np.array([a + n for a, n in reqs]))).to(gpu)
        ops.attention_prefill_wide(c["q"], c["k"], c["v"], o, block_table=c["table"], blocks=blocks, req_info=c["info"], H=H, Hkv=Hkv, hd=hd,
                                   vd=vd, page_size=ps, max_ctx_len=c["longest"], window=c["window"], scale=0.2, sinks=c["sinks"],
                                   slopes=c["slopes"], log_distance=c["logd"], all_values=True)
        got = torch.zeros(c["T"], H * vd, dtype=torch.float32, device=gpu)
        ops.head_mix_gate(o, got, H=H, Hkv=Hkv, vd=vd, talk=c["talk"], gates=None)
        assert (got - want).abs().max() <= 3e-5 * max(1.0, float(want.abs().max())), opts


@pytest.mark.parametrize("H, Hkv, hd, vd, ps", [(32, 8, 64, 64, 16), (8, 8, 64, 64, 48), (10, 5, 64, 24, 16), (6, 6, 16, 32, 32), (12, 3, 40, 64, 80),
                                                (10, 5, 32, 32, 16)])
def test_long_requests_of_mixed_heads_have_the_same_bits_alone_and_in_company(gpu, H, Hkv, hd, vd, ps):
    """A portion alone is a launch of few workgroups, which take two kv heads each; among many short requests the same portion goes
    through the kernel that takes four.  Whole blocks of 128 columns over more than 1,024 and 2,048 keys (the places of pages are worked
    out for 1,024 at a time), with windows that reach into the portion and beyond; beside the general kernel to float32's rounding.
    (Heads of at most 32 channels stay by themselves in the small launches, and where four would leave places empty.)"""
    from tuff_amd.csrc import ops
    long = [(1500, 200), (2040, 130), (0, 250)]
    reqs = [(5 + i % 40, 1) for i in range(40)] + long + [(i, 1) for i in range(24)]
    small = lambda blocks: blocks.shape[0] * Hkv * -(-Hkv // 2) <= 256
    for opts in [(0, 0, 0, 1, 1, 0), (100, 1, 0, 1, 1, 0), (1500, 0, 1, 0, 1, 0)]:
        c = _paged_case(gpu, H, Hkv, hd, vd, reqs, opts, ps=ps, seed=H + hd)
        want = _general({**c, "gates": None}, H, Hkv, hd, vd, ps=ps)

        def sums(first, which):
            n = np.array([m for _, m in which])
            ends = np.array([a + m for a, m in which])
            starts = np.concatenate([[0], np.cumsum(n)])
            T, at = int(n.sum()), sum(m for _, m in reqs[:first])
            info = torch.tensor([[int(s), m, a, 0] for s, (a, m) in zip(starts, which)], dtype=torch.int32, device=gpu)
            blocks = torch.from_numpy(ops.query_blocks(n, H // Hkv, 8, ends))
            assert small(blocks) == (len(which) == 1)
            o = torch.full((T, H * Hkv * vd), float("nan"), device=gpu)
            ops.attention_prefill_wide(c["q"][at:at + T], c["k"], c["v"], o, block_table=c["table"][first:first + len(which)], blocks=blocks.to(gpu),
                                       req_info=info, H=H, Hkv=Hkv, hd=hd, vd=vd, page_size=ps, max_ctx_len=int(ends.max()), window=c["window"],
                                       scale=0.2, sinks=c["sinks"], slopes=c["slopes"], log_distance=c["logd"], all_values=True)
            return o
        every = sums(0, reqs)
        for i, (_, m) in enumerate(long):
            at = 40 + sum(k for _, k in long[:i])
            assert torch.equal(sums(40 + i, [long[i]]), every[at:at + m]), (opts, i)
        got = torch.zeros(c["T"], H * vd, device=gpu)
        ops.head_mix_gate(every, got, H=H, Hkv=Hkv, vd=vd, talk=c["talk"], gates=None)
        assert (got - want).abs().max() <= 3e-5 * max(1.0, float(want.abs().max())), opts


@pytest.mark.parametrize("H, Hkv, hd, vd", SHAPES)
def test_single_token_kernels_with_float32_weights_against_the_general_kernel(gpu, H, Hkv, hd, vd):
    """Single tokens at the first position, on both sides of a part's 256 keys and far behind them."""
    from tuff_amd.csrc import ops
    reqs = [(n, 1) for n in (0, 5, 255, 256, 257, 700, 1023, 15)]
    for opts in OPTIONS:
        c = _paged_case(gpu, H, Hkv, hd, vd, reqs, opts, seed=H + vd)
        want = _general(c, H, Hkv, hd, vd)
        got = torch.zeros(c["T"], H * vd, dtype=torch.float32, device=gpu)
        ops.attention_decode_exact(c["q"], c["k"], c["v"], got, block_table=c["table"], req_of_token=c["req_of"], positions=c["pos"], H=H,
                                   Hkv=Hkv, hd=hd, vd=vd, page_size=16, max_ctx_len=c["longest"], window=c["window"], scale=0.2,
                                   sinks=c["sinks"], slopes=c["slopes"], log_distance=c["logd"], talk=c["talk"], gates=c["gates"])
        tol = 3e-5 if c["talk"] is not None else 0.01            # (the general kernel's own output is bfloat16 where heads are not mixed)
        assert (got - want).abs().max() <= tol * max(1.0, float(want.abs().max())), opts


def test_forget_scan_carries_its_state_across_any_cut(gpu):
    """The recurrence's kernel on its own, at key sizes on both sides of a wave's 64 lanes and value sizes of one and
    several blocks: a sequence in one call against the same sequence in portions of 1, 2 and more through the state, in
    a slot between slots of NaN, against the plain loop.  Gates near 0 and near 1 are among them."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(5)
    for H, D, Dv in [(2, 16, 16), (3, 40, 72), (1, 100, 130), (2, 200, 24), (1, 256, 8), (4, 48, 64), (1, 1, 1)]:
        n = 23
        x = torch.randn(n, 2 * H * D + H * Dv, generator=gen)
        x[:, H * D:2 * H * D] *= 6.0                                  # gate logits: many gates at their bounds
        fb, lower = torch.randn(H * D, generator=gen), 0.02 + 0.96 * torch.rand(H * D, generator=gen)
        xd = x.double()
        q = torch.nn.functional.silu(xd[:, :H * D]).view(n, H, D)
        f = (lower.double() + (1 - lower.double()) * torch.sigmoid(xd[:, H * D:2 * H * D] + fb.double())).view(n, H, D)
        v = xd[:, 2 * H * D:].view(n, H, Dv)
        S = torch.zeros(H, D, Dv, dtype=torch.float64)
        want = torch.zeros(n, H, Dv, dtype=torch.float64)
        for t in range(n):
            S = f[t][:, :, None] * S + (1 - f[t])[:, :, None] * v[t][:, None, :]
            want[t] = torch.einsum("hij,hi->hj", S, q[t])
        dev = lambda t: t.to(gpu).contiguous()
        i32 = lambda *v_: torch.tensor(v_, dtype=torch.int32, device=gpu)
        for cuts in ([n], [1] * n, [2, 1, 7, 2, 11]):
            state = torch.full((3, H, D, Dv), float("nan"), device=gpu)
            state[1] = 0
            out, pos = [], 0
            for c in cuts:
                o = torch.empty(c, H * Dv, device=gpu)
                ops.forget_scan(dev(x[pos:pos + c]), dev(fb), dev(lower), state, o, q_start=i32(0), q_len=i32(c),
                                state_slot=i32(1), H=H, D=D, Dv=Dv)
                out.append(o.cpu())
                pos += c
            got = torch.cat(out).view(n, H, Dv).double()
            assert (got - want).abs().max() <= 2e-5 * max(1.0, float(want.abs().max())), (H, D, Dv, cuts)
            assert (state[1].double().cpu() - S).abs().max() <= 2e-5 * max(1.0, float(S.abs().max())), (H, D, Dv, cuts)
            assert torch.isnan(state[0]).all() and torch.isnan(state[2]).all()


@pytest.mark.parametrize("H, D, Dv", [(2, 16, 16), (3, 32, 80), (2, 48, 256), (2, 64, 128)])
@pytest.mark.parametrize("gates", ["spread", "at their bounds"])
def test_forget_scan_in_chunks_against_the_loop(gpu, H, D, Dv, gates):
    """The chunked form against the plain loop in float64: requests of 1 to 200 tokens and of none side by side, more of them
    than a wave has lanes, chunks and blocks that are full, partial and of one token, states in slots between slots of NaN; a second step goes
    on from the first's states.  Gates of exactly zero and one are among those at their bounds.  A rounding a token and some
    twenty a sum: 200 + 20 times 2^-24 of the sum of the magnitudes, 1.3e-5."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(H + D + Dv)
    lens = [200, 1, 0, 64, 65, 16, 17, 129] + [0, 1, 2] * 22
    R, T = len(lens), sum(lens)
    x = torch.randn(T, 2 * H * D + H * Dv, generator=gen)
    fb, lower = torch.randn(H * D, generator=gen), 0.9 * torch.rand(H * D, generator=gen)
    if gates != "spread":
        x[:, H * D:2 * H * D] *= 300.0                    # sigmoids of 0 and 1
        lower[::2] = 0.0
    q = torch.nn.functional.silu(x[:, :H * D].double()).view(T, H, D)
    f = (lower.double() + (1 - lower.double()) * torch.sigmoid(x[:, H * D:2 * H * D].double() + fb.double())).view(T, H, D)
    v = x[:, 2 * H * D:].double().view(T, H, Dv)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=gpu)
    S = [torch.randn(H, D, Dv, generator=gen) * (r % 2) for r in range(R)]
    state = torch.full((2 * R + 1, H, D, Dv), float("nan"), device=gpu)
    for r in range(R):
        state[2 * r + 1] = S[r].to(gpu)
    S = [s.double() for s in S]
    starts = [sum(lens[:r]) for r in range(R)]
    for step in range(2):
        out = torch.full((T, H * Dv), float("nan"), device=gpu)
        ops.forget_chunked(x.to(gpu), fb.to(gpu), lower.to(gpu), state, out, q_start=i32(starts), q_len=i32(lens),
                           state_slot=i32([2 * r + 1 for r in range(R)]), H=H, D=D, Dv=Dv)
        for r, n in enumerate(lens):
            for t in range(starts[r], starts[r] + n):
                S[r] = f[t][:, :, None] * S[r] + (1 - f[t])[:, :, None] * v[t][:, None, :]
                want, sizes = (S[r] * q[t][:, :, None]).sum(1), (S[r] * q[t][:, :, None]).abs().sum(1)
                assert ((out[t].double().cpu().view(H, Dv) - want).abs() <= 1.3e-5 * sizes.clamp(min=1.0)).all(), (step, r, t)
            assert (state[2 * r + 1].double().cpu() - S[r]).abs().max() <= 1.3e-5 * max(1.0, float(S[r].abs().max())), (step, r)
    assert all(torch.isnan(state[2 * r]).all() for r in range(R + 1))


@pytest.mark.parametrize("H, D, Dv", [(8, 64, 128), (8, 48, 256), (8, 32, 80), (16, 16, 16)])
@pytest.mark.parametrize("spread, lowest, mean", [(1.0, 0.9, 0.0), (4.0, 0.9, 0.0), (0.3, 0.99, 0.0), (300.0, 0.9, 0.0), (1.0, 0.0, -3.0)])
def test_forget_scan_in_chunks_is_no_further_from_64_bits(gpu, H, D, Dv, spread, lowest, mean):
    """Outputs and states of a request of 512 tokens and one of 300, token by token and in chunks, against the loop in float64:
    the norm of the difference is no larger in chunks, for gates of short and long memories and at their bounds."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(D)
    lens = [512, 300]
    T = sum(lens)
    x = torch.randn(T, 2 * H * D + H * Dv, generator=gen)
    x[:, H * D:2 * H * D] = x[:, H * D:2 * H * D] * spread + mean
    x, fb, lower = x.to(gpu), torch.randn(H * D, generator=gen).to(gpu), (lowest * torch.rand(H * D, generator=gen)).to(gpu)
    q = torch.nn.functional.silu(x[:, :H * D].double()).view(T, H, D)
    f = (lower.double() + (1 - lower.double()) * torch.sigmoid(x[:, H * D:2 * H * D].double() + fb.double())).view(T, H, D)
    v = x[:, 2 * H * D:].double().view(T, H, Dv)
    want, S = torch.empty(T, H, Dv, dtype=torch.float64, device=gpu), torch.zeros(2, H, D, Dv, dtype=torch.float64, device=gpu)
    for t in range(T):
        r = int(t >= lens[0])
        S[r] = f[t][:, :, None] * S[r] + (1 - f[t])[:, :, None] * v[t][:, None, :]
        want[t] = (S[r] * q[t][:, :, None]).sum(1)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=gpu)
    off = []
    for fn in (ops.forget_scan, ops.forget_chunked):
        out, state = torch.empty(T, H * Dv, device=gpu), torch.zeros(2, H, D, Dv, device=gpu)
        fn(x, fb, lower, state, out, q_start=i32([0, lens[0]]), q_len=i32(lens), state_slot=i32([0, 1]), H=H, D=D, Dv=Dv)
        off.append((float((out.view_as(want) - want).norm()), float((state - S).norm())))
    assert off[1][0] <= off[0][0] and off[1][1] <= off[0][1], off


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("H, D, Dv", [(2, 64, 128), (3, 32, 48)])
def test_forget_scan_in_chunks_with_a_value_that_is_not_finite(gpu, H, D, Dv, bad):
    """One value of one head and channel in the middle of a block: every output before its token is what it is without it, and
    so is every other channel's; from its token on the channel has none that is finite, as token by token.  The step's
    other request sees nothing of it."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(D)
    lens, at, head, ch = [100, 20], 73, 1, 5
    T = sum(lens)
    x = torch.randn(T, 2 * H * D + H * Dv, generator=gen).to(gpu)
    fb, lower = torch.randn(H * D, generator=gen).to(gpu), (0.9 * torch.rand(H * D, generator=gen)).to(gpu)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=gpu)
    spoilt = x.clone()
    spoilt[at, 2 * H * D + head * Dv + ch] = bad
    got = []
    for fn, rows in ((ops.forget_chunked, x), (ops.forget_chunked, spoilt), (ops.forget_scan, spoilt)):
        out, state = torch.empty(T, H * Dv, device=gpu), torch.zeros(2, H, D, Dv, device=gpu)
        fn(rows, fb, lower, state, out, q_start=i32([0, lens[0]]), q_len=i32(lens), state_slot=i32([0, 1]), H=H, D=D, Dv=Dv)
        got.append((out.view(T, H, Dv), state))
    (clean, clean_state), (out, state), (token_by_token, _) = got
    touched = torch.zeros(T, H, Dv, dtype=torch.bool, device=gpu)
    touched[at:lens[0], head, ch] = True
    assert not torch.isfinite(out[touched]).any() and not torch.isfinite(token_by_token[touched]).any()
    # (the block with the value adds in 64 bits in another order: the last bit of a few of its outputs)
    assert ((out - clean)[~touched].abs() <= 2.0 ** -23 * clean[~touched].abs()).all() and torch.isfinite(token_by_token[~touched]).all()
    assert torch.equal(out[:64], clean[:64]) and torch.equal(out[lens[0]:], clean[lens[0]:]) and torch.equal(state[1], clean_state[1])
    assert not torch.isfinite(state[0, head, :, ch]).any()
    state[0, head, :, ch] = clean_state[0, head, :, ch]
    assert torch.equal(state[0], clean_state[0])


@pytest.mark.parametrize("n", [287, 288, 400, 700])
def test_forget_gate_of_a_request_has_the_same_bits_alone_and_in_company(gpu, n):
    """The mixer's step for one request alone, and among others with single tokens, short portions and long ones: outputs and
    state of every request are what the request has alone, whichever form its number of tokens takes."""
    import types
    from tuff_amd.engine.batch import StepEntry, build_context
    from tuff_amd.parts.base import Runtime
    from tuff_amd.parts.recurrent import ForgetGateMixer
    H, D, Dv = 4, 64, 32
    eng = engine("wide", "bfloat16", max_tokens=4096, max_requests=8)
    gen = torch.Generator().manual_seed(n)
    m = ForgetGateMixer(96, H, D, Dv, 1e-5, names={k: k for k in ("q", "f", "f.b", "lower", "v", "norm", "o")})
    m.rt = Runtime(gpu, torch.bfloat16)
    m.f_bias, m.lower = torch.randn(H * D, generator=gen).to(gpu), (0.9 * torch.rand(H * D, generator=gen)).to(gpu)
    m.norm_w = torch.ones(Dv, device=gpu)
    lens = {"a": 1, "b": n, "c": 30, "d": 1, "e": 290, "f": 287, "g": 1}
    rows = {k: torch.randn(v, H * (2 * D + Dv), generator=gen).to(gpu) for k, v in lens.items()}
    S0 = torch.randn(8, H, D, Dv, generator=gen).to(gpu)

    def step(ids):
        for k in ids:
            eng.begin(k)
            eng.manager.extend(k, lens[k])
        ctx = build_context([StepEntry(k, [0] * lens[k], []) for k in ids], eng.manager, gpu, 333)
        slots = [eng.manager.slot(k) for k in ids]
        state = torch.full_like(S0, float("nan"))
        for k, slot in zip(ids, slots):
            state[slot] = S0[list(lens).index(k)]
        kept = []
        m.qfv = types.SimpleNamespace(forward=lambda h, out_dtype: torch.cat([rows[k] for k in ids]))
        m.out = types.SimpleNamespace(forward=lambda y, **kw: kept.append(y))
        m.forward(torch.empty(ctx.T, 96, dtype=torch.bfloat16, device=gpu), ctx, types.SimpleNamespace(state=state), None)
        for k in ids:
            eng.end(k)
        return {k: (y.float(), state[slot]) for k, y, slot in zip(ids, kept[0].split([lens[k] for k in ids]), slots)}

    together = step(list(lens))
    for k in lens:
        alone = step([k])[k]
        assert torch.isfinite(alone[0]).all() and torch.isfinite(alone[1]).all()
        assert torch.equal(alone[0], together[k][0]) and torch.equal(alone[1], together[k][1]), k


def _counted(monkeypatch):
    """How often each form of the forget gate's recurrence was launched."""
    from tuff_amd.csrc import ops
    calls = {"forget_scan": 0, "forget_chunked": 0}
    for name in calls:
        def wrapped(*a, _name=name, _fn=getattr(ops, name), **kw):
            calls[_name] += 1
            return _fn(*a, **kw)
        monkeypatch.setattr(ops, name, wrapped)
    return calls


@pytest.mark.parametrize("how", ["whole", "then single tokens", "in portions", "beside others"])
def test_prompts_long_enough_for_the_recurrence_in_chunks(gpu, monkeypatch, how):
    """Prompts of 288 tokens and more through the engine, whole, decoded on token by token, in portions on both sides of that
    length, and beside single tokens and short requests: the logits of the plain model every time."""
    calls = _counted(monkeypatch)
    reqs = requests("wide", [450, 300] if how == "beside others" else [700, 289], seed=11)
    if how == "whole":
        plan = util.plan_whole(reqs)
    elif how == "then single tokens":
        plan = util.plan_tail(reqs, tail=33)
    elif how == "in portions":
        plan = util.plan_chunks(reqs, sizes=(300, 7, 1, 290, 64, 2))
    else:
        reqs.update({"x": util.rand_tokens(24, 333, 7), "y": util.rand_tokens(60, 333, 8)})
        at = {k: 0 for k in reqs}
        plan = []
        for sizes in ({"x": 20}, {"x": 1, "r0": 400, "y": 40}, {"x": 1, "r1": 290, "y": 10, "r0": 20}, {"x": 1, "y": 8, "r1": 10, "r0": 28},
                      {"x": 1, "y": 2, "r0": 2}):
            entries = []
            for k, n in sizes.items():
                entries.append({"id": k, "tokens": reqs[k][at[k]:at[k] + n], "want": list(range(n))})
                at[k] += n
            plan.append({"step": len(plan), "entries": entries, "end": [k for k in sizes if at[k] == len(reqs[k])]})
    check("wide", "bfloat16", plan, reqs, max_tokens=2048)
    assert calls["forget_chunked"] > 0 and (how == "whole" or calls["forget_scan"] > 0)


def test_recorded_steps_of_long_portions_short_ones_and_both(gpu):
    """Steps of one number of tokens, as one long portion, as four short ones and as a long one beside short ones, in turn and often
    enough to be recorded and replayed: every logit is the eager step's, and there is a recording of each kind."""
    reqs = {k: util.rand_tokens(3000, 333, 20 + i) for i, k in enumerate("abcd")}
    at, steps = {k: 0 for k in reqs}, []
    for _ in range(6):
        for sizes in ({"a": 448}, {k: 112 for k in "abcd"}, {"b": 400, "c": 24, "d": 24}):
            entries = []
            for k, n in sizes.items():
                at[k] = at[k] if at[k] + n <= 3000 else 0
                entries.append({"id": k, "tokens": reqs[k][at[k]:at[k] + n], "want": [0, n - 1]})
                at[k] += n
            steps.append({"step": len(steps), "entries": entries, "end": []})
        steps.append({"step": len(steps), "entries": [{"id": k, "tokens": reqs[k][:1], "want": [0]} for k in "abcd"], "end": []})
    steps[-1]["end"] = list("abcd")
    kw = dict(max_tokens=16384, max_requests=6)
    want = util.run_plan(engine("wide", "bfloat16", use_graphs=False, **kw), steps)
    eng = engine("wide", "bfloat16", **kw)
    got = util.run_plan(eng, steps)
    assert eng.section_recordings == 3 and eng.section_replays == 3 * 4
    for k in reqs:
        wanted = ~torch.isnan(want[k][:, 0])
        assert wanted.any() and torch.equal(got[k][wanted], want[k][wanted]), k


def test_forget_scan_in_chunks_takes_as_many_requests_as_the_scan(gpu):
    """More requests than a grid's second axis holds, all but the last without tokens: what the last has alone.  A state that lies on no
    16-byte border is refused (the mixer then takes the scan)."""
    from tuff_amd.csrc import ops
    H, D, Dv, n, R = 1, 16, 16, 70, 70000
    gen = torch.Generator().manual_seed(1)
    x, lower = torch.randn(n, 2 * H * D + H * Dv, generator=gen).to(gpu), (0.9 * torch.rand(H * D, generator=gen)).to(gpu)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=gpu)
    got = []
    for many in (1, R):
        out, state = torch.empty(n, H * Dv, device=gpu), torch.zeros(2, H, D, Dv, device=gpu)
        ops.forget_chunked(x, None, lower, state, out, q_start=i32([0] * many), q_len=i32([0] * (many - 1) + [n]),
                           state_slot=i32([0] * (many - 1) + [1]), H=H, D=D, Dv=Dv)
        got.append((out, state))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and not got[1][1][0].any()
    off = torch.zeros(2 * H * D * Dv + 1, device=gpu)[1:].view(2, H, D, Dv)
    assert ops.forget_chunked_supported(D, Dv) and not ops.forget_chunked_supported(D, Dv, off)
    with pytest.raises(ops.KernelError):
        ops.forget_chunked(x, None, lower, off, got[0][0], q_start=i32([0]), q_len=i32([n]), state_slot=i32([1]), H=H, D=D, Dv=Dv)


@pytest.mark.parametrize("name, dtype", [("wide", "float32"), ("mixed", "bfloat16")])
def test_one_recording_a_number_of_tokens_where_no_part_asks_for_long_runs(gpu, name, dtype):
    """float32, and sizes that the chunks do not take: a step of one long portion and one of short ones launch the same and
    share a recording."""
    reqs = {k: util.rand_tokens(448 * 4, lu.CONFIGS[name]["vocab"], 30 + i) for i, k in enumerate("ab")}
    steps = [{"step": i, "entries": [{"id": k, "tokens": reqs[k][n * i:n * (i + 1)], "want": [n - 1]} for k, n in sizes], "end": []}
             for i in range(4) for sizes in ([("a", 448)], [("a", 224), ("b", 224)])]
    steps[-1]["end"] = ["a", "b"]
    eng = engine(name, dtype, max_tokens=8192)
    util.run_plan(eng, steps)
    assert eng.section_recordings == 1 and eng.section_replays == 6 and len(eng._sectioned) == 1


@pytest.mark.parametrize("H, Hkv, vd", [(4, 2, 64), (32, 8, 64), (12, 3, 5), (16, 2, 130), (8, 1, 70), (6, 2, 33), (5, 5, 16), (1, 1, 1)])
def test_mix_of_heads_against_the_sum_in_float64(gpu, H, Hkv, vd):
    """Two, four and eight heads a kv head (with and without heads left over after eight at a time) and the others: to the
    rounding of H float32 steps, and of the output's type."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(H + vd)
    o, talk, gates = (torch.randn(*s, generator=gen) for s in ((7, H * Hkv * vd), (H, H), (7, H + 3)))
    ov, t64 = o.double().view(7, H, Hkv, vd), talk.double()
    kv_of = torch.arange(H) // (H // Hkv)
    picked = ov[:, :, kv_of, :]                                  # [t][summed head][h][vd]
    want = torch.stack([(t64[h][None, :, None] * picked[:, :, h]).sum(1) for h in range(H)], 1)
    size = torch.stack([(t64[h].abs()[None, :, None] * picked[:, :, h].abs()).sum(1) for h in range(H)], 1)
    for gated in (False, True):
        f = torch.sigmoid(gates[:, :H].double())[:, :, None] if gated else 1.0
        for dt, unit in ((torch.float32, 2.0 ** -24), (torch.bfloat16, 2.0 ** -8)):
            out = torch.full((7, H * vd), float("nan"), dtype=dt, device=gpu)
            ops.head_mix_gate(o.to(gpu), out, H=H, Hkv=Hkv, vd=vd, talk=talk.to(gpu), gates=gates.to(gpu) if gated else None)
            err = (out.cpu().double().view(7, H, vd) - want * f).abs()
            # H + 1 roundings of the sum and the gate's few units; then the output's own
            assert (err <= (H + 8) * 2.0 ** -24 * size * f + unit * (want * f).abs()).all(), (dt, gated)


@pytest.mark.parametrize("H, Hkv, vd", [(32, 2, 64), (24, 2, 130), (12, 2, 65), (20, 2, 33), (8, 1, 256), (4, 2, 512), (6, 1, 70), (3, 1, 64)])
def test_mix_of_heads_of_few_tokens_and_of_many(gpu, H, Hkv, vd):
    """Kv heads of 2, 3, 6, 10, 12 and 16 heads: few tokens (a wave for every 64 channels) and many (a wave all of them) to the same
    bits, and those to H + 1 float32 roundings of the sum in float64."""
    from tuff_amd.csrc import ops
    T = 1024 * 4 // H + 5
    gen = torch.Generator().manual_seed(H * vd)
    o, talk = (torch.randn(*s, generator=gen) for s in ((T, H * Hkv * vd), (H, H)))
    od, td = o.to(gpu), talk.to(gpu)
    out = torch.full((T, H * vd), float("nan"), device=gpu)
    ops.head_mix_gate(od, out, H=H, Hkv=Hkv, vd=vd, talk=td)
    for t0, n in ((0, 1), (T - 7, 7)):
        few = torch.full((n, H * vd), float("nan"), device=gpu)
        ops.head_mix_gate(od[t0:t0 + n].contiguous(), few, H=H, Hkv=Hkv, vd=vd, talk=td)
        assert torch.equal(few, out[t0:t0 + n])
    picked = o.double().view(T, H, Hkv, vd)[:, :, torch.arange(H) // (H // Hkv), :]
    want = torch.stack([(talk[h].double()[None, :, None] * picked[:, :, h]).sum(1) for h in range(H)], 1)
    size = torch.stack([(talk[h].double().abs()[None, :, None] * picked[:, :, h].abs()).sum(1) for h in range(H)], 1)
    assert ((out.cpu().double().view(T, H, vd) - want).abs() <= (H + 1) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("D", [24, 64, 68, 128, 256])
def test_scan_gives_the_same_bits_for_any_company_and_alignment(gpu, D):
    """The recurrence's kernel over nine requests of 0 to 41 tokens (edges of the eight tokens it stages at a time), with
    heads that do not fill rounds of the chip's eight parts, against each request alone, and with inputs that a wide load
    cannot fetch: the same bits."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(11)
    H, lens = 3, [7, 0, 8, 9, 1, 16, 41, 2, 24]
    T = sum(lens)
    r, k, v = (torch.randn(T, H * D, generator=gen) for _ in range(3))
    lw, w0, u = torch.randn(T, H * D, generator=gen), torch.randn(H * D, generator=gen).to(gpu), torch.randn(H, D, generator=gen).to(gpu)
    state0 = torch.randn(len(lens), H, D, D, generator=gen)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=gpu)
    starts = [sum(lens[:i]) for i in range(len(lens))]

    def scan(sel, q_start, q_len, slots, shift, dt):
        def put(t, d):
            t = t[sel].to(d)
            room = torch.zeros(t.numel() + shift, dtype=d, device=gpu)
            room[shift:] = t.flatten().to(gpu)
            return room[shift:].view(t.shape)
        state, out = state0.to(gpu), torch.full((len(range(T)[sel]), H * D), float("nan"), device=gpu)
        ops.wkv_scan(put(r, dt), put(k, dt), put(v, dt), put(lw, torch.float32), w0, u, state, out, q_start=i32(q_start), q_len=i32(q_len),
                     state_slot=i32(slots), H=H, D=D)
        return out.cpu(), state.cpu()

    for dt in (torch.bfloat16, torch.float32):
        out, state = scan(slice(0, T), starts, lens, list(range(len(lens))), 0, dt)
        assert torch.isfinite(out).all()
        out1, state1 = scan(slice(0, T), starts, lens, list(range(len(lens))), 1, dt)
        assert torch.equal(out, out1) and torch.equal(state, state1), "the result depends on the alignment"
        for i, n in enumerate(lens):
            if n:
                alone, s = scan(slice(starts[i], starts[i] + n), [0], [n], [i], 0, dt)
                assert torch.equal(alone, out[starts[i]:starts[i] + n]) and torch.equal(s[i], state[i]), (dt, i)
            else:
                assert torch.equal(state[i], state0[i])


@pytest.mark.parametrize("C, K, bias, act", [(3072, 4, False, None), (1028, 3, True, "silu"), (516, 2, True, None), (8, 4, False, "silu")])
@pytest.mark.parametrize("dtype, out", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16), (torch.float32, torch.float32)])
def test_convolution_of_four_channels_a_thread_has_the_bits_of_one(gpu, C, K, bias, act, dtype, out):
    """Few tokens and many, requests that begin inside a run of four, portions shorter than the taps; rows off a border of four
    elements take the kernel of one channel a thread."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(C + K)
    for lens in ([1], [1, 2, 3, 1], [40, 1, 2, 700, 3, 1, 601]):
        T, R = sum(lens), len(lens)
        x, taps, state = (torch.randn(*s, generator=gen) for s in ((T, C), (C, K), (R, K - 1, C)))
        b = torch.randn(C, generator=gen).to(gpu) if bias else None
        i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=gpu)
        got = []
        for ld in (C, C + 1):
            rows = torch.zeros(T, ld, dtype=dtype, device=gpu)
            rows[:, :C] = x.to(gpu)
            st, y = state.to(gpu), torch.full((T, C), float("nan"), dtype=out, device=gpu)
            more = {} if b is None else {"bias": b}
            ops.conv_act(rows[:, :C], taps.to(gpu), st, y, req_of_token=i32(sum([[r] * n for r, n in enumerate(lens)], [])),
                         q_start=i32([sum(lens[:r]) for r in range(R)]), q_len=i32(lens), state_slot=i32(list(range(R))), activation=act, **more)
            got.append((y, st))
        assert all(torch.equal(a, b_) for a, b_ in zip(*got)), lens


@pytest.mark.parametrize("T, H, vd", [(1, 1, 8), (3, 5, 24), (700, 32, 64), (129, 3, 136)])
def test_gates_and_biases_of_several_numbers_a_thread_have_the_bits_of_one(gpu, T, H, vd):
    """Rows off a 16-byte border take the kernels of one number a thread."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(T)
    o, gates = torch.randn(T * H * vd, generator=gen).bfloat16().to(gpu), torch.randn(T, H, generator=gen).to(gpu)
    x, bias = torch.randn(T * H * vd, generator=gen).to(gpu), torch.randn(H * vd, generator=gen).to(gpu)
    got = []
    for off in (0, 1):
        at = lambda like: torch.empty(like.numel() + 1, dtype=like.dtype, device=gpu)[off:off + like.numel()].copy_(like)
        y = torch.empty(T, H * vd, dtype=torch.bfloat16, device=gpu)
        ops.head_mix_gate(at(o).view(T, H * vd), y, H=H, Hkv=1, vd=vd, gates=gates)
        casts = [torch.empty(T, H * vd, dtype=dt, device=gpu) for dt in (torch.bfloat16, torch.float32)]
        for c in casts:
            ops.cast(at(x).view(T, H * vd), c, bias)
        got.append([y] + casts)
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("T", [1, 17, 300])
@pytest.mark.parametrize("H, G, rot, norm, ps", [(32, 8, 32, True, 16), (3, 3, 64, False, 48), (5, 1, 20, True, 32), (4, 2, 0, True, 16), (4, 4, 0, False, 64)])
def test_heads_of_64_turned_in_pairs_or_not_at_all(gpu, T, H, G, rot, norm, ps):
    """The kernel of sixteen lanes a head has the bits of the one of a wave a head, which rows off a 16-byte border take: what
    comes out does not depend on where a row lies."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(T + H)
    width = (H + 2 * G) * 64
    qkv = torch.randn(T * width, generator=gen).bfloat16().to(gpu)
    w = [(torch.rand(64, generator=gen) + 0.5).to(gpu) for _ in "qk"] if norm else [None, None]
    inv = (10000.0 ** (-torch.arange(rot // 2) * 2 / rot)).float().to(gpu) if rot else None
    pos = torch.arange(5, 5 + T, dtype=torch.int32, device=gpu)
    got = []
    for off in (0, 1):
        at = torch.empty(T * width + 1, dtype=torch.bfloat16, device=gpu)[off:off + T * width]
        at.copy_(qkv)
        q = torch.zeros(T, H * 64, dtype=torch.bfloat16, device=gpu)
        P = -(-(T + 5) // ps) + 1
        k, v = torch.zeros(P, G, ps, 64, dtype=torch.bfloat16, device=gpu), torch.zeros(P, G, 64, ps, dtype=torch.bfloat16, device=gpu)
        ops.qkv_post(at.view(T, width), q, H=H, Hkv=G, hd=64, positions=pos, eps=1e-5, q_norm_w=w[0], k_norm_w=w[1], inv_freq=inv,
                     rotary_dim=rot, interleaved=True, k_cache=k, v_cache=v, slot_mapping=pos + ps, page_size=ps)
        got.append((q, k, v))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind, H, D, Dv", [("forget", 3, 40, 33), ("forget", 2, 64, 128), ("forget", 5, 65, 32), ("ssd", 4, 64, 40),
                                            ("ssd", 2, 128, 64), ("delta", 3, 100, 130), ("delta", 2, 192, 48), ("wkv", 3, 72, 72),
                                            ("wkv", 1, 128, 128)])
def test_runs_in_four_waves_have_the_bits_of_short_runs(gpu, kind, H, D, Dv, dtype):
    """Long runs, whose waves bring rows into LDS for each other, in one step with shorter ones; and the same
    tokens in steps of up to 20, which waves take alone: numbers of tokens around sixteen, channels that fill no tile."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(H + D + Dv)
    rnd = lambda *shape: torch.randn(*shape, generator=gen)
    lens = [65, 31, 48, 1, 111 if kind != "ssd" or D > 64 else 1511]      # (the last takes them from 320 tokens a request on)
    T, R = sum(lens), len(lens)
    if kind == "forget":
        rows = [rnd(T, 2 * H * D + H * Dv).to(dtype)]
        bias, lower = rnd(H * D).to(gpu), torch.rand(H * D, generator=gen).to(gpu)
        call = lambda x, s, o, **kw: ops.forget_scan(x, bias, lower, s, o, H=H, D=D, Dv=Dv, **kw)
    elif kind == "ssd":
        rows = [rnd(T, H * Dv + 2 * D).to(dtype), rnd(T, H)]
        b, A, skip = (rnd(H).to(gpu) for _ in range(3))
        call = lambda x, r, s, o, **kw: ops.ssd_scan(x, r, b, A, skip, s, o, H=H, G=1, N=D, P=Dv, **kw)
    elif kind == "delta":
        rows = [rnd(T, H * D).to(dtype), rnd(T, H * D).to(dtype), rnd(T, H * Dv).to(dtype), rnd(T, H * D), rnd(T, H)]
        b, A = rnd(H * D).to(gpu), rnd(H).to(gpu)
        call = lambda q, k, v, a, beta, s, o, **kw: ops.delta_scan(q, k, v, a, b, A, beta, s, o, H=H, Hk=H, D=D, Dv=Dv, **kw)
    else:
        rows = [rnd(T, H * D).to(dtype) for _ in range(3)] + [rnd(T, H * D) * 0.5]
        w0, u = rnd(H * D).to(gpu), rnd(H, D).to(gpu)
        call = lambda r, k, v, lw, s, o, **kw: ops.wkv_scan(r, k, v, lw, w0, u, s, o, H=H, D=D, **kw)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device=gpu)
    first = [sum(lens[:i]) for i in range(R)]
    state = rnd(R, H, D, Dv).to(gpu)
    whole, out = state.clone(), torch.full((T, H * Dv), float("nan"), device=gpu)
    call(*[t.to(gpu) for t in rows], whole, out, q_start=i32(first), q_len=i32(lens), state_slot=i32(list(range(R))))
    cut, parts = state.clone(), torch.full((T, H * Dv), float("nan"), device=gpu)
    for r, n in enumerate(lens):
        for at in range(first[r], first[r] + n, 20):
            m = min(20, first[r] + n - at)
            piece = torch.empty(m, H * Dv, device=gpu)
            call(*[t[at:at + m].to(gpu) for t in rows], cut, piece, q_start=i32([0]), q_len=i32([m]), state_slot=i32([r]))
            parts[at:at + m] = piece
    assert torch.equal(out, parts) and torch.equal(whole, cut)


@pytest.mark.parametrize("D, Dv", [(16, 16), (30, 50), (32, 64), (64, 128), (96, 20), (130, 130), (256, 24)])
def test_single_tokens_of_a_scan_have_the_bits_of_a_run(gpu, D, Dv):
    """A request with one token takes no stop in LDS; portions that end inside the tokens staged at a time stage only their own:
    thirteen tokens in any cut, the same outputs and state."""
    from tuff_amd.csrc import ops
    gen = torch.Generator().manual_seed(D)
    H, n = 2, 13
    rnd = lambda *shape: torch.randn(*shape, generator=gen).to(gpu)
    i32 = lambda x: torch.tensor([x], dtype=torch.int32, device=gpu)
    state0, hd, h = rnd(1, H, D, Dv), rnd(H * D), [rnd(H) for _ in range(3)]
    for dt in (torch.bfloat16, torch.float32):
        x, q, k, v, xbc = (rnd(n, w).to(dt) for w in (2 * H * D + H * Dv, H * D, H * D, H * Dv, H * Dv + 2 * D))
        a, b = rnd(n, H * D), rnd(n, H)
        lower = torch.rand(H * D, generator=gen).to(gpu)
        kinds = {
            "forget": lambda t, st, o, kw: ops.forget_scan(x[t], hd, lower, st, o, H=H, D=D, Dv=Dv, **kw),
            "delta": lambda t, st, o, kw: ops.delta_scan(q[t], k[t], v[t], a[t].clone(), hd, h[0], b[t], st, o, H=H, Hk=H, D=D, Dv=Dv, **kw),
            "state space": lambda t, st, o, kw: ops.ssd_scan(xbc[t], b[t], *h, st, o, H=H, G=1, N=D, P=Dv, **kw)}
        if D == Dv:
            kinds["wkv"] = lambda t, st, o, kw: ops.wkv_scan(q[t], k[t], v[t], a[t].clone(), hd, hd.view(H, D), st, o, H=H, D=D, **kw)
        for name, scan in kinds.items():
            results = []
            for cuts in ([n], [1] * n, [1, 2, 3, 7], [4, 1, 8], [5, 6, 1, 1]):
                state, out, at = state0.clone(), torch.full((n, H * Dv), float("nan"), device=gpu), 0
                for c in cuts:
                    scan(slice(at, at + c), state, out[at:at + c], dict(q_start=i32(0), q_len=i32(c), state_slot=i32(0)))
                    at += c
                results.append((out, state))
            assert torch.isfinite(results[0][0]).all(), name
            for out, state in results[1:]:
                assert torch.equal(out, results[0][0]) and torch.equal(state, results[0][1]), (name, dt)


# ------------------------------------------------------------------- generation, command line
def test_greedy_generation_through_the_scheduler(gpu):
    from tuff_amd.engine.llm import LLM
    from tuff_amd.sampling.params import SamplingParams
    reqs = requests("mixed", [5, 21, 1, 12, 30, 8], seed=9)
    _, raw, w = model("mixed")
    eng = engine("mixed", "float32", max_tokens=512, max_requests=3)
    llm = LLM(engine=eng, max_num_seqs=3, max_batched_tokens=16, ctx_size=128, ignore_eos=True)
    outs = llm.generate(list(reqs.values()), SamplingParams(temp=0.0, max_new_tokens=10, ignore_eos=True))
    for g, prompt in zip(outs, reqs.values()):
        assert list(g.token_ids) == plain.greedy(raw, w, prompt, 10), prompt
    eng.manager.check()
    assert not eng.manager.live()


def test_command_line_and_trace_replay(gpu, tmp_path):
    folder, raw, w = model("wide")
    prompt = util.rand_tokens(9, raw["vocab"], 3)
    p = subprocess.run([sys.executable, os.path.join(util.ROOT, "bin", "tuff"), "--model", folder, "--prompt-ids",
                        ",".join(map(str, prompt)), "--dump-tokens", "-n", "6", "--dtype", "fp32", "--temp", "0"],
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-2000:]
    assert [int(x) for x in p.stdout.split()] == plain.greedy(raw, w, prompt, 6)
    q = subprocess.run([sys.executable, os.path.join(util.ROOT, "bin", "tuff"), "--model", folder, "--inspect"],
                       capture_output=True, text=True, timeout=300)
    assert q.returncode == 0 and "PairMixer" in q.stdout and "ForgetGateMixer" in q.stdout, q.stderr[-2000:]
    # the trace runner: a mixed plan through a child process, four slots, a pool no larger than the plan's peak
    reqs = requests("wide", [50, 3, 70, 20, 31], seed=10)
    plan = util.plan_mixed(reqs, seed=2)
    out = tmp_path / "out"
    cmd = [sys.executable, os.path.join(util.ROOT, "bin", "trace_run"), "--model", folder, "--dtype", "float32",
           "--out", str(out), "--max-tokens", str(util.live_tokens_peak(plan))]
    proc = subprocess.Popen(cmd, stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True)
    try:
        for s in plan:
            proc.stdin.write(json.dumps(s) + "\n")
            proc.stdin.flush()
            assert proc.stdout.readline().strip() == f"done {s['step']}"
        proc.stdin.close()
        assert proc.wait(timeout=120) == 0
    finally:
        if proc.poll() is None:
            proc.kill()
    fed = {rid: 0 for rid in reqs}
    for s in plan:
        n_want = sum(len(e["want"]) for e in s["entries"])
        data = torch.from_numpy(np.fromfile(out / f"{s['step']}.f32", dtype="<f4").reshape(n_want, raw["vocab"]).copy())
        i = 0
        for e in s["entries"]:
            want = expected("wide", reqs[e["id"]]).want
            rows = [fed[e["id"]] + w_ for w_ in e["want"]]
            util.assert_close_f32(data[i:i + len(rows)], want[rows], f"step {s['step']} {e['id']}")
            i += len(rows)
            fed[e["id"]] += len(e["tokens"])
