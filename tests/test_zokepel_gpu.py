"""Zokepel on the GPU against the plain implementation, in 32-bit and in bfloat16: every mixer kind alone; whole
prompts; most of a prompt in one step and its last tokens one by one; portions of changing size down to two tokens;
mixed batches in a pool so small that pages and slots are used again; long decoding; the first tokens; kernels with
inputs made so that one far key, one distance bucket or one old write stands out; generation through the scheduler,
the replay program and the command line."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from tests import helpers as H
from tests import zokepel_helpers as ZH
from tests.plain import zokepel_plain as Z
from tests.test_engine_gpu import mixed_schedule, portions, run_steps

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DTYPES = ["float32", "bfloat16"]
NAMES = ["P", "Q", "R", "S"]
LENGTHS = {"P": 150, "Q": 210, "R": 120, "S": 330}
# bfloat16 against the plain implementation, per row: relative L2 error of the logits (1.5 x the worst row measured
# for these models; a wrong bucket, a lost state or a missing scale shows as tens of percent)
BF16_REL_L2 = 0.06
# A sequence's first token gets more: every state is empty there, so each recurrent head's read-out is one outer
# product, (k . q) u for the delta rule and (sum_i bonus_i k_i r_i) v for the time mixing, and dividing it by its root
# mean square leaves a direction times a factor that depends on that one inner product and the norm's eps alone:
# where the products' terms cancel, their bfloat16 rounding is amplified (measured up to 8.4 % for one sequence,
# the same in every batching; 32-bit is not affected).
BF16_REL_L2_FIRST = 0.15
# The same amplification happens at single later tokens where a head's read-out nearly cancels before it is divided
# by its root mean square (random weights; measured: one row in some sequences at 10 % between neighbours at 1 %, bit
# for bit the same alone, in portions, decoded and beside other requests).  One row in fifty may therefore exceed
# the bound, none twice the first token's.
BF16_ROWS_OVER = 0.02
BF16_REL_L2_WORST = 0.3


@pytest.fixture(scope="module")
def dirs(tmp_path_factory):
    root = tmp_path_factory.mktemp("zokepel")
    out = {n: ZH.make_model_dir(str(root), ZH.MODELS[n], n, seed=31 + i) for i, n in enumerate(NAMES)}
    for kind in ("delta", "channel_delta", "parallel"):
        out[kind] = ZH.make_model_dir(str(root), ZH.single_layer(kind), kind, seed=5)
    return out


def make_engine(model_dir, dtype, **kw):
    from gibbs_amd import Engine
    kw.setdefault("max_tokens", 2048)
    kw.setdefault("max_requests", 4)
    return Engine(model_dir, dtype=dtype, **kw)


def close(got, want, dtype, what, places=None):
    """`places`: the rows' positions in their sequence (position 0 has a bound of its own in bfloat16)."""
    got, want = np.asarray(got, dtype=np.float64), np.asarray(want, dtype=np.float64)
    assert got.shape == want.shape, (what, got.shape, want.shape)
    if dtype == "float32":
        err = np.abs(got - want).max(-1)
        bound = 2e-5 * np.abs(want).max()
        assert err.max() <= bound, f"{what}: max error {err.max():.3e} at row {int(err.argmax())} above {bound:.3e}; first bad row {int((err > bound).argmax())}"
        return
    rel = np.sqrt(((got - want) ** 2).sum(-1) / (want ** 2).sum(-1))
    bound = np.full(rel.shape, BF16_REL_L2)
    if places is not None:
        bound[np.asarray(places) == 0] = BF16_REL_L2_FIRST
    over = int((rel > bound).sum())
    assert over <= max(1, int(BF16_ROWS_OVER * rel.size)) and rel.max() <= BF16_REL_L2_WORST, (
        f"{what}: {over} of {rel.size} rows over their bound, relative L2 error {rel.max():.3e} at row {int(rel.argmax())}; "
        f"first bad row {int((rel > bound).argmax())}")


def check(model_dir, seqs, got, dtype, what):
    for rid, ids in seqs.items():
        want = ZH.plain_logits(model_dir, ids)
        places = sorted(p for r, p in got if r == rid)
        assert places, f"{what}: no logits for {rid}"
        close(np.stack([got[(rid, p)] for p in places]), want[places], dtype, f"{what} request {rid}", places)


def vocab_of(model_dir):
    with open(os.path.join(model_dir, "config.json")) as f:
        return json.load(f)["vocab"]


# ----------------------------------------------------------------------------------------------- whole models
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("kind", ["delta", "channel_delta", "parallel"])
def test_each_mixer_alone(dirs, kind, dtype):
    d = dirs[kind]
    ids = ZH.tokens(1, 90, vocab_of(d))
    eng = make_engine(d, dtype)
    got = run_steps(eng, [([("r", ids[:61], list(range(61)))], []), ([("r", ids[61:], list(range(29)))], ["r"])])
    check(d, {"r": ids}, got, dtype, f"{kind} alone {dtype}")
    assert eng.cache.free_slots() == 4


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_whole(dirs, name, dtype):
    d = dirs[name]
    ids = ZH.tokens(2, LENGTHS[name], vocab_of(d))
    eng = make_engine(d, dtype)
    got = run_steps(eng, [([("r", ids, list(range(len(ids))))], ["r"])])
    check(d, {"r": ids}, got, dtype, f"whole {name} {dtype}")
    eng.cache.check()
    assert all(eng.cache.free_pages(g) == eng.cache.pools[g].num_pages for g in range(eng.cache.n_groups))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_bulk_then_last_32_one_by_one(dirs, name, dtype):
    d = dirs[name]
    ids = ZH.tokens(3, LENGTHS[name], vocab_of(d))
    cut = len(ids) - 32
    steps = [([("r", ids[:cut], list(range(cut)))], [])] + [([("r", [t], [0])], []) for t in ids[cut:]]
    got = run_steps(make_engine(d, dtype), steps)
    check(d, {"r": ids}, got, dtype, f"bulk+tail {name} {dtype}")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_changing_portions_down_to_two_tokens(dirs, name, dtype):
    d = dirs[name]
    ids = ZH.tokens(4, LENGTHS[name], vocab_of(d))
    cuts = portions(len(ids) - 9, [7, 2, 13, 3, 2, 64, 5, 2, 17, 1, 2]) + [(len(ids) - 9 + i, len(ids) - 8 + i) for i in range(9)]
    steps = [([("r", ids[a:b], list(range(b - a)))], []) for a, b in cuts]
    got = run_steps(make_engine(d, dtype), steps)
    check(d, {"r": ids}, got, dtype, f"portions {name} {dtype}")


@pytest.mark.parametrize("name", NAMES)
def test_cutting_changes_no_bit_in_32_bit(dirs, name):
    """The recurrences add in one order per token and the products in one order of k, so 32-bit logits do not depend on how
    the prompt was cut or on what else was in the batch."""
    d = dirs[name]
    ids = ZH.tokens(5, 77, vocab_of(d))
    other = ZH.tokens(6, 41, vocab_of(d))
    whole = run_steps(make_engine(d, "float32"), [([("r", ids, list(range(77)))], [])])
    eng = make_engine(d, "float32")
    steps = [([("o", other[:20], []), ("r", ids[:2], [0, 1])], []), ([("r", ids[2:50], list(range(48))), ("o", other[20:21], [])], []),
             ([("o", other[21:], []), ("r", ids[50:51], [0])], ["o"]), ([("r", ids[51:], list(range(26)))], [])]
    cut = run_steps(eng, steps)
    for p in range(77):
        assert np.abs(cut[("r", p)] - whole[("r", p)]).max() <= 2e-6 * np.abs(whole[("r", p)]).max(), p


@pytest.mark.parametrize("name", ["Q", "S"])
def test_long_portions_and_what_shares_their_step_change_no_bit_in_32_bit(dirs, name):
    """The same where portions are long enough for the rules in chunks of a bfloat16 run, and a decoded token, a short and a long portion share a step."""
    d = dirs[name]
    ids, other = ZH.tokens(21, 230, vocab_of(d)), ZH.tokens(22, 180, vocab_of(d))
    whole = run_steps(make_engine(d, "float32"), [([("r", ids, list(range(230)))], [])])
    steps = [([("r", ids[:30], list(range(30))), ("o", other[:140], [])], []), ([("r", ids[30:31], [0]), ("o", other[140:150], [])], []),
             ([("o", other[150:151], []), ("r", ids[31:180], list(range(149)))], []), ([("r", ids[180:], list(range(50)))], [])]
    cut = run_steps(make_engine(d, "float32"), steps)
    for p in range(230):
        assert np.array_equal(cut[("r", p)], whole[("r", p)]), (p, np.abs(cut[("r", p)] - whole[("r", p)]).max())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", NAMES)
def test_mixed_batches_with_pages_and_slots_used_again(dirs, name, dtype):
    d = dirs[name]
    rng = np.random.default_rng(7)
    seqs = {f"q{i}": ZH.tokens(100 + i, int(n), vocab_of(d)) for i, n in enumerate([70, 45, 90, 33, 64, 81, 50, 3, 2])}
    steps = mixed_schedule(seqs, rng)
    assert max(len(e) for e, _ in steps) >= 3
    assert any(len(t) > 1 for e, _ in steps for _, t, _ in e) and any(len(t) == 1 for e, _ in steps for _, t, _ in e)
    eng = make_engine(d, dtype, max_tokens=384, max_requests=4, page_size=16)
    assert sum(-(-len(s) // 16) for s in seqs.values()) > eng.cache.pools[0].num_pages, "the pool must be too small to avoid reuse"
    got = run_steps(eng, steps)
    check(d, seqs, got, dtype, f"mixed {name} {dtype}")
    eng.cache.check()
    assert eng.cache.free_slots() == 4 and all(eng.cache.free_pages(g) == eng.cache.pools[g].num_pages for g in range(eng.cache.n_groups))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("short", [1, 60])
@pytest.mark.parametrize("name", ["Q", "S"])
def test_decoding_beside_a_long_and_short_portions(dirs, name, short, dtype):
    """Steps of three decoding requests, one portion of 110 rows and `short` of five to seven, then of decoding alone: in bfloat16 the one-row kernels
    for the requests at the head of the step, and for those behind them, from a row and a request above 0, the rules in chunks (one short
    portion) or the delta rule's walk (sixty)."""
    from gibbs_amd.ops.lib import library
    d = dirs[name]
    n = 4 + short
    assert all(library().gibbs_rule_chunked(0, 110 + 6 * short, 1 + short, 110, *head) == (short == 1) for head in ((2, 128, 64), (4, 64, 32), (4, 128, 64)))
    assert short > 1 or all(library().gibbs_rule_chunked(1, 116, 2, 110, *head) for head in ((2, 64, 64), (4, 64, 64), (8, 32, 32)))
    ids = {f"d{i}": ZH.tokens(40 + i, 14 + i, vocab_of(d)) for i in range(3)}
    ids["long"] = ZH.tokens(50, 120, vocab_of(d))
    ids.update({f"s{i}": ZH.tokens(60 + i, 8 + i % 3, vocab_of(d)) for i in range(short)})
    every = lambda a, b: list(range(b - a))
    at = {r: len(x) - 4 if r[0] == "d" else (len(x) - 10 if r == "long" else len(x) - 3) for r, x in ids.items()}
    steps = [([(r, ids[r][:at[r]], every(0, at[r]))], []) for r in ids if r[0] == "d"]
    steps.append(([(r, ids[r][at[r]:at[r] + 1], [0]) for r in ids if r[0] == "d"] + [(r, ids[r][:at[r]], every(0, at[r])) for r in ids if r[0] != "d"], []))
    steps += [([(r, ids[r][at[r] + i + (r[0] == "d"):][:1], [0]) for r in ids], []) for i in range(3)]
    got = run_steps(make_engine(d, dtype, max_requests=n), steps)
    check(d, {r: x for r, x in ids.items() if r[0] != "s"}, got, dtype, f"{short} short {name} {dtype}")
    # the short ones against themselves alone, whole: sixty beginnings hold one whose first token's inner product nearly cancels (42 % of the plain
    # implementation's logits off in bfloat16, alone as here), see BF16_REL_L2_FIRST
    eng = make_engine(d, dtype)
    for r, x in ids.items():
        if r[0] == "s":
            alone = run_steps(eng, [([(r, x, every(0, len(x)))], [r])])
            close(np.stack([got[(r, p)] for p in range(len(x))]), np.stack([alone[(r, p)] for p in range(len(x))]), dtype, f"{r} of {short} {name} {dtype}", range(len(x)))


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding(dirs, dtype):
    d = dirs["P"]
    ids = ZH.tokens(9, 330, vocab_of(d))
    steps = [([("r", ids[:5], list(range(5)))], [])] + [([("r", [t], [0])], []) for t in ids[5:]]
    got = run_steps(make_engine(d, dtype), steps)
    check(d, {"r": ids}, got, dtype, f"long decoding {dtype}")


@pytest.mark.parametrize("dtype", DTYPES)
def test_first_tokens(dirs, dtype):
    """Sequences of one, two and three tokens, alone and side by side: zeros before the start in the convolutions
    and the shift, empty states, a single visible key."""
    d = dirs["P"]
    seqs = {f"s{n}": ZH.tokens(20 + n, n, vocab_of(d)) for n in (1, 2, 3, 5)}
    got = run_steps(make_engine(d, dtype), [([(r, ids, list(range(len(ids)))) for r, ids in seqs.items()], list(seqs))])
    check(d, seqs, got, dtype, f"first tokens together {dtype}")
    eng = make_engine(d, dtype)
    for r, ids in seqs.items():
        got = run_steps(eng, [([(r, ids[:1], [0])], [])] + [([(r, [t], [0])], []) for t in ids[1:]] + [([], [r])][:0])
        check(d, {r: ids}, got, dtype, f"first tokens one by one {dtype}")
        eng.release(r)


# ----------------------------------------------------------------------------------------------- kernels with made-up inputs
def paged(keys, values, page_size, n_pages, order):
    """Key and value pages [page, 1, slot, size] of one request whose logical pages lie at `order` in the pool."""
    T = keys.shape[0]
    kp = torch.zeros((n_pages, 1, page_size, keys.shape[1]), dtype=keys.dtype, device="cuda")
    vp = torch.zeros((n_pages, 1, page_size, values.shape[1]), dtype=keys.dtype, device="cuda")
    for t in range(T):
        kp[order[t // page_size], 0, t % page_size] = keys[t]
        vp[order[t // page_size], 0, t % page_size] = values[t]
    return kp, vp


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_far_key_and_every_distance_of_the_bias(dtype):
    """One query head over 700 keys in pages of 16 scattered over the pool, values of a size of their own.  A single key
    far back is made to dominate (its score stands out by 12), at a page's border and in the middle of one; then the
    bias alone decides: a table whose row for one distance stands out, for distances just inside and just beyond the
    table's end (all longer distances share the last row)."""
    from gibbs_amd import ops
    rng = np.random.default_rng(0)
    T, hd, vd, ps = 700, 24, 40, 16
    n_pages = 64
    order = rng.permutation(n_pages)[:-(-T // ps)].tolist()
    keys = torch.tensor(rng.normal(size=(T, hd)) * 0.1, dtype=dtype, device="cuda")
    values = torch.tensor(rng.normal(size=(T, vd)), dtype=dtype, device="cuda")
    table = torch.tensor([order], dtype=torch.int32, device="cuda")
    rows = torch.tensor([T - 1, T - 2, 300], dtype=torch.int32, device="cuda")
    row_req = torch.zeros(3, dtype=torch.int32, device="cuda")
    q = torch.tensor(rng.normal(size=(3, hd)) * 0.1, dtype=dtype, device="cuda")
    flat = torch.zeros((50, 1), dtype=torch.float32, device="cuda")
    for far in (15, 16, 17, 200, 0):
        k2 = keys.clone()
        k2[far] = (q[0].float() / q[0].float().norm() ** 2 * 12.0).to(dtype)     # q0 . k = 12
        kp, vp = paged(k2, values, ps, n_pages, order)
        out = ops.attention_plain(q, 3, 1, 1, hd, kp, vp, table, 1, rows, row_req, 1.0, bias=flat).float().cpu().numpy()
        s = (q.float() @ k2.float().T).cpu().numpy()
        for i, p in enumerate(rows.tolist()):
            w = np.exp(s[i, :p + 1] - s[i, :p + 1].max())
            want = (w / w.sum()) @ values.float().cpu().numpy()[:p + 1]
            assert np.abs(out[i] - want).max() <= (2e-5 if dtype == torch.float32 else 2e-2), (far, i)
        assert np.abs(out[0] - values[far].float().cpu().numpy()).max() < 0.05, f"the far key {far} does not dominate"
    kp, vp = paged(keys * 0, values, ps, n_pages, order)
    for length, hot in ((50, 48), (50, 49), (50, 7), (3, 2), (3, 1)):
        bias = torch.zeros((length, 1), dtype=torch.float32, device="cuda")
        bias[hot, 0] = 14.0
        out = ops.attention_plain(q, 3, 1, 1, hd, kp, vp, table, 1, rows, row_req, 1.0, bias=bias).float().cpu().numpy()
        for i, p in enumerate(rows.tolist()):
            dist = np.minimum(p - np.arange(p + 1), length - 1)
            w = np.exp(np.where(dist == hot, 14.0, 0.0))
            want = (w / w.sum()) @ values.float().cpu().numpy()[:p + 1]
            assert np.abs(out[i] - want).max() <= (2e-5 if dtype == torch.float32 else 2e-2), (length, hot, i)


def test_unit_norm_temperature_and_cache_write():
    from gibbs_amd import ops
    rng = np.random.default_rng(1)
    nh, nkv, hd, vd, ps = 4, 2, 24, 40, 16
    pos = torch.tensor([0, 7, 8, 15, 16, 31, 250], dtype=torch.int32, device="cuda")
    n = pos.numel()
    rows = torch.tensor(rng.normal(size=(n, (nh + nkv) * hd + nkv * vd)), dtype=torch.float32, device="cuda")
    before = rows.cpu().numpy().copy()
    kp = torch.zeros((20, nkv, ps, hd), dtype=torch.float32, device="cuda")
    vp = torch.zeros((20, nkv, ps, vd), dtype=torch.float32, device="cuda")
    table = torch.arange(19, -1, -1, dtype=torch.int32, device="cuda").view(1, 20).contiguous()
    ops.qk_unit_kv(rows, nh, nkv, hd, vd, kpages=kp, vpages=vp, table=table, pos=pos, row_req=torch.zeros(n, dtype=torch.int32, device="cuda"),
                   eps=1e-5, unit=True, temp_coef=0.7, temp_every=8)
    after = rows.cpu().numpy()
    for i, p in enumerate(pos.tolist()):
        heads = before[i, :(nh + nkv) * hd].reshape(nh + nkv, hd)
        unit = heads / np.sqrt((heads ** 2).mean(-1, keepdims=True) + 1e-5)
        unit[:nh] *= 1.0 + 0.7 * np.log((p + 1) // 8 + 1.0)             # positions 7 and 8, 15 and 16 lie on both sides of a step
        assert np.allclose(after[i, :(nh + nkv) * hd].reshape(nh + nkv, hd), unit, rtol=2e-6, atol=1e-6)
        page = 19 - p // ps
        assert np.allclose(kp[page, :, p % ps].cpu().numpy(), unit[nh:], rtol=2e-6, atol=1e-6)
        assert np.array_equal(vp[page, :, p % ps].cpu().numpy().reshape(-1), before[i, (nh + nkv) * hd:])


def test_heads_of_unequal_sizes_are_stored_padded_in_bfloat16_only(dirs):
    """Keys of 24 and values of 40 (model P) run as heads of 48 in a bfloat16 engine (zeros behind each head's channels, in
    the projections and in the pages: what the matrix-core attention kernels take) and at their own sizes in 32-bit; the
    logits of both are held against the plain implementation by the tests above."""
    for dtype, sizes in (("bfloat16", (48, 48)), ("float32", (24, 40))):
        eng = make_engine(dirs["P"], dtype)
        left = eng.model.blocks[1].left
        assert left.stored_dims() == sizes and (left.head_dim, left.v_head_dim) == (24, 40)
        group = eng.cache.group_needs.index(left.cache_need())
        assert eng.device_cache.kpages[group].shape[-1] == sizes[0] and eng.device_cache.vpages[group].shape[-1] == sizes[1]
        assert left.w_qkv.shape[0] == 6 * sizes[0] + 3 * sizes[0] + 3 * sizes[1] and left.w_out.shape[1] == 6 * sizes[1]
        if dtype == "bfloat16":
            q = left.w_qkv[:6 * 48].view(6, 48, -1)
            assert float(q[:, 24:].abs().max()) == 0.0 and float(left.w_out.view(-1, 6, 48)[:, :, 40:].abs().max()) == 0.0


def test_unit_norm_of_padded_heads_divides_by_the_true_size():
    from gibbs_amd import ops
    rng = np.random.default_rng(8)
    nh, nkv, true, pad = 2, 1, 24, 32
    rows = np.zeros((3, (nh + 2 * nkv) * pad), dtype=np.float32)
    rows.reshape(3, nh + 2 * nkv, pad)[:, :, :true] = rng.normal(size=(3, nh + 2 * nkv, true))
    dev = torch.tensor(rows, device="cuda")
    pos = torch.tensor([0, 1, 2], dtype=torch.int32, device="cuda")
    ops.qk_unit_kv(dev, nh, nkv, pad, pad, kpages=None, vpages=None, table=None, pos=pos, row_req=torch.zeros(3, dtype=torch.int32, device="cuda"),
                   eps=1e-6, unit=True, norm_dim=true)
    heads = rows.reshape(3, nh + 2 * nkv, pad)[:, :nh + nkv]
    want = heads / np.sqrt((heads[:, :, :true] ** 2).mean(-1, keepdims=True) + 1e-6)
    got = dev.cpu().numpy().reshape(3, nh + 2 * nkv, pad)[:, :nh + nkv]
    assert np.allclose(got, want, rtol=2e-6, atol=1e-6) and np.abs(got[:, :, true:]).max() == 0.0


@pytest.mark.parametrize("per_channel", [False, True])
def test_delta_rule_keeps_an_old_write_through_portions_and_slots(per_channel):
    """A value written at the first token with a key of its own is read back 500 tokens later (no decay on that key's
    channel, random writes on the others in between), whole, in portions of 1, 2, 7 and 64 tokens, and in a slot that
    another request used before; the kernel's result equals the plain rule's."""
    from gibbs_amd import ops
    rng = np.random.default_rng(2)
    T, H, G, D, V = 501, 4, 2, 20, 24
    k = rng.normal(size=(T, G, D)); k[:, :, 0] = 0; k[0] = 0; k[0, :, 0] = 1
    k /= np.linalg.norm(k, axis=-1, keepdims=True)
    q = rng.normal(size=(T, G, D)) * 0.2; q[-1] = 0; q[-1, :, 0] = 1
    v = rng.normal(size=(T, H, V))
    beta = rng.uniform(0.2, 1.0, size=(T, H)); beta[0] = 1
    decay = rng.uniform(0.8, 1.0, size=(T, H, D) if per_channel else (T, H))
    if per_channel:
        decay[:, :, 0] = 1
    want = np.stack([Z.delta_rule(q[:, h // 2], k[:, h // 2], v[:, h], beta[:, h], decay[:, h]) for h in range(H)], axis=1)
    if per_channel:
        assert np.allclose(want[-1], v[0]), "the plain rule itself must recall the first write"
    dev = lambda a: torch.tensor(a.reshape(T, -1), dtype=torch.float32, device="cuda")
    dq, dk, dv, db, dd = dev(q), dev(k), dev(v), dev(beta), dev(decay)
    state = torch.zeros((3, H, D, V), dtype=torch.float32, device="cuda")
    for slot, sizes in ((1, [T]), (2, [1, 2, 7, 64, 1, 1, 300, 2]), (1, [64, 63, 2])):
        state[slot].zero_()                       # (a slot is cleared when a request takes it)
        at, outs, i = 0, [], 0
        while at < T:
            n = min(sizes[i % len(sizes)], T - at)
            cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
            outs.append(ops.delta_rule(dq[at:at + n].contiguous(), dk[at:at + n].contiguous(), dv[at:at + n].contiguous(),
                                       db[at:at + n].contiguous(), dd[at:at + n].contiguous(), state, cu,
                                       torch.tensor([slot], dtype=torch.int32, device="cuda"), H, G))
            at += n; i += 1
        got = torch.cat(outs).cpu().numpy().reshape(T, H, V)
        assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max(), (slot, sizes)


@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("lens,H,G,D,V,strength", [([1], 2, 1, 16, 16, 1), ([64], 4, 2, 64, 48, 1), ([65, 1, 17], 2, 2, 128, 128, 1), ([130, 63], 2, 1, 48, 32, 1),
                                                   ([200], 3, 3, 96, 16, 1), ([300], 2, 2, 64, 64, 300), ([300], 2, 2, 128, 32, 1e-6)])
def test_delta_rule_in_chunks_equals_the_walk(lens, H, G, D, V, strength, per_channel):
    """Chunks of 64 tokens against the rule token by token in 64 bits: whole chunks, remainders, requests side by side in scattered
    slots, decays that forget within a token and decays that forget nothing.  A read-out is a sum over D products of a state that is
    itself a sum over the tokens; 32 roundings of 2^-24 stand for both (measured: 5)."""
    from gibbs_amd import ops
    rng = np.random.default_rng(sum(lens) + D)
    n = sum(lens)
    q, k = rng.normal(size=(n, G, D)), rng.normal(size=(n, G, D))
    k[1:] = 0.6 * k[1:] + 0.4 * k[:-1]
    q, k = q / np.linalg.norm(q, axis=-1, keepdims=True) * D ** -0.5, k / np.linalg.norm(k, axis=-1, keepdims=True)
    v, beta = rng.normal(size=(n, H, V)), rng.uniform(0, 1, size=(n, H))
    decay = np.exp(-strength * np.exp(rng.normal(size=(n, H, D) if per_channel else (n, H)) - 3))
    q, k, v, beta, decay = (x.astype(np.float32).astype(np.float64) for x in (q, k, v, beta, decay))
    dev = lambda a: torch.tensor(a.reshape(n, -1), dtype=torch.float32, device="cuda")
    cu = np.concatenate([[0], np.cumsum(lens)])
    slots = rng.permutation(len(lens) + 2)[:len(lens)]
    start = rng.normal(size=(len(lens) + 2, H, D, V)).astype(np.float32)
    state = torch.tensor(start, device="cuda")
    got = ops.delta_rule(dev(q), dev(k), dev(v), dev(beta), dev(decay), state, torch.tensor(cu, dtype=torch.int32, device="cuda"),
                         torch.tensor(slots, dtype=torch.int32, device="cuda"), H, G, chunks=True).cpu().numpy().reshape(n, H, V)
    after = state.cpu().numpy()
    for i, slot in enumerate(slots):
        at = slice(cu[i], cu[i + 1])
        for h in range(H):
            S, want = start[slot, h].astype(np.float64), []
            for t in range(cu[i], cu[i + 1]):
                S = S * (decay[t, h][:, None] if per_channel else decay[t, h])
                S = S + np.outer(k[t, h // (H // G)], beta[t, h] * (v[t, h] - S.T @ k[t, h // (H // G)]))
                want.append(S.T @ q[t, h // (H // G)])
            for mine, true in ((got[at, h], np.stack(want)), (after[slot, h], S)):
                assert np.linalg.norm(mine - true) <= 32 * 2.0 ** -24 * np.linalg.norm(true), (i, h)
    others = [s for s in range(len(lens) + 2) if s not in slots]
    assert np.array_equal(after[others], start[others])


# decays: moderate, hardly any, all hard, hard ones among gentle ones, and resets among gentle ones
DECAYS = {"moderate": lambda r, shape: np.exp(-np.exp(r.normal(size=shape) - 3)), "slow": lambda r, shape: np.exp(-1e-6 * np.exp(r.normal(size=shape))),
          "hard": lambda r, shape: np.exp(-np.minimum(300 * np.exp(r.normal(size=shape) - 3), 87)),
          "mixed": lambda r, shape: np.where(r.random(shape) < 0.3, 2.0 ** -28, 2.0 ** -0.02),
          "resets": lambda r, shape: np.where(r.random(shape) < 0.05, 2.0 ** -60, 2.0 ** -0.01)}


@pytest.mark.parametrize("kind", sorted(DECAYS))
@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("D", [64, 128])
def test_delta_rule_in_chunks_is_as_exact_as_the_walk(D, per_channel, kind):
    """The chunks' error against 64 bits is the walk's or less, for read-outs and state; a quarter more is allowed for the sample (measured: at most
    1.07 times the walk's, mostly 0.4 to 0.95).  Resets come with writes that are nearly nothing, so that what is left behind them counts."""
    from gibbs_amd import ops
    rng = np.random.default_rng(D)
    n, H, V = 256, 4, 64
    q, k = rng.normal(size=(n, H, D)), rng.normal(size=(n, H, D))
    k[1:] = 0.6 * k[1:] + 0.4 * k[:-1]
    q, k = q / np.linalg.norm(q, axis=-1, keepdims=True) * D ** -0.5, k / np.linalg.norm(k, axis=-1, keepdims=True)
    v, beta = rng.normal(size=(n, H, V)), rng.uniform(0, 1, size=(n, H))
    decay = DECAYS[kind](rng, (n, H, D) if per_channel else (n, H))
    if kind == "resets":
        beta = np.where(rng.random((n, H)) < 0.5, 1e-6, beta)
    q, k, v, beta, decay = (x.astype(np.float32).astype(np.float64) for x in (q, k, v, beta, decay))
    start = rng.normal(size=(1, H, D, V)).astype(np.float32)
    S, want = start[0].astype(np.float64), []
    for t in range(n):
        S = S * (decay[t][:, :, None] if per_channel else decay[t][:, None, None])
        S = S + k[t][:, :, None] * (beta[t][:, None] * (v[t] - np.einsum("hdv,hd->hv", S, k[t])))[:, None, :]
        want.append(np.einsum("hdv,hd->hv", S, q[t]))
    dev = lambda a: torch.tensor(a.reshape(n, -1), dtype=torch.float32, device="cuda")
    cu, slot = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([0, n], [0]))
    far = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)
    errors = []
    for chunks in (False, True):
        state = torch.tensor(start, device="cuda")
        got = ops.delta_rule(dev(q), dev(k), dev(v), dev(beta), dev(decay), state, cu, slot, H, H, chunks=chunks)
        errors.append((far(got.cpu().numpy().reshape(n, H, V), np.stack(want)), far(state[0].cpu().numpy(), S)))
    for walk, mine in zip(*errors):
        assert mine <= 1.25 * walk, errors


@pytest.mark.parametrize("what", ["q", "k", "v", "beta", "decay"])
@pytest.mark.parametrize("per_channel", [False, True])
def test_delta_rule_in_chunks_keeps_a_value_that_is_not_finite_behind_it(per_channel, what):
    """The read-outs in front of such a value are what they are without it, to the bit, and another request's too; from it on what the walk leaves not
    finite is not finite here either, and the rest (a column of v, a row of q) agrees with the walk to rounding, the state likewise."""
    from gibbs_amd import ops
    rng = np.random.default_rng(5)
    n, H, D, V, lens = 200, 2, 48, 32, [150, 50]
    q, k = rng.normal(size=(n, H, D)), rng.normal(size=(n, H, D))
    q, k = q / np.linalg.norm(q, axis=-1, keepdims=True), k / np.linalg.norm(k, axis=-1, keepdims=True)
    values = {"q": q, "k": k, "v": rng.normal(size=(n, H, V)), "beta": rng.uniform(0, 1, size=(n, H)),
              "decay": rng.uniform(0.8, 1, size=(n, H, D) if per_channel else (n, H))}
    start = torch.tensor(rng.normal(size=(2, H, D, V)), dtype=torch.float32, device="cuda")
    cu, slot = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([0, 150, 200], [1, 0]))
    def run(x, chunks):
        dev = {name: torch.tensor(a.reshape(n, -1), dtype=torch.float32, device="cuda") for name, a in x.items()}
        state = start.clone()
        return ops.delta_rule(*(dev[name] for name in ("q", "k", "v", "beta", "decay")), state, cu, slot, H, H, chunks=chunks).reshape(n, H, V), state
    clean, _ = run(values, True)
    for t, bad in ((7, np.nan), (77, np.inf), (64, -np.inf), (149, np.nan)):
        x = {name: a.copy() for name, a in values.items()}
        x[what][(t, 1) + (3,) * (x[what].ndim - 2)] = bad
        (got, mine), (want, state) = run(x, True), run(x, False)
        assert bool((got[:t] == clean[:t]).all() and (got[:, 0] == clean[:, 0]).all() and (got[150:] == clean[150:]).all()), (t, bad)
        assert not want[t, 1].isfinite().all()
        for a, b in ((got, want), (mine, state)):
            assert bool((a.isfinite() == b.isfinite()).all()), (t, bad)
            assert float((a - b)[b.isfinite()].norm()) <= 32 * 2.0 ** -24 * float(b[b.isfinite()].norm())


@pytest.mark.parametrize("lead", [1, 3])
def test_rules_in_chunks_from_a_request_on(lead):
    """`cu` and `slot` from a request on, its rows addressed by the step's: read-outs and states are those of the requests alone, to the bit, and
    rows and slots in front are left as they are."""
    from gibbs_amd.ops.lib import call, library, ptr, stream
    lens, H, D = [1] * lead + [130, 5], 2, 64
    n, C, R, rest = sum(lens), H * D, len(lens), sum(lens) - lead
    g = torch.Generator(device="cuda").manual_seed(lead)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    unit = lambda: torch.nn.functional.normalize(rnd(n, H, D), dim=-1).reshape(n, C)
    cu, slot = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in (np.concatenate([[0], np.cumsum(lens)]), range(R)))
    alone = cu[lead:] - lead
    q, k, v, beta, decay, start = unit(), unit(), rnd(n, C), torch.rand((n, H), generator=g, device="cuda"), 1 - 0.1 * torch.rand((n, C), generator=g, device="cuda"), rnd(R, H, D, D)
    mark = 7.0
    results = []
    for c, skip in ((cu[lead:], 0), (alone, lead)):
        state, out = start.clone(), torch.full((n, C), mark, device="cuda")
        work = torch.empty(library().gibbs_delta_chunks_workspace(rest, 2, H, D, D), device="cuda")
        rows = [x[skip:] for x in (q, k, v, beta, decay, out)]
        call("gibbs_delta_chunks", ptr(rows[0]), ptr(rows[1]), C, ptr(rows[2]), C, ptr(rows[3]), ptr(rows[4]), 1, ptr(state), state.stride(0), ptr(c), ptr(slot[lead:]),
             ptr(rows[5]), ptr(work), rest, 2, H, H, D, D, stream())
        results.append((out, state))
    rows, z, bias, bonus, gain = torch.stack([q, k, v, rnd(n, C)]), rnd(n, C), rnd(C) - 3, rnd(C), rnd(C)
    for c, skip in ((cu[lead:], 0), (alone, lead)):
        state, out = start.clone(), torch.full((n, C), mark, device="cuda")
        work = torch.empty(library().gibbs_decayed_outer_chunks_workspace(rest, 2, H, D), device="cuda")
        call("gibbs_decayed_outer_chunks", ptr(rows[0, skip:]), C, n * C, 2 * n * C, 3 * n * C, ptr(z[lead:]), ptr(bias), ptr(bonus), ptr(gain), 1e-6, ptr(state),
             state.stride(0), ptr(c), ptr(slot[lead:]), ptr(out[skip:]), ptr(work), 0, rest, 2, H, D, stream())
        results.append((out, state))
    for (out, state), (other, other_state) in (results[:2], results[2:]):
        assert torch.equal(out, other) and torch.equal(state, other_state)
        assert bool((out[:lead] == mark).all() and out[lead:].isfinite().all() and (out[lead:] != mark).any()) and torch.equal(state[:lead], start[:lead])
        assert not torch.equal(state[lead:], start[lead:])


@pytest.mark.parametrize("lens,H", [([1100, 70], 64), ([64 * 65536 + 1], 1)])
def test_delta_rule_in_chunks_of_long_prompts(lens, H):
    """More chunks than the workspace holds at once, two requests across its border, and more than a launch's second dimension could be: the
    workspace stays below 256 MB, and what comes out is the walk's to rounding (32 of 2^-24, as above)."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import library
    assert all(library().gibbs_delta_chunks_workspace(rows, 3, 16, 128, 128) * 4 <= 2 ** 28 for rows in (100, 16384, 2 ** 30))
    n, D = sum(lens), 16
    g = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    q, k = (torch.nn.functional.normalize(rnd(n, H, D), dim=-1).reshape(n, -1) for _ in range(2))
    v, beta, decay, start = rnd(n, H * D), torch.rand((n, H), generator=g, device="cuda"), 1 - 0.1 * torch.rand((n, H), generator=g, device="cuda"), rnd(len(lens), H, D, D)
    cu, slot = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in (np.concatenate([[0], np.cumsum(lens)]), range(len(lens))))
    states = [start.clone(), start.clone()]
    walk, mine = (ops.delta_rule(q, k, v, beta, decay, s, cu, slot, H, H, chunks=c) for s, c in zip(states, (False, True)))
    for got, want in [(mine, walk)] + list(zip(states[1], states[0])):
        assert (got - want).norm() <= 32 * 2.0 ** -24 * want.norm()
    assert (mine - walk)[-64:].norm() <= 32 * 2.0 ** -24 * walk[-64:].norm()


def test_decayed_outer_rule_two_requests_side_by_side():
    from gibbs_amd import ops
    rng = np.random.default_rng(3)
    H, D = 3, 12
    lens = [37, 5]
    r, k, v = (rng.normal(size=(sum(lens), H, D)) * 0.5 for _ in range(3))
    w = rng.uniform(0.5, 1.0, size=(sum(lens), H, D)); w[:, :, 1] = 1.0          # channel 1 never forgets
    bonus = rng.normal(size=(H, D))
    want = np.zeros((sum(lens), H, D))
    at = 0
    for n in lens:
        for h in range(H):
            S = np.zeros((D, D))
            for t in range(at, at + n):
                kv = np.outer(k[t, h], v[t, h])
                want[t, h] = (S + bonus[h][:, None] * kv).T @ r[t, h]
                S = w[t, h][:, None] * S + kv
        at += n
    dev = lambda a: torch.tensor(a.reshape(a.shape[0], -1), dtype=torch.float32, device="cuda")
    state = torch.zeros((4, H, D, D), dtype=torch.float32, device="cuda")
    slot = torch.tensor([3, 0], dtype=torch.int32, device="cuda")
    dr, dk, dv, dw = dev(r), dev(k), dev(v), dev(w)
    # first 30 + 2 tokens in one call, the rest in another (rows of the two requests side by side)
    idx1 = list(range(30)) + [37, 38]
    idx2 = list(range(30, 37)) + [39, 40, 41]
    outs = {}
    for idx, cu in ((idx1, [0, 30, 32]), (idx2, [0, 7, 10])):
        sel = torch.tensor(idx, device="cuda")
        o = ops.decayed_outer_rule(dr[sel].contiguous(), dk[sel].contiguous(), dv[sel].contiguous(), dw[sel].contiguous(),
                                   torch.tensor(bonus, dtype=torch.float32, device="cuda"), state,
                                   torch.tensor(cu, dtype=torch.int32, device="cuda"), slot, H)
        for i, t in enumerate(idx):
            outs[t] = o[i].cpu().numpy().reshape(H, D)
    got = np.stack([outs[t] for t in range(sum(lens))])
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("n,H,G,D,V", [(1, 1, 1, 4, 4), (8, 4, 2, 128, 128), (3, 2, 2, 20, 24), (2, 3, 1, 64, 256), (2, 2, 1, 256, 64), (5, 2, 2, 12, 512)])
def test_delta_step_equals_its_parts(n, H, G, D, V, per_channel, dtype):
    """One row per request in one kernel against the row preparation, the walk and the gated norm one after the other: the same arithmetic
    but for the order of two sums over D products and of one over V squares (32-bit: 32 roundings of 2^-24; the bfloat16 result adds its own)."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, library, ptr, stream
    g = torch.Generator().manual_seed(n + D)
    rnd = lambda *shape, t=torch.float32: torch.randn(*shape, generator=g).to(t).cuda()
    kind, C, eps, unit_eps, scale = (0 if dtype == torch.float32 else 1), 2 * G * D + H * V, 1e-6, 1e-6, D ** -0.5
    qkv, braw, araw, gate = rnd(n, C), rnd(n, H, t=dtype), rnd(n, H, t=dtype), rnd(n, H * V, t=dtype)
    channel = rnd(n, H * D) if per_channel else None
    dt_bias, a_log, gain = rnd(H * D if per_channel else H) - 3, rnd(H) * 0.5, 1 + 0.1 * rnd(V)
    state = rnd(n + 2, H, D, V)
    slot = torch.randperm(n + 2, generator=g)[:n].to(torch.int32).cuda()
    mine, y = state.clone(), torch.empty((n, H * V), dtype=dtype, device="cuda")
    assert library().gibbs_delta_step_takes(D, V)
    decays = (None if channel is None else ptr(channel), ptr(dt_bias), ptr(a_log))
    call("gibbs_delta_step", ptr(qkv), C, ptr(braw), ptr(araw), H, kind, *decays, ptr(gate), H * V, 1, ptr(gain), eps, ptr(mine),
         mine.stride(0), ptr(slot), ptr(y), n, G, H, D, V, scale, unit_eps, stream())
    rows, beta, decay = qkv.clone(), torch.empty((n, H), device="cuda"), torch.empty((n, H * D if per_channel else H), device="cuda")
    call("gibbs_delta_prep", ptr(rows), ptr(rows[:, G * D:]), C, ptr(braw), ptr(araw), H, kind, *decays, ptr(beta), ptr(decay), n, G, H, D, scale, unit_eps, stream())
    o = ops.delta_rule(rows[:, :G * D].contiguous(), rows[:, G * D:2 * G * D].contiguous(), rows[:, 2 * G * D:].contiguous(), beta, decay, state,
                       torch.arange(n + 1, dtype=torch.int32, device="cuda"), slot, H, G)
    want = torch.empty_like(y)
    call("gibbs_head_norm_gate", ptr(o), ptr(gain), V, ptr(gate), H * V, ptr(want), kind, n, H, V, eps, 1, stream())
    far = lambda a, b: ((a.double() - b.double()).norm() / b.double().norm()).item()
    assert far(mine, state) <= 32 * 2.0 ** -24, far(mine, state)
    assert far(y, want) <= 32 * 2.0 ** -24 + (2.0 ** -8 if kind else 0), far(y, want)


@pytest.mark.parametrize("V", [4, 32, 36, 64, 100, 128, 256, 512])
def test_delta_step_sums_a_heads_squares_in_one_order(V):
    """Empty states, keys and queries of one channel and a full write leave the values themselves as the read-out, so that what comes out is their norm
    alone: a lane's own square fused with the rounded one 32 lanes on, lanes by halves, waves in turn, to the bit."""
    from gibbs_amd.ops.lib import call, ptr, stream
    n, D, eps = 200, 4, 1e-6
    g = torch.Generator().manual_seed(V)
    v = torch.randn(n, V, generator=g)
    one = torch.zeros(n, D)
    one[:, 0] = 1.0
    qkv, sure = torch.cat([one, one, v], 1).cuda(), torch.full((n, 1), 200.0, device="cuda")      # (a sigmoid of 1: beta and the gate)
    zero, gain, gate = torch.zeros(1, device="cuda"), torch.ones(V, device="cuda"), torch.full((n, V), 200.0, device="cuda")
    state, slot = torch.zeros(n, 1, D, V, device="cuda"), torch.arange(n, dtype=torch.int32, device="cuda")
    y = torch.empty(n, V, device="cuda")
    call("gibbs_delta_step", ptr(qkv), 2 * D + V, ptr(sure), ptr(sure), 1, 0, None, ptr(zero), ptr(zero), ptr(gate), V, 1, ptr(gain), eps, ptr(state),
         state.stride(0), ptr(slot), ptr(y), n, 1, 1, D, V, 1.0, 0.0, stream())
    f32, f64 = np.float32, np.float64
    x = np.zeros((n, 8, 64), f32)
    x.reshape(n, 512)[:, :V] = v.numpy()
    far = np.roll(x, 32, axis=2)
    lanes = (x.astype(f64) ** 2 + (far * far).astype(f64)).astype(f32)[:, :, :32]
    for half in (16, 8, 4, 2, 1):
        lanes = lanes + lanes[:, :, np.arange(32) ^ half]
    total = np.zeros(n, f32)
    for w in range(8):
        total = total + lanes[:, w, 0]
    scale = f32(1) / np.sqrt(total / f32(V) + f32(eps))
    assert np.array_equal(y.cpu().numpy(), v.numpy() * scale[:, None])


@pytest.mark.parametrize("how", ["chunks", "rows"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens,H,D,shift", [([1], 2, 16, 0), ([1, 1, 1], 2, 64, -3), ([64], 3, 64, -3), ([65, 1, 17], 2, 64, -3), ([130, 63], 2, 24, 1), ([200], 2, 32, 4),
                                            ([96], 1, 12, -8)])
def test_decayed_outer_rule_with_norm_and_gate(lens, H, D, shift, dtype, how):
    """Chunks of 64 tokens, and row by row, with the decays, the heads' norm and the gate, against the rule token by token in 64 bits: whole chunks and
    remainders, requests in scattered slots, head sizes that are no multiple of 16, decays that forget at once (shift 4) and hardly
    ever (-8).  32-bit: 64 roundings of 2^-24 for the sums over channels and tokens and the factors that decays are split into; the
    bfloat16 result adds its own rounding."""
    from gibbs_amd.ops.lib import call, library, ptr, stream
    rng = np.random.default_rng(sum(lens) + D)
    n, C, eps = sum(lens), H * D, 1e-6
    q, k, v, g = (torch.tensor(rng.normal(size=(n, C)), dtype=dtype, device="cuda") for _ in range(4))
    z, bias, bonus = rng.normal(size=(n, C)), rng.normal(size=C) * 0.5 + shift, rng.normal(size=C)
    gain = 1 + 0.1 * rng.normal(size=C)
    z, bias, bonus, gain = (torch.tensor(x, dtype=torch.float32, device="cuda") for x in (z, bias, bonus, gain))
    rows = torch.stack([q, k, v, g])
    slots = rng.permutation(len(lens) + 2)[:len(lens)]
    start = rng.normal(size=(len(lens) + 2, H, D, D)).astype(np.float32)
    state, out = torch.tensor(start, device="cuda"), torch.empty((n, C), dtype=dtype, device="cuda")
    cu = np.concatenate([[0], np.cumsum(lens)])
    dcu, dslot = torch.tensor(cu, dtype=torch.int32, device="cuda"), torch.tensor(slots, dtype=torch.int32, device="cuda")
    operands = (ptr(rows), C, n * C, 2 * n * C, 3 * n * C, ptr(z), ptr(bias), ptr(bonus), ptr(gain), eps, ptr(state), state.stride(0))
    kind = 0 if dtype == torch.float32 else 1
    if how == "chunks":
        assert library().gibbs_decayed_outer_chunks_take(D)
        work = torch.empty(library().gibbs_decayed_outer_chunks_workspace(n, len(lens), H, D), dtype=torch.float32, device="cuda")
        call("gibbs_decayed_outer_chunks", *operands, ptr(dcu), ptr(dslot), ptr(out), ptr(work), kind, n, len(lens), H, D, stream())
    else:
        assert library().gibbs_decayed_outer_rows_take(D)
        call("gibbs_decayed_outer_rows", *operands, None if n == len(lens) else ptr(dcu), ptr(dslot), ptr(out), kind, len(lens), H, D, stream())
    q, k, v, g, z, bias, bonus, gain = (x.double().cpu().numpy() for x in (q, k, v, g, z, bias, bonus, gain))
    decay = np.exp(-np.exp(z + bias)).reshape(n, H, D)
    got, after = out.double().cpu().numpy(), state.cpu().numpy()
    tol = 64 * 2.0 ** -24 + (2.0 ** -8 if dtype == torch.bfloat16 else 0)
    q, k, v = (x.reshape(n, H, D) for x in (q, k, v))
    for i, slot in enumerate(slots):
        want = np.zeros((lens[i], H, D))
        for h in range(H):
            S = start[slot, h].astype(np.float64)
            for t in range(cu[i], cu[i + 1]):
                kv = np.outer(k[t, h], v[t, h])
                want[t - cu[i], h] = (S + bonus.reshape(H, D)[h][:, None] * kv).T @ q[t, h]
                S = decay[t, h][:, None] * S + kv
            assert np.linalg.norm(after[slot, h] - S) <= 64 * 2.0 ** -24 * np.linalg.norm(S), (i, h)
        want = want / np.sqrt((want ** 2).mean(-1, keepdims=True) + eps)
        want = want.reshape(lens[i], C) * gain * (g / (1 + np.exp(-g)))[cu[i]:cu[i + 1]]
        assert np.linalg.norm(got[cu[i]:cu[i + 1]] - want) <= tol * np.linalg.norm(want), i
    others = [s for s in range(len(lens) + 2) if s not in slots]
    assert np.array_equal(after[others], start[others])


def test_decayed_outer_rows_of_as_many_requests_as_the_walk_takes():
    """65,537 requests of one token in one call: the last ones' read-outs and states are those of a call of their own, to the bit; a step that long
    never takes the rules in chunks, whose launches have a dimension for the requests."""
    from gibbs_amd.ops.lib import call, library, ptr, stream
    assert not any(library().gibbs_rule_chunked(t, 65536 + 2000, 65536, 2000, 1, 16, 16) for t in (0, 1))
    n, D, last = 65537, 4, 5
    g = torch.Generator(device="cuda").manual_seed(0)
    rows, z, bias, bonus, gain = (torch.randn(s, generator=g, device="cuda") for s in ((4, n, D), (n, D), D, D, D))
    start, slot = torch.randn((n, 1, D, D), generator=g, device="cuda"), torch.arange(n, dtype=torch.int32, device="cuda")
    results = []
    for first in (0, n - last):
        state, out = start.clone(), torch.zeros((n, D), device="cuda")
        call("gibbs_decayed_outer_rows", ptr(rows[0, first:]), D, n * D, 2 * n * D, 3 * n * D, ptr(z[first:]), ptr(bias), ptr(bonus), ptr(gain), 1e-6, ptr(state),
             state.stride(0), None, ptr(slot[first:]), ptr(out[first:]), 0, n - first, 1, D, stream())
        results.append((out[-last:], state[-last:]))
    assert all(torch.equal(a, b) and a.isfinite().all() and (a != 0).any() for a, b in zip(*results))


@pytest.mark.parametrize("kind", sorted(DECAYS))
@pytest.mark.parametrize("D", [24, 64, 96])
def test_decayed_outer_rule_in_chunks_is_as_exact_as_the_walk(D, kind):
    """As for the delta rule: the error of normed read-outs and state against 64 bits is the walk's or less, a quarter more allowed for the sample
    (measured: 0.2 to 1.06 times the walk's)."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, library, ptr, stream
    rng = np.random.default_rng(D)
    n, H, eps = 256, 4, 1e-6
    C = H * D
    f32 = lambda x: np.asarray(x, dtype=np.float32)
    rows = f32(rng.normal(size=(4, n, C)))
    bias = f32(rng.normal(size=C))
    z = f32(np.log(-np.log(DECAYS[kind](rng, (n, C)))) - bias)
    bonus, gain, start = f32(0.5 * rng.normal(size=C)), f32(1 + 0.1 * rng.normal(size=C)), f32(rng.normal(size=(1, H, D, D)))
    q, k, v, g = (x.astype(np.float64).reshape(n, H, D) for x in rows)
    decay, u = np.exp(-np.exp(z.astype(np.float64) + bias)).reshape(n, H, D), bonus.astype(np.float64).reshape(H, D)
    S, want = start[0].astype(np.float64), []
    for t in range(n):
        y = np.einsum("hdv,hd->hv", S, q[t]) + (q[t] * u * k[t]).sum(-1, keepdims=True) * v[t]
        S = decay[t][:, :, None] * S + k[t][:, :, None] * v[t][:, None, :]
        want.append(y / np.sqrt((y ** 2).mean(-1, keepdims=True) + eps) * gain.reshape(H, D) * (g[t] / (1 + np.exp(-g[t]))))
    rows, z, bias, bonus, gain = (torch.tensor(x, device="cuda") for x in (rows, z, bias, bonus, gain))
    cu, slot = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([0, n], [0]))
    states, outs = [torch.tensor(start, device="cuda") for _ in range(2)], [torch.empty((n, C), device="cuda") for _ in range(2)]
    read = ops.decayed_outer_rule(rows[0], rows[1], rows[2], torch.exp(-torch.exp(z + bias)), bonus.reshape(H, D), states[0], cu, slot, H)
    call("gibbs_head_norm_gate", ptr(read), ptr(gain), C, ptr(rows[3]), C, ptr(outs[0]), 0, n, H, D, eps, 0, stream())
    work = torch.empty(library().gibbs_decayed_outer_chunks_workspace(n, 1, H, D), dtype=torch.float32, device="cuda")
    call("gibbs_decayed_outer_chunks", ptr(rows), C, n * C, 2 * n * C, 3 * n * C, ptr(z), ptr(bias), ptr(bonus), ptr(gain), eps, ptr(states[1]),
         states[1].stride(0), ptr(cu), ptr(slot), ptr(outs[1]), ptr(work), 0, n, 1, H, D, stream())
    far = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)
    errors = [(far(o.cpu().numpy().reshape(n, H, D), np.stack(want)), far(s[0].cpu().numpy(), S)) for o, s in zip(outs, states)]
    for walk, mine in zip(*errors):
        assert mine <= 1.25 * walk, errors


@pytest.mark.parametrize("what", ["q", "k", "v", "z"])
def test_decayed_outer_rule_in_chunks_keeps_a_value_that_is_not_finite_behind_it(what):
    """The same for time mixing: a NaN or an infinity in a row (a rate of infinity is a decay of 0)."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, library, ptr, stream
    rng = np.random.default_rng(5)
    n, H, D = 200, 2, 40
    C = H * D
    dev = lambda a: torch.tensor(a, dtype=torch.float32, device="cuda")
    values = {name: rng.normal(size=(n, C)) for name in ("q", "k", "v", "g")}
    values["z"] = rng.normal(size=(n, C)) - 2
    bias, bonus, gain, start = dev(rng.normal(size=C)), dev(rng.normal(size=(H, D))), dev(np.ones(C)), dev(rng.normal(size=(2, H, D, D)))
    cu, slot = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([0, 150, 200], [1, 0]))
    def run(x, chunks):
        rows, z, state, out = dev(np.stack([x[name] for name in ("q", "k", "v", "g")])), dev(x["z"]), start.clone(), torch.empty((n, C), device="cuda")
        if chunks:
            work = torch.empty(library().gibbs_decayed_outer_chunks_workspace(n, 2, H, D), dtype=torch.float32, device="cuda")
            call("gibbs_decayed_outer_chunks", ptr(rows), C, n * C, 2 * n * C, 3 * n * C, ptr(z), ptr(bias), ptr(bonus), ptr(gain), 1e-6, ptr(state),
                 state.stride(0), ptr(cu), ptr(slot), ptr(out), ptr(work), 0, n, 2, H, D, stream())
        else:
            read = ops.decayed_outer_rule(rows[0], rows[1], rows[2], torch.exp(-torch.exp(z + bias)), bonus, state, cu, slot, H)
            call("gibbs_head_norm_gate", ptr(read), ptr(gain), C, ptr(rows[3]), C, ptr(out), 0, n, H, D, 1e-6, 0, stream())
        return out.reshape(n, H, D), state
    clean, _ = run(values, True)
    for t, bad in ((7, np.nan), (77, np.inf), (64, np.nan), (149, np.nan)):
        x = {name: a.copy() for name, a in values.items()}
        x[what][t, D + 3] = bad
        (got, mine), (want, state) = run(x, True), run(x, False)
        assert bool((got[:t] == clean[:t]).all() and (got[:, 0] == clean[:, 0]).all() and (got[150:] == clean[150:]).all()), (t, bad)
        if what != "z" and bad != bad:      # (an infinite read-out is divided by its norm: NaN or 0)
            for a, b in ((got, want), (mine, state)):
                assert bool((a.isnan() == b.isnan()).all()), (t, bad)
        ok = want.isfinite() & got.isfinite()
        assert float((got - want)[ok].norm()) <= 64 * 2.0 ** -24 * float(want[ok].norm())


def test_short_convolution_across_portions_shorter_than_its_taps():
    from gibbs_amd import ops
    rng = np.random.default_rng(4)
    T, C, K = 23, 70, 5
    x = rng.normal(size=(T, C))
    taps = rng.normal(size=(C, K))
    want = Z.silu(Z.causal_conv(x, taps))
    dx = torch.tensor(x, dtype=torch.float32, device="cuda")
    dt = torch.tensor(taps, dtype=torch.float32, device="cuda")
    state = torch.zeros((2, K - 1, C), dtype=torch.float32, device="cuda")
    slot = torch.tensor([1], dtype=torch.int32, device="cuda")
    at, outs = 0, []
    for n in [1, 1, 2, 3, 1, 9, 2, 4]:
        cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
        outs.append(ops.causal_conv_silu(dx[at:at + n].contiguous(), dt, state, torch.zeros(n, dtype=torch.int32, device="cuda"), cu, slot))
        at += n
    assert at == T
    assert np.abs(torch.cat(outs).cpu().numpy() - want).max() <= 1e-5


# ----------------------------------------------------------------------------------------------- entry points
def plain_greedy(model_dir, prompt, n):
    seq, out = list(prompt), []
    for _ in range(n):
        t = int(np.argmax(ZH.plain_logits(model_dir, seq)[-1]))
        out.append(t); seq.append(t)
    return out


@pytest.mark.parametrize("dtype", DTYPES)
def test_greedy_generation_through_the_scheduler(dirs, dtype):
    """`generate` (scheduler, prompt steps, bursts of captured decode steps) gives the plain implementation's greedy
    tokens; in bfloat16 wherever the plain logits' lead exceeds the precision's error."""
    from gibbs_amd import Engine, generate
    held = 0
    for name, lens in (("P", [7, 13, 2]), ("R", [5])):
        d = dirs[name]
        eng = Engine(d, dtype=dtype, max_tokens=512, max_requests=4)
        prompts = [ZH.tokens(40 + i, n, vocab_of(d)) for i, n in enumerate(lens)]
        outs = generate(eng, prompts, max_tokens=20, temperature=0.0, ignore_eos=True)
        for p, o in zip(prompts, outs):
            assert o.finish_reason == "length" and len(o.tokens) == 20
            if dtype == "float32":
                assert o.tokens == plain_greedy(d, p, 20)
                held += 20
                continue
            logits = ZH.plain_logits(d, list(p) + list(o.tokens))
            for i, t in enumerate(o.tokens):
                row = logits[len(p) - 1 + i]
                best, second = np.sort(row)[[-1, -2]]
                margin = 2 * 0.04 * np.abs(row).max()
                if best - second > margin:
                    held += 1
                    assert t == int(np.argmax(row)), f"token {i}"
                else:
                    assert row[t] >= best - margin, f"token {i}"
        eng.cache.check()
        assert eng.cache.free_slots() == 4
    assert held >= 20


def test_decode_bursts_change_nothing(dirs):
    from gibbs_amd import Engine, Generator, SamplingParams
    d = dirs["Q"]
    prompts = [ZH.tokens(70 + i, n, vocab_of(d)) for i, n in enumerate([9, 21, 5])]
    runs = []
    for burst in (0, 16):
        eng = Engine(d, dtype="float32", max_tokens=1024, max_requests=4)
        gen = Generator(eng, decode_burst=burst, eos_token_ids=())
        rids = [gen.submit(p, SamplingParams(temperature=0.0, max_new_tokens=n), rid=f"r{i}") for i, (p, n) in enumerate(zip(prompts, [37, 20, 9]))]
        res = gen.run()
        runs.append([res[r].tokens for r in rids])
    assert runs[0] == runs[1]
    assert runs[0][0] == plain_greedy(d, prompts[0], 37)


@pytest.mark.parametrize("dtype", DTYPES)
def test_replay_program(dirs, dtype, tmp_path):
    d = dirs["R"]
    ids = ZH.tokens(50, 40, vocab_of(d))
    other = ZH.tokens(51, 9, vocab_of(d))
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": ids[:17], "want": [0, 16]}, {"id": "b", "tokens": other[:2], "want": []}], "end": []},
             {"step": 1, "entries": [{"id": "b", "tokens": other[2:], "want": [6]}], "end": ["b"]},
             {"step": 2, "entries": [{"id": "a", "tokens": ids[17:39], "want": [21]}], "end": []},
             {"step": 3, "entries": [{"id": "a", "tokens": ids[39:], "want": [0]}], "end": ["a"]}]
    out = tmp_path / "out"
    proc = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", d, "--dtype", dtype, "--out", str(out), "--max-tokens", "128"],
                          input="\n".join(json.dumps(s) for s in steps) + "\n", capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stderr[-2000:]
    assert [l for l in proc.stdout.splitlines() if l.startswith("done")] == [f"done {i}" for i in range(4)]
    want_a, want_b = ZH.plain_logits(d, ids), ZH.plain_logits(d, other)
    read = lambda i: np.fromfile(out / f"{i}.f32", dtype="<f4").reshape(-1, vocab_of(d))
    close(read(0), want_a[[0, 16]], dtype, "step 0", [0, 16])
    close(read(1), want_b[[8]], dtype, "step 1")
    close(read(2), want_a[[38]], dtype, "step 2")
    close(read(3), want_a[[39]], dtype, "step 3")


def test_command_line(dirs):
    d = dirs["P"]
    prompt = ZH.tokens(60, 6, vocab_of(d))
    proc = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "gibbs"), "--model", d, "--dtype", "float32", "--prompt-ids",
                           ",".join(map(str, prompt)), "--max-tokens", "8", "--temperature", "0", "--ignore-eos"],
                          capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stderr[-2000:]
    assert "⚡ Prefill: 6 tokens" in proc.stdout and "📈 Roofline:" in proc.stdout
    line = proc.stdout.split("✨ Output:\n")[1].splitlines()[0]
    assert [int(t) for t in line.split()] == plain_greedy(d, prompt, 8)
    proc = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "gibbs"), "--model", d, "--arch-dump"], capture_output=True, text=True, timeout=600)
    dump = json.loads(proc.stdout)
    assert dump["architecture"] == "Zokepel" and dump["unconsumed"] == [] and dump["missing"] == []
    assert dump["derived"]["order"] == [0, 1, 2, 1, 2, 1, 2, 3]


@pytest.mark.parametrize("lens", [[64], [1] * 70, [3, 1, 2, 1, 300, 1, 210], [517], [1, 1, 1, 509, 4]])
@pytest.mark.parametrize("K,G,D,V", [(4, 2, 128, 40), (2, 3, 16, 8), (3, 1, 64, 24), (5, 2, 32, 72), (4, 5, 128, 600)])
def test_delta_convolution_makes_unit_vectors(lens, K, G, D, V):
    """Rows of several requests that meet inside a thread's run of rows, with and without history, few and many rows: the convolution is
    `causal_conv_silu`'s (the same sums, taken one by one), q and k its results over their norms; a sum of D squares and the rest are
    D + 8 roundings of 2^-24 at most."""
    from gibbs_amd import ops
    g = torch.Generator(device="cuda").manual_seed(5)
    N, C = sum(lens), 2 * G * D + V
    x = torch.randn((N, C), generator=g, device="cuda").bfloat16()
    taps = torch.randn((C, K), generator=g, device="cuda")
    state = torch.randn((len(lens) + 1, K - 1, C), generator=g, device="cuda")
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
    row_req = torch.repeat_interleave(torch.arange(len(lens), device="cuda"), torch.tensor(lens, device="cuda")).to(torch.int32)
    slot = torch.arange(1, len(lens) + 1, dtype=torch.int32, device="cuda").flip(0).contiguous()
    first = 3 if len(lens) > 4 else 0
    padded = [torch.cat([state[s].double(), x[a:b].double()]) for s, a, b in zip(slot.tolist(), cu.tolist(), cu.tolist()[1:])]
    conv = torch.cat([sum(p[j:j + n] * taps[:, j].double() for j in range(K)) for p, n in zip(padded, lens)])
    want = conv * torch.sigmoid(conv)
    heads = want[first:, :2 * G * D].unflatten(1, (2, G, D))
    unit = heads / torch.sqrt((heads * heads).sum(-1, keepdim=True) + 1e-6) * torch.tensor([0.25, 1.0], device="cuda", dtype=torch.float64)[:, None, None]
    want[first:, :2 * G * D] = unit.flatten(1)
    kept = state.clone()
    got = ops.delta_conv(x, taps, state, row_req, cu, slot, G, D, 0.25, 1e-6, first)
    err = (got.double() - want).abs()
    # (the convolution's own K + 8 roundings are relative to the sum of its terms' magnitudes, at most 60 here; the norm passes them on)
    assert err[:first].max().item() <= (K + 8) * 2.0 ** -24 * 60 if first else True
    assert err[first:, 2 * G * D:].max().item() <= (K + 8) * 2.0 ** -24 * 60
    head = got[first:, :2 * G * D].double().unflatten(1, (2, G, D)) - unit
    terms = torch.cat([sum((p[j:j + n] * taps[:, j].double()).abs() for j in range(K)) for p, n in zip(padded, lens)])[first:, :2 * G * D].unflatten(1, (2, G, D))
    scale = unit.norm(dim=-1) / (heads.norm(dim=-1) + 1e-30)
    bound = 2.0 ** -24 * (2 * (K + 8) * terms.norm(dim=-1) * scale + (D + 8) * unit.norm(dim=-1))
    assert (head.norm(dim=-1) <= bound).all()
    for i, s in enumerate(slot.tolist()):
        assert torch.equal(state[s], padded[i][-(K - 1):].float())
    assert torch.equal(state[0], kept[0])


@pytest.mark.parametrize("n,nh,nkv,hd,vd,norm_dim,unit,every", [(1, 4, 1, 64, 64, 0, True, 7), (70, 16, 4, 128, 128, 0, True, 1024), (9, 3, 3, 16, 24, 13, True, 0),
                                                              (33, 40, 8, 64, 128, 0, False, 5), (5, 2, 0, 32, 8, 0, True, 3), (3, 64, 64, 128, 128, 0, True, 2)])
def test_unit_heads_in_whole_16_bytes_like_float32(n, nh, nkv, hd, vd, norm_dim, unit, every):
    """bfloat16 heads eight channels a lane against the float32 kernel on the same values: one rounding to bfloat16 apart (2^-8), values unchanged."""
    from gibbs_amd import ops
    g = torch.Generator(device="cuda").manual_seed(n + nh)
    W = (nh + nkv) * hd + nkv * vd
    x = torch.randn((n, W), generator=g, device="cuda").bfloat16()
    page_size, pages = 4, 40
    pos = torch.randint(0, 100, (n,), generator=g, device="cuda", dtype=torch.int32)
    req = torch.zeros(n, dtype=torch.int32, device="cuda")
    table = torch.randperm(pages, generator=g, device="cuda").to(torch.int32)[:25].reshape(1, -1).contiguous()
    outs = []
    for kind in (torch.float32, torch.bfloat16):
        rows = x.to(kind).clone()
        kp = torch.zeros((pages, nkv, page_size, hd), dtype=kind, device="cuda") if nkv else None
        vp = torch.zeros((pages, nkv, page_size, vd), dtype=kind, device="cuda") if nkv else None
        for i in range(n):        # (rows of one position would race for a place in the pages)
            ops.qk_unit_kv(rows[i:i + 1], nh, nkv, hd, vd, kpages=kp, vpages=vp, table=table if nkv else None, pos=pos[i:i + 1], row_req=req[:1], eps=1e-6, unit=unit,
                           temp_coef=0.1, temp_every=every, norm_dim=norm_dim)
        outs.append([rows.float()] + ([kp.float(), vp.float()] if nkv else []))
        if kind == torch.bfloat16:
            again = x.clone()
            ops.qk_unit_kv(again, nh, nkv, hd, vd, kpages=None, vpages=None, table=None, pos=pos, row_req=req, eps=1e-6, unit=unit, temp_coef=0.1, temp_every=every,
                           norm_dim=norm_dim)
            assert torch.equal(again, rows)
    for want, got in zip(*outs):
        assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-30).all()


@pytest.mark.parametrize("n,H,V,gains", [(1, 1, 16, 16), (7, 3, 32, 96), (300, 16, 128, 128), (130, 5, 64, 64)])
@pytest.mark.parametrize("gated", [False, True])
def test_head_norm_in_whole_16_bytes_like_float32(n, H, V, gains, gated):
    """The bfloat16 kernel with a few lanes a head against the float32 kernel: one rounding to bfloat16 apart."""
    from gibbs_amd.ops.lib import call, ptr, stream
    g = torch.Generator(device="cuda").manual_seed(n)
    o = torch.randn((n, H * V), generator=g, device="cuda")
    gain = torch.randn(gains, generator=g, device="cuda")
    gate = torch.randn((n, H * V + 8), generator=g, device="cuda").bfloat16()
    outs = []
    for kind, code in ((torch.float32, 0), (torch.bfloat16, 1)):
        y, z = torch.empty((n, H * V), dtype=kind, device="cuda"), gate.to(kind)
        call("gibbs_head_norm_gate", ptr(o), ptr(gain), gains, ptr(z) if gated else None, H * V + 8 if gated else 0, ptr(y), code, n, H, V, 1e-6, 0, stream())
        outs.append(y.float())
    assert ((outs[1] - outs[0]).abs() <= 2.0 ** -8 * outs[0].abs() + 1e-30).all()


@pytest.mark.parametrize("lens", [[64], [1] * 66, [1025], [5, 1, 1, 1500, 2, 1]])
@pytest.mark.parametrize("W,mixes", [(8, 1), (2056, 5)])
def test_token_shift_in_whole_16_bytes_like_float32(lens, W, mixes):
    """Eight channels a thread, a row or four of them, requests that meet inside a thread's rows: the float32 kernel's results rounded, to the bit, and its state."""
    from gibbs_amd.ops.lib import call, ptr, stream
    g = torch.Generator(device="cuda").manual_seed(W)
    n = sum(lens)
    h = torch.randn((n, W), generator=g, device="cuda").bfloat16()
    mu = torch.randn((mixes, W), generator=g, device="cuda")
    kept = torch.randn((len(lens) + 1, W), generator=g, device="cuda")
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
    req = torch.repeat_interleave(torch.arange(len(lens), device="cuda"), torch.tensor(lens, device="cuda")).to(torch.int32)
    slot = torch.arange(1, len(lens) + 1, dtype=torch.int32, device="cuda").flip(0).contiguous()
    outs = []
    for kind, code in ((torch.float32, 0), (torch.bfloat16, 1)):
        x, state, out = h.to(kind), kept.clone(), torch.empty((mixes, n, W), dtype=kind, device="cuda")
        call("gibbs_token_shift", ptr(x), code, ptr(mu), mixes, ptr(state), W, ptr(req), ptr(cu), ptr(slot), ptr(out), n, len(lens), W, 1, int(n == len(lens)), stream())
        outs.append((out, state))
    assert torch.equal(outs[0][0].bfloat16(), outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("hd", [16, 32, 64, 128])
@pytest.mark.parametrize("unit,every", [(True, 7), (True, 0), (False, 3)])
def test_unit_heads_in_whole_16_bytes_are_the_general_kernels(hd, unit, every):
    """Rows of whole 16 bytes and the same rows two values further apart, which take the kernel with a wave a head: rows and pages are the same bits, with an infinity
    and a NaN among them.  (A norm that is one float32 step off moves one of some 2^16 bfloat16 results, so there are over a million.)"""
    from gibbs_amd.ops.lib import call, ptr, stream
    g = torch.Generator(device="cuda").manual_seed(hd)
    n, nh, nkv, vd, page_size, pages = 1031 * 128 // hd, 8, 3, 24, 16, 600
    W = (nh + nkv) * hd + nkv * vd
    x = torch.randn((n, W), generator=g, device="cuda").bfloat16()
    x[3, 1], x[9, nh * hd + 5] = float("inf"), float("nan")
    pos = torch.arange(n, dtype=torch.int32, device="cuda")
    req = torch.zeros(n, dtype=torch.int32, device="cuda")
    table = torch.randperm(pages, generator=g, device="cuda").to(torch.int32)[:520].reshape(1, -1).contiguous()
    outs = []
    for ld in (W, W + 2):
        rows = torch.zeros((n, ld), dtype=torch.bfloat16, device="cuda")
        rows[:, :W] = x
        kp, vp = (torch.zeros((pages, nkv, page_size, d), dtype=torch.bfloat16, device="cuda") for d in (hd, vd))
        call("gibbs_qk_unit_kv", ptr(rows), ld, ptr(kp), ptr(vp), 1, ptr(pos), ptr(req), ptr(table), 520, page_size, pages, n, nh, nkv, hd, vd, 1e-6, int(unit),
             hd - 3, 0.1, every, stream())
        outs.append([t.contiguous().nan_to_num(nan=5.0, posinf=7.0, neginf=-7.0) for t in (rows[:, :W], kp, vp)])
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("lens", [[64], [3, 1, 2, 1, 300, 1, 210], [1] * 515])
@pytest.mark.parametrize("K,G,D,V", [(4, 2, 128, 40), (2, 3, 16, 8), (3, 1, 64, 24), (5, 2, 32, 72)])
def test_delta_convolution_is_the_convolution_and_then_the_unit_vectors(lens, K, G, D, V):
    """One kernel against the two that it stands for, whose results a row's do not differ from whichever way a step takes: rows and states to the bit, with
    an infinity, a NaN and a head of zeros among the rows; rows of a request each, which move all their states on, too."""
    from gibbs_amd import ops
    from gibbs_amd.ops.lib import call, ptr, stream
    g = torch.Generator(device="cuda").manual_seed(D)
    N, C, H = sum(lens), 2 * G * D + V, 2 * G
    x = torch.randn((N, C), generator=g, device="cuda").bfloat16()
    x[1, 2], x[2, 3], x[7:14, :D] = float("inf"), float("nan"), 0.0
    taps = torch.randn((C, K), generator=g, device="cuda")
    state = torch.randn((len(lens) + 1, K - 1, C), generator=g, device="cuda")
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
    row_req = torch.repeat_interleave(torch.arange(len(lens), device="cuda"), torch.tensor(lens, device="cuda")).to(torch.int32)
    slot = torch.arange(1, len(lens) + 1, dtype=torch.int32, device="cuda").flip(0).contiguous()
    first, other = (3 if len(lens) > 4 else 0), state.clone()
    got = ops.delta_conv(x, taps, state, row_req, cu, slot, G, D, 0.25, 1e-6, first)
    want = ops.causal_conv_silu(x, taps, other, row_req, cu, slot)
    rest, m = want[first:], N - first
    raw = torch.zeros((m, 2 * H), dtype=torch.bfloat16, device="cuda")
    gates = torch.zeros(H, device="cuda")
    beta, decay = torch.empty((m, H), device="cuda"), torch.empty((m, H), device="cuda")
    call("gibbs_delta_prep", ptr(rest), ptr(rest[:, G * D:]), C, ptr(raw), ptr(raw[:, H:]), 2 * H, 1, None, ptr(gates), ptr(gates), ptr(beta), ptr(decay), m, G, H, D,
         0.25, 1e-6, stream())
    for a, b in ((got, want), (state, other)):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(nan=7.0), b.nan_to_num(nan=7.0))


@pytest.mark.parametrize("lens", [[1] * 1027, [1026], [5, 1, 1, 700, 2, 1, 330]])
@pytest.mark.parametrize("W,mixes", [(512, 5), (3072, 2), (3080, 5), (6152, 1)])
def test_token_shift_of_many_values_is_float32s(lens, W, mixes):
    """Eight channels a thread, of a row (the first width) and of four, where rows and channels are enough for that: the float32 kernel's results rounded, to the bit,
    and its state; requests that meet inside a thread's rows, and rows of a request each, whose states one thread reads and moves on."""
    from gibbs_amd.ops.lib import call, ptr, stream
    g = torch.Generator(device="cuda").manual_seed(W)
    n = sum(lens)
    h = torch.randn((n, W), generator=g, device="cuda").bfloat16()
    mu = torch.randn((mixes, W), generator=g, device="cuda")
    kept = torch.randn((len(lens) + 1, W), generator=g, device="cuda")
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
    req = torch.repeat_interleave(torch.arange(len(lens), device="cuda"), torch.tensor(lens, device="cuda")).to(torch.int32)
    slot = torch.arange(1, len(lens) + 1, dtype=torch.int32, device="cuda").flip(0).contiguous()
    outs = []
    for kind, code in ((torch.float32, 0), (torch.bfloat16, 1)):
        x, state, out = h.to(kind), kept.clone(), torch.empty((mixes, n, W), dtype=kind, device="cuda")
        call("gibbs_token_shift", ptr(x), code, ptr(mu), mixes, ptr(state), W, ptr(req), ptr(cu), ptr(slot), ptr(out), n, len(lens), W, 1, int(n == len(lens)), stream())
        outs.append((out, state))
    assert torch.equal(outs[0][0].bfloat16(), outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("K,C", [(4, 9216), (3, 4608), (2, 24640), (4, 4616)])
@pytest.mark.parametrize("lens", [[1] * 1027, [1026], [3, 1, 2, 1, 700, 1, 4, 313]])
def test_convolution_of_four_rows_a_thread_is_float32s(K, C, lens):
    """Rows and channels enough that a thread takes four rows: bfloat16 rows against the same values in float32, a channel a thread, to the bit (sums are
    float32 in ascending order in both); requests that meet inside a thread's rows, and one row of each with its state moved on in the same kernel.  With unit
    vectors (heads of 128, the first channels) the other channels are the same bits, and q and k unit vectors."""
    from gibbs_amd import ops
    g = torch.Generator(device="cuda").manual_seed(K)
    N = sum(lens)
    x = torch.randn((N, C), generator=g, device="cuda").bfloat16()
    x[1, 2], x[5, C - 1] = float("inf"), float("nan")
    taps = torch.randn((C, K), generator=g, device="cuda")
    state = torch.randn((len(lens) + 1, K - 1, C), generator=g, device="cuda")
    cu = torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32, device="cuda")
    row_req = torch.repeat_interleave(torch.arange(len(lens), device="cuda"), torch.tensor(lens, device="cuda")).to(torch.int32)
    slot = torch.arange(1, len(lens) + 1, dtype=torch.int32, device="cuda").flip(0).contiguous()
    states = [state.clone() for _ in range(3)]
    want = ops.causal_conv_silu(x.float(), taps, states[0], row_req, cu, slot)
    got = ops.causal_conv_silu(x, taps, states[1], row_req, cu, slot)
    unit = ops.delta_conv(x, taps, states[2], row_req, cu, slot, 2, 128, 0.25, 1e-6, 2)
    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(nan=7.0), b.nan_to_num(nan=7.0))
    assert same(got, want) and same(states[1], states[0]) and same(states[2], states[0])
    assert same(unit[:, 512:], want[:, 512:]) and same(unit[:2], want[:2])
    heads = unit[2:, :512].unflatten(1, (4, 128)).double().norm(dim=-1)[8:]
    assert (heads - torch.tensor([0.25, 0.25, 1.0, 1.0], device="cuda")).abs().max() < 1e-5


@pytest.mark.parametrize("V", [16, 32, 64, 128])
@pytest.mark.parametrize("gated", [False, True])
def test_head_norm_in_whole_16_bytes_is_the_general_kernels(V, gated):
    """Results in whole 16 bytes and the same results one value further on, which take the kernel with a wave a head: the same bits, with an infinity, a NaN and a
    head of zeros.  (Over a million results: a norm that is one float32 step off moves one of some 2^16.)"""
    from gibbs_amd.ops.lib import call, ptr, stream
    g = torch.Generator(device="cuda").manual_seed(V)
    H, n = 8, 1031 * 128 // V
    o = torch.randn((n, H * V), generator=g, device="cuda")
    o[3, 1], o[9, V + 5], o[11, :V] = float("inf"), float("nan"), 0.0
    gain, gate = torch.randn(V, generator=g, device="cuda"), torch.randn((n, H * V), generator=g, device="cuda").bfloat16()
    outs = []
    for shift in (0, 1):
        y = torch.zeros(n * H * V + 8, dtype=torch.bfloat16, device="cuda")[shift:shift + n * H * V]
        call("gibbs_head_norm_gate", ptr(o), ptr(gain), V, ptr(gate) if gated else None, H * V if gated else 0, ptr(y), 1, n, H, V, 1e-6, 1, stream())
        outs.append(y.clone())
    assert torch.equal(outs[0].isnan(), outs[1].isnan()) and torch.equal(outs[0].nan_to_num(nan=7.0), outs[1].nan_to_num(nan=7.0))
