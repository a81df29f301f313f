"""Row-kernel cases the sweep does not reach: peaked bf16 rows, where the resident
kernel's f16 softmax terms matter, and calls that leave dead rows unwritten
(PCP_FLAG_NO_ZERO_FILL) on every row kernel. Bars: tests/parity_tol.py."""
import threading

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from pcp_amd import grpo
from pcp_amd._lib import LossMode
from parity_tol import (assert_dlogits, dev, full_floor, full_loss_tol, host_bits, token_scale,
                        tok_to_rows)

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def peaked_case(V, S, T, seed):
    """bf16 rows whose two largest logits sit in one 16-byte vector (so one lane holds
    both, and the lane's largest term is 1), near-tied, with softmax mass 0.3-0.5 each."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((S, T, V)).astype(np.float32)
    ids = rng.integers(0, V, size=(S, T)).astype(np.int64)
    level = np.log(2.0 * V * np.exp(0.5))            # e^level = 2 * sum of the other terms
    for s in range(S):
        for t in range(T):
            q = int(rng.integers(0, V // 8))
            a, b = rng.choice(8, size=2, replace=False)
            i, j = 8 * q + a, 8 * q + b
            x[s, t, i] = level + rng.uniform(0.0, 0.3)
            x[s, t, j] = level + rng.uniform(0.0, 0.3)
            r = rng.random()
            ids[s, t] = i if r < 0.3 else (j if r < 0.5 else ids[s, t])
    ref = x + rng.standard_normal(x.shape).astype(np.float32) * 0.1
    lengths = rng.integers(T // 2, T + 1, size=S)
    mask = (np.arange(T)[None] < lengths[:, None]).astype(np.float32)
    rewards = rng.random(S).astype(np.float32)
    return orc.bf16_from_f32(x), orc.bf16_from_f32(ref), ids, mask, rewards


@pytest.mark.parametrize("V,S,T,among", [(1000, 8, 16, 8), (151936, 4, 8, 4), (151936, 4, 8, 100)])
def test_peaked_bf16_rows(V, S, T, among):
    """Two near-tied dominant logits per row (p ~ 0.3-0.5 each) in one lane. By default
    the kernel's f16 softmax terms carry up to 2^-11 of these large dlogits, inside the
    cached bar; with PCP_FLAG_EXACT_BF16 every output is the f32 result rounded once,
    inside the exact bar. Where the term is in f16's normal range (|d| >= 2^-14 |c|) the
    two differ by at most one bf16 ulp, since 2^-11 of a value is under half its ulp. The
    case's S sequences are the first of `among`, the others masked: with few wide rows both
    calls run in parts, which have no f16 terms, so the widest instance needs the 800 rows."""
    x, ref, ids, mask, rewards = peaked_case(V, S, T, seed=V + S)
    G = 2
    sel = np.ascontiguousarray(x).reshape(S * T, V)
    lp, _ = orc.logprob(sel, ids.reshape(-1), dtype=orc.BF16)
    old = (lp.reshape(S, T) + np.random.default_rng(1).standard_normal((S, T)) * 0.05).astype(np.float32)
    want = orc.grpo_full(x, ids, mask, rows=T, rewards=rewards, group_size=G, ref_logits=ref, old_logp=old,
                         loss_mode=orc.CLIP_KL, dtype=orc.BF16)
    # The rows are peaked as intended: the largest softmax term of every row is 0.25 or more.
    xs = orc.bf16_to_f32(sel).astype(np.float64)
    p = np.exp(xs - xs.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    assert p.max(1).min() >= 0.25
    ts = token_scale(x, ids, T, 0, orc.BF16)
    fl = tok_to_rows(full_floor(want, mask, old, S, False, 0.04, 0.2, ts), T, 0, T)
    bits = {}

    def all_rows(a):
        a = dev(a)
        return torch.cat([a, torch.zeros((among - S, *a.shape[1:]), dtype=a.dtype, device=DEV)])

    for exact in (False, True):
        print(f"peaked bf16 rows: V={V} S={S} T={T} among {among} exact={exact}", flush=True)
        out = grpo.grpo_loss_fwd_bwd(all_rows(x), all_rows(ids), all_rows(mask), rewards=all_rows(rewards), group_size=G,
                                     ref_logits=all_rows(ref), old_logp=all_rows(old), loss_norm=float(S),
                                     loss_mode=LossMode.GRPO_CLIP_KL, exact_bf16=exact)
        torch.cuda.synchronize()
        assert np.all(np.abs(out.logp[:S].cpu().numpy() - want.lp) <= 1e-5 * ts)
        bits[exact] = host_bits(out.dlogits[:S])
        got = orc.bf16_to_f32(bits[exact])
        assert_dlogits(got, want.dlogits, fl, True, exact=exact)
        err = np.abs(got.astype(np.float64) - want.dlogits)
        cabs = np.abs(want.coef)[..., None]
        big = (np.abs(want.dlogits) >= 0.05 * cabs) & (cabs > 0)
        rel = (err[big] / np.abs(want.dlogits[big])).max()
        print(f"  worst relative error where |d| >= 0.05|c|: {rel:.3e} (bf16 unit roundoff {2.0 ** -8:.3e})",
              flush=True)
        assert abs(float(out.loss.cpu()) - want.loss) <= full_loss_tol(want, x, ids, mask, T, 0, orc.BF16, False,
                                                                       0.04, S)
    c = np.abs(want.coef)[..., None] * np.ones((1, 1, V))
    normal = np.abs(want.dlogits) >= 2.0 ** -14 * c
    a = bits[False].astype(np.int32)
    b = bits[True].astype(np.int32)
    same_sign = (a >> 15) == (b >> 15)
    ulps = np.abs((a & 0x7FFF) - (b & 0x7FFF))
    assert np.all(same_sign[normal] | (ulps[normal] == 0)) and ulps[normal].max() <= 1
    in_parts = V >= 32768 and among * T <= 768
    assert in_parts == bool((a == b).all())
    print(f"  cached vs exact: {np.mean(ulps[normal] != 0):.2%} of normal-range elements one ulp apart", flush=True)


# (kind, logits dtype, V, dlogits dtype, force_streaming, shifted layout, live fraction of the mask)
ZF_CASES = [
    ("resident", "bf16", 4096, "bf16", False, False, 0.7),
    ("resident-sparse", "bf16", 4096, "bf16", False, False, 0.25),
    ("resident-shifted", "bf16", 151936, "bf16", False, True, 0.7),
    ("resident-shifted-sparse", "bf16", 151936, "bf16", False, True, 0.2),
    ("resident-edge", "bf16", 5003, "bf16", False, True, 0.7),
    ("resident-edge-sparse", "bf16", 5003, "bf16", False, False, 0.3),
    ("resident-f32", "f32", 3000, "f32", False, False, 0.7),
    ("resident-f32-sparse", "f32", 3000, "f32", False, True, 0.25),
    ("resident-bf16-to-f32", "bf16", 4096, "f32", False, True, 0.7),
    ("resident-bf16-to-f32-qwen", "bf16", 151936, "f32", False, False, 0.7),
    ("resident-bf16-to-f32-qwen-sparse", "bf16", 151936, "f32", False, True, 0.25),
    ("stream-vec", "bf16", 4096, "bf16", True, True, 0.7),
    ("stream-scalar", "bf16", 5003, "f32", False, False, 0.7),
]


@pytest.mark.parametrize("kind,dt,V,odt,stream,shifted,live", ZF_CASES, ids=[c[0] for c in ZF_CASES])
def test_no_zero_fill_leaves_dead_rows(kind, dt, V, odt, stream, shifted, live):
    """PCP_FLAG_NO_ZERO_FILL: dlogits rows of masked, ignored (-100) and pad tokens keep
    what the caller put there, bit for bit; live rows match the oracle. Resident
    (aligned and off-16-byte rows), f32 and mixed-precision, and both streaming kernels.
    The persistent kernels visit only the listed live rows when fewer than half the rows
    are live (the sparse cases) and every row otherwise."""
    rng = np.random.default_rng(V + 7 * len(kind))
    S, T, G = 4, 9, 2
    rows, off = (T - 1, 1) if shifted else (T, 0)
    x32 = rng.standard_normal((S, T, V)).astype(np.float32) * 3
    r32 = x32 + rng.standard_normal((S, T, V)).astype(np.float32) * 0.1
    if dt == "bf16":
        x, ref, odt_orc = orc.bf16_from_f32(x32), orc.bf16_from_f32(r32), orc.BF16
    else:
        x, ref, odt_orc = x32, r32, orc.F32
    ids = rng.integers(0, V, size=(S, T)).astype(np.int64)
    ids[rng.random((S, T)) < 0.15] = -100
    mask = (rng.random((S, T)) < live).astype(np.float32)
    mask[1] = 0.0                                        # one empty sequence
    rewards = np.array([1.0, 0.0, 0.25, 0.75], np.float32)
    sel = np.ascontiguousarray(x[:, :rows]).reshape(S * rows, V)
    lp, _ = orc.logprob(sel, np.clip(ids[:, off:off + rows].reshape(-1), 0, None), dtype=odt_orc)
    old = np.zeros((S, T), np.float32)
    old[:, off:off + rows] = (lp.reshape(S, rows) + rng.standard_normal((S, rows)) * 0.05).astype(np.float32)
    tdt = {"bf16": torch.bfloat16, "f32": torch.float32}[odt]
    sentinel = -3.5
    dl = torch.full((S, T, V), sentinel, dtype=tdt, device=DEV)
    print(f"no zero-fill: {kind} {dt}->{odt} V={V} streaming={stream} shifted={shifted}", flush=True)
    out = grpo.grpo_loss_fwd_bwd(dev(x), dev(ids), dev(mask), rewards=dev(rewards), group_size=G,
                                 ref_logits=dev(ref), old_logp=dev(old), loss_mode=LossMode.GRPO_CLIP_KL,
                                 rows=rows, tok_offset=off, dlogits=dl, zero_fill=False, force_streaming=stream)
    torch.cuda.synchronize()
    want = orc.grpo_full(x, ids, mask, rows=rows, tok_offset=off, rewards=rewards, group_size=G, ref_logits=ref,
                         old_logp=old, loss_mode=orc.CLIP_KL, dtype=odt_orc)
    got_bits = host_bits(out.dlogits)
    sent_bits = host_bits(torch.full((1,), sentinel, dtype=tdt))[0]
    dead = np.zeros((S, T), bool)
    for s in range(S):
        for t in range(T):
            dead[s, t] = t >= rows or mask[s, off + t] == 0 or ids[s, off + t] == -100
    assert dead.any() and (~dead).any()
    assert np.all(got_bits[dead] == sent_bits), "a dead row was written"
    ts = token_scale(x, ids, rows, off, odt_orc)
    fl = tok_to_rows(full_floor(want, mask, old, S, False, 0.04, 0.2, ts), rows, off, T)
    got = orc.bf16_to_f32(got_bits) if odt == "bf16" else got_bits.astype(np.float32)
    assert_dlogits(got[~dead], want.dlogits[~dead], fl[~dead], odt == "bf16")
    assert abs(float(out.loss.cpu()) - want.loss) <= full_loss_tol(want, x, ids, mask, rows, off, odt_orc, False,
                                                                   0.04, S)


# (logits dtype, V, dlogits dtype): aligned rows, several listed rows per workgroup
LISTED_CASES = [("bf16", 32768, "bf16"), ("bf16", 32768, "f32"), ("f32", 8192, "f32"), ("f32", 10000, "f32")]


@pytest.mark.parametrize("dt,V,odt", LISTED_CASES, ids=[f"{c[0]}-{c[1]}-{c[2]}" for c in LISTED_CASES])
def test_no_zero_fill_listed_rows_prefetch(dt, V, odt):
    """Without zero-fill and a quarter of the rows live, the resident kernel walks the
    listed live rows, several per workgroup here, loading each next row's policy chunks
    during the current row's dlogits pass (on 1024-lane instances of 4 chunks, whose rows
    are claimed from the counter, the 256-lane instance of 8, whose rows are dealt in
    strides, and the split-half bf16 -> f32 instance). Every live row against the oracle, dead rows
    untouched bit for bit."""
    rng = np.random.default_rng(V + len(dt) + len(odt))
    S, T, G = 16, 512, 4
    x32 = rng.standard_normal((S, T, V)).astype(np.float32) * 3
    r32 = x32 + rng.standard_normal((S, T, V)).astype(np.float32) * 0.1
    if dt == "bf16":
        x, ref, odt_orc = orc.bf16_from_f32(x32), orc.bf16_from_f32(r32), orc.BF16
    else:
        x, ref, odt_orc = x32, r32, orc.F32
    del x32, r32
    ids = rng.integers(0, V, size=(S, T)).astype(np.int64)
    ids[rng.random((S, T)) < 0.05] = -100
    mask = (rng.random((S, T)) < 0.27).astype(np.float32)
    rewards = rng.random(S).astype(np.float32)
    lp, _ = orc.logprob(np.ascontiguousarray(x).reshape(S * T, V), np.clip(ids.reshape(-1), 0, None), dtype=odt_orc)
    old = (lp.reshape(S, T) + rng.standard_normal((S, T)) * 0.05).astype(np.float32)
    tdt = {"bf16": torch.bfloat16, "f32": torch.float32}[odt]
    sentinel = -3.5
    dl = torch.full((S, T, V), sentinel, dtype=tdt, device=DEV)
    dead = (mask == 0) | (ids == -100)
    assert 2 * int((~dead).sum()) < S * T          # the listed path
    print(f"listed rows: {dt}->{odt} V={V}, {int((~dead).sum())} live of {S * T}", flush=True)
    out = grpo.grpo_loss_fwd_bwd(dev(x), dev(ids), dev(mask), rewards=dev(rewards), group_size=G,
                                 ref_logits=dev(ref), old_logp=dev(old), loss_mode=LossMode.GRPO_CLIP_KL,
                                 dlogits=dl, zero_fill=False)
    torch.cuda.synchronize()
    want = orc.grpo_full(x, ids, mask, rows=T, rewards=rewards, group_size=G, ref_logits=ref, old_logp=old,
                         loss_mode=orc.CLIP_KL, dtype=odt_orc)
    got_bits = host_bits(out.dlogits)
    sent_bits = host_bits(torch.full((1,), sentinel, dtype=tdt))[0]
    assert np.all(got_bits[dead] == sent_bits), "a dead row was written"
    ts = token_scale(x, ids, T, 0, odt_orc)
    fl = tok_to_rows(full_floor(want, mask, old, S, False, 0.04, 0.2, ts), T, 0, T)
    got = orc.bf16_to_f32(got_bits) if odt == "bf16" else got_bits.astype(np.float32)
    assert_dlogits(got[~dead], want.dlogits[~dead], fl[~dead], odt == "bf16")
    assert abs(float(out.loss.cpu()) - want.loss) <= full_loss_tol(want, x, ids, mask, T, 0, odt_orc, False, 0.04, S)


# Live-row counts around the persistent grid's size (one workgroup per resident slot,
# a few hundred to about a thousand here): none, one, fewer than the grid, between one
# and two grids (the second rows come from the first claim, not the counter), more,
# and either side of the switch to visiting every row (half of 8192 rows). At V = 4096
# the rows past the first grid are dealt in strides; bf16 20,000 and f32 10,000 claim them.
LIVE_COUNTS = [0, 1, 37, 255, 256, 257, 511, 512, 513, 767, 1023, 1024, 1025, 1537, 2049, 4095, 4096]


@pytest.fixture(scope="module", params=[4096, 20000])
def count_inputs(request):
    S, T, V = 16, 512, request.param
    gen = torch.Generator(device=DEV)
    gen.manual_seed(77)
    x = torch.randn((S, T, V), generator=gen, device=DEV) * 3
    r = x + torch.randn((S, T, V), generator=gen, device=DEV) * 0.1
    ids = torch.randint(0, V, (S, T), generator=gen, device=DEV)
    old = torch.randn((S, T), generator=gen, device=DEV) * 0.05 - float(np.log(V))
    rewards = torch.rand((S,), generator=gen, device=DEV)
    if V > 4096:
        W = V // 2
        return dict(S=S, T=T, V={"bf16": V, "f32": W}, x={"bf16": x.to(torch.bfloat16), "f32": x[..., :W].contiguous()},
                    r={"bf16": r.to(torch.bfloat16), "f32": r[..., :W].contiguous()}, ids=ids % W, old=old,
                    rewards=rewards)
    return dict(S=S, T=T, V={"bf16": V, "f32": V}, x={"bf16": x.to(torch.bfloat16), "f32": x},
                r={"bf16": r.to(torch.bfloat16), "f32": r}, ids=ids, old=old, rewards=rewards)


@pytest.mark.parametrize("dt", ["bf16", "f32"])
@pytest.mark.parametrize("n_live", LIVE_COUNTS)
def test_no_zero_fill_live_counts(count_inputs, n_live, dt):
    """Exactly n_live live rows at random places: the call without zero-fill (listed rows
    with the next-row prefetch below half live, every row in order from half on) gives
    the zero-fill call's outputs bit for bit on live rows and leaves every dead row's
    dlogits as they were."""
    c = count_inputs
    S, T, V = c["S"], c["T"], c["V"][dt]
    rng = np.random.default_rng(1000 + n_live)
    flat = np.zeros(S * T, np.float32)
    flat[rng.choice(S * T, size=n_live, replace=False)] = 1.0
    mask = torch.from_numpy(flat.reshape(S, T)).to(DEV)
    kw = dict(rewards=c["rewards"], group_size=4, ref_logits=c["r"][dt], old_logp=c["old"],
              loss_mode=LossMode.GRPO_CLIP_KL)
    x = c["x"][dt]
    sentinel = -3.5
    dl = torch.full((S, T, V), sentinel, dtype=x.dtype, device=DEV)
    print(f"live rows {n_live} of {S * T} ({dt})", flush=True)
    got = grpo.grpo_loss_fwd_bwd(x, c["ids"], mask, dlogits=dl, zero_fill=False, **kw)
    want = grpo.grpo_loss_fwd_bwd(x, c["ids"], mask, **kw)
    torch.cuda.synchronize()
    live = mask != 0
    assert torch.equal(got.dlogits[live], want.dlogits[live])
    assert bool((got.dlogits[~live] == sentinel).all()), "a dead row was written"
    assert bool((want.dlogits[~live] == 0).all())
    for f in ("loss", "logp", "ref_logp", "token_loss", "advantages"):
        assert torch.equal(getattr(got, f), getattr(want, f)), f


@pytest.mark.parametrize("zero_fill, longest", [(True, 128), (False, 128), (False, 40)])
@pytest.mark.parametrize("dtype, V", [("bf16", 64), ("bf16", 1001), ("bf16", 16384), ("bf16", 16392), ("f32", 8192),
                                      ("f32", 1030), ("f16", 8200)])
def test_rows_past_the_first_grid(dtype, V, zero_fill, longest):
    """Narrow rows (256 lanes x 1 to 8 chunks, aligned and not) are dealt in grid strides, wider
    ones from the counter. A row's outputs depend on its own data only, so the last 4 of 72
    sequences (9,216 rows, more than two grids of the widest launch) must come out bit for bit
    as in a call of their own (512 rows: one grid). longest 40 lists under half of the rows."""
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    S, T = 72, 128
    gen = torch.Generator(device="cuda").manual_seed(V)
    x = (torch.randn((S, T, V), generator=gen, device="cuda") * 3).to(dt)
    r = (x.float() + 0.1 * torch.randn((S, T, V), generator=gen, device="cuda")).to(dt)
    ids = torch.randint(0, V, (S, T), generator=gen, device="cuda")
    lengths = torch.randint(1, longest + 1, (S, 1), generator=gen, device="cuda")
    mask = (torch.arange(T, device="cuda")[None] < lengths).float()
    adv = torch.randn(S, generator=gen, device="cuda")
    old = -torch.rand((S, T), generator=gen, device="cuda") * 9

    def call(sl):
        out = grpo.grpo_loss_fwd_bwd(x[sl], ids[sl], mask[sl], advantages=adv[sl], ref_logits=r[sl], old_logp=old[sl],
                                     loss_mode=LossMode.GRPO_CLIP_KL, loss_norm=float(S), zero_fill=zero_fill,
                                     dlogits=torch.full_like(x[sl], 7.0))
        return out.dlogits, out.logp, out.ref_logp, out.token_loss

    for whole, own in zip(call(slice(0, S)), call(slice(S - 4, S))):
        assert torch.equal(whole[S - 4:], own)


@pytest.mark.parametrize("T", [1, 96, 128, 509, 1024])
@pytest.mark.parametrize("dtype, V", [("bf16", 64), ("bf16", 16384), ("f32", 1030)])
def test_every_row_is_dealt_once(dtype, V, T):
    """Rows dealt in grid strides that move on within the sequence: every row of calls of several
    grids and a part comes out as in the streaming kernel, which takes a workgroup for each (to
    2^-8 of the largest, a bf16 rounding and the f16 softmax terms; dead rows are zero in both)."""
    dt = {"bf16": torch.bfloat16, "f32": torch.float32}[dtype]
    S = 9001 // T
    gen = torch.Generator(device="cuda").manual_seed(V + T)
    x = torch.randn((S, T, V), generator=gen, device="cuda").to(dt)
    ids = torch.randint(0, V, (S, T), generator=gen, device="cuda")
    mask = (torch.arange(T, device="cuda")[None] < torch.randint(0, T + 1, (S, 1), generator=gen, device="cuda")).float()
    adv = torch.rand(S, generator=gen, device="cuda") + 0.5

    def call(**kw):
        out = grpo.grpo_loss_fwd_bwd(x, ids, mask, advantages=adv, loss_norm=1.0, dlogits=torch.full_like(x, 7.0), **kw)
        return out.dlogits.flatten(0, 1), out.logp.flatten()

    got, want = call(), call(force_streaming=True)
    assert bool(((got[1] - want[1]).abs() <= 1e-5 * want[1].abs()).all())
    top = want[0].float().abs().amax(1)
    assert bool(((got[0].float() - want[0].float()).abs().amax(1) <= 2 ** -8 * top).all())
    assert bool(((mask.flatten() > 0) == (top > 0)).all())


PARTS_CASES = [("bf16", 32768, "bf16"), ("bf16", 50257, "bf16"), ("bf16", 151936, "bf16"), ("bf16", 151937, "bf16"),
               ("bf16", 65544, "f32"), ("bf16", 262152, "bf16"), ("f32", 16384, "f32"), ("f32", 50257, "f32"),
               ("f32", 151936, "f32"), ("f16", 50257, "f16"), ("f16", 32776, "f32")]


@pytest.mark.parametrize("zero_fill", [True, False])
@pytest.mark.parametrize("dt,V,odt", PARTS_CASES, ids=[f"{c[0]}-{c[1]}-{c[2]}" for c in PARTS_CASES])
def test_few_rows_in_parts_and_many_whole(dt, V, odt, zero_fill):
    """Wide rows of a small call run in parts, each dlogit the f32 result rounded once; among more
    rows (1,600 here) the same rows run one to a workgroup (or stream). Both against the oracle:
    the narrowest vocabularies in parts, ragged last parts, rows off 16 bytes, a shifted layout,
    targets in the first and the last vector and in the head and tail, dead and ignored rows."""
    rng = np.random.default_rng(V + len(odt))
    S, T = 3, 5
    rows, off = T - 1, 1
    x32 = rng.standard_normal((S, T, V)).astype(np.float32) * 3
    r32 = x32 + rng.standard_normal((S, T, V)).astype(np.float32) * 0.1
    to, code = {"f32": (np.float32, orc.F32), "f16": (np.float16, orc.F16), "bf16": (orc.bf16_from_f32, orc.BF16)}[dt]
    x, ref = (a.copy() if dt == "f32" else to(a) for a in (x32, r32))
    ids = rng.integers(0, V, size=(S, T)).astype(np.int64)
    ids[0, 1:] = [0, V - 1, V // 2, 7]
    ids[1, 2] = -100
    mask = (np.arange(T)[None] < np.array([5, 5, 3])[:, None]).astype(np.float32)
    adv = np.array([0.75, -1.25, 0.5], np.float32)
    old = np.zeros((S, T), np.float32)
    lp, _ = orc.logprob(np.ascontiguousarray(x[:, :rows]).reshape(S * rows, V), np.clip(ids[:, 1:].reshape(-1), 0, None),
                        dtype=code)
    old[:, 1:] = lp.reshape(S, rows) + rng.standard_normal((S, rows)) * 0.05
    want = orc.grpo_full(x, ids, mask, rows=rows, tok_offset=off, advantages_in=adv, ref_logits=ref, old_logp=old,
                         loss_mode=orc.CLIP_KL, loss_norm=3.0, dtype=code)
    ts = token_scale(x, ids, rows, off, code)
    fl = tok_to_rows(full_floor(want, mask, old, S, False, 0.04, 0.2, ts), rows, off, T)
    dead = np.ones((S, T), bool)
    dead[:, :rows] = (mask[:, 1:] == 0) | (ids[:, 1:] == -100)
    tdt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[odt]

    def padded(a, n):   # n - S sequences of masked tokens after the case's own
        a = dev(a)
        return torch.cat([a, torch.zeros((n - S, *a.shape[1:]), dtype=a.dtype, device=DEV)])

    for n in (S, 320):
        print(f"rows in parts / whole: {dt}->{odt} V={V} sequences={n} zero_fill={zero_fill}", flush=True)
        dl = torch.full((n, T, V), -3.5, dtype=tdt, device=DEV)
        out = grpo.grpo_loss_fwd_bwd(padded(x, n), padded(ids, n), padded(mask, n), advantages=padded(adv, n),
                                     ref_logits=padded(ref, n), old_logp=padded(old, n), rows=rows, tok_offset=off,
                                     loss_mode=LossMode.GRPO_CLIP_KL, loss_norm=3.0, dlogits=dl, zero_fill=zero_fill)
        assert np.all(np.abs(out.logp[:S].cpu().numpy()[:, 1:] - want.lp[:, 1:]) <= 1e-5 * ts[:, 1:])
        assert abs(float(out.loss.cpu()) - want.loss) <= full_loss_tol(want, x, ids, mask, rows, off, code, False,
                                                                       0.04, S)
        bits = host_bits(out.dlogits[:S])
        got = orc.bf16_to_f32(bits) if odt == "bf16" else bits
        assert_dlogits(got[~dead], want.dlogits[~dead], fl[~dead], odt != "f32", exact=n == S, f16_out=odt == "f16")
        fill = 0.0 if zero_fill else -3.5
        assert np.all(got[dead] == fill) and bool((dl[S:] == fill).all())


@pytest.mark.parametrize("dt,V", [("bf16", 50257), ("bf16", 151936), ("f32", 50257)])
def test_rows_in_parts_in_place(dt, V):
    """dlogits written over the logits: the same bits as into a buffer of their own, with targets
    in every part of the row and in its head and tail."""
    gen = torch.Generator(device=DEV).manual_seed(V)
    S, T = 4, 48
    x = (torch.randn((S, T, V), generator=gen, device=DEV) * 3).to({"bf16": torch.bfloat16, "f32": torch.float32}[dt])
    ref = (x.float() + 0.1 * torch.randn((S, T, V), generator=gen, device=DEV)).to(x.dtype)
    ids = torch.linspace(0, V - 1, S * T, device=DEV).long().view(S, T)
    mask = (torch.arange(T, device=DEV)[None] < torch.tensor([[48], [31], [48], [9]], device=DEV)).float()
    kw = dict(advantages=torch.tensor([0.75, -1.25, 0.5, 1.0], device=DEV), ref_logits=ref,
              old_logp=-torch.rand((S, T), generator=gen, device=DEV) * 9, loss_mode=LossMode.GRPO_CLIP_KL)
    want = grpo.grpo_loss_fwd_bwd(x, ids, mask, dlogits=torch.empty_like(x), **kw)
    f32 = dict(dtype=torch.float32, device=DEV)
    # The new log-probs over the old ones.
    over = grpo.GrpoOutputs(loss=torch.zeros((), **f32), dlogits=torch.empty_like(x), logp=kw["old_logp"].clone(),
                            ref_logp=torch.zeros((S, T), **f32), token_loss=torch.zeros((S, T), **f32),
                            advantages=torch.zeros(S, **f32))
    got = grpo.grpo_loss_fwd_bwd(x, ids, mask, outputs=over, **{**kw, "old_logp": over.logp})
    for f in ("loss", "dlogits", "logp", "ref_logp", "token_loss"):
        assert torch.equal(getattr(got, f), getattr(want, f)), f
    got = grpo.grpo_loss_fwd_bwd(x, ids, mask, dlogits=x, **kw)
    for f in ("loss", "dlogits", "logp", "ref_logp", "token_loss"):
        assert torch.equal(getattr(got, f), getattr(want, f)), f


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("V", [32776, 95992, 151944])
def test_f32_dlogits_of_16_bit_rows_in_parts(dt, V):
    """f32 dlogits of 16-bit logits in parts against c * (onehot - softmax) in 64 bits, with targets
    all over the row (both halves of a wave's slots, ragged last parts) and a dead row. A term is
    one exponential of an argument below 40 in f32: 2^-24 * 40 * ln 2 of it, under 1e-5 of |c|."""
    gen = torch.Generator(device=DEV).manual_seed(V)
    S, T = 2, 41
    x = (torch.randn((S, T, V), generator=gen, device=DEV) * 3).to({"bf16": torch.bfloat16, "f16": torch.float16}[dt])
    ids = torch.linspace(0, V - 1, S * T, device=DEV).long().view(S, T)
    mask = torch.ones((S, T), device=DEV)
    mask[1, 7] = 0
    adv = torch.tensor([0.75, -1.25], device=DEV)
    out = grpo.grpo_loss_fwd_bwd(x, ids, mask, advantages=adv, dlogits=torch.full((S, T, V), 7.0, device=DEV))
    c = (-adv.double() / (S * mask.double().sum(1)))[:, None] * mask.double()
    want = -torch.softmax(x.double(), -1)
    want.scatter_add_(2, ids[..., None], torch.ones_like(want[..., :1]))
    want *= c[..., None]
    err = (out.dlogits.double() - want).abs().amax(-1)
    assert bool((err <= 1e-5 * c.abs()).all())


def test_async_logprobs_share_a_context():
    """Log-probs enqueued on several streams through one context, beside losses and a synchronous
    call: each gives the bits that it gives alone (they use no memory of the context)."""
    gen = torch.Generator(device=DEV).manual_seed(4)
    V, sizes = 151936, [150, 40, 97, 64]
    x = [torch.randn((1, n, V), generator=gen, device=DEV).to(torch.bfloat16) for n in sizes]
    ids = [torch.randint(0, V, (1, n), generator=gen, device=DEV) for n in sizes]
    ctx = grpo.Context(0)
    want = []
    for a, i in zip(x, ids):
        want.append(grpo.logprob_fwd(a, i, sync=False, ctx=ctx)[0])
        ctx.sync()
    kw = dict(advantages=torch.ones(1, device=DEV), dlogits=torch.empty_like(x[0]), ctx=ctx)
    loss = grpo.grpo_loss_fwd_bwd(x[0], ids[0], **kw)
    lp, dl = loss.logp.clone(), loss.dlogits.clone()
    streams = [torch.cuda.Stream() for _ in sizes]
    torch.cuda.synchronize()
    for rep in range(5):
        print(f"overlapping log-probs {rep}", flush=True)
        with torch.cuda.stream(streams[0]):
            loss = grpo.grpo_loss_fwd_bwd(x[0], ids[0], sync=False, **kw)
        got = []
        for s, a, i in zip(streams[1:], x[1:], ids[1:]):
            with torch.cuda.stream(s):
                got.append(grpo.logprob_fwd(a, i, sync=False, ctx=ctx)[0])
        alone = grpo.logprob_fwd(x[3], ids[3], ctx=ctx)[0]
        ctx.sync()
        torch.cuda.synchronize()
        assert all(torch.equal(g, w) for g, w in zip(got, want[1:]))
        assert torch.equal(loss.logp, lp) and torch.equal(loss.dlogits, dl)
        assert bool(((alone - want[3]).abs() <= 1e-5 * want[3].abs()).all())


def test_logprobs_of_several_threads():
    """Synchronous log-probs of two threads, each on its own stream, through one context. The
    library's calls run outside the interpreter lock, so they overlap."""
    gen = torch.Generator(device=DEV).manual_seed(5)
    V, n = 151936, 96
    x = [torch.randn((1, n, V), generator=gen, device=DEV) for _ in range(2)]
    ids = [torch.randint(0, V, (1, n), generator=gen, device=DEV) for _ in range(2)]
    want = [torch.log_softmax(a.double(), -1).gather(2, i[..., None])[..., 0] for a, i in zip(x, ids)]
    ctx = grpo.Context(0)
    torch.cuda.synchronize()
    worst = [0.0, 0.0]

    def work(k):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(50):
                lp, _ = grpo.logprob_fwd(x[k], ids[k], ctx=ctx)
                worst[k] = max(worst[k], float(((lp - want[k]) / want[k]).abs().max()))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert max(worst) <= 1e-6


@pytest.mark.parametrize("S,T,V,kw", [(2, 6, 1000, {}), (2, 6, 5003, dict(force_streaming=True)), (2, 6, 50257, {}),
                                      (2, 400, 33000, {})], ids=["resident", "streaming", "parts", "wide"])
def test_target_of_probability_zero(S, T, V, kw):
    """A live token whose own logit is -inf (masked vocabulary) on-policy: rho = exp(lp - lp) is NaN
    for it, as in the oracle; other rows are untouched."""
    gen = torch.Generator(device=DEV).manual_seed(6)
    x = torch.randn((S, T, V), generator=gen, device=DEV)
    ids = torch.randint(0, V, (S, T), generator=gen, device=DEV)
    x[1, 2, ids[1, 2]] = -float("inf")
    ref = x + 0.1 * torch.randn((S, T, V), generator=gen, device=DEV)
    ref[1, 2, ids[1, 2]] = 0.0
    adv = torch.tensor([0.5, -0.5], device=DEV)
    out = grpo.grpo_loss_fwd_bwd(x, ids, advantages=adv, ref_logits=ref, loss_mode=LossMode.GRPO_CLIP_KL, **kw)
    few = slice(0, 4)                                    # rows are independent: the oracle takes the first few
    want = orc.grpo_full(x[:, few].cpu().numpy(), ids[:, few].cpu().numpy(), np.ones((S, 4), np.float32), rows=4,
                         advantages_in=adv.cpu().numpy(), ref_logits=ref[:, few].cpu().numpy(),
                         loss_mode=orc.CLIP_KL, dtype=orc.F32)
    bad = np.zeros((S, T), bool)
    bad[1, 2] = True
    assert np.isnan(want.token_loss[1, 2]) and np.isfinite(np.delete(want.token_loss.ravel(), 4 + 2)).all()
    assert np.array_equal(np.isnan(out.token_loss.cpu().numpy()), bad)
    assert float(out.logp[1, 2]) == -float("inf")
    assert np.array_equal(torch.isnan(out.dlogits).any(-1).cpu().numpy(), bad)


@pytest.mark.parametrize("V,lo,hi", [(50257, 0, 17000), (50257, 33000, 50257), (33000, 11000, 22000), (33000, 0, 32999)])
@pytest.mark.parametrize("dt", ["bf16", "f32"])
def test_rows_in_parts_with_masked_vocabulary(dt, V, lo, hi):
    """A whole part of a row at -inf (with the row's head or tail off 16 bytes), and all of it but
    one entry: log-probs and dlogits against 64 bits, zeros where the probability is."""
    gen = torch.Generator(device=DEV).manual_seed(V + lo)
    x = torch.randn((2, 9, V), generator=gen, device=DEV).to({"bf16": torch.bfloat16, "f32": torch.float32}[dt])
    x[0, 2, lo:hi] = -float("inf")
    ids = torch.randint(0, V, (2, 9), generator=gen, device=DEV)
    ids[0, 2] = hi if hi < V else 5
    adv = torch.tensor([0.75, -1.25], device=DEV)
    out = grpo.grpo_loss_fwd_bwd(x, ids, advantages=adv)
    lp = torch.log_softmax(x.double(), -1)
    want_lp = lp.gather(2, ids[..., None])[..., 0]
    assert bool(((out.logp - want_lp).abs() <= 1e-6 * want_lp.abs().clamp(min=1)).all())
    want = lp.exp().neg()
    want.scatter_add_(2, ids[..., None], torch.ones_like(want[..., :1]))
    want *= -adv.double()[:, None, None] / (2 * 9)
    rel = 2.0 ** -8 if dt == "bf16" else 2.0 ** -16
    assert bool(((out.dlogits.double() - want).abs() <= rel * want.abs() + 1e-7).all())
    assert bool((out.dlogits[0, 2, lo:hi] == 0).all())
