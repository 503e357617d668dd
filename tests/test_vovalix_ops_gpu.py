"""Every mechanism of the Vovalix decoder alone: the kernel against the plain function of
``tests/plain/vovalix.py``, at sizes of the tests' own, whole and in steps, beside other
requests and padding, from slots that hold another request's leftovers, with inputs made so
that a far token, a chunk's edge or a lost state shows."""

from __future__ import annotations

import math

import pytest
import torch

from tests.plain import vovalix as plain
from tests.vovalix_helpers import batch_tensors

pytestmark = pytest.mark.gpu

DEV = "cuda"


def gpu(t, dtype=torch.float32):
    return t.to(device=DEV, dtype=dtype).contiguous()


def rel(got, want):
    return float((got.double().cpu() - want).pow(2).mean().sqrt() / (want.pow(2).mean().sqrt() + 1e-30))


# ------------------------------------------------------------------ the matrix state
def new_state(slots, heads, dim, vdim, fill=float("nan")):
    """Slots as the engine keeps them (NaN where a request must not read: another's leftovers)."""
    from kvcore_amd.ops import library as ops

    return torch.full((slots, heads, ops.linear_state_rows(dim), vdim), fill, device=DEV)


def run_scan(q, k, v, decay, beta, state, reqs, *, heads, qk_heads, dim, vdim, delta, q_scale=1.0):
    from kvcore_amd.ops import library as ops

    batch, T = batch_tensors(reqs)
    out = torch.full((T, heads * vdim), float("nan"), device=DEV)
    ops.linear_state_scan(out, q, k, v, decay, beta, state, heads=heads, qk_heads=qk_heads, dim=dim, vdim=vdim,
                          delta_rule=delta, q_scale=q_scale, **batch)
    return out


@pytest.mark.parametrize("heads,qk_heads,dim,vdim", [(3, 3, 24, 40), (1, 1, 8, 5), (2, 2, 200, 80), (4, 4, 64, 64),
                                                       (2, 2, 32, 130)])
def test_key_decay_recurrence_whole_in_steps_and_beside_others(heads, qk_heads, dim, vdim):
    gen = torch.Generator().manual_seed(dim + vdim)
    T = 83
    q = torch.randn(T, heads, dim, generator=gen, dtype=torch.float64)
    k = torch.randn(T, heads, dim, generator=gen, dtype=torch.float64) * 0.5
    v = torch.randn(T, heads, vdim, generator=gen, dtype=torch.float64)
    a = torch.rand(T, heads, dim, generator=gen, dtype=torch.float64) * 0.5 + 0.5
    want = torch.stack([plain.gated_linear_recurrence(q[:, h] * 0.3, k[:, h], v[:, h], a[:, h]) for h in range(heads)], 1)
    want = want.reshape(T, -1)
    qg, kg, vg, ag = (gpu(t.reshape(T, -1)) for t in (q, k, v, a))
    kw = dict(heads=heads, qk_heads=qk_heads, dim=dim, vdim=vdim, delta=False, q_scale=0.3)
    # the slots hold another request's leftovers (NaN where nothing may be read)
    state = new_state(3, heads, dim, vdim)
    out = run_scan(qg, kg, vg, ag, None, state, [(1, 0, T)], **kw)
    assert rel(out, want) < 2e-6
    # in steps of every size down to one token, cut inside the stages of 16
    state = new_state(3, heads, dim, vdim)
    at, got = 0, []
    for n in (2, 1, 17, 3, 1, 16, 31, 2, 10):
        got.append(run_scan(qg[at:at + n], kg[at:at + n], vg[at:at + n], ag[at:at + n], None, state, [(2, at, n)], **kw))
        at += n
    assert at == T
    assert rel(torch.cat(got), want) < 2e-6
    # beside a padded row and another request that is further on: rows [other | pad | this]
    other = new_state(3, heads, dim, vdim, 0.0)
    mixed_q = torch.cat([qg[40:41], qg[:1], qg[:20]])
    mixed_k = torch.cat([kg[40:41], kg[:1], kg[:20]])
    mixed_v = torch.cat([vg[40:41], vg[:1], vg[:20]])
    mixed_a = torch.cat([ag[40:41], ag[:1], ag[:20]])
    run_scan(qg[:40], kg[:40], vg[:40], ag[:40], None, other, [(0, 0, 40)], **kw)
    out = run_scan(mixed_q, mixed_k, mixed_v, mixed_a, None, other, [(0, 40, 1), None, (1, 0, 20)], **kw)
    assert rel(out[0:1], want[40:41]) < 2e-6 and rel(out[2:], want[:20]) < 2e-6
    assert float(out[1].abs().max()) == 0.0


@pytest.mark.parametrize("heads,qk_heads,dim,vdim", [(4, 2, 24, 20), (1, 1, 8, 1), (3, 1, 8, 1), (2, 1, 130, 72),
                                                       (2, 2, 64, 64)])
def test_delta_rule_whole_in_steps_and_beside_others(heads, qk_heads, dim, vdim):
    gen = torch.Generator().manual_seed(dim * 3 + vdim)
    T = 70
    q = plain.unit_vector(torch.randn(T, qk_heads, dim, generator=gen, dtype=torch.float64))
    k = plain.unit_vector(torch.randn(T, qk_heads, dim, generator=gen, dtype=torch.float64))
    v = torch.randn(T, heads, vdim, generator=gen, dtype=torch.float64)
    beta = torch.rand(T, heads, generator=gen, dtype=torch.float64)
    g = torch.rand(T, heads, generator=gen, dtype=torch.float64) * 0.3 + 0.7
    rep = heads // qk_heads
    want = torch.stack([plain.delta_recurrence(q[:, h // rep], k[:, h // rep], v[:, h], beta[:, h], g[:, h])
                        for h in range(heads)], 1).reshape(T, -1)
    qg, kg, vg = (gpu(t.reshape(T, -1)) for t in (q, k, v))
    bg, gg = gpu(beta), gpu(g)
    kw = dict(heads=heads, qk_heads=qk_heads, dim=dim, vdim=vdim, delta=True)
    state = new_state(2, heads, dim, vdim)
    out = run_scan(qg, kg, vg, gg, bg, state, [(1, 0, T)], **kw)
    assert rel(out, want) < 5e-6
    state = new_state(2, heads, dim, vdim)
    at, got = 0, []
    for n in (1, 2, 16, 1, 19, 2, 29):
        got.append(run_scan(qg[at:at + n], kg[at:at + n], vg[at:at + n], gg[at:at + n], bg[at:at + n], state,
                            [(0, at, n)], **kw))
        at += n
    assert at == T
    assert rel(torch.cat(got), want) < 5e-6
    # a column view of a wider row, as the mixers hand their projections over
    wide = torch.cat([qg, kg, vg], dim=1).contiguous()
    nq = qk_heads * dim
    state = new_state(2, heads, dim, vdim, 0.0)
    out = run_scan(wide[:, :nq], wide[:, nq:2 * nq], wide[:, 2 * nq:], gg, bg, state, [(0, 0, T)], **kw)
    assert rel(out, want) < 5e-6


@pytest.mark.parametrize("rule", ["decay", "delta", "gates"])
@pytest.mark.parametrize("heads,dim,vdim", [(2, 32, 16), (2, 64, 40), (1, 128, 130), (70, 32, 64)])
def test_whole_stages_of_tokens_give_the_bits_of_single_ones(rule, heads, dim, vdim):
    """Stages of sixteen tokens keep a token's values in registers ahead of the work; one token at a time is the way without: the same
    products and sums in the same order."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(dim + vdim)
    T = 48
    unit = lambda: gpu(plain.unit_vector(torch.randn(T, heads, dim, generator=gen, dtype=torch.float64)).reshape(T, -1))
    q, k = unit(), unit()
    v = gpu(torch.randn(T, heads * vdim, generator=gen))
    beta = gpu(torch.rand(T, heads, generator=gen))
    decay = gpu(torch.rand(T, heads * (dim if rule == "decay" else 1), generator=gen) * 0.3 + 0.7)

    def scan(state, first, n):
        batch, _ = batch_tensors([(0, first, n)])
        out = torch.full((n, heads * vdim), float("nan"), device=DEV)
        at = slice(first, first + n)
        ops.linear_state_scan(out, q[at], k[at], v[at], decay[at], None if rule == "decay" else beta[at], state, heads=heads,
                              qk_heads=heads, dim=dim, vdim=vdim, delta_rule=rule == "delta", scalar_gates=rule == "gates", **batch)
        return out

    whole, single = new_state(1, heads, dim, vdim), new_state(1, heads, dim, vdim)
    out = scan(whole, 0, T)
    assert torch.equal(out, torch.cat([scan(single, t, 1) for t in range(T)]))
    assert torch.equal(whole, single)


@pytest.mark.parametrize("rule", ["decay", "delta", "gates"])
@pytest.mark.parametrize("dim", [64, 256])
def test_chains_that_leave_room_for_one_two_and_more_on_a_unit(rule, dim):
    """128, 256 and 384 blocks ask for different shares of a unit's LDS: the first request has the same bits in each, and without any."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(dim)
    heads, vdim, n = 16, 128, 37
    asked = [ops.load().kvc_linear_state_scan_lds(128 * R) for R in (1, 2, 3)]
    assert asked[0] > asked[1] > asked[2] == 0
    unit = lambda: gpu(plain.unit_vector(torch.randn(3 * n, heads, dim, generator=gen, dtype=torch.float64)).reshape(3 * n, -1))
    q, k = unit(), unit()
    v = gpu(torch.randn(3 * n, heads * vdim, generator=gen))
    beta = gpu(torch.rand(3 * n, heads, generator=gen))
    decay = gpu(torch.rand(3 * n, heads * (dim if rule == "decay" else 1), generator=gen) * 0.3 + 0.7)
    got = []
    for R, chains in ((1, 0), (1, 1), (2, 2), (3, 3), (3, 1)):
        batch, T = batch_tensors([(r, 0, n) for r in range(R)])
        state = new_state(3, heads, dim, vdim)
        out = torch.full((T, heads * vdim), float("nan"), device=DEV)
        ops.linear_state_scan(out, q[:T], k[:T], v[:T], decay[:T], None if rule == "decay" else beta[:T], state, heads=heads,
                              qk_heads=heads, dim=dim, vdim=vdim, delta_rule=rule == "delta", scalar_gates=rule == "gates", chains=chains, **batch)
        got.append((out[:n], state[0]))
    assert torch.isfinite(got[0][0]).all()
    for out, state in got[1:]:
        assert torch.equal(out, got[0][0]) and torch.equal(state, got[0][1])


def test_a_token_written_six_hundred_tokens_ago_is_still_read():
    """A decay of almost one: the first token's value, written at a key of its own, comes back
    for a query of that key 600 tokens later (in one step, and token by token), scaled by the
    decay's 600th power; with the state lost on the way it would be zero."""
    T, d, dv = 601, 16, 8
    gen = torch.Generator().manual_seed(4)
    k = torch.randn(T, 1, d, generator=gen, dtype=torch.float64) * 0.05
    k[:, 0, 0] = 0.0
    k[0, 0] = 0.0
    k[0, 0, 0] = 1.0  # channel 0 is the first token's alone
    v = torch.randn(T, 1, dv, generator=gen, dtype=torch.float64)
    q = torch.zeros(T, 1, d, dtype=torch.float64)
    q[:, 0, 0] = 1.0
    a = torch.full((T, 1, d), 0.999, dtype=torch.float64)
    want = plain.gated_linear_recurrence(q[:, 0], k[:, 0], v[:, 0], a[:, 0])
    assert torch.allclose(want[600], v[0, 0] * 0.999 ** 600, atol=1e-9)
    qg, kg, vg, ag = (gpu(t.reshape(T, -1)) for t in (q, k, v, a))
    kw = dict(heads=1, qk_heads=1, dim=d, vdim=dv, delta=False)
    state = new_state(1, 1, d, dv)
    out = run_scan(qg, kg, vg, ag, None, state, [(0, 0, T)], **kw)
    assert rel(out[600], want[600]) < 1e-4
    state = new_state(1, 1, d, dv)
    run_scan(qg[:300], kg[:300], vg[:300], ag[:300], None, state, [(0, 0, 300)], **kw)
    for t in range(300, T):
        out = run_scan(qg[t:t + 1], kg[t:t + 1], vg[t:t + 1], ag[t:t + 1], None, state, [(0, t, 1)], **kw)
    assert rel(out[0], want[600]) < 1e-4


def test_small_kernels_around_the_recurrences():
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(8)
    T = 37
    # sigmoid(z + b) ^ (1 / tau), through the logarithm, also far out in the tails
    z = torch.randn(T, 48, generator=gen, dtype=torch.float64) * 6
    b = torch.randn(48, generator=gen, dtype=torch.float64)
    out = torch.empty(T, 48, device=DEV)
    ops.sigmoid_power(out, gpu(z), gpu(b), 1 / 12.0)
    assert rel(out, torch.sigmoid(z + b).pow(1 / 12.0)) < 1e-6
    # decay and write strength of the delta rule
    a_raw, b_raw = (torch.randn(T, 5, generator=gen, dtype=torch.float64) * 3 for _ in range(2))
    a_log, dt_bias = (torch.randn(5, generator=gen, dtype=torch.float64) for _ in range(2))
    g, beta = torch.empty(T, 5, device=DEV), torch.empty(T, 5, device=DEV)
    wide = gpu(torch.cat([a_raw, b_raw], 1))
    ops.decay_and_write_gates(g, beta, wide[:, :5], wide[:, 5:], gpu(a_log), gpu(dt_bias))
    assert rel(g, torch.exp(-torch.exp(a_log) * plain.softplus(a_raw + dt_bias))) < 1e-6
    assert rel(beta, torch.sigmoid(b_raw)) < 1e-6
    # unit vectors per head, in place, in a column view
    x = torch.randn(T, 3 * 24 + 7, generator=gen, dtype=torch.float64)
    xg = gpu(x)
    ops.unit_heads(xg[:, :72], 3, 24, 1e-6, 24 ** -0.5)
    want = plain.unit_vector(x[:, :72].reshape(T, 3, 24)).reshape(T, 72) * 24 ** -0.5
    assert rel(xg[:, :72], want) < 1e-6 and torch.equal(xg[:, 72:].cpu().double(), x[:, 72:].float().double())
    # the first heads with a scale of their own (q before k in one launch)
    xg = gpu(x)
    ops.unit_heads(xg[:, :72], 3, 24, 1e-6, 1.0, first_heads=1, first_scale=0.25)
    want = plain.unit_vector(x[:, :72].reshape(T, 3, 24))
    want[:, 0] *= 0.25
    assert rel(xg[:, :72], want.reshape(T, 72)) < 1e-6
    # the head norm with its gate, heads of 40 and of 1 and of 130 values
    for heads, dv in ((3, 40), (4, 1), (2, 130)):
        o = torch.randn(T, heads, dv, generator=gen, dtype=torch.float64)
        gate = torch.randn(T, heads * dv, generator=gen, dtype=torch.float64)
        gain = torch.randn(dv, generator=gen, dtype=torch.float64)
        want = (plain.rms_unit(o, 1e-5) * gain).reshape(T, -1) * plain.silu(gate)
        for dtype, tol in ((torch.float32, 2e-6), (torch.bfloat16, 6e-3)):
            out = torch.empty(T, heads * dv, device=DEV, dtype=dtype)
            gate_rows = gpu(gate) if dtype == torch.float32 else gpu(gate, torch.bfloat16)
            ref = want if dtype == torch.float32 else (plain.rms_unit(o, 1e-5) * gain).reshape(T, -1) * plain.silu(
                gate.to(torch.bfloat16).double())
            ops.head_rmsnorm_gate(out, gpu(o.reshape(T, -1)), gate_rows, gpu(gain), 1e-5, heads, dv)
            assert rel(out, ref) < tol
    # the experts' activation
    gu = torch.randn(T, 2 * 24, generator=gen, dtype=torch.float64) * 3
    out = torch.empty(T, 24, device=DEV)
    ops.clamped_glu(out, gpu(gu), 1.3, 1.702)
    gg, uu = torch.clamp(gu[:, :24], max=1.3), torch.clamp(gu[:, 24:], -1.3, 1.3)
    assert rel(out, gg * torch.sigmoid(1.702 * gg) * (uu + 1)) < 1e-6


@pytest.mark.parametrize("act", ["sigmoid", "silu"])
def test_sigmoid_and_silu_have_the_division_s_bits_for_every_float32(act):
    """All 2^32 values as gates of rows whose norm is one: a reciprocal and a correction in the kernel, a division here."""
    from kvcore_amd.ops import library as ops

    T, heads, dim = 65536, 16, 64
    ones, gain = torch.ones(T, heads * dim, device=DEV), torch.ones(dim, device=DEV)
    out = torch.empty_like(ones)
    count = ones.numel()
    for first in range(-2 ** 31, 2 ** 31, count):
        gate = torch.arange(first, first + count, dtype=torch.int64, device=DEV).to(torch.int32).view(torch.float32).view(T, -1)
        ops.head_rmsnorm_gate(out, ones, gate, gain, 0.0, heads, dim, act=act)
        want = (gate if act == "silu" else ones) / (1.0 + torch.exp(-gate))
        same = (out.view(torch.int32) == want.view(torch.int32)) | (out.isnan() & want.isnan())
        assert bool(same.all()), (first, gate[~same][:4].tolist(), out[~same][:4].tolist(), want[~same][:4].tolist())


# ------------------------------------------------------------------------- attention
def paged(q, k, v, page, *, scale, slopes, chunk, dtype, positions=None, shuffle=True, kernel="general"):
    """Attention of ``q [T, H, d]`` (tokens at ``positions``, default 0..T-1) over keys and values
    ``k, v [S, G, d / dv]`` laid into pages in a shuffled order, through the general kernel, or
    (bfloat16) the matrix-core kernel for portions (``"portion"``) or for single tokens
    (``"single"``, one launch a token)."""
    from kvcore_amd.ops import library as ops

    S, G, d = k.shape
    dv = v.shape[2]
    T, H, _ = q.shape
    n_pages = -(-S // page)
    order = torch.randperm(n_pages, generator=torch.Generator().manual_seed(1)) if shuffle else torch.arange(n_pages)
    k_cache = torch.full((n_pages + 1, G, page, d), float("nan"), dtype=dtype, device=DEV)
    v_cache = torch.full((n_pages + 1, G, dv, page), float("nan"), dtype=dtype, device=DEV)
    table = torch.zeros((2, n_pages), dtype=torch.int32, device=DEV)
    for p in range(n_pages):
        pid = int(order[p]) + 1
        table[1, p] = pid
        n = min(page, S - p * page)
        k_cache[pid, :, :n] = gpu(k[p * page:p * page + n].transpose(0, 1), dtype)
        v_cache[pid, :, :, :n] = gpu(v[p * page:p * page + n].permute(1, 2, 0), dtype)
    pos = list(range(T)) if positions is None else positions
    out = torch.empty(T, H * dv, dtype=dtype, device=DEV)
    slope_t = None if slopes is None else gpu(torch.tensor(slopes))
    if kernel == "portion":
        assert ops.prefill_attention_supported(H, G, d, page, dtype) and dv == d
        ops.prefill_attention(out, gpu(q.reshape(T, -1), dtype), k_cache, v_cache, table=table,
                              positions=torch.tensor(pos, dtype=torch.int32, device=DEV),
                              q_start=torch.tensor([0, T], dtype=torch.int32, device=DEV),
                              slots=torch.tensor([1], dtype=torch.int32, device=DEV), num_reqs=1, nh=H, nkv=G, d=d,
                              scale=scale, slopes=slope_t, chunk=chunk)
        assert ops.last_variant("prefill_attention").startswith("prefill_attention_kernel")
        return out.double().cpu().view(T, H, dv)
    if kernel == "single":
        assert ops.decode_attention_supported(H, G, d, page, dtype) and dv == d
        for i in range(T):
            ops.decode_attention(out[i:i + 1], gpu(q[i:i + 1].reshape(1, -1), dtype), k_cache, v_cache, table=table,
                                 positions=torch.tensor(pos[i:i + 1], dtype=torch.int32, device=DEV),
                                 token_req=torch.zeros(1, dtype=torch.int32, device=DEV),
                                 slots=torch.tensor([1], dtype=torch.int32, device=DEV), nh=H, nkv=G, d=d,
                                 scale=scale, slopes=slope_t, chunk=chunk)
        return out.double().cpu().view(T, H, dv)
    ops.paged_attention(out, gpu(q.reshape(T, -1), dtype), k_cache, v_cache, table=table,
                        positions=torch.tensor(pos, dtype=torch.int32, device=DEV),
                        token_req=torch.zeros(T, dtype=torch.int32, device=DEV),
                        slots=torch.tensor([1], dtype=torch.int32, device=DEV), nh=H, nkv=G, d=d, dv=dv,
                        scale=scale, slopes=None if slopes is None else gpu(torch.tensor(slopes)), chunk=chunk)
    return out.double().cpu().view(T, H, dv)


def normalised(x):
    """Heads with a mean square of exactly one, which the plain function's own norm leaves alone."""
    return x / x.pow(2).mean(dim=-1, keepdim=True).sqrt()


@pytest.mark.parametrize("H,G,d,dv,chunk,page", [(4, 2, 32, 16, 24, 8), (6, 6, 16, 16, 10, 16), (1, 1, 16, 32, 1, 4),
                                                  (2, 1, 16, 16, 0, 4), (3, 1, 48, 72, 100, 16)])
def test_chunked_attention_with_a_distance_bias(H, G, d, dv, chunk, page):
    gen = torch.Generator().manual_seed(H * 100 + chunk)
    T = 131
    q = normalised(torch.randn(T, H, d, generator=gen, dtype=torch.float64))
    k = normalised(torch.randn(T, G, d, generator=gen, dtype=torch.float64))
    v = torch.randn(T, G, dv, generator=gen, dtype=torch.float64)
    want = plain.chunked_distance_attention(q, k, v, 0.3, chunk or None, 0.0)
    got = paged(q, k, v, page, scale=0.3, slopes=plain.distance_slopes(H), chunk=chunk, dtype=torch.float32)
    assert rel(got, want) < 2e-6
    # the bias matters: without it the result differs
    flat = paged(q, k, v, page, scale=0.3, slopes=None, chunk=chunk, dtype=torch.float32)
    if chunk != 1:
        assert rel(flat, want) > 1e-3
    got = paged(q, k, v, page, scale=0.3, slopes=plain.distance_slopes(H), chunk=chunk, dtype=torch.bfloat16)
    qb, kb, vb = (t.to(torch.bfloat16).double() for t in (q, k, v))
    want_b = plain.chunked_distance_attention(qb, kb, vb, 0.3, chunk or None, 0.0)
    # q and k are rounded after their norm here, which moves their mean squares by 1e-3
    assert rel(got, want_b) < 2e-2


@pytest.mark.parametrize("single", [False, True], ids=["portion", "single"])
def test_a_key_that_stands_out_at_a_chunk_s_edges_and_far_back(single):
    """One key is made to outscore all others for every query.  A query sees it iff it lies in
    the query's chunk and not after it: the first position of the chunk (just inside), the last
    of the chunk before (just outside), a page's first and last slot, a key hundreds of tokens
    back in a long chunk.  The queries come as a portion of a prompt or as single tokens."""
    H, G, d, dv, page = 2, 1, 16, 8, 16
    for chunk, T, marked, query in ((64, 200, 64, 127), (64, 200, 63, 64), (64, 200, 128, 128), (64, 200, 127, 191),
                                    (400, 420, 0, 399), (400, 420, 15, 399), (400, 420, 16, 399), (400, 420, 399, 400),
                                    (0, 420, 3, 419), (48, 200, 95, 96), (48, 200, 96, 143), (48, 200, 96, 144)):
        gen = torch.Generator().manual_seed(marked + query)
        k = torch.randn(T, G, d, generator=gen, dtype=torch.float64) * 0.3
        k[:, 0, 0] = 0.0
        k[marked, 0] = 0.0
        k[marked, 0, 0] = 1.0
        v = torch.randn(T, G, dv, generator=gen, dtype=torch.float64)
        q = torch.randn(T, H, d, generator=gen, dtype=torch.float64) * 0.3
        q[:, :, 0] = 60.0
        visible = marked <= query and (chunk == 0 or marked // chunk == query // chunk)
        want = plain.chunked_distance_attention(normalised(q), normalised(k), v, 1.0, chunk or None, 0.0)
        # head 1's slope is 2^-8: the marked key wins even from 400 tokens away
        assert torch.allclose(want[query, 1], v[marked, 0], atol=1e-3) == visible
        qs = normalised(q)[query:query + 1] if single else normalised(q)[query - 2:query + 1]
        pos = [query] if single else [query - 2, query - 1, query]
        got = paged(qs, normalised(k), v, page, scale=1.0, slopes=plain.distance_slopes(H), chunk=chunk,
                    dtype=torch.float32, positions=pos)
        assert rel(got[-1], want[query]) < 1e-5, (chunk, marked, query)
        assert torch.allclose(got[-1, 1], v[marked, 0], atol=1e-3) == visible, (chunk, marked, query)


@pytest.mark.parametrize("kernel", ["portion", "single"])
@pytest.mark.parametrize("H,G,d,chunk", [(8, 2, 64, 48), (4, 4, 128, 0), (8, 1, 64, 200), (16, 2, 64, 1)])
def test_matrix_core_kernels_with_bias_and_chunks(kernel, H, G, d, chunk):
    """The bfloat16 kernels for portions and for single tokens against the plain function on the
    same rounded values: every position of a prompt of 300 tokens (chunks that are no multiple of
    the kernels' tiles of 16 and 64 keys, a chunk of one position, no chunk), then the key that
    stands out at a chunk's edges."""
    gen = torch.Generator().manual_seed(H + d + chunk)
    T, page = 300, 16
    q = normalised(torch.randn(T, H, d, generator=gen, dtype=torch.float64)).to(torch.bfloat16).double()
    k = normalised(torch.randn(T, G, d, generator=gen, dtype=torch.float64)).to(torch.bfloat16).double()
    v = torch.randn(T, G, d, generator=gen, dtype=torch.float64).to(torch.bfloat16).double()
    # the plain function norms again: take that out by its own factor (the rounded rows' mean squares are not 1)
    want = plain.chunked_distance_attention(q * q.pow(2).mean(-1, keepdim=True).sqrt(),
                                            k * k.pow(2).mean(-1, keepdim=True).sqrt(), v, 0.3, chunk or None, 0.0)
    rows = list(range(T)) if kernel == "portion" else [0, 1, 15, 16, 47, 48, 95, 96, 143, 144, 199, 200, 255, 256, 299]
    got = paged(q[rows] if kernel == "single" else q, k, v, page, scale=0.3, slopes=plain.distance_slopes(H),
                chunk=chunk, dtype=torch.bfloat16, positions=rows, kernel=kernel)
    assert rel(got, want[rows]) < 1e-2
    for size, marked, query in ((48, 95, 96), (48, 96, 143), (48, 96, 144), (48, 48, 95), (200, 0, 199), (200, 15, 199),
                                (200, 199, 200), (0, 3, 299)):
        k2 = (torch.randn(T, G, d, generator=gen, dtype=torch.float64) * 0.3)
        k2[:, :, 0] = 0.0
        k2[marked] = 0.0
        k2[marked, :, 0] = 1.0
        q2 = torch.randn(T, H, d, generator=gen, dtype=torch.float64) * 0.3
        q2[:, :, 0] = 60.0
        q2, k2 = normalised(q2).to(torch.bfloat16).double(), normalised(k2).to(torch.bfloat16).double()
        visible = marked <= query and (size == 0 or marked // size == query // size)
        rows = [query - 2, query - 1, query] if kernel == "portion" else [query]
        got = paged(q2[rows], k2, v, page, scale=1.0, slopes=plain.distance_slopes(H), chunk=size,
                    dtype=torch.bfloat16, positions=rows, kernel=kernel)
        # the last head's slope is 2^-8: the marked key wins even from 300 tokens away
        assert torch.allclose(got[-1, H - 1], v[marked, G - 1], atol=2e-2) == visible, (size, marked, query)


# --------------------------------------------------------------------- routed experts
@pytest.mark.parametrize("E,top,groups,keep", [(6, 2, 3, 2), (8, 3, 1, 1), (2, 2, 2, 2), (3, 1, 3, 1), (16, 4, 4, 1),
                                               (16, 4, 4, 2), (12, 3, 4, 3), (5, 5, 1, 1), (70, 6, 10, 3)])
def test_routing_against_the_plain_rule(E, top, groups, keep):
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(E * 7 + top)
    T = 57
    logits = torch.randn(T, E, generator=gen, dtype=torch.float64) * 2
    logits[3] = 0.0  # all equal: the lowest indices of the first groups
    logits = logits.float().double()
    choice = torch.empty(T, top, dtype=torch.int32, device=DEV)
    weight = torch.empty(T, top, dtype=torch.float32, device=DEV)
    ops.moe_route(choice, weight, gpu(logits), top=top, groups=groups, keep=keep)
    scores = torch.softmax(logits, dim=-1)
    for t in range(T):
        want_e, want_w = plain.route(scores[t], top, groups, keep)
        got_e = choice[t].tolist()
        live = min(top, keep * (E // groups))  # fewer allowed experts than choices: the rest weigh nothing
        assert got_e[:live] == want_e[:live], t
        assert torch.allclose(weight[t, :live].double().cpu(), want_w[:live], atol=1e-6), t
        assert float(weight[t, live:].abs().sum()) == 0.0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("E,top,groups,keep,H,T", [(6, 2, 3, 2, 96, 75), (32, 4, 8, 4, 256, 1100), (2, 2, 2, 2, 40, 1),
                                                   (70, 6, 10, 3, 130, 9), (130, 3, 1, 1, 64, 20)])
def test_router_product_and_choice_in_one_kernel(dtype, E, top, groups, keep, H, T):
    """The fused router against the plain rule on the same rows; the logits are float32 sums of the
    rows as they are, the same for a token alone and among a thousand (blocks of 4 and of 16 tokens)."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(E + T)
    x = torch.randn(T, H, generator=gen, dtype=torch.float64)
    x = x.to(dtype).double()
    w = (torch.randn(E, H, generator=gen, dtype=torch.float64) * 0.5).float().double()
    choice = torch.empty(T, top, dtype=torch.int32, device=DEV)
    weight = torch.empty(T, top, dtype=torch.float32, device=DEV)
    ops.moe_router(choice, weight, gpu(x, dtype), gpu(w), top=top, groups=groups, keep=keep)
    logits = x @ w.T
    scores = torch.softmax(logits, dim=-1)
    checked = 0
    for t in range(T):
        if plain.route_margin(logits[t], top, groups, keep) < 1e-4:
            continue  # a tie within float32's reach
        want_e, want_w = plain.route(scores[t], top, groups, keep)
        assert choice[t].tolist() == want_e, t
        assert torch.allclose(weight[t].double().cpu(), want_w, atol=1e-5), t
        checked += 1
    assert checked >= T * 0.9
    # a token's result does not depend on the batch: the first rows alone give the same bits
    n = min(T, 3)
    c2 = torch.empty(n, top, dtype=torch.int32, device=DEV)
    w2 = torch.empty(n, top, dtype=torch.float32, device=DEV)
    ops.moe_router(c2, w2, gpu(x[:n], dtype), gpu(w), top=top, groups=groups, keep=keep)
    assert torch.equal(c2, choice[:n]) and torch.equal(w2, weight[:n])


def expert_weights(E, H, I, gen, shared=0):
    w = {"router": torch.randn(E, H, generator=gen, dtype=torch.float64) * 0.5}
    for e in range(E):
        w[f"e{e}.gate"] = torch.randn(I, H, generator=gen, dtype=torch.float64) * 0.3
        w[f"e{e}.up"] = torch.randn(I, H, generator=gen, dtype=torch.float64) * 0.3
        w[f"e{e}.down"] = torch.randn(H, I, generator=gen, dtype=torch.float64) * 0.3
    if shared:
        w["shared.gate"] = torch.randn(shared, H, generator=gen, dtype=torch.float64) * 0.3
        w["shared.up"] = torch.randn(shared, H, generator=gen, dtype=torch.float64) * 0.3
        w["shared.down"] = torch.randn(H, shared, generator=gen, dtype=torch.float64) * 0.3
    return w


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("E,top,groups,keep,H,I,shared,T", [(6, 2, 3, 2, 96, 40, 56, 75), (8, 3, 1, 1, 128, 64, 0, 300),
                                                            (2, 2, 2, 2, 40, 8, 0, 1), (3, 1, 3, 1, 40, 16, 8, 2),
                                                            (16, 4, 4, 1, 64, 32, 32, 33), (5, 2, 1, 1, 36, 20, 12, 19),
                                                            (4, 2, 1, 1, 96, 32, 0, 200), (2, 1, 1, 1, 160, 96, 16, 150),
                                                            (2, 2, 2, 2, 64, 32, 0, 300), (3, 1, 1, 1, 96, 64, 24, 800)])
def test_the_feed_forward_of_routed_experts(dtype, E, top, groups, keep, H, I, shared, T):
    """The part itself on rows of its own: routing, the arrangement by expert, both products,
    the weighted sum and the shared expert, against the plain function token by token.  Sizes
    that 16-byte loads do not divide (36, 20, 12) take the kernel without them; many rows an expert
    take tiles of 64 rows (also with sums of 96, 160 and 32 terms, which end inside a pass of 64)."""
    from kvcore_amd.engine.context import StepBuffers, StepContext
    from kvcore_amd.parts.base import Runtime
    from kvcore_amd.parts.moe import RoutedExperts

    gen = torch.Generator().manual_seed(E + T)
    w = expert_weights(E, H, I, gen, shared)
    if dtype == torch.bfloat16:
        w = {k: (v if k == "router" else v.to(torch.bfloat16).double()) for k, v in w.items()}
    part = RoutedExperts(hidden_size=H, experts=E, top=top, expert_size=I, limit=1.2, groups=groups, keep=keep,
                         shared_size=shared, shared_limit=0.8,
                         tensor_names={"router": "router", "expert": "e{e}", "shared": "shared", "gate": "gate",
                                       "up": "up", "down": "down"})
    part.setup(Runtime(dtype=dtype, device=torch.device(DEV)))
    params = {}
    for ps in part.param_specs():
        t = torch.empty(ps.shape, dtype=torch.float32 if ps.kind == "vector" else dtype, device=DEV)
        for src in ps.resolved_sources():
            t[src.row:src.row + src.rows] = gpu(w[src.name], t.dtype)
        params[ps.name] = t
    part.bind(params)
    x = torch.randn(T, H, generator=gen, dtype=torch.float64)
    if dtype == torch.bfloat16:
        x = x.to(torch.bfloat16).double()
    mlp = {"router": {"experts": E, "top": top, "groups": {"count": groups, "keep": keep}},
           "expert": {"ff": I, "limit": 1.2}, "shared": {"ff": shared, "limit": 0.8} if shared else None}
    want = plain.moe_feed_forward(x, {f"p.{k}": v for k, v in w.items()}, "p", mlp)
    buffers = StepBuffers(torch.device(DEV), token_capacity=T)
    none = torch.zeros(1, dtype=torch.int32, device=DEV)
    ctx = StepContext(num_tokens=T, num_reqs=1, token_ids=none, positions=none, token_req=none, q_start=none,
                      seq_lens=none, slots=none, groups=[], states=[], buffers=buffers, dtype=dtype,
                      device=torch.device(DEV))
    out = part.forward(gpu(x, dtype), ctx, None)
    assert out.dtype == torch.float32 and out.shape == (T, H)
    assert rel(out, want) < (3e-6 if dtype == torch.float32 else 8e-3)
    # the form that adds into a stream, with another branch's rows taken along
    stream = torch.randn(T, H, generator=gen, dtype=torch.float64)
    other = torch.randn(T, H, generator=gen, dtype=torch.float64)
    first = out.double().cpu().clone()
    stream_gpu = gpu(stream)
    part.forward_into(stream_gpu, gpu(x, dtype), ctx, None, add=gpu(other))
    assert rel(stream_gpu, stream.float().double() + (other.float().double() + first)) < 1e-6
    # the same rows again among others, in another order: a row's result does not depend on its place
    out = part.forward(gpu(x, dtype), ctx, None)
    if T > 2:
        first = out.cpu().clone()  # the result lives in a step buffer that the next call rewrites
        perm = torch.randperm(T, generator=gen)
        again = part.forward(gpu(x[perm], dtype), ctx, None)
        assert rel(again, first[perm].double()) < 1e-6


@pytest.mark.parametrize("gated", [True, False], ids=["gated", "plain"])
@pytest.mark.parametrize("tile_rows", [16, 64, 128, 384])
@pytest.mark.parametrize("T", [1, 129, 700])
def test_experts_with_a_shared_one_of_their_size_beside_another_branch(monkeypatch, T, tile_rows, gated):
    """The part with its shared expert in the routed ones' launches, with and without another branch: the same bits, each against the
    weighted sum in 64 bits; the branch starts behind the mark."""
    from kvcore_amd.engine.context import StepBuffers, StepContext
    from kvcore_amd.ops import library as ops
    from kvcore_amd.parts.base import Runtime
    from kvcore_amd.parts.moe import RoutedExperts

    E, top, H, I = 6, 2, 192, 128
    gen = torch.Generator().manual_seed(T + tile_rows)
    part = RoutedExperts(hidden_size=H, experts=E, top=top, expert_size=I, limit=1.2, shared_size=I, shared_limit=0.8,
                         activation=None if gated else "relu_squared")
    part.setup(Runtime(dtype=torch.bfloat16, device=torch.device(DEV)))
    params = {}
    for ps in part.param_specs():
        t = torch.randn(ps.shape, generator=gen) * ps.shape[1] ** -0.5
        params[ps.name] = gpu(t, torch.float32 if ps.kind == "vector" else torch.bfloat16)
    part.bind(params)
    x = gpu(torch.randn(T, H, generator=gen), torch.bfloat16)
    monkeypatch.setattr(ops, "moe_wide_tile_rows", lambda *of: 384 if tile_rows == 384 else 0)
    monkeypatch.setattr(ops, "moe_one_tile_rows", lambda *of: 0)
    monkeypatch.setattr(ops, "moe_tile_rows", lambda *of: tile_rows)
    monkeypatch.setattr(ops, "moe_shared_tile_rows", lambda pairs, experts, sizes, gated, tokens, alone, beside=False: alone)
    none = torch.zeros(1, dtype=torch.int32, device=DEV)
    called, got = [], []
    for longer in (None, False, True):
        monkeypatch.setattr("kvcore_amd.parts.moe.LONG_BRANCH_BYTES", 0 if longer else 1e18)
        ctx = StepContext(num_tokens=T, num_reqs=1, token_ids=none, positions=none, token_req=none, q_start=none,
                          seq_lens=none, slots=none, groups=[], states=[], buffers=StepBuffers(torch.device(DEV), token_capacity=T),
                          dtype=torch.bfloat16, device=torch.device(DEV))
        branch = {} if longer is None else dict(fork=lambda: called.append("fork"), beside=lambda: called.append("beside"))
        rows = part.forward_weighted(x, ctx, None, **branch)
        assert rows.data.shape[0] == T * (top + 1) and rows.add.shape == (T, H) and rows.add.data_ptr() == rows.data[T * top:].data_ptr()
        out = torch.empty(T, H, device=DEV)
        ops.moe_combine(out, rows.data, rows.weight, None, rows.add, add1_gate=rows.add_gate, count=rows.count)
        got.append((out, rows.weight.clone(), ctx.buffers.get(f"moe_choice:{top}", T, top, torch.int32)))
    assert called == ["fork", "beside"] * 2
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][0], got[2][0])

    w = {k: v.double().cpu() for k, v in params.items()}
    xs = x.double().cpu()

    def expert(rows, first, down, limit):
        h = rows @ first.T
        if gated:
            g, u = h[:, :I].clamp(max=limit), h[:, I:].clamp(-limit, limit)
            h = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        else:
            h = h.clamp(min=0) ** 2
        return h @ down.T

    want = expert(xs, w[f"shared.{part.first}"], w["shared.down"], 0.8)
    weight, choice = got[0][1].double().cpu(), got[0][2].cpu()
    per = w[f"experts.{part.first}"].shape[0] // E
    for e in range(E):
        rows = expert(xs, w[f"experts.{part.first}"][e * per:(e + 1) * per], w["experts.down"][e * H:(e + 1) * H], 1.2)
        want += rows * (weight * (choice == e)).sum(1, keepdim=True)
    assert rel(got[0][0], want) < 3e-3  # one rounding of the activations to bfloat16, float32 sums


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("E,top,groups,keep,H,T,score,gated", [
    (32, 4, 8, 4, 2048, 8, "softmax", False), (64, 8, 1, 1, 520, 64, "logit", True), (33, 5, 3, 2, 100, 17, "sigmoid", True),
    (2, 2, 2, 1, 8, 1, "sigmoid", False), (40, 3, 10, 9, 2040, 256, "softmax", True), (1, 1, 1, 1, 32, 16, "logit", False), (16, 2, 4, 2, 64, 1000, "softmax", False),
    (3, 2, 1, 1, 64, 1000, "softmax", False)])
@pytest.mark.parametrize("tile_rows", [16, 384])
def test_spread_router_and_tiles_are_those_of_the_two_kernels(dtype, E, top, groups, keep, H, T, score, gated, tile_rows):
    """The same bits for choices, weights and gates, and the same tiles; a tile's pairs may stand in any order."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(E + T)
    x = gpu(torch.randn(T, H, generator=gen), dtype)
    x[T // 2] = 0  # every expert alike: the lowest indices
    w = gpu(torch.randn(E + gated, H, generator=gen) * H ** -0.5)
    bias = gpu(torch.randn(E, generator=gen) * 0.1) if score != "softmax" else None
    correction = gpu(torch.randn(E, generator=gen)) if score == "sigmoid" else None
    rule = dict(top=top, groups=groups, keep=keep, score=score, bias=bias, correction=correction, weight_scale=1.5,
                group_best=2 if score == "sigmoid" else 1, renormalize=score != "sigmoid")
    i32 = dict(dtype=torch.int32, device=DEV)
    results = []
    for few in (False, True):
        choice, weight = torch.full((T, top), -1, **i32), torch.full((T, top), float("nan"), device=DEV)
        gate = torch.full((T,), float("nan"), device=DEV) if gated else None
        sorted_pairs, num = torch.full((T * top,), -1, **i32), torch.empty(1, **i32)
        tiles = torch.full((ops.moe_max_tiles(T * top, E, tile_rows), 3), -1, **i32)
        if few:
            work = torch.full((ops.moe_router_spread_floats(T, E),), float("nan"), device=DEV)
            ops.moe_router_spread(choice, weight, sorted_pairs, tiles, num, x, w, work, tile_rows=tile_rows, gate=gate, **rule)
        else:
            ops.moe_router(choice, weight, x, w, gate=gate, **rule)
            ops.moe_align(sorted_pairs, tiles, num, choice, E, tile_rows)
        listed = tiles[: int(num)].tolist()
        pairs = sorted_pairs.tolist()
        starts = {e: min(a for f, a, _ in listed if f == e) for e, _, _ in listed}
        held = {e: sorted(pairs[starts[e]: starts[e] + sum(n for f, _, n in listed if f == e)]) for e in starts}
        results.append((choice, weight, gate, listed, held))
    (c0, w0, g0, l0, h0), (c1, w1, g1, l1, h1) = results
    assert torch.equal(c0, c1) and torch.equal(w0, w1) and l0 == l1 and h0 == h1
    assert g0 is None or torch.equal(g0, g1)
    assert sum(len(v) for v in h1.values()) == T * top


@pytest.mark.parametrize("tile_rows", [16, 64, 128])
@pytest.mark.parametrize("packed", [False, True], ids=["rows", "packed"])
@pytest.mark.parametrize("gated,N,K,out_dtype", [(True, 1024, 64, torch.bfloat16), (True, 176, 192, torch.bfloat16),
                                                 (False, 2048, 128, torch.float32), (False, 48, 64, torch.float32),
                                                 (True, 40, 96, torch.float32), (False, 300, 160, torch.bfloat16)])
def test_products_of_experts_over_tiles_of_many_rows(tile_rows, packed, gated, N, K, out_dtype):
    """Experts with no row, one, a few, exactly a tile's, one more and several tiles' worth; columns that end
    inside a block; sums that end inside a pass (a packed matrix has none of the two)."""
    from kvcore_amd.ops import library as ops

    if packed and (N % 16 or K % 64):
        pytest.skip("a packed matrix has experts of a multiple of 16 rows of a multiple of 64")
    gen = torch.Generator().manual_seed(N + K)
    counts = [0, 1, 16, 17, tile_rows - 1, tile_rows, tile_rows + 1, 3, 2 * tile_rows + 5, 0]
    E, T = len(counts), sum(counts)
    choice = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=gen)]
    x = torch.randn(T, K, generator=gen).to(torch.bfloat16)
    w = (torch.randn(E * N * (2 if gated else 1), K, generator=gen) * K ** -0.5).to(torch.bfloat16)
    scale = torch.rand(T, generator=gen) + 0.5
    wg = gpu(w, torch.bfloat16)
    if packed:
        ops.pack_weight(wg)
    i32 = dict(dtype=torch.int32, device=DEV)
    sorted_pairs, num = torch.empty(T, **i32), torch.empty(1, **i32)
    tiles = torch.empty(ops.moe_max_tiles(T, E, tile_rows), 3, **i32)
    ops.moe_align(sorted_pairs, tiles, num, choice.to(**i32).view(T, 1), E, tile_rows)
    listed = tiles[: int(num)].tolist()
    assert all(1 <= n <= tile_rows for _, _, n in listed)
    assert [sum(n for e, _, n in listed if e == which) for which in range(E)] == counts
    out = torch.full((T, N), float("nan"), dtype=out_dtype, device=DEV)
    ops.moe_gemm(out, gpu(x, torch.bfloat16), wg, sorted_pairs, tiles, num, pairs=T, experts=E, in_div=1, out_sorted=False,
                 gated=gated, limit=1.2, alpha=1.702, up_shift=1.0, tile_rows=tile_rows, row_scale=gpu(scale),
                 act=None if gated else "relu_squared")
    want = torch.empty(T, N, dtype=torch.float64)
    per = w.double().view(E, -1, K)
    for e in range(E):
        at = choice == e
        y = (x[at].double() @ per[e].T) * scale[at, None].double()
        if gated:
            g, u = y[:, :N].clamp(max=1.2), y[:, N:].clamp(-1.2, 1.2)
            want[at] = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        else:
            want[at] = y.clamp(min=0) ** 2
    # float32 sums of exact products; a bfloat16 result adds one rounding of 2^-9
    assert rel(out, want) < (2e-6 if out_dtype == torch.float32 else 3e-3)


@pytest.mark.parametrize("packed", [False, True], ids=["rows", "packed"])
@pytest.mark.parametrize("gated,N,K,out_dtype", [(True, 256, 64, torch.bfloat16), (True, 176, 192, torch.float32),
                                                 (False, 512, 128, torch.float32), (False, 304, 320, torch.bfloat16),
                                                 (True, 42, 64, torch.bfloat16), (False, 301, 448, torch.float32)])
def test_products_of_experts_over_tiles_of_384_rows(packed, gated, N, K, out_dtype):
    """Tiles at each number of row blocks a wave takes, and at its edges; two, four and more stages along K, so that the
    last ones find nothing left to fetch; columns that end inside a wave's, and results that four at a time do not
    divide; the same bits as tiles of 128 rows."""
    from kvcore_amd.ops import library as ops

    if packed and N % 16:
        pytest.skip("a packed matrix has experts of a multiple of 16 rows")
    gen = torch.Generator().manual_seed(N + K)
    counts = [0, 1, 31, 32, 33, 65, 100, 129, 160, 192, 223, 225, 256, 257, 288, 289, 320, 321, 352, 353, 384, 385, 800]
    E, T = len(counts), sum(counts)
    choice = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=gen)]
    x = torch.randn(T, K, generator=gen).to(torch.bfloat16)
    w = (torch.randn(E * N * (2 if gated else 1), K, generator=gen) * K ** -0.5).to(torch.bfloat16)
    scale = torch.rand(T, generator=gen) + 0.5
    xg, wg, i32 = gpu(x, torch.bfloat16), gpu(w, torch.bfloat16), dict(dtype=torch.int32, device=DEV)
    if packed:
        ops.pack_weight(wg)
    outs = []
    for tile_rows in (384, 128):
        sorted_pairs, num = torch.empty(T, **i32), torch.empty(1, **i32)
        tiles = torch.empty(ops.moe_max_tiles(T, E, tile_rows), 3, **i32)
        ops.moe_align(sorted_pairs, tiles, num, choice.to(**i32).view(T, 1), E, tile_rows)
        listed = tiles[: int(num)].tolist()
        assert all(1 <= n <= tile_rows for _, _, n in listed)
        assert [sum(n for e, _, n in listed if e == which) for which in range(E)] == counts
        out = torch.full((T, N + 3), float("nan"), dtype=out_dtype, device=DEV)
        ops.moe_gemm(out[:, :N], xg, wg, sorted_pairs, tiles, num, pairs=T, experts=E, in_div=1, out_sorted=False,
                     gated=gated, limit=1.2, alpha=1.702, up_shift=1.0, tile_rows=tile_rows, row_scale=gpu(scale),
                     act=None if gated else "relu_squared")
        assert out[:, N:].isnan().all()
        outs.append(out[:, :N])
    assert torch.equal(*outs)
    want = torch.empty(T, N, dtype=torch.float64)
    per = w.double().view(E, -1, K)
    for e in range(E):
        at = choice == e
        y = (x[at].double() @ per[e].T) * scale[at, None].double()
        if gated:
            g, u = y[:, :N].clamp(max=1.2), y[:, N:].clamp(-1.2, 1.2)
            want[at] = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        else:
            want[at] = y.clamp(min=0) ** 2
    # float32 sums of exact products; a bfloat16 result adds one rounding of 2^-9
    assert rel(outs[0], want) < (2e-6 if out_dtype == torch.float32 else 3e-3)


@pytest.mark.parametrize("gated,N", [(True, 176), (False, 272), (True, 4224)])
@pytest.mark.parametrize("counts", [[300] * 7, [300] * 8, [40, 385] * 4 + [0, 200], [500] * 5, [33] * 67, [20] * 60 + [385] * 8,
                                    [390, 10] * 33], ids=lambda c: f"{len(c)}x{c[0]}")
def test_tiles_of_384_rows_dealt_to_the_dies_by_tile_and_by_column(counts, gated, N):
    """Fewer tiles than dies, as many, more than a wave looks at at once; one tile an expert, a few of two, all of two;
    one column block, two, and more than a die takes in a round: the same bits as tiles of 128 rows."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(N + len(counts))
    E, T, K = len(counts), sum(counts), 64
    i32 = dict(dtype=torch.int32, device=DEV)
    choice = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=gen)].to(**i32)
    xg = gpu(torch.randn(T, K, generator=gen), torch.bfloat16)
    wg = gpu(torch.randn(E * N * (2 if gated else 1), K, generator=gen), torch.bfloat16)
    ops.pack_weight(wg)
    outs = []
    for tile_rows in (384, 128):
        sorted_pairs, num = torch.empty(T, **i32), torch.empty(1, **i32)
        tiles = torch.empty(ops.moe_max_tiles(T, E, tile_rows), 3, **i32)
        ops.moe_align(sorted_pairs, tiles, num, choice.view(T, 1), E, tile_rows)
        out = torch.full((T, N), float("nan"), dtype=torch.float32, device=DEV)
        ops.moe_gemm(out, xg, wg, sorted_pairs, tiles, num, pairs=T, experts=E, in_div=1, out_sorted=False, gated=gated,
                     tile_rows=tile_rows)
        outs.append(out)
    assert torch.equal(*outs) and outs[0].isfinite().all()


@pytest.mark.parametrize("tile_rows", [64, 128])
@pytest.mark.parametrize("gated,N,K", [(True, 176, 448), (False, 304, 512), (True, 2064, 576)])
def test_tiles_of_experts_with_and_without_streaming_loads(tile_rows, gated, N, K):
    """Sums shorter, as long and longer than those from which the experts' tiles are read by streaming loads; experts with
    one tile in the mean (some of none, of two and of three among them) and with more, whose kernel has no such loads; from a
    packed matrix and from rows, which give the same bits."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(N + K)
    counts = [0, 1, tile_rows // 3, tile_rows, tile_rows + 1, 3, 2 * tile_rows + 5, tile_rows // 4]
    i32 = dict(dtype=torch.int32, device=DEV)
    for counts in (counts, [n + tile_rows for n in counts]):
        E, T = len(counts), sum(counts)
        choice = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=gen)]
        x = torch.randn(T, K, generator=gen).to(torch.bfloat16)
        w = (torch.randn(E * N * (2 if gated else 1), K, generator=gen) * K ** -0.5).to(torch.bfloat16)
        sorted_pairs, num = torch.empty(T, **i32), torch.empty(1, **i32)
        tiles = torch.empty(ops.moe_max_tiles(T, E, tile_rows), 3, **i32)
        ops.moe_align(sorted_pairs, tiles, num, choice.to(**i32).view(T, 1), E, tile_rows)
        outs = []
        for packed in (False, True):
            wg = gpu(w, torch.bfloat16)
            if packed:
                ops.pack_weight(wg)
            outs.append(torch.full((T, N), float("nan"), device=DEV))
            ops.moe_gemm(outs[-1], gpu(x, torch.bfloat16), wg, sorted_pairs, tiles, num, pairs=T, experts=E, in_div=1,
                         out_sorted=False, gated=gated, limit=1.2, alpha=1.702, tile_rows=tile_rows)
        assert torch.equal(*outs)
        per = w.double().view(E, -1, K)
        want = torch.empty(T, N, dtype=torch.float64)
        for e in range(E):
            y = x[choice == e].double() @ per[e].T
            if gated:
                g, u = y[:, :N].clamp(max=1.2), y[:, N:].clamp(-1.2, 1.2)
                y = g * torch.sigmoid(1.702 * g) * (u + 1.0)
            want[choice == e] = y
        assert rel(outs[0], want) < 2e-6  # float32 sums of exact products


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,top", [(1, 8, 1), (3, 2048, 4), (67, 2056, 3), (2, 4096, 8), (5, 16384, 5), (5, 16392, 2), (4, 2047, 4)])
def test_experts_sums_with_the_next_norm(T, H, top, dtype):
    """Rows of one chunk a block, a few, all that its registers hold, and those that take two kernels: the bits of the
    two kernels, with and without weights, a further row and its gate, and the mixer's rows."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(T + H)
    draw = lambda *shape: gpu(torch.randn(*shape, generator=gen))  # noqa: E731
    y, gain, start = draw(T * top, H), draw(H), draw(T, H)
    for weight, shared, gate, other in ((draw(T, top), draw(T, H), draw(T, 1), draw(T, H)), (None, None, None, None),
                                        (draw(T, top), draw(T, H), None, None), (None, None, None, draw(T, H))):
        want, got = start.clone(), start.clone()
        rows, x = (torch.empty(T, H, dtype=dtype, device=DEV) for _ in range(2))
        ops.moe_combine(want, y, weight, other, shared, accumulate=True, add1_gate=gate, count=top)
        ops.add_rmsnorm(rows, want, None, gain, 1e-5)
        ops.moe_combine_norm(x, got, ops.WeightedRows(y, weight, shared, gate, count=top), gain, 1e-5, add=other)
        assert torch.equal(got, want) and torch.equal(x, rows)


@pytest.mark.parametrize("E", [1, 31, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("counts_of", ["equal", "edges", "drawn"])
def test_tiles_of_384_rows_hold_every_pair_once(E, counts_of):
    """The list of tiles for up to 32, up to 64 and more experts, with equal counts, without rows and with up to three tiles
    an expert: as many tiles as the rows ask for, each pair in one of them, no row beyond an expert's own, and up to 64
    experts those with more rows a tile first."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(E)
    edges = [0, 1, 383, 384, 385, 768, 769, 1000, 384, 0, 1, 16, 17]
    counts = {"equal": [200] * E, "edges": [edges[i % len(edges)] for i in range(E)],
              "drawn": torch.randint(0, 500, (E,), generator=gen).tolist()}[counts_of]
    if not sum(counts):
        counts[0] = 5
    pairs = sum(counts)
    choice = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(pairs, generator=gen)]
    i32 = dict(dtype=torch.int32, device=DEV)
    sorted_pairs, num = torch.full((pairs,), -1, **i32), torch.empty(1, **i32)
    tiles = torch.full((ops.moe_max_tiles(pairs, E, 384), 3), -1, **i32)
    ops.moe_align(sorted_pairs, tiles, num, choice.to(**i32).view(pairs, 1), E, 384)
    assert int(num) == sum(-(-n // 384) for n in counts)
    assert (tiles[int(num):] == -1).all()
    listed, order = tiles[: int(num)].tolist(), sorted_pairs.tolist()
    rows = [r for _, first, n in listed for r in range(first, first + n)]
    assert sorted(rows) == list(range(pairs)) and sorted(order) == list(range(pairs))
    for e, first, n in listed:
        assert 1 <= n <= 384 and all(choice[order[r]] == e for r in range(first, first + n))
    if E <= 64:
        most = {e: max(n for f, _, n in listed if f == e) for e, _, _ in listed}
        assert [e for e, _, _ in listed] == sorted((e for e, _, _ in listed), key=lambda e: (-most[e], e))


@pytest.mark.parametrize("packed", [False, True], ids=["rows", "packed"])
@pytest.mark.parametrize("gated", [True, False], ids=["gated", "plain"])
@pytest.mark.parametrize("tile_rows,E,T", [(16, 5, 1), (16, 70, 33), (64, 5, 65), (64, 64, 128), (128, 3, 129), (384, 5, 385), (384, 70, 30)])
def test_an_expert_of_every_token_in_the_others_launches(tile_rows, E, T, gated, packed):
    """Both products with the shared expert as one more expert: its rows (one tile, a tile and one row, whole tiles) against
    64-bit sums with its own limit, and the routed experts' rows, which have the bits that they have without it."""
    from kvcore_amd.ops import library as ops

    H, I, top = 192, 128, 2
    gen = torch.Generator().manual_seed(T)
    choice = torch.randint(0, E, (T, top), generator=gen)
    x = torch.randn(T, H, generator=gen).to(torch.bfloat16)
    branches = 2 if gated else 1
    weights = [(torch.randn(*shape, generator=gen) * shape[1] ** -0.5).to(torch.bfloat16)
               for shape in ((E * branches * I, H), (E * H, I), (branches * I, H), (H, I))]
    on = [gpu(w, torch.bfloat16) for w in weights]
    if packed:
        for w in on:
            ops.pack_weight(w)
    i32 = dict(dtype=torch.int32, device=DEV)
    pairs = T * top

    def products(also):
        sorted_pairs, num = torch.full((pairs + also,), -1, **i32), torch.empty(1, **i32)
        tiles = torch.full((ops.moe_max_tiles(pairs, E, tile_rows, also), 3), -7, **i32)
        ops.moe_align(sorted_pairs, tiles, num, choice.to(**i32), E, tile_rows, also)
        listed = tiles[: int(num)].tolist()
        assert sorted(r for _, f, n in listed for r in range(f, f + n)) == list(range(pairs + also))
        assert sum(n for e, _, n in listed if e < 0) == also
        act = torch.full((pairs + also, I), float("nan"), dtype=torch.bfloat16, device=DEV)
        y = torch.full((pairs + also, H), float("nan"), device=DEV)
        ops.moe_gemm(act, gpu(x, torch.bfloat16), on[0], sorted_pairs, tiles, num, pairs=pairs, experts=E, in_div=top,
                     out_sorted=True, gated=gated, limit=1.2, alpha=1.702, tile_rows=tile_rows,
                     act=None if gated else "relu_squared", shared=on[2] if also else None, shared_rows=also, shared_limit=0.7)
        ops.moe_gemm(y, act, on[1], sorted_pairs, tiles, num, pairs=pairs, experts=E, in_div=0, out_sorted=False, gated=False,
                     tile_rows=tile_rows, shared=on[3] if also else None, shared_rows=also)
        return y

    y, alone = products(T), products(0)
    assert torch.equal(y[:pairs], alone)
    h = x.double() @ weights[2].double().T
    if gated:
        g, u = h[:, :I].clamp(max=0.7), h[:, I:].clamp(-0.7, 0.7)
        h = g * torch.sigmoid(1.702 * g) * (u + 1.0)
    else:
        h = h.clamp(min=0) ** 2
    # one rounding of the activations to bfloat16, float32 sums
    assert rel(y[pairs:], h @ weights[3].double().T) < 3e-3


@pytest.mark.parametrize("gated", [True, False])
def test_experts_results_of_infinite_and_missing_sums(gated):
    """Sums that are infinite or no number leave tiles of 64, 128 and 384 rows as the activation says, a sum whose
    exponential overflows as zero."""
    from kvcore_amd.ops import library as ops

    T, N, K = 7, 16, 64
    rows = torch.zeros(T, K, dtype=torch.bfloat16)
    rows[:, 0] = torch.tensor([1.0, -1.0, 300.0, -300.0, float("inf"), float("-inf"), float("nan")])
    w = torch.zeros(N * (2 if gated else 1), K, dtype=torch.bfloat16)
    w[:, 0] = 1.0
    i32 = dict(dtype=torch.int32, device=DEV)
    zero = torch.zeros(T, 1, **i32)
    for tile_rows in (64, 128, 384):
        sorted_pairs, num = torch.empty(T, **i32), torch.empty(1, **i32)
        tiles = torch.empty(ops.moe_max_tiles(T, 1, tile_rows), 3, **i32)
        ops.moe_align(sorted_pairs, tiles, num, zero, 1, tile_rows)
        out = torch.empty(T, N, device=DEV)
        ops.moe_gemm(out, gpu(rows, torch.bfloat16), gpu(w, torch.bfloat16), sorted_pairs, tiles, num, pairs=T, experts=1,
                     in_div=1, out_sorted=False, gated=gated, limit=float("inf"), alpha=1.0, up_shift=0.0,
                     tile_rows=tile_rows, act=None if gated else "relu_squared")
        v = rows[:, 0].float()
        limit = torch.tensor(float("inf"))  # the clamps take the limit for what is no number
        g, u = torch.fmin(v, limit), torch.fmin(torch.fmax(v, -limit), limit)
        want = g / (1.0 + torch.exp(-g)) * u if gated else torch.fmax(v, torch.zeros(())) ** 2
        assert torch.allclose(out[:, 0].cpu(), want, rtol=1e-6, atol=1e-30, equal_nan=True)


@pytest.mark.parametrize("packed", [False, True], ids=["rows", "packed"])
@pytest.mark.parametrize("gated,N,K,whole", [
    (True, 64, 2048, False),    # 32 passes of 64: eight a wave, more than are on their way at once
    (False, 48, 1088, False),   # 17 passes
    (True, 32, 1000, False),    # a ragged end along K
    (False, 2048, 576, False),  # many waves, K too long for a whole one
    (True, 496, 512, False), (False, 160, 256, False),  # 744 and 240 waves: just too few
    (True, 512, 512, True), (False, 176, 256, True), (False, 1000, 456, True), (False, 1040, 64, True), (True, 999, 8, True)])
def test_few_rows_take_shares_of_k_or_all_of_it(gated, N, K, whole, packed):
    """Both sides of the line between the two, with 24 tiles of up to 16 rows (the line: K of at most 512, from a wave of
    16 columns a unit on up to K of 256, from three beyond)."""
    from kvcore_amd.ops import library as ops

    if packed and (N % 16 or K % 64):
        pytest.skip("a packed matrix has experts of a multiple of 16 rows of a multiple of 64")
    gen = torch.Generator().manual_seed(N + K)
    E, T = 8, 16 * 16
    choice = torch.randint(1, E, (T,), generator=gen)
    choice[:17] = 3
    x = torch.randn(T, K, generator=gen).to(torch.bfloat16)
    w = (torch.randn(E * N * (2 if gated else 1), K, generator=gen) * K ** -0.5).to(torch.bfloat16)
    wg = gpu(w, torch.bfloat16)
    if packed:
        ops.pack_weight(wg)
    i32 = dict(dtype=torch.int32, device=DEV)
    sorted_pairs, num = torch.empty(T, **i32), torch.empty(1, **i32)
    tiles = torch.empty(ops.moe_max_tiles(T, E, 16), 3, **i32)
    assert tiles.shape[0] == 24
    ops.moe_align(sorted_pairs, tiles, num, choice.to(**i32).view(T, 1), E, 16)
    out = torch.full((T, N), float("nan"), device=DEV)
    ops.moe_gemm(out, gpu(x, torch.bfloat16), wg, sorted_pairs, tiles, num, pairs=T, experts=E, in_div=1, out_sorted=False,
                 gated=gated, limit=1.2, alpha=1.702, up_shift=1.0, tile_rows=16)
    assert ops.last_variant("moe_gemm") == "moe_gemm_few_kernel, " + ("whole K" if whole else "shares of K")
    per, want = w.double().view(E, -1, K), torch.empty(T, N, dtype=torch.float64)
    for e in range(E):
        at = choice == e
        y = x[at].double() @ per[e].T
        if gated:
            g, u = y[:, :N].clamp(max=1.2), y[:, N:].clamp(-1.2, 1.2)
            y = g * torch.sigmoid(1.702 * g) * (u + 1.0)
        want[at] = y
    assert rel(out, want) < 2e-6  # float32 sums of exact products


def test_more_tiles_of_few_rows_than_a_grid_dimension_holds():
    """K that tiles of 64 rows do not take, and 65,536 tiles of 16."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(1)
    E, T, N, K = 3, 65536 * 16 - 40, 16, 8
    choice = torch.randint(0, E, (T, 1), generator=gen).to(device=DEV, dtype=torch.int32)
    x, w = (gpu(torch.randn(n, K, generator=gen), torch.bfloat16) for n in (T, E * N))
    i32 = dict(dtype=torch.int32, device=DEV)
    sorted_pairs, num, tiles = torch.empty(T, **i32), torch.empty(1, **i32), torch.empty(ops.moe_max_tiles(T, E, 16), 3, **i32)
    assert tiles.shape[0] > 65535
    ops.moe_align(sorted_pairs, tiles, num, choice, E, 16)
    out = torch.full((T, N), float("nan"), device=DEV)
    ops.moe_gemm(out, x, w, sorted_pairs, tiles, num, pairs=T, experts=E, in_div=1, out_sorted=False, gated=False, tile_rows=16)
    every = (x.float() @ w.float().T).view(T, E, N)  # eight exact products a sum
    want = every.gather(1, choice.long()[:, :, None].expand(-1, -1, N))[:, 0]
    assert torch.allclose(out, want, atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("E", [65, 1500, 5000])
def test_tiles_of_very_many_experts(E):
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(E)
    T, top = 3000, 3
    choice = torch.randint(0, E, (T, top), generator=gen)
    choice[:200] = E - 1
    i32 = dict(dtype=torch.int32, device=DEV)
    sorted_pairs, num = torch.full((T * top,), -1, **i32), torch.empty(1, **i32)
    tiles = torch.full((ops.moe_max_tiles(T * top, E, 64), 3), -1, **i32)
    ops.moe_align(sorted_pairs, tiles, num, choice.to(**i32), E, 64)
    of_pair, at = choice.flatten(), 0
    order = sorted_pairs.cpu().long()
    assert torch.equal(order.sort().values, torch.arange(T * top))
    assert torch.equal(of_pair[order], of_pair.sort().values)
    for e, first, n in tiles[: int(num)].tolist():
        assert first == at and 1 <= n <= 64 and (of_pair[order[first: first + n]] == e).all()
        at += n
    assert at == T * top
    too_many = torch.zeros(1, 1, **i32)
    with pytest.raises(ops.KernelError, match="too many experts"):
        ops.moe_align(sorted_pairs, torch.empty(ops.moe_max_tiles(1, 5001, 16), 3, **i32), num, too_many, 5001, 16)


def test_offset_norm_keeps_a_gain_of_one_plus_the_stored_weight():
    from kvcore_amd.parts.base import Runtime
    from kvcore_amd.parts.rmsnorm import RMSNorm

    gen = torch.Generator().manual_seed(2)
    H, T = 96, 9
    w = torch.randn(H, generator=gen, dtype=torch.float64) * 0.2
    r = torch.randn(T, H, generator=gen, dtype=torch.float64) * 3
    norm = RMSNorm(hidden_size=H, eps=1e-5, weight_offset=1.0, weight_name="")
    assert [s.name for s in norm.param_specs()[0].resolved_sources()] == [""]
    norm.setup(Runtime(dtype=torch.float32, device=torch.device(DEV)))
    norm.bind({"weight": gpu(w)})
    norm.weights_loaded()
    out = torch.empty(T, H, device=DEV)
    norm.forward_fused(out, gpu(r), None)
    assert rel(out, plain.offset_rms_norm(r, w, 1e-5)) < 1e-6
    assert math.isclose(float(norm.as_gain()[0][0]), 1.0 + float(w[0].float()), rel_tol=1e-6)
