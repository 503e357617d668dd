"""The matrix-state recurrences over portions of prompts in chunks, against the recurrence token by token in float64
and against the scan kernels, at the edges of chunks (64 tokens) and of the runs inside them (16)."""

from __future__ import annotations

import pytest
import torch

from tests.vovalix_helpers import batch_tensors

pytestmark = pytest.mark.gpu

DEV = "cuda"


def gpu(t, dtype=torch.float32):
    return t.to(device=DEV, dtype=dtype).contiguous()


def rel(got, want):
    return float((got.double().cpu() - want).pow(2).mean().sqrt() / (want.pow(2).mean().sqrt() + 1e-30))


def in_chunks(reqs, start, heads, key_heads, rows, cols):
    """The arguments that say which requests are cut into chunks, and their workspace (nothing in it to be read)."""
    from kvcore_amd.ops import library as ops

    chunks = ops.gated_chunk_count([1 if r is None else r[2] for r in reqs], start)
    work = torch.full((chunks, ops.load().kvc_gated_chunk_floats(heads, key_heads, rows, cols)), float("nan"), device=DEV)
    return work, dict(chunks=chunks, start=start)


def walk(q, k, v, g, b, S):
    """``q, k [T, heads, d]``, ``v [T, heads, dv]``, ``g, b [T, heads]``, ``S [heads, d, dv]``: results and last state."""
    out = []
    for t in range(q.shape[0]):
        S = g[t][:, None, None] * S + b[t][:, None, None] * k[t][:, :, None] * v[t][:, None, :]
        out.append(torch.einsum("hdv,hd->hv", S, q[t]))
    return torch.stack(out), S


# requests side by side: lengths at and around the chunk's and the run's edges, a padded one between them
LENGTHS = [1, 64, 65, 15, 16, 17, 200, 63, 130]


def requests(lengths, start):
    reqs = [(i, start, n) for i, n in enumerate(lengths)]
    return reqs[:4] + [None] + reqs[4:]


def spans(reqs):
    at, out = 0, []
    for r in reqs:
        n = 1 if r is None else r[2]
        if r is not None:
            out.append((r[0], at, at + n))
        at += n
    return out, at


def memory_inputs(heads, qk_heads, d, dv, ones, T, gen):
    q, k = (torch.randn(T, qk_heads, d, generator=gen) for _ in range(2))
    v = torch.randn(T, heads, dv - ones, generator=gen)
    g = torch.rand(T, heads, generator=gen) ** 0.2
    g[torch.rand(T, heads, generator=gen) < 0.03] = 0.0   # a state that is forgotten at once
    g[:, 0] = 0.999
    return q, k * d ** -0.5, v, g, torch.rand(T, heads, generator=gen) * 2


def both(q, k, v, g, b, state, reqs, *, heads, qk_heads, d, dv, ones, start=1):
    """(results, states) of the scan and of the chunks, from copies of ``state``."""
    from kvcore_amd.ops import library as ops

    batch, T = batch_tensors(reqs)
    # column views of wider rows, as the mixers hand them in
    wide = torch.cat([q.flatten(1), k.flatten(1), v.flatten(1), g, b], 1)
    wide = gpu(torch.cat([wide, torch.zeros(T, -wide.shape[1] % 4)], 1))
    a, c = qk_heads * d, heads * (dv - ones)
    rows = (wide[:, :a], wide[:, a:2 * a], wide[:, 2 * a:2 * a + c], wide[:, 2 * a + c:2 * a + c + heads],
            wide[:, 2 * a + c + heads:2 * a + c + 2 * heads])
    sizes = dict(heads=heads, qk_heads=qk_heads, dim=d, vdim=dv, q_scale=0.5, ones_column=bool(ones))
    out = []
    for chunked in (False, True):
        y, s = torch.full((T, heads * dv), float("nan"), device=DEV), state.clone()
        if chunked:
            work, cut = in_chunks(reqs, start, heads, qk_heads, d, dv)
            ops.scalar_gate_chunks(y, *rows, s, work, **cut, **sizes, **batch)
            if start > 1:  # the shorter requests the other way
                ops.linear_state_scan(y, *rows, s, scalar_gates=True, below=start, **sizes, **batch)
        else:
            ops.linear_state_scan(y, *rows, s, scalar_gates=True, **sizes, **batch)
        out.append((y, s))
    return out


@pytest.mark.parametrize("start,from_", [(0, 1), (7, 1), (7, 64)])
@pytest.mark.parametrize("heads,qk_heads,d,dv,ones", [(2, 2, 64, 129, 1), (3, 1, 24, 40, 0), (2, 2, 100, 80, 0),
                                                        (1, 1, 8, 5, 1), (2, 1, 128, 64, 0), (2, 2, 30, 145, 1)])
def test_scalar_gates_in_chunks(heads, qk_heads, d, dv, ones, start, from_):
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(d + dv)
    reqs = requests(LENGTHS, start)
    where, T = spans(reqs)
    q, k, v, g, b = memory_inputs(heads, qk_heads, d, dv, ones, T, gen)
    # what the slots hold: another request's leftovers where a request starts, its own state otherwise
    rows = ops.linear_state_rows(d)
    held = torch.randn(len(LENGTHS), heads, rows, dv, generator=gen)
    state = torch.full_like(held, float("nan")) if start == 0 else held
    results = both(q, k, v, g, b, gpu(state), reqs, heads=heads, qk_heads=qk_heads, d=d, dv=dv, ones=ones,
                   start=from_)
    rep = heads // qk_heads
    errors = []
    for y, s in results:
        got, want, gs, ws = [], [], [], []
        for slot, lo, hi in where:
            value = v[lo:hi].double()
            if ones:
                value = torch.cat([value, torch.ones(hi - lo, heads, 1, dtype=torch.float64)], -1)
            # a head's rows lie in fours: [rows / 4, dv, 4]
            plain = held[slot].view(heads, rows // 4, dv, 4).permute(0, 1, 3, 2).reshape(heads, rows, dv)[:, :d]
            first = plain.double() if start else torch.zeros(heads, d, dv, dtype=torch.float64)
            o, last = walk(q[lo:hi].double().repeat_interleave(rep, 1) * 0.5, k[lo:hi].double().repeat_interleave(rep, 1),
                           value, g[lo:hi].double(), b[lo:hi].double(), first)
            got.append(y[lo:hi].view(hi - lo, heads, dv).cpu())
            want.append(o)
            gs.append(s[slot].view(heads, rows // 4, dv, 4).permute(0, 1, 3, 2).reshape(heads, rows, dv)[:, :d].cpu())
            ws.append(last)
        errors.append((rel(torch.cat(got), torch.cat(want)), rel(torch.stack(gs), torch.stack(ws))))
    pad = sum(LENGTHS[:4])
    assert float(results[1][0][pad].abs().sum()) == 0.0  # the padded request's row
    (scan_y, scan_s), (chunk_y, chunk_s) = errors
    assert chunk_y < 1e-6 and chunk_s < 1e-6, errors
    # the chunks round no more than the scan does (both some 1e-7: a quarter more is their scatter)
    assert chunk_y < 1.25 * scan_y + 2e-8 and chunk_s < 1.25 * scan_s + 2e-8, errors


@pytest.mark.parametrize("heads,P,N,groups", [(16, 64, 128, 2), (16, 64, 64, 1), (8, 100, 30, 2)])
def test_state_space_chunks_round_no_more_than_the_scan(heads, P, N, groups):
    """Decays and steps as such layers have them; the mean of four draws, whose ratios scatter by some 3%."""
    from kvcore_amd.ops import library as ops

    T, inner, errors = 256, heads * P, []
    for seed in range(4):
        gen = torch.Generator().manual_seed(seed)
        z = torch.randn(T, inner + 2 * groups * N, generator=gen)
        xbc, dt = gpu(z * torch.sigmoid(z)), gpu(torch.randn(T, heads, generator=gen))
        bias = gpu(torch.log(torch.expm1(0.001 * torch.exp(4.6 * torch.rand(heads, generator=gen)))))
        a_log, skip = gpu(torch.log(1 + 15 * torch.rand(heads, generator=gen))), gpu(torch.ones(heads))
        step = torch.nn.functional.softplus(dt.double() + bias.double(), threshold=100).cpu()
        x = xbc[:, :inner].double().cpu().view(T, heads, P)
        B, C = (xbc[:, inner + i * groups * N: inner + (i + 1) * groups * N].double().cpu().view(T, groups, N)
                .repeat_interleave(heads // groups, 1) for i in (0, 1))
        want, _ = walk(C, B, x, torch.exp(-torch.exp(a_log.double().cpu()) * step), step,
                       torch.zeros(heads, N, P, dtype=torch.float64))
        want = (want + x).reshape(T, inner)
        batch, _ = batch_tensors([(0, 0, T)])
        sizes = dict(heads=heads, head_dim=P, state_size=N, groups=groups)
        both_ways = []
        for chunked in (False, True):
            y, s = torch.empty(T, inner, device=DEV), torch.zeros(1, heads, N, P, device=DEV)
            if chunked:
                work, cut = in_chunks([(0, 0, T)], 1, heads, groups, N, P)
                ops.ssm_chunks(y, xbc, dt, bias, a_log, skip, s, work, **cut, **sizes, **batch)
            else:
                ops.ssm_scan(y, xbc, dt, bias, a_log, skip, s, **sizes, **batch)
            both_ways.append(rel(y, want))
        errors.append(both_ways)
    scan, chunks = torch.tensor(errors).mean(0).tolist()
    assert chunks < 1.08 * scan, errors


def test_what_is_not_finite_reaches_no_earlier_token_and_no_other_request():
    gen = torch.Generator().manual_seed(4)
    heads, d, dv = 2, 16, 20
    reqs = requests([40, 70, 30, 64, 90], 0)
    where, T = spans(reqs)
    q, k, v, g, b = memory_inputs(heads, heads, d, dv, 0, T, gen)
    state = torch.zeros(5, heads, d, dv, device=DEV)
    kw = dict(heads=heads, qk_heads=heads, d=d, dv=dv, ones=0)
    clean = both(q, k, v, g, b, state, reqs, **kw)[1][0]
    (slot, lo, hi) = where[1]
    at = lo + 37
    for which, value in (("v", float("inf")), ("v", float("nan")), ("k", float("nan")), ("q", float("inf")), ("b", float("nan"))):
        parts = dict(q=q.clone(), k=k.clone(), v=v.clone(), g=g.clone(), b=b.clone())
        parts[which][at] = value
        dirty = both(*parts.values(), state, reqs, **kw)[1][0]
        keep = torch.ones(T, dtype=torch.bool)
        keep[at:hi] = False
        keep = keep.to(DEV)
        assert rel(dirty[keep], clean[keep].double().cpu()) < 1e-6, which
        assert not torch.isfinite(dirty[at]).all(), which


@pytest.mark.parametrize("start,from_", [(0, 1), (5, 1), (5, 65)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("heads,groups,N,P", [(4, 2, 128, 64), (2, 1, 30, 20), (3, 3, 16, 100), (2, 2, 100, 16), (2, 1, 5, 3)])
def test_state_space_recurrence_in_chunks(heads, groups, N, P, dtype, start, from_):
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(N + P)
    reqs = requests(LENGTHS, start)
    where, T = spans(reqs)
    batch, _ = batch_tensors(reqs)
    inner = heads * P
    xbc = torch.randn(T, inner + 2 * groups * N, generator=gen)
    xbc[:, inner:] *= N ** -0.5
    dt = torch.randn(T, heads + 3, generator=gen).to(dtype)
    dt_bias, skip = torch.randn(heads, generator=gen) - 3, torch.randn(heads, generator=gen)
    a_log = torch.linspace(0.0, 2.7, heads)
    held = torch.randn(len(LENGTHS), heads, N, P, generator=gen)
    state = torch.full_like(held, float("nan")) if start == 0 else held
    dts = gpu(dt, dtype)[:, 3:]
    common = (gpu(xbc), dts, gpu(dt_bias), gpu(a_log), gpu(skip))
    sizes = dict(heads=heads, head_dim=P, state_size=N, groups=groups)
    errors = []
    for chunked in (False, True):
        y, s = torch.full((T, inner), float("nan"), device=DEV), gpu(state)
        if chunked:
            work, cut = in_chunks(reqs, from_, heads, groups, N, P)
            ops.ssm_chunks(y, *common, s, work, **cut, **sizes, **batch)
            if from_ > 1:
                ops.ssm_scan(y, *common, s, below=from_, **sizes, **batch)
        else:
            ops.ssm_scan(y, *common, s, **sizes, **batch)
        got, want, ws = [], [], []
        for slot, lo, hi in where:
            x = xbc[lo:hi, :inner].double().view(-1, heads, P)
            B, C = (xbc[lo:hi, inner + i * groups * N: inner + (i + 1) * groups * N].double().view(-1, groups, N)
                    .repeat_interleave(heads // groups, 1) for i in (0, 1))
            step = torch.nn.functional.softplus(dt[lo:hi, 3:].double() + dt_bias.double(), threshold=100)
            first = held[slot].double() if start else torch.zeros(heads, N, P, dtype=torch.float64)
            o, last = walk(C, B, x, torch.exp(-torch.exp(a_log.double()) * step), step, first)
            got.append(y[lo:hi].view(-1, heads, P).cpu())
            want.append(o + skip.double()[:, None] * x)
            ws.append(last)
        errors.append((rel(torch.cat(got), torch.cat(want)), rel(s, torch.stack(ws))))
        assert float(y[sum(LENGTHS[:4])].abs().sum()) == 0.0
    (scan_y, scan_s), (chunk_y, chunk_s) = errors
    assert chunk_y < 1e-6 and chunk_s < 1e-6, errors
    assert chunk_y < 1.25 * scan_y + 2e-8 and chunk_s < 1.25 * scan_s + 2e-8, errors


@pytest.mark.parametrize("start,from_", [(0, 1), (7, 1), (7, 64)])
@pytest.mark.parametrize("heads,qk_heads,d,dv", [(2, 2, 64, 128), (3, 1, 24, 40), (2, 2, 100, 80), (1, 1, 7, 5),
                                                  (2, 1, 128, 130), (2, 2, 30, 64)])
def test_channel_factors_in_chunks(heads, qk_heads, d, dv, start, from_):
    """Factors from zero to one, some channels that forget at once and some that keep for ever."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(d + dv)
    reqs = requests(LENGTHS, start)
    where, T = spans(reqs)
    q, k = (torch.randn(T, qk_heads, d, generator=gen) for _ in range(2))
    k = k * d ** -0.5
    v = torch.randn(T, heads, dv, generator=gen)
    a = torch.rand(T, heads, d, generator=gen) ** (10.0 ** (torch.rand(heads, d, generator=gen) * -3 + 1))
    a[torch.rand(T, heads, d, generator=gen) < 0.02] = 0.0
    a[:, 0, 0] = 1.0
    rows = ops.linear_state_rows(d)
    held = torch.randn(len(LENGTHS), heads, rows, dv, generator=gen)
    state = gpu(torch.full_like(held, float("nan")) if start == 0 else held)
    batch, _ = batch_tensors(reqs)
    wide = torch.cat([q.flatten(1), k.flatten(1), v.flatten(1)], 1)
    wide = gpu(torch.cat([wide, torch.zeros(T, -wide.shape[1] % 4)], 1))
    c = qk_heads * d
    views = (wide[:, :c], wide[:, c:2 * c], wide[:, 2 * c:2 * c + heads * dv])
    sizes = dict(heads=heads, qk_heads=qk_heads, dim=d, vdim=dv, q_scale=0.5, **batch)
    errors = []
    for chunked in (False, True):
        y, s = torch.full((T, heads * dv), float("nan"), device=DEV), state.clone()
        if chunked:
            chunks = ops.gated_chunk_count([1 if r is None else r[2] for r in reqs], from_)
            work = torch.full((chunks, ops.load().kvc_channel_chunk_floats(heads, d, dv)), float("nan"), device=DEV)
            ops.channel_gate_chunks(y, *views, gpu(a.flatten(1)), s, work, chunks=chunks, start=from_, **sizes)
            if from_ > 1:
                ops.linear_state_scan(y, *views, gpu(a.flatten(1)), None, s, below=from_, **sizes)
        else:
            ops.linear_state_scan(y, *views, gpu(a.flatten(1)), None, s, **sizes)
        got, want, gs, ws = [], [], [], []
        rep = heads // qk_heads
        for slot, lo, hi in where:
            S = held[slot].double().view(heads, rows // 4, dv, 4).permute(0, 1, 3, 2).reshape(heads, rows, dv)[:, :d]
            S = S * (start > 0)
            for t in range(lo, hi):
                kt, qt = (x[t].double().repeat_interleave(rep, 0) for x in (k, q))
                S = a[t].double()[:, :, None] * S + kt[:, :, None] * v[t].double()[:, None, :]
                want.append(torch.einsum("hdv,hd->hv", S, qt * 0.5).flatten())
            got.append(y[lo:hi])
            gs.append(s[slot].view(heads, rows // 4, dv, 4).permute(0, 1, 3, 2).reshape(heads, rows, dv)[:, :d])
            ws.append(S)
        errors.append((rel(torch.cat(got), torch.stack(want)), rel(torch.stack(gs), torch.stack(ws))))
        if None in reqs:
            at = sum(r[2] for r in reqs[:4])
            assert (y[at] == 0).all()
    # the same number of products and sums is rounded either way: no worse than the scan but for chance (factors that
    # forget at once leave the last few tokens' roundings, of which the scan has two a token and the chunks three)
    assert errors[1][0] < 1.2 * errors[0][0] and errors[1][1] < 1.5 * errors[0][1], errors


def test_channel_factors_in_chunks_keep_to_their_own_tokens():
    """A value or key that is not finite reaches the tokens from its own on and no earlier one, and its own column or all."""
    from kvcore_amd.ops import library as ops

    gen = torch.Generator().manual_seed(2)
    T, d, dv = 100, 64, 128
    q, k, v = (torch.randn(T, n, generator=gen) for n in (d, d, dv))
    a = torch.rand(T, d, generator=gen)
    v[37, 5], k[70, 3] = float("inf"), float("nan")
    batch, _ = batch_tensors([(0, 0, T)])
    y, s = torch.zeros(T, dv, device=DEV), torch.zeros(1, 1, d, dv, device=DEV)
    work = torch.empty(2, ops.load().kvc_channel_chunk_floats(1, d, dv), device=DEV)
    ops.channel_gate_chunks(y, gpu(q), gpu(k), gpu(v), gpu(a), s, work, chunks=2, heads=1, qk_heads=1, dim=d, vdim=dv,
                            **batch)
    fine = torch.isfinite(y.cpu())
    assert fine[:37].all() and not fine[37:, 5].any() and not fine[70:].any()
    others = torch.arange(dv) != 5
    assert fine[37:70][:, others].all()
