"""A layer's two branches side by side, on the CPU: what a parallel block hands to its parts, and what orders the streams."""

from __future__ import annotations

import contextlib
from types import SimpleNamespace

import pytest
import torch

from kvcore_amd.engine.context import LayerCall, SideStream
from kvcore_amd.parts.base import FeedForward, Mixer, Norm
from kvcore_amd.parts.block import ParallelResidualBlock
from kvcore_amd.parts.moe import RoutedExperts


class CopyNorm(Norm):
    def forward_fused(self, out, residual, delta):
        out.copy_(residual)

    def as_gain(self):
        return torch.ones(4), 1e-5


class DoublingMixer(Mixer):
    float32_result = True

    def __init__(self, log):
        self.log = log

    def forward(self, x, ctx, call, sink=None):
        self.log.append("mixer")
        return 2.0 * x


class Side:
    """In the place of a ``SideStream``: notes what it is asked."""

    def __init__(self, log):
        self.log = log

    def fork(self):
        self.log.append("fork")

    def branch(self, work):
        self.log.append("branch")
        return work()

    def join(self):
        self.log.append("join")


def experts(log, fails=False):
    part = RoutedExperts(hidden_size=4, experts=2, top=1, expert_size=4, limit=None)

    def forward_weighted(x, ctx, call, fork=None, beside=None):
        if beside is not None:
            fork()
            beside()
        log.append("experts")
        if fails:
            raise RuntimeError("no room")
        return "rows"

    part.forward_weighted = forward_weighted
    part.forward_into = lambda residual, x, ctx, call, add=None, rows=None: (log.append(("into", rows)), residual.add_(add))
    return part


def step(ffn, log, side=True, next_block=None):
    block = ParallelResidualBlock(mixer=DoublingMixer(log), ffn=ffn, norms={"n": CopyNorm()})
    ctx = SimpleNamespace(side=Side(log) if side else None, scratch={}, buf=lambda name, cols: torch.zeros(3, cols))
    residual = torch.ones(3, 4)
    block.forward(None, residual, ctx, LayerCall(0, 0), next_block=next_block)
    return residual


def test_the_streams_are_joined_when_the_experts_raise():
    log = []
    with pytest.raises(RuntimeError, match="no room"):
        step(experts(log, fails=True), log)
    assert log == ["fork", "branch", "mixer", "experts", "join"]


class Event:
    def __init__(self, name, log):
        self.name, self.log = name, log

    def record(self, stream=None):
        self.log.append((self.name, "record", stream))

    def wait(self, stream=None):
        self.log.append((self.name, "wait", stream))


def side_stream(monkeypatch, log, beside=True, made=None):
    """A ``SideStream`` over streams and events that only note what is asked of them; the current stream is "main"."""
    made = [] if made is None else made
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: "main")
    monkeypatch.setattr(torch.cuda, "set_stream", lambda stream: log.append(stream))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: "capturing" in made)
    monkeypatch.setattr(SideStream, "_works_beside", lambda self: beside)
    monkeypatch.setattr(torch.cuda, "Stream", lambda device=None: made.append("side") or "side")
    monkeypatch.setattr(torch.cuda, "device", lambda device: contextlib.nullcontext())
    events = iter((Event("forked", log), Event("done", log)))
    monkeypatch.setattr(torch.cuda, "Event", lambda: next(events))
    return SideStream(torch.device("cpu")), made


def test_a_join_waits_for_the_branch_that_was_started_last_and_for_nothing_else(monkeypatch):
    log = []
    side, _ = side_stream(monkeypatch, log)

    def fails():
        raise ValueError("in the branch")

    side.fork()
    side.join()  # an error before the branch: an event that this step has not recorded is not waited for
    assert log == [("forked", "record", "main")]
    log.clear()
    with pytest.raises(ValueError, match="in the branch"):
        side.branch(fails)
    side.join()
    side.join()
    assert log == [("forked", "wait", "side"), "side", ("done", "record", "side"), "main", ("done", "wait", "main")]


def test_where_no_stream_works_beside_the_current_one(monkeypatch):
    """Branches run in line, one after the other, but for captured steps, whose graph has branches of its own."""
    log = []
    side, made = side_stream(monkeypatch, log, beside=False)
    assert not side.apart and len(made) == 8
    side.fork()
    assert side.branch(lambda: log.append("work") or 7) == 7
    side.join()
    assert log == ["work"]
    log.clear()
    made.append("capturing")
    side.begin_capture()
    side.fork()
    side.branch(lambda: log.append("work"))
    side.join()
    assert log == [("forked", "record", "main"), ("forked", "wait", "side"), "side", "work", ("done", "record", "side"), "main",
                   ("done", "wait", "main")]
    side, made = side_stream(monkeypatch, log)
    assert side.apart and len(made) == 1


def test_a_process_captures_so_many_steps_with_branches(monkeypatch):
    log = []
    monkeypatch.setattr(SideStream, "_graphs", 0)
    monkeypatch.setattr(SideStream, "MOST_GRAPHS", 2)
    side, made = side_stream(monkeypatch, log)
    other, _ = side_stream(monkeypatch, log, made=made)
    ways = []
    for s in (side, other, side, other):
        made.append("capturing")
        s.begin_capture()
        log.clear()
        s.fork()
        s.branch(lambda: None)
        s.join()
        ways.append(bool(log))
        made.remove("capturing")
        log.clear()
        s.fork()  # a step that is not captured
        s.branch(lambda: None)
        s.join()
        assert log
    assert ways == [True, True, False, False]


def test_experts_beside_a_mixer_take_the_rows_that_they_have_made():
    log = []
    assert torch.equal(step(experts(log), log), torch.full((3, 4), 3.0))
    assert log == ["fork", "branch", "mixer", "experts", "join", ("into", "rows")]
    log.clear()
    step(experts(log), log, side=False)
    assert log == ["mixer", ("into", None)]


class AddingFeedForward(FeedForward):
    """As the documented signatures have it, and no more."""

    gives_weighted_rows = True

    def __init__(self, log):
        self.log = log

    def forward_weighted(self, x, ctx, call):
        raise AssertionError("not this block's")

    def forward_into(self, residual, x, ctx, call, add=None):
        self.log.append("into")
        residual.add_(add).add_(x)


class NormedFeedForward(AddingFeedForward):
    def forward_into_normed(self, out, residual, x, ctx, call, gain, eps, add=None):
        self.log.append("normed")
        residual.add_(add).add_(x)


class OwnExperts(RoutedExperts):
    """Experts with a ``forward_weighted`` of the three arguments that a block without a second stream passes."""

    def forward_weighted(self, x, ctx, call):
        self.log.append("weighted")
        return "rows"

    def forward_into(self, residual, x, ctx, call, add=None):
        assert self.forward_weighted(x, ctx, call) == "rows"
        residual.add_(add).add_(x)


@pytest.mark.parametrize("side", [False, True], ids=["one stream", "a second stream"])
@pytest.mark.parametrize("kind", ["into", "normed", "experts"])
def test_a_feed_forward_that_knows_nothing_of_branches(kind, side):
    """A registered part with the documented methods is called with their arguments, on one stream."""
    log = []
    following = None
    if kind == "experts":
        ffn = OwnExperts(hidden_size=4, experts=2, top=1, expert_size=4, limit=None)
        ffn.log = log
    else:
        ffn = (NormedFeedForward if kind == "normed" else AddingFeedForward)(log)
        following = ParallelResidualBlock(mixer=DoublingMixer(log), ffn=ffn, norms={"n": CopyNorm()})
        assert not following.has_branches
    assert torch.equal(step(ffn, log, side, following), torch.full((3, 4), 4.0))
    assert log == ["mixer", {"into": "into", "normed": "normed", "experts": "weighted"}[kind]]


def test_a_subclass_of_the_experts_that_says_so_runs_beside():
    class Same(RoutedExperts):
        pass

    class Own(RoutedExperts):
        runs_beside = True

        def forward_weighted(self, x, ctx, call, fork=None, beside=None):
            return super().forward_weighted(x, ctx, call, fork, beside)

    assert RoutedExperts.runs_beside and Same.runs_beside and Own.runs_beside and not OwnExperts.runs_beside


def test_the_requests_whose_scans_leave_units_to_the_other_stream():
    from kvcore_amd.parts.linear_attention import CHAIN_TOKENS, GatedDeltaRule

    lengths = [3500, 1, CHAIN_TOKENS, CHAIN_TOKENS - 1]
    beside = SimpleNamespace(side=object(), host_query_lens=lengths)
    assert GatedDeltaRule._chains(beside) == 2
    assert GatedDeltaRule._chains(beside, below=300) == 1  # the longer ones go in chunks
    assert GatedDeltaRule._chains(SimpleNamespace(side=None, host_query_lens=lengths)) == 0
    assert GatedDeltaRule._chains(SimpleNamespace(side=object(), host_query_lens=[1] * 8)) == 0


def blocks_of(layers):
    return [ParallelResidualBlock(mixer=DoublingMixer([]), ffn=RoutedExperts(hidden_size=H, experts=E, top=top, expert_size=I, limit=None,
                                                                             shared_size=I), norms={"n": CopyNorm()})
            for E, top, H, I in layers]


def test_where_two_branches_are_worth_a_fork_and_a_join():
    """Not captured: where a layer's kernels take longer than the host for its launches and the fork; captured: from some weights on."""
    from kvcore_amd.engine.runner import SIDE_TOKENS, branches_pay

    small, middle = blocks_of([(16, 4, 1024, 1024)] * 8), blocks_of([(32, 4, 2048, 2048)] * 16)
    for blocks, wanted in ((small, {640: False, 1000: False, 1250: False, 2048: True, 4096: True}),
                           (middle, {300: False, SIDE_TOKENS - 1: False, SIDE_TOKENS: True, 2048: True}),
                           (blocks_of([(128, 8, 2048, 1024)]), {639: False, 640: True}),
                           (blocks_of([(16, 2, 4096, 4096)]), {640: True})):
        assert {T: branches_pay(blocks, T, 2, False) for T in wanted} == wanted
    assert {T: branches_pay(small, T, 2, True) for T in (1, 2, 8, 64)} == {1: False, 2: True, 8: True, 64: True}
    assert branches_pay(middle, 1, 2, True) and branches_pay(small, 1, 4, True)
    plain = ParallelResidualBlock(mixer=DoublingMixer([]), ffn=AddingFeedForward([]), norms={"n": CopyNorm()})
    assert not branches_pay([plain], 4096, 2, False) and not branches_pay([plain], 64, 2, True)
    assert branches_pay([plain, *middle], 4096, 2, False)  # a block without branches has no say


def test_what_a_step_of_routed_experts_reads_and_multiplies():
    gated = RoutedExperts(hidden_size=8, experts=4, top=2, expert_size=16, limit=None, shared_size=24)
    read, ops_done = gated.beside_cost(10_000, 2)
    assert read == pytest.approx(3 * 8 * (4 * 16 + 24) * 2) and ops_done == 2 * 10_000 * 3 * 8 * (2 * 16 + 24)
    plain = RoutedExperts(hidden_size=8, experts=4, top=2, expert_size=16, limit=None, activation="relu_squared")
    assert plain.beside_cost(10_000, 4)[0] == pytest.approx(2 * 8 * 4 * 16 * 4)
