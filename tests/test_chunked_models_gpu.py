"""The decoders with recurrent states over portions long enough to be cut into chunks, in bfloat16 in the engine, against
the plain implementations: a long portion beside a single token, a second long portion that starts from the states
which the first left, beside one that stays with the scan, and decoding from what the chunks left."""

from __future__ import annotations

import pytest
import torch

from tests import dirulorn_helpers, tazunex_helpers, vovalix_helpers
from tests import test_dirulorn_model_gpu as dirulorn
from tests import test_tazunex_model_gpu as tazunex
from tests import test_vovalix_model_gpu as vovalix
from tests.helpers import random_tokens

pytestmark = pytest.mark.gpu

# decoder, configuration, its chunk operation and the scan
CASES = [(dirulorn, dirulorn_helpers, "P", "ssm_chunks", "ssm_scan"), (dirulorn, dirulorn_helpers, "Q", "ssm_chunks", "ssm_scan"),
         (dirulorn, dirulorn_helpers, "M", "ssm_chunks", "ssm_scan"),
         (tazunex, tazunex_helpers, "A", "scalar_gate_chunks", "linear_state_scan"),
         (tazunex, tazunex_helpers, "B", "scalar_gate_chunks", "linear_state_scan"),
         (vovalix, vovalix_helpers, "A", "channel_gate_chunks", "linear_state_scan"),
         (vovalix, vovalix_helpers, "B", "channel_gate_chunks", "linear_state_scan")]


@pytest.mark.parametrize("module,helpers,name,chunks,scan", CASES, ids=lambda v: v if isinstance(v, str) else "")
def test_long_portions_then_more_of_them_then_single_tokens(module, helpers, name, chunks, scan, tmp_path, monkeypatch):
    from kvcore_amd.ops import library as ops

    config, page = helpers.CONFIGS[name]
    folder = helpers.make_model_dir(tmp_path, config, seed=91)
    cfg, weights = module.plain.load_model_folder(folder)
    V = cfg["vocab"]
    seqs = {"a": random_tokens(618, V, 21), "b": random_tokens(338, V, 22), "c": random_tokens(9, V, 23)}
    want = {k: module.oracle(f"long {name}", cfg, weights, v) for k, v in seqs.items()}
    calls: dict[str, list] = {chunks: [], scan: []}
    for op in calls:
        def spy(*args, _real=getattr(ops, op), _seen=calls[op], **kw):
            _seen.append(kw.get("start") or kw.get("below"))
            return _real(*args, **kw)
        monkeypatch.setattr(ops, op, spy)
    s = module.session_for(folder, torch.bfloat16, page, 1100)
    at = dict.fromkeys(seqs, 0)
    got, layers = {}, None
    plan = [dict(a=270, c=1), dict(a=340, b=100, c=1), dict(b=230, a=1, c=1)] + [dict(a=1, b=1, c=1)] * 6
    for i, entries in enumerate(plan):
        for seen in calls.values():
            seen.clear()
        record = {"step": i, "entries": [], "end": []}
        for k, n in entries.items():
            # every position around the edges of chunks and of the portion, and some between
            places = sorted({p for p in range(n) if p % 64 in (0, 1, 15, 16, 63) or p % 11 == 5} | {n - 1})
            record["entries"].append({"id": k, "tokens": seqs[k][at[k]: at[k] + n], "want": places})
        logits = s.run_step(record).logits.detach().cpu().double()
        row = iter(logits)
        for item in record["entries"]:
            for p in item["want"]:
                got[(item["id"], at[item["id"]] + p)] = next(row)
            at[item["id"]] += len(item["tokens"])
        if i < 3:  # chunks for the long portion of every such layer, the scan for the rest
            start = calls[chunks][0]
            layers = layers or len(calls[chunks])
            assert calls[chunks] == [start] * layers and calls[scan].count(start) == layers and start > 100, (i, calls)
        else:
            assert not calls[chunks]
    assert all(at[k] >= len(v) - 3 for k, v in seqs.items()) and s.runner.graph_replays > 0
    extra = {}
    if module is tazunex:
        extra["floors"] = {k: module.rounding_floor(cfg, weights, v, want[k], torch.bfloat16) for k, v in seqs.items()}
    module.compare(got, want, torch.bfloat16, **extra)
