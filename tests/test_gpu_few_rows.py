"""GPU parity of the sampler's hand-off for few rows (more than 8 chunks a
row: the last workgroup to arrive selects from all the chunks' lists) against the
CPU oracle: 1-63 rows, top-k 1-64 across the two list widths, batches that mix
greedy and sampled rows, and inputs that defeat the selection's bound (ties,
all best entries in one chunk, fewer finite logits than top-k).  Tokens and
logits must be the oracle's bit for bit, except where its draw lies within
1e-6 of a boundary."""
import numpy as np
import pytest

import fg_hip
import workloads as W
from test_gpu_sampler import check, run_hip

pytestmark = pytest.mark.gpu


def batch(rows, vocab, k, kind, seed):
    rng = np.random.default_rng(seed)
    x = (rng.normal(0, 3, (rows, vocab))).astype(np.float32)
    if kind == "one_chunk":  # every row's best side by side, in one wave's slice
        n = min(200, vocab)
        first = rng.integers(0, vocab - n + 1, rows)
        for r in range(rows):
            x[r, first[r]:first[r] + n] += np.float32(30.0)
    elif kind == "eight_chunks":  # 8 spans of 80: more past the bound than is ranked at top-k 64
        for r in range(rows):
            for at in rng.integers(0, vocab - 80, 8):
                x[r, at:at + 80] += np.float32(30.0)
    elif kind == "equal":
        x[:] = np.float32(1.5)
    elif kind == "tied":
        x = (np.round(x / 0.5) * 0.5).astype(np.float32)
    elif kind == "sparse":  # 20 finite logits a row, NaN and -inf elsewhere
        y = np.full_like(x, -np.inf)
        y[:, ::3] = np.nan
        for r in range(rows):
            at = rng.choice(vocab, min(20, vocab), replace=False)
            y[r, at] = x[r, at]
        x = y
    base = [W.cfg(0.7, 0.9, k, presence=1.0, repetition=1.05), W.cfg(1.1, 1.0, k),
            W.cfg(0.0, 1.0, 1, repetition=1.1), W.cfg(0.9, 0.8, max(1, k // 2), frequency=0.3)]
    configs = [base[(r if rows > 2 else 2 * r) % len(base)] for r in range(rows)]
    counts = W.O.build_counts(W.O.gen_uniform_ids(rows, 64, vocab, seed, 5), vocab)
    return dict(logits=x, counts=counts, configs=configs, logprobs=0,
                uniforms=rng.random(rows).astype(np.float32))


@pytest.mark.parametrize("rows,vocab,k,kind", [
    (1, 248_320, 20, "normal"), (1, 262_144, 64, "normal"), (1, 262_145, 20, "normal"),
    (3, 4_099, 32, "normal"), (9, 50_257, 33, "normal"), (24, 50_257, 1, "normal"),
    (56, 9_001, 64, "normal"), (57, 9_001, 50, "normal"), (63, 20_000, 20, "normal"),
    (5, 50_257, 20, "one_chunk"), (5, 50_257, 64, "one_chunk"), (12, 30_000, 64, "eight_chunks"),
    (2, 151_936, 64, "eight_chunks"), (4, 30_001, 20, "equal"), (4, 30_001, 64, "equal"),
    (50, 30_001, 64, "equal"), (16, 50_000, 64, "tied"), (8, 40_000, 50, "sparse"),
    (8, 300, 40, "normal"), (40, 70, 64, "normal")])
def test_few_rows_match_the_oracle(dev, rows, vocab, k, kind):
    w = batch(rows, vocab, k, kind, seed=rows * 1000 + k)
    ref = W.oracle_run(w)
    s = fg_hip.HipSampler(vocab, rows)
    for call in range(3):
        check(w, run_hip(w, dev, sampler=s), ref, f"{kind} call {call}")


@pytest.mark.parametrize("rows,vocab,k,kind", [(1, 248_320, 20, "normal"), (2, 100_000, 64, "normal"),
                                               (8, 100_000, 40, "tied"), (63, 20_000, 64, "normal"),
                                               (70, 20_000, 20, "normal")])
def test_no_row_waits(dev, rows, vocab, k, kind):
    """Batches of fewer than 64 rows with a top list, and batches that mix
    greedy and sampled rows, wait for nobody: a wait limit of 0 fails no row."""
    w = batch(rows, vocab, k, kind, seed=rows + k)
    ref = W.oracle_run(w)
    s = fg_hip.HipSampler(vocab, rows)
    s.set_wait_limit(0)
    for call in range(2):
        check(w, run_hip(w, dev, sampler=s), ref, f"call {call}")
