"""The GEMM's 128-token tiles, with two workgroups per CU (one wave group, two
LDS stages) and with one (two wave groups, four stages), against the CPU oracle
at ragged rows and tokens: one, three and five K steps (fewer than the stages,
odd counts), widths 64, 128 and 192 (256 with two wave groups), both groups;
rows too long for the scale preload, min-term operands read word by word over
several blocks, and long rows whose token tiles go in runs of four.  Each case
names the form it is there for, which the plan has to give.

Every row of the first and the last 32 tokens and of a band around a tile
border, sampled tokens elsewhere, within rel 1e-5 (max-norm) of the oracle,
the bar of the other GEMM tests; the group-sum dump runs the same instances
and gives the same bits.
"""
import os
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from oracle import reference as ref
from webyiq_amd import ops
from conftest import gemm_form, rel_err

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# M, K, N, G, mode, rows per tile, waves per workgroup (four: one wave group)
CASES = [
    (3638, 384, 1029, 128, 0, 64, 4),
    (3049, 384, 655, 128, 2, 64, 4),
    (3210, 384, 2322, 128, 1, 128, 4),
    (3224, 384, 1176, 128, 2, 128, 4),
    (4000, 128, 2050, 128, 0, 192, 4),   # a single step
    (403, 640, 8475, 128, 2, 192, 4),    # five steps
    (824, 384, 4639, 32, 1, 64, 4),
    (641, 384, 8717, 32, 0, 128, 4),
    (404, 384, 5968, 32, 2, 192, 4),
    (594, 384, 423, 128, 2, 64, 8),
    (533, 384, 3484, 128, 2, 192, 8),
    (389, 640, 6633, 128, 2, 256, 8),
    (384, 384, 3484, 32, 2, 128, 8),     # group 32, two wave groups
    (900, 1152, 3484, 32, 1, 128, 8),    # nine steps over two wave groups
    (403, 3712, 8475, 128, 2, 192, 4),   # 29 scale words per row: staged with each step
    (395, 3712, 16870, 128, 0, 192, 4),
    (2496, 7552, 3164, 128, 0, 128, 4),  # 59 of them
    (533, 2176, 3484, 128, 2, 192, 8),   # 17 groups: min-term operands word by word
    (1024, 2176, 2050, 128, 0, 128, 8),
    (389, 2176, 6633, 128, 2, 256, 8),
    (403, 2176, 8475, 128, 2, 192, 4),
    (640, 4096, 3000, 128, 2, 128, 8),   # five token tiles: a run of four and one more
    (1290, 4224, 1000, 128, 1, 64, 8),   # eleven, 33 steps
]


@pytest.mark.parametrize("M,K,N,G,mode,rows,waves", CASES)
def test_shared_tiles(M, K, N, G, mode, rows, waves):
    form = gemm_form(M, K, N, G, None, mode)
    assert form == ("tiles", rows, waves, False), form
    print(f"[case] shared tiles M={M} K={K} N={N} G={G} mode={mode}", flush=True)
    rng = np.random.default_rng(M + K + N)
    wq, ws = ref.make_weight(rng, 2 * N if mode == 2 else N, K, G)
    xq, dx, xs = orc.quant_act(ref.make_activations(rng, M, K), None, G)
    y0 = rng.normal(size=(M, N)).astype(np.float32) if mode == 1 else None
    w = ops.Q4Tensor.from_numpy(wq, ws, K, G)
    a = ops.Acts(dev(xq), dev(dx), dev(xs), K, G)
    got = ops.gemm(w, a, mode=mode, y=None if y0 is None else dev(y0)).cpu().numpy()
    idx = np.unique(np.concatenate([np.arange(32), np.arange(112, 144), np.arange(M - 32, M), np.arange(5, M, 37)]))
    parts = np.array_split(idx, min(16, os.cpu_count() or 1))
    with ThreadPoolExecutor(len(parts)) as ex:
        want = np.concatenate(list(ex.map(
            lambda i: orc.linear(wq, ws, K, G, xq[i], dx[i], xs[i], mode=mode, y=None if y0 is None else y0[i]), parts)))
    assert rel_err(got[idx], want) < 1e-5
    assert np.isfinite(got).all()
    y, acc = ops.group_sums(ops.PATH_PREFILL, w, a, mode=mode, y=None if y0 is None else dev(y0))
    assert np.array_equal(y.cpu().numpy().view(np.uint32), got.view(np.uint32))
    t = np.array([0, 130, M - 1])
    assert np.array_equal(acc[dev(t)].cpu().numpy(), orc.group_acc(wq, K, G, xq[t]))
