"""The GEMM with K split between the waves of a workgroup (gemm_wave.hip),
against the CPU oracle at the edges of its tiles: 32 tokens x 32 or 64 rows,
1, 4 or 8 waves, fewer K steps than waves and step counts the waves do not
share evenly, ragged rows and tokens, and scale, sum and dx arrays that are
only 4-byte aligned (the kernel reads their four-word pieces word by word
then).  Each case names the form it is there for, which the plan has to give.

fp32 outputs within rel 1e-5 (max-norm) of the oracle, the bar of the other
GEMM tests: the int32 group sums are exact, and the fp32 sums of K / G terms
differ from the oracle's order by a few 2^-24 relative to the largest term.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from oracle import reference as ref
from webyiq_amd import ops
from conftest import gemm_form, rel_err

pytestmark = pytest.mark.gpu


def dev(a, shift=0):
    """a on the GPU, its first element `shift` elements past a 256-byte boundary."""
    t = torch.empty(a.size + 64, dtype=torch.from_numpy(a).dtype, device="cuda")
    t = t[shift:shift + a.size].view(a.shape)
    t.copy_(torch.from_numpy(np.ascontiguousarray(a)))
    return t


FORMATS = [(128, None), (32, None), (32, 32), (128, 32)]

# M, K, N, mode, shift, rows per tile and waves per workgroup, in every format
EDGES = [
    (1, 128, 1, 0, 0, 32, 8),        # one step: seven waves without work
    (33, 1152, 33, 1, 0, 32, 8),     # nine steps over eight waves, one token and one row past a tile
    (31, 640, 65, 2, 1, 64, 8),      # gate/up pairs, five steps, unaligned arrays
    (32, 2048, 97, 0, 3, 32, 8),     # unaligned arrays
]
# (groups of 32 keep narrow tiles up to 768 of them, and the 128-token tiles
# take many of the per-token shapes: each format has its own)
FOUR_WAVES = [
    (130, 640, 1700, 2, 1, 128, None),   # gate/up pairs, five steps over four waves, unaligned arrays
    (130, 640, 1700, 2, 1, 32, None),
    (130, 640, 1700, 2, 1, 32, 32),
    (130, 640, 1700, 2, 1, 128, 32),
    (130, 384, 1700, 2, 0, 32, None),    # three steps over four waves
    (130, 384, 1700, 2, 0, 32, 32),
    (130, 384, 1700, 2, 0, 128, 32),
    (520, 1152, 1555, 0, 2, 32, None),   # nine steps, unaligned arrays
    (520, 1152, 1555, 0, 2, 32, 32),
    (520, 1152, 1555, 0, 2, 128, 32),
    (840, 640, 1025, 1, 0, 32, None),    # eight tokens and one row past a tile
    (840, 640, 1025, 1, 0, 32, 32),
    (840, 640, 1025, 1, 0, 128, 32),
    (300, 1024, 2048, 0, 1, 128, None),
    (700, 1024, 1024, 1, 0, 128, None),
]
CASES = [(*c, G, GA) for c in EDGES for G, GA in FORMATS] + [(*c[:5], 64, 4, *c[5:]) for c in FOUR_WAVES]


@pytest.mark.parametrize("M,K,N,mode,shift,rows,waves,G,GA", CASES)
def test_wave_gemm_edges(M, K, N, mode, shift, rows, waves, G, GA):
    form = gemm_form(M, K, N, G, GA, mode)
    assert form == ("waves", rows, waves, False), form
    print(f"[case] wave gemm M={M} K={K} N={N} G={G} GA={GA} mode={mode} shift={shift}", flush=True)
    rng = np.random.default_rng(M + K + N + mode)
    wq, ws = ref.make_weight(rng, 2 * N if mode == 2 else N, K, G)
    x = ref.make_activations(rng, M, K)
    gaa = K if GA is None else GA
    xq, dx, xs = orc.quant_act(x, GA, G)
    y0 = rng.normal(size=(M, N)).astype(np.float32) if mode == 1 else None
    want = orc.linear(wq, ws, K, G, xq, dx, xs, mode=mode, y=y0, GA=gaa)
    w = ops.Q4Tensor(dev(wq.view("int32")), dev(ws.view("int32"), shift), K, G)
    a = ops.Acts(dev(xq), dev(dx, shift), dev(xs, shift), gaa, G)

    def run(m=None):
        y = dev(y0) if mode == 1 else torch.full((M, N), float("nan"), device="cuda")
        ops.gemm(w, a, mode=mode, y=y, params=None if m is None else ops.make_params(m=m))
        torch.cuda.synchronize()
        return y.cpu().numpy()
    got = run()
    assert rel_err(got, want) < 1e-5
    m = (M + 1) // 2  # device Params below the capacity: the same rows, the others untouched
    part = run(m)
    assert np.array_equal(part[:m].view(np.uint32), got[:m].view(np.uint32))
    base = y0 if mode == 1 else np.full((M, N), np.nan, np.float32)
    assert np.array_equal(part[m:].view(np.uint32), base[m:].view(np.uint32))


def sampled(M):
    """Every token of the first and the last tile, and some of each between."""
    return np.unique(np.concatenate([np.arange(min(M, 33)), np.arange(max(0, M - 33), M), np.arange(0, M, 29)]))


@pytest.mark.parametrize("M,K,N,G,GA,mode,kernel,waves", [
    (1050, 128, 2017, 32, 32, 0, "waves", 1),     # one step: one wave per tile
    (1050, 128, 2600, 128, 32, 1, "waves", 1),
    (1050, 128, 1050, 32, 32, 2, "waves", 1),
    (1050, 128, 1950, 128, 32, 2, "waves", 1),
    (1050, 128, 2000, 32, 32, 1, "waves", 4),     # under the line for mode 1
    (1050, 384, 4100, 32, 32, 1, "waves", 4),     # old values read late
    (1050, 256, 4100, 128, 32, 1, "waves", 4),
    (1050, 128, 4100, 128, None, 0, "tiles", 8),  # one step per token: the 128-token tiles
    (1050, 128, 4100, 32, None, 1, "tiles", 4),
])
def test_short_rows_many_tiles(M, K, N, G, GA, mode, kernel, waves):
    """Rows of one to three steps under many tiles, ragged in tokens and rows;
    the group-sum dump gives the same bits."""
    form = gemm_form(M, K, N, G, GA, mode)
    assert (form[0], form[2]) == (kernel, waves), form
    print(f"[case] short rows M={M} K={K} N={N} G={G} GA={GA} mode={mode}", flush=True)
    rng = np.random.default_rng(M + K + N + mode)
    wq, ws = ref.make_weight(rng, 2 * N if mode == 2 else N, K, G)
    gaa = K if GA is None else GA
    xq, dx, xs = orc.quant_act(ref.make_activations(rng, M, K), GA, G)
    y0 = rng.normal(size=(M, N)).astype(np.float32) if mode == 1 else None
    w = ops.Q4Tensor.from_numpy(wq, ws, K, G)
    a = ops.Acts(dev(xq), dev(dx), dev(xs), gaa, G)
    got = ops.gemm(w, a, mode=mode, y=None if y0 is None else dev(y0)).cpu().numpy()
    t = sampled(M)
    want = orc.linear(wq, ws, K, G, xq[t], dx[t], xs[t], mode=mode, y=None if y0 is None else y0[t], GA=gaa)
    assert rel_err(got[t], want) < 1e-5
    assert np.isfinite(got).all()
    y, acc = ops.group_sums(ops.PATH_PREFILL, w, a, mode=mode, y=None if y0 is None else dev(y0))
    assert np.array_equal(y.cpu().numpy().view(np.uint32), got.view(np.uint32))
    assert np.array_equal(acc[dev(t)].cpu().numpy(), orc.group_acc(wq, K, min(G, gaa), xq[t]))


@pytest.mark.parametrize("m", [0, 1, 32, 33, 96, 129, 130, 200])
def test_wave_gemm_active_tokens(m):
    """Device Params number the tiles of the step's m tokens only: rows below
    min(m, M) are those of the call on the whole capacity M, bit for bit (M
    picks the kernel and with it a row's order of sums), the rest keep their
    contents."""
    M, K, N, G = 130, 512, 1090, 32  # 5 token tiles x 18 or 35 row tiles: no multiple of the XCDs
    print(f"[case] wave gemm params m={m}", flush=True)
    rng = np.random.default_rng(4)
    for mode, rows in ((0, N), (2, 2 * N)):
        w = ops.Q4Tensor.from_numpy(*ref.make_weight(rng, rows, K, G), K, G)
        a = ops.Acts(*(dev(v) for v in orc.quant_act(ref.make_activations(rng, M, K), 32, G)), 32, G)
        full = ops.gemm(w, a, mode=mode).cpu().numpy()
        y = torch.full((M, N), float("nan"), device="cuda")
        ops.gemm(w, a, mode=mode, y=y, params=ops.make_params(m=m))
        got, k = y.cpu().numpy(), min(m, M)
        assert np.array_equal(got[:k].view(np.uint32), full[:k].view(np.uint32))
        assert np.isnan(got[k:]).all()


@pytest.mark.parametrize("M,K,N,G,mode", [
    (256, 6144, 2048, 128, 0), (384, 4096, 2048, 32, 0), (200, 8192, 640, 128, 1),
])
def test_wave_gemm_ignores_workspace(M, K, N, G, mode):
    """Long rows under too few tokens for pairs of workgroups: these calls ask
    for no workspace, and leave one that they are given alone."""
    assert gemm_form(M, K, N, G, None, mode, workspace=True)[0] == "waves"
    print(f"[case] wave gemm with a workspace M={M} K={K} N={N} G={G} mode={mode}", flush=True)
    rng = np.random.default_rng(M + K + N)
    wq, ws = ref.make_weight(rng, N, K, G)
    xq, dx, xs = orc.quant_act(ref.make_activations(rng, M, K), None, G)
    y0 = rng.normal(size=(M, N)).astype(np.float32)
    w = ops.Q4Tensor.from_numpy(wq, ws, K, G)
    a = ops.Acts(dev(xq), dev(dx), dev(xs), K, G)
    plain = ops.gemm(w, a, mode=mode, y=dev(y0))
    wsp = torch.zeros(8 << 20, dtype=torch.uint8, device="cuda")
    given = ops.gemm(w, a, mode=mode, y=dev(y0), workspace=wsp)
    assert torch.equal(given.view(torch.int32), plain.view(torch.int32))
    assert not wsp.any()
    t = sampled(M)
    want = orc.linear(wq, ws, K, G, xq[t], dx[t], xs[t], mode=mode, y=y0[t] if mode == 1 else None)
    assert rel_err(plain.cpu().numpy()[t], want) < 1e-5


def test_wave_gemm_beyond_one_grid():
    """More tiles than a grid of 2^32 threads holds: the call goes out as two
    launches, the second starting with columns 1024 (2^23 tiles of 64 rows are
    16 columns of 524,288 token tiles)."""
    M, K, N, G = (1 << 24) - 1, 256, 1030, 32
    if torch.cuda.mem_get_info()[0] < 110e9:
        pytest.skip("the outputs take 69 GB")
    assert gemm_form(M, K, N, G, 32) == ("waves", 64, 4, False)
    print(f"[case] wave gemm in two launches M={M} K={K} N={N}", flush=True)
    rng = np.random.default_rng(6)
    wq, ws = ref.make_weight(rng, N, K, G)
    base = orc.quant_act(ref.make_activations(rng, 4099, K), 32, G)  # repeated: row t is row t % 4099
    n = -(-M // 4099)
    xq, dx, xs = (dev(v).repeat(n, 1)[:M].contiguous() for v in base)
    y = torch.empty((M, N), device="cuda")
    for r in range(0, M, 1 << 22):
        y[r:r + (1 << 22)] = float("nan")
    ops.gemm(ops.Q4Tensor.from_numpy(wq, ws, K, G), ops.Acts(xq, dx, xs, 32, G), y=y)
    want = orc.linear(wq, ws, K, G, *base, GA=32)
    first = y[:4099].clone()
    assert rel_err(first.cpu().numpy(), want) < 1e-5
    for r in range(0, M, 4099 * 1024):  # every row like its copy among the first ones
        part = y[r:r + 4099 * 1024]
        k = part.shape[0] // 4099
        assert (part[:k * 4099].view(k, 4099, N) == first).all()
        assert torch.equal(part[k * 4099:], first[:part.shape[0] - k * 4099])


@pytest.mark.parametrize("GA", [None, 32])
def test_wave_gemm_special_values(GA):
    """NaN and infinite scales stay in their own rows and columns: a NaN
    activation scale spoils its token, an infinite weight scale its column,
    a zero activation scale gives a zero row; everything else is unchanged."""
    M, K, N, G = 40, 512, 70, 32
    rng = np.random.default_rng(9)
    wq, ws = ref.make_weight(rng, N, K, G)
    xq, dx, xs = orc.quant_act(ref.make_activations(rng, M, K), GA, G)
    gaa = K if GA is None else GA
    want = orc.linear(wq, ws, K, G, xq, dx, xs, GA=gaa)
    dx, ws = dx.copy(), ws.copy()
    dx[3] = np.nan
    dx[7] = 0.0
    ws[11, 5] = (ws[11, 5] & 0xFFFF0000) | 0x7C00  # scale = +inf
    y = ops.gemm(ops.Q4Tensor.from_numpy(wq, ws, K, G), ops.Acts(dev(xq), dev(dx), dev(xs), gaa, G))
    got = y.cpu().numpy()
    assert np.isnan(got[3]).all()
    rest = np.delete(np.arange(M), [3, 7])
    cols = np.delete(np.arange(N), 11)
    assert np.array_equal(got[7, cols], np.zeros(N - 1, np.float32))
    assert not np.isfinite(got[rest, 11]).any()
    assert rel_err(got[np.ix_(rest, cols)], want[np.ix_(rest, cols)]) < 1e-5
