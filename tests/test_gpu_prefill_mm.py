"""GPU parity of the grouped prefill product (k_q2g_mm) at the edges of its tiles and dispatch.

The fp64 oracle on every row; weights, h and the output are each rounded once to fp16, a relative
error of at most 2^-11 each, so the 2-norm of a segment's error is within 3 * 2^-11 of its own.
* contraction lengths with one group, a last step of one half (at most 4 groups) and of two clamped
  halves, whole steps, and the longest (2560); segments of 0, 1, 16, 17, 64, 65 and 130 rows; blob
  pools and the 9-tensor form with fp16 and bf16 scales; output columns below and above one tile;
* more segments than threads in a block, over a pool of few slots, with long and empty ones mixed in; blocks that
  take several column tiles of a segment, shares in 64-row batches, more than 4096 rows of a short contraction;
* the same rows in calls of different sizes, which select different kernels, give the same bits;
* an output that starts 2 bytes past a 16-byte boundary, and rows that name no source row, no output
  row and no slot, are handled alike in k_q2g_mm and, with short segments, the whole-K kernels.
"""
import numpy as np
import pytest

from helpers import expert_fn, experts_bf16, experts_np
from oracle import q2
from test_gpu_q2t import _grouped_t, _pools

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
BOUND = 3 * 2.0 ** -11
LONG = [0, 1, 16, 17, 64, 65, 130, 3, 0, 40]
SHORT = [1, 0, 2, 5, 17, 1, 3, 1, 0, 4]


def _plan(counts, n_tok, rng):
    m = int(sum(counts))
    seg_start = np.append(0, np.cumsum(counts)).astype(np.int32)
    return rng.integers(0, n_tok, m).astype(np.int32), rng.permutation(m).astype(np.int32), seg_start


def _check(y, x, row_tok, row_out, seg_start, seg_slot, fn, sdtype=None):
    for u, e in enumerate(seg_slot):
        r = np.arange(seg_start[u], seg_start[u + 1])
        if r.size:
            want = q2.switch_glu_expert(x[row_tok[r]].astype(np.float64), *fn(int(e)), bits=2, group=64, sdtype=sdtype)
            err = np.linalg.norm(y[row_out[r]].astype(np.float64) - want) / np.linalg.norm(want)
            assert err <= BOUND, (u, r.size, err)


@pytest.mark.parametrize("counts", [LONG, SHORT], ids=["long", "short"])
@pytest.mark.parametrize("form", ["blob", "fp16", "bf16"])
@pytest.mark.parametrize("hidden,inter", [(64, 64), (320, 192), (512, 576), (1152, 320), (2048, 512), (2560, 640)])
def test_mm_matches_oracle(hidden, inter, form, counts):
    from moe_offload import _lib, ops
    dev = torch.device("cuda")
    n_exp = len(counts)
    rng = np.random.default_rng(hidden + inter)
    mlx, blobs = experts_np(n_exp, hidden, inter, seed=3)
    if form == "bf16":
        mlx = experts_bf16(n_exp, hidden, inter, seed=4)
    x = rng.standard_normal((50, hidden)).astype(np.float16)
    row_tok, row_out, seg_start = _plan(counts, 50, rng)
    seg_slot = rng.permutation(n_exp).astype(np.int32)
    t = lambda a: torch.from_numpy(a).to(dev)
    if form == "blob":
        y = ops.q2_grouped_switch_glu(t(x), t(row_tok), t(seg_start), t(blobs), hidden, inter, row_out=t(row_out),
                                      n_out_rows=row_tok.size, seg_slot=t(seg_slot)).cpu().numpy()
    else:
        ts, ptrs, nbytes = _pools(mlx, dev)
        y = _grouped_t(_lib.lib(), t(x), t(row_tok), t(row_out), t(seg_start), t(seg_slot), ptrs, nbytes,
                       int(form == "bf16"), n_exp, hidden, inter, row_tok.size)
    _check(y, x, row_tok, row_out, seg_start, seg_slot, expert_fn(mlx), "bf16" if form == "bf16" else None)


def _few_rows():
    counts = np.random.default_rng(7).integers(0, 4, 1300)
    counts[[5, 700, 1299]] = [150, 64, 33]
    counts[100:180] = 0
    return counts


@pytest.mark.parametrize("hidden,inter,counts", [
    (512, 128, _few_rows()), (1088, 256, _few_rows()),
    # one block per segment and 3 of 16 column tiles (gate/up), for segments of one and two batches
    (640, 1024, np.random.default_rng(8).integers(1, 12, 300) + 12 * (np.arange(300) % 40 == 7)),
    # shares over more segments than a block has threads, 64-row batches (gate/up)
    (1088, 128, np.random.default_rng(9).integers(2, 20, 600)),
    # the same with few long segments, at a K of part of a step and of one whole step
    (320, 512, np.array([900, 0, 1200, 63, 700, 1500, 1, 65])),
    (512, 320, np.array([900, 0, 1200, 63, 700, 1500, 1, 65])),
], ids=["many_512", "many_1088", "span_640", "shares_1088", "long_320", "long_512"])
def test_mm_many_segments(hidden, inter, counts):
    from moe_offload import ops
    dev = torch.device("cuda")
    rng = np.random.default_rng(7)
    n_seg = counts.size
    mlx, blobs = experts_np(6, hidden, inter, seed=5)
    x = rng.standard_normal((60, hidden)).astype(np.float16)
    row_tok, row_out, seg_start = _plan(counts, 60, rng)
    seg_slot = rng.integers(0, 6, n_seg).astype(np.int32)
    t = lambda a: torch.from_numpy(a).to(dev)
    y = ops.q2_grouped_switch_glu(t(x), t(row_tok), t(seg_start), t(blobs), hidden, inter, row_out=t(row_out),
                                  n_out_rows=row_tok.size, seg_slot=t(seg_slot)).cpu().numpy()
    slot_of = np.repeat(seg_slot, counts)
    order = np.argsort(slot_of, kind="stable")               # one oracle call per slot
    starts = np.searchsorted(slot_of[order], np.arange(7))
    _check(y, x, row_tok[order], row_out[order], starts, np.arange(6), expert_fn(mlx))
    # the same rows as six long segments: other kernels, the same bits
    y6 = ops.q2_grouped_switch_glu(t(x), t(row_tok[order]), t(starts.astype(np.int32)), t(blobs), hidden, inter,
                                   row_out=t(row_out[order]), n_out_rows=row_tok.size).cpu().numpy()
    assert np.array_equal(y6, y)


@pytest.mark.parametrize("hidden,inter", [(320, 192), (192, 320), (2048, 512)])
@pytest.mark.parametrize("counts", [LONG, SHORT], ids=["long", "short"])
def test_mm_out_of_range_and_unaligned(counts, hidden, inter):
    from moe_offload import ops
    dev = torch.device("cuda")
    n_exp = len(counts)
    rng = np.random.default_rng(9)
    mlx, blobs = experts_np(n_exp, hidden, inter, seed=6)
    x = rng.standard_normal((30, hidden)).astype(np.float16)
    row_tok, row_out, seg_start = _plan(counts, 30, rng)
    m = row_tok.size
    seg_slot = np.arange(n_exp, dtype=np.int32)
    seg_slot[3] = n_exp                                       # no such slot: its rows are not written
    bad_tok, bad_out = int(seg_start[4]), int(seg_start[4]) + 1
    keep_out = int(row_out[bad_out])
    row_tok[bad_tok], row_out[bad_out] = 30, m
    buf = torch.full((m * hidden + 1,), 7.0, dtype=torch.float16, device=dev)
    y = buf[1:].view(m, hidden)
    t = lambda a: torch.from_numpy(a).to(dev)
    ops.q2_grouped_switch_glu(t(x), t(row_tok), t(seg_start), t(blobs), hidden, inter, row_out=t(row_out), n_out_rows=m,
                              seg_slot=t(seg_slot), out=y)
    got = y.cpu().numpy()
    assert float(buf[0]) == 7.0 and (got[keep_out] == 7).all() and (got[row_out[bad_tok]] == 0).all()
    skipped = np.arange(seg_start[3], seg_start[4])
    assert (got[row_out[skipped]] == 7).all()
    good = np.setdiff1d(np.arange(m), np.append(skipped, [bad_tok, bad_out]))
    for u in range(n_exp):
        r = good[(good >= seg_start[u]) & (good < seg_start[u + 1])]
        if r.size:
            want = q2.switch_glu_expert(x[row_tok[r]].astype(np.float64), *expert_fn(mlx)(u), bits=2, group=64)
            err = np.linalg.norm(got[row_out[r]].astype(np.float64) - want) / np.linalg.norm(want)
            assert err <= BOUND, (u, err)


@pytest.mark.parametrize("hidden,inter", [(2048, 512), (2048, 576), (384, 512), (2560, 192), (320, 256), (192, 128),
                                          (64, 64)])
@pytest.mark.parametrize("form", ["blob", "fp16", "bf16"])
def test_same_bits_whatever_the_call(hidden, inter, form):
    """At K = 2048 (gate/up), K = 512 (down) and up to K = 256 the whole-K kernels take the calls with few rows per
    segment and k_q2g_mm the others, in its several forms there and at every other K; a row's result does not depend
    on which: all rows in one call, one call per segment and one-tile segments give the same bits, also with a last
    slice only partly in range (inter 576, hidden 384, 320 and 192)."""
    from moe_offload import _lib, ops, prefill
    dev = torch.device("cuda")
    n_exp = 10
    rng = np.random.default_rng(hidden + inter)
    mlx, blobs = experts_np(n_exp, hidden, inter, seed=8)
    if form == "bf16":
        mlx = experts_bf16(n_exp, hidden, inter, seed=8)
    counts = np.array([130, 40, 1, 16, 64, 17, 70, 31, 90, 15])
    x = rng.standard_normal((50, hidden)).astype(np.float16)
    row_tok, row_out, seg_start = _plan(counts, 50, rng)
    seg_slot = rng.permutation(n_exp).astype(np.int32)
    t = lambda a: torch.from_numpy(a).to(dev)
    pools = _pools(mlx, dev) if form != "blob" else None

    def call(rt, ro, ss, sl):
        if form == "blob":
            out = torch.zeros((row_tok.size, hidden), dtype=torch.float16, device=dev)
            return ops.q2_grouped_switch_glu(t(x), t(rt), t(ss), t(blobs), hidden, inter, row_out=t(ro),
                                             n_out_rows=row_tok.size, seg_slot=t(sl), out=out).cpu().numpy()
        return _grouped_t(_lib.lib(), t(x), t(rt), t(ro), t(ss), t(sl), pools[1], pools[2], int(form == "bf16"), n_exp,
                          hidden, inter, row_tok.size)

    want = call(row_tok, row_out, seg_start, seg_slot)          # 474 rows over 10 segments
    tiles = prefill.tile_segments(seg_start, seg_slot)
    assert np.array_equal(call(row_tok, row_out, *tiles), want)
    for u in range(n_exp):
        r = slice(int(seg_start[u]), int(seg_start[u + 1]))
        got = call(row_tok[r], row_out[r], np.array([0, counts[u]], np.int32), seg_slot[u:u + 1])
        assert np.array_equal(got[row_out[r]], want[row_out[r]]), (u, int(counts[u]))
    _check(want, x, row_tok, row_out, seg_start, seg_slot, expert_fn(mlx), "bf16" if form == "bf16" else None)
