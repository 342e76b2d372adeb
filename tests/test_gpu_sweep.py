"""Seeded random shapes against the oracle, beyond the hand-picked cases:
chunked prefill at random (pos0, N, window) for both head widths, and
ragged decode batches of random sizes, lengths and windows (through the
streamed path and the per-sequence split grid, whichever the launcher
picks).  Every query row and every sequence is checked, to the tolerance
of the other parity tests: 1e-4 relative
(crates/llm-gemma4/tests/synthetic_generate.rs:74-83).
"""
import numpy as np
import pytest
import torch

import inputs as I
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu
TOL = 1e-4


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _prefill_shapes():
    rng = np.random.default_rng(20261202)
    shapes = []
    for i in range(12):
        d = (256, 512)[i % 2]
        window = int(rng.choice([0, 512, 1, 7, 100, 4096])) if d == 256 else int(rng.choice([0, 0, 33]))
        shapes.append((d, window, int(rng.integers(0, 3000)), int(rng.integers(1, 400))))
    return shapes


@pytest.mark.parametrize("d,window,pos0,N", _prefill_shapes())
def test_prefill_random_shapes(ctx, d, window, pos0, N):
    print(f"[case] prefill sweep d={d} W={window} pos0={pos0} N={N}", flush=True)
    freqs = I.rope_freqs(pos0 + 1, d) if d == 512 else None
    base = I.GLOBAL_BASE if d == 512 else I.LOCAL_BASE
    K, V = I.kv_rows(3 * pos0 + N, pos0 + N, d, base, freqs)
    q = I.queries(5 * pos0 + N, N, d, base, freqs, pos0)
    out = torch.zeros(N * 8 * d, device="cuda")
    ctx.attend_prefill(dev(q), dev(K), dev(V), pos0, N, window, 8, 1, d, out)
    ctx.check_status()
    got = out.cpu().numpy().reshape(N, 8 * d)
    ref, status = orc.attend_prefill(q, K, V, pos0, window, 8, 1)
    assert not status.any()
    worst = max(I.rel_err(got[i], ref[i]) for i in range(N))
    print(f"[parity] prefill sweep d={d} W={window} pos0={pos0} N={N}: worst rel err {worst:.2e}")
    assert worst <= TOL


def _ragged_shapes():
    rng = np.random.default_rng(4242)
    shapes = []
    for i in range(10):
        d = (256, 512)[i % 2]
        B = int(rng.choice([1, 2, 5, 17, 40, 100]))
        hi = int(rng.choice([40, 600, 5000, 20000]))
        hi = max(1, min(hi, 120000 // B))  # keeps the host arrays and the oracle small
        window = int(rng.choice([0, 512])) if d == 256 else 0
        shapes.append((d, window, rng.integers(1, hi + 1, size=B).astype(np.int64).tolist()))
    return shapes


@pytest.mark.parametrize("d,window,lens", _ragged_shapes())
def test_ragged_decode_random_batches(ctx, d, window, lens):
    lens = np.array(lens, np.int64)
    B = lens.size
    print(f"[case] ragged sweep d={d} W={window} B={B} max={lens.max()} total={lens.sum()}", flush=True)
    rng = np.random.default_rng(int(lens.sum()) + d)
    gap = 2  # NaN rows between the sequences' caches: reading one poisons the result
    row0 = np.zeros(B, np.int64)
    at = 0
    for s in range(B):
        row0[s] = at
        at += int(lens[s]) + gap
    K = np.full((at, d), np.nan, np.float32)
    V = np.full((at, d), np.nan, np.float32)
    for s in range(B):
        K[row0[s]:row0[s] + lens[s]] = rng.standard_normal((int(lens[s]), d), dtype=np.float32)
        V[row0[s]:row0[s] + lens[s]] = rng.standard_normal((int(lens[s]), d), dtype=np.float32)
    q = rng.standard_normal((B, 8 * d), dtype=np.float32) * 0.1
    begin = np.array([I.attended_range(int(L) - 1, window)[0] for L in lens], np.int64)
    out = torch.zeros(B * 8 * d, device="cuda")
    ctx.attend_decode_batch(dev(q), dev(K), dev(V), dev(row0), dev(begin), dev(lens), int((lens - begin).max()),
                            8, 1, d, out)
    ctx.check_status()
    got = out.cpu().numpy().reshape(B, -1)
    worst = 0.0
    for s in range(B):
        rows = slice(row0[s] + begin[s], row0[s] + lens[s])
        worst = max(worst, I.rel_err(got[s], orc.attend(q[s], K[rows], V[rows], 8, 1)))
    print(f"[parity] ragged sweep d={d} W={window} B={B}: worst rel err {worst:.2e}")
    assert worst <= TOL


@pytest.mark.parametrize("d", [256, 512])
@pytest.mark.parametrize("B,bound", [(1, 33), (3, 90), (12, 512), (13, 512), (23, 512), (24, 512), (63, 512), (7, 2339)])
def test_ragged_decode_split_sizes(ctx, d, B, bound):
    """Batches on each side of the lines between split sizes (16 keys, then
    whole pairs of 32), with sequences of one key, of the bound, and around
    the sizes' multiples."""
    near = [1, 15, 16, 17, 31, 32, 33, 48, 64, 65, bound - 1, bound]
    lens = np.array([min(bound, near[(B + 5 * s) % len(near)]) for s in range(B)], np.int64)
    lens[B // 2] = bound
    print(f"[case] ragged splits d={d} B={B} bound={bound}", flush=True)
    test_ragged_decode_random_batches(ctx, d, 0, lens.tolist())


@pytest.mark.parametrize("d,bound", [(256, 512), (512, 250), (256, 130)])
def test_ragged_decode_after_non_finite_partials(ctx, d, bound):
    """The merge reads split slots past a short sequence's count: outputs
    left full of NaN there by an earlier batch's V must not reach its own.
    (Those batches' maxima and sums are finite; a test below poisons
    them.)"""
    B = 6
    K = np.random.default_rng(d).standard_normal((B * bound, d), dtype=np.float32) * 0.1
    V = np.full((B * bound, d), np.nan, np.float32)
    q = np.random.default_rng(bound).standard_normal((B, 8 * d), dtype=np.float32) * 0.1
    row0 = np.arange(B, dtype=np.int64) * bound
    begin = np.zeros(B, np.int64)
    out = torch.zeros(B * 8 * d, device="cuda")
    ctx.attend_decode_batch(dev(q), dev(K), dev(V), dev(row0), dev(begin), dev(begin + bound), bound, 8, 1, d, out)
    torch.cuda.synchronize()
    assert torch.isnan(out).all()
    V = np.random.default_rng(3).standard_normal((B * bound, d), dtype=np.float32)
    lens = np.array([1, 17, 33, bound // 2, bound - 1, bound], np.int64)
    ctx.attend_decode_batch(dev(q), dev(K), dev(V), dev(row0), dev(begin), dev(lens), bound, 8, 1, d, out)
    ctx.check_status()
    got = out.cpu().numpy().reshape(B, -1)
    for s in range(B):
        rows = slice(row0[s], row0[s] + lens[s])
        assert I.rel_err(got[s], orc.attend(q[s], K[rows], V[rows], 8, 1)) <= TOL


def _poison_and_check(ctx, d, poison, K, V, q, bound, lens, row0):
    """poison() leaves its partials in the workspace and fails its own status
    check; the batch over `lens` that follows must not see them."""
    import g4hip
    poison()
    with pytest.raises(g4hip.EngError):
        ctx.check_status()
    B = len(lens)
    out = torch.zeros(B * 8 * d, device="cuda")
    begin = np.zeros(B, np.int64)
    ctx.attend_decode_batch(dev(q), dev(K), dev(V), dev(row0), dev(begin), dev(lens), bound, 8, 1, d, out)
    ctx.check_status()
    got = out.cpu().numpy().reshape(B, -1)
    for s in range(B):
        rows = slice(row0[s], row0[s] + lens[s])
        assert I.rel_err(got[s], orc.attend(q[s], K[rows], V[rows], 8, 1)) <= TOL, s


@pytest.mark.parametrize("value", [np.nan, 1e38])
@pytest.mark.parametrize("d,bound", [(256, 135), (256, 250), (512, 144), (256, 260), (512, 400), (512, 512)])
def test_ragged_decode_after_non_finite_softmax_sums(ctx, d, bound, value):
    """9 to 32 split slots per sequence, each left with a NaN maximum or sum
    by a batch whose keys hold NaN, or overflow their scores: a shorter
    sequence in the slot's place must not see them.  (Splits are 16 keys.)"""
    B = 6
    rng = np.random.default_rng(d + bound)
    K = rng.standard_normal((B * bound, d), dtype=np.float32) * 0.1
    V = rng.standard_normal((B * bound, d), dtype=np.float32)
    q = rng.standard_normal((B, 8 * d), dtype=np.float32) * 0.1
    row0 = np.arange(B, dtype=np.int64) * bound
    bad = K.copy()
    bad[::5] = value  # every split holds some
    hot = np.full_like(q, 50.0)
    ends = np.full(B, bound, np.int64)
    out = torch.zeros(B * 8 * d, device="cuda")
    lens = np.array([1, 17, 33, bound // 2, bound - 17, bound], np.int64)
    _poison_and_check(ctx, d, lambda: ctx.attend_decode_batch(dev(hot), dev(bad), dev(V), dev(row0), dev(ends * 0),
                                                              dev(ends), bound, 8, 1, d, out),
                      K, V, q, bound, lens, row0)


@pytest.mark.parametrize("d", [256, 512])
def test_ragged_decode_over_another_bounds_outputs(ctx, d):
    """A batch with a larger bound leaves NaN outputs where a later batch's
    (m, l) pairs lie."""
    B, wide, bound = 6, 512, 200
    rng = np.random.default_rng(d)
    K = rng.standard_normal((B * wide, d), dtype=np.float32) * 0.1
    V = rng.standard_normal((B * wide, d), dtype=np.float32)
    q = rng.standard_normal((B, 8 * d), dtype=np.float32) * 0.1
    row0 = np.arange(B, dtype=np.int64) * wide
    ends = np.full(B, wide, np.int64)
    bad = K.copy()
    bad[::16] = np.nan
    nan_v = np.full_like(V, np.nan)
    out = torch.zeros(B * 8 * d, device="cuda")
    lens = np.array([1, 17, 33, bound // 2, bound - 17, bound], np.int64)
    _poison_and_check(ctx, d, lambda: ctx.attend_decode_batch(dev(q), dev(bad), dev(nan_v), dev(row0), dev(ends * 0),
                                                              dev(ends), wide, 8, 1, d, out),
                      K, V, q, bound, lens, row0)


@pytest.mark.parametrize("chunk,pos0,N", [(0, 890, 40), (16, 0, 300)])
def test_generic_prefill_after_non_finite_softmax_sums(ctx, chunk, pos0, N):
    """The same through a prompt chunk of a shape outside the MFMA prefill (4
    heads on one KV head), whose queries have different split counts."""
    import g4hip
    d, heads = 256, 4
    rng = np.random.default_rng(pos0 + N)
    K = rng.standard_normal((pos0 + N, d), dtype=np.float32) * 0.1
    V = rng.standard_normal((pos0 + N, d), dtype=np.float32)
    q = rng.standard_normal((N, heads * d), dtype=np.float32) * 0.1
    out = torch.zeros(N * heads * d, device="cuda")
    ctx.set_decode_chunk(chunk)
    try:
        bad = K.copy()
        bad[::5] = np.nan
        ctx.attend_prefill(dev(q), dev(bad), dev(V), pos0, N, 0, heads, 1, d, out)
        with pytest.raises(g4hip.EngError):
            ctx.check_status()
        ctx.attend_prefill(dev(q), dev(K), dev(V), pos0, N, 0, heads, 1, d, out)
        ctx.check_status()
    finally:
        ctx.set_decode_chunk(0)
    got = out.cpu().numpy().reshape(N, -1)
    for i in range(N):
        assert I.rel_err(got[i], orc.attend(q[i], K[:pos0 + i + 1], V[:pos0 + i + 1], heads, 1)) <= TOL, i


@pytest.mark.parametrize("d", [256, 512])
@pytest.mark.parametrize("B,bound", [(32, 33), (32, 64), (33, 64), (43, 48), (85, 128), (86, 65), (86, 96), (86, 128),
                                     (86, 129), (150, 40), (255, 128)])
def test_ragged_short_contexts(ctx, d, B, bound):
    """Batches on both sides of the line where each short context stays one
    split, lengths from 1 to the bound."""
    rng = np.random.default_rng(B * bound + d)
    lens = rng.integers(1, bound + 1, B)
    lens[:3] = 1, bound, (bound + 1) // 2
    row0 = np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int64)
    K = rng.standard_normal((int(lens.sum()), d), dtype=np.float32) * 0.1
    V = rng.standard_normal((int(lens.sum()), d), dtype=np.float32)
    q = rng.standard_normal((B, 8 * d), dtype=np.float32)
    out = torch.full((B * 8 * d,), float("nan"), device="cuda")
    ctx.attend_decode_batch(dev(q), dev(K), dev(V), dev(row0), dev(np.zeros(B, np.int64)), dev(lens.astype(np.int64)),
                            bound, 8, 1, d, out)
    ctx.check_status()
    got = out.cpu().numpy().reshape(B, -1)
    for s in range(B):
        rows = slice(row0[s], row0[s] + lens[s])
        assert I.rel_err(got[s], orc.attend(q[s], K[rows], V[rows], 8, 1)) <= TOL, s
