"""The device entry points inside captured HIP graphs.

A serving loop captures its per-token work once and replays it.  Each test
warms the call up eagerly (so that workspaces and prefill unit tables
exist), captures it, then replays the graph several times with new inputs
copied in between -- eager work and synchronisations between the replays --
and checks every replay against an eager call on the same inputs, bit for
bit (the kernels are deterministic).
"""
import numpy as np
import pytest
import torch

import inputs as I

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def replay_and_check(ctx, run, inputs, outputs, fresh, n=4):
    """run() launches the work on the current stream reading `inputs`
    (tensors) and writing `outputs`; fresh(i) gives new input values."""
    run()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run()
    torch.cuda.synchronize()
    for i in range(n):
        for t, v in zip(inputs, fresh(i)):
            t.copy_(v)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = [o.clone() for o in outputs]
        for o in outputs:
            o.fill_(float("nan"))
        run()  # eager, same inputs
        torch.cuda.synchronize()
        for a, b in zip(got, outputs):
            assert torch.equal(a, b), f"replay {i} differs from the eager call"
    ctx.check_status()


@pytest.mark.parametrize("T,d", [(4096, 512), (512, 256), (40, 256)])
def test_decode_in_a_graph(ctx, T, d):
    rng = np.random.default_rng(T + d)
    q = dev(rng.standard_normal(8 * d).astype(np.float32))
    K = dev(rng.standard_normal((T, d)).astype(np.float32))
    V = dev(rng.standard_normal((T, d)).astype(np.float32))
    out = torch.zeros(8 * d, device="cuda")
    replay_and_check(ctx, lambda: ctx.attend_decode(q, K, V, 0, T, 8, 1, d, out), [q, K], [out],
                     lambda i: [torch.randn(8 * d, device="cuda"), torch.randn(T, d, device="cuda")])


def test_ragged_stream_decode_in_a_graph(ctx):
    lens = np.array([5, 40, 20000, 3000, 700] * 4, np.int64)
    d = 512
    rng = np.random.default_rng(1)
    total = int(lens.sum())
    K = dev(rng.standard_normal((total, d)).astype(np.float32))
    V = dev(rng.standard_normal((total, d)).astype(np.float32))
    q = dev(rng.standard_normal((len(lens), 8 * d)).astype(np.float32))
    row0 = dev(np.concatenate([[0], np.cumsum(lens)[:-1]]).astype(np.int64))
    begin = dev(np.zeros(len(lens), np.int64))
    end = dev(lens)
    out = torch.zeros(len(lens) * 8 * d, device="cuda")
    replay_and_check(ctx, lambda: ctx.attend_decode_batch(q, K, V, row0, begin, end, int(lens.max()), 8, 1, d, out),
                     [q], [out], lambda i: [torch.randn(len(lens), 8 * d, device="cuda")])


@pytest.mark.parametrize("d,window", [(512, 0), (256, 512)])
def test_prefill_in_a_graph(ctx, d, window):
    N = 300
    rng = np.random.default_rng(d)
    q = dev(rng.standard_normal((N, 8 * d)).astype(np.float32))
    K = dev(rng.standard_normal((N, d)).astype(np.float32))
    V = dev(rng.standard_normal((N, d)).astype(np.float32))
    out = torch.zeros(N * 8 * d, device="cuda")
    replay_and_check(ctx, lambda: ctx.attend_prefill(q, K, V, 0, N, window, 8, 1, d, out), [q, V], [out],
                     lambda i: [torch.randn(N, 8 * d, device="cuda"), torch.randn(N, d, device="cuda")])


@pytest.mark.parametrize("d,window,pos0,N", [(512, 0, 0, 300), (256, 512, 700, 40), (512, 0, 4000, 17)])
def test_prefill_graph_outlives_its_shapes_turn_in_the_table_cache(d, window, pos0, N):
    """A context keeps the schedule tables of the last 128 prefill shapes; a
    captured graph's table stays beyond that.  The graph replays between and
    after eager calls of 160 other shapes."""
    import g4hip
    rng = np.random.default_rng(d + pos0)
    q = dev(rng.standard_normal((N, 8 * d)).astype(np.float32))
    K = dev(rng.standard_normal((pos0 + N, d)).astype(np.float32))
    V = dev(rng.standard_normal((pos0 + N, d)).astype(np.float32))
    out = torch.zeros(N * 8 * d, device="cuda")
    other = torch.zeros(300 * 8 * d, device="cuda")
    with g4hip.Context(0) as ctx:
        big = torch.zeros(1024, 8 * 512, device="cuda")  # the largest workspace first: it does not grow later
        ctx.attend_prefill(big, big, big, 0, 1024, 0, 8, 1, 512, torch.zeros_like(big))
        deep = torch.zeros(8200, 512, device="cuda")
        ctx.attend_prefill(big, deep, deep, 8000, 64, 0, 8, 1, 512, torch.zeros_like(big))

        def run():
            ctx.attend_prefill(q, K, V, pos0, N, window, 8, 1, d, out)

        run()
        ref = out.clone()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            run()
        for i in range(160):
            n = 1 + i % min(N, pos0 + N - 1)
            ctx.attend_prefill(q, K, V, i % (pos0 + N - n), n, 1 + i, 8, 1, d, other)
            if i % 40 == 39:
                out.fill_(float("nan"))
                torch.cuda.synchronize()
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(out, ref), f"after {i + 1} other shapes"
        run()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
        ctx.check_status()


@pytest.mark.parametrize("captured", [1, 0])
@pytest.mark.parametrize("d,window,pos0,N", [(512, 0, 0, 300), (256, 512, 700, 40), (512, 0, 4000, 17)])
def test_prefill_capture_in_the_other_form_than_the_warm_up(d, window, pos0, N, captured):
    """One eager call makes a shape's capture possible in either product form:
    nothing is allocated or copied then."""
    import g4hip
    from oracle import pyoracle as orc
    rng = np.random.default_rng(d + pos0 + captured)
    qn = rng.standard_normal((N, 8 * d), dtype=np.float32) * 0.3
    Kn, Vn = (rng.standard_normal((pos0 + N, d), dtype=np.float32) for _ in range(2))
    q, K, V = dev(qn), dev(Kn), dev(Vn)
    out = torch.zeros(N * 8 * d, device="cuda")
    ref, status = orc.attend_prefill(qn, Kn, Vn, pos0, window, 8, 1)
    assert not status.any()
    with g4hip.Context(0) as ctx:
        def run():
            ctx.attend_prefill(q, K, V, pos0, N, window, 8, 1, d, out)

        big = torch.zeros(8200, 8 * 512, device="cuda")  # a workspace large enough for both forms
        ctx.attend_prefill(big, big, big, 8000, 64, 0, 8, 1, 512, torch.zeros(64, 8 * 512, device="cuda"))
        ctx.set_prefill_exact(1 - captured)
        run()
        torch.cuda.synchronize()
        ctx.set_prefill_exact(captured)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            run()
        for _ in range(3):
            out.fill_(float("nan"))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            got = out.cpu().numpy().reshape(N, -1)
            assert max(I.rel_err(got[i], ref[i]) for i in range(N)) <= 1e-4
            run()  # the form's own table from here on
            torch.cuda.synchronize()
            got = out.cpu().numpy().reshape(N, -1)
            assert max(I.rel_err(got[i], ref[i]) for i in range(N)) <= 1e-4
        ctx.check_status()


def test_prepare_and_decode_step_in_a_graph(ctx):
    """A global layer step: fused q/k/v preparation with the append into the
    cache, then the decode over the cache."""
    d, T = 512, 1024
    rng = np.random.default_rng(7)
    K = dev(rng.standard_normal((T, d)).astype(np.float32))
    V = dev(rng.standard_normal((T, d)).astype(np.float32))
    q, k, v = (dev(rng.standard_normal(n).astype(np.float32)) for n in (8 * d, d, d))
    wq, wk = dev(rng.uniform(0.5, 1.5, d).astype(np.float32)), dev(rng.uniform(0.5, 1.5, d).astype(np.float32))
    freqs = dev(I.rope_freqs(3, d))
    out = torch.zeros(8 * d, device="cuda")
    qs, ks, vs = q.clone(), k.clone(), v.clone()

    def run():
        q.copy_(qs), k.copy_(ks), v.copy_(vs)  # the preparation works in place
        ctx.prepare_qkv(q, k, v, 1, T - 1, 8, 1, d, wq, wk, 1e-6, I.GLOBAL_BASE, freqs,
                        k_rows=K.view(-1)[(T - 1) * d:], v_rows=V.view(-1)[(T - 1) * d:], row_stride=d)
        ctx.attend_decode(q, K, V, 0, T, 8, 1, d, out)

    replay_and_check(ctx, run, [qs, ks, vs], [out],
                     lambda i: [torch.randn(8 * d, device="cuda"), torch.randn(d, device="cuda"),
                                torch.randn(d, device="cuda")])


@pytest.mark.parametrize("rows,cols", [(4096, 1536), (70000, 1536)])
def test_q8_0_matvecs_in_a_graph(ctx, rows, cols):
    """Most matrices quantize inside the mat-vec; the gate and up pair of
    70,000 rows (228 MB) quantizes into the context's workspace first (a
    second kernel in the graph)."""
    w = dev(I.q8_0_bytes(np.random.default_rng(rows).uniform(-1, 1, rows * cols).astype(np.float32)))
    up = dev(I.q8_0_bytes(np.random.default_rng(rows + 1).uniform(-1, 1, rows * cols).astype(np.float32)))
    x = torch.randn(cols, device="cuda")
    a, b = torch.zeros(rows, device="cuda"), torch.zeros(rows, device="cuda")

    def run():
        ctx.logits_q8_0(w, rows, cols, x, 30.0, a)
        ctx.gated_ffn_q8_0(w, up, rows, cols, x, b)

    replay_and_check(ctx, run, [x], [a, b], lambda i: [torch.randn(cols, device="cuda") * (i + 1)])


def test_fused_decode_step_in_a_graph(ctx):
    """A global layer step as g4_layer_attention runs it: one launch that
    prepares q and the new row, appends the row and attends (plus the merge)."""
    d, T = 512, 2048
    rng = np.random.default_rng(9)
    K = dev(rng.standard_normal((T, d)).astype(np.float32))
    V = dev(rng.standard_normal((T, d)).astype(np.float32))
    q, k, v = (dev(rng.standard_normal(n).astype(np.float32)) for n in (8 * d, d, d))
    wq, wk = dev(rng.uniform(0.5, 1.5, d).astype(np.float32)), dev(rng.uniform(0.5, 1.5, d).astype(np.float32))
    freqs = dev(I.rope_freqs(4, d))
    out = torch.zeros(8 * d, device="cuda")

    def run():
        ctx.decode_step_fused(q, k, v, wq, wk, 1e-6, I.GLOBAL_BASE, freqs, T - 1, K, V, d, T,
                              K.view(-1)[(T - 1) * d:], V.view(-1)[(T - 1) * d:], 8, 1, d, out)

    replay_and_check(ctx, run, [q, k, v], [out],
                     lambda i: [torch.randn(8 * d, device="cuda"), torch.randn(d, device="cuda"),
                                torch.randn(d, device="cuda")])


def _rows(rng, n, width):
    return dev(rng.standard_normal((n, width), dtype=np.float32) * 0.3)


@pytest.mark.parametrize("call", ["decode", "ragged", "ragged_row0", "stream", "prefill", "few_queries", "softcap"])
def test_graphs_outlive_the_growth_of_the_workspace(call):
    """A captured call keeps the context's buffers of its time; larger eager
    calls grow them twice between replays."""
    import g4hip
    rng = np.random.default_rng(5)
    d = 512
    out = torch.zeros(64 * 8 * d, device="cuda")
    with g4hip.Context(0) as ctx:
        if call == "decode":
            q, K, V, n = _rows(rng, 1, 8 * d), _rows(rng, 1000, d), _rows(rng, 1000, d), 8 * d
            run = lambda: ctx.attend_decode(q, K, V, 0, 1000, 8, 1, d, out)
        elif call in ("ragged", "ragged_row0", "stream"):
            lens = np.array([5, 700, 64, 333], np.int64) * (30 if call == "stream" else 1)
            longest, n = int(lens.max()), 4 * 8 * d
            q, K, V = _rows(rng, 4, 8 * d), _rows(rng, longest, d), _rows(rng, longest, d)
            begin, end, row0 = dev(lens * 0), dev(lens), dev(lens * 0) if call != "ragged_row0" else None
            run = lambda: ctx.attend_decode_batch(q, K, V, row0, begin, end, longest, 8, 1, d, out)
        elif call == "softcap":
            x = _rows(rng, 1, 1536)
            w = dev(np.tile(I.q8_0_bytes(rng.uniform(-1, 1, 1000 * 1536).astype(np.float32)), 90))
            n = 90000
            run = lambda: ctx.logits_q8_0(w, 90000, 1536, x, 30.0, out)
        else:
            pos0, N = (0, 60) if call == "prefill" else (600, 9)
            q, K, V, n = _rows(rng, N, 8 * d), _rows(rng, pos0 + N, d), _rows(rng, pos0 + N, d), N * 8 * d
            run = lambda: ctx.attend_prefill(q, K, V, pos0, N, 0, 8, 1, d, out)
        run()
        ref = out.clone()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            run()
        big = _rows(rng, 20000, d)
        bigq, bigout = _rows(rng, 64, 8 * d), torch.zeros(64 * 8 * d, device="cuda")
        for rows, B in ((8000, 1500), (20000, 3000)):
            ctx.attend_prefill(bigq, big, big, rows - 64, 64, 0, 8, 1, d, bigout)
            ones = torch.ones(B, dtype=torch.int64, device="cuda")  # a batch that needs more row offsets
            wide = torch.zeros(B, 8 * 256, device="cuda")
            ctx.attend_decode_batch(wide, big, big, None, ones * 0, ones, 1, 8, 1, 256, torch.zeros_like(wide))
            for _ in range(2):
                out.fill_(float("nan"))
                torch.cuda.synchronize()
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(out[:n], ref[:n])
        run()
        torch.cuda.synchronize()
        assert torch.equal(out[:n], ref[:n])
        ctx.check_status()
