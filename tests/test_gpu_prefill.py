"""Prefill path (FastExperts) on the GPU: MFMA grouped GEMMs against the CPU oracle (one full-K chain a row,
exl3_prefill.cu:14-23), the reference probe's row cases (fast_experts.rs:247-286), shared-X == separate-X,
graph replays byte-identical, and the MoE layer at the 8K-token prefill shape."""
import numpy as np
import pytest
import torch

from refs import DecodedExperts, assert_close, assert_rows_close, graph_kernels, np_u16, window_reference

pytestmark = pytest.mark.gpu

D, N, BITS = 2048, 1536, 4


def _probe_picks(rows, E, slots):
    # fast_experts.rs:247-286: (r * 7 + slot) % 16 for the routed slots, the shared expert last
    return np.array([[(E if s == slots - 1 else (r * 7 + s) % 16) for s in range(slots)] for r in range(rows)],
                    np.int32)


@pytest.fixture(scope="module")
def weights():
    import synth
    return synth.experts(17, D, N, BITS, seed=77)


@pytest.mark.parametrize("rows,maxm", [(1, 129), (63, 129), (64, 129), (65, 129), (129, 129)])
def test_fast_experts_reference_cases(gfr, oracle, weights, rows, maxm):
    import synth
    slots = 5
    w = weights
    picks_np = _probe_picks(rows, 16, slots)
    picks = torch.from_numpy(picks_np).cuda()
    x = synth.activations(rows, D, 3 + rows)
    g = gfr.Grouping(17, slots, maxm)
    g.run(picks, rows)
    fx = gfr.FastExperts(D, N, slots, slots, 17, maxm)
    fx.run(w, x, picks, g.ids, g.count, g.members, rows, maxm, shared_x=False)
    torch.cuda.synchronize()
    y = fx.output[:rows * slots].cpu().numpy()
    assert np.all(np.isfinite(y))
    dec = DecodedExperts(oracle, w)
    xb = np_u16(x)
    for r, s in [(0, 0), (rows - 1, slots - 1)]:
        want, _ = dec.row(xb[r], int(picks_np[r, s]), sk_gu=1, sk_d=1, warps=1)
        assert_close(y[r * slots + s], want, what=f"rows {rows} row {r} slot {s}")
    # every (row, slot) output (fast_experts.rs:353-361 compares every output of the window)
    assert_rows_close(y, window_reference(oracle, w, x, picks_np).reshape(rows * slots, D), what=f"rows {rows}")


def test_shared_x_equals_separate_x(gfr, weights):
    """With suh_g == suh_u, the shared-rotation launch is byte-identical to the separate one (fast_experts.rs:369-381)."""
    import synth
    import dataclasses
    w = dataclasses.replace(weights, suh_u=weights.suh_g)
    rows, slots, maxm = 70, 5, 70
    picks = torch.from_numpy(_probe_picks(rows, 16, slots)).cuda()
    x = synth.activations(rows, D, 9)
    g = gfr.Grouping(17, slots, maxm)
    g.run(picks, rows)
    fx = gfr.FastExperts(D, N, slots, slots, 17, maxm)
    fx.run(w, x, picks, g.ids, g.count, g.members, rows, maxm, shared_x=True)
    a = fx.output[:rows * slots].clone()
    fx.run(w, x, picks, g.ids, g.count, g.members, rows, maxm, shared_x=False)
    assert torch.equal(a, fx.output[:rows * slots])


def test_prefill_graph_replays(gfr, weights):
    import synth
    rows, slots, maxm = 200, 5, 256
    picks = torch.from_numpy(_probe_picks(rows, 16, slots)).cuda()
    x = synth.activations(rows, D, 10)
    g = gfr.Grouping(17, slots, maxm)
    fx = gfr.FastExperts(D, N, slots, slots, 17, maxm)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        g.run(picks, rows, stream=s)
        fx.run(weights, x, picks, g.ids, g.count, g.members, rows, maxm, False, stream=s)
        s.synchronize()
        eager = fx.output[:rows * slots].clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            g.run(picks, rows, stream=s)
            fx.run(weights, x, picks, g.ids, g.count, g.members, rows, maxm, False, stream=s)
    for _ in range(3):
        fx.output.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(fx.output[:rows * slots], eager)


def test_moe_prefill_config4_tokens(gfr, oracle):
    """Config 4 shape: 8192 tokens, 64 routed + 1 shared, top-4, uniform routing: routing exact; three tokens against
    the oracle's own row order, and every token's output against the whole-window reference."""
    import synth
    E, topk, rows = 64, 4, 8192
    w = synth.experts(E + 1, D, N, BITS, seed=5)
    x = synth.activations(rows, D, 6)
    lg = synth.logits(rows, E, 7)
    m = gfr.Moe(D, N, E, topk, rows)
    m.run(w, x, lg, rows)
    torch.cuda.synchronize()
    out = m.output[:rows].cpu().numpy()
    assert np.all(np.isfinite(out))
    p, wt = oracle.route(lg.cpu().numpy(), topk, E)
    assert np.array_equal(m.picks[:rows].cpu().numpy(), p)
    dec = DecodedExperts(oracle, w)
    xb = np_u16(x)
    for r in (0, 4097, rows - 1):
        ys = np.stack([dec.row(xb[r], int(e), sk_gu=1, sk_d=1, warps=1)[0] for e in p[r]])
        want = oracle.combine(ys, wt[r:r + 1], 1, topk + 1)
        assert_close(out[r], want[0], what=f"token {r}")
    y = window_reference(oracle, w, x, p, workers=16)
    assert_rows_close(out, oracle.combine(y, wt, rows, topk + 1), what="config 4, every token")


@pytest.mark.parametrize("bits", [2, 3, 4, 5])
@pytest.mark.parametrize("rows", [40, 320])
def test_fast_experts_bit_widths(gfr, oracle, bits, rows):
    """K = 2, 3, 4, 5 (config 5's mixed bit rates) at C5's hidden size against the oracle: every width decodes its
    trellis straight into MFMA A fragments, through one funnel shift a group of four values. 40 rows (360 pairs) run the split-K programs, 320 rows (2880 pairs) the full-K items with the fused
    epilogues."""
    import synth
    Dk, Nk, E, slots, maxm = 5120, 1536, 9, 9, rows
    w = synth.experts(E, Dk, Nk, bits, seed=90 + bits)
    picks_np = np.array([[(r * 3 + s) % (E - 1) if s < slots - 1 else E - 1 for s in range(slots)]
                         for r in range(rows)], np.int32)
    picks_np[:, :slots - 1] = np.sort(picks_np[:, :slots - 1], axis=1)
    picks = torch.from_numpy(picks_np).cuda()
    x = synth.activations(rows, Dk, 5 + bits)
    g = gfr.Grouping(E, slots, maxm)
    g.run(picks, rows)
    fx = gfr.FastExperts(Dk, Nk, slots, slots, E, maxm)
    fx.run(w, x, picks, g.ids, g.count, g.members, rows, maxm, shared_x=False)
    torch.cuda.synchronize()
    y = fx.output[:rows * slots].cpu().numpy()
    assert np.all(np.isfinite(y))
    dec = DecodedExperts(oracle, w)
    xb = np_u16(x)
    for r, s in [(0, 0), (rows - 1, 5)]:
        want, _ = dec.row(xb[r], int(picks_np[r, s]), sk_gu=1, sk_d=1, warps=1)
        assert_close(y[r * slots + s], want, what=f"K={bits} row {r} slot {s}")
    assert_rows_close(y, window_reference(oracle, w, x, picks_np).reshape(rows * slots, Dk),
                      what=f"K={bits} rows {rows}, every (row, slot)")


@pytest.mark.parametrize("bits", [2, 3, 4, 5])
def test_moe_prefill_config5_chunk(gfr, oracle, bits):
    """Config 5's prefill chunk at each of the stack's bit widths: 16384 tokens, hidden 5120, 160 routed + 1 shared,
    top-8, Zipf(1.1) routing; routing exact, the first, a middle and the last token against the oracle, and 64 spread
    tokens against the whole-window reference."""
    import synth
    E, Dk, Nk, topk, rows = 160, 5120, 1536, 8, 16384
    w = synth.experts(E + 1, Dk, Nk, bits, seed=71 if bits == 3 else 71 + 10 * bits)
    x = synth.activations(rows, Dk, 72)
    lg = synth.zipf_logits(rows, E, topk, 1.1, 73)
    m = gfr.Moe(Dk, Nk, E, topk, rows)
    m.run(w, x, lg, rows)
    torch.cuda.synchronize()
    out = m.output[:rows].cpu().numpy()
    assert np.all(np.isfinite(out))
    p, wt = oracle.route(lg.cpu().numpy(), topk, E)
    assert np.array_equal(m.picks[:rows].cpu().numpy(), p)
    dec = DecodedExperts(oracle, w)
    xb = np_u16(x)
    for r in (0, rows // 2 + 1, rows - 1):
        ys = np.stack([dec.row(xb[r], int(e), sk_gu=1, sk_d=1, warps=1)[0] for e in p[r]])
        want = oracle.combine(ys, wt[r:r + 1], 1, topk + 1)
        assert_close(out[r], want[0], what=f"config 5 K={bits} token {r}")
    sel = np.linspace(0, rows - 1, 64).astype(np.int64)
    y = window_reference(oracle, w, x[torch.from_numpy(sel).cuda()], p[sel], workers=16)
    assert_rows_close(out[sel], oracle.combine(y, wt[sel], len(sel), topk + 1), what=f"config 5 K={bits}, 64 tokens")


def _unpair(rows_u16):
    """Pair order of the prefill B operand (pair m of a 16-value k tile = (x[m + 8] low, x[m] high)) -> natural."""
    t = rows_u16.reshape(rows_u16.shape[0], -1, 8, 2)
    return np.concatenate([t[:, :, :, 1], t[:, :, :, 0]], axis=2).reshape(rows_u16.shape)


@pytest.mark.parametrize("hidden,slots,rows,shared_x", [
    (2048, 5, 37, False),     # the config 2-4 shape: 10 (slot, matrix) rows, up to 16 a launch form
    (1280, 5, 1, True),       # shared rotation: 5 rows
    (5120, 9, 13, False),     # config 5: 18 rows, up to 32
    (1280, 17, 3, False),     # 34 rows, up to 64
])
def test_prefill_rotation_bitexact(gfr, oracle, hidden, slots, rows, shared_x):
    """The prefill input rotation (prefill_rot_kernel) is rot_in (exl3.cu:224-241) bit for bit, for every pair and
    both matrices, at every (slot, matrix) row count the launch distinguishes."""
    import synth
    import dataclasses
    E = slots + 3
    w = synth.experts(E, hidden, 256, 2, seed=hidden + slots)
    if shared_x:
        w = dataclasses.replace(w, suh_u=w.suh_g)
    rng = np.random.default_rng(slots)
    picks_np = np.stack([rng.permutation(E)[:slots] for _ in range(rows)]).astype(np.int32)
    picks = torch.from_numpy(picks_np).cuda()
    x = synth.activations(rows, hidden, slots + 1)
    g = gfr.Grouping(E, slots, rows)
    g.run(picks, rows)
    fx = gfr.FastExperts(hidden, 256, slots, slots, E, rows)
    fx.run(w, x, picks, g.ids, g.count, g.members, rows, rows, shared_x=shared_x)
    torch.cuda.synchronize()
    xs = np_u16(x)
    for m in ((0,) if shared_x else (0, 1)):
        got = _unpair(np_u16(fx.rotated[m][:rows * slots]))
        suh = np_u16(w.suh_u if m else w.suh_g)
        for r in range(rows):
            for s in range(slots):
                want = oracle.rot(xs[r], suh[picks_np[r, s]])
                assert np.array_equal(got[r * slots + s], want), \
                    f"matrix {m} row {r} slot {s}: {np.sum(got[r * slots + s] != want)} values differ"


@pytest.mark.parametrize("hidden,routed,topk,rows,glm", [
    (2048, 64, 4, 37, False),     # config 3's shape: softmax gate, 5 slots
    (1024, 288, 8, 9, True),      # the reference's router: GLM's biased sigmoid gate over 288 experts, 9 slots
    (1024, 288, 8, 12, True),     # 96 picks
    (1024, 288, 8, 13, True),     # ... and 104, in two rounds of eight rows
    (1024, 288, 8, 16, True),     # the most rows above 100 picks that one launch routes, groups and rotates ...
    (1024, 288, 8, 17, True),     # ... a launch that routes, then one that groups and rotates
    (1024, 64, 4, 25, False),     # 100 picks: still one launch ...
    (1024, 64, 4, 26, False),     # ... 104: two
    (512, 16, 2, 256, False),     # the largest window of those launches
    (512, 16, 2, 300, False),     # larger windows: the rotation rides on the grouping's scatter launch
    (1024, 288, 8, 260, True),    # ... with GLM's gate, full-K items
])
def test_moe_fused_rotation_bitexact(gfr, oracle, hidden, routed, topk, rows, glm):
    """Windows of at most 256 rows on the prefill engine route, group and rotate in one launch: workgroup 0 routes and
    groups, the others route their own token again and rotate its pairs; larger windows rotate in the grouping's
    scatter launch, from the routed picks. Both routings must pick the same experts:
    every rotated (pair, matrix) row against rot_in (exl3.cu:224-241) of the layer's pick for it, bit for bit, and
    the softmax gate's picks against the oracle's."""
    import synth
    w = synth.experts(routed + 1, hidden, 256, 2, seed=hidden + rows)
    x = synth.activations(rows, hidden, rows + 3)
    lg = synth.logits(rows, routed, rows + 4)
    m = gfr.Moe(hidden, 256, routed, topk, rows)
    bias = None
    if glm:
        bias = torch.randn(routed, generator=torch.Generator(device="cuda").manual_seed(5), device="cuda") * 0.1
        m.set_router(bias, 2.5)
    m.run(w, x, lg, rows)
    torch.cuda.synchronize()
    # the rotating workgroups must have used the picks workgroup 0 wrote (the routers themselves against the oracle,
    # near-ties of GLM's gate included, are tested with the decode path)
    p = m.picks[:rows].cpu().numpy()
    if not glm:
        assert np.array_equal(p, oracle.route(lg.cpu().numpy(), topk, routed)[0])
    xs = np_u16(x)
    for mat in (0, 1):
        got = _unpair(np_u16(m.rotated(mat, rows)))
        suh = np_u16(w.suh_u if mat else w.suh_g)
        for r in range(rows):
            for s in range(topk + 1):
                want = oracle.rot(xs[r], suh[p[r, s]])
                assert np.array_equal(got[r * (topk + 1) + s], want), \
                    f"matrix {mat} row {r} slot {s}: {np.sum(got[r * (topk + 1) + s] != want)} values differ"


@pytest.mark.parametrize("N,bits", [(512, 4), (256, 4), (256, 3)])
@pytest.mark.parametrize("rows", [32, 300, 1024])
def test_moe_prefill_graph_replays(gfr, rows, N, bits):
    """A captured prefill-engine layer replays to the eager bytes, across two weight sets and routings: a small window
    (route + group + rotation in one launch), a larger one (the rotation in the grouping's scatter launch), both on the
    split-K programs at inter 512 and on the few-row items at 256, which has no split-K form, and a window on the largest
    items. Each replay follows eager work that clears the output."""
    import synth
    E, D, topk = 16, 512, 2
    ws = [synth.experts(E + 1, D, N, bits, seed=s) for s in (31, 32)]
    xs = [synth.activations(rows, D, 33 + j) for j in range(2)]
    lgs = [synth.logits(rows, E, 35 + j) for j in range(2)]
    m = gfr.Moe(D, N, E, topk, rows)
    s = torch.cuda.Stream()
    eager = []
    with torch.cuda.stream(s):
        for j in range(2):
            m.run(ws[j], xs[j], lgs[j], rows, stream=s)
            s.synchronize()
            eager.append(m.output[:rows].clone())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            m.run(ws[0], xs[0], lgs[0], rows, stream=s)
            m.run(ws[1], xs[1], lgs[1], rows, stream=s)
    assert not torch.equal(eager[0], eager[1])
    for _ in range(3):
        m.output.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(m.output[:rows], eager[1])


@pytest.mark.parametrize("routed,topk,rows,launches", [
    (160, 8, 12, 5), (160, 8, 13, 5), (288, 8, 16, 5), (288, 8, 17, 6), (64, 4, 25, 5), (64, 4, 26, 6), (64, 1, 100, 5),
    (64, 1, 101, 6)])
def test_window_launches(gfr, routed, topk, rows, launches):
    """A window's launches: route + group + rotation, gate/up programs, their epilogue, down programs, finish; above 16
    rows and 100 picks the routing is a launch of its own."""
    import synth
    w = synth.experts(routed + 1, 512, 512, 2, seed=30)
    x, lg = synth.activations(rows, 512, 31), synth.logits(rows, routed, 32)
    m = gfr.Moe(512, 512, routed, topk, rows)
    assert graph_kernels(lambda s: m.run(w, x, lg, rows, stream=s)) == launches


def test_split_window_with_many_experts(gfr, oracle):
    """A split-K window (at most 2048 pairs, 32-row items) whose routing spreads over 1023 experts with one member each
    plus a shared expert with every row: the plan holds 1023 + 32 items, more than an item count sized for 128-row
    items would hold. Sampled tokens against the oracle."""
    import synth
    routed, topk, rows, Dk, Nk, bits = 1023, 1, 1024, 512, 512, 4
    w = synth.experts(routed + 1, Dk, Nk, bits, seed=1023)
    x = synth.activations(rows, Dk, 11)
    lg = torch.randn((rows, routed), generator=torch.Generator(device="cuda").manual_seed(12), device="cuda")
    target = torch.arange(rows, device="cuda") % routed
    lg[torch.arange(rows, device="cuda"), target] = 10.0
    m = gfr.Moe(Dk, Nk, routed, topk, rows)
    m.run(w, x, lg, rows)
    torch.cuda.synchronize()
    out = m.output[:rows].cpu().numpy()
    assert np.all(np.isfinite(out))
    p, wt = oracle.route(lg.cpu().numpy(), topk, routed)
    assert np.array_equal(m.picks[:rows].cpu().numpy(), p)
    assert len(set(p[:, 0].tolist())) == routed
    dec = DecodedExperts(oracle, w)
    xb = np_u16(x)
    for r in (0, 511, 1022, 1023):
        ys = np.stack([dec.row(xb[r], int(e), sk_gu=1, sk_d=1, warps=1)[0] for e in p[r]])
        want = oracle.combine(ys, wt[r:r + 1], 1, topk + 1)
        assert_close(out[r], want[0], what=f"token {r}")
    y = window_reference(oracle, w, x, p, workers=16)
    assert_rows_close(out, oracle.combine(y, wt, rows, topk + 1), what="1023 experts, every token")


@pytest.mark.parametrize("bits", [2, 3, 4, 5])
@pytest.mark.parametrize("form,hidden,inter", [("few", 256, 256), ("few", 768, 512), ("large", 256, 256),
                                               ("large", 1280, 256)])
def test_prefill_item_bodies(gfr, oracle, bits, form, hidden, inter):
    """Experts with member counts around every body's and item's rows (16-row blocks, the 32- and 96-row bodies, the
    form's item), at K depths shorter and longer than the staged steps: every output against the oracle. Hidden sizes
    that are not multiples of 512 have no split-K form; fewer than 100 pairs an expert run the few-row form."""
    import synth
    bm = {2: 176, 3: 160, 4: 176, 5: 144}[bits]
    counts = [1, 15, 16, 17, 31, 32, 33, 95, 96, 97, 193] if form == "few" else [1, 32, 33, 96, 97, bm - 1, bm, bm + 1,
                                                                              2 * bm + 1]
    E, rows = len(counts), sum(counts)
    assert (rows < 100 * E) == (form == "few")
    rng = np.random.default_rng(bits)
    picks_np = rng.permutation(np.repeat(np.arange(E, dtype=np.int32), counts)).reshape(rows, 1)
    picks = torch.from_numpy(picks_np).cuda()
    w = synth.experts(E, hidden, inter, bits, seed=600 + bits)
    x = synth.activations(rows, hidden, 31 + bits)
    g = gfr.Grouping(E, 1, rows)
    g.run(picks, rows)
    fx = gfr.FastExperts(hidden, inter, 1, 1, E, rows)
    fx.run(w, x, picks, g.ids, g.count, g.members, rows, rows, shared_x=False)
    torch.cuda.synchronize()
    # the sums' order differs from the oracle's, so an activation's bf16 rounding may go the other way: 2^-8 of one value
    # of at most 150 (10 * 10 * a suh_d of 1.5) in a row whose norm is about 80 sqrt(inter / 2) (half the gates are
    # negative); nine of them add up to three
    bound = 3 * 2.0 ** -8 * 150 / (80 * (inter / 2) ** 0.5)
    assert_rows_close(fx.output[:rows].cpu().numpy(), window_reference(oracle, w, x, picks_np).reshape(rows, hidden),
                      rel_rms=bound, what=f"{form} K={bits} {hidden}x{inter}")


@pytest.mark.parametrize("bits", [3, 4])
def test_split_windows_do_not_depend_on_the_window(gfr, bits):
    """Windows of up to 2048 pairs at a shape with the split-K programs run those, however many rows an expert has and
    however many programs: a pair's output is the same bytes in a window of 256 rows (2048 pairs, 17 rows an expert) and
    of 100 rows (6 an expert) as in one of 9 rows."""
    import synth
    E, hidden, inter, slots, rows = 120, 2048, 1536, 8, 256
    w = synth.experts(E, hidden, inter, bits, seed=700 + bits)
    x = synth.activations(rows, hidden, 701)
    rng = np.random.default_rng(bits)
    picks = torch.from_numpy(np.stack([rng.permutation(E)[:slots] for _ in range(rows)]).astype(np.int32)).cuda()
    g = gfr.Grouping(E, slots, rows)
    fx = gfr.FastExperts(hidden, inter, slots, slots, E, rows)

    def window(r0, n):
        p = picks[r0:r0 + n].contiguous()
        g.run(p, n)
        fx.run(w, x[r0:r0 + n].contiguous(), p, g.ids, g.count, g.members, n, rows, shared_x=False)
        return fx.output[:n * slots].view(n, slots, hidden).clone()

    small = torch.cat([window(r, min(9, rows - r)) for r in range(0, rows, 9)])
    for n in (100, 256):
        got = window(0, n)
        assert torch.isfinite(got).all()
        diff = (got != small[:n]).any(dim=2).any(dim=1).sum().item()
        assert diff == 0, f"{diff} of {n} rows differ between a window of {n} rows and windows of 9"


@pytest.mark.parametrize("bits", [2, 3, 4, 5])
@pytest.mark.parametrize("hidden,inter,topk", [(2048, 1536, 4), (2560, 768, 7), (5120, 1536, 8)])
def test_moe_small_windows_on_the_default_engine(gfr, oracle, hidden, inter, topk, bits):
    """The default border is 4 rows at every width and bit width: windows of 1 to 4 rows run the decode engine (the
    prefill engine's rotated rows, a probe, stay untouched), and the windows of 2 to 4 give every token the same bytes as a
    window of two of it; 5 rows run the prefill engine. A layer of at most 4 rows has no prefill engine to leave rows for."""
    import synth
    E = topk + 2
    w = synth.experts(E + 1, hidden, inter, bits, seed=800 + topk)
    m = gfr.Moe(hidden, inter, E, topk, 5)
    for rows in range(1, 6):
        x, lg = synth.activations(rows, hidden, 810 + rows), synth.zipf_logits(rows, E, topk, 1.1, 820 + rows)
        pairs = []
        for r in range(rows):
            m.run(w, x[[r, r]].contiguous(), lg[[r, r]].contiguous(), 2)
            pairs.append(m.output[:1].clone())
        for mat in (0, 1):
            m.rotated(mat, 5).zero_()
        m.run(w, x, lg, rows)
        torch.cuda.synchronize()
        got = m.output[:rows].clone()
        prefill = bool((m.rotated(0, 5) != 0).any())
        assert prefill == (rows == 5), rows
        if 1 < rows < 5:
            assert torch.equal(got, torch.cat(pairs)), rows
        p, wt = oracle.route(lg.cpu().numpy(), topk, E)
        y = window_reference(oracle, w, x, p)
        want = np.einsum("rs,rsd->rd", wt.astype(np.float64), y.astype(np.float64))
        # the decode engine multiplies unrounded codebook sums (within 1e-2 of the reference's fp16 weights)
        assert_rows_close(got.cpu().numpy(), want, rel_rms=2e-3 if prefill else 1e-2, what=f"{rows} rows")
    small = gfr.Moe(hidden, inter, E, topk, 3)
    small.set_decode_rows(3)
    with pytest.raises(gfr.GfrError, match="lacks"):
        small.set_decode_rows(2)
