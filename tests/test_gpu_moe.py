"""MoE expert path through the C ABI against the oracle (reference dispatch order)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel_err(y, ref):
    return float(np.abs(y.astype(np.float64) - ref).max() / np.abs(ref).max())


def test_route_matches_reference_softmax_topk(O, tfq, gpu):
    import torch
    T, E, K = 16, 8, 2
    logits = O.rng_normal(45, T * E, 1.0).reshape(T, E)
    probs, idx, w = O.softmax_topk(logits, K)
    p_d, i_d, w_d = tfq.moe_route(torch.from_numpy(logits).to(gpu), K)
    assert np.array_equal(i_d.cpu().numpy().astype(np.int64), idx)
    assert np.abs(p_d.cpu().numpy() - probs).max() <= 2e-7
    assert np.abs(w_d.cpu().numpy() - w).max() <= 2e-7
    # closed form: rows sum to one, weights are the k largest probabilities, not renormalised
    pn = p_d.cpu().numpy()
    assert np.abs(pn.sum(axis=1) - 1).max() < 1e-6
    assert np.allclose(np.sort(pn, axis=1)[:, ::-1][:, :K], w_d.cpu().numpy(), atol=0, rtol=0)
    # k is clamped into 1..E like the reference does
    assert tfq.moe_route(torch.from_numpy(logits).to(gpu), 99)[1].shape == (T, E)


@pytest.mark.parametrize("T,E,K", [(1, 3, 2), (5, 64, 6), (16, 130, 8), (3, 257, 8), (7, 1024, 4), (2, 1100, 3)])
def test_route_many_experts_and_ties(O, tfq, gpu, T, E, K):
    """Expert counts around the wavefront width and the limit of the one-wavefront-per-token kernel (1100 experts take
    the one-lane form), against the oracle; and logits with exact duplicates: equal probabilities are picked in
    ascending expert order, the k picks of a token are distinct, and the weights are the picked probabilities."""
    import torch
    logits = O.rng_normal(70 + E, T * E, 1.0).reshape(T, E)
    probs, idx, w = O.softmax_topk(logits, K)
    p_d, i_d, w_d = tfq.moe_route(torch.from_numpy(logits).to(gpu), K)
    assert np.array_equal(i_d.cpu().numpy().astype(np.int64), idx)
    assert np.abs(p_d.cpu().numpy() - probs).max() <= 2e-7
    assert np.abs(w_d.cpu().numpy() - w).max() <= 2e-7
    tied = logits.copy()
    tied[:, 1::2] = tied[:, 0::2][:, :tied[:, 1::2].shape[1]]  # every odd expert repeats the even one before it
    probs, idx, w = O.softmax_topk(tied, K)
    p_d, i_d, w_d = tfq.moe_route(torch.from_numpy(tied).to(gpu), K)
    i_n, p_n, w_n = i_d.cpu().numpy().astype(np.int64), p_d.cpu().numpy(), w_d.cpu().numpy()
    assert np.array_equal(i_n, idx)
    for t in range(T):
        assert len(set(i_n[t].tolist())) == K
        assert np.array_equal(p_n[t, i_n[t]], w_n[t])
        order = sorted(range(E), key=lambda e: (-p_n[t, e], e))[:K]
        assert order == i_n[t].tolist()


@pytest.mark.parametrize("xdt", ["f32", "bf16"])
def test_router_linear_then_route(O, tfq, gpu, xdt):
    """tfq_moe_router: logits = x . Wr^T + b (float64 numpy as the check, 1e-5 of the largest logit), then the
    route of those very logits equals the oracle's softmax_topk of them."""
    import torch
    T, D, E, K = 16, 4096, 8, 2
    x = O.rng_normal(43, T * D, 1.0).reshape(T, D)
    if xdt == "bf16":
        x = O.bf16_round(x)
    Wr = O.rng_normal(46, E * D, 0.05).reshape(E, D)
    b = O.rng_normal(47, E, 0.1)
    xd = torch.from_numpy(x).to(gpu)
    if xdt == "bf16":
        xd = xd.bfloat16()
    logits, probs, idx, w = tfq.moe_router(xd, torch.from_numpy(Wr).to(gpu), K, bias=torch.from_numpy(b).to(gpu))
    ref = x.astype(np.float64) @ Wr.astype(np.float64).T + b
    got = logits.cpu().numpy()
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
    p_ref, i_ref, w_ref = O.softmax_topk(got, K)
    assert np.array_equal(idx.cpu().numpy().astype(np.int64), i_ref)
    assert np.abs(probs.cpu().numpy() - p_ref).max() <= 2e-7
    assert np.abs(w.cpu().numpy() - w_ref).max() <= 2e-7


@pytest.mark.parametrize("T,D,E,K,bias", [(1, 64, 1, 1, False), (3, 1023, 3, 2, True), (17, 1024, 16, 4, False), (5, 4097, 17, 8, True),
                                          (2, 2112, 130, 6, False), (2, 256, 1100, 3, True)])
def test_router_in_one_launch(O, tfq, gpu, T, D, E, K, bias):
    """The router Linear and the route of its logits over the edges of both its forms (one and two launches, D off the
    steps of 1024, more experts than a wavefront routes): logits against float64, and the route equal to tfq_moe_route's of those
    very logits."""
    import torch
    x = torch.from_numpy(O.rng_normal(48, T * D, 1.0).reshape(T, D)).to(gpu)
    Wr = torch.from_numpy(O.rng_normal(49, E * D, 0.05).reshape(E, D)).to(gpu)
    b = torch.from_numpy(O.rng_normal(50, E, 0.1)).to(gpu) if bias else None
    for xd in (x, x.bfloat16()):
        logits, probs, idx, w = tfq.moe_router(xd, Wr, K, bias=b)
        ref = xd.double() @ Wr.double().T + (b.double() if bias else 0.0)
        assert float((logits.double() - ref).abs().max()) <= 1e-5 * float(ref.abs().max())
        p2, i2, w2 = tfq.moe_route(logits, K)
        assert torch.equal(probs, p2) and torch.equal(idx, i2) and torch.equal(w, w2)


@pytest.mark.parametrize("E,T", [(12, 1), (13, 153), (13, 154), (24, 175), (24, 176), (64, 255), (64, 256), (65, 258)])
def test_router_one_launch_or_two(tfq, gpu, E, T):
    """Few experts, or many tokens, take the one-launch kernel and everything else two launches: on both sides of the line a
    token's logits and route are, bit for bit, those of a call with that token alone (two launches from thirteen experts on),
    and the route is tfq_moe_route's of the logits."""
    import torch
    D, K = 1088, 3
    gen = torch.Generator().manual_seed(E * 1000 + T)
    x = torch.randn(T, D, generator=gen).to(gpu)
    Wr = (torch.randn(E, D, generator=gen) * 0.05).to(gpu)
    got = tfq.moe_router(x, Wr, K)
    ref = x.double() @ Wr.double().T
    assert float((got[0].double() - ref).abs().max()) <= 1e-5 * float(ref.abs().max())
    assert all(torch.equal(a, b) for a, b in zip(got[1:], tfq.moe_route(got[0], K)))
    for t in (0, T // 2, T - 1):
        alone = tfq.moe_router(x[t:t + 1].contiguous(), Wr, K)
        assert all(torch.equal(a[t:t + 1], b) for a, b in zip(got, alone))


@pytest.mark.parametrize("E", [1, 2, 4, 5, 7, 8, 9])
def test_router_of_few_experts_ties(tfq, gpu, E):
    """Up to eight experts meet over eight lanes, one more over all: every k up to E, rows of the router repeated so that logits and
    probabilities tie exactly, all of them in one token.  Probabilities, picks and weights are, bit for bit, tfq_moe_route's
    of the logits (which has the general form), and the picks are in order, the lower index first among equals."""
    import torch
    T, D = 37, 1088
    gen = torch.Generator().manual_seed(E)
    x = torch.randn(T, D, generator=gen).to(gpu)
    x[3] = 0.0
    Wr = (torch.randn(E, D, generator=gen) * 0.05).to(gpu)
    Wr[1::2] = Wr[0::2][:E // 2]
    for k in range(1, E + 1):
        logits, probs, idx, w = tfq.moe_router(x, Wr, k)
        assert torch.equal(logits[:, 1::2], logits[:, 0::2][:, :E // 2])
        for a, b in zip((probs, idx, w), tfq.moe_route(logits, k)):
            assert torch.equal(a, b), k
        order = [sorted(range(E), key=lambda e: (-p[e], e))[:k] for p in probs.cpu().tolist()]
        assert idx.cpu().tolist() == order


def _experts(O, tfq, fmt, E, D, F, seed):
    gate, up, down, hg, hu, hd = [], [], [], [], [], []
    for e in range(E):
        for lst, hst, n, k, off in ((gate, hg, F, D, 0), (up, hu, F, D, 1), (down, hd, D, F, 2)):
            pay = O.encode_tensor(fmt, O.rng_normal(seed + 10 * e + off, n * k, 0.02))
            hst.append(pay)
            lst.append(tfq.Weight(fmt, n, k, pay))
    return gate, up, down, hg, hu, hd


@pytest.mark.parametrize("fmt", ["Q_G_4", "B32S4"])
@pytest.mark.parametrize("xdt,mid_bf16,tol", [("bf16", True, 1e-2), ("f32", False, 1e-3)])
def test_moe_ffn_small(O, tfq, gpu, fmt, xdt, mid_bf16, tol):
    """8 experts, top-2, 16 tokens: the Mixtral-style configuration at reduced width."""
    import torch
    E, Ktop, T, D, F = 8, 2, 16, 512, 1024
    gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, E, D, F, 300)
    logits = O.rng_normal(45, T * E, 1.0).reshape(T, E)
    _, idx, w = O.softmax_topk(logits, Ktop)
    x = O.rng_normal(43, T * D, 1.0).reshape(T, D)
    if xdt == "bf16":
        x = O.bf16_round(x)
        xt = torch.from_numpy(x).to(gpu).bfloat16()
    else:
        xt = torch.from_numpy(x).to(gpu)
    ref = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=mid_bf16)
    y = tfq.moe_ffn(gate, up, down, idx, w, xt, mid_dtype=torch.bfloat16 if mid_bf16 else torch.float32).cpu().numpy()
    assert rel_err(y, ref) <= tol
    # invariants: every (token, slot) pair is dispatched once; weights in (0, 1]
    assert sum((idx == e).sum() for e in range(E)) == T * Ktop and np.all((w > 0) & (w <= 1))
    # an expert nobody routes to, a dropped (non-positive) weight and an out-of-range id are skipped
    idx2, w2 = idx.copy(), w.copy()
    idx2[idx2 == 3] = 5
    w2[0, 0] = 0.0
    idx2[1, 1] = 99
    for t in range(T):  # keep the two slots of a token distinct
        if idx2[t, 0] == idx2[t, 1]:
            idx2[t, 1] = (idx2[t, 0] + 1) % E if (idx2[t, 0] + 1) % E != 3 else (idx2[t, 0] + 2) % E
    ref2 = O.moe_ffn(fmt, hg, hu, hd, D, F, idx2, w2, x, mid_bf16=mid_bf16)
    y2 = tfq.moe_ffn(gate, up, down, idx2, w2, xt, mid_dtype=torch.bfloat16 if mid_bf16 else torch.float32).cpu().numpy()
    assert rel_err(y2, ref2) <= tol
    yb = tfq.moe_ffn(gate, up, down, idx, w, xt, out_dtype=torch.bfloat16,
                     mid_dtype=torch.bfloat16 if mid_bf16 else torch.float32).float().cpu().numpy()
    assert rel_err(yb, ref) <= 1e-2
    for wl in gate + up + down:
        wl.close()


@pytest.mark.parametrize("fmt", ["B32S4", "Q_G_8", "Q_G_3"])
def test_moe_ffn_skewed_routing(O, tfq, gpu, fmt):
    """One expert takes most tokens (more rows than one pass of the GEMV carries, so its rows are cut into
    chunks), some experts take none; formats with the grouped launch and one without it."""
    import torch
    E, Ktop, T, D, F = 6, 2, 24, 512, 1024
    gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, E, D, F, 700)
    logits = O.rng_normal(46, T * E, 1.0).reshape(T, E)
    logits[:, 2] += 6.0      # every token picks expert 2 first
    logits[:, 4] -= 20.0     # nobody picks expert 4
    _, idx, w = O.softmax_topk(logits, Ktop)
    assert (idx == 2).sum() == T and (idx == 4).sum() == 0
    x = O.bf16_round(O.rng_normal(43, T * D, 1.0).reshape(T, D))
    ref = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=True)
    y = tfq.moe_ffn(gate, up, down, idx, w, torch.from_numpy(x).to(gpu).bfloat16(), mid_dtype=torch.bfloat16).cpu().numpy()
    assert rel_err(y, ref) <= 1e-2
    ref32 = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=False)
    y32 = tfq.moe_ffn(gate, up, down, idx, w, torch.from_numpy(x).to(gpu), mid_dtype=torch.float32).cpu().numpy()
    assert rel_err(y32, ref32) <= 1e-3
    for wl in gate + up + down:
        wl.close()


@pytest.mark.parametrize("fmt,xdt,mid_bf16,tol", [("B32S4", "bf16", True, 1e-2), ("Q_G_8", "bf16", True, 1e-2),
                                                  ("Q_G_4", "f32", False, 1e-3)])
def test_moe_ffn_many_tokens_per_expert(O, tfq, gpu, fmt, xdt, mid_bf16, tol):
    """A prefill-sized call: 200 tokens over 4 experts, top-2, so every expert holds far more than 16 rows and
    the expert products go through the prefill entry (the matrix-core GEMM for bf16 rows)."""
    import torch
    E, Ktop, T, D, F = 4, 2, 200, 256, 512
    gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, E, D, F, 700)
    logits = O.rng_normal(46, T * E, 1.0).reshape(T, E)
    _, idx, w = O.softmax_topk(logits, Ktop)
    assert min((idx == e).sum() for e in range(E)) > 32
    x = O.rng_normal(47, T * D, 1.0).reshape(T, D)
    if xdt == "bf16":
        x = O.bf16_round(x)
        xt = torch.from_numpy(x).to(gpu).bfloat16()
    else:
        xt = torch.from_numpy(x).to(gpu)
    ref = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=mid_bf16)
    y = tfq.moe_ffn(gate, up, down, idx, w, xt, mid_dtype=torch.bfloat16 if mid_bf16 else torch.float32).cpu().numpy()
    assert rel_err(y, ref) <= tol
    for W in gate + up + down:
        W.close()


@pytest.mark.parametrize("fmt", ["B32S4", "Q_G_8", "Q_G_3"])
def test_moe_ffn_prefill_sized_with_uneven_experts(O, tfq, gpu, fmt):
    """A prefill-sized call (bf16 rows and mid activations: the experts' products are grouped launches of the
    matrix-core tile kernel) in which one expert holds hundreds of rows (two token tiles), others a few dozen, one
    a handful and one none."""
    import torch
    E, Ktop, T, D, F = 6, 2, 300, 256, 512
    gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, E, D, F, 1300)
    logits = O.rng_normal(54, T * E, 1.0).reshape(T, E)
    logits[:, 1] += 6.0      # every token picks expert 1 first: 300 rows
    logits[:, 4] -= 20.0     # nobody picks expert 4
    logits[:, 5] -= 3.5      # a handful pick expert 5
    _, idx, w = O.softmax_topk(logits, Ktop)
    counts = [int((idx == e).sum()) for e in range(E)]
    assert counts[1] == T and counts[4] == 0 and 0 < counts[5] <= 16, counts
    x = O.bf16_round(O.rng_normal(55, T * D, 1.0).reshape(T, D))
    ref = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=True)
    y = tfq.moe_ffn(gate, up, down, idx, w, torch.from_numpy(x).to(gpu).bfloat16(), mid_dtype=torch.bfloat16).cpu().numpy()
    assert rel_err(y, ref) <= 1e-2
    for W in gate + up + down:
        W.close()


@pytest.mark.parametrize("fmt", ["B32S4", "B32S8"])
def test_moe_ffn_long_down_rows_five_to_sixteen(O, tfq, gpu, fmt):
    """Experts with five to sixteen tokens and a down product too long for their staged rows (K = 5120: twenty
    block columns, so some wavefronts of the sixteen-row kernel own two): bf16 mid activations take the grouped
    sixteen-row launch, which reads every down matrix once; fp32 mid activations keep the two-row passes."""
    import torch
    E, Ktop, T, D, F = 4, 2, 18, 256, 5120
    gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, E, D, F, 900)
    logits = O.rng_normal(48, T * E, 1.0).reshape(T, E)
    logits[:, 3] -= 20.0  # three experts share the tokens: twelve each
    _, idx, w = O.softmax_topk(logits, Ktop)
    counts = [int((idx == e).sum()) for e in range(E)]
    assert counts[3] == 0 and min(counts[:3]) > 4 and max(counts) <= 16, counts
    x = O.bf16_round(O.rng_normal(49, T * D, 1.0).reshape(T, D))
    ref = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=True)
    y = tfq.moe_ffn(gate, up, down, idx, w, torch.from_numpy(x).to(gpu).bfloat16(), mid_dtype=torch.bfloat16).cpu().numpy()
    assert rel_err(y, ref) <= 1e-2
    ref32 = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=False)
    y32 = tfq.moe_ffn(gate, up, down, idx, w, torch.from_numpy(x).to(gpu).bfloat16(), mid_dtype=torch.float32).cpu().numpy()
    assert rel_err(y32, ref32) <= 1e-3
    for wl in gate + up + down:
        wl.close()


@pytest.mark.parametrize("fmt,D,F,T", [("B32S4", 256, 6144, 20), ("B32S4", 768, 6400, 20), ("Q_G_4", 512, 6144, 20),
                                       ("B32S8", 256, 6144, 20), ("Q_G_8", 512, 6144, 20), ("B32S4", 512, 6144, 24),
                                       ("B32S4", 256, 6144, 40)])
def test_moe_ffn_tall_gate_up_with_five_to_eight_rows(O, tfq, gpu, fmt, D, F, T):
    """Gate / up matrices with thousands of rows and experts of five to eight tokens: enough tiles for the grouped
    launch whose wavefronts own whole tiles (a workgroup per compute unit, twelve tile pairs or more each), at one,
    two and three block columns.  Host-side and device-side routing, against the oracle.  With 24 and 40 tokens
    some experts hold nine to seventeen rows: their rows go in chunks of eight (9 and 13 problems), and the
    wavefronts take more tile pairs each so that the workgroups still fit one round."""
    import torch
    E, Ktop = 8, 2
    gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, E, D, F, 1100)
    logits = O.rng_normal(52, T * E, 1.0).reshape(T, E)
    _, idx, w = O.softmax_topk(logits, Ktop)
    counts = [int((idx == e).sum()) for e in range(E)]
    assert 4 < max(counts) and (T > 20 or max(counts) <= 8), counts
    x = O.bf16_round(O.rng_normal(53, T * D, 1.0).reshape(T, D))
    ref = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=True)
    xt = torch.from_numpy(x).to(gpu).bfloat16()
    y = tfq.moe_ffn(gate, up, down, idx, w, xt, mid_dtype=torch.bfloat16)
    assert rel_err(y.cpu().numpy(), ref) <= 1e-2
    routed = tfq.RoutedMoe(gate, up, down, T, Ktop)
    yr = torch.empty(T, D, device=gpu)
    routed(torch.from_numpy(idx.astype(np.int32)).to(gpu), torch.from_numpy(w.astype(np.float32)).to(gpu), xt, yr)
    assert rel_err(yr.cpu().numpy(), ref) <= 1e-2
    assert float((yr - y).abs().max()) <= 1e-5 * float(y.abs().max())
    for wl in gate + up + down:
        wl.close()


@pytest.mark.parametrize("fmt", ["B32S4", "Q_G_8"])
def test_moe_ffn_routed_builds_its_lists_on_the_device(O, tfq, gpu, fmt):
    """tfq_moe_ffn_routed: routing arrays stay on the device, lists and launch tables are built there.  Skewed
    routing (an expert with more rows than one pass, an expert with none, a slot whose id is out of range) against
    the oracle and against tfq_moe_ffn with the same routing on the host."""
    import torch
    E, Ktop, T, D, F = 6, 2, 24, 512, 1024
    gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, E, D, F, 800)
    logits = O.rng_normal(50, T * E, 1.0).reshape(T, E)
    logits[:, 2] += 6.0      # every token picks expert 2 first: 24 rows, three passes of eight
    logits[:, 4] -= 20.0     # nobody picks expert 4
    _, idx, w = O.softmax_topk(logits, Ktop)
    idx = idx.copy()
    idx[5, 1] = E + 3        # an id outside 0..E-1: the slot is skipped
    x = O.bf16_round(O.rng_normal(51, T * D, 1.0).reshape(T, D))
    ref = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=True)
    xt = torch.from_numpy(x).to(gpu).bfloat16()
    host = tfq.moe_ffn(gate, up, down, idx, w, xt, mid_dtype=torch.bfloat16)
    routed = tfq.RoutedMoe(gate, up, down, T, Ktop)
    y = torch.empty(T, D, device=gpu)
    routed(torch.from_numpy(idx.astype(np.int32)).to(gpu), torch.from_numpy(w.astype(np.float32)).to(gpu), xt, y)
    assert rel_err(y.cpu().numpy(), ref) <= 1e-2
    assert float((y - host).abs().max()) <= 1e-5 * float(host.abs().max())
    for wl in gate + up + down:
        wl.close()


@pytest.mark.parametrize("fmt,D,F", [("B32S4", 512, 1024), ("Q_G_4", 256, 768), ("B32S8", 256, 512), ("Q_G_8", 512, 512), ("B32S4", 4096, 14336)])
def test_moe_ffn_routed_single_token(O, tfq, gpu, fmt, D, F):
    """One token, top-2: the routed call is two launches that look the slots' experts up themselves and add the
    weighted down products into y with atomics.  Against the oracle (the small shapes), against the host-list
    call bit for bit, and with the irregular slots: an id outside 0..E-1, a weight that is not positive, both
    slots naming one expert, no slot with an expert at all (y = 0); ten calls in a row give the same bits."""
    import torch
    E, Ktop, T = 8, 2, 1
    small = D * F <= 1 << 20
    if small:
        gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, E, D, F, 1500)
    else:
        gen = torch.Generator(device="cuda").manual_seed(3)
        gate, up, down = [], [], []
        for e in range(E):
            for lst, n, k in ((gate, F, D), (up, F, D), (down, D, F)):
                lst.append(tfq.Weight(fmt, n, k, tfq.encode(fmt, torch.randn(n * k, device=gpu, generator=gen) * 0.02)))
    x = O.bf16_round(O.rng_normal(57, T * D, 1.0).reshape(T, D))
    xt = torch.from_numpy(x).to(gpu).bfloat16()
    routed = tfq.RoutedMoe(gate, up, down, T, Ktop)
    cases = [([3, 6], [0.7, 0.3]), ([5, 0], [0.25, 0.75]), ([2, E + 1], [0.6, 0.4]), ([-1, 4], [0.5, 0.5]),
             ([1, 7], [0.0, 1.0]), ([4, 4], [0.6, 0.4]), ([-1, E + 2], [0.5, 0.5])]
    for ids, wts in cases:
        idx = np.array([ids], np.int64)
        w = np.array([wts], np.float32)
        host = tfq.moe_ffn(gate, up, down, idx, w, xt, mid_dtype=torch.bfloat16)
        y = torch.full((T, D), 7.0, device=gpu)
        di, dw = torch.from_numpy(idx.astype(np.int32)).to(gpu), torch.from_numpy(w).to(gpu)
        routed(di, dw, xt, y)
        assert torch.equal(y, host), (ids, wts, float((y - host).abs().max()))
        if not any(0 <= i < E for i in ids):
            assert float(y.abs().max()) == 0.0
        if small and ids[0] != ids[1] and any(0 <= i < E for i in ids):
            ref = O.moe_ffn(fmt, hg, hu, hd, D, F, idx, w, x, mid_bf16=True)
            assert rel_err(y.cpu().numpy(), ref) <= 1e-2
        for _ in range(10):
            y2 = torch.full((T, D), -3.0, device=gpu)
            routed(di, dw, xt, y2)
            assert torch.equal(y2, y)
    for wl in gate + up + down:
        wl.close()


@pytest.mark.parametrize("Ktop", [1, 2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("D", [256, 768])
def test_moe_ffn_combine(tfq, gpu, Ktop, D):
    """The step that adds a token's pairs, in batches of four and two with a rest, tokens without a pair or with one among them.
    Against the sum of one-pair mixtures of the same rows in float64: fp32 sums of
    up to nine rows (their products may come from other kernels: 1e-5, as in test_moe_ffn_routed_shapes), bf16 by one rounding more."""
    import torch
    E, F, T = 12, 256, 9
    g = torch.Generator(device="cuda").manual_seed(41)
    mat = lambda n, k: tfq.Weight("B32S4", n, k, tfq.encode("B32S4", torch.randn(n * k, device=gpu, generator=g) * 0.05))
    ws = [[mat(F, D) for _ in range(E)], [mat(F, D) for _ in range(E)], [mat(D, F) for _ in range(E)]]
    x = torch.randn(T, D, device=gpu, generator=g)
    rng = np.random.default_rng(42)
    idx = np.stack([rng.permutation(E)[:Ktop] for _ in range(T)]).astype(np.int64)
    w = rng.uniform(0.1, 1.0, (T, Ktop)).astype(np.float32)
    w[1, :] = 0.0
    w[2, 1:] = 0.0
    w[3, :-1] = 0.0
    want = torch.zeros(T, D, dtype=torch.float64, device=gpu)
    for j in range(Ktop):
        want += tfq.moe_ffn(*ws, idx[:, j:j + 1].copy(), w[:, j:j + 1].copy(), x, mid_dtype=torch.float32).double()
    top = float(want.abs().max())
    y = tfq.moe_ffn(*ws, idx, w, x, mid_dtype=torch.float32)
    yb = tfq.moe_ffn(*ws, idx, w, x, mid_dtype=torch.float32, out_dtype=torch.bfloat16)
    assert float((y.double() - want).abs().max()) <= 1e-5 * top
    assert torch.equal(yb, y.bfloat16())
    assert not y[1].any() and not yb[1].any()
    for wl in sum(ws, []):
        wl.close()


@pytest.mark.parametrize("T,Ktop,E", [(1, 1, 3), (7, 3, 5), (64, 2, 4), (128, 8, 16), (5, 2, 40)])
def test_moe_ffn_routed_shapes(O, tfq, gpu, T, Ktop, E):
    """Call shapes of the routed form: one pair, odd counts, experts with several passes of eight and sixteen
    rows, the largest call it takes (1024 pairs), more experts than pairs.  Against tfq_moe_ffn with the same
    routing read back to the host (which cuts the rows into passes by its own rules: equal to rounding, or to the
    bf16 tolerance where it takes the prefill GEMM)."""
    import torch
    fmt, D, F = "B32S4", 256, 512
    gate, up, down, _, _, _ = _experts(O, tfq, fmt, E, D, F, 840)
    logits = torch.from_numpy(O.rng_normal(53, T * E, 1.0).reshape(T, E)).to(gpu)
    _, idx, w = tfq.moe_route(logits, Ktop)
    xt = torch.from_numpy(O.rng_normal(54, T * D, 1.0).reshape(T, D)).to(gpu).bfloat16()
    host = tfq.moe_ffn(gate, up, down, idx.cpu().numpy().astype(np.int64), w.cpu().numpy(), xt, mid_dtype=torch.bfloat16)
    y = torch.empty(T, D, device=gpu)
    tfq.RoutedMoe(gate, up, down, T, Ktop)(idx, w, xt, y)
    # with more than 32 rows on an expert the host-list call multiplies through the prefill GEMM, whose weights are
    # rounded to bf16; the routed call always takes the decode kernels
    counts = [int((idx == e).sum()) for e in range(E)]
    tol = 1e-2 if max(counts) > 32 else 1e-5
    assert float((y - host).abs().max()) <= tol * float(host.abs().max())
    for wl in gate + up + down:
        wl.close()


@pytest.mark.parametrize("T,Ktop,E", [(1, 3, 2), (21, 3, 64), (13, 5, 65), (128, 8, 200), (256, 4, 256)])
def test_moe_ffn_routed_lists(tfq, gpu, T, Ktop, E):
    """The lists of a routed call: slots of one wavefront and of all sixteen, as many experts as lanes, one more, and the most that
    are taken; ids out of range, an expert with most of the tokens.  Against tfq_moe_ffn with the same routing (its rows are cut
    into passes by other rules: 1e-5 as in test_moe_ffn_routed_shapes, 1e-2 where it takes the prefill GEMM)."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(43)
    D = F = 256
    print(f"routed lists T={T} k={Ktop} E={E}", flush=True)
    mat = lambda: tfq.Weight("B32S4", D, F, tfq.encode("B32S4", torch.randn(D * F, device=gpu, generator=g) * 0.05))
    gate, up, down = ([mat() for _ in range(E)] for _ in range(3))
    rng = np.random.default_rng(44)
    idx = np.stack([rng.permutation(E + 2)[:Ktop] - 1 for _ in range(T)]).astype(np.int64)  # (-1 and E: no expert)
    for t in range(0, T, 3):
        if not (idx[t] == E - 1).any():
            idx[t, 0] = E - 1
    w = rng.uniform(0.1, 1.0, (T, Ktop)).astype(np.float32)
    x = torch.randn(T, D, device=gpu, generator=g).bfloat16()
    host = tfq.moe_ffn(gate, up, down, idx, w, x, mid_dtype=torch.bfloat16)
    y = torch.empty(T, D, device=gpu)
    call = tfq.RoutedMoe(gate, up, down, T, Ktop)
    call(torch.from_numpy(idx.astype(np.int32)).to(gpu), torch.from_numpy(w).to(gpu), x, y)
    tol = 1e-2 if max(int((idx == e).sum()) for e in range(E)) > 32 else 1e-5
    assert float((y - host).abs().max()) <= tol * float(host.abs().max())
    for wl in gate + up + down:
        wl.close()


@pytest.mark.parametrize("E,T,busy,exact", [(16, 512, 0, True), (16, 512, 512, True), (16, 1280, 0, False), (16, 1280, 900, False), (4, 256, 0, True)])
def test_moe_ffn_rows_of_each_expert_choose_the_kernel(tfq, gpu, E, T, busy, exact):
    """Prefill-sized calls with the lists on the host, `busy` tokens on expert 0 and the rest spread: up to 1024 pairs go through
    the integer tile kernel, which does not round weights, however they are spread; 160 rows an expert on average through the
    bf16 tile kernel, whose rounded weights show as 1e-3 of the output's norm.  Against float64 with the mid activations in bf16."""
    import torch
    D, F = 1024, 2816
    gen = torch.Generator().manual_seed(E + T + busy)
    ws, dense = [], []
    for n, k in ((F, D), (F, D), (D, F)):
        pays = [tfq.encode("B32S4", torch.randn(n * k, generator=gen).to(gpu) * 0.03) for _ in range(E)]
        ws.append([tfq.Weight("B32S4", n, k, p) for p in pays])
        dense.append([tfq.decode("B32S4", p, n * k).reshape(n, k).double() for p in pays])
    idx = torch.stack([torch.randperm(E, generator=gen)[:2] for _ in range(T)])
    for t in range(busy):
        idx[t] = torch.tensor([0, 1 + t % (E - 1)])
    w = torch.rand(T, 2, generator=gen) * 0.5 + 0.25
    x = torch.randn(T, D, generator=gen).to(gpu).bfloat16()
    want = torch.zeros(T, D, dtype=torch.float64, device=gpu)
    for e in range(E):
        t, j = (idx == e).nonzero(as_tuple=True)
        if len(t) == 0:
            continue
        xe = x[t.to(gpu)].double()
        mid = (torch.nn.functional.silu(xe @ dense[0][e].T) * (xe @ dense[1][e].T)).float().bfloat16().double()
        want.index_add_(0, t.to(gpu), (mid @ dense[2][e].T) * w[t, j].to(gpu).double()[:, None])
    y = tfq.moe_ffn(*ws, idx.numpy(), w.numpy(), x, mid_dtype=torch.bfloat16).double()
    err = float((y - want).norm() / want.norm())
    assert err <= 1e-2
    assert (err <= 3e-4) == exact, err
    for wl in ws:
        for W in wl:
            W.close()


def test_moe_ffn_routed_refuses_what_it_does_not_serve(O, tfq, gpu):
    """More than 1024 pairs, or a format without the grouped kernels: no workspace size, and the call fails."""
    gate, up, down, _, _, _ = _experts(O, tfq, "B32S4", 2, 256, 512, 860)
    with pytest.raises(tfq.TfqError):
        tfq.RoutedMoe(gate, up, down, 600, 2)
    g3, u3, d3, _, _, _ = _experts(O, tfq, "Q_G_3", 2, 256, 512, 870)
    with pytest.raises(tfq.TfqError):
        tfq.RoutedMoe(g3, u3, d3, 4, 2)
    for wl in gate + up + down + g3 + u3 + d3:
        wl.close()


def test_moe_ffn_routed_in_a_graph(O, tfq, gpu):
    """The routed call captured into a graph together with the router: replays with other activations (hence other
    routing) equal the eager calls bit for bit, with eager work and synchronizations between the replays."""
    import torch
    fmt, E, Ktop, T, D, F = "B32S4", 8, 2, 16, 512, 1536
    gate, up, down, _, _, _ = _experts(O, tfq, fmt, E, D, F, 820)
    Wr = torch.from_numpy(O.rng_normal(52, E * D, 0.05).reshape(E, D).astype(np.float32)).to(gpu)
    routed = tfq.RoutedMoe(gate, up, down, T, Ktop)
    xs = [torch.from_numpy(O.rng_normal(60 + i, T * D, 1.0).reshape(T, D).astype(np.float32)).to(gpu).bfloat16() for i in range(4)]
    x = xs[0].clone()
    y = torch.zeros(T, D, device=gpu)

    def step():
        _, _, idx, wts = tfq.moe_router(x, Wr, Ktop)
        routed(idx, wts, x, y)
        return idx

    step()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    seen = set()
    for i in (1, 2, 3, 0, 2):
        x.copy_(xs[i])
        g.replay()
        torch.cuda.synchronize()
        got = y.clone()
        y.zero_()
        idx = step()
        torch.cuda.synchronize()
        seen.add(tuple(idx.cpu().numpy().reshape(-1).tolist()))
        assert torch.equal(got, y), i
    assert len(seen) >= 3  # the replays really saw different routing
    for wl in gate + up + down:
        wl.close()


def test_moe_single_token_equals_plain_mlp(O, tfq, gpu):
    """One token, one expert, weight 1: the MoE path reduces to the SwiGLU MLP step."""
    import torch
    fmt, D, F = "B32S4", 512, 768
    gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, 1, D, F, 500)
    x = O.bf16_round(O.rng_normal(7, D, 1.0).reshape(1, D))
    xt = torch.from_numpy(x).to(gpu).bfloat16()
    y = tfq.moe_ffn(gate, up, down, np.zeros((1, 1), np.int64), np.ones((1, 1), np.float32), xt,
                    mid_dtype=torch.float32).cpu().numpy()
    g = O.matmul(fmt, hg[0], F, D, x)
    u = O.matmul(fmt, hu[0], F, D, x)
    want = O.matmul(fmt, hd[0], D, F, O.silu_mul(g, u))
    assert rel_err(y, want) <= 1e-3
    for wl in gate + up + down:
        wl.close()


def test_config5_mixtral_layer_full_size(tfq, gpu):
    """8 experts, top-2, 16 tokens, gate/up 14336x4096 and down 4096x14336, B32S4 weights from
    N(0, 0.02), bf16 activations: checked against a dense torch evaluation of the same decoded
    weights (the oracle takes minutes at this size), plus conservation under weight scaling."""
    import torch
    E, Ktop, T, D, F = 8, 2, 16, 4096, 14336
    g = torch.Generator(device="cuda").manual_seed(5)
    gate, up, down = [], [], []
    for e in range(E):
        for lst, n, k in ((gate, F, D), (up, F, D), (down, D, F)):
            w = torch.randn(n * k, device=gpu, generator=g) * 0.02
            lst.append(tfq.Weight("B32S4", n, k, tfq.encode("B32S4", w)))
            del w
    logits = torch.randn(T, E, device=gpu, generator=g)
    _, idx, wts = tfq.moe_route(logits, Ktop)
    idx_h, w_h = idx.cpu().numpy().astype(np.int64), wts.cpu().numpy()
    x = torch.randn(T, D, device=gpu, generator=g).bfloat16()
    y = tfq.moe_ffn(gate, up, down, idx_h, w_h, x, mid_dtype=torch.bfloat16)
    want = torch.zeros(T, D, device=gpu, dtype=torch.float64)
    xf = x.double()
    for e in range(E):
        toks = [t for t in range(T) if e in idx_h[t]]
        if not toks:
            continue
        Wg, Wu, Wd = gate[e].decode().double(), up[e].decode().double(), down[e].decode().double()
        xe = xf[toks]
        gg, uu = (xe @ Wg.T).float(), (xe @ Wu.T).float()
        h = (gg / (1 + torch.exp(-gg)) * uu).bfloat16().double()
        o = h @ Wd.T
        for i, t in enumerate(toks):
            want[t] += float(w_h[t][list(idx_h[t]).index(e)]) * o[i]
        del Wg, Wu, Wd
    err = float((y.double() - want).abs().max() / want.abs().max())
    assert err <= 1e-2, err
    # linear in the routing weights: doubling them doubles the output exactly (power of two)
    y2 = tfq.moe_ffn(gate, up, down, idx_h, 2 * w_h, x, mid_dtype=torch.bfloat16)
    assert torch.equal(y2, 2 * y)
    for wl in gate + up + down:
        wl.close()


@pytest.mark.parametrize("fmt", ["B32S4", "Q_G_4", "Q_G_8", "Q_G_6"])
@pytest.mark.parametrize("B,xdt,mid", [(1, "f32", "f32"), (3, "bf16", "bf16"), (16, "bf16", "bf16"), (20, "bf16", "f32")])
def test_mlp_step_matches_the_oracle(O, tfq, gpu, fmt, B, xdt, mid):
    """Dense SwiGLU feed-forward (Qwen35Engine::mlp_step): y = down(silu(gate x) * (up x)) against the oracle's
    block-row matmuls and silu step; formats with and without the multi-matrix kernel, decode and prefill row counts."""
    import torch
    D, F = 512, 768
    print(f"mlp_step {fmt} B={B} {xdt} mid={mid}", flush=True)
    pays = [O.encode_tensor(fmt, O.rng_normal(70 + i, n * k, 0.02)) for i, (n, k) in enumerate(((F, D), (F, D), (D, F)))]
    x = O.rng_normal(9, B * D, 1.0).reshape(B, D)
    if xdt == "bf16":
        x = O.bf16_round(x)
    g = O.matmul(fmt, pays[0], F, D, x)
    u = O.matmul(fmt, pays[1], F, D, x)
    h = O.silu_mul(g.reshape(-1), u.reshape(-1)).reshape(B, F)
    if mid == "bf16":
        h = O.bf16_round(h)
    want = O.matmul(fmt, pays[2], D, F, h)
    Ws = [tfq.Weight(fmt, n, k, p) for p, (n, k) in zip(pays, ((F, D), (F, D), (D, F)))]
    xt = torch.from_numpy(x).to(gpu)
    if xdt == "bf16":
        xt = xt.bfloat16()
    y = tfq.mlp_step(Ws[0], Ws[1], Ws[2], xt, mid_dtype=torch.bfloat16 if mid == "bf16" else torch.float32).cpu().numpy()
    tol = 1e-3 if xdt == "f32" and mid == "f32" else 1e-2
    assert float(np.abs(y - want).max()) <= tol * float(np.abs(want).max())
    for W in Ws:
        W.close()


@pytest.mark.parametrize("fmt", ["B32S4", "Q_G_8", "Q_G_3", "SB256A3", "Q_G_6"])
@pytest.mark.parametrize("B", [2, 3, 8, 9, 16, 17])
def test_mlp_step_fp32_rows_match_the_oracle(O, tfq, gpu, fmt, B):
    """The same with fp32 activations throughout, at the row counts where the launches change: the paired launch up to
    two, with two slot sets up to four, launches of their own for the elementwise step and down up to sixteen, the prefill
    entry above.  Three products of 16-bit activations are within
    3 x 2^-17 of a value, the companded grid's line within 7.5e-5 of its levels (on the norm; SiLU's slope is below 1.1)."""
    import torch
    D, F = 512, 768
    print(f"mlp_step {fmt} B={B} f32", flush=True)
    pays = [O.encode_tensor(fmt, O.rng_normal(70 + i, n * k, 0.02)) for i, (n, k) in enumerate(((F, D), (F, D), (D, F)))]
    x = O.rng_normal(9, B * D, 1.0).reshape(B, D)
    g = O.matmul(fmt, pays[0], F, D, x)
    u = O.matmul(fmt, pays[1], F, D, x)
    want = O.matmul(fmt, pays[2], D, F, O.silu_mul(g.reshape(-1), u.reshape(-1)).reshape(B, F)).astype(np.float64)
    Ws = [tfq.Weight(fmt, n, k, p) for p, (n, k) in zip(pays, ((F, D), (F, D), (D, F)))]
    y = tfq.mlp_step(Ws[0], Ws[1], Ws[2], torch.from_numpy(x).to(gpu)).cpu().numpy()
    assert np.linalg.norm(y - want) <= (3e-4 if fmt == "Q_G_8" else 3e-5) * np.linalg.norm(want)
    for W in Ws:
        W.close()


@pytest.mark.parametrize("fmt,counts,D,F", [
    ("B32S4", (0, 1, 31, 33, 64, 65), 512, 768),        # tiles of 64 rows, an expert without a row
    ("Q_G_8", (0, 32, 33, 1, 63, 0), 256, 1280),        # tiles of 32 rows
    ("Q_G_4", (97, 0, 0, 16), 768, 512),
    ("B32S8", tuple([0] * 3 + [17, 40] * 36 + [5]), 256, 256),  # more experts than a wavefront scans at once
])
def test_moe_ffn_grouped_tiles(O, tfq, gpu, fmt, counts, D, F):
    """Experts of some sixteen rows and more on average, top-1: one launch over the tiles of all experts, from routing arrays
    on the host and, where they are few enough, on the device: the two calls agree bit for bit, and match the float64 product
    of the decoded matrices to the bound of bf16 mid activations."""
    import ctypes as C
    import torch
    E, T = len(counts), sum(counts)
    print(f"moe groups {fmt} E={E} T={T} D={D} F={F}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(81)
    make = lambda n, k: tfq.Weight(fmt, n, k, tfq.encode(fmt, torch.randn(n * k, device=gpu, generator=g) * 0.02))
    gate, up, down = [[make(*nk) for _ in range(E)] for nk in ((F, D), (F, D), (D, F))]
    x = torch.randn(T, D, device=gpu, generator=g).bfloat16()
    idx = np.repeat(np.arange(E), counts)[np.random.RandomState(5).permutation(T)].astype(np.int32).reshape(T, 1)
    w = np.linspace(0.2, 1.0, T).astype(np.float32).reshape(T, 1)
    y = tfq.moe_ffn(gate, up, down, idx, w, x)
    want = torch.zeros(T, D, device=gpu, dtype=torch.float64)
    for e in range(E):
        rows = torch.from_numpy(np.nonzero(idx[:, 0] == e)[0]).to(gpu)
        if rows.numel() == 0:
            continue
        a, b, d = (W.decode().reshape(n, k).double() for W, (n, k) in ((gate[e], (F, D)), (up[e], (F, D)), (down[e], (D, F))))
        xe = x[rows].double()
        u = xe @ a.T
        h = (u * torch.sigmoid(u) * (xe @ b.T)).bfloat16().double()
        want[rows] = (h @ d.T) * torch.from_numpy(w).to(gpu)[rows].double()
    err = lambda v: float((v.double() - want).norm() / want.norm())
    assert err(y) <= 5e-3
    if T <= 1024:
        z = torch.full((T, D), 9.0, device=gpu)
        tfq.RoutedMoe(gate, up, down, T, 1)(torch.from_numpy(idx).to(gpu), torch.from_numpy(w).to(gpu), x, z)
        assert torch.equal(z, y)
    for W in gate + up + down:
        W.close()


@pytest.mark.parametrize("fmt,B,D,F,xdt,mid,plan", [  # plan: shape (4: 32 x 32 tiles, 1: activations split beforehand) and K parts of the pair
    ("B32S4", 9, 512, 8448, "f32", "f32", (3, 1)),
    ("Q_G_8", 16, 768, 4352, "f32", "f32", (4, 1)),
    ("Q_G_4", 33, 512, 768, "bf16", "bf16", (4, 1)),
    ("SB256A3", 65, 256, 1280, "f32", "bf16", (4, 1)),
    ("B32S8", 129, 768, 512, "f32", "f32", (4, 1)),
    ("B32S4", 9, 4096, 768, "f32", "f32", (4, 5)),      # (with the least workspace in one part of another shape)
    ("Q_G_3", 16, 2304, 512, "f32", "f32", (4, 5)),     # parts of one and two blocks
    ("Q_G_8", 32, 6400, 256, "bf16", "bf16", (4, 5)),
    ("Q_G_4", 33, 3072, 512, "bf16", "f32", (4, 5)),
    ("SB256A3", 20, 4352, 256, "f32", "f32", (4, 5)),
    ("Q_G_2", 40, 2560, 1024, "bf16", "bf16", (3, 5)),
    ("B32S8", 130, 2560, 1792, "bf16", "bf16", (1, 5)),
    ("Q_G_4", 259, 1536, 2048, "f32", "f32", (1, 3)),
])
def test_mlp_step_pair_on_integer_operands(O, tfq, gpu, rules, fmt, B, D, F, xdt, mid, plan):
    """gate and up in one launch of the integer tile kernel, whole and in K parts: against the float64 products of the
    decoded matrices (the companded line 3e-4, bf16 mid activations 5e-3, otherwise 3e-5 as above); a buffer behind the
    workspace stays as it was."""
    import ctypes
    import torch
    print(f"mlp_step {fmt} B={B} D={D} F={F} {xdt} mid={mid}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(82)
    Ws = [tfq.Weight(fmt, n, k, tfq.encode(fmt, torch.randn(n * k, device=gpu, generator=g) * 0.02)) for n, k in ((F, D), (F, D), (D, F))]
    x = torch.randn(B, D, device=gpu, generator=g)
    x = x.bfloat16() if xdt == "bf16" else x
    a, b, d = (W.decode().reshape(n, k).double() for W, (n, k) in zip(Ws, ((F, D), (F, D), (D, F))))
    u = x.double() @ a.T
    h = u * torch.sigmoid(u) * (x.double() @ b.T)
    want = (h.bfloat16().double() if mid == "bf16" else h) @ d.T
    tol = 5e-3 if mid == "bf16" else 3e-4 if fmt == "Q_G_8" else 3e-5
    L = tfq.lib()
    part = (B * F * 4 + 255) // 256 * 256
    least = 3 * part + (min(8 * B * F * 4, 256 * 256 * 256 * 4) + 255) // 256 * 256 * (B > 16)
    taken = rules.pair(fmt, F, D, xdt == "f32", B, L.tfq_mlp_workspace_bytes(B, F) - part)
    assert (taken.shape, taken.ksplit) == plan
    for size in (L.tfq_mlp_workspace_bytes(B, F), least):
        buf = torch.full((size + 4096,), 77, device=gpu, dtype=torch.uint8)
        y = torch.empty(B, D, device=gpu)
        rc = L.tfq_mlp_step(Ws[0].handle, Ws[1].handle, Ws[2].handle, ctypes.c_void_p(x.data_ptr()), 1 if xdt == "bf16" else 0, B,
                            ctypes.c_void_p(y.data_ptr()), 0, 1 if mid == "bf16" else 0, ctypes.c_void_p(buf.data_ptr()), size,
                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        assert float((y.double() - want).norm() / want.norm()) <= tol, size
        assert bool((buf[size:] == 77).all()), size
    for W in Ws:
        W.close()


@pytest.mark.parametrize("fmt,B,D,F,xdt", [("Q_4", 17, 512, 4352, "f32"), ("Q_4", 129, 4352, 512, "f32"), ("Q_G_6", 200, 768, 768, "bf16"),
                                           ("B32S4", 300, 256, 1280, "bf16"), ("Q_G_3", 333, 1280, 256, "f32")])
def test_mlp_step_scratch_in_the_areas_not_in_use(tfq, gpu, fmt, B, D, F, xdt):
    """More than sixteen rows, gate, up and down one after the other (the wire formats) or as the models choose: each product's
    scratch lies in areas that the later ones fill.  Against the float64 products of the decoded matrices (fp32 throughout 3e-5,
    bf16 rows and mid activations 5e-3); a buffer behind the workspace stays as it was."""
    import ctypes
    import torch
    g = torch.Generator(device="cuda").manual_seed(83)
    Ws = [tfq.Weight(fmt, n, k, tfq.encode(fmt, torch.randn(n * k, device=gpu, generator=g) * 0.02)) for n, k in ((F, D), (F, D), (D, F))]
    x = torch.randn(B, D, device=gpu, generator=g)
    x = x.bfloat16() if xdt == "bf16" else x
    a, b, d = (W.decode().reshape(n, k).double() for W, (n, k) in zip(Ws, ((F, D), (F, D), (D, F))))
    u = x.double() @ a.T
    h = u * torch.sigmoid(u) * (x.double() @ b.T)
    want = (h.bfloat16().double() if xdt == "bf16" else h) @ d.T
    L, code = tfq.lib(), 1 if xdt == "bf16" else 0
    size = L.tfq_mlp_workspace_bytes(B, F)
    buf = torch.full((size + 4096,), 77, device=gpu, dtype=torch.uint8)
    y = torch.empty(B, D, device=gpu)
    rc = L.tfq_mlp_step(Ws[0].handle, Ws[1].handle, Ws[2].handle, ctypes.c_void_p(x.data_ptr()), code, B, ctypes.c_void_p(y.data_ptr()), 0, code,
                        ctypes.c_void_p(buf.data_ptr()), size, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    assert float((y.double() - want).norm() / want.norm()) <= (5e-3 if xdt == "bf16" else 3e-5)
    assert bool((buf[size:] == 77).all())
    for W in Ws:
        W.close()


@pytest.mark.parametrize("fmt,B,D,F,xdt,mid", [
    ("B32S4", 3, 512, 8448, "f32", "f32"),    # down's K in three parts
    ("Q_G_8", 4, 8192, 768, "f32", "f32"),    # the longest D of the paired launch with two slot sets
    ("Q_G_4", 3, 8448, 512, "f32", "f32"),    # one block longer: gate, up and the elementwise step apart
    ("B32S8", 5, 512, 4352, "bf16", "f32"),
    ("Q_G_4", 8, 768, 4352, "bf16", "bf16"),
])
def test_mlp_step_two_slot_sets(O, tfq, gpu, fmt, B, D, F, xdt, mid):
    """Three or four fp32 rows and five to eight bf16 ones, with the workspace that is asked for and with the three areas
    alone (down unsplit): against the oracle within the bounds of the tests above; a buffer behind the workspace stays as
    it was."""
    import ctypes
    import torch
    print(f"mlp_step {fmt} B={B} D={D} F={F} {xdt} mid={mid}", flush=True)
    pays = [O.encode_tensor(fmt, O.rng_normal(70 + i, n * k, 0.02)) for i, (n, k) in enumerate(((F, D), (F, D), (D, F)))]
    x = O.rng_normal(9, B * D, 1.0).reshape(B, D)
    if xdt == "bf16":
        x = O.bf16_round(x)
    g = O.matmul(fmt, pays[0], F, D, x)
    u = O.matmul(fmt, pays[1], F, D, x)
    h = O.silu_mul(g.reshape(-1), u.reshape(-1)).reshape(B, F)
    if mid == "bf16":
        h = O.bf16_round(h)
    want = O.matmul(fmt, pays[2], D, F, h).astype(np.float64)
    Ws = [tfq.Weight(fmt, n, k, p) for p, (n, k) in zip(pays, ((F, D), (F, D), (D, F)))]
    xt = torch.from_numpy(x).to(gpu)
    if xdt == "bf16":
        xt = xt.bfloat16()
    tol = 5e-3 if mid == "bf16" else 3e-4 if fmt == "Q_G_8" else 3e-5
    L = tfq.lib()
    least = 3 * ((B * F * 4 + 255) // 256 * 256)
    for size in (L.tfq_mlp_workspace_bytes(B, F), least):
        buf = torch.full((size + 256,), 77, device=gpu, dtype=torch.uint8)
        y = torch.empty(B, D, device=gpu)
        rc = L.tfq_mlp_step(Ws[0].handle, Ws[1].handle, Ws[2].handle, ctypes.c_void_p(xt.data_ptr()), 1 if xdt == "bf16" else 0, B,
                            ctypes.c_void_p(y.data_ptr()), 0, 1 if mid == "bf16" else 0, ctypes.c_void_p(buf.data_ptr()), size,
                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        err = np.linalg.norm(y.cpu().numpy() - want) / np.linalg.norm(want)
        assert err <= tol, (size, err)
        assert bool((buf[size:] == 77).all())
    for W in Ws:
        W.close()


def test_capacity_dispatch_matches_oracle(O, tfq, gpu):
    """moe_engine::plan_dispatch / gather / combine (engines/trainer/moe/dispatch.cpp:9-78) through the C ABI."""
    import torch
    fmt, E, D, F, T, K, slots = "B32S4", 4, 1024, 2048, 16, 2, 5
    gate, up, down, hg, hu, hd = _experts(O, tfq, fmt, E, D, F, 900)
    x = O.rng_normal(11, T * D, 1.0).reshape(T, D)
    rng = np.random.default_rng(12)
    idx = rng.integers(0, E, size=(T, K)).astype(np.int32)
    w = rng.standard_normal((T, K)).astype(np.float32)
    # the plan alone: the library's host-side lists equal the oracle's
    for a, b in zip(tfq.moe_plan_dispatch(idx, w, E, slots), O.moe_plan_dispatch(idx, w, E, slots)):
        assert np.array_equal(a, b)
    ref, nd_ref = O.moe_ffn_capacity(fmt, hg, hu, hd, D, F, idx, w, slots, x)
    y, nd = tfq.moe_ffn_capacity(gate, up, down, idx, w, slots, torch.from_numpy(x).to(gpu), mid_dtype=torch.float32)
    assert nd == nd_ref and nd > 0
    assert rel_err(y.cpu().numpy(), ref) <= 1e-3
    # bf16 activations and intermediate
    xb = O.bf16_round(x)
    refb, _ = O.moe_ffn_capacity(fmt, hg, hu, hd, D, F, idx, w, slots, xb, mid_bf16=True)
    yb, _ = tfq.moe_ffn_capacity(gate, up, down, idx, w, slots, torch.from_numpy(xb).to(gpu).bfloat16(), out_dtype=torch.float32)
    assert rel_err(yb.cpu().numpy(), refb) <= 1e-2
    # an expert id outside 0..E-1 is an error, as in the reference
    bad = idx.copy()
    bad[0, 0] = E
    with pytest.raises(tfq.TfqError):
        tfq.moe_ffn_capacity(gate, up, down, bad, w, slots, torch.from_numpy(x).to(gpu))
