"""The dispatch rules of the tiled products and the native launch sequence at
the sizes where they change: K splits of small launches, the chunks of the
weight gradients, the small-group limit, the top-k over a token's lanes."""
import pytest
import torch

from fusionllm_amd import DeepSeekMoE, configs
from fusionllm_amd import _kernels as K
from fusionllm_amd._lib import FusionMoEError

pytestmark = pytest.mark.gpu


def _bf(*shape, g, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).bfloat16()


def _groups(counts, device):
    off = torch.tensor([0, *torch.tensor(counts).cumsum(0).tolist()], dtype=torch.int32, device=device)
    return off, sum(counts)


# bf16 outputs of fp32 sums of bf16 operands: one rounding (rms 1.5e-3 relative,
# 2^-9 at most) and the sums' own error (K 2^-24, below it); up to three roundings
# in a row for h, da and db (rms 2.6e-3): rel-L2 bound 4e-3.
BOUND = 4e-3


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30))


@pytest.mark.parametrize("counts,shared,d,I", [
    # (each launch has more than 256 routed rows, so that none goes to the small-group kernel)
    ([0, 15, 16, 17, 300], 0, 512, 1024),   # down: 16 steps, the fewest that split; slices of 16 rows
    ([255, 256, 257, 1], 300, 1024, 576),   # tile edges, columns that do not fill a tile
    ([700, 0, 3, 120], 1000, 64, 1088),     # one K step forward, two ranges of the down product
    ([300, 0, 40, 513], 200, 1024, 1408),   # gate/up and down backward split over ragged groups and an empty one
    ([130] * 16, 0, 1024, 512),             # one row tile of each group, half full
])
def test_row_products_of_small_launches(gpu_device, counts, shared, d, I):
    D = gpu_device
    g = torch.Generator().manual_seed(sum(counts) + d)
    E, G = len(counts), len(counts) + (1 if shared else 0)
    off, rr = _groups(counts, D)
    x, h = _bf(rr, d, g=g).to(D), _bf(rr + shared, I, g=g).to(D)
    xs = _bf(shared, d, g=g).to(D) if shared else None
    dab = _bf(rr + shared, 2 * I, g=g, scale=0.1).to(D)
    w1 = [_bf(I, d, g=g, scale=0.05).to(D) for _ in range(G)]
    w3 = [_bf(I, d, g=g, scale=0.05).to(D) for _ in range(G)]
    w2 = [_bf(d, I, g=g, scale=0.05).to(D) for _ in range(G)]
    dor = _bf(rr, d, g=g).to(D)
    dos = _bf(shared, d, g=g).to(D) if shared else None
    abi = _bf(rr + shared, 2 * I, g=g).to(D)
    ab, hf = K.gateup_fwd(x, xs, off, E, w1, w3, I)
    o = K.down_fwd(h, off, E, rr, shared, w2, d)
    dd = K.down_bwd_dx(dor, dos, off, E, w2, abi, I)
    dx = K.gateup_bwd_dx(dab, off, E, rr, shared, w1, w3, d)
    bounds = [0, *torch.tensor(counts).cumsum(0).tolist()] + ([rr + shared] if shared else [])
    xa = torch.cat([x, xs]) if shared else x
    da = torch.cat([dor, dos]) if shared else dor
    for q in range(G):
        r = slice(bounds[q], bounds[q + 1])
        if r.stop == r.start:
            continue
        f = lambda t: t.float()
        assert _rel(ab[r, :I], f(xa[r]) @ f(w1[q]).t()) < BOUND
        assert _rel(ab[r, I:], f(xa[r]) @ f(w3[q]).t()) < BOUND
        assert _rel(o[r], f(h[r]) @ f(w2[q]).t()) < BOUND
        assert _rel(dx[r], f(dab[r, :I]) @ f(w1[q]) + f(dab[r, I:]) @ f(w3[q])) < BOUND
        # h from the a|b of the same launch; da, db: the SwiGLU's derivative at abi
        assert _rel(hf[r], torch.nn.functional.silu(f(ab[r, :I])) * f(ab[r, I:])) < BOUND
        a, b = f(abi[r, :I]), f(abi[r, I:])
        sg, dh = torch.sigmoid(a), f(da[r]) @ f(w2[q])
        assert _rel(dd[r, :I], dh * b * sg * (1 + a * (1 - sg))) < BOUND
        assert _rel(dd[r, I:], dh * a * sg) < BOUND


@pytest.mark.parametrize("rows", [512, 513])    # 8 rows for each of 64 experts, and one more: all tiled
@pytest.mark.parametrize("shared", [0, 85, 200])  # none, small slabs, tiled
@pytest.mark.parametrize("big", [True, False])  # a group above 128 rows beside small ones; none (512 rows: no tiles at all)
def test_forward_products_at_the_small_group_limit(gpu_device, rows, shared, big):
    D, E, d, I = gpu_device, 64, 1024, 1024
    g = torch.Generator().manual_seed(rows + shared)
    counts = [130 if big else 127, 128, 1, 0, 0]
    rest = rows - sum(counts)
    counts += [rest // 59 + (1 if e < rest % 59 else 0) for e in range(59)]
    assert sum(counts) == rows and len(counts) == E
    G = E + (1 if shared else 0)
    off, rr = _groups(counts, D)
    x, h = _bf(rr, d, g=g).to(D), _bf(rr + shared, I, g=g).to(D)
    xs = _bf(shared, d, g=g).to(D) if shared else None
    gd = torch.Generator(device=D).manual_seed(1)
    ws = torch.randn(3, G, d, I, generator=gd, device=D, dtype=torch.bfloat16).mul_(0.05)
    w1, w3, w2 = (list(w.unbind(0)) for w in ws)
    ab, hf = K.gateup_fwd(x, xs, off, E, w1, w3, I)
    o = K.down_fwd(h, off, E, rr, shared, w2, d)
    bounds = [0, *torch.tensor(counts).cumsum(0).tolist()] + ([rr + shared] if shared else [])
    xa = torch.cat([x, xs]) if shared else x
    for q in range(G):
        r = slice(bounds[q], bounds[q + 1])
        if r.stop == r.start:
            continue
        f = lambda t: t.float()
        assert _rel(ab[r, :I], f(xa[r]) @ f(w1[q]).t()) < BOUND
        assert _rel(ab[r, I:], f(xa[r]) @ f(w3[q]).t()) < BOUND
        assert _rel(hf[r], torch.nn.functional.silu(f(ab[r, :I])) * f(ab[r, I:])) < BOUND
        assert _rel(o[r], f(h[r]) @ f(w2[q]).t()) < BOUND


def test_split_tiles_match_whole_tiles_in_every_product(gpu_device):
    # At 16 K steps and more every product of a launch of fewer tiles than CUs
    # is split. Only the fp32 summation order differs from the same launch
    # without a workspace: outputs agree to a few bf16 roundings (one on the
    # sum, up to three more in the SwiGLU epilogues), and do differ somewhere.
    from tests.gpu_util import close, rel_l2
    from tests.test_gpu_kernels import _row_products
    D, d, I = gpu_device, 1024, 1088
    g = torch.Generator().manual_seed(11)
    counts, shared = [1500, 700, 0, 300], 500
    E, G = 4, 5
    off, rr = _groups(counts, D)
    t = lambda *s, scale=1.0: _bf(*s, g=g, scale=scale).to(D)
    args = (D, t(rr, d), t(shared, d), t(rr, d), t(shared, d), off, E, [t(I, d, scale=.05) for _ in range(G)],
            [t(I, d, scale=.05) for _ in range(G)], [t(d, I, scale=.05) for _ in range(G)], t(rr + shared, 2 * I),
            t(rr + shared, I, scale=.3), t(rr + shared, 2 * I, scale=.05))
    split, whole = _row_products(*args, split=True), _row_products(*args, split=False)
    for name, a, b in zip(("ab", "h", "out", "d_ab", "dx_rows"), split, whole):
        close(a, b, rtol=3.2e-2, atol=2e-3)
        assert rel_l2(a, b.float()) < 2e-3, name
        assert not torch.equal(a, b), f"{name}: no tile was split"


@pytest.mark.parametrize("counts,shared,m,n", [
    ([0, 1, 63, 64, 65], 0, 256, 320),       # groups without rows, one stage and its edges
    ([1151, 1152, 1153, 0], 0, 512, 256),    # one chunk or two (kc = 768: from 1152 rows)
    ([100, 2000], 5000, 64, 704),            # shared group in several chunks, a partial tile
    ([10766, 5], 0, 64, 704),                # 14 chunks of 832 rows: the last one empty, a zero partial
    ([1216], 0, 320, 256),                   # one group: the chunk count that fills whole rounds, here one
    ([1217], 0, 320, 256),                   # ... and two from here
    ([5000], 0, 2048, 1536),                 # 48 tiles in five chunks, the last shorter
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_weight_gradient_chunks(gpu_device, counts, shared, m, n, dtype):
    D = gpu_device
    g = torch.Generator().manual_seed(sum(counts) + m)
    E, G = len(counts), len(counts) + (1 if shared else 0)
    off, rr = _groups(counts, D)
    a, b = _bf(rr, m, g=g).to(D), _bf(rr, n, g=g).to(D)
    sa, sb = (_bf(shared, m, g=g).to(D), _bf(shared, n, g=g).to(D)) if shared else (None, None)
    outs = [torch.full((m, n), float("nan"), dtype=dtype, device=D) for _ in range(G)]
    K.weight_grad(a, sa, b, sb, off, E, rr, shared, m, outs, None, dtype)
    bounds = [0, *torch.tensor(counts).cumsum(0).tolist()]
    for q in range(G):
        A, B = (sa, sb) if q == E else (a[bounds[q]:bounds[q + 1]], b[bounds[q]:bounds[q + 1]])
        want = A.double().t() @ B.double()
        if A.shape[0] == 0:
            assert not outs[q].any()  # a group without rows: zeros
        else:
            # fp32: sums of at most 11000 exact products, error about sqrt(rows) 2^-24 per unit
            assert _rel(outs[q], want) < (BOUND if dtype == torch.bfloat16 else 2e-6)


@pytest.mark.parametrize("T,shared,autocast", [(129, 1, False), (300, 0, False), (700, 1, True)])
def test_native_sequence_equals_the_entry_points(gpu_device, T, shared, autocast):
    # With timing on, the block runs through the per-entry-point wrappers; the
    # native sequence launches the same kernels: bit-equal.
    cfg = configs.BlockConfig("native", T, dim=256, inter=512, n_experts=8, topk=2, n_shared=shared, bias="skew")
    data = configs.make_block(cfg, seed=5)
    res = []
    for timer in ({}, None):
        torch.manual_seed(0)
        m = DeepSeekMoE(cfg.moe_config())
        m.load_state_dict(data.state_dict())
        m = m.to(gpu_device, torch.float32 if autocast else torch.bfloat16)
        x = data.x.to(gpu_device, torch.float32 if autocast else torch.bfloat16).requires_grad_()
        K.set_timer(timer)
        try:
            with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
                y = m(x)
            y.backward(data.dy.to(gpu_device, y.dtype))
        finally:
            K.set_timer(None)
        res.append([y.detach(), x.grad, m._last_indices, *[p.grad for _, p in m.named_parameters()]])
    for a, b in zip(*res):
        assert (a is None) == (b is None)
        assert a is None or torch.equal(a, b)


def test_native_sequence_reports_refused_shapes(gpu_device):
    # dim 96 is no multiple of 64: refused on the host, before any launch
    w, wt = _bf(64, 96, g=None), _bf(96, 64, g=None)
    x, gw, gb, w1, w2 = (t.to(gpu_device) for t in (_bf(200, 96, g=None), _bf(2, 96, g=None), _bf(2, g=None), w, wt))
    with pytest.raises(FusionMoEError, match="fmoe_route_and_dispatch"):
        K.block_host().forward(x, gw, gb, [w1] * 2, [w1] * 2, [w2] * 2, 1, 64, 1.0, False, torch.bfloat16, None, None,
                               K.stream_handle())


@pytest.mark.parametrize("E,k", [(1, 1), (15, 8), (16, 8), (17, 8), (33, 5), (64, 8)])
def test_topk_ties_and_nan_across_lanes(gpu_device, E, k):
    # Scores that tie across lanes and within one, and NaN scores: the lowest
    # expert index wins, NaN first, as torch's stable descending sort orders.
    T, d = 200, 64
    g = torch.Generator().manual_seed(E)
    x = torch.zeros(T, d).bfloat16()
    x[:, 0] = 1.0
    gw = torch.zeros(E, d).bfloat16()
    gw[:, 0] = torch.randint(-2, 3, (E,), generator=g).bfloat16()
    x[3, 1] = float("nan")  # a token whose every score is NaN
    gb = torch.zeros(E).bfloat16()
    idx, _, w, v = K.router_fwd(x.to(gpu_device), gw.to(gpu_device), gb.to(gpu_device), k, 1.0)
    want = torch.sort(gw[:, 0].float(), descending=True, stable=True).indices[:k]
    got = idx.cpu().long()
    keep = torch.ones(T, dtype=torch.bool)
    keep[3] = False
    assert torch.equal(got[keep], want.expand(T - 1, k))
    assert torch.equal(got[3], torch.arange(k)) and torch.isnan(v[3]).all()


def _mixed(m, which):
    """bf16 for some of an fp32 module's parameters (autocast takes any mix)."""
    for n, p in m.named_parameters():
        if {"shared": n.startswith("shared_expert"), "w3": n.endswith("w3.weight"),
            "w1, a w2": n.endswith("w1.weight") or n == "experts.2.w2.weight",
            "first expert": n.startswith("experts.0.")}[which]:
            p.data = p.data.bfloat16()
    return m


@pytest.mark.parametrize("which", ["shared", "w3", "w1, a w2", "first expert"])
@pytest.mark.parametrize("path", ["native", "wrappers", "operator"])
def test_weight_gradients_of_mixed_parameter_dtypes(gpu_device, which, path):
    # The values are bf16 ones, so the kernels read the same operands whatever
    # the parameters' dtypes: each gradient is the fp32 module's, rounded once
    # to its parameter's dtype.
    cfg = configs.BlockConfig("mixed", 300, dim=128, inter=192, n_experts=4, topk=2, n_shared=1, bias="skew")
    data = configs.make_block(cfg, seed=9)
    grads = []
    for mixed in (False, True):
        m = DeepSeekMoE(cfg.moe_config())
        m.load_state_dict({n: t.bfloat16().float() for n, t in data.state_dict().items()})
        m = m.to(gpu_device, torch.float32)
        m = _mixed(m, which) if mixed else m
        x = data.x.to(gpu_device).bfloat16().float()
        K.set_timer({} if path == "wrappers" else None)
        try:
            with torch.autocast("cuda", dtype=torch.bfloat16):
                if path == "operator":
                    y = torch.ops.fusionllm.moe_fwd(x, m.gate.weight, m.gate.bias, m._flat_weights(), 2, 1.0, True,
                                                    torch.float32)[0]
                else:
                    y = m(x)
            y.backward(data.dy.to(gpu_device, y.dtype))
        finally:
            K.set_timer(None)
        grads.append({n: (p.dtype, p.grad) for n, p in m.named_parameters()})
    assert len({t for t, _ in grads[1].values()}) == 2
    for n, (t, got) in grads[1].items():
        want = grads[0][n][1]
        assert (got is None) == (want is None), n
        assert got is None or (got.dtype == t and torch.equal(got, want.to(t))), n


def test_weight_grad_refuses_outputs_that_do_not_fit(gpu_device):
    # on the host, before the launch
    off, rr = _groups([64, 64], gpu_device)
    a, b = (torch.zeros(rr, n, dtype=torch.bfloat16, device=gpu_device) for n in (128, 64))
    out = lambda *s, dtype=torch.float32: torch.empty(*s, dtype=dtype, device=gpu_device)
    for outs in ([out(128, 64), out(128, 64, dtype=torch.bfloat16)], [out(128, 64), out(64, 64)], [out(128, 64)],
                 [out(128, 64), out(64, 128).t()]):
        with pytest.raises(RuntimeError, match="outs_lo"):
            K.weight_grad(a, None, b, None, off, 2, rr, 0, 128, outs, None, torch.float32)


@pytest.mark.parametrize("counts,shared,m,n", [
    ([0, 1, 63, 64, 65], 0, 256, 320),        # one stage of 64 rows and its edges
    ([127, 129, 192, 193, 255], 300, 64, 64),  # two to four stages: fewer than are fetched ahead; a shared group
    ([512, 513, 577, 4000], 1100, 320, 576),   # past the eight stages of the index ring, several chunks
])
def test_gathered_weight_gradient_equals_the_copied_rows(gpu_device, counts, shared, m, n):
    D = gpu_device
    g = torch.Generator().manual_seed(sum(counts))
    E, G = len(counts), len(counts) + (1 if shared else 0)
    off, rr = _groups(counts, D)
    T, k = (rr + 2) // 3, 3
    x, a = _bf(T, n, g=g).to(D), _bf(rr, m, g=g).to(D)
    perm = torch.randperm(T * k, generator=g)[:rr].to(torch.int32).to(D)
    sa, sb = (_bf(shared, m, g=g).to(D), _bf(shared, n, g=g).to(D)) if shared else (None, None)
    outs = [[torch.full((m, n), float("nan"), device=D) for _ in range(G)] for _ in range(2)]
    K.weight_grad(a, sa, x[perm.long() // k].contiguous(), sb, off, E, rr, shared, m, outs[0], None, torch.float32)
    K.weight_grad(a, sa, x, sb, off, E, rr, shared, m, outs[1], None, torch.float32, b_gather=perm, k=k)
    for want, got in zip(*outs):
        assert torch.equal(want, got)


@pytest.mark.parametrize("path", ["native", "wrappers"])
@pytest.mark.parametrize("T,d,inter,splits", [(300, 256, 448, False), (300, 256, 576, True)])
def test_split_workspace_only_where_a_launch_can_split(gpu_device, T, d, inter, splits, path):
    # fewer than 16 K steps of 64 in every product (2 * 448 / 64 = 14): no split,
    # so no 64 MB of partials; 2 * 576 / 64 = 18 steps in the input gradient
    cfg = configs.BlockConfig("ws", T, dim=d, inter=inter, n_experts=4, topk=2, n_shared=1, bias="skew")
    data = configs.make_block(cfg, seed=1)
    m = DeepSeekMoE(cfg.moe_config())
    m.load_state_dict(data.state_dict())
    m = m.to(gpu_device, torch.bfloat16)
    x = data.x.to(gpu_device, torch.bfloat16).requires_grad_()
    dy = data.dy.to(gpu_device, torch.bfloat16)
    K.set_timer({} if path == "wrappers" else None)
    try:
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        m(x).backward(dy)
    finally:
        K.set_timer(None)
    assert (torch.cuda.max_memory_allocated() - before > 60 << 20) == splits


def test_forward_products_of_weights_at_8_byte_offsets(gpu_device):
    # Weights that are views into one buffer, 8 bytes past a 16-byte boundary:
    # 11 rows per expert, which aligned operands send to the tiled kernel, go to
    # the small-group kernel, whose loads take any such address.
    D, E, rows, d, I = gpu_device, 40, 11, 256, 128
    g = torch.Generator().manual_seed(3)
    off, rr = _groups([rows] * E, D)
    x, h = _bf(rr, d, g=g).to(D), _bf(rr, I, g=g).to(D)
    buf = _bf(E * (3 * I * d + 8), g=g, scale=0.05).to(D)
    w1, w3, w2 = [], [], []
    for e in range(E):
        at = e * (3 * I * d + 8) + 4
        for ws, shape in ((w1, (I, d)), (w3, (I, d)), (w2, (d, I))):
            ws.append(buf[at:at + I * d].view(shape))
            assert ws[-1].data_ptr() % 16 == 8
            at += I * d
    ab, _ = K.gateup_fwd(x, None, off, E, w1, w3, I)
    o = K.down_fwd(h, off, E, rr, 0, w2, d)
    for e in range(E):
        r = slice(e * rows, (e + 1) * rows)
        assert _rel(ab[r, :I], x[r].float() @ w1[e].float().t()) < BOUND
        assert _rel(ab[r, I:], x[r].float() @ w3[e].float().t()) < BOUND
        assert _rel(o[r], h[r].float() @ w2[e].float().t()) < BOUND


@pytest.mark.parametrize("E,k,nans", [(2, 1, [1]), (8, 2, [5]), (17, 3, [16]), (33, 5, [20, 4]), (64, 8, [63, 32, 31])])
def test_topk_with_nan_experts_among_finite_scores(gpu_device, E, k, nans):
    # A NaN score beats every finite one; several go to the lowest index first,
    # then the finite ones in order: torch's stable descending sort.
    T, d = 50, 64
    g = torch.Generator().manual_seed(E)
    x = torch.zeros(T, d).bfloat16()
    x[:, 0] = 1.0
    gw = torch.zeros(E, d).bfloat16()
    gw[:, 0] = torch.randint(-2, 3, (E,), generator=g).bfloat16()
    gw[nans, 1] = float("nan")  # 0 * NaN: this expert's score is NaN for every token
    score = gw[:, 0].float()
    score[nans] = float("nan")
    idx, _, w, v = K.router_fwd(x.to(gpu_device), gw.to(gpu_device), torch.zeros(E).bfloat16().to(gpu_device), k, 1.0)
    want = torch.sort(score, descending=True, stable=True).indices[:k]
    assert torch.equal(idx.cpu().long(), want.expand(T, k))
    assert torch.equal(torch.isnan(v.cpu()), torch.isnan(score[want]).expand(T, k))
