"""GPU parity (through the C ABI) of the fused Linear -> heads -> feature map launch
against torch's fp64 matmul and the CPU oracle's feature map.

Tolerances: the projections y are fp16 roundings of an fp32-accumulated product, compared
with the fp64 product of the same fp16 inputs: |dy| <= 1.5e-3 * max(1, |y|) (one fp16 ulp
is 9.8e-4 relative).  phi is compared (a) with the oracle applied to the y the kernel itself
returned (<= 2e-3 absolute, the feature-map bar) and (b) with the oracle applied to the
fp64 product rounded to fp16 (<= 4e-3: an ulp of difference in y moves the angle).
"""
import pytest
import torch

from oracle import rfa_oracle as O

pytestmark = pytest.mark.gpu

# L, B, E, H, d, D
SHAPES = [(128, 2, 256, 4, 64, 64), (300, 2, 512, 8, 64, 64), (70, 3, 128, 2, 64, 64), (33, 1, 256, 2, 128, 128), (5, 2, 64, 1, 64, 32),
          (1, 1, 192, 3, 64, 128), (257, 1, 128, 1, 128, 64)]


def _randn(*shape, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g, dtype=torch.float32)


def _inputs(L, B, E, H, d, seed, n):
    x = (_randn(L, B, E, seed=seed) * 0.8).half()
    ws = [(_randn(H * d, E, seed=seed + 1 + p) / E ** 0.5 * 1.5).half() for p in range(n)]
    bs = [(_randn(H * d, seed=seed + 11 + p) * 0.3).half() for p in range(n)]
    return x, ws, bs


def _rel(a, b):
    return ((a - b).norm() / b.norm()).item()


def _linear64(x, w, b, H, d):
    y = x.double() @ w.double().t()
    if b is not None:
        y = y + b.double()
    return y.view(*x.shape[:2], H, d)


@pytest.mark.parametrize("streaming", [False, True])
@pytest.mark.parametrize("L,B,E,H,d,D", SHAPES)
def test_qkv_projection_with_feature_map(L, B, E, H, d, D, streaming, knobs):
    """The tile height picked by itself and the tallest one (the "project_streaming" knob)."""
    from rfa_amd import rfa_hip
    knobs(project_streaming=1 if streaming else -1)
    x, ws, bs = _inputs(L, B, E, H, d, 900 + L, 3)
    bs[1] = None                                       # one projection without bias
    wf = (_randn(H, D, d, seed=77) * 0.9).half()
    print(f"project+phi L={L} B={B} E={E} H={H} d={d} D={D}", flush=True)
    dev = lambda t: None if t is None else t.cuda()
    ys, phis = rfa_hip.project_feature_map(x.cuda(), [w.cuda() for w in ws], [dev(b) for b in bs],
                                           [True, True, False], wf.cuda(), H, O.SCALE)
    assert phis[2] is None and phis[0].shape == (L, B, H, 2 * D)
    for p in range(3):
        want = _linear64(x, ws[p], bs[p], H, d)
        got = ys[p].double().cpu()
        assert ys[p].shape == (L, B, H, d)
        assert ((got - want).abs() <= 1.5e-3 * want.abs().clamp_min(1.0)).all(), (p, (got - want).abs().max().item())
        if p < 2:
            phi = phis[p].float().cpu()
            own = O.random_project(ys[p].float().cpu(), wf.float())
            assert (phi - own).abs().max().item() <= 2e-3
            ref = O.random_project(want.half().float(), wf.float())
            assert (phi - ref).abs().max().item() <= 4e-3


# rows around the three tile heights, one and several contraction rounds of the three-stage ring, odd
# numbers of 64-wide heads (half a column tile), every (d, D)
@pytest.mark.parametrize("rows_knob", [0, 1, 2])
@pytest.mark.parametrize("R,E,H,d,D,n", [(1, 64, 1, 64, 32, 1), (63, 128, 3, 64, 64, 1), (65, 64, 3, 64, 128, 3), (127, 192, 1, 128, 32, 2),
                                         (129, 64, 2, 128, 64, 1), (255, 128, 1, 128, 128, 3), (257, 320, 5, 64, 64, 2), (513, 64, 2, 64, 32, 3)])
def test_projection_tile_edges(R, E, H, d, D, n, rows_knob, knobs):
    from rfa_amd import rfa_hip
    knobs(project_streaming=rows_knob)
    x, ws, bs = _inputs(R, 1, E, H, d, 970 + R, n)
    wf = (_randn(H, D, d, seed=79) * 0.9).half()
    want_phi = [p != n - 1 or n == 1 for p in range(n)]
    print(f"project tile edges R={R} E={E} H={H} d={d} D={D} n={n} knob={rows_knob}", flush=True)
    ys, phis = rfa_hip.project_feature_map(x.cuda(), [w.cuda() for w in ws], [b.cuda() for b in bs], want_phi, wf.cuda(), H, O.SCALE)
    for p in range(n):
        want = _linear64(x, ws[p], bs[p], H, d)
        assert ((ys[p].double().cpu() - want).abs() <= 1.5e-3 * want.abs().clamp_min(1.0)).all(), p
        if want_phi[p]:
            own = O.random_project(ys[p].float().cpu(), wf.float())
            assert (phis[p].float().cpu() - own).abs().max().item() <= 2e-3


# the same edges with two groups of waves to a tile: one stage of 64 columns, two, an odd number, more than the ring holds
@pytest.mark.parametrize("rows_knob", [0, 3])
@pytest.mark.parametrize("R,E,H,d,D,n", [(1, 64, 1, 64, 32, 1), (65, 128, 3, 64, 128, 3), (127, 192, 1, 128, 128, 2), (129, 64, 2, 128, 64, 1),
                                         (257, 320, 5, 64, 64, 2), (500, 512, 2, 128, 32, 3)])
def test_projection_by_two_groups(R, E, H, d, D, n, rows_knob, knobs):
    test_projection_tile_edges(R, E, H, d, D, n, rows_knob, knobs)


@pytest.mark.parametrize("streaming", [False, True])
def test_projection_without_keeping_y(streaming, knobs):
    """keep_y=False (what the modules ask for when nothing requires a gradient): phi and the plain
    projection come out bit-identical to the keeping call, y of the phi projections is not produced."""
    from rfa_amd import rfa_hip
    from rfa_amd.projection import project_heads
    knobs(project_streaming=1 if streaming else -1)
    L, B, E, H, d, D = 200, 3, 256, 4, 64, 64
    x, ws, bs = _inputs(L, B, E, H, d, 4321, 3)
    wf = (_randn(H, D, d, seed=78) * 0.9).half().cuda()
    args = (x.cuda(), [w.cuda() for w in ws], [b.cuda() for b in bs], [True, True, False], wf, H, O.SCALE)
    print(f"project+phi without y, streaming={streaming}", flush=True)
    ys, phis = rfa_hip.project_feature_map(*args)
    ys0, phis0 = rfa_hip.project_feature_map(*args, keep_y=False)
    assert ys0[0] is None and ys0[1] is None and phis0[2] is None
    assert torch.equal(ys0[2], ys[2]) and torch.equal(phis0[0], phis[0]) and torch.equal(phis0[1], phis[1])
    layers = []
    for w, b in zip(ws, bs):
        lin = torch.nn.Linear(E, H * d).cuda().half()
        lin.weight.data.copy_(w); lin.bias.data.copy_(b)
        layers.append(lin)
    # the modules' entry: trainable layers under no_grad must take the keep_y=False launch, and the keeping one
    # (with the same bits) when a gradient can be asked for
    seen = []
    real = rfa_hip.project_feature_map

    def spy(*a, **kw):
        seen.append(a[7] if len(a) > 7 else kw.get("keep_y", True))
        return real(*a, **kw)
    rfa_hip.project_feature_map = spy
    try:
        with torch.no_grad():
            outs = project_heads(x.cuda(), layers, (True, True, False), H, wf, O.SCALE)
        kept = project_heads(x.cuda(), layers, (True, True, False), H, wf, O.SCALE)
    finally:
        rfa_hip.project_feature_map = real
    assert seen == [False, True] and all(p.requires_grad for lin in layers for p in lin.parameters())
    assert torch.equal(outs[0], phis[0]) and torch.equal(outs[1], phis[1]) and torch.equal(outs[2], ys[2])
    assert all(torch.equal(a, b) for a, b in zip(outs, kept)) and kept[0].requires_grad
    with pytest.raises(Exception, match="neither y nor phi"):
        from rfa_amd import _lib
        import ctypes
        arr = ctypes.c_void_p * 1
        xx = x.cuda()
        _lib.check(_lib.load().rfa_project_feature_map(xx.data_ptr(), arr(ws[0].cuda().data_ptr()), None, arr(None), None, 1,
                                                       None, L * B, E, H, D, d, O.SCALE, None))


def test_plain_projection_is_a_linear_layer():
    """No phi requested: out_proj-style use, one projection, with and without bias."""
    from rfa_amd import rfa_hip
    L, B, E, H, d = 130, 2, 512, 8, 64
    x, ws, bs = _inputs(L, B, E, H, d, 950, 1)
    for b in (bs[0], None):
        ys, phis = rfa_hip.project_feature_map(x.cuda(), [ws[0].cuda()], [None if b is None else b.cuda()], [False],
                                               None, H, O.SCALE)
        assert phis == [None]
        want = _linear64(x, ws[0], b, H, d)
        got = ys[0].double().cpu()
        assert ((got - want).abs() <= 1.5e-3 * want.abs().clamp_min(1.0)).all()
        ref16 = torch.nn.functional.linear(x.cuda(), ws[0].cuda(), None if b is None else b.cuda()).view(L, B, H, d)
        assert (ys[0].float() - ref16.float()).abs().max().item() <= 4e-3      # the library GEMM, for reference


def test_zero_rows_and_argument_checks():
    from rfa_amd import rfa_hip
    H, d, D, E = 2, 64, 64, 128
    x, ws, bs = _inputs(4, 1, E, H, d, 960, 2)
    x[1] = 0
    ws = [w.cuda() for w in ws]
    wf = (_randn(H, D, d, seed=78)).half().cuda()
    ys, phis = rfa_hip.project_feature_map(x.cuda(), ws, [None, None], [True, True], wf, H, O.SCALE)
    # a zero input row without bias projects to zero, whose phi is [0.., scale..]
    assert (ys[0][1] == 0).all()
    assert (phis[0][1, 0, :, :D] == 0).all() and (phis[0][1, 0, :, D:].float() - O.SCALE).abs().max() <= 1e-4
    with pytest.raises(ValueError):
        rfa_hip.project_feature_map(x.cuda(), ws, [None], [True, True], wf, H, O.SCALE)
    with pytest.raises(ValueError):
        rfa_hip.project_feature_map(x.cuda(), ws, [None, None], [True, False], None, H, O.SCALE)
    with pytest.raises((RuntimeError, ValueError)):
        rfa_hip.project_feature_map(x[..., :100].contiguous().cuda(), [w[:, :100].contiguous() for w in ws],
                                    [None, None], [False, False], None, H, O.SCALE)    # E not a multiple of 64
    with pytest.raises((RuntimeError, TypeError)):
        rfa_hip.project_feature_map(x, [w.cpu() for w in ws], [None, None], [False, False], None, H, O.SCALE)


@pytest.mark.parametrize("with_pad", [False, True])
def test_causal_module_fused_projections_match_unfused_chain(with_pad):
    """CausalAttention with the q/k/v projections + phi as one launch vs the same module running
    nn.Linear + random_project: outputs within 4e-3, every gradient within 1e-2 (relative
    Frobenius norm) of the unfused module's, and within 2e-2 of an fp64 autograd run of the
    oracle chain."""
    from rfa_amd import CausalAttention
    torch.manual_seed(5)
    T, B, E, H, d, D = 200, 3, 256, 4, 64, 64
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
    with torch.no_grad():
        m.sigma.mul_(1.0 + 0.1 * torch.randn_like(m.sigma))
        m.out_proj.bias.normal_(0, 0.1)
    W = O.make_w(d, D, H).cuda().half()
    x0 = (torch.randn(T, B, E) * 0.7).half()
    go = torch.randn(T, B, E).half().cuda()
    pad = None
    if with_pad:
        pad = torch.zeros(B, T, dtype=torch.bool)
        pad[1, 150:] = True
        pad = pad.cuda()

    def run(fused):
        m.fuse_projections = fused
        m.zero_grad(set_to_none=True)
        x = x0.clone().cuda().requires_grad_(True)
        y = m(x, W, key_padding_mask=pad)
        y.backward(go)
        return y.detach().float().cpu(), {"x": x.grad.float().cpu(),
                                          **{n: p.grad.float().cpu() for n, p in m.named_parameters()}}

    y_f, g_f = run(True)
    y_u, g_u = run(False)
    assert (y_f - y_u).abs().max().item() <= 4e-3
    rel = lambda a, b: ((a - b).norm() / b.norm().clamp_min(1e-30)).item()
    for name in g_u:
        assert torch.isfinite(g_f[name]).all(), name
        assert rel(g_f[name], g_u[name]) <= 1e-2, (name, rel(g_f[name], g_u[name]))

    # fp64 autograd through the oracle chain with the same fp16 parameters
    P = {n: p.detach().double().cpu().requires_grad_(True) for n, p in m.named_parameters()}
    x = x0.double().requires_grad_(True)
    lin = lambda n: x @ P[n + ".weight"].t() + P[n + ".bias"]
    q, k, v = (lin(n).reshape(T, B, H, d) for n in ("q_proj", "k_proj", "v_proj"))
    Wp = O.build_random_matrices(W.double().cpu(), 1.0, P["sigma"], True)
    pq, pk = O.random_project(q, Wp), O.random_project(k, Wp)
    if with_pad:
        pk = pk.masked_fill(pad.cpu().t()[:, :, None, None], 0.0)
    att = O.causal_forward_chunked(pq.reshape(T, B * H, 2 * D), pk.reshape(T, B * H, 2 * D), v.reshape(T, B * H, d))
    want = att.reshape(T, B, E) @ P["out_proj.weight"].t() + P["out_proj.bias"]
    assert (y_f.double() - want.detach()).abs().max().item() <= 1e-2
    want.backward(go.double().cpu())
    ref = {"x": x.grad, **{n: p.grad for n, p in P.items()}}
    for name in ref:
        assert rel(g_f[name].double(), ref[name]) <= 2e-2, (name, rel(g_f[name].double(), ref[name]))


@pytest.mark.parametrize("R,Eo,Ei,n", [(8192, 512, 512, 3), (300, 256, 512, 2), (70, 768, 256, 1), (200, 128, 256, 1), (1, 128, 128, 2), (4097, 256, 128, 3),
                                       (64, 384, 128, 1)])
def test_linear_weight_and_bias_gradients(R, Eo, Ei, n):
    """dW = dy^T x and db = column sums against fp64; fp16 outputs of fp32 sums: <= 1.5e-3 relative
    to max(1, |value|) per element, and <= 1e-3 relative Frobenius error."""
    from rfa_amd import rfa_hip
    x = (_randn(R, Ei, seed=970 + R) * 0.5).half()
    dys = [(_randn(R, Eo, seed=971 + p) * 0.05).half() for p in range(n)]
    want_bias = [p != 1 for p in range(n)]
    print(f"weight grad R={R} Eo={Eo} Ei={Ei} n={n}", flush=True)
    dws, dbs = rfa_hip.linear_weight_grad(x.cuda(), [d.cuda() for d in dys], want_bias)
    for p in range(n):
        ww = dys[p].double().t() @ x.double()
        got = dws[p].double().cpu()
        assert ((got - ww).abs() <= 1.5e-3 * ww.abs().clamp_min(1.0)).all(), (p, (got - ww).abs().max().item())
        assert ((got - ww).norm() / ww.norm()).item() <= 1e-3
        if want_bias[p]:
            wb = dys[p].double().sum(0)
            gb = dbs[p].double().cpu()
            assert ((gb - wb).abs() <= 1.5e-3 * wb.abs().clamp_min(1.0)).all()
        else:
            assert dbs[p] is None
    with pytest.raises(ValueError):
        rfa_hip.linear_weight_grad(x[:, :64].contiguous().cuda(), [d.cuda() for d in dys], want_bias)


# the ring of 32-row steps: one step (ragged), the ring's depth and one around it, the first row counts with a
# second split, a last split of a single ragged step
@pytest.mark.parametrize("R", [1, 31, 32, 33, 64, 95, 97, 1023, 1024, 1025, 1057, 1569])
def test_linear_weight_gradient_step_edges(R):
    """dW and db exactly (whole numbers: every product and sum is exact in fp32, every result below 2048)."""
    from rfa_amd import rfa_hip
    g = torch.Generator().manual_seed(990 + R)
    x = torch.randint(-1, 2, (R, 128), generator=g).half()
    dy = (torch.randint(-1, 2, (R, 256), generator=g)).half()
    (dw,), (db,) = rfa_hip.linear_weight_grad(x.cuda(), [dy.cuda()], [True])
    assert torch.equal(dw.double().cpu(), dy.double().t() @ x.double())
    assert torch.equal(db.double().cpu(), dy.double().sum(0))


@pytest.mark.parametrize("R", [1, 31, 33, 98, 1025, 8191])
def test_linear_weight_gradient_of_an_infinity_in_the_last_row(R):
    """Rows past the ragged end count for nothing, also where the last row, which stands in for them, holds an infinity:
    its column of dW is infinite with the sign of dy, as the product gives it, and the others are exact."""
    from rfa_amd import rfa_hip
    g = torch.Generator().manual_seed(R)
    x = torch.randint(-1, 2, (R, 128), generator=g).half()
    dy = (2 * torch.randint(0, 2, (R, 128), generator=g) - 1).half()
    want = dy.double().t() @ x.double()
    x[-1, 5], x[-1, 77] = float("inf"), float("-inf")
    want[:, 5], want[:, 77] = dy[-1].double() * float("inf"), dy[-1].double() * float("-inf")
    (dw,), _ = rfa_hip.linear_weight_grad(x.cuda(), [dy.cuda()], [False])
    assert torch.equal(dw.double().cpu(), want)


@pytest.mark.parametrize("wide_input", [True, False])
def test_linear_weight_gradient_wider_than_32_bit_offsets(wide_input):
    """The rows of a step (32) of a matrix 69 * 2^20 wide span more than 4 GiB: dW and db exactly (whole numbers)."""
    from rfa_amd import rfa_hip
    E, R = 69 << 20, 33
    gen = torch.Generator("cuda").manual_seed(69)
    print(f"wide weight gradient, wide_input={wide_input}", flush=True)
    big = torch.randint(-1, 2, (R, E), generator=gen, device="cuda", dtype=torch.int8).half()
    small = torch.randint(-1, 2, (R, 128), generator=gen, device="cuda", dtype=torch.int8).half()
    x, dy = (big, small) if wide_input else (small, big)
    (dw,), (db,) = rfa_hip.linear_weight_grad(x, [dy], [True])
    assert torch.equal(db, dy.float().sum(0).half())
    for c in range(0, E, 3 << 20):
        cut = slice(c, c + (3 << 20))
        if wide_input:
            assert torch.equal(dw[:, cut], (dy.float().t() @ x[:, cut].float()).half())
        else:
            assert torch.equal(dw[cut], (dy[:, cut].t().float() @ x.float()).half())


@pytest.mark.parametrize("R", [98, 128, 129, 257, 449, 600, 2000])
@pytest.mark.parametrize("e_out,e_in,n", [(128, 128, 1), (256, 384, 2), (512, 512, 3)])
def test_linear_weight_gradient_of_few_rows(R, e_out, e_in, n):
    """A few hundred rows split by the root of their steps, down to two steps and a last one of a single row: dW and
    db exactly (whole numbers)."""
    from rfa_amd import rfa_hip
    g = torch.Generator().manual_seed(R + n)
    x = torch.randint(-1, 2, (R, e_in), generator=g).half()
    dys = [torch.randint(-1, 2, (R, e_out), generator=g).half() for _ in range(n)]
    dws, dbs = rfa_hip.linear_weight_grad(x.cuda(), [dy.cuda() for dy in dys], [True] * n)
    for dy, dw, db in zip(dys, dws, dbs):
        assert torch.equal(dw.double().cpu(), dy.double().t() @ x.double())
        assert torch.equal(db.double().cpu(), dy.double().sum(0))


def test_cross_modules_fused_projections_match_unfused_chain():
    """CrossAttentionProjectLayer + CrossAttention with their projections on the fused launch vs
    the same modules on nn.Linear + random_project: output within 4e-3, gradients within 1e-2."""
    from rfa_amd import CrossAttention, CrossAttentionProjectLayer
    torch.manual_seed(6)
    S, T, B, E, H, d, D = 150, 70, 2, 256, 4, 64, 64
    proj = CrossAttentionProjectLayer(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
    att = CrossAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
    with torch.no_grad():
        proj.sigma.mul_(1.0 + 0.1 * torch.randn_like(proj.sigma))
        att.q_proj.bias.normal_(0, 0.1)
    W = O.make_w(d, D, H).cuda().half()
    enc0 = (torch.randn(S, B, E) * 0.7).half()
    q0 = (torch.randn(T, B, E) * 0.7).half()
    go = torch.randn(T, B, E).half().cuda()
    mask = torch.zeros(S, B, 1, 1, dtype=torch.bool)
    mask[120:, 1] = True
    mask = mask.cuda()

    def run(fused):
        proj.fuse_projections = att.fuse_projections = fused
        proj.zero_grad(set_to_none=True)
        att.zero_grad(set_to_none=True)
        enc = enc0.clone().cuda().requires_grad_(True)
        q = q0.clone().cuda().requires_grad_(True)
        y = att(q, proj(encoder_output=enc, random_matrices=W, mask=mask))
        y.backward(go)
        grads = {"enc": enc.grad, "q": q.grad}
        grads.update({"proj." + n: p.grad for n, p in proj.named_parameters()})
        grads.update({"att." + n: p.grad for n, p in att.named_parameters()})
        return y.detach().float().cpu(), {k: v.float().cpu() for k, v in grads.items()}

    y_f, g_f = run(True)
    y_u, g_u = run(False)
    assert (y_f - y_u).abs().max().item() <= 4e-3
    for name in g_u:
        r = ((g_f[name] - g_u[name]).norm() / g_u[name].norm().clamp_min(1e-30)).item()
        assert torch.isfinite(g_f[name]).all() and r <= 1e-2, (name, r)


def test_module_step_replays_from_a_hip_graph():
    """Forward + backward of CausalAttention captured once and replayed: every replay, with eager
    steps and synchronisations in between, gives bit-identical output and gradients to the eager step."""
    from rfa_amd import CausalAttention
    torch.manual_seed(7)
    T, B, E, H, d, D = 320, 2, 256, 4, 64, 64
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
    W = O.make_w(d, D, H).cuda().half()
    x = (torch.randn(T, B, E) * 0.6).half().cuda().requires_grad_(True)
    go = torch.randn(T, B, E).half().cuda()

    def step():
        m.zero_grad(set_to_none=True)
        x.grad = None
        y = m(x, W)
        y.backward(go)
        return y

    y_e = step().detach().clone()
    want = {"x": x.grad.detach().clone(), **{n: p.grad.detach().clone() for n, p in m.named_parameters()}}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    m.zero_grad(set_to_none=True)
    x.grad = None
    with torch.cuda.graph(graph):
        y_g = m(x, W)
        y_g.backward(go)
    captured = {"x": x.grad, **{n: p.grad for n, p in m.named_parameters()}}   # the graph's output buffers
    for rep in range(3):
        for t in captured.values():
            t.zero_()
        y_g.detach().zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y_g, y_e), rep
        for name, t in captured.items():
            assert torch.equal(t, want[name]), (rep, name)
        # eager work between the replays; it rebinds .grad, the graph keeps writing its own buffers
        grads_before = {k: v for k, v in captured.items()}
        step()
        torch.cuda.synchronize()
        captured = grads_before


def test_projection_backward_on_the_packed_gradient(monkeypatch):
    """q, k through the feature map and v plain: the backward that forms [dy_q | dy_k | dv] in one
    matrix (one GEMM for dx, one contraction for the three dW) against the one with a GEMM per
    projection.  dW, db and dW' carry the same bits (the same row-split sums); dx is one sum of 3E
    products in place of three rounded partial sums."""
    from rfa_amd import projection
    torch.manual_seed(11)
    L, B, E, H, d, D = 130, 3, 256, 4, 64, 64
    layers = [torch.nn.Linear(E, H * d).cuda().half() for _ in range(3)]
    layers[1].bias = None
    wf = (torch.randn(H, D, d) * 0.9).half().cuda().requires_grad_(True)
    x = (torch.randn(L, B, E) * 0.7).half().cuda().requires_grad_(True)
    gs = [torch.randn(L, B, H, 2 * D).half().cuda(), torch.randn(L, B, H, 2 * D).half().cuda(),
          torch.randn(L, B, H, d).half().cuda()]

    def run():
        for t in [x, wf] + [p for l in layers for p in l.parameters()]:
            t.grad = None
        outs = projection.project_heads(x, layers, [True, True, False], H, wf, O.SCALE)
        torch.autograd.backward(outs, gs)
        return [x.grad.clone(), wf.grad.clone()] + [p.grad.clone() for l in layers for p in l.parameters()]

    used = []
    real = projection.rfa_hip.feature_map_backward_pair_packed
    monkeypatch.setattr(projection.rfa_hip, "feature_map_backward_pair_packed",
                        lambda *a, **kw: (used.append(1), real(*a, **kw))[1])
    print("projection backward, packed gradient", flush=True)
    packed = run()
    assert used, "the packed path was not taken"
    key = tuple(id(l.weight) for l in layers)           # the stack of the weights is kept between eager steps ...
    stack = projection._STACKED[key].value
    again = run()
    assert projection._STACKED[key].value is stack and all(torch.equal(a, b) for a, b in zip(packed, again))
    with torch.no_grad():
        layers[2].weight.mul_(1.5)                      # ... until a weight changes
    changed = run()
    assert projection._STACKED[key].value is not stack and not torch.equal(changed[0], packed[0])
    with torch.no_grad():
        layers[2].weight.div_(1.5)                      # exact in fp16
    used.clear()
    packed = run()
    monkeypatch.setattr(projection, "_packed_backward_ok", lambda *a: False)
    plain = run()
    assert len(used) == 1 and len(packed) == len(plain) == 2 + 5
    scale = plain[0].float().abs().max().item()
    assert (packed[0].float() - plain[0].float()).abs().max().item() <= 4e-3 * scale
    for a, b in zip(packed[1:], plain[1:]):
        assert torch.equal(a, b)


def test_packed_backward_in_a_graph_follows_weight_updates():
    """The stacked weights [Wq; Wk; Wv] of the packed backward are kept between eager steps but
    formed inside a captured graph: a replay after an in-place weight update gives the eager
    gradients of the updated weights."""
    from rfa_amd import CausalAttention
    torch.manual_seed(13)
    T, B, E, H, d, D = 192, 2, 256, 4, 64, 64
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
    W = O.make_w(d, D, H).cuda().half()
    x = (torch.randn(T, B, E) * 0.6).half().cuda().requires_grad_(True)
    go = torch.randn(T, B, E).half().cuda()

    def step():
        m.zero_grad(set_to_none=True)
        x.grad = None
        m(x, W).backward(go)
        return x.grad.detach().clone()

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()                      # also fills the eager cache of the stacked weights
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    m.zero_grad(set_to_none=True)
    x.grad = None
    print("packed backward: capture", flush=True)
    with torch.cuda.graph(graph):
        m(x, W).backward(go)
    gx = x.grad
    for rep in range(3):
        with torch.no_grad():
            for p in (m.q_proj.weight, m.k_proj.weight, m.v_proj.weight):
                p.mul_(1.0 + 0.25 * (rep + 1))
        gx.zero_()
        torch.cuda.synchronize()
        print(f"packed backward: replay {rep}", flush=True)
        graph.replay()
        torch.cuda.synchronize()
        got = gx.clone()
        want = step()                   # eager, on the updated weights (rebinds x.grad; the graph keeps gx)
        torch.cuda.synchronize()
        assert torch.equal(got, want), rep


def test_empty_input():
    """No rows: the projections come back empty, the weight and bias gradients as zeros."""
    from rfa_amd import rfa_hip
    H, d, D, E = 2, 64, 64, 128
    x = torch.empty(0, 3, E, dtype=torch.float16).cuda()
    ws = [torch.randn(H * d, E).half().cuda() for _ in range(2)]
    wf = torch.randn(H, D, d).half().cuda()
    ys, phis = rfa_hip.project_feature_map(x, ws, [None, None], [True, False], wf, H, O.SCALE)
    assert ys[0].shape == (0, 3, H, d) and phis[0].shape == (0, 3, H, 2 * D) and phis[1] is None
    dws, dbs = rfa_hip.linear_weight_grad(x.view(0, E), [torch.empty(0, H * d, dtype=torch.float16).cuda()], [True])
    assert dws[0].shape == (H * d, E) and (dws[0] == 0).all() and (dbs[0] == 0).all()


@pytest.mark.parametrize("e_in,e_out", [(32, 16), (96, 48), (512, 1536), (992, 272), (1024, 3072)])
@pytest.mark.parametrize("R", [1, 15, 16, 17, 32, 33, 64, 65, 97, 130, 700, 3000])
def test_linear_rows(R, e_in, e_out):
    """The products without autograd against fp64, few rows at the edges of the row tiles, column tiles and wave
    splits of their kernel, more by the projection kernel: fp32
    sums of exact products, one rounding to fp16 (2^-11 of the value; sums of 1024 terms below 2^-16)."""
    from rfa_amd import projection, rfa_hip
    if rfa_hip.native is None:
        pytest.skip("the torch binding is not active")
    gen = torch.Generator("cuda").manual_seed(R)
    x = torch.randn(R, e_in, generator=gen, device="cuda").half()
    w = (torch.randn(e_out, e_in, generator=gen, device="cuda") / e_in ** 0.5).half()
    b = torch.randn(e_out, generator=gen, device="cuda").half()
    print(f"linear_rows R={R} {e_in}->{e_out}", flush=True)
    want = x.double() @ w.double().t()
    with torch.no_grad():
        for bias in (b, None):
            y = projection.linear_rows(x, w, bias)
            ref = want if bias is None else want + b.double()
            if R * e_in * e_out > 1 << 31 or (R > 256 and (e_in % 64 or e_out % 64)):
                assert y is None        # the library's
                continue
            assert ((y.double() - ref).abs() <= 2.0 ** -10 * ref.abs() + 2e-5).all()
        # what the kernel does not read as it is goes to the library
        assert projection.linear_rows(x.t().contiguous().t() if R > 1 else x.float(), w, b) is None
        assert projection.linear_rows(x, w[:, :e_in - 8], b) is None and projection.linear_rows(x.float(), w.float(), None) is None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert projection.linear_rows(x, w, b) is None
    assert projection.linear_rows(x, w, b) is None          # autograd is on


@pytest.mark.parametrize("R,e_in,e_out", [(1024, 512, 512), (1025, 512, 512), (320, 512, 1536), (321, 512, 1536), (512, 1024, 1024),
                                          (513, 1024, 1024), (129, 1024, 3072), (16, 2048, 6144), (32, 2080, 48), (33, 2048, 2048),
                                          (7, 160, 16), (19, 288, 32), (64, 992, 272)])
def test_linear_rows_where_the_choice_changes(R, e_in, e_out):
    """Both sides of one workgroup per CU and of the widest contraction, and contractions that end in a ragged batch of
    steps for one or more of the four waves, whose columns of W past the end are not numbers: against fp64."""
    from rfa_amd import projection, rfa_hip
    if rfa_hip.native is None:
        pytest.skip("the torch binding is not active")
    gen = torch.Generator("cuda").manual_seed(R)
    x = torch.randn(R, e_in, generator=gen, device="cuda").half()
    w = torch.full((e_out + 1, e_in), float("nan"), device="cuda", dtype=torch.float16)[:e_out]
    w.copy_(torch.randn(e_out, e_in, generator=gen, device="cuda") / e_in ** 0.5)
    b = torch.randn(e_out, generator=gen, device="cuda").half()
    print(f"linear_rows where the choice changes R={R} {e_in}->{e_out}", flush=True)
    with torch.no_grad():
        y = projection.linear_rows(x, w, b)
    if R > 32 and e_in > 1024:
        assert y is None        # the library's
        return
    want = x.double() @ w.double().t() + b.double()
    assert ((y.double() - want).abs() <= 2.0 ** -10 * want.abs() + 2e-5).all()


@pytest.mark.parametrize("e_in,e_out", [(512, 512), (512, 1536), (1024, 1024), (1024, 3072), (160, 48)])
def test_linear_rows_are_the_same_in_every_tile(e_in, e_out):
    """The tile goes by rounds of workgroups; every tile adds a row's products in one order, so a row has the same bits
    whatever rows it comes with: one at a time (16 x 16) against counts that take each tile, with rows past the last one."""
    from rfa_amd import projection, rfa_hip
    if rfa_hip.native is None:
        pytest.skip("the torch binding is not active")
    gen = torch.Generator("cuda").manual_seed(e_out)
    x = torch.randn(256, e_in, generator=gen, device="cuda").half()
    w = (torch.randn(e_out, e_in, generator=gen, device="cuda") / e_in ** 0.5).half()
    b = torch.randn(e_out, generator=gen, device="cuda").half()
    print(f"linear_rows in every tile {e_in}->{e_out}", flush=True)
    with torch.no_grad():
        one = [projection.linear_rows(x[r:r + 1], w, b) for r in (0, 17, 40)]
        for R in (41, 64, 79, 128, 160, 256):
            y = projection.linear_rows(x[:R], w, b)
            if -(-R // 64) * -(-e_out // 32) > torch.cuda.get_device_properties(0).multi_processor_count:
                continue                                     # another kernel's
            assert all(torch.equal(y[r:r + 1], o) for r, o in zip((0, 17, 40), one)), R


@pytest.mark.parametrize("e_in,e_out", [(32, 16), (160, 48), (512, 512), (1024, 1024), (512, 2064)])
@pytest.mark.parametrize("R", [1, 17, 64, 160])
def test_linear_rows_of_several_layers(R, e_in, e_out):
    """Layers side by side from where they are: the bits of one call over their stack, at widths where a tile of 32 columns
    spans two layers, with and without a bias."""
    import ctypes
    from rfa_amd import _lib
    lib = _lib.load()
    gen = torch.Generator("cuda").manual_seed(R + e_out)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").half()
    x, ws, bs = rand(R, e_in), [rand(e_out, e_in) for _ in range(3)], [rand(e_out) for _ in range(3)]
    stream = torch.cuda.current_stream().cuda_stream
    array = lambda ts: (ctypes.c_void_p * len(ts))(*[None if t is None else t.data_ptr() for t in ts])
    print(f"linear_rows_layers R={R} {e_in}->{e_out}", flush=True)
    for n in (1, 2, 3):
        for biases in (bs[:n], [None] * n, [bs[0]] + [None] * (n - 1)):
            got, want = (torch.full((R, n * e_out), float("nan"), device="cuda").half() for _ in range(2))
            stack = torch.cat(ws[:n], 0)
            bias = torch.cat([torch.zeros_like(bs[0]) if b is None else b for b in biases], 0)
            _lib.check(lib.rfa_linear_rows_layers(x.data_ptr(), array(ws[:n]), array(biases), n, got.data_ptr(), R, e_in, e_out, stream))
            _lib.check(lib.rfa_linear_rows(x.data_ptr(), stack.data_ptr(), bias.data_ptr(), want.data_ptr(), R, e_in, n * e_out, stream))
            assert torch.equal(got, want), (n, len(biases))
    _lib.check(lib.rfa_linear_rows_layers(x.data_ptr(), array(ws), None, 3, got.data_ptr(), R, e_in, e_out, stream))
    assert lib.rfa_linear_rows_layers(x.data_ptr(), array(ws), None, 4, got.data_ptr(), R, e_in, e_out, stream) == -2
    assert lib.rfa_linear_rows_layers(x.data_ptr(), array([ws[0], None]), None, 2, got.data_ptr(), R, e_in, e_out, stream) == -1


@pytest.mark.parametrize("e_in", [(1 << 22) + 128, (1 << 25) + 128])
def test_output_projection_wider_than_the_kernels_address(e_in):
    """Widths that the input-gradient launch (2^22) and the projection launch (2^25) refuse go to the library."""
    from rfa_amd import projection
    layer = torch.nn.Linear(128, 128, device="cuda", dtype=torch.float16)
    layer.weight = torch.nn.Parameter(torch.randn(128, e_in, device="cuda", dtype=torch.float16).mul_(e_in ** -0.5))
    x = torch.randn(1, e_in, device="cuda", dtype=torch.float16).requires_grad_()
    print(f"linear_out {e_in} -> 128", flush=True)
    y = projection.linear_out(x, layer)
    cut = [slice(c, c + (1 << 22)) for c in range(0, e_in, 1 << 22)]
    want = sum(x.detach()[:, c].double() @ layer.weight.detach()[:, c].double().t() for c in cut) + layer.bias.detach().double()
    assert _rel(y.detach().double(), want) <= 2.0 ** -10      # one rounding, fp32 sums of 2^25 terms of either sign
    if e_in < 1 << 25:
        dy = torch.randn_like(y)
        y.backward(dy)
        assert _rel(x.grad.double(), dy.double() @ layer.weight.detach().double()) <= 2.0 ** -11
    odd = torch.nn.Linear(64, 64, device="cuda", dtype=torch.float16)
    odd.weight = torch.nn.Parameter(torch.zeros(1, e_in - 64, device="cuda", dtype=torch.float16).expand(64, e_in - 64))
    assert projection.fused_projection_supported(x.detach()[None, :, 64:], [odd], 1) == (e_in - 64 <= 1 << 25)


@pytest.mark.parametrize("bias", [True, False])
def test_output_projection_differentiated_twice(bias):
    """The input gradient of the output layer under create_graph is itself differentiable (a gradient penalty):
    d/dW and d/dx of the sum of dx . r, where dx is the gradient of |x W^T + b|^2 / 2, against fp64."""
    from rfa_amd import projection
    torch.manual_seed(3)
    layer = torch.nn.Linear(128, 256, bias=bias).cuda().half()
    x, r = (torch.randn(37, 128, device="cuda").half() for _ in range(2))

    def second(x, weight, b, forward):
        x = x.detach().requires_grad_()
        y = forward(x)
        (dx,) = torch.autograd.grad(y, x, y, create_graph=True)
        return [dx] + list(torch.autograd.grad((dx * r.to(dx.dtype)).sum(), [weight, x]))

    got = second(x, layer.weight, layer.bias, lambda t: projection.linear_out(t, layer))
    w = layer.weight.detach().double().requires_grad_()
    b = layer.bias.detach().double() if bias else None
    want = second(x.double(), w, b, lambda t: torch.nn.functional.linear(t, w, b))
    for a, ref in zip(got, want):       # a few roundings to fp16, sums of up to 256 products of such terms
        assert _rel(a.double(), ref) <= 4 * 2.0 ** -11


def test_output_projection_keeps_its_hooks():
    """Without autograd the output layer may take the row kernel, but not past hooks or a forward of its own."""
    from rfa_amd import projection
    layer = torch.nn.Linear(64, 64).cuda().half()
    x = torch.randn(3, 64).cuda().half()
    seen = []
    with torch.no_grad():
        plain = projection.linear_out(x, layer)
        handle = layer.register_forward_hook(lambda *a: seen.append(1))
        assert torch.allclose(projection.linear_out(x, layer), plain, atol=2e-3) and seen == [1]
        handle.remove()
        layer.forward = lambda t: t * 0
        assert projection.linear_out(x, layer).abs().max().item() == 0


@pytest.mark.parametrize("e_out,e_in,n", [(32, 128, 1), (96, 128, 2), (128, 256, 3), (512, 512, 3), (64, 384, 2)])
@pytest.mark.parametrize("R", [1, 15, 63, 64, 65, 129, 257, 1000, 20000])
def test_linear_input_grad(R, e_out, e_in, n):
    """dx = sum_p dy_p W_p over the blocks of a packed gradient, at the edges of its row tiles (64, 128 and
    256 rows), against fp64: exact products, fp32 sums (a share 2^-20 of the sum of their magnitudes covers
    the order of up to 1536 of them) and one rounding to fp16."""
    import ctypes
    from rfa_amd import _lib
    gen = torch.Generator("cuda").manual_seed(R + e_out)
    dy = torch.randn(R, n * e_out, generator=gen, device="cuda").half()
    ws = [(torch.randn(e_out, e_in, generator=gen, device="cuda") / e_out ** 0.5).half() for _ in range(n)]
    dx = torch.full((R, e_in), float("nan"), dtype=torch.float16, device="cuda")
    array = lambda ptrs: (ctypes.c_void_p * n)(*ptrs)
    print(f"linear_input_grad R={R} {e_out}->{e_in} x {n}", flush=True)
    _lib.check(_lib.load().rfa_linear_input_grad(array([dy.data_ptr() + 2 * p * e_out for p in range(n)]), n * e_out,
                                                 array([w.data_ptr() for w in ws]), n, dx.data_ptr(), R, e_out, e_in,
                                                 torch.cuda.current_stream().cuda_stream))
    W = torch.cat(ws, 0).double()
    want, size = dy.double() @ W, dy.double().abs() @ W.abs()
    assert ((dx.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -20 * size + 2.0 ** -24).all()


@pytest.mark.parametrize("e_out", [32, 96, 128])
def test_linear_input_grad_of_a_tile_per_compute_unit(e_out):
    """As many columns as give every compute unit one tile, where widths that two groups of waves divide and others part."""
    test_linear_input_grad(50, e_out, 128 * torch.cuda.get_device_properties(0).multi_processor_count, 2)


@pytest.mark.parametrize("e_out,e_in,n", [(128, 128, 1), (128, 256, 3), (384, 128, 2), (512, 512, 3), (1024, 1024, 1)])
@pytest.mark.parametrize("R", [1, 31, 33, 64, 65, 200, 1000, 2049, 9000])
def test_linear_grads(R, e_out, e_in, n):
    """dx, dW and db from one launch over the blocks of a packed gradient, in every tile shape that the plan takes, against
    fp64: exact products, fp32 sums (a share 2^-20 of the sum of their magnitudes covers the order) and one rounding to
    fp16.  The last row holds an infinity in x: where rows past the end read it, nothing of it may show up."""
    import ctypes
    from rfa_amd import _lib
    lib = _lib.load()
    need = lib.rfa_linear_grads_workspace_bytes(R, e_out, e_in, n)
    assert need > 0
    gen = torch.Generator("cuda").manual_seed(R + e_out)
    x = torch.randn(R, e_in, generator=gen, device="cuda").half()
    x[-1, 5] = float("inf")
    dy = torch.randn(R, n * e_out, generator=gen, device="cuda").half()
    ws = [(torch.randn(e_out, e_in, generator=gen, device="cuda") / e_out ** 0.5).half() for _ in range(n)]
    new = lambda *shape: torch.full(shape, float("nan"), dtype=torch.float16, device="cuda")
    dx, dw, db = new(R, e_in), [new(e_out, e_in) for _ in range(n)], [new(e_out) for _ in range(n)]
    work = torch.empty(need, dtype=torch.uint8, device="cuda")
    array = lambda ptrs: (ctypes.c_void_p * n)(*ptrs)
    args = (x.data_ptr(), array([dy.data_ptr() + 2 * p * e_out for p in range(n)]), n * e_out, array([w.data_ptr() for w in ws]), n,
            dx.data_ptr(), array([w.data_ptr() for w in dw]), array([b.data_ptr() for b in db]), R, e_out, e_in, work.data_ptr())
    stream = torch.cuda.current_stream().cuda_stream
    print(f"linear_grads R={R} {e_out}->{e_in} x {n}", flush=True)
    _lib.check(lib.rfa_linear_grads(*args, need, stream))
    near = lambda got, want, size: ((got.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -20 * size + 2.0 ** -24).all()
    W = torch.cat(ws, 0).double()
    assert near(dx, dy.double() @ W, dy.double().abs() @ W.abs())
    keep = torch.arange(e_in, device="cuda") != 5
    for p in range(n):
        g = dy[:, p * e_out:(p + 1) * e_out].double()
        xk = x[:, keep].double()
        assert near(dw[p][:, keep], g.t() @ xk, g.t().abs() @ xk.abs()), p
        assert torch.isinf(dw[p][:, 5]).all() and (torch.sign(dw[p][:, 5]) == torch.sign(dy[-1, p * e_out:(p + 1) * e_out])).all()
        assert near(db[p], g.sum(0), g.abs().sum(0)), p
    assert lib.rfa_linear_grads(*args, need - 1, stream) == -5              # the workspace is checked
    assert lib.rfa_linear_grads_workspace_bytes(R, e_out + 64, e_in, n) == 0
    assert lib.rfa_linear_grads_workspace_bytes(1 << 20, e_out, e_in, n) == 0


@pytest.mark.parametrize("H,D,d,e_in,n,nphi", [(2, 64, 64, 128, 3, 2), (8, 64, 64, 512, 2, 1), (1, 128, 128, 256, 1, 1),
                                               (4, 32, 64, 128, 2, 2), (2, 64, 128, 256, 3, 1)])
@pytest.mark.parametrize("R", [1, 65, 300, 2049])
def test_project_grads(R, H, D, d, e_in, n, nphi):
    """Layers and the feature map behind the first of them, with one reduction for both: the bits of the calls of its parts."""
    import ctypes
    from rfa_amd import _lib
    lib = _lib.load()
    need = lib.rfa_project_grads_workspace_bytes(R, H, D, d, e_in, n, nphi)
    e_out = H * d
    assert need > 0
    gen = torch.Generator("cuda").manual_seed(R + e_in)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").half()
    new = lambda *shape: torch.full(shape, float("nan"), dtype=torch.float16, device="cuda")
    x, wf = rand(R, e_in), rand(H, D, d)
    y = [rand(R, e_out) for _ in range(nphi)]
    grad = [rand(R, 2 * H * D) for _ in range(nphi)] + [rand(R, e_out) for _ in range(n - nphi)]
    ws = [(rand(e_out, e_in) / e_out ** 0.5).half() for _ in range(n)]
    work = torch.empty(need, dtype=torch.uint8, device="cuda")
    array = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() if t is not None else None for t in ts])
    stream = torch.cuda.current_stream().cuda_stream
    print(f"project_grads R={R} H={H} D={D} d={d} E={e_in} layers={n} mapped={nphi}", flush=True)

    def whole(with_wf, with_bias, nbytes=need):
        dx, dw, dwf = new(R, e_in), [new(e_out, e_in) for _ in range(n)], new(H, D, d)
        db = [new(e_out) if with_bias else None for _ in range(n)]
        rc = lib.rfa_project_grads(x.data_ptr(), array(y), wf.data_ptr(), array(grad), array(ws), n, nphi, dx.data_ptr(), array(dw),
                                   array(db), dwf.data_ptr() if with_wf else None, R, H, D, d, e_in, 0.3, work.data_ptr(), nbytes,
                                   stream)
        return rc, dx, dw, db, dwf

    dy, dwf = [new(R, e_out) for _ in range(nphi)] + grad[nphi:], new(H, D, d)
    fbytes = 2 * lib.rfa_feature_map_backward_workspace_bytes(R, H, D, d)
    fwork = torch.empty(fbytes, dtype=torch.uint8, device="cuda")
    two = nphi == 2
    _lib.check(lib.rfa_feature_map_backward_half(
        y[0].data_ptr(), y[1].data_ptr() if two else None, wf.data_ptr(), grad[0].data_ptr(), grad[1].data_ptr() if two else None,
        None, dy[0].data_ptr(), dy[1].data_ptr() if two else None, None, dwf.data_ptr(), R, H, D, d, 0.3, fwork.data_ptr(), fbytes,
        stream))
    lbytes = lib.rfa_linear_grads_workspace_bytes(R, e_out, e_in, n)
    lwork = torch.empty(lbytes, dtype=torch.uint8, device="cuda")
    dx, dw, db = new(R, e_in), [new(e_out, e_in) for _ in range(n)], [new(e_out) for _ in range(n)]
    _lib.check(lib.rfa_linear_grads(x.data_ptr(), array(dy), e_out, array(ws), n, dx.data_ptr(), array(dw), array(db), R, e_out, e_in,
                                    lwork.data_ptr(), lbytes, stream))
    for with_wf, with_bias in ((True, True), (False, True), (True, False)):
        rc, gx, gw, gb, gwf = whole(with_wf, with_bias)
        _lib.check(rc)
        assert torch.equal(gx, dx) and all(torch.equal(a, b) for a, b in zip(gw, dw))
        assert not with_bias or all(torch.equal(a, b) for a, b in zip(gb, db))
        assert torch.equal(gwf, dwf) if with_wf else torch.isnan(gwf).all()
    assert whole(True, True, need - 1)[0] == -5                             # the workspace is checked
    assert lib.rfa_project_grads_workspace_bytes(R, H, D, 96, e_in, n, nphi) == 0
    assert lib.rfa_project_grads_workspace_bytes(1 << 20, H, D, d, e_in, n, nphi) == 0
    assert lib.rfa_project_grads_workspace_bytes(R, H, D, d, e_in, n, n + 1) == 0
