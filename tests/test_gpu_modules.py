"""GPU tests of the host-side mirror of the reference API (autograd Functions and
nn.Modules) against the oracle chain evaluated in fp32 on the CPU."""
import pytest
import torch

from oracle import rfa_oracle as O

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a - b).norm() / b.norm().clamp_min(1e-30)).item()


def _randn(*shape, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g, dtype=torch.float32)


def test_rfa_apply_autograd_matches_oracle_grad_check_recipe():
    """The recipe of the reference's grad_check.py (T=100, 5 sequences, K=128, d=64,
    U(-.5,.5) inputs L2-normalised, seed 3) through RFA.apply + autograd."""
    from rfa_amd import RFA
    torch.manual_seed(3)
    T, N, K, d = 100, 5, 128, 64
    nrm = lambda t: t / t.norm(p=2, dim=-1, keepdim=True)
    q, k, v = (nrm(torch.rand(T, N, n) - .5).half() for n in (K, K, d))
    g = nrm(torch.rand(T, N, d)).half()
    cq, ck, cv = (t.cuda().requires_grad_(True) for t in (q, k, v))
    out = RFA.apply(cq, ck, cv)
    out.backward(g.cuda())
    ref = O.causal_forward_cumsum(q.float(), k.float(), v.float())
    rq, rk, rv = O.causal_backward_cumsum(q.float(), k.float(), v.float(), g.float())
    # the reference's own pass rule: squared difference below 1e-4 everywhere
    assert ((out.float().cpu() - ref) ** 2 < 1e-4).all()
    for got, want in ((cq.grad, rq), (ck.grad, rk), (cv.grad, rv)):
        assert ((got.float().cpu() - want) ** 2 < 1e-4).all()
        assert _rel(got.float().cpu(), want) < 1e-2
    # static-method spellings used by the reference's callers
    assert torch.equal(RFA.forward_cuda(cq.detach(), ck.detach(), cv.detach()), out.detach())


def test_rfa_forward_matches_oracle_grad_check_forward_recipe():
    """The forward recipe of the reference's grad_check.py (:17-28): T=50, one sequence, K=128, d=64,
    U(-.5,.5) inputs that are NOT normalised, seed 3, compared with forward_torch under the
    reference's own pass rule."""
    from rfa_amd import RFA
    torch.manual_seed(3)
    T, N, K, d = 50, 1, 128, 64
    q, k, v = ((torch.rand(T, N, n) - .5).half() for n in (K, K, d))
    ref = O.causal_forward_cumsum(q.float(), k.float(), v.float())
    cq, ck, cv = (t.cuda() for t in (q, k, v))
    out = RFA.forward_cuda(cq, ck, cv)
    assert ((out.float().cpu() - ref) ** 2 < 1e-4).all()
    # outputs reach |out| ~ 10 with these inputs, where one fp16 step is 7.8e-3, and the intra-chunk weights q.k (up to ~10 here) pass through fp16
    assert ((out.float().cpu() - ref).abs() <= 2e-3 * ref.abs().clamp_min(1.0)).all()
    # forward_torch, the formula the reference compares its kernel with, on the same device tensors
    assert ((RFA.forward_torch(cq.float(), ck.float(), cv.float()).cpu() - ref) ** 2 < 1e-4).all()


def test_functional_chain_with_padding_mask_and_grads():
    """random_project -> cuda_causal_rfa with a key padding mask, gradients down to the
    raw q, k, v and the random matrix."""
    from rfa_amd.causal_attention import cuda_causal_rfa
    from rfa_amd.utils import random_project
    T, B, H, d, D = 150, 2, 2, 64, 64
    q, k, v, g = (_randn(T, B, H, d, seed=s).half() for s in (1, 2, 3, 4))
    W = (_randn(H, D, d, seed=5)).half()
    mask = torch.zeros(B, T, dtype=torch.uint8)
    mask[0, 100:] = 1
    mask[1, :3] = 1
    cq, ck, cv, cW = (t.cuda().requires_grad_(True) for t in (q, k, v, W))
    attn = cuda_causal_rfa(phi_q=random_project(x=cq, random_matrices=cW),
                           phi_k=random_project(x=ck, random_matrices=cW), v=cv,
                           key_padding_mask=mask.cuda())
    attn.backward(g.reshape(T, B, H * d).cuda())
    fq, fk, fv, fW = (t.float().requires_grad_(True) for t in (q, k, v, W))
    pq, pk = O.random_project(fq, fW), O.random_project(fk, fW)
    pk = pk.masked_fill(mask.bool().t()[:, :, None, None], 0.0)
    ref = O.causal_forward_chunked(pq.reshape(T, B * H, 2 * D), pk.reshape(T, B * H, 2 * D), fv.reshape(T, B * H, d))
    ref.backward(g.float().reshape(T, B * H, d))
    assert (attn.float().cpu().reshape(T, B * H, d) - ref.detach()).abs().max() <= 2e-3
    for name, got, want in (("dq", cq.grad, fq.grad), ("dk", ck.grad, fk.grad), ("dv", cv.grad, fv.grad), ("dW", cW.grad, fW.grad)):
        assert _rel(got.float().cpu(), want) <= 2e-2, (name, _rel(got.float().cpu(), want))


def test_causal_module_decode_equals_training_forward():
    from rfa_amd import CausalAttention
    torch.manual_seed(0)
    T, B, E, H, d, D = 40, 3, 128, 2, 64, 64
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half().eval()
    with torch.no_grad():
        m.sigma.copy_(1.0 + 0.1 * torch.randn_like(m.sigma))
    x = torch.randn(T, B, E).cuda().half()
    W = O.make_w(d, D, H).cuda().half()
    with torch.no_grad():
        full = m(x, W)
        state = {}
        rows = [m(x[t:t + 1], W, saved_state=state) for t in range(T)]
    assert state["prev_s"].dtype == torch.float32 and tuple(state["prev_s"].shape) == (B, H, 2 * D, d)
    assert tuple(state["prev_z"].shape) == (B, H, 2 * D)
    step = torch.cat(rows, 0)
    assert (step.float() - full.float()).abs().max().item() <= 4e-3
    # quadratic fallback agrees wherever the denominators are equal (den >= 1 from a few steps on)
    m.cuda_causal_rfa = False
    with torch.no_grad():
        quad = m(x, W, attn_mask=torch.triu(torch.full((T, T), float("-inf")), 1).cuda())
    assert (quad[8:].float() - full[8:].float()).abs().max().item() <= 2e-2


def test_causal_module_decode_leaves_earlier_states_alone():
    """The reference builds a new state every step (causal_attention.py:42-43, 262): a tensor the
    caller holds from step t is unchanged after step t + 1.  decode_inplace = True advances the
    tensors where they are, with the same numbers."""
    from rfa_amd import CausalAttention
    torch.manual_seed(3)
    T, B, E, H, d, D = 6, 2, 128, 2, 64, 64
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half().eval()
    x = torch.randn(T, B, E).cuda().half()
    W = O.make_w(d, D, H).cuda().half()
    with torch.no_grad():
        state, held, rows = {}, [], []
        for t in range(T):
            rows.append(m(x[t:t + 1], W, saved_state=state))
            held.append((state["prev_s"], state["prev_z"], state["prev_s"].clone(), state["prev_z"].clone()))
        for s, z, s_then, z_then in held:
            assert torch.equal(s, s_then) and torch.equal(z, z_then)
        assert len({h[0].data_ptr() for h in held}) == T
        m.decode_inplace = True
        state2, rows2 = {}, []
        for t in range(T):
            rows2.append(m(x[t:t + 1], W, saved_state=state2))
            if t == 1:
                ptr = state2["prev_s"].data_ptr()
        assert state2["prev_s"].data_ptr() == ptr
        assert torch.equal(torch.cat(rows), torch.cat(rows2)) and torch.equal(state["prev_s"], state2["prev_s"])
        # a user-supplied fp16 state is converted (a private copy), never written
        half_state = {"prev_s": held[2][0].half(), "prev_z": held[2][1].half()}
        keep = half_state["prev_s"].clone()
        m(x[3:4], W, saved_state=half_state)
        assert half_state["prev_s"].dtype == torch.float32 and torch.equal(keep, held[2][0].half())


def test_causal_module_decode_from_one_stacked_projection():
    """Without autograd a decoding step takes q, k, v from one Linear layer whose weight stacks the
    three projections, and keeps that weight and the scaled random matrices between calls.  Same
    numbers as the step with three projections (one fp16 rounding of a projection apart); a
    parameter changed in place, or another random_matrices tensor, is seen by the next call."""
    from rfa_amd import CausalAttention, rfa_hip
    torch.manual_seed(5)
    T, B, E, H, d, D = 12, 3, 128, 2, 64, 64
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half().eval()
    x = torch.randn(T, B, E).cuda().half()
    W = O.make_w(d, D, H).cuda().half()
    calls = []
    real = rfa_hip.incremental_qkv

    def spy(*a, **kw):
        calls.append(1)
        return real(*a, **kw)
    rfa_hip.incremental_qkv = spy
    try:
        with torch.no_grad():
            state, rows = {}, []
            for t in range(T):
                rows.append(m(x[t:t + 1], W, saved_state=state))
        assert len(calls) == T - 1                      # the first token finds no state and takes the general path
        m.requires_grad_(True)
        state2, rows2 = {}, []
        for t in range(T):                              # autograd on: three projections, nothing cached
            rows2.append(m(x[t:t + 1], W, saved_state=state2).detach())
        assert len(calls) == T - 1
        a, b = torch.cat(rows).float(), torch.cat(rows2).float()
        assert (a - b).abs().max().item() <= 4e-3
        assert _rel(state["prev_s"], state2["prev_s"]) <= 2e-3
        with torch.no_grad():
            before = m(x[3:4], W, saved_state=dict(state))
            again = m(x[3:4], W, saved_state=dict(state))
            assert torch.equal(before, again)
            m.q_proj.weight.mul_(1.5)                   # in place: the version counter moves, the stacked weight is rebuilt
            changed = m(x[3:4], W, saved_state=dict(state))
            assert not torch.equal(before, changed)
            ref_state = dict(state)
            m.requires_grad_(True)
        with torch.enable_grad():
            want = m(x[3:4], W, saved_state=ref_state).detach()
        assert (changed.float() - want.float()).abs().max().item() <= 4e-3
        with torch.no_grad():
            other = m(x[3:4], (W * 0.5).contiguous(), saved_state=dict(state))      # another matrix tensor: W' rebuilt
            m.sigma.mul_(0.8)
            other2 = m(x[3:4], (W * 0.5).contiguous(), saved_state=dict(state))
        assert not torch.equal(other, changed) and not torch.equal(other2, other)
        # a module with a filled cache copies and pickles (the cache stays behind), and the copy decodes alike
        import copy
        import io
        assert m.__dict__.get("_inference_cache")
        twin = copy.deepcopy(m)
        buf = io.BytesIO()
        torch.save(m, buf)
        assert "_inference_cache" not in twin.__dict__
        with torch.no_grad():
            assert torch.equal(twin(x[3:4], (W * 0.5).contiguous(), saved_state=dict(state)), other2)
    finally:
        rfa_hip.incremental_qkv = real


def _decode_module(seed, B=3):
    """A CausalAttention that advances its state in place, its matrices, tokens and a state after two of them."""
    from rfa_amd import CausalAttention
    torch.manual_seed(seed)
    m = CausalAttention(embed_dim=128, num_heads=2, head_dim=64, proj_dim=64).cuda().half().eval()
    W, x = O.make_w(64, 64, 2).cuda().half(), torch.randn(8, B, 128).cuda().half()
    first = {}
    with torch.no_grad():
        m(x[:2], W, saved_state=first)
    m.decode_inplace = True
    m.__dict__.pop("_inference_cache", None)
    return m, W, x, first


@pytest.fixture(params=["ext", "ctypes"])
def decode_binding(request):
    from rfa_amd import rfa_hip
    if request.param == "ext" and not rfa_hip.ext_available():
        pytest.skip("the torch binding has not been built")
    before = rfa_hip.binding()
    rfa_hip.use_binding(request.param)
    yield request.param
    rfa_hip.use_binding(before)


@pytest.mark.parametrize("B", [3, 600])          # the layers where they are, a stack of them
@pytest.mark.parametrize("warm", [False, True])
def test_captured_decode_step_reads_the_parameters_of_the_day(warm, B, decode_binding):
    """A decoding step in a graph, captured before (nothing kept yet) or after eager steps: eager steps before the first
    replay, changes of every parameter between replays and eager steps that make the kept values anew leave each replay
    with the eager step's bits."""
    m, W, x, first = _decode_module(21, B)
    other, oW, ox, ofirst = _decode_module(22, B)
    copy_of = lambda: {k: t.clone() for k, t in first.items()}
    eager = lambda t: m(x[t:t + 1], W, saved_state=copy_of())
    with torch.no_grad():
        other(ox[2:3], oW, saved_state={k: t.clone() for k, t in ofirst.items()})        # loads the kernels, fills its own cache
        if warm:
            eager(2)
        state, token, graph = copy_of(), x[2:3].clone(), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        print(f"decode capture {decode_binding} B={B} warm={warm}", flush=True)
        with torch.cuda.graph(graph):
            out = m(token, W, saved_state=state)
        assert state["prev_s"] is not first["prev_s"]
        want = eager(2)                                            # before any replay
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        for t, change in enumerate([m.q_proj.weight, m.k_proj.bias, m.v_proj.weight, m.out_proj.weight, m.sigma, W], 2):
            change.mul_(0.75)
            want = eager(t)                                        # what was kept is replaced and given back
            junk = [torch.full((384, 128), float("nan"), device="cuda").half() for _ in range(8)]
            del junk
            token.copy_(x[t:t + 1])
            for key in first:
                state[key].copy_(first[key])
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), t


@pytest.mark.parametrize("B", [3, 600])
def test_decode_steps_on_several_streams(B, decode_binding):
    """Each stream decodes with values that it made itself, also when there are more streams than values are kept for, and
    when a parameter changes in between."""
    m, W, x, first = _decode_module(23, B)
    copy_of = lambda: {k: t.clone() for k, t in first.items()}
    streams = [torch.cuda.current_stream()] + [torch.cuda.Stream() for _ in range(5)]
    with torch.no_grad():
        for round_ in range(3):
            got = []
            for s in streams + streams[::-1]:
                s.wait_stream(torch.cuda.default_stream())
                with torch.cuda.stream(s):
                    got.append(m(x[2:3], W, saved_state=copy_of()))
            torch.cuda.synchronize()
            assert all(torch.equal(g, got[0]) for g in got)
            m.q_proj.weight.mul_(0.5)
            assert round_ == 0 or not torch.equal(got[0], last)
            last = got[0]
    if decode_binding == "ctypes":
        assert len(m._inference_cache["derived"]) <= 8


@pytest.mark.parametrize("change", ["none", "replaced", "data", "in_place", "no_bias", "mixed_bias", "matrices", "tau", "sigma", "hook",
                                    "steps", "strided", "transposed", "matrices_transposed"])
def test_decode_step_sees_every_change(change):
    """A decoding step after one that filled the caches gives what a module without caches gives, whatever changed
    in between; the layers it is compared with run under autograd (nothing cached, three projections: a rounding of
    fp16 apart)."""
    import copy
    from rfa_amd import CausalAttention, rfa_hip
    torch.manual_seed(11)
    B, H, d, D = 3, 2, 64, 64
    E = H * d
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half().eval()
    W, x = O.make_w(d, D, H).cuda().half(), torch.randn(4, B, E).cuda().half()
    with torch.no_grad():
        first = {}
        m(x[:2], W, saved_state=first)
        m(x[2:3], W, saved_state=dict(first))                       # fills the caches
    seen, now, answered = [], x[3:4], []
    if rfa_hip.native is not None:                                   # and the native step is the one that answers below
        step = m._inference_cache["step"]

        class Spy:
            def rows(self, *args):
                rows = step.rows(*args)
                answered.append(rows is not None)
                return rows
        m._inference_cache["step"] = Spy()
    with torch.no_grad():
        if change == "replaced":
            m.k_proj = copy.deepcopy(m.k_proj)
            m.k_proj.weight.mul_(0.5)
        elif change == "data":
            m.v_proj.weight.data = m.v_proj.weight.data * 0.5
        elif change == "transposed":             # same object, version, address and shape
            m.q_proj.weight.data = m.q_proj.weight.data.t()
        elif change == "matrices_transposed":
            W.data = W.data.transpose(1, 2)
        elif change == "in_place":
            m.q_proj.bias.add_(0.5)
        elif change in ("no_bias", "mixed_bias"):
            for layer in (m.q_proj, m.k_proj, m.v_proj)[:3 if change == "no_bias" else 1]:
                layer.bias = None
        elif change == "matrices":
            W = W * 0.5
        elif change == "tau":
            m.tau = 2
        elif change == "sigma":
            m.sigma.mul_(0.7)
        elif change == "hook":
            m.out_proj.register_forward_hook(lambda mod, args, out: seen.append(1) or out * 2)
        elif change == "steps":
            now = x[2:4]
        elif change == "strided":
            now = torch.randn(1, E, B).cuda().half().transpose(1, 2)
        got_state, ref_state = dict(first), dict(first)
        got = m(now, W, saved_state=got_state)
    assert answered == ([] if rfa_hip.native is None else [change != "mixed_bias"])
    m.requires_grad_(True)
    with torch.enable_grad():
        want = m(now, W, saved_state=ref_state).detach()
    if change == "hook":            # called without autograd; a layer in training is one node
        assert len(seen) == 1
        got = got / 2
    assert (got.float() - want.float()).abs().max().item() <= 4e-3
    for key in ("prev_s", "prev_z"):
        assert _rel(got_state[key], ref_state[key]) <= 2e-3, key


def test_causal_module_training_step_runs_and_matches_oracle():
    from rfa_amd import CausalAttention
    torch.manual_seed(1)
    T, B, E, H, d, D = 96, 2, 128, 2, 64, 64
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
    x = torch.randn(T, B, E).cuda().half().requires_grad_(True)
    W = O.make_w(d, D, H).cuda().half()
    y = m(x, W)
    y.float().square().mean().backward()
    assert all(p.grad is not None and torch.isfinite(p.grad).all() for p in m.parameters())
    # oracle chain in fp32 with the same weights
    mf = {k_: v_.detach().float().cpu() for k_, v_ in m.state_dict().items()}
    xf = x.detach().float().cpu()
    lin = lambda n: xf @ mf[n + ".weight"].t() + mf[n + ".bias"]
    q, k, v = (lin(n).reshape(T, B, H, d) for n in ("q_proj", "k_proj", "v_proj"))
    Wp = O.build_random_matrices(W.float().cpu(), 1.0, mf["sigma"], True)
    pq, pk = O.random_project(q, Wp), O.random_project(k, Wp)
    att = O.causal_forward_chunked(pq.reshape(T, B * H, 2 * D), pk.reshape(T, B * H, 2 * D), v.reshape(T, B * H, d))
    want = att.reshape(T, B, E) @ mf["out_proj.weight"].t() + mf["out_proj.bias"]
    assert (y.detach().float().cpu() - want).abs().max().item() <= 1e-2


def test_cross_modules_forward_backward_match_oracle():
    from rfa_amd import CrossAttention, CrossAttentionProject
    torch.manual_seed(2)
    S, T, B, E, H, d, D, Lyr = 70, 33, 2, 128, 2, 64, 64, 2
    proj = CrossAttentionProject(num_layers=Lyr, embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half().eval()
    att = CrossAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
    enc = torch.randn(S, B, E).cuda().half().requires_grad_(True)
    qry = torch.randn(T, B, E).cuda().half().requires_grad_(True)
    pad = torch.zeros(B, S, dtype=torch.bool)
    pad[1, 50:] = True
    states = proj(encoder_output=enc, key_padding_mask=pad.cuda())
    assert len(states) == Lyr and states[0].s.dtype == torch.float32
    assert tuple(states[0].s.shape) == (B, H, 2 * D, d) and tuple(states[0].z.shape) == (B, H, 2 * D)
    y = att(qry, states[1])
    g = torch.randn(T, B, E).cuda().half()
    y.backward(g)
    # oracle in fp32
    L1 = proj.layers[1]
    f = lambda t: t.detach().float().cpu()
    encf, qryf = f(enc).requires_grad_(True), f(qry).requires_grad_(True)
    k = (encf @ f(L1.k_proj.weight).t() + f(L1.k_proj.bias)).reshape(S, B, H, d)
    v = (encf @ f(L1.v_proj.weight).t() + f(L1.v_proj.bias)).reshape(S, B, H, d)
    Wp = O.build_random_matrices(f(proj.random_matrices_eval), 1.0, f(L1.sigma), True)
    s, z = O.cross_state(O.random_project(k, Wp), v, pad.t())
    q = (qryf @ f(att.q_proj.weight).t() + f(att.q_proj.bias)).reshape(T, B, H, d)
    o = O.cross_readout(O.random_project(q, Wp), s, z).reshape(T, B, E)
    want = o @ f(att.out_proj.weight).t() + f(att.out_proj.bias)
    want.backward(f(g))
    assert _rel(f(states[1].s), s.detach()) <= 5e-3
    assert (f(y) - want.detach()).abs().max().item() <= 1e-2
    assert _rel(f(enc.grad), encf.grad) <= 3e-2
    assert _rel(f(qry.grad), qryf.grad) <= 3e-2


def test_incremental_rfa_out_of_place_and_inplace():
    from rfa_amd.causal_attention import incremental_rfa
    T, B, H, K, d = 3, 2, 2, 128, 64
    pq, pk = (0.1 * _randn(T, B, H, K, seed=8)).half().cuda(), (0.1 * _randn(T, B, H, K, seed=9)).half().cuda()
    v = _randn(T, B, H, d, seed=10).half().cuda()
    a1, s1, z1 = incremental_rfa(phi_q=pq[:2], phi_k=pk[:2], v=v[:2])
    s1c, z1c = s1.clone(), z1.clone()
    a2, s2, z2 = incremental_rfa(phi_q=pq[2:], phi_k=pk[2:], v=v[2:], s=s1, z=z1)
    assert torch.equal(s1, s1c) and torch.equal(z1, z1c) and s2.data_ptr() != s1.data_ptr()
    a3, s3, z3 = incremental_rfa(phi_q=pq[2:], phi_k=pk[2:], v=v[2:], s=s1, z=z1, inplace=True)
    assert s3.data_ptr() == s1.data_ptr() and torch.equal(s3, s2) and torch.equal(a2, a3)
    want, ws, wz = O.causal_forward_loop(pq.float().cpu().reshape(T, B * H, K), pk.float().cpu().reshape(T, B * H, K),
                                         v.float().cpu().reshape(T, B * H, d))
    got = torch.cat([a1, a2], 0).float().cpu().reshape(T, B * H, d)
    assert (got - want).abs().max().item() <= 2e-3


@pytest.mark.parametrize("T,B,H,d,D", [(1, 1, 1, 64, 64), (70, 2, 2, 64, 64), (1024, 1, 4, 64, 64), (200, 1, 2, 128, 32),
                                        (130, 1, 1, 128, 128)])
def test_prefill_state_equals_loop_state_and_decode_continues(T, B, H, d, D):
    """rfa_causal_prefill: the output is the causal forward, the returned state is what T
    single steps from a zero state leave behind (reference causal_attention.py:42-50), and a
    decode step taken from it reproduces row T of the forward over T + 1 steps."""
    from rfa_amd import rfa_hip
    q, k, v, _ = O.make_qkv(T + 1, B, H, d, seed=900 + T)
    W = O.make_w(d, D, H)
    N, K = B * H, 2 * D
    pq = O.random_project(q.float(), W).half().reshape(T + 1, N, K)
    pk = O.random_project(k.float(), W).half().reshape(T + 1, N, K)
    vv = v.reshape(T + 1, N, d)
    cq, ck, cv = pq.cuda(), pk.cuda(), vv.cuda()
    print(f"prefill T={T} N={N} K={K} d={d}", flush=True)
    out, s, z = rfa_hip.prefill(cq[:T].contiguous(), ck[:T].contiguous(), cv[:T].contiguous())
    assert torch.equal(out, rfa_hip.forward(cq[:T].contiguous(), ck[:T].contiguous(), cv[:T].contiguous()))
    _, s_ref, z_ref = O.causal_forward_loop(pq[:T].float(), pk[:T].float(), vv[:T].float())
    assert _rel(s.cpu(), s_ref) < 1e-5 and _rel(z.cpu(), z_ref) < 1e-5
    step = rfa_hip.incremental(cq[T:].contiguous(), ck[T:].contiguous(), cv[T:].contiguous(), s, z)
    full = O.causal_forward_chunked(pq.float(), pk.float(), vv.float()) if T > 256 else \
        O.causal_forward_cumsum(pq.float(), pk.float(), vv.float())
    assert (step.float().cpu() - full[T:]).abs().max().item() <= 2e-3


def test_module_prefill_then_decode_and_beam_reorder():
    """CausalAttention with saved_state: a prompt of several steps on an empty state (prefill),
    then single steps, equals the full causal forward; reorder_incremental_state permutes the
    batch entries of the state."""
    from rfa_amd.causal_attention import CausalAttention, reorder_incremental_state
    torch.manual_seed(11)
    T, B, E, H, d, D = 96, 3, 128, 2, 64, 64
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
    W = O.make_w(d, D, H).half().cuda()
    x = (torch.randn(T + 2, B, E) * 0.5).half().cuda()
    with torch.no_grad():
        full = m(x, W)
        state = {}
        a = m(x[:T], W, saved_state=state)                    # prefill
        b1 = m(x[T:T + 1], W, saved_state=state)               # decode steps
        b2 = m(x[T + 1:], W, saved_state=state)
    got = torch.cat([a, b1, b2], 0)
    assert (got.float() - full.float()).abs().max().item() <= 4e-3
    assert state["prev_s"].shape == (B, H, 2 * D, d) and state["prev_z"].dtype == torch.float32
    order = torch.tensor([2, 0, 0])
    before = {k_: t.clone() for k_, t in state.items()}
    reorder_incremental_state(state, order.cuda())
    for k_ in ("prev_s", "prev_z"):
        assert torch.equal(state[k_], before[k_][order.cuda()])
    assert reorder_incremental_state({}, order) == {}


def _masked_case(T, B, H, d, D, seed, with_pad, mask_kind):
    q, k, v, g = O.make_qkv(T, B, H, d, seed)
    W = O.make_w(d, D, H)
    pq = O.random_project(q.float(), W).half()
    pk = O.random_project(k.float(), W).half()
    pad = None
    if with_pad:
        pad = torch.zeros(B, T, dtype=torch.uint8)
        pad[0, max(T - 5, 1):] = 1
        if B > 1:
            pad[1, :2] = 1
    if mask_kind == "causal":
        am = torch.triu(torch.full((T, T), float("-inf")), 1)
    elif mask_kind == "band":       # an arbitrary pattern: causal band of width 40 plus a few holes
        i = torch.arange(T)
        am = torch.zeros(T, T)
        am[(i[None, :] > i[:, None]) | (i[:, None] - i[None, :] >= 40)] = -1.0
        am[i % 7 == 3, 0] = -1.0
    elif mask_kind == "stripes":    # whole 64 x 64 tiles masked, a fully masked row block, and a ragged edge
        am = torch.zeros(T, T)
        am[:64, :] = -1.0                       # queries 0..63 see nothing: zero output rows
        am[:, 128:192] = -1.0                   # keys 128..191 hidden from everybody
        am[200:, :70] = -1.0                    # a masked region that ends inside a tile
    else:
        am = None
    return pq, pk, v, g, pad, am


@pytest.mark.parametrize("T,B,H,d,D,with_pad,mask_kind", [
    (6, 2, 1, 64, 32, True, "causal"),
    (64, 1, 2, 64, 64, False, "causal"),
    (130, 2, 2, 64, 64, True, "causal"),
    (200, 1, 2, 64, 64, True, "band"),
    (96, 2, 1, 128, 64, False, None),
    (70, 1, 1, 128, 128, True, "causal"),
    (600, 1, 1, 64, 64, False, "causal"),      # ten blocks: more than one batch of tile flags
    (330, 1, 2, 64, 64, True, "stripes"),
])
def test_masked_rfa_matches_oracle_forward_and_backward(T, B, H, d, D, with_pad, mask_kind):
    """masked_rfa on the quadratic-form kernels against the oracle (causal_attention.py:57-109) and
    its autograd gradients, with key padding, the causal mask and an arbitrary mask."""
    from rfa_amd.causal_attention import masked_rfa
    pq, pk, v, g, pad, am = _masked_case(T, B, H, d, D, 4000 + T, with_pad, mask_kind)
    print(f"masked_rfa T={T} B={B} H={H} K={2*D} d={d} pad={with_pad} mask={mask_kind}", flush=True)
    cq, ck, cv = (t.cuda().requires_grad_(True) for t in (pq, pk, v))
    out = masked_rfa(phi_q=cq, phi_k=ck, v=cv, key_padding_mask=None if pad is None else pad.cuda(),
                     attn_mask=None if am is None else am.cuda())
    out.backward(g.reshape(T, B, H * d).cuda())
    fq, fk, fv = (t.float().requires_grad_(True) for t in (pq, pk, v))
    ref = O.masked_rfa(fq, fk, fv, pad, am)
    ref.backward(g.float())
    assert tuple(out.shape) == (T, B, H * d)
    # outputs are O(|v|) here (weights sum to 1 in magnitude): the forward gate of the path
    assert (out.float().cpu().view(T, B, H, d) - ref.detach()).abs().max().item() <= 4e-3
    for name, got, want in (("dphi_q", cq.grad, fq.grad), ("dphi_k", ck.grad, fk.grad), ("dv", cv.grad, fv.grad)):
        assert torch.isfinite(got).all(), name
        assert _rel(got.float().cpu(), want) <= 1e-2, (name, _rel(got.float().cpu(), want))
    if pad is not None:      # padded keys receive no gradient
        padded = pad.bool().t()[:, :, None, None].expand_as(ck.grad).cuda()
        assert ck.grad[padded].abs().max().item() == 0.0


def test_causal_attention_module_quadratic_fallback_matches_scan_module():
    """CausalAttention(cuda_causal_rfa=False) runs masked_rfa; with row sums far below 1 the
    scan path clamps at 1 while the quadratic form normalises, so compare against the oracle
    chain rather than the other module."""
    from rfa_amd.causal_attention import CausalAttention
    torch.manual_seed(3)
    T, B, E, H, d, D = 80, 2, 128, 2, 64, 64
    m = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D, cuda_causal_rfa=False).cuda().half()
    W = O.make_w(d, D, H).half().cuda()
    x = (torch.randn(T, B, E) * 0.5).half().cuda()
    am = torch.triu(torch.full((T, T), float("-inf")), 1).cuda()
    with torch.no_grad():
        y = m(x, W, attn_mask=am)
        f = lambda lin, t: torch.nn.functional.linear(t.float(), lin.weight.float(), lin.bias.float())
        q, k, v = (f(p_, x).view(T, B, H, d).cpu() for p_ in (m.q_proj, m.k_proj, m.v_proj))
        w = O.build_random_matrices(W.float().cpu(), m.tau, m.sigma.float().cpu(), True)
        attn = O.masked_rfa(O.random_project(q, w), O.random_project(k, w), v, None, am.cpu())
        want = f(m.out_proj, attn.reshape(T, B, E).cuda())
    assert (y.float() - want).abs().max().item() <= 2e-2


@pytest.mark.usefixtures("binding")
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 3, 63, 64, 65, 200])
def test_pack_negative_mask_matches_the_general_packing(T, dtype):
    """One launch against compare + pack_attn_mask, byte for byte: values around zero, infinities and
    NaN, and every stride order a mask may come with."""
    from rfa_amd import rfa_hip
    gen = torch.Generator().manual_seed(T)
    special = torch.tensor([0.0, -0.0, -1e-7, 1e-7, float("-inf"), float("inf"), float("nan"), -1.0, -3e38, 1e-38, -1e-38])
    base = special[torch.randint(0, len(special), (2 * T, 3 * T), generator=gen)].to(dtype).cuda()
    print(f"pack_negative_mask T={T} {dtype}", flush=True)
    row = base[0]
    for mask in (base[:T, :T].contiguous(), base[:T, :T].t(), base[::2, ::3], base[1:T + 1, T:2 * T] if T > 1 else base[1:2, 1:2],
                 row[None, :T].expand(T, T), row[:T, None].expand(T, T)):
        want = rfa_hip.pack_attn_mask(mask < 0.0)
        got = rfa_hip.pack_negative_mask(mask)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    if T == 3:
        with pytest.raises((RuntimeError, ValueError)):
            rfa_hip.pack_negative_mask(base[:2, :3])
        with pytest.raises((RuntimeError, TypeError)):
            rfa_hip.pack_negative_mask(base[:3, :3].to(torch.int32))


@pytest.mark.usefixtures("binding")
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_traced_masked_rfa_follows_its_mask(dtype):
    """A traced call packs the mask that it is given, not the one that it was traced with."""
    from rfa_amd.causal_attention import masked_rfa
    T, B, H, d = 70, 2, 2, 64
    q, k = (0.2 * torch.rand(T, B, H, 64, device="cuda").half() for _ in range(2))
    v = torch.randn(T, B, H, d, device="cuda").half()
    masks = [torch.full((T, T), float("-inf"), device="cuda", dtype=dtype).triu(n) for n in (1, 9)]
    call = lambda q, k, v, m: masked_rfa(phi_q=q, phi_k=k, v=v, attn_mask=m)
    traced = torch.jit.trace(call, (q, k, v, masks[0]), check_trace=False)
    for m in masks:
        assert torch.equal(traced(q, k, v, m), call(q, k, v, m))


def _native_forms(path, form):
    """(run, leaves) of one path in one form of its inputs; run() -> outputs whose sum of products is differentiated."""
    from rfa_amd import causal_attention as C, cross_attention as X, utils
    T, B, H, d, D = 37, 3, 2, 64, 32
    E = H * d
    gen = torch.Generator("cuda").manual_seed(5)
    grad = form != "no_grad"

    def leaf(*shape, scale=None):
        x = torch.randn(*shape, generator=gen, device="cuda")
        if scale is not None:           # feature values of one sign: no row sum near zero
            x = scale * x.abs()
        if form == "strided":       # every second entry of a wider tensor, batch and time swapped in memory
            wide = torch.zeros(shape[1], shape[0], *shape[2:-1], 2 * shape[-1], device="cuda", dtype=torch.float16)
            wide[..., ::2] = x.half().transpose(0, 1)
            return wide[..., ::2].transpose(0, 1).detach().requires_grad_(grad)
        return x.half().requires_grad_(grad)

    def layer(cls):
        torch.manual_seed(7)
        m = cls(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
        if form == "no_bias":
            for lin in m.children():
                lin.bias = None
        if form == "frozen":
            for p in m.parameters():
                p.requires_grad_(False)
        return m

    W = O.make_w(d, D, H).cuda().half()
    if path == "random_project":
        x = leaf(T, B, H, d)
        w = W.clone().requires_grad_(grad and form != "frozen")
        return lambda: utils.random_project(x=x, random_matrices=w), [x, w]
    if path in ("causal", "masked", "padded"):
        q, k, v = leaf(T, B, H, 2 * D, scale=0.1), leaf(T, B, H, 2 * D, scale=0.1), leaf(T, B, H, d)
        if form == "frozen":
            k = k.detach()
        if path == "causal":
            return lambda: C.cuda_causal_rfa(phi_q=q, phi_k=k, v=v), [q, k, v]
        pad = torch.zeros(B, T, dtype=torch.bool, device="cuda")
        pad[0, 30:] = True
        pad[2, 5] = True
        if path == "padded":
            pad = pad.t().contiguous().t() if form == "strided" else pad.byte() * 3 if form == "twice" else pad
            return lambda: C.cuda_causal_rfa(phi_q=q, phi_k=k, v=v, key_padding_mask=pad), [q, k, v]
        mask = torch.full((T, T), float("-inf"), device="cuda").triu(1)
        return lambda: C.masked_rfa(phi_q=q, phi_k=k, v=v, key_padding_mask=pad, attn_mask=mask), [q, k, v]
    x = leaf(T, B, E)
    if path == "module":
        m = layer(C.CausalAttention)
        return lambda: m(x, W), [x, *m.parameters()]
    enc = leaf(T + 4, B, E)
    src, m = layer(X.CrossAttentionProjectLayer), layer(X.CrossAttention)
    mask = torch.zeros(T + 4, B, 1, 1, dtype=torch.bool, device="cuda")
    mask[T:, 1] = True
    return (lambda: m(x, src(encoder_output=enc, random_matrices=W, mask=mask)),
            [x, enc, *src.parameters(), *m.parameters()])


@pytest.mark.parametrize("form", ["plain", "strided", "frozen", "no_bias", "no_grad", "hooks", "twice"])
@pytest.mark.parametrize("path", ["random_project", "causal", "padded", "masked", "module", "cross"])
def test_native_nodes_give_the_bits_of_the_python_functions(path, form, monkeypatch):
    """The C++ autograd nodes against the Python autograd functions over the same kernels: outputs and every
    gradient bit for bit (in the layers, whose Linear products are summed by another kernel and rounded to fp16
    at other places, within a few roundings), from strided inputs, with frozen or missing parameters, through saved-tensor
    hooks, and with two backward passes over one graph."""
    from rfa_amd import rfa_hip
    if rfa_hip.native is None:
        pytest.skip("the torch binding is not active")
    print(f"native nodes: {path} {form}", flush=True)
    monkeypatch.setattr("rfa_amd.projection.linear_rows", lambda *a: None)     # another sum than the library's
    run, leaves = _native_forms(path, form)
    results = []
    for native in (rfa_hip.native, None):
        monkeypatch.setattr(rfa_hip, "native", native)
        for t in leaves:
            t.grad = None
        packed = []
        if form == "hooks":
            with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.clone(), lambda t: t):
                out = run()
            assert packed
        else:
            with torch.set_grad_enabled(form != "no_grad"):
                out = run()
        assert out.is_contiguous() and out.requires_grad == (form != "no_grad")
        if form != "no_grad":
            g = torch.randn(out.shape, generator=torch.Generator("cuda").manual_seed(9), device="cuda").half()
            out.backward(g, retain_graph=form == "twice")
            if form == "twice":
                out.backward(g)
        results.append([out.detach()] + [None if t.grad is None else t.grad.clone() for t in leaves])
    for a, b in zip(*results):
        assert (a is None) == (b is None)
        if a is not None and path in ("module", "cross"):
            assert _rel(a.double().cpu(), b.double().cpu()) <= 4 * 2.0 ** -11
        elif a is not None:
            assert torch.equal(a, b)


@pytest.mark.parametrize("path", ["random_project", "causal", "padded", "masked", "module", "cross"])
def test_native_nodes_check_what_saved_tensor_hooks_return(path):
    """Each saved tensor in turn comes back with other strides (same values: what a hook may do), another type or
    another device.  The backward pass gives the gradients of the run without hooks (in the layers within the
    roundings of another product kernel) or raises; for another type or device it raises."""
    from rfa_amd import rfa_hip
    if rfa_hip.native is None:
        pytest.skip("the torch binding is not active")
    run, leaves = _native_forms(path, "plain")

    def gradients(change=None, which=-1):
        count = [0]

        def pack(t):
            count[0] += 1
            return t if count[0] - 1 != which else change(t)
        for t in leaves:
            t.grad = None
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
            out = run()
        out.backward(torch.randn(out.shape, generator=torch.Generator("cuda").manual_seed(9), device="cuda").half())
        return [t.grad.clone() for t in leaves], count[0]

    want, saved = gradients()
    refused = {"strides": 0, "type": 0, "device": 0}
    for which in range(saved):
        for name, change in (("strides", lambda t: t.transpose(0, 1).contiguous().transpose(0, 1) if t.dim() > 1 else t),
                             ("type", lambda t: t.double()), ("device", lambda t: t.cpu())):
            print(f"saved tensor {which} of {path}: other {name}", flush=True)
            try:
                got, _ = gradients(change, which)
            except (RuntimeError, ValueError, TypeError):
                refused[name] += 1
                continue
            assert name == "strides"
            for a, b in zip(got, want):
                assert _rel(a.double().cpu(), b.double().cpu()) <= (4 * 2.0 ** -11 if path in ("module", "cross") else 0)
    assert refused["type"] == refused["device"] == saved


@pytest.mark.parametrize("change", ["longer", "shorter", "narrower"])
def test_layers_check_the_shapes_of_what_saved_tensor_hooks_return(change):
    """An input or a weight of a layer comes back from a hook with another shape: the backward pass raises before it
    launches anything over rows or columns that are not there."""
    from rfa_amd import rfa_hip
    from rfa_amd.causal_attention import CausalAttention
    if rfa_hip.native is None:
        pytest.skip("the torch binding is not active")
    T, B, H, d, D = 70, 3, 2, 64, 32
    E = H * d
    new = {"longer": lambda t: torch.cat([t, t[:1]]), "shorter": lambda t: t[:-1].contiguous(),
           "narrower": lambda t: t[..., :E // 2].contiguous()}[change]
    layer = CausalAttention(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half().train()
    x = torch.randn(T, B, E, device="cuda").half().requires_grad_()
    W = O.make_w(d, D, H).half().cuda()
    seen, which, total = [0], [-1], 0

    def pack(t):
        if t.shape[-1:] != (E,) or t.dim() not in (2, 3):       # what the layers save, not the scan
            return t
        seen[0] += 1
        return new(t) if seen[0] - 1 == which[0] else t

    while True:
        seen[0] = 0
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
            out = layer(x, W)
        if which[0] < 0:
            out.backward(torch.ones_like(out))
            total = seen[0]
            assert total >= 6        # two inputs and four weights
        else:
            print(f"{change} saved tensor {which[0]}", flush=True)
            with pytest.raises((RuntimeError, ValueError)):
                out.backward(torch.ones_like(out))
        which[0] += 1
        if which[0] == total:
            break


def test_native_nodes_leave_odd_calls_to_the_python_functions():
    """Dispatch modes and tracing see the Python functions, and functorch transforms and forward-mode
    tangents meet the errors that those raise."""
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode
    from rfa_amd import rfa_hip
    from rfa_amd.causal_attention import cuda_causal_rfa
    if rfa_hip.native is None:
        pytest.skip("the torch binding is not active")
    q, k, v = (torch.randn(9, 2, 2, n, device="cuda").half().requires_grad_() for n in (64, 64, 64))
    call = lambda a: cuda_causal_rfa(phi_q=a, phi_k=k, v=v)
    assert rfa_hip.native.node_causal(q, k, v) is not None

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with Mode():
        assert rfa_hip.native.node_causal(q, k, v) is None
        call(q)
    assert rfa_hip.native.node_causal(q.float(), k, v) is None
    assert rfa_hip.native.node_causal(q.cpu(), k, v) is None
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda a: call(a).float().sum())(q.detach())
    with pytest.raises(RuntimeError), forward_ad.dual_level():
        call(forward_ad.make_dual(q.detach(), torch.ones_like(q)))


def test_traced_scan_follows_its_inputs():
    """While a call is traced the nodes step aside, so that the trace holds the Python functions."""
    from rfa_amd import rfa_hip
    from rfa_amd.causal_attention import cuda_causal_rfa
    if rfa_hip.native is None:
        pytest.skip("the torch binding is not active")
    aside = []

    def call(q, k, v):
        if torch.jit.is_tracing():
            aside.append(rfa_hip.native.node_causal(q, k, v) is None)
        return cuda_causal_rfa(phi_q=q, phi_k=k, v=v)
    first, second = ([0.1 * torch.rand(70, 2, 2, 64, device="cuda").half() for _ in range(3)] for _ in range(2))
    traced = torch.jit.trace(call, tuple(first), check_trace=False)
    assert aside == [True]
    assert torch.equal(traced(*second), call(*second))


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("T,B,H,d", [(70, 3, 3, 64), (205, 40, 8, 128)])
@pytest.mark.parametrize("path", ["module", "cross"])
def test_layer_gradients_where_the_library_multiplies(path, T, B, H, d, bias):
    """The nodes' other branches: widths that are no multiple of 128 (library products for every gradient, the stack
    of three weights) and rows above the own kernels' limits (library products for dx and y), outputs and every
    gradient against the formulas in fp64.  fp16 at some eight places on the way to each: 8 x 2^-11 / sqrt(3)."""
    from rfa_amd import causal_attention as C, cross_attention as X
    D, E = 32, H * d
    gen = torch.Generator("cuda").manual_seed(T)
    rand = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")
    W = rand(H, D, d).half()

    def layer(cls):
        m = cls(embed_dim=E, num_heads=H, head_dim=d, proj_dim=D).cuda().half()
        with torch.no_grad():
            for name, p in m.named_parameters():
                p.copy_(1 + 0.1 * rand(*p.shape) if name == "sigma" else rand(*p.shape) / (2 * E) ** 0.5)
        if not bias:
            for lin in m.children():
                lin.bias = None
        return m, {n: p.detach().double().requires_grad_() for n, p in m.named_parameters()}

    leaf = lambda t: t.half().requires_grad_()
    lin = lambda p, name, t: t @ p[name + ".weight"].t() + p.get(name + ".bias", 0.0)
    heads = lambda t: t.view(*t.shape[:2], H, d)
    x, g = leaf(rand(T, B, E)), rand(T, B, E).half()
    x64 = x.detach().double().requires_grad_()
    print(f"layer gradients {path} T={T} B={B} H={H} d={d} bias={bias}", flush=True)
    if path == "module":
        m, p = layer(C.CausalAttention)
        out = m(x, W)
        w = W.double() * p["sigma"]
        q, k, v = (heads(lin(p, n, x64)) for n in ("q_proj", "k_proj", "v_proj"))
        rows = lambda t: t.reshape(T, B * H, -1)
        attn = O.causal_forward_cumsum(rows(O.random_project(q, w)), rows(O.random_project(k, w)), rows(v))
        leaves, leaves64 = [x, *m.parameters()], [x64, *p.values()]
    else:
        src, ps = layer(X.CrossAttentionProjectLayer)
        m, p = layer(X.CrossAttention)
        enc = leaf(rand(T, B, E))
        enc64 = enc.detach().double().requires_grad_()
        pad = torch.zeros(T, B, 1, 1, dtype=torch.bool, device="cuda")
        pad[T - 9:, 1] = True
        out = m(x, src(encoder_output=enc, random_matrices=W, mask=pad))
        w = W.double() * ps["sigma"]
        k, v = (heads(lin(ps, n, enc64)) for n in ("k_proj", "v_proj"))
        phi_k = O.random_project(k, w).masked_fill(pad, 0.0)
        attn = O.cross_readout(O.random_project(heads(lin(p, "q_proj", x64)), w),
                               torch.einsum("tbhk,tbhd->bhkd", phi_k, v), phi_k.sum(0))
        leaves = [x, enc, *src.parameters(), *m.parameters()]
        leaves64 = [x64, enc64, *ps.values(), *p.values()]
    want = lin(p, "out_proj", attn.reshape(T, B, E))
    out.backward(g)
    want.backward(g.double())
    for a, b in [(out.detach(), want.detach())] + [(s.grad, t.grad) for s, t in zip(leaves, leaves64)]:
        err = _rel(a.double(), b)
        print(f"  {tuple(a.shape)} {err:.2e}", flush=True)
        assert err <= 8 * 2.0 ** -11 / 3 ** 0.5


@pytest.mark.parametrize("d,D", [(64, 32), (64, 64), (128, 32), (128, 64)])
@pytest.mark.parametrize("T", [2, 15, 64, 65, 127, 200])
def test_prefill_from_projected_rows(T, d, D):
    """The scan that forms phi(q), phi(k) itself against the feature-map launch followed by the scan,
    at short last chunks and with rows of zeros.  The formulas are the same; the compiler may contract them
    differently, which moves a phi value to the neighbouring fp16 value at most (2^-11)."""
    from rfa_amd import _lib, rfa_hip
    from rfa_amd.utils import random_project_pair
    if rfa_hip.native is None:
        pytest.skip("the torch binding is not active")
    H = 4
    B = 300 if T > 64 else 3        # sequences enough for one segment each
    assert _lib.load().rfa_causal_prefill_rows_supported(T, B * H, D, d)
    gen = torch.Generator("cuda").manual_seed(T)
    q, k, v = (torch.randn(T, B, H, d, generator=gen, device="cuda").half() for _ in range(3))
    q[T // 2, 1] = 0
    k[T - 1, 2] = 0
    W = O.make_w(d, D, H).half().cuda()
    print(f"prefill from rows T={T} d={d} D={D}", flush=True)
    attn, s, z = rfa_hip.native.node_prefill(q, k, v, W, O.SCALE)
    pq, pk = random_project_pair(x0=q, x1=k, random_matrices=W)
    want = rfa_hip.prefill(pq.view(T, B * H, 2 * D), pk.view(T, B * H, 2 * D), v.view(T, B * H, d))
    for got, ref in zip((attn, s, z), want):
        err = _rel(got.reshape(ref.shape).float().cpu(), ref.float().cpu())
        print(f"  {err:.2e}", flush=True)
        assert torch.isfinite(got).all() and err <= 2.0 ** -11
    assert rfa_hip.native.node_prefill(q[:, :1], k[:, :1], v[:, :1], W, O.SCALE) is None      # not contiguous


@pytest.mark.parametrize("T", [64, 65, 130, 300])
@pytest.mark.parametrize("with_mask", [True, False])
def test_masked_rfa_blocks_dealt_singly_and_in_pairs(T, with_mask):
    """Many sequences (row blocks dealt in pairs under a mask) give the bits of the same sequences a few
    at a time (dealt singly, every second round in reverse): the order of a row's sums does not depend on it."""
    from rfa_amd import rfa_hip
    H, d, D = 4, 64, 32
    B = -(-1000 // (H * -(-T // 64)))
    gen = torch.Generator("cuda").manual_seed(T)
    q, k = (torch.rand(T, B * H, 2 * D, generator=gen, device="cuda").half() for _ in range(2))
    v, g = (torch.randn(T, B * H, d, generator=gen, device="cuda").half() for _ in range(2))
    m = mt = None
    if with_mask:
        m, mt = rfa_hip.pack_attn_mask(torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1))
    print(f"masked blocks T={T} N={B * H} mask={with_mask}", flush=True)

    def run(b0, b1):
        cut = lambda t: t[:, b0 * H:b1 * H].contiguous()
        out, rsum = rfa_hip.masked_forward(cut(q), cut(k), cut(v), H, None, m)
        return [out, rsum, *rfa_hip.masked_backward(cut(q), cut(k), cut(v), cut(g), out, rsum, H, None, m, mt)]

    whole = run(0, B)
    for b0 in (0, B // 2, B - 17):
        for a, b in zip(whole, run(b0, b0 + 17)):
            assert torch.isfinite(b).all() and torch.equal(a[:, b0 * H:(b0 + 17) * H], b)


@pytest.mark.parametrize("d,D", [(64, 32), (64, 64), (64, 128), (128, 32), (128, 64), (128, 128)])
def test_masked_rfa_blocks_dealt_singly_and_in_pairs_at_every_width(d, D):
    """384 sequences of 4 row blocks go in pairs whatever a CU holds (one to four workgroups), 16 of them singly: the
    same bits, and 4 of them against the oracle in fp64 with a padded key and a row that keeps one key only."""
    from rfa_amd import rfa_hip
    T, H, B, few = 200, 4, 96, 4
    gen = torch.Generator("cuda").manual_seed(D)
    q, k = (torch.rand(T, B * H, 2 * D, generator=gen, device="cuda").half() / D ** 0.5 for _ in range(2))
    v, g = (torch.randn(T, B * H, d, generator=gen, device="cuda").half() for _ in range(2))
    masked = torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1)
    masked[70] = True
    masked[70, 3] = False
    m, mt = rfa_hip.pack_attn_mask(masked)
    pad = torch.zeros(B, T, dtype=torch.bool, device="cuda")
    pad[0, 190:] = True
    print(f"masked blocks at every width d={d} D={D}", flush=True)

    def run(b0, b1):
        cut = lambda t: t[:, b0 * H:b1 * H].contiguous()
        out, rsum = rfa_hip.masked_forward(cut(q), cut(k), cut(v), H, pad[b0:b1], m)
        return [out, rsum, *rfa_hip.masked_backward(cut(q), cut(k), cut(v), cut(g), out, rsum, H, pad[b0:b1], m, mt)]

    whole = run(0, B)
    for b0 in (0, B - few):
        for a, b in zip(whole, run(b0, b0 + few)):
            assert torch.isfinite(b).all() and torch.equal(a[:, b0 * H:(b0 + few) * H], b)
    wide = lambda t: t[:, :H].reshape(T, 1, H, -1).double().cpu().requires_grad_()
    q64, k64, v64 = wide(q), wide(k), wide(v)
    ref = O.masked_rfa(q64, k64, v64, pad[:1].cpu(), torch.zeros(T, T).masked_fill(masked.cpu(), float("-inf")).double())
    ref.backward(g[:, :H].reshape(ref.shape).double().cpu())
    for got, want in zip([whole[0]] + whole[2:], [ref.detach(), q64.grad, k64.grad, v64.grad]):
        assert _rel(got[:, :H].double().cpu().reshape(want.shape), want) <= 4 * 2.0 ** -11      # fp16 tiles and results
