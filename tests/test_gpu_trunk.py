"""The prefill trunk's kernels (q38moe_prefill.hip) against float64 restatements of the modules they
replace, next to the torch code of q38.prefill in the same dtype. Both evaluate the same formulas in
fp32 with other summation orders, so the bar is the torch code's own distance from float64: at most
1.5 times it, plus 2e-7 (a few fp32 roundings, where torch's happen to cancel)."""
import pytest
import torch
import torch.nn.functional as F

from q38 import prefill as P

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


def _hold(native, torch_code, exact, what):
    e, bar = _rel(native, exact), 1.5 * _rel(torch_code, exact) + 2e-7
    assert e <= bar, f"{what}: {e:.2e} from float64, bar {bar:.2e}"


def _fill(m, g, dev, std):
    for name, p in m.named_parameters():
        p.data = torch.randn(p.shape, generator=g, device=dev) * std(name)
    return m


def _mhc64(m, norm, X, y, cfg):
    """Sublayer input and the stream after output y, in float64 (modeling:994-1031)."""
    w = {n: p.detach().double() for n, p in m.named_parameters()}
    X, n = X.double(), 4
    f = X.flatten(2)
    f = f * torch.rsqrt(f.pow(2).mean(-1, keepdim=True) + 1e-6)
    z = torch.tanh(f @ w["A.weight"].t() @ w["B.weight"].t())
    pre = torch.sigmoid(w["b_pre"] + w["alphas"][0] * z[..., :n])
    post = 2 * torch.sigmoid(w["b_post"] + w["alphas"][1] * z[..., n:2 * n])
    logits = w["b_res"] + w["alphas"][2] * z[..., 2 * n:].unflatten(-1, (n, n))
    M = torch.exp(logits - logits.amax((-2, -1), keepdim=True))
    for _ in range(cfg.mhc_iters):
        M = M / M.sum(-1, keepdim=True)
        M = M / M.sum(-2, keepdim=True)
    x = (pre[..., None] * X).sum(2)
    x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + cfg.rms_eps) * (1 + norm.weight.detach().double())
    return x, M @ X + post[..., None] * y.double()[:, :, None]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,h", [(1, 1, 64),        # one token, a quarter of a wave's columns
                                   (2, 67, 320),      # a partial block of tokens, a partial chunk of columns
                                   (1, 64, 1024),
                                   (3, 2731, 256)])   # 16 tokens per block, the last one partial
def test_mhc_sublayer(gpu, dtype, B, S, h):
    """mhc_update (every mode) and mhc_pre around one sublayer."""
    from q38.hip import ops
    cfg = P.PrefillConfig(hidden=max(h, 64), layers=1)
    g = torch.Generator(device=gpu).manual_seed(S + h)
    m = _fill(P._MHC(cfg).to(gpu), g, gpu, lambda n: {"A.weight": 0.02, "B.weight": 0.2}.get(n, 1.0)).to(dtype)
    norm = _fill(P._Norm(h).to(gpu), g, gpu, lambda n: 0.05).to(dtype)
    e, d, y = (torch.randn(B, S, h, generator=g, device=gpu).to(dtype) for _ in range(3))
    noise = torch.randn(B, S, 4, h, generator=g, device=gpu)
    T = B * S
    ssq = torch.empty(T, device=gpu)
    with torch.no_grad():
        X = torch.empty(B, S, 4, h, device=gpu)
        ops.mhc_update(ops.MHC_INIT, X.view(T, 4, h), e.view(T, h), ssq)
        ref = e.float()[:, :, None].expand(-1, -1, 4, -1)
        assert torch.equal(X, ref)
        ops.mhc_update(ops.MHC_ADD, X.view(T, 4, h), d.view(T, h), ssq)
        assert torch.equal(X, ref + d.float()[:, :, None])
        assert torch.allclose(ssq.double(), X.double().pow(2).sum((2, 3)).view(-1), rtol=1e-6)
        X = X + noise
        ops.mhc_update(ops.MHC_ADD, X.view(T, 4, h), torch.zeros_like(d).view(T, h), ssq)
        start = X.clone()
        x, st = P._mhc_in(m, norm, X, ssq, cfg, dtype)
        X = P._mhc_out(X, y, st, ssq)
        xt, stt = P._mhc_in(m, norm, start, None, cfg, dtype)
        Xt = P._mhc_out(start, y, stt, None)
        x64, X64 = _mhc64(m, norm, start, y, cfg)
    assert x.dtype == dtype
    _hold(x, xt, x64, "sublayer input")
    _hold(X, Xt, X64, "stream")
    assert torch.allclose(ssq.double(), X.double().pow(2).sum((2, 3)).view(-1), rtol=1e-6)


class _Rank128(P.PrefillConfig):
    mhc_rank = 128


@pytest.mark.parametrize("B,S,h", [(1, 5, 1088), (1, 3, 1472), (2, 33, 2048),
                                   (1, 8193, 1792)])  # 16 tokens per block, the last one with one
def test_mhc_wide(gpu, monkeypatch, B, S, h):
    """Hidden sizes above 1024 at a rank the kernel takes (PrefillConfig's own, hidden / 8, is above it)."""
    monkeypatch.setattr(P, "PrefillConfig", _Rank128)
    test_mhc_sublayer(gpu, torch.bfloat16, B, S, h)


def _delta64(m, x, cfg):
    """The DeltaNet mixer in float64, token by token (modeling:352-413, 464-577)."""
    w = {n: p.detach().double() for n, p in m.named_parameters()}
    B, S, _ = x.shape
    nk, nv, d = cfg.lin_k_heads, cfg.lin_v_heads, cfg.lin_head_dim
    x = x.double()
    qkv = (x @ w["in_proj_qkv.weight"].t()).transpose(1, 2)
    qkv = F.silu(F.conv1d(F.pad(qkv, (3, 0)), w["conv1d.weight"], groups=qkv.shape[1]))
    q, k, v = (t.reshape(B, -1, d, S).transpose(2, 3) for t in qkv.split([nk * d, nk * d, nv * d], 1))
    q, k = ((t * torch.rsqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(nv // nk, 1) for t in (q, k))
    beta = torch.sigmoid(x @ w["in_proj_b.weight"].t()).transpose(1, 2)
    g = (-w["A_log"].exp() * F.softplus(x @ w["in_proj_a.weight"].t() + w["dt_bias"])).transpose(1, 2)
    state, out = x.new_zeros(B, nv, d, d), torch.empty_like(v)
    for t in range(S):
        state = state * g[:, :, t, None, None].exp()
        u = beta[:, :, t, None] * (v[:, :, t] - (k[:, :, t, None] @ state)[:, :, 0])
        state = state + k[:, :, t, :, None] * u[:, :, None]
        out[:, :, t] = (q[:, :, t, None] * d ** -0.5 @ state)[:, :, 0]
    o = out.transpose(1, 2)
    o = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + cfg.rms_eps) * w["norm.weight"]
    z = (x @ w["in_proj_z.weight"].t()).reshape(B, S, nv, d)
    return (o * F.silu(z)).reshape(B, S, nv * d) @ w["out_proj.weight"].t()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,nk,nv,slow", [(1, 64, 1, 1, False),    # one chunk, one head
                                            (2, 192, 2, 4, False),   # 8 heads, key heads shared by two
                                            (3, 320, 3, 3, True),    # slow decays: states reach far back
                                            (1, 1024, 13, 39, False)])
def test_delta_net(gpu, dtype, B, S, nk, nv, slow):
    """gdn_conv and gdn_delta inside the mixer; two runs agree bit for bit."""
    cfg = P.PrefillConfig(hidden=256, layers=1, lin_k_heads=nk, lin_v_heads=nv)
    g = torch.Generator(device=gpu).manual_seed(S + nv)
    m = _fill(P._DeltaNet(cfg).to(gpu), g, gpu, lambda n: 0.05 if "proj" in n else 0.3)
    m.A_log.data = torch.rand(nv, generator=g, device=gpu).mul(16).add(0.01).log() - (3.0 if slow else 0.0)
    m.norm.weight.data += 1
    m.dt_bias.data += 1
    m = m.to(dtype)
    x = torch.randn(B, S, 256, generator=g, device=gpu).to(dtype)
    with torch.no_grad():
        native, again = P._delta_net(m, x, cfg, True), P._delta_net(m, x, cfg, True)
        torch_code = P._delta_net(m, x, cfg, False)
        exact = _delta64(m, x, cfg)
    assert native.dtype == dtype and torch.equal(native, again)
    _hold(native, torch_code, exact, "mixer output")


def _qsa64(m, sel, x, cos, sin, cfg):
    """The QSA mixer in float64 over the given key blocks (modeling:1117-1165)."""
    w = {n: p.detach().double() for n, p in m.named_parameters()}
    B, S, _ = x.shape
    H, KV, d, nb = cfg.heads, cfg.kv_heads, cfg.head_dim, S // 64
    x, cos, sin = x.double(), cos.double(), sin.double()

    def heads(name, n):
        return (x @ w[name].t()).view(B, S, n, -1).transpose(1, 2)

    def norm_rope(t, name):
        t = t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + cfg.rms_eps) * (1 + w[name])
        r = cos.shape[-1]
        turned = torch.cat([-t[..., r // 2:r], t[..., :r // 2]], -1)
        return torch.cat([t[..., :r] * cos + turned * sin, t[..., r:]], -1)

    q, gate = heads("q_proj.weight", H).split([d, d], -1)
    q, k = norm_rope(q, "q_norm.weight"), norm_rope(heads("k_proj.weight", KV), "k_norm.weight")
    k, v = (t.repeat_interleave(H // KV, 1) for t in (k, heads("v_proj.weight", KV)))
    counts = torch.clamp(torch.arange(nb, device=x.device) + 1, max=sel.shape[-1])
    chosen = torch.zeros(B, nb, nb, dtype=torch.bool, device=x.device)
    for i in range(nb):
        chosen[:, i].scatter_(1, sel[:, i, :int(counts[i])], True)
    mask = chosen.repeat_interleave(64, 1).repeat_interleave(64, 2) & torch.ones(S, S, dtype=torch.bool,
                                                                                 device=x.device).tril()
    s = (q @ k.transpose(-1, -2) * d ** -0.5).masked_fill(~mask[:, None], float("-inf"))
    o = (torch.softmax(s, -1) @ v) * torch.sigmoid(gate)
    return o.transpose(1, 2).reshape(B, S, H * d) @ w["o_proj.weight"].t()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,H,KV,blocks,rotary,spread", [
    (1, 64, 2, 2, 8, 0.25, 1.0),     # one block, one head per workgroup
    (2, 320, 6, 2, 3, 0.5, 1.0),     # fewer blocks than the sequence has, an odd number of heads per key head
    (1, 1024, 38, 2, 8, 0.25, 1.0),
    (4, 1088, 10, 1, 8, 1.0, 6.0),   # one key head, all features rotated; peaked softmax
    (4, 1088, 38, 2, 8, 0.25, 6.0)])  # four heads per workgroup (bf16), three in the last
def test_qsa(gpu, dtype, B, S, H, KV, blocks, rotary, spread):
    """qsa_prep and qsa_attention inside the mixer, on the key blocks the indexer selects."""
    cfg = P.PrefillConfig(hidden=256, layers=1, heads=H, kv_heads=KV, qsa_blocks=blocks, partial_rotary=rotary)
    if H == 38 and B == 4:  # launch_qsa_attention's rule
        sets = -(-(H // KV) // 4)
        assert B * (S // 64) * KV * sets >= 2 * torch.cuda.get_device_properties(gpu).multi_processor_count
    g = torch.Generator(device=gpu).manual_seed(S + H)
    m = _fill(P._Attention(cfg).to(gpu), g, gpu, lambda n: spread if "norm" in n else 0.06).to(dtype)
    ix = _fill(P._Indexer(cfg).to(gpu), g, gpu, lambda n: 0.1).to(dtype)
    x = torch.randn(B, S, 256, generator=g, device=gpu).to(dtype)
    cos, sin = P.rope_tables(cfg, S, dtype, gpu)
    with torch.no_grad():
        native, again = P._qsa(m, ix, x, cos, sin, cfg, True), P._qsa(m, ix, x, cos, sin, cfg, True)
        torch_code = P._qsa(m, ix, x, cos, sin, cfg)
        sel, _ = P._qsa_select(ix, x, cos, sin, cfg)
        exact = _qsa64(m, sel, x, cos, sin, cfg)
    assert native.dtype == dtype and torch.equal(native, again)
    _hold(native, torch_code, exact, "mixer output")


def test_trunk_choice(gpu):
    """Which forwards take the kernels: plain bf16 or fp32 parameters on the GPU without gradients. Others
    run the torch code, and gradients still flow through it."""
    cfg = P.PrefillConfig(vocab=128, hidden=128, layers=1, lin_k_heads=1, lin_v_heads=2, moe_ffn=64, shared_ffn=64,
                          ngram_rows=64, experts=8, topk=2)
    ids = torch.arange(70, device=gpu)[None] % 128
    model = P.build(cfg, device=gpu, dtype=torch.float32, moe_forward=lambda block, x: 0.1 * x)
    M = model.model
    with torch.no_grad():
        assert P._native_trunk(M, cfg, ids) and not P._native_trunk(M, cfg, ids.cpu())
    native = model(ids)
    # A trainable MoE callable over frozen parameters gets its gradient.
    scale = torch.tensor(0.1, device=gpu, requires_grad=True)
    P.trunk_forward(M, cfg, ids, lambda block, x, r: scale * x).square().mean().backward()
    assert float(scale.grad.abs()) > 0
    # Autocast hands the mixers bf16 activations beside fp32 parameters: the torch code takes them (bf16
    # products, 2^-8 each, through a dozen of them in a row).
    with torch.autocast("cuda", torch.bfloat16):
        cast = model(ids)
    assert _rel(cast.float(), native.double()) < 12 * 2**-8
    M.requires_grad_(True)
    assert not P._native_trunk(M, cfg, ids)
    hs = P.trunk_forward(M, cfg, ids, lambda block, x, r: 0.1 * x)
    (hs @ M.embed_tokens.weight.t()).square().mean().backward()
    assert float(M.mhc[0].A.weight.grad.norm()) > 0 and float(M.layers[0].linear_attn.A_log.grad.norm()) > 0
    with torch.no_grad():
        assert P._native_trunk(M, cfg, ids)
        M.requires_grad_(False)
        M.norm.to(torch.float64)
        assert not P._native_trunk(M, cfg, ids)
        M.norm.to(torch.float32)
    assert _rel(native, (hs @ M.embed_tokens.weight.t()).detach().double()) < 1e-5


def _small_model(gpu, moe_forward=lambda block, x: 0.1 * x):
    """A period of the layer pattern in fp32, with 70 tokens."""
    cfg = P.PrefillConfig(vocab=128, hidden=128, layers=4, heads=4, kv_heads=2, lin_k_heads=1, lin_v_heads=2,
                          moe_ffn=64, shared_ffn=64, ngram_rows=64, experts=8, topk=2)
    model = P.build(cfg, device=gpu, dtype=torch.float32, moe_forward=moe_forward)
    return cfg, model, torch.arange(70, device=gpu)[None] % 128


@pytest.mark.parametrize("default", [torch.bfloat16, torch.float64])
def test_trunk_default_dtype(gpu, default):
    """The stream is fp32 whatever torch's default dtype is."""
    _, model, ids = _small_model(gpu)
    expected = model(ids)
    torch.set_default_dtype(default)
    try:
        got = model(ids)
    finally:
        torch.set_default_dtype(torch.float32)
    assert torch.equal(got, expected)


def _off_boundary(t):
    """A contiguous copy of t that does not start on a 16-byte boundary: a view into a flat buffer."""
    v = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    assert v.is_contiguous() and v.data_ptr() % 16
    return v.copy_(t)


@pytest.mark.parametrize("name", ["layers.0.input_layernorm.weight", "layers.0.linear_attn.conv1d.weight",
                                  "layers.0.linear_attn.norm.weight", "layers.3.self_attn.q_norm.weight",
                                  "layers.3.self_attn.k_norm.weight"])
def test_trunk_unaligned_parameter(gpu, name):
    """A parameter may be a view into a flat buffer."""
    _, model, ids = _small_model(gpu)
    expected = model(ids)
    p = model.model.get_parameter(name)
    p.data = _off_boundary(p.data)
    assert torch.equal(model(ids), expected)


def test_trunk_unaligned_moe_output(gpu):
    """The MoE callable's output may be any view."""
    _, model, ids = _small_model(gpu)
    expected = model(ids)
    model.moe_forward = lambda block, x: _off_boundary(0.1 * x)
    assert torch.equal(model(ids), expected)


def test_trunk_broadcast_moe_output(gpu):
    """The MoE callable's output may be broadcast over tokens or features, as the torch code's products take it."""
    _, model, ids = _small_model(gpu)
    for dims in ((-1,), (1,), (0, 1, 2)):
        model.moe_forward = lambda block, x: x.mean(dims, keepdim=True)
        got = model(ids)
        model.moe_forward = lambda block, x: x.mean(dims, keepdim=True).expand_as(x).contiguous()
        assert torch.equal(got, model(ids))


@pytest.mark.parametrize("where,value", [("b_res", float("nan")), ("b_res", float("inf")), ("b_res", -float("inf")),
                                         ("b_pre", float("nan")), ("b_post", float("inf")), ("B.weight", float("nan")),
                                         ("X", float("nan")), ("X", float("inf"))])
def test_mhc_not_finite(gpu, where, value):
    """NaN and infinities come out of mhc_pre where the torch code has them: a NaN residual logit makes the
    token's whole mix NaN, for the maximum and the clamped sums keep it."""
    cfg = P.PrefillConfig(hidden=128, layers=1)
    g = torch.Generator(device=gpu).manual_seed(7)
    m = _fill(P._MHC(cfg).to(gpu), g, gpu, lambda n: {"A.weight": 0.02, "B.weight": 0.2}.get(n, 1.0))
    norm = _fill(P._Norm(128).to(gpu), g, gpu, lambda n: 0.05)
    X = torch.randn(1, 5, 4, 128, generator=g, device=gpu)
    t = X if where == "X" else m.get_parameter(where).data
    t.view(-1)[{"X": 900, "B.weight": 9 * cfg.mhc_rank + 2}.get(where, t.numel() // 2)] = value
    with torch.no_grad():
        x, (post, mix) = P._mhc_in(m, norm, X, X.pow(2).sum((2, 3)).view(-1), cfg, torch.float32)
        xt, (postt, mixt) = P._mhc_in(m, norm, X, None, cfg, torch.float32)
    for got, want, what in ((x, xt, "input"), (post, postt, "post"), (mix, mixt, "mix")):
        torch.testing.assert_close(got.view(want.shape), want, rtol=1e-4, atol=1e-5, equal_nan=True, msg=what)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_qsa_infinite_value(gpu, dtype):
    """An infinite value comes through the weighted sum as an infinity, as in a product of fp32
    probabilities, and not as the NaN of an infinity times a zero part of a probability."""
    from q38.hip import ops
    B, S, H, KV = 1, 192, 4, 2
    g = torch.Generator(device=gpu).manual_seed(3)
    r = lambda n, d=64: torch.randn(B, S, n, d, generator=g, device=gpu).to(dtype)
    q, k, v, qg = r(H), r(KV), r(KV), r(H, 128)
    v[0, 5, 0, 3], v[0, 9, 1, 40], v[0, 11, 1, 41] = float("inf"), -float("inf"), float("nan")
    sel = torch.arange(3, device=gpu).expand(B, 3, 3).contiguous()
    got = ops.qsa_attention(q, k, v, qg, sel, 0.125)
    valid = torch.ones(3, 3, dtype=torch.bool, device=gpu).tril()
    o = P.block_sparse_attention(*(t.transpose(1, 2) for t in (q, k, v)), sel, valid, 0.125)
    want = o.transpose(1, 2).reshape(B, S, H * 64) * torch.sigmoid(qg[..., 64:].reshape(B, S, H * 64))
    assert want.isinf().any() and want.isnan().any()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isposinf(), want.isposinf())
    assert torch.equal(got.isneginf(), want.isneginf())
    ok = want.isfinite()
    tol = 2e-5 if dtype == torch.float32 else 2**-7  # two bf16 roundings
    torch.testing.assert_close(got[ok], want[ok], rtol=tol, atol=tol * 1e-1)
