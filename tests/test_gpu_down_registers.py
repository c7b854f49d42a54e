"""The down GEMM with its weights in registers (q38moe_gemm_wr.hip), through the stage entry points, where
its tiles and runs can go wrong: groups without rows, of one row, of exactly a tile and one more; columns
that fill part of a wave's or of a workgroup's block; every row length; one group over many runs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _routing(E, k, T, sizes, g):
    """Indices [T,k] whose experts 0, 1, ... get the given numbers of pairs, the rest spread evenly."""
    flat = torch.randint(len(sizes), E, (T * k,), generator=g, dtype=torch.int32)
    order = torch.randperm(T * k, generator=g)
    at = 0
    for e, n in enumerate(sizes):
        flat[order[at:at + n]] = e
        at += n
    return flat.view(T, k)


def _assert_rounded(actual, x, w, allowance, what):
    """|actual - exact| <= one bf16 ulp of the exact value + allowance * sum |x w|."""
    x, w = x.double(), w.double()
    exact = x @ w.t()
    ulp = torch.pow(2.0, torch.floor(torch.log2(exact.abs().clamp_min(1e-38))) - 7)
    excess = (actual.double() - exact).abs() - ulp - allowance * (x.abs() @ w.abs().t())
    assert float(excess.max()) <= 0, f"{what}: worst excess {float(excess.max()):.3e}"


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("E,k,T,K,N,sizes,shared", [
    (6, 2, 800, 256, 64, (0, 1, 64, 65), False),      # one active wave; empty, single-row and tile-edge groups
    (9, 3, 700, 384, 576, (63, 0, 128, 129), True),   # a second column block of one wave
    (64, 5, 2600, 512, 1024, (0, 1, 2, 700), True),   # runs that cross groups and column blocks
    (3, 1, 5000, 512, 1088, (), True)])               # few groups, each over many runs
def test_down(gpu, fp8, E, k, T, K, N, sizes, shared):
    """K in e4m3 values (half as many in bf16: the same row lengths). Each value within one bf16 rounding of
    the exact product plus an accumulation allowance: 2^-20 of the sum of |a w| for fp32 sums; 2^-16 for
    e4m3, whose MFMA aligns the 128 products it adds to the largest of them before it sums (2^-17.7 seen,
    on values near zero; the 32x32x64 form of the other kernels gives the same bits)."""
    from q38.hip import ops
    g = torch.Generator().manual_seed(T + K)
    I = K if fp8 else K // 2
    idx = _routing(E, k, T, sizes, g)
    rows = T * k + (T if shared else 0)
    assert rows >= 160 * (E + 1), "the shape must take the kernel under test"
    H = torch.randn(rows, I, generator=g).to(torch.bfloat16)
    W = (torch.randn(E, N, I, generator=g) * 0.05).to(torch.bfloat16)
    Ws = (torch.randn(N, I, generator=g) * 0.05).to(torch.bfloat16)
    di = idx.to(gpu)
    sr = T if shared else 0
    counts, starts, _, _, tiles, tc = ops.permute(di, ops.histogram(di, E), E, sr)
    if fp8:
        (hq, hs), (wq, ws), (sq, ss) = (ops.quantize_rows(t.to(gpu)) for t in (H, W, Ws))
        Y = ops.down_fp8(hq, hs, {"experts.down_proj": (wq, ws), "shared_expert.down_proj.weight": (sq, ss)}, tiles, tc,
                         T, k, shared_rows=sr).cpu()
        H, W, Ws = (q.view(torch.float8_e4m3fn).cpu().double() * s.cpu().double()[..., None]
                    for q, s in ((hq, hs), (wq, ws), (sq, ss)))
    else:
        Y = ops.down(H.to(gpu), W.to(gpu), tiles, tc, T, k, w_shared_down=Ws.to(gpu), shared_rows=sr).cpu()
    st, ct = starts.cpu().tolist(), counts.cpu().tolist()
    assert ct[:len(sizes)] == list(sizes)
    allowance = 2.0 ** (-16 if fp8 else -20)
    for e in range(E):
        if ct[e]:
            _assert_rounded(Y[st[e]:st[e] + ct[e]], H[st[e]:st[e] + ct[e]], W[e], allowance, f"expert {e}")
    if shared:
        _assert_rounded(Y[T * k:], H[T * k:], Ws, allowance, "shared expert")


@pytest.mark.parametrize("fp8", [False, True])
def test_down_tile_count(gpu, fp8):
    """Entries past *tile_count count for nothing, whatever a reused table still holds there."""
    from q38.hip import ops
    E, k, T, N, I = 6, 2, 800, 128, 256
    g = torch.Generator().manual_seed(1)
    idx = _routing(E, k, T, (0, 1, 300), g).to(gpu)
    H, W = (torch.randn(*s, generator=g).to(torch.bfloat16).to(gpu) for s in ((T * k, I), (E, N, I)))
    _, _, _, _, tiles, tc = ops.permute(idx, ops.histogram(idx, E), E)
    if fp8:
        (hq, hs), w = ops.quantize_rows(H), ops.quantize_rows(W)
        wq = {"experts.down_proj": w, "shared_expert.down_proj.weight": tuple(t[0].contiguous() for t in w)}
        run = lambda: ops.down_fp8(hq, hs, wq, tiles, tc, T, k)
    else:
        run = lambda: ops.down(H, W, tiles, tc, T, k)
    expected = run()
    assert int(tc) < len(tiles)
    tiles[int(tc):] = tiles[0]
    assert torch.equal(run(), expected)


@pytest.mark.parametrize("h,Is,rows", [
    (320, 128, (1, 64, 65, 129)),         # part of one column block
    (576, 256, (1, 64, 128, 129, 200)),   # a second block of one wave; both sides of 128 rows
    (768, 192, (128, 129, 7616, 7617, 16384, 16385)),  # both sides of one and two tiles per CU (256 CUs)
    (1024, 256, (1, 65, 5003))])
def test_down_dense(gpu, h, Is, rows):
    """Dense ranges (a shared expert by itself), from one row on, at the bar of test_down."""
    from q38.hip import ops
    g = torch.Generator().manual_seed(h)
    wg, wu, wd = ((torch.randn(*s, generator=g) * 0.05).to(torch.bfloat16).to(gpu) for s in ((Is, h), (Is, h), (h, Is)))
    ptr = lambda t: t.data_ptr()
    for T in rows:
        x = torch.randn(T, h, generator=g).to(torch.bfloat16).to(gpu)
        H, out = torch.empty(T, Is, dtype=torch.bfloat16, device=gpu), torch.empty_like(x)
        rc = ops.lib.q38moe_shared_expert(ptr(x), ptr(wg), ptr(wu), ptr(wd), ptr(H), ptr(out), T, h, Is, ops.BF16,
                                          torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        _assert_rounded(out, H, wd, 2.0**-20, f"{T} rows")


@pytest.mark.parametrize("T", [1, 130, 3000])
def test_down_dense_in_block(gpu, T):
    """The dense range of a block with 64 experts: with routed experts that give zeros and a shared gate of
    1/2, the block's output is half the shared expert's, bit for bit."""
    from q38.hip import ops
    E, k, h, I, Is = 64, 2, 512, 128, 256
    g = torch.Generator().manual_seed(T)
    r = lambda *s: (torch.randn(*s, generator=g) * 0.05).to(torch.bfloat16).to(gpu)
    x, wr, wgu, wg, wu, wd = r(T, h) * 20, r(E, h), r(E, 2 * I, h), r(Is, h), r(Is, h), r(h, Is)
    wdn, gate = torch.zeros(E, h, I, dtype=torch.bfloat16, device=gpu), torch.zeros(1, h, dtype=torch.bfloat16, device=gpu)
    with torch.inference_mode():
        out = ops.block_forward(x, wr, wgu, wdn, wg, wu, wd, gate, k)
        assert torch.equal(out, ops.shared_expert(x, wg, wu, wd) * 0.5)
