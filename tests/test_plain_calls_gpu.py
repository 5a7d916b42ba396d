"""The native one-call forms behind ops.ternary_linear, ternary_conv2d, ternary_dwconv2d, softstep_fwd_all and
softstep_bwd_all (torch_ext.cpp, plain_*) against the ctypes route they stand in for: the same kernels on the same data, so
the same bits, over types, layouts, epilogues and sizes -- and None, with nothing else done, for what is not the plain case."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def by_ctypes(monkeypatch):
    """Runs a call with the extension out of the way."""
    from tmq_amd import ops
    assert ops.ext is not None

    def run(fn, *a, **kw):
        with monkeypatch.context() as m:
            m.setattr(ops, "ext", None)
            return fn(*a, **kw)

    return run


def _weights(cuda, shape, seed):
    from tmq_amd import ops
    g = torch.Generator(device=cuda).manual_seed(seed)
    return ops.compactify_ternary(torch.randint(-1, 2, shape, device=cuda, generator=g).float())


@pytest.mark.parametrize("M,K,N", [(1, 4096, 512), (2, 512, 64), (5, 1000, 70), (17, 2048, 256), (33, 100, 64), (300, 192, 130), (1100, 128, 16)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_linear(cuda, by_ctypes, M, K, N, dtype):
    from tmq_amd import ops
    g = torch.Generator(device=cuda).manual_seed(M + K)
    nw = ops.NativeWeights(_weights(cuda, (N, K), K), N)
    scale, bias = torch.rand(N, device=cuda, generator=g) + 0.5, torch.randn(N, device=cuda, generator=g)
    for out in (torch.float32, torch.float16):
        res = torch.randn((M, N), device=cuda, generator=g).to(out)
        for shift in (0, 1):                               # a base that is not 16-byte aligned
            x = torch.randn(M * K + shift, device=cuda, generator=g).to(dtype)[shift:].view(M, K)
            for kw in ({}, {"scale": scale, "bias": bias}, {"bias": bias, "residual": res, "relu": True}):
                want = by_ctypes(ops.ternary_linear, x, nw, out_dtype=out, **kw)
                assert torch.equal(ops.ternary_linear(x, nw, out_dtype=out, **kw), want)
                prev = ops.set_fp32_prescale(False)
                try:
                    assert torch.equal(ops.ternary_linear(x, nw, out_dtype=out, **kw), by_ctypes(ops.ternary_linear, x, nw, out_dtype=out, **kw))
                finally:
                    ops.set_fp32_prescale(prev)


@pytest.mark.parametrize("B,C,H,W,N,k,s,p,d", [(2, 64, 9, 7, 48, 3, 1, 1, 1), (1, 20, 8, 8, 33, 3, 2, 1, 1), (3, 7, 5, 6, 5, 1, 1, 0, 1),
                                               (2, 32, 10, 11, 32, 3, 1, ((2, 0), (1, 3)), 2)])
@pytest.mark.parametrize("depthwise", [False, True])
def test_convolutions(cuda, by_ctypes, B, C, H, W, N, k, s, p, d, depthwise):
    from tmq_amd import ops
    g = torch.Generator(device=cuda).manual_seed(C + N)
    N = C if depthwise else N
    words = _weights(cuda, (N, 1 if depthwise else C, k, k), C)
    call, w = (ops.ternary_dwconv2d, words) if depthwise else (ops.ternary_conv2d, ops.NativeWeights(words, N, (k, k)))
    args = ((k, k), s, p, d) if depthwise else (s, p, d)
    scale, bias = torch.rand(N, device=cuda, generator=g) + 0.5, torch.randn(N, device=cuda, generator=g)
    base = torch.randn((B, C, H, W), device=cuda, generator=g)
    last = base.contiguous(memory_format=torch.channels_last)
    for x in (base, last, base.half(), last.half(), base.transpose(2, 3).contiguous().transpose(2, 3)):
        for out in (torch.float32, torch.float16):
            want = by_ctypes(call, x, w, *args, scale=scale, bias=bias, out_dtype=out)
            got = call(x, w, *args, scale=scale, bias=bias, out_dtype=out)
            assert torch.equal(got, want) and got.stride() == want.stride()
            res = torch.randn(want.shape, device=cuda, generator=g).to(out).contiguous(memory_format=torch.channels_last)
            assert torch.equal(call(x, w, *args, bias=bias, residual=res, relu=True, out_dtype=out),
                               by_ctypes(call, x, w, *args, bias=bias, residual=res, relu=True, out_dtype=out))
    with pytest.raises(RuntimeError):
        call(base[0] if depthwise else base[:, :-1], w, *args)
    with pytest.raises(RuntimeError):
        call(last.half(), w, *args, residual=torch.zeros(1, device=cuda))
    with pytest.raises(RuntimeError):
        call(last.half(), w, *args, scale=scale.cpu())


def test_soft_weights(cuda, by_ctypes):
    from tmq_amd import ops
    g = torch.Generator(device=cuda).manual_seed(1)
    ws = [2.2 * torch.rand(n, device=cuda, generator=g) - 1.1 for n in [(5,), (3, 7), (64, 3, 3, 3), (100003,)]]
    gs = [torch.randn(w.shape, device=cuda, generator=g) for w in ws]
    up = torch.full((1,), 0.7, device=cuda)
    for want_loss in (False, True):
        ys, loss = ops.softstep_fwd_all(ws, 3.5, want_loss, 5.0, 1e-3)
        ys2, loss2 = by_ctypes(ops.softstep_fwd_all, ws, 3.5, want_loss, 5.0, 1e-3)
        assert all(torch.equal(a, b) and a.stride() == b.stride() for a, b in zip(ys, ys2)) and len(ys) == len(ys2)
        assert (loss is None) == (not want_loss) and (loss is None or (loss.shape == loss2.shape and torch.equal(loss, loss2)))
        assert len({y.data_ptr() for y in ys}) == len(ys) and all(y.data_ptr() % 256 == 0 and not y.requires_grad for y in ys)
        ys[0].add_(1.0)                                    # tensors of their own: a write bumps its own version only
        assert ys[0]._version == 1 and ys[1]._version == 0
    for upstream in (None, up):
        for grads in (gs, [None] + gs[1:], [gs[0], gs[1].t().contiguous().t()] + gs[2:]):
            a = ops.softstep_bwd_all(ws, grads, upstream, 3.5, 5.0, 1e-3)
            b = by_ctypes(ops.softstep_bwd_all, ws, grads, upstream, 3.5, 5.0, 1e-3)
            assert all((p is None and q is None) or torch.equal(p, q) for p, q in zip(a, b)) and len(a) == len(b)
    strided = ws[1].t()
    assert torch.equal(ops.softstep_fwd_all([strided], 3.5)[0][0], by_ctypes(ops.softstep_fwd_all, [strided], 3.5)[0][0])
    with pytest.raises(ValueError):
        ops.softstep_fwd_all([], 3.5)
    with pytest.raises(ValueError):
        ops.softstep_fwd_all([ws[0].half()], 3.5)
    with pytest.raises(RuntimeError):
        ops.softstep_fwd_all([ws[0].cpu()], 3.5)


def test_linear_form_is_taken_and_declined(cuda):
    """plain_linear itself: a tensor for the plain case, None for everything else."""
    from tmq_amd import ops
    K, N = 512, 48
    nw = ops.NativeWeights(_weights(cuda, (N, K), 1), N)
    call = lambda x, scale=None, bias=None, residual=None, prescale=True: ops.ext.plain_linear(x, nw.buf, K, N, scale, bias, residual, False, False,
                                                                                               prescale)
    row, per = torch.randn(3, K, device=cuda), torch.ones(N, device=cuda)
    for x in (row, row[:1], row.half(), row[0], row.half().view(1, 3, K), torch.randn(40, K, device=cuda), torch.randn(40, K, device=cuda).half()):
        y = call(x, per, per)
        assert y is not None and y.shape == x.shape[:-1] + (N,)
        assert torch.equal(y, ops.ternary_linear(x, nw, scale=per, bias=per))
    flat = torch.randn(3 * K + 1, device=cuda)
    res = torch.zeros(3, N, device=cuda)
    assert call(row, residual=res) is not None
    for declined in (lambda: call(flat[1:].view(3, K)),                          # fp32 rows off a 16-byte boundary: the splitter's route
                     lambda: call(torch.randn(1100, K, device=cuda), prescale=False),     # the one-pass kernel's
                     lambda: call(row.double()), lambda: call(row.cpu()), lambda: call(row.t().contiguous().t()), lambda: call(row[:0]),
                     lambda: call(row[:, :-1].contiguous()), lambda: call(row, scale=per.cpu()), lambda: call(row, bias=per.double()),
                     lambda: call(row, scale=per[:-1]), lambda: call(row, bias=torch.ones(2 * N, device=cuda)[::2]),
                     lambda: call(row, residual=res[:2]), lambda: call(row, residual=res.half()), lambda: call(row, residual=res.t().contiguous().t())):
        assert declined() is None


@pytest.mark.parametrize("depthwise", [False, True])
def test_convolution_form_is_taken_and_declined(cuda, depthwise):
    from tmq_amd import ops
    C = 24
    N = C if depthwise else 40
    words = _weights(cuda, (N, 1 if depthwise else C, 3, 3), 2)
    w = words if depthwise else ops.NativeWeights(words, N, (3, 3)).buf
    geometry = (1, 1, 1, 1, 1, 1, 1, 1)
    call = lambda x, scale=None, bias=None, residual=None, prescale=True, words=w, geometry=geometry: \
        ops.ext.plain_conv(x, words, depthwise, C, N, 3, 3, geometry, scale, bias, residual, False, False, prescale)
    planar = torch.randn(2, C, 9, 8, device=cuda)
    last, per = planar.contiguous(memory_format=torch.channels_last), torch.ones(N, device=cuda)
    for x in (planar, last, last.half()):
        y = call(x, per, per)
        assert y is not None and y.shape == (2, N, 9, 8) and y.is_contiguous(memory_format=torch.channels_last)
    res = torch.zeros_like(y)
    assert call(last, residual=res) is not None and call(last.half(), prescale=False) is not None
    for declined in (lambda: call(planar.half()), lambda: call(planar, prescale=False), lambda: call(last.cpu()), lambda: call(last.double()),
                     lambda: call(planar.transpose(2, 3)), lambda: call(planar[0]), lambda: call(planar[:0]), lambda: call(planar[:, :-1].contiguous()),
                     lambda: call(last, scale=per.cpu()), lambda: call(last, bias=per[:-1]), lambda: call(last, scale=per.double()),
                     lambda: call(last, residual=res.contiguous()), lambda: call(last, residual=res[:1]), lambda: call(last, residual=res.half()),
                     lambda: call(last, words=w.cpu()), lambda: call(last, geometry=(1, 1, -9, 1, -9, 1, 1, 1))):
        assert declined() is None


def test_soft_weight_forms_are_taken_and_declined(cuda):
    from tmq_amd import ops
    ws = [torch.rand(n, device=cuda) for n in (5, 4096)]
    gs = [torch.randn_like(w) for w in ws]
    up = torch.ones(1, device=cuda)
    fwd = lambda w, loss=True: ops.ext.plain_softstep_fwd(w, 3.5, loss, 5.0, 1e-3)
    bwd = lambda w, g, u=None: ops.ext.plain_softstep_bwd(w, g, u, 3.5, 5.0, 1e-3)
    assert fwd(ws) is not None and fwd(ws, False)[1] is None and bwd(ws, gs) is not None and bwd(ws, gs, up) is not None
    many = [torch.rand(7, device=cuda) for _ in range(100)]                      # beyond the in-launch loss: with a workspace
    ys, loss = fwd(many)
    assert len(ys) == 100 and abs(loss.item() - sum(fwd([w])[1].item() for w in many)) <= 1e-5 * abs(loss.item())
    square = torch.rand(8, 8, device=cuda)
    for declined in (lambda: fwd([]), lambda: fwd([ws[0], ws[1].half()]), lambda: fwd([ws[0].cpu()]), lambda: fwd([square.t()]),
                     lambda: bwd(ws, gs[:1]), lambda: bwd(ws, [gs[0], gs[1].half()]), lambda: bwd(ws, [gs[1], gs[0]]),
                     lambda: bwd(ws, [gs[0], gs[1].cpu()]), lambda: bwd([square], [square.t()]), lambda: bwd(ws, gs, up.cpu()),
                     lambda: bwd(ws, gs, up.double()), lambda: bwd(ws, gs, torch.ones(2, device=cuda))):
        assert declined() is None
