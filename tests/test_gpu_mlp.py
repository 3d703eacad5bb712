"""The surrogate network's matrix-core kernels against the CPU (FP32 torch).

* pywrf_mlp_gemm, every epilogue, at shapes that leave partial tiles in M
  and N and with split-K: equal to the FP32 product of the same BF16 values
  (to FP32 summation order; BF16 outputs to one BF16 rounding);
* one training step (forward, loss, backward: all parameter gradients) equal
  to torch autograd on the CPU in FP32 of the same network, with the same
  BF16 roundings of the operands the kernels round (weights, inputs, hidden
  activations, output and hidden gradients);
* Adam equal to torch.optim.Adam.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bf(x):
    return x.to(torch.bfloat16)


def _rel(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return float((a - b).abs().max() / max(b.abs().max(), 1e-30))


@pytest.mark.parametrize("M,N,K,ksplit", [(256, 128, 64, 1), (300, 200, 96, 1), (1000, 288, 512, 1),
                                          (96, 512, 4096, 8), (51529 % 4096 + 7, 384, 384, 1),
                                          (700, 512, 288, 1), (512, 288, 8192, 16)])
def test_gemm_matches_cpu(M, N, K, ksplit):
    from pywrf_amd import surrogate as sg
    gen = torch.Generator().manual_seed(M * 7 + N)
    A = _bf(torch.randn(M, K, generator=gen))
    B = _bf(torch.randn(N, K, generator=gen))
    bias = torch.randn(N, generator=gen)
    ref = A.float() @ B.float().t()
    Ad, Bd, biasd = A.cuda(), B.cuda(), bias.cuda()
    if ksplit == 1:
        C = torch.full((M, N), 7.0, device="cuda")
        sg.gemm(0, Ad, Bd, C, biasd)
        assert _rel(C, ref + bias) < 1e-5
        Cb = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
        sg.gemm(1, Ad, Bd, Cb, biasd)
        want = torch.relu(ref + bias)
        assert _rel(Cb.float(), want) < 1e-2
        # one BF16 rounding: |Cb - want| <= 2^-8 |want| (+ summation-order slack)
        assert bool(((Cb.float().cpu() - want).abs() <= 2 ** -8 * want.abs() + 1e-3 * want.abs().max()).all())
        H = _bf(torch.randn(M, N, generator=gen))
        Cd = torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")
        sg.gemm(2, Ad, Bd, Cd, H=H.cuda())
        want = ref * (H.float() > 0)
        assert _rel(Cd.float(), want) < 1e-2
        Ct = torch.full((N, M + 5), 3.0, device="cuda")
        sg.gemm(4, Ad, Bd, Ct, biasd)
        assert _rel(Ct[:, :M].t(), ref + bias) < 1e-5
        assert bool((Ct[:, M:] == 3.0).all())
    C = torch.zeros(M, N, device="cuda")
    sg.gemm(3, Ad, Bd, C, ksplit=ksplit)
    assert _rel(C, ref) < 1e-5


def test_transpose_and_rowsum():
    from pywrf_amd import surrogate as sg
    x = _bf(torch.randn(300, 200)).cuda()
    t = torch.zeros(200, 300, dtype=torch.bfloat16, device="cuda")
    sg.transpose(x, t)
    assert torch.equal(t.cpu(), x.cpu().t())
    r = torch.zeros(300, device="cuda")
    sg.rowsum(x, r)
    assert _rel(r, x.float().cpu().sum(1)) < 1e-5


def _cpu_reference_step(net, X, T, w):
    """Forward / backward of the network in FP32 torch autograd on the CPU,
    rounding to BF16 where the kernels store BF16: weights, inputs, the
    hidden activations after ReLU, the output gradient and the hidden
    gradients."""
    W = [torch.nn.Parameter(_bf(x.cpu()).float()) for x in net.W]
    b = [torch.nn.Parameter(x.cpu().clone()) for x in net.b]

    class Round(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return _bf(x).float()

        @staticmethod
        def backward(ctx, g):
            return _bf(g).float()

    x = X.cpu().float()
    h1 = Round.apply(torch.relu(x @ W[0].t() + b[0]))
    h2 = Round.apply(torch.relu(h1 @ W[1].t() + b[1]))
    y = h2 @ W[2].t() + b[2]
    wc = w.cpu()
    M = x.shape[0]
    loss = ((y - T.cpu()) ** 2 * wc).sum() / (M * float(wc.sum()))
    y.register_hook(lambda g: _bf(g).float())
    loss.backward()
    return float(loss), [p.grad for p in W], [p.grad for p in b]


def test_training_step_gradients_match_cpu_autograd():
    from pywrf_amd import surrogate as sg
    M = 512
    gen = torch.Generator().manual_seed(3)
    net = sg.MLP(seed=5)
    for n in range(3):                       # non-zero biases
        net.b[n].copy_(0.1 * torch.randn(net.b[n].shape[0], generator=gen))
    net.b[2][sg.FOUT:] = 0.0
    X = torch.zeros(M, sg.KIN, dtype=torch.bfloat16)
    X[:, :sg.FIN] = _bf(torch.randn(M, sg.FIN, generator=gen))
    T = torch.zeros(M, sg.NO)
    T[:, :sg.FOUT] = torch.randn(M, sg.FOUT, generator=gen)
    w = sg.loss_weights("cpu")
    ws = sg.Workspace(M)
    Xd, Td, wd = X.cuda(), T.cuda(), w.cuda()
    sg.forward(net, Xd, ws)
    loss = float(sg.backward(net, Xd, Td, wd, ws, float(w.sum()), ksplit=4)[0])
    ref_loss, gW, gb = _cpu_reference_step(net, X, T, w)
    print("loss", loss, ref_loss)
    assert abs(loss - ref_loss) <= 1e-4 * ref_loss
    for n in range(3):
        eW, eb = _rel(ws.gW[n], gW[n]), _rel(ws.gb[n], gb[n])
        print("layer", n + 1, "dW %.2e  db %.2e" % (eW, eb))
        assert eW < 2e-3 and eb < 2e-3
    # padded input columns and the padded output row get zero gradient
    assert float(ws.gW[0][:, sg.FIN:].abs().max()) == 0.0
    assert float(ws.gW[2][sg.FOUT:].abs().max()) == 0.0


def test_adam_matches_torch():
    from pywrf_amd import surrogate as sg
    net = sg.MLP(seed=1)
    ws = sg.Workspace(32)
    p = [torch.nn.Parameter(x.cpu().clone()) for x in net.W + net.b]
    opt = torch.optim.Adam(p, lr=1e-3)
    gen = torch.Generator().manual_seed(0)
    for _ in range(3):
        grads = [torch.randn(x.shape, generator=gen) for x in p]
        for q, g in zip(p, grads):
            q.grad = g.clone()
        opt.step()
        for n in range(3):
            ws.gW[n].copy_(grads[n])
            ws.gb[n].copy_(grads[3 + n])
        sg.adam_step(net, ws, 1e-3)
    for mine, ref in zip(net.W + net.b, p):
        assert _rel(mine, ref.detach()) < 1e-5
    assert torch.equal(net.Wb[1].cpu(), _bf(net.W[1].cpu()))
    assert torch.equal(net.Wt[2].cpu(), _bf(net.W[2].cpu()).t())


@pytest.mark.parametrize("shapes", [[(64, 64)], [(8, 8), (72, 200), (300, 201), (129, 136)]])
def test_grouped_calls_and_conversion(shapes):
    """Matrices of aligned and ragged sides in one launch; FP32 rows of any
    length (and any row stride) into padded BF16 rows: the same bits as torch."""
    from pywrf_amd import surrogate as sg
    gen = torch.Generator().manual_seed(len(shapes))
    xs = [_bf(torch.randn(r, c, generator=gen)).cuda() for r, c in shapes]
    ts = [torch.zeros(c, r, dtype=torch.bfloat16, device="cuda") for r, c in shapes]
    sg.transpose_group(list(zip(xs, ts)))
    rs = [torch.zeros(r, device="cuda") for r, _ in shapes]
    sg.rowsum_group(list(zip(xs, rs)))
    for x, t, r in zip(xs, ts, rs):
        assert torch.equal(t.cpu(), x.cpu().t())
        # FP32 sums of at most 256 values: c eps / 2 of the sum of magnitudes, far below this
        assert float((r.cpu() - x.cpu().double().sum(1)).abs().max()) <= 1e-5 * float(x.cpu().double().abs().sum(1).max())
    for N, cols in ((287, 288), (369, 384), (5, 8), (600, 640)):
        x = torch.randn(7, N + 3, generator=gen).cuda()[:, :N]
        for y in (x, x[:1].expand(7, N), x.t().contiguous().t()):
            want = torch.zeros(7, cols, dtype=torch.bfloat16, device="cuda")
            want[:, :N] = y.to(torch.bfloat16)
            assert torch.equal(sg.to_bf16(y, cols), want)


@pytest.mark.parametrize("N,ldy", [(287, 288), (7, 9), (1, 4)])
def test_mse_rows_of_any_length(N, ldy):
    from pywrf_amd import surrogate as sg
    from pywrf_amd._lib import call, stream
    gen = torch.Generator().manual_seed(N)
    B = 700
    Y, T = torch.randn(B, ldy, generator=gen).cuda(), torch.randn(B, ldy, generator=gen).cuda()
    w = torch.rand(ldy, generator=gen).cuda()
    dY = torch.full((B, ldy), 7.0, dtype=torch.bfloat16, device="cuda")
    loss = torch.zeros(1, device="cuda")
    call("pywrf_mlp_mse", B, N, sg._vp(Y), ldy, sg._vp(T), ldy, sg._vp(w), 0.01, sg._vp(dY), ldy, sg._vp(loss), stream())
    d = (Y - T).double()[:, :N]
    # positive terms, FP32 sums over at most B N / 256 of them a workgroup: a few hundred roundings
    assert abs(float(loss) / float((w[:N] * d * d).sum() * 0.01) - 1) < 1e-5
    want = (2.0 * w[:N] * (Y - T)[:, :N] * 0.01)
    assert float((dY[:, :N].float() - want).abs().max()) <= 2 ** -8 * float(want.abs().max())
    assert bool((dY[:, N:] == 0).all())


@pytest.mark.parametrize("shape", [(32, 368), (32, 370), (32, 384), (64, 2), (32, 369, 1), (32,)])
def test_column_network_refuses_other_widths(shape):
    from pywrf_amd import adjoint, surrogate as sg
    net = sg.MLP(seed=1)
    with pytest.raises((ValueError, RuntimeError)):
        adjoint.SurrogateNet.apply(torch.zeros(shape, device="cuda"), net)


@pytest.mark.parametrize("M,splits", [(32, 1), (96, 1), (1024, 4), (4128, 8), (70048, 32)])
def test_weight_gradients_in_any_number_of_splits(M, splits):
    from pywrf_amd import surrogate as sg
    assert sg.weight_splits(M) == splits
    net, ws, w = sg.MLP(seed=2), sg.Workspace(M), sg.loss_weights()
    gen = torch.Generator(device="cuda").manual_seed(M)
    X = _bf(torch.randn(M, sg.KIN, device="cuda", generator=gen))
    T = torch.randn(M, sg.NO, device="cuda", generator=gen)
    sg.forward(net, X, ws)
    sg.backward(net, X, T, w, ws, float(w.sum()))
    got = [g.clone() for g in ws.gW]
    sg.backward(net, X, T, w, ws, float(w.sum()), ksplit=1)
    for n, (a, b) in enumerate(zip(got, ws.gW)):
        # FP32 sums over M terms in two orders: within sqrt(M) eps / 2 of the terms' root of summed squares each,
        # here over whole matrices of such sums
        assert float((a - b).norm()) <= 2 * M ** 0.5 * 6e-8 * float(b.norm()), n
