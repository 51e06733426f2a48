"""The BF16-MFMA perceptron kernels against the FP64 CPU reference
(tests/mlp_ref.py): the product kernel in its four operand layouts, the
forward pass, the loss gradient of every parameter, and Adam training."""
import gc

import numpy as np
import pytest

from . import mlp_ref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "GPU test without a HIP device"
    return torch


def _bf(torch, a):
    return torch.from_numpy(np.asarray(a, dtype=np.float32)).to(torch.bfloat16).cuda()


@pytest.mark.parametrize("a_kcontig,b_kcontig,M,N,K", [
    (True, True, 128, 192, 96), (True, True, 256, 256, 64), (True, True, 64, 128, 32), (True, False, 128, 192, 96),
    (False, True, 128, 192, 96), (False, False, 128, 192, 96)])
def test_gemm_layouts(torch_dev, a_kcontig, b_kcontig, M, N, K):
    """The product kernel in each operand layout and at several tile counts."""
    torch = torch_dev
    from tiger_nga_amd.mlp import MLP
    net = MLP(8, 8, 64, 1)
    rng = np.random.default_rng(7)
    A = rng.standard_normal((M, K))
    Bm = rng.standard_normal((K, N))
    Aq, Bq = mlp_ref.bf16(A), mlp_ref.bf16(Bm)
    if a_kcontig:
        Ad, sam, sak = _bf(torch, A), K, 1
    else:
        Ad, sam, sak = _bf(torch, A.T.copy()), 1, M
    if b_kcontig:
        Bd, sbk, sbn = _bf(torch, Bm.T.copy()), 1, K
    else:
        Bd, sbk, sbn = _bf(torch, Bm), N, 1
    C = torch.full((M, N), np.nan, dtype=torch.float32, device="cuda")
    net.gemm(Ad, sam, sak, Bd, sbk, sbn, M, N, K, C, N)
    torch.cuda.synchronize()
    ref = Aq @ Bq
    scale = np.abs(Aq) @ np.abs(Bq)
    err = np.abs(C.cpu().numpy() - ref) / scale
    assert err.max() < 1e-6, err.max()


def _net_case(torch, nin=38, nout=37, hidden=256, layers=4, B=128, seed=5):
    from tiger_nga_amd import mlp
    flat = mlp.init_params(nin, nout, hidden, layers, seed=seed)
    rng = np.random.default_rng(seed + 1)
    for l, (W, b) in enumerate(mlp.unflatten(flat, nin, nout, hidden, layers)):
        b[: (nout if l == layers else hidden)] = rng.standard_normal(nout if l == layers else hidden) * 0.05
    net = mlp.MLP(nin, nout, hidden, layers)
    net.set_params(flat)
    x = np.zeros((B, net.in_pad), dtype=np.float32)
    x[:, :nin] = rng.standard_normal((B, nin))
    tgt = rng.standard_normal((B, nout)).astype(np.float32) * 0.3
    params = mlp.unflatten(flat.astype(np.float64), nin, nout, hidden, layers)
    return net, flat, params, x, tgt


def test_forward_matches_reference(torch_dev):
    torch = torch_dev
    net, _, params, x, _ = _net_case(torch)
    out = net.forward(_bf(torch, x))
    torch.cuda.synchronize()
    ref, _, _ = mlp_ref.forward(params, x, quantize=True)
    got = out.cpu().numpy()
    err = np.abs(got - ref).max() / np.abs(ref).max()
    assert err < 5e-3, err   # bf16 activations: a rounding flip changes one activation by 2^-8
    assert np.all(got[:, 37:] == 0.0)
    exact, _, _ = mlp_ref.forward(params, x, quantize=False)
    print("\nforward: max rel err vs bf16-emulating FP64 %.2e, vs exact FP64 %.2e"
          % (err, np.abs(got - exact).max() / np.abs(exact).max()))


@pytest.mark.parametrize("B", [128, 1024])
def test_gradients_match_reference(torch_dev, B):
    """Every parameter's gradient: relative L2 error per tensor against the
    FP64 reference with the same bf16 rounding points (tight), and against
    the exact FP64 gradient of the same parameters (loose: bf16 operands)."""
    torch = torch_dev
    from tiger_nga_amd import mlp
    net, flat, params, x, tgt = _net_case(torch, B=B)   # B = 1024: weight gradients split over the batch
    g, loss = net.gradients(_bf(torch, x), torch.from_numpy(tgt).cuda())
    lq, gq = mlp_ref.loss_and_grad(params, x, tgt, 37, quantize=True)
    le, ge = mlp_ref.loss_and_grad(params, x, tgt, 37, quantize=False)
    assert abs(loss - lq) <= 1e-3 * lq, (loss, lq)
    got = mlp.unflatten(g, 38, 37, 256, 4)
    worst_q = worst_e = 0.0
    for l, ((dW, db), (rW, rb), (eW, eb)) in enumerate(zip(got, gq, ge)):
        for a, r, e in ((dW, rW, eW), (db, rb, eb)):
            nq = np.linalg.norm(a - r) / np.linalg.norm(r)
            ne = np.linalg.norm(a - e) / np.linalg.norm(e)
            worst_q, worst_e = max(worst_q, nq), max(worst_e, ne)
            assert nq < 1e-2, (l, nq)
            assert ne < 5e-2, (l, ne)
    print("\ngradients: loss %.6e (ref %.6e); worst rel L2 err vs bf16-emulating ref %.2e, vs exact FP64 %.2e"
          % (loss, lq, worst_q, worst_e))


def test_training_reduces_loss(torch_dev):
    """Adam on a smooth 38 -> 37 map: the loss falls by more than 20x."""
    torch = torch_dev
    from tiger_nga_amd import mlp
    nin, nout = 38, 37
    net = mlp.MLP(nin, nout, 256, 4)
    net.set_params(mlp.init_params(nin, nout, 256, 4, seed=9))
    rng = np.random.default_rng(10)
    P = rng.standard_normal((nin, nout)) / np.sqrt(nin)
    B = 2048
    x = np.zeros((B, net.in_pad), dtype=np.float32)
    x[:, :nin] = rng.uniform(-1, 1, (B, nin))
    tgt = np.tanh(x[:, :nin] @ P * 2.0).astype(np.float32)
    xd, td = _bf(torch, x), torch.from_numpy(tgt).cuda()
    l0 = net.train_step(xd, td, 1e-3, want_loss=True)
    for _ in range(400):
        net.train_step(xd, td, 1e-3)
    l1 = net.train_step(xd, td, 1e-3, want_loss=True)
    print("\ntraining: loss %.3e -> %.3e after 400 Adam steps" % (l0, l1))
    assert l1 < l0 / 20
    # the trained parameters round-trip through the host
    p = net.get_params()
    assert np.all(np.isfinite(p)) and p.size == net.nparam


@pytest.mark.parametrize("nin,nout,hidden,layers,B", [(8, 8, 64, 1, 64), (130, 200, 128, 2, 320), (38, 37, 256, 4, 8256),
                                                      (64, 256, 192, 3, 192), (38, 37, 320, 2, 128)])
def test_widths_and_batches(torch_dev, nin, nout, hidden, layers, B):
    """Forward and gradients at other widths (the last beyond the fused kernels),
    at batches of one 64-row tile, an odd number of 32-row slices and more
    than one row tile per CU; bounds as above."""
    torch = torch_dev
    from tiger_nga_amd import mlp
    net, flat, params, x, tgt = _net_case(torch, nin, nout, hidden, layers, B)
    got = net.forward(_bf(torch, x)).cpu().numpy()
    ref, _, _ = mlp_ref.forward(params, x, quantize=True)
    assert np.abs(got - ref).max() / np.abs(ref).max() < 5e-3 and np.all(got[:, nout:] == 0.0)
    g, loss = net.gradients(_bf(torch, x), torch.from_numpy(tgt).cuda())
    lq, gq = mlp_ref.loss_and_grad(params, x, tgt, nout, quantize=True)
    assert abs(loss - lq) <= 1e-3 * lq
    for (dW, db), (rW, rb) in zip(mlp.unflatten(g, nin, nout, hidden, layers), gq):
        for a, r in ((dW, rW), (db, rb)):
            assert np.linalg.norm(a - r) < 1e-2 * np.linalg.norm(r)


@pytest.mark.parametrize("B", [64, 320, 16448])
def test_fused_forward_equals_the_layered_one(torch_dev, B):
    """A network of 256 hidden units and the same one with 64 more of weight
    zero, which is too wide for the fused pass and goes layer by layer: the same
    products, sums, GELU and roundings, so the same outputs to the last bit."""
    torch = torch_dev
    from tiger_nga_amd import mlp
    net, flat, _, x, _ = _net_case(torch, B=B)
    wide = mlp.MLP(38, 37, 320, 4)
    wflat = np.zeros(wide.nparam, dtype=np.float32)
    for (W, b), (Wn, bn) in zip(mlp.unflatten(wflat, 38, 37, 320, 4), mlp.unflatten(flat, 38, 37, 256, 4)):
        W[:Wn.shape[0], :Wn.shape[1]] = Wn
        b[:bn.shape[0]] = bn
    wide.set_params(wflat)
    x = _bf(torch, 2.0 * x)
    assert torch.equal(net.forward(x), wide.forward(x))


@pytest.mark.parametrize("hidden", [256, 320])
def test_output_and_targets_at_any_offset(torch_dev, hidden):
    """Outputs and targets that are views one element past the start of a larger
    tensor, in the fused pass and layer by layer: the results of aligned ones,
    and nothing written outside.  Input rows must be 16-byte aligned."""
    torch = torch_dev
    from tiger_nga_amd import mlp
    net, _, _, x, tgt = _net_case(torch, hidden=hidden, B=192)
    x, tgt = _bf(torch, x), torch.from_numpy(tgt).cuda()
    want = net.forward(x)
    big = torch.full((want.numel() + 2,), 7.0, device="cuda")
    out = big[1:-1].view(want.shape)
    assert out.data_ptr() % 16 == 4
    assert torch.equal(net.forward(x, out=out), want) and float(big[0]) == float(big[-1]) == 7.0
    ts = torch.empty(tgt.numel() + 1, device="cuda")[1:].view(tgt.shape).copy_(tgt)
    for a, b in zip(net.gradients(x, tgt), net.gradients(x, ts)):
        assert np.array_equal(a, b)
    xs = torch.empty(x.numel() + 1, dtype=x.dtype, device="cuda")[1:].view(x.shape).copy_(x)
    for call in (lambda: net.forward(xs), lambda: net.gradients(xs, tgt), lambda: net.train_step(xs, tgt, 1e-3)):
        with pytest.raises(mlp.MLPError, match="16-byte aligned"):
            call()


def test_training_where_the_fused_workspace_does_not_fit(torch_dev):
    """A batch whose fused workspace (13.4 GB) is more than the free memory but
    whose layered one (10.0 GB) is not: the gradients, losses and trained
    parameters of the fused pass, then a small batch by the fused pass again."""
    torch = torch_dev
    from tiger_nga_amd import mlp
    B = 1 << 20
    nets = [_net_case(torch, B=64) for _ in range(2)]
    rng = torch.Generator(device="cuda").manual_seed(2)
    x = torch.zeros(B, 64, device="cuda", dtype=torch.bfloat16)
    x[:, :38] = torch.randn(B, 38, generator=rng, device="cuda").to(torch.bfloat16)
    tgt = torch.tanh(x[:, :37].float()).contiguous()

    def train(net):
        g, _ = net.gradients(x, tgt)
        losses = [net.train_step(x, tgt, 1e-3, want_loss=True) for _ in range(2)]
        small = [net.train_step(x[:256], tgt[:256], 1e-3, want_loss=True) for _ in range(2)]
        return g, np.array(losses + small), net.get_params()
    want = train(nets[0][0])
    nets[0][0].close()
    gc.collect()  # what earlier tests left
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hog, free0 = [], torch.cuda.mem_get_info()[0]
    while free0 > 11.8e9 and len(hog) < 8:  # memory freed before may come back late
        hog.append(torch.empty(free0 - int(11.7e9), dtype=torch.uint8, device="cuda"))
        torch.cuda.synchronize()
        free0 = torch.cuda.mem_get_info()[0]
    got = train(nets[1][0])
    taken = free0 - torch.cuda.mem_get_info()[0]
    del hog
    torch.cuda.empty_cache()
    assert free0 < 12.0e9 and 8.5e9 < taken < 10.6e9  # the layered workspace
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[2], want[2])
    assert np.abs(got[1] - want[1]).max() <= 1e-5 * want[1].max()  # sums of the squared errors in another order
