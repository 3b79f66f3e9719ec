"""GPU numerics of the U-Net kernels (csrc/unet.hip) against a plain
PyTorch FP32 reference of the same operations, computed on the CPU from the
same bf16-valued inputs and weights.

Bar: the kernels accumulate in FP32 on the matrix cores, in a different
order than the reference, so results agree to FP32 rounding of the sums
(relative 1e-4 of the output scale for one layer); whole-network results,
whose activations are rounded to bf16 between layers, agree to 2e-2 of the
output scale (a bf16 rounding flip of one activation moves the rest)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bf(t):
    import torch
    return t.to(torch.bfloat16).to(torch.float32)


def _ref_conv(x_nhwc, w_ck, b, cin, cout, relu):
    """x (n, h, w, cin) fp32, w [cout][9*cin] (k = tap*cin + ci) -> NHWC."""
    import torch
    import torch.nn.functional as F
    wt = w_ck.reshape(cout, 3, 3, cin).permute(0, 3, 1, 2).contiguous()
    y = F.conv2d(x_nhwc.permute(0, 3, 1, 2), wt, b, padding=1).permute(0, 2, 3, 1)
    return torch.relu(y) if relu else y


def _effective(x1, mode, x2):
    """The convolution's input: x1 through its mode, then x2's channels."""
    import torch
    import torch.nn.functional as F
    if mode == 1:
        x1 = _pool(x1)
    elif mode == 2:
        x1 = F.interpolate(x1.permute(0, 3, 1, 2), scale_factor=2,
                           mode="nearest").permute(0, 2, 3, 1)
    return torch.cat([x1, x2], dim=3) if x2 is not None else x1


def _pool(x):
    n, h, w, c = x.shape
    t = x.reshape(n, h // 2, 2, w // 2, 2, c)
    s = (t[:, :, 0, :, 0] + t[:, :, 0, :, 1]) + (t[:, :, 1, :, 0] + t[:, :, 1, :, 1])
    return _bf(s * 0.25)


def _dev(t, dtype=None):
    import torch
    return t.to(dtype or torch.bfloat16).to("cuda").contiguous()


def _conv_gpu(L, x1, c1, mode, x2, c2, wb, bias, cout, kpad, n, h, w, relu):
    import ctypes as C

    import torch
    out = torch.empty(n, h, w, cout, dtype=torch.float32, device="cuda")
    rc = L.m2d_unet_conv3x3(C.c_void_p(x1.data_ptr()), c1, mode,
                            C.c_void_p(x2.data_ptr()) if x2 is not None else None, c2,
                            C.c_void_p(wb.data_ptr()),
                            C.c_void_p(bias.data_ptr()) if bias is not None else None,
                            cout, cout, kpad, n, h, w, relu, None, C.c_void_p(out.data_ptr()), 0,
                            None)
    assert rc == 0
    torch.cuda.synchronize()
    return out.cpu()


CONV_CASES = [  # n, h, w, c1, mode, c2, cout, relu
    (2, 16, 24, 8, 0, 0, 16, 1), (1, 8, 8, 16, 1, 0, 32, 1), (2, 8, 16, 32, 2, 16, 16, 1),
    (1, 12, 20, 64, 0, 0, 128, 0), (3, 4, 8, 16, 0, 0, 8, 0)]


@pytest.mark.parametrize("case", CONV_CASES)
def test_conv3x3_matches_torch(gpu, case):
    import torch

    from mach2d import unet as U
    L = U._bind()
    n, h, w, c1, mode, c2, cout, relu = case
    g = torch.Generator().manual_seed(sum(case))
    sh1 = {0: (n, h, w, c1), 1: (n, 2 * h, 2 * w, c1), 2: (n, h // 2, w // 2, c1)}[mode]
    x1 = _bf(torch.randn(*sh1, generator=g))
    x2 = _bf(torch.randn(n, h, w, c2, generator=g)) if c2 else None
    cin = c1 + c2
    kpad = (9 * cin + 31) // 32 * 32
    cpad = (cout + 15) // 16 * 16
    wf = torch.zeros(cpad, kpad)
    wf[:cout, :9 * cin] = _bf(torch.randn(cout, 9 * cin, generator=g) * 0.2)
    b = torch.randn(cout, generator=g)
    got = _conv_gpu(L, _dev(x1), c1, mode, _dev(x2) if c2 else None, c2, _dev(wf),
                    _dev(b, torch.float32), cout, kpad, n, h, w, relu)
    xe = _effective(x1, mode, x2 if c2 else None)
    want = _ref_conv(xe, wf[:cout, :9 * cin], b, cin, cout, relu)
    scale = want.abs().max().item()
    assert torch.allclose(got, want, atol=1e-4 * scale, rtol=0), (case, (got - want).abs().max())


@pytest.mark.parametrize("case", CONV_CASES[:4])
def test_conv3x3_gradients_match_autograd(gpu, case):
    """wgrad kernel, input gradient (rotated weights through the forward
    kernel) and the gradient of the fused pool / upsampling against autograd
    of the FP32 reference."""
    import ctypes as C

    import torch

    from mach2d import unet as U
    L = U._bind()
    n, h, w, c1, mode, c2, cout, _ = case
    g = torch.Generator().manual_seed(7 + sum(case))
    sh1 = {0: (n, h, w, c1), 1: (n, 2 * h, 2 * w, c1), 2: (n, h // 2, w // 2, c1)}[mode]
    x1 = _bf(torch.randn(*sh1, generator=g))
    x2 = _bf(torch.randn(n, h, w, c2, generator=g)) if c2 else None
    cin = c1 + c2
    kpad, cpad = (9 * cin + 31) // 32 * 32, (cout + 15) // 16 * 16
    kpad_r, cin_pad = (9 * cout + 31) // 32 * 32, (cin + 15) // 16 * 16
    wf = torch.zeros(cpad, kpad)
    wf[:cout, :9 * cin] = _bf(torch.randn(cout, 9 * cin, generator=g) * 0.2)
    G = _bf(torch.randn(n, h, w, cout, generator=g))
    # reference: loss = sum(conv(x) * G), no bias / relu (the kernels take G
    # as the pre-activation gradient)
    x1r = x1.clone().requires_grad_(True)
    x2r = x2.clone().requires_grad_(True) if c2 else None
    wr_ = wf[:cout, :9 * cin].clone().requires_grad_(True)
    if mode == 1:
        n_, hh, ww, cc = x1r.shape
        t = x1r.reshape(n_, hh // 2, 2, ww // 2, 2, cc)
        pooled = ((t[:, :, 0, :, 0] + t[:, :, 0, :, 1]) + (t[:, :, 1, :, 0] + t[:, :, 1, :, 1])) * 0.25
        # the kernels read the pooled value rounded to bf16; its gradient is the pool's
        xe = _bf(pooled).detach() + (pooled - pooled.detach())
    else:
        xe = _effective(x1r, mode, None)
    if c2:
        xe = torch.cat([xe, x2r], dim=3)
    y = _ref_conv(xe, wr_, None, cin, cout, False)
    (y * G).sum().backward()
    # GPU: weight and bias gradients
    dw = torch.zeros(cpad, kpad, device="cuda")
    db = torch.zeros(cout, device="cuda")
    dx1, dx2, dG = _dev(x1), _dev(x2) if c2 else None, _dev(G)
    rc = L.m2d_unet_conv3x3_wgrad(C.c_void_p(dx1.data_ptr()), c1, mode,
                                  C.c_void_p(dx2.data_ptr()) if c2 else None, c2,
                                  C.c_void_p(dG.data_ptr()), cout, kpad, n, h, w,
                                  C.c_void_p(dw.data_ptr()), C.c_void_p(db.data_ptr()), None)
    assert rc == 0
    # input gradient: forward kernel on G with the rotated weights
    wfd = _dev(wf, torch.float32)
    wb = torch.empty(cpad, kpad, dtype=torch.bfloat16, device="cuda")
    wrot = torch.empty(cin_pad, kpad_r, dtype=torch.bfloat16, device="cuda")
    assert L.m2d_unet_pack_weights(C.c_void_p(wfd.data_ptr()), cout, cin, kpad,
                                   C.c_void_p(wb.data_ptr()), C.c_void_p(wrot.data_ptr()), kpad_r,
                                   cin_pad, None) == 0
    gi = _conv_gpu(L, dG, cout, 0, None, 0, wrot, None, cin, kpad_r, n, h, w, 0)
    gi_d = gi.to("cuda")
    g1 = torch.zeros(sh1, device="cuda")
    assert L.m2d_unet_mode_bwd(C.c_void_p(gi_d.data_ptr()), cin, 0, c1, mode, n, h, w,
                               C.c_void_p(g1.data_ptr()), None) == 0
    torch.cuda.synchronize()
    sw = wr_.grad.abs().max().item()
    assert torch.allclose(dw.cpu()[:cout, :9 * cin], wr_.grad, atol=1e-4 * sw, rtol=0)
    assert not dw.cpu()[:, 9 * cin:].any()
    assert torch.allclose(db.cpu(), G.sum(dim=(0, 1, 2)), atol=1e-4 * G.abs().sum().item() / cout)
    s1 = x1r.grad.abs().max().item()
    assert torch.allclose(g1.cpu(), x1r.grad, atol=1e-4 * s1, rtol=0)
    if c2:
        g2 = torch.zeros(n, h, w, c2, device="cuda")
        assert L.m2d_unet_mode_bwd(C.c_void_p(gi_d.data_ptr()), cin, c1, c2, 0, n, h, w,
                                   C.c_void_p(g2.data_ptr()), None) == 0
        torch.cuda.synchronize()
        s2 = x2r.grad.abs().max().item()
        assert torch.allclose(g2.cpu(), x2r.grad, atol=1e-4 * s2, rtol=0)


def _ref_net(net, x):
    """The whole network in FP32 on the CPU from the same weights, rounding
    activations to bf16 between layers as the kernels do."""
    import torch
    acts = {"x": x}
    n, h, w, _ = x.shape
    out = None
    for lay in net.layers:
        src = acts[lay.src]
        if lay.mode == 1:
            src = _pool(src)
        elif lay.mode == 2:
            src = _effective(src, 2, None)
        if lay.skip:
            src = torch.cat([src, acts[lay.skip]], dim=3)
        wv = _bf(lay.w.cpu()[:lay.cout, :9 * lay.cin])
        y = _ref_conv(src, wv, lay.b.cpu(), lay.cin, lay.cout, lay.relu)
        acts[lay.name] = y if lay.name == "head" else _bf(y)
        out = y
    return out


def test_unet_forward_matches_reference(gpu):
    import torch

    from mach2d import unet as U
    net = U.UNet(seed=3)
    g = torch.Generator().manual_seed(5)
    for lay in net.layers:   # non-zero biases exercise the bias path
        lay.b.copy_(torch.randn(lay.cout, generator=g) * 0.1)
    x = _bf(torch.randn(2, 16, 24, 8, generator=g))
    x[..., 6:] = 0
    got = net.forward(_dev(x)).cpu()
    torch.cuda.synchronize()
    want = _ref_net(net, x)
    scale = want[..., 0].abs().max().item()
    err = (got[..., 0] - want[..., 0]).abs().max().item()
    assert err <= 2e-2 * scale, (err, scale)


def test_unet_training_reduces_loss(gpu):
    """Adam on a fixed small batch: the loss falls well below its start."""
    import torch

    from mach2d import unet as U
    net = U.UNet(seed=1)
    g = torch.Generator().manual_seed(2)
    x = _bf(torch.randn(2, 16, 16, 8, generator=g))
    x[..., 6:] = 0
    target = (x[..., 0] * 0.5 + 0.25 * x[..., 1]).contiguous()
    xd, td = _dev(x), target.to("cuda")
    mask = torch.ones_like(td)
    losses = []
    for _ in range(60):
        loss = net.loss_and_backward(xd, td, mask)
        net.adam_step(lr=3e-3)
        losses.append(float(loss.item()))
    assert all(np.isfinite(losses))
    assert losses[-1] < 0.2 * losses[0], losses[::10]


def test_pack_input_and_guess_scale(gpu):
    """Network input channels from a 9-diagonal system, and the guess path
    (output times s) on the grid."""
    import ctypes as C

    import torch

    from mach2d import problems as P
    from mach2d import unet as U
    nx, ny = 20, 11
    s = P.pcorr_system(nx, ny, seed=4, q=1.05, rhs="gauss")
    net = U.UNet(seed=0)
    a = torch.tensor(s.a.reshape(-1), device="cuda")
    b = torch.tensor(s.rhs, device="cuda")
    x = net.pack_input(a, b, nx, ny, 2.0).cpu().float()
    h, w = U.UNet.padded(nx, ny)
    assert x.shape == (1, h, w, 8)
    A = s.a.reshape(9, ny, nx)
    ap = A[4]
    with np.errstate(divide="ignore", invalid="ignore"):
        want0 = np.where(ap != 0, s.rhs.reshape(ny, nx) / ap / 2.0, 0.0)
        want1 = np.where(ap != 0, A[3] / ap, 0.0)
    got = x[0, :ny, :nx].numpy()
    assert np.allclose(got[..., 0], want0, rtol=1e-2, atol=1e-6)
    assert np.allclose(got[..., 1], want1, rtol=1e-2, atol=1e-6)
    assert not x[0, ny:].any() and not x[0, :, nx:].any() and not x[..., 6:].any()
    var = torch.zeros(nx * ny, dtype=torch.float64, device="cuda")
    sc = net.guess(a, b, nx, ny, var)
    out = net.forward(net.pack_input(a, b, nx, ny, sc)).cpu()
    assert np.allclose(var.cpu().numpy().reshape(ny, nx), sc * out[0, :ny, :nx, 0].double().numpy())
    assert C.sizeof(C.c_void_p) == 8


def test_guess_scale_minimises_residual(gpu):
    """m2d_guess_scale: alpha = (Ag.b)/(Ag.Ag); the exact solution scales by
    1, a doubled one by 0.5, and a scaled arbitrary guess is never worse than
    the zero guess (first-order optimality: (A(alpha g) - b).Ag = 0)."""
    import torch

    from mach2d import problems as P
    s = P.pcorr_system(34, 18, seed=2, q=1.05, rhs="gauss")
    dev = gpu.DeviceMSI(s.nx, s.ny, "fp64")
    a = torch.tensor(s.a.reshape(-1), device="cuda")
    b = torch.tensor(s.rhs, device="cuda")
    A = np.zeros((s.N, s.N))
    nx = s.nx
    off = [-nx - 1, -nx, -nx + 1, -1, 0, 1, nx - 1, nx, nx + 1]
    for k, o in enumerate(off):
        for p in range(s.N):
            if 0 <= p + o < s.N and s.a[k, p] != 0.0:
                A[p, p + o] = s.a[k, p]
    x = np.linalg.solve(A, s.rhs)
    for mult, want in ((1.0, 1.0), (2.0, 0.5)):
        g = torch.tensor(mult * x, device="cuda")
        alpha = dev.guess_scale(a, b, g)
        assert abs(alpha - want) < 1e-10, (mult, alpha)
    rng = np.random.default_rng(3)
    g0 = rng.standard_normal(s.N)
    g = torch.tensor(g0, device="cuda")
    alpha = dev.guess_scale(a, b, g)
    Ag = A @ g0
    assert abs(alpha - (Ag @ s.rhs) / (Ag @ Ag)) < 1e-12 * abs(alpha) + 1e-300
    r = A @ (alpha * g0) - s.rhs
    assert abs(r @ Ag) < 1e-9 * np.linalg.norm(Ag) * np.linalg.norm(s.rhs)
    assert dev.residual_norm(a, b, g) <= dev.residual_norm(a, b, torch.zeros_like(g)) * (1 + 1e-12)
    dev.close()


def test_guess_scale_energy(gpu):
    """m2d_guess_scale_energy: alpha = (g.b)/(g.Ag); the exact solution
    scales by 1, a doubled one by 0.5; for an arbitrary guess the scaled
    one satisfies the first-order condition g.(A(alpha g) - b) = 0, and a
    guess with g.Ag <= 0 becomes zero."""
    import torch

    from mach2d import problems as P
    s = P.pcorr_system(34, 18, seed=2, q=1.05, rhs="gauss")
    dev = gpu.DeviceMSI(s.nx, s.ny, "fp64")
    a = torch.tensor(s.a.reshape(-1), device="cuda")
    b = torch.tensor(s.rhs, device="cuda")
    A = np.zeros((s.N, s.N))
    nx = s.nx
    off = [-nx - 1, -nx, -nx + 1, -1, 0, 1, nx - 1, nx, nx + 1]
    for k, o in enumerate(off):
        for p in range(s.N):
            if 0 <= p + o < s.N and s.a[k, p] != 0.0:
                A[p, p + o] = s.a[k, p]
    x = np.linalg.solve(A, s.rhs)
    for mult, want in ((1.0, 1.0), (2.0, 0.5)):
        g = torch.tensor(mult * x, device="cuda")
        alpha = dev.guess_scale(a, b, g, energy=True)
        assert abs(alpha - want) < 1e-10, (mult, alpha)
    g0 = np.random.default_rng(4).standard_normal(s.N)
    alpha = dev.guess_scale(a, b, torch.tensor(g0, device="cuda"), energy=True)
    assert abs(alpha - (g0 @ s.rhs) / (g0 @ (A @ g0))) < 1e-12 * abs(alpha)
    assert abs(g0 @ (A @ (alpha * g0) - s.rhs)) < 1e-9 * np.linalg.norm(g0) * np.linalg.norm(s.rhs)
    g = torch.zeros(s.N, dtype=torch.float64, device="cuda")
    assert dev.guess_scale(a, b, g, energy=True) == 0.0
    dev.close()


def test_guessed_solve_matches_zero_guess_solution(gpu):
    """Guess-then-MSI with an untrained network: the guess is scaled by the
    energy-minimising amplitude, the solve reaches gamma * ||b||, and the
    solution agrees with the zero-guess solution to 1e-8 relative."""
    import torch

    from mach2d import learned as Lr
    from mach2d import problems as P
    from mach2d import unet as U
    s = P.pcorr_system(66, 34, seed=5, q=1.05, rhs="gauss")
    net = U.UNet(seed=11)
    dev = gpu.DeviceMSI(s.nx, s.ny, "fp64")
    a = torch.tensor(s.a.reshape(-1), device="cuda")
    b = torch.tensor(s.rhs, device="cuda")
    dev.factor(a)
    v0 = torch.zeros(s.N, dtype=torch.float64, device="cuda")
    st0 = dev.solve(a, b, v0, 1e-10, 5000)
    v1 = torch.zeros_like(v0)
    st1, used, rg, rb = Lr.guessed_solve(dev, net, a, b, v1, s.nx, s.ny)
    assert st0.status == 0 and st1.status == 0
    assert st1.rn < 1e-10 * rb * (1 + 1e-9)
    rel = float(torch.linalg.norm(v1 - v0) / torch.linalg.norm(v0))
    assert rel < 1e-8, rel
    dev.close()


def test_guess_many_equals_single_guesses(gpu):
    """One network pass over several systems of one grid gives each system
    the guess it gets alone, bit for bit (the images are independent)."""
    import torch

    from mach2d import learned as Lr
    from mach2d import problems as P
    from mach2d import unet as U
    net = U.UNet()
    net.load(Lr.default_weights())
    nx, ny = 130, 66
    sys_ = [P.pcorr_system(nx, ny, seed=40 + q, rhs="gauss") for q in range(3)]
    a = [torch.tensor(s.a.reshape(-1), device="cuda") for s in sys_]
    b = [torch.tensor(s.rhs, device="cuda") for s in sys_]
    one = [torch.zeros(s.N, dtype=torch.float64, device="cuda") for s in sys_]
    many = [torch.zeros(s.N, dtype=torch.float64, device="cuda") for s in sys_]
    s1 = [net.guess(a[q], b[q], nx, ny, one[q]) for q in range(3)]
    s2 = net.guess_many(a, b, nx, ny, many)
    torch.cuda.synchronize()
    assert s1 == s2
    for q in range(3):
        assert torch.equal(one[q], many[q]), q
        assert float(one[q].abs().max()) > 0


def test_guess_prepare_many_matches_single_calls(gpu):
    """The batched scaling gives each system guess_scale's alpha (same sums
    in the same order) and residual_norm's ||rhs - A g|| to 1e-12."""
    import torch

    from mach2d import problems as P
    nx, ny = 97, 64
    sys_ = [P.pcorr_system(nx, ny, seed=60 + q, rhs="gauss") for q in range(3)]
    dev = gpu.DeviceMSI(nx, ny)
    a = [torch.tensor(s.a.reshape(-1), device="cuda") for s in sys_]
    b = [torch.tensor(s.rhs, device="cuda") for s in sys_]
    g0 = [torch.tensor(np.random.default_rng(q).uniform(-1, 1, s.N), device="cuda")
          for q, s in enumerate(sys_)]
    g1 = [x.clone() for x in g0]
    g2 = [x.clone() for x in g0]
    alphas, rn = dev.guess_prepare_many(a, b, g2, energy=True)
    for q in range(3):
        al = dev.guess_scale(a[q], b[q], g1[q], energy=True)
        assert al == alphas[q]
        assert torch.equal(g1[q], g2[q])
        assert rn[q] == pytest.approx(dev.residual_norm(a[q], b[q], g1[q]), rel=1e-12)
    dev.close()


def test_simplec_pairs_match_reference_fixture(gpu, tmp_path):
    """Training pairs generated on the GPU (device SIMPLEC time step, batched
    FP64 MSI targets) equal the pairs of the same time steps composed from
    the compiled reference's routines and solved by its class_solver_msi9d
    (tests/golden/simplec_pairs_34x18.m2dt): systems, right-hand sides and
    targets bit for bit (as stored, float32), the same step and itp
    metadata, the residual drop to 1e-3 relative (a residual 1e-13 of ||b||
    summed in another order and, on the host, from float64 values
    recomputed by the oracle)."""
    import os

    from mach2d import dataset as D
    from mach2d import learned as Lr
    path = str(tmp_path / "p.m2dt")
    n = Lr.simplec_pairs(path, variants=1, steps=12, nx=34, ny=18, seed=0)
    assert n == 12
    got = D.Dataset(path)
    want = D.Dataset(os.path.join(os.path.dirname(__file__), "golden",
                                  "simplec_pairs_34x18.m2dt"))
    assert (got.nx, got.ny, got.ndiag, len(got)) == (want.nx, want.ny, want.ndiag, len(want))
    for q in range(len(want)):
        for u, v in zip(got[q], want[q]):
            assert np.array_equal(u, v), q
        assert list(got.meta[q][:3]) == list(want.meta[q][:3])
        assert got.meta[q][3] == pytest.approx(want.meta[q][3], rel=1e-3)


# (n, h, w, c1, mode, c2, cout): tiles cut by the image's edge in both
# directions, output channels that leave a group of four or of 16, 32, 64
# open, channel counts of the network's layers and others (their taps' places
# are computed), and a staged input beyond 64 KB of LDS
TILE_CASES = [
    (1, 1, 1, 8, 0, 0, 8), (1, 9, 17, 8, 0, 0, 16), (2, 17, 33, 16, 0, 0, 16),
    (1, 7, 15, 16, 0, 0, 5), (1, 10, 18, 24, 0, 0, 12), (1, 16, 30, 32, 2, 16, 16),
    (1, 9, 31, 32, 0, 0, 48), (3, 5, 19, 16, 1, 0, 32), (1, 8, 16, 40, 0, 8, 32),
    (1, 12, 34, 64, 2, 32, 32), (1, 5, 17, 32, 0, 0, 64), (2, 3, 21, 64, 1, 0, 128),
    (1, 6, 18, 128, 2, 64, 64), (1, 5, 33, 64, 0, 0, 96), (1, 4, 16, 64, 0, 0, 192),
    (1, 6, 20, 392, 0, 0, 64), (1, 9, 20, 240, 0, 0, 16)]


def _conv_and_gradient(case, large):
    import ctypes as C

    import torch

    from mach2d import unet as U
    L = U._bind()
    n, h, w, c1, mode, c2, cout = case
    g = torch.Generator().manual_seed(11 + sum(case))
    sh1 = {0: (n, h, w, c1), 1: (n, 2 * h, 2 * w, c1), 2: (n, h // 2, w // 2, c1)}[mode]
    x1 = _bf(torch.randn(*sh1, generator=g))
    x2 = _bf(torch.randn(n, h, w, c2, generator=g)) if c2 else None
    cin = c1 + c2
    kpad, cpad = (9 * cin + 31) // 32 * 32, (cout + 15) // 16 * 16
    wf = torch.zeros(cpad, kpad)
    wf[:cout, :9 * cin] = _bf(torch.randn(cout, 9 * cin, generator=g) * 0.2)
    b = torch.randn(cout, generator=g)
    dx1, dx2 = _dev(x1), _dev(x2) if c2 else None
    got = _conv_gpu(L, dx1, c1, mode, dx2, c2, _dev(wf), _dev(b, torch.float32), cout, kpad,
                    n, h, w, 1)
    xe = _effective(x1, mode, x2)
    wr = wf[:cout, :9 * cin].clone().requires_grad_(True)
    want = _ref_conv(xe, wr, b, cin, cout, False)
    scale = want.abs().max().item()
    assert torch.allclose(got, torch.relu(want).detach(), atol=1e-4 * scale, rtol=0), case
    G = _bf(torch.randn(n, h, w, cout, generator=g))
    (want * G).sum().backward()
    dw, db, dG = torch.zeros(cpad, kpad, device="cuda"), torch.zeros(cout, device="cuda"), _dev(G)
    assert L.m2d_unet_conv3x3_wgrad(C.c_void_p(dx1.data_ptr()), c1, mode,
                                    C.c_void_p(dx2.data_ptr()) if c2 else None, c2,
                                    C.c_void_p(dG.data_ptr()), cout, kpad, n, h, w,
                                    C.c_void_p(dw.data_ptr()), C.c_void_p(db.data_ptr()),
                                    None) == 0
    torch.cuda.synchronize()
    sw = max(wr.grad.abs().max().item(), 1e-3)
    assert torch.allclose(dw.cpu()[:cout, :9 * cin], wr.grad, atol=1e-4 * sw, rtol=0), case
    assert not dw.cpu()[:, 9 * cin:].any() and not dw.cpu()[cout:].any()
    sb = G.sum(dim=(0, 1, 2))
    assert torch.allclose(db.cpu(), sb, atol=1e-4 * (sb.abs().max().item() if large else
                                                     G.abs().sum().item() / cout))


@pytest.mark.parametrize("case", TILE_CASES)
def test_conv3x3_tiles_match_torch(gpu, case):
    """Forward convolution and weight gradient at the edges of their tiles
    against PyTorch in FP32 (exact products of bf16 values, sums in another
    order: 1e-4 of the largest value, as above)."""
    _conv_and_gradient(case, False)


# Images large enough for the taller tiles (four rows a wave: 512 workgroups,
# 256 with 64 output channels) and for several tiles to a workgroup of the
# weight gradient, in uneven shares, cut at both edges: every number of output
# channels per workgroup, compiled and computed places of the taps, channel
# counts / 8 that are no multiple of four, staged tiles of 64 to 80 KB, every
# mode, one and two groups of 16 output channels of the gradient, many
# channels on few workgroups, output channels that no vector store takes
LARGE_CASES = [
    (2, 250, 257, 8, 0, 0, 16), (2, 243, 270, 16, 1, 0, 16), (2, 250, 258, 32, 2, 16, 16),
    (1, 250, 515, 120, 0, 0, 5), (2, 250, 257, 24, 0, 0, 12), (2, 243, 270, 16, 1, 0, 32),
    (1, 250, 514, 64, 2, 32, 32), (2, 250, 257, 24, 0, 0, 32), (1, 126, 250, 128, 2, 64, 64),
    (1, 125, 250, 216, 0, 0, 64), (1, 125, 130, 32, 1, 0, 128), (1, 130, 250, 64, 0, 0, 64),
    (1, 130, 250, 128, 0, 0, 64)]


@pytest.mark.parametrize("case", LARGE_CASES)
def test_conv3x3_large_images_match_torch(gpu, case):
    """The same for images that fill the chip.  That a case takes the path it
    is for is checked with the launch rules of csrc/unet.hip."""
    n, h, w, c1, mode, c2, cout = case
    cin, cpad = c1 + c2, (cout + 15) // 16 * 16
    nt = 4 if cpad % 64 == 0 else 2 if cpad % 32 == 0 else 1
    th = 8 if nt == 4 else 16
    lds = ((th + 2) * 18 * (cin + (0 if cin // 8 % 2 else 8)) + 8) * 2
    groups = -(-h // th) * -(-w // 16) * n * (cpad // (16 * nt))
    assert lds <= 80 * 1024 and groups >= (256 if nt == 4 else 512)
    tiles = -(-h // 16) * -(-w // 16) * n
    blocks = -(-cin // 16) * -(-cout // (32 if cout > 16 else 16))
    share = min(256, -(-512 // blocks))
    assert tiles > share and tiles % share
    _conv_and_gradient(case, True)


@pytest.mark.parametrize("n,h,w,c,m1,m2", [(1, 2, 2, 8, 1, None), (2, 6, 10, 16, 1, 0), (1, 3, 5, 24, 0, None),
                                           (1, 5, 3, 8, 2, None), (2, 4, 8, 32, 0, 2), (1, 8, 6, 40, 2, 1)])
def test_grad_in_is_its_pieces(gpu, n, h, w, c, m1, m2):
    """m2d_unet_grad_in against mode_bwd per input, to_bf16 and relu_bwd: the
    same bits, for every mode, one and two inputs, channel offsets."""
    import ctypes as C

    import torch

    from mach2d import unet as U
    L = U._bind()
    gen = torch.Generator().manual_seed(h * w + c)
    p = lambda t: C.c_void_p(t.data_ptr()) if t is not None else None  # noqa: E731
    src, ref = [], torch.zeros(n, h, w, c, device="cuda")
    for k, m in enumerate((m1, m2)):
        if m is None:
            src += [None, 0, 0, 0]
            continue
        hh, ww = {0: (h, w), 1: (h // 2, w // 2), 2: (2 * h, 2 * w)}[m]
        cs, c0 = c + 8 * k, 8 * k
        g = torch.randn(n, hh, ww, cs, generator=gen).to("cuda")
        src += [g, cs, c0, m]
        assert L.m2d_unet_mode_bwd(p(g), cs, c0, c, m, n, hh, ww, p(ref), None) == 0
    y = _dev(torch.relu(torch.randn(n, h, w, c, generator=gen)))
    want = torch.empty(n, h, w, c, dtype=torch.bfloat16, device="cuda")
    assert L.m2d_unet_to_bf16(p(ref), p(want), want.numel(), None) == 0
    assert L.m2d_unet_relu_bwd(p(want), p(y), want.numel(), None) == 0
    got = torch.empty_like(want)
    assert L.m2d_unet_grad_in(p(src[0]), *src[1:4], p(src[4]), *src[5:8], p(y), c, n, h, w, p(got),
                              None) == 0
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_empty_mask_is_refused(gpu):
    """A mask without a set pixel has no mean: the step raises before any
    gradient is written, weights and moments stay, and the next step on an
    ordinary mask runs; the kernel's loss and gradient for a count of 0 are 0."""
    import ctypes as C

    import torch

    from mach2d import unet as U
    net = U.UNet(seed=4)
    g = torch.Generator().manual_seed(9)
    x, target = _dev(torch.randn(1, 8, 16, 8, generator=g)), torch.ones(1, 8, 16, device="cuda")
    mask = torch.ones_like(target)
    net.loss_and_backward(x, target, mask)
    net.adam_step()
    keep = [t.clone() for lay in net.layers for t in (lay.w, lay.gw, lay.gb, lay.mw, lay.vw)]
    with pytest.raises(ZeroDivisionError):
        net.loss_and_backward(x, target, torch.zeros_like(mask))
    now = [t for lay in net.layers for t in (lay.w, lay.gw, lay.gb, lay.mw, lay.vw)]
    assert all(torch.equal(u, v) for u, v in zip(keep, now)) and net.step_count == 1
    assert bool(torch.isfinite(net.loss_and_backward(x, target, mask)))
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    pred, grad = torch.randn(300, 8, device="cuda"), torch.ones(300, 8, device="cuda").bfloat16()
    tgt, msk, cnt = (torch.zeros(k, device="cuda") for k in (300, 300, 1))
    part = torch.ones(2, device="cuda")
    assert net.L.m2d_unet_mse_count(p(pred), 8, p(tgt), p(msk), 300, p(cnt), p(grad), 8, p(part),
                                    None) == 0
    torch.cuda.synchronize()
    assert not part.any() and not grad.float().any()


@pytest.mark.parametrize("what", ["tensors", "storage", "one bias gradient"])
def test_training_follows_replaced_tensors(gpu, what):
    """Weights, gradients and moments that a caller puts in the place of the
    layers' own, as new tensors or as new storage of the old ones, are the
    ones that training reads and updates: the same steps as on the layers'
    own tensors (gradients to the order of their atomic additions)."""
    import torch

    from mach2d import unet as U
    g = torch.Generator().manual_seed(21)
    x, target = _dev(torch.randn(2, 16, 24, 8, generator=g)), torch.randn(2, 16, 24, generator=g).cuda()
    mask = torch.ones_like(target)
    own, net = U.UNet(seed=6), U.UNet(seed=6)
    names = ("w", "b", "gw", "gb", "mw", "mb", "vw", "vb")
    if what == "one bias gradient":
        net.layers[2].gb.data = torch.full_like(net.layers[2].gb, 7.0)
    else:
        for lay in net.layers:
            for k in names:
                if what == "tensors":
                    setattr(lay, k, getattr(lay, k).clone())
                else:
                    getattr(lay, k).data = getattr(lay, k).clone()
    before = [lay.w.clone() for lay in net.layers]
    for n in (own, net):
        losses = [float(n.loss_and_backward(x, target, mask))]
        n.adam_step()
        losses.append(float(n.loss_and_backward(x, target, mask)))
        n.losses = losses
    for u, v, w in zip(own.layers, net.layers, before):
        assert not torch.equal(v.w, w), v.name
        for k in names:
            a, b = getattr(u, k), getattr(v, k)
            # a step is at most lr = 1e-3; a gradient near zero may turn its sign
            tol = 2e-3 if k in ("w", "b") else 1e-2 * float(a.norm()) + 1e-12
            assert float((a - b).abs().max()) <= tol, (v.name, k)
    assert net.losses[0] == pytest.approx(own.losses[0], rel=1e-5)
    assert net.losses[1] < net.losses[0] and net.losses[1] == pytest.approx(own.losses[1], rel=1e-2)


def test_backward_follows_the_layer_table(gpu, monkeypatch):
    """A network of another table: a layer without ReLU, and one whose output
    three convolutions read.  Weight and bias gradients against autograd of
    the FP32 network (activations and their gradients rounded to bf16, as the
    kernels do): 2e-2 of a layer's gradient, the bound of a bf16 network; the
    cut of a missing ReLU or a reader left out is of the order of 1."""
    import torch

    from mach2d import unet as U
    table = [("a", "x", U.DIRECT, None, 16, False), ("b", "a", U.DIRECT, None, 16, True),
             ("c", "b", U.DIRECT, "a", 16, True), ("d", "c", U.DIRECT, "a", 16, True),
             ("e", "d", U.POOL, None, 16, False), ("f", "e", U.UP, "d", 16, True),
             ("head", "f", U.DIRECT, None, 8, False)]
    monkeypatch.setattr(U, "LAYERS", table)
    monkeypatch.setattr(U, "LEVEL", {n: int(n == "e") for n, *_ in table})
    net = U.UNet(seed=8)
    g = torch.Generator().manual_seed(3)
    x = _bf(torch.randn(2, 8, 24, 8, generator=g))
    target, mask = torch.randn(2, 8, 24, generator=g), torch.ones(2, 8, 24)
    mask[:, 3:5, 7:] = 0.0
    loss = net.loss_and_backward(_dev(x), target.cuda(), mask.cuda())

    def rnd(v):   # rounded to bf16 both ways
        v = v + (_bf(v) - v).detach()
        if v.requires_grad:
            v.register_hook(_bf)
        return v
    acts, params = {"x": x}, []
    for lay in net.layers:
        w = _bf(lay.w.cpu()[:lay.cout, :9 * lay.cin]).requires_grad_(True)
        b = lay.b.cpu().clone().requires_grad_(True)
        params.append((lay, w, b))
        src = acts[lay.src]
        if lay.mode == U.POOL:
            mean = src.unflatten(1, (-1, 2)).unflatten(3, (-1, 2)).mean(dim=(2, 4))
            src = _pool(src.detach()) + (mean - mean.detach())
        elif lay.mode == U.UP:
            src = _effective(src, 2, None)
        if lay.skip:
            src = torch.cat([src, acts[lay.skip]], dim=3)
        y = _ref_conv(src, w, b, lay.cin, lay.cout, False)
        if y.requires_grad and lay.name != "head":
            y.register_hook(_bf)
        acts[lay.name] = y if lay.name == "head" else rnd(torch.relu(y) if lay.relu else y)
    d = (acts["head"][..., 0] - target) * mask
    want = 0.5 * (d * d).sum() / mask.sum()
    want.backward()
    assert float(loss) == pytest.approx(float(want.detach()), rel=2e-2)
    for lay, w, b in params:
        for got, ref in ((lay.gw.cpu()[:lay.cout, :9 * lay.cin], w.grad), (lay.gb.cpu(), b.grad)):
            assert float((got - ref).norm()) <= 2e-2 * float(ref.norm()), lay.name
