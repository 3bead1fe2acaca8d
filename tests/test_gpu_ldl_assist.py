"""Block LDL on the GPU (qtip_ldl_hessian_device_updates): the factor must equal the host factorization's bit for bit
(every sum in the host code's order of operations), including ragged last panels, and must fail the same way on a matrix
that is not positive definite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)


def spd(n, seed, rows=None):
    rng = np.random.default_rng(seed)
    rows = rows or 2 * n
    X = rng.standard_normal((rows, n)).astype(np.float32) * np.linspace(0.2, 3.0, n, dtype=np.float32)
    X[:, 1:] += 0.8 * X[:, :-1]
    H = (X.T @ X / rows).astype(np.float32)
    H += 0.01 * np.float32(np.mean(np.diag(H))) * np.eye(n, dtype=np.float32)
    return H


# 6656: trailing matrices on both sides of the 6144 rows from which an update brings the next diagonal block with it
# 160, 176: the most that the form with host buffers leaves to the host, and the next; 1024, 1040: L goes down at the end, or
# in blocks of 1024 rows on the way
@pytest.mark.parametrize("n", [16, 160, 176, 496, 512, 1024, 1040, 1152, 2560, 6656])
def test_factor_equals_host_factor(qz, pkg, n):
    say("case: LDL with device updates, n = %d" % n)
    H = spd(n, 100 + n, rows=None if n < 4096 else n + 512)
    a = pkg.HessPrep(n=n, HRr=H.copy())
    b = pkg.HessPrep(n=n, HRr=H.copy())
    pkg.Quantizer.ldl_hessian(a, threads=16)
    qz.ldl_hessian_device_updates(b, threads=16)
    assert np.array_equal(a.L.view(np.uint32), b.L.view(np.uint32))
    # and once more through the same context (buffers reused, a smaller matrix after a larger one)
    if n == 2560:
        H2 = spd(1024, 7)
        a2 = pkg.HessPrep(n=1024, HRr=H2.copy())
        b2 = pkg.HessPrep(n=1024, HRr=H2.copy())
        pkg.Quantizer.ldl_hessian(a2, threads=16)
        qz.ldl_hessian_device_updates(b2, threads=16)
        assert np.array_equal(a2.L.view(np.uint32), b2.L.view(np.uint32))


@pytest.mark.parametrize("n", [16, 48, 160, 272, 1024, 1040, 2560])
def test_device_resident_form_equals_host_factor(qz, pkg, n):
    """qtip_ldl_hessian_device_updates_dev: the rotated Hessian stays on the device and is not written, L arrives in the
    device buffer and from there, row block by row block, in the host buffer; both equal the host factorization's words."""
    import torch
    say("case: LDL with device updates, Hessian resident on the device, n = %d" % n)
    H = spd(n, 300 + n)
    a = pkg.HessPrep(n=n, HRr=H.copy())
    pkg.Quantizer.ldl_hessian(a, threads=16)
    dH = torch.from_numpy(H).cuda()
    L_pin = torch.full((n, n), -1.0, dtype=torch.float32).pin_memory()
    dL = torch.full((n, n), -1.0, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    for _ in range(2):   # twice through the same context: its buffers are reused
        qz.ldl_hessian_device_resident(dH, n, L_pin, dL, threads=16)
        assert np.array_equal(L_pin.numpy().view(np.uint32), a.L.view(np.uint32))
        assert torch.equal(dL.cpu(), L_pin)
        assert torch.equal(dH.cpu(), torch.from_numpy(H))
    # without the device copy of L
    L2 = np.full((n, n), -1.0, np.float32)
    qz.ldl_hessian_device_resident(dH, n, L2, None, threads=16)
    assert np.array_equal(L2.view(np.uint32), a.L.view(np.uint32))


def test_factor_of_a_large_matrix_equals_host_factor(qz, pkg):
    """n = 12288: 24 panels whose diagonal block comes with the update before it, and 24 that have a launch of their own;
    the form with host buffers, and the one that stays on the device with L in both places."""
    import torch
    n = 12288
    say("case: LDL on the device, n = %d" % n)
    gen = torch.Generator(device="cuda").manual_seed(6)
    X = torch.randn(n + 1024, n, device="cuda", generator=gen) * torch.linspace(0.2, 3.0, n, device="cuda")
    X[:, 1:] += 0.8 * X[:, :-1].clone()
    dH = X.T @ X / X.shape[0]
    del X
    dH += 0.01 * dH.diagonal().mean() * torch.eye(n, device="cuda")
    dH = dH.contiguous()
    a = pkg.HessPrep(n=n, HRr=dH.cpu().numpy())
    pkg.Quantizer.ldl_hessian(a, threads=16)
    want = torch.from_numpy(a.L.view(np.int32))
    b = pkg.HessPrep(n=n, HRr=a.HRr)
    qz.ldl_hessian_device_updates(b, threads=16)
    assert torch.equal(torch.from_numpy(b.L.view(np.int32)), want)
    L, dL = torch.empty(n, n, pin_memory=True), torch.empty(n, n, device="cuda")
    torch.cuda.synchronize()
    qz.ldl_hessian_device_resident(dH, n, L, dL, threads=16)
    assert torch.equal(L.view(torch.int32), want) and torch.equal(dL.cpu().view(torch.int32), want)


@pytest.mark.parametrize("n", [32, 48, 256, 288])
def test_factor_of_uneven_matrix_equals_host_factor(qz, pkg, n):
    """Channels of very different scale, and pairs of channels that do not hang together at all (zeros in the factor)."""
    say("case: LDL on the device, uneven matrix, n = %d" % n)
    H = spd(n, 900 + n)
    scale = (2.0 ** np.random.default_rng(n).integers(-12, 13, n)).astype(np.float32)
    H = H * scale[:, None] * scale[None, :]
    H[n // 2:, :n // 2] = 0
    H[:n // 2, n // 2:] = 0
    a, b = pkg.HessPrep(n=n, HRr=H.copy()), pkg.HessPrep(n=n, HRr=H.copy())
    pkg.Quantizer.ldl_hessian(a, threads=4)
    qz.ldl_hessian_device_updates(b)
    assert np.array_equal(a.L.view(np.uint32), b.L.view(np.uint32))
    import torch
    dH, L = torch.from_numpy(H).cuda(), np.full((n, n), -1.0, np.float32)
    torch.cuda.synchronize()
    qz.ldl_hessian_device_resident(dH, n, L)
    assert np.array_equal(a.L.view(np.uint32), L.view(np.uint32))


def test_small_matrices_are_factored_where_they_are(pkg):
    """From host memory to host memory up to 160 columns: no launch, and nothing kept on the device."""
    say("case: LDL from host to host, 160 and 176 columns")
    q = pkg.Quantizer(0)
    for n, on_device in ((160, False), (176, True)):
        H = spd(n, 40 + n)
        before = pkg.device_alloc_calls()
        a, b = pkg.HessPrep(n=n, HRr=H.copy()), pkg.HessPrep(n=n, HRr=H.copy())
        q.ldl_hessian_device_updates(a)
        L, dw = q.nvfp4_prepare_device_updates(H)
        assert (pkg.device_alloc_calls() > before) == on_device
        pkg.Quantizer.ldl_hessian(b, threads=4)
        L0, dw0 = pkg.nvfp4_prepare(H, 1e-2, True, 4)
        assert np.array_equal(a.L.view(np.uint32), b.L.view(np.uint32))
        assert np.array_equal(L.view(np.uint32), L0.view(np.uint32)) and np.array_equal(dw, dw0)
    q.close()


def test_a_second_factorization_allocates_nothing(pkg):
    """The calls with host buffers keep what they need on the device: they run beside the quantization of other groups, and
    a device free would wait for all of it."""
    say("case: LDL on the device, second call of a size")
    q = pkg.Quantizer(0)
    n = 512
    H = spd(n, 3)
    for call in (lambda: q.ldl_hessian_device_updates(pkg.HessPrep(n=n, HRr=H.copy())), lambda: q.nvfp4_prepare_device_updates(H)):
        call()
        before = pkg.device_alloc_calls()
        call()
        assert pkg.device_alloc_calls() == before
    q.close()


def test_rank_deficient_matrix_is_refused(qz, pkg):
    say("case: LDL with device updates, matrix not positive definite")
    n = 1024
    rng = np.random.default_rng(5)
    X = rng.standard_normal((300, n)).astype(np.float32)      # rank 300 < n, no damping
    H = (X.T @ X / 300).astype(np.float32)
    H[700, 700] = -1.0
    hp = pkg.HessPrep(n=n, HRr=H)
    with pytest.raises(pkg.QtipError):
        qz.ldl_hessian_device_updates(hp, threads=16)
    assert hp.L is None
    # the context is usable afterwards
    ok = pkg.HessPrep(n=512, HRr=spd(512, 3))
    qz.ldl_hessian_device_updates(ok, threads=16)
    assert np.isfinite(ok.L).all()
