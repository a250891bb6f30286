"""The stress pass near the identity (series in Z = (b - I)(b + I)^-1, no
decomposition) and where it hands over to the SVD, through zsmpm_stress__rocm,
against a float64 eigendecomposition of b = F F^T.

Tolerances. Inside the series' range every entry is a chain of fewer than 40
float32 operations on terms no larger than the strain, 40 * 6e-8 < 3e-6 of
(2 mu + 3 lambda) vol |E| (sand: the strain measure includes logJp). Beyond it
the four-sweep SVD leaves up to 2.4e-4 of |F| unconverged: 1e-3 of
(2 mu + 3 lambda) vol. Reflections and rotations are exact inputs of both.
"""
import numpy as np
import pytest

from zpc_amd import scenes as S

pytestmark = pytest.mark.gpu


def _reference(mat, F, lj):
    """vol P F^T (n, 3, 3), the strain scale and the new logJp, float64."""
    f = np.float32
    E, nu, vol = float(f(mat.E)), float(f(mat.nu)), float(f(mat.volume))
    mu, lam = 0.5 * E / (1 + nu), E * nu / ((1 + nu) * (1 - 2 * nu))
    w, U = np.linalg.eigh(F @ F.transpose(0, 2, 1))
    sig = np.sqrt(np.maximum(w, 0))
    if mat.kind == S.FIXED_COROTATED:
        J = np.linalg.det(F)
        s = sig.copy()
        s[J < 0, 0] *= -1  # eigh sorts ascending: the smallest carries the sign
        tau = 2 * mu * (s - 1) * s + (lam * (J - 1) * J)[:, None]
        scale = np.abs(s - 1).max(1)
    else:
        coh, beta, ys = float(f(mat.cohesion)), float(f(mat.beta)), float(f(mat.yield_surface))
        eps = np.log(np.maximum(sig, 1e-4)) - coh
        tot = eps.sum(1)
        tr = tot + lj
        dev = eps - (tr / 3)[:, None]
        norm = np.sqrt((dev ** 2).sum(1))
        dg = norm + (3 * lam + 2 * mu) / (2 * mu) * tr * ys
        H = np.where((dg > 0)[:, None], eps - (dg / np.where(norm > 0, norm, 1))[:, None] * dev, eps) + coh
        H = np.where((tr >= 0)[:, None], coh, H)
        lj = np.where(tr >= 0, beta * tot + lj, 0.0)
        tau = 2 * mu * H + (lam * H.sum(1))[:, None]
        scale = np.abs(eps).max(1) + np.abs(tr)
    PF = vol * (U * tau[:, None, :]) @ U.transpose(0, 2, 1)
    return PF, (2 * mu + 3 * lam) * vol, scale, lj


@pytest.mark.parametrize("kind", [S.FIXED_COROTATED, S.DRUCKER_PRAGER])
@pytest.mark.parametrize("scale,turn", [(1e-5, "none"), (1e-2, "none"), (1e-2, "rotated"), (1e-2, "reflected"),
                                        (0.13, "none"), (0.5, "rotated")])
def test_stress_series_and_svd(kind, scale, turn):
    import torch

    from zpc_amd import rocm

    n = 64 * 5 + 7  # whole waves and a ragged one, near and far lanes mixed in a wave
    rng = np.random.default_rng(11)
    F = np.eye(3) + scale * rng.normal(size=(n, 3, 3))
    if turn != "none":
        Q, _ = np.linalg.qr(rng.normal(size=(n, 3, 3)))
        want = 1.0 if turn == "rotated" else -1.0
        Q *= (want * np.sign(np.linalg.det(Q)))[:, None, None]
        F = F @ Q
    F[0] = np.eye(3)
    F = F.astype(np.float32)
    mat = (S.Material(kind=kind, E=1e4, nu=0.3, volume=1e-6) if kind == S.FIXED_COROTATED else
           S.Material.drucker_prager(3.5e5, 0.3, 1e3, volume=1e-6, cohesion=1e-3))
    lj = (0.5 * scale * rng.normal(size=n)).astype(np.float32)
    ref, stiff, strain, lj_ref = _reference(mat, F.astype(np.float64), lj.astype(np.float64))
    pol = rocm.Policy()
    dF = torch.as_tensor(np.ascontiguousarray(F.transpose(0, 2, 1)).reshape(n, 9)).cuda()
    dl, PF = torch.as_tensor(lj).cuda(), torch.empty((n, 9), dtype=torch.float32, device="cuda")
    model = rocm.model_desc(mat)
    rocm.check(pol.L.zsmpm_stress__rocm(pol.h, rocm.C.byref(model), dF.data_ptr(), dl.data_ptr(), n, PF.data_ptr()),
               "stress")
    pol.sync()
    got = PF.cpu().numpy().reshape(n, 3, 3).transpose(0, 2, 1)
    F64 = F.astype(np.float64)
    b = F64 @ F64.transpose(0, 2, 1)
    Z = np.linalg.solve(b + np.eye(3), b - np.eye(3))
    near = (Z ** 2).sum((1, 2)) < 0.0899
    if kind == S.FIXED_COROTATED:
        near &= np.linalg.det(F64) > 0
    # rounding F to float32 is part of the input; a rotated F has |F - I| ~ 1, so
    # b - I carries 3 roundings of order 1 (1e-6) whatever the strain
    floor = 1e-6 if turn != "none" else 0.0
    tol = np.where(near, 3e-6 * strain + floor, 1e-3) * stiff
    err = np.abs(got - ref).max((1, 2))
    assert np.all(err <= tol + 1e-30), (err / tol).max()
    if kind == S.DRUCKER_PRAGER:
        ljtol = np.where(near, 3e-6 * strain + 3 * floor, 1e-3)
        assert np.all(np.abs(dl.cpu().numpy() - lj_ref) <= ljtol + 1e-30)


@pytest.mark.parametrize("stretch", [1e3, 2.0e6, 2.2e6, 2.5e6, 1e9])
def test_stress_of_huge_stretches(stretch):
    """Isotropic stretches around 2e6, where det(F F^T + I) is finite and its
    reciprocal is not: sand at the cone's tip, H = cohesion on each axis and
    logJp raised by the whole volume strain. log sigma is a float32 logarithm
    (2 ulp) and H exact up to its rounding: 1e-5."""
    import torch

    from zpc_amd import rocm

    n = 65
    mat = S.Material.drucker_prager(3.5e5, 0.3, 1e3, volume=1e-6, cohesion=1e-3)
    F = np.zeros((n, 9), np.float32)
    F[:, ::4] = np.float32(stretch) * (1 + np.arange(n, dtype=np.float32)[:, None] / 1024)
    F[0, ::4] = 1.0  # a near lane in the same wave
    dF, dl = torch.as_tensor(F).cuda(), torch.zeros(n, dtype=torch.float32, device="cuda")
    PF = torch.empty((n, 9), dtype=torch.float32, device="cuda")
    pol = rocm.Policy()
    model = rocm.model_desc(mat)
    rocm.check(pol.L.zsmpm_stress__rocm(pol.h, rocm.C.byref(model), dF.data_ptr(), dl.data_ptr(), n, PF.data_ptr()),
               "stress")
    pol.sync()
    M = F.astype(np.float64).reshape(n, 3, 3).transpose(0, 2, 1)
    ref, _, _, lj = _reference(mat, M, np.zeros(n))
    assert np.allclose(dl.cpu().numpy()[1:], lj[1:], rtol=1e-5, atol=0)
    got = PF.cpu().numpy().reshape(n, 3, 3).transpose(0, 2, 1)
    assert np.allclose(got[1:], ref[1:], rtol=1e-5, atol=1e-5 * np.abs(ref[1:]).max())
