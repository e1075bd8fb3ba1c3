"""GPU parity of the HIP path against the CPU oracle, through the C ABI.

Tolerances (FP32 path vs the FP64 oracle on FP32 parameters and FP32 walker
positions; u = 2^-24, kappa = the walker's largest 2-norm condition number of
its orbital matrices, from the oracle; bounds in tests/parity_util.py):
  log|psi|  : |d| <= 1e-5 |log psi| + 1e-4 + 4 e kappa (forward path vs the
              oracle), e = 16 u the relative error of the orbital entries and
              4 e kappa the first-order perturbation bound of log|det A|; the
              Laplacian-mode value vs the forward path the same bound (the two
              paths round differently)
  E_L       : per walker, relative error <= 1e-5 + 2 e kappa (first-order
              amplification of the entry error by the inverse); the median
              and the fraction of walkers within 1e-5 are printed (1e-5 holds
              for the well-conditioned walkers, kappa below ~10^2)
  grad      : |d| <= 2e-4 max(1, |grad|) per component (median), 5e-3 (max)
Metropolis decisions with identical proposals and uniforms agree wherever the
oracle's log ratio is farther from log u than 1e-6 plus twice the measured
difference between the GPU's and the oracle's log ratio (a decision can only
flip when the two log ratios straddle log u); the count inside that band is
printed.
"""

import numpy as np
import pytest

import os

from jaqmc_amd import params as P
from jaqmc_amd import systems as S
from oracle import hamiltonian as ham
from oracle import wavefunction as owf
from parity_util import ENTRY_ERR, U32, cancellation, el_report, logpsi_bound

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")

pytestmark = pytest.mark.gpu

CASES = {
    "li": ("li", {}),
    "n2_small": ("n2", dict(hidden_single=[32, 32, 32], hidden_double=[8, 16, 16], ndets=3)),
    "n2": ("n2", {}),
    "h60": ("h60", {}),
    "n2_iso": ("n2", dict(hidden_single=[64, 64], hidden_double=[16, 16], ndets=2, envelope="isotropic")),
}

_cache = {}


def _ring6():
    r = S.ring42()
    return S.make_system("ring6", r.atoms[:6] * 0.5, [1.0] * 6, (3, 3))


def _hydrogen():
    return S.make_system("H", [[0.0, 0.0, 0.0]], [1.0], (1, 0))


def _polarized_li():
    return S.make_system("Li(3,0)", [[0.0, 0.0, 0.0]], [3.0], (3, 0))


def _h17():
    return S.h_chain(17)


def _h24():
    return S.h_chain(24)


def _h20():
    return S.h_chain(20)


def _h26():
    return S.h_chain(26)


EDGE_CASES = {
    # 17 and 24 electrons: the FP64-MFMA determinant path at padded size 32
    "h17": (_h17, dict(hidden_single=[32, 32], hidden_double=[8, 8], ndets=2)),
    "h24": (_h24, dict(hidden_single=[32, 32], hidden_double=[8, 8], ndets=2)),
    # 20 and 26 electrons, 256-wide layers: the eight-wave FP16X3 layer GEMM
    # tiles at 64- and 96-row tangent units
    "h20_wide": (_h20, dict(hidden_single=[256, 256], hidden_double=[16, 16], ndets=2)),
    "h26_wide": (_h26, dict(hidden_single=[256, 256], hidden_double=[16, 16], ndets=2)),
    # the reference's hydrogen demo shape: one electron, one spin channel
    "h_atom": (_hydrogen, dict(hidden_single=[32, 32], hidden_double=[8, 8], ndets=2)),
    # fully polarized: a single non-empty spin channel (split_nonempty_channels)
    "li_polarized": (_polarized_li, dict(hidden_single=[32, 32], hidden_double=[8, 8], ndets=3)),
}

def _ring41():
    r = S.ring42()  # without its last hydrogen: 41 electrons
    return S.make_system("ring41", r.atoms[:11], r.charges[:11])


PSI_CASES = {
    # 6-electron piece of the ring, narrow Psiformer (heads_dim multiple of 32)
    "psi_small": (_ring6, dict(num_layers=2, num_heads=2, heads_dim=32, mlp_hidden=[32], ndets=2)),
    # full 42-electron ring with the 4-layer, 4-head, 256-wide Psiformer
    "ring42": (None, {}),
    # the ring less one hydrogen: 3N + 2 = 125 tangent rows in 128-row units (padding
    # rows), one MLP layer (the fused LayerNorm of the next layer written over
    # the MLP's own input)
    "psi41": (_ring41, dict(num_layers=2, mlp_hidden=[], ndets=2)),
}


def _setup(case, B):
    key = (case, B)
    if key in _cache:
        return _cache[key]
    if case in EDGE_CASES:
        mk, kw = EDGE_CASES[case]
        sysm, spec, *_ = S.workload("li")
        sysm = mk()
        spec.nspins = sysm.nspins
        spec.n_atoms = sysm.atoms.shape[0]
    elif case in PSI_CASES:
        mk, kw = PSI_CASES[case]
        sysm, spec, *_ = S.workload("ring42")
        if mk is not None:
            sysm = mk()
            spec.nspins = sysm.nspins
            spec.n_atoms = sysm.atoms.shape[0]
    else:
        name, kw = CASES[case]
        sysm, spec, *_ = S.workload(name)
    for k, v in kw.items():
        setattr(spec, k, v)
    p = P.init_params(spec, seed=11, bias_scale=0.1, env_jitter=0.2)
    x = S.init_walkers(sysm, B, seed=12)
    fx = os.path.join(GOLDEN, f"parity_{case}.npz")
    if case in CASES and os.path.exists(fx):
        # FP64 oracle references written by tests/golden/make_parity_fixtures.py
        # from the same seeds (the stored walkers are checked against them)
        with np.load(fx, allow_pickle=False) as f:
            ref = {k: f[k] for k in f.files}
        if ref["x"].shape[0] >= B:
            np.testing.assert_array_equal(ref["x"][:B], x)
            ref = {k: v[:B] for k, v in ref.items()}
            _cache[key] = (sysm, spec, p, x, ref)
            return _cache[key]
    p64 = P.cast_params(p, np.float64)
    ref = ham.local_energy(spec.as_oracle(), p64, x.astype(np.float64), sysm.atoms.astype(np.float64),
                           sysm.charges.astype(np.float64))
    A = np.asarray(owf.orbital_matrices(spec.as_oracle(), p64, x.astype(np.float64), sysm.atoms.astype(np.float64)))
    ref["kappa"] = np.linalg.cond(A).reshape(B, -1).max(axis=1)
    ref["cancel"] = cancellation(A)
    _cache[key] = (sysm, spec, p, x, ref)
    return _cache[key]


def _model(sysm, spec, p, prec="fp32", chunk=0):
    from jaqmc_amd.device import DeviceModel

    return DeviceModel(spec, sysm.atoms, sysm.charges, p, precision=prec, chunk_walkers=chunk)


@pytest.mark.parametrize("case,B", [("li", 16), ("n2_small", 16), ("n2", 32), ("h60", 8), ("n2_iso", 8),
                                    ("psi_small", 8), ("ring42", 8), ("h_atom", 16), ("li_polarized", 16),
                                    ("h17", 6), ("h24", 6)])
def test_logpsi_and_local_energy_fp32(cuda, case, B):
    import torch

    sysm, spec, p, x, ref = _setup(case, B)
    dm = _model(sysm, spec, p, chunk=5)
    xe = torch.from_numpy(x).to(cuda)
    lp, sg = dm.logpsi(xe)
    out = dm.local_energy(xe, with_grad=True)
    torch.cuda.synchronize()
    lp = lp.cpu().numpy()
    d_lp = np.abs(lp - ref["logpsi"])
    assert np.all(d_lp <= logpsi_bound(ref["logpsi"], ref["kappa"], "fp32", ref["cancel"])), (d_lp, ref["kappa"])
    np.testing.assert_array_equal(sg.cpu().numpy(), ref["sign"])
    d_lap = np.abs(out["logpsi"].cpu().numpy() - lp)
    assert np.all(d_lap <= logpsi_bound(lp, ref["kappa"], "fp32", ref["cancel"])), (d_lap, ref["kappa"])
    np.testing.assert_allclose(out["e_pot"].cpu().numpy(), ref["e_pot"], rtol=1e-6)
    rel, bnd = el_report(f"{case} B={B}", out["e_loc"].cpu().numpy(), ref["e_loc"], ref["kappa"], "fp32",
                         ref["cancel"])
    assert np.all(rel <= bnd), (rel, bnd)
    ek = out["e_kin"].cpu().numpy()
    np.testing.assert_allclose(ek + out["e_pot"].cpu().numpy(), out["e_loc"].cpu().numpy(), rtol=1e-12)
    g = out["grad"].cpu().numpy()
    gd = np.abs(g - ref["grad"]) / np.maximum(1.0, np.abs(ref["grad"]))
    gb = 5e-3 + 2 * ENTRY_ERR["fp32"] * U32 * (ref["kappa"] * ref["cancel"])[:, None]
    assert np.median(gd) <= 2e-4 and np.all(gd <= gb), (gd.max(), ref["kappa"])
    dm.close()


def test_chunking_is_bit_exact(cuda):
    import torch

    sysm, spec, p, x, _ = _setup("n2_small", 16)
    xe = torch.from_numpy(x).to(cuda)
    a = _model(sysm, spec, p, chunk=3)
    b = _model(sysm, spec, p, chunk=64)
    oa, ob = a.local_energy(xe), b.local_energy(xe)
    la, lb = a.logpsi(xe)[0], b.logpsi(xe)[0]
    torch.cuda.synchronize()
    assert torch.equal(oa["e_loc"], ob["e_loc"]) and torch.equal(la, lb)


@pytest.mark.parametrize("case", ["li", "n2_small", "n2"])
def test_metropolis_decisions_match_oracle(cuda, case):
    import torch

    sysm, spec, p, x, ref = _setup(case, 16)
    B, N = x.shape[:2]
    dm = _model(sysm, spec, p)
    rng = np.random.default_rng(21)
    steps, width = 4, 0.05
    normals = rng.standard_normal((steps, B, N, 3)).astype(np.float32)
    uniforms = rng.uniform(size=(steps, B)).astype(np.float32)
    xe = torch.from_numpy(x).to(cuda)
    logp = 2 * dm.logpsi(xe)[0]
    acc = dm.mh_steps(xe, logp, steps, width, normals=torch.from_numpy(normals).to(cuda),
                      uniforms=torch.from_numpy(uniforms).to(cuda))
    torch.cuda.synchronize()
    # oracle, step by step; the band of each decision is 1e-6 plus twice the
    # measured difference of the GPU's and the oracle's log ratio on the same
    # FP32 positions (GPU log|psi| from jq_logpsi, which the Metropolis
    # forward pass shares)
    xo = x.astype(np.float64)
    lpo = 2 * ref["logpsi"]
    p64 = P.cast_params(p, np.float64)
    at64 = sysm.atoms.astype(np.float64)
    nacc = np.zeros(B, int)
    ambiguous = np.zeros(B, bool)
    for s in range(steps):
        xp32 = (xo.astype(np.float32) + np.float32(width) * normals[s]).astype(np.float32)
        lg_x = 2 * dm.logpsi(torch.from_numpy(np.ascontiguousarray(xo.astype(np.float32))).to(cuda))[0].cpu().numpy()
        lg_p = 2 * dm.logpsi(torch.from_numpy(xp32).to(cuda))[0].cpu().numpy()
        xo, lpo_new, a, ratio, logu = ham.mh_step(spec.as_oracle(), p64, xo, lpo, at64, width,
                                                  normals[s].astype(np.float64), uniforms[s].astype(np.float64))
        delta = np.abs((lg_p - lg_x) - ratio)
        ambiguous |= np.abs(ratio - logu) < 1e-6 + 2 * delta
        lpo = lpo_new
        nacc += a
    print(f"[parity] metropolis {case}: {int(ambiguous.sum())} of {B} walkers with a decision inside the "
          f"FP32 band, max |ratio error| {delta.max():.2e}", flush=True)
    ok = ~ambiguous
    np.testing.assert_array_equal(acc.cpu().numpy()[ok], nacc[ok])
    np.testing.assert_allclose(xe.cpu().numpy()[ok], xo[ok], atol=1e-5)
    np.testing.assert_allclose(logp.cpu().numpy()[ok], lpo[ok], atol=2e-4 * np.abs(lpo).max())


def test_philox_sampler_is_keyed_by_walker(cuda):
    import torch

    sysm, spec, p, x, _ = _setup("li", 16)
    dm = _model(sysm, spec, p)
    xa = torch.from_numpy(x).to(cuda)
    xb = xa[:5].clone()
    la = 2 * dm.logpsi(xa)[0]
    lb = la[:5].clone()
    aa = dm.mh_steps(xa, la, 7, 0.1, seed=99, ctr=3)
    ab = dm.mh_steps(xb, lb, 7, 0.1, seed=99, ctr=3)
    torch.cuda.synchronize()
    assert torch.equal(xa[:5], xb) and torch.equal(aa[:5], ab)
    # a different seed gives a different trajectory
    xd = torch.from_numpy(x).to(cuda)[:5].clone()
    ld = la[:5].clone() * 0 + 2 * dm.logpsi(xd)[0]
    dm.mh_steps(xd, ld, 7, 0.1, seed=100, ctr=3)
    torch.cuda.synchronize()
    assert not torch.equal(xd, xb)


def test_reductions_match_numpy(cuda):
    import torch

    from jaqmc_amd.device import reduce_accepts, reduce_mean_var

    rng = np.random.default_rng(0)
    v = rng.standard_normal(10007) * 5 - 3
    v[[5, 77]] = np.nan
    v[100] = np.inf
    out = reduce_mean_var(torch.from_numpy(v).to(cuda)).cpu().numpy()
    ok = v[np.isfinite(v)]
    assert out[2] == ok.size
    assert out[0] == pytest.approx(ok.mean(), rel=1e-12)
    assert out[1] == pytest.approx(ok.var(), rel=1e-9)
    a = rng.integers(0, 20, 5000).astype(np.int32)
    assert reduce_accepts(torch.from_numpy(a).to(cuda)).item() == a.sum()


def test_full_size_n2_batch_properties(cuda):
    """C2 at its full size (4096 walkers): finite energies, swap antisymmetry
    on the GPU, and the batch mean consistent with the FP64 oracle on a sample."""
    import torch

    sysm, spec, B, _, _ = S.workload("n2")
    p = P.init_params(spec, seed=0)
    x = S.init_walkers(sysm, B, seed=0)
    dm = _model(sysm, spec, p)
    xe = torch.from_numpy(x).to(cuda)
    out = dm.local_energy(xe)
    lp, sg = dm.logpsi(xe)
    xs = xe.clone()
    xs[:, [0, 1]] = xs[:, [1, 0]]
    lps, sgs = dm.logpsi(xs)
    torch.cuda.synchronize()
    e = out["e_loc"].cpu().numpy()
    assert np.isfinite(e).mean() > 0.999
    np.testing.assert_allclose(lps.cpu().numpy(), lp.cpu().numpy(), rtol=1e-5, atol=1e-5)
    assert torch.all(sgs == -sg)
    ref = ham.local_energy(spec.as_oracle(), P.cast_params(p, np.float64), x[:32].astype(np.float64),
                           sysm.atoms.astype(np.float64), sysm.charges.astype(np.float64))["e_loc"]
    rel = np.abs(e[:32] - ref) / np.maximum(1, np.abs(ref))
    assert np.median(rel) < 2e-5


@pytest.mark.parametrize("prec,lp_tol,med_tol", [("bf16x6", 2e-3, 5e-5), ("bf16x3", 1e-2, 1e-3),
                                               ("fp16x3", 2e-3, 5e-5)])
def test_mixed_precision_modes(cuda, prec, lp_tol, med_tol):
    """Split 16-bit MFMA modes against the FP64 oracle on N2: bf16x6 (three
    BF16 terms, six products) stays at FP32-level error; bf16x3 (two terms) is
    ~2^-16; fp16x3 (two FP16 terms, three products) ~2^-22."""
    import torch

    sysm, spec, p, x, ref = _setup("n2", 32)
    dm = _model(sysm, spec, p, prec=prec)
    xe = torch.from_numpy(x).to(cuda)
    lp = dm.logpsi(xe)[0]
    out = dm.local_energy(xe)
    torch.cuda.synchronize()
    assert np.abs(lp.cpu().numpy() - ref["logpsi"]).max() < lp_tol  # kappa up to 10^5 on these walkers
    rel, bnd = el_report("n2 B=32", out["e_loc"].cpu().numpy(), ref["e_loc"], ref["kappa"],
                         prec if prec != "bf16x3" else "fp16x3", ref["cancel"])
    assert np.median(rel) < med_tol
    if prec != "bf16x3":
        assert np.all(rel <= bnd), (rel, bnd)


@pytest.mark.parametrize("case,B", [("ring42", 8), ("h60", 8), ("h20_wide", 4), ("h26_wide", 4)])
@pytest.mark.parametrize("prec", ["bf16x6", "fp16x3"])
def test_mixed_precision_large_configs(cuda, case, B, prec):
    """The mixed paths of the 42-electron ring (Psiformer) and H60 (FermiNet,
    60x60 FP64 determinants) against the FP64 oracle, with the kappa-scaled
    per-walker bounds of the FP32 path (entry error of the mode)."""
    import torch

    sysm, spec, p, x, ref = _setup(case, B)
    dm = _model(sysm, spec, p, prec=prec)
    xe = torch.from_numpy(x).to(cuda)
    lp = dm.logpsi(xe)[0]
    out = dm.local_energy(xe, with_grad=True)
    torch.cuda.synchronize()
    d_lp = np.abs(lp.cpu().numpy() - ref["logpsi"])
    assert np.all(d_lp <= logpsi_bound(ref["logpsi"], ref["kappa"], prec, ref["cancel"])), (d_lp, ref["kappa"])
    rel, bnd = el_report(f"{case} B={B}", out["e_loc"].cpu().numpy(), ref["e_loc"], ref["kappa"], prec,
                         ref["cancel"])
    assert np.all(rel <= bnd), (rel, bnd)


@pytest.mark.parametrize("prec", ["fp32", "fp16x3"])
def test_psiformer_padded_units_and_fused_layernorm(cuda, prec):
    """A 41-electron Psiformer (125 tangent rows in 128-row units, 256
    features, one MLP layer): in FP16X3 every LayerNorm runs in the epilogue
    of the preceding GEMM, including the one written over the MLP GEMM's own
    input, and the padding rows stay zero; log|psi| and E_L against the FP64
    oracle with the kappa-scaled bounds of the mode."""
    import torch

    sysm, spec, p, x, ref = _setup("psi41", 4)
    dm = _model(sysm, spec, p, prec=prec)
    xe = torch.from_numpy(x).to(cuda)
    lp = dm.logpsi(xe)[0]
    out = dm.local_energy(xe, with_grad=True)
    torch.cuda.synchronize()
    d_lp = np.abs(lp.cpu().numpy() - ref["logpsi"])
    assert np.all(d_lp <= logpsi_bound(ref["logpsi"], ref["kappa"], prec, ref["cancel"])), (d_lp, ref["kappa"])
    d_lap = np.abs(out["logpsi"].cpu().numpy() - ref["logpsi"])
    assert np.all(d_lap <= logpsi_bound(ref["logpsi"], ref["kappa"], prec, ref["cancel"])), (d_lap, ref["kappa"])
    rel, bnd = el_report(f"psi41 B=4", out["e_loc"].cpu().numpy(), ref["e_loc"], ref["kappa"], prec,
                         ref["cancel"])
    assert np.all(rel <= bnd), (rel, bnd)
    dm.close()


def test_empty_batch_is_a_no_op(cuda):
    import torch

    sysm, spec, p, x, _ = _setup("li", 16)
    dm = _model(sysm, spec, p)
    e = torch.empty(0, spec.n_elec, 3, dtype=torch.float32, device=cuda)
    lp, sg = dm.logpsi(e)
    out = dm.local_energy(e)
    acc = dm.mh_steps(e, torch.empty(0, device=cuda), 3, 0.1)
    torch.cuda.synchronize()
    assert lp.numel() == 0 and out["e_loc"].numel() == 0 and acc.numel() == 0


@pytest.mark.parametrize("case", ["n2_small", "h24"])
def test_coincident_electrons_are_data(cuda, case):
    """Two spin-up electrons at one point: that walker's orbital matrices are
    singular and its pair features divide by r = 0.  The walker's results are
    data (log|psi| far below its regular value or non-finite, no error) and
    every other walker of the batch is bit-identical to the regular run
    (estimator/base.py:44 treats non-finite E_L as data).  Covers the N <= 16
    and 16 < N <= 64 determinant kernels."""
    import torch

    sysm, spec, p, x, _ = _setup(case, 6)
    xs = x.copy()
    xs[2, 1] = xs[2, 0]
    dm = _model(sysm, spec, p)
    lp, _ = dm.logpsi(torch.from_numpy(xs).to(cuda))
    out = dm.local_energy(torch.from_numpy(xs).to(cuda))
    lp0, _ = dm.logpsi(torch.from_numpy(x).to(cuda))
    out0 = dm.local_energy(torch.from_numpy(x).to(cuda))
    torch.cuda.synchronize()
    keep = [0, 1, 3, 4, 5]
    assert torch.equal(lp[keep], lp0[keep])
    assert torch.equal(out["e_loc"][keep], out0["e_loc"][keep])
    v = lp[2].item()
    assert (not np.isfinite(v)) or v < lp0[2].item() - 5.0, (v, lp0[2].item())


@pytest.mark.parametrize("n", [20, 31, 33, 40, 47, 52, 57, 63])
def test_forward_logdet_every_padded_size(cuda, n):
    """log|psi| and sign on the forward (Metropolis) path for hydrogen chains
    whose electron counts reach every padded size of the register LU kernel
    (24 ... 64 in steps of 8), one determinant so log|psi| and sign are those
    of det A itself; against the FP64 oracle (jnp.linalg.slogdet,
    wavefunction/output/logdet.py:65) within the log|det| perturbation bound."""
    import torch

    sysm = S.h_chain(n)
    _, spec, *_ = S.workload("li")
    spec.nspins = sysm.nspins
    spec.n_atoms = n
    spec.hidden_single, spec.hidden_double, spec.ndets = [32, 32], [8, 8], 1
    p = P.init_params(spec, seed=5, bias_scale=0.1, env_jitter=0.2)
    x = S.init_walkers(sysm, 6, seed=6)
    p64 = P.cast_params(p, np.float64)
    at = sysm.atoms.astype(np.float64)
    sg_ref, lp_ref = owf.logpsi(spec.as_oracle(), p64, x.astype(np.float64), at, with_laplacian=False)
    A = np.asarray(owf.orbital_matrices(spec.as_oracle(), p64, x.astype(np.float64), at))
    kappa = np.linalg.cond(A).reshape(x.shape[0], -1).max(axis=1)
    dm = _model(sysm, spec, p)
    lp, sg = dm.logpsi(torch.from_numpy(x).to(cuda))
    torch.cuda.synchronize()
    d = np.abs(lp.cpu().numpy() - lp_ref.v)
    assert np.all(d <= logpsi_bound(lp_ref.v, kappa, "fp32")), (d, kappa)
    np.testing.assert_array_equal(sg.cpu().numpy(), np.asarray(sg_ref).reshape(-1))
    dm.close()


def test_psiformer_chunking_and_bf16x6(cuda):
    """Psiformer: chunked evaluation is bit-exact, and bf16x6 stays at FP32-level error."""
    import torch

    sysm, spec, p, x, ref = _setup("psi_small", 8)
    xe = torch.from_numpy(x).to(cuda)
    a = _model(sysm, spec, p, chunk=3)
    b = _model(sysm, spec, p, chunk=8)
    c = _model(sysm, spec, p, prec="bf16x6", chunk=8)
    oa, ob, oc = a.local_energy(xe), b.local_energy(xe), c.local_energy(xe)
    torch.cuda.synchronize()
    assert torch.equal(oa["e_loc"], ob["e_loc"])
    rel, bnd = el_report("psi_small B=8", oc["e_loc"].cpu().numpy(), ref["e_loc"], ref["kappa"], "bf16x6",
                         ref["cancel"])
    assert np.median(rel) < 2e-5 and np.all(rel <= bnd)


# batches on every tile of the plain GEMM's table (16 to 128 rows, 64 and 128
# columns; value rows of 14 electrons, 256-wide layers and 12 x 14 orbitals)
@pytest.mark.parametrize("prec", ["fp32", "fp16x3"])
def test_value_batches_are_bit_identical(cuda, prec):
    """A walker's log|psi| does not depend on the batch it is evaluated in, so
    neither on the tile that the batch's size selects."""
    import torch

    from jaqmc_amd import params as P
    from jaqmc_amd import systems as S
    from jaqmc_amd.device import DeviceModel

    sysm, spec, *_ = S.workload("n2")
    spec.ndets = 12
    p = P.init_params(spec, seed=71, bias_scale=0.1, env_jitter=0.3)
    x = torch.from_numpy(S.init_walkers(sysm, 4100, seed=72)).to(cuda)
    dm = DeviceModel(spec, sysm.atoms, sysm.charges, p, precision=prec)
    lp, sign = dm.logpsi(x)
    for n in (1, 7, 60, 333, 1201):
        for at in (0, 4100 - n):
            a, b = dm.logpsi(x[at:at + n].contiguous())
            assert torch.equal(a, lp[at:at + n]) and torch.equal(b, sign[at:at + n]), (n, at)
    dm.close()


# the padded sizes 4, 8, 12 and 16 of the column-per-lane kernel, full and not
@pytest.mark.parametrize("n", [1, 2, 4, 5, 8, 9, 12, 13, 16])
def test_forward_logdet_small_sizes(cuda, n):
    """As test_forward_logdet_every_padded_size, for up to 16 electrons (seven
    matrices: the last group of sixteen is not full)."""
    import torch

    sysm = S.h_chain(n)
    _, spec, *_ = S.workload("li")
    spec.nspins = sysm.nspins
    spec.n_atoms = n
    spec.hidden_single, spec.hidden_double, spec.ndets = [32, 32], [8, 8], 1
    p = P.init_params(spec, seed=5, bias_scale=0.1, env_jitter=0.2)
    x = S.init_walkers(sysm, 7, seed=6)
    p64 = P.cast_params(p, np.float64)
    at = sysm.atoms.astype(np.float64)
    sg_ref, lp_ref = owf.logpsi(spec.as_oracle(), p64, x.astype(np.float64), at, with_laplacian=False)
    A = np.asarray(owf.orbital_matrices(spec.as_oracle(), p64, x.astype(np.float64), at))
    kappa = np.linalg.cond(A).reshape(x.shape[0], -1).max(axis=1)
    dm = _model(sysm, spec, p)
    lp, sg = dm.logpsi(torch.from_numpy(x).to(cuda))
    torch.cuda.synchronize()
    d = np.abs(lp.cpu().numpy() - lp_ref.v)
    assert np.all(d <= logpsi_bound(lp_ref.v, kappa, "fp32")), (d, kappa)
    np.testing.assert_array_equal(sg.cpu().numpy(), np.asarray(sg_ref).reshape(-1))
    dm.close()


# the on-chip pair stream (every pair width 32): no, one, two and three layers,
# one electron, one spin channel, ragged 16-row blocks, eight-wave workgroups
PAIR_CASES = {
    "h5_1": (lambda: S.h_chain(5), 1),
    "h_2": (_hydrogen, 2),
    "h17_3": (_h17, 3),
    "li_polarized_4": (_polarized_li, 4),
    "h39_4": (lambda: S.h_chain(39), 4),
}


@pytest.mark.parametrize("case", list(PAIR_CASES))
def test_pair_stream_layers(cuda, case):
    """log|psi| and E_L against the FP64 oracle, to this file's bounds."""
    import torch

    mk, layers = PAIR_CASES[case]
    sysm = mk()
    _, spec, *_ = S.workload("li")
    spec.nspins, spec.n_atoms = sysm.nspins, sysm.atoms.shape[0]
    spec.hidden_single, spec.hidden_double, spec.ndets = [32] * layers, [32] * layers, 2
    p = P.init_params(spec, seed=81, bias_scale=0.1, env_jitter=0.5)
    x = S.init_walkers(sysm, 5, seed=82)
    p64, x64, at = P.cast_params(p, np.float64), x.astype(np.float64), sysm.atoms.astype(np.float64)
    ref = ham.local_energy(spec.as_oracle(), p64, x64, at, sysm.charges.astype(np.float64))
    A = np.asarray(owf.orbital_matrices(spec.as_oracle(), p64, x64, at))
    kappa, cancel = np.linalg.cond(A).reshape(5, -1).max(axis=1), cancellation(A)
    dm = _model(sysm, spec, p)
    xe = torch.from_numpy(x).to(cuda)
    lp, sg = dm.logpsi(xe)
    out = dm.local_energy(xe)
    bound = logpsi_bound(ref["logpsi"], kappa, "fp32", cancel)
    assert np.all(np.abs(lp.cpu().numpy() - ref["logpsi"]) <= bound)
    assert np.all(np.abs(out["logpsi"].cpu().numpy() - ref["logpsi"]) <= bound)
    np.testing.assert_array_equal(sg.cpu().numpy(), ref["sign"])
    rel, bnd = el_report(case, out["e_loc"].cpu().numpy(), ref["e_loc"], kappa, "fp32", cancel)
    assert np.all(rel <= bnd), (rel, bnd)
    dm.close()


# networks of the one-kernel value path: electrons per 16-row tile and its
# remainders, one channel, every envelope, shared orbitals, pair widths whose
# layers add the bias first (16) and last (8, 12), layers of 32 to 96
SMALL_CASES = {
    "h1": (_hydrogen, dict(hidden_single=[32, 32], hidden_double=[8, 8], ndets=2)),
    "li": (S.li_atom, dict(hidden_single=[64, 64], hidden_double=[16, 16], ndets=4, envelope="isotropic")),
    "li_polarized": (_polarized_li, dict(hidden_single=[32, 64, 64], hidden_double=[8, 12, 12], ndets=3)),
    "h5_shared": (lambda: S.h_chain(5), dict(hidden_single=[96, 96], hidden_double=[12, 16], ndets=5,
                                             orbitals_spin_split=False)),
    "h9_null": (lambda: S.h_chain(9), dict(hidden_single=[64], hidden_double=[16], ndets=1, envelope="null")),
    "h16": (lambda: S.h_chain(16), dict(hidden_single=[32, 32, 32, 32], hidden_double=[16, 16, 16, 16], ndets=2)),
}


@pytest.mark.parametrize("case", list(SMALL_CASES))
def test_small_network_kernel_is_bit_identical(cuda, case):
    """Walkers of a batch too large for the one-kernel path and the same walkers
    in a batch that takes it: the same log|psi|, signs and trajectories, with
    Philox and with given random numbers, and through the device sampler."""
    import torch

    mk, kw = SMALL_CASES[case]
    sysm = mk()
    _, spec, *_ = S.workload("li")
    spec.nspins, spec.n_atoms = sysm.nspins, sysm.atoms.shape[0]
    for k, v in kw.items():
        setattr(spec, k, v)
    p = P.init_params(spec, seed=91, bias_scale=0.1, env_jitter=0.5)
    N = spec.n_elec
    B, n = 5 * 256 * (16 // N) + 1, 77
    x = torch.from_numpy(S.init_walkers(sysm, B, seed=92)).to(cuda)
    dm = _model(sysm, spec, p)

    def evaluate(x):
        x = x.clone()
        lp, sg = dm.logpsi(x)
        logp = 2 * lp
        acc = dm.mh_steps(x, logp, 3, 0.3, seed=5, ctr=11)
        g = torch.Generator(device="cpu").manual_seed(3)
        normals, uniforms = torch.randn(2, n, N, 3, generator=g), torch.rand(2, n, generator=g)
        pad = len(x) - n  # the walkers compared have the same numbers in both batches
        normals = torch.cat([normals, torch.zeros(2, pad, N, 3)], 1).to(cuda)
        uniforms = torch.cat([uniforms, torch.full((2, pad), 0.5)], 1).to(cuda)
        dm.mh_steps(x, logp, 2, 0.2, normals=normals, uniforms=uniforms, n_accept=acc)
        moved = (x.clone(), logp.clone())
        state = torch.zeros(3 + 4, dtype=torch.float64, device=cuda)
        state[0] = 0.25
        logp2, acc2 = dm.sample(x, state, 2, 3, adapt_frequency=4, seed=9)
        return lp, sg, *moved, acc, x, logp2, acc2

    big, small = evaluate(x), evaluate(x[:n].contiguous())
    dm.close()
    for a, b in zip(big, small):
        assert torch.equal(a[:n], b)
    assert 0 < int(small[4].sum()) < 5 * n or N == 1


# 48-, 96- and 128-row units: a last tile of one unit of two, column blocks that
# are not full (24 x 13, 16 x 30, 12 x 42 orbitals), head-split projections
@pytest.mark.parametrize("n,ndets,B", [(13, 24, 159), (30, 16, 35), (42, 12, 25)])
def test_wide_projections_are_bit_identical(cuda, n, ndets, B):
    """In FP16X3 a batch whose projections run on whole row panels gives every
    walker the results of chunks too small for them."""
    import torch

    sysm = S.h_chain(n)
    _, spec, *_ = S.workload("ring42")
    spec.nspins, spec.n_atoms, spec.ndets, spec.num_layers = sysm.nspins, n, ndets, 2
    p = P.init_params(spec, seed=101, bias_scale=0.1, env_jitter=0.3)
    x = torch.from_numpy(S.init_walkers(sysm, B, seed=102)).to(cuda)
    out = []
    for chunk in (0, B // 3):
        dm = _model(sysm, spec, p, prec="fp16x3", chunk=chunk)
        out.append(dm.local_energy(x, with_grad=True))
        torch.cuda.synchronize()
        dm.close()
    for k, v in out[0].items():
        assert torch.equal(v, out[1][k]), k
    assert torch.isfinite(out[0]["e_loc"]).all()


# one to four dense layers, one layer (no projection after it), narrow heads,
# padding rows, fewer units than CUs and more
@pytest.mark.parametrize("n,B,kw", [
    (33, 2, dict(num_layers=2, mlp_hidden=[])),
    (32, 9, dict(num_layers=2, mlp_hidden=[256, 256, 256])),
    (37, 3, dict(num_layers=3, num_heads=8, heads_dim=32)),
    (42, 2, dict(num_layers=1, mlp_hidden=[256, 256])),
])
def test_psiformer_row_wise_chain(cuda, n, B, kw):
    """The row-wise part of 256-wide pre-LN layers in one kernel: log|psi| and
    E_L against the FP64 oracle, to this file's bounds."""
    import torch

    sysm = S.h_chain(n)
    _, spec, *_ = S.workload("ring42")
    spec.nspins, spec.n_atoms, spec.ndets = sysm.nspins, n, 2
    for k, v in kw.items():
        setattr(spec, k, v)
    p = P.init_params(spec, seed=111, bias_scale=0.1, env_jitter=0.3)
    x = S.init_walkers(sysm, B, seed=112)
    p64, x64, at = P.cast_params(p, np.float64), x.astype(np.float64), sysm.atoms.astype(np.float64)
    ref = ham.local_energy(spec.as_oracle(), p64, x64, at, sysm.charges.astype(np.float64))
    A = np.asarray(owf.orbital_matrices(spec.as_oracle(), p64, x64, at))
    kappa, cancel = np.linalg.cond(A).reshape(B, -1).max(axis=1), cancellation(A)
    dm = _model(sysm, spec, p, prec="fp16x3")
    out = dm.local_energy(torch.from_numpy(x).to(cuda))
    torch.cuda.synchronize()
    bound = logpsi_bound(ref["logpsi"], kappa, "fp16x3", cancel)
    assert np.all(np.abs(out["logpsi"].cpu().numpy() - ref["logpsi"]) <= bound)
    rel, bnd = el_report(f"chain {n}", out["e_loc"].cpu().numpy(), ref["e_loc"], kappa, "fp16x3", cancel)
    assert np.all(rel <= bnd), (rel, bnd)
    dm.close()


# one determinant of three exactly singular: zero at once, from its first column,
# at its last; full and not full sizes of the column-per-lane kernel, the
# row-per-lane kernel; fp32 at up to 16 electrons: the one-kernel network
@pytest.mark.parametrize("prec", ["fp32", "fp16x3"])
@pytest.mark.parametrize("n", [2, 3, 4, 9, 13, 16, 17, 33])
def test_singular_determinant_among_several(cuda, n, prec):
    """log|psi| and its sign are those of the other determinants (slogdet of a
    singular matrix is -inf), against the FP64 oracle to this file's bounds."""
    import torch

    sysm = S.h_chain(n)
    _, spec, *_ = S.workload("li")
    spec.nspins, spec.n_atoms = sysm.nspins, n
    spec.hidden_single, spec.hidden_double, spec.ndets = [32, 32], [8, 8], 3
    x = S.init_walkers(sysm, 7, seed=6)
    at = sysm.atoms.astype(np.float64)
    for orbitals in (slice(None), slice(0, 1), slice(n - 1, n)):
        p = P.init_params(spec, seed=5, bias_scale=0.1, env_jitter=0.2)
        for pi, _ in p["envelope"]:
            pi[orbitals, :, 1] = 0.0  # these columns of determinant 1 vanish
        p64 = P.cast_params(p, np.float64)
        A = np.asarray(owf.orbital_matrices(spec.as_oracle(), p64, x.astype(np.float64), at))
        assert np.all(np.linalg.slogdet(A[:, 1])[1] == -np.inf)
        others = A[:, [0, 2]]
        kappa, cancel = np.linalg.cond(others).max(axis=1), cancellation(others)
        s, l = np.linalg.slogdet(others)
        m = l.max(axis=1, keepdims=True)
        total = (s * np.exp(l - m)).sum(axis=1)
        ref = np.log(np.abs(total)) + m[:, 0]
        dm = _model(sysm, spec, p, prec=prec, chunk=7)
        lp, sg = dm.logpsi(torch.from_numpy(x).to(cuda))
        d = np.abs(lp.cpu().numpy() - ref)
        assert np.all(d <= logpsi_bound(ref, kappa, prec, cancel)), (orbitals, d)
        np.testing.assert_array_equal(sg.cpu().numpy(), np.sign(total))
        dm.close()


def test_singular_walker_with_a_nan_stays_nan(cuda):
    """A zero column does not hide a NaN in the matrix."""
    import torch

    for n in (3, 17):
        sysm = S.h_chain(n)
        _, spec, *_ = S.workload("li")
        spec.nspins, spec.n_atoms = sysm.nspins, n
        spec.hidden_single, spec.hidden_double, spec.ndets = [32, 32], [8, 8], 1
        p = P.init_params(spec, seed=5, bias_scale=0.1, env_jitter=0.2)
        for pi, _ in p["envelope"]:
            pi[0] = 0.0
            pi[1] = np.nan
        for prec in ("fp32", "fp16x3"):
            dm = _model(sysm, spec, p, prec=prec, chunk=7)
            lp, _ = dm.logpsi(torch.from_numpy(S.init_walkers(sysm, 7, seed=6)).to(cuda))
            assert torch.isnan(lp).all(), (n, prec)
            dm.close()


def test_small_network_launches_are_profiled(cuda):
    """JQ_PROF_FORWARD records the value path of a small network: one launch of
    log|psi|, one for the moves of a call, one per outer step of the sampler."""
    import torch

    from jaqmc_amd import _lib

    sysm, spec, *_ = S.workload("li")
    dm = _model(sysm, spec, P.init_params(spec, seed=0, bias_scale=0.1))
    x = torch.from_numpy(S.init_walkers(sysm, 64, seed=1)).to(cuda)
    logp = 2 * dm.logpsi(x)[0]
    state = torch.zeros(3 + 4, dtype=torch.float64, device=cuda)
    state[0] = 0.2
    counts = []
    for call in (lambda: dm.logpsi(x), lambda: dm.mh_steps(x, logp, 5, 0.1, seed=2),
                 lambda: dm.sample(x, state, 2, 3, adapt_frequency=4, seed=9)):
        _lib.profile_enable(True)
        call()
        _lib.profile_enable(False)
        ms, n = _lib.profile_read("forward")
        assert ms > 0
        counts.append(n)
    assert counts == [1, 1, 2]
    dm.close()


# workgroups (16 // electrons walkers each) on both sides of the lines between the
# one-kernel path and the general one: log|psi|, moves
@pytest.mark.parametrize("n,width,layers,most,most_moves", [
    (3, 64, 2, 1280, 1280), (14, 64, 2, 1024, 1024), (14, 96, 2, 512, 1024), (14, 128, 4, 512, 512),
    (16, 128, 4, 256, 256), (10, 192, 2, 256, 512), (3, 256, 2, 256, 512)])
def test_small_network_kernel_ends_where_it_loses(cuda, n, width, layers, most, most_moves):
    """A batch takes one launch up to the workgroups that a CU works off faster
    than the general path's launches, and that path's chunks beyond."""
    import torch

    from jaqmc_amd import _lib

    sysm = S.h_chain(n)
    _, spec, *_ = S.workload("li")
    spec.nspins, spec.n_atoms, spec.ndets = sysm.nspins, n, 4
    spec.hidden_single, spec.hidden_double = [width] * layers, [16] * layers
    dm = _model(sysm, spec, P.init_params(spec, seed=0, bias_scale=0.1), chunk=1)

    def launches(walkers, moves):
        x = torch.from_numpy(S.init_walkers(sysm, walkers, seed=1)).to(cuda)
        logp = torch.zeros(walkers, device=cuda)
        _lib.profile_enable(True)
        dm.mh_steps(x, logp, 1, 0.1, seed=2) if moves else dm.logpsi(x)
        _lib.profile_enable(False)
        return _lib.profile_read("forward")[1]

    G = 16 // n
    got = [launches(w, moves) for moves, line in ((False, most), (True, most_moves)) for w in (line * G, line * G + 1)]
    dm.close()
    assert got[0] == got[2] == 1 and got[1] > 1 and got[3] > 1, got


@pytest.mark.parametrize("prec", ["fp32", "bf16", "bf16x3", "bf16x6", "fp16x3"])
def test_bench_gemm_takes_every_plain_variant(cuda, prec):
    """jq_bench_gemm times plain rows with any variant: the tile it names, or the
    default where there is none of that name; Laplacian rows only with a tile."""
    import ctypes

    from jaqmc_amd import _lib

    lib = _lib.load()
    ms = ctypes.c_float()

    def bench(R, variant):
        ms.value = -1.0
        rc = lib.jq_bench_gemm(_lib.PRECISION[prec], R, 960, 64, 96, 0, variant, 2, ctypes.byref(ms))
        return rc, ms.value

    for variant in (0, 11, 21, 41, 82, 12, 42, 14, 24, 84, 142):
        rc, t = bench(1, variant)
        assert rc == 0 and t > 0, variant
    assert bench(48, 22)[0] == 0 and bench(48, 91)[0] == -1


# as test_psiformer_row_wise_chain, and heads of 128, several units a workgroup,
# every remainder of an MLP's depth
@pytest.mark.parametrize("n,B,kw", [
    (32, 2, dict(num_layers=2, mlp_hidden=[])),
    (33, 9, dict(num_layers=2, mlp_hidden=[256, 256])),
    (35, 1, dict(num_layers=2, num_heads=2, heads_dim=128)),
    (37, 3, dict(num_layers=3, num_heads=8, heads_dim=32)),
    (39, 20, dict(num_layers=1)),
    (42, 13, dict(num_layers=4)),
    (42, 2, dict(num_layers=2, mlp_hidden=[256, 256, 256])),
])
def test_psiformer_chain_is_bit_identical(cuda, n, B, kw):
    """Layers whose row-wise part runs in one kernel and the same layers in a
    launch a stage: the same log|psi|, energies and gradients."""
    import torch

    from jaqmc_amd.device import DeviceModel

    sysm = S.h_chain(n)
    _, spec, *_ = S.workload("ring42")
    spec.nspins, spec.n_atoms, spec.ndets = sysm.nspins, n, 2
    for k, v in kw.items():
        setattr(spec, k, v)
    p = P.init_params(spec, seed=121, bias_scale=0.1, env_jitter=0.3)
    x = torch.from_numpy(S.init_walkers(sysm, B, seed=122)).to(cuda)
    out = []
    for separate in (False, True):
        dm = DeviceModel(spec, sysm.atoms, sysm.charges, p, precision="fp16x3", chunk_walkers=B,
                         separate_launches=separate)
        out.append(dm.local_energy(x, with_grad=True))
        torch.cuda.synchronize()
        dm.close()
    for k, v in out[0].items():
        assert torch.equal(v, out[1][k]), k
    assert torch.isfinite(out[0]["e_loc"]).all()


def test_separate_launches_run_the_stages_apart(cuda):
    """JQ_OPT_SEPARATE_LAUNCHES: more layer launches for the Psiformer, chunks in
    place of the one-kernel value path for a small FermiNet."""
    import torch

    from jaqmc_amd import _lib
    from jaqmc_amd.device import DeviceModel

    sysm, spec, *_ = S.workload("ring42")
    p = P.init_params(spec, seed=0)
    counts = []
    for separate in (False, True):
        dm = DeviceModel(spec, sysm.atoms, sysm.charges, p, precision="fp16x3", chunk_walkers=2,
                         separate_launches=separate)
        x = torch.from_numpy(S.init_walkers(sysm, 2, seed=1)).to(cuda)
        dm.local_energy(x)
        _lib.profile_enable(True)
        dm.local_energy(x)
        _lib.profile_enable(False)
        counts.append(_lib.profile_read("gemm_layer_lap")[1])
        dm.close()
    L, stages = spec.num_layers, 2 + len(spec.mlp_hidden) + 1  # q k v, output projection, MLP
    assert counts == [1 + 1 + L, 1 + L * stages]  # the input projection; its first q k v; the layers
    sysm, spec, *_ = S.workload("li")
    dm = DeviceModel(spec, sysm.atoms, sysm.charges, P.init_params(spec, seed=0), chunk_walkers=1,
                     separate_launches=True)
    x = torch.from_numpy(S.init_walkers(sysm, 400, seed=1)).to(cuda)
    _lib.profile_enable(True)
    dm.logpsi(x)
    _lib.profile_enable(False)
    assert _lib.profile_read("forward")[1] > 1
    dm.close()
