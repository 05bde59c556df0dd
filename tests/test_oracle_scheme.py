"""CPU oracle: the QE scheme, the reference time grid and the Monte-Carlo estimator.

Pins (none of them restates the oracle's formulas):
 * QE variance step: the exact CIR conditional mean and variance (Andersen 2008, eqs. 17-18) are
   reproduced by both branches; the exponential branch's mass at 0 is p = (psi-1)/(psi+1).
 * Log-price step: exactly, given V and V', the increment is Andersen's eq. (33) with the central
   weights gamma1 = gamma2 = 1/2 (intercept and slope of the affine map Z -> d ln X over a grid of
   the draw's words, normals from scipy); planted CPU copies with other weights, a flipped rho/eps
   sign or no K0 fail the same check. Also: with rho = 0 the step is conditionally lognormal with
   E[X'/X] = 1 exactly; in the sigma -> 0 limit with v0 = theta the model is GBM, so European
   prices equal Black-Scholes.
 * Time grid (src/HSimulation.tpp:35-44) and the Asian finalisation quirk
   (src/inc/AsianContract.h:29-34): the case table of n* per (T, N), and the K = 0 invariant
   E[A] = S0 (N-1)/N when the last step lands on T, S0 otherwise.
 * Estimator: prices and standard errors equal numpy's mean and std of the per-path payoffs.
"""
import json
import os

import numpy as np
import pytest
from scipy.stats import norm

from oracle import oracle as O

GOLD = os.path.join(os.path.dirname(__file__), "golden")
BASE = [0.04, 0.04, -0.7, 2.0, 0.3]


def cir_moments(V, delta, theta, kappa, eps):
    e = np.exp(-kappa * delta)
    m = theta + (V - theta) * e
    s2 = V * eps * eps * e / kappa * (1 - e) + theta * eps * eps / (2 * kappa) * (1 - e) ** 2
    return m, s2


@pytest.mark.parametrize("V,delta,kappa,theta,eps", [
    (0.04, 1 / 52, 2.0, 0.04, 0.3),      # quadratic branch (psi small)
    (0.002, 1 / 252, 0.5, 0.04, 0.9),    # exponential branch (psi large)
    (0.01, 1 / 12, 1.0, 0.09, 1.0),      # mixed regime
    (0.0, 1 / 100, 3.0, 0.05, 0.6),      # from V = 0
])
def test_qe_step_reproduces_cir_moments(V, delta, kappa, theta, eps):
    params = [V, theta, -0.5, kappa, eps]
    n = 2_000_000
    r = O.qe_moments(params, delta, V, n, seed=11)
    m, s2 = cir_moments(V, delta, theta, kappa, eps)
    se_mean = np.sqrt(s2 / n)
    se_var = np.sqrt(max(r["m4"] - r["var"] ** 2, 1e-300) / n)
    assert abs(r["mean"] - m) < 5 * se_mean, (r["mean"], m, se_mean)
    assert abs(r["var"] - s2) < 5 * se_var, (r["var"], s2, se_var)
    psi = s2 / m ** 2
    if psi < 1.5:
        assert r["quad_frac"] == 1.0 and r["zero_frac"] == 0.0
    else:
        p = (psi - 1) / (psi + 1)
        assert r["quad_frac"] == 0.0
        assert abs(r["zero_frac"] - p) < 5 * np.sqrt(p * (1 - p) / n)


# ---- the log-price step, exactly -------------------------------------------------------------
# Andersen (2008), "Simple and efficient simulation of the Heston stochastic volatility model",
# J. Comput. Finance 11(3), eq. (33): given V(t) and V(t + D),
#   ln X(t + D) = ln X(t) + K0 + K1 V(t) + K2 V(t + D) + sqrt(K3 V(t) + K4 V(t + D)) Z,
#   K0 = -rho kappa theta D / eps,
#   K1 = g1 D (kappa rho / eps - 1/2) - rho / eps,   K2 = g2 D (kappa rho / eps - 1/2) + rho / eps,
#   K3 = g1 D (1 - rho^2),                           K4 = g2 D (1 - rho^2),
# with the central discretisation g1 = g2 = 1/2, the one src/HSimulation.tpp:75-80 takes.
GAMMA1 = GAMMA2 = 0.5


def andersen_eq33(params, delta, gamma1=GAMMA1, gamma2=GAMMA2):
    _, theta, rho, kappa, eps = params
    k0 = -rho * kappa * theta * delta / eps
    k1 = gamma1 * delta * (kappa * rho / eps - 0.5) - rho / eps
    k2 = gamma2 * delta * (kappa * rho / eps - 0.5) + rho / eps
    k3 = gamma1 * delta * (1.0 - rho * rho)
    k4 = gamma2 * delta * (1.0 - rho * rho)
    return k0, k1, k2, k3, k4


def words_midpoint(log2_n):
    """The midpoints of 2^log2_n equal intervals of the 32-bit words, and their uniforms
    u = (w + 1/2) 2^-32 as the oracle maps them; the normals come from scipy's ndtri."""
    from scipy.special import ndtri
    s = 32 - log2_n
    w = (np.arange(2 ** log2_n, dtype=np.uint64) << np.uint64(s)) | np.uint64(1 << (s - 1))
    return w.astype(np.uint32), ndtri((w.astype(np.float64) + 0.5) * 2.0 ** -32)


def check_log_step(step, params, delta, V, w_v, log2_n=12):
    """Fixes V and the variance draw's word (so V' is fixed) and runs `step` over a midpoint grid
    of the log-price draw's word. The log-price increment must be the affine function
    a + b Z of the draw's normal Z with a = K0 + K1 V + K2 V' and b^2 = K3 V + K4 V' of eq. (33)."""
    words, z = words_midpoint(log2_n)
    out = [step(params, delta, V, 0.0, int(w_v), int(wx)) for wx in words]
    vn = np.array([o[0] for o in out])
    dlx = np.array([o[1] for o in out])
    assert np.all(vn == vn[0])  # the variance step does not look at the log-price draw
    k0, k1, k2, k3, k4 = andersen_eq33(params, delta)
    a = k0 + k1 * V + k2 * vn[0]
    b2 = k3 * V + k4 * vn[0]
    A = np.stack([np.ones_like(z), z], axis=1)
    (fa, fb), *_ = np.linalg.lstsq(A, dlx, rcond=None)
    scale = abs(a) + abs(fb) * 4.0 + 1e-300
    ok = (np.max(np.abs(dlx - (fa + fb * z))) <= 1e-12 * scale and abs(fa - a) <= 1e-12 * scale and
          abs(fb * fb - b2) <= 1e-10 * b2 + 1e-300)
    return ok, (fa, a, fb * fb, b2, vn[0])


# (params, delta, V, w_v): both variance branches, V' far from V (where the split between K1 and
# K2 matters), V' = 0 from the exponential branch, the stiff benchmark's parameters
LOG_STEP_CASES = [
    ([0.04, 0.04, -0.7, 2.0, 0.3], 1 / 52, 0.04, 0x10000000),     # quadratic, Z_V = -1.15: V' < V
    ([0.04, 0.04, -0.7, 2.0, 0.3], 1 / 52, 0.02, 0xF8000000),     # quadratic, Z_V = +2.0: V' > V
    ([0.04, 0.04, -0.9, 0.5, 0.9], 1 / 2048, 0.00005, 0x20000000),  # exponential, U = 1/8 < p: V' = 0
    ([0.04, 0.04, -0.9, 0.5, 0.9], 1 / 52, 0.001, 0xFF000000),     # exponential, U near 1: V' >> V
    ([0.09, 0.04, 0.5, 3.0, 0.6], 0.25, 0.09, 0x40000000),         # positive rho, long step
]


@pytest.mark.parametrize("params,delta,V,w_v", LOG_STEP_CASES)
def test_log_step_equals_andersen_eq33_with_central_weights(params, delta, V, w_v):
    ok, info = check_log_step(O.qe_step, params, delta, V, w_v)
    assert ok, info


def _planted_step(gamma1, gamma2, flip_rho_over_eps=False, drop_k0=False):
    """A CPU copy of the oracle's step with a planted change in the log-price coefficients (the
    variance step is the oracle's own, so V' is the same)."""
    def step(params, delta, V, logX, w_v, w_x):
        vn, _, _ = O.qe_step(params, delta, V, logX, w_v, w_x)
        _, theta, rho, kappa, eps = params
        k0 = 0.0 if drop_k0 else -rho * kappa * theta * delta / eps
        s = -1.0 if flip_rho_over_eps else 1.0
        k1 = gamma1 * delta * (kappa * rho / eps - 0.5) - s * rho / eps
        k2 = gamma2 * delta * (kappa * rho / eps - 0.5) + s * rho / eps
        k3, k4 = gamma1 * delta * (1 - rho * rho), gamma2 * delta * (1 - rho * rho)
        z = O.normals_f64([w_x])[0]
        return vn, logX + k0 + k1 * V + k2 * vn + np.sqrt(k3 * V + k4 * vn) * z
    return step


@pytest.mark.parametrize("planted", ["euler_gamma1", "backward_gamma2", "rho_over_eps_sign", "no_k0"])
def test_log_step_check_rejects_planted_mistakes(planted):
    """The check above catches a re-weighting of gamma (which the rho = 0 martingale test and the
    sigma -> 0 limit cannot see: both hold for any gamma1 + gamma2 = 1), a sign error in the
    rho / eps terms and a dropped K0, on at least one of the cases; and it passes a correct copy."""
    step = {"euler_gamma1": _planted_step(1.0, 0.0), "backward_gamma2": _planted_step(0.0, 1.0),
            "rho_over_eps_sign": _planted_step(0.5, 0.5, flip_rho_over_eps=True),
            "no_k0": _planted_step(0.5, 0.5, drop_k0=True)}[planted]
    results = [check_log_step(step, *c, log2_n=8)[0] for c in LOG_STEP_CASES]
    assert not all(results), planted
    assert all(check_log_step(_planted_step(0.5, 0.5), *c, log2_n=8)[0] for c in LOG_STEP_CASES)


def test_log_step_is_martingale_without_correlation():
    r = O.qe_moments([0.04, 0.04, 0.0, 2.0, 0.5], 1 / 12, 0.04, 2_000_000, seed=3)
    assert abs(r["mean_exp_dlogx"] - 1.0) < 5 * np.sqrt(0.04 / 12 / 2_000_000) * 1.5


def bs_call(S, K, T, vol, r=0.0):
    d1 = (np.log(S / K) + (r + 0.5 * vol * vol) * T) / (vol * np.sqrt(T))
    return S * norm.cdf(d1) - K * np.exp(-r * T) * norm.cdf(d1 - vol * np.sqrt(T))


def test_black_scholes_limit():
    """sigma -> 0 with v0 = theta: every step is an exact GBM step with vol sqrt(theta); the
    rho/eps terms of the log-price step must combine to it (rho = -0.7 keeps them large)."""
    params = [0.04, 0.04, -0.7, 2.0, 1e-5]
    K = np.array([80.0, 100.0, 120.0])
    out = O.price(params, 100.0, [1.0], [3], K, steps=50, n_paths=400_000, seed=21, payoffs=O.EUROPEAN)
    ref = bs_call(100.0, K, 1.0, 0.2)
    assert np.all(np.abs(out["prices"] - ref) < 4 * out["std_errs"]), (out["prices"], ref, out["std_errs"])
    # with the drift and discount extensions the same holds at r = 5%
    out = O.price(params, 100.0, [1.0], [3], K, steps=50, n_paths=400_000, seed=22, r=0.05,
                  flags=O.DRIFT | O.DISCOUNT, payoffs=O.EUROPEAN)
    ref = bs_call(100.0, K, 1.0, 0.2, r=0.05)
    assert np.all(np.abs(out["prices"] - ref) < 4 * out["std_errs"]), (out["prices"], ref)


CASES = [(1.0, 252, 253), (1.0, 2048, 2048), (1.0, 1000, 1000), (0.1, 5, 5), (0.25, 13, 14), (0.5, 26, 27),
         (1.0, 52, 52), (2.0, 104, 105), (3.0, 156, 157), (4.0, 208, 209), (5.0, 260, 261)]


@pytest.mark.parametrize("T,N,nstar", CASES)
def test_time_grid_case_table(T, N, nstar):
    k, fs, fw = O.time_grid([T], [1], N)
    assert k == nstar and int(fs[0]) == nstar
    if nstar == N:  # case A: the N-th step lands on T; the interpolation weight is ~1
        assert abs(fw[0] - 1.0) < 1e-9
    else:           # case B: one more step; weight ~0
        assert 0.0 <= fw[0] < 1e-9


def test_time_grid_matches_product_host_builder():
    import hestonexotics_amd as H
    rng = np.random.default_rng(5)
    for _ in range(200):
        n = int(rng.integers(1, 6))
        T = np.sort(rng.uniform(0.05, 5.0, n))
        if np.any(np.diff(T) <= 0):
            continue
        ns = rng.integers(0, 4, n)
        if ns.sum() == 0:
            ns[-1] = 1
        N = int(rng.integers(1, 300))
        a = O.time_grid(T, ns, N)
        b = H.time_grid(T, ns, N)
        assert a[0] == b[0]
        np.testing.assert_array_equal(a[1], b[1])
        np.testing.assert_array_equal(a[2], b[2])


@pytest.mark.parametrize("T,N,case_a", [(0.1, 5, True), (0.25, 13, False), (1.0, 52, True), (0.5, 26, False)])
def test_asian_k0_invariant(T, N, case_a):
    """With K = 0 the Asian payoff is the average itself. Under the GBM limit E[X_t] = S0, so the
    reference's average has mean S0 (N-1)/N in case A (its last trapezoid is replaced by the
    price increment X_N - X_{N-1}) and S0 in case B (a proper trapezoid over [0, T])."""
    params = [0.04, 0.04, -0.7, 2.0, 1e-5]
    out = O.price(params, 100.0, [T], [1], [0.0], steps=N, n_paths=200_000, seed=9, payoffs=O.ASIAN)
    expect = 100.0 * (N - 1) / N if case_a else 100.0
    assert abs(out["prices"][0] - expect) < 5 * out["std_errs"][0], (out["prices"][0], expect)
    # the corrected-trapezoid extension removes the case A bias
    out = O.price(params, 100.0, [T], [1], [0.0], steps=N, n_paths=200_000, seed=9, payoffs=O.ASIAN,
                  flags=O.TRAPEZOID)
    assert abs(out["prices"][0] - 100.0) < 5 * out["std_errs"][0]


def test_estimator_matches_per_path_payoffs():
    K = np.array([90.0, 100.0, 110.0, 95.0])
    out = O.price(BASE, 100.0, [0.5, 1.0], [3, 1], K, steps=20, n_paths=5000, seed=4, want_finals=True,
                  r=0.03, flags=O.DISCOUNT)
    f = out["finals"]
    chain = [0, 0, 0, 1]
    asian = np.stack([np.maximum(f[:, c, 0] - k, 0) for c, k in zip(chain, K)])
    euro = np.stack([np.maximum(f[:, c, 1] - k, 0) for c, k in zip(chain, K)])
    pay = np.concatenate([asian, euro])
    disc = np.exp(-0.03 * np.array([0.5, 0.5, 0.5, 1.0] * 2))
    np.testing.assert_allclose(out["prices"], disc * pay.mean(axis=1), rtol=1e-12)
    np.testing.assert_allclose(out["std_errs"], disc * pay.std(axis=1, ddof=1) / np.sqrt(5000), rtol=1e-9)


def test_european_mc_agrees_with_closed_form():
    """The QE scheme (no martingale correction) at 52 steps/yr vs the closed-form Heston price:
    agreement within 4 standard errors plus a stated 0.5% discretisation allowance."""
    g = json.load(open(os.path.join(GOLD, "heston_closed_form.json")))
    case = [c for c in g["cases"] if c["S"] == 100.0 and c["T"] == 1.0][0]
    K = np.array(case["K"])
    params = [case["v0"], case["theta"], case["rho"], case["kappa"], case["sigma"]]
    out = O.price(params, 100.0, [1.0], [len(K)], K, steps=52, n_paths=300_000, seed=77, r=case["r"],
                  flags=O.DRIFT | O.DISCOUNT, payoffs=O.EUROPEAN)
    ref = np.array(case["price"])
    tol = 4 * out["std_errs"] + 0.005 * ref
    assert np.all(np.abs(out["prices"] - ref) < tol), (out["prices"], ref, out["std_errs"])


def test_results_independent_of_thread_count():
    a = O.price(BASE, 100.0, [1.0], [2], [95.0, 105.0], steps=30, n_paths=20_000, seed=1, n_threads=1)
    b = O.price(BASE, 100.0, [1.0], [2], [95.0, 105.0], steps=30, n_paths=20_000, seed=1, n_threads=4)
    np.testing.assert_array_equal(a["prices"], b["prices"])


def test_path_offset_selects_the_same_paths():
    full = O.price(BASE, 100.0, [1.0], [1], [100.0], steps=12, n_paths=300, seed=8, want_finals=True)["finals"]
    part = O.price(BASE, 100.0, [1.0], [1], [100.0], steps=12, n_paths=100, seed=8, path_offset=150,
                   want_finals=True)["finals"]
    np.testing.assert_array_equal(full[150:250], part)


def test_fast_oracle_leaves_subnormals_to_the_strict_one():
    """The timed build, compiled with -ffast-math, must not switch the process to flush-to-zero: at
    S0 = 1e-305 the average's last interval (X - Xp)(T - tp) is subnormal, and the strict oracle's finals
    are 1e-305 times those at S0 = 1 (to 1e-9: ln X = -702 carries 1e-13 a step; flushed, they are off
    by 8%)."""
    kw = dict(steps=9, n_paths=130, seed=13, want_finals=True)
    args = ([0.5], [1])
    O.price(BASE, 1.0, *args, [1.0], steps=2, n_paths=64, seed=1, kind="fast")
    one = O.price(BASE, 1.0, *args, [1.0], **kw)["finals"]
    tiny = O.price(BASE, 1e-305, *args, [1e-305], **kw)["finals"]
    np.testing.assert_allclose(tiny / 1e-305, one, rtol=1e-9)
