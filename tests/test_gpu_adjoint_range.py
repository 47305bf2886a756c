"""The reverse pass is linear in its seed: seeds scaled by a power of two give
gradients scaled by it, in all its forms, as long as the gradients themselves
are far from the ends of the float range.  The pairs' terms, which carry
factors of up to 10^16 (the kernels' normalisations at a support of 0.0056),
have to stay as far from them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORMS = (None, dict(), dict(force_staged=1, density_staged=1))


@pytest.mark.parametrize("h", [0.02, 0.0056])
@pytest.mark.parametrize("exponent", [-60, 50, 80])
def test_gradients_scale_with_their_seed(h, exponent):
    """Seeds of 1e-5 scaled by 2^-60, 2^50 and 2^80.  The adjoint of the acceleration
    is dt^2 = 1e-8 of the seed at first, 1e-31 at the small end, seven decades
    inside the range; gradients by position-like seeds are larger.  Scaled
    exactly, the results are equal bit for bit; 1e-6 of the largest allows for
    single terms that cancel below the range's end."""
    from simplefluid_amd import engine as E
    r = h / 4
    rng = np.random.default_rng(4)
    g = np.stack(np.meshgrid(*[np.arange(11)] * 3, indexing="ij"), -1).reshape(-1, 3) * (1.9 * r) + r
    x = (g + rng.uniform(-0.3 * r, 0.3 * r, g.shape)).astype(np.float32)
    v = rng.normal(0.0, 0.2, x.shape).astype(np.float32)
    seed = rng.normal(0.0, 1e-5, x.shape).astype(np.float32)
    p = E.make_params(kernel_radius=h, particle_radius=r, box_max=(40 * r,) * 3, dt=1e-4)
    for form in FORMS:
        e = E.Engine(p)
        e.set_particles(x, v)
        e.make_ready()
        if form is not None:
            e.set_tuning(**form)
        e.rollout_forward(6, 3)
        ref = e.rollout_backward(seed)
        got = e.rollout_backward(np.ldexp(seed, exponent))
        e.close()
        for name, a, b in zip(("dB", "dmu", "dv0"), ref, got):
            a64, b64 = a.astype(np.float64), np.ldexp(b.astype(np.float64), -exponent)
            err = np.abs(a64 - b64).max() / np.abs(a64).max()
            print(f"h {h} 2^{exponent} {form} {name}: largest {np.abs(a).max():.2e}, scaled {np.abs(b).max():.2e}, "
                  f"error {err:.1e}", flush=True)
            assert err <= 1e-6, name
