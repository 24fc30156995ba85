"""The detector hut's two forms: compiled steps, and the interpreted ones that
a wavefront takes when one of its events has slopes or a scattering angle that
are no track's."""
import numpy as np
import pytest

from simc_gfortran_amd import workloads as W

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from simc_gfortran_amd import api
    c = api.Spectrometers()
    yield c
    c.close()


ALL = [W.HMS_C0, W.SHMS_C1, W.SOS_1p5, W.HRSR_2, W.HRSL_3]


@pytest.mark.parametrize("wl", ALL, ids=lambda w: w.name)
def test_events_beside_a_track_that_is_not_a_number(ctx, oracle, wl):
    """A NaN slope passes every aperture that tests for being outside (all but
    the HMS dipole's entrance, which tests for being inside and stops it), so
    it reaches the hut and its wavefront interprets the steps: the other
    events' outputs stay bit for bit what they are without it, and its own stop
    code and draws are the oracle's."""
    n = 4099
    ev = W.generate_device(wl, n, seed=3, device=torch.device("cuda"))
    kw = dict(p_spec=wl.p_spec, m2=wl.m2, wire_sigma=wl.wire_sigma, seed=5)
    ref = ctx.run(wl.arm, ev, fit="fp64", **kw)
    odd = np.arange(0, n, 97)
    bad = {k: v.clone() for k, v in ev.items()}
    bad["dxdz"][torch.from_numpy(odd).cuda()] = float("nan")
    out = {k: v.cpu().numpy() for k, v in ctx.run(wl.arm, bad, fit="fp64", **kw).items()}
    keep = np.ones(n, bool)
    keep[odd] = False
    for k, v in ref.items():
        np.testing.assert_array_equal(out[k][keep], v.cpu().numpy()[keep], err_msg=k)
    assert int(ref["ok"].sum()) > n // 10
    cpu = oracle.run(wl.arm, {k: v.cpu().numpy() for k, v in bad.items()}, rng="philox", fit_f32=False, **kw)
    for k in ("stop", "used"):
        np.testing.assert_array_equal(out[k][odd], cpu[k][odd], err_msg=k)
    through = out["used"][odd].max()  # a track through the whole hut takes 176 to 202 uniforms
    assert through == 0 if wl.arm == W.HMS_C0.arm else through > 170


@pytest.mark.parametrize("wl", ALL, ids=lambda w: w.name)
def test_both_forms_of_the_hut_give_the_same_bits(ctx, oracle, wl):
    """At 0.1 keV/c the scattering angles' common factor is past the compiled
    form's limit, so every wavefront interprets the hut.  With the scattering
    off nothing depends on the momentum: the outputs equal those at the
    workload's momentum, which run compiled.  With it on the angles are no
    track's, and the stop codes and draws are the oracle's."""
    n = 4099
    ev = W.generate_device(wl, n, seed=3, device=torch.device("cuda"))
    kw = dict(m2=wl.m2, wire_sigma=wl.wire_sigma, seed=5)
    com = ctx.run(wl.arm, ev, p_spec=wl.p_spec, ms=False, fit="fp64", **kw)
    gen = ctx.run(wl.arm, ev, p_spec=1e-4, ms=False, fit="fp64", **kw)
    assert int(com["ok"].sum()) > n // 10
    for k, v in com.items():
        np.testing.assert_array_equal(gen[k].cpu().numpy(), v.cpu().numpy(), err_msg=k)
    out = ctx.run(wl.arm, ev, p_spec=1e-4, fit="fp64", **kw)
    cpu = oracle.run(wl.arm, {k: v.cpu().numpy() for k, v in ev.items()}, p_spec=1e-4, rng="philox", fit_f32=False, **kw)
    for k in ("stop", "used"):
        np.testing.assert_array_equal(out[k].cpu().numpy(), cpu[k], err_msg=k)
