"""Outputs made by the entry (written whole by the kernels) equal the same
run into cleared outputs (INOUT), where events stop at every stage."""
import numpy as np
import pytest

from simc_gfortran_amd import workloads as W

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
COLS = ("x_fp", "dx_fp", "y_fp", "dy_fp", "pathlen", "resmult", "m2")


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from simc_gfortran_amd import api
    c = api.Spectrometers()
    yield c
    c.close()


def cleared(ev, n, dev):
    out = {k: ev[k].clone() for k in ("dpp", "y", "dxdz", "dydz")}
    out.update({k: torch.zeros(n, dtype=torch.float64, device=dev) for k in COLS})
    out.update(ok=torch.zeros(n, dtype=torch.uint8, device=dev), stop=torch.zeros(n, dtype=torch.uint8, device=dev),
               used=torch.zeros(n, dtype=torch.int32, device=dev))
    return out


@pytest.mark.parametrize("pion", [False, True])
@pytest.mark.parametrize("n", [1, 257, 20_011])
@pytest.mark.parametrize("wl", [W.HMS_C0, W.SHMS_C1, W.SOS_1p5, W.HRSR_2], ids=lambda w: w.name)
def test_new_outputs_equal_cleared_ones(ctx, wl, n, pion):
    dev = torch.device("cuda")
    ev = W.generate_device(wl, n, seed=2, device=dev)
    kw = dict(p_spec=wl.p_spec, m2=W.MPI ** 2 if pion else wl.m2, wire_sigma=wl.wire_sigma, seed=9)
    if pion:
        kw.update(decay=True, ctau=780.4, coll=wl.arm in (1, 5))
    # what an allocation of this size held before must not show
    junk = [torch.full((n,), float("nan"), dtype=torch.float64, device=dev) for _ in range(16)]
    del junk
    new = ctx.run(wl.arm, ev, **kw)
    old = ctx.run(wl.arm, ev, out=cleared(ev, n, dev), **kw)
    torch.cuda.synchronize()
    assert set(new) == set(old)
    for k in old:
        np.testing.assert_array_equal(new[k].cpu().numpy(), old[k].cpu().numpy(), err_msg=k)
    host = {k: v.cpu().numpy() for k, v in ev.items()}
    got = ctx.run_host(wl.arm, host, **kw)
    for k in old:
        np.testing.assert_array_equal(got[k], old[k].cpu().numpy(), err_msg="host " + k)


def test_batch_with_a_gap_keeps_the_cleared_form(ctx):
    """Elements outside every setting's range are the inputs and zeros."""
    from simc_gfortran_amd import api
    wl, n = W.HMS_C0, 3000
    ev = W.generate_device(wl, n, seed=4, device=torch.device("cuda"))
    base = dict(arm=wl.arm, p_spec=wl.p_spec, m2=wl.m2, wire_sigma=wl.wire_sigma, fit="fp64")
    b = api.Batch(ctx, [dict(base, seed=1, offset=0, count=1000), dict(base, seed=2, offset=1500, count=1500)])
    out = b.run(ev)
    whole = api.Batch(ctx, [dict(base, seed=1, offset=0, count=1500), dict(base, seed=2, offset=1500, count=1500)])
    full = whole.run(ev)
    torch.cuda.synchronize()
    for k in out:
        gap = out[k][1000:1500].cpu().numpy()
        np.testing.assert_array_equal(gap, ev[k][1000:1500].cpu().numpy() if k in ev else np.zeros_like(gap), err_msg=k)
        for sl in (slice(0, 1000), slice(1500, 3000)):
            np.testing.assert_array_equal(out[k][sl].cpu().numpy(), full[k][sl].cpu().numpy(), err_msg=k)


def test_batch_allocates_only_the_columns_it_returns(ctx):
    """A batch's outputs are what the call takes: 74 bytes an event, and
    nothing else for its duration."""
    from simc_gfortran_amd import api
    wl, n = W.HMS_C0, 2_000_000
    ev = W.generate_device(wl, n, seed=4, device=torch.device("cuda"))
    b = api.Batch(ctx, [dict(arm=wl.arm, p_spec=wl.p_spec, m2=wl.m2, seed=1, offset=0, count=n)])
    b.run(ev)  # the library's own queues
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = b.run(ev)
    torch.cuda.synchronize()
    peak = torch.cuda.max_memory_allocated() - before
    returned = sum(v.numel() * v.element_size() for v in out.values())
    assert returned == 74 * n
    # a block's unsplit remainder is less than 1 MiB: eleven are less than one more column, 16 MB
    assert peak < returned + 8 * n, (peak, returned)


def test_new_outputs_have_the_inputs_shape(ctx):
    """dpp, y, dxdz and dydz come back in the shape of their inputs (as they do
    when they start as copies of them), also a column longer than a batch."""
    from simc_gfortran_amd import api
    wl, n = W.SHMS_C1, 3000
    inout = ("dpp", "y", "dxdz", "dydz")
    flat = W.generate_device(wl, n, seed=4, device=torch.device("cuda"))
    ev = {k: v.view(n // 3, 3) for k, v in flat.items()}
    kw = dict(p_spec=wl.p_spec, m2=wl.m2, seed=1)
    ref = ctx.run(wl.arm, flat, **kw)
    b = api.Batch(ctx, [dict(arm=wl.arm, offset=0, count=n, **kw)])
    host = {k: v.cpu().numpy().reshape(n, 1) for k, v in flat.items()}
    long = dict(flat, y=torch.cat([flat["y"], flat["y"][:5]]))
    for out in (ctx.run(wl.arm, ev, **kw), b.run(ev), ctx.run_host(wl.arm, host, **kw), b.run(long)):
        out = {k: torch.as_tensor(v).cpu() for k, v in out.items()}
        given = long if out["y"].numel() > n else host if out["y"].shape == (n, 1) else ev
        for k in inout:
            assert tuple(out[k].shape) == tuple(given[k].shape), k
        for k in inout + ("x_fp", "pathlen", "ok"):
            np.testing.assert_array_equal(out[k].reshape(-1)[:n].numpy(), ref[k].cpu().numpy(), err_msg=k)
        np.testing.assert_array_equal(out["y"].reshape(-1)[n:].numpy(), flat["y"][:out["y"].numel() - n].cpu().numpy())
