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


JUNK = {"ok": 0xFF, "stop": 0xFF, "used": -7}
ALL = [W.HMS_C0, W.SHMS_C1, W.SOS_1p5, W.HRSR_2, W.HRSL_3]
E_ARG = -6  # SIMC_E_ARG


def dirty(n):
    """Host columns holding what no run writes."""
    from simc_gfortran_amd import api
    kinds = {"ok": np.uint8, "stop": np.uint8, "used": np.int32}
    return {k: np.full(n, JUNK.get(k, np.nan), kinds.get(k, np.float64)) for k in api.OUT_FIELDS}


def structs(api, ev, out, ptr):
    return (api.EventsIn(*[ptr(ev.get(k)) for k in ("dpp", "x", "y", "z", "dxdz", "dydz", "fry")]),
            api.EventsOut(*[ptr(out.get(k)) for k in api.OUT_FIELDS]))


@pytest.mark.parametrize("rng", ["philox", "tape"])
@pytest.mark.parametrize("wl", ALL, ids=lambda w: w.name)
def test_every_column_of_dirty_outputs_is_written(ctx, wl, rng):
    """The C entries on outputs full of junk give what the cleared form gives;
    the tape is too short for the hut, so events end at it as well."""
    import ctypes as C
    from simc_gfortran_amd import api
    L, n, dev, stride = api.library(), 5003, torch.device("cuda"), 120
    ev = W.generate_device(wl, n, seed=6, device=dev)
    host = {k: v.cpu().numpy() for k, v in ev.items()}
    kw = dict(p_spec=wl.p_spec, m2=wl.m2, wire_sigma=wl.wire_sigma, fit="fp64")
    S = api.Settings(wl.p_spec, wl.m2, 0.0, 1, 1, 0, 0, api.FIT_FP64, 0, wl.wire_sigma)
    if rng == "tape":
        tape = W.uniform_tape(n, stride, seed=3)
        d_tape = torch.from_numpy(tape).to(dev)
        old = ctx.run(wl.arm, ev, out=cleared(ev, n, dev), rng="tape", tape=d_tape, stride=stride, **kw)
        R = api.Rng(api.RNG_TAPE, 0, 0, 0, d_tape.data_ptr(), stride)
        RH = api.Rng(api.RNG_TAPE, 0, 0, 0, tape.ctypes.data, stride)
    else:
        old = ctx.run(wl.arm, ev, out=cleared(ev, n, dev), seed=9, **kw)
        R = RH = api.Rng(api.RNG_PHILOX, 0, 9, 0, None, 0)
    old = {k: v.cpu().numpy() for k, v in old.items()}
    assert (old["stop"] == 250).any() == (rng == "tape")  # past the end of its tape

    new = {k: torch.from_numpy(v).to(dev) for k, v in dirty(n).items()}
    ein, eout = structs(api, ev, new, lambda t: None if t is None else t.data_ptr())
    st = torch.cuda.current_stream().cuda_stream
    assert L.simc_arm_run_fresh(ctx._h, wl.arm, C.byref(S), C.byref(ein), C.byref(eout), n, C.byref(R), C.c_void_p(st)) == 0
    torch.cuda.synchronize()
    got = dirty(n)
    hin, hout = structs(api, host, got, lambda a: None if a is None else a.ctypes.data)
    assert L.simc_arm_run_host_fresh(ctx._h, wl.arm, C.byref(S), C.byref(hin), C.byref(hout), n, C.byref(RH)) == 0
    for k in old:
        np.testing.assert_array_equal(new[k].cpu().numpy(), old[k], err_msg=k)
        np.testing.assert_array_equal(got[k], old[k], err_msg="host " + k)


def test_every_column_of_a_batch_is_written(ctx):
    import ctypes as C
    from simc_gfortran_amd import api
    dev, n = torch.device("cuda"), 9001
    ev = {k: torch.empty(n, dtype=torch.float64, device=dev) for k in ("dpp", "x", "y", "z", "dxdz", "dydz", "fry")}
    at, table = 0, []
    for i, wl in enumerate(ALL):
        m = 2003 if i < 4 else n - at
        W.generate_device(wl, m, seed=i, device=dev, out=ev, at=at)
        table.append(dict(arm=wl.arm, p_spec=wl.p_spec, m2=wl.m2, wire_sigma=wl.wire_sigma, fit="fp64", seed=i,
                          offset=at, count=m))
        at += m
    b = api.Batch(ctx, table)
    old = b.run(ev, out=b.new_outputs(ev))
    new = {k: torch.from_numpy(v).to(dev) for k, v in dirty(n).items() if k in old}
    ein, eout = structs(api, ev, new, lambda t: None if t is None else t.data_ptr())
    st = torch.cuda.current_stream().cuda_stream
    assert api.library().simc_batch_run_fresh(b._h, C.byref(ein), C.byref(eout), C.c_void_p(st)) == 0
    torch.cuda.synchronize()
    for k in old:
        np.testing.assert_array_equal(new[k].cpu().numpy(), old[k].cpu().numpy(), err_msg=k)


def test_the_sieve_is_refused(ctx):
    """Its forced angles are INOUT; the outputs stay as they are."""
    import ctypes as C
    from simc_gfortran_amd import api
    L, wl, n, dev = api.library(), W.HMS_C0, 300, torch.device("cuda")
    ev = W.generate_device(wl, n, seed=6, device=dev)
    host = {k: v.cpu().numpy() for k, v in ev.items()}
    S = api.Settings(wl.p_spec, wl.m2, 0.0, 1, 1, 0, 0, api.FIT_FP64, 1, wl.wire_sigma)
    R = api.Rng(api.RNG_PHILOX, 0, 9, 0, None, 0)
    new, got = {k: torch.from_numpy(v).to(dev) for k, v in dirty(n).items()}, dirty(n)
    ein, eout = structs(api, ev, new, lambda t: None if t is None else t.data_ptr())
    hin, hout = structs(api, host, got, lambda a: None if a is None else a.ctypes.data)
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    b = api.Batch(ctx, [dict(arm=wl.arm, p_spec=wl.p_spec, m2=wl.m2, sieve=1, seed=1, offset=0, count=n)])
    assert L.simc_arm_run_fresh(ctx._h, wl.arm, C.byref(S), C.byref(ein), C.byref(eout), n, C.byref(R), st) == E_ARG
    assert L.simc_arm_run_host_fresh(ctx._h, wl.arm, C.byref(S), C.byref(hin), C.byref(hout), n, C.byref(R)) == E_ARG
    assert L.simc_batch_run_fresh(b._h, C.byref(ein), C.byref(eout), st) == E_ARG
    torch.cuda.synchronize()
    for k, v in dirty(n).items():
        np.testing.assert_array_equal(new[k].cpu().numpy(), v, err_msg=k)
        np.testing.assert_array_equal(got[k], v, err_msg=k)
