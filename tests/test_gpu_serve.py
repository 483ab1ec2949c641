"""The registration pipeline (tiplhip_register: linear, then resample + cdm)
and the serving loop (tiplhip_server_*).

* the plain path recovers the ground-truth affine of seeded pairs;
* every served result equals the plain path's result for the same request,
  bit for bit (affine, matrix, cost, evaluation count, CDM iterations and
  field), whatever the mix and order it was served in -- batched costs are
  exact and the optimiser is deterministic;
* admission keeps the estimated device memory under the budget, rejects a
  request larger than the budget, and one failing request does not disturb
  the others."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _transform_error(T, truth, fixed_shape, moving_shape):
    """Voxel distance, over a grid of fixed points x, between x and M(T(x)):
    T is the found fixed->moving map; M (moving(q) = fixed(M q)) the truth's
    moving->fixed map, so T should be its inverse."""
    from tipl_amd import phantoms
    m = np.asarray(T, np.float64).reshape(-1)
    R, sh = m[:9].reshape(3, 3), m[9:12]
    mt, sht = phantoms.affine_matrix_np(truth, moving_shape, fixed_shape)
    zz, yy, xx = np.meshgrid(*[np.arange(0, n, 3.0) for n in fixed_shape], indexing="ij")
    pts = np.stack([xx, yy, zz], 0).reshape(3, -1)
    back = mt @ (R @ pts + sh[:, None]) + sht[:, None]
    d = np.linalg.norm(back - pts, axis=0)
    return float(d.mean()), float(d.max())


@pytest.fixture(scope="module")
def mix():
    """Eight requests of uneven sizes, dtypes and kinds (3 with CDM)."""
    from tipl_amd import phantoms
    specs = [((48, 56, 48), False, np.float32, "mi"), ((40, 40, 40), True, np.int16, "mi"),
             ((56, 48, 52), False, np.int16, "corr"), ((64, 64, 64), False, np.float32, "mi"),
             ((44, 52, 40), True, np.float32, "mi"), ((36, 44, 36), False, np.float32, "corr"),
             ((52, 52, 52), True, np.int16, "mi"), ((60, 50, 44), False, np.float32, "mi")]
    out = []
    for i, (shape, nl, dt, cost) in enumerate(specs):
        f, m, truth = phantoms.serving_pair(4000 + i, shape, nl, dt)
        out.append({"fixed": f, "moving": m, "truth": truth, "nonlinear": nl, "cost": cost})
    return out


def _same(a, b):
    assert a["status"] == b["status"] == 0
    assert np.array_equal(a["affine"].view(np.uint32), b["affine"].view(np.uint32))
    assert np.array_equal(a["T"].view(np.uint32), b["T"].view(np.uint32))
    assert a["cost"] == b["cost"] and a["evaluations"] == b["evaluations"]
    assert a["cdm_iterations"] == b["cdm_iterations"]
    assert a["r_linear"] == b["r_linear"] and a["r_nonlinear"] == b["r_nonlinear"]
    for k in ("field", "f2t", "to2from", "from2to", "warped"):
        if a.get(k) is not None or b.get(k) is not None:
            x, y = np.asarray(a[k]), np.asarray(b[k])
            if x.dtype == np.float32:
                x, y = x.view(np.uint32), y.view(np.uint32)
            assert np.array_equal(x, y), k


@pytest.fixture(scope="module")
def plain(ctx, mix):
    import tipl_amd
    out = []
    for i, r in enumerate(mix):
        print(f"plain request {i} shape={r['fixed'].shape} nonlinear={r['nonlinear']}", flush=True)
        out.append(tipl_amd.register(ctx, r["fixed"], r["moving"], cost=r["cost"],
                                     nonlinear=r["nonlinear"]))
    return out


@pytest.mark.parametrize("dtype", [np.float32, np.int16])
def test_plain_path_recovers_truth(ctx, dtype):
    """MI on config-0 blob pairs recovers the ground-truth affine (the nested-
    ellipsoid tissue phantom is close to rotation-symmetric, so only blob
    pairs pin it).  The compiled reference lands 0.13 / 0.18 voxel (mean) off
    on seeds 0 / 1."""
    import tipl_amd
    from tipl_amd import phantoms
    for seed in (0, 1):
        fixed, moving, truth = phantoms.blob_pair(seed, (64, 72, 60))
        f, m = fixed.astype(dtype), moving.astype(dtype)
        res = tipl_amd.register(ctx, f, m, cost="mi")
        mean, mx = _transform_error(res["T"], truth, f.shape, m.shape)
        print(f"blob seed={seed} dtype={np.dtype(dtype).name}: error mean {mean:.3f} "
              f"max {mx:.3f} voxel, {res['evaluations']} evaluations, {res['run_ms']:.1f} ms")
        assert mean < 0.5 and mx < 1.5


def test_plain_path_correlation_optimum(ctx, oracle):
    """Correlation with zero fill prefers a smaller overlap: on these pairs the
    compiled reference's own registration ends 3.6-4.9 voxels from the truth
    with scales near 0.84.  The bar is therefore the cost: the optimum found
    is no worse than the cost at the true transform."""
    import tipl_amd
    from tipl_amd import phantoms
    for seed in (0, 1):
        fixed, moving, truth = phantoms.blob_pair(seed, (64, 72, 60))
        f, m = fixed.astype(np.int16), moving.astype(np.int16)
        res = tipl_amd.register(ctx, f, m, cost="corr")
        M, sh = phantoms.affine_matrix_np(truth, m.shape, f.shape)
        Minv = np.linalg.inv(M)
        T_truth = np.concatenate([Minv.reshape(-1), -Minv @ sh]).astype(np.float32)
        f8 = phantoms.quantize(f.astype(np.float32))
        m8 = phantoms.quantize(m.astype(np.float32))
        found = oracle.corr_cost(f8, m8, res["T"])
        at_truth = oracle.corr_cost(f8, m8, T_truth)
        print(f"blob seed={seed}: corr cost {found:.6f} at the optimum, {at_truth:.6f} at the truth")
        assert found <= at_truth + 1e-6


def test_plain_path_nonlinear(mix, plain):
    for r, res in zip(mix, plain):
        print(f"shape={r['fixed'].shape} cost={r['cost']} nonlinear={r['nonlinear']}: "
              f"{res['evaluations']} evaluations, {res['cdm_iterations']} CDM iterations, "
              f"{res['run_ms']:.1f} ms")
        if r["nonlinear"]:
            # cdm() keeps its best field by cost: on a pair the affine step
            # already aligns well (r ~ 0.98) that can be the zero field, as
            # the oracle's cdm() gives for request 4 with the reference's
            # own linear() result
            assert res["cdm_iterations"] > 0
            assert np.isfinite(res["field"]).all()
            assert res["r_nonlinear"] >= res["r_linear"] - 0.01


@pytest.mark.parametrize("slots,order", [(4, "forward"), (8, "reverse")])
def test_served_equals_plain(mix, plain, slots, order):
    import tipl_amd
    idx = list(range(len(mix)))
    if order == "reverse":
        idx = idx[::-1]
    with tipl_amd.Server(0, slots=slots, hbm_budget=16 << 30) as srv:
        tickets = {i: srv.submit(mix[i]["fixed"], mix[i]["moving"], cost=mix[i]["cost"],
                                 nonlinear=mix[i]["nonlinear"]) for i in idx}
        got = {i: srv.wait(t) for i, t in tickets.items()}
        st = srv.stats()
    print(f"slots={slots}: {st}")
    for i in idx:
        _same(got[i], plain[i])
    assert st["completed"] == len(mix) and st["failed"] == 0
    assert st["batched_pairs"] > st["batch_launches"]  # candidate sets were merged
    assert st["latency_p50_ms"] <= st["latency_p95_ms"] <= st["latency_p99_ms"]


def test_admission_budget(mix, plain):
    import tipl_amd
    sizes = [tipl_amd.request_bytes(r["fixed"], r["moving"], nonlinear=r["nonlinear"]) for r in mix]
    budget = int(max(sizes) * 1.2)  # room for about one request at a time
    with tipl_amd.Server(0, slots=4, hbm_budget=budget) as srv:
        tickets = [srv.submit(r["fixed"], r["moving"], cost=r["cost"], nonlinear=r["nonlinear"])
                   for r in mix]
        got = [srv.wait(t) for t in tickets]
        st = srv.stats()
        assert st["hbm_peak"] <= budget
        big = np.zeros((128, 128, 128), np.float32)
        with pytest.raises(tipl_amd.TiplHipError):
            srv.submit(big, big, nonlinear=True)
    for a, b in zip(got, plain):
        _same(a, b)


def test_failure_is_isolated(mix, plain):
    """A nonlinear request on empty images fails in cdm (zero cost, as the
    reference returns false); the requests around it are unaffected."""
    import tipl_amd
    empty = np.zeros((32, 32, 32), np.float32)
    with tipl_amd.Server(0, slots=3, hbm_budget=16 << 30) as srv:
        t0 = srv.submit(mix[0]["fixed"], mix[0]["moving"], cost=mix[0]["cost"])
        tb = srv.submit(empty, empty, nonlinear=True)
        t1 = srv.submit(mix[1]["fixed"], mix[1]["moving"], cost=mix[1]["cost"], nonlinear=True)
        _same(srv.wait(t0), plain[0])
        with pytest.raises(tipl_amd.TiplHipError) as e:
            srv.wait(tb)
        assert e.value.code == tipl_amd.ERR_FAILED
        _same(srv.wait(t1), plain[1])
        st = srv.stats()
    assert st["failed"] == 1 and st["completed"] == 2


def test_mm_reg_preprocessing_served_equals_plain(ctx):
    """Requests with mm_reg's preprocessing (template_image_pre on fixed,
    subject_image_pre on moving, on the device): served == plain, and the
    subject preprocessing matches the oracle."""
    import tipl_amd
    from tipl_amd import phantoms
    reqs = [phantoms.serving_pair(4100 + i, s, nl, dt) for i, (s, nl, dt) in
            enumerate([((48, 52, 44), False, np.int16), ((40, 44, 40), True, np.float32),
                       ((56, 48, 48), False, np.float32)])]
    plain = [tipl_amd.register(ctx, f, m, nonlinear=(i == 1), preprocess="mm_reg")
             for i, (f, m, _) in enumerate(reqs)]
    with tipl_amd.Server(0, slots=3, hbm_budget=8 << 30) as srv:
        ts = [srv.submit(f, m, nonlinear=(i == 1), preprocess="mm_reg") for i, (f, m, _) in enumerate(reqs)]
        got = [srv.wait(t) for t in ts]
    for a, b in zip(got, plain):
        _same(a, b)


def test_bidirectional_served_equals_plain(ctx, mix):
    """mm_reg's full nonlinear half (reverse CDM on each slot's second stream,
    both mappings, the warped image and the r values): served == plain."""
    import tipl_amd
    outs = ("f2t", "to2from", "from2to", "warped")
    sel = [i for i, r in enumerate(mix) if r["nonlinear"]] + [0]
    kw = lambda i: dict(cost=mix[i]["cost"], nonlinear=mix[i]["nonlinear"],
                        reverse=mix[i]["nonlinear"],
                        outputs=outs if mix[i]["nonlinear"] else ("warped",))
    plain = [tipl_amd.register(ctx, mix[i]["fixed"], mix[i]["moving"], **kw(i)) for i in sel]
    for i, p in zip(sel, plain):
        if mix[i]["nonlinear"]:
            assert p["r_nonlinear"] >= p["r_linear"] - 0.01 and p["r_linear"] > 0.5
            assert np.isfinite(p["f2t"]).all() and np.isfinite(p["from2to"]).all()
    with tipl_amd.Server(0, slots=4, hbm_budget=16 << 30) as srv:
        ts = [srv.submit(mix[i]["fixed"], mix[i]["moving"], **kw(i)) for i in sel]
        got = [srv.wait(t) for t in ts]
    for a, b in zip(got, plain):
        _same(a, b)


@pytest.fixture(scope="module")
def cdm_mix():
    """Six nonlinear pairs of different shapes, for the batched CDM tests."""
    from tipl_amd import phantoms
    shapes = [(40, 48, 40), (64, 64, 64), (56, 44, 60), (72, 80, 64), (48, 48, 48), (96, 80, 72)]
    return [phantoms.serving_pair(4300 + i, s, True, np.float32)[:2] for i, s in enumerate(shapes)]


def test_cdm_batched_across_registrations(ctx, cdm_mix):
    """Six nonlinear registrations, both CDM directions, served together on
    six slots: the server's cdm() iterations go out as batched steps (more
    fields than steps, several fields per launch) and every result -- fields
    of both directions, mappings, iteration counts and r values -- equals
    the plain path's bit for bit."""
    import tipl_amd
    outs = ("f2t", "to2from", "from2to", "warped")
    kw = dict(nonlinear=True, reverse=True, outputs=outs)
    plain = []
    for f, m in cdm_mix:
        print(f"plain bidirectional {f.shape}", flush=True)
        plain.append(tipl_amd.register(ctx, f, m, **kw))
    with tipl_amd.Server(0, slots=6, hbm_budget=16 << 30) as srv:
        ts = [srv.submit(f, m, **kw) for f, m in cdm_mix]
        got = [srv.wait(t) for t in ts]
        st = srv.stats()
    print(f"batched CDM: {st['cdm_fields']} fields in {st['cdm_steps']} steps", flush=True)
    for a, b in zip(got, plain):
        _same(a, b)
    iters = sum(p["cdm_iterations"] for p in plain)
    assert st["cdm_steps"] > 0
    assert st["cdm_fields"] >= iters          # the forward ones at least
    assert st["cdm_fields"] >= 1.3 * st["cdm_steps"]


def test_cdm_batching_off(ctx, cdm_mix, monkeypatch):
    """TIPLHIP_SERVER_CDM_BATCH=0 at server creation: each registration runs
    its cdm() alone on its stream (no batched steps), same results."""
    import tipl_amd
    monkeypatch.setenv("TIPLHIP_SERVER_CDM_BATCH", "0")
    sel = cdm_mix[:3]
    plain = [tipl_amd.register(ctx, f, m, nonlinear=True) for f, m in sel]
    with tipl_amd.Server(0, slots=3, hbm_budget=16 << 30) as srv:
        ts = [srv.submit(f, m, nonlinear=True) for f, m in sel]
        got = [srv.wait(t) for t in ts]
        st = srv.stats()
    assert st["cdm_steps"] == 0 and st["cdm_fields"] == 0
    for a, b in zip(got, plain):
        _same(a, b)


def test_cdm_batching_mixed_levels_and_fallbacks(ctx, cdm_mix, monkeypatch):
    """Only levels up to 20000 voxels batched (TIPLHIP_CDM_BATCH_VOXELS), on
    two lanes: each registration runs its coarse levels as batched steps and
    its finer levels alone; a request with the 'd' gradient runs unbatched
    throughout.  Every result equals the plain path's bit for bit."""
    import tipl_amd
    monkeypatch.setenv("TIPLHIP_CDM_BATCH_VOXELS", "20000")
    monkeypatch.setenv("TIPLHIP_CDM_LANES", "2")
    reqs = [(f, m, {}) for f, m in cdm_mix[:4]] + [(cdm_mix[4][0], cdm_mix[4][1], {"gradient_type": "d"})]
    plain = [tipl_amd.register(ctx, f, m, nonlinear=True, **kw) for f, m, kw in reqs]
    with tipl_amd.Server(0, slots=5, hbm_budget=16 << 30) as srv:
        ts = [srv.submit(f, m, nonlinear=True, **kw) for f, m, kw in reqs]
        got = [srv.wait(t) for t in ts]
        st = srv.stats()
    print(f"batched CDM: {st['cdm_fields']} fields in {st['cdm_steps']} steps", flush=True)
    for a, b in zip(got, plain):
        _same(a, b)
    iters = sum(p["cdm_iterations"] for p in plain)
    assert 0 < st["cdm_fields"] < iters


def test_cdm_batching_one_lane_full_batches(ctx, cdm_mix, monkeypatch):
    """One lane (TIPLHIP_CDM_LANES=1): four bidirectional registrations put up
    to eight fields -- the most a step launch takes -- into each batched step;
    results equal the plain path's bit for bit."""
    import tipl_amd
    monkeypatch.setenv("TIPLHIP_CDM_LANES", "1")
    outs = ("f2t", "to2from", "from2to", "warped")
    kw = dict(nonlinear=True, reverse=True, outputs=outs)
    sel = [cdm_mix[0], cdm_mix[2], cdm_mix[4], cdm_mix[1]]
    plain = [tipl_amd.register(ctx, f, m, **kw) for f, m in sel]
    with tipl_amd.Server(0, slots=4, hbm_budget=16 << 30) as srv:
        ts = [srv.submit(f, m, **kw) for f, m in sel]
        got = [srv.wait(t) for t in ts]
        st = srv.stats()
    print(f"batched CDM: {st['cdm_fields']} fields in {st['cdm_steps']} steps", flush=True)
    for a, b in zip(got, plain):
        _same(a, b)
    assert st["cdm_fields"] >= 3 * st["cdm_steps"]


def test_cdm_batching_of_every_level(ctx, cdm_mix, monkeypatch):
    """Levels of up to 2^25 voxels batched (TIPLHIP_CDM_BATCH_VOXELS): the finest
    ones, of 262144 to 552960 voxels, take the large tiles of the gradient and of
    the field update, beside fields on the small tiles in the same step, both
    directions at a time.  Every iteration goes out as a batched step, and every
    result equals the plain path's bit for bit."""
    import tipl_amd
    monkeypatch.setenv("TIPLHIP_CDM_BATCH_VOXELS", str(1 << 25))
    monkeypatch.setenv("TIPLHIP_CDM_LANES", "2")
    sel = [cdm_mix[i] for i in (5, 1, 0, 3)]
    kw = dict(nonlinear=True, reverse=True, outputs=("f2t", "to2from", "from2to", "warped"))
    plain = [tipl_amd.register(ctx, f, m, **kw) for f, m in sel]
    with tipl_amd.Server(0, slots=4, hbm_budget=16 << 30) as srv:
        ts = [srv.submit(f, m, **kw) for f, m in sel]
        got = [srv.wait(t) for t in ts]
        st = srv.stats()
    for a, b in zip(got, plain):
        _same(a, b)
    iters = sum(p["cdm_iterations"] for p in plain)
    print(f"batched CDM: {st['cdm_fields']} fields in {st['cdm_steps']} steps, {iters} forward iterations")
    assert st["cdm_fields"] > iters  # the forward ones, and the reverse ones of the other direction
    assert st["cdm_fields"] > st["cdm_steps"]
