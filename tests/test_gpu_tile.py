"""The LDS-tiled GEMM form of the grouped matvec (64 x 64 tiles, CT_GEMM_LDS=1) at the edges of its tiles,
k-panels and 16 x 16 sub-tiles, against a dense FP64 contraction."""

import sys

import numpy as np
import pytest

import chemtensor_amd as ct

pytestmark = pytest.mark.gpu


def dense_problem(da, db, d, D, seed, density=1.0):
    """One sector on every axis: stage 1 is a (da d) x (D db) product with K = db, stage 3 da x (d db) with K = da D;
    a share `density` of the operator's entries is not zero."""
    rng = np.random.default_rng(seed)
    z = lambda n: np.zeros(n, dtype=np.int32)
    shapes = [(da, d, db), (D, d, d, D), (1, da, D, da), (db, D, db, 1)]
    dirs = [[1, 1, -1], [1, 1, -1, -1], [1, -1, -1, 1], [1, 1, -1, -1]]
    ts, vs = [], []
    for s, ad in zip(shapes, dirs):
        t = ct.HostTensor.zeros(s, ad, [z(n) for n in s])
        v = rng.standard_normal(s)
        if len(ts) == 1 and density < 1:
            v *= rng.random(s) < density
        t.deserialize(v.reshape(-1))
        ts.append(t)
        vs.append(v)
    th, w, l, r = vs
    t1 = np.tensordot(th, r[..., 0], axes=(2, 0))                       # a p n c
    t2 = np.tensordot(w, t1, axes=([2, 3], [1, 2]))                     # m q a c
    return ts, np.einsum("amx,mqac->xqc", l[0], t2, optimize=True).reshape(-1)


EDGES = [(1, 1, 1, 1), (1, 3, 2, 2), (15, 17, 1, 1), (16, 16, 2, 1), (17, 15, 3, 1), (33, 64, 1, 2), (48, 5, 1, 3),
                                 (63, 65, 2, 1), (64, 32, 1, 1), (65, 33, 2, 2), (130, 129, 1, 2), (3, 200, 4, 5), (200, 3, 4, 5)]


@pytest.mark.parametrize("stage3", ["tasks", "split"])
@pytest.mark.parametrize("da,db,d,D", EDGES)
def test_tile_form_edges(da, db, d, D, stage3, monkeypatch):
    monkeypatch.setenv("CT_GEMM_LDS", "1")
    monkeypatch.setenv("CT_STAGE12", "separate")
    monkeypatch.setenv("CT_STAGE3", stage3)
    ts, want = dense_problem(da, db, d, D, 100 * da + db)
    plan = ct.MatvecPlan(*ts, ct.GROUPED_FP64)
    forms = plan.forms()[0]
    print("case", da, db, d, D, "forms", forms, flush=True)
    sys.stdout.flush()
    assert forms[0] == 6 and forms[2] == (7 if stage3 == "split" else 6)
    x, y = ct.DeviceArray.from_numpy(ts[0].serialize()), ct.DeviceArray(plan.dim)
    plan.apply(x, y)
    plan.synchronize()
    # three chained FP64 products of at most 1000 terms: 2e-16 sqrt(1000) each way
    assert np.linalg.norm(y.numpy() - want) <= 2e-14 * np.linalg.norm(want)


@pytest.mark.parametrize("model,L,chi", [("hubbard", 8, 24), ("xxz", 32, 256), ("hubbard", 32, 256), ("xxz", 32, 1200)])
def test_split_stage3_and_its_lanczos(model, L, chi, monkeypatch):
    """The k range of every y block cut into slots (CT_STAGE3=split) against the tasks: the matvec, and the
    Lanczos recurrence whose step adds the slots and takes alpha from the tiles' partials (at 1200 states several
    reduction items per wavefront)."""
    monkeypatch.setenv("CT_STAGE12", "separate")
    p = ct.generate_matvec_problem(model, L, chi, 11)
    got = {}
    for stage3 in ("tasks", "split"):
        monkeypatch.setenv("CT_STAGE3", stage3)
        plan = ct.MatvecPlan(*p, ct.GROUPED_FP64)
        assert (plan.forms()[0][2] == 7) == (stage3 == "split")
        x, y = ct.DeviceArray.from_numpy(p[0].serialize()), ct.DeviceArray(plan.dim)
        plan.apply(x, y)
        plan.synchronize()
        first = plan.lanczos(x, 12)
        for _ in range(3):                    # the captured recurrence, then its replays
            again = plan.lanczos(x, 12)
            assert first[0] == again[0] and np.array_equal(first[1].numpy(), again[1].numpy())
        monkeypatch.setenv("CT_LANCZOS_GRAPH", "0")
        eager = plan.lanczos(x, 12)
        monkeypatch.delenv("CT_LANCZOS_GRAPH")
        assert eager[0] == first[0] and np.array_equal(eager[1].numpy(), first[1].numpy())
        got[stage3] = (y.numpy(), first[0], first[1].numpy())
    a, b = got["tasks"], got["split"]
    assert np.linalg.norm(a[0] - b[0]) <= 1e-14 * np.linalg.norm(a[0])
    # twelve steps of the recurrence, each carrying rounding of 1e-15 into the next
    assert abs(a[1] - b[1]) <= 1e-12 * abs(a[1])
    assert np.linalg.norm(a[2] - b[2]) <= 1e-10


@pytest.mark.parametrize("model,L,chi", [("hubbard", 8, 24), ("xxz", 20, 64)])
def test_partial_blocks_only_where_used(model, L, chi, monkeypatch):
    """A plan keeps the split's partial blocks (in its intermediate doubles) only where stage 3 runs on them:
    vectors this short do not take them into the Lanczos step."""
    p = ct.generate_matvec_problem(model, L, chi, 11)
    held = {}
    for stage3 in ("tasks", "split", None):
        if stage3:
            monkeypatch.setenv("CT_STAGE3", stage3)
        else:
            monkeypatch.delenv("CT_STAGE3")
        plan = ct.MatvecPlan(*p, ct.GROUPED_FP64)
        held[stage3] = (plan.forms()[0][2], plan.stats()["intermediate_doubles"])
    assert held["split"][0] == 7 and held["split"][1] > held["tasks"][1]
    assert held[None][1] == held["split" if held[None][0] == 7 else "tasks"][1]


def test_tiles_off(monkeypatch):
    """CT_GEMM_LDS=0: no stage on the LDS tiles, neither as tasks nor as slots of a cut k range (a bond that
    takes both without the switch)."""
    p = ct.generate_matvec_problem("xxz", 32, 256, 11)
    monkeypatch.setenv("CT_STAGE12", "separate")
    monkeypatch.setenv("CT_STAGE3", "tasks")
    tasks = ct.MatvecPlan(*p, ct.GROUPED_FP64).stats()["intermediate_doubles"]
    monkeypatch.delenv("CT_STAGE3")
    monkeypatch.setenv("CT_GEMM_LDS", "0")
    plan = ct.MatvecPlan(*p, ct.GROUPED_FP64)
    assert not {6, 7} & set(plan.forms()[0]) and plan.stats()["intermediate_doubles"] == tasks


@pytest.mark.parametrize("which", ["large", "all"])
@pytest.mark.parametrize("model,chi", [("hubbard", 1600), ("xxz", 515)])
def test_tiles_of_large_and_of_all_tasks(model, chi, which, monkeypatch):
    """Bonds with tasks on both sides of the limit: the large ones on the tiles and the others on the wavefront
    forms in a second launch, or all on the tiles, against the wavefront forms alone."""
    p = ct.generate_matvec_problem(model, 32, chi, 11)
    monkeypatch.setenv("CT_STAGE12", "separate")
    monkeypatch.setenv("CT_STAGE3", "tasks")
    x, got = ct.DeviceArray.from_numpy(p[0].serialize()), {}
    for lds in ("0", which):
        monkeypatch.setenv("CT_GEMM_LDS", lds)
        plan = ct.MatvecPlan(*p, ct.GROUPED_FP64)
        forms = plan.forms()[0]
        print("case", model, chi, lds, "forms", forms, flush=True)
        assert (forms[0] == 6 and forms[2] == 6) == (lds != "0")
        y = ct.DeviceArray(plan.dim)
        plan.apply(x, y)
        plan.synchronize()
        got[lds] = y.numpy()
    # the same products, added in an order of their own in some of the wavefront forms
    assert np.linalg.norm(got["0"] - got[which]) <= 1e-14 * np.linalg.norm(got["0"])


@pytest.mark.parametrize("density", [0.0, 0.02, 0.3, 1.0])
@pytest.mark.parametrize("da,db,d,D", [(1, 1, 2, 20), (3, 5, 4, 17), (17, 9, 2, 33), (5, 64, 3, 48), (33, 2, 2, 65), (1, 129, 1, 40)])
def test_row_tiles_of_wide_classes(da, db, d, D, density, monkeypatch):
    """Stage 2 as row tiles that keep the columns in use (CT_STAGE2=rowtiles): rows beyond a multiple of 64,
    columns beyond a multiple of 16, odd column counts, empty and full operators."""
    monkeypatch.setenv("CT_STAGE2", "rowtiles")
    ts, want = dense_problem(da, db, d, D, 7 * da + db, density)
    plan = ct.MatvecPlan(*ts, ct.GROUPED_FP64)
    print("case", da, db, d, D, density, "forms", plan.forms()[0], flush=True)
    assert plan.forms()[0][1] == 8
    assert plan.stage_flops()[1] == 2 * np.count_nonzero(ts[1].serialize()) * da * db
    x, y = ct.DeviceArray.from_numpy(ts[0].serialize()), ct.DeviceArray(plan.dim)
    plan.apply(x, y)
    plan.synchronize()
    assert np.linalg.norm(y.numpy() - want) <= 2e-14 * np.linalg.norm(want)


@pytest.mark.parametrize("da,db,d,D", [(2, 50, 2, 33), (3, 49, 2, 24), (17, 9, 2, 33), (5, 64, 3, 48), (33, 2, 2, 65), (7, 31, 1, 129)])
def test_tiles_of_several_column_runs(da, db, d, D, monkeypatch):
    """Stage 2 of a wide operator as products whose columns lie in several runs, one per row of the block pair:
    the 64 x 64 tiles that read any layout."""
    monkeypatch.setenv("CT_STAGE2", "mfma")
    monkeypatch.setenv("CT_GEMM_LDS", "large")
    ts, want = dense_problem(da, db, d, D, 5 * da + db)
    plan = ct.MatvecPlan(*ts, ct.GROUPED_FP64)
    print("case", da, db, d, D, "forms", plan.forms()[0], flush=True)
    assert plan.forms()[0][1] == 6
    x, y = ct.DeviceArray.from_numpy(ts[0].serialize()), ct.DeviceArray(plan.dim)
    plan.apply(x, y)
    plan.synchronize()
    assert np.linalg.norm(y.numpy() - want) <= 2e-14 * np.linalg.norm(want)


@pytest.mark.parametrize("stage2", ["rowtiles", "mfma"])
@pytest.mark.parametrize("n,chi", [(8, 96), (8, 150), (10, 160)])
def test_wide_classes_of_several_sectors(n, chi, stage2, monkeypatch):
    """Stage 2 of a molecular operator, with classes of many sectors and blocks that are absent, as row tiles and
    as tiles that read any layout, against the oracle."""
    from oracle import oracle as orc
    monkeypatch.setenv("CT_STAGE2", stage2)
    monkeypatch.setenv("CT_GEMM_LDS", "large")
    pm = ct.MPO.spin_molecular(*ct.molecular_coefficients(n, 5))
    p = orc.matvec_problem_mpo(orc.MPOView(pm.ptr, pm.nsites, pm.d, pm.qsite), orc.encode_pair(n, 0), chi, 2024)
    want = orc.apply_local_hamiltonian(*p).serialize()
    plan = ct.MatvecPlan(*p, ct.GROUPED_FP64)
    print("case", n, chi, stage2, "forms", plan.forms()[0], flush=True)
    assert plan.forms()[0][1] == (8 if stage2 == "rowtiles" else 6)
    x, y = ct.DeviceArray.from_numpy(p[0].serialize()), ct.DeviceArray(plan.dim)
    plan.apply(x, y)
    plan.synchronize()
    assert np.linalg.norm(y.numpy() - want) <= 2e-14 * np.linalg.norm(want)
