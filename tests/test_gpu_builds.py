"""The joins' build sides, run several to a launch, and the results' way back,
at the table sizes where their tiling can go wrong, against the plan oracle."""
import pytest

pytestmark = pytest.mark.gpu

from oracle import datagen, plan_oracle as PO  # noqa: E402
from sycldb_amd import plans as PL  # noqa: E402
from sycldb_amd import schema as S  # noqa: E402

PLANS = [("t1", {"date": ("year", 1992), "disc": (0, 10), "qty": ("lt", 51)}),
         ("t1", {"date": ("yearmonthnum", 199201), "disc": (1, 3), "qty": ("range", 2, 40)}),
         ("t1", {"date": ("year_range_and", 1992, 1993), "disc": (4, 6), "qty": ("lt", 25)}),
         ("t2", {"part": ("category", 1), "s_region": 1}), ("t2", {"part": ("brand_range", 40, 900), "s_region": 2}),
         ("t3", {"cust": ("region", 1), "supp": ("region", 1), "date": ("year_range", 1992, 1997), "group": "nation"}),
         ("t3", {"cust": ("city2", 3, 141), "supp": ("region", 0), "date": ("year_range", 1992, 1997), "group": "city"}),
         ("t3", {"cust": ("nation", 6), "supp": ("nation", 6), "date": ("yearmonthnum", 199202), "group": "city"}),
         ("t4", {"c_region": 1, "s_region": 1, "mfgr": (0, 1)}), ("t4", {"c_region": 0, "s_region": 2, "mfgr": (2, 4)})]


# 1,024 rows per block and step, 4 per thread: one row, fewer than a thread's,
# around a block's, around two; the batch holds more builds than one launch takes
@pytest.mark.parametrize("customer,supplier,part,ddate", [
    (1, 1, 1, 1), (3, 5, 2, 366), (1023, 1024, 1025, 2556), (2049, 4097, 2047, 1025)])
def test_build_sides_at_block_edges(customer, supplier, part, ddate):
    from sycldb_amd.engine import Engine
    sizes = {"customer": customer, "supplier": supplier, "part": part, "ddate": ddate}
    rows, seed = 20_011, 45
    tables = datagen.generate_tables(S, rows, seed, sizes)
    plans = [PL.build(t, **p) for t, p in PLANS]
    with Engine() as eng:
        eng.generate(rows, seed, sizes=sizes)
        want = [PO.execute_plan(p, tables).rows() for p in plans]
        for plan, w in zip(plans, want):
            assert eng.execute(plan).rows() == w, plan
        got, _ = eng.execute_batch(plans * 3)
        for g, p, w in zip(got, plans * 3, want * 3):
            assert g.rows() == w, p


def test_many_large_results_in_one_batch():
    """437,500-slot results: the first six are written to the host by the
    kernels that find their rows, the others (past the staging buffer's
    share) compacted and gathered, all beside dense results."""
    from sycldb_amd.engine import Engine
    rows, seed = 200_003, 45
    tables = datagen.generate_tables(S, rows, seed)
    plans = [PL.build("t3", cust=("region", i % 5), supp=("region", (i * 2 + 1) % 5), date=("year_range", 1992, 1997),
                      group="city") for i in range(8)]
    plans[3:3] = [PL.build("t1"), PL.build("t2", part=("category", 1), s_region=1)]
    plans.append(PL.build("t3", cust=("city2", 1, 2), supp=("city2", 3, 4), date=("yearmonthnum", 199712), group="city"))
    with Engine() as eng:
        eng.generate(rows, seed)
        for _ in range(2):
            got, _ = eng.execute_batch(plans)
            for g, p in zip(got, plans):
                assert g.rows() == PO.execute_plan(p, tables).rows(), p


@pytest.mark.parametrize("rows", [(4 << 20) - 1, 4 << 20, (16 << 20) - 1, 16 << 20])
def test_probe_tables_by_rows(rows):
    """Joins over fewer rows than these probe the reference tables, over more
    the compact ones (alone from 4M rows on, batched from 16M): the results of
    one kernel per operator."""
    from sycldb_amd.engine import Engine
    plans = [PL.build(t, **p) for t, p in PLANS]
    with Engine() as eng:
        eng.generate(rows, 45)
        eng.set_fusion(False)
        want = [eng.execute(p).rows() for p in plans]
        eng.set_fusion(True)
        assert [eng.execute(p).rows() for p in plans] == want
        got, batched = eng.execute_batch(plans)
        assert [g.rows() for g in got] == want and batched == len(plans)


@pytest.mark.parametrize("table,column,value", [("customer", 4, 6), ("supplier", 5, 1), ("customer", 4, 99)])
def test_results_that_are_no_groupby(table, column, value):
    """A filtered dimension as the result: 300,000 rows (not listed when they
    arrive) and 20,000 (listed), some rows selected and none."""
    import json
    from sycldb_amd.engine import Engine
    plan = json.loads(PL.to_json(PL.build("t3", cust=("nation", 6))))
    scan, keep = dict(plan["rels"][1], id=0, tables=["ssb", table]), dict(plan["rels"][2], id=1)
    keep["condition"]["operands"][0].update(input=column, name="$%d" % column)
    keep["condition"]["operands"][1]["literal"]["value"] = value
    tables = datagen.generate_tables(S, 1000, 45)
    for rels in ([scan, keep], [scan]):
        want = PO.execute_plan(dict(plan, rels=rels), tables).rows()
        for fusion in (True, False):
            with Engine(fusion=fusion) as eng:
                eng.generate(1000, 45)
                got = eng.execute(dict(plan, rels=rels))
                assert len(got.selected_rows) == len(want) and got.rows() == want
                assert int((got.flags != 0).sum()) == len(want)


def test_batch_reads_more_columns_than_the_shared_scan_holds():
    """A q3.x sum over each of the 17 fact columns (the scan holds 16): the
    column past it is read from memory.  Then a batch over a few of them in
    the same engine, and the first again."""
    import json
    import numpy as np
    from sycldb_amd.engine import Engine
    rows, seed = 120_003, 45
    tables = datagen.generate_tables(S, rows, seed)
    rng = np.random.default_rng(1)
    for c in set(range(17)) - set(tables["lineorder"]):
        tables["lineorder"][c] = rng.integers(-1000, 1000, rows).astype(np.int32)
    plans = []
    for c in range(17):
        p = json.loads(PL.to_json(PL.build("t3", cust=("region", 1), supp=("region", c % 5),
                                           date=("year_range", 1992, 1997), group="nation")))
        e = next(r for r in p["rels"] if r["relOp"] == "PROJECT")["exprs"][-1]
        e.update(input=c, name="$%d" % c)
        plans.append(p)
    want = [PO.execute_plan(p, tables).rows() for p in plans]
    with Engine() as eng:
        eng.load_tables(tables)
        for some in (plans, plans[2:5], plans):
            got, batched = eng.execute_batch(some)
            assert batched == len(some)
            assert [g.rows() for g in got] == [want[plans.index(p)] for p in some]


def _sum_plans(which):
    """q3.x sums, each over one of the 17 fact columns."""
    import json
    out = []
    for c in which:
        p = json.loads(PL.to_json(PL.build("t3", cust=("region", 1), supp=("region", c % 5),
                                           date=("year_range", 1992, 1997), group="nation")))
        e = next(r for r in p["rels"] if r["relOp"] == "PROJECT")["exprs"][-1]
        e.update(input=c, name="$%d" % c)
        out.append(p)
    return out


def _fact_tables(rows, seed):
    import numpy as np
    tables = datagen.generate_tables(S, rows, seed)
    rng = np.random.default_rng(seed)
    for c in set(range(17)) - set(tables["lineorder"]):
        tables["lineorder"][c] = rng.integers(-1000, 1000, rows).astype(np.int32)
    return tables


def test_batches_past_the_shared_scan_keep_their_kernels():
    """A batch over all 17 fact columns between others: what the table's
    batches compiled stays in use, whichever ran last."""
    from sycldb_amd import engine as E
    tables = _fact_tables(50_003, 45)
    one = _sum_plans(range(17))
    two, three = [PL.build("t1"), PL.build("t4")], [PL.build("t2"), PL.build("t2", s_region=3)]
    with E.Engine() as eng:
        eng.load_tables(tables)
        for some in (one, two, one, three):
            eng.execute_batch(some)
        assert E.codegen_wait(100)
        before = E.codegen_kernels_compiled()
        for some in (one, two, three):
            assert eng.execute_batch(some)[1] == len(some)
        assert E.codegen_wait(100) and E.codegen_kernels_compiled() == before


def test_batches_over_a_table_loaded_again():
    """The fact table replaced (its columns then lie elsewhere, the table
    itself maybe where it was): the batch's results are the new table's."""
    from sycldb_amd.engine import Engine
    plans = _sum_plans(range(4, 16))
    with Engine() as eng:
        for seed in (45, 46, 47):
            tables = _fact_tables(30_001 + seed, seed)
            eng.load_tables(tables)
            got, batched = eng.execute_batch(plans)
            assert batched == len(plans)
            assert [g.rows() for g in got] == [PO.execute_plan(p, tables).rows() for p in plans]


def test_result_staging_goes_back():
    """A batch of large results, thousands of small ones, the batch again."""
    from sycldb_amd.engine import Engine
    tables = datagen.generate_tables(S, 60_003, 45)
    large = [PL.build("t3", cust=("region", i), supp=("region", i), date=("year_range", 1992, 1997), group="city")
             for i in range(5)]
    small = PL.build("t1")
    w_large, w_small = [PO.execute_plan(p, tables).rows() for p in large], PO.execute_plan(small, tables).rows()
    with Engine() as eng:
        eng.load_tables(tables)
        assert [r.rows() for r in eng.execute_batch(large)[0]] == w_large
        for _ in range(2 * 4096 + 8):  # (its buffer then is a small one)
            eng.execute(small)
        for _ in range(3):
            assert eng.execute(small).rows() == w_small
        assert [r.rows() for r in eng.execute_batch(large)[0]] == w_large


# 1,000-row segments: those builds keep kernels of their own, in order
@pytest.mark.parametrize("customer,supplier,part,ddate", [(999, 1001, 2000, 2556), (3001, 1, 1000, 366)])
def test_segmented_build_sides(customer, supplier, part, ddate):
    from sycldb_amd.engine import Engine
    sizes = {"customer": customer, "supplier": supplier, "part": part, "ddate": ddate}
    rows, seed = 7_001, 45
    tables = datagen.generate_tables(S, rows, seed, sizes)
    with Engine(segment_size=1000) as eng:
        eng.generate(rows, seed, sizes=sizes)
        for t, p in PLANS:
            plan = PL.build(t, **p)
            assert eng.execute(plan).rows() == PO.execute_plan(plan, tables).rows(), plan


@pytest.mark.parametrize("rows", [(4 << 20) - 1, 4 << 20, (4 << 20) + 1])
def test_largest_build_side_of_a_shared_launch(rows):
    """Build sides of fewer than 4M rows share a launch, larger ones have
    kernels of their own: the results of one kernel per operator."""
    from sycldb_amd.engine import Engine
    plans = [PL.build(t, **p) for t, p in PLANS if t in ("t2", "t3", "t4")]
    with Engine() as eng:
        eng.generate(300_001, 45, sizes={"customer": rows, "part": rows})
        eng.set_fusion(False)
        want = [eng.execute(p).rows() for p in plans]
        eng.set_fusion(True)
        for _ in range(2):
            assert [eng.execute(p).rows() for p in plans] == want
        assert any(want)


ONE_BUFFER = """
import sys
sys.path.insert(0, "tests")
import quirk_plans as Q
from oracle import datagen, plan_oracle as PO
from sycldb_amd import plans as PL, schema as S
from sycldb_amd.engine import Engine
tables = datagen.generate_tables(S, 50_007, 45)
b = PL.PlanBuilder()  # its flags are the result
b.scan("lineorder")
b.filter(PL.expr("AND", PL.expr("=", PL.col(S.LO_DISCOUNT), PL.lit(2)), PL.expr("<", PL.col(S.LO_QUANTITY), PL.lit(9))))
plans = [PL.build("t4"), PL.build("t1"), Q.left_fold_or_and(), Q.left_fold_and_or(), Q.filter_after_join(), b.plan()]
with Engine(fusion=False) as eng:
    eng.load_tables(tables)
    for p in plans:
        print("plan", file=sys.stderr)
        assert eng.execute(p).rows() == PO.execute_plan(p, tables).rows()
"""


def test_which_operators_share_a_flag_buffer():
    """One kernel per operator: a chain whose flags nobody reads after it keeps
    them in one buffer, a filter that is the plan's result does not."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", ONE_BUFFER], cwd=root, capture_output=True, text=True, timeout=110,
                         env=dict(os.environ, SDB_DEBUG_FUSED="1"))
    assert out.returncode == 0, out.stderr[-4000:]
    forms = [[l.split("one_flag_buffer=")[1] for l in part.splitlines() if l.startswith("[unfused lineorder]")]
             for part in out.stderr.split("plan\n")[1:]]
    assert forms == [["1"]] * 5 + [["0"]]
