"""Forms of the fused fact kernels that only large or wide programs take,
against the same plans run one kernel per operator."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

from oracle import datagen, plan_oracle as PO  # noqa: E402
from sycldb_amd import plans as PL  # noqa: E402
from sycldb_amd import schema as S  # noqa: E402
from sycldb_amd.engine import Engine  # noqa: E402

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
T2 = (S.LO_PARTKEY, S.LO_SUPPKEY, S.LO_ORDERDATE, S.LO_REVENUE)


def _both(eng, plan):
    eng.set_fusion(True)
    fused = eng.execute(plan).rows()
    eng.set_fusion(False)
    return fused, eng.execute(plan).rows()


def test_presence_filter_of_a_wide_probe():
    """From 2^25 rows on, a selective probe of a table of 2^20 slots or more
    tests its keys against the folded presence bitmap in LDS first: a table
    larger than the filter, one that the filter holds whole, one slot range
    below the limit; 4 % and 0.1 % of the parts, one brand, and too many."""
    rows = (1 << 25) + 1027
    for parts in (1_400_000, 1 << 20, (1 << 20) - 1):
        with Engine(codegen="compile") as eng:
            eng.generate(rows, 11, sizes={"part": parts}, fact_columns=T2)
            for part in (("category", 3), ("brand", 77), ("brand_range", 120, 127), ("mfgr2", 0, 1)):
                print("parts", parts, part, flush=True)
                plan = PL.t2_plan(part, 2)
                fused, unfused = _both(eng, plan)
                assert fused == unfused and len(fused) > 0


# The groups a group-by is expected to meet decide its form: 6 x 10 x 10 in
# the LDS hash, 6 x 10 x 50 crowding it, 6 x 50 x 50 straight to the global
# arrays; a build side with keys outside the group's range (the slot's
# remainder) stays with the general form.
@pytest.mark.parametrize("cust,supp", [(("nation", 6), ("nation", 6)), (("nation", 6), ("region", 1)),
                                       (("region", 1), ("region", 3))])
@pytest.mark.parametrize("codegen", ["compile", "interpret"])
def test_groupby_forms(cust, supp, codegen):
    from sycldb_amd.engine import Engine
    plan = PL.build("t3", cust=cust, supp=supp, date=("year_range", 1992, 1997), group="city")
    tables = datagen.generate_tables(S, 300_007, 45)
    want = PO.execute_plan(plan, tables).rows()
    with Engine(codegen=codegen) as eng:
        eng.generate(300_007, 45)
        assert eng.execute(plan).rows() == want and len(want) > 100


# Run in a process of its own: the switch is read once.
EARLY = """
from sycldb_amd import plans as PL, schema as S
from sycldb_amd.engine import Engine
cols = (S.LO_QUANTITY, S.LO_CUSTKEY, S.LO_SUPPKEY, S.LO_REVENUE)
b = PL.PlanBuilder()
b.scan("lineorder")
lo = b.filter(PL.expr("<", PL.col(S.LO_QUANTITY), PL.lit(25)))
b.scan("customer")
cust = b.filter(PL.expr("=", PL.col(S.C_NATION), PL.lit(6)))
j1 = b.join(lo, cust, S.LO_CUSTKEY, S.C_CUSTKEY)
c_at = b.offset(lo) + S.C_NATION
b.scan("supplier")
supp = b.filter(PL.search(PL.col(S.S_CITY), PL.closed_range(20, 79)))
s_at = b.offset(j1) + S.S_NATION
b.join(j1, supp, S.LO_SUPPKEY, S.S_SUPPKEY)
b.project([PL.col(c_at), PL.col(s_at), PL.col(S.LO_REVENUE)], ["c_nation", "s_nation", "lo_revenue"])
b.aggregate([0, 1], 2, "revenue")
with Engine(codegen="compile") as eng:
    eng.generate((1 << 25) + 1027, 11, sizes={"customer": 1_400_000}, fact_columns=cols)
    fused = eng.execute(b.plan()).rows()
    eng.set_fusion(False)
    assert fused == eng.execute(b.plan()).rows() and len(fused) > 0
"""


def test_filtered_probe_issued_early():
    """SDB_JIT_HOIST=1 issues the customer probe's reads, behind their
    presence filter, with the supplier's value reads: rows that the supplier
    drops in between stay dropped."""
    out = subprocess.run([sys.executable, "-c", EARLY], cwd=ROOT, capture_output=True, text=True, timeout=110,
                         env=dict(os.environ, SDB_JIT_HOIST="1", SDB_DEBUG_FUSED="1"))
    print(out.stderr[-4000:])
    assert out.returncode == 0, out.stdout
    assert "fold=3" in out.stderr  # the filtered probe comes third
