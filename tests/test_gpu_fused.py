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


# 6 x 10 x 10 groups, 6 x 10 x 50, 6 x 50 x 50, through the LDS hash: the last
# are more than it holds, and a row looks at few of its slots.
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


FORMS = """
import numpy as np
from oracle import datagen, plan_oracle as PO
from sycldb_amd import plans as PL, schema as S
from sycldb_amd.engine import Engine
tables = datagen.generate_tables(S, 120_007, 45)
rng = np.random.default_rng(1)
for key, n in ((S.LO_CUSTKEY, 300_000), (S.LO_SUPPKEY, 20_000)):  # nine rows in ten in one group
    tables["lineorder"][key] = np.where(rng.random(120_007) < 0.9, 77, rng.integers(1, n, 120_007)).astype(np.int32)
where = [int(tables[t][c][76]) for t, c in (("customer", S.C_REGION), ("supplier", S.S_REGION))]
with Engine(codegen="%s") as eng:
    eng.load_tables(tables)
    for group in ("nation", "city"):
        plan = PL.build("t3", cust=("region", where[0]), supp=("region", where[1]), date=("year_range", 1992, 1997),
                        group=group)
        rows = eng.execute(plan).rows()
        assert rows == PO.execute_plan(plan, tables).rows()
        assert len(rows) > 50, len(rows)
"""


@pytest.mark.parametrize("codegen", ["compile", "interpret"])
def test_groupby_of_many_groups_keeps_the_hash(codegen):
    """Where one group takes most of the rows its sum belongs in LDS, however
    many groups there may be: 875 (32 tries) and 17,500 (4)."""
    out = subprocess.run([sys.executable, "-c", FORMS % codegen], cwd=ROOT, capture_output=True, text=True, timeout=110,
                         env=dict(os.environ, SDB_DEBUG_FUSED="1"))
    forms = [line.split("group=")[1].split(" fold")[0] for line in out.stderr.splitlines()
             if line.startswith("[fused lineorder]")]
    assert out.returncode == 0, out.stderr[-4000:]
    assert forms == ["2 tries=32", "2 tries=4"]


@pytest.mark.parametrize("spans,prod", [([(0, 599)], 600), ([(5, 3004)], 3000), ([(-7, 2), (1, 600)], 6000),
                                        ([(-7, 2), (1, 600)], 6001), ([(3, 9), (0, 40)], 100)])
def test_groupby_of_keys_outside_their_ranges(spans, prod):
    """A fused group-by whose keys leave the ranges it was given, in LDS (dense,
    hashed with many and with few tries) and where the ranges do not multiply
    to the slots: those rows take their slot's remainder, the others theirs."""
    import numpy as np
    import torch
    from oracle import oracle as O
    from sycldb_amd import _lib as L, ops
    from sycldb_amd.engine import codegen_wait
    n, rng = 70_003, np.random.default_rng(prod)
    keys = [rng.integers(a - 3, b + 4, n).astype(np.int32) for a, b in spans]
    agg = rng.integers(-2**31, 2**31, n).astype(np.int32)
    fl = (rng.random(n) < 0.7).astype(np.uint8)
    mins, maxs = [a for a, _ in spans], [b for _, b in spans]
    ws, wn = np.zeros(prod, np.uint64), np.zeros(prod, np.uint32)
    O.groupby_dense(keys, mins, maxs, agg, fl, [np.zeros(prod, np.int32) for _ in spans], ws, wn, prod)
    dk, da, df = [torch.from_numpy(k).cuda() for k in keys], torch.from_numpy(agg).cuda(), torch.from_numpy(fl).cuda()
    outk = [torch.zeros(prod, dtype=torch.int32, device="cuda") for _ in spans]
    sums, seen = (torch.zeros(prod, dtype=d, device="cuda") for d in (torch.int64, torch.int32))
    op = L.Op(kind=L.OP_GROUPBY, nkeys=len(spans), col=da.data_ptr(), in_flags=df.data_ptr(), sums=sums.data_ptr(),
              seen=seen.data_ptr(), prod=prod)
    for j in range(len(spans)):
        op.keys[j], op.out_keys[j], op.mins[j], op.maxs[j] = dk[j].data_ptr(), outk[j].data_ptr(), mins[j], maxs[j]
    for rep in range(2):  # the interpreter, then the compiled kernel
        sums.zero_(), seen.zero_()
        ops.bundle_exec([op], n)
        assert (sums.cpu().numpy().view(np.uint64) == ws).all() and (seen.cpu().numpy().view(np.uint32) == wn).all()
        assert codegen_wait(100)


FILTERED = """
from sycldb_amd import plans as PL, schema as S
from sycldb_amd.engine import Engine
T2 = (S.LO_PARTKEY, S.LO_SUPPKEY, S.LO_ORDERDATE, S.LO_REVENUE)
for rows, parts in (((1 << 25) + 3, 1_400_000), ((1 << 25) + 3, (1 << 20) - 1), ((1 << 25) - 1, 1_400_000)):
    with Engine(codegen="interpret") as eng:
        eng.generate(rows, 11, sizes={"part": parts}, fact_columns=T2)
        for cg in ("compile", "interpret"):
            eng.set_codegen(cg)
            for part in (("category", 3), ("mfgr2", 0, 1)):
                eng.execute(PL.t2_plan(part, 2))
"""


def test_presence_filter_is_taken():
    """Of the plans above, those with a presence filter: enough rows, a wide
    table, few matches, a compiled kernel."""
    out = subprocess.run([sys.executable, "-c", FILTERED], cwd=ROOT, capture_output=True, text=True, timeout=110,
                         env=dict(os.environ, SDB_DEBUG_FUSED="1"))
    assert out.returncode == 0, out.stderr[-4000:]
    folds = [line.split("fold=")[1] != "0" for line in out.stderr.splitlines() if line.startswith("[fused lineorder]")]
    assert folds == [True, False, False, False] + [False] * 8
