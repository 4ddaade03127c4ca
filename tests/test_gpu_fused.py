"""Forms of the fused fact kernels that only large or wide programs take,
against the same plans run one kernel per operator."""
import pytest

pytestmark = pytest.mark.gpu

from oracle import datagen, plan_oracle as PO  # noqa: E402
from sycldb_amd import plans as PL  # noqa: E402
from sycldb_amd import schema as S  # noqa: E402
from sycldb_amd.engine import Engine  # noqa: E402

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
