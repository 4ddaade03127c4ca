"""Performance cases: what a program built on this package has it do.

Five kinds of work, each through the public entry points:

  plan     Engine.execute: one star-join query over resident tables.
  batch    Engine.execute_batch: several queries that share one fact scan.
  bundle   ops.bundle_exec: a segment's operators handed over as one bundle.
  filter   the operator functions of a q1.x query, one call per operator:
           date build side, three selections, the fold, the semi join, the
           projected product, the sum.
  star     the operator functions of a q2.x query: three build sides, two
           full joins and a semi join over the fact table, the group-by.
  compact  flags to row ids, and the selected rows of two columns.

Tables have the star schema of sycldb_amd.schema with uniform values, filled
on the device by torch's generator, so exact() can make the same tables
without the package.  Every output is a whole number and is compared as such.
"""
import ctypes
import datetime
import json
import math

import numpy as np
import torch

from sycldb_amd import _lib as L
from sycldb_amd import engine as E
from sycldb_amd import ops
from sycldb_amd import plans as PL
from sycldb_amd import schema as S

DEV = "cuda"
# dimension rows: scale factor 100 as in the package's configurations, and 1
DIMS = {"sf100": {"customer": 300_000, "supplier": 20_000, "part": 1_400_000, "ddate": 2556},
        "sf1": {"customer": 30_000, "supplier": 2_000, "part": 200_000, "ddate": 2556}}
ANSWER = 5 * 50 * 50 * 7  # values of one query's answer at most
Q1, Q3 = '{"date": ["year", 1993], "disc": [1, 3], "qty": ["lt", 25]}', \
    '{"cust": ["region", 2], "supp": ["region", 2], "date": ["year_range", 1992, 1997], "group": "nation"}'
Q3_CITY = '{"cust": ["region", 1], "supp": ["region", 3], "date": ["year_range", 1992, 1997], "group": "city"}'
Q2 = '{"part": ["category", 1], "s_region": 1}'
Q4 = '{"c_region": 1, "s_region": 1, "mfgr": [0, 1]}'


def listed():
    return [
        # an interactive query on a small table: latency and launches
        {"name": "plan_q4_200k", "kind": "plan", "template": "t4", "params": Q4, "rows": 200_000, "dims": "sf100",
         "fusion": True},
        # the 6M-row configuration: date semi join, two filters, one sum
        {"name": "plan_q1_6m", "kind": "plan", "template": "t1", "params": Q1, "rows": 6_000_000, "dims": "sf100",
         "fusion": True},
        # the 60M-row configuration: three joins, 25 x 25 x 7 groups
        {"name": "plan_q3_60m", "kind": "plan", "template": "t3", "params": Q3, "rows": 60_000_000, "dims": "sf100",
         "fusion": True},
        # grouped by city: 437,500 possible groups, thousands of result rows; a ragged row count
        {"name": "plan_q3_city_30m", "kind": "plan", "template": "t3", "params": Q3_CITY, "rows": 30_000_003,
         "dims": "sf100", "fusion": True},
        # the 600M-row configuration: selective part and supplier joins
        {"name": "plan_q2_600m", "kind": "plan", "template": "t2", "params": Q2, "rows": 600_000_000, "dims": "sf100",
         "fusion": True},
        # four joins with one kernel per operator (the reference's own mode)
        {"name": "plan_q4_unfused_60m", "kind": "plan", "template": "t4", "params": Q4, "rows": 60_000_001,
         "dims": "sf100", "fusion": False},
        # a served batch: the mean batch of a loaded server, on its small table
        {"name": "batch_8_6m", "kind": "batch", "pipelines": 8, "pipeline_seed": 46, "rows": 6_000_000,
         "dims": "sf100"},
        # the batched configuration: 32 pipelines of uneven selectivity over 600M rows
        {"name": "batch_32_600m", "kind": "batch", "pipelines": 32, "pipeline_seed": 46, "rows": 600_000_000,
         "dims": "sf100"},
        # one fused bundle in place of an executor's operator queue
        {"name": "bundle_q1_6m", "kind": "bundle", "rows": 6_000_000, "disc_lo": 1, "disc_hi": 3, "qty": 25,
         "year": 1993},
        # q1.x operator by operator on an ordinary, odd-sized segment
        {"name": "filter_60m", "kind": "filter", "rows": 60_000_001, "disc_lo": 1, "disc_hi": 3, "qty": 25,
         "year": 1993},
        # q2.x operator by operator on a full segment (2^28 rows)
        {"name": "star_268m", "kind": "star", "rows": 1 << 28, "dims": "sf100", "category": 1, "region": 1},
        # bringing a segment's selected rows together: one row in twenty
        {"name": "compact_100m", "kind": "compact", "rows": 100_000_007, "density": 0.05},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plan", "plan", "plan", "batch", "bundle", "filter", "filter", "star", "star", "compact"])
    dims = rng.choice(["sf100", "sf100", "sf1"])
    if kind == "plan":
        t, params = PL.random_pipelines(4, rng.randrange(1 << 30))[rng.randrange(4)]
        fusion = rng.random() < 0.75
        return {"kind": kind, "template": t, "params": json.dumps(params),
                "rows": _log_int(rng, 100_000, 600_000_000 if fusion else 150_000_000), "dims": dims, "fusion": fusion}
    if kind == "batch":
        return {"kind": kind, "pipelines": rng.randint(3, 32), "pipeline_seed": rng.randrange(1 << 30),
                "rows": _log_int(rng, 1_000_000, 200_000_000), "dims": dims}
    lo, qty = rng.randint(0, 8), rng.randint(2, 50)
    q1 = {"disc_lo": lo, "disc_hi": lo + rng.randint(0, 2), "qty": qty, "year": rng.randint(1992, 1998)}
    if kind == "bundle":
        return {"kind": kind, "rows": _log_int(rng, 50_000, 200_000_000), **q1}
    if kind == "filter":
        return {"kind": kind, "rows": _log_int(rng, 50_000, 1 << 28), **q1}
    if kind == "star":
        return {"kind": kind, "rows": _log_int(rng, 50_000, 1 << 28), "dims": dims, "category": rng.randrange(25),
                "region": rng.randrange(5)}
    return {"kind": kind, "rows": _log_int(rng, 50_000, 1 << 28), "density": round(10 ** rng.uniform(-3, -0.3), 4)}


# ------------------------------------------------------------------- tables

def _dates():
    d = [datetime.date(1992, 1, 1) + datetime.timedelta(days=i) for i in range(DIMS["sf100"]["ddate"])]
    return {S.D_DATEKEY: [x.year * 10000 + x.month * 100 + x.day for x in d], S.D_YEAR: [x.year for x in d],
            S.D_YEARMONTHNUM: [x.year * 100 + x.month for x in d]}


def _gen(seed, table, col):
    return torch.Generator(DEV).manual_seed(((seed & 0xFFFFFFFF) << 16) + S.TABLE_IDS[table] * 64 + col)


def _column(table, col, rows, dims, seed, out=None, parent=None):
    """One column on the device (into `out` if given), a function of the
    seed; a column of a hierarchy takes its parent column."""
    if table == "ddate":
        v = torch.tensor(_dates()[col], dtype=torch.int32, device=DEV)
        return v if out is None else out.copy_(v)
    if out is None:
        out = torch.empty(rows, dtype=torch.int32, device=DEV)
    g = _gen(seed, table, col)
    if table == "lineorder":
        lo, hi = {S.LO_CUSTKEY: (1, dims["customer"]), S.LO_PARTKEY: (1, dims["part"]),
                  S.LO_SUPPKEY: (1, dims["supplier"]), S.LO_ORDERDATE: (0, dims["ddate"] - 1),
                  S.LO_QUANTITY: (1, 50), S.LO_EXTENDEDPRICE: (90_000, 10_500_000), S.LO_DISCOUNT: (0, 10),
                  S.LO_REVENUE: (100, 1_000_000), S.LO_SUPPLYCOST: (100, 100_000)}[col]
        out.random_(lo, hi + 1, generator=g)
        if col == S.LO_ORDERDATE:
            days = torch.tensor(_dates()[S.D_DATEKEY], dtype=torch.int32, device=DEV)
            for a in range(0, rows, 1 << 26):
                out[a:a + (1 << 26)] = days[out[a:a + (1 << 26)].long()]
        return out
    if col == 0:
        return torch.arange(1, rows + 1, dtype=torch.int32, device=DEV, out=out)
    if table == "part":
        up, mult, hi = {S.P_MFGR: (None, 0, 4), S.P_CATEGORY: (S.P_MFGR, 5, 4), S.P_BRAND1: (S.P_CATEGORY, 40, 39)}[col]
    else:
        up, mult, hi = {S.S_REGION: (None, 0, 4), S.S_NATION: (S.S_REGION, 5, 4), S.S_CITY: (S.S_NATION, 10, 9)}[col]
    out.random_(0, hi + 1, generator=g)
    if up is not None:
        out += mult * (parent if parent is not None else _column(table, up, rows, dims, seed))
    return out


DIM_COLUMNS = {"part": (S.P_PARTKEY, S.P_MFGR, S.P_CATEGORY, S.P_BRAND1),
               "supplier": (S.S_SUPPKEY, S.S_REGION, S.S_NATION, S.S_CITY),
               "customer": (S.C_CUSTKEY, S.C_REGION, S.C_NATION, S.C_CITY),
               "ddate": (S.D_DATEKEY, S.D_YEAR, S.D_YEARMONTHNUM)}
FACT_COLUMNS = {"t1": (S.LO_ORDERDATE, S.LO_QUANTITY, S.LO_EXTENDEDPRICE, S.LO_DISCOUNT),
                "t2": (S.LO_PARTKEY, S.LO_SUPPKEY, S.LO_ORDERDATE, S.LO_REVENUE),
                "t3": (S.LO_CUSTKEY, S.LO_SUPPKEY, S.LO_ORDERDATE, S.LO_REVENUE),
                "t4": (S.LO_CUSTKEY, S.LO_PARTKEY, S.LO_SUPPKEY, S.LO_ORDERDATE, S.LO_REVENUE, S.LO_SUPPLYCOST)}
DIM_TABLES = {"t1": ("ddate",), "t2": ("part", "supplier", "ddate"), "t3": ("customer", "supplier", "ddate"),
              "t4": ("customer", "supplier", "part", "ddate")}


def _pipes(case):
    if case["kind"] == "plan":
        return [(case["template"], json.loads(case["params"]))]
    return PL.random_pipelines(case["pipelines"], case["pipeline_seed"])


class _Memory:
    """A column of an engine's table as torch sees it."""

    def __init__(self, ptr, rows):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (rows,), "typestr": "<i4", "version": 2}


def _load(eng, table, cols, rows, dims, seed):
    eng.create_table(table, rows)
    made = {}
    for c in cols:
        t = torch.as_tensor(_Memory(eng.column_ptr(table, c), rows), device=DEV)
        parent = {S.P_CATEGORY: made.get(S.P_MFGR), S.P_BRAND1: made.get(S.P_CATEGORY)} if table == "part" else \
            {S.S_NATION: made.get(S.S_REGION), S.S_CITY: made.get(S.S_NATION)}
        made[c] = _column(table, c, rows, dims, seed, out=t, parent=parent.get(c) if table != "lineorder" else None)
    torch.cuda.synchronize()
    eng.finalize(table)


def _fact(cols, rows, dims, seed):
    return {c: _column("lineorder", c, rows, dims, seed) for c in cols}


def _dim(table, cols, dims, seed):
    return {c: _column(table, c, dims[table], dims, seed) for c in cols}


# ------------------------------------------------------------------ prepare

def prepare(case, seed):
    return {"plan": _prepare_engine, "batch": _prepare_engine, "bundle": _prepare_q1, "filter": _prepare_q1,
            "star": _prepare_star, "compact": _prepare_compact}[case["kind"]](case, int(seed))


def _prepare_engine(case, seed):
    pipes, dims = _pipes(case), DIMS[case["dims"]]
    used = sorted({t for t, _ in pipes})
    eng = E.Engine(fusion=case.get("fusion", True))
    for table in sorted({d for t in used for d in DIM_TABLES[t]}):
        _load(eng, table, DIM_COLUMNS[table], dims[table], dims, seed)
    _load(eng, "lineorder", sorted({c for t in used for c in FACT_COLUMNS[t]}), case["rows"], dims, seed)
    plans = [PL.to_json(PL.build(t, **p)) for t, p in pipes]
    # answers are laid one after another on a page: the rows and columns of a
    # query group by at most 50 x 50 cities x 7 years
    state = {"kind": case["kind"], "engine": eng, "plans": plans, "end": 0,
             "page": np.zeros(ANSWER * len(plans), np.int64), "sizes": np.zeros(len(plans), np.int64)}
    # a long-running program's kernels are compiled and tuned
    for _ in range(32):
        run(state)
        if E.codegen_pending() == 0:
            break
        E.codegen_wait(120)
    return state


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _op(kind, **kw):
    o = L.Op()
    o.kind = kind
    for k, v in kw.items():
        setattr(o, k, v.data_ptr() if isinstance(v, torch.Tensor) else v)
    return o


def _prepare_q1(case, seed):
    n, dims = case["rows"], DIMS["sf100"]
    s = {"case": case, "n": n, "kind": case["kind"], **_dim("ddate", (S.D_DATEKEY, S.D_YEAR), dims, seed)}
    s["lo"] = _fact(FACT_COLUMNS["t1"], n, dims, seed)
    s["min"], s["max"] = int(s[S.D_DATEKEY].min()), int(s[S.D_DATEKEY].max())
    s["len"] = s["max"] - s["min"] + 1
    s["ht"] = torch.zeros(s["len"], dtype=torch.uint8, device=DEV)
    s["dflags"] = torch.ones(dims["ddate"], dtype=torch.uint8, device=DEV)
    s["flags"] = torch.ones(n, dtype=torch.uint8, device=DEV)
    s["local"] = torch.zeros(n, dtype=torch.uint8, device=DEV)
    s["rev"] = torch.zeros(n, dtype=torch.int32, device=DEV)
    s["acc"] = torch.zeros(1, dtype=torch.int64, device=DEV)
    if case["kind"] == "bundle":
        _q1_build(s)
        lo, f = s["lo"], s["flags"]
        s["ops"] = [
            _op(L.OP_SELECT_LIT, cmp=L.GE, logic=L.NONE, value=case["disc_lo"], col=lo[S.LO_DISCOUNT], in_flags=f, out_flags=f),
            _op(L.OP_SELECT_LIT, cmp=L.LE, logic=L.AND, value=case["disc_hi"], col=lo[S.LO_DISCOUNT], in_flags=f, out_flags=f),
            _op(L.OP_SELECT_LIT, cmp=L.LT, logic=L.AND, value=case["qty"], col=lo[S.LO_QUANTITY], in_flags=f, out_flags=f),
            _op(L.OP_PROBE_SEMI, col=lo[S.LO_ORDERDATE], ht=s["ht"], ht_min=s["min"], ht_max=s["max"], in_flags=f, out_flags=f),
            _op(L.OP_BINOP_CC, binop=L.MUL, col=lo[S.LO_EXTENDEDPRICE], col2=lo[S.LO_DISCOUNT], res=s["rev"], in_flags=f),
            _op(L.OP_SUM, col=s["rev"], in_flags=f, acc=s["acc"])]
        for _ in range(32):
            run(s)
            torch.cuda.synchronize()
            if E.codegen_pending() == 0:
                break
            E.codegen_wait(120)
    return s


def _prepare_star(case, seed):
    n, dims = case["rows"], DIMS[case["dims"]]
    s = {"case": case, "n": n, "kind": "star", "part": _dim("part", (S.P_PARTKEY, S.P_CATEGORY, S.P_BRAND1), dims, seed),
         "supplier": _dim("supplier", (S.S_SUPPKEY, S.S_REGION), dims, seed),
         "ddate": _dim("ddate", (S.D_DATEKEY, S.D_YEAR), dims, seed), "lo": _fact(FACT_COLUMNS["t2"], n, dims, seed)}
    for t, pairs in (("part", 2), ("supplier", 1), ("ddate", 2)):
        key = s[t][0]
        s[t].update(min=int(key.min()), max=int(key.max()), rows=dims[t])
        s[t]["len"] = s[t]["max"] - s[t]["min"] + 1
        s[t]["ht"] = torch.zeros(pairs * s[t]["len"], dtype=torch.int32 if pairs == 2 else torch.uint8, device=DEV)
        s[t]["flags"] = torch.ones(dims[t], dtype=torch.uint8, device=DEV)
    s["flags"] = torch.ones(n, dtype=torch.uint8, device=DEV)
    s["brand"] = torch.zeros(n, dtype=torch.int32, device=DEV)
    s["year"] = torch.zeros(n, dtype=torch.int32, device=DEV)
    # group ranges: the key columns' load-time statistics
    s["gmin"] = [int(s["ddate"][S.D_YEAR].min()), int(s["part"][S.P_BRAND1].min())]
    s["gmax"] = [int(s["ddate"][S.D_YEAR].max()), int(s["part"][S.P_BRAND1].max())]
    prod = s["prod"] = (s["gmax"][0] - s["gmin"][0] + 1) * (s["gmax"][1] - s["gmin"][1] + 1)
    s["keys"] = [torch.zeros(prod, dtype=torch.int32, device=DEV) for _ in range(2)]
    s["sums"] = torch.zeros(prod, dtype=torch.int64, device=DEV)
    s["seen"] = torch.zeros(prod, dtype=torch.int32, device=DEV)
    s["gflags"] = torch.zeros(prod, dtype=torch.uint8, device=DEV)
    return s


def _compact_inputs(case, seed):
    g = torch.Generator(DEV).manual_seed(seed * 7919 + 17)
    n = case["rows"]
    flags = torch.empty(n, dtype=torch.uint8, device=DEV)
    for a in range(0, n, 1 << 26):
        m = min(1 << 26, n - a)
        flags[a:a + m] = torch.rand(m, generator=g, device=DEV) < case["density"]
    cols = [torch.empty(n, dtype=torch.int32, device=DEV).random_(100, 1_000_000, generator=g) for _ in range(2)]
    return flags, cols


def _prepare_compact(case, seed):
    n = case["rows"]
    flags, cols = _compact_inputs(case, seed)
    ids, *out = (torch.zeros(n, dtype=torch.int32, device=DEV) for _ in range(3))
    return {"kind": "compact", "n": n, "flags": flags, "cols": cols, "ids": ids, "out": out,
            "count": torch.zeros(1, dtype=torch.int32, device=DEV)}


# ---------------------------------------------------------------------- run

def run(state):
    return {"plan": _run_plan, "batch": _run_batch, "bundle": _run_bundle, "filter": _run_filter, "star": _run_star,
            "compact": _run_compact}[state["kind"]](state)


def _on_page(s, results):
    """The selected rows' numbers and columns of every result, one after another."""
    parts = []
    for i, r in enumerate(results):
        parts.append(r.selected_rows)
        parts.extend(r.selected_columns)
        s["sizes"][i] = len(parts[-1])
    end = sum(map(len, parts))
    np.concatenate(parts, out=s["page"][:end], casting="unsafe")
    s["page"][end:s["end"]] = 0
    s["end"] = end
    return s["sizes"], s["page"]


def _run_plan(s):
    return _on_page(s, [s["engine"].execute(s["plans"][0])])


def _run_batch(s):
    return _on_page(s, s["engine"].execute_batch(s["plans"])[0])


def _run_bundle(s):
    s["acc"].zero_()
    ops.bundle_exec(s["ops"], s["n"])
    return s["flags"], s["rev"], s["acc"]


def _q1_build(s):
    s["ht"].zero_()
    nd = s["dflags"].numel()
    ops.selection(s["dflags"], s[S.D_YEAR], "==", s["case"]["year"], "", nd)
    ops.build_keys_ht(s[S.D_DATEKEY], s["dflags"], nd, s["ht"], s["len"], s["min"])


def _run_filter(s):
    c, lo, n, flags, local = s["case"], s["lo"], s["n"], s["flags"], s["local"]
    _q1_build(s)
    ops.selection(local, lo[S.LO_DISCOUNT], ">=", c["disc_lo"], "", n)
    ops.selection(local, lo[S.LO_DISCOUNT], "<=", c["disc_hi"], "AND", n)
    ops.logical(flags, local, flags, ops.NONE, n)
    ops.selection(flags, lo[S.LO_QUANTITY], "<", c["qty"], "AND", n)
    ops.filter_join(lo[S.LO_ORDERDATE], flags, n, s["ht"], s["min"], s["max"])
    ops.perform_operation(s["rev"], lo[S.LO_EXTENDEDPRICE], lo[S.LO_DISCOUNT], flags, n, "*")
    s["acc"].zero_()
    ops.aggregate_operation(s["rev"], flags, n, s["acc"])
    return flags, s["rev"], s["acc"]


def _run_star(s):
    c, n, lo, flags = s["case"], s["n"], s["lo"], s["flags"]
    p, sup, d = s["part"], s["supplier"], s["ddate"]
    for t in (p, sup, d):
        t["ht"].zero_()
    ops.selection(p["flags"], p[S.P_CATEGORY], "==", c["category"], "", p["rows"])
    ops.build_key_vals_ht(p[S.P_PARTKEY], p[S.P_BRAND1], p["flags"], p["rows"], p["ht"], p["len"], p["min"])
    ops.selection(sup["flags"], sup[S.S_REGION], "==", c["region"], "", sup["rows"])
    ops.build_keys_ht(sup[S.S_SUPPKEY], sup["flags"], sup["rows"], sup["ht"], sup["len"], sup["min"])
    ops.build_key_vals_ht(d[S.D_DATEKEY], d[S.D_YEAR], d["flags"], d["rows"], d["ht"], d["len"], d["min"])
    flags.fill_(1)
    ops.full_join(lo[S.LO_PARTKEY], s["brand"], flags, n, p["ht"], p["min"], p["max"])
    ops.filter_join(lo[S.LO_SUPPKEY], flags, n, sup["ht"], sup["min"], sup["max"])
    ops.full_join(lo[S.LO_ORDERDATE], s["year"], flags, n, d["ht"], d["min"], d["max"])
    s["sums"].zero_()
    s["seen"].zero_()
    ops.group_by_aggregate([s["year"], s["brand"]], lo[S.LO_REVENUE], s["gmax"], s["gmin"], flags, n, 2, s["keys"],
                           s["sums"], s["seen"], s["prod"])
    ops.seen_to_flags(s["seen"], s["gflags"], s["prod"])
    return [flags, s["brand"], s["year"], *s["keys"], s["sums"], s["gflags"]]


def _run_compact(s):
    k = ops.count_true_flags(s["flags"], s["n"])
    ops.compact(s["flags"], s["ids"], s["count"], s["n"])
    for c, o in zip(s["cols"], s["out"]):
        ops.gather(c, s["ids"], k, o)
    return [k, s["count"], s["ids"], *s["out"]]


# --------------------------------------------------------- work and results

def work(case):
    n = case["rows"]
    if case["kind"] in ("plan", "batch"):
        pipes, dims = _pipes(case), DIMS[case["dims"]]
        used = {t for t, _ in pipes}
        cols = {c for t in used for c in FACT_COLUMNS[t]}
        dim = sum(4 * dims[d] * len(DIM_COLUMNS[d]) for d in {d for t in used for d in DIM_TABLES[t]})
        # a key test or an operand per column and row of each query
        return {"bytes": 4 * len(cols) * n + dim, "flops": sum(len(FACT_COLUMNS[t]) for t, _ in pipes) * n}
    if case["kind"] in ("bundle", "filter"):
        # four columns in, flags and the selected rows' products out
        sel = (case["disc_hi"] - case["disc_lo"] + 1) / 11 * min(1.0, max(0, case["qty"] - 1) / 50) / 7
        return {"bytes": int((16 + 1 + 4 * sel) * n), "flops": 6 * n}
    if case["kind"] == "star":
        # four columns in, flags, brands and years out
        return {"bytes": int((16 + 1 + 4 / 25 + 4 / 125) * n) + 12 * DIMS[case["dims"]]["part"], "flops": 5 * n}
    d = case["density"]
    return {"bytes": int((1 + 4 * d + 2 * 8 * d) * n), "flops": n}


def tolerance(case):
    return "exact"


def exact(case, seed):
    seed = int(seed)
    if case["kind"] in ("plan", "batch"):
        pipes, dims = _pipes(case), DIMS[case["dims"]]
        used = {t for t, _ in pipes}
        fact = _fact(sorted({c for t in used for c in FACT_COLUMNS[t]}), case["rows"], dims, seed)
        dim = {d: _dim(d, DIM_COLUMNS[d], dims, seed) for d in sorted({d for t in used for d in DIM_TABLES[t]})}
        out = [_exact_query(t, p, fact, dim) for t, p in pipes]
        page, all_of = np.zeros(ANSWER * len(pipes), np.int64), np.concatenate([c for a in out for c in a])
        page[:len(all_of)] = all_of
        return np.array([len(a[0]) for a in out]), page
    if case["kind"] in ("bundle", "filter"):
        n, dims = case["rows"], DIMS["sf100"]
        lo = _fact(FACT_COLUMNS["t1"], n, dims, seed)
        flags = torch.zeros(n, dtype=torch.uint8, device=DEV)
        rev = torch.zeros(n, dtype=torch.int32, device=DEV)
        flags[:] = (lo[S.LO_DISCOUNT] >= case["disc_lo"]) & (lo[S.LO_DISCOUNT] <= case["disc_hi"]) & \
            (lo[S.LO_QUANTITY] < case["qty"]) & (lo[S.LO_ORDERDATE] // 10000 == case["year"])
        at = flags.nonzero().squeeze(1)
        rev[at] = lo[S.LO_EXTENDEDPRICE][at] * lo[S.LO_DISCOUNT][at]
        return flags, rev, rev.long().sum().reshape(1)
    if case["kind"] == "star":
        n, dims = case["rows"], DIMS[case["dims"]]
        lo = _fact(FACT_COLUMNS["t2"], n, dims, seed)
        part = _dim("part", (S.P_CATEGORY, S.P_BRAND1), dims, seed)
        sup = _dim("supplier", (S.S_REGION,), dims, seed)
        brand, year = (torch.zeros(n, dtype=torch.int32, device=DEV) for _ in range(2))
        flags = torch.zeros(n, dtype=torch.uint8, device=DEV)
        for a in range(0, n, 1 << 26):
            x = slice(a, a + (1 << 26))
            pk, sk = lo[S.LO_PARTKEY][x].long() - 1, lo[S.LO_SUPPKEY][x].long() - 1
            hit = part[S.P_CATEGORY][pk] == case["category"]
            brand[x] = torch.where(hit, part[S.P_BRAND1][pk], 0)
            hit &= sup[S.S_REGION][sk] == case["region"]
            year[x] = torch.where(hit, lo[S.LO_ORDERDATE][x] // 10000, 0)
            flags[x] = hit
        bmin, bmax = int(part[S.P_BRAND1].min()), int(part[S.P_BRAND1].max())
        at = flags.nonzero().squeeze(1)
        slot = (year[at].long() - 1992) + 7 * (brand[at].long() - bmin)
        prod = 7 * (bmax - bmin + 1)
        sums = torch.zeros(prod, dtype=torch.int64, device=DEV).index_add_(0, slot, lo[S.LO_REVENUE][at].long())
        seen = torch.zeros(prod, dtype=torch.bool, device=DEV).index_fill_(0, slot, True)
        i = torch.arange(prod, device=DEV)
        keys = [torch.where(seen, 1992 + i % 7, 0).int(), torch.where(seen, bmin + i // 7, 0).int()]
        return [flags, brand, year, *keys, sums, seen.to(torch.uint8)]
    flags, cols = _compact_inputs(case, seed)
    at = flags.nonzero().squeeze(1)
    k = at.numel()
    ids, *out = (torch.zeros(case["rows"], dtype=torch.int32, device=DEV) for _ in range(3))
    ids[:k] = at
    for c, o in zip(cols, out):
        o[:k] = c[at]
    return [k, torch.tensor([k], dtype=torch.int32), ids, *out]


def _keep(col, p, points):
    """The rows of a dimension a predicate keeps."""
    c = col[points[p[0]]]
    if p[0] in ("city2", "mfgr2"):
        return (c == p[1]) | (c == p[2])
    if p[0] in ("year_range", "year_range_and", "brand_range"):
        return (c >= p[1]) & (c <= p[2])
    return c == p[1]


DATE_BY = {"year": S.D_YEAR, "year_range": S.D_YEAR, "year_range_and": S.D_YEAR, "yearmonthnum": S.D_YEARMONTHNUM}
PLACE_BY = {"region": S.S_REGION, "nation": S.S_NATION, "city": S.S_CITY, "city2": S.S_CITY}
PART_BY = {"category": S.P_CATEGORY, "brand": S.P_BRAND1, "brand_range": S.P_BRAND1, "mfgr2": S.P_MFGR}


def _exact_query(t, p, fact, dim):
    """Rows and columns of one query's answer, from a plain loop over slices of the fact table."""
    dd = dim["ddate"]
    at_day = torch.zeros(int(dd[S.D_DATEKEY].max()) + 1, dtype=torch.int64, device=DEV)
    at_day[dd[S.D_DATEKEY].long()] = torch.arange(len(dd[S.D_DATEKEY]), device=DEV)
    keep, joins, keys = {}, {}, []  # rows kept, fact key column, (dimension, column) of each group key
    if t == "t1":
        keep["ddate"] = _keep(dd, p["date"], DATE_BY)
    elif t == "t2":
        keep = {"part": _keep(dim["part"], p["part"], PART_BY), "supplier": dim["supplier"][S.S_REGION] == p["s_region"]}
        keys = [("ddate", S.D_YEAR), ("part", S.P_BRAND1)]
    elif t == "t3":
        keep = {"customer": _keep(dim["customer"], p["cust"], PLACE_BY), "supplier": _keep(dim["supplier"], p["supp"], PLACE_BY),
                "ddate": _keep(dd, p["date"], DATE_BY)}
        g = S.S_NATION if p["group"] == "nation" else S.S_CITY
        keys = [("customer", g), ("supplier", g), ("ddate", S.D_YEAR)]
    else:
        keep = {"customer": dim["customer"][S.C_REGION] == p["c_region"], "supplier": dim["supplier"][S.S_REGION] == p["s_region"],
                "part": _keep(dim["part"], ("mfgr2", p["mfgr"][0], p["mfgr"][1]), PART_BY)}
        keys = [("ddate", S.D_YEAR), ("customer", S.C_NATION)]
    joins = {"customer": S.LO_CUSTKEY, "supplier": S.LO_SUPPKEY, "part": S.LO_PARTKEY, "ddate": S.LO_ORDERDATE}
    lo = [int(dim[d][c].min()) for d, c in keys]
    size = [int(dim[d][c].max()) - m + 1 for (d, c), m in zip(keys, lo)]
    prod = math.prod(size)
    sums = torch.zeros(prod, dtype=torch.int64, device=DEV)
    seen = torch.zeros(prod, dtype=torch.bool, device=DEV)
    n = fact[S.LO_ORDERDATE].numel()
    for a in range(0, n, 1 << 26):
        f = {c: v[a:a + (1 << 26)] for c, v in fact.items()}

        def row_of(d):
            return at_day[f[S.LO_ORDERDATE].long()] if d == "ddate" else f[joins[d]].long() - 1
        hit = torch.ones(f[S.LO_ORDERDATE].numel(), dtype=torch.bool, device=DEV)
        for d, k in keep.items():
            hit &= k[row_of(d)]
        if t == "t1":
            q = f[S.LO_QUANTITY]
            hit &= (f[S.LO_DISCOUNT] >= p["disc"][0]) & (f[S.LO_DISCOUNT] <= p["disc"][1])
            hit &= q < p["qty"][1] if p["qty"][0] == "lt" else (q >= p["qty"][1]) & (q <= p["qty"][2])
        at = hit.nonzero().squeeze(1)
        f = {c: v[at] for c, v in f.items()}
        if t == "t1":
            v = f[S.LO_EXTENDEDPRICE].long() * f[S.LO_DISCOUNT]
        else:
            v = f[S.LO_REVENUE].long() - (f[S.LO_SUPPLYCOST] if t == "t4" else 0)
        slot, mult = torch.zeros(at.numel(), dtype=torch.int64, device=DEV), 1
        for (d, c), m, w in zip(keys, lo, size):
            slot += (dim[d][c][row_of(d)].long() - m) * mult
            mult *= w
        sums.index_add_(0, slot, v)
        seen[slot] = True
    if t == "t1":
        return [np.zeros(1, np.int64), sums.cpu().numpy()]
    rows = seen.nonzero().squeeze(1)
    out, rest = [rows.cpu().numpy()], rows
    for m, w in zip(lo, size):
        out.append((m + rest % w).int().cpu().numpy())
        rest = rest // w
    return out + [sums[rows].cpu().numpy()]
