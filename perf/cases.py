"""The queries whose time this repository answers for, as its users run them.

Every case is one pass of a compiled plan over tables that stay in device
memory, through the public entry points of ``dogqc_amd.runtime``.  What a
program has in hand before the call is made by ``prepare``: the columns, the
compiled plan, its input binding and the capacities that ``runtime.Feedback``
learned from an earlier run of the same query (the way HipCompiler.execute()
and the serving loop size repeated queries).  A pass is one of

  run      runtime.run: workspace, plan, status, and the result columns on the
           host (the call of HipCompiler.execute(); results of a few rows);
  enqueue  runtime.enqueue into a workspace the program keeps, results read
           where they lie by the torch code that follows on the same stream;
  graph    the same enqueue captured once with runtime.Graph and replayed.

Plans return rows in no particular order, as the reference's do, so a pass
ends with what a program does to them: sorts few rows, or places many by key.
(A few calls of torch or numpy on the result; they read no input table.)

The data follows the distributions of workloads.generate and tpch.generate,
made on the device from the seed.
"""
import ctypes
import functools

import numpy as np
import torch

from dogqc_amd import planlib, runtime as rt, tpch, workloads

DEV = "cuda"


def listed():
    return [
        # scan, two maps, eight aggregates into six groups: the size of the
        # workload's own definition, where launches and host work weigh most
        {"name": "pricing_1m", "kind": "pricing", "rows": 1000000, "how": "run"},
        # the same over a table that has to stream from memory
        {"name": "pricing_64m", "kind": "pricing", "rows": 67108864, "how": "run"},
        # PK-FK join and group-by at the size of a smoke test, replayed
        {"name": "lookup_80k", "kind": "lookup", "plan": "c1", "dim": 20000, "fact": 80000, "how": "graph"},
        # the same at its full size, the benchmark's default (lane refill)
        {"name": "lookup_6m", "kind": "lookup", "plan": "c1_refill", "dim": 1500000, "fact": 6000000,
         "how": "enqueue"},
        # expanding join on a Zipf-skewed key, match lists balanced over lanes
        {"name": "expand_16m", "kind": "expand", "build": 1000000, "probe": 16000000, "how": "enqueue"},
        # star join with a LIKE filter and two group-bys over a temp table, full size
        {"name": "star_60m", "kind": "star", "sales": 60000000, "item": 2000000, "cust": 200000, "how": "enqueue"},
        # the same over a small prefix, as the serving mix draws them; odd sizes
        {"name": "star_5m", "kind": "star", "sales": 4615385, "item": 153847, "cust": 15385, "how": "enqueue"},
        # TPC-H Q1, pricing summary: FLOAT columns, CHAR group keys
        {"name": "q1_sf10", "kind": "tpch", "query": 1, "sf": 10.0, "how": "run"},
        # TPC-H Q3: two joins, lane refill, a group per order
        {"name": "q3_sf1", "kind": "tpch", "query": 3, "sf": 1.0, "how": "enqueue"},
        # TPC-H Q10, the reference's published query: string group keys
        {"name": "q10_sf1", "kind": "tpch", "query": 10, "sf": 1.0, "how": "enqueue"},
        # TPC-H Q13: LIKE over order comments, outer join, group-by over a group-by
        {"name": "q13_sf1", "kind": "tpch", "query": 13, "sf": 1.0, "how": "run"},
        # TPC-H Q18: a group per order over all lineitems, then three joins
        {"name": "q18_sf1", "kind": "tpch", "query": 18, "sf": 1.0, "how": "run"},
    ]


def draw(rng):
    def spread(lo, hi):
        return lo * (hi / lo) ** rng.random()

    kind = rng.choice(["pricing", "lookup", "expand", "star", "tpch", "tpch"])
    if kind == "pricing":
        return {"kind": kind, "rows": int(spread(2e4, 6e7)), "how": "run"}
    if kind == "lookup":
        fact = int(spread(5e4, 2e7))
        return {"kind": kind, "plan": rng.choice(["c1", "c1_refill"]), "dim": int(fact / rng.uniform(2, 8)),
                "fact": fact, "how": "graph" if fact < 1000000 else "enqueue"}
    if kind == "expand":
        probe = int(spread(1e5, 1.6e7))
        return {"kind": kind, "build": int(probe / rng.uniform(12, 24)), "probe": probe, "how": "enqueue"}
    if kind == "star":
        sales = int(spread(3e5, 5e7))
        return {"kind": kind, "sales": sales, "item": int(sales / rng.uniform(20, 40)),
                "cust": int(sales / rng.uniform(200, 400)), "how": "enqueue"}
    query = rng.choice([1, 3, 10, 13, 18])
    return {"kind": kind, "query": query, "sf": round(spread(0.1, 2.0), 4),
            "how": "enqueue" if query in (3, 10) else "run"}


# ------------------------------------------------------------------ columns

class Gen(object):
    """Random columns on the device, from a seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def ints(self, lo, hi, n, dtype=torch.int32):
        """Uniform over lo..hi, both included."""
        return torch.randint(lo, hi + 1, (n,), generator=self.g, device=DEV, dtype=torch.int64).to(dtype)

    def decimals(self, lo, hi, n, div=100.0, dtype=torch.float64):
        return (self.ints(lo, hi, n, torch.int64).double() / div).to(dtype)

    def perm(self, n):
        return torch.randperm(n, generator=self.g, device=DEV).to(torch.int32)

    def uniform(self, n):
        return torch.rand(n, generator=self.g, device=DEV, dtype=torch.float64)


def _ymd(days):
    """yyyymmdd of days since 1992-01-01, from a table of the years 1992..1999."""
    d = np.arange(np.datetime64("1992-01-01"), np.datetime64("2000-01-01"))
    y, m = d.astype("datetime64[Y]"), d.astype("datetime64[M]")
    t = (y.astype(int) + 1970) * 10000 + ((m - y).astype(int) + 1) * 100 + (d - m).astype(int) + 1
    return torch.from_numpy(t.astype(np.int32)).to(DEV)[days]


def _tokens(words, picks, last):
    """A STRING column's char heap and the end of every token in it: the
    words picked, each followed by a space unless it is its row's last."""
    raw = [w.encode() for w in words]
    width = max(len(w) for w in raw) + 1
    table = torch.from_numpy(np.frombuffer(b"".join(w.ljust(width) for w in raw), dtype=np.uint8).copy())
    table = table.reshape(len(raw), width).to(DEV)
    lens = torch.tensor([len(w) for w in raw], device=DEV)[picks] + (~last).long()
    ends = torch.cumsum(lens, 0)
    tok = torch.repeat_interleave(torch.arange(len(picks), device=DEV), lens)
    at = torch.arange(int(ends[-1]), device=DEV) - (ends - lens)[tok]
    return table[picks[tok], at].contiguous(), ends


def _text(gen, words, n, lo, hi, plant=None, every=0):
    """n texts of lo..hi words; every `every`-th holds the two words of `plant` apart."""
    words = list(words)
    counts = gen.ints(lo, hi, n, torch.int64)
    if plant:
        hit = torch.arange(n, device=DEV) % every == every // 2
        counts = torch.where(hit, torch.clamp(counts, min=4), counts)
    ends = torch.cumsum(counts, 0)
    total = int(ends[-1])
    picks = gen.ints(0, len(words) - 1, total, torch.int64)
    if plant:
        words += list(plant)
        first = (ends - counts)[hit]
        picks[first] = len(words) - 2
        picks[first + 2] = len(words) - 1
    last = torch.zeros(total, dtype=torch.bool, device=DEV)
    last[ends - 1] = True
    chars, tokEnds = _tokens(words, picks, last)
    offs = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    offs[1:] = tokEnds[ends - 1]
    return offs, chars


def _choice(values, picks):
    """A STRING column of one of `values` per row."""
    chars, ends = _tokens(values, picks, torch.ones(len(picks), dtype=torch.bool, device=DEV))
    offs = torch.zeros(len(picks) + 1, dtype=torch.int64, device=DEV)
    offs[1:] = ends
    return offs, chars


def _pattern(form, fields):
    """A STRING column of fixed-width rows: `form` with its runs of '0'
    replaced by the decimal digits of `fields`, in order."""
    n = len(fields[0])
    out = torch.tensor(list(form.encode()), dtype=torch.uint8, device=DEV).repeat(n, 1)
    runs, k = [], 0
    while k < len(form):
        if form[k] == "0":
            e = k
            while e < len(form) and form[e] == "0":
                e += 1
            runs.append((k, e))
            k = e
        else:
            k += 1
    for (a, b), f in zip(runs, fields):
        f = f.long()
        for p in range(b - 1, a - 1, -1):
            out[:, p] = (f % 10 + 48).to(torch.uint8)
            f = f // 10
    offs = torch.arange(n + 1, device=DEV, dtype=torch.int64) * len(form)
    return offs, out.reshape(-1)


def _pricing(case, gen):
    n = case["rows"]
    return {"cfg0": (n, {"g1": gen.ints(0, 2, n, torch.int8), "g2": gen.ints(0, 1, n, torch.int8),
                         "qty": gen.ints(1, 50, n), "price": gen.decimals(90000, 10500000, n),
                         "disc": gen.decimals(0, 10, n), "tax": gen.decimals(0, 8, n),
                         "date": _ymd(gen.ints(0, 2556, n, torch.int64))})}


def _lookup(case, gen):
    nd, nf = case["dim"], case["fact"]
    return {"dim": (nd, {"d_key": gen.perm(nd), "d_cat": gen.ints(48, 52, nd, torch.int8),
                         "d_seg": gen.ints(0, 999999, nd)}),
            "fact": (nf, {"f_fk": gen.ints(0, nd - 1, nf), "f_price": gen.decimals(90000, 10500000, nf),
                          "f_disc": gen.decimals(0, 10, nf), "f_date": _ymd(gen.ints(0, 2556, nf, torch.int64))})}


def _expand(case, gen):
    nb, n = case["build"], case["probe"]
    nvals = min(100000, nb)
    cdf = np.cumsum(1.0 / np.arange(1, nvals + 1, dtype=np.float64))
    rank = torch.searchsorted(torch.from_numpy(cdf / cdf[-1]).to(DEV), gen.uniform(nb), right=True).clamp(max=nvals - 1)
    return {"build": (nb, {"b_key": gen.perm(nvals)[rank], "b_pay": gen.ints(1, (1 << 20) - 1, nb, torch.int64)}),
            "probe": (n, {"p_key": gen.ints(0, 2 * nvals - 1, n), "p_f": gen.ints(0, 99, n),
                          "p_pay": gen.ints(1, (1 << 20) - 1, n, torch.int64)})}


def _star(case, gen):
    ns, ni, nc = case["sales"], case["item"], case["cust"]
    w, words = workloads.TEXT_WIDTH, workloads.VOCAB
    width = max(len(v) for v in words) + 1
    table = np.zeros((len(words), width), dtype=np.uint8)
    lens = np.array([len(v) for v in words])
    for i, v in enumerate(words):
        table[i, :len(v)] = np.frombuffer(v.encode(), dtype=np.uint8)
    table, lens = torch.from_numpy(table).to(DEV), torch.from_numpy(lens).to(DEV)
    text = torch.full((ni, w + width), 32, dtype=torch.uint8, device=DEV)
    at = torch.zeros(ni, dtype=torch.int64, device=DEV)
    for _ in range(5):
        pick = gen.ints(0, len(words) - 1, ni, torch.int64)
        for c in range(width):
            ch = table[pick, c]
            text.scatter_(1, (at + c)[:, None], torch.where(ch == 0, 32, ch).to(torch.uint8)[:, None])
        at += lens[pick] + 1
    chars = text[:, :w].contiguous().reshape(-1)
    offs = torch.arange(ni + 1, device=DEV, dtype=torch.int64) * w
    return {"sales": (ns, {"s_item": gen.ints(0, ni - 1, ns), "s_cust": gen.ints(0, nc - 1, ns),
                           "s_nation": gen.ints(0, 24, ns), "s_qty": gen.ints(1, 50, ns),
                           "s_price": gen.decimals(90000, 10500000, ns)}),
            "item": (ni, {"i_key": gen.perm(ni), "i_text": (offs, chars)}),
            "cust": (nc, {"c_key": gen.perm(nc), "c_year": gen.ints(1992, 1998, nc)}),
            "nation": (25, {"n_key": gen.perm(25)})}


def _tpch(case, gen):
    """The columns of lineitem, orders, customer and nation that the query
    reads; keys, dates and text as tpch.generate makes them."""
    sf, query = case["sf"], case["query"]
    nC, nO = max(6, int(round(150000 * sf))), max(8, int(round(1500000 * sf)))
    i = torch.arange(nO, device=DEV)
    okey = (i // 8) * 32 + i % 8 + 1
    odays = gen.ints(0, 2405, nO, torch.int64)
    with_orders = torch.arange(1, nC + 1, device=DEV)
    with_orders = with_orders[with_orders % 3 != 0]
    orders = {"o_orderkey": okey.int(),
              "o_custkey": with_orders[gen.ints(0, len(with_orders) - 1, nO, torch.int64)].int(),
              "o_orderdate": _ymd(odays), "o_totalprice": gen.decimals(90000, 40000000, nO, dtype=torch.float32),
              "o_shippriority": torch.zeros(nO, dtype=torch.int32, device=DEV)}
    if query == 13:
        orders["o_comment"] = _text(gen, tpch.WORDS, nO, 3, 10, ("special", "requests"), 50)
    custkey = torch.arange(1, nC + 1, device=DEV, dtype=torch.int32)
    cnat = gen.ints(0, 24, nC)
    cust = {"c_custkey": custkey, "c_nationkey": cnat,
            "c_acctbal": gen.decimals(-99999, 999999, nC, dtype=torch.float32)}
    if query == 3:
        cust["c_mktsegment"] = _choice(tpch.SEGMENTS, gen.ints(0, 4, nC, torch.int64))
    if query in (10, 18):
        cust["c_name"] = _pattern("Customer#000000000", [custkey])
    if query == 10:
        cust["c_address"] = _text(gen, tpch.WORDS, nC, 1, 3)
        cust["c_comment"] = _text(gen, tpch.WORDS, nC, 4, 12)
        cust["c_phone"] = _pattern("00-000-000-0000", [cnat + 10, gen.ints(100, 999, nC), gen.ints(100, 999, nC),
                                                       gen.ints(1000, 9999, nC)])
    nation = {"n_nationkey": torch.arange(25, device=DEV, dtype=torch.int32),
              "n_name": _choice([n for n, _ in tpch.NATIONS], torch.arange(25, device=DEV))}
    tables = {"orders": (nO, orders), "customer": (nC, cust), "nation": (25, nation)}
    if query != 13:
        lo = torch.repeat_interleave(i, gen.ints(1, 7, nO, torch.int64))
        n = len(lo)
        ship = odays[lo] + gen.ints(1, 121, n, torch.int64)
        shipdate, receipt = _ymd(ship), _ymd(ship + gen.ints(1, 30, n, torch.int64))
        qty = gen.ints(1, 50, n)
        flag = torch.where(receipt <= tpch.CUTOFF, torch.where(gen.ints(0, 1, n) == 0, ord("R"), ord("A")), ord("N"))
        tables["lineitem"] = (n, {
            "l_orderkey": okey[lo].int(), "l_quantity": qty,
            "l_extendedprice": (qty * gen.decimals(90000, 200000, n)).float(),
            "l_discount": gen.decimals(0, 10, n, dtype=torch.float32), "l_tax": gen.decimals(0, 8, n, dtype=torch.float32),
            "l_returnflag": flag.to(torch.int8),
            "l_linestatus": torch.where(shipdate > tpch.CUTOFF, ord("O"), ord("F")).to(torch.int8),
            "l_shipdate": shipdate})
    return tables


TABLES = {"pricing": _pricing, "lookup": _lookup, "expand": _expand, "star": _star, "tpch": _tpch}


def plan_name(case):
    if case["kind"] == "tpch":
        return "tpch%d" % case["query"]
    return {"pricing": "c0", "expand": "c2_pushdown", "star": "c3_refill"}.get(case["kind"]) or case["plan"]


# -------------------------------------------------------------- preparation

class Resident(object):
    """Device memory of a tensor, in the form the runtime's store takes."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = ctypes.c_void_p(tensor.data_ptr())
        self.nbytes = tensor.numel() * tensor.element_size()


class TorchStream(object):
    """torch's current stream, for runtime calls."""

    def __init__(self):
        self.handle = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@functools.lru_cache(maxsize=None)
def _module(name):
    return rt.PlanModule(planlib.translate(name).compile(name))


DTYPES = {"int32_t": torch.int32, "uint32_t": torch.int32, "int64_t": torch.int64, "double": torch.float64,
          "int8_t": torch.int8, "dqc::str_offs": torch.int64}


def _views(ws, columns, offsets, count):
    """Result columns where they lie in the workspace (a string is its two offsets)."""
    out = {}
    for c, off in zip(columns, offsets):
        dt = DTYPES[c["ctype"]]
        per = 2 if c["ctype"] == "dqc::str_offs" else 1
        size = torch.empty(0, dtype=dt).element_size() * per * count
        v = ws[off:off + size].view(dt)
        out[c["name"]] = v.reshape(count, 2) if per == 2 else v
    return out


def prepare(case, seed):
    tables = TABLES[case["kind"]](case, Gen(seed))
    module = _module(plan_name(case))
    store = {}
    for c in module.desc["columns"]:
        col = tables[c["table"]][1][c["attr"]]
        if c["part"] is not None:
            col = col[0 if c["part"] == "offset" else 1]
        store[(c["table"], c["attr"], c["part"])] = Resident(col)
    s = {"case": case, "module": module, "store": store, "tables": tables, "stream": TorchStream()}
    s["inputs"] = rt.BoundInputs(module, None, store=store, rows={t: n for t, (n, _) in tables.items()})
    # the sizes an earlier run of this query measured
    torch.cuda.synchronize()
    feedback = rt.Feedback()
    rt.run(module, s["inputs"], rt.newTuning(), s["stream"], feedback=feedback).release()
    s["tuning"] = rt.newTuning()
    feedback.apply(module, s["inputs"], s["tuning"])
    # (retries, if the sizes still change with them, are kept in the tuning)
    rt.run(module, s["inputs"], s["tuning"], s["stream"]).release()
    if case["how"] == "run":
        return s
    lay = rt.layout(module, s["inputs"], s["tuning"])
    s["ws"] = Resident(torch.zeros(int(lay.ws_bytes), dtype=torch.uint8, device=DEV))
    rec = feedback.records[feedback.key(module)]
    s["result"] = _views(s["ws"].tensor, module.desc["result"], list(lay.result_offset), rec["result"])
    s["temps"] = {t["name"]: _views(s["ws"].tensor, t["columns"], [lay.temp_offset[c["slot"]] for c in t["columns"]],
                                    rec["temps"][t["index"]]) for t in module.desc["temps"]}
    if case["how"] == "graph":
        torch.cuda.synchronize()
        s["capture"] = rt.Stream()
        s["graph"] = rt.Graph(module, s["inputs"], s["tuning"], s["ws"], s["capture"])
    return s


# --------------------------------------------------------------------- pass

def _byKey(key, size, cols):
    """Columns as arrays indexed by an integer key (absent keys 0)."""
    key = key.long()
    return {n: torch.zeros((size,) + v.shape[1:], dtype=v.dtype, device=v.device).index_copy_(0, key, v)
            for n, v in cols.items()}


def _firstRows(cols, by, n):
    """The first n rows in the order of the columns `by` (the most
    significant last, as for lexsort); missing rows 0."""
    order = np.lexsort(by)[:n]
    out = {}
    for name, v in cols.items():
        v = v.view(np.uint64).reshape(-1, 2) if v.dtype.fields else v
        out[name] = np.zeros((n,) + v.shape[1:], dtype=v.dtype)
        out[name][:len(order)] = v[order]
    return out


def orderRow(okey):
    """Row of orders that holds an order key (runs of 8 keys per 32)."""
    return (okey // 32) * 8 + okey % 32 - 1


def run(s):
    case = s["case"]
    if case["how"] == "run":
        ex = rt.run(s["module"], s["inputs"], s["tuning"], s["stream"])
        c = ex.columns()
        ex.release()
        if case["kind"] == "pricing":
            return _firstRows(c, [c["g2"], c["g1"]], 6)
        if case["query"] == 1:
            return _firstRows(c, [c["l_linestatus"], c["l_returnflag"]], 4)
        if case["query"] == 13:
            return _firstRows(c, [c["c_count"]], 64)
        return _firstRows(c, [c["o_orderkey"], c["o_orderdate"], -c["o_totalprice"]], 100)
    if case["how"] == "graph":
        s["graph"].launch(s["stream"])
    else:
        rt.enqueue(s["module"], s["inputs"], s["tuning"], s["ws"], s["stream"])
    r = s["result"]
    if case["kind"] == "expand":
        return {"cnt": r["cnt"], "sum_prod": r["sum_prod"]}
    if case["kind"] == "lookup":
        return _byKey(r["d_key"], case["dim"], {"revenue": r["revenue"]})
    if case["kind"] == "star":
        t = s["temps"]["c3_by_nation_year"]
        return {"item": _byKey(r["i_key"], case["item"], {n: r[n] for n in ("sum_qty", "revenue", "cnt")}),
                "nation_year": _byKey(t["n_key"] * 7 + (t["c_year"] - 1992), 175,
                                      {n: t[n] for n in ("sum_qty", "revenue", "cnt")})}
    if case["query"] == 3:
        return _byKey(orderRow(r["l_orderkey"]), s["tables"]["orders"][0], r)
    return _byKey(r["c_custkey"], s["tables"]["customer"][0] + 1, r)


# --------------------------------------------------------------------- work

def work(case):
    k = case["kind"]
    if k == "pricing":
        return {"bytes": 34.0 * case["rows"], "flops": 11.0 * case["rows"]}
    if k == "lookup":
        return {"bytes": 24.0 * case["fact"] + 5.0 * case["dim"] + 8.0 * case["dim"], "flops": 0.1 * case["fact"]}
    if k == "expand":
        return {"bytes": 16.0 * case["probe"] + 12.0 * case["build"], "flops": 1.0 * case["probe"]}
    if k == "star":
        return {"bytes": 24.0 * case["sales"] + 67.0 * case["item"] + 8.0 * case["cust"] + 16.0 * case["item"],
                "flops": 0.2 * case["sales"]}
    sf = case["sf"]
    lines, orders, cust = 6.0e6 * sf, 1.5e6 * sf, 1.5e5 * sf
    if case["query"] == 1:      # quantity, price, discount, tax, two flags, shipdate
        return {"bytes": 22.0 * lines, "flops": 11.0 * lines}
    if case["query"] == 3:      # orderkey, shipdate, price, discount; three order columns and a priority; segment
        return {"bytes": 16.0 * lines + 16.0 * orders + 21.0 * cust, "flops": 0.5 * lines}
    if case["query"] == 10:     # orderkey, flag, price, discount; three order columns; names, texts and phones
        return {"bytes": 13.0 * lines + 12.0 * orders + 170.0 * cust, "flops": 0.3 * lines}
    if case["query"] == 13:     # orderkey, custkey, offsets and about 47 bytes of comment
        return {"bytes": 63.0 * orders + 4.0 * cust, "flops": orders}
    return {"bytes": 8.0 * lines + 16.0 * orders + 30.0 * cust, "flops": lines}   # Q18; lineitem is one input


# -------------------------------------------------------------------- exact

def _sums(n, at, **cols):
    return {k: torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, at, v) for k, v in cols.items()}


def exact(case, seed):
    if case["kind"] == "expand" or case.get("query") == 13:
        return None      # whole numbers only
    tables = {t: c for t, (_, c) in TABLES[case["kind"]](case, Gen(seed)).items()}
    if case["kind"] == "pricing" or case.get("query") == 1:
        if case["kind"] == "pricing":
            t = tables["cfg0"]
            keep = t["date"] <= 19981110
            names, code = ("g1", "g2", "qty"), t["g1"].long() * 256 + t["g2"].long()
            price, disc, tax = t["price"], t["disc"], t["tax"]
        else:
            t = tables["lineitem"]
            keep = t["l_shipdate"] <= 19980902
            names = ("l_returnflag", "l_linestatus", "l_quantity")
            code = t["l_returnflag"].long() * 256 + t["l_linestatus"].long()
            price, disc, tax = (t["l_" + c].double() for c in ("extendedprice", "discount", "tax"))
        qty = t[names[2]].double()
        code, qty, price, disc, tax = (x[keep] for x in (code, qty, price, disc, tax))
        groups, at = torch.unique(code, return_inverse=True)
        n = len(groups)
        dp = price * (1.0 - disc)
        s = _sums(n, at, qty=qty, price=price, disc=disc, dp=dp, charge=dp * (1.0 + tax), cnt=torch.ones_like(qty))
        return {names[0]: None, names[1]: None, "sum_qty": s["qty"], "sum_base_price": s["price"],
                "sum_disc_price": s["dp"], "sum_charge": s["charge"], "avg_qty": s["qty"] / s["cnt"],
                "avg_price": s["price"] / s["cnt"], "avg_disc": s["disc"] / s["cnt"], "count_order": None}
    if case["kind"] == "lookup":
        d, f = tables["dim"], tables["fact"]
        chosen = torch.zeros(case["dim"], dtype=torch.bool, device=DEV)
        chosen[d["d_key"][d["d_cat"] == ord("2")].long()] = True
        keep = (f["f_date"] >= 19950101) & (f["f_date"] < 19960101) & chosen[f["f_fk"].long()]
        return _sums(case["dim"], f["f_fk"].long()[keep], revenue=(f["f_price"] * (1.0 - f["f_disc"]))[keep])
    if case["kind"] == "star":
        offs, chars = tables["item"]["i_text"]
        text, word = chars.reshape(case["item"], -1), workloads.C3_WORD.encode()
        hit = torch.zeros(case["item"], dtype=torch.bool, device=DEV)
        for a in range(text.shape[1] - len(word) + 1):
            m = torch.ones_like(hit)
            for c, ch in enumerate(word):
                m &= text[:, a + c] == ch
            hit |= m
        green = torch.zeros_like(hit)
        green[tables["item"]["i_key"].long()] = hit
        year = torch.zeros(case["cust"], dtype=torch.int64, device=DEV)
        year[tables["cust"]["c_key"].long()] = tables["cust"]["c_year"].long()
        f = tables["sales"]
        item = f["s_item"].long()
        keep = green[item]
        ny = f["s_nation"].long() * 7 + year[f["s_cust"].long()] - 1992
        return {k: dict(_sums(n, at[keep], sum_qty=f["s_qty"][keep].double(), revenue=f["s_price"][keep]), cnt=None)
                for k, n, at in (("item", case["item"], item), ("nation_year", 175, ny))}
    # Q3, Q10 and Q18: sums per order and per customer
    li, od, cu = tables["lineitem"], tables["orders"], tables["customer"]
    row, nO, nC = orderRow(li["l_orderkey"].long()), len(od["o_orderkey"]), len(cu["c_custkey"])
    if case["query"] == 18:
        qty = _sums(nO, row, q=li["l_quantity"].double())["q"]
        big = (qty > 300).nonzero()[:, 0].cpu()
        c = {"o_totalprice": od["o_totalprice"].double().cpu()[big].numpy(), "quantity": qty.cpu()[big].numpy()}
        got = _firstRows(c, [big.numpy(), od["o_orderdate"].cpu()[big].numpy(), -c["o_totalprice"]], 100)
        return dict({n: None for n in ("c_name", "c_custkey", "o_orderkey", "o_orderdate")}, **got)
    rev = li["l_extendedprice"].double() * (1.0 - li["l_discount"].double())
    date, cust = od["o_orderdate"], od["o_custkey"].long()
    if case["query"] == 3:
        offs, chars = cu["c_mktsegment"]
        building = torch.zeros(nC + 1, dtype=torch.bool, device=DEV)
        building[1:] = chars[offs[:-1]] == ord("B")      # the only segment with that initial
        keep = (li["l_shipdate"] > 19950315) & ((date < 19950315) & building[cust])[row]
        return dict({n: None for n in ("l_orderkey", "o_orderdate", "o_shippriority")},
                    **_sums(nO, row[keep], revenue=rev[keep]))
    keep = (li["l_returnflag"] == ord("R")) & ((date >= 19931001) & (date < 19940101))[row]
    at = cust[row[keep]]
    bal = torch.zeros(nC + 1, dtype=torch.float64, device=DEV)
    bal[at] = cu["c_acctbal"].double()[at - 1]
    names = ("c_custkey", "c_name", "c_phone", "n_name", "c_address", "c_comment")
    return dict({n: None for n in names}, c_acctbal=bal, **_sums(nC + 1, at, revenue=rev[keep]))
