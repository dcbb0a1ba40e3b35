"""Performance cases of the numerical-agreement verdict.

A case is one verdict, or one call over several tensor pairs, as a harness that
judges operator outputs issues it: the pair already lies in device memory, the
call goes through a public entry point, and the record (or the meta dict built
from it) is the result.

Keys of a case:

* ``entry``   ``tensors``  ``verdict._compare_tensors`` (the drop-in, one pair)
              ``record``   ``verdict.verdict_record`` (the full device record)
              ``outputs``  ``verdict._compare_outputs`` (a nested output)
              ``pair``     ``kvv_verdict`` of the C library, issued asynchronously
              ``batch``    ``kvv_verdict_batch`` of the C library, likewise
* ``dtype``, ``rows``, ``cols``: the pair's element type and logical shape
* ``layout``  ``contiguous``  both tensors row-major
              ``pitched``     both with a row pitch of ``cols + pad``
              ``transposed``  the reference is the transposed view of a (cols, rows) tensor
              ``heads``       the reference is a (batch, seq, heads, cols) tensor viewed as
                              (batch, heads, seq, cols)
              ``sliced``      the reference is columns 1.. of a (rows, cols + 1) tensor
* ``data``    ``noise``      N(0, 1) against itself plus N(0, 1e-6), 0.1 % pushed by 1e-3..1e-1
              ``steps``      N(0, std), a fraction ``moved`` of the codes one step away, 0.01 % three
              ``nonfinite``  U(-60000, 60000) with 0.05 % NaN and 0.05 % Inf on both sides, 17 breaks
              ``integers``   the type's range, ``changed`` positions differ
* ``policy``  ``strict``, ``tolerant`` (near-zero diagnostics for 16-bit floats) or ``cosine``
"""

import ctypes
import math

import numpy as np
import torch

from kernelverse_amd import _lib, verdict
from kernelverse_amd.correctness_policy import resolve_correctness_policy

DEVICE = "cuda"
MAX_SAMPLES = 1_000_000

DTYPES = {
    "float32": (torch.float32, _lib.F32),
    "bfloat16": (torch.bfloat16, _lib.BF16),
    "float16": (torch.float16, _lib.F16),
    "float8_e4m3fn": (torch.float8_e4m3fn, _lib.F8E4M3FN),
    "int8": (torch.int8, _lib.I8),
    "int64": (torch.int64, _lib.I64),
}

# magnitude mask and first non-finite magnitude of the codes that "steps" moves
CODES = {
    "bfloat16": (torch.int16, 0x7FFF, 0x7F80),
    "float16": (torch.int16, 0x7FFF, 0x7C00),
    "float8_e4m3fn": (torch.int8, 0x7F, 0x7F),
}

# the tolerances operators configure for their outputs
TOLERANCES = {
    "FP32": {"rtol": 1e-5, "atol": 1e-5},
    "BF16": {"rtol": 1.6e-2, "atol": 1e-2},
    "FP16": {"rtol": 1e-3, "atol": 1e-3},
}
DTYPE_NAMES = {"float32": "FP32", "bfloat16": "BF16", "float16": "FP16"}
# a batch's pairs cycle through these, so that neighbours differ
BATCH_TOLERANCES = {
    "float32": ((1e-5, 1e-5), (1.3e-6, 1e-5), (5e-4, 5e-4), (1e-4, 1e-6)),
    "bfloat16": ((1.6e-2, 1e-2), (1.6e-2, 1e-3), (1e-2, 1e-2), (5e-3, 1e-3)),
}
POLICY_CATEGORY = {"strict": "activation", "tolerant": "gemm", "cosine": "attention"}


def _pair(name, entry, dtype, rows, cols, data, policy="strict", layout="contiguous", **more):
    return {"name": name, "entry": entry, "dtype": dtype, "rows": rows, "cols": cols, "data": data, "policy": policy,
            "layout": layout, **more}


def listed():
    return [
        # a small operator output (a few tokens' activations), judged on its own: launches and latency
        _pair("small_fp32", "tensors", "float32", 32, 128, "noise"),
        # an ordinary fp32 operator output, every element off by rounding noise
        _pair("fp32_1m", "tensors", "float32", 1024, 1024, "noise"),
        # a large fp32 output with a ragged length, verdicts issued back to back
        _pair("fp32_64m_odd", "pair", "float32", 8191, 8191, "noise"),
        # the headline workload: a 1 GiB bf16 pair with 5 % of its elements one ULP off
        _pair("bf16_256m", "pair", "bfloat16", 16384, 16384, "steps", moved=0.05, std=2.0),
        # a bf16 GEMM output whose kernel rounds elsewhere than the reference: half of the elements one ULP off,
        # judged with the tolerant policy's near-zero diagnostics
        _pair("bf16_64m_tolerant", "tensors", "bfloat16", 8192, 8192, "steps", "tolerant", moved=0.5, std=2.0),
        # an attention output: contiguous from the kernel, a permuted view from the reference
        _pair("fp16_heads_cosine", "tensors", "float16", 8 * 16 * 1024, 128, "steps", "cosine", "heads", batch=8, heads=16,
              moved=0.02, std=1.0),
        # fp16 logits with masked (infinite) and undefined entries in row-pitched storage
        _pair("fp16_pitched_nonfinite", "tensors", "float16", 4096, 32768, "nonfinite", "strict", "pitched", pad=128),
        # a quantised fp8 output, 2 % of the codes one step away
        _pair("fp8_128m", "record", "float8_e4m3fn", 16384, 8192, "steps", moved=0.02, std=4.0),
        # a quantised int8 output, equal except for a few positions
        _pair("int8_128m", "record", "int8", 16384, 8192, "integers", changed=1000),
        # an output the reference returns transposed while the kernel writes it contiguously
        _pair("bf16_transposed", "tensors", "bfloat16", 4096, 4096, "steps", "strict", "transposed", moved=0.05, std=1.0),
        # a layer's nested output: hidden state, a (key, value) pair, indices and scores, in one call
        {"name": "nested_layer", "entry": "outputs", "tokens": 2048, "width": 1024, "policy": "tolerant"},
        # a ragged batch of thousands of small and medium outputs in one call
        {"name": "batch_4096", "entry": "batch", "pairs": 4096, "lo": 1024, "hi": 1 << 20, "sizes": 5},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, lo, hi):
    """(rows, cols) of about a log-uniform number of elements in [lo, hi], odd ones among them."""
    n = _log_uniform(rng, lo, hi)
    cols = max(1, min(n, _log_uniform(rng, 32, 16384)))
    if rng.random() < 0.6:
        cols = max(64, cols // 64 * 64)
    return max(1, min(n, hi) // cols), cols


def draw(rng):
    kind = rng.random()
    if kind < 0.1:
        return {"entry": "batch", "pairs": _log_uniform(rng, 4, 3000), "lo": 1024, "hi": 1 << 20,
                "sizes": rng.randrange(1 << 20)}
    if kind < 0.25:
        return {"entry": "outputs", "tokens": _log_uniform(rng, 16, 8192), "width": 8 * _log_uniform(rng, 16, 256),
                "policy": rng.choice(("strict", "tolerant"))}
    dtype = rng.choice(("float32", "float32", "bfloat16", "float16", "float8_e4m3fn", "int8"))
    layout = rng.choice(("contiguous", "contiguous", "contiguous", "pitched", "heads", "transposed", "sliced"))
    # (a 32-bit pair is twice as heavy as a 16-bit one; strided views of up to 32 Mi elements)
    top = {"float32": 1 << 26, "bfloat16": 1 << 27, "float16": 1 << 27}.get(dtype, 1 << 27)
    rows, cols = _shape(rng, 1 << 10, top if layout in ("contiguous", "pitched") else 1 << 25)
    c = _pair("", rng.choice(("tensors", "pair")), dtype, rows, cols, "steps", "strict", layout)
    del c["name"]
    if dtype == "int8":
        c.update(data="integers", changed=rng.choice((0, 1, 1000)))
    elif dtype == "float32":
        c.update(data="noise", policy=rng.choice(("strict", "tolerant")))
    elif dtype == "float8_e4m3fn":
        c.update(moved=rng.choice((0.02, 0.2)), std=4.0)
    else:
        c.update(moved=rng.choice((0.005, 0.05, 0.5)), std=rng.choice((0.5, 2.0)),
                 policy=rng.choice(("strict", "tolerant", "cosine")))
        if layout == "pitched" and dtype == "float16":
            c.update(data="nonfinite")
    if dtype in ("float8_e4m3fn", "int8") and c["entry"] == "tensors":
        # (the drop-in refuses fp8, as torch's isfinite does; an int8 pair's meta is all counts)
        c["entry"] = "record"
    if layout == "pitched":
        c["pad"] = rng.choice((8, 64, 128))
    if layout == "heads":
        c["cols"] = rng.choice((64, 80, 128))
        rows = max(1, rows * cols // c["cols"])
        seq = max(1, min(rows, _log_uniform(rng, 16, 4096)))
        heads = max(1, min(32, rows // seq))
        c.update(heads=heads, batch=max(1, min(16, rows // (seq * heads))))
        c["rows"] = c["batch"] * heads * seq
    return c


# ------------------------------------------------------------ inputs
def _values(case, n, gen):
    """(generated, reference) of n elements, contiguous."""
    dtype = DTYPES[case["dtype"]][0]

    def uniform(k=n):
        return torch.rand(k, generator=gen, device=DEVICE)

    def normal(k=n):
        return torch.randn(k, generator=gen, device=DEVICE)

    if case["data"] == "noise":
        ref = normal()
        out = torch.add(ref, normal(), alpha=1e-6)
        hit = uniform() < 1e-3
        out += hit * (1e-3 + (1e-1 - 1e-3) * uniform())
        return out.to(dtype), ref.to(dtype)
    if case["data"] == "integers":
        ref = torch.randint(-128, 128, (n,), generator=gen, device=DEVICE, dtype=torch.int8)
        out = ref.clone()
        if case["changed"]:
            at = torch.randint(0, n, (case["changed"],), generator=gen, device=DEVICE)
            out[at] = (ref[at].to(torch.int16) + 77).to(torch.int8)
        return out, ref
    if case["data"] == "nonfinite":
        ref = (uniform() * 120000.0 - 60000.0).to(dtype)
        u = uniform()
        ref[u < 5e-4] = float("nan")
        ref[(u >= 5e-4) & (u < 7.5e-4)] = float("inf")
        ref[(u >= 7.5e-4) & (u < 1e-3)] = float("-inf")
        out = ref.clone()
        at = torch.randint(0, n, (17,), generator=gen, device=DEVICE)
        out[at] = torch.where(torch.isfinite(ref[at]), float("nan"), 1.0).to(dtype)
        return out, ref
    # steps of the codes
    x = normal() * case["std"]
    if case["dtype"] == "float8_e4m3fn":
        x.clamp_(-448, 448)
    ref = x.to(dtype)
    del x
    view, mask, nonfinite = CODES[case["dtype"]]
    u = uniform()
    steps = (u < case["moved"]).to(view)
    steps += 2 * (u >= 1 - 1e-4).to(view) + (u >= 1 - 1e-4).to(view) * (u >= case["moved"]).to(view)
    del u
    codes = ref.view(view)
    up = (codes & mask) + steps
    out = torch.where((up >= 0) & (up < nonfinite), codes + steps, codes - steps).view(dtype)
    return out, ref


def _in_layout(case, out, ref):
    rows, cols = case["rows"], case["cols"]
    layout = case["layout"]
    if layout == "heads":
        b, h = case["batch"], case["heads"]
        s = rows // (b * h)
        out, ref = out.view(b, h, s, cols), ref.view(b, h, s, cols)
        return out, ref.transpose(1, 2).contiguous().transpose(1, 2)
    out, ref = out.view(rows, cols), ref.view(rows, cols)
    if layout == "transposed":
        ref = ref.t().contiguous().t()
    elif layout == "pitched":
        def pitched(t):
            base = torch.zeros(rows, cols + case["pad"], dtype=t.dtype, device=t.device)
            view = base[:, :cols]
            view.copy_(t)
            return view
        out, ref = pitched(out), pitched(ref)
    elif layout == "sliced":
        base = torch.zeros(rows, cols + 1, dtype=ref.dtype, device=ref.device)
        base[:, 1:] = ref
        ref = base[:, 1:]
    return out, ref


def _generator(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    return gen


def _case_pair(case, seed):
    out, ref = _values(case, case["rows"] * case["cols"], _generator(seed))
    return _in_layout(case, out, ref)


def _nested(case, seed):
    gen = _generator(seed)
    t, w = case["tokens"], case["width"]

    def steps(rows, cols, moved):
        return tuple(x.view(rows, cols) for x in
                     _values({"dtype": "float16", "data": "steps", "moved": moved, "std": 1.0}, rows * cols, gen))

    hidden, key, value = steps(t, w, 0.05), steps(t, w // 4, 0.02), steps(t, w // 4, 0.02)
    ref_ids = torch.randint(0, 65536, (t, 8), generator=gen, device=DEVICE)
    ids = ref_ids.clone()
    ids.view(-1)[torch.randint(0, t * 8, (4,), generator=gen, device=DEVICE)] += 1
    scores = tuple(x.view(t, 8) for x in _values({"dtype": "float32", "data": "noise"}, t * 8, gen))
    return ((hidden[0], [key[0], value[0]], ids, scores[0]), (hidden[1], [key[1], value[1]], ref_ids, scores[1]))


def _batch_sizes(case):
    rng = np.random.default_rng(case["sizes"])
    u = rng.uniform(math.log(case["lo"]), math.log(case["hi"]), size=case["pairs"])
    return [int(min(case["hi"], max(case["lo"], round(math.exp(v))))) for v in u]


def _batch_pairs(case, seed):
    """[(generated, reference, dtype name)], fp32 and bf16 in turn, carved from one buffer per type at the
    alignment of an allocation."""
    gen = _generator(seed)
    sizes = _batch_sizes(case)
    parts = []
    for k, name in enumerate(("float32", "bfloat16")):
        step = 512 // DTYPES[name][0].itemsize
        offsets, at = [], 0
        for n in sizes[k::2]:
            offsets.append((at, n))
            at += (n + step - 1) // step * step
        out, ref = _values({"dtype": name, "data": "noise"}, at, gen) if at else (None, None)
        parts.append([(out[a:a + n], ref[a:a + n], name) for a, n in offsets])
    return [parts[i % 2][i // 2] for i in range(len(sizes))]


# ------------------------------------------------------------ the library's structures
def _kvv_tensor(t, code):
    k = _lib.KvvTensor()
    k.data, k.dtype, k.ndim = t.data_ptr(), code, t.dim()
    for i, (s, st) in enumerate(zip(t.shape, t.stride())):
        k.sizes[i], k.strides[i] = s, st
    return k


def _kvv_policy(case, dtype, rtol, atol):
    p = _lib.KvvPolicy()
    p.max_samples = MAX_SAMPLES
    if dtype in ("int8", "int64"):
        p.mode, p.max_abs_diff = _lib.MODE_MAX_ABS_DIFF, 1 if dtype == "int8" else 0
        return p
    p.mode, p.rtol, p.atol = _lib.MODE_ISCLOSE, rtol, atol
    row = _near_row(case.get("policy", "strict"), dtype)
    if row:
        p.flags = _lib.FLAG_NEAR_ZERO
        p.near_zero_abs, p.near_zero_bad_abs = row["near_zero_abs"], row["max_near_zero_bad_abs"]
    return p


def _columns(records, count):
    """Views of the record fields of `count` records (a pinned byte buffer)."""
    size = ctypes.sizeof(_lib.KvvResult)
    words = records.view(count, size).view(torch.int64)
    reals = records.view(count, size).view(torch.float64)
    cols = {}
    for name, kind in _lib.KvvResult._fields_:
        at = getattr(_lib.KvvResult, name).offset
        if name in ("status", "reserved"):
            continue
        if name == "ulp_hist":
            cols[name] = words[:, at // 8:at // 8 + _lib.HIST_BUCKETS]
        else:
            cols[name] = (reals if kind is ctypes.c_double else words)[:, at // 8]
    return cols


def _tolerance_of(dtype):
    t = TOLERANCES.get(DTYPE_NAMES.get(dtype), verdict.TOLERANCE_POLICY["fp32"])
    return t["rtol"], t["atol"]


def _policy(name):
    return resolve_correctness_policy({"category": POLICY_CATEGORY[name], "op_name": "perf"})


def _near_row(policy, dtype):
    """The near-zero thresholds the tolerant policy judges 16-bit floats with, else None."""
    if policy != "tolerant" or dtype not in ("bfloat16", "float16"):
        return None
    return _policy(policy)["thresholds"][DTYPE_NAMES[dtype]]


def prepare(case, seed):
    entry = case["entry"]
    state = {"entry": entry, "policy": _policy(case.get("policy", "strict")), "tolerance": TOLERANCES}
    if entry == "outputs":
        state["out"], state["ref"] = _nested(case, seed)
        return state
    if entry in ("tensors", "record"):
        state["out"], state["ref"] = _case_pair(case, seed)
        return state
    lib = state["lib"] = _lib.load()
    size = ctypes.c_size_t()
    if entry == "pair":
        out, ref = _case_pair(case, seed)
        state["keep"] = (out, ref)
        code = DTYPES[case["dtype"]][1]
        state["args"] = (_kvv_tensor(out, code), _kvv_tensor(ref, code),
                         _kvv_policy(case, case["dtype"], *_tolerance_of(case["dtype"])))
        _lib.check(lib.kvv_workspace_size(*state["args"], ctypes.byref(size)), "kvv_workspace_size")
        count = 1
    else:
        pairs = _batch_pairs(case, seed)
        count = len(pairs)
        state["keep"] = pairs
        gens, refs = (_lib.KvvTensor * count)(), (_lib.KvvTensor * count)()
        pols = (_lib.KvvPolicy * count)()
        for i, (out, ref, name) in enumerate(pairs):
            gens[i], refs[i] = _kvv_tensor(out, DTYPES[name][1]), _kvv_tensor(ref, DTYPES[name][1])
            pols[i] = _kvv_policy(case, name, *BATCH_TOLERANCES[name][(i // 2) % 4])
        state["args"] = (count, gens, refs, pols)
        _lib.check(lib.kvv_batch_workspace_size(*state["args"], ctypes.byref(size)), "kvv_batch_workspace_size")
    state["workspace"] = torch.empty(size.value, dtype=torch.uint8, device=DEVICE)
    records = torch.zeros(count * ctypes.sizeof(_lib.KvvResult), dtype=torch.uint8, pin_memory=True)
    state["records"], state["columns"] = records, _columns(records, count)
    state["call"] = (*state["args"], records.data_ptr(), state["workspace"].data_ptr(), size.value,
                     torch.cuda.current_stream().cuda_stream)
    return state


def _numbers(meta, dims):
    """A meta without its texts; a pair without mismatches gets the entries that the others have."""
    out = {k: v for k, v in meta.items() if not isinstance(v, str)}
    if "max_abs" not in out:
        out["max_abs"] = out["max_rel"] = 0.0
        out["first_mismatch_index"] = (-1,) * dims
    return out


def run(state):
    entry = state["entry"]
    if entry == "tensors":
        ok, _, meta = verdict._compare_tensors(state["out"], state["ref"], "output", state["tolerance"], state["policy"])
        return {"ok": ok, "meta": _numbers(meta, state["ref"].dim())}
    if entry == "record":
        return verdict.verdict_record(state["out"], state["ref"], state["tolerance"], state["policy"])
    if entry == "outputs":
        ok, _, metas = verdict._compare_outputs(state["out"], state["ref"], "output", state["tolerance"], state["policy"])
        return {"ok": ok, "metas": _by_field([_numbers(m, 2) for m in metas])}
    call = state["lib"].kvv_verdict if entry == "pair" else state["lib"].kvv_verdict_batch
    rc = call(*state["call"])
    if rc:
        _lib.check(rc, "verdict")
    return state["columns"]


def _by_field(metas):
    """One array per field over the metas that hold it."""
    names = dict.fromkeys(k for m in metas for k, v in m.items() if isinstance(v, (bool, int, float)))
    return {k: np.array([m[k] for m in metas if isinstance(m.get(k), (bool, int, float))]) for k in names}


def work(case):
    if case["entry"] == "outputs":
        t, w = case["tokens"], case["width"]
        n16, n_small = t * (w + 2 * (w // 4)), t * 8
        n, moved = n16 + 2 * n_small, 2 * (2 * n16 + 8 * n_small + 4 * n_small)
    elif case["entry"] == "batch":
        sizes = _batch_sizes(case)
        n, moved = sum(sizes), 2 * (4 * sum(sizes[0::2]) + 2 * sum(sizes[1::2]))
    else:
        n = case["rows"] * case["cols"]
        moved = 2 * n * DTYPES[case["dtype"]][0].itemsize
    # per pair of elements: four sums of products, the difference, the bound and its comparison, the quotient
    return {"bytes": moved, "flops": 13 * n}


def tolerance(case):
    # counts, indices and histograms are whole numbers and equal; p99s and maxima are single elements' float32
    # values; the sums are declared to 1e-6 (16- and 8-bit codes: packed dot products in float32 per lane)
    return {"rel": 1e-6}


# ------------------------------------------------------------ the results in 64 bits
CHUNK = 1 << 25


def _strided(t, n, m):
    """The sampled values of a flat tensor: all, or element i*(n-1)//(m-1)."""
    if n <= m:
        return t
    return t[torch.arange(m, device=t.device, dtype=torch.int64) * (n - 1) // (m - 1)]


def _wide(t):
    return t.to(torch.float32).double() if "float8" in str(t.dtype) else t.double()


def _p99(t):
    return float(torch.quantile(t, 0.99))


def _cosine(gr, gg, rr):
    return min(1.0, max(-1.0, gr / math.sqrt(gg * rr))) if gg == gg and rr == rr else float("nan")


def _expected(out, ref, whole, rtol, atol, near):
    """The real-valued record fields of one pair, in float64."""
    out, ref = out.reshape(-1), ref.reshape(-1)
    n = ref.numel()
    sums = torch.zeros(4, dtype=torch.float64, device=ref.device)
    tops = {"max_abs": [], "max_rel": [], "mismatch_max_abs": [], "mismatch_max_rel": []}
    small, count = [], 0
    for a in range(0, n, CHUNK):
        g, r = _wide(out[a:a + CHUNK]), _wide(ref[a:a + CHUNK])
        d = (g - r).abs()
        rel = d / (r.abs() + 1e-12)
        if whole is not None:
            miss = d > whole
        else:
            miss = ~((g == r) | (torch.isfinite(d) & (d <= atol + (rtol * g).abs())))
        sums += torch.stack([(g * g).sum(), (r * r).sum(), (g * r).sum(), (d * d).sum()])
        count += int(miss.sum())
        tops["max_abs"].append(d.max())
        tops["max_rel"].append(rel.max())
        if bool(miss.any()):
            tops["mismatch_max_abs"].append(d[miss].max())
            tops["mismatch_max_rel"].append(rel[miss].max())
        if near is not None:
            small.append(d[r.abs() <= near])
    gg, rr, gr, dd = sums.tolist()
    e = {k: float(torch.stack(v).max()) if v else 0.0 for k, v in tops.items()}
    g, r = _wide(_strided(out, n, MAX_SAMPLES)), _wide(_strided(ref, n, MAX_SAMPLES))
    d = (g - r).abs()
    sg, sr, sx = float((g * g).sum()), float((r * r).sum()), float((g * r).sum())
    e.update(count=count, p99_abs=_p99(d), p99_rel=_p99(d / (r.abs() + 1e-12)), sample_sum_gg=sg, sample_sum_rr=sr,
             sample_sum_gr=sx, sample_cosine=_cosine(sx, sg, sr), sample_norm_ratio=math.sqrt(sg) / math.sqrt(sr),
             sum_gg=gg, sum_rr=rr, sum_gr=gr, sum_dd=dd, rel_l2=math.sqrt(dd) / math.sqrt(rr),
             cosine=_cosine(gr, gg, rr), near_zero_p99_abs=None, near_zero_mean_abs=None)
    if near is not None:
        v = torch.cat(small)
        v = _strided(v, v.numel(), MAX_SAMPLES)
        if v.numel():
            e.update(near_zero_p99_abs=_p99(v), near_zero_mean_abs=float(v.mean()))
    return e


RECORD_REALS = tuple(name for name, kind in _lib.KvvResult._fields_ if kind is ctypes.c_double)


def _expected_of(case, dtype, out, ref, rtol, atol):
    whole = {"int8": 1, "int64": 0}.get(dtype)
    row = _near_row(case.get("policy", "strict"), dtype)
    return _expected(out, ref, whole, rtol, atol, row["near_zero_abs"] if row else None)


def _expected_meta(e, dtype, n):
    """The real-valued meta entries of a pair (rounded as the metas are)."""
    meta = {"cosine_similarity": None, "norm_ratio": None, "mismatch_rate": round(e["count"] / n, 4),
            "p99_abs": e["p99_abs"], "p99_rel": e["p99_rel"]}
    if "int" not in dtype:
        meta["cosine_similarity"] = round(e["sample_cosine"], 4)
        meta["norm_ratio"] = round(e["sample_norm_ratio"], 4)
    if e["near_zero_p99_abs"] is not None:
        meta["near_zero_p99_abs"], meta["near_zero_mean_abs"] = e["near_zero_p99_abs"], e["near_zero_mean_abs"]
    meta["max_abs"], meta["max_rel"] = e["mismatch_max_abs"], e["mismatch_max_rel"]
    return meta


def exact(case, seed):
    entry = case["entry"]
    if entry == "outputs":
        out, ref = _nested(case, seed)
        leaves = [(out[0], ref[0], "float16"), (out[1][0], ref[1][0], "float16"), (out[1][1], ref[1][1], "float16"),
                  (out[2], ref[2], "int64"), (out[3], ref[3], "float32")]
        metas = [_expected_meta(_expected_of(case, name, g, r, *_tolerance_of(name)), name, r.numel())
                 for g, r, name in leaves]
        return {"ok": None, "metas": _by_field(metas)}
    if entry == "batch":
        rows = [_expected_of(case, name, out, ref, *BATCH_TOLERANCES[name][(i // 2) % 4])
                for i, (out, ref, name) in enumerate(_batch_pairs(case, seed))]
        nan = float("nan")
        return {k: torch.tensor([nan if e[k] is None else e[k] for e in rows], dtype=torch.float64)
                for k in RECORD_REALS}
    out, ref = _case_pair(case, seed)
    dtype = case["dtype"]
    e = _expected_of(case, dtype, out, ref, *_tolerance_of(dtype))
    if entry == "tensors":
        return {"ok": None, "meta": _expected_meta(e, dtype, ref.numel())}
    reals = {k: float("nan") if e[k] is None else e[k] for k in RECORD_REALS}
    return reals if entry == "record" else {k: torch.tensor([v], dtype=torch.float64) for k, v in reals.items()}
