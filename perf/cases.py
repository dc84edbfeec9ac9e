"""The calls of checkers_amd whose speed matters, as a user's program makes them.

Every case goes through the public Python entry points over the C ABI and is
one of seven kinds:

  compress        Encoder.compress of one tensor (histogram, table, encode)
  decode          Decoder.decode of one compressed tensor
  compress_many   a shard's tensors in one call
  decode_many     the same shard restored in one call
  roundtrip       compress and decode of one tensor, a written checkpoint verified
  analyze         the statistics pass over a rank's records
  repair          a group's grammar built on one tensor and applied to another

A case names its tensors as "role:elements role:elements ..."; a role fixes the
element type and the distribution of the values (ROLES).  Sizes are those of
the Llama-3-8B shapes and ZeRO-3 ranks that the tests and the benchmark use, at
the whole or at ragged fractions of them.
"""
import math

import numpy as np
import torch

import checkers_amd as ck

KIB64, MIB = 65536, 1 << 20

# role: (dtype tag, bytes per element, sidecar bytes per element, coded bytes
# per element).  The coded size is the order-0 entropy of the masked bytes under
# the tensor's one table, from samples of each distribution.
ROLES = {
    "params": (ck.BF16, 2, 1, 0.59),      # bf16 weights, N(0, 0.02)
    "half": (ck.F16, 2, 1, 0.91),         # fp16 weights, N(0, 0.02)
    "norm": (ck.BF16, 2, 1, 0.25),        # bf16 RMSNorm weights, near 1
    "master": (ck.F32, 4, 2, 2.05),       # fp32 master weights, upcast from bf16 steps
    "exp_avg": (ck.F32, 4, 2, 2.04),      # Adam first moment, N(0, 1e-3)
    "exp_avg_sq": (ck.F32, 4, 2, 2.03),   # Adam second moment
    "wide": (ck.F32, 4, 2, 2.19),         # fp32 over about 30 binades, zeros and infinities among them
    "quant8": (ck.I8, 1, 0, 0.88),        # 8-bit optimizer state
    "ids32": (ck.I32, 4, 0, 2.3),         # int32 indices below a vocabulary size
}

# one Llama-3-8B decoder layer, in parameter order
LAYER = [("params", 4096 * 4096), ("params", 1024 * 4096), ("params", 1024 * 4096), ("params", 4096 * 4096),
         ("params", 14336 * 4096), ("params", 14336 * 4096), ("params", 4096 * 14336), ("norm", 4096), ("norm", 4096)]
LLAMA8B = 8_030_261_248


def _spec(tensors):
    return " ".join(f"{role}:{n}" for role, n in tensors)


def _parse(case):
    return [(r, int(n)) for r, n in (t.split(":") for t in case["tensors"].split())]


def _rank_shard(world):
    """One ZeRO-3 rank's flat tensors: bf16 parameters and the three fp32 states."""
    n = LLAMA8B // world
    return [("params", n), ("master", n), ("exp_avg", n), ("exp_avg_sq", n)]


def _rank_records(layers, world):
    """The records a ZeRO-3 rank discovers: per parameter its bf16 slice, then
    the master weights and the two moments of that slice."""
    out = []
    for _ in range(layers):
        for role, n in LAYER:
            out += [(role, n // world), ("master", n // world), ("exp_avg", n // world), ("exp_avg_sq", n // world)]
    return out


def listed():
    return [
        # the smallest tensor of a checkpoint: a normalisation weight
        dict(name="compress_norm", kind="compress", tensors=_spec([("norm", 4096)]), unit=KIB64),
        # one optimizer state of an attention projection, both directions
        dict(name="compress_matrix", kind="compress", tensors=_spec([("exp_avg", 4096 * 4096)]), unit=KIB64),
        dict(name="decode_matrix", kind="decode", tensors=_spec([("exp_avg", 4096 * 4096)]), unit=KIB64, check=True),
        # a decoder layer's parameters, both directions: a layer-wise checkpoint
        dict(name="compress_layer", kind="compress_many", tensors=_spec(LAYER), unit=KIB64),
        dict(name="decode_layer", kind="decode_many", tensors=_spec(LAYER), unit=KIB64, check=False),
        # a rank's whole optimizer shard (rank 0 of 32), both directions
        dict(name="compress_shard", kind="compress_many", tensors=_spec(_rank_shard(32)), unit=KIB64),
        dict(name="decode_shard", kind="decode_many", tensors=_spec(_rank_shard(32)), unit=KIB64, check=False),
        # 1 MiB units, the choice for the largest models, with a ragged end
        dict(name="compress_1mib_units", kind="compress", tensors=_spec([("exp_avg", 268_435_456 - 98_765)]), unit=MIB),
        # the reference's own layout (one stream per tensor), written and verified
        dict(name="roundtrip_one_stream", kind="roundtrip", tensors=_spec([("params", 4096 * 4096)]), unit=0, check=True),
        # an 8-bit optimizer state, written and verified
        dict(name="roundtrip_int8", kind="roundtrip", tensors=_spec([("quant8", 14336 * 4096)]), unit=KIB64, check=True),
        # the statistics pass before a checkpoint: four layers of a rank of 8, 144 records
        dict(name="analyze_layers", kind="analyze", tensors=_spec(_rank_records(4, 8)), bins=256),
        # prefix-mask repair of a group: rules from one projection applied to its sibling
        dict(name="repair_group", kind="repair", tensors=_spec([("params", 1024 * 4096), ("params", 1024 * 4096)]),
             rules=50),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["compress", "decode", "compress_many", "decode_many", "roundtrip", "analyze", "repair"])
    masked = ["params", "half", "norm", "master", "exp_avg", "exp_avg_sq", "wide"]
    if kind in ("compress", "decode"):
        case = dict(kind=kind, tensors=_spec([(rng.choice(masked), _log_uniform(rng, 1000, 1 << 27))]),
                    unit=rng.choice([16384, KIB64, KIB64, KIB64, 4 * KIB64, MIB]))
    elif kind in ("compress_many", "decode_many"):
        top = rng.choice([1 << 18, 1 << 23, 1 << 25, 1 << 27])
        case = dict(kind=kind, tensors=_spec([(rng.choice(masked), _log_uniform(rng, max(1000, top >> 8), top))
                                              for _ in range(rng.randint(2, 6))]),
                    unit=rng.choice([KIB64, KIB64, KIB64, MIB]))
    elif kind == "roundtrip":
        if rng.random() < 0.5:  # one stream per tensor
            case = dict(kind=kind, tensors=_spec([(rng.choice(masked), _log_uniform(rng, 1000, 1 << 23))]), unit=0)
        else:
            case = dict(kind=kind, tensors=_spec([(rng.choice(["quant8", "ids32"]), _log_uniform(rng, 1000, 1 << 24))]),
                        unit=rng.choice([16384, KIB64]))
    elif kind == "analyze":
        top = rng.choice([1 << 14, 1 << 20, 1 << 24])
        return dict(kind=kind, tensors=_spec([(rng.choice(sorted(set(ROLES) - {"wide"})), _log_uniform(rng, 100, top))
                                              for _ in range(rng.randint(1, 64))]), bins=rng.choice([64, 256, 256]))
    else:
        n = _log_uniform(rng, 1000, 1 << 22)
        role = rng.choice(["params", "half"])
        return dict(kind=kind, tensors=_spec([(role, n), (role, max(1, n - rng.randint(0, n // 2)))]),
                    rules=rng.choice([10, 50]))
    case["check"] = rng.random() < 0.5
    return case


def _make(role, n, gen):
    """One tensor of a role on the GPU."""
    dev = "cuda"
    r = torch.randn(n, generator=gen, device=dev)
    if role == "params":
        return (r * 0.02).to(torch.bfloat16)
    if role == "half":
        return (r * 0.02).to(torch.float16)
    if role == "norm":
        return (1.0 + 0.01 * r).to(torch.bfloat16)
    if role == "master":  # bf16 weights after a few fp32 optimizer steps
        return (r * 0.02).to(torch.bfloat16).float() + 1e-5 * torch.randn(n, generator=gen, device=dev)
    if role == "exp_avg":
        return r * 1e-3
    if role == "exp_avg_sq":
        return (r * 1e-3).square_().add_(1e-12)
    if role == "wide":
        x = torch.exp(r * 5.0 - 12.0)
        x[torch.randint(0, n, (n // 1000,), generator=gen, device=dev)] = 0.0
        x[torch.randint(0, n, (n // 100000,), generator=gen, device=dev)] = float("inf")
        return x
    if role == "quant8":
        return (r * 32.0).round_().clamp_(-127, 127).to(torch.int8)
    return torch.randint(0, 128256, (n,), generator=gen, device=dev, dtype=torch.int32)


def _inputs(case, seed):
    out = []
    for k, (role, n) in enumerate(_parse(case)):
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed * 1009 + k)
        out.append(_make(role, n, gen))
    return out


def prepare(case, seed):
    """The inputs, and the encoders, decoders, analyzer or repairer (buffers and
    workspaces) that a program keeps from call to call."""
    xs = _inputs(case, seed)
    roles = _parse(case)
    tags = [ROLES[r][0] for r, _ in roles]
    st = dict(kind=case["kind"], xs=xs, check=case.get("check", True))
    if case["kind"] == "analyze":
        st["analyzer"] = ck.Analyzer(xs, tags, case["bins"])
    elif case["kind"] == "repair":
        st["repairer"] = ck.Repairer(max(n for _, n in roles), tags[0], None, case["rules"])
    else:
        st["encs"] = [ck.Encoder(n, tag, case["unit"]) for (_, n), tag in zip(roles, tags)]
        for e in st["encs"]:
            e.out.zero_()
        if case["kind"] not in ("compress", "compress_many"):
            st["decs"] = [ck.Decoder(n, tag, case["unit"]) for (_, n), tag in zip(roles, tags)]
            st["dsts"] = [torch.empty(x.nbytes, dtype=torch.uint8, device="cuda") for x in xs]
        if case["kind"] in ("decode", "decode_many"):  # what was read back from a checkpoint
            st["coded"] = ck.compress_many(st["encs"], xs)
            torch.cuda.synchronize()
    return st


def _coded_outputs(e):
    """Everything a compress call returns: the packed streams (in their whole
    buffer, cleared by prepare, of which a call writes the first e.total bytes),
    their size, headers and offsets, the sidecar, and the frequency table's
    counts, which its other arrays restate."""
    out = dict(data=e.data, total=e.total, headers=e.headers, unit_offsets=e.unit_offsets, table=e.table.norm)
    if e.sidecar is not None:
        out["sidecar"] = e.sidecar
    return out


def _decode(st, e):
    bad = st["decs"][0].decode(e.data, e.headers, e.unit_offsets, e.table, e.sidecar, st["dsts"][0], check=st["check"])
    return dict(dst=st["dsts"][0], bad=-1 if bad is None else bad)


def run(st):
    kind = st["kind"]
    if kind == "compress":
        return _coded_outputs(st["encs"][0].compress(st["xs"][0]))
    if kind == "decode":
        return _decode(st, st["coded"][0])
    if kind == "compress_many":
        return [_coded_outputs(e) for e in ck.compress_many(st["encs"], st["xs"])]
    if kind == "decode_many":
        bad = ck.decode_many(st["decs"], st["coded"], st["dsts"], check=st["check"])
        return dict(dst=st["dsts"], bad=-1 if bad is None else list(bad))
    if kind == "roundtrip":
        e = st["encs"][0].compress(st["xs"][0])
        return [_coded_outputs(e), _decode(st, e)]
    if kind == "analyze":
        a = st["analyzer"]
        a.run()
        return dict(hist=a.hist, moments=a.mom, minmax=a.mm, fingerprint=a.fp)
    r = st["repairer"].build(st["xs"][0])
    tokens = st["repairer"].apply(st["xs"][1], r["rules"])
    return dict(rules=np.array(r["rules"], np.uint64).reshape(-1, 4), out_len=r["out_len"], max_pair=r["max_pair"],
                applied=tokens)


def work(case):
    """Each input read once, each output written once.  A coded tensor is its
    packed streams, 4104 bytes of headers and offset per unit, and its sidecar;
    a repair reads its two tensors."""
    total = 0
    for role, n in _parse(case):
        _, es, spe, coded = ROLES[role]
        total += n * es
        if case["kind"] in ("analyze", "repair"):
            continue
        unit = case["unit"] or n * es
        out = n * (spe + coded) + -(-n * es // unit) * 4104
        total += out
        if case["kind"] == "roundtrip":
            total += out + n * es
    return dict(bytes=int(total), flops=0)


def tolerance(case):
    """Streams, counts and decoded bytes are exact.  The moments are fp32 values
    of fp64 sums over fp32 powers: they measured within 7e-8 of exact()'s."""
    if case["kind"] == "analyze":
        return dict(rel=4e-7, max=4e-6)
    return "exact"


def exact(case, seed):
    """Decoded bytes: the source's.  Statistics: the reference's formulas in 64
    bits (the histogram bins follow fp32 arithmetic and have no such value)."""
    kind = case["kind"]
    if kind == "analyze":
        xs = _inputs(case, seed)
        nb = min(case["bins"], 256)
        mom = torch.empty((len(xs), 4), dtype=torch.float64)
        mm = torch.empty((len(xs), 2), dtype=torch.float64)
        for i, x in enumerate(xs):
            d = x.double()
            lo, hi = d.min().item(), d.max().item()
            mean = d.mean().item()
            d -= mean
            var = d.square().mean().item()
            skew = kurt = 0.0
            if var > 1e-9:  # below it the reference reports no shape
                skew = d.pow(3).mean().item() / (var * math.sqrt(var))
                kurt = d.pow(4).mean().item() / (var * var)
            mom[i] = torch.tensor([mean, var, skew, kurt], dtype=torch.float64)
            mm[i] = torch.tensor([lo, hi], dtype=torch.float64)
        fp = torch.cat([mom, (mm[:, 1] - mm[:, 0]).unsqueeze(1)], 1)
        return dict(hist=None, moments=mom, minmax=mm, fingerprint=fp)
    if kind == "decode":
        return dict(dst=_inputs(case, seed)[0].view(torch.uint8), bad=None)
    if kind == "decode_many":
        return dict(dst=[x.view(torch.uint8) for x in _inputs(case, seed)], bad=None)
    return None
