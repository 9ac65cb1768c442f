"""The work that users of the batched multi-LoRA INT4 linear have it do, as timed cases.

Kinds of case, each through the package's public entry points:
- "layer": one decoder layer (RMSNorm, qkv, o with the residual add, RMSNorm, gate_up with SiLU(gate) * up, down with
  the residual add) recorded once as a HIP graph and replayed, as an engine runs every layer of a recorded pass. The
  inputs are already in the recorded tensors, where the layer before wrote them. Outputs: the qkv product, the gated
  activation and the residual stream.
- "product": routing and one INT4 product called eagerly, with each request's last-token rows gathered.
- "pass": a whole recorded decoder pass with the decision head; a batch's rows are copied into the recorded tensors
  and the graph is replayed. Outputs: the option probabilities.
- "mlp": the MLP of a bfloat16 base called eagerly: add_rms, the library product plus lora_add, silu_mul, the library
  product plus lora_add.
- "linear": one bfloat16 group called eagerly (the library product plus lora_add).
- "head": the decision head on the last-token rows of a pass, called eagerly.

Sizes: decoder shapes up to hidden 2048 / intermediate 6144 with 4-bit weights in groups of 64 (symmetric) or 128
(asymmetric); 1 to 1024 adapters of ranks 8 to 64; passes from one decode row to 160 k prefill tokens."""

from __future__ import annotations

import math

import numpy as np
import torch

from jeff_amd.epilogues import add_rms, rms, silu_mul
from jeff_amd.fast_path import AdapterPool, Lin, Workspace
from jeff_amd.int4 import pack_kernel, pack_kernel_asym
from jeff_amd.int4_kernels import int4_product
from jeff_amd.passes import DecoderInputs, RecordedPass, decoder_pass
from jeff_amd.readout import readout_rows

BF16 = torch.bfloat16
OPTIONS = 255  # answer options of the decision head
DEVICE = "cuda"


# --- the cases ------------------------------------------------------------------------------------------------------

def _layer(tokens: int, requests: int, adapters: int, rank, spread: str = "one", hidden: int = 2048, inter: int = 6144,
           kv: int = 1024, group: int = 128) -> dict:
    return {"kind": "layer", "tokens": tokens, "requests": requests, "spread": spread, "adapters": adapters,
            "rank": rank, "hidden": hidden, "inter": inter, "kv": kv, "group": group}


def listed() -> list[dict]:
    return [
        # a few requests decoding: the smallest call, where latency and launches count
        {"name": "decode-4", **_layer(4, 4, 4, 16)},
        # one request's 32 new tokens through its one adapter: a decision on a cached prefix
        {"name": "decision-32", **_layer(32, 1, 16, 16, "even")},
        # three such decisions of about 128 new tokens served together, symmetric weights in groups of 64
        {"name": "decisions-384", **_layer(384, 3, 16, 32, "near", group=64)},
        # a full decode batch over 64 adapters with ranks 8, 16, 32 and 64
        {"name": "decode-256", **_layer(256, 256, 64, "mixed")},
        # a larger decode batch, an odd number of rows, between the narrow and the large tiles
        {"name": "decode-643", **_layer(643, 643, 128, "mixed")},
        # decode over a large adapter pool: 4096 rows, 1024 adapters of rank 64
        {"name": "decode-pool-4096", **_layer(4096, 4096, 1024, 64)},
        # one layer's product over a ragged prefill of 64 requests, 16 adapters of rank 16
        {"name": "prefill-8855", "kind": "product", "tokens": 8855, "requests": 64, "spread": "uniform", "adapters": 16,
         "rank": 16, "k": 1024, "out": 3072, "group": 128},
        # a large prefill: 512 requests of log-normal length, 128 adapters of rank 32 with skewed popularity
        {"name": "prefill-159488", **_layer(159488, 512, 128, 32, "lognormal")},
        # a whole recorded pass of two layers over a ragged batch, decision head included
        {"name": "pass-2311", **_layer(2311, 24, 16, 16, "lognormal"), "kind": "pass", "layers": 2},
        # a bfloat16 base: one projection over 8 requests of 32 tokens
        {"name": "bf16-256", "kind": "linear", "tokens": 256, "requests": 8, "spread": "even", "adapters": 4,
         "rank": 16, "k": 1024, "out": 1024},
        # a bfloat16 base: the MLP of a prefill of 32 ragged requests
        {"name": "bf16-mlp-4501", "kind": "mlp", "tokens": 4501, "requests": 32, "spread": "lognormal", "adapters": 16,
         "rank": 16, "hidden": 2048, "inter": 6144},
        # the decision head on 512 requests' last-token rows
        {"name": "head-512", "kind": "head", "requests": 512, "adapters": 128, "hidden": 2048, "options": OPTIONS},
    ]


def _log(rng, low: int, high: int) -> int:
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng) -> dict:
    kind = rng.choices(("decode", "prompt", "product", "pass", "linear", "mlp", "head"), (4, 4, 2, 1, 1, 1, 1))[0]
    adapters = _log(rng, 1, 256)
    rank = rng.choice((8, 16, 32, 64, "mixed"))
    if kind == "head":
        return {"kind": "head", "requests": _log(rng, 1, 1024), "adapters": adapters, "hidden": 64 * rng.randint(8, 32),
                "options": rng.randint(2, 256)}
    requests = _log(rng, 1, 512)
    tokens = min(requests * _log(rng, 12, 400) + rng.randint(0, 11), 120000)
    spread = rng.choice(("near", "uniform", "lognormal"))
    if kind == "linear":
        return {"kind": "linear", "tokens": min(tokens, 20000), "requests": requests, "spread": spread,
                "adapters": adapters, "rank": rank, "k": 64 * rng.randint(8, 32), "out": 8 * rng.randint(64, 512)}
    if kind == "product":
        group = rng.choice((64, 128))
        return {"kind": "product", "tokens": min(tokens, 60000), "requests": requests, "spread": spread,
                "adapters": adapters, "rank": rank, "k": group * rng.randint(512 // group, 4096 // group),
                "out": 8 * rng.randint(64, 768), "group": group}
    hidden = 128 * rng.randint(4, 16)
    inter = 128 * rng.randint(2 * hidden // 128, 3 * hidden // 128)
    if kind == "mlp":
        return {"kind": "mlp", "tokens": min(tokens, 20000), "requests": requests, "spread": spread,
                "adapters": adapters, "rank": rank, "hidden": hidden, "inter": inter}
    shape = {"hidden": hidden, "inter": inter, "kv": 64 * rng.randint(1, hidden // 64),
             "group": rng.choice((64, 128))}
    if kind == "decode":
        rows = _log(rng, 1, 4096)
        return _layer(rows, rows, _log(rng, 1, 1024), rank, **shape)
    if kind == "pass":
        return {**_layer(min(tokens, 20000), requests, adapters, rank, spread, **shape), "kind": "pass", "layers": 2}
    return _layer(tokens, requests, adapters, rank, spread, **shape)


# --- inputs, from the seed alone --------------------------------------------------------------------------------------

def _rank_of(case: dict, adapter: int) -> int:
    """The rank of pool row `adapter` (1 to case["adapters"])."""
    return (8, 16, 32, 64)[adapter % 4] if case["rank"] == "mixed" else int(case["rank"])


def _cap(case: dict) -> int:
    return 64 if case["rank"] == "mixed" else int(case["rank"])


def _groups(case: dict) -> list[dict[str, tuple[list[str], list[int], int]]]:
    """Per layer, the fused groups: label -> (matrix names, outputs, inputs)."""
    if case["kind"] in ("product", "linear"):
        return [{"proj": (["up_proj"], [case["out"]], case["k"])}]
    h, inter = case["hidden"], case["inter"]
    mlp = {"gate_up": (["gate_proj", "up_proj"], [inter, inter], h), "down": (["down_proj"], [h], inter)}
    if case["kind"] == "mlp":
        return [mlp]
    kv = case["kv"]
    one = {"qkv": (["q_proj", "k_proj", "v_proj"], [h, kv, kv], h), "o": (["o_proj"], [h], h), **mlp}
    return [one] * case.get("layers", 1)


def _requests(case: dict, rng: np.random.Generator) -> tuple[np.ndarray, np.ndarray]:
    """(token offsets (requests + 1), pool row of each request): lengths of the case's spread scaled to its tokens."""
    n, tokens = case["requests"], case["tokens"]
    if case["spread"] == "one":
        cu = np.arange(n + 1)
    else:
        size = {"even": lambda: np.ones(n), "near": lambda: rng.uniform(0.8, 1.2, n),
                "uniform": lambda: rng.uniform(16, 256, n),
                "lognormal": lambda: np.clip(rng.lognormal(math.log(200.0), 1.0, n), 16, 2048)}[case["spread"]]()
        spare = tokens - n  # every request has a token
        cu = np.concatenate([[0], np.rint(np.cumsum(size) / size.sum() * spare).astype(np.int64) + np.arange(1, n + 1)])
    if case["spread"] == "lognormal":  # prefill: a few adapters take most requests
        p = np.arange(1, case["adapters"] + 1, dtype=np.float64) ** -1.1
        ids = rng.choice(case["adapters"], n, p=p / p.sum()) + 1
    else:
        ids = rng.integers(1, case["adapters"] + 1, n)
    return cu.astype(np.int32), ids.astype(np.int32)


class _Inputs:
    """Everything a case is given, as plain tensors on the GPU."""

    def __init__(self, case: dict, seed: int) -> None:
        gen = torch.Generator(device=DEVICE).manual_seed(seed)
        rng = np.random.default_rng(seed)

        def normal(*shape: int, std: float = 1.0) -> torch.Tensor:
            return torch.randn(*shape, generator=gen, device=DEVICE).mul_(std)

        if case["kind"] in ("head", "pass"):
            rows = case["adapters"] + 1
            options = case.get("options", OPTIONS)
            self.readout = normal(rows, options, case["hidden"], std=0.05).to(BF16)
            self.temperature = 0.5 + 1.5 * torch.rand(rows, generator=gen, device=DEVICE)
            self.counts = torch.tensor(rng.integers(1, options + 1, case["requests"]).astype(np.int32), device=DEVICE)
        if case["kind"] == "head":
            self.adp = torch.tensor(rng.integers(1, rows, case["requests"]).astype(np.int32), device=DEVICE)
            self.hidden = normal(case["requests"], case["hidden"]).to(BF16)
            return
        cu, ids = _requests(case, rng)
        self.cu_host, self.ids_host = cu, ids
        self.cu, self.adp = torch.tensor(cu, device=DEVICE), torch.tensor(ids, device=DEVICE)
        self.groups = _groups(case)
        width = case.get("hidden", case.get("k"))
        self.x = normal(case["tokens"], width).to(BF16)
        if case["kind"] == "mlp":
            self.d = normal(case["tokens"], width).to(BF16)
        if case["kind"] in ("layer", "pass", "mlp"):
            self.norms = [(1 + normal(width, std=0.1), 1 + normal(width, std=0.1)) for _ in self.groups]
            self.final_norm = 1 + normal(width, std=0.1)
        # weights: 4-bit codes, scales U(0.005, 0.02) and, in groups of 128, zero points; or bfloat16 N(0, 0.02)
        self.weights: list[dict] = []
        for layer in self.groups:
            made = {}
            for label, (_, sizes, k) in layer.items():
                if "group" in case:
                    g, out = case["group"], sum(sizes)
                    codes = torch.randint(0, 16, (out, k), generator=gen, device=DEVICE, dtype=torch.uint8)
                    scales = (torch.rand(out, k // g, generator=gen, device=DEVICE) * 0.015 + 0.005).to(BF16)
                    zeros = torch.randint(0, 16, (out, k // g), generator=gen, device=DEVICE, dtype=torch.uint8) \
                        if g == 128 else None
                    made[label] = (codes, scales, zeros)
                else:
                    made[label] = [normal(n, k, std=0.02).to(BF16) for n in sizes]
            self.weights.append(made)
        # adapters: A ~ N(0, 1/32), the scaled second factor ~ N(0, 0.04), per pool row, layer and matrix
        self.adapters: list[list[dict[str, list[tuple[torch.Tensor, torch.Tensor]]]]] = []
        for a in range(1, case["adapters"] + 1):
            r = _rank_of(case, a)
            shapes = [(li, label, n, k) for li, layer in enumerate(self.groups)
                      for label, (_, sizes, k) in layer.items() for n in sizes]
            flat = normal(sum(r * (n + k) for _, _, n, k in shapes)).to(BF16)
            rows: list[dict] = [{label: [] for label in layer} for layer in self.groups]
            at = 0
            for li, label, n, k in shapes:
                first = flat[at:at + r * k].view(r, k).mul_(1 / 32)
                second = flat[at + r * k:at + r * (k + n)].view(n, r).mul_(0.04)
                rows[li][label].append((first, second))
                at += r * (k + n)
            self.adapters.append(rows)


# --- what a program keeps, and one pass -------------------------------------------------------------------------------

class _State:
    pass


def prepare(case: dict, seed: int) -> _State:
    data = _Inputs(case, seed)
    st = _State()
    st.kind = case["kind"]
    if st.kind == "head":
        st.hidden, st.readout, st.temperature = data.hidden, data.readout, data.temperature
        st.adp, st.counts = data.adp, data.counts
        return st
    cap = _cap(case)
    layers = []
    for li, layer in enumerate(data.groups):
        lins = {}
        for label, (names, sizes, k) in layer.items():
            names = [f"layers.{li}.{n}" for n in names]
            ranks = [cap] * len(sizes)
            if "group" in case:
                lin = Lin(names, sizes=sizes, k=k, ranks=ranks)
                codes, scales, zeros = data.weights[li][label]
                lin.int4 = pack_kernel(codes.to(torch.int8) - 8, scales, case["group"]) if zeros is None else \
                    pack_kernel_asym(codes, scales, zeros, case["group"])
            else:
                lin = Lin(names, data.weights[li][label], ranks=ranks)
            lins[label] = lin
        layers.append(lins)
    lins = [lin for layer in layers for lin in layer.values()]
    st.pool = AdapterPool(lins, case["adapters"])
    for a, rows in enumerate(data.adapters, 1):
        updates = {name: pair for li, layer in enumerate(layers) for label, lin in layer.items()
                   for name, pair in zip(lin.names, rows[li][label])}
        st.pool.add_adapter(f"adapter-{a}", updates)
    data.adapters.clear()
    st.layers, st.tokens, st.pool_rows = layers, case["tokens"], case["adapters"] + 1
    st.adp, st.x = data.adp, data.x
    st.cu = None if case["spread"] == "one" else data.cu
    st.ws = Workspace(case["tokens"], 1, {(lin.k, lin.out) for lin in lins},
                      max_rank=max(lin.rank for lin in lins), max_requests=case["requests"])
    if st.kind == "layer":
        st.norms = data.norms[0]
        st.recorded = RecordedPass(lambda: _layer_body(st))
    elif st.kind == "pass":
        ends = (data.cu[1:] - 1).to(torch.int64)
        st.batch = (data.x, data.adp, data.cu, ends, data.counts)
        st.inputs = DecoderInputs(data.x.clone(), data.adp.clone(), data.cu.clone(), ends.clone(), data.counts.clone())
        st.readout, st.temperature = data.readout, data.temperature
        st.recorded = RecordedPass(decoder_pass(layers, data.norms, data.final_norm, st.ws, st.inputs, st.tokens,
                                                st.readout, st.temperature))
    elif st.kind == "product":
        st.last = torch.empty(case["requests"], case["out"], device=DEVICE, dtype=BF16)
    elif st.kind == "mlp":
        st.d, st.norm = data.d, data.norms[0][0]
    return st


def _layer_body(st: _State) -> tuple[torch.Tensor, ...]:
    layer, ws, adp = st.layers[0], st.ws, st.adp
    ws.route(adp, st.pool_rows, tokens=st.tokens, cu_seqlens=st.cu)
    x = st.x.clone()  # the residual stream
    qkv = int4_product(layer["qkv"], rms(x, st.norms[0]), ws, adp)
    # the query columns stand in for attention's output
    int4_product(layer["o"], qkv[:, :layer["o"].k], ws, adp, epilogue="residual", residual=x)
    act = int4_product(layer["gate_up"], rms(x, st.norms[1]), ws, adp, epilogue="silu_mul")
    int4_product(layer["down"], act, ws, adp, epilogue="residual", residual=x)
    return qkv, act, x


def run(st: _State):
    if st.kind == "layer":
        return st.recorded.replay()
    if st.kind == "pass":
        into = st.inputs
        for recorded, rows in zip((into.x, into.adp, into.cu_seqlens, into.ends, into.counts), st.batch):
            recorded.copy_(rows)
        return st.recorded.replay()
    if st.kind == "head":
        return readout_rows(st.hidden, st.readout, st.temperature, st.adp, st.counts)
    ws, layer = st.ws, st.layers[0]
    ws.route(st.adp, st.pool_rows, tokens=st.tokens, cu_seqlens=st.cu)
    if st.kind == "product":
        return int4_product(layer["proj"], st.x, ws, st.adp, last_out=st.last), st.last
    if st.kind == "linear":
        return layer["proj"](st.x, ws, st.adp)
    x, h = add_rms(st.x, st.d, st.norm)
    act = silu_mul(layer["gate_up"](h, ws, st.adp))
    return x, act, layer["down"](act, ws, st.adp)


# --- what a pass cannot do without, and what its results may differ by ------------------------------------------------

def _present(case: dict) -> float:
    """Expected number of distinct adapters among the requests, each adapter taken alike."""
    n = case["adapters"]
    if case.get("spread") == "lognormal":
        p = np.arange(1, n + 1, dtype=np.float64) ** -1.1
        return float((1 - (1 - p / p.sum()) ** case["requests"]).sum())
    return n * (1 - (1 - 1 / n) ** case["requests"])


def work(case: dict) -> dict:
    present = _present(case)
    if case["kind"] == "head":
        n, dim, options = case["requests"], case["hidden"], case["options"]
        return {"bytes": 2 * present * options * dim + n * (2 * dim + 4 * options + 8),
                "flops": 2 * n * options * dim}
    tokens = case["tokens"]
    rank = float(np.mean([_rank_of(case, a) for a in range(1, case["adapters"] + 1)]))
    nbytes, flops = 8.0 * case["requests"], 0.0
    for layer in _groups(case):
        for _, sizes, k in layer.values():
            out = sum(sizes)
            if "group" in case:  # codes, scales and, in groups of 128, zero points
                nbytes += out * k / 2 + out * (k // case["group"]) * (3 if case["group"] == 128 else 2)
            else:
                nbytes += 2 * out * k
            nbytes += sum(2 * present * rank * (k + n) for n in sizes)
            flops += 2 * tokens * k * out + sum(2 * tokens * rank * (k + n) for n in sizes)
    if case["kind"] in ("product", "linear"):
        nbytes += 2 * tokens * (case["k"] + case["out"])
        if case["kind"] == "product":
            nbytes += 2 * case["requests"] * case["out"]
    elif case["kind"] == "pass":
        h, n = case["hidden"], case["requests"]
        nbytes += 2 * tokens * h + 2 * present * OPTIONS * h + n * 4 * OPTIONS
        flops += 2 * n * OPTIONS * h
    else:
        h = case["hidden"]
        extra = h + 2 * case["kv"] if case["kind"] == "layer" else 2 * h  # qkv out; or the second input and result
        nbytes += 2 * tokens * (2 * h + case["inter"] + extra)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict) -> dict:
    """Outputs are bfloat16 sums (one rounding is 1.7e-3 of a result in the 2-norm). About four times what the same
    work shows with its sums in another order (the products' other kernels): through a layer, a flipped last place of
    qkv or of a norm travels on (1.1e-3, largest difference 0.019); through a whole pass to the probabilities 5.6e-3
    and 0.061. A lone product shows under 1e-4 and one last place, 0.008. The head flips only logits at a rounding
    boundary (a last place is up to 3% of a probability at the largest logits and half that temperature)."""
    if case["kind"] in ("product", "linear"):
        return {"rel": 1e-3, "max": 0.03}
    if case["kind"] == "head":
        return {"rel": 4e-3, "max": 0.1}
    if case["kind"] == "pass":
        return {"rel": 2.2e-2, "max": 0.25}
    return {"rel": 5e-3, "max": 0.08}


# --- the results in 64 bits -------------------------------------------------------------------------------------------

def _norm64(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt((x * x).mean(dim=1, keepdim=True) + 1e-6) * w.double()


class _Exact:
    """The groups' products in 64 bits: weights are the bfloat16 values that codes, scales and zero points stand for."""

    def __init__(self, case: dict, data: _Inputs) -> None:
        self.data = data
        self.rows = np.repeat(data.ids_host, np.diff(data.cu_host))  # each token's pool row
        self.weights = []
        for layer in data.weights:
            made = {}
            for label, w in layer.items():
                if "group" in case:
                    codes, scales, zeros = w
                    z = 8.0 if zeros is None else zeros.float().repeat_interleave(case["group"], 1)
                    made[label] = ((codes.float() - z) * scales.float().repeat_interleave(case["group"], 1)).to(BF16)
                else:
                    made[label] = torch.cat(list(w))
            self.weights.append(made)

    def product(self, li: int, label: str, x: torch.Tensor, t0: int) -> torch.Tensor:
        """Rows t0 .. of the pass through a group, in 64 bits."""
        w = self.weights[li][label].double()
        y = x @ w.T.contiguous()
        _, sizes, _ = self.data.groups[li][label]
        rows = self.rows[t0:t0 + x.shape[0]]
        order = np.argsort(rows, kind="stable")
        ids, starts = np.unique(rows[order], return_index=True)
        index = torch.from_numpy(order).to(DEVICE)
        for a, s, e in zip(ids, starts, np.append(starts[1:], len(rows))):
            at = index[int(s):int(e)]
            xs, col = x[at], 0
            for n, (first, second) in zip(sizes, self.data.adapters[int(a) - 1][li][label]):
                y[at, col:col + n] += (xs @ first.double().T.contiguous()) @ second.double().T.contiguous()
                col += n
        return y


def exact(case: dict, seed: int):
    data = _Inputs(case, seed)
    if case["kind"] == "head":
        return _head64(data.hidden.double(), data)
    ex = _Exact(case, data)
    chunks = []
    for t0 in range(0, case["tokens"], 16384):
        chunks.append(_rows64(case, data, ex, t0, min(t0 + 16384, case["tokens"])))
    outs = tuple(torch.cat(parts) for parts in zip(*chunks))
    if case["kind"] == "pass":
        last = outs[0][data.cu[1:].long() - 1]
        return _head64(_norm64(last, data.final_norm), data)
    if case["kind"] == "linear":
        return outs[0]
    if case["kind"] == "product":
        return outs[0], outs[0][data.cu[1:].long() - 1]
    return outs


def _rows64(case: dict, data: _Inputs, ex: _Exact, t0: int, t1: int) -> tuple[torch.Tensor, ...]:
    """Rows t0 .. t1 - 1 of the case's outputs (of a pass: its residual stream)."""
    x = data.x[t0:t1].double()
    if case["kind"] in ("product", "linear"):
        return (ex.product(0, "proj", x, t0),)
    inter = case["inter"]
    if case["kind"] == "mlp":
        x = x + data.d[t0:t1].double()
        gu = ex.product(0, "gate_up", _norm64(x, data.norms[0][0]), t0)
        act = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
        return x, act, ex.product(0, "down", act, t0)
    for li in range(len(data.groups)):
        qkv = ex.product(li, "qkv", _norm64(x, data.norms[li][0]), t0)
        x = x + ex.product(li, "o", qkv[:, :case["hidden"]], t0)
        gu = ex.product(li, "gate_up", _norm64(x, data.norms[li][1]), t0)
        act = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
        x = x + ex.product(li, "down", act, t0)
    return (x,) if case["kind"] == "pass" else (qkv, act, x)


def _head64(hidden: torch.Tensor, data: _Inputs) -> torch.Tensor:
    rows = data.adp.long()
    logits = torch.empty(hidden.shape[0], data.readout.shape[1], device=DEVICE, dtype=torch.float64)
    for i in range(0, len(rows), 64):  # 64 requests' readouts at a time
        logits[i:i + 64] = (data.readout[rows[i:i + 64]].double() * hidden[i:i + 64, None, :]).sum(dim=2)
    option = torch.arange(logits.shape[1], device=DEVICE)
    logits = torch.where(option < data.counts[:, None], logits, -1e9)
    return torch.softmax(logits / data.temperature.double()[rows][:, None], dim=1)
