"""The sliced product (csrc/sliced.hip: the inputs sliced over a workgroup's waves) and the first factors in 32-row tiles
(shrink_rows_kernel) at the sizes where they can go wrong, against the oracle's bound (needs a gfx950 GPU; marked gpu):
row counts around the tiles' 32, 64 and 96 rows in each of the four forms, chunk counts that do not divide over the
slices or fill the ring, columns of several matrices in one tile, ranks past one 64-rank pass, every adapter segment
pattern (one, several, one per row, the base row among them) and the three epilogues, whose bits must agree."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from jeff_amd import _lib
from jeff_amd.epilogues import silu_mul
from jeff_amd.fast_path import DT, Workspace
from jeff_amd.int4_kernels import int4_product
from oracle.layer import exact_and_bound, step, within_tolerance
from tests.gpu_cases import Case, make_case, oracle_adapters, reference_f32_gpu, token_ids

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu() -> None:
    assert torch.cuda.is_available(), "the gpu tests need an AMD GPU"
    _lib.lib()


# name: (lengths of the requests, matrix widths, inputs, group, rank capacities, live ranks by adapter)
CASES = {
    "one-row-past": ([33], [320], 576, 64, [16], {1: [16]}),               # 9 chunks over 8 slices
    "one-chunk": ([20, 12], [64], 64, 64, [8], {1: [8], 2: [3]}),           # 7 slices hold no chunk
    "mixed": ([40, 1, 0, 22, 90], [104, 24, 200], 1600, 64, [16, 24, 0],  # matrices change inside a tile, 25 chunks
              {1: [16, 24, 0], 2: [3, 17, 0], 3: [0, 9, 0]}),
    "big-ranks": ([64, 65], [128, 96], 256, 128, [128, 72], {1: [128, 72], 2: [65, 40]}),
    "rows-64": ([191, 192], [2048], 576, 64, [32], {1: [32], 2: [24]}),        # 64-row tiles, 8 slices
    "rows-64-wide": ([129, 255], [2048, 1024, 1000], 832, 64, [16, 16, 16],    # 64-row tiles, 4 slices, 13 chunks
                     {1: [16, 8, 16], 2: [9, 16, 0]}),
    "rows-96": ([97, 286], [6144, 6144], 192, 64, [64, 64], {1: [64, 40], 2: [8, 64]}),  # 96-row tiles, 3 chunks
    "short": ([1] * 300, [2048], 512, 128, [64], {a: [(8, 16, 32, 64)[a % 4]] for a in range(1, 41)}),
}


def routed(lengths: list[int], adapters: int, pool_rows: int, seed: int, ws_rank: int):
    rng = np.random.default_rng(seed)
    adp = torch.tensor(rng.integers(0, adapters + 1, len(lengths)).astype(np.int32), device="cuda")
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32), device="cuda")
    tokens = int(sum(lengths))
    ws = Workspace(tokens, 1, max_rank=ws_rank, max_requests=len(lengths))
    ws.route(adp, pool_rows, tokens=tokens, cu_seqlens=cu)
    return ws, adp, cu


def assert_within_bound(case: Case, x: torch.Tensor, tok_adp: np.ndarray, got: torch.Tensor) -> None:
    """The output within the forward error bound of exact arithmetic, the first factors' rounding at its largest.
    Rounding a value to bfloat16's 8 significant bits costs up to 2^-8 of it; the oracle's bound prices that at 2^-9,
    which holds where many ranks average it out and not at the few ranks of these cases (8 and 3 live ranks, 64 inputs: a
    correct result, float64 sums and the two roundings, passes it in 77 of 300 draws, by up to 1.35 times). So
    |got - exact| <= p + step(|exact| + p) / 2 with p = slack + 2^-8 |x A^T| |sB|^T; `slack + 2^-9 ...` is at most the
    oracle's bound less step(|exact|) / 2."""
    lin = case.lin
    adapters = oracle_adapters(lin, np.unique(tok_adp))
    xc = x.cpu()
    exact, bound = exact_and_bound(xc, case.w, tok_adp, adapters, lin.sizes, lin.rank)
    p = bound - step(exact.abs()) / 2
    edges = np.concatenate([[0], np.cumsum(lin.sizes)]).astype(int)
    for a, updates in adapters.items():
        idx = torch.from_numpy(np.nonzero(tok_adp == a)[0])
        for j, upd in enumerate(updates):
            if upd is not None and len(idx):
                a_mat, sb = (t.double() for t in upd)
                lora = 2.0 ** -9 * ((xc[idx].double() @ a_mat.T).abs() @ sb.abs().T)
                p[idx, int(edges[j]):int(edges[j + 1])] += lora
    err = (got.cpu().double() - exact).abs()
    worst = float((err / (p + step(exact.abs() + p) / 2)).max())
    assert bool(torch.isfinite(got.float()).all()) and worst <= 1.0, worst
    assert bool(within_tolerance(got, reference_f32_gpu(lin, case.w, x, tok_adp)).all())


def normal(rows: int, cols: int, seed: int) -> torch.Tensor:
    return torch.randn(rows, cols, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda").to(DT)


@pytest.mark.parametrize("name", list(CASES))
def test_sliced_products_are_within_the_bound(name: str) -> None:
    lengths, sizes, k, group, caps, ranks = CASES[name]
    print(f"sliced {name}", flush=True)
    case = make_case(sizes, k, group, group == 128, ranks, caps, 7 + len(name))
    lin = case.lin
    ws, adp, cu = routed(lengths, len(ranks), lin.pool.shape[0], len(name), lin.rank)
    tokens = int(sum(lengths))
    x = normal(tokens, k, tokens)
    last = torch.zeros(len(lengths), lin.out, dtype=DT, device="cuda")
    got = int4_product(lin, x, ws, adp, last_out=last)
    ends = np.cumsum(lengths) - 1
    for i, n in enumerate(lengths):
        if n:
            assert torch.equal(last[i], got[int(ends[i])]), f"{name}: last row of request {i}"
    assert_within_bound(case, x, token_ids(adp, lin.pool.shape[0], cu=cu), got)
    assert torch.equal(got, int4_product(lin, x, ws, adp)), f"{name}: two runs differ"
    res0 = normal(tokens, lin.out, tokens + 1)
    res = res0.clone()
    int4_product(lin, x, ws, adp, epilogue="residual", residual=res)
    assert torch.equal(res, (res0.float() + got.float()).to(DT)), f"{name}: the residual epilogue's bits"
    if len(sizes) == 2 and sizes[0] == sizes[1] and sizes[0] % 128 == 0 and caps[0] == caps[1] <= 64:
        assert torch.equal(int4_product(lin, x, ws, adp, epilogue="silu_mul"), silu_mul(got)), f"{name}: gated bits"


def test_an_infinity_stays_in_its_row() -> None:
    """One infinite input: its row is infinite (or NaN where the weight is zero), every other row unchanged, also where
    a slice has no chunk in the last step (its weights are then zero, and 0 * inf would be NaN)."""
    k = 576  # 9 chunks over 8 slices
    case = make_case([128], k, 64, False, {1: [8]}, [8], 3)
    lin = case.lin
    ws, adp, _ = routed([40], 0, lin.pool.shape[0], 1, lin.rank)
    x = normal(40, k, 40)
    want = int4_product(lin, x, ws, adp)
    for at in (3, 64 + 5, 575):
        xi = x.clone()
        xi[17, at] = float("inf")
        got = int4_product(lin, xi, ws, adp)
        keep = torch.arange(40, device="cuda") != 17
        assert torch.equal(got[keep], want[keep])
        w = case.w[:, at].cuda().float()
        assert torch.equal(torch.isnan(got[17]), w == 0)
        assert torch.equal(got[17][w != 0].float(), torch.sign(w[w != 0]) * float("inf"))
