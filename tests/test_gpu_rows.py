"""keep_vq_rows, the routed mat-vecs on the matrix cores, against the float64
oracle: 8-bit E8 and E8P codes, fp16 and bf16 rows, one and several K slices
(groups of waves that fill the block or leave some idle), units past the last
output, per-row and grouped scales, odd scale counts, tiles of one route, of
exactly 16 and of more (one expert, one matrix), routes planned in the kernel
(<= 128) and by a route plan, experts and rows out of range (NaN), and the
same bits whatever the grouping."""

import numpy as np
import pytest
import torch

import keep_amd
from keep_amd import ops as kops
from oracle import e8p, ops

pytestmark = pytest.mark.gpu
TOL = 2e-3


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a.view(np.int16) if a.dtype == np.uint16 else a)).to(dev)


def _make(E, N, K, G, bits, seed, sdt=np.float16):
    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 1 << bits, (E, N, K // 8)).astype(np.uint8 if bits == 8 else np.uint16)
    scales = np.exp(rng.normal(0, 0.3, (E, N, G))).astype(sdt)
    vals = (e8p.decode_e8_1bit(codes) if bits == 8 else e8p.decode_e8p(codes)).astype(np.float64)
    return codes, scales, vals.reshape(E, N, K) * np.repeat(scales.astype(np.float64), K // G, -1)


def _check(got, want, xdt):
    # the fp32 sums, then one rounding to the rows' type
    ulp = 2.0 ** -11 if xdt == torch.float16 else 2.0 ** -8
    assert ops.max_rel_err(got, want) <= TOL + ulp
    assert ops.elementwise_ok(got, want, rtol=TOL + ulp)


CASES = [(8, torch.float16, 3, 32, 512, 1), (8, torch.bfloat16, 5, 65, 1536, 3), (8, torch.float16, 4, 96, 4096, 8),
         (8, torch.bfloat16, 2, 33, 3584, 1), (8, torch.float16, 2, 40, 8192, 4), (16, torch.float16, 3, 32, 256, 1),
         (16, torch.float16, 4, 71, 1280, 5), (16, torch.float16, 2, 64, 4096, 1)]


@pytest.mark.parametrize("bits,xdt,E,N,K,G", CASES)
def test_rows_vs_oracle_and_grouping(dev, bits, xdt, E, N, K, G):
    codes, scales, dense = _make(E, N, K, G, bits, seed=N + K, sdt=np.float32 if N == 71 else np.float16)
    rng = np.random.default_rng(K)
    cb = kops._default_codebook(bits, dev)
    kw = dict(input_dims=K, output_dims=N, group_size=K // G, code_bits=bits)
    c, s = _t(codes, dev), _t(scales, dev)
    for T, k in ((1, 1), (7, 3), (50, 3)):  # 150 routes: a route plan
        x = torch.from_numpy(rng.standard_normal((T, K)).astype(np.float32)).to(dev).to(xdt)
        rhs = rng.integers(0, E, (T, k)).astype(np.int32)
        if T == 7:
            rhs[2, 1], rhs[5, 0] = E, -3
            rhs[:, 2] = 0
        flat = _t(rhs.reshape(-1), dev)
        assert kops.rows_eligible(x, c, s, cb, code_bits=bits, input_dims=K, group_size=K // G)
        y = kops.rows_matvec(x, c, s, cb, flat, x_div=k, grouped=True, **kw)
        z = kops.rows_matvec(x, c, s, cb, flat, x_div=k, grouped=False, **kw)
        good = (rhs.reshape(-1) >= 0) & (rhs.reshape(-1) < E)
        yc = y.float().cpu().numpy()
        assert np.isnan(yc[~good]).all() and not np.isnan(yc[good]).any()
        assert np.array_equal(yc, z.float().cpu().numpy(), equal_nan=True)
        xd = x.double().cpu().numpy()
        want = np.stack([dense[e] @ xd[i // k] for i, e in enumerate(rhs.reshape(-1)) if 0 <= e < E])
        _check(yc[good], want, xdt)
    lhs = _t(np.array([3, 0, 60, 2], np.int32), dev)  # row 60 is out of range
    w = kops.rows_matvec(x, c, s, cb, _t(np.array([1, 0, 1, 1], np.int32), dev), lhs=lhs, grouped=True, **kw)
    wc = w.float().cpu().numpy()
    assert np.isnan(wc[2]).all()
    _check(wc[[0, 1, 3]], np.stack([dense[1] @ xd[3], dense[0] @ xd[0], dense[1] @ xd[2]]), xdt)


@pytest.mark.parametrize("bits,xdt,E,N,K,G", CASES)
@pytest.mark.parametrize("M", [1, 16, 17, 49])
def test_rows_one_matrix_vs_oracle(dev, bits, xdt, E, N, K, G, M):
    codes, scales, dense = _make(1, N, K, G, bits, seed=N + K)
    x = torch.from_numpy(np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)).to(dev).to(xdt)
    y = kops.rows_matvec(x, _t(codes, dev), _t(scales, dev), kops._default_codebook(bits, dev), None, input_dims=K,
                         output_dims=N, group_size=K // G, code_bits=bits)
    _check(y.float().cpu().numpy(), x.double().cpu().numpy() @ dense[0].T, xdt)


def test_rows_through_the_operators(dev):
    """Sizes at which vq_qmm, gather_vqmm (direct and sorted) and the verify
    operator take the rows kernel, replayed in a graph: every replay equals
    the eager call, and the verify groupings agree with the single-row gather."""
    E, N, K, G, T, k = 6, 1024, 2048, 4, 5, 3
    codes, scales, dense = _make(E, N, K, G, 8, seed=9)
    c, s = _t(codes, dev), _t(scales, dev)
    rng = np.random.default_rng(10)
    x = torch.from_numpy(rng.standard_normal((T, K)).astype(np.float16)).to(dev)
    rhs = _t(rng.integers(0, E, (T, k)).astype(np.int32), dev)
    kw = dict(input_dims=K, output_dims=N, group_size=K // G)
    assert N * K >= kops.ROWS_MATRIX
    calls = {
        "expert": lambda: kops.gather_vqmm_verify_rows(x, c, s, None, rhs, grouping="expert", **kw),
        "flat": lambda: kops.gather_vqmm_verify_rows(x, c, s, None, rhs, grouping="flat", **kw),
        "direct": lambda: kops.gather_vqmm(x, c, s, None, rhs, code_bits=8, **kw),
        "sorted": lambda: kops.gather_vqmm(x, c, s, None, rhs, code_bits=8, route_strategy="sorted_tiled", **kw),
        "qmm": lambda: kops.vq_qmm(x.repeat(8, 1), c[0], s[0], in_dim=K, out_dim=N, group_size=K // G),
    }
    with keep_amd.trace_gather_vqmm_calls() as tr:
        eager = {n: f() for n, f in calls.items()}
    assert [t["implementation"] for t in tr] == ["mfma_rows"] * 4
    torch.cuda.synchronize()
    for n in ("flat", "direct", "sorted"):
        assert torch.equal(eager["expert"], eager[n]), n
    one = kops.gather_vqmm(x[2:3], c, s, None, rhs[2:3], code_bits=8, **kw)
    assert torch.equal(one[0], eager["flat"][2])
    xd, r = x.double().cpu().numpy(), rhs.cpu().numpy()
    _check(eager["expert"].float().cpu().numpy(), np.stack([[dense[e] @ xd[t] for e in r[t]] for t in range(T)]),
           torch.float16)
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        held = {n: f() for n, f in calls.items()}
    for _ in range(3):
        for h in held.values():
            h.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for n in calls:
            assert torch.equal(held[n], eager[n]), n


@pytest.mark.parametrize("bits, xdt", [(8, torch.float16), (8, torch.bfloat16), (16, torch.float16)])
def test_rows_non_finite_rows(dev, bits, xdt):
    """Infinities and NaN in a row: the plain product's, for that row's routes alone."""
    E, N, K, G, T, k = 3, 72, 1024, 2, 9, 2
    codes, scales, dense = _make(E, N, K, G, bits, seed=bits)
    rng = np.random.default_rng(7)
    x = torch.from_numpy(rng.standard_normal((T, K)).astype(np.float32)).to(dev).to(xdt)
    inf = float("inf")
    for r, vals in {1: {5: inf}, 2: {K - 1: -inf}, 3: {7: inf, 90: -inf}, 4: {9: float("nan")}, 8: {700: inf}}.items():
        for i, v in vals.items():
            x[r, i] = v
    rhs = rng.integers(0, E, T * k).astype(np.int32)
    y = kops.rows_matvec(x, _t(codes, dev), _t(scales, dev), kops._default_codebook(bits, dev), _t(rhs, dev), x_div=k,
                         grouped=True, input_dims=K, output_dims=N, group_size=K // G, code_bits=bits)
    xd = x.double().cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = np.stack([(dense[e] * xd[i // k]).sum(1) for i, e in enumerate(rhs)])
    got = y.double().cpu().numpy()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    good = np.isfinite(want).all(1)
    _check(got[good], want[good], xdt)


def _units(bits, N, K, tiles, n_tiles):
    """(units per group of waves, whether a group's run crosses tiles), as the launch shares them out: a group of
    K / 512 (E8P: / 256) of a block's 16 waves, units of 32 columns, up to 256 blocks."""
    upt, groups = -(-N // 32), 16 // (K // (512 if bits == 8 else 256))
    per = -(-tiles * upt // (min(n_tiles * upt, 256) * groups))
    return per, any((u // upt) != ((min(u + per, tiles * upt) - 1) // upt) for u in range(0, tiles * upt, per))


# K slices that leave one, two and sixteen groups per block; ragged last units; odd counts of scales and rows
LONG = [(8, torch.float16, 90, 520, 8192, 16), (8, torch.bfloat16, 110, 1031, 3584, 7),
        (16, torch.float16, 90, 520, 4096, 1), (8, torch.bfloat16, 90, 1080, 4096, 8)]


@pytest.mark.parametrize("bits,xdt,E,N,K,G", LONG)
@pytest.mark.parametrize("form", ["planned", "plan", "flat", "matrix"])
def test_rows_long_runs_vs_oracle(dev, bits, xdt, E, N, K, G, form):
    """At least five units per group of waves: code buffers refilled, both
    partial-sum buffers used again, and runs that cross from one expert's tile
    (or one matrix's rows) to the next, invalid routes among them."""
    g = torch.Generator(device=dev).manual_seed(K + N)
    one = form == "matrix"
    E = 1 if one else E
    codes = torch.randint(0, 256, (E, N, K // 8 * (bits // 8)), dtype=torch.uint8, device=dev, generator=g)
    grid = e8p.decode_e8_1bit(np.arange(256, dtype=np.uint8)) if bits == 8 else e8p.e8p_full_grid()
    grid = torch.from_numpy(grid.astype(np.float32)).to(dev)
    index = codes if bits == 8 else (codes.view(torch.int16).int() & 0xFFFF)
    codes = codes if bits == 8 else codes.view(torch.int16)
    scales = torch.exp(0.3 * torch.randn((E, N, G), device=dev, generator=g)).half()
    T, k = {"planned": (32, 4), "plan": (70, 4), "flat": (32, 4), "matrix": (2055, 1)}[form]
    x = torch.randn((T, K), device=dev, generator=g).to(xdt)
    kw = dict(input_dims=K, output_dims=N, group_size=K // G, code_bits=bits)
    cb = kops._default_codebook(bits, dev)

    def dense(e):
        return grid[index[e].int()].reshape(N, K).double() * scales[e].double().repeat_interleave(K // G, 1)

    if one:
        tiles = n_tiles = -(-T // 16)
        y = kops.rows_matvec(x, codes, scales, cb, None, **kw)
        want = x.double() @ dense(0).T
        good = torch.ones(T, dtype=torch.bool, device=dev)
    else:
        rhs = torch.randint(0, E, (T * k,), device=dev, generator=g, dtype=torch.int32)
        rhs[[5, 61, 90]] = torch.tensor([E, -2, E + 7], dtype=torch.int32, device=dev)
        flat = rhs.cpu().numpy()
        good = (rhs >= 0) & (rhs < E)
        count = np.bincount(np.where((flat < 0) | (flat >= E), E, flat), minlength=E + 1)
        tiles = n_tiles = T * k
        if form != "flat":
            tiles = int((-(-count // 16)).sum())
        if form == "plan":
            tiles = n_tiles = min(-(-T * k // 16) + E, T * k)
        y = kops.rows_matvec(x, codes, scales, cb, rhs, x_div=k, grouped=form != "flat", **kw)
        want = torch.zeros((T * k, N), dtype=torch.float64, device=dev)
        for e in np.unique(flat[good.cpu().numpy()]):
            r = torch.nonzero(rhs == int(e))[:, 0]
            want[r] = x[r // k].double() @ dense(int(e)).T
    per, crosses = _units(bits, N, K, tiles, n_tiles)
    assert per >= 5 and crosses, (per, crosses)
    y = y.float().cpu().numpy()
    good = good.cpu().numpy()
    assert np.isnan(y[~good]).all()
    _check(y[good], want.cpu().numpy()[good], xdt)
