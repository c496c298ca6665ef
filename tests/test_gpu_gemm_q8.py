"""GPU parity of the prefill grouped GEMM (keep_vq_grouped_gemm_q8, fp16
matrix cores) and its fused gate/up + SwiGLU form (keep_vq_grouped_swiglu_q8)
against the float64 oracle: partial column blocks, tiles of one and two
32-route m-tiles, per-row and grouped scales, fp16 / bf16 / fp32
activations, work items of 256 and of 512 columns, the scatter back to route
order, and NaN rows / out-of-range experts (the sorted-route prefill of
src/ramp/ops/vq_switch.py:620-913 and src/ramp/models/glm4_moe_adapter.py:274-353)."""

import numpy as np
import pytest
import torch

import keep_amd
from keep_amd import ops as kops
from keep_amd import synth
from oracle import cpu, e8p, ops

pytestmark = pytest.mark.gpu
TOL = 2e-3


def _t(a, dev):
    if a.dtype == np.uint16:
        a = a.view(np.int16)
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _check(got, want, tol=TOL):
    g = got.float().cpu().numpy()
    err = ops.max_rel_err(g, want)
    assert err <= tol, f"max rel err {err:.3e}"
    assert ops.elementwise_ok(g, want, rtol=tol), "elementwise bound violated"
    return err


def _plan(rhs, E, k, dev):
    flat = _t(rhs.reshape(-1).astype(np.int32), dev)
    order, inverse, counts, _, te, to, tc, _ = keep_amd.route_plan(flat, E, 64)
    lhs = (torch.arange(flat.numel(), device=dev, dtype=torch.int32) // k)[order.long()].contiguous()
    return flat, order, inverse, counts, (te, to, tc), lhs


@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("G", [1, 4])
def test_grouped_gemm_q8_vs_oracle(dev, xdt, G):
    """N = 320: a full and a partial 256-column block; Zipf routing gives
    experts with > 64, 33..64 and <= 32 routes."""
    E, N, K, T, k = 12, 320, 512, 100, 4
    codes, scales = synth.projection_np(E, N, K, group_size=K // G, seed=G)
    rhs = synth.zipf_routes(T, E, k, seed=3)
    x = synth.rht_activations(T, K, seed=4, device=dev, dtype=xdt)
    flat, order, inverse, counts, tiles, lhs = _plan(rhs, E, k, dev)
    c = counts.cpu().numpy()
    assert c.max() > 64 and ((c > 32) & (c <= 64)).any() and ((c > 0) & (c <= 32)).any()
    cb = kops._default_codebook(16, dev)
    want = ops.gather_token(x.float().cpu().numpy(), codes, scales, rhs)
    y = kops.grouped_gemm(x, _t(codes, dev), _t(scales, dev), cb, tiles, lhs=lhs, routes=flat.numel(),
                          input_dims=K, output_dims=N, group_size=K // G, out_dtype=torch.float32)
    _check(y[inverse.long()].reshape(T, k, N), want)
    # the same rows scattered straight to route order
    y2 = kops.grouped_gemm(x, _t(codes, dev), _t(scales, dev), cb, tiles, lhs=lhs, routes=flat.numel(),
                           input_dims=K, output_dims=N, group_size=K // G, out_dtype=torch.float32, out_index=order)
    assert torch.equal(y2, y[inverse.long()])


@pytest.mark.parametrize("limit", [0.0, 7.0])
def test_grouped_swiglu_q8_vs_oracle(dev, limit):
    """I = 320: two full 128-row blocks and a partial one."""
    E, H, I, T, k = 10, 512, 320, 60, 3
    gate = synth.projection_np(E, I, H, seed=31)
    up = synth.projection_np(E, I, H, seed=32)
    rhs = synth.zipf_routes(T, E, k, seed=33)
    x = synth.rht_activations(T, H, seed=34, device=dev)
    flat, order, inverse, _, tiles, lhs = _plan(rhs, E, k, dev)
    cb = kops._default_codebook(16, dev)
    h = kops.grouped_swiglu(x, _t(gate[0], dev), _t(gate[1], dev), _t(up[0], dev), _t(up[1], dev), cb, tiles,
                            lhs=lhs, routes=flat.numel(), input_dims=H, hidden_dims=I, group_size=H, limit=limit)
    xf = x.float().cpu().numpy()
    g = ops.gather_token(xf, gate[0], gate[1], rhs)
    u = ops.gather_token(xf, up[0], up[1], rhs)
    want = ops.round_bf16(ops.swiglu(g, u, limit))
    # bf16-stored h on both sides: two nearly equal values can round one bf16
    # ulp apart, 2**-7 of the smaller where they straddle a power of two
    _check(h[inverse.long()].reshape(T, k, I), want, TOL + 2.0 ** -7)


def test_grouped_gemm_q8_nan_row_and_bad_expert(dev):
    E, N, K, T, k = 4, 256, 256, 40, 2
    codes, scales = synth.projection_np(E, N, K, seed=41)
    rng = np.random.default_rng(42)
    rhs = rng.integers(0, E, size=(T, k)).astype(np.int32)
    rhs[5, 1] = 7  # out of range: its route's row is NaN
    x = synth.rht_activations(T, K, seed=43, device=dev)
    x[9, 17] = float("nan")  # token 9's routes are NaN
    flat = _t(rhs.reshape(-1), dev)
    order, inverse, _, _, te, to, tc, _ = keep_amd.route_plan(flat, E, 64)  # expert 7: a tile of expert -1
    lhs = (torch.arange(flat.numel(), device=dev, dtype=torch.int32) // k)[order.long()].contiguous()
    cb = kops._default_codebook(16, dev)
    y = kops.grouped_gemm(x, _t(codes, dev), _t(scales, dev), cb, (te, to, tc), lhs=lhs, routes=flat.numel(),
                          input_dims=K, output_dims=N, group_size=K, out_dtype=torch.float32,
                          out_index=order).reshape(T, k, N).cpu()
    bad = np.zeros((T, k), dtype=bool)
    bad[5, 1] = True
    bad[9, :] = True
    assert torch.isnan(y[torch.from_numpy(bad)]).all()
    good = ~bad
    assert not torch.isnan(y[torch.from_numpy(good)]).any()
    rr = np.where(rhs < E, rhs, 0)
    want = ops.gather_token(np.nan_to_num(x.float().cpu().numpy()), codes, scales, rr)
    _check(y[torch.from_numpy(good)], want[good])


@pytest.mark.parametrize("G", [1, 2])
def test_grouped_residual_add_vs_oracle(dev, G):
    """The 8-bit E8 residual form: tiles of routes grouped by residual row
    (route_plan over the routes' rows, -1 = none, sorted past every tile) add
    R[row] . x into an fp32 output at out_index; routes off the tier keep
    their value."""
    from oracle import e8p

    Hh, N, K, T, k = 5, 320, 512, 60, 3
    rng = np.random.default_rng(101)
    rc = rng.integers(0, 256, (Hh, N, K // 8), dtype=np.uint8)
    rs = (np.exp(rng.normal(0, 0.3, (Hh, N, G))) * 0.1).astype(np.float16)
    dense = e8p.decode_e8_1bit(rc).astype(np.float64).reshape(Hh, N, K) * np.repeat(rs.astype(np.float64), K // G, -1)
    rows = rng.integers(-1, Hh, size=T * k).astype(np.int32)
    x = synth.rht_activations(T, K, seed=102, device=dev)
    flat = _t(rows, dev)
    order, _, _, _, te, to, tc, _ = keep_amd.route_plan(flat, Hh, 64)
    lhs = (torch.arange(T * k, device=dev, dtype=torch.int32) // k)[order.long()].contiguous()
    base = torch.randn(T * k, N, device=dev)
    out = base.clone()
    kops.grouped_residual_add(out, x, _t(rc, dev), _t(rs, dev), (te, to, tc), lhs=lhs, out_index=order,
                              routes=T * k, input_dims=K, output_dims=N, group_size=K // G)
    xf = x.float().cpu().numpy().astype(np.float64)
    want = np.stack([dense[r] @ xf[i // k] if r >= 0 else np.zeros(N) for i, r in enumerate(rows)])
    got = (out - base).cpu().numpy()
    assert (got[rows < 0] == 0).all()
    assert ops.max_rel_err(got, want) <= TOL


def test_out_of_range_route_is_nan_through_gather_and_glu(dev):
    """R >= 128 takes the sorted-route GEMM: a route whose expert is out of
    range sorts past every valid tile and its row comes back NaN (not
    unwritten memory), through gather_vqmm and through the shared-plan
    prefill of QuantizedVQSwitchGLU; every other row matches the oracle."""
    from keep_amd.nn import QuantizedVQSwitchGLU, QuantizedVQSwitchLinear

    E, H, I, T, k = 6, 256, 256, 48, 4
    gate, up, down = (synth.projection_np(E, I, H, seed=61), synth.projection_np(E, I, H, seed=62),
                      synth.projection_np(E, H, I, seed=63))
    rng = np.random.default_rng(64)
    rhs = rng.integers(0, E, size=(T, k)).astype(np.int32)
    rhs[3, 2], rhs[17, 0], rhs[40, 3] = E, -1, E + 9
    bad = (rhs < 0) | (rhs >= E)
    x = synth.rht_activations(T, H, seed=65, device=dev)
    for trial in range(2):  # the output buffer of the second call is recycled memory
        y = kops.gather_vqmm(x, _t(gate[0], dev), _t(gate[1], dev), None, _t(rhs, dev), input_dims=H,
                             output_dims=I, group_size=H, code_bits=16)
        assert y.shape == (T, k, I)
        yc = y.float().cpu()
        assert torch.isnan(yc[torch.from_numpy(bad)]).all()
        assert not torch.isnan(yc[torch.from_numpy(~bad)]).any()
    want = ops.gather_token(x.float().cpu().numpy(), gate[0], gate[1], np.where(bad, 0, rhs))
    _check(yc[torch.from_numpy(~bad)], want[~bad])

    def lin(p, K, N):
        return QuantizedVQSwitchLinear(input_dims=K, output_dims=N, num_experts=E, codes=_t(p[0], dev),
                                       scales=_t(p[1], dev), group_size=K, code_bits=16)

    glu = QuantizedVQSwitchGLU(gate_proj=lin(gate, H, I), up_proj=lin(up, H, I), down_proj=lin(down, I, H))
    out = glu(x, _t(rhs, dev)).float().cpu()
    assert out.shape == (T, k, H)
    assert torch.isnan(out[torch.from_numpy(bad)]).all()
    assert not torch.isnan(out[torch.from_numpy(~bad)]).any()


def test_grouped_gemm_q8_blocks_run_many_items(dev):
    """More work items than blocks: at N = 2048 (eight 256-column blocks)
    and ~100 tiles every persistent block runs two or more non-empty items
    back to back, so a block's next item must not overwrite the row scales
    and output rows that its lagging waves still read in the previous
    item's epilogue. Checked against the C oracle on every route."""
    from oracle import cpu

    E, N, K, T, k = 40, 2048, 512, 1200, 4
    codes, scales = synth.projection_np(E, N, K, seed=71)
    rhs = synth.zipf_routes(T, E, k, s=1.1, seed=72)
    x = synth.rht_activations(T, K, seed=73, device=dev)
    flat, order, inverse, counts, tiles, lhs = _plan(rhs, E, k, dev)
    n_tiles = int((tiles[2] > 0).sum().item())
    assert n_tiles * (N // 256) > 2 * 256, "fewer work items than two per block"
    cb = kops._default_codebook(16, dev)
    y = kops.grouped_gemm(x, _t(codes, dev), _t(scales, dev), cb, tiles, lhs=lhs, routes=flat.numel(),
                          input_dims=K, output_dims=N, group_size=K, out_dtype=torch.float32, out_index=order)
    want = cpu.routed_matvec(x.float().cpu().numpy(), codes, scales.astype(np.float32),
                             kops.e8p_packed_abs_grid(), rhs.reshape(-1), x_div=k, group_size=K)
    _check(y, want.astype(np.float64))


@pytest.mark.parametrize("G", [1, 2])
@pytest.mark.parametrize("form", ["plain", "swiglu"])
def test_grouped_gemm_wide_items(dev, form, G):
    """Enough route tiles for work items of 512 columns (two n-tiles per
    wave): 160 experts with ~32 routes each (tiles of one and two m-tiles),
    N = 4096 (plain) or I = 2048 (gate/up + SwiGLU), per-row and grouped
    scales, against the C oracle's fp32 row dots."""
    E, K, T, k = 160, 256, 2560, 2
    rng = np.random.default_rng(50 + G)
    rhs = rng.integers(0, E, (T, k)).astype(np.int32)
    x = synth.rht_activations(T, K, seed=51, device=dev)
    flat, order, inverse, counts, tiles, lhs = _plan(rhs, E, k, dev)
    c = counts.cpu().numpy()
    assert tiles[0].numel() >= 128 and (c > 32).any() and ((c > 0) & (c <= 32)).any()
    cb = kops._default_codebook(16, dev)
    tab = e8p.e8p_packed_abs_grid()
    xf = x.float().cpu().numpy()
    R = flat.numel()

    def oracle(codes, scales):
        return cpu.routed_matvec(xf, codes, scales.astype(np.float32), tab, rhs.reshape(-1), x_div=k,
                                 group_size=K // G).astype(np.float64)
    if form == "plain":
        N = 4096
        codes, scales = synth.projection_np(E, N, K, group_size=K // G, seed=52)
        y = kops.grouped_gemm(x, _t(codes, dev), _t(scales, dev), cb, tiles, lhs=lhs, routes=R, input_dims=K,
                              output_dims=N, group_size=K // G, out_dtype=torch.float32)
        _check(y[inverse.long()], oracle(codes, scales))
    else:
        I = 2048
        gate = synth.projection_np(E, I, K, group_size=K // G, seed=53)
        up = synth.projection_np(E, I, K, group_size=K // G, seed=54)
        h = kops.grouped_swiglu(x, _t(gate[0], dev), _t(gate[1], dev), _t(up[0], dev), _t(up[1], dev), cb, tiles,
                                lhs=lhs, routes=R, input_dims=K, hidden_dims=I, group_size=K // G, limit=7.0)
        with np.errstate(over="ignore"):
            want = ops.round_bf16(ops.swiglu(oracle(*gate), oracle(*up), limit=7.0))
        got = h[inverse.long()].float().cpu().numpy()
        assert ops.elementwise_ok(got, want, rtol=TOL + 2.0 ** -7), "h beyond one bf16 ulp of the oracle's"


@pytest.mark.parametrize("code_bits", [8, 16])
@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,G", [(1024, 64, 128, 1), (129, 513, 640, 5), (2112, 1040, 256, 2), (65, 2056, 384, 1)])
def test_one_matrix_gemm_vs_oracle(dev, code_bits, xdt, M, N, K, G):
    """vq_qmm on the MFMA GEMM: partial row tiles (65 = one row past a tile),
    partial column blocks, one K block, per-row and grouped scales (items of
    256 columns; 512 in the test below). fp32 row dots against the fp64 oracle: within the rounding of the
    16-bit output plus the path's bound."""
    rng = np.random.default_rng(M + N)
    codes = rng.integers(0, 1 << code_bits, (N, K // 8)).astype(np.uint8 if code_bits == 8 else np.uint16)
    scales = np.exp(rng.normal(0, 0.3, (N, G))).astype(np.float16)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(dev).to(xdt)
    assert M * N >= kops.MATRIX_GEMM_CELLS
    y = kops.vq_qmm(x, _t(codes, dev), _t(scales, dev), in_dim=K, out_dim=N, group_size=K // G, code_bits=code_bits)
    assert y.dtype == xdt
    dense = (e8p.decode_e8_1bit(codes) if code_bits == 8 else e8p.decode_e8p(codes)).astype(np.float64)
    dense = dense.reshape(N, K) * np.repeat(scales.astype(np.float64), K // G, -1)
    want = x.double().cpu().numpy() @ dense.T
    ulp = 2.0 ** -9 if xdt == torch.float16 else 2.0 ** -8
    _check(y, want, tol=TOL + ulp)


@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("E,T,k,N,K,G", [(7, 43, 3, 72, 128, 1), (3, 90, 2, 520, 512, 4), (200, 700, 4, 1032, 256, 2)])
def test_routed_8bit_gemm_vs_oracle(dev, xdt, E, T, k, N, K, G):
    """8-bit E8 routes on the sorted-route GEMM (tiles of one and two m-tiles,
    partial column blocks, items of 256 columns; 512 in the test below), an out-of-range route
    (NaN), and gather_vqmm_sorted_routes on unsorted routes: each row its own."""
    rng = np.random.default_rng(E + T)
    codes = rng.integers(0, 256, (E, N, K // 8), dtype=np.uint8)
    scales = np.exp(rng.normal(0, 0.3, (E, N, G))).astype(np.float16)
    rhs = rng.integers(0, E, (T, k)).astype(np.int32)
    rhs[1, 0] = E
    x = torch.from_numpy(rng.standard_normal((T, K)).astype(np.float32)).to(dev).to(xdt)
    dense = e8p.decode_e8_1bit(codes).astype(np.float64).reshape(E, N, K) * np.repeat(
        scales.astype(np.float64), K // G, -1)
    flat = rhs.reshape(-1)
    good = flat < E
    xd = x.double().cpu().numpy()
    want = np.stack([dense[min(e, E - 1)] @ xd[i // k] for i, e in enumerate(flat)])
    ulp = 2.0 ** -9 if xdt == torch.float16 else 2.0 ** -8
    kw = dict(input_dims=K, output_dims=N, group_size=K // G, code_bits=8)
    with keep_amd.trace_gather_vqmm_calls() as tr:
        y = kops.gather_vqmm(x, _t(codes, dev), _t(scales, dev), None, _t(rhs, dev), route_strategy="sorted_tiled",
                             **kw).reshape(T * k, N)  # (the two small cases are the mat-vec's by themselves)
    assert tr[0]["implementation"] == "mfma_grouped_gemm"
    lhs = torch.arange(T * k, device=dev, dtype=torch.int32) // k
    z = kops.gather_vqmm_sorted_routes(x, _t(codes, dev), _t(scales, dev), None, _t(flat, dev), lhs, **kw)
    for out in (y, z):
        assert torch.isnan(out[torch.from_numpy(~good)]).all()
        _check(out[torch.from_numpy(good)], want[good], tol=TOL + ulp)


def _dense(codes, scales, code_bits, K):
    """Decoded weights in float64 on the GPU, from the oracle's grid."""
    grid = e8p.decode_e8_1bit(np.arange(256, dtype=np.uint8)) if code_bits == 8 else e8p.e8p_full_grid()
    index = codes.int() if code_bits == 8 else codes.int() & 0xFFFF
    w = torch.from_numpy(grid.astype(np.float64)).to(codes.device)[index].flatten(-2)
    return w * scales.double().repeat_interleave(K // scales.shape[-1], -1)


def _codes(code_bits, shape, K, dev, g):
    c = torch.randint(0, 256, (*shape, K // 8 * (code_bits // 8)), dtype=torch.uint8, device=dev, generator=g)
    return c if code_bits == 8 else c.view(torch.int16)


@pytest.mark.parametrize("code_bits", [8, 16])
@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("G", [1, 2])
def test_one_matrix_gemm_wide_items(dev, code_bits, xdt, G):
    """Rows and columns enough that 512-column items take fewer rounds of the
    chip: 2001 x 4088, a partial tile of rows and a partial last item."""
    M, N, K = 2001, 4088, 256
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    rounds = [-(-(-(-M // 64) * -(-N // w)) // cus) for w in (256, 512)]
    assert 8 * rounds[1] <= 5 * rounds[0], "items of 512 columns"
    g = torch.Generator(device=dev).manual_seed(G + code_bits)
    codes = _codes(code_bits, (N,), K, dev, g)
    scales = torch.exp(0.3 * torch.randn((N, G), device=dev, generator=g)).half()
    x = torch.randn((M, K), device=dev, generator=g).to(xdt)
    y = kops.matrix_gemm(x, codes, scales, kops._default_codebook(code_bits, dev), input_dims=K, output_dims=N,
                         group_size=K // G, code_bits=code_bits)
    ulp = 2.0 ** -9 if xdt == torch.float16 else 2.0 ** -8
    _check(y, (x.double() @ _dense(codes, scales, code_bits, K).T).cpu().numpy(), tol=TOL + ulp)


@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("G", [1, 2])
def test_routed_8bit_gemm_wide_items(dev, xdt, G):
    """Four items of 512 columns per CU: 160 experts of 4096 outputs, tiles of one and of two m-tiles, an
    out-of-range route (NaN)."""
    E, N, K, T, k = 160, 4096, 256, 2560, 2
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert (-(-T * k // 64) + E) * -(-N // 512) >= 4 * cus, "items of 512 columns"
    g = torch.Generator(device=dev).manual_seed(G)
    codes = _codes(8, (E, N), K, dev, g)
    scales = torch.exp(0.3 * torch.randn((E, N, G), device=dev, generator=g)).half()
    x = torch.randn((T, K), device=dev, generator=g).to(xdt)
    rhs = torch.randint(0, E, (T, k), device=dev, generator=g, dtype=torch.int32)
    rhs[7, 1] = E
    count = torch.bincount(rhs.reshape(-1).long())
    assert (count > 32).any() and ((count > 0) & (count <= 32)).any()
    with keep_amd.trace_gather_vqmm_calls() as tr:
        y = kops.gather_vqmm(x, codes, scales, None, rhs, input_dims=K, output_dims=N, group_size=K // G, code_bits=8)
    assert tr[0]["implementation"] == "mfma_grouped_gemm"
    assert torch.isnan(y[7, 1]).all()
    flat, y = rhs.reshape(-1), y.reshape(T * k, N)
    want = torch.zeros((T * k, N), dtype=torch.float64, device=dev)
    for e in range(E):
        r = torch.nonzero(flat == e)[:, 0]
        want[r] = x[r // k].double() @ _dense(codes[e], scales[e], 8, K).T
    good = flat < E
    ulp = 2.0 ** -9 if xdt == torch.float16 else 2.0 ** -8
    _check(y[good], want[good].cpu().numpy(), tol=TOL + ulp)


@pytest.mark.parametrize("tail", [1, 700])
@pytest.mark.parametrize("gap", [False, True])
def test_empty_tiles_of_a_plan_change_nothing(tail, gap):
    # N = 1544: four column blocks of 512 (the last ragged), so the items do not divide by the XCDs; the arrays end
    # in `tail` empty tiles, and one may lie between live ones. Every row is computed alike: the bits are the same.
    E, N, K, R = 9, 1544, 256, 200
    g = torch.Generator().manual_seed(tail + gap)
    codes = torch.randint(-32768, 32768, (E, N, K // 8), dtype=torch.int16, generator=g).cuda()
    scales = torch.rand((E, N, 1), generator=g).half().cuda()
    x = torch.randn((R, K), generator=g).half().cuda()
    rhs = torch.randint(0, E, (R,), dtype=torch.int32, generator=g).cuda()
    order, _, _, _, te, to, tc, _ = kops.route_plan(rhs, E, kops.GEMM_ROUTE_TILE)
    n = int((tc > 0).sum())
    cb = kops._default_codebook(16, x.device)

    def gemm(*tiles):
        return kops.grouped_gemm(x, codes, scales, cb, tuple(t.contiguous() for t in tiles), lhs=order, routes=R,
                                input_dims=K, output_dims=N, group_size=K, out_index=order)

    want = gemm(te[:n], to[:n], tc[:n])
    hole = torch.zeros(1, dtype=torch.int32, device=x.device)
    parts = [[t[:2], hole, t[2:n]] if gap else [t[:n]] for t in (te, to, tc)]
    got = gemm(*(torch.cat(p + [hole.repeat(tail)]) for p in parts))
    assert not torch.isnan(want).any() and torch.equal(got, want)


def _same_values(got, want, tol):
    """NaN and infinities where the float64 product has them, finite values within tol of their row's largest."""
    got = got.double().cpu().numpy()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    np.testing.assert_array_equal(np.isinf(got), inf)
    np.testing.assert_array_equal(got[inf], want[inf])
    fin = np.where(np.isfinite(want), want, 0)
    assert (np.abs(np.where(np.isfinite(want), got, 0) - fin) <= tol * np.abs(fin).max(-1, keepdims=True)).all()


@pytest.mark.parametrize("code_bits", [8, 16])
@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M, N, K, G", [(90, 1040, 384, 3), (128, 1024, 512, 1)])
def test_one_matrix_gemm_non_finite_rows(dev, code_bits, xdt, M, N, K, G):
    """vq_qmm on the GEMM with infinities and NaN in its rows: the plain
    product's, and where the mat-vec has an infinity, that infinity."""
    rng = np.random.default_rng(M)
    codes = rng.integers(0, 1 << code_bits, (N, K // 8)).astype(np.uint8 if code_bits == 8 else np.uint16)
    scales = np.exp(rng.normal(0, 0.3, (N, G))).astype(np.float16)
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).to(dev).to(xdt)
    inf, nan = float("inf"), float("nan")
    for r, vals in {1: {5: inf}, 2: {K - 1: -inf}, 3: {7: inf, 90: -inf}, 4: {9: nan}, 5: {2: inf, 3: inf},
                    M - 1: {0: inf, 1: nan}}.items():
        for i, v in vals.items():
            x[r, i] = v
    x[6] = inf
    kw = dict(input_dims=K, output_dims=N, group_size=K // G, code_bits=code_bits)
    c, s, cb = _t(codes, dev), _t(scales, dev), kops._default_codebook(code_bits, dev)
    assert M * N >= kops.BF16_E8P_GEMM_CELLS
    y = kops.vq_qmm(x, c, s, in_dim=K, out_dim=N, group_size=K // G, code_bits=code_bits)
    dense = (e8p.decode_e8_1bit(codes) if code_bits == 8 else e8p.decode_e8p(codes)).astype(np.float64)
    dense = dense.reshape(N, K) * np.repeat(scales.astype(np.float64), K // G, -1)
    with np.errstate(invalid="ignore"):
        want = np.stack([(dense * r).sum(1) for r in x.double().cpu().numpy()])
    assert code_bits == 8 or np.isinf(want[[1, 2]]).all()
    _same_values(y, want, TOL + 2.0 ** -7)
    old = kops.routed_matvec(x, c.reshape(1, N, -1), s.reshape(1, N, -1), cb, None, routes=M, **kw)
    assert torch.equal(y[torch.isinf(old)], old[torch.isinf(old)])
