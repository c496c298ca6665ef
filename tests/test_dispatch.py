"""Which entry points the operators reach, on the CPU with the launches
recorded instead of made: no launch on tensors the GPU does not own."""

from types import SimpleNamespace

import pytest
import torch

import keep_amd
from keep_amd import _lib, ops


@pytest.fixture
def launches(monkeypatch):
    """The entry points called, none of them run; a GPU's stream and capture state stubbed."""
    calls, real = [], _lib.call
    host = ("keep_e8p_packed_abs_grid", "keep_e8_1bit_packed")  # tables built on the host

    def call(name, *args):
        if name in host:
            return real(name, *args)
        calls.append(name)
        if name == "keep_route_plan" and args[2] > 1024:
            raise ValueError("E must be in 1..1024")  # the library's check
    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(ops, "_raw_stream", lambda index: 0)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(ops, "_PREPARED", {})
    monkeypatch.setattr(ops, "_DEFAULT_PREPARED", {})
    return calls


def _moe(T, H=512, I=256, E=4, k=2):
    def codes(n, K):
        return torch.zeros((E, n, K // 8), dtype=torch.int16), torch.ones((E, n, 1), dtype=torch.float16)
    return (torch.zeros((T, H), dtype=torch.float16), torch.zeros((T, E)), (codes(I, H), codes(I, H), codes(H, I)),
            torch.zeros((T, k), dtype=torch.int32), torch.ones((T, k)))


@pytest.mark.parametrize("call", ["decode", "decode_packed", "tiles_layer", "layer", "wide"])
def test_cpu_activations_are_refused_before_any_launch(launches, call):
    x, z, pool, idx, w = _moe(1 if call == "layer" else 3, **({"H": 4096, "I": 512} if call == "layer" else
                                                              {"H": 4608} if call == "wide" else {}))
    with pytest.raises(ValueError, match="cuda device"):
        if call in ("decode", "wide"):
            keep_amd.moe_decode(x, idx, w, *pool)
        elif call == "decode_packed":
            keep_amd.moe_decode(x, idx, w, *pool, prepared=False)
        elif call == "tiles_layer":
            keep_amd.moe_tiles_layer(x, z, *pool, k=2)
        else:
            keep_amd.moe_layer(x, z, *pool, k=2)
    assert launches == []


def test_a_table_prepared_under_capture_is_not_kept(launches, monkeypatch):
    """It holds nothing before that graph's first replay: the next eager call builds its own, once."""
    cb = torch.from_numpy(ops.e8p_packed_abs_grid().view("int32"))
    monkeypatch.setattr(ops, "_stream", lambda device: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: SimpleNamespace(synchronize=lambda: None))
    captured = ops.prepared_table(cb)
    assert launches == ["keep_e8p_prepare"] and not ops._may_prepare(cb)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert ops._may_prepare(cb)
    eager = ops.prepared_table(cb)
    assert eager is not captured and launches == ["keep_e8p_prepare"] * 2
    assert ops.prepared_table(cb) is eager
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert ops._may_prepare(cb) and ops.prepared_table(cb) is eager
    assert len(launches) == 2


@pytest.fixture
def routed(launches, monkeypatch):
    """The operators on CPU tensors taken for the GPU's; the entry points that one call reached."""
    monkeypatch.setattr(ops, "_device_of", lambda *ts: torch.device("cpu"))
    monkeypatch.setattr(ops, "_stream", lambda device: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: SimpleNamespace(synchronize=lambda: None))

    def run(fn, *args, **kw):
        launches.clear()
        fn(*args, **kw)
        return list(launches)
    return run


def _switch(E, N, K, bits=8, G=1):
    codes = torch.empty((E, N, K // 8), dtype=torch.uint8 if bits == 8 else torch.int16)  # never read
    return codes, torch.empty((E, N, G), dtype=torch.float16), dict(input_dims=K, output_dims=N, group_size=K // G)


@pytest.mark.parametrize("T", [2, 65])
def test_more_experts_than_a_plan_holds(routed, T):
    """Route plans hold 1024 experts. Calls that never needed one are served beyond, by the mat-vec."""
    N, K, k = 4096, 512, 2
    x, rhs = torch.empty((T, K), dtype=torch.float16), torch.zeros((T, k), dtype=torch.int32)
    flat, lhs = rhs.reshape(-1), torch.arange(T * k, dtype=torch.int32) // k
    for E in (1024, 1025):
        c, s, kw = _switch(E, N, K)
        assert N * K >= ops.ROWS_MATRIX
        got = {
            "auto": routed(ops.gather_vqmm, x, c, s, None, rhs, code_bits=8, **kw),
            "direct": routed(ops.gather_vqmm, x, c, s, None, rhs, code_bits=8, route_strategy="direct", **kw),
            "sorted": routed(ops.gather_vqmm_sorted_routes, x, c, s, None, flat, lhs, code_bits=8, **kw),
            "flat": routed(ops.gather_vqmm_verify_rows, x, c, s, None, rhs, grouping="flat", **kw),
        }
        for name, calls in got.items():
            if E > 1024:
                assert calls == ["keep_vq_matvec"], (name, calls)
            elif name != "sorted" or T * k >= ops.GEMM_ROUTE_THRESHOLD:
                assert calls[-1] == "keep_vq_rows", (name, calls)
    # what a plan refused it refuses
    for fn, over in ((ops.gather_vqmm, dict(code_bits=8, route_strategy="sorted_tiled")),
                     (ops.gather_vqmm_verify_rows, dict(grouping="expert"))):
        with pytest.raises(ValueError, match="1024"):
            routed(fn, x, c, s, None, rhs, **over, **kw)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bits", [8, 16])
@pytest.mark.parametrize("E, N, K, G, T, k", [(4, 4096, 512, 1, 2, 2), (4, 4096, 512, 1, 65, 2), (4, 512, 512, 1, 65, 2),
                                              (2, 64, 512, 1, 200, 2), (8, 64, 128, 1, 65, 2), (4, 72, 640, 5, 70, 2),
                                              (8, 4096, 512, 2, 10, 2), (4, 520, 8704, 17, 40, 4)])
@pytest.mark.parametrize("strategy", ["auto", "direct", "sorted_tiled", "verify"])
def test_trace_names_the_kernel_that_runs(routed, monkeypatch, dtype, bits, E, N, K, G, T, k, strategy):
    c, s, kw = _switch(E, N, K, bits, G)
    x, rhs = torch.empty((T, K), dtype=dtype), torch.zeros((T, k), dtype=torch.int32)
    monkeypatch.setattr(ops, "route_plan", lambda rhs, E, tile: tuple(
        torch.arange(rhs.numel(), dtype=torch.int32) for _ in range(8)))
    with keep_amd.trace_gather_vqmm_calls() as tr:
        if strategy == "verify":
            calls = routed(ops.gather_vqmm_verify_rows, x, c, s, None, rhs, grouping="expert", **kw)
        else:
            calls = routed(ops.gather_vqmm, x, c, s, None, rhs, code_bits=bits, route_strategy=strategy, **kw)
    want = {"keep_vq_rows": "mfma_rows", "keep_vq_grouped_gemm_e8": "mfma_grouped_gemm",
            "keep_vq_grouped_gemm_q8": "mfma_grouped_gemm", "keep_vq_matvec": "hip_matvec",
            "keep_vq_matvec_tiles": "hip_matvec"}
    assert [t["implementation"] for t in tr] == [want[calls[-1]]]


def test_written_tables_are_not_the_default(routed, launches):
    """A layer's own copy of the default E8P table takes the matrix cores and the one prepared table of all
    copies; written to, it is a table like any other: the mat-vec, and prepared again."""
    cpu = torch.device("cpu")
    N, K, M = 4096, 512, 128
    c, s, kw = _switch(1, N, K, bits=16)
    x = torch.empty((M, K), dtype=torch.float16)

    def qmm(cb):
        return routed(ops.vq_qmm, x, c[0], s[0], cb, in_dim=K, out_dim=N, group_size=K, code_bits=16)

    a, b = ops._new_codebook(16, cpu), ops._new_codebook(16, cpu)
    assert qmm(a) == ["keep_e8p_prepare", "keep_vq_rows"] and qmm(b) == ["keep_vq_rows"] and qmm(None) == ["keep_vq_rows"]
    shared = ops.prepared_table(b)
    a[3] = a[4]
    assert qmm(a) == ["keep_vq_matvec"] and qmm(b) == ["keep_vq_rows"]
    first = ops.prepared_table(a)
    assert first is not shared and ops.prepared_table(a) is first and ops.prepared_table(b) is shared
    with torch.inference_mode():
        a[5] = 0
    assert ops.prepared_table(a) is not first
    assert qmm(b.clone()) == ["keep_vq_matvec"]  # a table of the caller's
    n = len(ops._E8P_TABLES)
    del b
    assert len(ops._E8P_TABLES) == n - 1


def test_router_outputs_have_version_counters_of_their_own():
    """Writing to one output leaves another that autograd has saved usable."""
    from keep_amd.nn import _router_output

    r = _router_output(3, 5, torch.device("cpu"))
    assert [t.dtype for t in r] == [torch.int32, torch.float32, torch.int32, torch.float32, torch.uint8]
    assert all(t.shape == (3, 5) and t.is_contiguous() and not t._is_view() for t in (r.idx, r.want, r.admit))
    spans = sorted((t.data_ptr(), t.data_ptr() + t.nbytes) for t in r)
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
    r.weight.fill_(0.5)
    y = torch.ones((3, 5), requires_grad=True)
    z = (y * r.weight).sum()
    r.idx.zero_()
    z.backward()
    assert torch.equal(y.grad, r.weight)


@pytest.mark.parametrize("T, H, I, E, k, wide", [(2, 7168, 2048, 1, 1, False), (3, 7168, 2048, 1, 1, True),
                                                 (2, 6144, 1024, 4, 2, False), (4, 6144, 1024, 4, 2, True),
                                                 (1, 8192, 256, 4, 2, False), (2, 8192, 256, 4, 2, True)])
def test_few_routes_of_wide_layers_stay_on_the_packed_kernels(routed, T, H, I, E, k, wide):
    x, _, pool, idx, w = _moe(T, H=H, I=I, E=E, k=k)
    assert routed(keep_amd.moe_decode, x, idx, w, *pool)[-1] == ("keep_moe_wide" if wide else "keep_moe_decode")


@pytest.mark.parametrize("T, E, N, K, G, last", [
    (64, 32, 64, 1024, 2, "keep_vq_matvec"), (64, 32, 256, 1024, 2, "keep_vq_matvec"),
    (64, 32, 512, 1024, 2, "keep_vq_rows"), (64, 32, 256, 4096, 8, "keep_vq_rows"),
    (32, 32, 64, 2048, 4, "keep_vq_matvec"), (32, 32, 512, 1024, 2, "keep_vq_rows"),
    (256, 4, 64, 4096, 8, "keep_vq_matvec"), (256, 4, 256, 1024, 2, "keep_vq_grouped_gemm_e8"),
    (32, 32, 64, 128, 1, "keep_vq_matvec"), (256, 32, 1024, 128, 1, "keep_vq_grouped_gemm_e8")])
def test_8bit_routes_leave_the_matvec_with_enough_work(routed, monkeypatch, T, E, N, K, G, last):
    """4 routes a token, through gather_vqmm (also told that they are sorted) and gather_vqmm_sorted_routes."""
    monkeypatch.setattr(ops, "route_plan", lambda rhs, E, tile: tuple(
        torch.arange(rhs.numel(), dtype=torch.int32) for _ in range(8)))
    c, s, kw = _switch(E, N, K, G=G)
    x, rhs = torch.empty((T, K), dtype=torch.float16), torch.zeros((T, 4), dtype=torch.int32)
    lhs = torch.arange(T * 4, dtype=torch.int32) // 4
    assert N * K < ops.ROWS_MATRIX
    for sort in (False, True):
        assert routed(ops.gather_vqmm, x, c, s, None, rhs, code_bits=8, sorted_indices=sort, **kw)[-1] == last
    assert routed(ops.gather_vqmm_sorted_routes, x, c, s, None, rhs.reshape(-1), lhs, code_bits=8, **kw)[-1] == last
    assert routed(ops.gather_vqmm, x, c, s, None, rhs, code_bits=8, route_strategy="sorted_tiled",
                  **kw)[-1] != "keep_vq_matvec"
