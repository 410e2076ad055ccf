"""mi355x_qgemv_noalloc, the entry point that allocates nothing, against mi355x_qgemv: the same kernels
over a fixed scratch block, so the results must be the same bits (and within the product's bound of
the oracle). Two calls in a row per case, the second with a smaller input, since the block keeps the
last call's contents. That nothing is allocated is shown twice: the device's free memory does not move
across the calls, and the calls are made under stream capture on a stream the library has never seen
(where an allocation is refused, the library's growing scratch included), then replayed from the graph."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from mimir_amd import capi
from tests import gpu, helpers

pytestmark = pytest.mark.gpu

DT = {"q4_0": (capi.Q4_0, O.Q4_0), "q8_0": (capi.Q8_0, O.Q8_0), "q4_K": (capi.Q4_K, O.Q4_K), "q6_K": (capi.Q6_K, O.Q6_K)}

# (M, N, K): twelve rows (every dtype converts them into the block: Q4_0 and Q8_0 do so from nine rows on, the
# K-quants from two), then three, then one
CASES = ((12, 384, 2048), (3, 160, 512), (1, 96, 256))


def _blocks(rng, name, odt, n, k):
    # scales as the configurations draw them for the dtypes whose float32 sums differ in order from the oracle's
    return helpers.bench_blocks(rng, odt, n * k) if name in ("q4_0", "q8_0") else helpers.random_blocks(rng, odt, n * k)


def _both(dt, w, x, n, k):
    l = gpu.lib()
    m = x.shape[0]
    ys = []
    for fn in (l.mi355x_qgemv, l.mi355x_qgemv_noalloc):
        y = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
        capi.check(fn(dt, w.data_ptr(), x.data_ptr(), y.data_ptr(), m, n, k, k, gpu.stream()))
        gpu.sync()
        ys.append(y.cpu().numpy())
    return ys


@pytest.mark.parametrize("name", ["q4_0", "q8_0", "q4_K", "q6_K"])
def test_noalloc_equals_qgemv_twice_second_smaller(name):
    dt, odt = DT[name]
    rng = np.random.default_rng(7)
    # the first call fills more of the block than the second reads
    for (m, n, k) in CASES:
        raw = _blocks(rng, name, odt, n, k)
        x = rng.normal(size=(m, k)).astype(np.float32)
        gpu.say(f"qgemv_noalloc {name} M={m} N={n} K={k}")
        w, xd = gpu.dev(raw), gpu.dev(x)
        got, got_fixed = _both(dt, w, xd, n, k)
        assert np.array_equal(got.view(np.uint32), got_fixed.view(np.uint32))
        want = O.qmatmul(odt, raw, x, n, k)
        tol = 1e-3 if name == "q4_0" else 1e-4 if name == "q8_0" else 1e-5  # the K-quant kernels give the oracle's bits
        assert np.all(np.abs(got_fixed - want) <= tol * np.maximum(1, np.abs(want)))


@pytest.mark.parametrize("name", ["q4_0", "q8_0", "q4_K", "q6_K"])
def test_noalloc_allocates_nothing(name):
    """Free device memory is the same before and after; and the calls succeed under stream capture on a fresh
    stream, where hipMalloc is refused (so a route back to the library's growing scratch would fail there), the
    graph's replays giving the bits of the eager mi355x_qgemv."""
    dt, odt = DT[name]
    l = gpu.lib()
    rng = np.random.default_rng(11)
    prepared = []
    for (m, n, k) in CASES:
        raw = _blocks(rng, name, odt, n, k)
        x = rng.normal(size=(m, k)).astype(np.float32)
        w, xd = gpu.dev(raw), gpu.dev(x)
        want = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
        capi.check(l.mi355x_qgemv(dt, w.data_ptr(), xd.data_ptr(), want.data_ptr(), m, n, k, k, gpu.stream()))  # also loads the kernels
        y = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
        prepared.append((m, n, k, w, xd, y, want))
    gpu.sync()
    torch.cuda.synchronize()
    free_before = torch.cuda.mem_get_info()[0]
    for (m, n, k, w, xd, y, want) in prepared:
        gpu.say(f"qgemv_noalloc {name} M={m} N={n} K={k}: free memory")
        capi.check(l.mi355x_qgemv_noalloc(dt, w.data_ptr(), xd.data_ptr(), y.data_ptr(), m, n, k, k, gpu.stream()))
    gpu.sync()
    assert torch.cuda.mem_get_info()[0] == free_before
    for (_, _, _, _, _, y, want) in prepared:
        assert torch.equal(y.view(torch.int32), want.view(torch.int32))
        y.fill_(float("nan"))
    fresh = torch.cuda.Stream()  # the library holds no scratch for it
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    gpu.say(f"qgemv_noalloc {name}: under stream capture")
    with torch.cuda.stream(fresh):
        with torch.cuda.graph(graph, stream=fresh):
            for (m, n, k, w, xd, y, want) in prepared:
                capi.check(l.mi355x_qgemv_noalloc(dt, w.data_ptr(), xd.data_ptr(), y.data_ptr(), m, n, k, k, fresh.cuda_stream))
        for replay in range(2):
            graph.replay()
            fresh.synchronize()
            # the last case is the block's current content; every case's result was written by its own replayed launch
            for (_, _, _, _, _, y, want) in prepared:
                assert torch.equal(y.view(torch.int32), want.view(torch.int32)), replay
                y.fill_(float("nan"))
            fresh.synchronize()


def test_noalloc_rejects_what_the_block_cannot_hold():
    l = gpu.lib()
    k, n, m = 4096, 32, 300  # 300 rows of q8_0 activations: 4608 bytes each, more than 1 MiB
    w = torch.zeros(n * k // 32 * 34, dtype=torch.uint8, device="cuda:0")
    x = torch.zeros((m, k), dtype=torch.float32, device="cuda:0")
    y = torch.zeros((m, n), dtype=torch.float32, device="cuda:0")
    st = l.mi355x_qgemv_noalloc(capi.Q8_0, w.data_ptr(), x.data_ptr(), y.data_ptr(), m, n, k, k, gpu.stream())
    assert st == capi.ERR_SHAPE and "fixed scratch" in capi.last_error()
    # and the growing entry point takes the same call
    capi.check(l.mi355x_qgemv(capi.Q8_0, w.data_ptr(), x.data_ptr(), y.data_ptr(), m, n, k, k, gpu.stream()))
    gpu.sync()


def test_noalloc_rejects_by_the_size_that_act_bytes_tells():
    """K-quant rows of which sixteen laid out for the matrix cores would fit the block, though mi355x_act_bytes a row says more than 1 MiB."""
    l = gpu.lib()
    m, n, k = 128, 4096, 31 * 256
    w = torch.zeros(n * k // 256 * 144, dtype=torch.uint8, device="cuda:0")
    x, y = torch.zeros((m, k), device="cuda:0"), torch.zeros((m, n), device="cuda:0")
    assert m * l.mi355x_act_bytes(capi.Q4_K, k) > 1 << 20
    st = l.mi355x_qgemv_noalloc(capi.Q4_K, w.data_ptr(), x.data_ptr(), y.data_ptr(), m, n, k, k, gpu.stream())
    assert st == capi.ERR_SHAPE and "fixed scratch" in capi.last_error()
    capi.check(l.mi355x_qgemv_noalloc(capi.Q4_K, w.data_ptr(), x.data_ptr(), y.data_ptr(), m - 16, n, k, k, gpu.stream()))
    gpu.sync()


def test_a_call_of_more_rows_under_capture_after_one_of_few():
    """What a stream's first call leaves is enough for whatever fills no more than 1 MiB in fixed point: 32 rows by W read where it lies,
    whose rows and shares of K take 4.8 MB, recorded into a graph after a call of eight rows, and replayed."""
    l, n, k = gpu.lib(), 14336, 4096
    rng = np.random.default_rng(5)
    w = gpu.dev(helpers.bench_blocks(rng, O.Q4_0, n * k))
    xs = [gpu.dev(rng.normal(size=(32, k)).astype(np.float32)) for _ in range(3)]
    x, y, want = xs[0].clone(), torch.empty((32, n), device="cuda:0"), []

    def call(m, stream, out=y):
        capi.check(l.mi355x_qgemv(capi.Q4_0, w.data_ptr(), x.data_ptr(), out.data_ptr(), m, n, k, k, stream))
    gpu.say("qgemv under capture after a call of few rows")
    for v in xs:
        x.copy_(v)
        out = torch.empty_like(y)
        call(32, gpu.stream(), out)
        want.append(out)
    torch.cuda.synchronize()
    fresh, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(fresh):
        call(8, fresh.cuda_stream)
        fresh.synchronize()
        with torch.cuda.graph(graph, stream=fresh):
            call(32, fresh.cuda_stream)
        for v, expected in zip(xs, want):
            x.copy_(v)
            y.fill_(float("nan"))
            graph.replay()
            fresh.synchronize()
            assert torch.equal(y.view(torch.int32), expected.view(torch.int32))


def last_kernel():
    buf = C.create_string_buffer(200)
    capi.check(gpu.lib().mi355x_last_kernel(buf, 200))
    return buf.value.decode()


@pytest.mark.parametrize("m,n,k,kernels", [
    (32, 14336, 4096, ("qgemm_q4_0_parts_kernel", "qgemm_q4_0_parts_kernel")), (48, 5120, 5120, ("qgemm_q4_0_parts_kernel", "qgemm_q4_0_parts_kernel")),
    (200, 32768, 1024, ("qgemm_q4_0_direct_kernel", "qgemm_q4_0_direct_kernel")), (256, 32768, 1024, ("qgemm_q4_0_direct_kernel", "qgemm_q4_0_direct_kernel")),
    (300, 65536, 1024, ("qgemm_q4_0_fx16_kernel", "qgemm_q4_0_fx_kernel")), (512, 32768, 512, ("qgemm_q4_0_fx16_kernel", "qgemm_q4_0_fx_kernel")),
    (1000, 2048, 256, ("qgemm_q4_0_fx_kernel", "qgemm_q4_0_fx_kernel"))])
def test_noalloc_equals_qgemv_at_many_rows(m, n, k, kernels):
    """Whatever the fixed block takes has mi355x_qgemv's bits there: W read where it lies, by the same kernel in the same shares of K; from
    256 rows on the int8 form, whose bits mi355x_qgemv's panel of digits gives. Against 64 bits within the product's bound."""
    rng = np.random.default_rng(m)
    raw = helpers.bench_blocks(rng, O.Q4_0, 64 * k)
    w = gpu.dev(raw).repeat(n // 64)
    x = gpu.dev(rng.normal(size=(m, k)).astype(np.float32))
    gpu.say(f"qgemv_noalloc q4_0 M={m} N={n} K={k}")
    l, ys, ran = gpu.lib(), [], []
    for fn in (l.mi355x_qgemv, l.mi355x_qgemv_noalloc):
        y = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
        capi.check(fn(capi.Q4_0, w.data_ptr(), x.data_ptr(), y.data_ptr(), m, n, k, k, gpu.stream()))
        ran.append(last_kernel())
        ys.append(y)
    gpu.sync()
    assert all(r.startswith(want) for r, want in zip(ran, kernels)), ran
    assert torch.equal(ys[0].view(torch.int32), ys[1].view(torch.int32))
    fresh, graph, y = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.empty_like(ys[0])  # a stream that the library holds no scratch for
    torch.cuda.synchronize()
    with torch.cuda.stream(fresh):
        with torch.cuda.graph(graph, stream=fresh):
            capi.check(l.mi355x_qgemv_noalloc(capi.Q4_0, w.data_ptr(), x.data_ptr(), y.data_ptr(), m, n, k, k, fresh.cuda_stream))
        for replay in range(2):
            y.fill_(float("nan"))
            graph.replay()
            fresh.synchronize()
            assert torch.equal(y.view(torch.int32), ys[0].view(torch.int32)), replay
    w64, x64 = gpu.dev(O.dequantize(O.Q4_0, raw).reshape(64, k)).double(), x.double()
    bound = 2e-6 * (x64.abs() @ w64.abs().T) + 2.0 ** -23 * (x64.abs().reshape(m, -1, 32).amax(2) @ w64.abs().reshape(64, -1, 32).sum(2).T)
    for n0 in (0, n - 64):
        assert ((ys[1][:, n0:n0 + 64].double() - x64 @ w64.T).abs() <= bound).all()
