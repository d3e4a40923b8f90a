"""The entry point that allocates nothing (rocm_wmma_gemm_noalloc) against the ordinary
entry points, through the C ABI: same problems, same bits, on calls in a row that share
the fixed per-GPU scratch array, the later ones smaller than the first."""
import numpy as np
import pytest

import oracle as O
from gemm_harness import TYPE_PAIRS, check_against_oracle, make_inputs, to_device, to_host, torch_dtype

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def loader():
    import torch

    import rocm_wmma_gemm_amd as R

    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    torch.cuda.set_device(0)
    return R.Loader()  # raises if the HIP library is missing: no fallback


def _both_ways(loader, M, N, K, lc, la, lb, tname, batch=1):
    import torch

    din, dout = TYPE_PAIRS[tname]
    A = np.concatenate([O.init_matrix(M, K, la, din, seed=1 + b) for b in range(batch)])
    B = np.concatenate([O.init_matrix(K, N, lb, din, seed=101 + b) for b in range(batch)])
    dA, dB = to_device(A, din), to_device(B, din)
    want = torch.full((M * N * batch,), float("nan"), dtype=torch_dtype(dout), device="cuda")
    got = torch.full_like(want, float("nan"))
    loader.gemm(want, dA, dB, M, N, K, lc, la, lb, batch_count=batch)
    rc = loader.gemm_noalloc(got, dA, dB, M, N, K, lc, la, lb, batch_count=batch)
    torch.cuda.synchronize()
    return rc, want, got, A, B


def test_noalloc_entry_point_matches_the_ordinary_one_on_calls_in_a_row(loader):
    import torch

    import rocm_wmma_gemm_amd.loader as RL

    cases = [  # the first is the largest user of the scratch array, the rest are smaller
        (128, 8192, 8192, 0, 0, 1, "f32_f16", 1),    # split-K: fp32 partial planes
        (64, 4096, 4096, 1, 1, 0, "f16_f16", 1),     # split-K, fewer and smaller planes
        (1025, 1031, 2049, 0, 0, 1, "bf16_bf16", 1),  # ragged: padded copies (and partial tiles)
        (16, 2048, 1024, 0, 1, 1, "f32_bf16", 3),    # small batched split
        (512, 768, 1024, 0, 0, 1, "f16_f16", 1),     # whole tiles: no scratch memory at all
    ]
    for rnd in range(2):  # and once more from the top, over what the last round left behind
        for (M, N, K, lc, la, lb, tname, batch) in cases:
            rc, want, got, A, B = _both_ways(loader, M, N, K, lc, la, lb, tname, batch)
            assert rc == RL.OK, (rc, M, N, K, tname)
            assert not torch.isnan(got.float()).any()
            # same plan, same kernels, same order of additions: the same bits
            assert torch.equal(got, want), (rnd, M, N, K, lc, la, lb, tname)
            if rnd == 0 and batch == 1:
                din, dout = TYPE_PAIRS[tname]
                check_against_oracle(to_host(got, dout), A, B, M, N, K, lc, la, lb, din, dout)


def test_noalloc_entry_point_rejects_what_its_scratch_array_cannot_hold(loader):
    import torch

    import rocm_wmma_gemm_amd.loader as RL

    # ragged in every extent, rows not 16-byte aligned: the plan is padded copies of both
    # operands, 2 x 8192 x 8192 x 2 bytes = 256 MiB, four times the array
    M = N = K = 8191
    dA = torch.zeros(M * K, dtype=torch.float16, device="cuda")
    dB = torch.zeros(K * N, dtype=torch.float16, device="cuda")
    dC = torch.full((M * N,), float("nan"), dtype=torch.float16, device="cuda")
    assert loader.gemm_noalloc(dC, dA, dB, M, N, K, 0, 0, 1) == RL.ERR_SCRATCH
    torch.cuda.synchronize()
    assert bool(torch.isnan(dC).all()), "a rejected call must enqueue nothing"
    # bad arguments are reported, not ignored
    assert loader._lib.rocm_wmma_gemm_noalloc(7, 0, 0, 0, 16, 16, 16, 1, 0, 0, 0, None) == RL.ERR_ARGUMENT
    assert loader._lib.rocm_wmma_gemm_noalloc(0, 0, 0, 0, 16, 16, 16, 1, 0, 2, 0, None) == RL.ERR_ARGUMENT
    # and the array still serves the next call
    rc, want, got, _, _ = _both_ways(loader, 64, 8192, 8192, 0, 1, 0, "f32_f16")
    assert rc == RL.OK and torch.equal(got, want)


@pytest.mark.parametrize("M,N,K,layouts,type_name", [
    (1068, 1080, 4968, (0, 0, 1), "f16_f16"),       # ragged rows: the estimate's plan walks by K tile or copies
    (947, 1472, 8896, (0, 0, 1), "bf16_bf16"),
    (158, 11456, 12224, (0, 0, 0), "f32_f16"),      # ... and would copy the large operand here
    (133, 2000, 30001, (0, 1, 1), "f16_f16"),       # copies of both that only just pay
    (431, 831, 20181, (0, 1, 1), "f32_bf16"),       # odd in every extent
])
def test_noalloc_entry_point_takes_a_leaner_plan_where_the_first_does_not_fit(loader, M, N, K, layouts, type_name):
    """Extents whose rows do not start on 16 bytes, which the estimate would serve with more scratch
    memory than the array holds: the tables' plan, which fits, serves them.  The same for
    the ordinary entry point on a capturing stream without a buffer."""
    import torch

    import rocm_wmma_gemm_amd.loader as RL

    lc, la, lb = layouts
    din, dout = TYPE_PAIRS[type_name]
    A, B = make_inputs(M, N, K, la, lb, din, seed_a=31, seed_b=32)
    dA, dB = to_device(A, din), to_device(B, din)
    got = torch.full((M * N,), float("nan"), dtype=torch_dtype(dout), device="cuda")
    assert loader.gemm_noalloc(got, dA, dB, M, N, K, lc, la, lb) == RL.OK
    torch.cuda.synchronize()
    assert not torch.isnan(got.float()).any()
    rows = (M - 8, M)
    check_against_oracle(to_host(got, dout), A, B, M, N, K, lc, la, lb, din, dout, rows=rows)
    if loader.workspace_release() != 0:
        return  # (a graph of an earlier test holds the buffer: it would serve the capture)
    out = torch.full_like(got, float("nan"))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        loader.gemm(out, dA, dB, M, N, K, lc, la, lb)
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert not torch.isnan(out.float()).any()
        check_against_oracle(to_host(out, dout), A, B, M, N, K, lc, la, lb, din, dout, rows=rows)


def test_noalloc_and_ordinary_shared_tile_calls_on_two_streams(loader):
    """Calls whose workgroups share tiles (whole-K streaming kernel, several workgroups per
    tile) count their arrivals in per-GPU counters.  The ordinary entry points and the one
    that allocates nothing each have counters of their own, so an ordinary call on one stream
    and a no-alloc call on another may run at the same time: every result has the bits of
    the same call run alone."""
    import torch

    import rocm_wmma_gemm_amd.loader as RL

    M, N, K = 16, 1024, 8192
    variant, _, split = loader.select(M, N, K, 0, 0, 0, 1)
    assert loader.variants()[variant].pipeline == 7 and split > 1, (variant, split)
    A, B = make_inputs(M, N, K, 0, 1, O.F16, seed_a=11, seed_b=12)
    dA, dB = to_device(A, O.F16), to_device(B, O.F16)
    want = torch.zeros(M * N, dtype=torch.float16, device="cuda")
    loader.gemm(want, dA, dB, M, N, K, 0, 0, 1)
    torch.cuda.synchronize()
    check_against_oracle(to_host(want, O.F16), A, B, M, N, K, 0, 0, 1, O.F16, O.F16)
    rounds = 40
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    out1 = [torch.full_like(want, float("nan")) for _ in range(rounds)]
    out2 = [torch.full_like(want, float("nan")) for _ in range(rounds)]
    for r in range(rounds):
        loader.gemm(out1[r], dA, dB, M, N, K, 0, 0, 1, stream=s1)
        assert loader.gemm_noalloc(out2[r], dA, dB, M, N, K, 0, 0, 1, stream=s2) == RL.OK
    s1.synchronize()
    s2.synchronize()
    for r in range(rounds):
        assert torch.equal(out1[r], want), ("ordinary", r)
        assert torch.equal(out2[r], want), ("no-alloc", r)


def test_noalloc_entry_point_under_graph_capture_without_a_library_buffer(loader):
    """What the entry point is for: a caller that cannot allocate.  With the library's own
    scratch buffer released, a split-K plan, a padded-copy plan and a shared-tile plan are
    recorded into a HIP graph through the no-alloc entry point (a capture forbids
    allocation and synchronisation: either would fail the capture), replayed with eager
    work in between, and compared bit for bit with the eager results; device memory in use
    does not change across the calls."""
    import torch

    import rocm_wmma_gemm_amd.loader as RL

    cases = [(128, 4096, 4096, 1, 1, 0, "f16_f16"),      # split-K planes
             (1025, 1031, 2049, 0, 0, 1, "bf16_bf16"),   # padded copies
             (16, 1024, 8192, 0, 0, 1, "f16_f16")]       # workgroups that share tiles
    dev = []
    for (M, N, K, lc, la, lb, tname) in cases:
        din, dout = TYPE_PAIRS[tname]
        A, B = make_inputs(M, N, K, la, lb, din, seed_a=21, seed_b=22)
        dA, dB = to_device(A, din), to_device(B, din)
        want = torch.full((M * N,), float("nan"), dtype=torch_dtype(dout), device="cuda")
        # (eager warm-up of the entry point: the one-time hipGetSymbolAddress per device)
        assert loader.gemm_noalloc(want, dA, dB, M, N, K, lc, la, lb) == RL.OK
        dev.append((dA, dB, want, torch.full_like(want, float("nan"))))
    torch.cuda.synchronize()
    # (gives the library's own buffer back, unless a graph captured by an earlier test
    # holds it: either way the calls below must not touch, create or grow it)
    loader.workspace_release()
    free_before, _ = torch.cuda.mem_get_info()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for (M, N, K, lc, la, lb, tname), (dA, dB, want, out) in zip(cases, dev):
            assert loader.gemm_noalloc(out, dA, dB, M, N, K, lc, la, lb) == RL.OK
    for replay in range(3):
        for (_, _, _, out) in dev:
            out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for case, (_, _, want, out) in zip(cases, dev):
            assert torch.equal(out, want), (replay, case)
        # eager no-alloc work between the replays
        M, N, K, lc, la, lb, tname = cases[0]
        assert loader.gemm_noalloc(dev[0][3], dev[0][0], dev[0][1], M, N, K, lc, la, lb) == RL.OK
        torch.cuda.synchronize()
    free_after, _ = torch.cuda.mem_get_info()
    assert free_after >= free_before - (8 << 20), (free_before, free_after)  # (the graph's own nodes)
