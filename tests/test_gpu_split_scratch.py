"""Calls whose partial sums pass through scratch (K runs, the weight-streaming W4A16 kernel), where the
life of that scratch matters: recorded in graphs, and several at once on one artifact. Every output is
compared bit for bit with the same call made alone: runs are added in order, so it does not vary."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import intent_amd as intent
from intent_amd import inputs

pytestmark = pytest.mark.gpu


def _dev(d, *names):
    return tuple(torch.from_numpy(np.ascontiguousarray(d[n])).cuda() for n in names)


def _w4(M, K, N):
    return lambda seed: _dev(inputs.config1_w4a16_decode(seed, M=M, K=K, N=N), "x", "packed", "scales", "zeros")


def _fp8(M, KB, N):
    def make(seed):
        rng = np.random.default_rng(seed)
        bits = [torch.from_numpy(rng.integers(0, 0x78, size=(r, KB, 128), dtype=np.uint8)).cuda().view(torch.float8_e4m3fn)
                for r in (M, N)]
        scales = [torch.from_numpy(rng.random((r, KB), dtype=np.float32) + 0.25).cuda() for r in (M, (N + 127) // 128)]
        return (*bits, *scales)
    return make


# name: definition, inputs of a seed, start of the kernel's name. The streaming kernel at 128 rows asks for more
# than the default 64 KB of LDS on each launch.
CASES = {
    "w4a16_m12": (intent.weight_only_int4_asym_matmul, _w4(12, 4096, 11008), "w4a16_skinny"),
    "w4a16_m128": (intent.weight_only_int4_asym_matmul, _w4(128, 4096, 1024), "w4a16_skinny"),
    "w4a16_m200": (intent.weight_only_int4_asym_matmul, _w4(200, 4096, 1024), "w4a16_gemm<"),
    "w8a16_m48": (intent.weight_only_int8_matmul,
                  lambda seed: _dev(inputs.config0_w8a16(seed, M=48, K=4096, N=640), "x", "w", "scales"), "w8a16_matmul<"),
    "w8a8_m32": (intent.w8a8_scaled_matmul,
                 lambda seed: _dev(inputs.config3_w8a8(seed, M=32, K=8192, N=1024), "a", "a_scales", "w", "w_scales"),
                 "w8a8_gemm<"),
    "fp8_m40": (intent.deepgemm_fp8_2xacc, _fp8(40, 32, 1030), "deepgemm_fp8<"),
}


def _case(name):
    defn, make, kernel = CASES[name]
    art = intent.compile(defn, target=intent.MI355XTarget(0))
    return art, make, kernel


def _bits(t):
    return t.view(torch.int16)


def _alone(art, args, kernel):
    y = art.run(*args)
    torch.cuda.synchronize()
    name = art.observation.kernel
    assert name.startswith(kernel) and ("runs" in name or name == "w4a16_skinny"), name
    return _bits(y).clone()


def _churn():
    """Eager work that takes and gives back blocks of the allocator, as a program does between replays."""
    for mb in (1, 2, 4, 8, 16):
        torch.full((mb << 18,), float("nan"), device="cuda")
    torch.cuda.synchronize()


def _replays(art, args, make, kernel, out, replay):
    """Several replays with new inputs in place and eager work between them, each against the eager result."""
    for seed in (11, 12, 11, 13):
        for dst, src in zip(args, make(seed)):
            dst.copy_(src)
        want = _alone(art, args, kernel)
        _churn()
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        replay()
        torch.cuda.synchronize()
        assert torch.equal(_bits(out), want), seed


@pytest.mark.parametrize("name", sorted(CASES))
def test_split_call_in_a_graph(gpu, name):
    art, make, kernel = _case(name)
    args = make(11)
    _alone(art, args, kernel)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = art.run(*args)
    _replays(art, args, make, kernel, out, graph.replay)


@pytest.mark.parametrize("name", sorted(CASES))
def test_prepared_split_call_in_a_stream_capture(gpu, name):
    # A plain capture of the stream: no private pool keeps what is allocated inside it, and a prepared launch
    # allocates nothing.
    art, make, kernel = _case(name)
    args = make(11)
    _alone(art, args, kernel)
    call = art.prepare(*args)
    hip = ctypes.CDLL("libamdhip64.so")
    stream = torch.cuda.Stream()
    handle, graph, execution = ctypes.c_void_p(stream.cuda_stream), ctypes.c_void_p(), ctypes.c_void_p()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        call.launch()
        torch.cuda.synchronize()
        assert hip.hipStreamBeginCapture(handle, 1) == 0  # thread-local
        call.launch()
        assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(execution), graph, None, None, ctypes.c_size_t(0)) == 0
    try:
        def replay():
            assert hip.hipGraphLaunch(execution, handle) == 0

        _replays(art, args, make, kernel, call.result(), replay)
    finally:
        torch.cuda.synchronize()
        hip.hipGraphExecDestroy(execution)
        hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("name", sorted(CASES))
def test_split_calls_on_streams_and_threads(gpu, name):
    art, make, kernel = _case(name)
    sets = [make(seed) for seed in (21, 22, 23)]
    want = [_alone(art, args, kernel) for args in sets]
    errors = []

    def work(args, want):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                outs = [art.run(*args) for _ in range(20)]
                prepared = art.prepare(*args)
                prepared.launch()
            stream.synchronize()
            for y in (*outs, prepared.result()):
                assert torch.equal(_bits(y), want)
            stream.synchronize()
        except Exception as error:  # noqa: BLE001 - reported by the test's own thread
            errors.append(error)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=pair) for pair in zip(sets, want)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


def test_prepared_split_call_on_another_stream_is_dropped(gpu):
    # Its scratch belongs to the stream that prepared it; a launch on another one keeps it from being reused
    # there until that launch is over.
    art, make, kernel = _case("w8a8_m32")
    args = make(31)
    want = _alone(art, args, kernel)
    side = torch.cuda.Stream()
    outs = []
    for _ in range(20):
        call = art.prepare(*args)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            call.launch()
        outs.append(call.result())
        size = call._binding.workspace.numel()
        del call
        torch.full((size,), 0x7F, dtype=torch.uint8, device="cuda")  # would take the block of the scratch
    torch.cuda.synchronize()
    for y in outs:
        assert torch.equal(_bits(y), want)
