"""Int8 matrices without their copy in MFMA operand order (no memory for it,
or past the context's limit, which the tests lower through
nd_test_copy_limit): every entry point that takes the matrix still does, on
the row-major codes.  The products of nd_matmul are exact integer sums, so
their results equal those with the copy bit for bit; the models stay within
the bars of the tests they are run through.
"""

import ctypes as C
import sys

import numpy as np
import pytest

import oracle
from helpers import hip_runtime
from needle_hip import HipBackend, Int8Matrix, MatrixRowRange, NeedleModel, synth
from needle_hip import lib as L
from needle_hip.models import (ConstrainedWorkload, DecoderGeometry, DecoderWeights,
                               HipDecoder)
from needle_hip.needle2 import Needle2Geometry, Needle2Weights
from test_gpu_decoder import matmul, run_case
from test_gpu_needle2 import SMALL, check_kv, close
from test_gpu_prefill import compare

pytestmark = pytest.mark.gpu


def say(*args):
    print("[case]", *args, file=sys.stderr, flush=True)


@pytest.fixture(scope="module", params=[0, 1 << 20])
def bare(request):
    """A context without copies, and one whose copies end at 1 MiB: its small
    matrices have one and its models' later ones do not."""
    with HipBackend() as backend:
        backend._check(backend.lib.nd_test_copy_limit(backend.ctx, request.param))
        yield backend


@pytest.mark.parametrize("rows,n,k", [(1, 300, 512), (33, 65, 128), (64, 9000, 512),
                                      (129, 512, 512), (700, 512, 2048)])
def test_matmul_from_row_major_codes(hip, bare, rows, n, k):
    say("matmul without copy", rows, n, k)
    w, s = synth.int8_matrix(81, f"bare{n}x{k}", n, k, k)
    m = Int8Matrix(w, s, k)
    x = synth.Stream(81, f"barex{rows}").normal((rows, k))
    got, want = matmul(bare, m, x), matmul(hip, m, x)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n,k,g,batch", [(70, 256, 32, 3), (100, 512, 64, 12), (65, 4096, 32, 8)])
def test_batched_matvec_from_row_major_codes(bare, n, k, g, batch):
    """At most k + 1 fp32 roundings a row on the vector kernel: 2^-24 (k + 1) of
    the absolute sum."""
    say("matvec without copy", n, k, g, batch)
    w, s = synth.int8_matrix(82, f"barev{n}x{k}", n, k, g)
    x = synth.Stream(82, f"barevx{batch}").normal((batch, k))
    full = w.astype(np.float64) * np.repeat(s.astype(np.float64), g, axis=1)
    got = bare.matvec(Int8Matrix(w, s, g), x, MatrixRowRange(1, n - 1)).astype(np.float64)
    want = x.astype(np.float64) @ full[1:].T
    bound = 2.0 ** -24 * (k + 1) * (np.abs(x).astype(np.float64) @ np.abs(full[1:]).T)
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) / bound)


def test_prefill_from_row_major_codes(bare):
    say("prefill without copy")
    compare(bare, DecoderGeometry(layers=2, vocab=4096), 300, 5)


def test_batch_decode_from_row_major_codes(bare):
    say("batch decode without copy")
    g = DecoderGeometry(layers=2, vocab=4096)
    run_case(bare, g, ConstrainedWorkload(batch=3, steps=3, min_context=1, max_context=300,
                                          vocab=g.vocab), seed=11)


def test_copies_take_their_share_and_no_more(hip):
    """The copies counted through free memory: 64 MB more for 64 MB of codes, none
    for groups that no matrix-core kernel reads or past the limit, and given
    back with the matrix; a decoder keeps one form of its joined projections."""
    say("memory of the copies")
    lib, mb = hip_runtime(), 1 << 20
    lib.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    free, total = C.c_size_t(), C.c_size_t()

    def now():
        assert lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    n, k = 16384, 4096
    w = np.ones((n, k), np.int8)

    def taken(backend, g):
        s = np.ones((n, k // g), np.float32)
        handle, before = C.c_void_p(), now()
        backend._check(backend.lib.nd_mat_upload_i8(backend.ctx, L.ptr(w), L.ptr(s), n, k, g,
                                                    C.byref(handle)))
        grown = before - now()
        backend._check(backend.lib.nd_mat_free(backend.ctx, handle))
        assert abs(before - now()) < 4 * mb
        return grown / mb

    with HipBackend() as backend:
        assert abs(taken(backend, 4096) - 128) < 8
        assert abs(taken(backend, 16) - 80) < 8  # codes and 16 MB of scales
        backend._check(backend.lib.nd_test_copy_limit(backend.ctx, 60 * mb))
        assert abs(taken(backend, 4096) - 64) < 8
    with HipBackend() as backend:
        g = DecoderGeometry(layers=4, dim=2048, heads=32, kv_heads=32, ffn=2048, vocab=64)
        weights = DecoderWeights(g, 1)
        for role in ("wq", "wk", "wv", "wo", "wup", "wdown"):
            for m in getattr(weights, role):
                backend.upload(m)
        backend.upload(weights.embedding)
        before = now()
        dec = HipDecoder(backend, weights)
        # 4 layers of 6144 x 2048, and one more that the runtime may give back
        # only with the stream's next work.
        assert -8 < (before - now()) / mb - 4 * 12 < 12 + 8
        dec.free()


def test_needle_prompt_from_row_major_codes(bare):
    say("needle2 without copy")
    g = Needle2Geometry(**{**SMALL.__dict__, "kv_window": 160, "max_length": 200})
    w = Needle2Weights(g, 46)
    model = NeedleModel(bare, w)
    try:
        rt = model.create_resident_runtime()
        rt.reset(g.max_length, 3)
        ref = oracle.Needle2(w).runtime(g.max_length, 3)
        ref.capture_kv(0, g.max_length)
        tokens = synth.Stream(15, "n2bare").integers(134, 0, g.vocab - 1)
        got = rt.prefill(tokens[:130])
        for t in tokens[:130]:
            want = ref.step(int(t))
        close(got, want, "prompt")
        check_kv(model, ref, g, 130, 3, "prompt without copies")
        for t in tokens[130:]:
            close(rt.step(int(t)), ref.step(int(t)), "step")
    finally:
        model.dispose()
