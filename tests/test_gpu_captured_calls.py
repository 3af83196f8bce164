"""Calls under stream capture, in a workspace that an earlier, larger call has grown: the graph stays
valid through any smaller call, whatever workspace that one would like."""
import ctypes

import numpy as np
import pytest

import oracle as O
from fk20_amd import ops, synthetic as S
from fk20_amd.lib import DeviceBuffer, Stream, call, lib, synchronize

pytestmark = pytest.mark.gpu


def hip(name, *args):
    f = getattr(lib(), name)  # of the runtime the library is linked with
    f.restype = ctypes.c_int
    assert f(*args) == 0, name


class Graph:
    """The calls that `record(stream)` makes, captured."""

    def __init__(self, record):
        self.stream = Stream()
        s = ctypes.c_void_p(self.stream.handle)
        graph, self.exe = ctypes.c_void_p(), ctypes.c_void_p()
        hip("hipStreamBeginCapture", s, 1)  # thread-local
        try:
            record(self.stream.handle)
        finally:
            hip("hipStreamEndCapture", s, ctypes.byref(graph))
        hip("hipGraphInstantiate", ctypes.byref(self.exe), graph, None, None, ctypes.c_size_t(0))
        hip("hipGraphDestroy", graph)

    def replay(self):
        hip("hipGraphLaunch", self.exe, ctypes.c_void_p(self.stream.handle))
        self.stream.synchronize()

    def destroy(self):
        hip("hipGraphExecDestroy", self.exe)
        self.stream.destroy()


def test_drop_in_calls():
    N, n = 1024, 128
    xext = O.xext_fft_from_tau(S.random_secret(71), N)
    poly = S.random_polys(3, N, 72)
    x = ops.g1p_op("mul", np.tile(O.g1p_gen(), (12 * n, 1)), k=S.random_fr(12 * n, 73)).reshape(12, n, 18)
    tc = S.random_fr(20 * 16 * n, 74).reshape(20, 16, n, 4)
    # the largest workspace of them all: every later call's need fits in it
    big = ops.g1p_op("mul", np.tile(O.g1p_gen(), (512 * 256, 1)), k=S.random_fr(512 * 256, 75)).reshape(512, 256, 18)
    ops.g1p_fft(big)
    want = {"g1p_fft": ops.g1p_fft(x[:2]), "g1p_ift": ops.g1p_fft(x, inverse=True),
            "fk20_hext_fft2h_fft": ops.hext_fft2h_fft(x[:3]), "fk20_poly2h_fft": ops.poly2h_fft(poly, xext),
            "fk20_msm": ops.to_affine(ops.msm(tc, xext))}
    xb, pb, tb, eb = (DeviceBuffer.from_array(a) for a in (x, poly, tc, xext))
    args = {"g1p_fft": (2, (xb.ptr, 2, n)), "g1p_ift": (12, (xb.ptr, 12, n)),
            "fk20_hext_fft2h_fft": (3, (xb.ptr, 3, n)), "fk20_poly2h_fft": (3, (pb.ptr, eb.ptr, 3, N)),
            "fk20_msm": (20, (tb.ptr, eb.ptr, 20, n))}
    outs = {f: DeviceBuffer(rows * n * 144) for f, (rows, _) in args.items()}
    graphs = {f: Graph(lambda s, f=f, a=a: call(f, outs[f].ptr, *a, s)) for f, (_, a) in args.items()}
    for again in range(3):
        for f, g in graphs.items():
            outs[f].fill(0x5A)
            g.replay()
            got = outs[f].download((args[f][0], n, 18))
            assert np.array_equal(ops.to_affine(got) if f == "fk20_msm" else got, want[f]), (f, again)
        # calls whose needs are smaller and whose wishes are not
        ops.msm(S.random_fr(66 * 16 * n, again).reshape(66, 16, n, 4), xext)
        ops.g1p_fft(big[: 2 + again])
        ops.g1p_fft(x[: 5 + again], inverse=True)
        synchronize()
    for g in graphs.values():
        g.destroy()
