"""A kernel launch that the runtime refuses is reported by the call that made it.

The refusal is the runtime's own, on the host: a launch on a stream whose capture has been invalidated (here by
waiting for the stream while it captures) returns an error and nothing runs.  Every apply route must pass it on;
once the capture has ended the same calls succeed."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _InvalidatedCapture:
    """a stream of its own, set as the library's, whose capture has been invalidated"""

    def __init__(self, hip):
        from lfric_core_amd import _lib
        self.lib = _lib.lib()
        self.rt = ctypes.CDLL(str(_lib.LIB_PATH))  # its dependency is the HIP runtime in use
        self.stream = ctypes.c_void_p()

    def __enter__(self):
        assert self.rt.hipStreamCreateWithFlags(ctypes.byref(self.stream), 1) == 0
        assert self.rt.hipStreamBeginCapture(self.stream, 2) == 0  # relaxed: other streams are not concerned
        assert self.rt.hipStreamSynchronize(self.stream) != 0
        assert self.lib.lfric_set_stream(self.stream) == 0

    def __exit__(self, *exc):
        self.lib.lfric_set_stream(None)
        graph = ctypes.c_void_p()
        assert self.rt.hipStreamEndCapture(self.stream, ctypes.byref(graph)) != 0 and not graph.value
        self.rt.hipGetLastError()
        assert self.rt.hipStreamDestroy(self.stream) == 0


def _operators(hip):
    w0, w01 = hip.FunctionSpace.cubedsphere(4, 3), hip.FunctionSpace.cubedsphere(3, 2, hip.W0, 1)
    w2 = hip.FunctionSpace.cubedsphere(4, 3, hip.W2, 0)
    for fs, kw in ((w0, {}), (w01, {}), (w2, dict(shift=1.0))):
        op = hip.LmaOperator(fs).generate_spd(1, **kw)
        yield op
        yield op.convert(hip.R32)
    for copy in ("prepare_rows", "prepare_symmetric"):
        op = hip.LmaOperator(w0).generate_spd(1)
        getattr(op, copy)()
        yield op
    op = hip.LmaOperator(w01).generate_spd(1)
    op.prepare_symmetric()
    yield op


def test_refused_launches_are_reported(hip):
    for op in _operators(hip):
        x, y = hip.FieldVector(op.fs_to, op.precision).fill_uniform(1), hip.FieldVector(op.fs_to, op.precision)
        linop = hip.LinearOperator.from_lma(op)
        calls = [op.apply, op.apply_gather, linop.apply]
        if op.fs_to.ndf == 6:
            calls.append(hip.LinearOperator.mass_matrix(op, True).apply)
        good = []
        for call in calls:  # builds the lists
            call(x, y)
            good.append(y.export_raw())
        hip.synchronize()
        with _InvalidatedCapture(hip):
            for call in calls:
                with pytest.raises(hip.LfricError):
                    call(x, y)
        for call, want in zip(calls, good):
            y.set_scalar(7.0)
            call(x, y)
            np.testing.assert_array_equal(y.export_raw(), want)
