"""The joined packing of host traces equals the trace-by-trace copy for every form that the entry
point takes: equal and ragged lengths, one trace, empty ones, strided and reversed views, other
dtypes and byte orders, lists, read-only arrays and mixtures."""
import numpy as np
import pytest

from crava_amd import _pack_traces


def _plain(traces):
    stride = max(len(t) for t in traces)
    s = np.zeros((len(traces), stride), dtype=np.float32)
    for k, t in enumerate(traces):
        s[k, :len(t)] = np.asarray(t, dtype=np.float32)
    return s


RNG = np.random.default_rng(3)
A = RNG.standard_normal((7, 12)).astype(np.float32)
FROZEN = A[0].copy()
FROZEN.setflags(write=False)
FORMS = {
    "rows": list(A), "one": [A[0]], "array": A, "ragged": [A[k, :12 - k] for k in range(7)],
    "with an empty one": [A[0], A[1, :0], A[2, :5]], "columns": list(A.T), "reversed": [r[::-1] for r in A],
    "every other": [r[::2] for r in A], "double": list(A.astype(np.float64)), "integers": list((10 * A).astype(np.int32)),
    "big-endian": list(A.astype(">f4")), "lists": [list(map(float, r)) for r in A], "read-only": [FROZEN, A[1]],
    "mixed": [A[0], A[1].astype(np.float64), list(map(float, A[2]))], "transposed array": np.asfortranarray(A),
}


@pytest.mark.parametrize("name", list(FORMS))
def test_pack_traces(name):
    samples, length = _pack_traces(FORMS[name])
    want = _plain(FORMS[name])
    assert samples.dtype == np.float32 and samples.flags.c_contiguous and length.dtype == np.int32
    assert np.array_equal(samples.view(np.uint32), want.view(np.uint32))
    assert list(length) == [len(t) for t in FORMS[name]]


def test_pack_traces_refuses_what_the_copy_refuses():
    for bad in ([np.zeros((3, 2), np.float32), np.zeros(3, np.float32)], [], [np.float32(1.0)],
                [np.zeros((3, 1), np.float32)] * 2):
        with pytest.raises((ValueError, TypeError)):
            _pack_traces(bad)
