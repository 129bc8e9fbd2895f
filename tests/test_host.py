"""Host-side logic of the Python mirror of the reference API (no GPU):
operator/map resolution, dims normalisation and routing, layout merging."""
import operator

import pytest
import torch


def test_operator_and_map_resolution(kf):
    L = kf._lib
    assert kf._op_code(operator.add) == L.OP_ADD == kf._op_code("+")
    assert kf._op_code(max) == L.OP_MAX and kf._op_code(min) == L.OP_MIN
    assert kf._op_code(kf.affine) == L.OP_AFFINE
    assert kf._map_code(kf.identity) == L.MAP_IDENTITY and kf._map_code(kf.abs2) == L.MAP_ABS2
    assert kf._op_code(operator.mul) == L.OP_MUL == kf._op_code("*")
    with pytest.raises(kf.ArgumentError):
        kf._op_code(operator.truediv)
    with pytest.raises(kf.ArgumentError):
        kf._map_code(lambda x: x)


def test_affine_op_is_the_recurrence(kf):
    # (a1,b1) o (a2,b2) applied to x equals applying map 1 then map 2
    p, q, x = (2.0, 1.0), (3.0, 5.0), 7.0
    a, b = kf.affine(p, q)
    assert a * x + b == q[0] * (p[0] * x + p[1]) + q[1]


def test_normalize_and_validate_dims(kf):
    assert kf._normalize_dims(2, 3) == (2,)
    assert kf._normalize_dims((3, 1), 3) == (1, 3)
    with pytest.raises(kf.ArgumentError):
        kf._normalize_dims(4, 3)
    with pytest.raises(kf.ArgumentError):
        kf._normalize_dims(0, 3)
    with pytest.raises(kf.ArgumentError):
        kf._normalize_dims((1, 1), 3)
    # non-positive dims count from the end (reference src/helpers.jl:194-198):
    # d -> nd + d + 1, so -1 is the last dim and 0 is one past it
    assert kf._normalize_dims(-1, 3) == (3,)
    assert kf._normalize_dims((-1, 1), 3) == (1, 3)
    assert kf._normalize_dims(-3, 3) == (1,)
    with pytest.raises(kf.ArgumentError):
        kf._normalize_dims(-4, 3)
    with pytest.raises(kf.ArgumentError):
        kf._normalize_dims((3, -1), 3)


@pytest.mark.parametrize("dims,nd,expected", [
    ((1,), 3, (1, 2)),          # leading only
    ((1, 2), 3, (2, 3)),        # leading block
    ((3,), 3, (0, 1)),          # trailing only
    ((2, 3), 3, (0, 1)),        # trailing block
    ((1, 3), 3, (1, 2)),        # leading + trailing
    ((1, 2, 3), 3, (3, 4)),     # one block touching both ends -> leading
    ((2,), 3, (0, 2)),          # middle -> general
    ((2, 4, 5), 5, (0, 4)),     # not two blocks covering dims -> general
    ((1, 4, 5), 5, (1, 2)),     # lead {1}, tail {4,5}
])
def test_classify_dims_matches_reference_rules(kf, dims, nd, expected):
    # rules of reference src/mapreduce/mapreduce.jl:272-298
    assert kf._classify_dims(dims, nd) == expected


def test_merge_and_matrix_views(kf):
    A = torch.empty(65536, 4096).T          # 4096 x 65536 column-major
    assert kf._as_matrix(A, 1) == (4096, 65536, 4096)
    V = A[:, ::2]                            # view(A, :, 1:2:end)
    assert kf._as_matrix(V, 1) == (4096, 32768, 8192)
    B = torch.empty(4, 5, 6).permute(2, 1, 0)  # 6x5x4 column-major
    assert kf._as_matrix(B, 2) == (30, 4, 30)
    assert kf._as_matrix(B, 1) == (6, 20, 6)
    with pytest.raises(NotImplementedError):
        kf._as_matrix(torch.empty(3, 4), 1)   # row-major: rows are not unit-stride


def test_cpu_tensors_are_rejected(kf):
    x = torch.zeros(10)
    with pytest.raises(kf.ArgumentError, match="GPU"):
        kf.scan("+", x)
    with pytest.raises(kf.ArgumentError, match="GPU"):
        kf.mapreduce(kf.identity, "+", x)


def test_scratch_family_check(kf):
    # a scan buffer must not serve reductions and vice versa (reduction
    # partials written over scan descriptors could read as current ones)
    cpu = torch.device("cpu")
    sbuf = kf.KernelBuffer(kf.Scan1D, 1024, cpu)
    rbuf = kf.KernelBuffer(kf.MapReduce1D, 1024, cpu)
    with pytest.raises(kf.ArgumentError):
        kf._scratch(kf.MapReduce1D, 256, cpu, sbuf)
    with pytest.raises(kf.ArgumentError):
        kf._scratch(kf.MapReduce2D, 256, cpu, sbuf)
    with pytest.raises(kf.ArgumentError):
        kf._scratch(kf.Scan1D, 256, cpu, rbuf)
    assert kf._scratch(kf.MapReduce2D, 256, cpu, rbuf) is rbuf      # one family: shared
    with pytest.raises(kf.ArgumentError):
        kf._scratch(kf.MapReduce1D, 4096, cpu, rbuf)                  # too small


@pytest.mark.parametrize("multi", [False, True])
@pytest.mark.parametrize("error,sync_rc,synced,reused", [
    ("KernelForgeError", 0, True, True),      # a HIP error: the kernel may be queued, so wait for it
    ("KernelForgeError", 1, True, False),     # the wait fails: the slot stays out of the pool
    ("ArgumentError", 0, False, True)])       # refused before any launch
def test_result_slot_of_a_failed_call(kf, monkeypatch, multi, error, sync_rc, synced, reused):
    # a call whose launch check reports a HIP error may have queued the kernel
    # that writes its result slot: the slot must not serve another call before
    # the stream was waited for
    class Lib:
        calls = []

        def hipStreamSynchronize(self, stream):
            self.calls.append(stream)
            return sync_rc

        def hipGetLastError(self):
            return 0

    def fail(*args, **kwargs):
        raise {"KernelForgeError": kf._lib.KernelForgeError, "ArgumentError": kf.ArgumentError}[error]("as a launch does")

    import contextlib
    x, slot, fake = torch.zeros(4), torch.zeros(1), Lib()
    fake.calls.clear()
    monkeypatch.setattr(kf, "_require_device", lambda *ts: None)
    monkeypatch.setattr(kf, "_reduce_full_into", fail)
    monkeypatch.setattr(kf, "_reduce2_into", fail)
    monkeypatch.setattr(kf, "_raw_stream", lambda device: 7)
    monkeypatch.setattr(kf, "_on", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(kf._lib, "lib", lambda: fake)
    monkeypatch.setattr(kf, "_scalar_free", {torch.float32: [slot]})
    with pytest.raises((kf._lib.KernelForgeError, kf.ArgumentError), match="as a launch does"):
        kf.mapreduce("mul", "+", (x, x)) if multi else kf.mapreduce(kf.identity, "+", x)
    assert fake.calls == ([7] if synced else [])
    assert kf._scalar_free[torch.float32] == ([slot] if reused else [])


def test_leading_first_takes_no_layout_that_trailing_first_refuses(kf):
    # the order of the two passes is a matter of speed: which layouts are
    # refused must not depend on it
    import itertools
    taken = 0
    for shape in itertools.product((1, 2, 3, 5), (1, 2, 4), (1, 3), (1, 2, 3)):
        for pad in itertools.product((0, 1), repeat=4):
            full = [s + p for s, p in zip(shape, pad)]
            t = torch.empty(tuple(reversed(full))).permute(3, 2, 1, 0)
            t = t[:shape[0], :shape[1], :shape[2], :shape[3]]
            for lead_end, k in ((1, 3), (1, 2), (2, 3)):
                if kf._leading_first(t, lead_end, None):
                    taken += 1
                    kf._as_matrix(t, k)  # raises where trailing-first refuses
    assert taken > 100
