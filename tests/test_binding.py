"""The Python binding extension (csrc/binding.cpp): every argument check that
kernels.py made in Python still refuses what it refused, with the same error,
and the launches go to the current stream."""
from __future__ import annotations

import threading

import pytest

torch = pytest.importorskip("torch")

from qwenasr_amd import _lib, kernels as K  # noqa: E402


def test_every_bound_entry_point_is_in_the_table():
    bound = _lib.bind(K._need, (K.F32, K.I8, K.I32, K.U16))
    assert set(bound) <= set(_lib.SIGNATURES)
    with pytest.raises(AttributeError):
        K._call.qasr_no_such_entry


def test_cpu_tensors_and_wrong_objects_are_refused():
    t = torch.empty(8)
    for bad, text in ((t, "must be a device tensor"), (None, "expected a torch tensor"), (3, "expected a torch tensor")):
        with pytest.raises(TypeError, match="out: " + text):
            K.rms_norm(bad, t, t, 1, 8, 1e-6)
    with pytest.raises(ValueError, match="one output per weight"):
        K.linear_nobias_int8_multi([t], [], t, 1, 8)
    with pytest.raises(TypeError, match="too few arguments"):
        K._call.qasr_add_inplace_f32()


def test_a_host_without_the_headers_gets_the_libraries(monkeypatch, tmp_path, capsys):
    """Without torch, its headers, Python's or g++ the build leaves the binding out and says
    why; with them a failing compile is still an error."""
    import sys

    from qwenasr_amd import build

    assert build.binding_missing() == ""
    so = tmp_path / "_binding.so"
    monkeypatch.setattr(build, "BINDING", so)
    monkeypatch.setattr(build, "BUILD", tmp_path)
    for change, text in ((lambda m: m.setitem(sys.modules, "torch", None), "torch cannot be imported"),
                         (lambda m: m.setattr(build, "_binding_includes", lambda: [tmp_path]), "no torch/csrc"),
                         (lambda m: m.setattr(build.shutil, "which", lambda _: None), "no g++")):
        so.write_bytes(b"old")
        with monkeypatch.context() as m:
            change(m)
            assert build.build_binding() is None
        assert not so.exists() and "not built: " + text in capsys.readouterr().err
    with monkeypatch.context() as m:
        m.setattr(build, "CSRC", tmp_path)  # no source there
        with pytest.raises(RuntimeError, match="command failed"):
            build.build_binding()


@pytest.mark.gpu
def test_checks_on_device_tensors(dev):
    x, w = torch.ones(64, device=dev), torch.ones(16, device=dev)
    out = torch.empty(64, device=dev)
    with pytest.raises(IndexError, match="x: range end index 80 out of range for slice of length 64"):
        K.rms_norm(torch.empty(80, device=dev), x, w, 5, 16, 1e-6)
    with pytest.raises(TypeError, match="weight: expected torch.float32, got torch.float64"):
        K.rms_norm(out, x, w.double(), 4, 16, 1e-6)
    with pytest.raises(ValueError, match="x: must be contiguous"):
        K.rms_norm(out, torch.ones(64, 2, device=dev)[:, 0], w, 4, 16, 1e-6)
    with pytest.raises(TypeError):
        K.rms_norm(out, x, w, 4.0, 16, 1e-6)
    with pytest.raises(TypeError, match="delta: expected a torch tensor, got NoneType"):
        K.add_rms_norm(x, None, w, out, 4, 16, 1e-6)
    with pytest.raises(K.QasrError) as e:  # an odd head size: the library's own status and message
        K.apply_rope_neox(x, x, x, 1, 1, 15)
    assert e.value.code == _lib.QASR_ERR_INVALID_ARG and "even" in e.value.msg
    q = K.QuantWeight(torch.ones(16 * 16, dtype=torch.int8, device=dev), torch.ones(16, device=dev), 16, 16)
    with pytest.raises(IndexError, match="w: range end index 512"):
        K.linear_nobias_int8_multi([out], [q], x, 2, 32)
    # parameters and views are tensors like any other; None where the entry allows it
    K.rms_norm(out, torch.nn.Parameter(x), w, 4, 16, 1e-6)
    K.linear_int8(out, x, q.data, q.scales, None, 4, 16, 16)
    assert torch.equal(out, torch.full_like(out, 16.0))


@pytest.mark.gpu
def test_launches_follow_the_current_stream_and_thread(dev):
    a, b = torch.zeros(1 << 20, device=dev), torch.ones(1 << 20, device=dev)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    parts = [a[: 1 << 19], a[1 << 19:]]

    def work(i):
        with torch.cuda.stream(streams[i]):
            for _ in range(50):
                K.add_inplace(parts[i], b, 1 << 19)
            streams[i].synchronize()

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert torch.equal(a, torch.full_like(a, 50.0))
    g, s = torch.cuda.CUDAGraph(), torch.zeros(64, device=dev)
    with torch.cuda.graph(g):  # a capture sees the launch only on its own stream
        K.add_inplace(s, b, 64)
    for rep in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(s, torch.full_like(s, rep + 1.0))
