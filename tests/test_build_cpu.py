"""The incremental build compiles an object again when a header it includes is newer."""
import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_objects_depend_on_every_kernel_header(monkeypatch):
    spec = importlib.util.spec_from_file_location("_tpr_build", os.path.join(ROOT, "tensorplay_amd", "build.py"))
    B = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(B)
    seen = {}
    monkeypatch.setattr(B, "_newer", lambda target, deps: seen.setdefault(target, deps) and False)
    _, objs = B._tpr_compiles(False, False)
    rocm = os.path.join(B.CSRC, "rocm")
    headers = {os.path.join(rocm, h) for h in os.listdir(rocm) if h.endswith(".h")}
    headers.add(os.path.join(ROOT, "include", "tpr_rocm.h"))
    assert len(headers) >= 4
    for o in objs:
        assert headers <= set(seen[o]), (o, headers - set(seen[o]))
