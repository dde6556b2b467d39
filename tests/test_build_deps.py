"""What makes a compiled object stale: its source, every header, and the file that holds the compiler's flags."""
import importlib.util
import os

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-hw3_amd")


@pytest.mark.parametrize("target,header", [("qlinear", "ql_gemm_wide.h"), ("seqmix", "sm_common.h"), ("hymix", "hm_attn_tile.h")])
def test_an_object_depends_on_its_flags(monkeypatch, target, header):
    spec = importlib.util.spec_from_file_location("build_under_test", os.path.join(PKG, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    seen = {}
    monkeypatch.setattr(build, "_hipcc", lambda: "hipcc")
    monkeypatch.setattr(build, "_stale", lambda obj, deps: seen.update({obj: [os.path.realpath(d) for d in deps]}))      # (falsy: nothing is built)
    build.build(verbose=False, target=target)
    objects = [deps for obj, deps in seen.items() if obj.endswith(".o")]
    assert objects
    for deps in objects:
        assert os.path.realpath(os.path.join(PKG, "build.py")) in deps
        assert any(os.path.basename(d) == header for d in deps) and any(d.endswith(".hip") for d in deps)
