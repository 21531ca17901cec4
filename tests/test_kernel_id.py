"""The id a build gives its kernel sources: the same for the same code, whatever its
comments and line breaks, another for other code or other flags."""
from octotiger_amd import build


def test_source_id_follows_the_code_only():
    code = "int f(int a) {\n    return a + 1;   // one more\n}\n"
    assert build.source_id([code]) == build.source_id(["/* f */ int f(int a) {\n  return a + 1;\n}"])
    assert build.source_id([code]) != build.source_id([code.replace("+ 1", "+ 2")])
    assert build.source_id([code, "x"]) != build.source_id(["x", code])


def test_kernel_id_depends_on_flags(monkeypatch):
    first = build.kernel_id()
    assert len(first) == 12 and first == build.kernel_id()
    monkeypatch.setattr(build, "HIP_FLAGS", build.HIP_FLAGS + ["-DX"])
    assert build.kernel_id() != first
