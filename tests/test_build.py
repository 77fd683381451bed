"""What the build runs, in which order (CPU, nothing is compiled)."""
import pytest

from retrievalattention_amd import build


def test_the_library_and_its_example_do_not_wait_for_the_python_module(monkeypatch):
    """The module for Python is the only part that needs torch's headers: without them the library and the C program over it are
    there all the same, and the build still fails.  One compiler makes everything, with its warnings on."""
    made = []

    def run(command):
        if any(x.endswith("step_calls.cpp") for x in command):
            raise RuntimeError("no headers")
        made.append(command)
        return ""
    monkeypatch.setattr(build, "_run", run)
    with pytest.raises(RuntimeError, match="no headers"):
        build.build()
    outputs = [c[c.index("-o") + 1] for c in made]
    assert build.LIB in outputs and build.CAPI_EXAMPLE in outputs
    module = build.step_calls_command(made[0][0])
    assert {c[0] for c in made} == {module[0]}
    assert "-w" not in module and "-Wall" in module and sum(x.startswith("-O") for x in module) == 1
