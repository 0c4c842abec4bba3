"""What is built from what (no GPU, nothing is compiled)."""
import subprocess


def _commands(*goals):
    import fieldfare_moe as ff
    return subprocess.run(["make", "-n", "-B", "-C", str(ff.CSRC), "PYTHON=false", *goals], capture_output=True, text=True).stdout


def test_the_library_is_the_default_and_needs_no_torch():
    lib = _commands()
    assert "libfieldfare_moe_hip.so" in lib and "HASH_PATH" in lib
    assert "binding" not in lib.lower() and "torch" not in lib
    both = _commands("all")
    assert "binding.cpp" in both and "BINDING_HASH_PATH" in both and "libfieldfare_moe_hip.so" in both


def test_a_change_of_flags_rebuilds_what_they_build():
    # the digest beside each covers the Makefile: an object with the old flags would pass for one with the new
    import fieldfare_moe as ff
    lines = subprocess.run(["make", "-n", "-W", "Makefile", "-C", str(ff.CSRC), "PYTHON=false", "all"], capture_output=True, text=True).stdout
    for source in ff.CSRC.glob("*.hip"):
        assert f"-c {source.name} -o {source.stem}.o" in lines, source.name
    assert "binding.cpp -o" in lines


def test_a_module_for_another_torch_is_stale(monkeypatch):
    import torch
    import fieldfare_moe as ff
    assert not ff.is_stale()
    monkeypatch.setattr(torch, "__version__", torch.__version__ + ".other")
    assert ff.is_stale()
    monkeypatch.undo()
    monkeypatch.setattr(ff, "HASH_PATH", ff.HASH_PATH.with_name("none"))
    assert ff.is_stale()
