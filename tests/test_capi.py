"""The C-ABI library loads and exports every symbol include/*.h declares
(no device calls; runs without a GPU)."""
import re
from pathlib import Path

import daxtoolkit_amd
from daxtoolkit_amd import _lib

ROOT = Path(__file__).resolve().parent.parent


def declared_in_headers():
    names = set()
    for h in (ROOT / "include").glob("*.h"):
        text = re.sub(r"/\*.*?\*/", "", h.read_text(), flags=re.S)
        for m in re.finditer(r"^\s*[A-Za-z_][\w\s\*]*?\b(dax_hip_\w+)\s*\(", text, flags=re.M):
            names.add(m.group(1))
    return names


def test_library_exports_every_declared_symbol():
    lib = daxtoolkit_amd.load_library()
    names = declared_in_headers()
    assert len(names) >= 20
    missing = [n for n in sorted(names) if not hasattr(lib, n)]
    assert not missing, missing


def test_python_binding_covers_header():
    names = declared_in_headers()
    bound = set(_lib.declared_symbols())
    assert names == bound, (sorted(names - bound), sorted(bound - names))


def test_version_and_error_string():
    lib = daxtoolkit_amd.load_library()
    assert lib.dax_hip_version().startswith(b"daxhip")
    assert isinstance(lib.dax_hip_last_error(), bytes)


def test_workspace_size_is_host_only():
    lib = daxtoolkit_amd.load_library()
    assert lib.dax_hip_mc_workspace_bytes(0, 1, 1) == 0
    b = lib.dax_hip_mc_workspace_bytes(512, 512, 512)
    # bit words (P/8), prefixes (4 bytes a word), endpoint words and prefixes (10)
    assert 512**3 // 8 <= b < 512**3 // 8 * 3


def test_span_threshold_setter_is_host_only():
    lib = daxtoolkit_amd.load_library()
    assert lib.dax_hip_mc_backward_set_span_threshold(-1) != 0
    assert b"negative" in lib.dax_hip_last_error()
    assert lib.dax_hip_mc_backward_set_span_threshold(0) == 0
    assert lib.dax_hip_mc_backward_set_span_threshold(16) == 0


def test_default_tuning_as_set():
    """Sizes without a tuning of their own take the default that a caller sets,
    whatever it is; before that they follow from the size (a process of its
    own: the default holds for the process)."""
    import subprocess
    import sys
    code = """
from daxtoolkit_amd import mc
shapes = [(300, 300, 300), (20, 20, 20), (700, 700, 700)]
built_in = mc.get_tuning((0, 0, 0))
by_size = [mc.get_tuning(s) for s in shapes]
assert any(t != built_in for t in by_size)
mc.set_tuning((20, 20, 20), [8, 1, 2, 128, 1])
for default in (built_in, [2, 4, 1, 256, 0], built_in):
    mc.set_tuning((0, 0, 0), default)
    assert mc.get_tuning((0, 0, 0)) == default
    assert mc.get_tuning(shapes[0]) == mc.get_tuning(shapes[2]) == default
    assert mc.get_tuning(shapes[1]) == [8, 1, 2, 128, 1]
"""
    subprocess.run([sys.executable, "-c", code], check=True, cwd=ROOT, timeout=300)
