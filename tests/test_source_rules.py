"""Rules that the sources keep, checked on their text (CPU)."""
import ast
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_wave_barriers_carry_fences():
    """A wave barrier alone orders no memory access: lanes that exchange data through LDS do so across a barrier with a
    wavefront-scope release fence before it and an acquire fence after it."""
    found = 0
    for path in glob.glob(os.path.join(ROOT, "nibble_amd", "csrc", "**", "*"), recursive=True):
        if not path.endswith((".hip", ".h")):
            continue
        with open(path) as f:
            text = f.read()
        fenced = re.findall(r'__builtin_amdgcn_fence\(__ATOMIC_RELEASE, "wavefront"\);\s*'
                            r'__builtin_amdgcn_wave_barrier\(\);\s*'
                            r'__builtin_amdgcn_fence\(__ATOMIC_ACQUIRE, "wavefront"\);', text)
        found += len(fenced)
        assert text.count("__builtin_amdgcn_wave_barrier") == len(fenced), os.path.relpath(path, ROOT)
    assert found


def test_every_test_is_collected():
    """A module's second definition of a name replaces the first, which pytest then never sees."""
    for path in glob.glob(os.path.join(ROOT, "tests", "*.py")):
        with open(path) as f:
            tree = ast.parse(f.read())
        scopes = [tree] + [n for n in tree.body if isinstance(n, ast.ClassDef)]
        for scope in scopes:
            names = [n.name for n in scope.body if isinstance(n, (ast.FunctionDef, ast.ClassDef))]
            twice = sorted({n for n in names if names.count(n) > 1})
            assert not twice, (os.path.basename(path), twice)
