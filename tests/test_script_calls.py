"""Scripts that call entries of the kernel library themselves pass as many arguments as the library's bindings declare."""
import ast
import glob
import os

import pytest

from llm_sharding_amd.ops import hip

SCRIPTS = sorted(glob.glob(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "scripts", "*.py")))


def _calls(path):
    """(line, entry, arguments) of the calls without starred arguments, and of declarations written out."""
    with open(path) as fh:
        tree = ast.parse(fh.read())
    for n in ast.walk(tree):
        if isinstance(n, ast.Call) and isinstance(n.func, ast.Attribute) and n.func.attr.startswith("lsa_") \
                and not any(isinstance(a, ast.Starred) for a in n.args):
            yield n.lineno, n.func.attr, len(n.args)
        if isinstance(n, ast.Assign) and isinstance(n.value, ast.List) and isinstance(n.targets[0], ast.Attribute) \
                and n.targets[0].attr == "argtypes" and isinstance(n.targets[0].value, ast.Attribute):
            yield n.lineno, n.targets[0].value.attr, len(n.value.elts)


@pytest.mark.skipif(not os.path.exists(hip.KERNELS_SO), reason="kernel library not built")
def test_arguments():
    lib, wrong, seen = hip.lib(), [], 0
    for path in SCRIPTS:
        for line, name, given in _calls(path):
            declared = getattr(getattr(lib, name, None), "argtypes", None)  # None: of a probe's own library
            seen += declared is not None
            if declared is not None and given != len(declared):
                wrong.append(f"{os.path.basename(path)}:{line}: {name} with {given} of {len(declared)} arguments")
    assert seen >= 8 and not wrong, wrong
