"""CPU check of the suite itself: no test shadows another of the same name."""
import ast
import collections
import glob
import os

HERE = os.path.dirname(os.path.abspath(__file__))


def test_names_are_defined_once():
    twice = {}
    for path in glob.glob(os.path.join(HERE, "*.py")):
        names = collections.Counter(f.name for f in ast.parse(open(path).read()).body
                                    if isinstance(f, ast.FunctionDef))
        twice.update({(os.path.basename(path), n): c for n, c in names.items() if c > 1})
    assert not twice, twice
