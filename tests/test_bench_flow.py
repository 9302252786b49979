"""Statements of bench.py that no run reaches (one of them set what the plate workload needs)."""
import ast
import os

from conftest import ROOT


def test_no_statement_stands_behind_a_return():
    tree = ast.parse(open(os.path.join(ROOT, "bench.py")).read())
    for node in ast.walk(tree):
        for body in (getattr(node, k, None) for k in ("body", "orelse", "finalbody")):
            if isinstance(body, list):
                ends = [i for i, s in enumerate(body) if isinstance(s, (ast.Return, ast.Raise))]
                assert not ends or ends[0] == len(body) - 1, f"bench.py:{body[ends[0] + 1].lineno}"
