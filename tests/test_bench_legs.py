"""bench.py's legs: each stands in main() once, and runs on its own (--only) with what main() has set up ahead of the legs."""
import ast
import builtins
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def legs_and_rest():
    with open(os.path.join(ROOT, "bench.py")) as f:
        module = ast.parse(f.read())
    main = next(n for n in module.body if isinstance(n, ast.FunctionDef) and n.name == "main")

    def leg(stmt):  # if args.only in (None, "<leg>"):
        t = stmt.test if isinstance(stmt, ast.If) else None
        if isinstance(t, ast.Compare) and isinstance(t.left, ast.Attribute) and t.left.attr == "only":
            return [c.value for c in t.comparators[0].elts if c.value is not None][0]

    return module, [(leg(s), s) for s in main.body if leg(s)], [s for s in main.body if not leg(s)]


def bound(node):
    """Names that are given a value anywhere below the node."""
    out = set()
    for n in ast.walk(node):
        if isinstance(n, ast.Name) and isinstance(n.ctx, (ast.Store, ast.Del)):
            out.add(n.id)
        elif isinstance(n, (ast.FunctionDef, ast.ClassDef)):
            out.add(n.name)
        elif isinstance(n, ast.arg):
            out.add(n.arg)
        elif isinstance(n, ast.ExceptHandler) and n.name:
            out.add(n.name)
        elif isinstance(n, (ast.Import, ast.ImportFrom)):
            out.update((a.asname or a.name).split(".")[0] for a in n.names)
    return out


def test_every_leg_stands_once_and_uses_no_other_leg():
    module, legs, rest = legs_and_rest()
    names = [name for name, _ in legs]
    assert len(names) >= 8 and len(names) == len(set(names)), names
    outside = set(dir(builtins)) | {"__file__"}
    for s in module.body:
        outside |= bound(s) if not isinstance(s, ast.FunctionDef) else {s.name}
    first = legs[0][1].lineno
    for s in rest:
        if s.lineno < first:
            outside |= bound(s)
    for name, s in legs:
        used = {n.id for n in ast.walk(s) if isinstance(n, ast.Name) and isinstance(n.ctx, ast.Load)}
        assert not used - outside - bound(s), f"leg {name}: {sorted(used - outside - bound(s))}"
