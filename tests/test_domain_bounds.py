"""The bounds by which the code generator leaves fix out (tsi_jit.cpp bound_rule): records whose values
leave +-1e6 somewhere on the domain (cells in [-5,5]^3) keep it, by every rule that takes a minimum or a
maximum of two bounds, and tapes that depend on the clamp match the oracle."""
import numpy as np
import pytest

import oracle
import temporalsetinversion_amd as T
from helpers import run_pair, assert_same_nodes
from temporalsetinversion_amd.scenes import Tape


def tape(f):
    B = Tape()
    return B.to_ll(f(B))


# (field, records that keep fix: those whose bound leaves +-1e6, and everything computed from them)
FIELDS = {
    # 5000 x 5000: the product and the RET
    "product": (lambda B: B.mul(B.mul(B.x, 1000.0), B.mul(B.y, 1000.0)), 2),
    # [-500, 2500]^2: the square and the RET
    "square": (lambda B: B.sq(B.add(B.mul(B.x, 300.0), 1000.0)), 2),
    # [-5, 5] / -1e-6: the quotient and the RET
    "quotient": (lambda B: B.div(B.x, -1e-6), 2),
    # max(x, 2e6), min(x, -2e6)
    "max-literal": (lambda B: B.max(B.x, 2e6), 2),
    "min-literal": (lambda B: B.min(B.x, -2e6), 2),
    # sums of 3 up to 9e5 each: the sums beyond the first, the RET
    "sum": (lambda B: B.add(B.add(B.mul(B.sq(B.x), 3.6e4), B.mul(B.sq(B.y), 3.6e4)), B.mul(B.sq(B.z), 3.6e4)), 3),
    # inside: nothing is kept
    "root": (lambda B: B.sub(B.sqrt(B.sub(B.add(B.sq(B.x), B.sq(B.z)), 0.01)), 0.1), 0),
    "mixed": (lambda B: B.max(B.min(B.abs(B.mul(B.x, -100.0)), B.mul(B.y, B.z)), B.sub(3.0, B.x)), 0),
    "asymmetric": (lambda B: B.sq(B.sub(B.sq(B.add(B.x, 4.0)), 60.0)), 0),   # ([0, 81] - 60)^2 <= 3600
}


@pytest.mark.parametrize("name", sorted(FIELDS))
def test_records_that_may_clamp_keep_fix(name):
    field, kept = FIELDS[name]
    info = T.precompile(tape(field), prune=False)
    assert info["specialized"] and info["fix_kept"] == kept


# surfaces where the clamped value crosses 0 and the unclamped one does not, or the other way round
CLAMPED = {
    "product": lambda B: B.sub(B.min(B.mul(B.mul(B.x, 1000.0), B.mul(B.y, 1000.0)), B.mul(B.z, 1e3)), 1.5e3),
    "product-beyond": lambda B: B.add(B.sub(B.mul(B.mul(B.x, 1000.0), B.mul(B.y, 1000.0)), 1.5e6), B.mul(B.z, 4e5)),
    "square": lambda B: B.sub(B.sq(B.add(B.mul(B.x, 300.0), 1000.0)), B.add(B.mul(B.y, 2e5), 9e5)),
    "quotient": lambda B: B.add(B.div(B.x, -1e-6), B.mul(B.y, 3e5)),
}


@pytest.mark.gpu
@pytest.mark.parametrize("prune", [False, True])
@pytest.mark.parametrize("name", sorted(CLAMPED))
def test_tapes_that_clamp_match_the_oracle(name, prune):
    t = oracle.parse_ll(tape(CLAMPED[name]))
    for k, g, o, gs, os_, _, _ in run_pair(t, [0.0, 1 / 60, 0.2], localsubdiv=5, prune=prune):
        print(f"{name} prune={prune} frame {k}: {len(o)} nodes", flush=True)
        assert_same_nodes(g, o, f"{name} frame {k}")
    assert len(o) > 1
