"""The operation counts of bench.py's roofline: the transforms' counts against
arithmetic that counts itself, and the column kernel's total against what its
measured vector instructions can have carried out."""
import pytest

import bench

SHAPES = [(3, 4), (4, 5), (4, 6), (5, 7), (6, 8), (7, 9)]


class Counted:
    ops = 0

    def _op(self, other):
        Counted.ops += 1
        return Counted()

    __add__ = __sub__ = __mul__ = _op


def count(f):
    Counted.ops = 0
    f()
    return Counted.ops


def dot(n):
    v = Counted() * Counted()
    for _ in range(n - 1):
        v = v + Counted() * Counted()
    return v


@pytest.mark.parametrize("K,M", SHAPES)
def test_even_odd_transforms(K, M):
    def to_points():
        for p in range((M + 1) // 2):
            even = dot((K + 1) // 2)
            if p < M // 2:
                odd = dot(K // 2)
                even + odd
                even - odd

    def to_modes():
        x = [Counted() for _ in range(M)]
        for p in range(M // 2):
            x[p] + x[M - 1 - p]
            x[p] - x[M - 1 - p]
        for q in range(K):
            dot((M + 1) // 2 if q % 2 == 0 else M // 2)

    assert bench.to_points_flops(K, M) == count(to_points)
    assert bench.to_modes_flops(K, M) == count(to_modes)


@pytest.mark.parametrize("M", [4, 5, 6, 7, 8, 9])
def test_line_derivative(M):
    def line():
        x = [Counted() for _ in range(M)]
        for b in range(M // 2):
            x[b] + x[M - 1 - b]
            x[b] - x[M - 1 - b]
        if M % 2:
            dot(M // 2)
        for _ in range(M // 2):
            u, v = dot(M // 2), dot(M // 2)
            if M % 2:
                u = u + Counted() * Counted()
            v + u
            v - u

    assert bench.line_derivative_flops(M) == count(line)


def test_column_kernel_within_its_instructions():
    """At (5, 7) with five iterations of the solve an element's wave carries out
    4,332 FP64 multiply-adds, 2,080 products and 1,295 sums on at most 64 lanes."""
    most = 64 * (2 * 4332 + 2080 + 1295)
    assert 0.5 * most < bench.column_kernel_flops(5, 7, 5.03) < most
    for K, M in SHAPES:
        assert bench.column_kernel_flops(K, M, 5.0) < bench.workgroup_kernel_flops(K, M, 5.0)
