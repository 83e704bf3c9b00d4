"""Graphs over [rows, columns] spaces with as many rows as columns, in which a value per row is also read per column: each returns the Vars
that are asked for and what numpy makes of them in float64."""
import numpy as np

import jittor_amd as jt


def _spread(v, shape, dims):
    return jt.broadcast(v, shape, dims)


def minus_sum(x, X, e, E):                         # x[i][j] - s[j]
    return [(x - x.sum([1]), X - X.sum(1))]


def over_root(x, X, e, E):                         # the ops in front of the broadcast are taken into it
    return [(x / x.sum([1]).sqrt(), X / np.sqrt(X.sum(1)))]


def adjacency(x, X, e, E):                         # A / d[:, None] / d[None, :]
    n = len(X)
    d, D = x.sum([1]), X.sum(1)
    return [(x / _spread(d, [n, n], [1]) / _spread(d, [n, n], [0]), X / D[:, None] / D[None, :])]


def adjacency_rooted(x, X, e, E):
    n = len(X)
    d, D = x.sum([1]).sqrt(), np.sqrt(X.sum(1))
    return [(x / _spread(d, [n, n], [1]) / _spread(d, [n, n], [0]), X / D[:, None] / D[None, :]), (d, D)]


def group_of_columns(x, X, e, E):                  # a group of [columns] that nothing here reads per row
    d, D = x - x.mean([1], keepdims=True), X - X.mean(1, keepdims=True)
    c, C = e * 2.0 + 1.0, E * 2.0 + 1.0
    return [(d / (d * d).mean([1], keepdims=True).sqrt() * c, D / np.sqrt((D * D).mean(1, keepdims=True)) * C), (c, C)]


def group_of_both(x, X, e, E):                     # a group behind the row sums, read per row and per column
    n = len(X)
    t, T = x.sum([1]) * e + e, X.sum(1) * E + E
    y, Y = x - _spread(t, [n, n], [1]), X - T[:, None]
    return [(y * y.sum([1], keepdims=True), Y * Y.sum(1, keepdims=True)), (x - t, X - T), (t, T)]


def per_row_only(x, X, e, E):
    p, P = (x - x.max([1], keepdims=True)).exp(), np.exp(X - X.max(1, keepdims=True))
    return [(p / p.sum([1], keepdims=True) * e, P / P.sum(1, keepdims=True) * E)]


def column_sums(x, X, e, E):                       # sums over the rows, read per column as they should be
    p, P = x / x.sum([1], keepdims=True), X / X.sum(1, keepdims=True)
    s, S = p.sum([0]), P.sum(0)
    return [(p - s, P - S), (s, S)]


GRAPHS = [minus_sum, over_root, adjacency, adjacency_rooted, group_of_columns, group_of_both, per_row_only, column_sums]


def several_axes(x, X):                            # [a, b, a, b]: rows and columns of two axes each
    return [(x - x.sum([2, 3]), X - X.sum((2, 3))), (x / x.sum([2, 3], keepdims=True), X / X.sum((2, 3), keepdims=True))]
