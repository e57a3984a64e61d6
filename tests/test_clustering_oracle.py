"""The clustering restatement in the oracle and the host tree functions,
checked against the reference's own clustering tests
(bioshell-clustering/tests/test_hierarchical.rs) and against results the
mathematics fixes (single-link heights are the minimum spanning tree's edges;
single and complete linkage heights agree with scipy, and average linkage
does where the reference's bookkeeping leaves the sizes correct)."""
import os

import numpy as np
import pytest

from bioshell_amd import clustering as C
from oracle import oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))


def packed(n, d):
    """Packed triangle from d(i, j), called with i > j like the reference."""
    return np.array([d(j, i) for i in range(n) for j in range(i + 1, n)], dtype=np.float32)


def oracle_tree(n, d, linkage="single"):
    up = packed(n, d)
    mi, mj, md = O.hclust(up, n, linkage)
    return C.tree_from_merges(n, mi, mj, md), up


def test_reference_cluster_numbers():
    """test_hierarchical.rs:9-24"""
    data = np.array([6.0, 2.0, 2.5, 5.9], dtype=np.float32)
    d = lambda a, b: float(np.abs(data[a] - data[b]))  # f32 arithmetic, as in the test
    root, _ = oracle_tree(4, d)
    assert root.cluster_size == 4
    assert [float(v) for v in C.retrieve_data(root, data)] == [6.0, np.float32(5.9), 2.0, 2.5]
    C.balance_clustering_tree(root, d)
    assert [float(v) for v in C.retrieve_data(root, data)] == [6.0, np.float32(5.9), 2.5, 2.0]


def test_reference_cluster_letters():
    """test_hierarchical.rs:26-43"""
    data = ['A', 'Z', 'D', 'Y', 'C', 'X', 'B', 'W', 'F', 'V']
    d = lambda a, b: float(abs(ord(data[a]) - ord(data[b])))
    root, _ = oracle_tree(len(data), d)
    assert root.cluster_size == len(data)
    assert C.retrieve_data(root, data) == ['A', 'B', 'D', 'C', 'F', 'Z', 'Y', 'X', 'W', 'V']
    C.balance_clustering_tree(root, d)
    assert C.retrieve_data(root, data) == ['A', 'B', 'C', 'D', 'F', 'V', 'W', 'X', 'Y', 'Z']


def read_tsv(path):
    """label_i <tab> label_j <tab> value lines, symmetric; labels numbered in
    order of first appearance."""
    ids, vals = {}, {}
    for line in open(path):
        a, b, v = line.split()
        for x in (a, b):
            ids.setdefault(x, len(ids))
        vals[(ids[a], ids[b])] = vals[(ids[b], ids[a])] = float(v)
    n = len(ids)
    return n, (lambda i, j: 0.0 if i == j else float(np.float32(vals.get((i, j), 100.0)))), list(ids)


def test_reference_d5_clusters():
    """test_hierarchical.rs:45-69 on the reference's d5.tsv fixture"""
    n, d, _ = read_tsv(os.path.join(HERE, "golden", "d5.tsv"))
    root, _ = oracle_tree(n, d)
    clusters = sorted(C.retrieve_clusters(root, 0.11), key=lambda c: c.cluster_size)
    assert len(clusters) == 4
    assert sum(c.cluster_size for c in clusters) == 5
    assert clusters[3].cluster_size == 2
    for c in clusters[:3]:
        assert C.medoid_by_min_max(c, d) == C.retrieve_data_id(c)[0]


def mst_weights(D):
    n = len(D)
    inside = [0]
    best = D[0].copy()
    out = []
    used = np.zeros(n, bool)
    used[0] = True
    for _ in range(n - 1):
        cand = np.where(used, np.inf, best)
        k = int(np.argmin(cand))
        out.append(cand[k])
        used[k] = True
        best = np.minimum(best, D[k])
    return np.sort(np.array(out, dtype=np.float32))


@pytest.mark.parametrize("seed", range(4))
def test_single_link_heights_are_the_mst(seed):
    rng = np.random.default_rng(seed)
    n = 40
    D = rng.uniform(0.5, 9.0, size=(n, n)).astype(np.float32)
    D = np.minimum(D, D.T)
    np.fill_diagonal(D, 0)
    root, up = oracle_tree(n, lambda a, b: float(D[a, b]))
    _, _, md = O.hclust(up, n, "single")
    assert np.array_equal(np.sort(md), mst_weights(D))


@pytest.mark.parametrize("linkage", ["single", "complete"])
def test_heights_agree_with_scipy(linkage):
    """Size-independent rules: the merge heights are scipy's."""
    from scipy.cluster.hierarchy import linkage as sp_linkage

    rng = np.random.default_rng(7)
    n = 60
    pts = rng.normal(size=(n, 3)) * 3
    D = np.sqrt(((pts[:, None] - pts[None]) ** 2).sum(-1)).astype(np.float32)
    up = np.array([D[i, j] for i in range(n) for j in range(i + 1, n)], dtype=np.float32)
    _, _, md = O.hclust(up, n, linkage)
    Z = sp_linkage(up.astype(np.float64), method=linkage)
    assert np.allclose(np.sort(md), np.sort(Z[:, 2]), rtol=1e-6, atol=1e-6)


def test_average_link_is_upgma_when_nothing_moves():
    """Points on a line whose gaps halve from left to right: the cluster
    growing at the right end is always closer to its neighbour than the next
    gap, so every merge takes the last active index, no cluster is moved (the
    reference never moves sizes[]) and average linkage must be exactly UPGMA."""
    from scipy.cluster.hierarchy import linkage as sp_linkage

    n = 20
    x = np.cumsum(np.r_[0.0, 2.0 ** np.arange(n - 2, -1, -1)]).astype(np.float32)
    D = np.abs(x[:, None] - x[None]).astype(np.float32)
    up = np.array([D[i, j] for i in range(n) for j in range(i + 1, n)], dtype=np.float32)
    mi, mj, md = O.hclust(up, n, "average")
    order = n - np.arange(n - 1)
    assert np.array_equal(mj, order - 1)  # every merge takes the last index
    Z = sp_linkage(up.astype(np.float64), method="average")
    assert np.allclose(np.sort(md), np.sort(Z[:, 2]), rtol=1e-5)


@pytest.mark.parametrize("linkage", ["centroid", "median"])
def test_centroid_and_median_rules_match_scipy_on_squared_distances(linkage):
    """Both Lance-Williams rules are exact on squared Euclidean distances: the
    merge heights are the squared distances between cluster centroids
    (centroid) or between the midpoints of merged pairs (median, WPGMC), which
    scipy computes from the points themselves.  On the halving-gap chain every
    merge takes the last active index, so the reference's size bookkeeping
    (sizes[] not moved) never comes into play."""
    from scipy.cluster.hierarchy import linkage as sp_linkage

    n = 18
    x = np.cumsum(np.r_[0.0, 2.0 ** np.arange(n - 2, -1, -1)])
    D2 = ((x[:, None] - x[None]) ** 2).astype(np.float32)
    up = np.array([D2[i, j] for i in range(n) for j in range(i + 1, n)], dtype=np.float32)
    mi, mj, md = O.hclust(up, n, linkage)
    assert np.array_equal(mj, n - 1 - np.arange(n - 1))  # every merge takes the last index
    Z = sp_linkage(x[:, None], method=linkage)
    assert np.allclose(np.sqrt(np.sort(md.astype(np.float64))), np.sort(Z[:, 2]), rtol=2e-6)


def test_wards_first_merge_is_textbook():
    """The reference's Ward rule takes sizes[j] for size_k; while every
    cluster is a singleton that equals the textbook Lance-Williams Ward
    update, so the first merged row must be scipy's Ward distances of the
    merged pair to each other point (squared Euclidean inputs)."""
    rng = np.random.default_rng(4)
    n = 12
    P = rng.normal(size=(n, 3))
    D2 = ((P[:, None] - P[None]) ** 2).sum(-1).astype(np.float32)
    up = np.array([D2[i, j] for i in range(n) for j in range(i + 1, n)], dtype=np.float32)
    mi, mj, md = O.hclust(up, n, "wards")
    i, j = int(mi[0]), int(mj[0])
    assert md[0] == D2[np.triu_indices(n, 1)].min()
    # the textbook update for singletons: d(k, i+j) = (2 d_ik + 2 d_jk - d_ij) / 3
    want = {k: (2 * D2[i, k] + 2 * D2[j, k] - D2[i, j]) / 3 for k in range(n) if k not in (i, j)}
    # the second merge is the smallest of the updated and untouched distances
    rest = [D2[a, b] for a in range(n) for b in range(a + 1, n) if a not in (i, j) and b not in (i, j)]
    assert md[1] == pytest.approx(min(min(want.values()), min(rest)), rel=1e-6)


def test_oracle_keeps_reference_quirks():
    """clust --median/--centroid map to average/wards (clust.rs:66-80)."""
    assert C.linkage_of_cli(median=True) == "average"
    assert C.linkage_of_cli(centroid=True) == "wards"
    assert C.linkage_of_cli() == "single"


# Hand-traced agglomeration of six elements in which a merged cluster is moved
# and then merged again, so that the sizes the reference keeps in place
# (clustering_matrix.rs:47-53: rows swapped, columns copied, sizes untouched)
# and the sizes[j] it passes as the rule's third argument
# (clustering_matrix.rs:66) decide the later heights.
F = np.float32


def _average(si, sj, sk, dij, dik, djk):  # strategies/mod.rs average_link, f32
    d = F(1.0) / F(si + sj)
    return F(F(d * F(si)) * dik) + F(F(d * F(sj)) * djk)


def _centroid(si, sj, sk, dij, dik, djk):  # strategies/mod.rs centroid_link, f32
    d = F(1.0) / F(si + sj)
    return (F(F(d * F(si)) * dik) + F(F(d * F(sj)) * djk)) - F(F(F(F(si) * F(sj)) * d) * d) * dij


def _wards(si, sj, sk, dij, dik, djk):  # strategies/mod.rs wards_method, f32
    d = F(1.0) / F(si + sj + sk)
    return (F(F(d * F(si + sk)) * dik) + F(F(d * F(sj + sk)) * djk)) - F(F(sk) * d) * dij


def _six():
    """d(4,5) = 1 merges first (no move: 5 is last); d(0,1) = 2 next, after which
    the pair {4,5} at index 4 moves to index 1 while sizes[1] stays 1."""
    D = np.zeros((6, 6), np.float32)
    for (a, b), v in {(0, 1): 2, (4, 5): 1, (2, 4): 3, (2, 5): 3, (0, 2): 10, (1, 2): 10,
                      (0, 3): 30, (1, 3): 30, (0, 4): 8, (0, 5): 12, (1, 4): 8, (1, 5): 12,
                      (2, 3): 16, (3, 4): 20, (3, 5): 24}.items():
        D[a, b] = D[b, a] = v
    return D


def _hand_trace(rule):
    """Expected (i, j, height) of the five merges, step by step."""
    D = _six()
    P = {k: rule(1, 1, 1, D[4, 5], D[4, k], D[5, k]) for k in (0, 1, 2, 3)}  # step 1: {4,5} at 4
    # step 2: (0, 1) at 2; row 0 becomes A = {0,1}; sizes[1] = 1 is the third argument
    A = {2: rule(1, 1, 1, D[0, 1], D[0, 2], D[1, 2]), 3: rule(1, 1, 1, D[0, 1], D[0, 3], D[1, 3]),
         "P": rule(1, 1, 1, D[0, 1], P[0], P[1])}
    # {4,5} moves to index 1; sizes stay [2, 1, 1, 1 | 2]: index 1 still says 1
    # step 3: (1, 2) = ({4,5}, {2}) with size_i = 1 (not 2), size_j = 1, sizes[j] = 1
    dP2 = P[2]
    Q = {"A": rule(1, 1, 1, dP2, A["P"], A[2]), 3: rule(1, 1, 1, dP2, P[3], D[2, 3])}
    # {3} (index 3, the last) moves to index 2; sizes[1] = 1 + 1 = 2 (the cluster holds 3)
    # step 4: (0, 1) = (A, Q), size_i = 2, size_j = 2, sizes[j] = 2
    dAQ = Q["A"]
    AQ3 = rule(2, 2, 2, dAQ, A[3], Q[3])
    # {3} moves to index 1; step 5: (0, 1) at AQ3
    return [(4, 5, F(1)), (0, 1, F(2)), (1, 2, dP2), (0, 1, dAQ), (0, 1, AQ3)]


@pytest.mark.parametrize("linkage,rule", [("average", _average), ("centroid", _centroid), ("wards", _wards)])
def test_moved_cluster_heights_hand_traced(linkage, rule):
    D = _six()
    up = D[np.triu_indices(6, 1)]
    want = _hand_trace(rule)
    mi, mj, md = O.hclust(up, 6, linkage)
    got = list(zip(mi.tolist(), mj.tolist(), md.tolist()))
    assert [(i, j) for i, j, _ in got] == [(i, j) for i, j, _ in want]
    assert np.array_equal(md.view(np.uint32), np.array([h for _, _, h in want], np.float32).view(np.uint32)), \
        (got, want)
    # and the values are the ones worked out on paper for average linkage
    if linkage == "average":
        assert [float(h) for _, _, h in want] == [1.0, 2.0, 3.0, 10.0, 24.5]
    if linkage == "centroid":
        assert [float(h) for _, _, h in want] == [1.0, 2.0, 2.75, 8.6875, 21.671875]
    # planted mistakes: sizes moved with the row changes the last height for
    # every size-weighted rule; sizes[k] as the third argument changes Ward's
    moved = O.hclust(up, 6, linkage, planted_mistake=1)[2]
    assert not np.array_equal(moved, md)
    by_k = O.hclust(up, 6, linkage, planted_mistake=2)[2]
    assert np.array_equal(by_k, md) == (linkage != "wards")


def test_wards_moved_cluster_hand_computed():
    """Ward's rule on the same six elements, worked out on paper (exact
    fractions; f32 agrees to a few ulps): d(P,k) = (2(d4k + d5k) - 1)/3, so
    P = {0: 13, 1: 13, 2: 11/3, 3: 29}; A = {2: 38/3, 3: 118/3, P: 50/3};
    step 3 with the stale size 1: Q = {A: (2(50/3 + 38/3) - 11/3)/3 = 55/3,
    3: (2(29 + 16) - 11/3)/3 = 259/9}; step 4 with sizes 2, 2, 2:
    (4 * 118/3 + 4 * 259/9 - 2 * 55/3)/6 = 1061/27."""
    D = _six()
    md = O.hclust(D[np.triu_indices(6, 1)], 6, "wards")[2].astype(np.float64)
    assert md == pytest.approx([1.0, 2.0, 11 / 3, 55 / 3, 1061 / 27], rel=2e-7)
    # with the moved cluster's true size 2 at step 3, Q = {A: 215/12, 3: 173/6}
    # and step 4 (sizes 2, 3, 3) gives 5/8 * 118/3 + 6/8 * 173/6 - 3/8 * 215/12
    moved = O.hclust(D[np.triu_indices(6, 1)], 6, "wards", planted_mistake=1)[2].astype(np.float64)
    assert moved[4] == pytest.approx(5 / 8 * 118 / 3 + 6 / 8 * 173 / 6 - 3 / 8 * 215 / 12, rel=2e-7)
    assert abs(moved[4] - 1061 / 27) > 0.1


def test_row_stats_oracle():
    rng = np.random.default_rng(3)
    n = 37
    D = rng.uniform(0, 5, size=(n, n)).astype(np.float32)
    D = np.minimum(D, D.T)
    np.fill_diagonal(D, np.nan)
    up = np.array([D[i, j] for i in range(n) for j in range(i + 1, n)], dtype=np.float32)
    lo, hi = O.row_stats(up, n)
    assert np.array_equal(lo, np.nanmin(D, axis=1))
    assert np.array_equal(hi, np.nanmax(D, axis=1))


@pytest.mark.parametrize("mi,mj", [([0, -1], [1, 0]), ([0, 0], [1, -1]), ([0, 0], [-2, 1]), ([0, 0], [3, 1]),
                                   ([5, 0], [1, 1]), ([0, 0], [1, 2]), ([0, 0, 0], [2, 1, 0]), ([0, 0, 0], [2, 1, 1])])
def test_tree_refuses_indices_of_no_cluster(mi, mj):
    """Negative indices, indices past the active clusters and one merge too
    many: three elements, two merges at most."""
    with pytest.raises(KeyError):
        C.tree_from_merges(3, mi, mj, [1.0, 2.0, 3.0][:len(mi)])


def test_tree_from_other_number_types():
    """Any iterables of numbers: the tree is that of the integer arrays."""
    mi, mj, md = [0, 0, 0], [3, 1, 1], [1, 2, 3]
    want = C.tree_from_merges(4, np.array(mi, np.uint32), np.array(mj, np.uint32), np.array(md, np.float32))
    for make in (lambda v: [float(x) for x in v], lambda v: (x for x in v), lambda v: np.array(v, np.float64),
                 lambda v: tuple(np.int64(x) for x in v)):
        root = C.tree_from_merges(4, make(mi), make(mj), make(md))
        assert C.retrieve_data_id(root) == C.retrieve_data_id(want)
        assert type(root.merging_distance) is float and root.merging_distance == 3.0
