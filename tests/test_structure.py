"""Structure learning (pairwise mutual information, Chow-Liu tree): the oracle against library
routines and closed forms (CPU), the HIP path against the oracle (GPU)."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "oracle"))
sys.path.insert(0, os.path.join(ROOT, "lvd-pg_amd"))

import structure_oracle as S  # noqa: E402


def _data(N, V, C, seed, corr=0.7):
    """Columns copied from their predecessor with probability `corr`, else uniform."""
    rng = np.random.default_rng(seed)
    x = np.zeros((N, V), np.uint8)
    x[:, 0] = rng.integers(0, C, N)
    for v in range(1, V):
        src = rng.integers(0, v)
        keep = rng.random(N) < corr
        x[:, v] = np.where(keep, x[:, src], rng.integers(0, C, N))
    return x


# ---- the oracle, pinned ------------------------------------------------------------------

def test_oracle_mi_matches_sklearn_without_pseudocount():
    from sklearn.metrics import mutual_info_score
    x = _data(500, 5, 6, 0)
    mi = S.pairwise_mi(x, 6, pseudocount=0.0)
    for u in range(5):
        for v in range(5):
            assert abs(mi[u, v] - mutual_info_score(x[:, u], x[:, v])) < 1e-10


def test_oracle_mi_closed_forms():
    rng = np.random.default_rng(1)
    N, C = 4000, 4
    a = rng.integers(0, C, N)
    b = rng.integers(0, C, N)
    x = np.stack([a, a, b], axis=1).astype(np.uint8)
    mi = S.pairwise_mi(x, C, pseudocount=0.0)
    p = np.bincount(a, minlength=C) / N
    H = -(p * np.log(p)).sum()
    assert abs(mi[0, 1] - H) < 1e-12 and abs(mi[0, 0] - H) < 1e-12      # MI(x, x) = H(x)
    assert 0 <= mi[0, 2] < 5e-3                                           # independent columns
    assert np.allclose(mi, mi.T)
    # the pseudocount enters as information.jl:52-58 says: every cell pc/C^2, every category pc/C, Z = N + pc
    pair, single = S.marginals(x.astype(np.int64), C, 0.5)
    assert abs(pair[0, 2].sum() - 1) < 1e-12 and abs(single[1].sum() - 1) < 1e-12
    assert abs(pair[0, 1][0, 1] - 0.5 / 16 / (N + 0.5)) < 1e-15           # an empty cell


def test_oracle_tree_is_a_maximum_spanning_tree_rooted_at_the_centre():
    from scipy.sparse.csgraph import minimum_spanning_tree
    x = _data(800, 12, 5, 2)
    mi = S.pairwise_mi(x, 5)
    parent = S.chow_liu_tree(mi)
    assert (parent < 0).sum() == 1
    w = mi.max() + 1.0 - mi
    np.fill_diagonal(w, 0)
    ref = minimum_spanning_tree(w).toarray()
    ref_weight = sum(mi[i, j] for i, j in zip(*np.nonzero(ref)))
    assert abs(S.tree_weight(mi, parent) - ref_weight) < 1e-9
    # path graph 0-1-2-3-4: the centre is 2; with six vertices the centres are 2 and 3 -> 2
    for V, root in ((5, 2), (6, 2)):
        m = np.zeros((V, V))
        for i in range(V - 1):
            m[i, i + 1] = m[i + 1, i] = 1.0
        p = S.chow_liu_tree(m)
        assert int(np.where(p < 0)[0][0]) == root


# ---- the C ABI on the host ----------------------------------------------------------------

def test_chow_liu_tree_host_entry_matches_oracle():
    import pcmi355 as P
    x = _data(600, 20, 4, 3)
    mi = S.pairwise_mi(x, 4).astype(np.float32)
    got = P.chow_liu_tree(mi)
    want = S.chow_liu_tree(mi.astype(np.float64))
    assert abs(S.tree_weight(mi, got) - S.tree_weight(mi, want)) < 1e-5
    assert np.array_equal(got, want)        # same tie rule, same centre
    with pytest.raises(P.PcmError):
        P.chow_liu_tree(np.full((3, 3), np.nan, np.float32))


@pytest.mark.parametrize("V", [2, 7, 10, 19])
def test_chow_liu_tree_and_single_nans(V):
    """A NaN among the first vertex's links is refused wherever it stands, as is a vertex without a link; any other NaN is
    a link that is not there."""
    import pcmi355 as P
    rng = np.random.default_rng(V)
    mi = rng.random((V, V)).astype(np.float32)
    mi = mi + mi.T
    for v in range(1, V):
        bad = mi.copy()
        bad[0, v] = np.nan
        with pytest.raises(P.PcmError):
            P.chow_liu_tree(bad)
        bad[0, v], bad[:, v] = 1.0, -np.inf
        bad[v] = -np.inf
        with pytest.raises(P.PcmError):
            P.chow_liu_tree(bad)
    for u in range(1, V):
        for v in range(V):
            odd, none = mi.copy(), mi.copy()
            odd[u, v], none[u, v] = np.nan, -np.inf
            assert np.array_equal(P.chow_liu_tree(odd), P.chow_liu_tree(none))


def test_tree_from_its_edges():
    """`pcm_chow_liu_root`: the edges of a tree in any order and direction give the parent array that the matrix gave;
    what is no tree is refused."""
    import ctypes
    import pcmi355 as P
    from pcmi355._lib import lib, np_ptr
    rng = np.random.default_rng(3)
    for V in (1, 2, 3, 17, 200):
        a = rng.normal(size=(V, V)).astype(np.float32)
        want = P.chow_liu_tree(a + a.T)
        kids = rng.permutation(np.flatnonzero(want >= 0))
        edges = np.stack([kids, want[kids]], 1).astype(np.int32)
        flip = rng.random(len(edges)) < 0.5
        edges[flip] = edges[flip][:, ::-1]
        edges, got = np.ascontiguousarray(edges.reshape(-1)), np.empty(V, np.int32)
        padded = np.concatenate([edges, np.zeros(2, np.int32)])
        assert lib.pcm_chow_liu_root(np_ptr(padded), V, np_ptr(got)) == 0
        assert np.array_equal(got, want)
    for bad in ([0, 1, 1, 2, 2, 0], [0, 1, 0, 1, 2, 3], [0, 4, 1, 2, 2, 3], [0, -1, 1, 2, 2, 3], [0, 0, 1, 2, 2, 3]):
        assert lib.pcm_chow_liu_root(np_ptr(np.array(bad, np.int32)), 4, np_ptr(np.empty(4, np.int32))) == -1
    assert lib.pcm_chow_liu_edges_workspace(1) == 0 and lib.pcm_chow_liu_edges_workspace(8193) == 0
    assert lib.pcm_chow_liu_edges_workspace(8192) > 0


# ---- the HIP path -------------------------------------------------------------------------

@pytest.fixture(scope="module")
def gpu():
    import torch
    assert torch.cuda.is_available(), "these tests need the GPU box"
    import pcmi355
    return torch, pcmi355


@pytest.mark.gpu
@pytest.mark.parametrize("N,V,C,pc", [(300, 7, 5, 0.1), (1000, 9, 16, 0.0), (4097, 6, 256, 0.1), (64, 3, 2, 1.0),
                                      (5000, 4, 200, 0.1), (65535, 3, 256, 0.1), (65536, 3, 256, 0.1), (70001, 4, 256, 0.1),
                                      (140000, 3, 7, 0.0), (66000, 3, 200, 0.1), (12000, 5, 64, 0.1), (30000, 3, 256, 0.1)])
def test_pairwise_mi_matches_oracle(gpu, N, V, C, pc):
    """Tolerance: 1e-4 of the largest entry (float32 output of float64 sums).  Beyond 65535 examples
    the cells are counted in 32 bits, band by band of the first variable's categories (two bands at
    256 categories, one at 200 and 7)."""
    torch, P = gpu
    x = _data(N, V, C, N + V)
    want = S.pairwise_mi(x, C, pc)
    got = P.pairwise_MI(torch.from_numpy(x).cuda(), C, pc).cpu().numpy()
    assert np.abs(got - want).max() < 1e-4 * np.abs(want).max()
    assert np.array_equal(got, got.T)
    xt = torch.from_numpy(np.ascontiguousarray(x.T)).cuda().t()          # column-major, as Julia holds it
    assert np.array_equal(P.pairwise_MI(xt, C, pc).cpu().numpy(), got)


@pytest.mark.gpu
@pytest.mark.parametrize("N,V,C", [(1, 2, 256), (3, 3, 255), (1500, 4, 100), (2049, 4, 100), (40000, 3, 64), (20000, 3, 2),
                                   (12384, 3, 256), (12385, 3, 256), (32769, 3, 129), (16387, 4, 33)])
def test_pairwise_mi_at_the_edges_of_its_launch_rules(gpu, N, V, C):
    """Both ways of clearing the table on either side of their line, both workgroup sizes, rounds beyond the words a
    thread keeps, counts past the part of the term table that the LDS holds (two categories), odd category counts, and
    a constant column beside the others.  Same tolerance as above."""
    torch, P = gpu
    x = _data(N, V, C, N + V + C)
    x[:, 0] = C - 1
    want = S.pairwise_mi(x, C, 0.1)
    got = P.pairwise_MI(torch.from_numpy(x).cuda(), C, 0.1).cpu().numpy()
    assert np.abs(got - want).max() < 1e-4 * np.abs(want).max()
    assert np.array_equal(got, got.T)


@pytest.mark.gpu
@pytest.mark.parametrize("N,V,C", [(1, 510, 256), (17, 521, 255), (300, 1100, 129), (2000, 1030, 130), (2500, 700, 256),
                                   (2500, 700, 200), (4096, 640, 256), (4097, 1000, 128), (14000, 1152, 64), (15000, 1100, 33),
                                   (16000, 1024, 256), (3000, 900, 1), (3000, 900, 100)])
def test_pairwise_mi_with_a_pair_per_two_lanes(gpu, N, V, C):
    """Enough variables for the kernel that sorts a variable's examples by category, against the one with a pair per
    workgroup (`pcm_pairwise_mi_static`, the kernel of the oracle tests): both add the same integers, so the results are the same
    bits.  Columns whose categories hold 8, 9, 16, 17, 255, 256 and 257 examples (ends of chunks, the last 8-bit count), one
    that is constant, one with nine tenths of its examples in one category (counts past the terms in LDS); variables past a
    whole block of 32; a category of a thousand and more examples whose counts pass 255 and one whose do not; categories shared out among several waves and not."""
    torch, P = gpu
    from pcmi355._lib import lib, check
    rng = np.random.default_rng(N + V + C)
    base = rng.normal(size=(N, 1)) * 0.6 + rng.normal(size=(N, V))
    x = np.clip((base / 6 + 0.5) * C, 0, C - 1).astype(np.uint8)
    edges = np.repeat(np.arange(7), [8, 9, 16, 17, 255, 256, 257])[:N] % C
    for v in (0, 64, V - 1):
        x[:, v] = C - 1
        x[:len(edges), v] = edges
        x[:, v] = x[rng.permutation(N), v]
    x[:, 5] = C // 2
    x[rng.random(N) < 0.9, 9] = 0
    x[:, 10] = np.arange(N) % 3 % C          # counts past 255 (2500 examples) between this column and the next, not with noise
    x[:, 11] = x[:, 10]
    x[rng.random(N) < 0.9, 70] = C - 1
    d = torch.from_numpy(x).cuda()
    got = P.pairwise_MI(d, C, 0.1)
    want = torch.full((V, V), float("nan"), device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    check(lib.pcm_pairwise_mi_static(d.data_ptr(), d.stride(0), d.stride(1), N, V, C, 0.1, want.data_ptr(), stream))
    assert torch.equal(got, want)
    wide = torch.zeros((N, V + 3), dtype=torch.uint8, device="cuda")
    wide[:, 1:V + 1] = d
    assert torch.equal(P.pairwise_MI(wide[:, 1:V + 1], C, 0.1), got)
    assert torch.equal(P.pairwise_MI(d.t().contiguous().t(), C, 0.1), got)


def _mi_plan(N, V, C):
    """[lanes of a pair, shares of a variable's categories, bytes of scratch] of `pairwise_MI`"""
    from pcmi355._lib import lib, check, np_ptr
    plan = np.zeros(3, np.int64)
    check(lib.pcm_pairwise_mi_plan(N, V, C, np_ptr(plan)))
    return plan.tolist()


@pytest.mark.gpu
def test_which_pairs_go_to_lanes(gpu):
    """The sizes of the tests above and below reach the kernel they name, at one share and at several, and a call's scratch is
    what its kernels use: staged data, marginals, terms; codes, lists, starts and, with several shares, the pairs' sums."""
    up = lambda n: (n + 255) // 256 * 256
    lanes = [(1, 510, 256), (17, 521, 255), (300, 1100, 129), (2000, 1030, 130), (2500, 700, 256), (2500, 700, 200), (4096, 640, 256),
             (4097, 1000, 128), (14000, 1152, 64), (15000, 1100, 33), (16000, 1024, 256), (3000, 900, 1), (3000, 900, 100),
             (4000, 545, 200), (3500, 813, 256), (65535, 801, 64), (65535, 801, 256)]
    shares = set()
    for N, V, C in lanes + [(1000, 100, 256), (16384, 400, 256), (65536, 3072, 256), (4097, 640, 256)]:
        two, parts, size = _mi_plan(N, V, C)
        Np, blocks = (N + 63) // 64 * 64, (V + 31) // 32
        want = up(V * Np) + up(16 * V) + up(8 * (N + 1))
        if two:
            stride = (N + 31 * min(N, C) + 64 + 63) // 64 * 64
            want += up(blocks * N * 128) + up(4 * V * stride) + up(4 * V * (parts + 1)) + (up(8 * V * 32 * blocks) if parts > 1 else 0)
            shares.add(parts > 1)
        assert (two == 2) == ((N, V, C) in lanes) and (two or parts == 1) and size == want, (N, V, C, two, parts, size, want)
    assert shares == {False, True}


@pytest.mark.gpu
@pytest.mark.parametrize("N,V,C", [(4000, 545, 200), (3500, 813, 256), (65535, 801, 64), (65535, 801, 256)])
def test_counts_past_their_bits_in_lanes(gpu, N, V, C):
    """Few categories of many examples, so that only lanes without a pair count past 255 (the last block's, past the last
    variable); and as many examples as 16-bit counts hold, with columns of one category (a count of 65535) beside others."""
    torch, P = gpu
    from pcmi355._lib import lib, check
    rng = np.random.default_rng(N + V + C)
    x = rng.integers(0, 10, size=(N, V)).astype(np.uint8) * np.uint8(C // 10)
    if N == 65535:
        for v in (0, 31, 32, 500, V - 1):
            x[:, v] = C - 1 - v % 2
        x[:, 7] = x[:, 501] = np.arange(N) < 33000     # counts past 32767
    assert _mi_plan(N, V, C)[0] == 2
    d = torch.from_numpy(x).cuda()
    got = P.pairwise_MI(d, C, 0.1)
    part = 240 if N == 65535 else V      # (the other kernel's memory of its own holds 16 MB of data)
    for v0 in sorted({0, V - part} | ({480} if N == 65535 else set())):
        want = torch.empty((part, part), device="cuda")
        cols = d[:, v0:v0 + part]
        check(lib.pcm_pairwise_mi_static(cols.data_ptr(), cols.stride(0), cols.stride(1), N, part, C, 0.1, want.data_ptr(),
                                         torch.cuda.current_stream().cuda_stream))
        assert torch.equal(got[v0:v0 + part, v0:v0 + part], want)
    assert torch.equal(got, got.t())


@pytest.mark.gpu
def test_lanes_without_a_pair_cost_nothing(gpu):
    """784 variables are 24 blocks of 32 and a half: the lanes past the last variable count every example of a category in one
    place, more than 255 of them here, but no pair does, so the half block takes no second pass.  4 % more pairs than with 768
    variables; 1.6 times as long where those lanes were heeded, so 1.3 lies half way and far from either."""
    import time
    torch, P = gpu
    g = torch.Generator(device="cuda").manual_seed(5)
    d = torch.randint(0, 10, (4000, 784), device="cuda", generator=g, dtype=torch.uint8) * 25
    assert _mi_plan(4000, 768, 256)[:2] == _mi_plan(4000, 784, 256)[:2] and _mi_plan(4000, 784, 256)[0] == 2
    least = {}
    for V in 3 * (768, 784):
        x = d[:, :V].contiguous()
        for _ in range(8):
            torch.cuda.synchronize()
            t = time.perf_counter()
            P.pairwise_MI(x, 256, 0.1)
            torch.cuda.synchronize()
            least[V] = min(least.get(V, 1.0), time.perf_counter() - t)
    assert least[784] < 1.3 * least[768]


@pytest.mark.gpu
def test_learned_tree_and_hclt(gpu):
    torch, P = gpu
    x = _data(2000, 30, 8, 11)
    d = torch.from_numpy(x).cuda()
    mi = P.pairwise_MI(d, 8, 0.1).cpu().numpy()
    parent = P.learn_chow_liu_tree(d, 8, 0.1)
    want = S.chow_liu_tree(S.pairwise_mi(x, 8, 0.1))
    assert abs(S.tree_weight(mi, parent) - S.tree_weight(mi, want)) < 1e-3
    bpc = P.hclt(d, 16, num_cats=8)
    assert bpc.size("variables") == 30
    lls = P.mini_batch_em_with_reg(bpc, d, 3, batch_size=500, pseudocount=0.1, param_inertia=0.9, shuffle="none")
    assert lls[-1] > lls[0]


@pytest.mark.gpu
def test_hclt_over_variable_groups_and_for_colored_images(gpu):
    """`hclt(data, K, variable_groups)` and `hclt_for_colored_images` (src/structures/hclts.jl:7-98): the tree is
    learned on the groups' first variables, a tree node's leaf is the product of one categorical per variable of
    its group; the circuit is the one `hclt_pc` builds from that tree, it covers exactly the grouped variables,
    and it trains."""
    torch, P = gpu
    from pcmi355 import nodes as N
    nc, h, w, K, C, n = 3, 4, 4, 4, 6, 600
    x = _data(n, nc * h * w, C, 23)
    d = torch.from_numpy(x).cuda()
    for mode, offset in (("red_only", 0), ("green_only", h * w), ("blue_only", 2 * h * w), ("cat_channels", None)):
        pc, leaves = P.hclt_for_colored_images(d, nc, h, w, K, num_cats=C, mode=mode, patch_size=2)
        groups = (P.group_vars_by_cgrid(h, w, nc, 2, 2, 0) if offset is None else P.group_vars_by_grid(h, w, 1, 2, 2, offset))
        assert len(leaves) == len(groups) == 4 and all(len(l) == K for l in leaves)
        want_vars = sorted(v for g in groups for v in g[1])
        assert N.variables(pc) == want_vars and len(want_vars) == (4 * nc if offset is None else 4) * 4
        firsts = [g[0] for g in groups]
        clt = P.learn_chow_liu_tree(d[:, firsts].contiguous(), C, 0.1)
        same, _ = N.describe(P.hclt_pc(clt, C, K, groups))
        got, _ = N.describe(pc)
        for k in same:
            np.testing.assert_array_equal(got[k], same[k], err_msg=f"{mode} {k}")
        for i, g in enumerate(groups):                          # a leaf circuit: sum over the product of its group's inputs
            prod = leaves[i][0].inputs[0]
            assert [c.var for c in prod.inputs] == list(g[1])
    with pytest.raises(ValueError):
        P.hclt_for_colored_images(d, nc, h, w, K, num_cats=C, mode="grey")
    N.init_parameters(pc, perturbation=0.4, rng=np.random.default_rng(1))
    bpc = P.CuBitsProbCircuit(pc, nc * h * w)
    lls = P.mini_batch_em_with_reg(bpc, d, 3, batch_size=200, pseudocount=0.1, param_inertia=0.9, shuffle="none")
    assert lls[-1] > lls[0]


@pytest.mark.gpu
@pytest.mark.parametrize("V", [2, 3, 63, 64, 65, 500, 1030])
def test_tree_found_on_the_device(gpu, V):
    """Where the maximum spanning tree is unique the device's edges give the host's tree, bit for bit; two largest edges of a
    component, asymmetry, NaN and infinities are left to the host, which answers as before."""
    torch, P = gpu
    from pcmi355 import structures
    from pcmi355._lib import lib, check, np_ptr
    rng = np.random.default_rng(V)
    for scale in (1e-6, 1.0, -3.0):
        a = rng.normal(size=(V, V)).astype(np.float32)
        a = np.maximum(a, a.T) * np.float32(scale)
        edges = structures._unique_tree_edges(torch.from_numpy(a).cuda())
        parent = np.empty(V, np.int32)
        check(lib.pcm_chow_liu_root(np_ptr(edges), V, np_ptr(parent)))
        assert np.array_equal(parent, P.chow_liu_tree(a))
        assert np.array_equal(P.chow_liu_tree(torch.from_numpy(a).cuda().double()), parent)
    if V < 63:
        return
    for kind in ("ties", "twin", "zeros", "asymmetric", "nan", "inf", "-inf"):
        b = a.copy()
        if kind == "ties":
            b = np.round(b)
        elif kind == "twin":                      # two columns of the data alike
            b[2], b[:, 2] = b[4], b[:, 4]
        elif kind == "zeros":                     # the two zeros are one weight
            b[...] = np.where(rng.random(V) < 0.5, np.float32(0.0), np.float32(-0.0))
        elif kind == "asymmetric":
            b[5, 7] += 1.0
        else:
            b[5, 7] = b[7, 5] = float(kind)
        m = torch.from_numpy(b).cuda()
        assert structures._unique_tree_edges(m) is None or kind in ("ties", "twin")   # (ties that no component meets)
        assert np.array_equal(P.chow_liu_tree(m), P.chow_liu_tree(b))
    none = np.full((V, V), -np.inf, np.float32)
    with pytest.raises(P.PcmError):
        P.chow_liu_tree(torch.from_numpy(none).cuda())


@pytest.mark.gpu
def test_pairwise_mi_full_size_properties(gpu):
    """4096 examples x 512 variables x 256 categories: symmetry, MI(x, x) = smoothed entropy
    identity against the oracle on a few pairs, duplicated column gives the same row."""
    torch, P = gpu
    from pcmi355 import workloads
    data = workloads.grf_images(4096, 16, 16, 2, 3.0, 0.8, seed=77)        # [4096, 512]
    data[:, 100] = data[:, 7]
    d = torch.from_numpy(data).cuda()
    mi = P.pairwise_MI(d, 256, 0.1).cpu().numpy()
    assert np.array_equal(mi, mi.T)
    assert np.allclose(mi[100], mi[7], rtol=0, atol=1e-6)
    sub = [0, 7, 100, 511]
    want = S.pairwise_mi(data[:, sub], 256, 0.1)
    assert np.abs(mi[np.ix_(sub, sub)] - want).max() < 1e-4 * np.abs(want).max()
