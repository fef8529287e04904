"""What a user of this package has it do, as cases that can be timed and compared: scoring, mini-batch EM on hidden
Chow-Liu trees (single, many heads, a forest of patches, soft evidence), the variational queries, sampling and structure
learning, from one small batch to the 3072-variable image circuit.

A case is a dict of plain values.  `prepare` makes what a program holds before the call (data, compiled circuit with
its parameters), `run` is one pass through the package's public entry points, `work` what that pass cannot do without,
`tolerance` what another correct implementation at the same precision may differ by."""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "lvd-pg_amd"))

import pcmi355 as P  # noqa: E402

TRAIN = 4096    # images a circuit's tree is learned from
INNER = 0.8     # share of a Chow-Liu tree's nodes that have children, on image data
KINDS = ("score", "em", "em", "heads", "forest", "soft", "kl", "relaxed", "sample", "structure")


# ---- cases ------------------------------------------------------------------------------------------------------

def listed():
    return [
        # a served request: one small batch scored by the 64-variable, K = 16 circuit of an 8 x 8 patch
        dict(name="score_patch", kind="score", h=8, w=8, ch=1, K=16, C=256, n=100, batch=100),
        # a held-out set of 32 x 32 x 3 images scored in batches of a thousand, the last one ragged
        dict(name="score_images", kind="score", h=32, w=32, ch=3, K=32, C=256, n=10300, batch=1000),
        # an epoch of EM on 28 x 28 grey digits at the batch size the trainers use
        dict(name="em_digits", kind="em", h=28, w=28, ch=1, K=32, C=256, n=8192, batch=512, weighted=False),
        # the headline circuit: 3072 variables, K = 32, batches of 4096, an epoch of 20 batches
        dict(name="em_images", kind="em", h=32, w=32, ch=3, K=32, C=256, n=81920, batch=4096, weighted=False),
        # ten EM steps on the wide K = 128 circuit of a 4 x 4 x 3 patch
        dict(name="em_wide", kind="em", h=4, w=4, ch=3, K=128, C=256, n=40960, batch=4096, weighted=False),
        # a patch circuit in the middle of progressive growing: 128 cluster heads over a body that lost two fifths of
        # its edges to pruning, so that no two sums of a layer have the same children
        dict(name="heads_pruned", kind="heads", h=8, w=8, ch=3, K=32, C=256, heads=128, keep=0.6, n=8192, batch=512),
        # sixteen 8 x 8 x 3 patch circuits of 32 x 32 x 3 images, 128 heads each, trained side by side
        dict(name="forest_patches", kind="forest", side=4, ph=8, pw=8, ch=3, K=32, C=256, heads=128, n=8192, batch=512),
        # the circuit over an image's patches, trained on per-cluster log-likelihoods instead of pixels
        dict(name="soft_top", kind="soft", V=64, K=64, C=128, n=8192, batch=1024),
        # KL between two matrices of parameter rows of the image circuit, and its gradient
        dict(name="kl_images", kind="kl", h=32, w=32, ch=3, K=32, C=256, rows=16),
        # a variational model's sampling step on a 16 x 16 x 3 circuit: relaxed samples, one parameter row per example,
        # and the gradient back to the rows
        dict(name="relaxed_rows", kind="relaxed", h=16, w=16, ch=3, K=16, C=256, rows=100, gumbel=True),
        # 4096 images drawn from the image circuit with supplied noise
        dict(name="sample_images", kind="sample", h=32, w=32, ch=3, K=32, C=256, n=4096),
        # the tree of the image circuit learned from 16384 training images
        dict(name="structure_images", kind="structure", h=32, w=32, ch=3, C=256, n=16384),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _image(rng, lo, hi):
    """height, width, channels with about lo..hi variables, any height and width among them"""
    ch = rng.choice((1, 3))
    v = _between(rng, lo, hi) / ch
    h = max(2, int(round(math.sqrt(v) * rng.uniform(0.8, 1.25))))
    return dict(h=h, w=max(2, int(v / h)), ch=ch)


def draw(rng):
    kind = rng.choice(KINDS)
    cats = rng.choice((256, 256, 256, 128, 100, 64))
    if kind == "score":
        K = rng.choice((16, 32, 32, 64, 128))
        img = _image(rng, 40, {16: 3072, 32: 3072, 64: 256, 128: 96}[K])
        n = _between(rng, 50, 10000)
        return dict(kind=kind, **img, K=K, C=cats, n=n, batch=min(n, _between(rng, 50, 4096)))
    if kind == "em":
        K = rng.choice((16, 32, 32, 64, 128))
        img = _image(rng, 40, {16: 3072, 32: 3072, 64: 256, 128: 96}[K])
        batch = _between(rng, 64, 4096)
        return dict(kind=kind, **img, K=K, C=cats, n=batch * rng.randint(4, 16), batch=batch, weighted=rng.random() < 0.2)
    if kind == "heads":
        batch = _between(rng, 64, 1024)
        return dict(kind=kind, **_image(rng, 40, 192), K=rng.choice((16, 32)), C=cats, heads=_between(rng, 8, 128),
                    keep=rng.choice((1.0, 0.8, 0.6, 0.4)), n=batch * rng.randint(4, 12), batch=batch)
    if kind == "forest":
        batch = _between(rng, 64, 1024)
        return dict(kind=kind, side=rng.randint(2, 4), ph=rng.randint(4, 8), pw=rng.randint(4, 8), ch=rng.choice((1, 3)),
                    K=rng.choice((16, 32)), C=cats, heads=_between(rng, 8, 128), n=batch * rng.randint(4, 12), batch=batch)
    if kind == "soft":
        batch = _between(rng, 64, 1024)
        return dict(kind=kind, V=_between(rng, 16, 64), K=rng.choice((16, 32, 64)), C=_between(rng, 20, 128),
                    n=batch * rng.randint(4, 8), batch=batch)
    if kind in ("kl", "relaxed"):
        K = rng.choice((16, 32))
        img = _image(rng, 40, 3072)
        most = max(1, int(16 * 3072 * 32 * 256 / (img["h"] * img["w"] * img["ch"] * K * cats)))
        case = dict(kind=kind, **img, K=K, C=cats, rows=min(_between(rng, 1, 256), most))
        return dict(case, gumbel=rng.random() < 0.7) if kind == "relaxed" else case
    if kind == "sample":
        return dict(kind=kind, **_image(rng, 40, 3072), K=rng.choice((16, 32)), C=cats, n=_between(rng, 16, 4096))
    return dict(kind=kind, **_image(rng, 100, 3072), C=cats, n=_between(rng, 1000, 16384))


# ---- inputs -----------------------------------------------------------------------------------------------------

def _variables(case):
    if case["kind"] == "forest":
        return case["side"] ** 2 * case["ph"] * case["pw"] * case["ch"]
    return case["V"] if "V" in case else case["h"] * case["w"] * case["ch"]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _images(n, h, w, ch, cats, gen, scale=3.0, corr=0.8):
    """[n, ch * h * w] uint8: smooth random fields whose channels are correlated, quantised to `cats` grey levels"""
    fy = torch.fft.fftfreq(h, device="cuda")[:, None]
    fx = torch.fft.rfftfreq(w, device="cuda")[None, :]
    filt = torch.exp(-2.0 * (math.pi * scale) ** 2 * (fx ** 2 + fy ** 2))
    filt = filt / torch.sqrt((filt ** 2).mean())
    out = torch.empty((n, ch, h, w), dtype=torch.uint8, device="cuda")
    for s in range(0, n, 8192):
        m = min(8192, n - s)
        f = torch.randn((m, ch + 1, h, w), device="cuda", generator=gen)
        f = torch.fft.irfft2(torch.fft.rfft2(f) * filt, s=(h, w))
        f = math.sqrt(corr) * f[:, :1] + math.sqrt(1.0 - corr) * f[:, 1:]
        out[s:s + m] = ((f / 9.0 + 0.5) * cats).floor_().clamp_(0, cats - 1).to(torch.uint8)
    return out.reshape(n, ch * h * w)


def _tree(data):
    """The Chow-Liu tree of the data's Gaussian mutual information, as a parent array"""
    x = data.double()
    x = x - x.mean(0)
    x = x / x.std(0).clamp_(min=1e-9)
    rho = (x.t() @ x / x.shape[0]).clamp_(-0.999999, 0.999999)
    return P.chow_liu_tree((-0.5 * torch.log1p(-rho ** 2)).float())


def _log_rows(shape, gen, flat=True):
    """Log-probabilities along the last axis: uniform within 40 % (what training starts from), or Dirichlet(1)"""
    x = torch.rand(shape, device="cuda", generator=gen)
    x = x.mul_(0.8).add_(0.6) if flat else x.clamp_(1e-7, 1 - 1e-7).log_().neg_()
    return x.div_(x.sum(-1, keepdim=True)).log_()


def _hclt(parent, K, C, gen, flat=True):
    bpc = P.hclt_from_clt(parent, C, K)
    V = len(parent)
    bpc.set_params(_log_rows((V, K, K), gen, flat).cpu().numpy(), _log_rows((V, K, C), gen, flat).cpu().numpy())
    return bpc


def _clusters(n, heads, gen):
    """[n, heads] one-hot head masks of uniform cluster ids"""
    mask = torch.zeros((n, heads), device="cuda")
    mask[torch.arange(n, device="cuda"), torch.randint(heads, (n,), device="cuda", generator=gen)] = 1.0
    return mask


def _pruned_heads(parent, K, C, heads, keep, gen):
    """`heads` roots over one HCLT body whose sums keep about `keep` of their K children (two at least), compiled as the
    flat description of its nodes: input nodes, then per tree node, children first, its products and its sums."""
    V, rng = len(parent), np.random.default_rng(17)
    children = [[] for _ in range(V)]
    for v, p in enumerate(parent):
        if p >= 0:
            children[p].append(v)
    root = int(np.flatnonzero(parent < 0)[0])
    order, stack = [], [root]
    while stack:
        order.append(stack.pop())
        stack.extend(children[order[-1]])
    first_of = {v: v * K for v in range(V)}      # first of the K nodes a parent's products take: inputs, or sums
    kinds, sizes, lists = [np.zeros(V * K, np.uint8)], [np.zeros(V * K, np.int64)], []
    at = V * K
    for v in reversed(order):
        if not children[v]:
            continue
        parts = [v * K] + [first_of[c] for c in children[v]]
        kinds.append(np.full(K, 2, np.uint8))
        sizes.append(np.full(K, len(parts), np.int64))
        lists.append((np.arange(K)[:, None] + np.array(parts)).reshape(-1))
        products = at + np.arange(K)
        at += K
        sums = heads if v == root else K
        kept = rng.random((sums, K)) < (1.0 if v == root else keep)
        kept[np.arange(sums)[:, None], np.stack([rng.choice(K, 2, replace=False) for _ in range(sums)])] = True
        kinds.append(np.ones(sums, np.uint8))
        sizes.append(kept.sum(1))
        lists.append(np.broadcast_to(products, (sums, K))[kept])
        first_of[v] = at
        at += sums
    ptr = np.concatenate([[0], np.cumsum(np.concatenate(sizes))])
    kinds, lists = np.concatenate(kinds), np.concatenate(lists)
    weight = torch.rand(len(lists), device="cuda", generator=gen).cpu().numpy() * 0.8 + 0.6
    total = np.add.reduceat(weight, ptr[V * K:-1])
    logp = np.log(weight / np.repeat(total, np.diff(ptr)[V * K:]))
    return P.compile_multihead(kinds, ptr, lists, logp, np.repeat(np.arange(V), K), _log_rows((V * K, C), gen).cpu().numpy(),
                               V, C, heads)


def _forest(case, data, gen):
    """One tree per patch over the pixels of the whole image (variable = channel, row, column)"""
    side, ph, pw, ch = (case[k] for k in ("side", "ph", "pw", "ch"))
    pixel = np.arange(_variables(case)).reshape(ch, side * ph, side * pw)
    parent = np.empty(pixel.size, np.int32)
    for i in range(side):
        for j in range(side):
            own = pixel[:, i * ph:(i + 1) * ph, j * pw:(j + 1) * pw].reshape(-1)
            tree = _tree(data[:, torch.from_numpy(own).cuda()])
            parent[own] = np.where(tree < 0, -1, own[tree])
    bpc = P.hclt_forest_from_clts(parent, case["C"], case["K"], case["heads"])
    bpc.set_params(_log_rows((len(parent), case["K"], case["K"]), gen).cpu().numpy(),
                   _log_rows((len(parent), case["K"], case["C"]), gen).cpu().numpy())
    return bpc


def _parameter_rows(bpc, rows, K, C, gen):
    """[rows, num_parameters]: every sum's K and every input node's C log-parameters normalised"""
    ns = bpc.num_inner_params()
    out = torch.empty((rows, bpc.num_parameters()), device="cuda")
    for r in range(rows):
        out[r, :ns] = _log_rows((ns // K, K), gen, False).view(-1)
        out[r, ns:] = _log_rows((bpc.num_input_params() // C, C), gen, False).view(-1)
    return out


def _gumbel(shape, gen):
    x = torch.empty(shape, device="cuda")
    for part in x.view(shape[0], -1).split(512):
        part.uniform_(1e-7, 1 - 1e-7, generator=gen).log_().neg_().log_().neg_()
    return x


def prepare(case, seed):
    """Data and parameters come from the seed; the structure of the circuit is the case's, learned (and pruned) from a
    training set of its own."""
    gen, fixed, kind = _generator(seed), _generator(17), case["kind"]
    if kind == "soft":
        V, C, n = case["V"], case["C"], case["n"]
        ids = _images(n, V, 1, 1, C, gen)
        tree = _tree(_images(TRAIN, V, 1, 1, C, fixed))
        # log-likelihoods of every cluster's circuit on a patch: a common level, the image's own cluster ahead
        ev = torch.empty((n, V, C), device="cuda")
        ev.uniform_(1e-7, 1 - 1e-7, generator=gen).log_().neg_().log_().mul_(-8.0)
        ev += -600.0 + 30.0 * torch.randn((n, V, 1), device="cuda", generator=gen)
        ev.scatter_add_(2, ids.long()[:, :, None], torch.full((n, V, 1), 20.0, device="cuda"))
        return dict(kind=kind, case=case, seed=seed, bpc=_hclt(tree, case["K"], C, gen), data=ev)
    if kind == "forest":
        size = case["side"] * case["ph"], case["side"] * case["pw"], case["ch"], case["C"]
        bpc, data = _forest(case, _images(TRAIN, *size, fixed), gen), _images(case["n"], *size, gen)
        masks = torch.stack([_clusters(case["n"], case["heads"], gen) for _ in range(case["side"] ** 2)])
        return dict(kind=kind, case=case, seed=seed, bpc=bpc, data=data, masks=masks)
    n, size = case.get("n"), (case["h"], case["w"], case["ch"], case["C"])
    data = _images(n, *size, gen) if kind in ("score", "em", "heads", "structure") else None
    if kind == "structure":
        return dict(kind=kind, case=case, data=data)
    K, C, parent = case["K"], case["C"], _tree(_images(TRAIN, *size, fixed))
    if kind == "score":
        return dict(kind=kind, case=case, bpc=_hclt(parent, K, C, gen), data=data)
    if kind == "em":
        weights = torch.rand(n, device="cuda", generator=gen) if case["weighted"] else None
        return dict(kind=kind, case=case, seed=seed, bpc=_hclt(parent, K, C, gen), data=data, weights=weights)
    if kind == "heads":
        bpc = _pruned_heads(parent, K, C, case["heads"], case["keep"], gen)
        return dict(kind=kind, case=case, seed=seed, bpc=bpc, data=data, mask=_clusters(n, case["heads"], gen))
    bpc = _hclt(parent, K, C, gen, flat=False)
    if kind == "sample":
        noise = case["n"], bpc.size("inner_tree_nodes") * K
        return dict(kind=kind, bpc=bpc, node_noise=_gumbel(noise, gen), leaf_noise=_gumbel((case["n"], len(parent), C), gen))
    p = _parameter_rows(bpc, case["rows"], K, C, gen)
    if kind == "kl":
        return dict(kind=kind, bpc=bpc, p=p, q=_parameter_rows(bpc, case["rows"], K, C, gen))
    noise = _gumbel((case["rows"], bpc.num_inner_params()), gen) if case["gumbel"] else None
    grads = torch.randn((case["rows"], len(parent), C), device="cuda", generator=gen)
    return dict(kind=kind, bpc=bpc, p=p, noise=noise, grads=grads)


# ---- one pass ---------------------------------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "score":
        return P.loglikelihoods(state["bpc"], state["data"], batch_size=state["case"]["batch"])
    if kind == "structure":
        mi = P.pairwise_MI(state["data"], state["case"]["C"], 0.1)
        return mi, P.chow_liu_tree(mi)
    if kind == "kl":
        return P.kld(state["bpc"], state["p"], state["q"]), P.kld_backward(state["bpc"], state["p"], state["q"])
    if kind == "relaxed":
        soft = P.gumbel_sample_rows(state["bpc"], state["p"], temperature=0.7, noise=state["noise"])
        return soft, P.gumbel_sample_backward_rows(state["bpc"], state["p"], state["grads"], temperature=0.7, noise=state["noise"])
    if kind == "sample":
        return P.sample(state["bpc"], state["node_noise"], state["leaf_noise"])
    # an epoch of mini-batch EM, shuffled from the state's own seed, and the trained parameters back on the host
    bpc, data = state["bpc"], state["data"]
    how = dict(batch_size=state["case"]["batch"], pseudocount=0.1, param_inertia=0.9,
               generator=torch.Generator().manual_seed(state["seed"]))
    if kind == "forest":
        lls = P.mini_batch_em_for_forest(bpc, data, state["masks"], 1, **how)
        return lls, bpc.get_params(), bpc.get_heads()
    if kind == "heads":
        lls = P.mini_batch_em_for_multihead_pc(bpc, data, state["mask"], 1, **how)
    elif kind == "soft":
        lls = P.mini_batch_em_with_reg(bpc, data, 1, **how)
    else:
        lls = P.mini_batch_em(bpc, data, 1, weights=state["weights"], **how)
    return lls, P.vectorize_parameters(bpc)


def work(case):
    """Bytes: data, noise and parameters in once, results out once.  Flops: two per multiply-add of the K x K blocks
    (up, down and the statistics for a training pass), and what the leaf terms take."""
    kind, V, C = case["kind"], _variables(case), case["C"]
    if kind == "structure":
        return dict(bytes=case["n"] * V + 4 * V * V, flops=case["n"] * V * V)
    K = case["K"]
    sums, leaves = int(INNER * V) * K * K, V * K * C
    n = case.get("n", 0)
    if kind == "score":
        return dict(bytes=n * V + 4 * (sums + leaves) + 4 * n, flops=2 * sums * n)
    if kind == "em":
        return dict(bytes=n * V + 8 * (sums + leaves), flops=6 * sums * n)
    if kind == "heads":
        sums = int(sums * case["keep"]) + case["heads"] * K
        return dict(bytes=n * (V + 4 * case["heads"]) + 8 * (sums + leaves), flops=6 * sums * n)
    if kind == "forest":
        trees = case["side"] ** 2
        sums += trees * case["heads"] * K
        return dict(bytes=n * (V + 4 * trees * case["heads"]) + 8 * (sums + leaves), flops=6 * sums * n)
    if kind == "soft":
        return dict(bytes=4 * n * V * C + 8 * (sums + leaves), flops=6 * sums * n + 6 * leaves * n)
    if kind == "sample":
        return dict(bytes=4 * n * (int(INNER * V) * K + V * C) + 4 * (sums + leaves) + n * V, flops=n * (int(INNER * V) * K + V * C))
    rows = case["rows"]
    if kind == "kl":
        return dict(bytes=16 * rows * (sums + leaves), flops=12 * rows * (sums + leaves))
    return dict(bytes=rows * (8 * (sums + leaves) + 8 * V * C + (4 * sums if case["gumbel"] else 0)), flops=12 * rows * (sums + leaves))


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "structure":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 1e-5, "max": 1e-3}
