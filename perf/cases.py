"""Measured workloads of the matcher: what its users call, over the sizes that they use.

listed() names the workloads, draw() gives more of the same ranges, prepare() makes what a
caller has in hand before the call, run() is one pass through the public Python API, work()
the bytes and operations of a pass, exact() its result in float64 where outputs are
computed numbers (match lists and visual words are whole numbers).

Descriptors are SIFT-like as in v3dmatch.synth (Gamma(0.5) components, L2 normalised,
clipped at 0.2, renormalised, quantised as round(512 x)); a share of the right set are noisy
copies (sigma 0.05 per component) of left descriptors, the rest unrelated.  They are drawn
with torch on the GPU, since a batch holds millions.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "eth-v3d-lgpl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import v3dmatch  # noqa: E402
from v3dmatch import learned, voctree  # noqa: E402

FORMS = {"fp32": v3dmatch.PREC_FP32, "bf16": v3dmatch.PREC_BF16, "fp8": v3dmatch.PREC_FP8,
         "learned": v3dmatch.PREC_LEARNED}
SIGMA = 0.05
TAU = 0.05


def listed():
    return [
        # the reference's own call sequence (set both sides, findPutativeMatches) on the
        # smallest images: latency of uploads, launches and the result copy
        {"name": "pair_512_host", "kind": "pair", "form": "fp32", "nL": 512, "nR": 480, "upload": "host_f32",
         "min_score": 0.9, "min_ratio": 0.8},
        # an ordinary photo pair uploaded as uint8 SIFT descriptors, ragged counts
        {"name": "pair_2085_u8", "kind": "pair", "form": "fp32", "nL": 2085, "nR": 1893, "upload": "host_u8",
         "min_score": 0.9, "min_ratio": 0.8},
        # descriptors extracted on the GPU and handed over as device pointers, the exact form
        {"name": "pair_4096", "kind": "pair", "form": "fp32", "nL": 4096, "nR": 4096, "upload": "device",
         "min_score": 0.9, "min_ratio": 0.8},
        # the largest ordinary images (16k features a side), the exact form
        {"name": "pair_16384", "kind": "pair", "form": "fp32", "nL": 16384, "nR": 16384, "upload": "device",
         "min_score": 0.9, "min_ratio": 0.8},
        # the BF16 shortlist on large ragged images
        {"name": "pair_13k_bf16", "kind": "pair", "form": "bf16", "nL": 13107, "nR": 15843, "upload": "device",
         "min_score": 0.9, "min_ratio": 0.8},
        # the FP8 shortlist on a very large pair (stitched or gigapixel images)
        {"name": "pair_32768_fp8", "kind": "pair", "form": "fp8", "nL": 32768, "nR": 32768, "upload": "device",
         "min_score": 0.9, "min_ratio": 0.8},
        # the learned shortlist with its sampled check, one pair at a time
        {"name": "pair_16384_learned", "kind": "pair", "form": "learned", "nL": 16384, "nR": 16384,
         "upload": "device", "min_score": 0.9, "min_ratio": 0.8},
        # guided matching: a find, then the epipolar guided call the SfM callers make after
        # estimating F
        {"name": "guided_8k", "kind": "guided", "matrix": "F", "nL": 7950, "nR": 8192, "threshold": 3.0,
         "min_score": 0.9, "min_ratio": 0.8},
        # the exact form over a batch of uneven pairs (one image collection, resident)
        {"name": "batch256_fp32", "kind": "batch", "form": "fp32", "pairs": 256, "layout": 1, "dtype": "u8",
         "min_score": 0.9, "min_ratio": 0.8},
        # the same in the learned form: the framework's headline workload
        {"name": "batch256_learned", "kind": "batch", "form": "learned", "pairs": 256, "layout": 1, "dtype": "u8",
         "min_score": 0.9, "min_ratio": 0.8},
        # vocabulary-tree quantisation of a collection's descriptors
        {"name": "voctree_1m", "kind": "voctree", "branch": 50, "depth": 3, "n": 1000000},
        # forward and backward of the shortlist network on one training minibatch
        {"name": "train_grads_4096", "kind": "grads", "batch": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pair", "pair", "pair", "pair", "batch", "batch", "guided", "voctree", "grads"])
    minimum = rng.choice([0.9, 0.9, 0.85, 0.93])
    ratio = rng.choice([0.8, 0.8, 0.8, 0.7, -1.0])  # -1: the reference's variant without the ratio test
    if kind == "pair":
        form = rng.choice(["fp32", "fp32", "fp32", "bf16", "fp8", "learned"])
        return {"kind": kind, "form": form, "nL": _log_int(rng, 64, 24000), "nR": _log_int(rng, 64, 24000),
                "upload": rng.choice(["host_f32", "host_u8", "device"]), "min_score": minimum, "min_ratio": ratio}
    if kind == "batch":
        return {"kind": kind, "form": rng.choice(["fp32", "bf16", "learned"]), "pairs": _log_int(rng, 3, 160),
                "layout": rng.randrange(2, 1000), "dtype": rng.choice(["u8", "f32"]), "min_score": minimum,
                "min_ratio": ratio}
    if kind == "guided":
        return {"kind": kind, "matrix": rng.choice(["F", "H"]), "nL": _log_int(rng, 200, 16384),
                "nR": _log_int(rng, 200, 16384), "threshold": rng.choice([1.5, 3.0, 6.0]), "min_score": minimum,
                "min_ratio": ratio}
    if kind == "voctree":
        branch, depth = rng.choice([(50, 3), (10, 3), (8, 4), (10, 5), (64, 2), (300, 2)])
        return {"kind": kind, "branch": branch, "depth": depth, "n": _log_int(rng, 1000, 1000000)}
    return {"kind": kind, "batch": _log_int(rng, 64, 4096)}


# ---------------------------------------------------------------------------------- inputs

def _unit(x):
    return x / x.norm(dim=1, keepdim=True).clamp_min(1e-12)


def _quantise(x):
    return (512.0 * x).round().clamp(0, 255).to(torch.uint8)


def _fresh(g, n):
    """n unrelated uint8 descriptors (Gamma(0.5, 1) is half the square of a normal)."""
    x = _unit(torch.randn((n, 128), generator=g, device="cuda").square())
    return _quantise(_unit(x.clamp_max(0.2)))


def _dequantise(q):
    f = q.float()
    return f * (1.0 / f.square().sum(1, keepdim=True).sqrt())


def _pair(g, nL, nR, copies=0.4):
    """uint8 (nL, 128), uint8 (nR, 128) and, per right descriptor, its left source or -1."""
    qL = _fresh(g, nL)
    n = int(copies * min(nL, nR) + 0.5)
    src = torch.randperm(nL, generator=g, device="cuda")[:n]
    noisy = _dequantise(qL[src]) + SIGMA * torch.randn((n, 128), generator=g, device="cuda")
    qR = torch.cat([_quantise(_unit(noisy.clamp_min(0.0))), _fresh(g, nR - n)])
    truth = torch.cat([src, torch.full((nR - n,), -1, device="cuda", dtype=src.dtype)])
    order = torch.randperm(nR, generator=g, device="cuda")
    return qL, qR[order].contiguous(), truth[order]


def _batch_sizes(case):
    """500 to 16000 features an image (log-uniform) and 30-60% copies a pair."""
    rng = np.random.RandomState(case["layout"])
    n = np.exp(rng.uniform(math.log(500), math.log(16000), (case["pairs"], 2))).astype(int)
    return n, rng.uniform(0.3, 0.6, case["pairs"])


def _down32(n):
    return n - n % 32


def _geometry(nL, nR, truth, seed):
    """Pixel positions of a two-view scene (copies project the same point) with F and H."""
    rng = np.random.RandomState(seed % (2 ** 31))
    K = np.array([[800.0, 0, 512], [0, 800.0, 384], [0, 0, 1]])
    a = rng.standard_normal(3) * 0.05
    th = np.linalg.norm(a)
    k = a / th
    S = np.array([[0, -k[2], k[1]], [k[2], 0, -k[0]], [-k[1], k[0], 0]])
    R = np.eye(3) + np.sin(th) * S + (1 - np.cos(th)) * S @ S
    t = np.array([1.0, 0.1, 0.05]) + rng.standard_normal(3) * 0.02
    T = np.array([[0, -t[2], t[1]], [t[2], 0, -t[0]], [-t[1], t[0], 0]])
    uv = np.stack([rng.uniform(0, 1024, nL), rng.uniform(0, 768, nL)], 1)
    depth = rng.uniform(6, 20, nL)
    Ki = np.linalg.inv(K)
    p = (K @ (R @ ((Ki @ np.c_[uv, np.ones(nL)].T) * depth) + t[:, None])).T
    p = p[:, :2] / p[:, 2:3]
    right = np.stack([rng.uniform(0, 1024, nR), rng.uniform(0, 768, nR)], 1)
    cp = truth >= 0
    right[cp] = p[truth[cp]] + 0.7 * rng.standard_normal((int(cp.sum()), 2))
    F = Ki.T @ T @ R @ Ki
    H = K @ (R + np.outer(t, [0, 0, 1.0]) / np.median(depth)) @ Ki
    return uv.astype(np.float32), right.astype(np.float32), F / np.linalg.norm(F), H / H[2, 2]


def _tree(g, branch, depth, spread=0.35):
    """A k-means-like tree, level after level, every node's children near its direction."""
    levels = [_unit(torch.randn((branch, 128), generator=g, device="cuda").abs())]
    for _ in range(1, depth):
        kids = levels[-1][:, None, :] + spread * torch.randn((levels[-1].shape[0], branch, 128), generator=g,
                                                             device="cuda").abs() / math.sqrt(128)
        levels.append(_unit(kids.reshape(-1, 128)))
    return torch.cat(levels), levels[-1]


def _partners(pairs, out):
    """The matches as the callers keep them: per left feature its right feature, or -1."""
    out.fill(-1)
    out[pairs[:, 0]] = pairs[:, 1]
    return out


def _matcher(form):
    m = v3dmatch.SIFT_Matching(0)
    m.enableRoundingWarning(False)
    m.set_precision(FORMS[form])
    if form == "learned":
        learned.Network(m).load(learned.WEIGHTS_PATH)
    return m


def _upload(q, kind):
    if kind == "host_u8":
        return q.cpu().numpy()
    f = _dequantise(q).contiguous()
    return f if kind == "device" else f.cpu().numpy()


def _training(seed, batch):
    """Pool rows and one minibatch of (anchor, positive, negative) triplets."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    qA = _fresh(g, batch)
    noisy = _dequantise(qA) + SIGMA * torch.randn((batch, 128), generator=g, device="cuda")
    qP = _quantise(_unit(noisy.clamp_min(0.0)))
    pool = torch.cat([_dequantise(qA), _dequantise(qP), _dequantise(_fresh(g, batch))]).cpu().numpy()
    i = np.arange(batch, dtype=np.int32)
    tri = np.stack([i, batch + i, 2 * batch + i], 1)
    rng = np.random.RandomState(seed % (2 ** 31))
    params = {"W1": (rng.standard_normal((256, 128)) * math.sqrt(2.0 / 128)).astype(np.float32),
              "b1": (0.05 * rng.standard_normal(256)).astype(np.float32),
              "W2": (rng.standard_normal((32, 256)) * math.sqrt(1.0 / 256)).astype(np.float32),
              "b2": (0.05 * rng.standard_normal(32)).astype(np.float32)}
    return pool, tri, params


def prepare(case, seed):
    kind = case["kind"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    s = {"case": case}
    if kind in ("pair", "guided"):
        s["found"], s["guided"] = np.empty(case["nL"], np.int32), np.empty(case["nL"], np.int32)
    if kind == "pair":
        qL, qR, _ = _pair(g, case["nL"], case["nR"])
        s["L"], s["R"] = _upload(qL, case["upload"]), _upload(qR, case["upload"])
        s["m"] = m = _matcher(case["form"])
        m.allocate(case["nL"], case["nR"])
    elif kind == "guided":
        qL, qR, truth = _pair(g, case["nL"], case["nR"])
        s["L"], s["R"] = _upload(qL, "device"), _upload(qR, "device")
        s["lxy"], s["rxy"], F, H = _geometry(case["nL"], case["nR"], truth.cpu().numpy(), seed)
        s["M"] = F if case["matrix"] == "F" else H
        s["m"] = m = _matcher("fp32")
        m.allocate(case["nL"], case["nR"], True)
    elif kind == "batch":
        n, copies = _batch_sizes(case)
        parts = []
        for (a, b), c in zip(n, copies):
            qL, qR, _ = _pair(g, int(a), int(b), float(c))
            parts += [qL, qR]
        q = torch.cat(parts)
        del parts
        s["m"] = m = _matcher(case["form"])
        m.set_derived_cache(False)  # every pass converts or embeds the images, as on new ones
        m.batch_set_images(n.reshape(-1), q.cpu().numpy() if case["dtype"] == "u8" else _dequantise(q).cpu().numpy())
        left = np.arange(0, 2 * case["pairs"], 2, dtype=np.int32)
        m.batch_set_pairs(left, left + 1)
        s["pairs"] = np.full((int(n.min(1).sum()), 2), -1, np.int32)
    elif kind == "voctree":
        nodes, leaves = _tree(g, case["branch"], case["depth"])
        at = torch.randint(0, leaves.shape[0], (case["n"],), generator=g, device="cuda")
        noise = 0.08 * torch.randn((case["n"], 128), generator=g, device="cuda")
        s["keys"] = _unit((leaves[at] + noise).abs()).contiguous()
        s["words"] = torch.empty(case["n"], dtype=torch.int32, device="cuda")
        s["tree"] = t = voctree.VocabularyTree(case["branch"], case["depth"])
        t.setNodes(nodes.cpu().numpy())
    else:
        pool, tri, params = _training(seed, case["batch"])
        s["m"] = v3dmatch.SIFT_Matching(0)
        s["net"] = net = learned.Network(s["m"])
        net.set_params(params)
        net.set_training(pool, tri)
        s["idx"] = np.arange(case["batch"], dtype=np.int32)
    torch.cuda.synchronize()  # the library works on streams of its own
    return s


# ---------------------------------------------------------------------------------- one pass

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("pair", "guided"):
        m, L, R = s["m"], s["L"], s["R"]
        if kind == "guided" or case["upload"] == "device":
            m.set_left_device(case["nL"], L.data_ptr())
            m.set_right_device(case["nR"], R.data_ptr())
        elif case["upload"] == "host_u8":
            m.set_left_u8(L)
            m.set_right_u8(R)
        else:
            m.setLeftFeatures(case["nL"], L)
            m.setRightFeatures(case["nR"], R)
        found = _partners(m.find_putative_matches_array(case["min_score"], case["min_ratio"]), s["found"])
        if kind == "pair":
            return found
        kept = m.run_guided_array(case["matrix"] == "H", s["M"], case["threshold"], s["lxy"], s["rxy"],
                                  case["min_score"], case["min_ratio"])
        return {"found": found, "guided": _partners(kept, s["guided"])}
    if kind == "batch":
        s["m"].batch_match_async(case["min_score"], case["min_ratio"])
        offsets, pairs = s["m"].batch_get_matches()
        s["pairs"][:len(pairs)] = pairs  # the caller's own store, the same size for every pass
        return {"offsets": offsets, "pairs": s["pairs"]}
    if kind == "voctree":
        s["tree"].traverse_device(case["n"], s["keys"].data_ptr(), s["words"].data_ptr())
        s["tree"].synchronize()
        return s["words"]
    loss, grads, hard = s["net"].gradients(s["idx"], TAU)
    return {"loss": loss, "grads": grads, "hard": hard}


# ---------------------------------------------------------------------------------- work

def _form_flops(form, rows, scores):
    if form == "learned":  # embedding, then one 32-d code product a score
        return 2.0 * rows * (128 * 256 + 256 * 32) + 2.0 * scores * 32
    return 2.0 * scores * 128


def work(case):
    kind = case["kind"]
    if kind in ("pair", "guided"):
        a, b = _down32(case["nL"]), _down32(case["nR"])
        element = 1 if case.get("upload") == "host_u8" else 4
        moved = (a + b) * 128 * element + 8 * 0.3 * min(a, b)
        if kind == "pair":
            return {"bytes": moved, "flops": _form_flops(case["form"], a + b, float(a) * b)}
        # the scores of the find and of the guided call, and about 20 operations a distance
        return {"bytes": moved + 8 * (a + b), "flops": (4.0 * 128 + 20) * a * b}
    if kind == "batch":
        n = _batch_sizes(case)[0]
        n = n - n % 32
        scores = float((n[:, 0].astype(float) * n[:, 1]).sum())
        rows = int(n.sum())
        return {"bytes": rows * 128.0 * (1 if case["dtype"] == "u8" else 4) + 8 * 0.15 * rows,
                "flops": _form_flops(case["form"], rows, scores)}
    if kind == "voctree":
        nodes = sum(case["branch"] ** (d + 1) for d in range(case["depth"]))
        return {"bytes": 512.0 * (case["n"] + nodes) + 4 * case["n"],
                "flops": 2.0 * 128 * case["n"] * case["branch"] * case["depth"]}
    # forward and backward of 3 rows a triplet, and every anchor against every positive
    b = case["batch"]
    return {"bytes": 512.0 * 3 * b + 2 * 4.0 * learned.N_PARAMS,
            "flops": 3 * 2.0 * 3 * b * (128 * 256 + 256 * 32) + 2.0 * b * b * 32}


# ---------------------------------------------------------------------------------- float64

def exact(case, seed):
    if case["kind"] != "grads":
        return None  # whole numbers
    pool, tri, params = _training(seed, case["batch"])
    p = {k: v.astype(np.float64) for k, v in params.items()}
    b = case["batch"]
    x = pool[tri.T.reshape(-1)].astype(np.float64)
    a = x @ p["W1"].T + p["b1"]
    h = np.maximum(a, 0.0)
    z = h @ p["W2"].T + p["b2"]
    n = np.maximum(np.linalg.norm(z, axis=1, keepdims=True), 1e-12)
    c = z / n
    ca, cp, cn = c[:b], c[b:2 * b], c[2 * b:]
    sp, sn = (ca * cp).sum(1), (ca * cn).sum(1)
    S = ca @ cp.T
    np.fill_diagonal(S, -np.inf)
    hard = S.argmax(1)
    sh = S[np.arange(b), hard]
    loss = (np.logaddexp(0, (sn - sp) / TAU) + np.logaddexp(0, (sh - sp) / TAU)).mean()
    gn = 0.5 * (1 + np.tanh((sn - sp) / (2 * TAU))) / (TAU * b)
    gh = 0.5 * (1 + np.tanh((sh - sp) / (2 * TAU))) / (TAU * b)
    dc = np.concatenate([gn[:, None] * (cn - cp) + gh[:, None] * (cp[hard] - cp), -(gn + gh)[:, None] * ca,
                         gn[:, None] * ca])
    np.add.at(dc, b + hard, gh[:, None] * ca)
    dz = (dc - c * (c * dc).sum(1, keepdims=True)) / n
    dh = (dz @ p["W2"]) * (a > 0)
    grads = {"W1": dh.T @ x, "b1": dh.sum(0), "W2": dz.T @ h, "b2": dz.sum(0)}
    return {"loss": float(loss), "grads": grads, "hard": None}
