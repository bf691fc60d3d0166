"""The measured work of this framework: what a user has it do, through nscale_amd.gpu's public calls.

Cases (h x w pixels):
 * recon      morphological reconstruction of one (marker, mask) pair: from a region of interest, where
              launches and host reads count, to a whole 4096 x 4096 tile; uint8, float32 and int32 planes;
 * batch      a set of uint8 pairs of uneven sizes and mixed connectivity in one call (the tiles of a slide
              that wait for the same operator);
 * hmin       what separates touching nuclei: distance transform of each mask, then h-minima (float32) of
              the negated distances of the whole set;
 * label      the labelling family on a binary mask: area opening, labels, canonical labels, boxes and areas;
 * normalize  colour normalization of a tile to a target's statistics;
 * features   geometry, intensity and gradient features of every nucleus of a tile;
 * chain      segmentNuclei on a tile, with the reference's labels, or canonical labels with boxes and areas;
 * served     a queue of tiles of mixed sizes through the continuous-batching server.

Sizes are those of this repository's benchmark and tests: tiles with sides of 512 to 4096 pixels, the short
side log-uniform and the long one up to twice it, odd sizes as they come, and regions of interest below that.
"""
import math
import random

import torch

from nscale_amd import gpu

# ---- cases --------------------------------------------------------------------------------------------


def listed():
    return [
        # a region of interest: launch latency and host reads
        {"name": "recon_roi", "kind": "recon", "h": 256, "w": 320, "conn": 4, "dtype": "u8"},
        # the reconstruction benchmark: a whole tile of ellipses with noise, marker = mask - 10
        {"name": "recon_4096", "kind": "recon", "h": 4096, "w": 4096, "conn": 8, "dtype": "u8"},
        # the batched benchmark's size distribution, a quarter of its pairs
        {"name": "batch_64", "kind": "batch", "n": 64, "lo": 512, "hi": 4096, "sizes": 2026},
        # h-minima of distance maps, a set of ordinary tiles
        {"name": "hmin_16", "kind": "hmin", "n": 16, "lo": 512, "hi": 2048, "sizes": 7},
        # labels, boxes and areas of a large odd tile's binary mask
        {"name": "label_4096", "kind": "label", "h": 4096, "w": 3071, "conn": 8},
        # a tile of the size that whole slides are cut into
        {"name": "normalize_4096", "kind": "normalize", "h": 4096, "w": 4096},
        # a small tile: fixed costs of the two passes
        {"name": "normalize_600", "kind": "normalize", "h": 600, "w": 517},
        # the features of about 2000 nuclei
        {"name": "features_2048", "kind": "features", "h": 2048, "w": 2048},
        # the smallest tile of the served distribution: a chain of about a hundred dependent launches
        {"name": "chain_512", "kind": "chain", "h": 512, "w": 512, "params": "default", "boxes": False},
        # an ordinary odd tile with the reference test's own parameters, canonical labels, boxes and areas
        {"name": "chain_odd", "kind": "chain", "h": 1531, "w": 2243, "params": "test", "boxes": True},
        # the default benchmark's tile
        {"name": "chain_4096", "kind": "chain", "h": 4096, "w": 4096, "params": "default", "boxes": False},
        # twelve tiles of mixed sizes on eight slots
        {"name": "served_12", "kind": "served", "n": 12, "lo": 512, "hi": 2896, "sizes": 3, "slots": 8},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _tile(rng, lo=512, hi=4096, area=4096 * 4096):
    """Short side log-uniform in [lo, hi], long side up to twice it (within the area), either way up."""
    a = _log_uniform(rng, lo, hi)
    b = min(int(round(a * rng.uniform(1.0, 2.0))), area // a)
    return (a, b) if rng.random() < 0.5 else (b, a)


def draw(rng):
    kind = rng.choice(["recon", "recon", "batch", "hmin", "label", "normalize", "features", "chain", "chain", "served"])
    case = {"kind": kind}
    if kind == "batch":
        case.update(n=_log_uniform(rng, 2, 64), lo=rng.randint(200, 512), hi=rng.randint(1024, 2896),
                    sizes=rng.randrange(1 << 30))
    elif kind == "hmin":
        case.update(n=_log_uniform(rng, 1, 16), lo=rng.randint(200, 512), hi=rng.randint(1024, 1800),
                    sizes=rng.randrange(1 << 30))
    elif kind == "served":
        case.update(n=rng.randint(2, 10), lo=512, hi=rng.randint(1024, 2000), sizes=rng.randrange(1 << 30), slots=8)
    else:
        small = kind in ("recon", "label", "normalize", "features")
        h, w = _tile(rng, lo=96 if small else 512, area=2048 * 2048 if kind == "features" else 4096 * 4096)
        case.update(h=h, w=w)
    if kind == "recon":
        case.update(conn=rng.choice([4, 8]), dtype=rng.choice(["u8", "u8", "f32", "i32"]))
    elif kind == "label":
        case.update(conn=rng.choice([4, 8]))
    elif kind == "chain":
        case.update(params=rng.choice(["default", "test"]), boxes=rng.random() < 0.5)
    return case


def _sizes(case):
    """The (h, w) of the images of a set."""
    rng = random.Random(case["sizes"])
    return [_tile(rng, case["lo"], case["hi"]) for _ in range(case["n"])]


def work(case):
    """Bytes and operations of one pass: each input read once, each output written once; the operations
    are those of the arithmetic that the method is defined by (comparisons are not counted)."""
    kind = case["kind"]
    if "n" in case:
        px = sum(h * w for h, w in _sizes(case))
    else:
        px = case["h"] * case["w"]
    if kind == "recon":
        return {"bytes": 3 * px * (1 if case["dtype"] == "u8" else 4), "flops": 0}
    if kind == "batch":
        return {"bytes": 3 * px, "flops": 0}
    if kind == "hmin":  # mask in, distances out; distances in, h-minima out
        return {"bytes": (1 + 4 + 4 + 4) * px, "flops": 0}
    if kind == "label":  # area opening: 1 in, 1 out; labels: 1 in, 4 out; relabelled and boxed in place
        return {"bytes": (1 + 1 + 1 + 4) * px, "flops": 0}
    if kind == "normalize":  # two colour transforms: four 3 x 3 products, six transcendental functions
        return {"bytes": 6 * px, "flops": 4 * 15 * px + 6 * px}
    if kind == "features":  # labels and a BGR image in
        return {"bytes": (4 + 3) * px, "flops": 0}
    return {"bytes": (3 + 4) * px, "flops": 0}  # chain, served: BGR in, labels out


# ---- inputs -------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cpu").manual_seed(seed)


def _device_gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _shapes(h, w, cell, lo, hi, inside, seed, margin=0, turn=0):
    """One ellipse per cell x cell square with semi-axes U[lo, hi]: the (h, w) index of the last ellipse
    that covers each pixel, -1 where none does.  inside keeps each ellipse within its square, margin pixels
    from its sides, so that no two meet, and leaves out the squares that the image cuts; otherwise centres
    are uniform and ellipses overlap.  turn exchanges the axes and turns the ellipses about the same centres."""
    gh, gw = h // cell + 3, w // cell + 3
    u = torch.rand(5, gh, gw, generator=_gen(seed)).cuda()
    a, b = lo + (hi - lo) * u[2], lo + (hi - lo) * u[3]
    r = torch.maximum(a, b)
    gy = torch.arange(gh, device="cuda").view(-1, 1) - 1
    gx = torch.arange(gw, device="cuda").view(1, -1) - 1
    if inside:
        r = r + margin
        cx, cy = gx * cell + r + u[0] * (cell - 2 * r), gy * cell + r + u[1] * (cell - 2 * r)
    else:
        cx, cy = (gx + u[0]) * cell, (gy + u[1]) * cell
    if turn:
        a, b = b, a
    co, si = torch.cos(math.pi * u[4] + turn), torch.sin(math.pi * u[4] + turn)
    y = torch.arange(h, device="cuda").view(-1, 1)
    x = torch.arange(w, device="cuda").view(1, -1)
    iy, ix = torch.div(y, cell, rounding_mode="floor") + 1, torch.div(x, cell, rounding_mode="floor") + 1
    out = torch.full((h, w), -1, dtype=torch.int32, device="cuda")
    reach = [0] if inside else [-1, 0, 1]
    for dy in reach:
        for dx in reach:
            k = (iy + dy) * gw + (ix + dx)
            ex, ey = x + 0.5 - cx.flatten()[k], y + 0.5 - cy.flatten()[k]
            c, s = co.flatten()[k], si.flatten()[k]
            p, q = (ex * c + ey * s) / a.flatten()[k], (ey * c - ex * s) / b.flatten()[k]
            out = torch.where(p * p + q * q <= 1.0, k.to(torch.int32), out)
    if inside:
        whole = (y < h // cell * cell) & (x < w // cell * cell)
        out = torch.where(whole, out, torch.full_like(out, -1))
    return out, gh * gw


def _grey_mask(h, w, seed):
    """Background 220, overlapping ellipses of U[60, 120], Gaussian noise of sigma 8 (uint8)."""
    idx, cells = _shapes(h, w, 20, 4.0, 12.0, False, seed)
    val = torch.randint(60, 121, (cells,), generator=_gen(seed + 1)).float().cuda()
    base = torch.where(idx >= 0, val[idx.clamp(min=0).long()], torch.full((), 220.0, device="cuda"))
    noise = torch.randn(h, w, generator=_device_gen(seed + 2), device="cuda")
    return (base + 8.0 * noise).round_().clamp_(0, 255).to(torch.uint8)


def _pair(h, w, seed):
    mask = _grey_mask(h, w, seed)
    return (mask.to(torch.int16) - 10).clamp_(min=0).to(torch.uint8), mask


def _speckled_mask(h, w, seed):
    """Binary mask (255 / 0) of separate irregular nuclei, one per full cell, and specks too small to keep."""
    a, _ = _shapes(h, w, 34, 4.0, 14.0, True, seed, 2)
    b, _ = _shapes(h, w, 34, 4.0, 14.0, True, seed, 2, turn=1)
    mask = (a >= 0) | (b >= 0)
    near = torch.nn.functional.max_pool2d(mask[None].half(), 7, 1, 3)[0] > 0
    speck = torch.rand(h, w, generator=_device_gen(seed + 1), device="cuda") < 0.004
    return (mask | (speck & ~near)).to(torch.uint8) * 255


def _nuclei_mask(h, w, seed):
    """Binary mask of nuclei, touching ones among them (255 / 0)."""
    idx, _ = _shapes(h, w, 30, 4.0, 14.0, False, seed)
    return (idx >= 0).to(torch.uint8) * 255


def _labelled(h, w, seed):
    """Labels 1..n of separate nuclei (background 0), their (5, n) boxes and a BGR image of them."""
    idx, cells = _shapes(h, w, 40, 4.0, 14.0, True, seed)
    present = torch.unique(idx)
    present = present[present >= 0].long()
    n = int(present.numel())
    number = torch.zeros(cells + 1, dtype=torch.int32, device="cuda")
    number[present + 1] = torch.arange(1, n + 1, dtype=torch.int32, device="cuda")
    labels = number[(idx + 1).long()].contiguous()
    ys, xs = torch.nonzero(labels, as_tuple=True)
    lab = labels[ys, xs].long() - 1
    box = [torch.arange(1, n + 1, device="cuda")]
    for v in (xs, ys):
        box.append(torch.full((n,), 1 << 30, device="cuda").scatter_reduce(0, lab, v, "amin"))
        box.append(torch.full((n,), -1, device="cuda").scatter_reduce(0, lab, v, "amax"))
    tint = torch.randint(-20, 21, (n + 1, 3), generator=_gen(seed + 2)).cuda()
    tint[0] = torch.tensor([90, 160, 140])  # background (230, 220, 230) as an offset from the nuclei's colour
    noise = torch.randint(-6, 7, (h, w, 3), generator=_device_gen(seed + 3), device="cuda")
    bgr = (torch.tensor([140, 60, 90], device="cuda") + tint[labels.long()] + noise).clamp_(0, 255).to(torch.uint8)
    return labels, torch.stack(box).to(torch.int32).contiguous(), bgr.contiguous()


def _he_tile(h, w, seed):
    """A tile of the procedural H&E slide: nuclei, red blood cells, uneven stain, noise (BGR)."""
    return gpu.synth_slide_tile(64 * (seed % 97), 64 * (seed % 89), w, h, seed=seed)


def _params(which):
    p = gpu.default_params()
    if which == "test":  # the reference test's own parameter set
        p.T1, p.T2, p.G1, p.minSize, p.maxSize, p.G2 = 4.0, 3.5, 44, 5, 9000, 31
        p.minSizePl, p.minSizeSeg, p.maxSizeSeg = 20, 5, 1150
        p.fillHolesConnectivity = p.reconConnectivity = p.watershedConnectivity = 4
    return p


# capacity of the box tables of a tile, and the number of columns of the table that a caller keeps of it
MAX_BOXES = 1 << 16
KEPT_BOXES = 1 << 14


def _table(boxes, areas):
    """Boxes and areas in a table of fixed size, one row of a slide's table of tiles."""
    pad = (0, KEPT_BOXES - int(boxes.shape[1]))
    return torch.nn.functional.pad(boxes, pad), torch.nn.functional.pad(areas, pad)



def prepare(case, seed):
    kind = case["kind"]
    if kind == "recon":
        marker, mask = _pair(case["h"], case["w"], seed)
        if case["dtype"] == "f32":
            marker, mask = marker.float() / 255.0, mask.float() / 255.0
        elif case["dtype"] == "i32":
            marker, mask = marker.int() * 257, mask.int() * 257
        return {"kind": kind, "marker": marker, "mask": mask, "conn": case["conn"]}
    if kind == "batch":
        rng = random.Random(seed)
        pairs, conns = [], []
        for k, (h, w) in enumerate(_sizes(case)):
            pairs.append(_pair(h, w, 1000 * seed + 10 * k))
            conns.append(rng.choice([4, 8]))
        return {"kind": kind, "pairs": pairs, "conns": conns}
    if kind == "hmin":
        rng = random.Random(seed)
        masks = [_nuclei_mask(h, w, 1000 * seed + 10 * k) for k, (h, w) in enumerate(_sizes(case))]
        return {"kind": kind, "masks": masks, "conns": [rng.choice([4, 8]) for _ in masks]}
    if kind == "label":
        return {"kind": kind, "mask": _speckled_mask(case["h"], case["w"], seed), "conn": case["conn"]}
    if kind == "normalize":
        mean, std, _ = gpu.normalization_target_parameters(_he_tile(512, 512, seed + 1))
        return {"kind": kind, "bgr": _he_tile(case["h"], case["w"], seed), "mean": mean, "std": std}
    if kind == "features":
        labels, box, bgr = _labelled(case["h"], case["w"], seed)
        return {"kind": kind, "labels": labels, "box": box, "bgr": bgr}
    if kind == "chain":
        h, w = case["h"], case["w"]
        return {"kind": kind, "bgr": _he_tile(h, w, seed), "params": _params(case["params"]), "boxes": case["boxes"],
                "ws": gpu.Workspace(w, h)}
    sizes = _sizes(case)
    return {"kind": kind, "tiles": [_he_tile(h, w, 100 * seed + k) for k, (h, w) in enumerate(sizes)],
            "server": gpu.Server(slots=case["slots"], max_w=4096, max_h=4096)}


def run(state):
    kind = state["kind"]
    if kind == "recon":
        return gpu.imreconstruct(state["marker"], state["mask"], state["conn"])
    if kind == "batch":
        return gpu.imreconstruct_batched(state["pairs"], state["conns"])
    if kind == "hmin":
        dist = [gpu.dist_transform(m) for m in state["masks"]]
        return {"dist": dist, "hmin": gpu.imhmin_batched([-d for d in dist], 1.0, state["conns"])}
    if kind == "label":
        opened, kept = gpu.bwareaopen2(state["mask"], 30, 1500, state["conn"])
        labels = gpu.bwlabel2(opened, state["conn"])
        n = gpu.cc_relabel(labels)
        boxes, areas = gpu.bounding_boxes(labels, n)
        return {"opened": opened, "kept": kept, "labels": labels, "n": n, "boxes": boxes, "areas": areas}
    if kind == "normalize":
        return gpu.normalization(state["bgr"], state["mean"], state["std"])
    if kind == "features":
        return gpu.object_features(state["labels"], state["box"], state["bgr"], channel=2)
    if kind == "chain":
        if state["boxes"]:
            status, labels, n, nuclei, boxes, areas, _ = gpu.segment_nuclei_io(
                state["bgr"], params=state["params"], ws=state["ws"], canonical=True, bbox_mode=gpu.BBOX_ALL,
                max_boxes=MAX_BOXES, with_area=True)
            boxes, areas = _table(boxes, areas)
            return {"status": status, "labels": labels, "n": n, "nuclei": nuclei, "boxes": boxes, "areas": areas}
        status, labels, n, _, _ = gpu.segment_nuclei(state["bgr"], params=state["params"], ws=state["ws"])
        return {"status": status, "labels": labels, "n": n}
    server = state["server"]
    tickets = [server.submit(t, canonical=True, max_labels=MAX_BOXES) for t in state["tiles"]]
    out = []
    for t in tickets:
        status, n, labels, boxes, areas, _ = server.wait(t)
        boxes, areas = _table(boxes, areas)
        out.append({"status": status, "n": n, "labels": labels, "boxes": boxes, "areas": areas})
    return out


# ---- 64-bit values ------------------------------------------------------------------------------------


def _exact_dist(mask):
    """Distance of every nonzero pixel to the nearest zero pixel, by columns and then along rows."""
    h, w = mask.shape
    y = torch.arange(h, device=mask.device, dtype=torch.float64).view(-1, 1).expand(h, w)
    far = 4.0 * (h + w)
    above = torch.where(mask == 0, y, torch.full_like(y, -far)).cummax(0).values
    below = torch.where(mask == 0, y, torch.full_like(y, h + far)).flip(0).cummin(0).values.flip(0)
    g2 = torch.minimum(y - above, below - y).square()
    d2 = g2.clone()
    k = 1
    while k < w and k * k < float(d2.max()):
        d2[:, k:] = torch.minimum(d2[:, k:], g2[:, :-k] + k * k)
        d2[:, :-k] = torch.minimum(d2[:, :-k], g2[:, k:] + k * k)
        k += 1
    return d2.sqrt()


def _exact_hmin(dist, depth, conn):
    """h-minima of -dist: the reconstruction of dist - depth under dist, negated."""
    m = dist - depth
    while True:
        p = torch.nn.functional.pad(m, (1, 1, 1, 1), value=-math.inf)
        h, w = m.shape
        up = m
        for dy in (0, 1, 2):
            for dx in (0, 1, 2):
                if conn == 8 or dy == 1 or dx == 1:
                    up = torch.maximum(up, p[dy:dy + h, dx:dx + w])
        up = torch.minimum(up, dist)
        if torch.equal(up, m):
            return -m
        m = up


def _exact_histogram(value, lab, n):
    """Mean, maximum, minimum, standard deviation, entropy, energy, skewness and kurtosis per label."""
    hist = torch.zeros(n * 256, dtype=torch.float64, device=value.device)
    hist.scatter_add_(0, lab * 256 + value.long(), torch.ones_like(value, dtype=torch.float64))
    hist = hist.view(n, 256)
    v = torch.arange(256, device=value.device, dtype=torch.float64)
    count = hist.sum(1, keepdim=True)
    p = hist / count
    mean = (p * v).sum(1, keepdim=True)
    d = v - mean
    m2, m3, m4 = ((p * d ** k).sum(1) for k in (2, 3, 4))
    top = torch.where(hist > 0, v, torch.full_like(v, -1.0)).amax(1)
    low = torch.where(hist > 0, v, torch.full_like(v, 256.0)).amin(1)
    ent = -(p * torch.where(p > 0, p, torch.ones_like(p)).log2()).sum(1)
    skew = torch.where(m2 > 0, m3 / m2 ** 1.5, torch.zeros_like(m2))
    kurt = torch.where(m2 > 0, m4 / m2 ** 2, torch.zeros_like(m2))
    return torch.stack([mean[:, 0], top, low, m2.sqrt(), ent, (p * p).sum(1), skew, kurt], 1)


def _exact_gradient(grey):
    """Magnitude of central differences (one-sided at the borders), rounded half up, at most 255."""
    g = grey.double()
    gy, gx = torch.gradient(g)
    return ((gx * gx + gy * gy).sqrt() + 0.5).floor().clamp(max=255)


def _exact_perimeter(labels, n):
    """Weights of the 2 x 2 cells along each label's outline."""
    p = torch.nn.functional.pad(labels, (1, 1, 1, 1))
    corners = [p[:-1, :-1], p[:-1, 1:], p[1:, 1:], p[1:, :-1]]
    weight = torch.tensor([0.0, 0.70710678118, 1.0, 0.70710678118, 0.0], dtype=torch.float64, device=labels.device)
    out = torch.zeros(n + 1, dtype=torch.float64, device=labels.device)
    for k, lab in enumerate(corners):
        same = [c == lab for c in corners]
        first = lab > 0
        for j in range(k):
            first = first & ~same[j]
        wt = weight[sum(s.long() for s in same)]
        diagonal = (same[0] & same[2] & ~same[1] & ~same[3]) | (same[1] & same[3] & ~same[0] & ~same[2])
        wt = torch.where(diagonal, torch.full_like(wt, 1.41421356237), wt)
        out.scatter_add_(0, lab[first].long(), wt[first])
    return out[1:]


def _exact_features(labels, box, bgr):
    n = int(box.shape[1])
    ys, xs = torch.nonzero(labels, as_tuple=True)
    lab = labels[ys, xs].long() - 1

    def per_label(v):
        return torch.zeros(n, dtype=torch.float64, device=v.device).scatter_add_(0, lab, v)

    b = box.double()
    cx, cy = xs - ((b[1] + b[2]) / 2)[lab], ys - ((b[3] + b[4]) / 2)[lab]
    area = per_label(torch.ones_like(cx))
    mx, my = per_label(cx) / area, per_label(cy) / area
    mxx = per_label(cx * cx) / area - mx * mx + 1.0 / 12.0
    myy = per_label(cy * cy) / area - my * my + 1.0 / 12.0
    mxy = per_label(cx * cy) / area - mx * my
    delta = ((mxx - myy) ** 2 + 4.0 * mxy * mxy).sqrt()
    major, minor = (8.0 * (mxx + myy + delta)).sqrt(), (8.0 * (mxx + myy - delta)).sqrt()
    per = _exact_perimeter(labels, n)
    grey = bgr[:, :, 2]
    return {"area": None, "perimeter": per, "major_axis": major, "minor_axis": minor,
            "eccentricity": (major * major - minor * minor).abs().sqrt() / major,
            "extent_ratio": area / ((b[2] - b[1] + 1) * (b[4] - b[3] + 1)),
            "circularity": 4.0 * 3.14159265359 * area / (per * per),
            "intensity": _exact_histogram(grey[ys, xs], lab, n),
            "gradient": _exact_histogram(_exact_gradient(grey)[ys, xs], lab, n)[:, [0, 3, 4, 5, 6, 7]]}


def exact(case, seed):
    """What run returns, in 64 bits and without this framework; None where the outputs are whole numbers or
    are the inputs' own values (the reconstructions select among them, the float one included)."""
    if case["kind"] == "hmin":
        state = prepare(case, seed)
        dist = [_exact_dist(m) for m in state["masks"]]
        return {"dist": dist, "hmin": [_exact_hmin(d, 1.0, c) for d, c in zip(dist, state["conns"])]}
    if case["kind"] == "features":
        return _exact_features(*_labelled(case["h"], case["w"], seed))
    return None
