"""The work a user of this library has it do, as measurable cases.

The library encodes video frames: the device-resident step of one frame or of a
batch of uneven streams, the allocation-free single-frame call, the learned
search and the training and forward pass of its networks, and the host-buffer
encoder with its stream writer and reader.  Sizes, search areas and thresholds
are those of mptc_amd/workloads.py and bench.py or generic ones; frames are a
colour gradient with moving rectangles and noise, as that module's generator
draws them, made on the GPU.

Device buffers are torch tensors.  torch is imported before the library, so the
process has the one HIP runtime that torch brings.
"""
from __future__ import annotations

import random

import numpy as np
import torch

from mptc_amd import codec, lib

DEV = "cuda"
STREAM_SIZES = [(640, 360), (1280, 720), (1920, 1080), (3840, 2160)]


def listed():
    return [
        # a thumbnail or atlas tile: the smallest call, all launches and latency
        dict(name="tile_64_s8_t0", kind="frame", w=64, h=64, S=8, thr=0, intra=False, rects=4),
        # a serving loop that may not allocate: one 720p frame, no context
        dict(name="noalloc_720p_s8_t0", kind="noalloc", w=1280, h=720, S=8, thr=0, intra=False, rects=32),
        # the 1080p sequence at threshold 0: seven of its eight frames are inter
        dict(name="hd_s8_t0_inter", kind="frame", w=1920, h=1080, S=8, thr=0, intra=False, rects=32),
        # the same sequence at threshold 8, its intra-refresh frame: long reuse chains
        dict(name="hd_s8_t8_intra", kind="frame", w=1920, h=1080, S=8, thr=8, intra=True, rects=32),
        # the 64 x 64 block window: a 4K frame at threshold 0 and a 1080p refresh frame at a rate-leaning threshold
        dict(name="uhd_s32_t0_inter", kind="frame", w=3840, h=2160, S=32, thr=0, intra=False, rects=32),
        dict(name="hd_s32_t32_intra", kind="frame", w=1920, h=1080, S=32, thr=32, intra=True, rects=32),
        # a server's step: the next frame of twelve uneven streams in one call
        dict(name="streams12_s8_t8_inter", kind="batch", n=12, S=8, thr=8, intra=False, rects=32, scale=4),
        # the learned search of the 1080p sequence: top-4 proposals, similarity scores on the inter ranking
        dict(name="learned_hd_k4_inter", kind="learned", w=1920, h=1080, S=8, thr=0, k=4, intra=False, rects=32),
        # training of a proposal network: weights in, weights out
        dict(name="train_b4096_x200", kind="train", pairs=131072, batch=4096, steps=200, net=0),
        # a network's outputs for every block of a 1080p frame
        dict(name="forward_hd", kind="forward", rows=129600, net=0),
        # the encoder program on host frames: fit, re-encode and .mptc stream of a short clip
        dict(name="clip_256_s8_t8_write", kind="write", w=256, h=256, S=8, thr=8, frames=8, interval=8, rects=4),
        # the player's side: a stream decoded to blocks
        dict(name="clip_512_s8_t8_read", kind="read", w=512, h=256, S=8, thr=8, frames=8, interval=4, rects=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _frame_dims(rng, lo, hi):
    """A block grid of lo..hi blocks, spread over the logarithm, of ordinary aspect; any width, odd grids included."""
    nb = _log_int(rng, lo, hi)
    bw = max(4, int(round((nb * rng.uniform(0.8, 2.4)) ** 0.5)))
    return 4 * bw, 4 * max(4, nb // bw)


def draw(rng):
    kind = rng.choice(["frame"] * 6 + ["batch", "noalloc", "learned", "train", "forward", "write", "read"])
    thr = rng.choice([0, 0, 0, 2, 4, 8, 8, 16, 32, 128])
    intra = rng.random() < 0.4
    if kind == "frame":
        S = rng.choice([8, 8, 8, 16, 32, rng.randint(1, 63)])
        # window positions per frame at most the 1080p, S = 32 frame's (long chains cost most there)
        most = min(518400, int(5.3e8 / (4 * S * S)))
        w, h = _frame_dims(rng, 64, max(most, 256))
        return dict(kind=kind, w=w, h=h, S=S, thr=thr, intra=intra, rects=rng.choice([4, 32]))
    if kind == "noalloc":
        w, h = _frame_dims(rng, 64, 60000)
        return dict(kind=kind, w=w, h=h, S=rng.randint(1, 8), thr=thr, intra=intra, rects=rng.choice([4, 32]))
    if kind == "batch":
        return dict(kind=kind, n=rng.randint(2, 12), S=rng.choice([4, 8]), thr=rng.choice([0, 2, 8, 8]), intra=intra, rects=32,
                    scale=rng.randint(1, 4))
    if kind == "learned":
        w, h = _frame_dims(rng, 1024, 230400)
        return dict(kind=kind, w=w, h=h, S=8, thr=rng.choice([0, 0, 8]), k=rng.choice([1, 2, 4, 8, 16]), intra=intra, rects=32)
    if kind == "train":
        batch = rng.choice([1024, 2048, 4096, 4096, rng.randint(500, 5000)])
        return dict(kind=kind, pairs=batch * rng.randint(2, 40) + rng.randint(0, 999), batch=batch, steps=rng.randint(20, 300),
                    net=rng.randint(0, 1))
    if kind == "forward":
        return dict(kind=kind, rows=_log_int(rng, 256, 400000), net=rng.randint(0, 1))
    # streams need a block grid of multiples of 64
    w, h = rng.choice([(256, 256), (512, 256), (512, 512), (768, 256)])
    n = rng.choice([2, 4, 8])
    return dict(kind=kind, w=w, h=h, S=rng.choice([8, 8, 16]), thr=rng.choice([0, 4, 8]), frames=n,
                interval=rng.choice([x for x in (2, 4, 8) if x <= n]), rects=rng.choice([4, 8]))


# ---- inputs -----------------------------------------------------------------
def _video(w, h, rects, seed, first, n):
    """Frames first .. first + n - 1 of a seeded clip, uint8 n x h x w x 3 on the GPU."""
    r = random.Random(seed * 7919 + w * 31 + h)
    base = torch.tensor([[r.randrange(256), r.randrange(-128, 129), r.randrange(-128, 129)] for _ in range(3)], device=DEV)
    y = torch.arange(h, device=DEV).view(h, 1, 1)
    x = torch.arange(w, device=DEV).view(1, w, 1)
    grad = base[:, 0] + torch.div(base[:, 1] * x, w, rounding_mode="trunc") + torch.div(base[:, 2] * y, h, rounding_mode="trunc")
    grad = grad.clamp_(0, 255).to(torch.uint8)
    boxes = []
    for _ in range(rects):
        boxes.append((r.randint(max(1, w // 16), max(1, w // 4)), r.randint(max(1, h // 16), max(1, h // 4)), r.randrange(w),
                      r.randrange(h), [r.randrange(256) for _ in range(3)], r.randint(-4, 4), r.randint(-4, 4)))
    gen = torch.Generator(device=DEV).manual_seed(seed)
    out = torch.empty((n, h, w, 3), dtype=torch.uint8, device=DEV)
    for t in range(first + n):
        noise = torch.randint(-8, 9, (h, w, 3), generator=gen, dtype=torch.int16, device=DEV)
        if t < first:
            continue
        f = grad.to(torch.int16)
        for rw, rh, x0, y0, col, vx, vy in boxes:
            ys = (torch.arange(rh, device=DEV) + y0 + vy * t) % h
            xs = (torch.arange(rw, device=DEV) + x0 + vx * t) % w
            f[ys[:, None], xs[None, :]] = torch.tensor(col, dtype=torch.int16, device=DEV)
        out[t - first] = (f + noise).clamp_(0, 255).to(torch.uint8)
    return out


def _outputs(nb):
    return dict(phys=torch.zeros(nb, dtype=torch.int64, device=DEV), motion=torch.zeros(2 * nb, dtype=torch.uint8, device=DEV),
                unique=torch.zeros(nb, dtype=torch.int32, device=DEV), n_unique=torch.zeros(1, dtype=torch.int32, device=DEV),
                eps=torch.zeros(6 * nb, dtype=torch.uint8, device=DEV), kind=torch.zeros(nb, dtype=torch.uint8, device=DEV))


def _blocks(w, h):
    return (w // 4) * (h // 4)


def _job(rgb, ref, o, w, h, intra):
    return dict(d_rgb=rgb, width=w, height=h, is_intra=intra, d_ref=ref, d_phys=o["phys"], d_motion=o["motion"],
                d_unique=o["unique"], d_n_unique=o["n_unique"], d_eps=o["eps"], d_kind=o["kind"])


def _batch_sizes(case):
    """Uneven streams as evenly spread over the first `scale` stream sizes as they come."""
    return [STREAM_SIZES[i * case["scale"] // case["n"]] for i in range(case["n"])]


def _weights(seed):
    """A network's parameters at the scale training leaves them: He-normal hidden layers, a small logit layer."""
    r = np.random.default_rng(seed)
    w = [r.normal(0, (2 / 48) ** 0.5, 48 * 256), r.normal(0, 0.05, 256), r.normal(0, (2 / 256) ** 0.5, 256 * 256),
         r.normal(0, 0.05, 256), r.normal(0, 0.3 * (1 / 256) ** 0.5, 256 * 262), r.normal(0, 0.05, 262)]
    return np.concatenate(w).astype(np.float32)


def _nearest(net):
    """Base scores that rank near offsets first."""
    L = np.arange(256)
    dx, dy = L % 16 - 8, (L // 16 - 8 if net == 0 else L // 16)
    return (-(dx * dx + dy * dy) - 1e-3 * L).astype(np.float32)


def _pixels(n, seed):
    """n blocks of 48 bytes cut from a seeded clip's frames."""
    w = 1920
    h = 4 * max(1, -(-4 * n // w))
    f = _video(w, h, 32, seed, 0, 1)[0]
    px = f.view(h // 4, 4, w // 4, 4, 3).permute(0, 2, 1, 3, 4).reshape(-1, 48)
    return px[:n].contiguous()


# ---- prepare and run ----------------------------------------------------------
def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_frame(case, seed):
    w, h = case["w"], case["h"]
    rgb = _video(w, h, case["rects"], seed, 0, 2)
    enc = lib.Encoder(w, h, case["S"], case["thr"])
    return _frame_state(case, enc, rgb)


def _frame_state(case, enc, rgb):
    w, h, nb = case["w"], case["h"], _blocks(case["w"], case["h"])
    stream = torch.cuda.Stream()
    ref = None
    torch.cuda.synchronize()
    if not case["intra"]:  # the previous frame, encoded by the same program
        o = _outputs(nb)
        torch.cuda.synchronize()
        enc.encode_frame_device(rgb[0], w, h, True, None, o["phys"], o["motion"], o["unique"], o["n_unique"], o["eps"],
                                o["kind"], stream=stream.cuda_stream)
        ref = o["phys"]
    return dict(run=_run_frame, enc=enc, stream=stream, rgb=rgb[1], ref=ref, out=_outputs(nb), w=w, h=h, intra=case["intra"])


def _run_frame(s):
    o = s["out"]
    s["enc"].encode_frame_device(s["rgb"], s["w"], s["h"], s["intra"], s["ref"], o["phys"], o["motion"], o["unique"],
                                 o["n_unique"], o["eps"], o["kind"], stream=s["stream"].cuda_stream)
    return o


def _prepare_noalloc(case, seed):
    w, h, nb = case["w"], case["h"], _blocks(case["w"], case["h"])
    rgb = _video(w, h, case["rects"], seed, 0, 2)
    s = dict(run=_run_noalloc, rgb=rgb[1], ref=None, w=w, h=h, S=case["S"], thr=case["thr"], intra=case["intra"],
             stream=torch.cuda.Stream())
    torch.cuda.synchronize()
    if not case["intra"]:
        o = _run_noalloc(dict(s, rgb=rgb[0], intra=True, out=_outputs(nb)))
        s["ref"] = o["phys"]
    s["out"] = _outputs(nb)
    return s


def _run_noalloc(s):
    o = s["out"]
    lib.encode_frame_noalloc(0, s["rgb"], s["w"], s["h"], s["S"], s["thr"], s["intra"], s["ref"], o["phys"], o["motion"],
                             o["unique"], o["n_unique"], o["eps"], o["kind"], stream=s["stream"].cuda_stream)
    return o


def _prepare_batch(case, seed):
    sizes = _batch_sizes(case)
    enc = lib.Encoder(max(w for w, _ in sizes), max(h for _, h in sizes), case["S"], case["thr"], max_batch_frames=len(sizes),
                      max_batch_blocks=sum(_blocks(w, h) for w, h in sizes))
    stream = torch.cuda.Stream()
    clips = [_video(w, h, case["rects"], seed * 64 + i, 0, 2) for i, (w, h) in enumerate(sizes)]
    first = [_outputs(_blocks(w, h)) for w, h in sizes]
    out = [_outputs(_blocks(w, h)) for w, h in sizes]
    torch.cuda.synchronize()
    if not case["intra"]:
        enc.encode_batch_device([_job(c[0], None, o, w, h, True) for c, o, (w, h) in zip(clips, first, sizes)],
                                stream=stream.cuda_stream)
    jobs = [_job(c[1], None if case["intra"] else f["phys"], o, w, h, case["intra"])
            for c, f, o, (w, h) in zip(clips, first, out, sizes)]
    return dict(run=_run_batch, enc=enc, stream=stream, jobs=jobs, out=out)


def _run_batch(s):
    s["enc"].encode_batch_device(s["jobs"], stream=s["stream"].cuda_stream)
    keys = ("phys", "motion", "unique", "n_unique", "eps")  # the kinds are written too; 64 outputs are the most
    return [{k: o[k] for k in keys} for o in s["out"]]


def _prepare_learned(case, seed):
    w, h = case["w"], case["h"]
    rgb = _video(w, h, case["rects"], seed, 0, 2)
    enc = lib.Encoder(w, h, case["S"], case["thr"])
    for net in (lib.NET_INTER, lib.NET_INTRA):
        enc.net_set_params(net, _weights(100 * seed + net))
        enc.net_set_base(net, 0.25 * _nearest(net))
    # log acceptance rate by differing indices: near words pass more often
    enc.net_set_similarity(lib.NET_INTER, (-1.0 - 0.35 * np.arange(lib.SIM_BINS)).astype(np.float32))
    enc.set_search_mode(lib.SEARCH_LEARNED, case["k"])
    return _frame_state(case, enc, rgb)


def _prepare_train(case, seed):
    n = case["pairs"]
    gen = torch.Generator(device=DEV).manual_seed(seed)
    px = _pixels(n, seed)
    # target sets: one to a few dozen of 256 offsets, most of them few; endpoints near the block's own extremes
    keep = torch.rand((n, 1), generator=gen, device=DEV) ** 4 * 0.12
    bits = torch.rand((n, 256), generator=gen, device=DEV) < keep
    bits[torch.arange(n, device=DEV), torch.randint(0, 256, (n,), generator=gen, device=DEV)] = True
    place = torch.tensor([1 << i for i in range(32)], dtype=torch.int64, device=DEV)
    words = (bits.view(n, 8, 32).to(torch.int64) * place).sum(2)
    target = torch.where(words >= 1 << 31, words - (1 << 32), words).to(torch.int32).contiguous()
    rgb = px.view(n, 16, 3)
    eps = torch.cat([rgb.amax(1), rgb.amin(1)], 1).contiguous()
    enc = lib.Encoder(64, 64, 8, 0)
    enc.net_set_base(case["net"], 0.25 * _nearest(case["net"]))
    return dict(run=_run_train, enc=enc, net=case["net"], px=px, target=target, eps=eps, n=n, batch=case["batch"],
                steps=case["steps"], start=lib.zero_logit_layer(_weights(100 * seed + 7)))


def _run_train(s):
    e = s["enc"]
    e.net_set_params(s["net"], s["start"])
    losses = e.net_train(s["net"], s["px"], s["target"], s["eps"], s["n"], batch=s["batch"], steps=s["steps"], lr=2e-3,
                         seed_weight=1.0, seed=7, lr_final=1e-4)
    return dict(losses=losses, params=e.net_params(s["net"]))


def _prepare_forward(case, seed):
    enc = lib.Encoder(64, 64, 8, 0)
    enc.net_set_params(case["net"], _weights(100 * seed + 3))
    enc.net_set_base(case["net"], 0.25 * _nearest(case["net"]))
    out = torch.zeros((case["rows"], lib.NET_OUT), dtype=torch.float32, device=DEV)
    return dict(run=_run_forward, enc=enc, net=case["net"], px=_pixels(case["rows"], seed), rows=case["rows"], out=out)


def _run_forward(s):
    s["enc"].net_forward(s["net"], s["px"], s["rows"], s["out"])
    return s["out"]


def _prepare_write(case, seed):
    frames = _video(case["w"], case["h"], case["rects"], seed, 0, case["frames"]).cpu().numpy()
    return dict(run=_run_write, enc=lib.Encoder(case["w"], case["h"], case["S"], case["thr"]), clip=frames, w=case["w"],
                h=case["h"], S=case["S"], interval=case["interval"])


def _padded(a, n):
    """The array in one of n elements, zeros behind it, and its own length."""
    out = np.zeros(n, a.dtype)
    out[:len(a)] = a
    return out, len(a)


def _run_write(s):
    coded = s["enc"].encode_sequence(s["clip"], s["interval"])
    data = codec.write_stream(coded, s["w"], s["h"], s["S"], s["interval"])
    return dict(stream=_padded(np.frombuffer(data, np.uint8), s["clip"].size), phys=np.stack([f["phys"] for f in coded]).view(np.int64),
                motion=np.stack([f["motion"] for f in coded]))


def _prepare_read(case, seed):
    s = _prepare_write(case, seed)
    coded = s["enc"].encode_sequence(s["clip"], s["interval"])
    return dict(run=_run_read, data=codec.write_stream(coded, s["w"], s["h"], s["S"], s["interval"]))


def _run_read(s):
    info, frames = codec.read_stream(s["data"])
    return dict(info=info, phys=np.stack([f["phys"] for f in frames]).view(np.int64), motion=np.stack([f["motion"] for f in frames]),
                unique=[_padded(f["unique"].view(np.int32), len(f["phys"])) for f in frames])


# ---- what a pass cannot do without ---------------------------------------------
# Lane operations of one 4x4 block's endpoint fit and of one exact candidate
# evaluation; a frame's search cannot decide without each window position's
# word being tried or bounded, and the cheapest bound is a 16-pixel scatter.
_FIT, _BOUND = 2000, 78
_ROW_FLOPS = 2 * (48 * 256 + 256 * 256 + 256 * 262)


def _frame_work(w, h, S, intra):
    nb = _blocks(w, h)
    window = (2 * S) * (2 * S) - S if intra else (2 * S) * (2 * S)
    return nb * (48 + (0 if intra else 8) + 8 + 2 + 6 + 1), nb * (_FIT + _BOUND * window)


def work(case):
    k = case["kind"]
    if k in ("frame", "noalloc"):
        b, f = _frame_work(case["w"], case["h"], case["S"], case["intra"])
    elif k == "batch":
        each = [_frame_work(w, h, case["S"], case["intra"]) for w, h in _batch_sizes(case)]
        b, f = sum(x[0] for x in each), sum(x[1] for x in each)
    elif k == "learned":
        nb = _blocks(case["w"], case["h"])
        nets = 1 if case["intra"] else 2
        b, f = _frame_work(case["w"], case["h"], 1, case["intra"])[0], nb * (_FIT + nets * (_ROW_FLOPS + 600 * case["k"]))
    elif k == "train":
        rows = case["batch"] * case["steps"]
        b, f = min(case["pairs"], rows) * (48 + 32 + 6) + 2 * 4 * lib.NET_PARAMS, 3 * rows * _ROW_FLOPS
    elif k == "forward":
        b, f = case["rows"] * (48 + 4 * lib.NET_OUT), case["rows"] * _ROW_FLOPS
    else:  # the first frame of every interval is intra
        n = case["frames"]
        each = [_frame_work(case["w"], case["h"], case["S"], i % case["interval"] == 0) for i in range(n)]
        b = sum(x[0] for x in each)
        f = sum(x[1] for x in each) if k == "write" else 100 * n * _blocks(case["w"], case["h"])
    return {"bytes": b, "flops": f}


def exact(case, seed):
    """The network's outputs in 64 bits.  Every other output is whole numbers
    and bytes, or (training) follows the library's own shuffle of the pairs."""
    if case["kind"] != "forward":
        return None
    p = torch.from_numpy(_weights(100 * seed + 3)).to(DEV, torch.float64)
    parts = torch.split(p, [48 * 256, 256, 256 * 256, 256, 256 * 262, 262])
    x = _pixels(case["rows"], seed).to(torch.float64) / 255.0
    x = torch.relu(x @ parts[0].view(48, 256) + parts[1])
    x = torch.relu(x @ parts[2].view(256, 256) + parts[3])
    y = x @ parts[4].view(256, 262) + parts[5]
    y[:, :256] += torch.from_numpy(0.25 * _nearest(case["net"])).to(DEV, torch.float64)
    return y
