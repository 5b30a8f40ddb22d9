"""The work that users of the Toeplitz-hashing engine have it do, as measurable cases.

Four forms of it, each through the public Python API (privacyamplification_amd.Engine):
  block   one block whose key and seed are already in device memory (block_device with a fresh
          seed, block_device_seeded with a resident one): what a front-end that receives into GPU
          memory calls per block;
  host    one block from and to host memory (amplify): the whole synchronous call;
  batch   many blocks of uneven length in one call (batch_device);
  serve   a filled input cache handed to the serving scheduler (serve_submit_many, serve_wait),
          pinned host buffers in and out.
Block lengths run from 2^10 to 2^29 bits (the reference's factor_exp range 10..27 and the two
lengths this engine adds), powers of two and ragged multiples of 32, m / n from 1/8 to 7/8, with and
without the key-rest XOR and compression.  Keys and seeds are uniformly random bits, as a QKD link
and its seed server deliver them.  Every output is the packed bit string, compared byte for byte.
"""
import ctypes
import math

import numpy as np
import torch

import privacyamplification_amd as P

XOR, COMPRESS = P.XOR_KEY_REST, P.COMPRESS
BOTH = XOR | COMPRESS


def _m(n, eighths):
    return max(32, n * eighths // 8 // 32 * 32)


def _block(name, n, m, static=False, flags=BOTH, kind="block"):
    return {"name": name, "kind": kind, "n": n, "m": m, "static": static, "flags": flags}


def listed():
    return [
        # the smallest blocks: short sifted keys of a slow link, one call each; latency is all
        _block("block_2^12", 1 << 12, _m(1 << 12, 3)),
        # a short block from and to host memory, one synchronous call: link bring-up, tests, tools
        _block("host_2^17", 1 << 17, _m(1 << 17, 3), kind="host"),
        # the mid-size block of the reference's speedtest range, fresh and resident seed
        _block("block_2^20", 1 << 20, _m(1 << 20, 3)),
        _block("block_2^20_static", 1 << 20, _m(1 << 20, 3), static=True),
        # a key of whatever length sifting left: not a power of two, low secret-key rate
        _block("block_ragged_3e6", 3000032, _m(3000032, 2)),
        # the plain product: no key-rest XOR and no compression (both frames zero); n/2 bits out
        _block("block_2^24_plain", 1 << 24, _m(1 << 24, 3), flags=0),
        # the headline block: the reference's largest and default length, fresh seed per block
        _block("block_2^27", 1 << 27, _m(1 << 27, 3)),
        # the same with a reused (resident) seed
        _block("block_2^27_static", 1 << 27, _m(1 << 27, 3), static=True),
        # the largest length: beyond the reference's, for finite-size effects of long links
        _block("block_2^29", 1 << 29, _m(1 << 29, 3)),
        # the 256 uneven blocks of the benchmark: several links' blocks gathered into one call,
        # graph replayed and launch shapes tuned, as a program that repeats a shape asks for
        {"name": "batch_mix_256", "kind": "batch", "count": 256, "lo": 16.0, "hi": 25.0, "mix": 1, "static": False,
         "flags": BOTH, "options": P.BATCH_GRAPH | P.BATCH_TUNE},
        # many short blocks on one resident seed, launched directly
        {"name": "batch_short_64_static", "kind": "batch", "count": 64, "lo": 18.0, "hi": 18.0, "mix": 2,
         "static": True, "flags": BOTH, "options": 0},
        # a full input cache of a key server: 64 blocks, three in four on resident seeds
        {"name": "serve_64", "kind": "serve", "count": 64, "lo": 16.0, "hi": 24.0, "mix": 3},
    ]


def draw(rng):
    kind = rng.choices(["block", "host", "batch", "serve"], [10, 2, 4, 2])[0]
    if kind in ("block", "host"):
        u = rng.uniform(10.0, 28.0 if kind == "block" else 24.0)
        n = 1 << round(u) if rng.random() < 0.5 else max(1024, int(2.0 ** u) // 32 * 32)
        pow2 = n & (n - 1) == 0
        m = min(n - 32, max(32, int(n * rng.uniform(0.125, 0.875)) // 32 * 32))
        flags = BOTH if rng.random() < 0.6 else rng.choice([0, XOR, COMPRESS] if pow2 else [COMPRESS])
        return {"kind": kind, "n": n, "m": m, "static": kind == "block" and rng.random() < 0.4, "flags": flags}
    lo = rng.uniform(12.0, 18.0)
    hi = rng.uniform(lo, 24.0)
    mean = 2.0 ** lo if hi - lo < 1e-3 else (2.0 ** hi - 2.0 ** lo) / ((hi - lo) * math.log(2.0))
    most = min(256, int(1.0e9 / mean)) if kind == "batch" else min(96, int(2.5e8 / mean))
    count = max(2, min(most, round(2.0 ** rng.uniform(2.0, 8.0))))
    case = {"kind": kind, "count": count, "lo": lo, "hi": hi, "mix": rng.randrange(1 << 30)}
    if kind == "batch":
        case.update(static=rng.random() < 0.3, flags=rng.choice([BOTH, BOTH, COMPRESS]),
                    options=rng.choice([0, P.BATCH_GRAPH, P.BATCH_GRAPH | P.BATCH_TUNE]))
    return case


def _shapes(case):
    """(n, m) of each block: n = 32 floor(2^U / 32), U uniform in [lo, hi], m / n in eighths."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for _ in range(case["count"]):
        n = max(64, int(2.0 ** rng.uniform(case["lo"], case["hi"])) // 32 * 32)
        out.append((n, min(n - 32, _m(n, int(rng.integers(1, 5))))))
    return out


def _roles(case):
    """Per block of a serve case its resident seed stream, or -1 for a fresh seed; and the streams'
    shapes, each that of the first block in it."""
    shapes = _shapes(case)
    rng = np.random.default_rng(case["mix"] + 1)
    firsts = [int(i) for i in rng.choice(len(shapes), size=min(4, len(shapes)), replace=False)]
    role = [int(rng.integers(0, len(firsts))) if rng.random() < 0.75 else -1 for _ in shapes]
    shapes = [shapes[firsts[r]] if r >= 0 else sh for sh, r in zip(shapes, role)]
    return shapes, role, [shapes_of for shapes_of in (_shapes(case)[i] for i in firsts)]


# ------------------------------------------------------------------ inputs ----
def _key_words(n):
    return n // 32 + 1


def _spans(sizes, align):
    """Start of each of `sizes` in one buffer, each aligned, and the buffer's size."""
    offs, at = [], 0
    for s in sizes:
        offs.append(at)
        at += (s + align - 1) // align * align
    return offs, max(at, align)


def _words_dev(count, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randint(-(1 << 31), 1 << 31, (count,), dtype=torch.int32, device="cuda", generator=g)


def _words_host(count, seed):
    return np.random.default_rng(seed).integers(0, 1 << 32, count, dtype=np.uint32)


def _inputs(case, seed):
    """The random words of a case: block / host / batch: (keys, seeds), serve: (keys, fresh seeds,
    resident seeds); each a list of arrays.  Used by prepare and by exact."""
    kind = case["kind"]
    if kind == "block":
        n = case["n"]
        keys = [_words_dev(_key_words(n), 2 * seed + 1)]
        seeds = [_words_host(n // 32, 2 * seed + 2) if case["static"] else _words_dev(n // 32, 2 * seed + 2)]
        return keys, seeds
    if kind == "host":
        n = case["n"]
        return [_words_host(_key_words(n), 2 * seed + 1)], [_words_host(n // 32, 2 * seed + 2)]
    if kind == "batch":
        shapes = _shapes(case)
        ko, kw = _spans([_key_words(n) for n, _ in shapes], 64)
        k = _words_dev(kw, 2 * seed + 1)
        keys = [k[o: o + _key_words(n)] for o, (n, _) in zip(ko, shapes)]
        if case["static"]:  # one resident seed per length
            seeds = {n: _words_host(n // 32, 2 * seed + 2 + n) for n, _ in shapes}
            return keys, [seeds[n] for n, _ in shapes]
        so, sw = _spans([n // 32 for n, _ in shapes], 64)
        s = _words_dev(sw, 2 * seed + 2)
        return keys, [s[o: o + n // 32] for o, (n, _) in zip(so, shapes)]
    shapes, role, streams = _roles(case)
    ko, kw = _spans([_key_words(n) for n, _ in shapes], 64)
    k = _words_host(kw, 2 * seed + 1)
    so, sw = _spans([n // 32 if r < 0 else 0 for (n, _), r in zip(shapes, role)], 64)
    s = _words_host(sw, 2 * seed + 2)
    resident = [_words_host(n // 32, 2 * seed + 3 + 1000 * i) for i, (n, _) in enumerate(streams)]
    return ([k[o: o + _key_words(n)] for o, (n, _) in zip(ko, shapes)],
            [s[o: o + n // 32] if r < 0 else None for o, (n, _), r in zip(so, shapes, role)], resident)


# ------------------------------------------------------------------ the program ----
_engines = {}


def _engine(serving=False):
    """One engine per process (a second one runs the server), as a front-end keeps it."""
    if serving not in _engines:
        eng = P.Engine(max_n_log2=29, hbm_budget_bytes=160 << 30)
        if serving:
            eng.serve_start(slots=3, max_batch=256, hbm_budget_bytes=64 * 10 ** 9)
        _engines[serving] = (eng, torch.cuda.Stream())
    return _engines[serving]


class _Prepared:
    """A prepared case: its inputs, its output buffer and its resident seeds (dropped with it)."""

    def __init__(self, case, seed):
        self.case = case
        self.eng, self.stream = _engine(case["kind"] == "serve")
        self.sids = []
        getattr(self, "_" + case["kind"])(case, seed)
        torch.cuda.synchronize()

    def __del__(self):
        try:
            for sid in set(self.sids):
                self.eng.seed_drop(sid)
        except Exception:
            pass

    def _block(self, case, seed):
        n, m = case["n"], case["m"]
        (self.key,), (s,) = _inputs(case, seed)
        if case["static"]:
            self.sids = [self.eng.seed_put(s, n, m)]
        else:
            self.seed = s
        self.out = torch.zeros(P.out_bytes(n, m, case["flags"] & COMPRESS), dtype=torch.uint8, device="cuda")

    def _host(self, case, seed):
        (self.key,), (self.seed,) = _inputs(case, seed)

    def _batch(self, case, seed):
        self.shapes = _shapes(case)
        self.keys, self.seeds = _inputs(case, seed)
        oo, ob = _spans([P.out_bytes(n, m, case["flags"] & COMPRESS) for n, m in self.shapes], 256)
        self.out = torch.zeros(ob, dtype=torch.uint8, device="cuda")
        if case["static"]:
            by_n = {}
            for (n, m), s in zip(self.shapes, self.seeds):
                # a resident seed serves one (n, m) where n is not a power of two
                if (n, m) not in by_n:
                    by_n[(n, m)] = self.eng.seed_put(s, n, m)
            self.sids = [by_n[sh] for sh in self.shapes]
        self.blocks = (P.PaBlock * len(self.shapes))()
        for i, (n, m) in enumerate(self.shapes):
            b = self.blocks[i]
            b.key, b.n, b.m, b.flags = self.keys[i].data_ptr(), n, m, case["flags"]
            b.out = self.out.data_ptr() + oo[i]
            if case["static"]:
                b.seed_id = self.sids[i]
            else:
                b.seed = self.seeds[i].data_ptr()

    def _serve(self, case, seed):
        shapes, role, streams = _roles(case)
        keys, fresh, resident = _inputs(case, seed)
        self.sids = [self.eng.seed_put(s, n, m) for s, (n, m) in zip(resident, streams)]
        # the input and output caches: one pinned buffer each
        ko, kw = _spans([k.size for k in keys], 64)
        so, sw = _spans([0 if s is None else s.size for s in fresh], 64)
        oo, ob = _spans([m // 8 for _, m in shapes], 256)
        kbuf, sbuf = self.eng.host_empty(kw, np.uint32), self.eng.host_empty(sw, np.uint32)
        self.out = self.eng.host_empty(ob, np.uint8)
        self.out[:] = 0
        self.requests = []
        for i, (n, m) in enumerate(shapes):
            k = kbuf[ko[i]: ko[i] + keys[i].size]
            k[:] = keys[i]
            s = None
            if fresh[i] is not None:
                s = sbuf[so[i]: so[i] + fresh[i].size]
                s[:] = fresh[i]
            o = self.out[oo[i]: oo[i] + m // 8]
            self.requests.append((k, n, m, o, s, self.sids[role[i]] if role[i] >= 0 else 0))


def prepare(case, seed):
    return _Prepared(case, seed)


def run(state):
    case, eng, kind = state.case, state.eng, state.case["kind"]
    if kind == "block":
        n, m, flags, sptr = case["n"], case["m"], case["flags"], state.stream.cuda_stream
        if case["static"]:
            eng.block_device_seeded(state.key.data_ptr(), state.sids[0], n, m, flags, state.out.data_ptr(), sptr)
        else:
            eng.block_device(state.key.data_ptr(), state.seed.data_ptr(), n, m, flags, state.out.data_ptr(), sptr)
        return state.out
    if kind == "host":
        return eng.amplify(state.key, state.seed, case["n"], case["m"], bool(case["flags"] & XOR),
                           bool(case["flags"] & COMPRESS))
    if kind == "batch":
        eng.batch_device(state.blocks, case["options"], state.stream.cuda_stream)
        return state.out
    for ticket in eng.serve_submit_many(state.requests):
        eng.serve_wait(ticket)
    return state.out


# ------------------------------------------------------------------ what it cannot do without ----
def _work_block(n, m, flags, static):
    """Inputs read once and outputs written once (a resident seed is its spectrum of n/2 + 1 complex
    FP32 values); the operations are those of two real transforms and a pointwise product (three
    transforms with a fresh seed) of the padded length, 2.5 L log2 L each."""
    length = 1 << (n - 1).bit_length()
    bits = m if flags & COMPRESS else n // 2
    key = n if flags & XOR else n - m
    nbytes = key / 8 + bits / 8 + (4 * length if static else n / 8)
    return nbytes, (2 if static else 3) * 2.5 * length * math.log2(length) + 3 * length


def work(case):
    if case["kind"] in ("block", "host"):
        parts = [_work_block(case["n"], case["m"], case["flags"], case["static"])]
    elif case["kind"] == "batch":
        parts = [_work_block(n, m, case["flags"], case["static"]) for n, m in _shapes(case)]
    else:
        shapes, role, _ = _roles(case)
        parts = [_work_block(n, m, BOTH, r >= 0) for (n, m), r in zip(shapes, role)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# ------------------------------------------------------------------ exact outputs ----
def _bits(words):
    """The bits of RefBits words, in stream order, as a float64 tensor on the GPU."""
    w = words if isinstance(words, torch.Tensor) else torch.from_numpy(np.ascontiguousarray(words).view(np.int32))
    sh = torch.arange(31, -1, -1, dtype=torch.int32, device="cuda")
    return ((w.cuda()[:, None] >> sh) & 1).reshape(-1).to(torch.float64)


def _exact_block(key, seed, n, m, flags):
    """amp_out by a float64 convolution: y[p] = sum_{j <= h} x[j] s[(p - j) mod n], h = n - m, mod 2,
    xor key bit h + 1 + p where p < m and the key rest is wanted."""
    h, length = n - m, 1 << (n - 1).bit_length()
    kb = _bits(key)
    x = torch.zeros(length, dtype=torch.float64, device="cuda")
    x[: h + 1] = kb[: h + 1]
    t = torch.zeros(length, dtype=torch.float64, device="cuda")
    t[:n] = torch.roll(_bits(seed), h)  # t[i] = s[(i - h) mod n]: y[p] is at index p + h
    conv = torch.fft.irfft(torch.fft.rfft(x) * torch.fft.rfft(t), n=length)
    bits = m if flags & COMPRESS else n // 2
    y = torch.round(torch.roll(conv, -h)[:bits]).to(torch.int64) & 1
    if flags & XOR:
        k = min(bits, m)
        y[:k] ^= kb[h + 1: h + 1 + k].to(torch.int64)
    place = 1 << torch.arange(7, -1, -1, dtype=torch.int64, device="cuda")
    return (y.reshape(-1, 8) * place).sum(1).to(torch.uint8)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("block", "host"):
        if case["n"] > 1 << 27:
            return None
        (key,), (s,) = _inputs(case, seed)
        y = _exact_block(key, s, case["n"], case["m"], case["flags"])
        return y.cpu().numpy() if kind == "host" else y
    if kind == "batch":
        shapes, (keys, seeds), flags = _shapes(case), _inputs(case, seed), case["flags"]
        if case["static"]:  # blocks of one length share the resident seed of the first of them
            first = {}
            seeds = [first.setdefault(sh, s) for sh, s in zip(shapes, seeds)]
    else:
        shapes, role, _ = _roles(case)
        keys, fresh, resident = _inputs(case, seed)
        seeds, flags = [resident[r] if r >= 0 else f for f, r in zip(fresh, role)], BOTH
    parts = [_exact_block(k, s, n, m, flags) for k, s, (n, m) in zip(keys, seeds, shapes)]
    oo, ob = _spans([p.numel() for p in parts], 256)
    out = torch.zeros(ob, dtype=torch.uint8, device="cuda")
    for o, p in zip(oo, parts):
        out[o: o + p.numel()] = p
    return out if kind == "batch" else out.cpu().numpy()
