"""The work that a user of this library has it do, as cases that can be timed: one dense product, the dense half of a
decode step, single MoE layers, stacks of them with and without the hyper-connection, a ragged step cut by the planner,
and ragged batches through the packing path up to a prefill segment.

A case is a dict of plain values; "kind" says which of the paths below it takes:
  matvec  one quantized matrix (N rows of K values, ggml type fmt) times nb activations
  dense   per layer q / k / v / indexer projections in one launch and an output projection, then the vocabulary projection
  stack   MoE layers one after the other over resident weights; layers = 1 with host = True is a caller that keeps its
          activations, logits and selection in ordinary buffers, as the reference's engine does
  hyper   hyper-connection -> MoE layer, layer after layer
  vstep   a step of several conversations with a few rows each, cut into groups by the planner
  pack    rows of many tokens with known routing through count -> plan -> scatter -> grouped products -> combine
Shapes are those of the benchmark (D = 2048, I = 512, 512 experts, top-10), of the reference model's own layer (D = 2560,
I = 640) and of the tests (fewer experts, D = 1024, I = 256)."""
import ctypes as C
import math

import numpy as np
import torch

import qwental_amd as q
from qwental_amd import synth
from qwental_amd.gpu import Buf, QwBuf, QwHyperW, QwMoeLayer

# ggml types: 1 F16, 8 Q8_0, 12 Q4_K, 14 Q6_K, 20 IQ4_NL, 21 IQ3_S, 23 IQ4_XS, 30 BF16
# layer recipes: (routed gate and up, routed down, shared gate, shared up, shared down)
RECIPES = {
    "iq3_s": (21, 21, 21, 21, 21),   # the benchmark's layer; every fourth one has its shared expert in Q8_0
    "iq4_nl": (21, 20, 12, 23, 20),  # the reference model's own layer
    "q4_k": (12, 14, 12, 12, 14),    # the common mix of Q4_K with Q6_K down rows
    "q8_0": (8, 8, 8, 8, 8),
}
DENSE = ((12, 2), (12, 0.25), (14, 0.25), (30, 0.0625))  # q, k, v, indexer: type and rows as a share of K (4096, 512, 512, 128 at K = 2048)


def listed():
    moe = {"D": 2048, "I": 512, "E": 512, "topk": 10, "router": 1}
    return [
        # the smallest call: one projection for one token (BASELINE's first configuration)
        {"name": "matvec_iq3_s_b1", "kind": "matvec", "fmt": 21, "N": 4096, "K": 2048, "nb": 1},
        # a projection of odd size for a few tokens
        {"name": "matvec_q8_0_b7", "kind": "matvec", "fmt": 8, "N": 5127, "K": 2560, "nb": 7},
        # the dense half of a decode step of four conversations, with the vocabulary at its end
        {"name": "dense_step_b4", "kind": "dense", "layers": 12, "K": 2048, "ofmt": 8, "vocab": 131072, "nb": 4},
        # one layer called by itself for two tokens (a draft of one beside the last token), everything visible to the host
        {"name": "moe_layer_b2", "kind": "stack", "recipe": "iq3_s", "layers": 1, "nb": 2, "host": True, **moe, "router": 30},
        # one conversation: a half stack at one token
        {"name": "stack_iq3_s_b1", "kind": "stack", "recipe": "iq3_s", "layers": 24, "nb": 1, "host": False, **moe},
        # the headline workload: the full 48-layer stack at sixteen tokens
        {"name": "stack_iq3_s_b16", "kind": "stack", "recipe": "iq3_s", "layers": 48, "nb": 16, "host": False, **moe},
        # the reference model's layer at eight tokens
        {"name": "stack_iq4_nl_b8", "kind": "stack", "recipe": "iq4_nl", "layers": 12, "nb": 8, "host": False, **moe, "D": 2560, "I": 640},
        # a file in the common K-quant mix at four tokens
        {"name": "stack_q4_k_b4", "kind": "stack", "recipe": "q4_k", "layers": 8, "nb": 4, "host": False, **moe},
        # the FFN halves of a decode step with their real dependency, five tokens
        {"name": "hyper_b5", "kind": "hyper", "recipe": "iq3_s", "layers": 24, "nb": 5, **moe},
        # sixteen conversations, most with one row, some with drafts
        {"name": "vstep_16_slots", "kind": "vstep", "recipe": "iq3_s", "slots": 16, "rows": 45, **moe},
        # a continuous-batching step of 69 rows (BASELINE's fourth configuration)
        {"name": "pack_69_rows", "kind": "pack", "recipe": "iq3_s", "rows": 69, "tm": 16, "skew": 1.1, **moe},
        # half a prefill segment of the reference (4096 tokens)
        {"name": "pack_2048_rows", "kind": "pack", "recipe": "iq3_s", "rows": 2048, "tm": 64, "skew": 1.1, **moe},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng, recipe):
    D, I = (2560, 640) if recipe == "iq4_nl" else rng.choice(((1024, 256), (1024, 512), (2048, 512), (2048, 512)))
    E = rng.choice((64, 128, 256, 512, 512))
    return {"D": D, "I": I, "E": E, "topk": rng.choice((4, 6, 8, 10, 10)), "router": rng.choice((1, 1, 30))}


def draw(rng):
    kind = rng.choice(("matvec", "dense", "stack", "stack", "stack", "hyper", "vstep", "pack", "pack"))
    nb = _log(rng, 1, 16)
    if kind == "matvec":
        return {"kind": kind, "fmt": rng.choice((21, 21, 8, 8, 12, 14, 20, 23, 1, 30)), "N": _log(rng, 100, 20000), "K": 256 * rng.randint(2, 16), "nb": nb}
    if kind == "dense":
        return {"kind": kind, "layers": _log(rng, 4, 16), "K": rng.choice((1024, 2048, 2560)), "ofmt": rng.choice((8, 21)), "vocab": 16 * _log(rng, 1500, 9000), "nb": nb}
    recipe = rng.choice(("iq3_s", "iq3_s", "iq4_nl", "q4_k", "q8_0"))
    if kind == "stack":
        host = rng.random() < 0.3
        return {"kind": kind, "recipe": recipe, "layers": 1 if host else _log(rng, 2, 24 if recipe == "iq3_s" else 8), "nb": nb, "host": host, **_shape(rng, recipe)}
    if kind == "hyper":
        recipe = rng.choice(("iq3_s", "iq3_s", "iq4_nl"))
        return {"kind": kind, "recipe": recipe, "layers": _log(rng, 2, 16 if recipe == "iq3_s" else 8), "nb": nb, **_shape(rng, recipe)}
    recipe = rng.choice(("iq3_s", "iq3_s", "iq4_nl")) if kind == "pack" else recipe
    if kind == "vstep":
        slots = rng.randint(2, 16)
        return {"kind": kind, "recipe": recipe, "slots": slots, "rows": min(64, slots + rng.randint(0, 4 * slots)), **_shape(rng, recipe)}
    rows = _log(rng, 17, 2048)
    return {"kind": kind, "recipe": recipe, "rows": rows, "tm": 16 if rows < 256 else rng.choice((32, 64)), "skew": round(rng.uniform(0.5, 1.1), 2), **_shape(rng, recipe)}


_gpu = None


def _device():
    global _gpu
    if _gpu is None:
        _gpu = q.Gpu()
    return _gpu


class _Buf(Buf):
    """A buffer given back when the last that refers to it goes away: the state, or a view of it."""

    def __del__(self):
        self.free()


class _Path(q.Path):
    def __del__(self):
        self.close()


class _Par(q.Par):
    def __del__(self):
        self.free()


class _Raw:
    """A device buffer in the form torch takes without a copy."""

    def __init__(self, buf, typestr, shape):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (buf.L.qw_hip_buf_devptr(buf.ref()), False), "version": 2}


def _view(buf, typestr, *shape):
    return torch.as_tensor(_Raw(buf, typestr, shape), device="cuda")


def _host(buf, dtype, *shape):
    raw = (C.c_uint8 * buf.size).from_address(buf.c.ptr)
    raw.buf = buf
    return np.frombuffer(raw, dtype, math.prod(shape)).reshape(shape)


class State:
    """What a program keeps: buffers, weights and handles."""

    def __init__(self, case, seed):
        self.case, self.gpu = case, _device()
        self.rng = np.random.default_rng(seed)
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed * 7 + 1)

    def buf(self, size, device_only=True):
        return _Buf(self.gpu, int(size), device_only=device_only)

    def upload(self, arr, device_only=True):
        b = self.buf(arr.nbytes, device_only)
        b.fill(arr)
        return b

    def path(self, D, I, E, topk, device_scratch=True):
        return _Path(self.gpu, D, I, E, topk, 16, device_scratch=device_scratch)

    def weights(self, pieces, scale):
        """One buffer holding (type, values) pieces one after the other, random blocks as in synth.blocks; their tensors."""
        sizes = [n // synth.BLOCK[f][0] * synth.BLOCK[f][1] for f, n in pieces]
        at = np.concatenate([[0], np.cumsum([(s + 255) // 256 * 256 for s in sizes])]).tolist()
        buf = self.buf(at[-1])
        raw = _view(buf, "|u1", at[-1])
        for (f, n), o, s in zip(pieces, at, sizes):
            v = raw[o:o + s]
            if f in (1, 30):
                w = torch.randn(n, generator=self.gen, device="cuda") * (0.02 * scale)
                v.copy_(w.to(torch.float16 if f == 1 else torch.bfloat16).view(torch.uint8))
                continue
            bb = synth.BLOCK[f][1]
            b = v.view(-1, bb)
            if f == 8:
                v.view(torch.int8).random_(-127, 128, generator=self.gen)
            else:
                raw[o:o + (s + 3) // 4 * 4].view(torch.int32).random_(-2**31, 2**31, generator=self.gen)
            offs, sigma = synth.SCALE_FIELDS[f] if f in synth.SCALE_FIELDS else ((0,), synth.D_SIGMA[f])
            for off in offs:
                d = torch.randn(b.shape[0], generator=self.gen, device="cuda").abs_().mul_(sigma * scale).to(torch.float16)
                b[:, off:off + 2] = d.view(torch.uint8).view(-1, 2)
        return [q.Tensor(buf, f, o) for (f, _), o in zip(pieces, at)]

    def moe_layer(self, recipe, l, D, I, E, router):
        gu, dn, sg, su, sd = RECIPES[recipe]
        if recipe == "iq3_s" and l % 4 == 3:
            sg = su = sd = 8
        g, u, d = self.weights([(gu, E * I * D), (gu, E * I * D), (dn, E * D * I)], synth.MOE_D_SCALE)
        a, b, c = self.weights([(sg, I * D), (su, I * D), (sd, D * I)], synth.MOE_D_SCALE)
        r, v = self.weights([(router, E * D), (router, D)], 1.0)
        return q.MoeLayer(router=r, sh_gate_w=v, gate=g, up=u, down=d, sh_gate=a, sh_up=b, sh_down=c)


def _moe_keys(case):
    return [case[k] for k in ("D", "I", "E", "topk")]


def prepare(case, seed):
    s = State(case, seed)
    kind, rng = case["kind"], s.rng
    if kind == "matvec":
        N, K, nb = case["N"], case["K"], case["nb"]
        s.p = s.path(2048, 512, 512, 10)
        s.W = s.weights([(case["fmt"], N * K)], 1.0)[0]
        s.x, s.y = s.upload(synth.activations(rng, nb, K), device_only=False), s.buf(nb * N * 4, device_only=False)
        s.out = {"y": _host(s.y, np.float32, nb, N)}
    elif kind == "dense":
        K, nb = case["K"], case["nb"]
        s.p = s.path(2048, 512, 512, 10)
        s.fmts, s.rows = [f for f, _ in DENSE], [int(K * m) for _, m in DENSE]
        s.proj = [s.weights([(f, n * K) for f, n in zip(s.fmts, s.rows)], 1.0) for _ in range(case["layers"])]
        s.oproj = [s.weights([(case["ofmt"], K * K)], 1.0)[0] for _ in range(case["layers"])]
        s.head = s.weights([(14, case["vocab"] * K)], 1.0)[0]
        s.x = s.upload(synth.activations(rng, nb, K), device_only=False)
        s.ys = [s.buf(nb * n * 4) for n in s.rows]
        s.yo, s.logits = s.buf(nb * K * 4), s.buf(nb * case["vocab"] * 4, device_only=False)
        s.out = {"logits": _host(s.logits, np.float32, nb, case["vocab"]), "o": _view(s.yo, "<f4", nb, K), **{"y%d" % i: _view(y, "<f4", nb, n) for i, (y, n) in enumerate(zip(s.ys, s.rows))}}
    elif kind in ("stack", "hyper"):
        D, nb, L, dev = case["D"], case["nb"], case["layers"], not case.get("host")
        s.p = s.path(*_moe_keys(case), device_scratch=dev)
        s.layers = [s.moe_layer(case["recipe"], l, D, case["I"], case["E"], case["router"]) for l in range(L)]
        s.layers_c = (QwMoeLayer * L)(*[m.c for m in s.layers])
        s.lg, s.sel = [s.buf(s.p.logits_bytes(nb), dev) for _ in range(L)], [s.buf(s.p.sel_bytes(nb), dev) for _ in range(L)]
        s.lg_c, s.sel_c = (QwBuf * L)(*[b.c for b in s.lg]), (QwBuf * L)(*[b.c for b in s.sel])
        s.o = s.buf(nb * D * 2, device_only=False)
        s.out = {"out": _host(s.o, np.float16, nb, D)}
        if kind == "stack":
            s.x = s.upload(synth.activations(rng, nb, D), device_only=dev)
            if case["host"]:
                s.out["logits"] = _host(s.lg[0], np.float32, nb, case["E"] + 1)
        else:
            w = synth.hyper_weights(rng, D)
            hw, s.hyper = [], []
            for l in range(L):
                c = QwHyperW()
                for k in ("hc_norm", "mix_down", "mix_up", "inject"):
                    s.hyper.append(s.upload(np.roll(w[k].ravel(), 977 * l)))
                    setattr(c, k, q.Tensor(s.hyper[-1], 0 if k == "hc_norm" else 30).c())
                hw.append(c)
            s.hyper_c = (QwHyperW * L)(*hw)
            s.h0, _, s.inj0 = synth.hyper_state(rng, nb, D)
            s.h, s.x = s.buf(s.h0.nbytes, False), s.buf(nb * D * 2)
            s.inj = [s.buf(s.inj0.nbytes, False), s.buf(s.inj0.nbytes, False)]
            s.inj_c = (QwBuf * 2)(*[b.c for b in s.inj])
            s.pd = s.buf(s.gpu.L.qw_path_hyper_pd_bytes(nb))
            s.out.update(h=_host(s.h, np.float32, nb, 4, D), inj=_host(s.inj[L % 2], np.float32, nb, 4, 4))
    elif kind == "vstep":
        D, R, B = case["D"], case["rows"], case["slots"]
        s.p = s.path(*_moe_keys(case))
        s.layer = s.moe_layer(case["recipe"], 0, D, case["I"], case["E"], case["router"])
        s.n = (1 + np.bincount(rng.integers(0, B, R - B), minlength=B)).tolist()  # every slot one row, the drafts spread over them
        s.x, s.o = s.upload(synth.activations(rng, R, D), device_only=False), s.buf(R * D * 2, device_only=False)
        s.par = _Par()
        s.out = {"out": _host(s.o, np.float16, R, D)}
    else:
        D, T, E, K = case["D"], case["rows"], case["E"], case["topk"]
        s.p = s.path(*_moe_keys(case))
        s.p.pf_reserve(T, case["tm"])
        s.layer = s.moe_layer(case["recipe"], 0, D, case["I"], E, case["router"])
        w = rng.uniform(0.05, 1.0, (T, K)).astype(np.float32)
        s.x, s.ids = s.upload(synth.activations(rng, T, D)), s.upload(_routing(rng, T, E, K, case["skew"]).ravel())
        s.w, s.o = s.upload((w / w.sum(axis=1, keepdims=True)).ravel()), s.buf(T * D * 2)
        s.out = {"out": _view(s.o, "<f2", T, D)}
    torch.cuda.synchronize()
    return s


def _routing(rng, T, E, K, skew):
    """synth.zipf_ids for many rows at once: the K largest of log p + Gumbel noise are K draws without replacement."""
    p = np.log(1.0 / np.arange(1, E + 1) ** skew)[rng.permutation(E)]
    return np.argsort(-(p + rng.gumbel(size=(T, E))), axis=1)[:, :K].astype(np.uint32)


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "vstep":
        s.p.par_vstep(s.par, s.layer, s.n, s.x, s.o)
        return s.out
    if kind == "hyper":  # the step starts from the embeddings' streams
        s.h.fill(s.h0)
        s.inj[0].fill(s.inj0)
    b = s.gpu.batch()
    if kind == "matvec":
        s.p.qmv_gg(b, s.W, case["N"], case["K"], s.x, s.y, case["nb"])
    elif kind == "dense":
        for ws, o in zip(s.proj, s.oproj):
            s.p.qmv_ggm(b, ws, s.rows, case["K"], s.x, s.ys, case["nb"])
            s.p.qmv_gg(b, o, case["K"], case["K"], s.x, s.yo, case["nb"])
        s.p.qmv_gg(b, s.head, case["vocab"], case["K"], s.x, s.logits, case["nb"])
    elif kind == "stack":
        s.p.gg_moe_stack(b, s.layers_c, case["layers"], case["nb"], s.x, s.lg_c, s.sel_c, s.o)
    elif kind == "hyper":
        s.p.hyper_moe_stack(b, s.hyper_c, s.layers_c, case["layers"], case["nb"], False, s.h, s.inj_c, s.pd, s.x, s.lg_c, s.sel_c, s.o)
    else:
        s.p.pf_moe(b, s.layer, case["rows"], s.x, s.ids, s.w, s.o)
    b.end()
    return s.out


def work(case):
    kind = case["kind"]
    rb = synth.row_bytes
    if kind == "matvec":
        N, K, nb = case["N"], case["K"], case["nb"]
        return {"bytes": N * rb(case["fmt"], K) + nb * (K * 2 + N * 4), "flops": 2 * nb * N * K}
    if kind == "dense":
        K, nb = case["K"], case["nb"]
        layer = [(f, int(K * m)) for f, m in DENSE] + [(case["ofmt"], K)]
        rows = case["layers"] * sum(n for _, n in layer) + case["vocab"]
        w = case["layers"] * sum(n * rb(f, K) for f, n in layer) + case["vocab"] * rb(14, K)
        return {"bytes": w + nb * (K * 2 + sum(n for _, n in layer) * 4 + case["vocab"] * 4), "flops": 2 * nb * rows * K}
    D, I, E, K = _moe_keys(case)
    gu, dn, sg, su, sd = RECIPES[case["recipe"]]
    expert = 2 * I * rb(gu, D) + D * rb(dn, I)
    shared = I * (rb(sg, D) + rb(su, D)) + D * rb(sd, I)
    router = (E + 1) * D * 2
    flops = 6 * D * I  # of one expert for one row
    if kind == "pack":
        T = case["rows"]
        ids = _routing(np.random.default_rng(1), T, E, K, case["skew"])
        return {"bytes": len(np.unique(ids)) * expert + T * (D * 4 + K * 8), "flops": T * K * flops}
    T, L = (case["rows"], 1) if kind == "vstep" else (case["nb"], case["layers"])
    U = E * (1 - (1 - K / E) ** T)  # distinct experts of T tokens
    w = L * (U * expert + shared + router)
    f = L * T * ((K + 1) * flops + 2 * (E + 1) * D)
    if kind == "hyper":
        w += L * ((320 + 4) * 4 * D * 2 + 4 * D * 320 * 2 + 4 * D * 4) + T * 4 * D * 4 * 2
        f += L * T * 2 * (2 * 320 + 4) * 4 * D
    return {"bytes": w + T * D * 4, "flops": f}


def tolerance(case):
    if case["kind"] in ("matvec", "dense"):
        return {"rel": 1e-5}  # sums in binary32 over exact weights
    if case["kind"] == "hyper":
        return {"rel": 3e-3}  # every layer's activations are rounded to binary16
    return {"rel": 2e-3 if case["kind"] == "pack" else 1e-3}  # binary16 results (packing: binary16 intermediates too)
