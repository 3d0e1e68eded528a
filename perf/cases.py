"""The work that users of klearu_amd have it do, as cases to time and compare.

A case is a dict of plain values; its "kind" names the path:

  mlp      Deja Vu sparse SwiGLU MLP blocks of a decoder: norm, low-rank predictor, exact top-k,
           gathered FFN, residual (mlp_block / mlp_block_batch), each layer on its own hidden rows
  attn     head-sparse decode attention blocks: a prefill's K/V handed to the cache, then a few
           decode steps (attn_block / attn_block_batch), each on its own hidden rows
  slide    one SLIDE LSH layer on a batch of dense inputs (kh_slide_layer_forward)
  xc       extreme classification: a dense hidden layer over sparse inputs, then an LSH-sampled
           softmax output layer
  train    one Network.train_step_sparse; the updated weights come back
  predict  Network.predict_batch of a trained network
  layer    the klearu-dejavu transformer layer in f32: SparseMlp and SparseAttention
  accel    klearu-accel entry points: dense rows times a vector, a BF16 round trip of the rows, one
           row's BF16 dot, an example's sparse dot and scatter-add
  index    an LSH index rebuilt from a weight matrix and queried, as SLIDE training does at
           intervals

Inputs are made from the seed on the GPU, with the weight and input distributions of bench.py.
exact() gives the outputs in 64 bits in plain torch / numpy.  Which neurons or heads are selected is
decided by f32 sums in a fixed order, so exact() replays those sums (and only those) in f32.
"""
from __future__ import annotations

import math

import numpy as np
import torch

EPS = 1e-5
THETA = 10000.0
CAP = 128          # bucket capacity of every LSH index here (the reference's default)
LABELS = 5         # at most this many labels per training example


# ------------------------------------------------------------------ cases
def listed():
    return [
        # A toy model's two layers, one token: launches and latency are all there is.
        dict(name="mlp_tiny_b1", kind="mlp", hidden=512, inter=1408, rank=64, k=212, batch=1, layers=2),
        # 7B-class decode of one sequence, the headline workload: 15% of 11008 neurons.
        dict(name="mlp_7b_b1", kind="mlp", hidden=4096, inter=11008, rank=256, k=1652, batch=1, layers=4),
        # The same model serving 16 sequences that share the union of their neurons.
        dict(name="mlp_7b_b16", kind="mlp", hidden=4096, inter=11008, rank=256, k=1652, batch=16, layers=2),
        # 7B-class attention of one sequence: half of the heads over a prefix of about 2000 positions.
        dict(name="attn_7b_b1", kind="attn", hidden=4096, heads=32, kv_heads=32, dim=128, rank=128, k=16,
             prefix=1999, batch=1, tokens=8, layers=2),
        # Eight sequences that start from one shared prompt.
        dict(name="attn_7b_b8", kind="attn", hidden=4096, heads=32, kv_heads=32, dim=128, rank=128, k=16,
             prefix=1999, batch=8, tokens=8, layers=1),
        # SLIDE hidden layer on 784-d inputs that are 80% zeros.
        dict(name="slide_784_b128", kind="slide", dim=784, neurons=1024, bits=6, tables=50, batch=128),
        # Extreme classification: 135909-d sparse inputs, 670091 classes.
        dict(name="xc_670k_b256", kind="xc", dim=135909, hidden=128, neurons=670091, bits=9, tables=50,
             nnz=75, batch=256),
        # A training step of a smaller net of that form.
        dict(name="train_8k_b32", kind="train", dim=8192, hidden=128, neurons=8191, bits=6, tables=50, nnz=75,
             batch=32, optimizer="Adam"),
        # Inference of a trained classifier with a sparse hidden layer.
        dict(name="predict_784_b128", kind="predict", dim=784, hidden=1024, neurons=32, bits=6, tables=50,
             nnz=157, batch=128),
        # The f32 transformer layer of klearu-dejavu, a few tokens, no size a round number.
        dict(name="layer_f32_b3", kind="layer", hidden=1000, inter=2741, heads=20, dim=50, keep=0.3, batch=3),
        # A weight matrix of a 7B layer through the accel entry points.
        dict(name="accel_11008x4096", kind="accel", rows=11008, n=4096, nnz=75, dim=135909),
        # Index maintenance over an output layer.
        dict(name="index_200k", kind="index", dim=128, neurons=200003, bits=9, tables=50, batch=64),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "attn", "attn", "slide", "xc", "train", "predict", "layer", "accel", "index"])
    if kind == "mlp":
        inter = _logint(rng, 1024, 11008)
        hidden = 64 * rng.randint(8, 64)
        batch = rng.choice([1, 1, _logint(rng, 2, 16)])
        return dict(kind=kind, hidden=hidden, inter=inter, rank=_logint(rng, 32, 256),
                    k=max(1, int(inter * rng.uniform(0.05, 0.3))), batch=batch, layers=rng.randint(1, 2))
    if kind == "attn":
        dim = rng.choice([64, 128])
        kv = rng.choice([4, 8, 16, 32])
        heads = min(64 if dim == 64 else 32, kv * rng.choice([1, 2, 4]))
        kv = min(kv, heads)
        return dict(kind=kind, hidden=1024 * rng.randint(1, 4), heads=heads, kv_heads=kv, dim=dim,
                    rank=_logint(rng, 32, 128), k=rng.randint(1, heads), prefix=_logint(rng, 16, 4000),
                    batch=rng.choice([1, 1, _logint(rng, 2, 8)]), tokens=8, layers=1)
    if kind == "slide":
        return dict(kind=kind, dim=_logint(rng, 64, 2048), neurons=_logint(rng, 100, 8000), bits=rng.randint(4, 9),
                    tables=rng.randint(10, 50), batch=_logint(rng, 1, 512))
    if kind == "xc":
        return dict(kind=kind, dim=_logint(rng, 5000, 135909), hidden=4 * rng.randint(8, 32),
                    neurons=_logint(rng, 10000, 400000), bits=rng.randint(7, 9), tables=rng.randint(20, 50),
                    nnz=_logint(rng, 20, 300), batch=_logint(rng, 1, 256))
    if kind == "train":
        return dict(kind=kind, dim=_logint(rng, 128, 8192), hidden=_logint(rng, 32, 128), neurons=_logint(rng, 10, 8191),
                    bits=rng.randint(4, 6), tables=rng.randint(10, 50), nnz=_logint(rng, 20, 100),
                    batch=_logint(rng, 4, 32), optimizer=rng.choice(["Sgd", "Adam"]))
    if kind == "predict":
        return dict(kind=kind, dim=_logint(rng, 128, 4096), hidden=_logint(rng, 64, 1024), neurons=_logint(rng, 10, 4000),
                    bits=rng.randint(4, 7), tables=rng.randint(10, 50), nnz=_logint(rng, 20, 120),
                    batch=_logint(rng, 1, 128))
    if kind == "layer":
        return dict(kind=kind, hidden=_logint(rng, 64, 2048), inter=_logint(rng, 128, 5632), heads=rng.randint(4, 16),
                    dim=rng.randint(16, 64), keep=rng.uniform(0.1, 0.5), batch=_logint(rng, 1, 32))
    if kind == "accel":
        return dict(kind=kind, rows=_logint(rng, 1, 11008), n=_logint(rng, 64, 4096), nnz=_logint(rng, 8, 1000),
                    dim=_logint(rng, 2000, 135909))
    return dict(kind=kind, dim=_logint(rng, 16, 256), neurons=_logint(rng, 1024, 200003), bits=rng.randint(5, 9),
                tables=rng.randint(10, 50), batch=_logint(rng, 1, 256))


# ------------------------------------------------------------------ inputs
class Inputs:
    pass


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, device="cuda") * scale


def _bf(t):
    """f32 values that are BF16 values."""
    return t.to(torch.bfloat16).float()


def _bits(t):
    """BF16 bit patterns of t as a host uint16 array."""
    return t.to(torch.bfloat16).view(torch.int16).cpu().numpy().view(np.uint16)


def _planes(g, tables, bits, dim):
    """Ternary hyperplanes with SimHash's probabilities (1/6, 2/3, 1/6)."""
    u = torch.rand((tables, bits, dim), generator=g, device="cuda")
    return (u >= 5 / 6).to(torch.int8) - (u < 1 / 6).to(torch.int8)


def _positions(g, rows, nnz, dim):
    """rows x nnz ascending distinct positions below dim, one in each of nnz equal parts."""
    edge = torch.arange(nnz + 1, device="cuda", dtype=torch.int64) * dim // nnz
    width = (edge[1:] - edge[:-1]).double()
    u = torch.rand((rows, nnz), generator=g, device="cuda", dtype=torch.float64)
    return edge[:-1] + torch.minimum((u * width).long(), width.long() - 1)


def _csr(g, rows, nnz, dim):
    """Sparse examples of nnz entries in U[0, 1): (offsets, positions, values)."""
    nnz = min(nnz, dim)
    idx = _positions(g, rows, nnz, dim)
    val = torch.rand((rows, nnz), generator=g, device="cuda")
    off = torch.arange(rows + 1, device="cuda", dtype=torch.int64) * nnz
    return off, idx, val


def _inputs(case, seed):
    c, g, s = case, _gen(seed), Inputs()
    kind = c["kind"]
    if kind == "mlp":
        H, I, R, L = c["hidden"], c["inter"], c["rank"], c["layers"]
        s.ffn = [[_randn(g, I, H, scale=0.02).to(torch.bfloat16), _randn(g, I, H, scale=0.02).to(torch.bfloat16),
                  _randn(g, H, I, scale=0.02).to(torch.bfloat16)] for _ in range(L)]
        s.pred = [[_bf(_randn(g, R, H, scale=0.02)), _bf(_randn(g, I, R, scale=0.02))] for _ in range(L)]
        s.norm = 1.0 + _randn(g, L, H, scale=0.1)
        s.x = _randn(g, L, c["batch"], H)
    elif kind == "attn":
        H, nh, nk, d, R, L = c["hidden"], c["heads"], c["kv_heads"], c["dim"], c["rank"], c["layers"]
        s.proj = [[_randn(g, *shape, scale=0.02).to(torch.bfloat16)
                   for shape in ((nh * d, H), (nk * d, H), (nk * d, H), (H, nh * d))] for _ in range(L)]
        s.pred = [[_bf(_randn(g, R, H, scale=0.02)), _bf(_randn(g, nh, R, scale=0.1))] for _ in range(L)]
        s.kv = [[_bf(_randn(g, nk, c["prefix"], d)) for _ in range(2)] for _ in range(L)]
        s.norm = 1.0 + _randn(g, L, H, scale=0.1)
        s.x = _randn(g, c["tokens"], L, c["batch"], H)
    elif kind == "slide":
        s.planes = _planes(g, c["tables"], c["bits"], c["dim"])
        s.W = _randn(g, c["neurons"], c["dim"], scale=0.01)
        s.b = _randn(g, c["neurons"], scale=0.01)
        s.x = torch.rand((c["batch"], c["dim"]), generator=g, device="cuda")
        s.x *= torch.rand(s.x.shape, generator=g, device="cuda") >= 0.8
    elif kind == "xc":
        s.planes = _planes(g, c["tables"], c["bits"], c["hidden"])
        s.W1 = _randn(g, c["hidden"], c["dim"], scale=0.01)
        s.b1 = torch.zeros(c["hidden"], device="cuda")
        s.W2 = _randn(g, c["neurons"], c["hidden"], scale=0.01)
        s.b2 = torch.zeros(c["neurons"], device="cuda")
        s.csr = _csr(g, c["batch"], c["nnz"], c["dim"])
    elif kind in ("train", "predict"):
        dims, n, wide = (c["dim"], c["hidden"]), (c["hidden"], c["neurons"]), kind == "train"
        # training: every hidden neuron is active (one-bit tables, top-k of all), the output layer
        # takes the union of its buckets; inference: both layers keep the neurons hit most often
        s.bits = (1 if wide else c["bits"], c["bits"])
        s.sampling = ("TopK", "Vanilla" if wide else "TopK")
        s.top_k = (n[0] if wide else max(1, n[0] // 4), n[1])
        s.planes = [_planes(g, c["tables"], s.bits[i], dims[i]) for i in range(2)]
        s.W = [_randn(g, n[i], dims[i], scale=(2.0 / dims[i]) ** 0.5 if i else 0.01 if wide else 0.1) for i in range(2)]
        s.b = [_randn(g, n[i], scale=0.01) for i in range(2)]
        s.csr = _csr(g, c["batch"], c["nnz"], c["dim"])
        s.labels = torch.randint(0, c["neurons"], (c["batch"], LABELS), generator=g, device="cuda")
        s.n_labels = torch.randint(1, LABELS + 1, (c["batch"],), generator=g, device="cuda")
    elif kind == "layer":
        H, I, A = c["hidden"], c["inter"], c["heads"] * c["dim"]
        shapes = dict(gate=(I, H), up=(I, H), down=(H, I), q=(A, H), k=(A, H), v=(A, H), o=(H, A))
        s.w = {n: _randn(g, *sh, scale=(2.0 / sum(sh)) ** 0.5) for n, sh in shapes.items()}
        s.wb = {n: _randn(g, sh[0], scale=0.05) for n, sh in shapes.items()}
        s.neurons = torch.randperm(I, generator=g, device="cuda")[:max(1, int(I * c["keep"]))].cpu().numpy()
        s.heads = torch.randperm(c["heads"], generator=g, device="cuda")[:max(1, int(c["heads"] * c["keep"]))].cpu().numpy()
        s.x = _randn(g, c["batch"], H)
    elif kind == "accel":
        s.a = _randn(g, c["rows"], c["n"], scale=0.02)
        s.v = _randn(g, c["n"])
        _, idx, val = _csr(g, 1, c["nnz"], c["dim"])
        s.idx, s.val = idx[0].to(torch.int32), val[0].contiguous()
        s.dense = _randn(g, c["dim"], scale=0.01)
    else:
        s.planes = _planes(g, c["tables"], c["bits"], c["dim"])
        s.W = _randn(g, c["neurons"], c["dim"], scale=0.01)
        s.x = torch.relu(_randn(g, c["batch"], c["dim"]))
    return s


# ------------------------------------------------------------------ prepare
def _host(t):
    return np.ascontiguousarray(t.cpu().numpy())


def _predictor(w1, w2):
    from klearu_amd.dejavu import SparsityPredictor
    return SparsityPredictor(_host(w1), np.zeros(w1.shape[0], np.float32), _host(w2), np.zeros(w2.shape[0], np.float32))


def _layer(planes, W, b, activation, sampling, top_k, bucket):
    from klearu_amd.lsh import FIFO, RESERVOIR, HashFamily, LshConfig, LshIndex
    from klearu_amd.slide import Layer, LayerConfig
    tables, bits, dim = planes.shape
    index = LshIndex(HashFamily.from_planes(_host(planes)), FIFO if bucket == "Fifo" else RESERVOIR, CAP)
    cfg = LayerConfig(dim, W.shape[0], activation, LshConfig(num_tables=tables, num_hashes=bits, bucket_capacity=CAP,
                                                             bucket_type=bucket), sampling, 2, top_k)
    return Layer(cfg, _host(W), _host(b), 0, index=index)


def _bound(c):
    """Entries that a CSR result can have here: the tables' full buckets, each neuron at most once."""
    return c["batch"] * min(c["neurons"], c["tables"] * CAP)


def _csr_buffers(st, c, kinds):
    """A caller's own result buffers, with room for every row's worst case (an input that hits
    nothing takes every neuron), so that a call need not wait for its total."""
    st.cap = c["batch"] * max(c["neurons"], c["tables"] * CAP)
    st.off = torch.zeros(c["batch"] + 1, dtype=torch.int64, device="cuda")
    st.out = [torch.zeros(st.cap, dtype=k, device="cuda") for k in kinds]


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    kind = c["kind"]
    st = Inputs()
    st.case = c
    if kind == "mlp":
        from klearu_amd.dejavu import Mlp
        st.mlp = [Mlp(*(_bits(w) for w in ws), max_batch=c["batch"]) for ws in s.ffn]
        st.pred = [_predictor(*ws) for ws in s.pred]
        st.norm, st.x = list(s.norm), s.x
    elif kind == "attn":
        from klearu_amd.attention import SparseAttention
        st.attn = [SparseAttention(c["hidden"], c["heads"], c["kv_heads"], c["dim"], *ws, c["prefix"] + c["tokens"],
                                   c["batch"], THETA) for ws in s.proj]
        st.pred = [_predictor(*ws) for ws in s.pred]
        st.norm, st.x, st.kv = list(s.norm), s.x, s.kv
    elif kind == "slide":
        st.layer = _layer(s.planes, s.W, s.b, "Relu", "Vanilla", 0, "Fifo")
        st.x = s.x
        _csr_buffers(st, c, (torch.int32, torch.float32, torch.float32))
    elif kind == "xc":
        from klearu_amd.slide import DenseLayer
        st.hidden = DenseLayer(_host(s.W1), _host(s.b1), "Relu")
        st.layer = _layer(s.planes, s.W2, s.b2, "Softmax", "Vanilla", 0, "Reservoir")
        off, idx, val = s.csr
        st.csr = off, idx.to(torch.int32).reshape(-1).contiguous(), val.reshape(-1).contiguous()
        _csr_buffers(st, c, (torch.int32, torch.float32, torch.float32))
    elif kind in ("train", "predict"):
        from klearu_amd.slide import Network
        st.layers = [_layer(s.planes[i], s.W[i], s.b[i], ("Relu", "Softmax")[i], s.sampling[i], s.top_k[i], "Fifo")
                     for i in range(2)]
        st.net = Network(st.layers, c.get("optimizer", "Sgd"))
        off, idx, val = s.csr
        if kind == "train":
            st.csr = off, idx.to(torch.int32).reshape(-1).contiguous(), val.reshape(-1).contiguous()
            st.labels = [sorted(set(row[:n])) for row, n in zip(s.labels.tolist(), s.n_labels.tolist())]
        else:
            st.x = torch.zeros((c["batch"], c["dim"]), device="cuda").scatter_(1, idx, val)
    elif kind == "layer":
        from klearu_amd.dejavu_transformer import Linear, SparseAttention, SparseMlp
        st.lin = {n: Linear(_host(w), _host(s.wb[n])) for n, w in s.w.items()}
        st.mlp = SparseMlp(c["hidden"], c["inter"])
        st.attn = SparseAttention(c["hidden"], c["heads"], c["dim"])
        st.neurons, st.heads, st.x = s.neurons, s.heads, s.x
    elif kind == "accel":
        st.a, st.v, st.idx, st.val, st.dense = s.a, s.v, s.idx, s.val, s.dense
    else:
        from klearu_amd.lsh import FIFO, HashFamily, LshIndex
        st.index = LshIndex(HashFamily.from_planes(_host(s.planes)), FIFO, CAP)
        st.ids = torch.arange(c["neurons"], device="cuda", dtype=torch.int32)
        st.W, st.x = s.W, s.x
        _csr_buffers(st, c, (torch.int32, torch.int32))
    return st


# ------------------------------------------------------------------ run
def run(st):
    from klearu_amd import _lib
    from klearu_amd._dev import ptr, stream_ptr
    c = st.case
    kind = c["kind"]
    if kind == "mlp":
        from klearu_amd.dejavu import mlp_block, mlp_block_batch
        hidden, active = st.x.clone(), []
        for l in range(c["layers"]):
            if c["batch"] == 1:
                active.append(mlp_block(st.pred[l], st.mlp[l], hidden[l, 0], st.norm[l], EPS, c["k"]))
            else:
                active.append(mlp_block_batch(st.pred[l], st.mlp[l], hidden[l], st.norm[l], EPS, c["k"]))
        return {"hidden": hidden, "active": active}
    if kind == "attn":
        from klearu_amd.attention import attn_block, attn_block_batch
        hidden, heads = st.x.clone(), []
        for l in range(c["layers"]):
            for b in range(c["batch"]):
                st.attn[l].load_cache_dev(b, *st.kv[l])
        for t in range(c["tokens"]):
            for l in range(c["layers"]):
                if c["batch"] == 1:
                    heads.append(attn_block(st.pred[l], st.attn[l], hidden[t, l, 0], st.norm[l], EPS, c["k"]))
                else:
                    heads.append(attn_block_batch(st.pred[l], st.attn[l], hidden[t, l], st.norm[l], EPS, c["k"]))
        return {"hidden": hidden, "heads": heads}
    if kind in ("slide", "xc"):
        x = st.x if kind == "slide" else st.hidden.forward_sparse_csr(*st.csr, c["batch"])
        _lib.call("kh_slide_layer_forward", st.layer._h, ptr(x), c["batch"], ptr(st.off), *map(ptr, st.out), st.cap,
                  stream_ptr())
        return {"off": st.off, **{n: o[:_bound(c)] for n, o in zip(("ids", "pre", "act"), st.out)}}
    if kind == "train":
        loss = st.net.train_step_sparse(None, st.labels, 0.001, csr=st.csr)
        (w0, b0), (w1, b1) = st.layers[0].weights(), st.layers[1].weights()
        return {"loss": loss, "w0": w0, "b0": b0, "w1": w1, "b1": b1}
    if kind == "predict":
        return {"out": st.net.predict_batch(st.x)}
    if kind == "layer":
        p = st.lin
        return {"mlp": st.mlp.forward(st.x, p["gate"], p["up"], p["down"], st.neurons),
                "attn": st.attn.forward(st.x, p["q"], p["k"], p["v"], p["o"], st.heads)}
    if kind == "accel":
        from klearu_amd.accel import (Bf16Weights, dense_dot_dense_simd, scatter_add_simd, sparse_dot_dense_simd)
        w = Bf16Weights.from_f32(st.a)
        return {"rows": dense_dot_dense_simd(st.a, st.v),
                "bf16": w.data, "back": w.to_f32(),
                "dot": Bf16Weights(w.data[:c["n"]]).dot_f32(st.v),
                "sparse": sparse_dot_dense_simd(st.idx, st.val, st.dense),
                "added": scatter_add_simd(st.idx, st.val, st.dense.clone(), 0.5)}
    st.index.clear()
    st.index.insert_batch(st.ids, st.W)
    _lib.call("kh_lsh_index_query", st.index._h, ptr(st.x), c["batch"], ptr(st.off), *map(ptr, st.out), st.cap, stream_ptr())
    return {"off": st.off, **{n: o[:_bound(c)] for n, o in zip(("ids", "counts"), st.out)}}


# ------------------------------------------------------------------ work
def _union(n, share, times):
    """Expected distinct picks of `times` draws that each take this share of n."""
    return n * (1.0 - (1.0 - min(1.0, share)) ** times)


def work(case):
    c = case
    kind = c["kind"]
    if kind == "mlp":
        H, I, R, k, B, L = c["hidden"], c["inter"], c["rank"], c["k"], c["batch"], c["layers"]
        U = _union(I, k / I, B)
        return {"bytes": L * (3 * U * H * 2 + (R * H + I * R) * 2 + 2 * B * H * 4 + B * k * 4),
                "flops": L * B * (2 * R * (H + I) + 6 * U * H)}
    if kind == "attn":
        H, d, B, k, T, L = c["hidden"], c["dim"], c["batch"], c["k"], c["tokens"], c["layers"]
        U = _union(c["heads"], k / c["heads"], B)
        kv, ctx = c["kv_heads"] * d, c["prefix"] + (c["tokens"] + 1) / 2
        # the cache rows that the selected heads share are read once per sequence
        rows = B * _union(c["kv_heads"], k / c["heads"], c["heads"] / c["kv_heads"]) * ctx * d * 2 * 2
        load = 2 * kv * c["prefix"] * (4 + 2 * B)
        step = (2 * kv + 2 * U * d) * H * 2 + rows + (c["rank"] * H + c["heads"] * c["rank"]) * 2 + 2 * B * H * 4
        return {"bytes": L * (load + T * step),
                "flops": L * T * B * (2 * H * (2 * kv + 2 * k * d + c["rank"]) + 4 * k * ctx * d)}
    if kind == "slide":
        n, B, dim = c["neurons"], c["batch"], c["dim"]
        A = _union(n, min(CAP, n / 2 ** c["bits"]) / n, c["tables"])
        return {"bytes": n * dim * 4 + B * dim * 4 + B * A * 12 + B * c["tables"] * min(CAP, n / 2 ** c["bits"]) * 4,
                "flops": B * A * 2 * 0.2 * dim + B * c["tables"] * c["bits"] * 2 * 0.2 * dim / 3}
    if kind == "xc":
        n, B, hd = c["neurons"], c["batch"], c["hidden"]
        slots = min(CAP, n / 2 ** c["bits"])
        A = _union(n, slots / n, c["tables"])
        rows = _union(n, A / n, B)
        return {"bytes": B * c["nnz"] * (hd * 4 + 8) + rows * hd * 4 + B * A * 12 + B * c["tables"] * slots * 4,
                "flops": B * (2 * c["nnz"] * hd + 2 * A * hd)}
    if kind in ("train", "predict"):
        n, hd, B, dim, wide = c["neurons"], c["hidden"], c["batch"], c["dim"], c["kind"] == "train"
        A = _union(n, min(CAP, n / 2 ** c["bits"]) / n, c["tables"])
        if not wide:
            return {"bytes": (hd * dim + n * hd) * 4 + B * (dim + n) * 4, "flops": 2 * B * (hd // 4 * c["nnz"] + A * hd // 4)}
        slots = 7 if c["optimizer"] == "Adam" else 5      # weight and state arrays read and written, once per example
        return {"bytes": B * slots * (hd * dim + A * hd) * 4 + 4 * (hd * dim + n * hd),
                "flops": B * (2 * hd * c["nnz"] + 6 * A * hd + 10 * (hd * dim + A * hd))}
    if kind == "layer":
        H, I, A, B = c["hidden"], c["inter"], c["heads"] * c["dim"], c["batch"]
        n, a = max(1, int(I * c["keep"])), max(1, int(c["heads"] * c["keep"])) * c["dim"]
        return {"bytes": 4 * (3 * n * H + 4 * a * H + 3 * B * H), "flops": 2 * B * (3 * n * H + 4 * a * H)}
    if kind == "accel":
        m = c["rows"] * c["n"]
        return {"bytes": m * 4 + m * 6 + m * 6 + c["nnz"] * 24 + c["dim"] * 8, "flops": 2 * m}
    n, B, dim, P = c["neurons"], c["batch"], c["dim"], c["tables"] * c["bits"]
    kept = c["tables"] * min(n, CAP * 2 ** c["bits"])
    return {"bytes": n * dim * 4 + n * c["tables"] * 4 + kept * 4 + B * c["tables"] * CAP * 12, "flops": 2 * (n + B) * dim * P}


def tolerance(case):
    """About four times the distance to exact() that these sums show."""
    kind = case["kind"]
    if kind == "mlp":      # batches multiply on BF16 hi + lo halves of the activations
        return {"rel": 1.6e-5, "max": 2e-4}
    if kind == "train":    # Adam's first steps are lr * sign(gradient): a sum near zero can change one
        return {"rel": 6e-5, "max": 0.3}
    if kind == "index":
        return "exact"
    return {"rel": 4e-6, "max": 4e-5}


# ------------------------------------------------------------------ exact
def _seq32(W, X):
    """Sequential f32 dot products X [b][n] with the rows of W [m][n], each product rounded: [b][m]."""
    acc = torch.zeros((X.shape[0], W.shape[0]), device="cuda")
    WT, XT = W.t().contiguous(), X.t().contiguous()
    for i in range(W.shape[1]):
        acc += XT[i][:, None] * WT[i][None, :]
    return acc


def _rows32(hidden, w):
    """RmsNorm of the rows in f32, the sum of squares sequential."""
    x = _host(hidden)
    sq = np.add.accumulate(x * x, axis=1, dtype=np.float32)[:, -1]
    inv = np.float32(1.0) / np.sqrt(sq / np.float32(x.shape[1]) + np.float32(EPS))
    return torch.from_numpy((x * inv[:, None]) * _host(w)[None, :]).cuda()


def _top_k(rows, w1, w2, k):
    """The predictor's top k per row, ascending: scores in f32, ties to the lower index."""
    h = torch.relu(_seq32(w1, rows))
    z = _host(_seq32(w2, h))
    score = np.float32(1.0) / (np.float32(1.0) + np.exp(-z))
    order = np.argsort(-score, axis=1, kind="stable")[:, :k]
    return torch.from_numpy(np.sort(order, axis=1)).cuda()


def _exact_mlp(c, s):
    out = torch.empty(s.x.shape, dtype=torch.float64, device="cuda")
    for l in range(c["layers"]):
        rows = _rows32(s.x[l], s.norm[l])
        ids = _top_k(rows, *s.pred[l], c["k"])
        on = torch.unique(ids)
        x = s.x[l].double()
        x = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * s.norm[l].double()
        wg, wu, wd = s.ffn[l]
        g, u = x @ wg[on].double().t(), x @ wu[on].double().t()
        out[l] = s.x[l].double() + (g * torch.sigmoid(g) * u) @ wd[:, on].double().t()
    return {"hidden": out, "active": [None] * c["layers"]}


def _rope(v, pos):
    half = v.shape[-1] // 2
    f = (np.float32(1.0) / np.power(np.float32(THETA), (2.0 * np.arange(half, dtype=np.float32)) / np.float32(2 * half),
                                    dtype=np.float32)).astype(np.float32)
    ang = torch.from_numpy((np.float32(pos) * f).astype(np.float64)).cuda()   # f32 angles, as RoPE tables hold
    co, si = torch.cos(ang), torch.sin(ang)
    a, b = v[..., :half], v[..., half:]
    return torch.cat([a * co - b * si, b * co + a * si], -1)


def _exact_attn(c, s):
    nh, nk, d, B, P = c["heads"], c["kv_heads"], c["dim"], c["batch"], c["prefix"]
    out = torch.empty(s.x.shape, dtype=torch.float64, device="cuda")
    for l in range(c["layers"]):
        flat = s.x[:, l].reshape(-1, c["hidden"])
        ids = _top_k(_rows32(flat, s.norm[l]), *s.pred[l], c["k"]).reshape(c["tokens"], B, -1)
        wq, wk, wv, wo = (w.double() for w in s.proj[l])
        x = flat.double()
        x = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * s.norm[l].double()
        q, kk, vv = ((x @ w.t()).reshape(c["tokens"], B, -1, d) for w in (wq, wk, wv))
        ks = [s.kv[l][0].double()[None].expand(B, -1, -1, -1)]
        vs = [s.kv[l][1].double()[None].expand(B, -1, -1, -1)]
        for t in range(c["tokens"]):
            ks = [torch.cat(ks + [_rope(kk[t], P + t)[:, :, None]], 2)]
            vs = [torch.cat(vs + [vv[t][:, :, None]], 2)]
            qt = _rope(q[t], P + t)
            cat = torch.zeros((B, nh, d), dtype=torch.float64, device="cuda")
            for b in range(B):
                h = ids[t, b]
                kv = h // (nh // nk)
                sc = torch.einsum("hd,hjd->hj", qt[b, h], ks[0][b, kv]) / math.sqrt(d)
                cat[b, h] = (torch.softmax(sc, 1)[:, :, None] * vs[0][b, kv]).sum(1)
            out[t, l] = s.x[t, l].double() + cat.reshape(B, -1) @ wo.t()
    return {"hidden": out, "heads": [None] * (c["tokens"] * c["layers"])}


def _codes(planes, X):
    """SimHash codes [row][table]: the signs of sequential f32 sums."""
    T, K, dim = planes.shape
    got = []
    for r0 in range(0, X.shape[0], 65536):
        x = X[r0:r0 + 65536].t().contiguous()
        acc = torch.zeros((x.shape[1], T * K), device="cuda")
        p = planes.reshape(T * K, dim).t().float().contiguous()
        for i in range(dim):
            acc += x[i][:, None] * p[i][None, :]
        bit = (acc >= 0).reshape(-1, T, K).to(torch.int64)
        got.append((bit << torch.arange(K, device="cuda")).sum(2))
    return _host(torch.cat(got))


def _mix(z):
    z = z + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _buckets(codes, bits, bucket):
    """Per table and bucket the ids held after inserting 0..n-1 in order."""
    tables = []
    for t in range(codes.shape[1]):
        order = np.argsort(codes[:, t], kind="stable")
        edge = np.searchsorted(codes[order, t], np.arange(2 ** bits + 1))
        if bucket == "Fifo":
            tables.append([order[max(a, b - CAP):b] for a, b in zip(edge[:-1], edge[1:])])
            continue
        size = edge[1:] - edge[:-1]
        j = np.arange(order.size) - np.repeat(edge[:-1], size)
        with np.errstate(over="ignore"):
            count = (j + 1).astype(np.uint64)
            key = count * np.uint64(0x517CC1B727220A95) + order.astype(np.uint64)
            slot = np.where(_mix(key) % count < CAP, (_mix(key + np.uint64(1)) % np.uint64(CAP)).astype(np.int64), -1)
        slot = np.where(j < CAP, j, slot)
        held = np.full((2 ** bits, CAP), -1, np.int64)
        at = np.repeat(np.arange(2 ** bits), size)
        ok = slot >= 0
        held[at[ok], slot[ok]] = order[ok]      # later inserts win
        tables.append([h[h >= 0] for h in held])
    return tables


def _hits(buckets, code):
    ids, n = np.unique(np.concatenate([buckets[t][code[t]] for t in range(len(buckets))]), return_counts=True)
    return ids, n


def _forward(x64, W64, b64, ids, activation):
    """Pre-activations and activations of one input's active neurons."""
    i = torch.from_numpy(np.ascontiguousarray(ids)).cuda()
    pre = W64[i] @ x64 + b64[i]
    return i, pre, torch.relu(pre) if activation == "Relu" else torch.softmax(pre, 0)


def _exact_rows(c, s, x32, x64, W, b, activation, bucket):
    tables = _buckets(_codes(s.planes, W), c["bits"], bucket)
    q = _codes(s.planes, x32)
    W64, b64, rows = W.double(), b.double(), []
    for r in range(c["batch"]):
        ids, _ = _hits(tables, q[r])
        if not ids.size:
            ids = np.arange(c["neurons"])
        rows.append(_forward(x64[r], W64, b64, ids, activation))
    off = torch.tensor([0] + [r[0].numel() for r in rows], device="cuda").cumsum(0)
    pad = torch.zeros(_bound(c) - int(off[-1]), dtype=torch.float64, device="cuda")
    return {"off": None, "ids": None, **{n: torch.cat([r[i] for r in rows] + [pad]) for i, n in ((1, "pre"), (2, "act"))}}


def _exact_xc(c, s):
    _, idx, val = s.csr
    WT = s.W1.t().contiguous()
    acc = torch.zeros((c["batch"], c["hidden"]), device="cuda")
    for e in range(idx.shape[1]):
        acc += val[:, e][:, None] * WT[idx[:, e]]
    h64 = torch.relu((val.double()[:, :, None] * WT[idx].double()).sum(1) + s.b1.double())
    return _exact_rows(c, s, torch.relu(acc + s.b1), h64, s.W2, s.b2, "Softmax", "Reservoir")


def _exact_net(c, s):
    """Both layers' examples one by one; training updates the weights as it goes (Adam's or SGD's first step)."""
    act, train = ("Relu", "Softmax"), c["kind"] == "train"
    tables = [_buckets(_codes(s.planes[i], s.W[i]), s.bits[i], "Fifo") for i in range(2)]
    _, idx, val = s.csr
    X = torch.zeros((c["batch"], c["dim"]), dtype=torch.float64, device="cuda").scatter_(1, idx, val.double())
    W, b = [w.double() for w in s.W], [v.double() for v in s.b]
    m1, m2 = ([torch.zeros_like(w) for w in W + b] for _ in range(2))
    first = _codes(s.planes[0], X.float())
    out, loss = torch.zeros((c["batch"], c["neurons"]), dtype=torch.float64, device="cuda"), 0.0
    for r in range(c["batch"]):
        x, seen = X[r], []
        for i in range(2):
            code = first[r] if i == 0 else _codes(s.planes[1], x.float()[None])[0]
            ids, hit = _hits(tables[i], code)
            if s.sampling[i] == "TopK":
                ids = ids[np.lexsort((ids, -hit))][:s.top_k[i]]
            if not ids.size:
                ids = np.arange(W[i].shape[0])
            on, pre, a = _forward(x, W[i], b[i], ids, act[i])
            seen.append((x, on, pre, a))
            x = torch.zeros(W[i].shape[0], dtype=torch.float64, device="cuda")
            x[on] = a
        out[r] = x
        if not train:
            continue
        labels = sorted(set(s.labels[r, :int(s.n_labels[r])].tolist()))
        loss += sum(-math.log(max(float(x[v]), 1e-7)) for v in labels) / len(labels)
        grad = x.clone()
        grad[labels] -= 1.0 / len(labels)
        for i in (1, 0):
            inp, on, pre, a = seen[i]
            g = grad[on]
            lg = a * (g - (g * a).sum()) if act[i] == "Softmax" else g * (pre > 0)
            grad = lg @ W[i][on]
            for p, dw, j in ((W[i], lg[:, None] * inp[None, :], i), (b[i], lg, 2 + i)):
                if c["optimizer"] == "Adam":
                    m1[j][on] = 0.9 * m1[j][on] + (1 - 0.9) * dw
                    m2[j][on] = 0.999 * m2[j][on] + (1 - 0.999) * dw * dw
                    p[on] -= 0.001 * (m1[j][on] / (1 - 0.9)) / (torch.sqrt(m2[j][on] / (1 - 0.999)) + 1e-8)
                else:
                    m1[j][on] = 0.9 * m1[j][on] - 0.001 * dw
                    p[on] += m1[j][on]
    if not train:
        return {"out": out}
    return {"loss": loss / c["batch"], "w0": W[0], "b0": b[0], "w1": W[1], "b1": b[1]}


def _exact_layer(c, s):
    w, wb, x, d = {n: v.double() for n, v in s.w.items()}, {n: v.double() for n, v in s.wb.items()}, s.x.double(), c["dim"]
    on = torch.from_numpy(s.neurons).cuda()
    g, u = x @ w["gate"][on].t() + wb["gate"][on], x @ w["up"][on].t() + wb["up"][on]
    mlp = (g * torch.sigmoid(g) * u) @ w["down"][:, on].t() + wb["down"]
    q, k, v = ((x @ w[n].t() + wb[n]).reshape(c["batch"], c["heads"], d) for n in "qkv")
    att = torch.zeros_like(v)
    for h in s.heads:
        att[:, h] = torch.sigmoid((q[:, h] * k[:, h]).sum(1, keepdim=True) / math.sqrt(d)) * v[:, h]
    return {"mlp": mlp, "attn": att.reshape(c["batch"], -1) @ w["o"].t() + wb["o"]}


def _exact_accel(c, s):
    i, added = s.idx.long(), s.dense.double()
    added[i] += s.val.double() * 0.5
    back = _bf(s.a).reshape(-1).double()
    return {"rows": s.a.double() @ s.v.double(), "bf16": None, "back": back, "dot": back[:c["n"]] @ s.v.double(),
            "sparse": s.val.double() @ s.dense.double()[i], "added": added}


def exact(case, seed):
    c, s = case, _inputs(case, seed)
    kind = c["kind"]
    if kind == "mlp":
        return _exact_mlp(c, s)
    if kind == "attn":
        return _exact_attn(c, s)
    if kind == "slide":
        return _exact_rows(c, s, s.x, s.x.double(), s.W, s.b, "Relu", "Fifo")
    if kind == "xc":
        return _exact_xc(c, s)
    if kind in ("train", "predict"):
        return _exact_net(c, s)
    if kind == "layer":
        return _exact_layer(c, s)
    if kind == "accel":
        return _exact_accel(c, s)
    return None       # ids and counts only
