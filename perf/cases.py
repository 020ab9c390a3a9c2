"""Performance cases: the calls that an engine built on this library makes.

Each case is one kind of call at one size, made through the public entry
points (the C ABI of include/mllm.h, by way of mojollama_amd.kernels):

  host    quant_matmul_omp on host buffers, one token: the drop-in call that a
          ctypes caller makes for every matrix
  decode  a stack of transformer blocks and the output head for B sequences,
          one token each, through mllm_gemv_fused (RMSNorm into q/k/v and
          gate/up, residual adds into o and down, SiLU product in gate/up),
          replayed from a captured graph as a decode loop runs it
  matmul  one dense matrix times M tokens (prefill; 9 <= M), mllm_gemv
  moe     one routed MoE layer for T tokens (T = 1: decode of one sequence;
          tens: batched decode; hundreds and more: prefill), mllm_moe_forward
  attn    decode attention of B sequences over cached K/V, contiguous or paged
  step    one decode token through every layer of a gpt-oss model and its
          output projection, mllm_gptoss_step

Weights are raw GGUF blocks of every type that the entry points take, with
zero-mean values of standard deviation about 1/sqrt(columns), so that a stack
of matrices keeps activations of order one; activations are N(0, 1) in fp32.
"""
import ctypes
import math

import numpy as np
import torch

from mojollama_amd import kernels as K

Q4_0, Q8_0, Q4_K, Q5_K, Q6_K, MXFP4 = 2, 8, 12, 13, 14, 39
BLOCK = {Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210), MXFP4: (32, 17)}
EPS = 1e-5


def listed():
    return [
        # the drop-in call of one FFN matrix for one token (Q8_0 5632 x 2048)
        dict(name="host_q8_0", kind="host", qt=Q8_0, rows=5632, cols=2048),
        # decode of one sequence: TinyLlama-1.1B Q4_K_M blocks and its head
        dict(name="decode_b1", kind="decode", B=1, layers=4, N=2048, kv=256, M=5632, V=32000, qt=Q4_K, qt_down=Q6_K),
        # the same for a small batch, where the vector kernels hand over to the matrix cores
        dict(name="decode_b8", kind="decode", B=8, layers=4, N=2048, kv=256, M=5632, V=32000, qt=Q4_K, qt_down=Q6_K),
        # batched serving: 32 sequences, past the eight that the decode kernels take at once
        dict(name="decode_b32", kind="decode", B=32, layers=4, N=2048, kv=256, M=5632, V=32000, qt=Q4_K, qt_down=Q6_K),
        # prefill of a long prompt: the FFN gate, Q4_K
        dict(name="matmul_q4k_1280", kind="matmul", qt=Q4_K, rows=5632, cols=2048, M=1280),
        # prefill of an ordinary prompt of odd length: the FFN down projection, Q6_K
        dict(name="matmul_q6k_517", kind="matmul", qt=Q6_K, rows=2048, cols=5632, M=517),
        # prefill in a Q8_0 model (32-element blocks)
        dict(name="matmul_q8_0_256", kind="matmul", qt=Q8_0, rows=5632, cols=2048, M=256),
        # batched decode through a gpt-oss MoE layer (32 MXFP4 experts, top 4)
        dict(name="moe_gptoss_16", kind="moe", qts="39,39,39", N=2880, M=2880, E=32, K=4, T=16),
        # batched decode through a Qwen3-MoE layer (128 Q4_K / Q6_K experts, top 8)
        dict(name="moe_qwen3_64", kind="moe", qts="12,12,14", N=2048, M=768, E=128, K=8, T=64),
        # prefill through the gpt-oss MoE layer
        dict(name="moe_gptoss_1280", kind="moe", qts="39,39,39", N=2880, M=2880, E=32, K=4, T=1280),
        # decode attention of eight sequences of unequal length on 64-row pages (gpt-oss heads)
        dict(name="attn_paged_b8", kind="attn", B=8, NH=64, NKH=8, HD=64, max_seq=4096, page=64, mode=0),
        # one token through a quarter of gpt-oss-20b (6 of 24 layers, a quarter of its vocabulary), early in a
        # generation: up to seven positions every weight is an exponential, while past them mode 1's weights have
        # both signs, and where a head's sum of them comes near zero a stack of layers has no digits to compare
        dict(name="step_gptoss", kind="step", L=6, N=2880, NH=64, NKH=8, HD=64, E=32, K=4, M=2880, V=50272, ctx=1024,
             seq=6),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "decode", "decode", "matmul", "matmul", "matmul", "moe", "moe", "moe", "attn", "attn",
                       "step"])
    if kind == "host":
        return dict(kind=kind, qt=rng.choice([Q8_0, Q6_K, MXFP4]), rows=_log(rng, 256, 16384),
                    cols=256 * _log(rng, 2, 24))
    if kind == "decode":
        qt, qd = rng.choice([(Q4_K, Q6_K), (Q4_K, Q6_K), (Q8_0, Q8_0), (MXFP4, MXFP4), (Q4_0, Q4_0)])
        N = 256 * rng.randint(2, 16)
        return dict(kind=kind, B=_log(rng, 1, 64), layers=rng.randint(2, 4), N=N, kv=64 * rng.randint(1, N // 128),
                    M=256 * rng.randint(N // 256, 3 * N // 256), V=_log(rng, 1000, 40000), qt=qt, qt_down=qd)
    if kind == "matmul":
        return dict(kind=kind, qt=rng.choice([Q4_K, Q6_K, Q8_0, Q5_K, Q4_0, MXFP4]), rows=_log(rng, 256, 8192),
                    cols=256 * _log(rng, 2, 32), M=_log(rng, 9, 1280))
    if kind == "moe":
        T = _log(rng, 1, 1024)
        if rng.random() < 0.5:
            return dict(kind=kind, qts="39,39,39", N=32 * rng.randint(16, 90), M=32 * rng.randint(16, 90),
                        E=rng.randint(8, 64), K=rng.randint(2, 6), T=T)
        return dict(kind=kind, qts=rng.choice(["12,12,14", "14,14,14", "2,2,2"]), N=256 * rng.randint(2, 10),
                    M=256 * rng.randint(2, 6), E=rng.randint(8, 128), K=rng.randint(2, 8), T=T)
    if kind == "attn":
        return dict(kind=kind, B=_log(rng, 1, 32), NH=8 * (g := rng.choice([1, 2, 4, 8])), NKH=rng.choice([8, 4 * g]),
                    HD=rng.choice([64, 64, 128]), max_seq=_log(rng, 48, 6000), page=rng.choice([0, 16, 64]),
                    mode=rng.choice([0, 1]))
    return dict(kind=kind, L=rng.randint(2, 5), N=32 * rng.randint(32, 90), NH=64, NKH=8, HD=64,
                E=rng.randint(8, 32), K=rng.randint(2, 4), M=32 * rng.randint(32, 90), V=_log(rng, 4000, 60000),
                ctx=1024, seq=rng.randint(0, 6))


# ------------------------------------------------------------------ weights
def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFFFFFFFFF)


def _f16(v):
    return v.to(torch.float16).view(torch.uint8).view(-1, 2)


def _weights(g, qt, rows, cols):
    """Raw GGUF blocks (uint8, GPU) of a rows x cols matrix of zero-mean values."""
    be, bb = BLOCK[qt]
    nb = rows * (cols // be)
    blk = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, device="cuda", generator=g)
    s = (0.5 + torch.rand(nb, device="cuda", generator=g)) / math.sqrt(cols)   # target deviation of the block
    if qt == Q4_0:
        blk[:, 0:2] = _f16(s / 4.6)
    elif qt == Q8_0:
        blk[:, 0:2] = _f16(s / 73.6)
    elif qt in (Q4_K, Q5_K):
        # scales 0..63, minima that centre the codes: dmin * m = d * sc * mean code
        d = (s / (36.0 * (4.6 if qt == Q4_K else 9.2))).to(torch.float16).float()
        sc = torch.randint(0, 64, (nb, 8), device="cuda", generator=g)
        m = torch.round(sc * 7.5 / 8).long() if qt == Q4_K else torch.round(sc * 15.5 / 16).long()
        q = torch.zeros(nb, 12, dtype=torch.long, device="cuda")
        q[:, 0:4] = sc[:, 0:4] | ((sc[:, 4:8] >> 4) << 6)
        q[:, 4:8] = m[:, 0:4] | ((m[:, 4:8] >> 4) << 6)
        q[:, 8:12] = (sc[:, 4:8] & 15) | ((m[:, 4:8] & 15) << 4)
        blk[:, 0:2] = _f16(d)
        blk[:, 2:4] = _f16(d * (8 if qt == Q4_K else 16))
        at = 4 if qt == Q4_K else 164
        blk[:, at:at + 12] = q.to(torch.uint8)
    elif qt == Q6_K:
        blk[:, 192:208] = torch.randint(-32, 32, (nb, 16), dtype=torch.int8, device="cuda", generator=g).view(torch.uint8)
        blk[:, 208:210] = _f16(s / (18.5 * 18.5))
    elif qt == MXFP4:
        e = torch.randint(-3, 2, (nb,), device="cuda", generator=g) + int(round(math.log2(1 / (4.6 * math.sqrt(cols)))))
        blk[:, 16] = (127 + e).to(torch.uint8)
    return blk.reshape(-1)


def _h(b):
    return b.contiguous().view(torch.float16).to(torch.float64)


def _k4(q):
    """The eight 6-bit (scale, minimum) pairs of 12 bytes, [nb][8] each."""
    q = q.long()
    sc = torch.cat([q[:, 0:4] & 63, (q[:, 8:12] & 15) | ((q[:, 0:4] >> 6) << 4)], 1)
    m = torch.cat([q[:, 4:8] & 63, (q[:, 8:12] >> 4) | ((q[:, 4:8] >> 6) << 4)], 1)
    return sc.double(), m.double()


def _nibbles(b):
    """[nb][n] bytes -> [nb][2n] codes, low nibble first."""
    b = b.long()
    return torch.stack([b & 15, b >> 4], -1).reshape(b.shape[0], -1)


def _dequant(qt, raw, rows, cols, lownib=False):
    """The weights in 64 bits: [rows][cols].  lownib: Q6_K as the MoE entry
    points read it (every quadrant from the low nibble); else its sequential order."""
    be, bb = BLOCK[qt]
    b = raw.view(-1, bb)
    if qt == Q4_0:
        q = b[:, 2:].long()
        w = (torch.cat([q & 15, q >> 4], 1) - 8).double() * _h(b[:, 0:2])
    elif qt == Q8_0:
        w = b[:, 2:].contiguous().view(torch.int8).double() * _h(b[:, 0:2])
    elif qt == Q4_K:
        sc, m = _k4(b[:, 4:16])
        q = b[:, 16:].long().view(-1, 4, 32)
        c = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        w = c * (_h(b[:, 0:2]) * sc)[:, :, None] - (_h(b[:, 2:4]) * m)[:, :, None]
    elif qt == Q5_K:   # the batch entry point's own layout: d, dmin, qh[32], ql[128], scales[12]
        sc, m = _k4(b[:, 164:176])
        hi = ((b[:, 4:36].long()[:, :, None] >> torch.arange(8, device=raw.device)) & 1).reshape(-1, 256)
        c = (_nibbles(b[:, 36:164]) | (hi << 4)).double().view(-1, 8, 32)
        w = c * (_h(b[:, 0:2]) * sc)[:, :, None] - (_h(b[:, 2:4]) * m)[:, :, None]
    elif qt == Q6_K:
        d = _h(b[:, 208:210])
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        qh = b[:, 128:192].long()
        if not lownib:
            hi = ((qh[:, :, None] >> (2 * torch.arange(4, device=raw.device))) & 3).reshape(-1, 256)
            w = ((_nibbles(b[:, 0:128]) | (hi << 4)) - 32).double().view(-1, 16, 16) * (d * sc)[:, :, None]
        else:
            ql = (b[:, 0:128].long() & 15).view(-1, 2, 2, 32)                       # [half][Q & 1][l]
            low = torch.cat([ql, ql], 2)                                             # [half][Q][l]
            hi = (qh.view(-1, 2, 1, 32) >> (2 * torch.arange(4, device=raw.device)).view(1, 1, 4, 1)) & 3
            s = sc.view(-1, 2, 4, 2).repeat_interleave(16, 3)                        # sc[8 half + l/16 + 2 Q]
            w = ((low | (hi << 4)) - 32).double() * s * d.view(-1, 1, 1, 1)
    else:
        v = _nibbles(b[:, 0:16])
        w = torch.where(v >= 8, v - 16, v).double() * torch.exp2(b[:, 16:17].double() - 127)
    return w.reshape(rows, cols)


def _q8(x):
    """The Q8_0 activations of x [n][cols] fp32: codes and fp16 scales, in 64 bits."""
    v = x.float().view(x.shape[0], -1, 32)
    d = v.abs().amax(-1, keepdim=True) / 127.0
    d = torch.where(d == 0, torch.ones_like(d), d)
    q = torch.round((v * (1.0 / d)).clamp(-127, 127))
    return q.double(), d.to(torch.float16).double()


def _dot(qt, entry, raw, rows, cols, x):
    """W x for the tokens of x [n][cols], in 64 bits, as the entry point
    defines it: "batch" (*_batch_matmul), "qmm" (quant_matmul_omp and the MoE
    gate / up rows) or "down" (the MoE down rows)."""
    if entry == "qmm" and qt == Q4_K:
        # the Q8_0-activation dot: codes of elements k < 16 of each sub-block, minima over k in 0-7 and 16-23
        b = raw.view(rows, -1, 144)
        nb = b.shape[1]
        flat = b.reshape(-1, 144)
        sc, _ = _k4(flat[:, 4:16])
        q = flat[:, 16:].long().view(-1, 4, 32)
        c = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32)[:, :, :16].double()
        w = (c * sc[:, :, None] * _h(flat[:, 0:2])[:, :, None]).reshape(rows, -1)
        xq, xd = _q8(x)
        xs = xq[:, :, :16].reshape(x.shape[0], -1)
        mins = (xd[:, :, 0] * (xq[:, :, 0:8].sum(-1) + xq[:, :, 16:24].sum(-1))).view(x.shape[0], nb, 8).sum(-1)
        return xs @ w.T - mins @ _h(flat[:, 2:4]).view(rows, nb).T
    w = _dequant(qt, raw, rows, cols, lownib=entry != "batch")
    if entry == "down" and qt == MXFP4:
        q, d = _q8(x)
        return (q * d).view(x.shape[0], -1) @ w.T
    return x.double() @ w.T


def _bytes(qt, rows, cols):
    be, bb = BLOCK[qt]
    return rows * (cols // be) * bb


# -------------------------------------------------------------------- cases
def _ops():
    return K.DeviceOps()


def _host_inputs(c, seed):
    g = _gen(seed)
    return _weights(g, c["qt"], c["rows"], c["cols"]), torch.randn(c["cols"], device="cuda", generator=g)


def _decode_inputs(c, seed):
    g = _gen(seed)
    N, kv, M = c["N"], c["kv"], c["M"]
    norm = lambda: 1 + 0.1 * torch.randn(N, device="cuda", generator=g)  # noqa: E731
    layers = [dict(qkv=_weights(g, c["qt"], N + 2 * kv, N), o=_weights(g, c["qt"], N, N),
                   gate_up=_weights(g, c["qt"], 2 * M, N), down=_weights(g, c["qt_down"], N, M), an=norm(), fn=norm())
              for _ in range(c["layers"])]
    head = _weights(g, c["qt_down"], c["V"], N)
    return layers, head, norm(), torch.randn(c["B"], N, device="cuda", generator=g)


def _moe_inputs(c, seed):
    g = _gen(seed)
    qts = [int(q) for q in c["qts"].split(",")]
    E, N, M = c["E"], c["N"], c["M"]
    mats = [[_weights(g, qt, *(s)) for _ in range(E)] for qt, s in zip(qts, ((M, N), (M, N), (N, M)))]
    router = torch.randn(E, N, device="cuda", generator=g) * 0.02
    return qts, mats, router, torch.randn(c["T"], N, device="cuda", generator=g)


def _attn_inputs(c, seed):
    g = _gen(seed)
    B, S, row = c["B"], c["max_seq"], c["NKH"] * c["HD"]
    page = c["page"]
    blocks = -(-S // page) if page else 0
    rows = B * blocks * page if page else B * S
    k = torch.randn(rows, row, device="cuda", generator=g)
    v = torch.randn(rows, row, device="cuda", generator=g)
    q = torch.randn(B, c["NH"] * c["HD"], device="cuda", generator=g)
    tables = torch.randperm(B * blocks, device="cuda", generator=g).to(torch.int32).view(B, blocks) if page else None
    # sequences of a running batch: between half and the whole of the longest
    lens = (S - torch.randint(0, S // 2 + 1, (B,), device="cuda", generator=g)).to(torch.int32)
    lens[0] = S
    return q, k, v, tables, lens


def _step_inputs(c, seed):
    g = _gen(seed)
    L, N, E, M = c["L"], c["N"], c["E"], c["M"]
    inner, kvd = c["NH"] * c["HD"], c["NKH"] * c["HD"]
    n = L - 1 + E   # expert e of layer l is matrix l + e
    w = dict(wQ=[_weights(g, MXFP4, inner, N) for _ in range(L)], wK=[_weights(g, MXFP4, kvd, N) for _ in range(L)],
             wV=[_weights(g, MXFP4, kvd, N) for _ in range(L)], wO=[_weights(g, MXFP4, N, inner) for _ in range(L)],
             w_gate_exps=[_weights(g, MXFP4, M, N) for _ in range(n)],
             w_up_exps=[_weights(g, MXFP4, M, N) for _ in range(n)],
             w_down_exps=[_weights(g, MXFP4, N, M) for _ in range(n)], wOut=[_weights(g, MXFP4, c["V"], N)])
    f = lambda *s, sc=1.0: torch.randn(*s, device="cuda", generator=g) * sc  # noqa: E731
    w.update(wAN=[1 + f(N, sc=0.1) for _ in range(L)], wFN=[1 + f(N, sc=0.1) for _ in range(L)],
             w_gate_inp=[f(E, N, sc=0.02) for _ in range(L)])
    j = torch.arange(c["HD"] // 2, device="cuda", dtype=torch.float64)
    th = torch.arange(c["ctx"], device="cuda", dtype=torch.float64)[:, None] / 10000.0 ** (2 * j / c["HD"])
    w["cos_t"], w["sin_t"] = [th.cos().float()], [th.sin().float()]
    kc, vc = f(L, c["ctx"], kvd), f(L, c["ctx"], kvd)
    return w, kc, vc, f(N)


class _Model:
    """A gpt-oss model handle (mllm_gptoss_create), released with the state."""

    def __init__(self, so, c, w):
        host = {k: [t.cpu().numpy() for t in v] for k, v in w.items()}
        ptr = lambda a: a.ctypes.data_as(K.cu if a.dtype == np.uint8 else K.cf)  # noqa: E731
        arr = {}
        for k, v in host.items():
            arr[k] = ptr(v[0]) if k in ("wOut", "cos_t", "sin_t") else \
                ((K.cu if v[0].dtype == np.uint8 else K.cf) * len(v))(*[ptr(a) for a in v])
        d = K.GptOssDesc(L=c["L"], N=c["N"], NH=c["NH"], NKH=c["NKH"], HD=c["HD"], E=c["E"], K=c["K"], M=c["M"],
                         max_ctx=c["ctx"], rope_dim=c["HD"], outNR=c["V"], eps=EPS, qt_gate=MXFP4, qt_up=MXFP4,
                         qt_down=MXFP4, **arr)
        self.so, self.h = so, so.mllm_gptoss_create(ctypes.byref(d))
        if not self.h:
            raise RuntimeError("mllm_gptoss_create: " + K.last_error(so))

    def __del__(self):
        if getattr(self, "h", None):
            torch.cuda.synchronize()
            self.so.mllm_gptoss_release(self.h)


def prepare(case, seed):
    c, kind, ops = case, case["kind"], _ops()
    if kind == "host":
        w, x = _host_inputs(c, seed)
        return dict(c=c, so=ops.so, W=w.cpu().numpy(), x=x.cpu().numpy(), out=np.zeros(c["rows"], np.float32))
    if kind == "decode":
        layers, head, on, x = _decode_inputs(c, seed)
        B, N, kv, M = c["B"], c["N"], c["kv"], c["M"]
        sem, sem_d = (ops.so.mllm_sem_for(K.ENT_BMM, q) for q in (c["qt"], c["qt_down"]))
        z = lambda n: torch.zeros(B, n, device="cuda")  # noqa: E731
        xa, xb, qkv, q, h, logits = z(N), z(N), z(N + 2 * kv), z(N), z(M), z(c["V"])
        calls, keep = [], []

        def add(sm, raw, rows, cols, inp, out, raw_rows=None, **fuse):
            p = ops.pack(sm, raw, raw_rows or rows, cols)
            f = ops.fusion(**fuse)
            n = ops.so.mllm_gemv_fused_workspace_size(sm, rows, cols, B, ctypes.byref(f))
            keep.append((fuse, n))
            calls.append((sm, p, inp, rows, cols, f, out))
        for L in layers:
            add(sem, L["qkv"], N + 2 * kv, N, xa, qkv, rms_w=L["an"], rms_eps=EPS)
            if B <= 8:   # q read in place from the stacked rows
                add(sem, L["o"], N, N, qkv.data_ptr(), xb, out_add=xa, x_ld=N + 2 * kv)
            else:
                add(sem, L["o"], N, N, q, xb, out_add=xa)
            add(sem, L["gate_up"], M, N, xb, h, raw_rows=2 * M, rms_w=L["fn"], rms_eps=EPS, silu_pair=True,
                silu_clamp=False)
            add(sem_d, L["down"], N, M, h, xa, out_add=xb)
        add(sem_d, head, c["V"], N, xa, logits, rms_w=on, rms_eps=EPS)
        ws = torch.empty(max([256] + [n for _, n in keep]), dtype=torch.uint8, device="cuda")

        def step():
            xa.copy_(x)
            for sm, p, inp, rows, cols, f, out in calls:
                if inp is q:
                    q.copy_(qkv[:, :N])
                ops.gemv_fused(sm, p, inp, rows, cols, f, out=out, ws=ws, B=B)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step()
        return dict(c=c, graph=graph, out=dict(hidden=xa, logits=logits), keep=(x, xb, qkv, q, h, ws, calls, keep))
    if kind == "matmul":
        g = _gen(seed)
        sem = ops.so.mllm_sem_for(K.ENT_BMM, c["qt"])
        packed = ops.pack(sem, _weights(g, c["qt"], c["rows"], c["cols"]), c["rows"], c["cols"])
        x = torch.randn(c["M"], c["cols"], device="cuda", generator=g)
        return dict(c=c, ops=ops, sem=sem, packed=packed, x=x, out=torch.empty(c["M"], c["rows"], device="cuda"),
                    ws=ops.workspace(sem, c["cols"], c["M"], x.device, c["rows"]))
    if kind == "moe":
        qts, mats, router, x = _moe_inputs(c, seed)
        layer = ops.moe_prepare(qts, c["N"], c["M"], c["E"], c["K"], *mats, router, 1)
        layer.workspace(c["T"])
        return dict(c=c, layer=layer, x=x, out=torch.empty(c["T"], c["N"], device="cuda"))
    if kind == "attn":
        q, k, v, tables, lens = _attn_inputs(c, seed)
        S, row = c["max_seq"], c["NKH"] * c["HD"]
        view = ops.kv_view(k, v, block_tables=tables, page_size=c["page"], n_pages=tables.numel()) if c["page"] else \
            ops.kv_view(k, v, seq_stride=S * row)
        ws = torch.empty(ops.so.mllm_gqa_workspace_size(c["B"], c["NH"], c["HD"], S), dtype=torch.uint8, device="cuda")
        return dict(c=c, ops=ops, q=q, kv=view, lens=lens, out=torch.empty_like(q), ws=ws)
    w, kc, vc, x = _step_inputs(c, seed)
    model = _Model(ops.so, c, w)
    seq = torch.full((c["L"],), c["seq"], dtype=torch.int32, device="cuda")
    return dict(c=c, ops=ops, model=model, kc=kc, vc=vc, x=x, seq=seq, lens=seq.clone(), pos=seq[:1].clone(),
                logits=torch.empty(c["V"], device="cuda"))


def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind == "host":
        s["so"].quant_matmul_omp(s["W"].ctypes.data_as(K.cu), s["x"].ctypes.data_as(K.cf),
                                 s["out"].ctypes.data_as(K.cf), c["rows"], c["cols"], c["qt"])
        return s["out"]
    if kind == "decode":
        s["graph"].replay()
        return s["out"]
    if kind == "matmul":
        return s["ops"].gemv(s["sem"], s["packed"], s["x"], c["rows"], c["cols"], out=s["out"], ws=s["ws"])
    if kind == "moe":
        return s["layer"].forward(s["x"], out=s["out"])
    if kind == "attn":
        return s["ops"].gqa_decode(c["mode"], s["q"], s["kv"], s["lens"], c["max_seq"], c["NH"], c["NKH"], c["HD"],
                                   out=s["out"], ws=s["ws"])
    s["lens"].copy_(s["seq"])   # the caller's sequence length of this step
    o = s["ops"]
    o._check(o.so.mllm_gptoss_step(s["model"].h, s["x"].data_ptr(), s["pos"].data_ptr(), s["lens"].data_ptr(),
                                   s["kc"].data_ptr(), s["vc"].data_ptr(), s["logits"].data_ptr(), o._stream()),
             "mllm_gptoss_step")
    return dict(logits=s["logits"], lens=s["lens"], k=s["kc"], v=s["vc"])


def work(case):
    c, kind = case, case["kind"]
    if kind in ("host", "matmul"):
        n = c.get("M", 1)
        return dict(bytes=_bytes(c["qt"], c["rows"], c["cols"]) + 4 * n * (c["rows"] + c["cols"]),
                    flops=2 * n * c["rows"] * c["cols"])
    if kind == "decode":
        N, kv, M, V, B = c["N"], c["kv"], c["M"], c["V"], c["B"]
        per = _bytes(c["qt"], N + 2 * kv, N) + _bytes(c["qt"], N, N) + _bytes(c["qt"], 2 * M, N) + \
            _bytes(c["qt_down"], N, M)
        el = c["layers"] * ((2 * N + 2 * kv) * N + 3 * M * N) + V * N
        return dict(bytes=c["layers"] * per + _bytes(c["qt_down"], V, N) + 4 * B * (2 * N + V), flops=2 * B * el)
    if kind == "moe":
        N, M, E, k, T = (c[n] for n in ("N", "M", "E", "K", "T"))
        qts = [int(q) for q in c["qts"].split(",")]
        per = _bytes(qts[0], M, N) + _bytes(qts[1], M, N) + _bytes(qts[2], N, M)
        touched = E * (1 - (1 - k / E) ** T)
        return dict(bytes=touched * per + 4 * E * N + 8 * T * N, flops=2 * T * (k * 3 * M * N + E * N))
    if kind == "attn":
        S = c["max_seq"]
        rows = S + (c["B"] - 1) * (S - S // 4)   # the mean length of the others
        return dict(bytes=8 * rows * c["NKH"] * c["HD"] + 8 * c["B"] * c["NH"] * c["HD"],
                    flops=4 * rows * c["NH"] * c["HD"])
    L, N, M, E, k, V = (c[n] for n in ("L", "N", "M", "E", "K", "V"))
    inner, kvd = c["NH"] * c["HD"], c["NKH"] * c["HD"]
    el = L * ((inner + 2 * kvd) * N + N * inner + 3 * k * M * N) + V * N
    return dict(bytes=_bytes(MXFP4, el // 32, 32) + L * (4 * E * N + 8 * (c["seq"] + 1) * kvd) + 4 * (N + V),
                flops=2 * el + L * (2 * E * N + 4 * (c["seq"] + 1) * inner))


def tolerance(case):
    """Relative 2-norm errors, about four times what the path shows against
    64 bits.  A value that the path quantises to Q8_0 on the way (the MXFP4
    MoE down projection) moves by a whole code where two sums round apart;
    mode 1 attention weights are steps of the score."""
    kind = case["kind"]
    if kind == "moe":
        return dict(rel=1e-3, max=0.1) if case["qts"].endswith("39") else dict(rel=1e-5, max=5e-4)
    if kind == "step":
        return dict(rel=1e-3, max=0.1)
    if kind == "attn":
        return dict(rel=1e-3, max=0.3) if case["mode"] == 1 else dict(rel=3e-6, max=2e-4)
    if kind == "decode":
        return dict(rel=2e-5, max=1e-3)
    return dict(rel=2e-5, max=1e-3)


# -------------------------------------------------------- the same in 64 bits
def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _route(router, x, k):
    p = torch.softmax(x.double() @ router.double().T, -1)
    v, i = p.topk(k, -1)
    return v / (v.sum(-1, keepdim=True) + 1e-10), i


def _experts(qts, mats, x, wt, idx, N, M):
    """sum_k w_k down_e(silu(gate_e x) * up_e x) with the gate clamped to +-80."""
    out = torch.zeros(x.shape[0], N, dtype=torch.float64, device=x.device)
    for e in range(len(mats[0])):
        t, slot = (idx == e).nonzero(as_tuple=True)
        if not t.numel():
            continue
        g = _dot(qts[0], "qmm", mats[0][e], M, N, x[t]).clamp(-80, 80)
        h = g / (1 + torch.exp(-g)) * _dot(qts[1], "qmm", mats[1][e], M, N, x[t])
        out.index_add_(0, t, wt[t, slot][:, None] * _dot(qts[2], "down", mats[2][e], N, M, h))
    return out


def _exp_steps(z):
    """The vector loop's weight of mode 1 (the reference's exp_ps_simd) on z <= 0, in 64 bits."""
    t = z.clamp(-80, 80) * float(np.float32(1.4426950408889634))
    n = torch.round(t + 0.5)
    f, p = t - n, torch.ones_like(t)
    for a in (0.6931471805599453, 0.2402265069591007, 0.0555041086648216, 0.0096181291076285, 0.0013333558146428):
        p = p * f + float(np.float32(a))
    return p * torch.exp2(n)


def _attend(mode, q, k, v):
    """One sequence: q [NH][HD], k and v [S][NKH][HD], 64 bits."""
    S, NKH, HD = k.shape
    G = q.shape[0] // NKH
    s = torch.matmul(q.view(NKH, G, HD), k.permute(1, 2, 0).contiguous()) / math.sqrt(HD)
    z = s - s.amax(-1, keepdim=True)
    e = torch.exp(z)
    if mode == 1:
        e[:, :, :S // 8 * 8] = _exp_steps(z[:, :, :S // 8 * 8])
    o = torch.matmul(e, v.permute(1, 0, 2).contiguous()) / (e.sum(-1, keepdim=True) + (1e-10 if mode == 1 else 0.0))
    return o.reshape(-1)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "host":
        w, x = _host_inputs(c, seed)
        return _dot(c["qt"], "qmm", w, c["rows"], c["cols"], x[None])[0].cpu().numpy()
    if kind == "decode":
        layers, head, on, x = _decode_inputs(c, seed)
        N, kv, M = c["N"], c["kv"], c["M"]
        x = x.double()
        for L in layers:
            qkv = _dot(c["qt"], "batch", L["qkv"], N + 2 * kv, N, _rms(x, L["an"]))
            x = x + _dot(c["qt"], "batch", L["o"], N, N, qkv[:, :N])
            gu = _dot(c["qt"], "batch", L["gate_up"], 2 * M, N, _rms(x, L["fn"]))
            x = x + _dot(c["qt_down"], "batch", L["down"], N, M, torch.nn.functional.silu(gu[:, :M]) * gu[:, M:])
        return dict(hidden=x, logits=_dot(c["qt_down"], "batch", head, c["V"], N, _rms(x, on)))
    if kind == "matmul":
        g = _gen(seed)
        w = _weights(g, c["qt"], c["rows"], c["cols"])
        return _dot(c["qt"], "batch", w, c["rows"], c["cols"],
                    torch.randn(c["M"], c["cols"], device="cuda", generator=g))
    if kind == "moe":
        qts, mats, router, x = _moe_inputs(c, seed)
        return _experts(qts, mats, x, *_route(router, x, c["K"]), c["N"], c["M"])
    if kind == "attn":
        q, k, v, tables, lens = _attn_inputs(c, seed)
        out = []
        for b in range(c["B"]):
            n = int(lens[b])
            p = torch.arange(n, device="cuda")
            r = tables[b].long()[p // c["page"]] * c["page"] + p % c["page"] if c["page"] else b * c["max_seq"] + p
            out.append(_attend(c["mode"], q[b].double().view(c["NH"], -1), k[r].double().view(n, c["NKH"], -1),
                               v[r].double().view(n, c["NKH"], -1)))
        return torch.stack(out)
    w, kc, vc, x = _step_inputs(c, seed)
    N, M, HD, NH, NKH, n = c["N"], c["M"], c["HD"], c["NH"], c["NKH"], c["seq"]
    kc, vc = kc.double(), vc.double()
    x = x.double()[None]
    cs, sn = w["cos_t"][0][n].double(), w["sin_t"][0][n].double()

    def rope(t):
        a, b = t[:, :HD // 2], t[:, HD // 2:]
        return torch.cat([a * cs - b * sn, b * cs + a * sn], 1)
    qts = (MXFP4, MXFP4, MXFP4)
    for i in range(c["L"]):
        xn = _rms(x, w["wAN"][i])
        q, k, v = (_dot(MXFP4, "qmm", w[m][i], r * HD, N, xn).view(r, HD)
                   for m, r in (("wQ", NH), ("wK", NKH), ("wV", NKH)))
        kc[i, n], vc[i, n] = rope(k).reshape(-1), v.reshape(-1)
        o = _attend(1, rope(q), kc[i, :n + 1].view(-1, NKH, HD), vc[i, :n + 1].view(-1, NKH, HD))
        att = x + _dot(MXFP4, "qmm", w["wO"][i], N, NH * HD, o[None])
        fn = _rms(att, w["wFN"][i])
        mats = [w[m][i:i + c["E"]] for m in ("w_gate_exps", "w_up_exps", "w_down_exps")]
        # the reference adds the FFN to the layer's input, and projects the last FFN-norm output
        x = x + _experts(qts, mats, fn, *_route(w["w_gate_inp"][i], fn, c["K"]), N, M)
    return dict(logits=_dot(MXFP4, "qmm", w["wOut"][0], c["V"], N, fn)[0], lens=None, k=kc, v=vc)
