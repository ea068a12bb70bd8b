"""The calls whose speed is measured: whole training steps and generation
through sejong_amd.model, and the single blocks a caller of the C ABI
(include/sejong_hip.h) drives itself: a feed-forward block, an attention
block, the output head with the loss, the optimizer update, a
mixture-of-experts block and the parameter-VJP update of a projection.

torch is imported first: the library then runs on torch's HIP runtime and
shares its devices and pointers.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from sejong_amd import _native as N
from sejong_amd import model as SM

BF, F32 = N.SJ_BF16, N.SJ_F32
DEV = "cuda"
EPS = 1e-6
THETA = 10000.0
V, VP = SM.VOCAB, (SM.VOCAB + 7) // 8 * 8


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the smallest real training step: one fp32 block on short sequences
        # (latency of about thirty launches; sj_gemm and the row kernels)
        dict(name="step_f32_small", kind="step", precision="f32", layers=1, heads=4, kv=2, head_dim=32, ffn=384,
             T=128, B=2, hier=False),
        # the benchmark's training step: 6 layers, 4096 tokens, AdamW, one graph
        dict(name="step_bf16", kind="step", precision="bf16", layers=6, heads=6, kv=2, head_dim=64, ffn=1024, T=512,
             B=8, hier=False),
        # the hierarchical training step: byte encoder and decoder of window
        # 128 around 8 global layers over patches of 4, 8192 bytes
        dict(name="step_hier", kind="step", precision="bf16", layers=8, heads=8, kv=2, head_dim=64, ffn=1376, T=1024,
             B=8, hier=True),
        # interactive use: a prompt, then one token at a time, each token's
        # logits read by the host that picks the next one
        dict(name="generate", kind="generate", layers=6, heads=6, kv=2, ffn=1024, prompt=200, new=24),
        # feed-forward block, forward and backward, at a ragged small size
        dict(name="ffn_ragged", kind="ffn", M=1000, D=384, F=1000),
        # the same at the large configuration: 16384 tokens
        dict(name="ffn_large", kind="ffn", M=16384, D=1024, F=2752),
        # attention block, forward and backward: the local windowed stage with
        # one query head per KV head
        dict(name="attn_window", kind="attn", B=8, T=1024, heads=4, kv=4, window=128),
        # grouped causal attention at the large configuration
        dict(name="attn_large", kind="attn", B=16, T=1024, heads=16, kv=4, window=0),
        # final norm, vocabulary head, cross entropy and their backward through
        # the reference-layout calls (fp32 gradients and master weights)
        dict(name="head", kind="head", M=4096, D=384),
        # gradient norm, clip and AdamW over a flat parameter arena
        dict(name="adamw", kind="adamw", n=9639552),
        # mixture of experts: routing, grouped products and their backward
        dict(name="moe", kind="moe", M=4096, D=512, E=8, K=2, F=1024),
        # parameter VJP of the gate|up projection at the large configuration:
        # selection, basis, factors, and the selected-row SGD update
        dict(name="pvjp", kind="pvjp", M=16384, D=1024, F=2752, rank=16, fraction=0.1),
    ]


def _log(rng, lo, hi, step=1):
    """A size between lo and hi, uniform in its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(-(-lo // step) * step, min(hi // step * step, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["step", "step", "generate", "ffn", "ffn", "attn", "attn", "head", "adamw", "moe", "pvjp"])
    if kind == "step":
        if rng.random() < 0.4:
            heads, kv, hd = rng.choice([(4, 2, 32), (4, 4, 16), (2, 1, 64), (8, 4, 32), (4, 2, 64), (8, 8, 32),
                                        (6, 2, 64), (8, 4, 64)])
            return dict(kind=kind, precision="f32", layers=rng.randint(1, 4), heads=heads, kv=kv, head_dim=hd,
                        ffn=_log(rng, 96, 1024), T=_log(rng, 24, 320), B=rng.randint(1, 6), hier=False)
        heads, kv = rng.choice([(2, 1), (2, 2), (4, 1), (4, 2), (6, 2), (6, 3), (8, 2), (8, 8), (9, 3), (12, 4)])
        T = _log(rng, 64, 1024, 64) if rng.random() < 0.8 else _log(rng, 60, 500, 4)
        B = max(1, min(12, int(4500 / T * rng.uniform(0.1, 1.0))))
        return dict(kind=kind, precision="bf16", layers=rng.randint(1, 5), heads=heads, kv=kv, head_dim=64,
                    ffn=_log(rng, 128, 2048, 8), T=T, B=B, hier=False)
    if kind == "generate":
        heads, kv = rng.choice([(2, 1), (4, 2), (6, 2), (8, 2), (8, 8), (12, 4), (16, 4)])
        return dict(kind=kind, layers=rng.randint(1, 12), heads=heads, kv=kv, ffn=_log(rng, 256, 2816, 8),
                    prompt=_log(rng, 1, 900), new=rng.randint(8, 32))
    if kind == "ffn":
        M, D = _log(rng, 16, 16384), _log(rng, 64, 1024, 8)
        return dict(kind=kind, M=M, D=D, F=_log(rng, 128, 2752, 8))
    if kind == "attn":
        heads, kv = rng.choice([(2, 1), (2, 2), (3, 1), (4, 4), (6, 2), (8, 2), (8, 4), (12, 4), (16, 4), (16, 16)])
        T = _log(rng, 64, 2048, 64)
        B = max(1, min(16, int(16384 / T * rng.uniform(0.05, 1.0))))
        return dict(kind=kind, B=B, T=T, heads=heads, kv=kv, window=rng.choice([0, 0, 0, 100, 128, 256]))
    if kind == "head":
        return dict(kind=kind, M=_log(rng, 32, 16384), D=_log(rng, 64, 1024, 8))
    if kind == "adamw":
        return dict(kind=kind, n=_log(rng, 1000, 60000000))
    if kind == "moe":
        E = rng.choice([2, 4, 8, 8, 8, 16])
        return dict(kind=kind, M=_log(rng, 64, 8192), D=_log(rng, 128, 1024, 64), E=E, K=rng.choice([1, 2, 2, min(4, E)]),
                    F=_log(rng, 128, 1024, 8))
    return dict(kind=kind, M=_log(rng, 512, 16384, 8), D=_log(rng, 128, 1024, 8), F=_log(rng, 256, 2752, 8),
                rank=rng.choice([8, 16, 16, 32]), fraction=rng.choice([0.1, 0.25]))


# ---------------------------------------------------------------- helpers

class _Device:
    """A device buffer of a model as torch sees it; the tensor made of it
    holds this object, and so the model that owns the memory."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(ptr, False), version=3,
                                             strides=None)


def _view(model, what, shape=None):
    ptr, n = model.buffer(what)
    return torch.as_tensor(_Device(model, ptr, shape or (n,), "<f4"), device=DEV)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _p(t, elements=0):
    return None if t is None else ctypes.c_void_p(t.data_ptr() + elements * t.element_size())


def _planes(x):
    """fp32 -> (hi, lo) bf16 planes."""
    hi = x.to(torch.bfloat16)
    return hi, (x - hi.float()).to(torch.bfloat16)


class _S:
    """What a case's program holds."""


class _Out(dict):
    """Outputs that are a model's own buffers, with the model that owns them."""
    model = None


def _normal(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device=DEV)


def _bytes(n):
    return torch.zeros(max(int(n), 256), dtype=torch.uint8, device=DEV)


def _configs(c):
    if c["kind"] == "generate":
        mc = SM.ModelConfig(width=64 * c["heads"], layers=c["layers"], heads=c["heads"], kv_heads=c["kv"],
                            ffn_width=c["ffn"], context=1024, precision="bf16", norm_epsilon=EPS)
        return mc, SM.TrainConfig(sequence=64, batch=1)
    h = None
    if c["hier"]:
        h = SM.HierarchyConfig(patch_size=4, encoder_width=256, encoder_layers=2, encoder_heads=4,
                               encoder_ffn_width=768, decoder_width=256, decoder_layers=2, decoder_heads=4,
                               decoder_ffn_width=768, local_window=128)
    mc = SM.ModelConfig(width=c["heads"] * c["head_dim"], layers=c["layers"], heads=c["heads"], kv_heads=c["kv"],
                        ffn_width=c["ffn"], context=c["T"], precision=c["precision"], norm_epsilon=EPS, hierarchy=h)
    return mc, SM.TrainConfig(sequence=c["T"], batch=c["B"], learning_rate=3e-4, weight_decay=0.01, epsilon=1e-8)


def _params(mc, seed):
    """Flat fp32 masters in the reference order: N(0, 0.02) matrices, norms near 1."""
    g = _gen(seed)
    flat = torch.randn(SM.param_count(mc), generator=g, device=DEV) * 0.02
    o = 0
    for name, shape, norm in SM.layout(mc):
        n = math.prod(shape)
        if norm:
            flat[o:o + n] = 1.0 + 5.0 * flat[o:o + n]
        o += n
    return flat.cpu().numpy()


def _tokens(seed, batch, T):
    """Text-like bytes: the low codes are drawn more often."""
    g = _gen(seed * 7 + 1)
    r = torch.rand(batch, T + 1, generator=g, device=DEV)
    t = (r * r * 256.0).to(torch.int32).clamp(0, 255)
    return t[:, :-1].reshape(-1).contiguous(), t[:, 1:].reshape(-1).contiguous()


def _rope_table(T, hd):
    t = _empty(T, hd)
    N.api.sj_rope_table(None, _p(t), T, hd, ctypes.c_float(THETA))
    return t


# ---------------------------------------------------------------- prepare

def prepare(case, seed):
    N.load()
    s = _S()
    s.kind, s.c = case["kind"], case
    globals()["_prepare_" + s.kind](s, case, seed)
    if s.kind not in ("step", "generate"):
        s.calls = _Calls()
        s.out = globals()["_calls_" + s.kind](s, s.calls)
    torch.cuda.synchronize()
    return s


def run(s):
    if s.kind == "step":
        return _run_step(s)
    if s.kind == "generate":
        return _run_generate(s)
    check = N.check
    for fn, args in s.calls.all:
        check(fn(*args))
    return s.out


class _Calls:
    """The C ABI calls of a block with their arguments, as a compiled caller
    has them: a pass then costs the calls themselves, not Python's packing
    of pointers."""

    def __init__(self):
        self.all = []

    def __getattr__(self, name):
        fn = getattr(N.load(), name)
        return lambda *args: self.all.append((fn, args))


# a training loop: the batch is on the device, the step one captured graph
def _prepare_step(s, c, seed):
    mc, tc = _configs(c)
    s.model = SM.Model(mc, tc)
    s.model.set_params(_params(mc, seed))
    s.ids, s.targets = _tokens(seed, tc.batch, tc.sequence)
    s.model.use_graph(True)
    rows = tc.batch * tc.sequence
    s.out = _Out(logits=_view(s.model, "logits", (rows, VP))[:, :V], loss=_view(s.model, "loss_rows"),
                 grads=_view(s.model, "grads"), params=_view(s.model, "params"))
    s.out.model = s.model


def _run_step(s):
    s.model.set_batch_device(s.ids.data_ptr(), s.targets.data_ptr())
    s.model.train_step()
    return s.out


def _prepare_generate(s, c, seed):
    mc, tc = _configs(c)
    s.model = SM.Model(mc, tc)
    s.model.set_params(_params(mc, seed))
    s.cache = s.model.new_cache(1024)
    s.tokens = _tokens(seed, 1, c["prompt"] + c["new"])[0].cpu().numpy()


def _run_generate(s):
    P = s.c["prompt"]
    s.cache.reset()
    out = [s.model.forward_cached(s.tokens[:P], s.cache)]
    for i in range(P, P + s.c["new"]):
        out.append(s.model.forward_cached(s.tokens[i:i + 1], s.cache))
    return np.stack(out)


def _prepare_ffn(s, c, seed):
    M, D, F = c["M"], c["D"], c["F"]
    g = _gen(seed)
    s.x = _normal(g, M, D, dtype=torch.bfloat16)
    s.wn = (1.0 + 0.1 * _normal(g, D)).to(torch.bfloat16)
    s.wgu = _normal(g, D, 2 * F, std=D ** -0.5, dtype=torch.bfloat16)
    s.wgu_t = s.wgu.t().contiguous()
    s.wd = _normal(g, F, D, std=F ** -0.5, dtype=torch.bfloat16)
    s.wd_t = s.wd.t().contiguous()
    s.dy = _normal(g, M, D, std=1e-3)
    s.dyh, s.dyl = _planes(s.dy)
    bf = torch.bfloat16
    s.z, s.y = _empty(M, D, dtype=bf), _empty(M, D, dtype=bf)
    s.g, s.u, s.h = (_empty(M, F, dtype=bf) for _ in range(3))
    s.dgh, s.dgl = _empty(M, 2 * F, dtype=bf), _empty(M, 2 * F, dtype=bf)
    s.dz, s.dx, s.dw = _empty(M, D), _empty(M, D), _empty(D)
    s.dxh, s.dxl = _empty(M, D, dtype=bf), _empty(M, D, dtype=bf)
    s.dwd, s.dwgu = _empty(F, D), _empty(D, 2 * F)
    lib = N.load()
    s.ws = _bytes(max(lib.sj_gemm_planes_workspace_bytes(M, D, 2 * F), lib.sj_gemm_planes_workspace_bytes(F, D, M),
                      lib.sj_gemm_planes_workspace_bytes(D, 2 * F, M), lib.sj_rmsnorm_bwd_p_workspace_bytes(M, D)))


def _calls_ffn(s, a):
    M, D, F = s.c["M"], s.c["D"], s.c["F"]
    e = ctypes.c_float(EPS)
    ws, wb = _p(s.ws), s.ws.numel()
    ldt = (M + 7) // 8 * 8
    a.sj_rmsnorm_fwd_t(None, _p(s.x), _p(s.wn), _p(s.z), None, ldt, M, D, e)
    a.sj_gate_up_fwd_t(None, _p(s.z), D, M, D, _p(s.wgu_t), _p(s.wgu_t, F * D), D, F, _p(s.g), _p(s.u), _p(s.h), F,
                       None, 0)
    a.sj_linear_residual_fwd_t(None, _p(s.h), F, M, F, _p(s.wd_t), F, D, _p(s.x), D, _p(s.y), D)
    a.sj_down_bwd_swiglu_p(None, _p(s.dyh), _p(s.dyl), D, M, D, _p(s.wd), D, F, _p(s.g), _p(s.u), F, _p(s.dgh),
                           _p(s.dgl), 2 * F, None, None, ldt)
    a.sj_gemm_planes_tn(None, F, D, M, _p(s.h), None, F, _p(s.dyh), _p(s.dyl), D, _p(s.dwd), F32, D, 0, ws, wb)
    a.sj_gemm_planes(None, M, D, 2 * F, _p(s.dgh), _p(s.dgl), 2 * F, _p(s.wgu), None, 2 * F, _p(s.dz), F32, D, 0, ws,
                     wb)
    a.sj_gemm_planes_tn(None, D, 2 * F, M, _p(s.z), None, D, _p(s.dgh), _p(s.dgl), 2 * F, _p(s.dwgu), F32, 2 * F, 0,
                        ws, wb)
    a.sj_rmsnorm_bwd_p(None, _p(s.x), _p(s.wn), _p(s.dz), _p(s.dy), _p(s.dx), _p(s.dw), _p(s.dxh), _p(s.dxl), None,
                       None, ldt, M, D, e, ws, wb)
    return dict(y=s.y, dx=s.dx, dw_norm=s.dw, dw_gate_up=s.dwgu, dw_down=s.dwd)


def _prepare_attn(s, c, seed):
    B, T, HQ, HK = c["B"], c["T"], c["heads"], c["kv"]
    M, D, J = B * T, 64 * HQ, 64 * HK
    NQ = D + 2 * J
    g = _gen(seed)
    bf = torch.bfloat16
    s.x = _normal(g, M, D, dtype=bf)
    s.wn = (1.0 + 0.1 * _normal(g, D)).to(bf)
    s.wqkv = _normal(g, D, NQ, std=D ** -0.5, dtype=bf)
    s.wqkv_t = s.wqkv.t().contiguous()
    s.wo = _normal(g, D, D, std=D ** -0.5, dtype=bf)
    s.wo_t = s.wo.t().contiguous()
    s.dy = _normal(g, M, D, std=1e-3)
    s.dyh, s.dyl = _planes(s.dy)
    s.rope = _rope_table(T, 64)
    s.ldt = (M + 7) // 8 * 8
    s.z, s.o, s.y = (_empty(M, D, dtype=bf) for _ in range(3))
    s.qkv = _empty(M, NQ, dtype=bf)
    s.lse, s.lse_t, s.delta = _empty(M, HQ), _empty(HQ, s.ldt), _empty(HQ, s.ldt)
    s.doh, s.dol = _empty(M, D, dtype=bf), _empty(M, D, dtype=bf)
    s.gh, s.gl = _empty(M, NQ, dtype=bf), _empty(M, NQ, dtype=bf)
    s.dz, s.dx, s.dw = _empty(M, D), _empty(M, D), _empty(D)
    s.dxh, s.dxl = _empty(M, D, dtype=bf), _empty(M, D, dtype=bf)
    s.dwo, s.dwqkv = _empty(D, D), _empty(D, NQ)
    lib = N.load()
    s.ws = _bytes(max(lib.sj_gemm_planes_workspace_bytes(M, D, NQ), lib.sj_gemm_planes_workspace_bytes(D, D, M),
                      lib.sj_gemm_planes_workspace_bytes(D, NQ, M), lib.sj_rmsnorm_bwd_p_workspace_bytes(M, D)))
    s.wsa = _bytes(lib.sj_attention_bwd_tt_workspace_bytes(B, T, HQ, HK, 64))
    s.wsa_bytes = lib.sj_attention_bwd_tt_workspace_bytes(B, T, HQ, HK, 64)


def _calls_attn(s, a):
    c = s.c
    B, T, HQ, HK, W = c["B"], c["T"], c["heads"], c["kv"], c["window"]
    M, D, J = B * T, 64 * HQ, 64 * HK
    NQ = D + 2 * J
    e = ctypes.c_float(EPS)
    ws, wb, ldt = _p(s.ws), s.ws.numel(), s.ldt
    a.sj_rmsnorm_fwd_t(None, _p(s.x), _p(s.wn), _p(s.z), None, ldt, M, D, e)
    a.sj_qkv_fwd_t(None, _p(s.z), D, M, D, _p(s.wqkv_t), D, D, J, _p(s.qkv), NQ, _p(s.rope), T, 64, None, ldt)
    a.sj_attention_fwd_tt(None, _p(s.qkv), NQ, ldt, B, T, HQ, HK, 64, W, _p(s.o), D, _p(s.lse), _p(s.lse_t), None, ldt)
    a.sj_linear_residual_fwd_t(None, _p(s.o), D, M, D, _p(s.wo_t), D, D, _p(s.x), D, _p(s.y), D)
    a.sj_gemm_planes_split_out(None, M, D, D, _p(s.dyh), _p(s.dyl), D, _p(s.wo), D, _p(s.doh), _p(s.dol), D, None,
                               None, 0, _p(s.o), D, _p(s.delta), ldt)
    a.sj_gemm_planes_tn(None, D, D, M, _p(s.o), None, D, _p(s.dyh), _p(s.dyl), D, _p(s.dwo), F32, D, 0, ws, wb)
    a.sj_attention_bwd_tt(None, _p(s.qkv), NQ, ldt, _p(s.o), D, _p(s.lse_t), _p(s.doh), _p(s.dol), D, _p(s.delta), B,
                          T, HQ, HK, 64, W, _p(s.rope), _p(s.gh), _p(s.gl), NQ, None, None, ldt, _p(s.wsa),
                          s.wsa_bytes)
    a.sj_gemm_planes(None, M, D, NQ, _p(s.gh), _p(s.gl), NQ, _p(s.wqkv), None, NQ, _p(s.dz), F32, D, 0, ws, wb)
    a.sj_gemm_planes_tn(None, D, NQ, M, _p(s.z), None, D, _p(s.gh), _p(s.gl), NQ, _p(s.dwqkv), F32, NQ, 0, ws, wb)
    a.sj_rmsnorm_bwd_p(None, _p(s.x), _p(s.wn), _p(s.dz), _p(s.dy), _p(s.dx), _p(s.dw), _p(s.dxh), _p(s.dxl), None,
                       None, ldt, M, D, e, ws, wb)
    return dict(y=s.y, o=s.o, lse=s.lse, dx=s.dx, dw_norm=s.dw, dw_out=s.dwo, dw_qkv=s.dwqkv)


def _prepare_head(s, c, seed):
    M, D = c["M"], c["D"]
    g = _gen(seed)
    s.x = _normal(g, M, D, dtype=torch.bfloat16)
    s.wn = (1.0 + 0.1 * _normal(g, D)).to(torch.bfloat16)
    s.w = _normal(g, D, V, std=D ** -0.5)
    s.ids, s.targets = (t.contiguous() for t in _tokens(seed, 1, M))
    s.hn = _empty(M, D, dtype=torch.bfloat16)
    s.logits, s.dlogits = _empty(M, VP), _empty(M, VP)
    s.rows, s.loss = _empty(M), _empty(1, dtype=torch.float64)
    s.dh, s.dx, s.dw, s.dwn, s.demb = _empty(M, D), _empty(M, D), _empty(D, V), _empty(D), _empty(V, D)
    lib = N.load()
    s.ws = _bytes(max(lib.sj_gemm_workspace_bytes(M, V, D), lib.sj_gemm_workspace_bytes(M, D, V),
                      lib.sj_gemm_workspace_bytes(D, V, M), lib.sj_rmsnorm_bwd_workspace_bytes(M, D),
                      lib.sj_embedding_bwd_workspace_bytes(M, V)))


def _calls_head(s, a):
    M, D = s.c["M"], s.c["D"]
    e = ctypes.c_float(EPS)
    ws, wb = _p(s.ws), s.ws.numel()
    a.sj_rmsnorm_fwd(None, _p(s.x), BF, _p(s.wn), BF, _p(s.hn), M, D, e)
    a.sj_gemm(None, 0, 0, M, V, D, _p(s.hn), BF, D, _p(s.w), F32, V, _p(s.logits), F32, VP, 0, ws, wb)
    a.sj_cross_entropy(None, _p(s.logits), VP, _p(s.targets), _p(s.rows), _p(s.dlogits), VP, M, V, None,
                       ctypes.c_float(1.0 / M))
    a.sj_loss_summary(None, _p(s.rows), M, _p(s.loss), 0, ctypes.c_float(1.0))
    a.sj_gemm(None, 0, 1, M, D, V, _p(s.dlogits), F32, VP, _p(s.w), F32, V, _p(s.dh), F32, D, 0, ws, wb)
    a.sj_gemm(None, 1, 0, D, V, M, _p(s.hn), BF, D, _p(s.dlogits), F32, VP, _p(s.dw), F32, V, 0, ws, wb)
    a.sj_rmsnorm_bwd(None, _p(s.x), BF, _p(s.wn), BF, _p(s.dh), None, _p(s.dx), _p(s.dwn), M, D, e, ws, wb)
    a.sj_embedding_bwd(None, _p(s.dx), _p(s.ids), _p(s.demb), M, D, V, ws, wb)
    return dict(logits=s.logits[:, :V], loss=s.loss, rows=s.rows, dx=s.dx, dw=s.dw, dw_norm=s.dwn, dw_embedding=s.demb)


def _prepare_adamw(s, c, seed):
    n = c["n"]
    g = _gen(seed)
    s.w, s.g = _normal(g, n, std=0.02), _normal(g, n, std=1e-3)
    s.m, s.v = _normal(g, n, std=1e-3), _normal(g, n, std=1e-3).square()
    s.mirror = _empty(n, dtype=torch.bfloat16)
    s.nodecay = min(n, 4096)
    st = N.AdamStep(lr=3e-4, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.1, inv_b1=1.25, inv_b2=1.5,
                    clip_norm=1.0, loss_scale=1.0, clip_enabled=1)
    s.step = torch.frombuffer(bytearray(bytes(st)), dtype=torch.uint8).to(DEV)
    s.sumsq, s.status = _empty(1, dtype=torch.float64), torch.zeros(1, dtype=torch.int32, device=DEV)
    s.ws = _bytes(N.load().sj_sum_squares_workspace_bytes(n))


def _calls_adamw(s, a):
    n = s.c["n"]
    a.sj_sum_squares(None, _p(s.g), n, _p(s.sumsq), _p(s.ws), s.ws.numel())
    a.sj_adamw_multi(None, _p(s.w), _p(s.g), _p(s.m), _p(s.v), _p(s.mirror), n, s.nodecay, _p(s.step), _p(s.sumsq),
                         _p(s.status))
    return dict(w=s.w, m=s.m, v=s.v, mirror=s.mirror, sumsq=s.sumsq)


def _prepare_moe(s, c, seed):
    M, D, E, K, F = c["M"], c["D"], c["E"], c["K"], c["F"]
    g = _gen(seed)
    bf = torch.bfloat16
    s.z, s.x = _normal(g, M, D, dtype=bf), _normal(g, M, D, dtype=bf)
    s.wr = _normal(g, D, E, std=D ** -0.5, dtype=bf)
    s.wgu = _normal(g, E, D, 2 * F, std=D ** -0.5, dtype=bf)
    s.wgu_t = s.wgu.transpose(1, 2).contiguous()
    s.wd = _normal(g, E, F, D, std=F ** -0.5, dtype=bf)
    s.wd_t = s.wd.transpose(1, 2).contiguous()
    s.dy = _normal(g, M, D, std=1e-3)
    lib = N.load()
    S = M * K
    s.cap = cap = lib.sj_route_pack_capacity(S, E)
    i32 = lambda n: torch.zeros(n, dtype=torch.int32, device=DEV)
    s.logits, s.ids, s.wts = _empty(M, E, dtype=bf), i32(S), _empty(S)
    s.cnt, s.off, s.ps, s.pp = i32(E), i32(E + 1), i32(cap), i32(S)
    s.zp, s.yp, s.out = _empty(cap, D, dtype=bf), _empty(cap, D, dtype=bf), _empty(M, D, dtype=bf)
    s.g, s.u, s.h = (torch.zeros(cap, F, dtype=bf, device=DEV) for _ in range(3))
    s.dxh, s.dxl = _empty(cap, D, dtype=bf), _empty(cap, D, dtype=bf)
    s.dwts = _empty(S)
    s.dgh, s.dgl = _empty(cap, 2 * F, dtype=bf), _empty(cap, 2 * F, dtype=bf)
    s.dzp, s.dz, s.dlog = _empty(cap, D), _empty(M, D), _empty(M, E)
    s.dwgu, s.dwd, s.dwr = _empty(E, D, 2 * F), _empty(E, F, D), _empty(D, E)
    s.ws = _bytes(lib.sj_gemm_workspace_bytes(D, E, M))


def _calls_moe(s, a):
    c, cap = s.c, s.cap
    M, D, E, K, F = c["M"], c["D"], c["E"], c["K"], c["F"]
    a.sj_router_topk(None, _p(s.z), D, _p(s.wr), D, M, E, K, _p(s.logits), _p(s.ids), _p(s.wts))
    a.sj_route_pack(None, _p(s.ids), M, K, E, None, None, _p(s.cnt), _p(s.off), _p(s.ps), _p(s.pp), cap)
    a.sj_moe_gather(None, _p(s.z), D, D, _p(s.ps), K, cap, _p(s.zp), None, cap)
    a.sj_moe_gate_up_fwd(None, _p(s.off), E, cap, _p(s.zp), D, D, _p(s.wgu_t), _p(s.wgu_t, F * D), D, 2 * F * D, F,
                         _p(s.g), _p(s.u), _p(s.h), F, None, cap)
    a.sj_moe_down_fwd(None, _p(s.off), E, cap, _p(s.h), F, F, _p(s.wd_t), F, D * F, D, _p(s.yp), D)
    a.sj_moe_combine(None, _p(s.yp), D, D, _p(s.ids), _p(s.pp), _p(s.wts), M, K, _p(s.x), D, _p(s.out), D)
    a.sj_moe_combine_bwd(None, _p(s.yp), D, D, _p(s.ps), _p(s.wts), K, cap, _p(s.dy), D, _p(s.dxh), _p(s.dxl), None,
                         None, cap, _p(s.dwts))
    a.sj_moe_down_bwd_swiglu_p(None, _p(s.off), E, cap, _p(s.dxh), _p(s.dxl), D, D, _p(s.wd), D, F * D, F, _p(s.g),
                               _p(s.u), F, _p(s.dgh), _p(s.dgl), 2 * F, None, None, cap)
    a.sj_moe_gemm_dw_tn(None, _p(s.off), E, cap, F, D, _p(s.h), F, _p(s.dxh), _p(s.dxl), D, _p(s.dwd), D, F * D)
    a.sj_moe_gemm_rows(None, _p(s.off), E, cap, D, 2 * F, _p(s.dgh), _p(s.dgl), 2 * F, _p(s.wgu), 2 * F, D * 2 * F,
                       _p(s.dzp), D, 0)
    a.sj_moe_gemm_dw_tn(None, _p(s.off), E, cap, D, 2 * F, _p(s.zp), D, _p(s.dgh), _p(s.dgl), 2 * F, _p(s.dwgu),
                        2 * F, D * 2 * F)
    a.sj_moe_gather_bwd(None, _p(s.dzp), D, D, _p(s.ids), _p(s.pp), _p(s.wts), _p(s.logits), _p(s.dwts), _p(s.wr), M,
                        K, E, None, D, _p(s.dz), D, _p(s.dlog))
    a.sj_gemm(None, 1, 0, D, E, M, _p(s.z), BF, D, _p(s.dlog), F32, E, _p(s.dwr), F32, E, 0, _p(s.ws), s.ws.numel())
    return dict(ids=s.ids, weights=s.wts, out=s.out, dz=s.dz, dw_gate_up=s.dwgu, dw_down=s.dwd, dw_router=s.dwr)


def _prepare_pvjp(s, c, seed):
    M, D, F = c["M"], c["D"], c["F"]
    lib = N.load()
    r, b, k = ctypes.c_long(), ctypes.c_long(), ctypes.c_long()
    N.api.sj_pvjp_budget(c["rank"], c["fraction"], 32, M, D, F, ctypes.byref(r), ctypes.byref(b), ctypes.byref(k))
    s.rank, s.blocks, s.sel = r.value, b.value, k.value
    s.k = s.sel * 32
    s.seed = 0x9E37 + int(seed)
    g = _gen(seed)
    bf = torch.bfloat16
    s.x = _normal(g, M, D, dtype=bf)
    s.donor = _normal(g, M, F, dtype=bf)
    s.dyh, s.dyl = _planes(_normal(g, M, 2 * F, std=1e-4))
    s.w = _normal(g, D, 2 * F, std=0.02)
    s.mirror = _empty(D, 2 * F, dtype=bf)
    i32 = lambda n: torch.zeros(n, dtype=torch.int32, device=DEV)
    s.scr, s.cols, s.rowsel, s.map = i32(F + s.blocks), i32(s.rank), i32(s.k), i32(D)
    s.q, s.left, s.coef = _empty(M, s.rank), _empty(D, s.rank), _empty(s.rank + s.k, 2 * F)
    s.eh, s.el = _empty(s.rank + s.k, M, dtype=bf), _empty(s.rank + s.k, M, dtype=bf)
    s.eps = lib.sj_pvjp_basis_tolerance(M, s.rank)
    s.ws = _bytes(max(lib.sj_pvjp_basis_workspace_bytes(M, s.rank), lib.sj_pvjp_prepare_workspace_bytes(D, M, s.rank),
                      lib.sj_pvjp_vjp_workspace_bytes(s.rank + s.k, 2 * F, M)))
    # gate and up: two column blocks of one matrix, as a model holds them
    terms, params = [], []
    for j in range(2):
        terms.append(N.FactoredTerm(s.left.data_ptr(), s.coef.data_ptr() + 4 * j * F,
                                    s.coef.data_ptr() + 4 * (s.rank * 2 * F + j * F), s.map.data_ptr(), s.rank, 1.0,
                                    2 * F))
        params.append(N.FactoredParam(s.w.data_ptr() + 4 * j * F, None, D, F, 1, j, 1, 2 * F,
                                      s.mirror.data_ptr() + 2 * j * F))
    PA, TA = (N.FactoredParam * 2)(*params), (N.FactoredTerm * 2)(*terms)
    nb = lib.sj_factored_meta_bytes(PA, 2, 2)
    host, tiles = np.zeros(nb, np.uint8), ctypes.c_long()
    N.api.sj_factored_pack(PA, 2, TA, 2, ctypes.c_void_p(host.ctypes.data), nb, ctypes.byref(tiles))
    s.meta, s.tiles = torch.from_numpy(host).to(DEV), tiles.value
    s.part, s.norm = _empty(s.tiles, dtype=torch.float64), _empty(1, dtype=torch.float64)


def _calls_pvjp(s, a):
    c = s.c
    M, D, F = c["M"], c["D"], c["F"]
    ws, wb = _p(s.ws), s.ws.numel()
    cf = ctypes.c_float
    a.sj_pvjp_indices(None, s.seed, D, F, s.blocks, s.sel, s.rank, 32, _p(s.scr), _p(s.cols), _p(s.rowsel), _p(s.map))
    a.sj_pvjp_basis(None, _p(s.donor), BF, F, M, _p(s.cols), s.rank, cf(s.eps), _p(s.q), ws, wb)
    a.sj_pvjp_prepare_rows(None, _p(s.x), D, D, M, _p(s.q), s.rank, _p(s.rowsel), s.k, cf(s.blocks / s.sel), _p(s.left),
                           None, _p(s.eh), _p(s.el), M, ws, wb)
    a.sj_pvjp_vjp_rows(None, _p(s.eh), _p(s.el), M, s.rank + s.k, M, _p(s.dyh), _p(s.dyl), 2 * F, 2 * F, _p(s.coef),
                       2 * F, ws, wb)
    a.sj_factored_apply(None, _p(s.meta), s.tiles, 2, cf(0), cf(0), _p(s.part))
    a.sj_sum_f64(None, _p(s.part), s.tiles, _p(s.norm))
    a.sj_factored_apply(None, _p(s.meta), s.tiles, 1, cf(1e-2), cf(1e-4), None)
    return dict(columns=s.cols, rows=s.rowsel, q=s.q, left=s.left, coefficients=s.coef, w=s.w, mirror=s.mirror,
                norm=s.norm)


# ------------------------------------------------------------------- work

def _pairs(T, window):
    if window and window < T:
        return window * (window + 1) / 2 + (T - window) * window
    return T * (T + 1) / 2


def _block_flops(M, T, B, d, heads, kv, ffn, hd, window=0):
    """Forward products and attention of one block."""
    nq = d + 2 * kv * hd
    return 2 * M * d * (nq + d + 3 * ffn) + B * heads * 4 * hd * _pairs(T, window)


def work(case):
    """Each input read once and each output written once; products once
    (forward, dX and dW), attention backward 2.5 times its forward."""
    c, k = case, case["kind"]
    if k == "step":
        mc, tc = _configs(c)
        M, P = tc.batch * tc.sequence, SM.param_count(mc)
        d, hd, T, B = mc.width, mc.head_dim, tc.sequence, tc.batch

        def stage(L, M, T, d, heads, kv, ffn, window=0):
            lin = 2 * M * d * (2 * d + 2 * kv * (d // heads) + 3 * ffn)
            return L * (3 * lin + 3.5 * B * heads * 4 * (d // heads) * _pairs(T, window))
        fl = 6.0 * M * d * V
        if c["hier"]:
            h = mc.hierarchy
            Tg = -(-T // h.patch_size)
            fl += stage(h.encoder_layers, M, T, h.encoder_width, h.encoder_heads, h.encoder_heads, h.encoder_ffn_width,
                        h.local_window)
            fl += stage(h.decoder_layers, M, T, h.decoder_width, h.decoder_heads, h.decoder_heads, h.decoder_ffn_width,
                        h.local_window)
            fl += stage(mc.layers, B * Tg, Tg, d, mc.heads, mc.kv, mc.ffn_width)
            fl += 6.0 * (B * Tg * d * (h.encoder_width + h.decoder_width)
                         + M * h.decoder_width * (h.encoder_width + d))
        else:
            fl += stage(mc.layers, M, T, d, mc.heads, mc.kv, mc.ffn_width)
        # w, m, v read and written, the gradient written (and read by the norm and update)
        return dict(bytes=4.0 * P * 8 + 4.0 * M * V + 8 * M, flops=fl)
    if k == "generate":
        mc, _ = _configs(c)
        P = SM.param_count(mc) - V * mc.width
        n, J = c["prompt"] + c["new"], 64 * c["kv"]
        # every call reads the weights (bf16; the fp32 head) and the cache so far
        head = mc.width * V
        per_call = 2.0 * (P - head) + 4.0 * head
        cache = sum(4.0 * J * (c["prompt"] + i + 1) for i in range(c["new"])) * mc.layers
        return dict(bytes=per_call * (c["new"] + 1) + cache,
                    flops=2.0 * (P - head) * n + 2.0 * head * (c["new"] + 1)
                    + mc.layers * c["heads"] * 256.0 * _pairs(n, 0))
    if k == "ffn":
        M, D, F = c["M"], c["D"], c["F"]
        return dict(bytes=M * D * (2 + 4 + 4 + 2 + 4.0) + 3 * D * F * (2 + 4.0) + 8 * D, flops=18.0 * M * D * F)
    if k == "attn":
        B, T, HQ, HK = c["B"], c["T"], c["heads"], c["kv"]
        M, D, NQ = B * T, 64 * HQ, 64 * (HQ + 2 * HK)
        return dict(bytes=M * D * (2 + 4 + 4 + 2 + 2 + 4.0) + M * HQ * 4 + D * (NQ + D) * 6.0,
                    flops=6.0 * M * D * (NQ + D) + 3.5 * B * HQ * 256 * _pairs(T, c["window"]))
    if k == "head":
        M, D = c["M"], c["D"]
        return dict(bytes=M * D * (2 + 4.0) + M * V * 4.0 + M * 12 + 4.0 * V * D * 3 + 8 * D, flops=6.0 * M * D * V)
    if k == "adamw":
        return dict(bytes=30.0 * c["n"], flops=0.0)
    if k == "moe":
        M, D, E, K, F = c["M"], c["D"], c["E"], c["K"], c["F"]
        return dict(bytes=M * D * (2 + 2 + 2 + 4 + 4.0) + 3 * E * D * F * (2 + 4.0) + M * K * 8 + D * E * 6,
                    flops=18.0 * M * K * D * F + 6.0 * M * D * E)
    M, D, F = c["M"], c["D"], c["F"]
    blocks = -(-D // 32)
    rows = c["rank"] + 32 * max(1, math.ceil(blocks * c["fraction"]))
    return dict(bytes=M * (2.0 * D + 2.0 * c["rank"] + 4.0 * c["rank"] + 8.0 * F) + 2 * F * (rows * 4.0 + D * 10.0),
                flops=2.0 * M * rows * 2 * F + 2.0 * M * D * c["rank"] + 2.0 * D * 2 * F * c["rank"])


# -------------------------------------------------------------- tolerance

def tolerance(case):
    """Up to about four times the error against exact() that the calls showed
    over the listed and several drawn cases."""
    k = case["kind"]
    if k == "step":
        # fp32 products on hi/lo bf16 planes (seen: 9e-6); AdamW divides a
        # gradient by its own size, so single weights may move by 2 lr a step
        if case["precision"] == "f32":
            return dict(rel=5e-5, max=0.2)
        # a bf16 rounding that flips in one layer travels through the others
        # (seen: 7e-3 on the logits, 4e-3 on the gradients)
        return dict(rel=2e-2, max=0.9)
    if k == "generate":
        return dict(rel=2e-2, max=0.3)  # seen: 6e-3
    if k in ("ffn", "attn"):
        return dict(rel=1e-2, max=0.3)  # bf16 activations between the products; seen: 5e-3
    if k == "head":
        return dict(rel=5e-3, max=0.2)  # bf16 normed rows; seen: 1.7e-3
    if k == "adamw":
        return dict(rel=2e-4, max=1e-2)  # the bf16 mirror's rare other neighbour; the rest to fp32 rounding
    if k == "moe":
        return dict(rel=1e-2, max=0.3, differ=1e-3)  # seen: 4e-3; near-ties of the router may pick the other expert
    return dict(rel=5e-4, max=5e-2)  # hi/lo products (seen: 4e-6) and a bf16 mirror


# ------------------------------------------------------------------ exact
# The same calls in 64 bits with plain torch: inputs as prepare makes them,
# no storage roundings between the operations (weights enter in the storage
# type the framework multiplies them in).

def _d(t):
    return t.double()


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _rope(x, T):
    """x [B, T, H, hd], interleaved pairs."""
    hd = x.shape[-1]
    i = torch.arange(hd // 2, device=x.device, dtype=torch.float64)
    f = torch.arange(T, device=x.device, dtype=torch.float64)[:, None] * (THETA ** (-2.0 * i / hd))[None]
    c, s = f.cos()[None, :, None], f.sin()[None, :, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)


def _attend(q, k, v, window):
    """q [B, T, HQ, hd], k and v [B, T, HK, hd] -> (o, lse), one KV head at a time."""
    B, T, HQ, hd = q.shape
    HK = k.shape[2]
    G = HQ // HK
    i = torch.arange(T, device=q.device)
    keep = i[None, :] <= i[:, None]
    if window:
        keep &= i[None, :] > i[:, None] - window
    os, ls = [], []
    for h in range(HK):
        qh = q[:, :, h * G:(h + 1) * G].transpose(1, 2)
        kh, vh = k[:, :, h].unsqueeze(1), v[:, :, h].unsqueeze(1)
        sc = torch.matmul(qh, kh.transpose(-1, -2).contiguous()) * hd ** -0.5
        sc = sc.masked_fill(~keep, -math.inf)
        ls.append(torch.logsumexp(sc, -1))
        os.append(torch.matmul(torch.softmax(sc, -1), vh).transpose(1, 2))
    return torch.cat(os, 2), torch.cat(ls, 1)


def _block(x, w, B, T, heads, kv, window=0):
    d = x.shape[-1]
    hd = d // heads
    z = _rms(x, w["attention_norm"])
    q = _rope((z @ w["query"]).view(B, T, heads, hd), T)
    k = _rope((z @ w["key"]).view(B, T, kv, hd), T)
    v = (z @ w["value"]).view(B, T, kv, hd)
    x = x + _attend(q, k, v, window)[0].reshape(B * T, d) @ w["attention_output"]
    z = _rms(x, w["ffn_norm"])
    return x + (torch.nn.functional.silu(z @ w["gate"]) * (z @ w["up"])) @ w["down"]


def _exact_model(mc, flat, ids, B, T):
    """(logits of every position, the weights as leaves by name)."""
    W, o = {}, 0
    for name, shape, norm in SM.layout(mc):
        n = math.prod(shape)
        t = torch.from_numpy(flat[o:o + n]).to(DEV).view(shape)
        if mc.precision == "bf16" and name != "output":
            t = t.to(torch.bfloat16)
        W[name] = t.double().requires_grad_(True)
        o += n
    x = W["embedding"][ids.long()]
    for l in range(mc.layers):
        p = "layers.%d." % l
        x = _block(x, {n[len(p):]: t for n, t in W.items() if n.startswith(p)}, B, T, mc.heads, mc.kv)
    return _rms(x, W["final_norm"]) @ W["output"], W


def _exact_step(c, seed):
    if c["hier"]:
        return None
    mc, tc = _configs(c)
    flat = _params(mc, seed)
    ids, tg = _tokens(seed, tc.batch, tc.sequence)
    logits, W = _exact_model(mc, flat, ids, tc.batch, tc.sequence)
    rows = torch.nn.functional.cross_entropy(logits, tg.long(), reduction="none")
    rows.mean().backward()
    # the arena's order: norms, embedding, then per layer q|k|v, the attention
    # output, gate|up and down, the head padded to a multiple of 8 columns;
    # every matrix starts at a multiple of 64
    parts = []

    def put(t):
        parts.append(t.reshape(-1))
        if t.numel() % 64:
            parts.append(torch.zeros(64 - t.numel() % 64, dtype=torch.float64, device=DEV))
    G = {n: t.grad for n, t in W.items()}
    for l in range(mc.layers):
        put(G["layers.%d.attention_norm" % l])
        put(G["layers.%d.ffn_norm" % l])
    put(G["final_norm"])
    put(G["embedding"])
    for l in range(mc.layers):
        p = "layers.%d." % l
        put(torch.cat([G[p + "query"], G[p + "key"], G[p + "value"]], 1))
        put(G[p + "attention_output"])
        put(torch.cat([G[p + "gate"], G[p + "up"]], 1))
        put(G[p + "down"])
    put(torch.nn.functional.pad(G["output"], (0, VP - V)))
    return dict(logits=logits.detach(), loss=rows.detach(), grads=torch.cat(parts), params=None)


def _exact_generate(c, seed):
    mc, _ = _configs(c)
    n = c["prompt"] + c["new"]
    ids = _tokens(seed, 1, n)[0]
    with torch.no_grad():
        logits, _ = _exact_model(mc, _params(mc, seed), ids, 1, n)
    return logits[c["prompt"] - 1:].cpu().numpy()


def _exact_ffn(c, seed):
    s = _S()
    _prepare_ffn(s, c, seed)
    F = c["F"]
    x, wn, wgu, wd = (_d(t).requires_grad_(True) for t in (s.x, s.wn, s.wgu, s.wd))
    gu = _rms(x, wn) @ wgu
    y = x + (torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]) @ wd
    y.backward(_d(s.dy))
    return dict(y=y.detach(), dx=x.grad, dw_norm=wn.grad, dw_gate_up=wgu.grad, dw_down=wd.grad)


def _exact_attn(c, seed):
    B, T, HQ, HK = c["B"], c["T"], c["heads"], c["kv"]
    if B * HQ * T * T > 1.1e9:  # the scores alone would take over 9 GB a copy
        return None
    s = _S()
    _prepare_attn(s, c, seed)
    M, D, J = B * T, 64 * HQ, 64 * HK
    x, wn, wqkv, wo = (_d(t).requires_grad_(True) for t in (s.x, s.wn, s.wqkv, s.wo))
    qkv = _rms(x, wn) @ wqkv
    q, k = _rope(qkv[:, :D].view(B, T, HQ, 64), T), _rope(qkv[:, D:D + J].view(B, T, HK, 64), T)
    o, lse = _attend(q, k, qkv[:, D + J:].view(B, T, HK, 64), c["window"])
    o = o.reshape(M, D)
    y = x + o @ wo
    y.backward(_d(s.dy))
    return dict(y=y.detach(), o=o.detach(), lse=lse.detach().transpose(1, 2).reshape(M, HQ), dx=x.grad,
                dw_norm=wn.grad, dw_out=wo.grad, dw_qkv=wqkv.grad)


def _exact_head(c, seed):
    s = _S()
    _prepare_head(s, c, seed)
    x, wn, w = (_d(t).requires_grad_(True) for t in (s.x, s.wn, s.w))
    logits = _rms(x, wn) @ w
    rows = torch.nn.functional.cross_entropy(logits, s.targets.long(), reduction="none")
    rows.mean().backward()
    demb = torch.zeros(V, c["D"], dtype=torch.float64, device=DEV).index_add_(0, s.ids.long(), x.grad)
    return dict(logits=logits.detach(), loss=rows.mean().detach().view(1), rows=rows.detach(), dx=x.grad, dw=w.grad,
                dw_norm=wn.grad, dw_embedding=demb)


def _exact_adamw(c, seed):
    s = _S()
    _prepare_adamw(s, c, seed)
    w, g, m, v = (_d(t) for t in (s.w, s.g, s.m, s.v))
    sumsq = g.square().sum().view(1)
    norm = float(sumsq.sqrt())
    gi = g * (1.0 / norm if norm > 1.0 else 1.0)
    f = lambda x: float(np.float32(x))
    b1, b2, lr, wdec = f(0.9), f(0.95), f(3e-4), f(0.1)
    m = b1 * m + (1 - b1) * gi
    v = b2 * v + (1 - b2) * gi * gi
    keep = torch.ones_like(w)
    keep[s.nodecay:] = 1 - lr * wdec
    w = w * keep - lr * (m * 1.25) / ((v * 1.5).sqrt() + f(1e-8))
    return dict(w=w, m=m, v=v, mirror=w, sumsq=sumsq)


def _exact_moe(c, seed):
    s = _S()
    _prepare_moe(s, c, seed)
    M, D, E, K, F = c["M"], c["D"], c["E"], c["K"], c["F"]
    z, wr, wgu, wd = (_d(t).requires_grad_(True) for t in (s.z, s.wr, s.wgu, s.wd))
    logits = z @ wr
    # the stored logits decide (lowest index on ties), so the choice is of
    # their bf16 roundings
    probs = torch.softmax(logits + (logits.to(torch.bfloat16).double() - logits).detach(), -1)
    p = probs.detach().clone()
    ids = []
    for _ in range(K):
        ids.append((p == p.max(-1, keepdim=True).values).int().argmax(-1))
        p[torch.arange(M, device=DEV), ids[-1]] = -1.0
    ids = torch.stack(ids, 1)
    wts = probs.gather(1, ids)
    out = _d(s.x)
    for e in range(E):
        tok, slot = (ids == e).nonzero(as_tuple=True)
        gu = z[tok] @ wgu[e]
        y = (torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]) @ wd[e]
        out = out.index_add(0, tok, y * wts[tok, slot][:, None])
    out.backward(_d(s.dy))
    return dict(ids=None, weights=wts.detach().reshape(-1), out=out.detach(), dz=z.grad, dw_gate_up=wgu.grad,
                dw_down=wd.grad, dw_router=wr.grad)


def _exact_pvjp(c, seed):
    s = _S()
    _prepare_pvjp(s, c, seed)
    M, D, F = c["M"], c["D"], c["F"]
    # partial Fisher-Yates over the donor columns, then over the feature
    # blocks, on one SplitMix64 stream
    mask, state = (1 << 64) - 1, [s.seed & ((1 << 64) - 1)]

    def index(n):
        while True:
            state[0] = (state[0] + 0x9E3779B97F4A7C15) & mask
            x = state[0]
            x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & mask
            x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & mask
            x ^= x >> 31
            if x >= ((1 << 64) - n) % n:
                return x % n

    def pick(size, count):
        a = list(range(size))
        for i in range(count):
            j = i + index(size - i)
            a[i], a[j] = a[j], a[i]
        return a[:count]
    cols, blocks = pick(F, s.rank), pick(s.blocks, s.sel)
    rows = [b * 32 + i if b * 32 + i < D else -1 for b in blocks for i in range(32)]
    q, r = torch.linalg.qr(_d(s.donor)[:, cols])
    q = q * torch.sign(torch.diagonal(r))
    x, dy = _d(s.x), _d(s.dyh) + _d(s.dyl)
    left = x.t() @ q
    at = torch.tensor(rows, device=DEV)
    ok = at >= 0
    res = torch.zeros(s.k, M, dtype=torch.float64, device=DEV)
    res[ok] = (x[:, at[ok]].t() - left[at[ok]] @ q.t()) * (s.blocks / s.sel)
    coef = torch.cat([q.t(), res]) @ dy
    grad = left @ coef[:s.rank]
    grad[at[ok]] += coef[s.rank:][ok]
    w = _d(s.w) * (1 - 1e-4) - 1e-2 * grad
    return dict(columns=None, rows=None, q=q, left=left, coefficients=coef, w=w, mirror=w,
                norm=grad.square().sum().view(1))


def exact(case, seed):
    N.load()
    return globals()["_exact_" + case["kind"]](case, seed)
