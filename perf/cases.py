"""The calls this framework is used for, as cases that can be timed and checked.

A case is a dict of plain values. `listed()` names the standing ones, `draw(rng)`
gives more of the same ranges, `prepare` makes what a program holds before the
call, `run` makes the call, `exact` computes the same in 64 bits with torch alone.

Kinds:
  linear_i8   vla_dense_linear_i8_dev: per-row int8 quantization of fp32
              activations, int8 GEMM, bias and activation (every int8 layer)
  linear_f32  vla_dense_linear_dev: the same layer where a model's int8 mask
              leaves it in fp32
  attention   vla_attention_dev: fp32 masked GQA attention
  conv_i8     vla_conv2d_i8_dev: the W8A8 convolution of the image trunks
  trunk       vla_act_encode_dev: camera frame -> ResNet-18 feature map
  vision      vla_siglip_tf_encode_dev: the whole SigLIP tower and connector
"""

from __future__ import annotations

import hashlib
import importlib.util
import json
import math
import os
import shutil
import sys
import tempfile

import numpy as np
import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"


def _pkg():
    if "vla_simd_amd" not in sys.modules:
        d = os.path.join(ROOT, "vla.simd_amd")
        spec = importlib.util.spec_from_file_location("vla_simd_amd", os.path.join(d, "__init__.py"),
                                                      submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["vla_simd_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["vla_simd_amd"]


def listed():
    return [
        # one decode row through a SmolLM2 MLP up projection: the smallest call
        dict(name="linear_i8_row", kind="linear_i8", M=1, K=960, N=2560, act="none", bias=True),
        # ACT's action chunk of 100 rows through the decoder's first FFN layer
        dict(name="linear_i8_chunk", kind="linear_i8", M=100, K=512, N=3200, act="relu", bias=True),
        # Octo-base's 690 tokens through its first MLP layer
        dict(name="linear_i8_tokens", kind="linear_i8", M=690, K=768, N=3072, act="gelu_tanh", bias=True),
        # the largest GEMM of the throughput sweep
        dict(name="linear_i8_large", kind="linear_i8", M=8192, K=4096, N=4096, act="none", bias=True),
        # ACT's decoder FFN with the int8 bit of w1 off
        dict(name="linear_f32_chunk", kind="linear_f32", M=100, K=512, N=3200, act="relu", bias=True),
        # Octo-base's first MLP layer with the int8 bit of w1 off
        dict(name="linear_f32_tokens", kind="linear_f32", M=690, K=768, N=3072, act="gelu_tanh", bias=True),
        # one denoise step of SmolVLA's action expert: 50 suffix queries over
        # 177 prefix and 50 suffix keys, 15 query heads on 5 kv heads
        dict(name="attn_suffix", kind="attention", sq=50, sk=227, n_q=15, n_kv=5, hd=64, mask="suffix"),
        # Octo-base over two timesteps, block-causal over its token groups
        dict(name="attn_blocks", kind="attention", sq=690, sk=690, n_q=12, n_kv=12, hd=64, mask="blocks"),
        # SigLIP over the 1024 patches of one 512 x 512 image
        dict(name="attn_vision", kind="attention", sq=1024, sk=1024, n_q=12, n_kv=12, hd=64, mask="none"),
        # a 3 x 3 layer of ResNet-18's second stage for a 480 x 640 frame
        dict(name="conv_i8_stage2", kind="conv_i8", H=60, W=80, Cin=128, Cout=128, k=3, stride=1),
        # ACT's image trunk as it runs unless its int8 bit is set
        dict(name="trunk_f32", kind="trunk", H=480, W=640, cams=1, int8=False),
        # SmolVLA's vision tower for one camera image, every layer int8
        dict(name="vision_i8", kind="vision", side=32, heads=12, inter=3072, layers=12, out=960, int8=15),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear_i8"] * 4 + ["linear_f32"] * 3 + ["attention"] * 4 + ["conv_i8"] * 2 + ["trunk", "vision"])
    if kind in ("linear_i8", "linear_f32"):
        K, N = _log(rng, 256, 4096), _log(rng, 240, 4096)
        if rng.random() < 0.7:  # model widths are multiples of 16; the rest are as they come
            K, N = (K + 15) // 16 * 16, (N + 15) // 16 * 16
        M = _log(rng, 1, 8192 if kind == "linear_i8" else 2048)
        return dict(kind=kind, M=M, K=K, N=N, act=rng.choice(["none", "relu", "gelu_tanh", "gelu_erf"]),
                    bias=rng.random() < 0.8)
    if kind == "attention":
        n_q, n_kv = rng.choice([(8, 8), (12, 12), (15, 5), (16, 4), (6, 6)])
        mask = rng.choice(["none", "causal", "dense", "blocks", "suffix"])
        sq = _log(rng, 1, 1024)
        if mask == "none":
            sk = _log(rng, 16, 1024)
        elif mask == "blocks":
            sq = sk = max(sq, 40)
        else:
            sk = sq + rng.choice([0, rng.randint(1, 300)])
            sk = max(sk, 16) if mask != "suffix" else max(sk, sq + 16)
            if mask == "suffix":
                sq = min(sq, 200)  # an action chunk: a group of its own per query, 256 groups at most
                sk = sq + rng.randint(16, 400)
        return dict(kind=kind, sq=sq, sk=sk, n_q=n_q, n_kv=n_kv, hd=rng.choice([32, 64, 64, 64, 128]), mask=mask)
    if kind == "conv_i8":
        k = rng.choice([1, 3, 3])
        return dict(kind=kind, H=rng.randint(12, 120), W=rng.randint(12, 160), Cin=rng.choice([3, 64, 96, 128, 256]),
                    Cout=rng.choice([64, 128, 256]), k=k, stride=rng.choice([1, 1, 2]))
    if kind == "trunk":
        return dict(kind=kind, H=rng.randint(96, 480), W=rng.randint(96, 640), cams=1, int8=rng.random() < 0.4)
    return dict(kind=kind, side=4 * rng.randint(2, 8), heads=rng.choice([4, 6, 12]), inter=rng.choice([1024, 2048, 3072]),
                layers=rng.randint(1, 4), out=rng.choice([576, 960]), int8=rng.choice([0, 7, 15, 15]))


# ---------------------------------------------------------------- inputs --

def _gen(seed):
    return torch.Generator(DEV).manual_seed(int(seed) * 7919 + 17)


def _n(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _kpad(K):
    return (K + 3) // 4 * 4


def _linear_inputs(c, seed):
    g = _gen(seed)
    M, K, N = c["M"], c["K"], c["N"]
    x = _n(g, M, K)
    b = _n(g, N, std=0.02) if c["bias"] else None
    if c["kind"] == "linear_f32":
        return x, (torch.rand(N, K, generator=g, device=DEV) * 2 - 1) / math.sqrt(K), None, b
    W = torch.zeros(N, _kpad(K), dtype=torch.int8, device=DEV)
    W[:, :K] = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    return x, W, 1e-3 + 9e-3 * torch.rand(N, generator=g, device=DEV), b


def _groups(c):
    """(query group, key group, allow[G, G]) of the group masks, on the host."""
    sq, sk = c["sq"], c["sk"]
    if c["mask"] == "suffix":  # the prefix is one group, every suffix query sees it and the suffix up to itself
        n = sk - sq
        q = np.arange(1, sq + 1, dtype=np.uint8)
        k = np.concatenate([np.zeros(n, np.uint8), q])
        allow = np.tril(np.ones((sq + 1, sq + 1), np.uint8))
        return q, k, allow
    # task tokens, then two timesteps of observation tokens and one readout
    # each: everyone sees the task, observations see earlier observations,
    # readouts see observations and earlier readouts, nobody else sees readouts
    n_task = min(16, sk // 4)
    per = (sk - n_task) // 2
    ids = [0] * n_task + [1] * (per - 1) + [2] + [3] * (sk - n_task - per - 1) + [4]
    q = np.array(ids, np.uint8)
    allow = np.array([[1, 0, 0, 0, 0], [1, 1, 0, 0, 0], [1, 1, 1, 0, 0], [1, 1, 0, 1, 0], [1, 1, 1, 1, 1]], np.uint8)
    return q, q.copy(), allow


def _keep(c):
    """[sq, sk] truth values of the mask, on the host (None: everything)."""
    i, j = np.arange(c["sq"])[:, None], np.arange(c["sk"])[None, :]
    if c["mask"] == "causal":
        return j <= i + (c["sk"] - c["sq"])
    if c["mask"] == "dense":  # the last eighth of the keys is padding
        return np.broadcast_to(j < c["sk"] - c["sk"] // 8, (c["sq"], c["sk"]))
    if c["mask"] in ("suffix", "blocks"):
        q, k, allow = _groups(c)
        return allow[q[:, None], k[None, :]].astype(bool)
    return None


def _attention_inputs(c, seed):
    g = _gen(seed)
    return (_n(g, c["sq"], c["n_q"] * c["hd"]), _n(g, c["sk"], c["n_kv"] * c["hd"]), _n(g, c["sk"], c["n_kv"] * c["hd"]))


def _conv_inputs(c, seed):
    g = _gen(seed)
    K = c["k"] * c["k"] * c["Cin"]
    x = torch.relu(_n(g, c["H"], c["W"], c["Cin"]))  # maps reach a convolution through a ReLU
    W = (torch.rand(c["Cout"], K, generator=g, device=DEV) * 2 - 1) * math.sqrt(3.0 / K)
    return x, W, _n(g, c["Cout"], std=0.05)


def _frames(c, seed):
    return torch.randint(0, 256, (c["cams"], c["H"], c["W"], 3), generator=_gen(seed), device=DEV, dtype=torch.uint8)


def _trunk_cfg(c):
    # the transformer behind the trunk is not run here and kept small
    return dict(_pkg_checkpoints().ACT_MODEL_BASE, img_h=c["H"], img_w=c["W"], n_cams=c["cams"], n_enc=1, ff=256)


def _vision_cfg(c):
    return dict(_pkg_checkpoints().SIGLIP_BASE, hidden=64 * c["heads"], n_heads=c["heads"], inter=c["inter"],
                n_layers=c["layers"], img=16 * c["side"], n_patches=c["side"] ** 2, mm_out=c["out"],
                n_img_tok=(c["side"] // 4) ** 2)


def _pkg_checkpoints():
    _pkg()
    import vla_simd_amd.checkpoints as ck
    return ck


def _checkpoint(what, cfg):
    """A random-init checkpoint of this shape, written once (a user has it on disk)."""
    ck = _pkg_checkpoints()
    key = hashlib.sha1(json.dumps([what, cfg], sort_keys=True).encode()).hexdigest()[:16]
    d = os.path.join(tempfile.gettempdir(), f"vla_cases_{os.getuid()}_{what}_{key}")
    if not os.path.isdir(d):
        tmp = tempfile.mkdtemp(prefix="vla_cases_")
        (ck.write_siglip if what == "vision" else ck.write_act_model)(tmp, cfg)
        try:
            os.rename(tmp, d)
        except OSError:  # another process was first
            shutil.rmtree(tmp, ignore_errors=True)
    return d


# ------------------------------------------------------------ the calls --

def prepare(case, seed):
    vla, c = _pkg(), case
    s = {"case": c, "vla": vla}
    if c["kind"] in ("linear_i8", "linear_f32"):
        s["x"], s["W"], s["ws"], s["b"] = _linear_inputs(c, seed)
        s["out"] = torch.empty(c["M"], c["N"], device=DEV)
        s["act"] = vla.ACT[c["act"]]
        if c["kind"] == "linear_i8":
            s["xq"] = torch.empty(c["M"], _kpad(c["K"]), dtype=torch.int8, device=DEV)
            s["sa"] = torch.empty(c["M"], device=DEV)
    elif c["kind"] == "attention":
        s["q"], s["k"], s["v"] = _attention_inputs(c, seed)
        s["out"] = torch.empty_like(s["q"])
        s["scale"] = 1.0 / math.sqrt(c["hd"])
        m = None
        if c["mask"] == "causal":
            m = vla.VlaMask(kind=vla.MASK_CAUSAL, causal_offset=c["sk"] - c["sq"])
        elif c["mask"] == "dense":
            keep = torch.from_numpy(np.ascontiguousarray(_keep(c))).to(DEV)
            s["dense"] = torch.where(keep, 0.0, torch.finfo(torch.float32).min).to(torch.float32).contiguous()
            m = vla.VlaMask(kind=vla.MASK_DENSE, dense=s["dense"].data_ptr())
        elif c["mask"] in ("suffix", "blocks"):
            s["groups"] = [torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in _groups(c)]
            q, k, allow = s["groups"]
            m = vla.VlaMask(kind=vla.MASK_GROUPS, n_groups=allow.shape[0], q_group=q.data_ptr(),
                            k_group=k.data_ptr(), allow=allow.data_ptr())
        s["mask"] = m
    elif c["kind"] == "conv_i8":
        s["x"], W, b = _conv_inputs(c, seed)
        s["lin"] = vla.LinearI8.from_f32(W.cpu().numpy(), b.cpu().numpy())
        Ho, Wo = _conv_out(c)
        s["out"] = torch.empty(Ho, Wo, c["Cout"], device=DEV)
        n = vla.conv2d_i8_workspace_bytes(c["H"], c["W"], c["Cin"], c["Cout"], c["k"], c["stride"], c["k"] // 2)
        s["work"] = torch.empty(n, dtype=torch.uint8, device=DEV)
    elif c["kind"] == "trunk":
        os.environ["ACT_INT8"] = "63" if c["int8"] else "31"  # read when the model loads
        s["model"] = vla.ActModel(_checkpoint("trunk", _trunk_cfg(c)))
        s["x"] = _frames(c, seed)
        m = s["model"]
        s["out"] = torch.empty(m.n_cams * m.feat_h * m.feat_w, m.feat_ch, device=DEV)
    else:
        cfg = _vision_cfg(c)
        s["model"] = vla.SiglipVision(_checkpoint("vision", cfg), c["int8"])
        s["x"] = torch.rand(3, cfg["img"], cfg["img"], generator=_gen(seed), device=DEV) * 2 - 1
        s["out"] = torch.empty(cfg["n_img_tok"], cfg["mm_out"], device=DEV)
    return s


def run(s):
    c, vla = s["case"], s["vla"]
    if c["kind"] == "linear_i8":
        vla.dense_linear_i8_dev(s["out"], s["x"], s["W"], s["ws"], s["b"], c["K"], s["xq"], s["sa"], act=s["act"])
    elif c["kind"] == "linear_f32":
        vla.dense_linear_dev(s["out"], s["x"], s["W"], s["b"], act=s["act"])
    elif c["kind"] == "attention":
        vla.attention_dev(s["out"], s["q"], s["k"], s["v"], c["n_q"], c["n_kv"], c["hd"], s["scale"], s["mask"])
    elif c["kind"] == "conv_i8":
        vla.conv2d_i8_dev(s["lin"], s["out"], s["x"], c["k"], c["stride"], c["k"] // 2, s["work"])
    else:
        (s["model"].encode_dev)(s["x"], s["out"])
    return s["out"]


# ------------------------------------------------- what a pass has to do --

def _conv_out(c):
    p = c["k"] // 2
    return (c["H"] + 2 * p - c["k"]) // c["stride"] + 1, (c["W"] + 2 * p - c["k"]) // c["stride"] + 1


def _trunk_layers(c):
    """(H, W, Cin, Cout, k, stride, pad) of ResNet-18's convolutions, in the order of backbone.bin."""
    h, w = c["H"], c["W"]
    out = [(h, w, 3, 64, 7, 2, 3)]
    h, w = (h - 1) // 2 + 1, (w - 1) // 2 + 1  # the stem
    h, w = (h - 1) // 2 + 1, (w - 1) // 2 + 1  # the max pool
    cin = 64
    for stage in range(4):
        for b in range(2):
            cout, st = 64 << stage, 2 if stage and not b else 1
            out.append((h, w, cin, cout, 3, st, 1))
            oh, ow = (h - 1) // st + 1, (w - 1) // st + 1
            out.append((oh, ow, cout, cout, 3, 1, 1))
            if st != 1:
                out.append((h, w, cin, cout, 1, st, 0))
            h, w, cin = oh, ow, cout
    return out, h, w


def work(case):
    c = case
    if c["kind"] == "linear_i8":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 4 * M * K + N * K + 8 * N + 4 * M * N, "flops": 2 * M * N * K}
    if c["kind"] == "linear_f32":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": 4 * (M * K + N * K + N + M * N), "flops": 2 * M * N * K}
    if c["kind"] == "attention":
        keep = _keep(c)
        pairs = c["sq"] * c["sk"] if keep is None else int(keep.sum())
        return {"bytes": 4 * c["hd"] * (2 * c["sq"] * c["n_q"] + 2 * c["sk"] * c["n_kv"]) +
                (4 * c["sq"] * c["sk"] if c["mask"] == "dense" else 0), "flops": 4 * pairs * c["hd"] * c["n_q"]}
    if c["kind"] == "conv_i8":
        Ho, Wo = _conv_out(c)
        K = c["k"] ** 2 * c["Cin"]
        return {"bytes": 4 * c["H"] * c["W"] * c["Cin"] + c["Cout"] * (K + 8) + 4 * Ho * Wo * c["Cout"],
                "flops": 2 * Ho * Wo * c["Cout"] * K}
    if c["kind"] == "trunk":
        layers, fh, fw = _trunk_layers(c)
        flops = wb = 0
        for h, w, cin, cout, k, st, p in layers:
            n = ((h + 2 * p - k) // st + 1) * ((w + 2 * p - k) // st + 1)
            flops += 2 * n * cout * cin * k * k
            wb += cout * (cin * k * k * (1 if c["int8"] else 4) + 8)
        return {"bytes": c["cams"] * (3 * c["H"] * c["W"] + 4 * fh * fw * 512) + wb, "flops": c["cams"] * flops}
    H, T, I = 64 * c["heads"], c["side"] ** 2, c["inter"]
    n_tok = (c["side"] // 4) ** 2
    lin = H * 768 + c["layers"] * (4 * H * H + 2 * H * I)
    per = 1 if c["int8"] == 15 else 2 if c["int8"] else 4
    return {"bytes": 4 * 3 * (16 * c["side"]) ** 2 + per * (lin + 16 * H * c["out"]) + 4 * T * H + 4 * n_tok * c["out"],
            "flops": 2 * T * lin + 2 * n_tok * 16 * H * c["out"] + c["layers"] * 4 * T * T * H}


def tolerance(case):
    k = case["kind"]
    if k in ("linear_i8", "conv_i8"):
        # exact integer sums; what is left is the fp32 rounding of the epilogue
        # and of the activation function (seen against 64 bits: rel 4e-8)
        return {"rel": 4e-7, "max": 4e-6}
    if k == "attention":  # sums in another order: rel 3.4e-7, max 2.4e-6
        return {"rel": 2e-6, "max": 2e-5}
    if k == "linear_f32":  # against 64 bits: rel 6e-7 at K = 768, more with longer sums
        return {"rel": 4e-6, "max": 4e-5}
    if k == "trunk" and not case["int8"]:  # against 64 bits: rel 8.3e-7, max 5e-6
        return {"rel": 4e-6, "max": 4e-5}
    if k == "vision" and not case["int8"]:  # against 64 bits: rel 1.3e-6
        return {"rel": 6e-6, "max": 1e-4}
    # one rounding changed ahead of an int8 quantization moves bytes by a whole
    # step, which every later layer sees: the attention's sums in another order
    # alone give rel 0.019, max 0.09 over the 12-layer tower
    return {"rel": 0.03, "max": 0.4}


# ------------------------------------------------------- 64-bit results --

def _act64(v, act):
    if act == "relu":
        return torch.relu(v)
    if act == "gelu_tanh":
        return F.gelu(v, approximate="tanh")
    if act == "gelu_erf":
        return F.gelu(v)
    return v


def _quant_rows(x):
    """The framework's row quantizer: (values on the int8 grid, scale), both in x's type."""
    amax = x.abs().amax(dim=-1, keepdim=True)
    one = torch.ones_like(amax)  # tensors divide: a division by a number is a product with its reciprocal
    s = torch.where(amax > 0, (amax / (127 * one)).clamp_min(torch.finfo(torch.float32).tiny), one)
    return torch.round(x * (one / s)).clamp(-127, 127), s


def _linear64(x, W, b, int8):
    """x in 64 bits through a layer with fp32 weights W, quantized as the layer is when int8."""
    if not int8:
        y = x @ W.double().t()
    else:
        wq, ws = _quant_rows(W.float())
        xq, xs = _quant_rows(x)
        y = (xq @ wq.double().t()) * ws.double().t() * xs
    return y if b is None else y + b.double()


def _exact_conv(x, W, b, k, stride, pad, int8):
    """x [n, Cin, H, W] in 64 bits, W [Cout, k, k, Cin] fp32."""
    Wd = W.float()
    if int8:
        q, ws = _quant_rows(Wd.reshape(W.shape[0], -1))
        Wd = (q.double() * ws.double()).reshape(W.shape)
        xq, s = _quant_rows(x.reshape(-1))
        x = (xq * s).reshape(x.shape)
    # as a product of patches: 64-bit convolutions have no fast library path
    n, cin, h, w = x.shape
    cols = F.unfold(x, k, padding=pad, stride=stride)  # [n, Cin k k, pixels]
    Wm = Wd.double().permute(0, 3, 1, 2).reshape(W.shape[0], -1)
    y = torch.stack([Wm @ cols[i] for i in range(n)]) + b.double()[None, :, None]
    return y.reshape(n, W.shape[0], (h + 2 * pad - k) // stride + 1, (w + 2 * pad - k) // stride + 1)


def exact(case, seed):
    c = case
    if c["kind"] in ("linear_i8", "linear_f32"):
        x, W, ws, b = _linear_inputs(c, seed)
        if c["kind"] == "linear_f32":
            return _act64(_linear64(x.double(), W, b, False), c["act"])
        xq, xs = _quant_rows(x)  # the quantizer is defined in 32 bits
        y = (xq.double() @ W[:, :c["K"]].double().t()) * ws.double()[None, :] * xs.double()
        return _act64(y if b is None else y + b.double(), c["act"])
    if c["kind"] == "attention":
        q, k, v = (t.double() for t in _attention_inputs(c, seed))
        hd, rep = c["hd"], c["n_q"] // c["n_kv"]
        keep = _keep(c)
        keep = None if keep is None else torch.from_numpy(np.ascontiguousarray(keep)).to(DEV)
        out = []
        for h in range(c["n_q"]):
            kv = slice(h // rep * hd, (h // rep + 1) * hd)
            s = (q[:, h * hd:(h + 1) * hd] @ k[:, kv].t().contiguous()) * float(np.float32(1.0 / math.sqrt(hd)))
            if keep is not None:
                s = s.masked_fill(~keep, -math.inf)
            out.append(torch.softmax(s, dim=-1) @ v[:, kv].contiguous())
        return torch.cat(out, dim=1)
    if c["kind"] == "conv_i8":
        x, W, b = _conv_inputs(c, seed)
        k = c["k"]
        # the activation scale and the bytes are defined in 32 bits
        xq, s = _quant_rows(x.reshape(-1))
        xq = xq.reshape(x.shape).double()
        q, ws = _quant_rows(W)
        y = _exact_conv(xq.permute(2, 0, 1)[None], q.reshape(c["Cout"], k, k, c["Cin"]), torch.zeros_like(b), k,
                        c["stride"], k // 2, False)[0]
        y = y.permute(1, 2, 0) * ws.double().reshape(-1) * s.double() + b.double()
        return y.contiguous()
    if c["kind"] == "trunk":
        cfg = _trunk_cfg(c)
        raw = torch.from_numpy(np.fromfile(os.path.join(_checkpoint("trunk", cfg), "backbone.bin"), np.float32)).to(DEV)
        layers, at = [], 0
        for h, w, cin, cout, k, st, p in _trunk_layers(c)[0]:
            n = cout * k * k * cin
            layers.append((raw[at:at + n].reshape(cout, k, k, cin), raw[at + n:at + n + cout], k, st, p, c["int8"]))
            at += n + cout
        mean = torch.tensor([0.485, 0.456, 0.406], device=DEV).double()
        std = torch.tensor([0.229, 0.224, 0.225], device=DEV).double() + cfg["norm_eps"]
        x = ((_frames(c, seed).double() / 255 - mean) / std).permute(0, 3, 1, 2)
        x = F.max_pool2d(torch.relu(_exact_conv(x, *layers[0])), 3, 2, 1)
        i = 1
        for stage in range(4):
            for b in range(2):
                down = stage > 0 and b == 0
                y = torch.relu(_exact_conv(x, *layers[i]))
                y = _exact_conv(y, *layers[i + 1])
                idn = _exact_conv(x, *layers[i + 2]) if down else x
                x = torch.relu(y + idn)
                i += 3 if down else 2
        return x.permute(0, 2, 3, 1).reshape(-1, x.shape[1]).contiguous()
    return _exact_vision(c, seed)


def _exact_vision(c, seed):
    cfg = _vision_cfg(c)
    H, I, T, NL, P, side = cfg["hidden"], cfg["inter"], cfg["n_patches"], cfg["n_layers"], cfg["patch"], c["side"]
    raw = np.fromfile(os.path.join(_checkpoint("vision", cfg), "vit.bin"), np.uint8)
    n32 = H + T * H + NL * (8 * H + I + H) + 2 * H
    f = torch.from_numpy(raw[:4 * n32].view(np.float32).copy()).to(DEV)
    w = torch.from_numpy(raw[4 * n32:].view(np.int16).copy()).view(torch.bfloat16).to(DEV)
    at = [0, 0]

    def vec(*shape):
        n = math.prod(shape)
        at[0] += n
        return f[at[0] - n:at[0]].double().reshape(shape)

    def mat(N, K):
        at[1] += N * K
        return w[at[1] - N * K:at[1]].float().reshape(N, K)

    def ln(v, s, b):
        return F.layer_norm(v, (H,), s, b, float(np.float32(cfg["ln_eps"])))

    m = c["int8"]
    g = _gen(seed)
    px = (torch.rand(3, cfg["img"], cfg["img"], generator=g, device=DEV) * 2 - 1).double()
    patch_b, pos = vec(H), vec(T, H)
    lf = [dict(ln1s=vec(H), ln1b=vec(H), bq=vec(H), bk=vec(H), bv=vec(H), bo=vec(H), ln2s=vec(H), ln2b=vec(H),
               b1=vec(I), b2=vec(H)) for _ in range(NL)]
    post_s, post_b = vec(H), vec(H)
    rows = px.reshape(3, side, P, side, P).permute(1, 3, 0, 2, 4).reshape(T, 3 * P * P)
    x = _linear64(rows, mat(H, 3 * P * P), patch_b, bool(m & 8)) + pos
    heads, hd = c["heads"], 64
    for p in lf:
        h = ln(x, p["ln1s"], p["ln1b"])
        q, k, v = (_linear64(h, mat(H, H), p[b], bool(m & 1)) for b in ("bq", "bk", "bv"))
        o = []
        for i in range(heads):
            sl = slice(i * hd, (i + 1) * hd)
            s = torch.softmax((q[:, sl] @ k[:, sl].t().contiguous()) * float(np.float32(1.0 / math.sqrt(hd))), dim=-1)
            o.append(s @ v[:, sl].contiguous())
        x = x + _linear64(torch.cat(o, dim=1), mat(H, H), p["bo"], bool(m & 1))
        h = ln(x, p["ln2s"], p["ln2b"])
        h = F.gelu(_linear64(h, mat(I, H), p["b1"], bool(m & 2)), approximate="tanh")
        x = x + _linear64(h, mat(H, I), p["b2"], bool(m & 4))
    x = ln(x, post_s, post_b)
    sf = cfg["scale_factor"]
    g2 = side // sf
    x = x.reshape(g2, sf, g2, sf, H).permute(0, 2, 1, 3, 4).reshape(g2 * g2, sf * sf * H)
    return _linear64(x, mat(cfg["mm_out"], sf * sf * H), None, bool(m & 8))
