"""The work that this library is measured by: what a text-to-image program has it do, through the C device API.

A picture takes, once, the layers of the text encoder; then, for every sampling step, the blocks of a transformer over
the joint text + image rows; at the end (or, for an image given as input, at the start) the stages of the VAE. Each kind
of case below is one such piece, issued call by call as a host program issues it. Sizes follow the picture: 256 x 256
pixels are 256 image tokens, 1024 x 1024 are 4096, two reference images triple that; text is padded to a fixed length.

Rows are bf16, the residual stream and the images are f32, weights are bf16: the only types the API has. Weights and
workspaces are laid out once (`prepare`), as a program that holds a model keeps them.
"""
import math

import torch

import iris_c_amd

HD = 128                                        # head size of every transformer here
ENC = dict(hidden=2560, inter=9728, heads=32, kv=8)   # the text encoder: grouped keys, causal, split-half rotation
EPS = 1e-6
GROUPS = 32                                     # group norm of the VAE

_dev = None


def _lib():
    global _dev
    if _dev is None:
        _dev = iris_c_amd.IrisDev()
    return _dev.lib


# ---------------------------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # Q and K normalised and rotated in place, then joint attention: the pair of operators the library is built
        # around. The smallest picture, the usual one, a pair of guidance halves whose second one masks its padding, and
        # an edit with two reference images.
        dict(name="step_320", kind="step", heads=24, seq=320, valid=320),
        dict(name="step_4608", kind="step", heads=24, seq=4608, valid=4608),
        dict(name="step_4352_masked", kind="step", heads=30, seq=4352, valid=4233),
        dict(name="step_12800", kind="step", heads=24, seq=12800, valid=12800),
        # a text-encoder layer over a prompt of 118 tokens in the usual 512
        dict(name="encoder_512", kind="encoder", seq=512, valid=118),
        # a single-stream transformer block: the smallest picture with a short text, and the usual one
        dict(name="single_320", kind="single", heads=24, seq=320),
        dict(name="single_4608", kind="single", heads=24, seq=4608),
        # a double-stream block, text and image rows with weights of their own; an image of no round size (720 x 752 pixels)
        dict(name="double_2627", kind="double", heads=24, txt=512, img=2115),
        # the VAE around a 1024 x 1024 picture: attention over all latent positions, a decoder stage (256 -> 512 pixels
        # wide), the first encoder stage, and the last layer of the decoder
        dict(name="vae_attention_16384", kind="vae_attention", h=128, w=128),
        dict(name="vae_up_256", kind="vae_up", h=256, w=256, cin=256, cout=128),
        dict(name="vae_down_512", kind="vae_down", h=512, w=512),
        dict(name="vae_out_1024", kind="vae_out", h=1024, w=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "encoder", "single", "single", "double", "double", "vae_attention", "vae_up",
                       "vae_down", "vae_out"])
    if kind == "step":
        heads = rng.choice([24, 30, 32])
        seq = _log(rng, 80, 12800 if heads == 24 else 11000)
        # a mask in a third of the cases: the last rows are the padding of a text of at most 512 tokens
        return dict(kind=kind, heads=heads, seq=seq, valid=seq - rng.randrange(1, min(seq, 512)) if rng.random() < 0.34 else seq)
    if kind == "encoder":
        seq = _log(rng, 80, 1280)
        return dict(kind=kind, seq=seq, valid=rng.randrange(min(8, seq), seq + 1))
    if kind == "single":
        heads = rng.choice([24, 32])
        return dict(kind=kind, heads=heads, seq=_log(rng, 80, 4608 if heads == 24 else 2600))
    if kind == "double":
        heads = rng.choice([24, 32])
        return dict(kind=kind, heads=heads, txt=_log(rng, 64, 512), img=_log(rng, 256, 4096 if heads == 24 else 2600))
    # the VAE at 256 .. 1024 pixels a side
    if kind == "vae_attention":
        return dict(kind=kind, h=rng.randrange(32, 129), w=rng.randrange(32, 129))
    if kind == "vae_up":
        cin, cout = rng.choice([(512, 512), (512, 256), (256, 128)])
        most = 128 if cin == 512 else 256
        return dict(kind=kind, h=rng.randrange(most // 4, most + 1), w=rng.randrange(most // 4, most + 1), cin=cin, cout=cout)
    most = 512 if kind == "vae_down" else 1024
    return dict(kind=kind, h=rng.randrange(most // 4, most + 1), w=rng.randrange(most // 4, most + 1))


# --------------------------------------------------------------------------------------------------------------- inputs
class _Make:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def f32(self, *shape, s=1.0, at=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda").mul_(s).add_(at)

    def bf16(self, *shape, s=1.0):
        return self.f32(*shape, s=s).to(torch.bfloat16)

    def weight(self, out, cin):
        return self.bf16(out, cin, s=1.0 / math.sqrt(cin))

    def tables(self, seq):
        """cos and sin of angles that cover the circle [seq, 64], as the higher frequencies of a rotary table do"""
        ang = torch.rand(seq, HD // 2, generator=self.g, device="cuda").mul_(6.2).sub_(3.1)
        return torch.cos(ang), torch.sin(ang)


def _empty(*shape, dtype):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    _lib()
    s = dict(case)
    globals()["_prepare_" + case["kind"]](s, _Make(seed))
    torch.cuda.synchronize()
    return s


def _prepare_step(s, m):
    seq, dim = s["seq"], s["heads"] * HD
    s["h"] = m.bf16(seq, 3 * dim)
    # norm weights at their initial value: the norm of a row that a pass has already normalised is then as good an
    # input as the first
    s["wq"], s["wk"] = torch.ones(HD, device="cuda"), torch.ones(HD, device="cuda")
    s["cos"], s["sin"] = m.tables(seq)
    s["mask"] = (torch.arange(seq, device="cuda") < s["valid"]).to(torch.int32) if s["valid"] < seq else None
    s["out"] = _empty(seq, dim, dtype=torch.bfloat16)


def _prepare_encoder(s, m):
    seq, hid, inter, q, kv = s["seq"], ENC["hidden"], ENC["inter"], ENC["heads"] * HD, ENC["kv"] * HD
    s["x"] = m.f32(seq, hid, s=1.5)
    s["n1"], s["n2"] = m.f32(hid, s=0.05, at=1.0), m.f32(hid, s=0.05, at=1.0)
    s["wqkv"], s["wo"] = m.weight(q + 2 * kv, hid), m.weight(hid, q)
    s["wgu"], s["wdown"] = m.weight(2 * inter, hid), m.weight(hid, inter)
    s["wq"], s["wk"] = m.f32(HD, s=0.05, at=1.0), m.f32(HD, s=0.05, at=1.0)
    s["cos"], s["sin"] = m.tables(seq)
    s["mask"] = (torch.arange(seq, device="cuda") < s["valid"]).to(torch.int32)
    s["norm"], s["qkv"], s["att"] = (_empty(seq, n, dtype=torch.bfloat16) for n in (hid, q + 2 * kv, q))
    s["gu"], s["act"] = (_empty(seq, n, dtype=torch.bfloat16) for n in (2 * inter, inter))
    s["out"] = _empty(seq, hid, dtype=torch.float32)


def _prepare_single(s, m):
    seq, dim = s["seq"], s["heads"] * HD
    mlp = 3 * dim
    s["x"], s["mod"] = m.f32(seq, dim, s=1.5), m.f32(3 * dim, s=0.3)
    s["win"], s["wout"] = m.weight(3 * dim + 2 * mlp, dim), m.weight(dim, dim + mlp)
    s["wq"], s["wk"] = m.f32(HD, s=0.05, at=1.0), m.f32(HD, s=0.05, at=1.0)
    s["cos"], s["sin"] = m.tables(seq)
    s["norm"], s["h"], s["cat"] = (_empty(seq, n, dtype=torch.bfloat16) for n in (dim, 3 * dim + 2 * mlp, dim + mlp))
    s["out"] = _empty(seq, dim, dtype=torch.float32)


def _prepare_double(s, m):
    seq, dim = s["txt"] + s["img"], s["heads"] * HD
    mlp = 3 * dim
    s["x"] = m.f32(seq, dim, s=1.5)
    s["cos"], s["sin"] = m.tables(seq)
    s["streams"] = [dict(mod=m.f32(6 * dim, s=0.3), wqkv=m.weight(3 * dim, dim), wproj=m.weight(dim, dim),
                         wff1=m.weight(2 * mlp, dim), wff2=m.weight(dim, mlp),
                         wq=m.f32(HD, s=0.05, at=1.0), wk=m.f32(HD, s=0.05, at=1.0)) for _ in range(2)]
    s["norm"], s["cat"] = _empty(seq, dim, dtype=torch.bfloat16), _empty(seq, mlp, dtype=torch.bfloat16)
    s["h"] = _empty(seq, 2 * mlp, dtype=torch.bfloat16)
    s["out"] = _empty(seq, dim, dtype=torch.float32)


def _conv(m, cin, cout, k):
    return m.weight(cout, k * k * cin), m.f32(cout, s=0.1)


def _affine(m, c):
    return m.f32(c, s=0.1, at=1.0), m.f32(c, s=0.1)


def _prepare_vae_attention(s, m):
    hw, c = s["h"] * s["w"], 512
    s["x"], s["gn"] = m.f32(hw, c), _affine(m, c)
    s["qkv_w"], s["qkv_b"] = _conv(m, c, 3 * c, 1)
    s["o_w"], s["o_b"] = _conv(m, c, c, 1)
    s["t1"], s["t2"], s["out"] = (_empty(hw, n, dtype=torch.float32) for n in (c, 3 * c, c))
    s["qkv"], s["att"] = (_empty(hw, n, dtype=torch.bfloat16) for n in (3 * c, c))


def _resblock_weights(s, m, cin, cout):
    s["gn1"], s["gn2"] = _affine(m, cin), _affine(m, cout)
    s["c1"], s["c2"] = _conv(m, cin, cout, 3), _conv(m, cout, cout, 3)
    s["skip"] = _conv(m, cin, cout, 1) if cin != cout else None


def _prepare_vae_up(s, m):
    hw, cin, cout = s["h"] * s["w"], s["cin"], s["cout"]
    s["x"] = m.f32(hw, cin)
    s["up"] = _conv(m, cin, cin, 3)
    _resblock_weights(s, m, cin, cout)
    s["t0"], s["t1"], s["t2"], s["out"] = (_empty(4 * hw, n, dtype=torch.float32) for n in (cin, cin, cin, cout))


def _prepare_vae_down(s, m):
    hw, c = s["h"] * s["w"], 128
    s["x"] = m.f32(hw, 3, s=0.5)
    s["first"], s["down"] = _conv(m, 3, c, 3), _conv(m, c, c, 3)
    _resblock_weights(s, m, c, c)
    s["t0"], s["t1"], s["t2"], s["res"] = (_empty(hw, c, dtype=torch.float32) for _ in range(4))
    s["out"] = _empty(((s["h"] - 2) // 2 + 1) * ((s["w"] - 2) // 2 + 1), c, dtype=torch.float32)


def _prepare_vae_out(s, m):
    hw, c = s["h"] * s["w"], 128
    s["x"], s["gn"] = m.f32(hw, c), _affine(m, c)
    s["last"] = _conv(m, c, 3, 3)
    s["t1"], s["out"] = _empty(hw, c, dtype=torch.float32), _empty(hw, 3, dtype=torch.float32)


# ----------------------------------------------------------------------------------------------------------------- runs
def run(s):
    return globals()["_run_" + s["kind"]](_lib(), s)


def _p(t, elems=0):
    return t.data_ptr() + elems * t.element_size() if t is not None else None


_SCALE = 1.0 / math.sqrt(HD)


def _run_step(L, s):
    """iris_dev_head_norm_rope on Q and on K, iris_dev_attention"""
    seq, heads = s["seq"], s["heads"]
    dim = heads * HD
    h, cos, sin = s["h"], _p(s["cos"]), _p(s["sin"])
    L.iris_dev_head_norm_rope(_p(h), 3 * dim, _p(s["wq"]), cos, sin, seq, heads, HD, EPS, 0)
    L.iris_dev_head_norm_rope(_p(h, dim), 3 * dim, _p(s["wk"]), cos, sin, seq, heads, HD, EPS, 0)
    L.iris_dev_attention(_p(s["out"]), dim, _p(h), _p(h, dim), _p(h, 2 * dim), 3 * dim, seq, seq, heads, heads, HD, _SCALE, 0,
                         _p(s["mask"]))
    return h, s["out"]


def _run_encoder(L, s):
    """A layer of the text encoder: norm, q | k | v, norm + rope, causal attention under a padding mask, projection, MLP."""
    seq, hid, inter, heads, kv = s["seq"], ENC["hidden"], ENC["inter"], ENC["heads"], ENC["kv"]
    qd, ld = heads * HD, (heads + 2 * kv) * HD
    x, norm, qkv, gu, out = s["x"], _p(s["norm"]), s["qkv"], s["gu"], _p(s["out"])
    cos, sin = _p(s["cos"]), _p(s["sin"])
    L.iris_dev_rms_norm(norm, _p(x), _p(s["n1"]), seq, hid, EPS)
    L.iris_dev_linear_bf16(_p(qkv), norm, _p(s["wqkv"]), seq, hid, ld)
    L.iris_dev_head_norm_rope(_p(qkv), ld, _p(s["wq"]), cos, sin, seq, heads, HD, EPS, 1)
    L.iris_dev_head_norm_rope(_p(qkv, qd), ld, _p(s["wk"]), cos, sin, seq, kv, HD, EPS, 1)
    L.iris_dev_attention(_p(s["att"]), qd, _p(qkv), _p(qkv, qd), _p(qkv, qd + kv * HD), ld, seq, seq, heads, kv, HD, _SCALE, 1,
                         _p(s["mask"]))
    L.iris_dev_linear_f32(out, _p(s["att"]), _p(s["wo"]), seq, qd, hid)
    L.iris_dev_residual(_p(x), out, None, seq, hid)
    L.iris_dev_rms_norm(norm, _p(x), _p(s["n2"]), seq, hid, EPS)
    L.iris_dev_linear_bf16(_p(gu), norm, _p(s["wgu"]), seq, hid, 2 * inter)
    L.iris_dev_swiglu(_p(s["act"]), inter, _p(gu), _p(gu, inter), 2 * inter, seq, inter)
    L.iris_dev_linear_f32(out, _p(s["act"]), _p(s["wdown"]), seq, inter, hid)
    L.iris_dev_residual(_p(x), out, None, seq, hid)
    return x


def _run_single(L, s):
    """A single-stream block; the projection normalises its own Q and K columns."""
    seq, heads = s["seq"], s["heads"]
    dim, mlp = heads * HD, 3 * heads * HD
    ldh, ldc = 3 * dim + 2 * mlp, dim + mlp
    x, mod, h, cat, norm = s["x"], s["mod"], s["h"], s["cat"], _p(s["norm"])
    L.iris_dev_layer_norm_mod(norm, _p(x), _p(mod), _p(mod, dim), seq, dim, EPS)
    L.iris_dev_linear_bf16_qknorm(_p(h), norm, _p(s["win"]), seq, dim, ldh, heads, heads, HD, _p(s["wq"]), _p(s["wk"]),
                                  _p(s["cos"]), _p(s["sin"]), EPS, 0)
    L.iris_dev_attention(_p(cat), ldc, _p(h), _p(h, dim), _p(h, 2 * dim), ldh, seq, seq, heads, heads, HD, _SCALE, 0, None)
    L.iris_dev_swiglu(_p(cat, dim), ldc, _p(h, 3 * dim), _p(h, 3 * dim + mlp), ldh, seq, mlp)
    L.iris_dev_linear_f32(_p(s["out"]), _p(cat), _p(s["wout"]), seq, ldc, dim)
    L.iris_dev_residual(_p(x), _p(s["out"]), _p(mod, 2 * dim), seq, dim)
    return x


def _run_double(L, s):
    """A double-stream block: every stream its own projections and norms, one attention over the rows of both."""
    txt, img, heads = s["txt"], s["img"], s["heads"]
    seq, dim, mlp = txt + img, heads * HD, 3 * heads * HD
    x, h, cat, norm, out = s["x"], s["h"], s["cat"], _p(s["norm"]), _p(s["out"])
    parts = ((0, txt, s["streams"][0]), (txt, img, s["streams"][1]))
    for first, n, w in parts:
        L.iris_dev_layer_norm_mod(norm, _p(x, first * dim), _p(w["mod"]), _p(w["mod"], dim), n, dim, EPS)
        L.iris_dev_linear_bf16(_p(h, 3 * first * dim), norm, _p(w["wqkv"]), n, dim, 3 * dim)
    a, b = s["streams"]
    L.iris_dev_head_norm_rope_qk_streams(_p(h), _p(h, dim), 3 * dim, _p(a["wq"]), _p(a["wk"]), _p(b["wq"]), _p(b["wk"]), txt,
                                         _p(s["cos"]), _p(s["sin"]), seq, heads, heads, HD, EPS, 0)
    L.iris_dev_attention(_p(cat), dim, _p(h), _p(h, dim), _p(h, 2 * dim), 3 * dim, seq, seq, heads, heads, HD, _SCALE, 0, None)
    for first, n, w in parts:
        L.iris_dev_linear_f32(out, _p(cat, first * dim), _p(w["wproj"]), n, dim, dim)
        L.iris_dev_residual(_p(x, first * dim), out, _p(w["mod"], 2 * dim), n, dim)
    for first, n, w in parts:
        xs = _p(x, first * dim)
        L.iris_dev_layer_norm_mod(norm, xs, _p(w["mod"], 3 * dim), _p(w["mod"], 4 * dim), n, dim, EPS)
        L.iris_dev_linear_bf16(_p(h), norm, _p(w["wff1"]), n, dim, 2 * mlp)
        L.iris_dev_swiglu(_p(cat), mlp, _p(h), _p(h, mlp), 2 * mlp, n, mlp)
        L.iris_dev_linear_f32(out, _p(cat), _p(w["wff2"]), n, mlp, dim)
        L.iris_dev_residual(xs, out, _p(w["mod"], 5 * dim), n, dim)
    return x


def _run_vae_attention(L, s):
    """The VAE's attention block: group norm, q | k | v as a 1 x 1 convolution, one head of 512, projection, skip."""
    hw, c = s["h"] * s["w"], 512
    t1, t2, qkv, out = _p(s["t1"]), _p(s["t2"]), s["qkv"], _p(s["out"])
    L.iris_dev_group_norm(t1, _p(s["x"]), _p(s["gn"][0]), _p(s["gn"][1]), hw, c, GROUPS, EPS, 0)
    L.iris_dev_conv2d(t2, t1, _p(s["qkv_w"]), _p(s["qkv_b"]), hw, 1, c, 3 * c, 1, 1, 0, 0)
    L.iris_dev_f32_to_bf16(_p(qkv), t2, hw * 3 * c)
    L.iris_dev_attention(_p(s["att"]), c, _p(qkv), _p(qkv, c), _p(qkv, 2 * c), 3 * c, hw, hw, 1, 1, c, 1.0 / math.sqrt(c), 0, None)
    L.iris_dev_linear_f32(out, _p(s["att"]), _p(s["o_w"]), hw, c, c)
    L.iris_dev_add_bias(out, _p(s["o_b"]), hw, c)
    L.iris_dev_add(out, _p(s["x"]), hw * c)
    return s["out"]


def _resblock(L, s, out, x, h, w, cin, cout, t1, t2):
    """out = skip(x) + conv(silu(norm(conv(silu(norm(x))))))"""
    hw = h * w
    L.iris_dev_group_norm(t1, x, _p(s["gn1"][0]), _p(s["gn1"][1]), hw, cin, GROUPS, EPS, 1)
    L.iris_dev_conv2d(t2, t1, _p(s["c1"][0]), _p(s["c1"][1]), h, w, cin, cout, 3, 1, 1, 1)
    L.iris_dev_group_norm(t1, t2, _p(s["gn2"][0]), _p(s["gn2"][1]), hw, cout, GROUPS, EPS, 1)
    L.iris_dev_conv2d(out, t1, _p(s["c2"][0]), _p(s["c2"][1]), h, w, cout, cout, 3, 1, 1, 1)
    if s["skip"] is not None:
        L.iris_dev_conv2d(t2, x, _p(s["skip"][0]), _p(s["skip"][1]), h, w, cin, cout, 1, 1, 0, 0)
        L.iris_dev_add(out, t2, hw * cout)
    else:
        L.iris_dev_add(out, x, hw * cout)


def _run_vae_up(L, s):
    """Between two decoder stages: nearest-neighbour upsampling, its convolution, the next stage's first residual block."""
    h, w, cin, cout = s["h"], s["w"], s["cin"], s["cout"]
    t0, t1, t2 = _p(s["t0"]), _p(s["t1"]), _p(s["t2"])
    L.iris_dev_upsample2x(t1, _p(s["x"]), h, w, cin)
    L.iris_dev_conv2d(t0, t1, _p(s["up"][0]), _p(s["up"][1]), 2 * h, 2 * w, cin, cin, 3, 1, 1, 1)
    _resblock(L, s, _p(s["out"]), t0, 2 * h, 2 * w, cin, cout, t1, t2)
    return s["out"]


def _run_vae_down(L, s):
    """The first encoder stage: 3 channels to 128, a residual block, halved by a convolution of stride 2."""
    h, w, c = s["h"], s["w"], 128
    t0, res = _p(s["t0"]), _p(s["res"])
    L.iris_dev_conv2d(t0, _p(s["x"]), _p(s["first"][0]), _p(s["first"][1]), h, w, 3, c, 3, 1, 1, 1)
    _resblock(L, s, res, t0, h, w, c, c, _p(s["t1"]), _p(s["t2"]))
    L.iris_dev_conv2d(_p(s["out"]), res, _p(s["down"][0]), _p(s["down"][1]), h, w, c, c, 3, 2, 0, 1)
    return s["out"]


def _run_vae_out(L, s):
    """The end of the decoder: norm, SiLU, 128 channels to the picture's 3."""
    h, w, c = s["h"], s["w"], 128
    L.iris_dev_group_norm(_p(s["t1"]), _p(s["x"]), _p(s["gn"][0]), _p(s["gn"][1]), h * w, c, GROUPS, EPS, 1)
    L.iris_dev_conv2d(_p(s["out"]), _p(s["t1"]), _p(s["last"][0]), _p(s["last"][1]), h, w, c, 3, 3, 1, 1, 1)
    return s["out"]


# ----------------------------------------------------------------------------------------------------------------- work
def _keys(seq, valid, causal):
    """(query, valid key) pairs"""
    if not causal:
        return seq * valid
    return valid * (valid + 1) // 2 + (seq - valid) * valid


def work(case):
    k = case["kind"]
    if k in ("step", "encoder", "single"):
        seq = case["seq"]
    if k == "step":
        dim = case["heads"] * HD
        # q | k | v and both tables in, q, k and the attention output out
        return {"bytes": 2 * seq * 6 * dim + 4 * seq * HD, "flops": 4 * dim * _keys(seq, case["valid"], False)}
    if k == "encoder":
        hid, inter, q, kv = ENC["hidden"], ENC["inter"], ENC["heads"] * HD, ENC["kv"] * HD
        w = (q + 2 * kv) * hid + hid * q + 3 * inter * hid
        return {"bytes": 2 * w + 8 * seq * hid + 4 * seq * HD, "flops": 2 * seq * w + 4 * q * _keys(seq, case["valid"], True)}
    if k == "single":
        dim = case["heads"] * HD
        w = 9 * dim * dim + 4 * dim * dim
        return {"bytes": 2 * w + 8 * seq * dim + 4 * seq * HD, "flops": 2 * seq * w + 4 * dim * seq * seq}
    if k == "double":
        seq, dim = case["txt"] + case["img"], case["heads"] * HD
        w = (3 + 1 + 6 + 3) * dim * dim
        return {"bytes": 2 * 2 * w + 8 * seq * dim + 4 * seq * HD, "flops": 2 * seq * w + 4 * dim * seq * seq}
    hw = case["h"] * case["w"]
    if k == "vae_attention":
        return {"bytes": 8 * hw * 512 + 2 * 4 * 512 * 512, "flops": 2 * hw * 4 * 512 * 512 + 4 * 512 * hw * hw}
    if k == "vae_up":
        cin, cout = case["cin"], case["cout"]
        w = 9 * cin * cin + 9 * cin * cout + 9 * cout * cout + (cin * cout if cin != cout else 0)
        return {"bytes": 4 * hw * cin + 4 * 4 * hw * cout + 2 * w, "flops": 2 * 4 * hw * w}
    if k == "vae_down":
        out = ((case["h"] - 2) // 2 + 1) * ((case["w"] - 2) // 2 + 1)
        return {"bytes": 4 * hw * 3 + 4 * out * 128 + 2 * 9 * (3 + 3 * 128) * 128,
                "flops": 2 * 9 * 128 * (hw * (3 + 2 * 128) + out * 128)}
    return {"bytes": 4 * hw * (128 + 3) + 2 * 9 * 128 * 3, "flops": 2 * hw * 9 * 128 * 3}


def tolerance(case):
    return dict(TOLERANCE[case["kind"]])


# About four times the distance of a pass from the same chain in 64-bit arithmetic (rel / max): step 3.3e-3 / 2.3e-2 (the
# attention output; q and k 1.4e-3), encoder 1.6e-3 / 1.0e-2, single 5.0e-4 / 6.9e-3, double 5.6e-4 / 7.1e-3 (the residual
# stream, most of which a pass leaves alone), vae_attention 2.9e-4 / 1.5e-3 (likewise), vae_up 2.5e-3 / 1.4e-2,
# vae_down 3.0e-3 / 1.7e-2, vae_out 1.5e-3 / 7.0e-3.
TOLERANCE = {
    "step": {"rel": 1.2e-2, "max": 0.09},
    "encoder": {"rel": 6e-3, "max": 0.04},
    "single": {"rel": 2e-3, "max": 0.028},
    "double": {"rel": 2.2e-3, "max": 0.028},
    "vae_attention": {"rel": 1.2e-3, "max": 0.006},
    "vae_up": {"rel": 1e-2, "max": 0.055},
    "vae_down": {"rel": 1.2e-2, "max": 0.07},
    "vae_out": {"rel": 6e-3, "max": 0.03},
}
