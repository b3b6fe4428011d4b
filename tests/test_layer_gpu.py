"""The decoder layer's fused operations (csrc/layer.hip through engine/hip_layer.py) against the same operations in
fp64, and a layer on the kernels against the same layer on torch operations.

Bound, for results of N(0, 1) inputs: the output's own bf16 rounding is at most 2^-9 of each value (2^-9 / sqrt(3) =
1.1e-3 in the 2-norm at worst); a normalised operand x * w rounded to bf16 adds a relative error of the same size to
every term of a product, independent from term to term, so again at most 1.1e-3 in the 2-norm, and the gated product
of SwiGLU carries it twice. Together under 2^-8 = 3.9e-3.
"""

import pytest
import torch
import torch.nn.functional as F

from cases import fragmented_manager
from engine import hip_layer
from engine.config import ModelConfig
from engine.model import Layer, Qwen2Model, rms_norm, rotate
from engine.paged_cache import PagedKVCache, build_metadata

pytestmark = pytest.mark.gpu

BOUND = 2.0 ** -8
EPS = 1e-6
TOKENS = [1, 2, 15, 16, 17, 31, 32, 33, 64, 65, 129, 300]


def rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


def randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.bfloat16)


def norm64(x, w):
    x = x.double()
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def rotate64(x, cos, sin):
    h = x.shape[-1] // 2
    return x * cos.double() + torch.cat([x[..., h:], x[..., :h]], -1) * sin.double()


# (hidden, heads, rotated heads, head_dim): the two model shapes, one slice of K, more slices than waves take at once
SHAPES = [(896, 18, 16, 64), (1536, 16, 14, 128), (64, 3, 2, 16), (4096, 2, 1, 32)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("T", TOKENS)
def test_projection_with_norm_and_rotary(T, shape):
    hidden, heads, rotated, d = shape
    g = torch.Generator(device="cuda").manual_seed(T)
    x, nw, w, b = randn(g, T, hidden), 1 + 0.1 * randn(g, hidden), randn(g, heads * d, hidden) * 0.05, randn(g, heads * d)
    rot = randn(g, T, 1, d), randn(g, T, 1, d)
    print(f"case rotary T {T} {shape}", flush=True)
    out = hip_layer.fused_linear(x, w, hip_layer.ROPE, norm_weight=nw, eps=EPS, bias=b, rot=rot, head_dim=d,
                                 rot_channels=rotated * d)
    y = (norm64(x, nw) @ w.double().t() + b.double()).view(T, heads, d)
    ref = torch.cat([rotate64(y[:, :rotated], *rot), y[:, rotated:]], 1).view(T, -1)
    assert rel(out, ref) < BOUND


@pytest.mark.parametrize("inter,hidden", [(4864, 896), (8960, 1536), (8, 64)])
@pytest.mark.parametrize("T", TOKENS)
def test_gated_projection(T, inter, hidden):
    g = torch.Generator(device="cuda").manual_seed(T)
    x, nw, w = randn(g, T, hidden), 1 + 0.1 * randn(g, hidden), randn(g, 2 * inter, hidden) * 0.05
    print(f"case gated T {T} {inter} x {hidden}", flush=True)
    out = hip_layer.fused_linear(x, w, hip_layer.SILU, norm_weight=nw, eps=EPS)
    y = norm64(x, nw) @ w.double().t()
    assert rel(out, F.silu(y[:, :inter]) * y[:, inter:]) < BOUND


@pytest.mark.parametrize("out_f,in_f", [(896, 4864), (1536, 8960), (896, 896), (16, 64), (48, 320)])
@pytest.mark.parametrize("splits", [0, 1, 2, 7])
@pytest.mark.parametrize("T", [1, 16, 17, 33, 65, 300])
def test_projection_with_residual(T, splits, out_f, in_f):
    """Split K too: more splits than slices of K among them; a second call finds the counters at zero."""
    g = torch.Generator(device="cuda").manual_seed(T)
    x, w, res = randn(g, T, in_f), randn(g, out_f, in_f) * 0.05, randn(g, T, out_f)
    print(f"case residual T {T} splits {splits} {out_f} x {in_f}", flush=True)
    ref = x.double() @ w.double().t() + res.double()
    first = hip_layer.fused_linear(x, w, hip_layer.RESIDUAL, residual=res, num_splits=splits)
    again = hip_layer.fused_linear(x, w, hip_layer.RESIDUAL, residual=res, num_splits=splits)
    assert rel(first, ref) < BOUND
    assert torch.equal(first, again)


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("T", [1, 16, 33, 129])
def test_every_tile_shape(tile, T):
    """Each tile of the projection kernels with each epilogue, at row counts that fill no whole tile (120 rows of 16 for
    tiles of up to 128) and a K of 5 slices (less and more than the slices in flight)."""
    if tile == 6 and T > 16:
        return
    g = torch.Generator(device="cuda").manual_seed(T)
    K, d, heads, inter = 320, 48, 5, 120
    x, nw, res, b = randn(g, T, K), 1 + 0.1 * randn(g, K), randn(g, T, heads * d), randn(g, heads * d)
    w, gu = randn(g, heads * d, K) * 0.05, randn(g, 2 * inter, K) * 0.05
    rot = randn(g, T, 1, d), randn(g, T, 1, d)
    print(f"case tile {tile} T {T}", flush=True)
    xn = norm64(x, nw)
    y = (xn @ w.double().t() + b.double()).view(T, heads, d)
    out = hip_layer.fused_linear(x, w, hip_layer.ROPE, norm_weight=nw, eps=EPS, bias=b, rot=rot, head_dim=d,
                                 rot_channels=3 * d, tile=tile)
    assert rel(out, torch.cat([rotate64(y[:, :3], *rot), y[:, 3:]], 1).view(T, -1)) < BOUND
    out = hip_layer.fused_linear(x, gu, hip_layer.SILU, norm_weight=nw, eps=EPS, tile=tile)
    y = xn @ gu.double().t()
    assert rel(out, F.silu(y[:, :inter]) * y[:, inter:]) < BOUND
    ref = x.double() @ w.double().t() + res.double() + b.double()
    for splits in (1, 2) if tile < 6 else (1,):
        out = hip_layer.fused_linear(x, w, hip_layer.RESIDUAL, bias=b, residual=res, num_splits=splits, tile=tile)
        assert rel(out, ref) < BOUND


@pytest.mark.parametrize("tile", [0, 1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("T", [1, 16, 33, 129])
def test_epilogues_with_and_without_norm(tile, T):
    """The forms that a Qwen2 layer does not use: a residual after a normed product, rotary and gated ones without norm."""
    if tile == 6 and T > 16:
        return
    g = torch.Generator(device="cuda").manual_seed(T)
    K, d, heads, inter = 320, 48, 5, 120
    x, nw, res, b = randn(g, T, K), 1 + 0.1 * randn(g, K), randn(g, T, heads * d), randn(g, heads * d)
    w, gu = randn(g, heads * d, K) * 0.05, randn(g, 2 * inter, K) * 0.05
    rot = randn(g, T, 1, d), randn(g, T, 1, d)
    print(f"case forms tile {tile} T {T}", flush=True)
    out = hip_layer.fused_linear(x, w, hip_layer.RESIDUAL, norm_weight=nw, eps=EPS, bias=b, residual=res, tile=tile)
    assert rel(out, norm64(x, nw) @ w.double().t() + b.double() + res.double()) < BOUND
    y = (x.double() @ w.double().t() + b.double()).view(T, heads, d)
    out = hip_layer.fused_linear(x, w, hip_layer.ROPE, bias=b, rot=rot, head_dim=d, rot_channels=3 * d, tile=tile)
    assert rel(out, torch.cat([rotate64(y[:, :3], *rot), y[:, 3:]], 1).view(T, -1)) < BOUND
    out = hip_layer.fused_linear(x, gu, hip_layer.SILU, tile=tile)
    y = x.double() @ gu.double().t()
    assert rel(out, F.silu(y[:, :inter]) * y[:, inter:]) < BOUND


@pytest.mark.parametrize("hidden,inter,Hq,d", [(896, 4864, 14, 64), (1536, 8960, 12, 128)])
@pytest.mark.parametrize("T", [400, 544, 700, 1000, 1024])
def test_projections_of_larger_batches(T, hidden, inter, Hq, d):
    """Both model shapes' four projections at the tiles and splits that the library takes itself."""
    g = torch.Generator(device="cuda").manual_seed(T)
    heads = Hq + 4
    x, nw, b = randn(g, T, hidden), 1 + 0.1 * randn(g, hidden), randn(g, heads * d)
    rot = randn(g, T, 1, d), randn(g, T, 1, d)
    print(f"case larger T {T} {hidden}", flush=True)
    xn = norm64(x, nw)
    w = randn(g, heads * d, hidden) * 0.05
    out = hip_layer.fused_linear(x, w, hip_layer.ROPE, norm_weight=nw, eps=EPS, bias=b, rot=rot, head_dim=d,
                                 rot_channels=(Hq + 2) * d)
    y = (xn @ w.double().t() + b.double()).view(T, heads, d)
    assert rel(out, torch.cat([rotate64(y[:, :Hq + 2], *rot), y[:, Hq + 2:]], 1).view(T, -1)) < BOUND
    w = randn(g, 2 * inter, hidden) * 0.05
    y = xn @ w.double().t()
    assert rel(hip_layer.fused_linear(x, w, hip_layer.SILU, norm_weight=nw, eps=EPS),
               F.silu(y[:, :inter]) * y[:, inter:]) < BOUND
    for K in (hidden, inter):
        a, w, res = randn(g, T, K), randn(g, hidden, K) * 0.05, randn(g, T, hidden)
        out = hip_layer.fused_linear(a, w, hip_layer.RESIDUAL, residual=res)
        assert rel(out, a.double() @ w.double().t() + res.double()) < BOUND


@pytest.mark.parametrize("K", [8, 896, 1024, 1032, 1536, 2056, 8192])
@pytest.mark.parametrize("T", [1, 4, 5, 300])
def test_rms_norm_rows(T, K):
    """The kernel rounds where the torch operations do: equal but for the order of the sum of squares (a row factor one
    fp32 step off flips few roundings), the residual sum bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(K)
    x, add, w = randn(g, T, K), randn(g, T, K), 1 + 0.1 * randn(g, K)
    out, s = hip_layer.rms_norm(x, w, EPS, add=add)
    assert torch.equal(s, x + add)
    ref = rms_norm(x + add, w, EPS)
    assert (out != ref).float().mean() < 0.01 and rel(out, ref.double()) < 2 ** -9
    assert torch.equal(hip_layer.rms_norm(s, w, EPS), out)


@pytest.mark.parametrize("T,heads,extra,d", [(1, 1, 0, 16), (7, 16, 2, 64), (300, 14, 2, 128)])
def test_rope_and_silu_rows(T, heads, extra, d):
    g = torch.Generator(device="cuda").manual_seed(T)
    x = randn(g, T, (heads + extra) * d)
    rot = randn(g, T, 1, d), randn(g, T, 1, d)
    y = x.clone()
    hip_layer.rope_(y, rot, heads, d)
    ref = rotate64(x.view(T, -1, d)[:, :heads].double(), *rot).reshape(T, -1)
    assert rel(y[:, :heads * d], ref) < 2 ** -9
    assert torch.equal(y[:, heads * d:], x[:, heads * d:])
    gu = randn(g, T, 2 * heads * d)
    half = heads * d
    assert rel(hip_layer.silu_mul(gu), F.silu(gu[:, :half].double()) * gu[:, half:].double()) < 2 ** -9


@pytest.mark.parametrize("T", [1, 16, 33, 130, 1025])
def test_layer_on_kernels_matches_torch_operations(T):
    """layer_forward under inference_mode (the kernels) against the same call outside it (the torch operations), and
    what the layer wrote into the cache."""
    for a, b in zip(*run_layer_both_ways(T, 896, 4864, 14, 64)[0]):
        # the torch side rounds up to 16 times along a chain of operations (norm 2, projection, rotary 3, attention,
        # projection, sum, norm 2, projection, gate 2, projection, sum), at most 2^-9 of the value each and independent:
        # sqrt(16) 2^-9 = 2^-7 a side, 2^-6 between two sides
        assert rel(a, b.double()) < 2.0 ** -6


@pytest.mark.parametrize("hidden,inter,Hq,d", [(896, 4864, 14, 64), (1536, 8960, 12, 128)])
@pytest.mark.parametrize("T", ["below", "above", 1024, 1025])
def test_layer_on_either_side_of_the_gated_limit(T, hidden, inter, Hq, d):
    """The last batch whose gated projection is fused, the first whose goes to the library between fused projections, the
    last and first batch around MAX_TOKENS, against 64 bits: no further from it than the torch operations, whose roundings
    are a superset of the kernels' (2% for the draw of the others)."""
    most = int(hip_layer.MAX_GATED_FLOPS / (4.0 * hidden * inter))
    assert most < 1024
    T = {"below": most, "above": most + 1}.get(T, T)
    (kernels, torch_ops), (x, w, rot) = run_layer_both_ways(T, hidden, inter, Hq, d)
    qkv = (norm64(x, w.input_norm) @ w.qkv_w.double().t() + w.qkv_b.double()).view(T, Hq + 4, d)
    qk, v = rotate64(qkv[:, :Hq + 2], *rot), qkv[:, Hq + 2:]
    k, v = (t.transpose(0, 1).repeat_interleave(Hq // 2, 0) for t in (qk[:, Hq:], v))
    score = torch.bmm(qk[:, :Hq].transpose(0, 1), k.transpose(1, 2).contiguous()) * d ** -0.5
    score.masked_fill_(torch.ones(T, T, device="cuda", dtype=torch.bool).triu(1), -torch.inf)
    attn = torch.bmm(torch.softmax(score, -1), v.contiguous()).transpose(0, 1).reshape(T, Hq * d)
    ref = layer_out64(x, attn, w)
    assert rel(kernels[0], ref) <= 1.02 * rel(torch_ops[0], ref) < 2.0 ** -5
    for a, b in zip(kernels[1:], torch_ops[1:]):  # K (rounded four times less) and V in the pools
        assert rel(a, b.double()) < 2.0 ** -7


def run_layer_both_ways(T, hidden, inter, Hq, d):
    """([hidden states and pools on the kernels, the same on torch operations], (x, weights, rotary rows))"""
    cfg = ModelConfig(vocab_size=64, hidden_size=hidden, intermediate_size=inter, num_layers=1, num_q_heads=Hq,
                      num_kv_heads=2, head_dim=d)
    model = Qwen2Model(cfg, "cuda", torch.bfloat16, seed=1, max_positions=2048, std=0.05)
    g = torch.Generator(device="cuda").manual_seed(2)
    x = randn(g, T, hidden)
    print(f"case layer T {T} {hidden}", flush=True)
    results = []
    for fused in (True, False):
        m = fragmented_manager(128, 16, torch.Generator().manual_seed(3))
        cache = PagedKVCache(cfg, m.num_blocks, 16, "cuda", torch.bfloat16, attn_backend="hip")
        cache.k.zero_()
        cache.v.zero_()
        m.allocate(0, T)
        meta = build_metadata(m, [(0, 0, T)], "cuda")
        cache.begin(T, meta)
        rot = model.rotary.rows(meta.positions, torch.bfloat16)
        with torch.inference_mode() if fused else torch.no_grad():
            assert hip_layer.supported(x, model.layers[0], rot, Hq + 4, d) == fused
            results.append((model.layer_forward(0, x, meta.positions, cache, rot), cache.k, cache.v))
    return results, (x, model.layers[0], rot)


def test_rotate_reference_matches_the_model():
    g = torch.Generator(device="cuda").manual_seed(9)
    x, rot = randn(g, 5, 3, 32), (randn(g, 5, 1, 32), randn(g, 5, 1, 32))
    assert rel(rotate(x, *rot), rotate64(x.double(), *rot)) < BOUND


@pytest.mark.parametrize("T", [1, 16, 17, 64, 300])
@pytest.mark.parametrize("d,Hq,Hkv", [(64, 14, 2), (128, 12, 2), (16, 4, 4)])
def test_projection_stores_to_the_paged_pools(T, d, Hq, Hkv):
    """K and V stored by the projection: the bits that the projection without pools and store_tokens give, nothing else
    in the pools touched, and the same queries."""
    from engine.hip_quant import store_tokens

    hidden, heads = 320, Hq + 2 * Hkv
    g = torch.Generator(device="cuda").manual_seed(T)
    x, nw, w, b = randn(g, T, hidden), 1 + 0.1 * randn(g, hidden), randn(g, heads * d, hidden) * 0.05, randn(g, heads * d)
    rot = randn(g, T, 1, d), randn(g, T, 1, d)
    cfg = ModelConfig(vocab_size=64, hidden_size=hidden, intermediate_size=64, num_layers=3, num_q_heads=Hq,
                      num_kv_heads=Hkv, head_dim=d)
    m = fragmented_manager(64, 16, torch.Generator().manual_seed(4))
    cache = PagedKVCache(cfg, m.num_blocks, 16, "cuda", torch.bfloat16, attn_backend="hip")
    m.allocate(0, T + 5)
    meta = build_metadata(m, [(0, 5, T)], "cuda")
    cache.begin(T, meta)
    cache.k.fill_(7)
    cache.v.fill_(9)
    kw = dict(norm_weight=nw, eps=EPS, bias=b, rot=rot, head_dim=d, rot_channels=(Hq + Hkv) * d)
    store = cache.store_target(1, x, Hkv, d)
    q = hip_layer.fused_linear(x, w, hip_layer.ROPE, store=store, **kw).view(T, heads, d)[:, :Hq]
    ref = hip_layer.fused_linear(x, w, hip_layer.ROPE, **kw).view(T, heads, d)
    k, v = torch.full_like(cache.k, 7), torch.full_like(cache.v, 9)
    store_tokens(ref[:, Hq:Hq + Hkv], meta.slot_blocks, meta.slot_offsets, k[1], x2=ref[:, Hq + Hkv:], pool2=v[1])
    assert torch.equal(q, ref[:, :Hq]) and torch.equal(cache.k, k) and torch.equal(cache.v, v)


def test_caches_that_write_their_own_way_are_asked_to():
    cfg = ModelConfig(vocab_size=64, hidden_size=896, intermediate_size=64, num_layers=1, num_q_heads=14, num_kv_heads=2,
                      head_dim=64)
    m = fragmented_manager(64, 16, torch.Generator().manual_seed(4))

    class Own(PagedKVCache):
        def write(self, layer, k, v):
            super().write(layer, k, v)

    x = torch.zeros(4, 896, device="cuda", dtype=torch.bfloat16)
    m.allocate(0, 4)
    meta = build_metadata(m, [(0, 0, 4)], "cuda")
    for make, dtype, taken in ((PagedKVCache, torch.bfloat16, True), (Own, torch.bfloat16, False),
                               (PagedKVCache, torch.float32, False)):
        cache = make(cfg, m.num_blocks, 16, "cuda", dtype, attn_backend="hip")
        assert cache.store_target(0, x, 2, 64) is None  # no forward begun
        cache.begin(4, meta)
        assert (cache.store_target(0, x, 2, 64) is not None) == taken
        assert cache.store_target(0, x[:3], 2, 64) is None and cache.store_target(0, x, 4, 64) is None
        assert cache.store_target(0, x.cpu(), 2, 64) is None
        cache.write = lambda layer, k, v: None
        assert cache.store_target(0, x, 2, 64) is None


def test_a_wrapped_cache_keeps_its_write():
    """An object that passes names on to a cache, and a subclass whose write is found by __getattribute__, see every write
    of a layer."""
    cfg = ModelConfig(vocab_size=64, hidden_size=128, intermediate_size=64, num_layers=1, num_q_heads=4, num_kv_heads=2,
                      head_dim=32)
    model = Qwen2Model(cfg, "cuda", torch.bfloat16, seed=1, max_positions=64, std=0.05)
    m = fragmented_manager(16, 16, torch.Generator().manual_seed(4))
    m.allocate(0, 5)
    meta = build_metadata(m, [(0, 0, 5)], "cuda")
    seen = []

    class Wrapper:
        def __init__(self, cache):
            self.cache = cache

        def __getattr__(self, name):
            return getattr(self.cache, name)

        def write(self, layer, k, v):
            seen.append((k.clone(), v.clone()))
            self.cache.write(layer, k, v)

    class Watched(PagedKVCache):
        def __getattribute__(self, name):
            found = super().__getattribute__(name)
            if name != "write":
                return found
            return lambda layer, k, v: (seen.append((k.clone(), v.clone())), found(layer, k, v))

    x = randn(torch.Generator(device="cuda").manual_seed(2), 5, 128)
    rot = model.rotary.rows(meta.positions, torch.bfloat16)
    results = []
    for make in (PagedKVCache, lambda *a, **kw: Wrapper(PagedKVCache(*a, **kw)), Watched):
        cache = make(cfg, m.num_blocks, 16, "cuda", torch.bfloat16, attn_backend="hip")
        cache.begin(5, meta)
        seen.clear()
        with torch.inference_mode():
            results.append(model.layer_forward(0, x, meta.positions, cache, rot))
        assert len(seen) == (make is not PagedKVCache)
        for k, v in seen:
            assert torch.equal(cache.k[0][:, meta.slot_blocks, meta.slot_offsets], k.transpose(0, 1))
            assert torch.equal(cache.v[0][:, meta.slot_blocks, meta.slot_offsets], v.transpose(0, 1))
    assert torch.equal(results[0], results[1]) and torch.equal(results[0], results[2])


@pytest.mark.parametrize("T", [1, 3, 40])
def test_attention_results_of_other_forms(T):
    """What a cache's attend returns is read by the kernels only in the form that they take: other strides and offsets
    give the layer's result all the same, other types and sizes raise as the torch operations do."""
    cfg = ModelConfig(vocab_size=64, hidden_size=128, intermediate_size=64, num_layers=1, num_q_heads=4, num_kv_heads=2,
                      head_dim=32)
    model = Qwen2Model(cfg, "cuda", torch.bfloat16, seed=1, max_positions=64, std=0.05)
    g = torch.Generator(device="cuda").manual_seed(2)
    x, pos, attn = randn(g, T, 128), torch.arange(T, device="cuda"), randn(g, T, 128)
    rot = model.rotary.rows(pos, torch.bfloat16)

    class Given:
        def write(self, layer, k, v):
            pass

        def attend(self, layer, q, positions, scale):
            return self.out

    cache = Given()

    def layer(out):
        cache.out = out
        with torch.inference_mode():
            return model.layer_forward(0, x, pos, cache, rot)

    ref = layer(attn)
    wide = torch.zeros(T, 256, device="cuda", dtype=torch.bfloat16)
    odd = torch.zeros(T * 128 + 1, device="cuda", dtype=torch.bfloat16)
    for view in (wide[:, 64:192], wide[:, ::2], wide[:, 3:131], odd[1:].view(T, 128),
                 torch.zeros(128, T, device="cuda", dtype=torch.bfloat16).t()):
        view.copy_(attn)
        assert rel(layer(view), ref.double()) < 2.0 ** -6  # torch operations against kernels, as above
    bad_rows = [attn.repeat(2, 1)] if T > 1 else []  # one row of x broadcasts over them
    for bad in [attn.float(), attn[:, :64].contiguous(), torch.cat([attn, attn], 1), attn.cpu()] + bad_rows:
        with pytest.raises(RuntimeError):
            layer(bad)


def test_autocast_keeps_the_torch_operations():
    cfg = ModelConfig(vocab_size=64, hidden_size=128, intermediate_size=64, num_layers=1, num_q_heads=4, num_kv_heads=2,
                      head_dim=32)
    model = Qwen2Model(cfg, "cuda", torch.bfloat16, seed=1, max_positions=64, std=0.05)
    x = torch.zeros(4, 128, device="cuda", dtype=torch.bfloat16)
    rot = model.rotary.rows(torch.arange(4, device="cuda"), torch.bfloat16)
    with torch.inference_mode():
        assert hip_layer.supported(x, model.layers[0], rot, 8, 32)
        with torch.autocast("cuda", torch.float16):
            assert not hip_layer.supported(x, model.layers[0], rot, 8, 32)
            assert not hip_layer.rows_ok(x, model.final_norm)


def layer_weights(g, hidden, attn, inter):
    return Layer(None, None, None, randn(g, hidden, attn) * 0.05, 1 + 0.1 * randn(g, hidden), randn(g, 2 * inter, hidden) * 0.05,
                 randn(g, hidden, inter) * 0.05)


def layer_out64(x, attn, w):
    h = x.double() + attn.double() @ w.o_w.double().t()
    gate, up = (norm64(h, w.post_norm) @ w.gate_up_w.double().t()).chunk(2, -1)
    return h + (F.silu(gate) * up) @ w.down_w.double().t()


@pytest.mark.parametrize("T,hidden,attn,inter", [(8, 896, 896, 4864), (128, 896, 896, 4864), (512, 1536, 1536, 8960),
                                                 (20, 128, 4096, 4096)])
def test_captured_layers_own_their_merge_counters(T, hidden, attn, inter):
    """Layers whose projections share K among workgroups, captured twice on a stream without a workspace: the second
    graph is replayed before the first, the stream's workspace is made, replaced and overwritten in between, and the two
    are replayed side by side on two streams. Every replay gives the eager result."""
    from engine.hip_decode import reserve_workspace

    g = torch.Generator(device="cuda").manual_seed(T)
    w = layer_weights(g, hidden, attn, inter)
    inputs = [(randn(g, T, hidden), randn(g, T, attn)) for _ in range(2)]
    print(f"case captured layer T {T} {hidden} {attn} {inter}", flush=True)
    s, other = torch.cuda.Stream(), torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        eager = [hip_layer.layer_out(x, a, w, EPS) for x, a in inputs]
    torch.cuda.synchronize()
    for (x, a), out in zip(inputs, eager):
        # h, the activations and the sum are rounded to bf16, each 2^-9 at worst, beside the gated product's bound
        assert rel(out, layer_out64(x, a, w)) < 2 * BOUND
    torch.cuda.synchronize()
    graphs = []
    for x, a in inputs:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            outs = [hip_layer.layer_out(x, a, w, EPS) for _ in range(3)]
        graphs.append((graph, outs))
    torch.cuda.synchronize()

    def check(i):
        torch.cuda.synchronize()
        for out in graphs[i][1]:
            assert torch.equal(out, eager[i])
            out.fill_(7)
        torch.cuda.synchronize()

    for i in (1, 0, 1):
        graphs[i][0].replay()
        check(i)
    for nbytes in (1 << 20, 8 << 20, 24 << 20):
        ws = reserve_workspace(torch.device("cuda"), s.cuda_stream, nbytes)
        torch.cuda.synchronize()
        junk = [torch.full((1 << 18,), 0x5a5a5a5a, device="cuda", dtype=torch.int32) for _ in range(8)]
        graphs[0][0].replay()
        check(0)
        assert not ws.any()
        del junk
    if 4.0 * T * hidden * inter > hip_layer.MAX_GATED_FLOPS:
        return  # a library product among them: torch gives the stream's graphs one library workspace
    for _ in range(5):
        with torch.cuda.stream(s):
            graphs[0][0].replay()
        with torch.cuda.stream(other):
            graphs[1][0].replay()
        check(0)
        check(1)


def test_transforms_and_modes_keep_the_torch_operations():
    """vmap over a layer, and modes that are to see each of its operations, under inference_mode: what the torch operations
    give; the default device's own mode changes nothing."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    cfg = ModelConfig(vocab_size=64, hidden_size=128, intermediate_size=64, num_layers=1, num_q_heads=4, num_kv_heads=2,
                      head_dim=32)
    model = Qwen2Model(cfg, "cuda", torch.bfloat16, seed=1, max_positions=64, std=0.05)
    g = torch.Generator(device="cuda").manual_seed(2)
    xs, pos = randn(g, 3, 4, 128), torch.arange(4, device="cuda")
    rot = model.rotary.rows(pos, torch.bfloat16)

    class Values:  # each query head returns its group's values
        def write(self, layer, k, v):
            self.v = v

        def attend(self, layer, q, positions, scale):
            return self.v.repeat_interleave(2, 1).reshape(q.shape[0], -1)

    def layer(x):
        return model.layer_forward(0, x, pos, Values(), rot)

    linears = []

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            linears.append(func is F.linear)
            return func(*args, **(kwargs or {}))

    class Operations(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            linears.append(func in (torch.ops.aten.mm.default, torch.ops.aten.addmm.default, torch.ops.aten.linear.default))
            return func(*args, **(kwargs or {}))

    with torch.no_grad():
        ref = [layer(x) for x in xs]
    with torch.inference_mode():
        assert hip_layer.supported(xs[0], model.layers[0], rot, 8, 32)
        with torch.device("cuda"):
            assert hip_layer.supported(xs[0], model.layers[0], rot, 8, 32)
        out = torch.func.vmap(layer)(xs)
        for mode in (Functions, Operations):
            linears.clear()
            with mode():
                seen = layer(xs[0])
            assert sum(linears) == 4 and torch.equal(seen, ref[0])
        traced = torch.jit.trace(layer, (xs[0],), check_trace=False)(xs[1])
    assert torch.equal(traced, ref[1])
    for a, b in zip(out, ref):
        assert rel(a, b.double()) < 2.0 ** -6
