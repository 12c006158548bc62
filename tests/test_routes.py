"""Which calls take the faster forms of products, embeddings and attention: a call outside what a form reads stays with the general one."""
import pytest
import torch

from msa_amd import seq_ops


@pytest.fixture
def anywhere(monkeypatch):
    monkeypatch.setattr(seq_ops, "_cuda", lambda *a: None)


def test_prefill_attention_of_other_types(anywhere):
    q, k = torch.zeros((600, 512)), torch.zeros((600, 512))
    batch = seq_ops.StepBatch([600], [0], [0], "cpu")
    ok = lambda q, k, v: seq_ops.takes_flash_rows(q, k, v, 4, 4, 128, 128, 0, batch)
    assert ok(q.bfloat16(), k.bfloat16(), k.bfloat16())
    for a, b, c in ((q, k, k), (q.half(), k.half(), k.half()), (q.bfloat16(), k, k), (q.bfloat16(), k.bfloat16(), k)):
        assert not ok(a, b, c)


class _Doubled(torch.nn.Linear):
    def forward(self, x):
        return 2 * super().forward(x)


def test_modules_whose_call_is_not_their_class_s_own():
    from torch.nn.modules import module as m
    from msa_amd import ops
    plain = lambda x: ops.plain_module(x, torch.nn.Linear)
    lin = torch.nn.Linear(4, 4)
    assert plain(lin) and not plain(_Doubled(4, 4)) and not plain(torch.nn.Identity()) and not plain(object())
    for register in (lin.register_forward_hook, lin.register_forward_pre_hook, lin.register_full_backward_hook, m.register_module_forward_hook,
                     m.register_module_forward_pre_hook, m.register_module_full_backward_hook):
        h = register(lambda *a: None)
        assert not plain(lin)
        h.remove()
        assert plain(lin)
    lin.forward = lambda x: x
    assert not plain(lin)
    del lin.forward
    assert plain(lin)


@pytest.fixture
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from msa_amd import ops
    return ops


@pytest.mark.gpu
def test_an_mlp_with_a_call_of_its_own(gpu):
    """A layer adds what calling its MLP gives: a subclass's, an instance's or another module's forward, and a hook's result."""
    from torch.nn.modules import module as m
    from msa_amd.config import MSAConfig
    from msa_amd.model import MLP, MSADecoderLayer

    class Attention(torch.nn.Module):
        def forward(self, x, *a, **k):
            return x * 0.5, None

    class Tripled(MLP):
        def forward(self, x):
            return 3 * super().forward(x)

    cfg = MSAConfig(hidden_size=1024, intermediate_size=3072, num_hidden_layers=1)
    torch.manual_seed(0)
    layer = MSADecoderLayer(cfg, 0)
    layer.self_attn = Attention()
    tripled = Tripled(cfg)
    layer, tripled = layer.cuda().bfloat16().requires_grad_(False), tripled.cuda().bfloat16().requires_grad_(False)
    tripled.load_state_dict(layer.mlp.state_dict())
    own = layer.mlp
    x = torch.randn((1, 9600, 1024), device="cuda").bfloat16()       # (the products of 9600 rows are tiled ones)

    def added():
        """What the layer adds behind its attention, and that times one over the plain MLP's output."""
        h = x.clone()
        y = layer(h, None, None, None, None)
        return (y.float() - (x + gpu.rmsnorm(x, layer.input_layernorm.weight, 1e-6) * 0.5).float())
    base = added()
    assert gpu.linear_ok(own.down_proj, torch.empty((1, 9600, 3072), device="cuda").bfloat16(), end=True)
    # (rounding the stream to bf16 leaves 2^-9 of values some ten times the MLP's, three times over)
    close = lambda got, times: ((got - times * base).norm() / base.norm()).item() < 0.06 * max(1, times)
    layer.mlp = tripled
    print("[routes] subclass", flush=True)
    assert close(added(), 3)
    layer.mlp = own
    inner = own.forward
    own.forward = lambda x: 2 * inner(x)
    assert close(added(), 2)
    del own.forward
    assert close(added(), 1)
    h = m.register_module_forward_hook(lambda mod, i, o: o * 0 if mod is own else None)
    assert close(added(), 0)
    h.remove()
    layer.mlp = torch.nn.Identity()
    n = gpu.rmsnorm(x + gpu.rmsnorm(x, layer.input_layernorm.weight, 1e-6) * 0.5, layer.post_attention_layernorm.weight, 1e-6).float()
    assert ((added() - n).norm() / n.norm()).item() < 0.02


@pytest.mark.gpu
def test_linear_and_embedding_with_a_call_of_their_own(gpu):
    lin = torch.nn.Linear(1024, 4096, bias=False).cuda().bfloat16().requires_grad_(False)
    x = torch.randn((4096, 1024), device="cuda").bfloat16()
    assert gpu.linear_ok(lin, x)
    lin.forward = lambda x: x[:, :8]
    assert not gpu.linear_ok(lin, x) and torch.equal(gpu.linear(lin, x), x[:, :8])


@pytest.mark.parametrize("interleaved", [False, True])
def test_joined_weights_follow_their_parts(interleaved):
    """Also of a model made in inference mode, whose tensors have no version."""
    from msa_amd import ops
    from msa_amd.config import MSAConfig
    from msa_amd.model import MLP
    want = lambda m: (ops.interleave_gate_up if interleaved else lambda *w: torch.cat(w))(m.gate_proj.weight, m.up_proj.weight)
    cfg = MSAConfig(hidden_size=64, intermediate_size=128)
    with torch.inference_mode():
        m = MLP(cfg)
        assert torch.equal(m._gate_up(interleaved), want(m))
    m = MLP(cfg).requires_grad_(False)
    first = m._gate_up(interleaved)
    assert torch.equal(first, want(m)) and m._gate_up(interleaved) is first
    m.up_proj.weight.mul_(2)
    assert torch.equal(m._gate_up(interleaved), want(m))
    m.gate_proj.weight = torch.nn.Parameter(torch.randn(128, 64))
    assert torch.equal(m._gate_up(interleaved), want(m))
    # a captured step goes on reading the memory that it was captured with
    assert m._gate_up(interleaved).data_ptr() == first.data_ptr() and torch.equal(first, want(m))
    m.double()
    assert m._gate_up(interleaved).dtype == torch.float64 and torch.equal(m._gate_up(interleaved), want(m))


class _On:
    """What a route looks at of a dense bf16 matrix on some device."""
    dtype, is_cuda, requires_grad = torch.bfloat16, True, False

    def __init__(self, device, *shape):
        self.device, self.shape = torch.device(device), shape

    dim = lambda self: len(self.shape)
    numel = lambda self: self.shape[0] * self.shape[1]
    is_contiguous = lambda self: True
    stride = lambda self, i: (self.shape[1], 1)[i]
    data_ptr = lambda self: 4096


def test_operands_of_different_devices(monkeypatch):
    from msa_amd import ops
    x, w = _On("cuda:0", 8192, 2048), _On("cuda:0", 4096, 2048)
    assert ops.tile_linear_ok(x, w) and ops.tile_linear_ok(x, w, end=False)
    assert not ops.tile_linear_ok(x, _On("cuda:1", 4096, 2048))
    # without an end a round of whole tiles is the vendor's, unless its tiles do not fit the columns either
    few = _On("cuda:0", 4000, 2048)
    assert ops.tile_linear_ok(few, w) and not ops.tile_linear_ok(few, w, end=False)
    assert ops.tile_linear_ok(few, _On("cuda:0", 3000, 2048), end=False)
    monkeypatch.setattr(ops, "_need_cuda", lambda *a: None)
    with pytest.raises(ValueError, match="device"):
        ops.tile_linear(x, _On("cuda:1", 4096, 2048))
    with pytest.raises(ValueError, match="device"):
        ops.tile_linear(x, w, out=_On("cuda:1", 8192, 4096))


@pytest.mark.parametrize("rows", [0, 1, 300])
def test_products_of_no_depth(rows):
    from msa_amd import ops
    x, w = torch.zeros((rows, 0)), torch.zeros((5, 0))
    assert not ops.tile_linear_ok(x, w) and not ops.tile_linear_ok(x[None], w, 2) and not ops.block_linear_ok(x, w)
    assert seq_ops.product(x, w).shape == (rows, 5)


@pytest.mark.parametrize("T,K,N,taken", [(450, 2560, 2560, True), (769, 9728, 2560, True), (48, 9728, 2560, True), (640, 2560, 7680, True), (1200, 2560, 2560, True),
                                         (1119, 1024, 4256, True), (33, 3072, 1024, True), (769, 2560, 2560, True), (573, 2560, 12384, False), (1000, 2560, 7680, False),
                                         (1793, 4096, 4096, False), (640, 4096, 2560, False), (400, 4096, 4096, False), (257, 4096, 2560, False), (300, 5120, 2560, False)])
def test_products_that_another_form_makes_sooner(T, K, N, taken):
    """Plain products of one round of mid-sized tiles: those that are behind the vendor's or the smaller tiles go there.  With an end, which costs
    the vendor's another launch, they stay where the smaller tiles are not asked for."""
    from msa_amd import _lib
    lib = _lib.load()
    assert (lib.msa_flow_linear_us(T, K, N, _lib.TILE_STORE) > 0) == taken
    if lib.msa_block_linear_us(T, K, N) > 23:
        assert lib.msa_flow_linear_us(T, K, N, _lib.TILE_GELU) > 0


def _err(got, want):
    return ((got.float() - want).norm() / want.norm()).item()


@pytest.mark.gpu
@pytest.mark.parametrize("T,K,N", [(2500, 1024, 8192), (2500, 1024, 5136), (1900, 1024, 4096)])
def test_products_of_a_step(gpu, monkeypatch, T, K, N):
    """The decoders' products against fp32 where the tiled form takes them (the first two; the third with the vendor's or the small tiles'):
    one rounding to bf16, 1.7e-3 over many values; three for the gated unit and gelu, the gate's passed on by up to 1.3 (4e-3)."""
    taken = []
    inner = gpu.tile_linear
    monkeypatch.setattr(gpu, "tile_linear", lambda x, w, **k: (taken.append(sorted(k)), inner(x, w, **k))[1])
    g = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn((T, K + 32), generator=g, device="cuda").bfloat16()[:, 8:K + 8]
    w = (torch.randn((N, K), generator=g, device="cuda") * K ** -0.5).bfloat16()
    want = x.float() @ w.float().t()
    assert _err(seq_ops.product(x, w), want) < 3e-3
    n = N // 2 // 128 * 128 + 8
    act = torch.nn.functional.gelu(want[:, :n], approximate="tanh")
    got = seq_ops.product_gelu(x, w, n)
    assert _err(got[:, :n], act) < 4e-3 and _err(got[:, n:], want[:, n:]) < 3e-3
    gate, up = want[:, 0::2].clamp(max=1.5), want[:, 1::2].clamp(-1.5, 1.5)
    got = seq_ops.product_glu(x, w, 1.5)
    assert _err(got, gate * torch.sigmoid(seq_ops.GLU_ALPHA * gate) * (up + seq_ops.GLU_SHIFT)) < 4e-3
    assert taken == ([[], ["gelu_n"], ["glu"]] if T * N >= gpu.TILE_MIN else [])


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 300, 1400, 1700, 9300])
def test_mlp(gpu, T):
    """Both sides of the lines of the two products, before and after an update of a weight in place.  The activation and the output are
    rounded to bf16, and the gate and up sums may be: four roundings, each of 1.7e-3 over many values."""
    from msa_amd.config import MSAConfig
    from msa_amd.model import MLP
    print(f"[routes] mlp T={T}", flush=True)
    torch.manual_seed(T)
    m = MLP(MSAConfig(hidden_size=1024, intermediate_size=3072)).cuda().bfloat16().requires_grad_(False)
    x, base = torch.randn((1, T, 1024), device="cuda").bfloat16(), torch.randn((1, T, 1024), device="cuda").bfloat16()
    for _ in range(2):
        gate, up, down = (p.weight.float() for p in (m.gate_proj, m.up_proj, m.down_proj))
        want = (torch.nn.functional.silu(x.float() @ gate.t()) * (x.float() @ up.t())) @ down.t()
        assert _err(m(x), want) < 5e-3
        out = base.clone()
        assert m.add_to(out, x).data_ptr() == out.data_ptr() and _err(out, base.float() + want) < 5e-3
        m.up_proj.weight.mul_(-1.5)
