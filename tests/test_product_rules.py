"""Which operands the products of a few rows take to their fused kernels: rules on the host, checked without a GPU."""
import copy
import types
import weakref

import pytest
import torch

from prelude_amd.models.causal_lm import CausalLM
from prelude_amd.ops import kernels as K
from prelude_amd.parts.attention import GQAAttention
from prelude_amd.parts.base import FeedForward
from prelude_amd.parts.block import PreNormBlock
from prelude_amd.parts.mlp import GatedMLP
from prelude_amd.parts.norm import RMSNorm


def tiled(n, k):
    return K.LinearWeight(torch.zeros(n, k, dtype=torch.bfloat16), K.TiledWeight(torch.zeros(1, dtype=torch.bfloat16), n, k))


def view(shape, off, dtype=torch.bfloat16):
    """A contiguous tensor whose first element lies ``off`` elements behind a 16-byte boundary."""
    n = int(torch.Size(shape).numel())
    buf = torch.zeros(n + 16, dtype=dtype)
    skip = (-buf.data_ptr() % 16) // buf.element_size() + off
    return buf[skip: skip + n].view(shape)


@pytest.mark.parametrize("off", [0, 1, 4, 7, 8])
def test_an_activation_rides_in_a_product_of_aligned_rows_alone(off):
    """The kernel reads rows in 16-byte pieces: an aligned tensor is taken (and refused here, for there is no GPU), another
    goes the way of the product and the activation apart."""
    x, w = view((3, 64), off), tiled(32, 64)
    if off % 8 == 0:
        with pytest.raises(K.NativeError):
            K._linear_few_act(x, w, 1)
    else:
        assert K._linear_few_act(x, w, 1) is None


@pytest.mark.parametrize("which", ["rows", "slices", "residual", "gain"])
def test_the_norm_rides_in_a_product_of_aligned_operands_alone(which):
    off = {"rows": 0, "slices": 0, "residual": 0, "gain": 0, which: 1}
    w, gain = tiled(64, 512), view((512,), off["gain"], torch.float32)
    x = K.SliceSums(view((2, 3, 512), off["slices"], torch.float32), torch.bfloat16) if which == "slices" else view((3, 512), off["rows"])
    assert not K.after_norm_few_supported(x, view((3, 512), off["residual"]), w, gain)
    whole = K.SliceSums(view((2, 3, 512), 0, torch.float32), torch.bfloat16) if which == "slices" else view((3, 512), 0)
    assert K.after_norm_few_supported(whole, view((3, 512), 0), w, view((512,), 0, torch.float32))


class PlainNorm:
    """Stands for an RMS norm: one that a kernel behind it could take in."""
    TAKES_SLICE_SUMS = TAKES_BRANCHES = True

    def as_rms(self):
        return torch.ones(512), 1e-6

    def forward_residual(self, x, residual):
        return residual + x, ("normed", residual + x)


def test_a_part_with_a_forward_of_its_own_keeps_it_behind_a_norm(monkeypatch):
    """Classes derived from the parts that take a norm into their first product, and an instance whose forward was wrapped, run
    their own forward; the parts themselves take the norm in."""
    for name in ("after_norm_few_supported", "gated_after_norm_supported"):
        monkeypatch.setattr(K, name, lambda *a: True)
    monkeypatch.setattr(K, "linear_after_norm_few", lambda x, residual, *a, **kw: (residual + x, "one kernel"))
    monkeypatch.setattr(K, "linear_gated_after_norm", lambda x, residual, *a, **kw: (residual + x, "one kernel"))
    monkeypatch.setattr(K, "linear", lambda h, *a, **kw: h)
    monkeypatch.setattr(GQAAttention, "_fused_decode", lambda self, x, step, cache: True)
    monkeypatch.setattr(GQAAttention, "_decode", lambda self, qkv, step, cache: torch.ones(2))

    class Scaled(GQAAttention):
        def forward(self, x, step, cache, write_cache=True):
            assert x[0] == "normed"
            return torch.full((2,), 7.0)

    class Own(GatedMLP):
        def forward(self, x):
            return x, "own"

    def heads(cls):
        mixer = cls.__new__(cls)
        mixer.w_qkv = mixer.b_qkv = None
        return mixer

    def feed_forward(cls):
        ffn = cls.__new__(cls)
        ffn.gate_up, ffn.down, ffn.activation = None, None, "silu"
        return ffn

    x, residual = torch.zeros(2), torch.zeros(2)

    def run(mixer, ffn):
        return PreNormBlock(PlainNorm(), mixer, PlainNorm(), ffn).forward(x, residual, None, None)

    h, res = run(heads(GQAAttention), feed_forward(GatedMLP))
    assert h == "one kernel" and torch.equal(res, torch.ones(2))
    h, res = run(heads(Scaled), feed_forward(Own))
    assert h[1] == "own" and torch.equal(res, torch.full((2,), 7.0))
    wrapped = heads(GQAAttention)
    wrapped.forward = types.MethodType(Scaled.forward, wrapped)
    assert torch.equal(run(wrapped, feed_forward(GatedMLP))[1], torch.full((2,), 7.0))


def test_a_norm_with_a_residual_step_of_its_own_is_not_taken_for_the_plain_one():
    class Halved(RMSNorm):
        def forward_residual(self, x, residual):
            residual, h = super().forward_residual(x, residual)
            return residual, h / 2

    class Named(RMSNorm):
        pass

    assert RMSNorm(8, 1e-6).as_rms() is not None and Named(8, 1e-6).as_rms() is not None
    assert Halved(8, 1e-6).as_rms() is None
    wrapped = RMSNorm(8, 1e-6)
    wrapped.forward_residual = lambda x, residual: (residual, x)
    assert wrapped.as_rms() is None


@pytest.mark.parametrize("limit", [0.0, -1.0, float("nan")])
def test_a_clamped_pair_without_a_clamp_is_refused_at_any_number_of_rows(monkeypatch, limit):
    """At many rows (``gemm_block``) as at few, before anything is launched: what stands for the tensors is never read."""
    monkeypatch.setattr(K, "_dev", lambda *ts: None)
    monkeypatch.setattr(K, "_stream", lambda: None)
    w = tiled(2048, 64)
    for rows in (3, 200):
        with pytest.raises(K.NativeError, match="clamp"):
            K.linear_clamped_gate(view((rows, 64), 0), w, limit, 1.702)
    with pytest.raises(K.NativeError, match="clamp"):
        K.gemm_block(view((200, 64), 0), w.tiles, activation="clamped", limit=limit, shape=0)


def model_of(*blocks):
    model = CausalLM.__new__(CausalLM)
    model.blocks = [types.SimpleNamespace(**b) for b in blocks]
    model.spec = types.SimpleNamespace(order=[types.SimpleNamespace(layer=i) for i in range(len(blocks))])
    return model


def attention(w_qkv, w_o):
    mixer = GQAAttention(64, 2, 1, 32)
    mixer.w_qkv, mixer.w_o = w_qkv, w_o
    return mixer


def feed_forward_of(gate_up, down):
    ffn = GatedMLP(64, 128)
    ffn.gate_up, ffn.down = gate_up, down
    return ffn


def test_weights_without_tiles_are_not_read_ahead():
    """Parts of a program's own may keep a weight as a tensor (``linear`` takes it), or under another name: the list ends there."""
    class Own(GatedMLP):
        def __init__(self, weight):
            self.w = weight

    o, gate_up, down, plain = tiled(64, 64), tiled(256, 64), tiled(64, 128), torch.zeros(64, 64)
    qkv = tiled(128, 64)
    for ffn, want in ((feed_forward_of(gate_up, down), [o, gate_up, down, qkv]), (feed_forward_of(gate_up, plain), [o, gate_up]),
                      (feed_forward_of(gate_up, K.LinearWeight(plain)), [o, gate_up]), (Own(plain), [o])):
        first, second = attention(qkv, o), attention(qkv, plain)
        model_of(dict(mixer=first, ffn=ffn), dict(mixer=second, ffn=feed_forward_of(gate_up, down)))._order_streams()
        assert first.ahead.tiles == [w.tiles for w in want] and second.ahead.tiles == []


def test_what_is_read_ahead_ends_at_a_part_that_does_not_name_its_weights():
    """Experts, say, stream weights of their own in front of the next layer's projection."""
    class Unnamed(FeedForward):
        pass

    o, gate_up, down, qkv = tiled(64, 64), tiled(256, 64), tiled(64, 128), tiled(128, 64)
    last = dict(mixer=attention(qkv, o), ffn=feed_forward_of(gate_up, down))
    for first, want in ((dict(mixer=attention(qkv, o), ffn=Unnamed()), [o]), (dict(mixer=attention(qkv, o)), [o, qkv]),
                        (dict(mixer=attention(qkv, o), ffn=feed_forward_of(gate_up, down)), [o, gate_up, down, qkv])):
        model_of(first, last)._order_streams()
        assert first["mixer"].ahead.tiles == [w.tiles for w in want] and last["mixer"].ahead.tiles == [o.tiles, gate_up.tiles, down.tiles]


def test_the_list_of_what_is_read_ahead_is_made_once_and_holds_its_weights():
    """An attention passes it at every launch; what it points to stays alive as long as it does."""
    ahead = K.ReadAhead([tiled(64, 100), tiled(40, 64)])
    words = ahead.words()
    assert ahead.words() is words
    assert list(words) == [2, ahead.tiles[0].data.data_ptr(), 2 * 2048, 4, ahead.tiles[1].data.data_ptr(), 2048, 3]
    first = weakref.ref(ahead.tiles[0].data)
    ahead.tiles[0].data = torch.zeros(1, dtype=torch.bfloat16)   # a weight laid out anew
    assert first() is not None and ahead.words()[1] == first().data_ptr()
    copied = copy.deepcopy(ahead)
    assert copied.words()[1] == copied.tiles[0].data.data_ptr() and copied.words()[4] == copied.tiles[1].data.data_ptr() != words[4]


def test_few_rows_are_told_by_their_number_alone():
    """What a direct step of few rows pays the rule of the many-row products for is one comparison."""
    class Weight(K.LinearWeight):
        def __init__(self):
            pass

        def __getattribute__(self, name):
            raise AssertionError(f"{name} was asked for")

    assert K._block_operands(torch.zeros(K.BLOCK_MORE_THAN_ROWS, 64, dtype=torch.bfloat16), Weight()) is False


@pytest.mark.parametrize("kind,n,k,m,wanted", [
    # us where it went before there was gemm_block / in gemm_block
    ("gated", 19456, 2560, 80, "gemm_mid"),        # 28.9 / 30.0
    ("gated", 19456, 2560, 96, "gemm_mid"),        # 29.7 / 31.6
    ("gated", 19456, 2560, 128, "gemm_block"),     # 33.7 / 33.3
    ("gated", 16384, 2560, 96, "gemm_block"),      # 29.0 / 23.9
    ("gated", 28672, 2560, 96, "gemm_block"),      # 46.8 / 37.3
    ("gated", 24576, 4096, 65, "gemm_block"),      # 45.1 / 42.7
    ("tensor", 4096, 1024, 300, "gemm_block"),     # level, and the host launches it in half the time
    ("norm", 2560, 9728, 65, "gemm_block"),        # 22.4 / 21.7
    ("norm", 5120, 25600, 65, "gemm_block"),       # 73.5 / 69.2
    ("tensor", 3072, 1024, 2048, "library"),       # 18.4 / 22.1
    ("tensor", 6144, 1024, 1024, "library"),       # 18.5 / 22.3
    ("tensor", 6144, 4096, 1024, "library"),       # 51.0 / 55.3
    ("tensor", 6144, 2560, 96, "gemm_block"),      # 17.2 / 14.9
])
def test_many_rows_go_where_they_were_measured_faster(monkeypatch, kind, n, k, m, wanted):
    """Products whose price was close, either side of the line."""
    took = []

    def stand_in(name):
        def taken(x, w, *a, slices=1, **kw):
            took.append(name)
            return torch.empty((x.shape[0], 1))
        return taken
    for name in ("gemm_block", "gemm_mid", "gemm_tall"):
        monkeypatch.setattr(K, name, stand_in(name))
    monkeypatch.setattr(K, "gemm_library", stand_in("library"))
    monkeypatch.setattr(K, "silu_mul", lambda y, activation: y)
    monkeypatch.setattr(K, "_dev", lambda *ts: None)
    w = K.LinearWeight(torch.empty((n, k), dtype=torch.bfloat16), K.TiledWeight(torch.zeros(1, dtype=torch.bfloat16), n, k))
    {"gated": K.linear_gated, "norm": K.linear_for_norm, "tensor": K.linear}[kind](torch.empty((m, k), dtype=torch.bfloat16), w)
    assert took == [wanted]


@pytest.mark.parametrize("outputs", [0, 3])
def test_a_gated_product_of_no_pairs_is_refused(monkeypatch, outputs):
    """In 32-bit as in bfloat16: gate and up come in pairs, one at least."""
    monkeypatch.setattr(K, "_dev", lambda *ts: None)
    monkeypatch.setattr(K, "_stream", lambda: None)
    with pytest.raises(K.NativeError):
        K.linear_gated(torch.zeros(2, 64), torch.zeros(outputs, 64))


def test_splits_of_latents_are_one_block_only_while_they_do_not_outnumber_the_compute_units():
    for n, context, heads, keys in [(1, 64, 16, 64), (1, 16384, 16, 64), (1, 16448, 16, 128), (8, 2048, 16, 64), (8, 2112, 16, 128),
                                    (4, 2048, 32, 64), (4, 2049, 17, 128), (256, 64, 16, 64), (257, 64, 16, 128), (8, 4096, 16, 128),
                                    (64, 4096, 16, 512), (600, 8192, 16, 1024), (1, 64 * 4096 * 9, 16, 1024)]:
        assert K.latent_split_keys(n, context, heads) == keys, (n, context, heads)
