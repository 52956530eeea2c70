"""The order of the operator calls in layer.decode_layer_calls (reference: src/model_gpu.cu:251-293), without a GPU."""
import pytest

from orin_llm_amd import layer


class Calls:
    """Stands in for the operators; a product over more elements than were staged is refused, as the library refuses it."""

    def __init__(self):
        self.staged, self.products = 0, []

    def quantize_activation(self, x, n_in):
        assert n_in <= len(x)
        self.staged = n_in

    def _product(self, what, n_in):
        assert n_in <= self.staged, f"{what}: {n_in} elements of {self.staged} staged"
        self.products.append((what, n_in))

    def gemv_q8(self, wtype, W, y, n_in, n_out):
        self._product(W, n_in)

    def gemv_q8_bias(self, wtype, W, bias, y, n_in, n_out):
        self._product(W, n_in)

    def gemv_q8_add(self, wtype, W, y, n_in, n_out):
        self._product(W, n_in)

    def gemv_fused_gate_up_swiglu(self, wtype, Wg, Wu, out, n_in, n_out):
        self._product(Wg, n_in)

    def __getattr__(self, name):
        return lambda *args: None


@pytest.mark.parametrize("n_head, head_dim, n_embd", [(16, 128, 1024), (12, 128, 1536), (8, 64, 768)])
def test_every_product_finds_its_whole_activation_staged(n_head, head_dim, n_embd):
    """Heads wider than the model, as wide, and narrower."""
    n_kv, n_ff, nq = 4, 3072, n_head * head_dim
    hp = dict(n_embd=n_embd, n_head=n_head, n_kv=n_kv, head_dim=head_dim, n_ff=n_ff, n_rot=head_dim, neox=1, rms_eps=1e-6, rope_theta=1e6)
    L = {k: (layer.Q4_K, k) for k in ("wq", "wk", "wv", "wo", "ffn_gate", "ffn_up", "ffn_down")}
    L.update(attn_norm=None, ffn_norm=None)
    sizes = dict(x=n_embd, xn=n_embd, xn2=n_embd, q=nq, k=n_kv * head_dim, v=n_kv * head_dim, attn=max(nq, n_embd), act=n_ff)
    ops = Calls()
    layer.decode_layer_calls(hp, L, {k: range(n) for k, n in sizes.items()}, None, None, None, 512, ops=ops)
    assert ops.products == [("wq", n_embd), ("wk", n_embd), ("wv", n_embd), ("wo", nq), ("ffn_gate", n_embd), ("ffn_down", n_ff)]
