"""Host logic of the model's steps that needs no GPU."""
import torch

from starkv_serve import model as M
from starkv_serve.kernels import model_ops


def test_decode_step_of_no_tokens():
    """A step without requests through uncompressed layers: empty logits, nothing launched."""
    shape = M.LlamaShape(hidden_size=64, num_layers=2, num_heads=4, num_kv_heads=2, head_dim=128,
                         intermediate_size=32, vocab_size=10)
    model = M.StarKVLlamaForCausalLM(shape, None, max_model_len=64, device="cpu", seed=2)
    model.allocate_kv_cache(2)
    none = torch.zeros(0, dtype=torch.int64)
    bt = torch.zeros(0, 4, dtype=torch.int32)
    assert model.decode_step(none, none, M.decode_metadata(bt, none, 16, 1)).shape == (0, 10)


def test_kernels_are_not_given_memory_of_another_device():
    """Weights, caches or slots beside the step's own device go to the calls that refuse them."""
    bf = dict(dtype=torch.bfloat16)
    x, w, ln = (torch.zeros(*s, device="meta", **bf) for s in ((2, 64), (32, 64), (64,)))
    assert model_ops.few_fits(x, w, ln)
    assert not model_ops.few_fits(x, torch.zeros(32, 64, **bf), ln)
    assert not model_ops.few_fits(x, w, torch.zeros(64, **bf))
    q, k, cs = (torch.zeros(*s, device="meta", **bf) for s in ((2, 4, 128), (2, 2, 128), (9, 128)))
    kc, pos, slots = torch.zeros(3, 16, 2, 128, **bf), torch.zeros(2, device="meta").long(), torch.zeros(2).long()
    for a in ((kc, kc, slots), (kc.to("meta"), kc, slots.to("meta")), (kc.to("meta"), kc.to("meta"), slots)):
        assert not model_ops.rope_write_fits(cs, pos, q, k, k, *a)
