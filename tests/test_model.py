"""Host logic of the model's steps that needs no GPU."""
import torch

from starkv_serve import model as M


def test_decode_step_of_no_tokens():
    """A step without requests through uncompressed layers: empty logits, nothing launched."""
    shape = M.LlamaShape(hidden_size=64, num_layers=2, num_heads=4, num_kv_heads=2, head_dim=128,
                         intermediate_size=32, vocab_size=10)
    model = M.StarKVLlamaForCausalLM(shape, None, max_model_len=64, device="cpu", seed=2)
    model.allocate_kv_cache(2)
    none = torch.zeros(0, dtype=torch.int64)
    bt = torch.zeros(0, 4, dtype=torch.int32)
    assert model.decode_step(none, none, M.decode_metadata(bt, none, 16, 1)).shape == (0, 10)
