"""Host logic of the model's steps that needs no GPU."""
import ctypes
import os
import subprocess

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx

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


def test_index_rules_are_those_of_torch(tmp_path):
    """The positions a decode step's kernels take (csrc/index_rules.hpp, built for the host): those torch's index
    takes, at the same places; at every other the kernels end the launch."""
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(M.__file__))), "csrc")
    src, so = tmp_path / "rules.cpp", tmp_path / "rules.so"
    src.write_text('#include "index_rules.hpp"\n'
                   'extern "C" int wrap(int64_t* i, int64_t n) { return starkv::wrap_index(*i, n); }\n'
                   'extern "C" int split(int64_t p, int64_t bs, int64_t w, int64_t* b, int64_t* in) '
                   '{ return starkv::split_position(p, bs, w, *b, *in); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{csrc}", str(src), "-o", str(so)], check=True)
    L, i64 = ctypes.CDLL(str(so)), ctypes.c_int64
    table, row, bs = torch.arange(50), torch.arange(7), 16
    for p in list(range(-130, 130)) + [2 ** 40, -2 ** 40, 2 ** 63 - 1, -2 ** 63]:
        for rule in ("table", "row"):
            pos, a, b = torch.tensor([p]), i64(p), i64()
            if rule == "table":
                ok = L.wrap(ctypes.byref(a), i64(50))
            else:
                ok = L.split(i64(p), i64(bs), i64(7), ctypes.byref(a), ctypes.byref(b))
            try:
                want = table[pos] if rule == "table" else row[pos // bs]
            except IndexError:
                assert not ok, (rule, p)
                continue
            assert ok and a.value == want.item(), (rule, p)
            if rule == "row":
                assert b.value == (pos % bs).item(), p
    kernels = open(os.path.join(csrc, "model_ops.hip")).read()
    assert kernels.count("__builtin_trap()") == 2 and "wrap_index(pos, p.cs_rows)" in kernels
    assert "split_position(p, block_size, width, blk, in)" in kernels


@pytest.mark.parametrize("how", ["compile", "jit", "make_fx"])
def test_rotary_and_slots_compile_and_trace(how):
    """One graph, of torch's operations, with the plain calls' values."""
    rot = M.Rotary(50, torch.float32, "cpu", 10000.0)
    pos, x = torch.tensor([0, 49, 7]), torch.randn(3, 4, 128)
    bt = torch.arange(12, dtype=torch.int32).view(3, 4)

    def slots(bt, pos):
        md = M.decode_metadata(bt, pos, 16, 64)
        return md.slot_mapping, md.seq_lens

    for f, args in ((lambda p, t: rot.apply(p, t), (pos, x)), (slots, (bt, pos))):
        g = {"compile": lambda: torch.compile(f, fullgraph=True, backend="eager"),
             "jit": lambda: torch.jit.trace(f, args, check_trace=False), "make_fx": lambda: make_fx(f)(*args)}[how]()
        got, want = g(*args), f(*args)
        assert all(torch.equal(a, b) for a, b in zip(*((t if isinstance(t, tuple) else (t,)) for t in (got, want))))
