"""The vLLM-free STAR-KV Llama decode step (starkv_serve/model.py) on a shrunk shape:
4 layers (1 and 2 compressed from a fused checkpoint, 0 and 3 full), 4 heads x 128,
3 requests. The prompts' cache rows are written through the layers' own write paths
(the fused codes write for compressed layers, K/V scatter for full ones); then two
decode steps run, and each layer's attention output of each step is compared with the
float64 oracle over the cache as it stands after that step's write: compressed layers
with oracle/ref.py's decode (bf16 codes or the 3.2-bit rows), full layers with plain
softmax attention over the gathered K/V. Tolerance as the decode tests (max-abs 2e-2,
mean-rel 1e-3). Also the stock model (every layer full) and the uncompressed-attention
kernel alone against the oracle, with GQA, and the step captured in a HIP graph
(DecodeGraph) against the same steps run eagerly over the same span."""
import numpy as np
import pytest
import torch

from oracle import ref
from starkv_serve import checkpoint as ck
from starkv_serve import model as M
from starkv_serve.kernels.stock_decode import paged_decode_full, write_kv_full
from test_gpu_decode import assert_close

pytestmark = pytest.mark.gpu

SHAPE = M.LlamaShape(hidden_size=512, num_layers=4, num_heads=4, num_kv_heads=4, head_dim=128,
                     intermediate_size=1024, vocab_size=1000)
PROMPTS = [100, 37, 260]
STEPS = 2


def full_attention_truth(q, kc, vc, bt, seq_lens, scale):
    """float64 softmax attention of q [n, Hq, D] over the gathered caches."""
    q = q.float().cpu().numpy().astype(np.float64)
    kc, vc = kc.float().cpu().numpy(), vc.float().cpu().numpy()
    n, Hq, D = q.shape
    G = Hq // kc.shape[2]
    out = np.zeros((n, Hq, D))
    for b in range(n):
        L = int(seq_lens[b])
        l = np.arange(L)
        K = kc[bt[b, l // 16], l % 16].astype(np.float64)
        V = vc[bt[b, l // 16], l % 16].astype(np.float64)
        for h in range(Hq):
            s = K[:, h // G] @ q[b, h] * scale
            p = np.exp(s - s.max())
            out[b, h] = (p / p.sum()) @ V[:, h // G]
    return out


def decode_layer_truth(model, c, bt_host, seq):
    """float64 truth of one layer's decode output `c` (a decode_step capture entry) over
    the layer's cache as the step left it: oracle/ref.py's decode for a compressed layer
    (bf16 codes or 3.2-bit rows), softmax attention over the gathered K/V for a full one."""
    li, layer = c["layer"], model.layers[c["layer"]]
    if not layer.compressed:
        kc, vc = model.kv_caches[li]
        return full_attention_truth(c["q"], kc, vc, bt_host, seq, model.scale)
    imp = layer.impl
    q = c["q"].float().cpu().numpy()
    vq = imp.v_up_by_q.float().cpu().numpy()
    cs = imp.rotary_emb.cos_sin_cache.float().cpu().numpy()
    ranks = imp.w.k_head_ranks.tolist()
    if imp.row is None:
        cache = model.kv_caches[li].float().cpu().numpy()
        return ref.lowrank_decode(q, cache, bt_host, seq, int(seq.max()), imp.k_up.float().cpu().numpy(), ranks,
                                  imp.k_head_offsets.tolist(), imp.k_width, vq, cs, imp.scale)
    lay = ref.row_layout(imp.k_width, len(ranks), imp.w.v_rank)
    return ref.quant_decode(q, model.kv_caches[li].cpu().numpy(), bt_host, seq, int(seq.max()), lay, ranks,
                            imp.k_up.float().cpu().numpy(), vq, cs, imp.scale)


def build(cuda, tmp_path, kv_quant, stock=False):
    path = str(tmp_path / "fused_weights.pt")
    comp = {1: ([16, 32, 16, 48], 64), 2: ([32, 16, 16, 16], 96)}
    ck.write_fused_checkpoint(path, SHAPE.num_layers, SHAPE.num_kv_heads, SHAPE.head_dim, SHAPE.hidden_size, comp,
                              seed=11)
    c = ck.load_fused_checkpoint(path, SHAPE.num_layers, SHAPE.num_kv_heads, SHAPE.head_dim, dtype=torch.bfloat16,
                                 kv_quant=kv_quant)
    model = M.StarKVLlamaForCausalLM(SHAPE, c, max_model_len=512, device=cuda, seed=12, stock=stock)
    pages = [(L + STEPS + 15) // 16 for L in PROMPTS]
    g = torch.Generator().manual_seed(13)
    perm = (torch.randperm(sum(pages), generator=g) + 1).to(torch.int32)
    # Rows cover max_model_len (512) positions; columns past a request's pages hold the null block.
    bt = torch.zeros(len(PROMPTS), 512 // 16, dtype=torch.int32)
    o = 0
    for b, p in enumerate(pages):
        bt[b, :p] = perm[o:o + p]
        o += p
    model.allocate_kv_cache(sum(pages) + 1)
    bt = bt.to(cuda)
    # The prompts' rows, through each layer's write path.
    rows = torch.cat([torch.full((L,), b) for b, L in enumerate(PROMPTS)]).to(cuda)
    pos = torch.cat([torch.arange(L) for L in PROMPTS]).to(cuda)
    slots = bt[rows, pos // 16].long() * 16 + pos % 16
    for li, layer in enumerate(model.layers):
        hid = torch.randn(len(pos), SHAPE.hidden_size, generator=g).to(torch.bfloat16).to(cuda)
        if layer.compressed:
            layer.impl.write_from_hidden(hid, model.kv_caches[li], slots)
        else:
            kc, vc = model.kv_caches[li]
            kc[slots // 16, slots % 16] = torch.randn(len(pos), 4, 128, generator=g).to(torch.bfloat16).to(cuda)
            vc[slots // 16, slots % 16] = torch.randn(len(pos), 4, 128, generator=g).to(torch.bfloat16).to(cuda)
    return model, bt


@pytest.mark.parametrize("kv_quant", [False, True])
def test_model_decode_steps_against_oracle(cuda, tmp_path, kv_quant):
    print(f"\n[model] shrunk Llama, kv_quant={kv_quant}", flush=True)
    model, bt = build(cuda, tmp_path, kv_quant)
    bt_host = bt.cpu().numpy()
    tokens = torch.tensor([5, 17, 999], device=cuda)
    for step in range(STEPS):
        positions = torch.tensor(PROMPTS, device=cuda) + step
        md = M.decode_metadata(bt, positions, 16, int(positions.max()) + 1)
        cap = []
        logits = model.decode_step(tokens, positions, md, capture=cap)
        torch.cuda.synchronize()
        assert torch.isfinite(logits).all()
        seq = (positions + 1).cpu().numpy()
        assert [c["layer"] for c in cap] == [0, 1, 2, 3]
        for c in cap:
            assert_close(c["out"], decode_layer_truth(model, c, bt_host, seq), f"step {step} layer {c['layer']}")
        tokens = logits.argmax(-1)


def test_stock_model_and_gqa_kernel(cuda, tmp_path):
    model, bt = build(cuda, tmp_path, False, stock=True)
    assert not any(layer.compressed for layer in model.layers)
    positions = torch.tensor(PROMPTS, device=cuda)
    md = M.decode_metadata(bt, positions, 16, int(positions.max()) + 1)
    cap = []
    logits = model.decode_step(torch.tensor([1, 2, 3], device=cuda), positions, md, capture=cap)
    assert torch.isfinite(logits).all()
    seq = (positions + 1).cpu().numpy()
    for c in cap:
        kc, vc = model.kv_caches[c["layer"]]
        assert_close(c["out"], full_attention_truth(c["q"], kc, vc, bt.cpu().numpy(), seq, model.scale),
                     f"stock layer {c['layer']}")
    # the kernel alone: GQA groups of 2 and 4, many splits (one long request), block size 32
    g = torch.Generator().manual_seed(21)
    for Hq, Hkv, lens, bs in ((8, 4, [3000, 5], 16), (16, 4, [700], 32), (4, 4, [1, 16, 17], 16)):
        pages = [(L + bs - 1) // bs for L in lens]
        nb = sum(pages) + 1
        kc = torch.randn(nb, bs, Hkv, 128, generator=g).to(torch.bfloat16)
        vc = torch.randn(nb, bs, Hkv, 128, generator=g).to(torch.bfloat16)
        btk = torch.zeros(len(lens), max(pages), dtype=torch.int32)
        perm = torch.randperm(nb - 1, generator=g) + 1
        o = 0
        for b, p in enumerate(pages):
            btk[b, :p] = perm[o:o + p]
            o += p
        q = torch.randn(len(lens), Hq, 128, generator=g).to(torch.bfloat16)
        out = paged_decode_full(q.to(cuda), kc.to(cuda), vc.to(cuda), btk.to(cuda),
                                torch.tensor(lens, dtype=torch.int32, device=cuda), max(lens), 128 ** -0.5)
        # the truth gathers with block_size bs: fold the block into 16-token pages
        truth = np.zeros((len(lens), Hq, 128))
        qn, kn, vn = q.double().numpy(), kc.double().numpy(), vc.double().numpy()
        for b, L in enumerate(lens):
            l = np.arange(L)
            K = kn[btk[b, l // bs].numpy(), l % bs]
            V = vn[btk[b, l // bs].numpy(), l % bs]
            for h in range(Hq):
                s = K[:, h // (Hq // Hkv)] @ qn[b, h] * 128 ** -0.5
                p = np.exp(s - s.max())
                truth[b, h] = (p / p.sum()) @ V[:, h // (Hq // Hkv)]
        assert_close(out, truth, f"stock kernel Hq={Hq} Hkv={Hkv} lens={lens} bs={bs}")


@pytest.mark.parametrize("mode", ["bf16", "quant", "stock"])
def test_decode_graph_replays_match_eager(cuda, tmp_path, mode):
    """Three greedy steps replayed from one captured step equal three eager steps over the
    graph's span bit for bit (logits and tokens), with eager work and synchronizations
    between the replays; then a reset and a replay repeat the first step."""
    print(f"\n[model graph] {mode}", flush=True)
    model, bt = build(cuda, tmp_path, mode == "quant", stock=mode == "stock")
    tokens = torch.tensor([5, 17, 999], device=cuda)
    positions = torch.tensor(PROMPTS, device=cuda)
    dg = M.DecodeGraph(model, bt, tokens, positions)
    want, tok, pos = [], tokens.clone(), positions.clone()
    for _ in range(3):
        md = M.decode_metadata(bt, pos, 16, model.max_model_len)
        logits = model.decode_step(tok, pos, md, in_graph=True)
        tok = logits.argmax(-1)
        pos = pos + 1
        want.append((logits.clone(), tok.clone()))
    torch.cuda.synchronize()
    dg.reset(tokens, positions)
    for step, (lw, tw) in enumerate(want):
        dg.replay()
        torch.cuda.synchronize()
        assert torch.equal(dg.logits, lw), f"step {step}"
        assert torch.equal(dg.tokens, tw), f"step {step}"
        assert torch.equal(dg.positions, positions + step + 1)
        torch.randn(1000, device=cuda).sum().item()  # eager work between replays
    dg.reset(tokens, positions)
    dg.replay()
    torch.cuda.synchronize()
    assert torch.equal(dg.logits, want[0][0])


@pytest.mark.parametrize("slot_dtype", [torch.int32, torch.int64])
def test_stock_write_matches_index_put(cuda, slot_dtype):
    """write_kv_full against torch's index_put on the same caches: bit-exact, slot -1
    writes nothing, strided key/value rows (views of one QKV output), block size 32."""
    print(f"\n[stock write] slots {slot_dtype}", flush=True)
    g = torch.Generator().manual_seed(31)
    nb, bs, Hkv, n = 9, 32, 4, 12
    qkv = torch.randn(n, (8 + 2 * Hkv) * 128, generator=g).to(torch.bfloat16).to(cuda)
    k = qkv[:, 8 * 128:(8 + Hkv) * 128].view(n, Hkv, 128)
    v = qkv[:, (8 + Hkv) * 128:].view(n, Hkv, 128)
    slots = torch.randperm(nb * bs, generator=g)[:n].to(slot_dtype)
    slots[3] = -1
    slots = slots.to(cuda)
    kc = torch.randn(nb, bs, Hkv, 128, generator=g).to(torch.bfloat16).to(cuda)
    vc = torch.randn(nb, bs, Hkv, 128, generator=g).to(torch.bfloat16).to(cuda)
    want_k, want_v = kc.clone(), vc.clone()
    ok = slots >= 0
    s = slots[ok].long()
    want_k[s // bs, s % bs] = k[ok]
    want_v[s // bs, s % bs] = v[ok]
    write_kv_full(k, v, kc, vc, slots)
    torch.cuda.synchronize()
    assert torch.equal(kc, want_k) and torch.equal(vc, want_v)


@pytest.mark.parametrize("lens", [[3100, 1, 16, 2049, 0, 700, 3099, 17, 5], [3072 + 64 * i for i in range(17)]])
def test_stock_decode_splits_of_larger_batches(cuda, lens):
    """More (request, head) pairs than CUs with long spans: 5 splits (9 requests) and 3 (17), some of
    them past a request's end, an empty request (NaN). Against float64 in torch, and by the decode
    tolerance."""
    g = torch.Generator().manual_seed(len(lens))
    H, bs, n = 32, 16, len(lens)
    pages = [(L + bs - 1) // bs for L in lens]
    nb = sum(pages) + 1
    kc, vc = (torch.randn(nb, bs, H, 128, generator=g).to(torch.bfloat16).to(cuda) for _ in range(2))
    bt, o = torch.zeros(n, max(pages), dtype=torch.int32), 1
    for b, p in enumerate(pages):
        bt[b, :p] = torch.arange(o, o + p)
        o += p
    q = torch.randn(n, H, 128, generator=g).to(torch.bfloat16).to(cuda)
    out = paged_decode_full(q, kc, vc, bt.to(cuda), torch.tensor(lens, dtype=torch.int32, device=cuda), max(lens),
                            128 ** -0.5)
    live = [b for b in range(n) if lens[b]]
    truth = torch.empty(len(live), H, 128, dtype=torch.float64, device=cuda)
    for i, b in enumerate(live):
        K, V = (t[bt[b, :pages[b]].long().to(cuda)].reshape(-1, H, 128)[:lens[b]].double() for t in (kc, vc))
        for h in range(H):
            truth[i, h] = torch.softmax(K[:, h] @ q[b, h].double() * 128 ** -0.5, 0) @ V[:, h]
    assert_close(out[live], truth.cpu().numpy(), f"stock splits n={n}")
    assert all(bool(out[b].isnan().all()) for b in range(n) if not lens[b])


@pytest.mark.parametrize("Hkv", [4, 2])
@pytest.mark.parametrize("shape", ["rising", "falling", "jumps", "flat"])
def test_gqa_decode_moves_its_reference_max(cuda, Hkv, shape):
    """Two query heads a row, with scores that pass the reference max by more than 2^8 slowly, never,
    or from page to page (the last page partly filled). Against float64: bf16 output (half an ulp is at
    most 2^-8 of the value); a float32 score of up to 100 over 128 terms is off by at most 100 * 8 * 2^-24
    = 5e-5, and so are the weights, times |V| < 5."""
    g = torch.Generator().manual_seed(Hkv)
    Hq, bs, lens = 8, 16, [1003, 70, 16]
    pages = [(L + bs - 1) // bs for L in lens]
    nb = sum(pages) + 1
    kc, vc = (torch.randn(nb, bs, Hkv, 128, generator=g).to(torch.bfloat16) for _ in range(2))
    vc.clamp_(-4.5, 4.5)
    q = torch.randn(len(lens), Hq, 128, generator=g).to(torch.bfloat16)
    q[..., 0] = 8
    bt, o = torch.zeros(len(lens), max(pages), dtype=torch.int32), 1
    for b, p in enumerate(pages):
        bt[b, :p] = torch.arange(o, o + p)
        ramp = {"rising": torch.linspace(0, 60, p * bs), "falling": torch.linspace(60, 0, p * bs),
                "jumps": (60 * torch.rand(p, generator=g)).repeat_interleave(bs), "flat": torch.zeros(p * bs)}[shape]
        kc[o:o + p, :, :, 0] = ramp.view(p, bs, 1).to(torch.bfloat16)
        o += p
    out = paged_decode_full(q.to(cuda), kc.to(cuda), vc.to(cuda), bt.to(cuda),
                            torch.tensor(lens, dtype=torch.int32, device=cuda), max(lens), 128 ** -0.5).double().cpu()
    for b, L in enumerate(lens):
        K, V = (t[bt[b, :pages[b]].long()].reshape(-1, Hkv, 128)[:L].double() for t in (kc, vc))
        for h in range(Hq):
            kv = h // (Hq // Hkv)
            want = torch.softmax(K[:, kv] @ q[b, h].double() * 128 ** -0.5, 0) @ V[:, kv]
            err = (out[b, h] - want).abs() - want.abs() * 2 ** -8
            assert err.max() < 2.5e-4, (shape, b, h, float(err.max()))


@pytest.mark.parametrize("Hq,Hkv,lens", [(32, 8, [8100 - 330 * i for i in range(24)]), (32, 8, [2900] * 5 + [0, 17]),
                                         (8, 1, [333, 1, 0]), (12, 3, [129] * 9), (32, 8, [700] * 33), (16, 2, [4097] * 33)])
def test_gqa_decode_units_and_splits(cuda, Hq, Hkv, lens):
    """Two or four workgroups of a (request, split, KV head), also where those are no multiple of 8:
    1, 3, 5 and many splits, some past a request's end, empty requests (NaN). Against float64 in torch,
    by the decode tolerance."""
    g = torch.Generator().manual_seed(len(lens))
    bs, n = 16, len(lens)
    pages = [(L + bs - 1) // bs for L in lens]
    nb = sum(pages) + 1
    kc, vc = (torch.randn(nb, bs, Hkv, 128, generator=g).to(torch.bfloat16).to(cuda) for _ in range(2))
    bt, o = torch.zeros(n, max(pages), dtype=torch.int32), 1
    for b, p in enumerate(pages):
        bt[b, :p] = torch.arange(o, o + p)
        o += p
    q = torch.randn(n, Hq, 128, generator=g).to(torch.bfloat16).to(cuda)
    out = paged_decode_full(q, kc, vc, bt.to(cuda), torch.tensor(lens, dtype=torch.int32, device=cuda), max(lens),
                            128 ** -0.5)
    live = [b for b in range(n) if lens[b]]
    truth = torch.empty(len(live), Hq, 128, dtype=torch.float64, device=cuda)
    for i, b in enumerate(live):
        K, V = (t[bt[b, :pages[b]].long().to(cuda)].reshape(-1, Hkv, 128)[:lens[b]].double() for t in (kc, vc))
        for h in range(Hq):
            kv = h // (Hq // Hkv)
            truth[i, h] = torch.softmax(K[:, kv] @ q[b, h].double() * 128 ** -0.5, 0) @ V[:, kv]
    assert_close(out[live], truth.cpu().numpy(), f"GQA units Hq={Hq} Hkv={Hkv} n={n}")
    assert all(bool(out[b].isnan().all()) for b in range(n) if not lens[b])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_logits_are_differentiable(cuda, dtype):
    """decode_step's logits carry a gradient to the norm and the head where one is wanted (the layers run
    without): bit for bit the values and gradients of torch's norm and product of the same rows."""
    model = M.StarKVLlamaForCausalLM(SHAPE, None, max_model_len=64, device=cuda, dtype=dtype, seed=2)
    model.allocate_kv_cache(9)
    bt = torch.arange(1, 9, device=cuda, dtype=torch.int32).view(2, 4)
    pos = torch.tensor([3, 0], device=cuda)
    tokens = torch.tensor([5, 6], device=cuda)
    x = model._layers(model.embed[tokens], pos, M.decode_metadata(bt, pos, 16, 4), None, False)
    leaves = [t.clone().requires_grad_() for t in (model.norm, model.lm_head)]
    want = torch.nn.functional.linear(torch.nn.functional.rms_norm(x, (SHAPE.hidden_size,), leaves[0],
                                                                   SHAPE.rms_norm_eps), leaves[1])
    model.norm.requires_grad_()
    model.lm_head.requires_grad_()
    logits = model.decode_step(tokens, pos, M.decode_metadata(bt, pos, 16, 4))
    assert torch.equal(logits, want)
    logits.float().square().sum().backward()
    want.float().square().sum().backward()
    for got, leaf in zip((model.norm, model.lm_head), leaves):
        assert torch.equal(got.grad, leaf.grad)


def test_decode_step_takes_weights_in_any_layout(cuda):
    """Weights as transposed views, and at starts and row strides that no wide load can take: torch's products,
    within bf16's rounding of the contiguous weights' logits."""
    shape = M.LlamaShape(hidden_size=512, num_layers=2, num_heads=4, num_kv_heads=2, head_dim=128,
                         intermediate_size=1024, vocab_size=999)
    model = M.StarKVLlamaForCausalLM(shape, None, max_model_len=64, device=cuda, seed=3)
    model.allocate_kv_cache(9)
    bt = torch.arange(1, 9, device=cuda, dtype=torch.int32).view(2, 4)
    pos = torch.tensor([0, 0], device=cuda)
    step = lambda: model.decode_step(torch.tensor([1, 2], device=cuda), pos, M.decode_metadata(bt, pos, 16, 1))  # noqa: E731
    want = step()

    def odd(t):  # the same values, 2 bytes off, rows 2 bytes longer
        return torch.cat([t.new_zeros(1), torch.nn.functional.pad(t, (0, 1)).reshape(-1)])[1:].view(
            t.shape[0], -1)[:, :t.shape[1]]

    for layout in (odd, lambda t: t.t().contiguous().t()):
        for layer in model.layers:
            layer.qkv_proj, layer.o_proj, layer.gate_up, layer.down = map(
                layout, (layer.qkv_proj, layer.o_proj, layer.gate_up, layer.down))
        model.lm_head = layout(model.lm_head)
        got = step()
        rel = (got.double() - want.double()).norm() / want.double().norm()
        # A dozen roundings of 2^-9 (rms about 2^-9 / sqrt(3)) on the way, either side.
        assert rel < 2 * 12 * 2.0 ** -9, float(rel)


def test_decode_step_of_no_tokens(cuda):
    """A step without requests: empty logits, through uncompressed layers."""
    model = M.StarKVLlamaForCausalLM(SHAPE, None, max_model_len=64, device=cuda, seed=2)
    model.allocate_kv_cache(2)
    none = torch.zeros(0, dtype=torch.int64, device=cuda)
    bt = torch.zeros(0, 4, dtype=torch.int32, device=cuda)
    assert model.decode_step(none, none, M.decode_metadata(bt, none, 16, 1)).shape == (0, SHAPE.vocab_size)


def test_decode_step_takes_other_slot_types(cuda):
    """Slots of an integer type the write has no form for are converted, as write_kv_full does."""
    model = M.StarKVLlamaForCausalLM(SHAPE, None, max_model_len=64, device=cuda, seed=2)
    model.allocate_kv_cache(9)
    bt = torch.arange(1, 9, device=cuda, dtype=torch.int32).view(2, 4)
    pos, tokens = torch.tensor([0, 0], device=cuda), torch.tensor([1, 2], device=cuda)
    md = M.decode_metadata(bt, pos, 16, 1)
    want = model.decode_step(tokens, pos, md)
    md.slot_mapping = md.slot_mapping.to(torch.int16)
    assert torch.equal(model.decode_step(tokens, pos, md), want)


def test_steps_refuse_caches_the_write_refuses(cuda):
    """Caches on the host, of another type, with different strides, of a block size the decode has no form for:
    write_kv_full's errors, nothing launched on them; a weight on the host: torch's."""
    model = M.StarKVLlamaForCausalLM(SHAPE, None, max_model_len=64, device=cuda, seed=2)
    bt = torch.arange(1, 9, device=cuda, dtype=torch.int32).view(2, 4)
    pos, tokens = torch.tensor([0, 0], device=cuda), torch.tensor([1, 2], device=cuda)
    md = M.decode_metadata(bt, pos, 16, 1)
    pmd, ppos = M.prefill_metadata(bt, [1, 1], 16)
    good = torch.zeros(9, 16, 4, 128, dtype=torch.bfloat16, device=cuda)
    wide = torch.zeros(9, 16, 8, 128, dtype=torch.bfloat16, device=cuda)[:, :, :4]
    for kc, vc in ((good.cpu(), good.cpu()), (good, good.cpu()), (good.float(), good.float()), (good, wide),
                   (good[:, :12], good[:, :12])):
        model.kv_caches = [(kc, vc)] * SHAPE.num_layers
        for step in (lambda: model.decode_step(tokens, pos, md), lambda: model.prefill_step(tokens, ppos, pmd)):
            with pytest.raises((RuntimeError, AssertionError)):
                step()
    model.kv_caches = [(good, good.clone()) for _ in range(SHAPE.num_layers)]
    want = model.decode_step(tokens, pos, md)
    model.lm_head = model.lm_head.cpu()
    with pytest.raises(RuntimeError):
        model.decode_step(tokens, pos, md)
    model.lm_head = model.lm_head.to(cuda)
    assert torch.equal(model.decode_step(tokens, pos, md), want)


@pytest.mark.parametrize("H,span,lens", [
    (32, 16384, [500, 0, 5000, 5461, 5462, 10922, 10923, 16384, 1, 16, 17]),  # 5 splits of 205 pages, at their edges
    (32, 8200, [0, 2736, 2737, 5472, 5473, 8200, 700, 33] * 2),               # 3 of 171, a whole round
    (5, 3100, [3100, 0, 5] * 23 + [620, 621, 3099]),                          # more than 64 requests
    (8, 4096, [30] * 130 + [4096, 1400])])
def test_stock_decode_splits_by_own_length(cuda, H, span, lens):
    """More (request, head) pairs than CUs over a span longer than most requests: each has the splits that its pages
    fill, some one, some none (NaN). Against float64 in torch, by the decode tolerance."""
    g = torch.Generator().manual_seed(H)
    bs, n = 16, len(lens)
    pages = [(L + bs - 1) // bs for L in lens]
    kc, vc = (torch.randn(sum(pages) + 1, bs, H, 128, generator=g).to(torch.bfloat16).to(cuda) for _ in range(2))
    bt, o = torch.zeros(n, (span + 15) // 16, dtype=torch.int32), 1
    for b, p in enumerate(pages):
        bt[b, :p] = torch.arange(o, o + p)
        o += p
    q = torch.randn(n, H, 128, generator=g).to(torch.bfloat16).to(cuda)
    out = paged_decode_full(q, kc, vc, bt.to(cuda), torch.tensor(lens, dtype=torch.int32, device=cuda), span, 128 ** -0.5)
    live = [b for b in range(n) if lens[b]]
    truth = torch.empty(len(live), H, 128, dtype=torch.float64, device=cuda)
    for i, b in enumerate(live):
        K, V = (t[bt[b, :pages[b]].long().to(cuda)].reshape(-1, H, 128)[:lens[b]].double() for t in (kc, vc))
        p = torch.softmax(torch.einsum("hd,lhd->hl", q[b].double(), K) * 128 ** -0.5, -1)
        truth[i] = torch.einsum("hl,lhd->hd", p, V)
    assert_close(out[live], truth.cpu().numpy(), f"own splits H={H} n={n}")
    assert all(bool(out[b].isnan().all()) for b in range(n) if not lens[b])


def test_a_rotation_of_the_callers_is_used(cuda):
    """A model whose rotary is replaced rotates with that one's apply in every layer, also where the kernel could."""
    class Half(M.Rotary):
        def apply(self, positions, x):
            return super().apply(positions, x) * 0.5

    model = M.StarKVLlamaForCausalLM(SHAPE, None, max_model_len=64, device=cuda, seed=2)
    bt = torch.arange(1, 9, device=cuda, dtype=torch.int32).view(2, 4)
    pos, tokens = torch.tensor([3, 5], device=cuda), torch.tensor([1, 2], device=cuda)
    model.rotary = Half(65, torch.bfloat16, cuda, 10000.0)
    model.allocate_kv_cache(9)
    cap = []
    model.decode_step(tokens, pos, M.decode_metadata(bt, pos, 16, 6), capture=cap)
    kc = model.kv_caches[0][0]
    assert torch.equal(kc[bt[:, 0].long(), pos], cap[0]["k"])
    h = cap[0]["h"].float() @ model.layers[0].qkv_proj.float().T
    k = M.Rotary.apply(model.rotary, pos, h[:, 512:1024].view(2, 4, 128)) * 0.5
    torch.testing.assert_close(cap[0]["k"].float(), k, rtol=0, atol=3 * 2.0 ** -8 * float(k.abs().max()))  # three roundings


def test_decode_graph_takes_a_head_of_any_width(cuda):
    """A head with more rows than the vocabulary, an odd number of them: the graph's tokens are the logits'
    argmax, replay by replay."""
    model = M.StarKVLlamaForCausalLM(SHAPE, None, max_model_len=64, device=cuda, seed=2)
    model.allocate_kv_cache(9)
    model.lm_head, model.embed = (torch.cat([t, t[:1] * 2]) for t in (model.lm_head, model.embed))
    bt = torch.arange(1, 9, device=cuda, dtype=torch.int32).view(2, 4)
    graph = M.DecodeGraph(model, bt, torch.tensor([1, 2], device=cuda), torch.tensor([3, 5], device=cuda))
    for step in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert graph.logits.shape == (2, 1001) and torch.equal(graph.tokens, graph.logits.argmax(-1))
        assert graph.positions.tolist() == [4 + step, 6 + step]
