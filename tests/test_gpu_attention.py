"""Every attention kernel on its own, through the C ABI (rtvla_attention), against fp32 scaled-dot-product attention with the
mask written out explicitly (the reference's predicate: /root/reference/pi0_infer.py:1089-1096, pi05_infer.py:294-299;
causal grouped-query: dm0_infer.py:913-918).  Shapes sit on the kernels' edges: one key block, keys = 1 mod 32, the state-row
mask, a valid prefix shorter than the allocated one, causal grouped-query heads, more than four key blocks per key split."""
import ctypes

import pytest
import torch

import rtvla_capi as capi

pytestmark = pytest.mark.gpu
_P = ctypes.c_void_p
KINDS = {  # kind: (head_dim, group)
    capi.ATTN_GEMMA_PREFIX: (256, 8), capi.ATTN_GEMMA_SUFFIX: (256, 8), capi.ATTN_GQA128_PREFIX: (128, 2), capi.ATTN_GQA128_SUFFIX: (128, 2),
    capi.ATTN_VIT64: (64, 1), capi.ATTN_SIGLIP: (72, 1), capi.ATTN_VIT64_EXP2: (64, 1)}
REL_TOL = 1e-2      # relative L2 of the bf16 output against the fp32 result (probabilities and outputs are rounded to bf16 once each)
ABS_TOL = 3e-2      # largest element error, outputs are O(1)
LN2 = 0.6931471805599453


def reference(kind, q, k, v, scale, prefix_alloc, valid_len, state_tokens):
    """fp32, mask as a dense boolean [tokens][keys]; q [T][B][G][D], k / v [K][B][D]."""
    T, B, G, D = q.shape
    K = k.shape[0]
    t = torch.arange(T, device=q.device)[:, None]
    j = torch.arange(K, device=q.device)[None, :]
    vis = torch.where(j < prefix_alloc, j < valid_len, (t >= state_tokens) | (j == prefix_alloc))
    if kind == capi.ATTN_GQA128_PREFIX:
        vis = vis & (j <= t)
    if kind == capi.ATTN_SIGLIP:
        vis = (t // 256) == (j // 256)
    logits = torch.einsum("tbgd,kbd->bgtk", q.float(), k.float()) * scale
    logits = logits.masked_fill(~vis[None, None], float("-inf"))
    return torch.einsum("bgtk,kbd->tbgd", torch.softmax(logits, -1), v.float())


def run(kind, tokens, keys, kv_heads, prefix_alloc=None, valid_len=None, state_tokens=0, seed=0, sharp=1.0, ramp=0.0):
    lib = capi.load()
    D, G = KINDS[kind]
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    q = (torch.randn(tokens, kv_heads, G, D, device="cuda:0", generator=g) * sharp).bfloat16()
    k = torch.randn(keys, kv_heads, D, device="cuda:0", generator=g).bfloat16()
    v = torch.randn(keys, kv_heads, D, device="cuda:0", generator=g).bfloat16()
    if ramp:            # logits that climb with the key index: the running maximum grows all the way through the key loop
        q = q.float(); q[..., 0] += 4.0; q = q.bfloat16()
        k = k.float(); k[..., 0] += ramp * torch.arange(keys, device="cuda:0")[:, None] / keys; k = k.bfloat16()
    scale = D ** -0.5
    if kind == capi.ATTN_VIT64_EXP2:
        q, scale = (q.float() * (scale / LN2)).bfloat16(), LN2
    out = torch.full_like(q, 9.0)
    prefix_alloc = keys if prefix_alloc is None else prefix_alloc
    vl = None if valid_len is None else torch.tensor([valid_len], dtype=torch.int32, device="cuda:0")
    need = lib.rtvla_attention_workspace_bytes(kind, tokens, keys, kv_heads)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    rc = lib.rtvla_attention(kind, _P(q.data_ptr()), _P(k.data_ptr()), _P(v.data_ptr()), _P(out.data_ptr()), tokens, keys, kv_heads,
                             ctypes.c_float(scale), prefix_alloc, _P(vl.data_ptr()) if vl is not None else None, state_tokens,
                             _P(ws.data_ptr()), need, _P(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, rc
    torch.cuda.synchronize()
    ref = reference(kind, q, k, v, scale, prefix_alloc, prefix_alloc if valid_len is None else valid_len, state_tokens)
    err = (out.float() - ref)
    rel = (err.norm() / ref.norm()).item()
    assert torch.isfinite(out.float()).all()
    assert rel <= REL_TOL and err.abs().max().item() <= ABS_TOL, (rel, err.abs().max().item())
    return rel


@pytest.mark.parametrize("tokens", [1, 17, 32, 33, 257, 788, 968])
def test_gemma_prefix_pass(tokens):
    run(capi.ATTN_GEMMA_PREFIX, tokens, tokens, 1, seed=tokens)


@pytest.mark.parametrize("tokens", [681, 682, 683, 767, 768, 769, 1023, 1024, 1025, 1224, 1536, 1537])
def test_gemma_prefix_pass_around_the_row_tiles_of_a_workgroup(tokens):
    """Half a 16-row tile per token, two tiles to a workgroup: even and odd numbers of tiles at which the workgroups are two, three and four rounds of the CUs' places for
    one tile."""
    run(capi.ATTN_GEMMA_PREFIX, tokens, tokens, 1, seed=tokens)


@pytest.mark.parametrize("tokens", [848, 849, 864, 1201])
def test_causal_prefix_pass_around_the_row_tiles_of_a_workgroup(tokens):
    """Eight heads of an eighth of a 16-row tile per token, two tiles to a workgroup: 106 tiles a head, 107 (the last workgroup has one), 108, 151."""
    run(capi.ATTN_GQA128_PREFIX, tokens, tokens, 8, seed=tokens)


@pytest.mark.parametrize("tokens", [184, 185, 192, 193, 208, 223, 224, 225, 255, 256, 257, 383, 384, 385, 607])
def test_causal_prefix_pass_in_blocks_of_32_rows(tokens):
    """32 rows are 16 tokens: sequences that end in the first or the second half of a block of 32 keys and of rows, one trip to several of each wave, waves that
    see nothing of their block in some rows."""
    run(capi.ATTN_GQA128_PREFIX, tokens, tokens, 8, seed=tokens)
    run(capi.ATTN_GQA128_PREFIX, tokens, tokens, 8, seed=tokens + 1, sharp=6.0)
    run(capi.ATTN_GQA128_PREFIX, tokens, tokens, 8, seed=tokens + 2, ramp=-60.0)


@pytest.mark.parametrize("kind,tokens,heads", [(capi.ATTN_GEMMA_PREFIX, 528, 1), (capi.ATTN_GEMMA_PREFIX, 788, 1), (capi.ATTN_GEMMA_PREFIX, 1024, 1), (capi.ATTN_GQA128_PREFIX, 607, 8)])
def test_prefix_pass_rounds_each_probability_once(kind, tokens, heads):
    """Sharp rows, where few keys hold the weight: relative to the row's largest, whose probability is then exactly 1, the probabilities add little to the rounding of the
    output to bf16 (1.02 times its error; relative to anything else 1.10 - 1.4 times)."""
    lib = capi.load()
    D, G = KINDS[kind]
    g = torch.Generator(device="cuda:0").manual_seed(tokens)
    q = (torch.randn(tokens, heads, G, D, device="cuda:0", generator=g) * 4.0).bfloat16()
    k = torch.randn(tokens, heads, D, device="cuda:0", generator=g).bfloat16()
    v = torch.randn(tokens, heads, D, device="cuda:0", generator=g).bfloat16()
    out = torch.zeros_like(q)
    need = lib.rtvla_attention_workspace_bytes(kind, tokens, tokens, heads)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    assert lib.rtvla_attention(kind, _P(q.data_ptr()), _P(k.data_ptr()), _P(v.data_ptr()), _P(out.data_ptr()), tokens, tokens, heads, ctypes.c_float(D ** -0.5), tokens,
                               None, 0, _P(ws.data_ptr()), need, _P(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    ref = reference(kind, q, k, v, D ** -0.5, tokens, tokens, 0)
    rounding = (ref.bfloat16().float() - ref).norm().item()
    assert (out.float() - ref).norm().item() <= 1.06 * rounding


# (64 and 100 tokens: the kernel for 16 rows)
@pytest.mark.parametrize("kind,tokens,heads", [(capi.ATTN_GEMMA_PREFIX, 64, 1), (capi.ATTN_GEMMA_PREFIX, 700, 1), (capi.ATTN_GQA128_PREFIX, 100, 8), (capi.ATTN_GQA128_PREFIX, 300, 8)])
@pytest.mark.parametrize("exponent,sign", [(20, 1), (35, 1), (35, -1), (40, 1), (40, -1)])
def test_prefix_pass_with_logits_of_any_size(kind, tokens, heads, exponent, sign):
    """One product to a logit, so that each is exact: +- 2^2n times 1 to 1.75, in steps of an eighth along the keys.  A row averages the keys that share its largest; those sums are of
    bf16 values with weights 1 / n, so what is left is the rounding of the output, and of a weight to bf16 (2^-9 each of the largest element)."""
    lib = capi.load()
    D, G = KINDS[kind]
    g = torch.Generator(device="cuda:0").manual_seed(tokens + exponent)
    q, k = torch.zeros(tokens, heads, G, D, device="cuda:0"), torch.zeros(tokens, heads, D, device="cuda:0")
    q[..., 3] = 2.0 ** exponent
    k[..., 3] = sign * (2.0 ** exponent * (1 + ((torch.arange(tokens, device="cuda:0") * 5) % 7) / 8))[:, None]
    q, k, v = q.bfloat16(), k.bfloat16(), torch.randn(tokens, heads, D, device="cuda:0", generator=g).bfloat16()
    out = torch.full_like(q, 9.0)
    need = lib.rtvla_attention_workspace_bytes(kind, tokens, tokens, heads)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    assert lib.rtvla_attention(kind, _P(q.data_ptr()), _P(k.data_ptr()), _P(v.data_ptr()), _P(out.data_ptr()), tokens, tokens, heads, ctypes.c_float(D ** -0.5), tokens,
                               None, 0, _P(ws.data_ptr()), need, _P(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    ref = reference(kind, q, k, v, D ** -0.5, tokens, tokens, 0)
    assert (out.float() - ref).abs().max().item() <= 2.0 ** -8 * v.float().abs().max().item()


@pytest.mark.parametrize("kind,tokens,heads", [(capi.ATTN_GEMMA_PREFIX, 64, 1), (capi.ATTN_GEMMA_PREFIX, 700, 1), (capi.ATTN_GQA128_PREFIX, 100, 8), (capi.ATTN_GQA128_PREFIX, 300, 8)])
def test_hidden_keys_have_no_weight_at_the_smallest_scales(kind, tokens, heads):
    """A scale at which all logits are as good as equal: a row is the mean of what it sees."""
    lib, valid = capi.load(), 33
    D, G = KINDS[kind]
    g = torch.Generator(device="cuda:0").manual_seed(tokens)
    q = torch.randn(tokens, heads, G, D, device="cuda:0", generator=g).bfloat16()
    k, v = (torch.randn(tokens, heads, D, device="cuda:0", generator=g).bfloat16() for _ in range(2))
    out, vl = torch.full_like(q, 9.0), torch.tensor([valid], dtype=torch.int32, device="cuda:0")
    need = lib.rtvla_attention_workspace_bytes(kind, tokens, tokens, heads)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    assert lib.rtvla_attention(kind, _P(q.data_ptr()), _P(k.data_ptr()), _P(v.data_ptr()), _P(out.data_ptr()), tokens, tokens, heads, ctypes.c_float(1e-30), tokens,
                               _P(vl.data_ptr()), 0, _P(ws.data_ptr()), need, _P(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    seen = v.float()[:valid]
    if kind == capi.ATTN_GQA128_PREFIX:
        last = torch.arange(tokens, device="cuda:0").clamp(max=valid - 1)
        mean = seen.cumsum(0)[last] / (last + 1)[:, None, None]
    else:
        mean = seen.mean(0, keepdim=True).expand(tokens, heads, D)
    assert (out.float() - mean[:, :, None]).abs().max().item() <= 2.0 ** -8 * v.float().abs().max().item()


@pytest.mark.parametrize("tokens,heads,valid", [(300, 8, 300), (300, 8, 299), (300, 8, 33), (300, 8, 32), (300, 8, 1), (400, 6, 250), (900, 3, 511)])
def test_causal_prefix_pass_with_a_valid_length(tokens, heads, valid):
    """Keys past the valid length are hidden from every row, and the number of K/V heads need not be that of the XCDs."""
    run(capi.ATTN_GQA128_PREFIX, tokens, tokens, heads, valid_len=valid, seed=valid)


# (tokens, row tiles per workgroup): one where that was the faster.  us of a launch with one / two: 512 tokens 9.2 / 9.6, 513 13.2 / 10.3, 682 16.3 / 11.9, 1 025 31.0 / 27.7, 1 536 43.4 / 36.0;
# DM0 177 5.11 / 5.16, 184 5.13 / 5.04, 185 5.07 / 5.06, 206 5.17 / 5.08, 848 15.9 / 9.9
@pytest.mark.parametrize("model,views,sizes", [("pi0", 1, [(256, 1), (682, 2), (683, 2)]), ("pi0", 2, [(512, 1), (513, 2)]), ("pi0", 4, [(1024, 2), (1025, 2), (1536, 2), (1537, 2), (2048, 2)]),
                                               ("dm0", 1, [(177, 1), (184, 1), (185, 2), (206, 2), (848, 2), (849, 2), (2107, 2)])])
def test_long_prefix_passes_take_two_row_tiles(model, views, sizes):
    """A workgroup with one row tile reads all keys for 16 rows: past 512 (DM0: about 190) tokens that is slower than for 32, by up to 70 %."""
    import synthetic as syn
    for tokens, tiles in sizes:
        if model == "pi0":
            from pi0_infer import Pi0Inference
            prompt = tokens - 256 * views
            m = Pi0Inference(syn.pi0_checkpoint(11, prompt, "cuda:0", vision_layers=1, llm_layers=2), views, 8)
        else:
            from dm0_infer import DM0Inference
            m = DM0Inference(syn.dm0_checkpoint(11, "cuda:0", 1, 2, vocab=64), num_images=views, max_lang_len=tokens - 169 * views)
        stream, names = torch.cuda.current_stream().cuda_stream, []
        while (r := m._engine.ctx.time_launch(capi.STAGE_PREFIX_LAYER, 0, 0, len(names), 1, stream)) is not None:
            names.append(r[1])
        assert "prefix attn [%d rows]" % (16 * tiles) in names, (tokens, names)


@pytest.mark.parametrize("tokens,valid", [(820, 789), (820, 1), (300, 288), (64, 64)])
def test_gemma_prefix_pass_with_a_valid_length_below_the_allocated_prefix(tokens, valid):
    """Pi05: prompt rows past valid_encoder_len are allocated but masked as keys (their own outputs are never read)."""
    lib = capi.load()
    D, G = 256, 8
    g = torch.Generator(device="cuda:0").manual_seed(valid)
    q = torch.randn(tokens, 1, G, D, device="cuda:0", generator=g).bfloat16()
    k = torch.randn(tokens, 1, D, device="cuda:0", generator=g).bfloat16()
    v = torch.randn(tokens, 1, D, device="cuda:0", generator=g).bfloat16()
    out = torch.zeros_like(q)
    vl = torch.tensor([valid], dtype=torch.int32, device="cuda:0")
    need = lib.rtvla_attention_workspace_bytes(capi.ATTN_GEMMA_PREFIX, tokens, tokens, 1)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    assert lib.rtvla_attention(capi.ATTN_GEMMA_PREFIX, _P(q.data_ptr()), _P(k.data_ptr()), _P(v.data_ptr()), _P(out.data_ptr()), tokens, tokens, 1,
                               ctypes.c_float(D ** -0.5), tokens, _P(vl.data_ptr()), 0, _P(ws.data_ptr()), need, _P(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    ref = reference(capi.ATTN_GEMMA_PREFIX, q, k, v, D ** -0.5, tokens, valid, 0)
    err = out.float()[:valid] - ref[:valid]
    assert (err.norm() / ref[:valid].norm()).item() <= REL_TOL


# (1 024 tokens: two row tiles per workgroup)  Blocks of 32 keys over four waves: none, fewer than waves, one each, an even and an odd number of trips, ends inside and at a block
@pytest.mark.parametrize("valid", [0, 1, 31, 32, 33, 97, 128, 129, 160, 255, 256, 257, 383, 1023])
def test_prefix_pass_of_many_rows_with_any_number_of_key_blocks(valid):
    if valid:
        test_gemma_prefix_pass_with_a_valid_length_below_the_allocated_prefix(1024, valid)
        return
    lib, tokens = capi.load(), 1024
    q, k, v = (torch.randn(tokens, n, 256, device="cuda:0").bfloat16() for n in (8, 1, 1))
    out, vl = torch.full_like(q, 9.0), torch.zeros(1, dtype=torch.int32, device="cuda:0")
    need = lib.rtvla_attention_workspace_bytes(capi.ATTN_GEMMA_PREFIX, tokens, tokens, 1)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    assert lib.rtvla_attention(capi.ATTN_GEMMA_PREFIX, _P(q.data_ptr()), _P(k.data_ptr()), _P(v.data_ptr()), _P(out.data_ptr()), tokens, tokens, 1,
                               ctypes.c_float(0.0625), tokens, _P(vl.data_ptr()), 0, _P(ws.data_ptr()), need, _P(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    assert not out.any()                                    # no key is visible


@pytest.mark.parametrize("tokens,ramp,sharp", [(700, 128.0, 1.0), (700, -128.0, 1.0), (771, 0.0, 6.0), (1600, 64.0, 1.0)])
def test_prefix_pass_of_many_rows_with_growing_maxima_and_sharp_rows(tokens, ramp, sharp):
    run(capi.ATTN_GEMMA_PREFIX, tokens, tokens, 1, seed=tokens, ramp=ramp, sharp=sharp)


# sizes about the one from which workgroups take two row tiles (513), an odd number of tiles and ends inside a block of keys among them
@pytest.mark.parametrize("tokens", [512, 513, 577, 640, 641])
def test_gemma_prefix_pass_around_the_row_tiles_of_a_workgroup_at_few_tokens(tokens):
    run(capi.ATTN_GEMMA_PREFIX, tokens, tokens, 1, seed=tokens)


# every part of the mask at once, on the edges of blocks of 32 keys: a suffix behind the prefix, a hole behind the valid keys, state rows that see the suffix's first key only
@pytest.mark.parametrize("prefix,state", [(900, 0), (1000, 3)])
def test_prefix_pass_of_many_rows_with_other_masks(prefix, state):
    run(capi.ATTN_GEMMA_PREFIX, 1000, 1000, 1, prefix_alloc=prefix, state_tokens=state, seed=prefix)


@pytest.mark.parametrize("prefix,state,valid", [(900, 5, None), (0, 3, None), (0, 0, None), (999, 2, 300), (512, 1, 33), (31, 4, 31), (32, 1, 0), (960, 1000, 1), (1000, 2, 700)])
def test_prefix_pass_of_many_rows_with_a_suffix_and_state_rows(prefix, state, valid):
    run(capi.ATTN_GEMMA_PREFIX, 1000, 1000, 1, prefix_alloc=prefix, state_tokens=state, valid_len=valid, seed=prefix + state)
    run(capi.ATTN_GEMMA_PREFIX, 1000, 1000, 1, prefix_alloc=prefix, state_tokens=state, valid_len=valid, seed=prefix + state, sharp=6.0)


@pytest.mark.parametrize("prefix,state,valid", [(200, 0, None), (200, 3, 150), (33, 2, 33), (1, 1, None), (299, 4, 100), (64, 300, 1)])
def test_causal_prefix_pass_with_a_suffix_and_state_rows(prefix, state, valid):
    run(capi.ATTN_GQA128_PREFIX, 300, 300, 8, prefix_alloc=prefix, state_tokens=state, valid_len=valid, seed=prefix + state)


@pytest.mark.parametrize("tokens,prefix,valid,state", [
    (51, 788, None, 1),      # the headline shape: 839 keys, 7 key splits, state-token row sees itself only
    (51, 270, None, 1),      # 321 keys = 1 mod 32: the last key block holds one key
    (51, 13, None, 1),       # 64 keys: a single key split of two blocks
    (1, 5, None, 0),         # one query token, six keys: one key block
    (50, 820, 789, 0),       # Pi05: no state token, valid prefix shorter than the allocated one
    (50, 820, 1, 0),         # ... down to one visible prefix key
    (64, 768, None, 1),      # chunk 63
    (101, 259, None, 1),     # two 64-row blocks of suffix rows
    (128, 261, 200, 0),      # the 128-row limit
    (21, 2256, None, 1),     # 2277 keys: more than four key blocks per split, the general kernel with a key split
])
def test_gemma_suffix_pass_masks_and_key_splits(tokens, prefix, valid, state):
    run(capi.ATTN_GEMMA_SUFFIX, tokens, prefix + tokens, 1, prefix_alloc=prefix, valid_len=valid, state_tokens=state, seed=prefix)


@pytest.mark.parametrize("tokens,heads", [(1, 8), (31, 8), (32, 8), (33, 1), (170, 8), (607, 8)])
def test_causal_grouped_query_prefix_pass(tokens, heads):
    run(capi.ATTN_GQA128_PREFIX, tokens, tokens, heads, seed=tokens)


@pytest.mark.parametrize("tokens,prefix,heads", [(50, 607, 8), (50, 33, 8), (64, 200, 2), (7, 1, 8)])
def test_grouped_query_suffix_pass(tokens, prefix, heads):
    run(capi.ATTN_GQA128_SUFFIX, tokens, prefix + tokens, heads, seed=prefix)


@pytest.mark.parametrize("tokens,heads", [(1, 16), (63, 3), (64, 8), (96, 2), (128, 4), (129, 16), (192, 3), (200, 2), (257, 5), (2705, 16)])
def test_vit_flash_attention(tokens, heads):
    """One to 43 key tiles of 64: a single tile, an odd number of 32-key blocks (the half-filled last tile), three and more
    tiles (the three LDS stages wrap), the DM0 shape."""
    run(capi.ATTN_VIT64, tokens, tokens, heads, seed=tokens)


@pytest.mark.parametrize("tokens", [96, 700, 2705])
def test_vit_flash_attention_with_a_maximum_that_keeps_growing(tokens):
    """The ViT kernel rescales its accumulator only when a row maximum grew by 2^8 and moves the probabilities of the block in
    flight to the new scale: logits that climb by ~90 bits over the keys take that path about a dozen times per row."""
    run(capi.ATTN_VIT64, tokens, tokens, 3, seed=tokens + 1, ramp=128.0)


@pytest.mark.parametrize("tokens,heads,ramp,sharp", [(1, 16, 0.0, 1.0), (31, 8, 0.0, 1.0), (32, 1, 0.0, 1.0), (33, 8, 0.0, 1.0), (63, 3, 0.0, 1.0), (64, 8, 0.0, 1.0),
                                                     (65, 3, 0.0, 1.0), (96, 2, 0.0, 1.0), (128, 4, 0.0, 1.0), (129, 16, 0.0, 1.0), (192, 3, 0.0, 1.0), (200, 2, 0.0, 1.0),
                                                     (257, 5, 0.0, 1.0), (385, 24, 0.0, 1.0), (449, 8, 0.0, 1.0), (512, 16, 0.0, 1.0), (2705, 16, 0.0, 1.0), (96, 3, 128.0, 1.0), (700, 3, 128.0, 1.0), (2705, 3, 128.0, 1.0),
                                                     (700, 3, -128.0, 1.0), (500, 4, 0.0, 6.0)])
def test_vit_flash_attention_as_the_forward_runs_it(tokens, heads, ramp, sharp):
    """Queries that carry their scale, S^T started from minus the running maximum: the edges of the instance without, a sequence that ends in its first
    block, last row blocks (which are dealt behind all others where the heads are a multiple of eight) of one row, of one to four waves, maxima that keep growing, that lie
    in the first block, and sharp rows."""
    run(capi.ATTN_VIT64_EXP2, tokens, tokens, heads, seed=tokens + 2, ramp=ramp, sharp=sharp)


def test_exponents_of_two_have_their_scale_built_in():
    lib, p = capi.load(), _P(4096)
    need = lib.rtvla_attention_workspace_bytes(capi.ATTN_VIT64_EXP2, 64, 64, 1)
    assert need > 0 and lib.rtvla_attention_workspace_bytes(capi.ATTN_VIT64_EXP2, 64, 65, 1) == 0
    for scale in (0.125, float("nan")):
        assert lib.rtvla_attention(capi.ATTN_VIT64_EXP2, p, p, p, p, 64, 64, 1, ctypes.c_float(scale), 64, None, 0, p, need, None) == capi.ERR_LIMIT
    assert lib.rtvla_attention(capi.ATTN_VIT64_EXP2, p, p, p, p, 64, 64, 1, ctypes.c_float(LN2), 63, None, 0, p, need, None) == capi.ERR_LIMIT


@pytest.mark.parametrize("views", [1, 3])
def test_siglip_attention_keeps_views_apart(views):
    run(capi.ATTN_SIGLIP, 256 * views, 256 * views, 16, seed=views)


@pytest.mark.parametrize("views", [1, 2, 3, 4])
def test_siglip_attention_with_maxima_that_grow_along_the_keys(views):
    """One, two and four waves to a workgroup: sharp logits, and keys whose logits climb, so that every block of 64 rescales what the ones before it left."""
    run(capi.ATTN_SIGLIP, 256 * views, 256 * views, 16, seed=40 + views, sharp=4.0)
    run(capi.ATTN_SIGLIP, 256 * views, 256 * views, 16, seed=50 + views, ramp=25.0 * views)


def test_peaked_softmax_rows_survive_the_running_maximum():
    """Large logits (|q| scaled up): one key dominates each row, the running-maximum rescale path is exercised in every kernel."""
    run(capi.ATTN_GEMMA_PREFIX, 300, 300, 1, seed=5, sharp=6.0)
    run(capi.ATTN_GEMMA_SUFFIX, 51, 839, 1, prefix_alloc=788, state_tokens=1, seed=6, sharp=6.0)
    run(capi.ATTN_VIT64, 500, 500, 4, seed=7, sharp=6.0)
    run(capi.ATTN_GQA128_PREFIX, 300, 300, 8, seed=8, sharp=6.0)
