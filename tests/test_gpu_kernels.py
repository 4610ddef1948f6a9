"""Per-kernel GPU parity through the C ABI: the large-M MFMA GEMM (every block tile, with and without split-K) and the
action-expert weight-streaming kernel on the shapes the models produce and on ragged ones, against torch.matmul in
fp32 on the same bf16 operands.  Tolerance: the result is one bf16 rounding of an fp32 sum whose order differs from
the checker's, so single-ulp flips are expected and nothing more: relative L2 <= 3e-3, and every element within
one bf16 spacing (2^-7 relative) plus 1e-3 of the output's RMS for the elements that cancel to nearly zero."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
_P = ctypes.c_void_p
REL_TOL = 3e-3


def _run(lib, capi, M, K, N, tile, nsplit, bias=True, seed=0):
    g = torch.Generator(device="cuda:0").manual_seed(seed * 7919 + M + K + N)
    x = torch.randn(M, K, device="cuda:0", generator=g).to(torch.bfloat16)
    w = (torch.randn(K, N, device="cuda:0", generator=g) * 0.05).to(torch.bfloat16)
    b = torch.randn(N, device="cuda:0", generator=g).to(torch.bfloat16) if bias else None
    need = lib.rtvla_linear_workspace_bytes(M, K, N, tile, nsplit)
    if need == 0:
        return None
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    out = torch.full((M, N), 77.0, dtype=torch.bfloat16, device="cuda:0")
    rc = lib.rtvla_linear(_P(x.data_ptr()), M, K, _P(w.data_ptr()), N, _P(b.data_ptr()) if bias else None, _P(out.data_ptr()),
                          _P(ws.data_ptr()), need, tile, nsplit, _P(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    if rc == capi.ERR_LIMIT:
        return None
    assert rc == 0, rc
    ref = x.float() @ w.float()
    if bias:
        ref = ref + b.float()
    got = out.float()
    rel = ((got - ref).norm() / ref.norm()).item()
    excess = (got - ref).abs() / (ref.abs() * 2.0 ** -7 + 1e-3 * ref.pow(2).mean().sqrt())
    return rel, excess.max().item()


def _tiles(lib):
    out, r, c = [], ctypes.c_int(), ctypes.c_int()
    t = 0
    while lib.rtvla_linear_tile_shape(t, ctypes.byref(r), ctypes.byref(c)) == 0:
        out.append((t, r.value, c.value)); t += 1
    return out


@pytest.mark.parametrize("M,K,N", [
    (768, 1152, 3456),      # SigLIP QKV
    (768, 1152, 1152),      # SigLIP O
    (768, 1152, 4304),      # SigLIP up (N = 16 * 269)
    (768, 4304, 1152),      # SigLIP down (K padded to 4352)
    (788, 2048, 2560),      # Gemma prefix QKV at the headline shape
    (788, 2048, 2048),      # prefix O
    (968, 2048, 2048),      # 968-token prefix
    (256, 1152, 2048),      # projector, one view
    (37, 136, 48),          # ragged everything: one partial row tile, K below one stage pair, three column tiles
    (225, 264, 272),        # one row past the largest tile, ragged K and N
])
def test_mfma_gemm_every_tile_and_split_against_fp32_matmul(M, K, N):
    import rtvla_capi as capi
    lib = capi.load()
    tiles = _tiles(lib)
    assert len(tiles) >= 4
    ran = 0
    for tile, rows, cols in tiles:
        for nsplit in (1, 2, 3, 4, 8):
            if nsplit > 1 and N > 2048:
                continue
            res = _run(lib, capi, M, K, N, tile, nsplit)
            if res is None:
                continue                                   # this tile cannot take this K / split (reported as RTVLA_ERR_LIMIT)
            ran += 1
            assert res[0] <= REL_TOL and res[1] <= 1.01, ("tile %dx%d split %d" % (rows, cols, nsplit), res)
    assert ran >= 4
    # the forward's own choice for this shape, one pass and through the partial + reduce route
    for nsplit in (1, 0):
        if nsplit == 0 and N > 2048:
            continue
        res = _run(lib, capi, M, K, N, capi.TILE_AUTO, nsplit, bias=(nsplit == 1))
        assert res is not None and res[0] <= REL_TOL and res[1] <= 1.01, (nsplit, res)


@pytest.mark.parametrize("M,K,N", [(51, 1024, 2560), (51, 2048, 1024), (51, 4096, 1024), (64, 1024, 4096), (1, 1024, 1024), (17, 2048, 48),
                                   (101, 1024, 2560), (128, 4096, 1024), (65, 2048, 1024)])      # (the last three: two 64-row blocks / up to eight 16-row blocks)
def test_weight_streaming_kernel_against_fp32_matmul(M, K, N):
    import rtvla_capi as capi
    lib = capi.load()
    res = _run(lib, capi, M, K, N, capi.TILE_SKINNY, 1)
    assert res is not None and res[0] <= REL_TOL and res[1] <= 1.01, res


def test_unit_entry_rejects_what_it_cannot_run():
    import rtvla_capi as capi
    lib = capi.load()
    assert lib.rtvla_linear_workspace_bytes(16, 12, 16, -1, 1) == 0          # K not a multiple of 8
    assert lib.rtvla_linear_workspace_bytes(16, 16, 24, -1, 1) == 0          # N not a multiple of 16
    assert lib.rtvla_linear_workspace_bytes(129, 1024, 64, capi.TILE_SKINNY, 1) == 0
    assert lib.rtvla_linear_workspace_bytes(16, 512, 64, capi.TILE_SKINNY, 1) == 0
    assert lib.rtvla_linear_workspace_bytes(64, 128, 4096, 0, 2) == 0        # split-K rows wider than the reduce kernel takes
    x = torch.zeros(16, 128, dtype=torch.bfloat16, device="cuda:0")
    ws = torch.empty(256, dtype=torch.uint8, device="cuda:0")
    rc = lib.rtvla_linear(_P(x.data_ptr()), 16, 128, _P(x.data_ptr()), 16, None, _P(x.data_ptr()), _P(ws.data_ptr()), 256, -1, 1, None)
    assert rc == capi.ERR_SIZE


def test_a_graph_captured_before_a_rebind_is_refused():
    """rtvla_bind after rtvla_graph_capture drops the graph: replaying it would read the old addresses."""
    import synthetic as syn
    import rtvla_capi as capi
    from pi0_infer import Pi0Inference
    ck = syn.pi0_checkpoint(5, 2, "cuda:0", 1, 1)
    img, state, noise = syn.observation(5, 1, 8, "cuda:0")
    m = Pi0Inference(ck, 1, 8)
    a = m.forward(img, state, noise).clone()
    ctx, stream = m._engine.ctx, torch.cuda.current_stream().cuda_stream
    other = torch.zeros_like(m.buffers["diffusion_noise"])
    ctx.bind("diffusion_noise", other.data_ptr(), other.numel() * 2)
    with pytest.raises(capi.RtvlaError) as e:
        ctx.graph_launch(stream)
    assert e.value.code == capi.ERR_STATE
    with pytest.raises(capi.RtvlaError):
        ctx.forward(stream)                                  # not prepared either
    m.buffers["diffusion_noise"] = other
    m._engine.prepare()
    m.record_infer_graph()
    b = m.forward(img, state, noise)
    assert b.data_ptr() == other.data_ptr() and torch.equal(a, b)


# ---------------------------------------------------------------------------------------------------------
# fused GEMM epilogues with a row-major output, and the reduce / normalise pass, each on its own
def _gelu_tanh(a):
    return a * torch.sigmoid(1.5957691216057308 * a * (1.0 + 0.044715 * a * a))


def _run_act(lib, capi, M, K, N, act, tile, seed=0):
    g = torch.Generator(device="cuda:0").manual_seed(seed * 104729 + M + K + N + act)
    x = torch.randn(M, K, device="cuda:0", generator=g).to(torch.bfloat16)
    w = (torch.randn(K, N, device="cuda:0", generator=g) * 0.05).to(torch.bfloat16)
    dual = act != capi.ACT_BIAS_GELU
    w2 = (torch.randn(K, N, device="cuda:0", generator=g) * 0.05).to(torch.bfloat16) if dual else None
    b = None if dual else torch.randn(N, device="cuda:0", generator=g).to(torch.bfloat16)
    need = lib.rtvla_linear_act_workspace_bytes(M, K, N, act, tile)
    if need == 0:
        return None
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    out = torch.full((M, N), 77.0, dtype=torch.bfloat16, device="cuda:0")
    rc = lib.rtvla_linear_act(_P(x.data_ptr()), M, K, _P(w.data_ptr()), _P(w2.data_ptr()) if dual else None, N, _P(b.data_ptr()) if b is not None else None,
                              act, _P(out.data_ptr()), _P(ws.data_ptr()), need, tile, _P(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    if rc == capi.ERR_LIMIT:
        return None
    assert rc == 0, rc
    a = x.float() @ w.float()
    if act == capi.ACT_BIAS_GELU:
        ref = _gelu_tanh(a + b.float())
    elif act == capi.ACT_GEGLU:
        ref = _gelu_tanh(a) * (x.float() @ w2.float())
    else:
        ref = a * torch.sigmoid(a) * (x.float() @ w2.float())
    got = out.float()
    rel = ((got - ref).norm() / ref.norm()).item()
    excess = (got - ref).abs() / (ref.abs() * 2.0 ** -7 + 2e-3 * ref.pow(2).mean().sqrt())      # (the activations use the hardware exp2 / rcp)
    return rel, excess.max().item()


@pytest.mark.parametrize("M,K,N,act", [
    (768, 1152, 4304, 1),       # SigLIP up-projection: bias + GELU
    (788, 2048, 16384, 2),      # Gemma prefix gate / up: GeGLU, 25 row tiles in mixed blocks
    (607, 2048, 6144, 3),       # DM0 prefix gate / up: SwiGLU
    (8115, 1024, 4096, 1),      # DM0 ViT fc: bias + GELU on the eight-wave tile
    (37, 136, 48, 1), (37, 136, 48, 2), (225, 264, 272, 3),      # ragged rows, K and columns
])
def test_fused_activation_epilogues_against_fp32(M, K, N, act):
    import rtvla_capi as capi
    lib = capi.load()
    ran = 0
    for tile, rows, cols in [(capi.TILE_AUTO, 0, 0)] + _tiles(lib):
        if M > 1000 and tile != capi.TILE_AUTO and rows < 128:
            continue                                        # (keeps the 8115-row case short)
        res = _run_act(lib, capi, M, K, N, act, tile)
        if res is None:
            continue                                        # a gated epilogue needs a 256-column tile; the large tiles need an even stage count
        ran += 1
        assert res[0] <= REL_TOL and res[1] <= 1.01, ("tile %dx%d" % (rows, cols), res)
    assert ran >= 3


# the eight-wave tiles deal the row tiles over more blocks than the least number where the last round of workgroups has room for them (56 row
# tiles: 8, 9 and 11 blocks instead of 7, 8 and 10 at 256 .. 272 columns); at 9 216 columns it has none
@pytest.mark.parametrize("M,K,N", [(1777, 264, 272), (1792, 136, 256), (1761, 136, 9216), (2720, 136, 3072)])
def test_eight_wave_tiles_with_more_row_blocks_than_the_least(M, K, N):
    import rtvla_capi as capi
    lib = capi.load()
    ran = 0
    for tile, rows, cols in _tiles(lib)[7:11]:
        assert rows in (256, 224, 192, 128) and cols == 256
        res = _run(lib, capi, M, K, N, tile, 1)
        if res is None:
            continue
        ran += 1
        assert res[0] <= REL_TOL and res[1] <= 1.01, ("tile %dx%d" % (rows, cols), res)
    assert ran >= 3


# what the cost model gives to the eight-wave tiles that a caller cannot name: 160 rows (85 row tiles by 12 blocks of columns), the residual epilogue
# (171 row tiles by 4) and a gated one (32 row tiles: 256 rows save a round); one row past a tile, K past a pair of stages, columns past a block
@pytest.mark.parametrize("M,K,N,act", [
    (2705, 136, 3072, 1), (2689, 72, 3056, 1), (5441, 72, 1008, 8), (5473, 264, 1024, 8), (1000, 264, 16384, 2), (993, 136, 16368, 3),
    # every tile with each kind of epilogue, in launches that mix its row blocks with those of 32 rows fewer: 128, 160, 192, 224 and 256 rows
    (1281, 136, 4096, 1), (2689, 136, 3056, 1), (3361, 136, 3056, 1), (4033, 136, 3056, 1), (4705, 136, 3056, 1),
    (10881, 72, 272, 8), (8193, 72, 1008, 8), (10241, 136, 1008, 8), (4033, 72, 3072, 8), (4705, 136, 3072, 8),
    (2689, 136, 16368, 2), (2241, 136, 6144, 3), (4737, 136, 6144, 2), (3841, 136, 16368, 3), (1121, 136, 6144, 2),
    # row blocks of one size: 160, 192, 224 and 256 rows; the output projection of four ViT images (192 and 160 rows)
    (3329, 72, 3072, 8), (4001, 136, 3072, 8), (4673, 72, 3072, 8), (5345, 136, 3072, 8), (10880, 1024, 1024, 8)])
def test_eight_wave_tiles_of_the_cost_model_against_fp32(M, K, N, act):
    import rtvla_capi as capi
    lib = capi.load()
    if act != capi.ACT_RESIDUAL:
        res = _run_act(lib, capi, M, K, N, act, capi.TILE_AUTO)
        assert res is not None and res[0] <= REL_TOL and res[1] <= 1.01, res
        return
    g = torch.Generator(device="cuda:0").manual_seed(M + K + N)
    x = torch.randn(M, K, device="cuda:0", generator=g).to(torch.bfloat16)
    w = (torch.randn(K, N, device="cuda:0", generator=g) * 0.05).to(torch.bfloat16)
    b = torch.randn(N, device="cuda:0", generator=g).to(torch.bfloat16)
    stream = (torch.randn(M + 1, N, device="cuda:0", generator=g) * 3).to(torch.bfloat16)
    out = stream.clone()
    need = lib.rtvla_linear_act_workspace_bytes(M, K, N, act, capi.TILE_AUTO)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    assert lib.rtvla_linear_act(_P(x.data_ptr()), M, K, _P(w.data_ptr()), None, N, _P(b.data_ptr()), act, _P(out.data_ptr()), _P(ws.data_ptr()), need,
                                capi.TILE_AUTO, _P(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    ref = x.float() @ w.float() + b.float() + stream[:M].float()
    got = out[:M].float()
    excess = (got - ref).abs() / (ref.abs() * 2.0 ** -7 + 1e-3 * ref.pow(2).mean().sqrt())
    assert ((got - ref).norm() / ref.norm()).item() <= REL_TOL and excess.max().item() <= 1.01
    assert torch.equal(out[M], stream[M])


# what the cost model gives to the tiles whose K is split between two groups of waves: 64 x 64 (128 workgroups of 64 x 128 and fewer), 64 x 128 and 96 x 128 (24 K
# stages and more), with rows that end in the first, in the second and behind the last row tile, odd numbers of stages for a group, columns past a block, and
# columns whose K the rule leaves to one group (26 stages in 2 splits of 13); bias, bias + GELU, residual, and partial sums (act None).  That the tiles are taken is asserted by
# name below, for launches of a forward
@pytest.mark.parametrize("M,K,N", [
    (33, 128, 64), (65, 264, 272), (1, 640, 16), (97, 1152, 1152), (256, 2048, 2560), (190, 1664, 2048),
    (532, 2048, 2560), (481, 1528, 2512), (449, 4096, 1536), (788, 2048, 2560), (865, 1536, 2544), (609, 4096, 2048)])
@pytest.mark.parametrize("act", [0, 1, 8, None])
def test_two_k_groups_of_the_cost_model_against_fp32(M, K, N, act):
    import rtvla_capi as capi
    lib = capi.load()
    if act is None:
        res = _run(lib, capi, M, K, min(N, 2048), capi.TILE_AUTO, 0)
    elif act == 0:
        res = _run(lib, capi, M, K, N, capi.TILE_AUTO, 1)
    elif act == 1:
        res = _run_act(lib, capi, M, K, N, act, capi.TILE_AUTO)
    else:
        test_residual_epilogue_in_place_against_fp32(M, K, N)
        return
    assert res is not None and res[0] <= REL_TOL and res[1] <= 1.01, res


def test_forward_takes_two_k_groups_where_workgroups_are_few():
    import synthetic as syn
    import rtvla_capi as capi
    from pi0_infer import Pi0Inference
    m = Pi0Inference(syn.pi0_checkpoint(5, 0, "cuda:0", 1, 1), 1, 8)
    names = [m._engine.ctx.time_launch(stage, 0, 0, 0, 1, torch.cuda.current_stream().cuda_stream)[1] for stage in (capi.STAGE_VISION_LAYER, capi.STAGE_PREFIX_LAYER)]
    assert names == ["vision qkv [64x64 2 K groups split 1]", "prefix qkv [64x64 2 K groups split 1]"]


# the scattering epilogues of both tiles, where each group has row tiles of its own: rows that end in the first, the second and the third row tile of a block, one block of 64 x 64 as well
@pytest.mark.parametrize("views,prompt,tile", [(1, 0, "64x64"), (1, 20, "64x64"), (2, 20, "64x128"), (2, 43, "64x128"), (3, 20, "96x128"), (3, 50, "96x128"), (3, 80, "96x128")])
def test_prefix_qkv_of_two_k_groups(views, prompt, tile):
    import synthetic as syn
    import rtvla_capi as capi
    from oracle import ops
    from pi0_infer import Pi0Inference
    tokens = 256 * views + prompt
    ck = syn.pi0_checkpoint(6, prompt, "cuda:0", 1, 1)
    e = Pi0Inference(ck, views, 8)._engine
    assert e.ctx.time_launch(capi.STAGE_PREFIX_LAYER, 0, 0, 0, 1, torch.cuda.current_stream().cuda_stream)[1] == "prefix qkv [%s 2 K groups split 1]" % tile
    x = torch.randn(tokens, 2048, device="cuda:0", generator=torch.Generator(device="cuda:0").manual_seed(tokens))
    e.buffers["encoder_x_norm"].copy_(x)
    e.buffers["encoder_Q"].fill_(3); e.buffers["encoder_K"].fill_(3); e.buffers["encoder_Vt"].fill_(3)
    e.run_stage(capi.STAGE_PREFIX_LAYER, 0, 0)
    torch.cuda.synchronize()
    qkv, table = x.bfloat16().float().cpu() @ ck["encoder_attn_qkv_w"][0].float().cpu(), ops.rope_table(0, tokens)
    # the result is rounded by at most 2^-9 of itself, the product ahead of the rotation at most likewise, which moves its pair's partner too: 2^-9 (1 + sqrt(2)) of a head's row at worst
    for name, want in (("encoder_Q", ops.rope_interleaved(qkv[:, :2048], table).reshape(-1, 256)), ("encoder_K", ops.rope_interleaved(qkv[:, 2048:2304], table)), ("encoder_V", qkv[:, 2304:])):
        got = e.reference_buffer(name).float().cpu().reshape(-1, 256)
        rows = want.shape[0]
        assert ((got[:rows] - want).norm(dim=1) / want.norm(dim=1)).max().item() <= 2.0 ** -9 * 2.42, name
        assert name == "encoder_Q" or bool((got[rows:] == 3).all()), name


@pytest.mark.parametrize("images,lang,tile", [(1, 7, "64x128"), (1, 37, "64x128"), (1, 69, "64x128"), (3, 100, "96x128"), (3, 109, "96x128"), (3, 139, "96x128")])
def test_prefix_heads_of_two_k_groups(images, lang, tile):
    """DM0, whose heads are normalised behind a barrier of the whole workgroup: by each group for the row tiles that it keeps."""
    import rtvla_capi as capi
    from test_gpu_dm0 import one_layer_policy, test_prefix_heads_are_normalised_by_their_gemm as heads_against_fp32
    m = one_layer_policy(images, lang)[0]
    assert m._engine.ctx.time_launch(capi.STAGE_PREFIX_LAYER, 0, 0, 0, 1, torch.cuda.current_stream().cuda_stream)[1] == "prefix qkv [%s 2 K groups split 1]" % tile
    heads_against_fp32(images, lang)


# a caller's own split with the cost model's tile: 10 stages in 2, 3 and 4 splits of 5, 4 and 3, which two groups cannot share; 32 in 2, 3 and 4
@pytest.mark.parametrize("M,K,N,nsplit", [(65, 640, 272, 2), (65, 640, 272, 3), (65, 640, 272, 4), (532, 2048, 1536, 3), (532, 2048, 1536, 4), (788, 2048, 2048, 3), (788, 2048, 2048, 2)])
def test_two_k_groups_with_a_callers_split(M, K, N, nsplit):
    import rtvla_capi as capi
    res = _run(capi.load(), capi, M, K, N, capi.TILE_AUTO, nsplit)
    assert res is not None and res[0] <= REL_TOL and res[1] <= 1.01, res


def test_eight_wave_tiles_give_what_their_offsets_cannot_reach_to_the_four_wave_kernel():
    import rtvla_capi as capi
    lib = capi.load()
    res = _run(lib, capi, 3, (1 << 21) + 8, 16, 7, 1)           # one 16-byte piece of K past what 32-bit offsets reach
    assert res is not None and res[0] <= REL_TOL and res[1] <= 1.01, res


# every tile that takes the epilogue, at whole and ragged tiles; the stream is read and written in place, rows behind it stay as they are
@pytest.mark.parametrize("M,K,N", [(2720, 1024, 1024), (2720, 4096, 1024), (224, 128, 256), (225, 264, 272), (37, 136, 48), (1, 64, 16), (97, 192, 144)])
def test_residual_epilogue_in_place_against_fp32(M, K, N):
    import rtvla_capi as capi
    lib = capi.load()
    g = torch.Generator(device="cuda:0").manual_seed(M + K + N)
    x = torch.randn(M, K, device="cuda:0", generator=g).to(torch.bfloat16)
    w = (torch.randn(K, N, device="cuda:0", generator=g) * 0.05).to(torch.bfloat16)
    b = torch.randn(N, device="cuda:0", generator=g).to(torch.bfloat16)
    stream = (torch.randn(M + 1, N, device="cuda:0", generator=g) * 3).to(torch.bfloat16)
    ref = x.float() @ w.float() + b.float() + stream[:M].float()
    ran = 0
    for tile, rows, cols in [(capi.TILE_AUTO, 0, 0)] + _tiles(lib):
        need = lib.rtvla_linear_act_workspace_bytes(M, K, N, capi.ACT_RESIDUAL, tile)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
        out = stream.clone()
        rc = lib.rtvla_linear_act(_P(x.data_ptr()), M, K, _P(w.data_ptr()), None, N, _P(b.data_ptr()), capi.ACT_RESIDUAL, _P(out.data_ptr()),
                                  _P(ws.data_ptr()), need, tile, _P(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        if rc == capi.ERR_LIMIT:
            continue                                        # the eight-wave tiles, and the large ones at an odd number of stages
        assert rc == 0
        ran += 1
        got = out[:M].float()
        excess = (got - ref).abs() / (ref.abs() * 2.0 ** -7 + 1e-3 * ref.pow(2).mean().sqrt())
        assert ((got - ref).norm() / ref.norm()).item() <= REL_TOL and excess.max().item() <= 1.01, (tile, rows, cols)
        assert torch.equal(out[M], stream[M])
    assert ran >= 5
    assert lib.rtvla_linear_act_workspace_bytes(M, K, N, 5, -1) == 0


@pytest.mark.parametrize("M", [1, 3, 5, 2720])
def test_layer_norm_of_1024_wide_rows_alone(M):
    """Four rows a workgroup, so row counts off by one; against float64: half a bf16 step of the result, and of the sum's terms fp32 errors."""
    import rtvla_capi as capi
    lib = capi.load()
    g = torch.Generator(device="cuda:0").manual_seed(M)
    x = (torch.randn(M, 1024, device="cuda:0", generator=g) * 2 + 0.5).bfloat16()
    w = (1 + 0.1 * torch.randn(1024, device="cuda:0", generator=g)).bfloat16()
    b = (0.1 * torch.randn(1024, device="cuda:0", generator=g)).bfloat16()
    out = torch.full((M + 1, 1024), 9.0, dtype=torch.bfloat16, device="cuda:0")
    assert lib.rtvla_reduce_norm(None, 0, M, 1024, None, _P(x.data_ptr()), 2, _P(w.data_ptr()), _P(b.data_ptr()), ctypes.c_float(1e-5),
                                 None, _P(out.data_ptr()), _P(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    ref = torch.nn.functional.layer_norm(x.double(), (1024,), w.double(), b.double(), 1e-5)
    assert ((out[:M].double() - ref).abs() <= ref.abs() * 2.0 ** -8 + 1e-5).all()
    assert (out[M] == 9.0).all()


# Groups of four columns past the row read the last one again: rows that end inside, at and just behind a pass of 256 groups, in place, next row untouched;
# against float64: half a bf16 step of the sum and of the result, and of the sum's terms fp32 errors.
@pytest.mark.parametrize("N", [4, 252, 1020, 1024, 1028, 2044, 2048])
@pytest.mark.parametrize("nsplit,norm", [(2, 2), (3, 1), (8, 0), (0, 2)])
def test_reduce_rows_that_end_around_a_pass(N, nsplit, norm):
    import rtvla_capi as capi
    lib = capi.load()
    g = torch.Generator(device="cuda:0").manual_seed(N + nsplit)
    M = 3
    parts = torch.randn(max(nsplit, 1), M, N, device="cuda:0", generator=g)
    bias, nw, nb = (torch.randn(N, device="cuda:0", generator=g).bfloat16() for _ in range(3))
    x = torch.full((M + 1, N), 9.0, dtype=torch.bfloat16, device="cuda:0")
    x[:M] = torch.randn(M, N, device="cuda:0", generator=g)
    res = x[:M].clone()
    xn = torch.full((M + 1, N), 9.0, dtype=torch.bfloat16, device="cuda:0")
    assert lib.rtvla_reduce_norm(_P(parts.data_ptr()) if nsplit else None, nsplit, M, N, _P(bias.data_ptr()), _P(x.data_ptr()), norm, _P(nw.data_ptr()),
                                 _P(nb.data_ptr()), ctypes.c_float(1e-5), _P(x.data_ptr()), _P(xn.data_ptr()) if norm else None,
                                 _P(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    terms = [bias.double().expand(M, N), res.double()] + [parts[i].double() for i in range(nsplit)]
    want, size = sum(terms), sum(t.abs() for t in terms)
    assert ((x[:M].double() - want).abs() <= want.abs() * 2.0 ** -8 + size * 2.0 ** -20).all()
    xb = x[:M].double()
    if norm:
        ref = torch.nn.functional.layer_norm(xb, (N,), nw.double(), nb.double(), 1e-5) if norm == 2 else xb * torch.rsqrt(xb.pow(2).mean(-1, keepdim=True) + 1e-5)
        assert ((xn[:M].double() - ref).abs() <= ref.abs() * 2.0 ** -8 + 1e-4).all()
        assert (xn[M] == 9.0).all()
    assert (x[M] == 9.0).all()


@pytest.mark.parametrize("M,N,nsplit,norm,has_bias,has_res", [
    (768, 1152, 2, 2, True, True),        # SigLIP O projection: split 2 + bias + residual + LayerNorm
    (768, 1152, 4, 2, True, True),        # SigLIP down projection
    (768, 1152, 0, 2, False, True),       # LayerNorm of a stream alone (first layer)
    (788, 2048, 1, 1, False, True),       # prefix O projection: one partial + residual + RMS norm
    (788, 2048, 4, 1, False, True),       # prefix down projection
    (968, 2048, 8, 1, False, True), (33, 2048, 6, 1, True, False), (5, 1024, 3, 0, True, True), (2705, 1024, 1, 2, True, True),
])
def test_reduce_bias_residual_norm_against_fp32(M, N, nsplit, norm, has_bias, has_res):
    import rtvla_capi as capi
    lib = capi.load()
    g = torch.Generator(device="cuda:0").manual_seed(M * 31 + N + nsplit)
    parts = torch.randn(max(nsplit, 1), M, N, device="cuda:0", generator=g)
    bias = torch.randn(N, device="cuda:0", generator=g).bfloat16() if has_bias else None
    res = (torch.randn(M, N, device="cuda:0", generator=g) * 2 + 0.5).bfloat16() if has_res else None
    nw = (1 + 0.1 * torch.randn(N, device="cuda:0", generator=g)).bfloat16()
    nb = (0.1 * torch.randn(N, device="cuda:0", generator=g)).bfloat16()
    x = torch.full((M, N), 9.0, dtype=torch.bfloat16, device="cuda:0")
    xn = torch.full((M, N), 9.0, dtype=torch.bfloat16, device="cuda:0")
    eps = 1e-5 if norm == 2 else 1e-6
    rc = lib.rtvla_reduce_norm(_P(parts.data_ptr()) if nsplit else None, nsplit, M, N, _P(bias.data_ptr()) if has_bias else None,
                               _P(res.data_ptr()) if has_res else None, norm, _P(nw.data_ptr()), _P(nb.data_ptr()), ctypes.c_float(eps),
                               _P(x.data_ptr()), _P(xn.data_ptr()) if norm else None, _P(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, rc
    torch.cuda.synchronize()
    want = (parts[:nsplit].sum(0) if nsplit else torch.zeros(M, N, device="cuda:0"))
    if has_bias:
        want = want + bias.float()
    if has_res:
        want = want + res.float()
    assert ((x.float() - want).norm() / want.norm()).item() <= REL_TOL
    assert ((x.float() - want).abs() <= want.abs() * 2.0 ** -7 + 1e-3).all()
    if norm:
        xb = x.float()                                      # the norm reads the rounded stream, as the forward's next GEMM input does
        if norm == 2:
            ref = torch.nn.functional.layer_norm(xb, (N,), nw.float(), nb.float(), eps)
        else:
            ref = xb * torch.rsqrt(xb.pow(2).mean(-1, keepdim=True) + eps)
        assert ((xn.float() - ref).norm() / ref.norm()).item() <= REL_TOL
        assert ((xn.float() - ref).abs() <= ref.abs() * 2.0 ** -7 + 2e-3).all()
