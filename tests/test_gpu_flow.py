"""The resident flow kernel (csrc/flow.hip) against the flow loop as launches, which a caller's own graph of rtvla_forward gets: the
same weights and noise at the suffix sizes where the kernel's row tiles end, and beside a second process on the same GPU."""
import ctypes
import os
import subprocess
import sys
import threading

import pytest
import torch

import rtvla_capi as capi
import synthetic as syn
from _engine import tile_ft, tile_vt, untile_ft, untile_vt

pytestmark = pytest.mark.gpu


def policy(model, seed, views, prompt, chunk, change=lambda checkpoint: None):
    """(policy, arguments of its forward) at one ViT layer and two decoder layers, of the seeded checkpoint after `change`"""
    if model == "dm0":
        from dm0_infer import DM0Inference
        ck = syn.dm0_checkpoint(seed, "cuda:0", 1, 2, vocab=300)
        change(ck)
        return DM0Inference(ck, num_images=views, max_lang_len=prompt), syn.dm0_observation(seed, views, "cuda:0", max_lang_len=prompt, vocab=300)
    images, state, noise = syn.observation(seed, views, chunk, "cuda:0")
    if model == "pi0":
        from pi0_infer import Pi0Inference
        ck = syn.pi0_checkpoint(seed, prompt, "cuda:0", vision_layers=1, llm_layers=2, norms="random")
        change(ck)
        return Pi0Inference(ck, views, chunk), (images, state, noise)
    from pi05_infer import Pi05Inference
    ck = syn.pi05_checkpoint(seed, prompt - 3, "cuda:0", state_tokens=3, vision_layers=1, llm_layers=2, norms="random")
    change(ck)
    return Pi05Inference(ck, views, chunk, discrete_state_input=False), (images, noise)


# suffix rows (Pi0: chunk + 1) at both sides of a pair of row tiles, and prefixes that end inside and at the end of a 32-key block and
# past the 1 024 keys one round of the attention phases covers
@pytest.mark.parametrize("model,views,prompt,chunk", [
    ("pi0", 1, 0, 31), ("pi0", 1, 31, 32), ("pi0", 1, 33, 63), ("pi0", 1, 7, 64), ("pi0", 2, 1, 95), ("pi0", 1, 5, 96), ("pi0", 4, 40, 127),
    ("pi05", 1, 32, 32), ("pi05", 1, 9, 65), ("pi05", 2, 21, 96), ("pi05", 1, 5, 97),
    ("dm0", 1, 23, 50), ("dm0", 2, 24, 50),
])
def test_resident_loop_equals_the_loop_as_launches(model, views, prompt, chunk):
    m, inputs = policy(model, 300 + chunk, views, prompt, chunk)
    engine, noise = m._engine, inputs[-1]
    resident = m.forward(*inputs).float().cpu()                              # also leaves the other inputs in the engine's buffers
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=side):
        engine.run_eager()
    launches = engine.ctx.launch_count()
    for _ in range(3):
        engine.buffers["diffusion_noise"].copy_(noise)
        graph.replay()
        torch.cuda.synchronize()
        as_launches = engine.buffers["diffusion_noise"].float().cpu().reshape(resident.shape)
        # two orders of bf16 rounding: each route is within 1e-2 of the oracle in the mean (test_gpu_parity.py), so they are within 2e-2 of each other
        assert torch.isfinite(resident).all() and (resident - as_launches).abs().mean().item() <= 2e-2
    assert launches > engine.graph_launches                                  # it was the other route
    assert torch.equal(m.forward(*inputs).float().cpu(), resident)


# 32-key blocks of the prefix and of the suffix: 14 + 2 (all shared by two workgroups), 15 + 2, 28 + 2 and 24 + 4 (the suffix's shared), 30 + 2 (none),
# 31 + 2 and 39 + 4 (blocks past the 32nd), 31 + 2 with adaptive norms, 33 + 2 with two query heads
BLOCKS = [("pi0", 1, 190, 50), ("pi0", 1, 200, 50), ("pi0", 3, 128, 50), ("pi0", 3, 0, 127), ("pi0", 3, 192, 50), ("pi0", 3, 200, 50),
          ("pi0", 4, 200, 127), ("pi05", 3, 200, 50), ("dm0", 2, 700, 50)]


@pytest.mark.parametrize("model,views,prompt,chunk", BLOCKS + [("pi05", 3, 200, 33)])
def test_key_blocks_dealt_in_every_way(model, views, prompt, chunk):
    test_resident_loop_equals_the_loop_as_launches(model, views, prompt, chunk)


@pytest.mark.parametrize("model,views,prompt,chunk", BLOCKS)
@pytest.mark.parametrize("limits", [(-1, -1), (0, 0)], ids=["resident", "one workgroup"])
def test_every_key_block_counts_once(model, views, prompt, chunk, limits):
    """One layer whose values tell the keys apart: V of prefix key k is the (k / 16)th unit vector and V of the suffix zero, so that the attention output
    is the probability of every 16 prefix keys."""
    heads, width = (16, 128) if model == "dm0" else (8, 256)                 # query heads; columns of one
    new_v = slice(3072, 4096) if model == "dm0" else slice(2304, 2560)
    m, inputs = policy(model, 970, views, prompt, chunk, lambda ck: ck["decoder_attn_qkv_w"][:, :, new_v].zero_())
    e = m._engine
    m.forward(*inputs)
    prefix, rows = views * (169 if model == "dm0" else 256) + prompt, chunk + (model == "pi0")
    x, cache = e.buffers["decoder_x"].clone(), e.buffers["kv_Vt" if model == "dm0" else "encoder_Vt"]
    keys_pad = cache.numel() // (2 * width * (8 if model == "dm0" else 1))   # (two layers)
    key = torch.arange(keys_pad, device="cuda:0")
    marked = tile_vt(((key // 16 == torch.arange(width, device="cuda:0")[:, None]) & (key < prefix)).to(torch.bfloat16))
    e.ctx.flow_limits(*limits)

    def probabilities(route):
        e.ctx.set_flow_route(route)
        cache.view(-1, marked.numel()).copy_(marked)
        e.buffers["decoder_x"].copy_(x)
        e.buffers["decoder_attn"].zero_()
        e.run_stage(capi.STAGE_SUFFIX_LAYER, 1, 4)
        torch.cuda.synchronize()
        assert e.ctx.flow_status()[0] == (route == capi.FLOW_RESIDENT)
        attn = e.buffers["decoder_attn"]
        return untile_ft(attn, attn.numel() // 2048, 2048)[:rows].double().cpu().view(rows, heads, width)

    # of 16 keys for a head, over the rows, relative: either route rounds it to bf16 (2^-9 at most, twice 2^-9 between two) after adding up 16
    # probabilities rounded to bf16 (2^-9 each, independent: a quarter of that)
    def differ(got, want):
        return ((got - want).norm(dim=0) / want.norm(dim=0).clamp_min(1e-30)).max().item() > 5e-3

    got, want = probabilities(capi.FLOW_RESIDENT), probabilities(capi.FLOW_LAUNCHES)
    halves = (prefix + 15) // 16
    assert (want[:, :, :halves].norm(dim=0) > 0).all() and not want[:, :, halves:].any() and not got[:, :, halves:].any()
    assert not differ(got, want)
    # what a mistake would look like: 16 keys, all 32 of a block or the smallest block of the suffix left out or counted twice
    of_suffix = 1 - want.sum(dim=2, keepdim=True)
    smallest = of_suffix * min(32, (rows - 1) % 32 + 1) / rows
    for times in (-1, 1):
        assert differ(want / (1 + times * smallest), want)
        for size in (1, 2):
            for j in range(0, halves, size):
                wrong = want.clone()
                wrong[:, :, j:j + size] *= 1 + times
                assert differ(wrong / (1 + times * want[:, :, j:j + size].sum(dim=2, keepdim=True)), want)


# suffix rows at the ends of every instance's range, a prefix that ends inside a 32-key block, past one round of the attention phases, and
# a prompt that is shorter than its allocation (Pi05)
SHAPES = [("pi0", 1, 5, 9), ("pi0", 1, 31, 50), ("pi0", 1, 7, 95), ("pi0", 4, 40, 127), ("pi05", 1, 9, 32), ("pi05", 1, 32, 64), ("pi05", 2, 21, 96),
          ("pi05", 1, 5, 128), ("dm0", 1, 23, 50), ("dm0", 2, 24, 50)]


# (the limits are the host's to set: a gate without patience closes before anybody reports, a loop without patience runs to its end at once)
@pytest.mark.parametrize("limits", [(0, 0, -1), (-1, -1, 0)], ids=["gates closed", "loop given up"])
@pytest.mark.parametrize("model,views,prompt,chunk", SHAPES)
def test_one_workgroup_gives_the_same_actions(model, views, prompt, chunk, limits):
    """Whatever keeps the resident kernel from finishing, the actions are those it would have given."""
    m, inputs = policy(model, 500 + chunk, views, prompt, chunk)
    ctx = m._engine.ctx
    want = m.forward(*inputs).clone()
    before = ctx.flow_status()[1]
    ctx.set_flow_route(capi.FLOW_RESIDENT)                                   # (else the second one would be launches)
    ctx.flow_limits(*limits)
    m._engine.capture()                                                      # (its eager forward is the first without patience)
    got = m.forward(*inputs).clone()
    torch.cuda.synchronize()
    assert torch.isfinite(want.float()).all() and torch.equal(got, want)
    assert ctx.flow_status() == (True, before + 2)
    ctx.flow_limits()
    m._engine.capture()
    again = m.forward(*inputs).clone()
    torch.cuda.synchronize()
    assert torch.equal(again, want) and ctx.flow_status() == (True, before + 2)


@pytest.mark.parametrize("model,views,prompt,chunk", SHAPES)
def test_the_second_launch_runs_where_the_first_gave_way(model, views, prompt, chunk):
    m, inputs = policy(model, 550 + chunk, views, prompt, chunk)
    want = m.forward(*inputs).clone()
    m._engine.ctx.flow_limits(0)
    for _ in range(3):
        assert torch.equal(m.forward(*inputs), want)
    torch.cuda.synchronize()
    assert torch.isfinite(want.float()).all() and m._engine.ctx.flow_status() == (True, 0)


@pytest.mark.parametrize("model", ["pi0", "pi05", "dm0"])
def test_one_workgroup_gives_the_same_layer(model):
    """The stages start from the caller's stream and noise; a loop that gave up half way has spoiled neither."""
    m, inputs = policy(model, 600, 1, 20, 40)
    e = m._engine
    e.ctx.set_flow_route(capi.FLOW_RESIDENT)
    m.forward(*inputs)
    x, noise = e.buffers["decoder_x"], e.buffers["diffusion_noise"]
    x0, n0 = x.clone(), noise.clone()
    results = []
    for limits in ((-1, -1, -1), (0, 0, -1), (-1, -1, 0)):
        e.ctx.flow_limits(*limits)
        for stage in (capi.STAGE_SUFFIX_STEP_BEGIN, capi.STAGE_SUFFIX_LAYER, capi.STAGE_SUFFIX_STEP_END):
            x.copy_(x0)
            noise.copy_(n0)
            e.run_stage(stage, 1, 3)
            torch.cuda.synchronize()
            results.append((x.clone(), noise.clone()))
    for k in range(3, 9):
        assert torch.equal(results[k][0], results[k % 3][0]) and torch.equal(results[k][1], results[k % 3][1]), k
    assert e.ctx.flow_status() == (True, 6)


# prefixes that end inside a 32-key block: its rows behind the prefix hold what the last forward's suffix left there
@pytest.mark.parametrize("route", [capi.FLOW_RESIDENT, capi.FLOW_LAUNCHES], ids=["resident", "launches"])
@pytest.mark.parametrize("model,views,prompt,chunk", [("pi0", 1, 20, 50), ("pi05", 1, 9, 33), ("dm0", 1, 24, 50), ("pi0", 1, 31, 9)])
@pytest.mark.parametrize("bad,which", [(float("nan"), -1), (float("inf"), -1), (float("nan"), 0)], ids=["nan noise", "inf noise", "nan images"])
def test_a_forward_on_bad_inputs_leaves_nothing_behind(model, views, prompt, chunk, route, bad, which):
    m, inputs = policy(model, 850, views, prompt, chunk)
    m._engine.ctx.set_flow_route(route)
    want = m.forward(*inputs).clone()
    spoiled = list(inputs)
    spoiled[which] = torch.full_like(inputs[which], bad)
    assert not torch.isfinite(m.forward(*spoiled).float()).any()
    assert torch.equal(m.forward(*inputs), want) and torch.isfinite(want.float()).all()


@pytest.mark.parametrize("model,views,prompt,chunk", [("pi0", 1, 20, 50), ("pi0", 1, 8, 90), ("pi05", 1, 9, 33), ("dm0", 1, 24, 50)])
def test_values_that_look_like_values_not_there_yet(model, views, prompt, chunk):
    """The workgroups wait for words that are not all ones: NaNs with every bit set, in the noise, must not be waited for."""
    m, inputs = policy(model, 870, views, prompt, chunk)
    want = m.forward(*inputs).clone()
    ones = torch.full(inputs[-1].shape, -1, dtype=torch.int16, device=inputs[-1].device).view(torch.bfloat16)
    assert not torch.isfinite(m.forward(*inputs[:-1], ones).float()).any()
    assert torch.equal(m.forward(*inputs), want)
    torch.cuda.synchronize()
    assert m._engine.ctx.flow_status() == (True, 0)


@pytest.mark.parametrize("route", [capi.FLOW_RESIDENT, capi.FLOW_LAUNCHES], ids=["resident", "launches"])
@pytest.mark.parametrize("staged_on", ["device", "host"])
def test_rows_behind_a_short_prompt_are_not_those_of_a_bad_forward(staged_on, route):
    """Pi05 with 40 rows for its prompt: the rows behind a shorter one keep their residual stream from call to call, and nobody may see them."""
    from pi05_infer import Pi05Inference
    rows, vocab = 40, 640
    ck = syn.pi05_checkpoint(860, 0, "cuda:0", 1, 2, state_tokens=0, norms="random")
    del ck["language_embeds"]
    table = syn.normal_bf16(860, "embedding_weight_small", (vocab, 2048), 0.02, "cuda:0")
    images, _, noise = syn.observation(860, 1, 33, "cuda:0")
    if staged_on == "device":
        m = Pi05Inference(dict(ck, embedding_weight=table), 1, 33, max_tokenize_len=rows, discrete_state_input=False)
        forward = lambda img, n: m.forward_ids(img, noise, syn.randint(860, "ids%d" % n, n, vocab)).clone()
    else:
        m = Pi05Inference(dict(ck, language_embeds=torch.zeros(rows, 2048, dtype=torch.bfloat16, device="cuda:0")), 1, 33, discrete_state_input=False)

        def forward(img, n):
            m.weights["language_embeds"] = (table[syn.randint(860, "ids%d" % n, n, vocab).to("cuda:0")].float() * (2048.0 ** 0.5)).to(torch.bfloat16)
            return m.forward(img, noise).clone()
    m._engine.ctx.set_flow_route(route)
    want = forward(images, 4)
    assert not torch.isfinite(forward(torch.full_like(images, float("nan")), 37).float()).any()
    assert torch.equal(forward(images, 4), want) and torch.isfinite(want.float()).all()


@pytest.mark.parametrize("model", ["pi0", "pi05", "dm0"])
def test_launches_after_a_loop_in_one_workgroup(model):
    """Whatever held the CUs may go on doing so: the next 64 forwards take the launches, then the resident kernel is tried again."""
    m, inputs = policy(model, 800, 1, 20, 50)
    ctx = m._engine.ctx
    want = m.forward(*inputs).clone()
    ctx.flow_limits(0, 0)
    assert torch.equal(m.forward(*inputs), want)                             # (alone; the host knows when it has ended)
    torch.cuda.synchronize()
    assert ctx.flow_status() == (True, 1)
    ctx.flow_limits()
    close = []
    for _ in range(64):
        out = m.forward(*inputs).float()
        close.append((out - want.float()).abs().mean())
        assert ctx.flow_status() == (False, 1)
    assert torch.stack(close).max().item() <= 2e-2                           # (as in the comparison of the two routes above)
    assert torch.equal(m.forward(*inputs), want) and ctx.flow_status() == (True, 1)
    ctx.set_flow_route(capi.FLOW_LAUNCHES)
    assert (m.forward(*inputs).float() - want.float()).abs().mean().item() <= 2e-2 and ctx.flow_status() == (False, 1)


@pytest.mark.parametrize("model,views,prompt,chunk", [("pi0", 1, 20, 50), ("pi0", 1, 3, 31), ("pi0", 2, 8, 127), ("pi05", 1, 32, 33), ("pi05", 1, 9, 128),
                                                      ("dm0", 1, 24, 50), ("dm0", 1, 23, 50)] + BLOCKS[1:])
@pytest.mark.parametrize("limits", [(-1, -1), (0, 0)], ids=["resident", "one workgroup"])
def test_the_activations_are_left_where_the_launches_leave_them(model, views, prompt, chunk, limits):
    """One input projection and one layer from the same stream and noise by either route: what `buffers` and `reference_buffer` show of them."""
    m, inputs = policy(model, 950, views, prompt, chunk)
    e = m._engine
    m.forward(*inputs)
    names = ["decoder_attn", "decoder_hidden"] + (["decoder_x_buf"] if model != "pi05" else []) + (["decoder_q_buf"] if model != "dm0" else [])
    caches = ["encoder_K", "encoder_Vt"] if model != "dm0" else []           # (behind the prefix DM0's are working memory)
    keep = {n: e.buffers[n].clone() for n in ["decoder_x", "diffusion_noise"] + caches}
    e.ctx.flow_limits(*limits)
    seen = {}
    for route in (capi.FLOW_RESIDENT, capi.FLOW_LAUNCHES):
        e.ctx.set_flow_route(route)
        for n in names:
            e.buffers[n].zero_()
        for n, t in keep.items():
            e.buffers[n].copy_(t)
        for c in caches:                                                     # rows behind the prefix: gone
            for part in e.buffers[c].view(2, -1):
                if c == "encoder_K":
                    cleared = untile_ft(part, part.numel() // 256, 256)
                    cleared[e.prefix_rows:] = 0
                    part.copy_(tile_ft(cleared))
                else:
                    cleared = untile_vt(part, 256, part.numel() // 256)
                    cleared[:, e.prefix_rows:] = 0
                    part.copy_(tile_vt(cleared))
        e.run_stage(capi.STAGE_SUFFIX_STEP_BEGIN, 0, 4)
        e.buffers["decoder_x"].copy_(keep["decoder_x"])
        e.run_stage(capi.STAGE_SUFFIX_LAYER, 1, 4)
        torch.cuda.synchronize()
        assert e.ctx.flow_status()[0] == (route == capi.FLOW_RESIDENT)
        seen[route] = {n: e.buffers[n].float().clone() for n in names + caches}
        if model != "dm0":
            seen[route].update({"untiled " + n: e.reference_buffer(n).float().clone() for n in names + ["encoder_K", "encoder_V"]})
    for n, want in seen[capi.FLOW_LAUNCHES].items():
        got = seen[capi.FLOW_RESIDENT][n]
        if "encoder_" not in n:
            assert want.norm() > 0
            rows = {"decoder_q_buf": 8}.get(n.split()[-1], 1) * (chunk + (model == "pi0") - (model == "pi0" and "x_buf" in n))
            if not n.startswith("untiled"):                                  # (rows past the suffix are the kernels' padding)
                got, want = (untile_ft(t, t.numel() // t.shape[1], t.shape[1])[:rows] for t in (got, want))
            else:
                got, want = got[:rows], want[:rows]
        # sums of up to 4 096 products in another order, each stage rounded to bf16 (2^-9) as often as on the other route: a few roundings that fall to the other side
        assert ((got - want).norm() / want.norm()).item() < 5e-3, n


def hip_runtime():
    """the HIP runtime of this process"""
    for line in open("/proc/self/maps"):
        if "libamdhip64.so" in line:
            return ctypes.CDLL(line.split()[-1])
    raise RuntimeError("no HIP runtime loaded")


@pytest.mark.parametrize("model", ["pi0", "dm0"])
def test_a_stream_that_may_not_use_every_compute_unit(model):
    """The resident kernel could not begin there: eager forwards and graph launches take the launches, on that stream only."""
    m, inputs = policy(model, 900, 1, 20, 50)
    e = m._engine
    want = m.forward(*inputs).clone()
    torch.cuda.synchronize()
    hip, handle = hip_runtime(), ctypes.c_void_p()
    mask = (ctypes.c_uint32 * 8)(*[0x0fffffff] * 8)                          # 28 of every 32
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(handle), 8, mask) == 0
    masked = torch.cuda.ExternalStream(handle.value)
    with torch.cuda.stream(masked):
        for eager in (True, False, False):
            e.buffers["diffusion_noise"].copy_(inputs[-1].reshape(e.buffers["diffusion_noise"].shape))
            e.run_eager() if eager else e.replay()
            got = e.buffers["diffusion_noise"].float().reshape(want.shape)
            assert e.ctx.flow_status() == (False, 0)
            assert (got - want.float()).abs().mean().item() <= 2e-2
    masked.synchronize()
    assert torch.equal(m.forward(*inputs), want) and e.ctx.flow_status() == (True, 0)
    torch.cuda.synchronize()
    assert hip.hipStreamDestroy(handle) == 0


def test_prepare_neither_waits_nor_judges_the_device_by_its_stream():
    """rtvla_prepare is enqueued, and a device that is busy or a stream that is masked during it decides nothing about later forwards."""
    m, inputs = policy("pi0", 910, 1, 20, 50)
    e = m._engine
    want = m.forward(*inputs).clone()
    torch.cuda.synchronize()
    hip, handle = hip_runtime(), ctypes.c_void_p()
    mask = (ctypes.c_uint32 * 8)(*[0x0fffffff] * 8)
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(handle), 8, mask) == 0
    masked = torch.cuda.ExternalStream(handle.value)
    with torch.cuda.stream(masked):
        for _ in range(100):
            e.replay()
        e.ctx.prepare(masked.cuda_stream)
        assert not masked.query()
    masked.synchronize()
    e.capture()
    assert torch.equal(m.forward(*inputs), want) and e.ctx.flow_status() == (True, 0)
    torch.cuda.synchronize()
    assert hip.hipStreamDestroy(handle) == 0


def test_policies_on_two_streams_and_threads():
    """The loops of one process take turns, whatever streams and threads they come from; each policy's actions are those it gives alone."""
    pairs = [policy(*args) for args in (("pi0", 701, 2, 20, 50), ("dm0", 702, 1, 24, 50))]
    want = [m.forward(*inputs).clone() for m, inputs in pairs]
    torch.cuda.synchronize()
    wrong, errors = [0, 0], []

    def run(k):
        m, inputs = pairs[k]
        try:
            for burst in range(10):                                          # (streams come and go: a new one may have the handle of an old one)
                stream = torch.cuda.Stream()
                with torch.cuda.stream(stream):
                    for _ in range(10):
                        wrong[k] += int(not torch.equal(m.forward(*inputs), want[k]))
        except Exception as e:                                               # (an exception in a thread is nobody's otherwise)
            errors.append(e)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not errors and wrong == [0, 0]
    assert [m._engine.ctx.flow_status() for m, _ in pairs] == [(True, 0)] * 2


def test_only_the_flow_loops_take_turns():
    """What comes before a loop does not wait for the loops of another stream.  Streams share a handful of hardware queues, and what is in one queue
    does wait: one stream of several that gets past the other's loops shows it."""
    (a, a_in), (b, b_in) = policy("pi0", 703, 1, 5, 50), policy("pi0", 704, 1, 5, 50)
    a.forward(*a_in)
    b.forward(*b_in)
    torch.cuda.synchronize()
    first, passed = torch.cuda.Stream(), False
    for second in [torch.cuda.Stream() for _ in range(8)]:
        with torch.cuda.stream(first):
            for _ in range(200):
                a._engine.replay()
        with torch.cuda.stream(second):
            b._engine.run_stage(capi.STAGE_VISION_LAYER, 0)
        second.synchronize()
        passed = not first.query()                                           # 200 forwards against one layer
        first.synchronize()
        if passed:
            break
    assert passed


WORKER = """
import sys
sys.path[:0] = %r
import torch
from test_gpu_flow import policy
m, inputs = policy("pi0", 401, 1, 5, 50)
first = m.forward(*inputs).clone()
print("ready", flush=True)
sys.stdin.readline()
same = sum(int(torch.equal(m.forward(*inputs), first)) for _ in range(500))
print("same", same, bool(torch.isfinite(first.float()).all()), flush=True)
"""


def test_two_processes_on_one_gpu():
    """Both processes' kernels want every CU: whichever is not whole gives way, and no forward is lost."""
    paths = [os.path.dirname(os.path.abspath(__file__)), os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "realtime-vla_amd")]
    workers = [subprocess.Popen([sys.executable, "-u", "-c", WORKER % paths], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True) for _ in range(2)]
    try:
        assert [w.stdout.readline().split() for w in workers] == [["ready"]] * 2
        for w in workers:
            w.stdin.write("go\n")
            w.stdin.flush()
        assert [w.stdout.readline().split() for w in workers] == [["same", "500", "True"]] * 2
    finally:
        for w in workers:
            w.stdin.close()
            w.wait(timeout=60)


def test_three_processes_on_one_gpu():
    """The CUs that one of three leaves may be shared by the other two, so that all of them get to the last launch, of one workgroup: no forward
    is lost there either, and with the route held to the resident kernel all of them are the same bits."""
    paths = [os.path.dirname(os.path.abspath(__file__)), os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "realtime-vla_amd")]
    code = (WORKER % paths).replace("first = ", "m._engine.ctx.set_flow_route(1)\nfirst = ").replace("range(500)", "range(100)")
    workers = [subprocess.Popen([sys.executable, "-u", "-c", code], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True) for _ in range(3)]
    try:
        assert [w.stdout.readline().split() for w in workers] == [["ready"]] * 3
        for w in workers:
            w.stdin.write("go\n")
            w.stdin.flush()
        assert [w.stdout.readline().split() for w in workers] == [["same", "100", "True"]] * 3
    finally:
        for w in workers:
            w.stdin.close()
            w.wait(timeout=60)
