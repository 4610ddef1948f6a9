"""GPU parity of the observation pre-/post-processing kernels against oracle/transforms.py (itself pinned against
Pillow and numpy in tests/test_oracle_transforms.py).  Bit-exact: integer images, IEEE double statistics."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _img(seed, h, w):
    rng = np.random.RandomState(seed)
    img = rng.randint(0, 256, size=(h, w, 3)).astype(np.uint8)
    yy, xx = np.mgrid[0:h, 0:w]
    img[..., 0] = ((xx * 255) // max(1, w - 1)).astype(np.uint8)
    img[h // 4: h // 2, w // 3: w // 2, 2] = 255
    return img


@pytest.mark.parametrize("h,w", [(480, 640), (720, 1280), (224, 224), (100, 150), (640, 480), (250, 224), (224, 300), (37, 53), (1080, 1920)])
def test_image_preprocessing_matches_the_pillow_restatement_bit_exactly(h, w):
    from oracle import transforms as T
    from obs_transforms import ObservationTransforms
    tr = ObservationTransforms("pi0")
    img = _img(h * 7 + w, h, w)
    want = torch.from_numpy(T.normalize_image(T.resize_with_pad(img))).to(torch.bfloat16)
    out = torch.full((224, 224, 3), 7.0, dtype=torch.bfloat16, device="cuda:0")
    tr.resize_pad_normalize_into(img, out)
    torch.cuda.synchronize()
    got = out.cpu()
    assert torch.equal(got, want), "mismatching elements: %d" % (got != want).sum().item()


# (either side of the rule for the threads of a block: 448 and 482 rows, of which a block has 24 and 25; 2 460 and 2 640 rows of as many, of which it has 58 and 65 in more blocks than CUs)
@pytest.mark.parametrize("h,w", [(1, 1), (4, 5), (9, 300), (300, 9), (223, 225), (448, 448), (482, 481), (479, 641), (717, 1279), (2700, 1801), (2460, 2460), (2640, 2640)])
@pytest.mark.parametrize("fmt", ["u8", "u8_chw", "f32", "f32_chw"])
def test_frame_formats_at_the_edges_of_the_tiles(h, w, fmt):
    """Every frame format on the device: single pixels, strips narrower than a tile, windows that end with the buffer, both tile heights."""
    from oracle import transforms as T
    from obs_transforms import ObservationTransforms
    tr = ObservationTransforms("pi0")
    img = np.random.RandomState(h * 31 + w).randint(0, 256, size=(h, w, 3)).astype(np.uint8)
    x = img if fmt.startswith("u8") else (img.astype(np.float32) + 0.3) / 255.0
    if fmt.endswith("chw"):
        x = x.transpose(2, 0, 1).copy()
    want = torch.from_numpy(T.normalize_image(T.resize_with_pad(T.parse_image(x)))).to(torch.bfloat16)      # (three rows are read as channels first)
    frame = torch.from_numpy(x).cuda()
    out = torch.full((224, 224, 3), 7.0, dtype=torch.bfloat16, device="cuda:0")
    tr.resize_pad_normalize_into(frame, out)
    assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("h,w", [(224, 224), (225, 224), (226, 301), (1080, 1920), (1920, 1079), (2065, 2065), (2066, 2066)])
@pytest.mark.parametrize("chw", [False, True])
def test_float_frames_staged_and_not(h, w, chw):
    """Either side of the rule that stages float frames in LDS (more than 4 taps, 76 KB); frames that start between two 16-byte pieces; values
    whose low byte counts."""
    from oracle import transforms as T
    from obs_transforms import ObservationTransforms
    tr = ObservationTransforms("pi0")
    x = (np.random.RandomState(h + w).rand(h, w, 3) * 3 - 1).astype(np.float32)
    if chw:
        x = x.transpose(2, 0, 1).copy()
    want = torch.from_numpy(T.normalize_image(T.resize_with_pad((255 * (x.transpose(1, 2, 0) if chw else x)).astype(np.int32).astype(np.uint8)))).to(torch.bfloat16)
    room = torch.empty(x.size + 1, dtype=torch.float32, device="cuda:0")
    frame = room[1:].view(x.shape)
    frame.copy_(torch.from_numpy(x))
    out = torch.full((224, 224, 3), 7.0, dtype=torch.bfloat16, device="cuda:0")
    tr.resize_pad_normalize_into(frame, out)
    assert torch.equal(out.cpu(), want)


def test_image_inputs_float_and_chw_and_errors():
    from oracle import transforms as T
    from obs_transforms import ObservationTransforms
    tr = ObservationTransforms("pi05")
    rng = np.random.RandomState(3)
    f = rng.rand(3, 120, 90).astype(np.float32)                          # CHW float in [0, 1]
    want = torch.from_numpy(T.normalize_image(T.resize_with_pad(T.parse_image(f)))).to(torch.bfloat16)
    out = torch.empty(224, 224, 3, dtype=torch.bfloat16, device="cuda:0")
    tr.resize_pad_normalize_into(f, out)
    assert torch.equal(out.cpu(), want)
    with pytest.raises(ValueError):
        tr.resize_pad_normalize_into(np.zeros((10, 10, 4), dtype=np.uint8), out)
    with pytest.raises(ValueError):
        tr.resize_pad_normalize_into(np.zeros((10, 10, 3), dtype=np.uint8), torch.empty(224, 224, 3, device="cuda:0"))
    with pytest.raises(RuntimeError):                                    # shrink factor above the supported 31
        tr.resize_pad_normalize_into(np.zeros((8000, 16, 3), dtype=np.uint8), out)


@pytest.mark.parametrize("version", ["pi0", "pi05"])
def test_state_and_action_transforms_match_numpy_bit_exactly(version):
    from oracle import transforms as T
    from obs_transforms import ObservationTransforms
    rng = np.random.RandomState(11)
    n = 14
    stats = {"state": {"mean": rng.randn(n).tolist(), "std": (rng.rand(n) + 0.1).tolist(),
                       "q01": (-1 - rng.rand(n)).tolist(), "q99": (1 + rng.rand(n)).tolist()},
             "actions": {"mean": rng.randn(n).tolist(), "std": (rng.rand(n) + 0.1).tolist(),
                         "q01": (-1 - rng.rand(n)).tolist(), "q99": (1 + rng.rand(n)).tolist()}}
    tr = ObservationTransforms(version, stats, state_len=n, action_dim=n)
    state = rng.randn(n) * 1.5
    state[0] = stats["state"]["q01"][0] - 3.0                            # far below the first bin edge
    state[1] = stats["state"]["q99"][1] + 3.0                            # far above the last one
    want = T.normalize_state(state, stats["state"], version)
    buf = torch.zeros(32, dtype=torch.bfloat16, device="cuda:0")
    z, bins = tr._normalize_state(state, want_bins=True, out_bf16=buf)
    torch.cuda.synchronize()
    assert np.array_equal(z.cpu().numpy(), want)
    assert torch.equal(buf.cpu(), torch.from_numpy(want.astype(np.float32)).to(torch.bfloat16))
    assert np.array_equal(bins.cpu().numpy(), T.digitize_state(want))
    edges = torch.tensor(T.DIGITIZE_BINS)                                # values exactly on bin edges
    a_stats = {"mean": [0.0] * 32, "std": [1.0 - 1e-6] * 32, "q01": [-1.0] * 32, "q99": [1.0 - 1e-6] * 32}
    tr2 = ObservationTransforms(version, {"state": a_stats}, state_len=32)
    for chunk in edges.split(32):
        zz, bb = tr2._normalize_state(chunk.numpy(), want_bins=True)
        assert np.array_equal(bb.cpu().numpy(), T.digitize_state(zz.cpu().numpy()))
    actions = torch.from_numpy(rng.randn(50, 32).astype(np.float32)).to(torch.bfloat16).cuda()
    got = tr.postprocess_actions(actions, state)
    ref = T.postprocess_actions(actions.cpu().float().numpy(), stats["actions"], version, state, n)
    assert got.shape == (50, n) and np.array_equal(got.cpu().numpy(), ref)
    tr7 = ObservationTransforms(version, stats, state_len=n, action_dim=7)
    assert np.array_equal(tr7.postprocess_actions(actions, state).cpu().numpy(),
                          T.postprocess_actions(actions.cpu().float().numpy(), stats["actions"], version, state, 7))


def test_whole_observation_through_the_policy():
    """infer(): camera frames + raw state -> actions, against the oracle transforms wrapped around the same policy."""
    import synthetic as syn
    from oracle import transforms as T
    from obs_transforms import ObservationTransforms
    from pi0_infer import Pi0Inference
    rng = np.random.RandomState(5)
    ck = syn.pi0_checkpoint(31, 2, "cuda:0", 1, 2)
    policy = Pi0Inference(ck, 2, 10)
    stats = {"state": {"mean": rng.randn(7).tolist(), "std": (rng.rand(7) + 0.5).tolist()},
             "actions": {"mean": rng.randn(7).tolist(), "std": (rng.rand(7) + 0.5).tolist()}}
    tr = ObservationTransforms("pi0", stats, state_len=7, action_dim=7)
    frames = {"base_0_rgb": _img(1, 480, 640), "left_wrist_0_rgb": _img(2, 360, 360), "right_wrist_0_rgb": _img(3, 10, 10)}
    state = rng.randn(7)
    noise = rng.randn(10, 32).astype(np.float32)
    out = tr.infer(policy, dict(frames, state=state), noise)["actions"]
    imgs = torch.stack([torch.from_numpy(T.normalize_image(T.resize_with_pad(frames[k]))) for k in ("base_0_rgb", "left_wrist_0_rgb")])
    st = torch.from_numpy(T.normalize_state(state, stats["state"], "pi0").astype(np.float32))
    ref_actions = policy.forward(imgs, st, torch.from_numpy(noise)).cpu().float().numpy()
    ref = T.postprocess_actions(ref_actions, stats["actions"], "pi0", state, 7)
    assert out.shape == (10, 7) and np.array_equal(out, ref)


def _outcome(call):
    try:
        return call()
    except Exception as e:
        return type(e), str(e)


@pytest.mark.parametrize("version", ["pi0", "pi05"])
def test_host_calls_and_the_general_way_agree(version):
    """What the host calls take and what they leave to the general way, accepted or refused: the same bits, the same errors."""
    from obs_transforms import ObservationTransforms, _GeneralWay
    rng = np.random.RandomState(41)
    stats = {g: {"mean": rng.randn(7).tolist(), "std": (rng.rand(7) + 0.5).tolist(), "q01": (-1 - rng.rand(7)).tolist(), "q99": (1 + rng.rand(7)).tolist()}
             for g in ("state", "actions")}
    plain, general = (ObservationTransforms(version, stats) for _ in range(2))
    general._host = _GeneralWay
    u8 = torch.from_numpy(rng.randint(0, 256, size=(61, 47, 3)).astype(np.uint8)).cuda()
    f32 = u8.float() / 255 + 0.001

    class Sub(torch.Tensor):
        pass

    frames = [u8, f32, u8.permute(2, 0, 1).contiguous(), f32.permute(2, 0, 1).contiguous(), u8.permute(1, 0, 2), f32.permute(2, 0, 1), u8[::2, 1:], u8.cpu(), u8.cpu().numpy(),
              f32.double(), f32.half(), u8.long(), u8.as_subclass(Sub), torch.nn.Parameter(f32), u8[:0], u8[..., :2], u8[0], u8[None], u8.bool(), u8[:1].expand(9000, 47, 3).contiguous()]
    for i, frame in enumerate(frames):
        for view in (lambda: torch.full((224, 224, 3), 7.0, dtype=torch.bfloat16, device="cuda:0"), lambda: torch.zeros(224, 224, 3, device="cuda:0"),
                     lambda: torch.zeros(3, 224, 224, 3, dtype=torch.bfloat16, device="cuda:0")[1], lambda: torch.zeros(224, 224, 6, dtype=torch.bfloat16, device="cuda:0")[..., :3]):
            got, want = (_outcome(lambda: tr.resize_pad_normalize_into(frame, view())) for tr in (plain, general))
            assert got == want if isinstance(want, tuple) else torch.equal(got, want), i
    st = rng.randn(7)
    states = [st, st.tolist(), st.astype(np.float32), st[::-1], np.concatenate([st, st])[::2], st.astype(">f8"), torch.from_numpy(st), np.float64(0.3), rng.randn(32), rng.randn(33),
              np.zeros(0), rng.randn(2, 7), np.arange(7), "no"]
    for i, values in enumerate(states):
        for bins in (False, True):
            for out in (None, 1):
                outs = [torch.full((32,), 5.0, dtype=torch.bfloat16, device="cuda:0") if out else None for _ in range(2)]
                got, want = (_outcome(lambda: tr._normalize_state(values, want_bins=bins, out_bf16=o)) for tr, o in zip((plain, general), outs))
                if not isinstance(want[0], torch.Tensor):
                    assert got == want, i
                    continue
                assert torch.equal(got[0], want[0]) and (torch.equal(got[1], want[1]) if bins else got[1] is want[1] is None), i
                assert got[0].dtype == want[0].dtype and (not out or torch.equal(*outs))
        acts = torch.from_numpy(rng.randn(50, 32).astype(np.float32)).to(torch.bfloat16).cuda()
        for a in (acts, acts[:1], acts[:0], acts[::2], acts.float(), acts[:, :7].contiguous(), acts.view(2, 25, 32), acts[0], acts.as_subclass(Sub)):
            got, want = (_outcome(lambda: tr.postprocess_actions(a, values)) for tr in (plain, general))
            assert got == want if isinstance(want, tuple) else torch.equal(got, want), i


def test_state_outputs_and_views_in_other_memory():
    """Pinned memory is written as device memory is; other types, strides, sizes and pageable memory are refused, before any launch, by the host calls and the general way alike."""
    from obs_transforms import ObservationTransforms, _GeneralWay
    rng = np.random.RandomState(42)
    stats = {"state": {"mean": rng.randn(7).tolist(), "std": (rng.rand(7) + 0.5).tolist()}, "actions": {"mean": [0.0] * 7, "std": [1.0] * 7}}
    plain, general = (ObservationTransforms("pi0", stats) for _ in range(2))
    general._host = _GeneralWay
    st, frame, dev = rng.randn(7), torch.from_numpy(rng.randint(0, 256, size=(61, 47, 3)).astype(np.uint8)).cuda(), "cuda:0"
    good, view = torch.zeros(32, dtype=torch.bfloat16, device=dev), torch.zeros(224, 224, 3, dtype=torch.bfloat16, device=dev)
    plain._normalize_state(st, out_bf16=good)
    plain.resize_pad_normalize_into(frame, view)
    for tr in (plain, general):
        for out in (torch.zeros(32, dtype=torch.bfloat16).pin_memory(), torch.zeros(2, 32, dtype=torch.bfloat16, device=dev)):
            tr._normalize_state(st, out_bf16=out)
            torch.cuda.synchronize()
            assert torch.equal(out.reshape(-1)[:32].cpu(), good.cpu())
        pinned = torch.zeros(224, 224, 3, dtype=torch.bfloat16).pin_memory()
        tr.resize_pad_normalize_into(frame, pinned)
        torch.cuda.synchronize()
        assert torch.equal(pinned, view.cpu())
        for out in (torch.zeros(32, device=dev), torch.zeros(31, dtype=torch.bfloat16, device=dev), torch.zeros(64, dtype=torch.bfloat16, device=dev)[::2], torch.zeros(32, dtype=torch.bfloat16)):
            with pytest.raises(ValueError, match="out_bf16"):
                tr._normalize_state(st, out_bf16=out)
        with pytest.raises(ValueError, match="out_view"):
            tr.resize_pad_normalize_into(frame, torch.zeros(224, 224, 3, dtype=torch.bfloat16))
        for acts in (torch.zeros(50, 32, dtype=torch.bfloat16), torch.zeros(32, dtype=torch.bfloat16, device=dev)):
            with pytest.raises(ValueError, match="actions"):
                tr.postprocess_actions(acts, st)


def test_host_calls_follow_the_current_stream_and_are_captured():
    from obs_transforms import ObservationTransforms
    rng = np.random.RandomState(43)
    stats = {g: {"mean": rng.randn(7).tolist(), "std": (rng.rand(7) + 0.5).tolist()} for g in ("state", "actions")}
    tr = ObservationTransforms("pi0", stats)
    frame = torch.from_numpy(rng.randint(0, 256, size=(300, 400, 3)).astype(np.uint8)).cuda()
    out, actions, st = torch.zeros(224, 224, 3, dtype=torch.bfloat16, device="cuda:0"), torch.randn(50, 32, device="cuda:0").to(torch.bfloat16), rng.randn(7)

    def observe():
        tr.resize_pad_normalize_into(frame, out)
        return tr._normalize_state(st, want_bins=True) + (tr.postprocess_actions(actions, st),)
    want = [t.clone() for t in observe()] + [out.clone()]
    torch.cuda.synchronize()
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    out.zero_()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = observe()
    side.synchronize()
    assert all(torch.equal(a, b) for a, b in zip((*got, out), want))
    with torch.cuda.graph(graph, stream=side):
        got = observe()
    for _ in range(3):
        for t in (*got, out):
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip((*got, out), want))
