"""Observation pre-/post-processing on the device, with the method names and semantics of the reference's evaluation
harness (/root/reference/test.py:88-201: `_parse_image`, `_resize_with_pad`, `_normalize_image`, `_normalize_state`,
`_digitize_state`, `_unnormalize_actions`, `_apply_input_transforms`, and the action post-processing of `infer`).
The reference runs these in numpy / Pillow on the host for every observation; here each is one or two HIP kernels of
librtvla.so writing straight into the model's input buffers.  PyTorch only owns the memory."""
import warnings

import numpy as np
import torch

import rtvla_capi as capi

_VIEW_SHAPE = (224, 224, 3)


def _reachable(tensor):
    """The kernels take bare pointers: device memory, or host memory that is mapped for the device."""
    return tensor.is_cuda or tensor.is_pinned()


class _GeneralWay:
    """In place of the module of host calls: takes nothing."""
    frame = state = actions = staticmethod(lambda *args: None)


def _host_calls():
    """The module of host calls, which is bound to one build of PyTorch.  The library alone is enough without it: the same launches, by Python and ctypes."""
    try:
        return capi.load_host()
    except (RuntimeError, ImportError) as e:
        warnings.warn("observation calls without _rtvla_host.so, which costs each 2 - 5 us: %s" % e, RuntimeWarning, stacklevel=3)
        return _GeneralWay


class ObservationTransforms:
    def __init__(self, model_version, norm_stats=None, state_len=7, action_dim=7, device=None):
        if model_version not in ("pi0", "pi05"):
            raise ValueError("model_version must be 'pi0' or 'pi05'")
        if not torch.cuda.is_available():
            raise RuntimeError("realtime-vla_amd needs a ROCm GPU (MI355X / gfx950); there is no CPU path")
        self.lib = capi.load()
        self._host = _host_calls()
        self.model_version = model_version
        self.mode = 0 if model_version == "pi0" else 1
        self.norm_stats = norm_stats
        self.state_len, self.action_dim = int(state_len), int(action_dim)
        self.device = torch.device(device) if device is not None else torch.device("cuda", torch.cuda.current_device())
        keys = ("mean", "std") if model_version == "pi0" else ("q01", "q99")
        self._stats = {}
        for group in ("state", "actions"):
            if norm_stats and group in norm_stats:
                a = torch.tensor(np.asarray(norm_stats[group][keys[0]], dtype=np.float64)[:32], device=self.device)
                b = torch.tensor(np.asarray(norm_stats[group][keys[1]], dtype=np.float64)[:32], device=self.device)
                self._stats[group] = (a, b, int(a.numel()))
        self._index = self.device.index if self.device.index is not None else torch.cuda.current_device()
        self.device = torch.device("cuda", self._index)
        # what results are allocated like: cheaper than naming a type and a device in each call
        self._row = torch.empty(32, dtype=torch.float64, device=self.device)
        self._bin_row = torch.empty(32, dtype=torch.int32, device=self.device)

    def _stream(self):
        return torch._C._cuda_getCurrentRawStream(self._index)      # the bare handle: the Stream object costs more than a launch

    @staticmethod
    def _check(rc, what):
        if rc != 0:
            raise RuntimeError("%s failed with rtvla status %d" % (what, rc))

    # ---- images ----
    def _parse_image(self, image):
        """test.py:88-94, but the result lives on the device as uint8 HWC."""
        image = torch.as_tensor(image)
        if image.is_floating_point():
            image = (255 * image).to(torch.uint8)                 # truncation, as numpy's astype
        if image.shape[0] == 3:
            image = image.permute(1, 2, 0)
        return image.to(self.device).contiguous()

    def _frame(self, image):
        """(contiguous tensor on the device, its frame format, height, width): float32 and channels-first frames go to the kernel as
        they are, everything else as _parse_image makes it."""
        if not isinstance(image, torch.Tensor):
            image = torch.as_tensor(image)
        dtype = image.dtype
        if (dtype is not torch.uint8 and dtype is not torch.float32) or image.dim() != 3:
            image, dtype = self._parse_image(image), torch.uint8
        chw = image.shape[0] == 3
        h, w, c = (image.shape[1], image.shape[2], 3) if chw else image.shape
        if c != 3 or image.dtype is not dtype:
            raise ValueError("expected an RGB uint8 image, got shape %s dtype %s" % ((h, w, c), image.dtype))
        if image.device != self.device:
            image = image.to(self.device)
        if not image.is_contiguous():
            image = image.contiguous()
        if dtype is torch.uint8:
            return image, (capi.FRAME_U8_CHW if chw else capi.FRAME_U8_HWC), h, w
        return image, (capi.FRAME_F32_CHW if chw else capi.FRAME_F32_HWC), h, w

    def resize_pad_normalize_into(self, image, out_view, static_scratch=False):
        """_resize_with_pad + _normalize_image of one image into out_view (bf16 [224, 224, 3], e.g. one view of the
        model's observation_images_normalized buffer).  Nothing is allocated for a frame that is on the device already;
        static_scratch (frames of at most 2160 rows at full width) is kept for its callers."""
        rc = None if static_scratch else self._host.frame(image, out_view, self._index)
        if rc is not None:                                        # a plain frame and view: launched
            if rc:
                self._check(rc, "rtvla_preprocess_frame")
            self._keep = image
            return out_view
        if out_view.dtype is not torch.bfloat16 or out_view.shape != _VIEW_SHAPE or not out_view.is_contiguous() or not _reachable(out_view):
            self._frame(image)                                    # (a bad image is reported first)
            raise ValueError("out_view must be a contiguous bf16 [224, 224, 3] tensor in device or pinned memory")
        img, fmt, h, w = self._frame(image)
        if static_scratch:
            img = self._parse_image(img)
            rc = self.lib.rtvla_preprocess_image_static(img.data_ptr(), h, w, out_view.data_ptr(), self._stream())
            if rc == capi.ERR_LIMIT:
                raise ValueError("a %d x %d frame does not fit the library's %d-byte static intermediate buffer (or shrinks by more "
                                 "than a factor of 31)" % (h, w, capi.STATIC_SCRATCH_BYTES))
            self._check(rc, "rtvla_preprocess_image_static")
        else:
            rc = self.lib.rtvla_preprocess_frame(img.data_ptr(), fmt, h, w, out_view.data_ptr(), self._stream())
            if rc:
                self._check(rc, "rtvla_preprocess_frame")
        self._keep = img                                           # alive until the stream has consumed it
        return out_view

    # ---- state ----
    def _normalize_state(self, state, want_bins=False, out_bf16=None):
        """test.py:121-137: returns (normalised float64 [32] on the device, 256-bin indices or None); optionally also
        writes the float32 -> bf16 value into out_bf16 (the model's observation_state_normalized buffer)."""
        if "state" not in self._stats:
            return None, None
        a, b, n_stats = self._stats["state"]
        done = self._host.state(state, a, b, n_stats, self.mode, self._row, self._bin_row if want_bins else None, out_bf16, self._index)
        if type(done) is tuple:                                    # plain values: launched
            return done
        if done is not None:
            self._check(done, "rtvla_preprocess_state_host")
        st = np.ascontiguousarray(state, dtype=np.float64)         # travels with the launch
        if out_bf16 is not None and (out_bf16.dtype is not torch.bfloat16 or out_bf16.numel() < 32 or not out_bf16.is_contiguous() or not _reachable(out_bf16)):
            raise ValueError("out_bf16 must be a contiguous bf16 tensor of 32 values in device or pinned memory")
        z = torch.empty_like(self._row)
        bins = torch.empty_like(self._bin_row) if want_bins else None
        rc = self.lib.rtvla_preprocess_state_host(st.tobytes(), st.size, a.data_ptr(), b.data_ptr(), n_stats, self.mode,
                                                  out_bf16.data_ptr() if out_bf16 is not None else None, z.data_ptr(),
                                                  bins.data_ptr() if bins is not None else None, self._stream())
        if rc:
            self._check(rc, "rtvla_preprocess_state_host")
        return z, bins

    # ---- actions ----
    def postprocess_actions(self, actions_bf16, ori_state):
        """test.py:196-201: un-normalise, add the current state, keep the grippers absolute -> float64 [chunk, action_dim]."""
        if "actions" not in self._stats:
            return None
        a, b, n_stats = self._stats["actions"]
        done = self._host.actions(actions_bf16, ori_state, a, b, n_stats, self.mode, self.action_dim, self._row, self._index)
        if type(done) is torch.Tensor:
            return done
        if done is not None:
            self._check(done, "rtvla_postprocess_actions_host")
        if actions_bf16.dtype is not torch.bfloat16 or actions_bf16.dim() < 2 or actions_bf16.shape[-1] != 32 or not actions_bf16.is_contiguous() or not _reachable(actions_bf16):
            raise ValueError("actions must be a contiguous bf16 [chunk, 32] tensor in device or pinned memory")
        chunk = actions_bf16.shape[0]
        st = np.ascontiguousarray(ori_state, dtype=np.float64)
        out = torch.empty((chunk, self.action_dim), dtype=torch.float64, device=self.device)
        rc = self.lib.rtvla_postprocess_actions_host(actions_bf16.data_ptr(), chunk, a.data_ptr(), b.data_ptr(), n_stats, self.mode,
                                                     st.tobytes(), st.size, self.action_dim, out.data_ptr(), self._stream())
        if rc:
            self._check(rc, "rtvla_postprocess_actions_host")
        return out

    # ---- the whole observation, as TritonInference.infer does around policy.forward (test.py:181-205) ----
    def infer(self, policy, inputs, noise):
        """inputs: {"state", "base_0_rgb", "left_wrist_0_rgb", "right_wrist_0_rgb"[, "prompt"]}; returns {"actions": ndarray}."""
        ori_state = np.asarray(inputs["state"]).copy()
        views = ["base_0_rgb", "left_wrist_0_rgb", "right_wrist_0_rgb"][: policy.num_views]
        img_buf = policy.buffers["observation_images_normalized"]
        for v, name in enumerate(views):
            self.resize_pad_normalize_into(inputs[name], img_buf[v])
        noise_t = torch.as_tensor(noise)
        if self.model_version == "pi0":
            self._normalize_state(ori_state, out_bf16=policy.buffers["observation_state_normalized"])
            actions = policy.forward(img_buf, policy.buffers["observation_state_normalized"], noise_t)
        else:
            _, bins = self._normalize_state(ori_state, want_bins=True)
            actions = policy.forward(img_buf, noise_t, inputs.get("prompt"), bins[: self.state_len].cpu().numpy())
        out = self.postprocess_actions(actions, ori_state)
        return {"actions": out.cpu().numpy()}
