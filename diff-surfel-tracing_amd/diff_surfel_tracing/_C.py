"""ctypes binding of libdst.so, shaped like the compiled `_C` module of the reference package
(reference ext.cpp:7-12): `OptiXStateWrapper`, `build_acceleration_structure`, `trace_surfels`,
`trace_surfels_backward` with the same positional arguments and return tuples
(reference trace_surfels.h:10-83).  There is no fallback: a missing library raises.
"""
import ctypes as C
import os
import threading
import warnings

import torch

_PKG_DIR = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_PKG_DIR, "libdst.so")

NUM_CHANNELS = 3          # reference optix_tracer/config.h:5
DEFAULT_AUX_CHANNELS = 2  # reference optix_tracer/config.h:6
DEFAULT_MAX_TRACE_DEPTH = 1  # reference optix_tracer/config.h:27: mid_val always holds at least two slots
MAX_AUX_CHANNELS = 8
MAX_TRACE_DEPTH = 3
FLAG_DETERMINISTIC = 1
FLAG_DISTORTION = 2
FLAG_SH_HALF = 4

_FP = C.c_void_p


class DstParams(C.Structure):
    """Field-for-field mirror of `DstParams` in include/dst_api.h."""
    _fields_ = (
        [(n, C.c_int32) for n in ("P", "H", "W", "D", "M", "aux", "mtd_alloc", "max_trace_depth", "training",
                                  "start_from_first")]
        + [("specular_threshold", C.c_float), ("scale_modifier", C.c_float)]
        + [(n, _FP) for n in ("ray_o", "ray_d", "vertices", "background", "means3D", "shs", "colors_precomp",
                              "others_precomp", "opacities", "scales", "rotations")]
        + [(n, _FP) for n in ("out_rgb", "out_dpt", "out_acc", "out_norm", "out_dist", "out_aux", "mid_val",
                              "a_weights", "counters", "hit_record")]
        + [("hit_record_blocks", C.c_uint32), ("flags", C.c_uint32), ("det_workspace", _FP), ("grad_rows", _FP)]
        + [(n, _FP) for n in ("dL_drgb", "dL_ddpt", "dL_dacc", "dL_ddist", "dL_dnorm", "dL_daux")]
        + [(n, _FP) for n in ("dL_dray_o", "dL_dray_d", "dL_dmeans3D", "dL_dgrads3D", "dL_dshs", "dL_dcolors",
                              "dL_dothers", "dL_dopacities", "dL_dscales", "dL_drotations")]
        + [("shs_half", _FP), ("grad_touched", _FP), ("hit_record_asked", _FP), ("dist_channels", C.c_int32),
           ("reserved", C.c_int32), ("scratch", _FP)]
    )


class DstAccelInfo(C.Structure):
    _fields_ = [("n_surfels", C.c_uint32), ("n_internal", C.c_uint32), ("root", C.c_uint32),
                ("node_bytes", C.c_uint32), ("leaf_bytes", C.c_uint32), ("scene_lo", C.c_float * 3),
                ("scene_hi", C.c_float * 3), ("max_abs", C.c_float), ("builds", C.c_uint32), ("refits", C.c_uint32),
                ("key_levels", C.c_uint32), ("agglomerated", C.c_uint32), ("depth", C.c_uint32)]


class DstTraceInfo(C.Structure):
    _fields_ = [("handover_mode", C.c_uint32), ("handover_steps", C.c_uint32), ("handover_capacity", C.c_uint32),
                ("small_quads", C.c_uint32), ("handover_active", C.c_uint32), ("det_out_of_range", C.c_uint32),
                ("tiles_handed_over", C.c_uint64)]


HANDOVER_OFF, HANDOVER_AUTO, HANDOVER_ALWAYS = 0, 1, 2


EXPORTS = ("dst_create", "dst_destroy", "dst_build_accel", "dst_trace_forward", "dst_trace_backward",
           "dst_last_error", "dst_accel_info", "dst_accel_download", "dst_version", "dst_sizeof_params",
           "dst_hit_record_layout", "dst_refit_accel_static", "dst_refit_from_surfels",
           "dst_det_workspace_words", "dst_trace_scratch_bytes",
           "dst_trace_scratch_needed", "dst_pack_sh_half", "dst_trace_info", "dst_set_handover", "dst_det_out_of_range")

_lib = None


def load_library():
    """Load libdst.so (once) and declare its prototypes.  Raises if the library is absent or stale."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise ImportError("diff_surfel_tracing: %s is missing; build it with `make -C csrc` (hipcc, gfx950). "
                          "There is no CPU or PyTorch fallback." % LIB_PATH)
    L = C.CDLL(LIB_PATH)
    L.dst_create.restype = C.c_void_p
    L.dst_create.argtypes = []
    L.dst_destroy.restype = None
    L.dst_destroy.argtypes = [C.c_void_p]
    L.dst_build_accel.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p, C.c_uint32, C.c_int, C.c_void_p]
    L.dst_refit_accel_static.argtypes = [C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p]
    L.dst_refit_from_surfels.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_uint32, C.c_void_p,
                                         C.c_void_p]
    L.dst_trace_forward.argtypes = [C.c_void_p, C.POINTER(DstParams), C.c_void_p]
    L.dst_trace_backward.argtypes = [C.c_void_p, C.POINTER(DstParams), C.c_void_p]
    L.dst_last_error.restype = C.c_char_p
    L.dst_last_error.argtypes = [C.c_void_p]
    L.dst_accel_info.argtypes = [C.c_void_p, C.POINTER(DstAccelInfo)]
    L.dst_accel_download.argtypes = [C.c_void_p] * 7
    L.dst_trace_info.argtypes = [C.c_void_p, C.POINTER(DstTraceInfo)]
    L.dst_det_out_of_range.argtypes = [C.c_void_p, C.POINTER(C.c_uint32), C.c_void_p]
    L.dst_set_handover.argtypes = [C.c_void_p, C.c_int, C.c_uint32]
    L.dst_det_workspace_words.restype = C.c_uint64
    L.dst_det_workspace_words.argtypes = [C.c_int32, C.c_int32, C.c_int]
    L.dst_trace_scratch_bytes.restype = C.c_uint64
    L.dst_trace_scratch_bytes.argtypes = [C.c_int32, C.c_int32, C.c_int32]
    L.dst_trace_scratch_needed.restype = C.c_uint64
    L.dst_trace_scratch_needed.argtypes = [C.c_void_p, C.POINTER(DstParams)]
    L.dst_pack_sh_half.argtypes = [C.c_void_p, C.c_void_p, C.c_uint64, C.c_void_p]
    L.dst_version.restype = C.c_char_p
    L.dst_sizeof_params.restype = C.c_size_t
    L.dst_hit_record_layout.restype = C.c_uint64
    L.dst_hit_record_layout.argtypes = [C.c_int32, C.c_int32, C.c_int32, C.c_uint32, C.POINTER(C.c_uint64),
                                        C.POINTER(C.c_uint32)]
    if L.dst_sizeof_params() != C.sizeof(DstParams):
        raise ImportError("diff_surfel_tracing: DstParams layout mismatch between _C.py and libdst.so")
    _lib = L
    return L


_streams = {}


def _current_stream():
    """torch.cuda.current_stream(), from a small cache of the objects (building one costs more than a launch)."""
    key = torch._C._cuda_getCurrentStream(torch._C._cuda_getDevice())
    s = _streams.get(key)
    if s is None:
        if len(_streams) >= 64:
            _streams.clear()
        s = _streams[key] = torch.cuda.Stream(stream_id=key[0], device_index=key[1], device_type=key[2])
    return s


def _stream():
    return C.c_void_p(torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice()))


def _check(ctx, rc):
    if rc != 0:
        msg = load_library().dst_last_error(ctx.handle)
        raise RuntimeError((msg or b"unknown error").decode() + " (status %d)" % rc)


def _cuda_f32(t, name):
    """The launcher's tensor contract: CUDA, fp32, contiguous (reference trace_surfels.cpp:23-24,252-277)."""
    if not isinstance(t, torch.Tensor):
        raise RuntimeError("%s must be a tensor" % name)
    if not t.is_cuda:
        raise RuntimeError("%s must be a CUDA tensor" % name)
    if t.dtype != torch.float32:
        t = t.float()
    return t if t.is_contiguous() else t.contiguous()


def _ptr(t):
    return None if t is None or t.numel() == 0 else t.data_ptr()


class HitRecord:
    """Device buffer in which a forward trace stores its per-chunk hit buffers so that the backward trace can
    replay them instead of walking the BVH again (see `hit_record` in include/dst_api.h).  `storage` is a
    caller- or pool-owned int64 tensor that is at least `words_needed(...)` long."""

    _layouts = {}   # (H, W, mtd_alloc) -> (header words, waves, words without blocks, words of a block)
    _slots = []     # free words of pinned host memory for the request counts (note_request)
    _late = []      # words given up before their copy had come: looked at again when new ones are needed

    @classmethod
    def layout(cls, H, W, mtd_alloc, blocks_per_wave):
        """(words of the whole buffer, header words to be zeroed, blocks, waves) for an (H,W) ray grid."""
        known = cls._layouts.get((H, W, mtd_alloc))
        if known is None:
            header, waves = C.c_uint64(0), C.c_uint32(0)
            lib = load_library()
            words = lib.dst_hit_record_layout(H, W, mtd_alloc, 0, C.byref(header), C.byref(waves))
            per_block = lib.dst_hit_record_layout(H, W, mtd_alloc, 1, None, None) - words
            if len(cls._layouts) >= 256:
                cls._layouts.clear()
            known = cls._layouts[(H, W, mtd_alloc)] = (int(header.value), max(1, waves.value), int(words), int(per_block))
        header, n_waves, bare, per_block = known
        blocks = max(1, int(n_waves * blocks_per_wave) + 1)
        return (bare + blocks * per_block if per_block else 0), header, blocks, n_waves

    def __init__(self, H, W, mtd_alloc, blocks_per_wave, device, storage=None):
        words, header, self.blocks, self.n_waves = self.layout(H, W, mtd_alloc, blocks_per_wave)
        if storage is None:
            storage = torch.empty(words, dtype=torch.int64, device=device)
        elif storage.numel() < words or storage.dtype != torch.int64 or not storage.is_cuda:
            raise RuntimeError("hit record storage must be a CUDA int64 tensor of at least %d elements" % words)
        self.words = storage
        self.words[:header].zero_()
        self._slot = None          # (numpy view, index, address) of a pinned word
        self._slot_stream = None

    def note_request(self):
        """Address of a pinned host word that the forward trace about to be launched copies word 0 (the blocks it asked
        for) to, stream-ordered and without anybody waiting; `asked()` reads it once the copy has happened."""
        if self._slot is None:
            try:
                self._slot = HitRecord._slots.pop()
            except IndexError:   # pinned memory by the page: a few hundred words at a time
                late, HitRecord._late = HitRecord._late, []
                HitRecord._slots.extend(s for s in late if s[0][s[1]] != -1)
                HitRecord._late.extend(s for s in late if s[0][s[1]] == -1)
                page = torch.empty(256, dtype=torch.int64, pin_memory=True)
                view, at = page.numpy(), page.data_ptr()
                HitRecord._slots.extend((view, k, at + 8 * k, page) for k in range(1, 256))
                self._slot = (view, 0, at, page)
        self._slot[0][self._slot[1]] = -1
        self._slot_stream = _current_stream()
        return self._slot[2]

    def __del__(self):
        # a word whose copy may still be under way is not handed to anybody else
        slot, self._slot = getattr(self, "_slot", None), None
        if slot is not None:
            (HitRecord._late if slot[0][slot[1]] == -1 else HitRecord._slots).append(slot)

    def asked(self, wait=False):
        """Blocks requested by the forward trace, or None while that is not known yet (never waits unless told to)."""
        if self._slot is None:
            return int(self.words[0].item()) if wait else None
        view, k = self._slot[:2]
        if view[k] == -1:
            if not wait:
                return None
            self._slot_stream.synchronize()
        return int(view[k])

    def requested_blocks(self):
        """Blocks the forward trace asked for (waits for it to finish)."""
        return self.asked(wait=True)

    def complete(self):
        return self.requested_blocks() <= self.blocks

    def broken_chains(self):
        """Chains a replaying backward trace found broken (waits); 0 for every record a forward trace wrote."""
        return int(self.words[1].item())


class OptiXStateWrapper:
    """Owner of the acceleration structure; keeps the reference's class name (ext.cpp:8) so callers need not
    change.  `pkg_dir` was where the reference looked for its PTX files and is ignored.

    Also owns the hit-record buffers of the autograd path: a small pool that forward calls draw from and
    backward calls return to (no allocation per call once warm), bounded by `record_max_bytes` per record and
    `record_pool_max_bytes` for the free storages together; a record that would be larger, or whose allocation
    fails, is not made and the backward pass walks the BVH again (`records_skipped` counts those calls, the first
    one warns)."""

    _pool_lock = threading.Lock()   # of the pools of all contexts: held for a few list operations, and nothing waits inside

    RECORD_POOL_SIZE = 4
    RECORD_FIRST_BLOCKS = 5.0   # blocks per wave and bounce before a forward trace has said what it needs
    RECORD_HEADROOM = 1.08      # a record is sized this much above the largest request seen so far

    def __init__(self, pkg_dir=None):
        lib = load_library()
        if not torch.cuda.is_available():
            raise RuntimeError("diff_surfel_tracing needs a GPU: no HIP device is visible")
        self.handle = lib.dst_create()
        if not self.handle:
            raise RuntimeError("dst_create failed: no usable HIP device")
        self.device = torch.cuda.current_device()
        self.num_surfels = 0
        self.record_blocks_per_wave = None  # sizing estimate for hit records: largest request seen, with headroom
        self.record_max_bytes = 32 << 30    # no record larger than this is made (backward then re-traces); a 4K image
                                            # of the 1M-surfel room scene needs 13 GB, of the card's 288
        self.record_pool_max_bytes = 48 << 30   # free storages kept for reuse, all together
        self.records_skipped = 0            # forward calls that made no record because of the two limits above
        self.deterministic = False          # True: a_weights and per-surfel gradients are bitwise reproducible
        self.deterministic_check = True     # with `deterministic`: warn after a backward trace whose sums left the range
        self._det_out_of_range = 0          # the library's count when last looked at
        self.gradient_rows = True           # backward sums per-surfel gradients in one row per surfel first (faster)
        self.distortion = False             # True: the dist output carries the 2DGS depth distortion (else zeros)
        self.sh_half = False                # True: the traces read the SH coefficients from a binary16 copy
        self._record_pool = []              # free storages (int64 tensors)
        self._record_events = {}            # id(storage) -> event recorded when the storage came back
        self._record_fixed = False          # True: only caller-provided storage is used, nothing is allocated
        self._record_watch = []             # records whose request count has not been read yet
        self._row_pool = []                 # (rows, marks, stream, event): per-surfel sums of backward calls, all zero
        self.row_pool_max_bytes = 8 << 30   # of them kept for reuse; 2M surfels, aux 4: 0.55 GB a pair, deterministic 1.1

    # ---- hit-record storage ---------------------------------------------------------------------------
    def use_record_storage(self, storage):
        """Use this caller-owned int64 CUDA tensor (and nothing else) for hit records; None returns to the
        pool.  One record is live at a time with a fixed storage: a forward call that finds it taken, or too
        small (HitRecord.layout gives the size), makes no record."""
        self._record_pool = [] if storage is None else [storage]
        self._record_fixed = storage is not None

    def update_record_estimate(self):
        """Raise the sizing estimate from records whose forward trace has finished.  Never waits, except in the
        deterministic mode: whether a backward trace replays a complete record or walks the BVH again changes its
        gradients in the last bit (the two kernels contract their gradient algebra differently), so there the
        sequence of record sizes must not depend on timing."""
        still = []
        for rec in self._record_watch:
            asked = rec.asked(wait=self.deterministic)
            if asked is None:
                still.append(rec)
            else:
                self.record_blocks_per_wave = max(self.record_blocks_per_wave or 0.0,
                                                  self.RECORD_HEADROOM * asked / rec.n_waves)
        self._record_watch = still[-8:]

    def acquire_record(self, H, W, mtd_alloc, device, max_trace_depth=None):
        """A record for an (H,W) grid traced with `mtd_alloc` mid_val slots - 1, or None.  Sized from what earlier
        forward traces asked for (with a little headroom); before any has finished, for RECORD_FIRST_BLOCKS blocks
        per wave and bounce actually traced (`max_trace_depth` + 1; `mtd_alloc` + 1 if that is not given): every bounce
        of a path opens at least one block per wave, so a multi-bounce run can replay from its first step."""
        self.update_record_estimate()
        per_wave = self.record_blocks_per_wave
        if per_wave is None:
            bounces = (mtd_alloc if max_trace_depth is None else max_trace_depth) + 1
            per_wave = self.RECORD_FIRST_BLOCKS * bounces
        words = HitRecord.layout(H, W, mtd_alloc, per_wave)[0]
        if 8 * words > self.record_max_bytes:
            self.records_skipped += 1
            if self.records_skipped == 1:
                warnings.warn("diff_surfel_tracing: a hit record for this %dx%d trace would take %.1f GiB (limit "
                              "record_max_bytes = %.1f GiB); backward passes walk the BVH again instead of replaying"
                              % (H, W, 8 * words / 2 ** 30, self.record_max_bytes / 2 ** 30))
            return None
        device = torch.device(device)
        if device.index is None:
            device = torch.device(device.type, torch.cuda.current_device())
        # (what a graph being captured writes must belong to that graph: a pooled storage would go on to other calls)
        captured = not self._record_fixed and torch.cuda.is_current_stream_capturing()
        with self._pool_lock:
            fit = [] if captured else [t for t in self._record_pool if t.numel() >= words and t.device == device]
            storage = min(fit, key=lambda t: t.numel()) if fit else None
            self._record_pool = [t for t in self._record_pool if t is not storage]
            done = self._record_events.pop(id(storage), None)
        if storage is not None:
            # the backward trace that last read this storage may still be running on another stream
            if done is not None:
                now = _current_stream()
                now.wait_event(done)
                storage.record_stream(now)   # (its allocator knows the stream it was made on, and no other)
        elif self._record_fixed:
            return None
        else:
            try:
                storage = torch.empty(words, dtype=torch.int64, device=device)
            except torch.OutOfMemoryError:
                self.records_skipped += 1
                return None
        return HitRecord(H, W, mtd_alloc, per_wave, device, storage=storage)

    def release_record(self, rec):
        """Back to the pool.  The storage's last reader (a backward trace just enqueued on the current stream) is
        marked with an event that the next user waits for, whatever stream that user runs on."""
        if rec is None or rec.words is None:
            return
        words, rec.words = rec.words, None
        done = None
        if words.is_cuda:
            if not self._record_fixed and torch.cuda.is_current_stream_capturing():
                return
            done, now = torch.cuda.Event(), _current_stream()
            done.record(now)
            words.record_stream(now)
        with self._pool_lock:
            pool = self._record_pool + [words]
            if done is not None:
                self._record_events[id(words)] = done
            while not self._record_fixed and len(pool) > 1 and (
                    len(pool) > self.RECORD_POOL_SIZE or 8 * sum(t.numel() for t in pool) > self.record_pool_max_bytes):
                smallest = min(pool, key=lambda t: t.numel())
                pool = [t for t in pool if t is not smallest]   # (list.remove() would compare tensors element-wise)
                self._record_events.pop(id(smallest), None)
            self._record_pool = pool

    # ---- per-surfel sums of the backward traces -------------------------------------------------------
    ROW_POOL_SIZE = 2

    def acquire_rows(self, P, words, dtype, device):
        """A zeroed buffer of at least `words` sums and one of at least P marks (DstParams.grad_touched).  The closing
        kernel of a backward trace leaves both zero, so they are filled once, not per call; at most ROW_POOL_SIZE pairs
        and `row_pool_max_bytes` are kept between calls.  A pair that this call's scene or mode has no use for is let
        go: the one made in its place is kept."""
        found, now = None, _current_stream()
        if not torch.cuda.is_current_stream_capturing():   # (a captured fill has not run yet)
            with self._pool_lock:
                fits = [p for p in self._row_pool if p[0].dtype == dtype and p[0].numel() >= words and
                        p[1].numel() >= P and p[0].device == device]
                found = next((p for p in fits if p[2] is now), fits[0] if fits else None)   # (nothing to wait for)
                self._row_pool = [p for p in fits if p is not found]
        if found is None:
            return torch.zeros(words, dtype=dtype, device=device), torch.zeros(P, dtype=torch.uint8, device=device)
        rows, marks, stream, event = found
        if stream is not now:   # its last user may still be running there, and when the pair is dropped, this one
            now.wait_event(event)
            rows.record_stream(now)
            marks.record_stream(now)
        return rows, marks

    def release_rows(self, rows, marks):
        """Back to the pool, behind a backward trace that has been launched (after a failed call they are dropped)."""
        size = rows.numel() * rows.element_size() + marks.numel()
        if torch.cuda.is_current_stream_capturing() or size > self.row_pool_max_bytes:
            return
        stream, event = _current_stream(), torch.cuda.Event()
        event.record(stream)
        with self._pool_lock:
            kept = [(rows, marks, stream, event)]
            for p in self._row_pool[:self.ROW_POOL_SIZE - 1]:
                size += p[0].numel() * p[0].element_size() + p[1].numel()
                if size <= self.row_pool_max_bytes:
                    kept.append(p)
            self._row_pool = kept

    def release_memory(self):
        """Give back what is kept between calls for reuse (hit records, rows of gradient sums; not a caller's own record
        storage).  The next training step allocates again."""
        self.update_record_estimate()
        with self._pool_lock:
            self._row_pool, self._record_watch = [], []   # (a record nobody traced backward through is held there alone)
            if not self._record_fixed:
                self._record_pool, self._record_events = [], {}

    def accel_info(self):
        info = DstAccelInfo()
        _check(self, load_library().dst_accel_info(self.handle, C.byref(info)))
        return info

    def trace_info(self):
        """Tile hand-over of the forward trace (include/dst_api.h): mode, step limit, list capacity, the small quads the
        last build counted, whether the next forward trace can hand over, tiles handed over so far; and the number of
        sums the deterministic mode has found out of its fixed-point range.  Waits."""
        info = DstTraceInfo()
        _check(self, load_library().dst_trace_info(self.handle, C.byref(info)))
        return info

    def check_deterministic_range(self):
        """Warn if sums of the deterministic mode have left their fixed-point range since the last look (gradients
        beyond about 6.7e7 for scales, rotations and means, 4.2e6 for the rest: they come out clamped or wrapped).
        Waits for the current stream.  Returns the number of such sums."""
        count = C.c_uint32(0)
        _check(self, load_library().dst_det_out_of_range(self.handle, C.byref(count), _stream()))
        seen = count.value
        new, self._det_out_of_range = (seen - self._det_out_of_range) & 0xFFFFFFFF, seen
        if new:
            warnings.warn("deterministic mode: %d per-surfel sums left the fixed-point range and are wrong; scale the "
                          "loss down or trace without the mode" % new, RuntimeWarning, stacklevel=3)
        return new

    def set_handover(self, mode, steps=0):
        """HANDOVER_OFF / HANDOVER_AUTO (only for scenes with many quads far smaller than the scene) / HANDOVER_ALWAYS;
        `steps`: what a tile's first walk may take before its rays are walked one by one (0: unchanged)."""
        _check(self, load_library().dst_set_handover(self.handle, int(mode), int(steps)))

    def __del__(self):
        h, self.handle = getattr(self, "handle", None), None
        if h and _lib is not None:
            _lib.dst_destroy(h)


def build_acceleration_structure(ctx, vertices, triangles, rebuild):
    """Reference BuildAccelerationStructure (trace_surfels.cpp:36-159)."""
    if vertices.dim() != 2 or vertices.size(1) != 3:
        raise RuntimeError("vertices must have dimensions (num_vertices, 3)")
    if triangles.dim() != 2 or triangles.size(1) != 3:
        raise RuntimeError("triangles must have dimensions (num_triangles, 3)")
    v = _cuda_f32(vertices, "vertices")
    if not triangles.is_cuda:
        raise RuntimeError("triangles must be a CUDA tensor")
    f = triangles.to(torch.int32).contiguous()
    rc = load_library().dst_build_accel(ctx.handle, v.data_ptr(), v.size(0), f.data_ptr(), f.size(0),
                                        int(bool(rebuild)), _stream())
    _check(ctx, rc)
    ctx.num_surfels = f.size(0) // 2


def refit_from_surfels(ctx, means3D, scales, rotations, vertices_out=None):
    """Refit the structure straight from the surfel parameters (dst_refit_from_surfels in include/dst_api.h) and
    return the quad corners (4P,3) the trace calls take as `vertices`, written by the same kernel.  No counterpart
    in the reference, whose callers regenerate the quads with tensor operations and then call
    build_acceleration_structure(v, f, rebuild=False)."""
    m, s, q = _cuda_f32(means3D, "means3D"), _cuda_f32(scales, "scales"), _cuda_f32(rotations, "rotations")
    P = m.size(0)
    if m.dim() != 2 or m.size(1) != 3 or tuple(s.shape) != (P, 2) or tuple(q.shape) != (P, 4):
        raise RuntimeError("means3D (P,3), scales (P,2) and rotations (P,4) are required")
    if vertices_out is None:
        vertices_out = torch.empty((4 * P, 3), dtype=torch.float32, device=m.device)
    elif (not vertices_out.is_cuda or vertices_out.dtype != torch.float32 or not vertices_out.is_contiguous()
          or vertices_out.numel() != 12 * P):
        raise RuntimeError("vertices_out must be a contiguous CUDA float32 tensor of shape (4P,3)")
    rc = load_library().dst_refit_from_surfels(ctx.handle, m.data_ptr(), s.data_ptr(), q.data_ptr(), P,
                                               vertices_out.data_ptr(), _stream())
    _check(ctx, rc)
    return vertices_out


def pack_sh_half(shs):
    """binary16 copy of an fp32 CUDA tensor of SH coefficients (dst_pack_sh_half: round to nearest even)."""
    shs = _cuda_f32(shs, "shs")
    out = torch.empty(shs.shape, dtype=torch.float16, device=shs.device)
    rc = load_library().dst_pack_sh_half(shs.data_ptr(), out.data_ptr(), shs.numel(), _stream())
    if rc != 0:
        raise RuntimeError("dst_pack_sh_half failed (status %d)" % rc)
    return out


def _use_sh_half(ctx, p, keep):
    """With `ctx.sh_half` set and SH coefficients given: pack them and point the launch parameters at the copy."""
    if getattr(ctx, "sh_half", False) and keep["shs"].numel() != 0:
        keep["shs_half"] = pack_sh_half(keep["shs"])
        p.shs_half = keep["shs_half"].data_ptr()
        p.flags |= FLAG_SH_HALF


def _common_params(ray_o, ray_d, vertices, background, means3D, shs, degree, colors_precomp, others_precomp,
                   opacities, scales, scale_modifier, rotations, max_trace_depth, specular_threshold,
                   start_from_first):
    if means3D.dim() != 2 or means3D.size(1) != 3:
        raise RuntimeError("means3D must have dimensions (num_points, 3)")
    # (one look at each of eleven tensors, and their addresses with it)
    p, t, f32, Tensor = DstParams(), {}, torch.float32, torch.Tensor
    for name, x in (("ray_o", ray_o), ("ray_d", ray_d), ("vertices", vertices), ("background", background),
                    ("means3D", means3D), ("shs", shs), ("colors_precomp", colors_precomp),
                    ("others_precomp", others_precomp), ("opacities", opacities), ("scales", scales),
                    ("rotations", rotations)):
        if not (isinstance(x, Tensor) and x.is_cuda and x.dtype is f32 and x.is_contiguous()):
            x = _cuda_f32(x, name)
        t[name] = x
        if x.numel() != 0:
            setattr(p, name, x.data_ptr())
    if t["ray_o"].dim() != 3 or t["ray_o"].size(2) != 3 or t["ray_d"].shape != t["ray_o"].shape:
        raise RuntimeError("ray_o and ray_d must have the same dimensions (H, W, 3) or (B, P, 3)")
    if t["scales"].numel() == 0 or t["rotations"].numel() == 0:
        raise RuntimeError("scales and rotations are required (a precomputed 3D covariance is not consumed by "
                           "the tracer)")
    p.P, p.H, p.W = means3D.size(0), t["ray_o"].size(0), t["ray_o"].size(1)
    p.D = int(degree)
    p.M = t["shs"].size(1) if p.shs else 0
    p.aux = t["others_precomp"].size(1) if p.others_precomp else DEFAULT_AUX_CHANNELS
    p.max_trace_depth = int(max_trace_depth)
    p.mtd_alloc = max(DEFAULT_MAX_TRACE_DEPTH, p.max_trace_depth)
    p.start_from_first = int(bool(start_from_first))
    p.specular_threshold = float(specular_threshold)
    p.scale_modifier = float(scale_modifier)
    return p, t


_scratch_bytes = {}   # (P, H, W) -> dst_trace_scratch_bytes


def _scratch(p, keep):
    """The forward call's scratch memory (DstParams.scratch): of the current stream's, given back when the call is done."""
    key = (p.P, p.H, p.W)
    size = _scratch_bytes.get(key)
    if size is None:
        if len(_scratch_bytes) >= 256:
            _scratch_bytes.clear()
        size = _scratch_bytes[key] = load_library().dst_trace_scratch_bytes(*key)
    if size != 0:
        size = load_library().dst_trace_scratch_needed(keep["context"].handle, C.byref(p))
    if size == 0:
        return
    try:
        keep["scratch"] = torch.empty(size, dtype=torch.uint8, device=keep["means3D"].device)
    except torch.OutOfMemoryError:   # (the same results without it)
        return
    p.scratch = keep["scratch"].data_ptr()


def trace_surfels(ctx, training, start_from_first, ray_o, ray_d, vertices, background, means3D, shs, degree,
                  colors_precomp, others_precomp, opacities, scales, scale_modifier, rotations, transMat_precomp,
                  viewmatrix, projmatrix, campos, prefiltered, debug, max_trace_depth, specular_threshold,
                  counters=None, events=None, hit_record=None, dist_channels=3):
    """Reference TraceSurfelsCUDA (trace_surfels.cpp:162-304): returns
    (out_rgb, out_dpt, out_acc, out_norm, out_dist, out_aux, mid_val, a_weights or None).
    Extras for measurement: `counters` (2 int64 on the device) receives the evaluated / composited hit totals;
    `events` (two torch.cuda.Event) are recorded on the launch stream right around the kernel launch;
    `hit_record` (a HitRecord) receives the hit buffers for a later replay by trace_surfels_backward.
    `dist_channels`: 3 as the reference's launcher returns them, 1 for the distortion alone."""
    p, keep = _common_params(ray_o, ray_d, vertices, background, means3D, shs, degree, colors_precomp,
                             others_precomp, opacities, scales, scale_modifier, rotations, max_trace_depth,
                             specular_threshold, start_from_first)
    H, W, P, dev = p.H, p.W, p.P, means3D.device
    mid_ch = (14 + p.aux) * (p.mtd_alloc + 1)
    p.dist_channels = int(dist_channels)
    new = keep["means3D"].new_empty   # (the kernel writes every element)
    out_rgb, out_dpt, out_acc = new((H, W, NUM_CHANNELS)), new((H, W, 1)), new((H, W, 1))
    out_norm, out_dist, out_aux, mid_val = (new((H, W, 3)), new((H, W, p.dist_channels)), new((H, W, p.aux)),
                                            new((H, W, mid_ch)))
    a_weights = keep["means3D"].new_zeros((P, 1)) if training else None
    p.training = int(bool(training))
    p.out_rgb, p.out_dpt, p.out_acc = out_rgb.data_ptr(), out_dpt.data_ptr(), out_acc.data_ptr()
    p.out_norm, p.out_dist, p.out_aux = out_norm.data_ptr(), out_dist.data_ptr(), out_aux.data_ptr()
    p.mid_val = mid_val.data_ptr()
    p.a_weights = _ptr(a_weights)
    p.counters = _ptr(counters)
    # (a captured copy of the request count would be made on every replay, long after the word has another owner)
    watch = hit_record is not None and not torch.cuda.is_current_stream_capturing()
    if hit_record is not None:
        p.hit_record, p.hit_record_blocks = hit_record.words.data_ptr(), hit_record.blocks
        if watch:
            p.hit_record_asked = hit_record.note_request()
    det_ws = None
    if getattr(ctx, "deterministic", False) and training:
        det_ws = torch.zeros(load_library().dst_det_workspace_words(P, p.aux, 0), dtype=torch.int64, device=dev)
        p.flags, p.det_workspace = FLAG_DETERMINISTIC, det_ws.data_ptr()
    if getattr(ctx, "distortion", False):
        p.flags |= FLAG_DISTORTION
    _use_sh_half(ctx, p, keep)
    if (p.flags == 0 or H < 8) and _scratch_bytes.get((P, H, W)) != 0:   # (images' kernels with the rare options take none)
        keep["context"] = ctx
        _scratch(p, keep)
    if events is not None:
        events[0].record()
    _check(ctx, load_library().dst_trace_forward(ctx.handle, C.byref(p), _stream()))
    if events is not None:
        events[1].record()
    if watch:
        ctx._record_watch.append(hit_record)
    del keep
    return out_rgb, out_dpt, out_acc, out_norm, out_dist, out_aux, mid_val, a_weights


def trace_surfels_backward(ctx, start_from_first, ray_o, ray_d, vertices, background, means3D, shs, degree,
                           colors_precomp, others_precomp, opacities, scales, scale_modifier, rotations,
                           transMat_precomp, viewmatrix, projmatrix, campos, prefiltered, debug, max_trace_depth,
                           specular_threshold, out_rgb, out_dpt, out_acc, out_norm, out_dist, out_aux, mid_val,
                           dL_dout_rgb, dL_dout_dpt, dL_dout_acc, dL_dout_norm, dL_dout_dist, dL_dout_aux,
                           events=None, hit_record=None, counters=None, wanted_only=False):
    """Reference TraceSurfelsBackwardCUDA (trace_surfels.cpp:307-464): returns (dL_dray_o, dL_dray_d, dL_dmeans3D,
    dL_dgrads3D, dL_dgrads3D_abs, dL_dshs, dL_dcolors, dL_dothers, dL_dopacities, dL_dscales, dL_drotations,
    dL_dtransMat_precomp).  `wanted_only`: None for the gradients of inputs that were not given, and for the two that are
    always zero."""
    p, keep = _common_params(ray_o, ray_d, vertices, background, means3D, shs, degree, colors_precomp,
                             others_precomp, opacities, scales, scale_modifier, rotations, max_trace_depth,
                             specular_threshold, start_from_first)
    H, W, P, dev = p.H, p.W, p.P, means3D.device
    saved = [_cuda_f32(x, n) for x, n in ((out_rgb, "out_rgb"), (out_dpt, "out_dpt"), (out_acc, "out_acc"),
                                          (out_norm, "out_norm"), (out_dist, "out_dist"), (out_aux, "out_aux"),
                                          (mid_val, "mid_val"))]
    mid_ch = (14 + p.aux) * (p.mtd_alloc + 1)
    if saved[6].numel() != H * W * mid_ch or saved[5].numel() != H * W * p.aux:
        raise RuntimeError("mid_val / out_aux do not match the settings they were traced with")
    p.out_rgb, p.out_dpt, p.out_acc, p.out_norm, p.out_dist, p.out_aux, p.mid_val = [x.data_ptr() for x in saved]
    ups = [_cuda_f32(x, n) for x, n in ((dL_dout_rgb, "dL_dout_rgb"), (dL_dout_dpt, "dL_dout_dpt"),
                                        (dL_dout_acc, "dL_dout_acc"), (dL_dout_norm, "dL_dout_norm"),
                                        (dL_dout_dist, "dL_dout_dist"), (dL_dout_aux, "dL_dout_aux"))]
    want = (3, 1, 1, 3, None, p.aux)
    for x, ch, n in zip(ups, want, ("rgb", "dpt", "acc", "norm", "dist", "aux")):
        if ch is not None and x.numel() != H * W * ch:
            raise RuntimeError("upstream gradient of %s has the wrong size" % n)
    p.dL_drgb, p.dL_ddpt, p.dL_dacc, p.dL_dnorm, p.dL_ddist, p.dL_daux = (
        ups[0].data_ptr(), ups[1].data_ptr(), ups[2].data_ptr(), ups[3].data_ptr(), _ptr(ups[4]), ups[5].data_ptr())
    det = bool(getattr(ctx, "deterministic", False))
    # The per-surfel gradients are summed in a buffer of their own first (a surfel's columns side by side; fixed point in
    # the deterministic mode), and a closing kernel writes them to the tensors; without it they are added to the tensors.
    by_rows = det or getattr(ctx, "gradient_rows", True)
    like = keep["means3D"]
    new = like.new_empty if by_rows else like.new_zeros
    dL_dray_o, dL_dray_d = like.new_empty((H, W, 3)), like.new_empty((H, W, 3))
    dL_dmeans3D, dL_dgrads3D = new((P, 3)), new((P, 3))
    dL_dshs = new((P, p.M, 3))
    lean = wanted_only and by_rows
    dL_dcolors = None if lean and not p.colors_precomp else new((P, NUM_CHANNELS))
    dL_dothers = None if lean and not p.others_precomp else new((P, p.aux))
    dL_dopacities, dL_dscales, dL_drotations = new((P, 1)), new((P, 2)), new((P, 4))
    dL_dgrads3D_abs = None if wanted_only else like.new_zeros((P, 3))
    dL_dtransMat = None if wanted_only else like.new_zeros((P, 9))
    p.dL_dray_o, p.dL_dray_d = dL_dray_o.data_ptr(), dL_dray_d.data_ptr()
    p.dL_dmeans3D, p.dL_dgrads3D, p.dL_dshs = dL_dmeans3D.data_ptr(), dL_dgrads3D.data_ptr(), _ptr(dL_dshs)
    p.dL_dcolors, p.dL_dothers = _ptr(dL_dcolors), _ptr(dL_dothers)
    p.dL_dopacities, p.dL_dscales, p.dL_drotations = (dL_dopacities.data_ptr(), dL_dscales.data_ptr(),
                                                      dL_drotations.data_ptr())
    if hit_record is not None:
        # the kernels decide on the device whether the record is complete (replay) or not (walk the BVH again):
        # nothing here waits for the forward trace
        p.hit_record, p.hit_record_blocks = hit_record.words.data_ptr(), hit_record.blocks
    p.counters = _ptr(counters)
    if by_rows:
        rows, marks = ctx.acquire_rows(P, load_library().dst_det_workspace_words(P, p.aux, 1),
                                       torch.int64 if det else torch.float32, like.device)
        p.grad_touched = marks.data_ptr()
        if det:
            p.flags, p.det_workspace = FLAG_DETERMINISTIC, rows.data_ptr()
        else:
            p.grad_rows = rows.data_ptr()
    if getattr(ctx, "sh_half", False) and keep["shs"].numel() != 0:
        # the backward trace reads fp32 coefficients: the values the forward trace used
        keep["shs"] = pack_sh_half(keep["shs"]).float()
        p.shs = keep["shs"].data_ptr()
    if events is not None:
        events[0].record()
    _check(ctx, load_library().dst_trace_backward(ctx.handle, C.byref(p), _stream()))
    if events is not None:
        events[1].record()
    if by_rows:
        ctx.release_rows(rows, marks)
    if p.flags & FLAG_DETERMINISTIC and getattr(ctx, "deterministic_check", False):
        ctx.check_deterministic_range()   # (the mode waits for the device elsewhere too: record sizes)
    del keep
    return (dL_dray_o, dL_dray_d, dL_dmeans3D, dL_dgrads3D, dL_dgrads3D_abs, dL_dshs, dL_dcolors, dL_dothers,
            dL_dopacities, dL_dscales, dL_drotations, dL_dtransMat)
