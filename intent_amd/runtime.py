"""HIP runtime behind a compiled artifact: binding, output allocation, launch.

Semantics follow the reference's GPU provider runtime
(python/intent/runtime/artifact.py:130-176, runtime/invocation.py:56-159,
runtime/gpu/program.py:68-124): the binder checks dtypes, ranks, shared
extents and strides against the public interface; ``run`` allocates declared
Out buffers with torch on the artifact's device; launches are asynchronous on
torch's current stream; ``infer_outputs`` builds outputs from shapes alone so
that torch fake tensors never touch data.
"""
from __future__ import annotations

from dataclasses import dataclass, field

from . import _native
from .definitions import KernelDefinition, Param, Scalar
from .interface import DTYPES, PublicInterface, ViewKind, torch_dtype


@dataclass(frozen=True)
class NativeObservation:
    """Facts of the latest launch, read without compiling or launching."""

    entry: str
    definition: str
    arch: str
    library: str
    constexprs: dict = field(default_factory=dict)
    kernel: str = ""  # the kernel variant the entry dispatched to


@dataclass(frozen=True)
class ConfigurationAssessment:
    entry: str
    eligible: bool
    reason: str


@dataclass(slots=True)
class Binding:
    views: dict
    env: dict
    outputs: tuple
    workspace: object = None


@dataclass(slots=True)
class _Layout:
    """What binding established for one combination of dtypes, devices, shapes and strides.

    Everything the checks of ``_bind`` derive from those alone: a call with the same
    combination needs only its addresses compared (``pairs``: the views of which one is
    writable, spans in bytes)."""

    env: dict
    names: tuple        # the supplied views, in argument order
    outputs: tuple      # allocated Out buffers: (name, shape, dtype)
    spans: tuple
    pairs: tuple
    workspace: int      # bytes, -1 without one
    scratch: int        # bytes of a launch's own scratch


MAX_LAYOUTS = 256  # layouts kept per artifact and calling form; the oldest go first


def _current_stream(device: int) -> int:
    import torch

    raw = getattr(torch._C, "_cuda_getCurrentRawStream", None)
    return raw(device) if raw is not None else torch.cuda.current_stream(device).cuda_stream


class HIPRuntime:
    def __init__(self, definition: KernelDefinition, device: int, constexprs: dict, arch: str):
        self.definition = definition
        self.device = device
        self.constexprs = constexprs
        self.arch = arch
        self._interface = definition.interface()
        self._workspace = None
        self._latest: tuple | None = None  # (entry, kernel name bytes) of the latest launch
        self._scalars = {p.name for p in definition.params if isinstance(p, Scalar)}
        self._writable = {p.name for p in definition.params if isinstance(p, Param) and p.access is not ViewKind.IN}
        self._supplied = tuple(p for p in definition.params if isinstance(p, Scalar) or p.access is not ViewKind.OUT)
        self._layouts: tuple[dict, dict] = ({}, {})  # by calling form: outputs allocated, outputs supplied
        self._home = None

    @property
    def interface(self) -> PublicInterface:
        return self._interface

    @property
    def observation(self) -> NativeObservation | None:
        if self._latest is None:
            return None
        entry, kernel = self._latest
        return NativeObservation(entry, self.definition.name, self.arch, str(_native.LIBRARY_PATH),
                                 dict(self.constexprs), kernel.decode("utf-8", "replace") if kernel else "")

    # ---- known layouts --------------------------------------------------------
    def _home_device(self):
        if self._home is None:
            import torch

            self._home = torch.device("cuda", self.device)
        return self._home

    def _layout_key(self, params: tuple, arguments: tuple):
        """Dtypes, devices, shapes and strides of the arguments; None unless all are plain tensors."""
        import torch

        key = []
        for p, a in zip(params, arguments):
            if p.name in self._scalars:
                continue
            if type(a) is not torch.Tensor and type(a) is not torch.nn.Parameter:
                return None
            if a.layout is not torch.strided:
                return None
            key += (a.dtype, a.device, a.shape, a.stride())
        return tuple(key)

    def rebind(self, arguments: tuple, supplied_outputs: bool) -> Binding | None:
        """The binding of a call whose layout has been bound before, or None (then ``_bind`` checks it)."""
        params = self.definition.params if supplied_outputs else self._supplied
        if len(arguments) != len(params):
            return None
        key = self._layout_key(params, arguments)
        known = self._layouts[supplied_outputs].get(key) if key is not None else None
        if known is None:
            return None
        env = known.env
        if self._scalars:
            env = dict(env)
            tensors = []
            for p, a in zip(params, arguments):
                if p.name in self._scalars:
                    env[p.name] = a
                else:
                    tensors.append(a)
        else:
            tensors = arguments
        if known.pairs:
            starts = [t.data_ptr() for t in tensors]
            for i, j in known.pairs:
                if starts[i] < starts[j] + known.spans[j] and starts[j] < starts[i] + known.spans[i]:
                    return None  # _bind names the overlap
        views = dict(zip(known.names, tensors))
        if known.outputs:
            import torch

            outputs = []
            for name, shape, dt in known.outputs:
                t = torch.empty(shape, dtype=dt, device=self._home_device())
                views[name] = t
                outputs.append(t)
            return Binding(views, env, tuple(outputs), self._buffer_of(known.workspace, known.scratch))
        outputs = ()
        if supplied_outputs:
            outputs = tuple(views[p.name] for p in params if p.name not in self._scalars and p.access is ViewKind.OUT)
        return Binding(views, env, outputs, self._buffer_of(known.workspace, known.scratch))

    def _remember(self, arguments: tuple, supplied_outputs: bool, binding: Binding, workspace: int, scratch: int) -> None:
        params = self.definition.params if supplied_outputs else self._supplied
        key = self._layout_key(params, arguments)
        if key is None:
            return
        views = [(p, a) for p, a in zip(params, arguments) if p.name not in self._scalars]
        spans = tuple(_span_bytes(t) for _, t in views)
        pairs = tuple((i, j) for i in range(len(views)) for j in range(i + 1, len(views))
                      if spans[i] and spans[j]
                      and (views[i][0].name in self._writable or views[j][0].name in self._writable))
        made = () if supplied_outputs else tuple((p.name, tuple(binding.views[p.name].shape), binding.views[p.name].dtype)
                                                 for p in self.definition.params
                                                 if p.name not in self._scalars and p.access is ViewKind.OUT)
        known = self._layouts[supplied_outputs]
        if len(known) >= MAX_LAYOUTS:
            for old in list(known)[:MAX_LAYOUTS // 2]:
                known.pop(old, None)
        known[key] = _Layout(dict(binding.env), tuple(p.name for p, _ in views), made, spans, pairs, workspace, scratch)

    # ---- binding ------------------------------------------------------------
    def _bind(self, arguments: tuple, explicit_outputs: tuple | None, abstract: bool = False) -> Binding:
        import torch

        d = self.definition
        params = d.params
        inputs = [p for p in params if isinstance(p, Scalar) or p.access is not ViewKind.OUT]
        outputs = [p for p in params if isinstance(p, Param) and p.access is ViewKind.OUT]
        if len(arguments) != len(inputs):
            raise TypeError(f"{d.name}: expected {len(inputs)} input arguments, got {len(arguments)}")
        env = dict(self.constexprs)
        views: dict = {}

        def observe(p: Param, t, supplied_by_caller: bool) -> None:
            if not isinstance(t, torch.Tensor):
                raise TypeError(f"{d.name}: {p.name} must be a torch.Tensor, got {type(t).__name__}")
            want = torch_dtype(DTYPES[p.dtype])
            if t.dtype != want:
                raise TypeError(f"{d.name}: {p.name} must have dtype {want}, got {t.dtype}")
            if t.dim() != len(p.dims):
                raise ValueError(f"{d.name}: {p.name} must have rank {len(p.dims)}, got {t.dim()}")
            for axis, dim in enumerate(p.dims):
                extent = int(t.shape[axis])
                if isinstance(dim, int):
                    if extent != dim:
                        raise ValueError(f"{d.name}: {p.name}.shape[{axis}] must be {dim}, got {extent}")
                elif isinstance(dim, str):
                    known = env.setdefault(dim, extent)
                    if known != extent:
                        raise ValueError(f"{d.name}: {p.name}.shape[{axis}] violates the declared interface "
                                         f"relation ({dim}={known}, got {extent})")
                else:
                    expected = int(dim(env))
                    if extent != expected:
                        raise ValueError(f"{d.name}: {p.name}.shape[{axis}] must be {expected}, got {extent}")
            if not abstract:
                self._check_layout(p, t)

        for p, value in zip(inputs, arguments):
            if isinstance(p, Scalar):
                env[p.name] = value
                continue
            observe(p, value, True)
            views[p.name] = value
        if d.check is not None:
            d.check(env)
        if explicit_outputs is None:
            outs = []
            device = next((v.device for v in views.values()), None)
            for p in outputs:
                shape = tuple(self._extent(p, dim, env) for dim in p.dims)
                t = torch.empty(shape, dtype=torch_dtype(DTYPES[p.dtype]), device=device)
                views[p.name] = t
                outs.append(t)
            outs = tuple(outs)
        else:
            if len(explicit_outputs) != len(outputs):
                raise TypeError(f"{d.name}: expected {len(outputs)} explicit output buffers, "
                                f"got {len(explicit_outputs)}")
            for p, t in zip(outputs, explicit_outputs):
                observe(p, t, True)
                views[p.name] = t
            outs = tuple(explicit_outputs)
        if not abstract:
            self._check_aliases(views)
        return Binding(views, env, outs)

    @staticmethod
    def _extent(p: Param, dim, env: dict) -> int:
        if isinstance(dim, int):
            return dim
        if isinstance(dim, str):
            if dim not in env:
                raise NotImplementedError(f"{p.name}: extent {dim} is not supplied by the inputs; "
                                          "provide explicit output buffers")
            return int(env[dim])
        return int(dim(env))

    def _check_layout(self, p: Param, t) -> None:
        expected = self._home_device()
        if t.device != expected:
            raise ValueError(f"compiled artifact is bound to {expected}, but {p.name} is on {t.device}")
        if t.numel() == 0 or p.free_strides:
            return
        if p.leading_stride and t.dim() == 2:
            if t.stride(1) != 1 and t.shape[1] > 1:
                raise ValueError(f"{p.name}.strides[1] violates the declared interface relation (must be 1)")
            if t.stride(0) < t.shape[1] and t.shape[0] > 1:
                raise ValueError(f"{p.name}.strides[0] is smaller than the row")
        elif not t.is_contiguous():
            raise ValueError(f"{p.name} must be contiguous")

    def _check_aliases(self, views: dict) -> None:
        """Writable views may not overlap any other view (noalias contract)."""
        writable = self._writable
        spans = {}
        for name, t in views.items():
            if t.numel() == 0:
                continue
            start = t.data_ptr()
            spans[name] = (start, start + _span_bytes(t))
        names = list(spans)
        for i, a in enumerate(names):
            for b in names[i + 1:]:
                if a not in writable and b not in writable:
                    continue
                (s0, e0), (s1, e1) = spans[a], spans[b]
                if s0 < e1 and s1 < e0:
                    raise ValueError(f"{self.definition.name}: {a} and {b} overlap; writable views must not alias")

    def _needs(self, env: dict) -> tuple[int, int]:
        """Bytes of the workspace (-1 without one) and of a launch's own scratch."""
        d = self.definition
        return (-1 if d.workspace is None else int(d.workspace(env)), 0 if d.scratch is None else int(d.scratch(env)))

    def _buffer_of(self, workspace: int, scratch: int):
        return self._scratch_of(scratch) if scratch > 0 else self._workspace_of(workspace)

    def _scratch_of(self, need: int):
        """Scratch of one launch: from torch's allocator on the launch stream (which reuses it only
        after that stream has passed the launch), so that calls of one artifact on several streams or
        threads never share it. None when memory is short: the call then runs without it."""
        import torch

        try:
            return torch.empty(need, dtype=torch.uint8, device=self._home_device())
        except torch.OutOfMemoryError:
            return None

    def _workspace_of(self, need: int):
        if need < 0:
            return None
        if self._workspace is None or self._workspace.numel() < need:
            import torch

            self._workspace = torch.empty(max(need, 16), dtype=torch.uint8, device=self._home_device())
        return self._workspace

    def _launch(self, binding: Binding) -> None:
        entry = self.definition.launch(binding.views, binding.env, _current_stream(self.device), binding.workspace)
        self._latest = (entry, _native.library().intent_amd_last_kernel())

    # ---- provider surface -------------------------------------------------------
    def launch_bound(self, binding: Binding):
        self._launch(binding)
        return _result(binding.outputs)

    def run(self, *arguments):
        binding = self._bind(arguments, None)
        needs = self._needs(binding.env)
        self._remember(arguments, False, binding, *needs)
        binding.workspace = self._buffer_of(*needs)
        return self.launch_bound(binding)

    def launch(self, *arguments):
        interface = self._interface
        n_in = len(interface.inputs)
        if len(arguments) != len(interface.parameters):
            raise TypeError(f"{self.definition.name}: expected {len(interface.parameters)} runtime arguments, "
                            f"got {len(arguments)}")
        ins = tuple(a for a, p in zip(arguments, interface.parameters) if not getattr(p, "output", False))
        outs = tuple(a for a, p in zip(arguments, interface.parameters) if getattr(p, "output", False))
        assert len(ins) == n_in
        binding = self._bind(ins, outs)
        needs = self._needs(binding.env)
        self._remember(arguments, True, binding, *needs)
        binding.workspace = self._buffer_of(*needs)
        self._launch(binding)
        return None

    def prepare_call(self, arguments: tuple, *, outputs: tuple | None = None) -> "HIPPreparedCall":
        binding = self._bind(tuple(arguments), outputs)
        workspace, scratch = self._needs(binding.env)
        binding.workspace = self._buffer_of(workspace, scratch)
        return HIPPreparedCall(self, binding, owns_scratch=scratch > 0)

    def infer_outputs(self, arguments: tuple):
        binding = self._bind(tuple(arguments), None, abstract=True)
        return _result(binding.outputs)

    def tuning_configurations(self, *arguments):
        return ()


def _span_bytes(t) -> int:
    """Bytes from a strided view's first element to the end of its last; 0 for an empty one."""
    if t.numel() == 0:
        return 0
    return (sum((extent - 1) * stride for extent, stride in zip(t.shape, t.stride())) + 1) * t.element_size()


def _result(outputs: tuple):
    if not outputs:
        return None
    return outputs[0] if len(outputs) == 1 else outputs


class HIPPreparedCall:
    """Invocation-owned arguments, outputs and scratch; launch() runs on torch's current stream.

    launch() allocates nothing, so a capture of it (torch.cuda.graph or a plain stream capture) holds
    only addresses that the prepared call keeps: it must outlive the graph."""

    def __init__(self, runtime: HIPRuntime, binding: Binding, owns_scratch: bool = False):
        self._runtime = runtime
        self._binding = binding
        # the stream whose order the allocator follows when the scratch is given back
        self._stream = _current_stream(runtime.device) if owns_scratch and binding.workspace is not None else None

    def compile(self) -> None:
        _native.library()  # the code objects are prebuilt; this validates the library and ABI

    def launch(self) -> None:
        if self._stream is not None and _current_stream(self._runtime.device) != self._stream:
            import torch

            self._binding.workspace.record_stream(torch.cuda.current_stream(self._runtime.device))
        self._runtime._launch(self._binding)

    def result(self):
        return _result(self._binding.outputs)

    @property
    def observation(self) -> NativeObservation | None:
        return self._runtime.observation

    def inspect_configurations(self) -> tuple[ConfigurationAssessment, ...]:
        d = self._runtime.definition
        if d.entry is None:
            return (ConfigurationAssessment(d.name, True, "single fixed kernel"),)
        env = self._binding.env
        chosen = d.entry(env, self._binding.workspace is not None)
        return tuple(ConfigurationAssessment(name, name == chosen and (limit is None or env["M"] <= limit), covers)
                     for name, covers, limit in d.entries)
