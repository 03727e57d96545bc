"""Step driver: forward -> loss -> backward for one micro-batch, with fp32 main-grad buffers.

Counterpart of `BaseRunner.forward_step` -> DeepSpeed `train_batch` (llm/runners/base_llm_runner.py:236-245)
for what lies inside this build: `loss = loss_fn(model(inputs), labels); loss.backward()`, weight
gradients landing in fp32 `main_grad` buffers (DeepSpeed's bf16 optimizer accumulates in fp32).
The optimizer step with global-norm clipping that follows lives in optimizer.py; loss scaling by the
number of accumulation steps and ZeRO partitioning are DeepSpeed's and are not reproduced.
"""
import torch

from .registry import MODULE_ZOO_REGISTRY
from . import functional as _F
from . import kernels as _K
from . import llama as _llama  # (registers the model builders)
from .losses import CrossEntropy
from .transformer import is_plain


def build_model(cfg):
    """cfg = {'type': 'llama_custom' | 'llama2_7b' | ..., 'kwargs': {...}} as in the reference's yaml `model:` node."""
    return MODULE_ZOO_REGISTRY.build(cfg)


def attach_main_grads(model):
    """One fp32 gradient buffer per parameter; marks them fresh (first write overwrites)."""
    for p in model.parameters():
        if p.requires_grad:
            p.main_grad = torch.zeros(p.shape, dtype=torch.float32, device=p.device)
            p.main_grad_fresh = True


def zero_main_grads(model):
    """zero_grad without a memset: the next gradient written to each buffer overwrites it."""
    for p in model.parameters():
        if getattr(p, "main_grad", None) is not None:
            p.main_grad_fresh = True
        p.grad = None


_LOSS_CALL = CrossEntropy.__call__


def _logits_stay_inside(model):
    """Nobody but this framework's own fused loss sees the model's output: no hook, subclass, replaced part or other loss in between.

    fp32_logits then only costs passes over memory: the fp32 logits hold bf16 values, the loss computes in fp32 from either, and
    its fp32 gradient is rounded to bf16 before the head's products.  Without the copies 4 x 1000 tokens at V = 32000 save 0.47 ms
    of 3.38 (a cast of the gradient, 146 us, and half the bytes of the head's result and of the loss)."""
    return (is_plain(model, _llama.LlamaModelPipe) and type(model.loss_fn) is CrossEntropy and model.loss_fn.fused
            and CrossEntropy.__call__ is _LOSS_CALL
            and is_plain(model.forward_funcs[-2], _llama.EmbedddingPipeNoTied))


def forward_step(model, inputs, labels):
    """One micro-batch: returns the loss tensor after backward has run."""
    with _F.input_checks_at_the_end():  # (before any gradient is written)
        output = model(inputs, cast_logits=False) if _logits_stay_inside(model) else model(inputs)
        loss = model.loss_fn(output, labels)
    loss.backward()
    return loss


def _tree_map(fn, x):
    if isinstance(x, torch.Tensor):
        return fn(x)
    if isinstance(x, (tuple, list)):
        return type(x)(_tree_map(fn, v) for v in x)
    return x


def _tree_pairs(dst, src):
    if isinstance(dst, torch.Tensor):
        return [(dst, src)]
    return [p for d, s in zip(dst, src) for p in _tree_pairs(d, s)] if isinstance(dst, (tuple, list)) else []


def _tree_copy(dst, src):
    """Tensors that lie alike on the current GPU in one launch; others (from the host, of another type or layout), and all of them where one (alike
    or not) is part of what another is copied to, one by one in their order."""
    pairs = _tree_pairs(dst, src)
    device = torch.cuda.current_device()
    alike = [type(s) is torch.Tensor and s.dtype is d.dtype and s.shape == d.shape and s.get_device() == d.get_device() == device
             and s.is_contiguous() and d.is_contiguous() and not s.is_neg() and not s.is_conj() for d, s in pairs]
    targets = {d.untyped_storage().data_ptr() for d, _ in pairs}
    if any(isinstance(s, torch.Tensor) and (type(s) is not torch.Tensor or s.layout is not torch.strided or s.untyped_storage().data_ptr() in targets)
           for _, s in pairs):  # (other kinds of tensors do not say what memory they read)
        alike = [False] * len(pairs)
    for a, (d, s) in zip(alike, pairs):
        if not a:
            d.copy_(s, non_blocking=True)
    if any(alike):
        _K.copy_list([d for a, (d, _) in zip(alike, pairs) if a], [s for a, (_, s) in zip(alike, pairs) if a])


class GraphedStep:
    """forward + loss + backward of one micro-batch captured once into a HIP graph and replayed.

    The captured kernels are exactly those of `forward_step`; replaying them removes the per-kernel host work and the
    launch gaps (about 180 launches per step for a 4-layer stack).  Shapes, document boundaries, the checkpoint plan and
    the gradient mode (first micro-batch overwrites `main_grad`, `accumulate=True` adds to it) are frozen at capture
    time; new token ids / labels of the same shape are copied into the static input buffers by `__call__`.  The loss is
    returned as a device tensor that the next replay overwrites.  The token-id range check of the embedding cannot
    raise inside a graph: its flag is read back after every replay and raised one call late, as in the deferred mode.
    """

    def __init__(self, model, inputs, labels, accumulate=False, warmup=2):
        from . import functional
        self.model = model
        self.inputs = _tree_map(lambda t: t.clone(), inputs)
        self.labels = _tree_map(lambda t: t.clone(), labels)
        self._accumulate = accumulate
        self._pending_flag = None

        grads = [p for p in model.parameters() if getattr(p, "main_grad", None) is not None]
        # The eager warm-up passes of an accumulating capture add the capture batch's gradients to the buffers; keep what
        # the buffers (and their "fresh" marks) held and put it back once the graph exists.
        saved = [(p.main_grad.clone(), getattr(p, "main_grad_fresh", False)) for p in grads] if accumulate else None

        def one_step():
            if accumulate:
                for p in grads:  # every captured gradient kernel must add: no buffer may be marked fresh here
                    p.main_grad_fresh = False
            else:
                zero_main_grads(model)
            return forward_step(model, self.inputs, self.labels)

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(warmup):
                one_step()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        for p in model.parameters():
            p.grad = None
        del functional.CAPTURED_ID_FLAGS[:]
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.loss = one_step()
        self._flags = list(functional.CAPTURED_ID_FLAGS)
        del functional.CAPTURED_ID_FLAGS[:]
        if saved is not None:
            torch.cuda.synchronize()
            for p, (buf, fresh) in zip(grads, saved):
                p.main_grad.copy_(buf)
                p.main_grad_fresh = fresh
        self._grads = grads
        self._host_flags = [torch.zeros(1, dtype=torch.int32, pin_memory=True) for _ in self._flags]
        self._flag_event = None

    def _check_previous(self):
        from . import functional
        if self._flag_event is not None:
            self._flag_event.synchronize()
            self._flag_event = None
            for host, (_, n) in zip(self._host_flags, self._flags):
                functional._raise_for_id_flag(int(host.item()), self.inputs[0] if isinstance(self.inputs, (tuple, list)) else self.inputs, n)

    def __call__(self, inputs=None, labels=None):
        self._check_previous()
        _tree_copy(*zip(*[(own, new) for own, new in ((self.inputs, inputs), (self.labels, labels)) if new is not None] or [((), ())]))
        if self._accumulate:
            for p in self._grads:  # the graph adds: a buffer marked fresh (zero_main_grads) starts from zero
                if getattr(p, "main_grad_fresh", False):
                    p.main_grad.zero_()
                    p.main_grad_fresh = False
        self.graph.replay()
        for host, (flag, _) in zip(self._host_flags, self._flags):
            host.copy_(flag, non_blocking=True)
        if self._flags:
            self._flag_event = torch.cuda.Event()
            self._flag_event.record()
        return self.loss

    def flush(self):
        """Raises for an out-of-range token id seen by the last replay."""
        self._check_previous()
