"""Autograd wiring of the trilinear query: forward, backward, backward of the
backward.  Two chained Functions with the same operands and return
conventions as the reference (ash/grid_query.py:10-283); each one is a single
call into the HIP library.
"""
import sys
import weakref
from typing import Literal

import torch

from .common import _get_c_extension

backend = _get_c_extension()

_N_TABLE_ARGS = 8  # grid_indices .. interpolation: operands without gradients

# One backward pass can reach the same embeddings through several nodes: a
# training step with a value loss and a gradient-norm loss runs both the first-
# and the second-order backward.  In the reference each zero-fills a dense
# gradient of the whole parameter and leaves the sum of the two to autograd (two
# fills and an add over the parameter: about a third of such a step).  The
# module's forward hands the second one to the first inside the graph
# (`grid._FusedGridForward`); `dense_grad` below also takes in what other nodes
# and an existing `.grad` contribute.
#
# which way the embedding gradient of the latest backward node went: "own"
# (a dense tensor of its own, handed to autograd), "contract" (added to the
# parameter's .grad inside a dense_grad block), "skipped" (nobody asked for it)
LAST_GRADIENT_PATH = None


# ---------------------------------------------------------------------------
# One dense gradient per step, by contract.
#
#     optimizer.zero_grad()
#     with ash.dense_grad(grid):          # or a Parameter, or several of either
#         loss.backward()
#     optimizer.step()
#
# Inside the block every backward node of the query adds its contribution for
# a registered parameter straight into `parameter.grad` (the library's
# `_accumulate` entries) and hands autograd no gradient for it: one zero fill
# per step instead of one per node plus autograd's additions over the whole
# parameter.  On entry a parameter whose `.grad` is None gets a zero-filled
# one (filled once); an existing `.grad` is accumulated onto, as
# `loss.backward()` would.  Nothing is handed to the engine and nothing is
# learnt from it: `.grad` is looked up when a node runs, other contributions to
# the parameter (a weight-decay term, say) reach the same tensor through
# autograd's own in-place accumulation, and hooks on other nodes may keep
# whatever they like.  What differs from plain `backward()`: hooks registered
# on the parameter itself do not see the query's contributions (they bypass
# its accumulation node), and under `create_graph=True` the block has no
# effect (an in-place addition would be invisible to the recorded graph).
# The block is for `loss.backward()`: a `torch.autograd.grad(..)` *with respect
# to a registered parameter* inside it would find the query's share in `.grad`
# and not in what it returns (gradients with respect to anything else, the
# positions for instance, are not affected).
_DENSE_TARGETS = {}   # id(parameter) -> (weak reference, nesting depth)


class dense_grad:
    """Context manager: see the comment above.  `targets` are Parameters or
    modules (every parameter of a module that is an `embeddings` operand of a
    query is simply one of its parameters).  `buffers` maps a parameter to the
    tensor to install as its `.grad` when it has none (default: a new one per
    entry)."""

    def __init__(self, *targets, buffers=None):
        self.parameters = []
        for t in targets:
            if isinstance(t, torch.nn.Module):
                self.parameters.extend(p for p in t.parameters() if p.requires_grad)
            elif isinstance(t, torch.Tensor):
                self.parameters.append(t)
            else:
                raise TypeError(f"dense_grad takes parameters or modules, got {type(t)}")
        self.buffers = buffers or {}

    def __enter__(self):
        for p in self.parameters:
            if p.grad is None:
                given = self.buffers.get(p)
                if given is not None:
                    if given.shape != p.shape or given.dtype != p.dtype or given.device != p.device:
                        raise RuntimeError("dense_grad: a buffer must be like its parameter")
                    p.grad = given.zero_()
                else:
                    p.grad = torch.zeros_like(p, memory_format=torch.contiguous_format)
            ref, depth = _DENSE_TARGETS.get(id(p), (weakref.ref(p), 0))
            _DENSE_TARGETS[id(p)] = (ref, depth + 1)
        return self

    def __exit__(self, *exc):
        for p in self.parameters:
            ref, depth = _DENSE_TARGETS[id(p)]
            if depth <= 1:
                del _DENSE_TARGETS[id(p)]
            else:
                _DENSE_TARGETS[id(p)] = (ref, depth - 1)
        return False


def _dense_target(embeddings):
    """The `.grad` tensor the running node is to add to, if `embeddings` is a
    parameter registered by a `dense_grad` block that applies, else None."""
    if not _DENSE_TARGETS or torch.is_grad_enabled():
        return None
    entry = _DENSE_TARGETS.get(id(embeddings))
    if entry is None or entry[0]() is not embeddings:
        return None
    grad = embeddings.grad
    if grad is None:
        # somebody dropped it inside the block: start a new one
        grad = embeddings.grad = torch.zeros_like(embeddings, memory_format=torch.contiguous_format)
    if (grad.shape != embeddings.shape or grad.dtype != embeddings.dtype
            or grad.device != embeddings.device or not grad.is_contiguous()):
        return None
    return grad


def _record_path(path: str) -> None:
    global LAST_GRADIENT_PATH
    LAST_GRADIENT_PATH = path


def _grad_requested(ctx, index: int, through: bool = False) -> bool:
    """Whether the running backward pass will consume the gradient of input
    `index`.  `ctx.needs_input_grad` only says that the input requires grad;
    in `autograd.grad(y, x)` the engine additionally knows which graph nodes it
    is going to execute, and the node behind an input it will not execute (the
    dense embeddings parameter, typically) needs no gradient from us.
    `through`: the input is the forward node's copy of the embeddings, and the
    node asked about is the one behind that node's own embeddings.  (In C++ where
    the native module is there: asked in Python each node of the graph becomes an
    object, and a leaf that the pass was asked for an exception, 20 us of a training
    step of 420.)"""
    host = getattr(backend, "host", None)
    if host is not None and hasattr(torch._C, "_will_engine_execute_node"):
        return host.grad_requested(ctx, index, through)
    if not ctx.needs_input_grad[index]:
        return False
    try:
        node = ctx.next_functions[index][0]
        if through:
            node = node.next_functions[0][0]
        return node is not None and torch._C._will_engine_execute_node(node)
    except Exception:  # outside an engine pass, or an older torch: be conservative
        return True


def _holders(t: torch.Tensor):
    """Who holds `t`: references to the Python object, to the tensor, to its
    storage."""
    return (sys.getrefcount(t), t._use_count(),
            torch._C._storage_Use_Count(t.untyped_storage()._cdata))


class _HoldersProbe(torch.autograd.Function):
    """A node of the shape of `grid._FusedGridForward` that notes what
    `_holders` says in its backward of a gradient that nobody else holds."""

    seen = None

    @staticmethod
    def forward(ctx, t):
        ctx.set_materialize_grads(False)
        return t.clone(), t.new_zeros(1), t.detach()

    @staticmethod
    def backward(ctx, z, _unused, carried):
        return _HoldersProbe.note(ctx, z, carried)

    @staticmethod
    def note(ctx, z, carried):
        _HoldersProbe.seen = _holders(carried)
        return carried


_HOLDERS_ALONE = None


def _learn_holders() -> None:
    """What `_holders` says in a backward node, one call below its `backward`,
    of a gradient that only the engine's call holds: learnt once from a node
    that is made for it.  False where this torch cannot tell; gradients are then
    never added in place."""
    global _HOLDERS_ALONE
    _HOLDERS_ALONE = False
    try:
        with torch.enable_grad():
            y, _, again = _HoldersProbe.apply(torch.zeros(1, requires_grad=True))
            (y.sum() + (2 * again).sum()).backward()
        _HOLDERS_ALONE = _HoldersProbe.seen or False
    except Exception:
        pass


# Queries from which second-order nodes leave their share to the forward node, by the wall
# time of training steps of 20 000 blocks, one after the other | each waited for (own share
# -> put off, us).  Fewer wait for the host, and the kernel time saved reaches nobody: 131 000
# of 1, 4, 5, 16 channels 308 -> 308, 428 -> 436, 425 -> 430, 437 -> 440; 262 000 307 -> 310,
# 428 -> 433, 419 -> 431, 439 -> 441 | 361 -> 363, 475 -> 483, 470 -> 478, 603 -> 570.  From
# here on the kernels of wide rows show, first where steps are waited for: 393 000 of 5, 8, 12,
# 16 channels 417 -> 425, 427 -> 429, 431 -> 435, 466 -> 436 | 462 -> 467, 490 -> 475, 562 ->
# 541, 640 -> 572; 524 000 421 -> 428, 427 -> 430, 431 -> 434, 569 -> 476 | 477 -> 466, 504 ->
# 482, 582 -> 561, 721 -> 635; 1 M of 1, 4, 5, 8, 12 310 -> 313, 434 -> 436, 430 -> 429, 465 ->
# 439, 630 -> 578 | 379 -> 358, 514 -> 480, 536 -> 478, 584 -> 551, 715 -> 663; 2 M of 1, 4, 5
# 432 -> 437, 544 -> 457, 628 -> 529.
PUT_OFF_FROM = 3 << 17


class _Pass:
    """What is put off in one pass of the engine, which holds this object, as one of
    the pass's final callbacks, until the pass ends, in whichever way."""

    __slots__ = ("parts", "__weakref__")

    def __init__(self):
        self.parts = []   # ((grad_grad_offsets, z), operands, parameter's .grad or None)

    def __call__(self):
        self.parts = []


class _Later:
    """What second-order nodes leave for the backward of the forward node they
    were recorded from: their contributions to the embedding gradient go to the
    same eight rows per query as that node's own, and both are bound by the
    requests for these rows, so the forward node adds the two in one pass over
    the queries (2^22 ray samples, rows of four: 187 + 184 -> 254 us).

    Put off is only what is certain to be taken up in the same pass, and seen by
    nobody in between: the engine is going to execute the forward node, which
    waits for the second-order node as it ever did, and no hook sits behind the
    one or before the other.  (They share a stream: the second-order node is
    recorded by the forward node's own backward, which the engine runs on the
    stream of the forward.)  Kept by the pass, so that what one leaves behind that
    fails in between is not taken up by another, and goes with it."""

    __slots__ = ("passes",)

    def __init__(self):
        self.passes = {}   # id of a pass -> weak reference to its _Pass

    def room(self, ctx):
        """The list of the running pass if `ctx`, a second-order node whose second
        input is the forward node's copy of the embeddings, may put off its
        contributions."""
        try:
            task = torch._C._current_graph_task_id()
            if (task < 0 or torch.is_grad_enabled()
                    or not torch._C._will_engine_execute_node(ctx.next_functions[1][0])
                    or not backend.host.hands_over_unseen(ctx, 1)):
                return None
            here = self._of(task)
            if here is None:
                here = _Pass()
                torch.autograd.Variable._execution_engine.queue_callback(here)
                for known, each in list(self.passes.items()):
                    if each() is None:
                        self.passes.pop(known, None)
                self.passes[task] = weakref.ref(here)
            return here.parts
        except Exception:  # outside an engine pass, or another torch
            return None

    def _of(self, task):
        each = self.passes.get(task)
        return None if each is None else each()

    def take(self):
        if not self.passes:
            return ()
        task = torch._C._current_graph_task_id()
        here = self._of(task)
        if here is None:
            return ()
        del self.passes[task]
        parts, here.parts = here.parts, []
        return parts


def add_put_off(parts, carried, grid_dim, interpolation, cell_size: float = 1.0):
    """The gradient `carried` with `parts` of a `_Later`, by themselves."""
    if any(target is None for _, _, target in parts):
        if carried is None:
            carried = torch.zeros_like(parts[0][1][0], memory_format=torch.contiguous_format)
        elif not (_HOLDERS_ALONE and _holders(carried) == _HOLDERS_ALONE and carried.is_contiguous()):
            carried = carried.clone(memory_format=torch.contiguous_format)
    for (u, z), operands, target in parts:
        backend.query_backward_backward_onto(carried if target is None else target, u, z, *operands,
                                             grid_dim, interpolation, **_per_cell(cell_size))
    return carried


def _per_cell(cell_size):
    """The argument for positions in units of a cell, which the native library alone
    knows and which is left out where it says nothing."""
    return {} if cell_size == 1.0 else {"cell_size": cell_size}


class SparseDenseGridQuery(torch.autograd.Function):
    """y[i] = sum over the 8 cell corners c of w_c(offsets[i]) * embeddings[row_c(i)].

    Differentiable with respect to `embeddings` and `offsets`; the indices,
    masks and neighbour tables only address memory.
    """

    @staticmethod
    def forward(
        ctx,
        embeddings: torch.Tensor,
        offsets: torch.Tensor,
        grid_indices: torch.Tensor,
        cell_indices: torch.Tensor,
        masks: torch.Tensor,
        lut_grid_nb2grid_idx: torch.Tensor,
        lut_cell_nb2cell_idx: torch.Tensor,
        lut_cell_nb2grid_nb: torch.Tensor,
        grid_dim: int,
        interpolation: Literal["linear", "smooth_step"] = "smooth_step",
    ) -> torch.Tensor:
        """embeddings (B, M, E), offsets (N, 3) in [0, 1), grid/cell indices and
        masks (N,), tables (B, 8), (M, 8), (M, 8); returns (N, E)."""
        operands = (
            embeddings,
            offsets,
            grid_indices,
            cell_indices,
            masks,
            lut_grid_nb2grid_idx,
            lut_cell_nb2cell_idx,
            lut_cell_nb2grid_nb,
        )
        ctx.save_for_backward(*operands)
        ctx.grid_dim = grid_dim
        ctx.interpolation = interpolation
        return backend.query_forward(*operands, grid_dim, interpolation)

    @staticmethod
    def backward(ctx, z: torch.Tensor):
        """Delegates to SparseDenseGridQueryBackward so that this step is itself
        differentiable (needed for gradient-norm losses)."""
        return first_order_backward(ctx, z, ctx.saved_tensors) + (None,) * _N_TABLE_ARGS


def first_order_backward(ctx, z, operands, embeddings_input: int = 0, offsets_input: int = 1,
                         again=None, carried=None, later=None, cell_size: float = 1.0):
    """(grad_embeddings, grad_offsets) of a forward node whose inputs number
    `embeddings_input` / `offsets_input` are the embeddings and the offsets, or
    positions of which the offsets are 1 / `cell_size`; `operands`
    = (embeddings, offsets, grid_indices, cell_indices, masks, three tables).
    `again`: the node's own copy of the embeddings, which a recorded backward is
    to depend on instead; `carried`: the gradient that has arrived for it;
    `later`: what belongs to that and has been put off."""
    need_embeddings = _grad_requested(ctx, embeddings_input)
    need_offsets = _grad_requested(ctx, offsets_input)
    parts = later.take() if later is not None else ()
    if not (need_embeddings or need_offsets):
        return None, None
    if not need_embeddings:
        carried, parts = None, ()
    along = _per_cell(cell_size)
    if parts:
        along["along"] = [pair for pair, _, _ in parts]
    # The reference always produces both gradients (ash/grid_query.py:104-116);
    # the dense embedding gradient (zero fill + atomics over the whole
    # parameter) is skipped when nobody asked for it, e.g. in
    # autograd.grad(y, x, create_graph=True).
    target = _dense_target(operands[0]) if need_embeddings else None
    _record_path("contract" if target is not None else "own" if need_embeddings else "skipped")
    if target is not None:
        # no graph is being recorded: the library is called directly
        _, grad_offsets = backend.query_backward_forward(
            z.contiguous(),
            *operands,
            ctx.grid_dim,
            ctx.interpolation,
            need_embeddings=True,
            need_offsets=need_offsets,
            accumulate_into=target,
            **along,
        )
        return carried, grad_offsets
    if (
        carried is not None
        and not torch.is_grad_enabled()
        and _HOLDERS_ALONE
        and _holders(carried) == _HOLDERS_ALONE
        and carried.is_contiguous()
        and hasattr(backend, "query_backward_forward_onto")
    ):
        # the tensor is this call's alone: the node's own contribution goes on top
        grad_offsets = backend.query_backward_forward_onto(
            carried, z.contiguous(), *operands, ctx.grid_dim, ctx.interpolation,
            need_offsets=need_offsets, **along)
        return carried, grad_offsets
    if parts:
        grad_embeddings, grad_offsets = backend.query_backward_forward(
            z.contiguous(), *operands, ctx.grid_dim, ctx.interpolation, need_offsets=need_offsets, **along)
        return grad_embeddings if carried is None else grad_embeddings + carried, grad_offsets
    owner = None
    if again is not None and torch.is_grad_enabled():
        owner = weakref.ref(operands[0])
        operands = (again, *operands[1:])
    else:
        later = None
    grad_embeddings, grad_offsets = SparseDenseGridQueryBackward.apply(
        z.contiguous(),
        *operands,
        ctx.grid_dim,
        ctx.interpolation,
        need_embeddings,
        need_offsets,
        owner,
        later,
        cell_size,
    )
    if carried is not None:
        grad_embeddings = grad_embeddings + carried
    return grad_embeddings, grad_offsets


class SparseDenseGridQueryBackward(torch.autograd.Function):
    """(z, embeddings, offsets) -> (grad_embeddings, grad_offsets) with

        grad_embeddings[row_c(i)] += w_c(offsets[i]) * z[i]
        grad_offsets[i] = sum_c (embeddings[row_c(i)] . z[i]) * dw_c/doffsets

    `z` may carry a graph itself (autograd.grad(..., create_graph=True)).
    """

    @staticmethod
    def forward(
        ctx,
        z,
        embeddings,
        offsets,
        grid_indices,
        cell_indices,
        masks,
        lut_grid_nb2grid_idx,
        lut_cell_nb2cell_idx,
        lut_cell_nb2grid_nb,
        grid_dim,
        interpolation,
        need_grad_embeddings: bool = True,
        need_grad_offsets: bool = True,
        owner=None,
        later=None,
        cell_size: float = 1.0,
    ):
        """With both `need_*` flags at their default this is the reference's
        signature and result; an output that is not needed is returned as None
        and its work is skipped.  `owner`: weak reference to the embeddings that
        the operand is the forward node's copy of; `later`, `cell_size`: that
        node's."""
        operands = (
            z,
            embeddings,
            offsets,
            grid_indices,
            cell_indices,
            masks,
            lut_grid_nb2grid_idx,
            lut_cell_nb2cell_idx,
            lut_cell_nb2grid_nb,
        )
        ctx.save_for_backward(*operands)
        ctx.grid_dim = grid_dim
        ctx.interpolation = interpolation
        ctx.owner = owner
        ctx.later = later
        ctx.per_cell = _per_cell(cell_size)
        if need_grad_embeddings and need_grad_offsets:
            return backend.query_backward_forward(*operands, grid_dim, interpolation, **ctx.per_cell)
        return backend.query_backward_forward(
            *operands,
            grid_dim,
            interpolation,
            need_embeddings=need_grad_embeddings,
            need_offsets=need_grad_offsets,
            **ctx.per_cell,
        )

    @staticmethod
    def backward(ctx, grad_grad_embeddings: torch.Tensor, grad_grad_offsets: torch.Tensor):
        """Given u = d loss / d grad_offsets, returns

            grad_z[i]                = sum_c (dw_c/doffsets . u[i]) * embeddings[row_c(i)]
            grad_embeddings[row_c(i)] += (dw_c/doffsets . u[i]) * z[i]

        Exactly like the reference (ash/grid_query.py:209-283,
        ash/src/grid.cu:417-426) the incoming `grad_grad_embeddings` is not used
        and no gradient flows to `offsets` at second order.
        """
        owned = ctx.owner is not None
        need_z = _grad_requested(ctx, 0)
        need_embeddings = _grad_requested(ctx, 1, owned)
        n_rest = _N_TABLE_ARGS + 6  # offsets, tables, grid_dim, interpolation, 2 flags, owner, later, cell_size
        if grad_grad_offsets is None or not (need_z or need_embeddings):
            return (None, None) + (None,) * n_rest
        saved = ctx.saved_tensors
        embeddings = ctx.owner() if owned else saved[1]
        target = _dense_target(embeddings) if need_embeddings and embeddings is not None else None
        unused = {**getattr(backend, "WITHOUT_OFFSETS", {}), **ctx.per_cell}
        put_off = None
        if (need_embeddings and not need_z and ctx.later is not None
                and grad_grad_offsets.shape[0] >= PUT_OFF_FROM):
            put_off = ctx.later.room(ctx)
        if put_off is not None:
            put_off.append(((grad_grad_offsets, saved[0]), saved[1:], target))
            unused = {**unused, "later": True}
        _record_path("contract" if target is not None else "own" if need_embeddings else "skipped")
        if target is not None:
            grad_z, _, _ = backend.query_backward_backward(
                grad_grad_embeddings,
                grad_grad_offsets,
                *saved,
                ctx.grid_dim,
                ctx.interpolation,
                need_z=need_z,
                need_embeddings=True,
                accumulate_into=target,
                **unused,
            )
            return (grad_z, None) + (None,) * n_rest
        if need_z and need_embeddings:
            grad_z, grad_embeddings, _ = backend.query_backward_backward(
                grad_grad_embeddings,
                grad_grad_offsets,
                *saved,
                ctx.grid_dim,
                ctx.interpolation,
                **unused,
            )
        else:
            grad_z, grad_embeddings, _ = backend.query_backward_backward(
                grad_grad_embeddings,
                grad_grad_offsets,
                *saved,
                ctx.grid_dim,
                ctx.interpolation,
                need_z=need_z,
                need_embeddings=need_embeddings,
                **unused,
            )
        return (grad_z, grad_embeddings) + (None,) * n_rest
