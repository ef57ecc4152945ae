"""Rodas5P on MI355X: ``solve(ode_fn, y0, t_span, params, ...)``.

The API is the reference's (modax/rodas5P.py:1024-1237): the same arguments,
defaults and return shapes -- a ``(N, n_save, n_vars)`` history, optionally with
a stats dict of per-trajectory ``accepted_steps``/``rejected_steps``/
``loop_steps`` counters. Inputs may be numpy arrays (a numpy result comes back)
or torch tensors (the result is a torch tensor on the GPU, a view of the
structure-of-arrays history the kernel writes).

Only the right-hand side is supplied. ``df/dy`` and ``df/dt`` are generated by
forward-mode differentiation of the traced callback, one sweep per colour of
the Jacobian's column intersection graph. ``lu_precision`` picks the precision
of the iteration matrix, its LU factorisation and the stage vectors; state,
error norm and step control are always double.

Differentiation (modax/_sensitivity.py): when ``y0`` or ``params`` is a torch
tensor that requires grad or carries a forward-mode tangent, the solve
integrates the joint forward-sensitivity system for the blocks asked for and
returns a tensor whose ``backward`` and ``jvp`` contract ``S = dy/dtheta``
(``sens_error_control`` and ``sens_param_columns`` as in the reference).
``adjoint=True`` makes the backward a discrete-adjoint kernel instead
(checkpointed every ``ckpt_every`` accepted steps, or keeping a record of each
where they fit: ``_autodiff._records_whole``); ``adjoint_gradients`` and
``solve_sensitivities`` expose both directly. ``torch.func.vmap`` over
single-trajectory solves lowers to one ensemble launch (the reference's
``custom_vmap``). ``save_hook``/``hook_size``/``save_history`` run a traced hook
at every save inside the kernel; ``array_rhs`` gives an array-form right-hand
side for the stage evaluations.

Beyond the reference: ``refill`` selects the persistent kernel in which a lane
takes the next trajectory from a device queue as soon as its own ends
(``None`` = decide from the ensemble size), ``work_order`` is the order in
which that queue hands trajectories out (a permutation of 0..N-1; claiming the
expensive ones first -- ``_common.cost_order`` of an earlier solve's step
counts -- shortens the ensemble's tail; ``"pilot"`` estimates that order with a
short pilot of every trajectory on the device, which the solve then resumes;
``None`` = the pilot's order when the ensemble's size picks the persistent
launch, index order when the caller set ``refill=True``: the same bits either
way, and on the 100,000-trajectory uneven stiff ensemble 684 -> 555 ms with the
FP32 LU, 1.78 -> 1.13 s refined), ``stream`` names the torch stream to
launch on (after the current stream's work on the inputs; a GPU result is ready
when that stream has run, NumPy results and gradients are waited for),
``placement`` picks where the step keeps its vectors
(registers, scratch or LDS; ``None`` = by size), and ``tableau_in_registers``
whether the unrolled step holds the method's coefficients in registers rather
than rebuilding each from scalar moves at every use (``None`` = by size and
ensemble size, ``_kernels.tableau_in_registers``). Every trajectory computes
the same bits whichever is chosen.

``lu_refine=True`` (with ``lu_precision="fp32"``, a plain solve) keeps the FP32
factorisation and solves but refines each stage solve once: the residual of
the FP32 solution against the FP64 iteration matrix ``I/(h gamma) - J(y_n,
t_n)`` (``J x`` by one forward-mode sweep) is solved with the same FP32
factors and added, and the stage vectors are stored in FP64. The stages then
carry FP64 accuracy, so the solution follows the FP64-LU solve's to rounding
instead of differing from it by the accumulated FP32 rounding of the stage
vectors (the reference's FP32 typing, kept by default).
"""

from __future__ import annotations

import functools
from dataclasses import replace

from . import _autodiff, _common, _kernels, _runtime
from ._kernels import KernelOptions, trajectories_per_block_or_default
from ._sparsity import normalize_sparsity

#: refill pays once the ensemble outnumbers the lanes the device keeps resident:
#: up to that every trajectory has a lane of its own either way, above it the
#: plain launch runs its workgroups in rounds (the 100,000 x 50 uneven stiff
#: ensemble at 1.5x the rolled kernel's resident lanes: 1.98 s plain, 1.40 s
#: refill)
_REFILL_MIN_WAVES_PER_CU = 1


def solve(
    ode_fn,
    y0,
    t_span,
    params,
    *,
    rtol=1e-8,
    atol=1e-10,
    first_step=None,
    max_steps=100000,
    return_stats=False,
    error_weights=None,
    pcoeff=0.0,
    icoeff=1.0,
    dcoeff=0.0,
    lu_precision: str = "fp32",
    trajectories_per_block=None,
    sens_error_control=True,
    sens_param_columns=None,
    sparsity=None,
    ordering="amd",
    tf_index=None,
    max_registers=None,
    array_rhs=None,
    save_hook=None,
    hook_size: int = 0,
    save_history: bool = True,
    refill=None,
    stream=None,
    work_order=None,
    placement=None,
    adjoint=False,
    ckpt_every=64,
    tableau_in_registers=None,
    lu_refine=False,
):
    """Integrate an ensemble with Rodas5P; see the module docstring."""
    if _autodiff.under_vmap(y0, t_span, params):
        # torch.func.vmap over single-trajectory solves: one ensemble launch
        kwargs = dict(rtol=rtol, atol=atol, first_step=first_step, max_steps=max_steps,
                      return_stats=True, error_weights=error_weights, pcoeff=pcoeff,
                      icoeff=icoeff, dcoeff=dcoeff, lu_precision=lu_precision,
                      trajectories_per_block=trajectories_per_block, sparsity=sparsity,
                      ordering=ordering, tf_index=tf_index, max_registers=max_registers,
                      array_rhs=array_rhs, refill=refill, stream=stream, placement=placement,
                      tableau_in_registers=tableau_in_registers, lu_refine=lu_refine)

        def run(y, t, p):
            hist, stats = solve(ode_fn, y, t, p, **kwargs)
            return (hist, stats["accepted_steps"], stats["rejected_steps"], stats["loop_steps"])

        hist, acc, rej, loop = _autodiff.vmap_solve(
            run, *(_common.as_f64_device(x, _common.device()) for x in (y0, t_span, params)))
        if return_stats:
            return hist, _common.solver_stats(acc, rej, loop)
        return hist
    if save_hook is not None:
        if hook_size <= 0:
            raise ValueError("a save_hook needs a positive hook_size")
    elif not save_history:
        raise ValueError("save_history=False needs a save_hook to consume the saves")
    dev = _common.device()
    y0_t, p_t, n, n_vars = _common.normalize_y0_params(y0, params, dev)
    n_params = p_t.shape[1]
    if sparsity is not None:
        sparsity = normalize_sparsity(sparsity, n_vars)
    options = KernelOptions(
        pcoeff=float(pcoeff),
        icoeff=float(icoeff),
        dcoeff=float(dcoeff),
        lu_precision=lu_precision,
        trajectories_per_block=trajectories_per_block_or_default(trajectories_per_block),
        sparsity=sparsity,
        ordering=ordering,
        tf_index=-1 if tf_index is None else int(tf_index),
        max_registers=max_registers,
        unit_weights=error_weights is None,
        placement=placement,
        array_rhs=array_rhs,
        tableau_in_registers=_tableau(tableau_in_registers, n_vars, n, placement, max_registers),
        lu_refine=bool(lu_refine),
    )
    times = _common.as_f64_device(t_span, dev).contiguous()
    if times.ndim != 1 or times.numel() < 1:
        raise ValueError("t_span must be a non-empty 1-D array of save times")
    launch_kw = dict(dt0=_common.initial_step(first_step), rtol=rtol, atol=atol,
                     max_steps=max_steps, refill=refill, stream=stream,
                     order=_common.work_order_arg(work_order, n, dev))
    if save_hook is not None:
        # a hooked solve is the plain launch: the hook's output carries no
        # derivative rule (modax/rodas5P.py:1204-1209)
        options = replace(options, save_hook=save_hook, hook_size=int(hook_size),
                          save_history=bool(save_history), hook_n_save=int(times.numel()))
        if tableau_in_registers is None:
            options = _fitting_tableau(options, ode_fn, n_vars, n_params, n)
        built = _kernels.rodas5p_kernel(ode_fn, n_vars, n_params, options)
        out = launch(built, y0_t.detach(), times, p_t.detach(), n,
                     weights=_common.error_weights_soa(error_weights, n, n_vars, dev),
                     hook_size=int(hook_size), save_history=bool(save_history), **launch_kw)
        as_numpy = _common.wants_numpy(y0, params, t_span)
        if as_numpy:
            _common.join(stream, dev)
        hist = out.ensemble_view()
        hook_out = out.hook_out.t()
        stats = _common.solver_stats(out.accepted, out.rejected, out.loop)
        if as_numpy:
            hist, hook_out = hist.cpu().numpy(), hook_out.cpu().numpy()
            stats = {k: v.cpu().numpy() for k, v in stats.items()}
        return (hist, hook_out, stats) if return_stats else (hist, hook_out)
    wrt_y0, wrt_params = _autodiff.wanted(y0, params)
    if (wrt_y0 or wrt_params) and lu_refine:
        raise ValueError("lu_refine is for a plain solve: the adjoint and the forward "
                         "sensitivities differentiate the unrefined step")
    if (wrt_y0 or wrt_params) and adjoint:
        weights = _common.error_weights_soa(error_weights, n, n_vars, dev)
        job = _autodiff.AdjointJob(
            built=_kernels.rodas5p_kernel(ode_fn, n_vars, n_params, _sized(
                options, ode_fn, n_vars, n_params, n, trajectories_per_block,
                launch_kw["order"] is None and not refill, tableau_in_registers is None)),
            times=times, n=n, n_vars=n_vars, n_params=n_params, weights=weights,
            launch_kw=launch_kw, ckpt_every=int(ckpt_every),
            **_adjoint_kernels(options, ode_fn, n_vars, n_params, n, trajectories_per_block,
                               ckpt_every))
        hist, counters = _autodiff.adjoint_solve(job, y0_t, p_t)
        if return_stats:
            return hist, _common.solver_stats(*counters)
        return hist
    if wrt_y0 or wrt_params:
        n_aug = None
        if trajectories_per_block is None:
            # the joint vector differentiable_solve will integrate
            n_aug = _autodiff.SensitivitySpec(
                n_vars, n_params, bool(wrt_y0), bool(wrt_params), bool(sens_error_control),
                None if sens_param_columns is None else tuple(sens_param_columns)).n_aug
        job = _joint_job(ode_fn, options, times, n, n_vars, n_params, error_weights, dev,
                         launch_kw, n_aug=n_aug)
        state, counters = _autodiff.differentiable_solve(
            job, y0_t, p_t, wrt_y0, wrt_params, sens_error_control, sens_param_columns)
        if return_stats:
            return state, _common.solver_stats(*counters)
        return state
    options = _sized(options, ode_fn, n_vars, n_params, n, trajectories_per_block,
                     launch_kw["order"] is None and not refill, tableau_in_registers is None)
    built = _kernels.rodas5p_kernel(ode_fn, n_vars, n_params, options)
    if launch_kw["order"] is None and refill is None and _use_refill(built, n):
        launch_kw = dict(launch_kw, order="pilot")
    out = launch(built, y0_t.detach(), times, p_t.detach(), n,
                 weights=_common.error_weights_soa(error_weights, n, n_vars, dev), **launch_kw)
    as_numpy = _common.wants_numpy(y0, params, t_span)
    if as_numpy:
        _common.join(stream, dev)
    return finish(out, return_stats, as_numpy)


def _joint_job(ode_fn, options, times, n, n_vars, n_params, error_weights, dev, launch_kw,
               n_aug=None):
    if not launch_kw.get("refill") and launch_kw.get("order") is None:
        # the joint [y, S] solve of a small ensemble of a large dense system
        # takes the wave placement like the plain one; of a sparse system, the
        # workgroup size for its joint vector (n_aug long) when the caller gave
        # none
        options = replace(options, placement=_wave(options, n_vars, n))
        if n_aug is not None:
            options = _small_ensemble_block(options, n_aug, n)
    w = None
    if error_weights is not None:
        w = _common.as_f64_device(error_weights, dev)
        w = w.expand(n, n_vars) if w.ndim == 1 else w

    def build(spec, unit_weights):
        joint = replace(options, sens=spec, unit_weights=unit_weights)
        if n_aug is not None and _kernels.rodas5p_team(ode_fn, n_vars, n_params, joint):
            joint = replace(joint, placement=_kernels.TEAM,
                            trajectories_per_block=_kernels.DEFAULT_BLOCK)
        return _kernels.rodas5p_kernel(ode_fn, n_vars, n_params, joint)

    return _autodiff.JointJob(build=build, times=times, n=n, n_vars=n_vars, n_params=n_params,
                              weights=w, launch_kw=launch_kw)


def adjoint_gradients(ode_fn, y0, t_span, params, hist_cotangent, *, ckpt_every=64,
                      rtol=1e-8, atol=1e-10, first_step=None, max_steps=100000,
                      error_weights=None, pcoeff=0.0, icoeff=1.0, dcoeff=0.0,
                      lu_precision="fp32", trajectories_per_block=None, sparsity=None,
                      ordering="amd", tf_index=None, max_registers=None, stream=None,
                      placement=None):
    """Gradients of a loss of the solve's history by the discrete adjoint:
    ``hist_cotangent`` is dL/dhist ``(N, n_save, n_vars)`` for the solve
    ``solve(ode_fn, y0, t_span, params, ...)`` with the same options; returns
    ``(dL/dy0 (N, n_vars), dL/dparams (N, n_params))``. The accepted steps are
    differentiated with their sizes held fixed. With the default ``ckpt_every``
    the forward steps' records are kept where they fit in 8 GiB and a quarter of
    the free memory (8,192 trajectories of 20 variables and 1,400 steps: 2.2 GB);
    else, or with a smaller ``ckpt_every``, the forward solve is recomputed from
    checkpoints taken every ``ckpt_every`` accepted steps (0.14 GB).
    ``placement`` chooses where the kernels keep their per-lane vectors (by
    size when None; the adjoint uses registers, a team, or the rolled step with
    its stage arrays in LDS or scratch by ``_kernels.adjoint_block``); every
    placement gives the same bits."""
    import torch

    dev = _common.device()
    y0_t, p_t, n, n_vars = _common.normalize_y0_params(y0, params, dev)
    n_params = p_t.shape[1]
    if sparsity is not None:
        sparsity = normalize_sparsity(sparsity, n_vars)
    options = KernelOptions(
        pcoeff=float(pcoeff), icoeff=float(icoeff), dcoeff=float(dcoeff),
        lu_precision=lu_precision,
        trajectories_per_block=trajectories_per_block_or_default(trajectories_per_block),
        sparsity=sparsity, ordering=ordering, tf_index=-1 if tf_index is None else int(tf_index),
        max_registers=max_registers, unit_weights=error_weights is None, placement=placement,
    )
    times = _common.as_f64_device(t_span, dev).contiguous()
    launch_kw = dict(dt0=_common.initial_step(first_step), rtol=rtol, atol=atol,
                     max_steps=max_steps, refill=False, stream=stream)
    weights = _common.error_weights_soa(error_weights, n, n_vars, dev)
    job = _autodiff.AdjointJob(
        built=_kernels.rodas5p_kernel(ode_fn, n_vars, n_params, options),
        times=times, n=n, n_vars=n_vars, n_params=n_params, weights=weights,
        launch_kw=launch_kw, ckpt_every=int(ckpt_every),
        **_adjoint_kernels(options, ode_fn, n_vars, n_params, n, trajectories_per_block,
                           ckpt_every))
    y0_d, p_d = y0_t.detach(), p_t.detach()
    g = _common.as_f64_device(hist_cotangent, dev)
    if tuple(g.shape) != (n, times.numel(), n_vars):
        raise ValueError(f"hist_cotangent must be (N, n_save, n_vars) = "
                         f"{(n, times.numel(), n_vars)}; got {tuple(g.shape)}")
    gy, gp = _autodiff.adjoint_gradients(job, y0_d, p_d, g)
    if _common.wants_numpy(y0, params, t_span, hist_cotangent):
        return gy.cpu().numpy(), gp.cpu().numpy()
    del torch
    return gy, gp


def solve_sensitivities(ode_fn, y0, t_span, params, *, wrt_y0=True, wrt_params=True,
                        sens_error_control=True, sens_param_columns=None, return_stats=False,
                        rtol=1e-8, atol=1e-10, first_step=None, max_steps=100000,
                        error_weights=None, pcoeff=0.0, icoeff=1.0, dcoeff=0.0,
                        lu_precision="fp32", trajectories_per_block=None, sparsity=None,
                        ordering="amd", tf_index=None, max_registers=None, refill=None,
                        stream=None, placement=None):
    """One joint ``[y, S]`` solve: returns the state ``(N, n_save, n_vars)`` and
    ``S = dy/dtheta`` as ``(N, n_save, n_vars, n_sens)`` -- the initial-state
    directions first (when ``wrt_y0``), then the parameter columns (all, or
    ``sens_param_columns``) -- the quantities the reference's JVP rule
    contracts (modax/_sensitivity.py:331-413). Same options as ``solve``."""
    dev = _common.device()
    y0_t, p_t, n, n_vars = _common.normalize_y0_params(y0, params, dev)
    n_params = p_t.shape[1]
    if sparsity is not None:
        sparsity = normalize_sparsity(sparsity, n_vars)
    options = KernelOptions(
        pcoeff=float(pcoeff), icoeff=float(icoeff), dcoeff=float(dcoeff),
        lu_precision=lu_precision,
        trajectories_per_block=trajectories_per_block_or_default(trajectories_per_block),
        sparsity=sparsity, ordering=ordering, tf_index=-1 if tf_index is None else int(tf_index),
        max_registers=max_registers, unit_weights=error_weights is None, placement=placement,
    )
    times = _common.as_f64_device(t_span, dev).contiguous()
    launch_kw = dict(dt0=_common.initial_step(first_step), rtol=rtol, atol=atol,
                     max_steps=max_steps, refill=refill, stream=stream)
    spec = _autodiff.SensitivitySpec(
        n_vars, n_params, bool(wrt_y0), bool(wrt_params), bool(sens_error_control),
        None if sens_param_columns is None else tuple(int(c) for c in sens_param_columns))
    job = _joint_job(ode_fn, options, times, n, n_vars, n_params, error_weights, dev, launch_kw,
                     n_aug=spec.n_aug if trajectories_per_block is None else None)
    job.spec = spec
    out, state, sens = _autodiff.joint_solve(job, y0_t.detach(), p_t.detach())
    stats = _common.solver_stats(out.accepted, out.rejected, out.loop)
    if _common.wants_numpy(y0, params, t_span):
        state, sens = state.cpu().numpy(), sens.cpu().numpy()
        stats = {k: v.cpu().numpy() for k, v in stats.items()}
    return (state, sens, stats) if return_stats else (state, sens)


def launch(built, y0_t, times, p_t, n, *, dt0, rtol, atol, max_steps, weights=None, refill=None,
           stream=None, outputs=None, workspace=None, hook_size=0, save_history=True, grid=0,
           order=None):
    """One ensemble launch on prepared device tensors.

    ``y0_t``/``p_t`` are ``(N, k)`` tensors (views of structure-of-arrays storage
    cost no copy); ``weights`` is ``(n_vars, N)`` or ``None`` for a unit-weight
    kernel. ``grid`` overrides the number of workgroups (0: one lane per
    trajectory, or the resident grid for a persistent launch). ``order`` is an
    int64 device tensor, a permutation of the trajectories in the order a
    persistent launch claims them (see ``work_order``), or ``"pilot"`` to rank
    them by a short pilot first (``_pilot_order``). Returns the
    ``_common.Outputs``. This is the whole device-side job: the timed region of
    a benchmark is exactly this call.
    """
    import torch

    dev = y0_t.device
    n_vars = y0_t.shape[1]
    n_params = p_t.shape[1]
    y0_s = _common.soa(y0_t)
    p_s = _common.soa(p_t) if n_params else torch.zeros((1, n), dtype=torch.float64, device=dev)
    if weights is None and not built.unit_weights:
        raise ValueError("this kernel was built to read error weights")
    if outputs is None:
        outputs = _common.allocate_outputs(n, times.numel() if save_history else 1, n_vars, dev)
        if hook_size:
            outputs.hook_out = torch.empty((hook_size, n), dtype=torch.float64, device=dev)
    s = _common.launch_stream(stream, dev)
    resume = None
    if isinstance(order, str):
        if order != "pilot":
            raise ValueError(f"work_order must be a permutation or 'pilot', got {order!r}")
        if built.method in ("rodas5p", "tsit5") and built.refill and not hook_size:
            # the solve continues each trajectory where the pilot left it
            resume = torch.empty((_kernels.resume_rows(built.method, n_vars), n),
                                 dtype=torch.float64, device=dev)
        order = _pilot_order(built, y0_s, times, p_s, n, n_vars, n_params, dt0, rtol, atol,
                             weights, outputs, s, resume, max_steps)
        if order is None:
            resume = None  # no pilot ran: nothing to resume
    use_refill = _use_refill(built, n) if refill is None else bool(refill)
    if order is not None:
        if refill is not None and not refill:
            raise ValueError("a work order is a claim order: it needs the persistent (refill) launch")
        use_refill = True
    if use_refill and not built.refill:
        raise ValueError("the wave placement (one trajectory per workgroup) has no persistent "
                         "refill launch")
    handle = built.refill if use_refill else built.plain
    ws_bytes = _runtime.workspace_bytes(handle, n)
    if ws_bytes and workspace is None:
        workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    _runtime.solve_launch(
        handle, s.cuda_stream, int(grid), n, n_vars, n_params, times.numel(), _common.LAYOUT_SOA,
        y0_s.data_ptr(), times.data_ptr(), p_s.data_ptr(), dt0, rtol, atol, max_steps,
        0 if weights is None else weights.data_ptr(), outputs.hist.data_ptr(),
        outputs.accepted.data_ptr(), outputs.rejected.data_ptr(), outputs.loop.data_ptr(),
        outputs.hook_out.data_ptr() if hook_size else 0, int(hook_size),
        0 if workspace is None else workspace.data_ptr(), ws_bytes,
        order=0 if order is None else order.data_ptr(),
        resume=0 if resume is None else resume.data_ptr(),
    )
    _common.used_on(s, dev, y0_s, p_s, times, weights, order, workspace, resume, outputs.hist,
                    outputs.accepted, outputs.rejected, outputs.loop, outputs.hook_out)
    # keep the inputs alive until the stream has consumed them
    outputs._keep = (y0_s, p_s, times, weights, order, workspace, resume)
    outputs.workspace = workspace
    return outputs


#: steps each trajectory takes in the cost pilot of ``work_order="pilot"``. The
#: Rodas5P solve resumes each trajectory where its pilot left it, so the pilot's
#: steps are not taken twice; a longer pilot ranks better, while its
#: one-lane-per-trajectory launch leaves more lanes idle. The 100,000-trajectory
#: uneven stiff ensemble (FP32 / refined FP32 LU): 40 steps 570 / 1,171 ms,
#: 80 steps 551 / 1,090 ms, 160 steps 593 / 1,196 ms.
PILOT_STEPS = 80


def _pilot_order(built, y0_s, times, p_s, n, n_vars, n_params, dt0, rtol, atol, weights,
                 outputs, stream, resume=None, max_steps=PILOT_STEPS):
    """A claim order from a short pilot (``mdx_cost_pilot_launch``): every
    trajectory takes ``PILOT_STEPS`` steps in the one-lane-per-trajectory
    kernel, the steps it has left at its current step size rank it, costliest
    first. The pilot's saves go to ``outputs``; with a ``resume`` buffer
    (``_kernels.resume_rows`` by N) it also leaves each trajectory's step state
    there and the solve continues from it (``mdx_solve_launch_resumed``), else
    the solve starts over and overwrites them. The pilot takes no more steps than the
    solve's ``max_steps`` allows (a resumed trajectory carries its count on).
    Nothing leaves the device."""
    import torch

    if max_steps < 1:
        return None  # nothing to rank: the solve takes no step
    cost = torch.empty(n, dtype=torch.float64, device=y0_s.device)
    _runtime.cost_pilot_launch(
        built.plain, stream.cuda_stream, n, n_vars, n_params, times.numel(), _common.LAYOUT_SOA,
        y0_s.data_ptr(), times.data_ptr(), p_s.data_ptr(), dt0, rtol, atol,
        min(PILOT_STEPS, int(max_steps)),
        0 if weights is None else weights.data_ptr(), outputs.hist.data_ptr(),
        outputs.accepted.data_ptr(), outputs.rejected.data_ptr(), outputs.loop.data_ptr(),
        cost.data_ptr(), resume=0 if resume is None else resume.data_ptr())
    _common.used_on(stream, cost.device, cost)
    with torch.cuda.stream(stream):
        return torch.argsort(cost, descending=True, stable=True)


def _tableau(choice, n_vars, n, placement, max_registers):
    """``tableau_in_registers`` as the kernel options take it: the caller's
    choice, else the size rule for this device."""
    import torch

    if choice is not None:
        return bool(choice)
    n_cu = torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count
    return _kernels.tableau_in_registers(n_vars, n, n_cu, placement, max_registers)


def _wave(options, n_vars, n):
    """The plain solve's placement: the caller's, else the wave placement when
    the size rule picks it (``_kernels.wave_placement``)."""
    import torch

    if (options.placement is not None or options.max_registers is not None
            or options.lu_refine):
        return options.placement
    n_cu = torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count
    return _kernels.wave_placement(n_vars, n, n_cu, None, options.sparsity)


def _small_ensemble_block(options, n_aug, n):
    """``options`` with the workgroup size ``_kernels.rodas5p_block`` picks for
    a plain launch of ``n`` trajectories whose joint vector is ``n_aug`` long
    (the caller gave none)."""
    import torch

    if options.max_registers is not None:
        return options
    n_cu = torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count
    return replace(options, trajectories_per_block=_kernels.rodas5p_block(
        None, n_aug, options.lu_precision, n, n_cu, options.placement, options.sparsity,
        options.lu_refine))


def _sized(options, ode_fn, n_vars, n_params, n, requested_block, plain=True,
           tableau_by_rule=False):
    """``options`` of a plain solve of ``n`` trajectories by the size rules:
    where the caller left them open, a team (``_kernels.rodas5p_team``), the
    wave placement and a small ensemble's workgroup (``plain``: not for a
    persistent launch), an unrolled step's lanes a trajectory and workgroup
    (``_kernels.time_lanes``, ``_kernels.register_block``);
    ``tableau_by_rule``: ``_fitting_tableau`` applies."""
    if requested_block is None and _kernels.rodas5p_team(ode_fn, n_vars, n_params, options):
        return replace(options, placement=_kernels.TEAM,
                       trajectories_per_block=_kernels.DEFAULT_BLOCK)
    if plain:
        options = replace(options, placement=_wave(options, n_vars, n))
        if requested_block is None:
            options = _small_ensemble_block(options, n_vars, n)
    if (requested_block is None and n_vars <= _kernels.UNROLLED_MAX_VARS
            and options.placement in (None, "registers") and options.max_registers is None):
        lanes = (_kernels.time_lanes(ode_fn, n_vars, n_params, options, n, _common.n_cu())
                 if plain else 1)
        options = replace(options, lanes=lanes, trajectories_per_block=_kernels.register_block(
            n * lanes, _common.n_cu()) // lanes)
        if tableau_by_rule:
            options = _fitting_tableau(options, ode_fn, n_vars, n_params, n)
    return options


def _fitting_tableau(options, ode_fn, n_vars, n_params, n):
    """``options`` without the size rule's tableau in registers where an
    ensemble of more than a wavefront a SIMD would find only one resident with
    it: a right-hand side with calls, a save hook. (3 variables with ``exp``,
    FP64, 120,000 trajectories: 129 ms with it, 113 without; Robertson with a
    hook, FP64, 78,113: 0.94 and 0.58 ms.) Such ensembles come to at most two,
    so the kernel without it is bounded to two at most: with three resident the
    dispatcher gives some SIMDs three (Robertson FP64, 120,000: 746 us with
    three, 585 with two)."""
    if (options.tableau_in_registers and n > 4 * 64 * _common.n_cu()
            and _kernels.rodas5p_kernel(ode_fn, n_vars, n_params, options).extra["vgprs"]
            > _kernels.RESIDENT_VGPRS[2]):
        return replace(options, tableau_in_registers=False, resident=2)
    return options


def _adjoint_options(options, n_vars, n, requested_block):
    """``options`` for the adjoint kernel of an ensemble of ``n``: the rolled
    adjoint (more than ``ADJOINT_UNROLLED_MAX_VARS`` variables) takes the
    placement, workgroup size and stage cache of ``_kernels.adjoint_block`` unless the
    caller chose a workgroup size, a register cap or a placement other than
    LDS, or the pattern's sparse routines are table driven
    (``_kernels.adjoint_lds_supported``). A caller's team placement is the
    forward solve's: the team's adjoint has no checkpoints and comes in through
    ``_whole_adjoint`` alone."""
    options = _without_team(options)
    if (requested_block is not None or options.max_registers is not None
            or options.placement not in (None, "lds")
            or n_vars <= _kernels.ADJOINT_UNROLLED_MAX_VARS
            or not _kernels.adjoint_lds_supported(options.sparsity, options.ordering)):
        return options
    placement, block, cache = _kernels.adjoint_block(
        n_vars, _kernels.lu_size(n_vars, options.sparsity, options.ordering),
        options.lu_precision, n, _common.n_cu())
    return replace(options, placement=placement, trajectories_per_block=block,
                   adjoint_cache=cache)


def _without_team(options):
    """``options`` with a caller's team placement left to the size rules."""
    if options.placement == _kernels.TEAM:
        return replace(options, placement=None)
    return options


def _whole_adjoint(options, ode_fn, n_vars, n_params, n, requested_block) -> dict:
    """The ``AdjointJob`` fields of an adjoint kernel for an ensemble of ``n``
    that needs room for every step's record: the team's
    (``_kernels.rodas5p_adjoint_team``), or the unrolled one that keeps the
    stage vectors; none of them elsewhere."""
    options = _without_team(options)
    block = 0 if requested_block is not None else _kernels.rodas5p_adjoint_team(
        ode_fn, n_vars, n_params, options, n, _common.n_cu())
    if block:
        whole = replace(options, placement=_kernels.TEAM, trajectories_per_block=block)
    elif _kernels.adjoint_keeps_stages(n_vars, options, n, _common.n_cu()):
        whole = replace(options, adjoint_keep=True)
    else:
        return {}
    return dict(whole=lambda: _kernels.rodas5p_adjoint_kernel(ode_fn, n_vars, n_params, whole),
                whole_words=_kernels.adjoint_record_words(n_vars, whole))


def _adjoint_kernels(options, ode_fn, n_vars, n_params, n, requested_block, ckpt_every) -> dict:
    """The ``AdjointJob`` fields of a gradient's adjoint kernels: the one
    expected to run is built now, as the solve's own kernel is; the checkpoints'
    beside one that records every step only if it comes to that (compiling an
    adjoint takes 5-15 s for a system's first gradient)."""
    checkpoints = functools.partial(
        _kernels.rodas5p_adjoint_kernel, ode_fn, n_vars, n_params,
        _adjoint_options(options, n_vars, n, requested_block))
    whole = _whole_adjoint(options, ode_fn, n_vars, n_params, n, requested_block)
    if whole and int(ckpt_every) >= _autodiff.DEFAULT_CKPT_EVERY:
        whole["whole"]()
    else:
        checkpoints()
    return dict(adjoint=checkpoints, **whole)


def _use_refill(built, n):
    if not built.refill:
        return False  # a wave-per-trajectory kernel has no persistent form
    handle = built.refill
    grid = _runtime.persistent_grid(handle)
    return n > grid * built.block * _REFILL_MIN_WAVES_PER_CU


def finish(out, return_stats, as_numpy):
    hist = out.ensemble_view()
    stats = _common.solver_stats(out.accepted, out.rejected, out.loop)
    if as_numpy:
        hist = hist.cpu().numpy()
        stats = {k: v.cpu().numpy() for k, v in stats.items()}
    if return_stats:
        return hist, stats
    return hist


def _traced(ode_fn, y0, t_span, params, *, rtol=1e-8, atol=1e-10, first_step=None,
            max_steps=100000, return_stats=False, error_weights=None, pcoeff=0.0, icoeff=1.0,
            dcoeff=0.0, lu_precision="fp32", trajectories_per_block=None,
            sens_error_control=True, sens_param_columns=None, sparsity=None, ordering="amd",
            tf_index=None, max_registers=None, array_rhs=None, save_hook=None, hook_size=0,
            save_history=True, refill=None, stream=None, work_order=None, placement=None,
            adjoint=False, ckpt_every=64, tableau_in_registers=None, lu_refine=False):
    """``solve`` while ``torch.compile`` traces it: the custom operator for a
    plain solve (gradients through the adjoint kernel, ``adjoint=True``), or
    NotImplemented for what only the eager path does (error weights, hooks,
    array right-hand sides, streams, claim orders, forward-sensitivity
    gradients)."""
    from . import _ops

    if (error_weights is not None or array_rhs is not None or save_hook is not None
            or not save_history or stream is not None or work_order is not None
            or lu_refine):
        return NotImplemented
    options = (("pcoeff", float(pcoeff)), ("icoeff", float(icoeff)), ("dcoeff", float(dcoeff)),
               ("lu_precision", lu_precision),
               ("trajectories_per_block", trajectories_per_block),
               ("ordering", ordering), ("tf_index", -1 if tf_index is None else int(tf_index)),
               ("max_registers", max_registers), ("unit_weights", True),
               ("placement", placement))
    return _ops.traced_solve("rodas5p", ode_fn, y0, t_span, params, options=options,
                             sparsity=sparsity, tableau=tableau_in_registers, rtol=rtol,
                             atol=atol, first_step=first_step, max_steps=max_steps,
                             refill=refill, adjoint=adjoint, ckpt_every=ckpt_every,
                             return_stats=return_stats)


# Traced by torch.compile, a plain solve is one custom operator (menodax::
# ensemble_solve); everything else runs eagerly (see _common.eager_only).
solve = _common.compilable(solve, _traced)
adjoint_gradients = _common.eager_only(adjoint_gradients)
solve_sensitivities = _common.eager_only(solve_sensitivities)
