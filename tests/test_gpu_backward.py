"""Native float32 backward of the matrix tick (ns_dendritic_step_backward)
against the oracle's gradients.

The reference's native runtime records no graph of its own: whenever a
gradient is needed it runs its torch step (native_compartmental.py:104-108),
and autograd differentiates torch.sparse.mm and the update ops.  Here the
same gradients come from HIP kernels.  The expected values come from
oracle/grad.py: float64 autograd through the oracle's update on the dense
weight matrix, pinned by finite differences (tests/test_oracle_grad.py), on
the same float32 inputs, so the tolerance (1e-4 of the largest gradient of
each tensor) covers only the native float32 arithmetic.  Covers one tick with every input requiring a
gradient (states, [B,N] and [B,1] drives, the six parameters, the weights),
eight-tick backpropagation through time, scalar drives, stride-0 parameters,
repeatability, and the source-major weight copy the transposed product streams
from the second backward of a weight version on.
"""

from __future__ import annotations

import copy

import numpy as np
import pytest
import torch

from oracle import grad as og
from oracle import topology as otop
from neurosim_gpu import (DendriticDynamics, Dynamics, NativeDendriticMatrixRuntime,
                          SparseTopology)

pytestmark = pytest.mark.gpu


def graph(n: int, m: int, seed: int) -> otop.Graph:
    return otop.random_graph(n, m, seed=seed)


def topology(g: otop.Graph, dtype, device) -> SparseTopology:
    fields = dict(src=g.src, dst=g.dst, weight=g.weight, out_rowptr=g.out_rowptr,
                  in_rowptr=g.in_rowptr, in_col=g.in_col, out_weight_index=g.out_weight_index,
                  in_weight=g.in_weight)
    tensors = {k: torch.from_numpy(np.asarray(v)) for k, v in fields.items()}
    for k in ("weight", "in_weight"):
        tensors[k] = tensors[k].to(dtype)
    return SparseTopology(n_neurons=g.n, **{k: v.to(device) for k, v in tensors.items()})


def leaf(value: np.ndarray, dtype, device) -> torch.Tensor:
    return torch.tensor(value, dtype=dtype, device=device).requires_grad_(True)


def model(values: dict, dtype, device, expanded: bool) -> DendriticDynamics:
    def vec(name):
        if expanded and name in ("coupling", "strength"):
            return leaf(values[name][:1], dtype, device)[0].expand(values["alpha"].size)
        return leaf(values[name], dtype, device)
    return DendriticDynamics(Dynamics(vec("alpha"), vec("gain")), vec("rho_d"), vec("rho_a"),
                             vec("coupling"), vec("strength"))


def params_of(m: DendriticDynamics):
    return [m.soma.alpha, m.soma.gain, m.dendrite_decay, m.adaptation_decay, m.coupling,
            m.adaptation_strength]


def base(p):
    """The leaf behind a parameter (an expanded scalar's 0-d base)."""
    return p._base if p._base is not None else p


def run(runtime_cls, g, inputs, dtype, device, ticks, *, scalar_drives, expanded,
        source_major=True, transposed_panels=True, **kw):
    topo = topology(g, dtype, device)
    topo.in_weight.requires_grad_(True)
    mdl = model(inputs["params"], dtype, device, expanded)
    state0 = leaf(inputs["state"], dtype, device)
    rt = runtime_cls(topo, mdl, state0.detach(), **kw)
    if hasattr(rt, "source_major_weights"):
        rt.source_major_weights.enabled = source_major
    if hasattr(rt, "transposed_panels_enabled"):
        rt.transposed_panels_enabled = transposed_panels
    rt.state = state0
    rt.dendritic_state = leaf(inputs["dendrite"], dtype, device)
    rt.adaptation_state = leaf(inputs["adaptation"], dtype, device)
    dendrite0, adaptation0 = rt.dendritic_state, rt.adaptation_state
    if scalar_drives:
        drive, dendritic = 0.2, 0.1
    else:
        drive = leaf(inputs["drive"], dtype, device)
        dendritic = leaf(inputs["dendritic"], dtype, device)
    for _ in range(ticks):
        rt.step(drive, dendritic_drive=dendritic)
    r = {k: torch.tensor(v, dtype=dtype, device=device) for k, v in inputs["probe"].items()}
    loss = (rt.state * r["s"]).sum() + (rt.dendritic_state * r["d"]).sum() + \
        (rt.adaptation_state * r["a"]).sum()
    loss.backward()
    grads = {"weight": topo.in_weight.grad, "state": state0.grad, "dendrite": dendrite0.grad,
             "adaptation": adaptation0.grad}
    if not scalar_drives:
        grads["drive"], grads["dendritic"] = drive.grad, dendritic.grad
    for name, p in zip(("alpha", "gain", "rho_d", "rho_a", "coupling", "strength"), params_of(mdl)):
        grads[name] = base(p).grad
    return grads, rt


def inputs_for(g, batch, seed):
    rng = np.random.default_rng(seed)
    n = g.n
    return {
        "state": rng.uniform(0, 1, (batch, n)), "dendrite": rng.uniform(-1, 1, (batch, n)),
        "adaptation": rng.uniform(0, 1, (batch, n)),
        "drive": rng.uniform(-0.5, 0.8, (batch, n)), "dendritic": rng.uniform(-0.3, 0.3, (batch, 1)),
        "params": {"alpha": rng.uniform(0.5, 0.9, n), "gain": rng.uniform(0.5, 1.5, n),
                   "rho_d": rng.uniform(0.5, 0.95, n), "rho_a": rng.uniform(0.8, 0.99, n),
                   "coupling": rng.uniform(0.2, 0.8, n), "strength": rng.uniform(0.05, 0.4, n)},
        "probe": {"s": rng.standard_normal((batch, n)), "d": rng.standard_normal((batch, n)),
                  "a": rng.standard_normal((batch, n))},
    }


def oracle_gradients(g, inputs, ticks, *, scalar_drives, expanded) -> dict:
    """The oracle's gradients on the inputs as the native run sees them
    (rounded to float32), keyed like ``run``'s."""
    f32 = lambda v: np.asarray(v, np.float32).astype(np.float64)  # noqa: E731
    n = g.n
    params = {}
    for name, key in zip(og.PARAM_NAMES, ("alpha", "gain", "rho_d", "rho_a", "coupling", "strength")):
        value = f32(inputs["params"][key])
        params[name] = np.full(n, value[0]) if expanded and key in ("coupling", "strength") else value
    x = og.TickInputs(state=f32(inputs["state"]), dendrite=f32(inputs["dendrite"]),
                      adaptation=f32(inputs["adaptation"]),
                      drive=0.2 if scalar_drives else f32(inputs["drive"]),
                      dendritic=0.1 if scalar_drives else f32(inputs["dendritic"]),
                      params=params, probe={k: f32(inputs["probe"][k]) for k in ("s", "d", "a")})
    got = og.tick_gradients(g, x, ticks)
    out = {"weight": got["weight"], "state": got["state"], "dendrite": got["dendrite"],
           "adaptation": got["adaptation"]}
    if not scalar_drives:
        out["drive"], out["dendritic"] = got["drive"], got["dendritic"]
    for name in og.PARAM_NAMES:
        value = got[name]
        if expanded and name in ("coupling", "strength"):
            value = value.sum()                  # the gradient of the 0-d base
        out[name] = value
    return {k: torch.from_numpy(np.asarray(v, np.float64)) for k, v in out.items()}


def compare(native: dict, reference: dict, rtol: float = 1e-4) -> None:
    assert native.keys() == reference.keys()
    for name, want in reference.items():
        got = native[name]
        assert got is not None and want is not None, name
        got = got.detach().double().cpu().reshape(want.shape)
        scale = float(want.abs().max())
        err = float((got - want.cpu()).abs().max())
        assert err <= rtol * max(scale, 1e-12), f"{name}: max error {err:.3e}, scale {scale:.3e}"


@pytest.mark.parametrize("ticks,batch,scalar_drives,expanded", [
    (1, 3, False, False), (1, 1, True, True), (8, 2, False, True), (8, 4, True, False)])
def test_gradients_match_the_oracle(gpu, ticks, batch, scalar_drives, expanded):
    print(f"case backward ticks={ticks} batch={batch} scalar_drives={scalar_drives} "
          f"expanded={expanded}", flush=True)
    g = graph(600, 12_000, 9)
    inputs = inputs_for(g, batch, ticks * 10 + batch)
    kw = dict(scalar_drives=scalar_drives, expanded=expanded)
    native, rt = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, ticks, **kw)
    assert rt.last_backend == "native-autograd"
    compare(native, oracle_gradients(g, inputs, ticks, **kw))


@pytest.mark.parametrize("ticks,batch,width", [(2, 1, 1000), (4, 2, 1000), (3, 1, None)])
def test_transposed_product_on_panels_matches_the_oracle(gpu, ticks, batch, width):
    """With the forward on column panels the backward's transposed product
    W^T @ g runs, from the second backward of a weight version on, on a panel
    layout of the transposed matrix (rows = sources; three panels at width
    1000, so a second kernel adds the per-panel sums into d_state); the
    gradients through several ticks match the oracle, and the out-edge walk
    to float32 summation order."""
    print(f"case backward transposed panels ticks={ticks} batch={batch} width={width}",
          flush=True)
    g = graph(3000, 90_000, 17)
    inputs = inputs_for(g, batch, 40 + batch)
    kw = dict(scalar_drives=False, expanded=False, kernel="panels", panel_width=width)
    native, rt = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, ticks, **kw)
    assert rt._transposed is not None and rt._transposed._seen == ticks
    assert rt._transposed.layout._slot_weights is not None     # the panels ran
    assert rt._transposed.layout.n_panels == (3 if width else 1)
    compare(native, oracle_gradients(g, inputs, ticks, scalar_drives=False, expanded=False))
    walked, rt2 = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, ticks,
                      transposed_panels=False, **kw)
    assert rt2._transposed is None
    compare(native, {k: v.detach().double().cpu() for k, v in walked.items()}, rtol=1e-5)


@pytest.mark.parametrize("batch", [1, 2])
def test_first_backward_of_a_weight_version_reads_the_weights_in_place(gpu, batch):
    """One recorded tick per weight version (an optimizer step before every pass):
    the transposed product runs on the indexed plan, reading the CSR weights
    through the slots' edge numbers, where it used to walk the out-edges.  The
    gradients match the oracle and equal bitwise those of a second backward of the
    same version, which streams the slot-order copy."""
    print(f"case backward indexed transposed plan batch={batch}", flush=True)
    g = graph(3000, 90_000, 17)
    inputs = inputs_for(g, batch, 60 + batch)
    kw = dict(scalar_drives=False, expanded=False, kernel="panels", panel_width=1000)
    first, rt = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, 1, **kw)
    assert rt._transposed is not None and rt._transposed._seen == 1
    assert rt._transposed.layout._slot_weights is None      # the indexed plan ran
    compare(first, oracle_gradients(g, inputs, 1, scalar_drives=False, expanded=False))

    def again():
        """The same tick and loss once more, on the same weights (leaves reset)."""
        topo, mdl = rt.topology, rt.compartment_dynamics
        for t in [topo.in_weight, *params_of(mdl)]:
            base(t).grad = None
        state0 = leaf(inputs["state"], torch.float32, gpu)
        rt.state = state0
        rt.dendritic_state = leaf(inputs["dendrite"], torch.float32, gpu)
        rt.adaptation_state = leaf(inputs["adaptation"], torch.float32, gpu)
        drive = leaf(inputs["drive"], torch.float32, gpu)
        dendritic = leaf(inputs["dendritic"], torch.float32, gpu)
        rt.step(drive, dendritic_drive=dendritic)
        r = {k: torch.tensor(v, dtype=torch.float32, device=gpu)
             for k, v in inputs["probe"].items()}
        loss = (rt.state * r["s"]).sum() + (rt.dendritic_state * r["d"]).sum() + \
            (rt.adaptation_state * r["a"]).sum()
        loss.backward()
        return {"weight": topo.in_weight.grad, "state": state0.grad}

    second = again()
    assert rt._transposed.layout._slot_weights is not None  # the slot-order copy ran
    for name in second:
        assert torch.equal(first[name], second[name]), name


def test_backward_is_repeatable(gpu):
    print("case backward repeatable", flush=True)
    g = graph(2000, 60_000, 3)
    inputs = inputs_for(g, 2, 5)
    first, _ = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, 4,
                   scalar_drives=False, expanded=False)
    second, _ = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, 4,
                    scalar_drives=False, expanded=False)
    for name in first:
        assert torch.equal(first[name], second[name]), name


def test_source_major_weight_copy_changes_no_gradient(gpu):
    """Backpropagation through 6 ticks: from the second backward on, the transposed
    product streams a source-major copy of the weights instead of gathering them;
    the gradients are bitwise those of the gather."""
    print("case backward source-major weights", flush=True)
    g = graph(3000, 90_000, 12)
    inputs = inputs_for(g, 2, 21)
    kw = dict(scalar_drives=False, expanded=False)
    copied, rt = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, 6, **kw)
    assert rt.source_major_weights._values is not None, "the copy was built"
    assert rt.source_major_weights._seen == 6
    gathered, rt2 = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, 6,
                        source_major=False, **kw)
    assert rt2.source_major_weights._values is None
    for name in copied:
        assert torch.equal(copied[name], gathered[name]), name


def test_recorded_ticks_move_to_panels_for_a_reused_weight_version(gpu):
    """A recorded tick takes the row kernel the first time it sees a weight
    version and the panel kernel from the second on; an in-place weight update
    sends it back to the row kernel.  The states follow the inference ticks
    (panels) to float32 summation-order differences."""
    print("case backward recorded panel ticks", flush=True)
    g = graph(4000, 100_000, 6)
    topo = topology(g, torch.float32, gpu)
    topo.in_weight.requires_grad_(True)
    soma = Dynamics(torch.full((4000,), .72, device=gpu), torch.full((4000,), .8, device=gpu))
    mdl = DendriticDynamics.from_time_constants(soma, dt=1., tau_dendrite=4., tau_adaptation=25.)
    plain = NativeDendriticMatrixRuntime(topo, mdl, torch.zeros(1, 4000, device=gpu),
                                         kernel="panels")
    recorded = NativeDendriticMatrixRuntime(topo, mdl, torch.zeros(1, 4000, device=gpu),
                                            kernel="panels")
    assert recorded.kernel == "panels"
    for tick in range(5):
        with torch.no_grad():
            plain.step(0.2, dendritic_drive=0.1)
        recorded.step(0.2, dendritic_drive=0.1)
        assert (recorded._panel_struct_key is not None) == (tick >= 1)
    for name in ("state", "dendritic_state", "adaptation_state"):
        err = float((getattr(recorded, name) - getattr(plain, name)).abs().max())
        assert err <= 2e-6, (name, err)
    recorded.state.sum().backward()
    assert topo.in_weight.grad is not None and bool(torch.isfinite(topo.in_weight.grad).all())
    with torch.no_grad():
        topo.in_weight.mul_(0.5)                 # a new weight version: rows again, once
    recorded.step(0.2, dendritic_drive=0.1)
    assert recorded._recorded_seen == 1


def test_forward_of_a_recorded_tick_equals_the_inference_tick(gpu):
    """Recording for autograd changes nothing in the forward values."""
    print("case backward forward values", flush=True)
    g = graph(1000, 20_000, 0)
    topo = topology(g, torch.float32, gpu)
    soma = Dynamics(torch.full((1000,), .72, device=gpu), torch.full((1000,), .8, device=gpu))
    mdl = DendriticDynamics.from_time_constants(soma, dt=1., tau_dendrite=4., tau_adaptation=25.)
    plain = NativeDendriticMatrixRuntime(topo, mdl, torch.zeros(2, 1000, device=gpu), kernel="rows")
    recorded = NativeDendriticMatrixRuntime(topo, mdl, torch.zeros(2, 1000, device=gpu), kernel="rows")
    drive = torch.full((2, 1000), 0.2, device=gpu, requires_grad=True)
    for _ in range(5):
        with torch.no_grad():
            plain.step(drive.detach(), dendritic_drive=0.1)
        recorded.step(drive, dendritic_drive=0.1)
    assert recorded.last_backend == "native-autograd"
    assert torch.equal(plain.state, recorded.state.detach())
    assert torch.equal(plain.dendritic_state, recorded.dendritic_state.detach())


@pytest.mark.parametrize("n,m,batch", [
    (5, 12, 1), (300, 200, 2), (300, 900, 3), (257, 4000, 4), (130, 9000, 5), (200, 4000, 8),
    (64, 3000, 12), (100, 2000, 16), (90, 1500, 17), (80, 1600, 20)])
def test_edge_kernels_at_every_batch_form(gpu, n, m, batch):
    """The backward's edge kernels take whole neuron-major rows (batch 2 or a multiple
    of 4) or one column per lane, in lane groups sized to the mean degree: two ticks,
    so the second's state is neuron-major and the first's is not, from fewer than one
    edge per row to more than a wavefront's worth."""
    print(f"case backward forms n={n} m={m} batch={batch}", flush=True)
    g = graph(n, m, 31 + batch)
    inputs = inputs_for(g, batch, 70 + batch)
    kw = dict(scalar_drives=False, expanded=False)
    native, _ = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, 2, **kw)
    compare(native, oracle_gradients(g, inputs, 2, **kw))


@pytest.mark.parametrize("batch,kernel,walk", [(1, "panels", False), (2, "rows", True),
                                               (8, "rows", True)])
def test_start_state_without_gradient_changes_no_other_gradient(gpu, monkeypatch, batch, kernel,
                                                                walk):
    """A start state that needs no gradient leaves out the first tick's transposed
    product; with it (and with a row-major state copied to neuron-major first) the
    other gradients are bitwise the same."""
    print(f"case backward start state batch={batch} kernel={kernel}", flush=True)
    from neurosim_gpu import native_compartmental as nc

    g = graph(1500, 30_000, 4)
    inputs = inputs_for(g, batch, 90 + batch)
    results = {}
    for mode in ("full", "leaf", "copied"):
        monkeypatch.setattr(nc, "RELAYOUT_MIN_GATHERS", 0 if mode == "copied" else 1 << 60)
        topo = topology(g, torch.float32, gpu)
        topo.in_weight.requires_grad_(True)
        mdl = model(inputs["params"], torch.float32, gpu, False)
        state0 = leaf(inputs["state"], torch.float32, gpu)
        rt = NativeDendriticMatrixRuntime(topo, mdl, state0.detach(), kernel=kernel)
        rt.state = state0 if mode == "full" else state0.detach()
        rt.step(0.2, dendritic_drive=0.1)
        rt.step(0.3, dendritic_drive=0.1)
        (rt.state * rt.state).sum().backward()
        results[mode] = [topo.in_weight.grad, *(p.grad for p in params_of(mdl))]
        if mode != "full":
            assert (rt.source_major_weights._seen if walk else rt._transposed._seen) == 1
    # The copied state is read whole rows at a time, so its weight gradient may sum the
    # columns in another order: at most a few units in the last place of the terms.
    for a, b, c in zip(*(results[m] for m in ("full", "leaf", "copied"))):
        assert torch.equal(a, b)
        assert float((a - c).abs().max()) <= batch * 2.0 ** -22 * float(a.abs().max())


@pytest.mark.parametrize("batch,kernel", [(1, "panels"), (3, "rows"), (8, "rows")])
def test_gradients_summed_through_the_ticks_equal_separate_ones(gpu, batch, kernel):
    """A run of recorded ticks hands its weight and parameter gradients from tick to
    tick, each backward adding to them in place.  Against ticks recorded one by one
    (autograd adds their gradients, in the same order): bitwise, also through a second
    backward of the same graph, with some parameters frozen, and for a loss that leaves
    out the last ticks (the weight gradient to float32 rounding: it comes two ticks at
    a time)."""
    print(f"case backward linked ticks batch={batch} kernel={kernel}", flush=True)
    g = graph(900, 20_000, 8)
    inputs = inputs_for(g, batch, 50 + batch)

    def gradients(linked: bool, frozen: bool, early: bool):
        topo = topology(g, torch.float32, gpu)
        topo.in_weight.requires_grad_(True)
        mdl = model(inputs["params"], torch.float32, gpu, False)
        if frozen:
            mdl.soma.gain.requires_grad_(False)
            mdl.coupling.requires_grad_(False)
        rt = NativeDendriticMatrixRuntime(topo, mdl, torch.full((batch, 900), .3, device=gpu),
                                          kernel=kernel)
        states = []
        for t in range(4):
            rt.step(0.1 * t, dendritic_drive=0.1)
            states.append(rt.state)
            if not linked:
                rt._recording = None
        loss = (states[1 if early else 3] ** 2).sum() + (states[1] * 0.5).sum()
        wanted = [topo.in_weight, *(p for p in params_of(mdl) if p.requires_grad)]
        first = torch.autograd.grad(loss, wanted, retain_graph=True)
        second = torch.autograd.grad(loss, wanted)
        return first, second

    for frozen in (False, True):
        for early in (False, True):
            one, again = gradients(True, frozen, early)
            separate, _ = gradients(False, frozen, early)
            for k, (a, b, c) in enumerate(zip(one, separate, again)):
                if k == 0:
                    # Two ticks' weight gradients come from one chain of fused multiply-adds
                    # over 2B columns instead of two chains and an addition: at most two
                    # roundings of the partial sums (below twice the largest gradient) per term.
                    assert float((a - b).abs().max()) <= 8 * batch * 2.0 ** -23 * \
                        float(a.abs().max())
                else:
                    assert torch.equal(a, b)
                # the second backward recomputes j = W @ s on row blocks
                assert float((a - c).abs().max()) <= 1e-5 * float(a.abs().max())


def test_a_run_of_recorded_ticks_ends_where_its_inputs_change(gpu):
    """Detached states, restored states, an in-place update and a newly trained
    parameter each start a new run; gradients then match ticks recorded one by one."""
    print("case backward run boundaries", flush=True)
    g = graph(500, 6_000, 2)
    inputs = inputs_for(g, 2, 12)

    def gradients(linked: bool):
        topo = topology(g, torch.float32, gpu)
        topo.in_weight.requires_grad_(True)
        mdl = model(inputs["params"], torch.float32, gpu, False)
        mdl.coupling.requires_grad_(False)
        rt = NativeDendriticMatrixRuntime(topo, mdl, torch.full((2, 500), .3, device=gpu))

        def step(u):
            rt.step(u, dendritic_drive=0.1)
            if not linked:
                rt._recording = None

        step(0.1)
        step(0.2)
        kept = (rt.state, rt.dendritic_state, rt.adaptation_state)
        step(0.3)
        loss = rt.state.sum()
        rt.state, rt.dendritic_state, rt.adaptation_state = kept    # a second branch
        mdl.coupling.requires_grad_(True)
        step(0.4)
        step(0.1)
        loss = loss + (rt.state * 2).sum()
        rt.state = rt.state.detach()                                # truncated
        step(0.2)
        loss = loss + (rt.state ** 2).sum()
        return torch.autograd.grad(loss, [topo.in_weight, *params_of(mdl)])

    for a, b in zip(gradients(True), gradients(False)):
        # branches meet in another order of additions: a few roundings of the sum
        assert float((a - b).abs().max()) <= 2.0 ** -20 * float(b.abs().max())


@pytest.mark.parametrize("batch,kernel", [(1, "panels"), (3, "rows")])
@pytest.mark.parametrize("how", ["copy", "rewind"])
def test_a_run_is_continued_once(gpu, batch, kernel, how):
    """A simulation branched by a shallow copy of its runtime, or rewound to saved
    attributes: both branches start from the same recorded states, and only one may
    continue that run.  Gradients match those of ticks recorded one by one."""
    print(f"case backward branches batch={batch} kernel={kernel} {how}", flush=True)
    g = graph(500, 6_000, 6)
    inputs = inputs_for(g, batch, 21)

    def gradients(linked: bool):
        topo = topology(g, torch.float32, gpu)
        topo.in_weight.requires_grad_(True)
        mdl = model(inputs["params"], torch.float32, gpu, False)
        rt = NativeDendriticMatrixRuntime(topo, mdl, torch.full((batch, 500), .3, device=gpu),
                                          kernel=kernel)

        def step(runtime, u):
            runtime.step(u, dendritic_drive=0.1)
            if not linked:
                runtime._recording = None

        for u in (0.1, 0.2):
            step(rt, u)
        other = copy.copy(rt)
        kept = dict(vars(rt))
        step(rt, 0.5)              # odd numbers of ticks: both branches leave an entry pending
        loss = (rt.state ** 2).sum()
        if how == "rewind":
            vars(rt).update(kept)
            other = rt
        for u in (0.1, 0.4, 0.2):
            step(other, u)
        loss = loss + (other.state * 0.7).sum()
        return torch.autograd.grad(loss, [topo.in_weight, *params_of(mdl)])

    for a, b in zip(gradients(True), gradients(False)):
        # Five ticks of at most three columns meet in another order: 15 additions of
        # partial sums below twice the largest gradient.
        assert float((a - b).abs().max()) <= 2.0 ** -19 * float(b.abs().max())


@pytest.mark.parametrize("ticks", [2, 3])
@pytest.mark.parametrize("batch,kernel", [(1, "panels"), (3, "rows")])
def test_recorded_ticks_pass_anomaly_detection(gpu, batch, kernel, ticks):
    """No gradient that a tick hands on holds memory it has not written: with new memory
    filled with NaN, a backward under anomaly detection (which refuses NaN in any
    gradient, those between the ticks among them) passes and gives the gradients of
    ticks recorded one by one."""
    print(f"case backward anomaly batch={batch} kernel={kernel} ticks={ticks}", flush=True)
    g = graph(500, 6_000, 3)
    inputs = inputs_for(g, batch, 33)

    def gradients(linked: bool):
        topo = topology(g, torch.float32, gpu)
        topo.in_weight.requires_grad_(True)
        mdl = model(inputs["params"], torch.float32, gpu, False)
        rt = NativeDendriticMatrixRuntime(topo, mdl, torch.full((batch, 500), .3, device=gpu),
                                          kernel=kernel)
        for t in range(ticks):
            rt.step(0.1 + 0.1 * t, dendritic_drive=0.1)
            if not linked:
                rt._recording = None
        return torch.autograd.grad(rt.state, [topo.in_weight, *params_of(mdl)],
                                   grad_outputs=torch.ones_like(rt.state))

    separate = gradients(False)
    before = torch.are_deterministic_algorithms_enabled()
    torch.use_deterministic_algorithms(True, warn_only=True)    # fills new memory with NaN
    try:
        with torch.autograd.set_detect_anomaly(True):
            linked = gradients(True)
    finally:
        torch.use_deterministic_algorithms(before)
    for a, b in zip(linked, separate):
        # 3 ticks' products of at most 3 columns, summed two ticks at a time: nine
        # additions of partial sums below twice the largest gradient.
        assert float((a - b).abs().max()) <= 2.0 ** -19 * float(b.abs().max())


@pytest.mark.skip(reason="capturing a backward ended the process with a segmentation fault in "
                  "the runtime's end of capture, cause not known; it is refused since")
@pytest.mark.parametrize("batch,kernel,blocked", [(1, "panels", True), (1, "panels", False),
                                                  (3, "rows", False)])
@pytest.mark.parametrize("ticks", [1, 3])
def test_captured_training_pass_follows_its_weights(gpu, monkeypatch, batch, kernel, blocked,
                                                    ticks):
    """A forward and backward captured after one eager pass on the same weight version:
    replays after in-place updates of the weights give the states and gradients of eager
    passes on the new weights, the transposed product's among them."""
    print(f"case backward capture batch={batch} kernel={kernel} blocked={blocked} "
          f"ticks={ticks}", flush=True)
    from neurosim_gpu import native_compartmental as nc

    monkeypatch.setattr(nc, "BLOCKED_MIN_EDGES", 0 if blocked else 1 << 60)
    g = graph(1500, 30_000, 14)
    inputs = inputs_for(g, batch, 41)
    probe = torch.tensor(inputs["probe"]["s"], dtype=torch.float32, device=gpu)

    def build(weight):
        topo = topology(g, torch.float32, gpu)
        if weight is not None:
            topo.in_weight.copy_(weight)
        topo.in_weight.requires_grad_(True)
        start = [leaf(inputs[k], torch.float32, gpu) for k in ("state", "dendrite", "adaptation")]
        mdl = model(inputs["params"], torch.float32, gpu, False)
        rt = NativeDendriticMatrixRuntime(topo, mdl, start[0].detach(), kernel=kernel)

        def one_pass():
            rt.state, rt.dendritic_state, rt.adaptation_state = start
            for t in range(ticks):
                rt.step(0.1 + 0.1 * t, dendritic_drive=0.1)
            grads = torch.autograd.grad(rt.state, [*start, topo.in_weight, *params_of(mdl)],
                                        grad_outputs=probe)
            return (rt.state.detach(), *grads)

        return topo, one_pass

    topo, one_pass = build(None)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        one_pass()
        captured = torch.cuda.CUDAGraph()
        with torch.cuda.graph(captured, stream=side):
            replayed = one_pass()
    torch.cuda.current_stream().wait_stream(side)
    for scale in (0.5, -1.5, 1.0):
        with torch.no_grad():
            topo.in_weight.mul_(scale)
        captured.replay()
        want = build(topo.in_weight.detach())[1]()
        torch.cuda.synchronize()
        for a, b in zip(replayed, want):
            # float32 sums of the same terms, of at most a hundred each
            assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())


def test_recorded_ticks_under_capture_keep_no_copy_of_trained_weights(gpu, monkeypatch):
    """What a capture would bake in, without one (the query alone says that the stream is
    captured): the forward reads trained weights in place, also where a training loop's
    eager ticks have made a slot-order copy of them, and the backward is refused before
    it launches anything.  The eager pass after it is right."""
    print("case backward under capture", flush=True)
    from neurosim_gpu.native import PANEL_INDEXED

    g = graph(1500, 30_000, 14)
    inputs = inputs_for(g, 1, 41)
    topo = topology(g, torch.float32, gpu)
    topo.in_weight.requires_grad_(True)
    mdl = model(inputs["params"], torch.float32, gpu, False)
    start = leaf(inputs["state"], torch.float32, gpu)
    rt = NativeDendriticMatrixRuntime(topo, mdl, start.detach(), kernel="panels")
    zero = torch.zeros_like(start)

    def one_pass(ticks):
        rt.state, rt.dendritic_state, rt.adaptation_state = start, zero, zero
        for t in range(ticks):
            rt.step(0.1 + 0.1 * t, dendritic_drive=0.1)
        return rt.state

    def gradients(out):
        return torch.autograd.grad(out, [start, topo.in_weight],
                                   grad_outputs=torch.ones_like(out), retain_graph=True)

    gradients(one_pass(2))
    with torch.no_grad():
        topo.in_weight.mul_(0.5)
    out = one_pass(1)
    want = gradients(out)
    with monkeypatch.context() as patched:
        patched.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
        assert rt._recorded_panel_plan(topo.in_weight).flags & PANEL_INDEXED
        with pytest.raises(RuntimeError, match="cannot be captured"):
            gradients(out)
    for a, b in zip(gradients(one_pass(1)), want):
        # the same terms (panels against row blocks), of at most a hundred each
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())


@pytest.mark.parametrize("n,m,chunk,bucket", [
    (50, 400, None, None), (3000, 90_000, None, None), (3000, 90_000, 4, 64),
    (700, 9_217, 9216, 128), (2000, 60_000, 36_864, 36_864), (300, 5_001, 4_996, 18_432)])
def test_blocked_permutation_equals_the_slot_gather(gpu, n, m, chunk, bucket):
    """ns_permute_blocked (through LDS, chunk by chunk and bucket by bucket) against the
    gather slot by slot, bitwise: chunks and buckets of a few values, partial last ones,
    and values at an address that is not 16-byte aligned."""
    print(f"case blocked permutation n={n} m={m} chunk={chunk} bucket={bucket}", flush=True)
    from neurosim_gpu.native import BlockedPermutation
    from neurosim_gpu.native_compartmental import TransposedPanels

    topo = topology(graph(n, m, 3), torch.float32, gpu)
    layout = TransposedPanels(topo, 1, gpu).layout
    permutation = BlockedPermutation(layout.perm, topo.n_edges, chunk, bucket)
    for offset in (0, 1):
        held = torch.randn(topo.n_edges + offset, device=gpu)
        values = held[offset:]
        want, _ = layout.slot_weights(object(), values, None)
        assert torch.equal(permutation(values), want)
    with pytest.raises(RuntimeError, match="M contiguous float32"):
        permutation(held[: topo.n_edges - 1])


def test_blocked_transposed_weights_change_no_gradient(gpu, monkeypatch):
    """Two weight versions through two ticks each, with the transposed weights permuted
    in blocks before their first use: gradients bitwise those of the indexed plan."""
    print("case backward blocked transposed weights", flush=True)
    from neurosim_gpu import native_compartmental as nc

    g = graph(3000, 90_000, 17)
    inputs = inputs_for(g, 1, 77)
    kw = dict(scalar_drives=False, expanded=False, kernel="panels", panel_width=1000)
    indexed, rt = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, 1, **kw)
    assert rt._transposed.layout.blocked is None
    monkeypatch.setattr(nc, "BLOCKED_MIN_EDGES", 0)
    blocked, rt = run(NativeDendriticMatrixRuntime, g, inputs, torch.float32, gpu, 1, **kw)
    assert rt._transposed.layout.blocked is not None
    assert rt._transposed.layout._slot_weights is not None
    for name in indexed:
        assert torch.equal(indexed[name], blocked[name]), name
    with torch.no_grad():
        rt.topology.in_weight.mul_(0.5)
    before = rt._transposed.layout._slot_key
    rt.state = rt.state.detach().requires_grad_(True)
    rt.dendritic_state, rt.adaptation_state = (rt.dendritic_state.detach(),
                                               rt.adaptation_state.detach())
    rt.step(0.2)
    rt.state.sum().backward()
    assert rt._transposed.layout._slot_key != before
