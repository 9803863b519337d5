"""When a decode step writes its input embedding: right before the launch,
after every check, where the package's own interpreter and launcher run; before
anything else, and with no keyword that a stand-in does not know, otherwise."""

import functools

import pytest
import torch

import mk_llama
import mk_mixtral
from megakernels_amd.latency.mk import LatencyMK_Interpreter
from megakernels_amd.latency.scheduler import make_dag as llama_dag
from megakernels_amd.latency.scheduler import make_globals as llama_globals
from megakernels_amd.latency.synthetic import LLAMA_TINY, make_synthetic_llama
from megakernels_amd.mixtral.generate import MK_Generator
from megakernels_amd.mixtral.mk import MixtralMK_Interpreter
from megakernels_amd.mixtral.scheduler import make_dag, make_globals
from megakernels_amd.mixtral.synthetic import TINY, make_synthetic_mixtral
from megakernels_amd.scheduler import Schedule, assign_to_sms, tensorize_instructions

LAUNCHER = {"mixtral": mk_mixtral.mk_mixtral, "llama": mk_llama.mk_llama}
HIDDEN = {"mixtral": 17, "llama": 16}  # positional argument


@functools.lru_cache
def _model(vm):
    if vm == "mixtral":
        return make_synthetic_mixtral(TINY, "cpu", 3, full=True, kv_positions=16, prefill=4)
    return make_synthetic_llama(LLAMA_TINY, "cpu", 3, kv_positions=16, prefill=4)


def generator(vm, launcher=None, **kw):
    model = _model(vm)
    if vm == "mixtral":
        g, dag, interpreter = make_globals(model, seq_len=4, sm_count=8), make_dag, MixtralMK_Interpreter()
    else:
        g, dag, interpreter = llama_globals(model, seq_len=4, sm_count=8), llama_dag, LatencyMK_Interpreter()
    sched = Schedule(g, *dag(g))
    tensorize_instructions(g, assign_to_sms("rr", schedule=sched))
    if launcher is not None:
        interpreter.mk_func = launcher
    gen = MK_Generator(model, interpreter, sched, **kw)
    g.hidden_states.fill_(-7.0)
    return gen, g.hidden_states, model.embed_tokens


class Launcher:
    """Records the hidden state it was called with, and its keywords; with
    ``late`` it takes and runs ``before_launch``, as the package's own do."""

    def __init__(self, vm, late, fail=False):
        self.vm, self.fail, self.seen, self.keywords = vm, fail, [], []
        if late:
            self.takes_before_launch = self

    def __call__(self, *args, **kw):
        self.keywords.append(set(kw))
        self.seen.append(args[HIDDEN[self.vm]].clone())
        if self.fail:
            raise ValueError("refused")
        if "before_launch" in kw:
            kw["before_launch"]()
            self.seen.append(args[HIDDEN[self.vm]].clone())


TOKEN = torch.tensor([[5]])
VMS = pytest.mark.parametrize("vm", ["mixtral", "llama"])


@VMS
@pytest.mark.parametrize("device_argmax", [True, False])
def test_own_launcher_embeds_after_the_checks(vm, device_argmax):
    k = Launcher(vm, late=True)
    gen, hidden, table = generator(vm, k, device_argmax=device_argmax)
    gen.run(TOKEN, 4)
    before, after = k.seen
    assert bool((before == -7.0).all()) and torch.equal(after, table[5])


@VMS
def test_package_launchers_take_the_hook(vm):
    assert generator(vm)[0]._launch_takes_embed()
    assert LAUNCHER[vm].takes_before_launch is LAUNCHER[vm]


def _early(k, gen, hidden, table):
    gen.run(TOKEN, 4)
    assert torch.equal(k.seen[0], table[5])
    assert "before_launch" not in k.keywords[0]


@VMS
def test_other_launcher_gets_the_early_copy(vm):
    k = Launcher(vm, late=False)
    _early(k, *generator(vm, k))


@VMS
def test_wrapped_launcher_gets_the_early_copy(vm):
    k = Launcher(vm, late=False)

    @functools.wraps(LAUNCHER[vm])  # copies the attributes of the launcher it stands for
    def wrapped(*args, **kw):
        return k(*args, **kw)

    _early(k, *generator(vm, wrapped))


@VMS
def test_replaced_interpret_gets_the_early_copy(vm):
    """A method put on the instance sees the step's embedding and no keyword
    of the driver's own."""
    gen, hidden, table = generator(vm)
    seen = []

    def interpret(globs, argmax_out=None, next_embed_weights=None, reset_for_next_launch=False, work_sharing=False):
        seen.append(globs.hidden_states.clone())

    gen.interpreter.interpret = interpret
    gen.run(TOKEN, 4)
    assert torch.equal(seen[0], table[5])


@VMS
def test_interpreter_subclass_gets_the_early_copy(vm):
    base = MixtralMK_Interpreter if vm == "mixtral" else LatencyMK_Interpreter

    class Own(base):
        def interpret(self, globs, **kw):
            return super().interpret(globs, **kw)

    k = Launcher(vm, late=True)
    gen, hidden, table = generator(vm, k)
    own = Own()
    own.mk_func = k
    gen.interpreter = own
    _early(k, gen, hidden, table)


@VMS
def test_launch_on_a_named_stream_gets_the_early_copy(vm):
    k = Launcher(vm, late=True)
    _early(k, *generator(vm, k, stream=None))


@VMS
@pytest.mark.parametrize("kw,launches,embeds", [({"skip_mk": True}, 0, True), ({"skip_rest": True}, 1, False),
                                                ({"skip_mk": True, "skip_rest": True}, 0, False)])
def test_skips(vm, kw, launches, embeds):
    k = Launcher(vm, late=True)
    gen, hidden, table = generator(vm, k, **kw)
    gen.run(TOKEN, 4)
    assert len(k.keywords) == launches and all("before_launch" not in s for s in k.keywords)
    assert torch.equal(hidden, table[5]) if embeds else bool((hidden == -7.0).all())


@VMS
def test_embedded_step_copies_nothing(vm):
    """A chained step's embedding is the previous launch's work."""
    k = Launcher(vm, late=True)
    gen, hidden, _ = generator(vm, k)
    toks = torch.zeros(1, 4, dtype=torch.long)
    gen.generate(toks, prompt_len=4, ntok=3)
    assert ["before_launch" in s for s in k.keywords] == [True, False, False]
    assert len(k.seen) == 4


@VMS
def test_refused_launch_leaves_the_hidden_state(vm):
    """A failed check leaves ``hidden_states`` alone, and the step after it is
    whole: embedding, barriers and logits."""
    k = Launcher(vm, late=True, fail=True)
    gen, hidden, table = generator(vm, k)
    g = gen.schedule.globs
    with pytest.raises(ValueError, match="refused"):
        gen.run(TOKEN, 4)
    assert bool((hidden == -7.0).all())
    k.fail = False
    g.barriers.fill_(3)
    g.logits.fill_(3.0)
    gen.run(TOKEN, 4)
    assert torch.equal(hidden, table[5]) and not bool(g.barriers.any()) and not bool(g.logits.any())


@VMS
def test_package_launcher_checks_before_it_embeds(vm):
    """The real launchers refuse CPU tensors before they call the hook."""
    gen, hidden, _ = generator(vm)
    with pytest.raises(ValueError, match="needs GPU tensors"):
        gen.run(TOKEN, 4)
    assert bool((hidden == -7.0).all())
