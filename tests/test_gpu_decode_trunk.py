"""The decode step as one launch against the list of launches it stands for: the same bits.

The list is held to its oracle in test_gpu_decode_layer.py and test_ar_decode.py; the one launch adds its sums in
the same order, so every comparison here is exact.
"""

import types

import pytest
import torch

from visionrl_amd import _lib
from visionrl_amd.decode_step import NativeDecodeTrunk
from visionrl_amd.linear import Int4LlamaMLP, Int4Linear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HIDDEN, DIM = 2048, 128


def normal(gen, *shape, scale=1.0):
    return torch.randn(shape, generator=gen, device=DEV).mul_(scale).to(torch.bfloat16)


def linear(gen, K, N, prepack=True):
    words = lambda *s: torch.randint(-2 ** 31, 2 ** 31, s, generator=gen, device=DEV, dtype=torch.int64).to(torch.int32)
    scales = torch.randn((N, K // 128), generator=gen, device=DEV).abs_().clamp_(min=0.05).mul_(0.003)
    module = Int4Linear.from_packed(words(N, K // 8), scales.to(torch.bfloat16), words(N, (K // 128 + 7) // 8), 128)
    return module.prepack_() if prepack else module


class Step:
    """A trunk of random int4 layers over a random cache, its step as one launch and as the list."""

    def __init__(self, rows, layers=2, heads=16, kv_heads=16, inter=5632, length=1024, slot=(330,), padded=True,
                 final_norm=True, seed=1, edit=None):
        gen = torch.Generator(device=DEV).manual_seed(seed)
        norm = lambda: types.SimpleNamespace(weight=normal(gen, HIDDEN, scale=0.1).add_(1.0), variance_epsilon=1e-6)

        def layer():
            attn = types.SimpleNamespace(scaling=DIM ** -0.5, **{
                name: linear(gen, k, n) for name, k, n in (
                    ("q_proj", HIDDEN, heads * DIM), ("k_proj", HIDDEN, kv_heads * DIM),
                    ("v_proj", HIDDEN, kv_heads * DIM), ("o_proj", heads * DIM, HIDDEN))})
            mlp = Int4LlamaMLP(types.SimpleNamespace(
                gate_proj=linear(gen, HIDDEN, inter, False), up_proj=linear(gen, HIDDEN, inter, False),
                down_proj=linear(gen, inter, HIDDEN, False)), 128).prepack_()
            return types.SimpleNamespace(self_attn=attn, mlp=mlp, input_layernorm=norm(),
                                         post_attention_layernorm=norm())

        def rotary(x, position_ids):
            inv = 10000.0 ** (-torch.arange(0, DIM, 2, device=DEV).float() / DIM)
            angle = position_ids[..., None].float() * torch.cat([inv, inv])
            return angle.cos().to(x.dtype), angle.sin().to(x.dtype)

        trunk = types.SimpleNamespace(
            config=types.SimpleNamespace(hidden_size=HIDDEN, num_attention_heads=heads, num_key_value_heads=kv_heads,
                                         head_dim=DIM),
            layers=[layer() for _ in range(layers)], norm=norm(), rotary_emb=rotary)
        self.cache = [normal(gen, rows, kv_heads, length, DIM) for _ in range(2 * layers)]
        held = types.SimpleNamespace(layers=[
            types.SimpleNamespace(keys=k, values=v, is_initialized=True)
            for k, v in zip(self.cache[::2], self.cache[1::2])])
        self.mask = torch.ones((rows, length), dtype=torch.uint8, device=DEV)
        if padded:   # prompts padded on the left, by a different number of slots per row
            for m in range(rows):
                self.mask[m, :min(7 + 40 * m, min(slot) // 2)] = 0
        self.x = normal(gen, rows, 1, HIDDEN)
        self.slot = torch.tensor(slot, dtype=torch.int64, device=DEV)
        if edit is not None:
            edit(trunk)
        self.native = NativeDecodeTrunk(trunk, held, self.x, self.mask, self.slot, final_norm=final_norm)
        self.one = self.native._trunk

    def run(self, one: bool, short=False):
        """``(output, caches)`` of a step; the caches are put back."""
        before = [t.clone() for t in self.cache]
        self.native._trunk = self.one if one else None
        out = self.native.run(short)
        torch.cuda.synchronize()
        got = (self.native.final[0] if out is None else out).clone(), [t.clone() for t in self.cache]
        for t, b in zip(self.cache, before):
            t.copy_(b)
        self.native._trunk = self.one
        return got

    def check(self, short=False):
        assert self.one is not None
        want, want_cache = self.run(False, short)
        for _ in range(2):   # the second finds the numbers that the first left behind
            got, cache = self.run(True, short)
            assert torch.isfinite(got).all()
            assert torch.equal(got.view(torch.int16), want.view(torch.int16))
            assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(cache, want_cache))


@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("kv_heads", [4, 16])
@pytest.mark.parametrize("slot", [0, 1, 63, 64, 255, 256, 257, 511, 512, 513, 767, 768, 1023])
def test_one_launch_has_the_bits_of_the_list(rows, kv_heads, slot):
    print("decode trunk:", rows, kv_heads, slot, flush=True)
    step = Step(rows, kv_heads=kv_heads, slot=(slot,), layers=1 if slot in (63, 255, 257) else 2, seed=slot + rows)
    step.check()
    if step.native.short_form(slot):
        step.check(short=True)


@pytest.mark.parametrize("heads,kv_heads,inter,length,final_norm", [
    (16, 16, 5376, 640, True), (16, 2, 8192, 1024, True),      # remainders of the tiles per workgroup
    (16, 16, 5632, 320, False),                                # the last norm left to the head; no split form
    (16, 8, 5120, 1000, True), (12, 4, 5632, 700, True), (8, 8, 6144, 640, False),
])
@pytest.mark.parametrize("rows", [2, 4])
def test_other_shapes(rows, heads, kv_heads, inter, length, final_norm):
    print("decode trunk shapes:", rows, heads, kv_heads, inter, length, final_norm, flush=True)
    step = Step(rows, heads=heads, kv_heads=kv_heads, inter=inter, length=length, slot=(length - 5,),
                final_norm=final_norm)
    if (rows, heads) == (4, 8):   # eight workgroups per pair of four rows: not built
        assert step.one is None
    else:
        step.check()


@pytest.mark.parametrize("rows,slot", [(2, (0, 900)), (3, (511, 512, 40)), (4, (1023, 3, 767, 256)),
                                       (4, (5, 1024, 600, 9000)), (2, (1 << 40, 17))])
def test_rows_at_positions_of_their_own(rows, slot):
    """... also outside the cache, where a row appends nothing and its output means nothing."""
    print("decode trunk positions:", rows, slot, flush=True)
    step = Step(rows, slot=slot, seed=7)
    inside = [m for m in range(rows) if slot[m] < 1024]
    want, want_cache = step.run(False)
    got, cache = step.run(True)
    assert torch.equal(got[inside], want[inside])
    assert all(torch.equal(a, b) for a, b in zip(cache, want_cache))


@pytest.mark.parametrize("slot", [200, 800])
def test_masked_slots_and_stale_cache(slot):
    """A row that sees nothing, holes in the mask, and NaN in slots that the step must not read."""
    print("decode trunk masks:", slot, flush=True)
    step = Step(4, slot=(slot,))
    for t in step.cache:
        t[:, :, slot:] = float("nan")
    step.mask[0] = 0
    step.mask[1, ::3] = 0
    step.mask[2, :slot] = 0
    want, _ = step.run(False)
    for _ in range(2):
        got, _ = step.run(True)
        assert torch.isfinite(got).all() and torch.equal(got, want)


def test_graph_replays_between_eager_steps():
    print("decode trunk: graph", flush=True)
    step = Step(2, layers=3)
    want, _ = step.run(False)
    step.native.run()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step.native.run()
    for _ in range(4):
        out.zero_()
        graph.replay()
        assert torch.equal(out, want)
        step.x.add_(step.x)                       # eager work, another step, and the first one's input again
        step.native.run()
        torch.cuda.synchronize()
        step.x.mul_(0.5)


def test_steps_on_several_streams():
    """Launches that do not share a workspace, in flight together: each waits for the chip, none for another."""
    print("decode trunk: streams", flush=True)
    steps = [Step(2, seed=s, layers=4) for s in (1, 2, 3)]
    want = [s.run(False)[0] for s in steps]
    streams = [torch.cuda.Stream() for _ in steps]
    torch.cuda.synchronize()
    for _ in range(10):
        for s, stream in zip(steps, streams):
            with torch.cuda.stream(stream):
                s.native.run()
    torch.cuda.synchronize()
    assert all(torch.equal(s.native.normed, w) for s, w in zip(steps, want))


@pytest.mark.parametrize("workgroups", [1, 3, 100, 255])
@pytest.mark.parametrize("kwargs", [
    dict(rows=1, slot=(330,)), dict(rows=2, slot=(900,), kv_heads=4), dict(rows=3, slot=(0,), inter=5376),
    dict(rows=4, slot=(511, 900, 40, 2000)), dict(rows=4, slot=(800,), heads=12, kv_heads=4),
    dict(rows=2, slot=(130,), inter=8192, final_norm=False),
])
def test_a_part_of_the_chip_has_the_bits_of_the_list(workgroups, kwargs):
    """The parts of every product dealt out to fewer workgroups than they are laid out for."""
    print("decode trunk team:", workgroups, kwargs, flush=True)
    step = Step(**kwargs)
    for desc in step.one:
        desc.max_workgroups = workgroups
    slots = kwargs["slot"] if len(kwargs["slot"]) > 1 else kwargs["slot"] * kwargs["rows"]
    inside = [m for m, slot in enumerate(slots) if slot < 1024]
    want, want_cache = step.run(False)
    for _ in range(2):
        got, cache = step.run(True)
        assert torch.equal(got[inside].view(torch.int16), want[inside].view(torch.int16))
        assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(cache, want_cache))


@pytest.mark.parametrize("layers,heads,kv_heads", [(1, 8, 2), (1, 8, 8), (2, 8, 2)])
def test_workgroups_without_a_part_behind_the_last_exchange(layers, heads, kv_heads):
    """One row and few heads: some workgroups have gate|up tiles only, and in the last layer nobody needs to have
    seen them before the first ones end."""
    print("decode trunk few heads:", layers, heads, kv_heads, flush=True)
    step = Step(1, layers=layers, heads=heads, kv_heads=kv_heads, length=320, slot=(200,), final_norm=False)
    step.check()


def test_a_kernel_that_keeps_a_compute_unit():
    """A step beside a kernel that stays on the chip for long: neither waits for it nor gives anything up."""
    print("decode trunk: beside a kernel", flush=True)
    step = Step(2, layers=4)
    want, want_cache = step.run(False)
    side = torch.cuda.Stream()
    start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    start.record()
    torch.cuda._sleep(10_000_000)
    end.record()
    torch.cuda.synchronize()
    cycles = int(10_000_000 * 300 / start.elapsed_time(end))   # 0.3 s
    before = [t.clone() for t in step.cache]
    busy, done = torch.cuda.Event(), torch.cuda.Event()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(cycles)
        busy.record()
    got = step.native.run()
    done.record()
    done.synchronize()
    assert not busy.query()
    assert torch.equal(got, want)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(step.cache, want_cache))
    for t, b in zip(step.cache, before):
        t.copy_(b)
    got, _ = step.run(True)
    assert torch.equal(got, want)


def test_recorded_steps_on_several_streams():
    """Replays of steps with workspaces of their own, in flight together and beside an eager one."""
    print("decode trunk: recorded steps", flush=True)
    steps = [Step(2, seed=s, layers=4) for s in (1, 2, 3)]
    want = [s.run(False)[0] for s in steps]
    graphs = []
    for s in steps[:2]:
        s.native.run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            s.native.run()
        graphs.append(graph)
    streams = [torch.cuda.Stream() for _ in steps]
    torch.cuda.synchronize()
    for _ in range(10):
        for launch, stream in zip((graphs[0].replay, graphs[1].replay, steps[2].native.run), streams):
            with torch.cuda.stream(stream):
                launch()
    torch.cuda.synchronize()
    assert all(torch.equal(s.native.normed, w) for s, w in zip(steps, want))


def test_every_wait_ends():
    """One look per wave: nothing is waited for, the launch ends and its output says so; over a cleared workspace
    the next step is right again."""
    print("decode trunk: wait limit", flush=True)
    step = Step(2)
    want, _ = step.run(False)
    for desc in step.one:
        desc.wait_limit = 1
    got, _ = step.run(True)
    assert got.isnan().any()
    (workspace,) = [t for t in step.native._keep if torch.is_tensor(t) and t.data_ptr() == step.one[0].workspace]
    workspace.zero_()
    for desc in step.one:
        desc.wait_limit = 0
    got, _ = step.run(True)
    assert torch.equal(got, want)


@pytest.mark.parametrize("kwargs", [dict(rows=5), dict(rows=2, inter=4864), dict(rows=2, inter=8448),
                                    dict(rows=2, heads=32, kv_heads=32)])
def test_other_steps_keep_the_list(kwargs):
    print("decode trunk: list", kwargs, flush=True)
    step = Step(**kwargs)
    assert step.one is None
    assert torch.isfinite(step.run(False)[0]).all()


@pytest.mark.parametrize("final_norm", [True, False])
def test_a_workspace_that_was_given_up_on_says_so(final_norm):
    """Steps over it touch no cache and have NaN in every value, until it is zeroed."""
    print("decode trunk: given up", final_norm, flush=True)
    step = Step(3, final_norm=final_norm)
    want, want_cache = step.run(False)
    for desc in step.one:
        desc.wait_limit = 1
    assert step.run(True)[0].isnan().any()
    for desc in step.one:
        desc.wait_limit = 0
    for _ in range(2):
        got, cache = step.run(True)
        assert got.isnan().all() and all(torch.equal(a, b) for a, b in zip(cache, step.cache))
    (workspace,) = [t for t in step.native._keep if torch.is_tensor(t) and t.data_ptr() == step.one[0].workspace]
    workspace.zero_()
    got, cache = step.run(True)
    assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip(cache, want_cache))


def shifted(t):
    """The same values two bytes further on."""
    out = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    return out.copy_(t)


@pytest.mark.parametrize("which", ["input_layernorm", "post_attention_layernorm", "norm"])
@pytest.mark.parametrize("what", ["address", "eps"])
def test_norms_that_the_list_refuses_stay_refused(which, what):
    print("decode trunk: norms", which, what, flush=True)

    def edit(trunk):
        norm = trunk.norm if which == "norm" else getattr(trunk.layers[1], which)
        if what == "address":
            norm.weight = shifted(norm.weight)
        else:
            norm.variance_epsilon = -1.0

    step = Step(2, edit=edit)
    assert step.one is None
    with pytest.raises(ValueError):
        step.native.run()


def test_launches_says_what_run_enqueues():
    step = Step(2, layers=3)
    assert step.native.launches == 1
    step.native._trunk = None
    assert step.native.launches == 5 * 3 + 1


@pytest.mark.parametrize("code", _lib.NOT_COOPERATIVE)
def test_a_refused_cooperative_launch_leaves_the_step_to_the_list(monkeypatch, code):
    print("decode trunk: not cooperative", code, flush=True)
    step = Step(2)
    want, want_cache = step.run(False)
    monkeypatch.setattr(_lib.load(), "vrl_decode_trunk_bf16", lambda *args: code)
    got, cache = step.run(True)
    assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip(cache, want_cache))
    monkeypatch.setattr(_lib.load(), "vrl_decode_trunk_bf16", lambda *args: 1002)   # a mistake is still one
    with pytest.raises(ValueError):
        step.run(True)


def test_no_layers():
    print("decode trunk: no layers", flush=True)
    step = Step(2, layers=0)
    assert step.one is None
    got = step.native.run().float()
    x = step.x[:, 0].float()
    want = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * step.native._keep[-1].float()
    assert torch.allclose(got, want, rtol=2 ** -7, atol=1e-6)   # two roundings to bf16


def test_rotary_tables_at_any_address():
    print("decode trunk: rotary tables", flush=True)
    want, _ = Step(2).run(False)

    def edit(trunk):
        tables = trunk.rotary_emb
        trunk.rotary_emb = lambda *args, **kwargs: tuple(shifted(t) for t in tables(*args, **kwargs))

    step = Step(2, edit=edit)
    assert step.native.cos.data_ptr() % 4 == 2 and step.one is None
    assert torch.equal(step.native.run(), want)


def test_refusals():
    """Checks of the entry point, before any launch."""
    print("decode trunk: refusals", flush=True)
    import ctypes

    step = Step(2)
    lib = _lib.load()

    def code(**fields):
        desc = _lib.Trunk.from_buffer_copy(step.one[0])
        for name, value in fields.items():
            setattr(desc, name, value)
        return lib.vrl_decode_trunk_bf16(ctypes.byref(desc), None)

    assert lib.vrl_decode_trunk_bf16(None, None) == 1003
    for name in ("layers", "x", "mask", "cos", "sin", "norm", "position", "workspace"):
        assert code(**{name: None}) == 1003, name
    assert code(normed=None, h_out=None) == 1003
    assert code(M=0) == code(M=5) == code(hidden=4096) == code(group_size=64) == code(n_layers=0) == 1001
    assert code(x=step.one[0].x + 2) == code(workspace=step.one[0].workspace + 16) == 1002
    assert code(workspace_bytes=step.one[0].workspace_bytes - 1) == 1004
