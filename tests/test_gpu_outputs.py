"""The outputs that an entry point makes: as torch.empty makes them, whatever is in force around the call."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from tests.helpers import announce, gen, randn_bf16

pytestmark = pytest.mark.gpu


def _calls(gpu):
    from linghe_amd.quant.group import triton_group_quant
    from linghe_amd.utils.norm import triton_rms_norm_backward, triton_rms_norm_forward
    from linghe_amd.utils.silu import build_expert_plan, triton_silu_and_block_quant_forward

    g = gen(5)
    x, w = randn_bf16(g, 32, 256).to(gpu), randn_bf16(g, 256).to(gpu)
    counts = torch.tensor([3, 0, 200], device=gpu)
    return {
        "group": lambda: triton_group_quant(x),
        "norm": lambda: triton_rms_norm_forward(x, w),
        "norm_bwd": lambda: triton_rms_norm_backward(x, x, w),
        "swiglu": lambda: triton_silu_and_block_quant_forward(x, output_mode=0),
        "plan": lambda: (build_expert_plan(counts, [3, 0, 200]).table,),
    }


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.empties = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.empties += "empty" in func.__name__
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("name", ["group", "norm", "norm_bwd", "swiglu", "plan"])
def test_outputs_in_every_state_of_torch(gpu, name):
    announce("outputs", name)
    call = _calls(gpu)[name]
    plain = call()
    assert all(t.device == gpu and t.is_contiguous() and not t.is_inference() for t in plain)
    with _Seen() as seen:
        listened = call()
    assert seen.empties >= len(plain)
    with torch.inference_mode():
        inferred = call()
    assert all(t.is_inference() for t in inferred)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        beside = call()
    stream.synchronize()
    written = {"swiglu": 2}.get(name, len(plain))  # (mode 0 leaves the transposed outputs as they are)
    for other in (listened, inferred, beside):
        for a, b in list(zip(plain, other))[:written]:
            assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride()
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("name", ["group", "norm", "norm_bwd", "swiglu", "plan"])
def test_a_profiler_sees_the_outputs(gpu, name):
    announce("outputs, profiler", name)
    call = _calls(gpu)[name]
    outs = len(call())
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], acc_events=True) as seen:
        call()
    assert sum(e.name == "aten::empty" for e in seen.events()) >= outs


def test_deterministic_algorithms_fill_what_is_not_written(gpu):
    call = _calls(gpu)["swiglu"]
    torch.use_deterministic_algorithms(True)
    try:
        st = call()[3]
    finally:
        torch.use_deterministic_algorithms(False)
    assert st.isnan().all()


def test_output_keeps_the_strides_of_its_input(gpu):
    from linghe_amd.utils.norm import triton_rms_norm_forward

    w = torch.ones(256, dtype=torch.bfloat16, device=gpu)
    x = torch.randn(1, 8, 256, device=gpu).to(torch.bfloat16).as_strided((1, 8, 256), (77777, 256, 1))
    assert x.is_contiguous()
    assert triton_rms_norm_forward(x, w)[0].stride() == torch.empty_like(x).stride()
