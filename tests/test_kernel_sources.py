"""What a run on the GPU cannot show reliably, read from the kernels' sources."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "microllm-rocm_amd", "csrc")


def function(file: str, name: str) -> str:
    """The body of a kernel, comments left out."""
    with open(os.path.join(CSRC, file)) as source:
        text = re.sub(r"//[^\n]*", "", source.read())
    start = text.index(name + "(")
    depth, at = 0, text.index("{", start)
    for index in range(at, len(text)):
        depth += {"{": 1, "}": -1}.get(text[index], 0)
        if depth == 0:
            return text[at:index + 1]
    raise AssertionError(f"{name} has no end")


def test_weights_that_other_lanes_wrote_are_read_behind_a_fence():
    """Lanes of a wave hand their weights to each other through LDS without a barrier: between the last store and the first load
    stands a fence, without which the compiler may move a load above the stores of the other lanes."""
    body = function("linear_attention_chunks.hip", "gla_channel_out_kernel")
    stores = [match.end() for match in re.finditer(r"weights\[[^;=]*\]\[[^;=]*\] = [^=]", body)]
    loads = [match.start() for match in re.finditer(r"(own_weight|weight)\[j(?: / 4)?\] = [^;]*weights\[", body)]
    assert len(stores) == 2 and len(loads) == 2
    between = body[max(stores):min(loads)]
    assert re.search(r"__builtin_amdgcn_fence\(__ATOMIC_ACQ_REL, \"wavefront\"\)|__syncthreads\(\)", between)
