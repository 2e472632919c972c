"""The run_kernel.py-style harness end to end on the GPU: every case of KERNEL_ZOO compiled for the mi355x system,
checked against the torch system with the reference's report lines."""
import contextlib
import io

import pytest
import torch

from conftest import progress
from deepgengraph_amd import cases
from deepgengraph_amd.run_kernel import main

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", sorted(cases.KERNEL_ZOO))
def test_run_kernel_cli(gpu, name):
    progress(f"run_kernel -m {name}")
    buf = io.StringIO()
    with contextlib.redirect_stdout(buf):
        main(["-m", name, "-s", "mi355x", "--seqlen", "384"])
    text = buf.getvalue()
    assert "gflops=" in text and "speedup = " in text, text
    flags = [line for line in text.splitlines() if "isCorrect" in line]
    n_out = len(cases.KERNEL_ZOO[name].OUTPUTS)
    assert len(flags) == n_out and all(line.endswith("True") for line in flags), text


def test_stream_handle_takes_what_torch_takes(gpu):
    """A torch.device with and without an index, an index, None: each names torch's current stream there."""
    from deepgengraph_amd import _lib

    for dev in (gpu, torch.device("cuda"), gpu.index or 0, None):
        assert _lib.stream_handle(dev) == torch.cuda.current_stream(dev).cuda_stream
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert _lib.stream_handle(gpu) == side.cuda_stream
