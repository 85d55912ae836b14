"""CPU checks of how the Python operators pass streams to the library."""

import subprocess
import sys

from conftest import ROOT

_WITHOUT_RAW_STREAM = """
import types, torch
if hasattr(torch._C, "_cuda_getCurrentRawStream"):
    del torch._C._cuda_getCurrentRawStream
import heteromega_amd.ffn as ffn
torch.cuda.current_stream = lambda device=None: types.SimpleNamespace(cuda_stream=4096 + device.index)
assert ffn._stream(None, torch.device("cuda", 3)) == 4099
assert ffn._stream(17, torch.device("cuda", 3)) == 17
"""


def test_current_stream_without_torchs_private_handle():
    # The raw handle comes from a private function of torch; without it the public call serves.
    res = subprocess.run([sys.executable, "-c", _WITHOUT_RAW_STREAM], cwd=ROOT, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
