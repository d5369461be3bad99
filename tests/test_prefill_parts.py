"""The scratch that a prefill pass's attention asks for, from the built library on the CPU."""
import os
import subprocess
import sys

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sense-nova-server_amd", "libsnl.so")
PART_FLOATS = "_ZN3snl29attention_prefill_part_floatsEii"  # snl::attention_prefill_part_floats(int ctx, int n_heads)


def test_model_without_attention_needs_no_parts():
    """A model of DeltaNet layers alone may have no attention heads: it gets no scratch, and its engine
    is built (a division by its KV heads would end the process, so the call has one of its own)."""
    code = (f"import ctypes; f = ctypes.CDLL({LIB!r}).{PART_FLOATS}; f.restype = ctypes.c_size_t; "
            "print([f(c, 0) for c in (2, 128, 129, 4096, 32768)], f(4096, 16) > 0)")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stderr)
    assert r.stdout.split("\n")[0] == "[0, 0, 0, 0, 0] True"
