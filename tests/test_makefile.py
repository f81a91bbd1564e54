"""What make would run after a change, from its dry run."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "infer_amd", "csrc")


def commands(changed, target):
    """The commands behind a change of ``changed``, one a line."""
    done = subprocess.run(["make", "-C", CSRC, "PYTHON=true", "-n", "-W", changed, target], capture_output=True, text=True, check=True)
    return done.stdout.replace("\\\n", " ").splitlines()


def test_a_new_library_takes_the_decode_call_of_the_old_one_away():
    """``lib`` does not make the call, which needs torch: it must not leave one behind that knows the old library's arguments."""
    lines = commands("block_pool.cpp", "lib")
    gone = next(i for i, c in enumerate(lines) if c.startswith("rm ") and "_decode_call.so" in c)
    assert any("-o ../libinfer_kv.so" in c for c in lines[gone:]) and not any("decode_call.cpp" in c for c in lines)
    lines = commands("block_pool.cpp", "all")
    gone = next(i for i, c in enumerate(lines) if c.startswith("rm ") and "_decode_call.so" in c)
    assert any("decode_call.cpp" in c for c in lines[gone:])


def test_kernels_are_compiled_again_with_the_headers_they_include():
    """Two kernels of a call that agree on a record by a header, and one of them compiled with the old one, would read past it."""
    sources = [f for f in sorted(os.listdir(CSRC)) if f.endswith(".hip")]
    for header in sorted(f for f in os.listdir(CSRC) if f.endswith(".h")):
        lines = commands(header, "lib")
        for source in sources:
            if f'#include "{header}"' in open(os.path.join(CSRC, source)).read():
                assert any(f" -c {source} " in c for c in lines), (source, header)
