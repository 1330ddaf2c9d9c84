"""Host-side check of the library: names of the kernels that a captured step launches by the hundred stay short, since the host pays for them on every launch of the graph."""
import subprocess

from helpers.device import pkg


def test_names_of_the_one_token_products():
    names = {l.split()[-1] for l in subprocess.run(["nm", "-D", "--defined-only", pkg.lib_path()], capture_output=True, text=True, check=True).stdout.splitlines()}
    one = {n for n in names if n.startswith("_ZN3cai8gemv_one")}
    assert one and max(map(len, one)) < 110, max(one, key=len)
