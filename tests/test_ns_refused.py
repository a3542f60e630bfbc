"""ssx_ns_create on a device that does not grant the convection operator's
LDS: refused at creation, with nothing allocated, not in the middle of a
step.  The host side (ssx_ns.c) is linked with a stand-in for that one
device query that refuses; it must return the refusal before it calls
anything else (every other symbol is left unresolved and would end the
program)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
CSRC = os.path.join(ROOT, "ssenss_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

MAIN = r"""
#include <stdio.h>
#include <stdlib.h>
#include "ssx_internal.h"
void ssx_set_error(const char *fmt, ...) { (void) fmt; }
int ssxk_ns_conv_ready(int n) { return n == 10 ? SSX_EHIP : SSX_OK; }
int main(void)
{
	static ssx_ctx c;
	ssx_ns_params prm = { .dt = 1e-2, .visc = 0.5, .dens = 1.0 };
	ssx_ns *ns = (ssx_ns *) &c;
	c.lev[0].n = 10;
	c.nel = 1;
	c.lambda = (11.0 / 6.0) / (prm.dt * prm.visc);
	const int rc = ssx_ns_create(&ns, &c, &prm);
	printf("%d %d\n", rc == SSX_EHIP, ns == NULL);
	return 0;
}
"""


@pytest.mark.skipif(not shutil.which("gcc")
                    or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                    reason="needs gcc and the HIP headers")
def test_refused_at_creation(tmp_path):
    src, exe = tmp_path / "main.c", tmp_path / "main"
    src.write_text(MAIN)
    subprocess.run(
        ["gcc", "-O1", "-std=c99", "-D_GNU_SOURCE", "-D__HIP_PLATFORM_AMD__",
         "-I" + os.path.join(ROCM, "include"), "-I" + CSRC,
         "-I" + os.path.join(ROOT, "include"), str(src),
         os.path.join(CSRC, "ssx_ns.c"), "-o", str(exe), "-lm",
         "-Wl,--unresolved-symbols=ignore-all"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True,
                         timeout=60)
    assert (out.returncode, out.stdout.split()) == (0, ["1", "1"])
