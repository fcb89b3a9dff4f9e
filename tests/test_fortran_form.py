"""&gpucon fused of the Fortran host reaches hg_set_fused, 0 too, and without it
the context is left in the form it starts with.  The host runs against a
library of stand-ins that writes the argument down and stops it at the first
upload, so no GPU is needed."""
import os
import shutil
import subprocess

import pytest

from hormone_amd.build import DRIVER

STUB = """
#include <stdio.h>
#include <stdlib.h>
int hg_create(const void *d, void **c) { *c = (void *)16; return 0; }
int hg_set_fused(void *c, int on) {
  FILE *f = fopen(getenv("FORM_LOG"), "a");
  fprintf(f, "%d\\n", on);
  fclose(f);
  return 0;
}
int hg_upload(void *c, int f, const double *p) { return 2; }
int hg_last_error(const void *c, int *i, int *j, int *k, int *d) { return 0; }
int hg_destroy(void *c) { return 0; }
int hg_download(void *c, int f, double *p) { return 2; }
int hg_gravity() { return 2; }
int hg_hydro_step() { return 2; }
int hg_phidamp() { return 2; }
int hg_timestep() { return 2; }
"""


@pytest.mark.skipif(not os.path.exists(DRIVER) or not shutil.which("gcc"),
                    reason="needs the built Fortran host (amdflang) and gcc")
@pytest.mark.parametrize("text,want", [("fused=0", "0\n"), ("fused=1", "1\n"), ("fused=2", "2\n"),
                                       ("fused=-1", ""), ("", "")])
def test_fortran_host_passes_the_form_on(text, want, tmp_path):
    (tmp_path / "stub.c").write_text(STUB)
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", "-o", str(tmp_path / "libhormone_hip.so"),
                    str(tmp_path / "stub.c")], check=True)
    log = tmp_path / "form"
    log.write_text("")
    par = tmp_path / "parameters"
    par.write_text("&gridcon is=1 ie=16 js=1 je=16 ks=1 ke=1 /\n"
                   f"&gpucon outfile='{tmp_path}/out' {text} /\n")
    subprocess.run([DRIVER, str(par)], capture_output=True, timeout=60,
                   env=dict(os.environ, LD_LIBRARY_PATH=f"{tmp_path}:" + os.environ.get("LD_LIBRARY_PATH", ""),
                            FORM_LOG=str(log)))
    assert log.read_text() == want
