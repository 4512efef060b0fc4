"""Build recipe for the checker side (test infrastructure only).

1. oracle/_ref/liborc.so  -- the plain-C FP64 restatement (rhmc_oracle.c).
2. oracle/_ref/<cfg>/ref_harness -- the reference's own CPU path compiled with
   g++ -std=gnu++14 directly from the unmodified sources under
   /root/reference, one binary per compile-time configuration (the reference
   is configured through include/parameters.h; a generated parameters.h for
   each configuration is placed first on the include path).

Outputs go only into oracle/_ref/ (git-ignored).  Step 2 is skipped when
/root/reference does not hold the sources (e.g. on a machine without them).
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
OUT = os.path.join(HERE, "_ref")
REF = "/root/reference"

REF_SOURCES = [
    "lib/Main/Geometry/geometry.cc",
    "lib/Main/Conf/conf.cc",
    "lib/Action/su3.cc",
    "lib/Action/fermionmatrix.cc",
    "lib/Action/fermions.cc",
    "lib/Action/fermionforce.cc",
    "lib/Action/staples.cc",
    "lib/Action/action.cc",
    "lib/Action/Inverter/inverter.cc",
    "lib/Update/ipdot.cc",
    "lib/Update/momenta.cc",
    "lib/Update/update.cc",
    "lib/Update/MD_integrators/leapfrog.cc",
    "lib/Update/MD_integrators/minimum_norm2.cc",
    "lib/Update/MD_integrators/multistep_2MN.cc",
    "lib/Update/MD_integrators/multistep_4MN.cc",
    "lib/Tools/vec3.cc",
    "lib/Tools/gauss.cc",
    "lib/Tools/exception.cc",
    "lib/Tools/exist_file.cc",
    "lib/Tools/Rand/random.cc",
    "lib/Tools/RationalApprox/rationalapprox.cc",
    "lib/Measurements/gaugemeas.cc",
    "lib/Measurements/chiralmeas.cc",
]


def have_reference() -> bool:
    """Whether the reference's sources are there (its directory may be empty)."""
    return os.path.isfile(os.path.join(REF, REF_SOURCES[0]))


# Compile-time configurations for the golden vectors.  Keys are the constant
# names the reference reads from include/parameters.h.
CONFIGS = {
    # 4^4, two pseudofermions, multistep 2MN: exercises every path cheaply
    "t4": dict(nx=4, ny=4, nz=4, nt=4, no_flavours=2, beta=5.5, mass=0.1, no_ps=2,
               approx_metro=6, approx_md=5, no_md=3, use_multistep=1, gauge_scale=2,
               residue_metro=1e-12, residue_md=1e-12, max_cg=5000),
    # 4^4 Omelyan (minimum_norm2_A) with one pseudofermion
    "t4o": dict(nx=4, ny=4, nz=4, nt=4, no_flavours=2, beta=5.5, mass=0.1, no_ps=1,
                approx_metro=6, approx_md=5, no_md=3, use_multistep=0, gauge_scale=2,
                residue_metro=1e-12, residue_md=1e-12, max_cg=5000),
    # 4^4 multistep 4MN (use_multistep=2) with gauge_scale 2, one pseudofermion
    "t4m": dict(nx=4, ny=4, nz=4, nt=4, no_flavours=2, beta=5.5, mass=0.1, no_ps=1,
                approx_metro=6, approx_md=5, no_md=2, use_multistep=2, gauge_scale=2,
                residue_metro=1e-12, residue_md=1e-12, max_cg=5000),
    # 8^3x4 of the plain CPU RHMC configuration: am=0.05, beta=5.5, one
    # pseudofermion, 8 MD poles / 12 action poles, 10 Omelyan steps
    "c1": dict(nx=8, ny=8, nz=8, nt=4, no_flavours=2, beta=5.5, mass=0.05, no_ps=1,
               approx_metro=12, approx_md=8, no_md=10, use_multistep=0, gauge_scale=2,
               residue_metro=1e-10, residue_md=1e-10, max_cg=10000),
}

PARAM_TEMPLATE = """// generated by oracle/build_ref.py -- compile-time configuration {name}
#ifndef PARAMETERS_H_
#define PARAMETERS_H_
#include "include/global_macro.h"
const int nx={nx};
const int ny={ny};
const int nz={nz};
const int nt={nt};
const int no_flavours={no_flavours};
const REAL beta={beta!r};
const REAL mass={mass!r};
const int rand_seed=12345;
const int ferm_temp_bc=0;
const int start=1;
const int run_update_iterations=1;
const int therm_updates=0;
const int save_conf_every=1000000;
const int meas_every=1000000;
const int no_md={no_md};
const int use_multistep={use_multistep};
const int gauge_scale={gauge_scale};
const int rand_vect=1;
const int max_cg={max_cg};
const int no_ps={no_ps};
const int gmp_remez_precision=100;
const REAL inv_single_double_prec=1.0e-4;
const int approx_metro={approx_metro};
const REAL lambda_min_metro=1.0e-5;
const REAL residue_metro={residue_metro!r};
const int approx_md={approx_md};
const REAL lambda_min_md=1.0e-5;
const REAL residue_md={residue_md!r};
const int gpu_device_to_use=0;
#endif
"""


def run(cmd):
    print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)


def build_oracle_lib():
    os.makedirs(OUT, exist_ok=True)
    src = os.path.join(HERE, "rhmc_oracle.c")
    so = os.path.join(OUT, "liborc.so")
    if os.path.exists(so) and os.path.getmtime(so) >= max(os.path.getmtime(src),
                                                          os.path.getmtime(os.path.join(HERE, "rhmc_oracle.h"))):
        return so
    run(["gcc", "-O2", "-std=gnu11", "-fPIC", "-shared", "-fopenmp", src, "-o", so, "-lm"])
    return so


def build_ref(name: str, force: bool = False):
    if not have_reference():
        return None
    cfg = CONFIGS[name]
    bdir = os.path.join(OUT, name)
    exe = os.path.join(bdir, "ref_harness")
    harness = os.path.join(HERE, "ref_harness.cc")
    if os.path.exists(exe) and not force and os.path.getmtime(exe) >= os.path.getmtime(harness):
        return exe
    os.makedirs(os.path.join(bdir, "include"), exist_ok=True)
    with open(os.path.join(bdir, "include", "parameters.h"), "w") as fh:
        fh.write(PARAM_TEMPLATE.format(name=name, **cfg))
    objs = []
    dsfmt_o = os.path.join(bdir, "dSFMT.o")
    run(["gcc", "-O2", "-c", os.path.join(REF, "lib/Tools/Rand/RANDOM/dSFMT.c"), "-o", dsfmt_o])
    objs.append(dsfmt_o)
    inc = ["-I" + bdir, "-I" + REF]
    for s in REF_SOURCES + [os.path.join(HERE, "ref_harness.cc")]:
        path = s if os.path.isabs(s) else os.path.join(REF, s)
        o = os.path.join(bdir, os.path.basename(s).replace(".cc", ".o"))
        run(["g++", "-std=gnu++14", "-O2", "-w"] + inc + ["-c", path, "-o", o])
        objs.append(o)
    run(["g++", "-o", exe] + objs + ["-lm"])
    for o in objs:
        os.remove(o)
    return exe


def main(argv):
    build_oracle_lib()
    names = argv[1:] or list(CONFIGS)
    for n in names:
        build_ref(n, force="--force" in argv)


if __name__ == "__main__":
    main([a for a in sys.argv if a != "--force"] + (["--force"] if "--force" in sys.argv else []))
