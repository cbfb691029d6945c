"""The rates' kernels of a mechanism of many species keep to registers (the compiler's own report), where the
occupancy the nine-species mechanism is held to would spill."""

import re
import shutil
import subprocess

import support as sp
from peregrine_amd import build
from peregrine_amd.simulator import case_mechanism


def test_sixteen_species_rates_do_not_spill(tmp_path):
    mix = sp.mixture_of(sp.grown_mechanism(tmp_path, 16, 60))
    name, records, sets, _, _ = case_mechanism(mix)
    src = tmp_path / "peregrine_amd" / "csrc"
    (src / "generated").mkdir(parents=True)
    (tmp_path / "include").mkdir()
    shutil.copy2(build.HERE.parent / "include" / "peregrine_amd.h", tmp_path / "include")
    for path in [build.CSRC / "pga_stage.hip", *build.CSRC.glob("*.hpp")]:
        shutil.copy2(path, src)
    for file, text in build.variant_texts(mix.ns, mechanism=(name, records, sets)).items():
        (src / "generated" / file).write_text(text)
    r = subprocess.run([build.HIPCC, *build.FLAGS, "--offload-device-only", "-Rpass-analysis=kernel-resource-usage", "-c",
                        str(src / "pga_stage.hip"), "-o", str(tmp_path / "stage.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    scratch, kernel = {}, None
    for line in r.stderr.splitlines():
        if m := re.search(r"Function Name: (\S+)", line):
            kernel = m[1]
        elif m := re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line):
            scratch[kernel] = int(m[1])
    rates = {k: v for k, v in scratch.items() if "rates" in k}
    assert len(rates) == 2 and not any(rates.values()), rates
