"""Direct loads to LDS are written in one place, which names what they change and takes addresses."""

import pathlib
import re

CSRC = pathlib.Path(__file__).parent.parent / "automodel_amd" / "ops" / "csrc"


def test_direct_loads():
    places = [p.name for p in sorted(CSRC.iterdir()) if p.is_file() and "global_load_lds" in p.read_text()]
    assert places == ["lds_load.h"]
    text = (CSRC / "lds_load.h").read_text()
    blocks = re.findall(r"asm volatile\((.*?)\);", text, re.S)
    loads = [b for b in blocks if "m0" in b]
    assert loads and all(re.search(r':\s*"memory", "m0"\s*$', b) for b in loads)
    # every user passes an address of its shared memory, not an offset into it
    for p in CSRC.iterdir():
        if p.suffix == ".hip" and re.search(r"\bload_(tile<|lds16\()", p.read_text()):
            assert "lds_address(" in p.read_text(), p.name
