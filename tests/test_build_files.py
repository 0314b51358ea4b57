"""The library's Makefile names files that exist and builds every source."""
import os
import re

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "xpbd-fem_amd")


def test_makefile_names_every_source_and_no_other():
    text = open(os.path.join(PKG, "Makefile")).read()
    named = set(re.findall(r"\$\(HERE\)((?:csrc|\.\.)/[\w./]+\.(?:hip|cpp|h))", text))
    missing = [f for f in named if not os.path.exists(os.path.join(PKG, f))]
    assert not missing, missing
    objects = set(re.findall(r"\$\(OBJDIR\)/(\w+)\.o", text))
    sources = {os.path.splitext(f)[0] for f in os.listdir(os.path.join(PKG, "csrc"))
               if f.endswith((".hip", ".cpp"))}
    assert sources == objects, sources ^ objects
    headers = {f for f in os.listdir(os.path.join(PKG, "csrc")) if f.startswith("xf_") and f.endswith(".h")}
    used = {os.path.basename(f) for f in named}
    # xf_geo_gpu.h is the callers' header, not one of the library's
    assert headers - used == {"xf_geo_gpu.h"}, headers - used
