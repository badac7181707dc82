"""What the native code promises about host memory, read from its source (it cannot be
seen from the outside): the record that the host polls while a kernel writes it is
coherent memory, and the pools that instances give their memory back to outlive every
instance (a program may close one in a static destructor)."""
import os
import re

from conftest import ROOT

SOURCE = open(os.path.join(ROOT, "espreso_amd", "csrc", "feti.hip")).read()


def test_polled_record_is_coherent():
    call = re.search(r"hipHostMalloc\(&p, sizeof\(PcgRecord\), ([^)]*)\)", SOURCE)
    assert call and "hipHostMallocCoherent" in call.group(1)


def test_pools_outlive_instances():
    pools = set(re.findall(r"(\w+)\(\)\.give_back\(", SOURCE))
    assert pools >= {"workspace_cache", "pinned_pool", "record_pool", "host_stages"}
    for pool in pools:
        body = re.search(r"(\w+) &%s\(\) \{(.*?)\n\}" % pool, SOURCE, re.S)
        assert re.search(r"static %s \*\w+ = new %s;" % (body.group(1), body.group(1)), body.group(2)), pool
