"""What the native code promises about host memory, read from its source (it cannot be
seen from the outside): the record that the host polls while a kernel writes it is
coherent memory."""
import os
import re

from conftest import ROOT

SOURCE = open(os.path.join(ROOT, "espreso_amd", "csrc", "feti.hip")).read()


def test_polled_record_is_coherent():
    call = re.search(r"hipHostMalloc\(&p, sizeof\(PcgRecord\), ([^)]*)\)", SOURCE)
    assert call and "hipHostMallocCoherent" in call.group(1)
