"""Host build of the rule that picks the list build's form from the particles
and cells of an x-row (mdx::nbuild_form in mtcode_amd/csrc/mdx_device.h).  CPU
only."""
import os

import pytest

from test_wrap_host import HIPCC, host_build_and_run


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_form_of_the_list_build(tmp_path):
    r = host_build_and_run(tmp_path, "list_form_check")
    assert r.returncode == 0, r.stdout
    assert r.stdout.strip().endswith("ok")
