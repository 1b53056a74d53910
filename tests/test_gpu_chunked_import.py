"""ssd_chunked_scan imported under another default device than its inputs'."""
import importlib.util
import os

import pytest

pytestmark = pytest.mark.gpu


def test_import_under_a_default_device(cuda):
    import torch
    import ssd_chunked_scan
    spec = importlib.util.spec_from_file_location("ssd_chunked_scan_again", os.path.abspath(ssd_chunked_scan.__file__))
    again = importlib.util.module_from_spec(spec)
    with torch.device("meta"):
        spec.loader.exec_module(again)
    u = torch.randint(-1000, 1000, (1, 10, 8), dtype=torch.int32, device=cuda)
    n = torch.randint(16384, 32000, (1, 10, 8), dtype=torch.int32, device=cuda)
    for a, b in zip(again.ssd_chunked_scan_forward(u, n, 15, 4), ssd_chunked_scan.ssd_chunked_scan_forward(u, n, 15, 4)):
        assert a.device == b.device and torch.equal(a, b)
