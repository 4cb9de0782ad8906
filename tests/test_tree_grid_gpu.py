"""More workgroups to a tree than the second index of a grid is given: rows gathered into slot order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [262144, 262145 + 8, 300001])  # 32768 workgroups of a gather of 512-byte rows, and more
def test_rows_of_a_long_tree(n, gpu_device):
    from hira_amd.indexer.hip import HIPIndexer

    keys = torch.arange(2 * n, device=gpu_device, dtype=torch.float32).reshape(1, 2, n, 1).repeat(1, 1, 1, 128)
    index = HIPIndexer(1, 0, 32).build(keys, keys)
    torch.cuda.synchronize()
    assert torch.equal(index.perm[:, :n].cpu(), torch.arange(n, dtype=torch.int32).expand(2, n))
    assert torch.equal(index.keys_rowmajor()[:, :n], keys[0]) and torch.equal(index.values_buf[:, :n], keys[0])
