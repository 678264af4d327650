import ctypes
import os
import sys

import pytest

REPO_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if REPO_ROOT not in sys.path:
    sys.path.insert(0, REPO_ROOT)

import __graft_entry__ as entry  # noqa: E402


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def oracle():
    return entry.load_oracle()


@pytest.fixture(scope="session")
def nr_oracle():
    return entry.load_norm_rope_oracle()


@pytest.fixture(scope="session")
def dit_oracle():
    return entry.load_dit_attention_oracle()


@pytest.fixture(scope="session")
def block_oracle():
    return entry.load_dit_block_oracle()


@pytest.fixture(scope="session")
def net_oracle():
    return entry.load_dit_network_oracle()


@pytest.fixture(scope="session")
def pkg():
    """The package with its HIP library loaded; fails loudly when the library is not built."""
    return entry.load_package()


@pytest.fixture(scope="session")
def gpu():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return torch.device("cuda:0")


@pytest.fixture
def stream_override(pkg):
    """``stream_override(chunk=..., groups=...)`` steers short key sequences to (or away from) the query-streaming kernels through the
    library's own hook ``cosmos_attn_set_stream_override``; the library's choice is restored after the test."""
    lib = pkg._lib.load_library()

    def set_(chunk=0, groups=0):
        lib.cosmos_attn_set_stream_override(int(chunk), int(groups))

    yield set_
    lib.cosmos_attn_set_stream_override(0, 0)


@pytest.fixture
def forward_override(pkg):
    """``forward_override(rows=..., ranges=...)`` picks the workgroup shape and the key ranges of the forward-only kernel through
    ``cosmos_attn_set_forward_override``; the library's choice is restored after the test."""
    lib = pkg._lib.load_library()

    def set_(rows=0, ranges=0):
        assert lib.cosmos_attn_set_forward_override(int(rows), int(ranges)) == 0

    yield set_
    lib.cosmos_attn_set_forward_override(0, 0)


@pytest.fixture
def forward_plan(pkg):
    """``forward_plan((B, H, Lq, d), Lkv, dv=, causal=, padded=)``: (query rows, key groups, whole pairs, cut pairs, key ranges) that a
    forward-only call of dense tensors runs, or "streamed"."""
    L, lib = pkg._lib, pkg._lib.load_library()

    def plan_(shape_q, Lkv, dv=None, causal=False, padded=False):
        (B, H, Lq, d), dv = shape_q, dv or shape_q[3]
        D, plan, somewhere = L.AttnDesc(), L.AttnPlan(), 0x7F0000000000      # (never dereferenced)
        D.abi_version, D.dtype = L.ABI_VERSION, L.DTYPE_BF16
        D.B, D.H, D.Lq, D.Lkv, D.d_qk, D.d_v, D.causal, D.sm_scale = B, H, Lq, Lkv, d, dv, int(causal), d ** -0.5
        D.q = D.k = D.v = D.o = somewhere
        D.key_lens = somewhere if padded else None
        for name, rows, dim in (("q_stride", Lq, d), ("k_stride", Lkv, d), ("v_stride", Lkv, dv), ("o_stride", Lq, dv)):
            setattr(D, name, (ctypes.c_int64 * 3)(H * rows * dim, rows * dim, dim))
        assert lib.cosmos_attn_launch_plan(ctypes.byref(D), ctypes.c_size_t(-1).value, ctypes.byref(plan)) == 0
        return "streamed" if plan.streaming_workgroups else tuple(getattr(plan, name) for name, _ in plan._fields_[1:])

    return plan_
