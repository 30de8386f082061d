"""What the weight-streaming projections and the kernels that sum their
partials refuse, on the CPU: every buffer they write or read is checked before
the library is called."""

import pytest
import torch

import naivllm_amd.layers.qwen3 as qm

BF, F32 = torch.bfloat16, torch.float32


def z(*shape, dtype=BF):
    return torch.zeros(*shape, dtype=dtype)


M, N, K = 20, 1024, 256      # one split: y is written
SN, SK = 1024, 4096          # split: partials are written


def test_shapes_are_on_both_sides_of_the_split():
    assert qm.wide_splits(M, N, K) == 1 and qm.wide_splits(M, SN, SK) > 1


@pytest.mark.parametrize("y", [None, z(M, N, dtype=F32), z(M - 1, N), z(M, N - 16), z(M, 2 * N)[:, :N], z(M * N)])
def test_output_that_the_kernel_cannot_write(y):
    with pytest.raises(ValueError, match="y must be"):
        qm.wide_linear(z(M, K), z(N, K), y)


def test_swiglu_output_is_half_as_wide():
    with pytest.raises(ValueError, match="y must be"):
        qm.wide_linear(z(M, K), z(N, K), z(M, N), swiglu=True)


@pytest.mark.parametrize("x,w", [(z(M, K, dtype=F32), z(N, K)), (z(M, K), z(N, K, dtype=F32)), (z(K, M).t(), z(N, K))])
def test_operands(x, w):
    with pytest.raises(ValueError, match="contiguous bf16"):
        qm.wide_linear(x, w, z(M, N))


@pytest.mark.parametrize("scale,dtype", [(None, F32), (1, BF), (0.5, F32)])
def test_partials_of_a_split_projection(scale, dtype):
    splits = qm.wide_splits(M, SN, SK)
    part = None if scale is None else z(int(splits * M * SN * scale), dtype=dtype)
    with pytest.raises(ValueError, match="partials"):
        qm.wide_linear(z(M, SK), z(SN, SK), None, part)
    if part is not None:
        with pytest.raises(ValueError, match="partials"):
            qm.rms_norm_sum(part, splits, z(SN), 1e-6, z(M, SN), z(M, SN))
        with pytest.raises(ValueError, match="partials"):
            qm.qk_norm_rope_store_sum(part, splits, z(128), z(128), z(M, 128, dtype=F32), z(M, dtype=torch.int64),
                                      z(M, 4, 128), z(2, 16, 2, 128), z(2, 16, 2, 128), 4, 2, 128, 1e-6)


def test_sum_consumers_check_their_rows():
    part = z(2 * M * N, dtype=F32)
    for out, res, w in ((z(M, N), z(M - 1, N), z(N)), (z(M, N), z(M, N), z(N - 1)), (z(M, N), z(M, N, dtype=F32), z(N))):
        with pytest.raises(ValueError, match="rms_norm_sum"):
            qm.rms_norm_sum(part, 2, w, 1e-6, out, res)
    with pytest.raises(ValueError, match="slot_mapping"):
        qm.qk_norm_rope_store_sum(part, 2, z(128), z(128), z(M, 128, dtype=F32), z(M - 1, dtype=torch.int64),
                                  z(M, 4, 128), z(2, 16, 2, 128), z(2, 16, 2, 128), 4, 2, 128, 1e-6)


@pytest.mark.parametrize("M,N,K,taken", [
    (128, 16, 1 << 25, False),  # 2^30 bytes of weight, 2^33 of activations
    (128, 16, 1 << 23, False),  # 2^31 of activations, the first past an int
    (128, 16, (1 << 23) - (1 << 13), True),
    (1, 16, 1 << 25, False),    # one row is padded to two row tiles
    (128, 1 << 18, 4096, False),  # 2^31 of weight
    (128, 151936, 4096, True),
])
def test_shapes_past_32_bit_offsets_are_not_taken(M, N, K, taken):
    assert (qm.wide_splits(M, N, K) > 0) == taken


def test_packed_takes_the_packed_layouts_reductions():
    assert [qm.wide_splits(80, 1024, K, packed=True) for K in (512, 1024, 2048, 3072, 4096, 5120)] == [0, 1, 1, 0, 1, 0]


@pytest.mark.parametrize("hidden,rows,taken", [(1024, 81, False), (2048, 128, False), (2304, 13, True), (2304, 128, True),
                                               (2304, 129, False), (4096, 128, True)])
def test_layers_take_the_kernel_where_it_is_faster(hidden, rows, taken):
    # (up to hidden 2048 the library is, past the rows of the fused kernel)
    cfg = qm.Qwen3Config(vocab_size=64, hidden_size=hidden, num_layers=1, num_heads=2, num_kv_heads=1, head_dim=128,
                         intermediate_size=256, max_position=64)
    assert (qm.Qwen3Verify(cfg, "cpu")._wide_splits(rows) is not None) is taken
