"""Which kernel a 16-bit linear layer takes (hb_linear_kernel, no GPU call): the lines of the rule, at sizes where both sides were measured on 256 CUs."""
import ctypes

import pytest

from laya_hip import ffi as F

GEGLU, XP, YP = F.HB_EPI_GEGLU, F.HB_X_PANEL, F.HB_Y_PANEL


def kernel(M, N, K, flags=0, ldx=None, cus=256, bits=0):
    name = ctypes.create_string_buffer(64)
    n = F.native()
    n.call("linear_kernel", "hb_linear_kernel", cus, K if ldx is None else ldx, M, N, K, bits, flags, name, len(name))
    return name.value.decode()


@pytest.mark.parametrize("M,N,K,geglu,want", [
    (1, 768, 768, 0, "ring 32x64"), (93, 2304, 768, 0, "ring 32x64"), (256, 2304, 768, 0, "ring 64x64"),
    (768, 768, 3072, 0, "ring 64x64 long"), (512, 3072, 768, 0, "ring 128x64"), (512, 1152, 768, 1, "ring 128x64"),
    (1024, 2304, 768, 0, "ring 64x64 three"), (3840, 768, 768, 0, "ring 64x64 three"),
    (2048, 2304, 768, 0, "mfma 128x64"), (2048, 3072, 768, 0, "ring 128x256"), (3584, 2304, 768, 0, "ring 128x256"), (2560, 3072, 1024, 0, "ring 128x256"),
    # the 128-row kernel where the ring's tiles were slower: GeGLU, K = 3072, more than a round
    (2048, 1152, 768, 1, "mfma 128x64"), (3072, 1152, 768, 1, "mfma 128x128"), (2048, 2304, 3072, 0, "mfma 128x64"),
    (700, 2624, 1024, 1, "mfma 128x64"), (2048, 2624, 1024, 1, "mfma 128x128"), (3072, 2624, 1024, 1, "mfma 128x128"),
    (1536, 2304, 768, 0, "mfma 128x64"), (1024, 4096, 1024, 0, "mfma 128x64"), (3840, 4096, 1024, 0, "mfma 128x128"),
    (3840, 1024, 4096, 0, "mfma 128x64"), (700, 50368, 768, 0, "mfma 128x128"),
    # its 128 x 128 tiles just over two a CU: the ring's three rounds
    (3840, 2304, 768, 0, "ring 64x64 three"), (3072, 3072, 1024, 0, "ring 64x64 three"),
    (1792, 5248, 1024, 0, "mfma 128x128"),
    # other K; from M = 4096
    (512, 768, 776, 0, "mfma 128x64"), (4096, 2304, 768, 0, "arow 192"), (4096, 768, 768, 0, "ring 64x64 three"),
    (16384, 1024, 1024, 0, "arow 128"), (4096, 768, 776, 0, "arow 192 tail"),
    (4200, 1536, 384, 0, "ring 128x256"), (4200, 640, 768, 1, "ring 128x256"), (5500, 768, 3072, 0, "ring 128x256"),
])
def test_the_rule(M, N, K, geglu, want):
    assert kernel(M, N, K, GEGLU if geglu else 0) == want


def test_panel_order_operands_never_meet_the_kernel_without_them():
    """Every call that check_panel accepts below M = 4096 takes a kernel that reads
    and writes panel order, whatever the other operand's row stride."""
    for K in (64, 768, 1280, 2560):
        for N in (16, 48, 768, 2304, 8192):
            for M in (1, 33, 128, 500, 1300, 4000):
                for geglu in (0, GEGLU):
                    if 64 * K * (2 if geglu else 1) > 160 * 1024 or -(-N // 32) * -(-M // 128) > 256:
                        continue
                    for flags in (XP, YP, XP | YP):
                        for ldx in (K, (1 << 22) - 8, 1 << 22, 1 << 26):
                            got = kernel(M, N, K, geglu | flags, ldx)
                            assert not got.startswith("mfma"), (M, N, K, geglu, flags, ldx, got)
                            if not flags & XP and ldx >= 1 << 22:  # past 32-bit offsets
                                assert got.endswith("tail"), (M, N, K, ldx, got)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("M,N,K,geglu,want", [
    (1, 768, 768, 0, "ring 32x64"), (128, 2304, 768, 0, "ring 32x64"), (512, 768, 1152, 0, "ring 32x64"),
    (512, 1152, 768, 1, "ring 128x64"), (256, 2624, 1024, 1, "ring 128x64"), (1024, 3072, 1024, 0, "ring 64x64 three"),
    (2048, 2304, 768, 0, "ring 128x256"), (3072, 2304, 768, 0, "ring 128x256"), (3072, 2624, 1024, 1, "mfma 128x128"), (16384, 2304, 768, 0, "arow 192"),
    # a short K chain, or a weight that is wide against it: the loader was faster
    (1, 48, 64, 0, "codes mfma 128x64"), (4000, 48, 64, 0, "codes mfma 128x64"), (256, 16384, 768, 0, "codes mfma 128x64"),
    (1, 50368, 768, 0, "codes mfma 128x128"), (33, 256000, 1024, 0, "codes mfma 128x128"),
    # where the 16-bit call takes the 128-row kernel on few tiles; other K
    (1536, 2304, 768, 0, "codes mfma 128x64"), (700, 2624, 1024, 1, "codes mfma 128x64"),
    (2048, 1152, 768, 1, "codes mfma 128x64"), (512, 768, 776, 0, "codes mfma 128x64"),
])
def test_where_codes_are_dequantized(M, N, K, geglu, want, bits):
    assert kernel(M, N, K, GEGLU if geglu else 0, bits=bits) == want
