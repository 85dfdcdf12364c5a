"""What the entry points would launch, seen without a GPU: calls at sizes no test could run, on a stand-in for the HIP runtime
(hip_stub.c).  A process of its own, since the library takes the runtime it is loaded with."""
import ctypes as C
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
DEVICE = lambda k: k << 40   # an address that nothing reads


@pytest.fixture(scope="module")
def launches(lt, tmp_path_factory):
    """launches(entry point, arguments) -> {"rc", "error", "kernel", "launches": [[kernel, grid x, y, z, threads, LDS], ...]}.  An
    argument {"qparams": [scales, zero points]} stands for lten_hip_qparams."""
    stub = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", stub, os.path.join(HERE, "hip_stub.c")], check=True)

    def run(name, *args, variant=0):
        out = subprocess.run([sys.executable, __file__, stub, name, json.dumps(args), str(variant)], check=True, stdout=subprocess.PIPE, text=True)
        return json.loads(out.stdout.splitlines()[-1])
    return run


def call_on_the_stub(stub_path, name, args, variant):
    stub = C.CDLL(stub_path, mode=C.RTLD_GLOBAL)   # before the library, whose HIP calls it takes
    stub.stub_name.restype = C.c_char_p
    sys.path.insert(0, HERE)
    from conftest import load_package
    lt = load_package()
    lt.set_option("conv_variant", variant)
    rc = getattr(lt.lib(), name)(*[lt.qparams3(*a["qparams"]) if isinstance(a, dict) else a for a in args])
    seen, dims = [], (C.c_uint64 * 5)()
    for i in range(stub.stub_launches()):
        stub.stub_dims(i, dims)
        seen.append([stub.stub_name(i).decode(), *dims])
    return {"rc": rc, "error": (lt.lib().lten_hip_last_error() or b"").decode() if rc else "", "kernel": lt.last_kernel(), "launches": seen}


@pytest.mark.parametrize("N,C_in,H,W", [(65535, 4100, 1, 1), (1100, 1 << 18, 1, 3), (65535, 2, 2, 1)])
@pytest.mark.parametrize("entry", ["forward", "dgrad"])
def test_planes_of_less_than_a_quad_stay_within_32_bits(launches, entry, N, C_in, H, W):
    """Such planes are staged from a copy with four values each, by offsets of 32 bits: no part of it may reach 2^32 bytes, and
    the parts are all planes."""
    if entry == "forward":
        r = launches("lten_hip_conv2d_forward_f32", N, C_in, H, W, 64, 3, 3, 1, 1, 1, 1, DEVICE(1), DEVICE(2), None, DEVICE(3))
    else:
        r = launches("lten_hip_conv2d_dgrad_f32", N, 64, H, W, C_in, 3, 3, 1, 1, 1, 1, DEVICE(1), DEVICE(2), DEVICE(3), DEVICE(4))
    assert r["rc"] == 0, r["error"]
    copies = [x * threads for name, x, _, _, threads, _ in r["launches"] if "pad_planes" in name]
    assert ("pieces" in r["kernel"]) == bool(copies), r["kernel"]
    assert all(planes * 16 <= 1 << 32 for planes in copies), copies
    assert not copies or N * C_in <= sum(copies) < N * C_in + 256 * len(copies)


QP = {"qparams": [[0.02, 0.013, 0.9], [17, 125, 100]]}


@pytest.mark.parametrize("geo", [(65535, 8, 16000, 9, 1, 3, 3, 1, 1, 1, 1),       # bands of a few rows, many of them
                                 (16297, 5, 5225, 479, 124, 3, 3, 0, 2, 1, 1),
                                 (38160, 4, 2927, 152, 71, 2, 2, 1, 1, 1, 1),     # at most 64 taps
                                 (27108, 284, 3000, 29, 4, 3, 3, 2, 1, 1, 2)])    # no other kernel of one launch
def test_conv2dq_of_very_many_bands(launches, geo):
    """2^23 bands of 512 threads and more are no launch: the other kernels take the layer, or the same one with taller bands."""
    r = launches("lten_hip_conv2dq_forward", *geo, DEVICE(1), DEVICE(2), None, QP, DEVICE(3), DEVICE(4))
    assert r["rc"] == 0, r["error"]


@pytest.mark.parametrize("geo,kernel", [((4, 128, 120, 120, 32, 3, 3, 1, 1, 1, 1), "conv2dq_region"),
                                        ((127, 50, 10, 92, 15, 5, 5, 2, 4, 1, 1), "conv2dq_region"),
                                        ((64, 256, 100, 100, 256, 3, 3, 1, 1, 1, 1), "conv2dq_pixels")])
def test_conv2dq_layers_that_want_a_workspace(launches, geo, kernel):
    """Windows without a plan of one launch in 64 KB of LDS are refused without a workspace, whatever they run as with one."""
    r = launches("lten_hip_conv2dq_forward", *geo, DEVICE(1), DEVICE(2), None, QP, DEVICE(3), None)
    assert (r["rc"], r["error"]) == (2, "conv2dq: workspace is null")
    r = launches("lten_hip_conv2dq_forward", *geo, DEVICE(1), DEVICE(2), None, QP, DEVICE(3), DEVICE(4))
    assert (r["rc"], r["kernel"]) == (0, kernel), r["error"]


@pytest.mark.parametrize("geo,kernel", [((32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1), "conv2dq_region"),    # us in the band in LDS, two launches, the band kernel: 12.0, 16.1, 28.6
                                        ((52, 173, 32, 32, 80, 1, 1, 0, 0, 2, 2), "conv2dq_region"),   # 9.4, -, 23.0 (the pixels would not fit the workspace)
                                        ((3, 25, 72, 72, 32, 3, 3, 1, 1, 1, 1), "conv2dq_pixels"),     # 8.2, 6.9, -
                                        ((60, 48, 72, 72, 112, 3, 3, 1, 1, 2, 2), "conv2dq_pixels"),   # 24.2, 20.2, -
                                        ((1, 52, 15, 15, 220, 3, 3, 1, 1, 2, 2), "conv2dq_pixels"),    # 8.1, 6.3, -
                                        ((2, 26, 36, 36, 16, 3, 3, 1, 1, 2, 2), "conv2dq_band"),       # 8.0, -, 6.8
                                        ((21, 1, 89, 7, 473, 3, 3, 1, 1, 3, 3), "conv2dq_pixels")])    # 9.6, 7.1, -
def test_conv2dq_layers_run_as_what_is_quickest(launches, geo, kernel):
    """Layers whose kernels lie well apart, at the values of a measurement."""
    r = launches("lten_hip_conv2dq_forward", *geo, DEVICE(1), DEVICE(2), None, QP, DEVICE(3), DEVICE(4))
    assert (r["rc"], r["kernel"]) == (0, kernel), r["error"]


# (bands of an image, blocks of 32 channels a wavefront multiplies at once) of the layers that the GPU tests force on the band in LDS
@pytest.mark.parametrize("geo,bands,fn", [((32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1), 8, 2), ((64, 16, 112, 112, 60, 3, 3, 1, 1, 2, 2), 4, 2),
                                          ((64, 16, 56, 56, 32, 3, 3, 1, 1, 1, 1), 4, 1), ((64, 15, 57, 55, 29, 3, 3, 1, 1, 1, 1), 4, 1),
                                          ((40, 14, 111, 109, 70, 3, 3, 1, 1, 2, 2), 8, 2), ((64, 48, 28, 28, 120, 1, 1, 0, 0, 1, 1), 2, 2),
                                          ((3, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1), 56, 1)])
def test_conv2dq_region_bands(launches, geo, bands, fn):
    N, Cout = geo[0], geo[4]
    r = launches("lten_hip_conv2dq_forward", *geo, DEVICE(1), DEVICE(2), None, QP, DEVICE(3), DEVICE(4), variant=20)
    assert (r["rc"], r["kernel"], len(r["launches"])) == (0, "conv2dq_region", 1), r["error"]
    name, x, y, z, *_ = r["launches"][0]
    assert (x, y, z) == (N * bands, (Cout + 63) // 64, 1) and f"ELi{fn}E" in name, r["launches"]


@pytest.mark.parametrize("geo,kernel", [((23, 5, 111, 107, 15, 3, 3, 1, 0, 1, 1), "conv2d_patch_forward_3x3_32x4x128"),    # us there and on pieces: 22, 30
                                        ((18, 7, 100, 100, 205, 3, 3, 0, 1, 1, 1), "conv2d_patch_forward_3x3_32x4x128"),   # 86, 108 to 144
                                        ((23, 3, 88, 88, 20, 7, 7, 0, 0, 1, 1), "conv2d_forward_32x128x32"),               # 41, 50
                                        ((53, 8, 29, 29, 32, 5, 5, 0, 0, 1, 1), "conv2d_pieces_forward"),                  # 22, 17
                                        ((21, 372, 13, 124, 6, 3, 3, 1, 2, 1, 1), "conv2d_pieces_forward")])               # 199, 59
def test_conv2d_layers_run_as_what_is_quickest(launches, geo, kernel):
    """Forward layers whose routes lie well apart, at the values of a measurement."""
    r = launches("lten_hip_conv2d_forward_f32", *geo, DEVICE(1), DEVICE(2), None, DEVICE(3))
    assert (r["rc"], r["kernel"]) == (0, kernel), r["error"]


@pytest.mark.parametrize("geo,tile,tiles", [((208, 48, 22, 22, 13, 5, 5, 4, 2, 2, 2), "ILi64ELi128ELi2ELi2ELi210E", 244),   # 122 pixels to a tile: one round
                                            ((32, 64, 32, 32, 32, 5, 5, 2, 2, 1, 1), "ILi32ELi256E", 128)])              # not 64 rows for 32 channels
def test_conv2d_tiles_on_pieces(launches, geo, tile, tiles):
    """The tile and, up to the CUs, how many of them: pixels to a tile in no steps of 16, no tile half of whose rows are padding."""
    r = launches("lten_hip_conv2d_forward_f32", *geo, DEVICE(1), DEVICE(2), None, DEVICE(3))
    seen = [(name, x) for name, x, *_ in r["launches"] if "conv_split_kernel" in name]
    assert len(seen) == 1 and tile in seen[0][0] and seen[0][1] == (tiles + 7) // 8 * 8, seen


if __name__ == "__main__":
    print(json.dumps(call_on_the_stub(sys.argv[1], sys.argv[2], json.loads(sys.argv[3]), int(sys.argv[4]))))
