"""CPU-side checks of the drop-in boundary: the C-ABI library loads and exports every symbol the
header declares; host-only entry points (geometry, sizes, error reporting) behave."""
import os
import re

import pytest

from tests import refmath as rm

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    txt = open(os.path.join(ROOT, "include", "tcbnn_hip.h")).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(tcbnn_[a-z0-9_]+)\s*\(", txt)))


def test_library_exports_every_declared_symbol():
    from tcbnn_amd import _lib
    syms = _declared_symbols()
    assert len(syms) >= 30
    for s in syms:
        assert hasattr(_lib.lib, s), "libtcbnn_hip.so does not export %s" % s
    assert sorted(_lib.ABI) == syms, "Python binding table and header disagree"
    assert _lib.lib.tcbnn_abi_version() == 7
    # the build entry point refuses a library of another ABI version: it must expect this one
    import inspect
    import __graft_entry__
    assert "tcbnn_abi_version() == 7" in inspect.getsource(__graft_entry__.build)


def test_geometry_entry_points_match_reference_formulas():
    from tcbnn_amd import _lib
    for h in range(1, 40):
        for s in (1, 2, 4):
            for r in (1, 3, 7, 11):
                for pool in (1, 2):
                    pad, buf, out = rm.conv_pad_out(h, r, s, True, pool)
                    assert _lib.lib.tcbnn_conv_pad(h, r, s, 1) == pad
                    assert _lib.lib.tcbnn_conv_out(h, r, s, 1, pool) == out
                    assert _lib.lib.tcbnn_conv_pad(h, r, s, 0) == 0


def test_size_helpers():
    from tcbnn_amd import _lib
    L = _lib.lib
    assert L.tcbnn_fc_act_words(8192, 784) == 8192 * 28
    assert L.tcbnn_conv_act_words(56, 56, 256, 64) == 56 * 56 * 256 * 2
    assert L.tcbnn_fc_weight_words(784, 10) == 32 * 28 + 32 * 8 * 4  # sign-bit rows + the copy in lane order
    assert L.tcbnn_conv_filter_words(3, 3, 64, 64) == 64 * 9 * 2 * 2   # sign bits + a copy in MFMA lane order
    assert L.tcbnn_conv_filter_words(3, 3, 96, 64) == 64 * 9 * 3       # sign bits only
    assert L.tcbnn_conv_filter_words(5, 5, 64, 40) == 64 * 25 * 2
    assert L.tcbnn_inconv_filter_words(7, 7, 3, 64) == 49 * 64 * 5
    # packed first-layer input: (P - 1) stride + R rows and columns of [batch][3]
    assert L.tcbnn_inconv_packed_input_floats(256, 224, 224, 7, 7, 4, 4, 1) == 227 * 227 * 256 * 3
    assert L.tcbnn_inconv_packed_input_floats(5, 32, 30, 3, 5, 1, 2, 1) == 34 * 33 * 5 * 3
    assert L.tcbnn_inconv_packed_input_floats(5, 16, 16, 3, 3, 2, 2, 0) == 15 * 15 * 5 * 3  # the last row is unused
    assert L.tcbnn_inconv_packed_input_floats(0, 16, 16, 3, 3, 1, 1, 1) == 0
    assert L.tcbnn_inconv_packed_input_floats(4, 2, 16, 3, 3, 1, 1, 0) == 0   # no output row


def test_errors_are_codes_not_exits():
    from tcbnn_amd import _lib
    L = _lib.lib
    assert L.tcbnn_fc128_forward(None, None) == -2
    assert b"NULL" in L.tcbnn_last_error()
    d = _lib.Fc128Desc(1, 1, 1, 1, 0, 128, 128, 0, None, 0)  # batch 0; never launches
    assert L.tcbnn_fc128_forward(d, None) == -1
    assert L.tcbnn_bmm(1, 1, 1, 8, 8, 100, 1, None) == -1  # K not a multiple of 32
    assert L.tcbnn_set_default_variant(99) == -1
    assert L.tcbnn_inconv_pack_input(None, None, 4, 8, 8, 3, 3, 1, 1, 1, None) == -2
    assert L.tcbnn_inconv_pack_input(1, 1, 0, 8, 8, 3, 3, 1, 1, 1, None) == -1  # batch 0; never launches
    with pytest.raises(_lib.TcbnnError):
        _lib.check(-1)


def test_no_long_k_is_refused_for_its_lds():
    """Int32 products and convolutions whose K is too long for the LDS of one kernel go to another one: on both sides of
    every such limit a call fails for want of a device and of nothing else (where there is one, nothing is called: the
    pointers are made up)."""
    from tcbnn_amd import _lib
    L = _lib.lib
    if _lib.device_count() > 0:
        pytest.skip("made-up pointers")
    for m, n, k in ((32, 32, 128000), (32, 32, 128032), (1, 4096, 130816), (1, 4096, 130848)):
        assert L.tcbnn_bmm(16, 16, 16, m, n, k, _lib.VARIANT_MFMA_F4, None) == -3, (m, n, k, L.tcbnn_last_error())
    for b, hw, cin, cout in ((64, 28, 4736, 256), (64, 28, 4768, 256), (64, 28, 5120, 256), (64, 56, 4800, 512)):
        assert L.tcbnn_bconv(16, 16, 16, b, hw, hw, cin, cout, 5, 5, 1, 1, 2, 2, hw, hw, _lib.VARIANT_MFMA_F4, None) == -3, \
            (b, hw, cin, cout, L.tcbnn_last_error())


def test_large_products_test_for_odd_words_only_where_there_can_be_any():
    """Fully connected layers, whose rows are whole 128-bit units, run an instantiation without that test."""
    import ctypes as C
    from tcbnn_amd import _lib
    name = C.create_string_buffer(128)
    d = _lib.Fc128Desc(1, 1, 1, 1, 8192, 784, 1024, _lib.VARIANT_MFMA_F4, None, 0)
    _lib.check(_lib.lib.tcbnn_fc128_kernel_name(C.byref(d), name, 128))
    assert name.value == b"gemm_mfma_f4_kernel<2, 0, false>"


def _fc_kernel(batch, k, n, out=False):
    import ctypes as C
    from tcbnn_amd import _lib
    name = C.create_string_buffer(128)
    if out:
        d = _lib.Out128Desc(1, 1, 1, 1, 1, batch, k, n, _lib.VARIANT_MFMA_F4)
        _lib.check(_lib.lib.tcbnn_out128_kernel_name(C.byref(d), name, 128))
    else:
        d = _lib.Fc128Desc(1, 1, 1, 1, batch, k, n, _lib.VARIANT_MFMA_F4, None, 0)
        _lib.check(_lib.lib.tcbnn_fc128_kernel_name(C.byref(d), name, 128))
    return name.value.decode()


@pytest.mark.parametrize("out", [False, True])
def test_large_products_only_where_their_sums_are_exact(out):
    """The large-product kernel's rows are values of 0 .. 6 (13/4 on average where all signs agree), summed in fp32: taken
    while that stays below 2^24, over K rounded up to groups of sixteen words."""
    batch, n = 64, 16384  # 256 workgroups; 2 GiB of rows lie beyond the longest K
    served = [k for k in range(128 * 39000, 1 << 24, 128) if _fc_kernel(batch, k, n, out).startswith("gemm_mfma")]
    assert served, "the longest products that are exact stay with this kernel"
    sums = 13 * (-(-max(served) // 512) * 512) // 4
    assert (1 << 24) - 13 * 512 // 4 < sums <= 1 << 24, max(served)
    assert "gemm_mfma" not in _fc_kernel(batch, (1 << 24) - 1, n, out)


@pytest.mark.parametrize("batch,k,n,out,kernel", [
    (212, 8825, 3484, False, "<0, 0, true>"), (94, 8794, 8046, True, "<1, 0, true>"),  # 763 and 756 tiles: nine groups a wave
    (512, 8825, 1024, False, "<0, 7, true>"), (512, 8825, 1025, False, "<0, 0, true>")])  # 512 tiles: seven waves; 528
def test_fc_layers_of_many_tiles_take_four_waves(batch, k, n, out, kernel):
    """513 tiles and more: one wave to a SIMD, four workgroups to a compute unit; five waves leave a SIMD twice the work."""
    assert _fc_kernel(batch, k, n, out) == "fc_mfma_f4_kernel" + kernel


@pytest.mark.parametrize("frame,stride,served", [(1, 1, True), (2, 2, True), (5, 8, False), (3, 7, False)])
def test_large_products_read_the_first_pixel(frame, stride, served):
    """One output pixel of a 1x1 filter is the frame's first one only without padding: ((5 + 8 - 5)/8 - 1)*8 + 1 - 5 = -4,
    halved: the pixel at (2, 2) of a 5x5 frame."""
    import ctypes as C
    from tcbnn_amd import _lib
    d = _lib.Conv128Desc(1, 1, 1, 1, None, None, frame, frame, 256, 1, 1, 1024, 8192, stride, stride, 1, 1, 1, 0, 0, 0, 0, 0, 0,
                         _lib.VARIANT_MFMA_F4, 0, 0, 0)
    name = C.create_string_buffer(128)
    _lib.check(_lib.lib.tcbnn_conv128_kernel_name(C.byref(d), name, 128))
    assert (_lib.lib.tcbnn_conv_pad(frame, 1, stride, 1) == 0) == served
    assert name.value.decode().startswith("gemm_mfma") == served, name.value


@pytest.mark.parametrize("batch,frame,cout,fmt,kernel", [
    (166, 21, 256, 0, "conv1x1"), (69, 49, 192, 0, "bgemm_flat"),                                    # 80 and 137 MB of int32
    (136, 37, 384, 0, "conv1x1"), (185, 54, 512, 0, "bgemm_flat"), (185, 54, 512, 1, "conv1x1")])    # 301 MB; 1.1 GB, and in 16 bits
def test_1x1_layers_with_large_int32_residuals(batch, frame, cout, fmt, kernel):
    """Launches whose int32 stores a persistent grid would scatter go to the kernel whose workgroups are dealt in order."""
    import ctypes as C
    from tcbnn_amd import _lib
    d = _lib.Conv128Desc(1, 1, 1, 1, None, 16, frame, frame, 256, 1, 1, cout, batch, 1, 1, 1, 1, 1, 0, 1, 0, 0, 0, 0,
                         _lib.VARIANT_MFMA_F4, 0, fmt, 0)
    name = C.create_string_buffer(128)
    _lib.check(_lib.lib.tcbnn_conv128_kernel_name(C.byref(d), name, 128))
    assert name.value.decode().startswith(kernel), name.value


def _device_kernels():
    """Name -> record of every kernel in the library, as its code objects describe them (their AMDGPU metadata notes)."""
    import struct
    msgpack = pytest.importorskip("msgpack")
    blob = open(os.path.join(ROOT, "tcbnn_amd", "libtcbnn_hip.so"), "rb").read()
    kernels, at = {}, blob.find(b"\x7fELF")
    while at >= 0:
        machine, = struct.unpack_from("<H", blob, at + 18)
        if machine == 224:  # EM_AMDGPU
            headers, = struct.unpack_from("<Q", blob, at + 32)
            size, count = struct.unpack_from("<HH", blob, at + 54)
            for i in range(count):
                kind, _, offset, _, _, length = struct.unpack_from("<IIQQQQ", blob, at + headers + i * size)
                note, end = at + offset, at + offset + length
                while kind == 4 and note < end:  # PT_NOTE
                    name, desc, which = struct.unpack_from("<III", blob, note)
                    body = note + 12 + (name + 3) // 4 * 4
                    if which == 32:  # NT_AMDGPU_METADATA
                        for k in msgpack.unpackb(blob[body:body + desc])["amdhsa.kernels"]:
                            kernels[k[".name"]] = k
                    note = body + (desc + 3) // 4 * 4
        at = blob.find(b"\x7fELF", at + 4)
    return kernels


def test_twelve_waves_of_the_3x3_kernel_do_not_spill():
    """Twelve waves a workgroup leave a wave 168 registers: taken only by the instantiations that fit them."""
    twelve = {name: k for name, k in _device_kernels().items() if "conv3x3_mfma" in name and k[".max_flat_workgroup_size"] == 768}
    assert len(twelve) >= 10
    assert not {name: k[".vgpr_spill_count"] for name, k in twelve.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}


def test_long_3x3_tiles_keep_their_operands_in_registers():
    """192 channels and more (three chunks a tile): requests between the products must not push operands out of registers."""
    spills = {name: k[".vgpr_spill_count"] for name, k in _device_kernels().items()
              if re.search(r"conv3x3_mfma_f4_kernelILi[3468]E", name) and k[".vgpr_spill_count"] > 1}
    assert not spills


_B = 8192  # (a batch at which two layers are faster together)


@pytest.mark.parametrize("run,moved,to,apart", [
    ("fc fc", None, None, True), ("in fc", None, None, True), ("fc out", None, None, True),
    # neighbours in memory, and one byte's worth too near
    ("fc fc", "output 1", ("input 0", _B * 16 * 4), True), ("fc fc", "output 1", ("input 0", _B * 16 * 4 - 4), False),
    ("fc fc", "output 1", ("input 0", -_B * 12 * 4), True), ("fc fc", "output 1", ("input 0", -_B * 12 * 4 + 4), False),
    # two buffers in turn; both outputs in one; an output over what a layer reads before or after it is written
    ("fc fc", "output 1", ("input 0", 0), False), ("fc fc", "output 1", ("output 0", 0), False), ("fc fc", "output 1", ("output 0", 16), False),
    ("fc fc", "weight 1", ("output 0", 64), False), ("fc fc", "scale 0", ("output 1", 4), False),
    ("in fc", "output 0", ("x", _B * 500 * 4 - 4), False), ("in fc", "output 0", ("x", _B * 500 * 4), True), ("in fc", "scale 0", ("input 0", 0), False),
    ("fc out", "output 1", ("input 0", 0), False), ("fc out", "output 1", ("output 0", -_B * 10 * 4 + 4), False),
    ("fc out", "output 1", ("output 0", -_B * 10 * 4), True), ("fc out", "bias", ("output 1", 8), False)])
def test_layers_that_share_memory_are_not_one_launch(run, moved, to, apart):
    """Layers launched one by one may write where an earlier one has read or written; inside one launch of a run nothing
    orders them, so such a run is not one."""
    import ctypes as C
    from tcbnn_amd import _lib
    widths = (500, 500, 10 if "out" in run else 380)
    at = {name: 0x10000000 * (1 + i) for i, name in enumerate(("x", "input 0", "weight 0", "scale 0", "output 0", "weight 1", "scale 1", "bias", "output 1"))}
    if moved is not None:
        at[moved] = at[to[0]] + to[1]
    fc = (_lib.Fc128Desc * 2)()
    fc[0] = _lib.Fc128Desc(at["input 0"], at["weight 0"], at["scale 0"], at["output 0"], _B, widths[0], widths[1], _lib.VARIANT_MFMA_F4, None, 0)
    fc[1] = _lib.Fc128Desc(at["output 0"], at["weight 1"], at["scale 1"], at["output 1"], _B, widths[1], widths[2], _lib.VARIANT_MFMA_F4, None, 0)
    fin = _lib.In128Desc(at["x"], at["input 0"], _B, widths[0])
    out = _lib.Out128Desc(at["output 0"], at["weight 1"], at["scale 1"], at["bias"], at["output 1"], _B, widths[1], widths[2], _lib.VARIANT_MFMA_F4)
    layers, n = (C.c_int * 4)(), C.c_int()
    _lib.check(_lib.lib.tcbnn_fc_chain_plan(C.byref(fin) if "in" in run else None, fc, 2 if run == "fc fc" else 1, C.byref(out) if "out" in run else None, layers, C.byref(n)))
    assert layers[:n.value] == ([2] if apart else [1, 1])


@pytest.mark.parametrize("batch,widths,with_in,with_out,launches", [
    # the MLP, at every batch; layers too wide for one compute unit until there are many images
    (1, (784, 1024, 1024, 1024, 10), True, True, [5]), (8192, (784, 1024, 1024, 1024, 10), True, True, [5]),
    (16384, (784, 1024, 1024, 1024, 10), True, True, [5]),
    (1024, (784, 2048, 2048, 2048, 10), True, True, [1] * 5), (2048, (784, 2048, 2048, 2048, 10), True, True, [5]),
    # two layers: where few images leave most compute units without work, launches of their own are faster
    (256, (1024, 1024, 10), False, True, [1, 1]), (768, (1024, 1024, 10), False, True, [1, 1]), (2048, (1024, 1024, 10), False, True, [1, 1]),
    (4096, (1024, 1024, 10), False, True, [2]), (8192, (64, 64, 10), False, True, [1, 1]), (1024, (512, 512, 10), False, True, [1, 1]),
    # many numbers to store; little to multiply for many images
    (64, (512, 1024, 1000), False, True, [1, 1]), (8, (256, 512, 512, 1000), True, True, [1] * 4), (16384, (200, 100, 50, 10), True, True, [1] * 4),
    (9000, (784, 128, 10), True, True, [3]), (12000, (64, 64, 64, 64, 64, 10), False, True, [1] * 5), (12000, (512, 512, 512, 10), False, True, [3]),
    # the input's signs and one layer
    (1, (784, 256), True, False, [2]), (64, (100, 50), True, False, [1, 1]), (1024, (512, 512), True, False, [1, 1]), (8192, (512, 512), True, False, [2])])
def test_which_layers_of_a_run_are_one_launch(batch, widths, with_in, with_out, launches):
    """The choice between one launch and one per layer, where both sides were timed."""
    import ctypes as C
    from tcbnn_amd import _lib
    n = len(widths) - 1 - int(with_out)
    fc, at = (_lib.Fc128Desc * n)(), [0x100000000 * (1 + i) for i in range(16)]
    for i in range(n):
        fc[i] = _lib.Fc128Desc(at[i], at[14] + 0x1000000 * i, at[15] + 0x1000000 * i, at[i + 1], batch, widths[i], widths[i + 1], _lib.VARIANT_MFMA_F4, None, 0)
    fin = _lib.In128Desc(at[13], at[0], batch, widths[0])
    out = _lib.Out128Desc(at[n], at[12], at[11], at[10], at[9], batch, widths[-2], widths[-1], _lib.VARIANT_MFMA_F4)
    layers, got = (C.c_int * 16)(), C.c_int()
    _lib.check(_lib.lib.tcbnn_fc_chain_plan(C.byref(fin) if with_in else None, fc, n, C.byref(out) if with_out else None, layers, C.byref(got)))
    assert layers[:got.value] == launches


def test_network_specs_match_reference_wiring():
    from tcbnn_amd import nets
    spec = nets.imagenet_resnet_spec(batch=256)
    assert len(spec) == 19
    by = {L["name"]: L for L in spec}
    assert by["Conv1"]["stride"] == 4 and by["Conv1"]["save_residual"]
    assert by["L2B1C2"]["residual_pool"] and by["L2B1C2"]["res_src"] == "L1B2C2"
    assert by["L3B1C2"]["residual_channels"] == 128 and by["L4B1C2"]["residual_channels"] == 256
    assert by["L1B2C2"]["residual_channels"] == 128 and by["L4B2C2"]["ahead_fc"]
    assert by["Fc1"]["inp"] == 7 * 7 * 512
    bops, flops = nets.binary_ops(spec)
    assert abs(bops / 256 / 1e9 - 3.379) < 0.01  # binary ops per image
    assert abs(flops / 1e9 - 15.1) < 0.1
    bops, _ = nets.binary_ops(nets.mnist_mlp_spec(8192))
    assert abs(bops / 1e9 - 47.68) < 0.05
    bops, _ = nets.binary_ops(nets.cifar10_vgg_spec(256))
    assert abs(bops / 1e9 - 314.1) < 0.5


def test_network_plans_its_runs_of_layers_once(monkeypatch):
    """forward() works out which layers go in one call when their order is new, not on every pass."""
    from tcbnn_amd import layers, nets
    calls, planned, plan = [], [], layers.fc_runs

    class Conv:
        def forward(self, stream=None):
            calls.append(self)

    def counted(order):
        planned.append(len(order))
        return plan(order)

    def together(run, stream=None):
        calls.extend(run)

    monkeypatch.setattr(nets, "fc_runs", counted)
    monkeypatch.setattr(nets, "fc_launches", lambda run: [run])
    monkeypatch.setattr(nets, "forward_fc_run", together)
    fc = [layers.Fc128LayerParam("Fc%d" % i, 8, 64, 64) for i in range(2)]
    out = layers.Out128LayerParam("Fout", 8, 64, 10)
    alone = layers.Out128LayerParam("Aux", 8, 64, 10)
    monkeypatch.setattr(alone, "forward", lambda stream=None: calls.append(alone), raising=False)
    net = nets.Network([], [], None)  # (plans the order that it makes: nothing here)
    assert planned == [0]
    del planned[:]
    net.order = [Conv(), Conv()] + fc + [out, alone]
    for _ in range(3):
        net.forward()
    assert planned == [6] and calls == 3 * net.order
    assert [len(run) for run in plan(net.order)] == [1, 1, 3, 1]
    del calls[:], planned[:]
    net.order.insert(1, Conv())  # in place
    net.forward()
    net.order = net.order[2:]
    net.forward()
    net.forward()
    assert planned == [7, 5] and len(calls) == 7 + 2 * 5


def test_a_run_of_layers_makes_no_types_of_its_own(monkeypatch):
    """The descriptors' array type outlives the call and a collection: a new network's first pass does not make it again."""
    import gc
    import weakref
    from tcbnn_amd import layers
    made = []

    class Lib:
        @staticmethod
        def tcbnn_fc_chain_forward(first, array, n, last, stream):
            made.append(weakref.ref(type(array)))
            return 0

    run = [layers.Fc128LayerParam("Fc%d" % i, 8, 64, 64) for i in range(3)] + [layers.Out128LayerParam("Fout", 8, 64, 10)]
    for layer in run:
        layer._desc = layers._lib.Out128Desc if layer is run[-1] else layers._lib.Fc128Desc
    monkeypatch.setattr(layers, "lib", Lib)
    for _ in range(2):
        layers.forward_fc_run(run)
        gc.collect()
    assert made[0]() is not None and made[0]() is made[1]()


def test_residual_formats_sizes_and_choice():
    """Host-only helpers of the residual storage formats: bytes per tensor, and the narrowest format a bound allows
    (12 bits need an even batch: the format's 128-bit accesses are aligned only then)."""
    from tcbnn_amd import _lib
    L = _lib.lib
    h, w, c, b = 5, 7, 64, 6
    assert L.tcbnn_residual_bytes(h, w, c, b, _lib.RES_I32) == h * w * c * b * 4
    assert L.tcbnn_residual_bytes(h, w, c, b, _lib.RES_I16) == h * w * c * b * 2
    assert L.tcbnn_residual_bytes(h, w, c, b, _lib.RES_I12) == h * w * c * b * 3 // 2
    # channels are stored in whole groups: 4 (int32), 8 (int16) or 16 (12 bits)
    assert L.tcbnn_residual_bytes(1, 1, 17, 2, _lib.RES_I32) == 20 * 2 * 4
    assert L.tcbnn_residual_bytes(1, 1, 17, 2, _lib.RES_I16) == 24 * 2 * 2
    assert L.tcbnn_residual_bytes(1, 1, 17, 2, _lib.RES_I12) == 32 * 2 * 3 // 2
    for bound, batch, want in ((0, 2, _lib.RES_I12), (2047, 256, _lib.RES_I12), (2048, 256, _lib.RES_I16),
                               (2047, 255, _lib.RES_I16), (32767, 8, _lib.RES_I16), (32768, 8, _lib.RES_I32),
                               (-1, 8, _lib.RES_I32), (2 ** 31 - 1, 8, _lib.RES_I32)):
        assert L.tcbnn_residual_format_narrowest(bound, batch) == want, (bound, batch)
    assert L.tcbnn_residual_format_for_bound(2047) == _lib.RES_I16  # (never 12 bits: it does not know the batch)
    assert L.tcbnn_conv_residual_bound(64, 3, 3, 155) == 155 + 576
    assert L.tcbnn_conv_residual_bound(64, 3, 3, 0) == 576


def test_first_layer_bound_of_input_is_the_largest_window_sum():
    """tcbnn_inconv_residual_bound_of_input against a brute-force window walk in numpy: no first-layer sum can
    exceed the largest sum of |x| over one filter window (all three channels), and the returned bound lies between
    that sum and that sum * 1.001 + 2."""
    import ctypes as C

    import numpy as np
    from tcbnn_amd import _lib
    L = _lib.lib
    rng = np.random.default_rng(11)
    for (b, h, w, r, s, sh, sw, padding) in ((2, 9, 11, 3, 3, 1, 1, 1), (3, 16, 13, 7, 7, 4, 4, 1), (1, 12, 12, 5, 3, 2, 1, 0),
                                             (2, 23, 19, 11, 11, 4, 4, 1), (1, 7, 7, 7, 7, 1, 1, 1)):
        x = (rng.standard_normal((b, 3, h, w)) * rng.uniform(0.1, 30)).astype(np.float32)
        pad_h, pad_w = L.tcbnn_conv_pad(h, r, sh, padding), L.tcbnn_conv_pad(w, s, sw, padding)
        oh, ow = L.tcbnn_conv_out(h, r, sh, padding, 1), L.tcbnn_conv_out(w, s, sw, padding, 1)
        a = np.abs(x.astype(np.float64)).sum(axis=1)
        worst = 0.0
        for y in range(oh):
            for xx in range(ow):
                y0, x0 = y * sh - pad_h, xx * sw - pad_w
                win = a[:, max(0, y0):min(h, y0 + r), max(0, x0):min(w, x0 + s)]
                worst = max(worst, float(win.sum(axis=(1, 2)).max()))
        got = L.tcbnn_inconv_residual_bound_of_input(x.ctypes.data_as(C.c_void_p), b, h, w, r, s, sh, sw, padding)
        assert worst <= got <= worst * 1.001 + 2, (got, worst)
        # and it is a bound: the largest |sum| any +-1 filter can reach is that window's sum of |x|
        assert got >= np.floor(worst)
    bad = np.ones((1, 3, 8, 8), np.float32)
    bad[0, 1, 3, 3] = np.nan
    assert L.tcbnn_inconv_residual_bound_of_input(bad.ctypes.data_as(C.c_void_p), 1, 8, 8, 3, 3, 1, 1, 1) == 2 ** 31 - 1
    assert L.tcbnn_inconv_residual_bound_of_input(None, 1, 8, 8, 3, 3, 1, 1, 1) == 2 ** 31 - 1


def test_host_abs_max_and_threaded_window_scan_on_a_large_batch():
    """tcbnn_host_abs_max against numpy (sizes below and above its threading threshold, NaN / infinity), and the
    window scan on a batch large enough for every host thread to take several images."""
    import numpy as np
    from tcbnn_amd import _lib
    L = _lib.lib
    rng = np.random.default_rng(12)
    for n in (1, 1000, (3 << 20) + 17):
        x = (rng.standard_normal(n) * 7).astype(np.float32)
        assert L.tcbnn_host_abs_max(x.ctypes.data, n) == float(np.abs(x).max())
        x[n // 2] = np.inf if n % 2 else np.nan
        assert L.tcbnn_host_abs_max(x.ctypes.data, n) == float("inf")
    assert L.tcbnn_host_abs_max(None, 5) == 0.0
    b, h, w = 70, 20, 24
    x = rng.standard_normal((b, 3, h, w)).astype(np.float32)
    x[41] *= 9.0  # the image that sets the bound sits in the middle of the batch
    a = np.abs(x.astype(np.float64)).sum(axis=1)
    worst = max(float(a[:, max(0, 4 * y - 3):4 * y + 4, max(0, 4 * q - 3):4 * q + 4].sum(axis=(1, 2)).max())
                for y in range(5) for q in range(6))
    got = L.tcbnn_inconv_residual_bound_of_input(x.ctypes.data, b, h, w, 7, 7, 4, 4, 1)
    assert worst <= got <= worst * 1.001 + 2, (got, worst)
