"""Work that users of this library have it do, as cases that can be timed and compared: whole networks of the layer
API with their inputs on the device, the serving call from a host array to logits, and the stand-alone bit matrix
product and bit convolution.  Sizes are those of the network drivers, the tests and the benchmark's sweep, plus
batches and shapes around them."""
import numpy as np
import torch

from tcbnn_amd import _lib, nets
from tcbnn_amd._lib import check, lib

# ops: "net" (forward pass, input resident), "serve" (set_input + forward + logits from host data), "bmm", "bconv".
# Largest batch that draw() takes for a network: ImageNet-sized nets up to twice their drivers' 256 where the pass
# stays cheaper than the largest listed case, CIFAR-sized ones up to 1024, the MLP up to twice its driver's 8192.
MAX_BATCH = {"imagenet_resnet": 512, "imagenet_resnet_textbook": 256, "cifar10_vgg": 1024, "cifar10_resnet": 1024,
             "mnist_mlp": 16384, "alexnet": 512, "imagenet_vgg": 192}


def listed():
    return [
        # offline classification at the drivers' configured batch: the headline benchmark
        dict(name="resnet18_b256", op="net", net="imagenet_resnet", batch=256),
        # the same network as an interactive service sees it: few images, launches and latency count
        dict(name="resnet18_b8", op="net", net="imagenet_resnet", batch=8),
        # the textbook wiring: 112x112 first layer, max-pool, 1x1 shortcut convolutions, average-pool head in fp32
        dict(name="resnet18_textbook_b256", op="net", net="imagenet_resnet_textbook", batch=256),
        # CIFAR classifier with pooled convolutions and three fully connected layers
        dict(name="vgg_small_b256", op="net", net="cifar10_vgg", batch=256),
        # residual network on small frames, with the odd batch that the tail of a data set leaves
        dict(name="cifar_resnet_b77", op="net", net="cifar10_resnet", batch=77),
        # fully connected layers alone, many rows
        dict(name="mlp_b8192", op="net", net="mnist_mlp", batch=8192),
        # 11x11 and 5x5 filters, pooled first layer, channel counts that are no powers of two, ragged batch
        dict(name="alexnet_b200", op="net", net="alexnet", batch=200),
        # the largest network of the drivers at its configured batch
        dict(name="vgg16_b256", op="net", net="imagenet_vgg", batch=256),
        # the stand-alone bit matrix product at the benchmark's smallest size ...
        dict(name="bmm_1024", op="bmm", m=1024, n=1024, k=1024),
        # ... and a large one whose sizes are multiples of 32 and of nothing larger
        dict(name="bmm_ragged", op="bmm", m=5000, n=3104, k=7200),
        # the stand-alone bit convolution, the largest output of the benchmark's sweep
        dict(name="bconv_56_c64_b256", op="bconv", batch=256, hw=56, cin=64, cout=64, r=3, stride=1),
        # a service's request: a batch of host images in, their logits on the host out
        dict(name="serve_resnet18_b64", op="serve", net="imagenet_resnet", batch=64),
    ]


def _log_int(rng, lo, hi):
    """An integer of lo..hi, evenly spread over its logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choice(["net"] * 5 + ["serve", "bmm", "bmm", "bconv", "bconv"])
    if op == "net":
        net = rng.choice(sorted(MAX_BATCH))
        return dict(op=op, net=net, batch=_log_int(rng, 1, MAX_BATCH[net]))
    if op == "serve":
        net = rng.choice(["imagenet_resnet", "cifar10_vgg", "mnist_mlp"])
        return dict(op=op, net=net, batch=_log_int(rng, 1, 128 if net == "imagenet_resnet" else 1024))
    if op == "bmm":
        return dict(op=op, m=_log_int(rng, 32, 8192), n=32 * _log_int(rng, 1, 256), k=32 * _log_int(rng, 2, 256))
    while True:
        c = dict(op=op, batch=_log_int(rng, 1, 256), hw=_log_int(rng, 7, 64),
                 cin=rng.choice([32, 64, 96, 128, 192, 256, 384, 512]),
                 cout=rng.choice([32, 64, 96, 128, 192, 256, 384, 512]), r=rng.choice([3, 3, 3, 1, 5]),
                 stride=rng.choice([1, 1, 2]))
        w = work(c)
        if w["flops"] <= 1e12 and w["bytes"] <= 8e8:
            return c


def _spec(case):
    return nets.SPECS[case["net"]](batch=case["batch"])


class _Weights:
    """Weight source of a network: one seeded array after the other, in the order the layers ask for them: +-1
    weights, thresholds N(0, sqrt(fan_in)), output scale N(1, 0.1) and bias N(0, 1), fp32 head N(0, 1/sqrt(C))."""

    def __init__(self, spec, gen):
        self._parts = []

        def normal(n, mean, std):
            self._parts.append(torch.randn(n, generator=gen, device="cuda").mul_(std).add_(mean))

        def signs(n):
            self._parts.append(torch.randint(0, 2, (n,), generator=gen, device="cuda", dtype=torch.int8).mul_(2).sub_(1))

        for L in spec:
            if L["kind"] in ("in", "pool"):
                continue
            if L["kind"] == "avgfc":
                normal(L["channels"] * L["out"], 0.0, L["channels"] ** -0.5)
                normal(L["out"], 0.0, 1.0)
                continue
            if L["kind"] in ("fc", "out"):
                fan_in, n_out = L["inp"], L["out"]
            else:
                fan_in, n_out = L["r"] * L["s"] * L["cin"], L["cout"]
            signs(fan_in * n_out)
            if L["kind"] == "out":
                normal(n_out, 1.0, 0.1)
                normal(n_out, 0.0, 1.0)
            else:
                normal(n_out, 0.0, fan_in ** 0.5)

    def launch_array(self, size):
        part = self._parts.pop(0)
        assert part.numel() == size, (part.numel(), size)
        return part.cpu().numpy()


class _DeviceView:
    """A device buffer of the library for torch.as_tensor; the tensor keeps the buffer's owner alive."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr="<f4", version=2, strides=None)


def _images(spec, gen):
    """A batch as the drivers' readers hand it over: fp32 on the host, normalised (ImageNet, CIFAR) or centred (MNIST)."""
    L = spec[0]
    if L["kind"] == "in":
        x = torch.rand((L["batch"], L["features"]), generator=gen, device="cuda").sub_(0.5)
    else:
        x = torch.randn((L["batch"], L["cin"], L["h"], L["w"]), generator=gen, device="cuda")
    return np.ascontiguousarray(x.cpu().numpy())


def _signs(shape, gen):
    return torch.randint(0, 2, shape, generator=gen, device="cuda", dtype=torch.int8).float().mul_(2).sub_(1)


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    op = case["op"]
    if op in ("net", "serve"):
        spec = _spec(case)
        x = _images(spec, gen)
        net = nets.Network(spec, _Weights(spec, gen), x)
        if op == "serve":
            return dict(op=op, net=net, images=x)
        out = net.order[-1].get_output_gpu()
        view = torch.as_tensor(_DeviceView(net, out.ptr, (case["batch"], spec[-1]["out"])), device="cuda")
        return dict(op=op, net=net, logits=view)
    if op == "bmm":
        m, n, k = case["m"], case["n"], case["k"]
        a = torch.empty(m * k // 32, dtype=torch.int32, device="cuda")
        b = torch.empty(n * k // 32, dtype=torch.int32, device="cuda")
        fa, fb = _signs((m, k), gen), _signs((k, n), gen)
        check(lib.tcbnn_pack_rows(fa.data_ptr(), a.data_ptr(), m, k, k, k // 32, None))
        check(lib.tcbnn_pack_cols(fb.data_ptr(), b.data_ptr(), k, n, k // 32, None))
        c = torch.empty((m, n), dtype=torch.int32, device="cuda")
        return dict(op=op, m=m, n=n, k=k, a=a, b=b, c=c)
    batch, hw, cin, cout, r, stride = (case[v] for v in ("batch", "hw", "cin", "cout", "r", "stride"))
    o = _bconv_out(case)
    x = torch.empty(lib.tcbnn_conv_act_words(hw, hw, batch, cin), dtype=torch.int32, device="cuda")
    f = torch.empty(lib.tcbnn_conv_filter_words(r, r, cin, cout), dtype=torch.int32, device="cuda")
    fx, ff = _signs((batch, hw, hw, cin), gen), _signs((r, r, cin, cout), gen)
    check(lib.tcbnn_pack_conv_input_nhwc(fx.data_ptr(), x.data_ptr(), batch, hw, hw, cin, None))
    check(lib.tcbnn_pack_conv_filter(ff.data_ptr(), f.data_ptr(), r, r, cin, cout, None))
    y = torch.empty((batch, o, o, cout), dtype=torch.int32, device="cuda")
    return dict(op=op, x=x, f=f, y=y, args=(batch, hw, hw, cin, cout, r, r, stride, stride, r // 2, r // 2, o, o))


def run(state):
    op = state["op"]
    if op == "net":
        state["net"].forward()
        return state["logits"]
    if op == "serve":
        net = state["net"]
        net.set_input(state["images"])
        net.forward()
        return net.logits()
    if op == "bmm":
        check(lib.tcbnn_bmm(state["a"].data_ptr(), state["b"].data_ptr(), state["c"].data_ptr(), state["m"], state["n"],
                            state["k"], _lib.VARIANT_AUTO, None))
        return state["c"]
    check(lib.tcbnn_bconv(state["x"].data_ptr(), state["f"].data_ptr(), state["y"].data_ptr(), *state["args"],
                          _lib.VARIANT_AUTO, None))
    return state["y"]


def _bconv_out(case):
    return (case["hw"] + 2 * (case["r"] // 2) - case["r"]) // case["stride"] + 1


def work(case):
    """Inputs, packed weights (one bit each) and outputs once; 2 operations per multiply-accumulate."""
    op = case["op"]
    if op in ("net", "serve"):
        spec = _spec(case)
        first = spec[0]
        x = first["batch"] * (first["features"] if first["kind"] == "in" else first["cin"] * first["h"] * first["w"])
        bits = floats = head = 0
        for L in spec:
            if L["kind"] in ("fc", "out"):
                bits += L["inp"] * L["out"]
                floats += L["out"] * (2 if L["kind"] == "out" else 1)
            elif L["kind"] in ("conv", "inconv"):
                bits += L["r"] * L["s"] * L["cin"] * L["cout"]
                floats += L["cout"]
            elif L["kind"] == "avgfc":
                floats += (L["channels"] + 1) * L["out"]
                head = 2 * L["batch"] * L["channels"] * L["out"]
        y = case["batch"] * spec[-1]["out"]
        return {"bytes": 4 * (x + floats + y) + bits // 8, "flops": sum(nets.binary_ops(spec)) + head}
    if op == "bmm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m + n) * k // 8 + 4 * m * n, "flops": 2 * m * n * k}
    batch, hw, cin, cout, r = (case[v] for v in ("batch", "hw", "cin", "cout", "r"))
    outputs = batch * _bconv_out(case) ** 2 * cout
    return {"bytes": (batch * hw * hw * cin + r * r * cin * cout) // 8 + 4 * outputs, "flops": 2 * outputs * r * r * cin}


def tolerance(case):
    """Sums of +-1 products are whole numbers; logits are whole numbers scaled and shifted in fp32, or an fp32 product."""
    return "exact" if case["op"] in ("bmm", "bconv") else {"rel": 1e-5}
