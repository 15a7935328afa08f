"""The C++ host layer (hdkx-aicompiler_amd/host): the reference's graph / compile / run interface with the
target switched.  The test program is built by `make -C hdkx-aicompiler_amd/host` (build() does it)."""
import json
import os
import subprocess
import tempfile

import numpy as np
import pytest

from oracle_lib import Oracle

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "hdkx-aicompiler_amd", "host")
BIN = os.path.join(HOST, "build", "host_tests")


def _ensure_built():
    if not os.path.exists(BIN):
        subprocess.check_call(["make", "-C", HOST, "-j8"])


def run(*args, timeout=600, env=None):
    _ensure_built()
    r = subprocess.run([BIN] + list(args), capture_output=True, text=True, timeout=timeout,
                       env=dict(os.environ, **env) if env else None)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    return r.stdout


def _write_resnet_inputs(synth, d, config, batch, hw):
    consts = synth.resnet18_consts(config)
    x = synth.resnet18_input(config, batch, hw)
    x.tofile(os.path.join(d, "input.bin"))
    for k, c in enumerate(consts):
        c.tofile(os.path.join(d, "const_%d.bin" % k))
    return x, consts


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


# ------------------------------------------------------------------ CPU (host C back end)
def test_op_numeric_known_answers_cpu():
    out = run("op_numeric", "cpu")
    assert "All operator numeric tests passed (cpu)" in out
    assert out.count("[PASS]") == 23          # 19 operators (softmax and cast included), 3 small models, the error cases


def test_device_info_contract():
    assert "device info ok" in run("device_info")


def test_packed_function_registry_cpu():
    """Registry::Global().Get / Set, KXC_REGISTER_GLOBAL, Args / RetValue conversions and the device_api.* functions on
    the host back end (include/base/registry.h:13-61, src/base/device_api.cc:442-658)."""
    assert "packed functions ok (cpu)" in run("packed_func", "cpu")


def _oracle_so():
    from oracle_lib import _build_if_missing
    return _build_if_missing("libkxc_oracle.so")


def test_split_batch_accepts_only_separable_graphs():
    """relay::SplitBatch (the shares of a batch the hip back end runs side by side): ResNet-18 splits, constants are
    shared; softmax / reduce_mean / transpose / flatten over the batch axis, reshape, a batched right-hand operand, an
    unbatched operand of batch extent and a batch that does not divide are refused; an explicit hip_batch_lanes on
    such a graph makes Compile throw."""
    out = run("split_batch")
    assert "split batch ok" in out and out.count("[PASS]") == 4


def test_quantised_operators_cpu():
    """qnn_quantize / qnn_conv2d / qnn_dense as graph operators (type rule, TE compute with the rint intrinsic, host
    back end): hand-worked answers, and the C oracle on seeded cases, element for element."""
    out = run("qnn", "cpu", _oracle_so())
    assert "quantised operators ok (cpu)" in out and out.count("[PASS]") == 16


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["hip", "hipgen"])
def test_quantised_operators_gpu(mode):
    """The same cases through the hand-written int8 launches (hip) and through kernels generated from the operators'
    TE compute (hipgen)."""
    out = run("qnn", mode, _oracle_so())
    assert "quantised operators ok (%s)" % mode in out and out.count("[PASS]") == 16


@pytest.mark.gpu
def test_shares_of_a_batch_with_generated_kernels():
    """conv -> relu -> global average pool -> flatten -> softmax at batch 8 in 1, 2 and 4 shares: the hand-written
    launches and the generated softmax kernels of every share give the one-share result bit for bit, and the saved
    plan rebuilds."""
    out = run("shares_generated")
    assert "shares with generated kernels ok" in out and out.count("[PASS]") == 3


@pytest.mark.gpu
def test_random_graphs_in_one_and_two_shares():
    """Eight seeded random convolutional graphs (plain / strided convolutions, pools, residual blocks with and without a
    downsample branch, dense head, softmax) at batch 4 and 8: hip back end in one share within the operator tolerance
    of the host back end, two shares within 1e-4 of one share, run twice over the same workspace."""
    out = run("shares_random")
    assert "random graphs in shares ok" in out and out.count("[PASS]") == 8


@pytest.mark.gpu
def test_generated_kernels_lds_schedules_bit_exact():
    """dense / matmul / reduce_mean shapes that take the generator's LDS-staged schedules (ragged chunks, fewer outputs
    than a workgroup, an operand that is not contiguous along the reduce axis, a padded window whose input load stays
    behind its select), and convolution-shaped nests in the register-tiled schedule (ragged blocks, stride and dilation,
    a 5x5 window, 1x1, the default block choice at a large and at a small shape): bit-identical to the host back end."""
    out = run("generated_numeric")
    assert "generated kernels ok" in out and out.count("[PASS]") == 12
    assert out.count("(reg_tile)") == 5


@pytest.mark.gpu
def test_non_finite_inputs_with_and_without_winograd():
    """The stated difference of the default path: with CompileConfig::hip_winograd = false an Inf / NaN input spreads
    exactly as in the CPU back end (nine outputs per channel, Inf stays Inf); with Winograd it reaches at most the
    sixteen outputs of the patches that hold it, where an Inf may come out as NaN; everything else is unaffected."""
    assert "non-finite ok" in run("nonfinite")


@pytest.mark.gpu
def test_packed_function_registry_hip():
    """The same registry on the GPU: allocation, copies with offsets on a stream, attributes, target.Build,
    device_info.hip.0.*, and a Relay function lowered to plan JSON and run from that JSON."""
    assert "packed functions ok (hip)" in run("packed_func", "hip")


def test_compiled_kernel_object_and_compile_config_surface_cpu():
    """codegen::CompiledKernel (fields, IsReady, call operator, error text), CompileConfig::profile_options / cache_dir
    and CompiledModule::GetProfileBundlePath on the host back end."""
    with tempfile.TemporaryDirectory() as d:
        assert "kernel object ok (cpu)" in run("kernel_object", "cpu", d)


@pytest.mark.gpu
def test_compiled_kernel_object_hip():
    """The same object owning a launch plan: ready exactly while the plan can run, "Kernel <name> returned error code
    N" when a launch is refused, resources alive as long as any handle."""
    with tempfile.TemporaryDirectory() as d:
        assert "kernel object ok (hip)" in run("kernel_object", "hip", d)
    assert "kernel object ok (hipgen)" in run("kernel_object", "hipgen")


def test_lowering_and_code_generators():
    assert "codegen ok" in run("codegen")


def test_resnet18_cpu_backend_equals_oracle_bit_for_bit(synth):
    """Relay graph -> TE -> TIR -> generated C on the host reproduces the pinned CPU oracle exactly: the
    lowering keeps the reference's loop and rounding order."""
    with tempfile.TemporaryDirectory() as d:
        x, consts = _write_resnet_inputs(synth, d, 3, 1, 64)
        out = run("resnet18", "cpu", d, "1", "64")
        assert "launches: 1" in out
        got = np.fromfile(os.path.join(d, "logits.bin"), np.float32).reshape(1, 1000)
    want = Oracle(fast=True).resnet18(x, consts)
    assert np.array_equal(bits(got), bits(want))


def test_resnet18_hip_plan_without_gpu():
    """Compiling for the hip target needs no GPU up to loading: 49 Relay calls become 20 launches (each block's
    downsample is the second output of the block's first convolution, at small batches with the reductions of both
    outputs split over workgroups; KXC_HIP_PAIR_SPLIT=0 gives such a downsample a launch of its own: 23).  By
    default a batch of 64 runs as
    two shares of 32 side by side, each those 20 launches; KXC_HIP_BATCH_LANES=1 keeps the batch whole."""
    with tempfile.TemporaryDirectory() as d:
        out = run("resnet18", "hip", d, "64", "224")
        shares = json.load(open(os.path.join(d, "plan.json")))
    assert "launches: 40" in out and len(shares["nodes"]) == 40
    # the two shares' launches alternate
    assert [n["kernel_symbol"] + " @share1" for n in shares["nodes"][0::2]] == [n["kernel_symbol"] for n in shares["nodes"][1::2]]
    assert [n["output_values"] for n in shares["nodes"][0::2]] == [n["output_values"] for n in shares["nodes"][1::2]]
    with tempfile.TemporaryDirectory() as d:
        out = run("resnet18", "hip", d, "64", "224", env={"KXC_HIP_BATCH_LANES": "1"})
        plan = json.load(open(os.path.join(d, "plan.json")))
    assert [n["kernel_symbol"] for n in plan["nodes"]] == [n["kernel_symbol"] for n in shares["nodes"][0::2]]
    assert "launches: 20" in out
    assert len(plan["nodes"]) == 20 and plan["schema_version"] == 1
    syms = [n["kernel_symbol"] for n in plan["nodes"]]
    assert sum("+add+relu" in s for s in syms) == 8          # residual tails folded into convolutions
    assert sum(s.startswith("kxc_conv2d") and s.endswith("+bias+relu") for s in syms) == 5
    # the first convolution takes the column maxima of the 3x3/2 max pool behind it; a 3x1 pool finishes the window
    assert syms[0].endswith("+bias+relu+maxpool3w") and syms[1] == "kxc_max_pool2d_f32"
    assert [n["op_name"] for n in plan["nodes"][:2]] == ["nn_conv2d", "nn_max_pool2d"]
    assert plan["nodes"][0]["output_values"] == plan["nodes"][1]["input_values"] == plan["nodes"][1]["output_values"]
    with tempfile.TemporaryDirectory() as d:
        run("resnet18", "hip", d, "64", "224", env={"KXC_HIP_FUSE_POOL": "0", "KXC_HIP_BATCH_LANES": "1"})
        unfused = json.load(open(os.path.join(d, "plan.json")))
    assert len(unfused["nodes"]) == 20 and unfused["nodes"][0]["kernel_symbol"].endswith("+bias+relu")
    assert unfused["nodes"][0]["output_values"] != unfused["nodes"][1]["output_values"]
    # each block's 1x1 downsample is the second output of the block's first 3x3/2 convolution
    pairs = [n for n in plan["nodes"] if n["kernel_symbol"].endswith("_ds+bias+relu|conv1x1+bias")]
    assert len(pairs) == 3 and all(len(n["output_values"]) == 2 and len(n["input_values"]) == 5 for n in pairs)
    assert len(plan["constant_value_ids"]) == 42 and len(plan["input_value_ids"]) == 1
    assert all(n["kind"] == "kernel" and n["worker_set"] == [0] for n in plan["nodes"])
    # at batch 64 every 3x3 stride-1 convolution (constant weights) takes the Winograd kernel, the rest do not
    assert sum(".winograd_f2k3" in s for s in syms) == 13 and sum(".mfma_" in s for s in syms) == 4
    with tempfile.TemporaryDirectory() as d:
        run("resnet18", "hip", d, "64", "224", env={"KXC_HIP_PAIR": "0", "KXC_HIP_BATCH_LANES": "1"})
        unpaired = json.load(open(os.path.join(d, "plan.json")))
    assert len(unpaired["nodes"]) == 23
    assert sum(n["kernel_symbol"].startswith("kxc_conv2d") and n["kernel_symbol"].endswith("+bias") for n in unpaired["nodes"]) == 3
    with tempfile.TemporaryDirectory() as d:
        run("resnet18", "hip", d, "64", "224", env={"KXC_HIP_WINOGRAD": "0", "KXC_HIP_BATCH_LANES": "1"})
        off = json.load(open(os.path.join(d, "plan.json")))
    assert not any("winograd" in n["kernel_symbol"] for n in off["nodes"])
    with tempfile.TemporaryDirectory() as d:
        run("resnet18", "hip", d, "1", "224")
        one = json.load(open(os.path.join(d, "plan.json")))
    # batch 1: the same thirteen layers (which of them run without the transform is settled when the plan is finalized); too
    # few tiles for the first layer's pooling epilogue to pay
    assert sum("winograd" in n["kernel_symbol"] for n in one["nodes"]) == 13
    assert not any("maxpool3w" in n["kernel_symbol"] for n in one["nodes"])
    with tempfile.TemporaryDirectory() as d:
        run("resnet18", "hip", d, "1", "224", env={"KXC_HIP_WINOGRAD_MIN_WORK": "512"})
        few = json.load(open(os.path.join(d, "plan.json")))
    # with the work threshold only the 56x56 layers have enough 2x2 blocks per input channel
    assert sum("winograd" in n["kernel_symbol"] for n in few["nodes"]) == 4


def test_quantised_resnet18_hip_plan_without_gpu():
    """The quantised ResNet-18 graph (qnn_quantize, qnn_conv2d, int8 max pool, qnn_global_avg_pool2d, qnn_dense)
    compiled for the hip target: the operators' layout hooks put every activation between the first convolution and
    the average pool into the channel-blocked layout of the int8 matrix cores, the input into the 4-channel layout,
    pair each downsample with its block's first convolution, and fold the max pool into the first convolution's
    kernel -- 24 calls, 20 launches, no converter (KXC_HIP_FUSE_POOL=0: 21, the pool a launch of its own).  With
    KXC_HIP_QNN_MFMA=0 every operator keeps NCHW and its reference-order kernel."""
    import importlib
    ha = importlib.import_module("hdkx-aicompiler_amd.hostapi")
    qr = importlib.import_module("hdkx-aicompiler_amd.qresnet18")
    layers = [{"name": n, "res_mult": 0.37 if n.endswith(".conv2") else 0.0} for (n, *_rest) in qr.layer_table()]
    model = {"layers": layers, "scale": {"last": 0.02}, "input_scale": 0.02, "gap_scale_out": 0.01, "last": "last"}
    mod = ha.CompiledQResNet18(model, 64, 224)
    sym = mod.launches()
    plan = json.loads(mod.plan_json())
    assert len(sym) == 20 and len(plan["nodes"]) == 20 and len(plan["constant_value_ids"]) == 63 and mod.num_args == 65
    assert sym[0] == "qnn_quantize kxc_quantize_f32_nchw_to_c4_i8"
    assert sym[1] == "qnn_conv2d kxc_qconv2d_c4_i8:qmfma_k7x7s2_c4+relu+maxpool3x3s2"
    # (the fused node produces the pooling call's value)
    assert plan["nodes"][1]["output_values"] != plan["nodes"][0]["output_values"] and plan["nodes"][2]["input_values"][0] == plan["nodes"][1]["output_values"][0]
    os.environ["KXC_HIP_FUSE_POOL"] = "0"
    try:
        unfused = ha.CompiledQResNet18(model, 64, 224)
        usym = unfused.launches()
        unfused.close()
    finally:
        del os.environ["KXC_HIP_FUSE_POOL"]
    assert len(usym) == 21 and usym[1] == "qnn_conv2d kxc_qconv2d_c4_i8:qmfma_k7x7s2_c4+relu" and usym[2] == "nn_max_pool2d kxc_max_pool2d_c16_i8"
    assert usym[3:] == sym[2:]
    sym = [sym[0], sym[1], "(pool)"] + sym[2:]                  # numbered as in the unfused plan below
    assert all(s.startswith(("qnn_conv2d kxc_qconv2d_c16_i8:qmfma", "qnn_conv2d kxc_qconv2d_c16_i8:qrows")) for s in sym[3:19])
    # the four 56 x 56 stride-1 layers take the kernel with the 64-position row pitch
    assert [":qrows_k3x3" in s for s in sym[3:19]] == [True] * 4 + [False] * 12
    assert sum(s.endswith("+relu|qconv1x1+bias") for s in sym) == 3 and sum(s.endswith("+add+relu") for s in sym) == 8
    pairs = [n for n in plan["nodes"] if "|qconv1x1" in n["kernel_symbol"]]
    assert all(len(n["output_values"]) == 2 and len(n["input_values"]) == 7 for n in pairs)
    assert sym[19:] == ["qnn_global_avg_pool2d kxc_global_avg_pool2d_c16_i8", "qnn_dense kxc_qdense_i8"]
    assert mod.constant_names[:3] == ["conv1.w", "conv1.b", "conv1.m"] and mod.constant_names[-3:] == ["fc.w", "fc.b", "fc.m"]
    # constants in depth-first argument order: a block's second convolution before its downsample
    k = mod.constant_names.index("l2.0.conv2.w")
    assert mod.constant_names[k - 3] == "l2.0.conv1.w" and mod.constant_names[k + 3] == "l2.0.down.w"
    mod.close()
    # a batch of 128 runs as two shares side by side; a graph cut at a convolution converts its result back to NCHW
    two = ha.CompiledQResNet18(model, 128, 224)
    assert len(two.launches()) == 40 and two.launches()[1].endswith(" @share1")
    two.close()
    cut = ha.CompiledQResNet18(model, 2, 64, result="l2.0.down")
    assert cut.launches()[-1] == "layout_convert kxc_i8_c16_to_nchw" and "qmfma_k1x1" in cut.launches()[-2]
    assert cut.constant_names[-1] == "l2.0.down.m" and "l2.0.conv1.w" not in cut.constant_names
    cut.close()
    os.environ["KXC_HIP_QNN_MFMA"] = "0"
    try:
        plain = ha.CompiledQResNet18(model, 2, 64)
        names = [s.split(" ", 1)[1] for s in plain.launches()]
        assert len(names) == 24 and names.count("kxc_qconv2d_nchw_i8") == 20 and names[0] == "kxc_quantize_f32_i8"
        assert "kxc_max_pool2d_i8" in names and "kxc_global_avg_pool2d_i8" in names
        plain.close()
    finally:
        del os.environ["KXC_HIP_QNN_MFMA"]


# ------------------------------------------------------------------ GPU
@pytest.mark.gpu
def test_op_numeric_known_answers_hip():
    assert "All operator numeric tests passed (hip)" in run("op_numeric", "hip")


@pytest.mark.gpu
def test_op_numeric_known_answers_generated_kernels():
    assert "All operator numeric tests passed (hipgen)" in run("op_numeric", "hipgen")


@pytest.mark.gpu
def test_resnet18_hip_matches_oracle(synth):
    from gpu_util import assert_close
    with tempfile.TemporaryDirectory() as d:
        x, consts = _write_resnet_inputs(synth, d, 3, 2, 224)
        out = run("resnet18", "hip", d, "2", "224")
        assert "execution plan replayed: 20 launches, identical output" in out
        assert "launches: 20" in out
        got = np.fromfile(os.path.join(d, "logits.bin"), np.float32).reshape(2, 1000)
        plan = json.load(open(os.path.join(d, "plan.json")))
        assert sum(n["kernel_symbol"].endswith("_ds+bias+relu|conv1x1+bias") for n in plan["nodes"]) == 3
    want = Oracle(fast=True).resnet18(x, consts)
    assert_close(got, want, what="C++ host layer, ResNet-18 logits", floor="scale")
    # a downsample of a launch that splits its reduction over workgroups as a launch of its own
    with tempfile.TemporaryDirectory() as d:
        _write_resnet_inputs(synth, d, 3, 2, 224)
        out = run("resnet18", "hip", d, "2", "224", env={"KXC_HIP_PAIR_SPLIT": "0"})
        assert "execution plan replayed: 23 launches, identical output" in out
        apart = np.fromfile(os.path.join(d, "logits.bin"), np.float32).reshape(2, 1000)
    assert_close(apart, want, what="C++ host layer, ResNet-18 logits, downsamples apart", floor="scale")


@pytest.mark.gpu
def test_resnet18_hip_winograd_matches_oracle(synth):
    """The same network with every 3x3 stride-1 convolution on the Winograd kernel and every downsample on the
    side lane (both forced at this small batch): logits within the fp32 tolerance, and the saved plan replays to
    the identical output."""
    from gpu_util import assert_close
    with tempfile.TemporaryDirectory() as d:
        x, consts = _write_resnet_inputs(synth, d, 3, 2, 224)
        out = run("resnet18", "hip", d, "2", "224", env={"KXC_HIP_WINOGRAD_MIN_WORK": "0", "KXC_HIP_CONCURRENT_MIN_ELEMS": "0", "KXC_HIP_PAIR_SPLIT": "0"})
        assert "execution plan replayed: 23 launches, identical output" in out
        plan = json.load(open(os.path.join(d, "plan.json")))
        assert sum(".winograd_f2k3" in n["kernel_symbol"] for n in plan["nodes"]) == 13
        got = np.fromfile(os.path.join(d, "logits.bin"), np.float32).reshape(2, 1000)
    want = Oracle(fast=True).resnet18(x, consts)
    assert_close(got, want, what="C++ host layer, ResNet-18 logits (Winograd)", floor="scale")


def _lanes(plan_json):
    """(lane, join, chain) of every node of the serialised launch plan (the three fields before the parameter count)."""
    text = json.loads(plan_json)["kxc_hip"]["launch_plan"]
    lines = [line.split() for line in text.splitlines() if line.startswith("node")]
    base = min(len(t) for t in lines)            # a node without parameters; each parameter adds two fields
    out = []
    for t in lines:
        assert (len(t) - base) % 2 == 0 and int(t[base - 1]) == (len(t) - base) // 2
        out.append((int(t[base - 4]), int(t[base - 3]), int(t[base - 2])))
    return out


def _compiled_resnet18_logits(synth, config, batch, module=None, env=None):
    """The plan bench.py times: ResNet-18 compiled by the C++ host layer with its DEFAULT configuration, run once
    eagerly and then replayed as a captured HIP graph; returns inputs, logits of both, and the module facts.
    env: switches the compiler reads from the environment, set for the compilation only."""
    import importlib
    import torch
    saved = {k: os.environ.get(k) for k in (env or {})}
    os.environ.update(env or {})
    try:
        return _compiled_resnet18_logits_now(synth, config, batch, importlib, torch)
    finally:
        for k, v in saved.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v


def _compiled_resnet18_logits_now(synth, config, batch, importlib, torch):
    hostapi = importlib.import_module("hdkx-aicompiler_amd.hostapi")
    consts_h = synth.resnet18_consts(config)
    x_h = synth.resnet18_input(config, batch)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    tensors = [dev(x_h)] + [dev(c) for c in consts_h]
    out = torch.zeros((batch, 1000), device="cuda")
    module = hostapi.CompiledResNet18(batch, 224, "hip", sync_after_run=False)
    try:
        packed = module.packed(tensors + [out])
        facts = {"launches": module.launches(), "lanes": _lanes(module.plan_json()), "workspace": module.workspace_bytes()}
        module.run_packed(packed, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        eager = out.cpu().numpy().copy()
        # second and third pass over the same workspace (liveness reuse, persistent transformed weights), as a graph
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            module.enable_graph_replay(True)
            for _ in range(3):
                out.zero_()
                module.run_packed(packed, stream.cuda_stream)
                stream.synchronize()
        replay = out.cpu().numpy().copy()
    finally:
        module.close()
    return x_h, consts_h, eager, replay, facts


@pytest.mark.gpu
def test_resnet18_benchmarked_plan_batch64_matches_oracle(synth):
    """Benchmark configuration 4 through the very plan the benchmark times (host layer, default configuration:
    thirteen Winograd launches, downsamples folded into the stride-2 convolutions): images 0 and 63 against the
    CPU path on those images, within the operator tolerance (the reference's acceptance metric,
    test/onnx_importer_test.cpp:146-179)."""
    from gpu_util import assert_close, assert_bit_exact
    x, consts, eager, replay, facts = _compiled_resnet18_logits(synth, 4, 64)
    syms = facts["launches"]
    # two shares of 32 images, each the whole network in 20 launches with the variants of the batch-64 launches
    assert len(syms) == 40 and sum(".winograd_f2k3" in s for s in syms) == 26 and sum("_ds+" in s for s in syms) == 6, syms
    assert [s + " @share1" for s in syms[0::2]] == syms[1::2]       # the shares' launches alternate in the plan
    assert facts["lanes"] == [(0, 0, 0), (0, 0, 1)] * 20              # the second share is a chain on a stream of its own
    assert_bit_exact(replay, eager, "graph replay of the batch-64 plan")
    # the whole batch in one share (20 launches, one stream): the same kernels; the 256-channel Winograd layers split
    # their reduction over two workgroups in the two-share plan only, so the logits agree to rounding, not bit for bit
    _, _, whole, whole_replay, whole_facts = _compiled_resnet18_logits(synth, 4, 64, env={"KXC_HIP_BATCH_LANES": "1"})
    assert whole_facts["launches"] == syms[0::2] and set(whole_facts["lanes"]) == {(0, 0, 0)}
    assert_close(eager, whole, what="two shares of the batch against the batch in one share", floor="scale")
    assert float(np.max(np.abs(eager - whole))) <= 1e-4 * float(np.max(np.abs(whole)))
    assert_bit_exact(whole_replay, whole, "graph replay of the one-share plan")
    # the first layer's pooling epilogue: the same logits bit for bit as convolution + 3x3 pool (the maximum is exact
    # and the 64 x 448 and 64 x 256 tiles add a pixel's products in the same order)
    assert syms[0].endswith("+bias+relu+maxpool3w")
    _, _, unfused, _, unfused_facts = _compiled_resnet18_logits(synth, 4, 64, env={"KXC_HIP_FUSE_POOL": "0"})
    assert not any("maxpool3w" in s for s in unfused_facts["launches"])
    assert_bit_exact(unfused, eager, "with and without the pooling epilogue")
    orc = Oracle(fast=True)
    for n in (0, 63):
        want = orc.resnet18(x[n:n + 1], consts)
        assert_close(eager[n:n + 1], want, what="host-layer plan, batch 64, image %d" % n, floor="scale")
        assert int(np.argmax(eager[n])) == int(np.argmax(want[0]))


@pytest.mark.gpu
def test_resnet18_two_shares_replay_from_saved_plan(synth):
    """Four images as two shares of two (forced at this size): the saved execution plan -- 2 x 20 launches, the
    second share's as a chain on argument offsets -- rebuilds into a module that reproduces the compiled one bit for
    bit.  Against one share of four the logits agree within the operator tolerance (at this size the reductions of
    the small launches are split over different numbers of workgroups; at batch 64 the two plans differ only in
    the split of the 256-channel layers and agree to rounding, see the batch-64 test)."""
    from gpu_util import assert_close
    logits = {}
    for lanes in ("1", "2"):
        with tempfile.TemporaryDirectory() as d:
            _write_resnet_inputs(synth, d, 3, 4, 224)
            out = run("resnet18", "hip", d, "4", "224", env={"KXC_HIP_BATCH_LANES": lanes})
            n = 20 * int(lanes)
            assert "execution plan replayed: %d launches, identical output" % n in out, out[-2000:]
            plan = json.load(open(os.path.join(d, "plan.json")))
            assert len(plan["nodes"]) == n
            logits[lanes] = np.fromfile(os.path.join(d, "logits.bin"), np.float32).reshape(4, 1000)
    assert_close(logits["2"], logits["1"], what="two shares of two images against one share of four", floor="scale")
    want = Oracle(fast=True).resnet18(synth.resnet18_input(3, 4, 224), synth.resnet18_consts(3))
    assert_close(logits["2"], want, what="two shares of two images against the CPU path", floor="scale")


@pytest.mark.gpu
def test_resnet18_benchmarked_plan_batch1_matches_oracle(synth):
    """Benchmark configuration 3 through the plan the benchmark times at batch 1: thirteen layers that the operators asked
    Winograd for, which at this size run on the kernel for small launches like the blocks' first convolutions."""
    from gpu_util import assert_close, assert_bit_exact
    x, consts, eager, replay, facts = _compiled_resnet18_logits(synth, 3, 1)
    assert sum(".winograd_f2k3" in s for s in facts["launches"]) == 13, facts["launches"]
    assert_bit_exact(replay, eager, "graph replay of the batch-1 plan")
    want = Oracle(fast=True).resnet18(x, consts)
    assert_close(eager, want, what="host-layer plan, batch 1", floor="scale")
    assert int(np.argmax(eager)) == int(np.argmax(want))


@pytest.mark.gpu
def test_resnet18_generated_kernels_equal_oracle_bit_for_bit(synth):
    """Every operator through the TIR -> HIP generator (no hand-written kernel): the generated kernels keep
    the CPU loop order and are compiled without contraction, so the logits are bit-identical."""
    with tempfile.TemporaryDirectory() as d:
        x, consts = _write_resnet_inputs(synth, d, 3, 1, 64)
        out = run("resnet18", "hipgen", d, "1", "64")
        assert "execution plan replayed:" in out and "identical output" in out      # generated kernels recompiled from the saved source
        assert "lds_row_reduce" in out          # global average pool: whole rows staged through LDS
        assert "lds_k_stage" in out             # the FC layer: rows of the weight staged a chunk of k at a time
        got = np.fromfile(os.path.join(d, "logits.bin"), np.float32).reshape(1, 1000)
    want = Oracle(fast=True).resnet18(x, consts)
    assert np.array_equal(bits(got), bits(want))


# ------------------------------------------------------------------ profiling bundle
EVENT_KEYS = ("trace_id", "session_id", "run_id", "span_id", "parent_span_id", "component", "event_type", "phase",
              "ts_ns", "duration_ns", "status", "severity", "device", "worker_id", "op_name", "pass_name",
              "kernel_symbol", "shape_signature", "message", "fields", "metrics")


def _read_bundle(d):
    for name in ("manifest.json", "events.jsonl", "trace.json", "summary.json", "diagnosis.json", "diagnosis.md"):
        assert os.path.exists(os.path.join(d, name)), name
    events = [json.loads(line) for line in open(os.path.join(d, "events.jsonl")) if line.strip()]
    manifest = json.load(open(os.path.join(d, "manifest.json")))
    trace = json.load(open(os.path.join(d, "trace.json")))
    summary = json.load(open(os.path.join(d, "summary.json")))
    assert manifest["schema_version"] == 1 and manifest["event_count"] == len(events) == summary["event_count"]
    assert len(trace["traceEvents"]) == len(events)
    for e in events:
        # the stable event fields of the reference's bundle (src/base/profiling.cc:740-771)
        assert tuple(e.keys()) == EVENT_KEYS
        assert e["fields"]["schema_version"] == "1" and e["duration_ns"] >= 0
    return events, manifest, summary


def test_profiling_bundle_cpu_target():
    with tempfile.TemporaryDirectory() as d:
        run("profile", "cpu", d)
        events, manifest, summary = _read_bundle(d)
        comps = {e["component"] for e in events}
        assert {"compiler", "relay.transform", "codegen", "test"} <= comps
        spans = {e["span_id"]: e for e in events}
        infer = [e for e in events if e["pass_name"] == "InferType"][0]
        assert spans[infer["parent_span_id"]]["event_type"] == "compile"       # nesting follows the call stack
        assert os.path.exists(os.path.join(d, "artifacts", "kernel_main.c"))


def _roctx_bundle(target):
    with tempfile.TemporaryDirectory() as off, tempfile.TemporaryDirectory() as on:
        run("profile", target, off)
        run("profile", target, on, env={"KXC_PROFILE_ROCTX": "1"})
        e_off, m_off, _ = _read_bundle(off)
        e_on, m_on, _ = _read_bundle(on)
    assert m_off["enable_roctx"] is False and m_on["enable_roctx"] is True
    # ROCm ships the marker library in this image: the spans really push and pop their ranges
    assert m_on["roctx_available"] is True
    # markers change nothing in the bundle: the same spans in the same order
    assert [(e["component"], e["event_type"], e["pass_name"]) for e in e_on if e["component"] != "device_api"] == \
           [(e["component"], e["event_type"], e["pass_name"]) for e in e_off if e["component"] != "device_api"]


def test_roctx_ranges_cpu_target():
    """ProfileOptions::enable_roctx (the reference's enable_nvtx, include/base/profiling.h:65): every ScopedSpan
    pushes a range named component:event_type into libroctx64, loaded with dlopen, and pops it when it ends."""
    _roctx_bundle("cpu")


@pytest.mark.gpu
def test_roctx_ranges_hip_target():
    _roctx_bundle("hip")


# ------------------------------------------------------------------ adaptive runtime
def _adaptive_events(d):
    events, _, _ = _read_bundle(d)
    return [(e["component"], e["event_type"]) for e in events], events


def test_adaptive_runtime_cpu_target():
    """RuntimeSession / KernelCache / ShapePredictor / BackgroundCompiler / KernelRunner with the reference's rules
    (cache miss -> fuzzy hit -> background compile -> exact hit, priority order, status text), and the profiling
    events a session leaves."""
    with tempfile.TemporaryDirectory() as d:
        assert "adaptive runtime ok (cpu)" in run("adaptive", "cpu", d)
        kinds, events = _adaptive_events(d)
    for want in ("runtime_session_warmup", "runtime_session_run", "cache_fuzzy_hit", "cache_exact_hit",
                 "cache_miss_sync_compile", "background_compile_submitted", "background_compile_completed",
                 "runtime_session_wait_all"):
        assert ("runtime_session", want) in kinds, want
    assert ("background_compiler", "background_compile_task") in kinds
    assert kinds.count(("runtime_session", "cache_fuzzy_hit")) == 2 and kinds.count(("runtime_session", "cache_exact_hit")) == 2
    assert kinds.count(("runtime_session", "background_compile_submitted")) == 1
    runs = [e for e in events if e["event_type"] == "runtime_session_run"]
    assert all(e["shape_signature"] == "[[2,3],[3]]" or "2" in e["shape_signature"] for e in runs)
    task = [e for e in events if e["event_type"] == "background_compile_task"][0]
    submit = [e for e in events if e["event_type"] == "background_compile_submitted"][0]
    assert task["run_id"] == submit["run_id"]                  # the worker thread reports under the caller's run


@pytest.mark.gpu
def test_adaptive_runtime_hip_target():
    """The same on the GPU: worker threads build launch plans (and, for generated kernels, compile with hipRTC
    and load modules) while the calling thread keeps running."""
    assert "adaptive runtime ok (hip)" in run("adaptive", "hip")
    with tempfile.TemporaryDirectory() as d:
        assert "adaptive runtime ok (hipgen)" in run("adaptive", "hipgen", d)
        kinds, _ = _adaptive_events(d)
    # on the hip target a module compiled for larger extents is never run on the caller's (smaller) device buffers:
    # the fuzzy candidate counts as a miss and the exact shape is compiled on the calling thread
    assert ("runtime_session", "cache_fuzzy_skipped_device_buffers") in kinds
    assert ("runtime_session", "cache_fuzzy_hit") not in kinds
    assert kinds.count(("runtime_session", "cache_miss_sync_compile")) >= 2


@pytest.mark.gpu
def test_profiling_bundle_hip_events():
    """A profiled Run yields one backend.hip event per launch with the kernel symbol and the launch geometry the
    reference's adapter records for CUDA kernels (grid_x..block_z, dynamic_shared_memory), device_api spans
    with byte counts, and the execution plan as an artifact."""
    with tempfile.TemporaryDirectory() as d:
        run("profile", "hip", d)
        events, manifest, summary = _read_bundle(d)
        assert manifest["gpu_activity_source"] == "hip_events"
        kernels = [e for e in events if e["component"] == "backend.hip" and e["event_type"] == "hip_kernel"]
        plan = json.load(open(os.path.join(d, "artifacts", "execution_plan.json")))
        assert len(kernels) == len(plan["nodes"]) >= 3
        run_span = [e for e in events if e["component"] == "runtime" and e["event_type"] == "kernel_run"][0]
        for k, node in zip(kernels, plan["nodes"]):
            assert k["kernel_symbol"] == node["kernel_symbol"] and k["kernel_symbol"]
            assert k["parent_span_id"] == run_span["span_id"] and k["device"] == "hip:0"
            m = k["metrics"]
            assert m["grid_x"] >= 1 and m["block_x"] >= 64 and m["grid_y"] == m["grid_z"] == m["block_y"] == m["block_z"] == 1
            assert "dynamic_shared_memory" in m and k["duration_ns"] > 0
        assert any(k["kernel_symbol"].startswith("mfma_") or k["kernel_symbol"] == "direct" or "conv" in k["kernel_symbol"]
                   for k in kernels)
        starts = [k["ts_ns"] for k in kernels]
        assert starts == sorted(starts)
        copies = [e for e in events if e["component"] == "device_api" and e["event_type"] == "copy"]
        assert copies and all(c["metrics"]["bytes"] > 0 for c in copies)
        assert summary["component_counts"]["backend.hip"] >= len(kernels)


@pytest.mark.gpu
def test_hip_smoke_bundle_has_every_activity_kind():
    """The HIP counterpart of the reference's only GPU test (test/cupti_smoke_test.cpp:95-267): device API calls, a
    fill, the run-time compiled `scale_add` kernel launched with hipModuleLaunchKernel on a device-API stream.  The
    bundle holds backend.hip events of all four kinds with the metric keys of the reference's CUDA records
    (src/base/profiling.cc:537-651), device_api spans the bundle analyser's rules read, and a diagnosis."""
    with tempfile.TemporaryDirectory() as d:
        assert "HIP bundle generated at:" in run("hip_smoke", d)
        events, manifest, summary = _read_bundle(d)
        diagnosis = json.load(open(os.path.join(d, "diagnosis.json")))
    hip = [e for e in events if e["component"] == "backend.hip"]
    by_type = {}
    for e in hip:
        by_type.setdefault(e["event_type"], []).append(e)
    assert set(by_type) == {"hip_runtime_api", "hip_memcpy", "hip_memset", "hip_kernel"}
    apis = {e["fields"]["backend.hip.api"] for e in by_type["hip_runtime_api"]}
    assert {"hipMalloc", "hipStreamCreate", "hipMemsetAsync", "hipMemcpyAsync", "hipModuleLaunchKernel",
            "hipStreamSynchronize", "hipFree"} <= apis
    assert all(e["fields"]["backend.hip.return_value"] == "0" for e in by_type["hip_runtime_api"])
    (kernel,) = by_type["hip_kernel"]
    assert kernel["kernel_symbol"] == "scale_add" and kernel["device"] == "hip:0"
    m = kernel["metrics"]
    assert (m["grid_x"], m["grid_y"], m["grid_z"], m["block_x"], m["block_y"], m["block_z"]) == (1, 1, 1, 128, 1, 1)
    assert m["dynamic_shared_memory"] == 0 and kernel["duration_ns"] > 0
    assert kernel["fields"]["backend.hip.timing_source"] == "hip_events"
    (fill,) = by_type["hip_memset"]
    assert fill["metrics"]["bytes"] == 256 and fill["metrics"]["value"] == 0
    copies = by_type["hip_memcpy"]
    assert len(copies) == 3 and all(c["metrics"]["bytes"] == 256 and c["metrics"]["copy_count"] == 1 for c in copies)
    assert sorted(c["fields"]["backend.hip.copy_kind"] for c in copies) == ["0", "0", "1"]
    # every device record is tied to the API call that enqueued it
    api_ids = {e["fields"]["backend.hip.correlation_id"] for e in by_type["hip_runtime_api"]}
    assert all(e["fields"]["backend.hip.correlation_id"] in api_ids for e in copies + [fill, kernel])
    # on the stream (the thread's current one): copy in, fill, copy in again, the kernel, the copy out
    order = sorted([fill, kernel] + copies, key=lambda e: e["ts_ns"])
    assert [e["event_type"] for e in order] == ["hip_memcpy", "hip_memset", "hip_memcpy", "hip_kernel", "hip_memcpy"]
    assert len({e["fields"]["backend.hip.stream_id"] for e in order}) == 1
    device_api = [e for e in events if e["component"] == "device_api"]
    assert {"alloc_data_space", "copy", "stream_sync", "free_data_space"} <= {e["event_type"] for e in device_api}
    assert manifest["enable_gpu_activity"] is True
    assert diagnosis["diagnostics"] and all({"category", "severity", "component", "summary"} <= set(x) for x in diagnosis["diagnostics"])


@pytest.mark.gpu
def test_hip_smoke_bundle_from_rocprofiler_sdk():
    """The same smoke test with the activity records taken from rocprofiler-sdk's buffered tracing
    (ProfileOptions::enable_gpu_activity = 2; the tool library registers itself before the process's first HIP
    call), which is how the reference's adapter uses CUPTI (src/base/profiling.cc:250-695): the profiler sees the
    whole process, so a copy the TEST enqueues with hipMemcpyAsync -- outside the HIP library of this build -- is in
    the bundle next to the library's own three copies, the fill and the kernel, every device record tied to the API
    call that caused it and timed by the profiler."""
    with tempfile.TemporaryDirectory() as d:
        assert "HIP bundle generated at:" in run("hip_smoke_sdk", d)
        events, manifest, summary = _read_bundle(d)
    assert manifest["gpu_activity_source"] == "rocprofiler_sdk"
    hip = [e for e in events if e["component"] == "backend.hip"]
    by_type = {}
    for e in hip:
        by_type.setdefault(e["event_type"], []).append(e)
    assert set(by_type) == {"hip_runtime_api", "hip_memcpy", "hip_memset", "hip_kernel"}
    apis = [e["fields"]["backend.hip.api"] for e in by_type["hip_runtime_api"]]
    assert {"hipMalloc", "hipStreamCreate", "hipMemsetAsync", "hipMemcpyAsync", "hipModuleLaunchKernel", "hipStreamSynchronize", "hipFree"} <= set(apis)
    assert apis.count("hipMemcpyAsync") == 4                    # three by the device API, one by the test
    (kernel,) = by_type["hip_kernel"]                           # the runtime's own copy / fill kernels are not listed as kernels
    assert kernel["kernel_symbol"] == "scale_add" and kernel["device"] == "hip:0" and kernel["duration_ns"] > 0
    m = kernel["metrics"]
    assert (m["grid_x"], m["grid_y"], m["grid_z"], m["block_x"], m["block_y"], m["block_z"]) == (1, 1, 1, 128, 1, 1)
    (fill,) = by_type["hip_memset"]
    assert fill["metrics"]["bytes"] == 256 and fill["metrics"]["value"] == 0
    copies = by_type["hip_memcpy"]
    assert sorted(c["metrics"]["bytes"] for c in copies) == [200, 256, 256, 256]
    assert sorted(c["fields"]["backend.hip.copy_kind"] for c in copies) == ["0", "0", "0", "1"]
    device_records = copies + [fill, kernel]
    assert all(e["fields"]["backend.hip.timing_source"] in ("rocprofiler_sdk", "host_clock") for e in device_records)
    assert kernel["fields"]["backend.hip.timing_source"] == "rocprofiler_sdk"
    api_ids = {e["fields"]["backend.hip.correlation_id"] for e in by_type["hip_runtime_api"]}
    assert all(e["fields"]["backend.hip.correlation_id"] in api_ids for e in device_records)


@pytest.mark.gpu
def test_rocprofiler_sdk_source_is_refused_once_hip_has_initialised(pkg):
    """A rocprofiler-sdk tool registered after the HIP runtime initialised would never receive a record; the library
    notices (its probe call does not come back) and says what to do, and the default source still works."""
    import ctypes as C
    import torch
    torch.zeros(4, device="cuda")
    torch.cuda.synchronize()
    lib = pkg.lib()
    assert lib.kxc_hip_activity_enable(2) != 0
    assert "before the first HIP call" in lib.kxc_hip_last_error().decode()
    assert lib.kxc_hip_activity_enable(1) == 0
    try:
        p = C.c_void_p()
        assert lib.kxc_hip_alloc(0, C.c_size_t(256), C.c_size_t(64), C.byref(p)) == 0
        assert lib.kxc_hip_free(0, p) == 0
        n = C.c_int32(0)
        assert lib.kxc_hip_activity_drain(None, 0, C.byref(n)) == 0 and n.value >= 2
        room = n.value + 64
        records = C.create_string_buffer(room * 208)             # sizeof(kxc_hip_activity_record)
        assert lib.kxc_hip_activity_drain(records, room, C.byref(n)) == 0
        names = {records.raw[208 * i + 4:208 * i + 100].split(b"\0", 1)[0] for i in range(n.value)}
        assert {b"hipMalloc", b"hipFree"} <= names
    finally:
        assert lib.kxc_hip_activity_enable(0) == 0


def test_bundle_diagnosis_rules_cpu():
    """kernel_launch_overhead / copy_dominance / sync_overhead as the reference's bundle analyser defines them
    (python/kxc_agent/services/diagnosis_engine.py:233-297), evaluated when a bundle is written."""
    with tempfile.TemporaryDirectory() as d:
        assert "diagnosis rules ok" in run("diagnosis", d)
        cats = {x["category"] for x in json.load(open(os.path.join(d, "diagnosis.json")))["diagnostics"]}
    assert {"kernel_launch_overhead", "copy_dominance", "sync_overhead"} <= cats


# ------------------------------------------------------------------ ONNX import wire format
def _onnx_case(synth, d, batch, hw):
    import copy
    import onnx_spec
    consts = synth.resnet18_consts(3)
    spec, blob = onnx_spec.resnet18_spec(batch, hw, consts)
    onnx_spec.write(d, spec, blob)
    return consts, onnx_spec.reference_input(batch, hw), spec


def test_onnx_import_cpu_backend_bit_exact(synth):
    """import.json + params.bin -> Relay function -> CPU back end: the imported ResNet-18 reproduces the CPU
    oracle bit for bit on the reference's acceptance input pattern (parameters keep their bytes and their order)."""
    with tempfile.TemporaryDirectory() as d:
        consts, x, _ = _onnx_case(synth, d, 1, 32)
        out = run("onnx", "cpu", d)
        assert "imported: 42 params, input input, output logits" in out
        got = np.fromfile(os.path.join(d, "logits.bin"), np.float32).reshape(1, 1000)
        want = Oracle().resnet18(x, consts)
        assert (bits(got) == bits(want)).all()


def test_onnx_import_error_messages(synth):
    import copy
    with tempfile.TemporaryDirectory() as d:
        _, _, spec = _onnx_case(synth, d, 1, 32)

        def variant(name, edit):
            s = copy.deepcopy(spec)
            edit(s)
            with open(os.path.join(d, name), "w") as f:
                json.dump(s, f)

        variant("bad_format.json", lambda s: s.update(format="kxc.onnx_import.v0"))
        variant("bad_op.json", lambda s: s["function"]["nodes"][1].update(op_name="identity"))
        variant("bad_input.json", lambda s: s["function"]["nodes"][1].update(name="relu0", inputs=["nowhere"]))
        variant("bad_range.json", lambda s: s["params"][0].update(offset=10 ** 12))
        variant("bad_order.json", lambda s: s.update(param_order=list(reversed(s["param_order"]))))
        assert "onnx error messages ok" in run("onnx_errors", d)


@pytest.mark.gpu
def test_onnx_import_runs_on_hip(synth):
    """The same files on the HIP target: the reference's acceptance criterion (max abs error <= 1e-3 or max
    relative error <= 1e-3 with denominator max(1, |ref|), test/onnx_importer_test.cpp:146-179) against the CPU oracle."""
    with tempfile.TemporaryDirectory() as d:
        consts, x, _ = _onnx_case(synth, d, 2, 224)
        out = run("onnx", "hip", d)
        assert "launches: 20" in out
        got = np.fromfile(os.path.join(d, "logits.bin"), np.float32).reshape(2, 1000)
        want = Oracle(fast=True).resnet18(x, consts)
        abs_err = np.abs(got - want)
        rel_err = abs_err / np.maximum(1.0, np.abs(want))
        assert abs_err.max() <= 1e-3 or rel_err.max() <= 1e-3, (abs_err.max(), rel_err.max())
