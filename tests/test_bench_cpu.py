"""bench.py's contract on a machine without a GPU: it measures one GPU's
share only, so a request for several GPUs (the flag, or a launcher's
WORLD_SIZE) ends with a message and a non-zero status before any device
work; and the kernels and arithmetic type it reports are the workload's."""
import importlib.util
import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.mark.parametrize("argv,env", [(["--gpus", "2"], {}), (["--gpus", "8"], {}), ([], {"WORLD_SIZE": "2"})])
def test_bench_refuses_more_than_one_gpu(argv, env):
    r = subprocess.run([sys.executable, str(ROOT / "bench.py"), *argv], cwd=ROOT, capture_output=True, text=True,
                       timeout=120, env={**os.environ, **env})
    assert r.returncode == 2, r.stderr
    assert "single MI355X" in r.stderr and "--gpus 1" in r.stderr
    assert r.stdout == ""   # no JSON line


@pytest.mark.parametrize("config,kernels,dtype", [
    ("cfg2", "pa_decode_f16_kernel<128> + pa_merge_kernel<1, 32>", "f16"),
    ("cfg2_f32", "pa_gen_mfma_kernel + pa_gen_merge_kernel", "f32"),
    ("cfg4", "pa_decode_q8_kernel<128> + pa_merge_kernel<1, 32>", "f16"),
    ("phi3_decode", "pa_decode_f16_kernel<96> + pa_merge_kernel<1, 32>", "f16"),
])
def test_bench_names_the_kernels_and_their_arithmetic(config, kernels, dtype):
    spec = importlib.util.spec_from_file_location("bench", ROOT / "bench.py")
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    import iian_amd as pa
    from iian_amd import synth
    sp = synth.spec(config)
    blocks = int((sp.seq_lens.max() + sp.block_size - 1) // sp.block_size)
    assert bench.launch_kernels(sp, pa, blocks, sp.block_size, 256) == kernels
    assert bench.arithmetic_type(kernels) == dtype
    sp.D, sp.kv_type = 264, pa.GGML_TYPE_F32   # a head size only the general fp32 kernel takes
    got = bench.launch_kernels(sp, pa, blocks, sp.block_size, 256)
    assert got.startswith("pa_general_kernel") and bench.arithmetic_type(got) == "f32"
