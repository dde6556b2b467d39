"""Build the package's HIP libraries (gfx950) in-tree with hipcc.  No GPU is needed to build.

Three libraries, each from its own folder of translation units, so that a model only waits for what it runs on:
  qlinear  csrc/*.hip         -> nanovllm/_lib/libqlinear.so   (quantized linears, Qwen3 operators, attention)
  seqmix   csrc/seqmix/*.hip  -> nanovllm/_lib/libseqmix.so    (multi-stream residuals, short convolutions, latent
                                                                attention with or without a rotated part and a window,
                                                                PolyNorm / gated / GELU / squared-ReLU feed-forwards,
                                                                expert routing)
  hymix    csrc/hymix/*.hip   -> nanovllm/_lib/libhymix.so     (gated, grouped-norm, tanh-norm and layer-norm residuals, token shift,
                                                                attention with sinks, windows, pooled blocks, chunked
                                                                masks, soft caps and sigmoid weights over a paged cache,
                                                                delta-rule, gated-delta, constant-decay, state-space and
                                                                selective-scan recurrences)
``python build.py [--force] [qlinear|seqmix|hymix]`` builds one of them, or all without a name."""
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "nanovllm", "_lib")
LIB = os.path.join(OUT_DIR, "libqlinear.so")
SEQMIX_LIB = os.path.join(OUT_DIR, "libseqmix.so")
HYMIX_LIB = os.path.join(OUT_DIR, "libhymix.so")
# The packed-f32 VALU forms stay off (plain f32 code only): some of them have given wrong results on this hardware.  Without them
# products and sums that were a packed multiply and a packed add, in the norms and the rotation among others, become fused
# multiply-adds: one rounding less, so their results differ from a build with the packed forms by up to a bf16 rounding.
FLAGS = ["--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-fno-gpu-rdc", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops"]
# Kernels of one wave per SIMD have 512 registers, and there the compiler puts the results of matrix instructions into the accumulation
# half, from which the vector unit has to copy every number that it reads.  These files' kernels read them all (softmax, splits, folds)
# and need few more than 256: results in the vector half take the copies out (the chunked recurrences' walk 1.09 x, latent decode
# attention 1.14 x; the same bits).  Tiles that hold 256 sums per lane (sm_moe_tiles) need the other half.
VECTOR_RESULTS = ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]
FILE_FLAGS = {f: VECTOR_RESULTS for f in ("hm_outer_chunk.hip", "hm_attn_mfma.hip", "sm_latent_decode.hip", "sm_latent_mfma.hip",
                                          "ql_gemm_inst_wide_bf16_i8.hip", "ql_gemm_inst_wide_bf16_fp8.hip")}
TARGETS = {
    "qlinear": dict(src=CSRC, lib=LIB, header="qlinear.h", flags=FLAGS, obj=""),
    "seqmix": dict(src=os.path.join(CSRC, "seqmix"), lib=SEQMIX_LIB, header="seqmix.h", flags=FLAGS, obj="seqmix_"),
    "hymix": dict(src=os.path.join(CSRC, "hymix"), lib=HYMIX_LIB, header="hymix.h", flags=FLAGS, obj="hymix_"),
}


def _hipcc():
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found")
    return exe


def _stale(target, deps):
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def build(force=False, verbose=True, target="qlinear"):
    """Compile one library (``target`` = "qlinear" | "seqmix") or all of them ("all"); returns the path of the (last) library."""
    if target == "all":
        for name in TARGETS:
            lib = build(force, verbose, name)
        return lib
    spec = TARGETS[target]
    CSRC, LIB, FLAGS = spec["src"], spec["lib"], spec["flags"]
    os.makedirs(OUT_DIR, exist_ok=True)
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    hipcc = _hipcc()
    shared = os.path.join(HERE, "csrc")                                   # headers of more than one library lie there
    headers = [os.path.join(d, f) for d in {CSRC, shared} for f in os.listdir(d) if f.endswith(".h")]
    headers += [os.path.join(HERE, "..", "include", spec["header"]), os.path.abspath(__file__)]       # (the flags are here)
    srcs = sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))      # every translation unit of the folder

    def compile_one(src):
        obj = os.path.join(objdir, spec["obj"] + src.replace(".hip", ".o"))
        path = os.path.join(CSRC, src)
        if force or _stale(obj, [path] + headers):
            cmd = [hipcc] + FLAGS + FILE_FLAGS.get(src, []) + ["-c", path, "-o", obj]
            if verbose:
                print(" ".join(cmd), flush=True)
            subprocess.check_call(cmd)
        return obj

    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(compile_one, srcs))
    if force or _stale(LIB, objs):
        cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.check_call(cmd)
    return LIB


if __name__ == "__main__":
    names = [a for a in sys.argv[1:] if not a.startswith("-")] or ["all"]
    for name in names:
        print(build(force="--force" in sys.argv, target=name))
