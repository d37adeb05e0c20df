"""The host-side rules that choose how products are launched, called directly: a small C++ program is compiled against the library's
internal headers and linked with it.  No device is visible to it, so a launch that a rule lets through ends at the runtime's
"no device" error, and one that a rule refuses with that rule's message."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def _run(pkg, tmp_path, body):
    """The lines a program prints whose main() has `body`."""
    lib = pkg.load_library()._name
    source, program = tmp_path / "rules.cpp", tmp_path / "rules"
    source.write_text("#include \"kernels.h\"\n#include <cstdio>\nusing namespace mynah;\nint main() {\n    char e[256] = \"\";\n%s\n}\n" % body)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I", os.path.join(ROOT, "include"), "-I",
                    os.path.join(ROOT, "mynah-tts_amd", "csrc"), str(source), lib, "-L", os.path.join(ROCM, "lib"), "-lamdhip64",
                    "-Wl,-rpath," + os.path.dirname(lib), "-Wl,-rpath," + os.path.join(ROCM, "lib"), "-o", str(program)], check=True)
    env = dict(os.environ, HIP_VISIBLE_DEVICES="", ROCR_VISIBLE_DEVICES="")
    return subprocess.run([str(program)], check=True, env=env, stdout=subprocess.PIPE, text=True).stdout.splitlines()


def test_list_of_products_that_the_rule_takes_is_launched(pkg, tmp_path):
    """What linear_takes_list accepts launches whatever the number of products: rows per workgroup grow with it, up to what the launch's
    packed arguments hold."""
    lines = _run(pkg, tmp_path, """
    const int shapes[][3] = {{768, 16, 24}, {768, 3, 64}, {49152, 3, 64}, {49152, 16, 64}, {65532, 4, 64}, {65532, 9, 64}, {65532, 16, 2}};
    for (const int storage : {MYNAH_HIP_F32, MYNAH_HIP_F16, MYNAH_HIP_INT8, MYNAH_HIP_INT4})
        for (const auto &s : shapes) {
            State st;
            static float at[4];
            LinearArgs a{};
            a.w = at; a.scales = at; a.qtype = storage; a.n = s[0]; a.k = 768; a.batch = s[1]; a.epilogue = EPI_NONE;
            for (int b = 0; b < a.batch && b < kBatchTile; ++b) { a.in[b] = at + (size_t)b * a.k; a.out[b] = at + (size_t)b * a.n; }
            const bool takes = linear_takes_list(a.qtype, a.n, a.k, a.batch, a.k, a.n);
            const int rc = launch_linear_products(&st, a, reinterpret_cast<const LinearProduct *>(at), s[2], e, sizeof e);
            printf("storage %d, %d x %d, %d products: %d %d %s\\n", storage, s[1], s[0], s[2], takes, rc, e);
        }""")
    assert len(lines) == 28
    for line in lines:
        assert ": 1 -1 " in line and "no ROCm-capable device" in line, line
