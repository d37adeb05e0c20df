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
    source.write_text("#include \"kernels.h\"\n#include \"head_rows.h\"\n#include <cstdio>\nusing namespace mynah;\nint main() {\n    char e[256] = \"\";\n%s\n}\n" % body)
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


def test_fold_of_many_streams_is_refused_where_the_build_cannot(pkg, tmp_path):
    """Only the side-by-side residual build folds for more than two streams: with a bias, a LayerNorm, a probe or a further output the general
    build would run, which multiplies the rows as they are -- such a launch is refused."""
    lines = _run(pkg, tmp_path, """
    static StepSlots slots;
    static float at[4];
    for (int what = 0; what < 10; ++what)
        for (const int batch : {2, 3, 8}) {
            State st;
            LinearArgs a{};
            a.w = at; a.scales = at; a.qtype = MYNAH_HIP_INT8; a.n = a.k = 768; a.batch = batch; a.epilogue = EPI_RESIDUAL;
            for (int b = 0; b < a.batch && b < kBatchTile; ++b) { a.in[b] = at + (size_t)b * a.k; a.out[b] = at + (size_t)b * a.n; }
            a.fold_partial = a.fold_partial_ml = at; a.fold_slots = &slots;
            a.fold_heads = 12; a.fold_head_width = 64; a.fold_max_units = 17; a.fold_is_self = 1;
            switch (what) {
                case 1: a.bias = at; break;
                case 2: a.ln_gain = at; break;
                case 3: a.probe_qx = reinterpret_cast<int8_t *>(at); break;
                case 4: a.probe_sx = at; break;
                case 5: a.probe_acc = reinterpret_cast<int32_t *>(at); break;
                case 6: a.ln_out = at; break;
                case 7: a.ln_out_slots = &slots; break;
                case 8: a.aux_out = at; break;
                case 9: a.act_out = at; break;
            }
            const int rc = launch_linear(&st, a, e, sizeof e);
            printf("%d %d %d %s\\n", what, batch, rc, e);
        }""")
    assert len(lines) == 30
    for line in lines:
        what, batch = map(int, line.split()[:2])
        refused = batch > 2 and what != 0
        assert ("streams to fold for" if refused else "no ROCm-capable device") in line, line


def test_head_leaves_the_graph_by_the_callers_changes(pkg, tmp_path):
    """Other rows for the head's results count once, however many forms of the step (short and long caches or memories) are captured again for
    them; a caller that changes them at every step has the head run behind the graph after eight."""
    lines = _run(pkg, tmp_path, """
    HeadRows running;                       // three stream counts, four forms each, the caller's rows changed twice
    for (unsigned long long rows = 1; rows <= 3; ++rows)
        for (int turn = 0; turn < 2; ++turn)
            for (int form = 0; form < 4; ++form)
                for (int count = 3; count <= 5; ++count) running.step(count, 100 * rows + count);
    printf("%d %d\\n", running.changes, running.in_graph());
    HeadRows restless;
    int taken = 0;
    for (unsigned long long rows = 1; rows <= 20 && restless.in_graph(); ++rows, ++taken) restless.step(1, rows);
    printf("%d %d\\n", taken, restless.in_graph());""")
    assert lines == ["6 1", "9 0"]
