"""What the compiler cannot check in the kernels' sources."""
import glob
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_inline_assembly_names_the_m0_it_writes():
    """An asm statement that writes m0 lists it as clobbered, so that the compiler places none of its own uses of m0 across it."""
    found = 0
    for path in sorted(glob.glob(os.path.join(ROOT, "spy_amd", "csrc", "*.hip")) + glob.glob(os.path.join(ROOT, "spy_amd", "csrc", "*.cuh"))):
        for m in re.finditer(r"\basm\s*(?:volatile)?\s*\((.*?)\);", open(path).read(), re.S):
            if re.search(r"\bs_mov_b32 m0\b", m.group(1)):
                found += 1
                assert m.group(1).rsplit(":", 1)[1].count('"m0"') == 1, (path, m.group(0))
    assert found >= 2


def test_the_number_of_compute_units_is_kept_per_device():
    """The launchers ask spy_num_cu (runtime.hip, one record per device) and keep no number of their own; an engine keeps that of its device (peaks.hip, the measured ceilings, asks on every call)."""
    for path in sorted(glob.glob(os.path.join(ROOT, "spy_amd", "csrc", "*.hip")) + glob.glob(os.path.join(ROOT, "spy_amd", "csrc", "*.cuh"))):
        if os.path.basename(path) not in ("runtime.hip", "engine.hip", "peaks.hip"):
            assert not re.search("multiprocessorcount", open(path).read(), re.I), path


def test_single_token_attention_reads_no_keys_behind_the_last_one(tmp_path):
    """What the one-launch attention of order 1 requests before it knows the position lies within n_kv keys and the 16-byte piece of a V^T row that holds the last
    token where the position is a number (spy_hip_attn_decode, a caller's caches), and within n_ctx where it is in device memory (the engine's)."""
    out = str(tmp_path / "attn_reach")
    subprocess.check_call(["g++", "-O1", "-std=c++20", "-o", out, os.path.join(ROOT, "tests", "host", "attn_reach.cpp")])
    r = subprocess.run([out], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
    kernel = open(os.path.join(ROOT, "spy_amd", "csrc", "attn_short.hip")).read()
    assert kernel.count("xf_keys_before(IN_STATE") == 1 and kernel.count("xf_row_pieces_before(IN_STATE") == 1 and kernel.count("if (state) xattn_short_kernel<true>") == 1 and kernel.count("key_piece(0, keys0)") == 1
    # ... and the score kernel: each head's keys by its own group, no work for a group without heads
    kernel = open(os.path.join(ROOT, "spy_amd", "csrc", "exact_decode.cuh")).read()
    kernel = kernel[kernel.index("void xattn_scores_kernel("):kernel.index("// ---- softmax + P.V^T in the host order")]
    assert [kernel.count(f) for f in ("xs_log2(n_head)", "xs_share(n_kv, nb, nt)", "xs_head(n_head, hg, slot)", "if (hg >= n_head) return;", "hg + 8 * slot < n_head")] == [1] * 5


def test_launches_of_a_single_token_pass_read_no_environment():
    """What enqueues the kernels of a single-token pass, eagerly or into a graph that outlives the call, asks the engine and not the environment: a variable set
    after a capture would change eager passes but not replays."""
    engine = open(os.path.join(ROOT, "spy_amd", "csrc", "engine.hip")).read()
    body = engine[engine.index("static int enqueue_one("):engine.index("// ---- passes over several tokens")]
    assert "xattn_scores_kernel" in body and "spy_attn_short" in body and "static int enqueue_pass_any(" in body
    for name, text in [("engine.hip", body)] + [(n, open(os.path.join(ROOT, "spy_amd", "csrc", n)).read()) for n in ("exact_launch.cuh", "decode_launch.cuh", "attn_short.hip")]:
        assert "getenv" not in text, name


def test_launches_of_a_single_token_pass_depend_on_no_state_of_an_earlier_call():
    """How many cached tokens a pass sees chooses its attention kernels: an argument of what enqueues them, not a field of the engine that a call which fails half-way
    would leave behind for the next one."""
    types = open(os.path.join(ROOT, "spy_amd", "csrc", "engine_types.cuh")).read()
    engine = open(os.path.join(ROOT, "spy_amd", "csrc", "engine.hip")).read()
    assert "kv_bound" not in types and "->kv_bound" not in engine and ".kv_bound" not in engine
    assert "static int enqueue_one(spy_hip_llama *m, hipStream_t st, int which, int il, int kv_bound)" in engine


def test_shapes_of_the_packed_activation_tests_reach_every_tile(tmp_path):
    """The tile choice (gemm_tiles.h, on 256 compute units) for the shapes of the GPU tests: every tile there is runs on a matrix with a remainder on both sides, and the
    tests named for one kernel run that one."""
    from tests import oracle_lib as O
    from tests import test_gpu_exact_order as E, test_gpu_gemm as G
    out = str(tmp_path / "gemm_tiles")
    subprocess.check_call(["g++", "-O1", "-std=c++20", "-o", out, os.path.join(ROOT, "tests", "host", "gemm_tiles.cpp")])

    def tiles(which, flag, shapes):
        text = "".join("%s %d %d %d 256\n" % (which, flag, M, T) for M, K, T in shapes)
        got = [int(v) for v in subprocess.run([out], input=text, capture_output=True, text=True, check=True).stdout.split()]
        assert len(got) == len(shapes)
        return got

    def ragged(which, flag, shapes, rows=16):
        return {t for t, (M, K, T) in zip(tiles(which, flag, shapes), shapes) if M % rows and T % 16}

    for q8 in (0, 1):
        assert ragged("t", q8, E.PACKED_SHAPES + E.NARROW_SHAPES, 32) == set(range(8))
        assert set(tiles("t", q8, E.NARROW_SHAPES)) == {0, 1}, "xn_kernel with four and with two slots, and nothing else"
        assert {1} == {t for t, (M, K, T) in zip(tiles("t", q8, E.NARROW_SHAPES), E.NARROW_SHAPES) if M in (12284, 8196)}, "... two slots: remainders, odd numbers of chunks"
    for q4 in (0, 1):
        assert ragged("k", q4, E.PACKED_SHAPES + E.ANY_SCALE_SHAPES) == set(range(5))
        assert set(tiles("k", q4, E.ANY_SCALE_SHAPES)) == {1, 2, 3, 4}
        assert [t for t, (M, K, T) in zip(tiles("k", q4, E.ANY_SCALE_SHAPES), E.ANY_SCALE_SHAPES) if M % 128 and (T + 15) // 16 % 8 and t == 4], "128 rows x 8 groups, part of either"
        own = [s[1:] for s in G.OWN_SHAPES if s[0] == (O.Q4_K if q4 else O.Q6_K)]
        assert ragged("o", q4, own + G.SPLIT_SHAPES, 32) == set(range(9)) - (set() if q4 else {2})       # (64 rows x 2 groups of Q6_K: chosen for no shape there is up to 36000 rows by 4096)
        split = list(zip(tiles("o", q4, G.SPLIT_SHAPES), G.SPLIT_SHAPES))
        assert {t for t, (M, K, T) in split if K == 256} >= {6, 7, 8}, "one super-block for all sets"
        assert {t for t, _ in split} == {0, 6, 7, 8}
    own = [s[1:] for s in G.OWN_SHAPES if s[0] == O.Q4_0]
    assert set(tiles("q", 0, own)) == {0} and set(tiles("q", 0, G.TILES_OF_32_SHAPES)) == {1}


def test_single_token_qkv_pairs_q4_0_and_q8_0_with_themselves_only(tmp_path):
    """The kernel undoes the factor 16 of Q4_0's high nibbles, and sums the activations that fold its -8, by the type of wq and wk: with another type of wv beside it, it does not compile."""
    import shutil
    from concurrent.futures import ThreadPoolExecutor
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

    def compiles(pair):
        src = tmp_path / ("%d_%d.hip" % pair)
        src.write_text('#include "%s/spy_amd/csrc/exact_decode.cuh"\nauto kernel = xgemv_kernel<%d, 1, 2, 1, EPI_QKV, %d>;\n' % (ROOT, pair[0], pair[1]))
        r = subprocess.run([hipcc, "--offload-arch=gfx950", "-std=c++20", "--cuda-device-only", "-fsyntax-only", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", str(src)],
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0 or "follow WT in every step" in r.stderr, r.stderr
        return r.returncode == 0

    from spy_amd._lib import Q4_0, Q4_K, Q6_K, Q8_0
    with ThreadPoolExecutor(4) as pool:
        assert list(pool.map(compiles, [(Q4_0, Q4_0), (Q4_K, Q6_K), (Q8_0, Q4_0), (Q4_0, Q8_0), (Q4_0, Q6_K)])) == [True, True, False, False, False]


def test_a_wave_releases_what_all_its_lanes_wrote_before_it_is_counted():
    """Waves of the single-token softmax meet on counters in LDS: one lane counts its wave, but what the others wait for was written by all 64, so the release is
    theirs too and stands ahead of the branch."""
    kernel = open(os.path.join(ROOT, "spy_amd", "csrc", "exact_decode.cuh")).read()
    body = re.search(r"void xp_arrive\(uint32_t \*c\) \{(.*?)\n\}", kernel, re.S).group(1)
    fence, barrier, branch, count = (body.index(x) for x in ('__builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup")', "__builtin_amdgcn_wave_barrier()", "if (", "__hip_atomic_fetch_add(c"))
    assert fence < barrier < branch < count
    await_ = re.search(r"void xp_await\(.*?\n", kernel).group(0)
    assert "__ATOMIC_ACQUIRE" in await_ and "if (" not in await_


def test_objects_are_remade_when_the_flags_change():
    """Flags lie in the Makefile, so every object depends on it, and on every header there is."""
    csrc = os.path.join(ROOT, "spy_amd", "csrc")
    sources = {os.path.basename(p) for p in glob.glob(os.path.join(csrc, "*.hip"))}
    for changed in ["Makefile"] + [os.path.basename(p) for p in glob.glob(os.path.join(csrc, "*.cuh")) + glob.glob(os.path.join(csrc, "*.h"))]:
        r = subprocess.run(["make", "-C", csrc, "-n", "-W", changed], capture_output=True, text=True, check=True, timeout=60)
        assert set(re.findall(r" -c (\S+\.hip) ", r.stdout)) == sources, changed
