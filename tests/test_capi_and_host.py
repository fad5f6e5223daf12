"""CPU-side checks of the boundary: the C-ABI library loads and exports every symbol that
include/ttmi.h declares, the pybind module and the drop-in package import, and the host
logic that needs no GPU (Tensor/DLPack semantics, allocator rounding, the npz reader, error
paths).  No compute entry point is called here.
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest
import torch

from turbotransformers_amd import capi


def test_header_declares_and_library_exports_every_entry_point():
    protos = capi.parse_header()
    assert len(protos) >= 45
    lib = ctypes.CDLL(capi.LIB_PATH)
    missing = [n for n in protos if not hasattr(lib, n)]
    assert not missing, missing
    # and nothing with C linkage is exported that the header does not declare
    out = subprocess.run(["nm", "-D", "--defined-only", capi.LIB_PATH], capture_output=True, text=True).stdout
    exported = {l.split()[-1] for l in out.splitlines() if " T " in l and l.split()[-1].startswith("ttmi_")}
    assert exported == set(protos), exported ^ set(protos)


def test_every_declaration_cites_or_explains_itself():
    text = open(capi.HEADER).read()
    assert text.count("TTMI_API int") >= 40 and "extern \"C\"" in text
    assert "torch" not in text.split("*/", 1)[1].lower().replace("pytorch", "")  # no torch types in signatures


def test_error_reporting_without_a_gpu():
    lib = capi.load()
    rc = lib.ttmi_layer_norm(None, None, None, 1, 8, 1e-12, capi.F32, None)
    assert rc == -1 and b"null tensor" in lib.ttmi_last_error()
    with pytest.raises(capi.TtmiError):
        capi.check(lib.ttmi_gemm(None, None, None, 1, 1, 1, 1, 1, 1, 0, 1.0, 0.0, capi.F32, None))
    n = ctypes.c_int(-1)
    assert lib.ttmi_device_count(ctypes.byref(n)) == 0 and n.value >= 0


def test_dropin_package_surface():
    import turbo_transformers as tt
    import turbo_transformers.turbo_transformers_cxx as cxx
    for name in ("BertModel", "BertLayer", "BertEncoder", "BertAttention", "BertIntermediate", "BertOutput",
                 "BertEmbeddings", "BertPooler", "SequencePool", "PoolingType", "ReturnType", "BertModelSmartBatch",
                 "MultiHeadedAttentionSmartBatch", "AlbertModel", "AlbertLayer", "MultiHeadedAttention",
                 "PositionwiseFeedForward", "DistrillFFN", "QBertModel", "pref_guard", "nparray2tensor", "tensor2nparrayf",
                 "tensor2nparrayl", "enable_perf", "disable_perf", "set_num_threads", "reset_allocator_schema",
                 "bert_opt_mem_allocate_api"):
        assert hasattr(tt, name), name
    for name in ("Tensor", "BERTEmbedding", "BertAttention", "MultiHeadedAttention", "MultiHeadedAttentionSmartBatch",
                 "BertIntermediate", "BertOutput", "SequencePool", "BertPooler", "PrepareBertMasks", "AlbertLayer",
                 "FusedAddBiasGELU", "FusedAddBiasLayerNorm", "PositionwiseFeedForward", "DistrillFFN", "nparray2tensor", "tensor2nparrayf", "tensor2nparrayl",
                 "set_num_threads", "reset_allocator_schema", "bert_opt_mem_allocate_api", "enable_perf", "disable_perf",
                 "set_stderr_verbose_level"):
        assert hasattr(cxx, name), name
    assert cxx.config.is_compiled_with_cuda() is True
    assert callable(tt.BertModel.from_torch)


def test_tensor_dlpack_round_trip_and_ownership():
    import turbo_transformers.turbo_transformers_cxx as cxx
    t = torch.arange(24, dtype=torch.float32).reshape(2, 3, 4)
    capsule = torch.utils.dlpack.to_dlpack(t)
    tt = cxx.Tensor.from_dlpack(capsule)
    assert tt.n_dim() == 3 and [tt.shape(i) for i in range(3)] == [2, 3, 4] and tt.shape(-1) == 4
    assert tt.float_data() == t.data_ptr()            # alias, not a copy
    with pytest.raises(RuntimeError):
        tt.shape(3)
    back = torch.utils.dlpack.from_dlpack(tt.to_dlpack())
    assert back.data_ptr() == t.data_ptr() and torch.equal(back, t)
    assert tt.is_null()                               # to_dlpack released ownership
    with pytest.raises(RuntimeError):
        tt.to_dlpack()
    assert cxx.Tensor.create_empty().is_null()
    i64 = cxx.Tensor.from_dlpack(torch.utils.dlpack.to_dlpack(torch.ones(3, dtype=torch.int64)))
    with pytest.raises(RuntimeError):                 # dtype check of data<float>()
        i64.float_data()


def test_numpy_converters_on_cpu():
    import turbo_transformers.turbo_transformers_cxx as cxx
    a = np.arange(12, dtype=np.float32).reshape(3, 4)
    t = cxx.nparray2tensor(a, "CPU")
    assert np.array_equal(cxx.tensor2nparrayf(t), a)
    ids = np.arange(5, dtype=np.int64)
    assert np.array_equal(cxx.tensor2nparrayl(cxx.nparray2tensor(ids, "CPU")), ids)
    with pytest.raises(RuntimeError):
        cxx.nparray2tensor(a, "TPU")


def test_layers_reject_cpu_tensors_and_bad_shapes():
    """No CPU fallback: a layer built on host tensors refuses to run; shape checks raise."""
    import turbo_transformers.turbo_transformers_cxx as cxx
    conv = lambda x: cxx.Tensor.from_dlpack(torch.utils.dlpack.to_dlpack(x))
    inter = cxx.BertIntermediate(conv(torch.zeros(8, 32)), conv(torch.zeros(32)))
    with pytest.raises(RuntimeError, match="not on the GPU"):
        inter(conv(torch.zeros(2, 8)), cxx.Tensor.create_empty())
    with pytest.raises(RuntimeError):  # weight/bias mismatch (bert_intermediate.cpp EnforceShapeAndType)
        cxx.BertIntermediate(conv(torch.zeros(8, 32)), conv(torch.zeros(31)))
    with pytest.raises(RuntimeError):
        cxx.SequencePool("Median")
    with pytest.raises(RuntimeError):
        cxx.reset_allocator_schema("no-such-schema")
    cxx.reset_allocator_schema("naive")
    import turbo_transformers as tt
    from transformers import BertConfig, BertModel
    tiny = BertModel(BertConfig(vocab_size=10, hidden_size=8, num_hidden_layers=1, num_attention_heads=2,
                                intermediate_size=16, max_position_embeddings=8))
    with pytest.raises(RuntimeError, match="GPU"):
        tt.BertModel.from_torch(tiny, torch.device("cpu"), "turbo")
    with pytest.raises(NotImplementedError):
        tt.BertModel.from_torch(tiny, torch.device("cpu"), "onnxrt")


def test_npz_reader_matches_numpy(tmp_path):
    import turbo_transformers.turbo_transformers_cxx as cxx
    rng = np.random.default_rng(0)
    arrays = {"embeddings.word_embeddings.weight": rng.standard_normal((7, 4)).astype(np.float32),
              "pooler.dense.bias": rng.standard_normal(4).astype(np.float32),
              "half": rng.standard_normal((2, 3)).astype(np.float16),
              "ids": np.arange(6, dtype=np.int64).reshape(2, 3)}
    path = str(tmp_path / "w.npz")
    np.savez(path, **arrays)
    loaded = cxx.load_npz(path)
    assert set(loaded) == set(arrays)
    for k, v in arrays.items():
        assert loaded[k].dtype == v.dtype and np.array_equal(loaded[k], v)
    # deflated members: what numpy.savez_compressed and the reference's converter
    # (tools/convert_huggingface_bert_pytorch_to_npz.py:71) write; a larger, compressible array as well
    arrays["big"] = np.tile(rng.standard_normal(1000).astype(np.float32), 300).reshape(600, 500)
    np.savez_compressed(path, **arrays)
    loaded = cxx.load_npz(path)
    assert set(loaded) == set(arrays)
    for k, v in arrays.items():
        assert loaded[k].dtype == v.dtype and np.array_equal(loaded[k], v)
    # a truncated archive is an error, not a crash
    data = open(path, "rb").read()
    bad = str(tmp_path / "bad.npz")
    open(bad, "wb").write(data[:len(data) // 2])
    with pytest.raises(RuntimeError):
        cxx.load_npz(bad)


def test_converter_writes_the_reference_key_scheme(tmp_path):
    """tools/convert_huggingface_bert_pytorch_to_npz.py:44-71: q/k/v packed into qkv.weight [hidden, 3*hidden] and
    qkv.bias, other dense weights transposed to [in, out]; the (deflated) file reads back through the C++ loader."""
    import torch
    from transformers import BertConfig, BertModel
    import turbo_transformers.turbo_transformers_cxx as cxx
    from turbotransformers_amd.convert_huggingface_bert_to_npz import save_bert_npz
    torch.manual_seed(0)
    model = BertModel(BertConfig(num_hidden_layers=2, hidden_size=64, num_attention_heads=4, intermediate_size=128, vocab_size=100))
    path = str(tmp_path / "m.npz")
    save_bert_npz(model, path)
    got = cxx.load_npz(path)
    sd = {k: v.detach().numpy() for k, v in model.named_parameters()}
    assert not any(".attention.self." in k for k in got)
    for i in range(2):
        p = "encoder.layer.%d." % i
        want = np.concatenate([sd[p + "attention.self.%s.weight" % x] for x in ("query", "key", "value")], 0).T
        assert np.array_equal(got[p + "attention.qkv.weight"], want) and want.shape == (64, 192)
        assert np.array_equal(got[p + "attention.qkv.bias"],
                              np.concatenate([sd[p + "attention.self.%s.bias" % x] for x in ("query", "key", "value")]))
        assert np.array_equal(got[p + "intermediate.dense.weight"], sd[p + "intermediate.dense.weight"].T)
        assert np.array_equal(got[p + "output.dense.weight"], sd[p + "output.dense.weight"].T)
        assert np.array_equal(got[p + "attention.output.dense.weight"], sd[p + "attention.output.dense.weight"].T)
    assert np.array_equal(got["pooler.dense.weight"], sd["pooler.dense.weight"].T)
    assert np.array_equal(got["embeddings.word_embeddings.weight"], sd["embeddings.word_embeddings.weight"])



def _stored_npz(path, members):
    """A zip archive of stored (uncompressed) members with the given raw bytes."""
    import zipfile
    with zipfile.ZipFile(path, "w", zipfile.ZIP_STORED) as z:
        for name, raw in members.items():
            z.writestr(name, raw)


def _npy(header_text, payload=b""):
    head = header_text.encode("latin1")
    return b"\x93NUMPY\x01\x00" + len(head).to_bytes(2, "little") + head + payload


@pytest.mark.parametrize("header", [
    "{'descr': '<f4', 'fortran_order': False, 'shape': (2, 3), }",                # payload missing
    "{'descr': '<f4', 'fortran_order': False, 'shape': (4611686018427387904, 4), }",  # product wraps around 2^64
    "{'descr': '<f4', 'fortran_order': False, 'shape': (99999999999999999999999, ), }",
    "{'descr': '<f4', 'fortran_order': False, 'shape' ",                          # no parenthesis
    "{'descr': '<f4', 'fortran_order': False }",                                   # no shape
    "{'descr': <f4, 'fortran_order': False, 'shape': (1, ), }",                    # unquoted dtype
    "{'descr': '<fx', 'fortran_order': False, 'shape': (1, ), }",                  # dtype size is not a number
    "{'descr'",                                                                    # nothing after the key
    "{'descr': '<f4', 'fortran_order':",                                           # ends inside a value
    "{'descr': '<f4', 'fortran_order': True, 'shape': (1, ), }",
    "{'descr': '<c8', 'fortran_order': False, 'shape': (1, ), }",
])
def test_npz_reader_refuses_malformed_members(tmp_path, header):
    """A malformed member ends in the loader's own error (RuntimeError), never in a crash or a C++ library exception
    of another type; a well-formed neighbour is no excuse."""
    import turbo_transformers.turbo_transformers_cxx as cxx
    path = str(tmp_path / "m.npz")
    _stored_npz(path, {"ok.npy": _npy("{'descr': '<f4', 'fortran_order': False, 'shape': (1, ), }".ljust(118) + "\n",
                                      np.float32(1).tobytes()),
                       "bad.npy": _npy(header.ljust(118) + "\n", b"\0" * 16)})
    with pytest.raises(RuntimeError):
        cxx.load_npz(path)


def test_npz_reader_refuses_sizes_beyond_the_file(tmp_path):
    import turbo_transformers.turbo_transformers_cxx as cxx
    path = str(tmp_path / "m.npz")
    np.savez(path, a=np.arange(4, dtype=np.float32))
    data = bytearray(open(path, "rb").read())
    cd = data.rfind(b"PK\x01\x02")
    data[cd + 20:cd + 28] = (0x7ffffff0).to_bytes(4, "little") * 2  # compressed and uncompressed size of the member
    open(path, "wb").write(bytes(data))
    with pytest.raises(RuntimeError):
        cxx.load_npz(path)


def test_gemm_describe_names_the_variant_without_a_device():
    """ttmi_gemm_describe runs the launchers' own selection with launching switched off, so it answers on a machine
    without a GPU: a family, the wavefronts per workgroup, the tile and the K split."""
    import ctypes
    import re
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)
    args = capi.EpilogueArgs()
    args.act = capi.ACT_GELU
    for m, n, k, epi in [(32768, 3072, 768, capi.EPI_BIAS_ACT), (32768, 768, 3072, capi.EPI_NONE), (128, 768, 3072, capi.EPI_NONE),
                         (2560, 768, 3072, capi.EPI_BIAS)]:
        capi.check(lib.ttmi_gemm_describe(m, n, k, epi, ctypes.byref(args), capi.F16, buf, 64))
        assert re.fullmatch(r"(reg|dma|dma_agpr|dma3_agpr|wave)\d+w_\d+x\d+(_splitk\d+)?", buf.value.decode()), buf.value
    assert lib.ttmi_gemm_describe(128, 768, 3072, capi.EPI_NONE, None, capi.F16, buf, 4) != 0  # too small for the answer


def test_one_short_sequence_splits_k_only_where_a_second_launch_pays():
    """128 tokens: the output projection and the second FFN product (24 tiles of 64 x 64) are cut along K; the
    intermediate Linear (96 tiles) keeps bias + GELU in the GEMM in 16-bit types, where the reduction kernel's launch
    costs more than the split saves, and is cut in fp32, where it does not."""
    import ctypes
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)
    args = capi.EpilogueArgs()
    args.act = capi.ACT_GELU

    def variant(m, n, k, epi, dt):
        capi.check(lib.ttmi_gemm_describe(m, n, k, epi, ctypes.byref(args), dt, buf, 64))
        return buf.value.decode()

    assert "_splitk" in variant(128, 768, 768, capi.EPI_NONE, capi.F16)
    assert "_splitk" in variant(128, 768, 3072, capi.EPI_NONE, capi.F16)
    assert variant(128, 3072, 768, capi.EPI_BIAS_ACT, capi.F16) == "wave1w_32x32"
    assert variant(128, 3072, 768, capi.EPI_BIAS_ACT, capi.BF16) == "wave1w_32x32"
    assert "_splitk" in variant(128, 3072, 768, capi.EPI_BIAS_ACT, capi.F32)


def test_up_to_128_rows_of_16_bit_operands_take_the_wavefront_kernel():
    """One wavefront per 32 x 32 tile, operand fragments straight from global memory: 16-bit types, at most 128 rows,
    K a multiple of the 128-byte step; fp32 and longer inputs stay on the LDS-tiled kernels."""
    import ctypes
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)

    def variant(m, n, k, dt):
        capi.check(lib.ttmi_gemm_describe(m, n, k, capi.EPI_NONE, None, dt, buf, 64))
        return buf.value.decode()

    for m in (1, 10, 40, 128):
        assert variant(m, 2304, 768, capi.F16).startswith("wave1w_32x32")  # cut along K while its tiles are few
        assert variant(m, 2304, 768, capi.BF16).startswith("wave1w_32x32")
        assert variant(m, 768, 3072, capi.F16).startswith("wave1w_32x32_splitk")
    assert not variant(128, 2304, 768, capi.F32).startswith("wave")
    assert not variant(129, 2304, 768, capi.F16).startswith("wave")
    assert not variant(128, 2304, 776, capi.F16).startswith("wave")


def test_transposed_v_of_sequences_shorter_than_8_stays_off_the_one_wavefront_per_simd_kernel():
    """That kernel stores a group of eight rows of a transposed V that leaves its sequence element by element into
    this sequence and the next one; with fewer than 8 positions per sequence a group would touch three, so such a
    QKV projection runs on the other kernels however many rows it has."""
    import ctypes
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)

    def variant(batch, seq, pitch):
        args = capi.EpilogueArgs()
        args.bias = args.q = args.k = args.v = 1 << 20  # never dereferenced: describe launches nothing
        args.seq, args.heads, args.head_dim, args.v_seq_pitch = seq, 12, 64, pitch
        capi.check(lib.ttmi_gemm_describe(batch * seq, 2304, 768, capi.EPI_QKV_SPLIT, ctypes.byref(args), capi.F16, buf, 64))
        return buf.value.decode()

    assert variant(1000, 12, 16).startswith("dma_agpr4w")
    assert variant(1500, 8, 8).startswith("dma_agpr4w")
    assert variant(2400, 5, 0).startswith("dma_agpr4w")  # row-major V: any length
    assert not variant(2400, 5, 8).startswith("dma_agpr4w")


def test_fp32_products_pick_tiles_by_rounds_over_the_compute_units():
    """fp32 is bound by the matrix pipe at every tile size, so the tile (and a cut along K) is chosen for whole
    rounds of tiles over the CUs: a few thousand rows by 768 columns run on 64 x 64 tiles where the 16-bit types take
    128 x 128, a last round that is nearly empty is filled by slices of K, large products keep the large tiles."""
    import ctypes
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)

    def variant(m, n, k, dt):
        capi.check(lib.ttmi_gemm_describe(m, n, k, capi.EPI_NONE, None, dt, buf, 64))
        return buf.value.decode()

    assert variant(4000, 768, 3072, capi.F32) == "reg4w_64x64"        # 756 tiles: three rounds of 256
    assert variant(4000, 768, 3072, capi.F16) == "dma4w_128x128"
    assert variant(1600, 768, 3072, capi.F32) == "reg4w_64x64_splitk5"  # 300 tiles are 1.17 rounds: 1500 slices, six
    assert variant(1600, 768, 768, capi.F32) == "reg4w_64x64"          # K too short for the cut to pay
    assert variant(32768, 3072, 768, capi.F32) == "dma8w_256x256"
    assert variant(128, 768, 3072, capi.F32) == "reg4w_64x64_splitk10"  # one short sequence: as before


def test_fused_products_off_the_ring_keep_the_kernels_for_their_size():
    """Widths that are no multiple of eight (vocabulary- and class-sized heads), operands of 2 GiB and more and heads that no
    16-byte store fits are refused by the ring tiles; they then run on the DMA tiles, the wavefront kernel or K slices that
    their size calls for, not all on the register-staged tiles."""
    import ctypes
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)

    def variant(m, n, k, dt, epi=capi.EPI_BIAS, args=None):
        capi.check(lib.ttmi_gemm_describe(m, n, k, epi, ctypes.byref(args or capi.EpilogueArgs()), dt, buf, 64))
        return buf.value.decode()

    for dt in (capi.F16, capi.BF16):
        assert variant(8192, 30522, 768, dt) == "dma8w_256x256"
        assert variant(600000, 768, 3072, dt) == "dma8w_256x256"
        assert variant(1000, 772, 3072, dt) == "dma4w_128x64"
        assert variant(200, 772, 3072, dt).startswith("reg4w_64x64_splitk")
        assert variant(128, 772, 3072, dt) == "wave1w_32x32"
        assert variant(10, 2, 768, dt) == "wave1w_32x32"
    assert variant(128, 772, 3072, capi.F32).startswith("reg4w_64x64_splitk")
    assert variant(8192, 30522, 768, capi.F32).startswith("dma8w")
    heads = capi.EpilogueArgs()
    heads.seq, heads.heads, heads.head_dim = 128, 12, 20
    assert variant(64 * 128, 720, 256, capi.F16, capi.EPI_QKV_SPLIT, heads).startswith("dma")


def test_gelu_products_of_65_to_128_rows_leave_the_ring_only_for_one_short_sequence():
    """The wavefront kernel (16-bit, whole) and the cut along K (fp32) are kept for the widths of an intermediate Linear over
    one short sequence; long K, few columns and wide outputs take the ring tiles, which the wavefront kernel trails by up to
    four times there."""
    import ctypes
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)
    args = capi.EpilogueArgs()
    args.act = capi.ACT_GELU

    def variant(m, n, k, dt):
        capi.check(lib.ttmi_gemm_describe(m, n, k, capi.EPI_BIAS_ACT, ctypes.byref(args), dt, buf, 64))
        return buf.value.decode()

    for dt in (capi.F16, capi.BF16):
        for m, n, k in ((128, 16384, 4096), (128, 8192, 2048), (128, 768, 3072), (100, 768, 768), (128, 256, 1024)):
            assert variant(m, n, k, dt).startswith("dma"), (m, n, k)
    for m, n, k in ((128, 8192, 512), (128, 16384, 4096)):
        assert "_splitk" not in variant(m, n, k, capi.F32), (m, n, k)


def test_picking_a_tile_costs_less_than_a_microsecond():
    """The selection of a ring tile and its K slices runs on the host in front of every launch, and the small cases are bound by
    the host.  Through ttmi_gemm_describe, whose own cost a plain product of the same size shares: 16 slices of at most eight
    tiles at some 3 ns each are 0.4 us; twice that is allowed (a plain search of all of them, run twice, takes 2.5 us more)."""
    import ctypes
    import time
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)
    args = ctypes.byref(capi.EpilogueArgs())

    def best_us(m, n, k, dt, epi):
        best = 1e9
        for _ in range(60):
            start = time.perf_counter()
            for _ in range(200):
                lib.ttmi_gemm_describe(m, n, k, epi, args, dt, buf, 64)
            best = min(best, (time.perf_counter() - start) / 200 * 1e6)
        return best

    for m, n, k, dt in ((128, 768, 3072, capi.F32), (896, 768, 3072, capi.F32), (8, 768, 3072, capi.F16), (128, 768, 3072, capi.F16)):
        assert best_us(m, n, k, dt, capi.EPI_BIAS) < best_us(m, n, k, dt, capi.EPI_NONE) + 0.8, (m, n, k, dt)


def test_kernel_forms_that_write_through_contain_such_stores(tmp_path):
    """The large tiles are compiled twice, with output stores that stay in L2 and with ones that go through it (the sc1 bit of a
    store): each form has the stores of its name, whatever epilogue it is for."""
    import re
    import shutil
    objdump = shutil.which("llvm-objdump", path=os.pathsep.join([os.environ.get("PATH", ""), "/opt/rocm/llvm/bin"]))
    if objdump is None:
        pytest.skip("no llvm-objdump")
    os.symlink(capi.LIB_PATH, tmp_path / "lib.so")
    subprocess.run([objdump, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    stores = {}
    for bundle in sorted(tmp_path.glob("lib.so.*gfx950")):
        if b"gemm_w4_kernel" not in bundle.read_bytes():
            continue
        text = subprocess.run([objdump, "-d", "-C", bundle], check=True, capture_output=True, text=True).stdout
        for name, body in re.findall(r"^[0-9a-f]+ <(void ttmi::gemm_w4_kernel<.*)>:\n((?:.+\n)+)", text, flags=re.M):
            found = re.findall(r"\b(?:buffer|global|flat)_store_dwordx4\b.*", body)
            stores[name] = (len(found), sum(" sc1" in s for s in found))
    assert len(stores) >= 40
    for name, (count, through) in stores.items():
        assert count > 0, name
        if re.search(r", true>\(", name):  # the last parameter
            assert through > 0, name
        else:
            assert through == 0, name


@pytest.mark.parametrize("layers,width,ffn,element,lens,reads", [
    # base: the tensors of some 1100 tokens push its weights out, those of one or a few sequences do not
    (12, 768, 3072, 2, 512, False), (12, 768, 3072, 2, 1000, False), (12, 768, 3072, 2, 1152, True), (12, 768, 3072, 2, 1536, True), (12, 768, 3072, 2, 2000, True),
    (13, 768, 3072, 2, 600, False), (13, 768, 3072, 2, 500, False), (13, 768, 3072, 2, 768, True), (14, 768, 3072, 2, 300, False), (17, 768, 1536, 2, 2048, True),
    # weights of 176 to 201 MB whose tensors add up to less than 200 MiB: narrower and wider layers, fp32
    (29, 512, 2048, 2, 1536, False), (32, 512, 2048, 2, 128, False), (7, 1024, 4096, 2, 768, False), (5, 1280, 5120, 2, 128, False), (5, 1280, 5120, 2, 256, False),
    (4, 1280, 5120, 2, 1024, False), (6, 768, 3072, 4, 512, False), (6, 768, 3072, 4, 600, False), (14, 512, 2048, 4, 768, False),
    # beyond: always, but for up to 32 rows
    (24, 1024, 4096, 2, 33, True), (24, 1024, 4096, 2, 32, False), (12, 768, 3072, 4, 128, True), (5, 1280, 5120, 2, 768, True), (6, 768, 3072, 4, 1024, True)])
def test_weights_are_read_ahead_where_they_leave_the_cache(layers, width, ffn, element, lens, reads):
    """The attention of a layer reads the following weights ahead where that was measured to gain: each line's time with and without
    stands at the rule."""
    from turbotransformers_amd import cxx
    weights = layers * (4 * width * width + 2 * width * ffn) * element
    assert cxx.weights_leave_cache(weights, lens, width, ffn, element) is reads


def test_the_layers_product_with_activation_has_no_named_form():
    """ttmi_gemm_bias_act takes the ring tiles where ttmi_gemm_fused keeps the form that ttmi_gemm_describe names for GELU over 65 to 128
    rows, and its own description says so; elsewhere the two run the same."""
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)
    args = capi.EpilogueArgs()

    def variants(m, n, k, act, dt):
        args.act = act
        capi.check(lib.ttmi_gemm_describe(m, n, k, capi.EPI_BIAS_ACT, ctypes.byref(args), dt, buf, 64))
        fused = buf.value.decode()
        capi.check(lib.ttmi_gemm_bias_act_describe(m, n, k, act, dt, buf, 64))
        return fused, buf.value.decode()

    for m in (65, 97, 128):
        for dt in (capi.F16, capi.BF16):
            assert variants(m, 3072, 768, capi.ACT_GELU, dt)[0] == "wave1w_32x32"
            assert variants(m, 3072, 768, capi.ACT_GELU, dt)[1].startswith("dma")
        assert "_splitk" in variants(m, 3072, 768, capi.ACT_GELU, capi.F32)[0]
        one, other = variants(m, 3072, 768, capi.ACT_GELU, capi.F32)
        assert other.startswith("dma") and "_splitk" not in other
    for m in (1, 10, 64, 129, 2000, 32768):
        for dt in (capi.F16, capi.BF16, capi.F32, capi.F32_PACKED):
            for act in (capi.ACT_GELU, capi.ACT_RELU):
                one, other = variants(m, 3072, 768, act, dt)
                assert one == other, (m, dt, act)
    one, other = variants(128, 3072, 768, capi.ACT_RELU, capi.F16)
    assert one == other
    assert lib.ttmi_gemm_bias_act_describe(128, 3072, 768, capi.ACT_GELU, capi.F16, buf, 4) != 0  # too small for the answer
    assert lib.ttmi_gemm_bias_act_describe(128, 3072, 768, 99, capi.F16, buf, 64) != 0


def test_encoder_stacks_as_one_launch_have_inner_rows_as_wide_as_the_hidden_ones():
    """The items of a step write the residual of the columns of their own number: with fewer items than column blocks some would
    never be written."""
    lib = capi.load()
    size = ctypes.c_int64(7)
    for heads, ffn, built in [(12, 768, True), (12, 704, False), (12, 512, False), (12, 256, False), (16, 1024, True), (16, 960, False), (4, 256, True),
                              (4, 192, False), (12, 4096, True)]:
        for dtype in (capi.F16, capi.BF16):
            capi.check(lib.ttmi_encoder_chain_workspace(2, 8, heads, heads * 64, ffn, dtype, ctypes.addressof(size)))
            assert (size.value > 0) == built, (heads, ffn)


_WALK = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "chain_walk.h"
// Workgroups of a chain, one round of waiting or one item a turn, in a random order; `resident` of them run at a time.  An item reads what the items of
// the step before have written, which arrives up to three turns later; one of them (lost_step, lost_item) reads something that nobody writes.
int main(int argc, char** argv) {
  const int workgroups = atoi(argv[1]), resident = atoi(argv[2]), resumes = atoi(argv[3]), lost_step = atoi(argv[4]), lost_item = atoi(argv[5]);
  srand(atoi(argv[6]));
  const std::vector<int> counts = {5, 2, 7, 2, 5, 2, 7, 2, 1};
  const int steps = (int)counts.size();
  std::vector<std::vector<long>> written(steps);
  for (int s = 0; s < steps; ++s) written[s].assign(counts[s], -1);
  struct Workgroup {
    ttmi::ChainWalk walk;
    int seen = 0;
    bool over = false, gave_up = false;
  };
  std::vector<Workgroup> all(workgroups);
  auto items = [&](int s) { return counts[s]; };
  long turns = 0;
  int started = 0, over = 0, gave_up = 0;
  std::vector<int> running;
  while (over < workgroups) {
    while ((int)running.size() < resident && started < workgroups) {
      const int me = started++;
      Workgroup& w = all[me];
      auto first_item = [&](int s) { return (me + s) % workgroups; };
      w.walk.item = me - workgroups;
      w.walk.forward(workgroups, steps, items, first_item);
      if (w.walk.step >= steps) ++over;
      else running.push_back(me);
    }
    if (running.empty()) continue;
    const int at = rand() % (int)running.size(), me = running[at];
    Workgroup& w = all[me];
    auto first_item = [&](int s) { return (me + s) % workgroups; };
    const int s = w.walk.step;
    bool there = !(s == lost_step && w.walk.item == lost_item);
    for (int i = 0; s > 0 && i < counts[s - 1]; ++i) there = there && written[s - 1][i] >= 0 && written[s - 1][i] <= turns;
    bool ends = false;
    if (there) {
      if (written[s][w.walk.item] < 0) written[s][w.walk.item] = turns + rand() % 4;
      if (!w.walk.solo()) w.seen = s;
      w.walk.executed(workgroups, steps, items, first_item);
      ends = w.walk.step >= steps;
    } else if (!w.walk.late(resumes ? w.seen : 0)) {
      ends = true, ++gave_up;
    }
    if (ends) running.erase(running.begin() + at), ++over;
    if (++turns > 20L * 1000 * 1000) return 3;
  }
  bool complete = true;
  for (const auto& step : written)
    for (long x : step) complete = complete && x >= 0;
  printf("%d %d\n", gave_up, (int)complete);
  return 0;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    folder = tmp_path_factory.mktemp("walk")
    source, program = folder / "walk.cpp", folder / "walk"
    source.write_text(_WALK)
    device = os.path.join(os.path.dirname(capi.HEADER), "..", "turbotransformers_amd", "csrc", "device")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", device, str(source), "-o", str(program)], check=True)

    def run(*args):
        done = subprocess.run([str(program)] + [str(a) for a in args], capture_output=True, text=True, timeout=100)
        assert done.returncode == 0, (args, done.returncode)  # (3: it would not have ended)
        return [int(x) for x in done.stdout.split()]

    return run


def test_workgroups_of_a_launch_add_up_to_one_unit(tmp_path):
    """Whoever has not added its share yet, of any number of workgroups, finds as many whole units as at the launch's start; at its end there is
    one more, also where 32 bits overflow."""
    (tmp_path / "share.cpp").write_text(r"""
#include <initializer_list>
#include "chain_walk.h"
int main() {
  using namespace ttmi;
  for (uint32_t g = 1; g <= (uint32_t)kChainMostWorkgroups; g = g < 600 ? g + 1 : g * 2 - g / 3)
    for (uint32_t start : {0u, 5 * kLaunchUnit, 0u - kLaunchUnit}) {
      uint32_t count = start;
      for (uint32_t r = 0; r < g; ++r) {
        if (count / kLaunchUnit != start / kLaunchUnit || launch_share(r, g) == 0) return 1;
        count += launch_share(r, g);
      }
      if (count != start + kLaunchUnit) return 2;
    }
  uint32_t sum = 0;
  for (int r = 0; r < kChainMostWorkgroups; ++r) sum += launch_share(r, kChainMostWorkgroups);
  return sum == kLaunchUnit ? 0 : 3;
}
""")
    device = os.path.join(os.path.dirname(capi.HEADER), "..", "turbotransformers_amd", "csrc", "device")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", device, str(tmp_path / "share.cpp"), "-o", str(tmp_path / "share")], check=True)
    assert subprocess.run([str(tmp_path / "share")], timeout=60).returncode == 0


@pytest.mark.parametrize("workgroups,resident", [(1, 1), (3, 1), (7, 2), (7, 7), (12, 5)])
@pytest.mark.parametrize("resumes", [0, 1])
def test_a_chain_of_steps_ends_whoever_is_resident(walk, workgroups, resident, resumes):
    """Workgroups that wait in vain compute what they miss: nobody gives up, and everything is written.  resumes: from the last step whose inputs
    were seen (encoder layers) or from the first (a decoder's blocks)."""
    for seed in range(20):
        assert walk(workgroups, resident, resumes, -1, -1, seed) == [0, 1]


@pytest.mark.parametrize("workgroups,resident", [(1, 1), (3, 1), (7, 2), (7, 7), (12, 5)])
@pytest.mark.parametrize("resumes", [0, 1])
@pytest.mark.parametrize("lost", [(0, 3), (3, 1), (6, 6), (8, 0)])
def test_a_chain_whose_item_reads_what_nobody_writes_ends_too(walk, workgroups, resident, resumes, lost):
    """A mistake in a shape or a rule is an error, not a launch that never ends."""
    gave_up, complete = walk(workgroups, resident, resumes, *lost, 1)
    assert gave_up > 0 and not complete


def _refused(rc):
    return rc == -1 and b"must share no memory" in capi.load().ttmi_last_error()


@pytest.mark.parametrize("dtype", [capi.F16, capi.BF16])
def test_a_stack_as_one_launch_refuses_a_result_over_what_it_reads(dtype):
    """Addresses only: the check stands in front of every device call.  A workgroup that starts late reads its input late."""
    lib = capi.load()
    rows, hidden = 10, 768
    weights = (ctypes.c_void_p * 12)(*[0x10000 * (i + 1) for i in range(12)])
    x, x32, mask, out, out32, memory = (0x40000000 + 0x100000 * i for i in range(6))
    good = dict(x=x, x32=x32, mask=mask, out=out, out32=out32)

    def call(**places):
        p = dict(good, **places)
        return lib.ttmi_encoder_chain(ctypes.addressof(weights), p["x"], p["x32"], p["mask"], p["out"], p["out32"], memory, 3, 1, 1, rows, 12, hidden, 3072, 1e-12,
                                      dtype, 0, 0, None)

    assert not _refused(call())  # (stopped by the turn, 3)
    assert not _refused(call(out=x + rows * hidden * 2)) and not _refused(call(x32=None, mask=None, out32=None))
    for places in (dict(out=x), dict(out=x + rows * hidden * 2 - 16), dict(out=x32 + 16), dict(out=mask), dict(out32=x), dict(out32=x32), dict(out32=mask - 16),
                   dict(out32=out), dict(out32=out + rows * hidden * 2 - 16)):
        assert _refused(call(**places)), places


@pytest.mark.parametrize("grows", [True, False])
def test_a_decoder_block_as_one_launch_refuses_results_over_what_it_reads_or_each_other(grows):
    lib = capi.load()
    rows, heads, hidden, keys = 8, 12, 768, 41
    names = ["x", "gamma", "beta", "w_in", "b_in", "w_out", "b_out", "k_past", "v_past", "k_out", "v_out", "mask", "probs", "out"]
    good = {n: 0x40000000 + 0x1000000 * i for i, n in enumerate(names)}
    if not grows:
        good.update(k_out=None, v_out=None)

    def call(**places):
        p = dict(good, **places)
        return lib.ttmi_decoder_attention(p["x"], p["gamma"], p["beta"], 1e-6, p["w_in"], p["b_in"], p["w_out"], p["b_out"], p["k_past"], p["v_past"], p["k_out"],
                                          p["v_out"], p["mask"], p["probs"], p["out"], 0x10000, 3, rows, heads, hidden, keys, 0.125, capi.F16, 0, 0, None)

    assert not _refused(call()) and not _refused(call(mask=None))
    places = [dict(out=good["x"]), dict(out=good["x"] + rows * hidden * 2 - 16), dict(out=good["probs"]), dict(probs=good["x"] + 16), dict(probs=good["mask"]),
              dict(out=good["v_past"] + 16), dict(probs=good["k_past"])]
    if grows:
        places += [dict(k_out=good["k_past"]), dict(v_out=good["k_past"]), dict(k_out=good["v_out"]), dict(out=good["k_out"]), dict(probs=good["v_out"] + 2)]
    for p in places:
        assert _refused(call(**p)), p

    def block(x, out):
        return lib.ttmi_decoder_feed_forward(x, 0x20000, 0x30000, 1e-12, 0x1000000, 0x40000, 0x2000000, 0x50000, out, 0x10000, 3, rows, hidden, 3072, capi.F16, 0, 0,
                                             None)

    assert not _refused(block(0x60000, 0x80000)) and _refused(block(0x60000, 0x60000)) and _refused(block(0x60000, 0x60010))


@pytest.mark.parametrize("hidden,inner,element,one", [(256, 1024, 2, True), (1024, 4096, 2, True), (64, 64, 2, True), (768, 3072, 4, True), (1024, 3072, 4, True),
                                                      (1024, 2048, 4, False), (768, 768, 4, False), (512, 2048, 4, False), (256, 3072, 4, False), (64, 256, 4, False)])
def test_feed_forward_blocks_run_as_one_launch_where_that_was_measured_to_gain(hidden, inner, element, one):
    from turbotransformers_amd import cxx
    assert cxx.feed_forward_runs_as_one_launch(hidden, inner, element) is one


@pytest.mark.parametrize("batch,seq,narrow", [(20, 100, True), (20, 200, True), (12, 460, True), (12, 500, True), (18, 464, False), (20, 440, False), (20, 480, False),
                                              (24, 500, False), (32, 500, False), (20, 128, False), (16, 300, False)])
def test_fp32_head_splits_take_the_tile_of_their_own_up_to_three_rounds(batch, seq, narrow):
    """96 x 192 where 128 x 192 would leave a quarter of the compute units idle; beyond three rounds of workgroups that was measured to lose."""
    lib = capi.load()
    buf = ctypes.create_string_buffer(64)
    args = capi.EpilogueArgs(bias=4096, q=4096, k=4096, v=4096, seq=seq, heads=12, head_dim=64, v_seq_pitch=(seq + 7) // 8 * 8)
    capi.check(lib.ttmi_gemm_describe(batch * seq, 2304, 768, capi.EPI_QKV_SPLIT, ctypes.byref(args), capi.F32_PACKED, buf, 64))
    assert ("96x192" in buf.value.decode()) == narrow, buf.value
