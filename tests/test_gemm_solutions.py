"""The GPT-2 engine's tuned GEMM solution file, checked on the CPU."""

def test_gemm_solution_file_is_tunableop_csv_with_validators():
    """The engine's GEMM solution file (dfattn.gpt2_step.GEMM_SOLUTIONS, written by tune_gemms) is a
    TunableOp results file: the library validators first, then one row per GEMM shape naming a
    default, hipBLASLt or rocBLAS solution and its measured time; exact fp32 ("float") ops and fast
    fp32 ("tf32") ops keep their own math mode."""
    from dfattn.gpt2_step import GEMM_SOLUTIONS

    rows = [line.rstrip("\n").split(",") for line in open(GEMM_SOLUTIONS) if line.strip()]
    validators = {r[1]: r[2] for r in rows if r[0] == "Validator"}
    for key in ("PT_VERSION", "HIP_VERSION", "HIPBLASLT_VERSION", "ROCBLAS_VERSION", "GCN_ARCH_NAME"):
        assert key in validators, key
    assert validators["GCN_ARCH_NAME"].startswith("gfx950")
    shapes = [r for r in rows if r[0] != "Validator"]
    assert len(shapes) >= 10
    for op, params, solution, ms in shapes:
        assert "_float_" in op or "_tf32_" in op, op
        assert solution == "Default" or solution.startswith(("Gemm_Hipblaslt_", "Gemm_Rocblas_")), solution
        assert float(ms) > 0
    assert len({(r[0], r[1]) for r in shapes}) == len(shapes)


def test_tune_gemms_steps_on_the_library_products(monkeypatch, tmp_path):
    """tune_gemms measures the library's products, so its steps take them at every site, also at sizes
    where the engine's own (dfgpt2_linear_*) are the rule; the library sees no other products. (The tuner
    and the model are stand-ins: the rule and the file's rows are what is checked.)"""
    from types import SimpleNamespace

    import torch

    from dfattn import gpt2_step as G

    engine = G._NativeEngine.__new__(G._NativeEngine)
    small = SimpleNamespace(seq_len=1024, d_model=768, d_ff=3072, fast_gemm=True)
    engine.m, engine.library_products = small, False
    assert engine._own_gemms()
    seen = []
    engine.step = lambda tokens, targets, tuned: seen.append(engine._own_gemms())
    model = SimpleNamespace(vocab_size=10, device="cpu", _engine=engine)
    monkeypatch.setattr(G, "StaticGPT2", lambda **kw: model)
    tuner = SimpleNamespace(is_enabled=lambda: False, tuning_is_enabled=lambda: False, set_filename=lambda f: None,
                            enable=lambda on: None, tuning_enable=lambda on: None,
                            get_validators=lambda: [("GCN_ARCH_NAME", "gfx950")],
                            get_results=lambda: [("GemmTunableOp_tf32_NT", "nt_1_2_3", "Default", 0.5)])
    monkeypatch.setattr(torch.cuda, "tunable", tuner)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    assert G.tune_gemms(tmp_path / "solutions.csv", steps=2) == 1
    assert seen == [False, False]
    assert (tmp_path / "solutions.csv").read_text() == "Validator,GCN_ARCH_NAME,gfx950\nGemmTunableOp_tf32_NT,nt_1_2_3,Default,0.5\n"
