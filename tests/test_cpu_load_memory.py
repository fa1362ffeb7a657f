"""The loader when device memory runs out, on the CPU: the library's host code built against a stand-in device of a
given size whose memory is the heap (allocations, copies and the sizes the device code reports; no kernels)."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

import l3m_amd as A

ROOT = Path(__file__).resolve().parents[1]
DEVICE = r"""
#include <stdlib.h>
#include <string.h>
#include "dev.h"
static size_t room, used;
static int sticky;
void stand_in(size_t bytes) { room = bytes; used = 0; sticky = 0; }
size_t stand_in_used(void) { return used; }
int stand_in_error(void) { return sticky; }
int l3m_dev_init(void) { return 0; }
int l3m_dev_sync(void) { return 0; }
const char *l3m_dev_error(void) { return sticky ? "out of memory" : NULL; }
void l3m_dev_clear_error(void) { sticky = 0; }
void *l3m_dev_alloc(size_t n) {
    if (used + n > room) { sticky = 1; return NULL; }
    size_t *p = calloc(1, n + 16);
    *p = n;
    used += n;
    return p + 2;
}
void l3m_dev_free(void *p) { if (p) { used -= ((size_t *)p)[-2]; free((size_t *)p - 2); } }
int l3m_dev_upload(void *d, const void *s, size_t n) { memcpy(d, s, n); return 0; }
void *l3m_dev_host_alloc(size_t n) { return calloc(1, n); }
void l3m_dev_host_free(void *p) { free(p); }
void *l3m_dev_event_new(void) { return malloc(1); }
void l3m_dev_event_free(void *e) { free(e); }
unsigned l3m_dev_lds_max(void) { return 163840; }
int l3m_dev_cus(void) { return 1; }
int l3m_attention_mode(int a, int b, int c, int d) { return (void)a, (void)b, (void)c, (void)d, 0; }
void l3m_group_layout(int a, int b, int c, int d, l3m_dgroup *g) { (void)a, (void)b, (void)c, (void)d, (void)g; }
void l3m_chunk_layout(int a, int b, l3m_dchunk *c) { (void)a, (void)b, (void)c; }
void l3m_model_layout(l3m_dmodel *m) { (void)m; }
unsigned l3m_lds_attn(int a, int b, int c, int d, const l3m_dgroup *g, int k) { return (void)a, (void)b, (void)c, (void)d, (void)g, (void)k, 1024; }
unsigned l3m_lds_ffn(int a, int b, const l3m_dchunk *c) { return (void)a, (void)b, (void)c, 1024; }
unsigned l3m_lds_head(int a, int b, int c, int d) { return (void)a, (void)b, (void)c, (void)d, 1024; }
int l3m_step_slots(int a, int b) { return (void)a, (void)b, 16; }
int l3m_step_a_dtype(int dt) { return dt == L3M_HIP_Q4_0 ? L3M_HIP_Q8_0 : dt; }
int l3m_prefill_fits(int a, int b, int c, int d) { return (void)a, (void)b, (void)c, (void)d, 1; }
l3m_graphs *l3m_graphs_build(const l3m_dmodel *m, const l3m_dlayer *l) { return (void)m, (void)l, malloc(1); }
void l3m_graphs_free(l3m_graphs *g) { free(g); }
l3m_pfgraphs *l3m_pfgraphs_new(void) { return malloc(1); }
void l3m_pfgraphs_free(l3m_pfgraphs *g) { free(g); }
"""
# what the host code calls after loading
NOT_REACHED = """act_bytes decode_fits decode_launch decode_pair decode_placement decode_timer_collect dev_download dev_download_async
dev_event_record dev_event_wait dev_evict dev_name dev_upload_async graphs_launch k_attend k_gemv k_ltiles k_step_mv ltile_bytes prefill prefill_graph
step_enqueue time_step_kernel""".split()


@pytest.fixture(scope="module")
def device(tmp_path_factory):
    d = tmp_path_factory.mktemp("stand_in")
    (d / "dev.c").write_text(DEVICE)
    (d / "rest.c").write_text("#include <stdlib.h>\n" + "".join(f"void l3m_{n}(void) {{ abort(); }}\n" for n in NOT_REACHED))
    src = ROOT / "l3m_amd" / "csrc"
    so = d / "libstand_in.so"
    subprocess.run(["gcc", "-std=c11", "-O1", "-fPIC", "-shared", "-D_GNU_SOURCE", "-Wl,-Bsymbolic-functions", f"-I{ROOT}/include", f"-I{src}", "-o", str(so),
                    str(d / "dev.c"), str(d / "rest.c"), *(str(src / f"{n}.c") for n in ("api", "file", "gen", "pack", "table", "vocab")), "-lm", "-lpthread"], check=True)
    lib = C.CDLL(str(so))
    lib.stand_in.argtypes, lib.stand_in_used.restype = [C.c_size_t], C.c_size_t
    lib.l3m_load.restype, lib.l3m_load.argtypes = C.c_void_p, [C.c_char_p, C.c_void_p]
    lib.l3m_free.argtypes = [C.c_void_p]
    return lib


@pytest.mark.parametrize("dtype", ["bf16", "q8_0", "q4_0", "mxfp4"])
def test_prompt_copies_do_not_cost_the_model(device, models, monkeypatch, dtype):
    """A device with room for the model but not for the second copy of its matrices that prompts run on: the model
    loads, at every size from its own need up, holds no more than that need where the copy does not fit, leaves no
    error behind, and gives everything back. One byte less than the need is refused."""
    cfg = A.Config("mem", dim=128, n_layers=3, n_heads=4, n_kv_heads=2, ffn_dim=256, vocab=256, ctx=64, dtype=dtype)
    path = str(models.get(cfg, dtype, seed=3)).encode()

    def load(room):
        device.stand_in(room)
        m = device.l3m_load(path, None)
        if not m:
            assert device.stand_in_used() == 0
            return None
        used = device.stand_in_used()
        assert not device.stand_in_error()
        device.l3m_free(m)
        assert device.stand_in_used() == 0
        return used

    monkeypatch.setenv("L3M_PREFILL", "0")
    need = load(1 << 40)
    monkeypatch.setenv("L3M_PREFILL", "1")
    full = load(1 << 40)
    assert full > need
    assert load(need - 1) is None
    for room in [need, *(need + (full - need) * i // 16 for i in range(1, 16)), full - 1]:
        assert load(room) == need, (room, need, full)
    assert load(full) == full
