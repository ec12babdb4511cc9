"""Pinned host memory and the copies of the caller's arrays, without a GPU: a C
program that brings its own runtime (device memory is malloc, kernels do nothing)
counts what the library asks of it."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

LIB_DIR = os.path.join(ROOT, "amr-demo_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

pytestmark = pytest.mark.skipif(shutil.which("gcc") is None or not os.path.isdir(os.path.join(ROCM, "include")),
                                reason="gcc or the HIP headers absent")

RUNTIME = r"""
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "amr_hip.h"
#include "amr_tagger.h"

/* what the library asked for */
static int host_allocs, copies, launches, copies_at_launch, cus = 256;
static dim3 grid;
static const void *copy_src[1024];
static void *copy_dst[1024];
static size_t copy_bytes[1024];
/* the caller's pinned array */
static char *mine;
static size_t mine_bytes;
static int reads_mine;      /* a copy from it may be under way */
static hipError_t launch_error = hipSuccess;

hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) { (void)flags; ++host_allocs; *p = calloc(n, 1); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { (void)k; memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    (void)k; (void)st;
    copy_src[copies % 1024] = s;
    copy_bytes[copies % 1024] = n;
    copy_dst[copies++ % 1024] = d;
    if (mine && (const char *)s >= mine && (const char *)s < mine + mine_bytes) reads_mine = 1;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    memset(a, 0, sizeof(*a));
    a->type = hipMemoryTypeUnregistered;
    if (mine && (const char *)p >= mine && (const char *)p < mine + mine_bytes) {
        a->type = hipMemoryTypeHost;
        a->hostPointer = (void *)p;
        a->devicePointer = (void *)p;
    }
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return launch_error; }
const char *hipGetErrorString(hipError_t e) { (void)e; return "error"; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) { (void)a; (void)d; *v = cus; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned f) { (void)f; *s = (hipStream_t)&copies; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; reads_mine = 0; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { (void)f; *e = (hipEvent_t)&launches; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t n, hipStream_t s) { (void)b; (void)n; (void)s; grid = g; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s)
{
    memset(g, 0, sizeof(*g)); memset(b, 0, sizeof(*b)); *n = 0; *s = 0;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t n, hipStream_t s)
{
    (void)f; (void)g; (void)b; (void)a; (void)n; (void)s;
    ++launches;
    copies_at_launch = copies;
    return hipSuccess;
}

#define MUST(x) do { int rc_ = (x); if (rc_) { printf("%s: %d %s\n", #x, rc_, amrgpu_last_error()); return 1; } } while (0)
#define HOLDS(x) do { if (!(x)) { printf("line %d: %s does not hold\n", __LINE__, #x); return 1; } } while (0)

/* nq quadrants of 2x2 cells with a wall on every side, zero state */
static int set_up_n(amrgpu_ctx *c, int nq, int ninst)
{
    int *ci = malloc(sizeof(int) * 3 * (size_t)nq), *fi = calloc((size_t)nq * 44, sizeof(int)), rc;
    double *u = calloc((size_t)nq * 16, sizeof(double));
    amrgpu_inst_t *in = calloc((size_t)ninst, sizeof(*in));
    for (int k = 0; k < ninst; ++k) { in[k].h_base = 1.0; in[k].cfl = 0.3; in[k].dt_cap = 1.0; }
    for (int q = 0; q < nq; ++q) {
        ci[3 * q] = 0; ci[3 * q + 1] = 5; ci[3 * q + 2] = 16 * q;
        for (int s = 0; s < 4; ++s) { int *f = fi + 11 * (4 * (size_t)q + s); f[0] = 1; f[1] = s; f[2] = q; }
    }
    rc = amrgpu_setup(c, 2, 3, ninst, in, nq, ci, NULL, 4 * nq, fi, NULL, u);
    free(ci); free(fi); free(u); free(in);
    return rc;
}
static int set_up(amrgpu_ctx *c, int nq) { return set_up_n(c, nq, 1); }
/* the same mesh again through a remesh */
static int remesh(amrgpu_ctx *c, int nq)
{
    int *lev = calloc((size_t)nq, sizeof(int)), *nbr = malloc(sizeof(int) * 8 * (size_t)nq), *src = calloc((size_t)nq, sizeof(int)), rc;
    for (size_t k = 0; k < 8 * (size_t)nq; ++k) nbr[k] = -1;
    rc = amrgpu_remesh_nbr(c, nq, lev, NULL, nbr, src);
    free(lev); free(nbr); free(src);
    return rc;
}
"""


def run(tmp_path, body):
    """the statements `body` of a program with that runtime; 0 is success"""
    src, exe = tmp_path / "t.c", tmp_path / "t"
    src.write_text(RUNTIME + "int main(void)\n{\n" + body + "    return 0;\n}\n")
    r = subprocess.run(["gcc", "-std=gnu11", "-O1", "-Wall", "-Wno-unused-function", f"-I{ROOT}/include",
                        f"-I{ROCM}/include", str(src), f"-L{LIB_DIR}", "-lamrhip", f"-Wl,-rpath,{LIB_DIR}",
                        "-rdynamic", f"-Wl,-rpath-link,{ROCM}/lib", "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("nq", [1, 100001, 1000000, 1500000])
def test_no_pinned_allocation_by_repeated_setups_and_remeshes(tmp_path, nq):
    """whatever the mesh's size, the pinned area its tables pass through is
    made once per context"""
    run(tmp_path, f"""
    amrgpu_ctx *c = amrgpu_create();
    for (int k = 0; k < 2; ++k) {{ MUST(set_up(c, {nq})); MUST(remesh(c, {nq})); }}
    const int before = host_allocs;
    for (int k = 0; k < 2; ++k) {{ MUST(set_up(c, {nq})); MUST(remesh(c, {nq})); }}
    HOLDS(host_allocs == before);
    amrgpu_destroy(c);
""")


@pytest.mark.parametrize("faces", [0, 1])
@pytest.mark.parametrize("nq", [1, 32767, 32768, 100001])
def test_a_remesh_uploads_the_table_and_remaps_a_large_mesh_ahead_of_it(tmp_path, nq, faces):
    """the device holds the face table, levels, instance ids and source map of
    the new mesh, one after the other; from 32768 quadrants on the remap is
    launched ahead of the table's copy: it runs while the host packs the table"""
    run(tmp_path, f"""
    enum {{ nq = {nq} }};
    static int lev[nq], inst[nq], nbr[8 * nq], src[nq], ci[3 * nq], fi[44 * nq];
    for (int q = 0; q < nq; ++q) {{
        lev[q] = q % 30; inst[q] = q % 3; src[q] = nq - 1 - q;
        ci[3 * q + 1] = lev[q]; ci[3 * q + 2] = 16 * q;
        for (int s = 0; s < 4; ++s) {{
            int *f = fi + 11 * (4 * q + s);
            f[0] = 1; f[1] = s; f[2] = q;
            nbr[8 * q + 2 * s] = {faces} ? -1 : (q * 7 + s) % nq;
            nbr[8 * q + 2 * s + 1] = -1;
        }}
    }}
    amrgpu_ctx *c = amrgpu_create();
    MUST(set_up_n(c, nq, 3));
    if ({faces}) MUST(amrgpu_remesh(c, nq, ci, inst, 4 * nq, fi, src));
    else MUST(amrgpu_remesh_nbr(c, nq, lev, inst, nbr, src));
    const int *d, *p;
    MUST(amrgpu_device_state(c, NULL, &d, NULL, NULL, NULL));
    p = d;
    HOLDS(memcmp(p, nbr, sizeof(nbr)) == 0); p += 8 * nq;
    HOLDS(memcmp(p, lev, sizeof(lev)) == 0); p += nq;
    HOLDS(memcmp(p, inst, sizeof(inst)) == 0); p += nq;
    HOLDS(memcmp(p, src, sizeof(src)) == 0);
    HOLDS(nq < 3 || (copies > copies_at_launch) == (nq >= 32768));    /* (every instance has quadrants) */
    amrgpu_destroy(c);
""")


def test_the_small_results_keep_no_transfer_chunks(tmp_path):
    """a context's small results take a block of their size, not the transfer
    chunks that wait for the next copy"""
    run(tmp_path, """
    amrgpu_ctx *c = amrgpu_create();
    static double t, dt, u[16 * 256];
    MUST(set_up(c, 256));
    MUST(amrgpu_get_time(c, &t, &dt));
    const int before = host_allocs;
    for (int k = 0; k < 3; ++k) { MUST(amrgpu_upload_soln(c, u)); MUST(amrgpu_get_time(c, &t, &dt)); }
    HOLDS(host_allocs == before);
    amrgpu_destroy(c);
""")


def test_the_pool_keeps_what_was_given_back_last(tmp_path):
    """pinned blocks of sizes that nobody asks for any more do not keep the pool
    full: contexts that come and go with the same mesh make no new ones"""
    run(tmp_path, """
    int before = 0;
    for (int nq = 150000; nq < 600000; nq += nq / 3) {       /* one size after the other, each larger than the last block */
        amrgpu_ctx *c = amrgpu_create();
        MUST(set_up(c, nq));
        amrgpu_destroy(c);
    }
    for (int k = 0; k < 4; ++k) {
        amrgpu_ctx *c = amrgpu_create();
        MUST(set_up(c, 600000));
        amrgpu_destroy(c);
        if (k == 1) before = host_allocs;
    }
    HOLDS(host_allocs == before);
""")


def test_the_callers_pinned_arrays_go_to_the_device_as_they_are(tmp_path):
    """no pass through the library's own chunks, in either direction"""
    run(tmp_path, """
    enum { nq = 4096, bytes = nq * 16 * 8 };
    mine = calloc(bytes, 1);
    mine_bytes = bytes;
    double *u = (double *)mine;
    amrgpu_ctx *c = amrgpu_create();
    MUST(set_up(c, nq));
    int k = copies;
    MUST(amrgpu_upload_soln(c, u));
    HOLDS(copies == k + 1 && copy_src[k] == u && copy_bytes[k] == bytes);
    k = copies;
    MUST(amrgpu_download_soln(c, u));
    HOLDS(copies == k + 1 && copy_dst[k] == u && copy_bytes[k] == bytes);
    k = copies;
    MUST(amrgpu_rhs(c, u));
    HOLDS(copies == k + 1 && copy_dst[k] == u && copy_bytes[k] == bytes);
    k = copies;
    MUST(amrgpu_indicator(c, u));
    HOLDS(copies == k + 1 && copy_dst[k] == u && copy_bytes[k] == nq * 8);
    k = copies;
    MUST(amrgpu_set_origins(c, u));
    HOLDS(copies == k + 1 && copy_src[k] == u && copy_bytes[k] == nq * 16);
    amrgpu_destroy(c);
""")


@pytest.mark.parametrize("nq,parts", [(1, 1), (16384, 1), (16385, 2), (100001, 7), (196608, 12), (196609, 1), (300000, 1)])
def test_an_upload_arrives_whole(tmp_path, nq, parts):
    """through the library's chunks of 2 MB up to 24 MB, left to the runtime beyond"""
    run(tmp_path, f"""
    const size_t bytes = {nq} * 128ul;
    unsigned char *u = malloc(bytes);
    for (size_t i = 0; i < bytes; ++i) u[i] = (unsigned char)(i * 2654435761u >> 13);
    amrgpu_ctx *c = amrgpu_create();
    MUST(set_up(c, {nq}));
    const int k = copies;
    MUST(amrgpu_upload_soln(c, (double *)u));
    HOLDS(copies == k + {parts} && (copy_src[k] == u) == (bytes > 24 << 20) && memcmp(copy_dst[k], u, bytes) == 0);
    amrgpu_destroy(c);
""")


@pytest.mark.parametrize("nq,parts", [(1, 1), (131072, 1), (131073, 2), (400000, 4)])
def test_the_corners_may_change_once_they_are_set(tmp_path, nq, parts):
    """they always pass through the chunks of 2 MB"""
    run(tmp_path, f"""
    const size_t bytes = {nq} * 16ul;
    unsigned char *u = malloc(bytes);
    for (size_t i = 0; i < bytes; ++i) u[i] = (unsigned char)(i * 2654435761u >> 13);
    amrgpu_ctx *c = amrgpu_create();
    MUST(set_up(c, {nq}));
    const int k = copies;
    MUST(amrgpu_set_origins(c, (double *)u));
    HOLDS(copies == k + {parts} && copy_src[k] != u && memcmp(copy_dst[k], u, bytes) == 0);
    amrgpu_destroy(c);
""")


@pytest.mark.parametrize("n", [2, 4, 8, 16])
def test_every_tile_launches_every_stage(tmp_path, n):
    """a step is the scheme's stages, after the dt kernel where the first stage
    does not form dt itself: no tile leaves one out"""
    run(tmp_path, f"""
    enum {{ nq = 4, n = {n} }};
    static int ci[3 * nq], fi[44 * nq], ppb[64], minw[64], design[64];
    static double u[4 * n * n * nq], rn;
    amrgpu_inst_t in;
    memset(&in, 0, sizeof(in));
    in.h_base = 1.0; in.cfl = 0.3; in.dt_cap = 1.0;
    for (int q = 0; q < nq; ++q) {{
        ci[3 * q + 2] = 4 * n * n * q;
        for (int s = 0; s < 4; ++s) {{ int *f = fi + 11 * (4 * q + s); f[0] = 1; f[1] = s; f[2] = q; }}
    }}
    const int tiles = amrgpu_tile_variants(n, ppb, minw, design, 64);
    HOLDS(tiles > 0 && tiles <= 64);
    for (int scheme = 1; scheme <= 5; ++scheme)
        for (int k = 0; k < tiles; ++k) {{
            amrgpu_ctx *c = amrgpu_create();
            MUST(amrgpu_setup(c, n, scheme, 1, &in, nq, ci, NULL, 4 * nq, fi, NULL, u));
            MUST(amrgpu_set_tile(c, ppb[k], minw[k], design[k]));
            const int l0 = launches;
            MUST(amrgpu_run(c, 1, 0, &rn));
            const int l1 = launches;
            MUST(amrgpu_run(c, 3, 0, &rn));
            const int step2 = (launches - l1) - (l1 - l0);       /* of two steps */
            HOLDS(step2 == 2 * scheme || step2 == 2 * (scheme + 1));
            amrgpu_destroy(c);
        }}
""")


@pytest.mark.parametrize("cus", [32, 256, 304])
def test_limits_follow_the_devices_compute_units(tmp_path, cus):
    """4x4 patches take four rows a step while their waves fit the device, 12 of
    4 patches a CU, and the tagger's inference two workgroups a CU at most"""
    run(tmp_path, f"""
    enum {{ most = {cus} * 48 + 1, n = 4 }};
    static int ci[3 * most], fi[44 * most];
    cus = {cus};
    amrgpu_inst_t in;
    memset(&in, 0, sizeof(in));
    in.h_base = 1.0; in.cfl = 0.3; in.dt_cap = 1.0;
    for (int q = 0; q < most; ++q) {{
        ci[3 * q + 2] = 4 * n * n * q;
        for (int s = 0; s < 4; ++s) {{ int *f = fi + 11 * (4 * q + s); f[0] = 1; f[1] = s; f[2] = q; }}
    }}
    amrgpu_ctx *c = amrgpu_create();
    for (int nq = most - 1; nq <= most; ++nq) {{
        int ppb, minw, design;
        MUST(amrgpu_setup(c, n, 3, 1, &in, nq, ci, NULL, 4 * nq, fi, NULL, NULL));
        MUST(amrgpu_get_tile(c, &ppb, &minw, &design));
        HOLDS(design == 3 && ppb == (nq < most ? 4 : 8));
    }}
    amrgpu_destroy(c);
    enum {{ rows = 2 * {cus} * 128 }};
    amr_mlp_t *m = amr_mlp_create(1);
    unsigned short *X = calloc((rows + 1) * (size_t)AMR_MLP_NIN, 2);
    float *z = calloc((rows + 1) * 3ul, sizeof(float));
    MUST(amr_mlp_forward(m, X, rows - 128, z));
    HOLDS(grid.x == 2 * {cus} - 1);
    MUST(amr_mlp_forward(m, X, rows + 1, z));
    HOLDS(grid.x == 2 * {cus});
    amr_mlp_destroy(m);
""")


def test_no_call_returns_while_the_callers_pinned_array_is_read(tmp_path):
    """not where it fails after the copy has been started, either"""
    run(tmp_path, """
    enum { nq = 64, bytes = nq * 16 * 8 };
    static int ci[3 * nq], fi[44 * nq];
    static double rhs[nq * 16];
    for (int q = 0; q < nq; ++q) {
        ci[3 * q + 2] = 16 * q;
        for (int s = 0; s < 4; ++s) { int *f = fi + 11 * (4 * q + s); f[0] = 1; f[1] = s; f[2] = q; }
    }
    mine = calloc(bytes, 1);
    mine_bytes = bytes;
    double *u = (double *)mine, dt = 1.0;
    amrgpu_ctx *c = amrgpu_create();
    MUST(set_up(c, nq));
    MUST(amrgpu_upload_soln(c, u));
    HOLDS(!reads_mine);
    MUST(amrgpu_set_origins(c, u));
    HOLDS(!reads_mine);
    launch_error = hipErrorInvalidValue;
    HOLDS(amrgpu_upload_soln(c, u) != 0 && !reads_mine);
    launch_error = hipSuccess;
    amrgpu_inst_t in;
    memset(&in, 0, sizeof(in));
    in.h_base = 1.0; in.cfl = 0.3; in.dt_cap = 1.0;
    MUST(amrgpu_setup(c, 2, 3, 1, &in, nq, ci, NULL, 4 * nq, fi, NULL, u));
    HOLDS(!reads_mine);
    launch_error = hipErrorInvalidValue;
    HOLDS(amrgpu_setup(c, 2, 3, 1, &in, nq, ci, NULL, 4 * nq, fi, NULL, u) != 0 && !reads_mine);
    launch_error = hipSuccess;
    amrgpu_destroy(c);
    /* the calls on host arrays, with walls that need the corners that are not given */
    physics_gpu_params_t p;
    physics_gpu_get_params(&p);
    p.dim = 2; p.nfields = 4; p.nelem_subgrid = 2; p.time_scheme = 3; p.time_steps = 10; p.dt = 1.0; p.cfl = 0.3;
    p.coarse_grid_h = 1.0;
    for (int s = 0; s < 4; ++s) p.bc[s] = AMRGPU_BC_SHOCK_TOP;
    physics_gpu_set_params(&p);
    int dim = 2, nf = 4, n = 2, ncell = nq, nface = 4 * nq, dof = nq * 16, z = 0, one = 1, istep = 0;
    double sec = 0.0;
    HOLDS(physics_rhs_structured_gpu(&dim, &nf, &n, &ncell, ci, NULL, &nface, fi, &dof, u, rhs) != 0 && !reads_mine);
    HOLDS(physics_go_gpu(&dim, &z, &nf, &n, &ncell, &z, &nface, &dof, ci, fi, &z, &z, &z, &z, &z, NULL, u, &istep, &z, &z, &z,
                         &one, NULL, &sec, &sec, &sec) != 0 && !reads_mine);
    MUST(physics_time_step_gpu(&dim, &nf, &n, &ncell, ci, NULL, u, &dt));
    HOLDS(!reads_mine);
""")
