"""The host side of the staged download of logits (qhip_dl_* of qhip_runtime.hip) on
the CPU: a small program takes the HIP calls' place and makes one fail, or leaves
the process no thread to start."""
import os
import subprocess

import pytest

import qlib

PROGRAM = r"""
#include <errno.h>
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static int fail_wait, no_threads;
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = malloc(1); return 0; }
int hipStreamDestroy(void *s) { free(s); return 0; }
int hipStreamSynchronize(void *s) { (void)s; return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { (void)s; (void)e; (void)f; return 0; }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = malloc(n); return *p ? 0 : 2; }
int hipHostFree(void *p) { free(p); return 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = malloc(1); return 0; }
int hipEventDestroy(void *e) { free(e); return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventSynchronize(void *e) { (void)e; return fail_wait ? 999 : 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)k; (void)st; memcpy(d, s, n); return 0; }
const char *hipGetErrorString(int e) { (void)e; return "made to fail"; }
int hipGetLastError(void) { return 0; }

int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x) {
  (void)t; (void)a; (void)f; (void)x;
  if (!no_threads) abort();               // nothing here starts a thread before the flag is set
  return EAGAIN;
}

void *qhip_dl_create(size_t);
void qhip_dl_free(void *);
int qhip_dl_mark(void *, int), qhip_dl_copy(void *, int, void *, const void *, size_t), qhip_dl_finish(void *);

int main(int argc, char **argv) {
  if (argc > 1 && !strcmp(argv[1], "failed_wait")) {
    unsigned char src[3000], a[3000], b[3000];
    memset(src, 7, sizeof src);
    void *h = qhip_dl_create(1000);       // three chunks: one is emptied on the way, two are left for the end
    if (!h || qhip_dl_mark(h, 0)) return 2;
    if (qhip_dl_copy(h, 0, a, src, 2000)) return 3;
    fail_wait = 1;
    if (!qhip_dl_finish(h)) return 4;     // reported
    fail_wait = 0;
    memset(a, 0xEE, sizeof a);            // the caller has its buffer back
    if (qhip_dl_copy(h, 0, b, src, sizeof b) || qhip_dl_finish(h)) return 5;
    for (size_t i = 0; i < sizeof a; i++) if (a[i] != 0xEE) return 6;
    if (memcmp(b, src, sizeof b)) return 7;
    qhip_dl_free(h);
  } else {
    const size_t n = ((size_t)33 << 20) + 5;
    unsigned char *src = malloc(n), *d = calloc(n, 1);
    if (!src || !d) return 2;
    for (size_t i = 0; i < n; i++) src[i] = (unsigned char)(i * 31 + (i >> 11));
    void *h = qhip_dl_create((size_t)16 << 20);
    no_threads = 1;
    if (!h || qhip_dl_mark(h, 0) || qhip_dl_copy(h, 0, d, src, n) || qhip_dl_finish(h)) return 3;
    if (memcmp(d, src, n)) return 4;
    qhip_dl_free(h);
  }
  puts("ok");
  return 0;
}
"""


@pytest.mark.parametrize("what", ["failed_wait", "no_threads"])
def test_staged_download_host_side(tmp_path, what):
    """failed_wait: a wait that fails is reported, and the next download does not write
    to the failed one's destination.  no_threads: where no copying thread can be
    started the calling thread copies, and the process goes on."""
    qlib.load().lib()
    src, exe = tmp_path / "dl.c", tmp_path / "dl"
    src.write_text(PROGRAM)
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-rdynamic", str(src), "-o", str(exe), "-L" + qlib.PKG, "-lqllama",
                    "-Wl,-rpath," + qlib.PKG + ":/opt/rocm/lib", "-Wl,-rpath-link,/opt/rocm/lib"], check=True)
    r = subprocess.run([str(exe), what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stderr[-400:])
