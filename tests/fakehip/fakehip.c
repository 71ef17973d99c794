/* A stand-in for the HIP runtime that the library's host code can be tested
 * against on the CPU: device memory is host memory, copies are done at once,
 * kernels do nothing but are logged, captured streams count their kernels.  It
 * has two devices and rejects what a runtime may reject: kernels, events and
 * memory of another device than the stream's, and launches while that device
 * is not current. */
#include <stdarg.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { unsigned x, y, z; } dim3_;
enum { OK = 0, EINVALID = 1, ENOMEM_ = 2, EHANDLE = 400 };
enum { DEVICE = 1, PINNED = 2 };

static __thread int cur_dev = 0, last_error = 0;
static char *log_buf;
static size_t log_len, log_cap;

/* knobs and counters for the tests */
int fake_fail_copy;                         /* the n-th copy from now on fails (0: none) */
int fake_fail_pinned;                       /* 1: pinned allocations fail, 2: every second one */
size_t fake_device_fill;                    /* device memory starts out as the doubles 0, 1, 2, ... */
size_t fake_device_limit = (size_t)-1;      /* largest device allocation that succeeds */
size_t fake_largest_pinned, fake_largest_device, fake_live_pinned;

static int fail(int e) { last_error = e; return e; }

static void note(const char *fmt, ...)
{
    char line[512];
    va_list ap;
    va_start(ap, fmt);
    int n = vsnprintf(line, sizeof line - 1, fmt, ap);
    va_end(ap);
    if (n > (int)sizeof line - 2) n = sizeof line - 2;
    line[n++] = '\n';
    if (log_len + n + 1 > log_cap) {
        log_cap = 2 * (log_len + n + 1);
        log_buf = realloc(log_buf, log_cap);
    }
    memcpy(log_buf + log_len, line, n);
    log_len += n;
    log_buf[log_len] = 0;
}
const char *fake_log(void) { return log_len ? log_buf : ""; }
void fake_log_clear(void) { log_len = 0; }

/* memory: ranges by kind and device */
typedef struct mem { char *p; size_t n; int kind, dev; struct mem *next; } mem;
static mem *mems;
static mem *find(const void *p)
{
    for (mem *m = mems; m; m = m->next)
        if ((const char *)p >= m->p && (const char *)p < m->p + m->n) return m;
    return 0;
}
static int add(void **p, size_t n, int kind)
{
    mem *m = malloc(sizeof *m);
    m->p = calloc(n ? n : 1, 1);
    m->n = n ? n : 1;
    if (kind == DEVICE && fake_device_fill)
        for (size_t k = 0; k < n / 8; k++) ((double *)m->p)[k] = (double)k;
    m->kind = kind;
    m->dev = cur_dev;
    m->next = mems;
    mems = m;
    *p = m->p;
    return OK;
}
static int drop(void *p, int kind)
{
    for (mem **q = &mems; *q; q = &(*q)->next)
        if ((*q)->p == p) {
            mem *m = *q;
            if (m->kind != kind) return fail(EINVALID);
            if (kind == PINNED) fake_live_pinned -= m->n;
            *q = m->next;
            free(m->p);
            free(m);
            return OK;
        }
    return p ? fail(EINVALID) : OK;
}
int hipMalloc(void **p, size_t n)
{
    if (n > fake_device_limit) return fail(ENOMEM_);
    if (n > fake_largest_device) fake_largest_device = n;
    return add(p, n, DEVICE);
}
int hipFree(void *p) { return drop(p, DEVICE); }
int hipHostMalloc(void **p, size_t n, unsigned flags)
{
    (void)flags;
    static int calls;
    if (fake_fail_pinned == 1 || (fake_fail_pinned == 2 && ++calls % 2 == 0)) return fail(ENOMEM_);
    if (n > fake_largest_pinned) fake_largest_pinned = n;
    fake_live_pinned += n;
    return add(p, n, PINNED);
}
int hipHostFree(void *p) { return drop(p, PINNED); }

int hipGetDevice(int *d) { *d = cur_dev; return OK; }
int hipSetDevice(int d) { if (d < 0 || d > 1) return fail(EINVALID); cur_dev = d; return OK; }
int hipGetLastError(void) { int e = last_error; last_error = OK; return e; }
const char *hipGetErrorString(int e)
{
    return e == OK ? "no error" : e == ENOMEM_ ? "out of memory" : e == EHANDLE ? "invalid resource handle" : "error";
}

typedef struct { int dev, capturing, kernels; } stream;
typedef struct { int dev; } event;
typedef struct { int kernels; } graph;
int hipStreamCreateWithFlags(stream **s, unsigned f)
{
    (void)f;
    *s = calloc(1, sizeof **s);
    (*s)->dev = cur_dev;
    return OK;
}
int hipStreamDestroy(stream *s) { free(s); return OK; }
int hipStreamSynchronize(stream *s) { return s && s->capturing ? fail(EINVALID) : OK; }
int hipEventCreateWithFlags(event **e, unsigned f)
{
    (void)f;
    *e = calloc(1, sizeof **e);
    (*e)->dev = cur_dev;
    return OK;
}
int hipEventCreate(event **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(event *e) { free(e); return OK; }
int hipEventRecord(event *e, stream *s) { return e->dev != s->dev ? fail(EHANDLE) : OK; }
int hipEventSynchronize(event *e) { (void)e; return OK; }
int hipEventElapsedTime(float *ms, event *a, event *b) { (void)a; (void)b; *ms = 1.f; return OK; }

static int on(const void *p, stream *s)
{
    mem *m = find(p);
    return !m || m->kind != DEVICE || !s || m->dev == s->dev;
}
int hipMemcpyAsync(void *d, const void *src, size_t n, int kind, stream *s)
{
    (void)kind;
    if (fake_fail_copy && --fake_fail_copy == 0) return fail(EINVALID);
    if (!on(d, s) || !on(src, s)) return fail(EINVALID);
    if (s && s->capturing) return fail(EINVALID);
    memmove(d, src, n);
    return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) { return hipMemcpyAsync(d, s, n, kind, 0); }
int hipMemsetAsync(void *d, int v, size_t n, stream *s)
{
    if (!on(d, s) || (s && s->capturing)) return fail(EINVALID);
    memset(d, v, n);
    return OK;
}

/* kernels, by the names they are registered with */
typedef struct { const void *f; const char *name; } kern;
static kern *kerns;
static size_t nkerns;
void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterVar(void **m, void *v, char *a, char *b, int c, size_t n, int d, int e)
{
    (void)m; (void)v; (void)a; (void)b; (void)c; (void)n; (void)d; (void)e;
}
void __hipRegisterFunction(void **m, const void *f, char *dn, const char *name, unsigned tl, void *a, void *b, void *c,
                           void *d, int *w)
{
    (void)m; (void)dn; (void)tl; (void)a; (void)b; (void)c; (void)d; (void)w;
    kerns = realloc(kerns, (nkerns + 1) * sizeof *kerns);
    kerns[nkerns].f = f;
    kerns[nkerns++].name = name;
}
static __thread struct { dim3_ g, b; size_t sh; void *s; } conf;
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t sh, void *s)
{
    conf.g = g; conf.b = b; conf.sh = sh; conf.s = s;
    return OK;
}
int __hipPopCallConfiguration(dim3_ *g, dim3_ *b, size_t *sh, void **s)
{
    *g = conf.g; *b = conf.b; *sh = conf.sh; *s = conf.s;
    return OK;
}
int hipLaunchKernel(const void *f, dim3_ g, dim3_ b, void **args, size_t sh, stream *s)
{
    (void)args; (void)sh; (void)b;
    if (s && s->dev != cur_dev) return fail(EHANDLE);
    const char *name = "?";
    for (size_t k = 0; k < nkerns; k++)
        if (kerns[k].f == f) name = kerns[k].name;
    if (s && s->capturing) {
        s->kernels++;
        note("captured %s", name);
    } else {
        note("launch %s %u", name, g.x);
    }
    return OK;
}
int hipGetSymbolAddress(void **p, const void *sym) { *p = (void *)sym; return OK; }

int hipStreamBeginCapture(stream *s, int mode) { (void)mode; s->capturing = 1; s->kernels = 0; return OK; }
int hipStreamEndCapture(stream *s, graph **g)
{
    s->capturing = 0;
    *g = calloc(1, sizeof **g);
    (*g)->kernels = s->kernels;
    return OK;
}
int hipGraphInstantiate(graph **x, graph *g, void *a, char *b, size_t c)
{
    (void)a; (void)b; (void)c;
    *x = calloc(1, sizeof **x);
    **x = *g;
    return OK;
}
int hipGraphDestroy(graph *g) { free(g); return OK; }
int hipGraphExecDestroy(graph *g) { free(g); return OK; }
int hipGraphLaunch(graph *g, stream *s)
{
    if (s->dev != cur_dev) return fail(EHANDLE);
    note("graph %d", g->kernels);
    return OK;
}
