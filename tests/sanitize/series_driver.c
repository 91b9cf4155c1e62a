/*
 * Host-only driver for what a search handle (accel_host.c, included here so
 * that a handle can be laid out by hand) promises about memory, streams and
 * events, built by tests/test_sanitize.py.
 * The device layer is replaced by test doubles that only book: an operation
 * stays pending on its stream, with the buffers it reads and writes, until
 * the stream, or an event recorded behind it, is waited for.
 *
 * Exits 0 when every check holds.
 */
#include "accel_host.c"

#define CHECK(c)                                                           \
    do {                                                                   \
        if (!(c)) {                                                        \
            fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__); \
            exit(1);                                                       \
        }                                                                  \
    } while (0)

/* ---- test doubles of the device layer ---- */

static struct {
    const void *stream, *rd, *wr;
} g_op[64];
static int g_nop;

struct event {
    const void *stream;
    int mark;   /* operations enqueued before it */
};

static void op(const void *stream, const void *rd, const void *wr)
{
    CHECK(g_nop < 64);
    g_op[g_nop].stream = stream;
    g_op[g_nop].rd = rd;
    g_op[g_nop++].wr = wr;
}

/* the first n operations of a stream are done */
static int done(const void *stream, int n)
{
    for (int i = 0; i < n; i++)
        if (g_op[i].stream == stream)
            g_op[i].rd = g_op[i].wr = NULL;
    return 0;
}

static int pending(const void *p)
{
    for (int i = 0; i < g_nop; i++)
        if (g_op[i].rd == p || g_op[i].wr == p)
            return 1;
    return 0;
}

static const char *g_fail = "";   /* the double that fails */

int agpu_malloc(void **p, size_t bytes) { return (*p = malloc(bytes)) == NULL; }
int agpu_free(void *p)
{
    CHECK(!p || !pending(p));   /* an arena hands a freed block out at once */
    free(p);
    return 0;
}
int agpu_h2d(void *dst, const void *src, size_t bytes, void *stream)
{
    (void) dst, (void) src, (void) bytes;
    return done(stream, g_nop);
}
int agpu_copy_d2d(void *dst, const void *src, size_t bytes, void *stream)
{
    (void) bytes;
    op(stream, src, dst);
    return 0;
}
int agpu_stream_sync(void *stream) { return done(stream, g_nop); }
int agpu_event_record(void *e, void *stream)
{
    ((struct event *) e)->stream = stream;
    ((struct event *) e)->mark = g_nop;
    return 0;
}
int agpu_event_sync(void *e)
{
    return done(((struct event *) e)->stream, ((struct event *) e)->mark);
}
const char *agpu_last_error(void) { return "double"; }
long long agpu_realfft_work(long long n) { return n; }
int agpu_realfft(const float *x, long long n, void *out, void *work, void *stream)
{
    (void) n, (void) work;
    if (!strcmp(g_fail, "realfft"))
        return -1;
    op(stream, x, out);
    return 0;
}
int agpu_deredden(void *spec, long long numbins, const agpu_window *blk, int nblk, int maxn,
                  float *mean, float im0, void *stream)
{
    (void) numbins, (void) blk, (void) nblk, (void) maxn, (void) mean, (void) im0;
    op(stream, spec, spec);
    return 0;
}

int agpu_memset(void *p, int v, size_t bytes, void *stream)
{
    (void) v, (void) bytes;
    op(stream, NULL, p);
    return 0;
}
int agpu_d2h(void *dst, const void *src, size_t bytes, void *stream)
{
    (void) src;
    memset(dst, 0, bytes);   /* no hits */
    return done(stream, g_nop);
}
int agpu_stream_wait_event(void *s, void *e) { return (void) s, (void) e, 0; }
int agpu_event_elapsed(float *ms, void *start, void *stop)
{
    *ms = (float) (((struct event *) stop)->mark - ((struct event *) start)->mark);
    return 0;
}
int agpu_block_norms(const void *spec, long long numbins, long long lobin, const agpu_window *win,
                     int nwin, int maxn, double *norm, float *nsq, void *stream)
{
    (void) numbins, (void) lobin, (void) win, (void) nwin, (void) maxn, (void) norm, (void) nsq;
    op(stream, spec, NULL);
    return 0;
}
int agpu_correlate(const void *spec, long long numbins, long long lobin, const void *T, int nt,
                   int L, int hw, int uselen, long long hb_end, float *plane, long long ntiles,
                   int groups, long long seg_lo, long long seg_hi, int bounds, void *stream)
{
    (void) numbins, (void) lobin, (void) T, (void) nt, (void) L, (void) hw, (void) uselen;
    (void) hb_end, (void) plane, (void) ntiles, (void) groups, (void) seg_lo, (void) seg_hi;
    (void) bounds;
    op(stream, spec, NULL);
    return 0;
}
int agpu_harmsum(const agpu_harmsum_args *a, long long c_lo, long long c_hi, void *stream)
{
    (void) a, (void) c_lo, (void) c_hi;
    op(stream, NULL, NULL);
    return 0;
}
int agpu_hit_sigmas(agpu_hitrec *hits, const unsigned *nhits, unsigned cap,
                    const agpu_numindep *ni, void *stream)
{
    (void) nhits, (void) cap, (void) ni;
    op(stream, NULL, hits);
    return 0;
}
/* linked, not reached: no bounds, standard norms */
int agpu_harmbound(const agpu_harmsum_args *a, const float *nb, void *stream)
{
    return (void) a, (void) nb, (void) stream, -1;
}
int agpu_bound_norms(const agpu_harmsum_args *a, long long hb_end, float *nb, void *stream)
{
    return (void) a, (void) hb_end, (void) nb, (void) stream, -1;
}
int agpu_inmem_nsq_table(const float *nsq, int npre, int nblocks, long long rh0, int cu,
                         long long hb_end, float *out, void *stream)
{
    (void) nsq, (void) npre, (void) nblocks, (void) rh0, (void) cu, (void) hb_end, (void) out;
    return (void) stream, -1;
}

/* ---- a handle with what the setters use ---- */

#define N 65536
static float g_series[N];
static struct event g_ev[8];

static accel_search *handle(void)
{
    accel_search *s = (accel_search *) calloc(1, sizeof(*s));
    s->g.numbins = N / 2;
    s->g.dt = 1e-3;
    s->stream = (void *) 1;
    s->stream2 = (void *) 2;
    s->ev_norms = &g_ev[0];
    s->ev_copy = &g_ev[1];
    for (int i = 0; i < 5; i++)
        s->ev[i] = &g_ev[2 + i];
    CHECK(agpu_malloc(&s->d_spec, sizeof(accel_fcomplex) * N / 2) == 0);
    s->own_spec = 1;
    g_nop = 0;
    g_fail = "";
    return s;
}

static void drop(accel_search *s)
{
    done(s->stream, g_nop);
    done(s->stream2, g_nop);
    if (s->own_spec)
        agpu_free(s->d_spec);
    agpu_free(s->d_fftwork);
    agpu_free(s->d_dblk);
    agpu_free(s->d_dmean);
    free(s);
}

/* The handle's own spectrum is freed only when nothing reads or writes it:
 * neither a preparation on the handle's stream nor norms on the second. */
static void spectrum_replaced(void)
{
    accel_fcomplex other;
    for (int k = 0; k < 3; k++) {
        accel_search *s = handle();
        if (k == 0)
            CHECK(accel_search_set_series(s, g_series, N) == 0);
        if (k == 1)
            CHECK(accel_search_set_device_series(s, g_series, N) == 0);
        if (k == 2)
            op(s->stream2, s->d_spec, NULL);
        CHECK(accel_search_set_device_spectrum(s, &other) == 0);
        CHECK(s->d_spec == &other && !s->own_spec);
        drop(s);
    }
}

/* The caller may free a device series when the call returns, also when the
 * preparation fails. */
static void series_returned(void)
{
    accel_search *s = handle();
    CHECK(accel_search_set_device_series(s, g_series, N) == 0);
    CHECK(!pending(g_series));
    drop(s);
    /* a host series is prepared when the call returns (a request's
     * preparation time is measured around it) */
    s = handle();
    CHECK(accel_search_set_series(s, g_series, N) == 0);
    CHECK(!pending(s->d_spec));
    drop(s);
    s = handle();
    g_fail = "realfft";
    CHECK(accel_search_set_device_series(s, g_series, N) != 0);
    CHECK(strstr(accel_last_error(), "double"));
    CHECK(!pending(g_series));
    drop(s);
}

/* The next series may be set while a search is launched and not collected:
 * the events that its timings come from stay as they are. */
static void launched_search(void)
{
    accel_search *s = handle();
    agpu_event_record(s->ev_norms, s->stream2);
    CHECK(accel_search_set_device_series(s, g_series, N) == 0);
    CHECK(g_ev[0].stream == s->stream2 && g_ev[0].mark == 0);
    drop(s);
}

/* The times of a search: one unit per operation between two events. */
static void timings(void)
{
    accel_search *s = handle();
    agpu_hitrec hits[2];
    float ms[5];
    s->d_hits = hits + 1;
    s->d_nhits = (unsigned *) hits;
    s->cap = 1;
    s->g.numharmstages = 1;
    CHECK(accel_search_launch(s) == 0 && accel_search_collect(s) == 0);
    CHECK(accel_search_timings(s, ms) == 0);
    CHECK(ms[0] == 1 && ms[1] == 1 && ms[2] == 0 && ms[3] == 1);
    CHECK(ms[4] == 4);   /* norms, correlation, harmonic sum and sigmas */
    free(s->hits);
    free(s->sigs);
    drop(s);
}

int main(void)
{
    timings();
    launched_search();
    spectrum_replaced();
    series_returned();
    printf("series checks passed\n");
    return 0;
}
