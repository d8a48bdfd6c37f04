/* cf_internal_host.h -- internal helpers shared by the host C files and
 * the HIP runtime of the chanflow library (not part of the public ABI). */
#ifndef CF_INTERNAL_HOST_H
#define CF_INTERNAL_HOST_H

#ifdef __cplusplus
extern "C" {
#endif

/* record a printf-style message for cf_last_error() on this thread */
void cf_set_error(const char *fmt, ...);

/* a plane statistic (CF_STAT_AVG, _CORR, _MOMENT) of a run into res[nz]
 * with caller-provided device work space (part: 3 CF_STAT_NBL nz doubles),
 * enqueued on the run's stream (returned as an opaque hipStream_t); part == NULL only reports nz, the
 * stream and the device */
struct cf_run;
cf_status cf_run_stat_plane_into(struct cf_run *r, int kind, int fa, int fb, double en, double *part,
                                 double *res, int *nz, void **stream, int *device);

/* a device buffer to host memory after what the stream holds, complete on
 * return; device is current */
cf_status cf_copy_to_host(void *host, const void *dev, size_t bytes, int device, void *stream);

/* a run is made (+1) or gone (-1): what the copies keep goes with the last.
 * The live runs come back (0 only asks) */
int cf_copy_users(int add);

#ifdef __cplusplus
}
#endif

#endif
