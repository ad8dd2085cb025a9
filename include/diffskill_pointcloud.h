/*
 * diffskill_pointcloud.h -- C ABI of the point-cloud kernels (gfx950), in the
 * same library as diffskill_mpm.h (libdiffskill_mpm.so).
 *
 * pc_nearest is the nearest-neighbour search under the reference's Chamfer
 * losses: compute_chamfer_loss_kernel (plb/engine/losses/loss.py:183-204,
 * inner loops over all targets) and the chamferdist.ChamferDistance loss
 * built by create_chamfer_loss (plb/engine/taichi_env.py:28-32, a
 * third-party dependency absent here); pc_nearest_pair gives the same results
 * from spatially sorted clouds, both directions at once, and pc_chamfer_loss /
 * pc_chamfer_grad the loss and its gradients from them.
 *
 * pc_softmin / pc_plan_grad are the pairwise kernels of the Sinkhorn
 * divergence behind the reference's EMD loss, create_emd_loss's
 * geomloss.SamplesLoss(loss='sinkhorn', p=1, blur=0.001)
 * (plb/engine/taichi_env.py:23-26, evaluated at :269-270 and :303; geomloss
 * is a third-party dependency absent here): the soft-min of its dual
 * updates and the transport-plan gradient of its last step.  pc_sinkhorn_solve
 * runs the whole annealing loop and pc_sinkhorn_grad forms the gradient.
 */
#ifndef DISKILL_POINTCLOUD_H
#define DISKILL_POINTCLOUD_H

#ifdef __cplusplus
extern "C" {
#endif

/* For every query point q[i] (nq x 3 floats, device) the nearest target of
 * t (nt x 3 floats, device), by exact fp32 squared Euclidean distance:
 * idx[i] its index (the smallest index among equal distances; -1 when nt is
 * 0) and d2[i] the squared distance (+inf when nt is 0).  work: nq 64-bit
 * device words of scratch, overwritten.  Asynchronous on stream (a
 * hipStream_t); no allocation, no host synchronisation, so the call can be
 * captured into a HIP graph.  Cost: nq * nt distance evaluations.  Returns 0,
 * or -1 with pc_last_error() describing the problem. */
int pc_nearest(const float *q, int nq, const float *t, int nt, unsigned long long *work, int *idx, float *d2, void *stream);
const char *pc_last_error(void);

/* pc_nearest without the workspace argument and without any allocation: no
 * counterpart in the reference; for callers that cannot allocate device
 * memory (code under HIP graph capture, tight serving loops, harnesses that
 * forbid hipMalloc).  The per-query scratch is a static device array of the
 * library, 2^20 queries (8 MiB) per GPU, held until the process ends; nq
 * above that is refused with an error (-1) before any GPU work.  Every call
 * on one GPU shares that GPU's array (cleared for its nq queries at the
 * start of each call): calls that overlap on one GPU -- on different
 * streams or threads -- race and must be serialised by the caller.  Same
 * outputs as pc_nearest on the same inputs. */
int pc_nearest_noalloc(const float *q, int nq, const float *t, int nt, int *idx, float *d2, void *stream);

/* Bytes of device scratch that pc_softmin and pc_plan_grad need for n rows
 * and m columns (-1 for negative counts). */
long long pc_sinkhorn_work_bytes(int n, int m);

/* out[i] = -eps log sum_j exp(h[j] - C(x_i, y_j) / eps), the weights h
 * given in log2 units (h2 = h * log2(e)), for the n rows x (n x 3
 * floats, device) against the m columns y (m x 3), C = |x - y| (p = 1) or
 * |x - y|^2 / 2 (p = 2); every pair is evaluated (n * m work), the columns
 * split over workgroups whose partial (max, sum) are combined in a fixed
 * order.  work: pc_sinkhorn_work_bytes(n, m) bytes of device scratch.
 * Asynchronous on stream, no allocation.  Returns 0, or -1 with
 * pc_last_error() (m must be positive, eps positive, p 1 or 2). */
int pc_softmin(const float *x, int n, const float *y, int m, const float *h2, float eps, int p, void *work, float *out,
               void *stream);

/* g[i] (n x 3, overwritten) = sum_j exp(h[j] + r[i] - C(x_i, y_j) / eps)
 * dC(x_i, y_j)/dx_i with h = h2 / log2(e), r = r2 / log2(e) (log2 units, as
 * pc_softmin), dC/dx = (x - y) / |x - y| for p = 1 (0 where x = y) and
 * x - y for p = 2: the transport plan's pull on every row point.  Same work
 * buffer, stream and error rules as pc_softmin. */
int pc_plan_grad(const float *x, int n, const float *y, int m, const float *h2, const float *r2, float eps, int p, void *work,
                 float *g, void *stream);

/* Bytes of device scratch (16-byte aligned) that pc_sinkhorn_step, _solve and
 * _grad need (-1 unless n, m are 1 to 2^28). */
long long pc_sinkhorn_step_work_bytes(int n, int m);

/* One annealing step of the debiased Sinkhorn loop (uniform weights) on the
 * potentials pot = [a_x, b_x, a_y, b_y, pa_x, pb_x, pa_y, pb_y] (device
 * floats, lengths n, n, m, m, n, n, m, m): the four soft-mins
 *   a_y <- softmin_x(log(1/n) + b_x / eps), b_x <- softmin_y(log(1/m) + a_y / eps),
 *   a_x <- softmin_x(log(1/n) + a_x / eps), b_y <- softmin_y(log(1/m) + b_y / eps)
 * all computed from the previous values; mode 0 takes the log weights alone
 * (the first eps) and stores the results, mode 1 stores (previous + result) / 2
 * (the symmetric update of every eps), mode 2 moves the previous values to
 * pa_x.. and stores the results (the last extrapolation).  Two launches on
 * stream, every pair evaluated, fixed combination order, no allocation.
 * Returns 0, or -1 with pc_last_error(). */
int pc_sinkhorn_step(const float *x, int n, const float *y, int m, float *pot, float eps, int p, int mode, void *work,
                     void *stream);

/* The whole annealing loop: a step of mode 0 at eps[0], one of mode 1 at each
 * of the n_eps values and the extrapolation of mode 2 at the last, one launch
 * each; eps is a host array (read before the call returns).  pot: 4 (n + m)
 * device floats, laid out as for pc_sinkhorn_step and overwritten.  loss (device
 * float, or null): the divergence mean(b_x - a_x) + mean(a_y - b_y).  work:
 * pc_sinkhorn_step_work_bytes(n, m) device bytes.  Asynchronous on stream, no
 * allocation.  Returns 0, or -1 with pc_last_error(). */
int pc_sinkhorn_solve(const float *x, int n, const float *y, int m, const float *eps, int n_eps, int p, float *pot, float *loss,
                      void *work, void *stream);

/* Gradient of the divergence in the points, times *go (device float; 1 when
 * null), from the potentials pc_sinkhorn_solve left at the last eps: the
 * transport plans' pulls towards the other cloud minus those within the own one
 * (pc_plan_grad's sums), over n and m.  gx (n x 3) and gy (m x 3) are
 * overwritten; either may be null.  work as for pc_sinkhorn_solve.  Two
 * launches. */
int pc_sinkhorn_grad(const float *x, int n, const float *y, int m, const float *pot, float eps, int p, const float *go, float *gx,
                     float *gy, void *work, void *stream);

/* out[0..2] = extents (max - min) of the bounding box of both clouds (device
 * floats), NaN where a coordinate is.  One launch. */
int pc_extent(const float *x, int n, const float *y, int m, float *out, void *stream);

/* Nearest neighbours of two clouds, in either direction or both: for every
 * point of x its nearest of y (idx_x, d2_x) and for every point of y its nearest
 * of x (idx_y, d2_y); a direction whose two outputs are null is left out.
 * Indices and squared distances are pc_nearest's, bit for bit, an empty target
 * cloud's included.  work: pc_nearest_pair_work_bytes(n, m) device bytes, 16-byte
 * aligned.  Either every pair is looked at, or both clouds are sorted spatially and
 * most pairs left out, whichever is the faster at these sizes.  Asynchronous on stream, no allocation.  Returns 0, or
 * -1 with pc_last_error(). */
long long pc_nearest_pair_work_bytes(int n, int m);
int pc_nearest_pair(const float *x, int n, const float *y, int m, void *work, int *idx_x, float *d2_x, int *idx_y, float *d2_y,
                    void *stream);

/* The Chamfer loss of pc_nearest_pair's distances: out[0] = mean_i d_i of x's
 * direction, plus that of y's unless d2_y is null; d the distances, or their
 * squares with squared != 0.  One launch. */
int pc_chamfer_loss(const float *d2_x, int n, const float *d2_y, int m, int squared, float *out, void *stream);

/* Search and loss in one call: pc_nearest_pair into idx_x, d2_x and, unless null,
 * idx_y, d2_y, and the loss of these directions to loss[0].  Both clouds non-empty;
 * work as for pc_nearest_pair. */
int pc_chamfer(const float *x, int n, const float *y, int m, int squared, void *work, int *idx_x, float *d2_x, int *idx_y, float *d2_y,
               float *loss, void *stream);

/* Its gradient times *go (device float) in both clouds, the indices held:
 * gx (n x 3) and gy (m x 3) are overwritten, either may be null; idx_y and d2_y
 * null for a loss of x's direction alone.  A point without a nearest target gets
 * NaN.  Two or three launches; sums over the points that share a target are atomic, in no
 * fixed order. */
int pc_chamfer_grad(const float *x, int n, const float *y, int m, const int *idx_x, const float *d2_x, const int *idx_y,
                    const float *d2_y, int squared, const float *go, float *gx, float *gy, void *stream);

#ifdef __cplusplus
}
#endif
#endif
