/*
 * sofi_frame.h - which cells lie in the absorbing frame, and the entries of
 * the CPML arrays that the update kernels fetch for them (sofi_kernels.hip).
 * No GPU is needed to check the ranges: tests/test_frame_entries.py compiles
 * this file on the host.  G is the kernels' Grid or any type with its members.
 */
#ifndef SOFI_FRAME_H
#define SOFI_FRAME_H

#ifdef __HIP__
#define SOFI_HD __host__ __device__ __forceinline__
#else
#define SOFI_HD inline
#endif

template <class G> SOFI_HD bool in_xframe(const G &g, int i) { return i <= g.gx2 || i > g.gx3; }
template <class G> SOFI_HD bool in_yframe(const G &g, int j) { return j <= g.gy2 || j > g.gy3; }
template <class G> SOFI_HD int hx(const G &g, int i) { return i <= g.gx2 ? i : i - g.nx + 2 * g.fw; }
template <class G> SOFI_HD int hy(const G &g, int j) { return j <= g.gy2 ? j : j - g.ny + 2 * g.fw; }

/* What is fetched for cell (i, j) with cpml_fetch: profiles at hx(i) and
 * x-frame memory at x_entry where frame_x, y-frame memory at y_entry where
 * frame_y.  PAST: also asked for cells past NX, as the shapes of several cells
 * per thread do; these get nothing (their entries would lie past the arrays'
 * ends), and nothing is fetched without a frame: the arrays, and the LDS they
 * go to, exist only with FW > 0.  (A cell 1..NX is then in no frame, so the
 * other shapes need no test.) */
template <bool PAST, class G> SOFI_HD bool frame_x(const G &g, int i) { return (!PAST || i <= g.nx) && in_xframe(g, i); }
template <bool PAST, class G> SOFI_HD bool frame_y(const G &g, int i, int j) { return (!PAST || i <= g.nx) && in_yframe(g, j); }
template <bool PAST, class G> SOFI_HD bool cpml_fetch(const G &g) { return g.abs_type == 1 && (!PAST || g.fw > 0); }
template <class G> SOFI_HD int x_entry(const G &g, int h, int j) { return j * g.wx + h; }
template <class G> SOFI_HD int y_entry(const G &g, int i, int j) { return hy(g, j) * g.wy + i; }

#endif /* SOFI_FRAME_H */
