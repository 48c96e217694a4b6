// jr_backward.hip -- reverse-mode pass of the forward rasteriser (gfx950).
//
// What jax.grad computes through renderer/pipeline.py with visibility held
// piecewise constant: the chosen primitive, the inside test, keep flags,
// floor/round texture and shadow lookups and all comparisons carry no
// gradient; gradients flow through the barycentrics b = e / sum(e) with
// e = (x, y, 1) M^-1 (so through jnp.linalg.inv: dM = -M^-T G M^-T), the
// window depth, the interpolated varyings, the shading formulas, texture and
// specular-map values (a gather transposes to a scatter-add at the same
// clamped index), the light and the camera matrices.  JAX's conventions are
// kept: max(a, b) splits the gradient 1/2-1/2 on ties, pow(x, y) has
// d/dy = log(x) x^y with log(0) read as log(1), and d/dx = 0 when y == 0.
//
// Nothing is stored from the forward but prim_id: for every written pixel the
// kernels recompute the chosen primitive's setup, edge values, barycentrics
// and fragment attributes with the forward's own code (jr_common.h,
// jr_shade.h), so they are bit-identical to what the forward used.
//
//   k_bwd_prepare / k_bwd_fill  check the workspace header; clear the
//                 per-triangle flags and accumulators only for a workspace that
//                 no earlier call left zero (each call clears what it used)
//   k_bwd_pixels  one wavefront per 16x16 tile (4 pixels per lane) or 8x16
//                 tile (2; the rule is in backward_body): each distinct
//                 primitive's setup and corner stage once, in LDS;
//                 per pixel, shading backward (texture / specular gradients
//                 summed per texel in LDS), the visibility backward (dL/dM^-1,
//                 dL/dz_clip, per-corner varying cotangents) summed per
//                 triangle across lanes and in LDS, then one set of global
//                 atomics per (tile, triangle) and per (tile, texel)
//   k_bwd_tris    one thread per triangle, the touched ones packed together:
//                 M^-1 -> M -> clip -> positions and the vertex stage of each
//                 corner (normals, colours, light, camera matrices)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "../../include/jrhip.h"
#include "jr_common.h"
#include "jr_math.h"
#include "jr_shade.h"

namespace jr {

// Per-triangle accumulators: dMinv[3][3] (row r, column k), dz_clip[3],
// dvar[3][3]; phong_darboux adds the cotangents of its face's NDC corners
// (3 x 3) and of their uvs (3 x 2).
constexpr int kAcc = 21;
constexpr int A_MINV = 0;
constexpr int A_Z = 9;
constexpr int A_VAR = 12;
constexpr int A_TRI = 21;
constexpr int A_TUV = 30;
template <int SHADER>
struct AccOf {
  static constexpr int N = kAcc;
};
template <>
struct AccOf<JR_SHADER_PHONG_DARBOUX> {
  static constexpr int N = kAcc + 15;
};

// Accumulator floats per triangle of a shader (host side).
inline int acc_floats(int shader) {
  return shader == JR_SHADER_PHONG_DARBOUX ? AccOf<JR_SHADER_PHONG_DARBOUX>::N : kAcc;
}

// per-scene sums of k_bwd_pixels, three floats each; a shader has the first
// scene_sums() of them.  S_DIR is the light direction that its fragment stage
// normalises: light_dir_eye of the reflection shaders, light_direction of phong
// and phong_darboux.  The reflection shaders sum c diff and c spec (c: the
// cotangent times the texel, times the shadow factor) into S_DIFFUSE and
// S_SPECULAR, from which the gradients of diffuse, specular and the light's colour
// follow; phong and phong_darboux sum the last one in S_DIFFUSE's place.
enum {
  S_DIR = 0,
  S_LIGHT_COLOUR = 3,
  S_DIFFUSE = 3,
  S_SPECULAR = 6,
  S_AMBIENT = 9,
  S_STRENGTH = 12,
  S_COUNT = 15
};
constexpr bool reflects(int shader) {
  return shader == JR_SHADER_PHONG_REFLECTION || shader == JR_SHADER_PHONG_REFLECTION_SHADOW;
}
constexpr int scene_sums(int shader) {
  return shader == JR_SHADER_PHONG_REFLECTION_SHADOW ? S_COUNT
         : shader == JR_SHADER_PHONG_REFLECTION      ? S_STRENGTH
         : shader == JR_SHADER_PHONG || shader == JR_SHADER_PHONG_DARBOUX ? S_SPECULAR
                                                                          : 0;
}

// y = v / |v|: dv = (dy - y (y . dy)) / |v|
JR_DEV void normalise_bwd(const float v[3], const float dy[3], float dv[3]) {
  float ss = v[0] * v[0];
  ss = ss + v[1] * v[1];
  ss = ss + v[2] * v[2];
  const float n = sqrtf(ss);
  const float y[3] = {v[0] / n, v[1] / n, v[2] / n};
  const float yd = dot3(y, dy);
  for (int q = 0; q < 3; ++q) dv[q] = (dy[q] - y[q] * yd) / n;
}

// d max(a, b) / da under JAX's balanced rule
JR_DEV float max_grad(float a, float b) {
  return a > b ? 1.0f : (a == b ? 0.5f : 0.0f);
}

// What one pixel hands to the sums: the cotangent dn of its interpolated
// 3-vector, the texel, specular-map and normal-map entry its gradients land on
// (u < 0: none) with the gradients, and phong_darboux's cotangents of the face's
// NDC corners and their uvs.
template <int SHADER>
struct PixGrad {
  static constexpr bool kDarboux = SHADER == JR_SHADER_PHONG_DARBOUX;
  float dn[3];
  int32_t u, v;            // diffuse texel
  int32_t us, vs;          // specular-map or normal-map entry
  float tex_g[3], spec_g, nmap_g[kDarboux ? 3 : 1];
  float more[kDarboux ? 15 : 1];
  JR_DEV PixGrad() {
    dn[0] = dn[1] = dn[2] = 0.0f;
    u = us = -1;
    v = vs = 0;
    tex_g[0] = tex_g[1] = tex_g[2] = spec_g = 0.0f;
    nmap_g[0] = 0.0f;
    if constexpr (kDarboux) {
      nmap_g[1] = nmap_g[2] = 0.0f;
#pragma unroll
      for (int k = 0; k < 15; ++k) more[k] = 0.0f;
    }
  }
};

// Reverse of Varyings<SHADER>::pixel.  vary: the corner stage; n: interp() of its
// first 9 floats; l: Varyings<SHADER>::scene_terms; sg: the lane's per-scene sums.
template <int SHADER>
struct ShadeBwd;

template <>
struct ShadeBwd<JR_SHADER_DEPTH> {};

// shaders/gouraud.py:90-124: col = sum_k b_k col_k
template <>
struct ShadeBwd<JR_SHADER_GOURAUD> {
  static JR_DEV void run(const jr_inputs&, const jr_scene&, const jr_grads&, const float*,
                         const float[3], const float[3], const float[3],
                         const float dcol[3], PixGrad<JR_SHADER_GOURAUD>& g, float*, int) {
#pragma unroll
    for (int q = 0; q < 3; ++q) g.dn[q] = dcol[q];
  }
};

// Texel of the wrapping shaders: floor(uv) mod the map's shape.
JR_DEV void wrapped_texel(const jr_scene& sc, const float* uvv, const float b[3], int32_t* u,
                          int32_t* v) {
  const float uu = interp(b, uvv[0], uvv[2], uvv[4]);
  const float vv = interp(b, uvv[1], uvv[3], uvv[5]);
  *u = floor_mod(f2i_sat(floorf(uu)), sc.tex_w);
  *v = floor_mod(f2i_sat(floorf(vv)), sc.tex_h);
}

// shaders/gouraud_texture.py:103-144: col = texture[uv] * sum_k b_k lc_k
template <>
struct ShadeBwd<JR_SHADER_GOURAUD_TEXTURE> {
  static JR_DEV void run(const jr_inputs& in, const jr_scene& sc, const jr_grads&,
                         const float* vary, const float light[3], const float b[3],
                         const float[3], const float dcol[3],
                         PixGrad<JR_SHADER_GOURAUD_TEXTURE>& g, float*, int) {
    wrapped_texel(sc, vary + 9, b, &g.u, &g.v);
    float tex[3];
    tex_rgb(in.textures, sc.tex_base, sc.tex_h, sc.tex_c, g.u, g.v, tex);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      g.tex_g[q] = dcol[q] * light[q];
      g.dn[q] = dcol[q] * tex[q];
    }
  }
};

// shaders/phong.py:106-164
template <>
struct ShadeBwd<JR_SHADER_PHONG> {
  static JR_DEV void run(const jr_inputs& in, const jr_scene& sc, const jr_grads&,
                         const float* vary, const float n[3], const float b[3],
                         const float ln[3], const float dcol[3],
                         PixGrad<JR_SHADER_PHONG>& g, float* sg, int) {
    int32_t u, v;
    wrapped_texel(sc, vary + 9, b, &u, &v);
    float tex[3], nn[3];
    tex_rgb(in.textures, sc.tex_base, sc.tex_h, sc.tex_c, u, v, tex);
    normalise3(n, nn);
    const float d = dot3(nn, ln);
    float lc[3];
    bool pos = true;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      lc[q] = sc.light_colour[q] * d;
      pos = pos && (lc[q] >= 0.0f);
    }
    if (!pos) return;  // the zero branch of the cond carries no gradient
    g.u = u;
    g.v = v;
    float dd = 0.0f, dnn[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      g.tex_g[q] = dcol[q] * lc[q];
      const float dlc = dcol[q] * tex[q];
      sg[S_LIGHT_COLOUR + q] = fmaf(dlc, d, sg[S_LIGHT_COLOUR + q]);
      dd += dlc * sc.light_colour[q];
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      dnn[q] = dd * ln[q];
      sg[S_DIR + q] = fmaf(dd, nn[q], sg[S_DIR + q]);  // normalise's backward applied per tile
    }
    normalise_bwd(n, dnn, g.dn);
  }
};

// shaders/phong_darboux.py:116-293: the forward of Varyings<PHONG_DARBOUX>::pixel
// with its intermediates, then its reverse.  Beyond phong's terms the
// gradient reaches the tangent frame: B = [i/|i|, j/|j|, n] with
// (i, j) = inv(A) @ [du, dv] and A = [t1 - t0; t2 - t0; n] built from the
// face's NDC corners t_m = to_cartesian(world_to_clip @ [p_m, 1]) and their
// uvs; d(inv(A)) transposes to dA = -inv(A)^T G inv(A)^T.  The corners'
// cotangents go to the per-triangle accumulators (k_bwd_tris takes them to
// positions, uvs and world_to_clip); the normal-map texel gets d(B @ nm).
template <>
struct ShadeBwd<JR_SHADER_PHONG_DARBOUX> {
  using V = Varyings<JR_SHADER_PHONG_DARBOUX>;
  static JR_DEV void run(const jr_inputs& in, const jr_scene& sc, const jr_grads& gr,
                         const float* vary, const float n_i[3], const float b[3],
                         const float ln[3], const float dcol[3],
                         PixGrad<JR_SHADER_PHONG_DARBOUX>& g, float* sg, int) {
    int32_t u, v;
    wrapped_texel(sc, vary + 9, b, &u, &v);
    float tex[3], nm[3];
    tex_rgb(in.textures, sc.tex_base, sc.tex_h, sc.tex_c, u, v, tex);
    const int32_t un = index_clamp(u, sc.nmap_w);
    const int32_t vn = index_clamp(v, sc.nmap_h);
    load3(in.normal_maps + sc.nmap_base, un * sc.nmap_h + vn, nm);
    float n[3], AI[9], iv[3], jv[3], in_[3], jn[3];
    normalise3(n_i, n);
    V::tangents(vary, n, AI, iv, jv);
    normalise3(iv, in_);
    normalise3(jv, jn);
    float bn[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      float s = in_[r] * nm[0];
      s = s + jn[r] * nm[1];
      s = s + n[r] * nm[2];
      bn[r] = s;
    }
    float n2[3];
    normalise3(bn, n2);
    const float d = dot3(n2, ln);
    float lc[3];
    bool pos = true;
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) {
      lc[ch] = sc.light_colour[ch] * d;
      pos = pos && (lc[ch] >= 0.0f);
    }
    if (!pos) return;  // the zero branch of the cond carries no gradient
    g.u = u;
    g.v = v;

    // colour = tex * light_colour * dot(n2, ln)
    float dd = 0.0f;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      g.tex_g[q] = dcol[q] * lc[q];
      const float dlc = dcol[q] * tex[q];
      sg[S_LIGHT_COLOUR + q] = fmaf(dlc, d, sg[S_LIGHT_COLOUR + q]);
      dd += dlc * sc.light_colour[q];
    }
    float dn2[3], dbn[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      dn2[q] = dd * ln[q];
      sg[S_DIR + q] = fmaf(dd, n2[q], sg[S_DIR + q]);  // normalise's backward applied per tile
    }
    normalise_bwd(bn, dn2, dbn);
    // bn = B @ nm with B's columns in_, jn, n
    float din[3], djn[3], dn[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      din[r] = dbn[r] * nm[0];
      djn[r] = dbn[r] * nm[1];
      dn[r] = dbn[r] * nm[2];
    }
    if (gr.d_normal_maps) {
      g.us = un;
      g.vs = vn;
      g.nmap_g[0] = dot3(dbn, in_);
      g.nmap_g[1] = dot3(dbn, jn);
      g.nmap_g[2] = dot3(dbn, n);
    }
    float div[3], djv[3];
    normalise_bwd(iv, din, div);
    normalise_bwd(jv, djn, djv);
    // (i, j) = AI @ (du, dv): dAI = div du^T + djv dv^T, d(du) = AI^T div
    const float* tuv = vary + V::kTuv;
    const float du1 = tuv[2] - tuv[0], du2 = tuv[4] - tuv[0];
    const float dv1 = tuv[3] - tuv[1], dv2 = tuv[5] - tuv[1];
    float dAI[9];
    float ddu1 = 0.0f, ddu2 = 0.0f, ddv1 = 0.0f, ddv2 = 0.0f;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      dAI[3 * r + 0] = div[r] * du1 + djv[r] * dv1;
      dAI[3 * r + 1] = div[r] * du2 + djv[r] * dv2;
      dAI[3 * r + 2] = div[r] * 0.0f + djv[r] * 0.0f;
      ddu1 += div[r] * AI[3 * r + 0];
      ddu2 += div[r] * AI[3 * r + 1];
      ddv1 += djv[r] * AI[3 * r + 0];
      ddv2 += djv[r] * AI[3 * r + 1];
    }
    float* dtuv = g.more + 9;
    dtuv[0] = -(ddu1 + ddu2);  // corner 0: u, v
    dtuv[1] = -(ddv1 + ddv2);
    dtuv[2] = ddu1;  // corner 1
    dtuv[3] = ddv1;
    dtuv[4] = ddu2;  // corner 2
    dtuv[5] = ddv2;
    // dA = -AI^T dAI AI^T
    float T1[9], dA[9];
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        float s = 0.0f;
#pragma unroll
        for (int r = 0; r < 3; ++r) s += AI[3 * r + p] * dAI[3 * r + k];
        T1[3 * p + k] = s;
      }
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < 3; ++k) s += T1[3 * p + k] * AI[3 * q + k];
        dA[3 * p + q] = -s;
      }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      g.more[0 + q] = -(dA[q] + dA[3 + q]);
      g.more[3 + q] = dA[q];
      g.more[6 + q] = dA[3 + q];
      dn[q] += dA[6 + q];
    }
    normalise_bwd(n_i, dn, g.dn);
  }
};

// shaders/phong_reflection.py:154-235 and phong_reflection_shadow.py:173-271
template <int SHADER>
struct ReflectionBwd {
  static constexpr bool SHADOW = SHADER == JR_SHADER_PHONG_REFLECTION_SHADOW;
  using V = Varyings<SHADER>;
  static JR_DEV void run(const jr_inputs& in, const jr_scene& sc, const jr_grads& gr,
                         const float* vary, const float n[3], const float b[3],
                         const float lh[3], const float dcol[3], PixGrad<SHADER>& g,
                         float* sg, int scene) {
    const float* uvv = vary + 9;  // uv of corner k: uvv[2k..2k+1]
    const int32_t ti = __float_as_int(vary[V::kTi]);
    float uv[2];
    uv[0] = interp(b, uvv[0], uvv[2], uvv[4]);
    uv[1] = interp(b, uvv[1], uvv[3], uvv[5]);
    // forward of reflection_terms with its intermediates
    const int32_t s0 = __float_as_int(vary[V::kShape]), s1 = __float_as_int(vary[V::kShape + 1]);
    float f0 = modf_frac(uv[0]), f1 = modf_frac(uv[1]);
    f0 = (f0 < 0.0f) ? f0 + 1.0f : f0;
    f1 = (f1 < 0.0f) ? f1 + 1.0f : f1;
    const int32_t shift = (int32_t)((uint32_t)ti * (uint32_t)sc.tex_offset);
    const int32_t u0 = f2i_sat(floorf(f0 * (float)s0 + (float)shift));
    const int32_t v0 = f2i_sat(floorf(f1 * (float)s1));
    g.u = index_clamp(u0, sc.tex_w);
    g.v = index_clamp(v0, sc.tex_h);
    g.us = index_clamp(u0, sc.spec_w);
    g.vs = index_clamp(v0, sc.spec_h);
    // the three lookups are issued together
    float tex[3], depth = 0.0f, sz = 0.0f;
    tex_rgb(in.textures, sc.tex_base, sc.tex_h, sc.tex_c, g.u, g.v, tex);
    const float S = in.specular_maps[sc.spec_base + (int64_t)g.us * sc.spec_h + g.vs];
    if (SHADOW) {
      const float* scd = vary + 15;  // homogeneous-normalised shadow clip of corner k
      float s4[4], sv[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) s4[q] = interp(b, scd[q], scd[4 + q], scd[8 + q]);
      apply4(sc.shadow_viewport, s4[0], s4[1], s4[2], s4[3], sv);
      sz = sv[2] / sv[3];
      const float* map = in.shadow_maps + (int64_t)scene * in.shadow_w * in.shadow_h;
      depth = shadow_get(map, in.shadow_w, in.shadow_h, sv[0] / sv[3], sv[1] / sv[3]);
    }
    float nh[3];
    normalise3(n, nh);
    const float d = dot3(nh, lh);
    const float diff = max_nan(d, 0.0f);
    const float two_d = 2.0f * d;
    float qv[3] = {two_d * nh[0] - lh[0], two_d * nh[1] - lh[1], two_d * nh[2] - lh[2]};
    float rh[3];
    normalise3(qv, rh);
    const float m = max_nan(rh[2], 0.0f);
    // the forward's power (pow_unit: within 3e-7 of powf for m in [0, 1]) and the
    // one of its derivative
    const float spec = pow_unit(m, S);
    const float slope = S == 0.0f ? 0.0f : S * pow_unit(m, S - 1.0f);
    const bool lit = !SHADOW || sz <= depth;

    float ddiff = 0.0f, dspec = 0.0f;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const float k = sc.diffuse[q] * diff + sc.specular[q] * spec;
      const float sh = lit ? 1.0f : 1.0f - sc.shadow_strength[q];
      const float ct = dcol[q] * tex[q];
      const float cs = SHADOW ? sh * ct : ct;
      const float dk = SHADOW ? dcol[q] * sh * tex[q] * sc.light_colour[q]
                              : dcol[q] * sc.light_colour[q] * tex[q];
      g.tex_g[q] = dcol[q] * (sc.ambient[q] + (SHADOW ? sh * k : k) * sc.light_colour[q]);
      sg[S_AMBIENT + q] += ct;
      if constexpr (SHADOW)
        sg[S_STRENGTH + q] =
            lit ? sg[S_STRENGTH + q]
                : fmaf(-k, ct * sc.light_colour[q], sg[S_STRENGTH + q]);
      sg[S_DIFFUSE + q] = fmaf(cs, diff, sg[S_DIFFUSE + q]);
      sg[S_SPECULAR + q] = fmaf(cs, spec, sg[S_SPECULAR + q]);
      ddiff += dk * sc.diffuse[q];
      dspec += dk * sc.specular[q];
    }
    if (gr.d_specular_maps)
      g.spec_g = dspec * logf(m == 0.0f ? 1.0f : m) * spec;
    else
      g.us = -1;
    const float dm = dspec * slope;
    const float dr[3] = {0.0f, 0.0f, dm * max_grad(rh[2], 0.0f)};
    float dq[3];
    normalise_bwd(qv, dr, dq);
    const float dtwo_d = dot3(dq, nh);
    const float dd = 2.0f * dtwo_d + ddiff * max_grad(d, 0.0f);
    float dnh[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      dnh[q] = two_d * dq[q] + dd * lh[q];
      // normalise's backward is linear in its cotangent: applied once per tile
      sg[S_DIR + q] += fmaf(dd, nh[q], -dq[q]);
    }
    normalise_bwd(n, dnh, g.dn);
  }
};

template <>
struct ShadeBwd<JR_SHADER_PHONG_REFLECTION> : ReflectionBwd<JR_SHADER_PHONG_REFLECTION> {};
template <>
struct ShadeBwd<JR_SHADER_PHONG_REFLECTION_SHADOW>
    : ReflectionBwd<JR_SHADER_PHONG_REFLECTION_SHADOW> {};

// v moved across lanes by the DPP pattern CTRL (lanes without a source get 0).
template <int CTRL>
JR_DEV float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// The totals over the 64 lanes of the wavefront of N <= 32 values a lane: lane l
// returns that of value l / 2 (l / 2 < N).  A step of the reduction halves the
// lanes that share a value and the values that a lane holds: in step 16 the
// lower half of the wavefront goes on with values 0..15 and the upper half with
// 16..31, and so on, so 32 values take 16 + 8 + 4 + 2 + 1 + 1 additions, where one
// value at a time takes six each, and their totals are added to memory by one
// instruction.  Call with every lane active.
template <int N>
JR_DEV float wave_totals(const float (&v)[N]) {
  static_assert(N <= 32, "one value per lane pair");
  float a[N];
#pragma unroll
  for (int i = 0; i < N; ++i) a[i] = v[i];
  const int lane = threadIdx.x & 63;
  int n = N;
#pragma unroll
  for (int half = 16; half >= 1; half >>= 1) {
#pragma unroll
    for (int i = 0; i < half && i < n; ++i) {
      const bool pair = i + half < n;
      const float x = a[i], y = pair ? a[i + half] : x;
      if (half >= 8) {
        const auto r = half == 16
                           ? __builtin_amdgcn_permlane32_swap(__float_as_uint(x),
                                                              __float_as_uint(y), false, false)
                           : __builtin_amdgcn_permlane16_swap(__float_as_uint(x),
                                                              __float_as_uint(y), false, false);
        a[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
      } else {
        const bool up = (lane & (2 * half)) != 0;
        const float keep = up ? y : x, give = up ? x : y;
        a[i] = keep + (half == 4   ? dpp_move<0x128>(give)    // row_ror:8
                       : half == 2 ? dpp_move<0x141>(give)    // row_half_mirror
                                   : dpp_move<0x4e>(give));   // quad_perm [2,3,0,1]
      }
    }
    n = n < half ? n : half;
  }
  return a[0] + dpp_move<0xb1>(a[0]);  // quad_perm [1,0,3,2]
}

// Sums per map entry in LDS: NC floats for each of up to CAP distinct keys, so
// that an entry which several pixels of the wavefront read costs one global
// atomic per channel.  What finds no place near its own is added to memory at
// once; its acknowledgement then holds up the loads issued after it (a wavefront's
// memory operations complete in order), so the table is as large as the number of
// pixels where nearly every pixel has its own entry.
constexpr int32_t kStageProbes = 16;

template <int CAP, int NC>
struct SumTable {
  int32_t key[CAP];
  float v[NC][CAP];
  JR_DEV void clear() {
    for (int e = threadIdx.x; e < CAP; e += 64) {
      key[e] = -1;
#pragma unroll
      for (int c = 0; c < NC; ++c) v[c][e] = 0.0f;
    }
  }
  // g to entry k; to_memory(k, c, x): x to channel c of an entry in memory
  template <class Add>
  JR_DEV void add(int32_t k, const float* g, Add to_memory) {
    const int32_t e = table_insert(key, CAP, k, kStageProbes);
    if (e >= 0) {
#pragma unroll
      for (int c = 0; c < NC; ++c) atomicAdd(&v[c][e], g[c]);
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c) to_memory(k, c, g[c]);
    }
  }
  // Adds the sums to memory.  Lanes take consecutive (entry, channel) pairs, so
  // the channels of one entry are added by neighbouring lanes of one instruction
  // (same cache line).
  template <class Add>
  JR_DEV void flush(Add to_memory) {
    for (int idx = threadIdx.x; idx < CAP * NC; idx += 64) {
      const int e = idx / NC, c = idx - NC * e;
      const int32_t k = key[e];
      if (k != -1) to_memory(k, c, v[c][e]);
    }
  }
};

struct BwdArgs {
  jr_inputs in;
  const jr_scene* scenes;
  jr_grads gr;
  const float* d_canvas;
  // fused L2 loss: with target set the canvas cotangent of a pixel is
  // l2_scale * (canvas - target), read in place of d_canvas
  const float* canvas;
  const float* target;
  float l2_scale;
  const float* d_zbuffer;
  const int32_t* prim_id;
  float* tacc;              // kAcc floats per triangle, zero between calls
  int32_t* touched;         // per triangle: its scene + 1 once a pixel adds to it, zero between calls
  uint32_t* header;         // workspace header (kHdr* words)
  int32_t W, H, n_scenes;
  // the 2x2 (or 1x2) pixel blocks of a scene (k_bwd_pixels), nq of them numbered:
  // FX x FY tiles of 8 x 8 blocks, rw and rh blocks left over right of and
  // below them; blocks [0, full_end) are the tiles', [full_end, bottom_end)
  // those below them; T wavefronts per scene
  int32_t nq, T, FX, FY, rw, rh, full_end, bottom_end;
  uint32_t T_m, fy_m, rh_m, rw_m;  // udiv31 by T, FY, rh and rw (by 1 for a zero)
  int32_t T_sh, fy_sh, rh_sh, rw_sh;
};

// Workspace header words.  The accumulators and flags are left zero by every
// call (k_bwd_tris clears what it consumed), so a call only clears them in
// full when the header does not describe this workspace yet.
constexpr int kHdrMagicLo = 0, kHdrMagicHi = 1, kHdrTris = 2, kHdrFill = 3, kHdrAcc = 4;
constexpr uint32_t kMagicLo = 0x6a724277u, kMagicHi = 0x73706b31u;

// The calling kernel's first argument, of type T, in the kernel argument segment.
template <class T>
using KernArgs = const __attribute__((address_space(4))) T*;
template <class T>
JR_DEV KernArgs<T> kernel_args() {
  return (KernArgs<T>)__builtin_amdgcn_kernarg_segment_ptr();
}

// A scene's pixels in blocks of 2x2 (PPL = 4) or 1x2 (PPL = 2), one wavefront per
// 64 consecutive blocks of this enumeration: the full tiles of 8 x 8 blocks first,
// tile by tile, so that each is one wavefront with lane l owning the block (8 tx +
// l / 8, 8 ty + l % 8); then the blocks below them (rh per row) and those right of
// them (rw per column), which share wavefronts instead of leaving most lanes of a
// partial tile idle (an 84 x 84 frame takes 28 wavefronts, not 36).  Where that
// saves few wavefronts every tile, partial ones included, is a wavefront of its own.
//
// A wavefront that shows no triangle leaves at once.  The others work in rounds of
// up to tri_cap() distinct triangles (mostly one round): their corners' clip
// positions and corner stage, one lane per corner, and their setup, one lane per
// triangle, go to LDS; then each lane goes over its pixels.  A lane sums
// consecutive pixels of one triangle, and of one texel, in registers and adds a run
// to the LDS sums when it ends, so neighbouring pixels, which mostly share both,
// cost one LDS atomic instead of four; the LDS sums reach memory once per
// (wavefront, triangle) and (wavefront, map entry).
//
// What bounds it: round trips to memory, then the LDS, which takes a turn for each
// lane of an atomic on one address.  On 512 frames of 480x270, where half of the
// wavefronts show nothing and half of the others one large triangle, and where it
// took 2,972 us: with the lanes' last runs summed across the wavefront (2,470 ->
// 1,320 LDS cycles per wavefront), a fourth wavefront per SIMD (162 registers ->
// 128: scalars read again for each pixel instead of spilt into vector registers, no
// own path for triangles beyond the table) and the scene's sums reduced together,
// 2,238 us; with the empty wavefronts gone at once, one chain of loads for corners
// and setup, and triangles numbered, so that only those there are are cleared and
// added, 1,758 us.  1,024 frames of 84x84: 573, 590, 538 us.
//
// 16 workgroups' LDS on a CU, 4 wavefronts per SIMD as 128 registers allow, takes
// at most 10 KiB each.  With a depth gradient the reflection shaders' three more sums
// and six more values per pixel do not fit 128 registers (22 and 41 of them were spilt,
// and 1,024 frames of 84x84 took 888 us): those two instances run 3 wavefronts of 168
// (804 us).
constexpr int tri_cap(int shader) {
  return shader == JR_SHADER_PHONG_REFLECTION_SHADOW || shader == JR_SHADER_PHONG_DARBOUX ? 28
                                                                                         : 32;
}
// distinct texels summed in LDS: the reflection shaders' maps repeat over a merged
// scene's objects, the others' have about a texel per pixel
constexpr int tex_cap(int shader) { return reflects(shader) ? 128 : 224; }
// Lanes on one triangle (texel) from which a sum across the wavefront (some 95
// instructions for 18 sums, 40 for 4) replaces their LDS atomics, and how many
// triangles (texels) are looked at.  Four lanes pay for it (64 gouraud views 411
// against 426 us), but with four pixels to a lane, where it makes no difference
// (512 frames of 480x270), eight leave the order of small triangles' sums as it was.
constexpr int shared_from(int ppl) { return ppl == 4 ? 8 : 4; }
constexpr int kSearched = 12;
constexpr int kTexShared = 16, kTexSearched = 4;
constexpr int kMapCap = 32;  // entries of a second map (normal map, specular map)

constexpr int pixel_waves(int shader, bool dz) {
  return shader == JR_SHADER_PHONG_DARBOUX ? 2 : dz && reflects(shader) ? 3 : 4;
}

template <int SHADER, bool DZ, int PPL>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(pixel_waves(SHADER, DZ), 8)))
void k_bwd_pixels(BwdArgs) {
  constexpr int BW = PPL / 2;  // a lane's block is BW x 2 pixels
  constexpr int kShared = shared_from(PPL);
  using V = Varyings<SHADER>;
  constexpr int NV = V::N;
  constexpr int NS = (12 + NV) | 1;  // record stride (odd: no LDS bank conflicts)
  constexpr int CAP = tri_cap(SHADER);
  constexpr int ACC = AccOf<SHADER>::N;
  // a triangle's sums in a lane and in LDS: its accumulators without A_Z where no
  // depth gradient comes in (DZ)
  constexpr int NR = DZ ? ACC : ACC - 3;
  constexpr int R_VAR = 9, R_Z = 18, R_TRI = DZ ? 21 : 18;
  constexpr int AS = NR | 1;  // odd row stride: lanes of different rows hit different banks
  constexpr bool DARBOUX = SHADER == JR_SHADER_PHONG_DARBOUX;
  constexpr bool REFLECT = reflects(SHADER);
  constexpr int NT = REFLECT ? 4 : 3;  // a texel's channels, and its specular exponent's
  constexpr int N2 = DARBOUX ? 3 : 1;
  __shared__ float trec[CAP * NS];
  __shared__ float acc[CAP][AS];
  __shared__ int32_t tab[CAP], ids[CAP];
  __shared__ float light[3];
  __shared__ SumTable<(NV > 9 ? tex_cap(SHADER) : 1), NT> tex_tab;
  __shared__ SumTable<DARBOUX || REFLECT ? kMapCap : 1, N2> map_tab;
  // The kernel's arguments and the scene's values are read where they are used
  // (scalar loads): kept over the whole kernel, with what is computed from them,
  // they take three times the scalar registers there are, and what has no place is
  // moved through vector registers lane by lane.  read_again() makes the compiler
  // forget the values it has.
  KernArgs<BwdArgs> ap = kernel_args<BwdArgs>();
  const jr_scene* sp = nullptr;
  auto read_again = [&]() { asm volatile("" : "+s"(ap), "+s"(sp)); };
  auto args = [&]() -> const BwdArgs& { return *(const BwdArgs*)ap; };
  auto scene = [&]() -> const jr_scene& { return *sp; };
  const int lane = threadIdx.x;
  const int32_t gt = (int32_t)blockIdx.x;
  const int32_t s = udiv31(gt, args().T_m, args().T_sh);
  // the first pixel (bi, bj) of the lane's block, number Q of the scene's blocks
  const int32_t Q = 64 * (gt - s * args().T) + lane;
  int32_t bi, bj;
  if (Q < args().full_end) {  // a full tile per wavefront, its blocks row by row
    const int32_t tile = Q >> 6;
    const int32_t tx = udiv31(tile, args().fy_m, args().fy_sh), ty = tile - tx * args().FY;
    bi = BW * (8 * tx + ((Q >> 3) & 7));
    bj = 16 * ty + 2 * (Q & 7);
  } else if (Q < args().bottom_end) {  // below the full tiles, rh blocks per row
    const int32_t q = Q - args().full_end;
    const int32_t row = udiv31(q, args().rh_m, args().rh_sh);
    bi = BW * row;
    bj = 16 * args().FY + 2 * (q - row * args().rh);
  } else {  // right of them over the whole height, rw blocks per column
    const int32_t q = Q - args().bottom_end;
    const int32_t col = udiv31(q, args().rw_m, args().rw_sh);
    bi = BW * (8 * args().FX + (q - col * args().rw));
    bj = 2 * col;
  }
  sp = args().scenes + s;
  const int64_t pix0 = (int64_t)s * args().W * args().H + (int64_t)bi * args().H + bj;
  // the block's pixels, q = 2 (i - bi) + (j - bj), that show a triangle
  auto pixel = [&](int q) { return pix0 + (q >> 1) * args().H + (q & 1); };
  uint32_t todo = 0u;
  {
    int32_t t[PPL];
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
      const bool in = Q < args().nq && bi + (q >> 1) < args().W && bj + (q & 1) < args().H;
      t[q] = in ? args().prim_id[pixel(q)] : -1;
    }
#pragma unroll
    for (int q = 0; q < PPL; ++q)
      todo |= t[q] >= 0 && t[q] < args().in.n_tris ? 1u << q : 0u;
  }
  if (__ballot(todo != 0u) == 0) return;
  const float* vp = scene().viewport;
  const float x0 = pix_x(bi, vp), x1 = pix_x(bi + 1, vp);
  const float y0 = pix_y(bj, vp), y1 = pix_y(bj + 1, vp);

  // sums per map entry.  A texel's specular exponent has the texel's number where
  // the two maps have one shape (uniform): then its gradient is the texel's
  // fourth channel.  A map of 2^32 texels and more is added to directly.
  const bool huge = (int64_t)scene().tex_w * scene().tex_h >= 0xFFFFFFFFLL ||
                    (REFLECT && (int64_t)scene().spec_w * scene().spec_h >= 0xFFFFFFFFLL) ||
                    (DARBOUX && (int64_t)scene().nmap_w * scene().nmap_h >= 0xFFFFFFFFLL);
  const bool one_map = REFLECT && args().gr.d_textures && args().gr.d_specular_maps &&
                       scene().tex_w == scene().spec_w && scene().tex_h == scene().spec_h;
  auto texel_at = [&](int64_t m, int c, float x) {
    if (x == 0.0f) return;
    if (REFLECT && c == 3)
      atomicAdd(args().gr.d_specular_maps + scene().spec_base + m, x);
    else if (c < scene().tex_c)
      atomicAdd(args().gr.d_textures + scene().tex_base + m * scene().tex_c + c, x);
  };
  auto entry_at = [&](int64_t m, int c, float x) {
    if (x == 0.0f) return;
    if (REFLECT) atomicAdd(args().gr.d_specular_maps + scene().spec_base + m, x);
    if (DARBOUX) atomicAdd(args().gr.d_normal_maps + scene().nmap_base + 3 * m + c, x);
  };
  auto add_texel = [&](int32_t key, int c, float x) { texel_at((uint32_t)key, c, x); };
  auto add_entry = [&](int32_t key, int c, float x) { entry_at((uint32_t)key, c, x); };
  if (lane == 0) {
    float l[3] = {0.0f, 0.0f, 0.0f};
    if constexpr (NV > 0) V::scene_terms(scene(), l);
    light[0] = l[0];
    light[1] = l[1];
    light[2] = l[2];
  }
  tex_tab.clear();
  if constexpr (REFLECT || DARBOUX) map_tab.clear();
  int32_t tex_key = -1;  // the lane's open run of pixels on one texel
  float tex_sum[NT];
#pragma unroll
  for (int c = 0; c < NT; ++c) tex_sum[c] = 0.0f;

  // the shader's sums, then the viewport's entries 10 and 11 (DZ)
  constexpr int NSH = scene_sums(SHADER), NSG = NSH + (DZ ? 2 : 0);
  float sg[NSG > 0 ? NSG : 1];
#pragma unroll
  for (int q = 0; q < NSG; ++q) sg[q] = 0.0f;

  while (__ballot(todo != 0u) != 0) {
    read_again();
    // the round's distinct triangles: an LDS set, whose entries are then numbered
    if (lane < CAP) tab[lane] = -1;
    __syncthreads();
    int32_t t4[PPL];
#pragma unroll
    for (int q = 0; q < PPL; ++q) t4[q] = (todo >> q) & 1u ? args().prim_id[pixel(q)] : -1;
    int32_t entry[PPL];
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
      entry[q] = -1;
      if (t4[q] >= 0)
        entry[q] = q > 0 && t4[q] == t4[q > 0 ? q - 1 : 0] ? entry[q > 0 ? q - 1 : 0]
                                                          : table_insert(tab, CAP, t4[q]);
    }
    __syncthreads();
    const int32_t found = lane < CAP ? tab[lane] : -1;
    const uint64_t used = __ballot(found >= 0);
    const int32_t nt = __popcll(used);
    const int32_t rank = __builtin_amdgcn_mbcnt_hi(
        (uint32_t)(used >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)used, 0u));
    if (found >= 0) ids[rank] = found;
    uint32_t slots = 0u;  // per pixel the number of its triangle, 255: not in this round
#pragma unroll
    for (int q = 0; q < PPL; ++q) {
      const int32_t r = __shfl(rank, entry[q] & 63);
      slots |= (entry[q] >= 0 ? (uint32_t)r : 255u) << (8 * q);
      if (entry[q] >= 0) todo &= ~(1u << q);
    }
    for (int k = lane; k < nt * AS; k += 64) (&acc[0][0])[k] = 0.0f;
    __syncthreads();
    // per corner, one lane each: its clip position (where the triangle's record goes
    // next) and its corner stage, whose loads are in flight together
#pragma unroll 1
    for (int idx = lane; idx < 3 * nt; idx += 64) {
      const int e = idx / 3, k = idx - 3 * e;
      const int32_t t = ids[e], slot = face_slot(args().in, t, k);
      float* row = trec + e * NS;
      float h[4];
      position_clip(args().in, scene().world_to_clip, slot, h);
      if constexpr (NV > 0)
        V::corner(args().in, scene(), slot, face_slot(args().in, t, 0), k, row + 12);
#pragma unroll
      for (int c = 0; c < 4; ++c) row[4 * k + c] = h[c];
    }
    __syncthreads();
    if (lane < nt) {
      TriSetup ts;
      float* r = trec + lane * NS;
#pragma unroll
      for (int k = 0; k < 12; ++k) ts.clip[k / 4][k % 4] = r[k];
      ts.det = tri_det(ts.clip, ts.M);
      tri_finish(ts);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const float4 c = rec_col(ts, k);
        r[4 * k + 0] = c.x;
        r[4 * k + 1] = c.y;
        r[4 * k + 2] = c.z;
        r[4 * k + 3] = c.w;
      }
    }
    __syncthreads();

    uint32_t run_slot = 255u;  // the lane's open run and its sums
    float run[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) run[k] = 0.0f;
    auto flush_tri = [&]() {
      if (run_slot != 255u) {
        float* row = acc[run_slot];
#pragma unroll
        for (int k = 0; k < NR; ++k)
          if (NV > 0 || k < R_VAR || k >= R_Z) atomicAdd(row + k, run[k]);
      }
#pragma unroll
      for (int k = 0; k < NR; ++k) run[k] = 0.0f;
    };
#pragma unroll 1
    for (int q = 0; q < PPL; ++q) {
      const uint32_t slot = (slots >> (8 * q)) & 255u;
      if (__ballot(slot != 255u) == 0) continue;
      if (slot != run_slot) {
        flush_tri();
        run_slot = slot;
      }
      PixGrad<SHADER> g;
      read_again();
      if (slot != 255u) {
        // the canvas cotangent, or the canvas and target that it is computed from:
        // first, and used last
        const int64_t pix = pixel(q);
        const float* from = args().target ? args().canvas : args().d_canvas;
        float dcol[3] = {0.0f, 0.0f, 0.0f}, tgt[3] = {0.0f, 0.0f, 0.0f};
        if (from) load3(from + 3 * pix, 0, dcol);
        if (args().target) load3(args().target + 3 * pix, 0, tgt);
        const float* r = trec + slot * NS;
        const float* vary = r + 12;
        const float x = q < 2 ? x0 : x1, y = q & 1 ? y1 : y0;
        float4 col[3];
        float e[3], b[3], db[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          col[k] = make_float4(r[4 * k], r[4 * k + 1], r[4 * k + 2], r[4 * k + 3]);
          e[k] = edge(col[k], x, y);
        }
        float wr = e[0] + e[1];
        wr = wr + e[2];
#pragma unroll
        for (int k = 0; k < 3; ++k) b[k] = e[k] / wr;
        if constexpr (NV > 0) {
          if (from) {
            if (args().target) {
#pragma unroll
              for (int c = 0; c < 3; ++c) dcol[c] = args().l2_scale * (dcol[c] - tgt[c]);
            }
            float n[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) n[c] = interp(b, vary[c], vary[3 + c], vary[6 + c]);
            ShadeBwd<SHADER>::run(args().in, scene(), args().gr, vary, n, b, light, dcol, g,
                                  sg, s);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              db[k] = dot3(g.dn, vary + 3 * k);
#pragma unroll
              for (int c = 0; c < 3; ++c) run[R_VAR + 3 * k + c] += b[k] * g.dn[c];
            }
          }
        }
        // b = e / sum(e)
        const float tdb = (db[0] * e[0] + db[1] * e[1]) + db[2] * e[2];
        const float all = tdb / (wr * wr);
        float de[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) de[k] = db[k] / wr - all;
        // zbuffer = (sum_k e_k z_k) * vp22 + vp23
        if constexpr (DZ) {
          const float dz = args().d_zbuffer[pix], vp22 = scene().viewport[10];
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            de[k] += dz * vp22 * col[k].w;
            run[R_Z + k] += dz * vp22 * e[k];
          }
          float zc = e[0] * col[0].w;
          zc = zc + e[1] * col[1].w;
          zc = zc + e[2] * col[2].w;
          sg[NSH] += dz * zc;
          sg[NSH + 1] += dz;
        }
        // e_k = x Minv[0][k] + y Minv[1][k] + Minv[2][k]
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          run[A_MINV + k] += x * de[k];
          run[A_MINV + 3 + k] += y * de[k];
          run[A_MINV + 6 + k] += de[k];
        }
        if constexpr (DARBOUX) {
#pragma unroll
          for (int k = 0; k < 15; ++k) run[R_TRI + k] += g.more[k];
        }
      }
      if constexpr (NV > 9) {
        const bool tex = g.u >= 0 && args().gr.d_textures;
        const int64_t m = (int64_t)g.u * scene().tex_h + g.v;
        if (scene().tex_c == 1) g.tex_g[0] = (g.tex_g[0] + g.tex_g[1]) + g.tex_g[2];
        if (!huge) {
          const int32_t key = tex ? (int32_t)(uint32_t)m : -1;
          if (key != tex_key) {
            if (tex_key != -1) tex_tab.add(tex_key, tex_sum, add_texel);
            tex_key = key;
#pragma unroll
            for (int c = 0; c < NT; ++c) tex_sum[c] = 0.0f;
          }
#pragma unroll
          for (int c = 0; c < 3; ++c) tex_sum[c] += tex ? g.tex_g[c] : 0.0f;
          if constexpr (REFLECT) tex_sum[NT - 1] += one_map ? g.spec_g : 0.0f;
        } else if (tex) {
          for (int c = 0; c < 3; ++c) texel_at(m, c, g.tex_g[c]);
        }
        if constexpr (REFLECT || DARBOUX) {
          if (g.us >= 0 && (huge || !one_map)) {
            const int64_t k = (int64_t)g.us * (DARBOUX ? scene().nmap_h : scene().spec_h) + g.vs;
            const float* mg = DARBOUX ? g.nmap_g : &g.spec_g;
            if (!huge) {
              map_tab.add((int32_t)(uint32_t)k, mg, add_entry);
            } else {
              for (int c = 0; c < N2; ++c) entry_at(k, c, mg[c]);
            }
          }
        }
      }
    }
    // The lanes' last runs: most end here, together.  An LDS atomic of n lanes on
    // one triangle takes the LDS n turns for each of the sums, so a triangle that
    // at least kShared lanes end on is summed across the wavefront first, and its
    // sums are added by a lane each.  The search is bounded: a wavefront of small
    // triangles has none to find.
    {
      uint64_t left = __ballot(run_slot != 255u);
      for (int n = 0; n < kSearched && __popcll(left) >= kShared; ++n) {
        const uint32_t one = __builtin_amdgcn_readlane(run_slot, __builtin_ctzll(left));
        const uint64_t same = __ballot(run_slot == one);
        left &= ~same;
        if (__popcll(same) < kShared) continue;
        const bool in = run_slot == one;
        constexpr int N1 = NR < 32 ? NR : 18;
        float v[N1];
#pragma unroll
        for (int k = 0; k < N1; ++k) v[k] = in ? run[k] : 0.0f;
        const float tot = wave_totals(v);
        if ((lane & 1) == 0 && (lane >> 1) < N1) atomicAdd(&acc[one][lane >> 1], tot);
        if constexpr (NR > N1) {
          float w[NR - N1];
#pragma unroll
          for (int k = 0; k < NR - N1; ++k) w[k] = in ? run[N1 + k] : 0.0f;
          const float more = wave_totals(w);
          if ((lane & 1) == 0 && (lane >> 1) < NR - N1)
            atomicAdd(&acc[one][N1 + (lane >> 1)], more);
        }
        if (in) run_slot = 255u;
      }
    }
    flush_tri();
    read_again();
    __syncthreads();
    // the round's sums to memory: lanes take consecutive accumulators of a
    // triangle's row, so that the addresses of one atomic instruction fall in
    // few cache lines
    if (lane < nt) args().touched[ids[lane]] = s + 1;
    for (int idx = lane; idx < nt * NR; idx += 64) {
      const int e = idx / NR, r = idx - e * NR;
      const int32_t t = ids[e];
      const float v = acc[e][r];
      const int k = r < R_VAR ? r : r < R_Z ? r - R_VAR + A_VAR
                                : r < R_TRI ? r - R_Z + A_Z : r - R_TRI + A_TRI;
      if (v != 0.0f) atomicAdd(args().tacc + (int64_t)t * ACC + k, v);
    }
    __syncthreads();  // the next round writes over what was read here
  }
  if constexpr (NV > 9) {
    // the lanes' last runs, as the triangles' above
    uint64_t left = __ballot(tex_key != -1);
    for (int n = 0; n < kTexSearched && __popcll(left) >= kTexShared; ++n) {
      const int32_t one = __builtin_amdgcn_readlane(tex_key, __builtin_ctzll(left));
      const uint64_t same = __ballot(tex_key == one);
      left &= ~same;
      if (__popcll(same) < kTexShared) continue;
      const bool in = tex_key == one;
      float v[NT];
#pragma unroll
      for (int c = 0; c < NT; ++c) v[c] = in ? tex_sum[c] : 0.0f;
      const float tot = wave_totals(v);
#pragma unroll
      for (int c = 0; c < NT; ++c)
        v[c] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tot), 2 * c));
      if (lane == 0) tex_tab.add(one, v, add_texel);
      if (in) tex_key = -1;
    }
    if (tex_key != -1) tex_tab.add(tex_key, tex_sum, add_texel);
    __syncthreads();
    tex_tab.flush(add_texel);
    if constexpr (REFLECT || DARBOUX)
      if (!one_map) map_tab.flush(add_entry);
  }
  // per-scene parameters: one reduction per wavefront, lane 2 j taking sum j.  The
  // pixels summed the cotangent of normalise(S_DIR's direction); normalise's
  // backward is linear in it, so it is applied to the sum.
  if (!args().gr.d_scene) return;
  float* row = args().gr.d_scene + (int64_t)s * JR_DSCENE_FLOATS;
  if constexpr (NSG > 0) {
    const float tot = wave_totals(sg);
    auto sum_of = [&](int j) {
      return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tot), 2 * j));
    };
    const int j = lane >> 1, q = j - 3 * (j / 3), group = j - q;
    const bool mine = (lane & 1) == 0;
    float v = tot;
    int at = -1;
    if (j >= NSH) {
      at = JR_DSCENE_VIEWPORT + 10 + j - NSH;
    } else if (group == S_DIR) {
      const float dy[3] = {sum_of(S_DIR), sum_of(S_DIR + 1), sum_of(S_DIR + 2)};
      float d[3] = {0.0f, 0.0f, 0.0f};
      if (dy[0] != 0.0f || dy[1] != 0.0f || dy[2] != 0.0f)
        normalise_bwd(REFLECT ? scene().light_dir_eye : scene().light_direction, dy, d);
      v = q == 0 ? d[0] : q == 1 ? d[1] : d[2];
      at = (REFLECT ? JR_DSCENE_LIGHT_DIR_EYE : JR_DSCENE_LIGHT_DIRECTION) + q;
    } else if (REFLECT && group == S_DIFFUSE) {
      v = tot * scene().light_colour[q];
      at = JR_DSCENE_DIFFUSE + q;
    } else if (REFLECT && group == S_SPECULAR) {
      v = tot * scene().light_colour[q];
      at = JR_DSCENE_SPECULAR + q;
    } else if (REFLECT && group == S_AMBIENT) {
      at = JR_DSCENE_AMBIENT + q;
    } else if (REFLECT && group == S_STRENGTH) {
      at = JR_DSCENE_SHADOW_STRENGTH + q;
    } else {
      at = JR_DSCENE_LIGHT_COLOUR + q;
    }
    if (mine && j < NSG && v != 0.0f) atomicAdd(row + at, v);
    if constexpr (REFLECT) {  // the light's colour, by the diffuse sums' lanes
      const float spec = __shfl(tot, (lane + 2 * (S_SPECULAR - S_DIFFUSE)) & 63);
      v = fmaf(scene().diffuse[q], tot, scene().specular[q] * spec);
      if (mine && j < NSH && group == S_DIFFUSE && v != 0.0f)
        atomicAdd(row + JR_DSCENE_LIGHT_COLOUR + q, v);
    }
  }
}

// vertex-stage backward of one slot for its varying cotangent dv: the
// gradient dn of the slot's normal row *nrow_out (and for gouraud dc of its
// colour row *crow_out; rows stay -1 when there is nothing to add).  dE: the
// sums of the light's direction and colour for the shaders lit here, else of the
// 3x3 rotation of world_to_eye_norm.
template <int SHADER>
JR_DEV void vertex_bwd(const BwdArgs& a, const jr_scene& sc, int32_t slot, const float dv[3],
                       float* dE, int64_t* nrow_out, float dn[3], int64_t* crow_out,
                       float dc[3]) {
  if (SHADER == JR_SHADER_DEPTH) return;
  if (dv[0] == 0.0f && dv[1] == 0.0f && dv[2] == 0.0f) return;
  const jr_inputs& in = a.in;
  const int32_t nrow = attr_row(in.nrm_index, slot);
  float n[3], nn[3];
  load3(in.normals, nrow, n);
  normalise3(n, nn);
  float dnn[3];
  if (SHADER == JR_SHADER_GOURAUD || SHADER == JR_SHADER_GOURAUD_TEXTURE) {
    float ln[3];
    normalise3(sc.light_direction, ln);
    const float it = dot3(nn, ln);
    float dI = 0.0f;
    if (SHADER == JR_SHADER_GOURAUD) {
      const int32_t crow = attr_row(in.col_index, slot);
      float col[3];
      load3(in.colours, crow, col);
      *crow_out = crow;
      for (int q = 0; q < 3; ++q) {
        dc[q] = dv[q] * sc.light_colour[q] * it;
        dE[3 + q] += dv[q] * col[q] * it;
        dI += dv[q] * col[q] * sc.light_colour[q];
      }
    } else {
      for (int q = 0; q < 3; ++q) {
        dE[3 + q] += dv[q] * it;
        dI += dv[q] * sc.light_colour[q];
      }
    }
    float dln[3], dL[3];
    for (int q = 0; q < 3; ++q) {
      dnn[q] = dI * ln[q];
      dln[q] = dI * nn[q];
    }
    normalise_bwd(sc.light_direction, dln, dL);
    for (int q = 0; q < 3; ++q) dE[q] += dL[q];
  } else {
    // ne = normalise((E @ [normalise(nn), 0])[:3])  (Camera.apply_vec)
    float u2[3];
    normalise3(nn, u2);
    float h[4];
    apply4(sc.world_to_eye_norm, u2[0], u2[1], u2[2], 0.0f, h);
    const float t3[3] = {h[0], h[1], h[2]};
    float dt3[3], du2[3], du1[3];
    normalise_bwd(t3, dv, dt3);
    for (int jj = 0; jj < 3; ++jj) {
      float s = 0.0f;
      for (int ii = 0; ii < 3; ++ii) {
        s += sc.world_to_eye_norm[4 * ii + jj] * dt3[ii];
        dE[3 * ii + jj] += dt3[ii] * u2[jj];
      }
      du2[jj] = s;
    }
    normalise_bwd(nn, du2, du1);
    for (int q = 0; q < 3; ++q) dnn[q] = du1[q];
  }
  normalise_bwd(n, dnn, dn);
  *nrow_out = nrow;
}

// Adds each lane's 3-float row g at d + 3 row (row < 0: nothing) with
// neighbouring lanes on the three floats of one row, so the adds of an atomic
// instruction share cache lines.  W: the wavefront's LDS staging; call with
// every lane of the wavefront.
struct WaveRows {
  int64_t at[64];
  float v[64][3];
};
JR_DEV void wave_row_adds(WaveRows& W, float* __restrict__ d, int64_t row, const float g[3]) {
  const int lane = threadIdx.x & 63;
  W.at[lane] = row;
  W.v[lane][0] = g[0];
  W.v[lane][1] = g[1];
  W.v[lane][2] = g[2];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int it = 0; it < 3; ++it) {
    const int idx = lane + 64 * it;
    const int e = idx / 3, c = idx - 3 * e;
    const int64_t r = W.at[e];
    const float x = W.v[e][c];
    if (r >= 0 && x != 0.0f) atomicAdd(d + 3 * r + c, x);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Triangle t (-1: none) of the calling lane; the accumulators are read and
// cleared only when `touched`.  Every lane computes its scene, so that a
// wavefront of one scene reduces its camera and light gradients once.
template <int SHADER>
JR_DEV void bwd_tri(const BwdArgs& a, int32_t t, int32_t s, bool touched, WaveRows& W) {
  // gradients of the scene's parameters: world_to_clip, the rotation of
  // world_to_eye_norm (or the light of a vertex-lit shader) and the viewport's
  // entries 0, 3, 5, 7
  constexpr bool LIT = SHADER == JR_SHADER_GOURAUD || SHADER == JR_SHADER_GOURAUD_TEXTURE;
  constexpr int NE = SHADER == JR_SHADER_DEPTH ? 0 : LIT ? 6 : 9;
  float dS[16 + 4 + NE];
#pragma unroll
  for (int q = 0; q < 16 + 4 + NE; ++q) dS[q] = 0.0f;
  float* dW = dS;
  float* dV = dS + 16;
  float* dE = dS + 20;
  if (__ballot(touched) == 0) return;  // nothing to add for this wavefront
  if (!touched) s = -1;
  constexpr int ACC = AccOf<SHADER>::N;
  float v[ACC];
  bool live = false;
  TriSetup ts;
  float dM[9];
  if (touched) {
    float* A = a.tacc + (int64_t)t * ACC;
    for (int q = 0; q < ACC; ++q) {
      v[q] = A[q];
      A[q] = 0.0f;
      live = live || (v[q] != 0.0f);
    }
    a.touched[t] = 0;
    if (live) {
      tri_setup(a.in, a.scenes[s], t, ts);
      // X = M^-1, G = dL/dX: dL/dM = -X^T G X^T
      const float* X = ts.Mi;
      float XtG[9];
      for (int p = 0; p < 3; ++p)
        for (int k = 0; k < 3; ++k) {
          float s2 = 0.0f;
          for (int r = 0; r < 3; ++r) s2 += X[3 * r + p] * v[A_MINV + 3 * r + k];
          XtG[3 * p + k] = s2;
        }
      for (int p = 0; p < 3; ++p)
        for (int q = 0; q < 3; ++q) {
          float s2 = 0.0f;
          for (int k = 0; k < 3; ++k) s2 += XtG[3 * p + k] * X[3 * q + k];
          dM[3 * p + q] = -s2;
        }
      // x = (i - vp03) / vp00, y = (j - vp13) / vp11: with dx = sum_k X[0][k] de_k at
      // a pixel, sum x dx = sum_k X[0][k] G[0][k] and sum dx = sum_k X[0][k] G[2][k]
      for (int k = 0; k < 3; ++k) {
        dV[0] -= X[k] * v[A_MINV + k];
        dV[1] -= X[k] * v[A_MINV + 6 + k];
        dV[2] -= X[3 + k] * v[A_MINV + 3 + k];
        dV[3] -= X[3 + k] * v[A_MINV + 6 + k];
      }
      const float* vp = a.scenes[s].viewport;
      dV[0] /= vp[0];
      dV[1] /= vp[0];
      dV[2] /= vp[5];
      dV[3] /= vp[5];
    }
  }
  // corner by corner, the lanes' position / normal / colour rows added
  // together (wave_row_adds), every lane taking part
  for (int k = 0; k < 3; ++k) {
    int64_t prow = -1, nrow = -1, crow = -1;
    float dp[3] = {0.0f, 0.0f, 0.0f}, dn[3] = {0.0f, 0.0f, 0.0f}, dc[3] = {0.0f, 0.0f, 0.0f};
    if (live) {
      const jr_scene& sc = a.scenes[s];
      const int32_t slot = face_slot(a.in, t, k);
      const float dclip[4] = {dM[3 * k + 0], dM[3 * k + 1], v[A_Z + k], dM[3 * k + 2]};
      prow = attr_row(a.in.pos_index, slot);
      float p[3];
      load3(a.in.positions, prow, p);
      const float ph[4] = {p[0], p[1], p[2], 1.0f};
      for (int jj = 0; jj < 4; ++jj) {
        float s2 = 0.0f;
        for (int ii = 0; ii < 4; ++ii) {
          s2 += sc.world_to_clip[4 * ii + jj] * dclip[ii];
          dW[4 * ii + jj] += dclip[ii] * ph[jj];
        }
        if (jj < 3) dp[jj] = s2;
      }
      const float dv[3] = {v[A_VAR + 3 * k], v[A_VAR + 3 * k + 1], v[A_VAR + 3 * k + 2]};
      vertex_bwd<SHADER>(a, sc, slot, dv, dE, &nrow, dn, &crow, dc);
    }
    if (a.gr.d_positions) wave_row_adds(W, a.gr.d_positions, prow, dp);
    if constexpr (SHADER != JR_SHADER_DEPTH)
      if (a.gr.d_normals) wave_row_adds(W, a.gr.d_normals, nrow, dn);
    if constexpr (SHADER == JR_SHADER_GOURAUD)
      if (a.gr.d_colours) wave_row_adds(W, a.gr.d_colours, crow, dc);
  }
  if (live) {
    {
      const jr_scene& sc = a.scenes[s];
      if constexpr (SHADER == JR_SHADER_PHONG_DARBOUX) {
        // the face of slot 0 (id_to_face) whose NDC corners and uvs built the
        // tangent frame: t_m = to_cartesian(h_m), h_m = world_to_clip @ [p_m, 1]
        const int32_t face = a.in.id_to_face[face_slot(a.in, t, 0)];
        for (int m = 0; m < 3; ++m) {
          const int32_t q = a.in.face_slots[3 * (int64_t)face + m];
          const float* dt = v + A_TRI + 3 * m;
          if (dt[0] != 0.0f || dt[1] != 0.0f || dt[2] != 0.0f) {
            const int32_t prow = attr_row(a.in.pos_index, q);
            float p[3], h[4];
            load3(a.in.positions, prow, p);
            position_clip(a.in, sc.world_to_clip, q, h);
            // where(w == 0, h[:3], h[:3] / w): x / w has d/dx = 1 / w and
            // d/dw = -x / w^2
            float dh[4];
            if (h[3] == 0.0f) {
              dh[0] = dt[0];
              dh[1] = dt[1];
              dh[2] = dt[2];
              dh[3] = 0.0f;
            } else {
              float dw = 0.0f;
              for (int c = 0; c < 3; ++c) {
                dh[c] = dt[c] / h[3];
                dw += -dt[c] * h[c] / (h[3] * h[3]);
              }
              dh[3] = dw;
            }
            const float ph[4] = {p[0], p[1], p[2], 1.0f};
            for (int jj = 0; jj < 4; ++jj) {
              float s2 = 0.0f;
              for (int ii = 0; ii < 4; ++ii) {
                s2 += sc.world_to_clip[4 * ii + jj] * dh[ii];
                dW[4 * ii + jj] += dh[ii] * ph[jj];
              }
              if (jj < 3 && a.gr.d_positions)
                atomicAdd(a.gr.d_positions + 3 * (int64_t)prow + jj, s2);
            }
          }
          const float* du = v + A_TUV + 2 * m;
          if (a.gr.d_uvs && (du[0] != 0.0f || du[1] != 0.0f)) {
            const int32_t urow = attr_row(a.in.uv_index, q);
            atomicAdd(a.gr.d_uvs + 2 * (int64_t)urow, du[0]);
            atomicAdd(a.gr.d_uvs + 2 * (int64_t)urow + 1, du[1]);
          }
        }
      }
    }
  }
  if (!a.gr.d_scene) return;
  // where dS[j] goes in a d_scene row
  auto slot_of = [&](int j) {
    if (j < 16) return JR_DSCENE_WORLD_TO_CLIP + j;
    if (j < 20)  // 0, 3, 5, 7
      return JR_DSCENE_VIEWPORT + (j == 16 ? 0 : 2 * (j - 16) + 1);
    const int k = j - 20;
    if (LIT)
      return k < 3 ? JR_DSCENE_LIGHT_DIRECTION + k : JR_DSCENE_LIGHT_COLOUR + k - 3;
    return JR_DSCENE_WORLD_TO_EYE_NORM + k + k / 3;  // 3x3 of a 4x4
  };
  // reduce over the wave when it holds one scene, else per lane
  const int32_t s0 = __shfl(s, 0);
  const bool uniform = __ballot(s == s0 || s < 0) == __ballot(true) && s0 >= 0;
  if (uniform) {
    const int lane = threadIdx.x & 63;
    const float tot = wave_totals(dS);
    if ((lane & 1) == 0 && (lane >> 1) < 20 + NE && tot != 0.0f)
      atomicAdd(a.gr.d_scene + (int64_t)s0 * JR_DSCENE_FLOATS + slot_of(lane >> 1), tot);
  } else if (s >= 0) {
    float* row = a.gr.d_scene + (int64_t)s * JR_DSCENE_FLOATS;
#pragma unroll
    for (int j = 0; j < 20 + NE; ++j)
      if (dS[j] != 0.0f) atomicAdd(row + slot_of(j), dS[j]);
  }
}

// One thread per triangle: the touched ones (flag = scene + 1) are packed to
// the front of the workgroup, read their accumulators and clear them with the
// flag for the next call; wavefronts left without one return at once.  At
// most 80 VGPRs (6 wavefronts per SIMD instead of 5): the kernel waits on its
// gathers most of the time, and more wavefronts hide more of that.
template <int SHADER>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6, 8)))
void k_bwd_tris(BwdArgs a) {
  __shared__ int2 items[256];
  __shared__ int32_t wave_n[4];
  __shared__ WaveRows rows[4];
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t flag = t < a.in.n_tris ? a.touched[t] : 0;
  const uint64_t bal = __ballot(flag != 0);
  if ((threadIdx.x & 63) == 0) wave_n[threadIdx.x >> 6] = __popcll(bal);
  __syncthreads();
  int32_t pos = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
  for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) pos += wave_n[w];
  if (flag != 0) items[pos] = make_int2(t, flag - 1);
  __syncthreads();
  const int32_t n = wave_n[0] + wave_n[1] + wave_n[2] + wave_n[3];
  const bool has = (int32_t)threadIdx.x < n;
  const int2 it = has ? items[threadIdx.x] : make_int2(-1, -1);
  bwd_tri<SHADER>(a, it.x, it.y, has, rows[threadIdx.x >> 6]);
}

// Reads the workspace header: if it does not describe this workspace (new,
// resized, or used for another triangle count or accumulator size), asks
// k_bwd_fill to clear the flags and accumulators.
__global__ void k_bwd_prepare(uint32_t* __restrict__ hdr, int32_t n_tris, int32_t acc) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const bool ok = hdr[kHdrMagicLo] == kMagicLo && hdr[kHdrMagicHi] == kMagicHi &&
                  hdr[kHdrTris] == (uint32_t)n_tris && hdr[kHdrAcc] == (uint32_t)acc;
  hdr[kHdrFill] = ok ? 0u : 1u;
  hdr[kHdrMagicLo] = kMagicLo;
  hdr[kHdrMagicHi] = kMagicHi;
  hdr[kHdrTris] = (uint32_t)n_tris;
  hdr[kHdrAcc] = (uint32_t)acc;
}

// Zeroes n 32-bit words after the header when k_bwd_prepare asked for it.
__global__ void k_bwd_fill(const uint32_t* __restrict__ hdr, uint32_t* __restrict__ p,
                           int64_t n) {
  if (hdr[kHdrFill] == 0u) return;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}


thread_local std::string g_bwd_err;

int32_t bfail(int32_t code, const char* msg) {
  g_bwd_err = msg;
  return code;
}

template <int SHADER>
void launch_bwd(const BwdArgs& a, int ppl, hipStream_t st) {
  const int64_t n_waves = (int64_t)a.T * a.n_scenes;
  const dim3 grid((unsigned)n_waves);
  if (a.d_zbuffer && ppl == 4)
    hipLaunchKernelGGL((k_bwd_pixels<SHADER, true, 4>), grid, dim3(64), 0, st, a);
  else if (a.d_zbuffer)
    hipLaunchKernelGGL((k_bwd_pixels<SHADER, true, 2>), grid, dim3(64), 0, st, a);
  else if (ppl == 4)
    hipLaunchKernelGGL((k_bwd_pixels<SHADER, false, 4>), grid, dim3(64), 0, st, a);
  else
    hipLaunchKernelGGL((k_bwd_pixels<SHADER, false, 2>), grid, dim3(64), 0, st, a);
  hipLaunchKernelGGL(k_bwd_tris<SHADER>, dim3((a.in.n_tris + 255) / 256), dim3(256), 0, st, a);
}

// Workspace: header (256 B), touched flags (4 B per triangle), accumulators
// (4 acc_floats(shader) B per triangle).
struct BwdLayout {
  int64_t touched, tacc, total;
};

BwdLayout bwd_layout(int32_t n_tris, int shader) {
  const int64_t n = std::max(n_tris, 1);
  BwdLayout L;
  L.touched = 256;
  L.tacc = L.touched + (4 * n + 255) / 256 * 256;
  L.total = L.tacc + (4 * (int64_t)acc_floats(shader) * n + 255) / 256 * 256;
  return L;
}

}  // namespace jr

using namespace jr;

extern "C" {

int64_t jr_backward_workspace_size(const jr_frame* frame, int32_t n_tris) {
  if (!frame || n_tris < 0) return -1;
  return bwd_layout(n_tris, frame->shader).total;
}

const char* jr_backward_last_error(void) { return g_bwd_err.c_str(); }

}  // extern "C"

namespace jr {
namespace {

// jr_backward and jr_backward_l2: the canvas cotangent is d_canvas, or
// l2_scale * (canvas - target) when target is set.
int32_t backward_body(const jr_frame* fr, const jr_inputs* in, const jr_scene* scenes,
                      const float* d_canvas, const float* canvas, const float* target,
                      float l2_scale, const float* d_zbuffer, const int32_t* prim_id,
                      jr_grads* grads, void* workspace, int64_t workspace_bytes,
                      jr_stream_t stream_) {
  if (!fr || !in || !scenes || !grads || !prim_id)
    return bfail(JR_E_INVALID, "frame, inputs, scenes, grads and prim_id are required");
  if (fr->width <= 0 || fr->height <= 0 || fr->n_scenes <= 0 || in->n_tris < 0)
    return bfail(JR_E_INVALID, "bad frame sizes");
  if (in->clip) return bfail(JR_E_UNSUPPORTED, "backward needs positions, not clip input");
  const int sh = fr->shader;
  if (sh == JR_SHADER_VISIBILITY || sh < 0 || sh >= JR_SHADER_COUNT)
    return bfail(JR_E_UNSUPPORTED, "shader has no backward pass");
  if (!d_canvas && !target && !d_zbuffer) return bfail(JR_E_INVALID, "no upstream gradient");
  if (!in->positions) return bfail(JR_E_INVALID, "positions are required");
  if (!in->faces && (int64_t)in->n_slots < 3 * (int64_t)in->n_tris)
    return bfail(JR_E_INVALID, "without faces, n_slots must be at least 3 n_tris");
  if (sh == JR_SHADER_GOURAUD && (!in->normals || !in->colours))
    return bfail(JR_E_INVALID, "gouraud needs normals and colours");
  if ((sh == JR_SHADER_GOURAUD_TEXTURE || sh == JR_SHADER_PHONG ||
       sh == JR_SHADER_PHONG_DARBOUX || sh == JR_SHADER_PHONG_REFLECTION ||
       sh == JR_SHADER_PHONG_REFLECTION_SHADOW) &&
      (!in->normals || !in->uvs || !in->textures))
    return bfail(JR_E_INVALID, "textured shaders need normals, uvs and textures");
  if (sh == JR_SHADER_PHONG_DARBOUX && (!in->id_to_face || !in->face_slots || !in->normal_maps))
    return bfail(JR_E_INVALID, "phong_darboux needs id_to_face, face_slots and normal_maps");
  if ((sh == JR_SHADER_PHONG_REFLECTION || sh == JR_SHADER_PHONG_REFLECTION_SHADOW) &&
      (!in->tex_index || !in->texture_shapes || !in->specular_maps))
    return bfail(JR_E_INVALID, "phong_reflection needs tex_index, texture_shapes, specular_maps");
  if (sh == JR_SHADER_PHONG_REFLECTION_SHADOW &&
      (!in->shadow_maps || in->shadow_w <= 0 || in->shadow_h <= 0))
    return bfail(JR_E_INVALID, "phong_reflection_shadow needs shadow maps");
  const int64_t need = jr_backward_workspace_size(fr, in->n_tris);
  if (!workspace || workspace_bytes < need) return bfail(JR_E_WORKSPACE, "workspace too small");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream_);
  BwdArgs a;
  a.in = *in;
  a.scenes = scenes;
  a.gr = *grads;
  a.d_canvas = (sh == JR_SHADER_DEPTH) ? nullptr : d_canvas;
  a.canvas = canvas;
  a.target = (sh == JR_SHADER_DEPTH) ? nullptr : target;
  a.l2_scale = l2_scale;
  a.d_zbuffer = d_zbuffer;
  a.prim_id = prim_id;
  const BwdLayout WL = bwd_layout(in->n_tris, sh);
  char* ws = static_cast<char*>(workspace);
  a.header = reinterpret_cast<uint32_t*>(ws);
  a.touched = reinterpret_cast<int32_t*>(ws + WL.touched);
  a.tacc = reinterpret_cast<float*>(ws + WL.tacc);
  a.W = fr->width;
  a.H = fr->height;
  a.n_scenes = fr->n_scenes;
  // Four pixels per lane (16 x 16 tiles) or two (8 x 16).  Two halve a wavefront's
  // chain of lookups and its triangles, for half as many pixels to pay for them: the
  // faster one where the 16 x 16 tiles, partial ones included, are few rounds of the
  // 4,096 wavefronts that the chip holds and a tile has triangles to set up (23 views
  // of 201x187, 3,588 tiles, 190 -> 167 us; 64 of 256x256 and 256 scenes of 128x128,
  // 16,384 each, 411 -> 381 and 790 -> 759 us), but not where there are more (1,024 of
  // 84x84, 36,864 tiles packed into 28,672 wavefronts, 1,399 against 1,428 us; 512 of
  // 480x270, 261,120, 4,100 against 4,480 us) or the triangles are larger (64 views of a
  // 200-triangle ball 258 against 274).  The line is six rounds of tiles, between the
  // largest measured gain and the smallest measured loss.  With a depth gradient, the
  // backward alone: 16 scenes of 100x75 139 -> 99 us, 256 of 84x84 311 -> 251, 64 phong
  // views of 256x256 297 -> 250, 4 of 128x128 108 -> 68.
  const int64_t tiles4 = (int64_t)((a.W + 15) / 16) * ((a.H + 15) / 16) * a.n_scenes;
  const int ppl = tiles4 <= 24576 && in->n_tris >= 4 * tiles4 ? 2 : 4;
  const int64_t QW = (a.W + ppl / 2 - 1) / (ppl / 2), QH = (a.H + 1) / 2, nq = QW * QH;
  const int64_t tiles_y = (QH + 7) / 8, tiles = (QW + 7) / 8 * tiles_y;
  // the leftover blocks are packed where that saves at least an eighth of the
  // wavefronts (84 x 84: 28 instead of 36, fwd+bwd 1.58 -> 1.52 ms on 1024
  // scenes); where it saves few (480 x 270: 507 instead of 510) plain tiles,
  // partial ones included, measured faster (the backward 3.88 against 3.98 ms
  // on 512 scenes).  Plain tiles are the first kind of block with FY = tiles_y
  // and every wavefront's blocks counted as a full tile's.
  const bool packed = 8 * ((nq + 63) / 64) <= 7 * tiles;
  const int64_t T = packed ? (nq + 63) / 64 : tiles;
  // block numbers (below 64 T) and wavefront numbers stay below 2^31
  if (64 * T > 0x7FFFFFFFLL || T * a.n_scenes > 0x7FFFFFFFLL)
    return bfail(JR_E_INVALID, "too many pixels");
  a.T = (int32_t)T;
  if (packed) {
    a.nq = (int32_t)nq;
    a.FX = (int32_t)(QW / 8);
    a.FY = (int32_t)(QH / 8);
    a.rw = (int32_t)(QW % 8);
    a.rh = (int32_t)(QH % 8);
    a.full_end = 64 * a.FX * a.FY;
    a.bottom_end = a.full_end + 8 * a.FX * a.rh;
  } else {
    a.nq = a.full_end = a.bottom_end = (int32_t)(64 * T);
    a.FX = (int32_t)(tiles / tiles_y);
    a.FY = (int32_t)tiles_y;
    a.rw = a.rh = 0;
  }
  magic31((uint32_t)a.T, &a.T_m, &a.T_sh);
  magic31((uint32_t)std::max(a.FY, 1), &a.fy_m, &a.fy_sh);
  magic31((uint32_t)std::max(a.rh, 1), &a.rh_m, &a.rh_sh);
  magic31((uint32_t)std::max(a.rw, 1), &a.rw_m, &a.rw_sh);
  if (in->n_tris == 0) return JR_OK;
  // flags and accumulators: everything after the header
  const int64_t nwords = (WL.total - WL.touched) / 4;
  hipLaunchKernelGGL(k_bwd_prepare, dim3(1), dim3(64), 0, st, a.header, in->n_tris,
                     acc_floats(sh));
  hipLaunchKernelGGL(k_bwd_fill, dim3((unsigned)std::min<int64_t>((nwords + 255) / 256, 8192)),
                     dim3(256), 0, st, a.header,
                     reinterpret_cast<uint32_t*>(ws + WL.touched), nwords);
  switch (sh) {
    case JR_SHADER_DEPTH: launch_bwd<JR_SHADER_DEPTH>(a, ppl, st); break;
    case JR_SHADER_GOURAUD: launch_bwd<JR_SHADER_GOURAUD>(a, ppl, st); break;
    case JR_SHADER_GOURAUD_TEXTURE: launch_bwd<JR_SHADER_GOURAUD_TEXTURE>(a, ppl, st); break;
    case JR_SHADER_PHONG: launch_bwd<JR_SHADER_PHONG>(a, ppl, st); break;
    case JR_SHADER_PHONG_DARBOUX: launch_bwd<JR_SHADER_PHONG_DARBOUX>(a, ppl, st); break;
    case JR_SHADER_PHONG_REFLECTION: launch_bwd<JR_SHADER_PHONG_REFLECTION>(a, ppl, st); break;
    default: launch_bwd<JR_SHADER_PHONG_REFLECTION_SHADOW>(a, ppl, st); break;
  }
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return bfail(JR_E_HIP, hipGetErrorString(err));
  return JR_OK;
}

}  // namespace
}  // namespace jr

extern "C" {

int32_t jr_backward(const jr_frame* fr, const jr_inputs* in, const jr_scene* scenes,
                    const float* d_canvas, const float* d_zbuffer, const int32_t* prim_id,
                    jr_grads* grads, void* workspace, int64_t workspace_bytes,
                    jr_stream_t stream) {
  return backward_body(fr, in, scenes, d_canvas, nullptr, nullptr, 0.0f, d_zbuffer, prim_id,
                       grads, workspace, workspace_bytes, stream);
}

int32_t jr_backward_l2(const jr_frame* fr, const jr_inputs* in, const jr_scene* scenes,
                       const float* canvas, const float* target, float scale,
                       const float* d_zbuffer, const int32_t* prim_id, jr_grads* grads,
                       void* workspace, int64_t workspace_bytes, jr_stream_t stream) {
  if (!canvas || !target) return bfail(JR_E_INVALID, "canvas and target are required");
  return backward_body(fr, in, scenes, nullptr, canvas, target, scale, d_zbuffer, prim_id,
                       grads, workspace, workspace_bytes, stream);
}

}  // extern "C"
