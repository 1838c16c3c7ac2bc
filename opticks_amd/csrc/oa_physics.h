/*
 * oa_physics.h : qsim propagation physics, photon generation and world trace
 * for gfx950. Function-by-function counterparts:
 *   fill                 qbnd::fill_state            qudarap/qbnd.h:192-223
 *   to_boundary          qsim::propagate_to_boundary qudarap/qsim.h:721-866
 *   rayleigh             qsim::rayleigh_scatter      qudarap/qsim.h:604-692
 *   at_boundary          qsim::propagate_at_boundary qudarap/qsim.h:1001-1208
 *   at_surface           qsim::propagate_at_surface  qudarap/qsim.h:1680-1758
 *   reflect_diffuse/specular, lambertian, marsaglia  qudarap/qsim.h:433-575,1988-2093
 *   propagate            qsim::propagate             qudarap/qsim.h:2229-2338
 *   gen_torch/gen_scint  storch::generate / qscint::generate
 *                        sysrap/storch.h:192-520, qudarap/qscint.h:66-200
 *   trace                optixTrace + IS/CH/MS       CSGOptiX/CSGOptiX7.cu:113-218,682-967
 */
#pragma once
#include "oa_device.h"

namespace oa {

/* ----------------------------------------------------------- tables */

/* Wrap addressing of a table of n texels: i0 = i mod n in [0, n) and its
   neighbour (i0 + 1) mod n. The integer divisions run only for an index
   outside the table (wavelengths beyond the domain), the results are the same. */
__device__ static __attribute__((noinline)) int wrap_index(int i, int n) { return ((i % n) + n) % n; }

OA_D void wrap_pair(int i, int n, int& i0, int& i1)
{
    i0 = i;
    if (i0 < 0 || i0 >= n) i0 = wrap_index(i0, n);
    i1 = i0 + 1 == n ? 0 : i0 + 1;
}

/* One lerped float4 of bnd row (2*line+k) at wavelength nm: the FP32 form of
   the linearly filtered, wrap-addressed texture fetch of qbnd::boundary_lookup. */
OA_D float4 bnd_lookup(const SimParams& P, float nm, int line, int k)
{
    const int nwl = P.n_wl;
    float fx = (nm - P.wl_low) / P.wl_step;
    float fl = floorf(fx);
    float a = fx - fl;
    int i0, i1;
    wrap_pair((int)fl, nwl, i0, i1);
    const float4* row = P.bnd + (int64_t)(2 * line + k) * nwl;
    float4 v0 = row[i0];
    float4 v1 = row[i1];
    return make_float4(v0.x + a * (v1.x - v0.x), v0.y + a * (v1.y - v0.y),
                       v0.z + a * (v1.z - v0.z), v0.w + a * (v1.w - v0.w));
}

struct State {
    float4 material1;     /* n, absorption, scattering, reemission */
    float  group_velocity;
    float  n2;
    float4 surface;       /* detect, absorb, specular, diffuse */
    int    ems;
    int    m1_line;       /* bnd line of the material the photon travels in */
};

/* Segment events reported to a Tape during propagate_to_boundary. */
enum : int { SEG_SAIL = 0, SEG_ABSORB = 1, SEG_SCATTER = 2 };

/* The forward kernels record nothing. Every propagation step makes exactly one
   segment call (propagate -> to_boundary), so a photon's step number is its
   segment number: `at` names it before the step, `finish` gets the count. */
struct NoTape {
    static constexpr bool keeps_seq = true;
    __device__ inline __attribute__((always_inline)) void begin(const SimParams&, int64_t) {}
    __device__ inline __attribute__((always_inline)) void at(const SimParams&, int64_t, int) {}
    __device__ inline __attribute__((always_inline)) void seg(const SimParams&, int, float, float, float, float, int) {}
    __device__ inline __attribute__((always_inline)) void finish(const SimParams&, int64_t, int) {}
};

/* A forward kernel run for a following adjoint keeps, per photon, the arguments
   of its segment calls -- bnd line, segment event, wavelength and segment length
   (the absorption and scattering lengths are the table values at that line and
   wavelength, looked up again when the record is read) -- up to P.tape_k of them,
   and the number it had. The adjoint then scores a hit from its records instead
   of replaying the photon. It adds no per-lane state: it holds the photon index
   and step number the lane keeps anyway, and forms the record address from them
   and the launch's fields only at the store. */
struct RecordTape {
    static constexpr bool keeps_seq = true;
    int64_t g, stride;
    int32_t step;
    __device__ inline __attribute__((always_inline)) void begin(const SimParams& P, int64_t n_photon)
    {
        stride = P.tape_stride ? P.tape_stride : n_photon;
    }
    __device__ inline __attribute__((always_inline)) void at(const SimParams&, int64_t g_, int step_)
    {
        g = g_; step = step_;
    }
    __device__ inline __attribute__((always_inline)) void seg(const SimParams& P, int line, float wl, float, float, float ell,
                                                              int ev)
    {
        if (step < P.tape_k) {
            /* streaming stores: the records are read back only by the adjoint, after the
               launch (0.38 -> 0.31 ms of taping on 10M photons against cached stores) */
            uint32_t* r = P.tape + 3 * ((int64_t)step * stride + g);
            __builtin_nontemporal_store((uint32_t)line | ((uint32_t)ev << 30), &r[0]);
            __builtin_nontemporal_store(__float_as_uint(wl), &r[1]);
            __builtin_nontemporal_store(__float_as_uint(ell), &r[2]);
        }
    }
    __device__ inline __attribute__((always_inline)) void finish(const SimParams& P, int64_t g, int steps)
    {
        P.tape_n[g] = (uint8_t)(steps < 255 ? steps : 255);
    }
};

/* record j of launch-local photon g */
OA_D const uint32_t* tape_record(const SimParams& P, int64_t g, int j)
{
    return P.tape + 3 * ((int64_t)j * P.tape_stride + g);
}

OA_D void fill(const SimParams& P, State& s, uint32_t boundary, float wl, float cosTheta)
{
    const int line = (int)boundary * 4;
    const int m1_line = cosTheta > 0.f ? line + 3 : line + 0;
    const int m2_line = cosTheta > 0.f ? line + 0 : line + 3;
    const int su_line = cosTheta > 0.f ? line + 2 : line + 1;
    s.m1_line = m1_line;
    s.material1 = bnd_lookup(P, wl, m1_line, 0);
    s.group_velocity = bnd_lookup(P, wl, m1_line, 1).x;
    s.n2 = bnd_lookup(P, wl, m2_line, 0).x;
    s.ems = P.optical[4 * su_line + 1];
    s.surface = (s.ems != EMS_NOSURFACE) ? bnd_lookup(P, wl, su_line, 0) : make_float4(0.f, 0.f, 0.f, 0.f);
}

OA_D float icdf_tex(const SimParams& P, float x, int layer)
{
    const int n = P.n_icdf;
    float xb = x * (float)n - 0.5f;
    float fl = floorf(xb);
    float a = xb - fl;
    int i0, i1;
    wrap_pair((int)fl, n, i0, i1);
    int L = layer < P.n_icdf_layer ? layer : 0;
    const float* row = P.icdf + (int64_t)L * n;
    float v0 = row[i0], v1 = row[i1];
    return v0 + a * (v1 - v0);
}

OA_D float scint_wavelength(const SimParams& P, float u0)
{
    if (P.icdf_hd == 0) return icdf_tex(P, u0, 0);
    if (P.icdf_hd == 10) {
        bool lhs = u0 < 0.1f, rhs = u0 > 0.9f;
        float x = lhs ? (u0 * 10.f) : (rhs ? (u0 - 0.9f) * 10.f : u0);
        return icdf_tex(P, x, lhs ? 1 : (rhs ? 2 : 0));
    }
    if (P.icdf_hd == 20) {
        bool lhs = u0 < 0.05f, rhs = u0 > 0.95f;
        float x = lhs ? (u0 * 20.f) : (rhs ? (u0 - 0.95f) * 20.f : u0);
        return icdf_tex(P, x, lhs ? 1 : (rhs ? 2 : 0));
    }
    return 0.f;
}

/* ---------------------------------------------------------- helpers */

OA_D void rotateUz(v3& d, v3 u)   /* sysrap/smath.h:95-115 */
{
    float up = u.x * u.x + u.y * u.y;
    if (up > 0.f) {
        up = sqrtf(up);
        float px = d.x, py = d.y, pz = d.z;
        d.x = (u.x * u.z * px - u.y * py) / up + u.x * pz;
        d.y = (u.y * u.z * px + u.x * py) / up + u.y * pz;
        d.z = -up * px + u.z * pz;
    } else if (u.z < 0.f) {
        d.x = -d.x;
        d.z = -d.z;
    }
}

OA_D v3 uniform_sphere(float u0, float u1)
{
    float phi = u0 * 2.f * OA_PI_F;
    float cosTheta = 2.f * u1 - 1.f;
    float sinTheta = sqrtf(1.f - cosTheta * cosTheta);
    float sp, cp;
    oa_sincosf(phi, &sp, &cp);
    return mk(cp * sinTheta, sp * sinTheta, cosTheta);
}

template <class R>
OA_D void marsaglia(v3& dir, R& rng)
{
    float u, v, b, a;
    int trials = 0;
    do {
        float w[2];
        draw<2>(rng, w);
        u = 2.f * w[0] - 1.f;
        v = 2.f * w[1] - 1.f;
        b = u * u + v * v;
    } while (b > 1.f && ++trials < OA_MAX_TRIALS);
    if (b > 1.f) { u = 0.f; v = 0.f; b = 0.f; }   /* bound reached: (0, 0, -1) */
    a = 2.f * sqrtf(1.f - b);
    dir = mk(a * u, a * v, 2.f * b - 1.f);
}

template <class R>
OA_D void lambertian(v3& dir, v3 normal, float orient, R& rng)
{
    float ndotv, u;
    int count = 0;
    do {
        count++;
        marsaglia(dir, rng);
        ndotv = dot(dir, normal) * orient;
        if (ndotv < 0.f) { dir = -1.f * dir; ndotv = -1.f * ndotv; }
        u = draw1(rng);
    } while (!(u < ndotv) && (count < 1024));
}

/* one trial of the rejection loop of qsim::rayleigh_scatter: whether it is accepted, and the
   direction and polarization it proposes */
OA_D bool rayleigh_trial(const Photon& p, const float (&u)[5], v3& direction, v3& polarization)
{
    const float u0 = u[0], u1 = u[1], u2 = u[2], u3 = u[3], u4 = u[4];
    float cosTheta = u0;
    float sinTheta = sqrtf(1.0f - u0 * u0);
    if (u1 < 0.5f) cosTheta = -cosTheta;
    float sinPhi, cosPhi;
    oa_sincosf(2.f * OA_PI_F * u2, &sinPhi, &cosPhi);
    direction = mk(sinTheta * cosPhi, sinTheta * sinPhi, cosTheta);
    rotateUz(direction, p.mom);
    float constant = -dot(direction, p.pol);
    polarization = mk(p.pol.x + constant * direction.x, p.pol.y + constant * direction.y,
                      p.pol.z + constant * direction.z);
    if (dot(polarization, polarization) == 0.f) {
        oa_sincosf(2.f * OA_PI_F * u3, &sinPhi, &cosPhi);
        polarization = mk(cosPhi, sinPhi, 0.f);
        rotateUz(polarization, direction);
    } else {
        if (u3 < 0.5f) polarization = -polarization;
    }
    polarization = normalize(polarization);
    float doCosTheta = dot(polarization, p.pol);
    return !(doCosTheta * doCosTheta < u4);
}

/* the new direction of a reemitted photon, or one trial of a scattered one's (the trial-th,
   from 0): false when another trial is needed */
template <class R>
OA_D bool redirect(const SimParams& P, int command, int trial, uint32_t& flag, R& rng, Photon& p)
{
    float u[5];
    draw<5>(rng, u);
    if (command == CMD_REEMIT) {        /* wavelength, direction (2), polarization (2) */
        p.wavelength = scint_wavelength(P, u[0]);
        p.mom = uniform_sphere(u[1], u[2]);
        p.pol = normalize(cross(uniform_sphere(u[3], u[4]), p.mom));
        flag = F_BULK_REEMIT;
        return true;
    }
    v3 direction, polarization;
    const bool accepted = rayleigh_trial(p, u, direction, polarization) || trial + 1 >= OA_MAX_TRIALS;
    if (accepted) {
        p.mom = direction;
        p.pol = polarization;
        flag = F_BULK_SCATTER;
    }
    return accepted;
}

/* ----------------------------------------------------------- physics */

template <class R, class Tape>
OA_D int to_boundary(const SimParams& P, uint32_t& flag, R& rng, Photon& p, const State& s, float dist, Tape& tape,
                     MaybeThird& third)
{
    const float absorption_length = s.material1.y;
    const float scattering_length = s.material1.z;
    const float reemission_prob = s.material1.w;
    const float gv = s.group_velocity;
    float u_scattering, u_absorption;
    third = draw2_maybe3(rng, u_scattering, u_absorption);
    const float scattering_distance = -scattering_length * oa_logf(u_scattering);
    const float absorption_distance = -absorption_length * oa_logf(u_absorption);
    /* the step's one segment: its length and the process that ends it (the
       branches below, in the same order) */
    {
        const bool absorbs = absorption_distance <= scattering_distance && absorption_distance <= dist;
        const bool scatters = !(absorption_distance <= scattering_distance) && scattering_distance <= dist;
        tape.seg(P, s.m1_line, p.wavelength, absorption_length, scattering_length,
                 absorbs ? absorption_distance : scatters ? scattering_distance : dist,
                 absorbs ? SEG_ABSORB : scatters ? SEG_SCATTER : SEG_SAIL);
    }
    if (absorption_distance <= scattering_distance) {
        if (absorption_distance <= dist) {
            p.time += absorption_distance / gv;
            p.pos = p.pos + absorption_distance * p.mom;
            float u_reemit = reemission_prob == 0.f ? 2.f : maybe_third(rng, third);
            if (u_reemit < reemission_prob) return CMD_REEMIT;
            flag = F_BULK_ABSORB;
            return CMD_BREAK;
        }
    } else if (scattering_distance <= dist) {
        p.time += scattering_distance / gv;
        p.pos = p.pos + scattering_distance * p.mom;
        return CMD_SCATTER;
    }
    p.pos = p.pos + dist * p.mom;
    p.time += dist / gv;
    return CMD_BOUNDARY;
}

template <class R>
OA_D int at_boundary(uint32_t& flag, R& rng, MaybeThird third, Photon& p, float n1, float n2, v3 normal)
{
    const float eta = n1 / n2;
    const float _c1 = -dot(p.mom, normal);
    const v3 on = _c1 < 0.f ? -normal : normal;
    const v3 trans = cross(p.mom, on);
    const float trans_length = length(trans);
    const bool normal_incidence = trans_length < 1e-6f;
    const v3 A_trans = normal_incidence ? p.pol : trans * (1.0f / trans_length);
    const float E1_perp = dot(p.pol, A_trans);
    const float c1 = fabsf(_c1);
    const float c2c2 = 1.f - eta * eta * (1.f - c1 * c1);
    const bool tir = c2c2 < 0.f;
    const float EdotN = dot(p.pol, on);
    const float c2 = tir ? 0.f : sqrtf(c2c2);
    const float n1c1 = n1 * c1, n2c2 = n2 * c2, n2c1 = n2 * c1, n1c2 = n1 * c2;
    float E1x, E1y;
    if (normal_incidence) { E1x = 0.f; E1y = 1.f; }
    else { E1x = E1_perp; E1y = length(p.pol - E1_perp * A_trans); }
    const float E2_tx = 2.f * n1c1 * E1x / (n1c1 + n2c2);
    const float E2_ty = 2.f * n1c1 * E1y / (n2c1 + n1c2);
    const float E2_rx = E2_tx - E1x;
    const float E2_ry = (n2 * E2_ty / n1) - E1y;
    const float invR = 1.0f / sqrtf(E2_rx * E2_rx + E2_ry * E2_ry);
    const float invT = 1.0f / sqrtf(E2_tx * E2_tx + E2_ty * E2_ty);
    const float TransCoeff = (tir || n1c1 == 0.f) ? 0.f : n2c2 * (E2_tx * E2_tx + E2_ty * E2_ty) / n1c1;
    const float u_reflect = maybe_third(rng, third);
    const bool reflect = u_reflect > TransCoeff;
    p.mom = reflect ? p.mom + (2.0f * c1) * on : eta * p.mom + (eta * c1 - c2) * on;
    const v3 A_paral = normalize(cross(p.mom, A_trans));
    if (normal_incidence) {
        p.pol = reflect ? p.pol * (n2 > n1 ? -1.f : 1.f) : p.pol;
    } else if (reflect) {
        p.pol = tir ? -p.pol + (2.f * EdotN) * on : (E2_rx * invR) * A_trans + (E2_ry * invR) * A_paral;
    } else {
        p.pol = (E2_tx * invT) * A_trans + (E2_ty * invT) * A_paral;
    }
    flag = reflect ? F_BOUNDARY_REFLECT : F_BOUNDARY_TRANSMIT;
    return CMD_CONTINUE;
}

template <class R>
OA_D int at_surface(uint32_t& flag, R& rng, MaybeThird third, Photon& p, const State& s, v3 normal)
{
    const float detect = s.surface.x, absorb = s.surface.y, diffuse = s.surface.w;
    const float u_surface = maybe_third(rng, third);
    const int action = u_surface < absorb + detect ? CMD_BREAK : CMD_CONTINUE;
    if (action == CMD_BREAK) {
        flag = u_surface < absorb ? F_SURFACE_ABSORB : F_SURFACE_DETECT;
    } else if (u_surface < absorb + detect + diffuse) {
        flag = F_SURFACE_DREFLECT;
        const v3 old_mom = p.mom;
        const float orient = dot(old_mom, normal) > 0.f ? -1.f : 1.f;
        lambertian(p.mom, normal, orient, rng);
        const v3 facet = normalize(p.mom - old_mom);
        const float EdotN = dot(p.pol, facet);
        p.pol = -1.f * p.pol + (2.f * EdotN) * facet;
    } else {
        flag = F_SURFACE_SREFLECT;
        const float PdotN = dot(p.mom, normal);
        p.mom = p.mom - (2.f * PdotN) * normal;
        const float EdotN = dot(p.pol, normal);
        p.pol = -1.f * p.pol + (2.f * EdotN) * normal;
    }
    return action;
}

/* up to the photon's fate in this step; CMD_REEMIT and CMD_SCATTER leave its new direction
   and flag to redirect() */
template <class R, class Tape>
OA_D int propagate(const SimParams& P, uint32_t& flag, R& rng, Photon& p, const Prd& prd, Tape& tape)
{
    const uint32_t boundary = prd.boundary;
    const uint32_t identity = prd.iindex_identity & 0xffffu;
    const uint32_t iindex = prd.iindex_identity >> 16;
    const v3 normal = prd.normal;
    const float cosTheta = dot(p.mom, normal);
    /* sphoton::set_prd (sysrap/sphoton.h:499-505) */
    p.obf = (p.obf & 0x8000ffffu) | ((boundary & 0x7fffu) << 16);
    p.identity = (p.identity & 0xff000000u) | (identity & 0x00ffffffu);
    p.obf = (p.obf & 0x7fffffffu) | ((cosTheta < 0.f ? 0x1u : 0x0u) << 31);
    p.hitcount_iindex = 0x00010000u | (0x0000ffffu & iindex);
    State s;
    fill(P, s, boundary, p.wavelength, cosTheta);
    MaybeThird third;
    int command = to_boundary(P, flag, rng, p, s, prd.t, tape, third);
    if (command == CMD_BOUNDARY) {
        if (s.ems == EMS_NOSURFACE) command = at_boundary(flag, rng, third, p, s.material1.x, s.n2, normal);
        else if (s.ems == EMS_SURFACE) command = at_surface(flag, rng, third, p, s, normal);
        else if (prd.lposcost < 0.f) command = at_surface(flag, rng, third, p, s, normal);
        else if (s.ems == EMS_ZPLUS_SENSOR_A) { (void)maybe_third(rng, third); flag = F_SURFACE_DETECT; command = CMD_BREAK; }
    }
    return command;
}

/* -------------------------------------------------------- generation */

enum : uint32_t { T_DISC = 1, T_LINE = 2, T_POINT = 3, T_CIRCLE = 4, T_RECTANGLE = 5, T_SPHERE_MARSAGLIA = 6, T_SPHERE = 7,
                  T_POINT_ISO = 100 };

OA_D void zero_flags_set(Photon& p, uint32_t flag)
{
    p.obf = 0u; p.identity = 0u; p.flagmask = 0u; p.hitcount_iindex = 0u;
    set_flag(p, flag);
}

template <class R>
OA_D void gen_torch(Photon& p, R& rng, const float4* gq, uint64_t photon_id)
{
    const float4 q0 = gq[0], q1 = gq[1], q2 = gq[2], q3 = gq[3], q4 = gq[4], q5 = gq[5];
    const uint32_t numphoton = __float_as_uint(q0.w);
    const uint32_t type = __float_as_uint(q5.w);
    const v3 gpos = mk(q1.x, q1.y, q1.z);
    const float gtime = q1.w;
    const v3 gmom = mk(q2.x, q2.y, q2.z);
    const float gweight = q2.w;
    const float gwl = q3.w;
    const float zx = q4.x, zy = q4.y, ax = q4.z, ay = q4.w;
    const float radius = q5.x, distance = q5.y;
    p.pos = mk(0.f, 0.f, 0.f); p.time = 0.f; p.mom = mk(0.f, 0.f, 0.f); p.pol = mk(0.f, 0.f, 0.f);
    p.wavelength = 0.f;
    if (type == T_SPHERE || type == T_POINT_ISO) {
        p.wavelength = gwl; p.time = gtime;
        float u0, u1;
        const MaybeThird third = draw2_maybe3(rng, u0, u1);
        float u_zenith = zx + u0 * (zy - zx);
        float u_azimuth = ax + u1 * (ay - ax);
        float phi = 2.f * OA_PI_F * u_azimuth;
        float sinPhi, cosPhi; oa_sincosf(phi, &sinPhi, &cosPhi);
        float cosTheta = 1.f - 2.0f * u_zenith;
        float sinTheta = sqrtf(1.0f - cosTheta * cosTheta);
        float flip = copysignf(1.f, radius);
        p.mom = mk(flip * sinTheta * cosPhi, flip * sinTheta * sinPhi, flip * cosTheta);
        float rad = fabsf(radius);
        p.pos = mk(sinTheta * cosPhi * rad, sinTheta * sinPhi * rad, cosTheta * rad);
        float phase = 2.f * OA_PI_F * distance;
        float sph, cph; oa_sincosf(phase, &sph, &cph);
        p.pol = mk(cph, sph, 0.f);
        rotateUz(p.pol, p.mom);
        if (type == T_POINT_ISO) {
            p.pos = p.pos + gpos;
            if (gweight > 0.f) p.wavelength = gwl + maybe_third(rng, third) * gweight;
        }
    } else if (type == T_DISC) {
        p.wavelength = gwl; p.time = gtime; p.mom = gmom;
        float u2[2];
        draw<2>(rng, u2);
        float u_zenith = zx + u2[0] * (zy - zx);
        float u_azimuth = ax + u2[1] * (ay - ax);
        float r = radius * u_zenith;
        float phi = 2.f * OA_PI_F * u_azimuth;
        float sinPhi, cosPhi; oa_sincosf(phi, &sinPhi, &cosPhi);
        p.pos = mk(r * cosPhi, r * sinPhi, 0.f);
        rotateUz(p.pos, p.mom);
        p.pos = p.pos + gpos;
        p.pol = mk(sinPhi, -cosPhi, 0.f);
        rotateUz(p.pol, p.mom);
    } else if (type == T_SPHERE_MARSAGLIA) {
        p.wavelength = gwl; p.time = gtime;
        float u, v, b, a;
        int trials = 0;
        do {
            float u2[2];
            draw<2>(rng, u2);
            float u0z = zx + u2[0] * (zy - zx);
            float u1a = ax + u2[1] * (ay - ax);
            u = 2.f * u0z - 1.f; v = 2.f * u1a - 1.f; b = u * u + v * v;
        } while (b > 1.f && ++trials < OA_MAX_TRIALS);
        if (b > 1.f) { u = 0.f; v = 0.f; b = 0.f; }
        a = 2.f * sqrtf(1.f - b);
        float rad = fabsf(radius);
        float flip = copysignf(1.f, radius);
        p.mom = mk(flip * a * u, flip * a * v, flip * (2.f * b - 1.f));
        p.pos = mk(a * u * rad, a * v * rad, (2.f * b - 1.f) * rad);
        float phase = 2.f * OA_PI_F * distance;
        float sph, cph; oa_sincosf(phase, &sph, &cph);
        p.pol = mk(cph, sph, 0.f);
        rotateUz(p.pol, p.mom);
    } else if (type == T_LINE) {
        p.wavelength = gwl; p.time = gtime; p.mom = gmom;
        float frac = (float)photon_id / (float)numphoton;
        float sfrac = 2.f * (frac - 0.5f);
        float r = radius * sfrac;
        p.pos = mk(r, 0.f, 0.f);
        rotateUz(p.pos, p.mom);
        p.pos = p.pos + gpos;
        p.pol = mk(0.f, -1.f, 0.f);
        rotateUz(p.pol, p.mom);
    } else if (type == T_POINT) {
        p.wavelength = gwl; p.time = gtime; p.mom = gmom;
        p.pos = mk(0.f, 0.f, 0.f);
        rotateUz(p.pos, p.mom);
        p.pos = p.pos + gpos;
        p.pol = mk(0.f, -1.f, 0.f);
        rotateUz(p.pol, p.mom);
    } else if (type == T_CIRCLE) {
        p.wavelength = gwl; p.time = gtime;
        float f = (float)photon_id / (float)numphoton;
        float frac = ax * (1.f - f) + ay * (f);
        float phi = 2.f * OA_PI_F * frac;
        float sinPhi, cosPhi; oa_sincosf(phi, &sinPhi, &cosPhi);
        float r = radius < 0.f ? -radius : radius;
        p.mom = mk(radius < 0.f ? -cosPhi : cosPhi, 0.f, radius < 0.f ? -sinPhi : sinPhi);
        p.pos = mk(r * cosPhi, 0.f, r * sinPhi);
        p.pos = p.pos + gpos;
        p.pol = mk(0.f, -1.f, 0.f);
        rotateUz(p.pol, p.mom);
    } else if (type == T_RECTANGLE) {
        /* storch.h:463-516: photons split over the four sides of the rectangle
           x in [azimuth.x, azimuth.y], z in [zenith.x, zenith.y] of the y = 0 plane,
           each pointing inwards; left, right, bottom, top. Fewer than 4 photons
           (side size 0, a division by zero in the reference) all go to side 0. */
        p.wavelength = gwl; p.time = gtime;
        const int side_size = (int)(numphoton / 4u);
        const uint64_t ss = side_size > 0 ? (uint64_t)side_size : 1ull;
        const int side = (int)(photon_id / ss);
        const int side_index = (int)(photon_id - (uint64_t)side * ss);
        const float frac = (float)side_index / (float)(side_size > 0 ? side_size : 1);
        if (side == 0 || side == 1) {
            p.pos = mk(side == 0 ? ax : ay, 0.f, (1.f - frac) * zx + frac * zy);
            p.mom = mk(side == 0 ? 1.f : -1.f, 0.f, 0.f);
        } else if (side == 2 || side == 3) {
            p.pos = mk((1.f - frac) * ax + frac * ay, 0.f, side == 2 ? zx : zy);
            p.mom = mk(0.f, 0.f, side == 2 ? 1.f : -1.f);
        }
        p.pos = p.pos + gpos;
        p.pol = mk(0.f, -1.f, 0.f);
        rotateUz(p.pol, p.mom);
    }
    zero_flags_set(p, F_TORCH);
}

template <class R>
OA_D void gen_scint(const SimParams& P, Photon& p, R& rng, const float4* gq)
{
    float ug[4];
    draw<4>(rng, ug);
    const float u0 = ug[0], u1 = ug[1], u2 = ug[2], u3 = ug[3];
    float cost = 1.f - 2.f * u0;
    float sint = sqrtf((1.f - cost) * (1.f + cost));
    float phi = 2.f * OA_PI_F * u1;
    float sinp, cosp; oa_sincosf(phi, &sinp, &cosp);
    p.mom = mk(sint * cosp, sint * sinp, cost);
    p.pol = mk(cost * cosp, cost * sinp, -sint);
    phi = 2.f * OA_PI_F * u2;
    oa_sincosf(phi, &sinp, &cosp);
    p.pol = normalize(cosp * p.pol + sinp * cross(p.mom, p.pol));
    p.wavelength = scint_wavelength(P, u3);
    const float4 q1 = gq[1], q2 = gq[2], q3 = gq[3], q5 = gq[5];
    const float charge = q3.y, meanVelocity = q3.w, step_length = q2.w, scint_time = q5.x;
    float ut[2];                    /* position along the step (charged), then the decay time */
    if (charge == 0.f) { ut[0] = 1.f; ut[1] = draw1(rng); }
    else draw<2>(rng, ut);
    const float fraction = ut[0];
    p.pos = mk(q1.x, q1.y, q1.z) + fraction * mk(q2.x, q2.y, q2.z);
    const float u4 = ut[1];
    float deltaTime = fraction * step_length / meanVelocity - scint_time * oa_logf(u4);
    p.time = q1.w + deltaTime;
    zero_flags_set(p, F_SCINTILLATION);
}

/* qcerenkov::generate (qudarap/qcerenkov.h): wavelength by reciprocal sampling
   flat in energy with rejection on sin^2(theta) against the medium's RINDEX
   from the bnd table (line = genstep matline), cone about the normalized step,
   emission point along the step by rejection on the linear N1 -> N2 yield */
template <class R>
OA_D void gen_cerenkov(const SimParams& P, Photon& p, R& rng, const float4* gq)
{
    const float4 q0 = gq[0], q1 = gq[1], q2 = gq[2], q3 = gq[3], q4 = gq[4], q5 = gq[5];
    const int matline = (int)__float_as_uint(q0.z);
    const v3 dpos = mk(q2.x, q2.y, q2.z);
    const float step_length = q2.w, preVelocity = q3.w;
    const float BetaInverse = q4.x, Wmin = q4.y, Wmax = q4.z;
    const float maxSin2 = q5.x, N1 = q5.y, N2 = q5.z, postVelocity = q5.w;
    const v3 p0 = normalize(dpos);
    float wavelength, cosTheta, sin2Theta, u_maxSin2;
    unsigned count = 0;
    do {
        float u[2];
        draw<2>(rng, u);
        const float w = Wmin + u[0] * (Wmax - Wmin);
        wavelength = Wmin * Wmax / w;
        const float4 props = bnd_lookup(P, wavelength, matline, 0);
        const float sampledRI = props.x;
        cosTheta = BetaInverse / sampledRI;
        sin2Theta = fmaxf(0.f, (1.f - cosTheta) * (1.f + cosTheta));
        u_maxSin2 = u[1] * maxSin2;
        count += 1;
    } while (u_maxSin2 > sin2Theta && count < 100);
    const float sinTheta = sqrtf(sin2Theta);
    const float phi = 2.f * OA_PI_F * draw1(rng);
    float sinPhi, cosPhi;
    oa_sincosf(phi, &sinPhi, &cosPhi);
    p.mom = mk(sinTheta * cosPhi, sinTheta * sinPhi, cosTheta);
    rotateUz(p.mom, p0);
    p.pol = mk(cosTheta * cosPhi, cosTheta * sinPhi, -sinTheta);
    rotateUz(p.pol, p0);
    p.wavelength = wavelength;
    float fraction, delta, NumberOfPhotons, N;
    const float MeanNumberOfPhotonsMax = fmaxf(N1, N2);
    const float DeltaN = (N1 - N2);
    int trials = 0;
    do {
        float w[2];
        draw<2>(rng, w);
        fraction = w[0];
        delta = fraction * step_length;
        NumberOfPhotons = N1 - fraction * DeltaN;
        N = w[1] * MeanNumberOfPhotonsMax;
    } while (N > NumberOfPhotons && ++trials < OA_MAX_TRIALS);
    const float midVelocity = preVelocity + fraction * (postVelocity - preVelocity) * 0.5f;
    p.time = q1.w + delta / midVelocity;
    p.pos = mk(q1.x, q1.y, q1.z) + fraction * dpos;
    zero_flags_set(p, F_CERENKOV);
}

/* ------------------------------------------------------------- trace */

/* slab test; on a hit tn is the entry distance clamped to tmin */
/* Ray data for slab tests: t = fma(plane, inv, -oi) with inv ~ 1/d (the hardware
   reciprocal, 1 ulp) and oi = o*inv. A direction component below 1e-20 in
   magnitude is replaced by +-1e-20 so inv and oi stay finite and the slab of a
   parallel ray gives huge t of the right sign. The reciprocal and the FMA form
   round differently from (plane - o)/d by a few ulp of o; box tests only prune
   (every box is padded by >= 1e-2 mm around what it holds), so the hits found
   do not depend on it. */
OA_D void slab_ray(v3 o, v3 d, v3& inv, v3& oi)
{
    const float e = 1e-20f;
    inv = mk(__builtin_amdgcn_rcpf(fabsf(d.x) < e ? copysignf(e, d.x) : d.x),
             __builtin_amdgcn_rcpf(fabsf(d.y) < e ? copysignf(e, d.y) : d.y),
             __builtin_amdgcn_rcpf(fabsf(d.z) < e ? copysignf(e, d.z) : d.z));
    oi = mk(o.x * inv.x, o.y * inv.y, o.z * inv.z);
}

/* entry distance into one child box, or +inf when the ray misses it in [tmin, tmax] */
OA_D float box_enter(float lx, float ly, float lz, float hx, float hy, float hz, v3 inv, v3 oi, float tmin,
                     float tmax)
{
    const float x0 = fmaf(lx, inv.x, -oi.x), x1 = fmaf(hx, inv.x, -oi.x);
    const float y0 = fmaf(ly, inv.y, -oi.y), y1 = fmaf(hy, inv.y, -oi.y);
    const float z0 = fmaf(lz, inv.z, -oi.z), z1 = fmaf(hz, inv.z, -oi.z);
    const float tn = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), tmin));
    const float tf = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), tmax));
    return tn <= tf ? tn : INFINITY;
}

OA_D void cswap(float& ta, uint32_t& ca, float& tb, uint32_t& cb)
{
    const bool s = tb < ta;
    const float t = s ? tb : ta;
    const uint32_t c = s ? cb : ca;
    tb = s ? ta : tb; cb = s ? ca : cb;
    ta = t; ca = c;
}

/* Visit one 4-wide node: returns the nearest hit child link (or EMPTY) and
   pushes the other hit children farthest first, so they pop nearest first.
   Leaf links go on the stack like node links, so both levels are traversed
   nearest-first and a shrinking tmax culls what is still pending. Equal entry
   distances keep the node's child order (leaves first). */
template <int STRIDE, bool SINGLE = false>
OA_D uint32_t visit(const BvhNode* nodes, uint32_t idx, v3 inv, v3 oi, float tmin, float tmax,
                    uint32_t* stk, int& sp)
{
    const float4* q = reinterpret_cast<const float4*>(nodes + idx);
    const float4 lx = q[0], ly = q[1], lz = q[2], hx = q[3], hy = q[4], hz = q[5];
    const uint4 ch = *reinterpret_cast<const uint4*>(q + 6);
    if constexpr (SINGLE) {
        /* a node with one child (the BLAS root of a one-prim solid): one box test.
           Empty slots hold boxes at +inf, which every test misses, so the full
           visit below would return the same link and push nothing. */
        if (ch.y == OA_BVH_EMPTY) {
            const float t = box_enter(lx.x, ly.x, lz.x, hx.x, hy.x, hz.x, inv, oi, tmin, tmax);
            return t < INFINITY ? ch.x : OA_BVH_EMPTY;
        }
    }
    float t0 = box_enter(lx.x, ly.x, lz.x, hx.x, hy.x, hz.x, inv, oi, tmin, tmax);
    float t1 = box_enter(lx.y, ly.y, lz.y, hx.y, hy.y, hz.y, inv, oi, tmin, tmax);
    float t2 = box_enter(lx.z, ly.z, lz.z, hx.z, hy.z, hz.z, inv, oi, tmin, tmax);
    float t3 = box_enter(lx.w, ly.w, lz.w, hx.w, hy.w, hz.w, inv, oi, tmin, tmax);
    uint32_t c0 = ch.x, c1 = ch.y, c2 = ch.z, c3 = ch.w;
    cswap(t0, c0, t1, c1);
    cswap(t2, c2, t3, c3);
    cswap(t0, c0, t2, c2);
    cswap(t1, c1, t3, c3);
    cswap(t1, c1, t2, c2);
    if (t3 < INFINITY) { stk[sp * STRIDE] = c3; sp++; }
    if (t2 < INFINITY) { stk[sp * STRIDE] = c2; sp++; }
    if (t1 < INFINITY) { stk[sp * STRIDE] = c1; sp++; }
    return t0 < INFINITY ? c0 : OA_BVH_EMPTY;
}

OA_D void inst_ray_rows(float4 r0, float4 r1, float4 r2, float4 r3, v3 o, v3 d, v3& oo, v3& od)
{
    oo = mk(r0.x * o.x + r1.x * o.y + r2.x * o.z + r3.x,
            r0.y * o.x + r1.y * o.y + r2.y * o.z + r3.y,
            r0.z * o.x + r1.z * o.y + r2.z * o.z + r3.z);
    od = mk(r0.x * d.x + r1.x * d.y + r2.x * d.z,
            r0.y * d.x + r1.y * d.y + r2.y * d.z,
            r0.z * d.x + r1.z * d.y + r2.z * d.z);
}
OA_D void inst_ray(const float4* m, v3 o, v3 d, v3& oo, v3& od) { inst_ray_rows(m[0], m[1], m[2], m[3], o, d, oo, od); }

/* a ray's nearest hit so far (exact ties: the smaller (instance, prim) key) */
struct Nearest {
    float t;
    uint64_t key;
    uint32_t inst, prim;
    Isect is;
};
OA_D void nearest_none(Nearest& best, float tmax)
{
    best.t = tmax; best.key = ~0ull; best.inst = 0xffffffffu; best.prim = 0u;
    best.is.x = best.is.y = best.is.z = best.is.w = 0.f;
}

/* one prim of one instance (entry k of the BLAS-ordered prim records) against the
   nearest hit so far (t, then the (instance, prim) key) */
template <bool EXT>
OA_D void consider_prim(const SimParams& P, uint32_t ii, uint32_t k, v3 oo, v3 od, float tmin, Nearest& best)
{
    const PrimRec pr = P.blas_prims[k];
    const uint32_t pi = pr.index;
    Isect is;
    if (!intersect_prim<EXT>(is, P.node + 4u * pr.node_offset, P.itra, P.plan, tmin, oo, od)) return;
    /* a reported hit outside [tmin, tmax] is ignored, as optixReportIntersection does
       (a convex polyhedron behind the ray reports valid with t = 0) */
    if (!(is.w >= tmin)) return;
    const uint64_t key = ((uint64_t)ii << 32) | (uint64_t)pi;
    if (is.w < best.t || (is.w == best.t && key < best.key)) {
        best.t = is.w; best.key = key; best.inst = ii; best.prim = pi; best.is = is;
    }
}

/* Whether a ray has anything to find in the TLAS beyond its nearest front hit at best_t, and
   from where (tlo): a lane whose segment from the origin to that hit lies in the free ball,
   which no TLAS instance meets, has nothing; one whose origin lies in it can meet an instance
   only after leaving it, so its box tests start there (boxes only prune: the prim tests keep
   tmin). */
OA_D bool beyond_free_ball(float4 fb, v3 o, v3 d, float tmin, float best_t, float& tlo)
{
    if (!(fb.w > 0.f)) return true;
    const v3 c = mk(fb.x, fb.y, fb.z);
    const v3 a = o - c, b = o + best_t * d - c;
    const float qa = dot(a, a) - fb.w;
    if (qa < 0.f) {
        if (dot(b, b) < fb.w) return false;
        const float dd = dot(d, d), bb = dot(a, d);
        const float t_exit = (sqrtf(bb * bb - dd * qa) - bb) / dd;
        tlo = fmaxf(tmin, t_exit);
    }
    return true;
}

/* Geometry records that are the same for a whole wave, read through the scalar cache: the
   constant address space tells the compiler that nothing writes them during the launch. */
typedef float cf4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) cf4* cptr4;
typedef const __attribute__((address_space(4))) uint32_t* cptr1;
OA_D cptr4 const_ptr(const void* p) { return (cptr4)(uintptr_t)p; }
OA_D float4 const_load(cptr4 p) { const cf4 v = *p; return make_float4(v.x, v.y, v.z, v.w); }

/*
 * The front instances (world-sized, tested by every trace), where their solids are leaf
 * prims of the common types: P.front_plain. Every lane tests the same prims, so their
 * records come by scalar loads and the leaf type is a scalar branch, where the leaf phase
 * below chains vector loads (item, instance, prim record, node) with a switch per lane.
 */
OA_D void trace_front(const SimParams& P, v3 o, v3 d, float tmin, Nearest& best)
{
    const uint32_t first = P.front_leaf & 0x00ffffffu, count = (P.front_leaf >> 24) & 0x7fu;
    for (uint32_t k = 0; k < count; ++k) {
        const uint32_t ii = ((cptr1)(uintptr_t)P.tlas_items)[first + k];
        const cptr4 m = const_ptr(P.inst + ii);
        OA_COUNT(OA_ST_INST);
        const float4 r0 = const_load(m), r1 = const_load(m + 1), r2 = const_load(m + 2), r3 = const_load(m + 3);
        v3 oo, od;
        inst_ray_rows(r0, r1, r2, r3, o, d, oo, od);
        const uint32_t link = __float_as_uint(r2.w);       /* a front instance's link: one leaf of all its prims */
        const uint32_t bf = link & 0x00ffffffu, bn = (link >> 24) & 0x7fu;
        for (uint32_t j = 0; j < bn; ++j) {
            OA_COUNT(OA_ST_PRIM);
            OA_WAVE_COUNT(OA_ST_W_PRIM, OA_ST_L_PRIM);
            const float4 pr = const_load(const_ptr(P.blas_prims + bf + j));
            const uint32_t pi = __float_as_uint(pr.w);
            const cptr4 nd = const_ptr(P.node + 4u * __float_as_uint(pr.x));
            const float4 q0 = const_load(nd), q1 = const_load(nd + 1), q3 = const_load(nd + 3);
            Isect is;
            if (!intersect_leaf_q<false>(is, q0, q1, __float_as_uint(q3.z), __float_as_uint(q3.w), P.itra, P.plan, tmin,
                                         oo, od))
                continue;
            if (!(is.w >= tmin)) continue;
            const uint64_t key = ((uint64_t)ii << 32) | (uint64_t)pi;
            if (is.w < best.t || (is.w == best.t && key < best.key)) {
                best.t = is.w; best.key = key; best.inst = ii; best.prim = pi; best.is = is;
            }
        }
    }
}

/* One iteration of the node walk: pop when the lane holds nothing, visit a node, and take a
   leaf (popped or the visit's nearest child) at once. True: nothing is left. */
template <int STRIDE>
OA_D bool walk_nodes(const SimParams& P, v3 inv, v3 oi, float tlo, const Nearest& best, uint32_t* stk, int& sp, uint32_t& cur,
                     uint32_t& leaf)
{
    if (cur == OA_BVH_EMPTY) {
        if (sp == 0) return true;
        sp--;
        cur = stk[sp * STRIDE];
    }
    if (!(cur & OA_BVH_LEAF_BIT)) {
        OA_COUNT(OA_ST_TLAS);
#ifdef OA_STATS
        const int sp0 = sp;
#endif
        cur = visit<STRIDE>(P.tlas, cur, inv, oi, tlo, best.t, stk, sp);
#ifdef OA_STATS
        if (cur == OA_BVH_EMPTY && sp == sp0) OA_COUNT(OA_ST_TLAS_DEAD);
#endif
    }
    if (cur != OA_BVH_EMPTY && (cur & OA_BVH_LEAF_BIT)) {
        leaf = cur;
        cur = OA_BVH_EMPTY;
    }
    return false;
}

/* the instances of a leaf link: ray into each frame, BLAS walk, prim tests. Returns the
   iterations this took. */
template <int STRIDE, bool EXT>
OA_D uint32_t test_leaf(const SimParams& P, uint32_t leaf, v3 o, v3 d, float tmin, float tlo, Nearest& best, uint32_t* stk,
                    int& sp)
{
    uint32_t iterations = 0;
    const uint32_t first = leaf & 0x00ffffffu, count = (leaf >> 24) & 0x7fu;
    for (uint32_t k = 0; k < count; ++k) {
        const uint32_t ii = P.tlas_items[first + k];
        OA_COUNT(OA_ST_INST);
        const float4* m = reinterpret_cast<const float4*>(P.inst + ii);
        v3 oo, od;
        inst_ray(m, o, d, oo, od);
        v3 inv2, oi2;
        slab_ray(oo, od, inv2, oi2);
        const int sp_base = sp;
        uint32_t bc = __float_as_uint(m[2].w);     /* BLAS root of this solid (front instances: one leaf of all its prims) */
        for (;;) {
            OA_WAVE_COUNT(OA_ST_W_P2, OA_ST_L_P2);
            iterations++;
            /* as in the node walk: pop, visit, and test a leaf's prims in one iteration */
            if (bc == OA_BVH_EMPTY) {
                if (sp == sp_base) break;
                sp--;
                bc = stk[sp * STRIDE];
            }
            if (!(bc & OA_BVH_LEAF_BIT)) {
                OA_COUNT(OA_ST_BLAS);
#ifdef OA_STATS
                const int sp0 = sp;
#endif
                bc = visit<STRIDE, true>(P.blas, bc, inv2, oi2, tlo, best.t, stk, sp);
#ifdef OA_STATS
                if (bc == OA_BVH_EMPTY && sp == sp0) OA_COUNT(OA_ST_BLAS_DEAD);
#endif
                if (bc == OA_BVH_EMPTY || !(bc & OA_BVH_LEAF_BIT)) continue;
            }
            const uint32_t bf = bc & 0x00ffffffu, bn = (bc >> 24) & 0x7fu;
            OA_CYC_MARK(c_prim);
            for (uint32_t j = 0; j < bn; ++j) {
                OA_COUNT(OA_ST_PRIM);
                OA_WAVE_COUNT(OA_ST_W_PRIM, OA_ST_L_PRIM);
                consider_prim<EXT>(P, ii, bf + j, oo, od, tmin, best);
            }
            OA_CYC_ADD(OA_ST_C_PRIM, c_prim);
            bc = OA_BVH_EMPTY;
        }
    }
    return iterations;
}

/* what a trace reports of its nearest hit */
OA_D void hit_record(const SimParams& P, const Nearest& best, v3 o, v3 d, Prd& prd)
{
    if (best.inst == 0xffffffffu) {
        prd.normal = mk(0.f, 0.f, 0.f); prd.t = 0.f; prd.lposcost = 0.f;
        prd.lx = 0.f; prd.ly = __uint_as_float(0x7fc00000u); prd.gprim = 0xffffu;
        prd.iindex_identity = 0xffffffffu; prd.boundary = 0xffffu;
        return;
    }
    const float4* m = reinterpret_cast<const float4*>(P.inst + best.inst);
    const float4 r0 = m[0], r1 = m[1], r2 = m[2];
    prd.normal = mk(r0.x * best.is.x + r0.y * best.is.y + r0.z * best.is.z,
                    r1.x * best.is.x + r1.y * best.is.y + r1.z * best.is.z,
                    r2.x * best.is.x + r2.y * best.is.y + r2.z * best.is.z);
    prd.t = best.t;
    v3 oo, od;
    inst_ray(m, o, d, oo, od);
    const v3 lpos = oo + best.t * od;
    prd.lposcost = lpos.z / sqrtf(dot(lpos, lpos));
    prd.lx = lpos.x;
    prd.ly = lpos.y;
    const uint32_t ident = __float_as_uint(r1.w);
    prd.iindex_identity = ((best.inst & 0xffffu) << 16) | (ident & 0xffffu);
    prd.boundary = P.prim[best.prim].boundary & 0xffffu;
    prd.gprim = P.prim[best.prim].global_prim;
}

/*
 * Nearest hit over instances x prims with t in (tmin, tmax); exact ties go to
 * the smaller (instance, prim) key so the answer does not depend on traversal
 * order. stk: this lane's LDS stack, entry k at stk[k*STRIDE].
 *
 * "while-while" traversal (Aila and Laine, "Understanding the efficiency of
 * ray traversal on GPUs", HPG 2009): lanes walk TLAS nodes until each holds
 * an instance leaf or is finished, then all pending leaves (instance ray
 * transform, BLAS walk, CSG prim tests) run together, so the expensive CSG
 * code executes with most lanes of the wave active instead of once per lane.
 *
 * Returns false, with nothing found out, for a lane that needs the TLAS walk while fewer
 * than walk_min lanes of the wave do and some lane does not, or others of the wave have
 * something else to do (`others`): it is traced again, front instances included, with its
 * wave's next step (they are tested on the whole wave anyway). Such a wave always has a
 * lane that gets on.
 */
template <int STRIDE, bool EXT = false>
OA_D bool trace(const SimParams& P, uint32_t* stk, v3 o, v3 d, float tmin, float tmax, Prd& prd, int walk_min = 0, bool others = false)
{
    OA_COUNT(OA_ST_TRACE);
    OA_WAVE_COUNT(OA_ST_W_TRACE, OA_ST_L_TRACE);
    OA_CYC_MARK(c_trace);
    v3 inv, oi;
    slab_ray(o, d, inv, oi);
    Nearest best;
    nearest_none(best, tmax);
    int sp = 0;
    uint32_t cur = P.tlas_empty ? OA_BVH_EMPTY : 0u;    /* TLAS root node */
    /* the front instances (world-sized boxes kept out of the TLAS) are tested on every
       lane together, by trace_front or as the first leaf phase; the walk then starts with
       their nearest hit as tmax */
    uint32_t leaf = P.front_plain ? OA_BVH_EMPTY : P.front_leaf;
    /* lower bound of the node and BLAS box tests of TLAS instances (set after the front phase) */
    float tlo = tmin;
    bool done = false;
    if (P.front_plain) {
        trace_front(P, o, d, tmin, best);
        done = !(cur == 0u && beyond_free_ball(const_load(const_ptr(P.free_ball)), o, d, tmin, best.t, tlo));
        /* the TLAS walk and the CSG trees behind it run for as long as their slowest lane:
           lanes that need them wait for company while others of the wave have a step to do */
        const unsigned long long walkers = __ballot(!done);
        if (__popcll(walkers) < walk_min && (others || walkers != __ballot(1))) {
            if (!done) return false;
        }
    }
#ifdef OA_STATS
    uint32_t n1 = 0, n2 = 0;
#endif
    while (!done) {
        /* phase 1: walk nodes until this lane has a leaf or nothing left */
        OA_CYC_MARK(c_p1);
        /* Once fewer than regroup_pct percent of the lanes that entered this walk
           still walk, the whole wave leaves it: the lanes holding a leaf run the
           leaf phase and the others resume from their own node and stack after it.
           Each lane still visits the same nodes and leaves in the same order, so
           only the wave's interleaving changes, never a result. 0 waits for all. */
        const int walk_floor = P.regroup_pct > 0 ? __popcll(__ballot(1)) * P.regroup_pct : 0;
        while (!done && leaf == OA_BVH_EMPTY) {
            if (__popcll(__ballot(1)) * 100 < walk_floor) break;
            OA_WAVE_COUNT(OA_ST_W_P1, OA_ST_L_P1);
#ifdef OA_STATS
            n1++;
#endif
            if (walk_nodes<STRIDE>(P, inv, oi, tlo, best, stk, sp, cur, leaf)) done = true;
        }
        OA_CYC_ADD(OA_ST_C_P1, c_p1);
        if (leaf == OA_BVH_EMPTY) continue;
        /* phase 2: the pending instance leaf */
        OA_CYC_MARK(c_p2);
        /* the leaf phase is chains of dependent loads (instance record, BLAS node, prim
           record, CSG nodes): waves in it issue first, so their next load starts sooner
           (0.6% on the 64 events against no priority; raising the walk instead lost 1%) */
        __builtin_amdgcn_s_setprio(2);
        const uint32_t at = leaf;
        leaf = OA_BVH_EMPTY;
        const uint32_t iterations = test_leaf<STRIDE, EXT>(P, at, o, d, tmin, tlo, best, stk, sp);
#ifdef OA_STATS
        n2 += iterations;
#endif
        (void)iterations;
        OA_CYC_ADD(OA_ST_C_P2, c_p2);
        __builtin_amdgcn_s_setprio(0);
        /* after a front leaf phase (the TLAS walk not begun: cur is still the root) */
        if (cur == 0u && !beyond_free_ball(*P.free_ball, o, d, tmin, best.t, tlo)) cur = OA_BVH_EMPTY;
    }
    OA_CYC_ADD(OA_ST_C_TRACE, c_trace);
#ifdef OA_STATS
    atomicAdd(&oa_hist[0][n1 ? 32 - __clz(n1) : 0], 1ull);
    atomicAdd(&oa_hist[1][n2 ? 32 - __clz(n2) : 0], 1ull);
    if (n1 > OA_SLOW_ITER) {
        const unsigned long long k = atomicAdd(&oa_slow_n, 1ull);
        if (k < OA_SLOW_MAX) {
            oa_slow[3 * k + 0] = make_float4(o.x, o.y, o.z, tmin);
            oa_slow[3 * k + 1] = make_float4(d.x, d.y, d.z, tmax);
            oa_slow[3 * k + 2] = make_float4(best.t, (float)n1, (float)n2, __uint_as_float(best.inst));
        }
    }
#endif
    hit_record(P, best, o, d, prd);
    return true;
}

} // namespace oa
