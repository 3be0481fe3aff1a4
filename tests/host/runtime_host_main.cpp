// Checks of the library's host side against the stand-in for the HIP runtime,
// where what a call asks of the device can be written down: no kernel of a
// compiled topology or tree runs, its launch is recorded instead.
//
//   runtime_host <check>
//
// Prints what it saw and returns 1 if that is wrong.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../include/gorilla_amd.h"
#include "../../gorilla-physics_amd/csrc/gp_internal.h"

namespace {
struct FastLaunch { int topo, n_steps, block; };
std::vector<FastLaunch> fast_launches;
}  // namespace

namespace gp {
int fast_topology_id(int, const int*, const int*, int) { return -1; }
int launch_fast_step(int topo, int, const BucketArgs&, double, int n_steps, int block, void*) {
  fast_launches.push_back({topo, n_steps, block});
  return hipSuccess;
}
int launch_fast_rk_step(int, int, int, const BucketArgs&, double, int, int, void*) { return hipErrorNotSupported; }
int launch_grouped_step(const GroupTable*, int, int, double, int, int, void*) { return hipErrorNotSupported; }
}  // namespace gp

static void need(bool c, const char* what) {
  if (!c) {
    std::printf("%s (%s)\n", what, gp_last_error());
    std::exit(1);
  }
}

// A floating body with a revolute one on it, a contact point and a plane: a
// tree that no compiled topology covers.
static gp_model* small_tree() {
  gp_body_desc body[2] = {};
  for (int i = 0; i < 2; ++i) {
    body[i].parent = i - 1;
    body[i].jtype = i == 0 ? GP_JOINT_FLOATING : GP_JOINT_REVOLUTE;
    body[i].axis[2] = 1.0;
    body[i].x_tree_quat[3] = 1.0;
    for (int k = 0; k < 3; ++k) body[i].moment[k] = 1.0;
    body[i].mass = 1.0;
  }
  gp_contact_desc contact{};
  contact.k = 50e3;
  gp_halfspace_desc plane{};
  plane.normal[2] = 1.0;
  plane.alpha = 0.9;
  plane.mu = 0.5;
  gp_model_desc d{};
  d.n_bodies = 2;
  d.bodies = body;
  d.n_contacts = 1;
  d.contacts = &contact;
  d.n_halfspaces = 1;
  d.halfspaces = &plane;
  d.gravity = 9.81;
  gp_model* m = nullptr;
  need(gp_model_create(&d, &m) == GP_OK, "gp_model_create");
  return m;
}

// A lone body on a joint of this type.
static gp_model* lone_body(int jtype) {
  gp_body_desc body{};
  body.parent = -1;
  body.jtype = jtype;
  body.axis[2] = 1.0;
  body.x_tree_quat[3] = 1.0;
  for (int k = 0; k < 3; ++k) body.moment[k] = 1.0;
  body.mass = 1.0;
  gp_model_desc d{};
  d.n_bodies = 1;
  d.bodies = &body;
  d.gravity = 9.81;
  gp_model* m = nullptr;
  need(gp_model_create(&d, &m) == GP_OK, "gp_model_create");
  return m;
}

static gp_batch* batch_of(gp_model* m, int64_t n, gp_batch_opts o) {
  o.separate_launches = 1;
  gp_batch* b = nullptr;
  need(gp_batch_create(&m, &n, 1, &o, &b) == GP_OK, "gp_batch_create");
  return b;
}

// The autotuner starts from the options that gp_step uses without it, tries
// sizes where a kernel has one, and adopts none that it has not measured to be
// faster (the stand-in's events measure nothing).
static void autotune() {
  gp_model* m = small_tree();
  for (int kernel : {GP_KERNEL_AUTO, GP_KERNEL_PLAIN}) {
    gp_batch_opts o{};
    o.kernel = kernel;
    gp_batch* b = batch_of(m, 3, o);
    fast_launches.clear();
    gp_batch_opts chosen{};
    double ms = -1.0;
    need(gp_batch_autotune(b, 1e-3, GP_SEMI_IMPLICIT_EULER, 50, &chosen, &ms) == GP_OK, "gp_batch_autotune");
    need(chosen.block_size == 0, "a workgroup size was adopted without a faster trial");
    const bool tree = kernel == GP_KERNEL_AUTO;
    need(tree == !fast_launches.empty(), "the tree kernel runs exactly by the automatic choice");
    if (tree) {
      need(fast_launches[0].block == 0, "the first trial is not the default's");
      for (int size : {64, 128, 256}) {
        bool tried = false;
        for (const FastLaunch& l : fast_launches) tried = tried || l.block == size;
        need(tried, "a workgroup size was not tried");
      }
      bool split = false;
      for (const FastLaunch& l : fast_launches) split = split || l.n_steps == 25;
      need(split, "fewer steps a launch were not tried");
    }
    gp_batch_destroy(b);
  }
  gp_model_destroy(m);
}

// Host calls reach the batch's device whatever device the calling thread has
// made current, and leave that as it was.
static void device() {
  gp_model* m[2] = {lone_body(GP_JOINT_FLOATING), lone_body(GP_JOINT_REVOLUTE)};
  const int64_t n[2] = {3, 2};
  gp_batch* b = nullptr;
  need(hipSetDevice(2) == hipSuccess && gp_batch_create(m, n, 2, nullptr, &b) == GP_OK, "gp_batch_create");
  need(hipSetDevice(5) == hipSuccess, "hipSetDevice");
  const int nq = 3 * 7 + 2, nv = 3 * 6 + 2, nm = 3 * 36 + 2;
  std::vector<double> q(nq, 0.5), v(nv, 0.25), out(nm), out2(nm);
  auto check = [&](int st, const char* call) {
    need(st == GP_OK, call);
    int now = -1;
    need(hipGetDevice(&now) == hipSuccess && now == 5, "the caller's device was changed");
    if (gp_host_null_stream_device != 2) {
      std::printf("%s launched on device %d, the batch is on 2\n", call, gp_host_null_stream_device);
      std::exit(1);
    }
    gp_host_null_stream_device = -1;
  };
  check(gp_batch_set_state(b, q.data(), v.data()), "gp_batch_set_state");
  check(gp_batch_set_tau(b, v.data()), "gp_batch_set_tau");
  check(gp_batch_get_state(b, out.data(), out2.data()), "gp_batch_get_state");
  check(gp_dynamics(b, nullptr, out.data()), "gp_dynamics");
  check(gp_dynamics(b, v.data(), out.data()), "gp_dynamics");
  check(gp_batch_get_vdot(b, out.data()), "gp_batch_get_vdot");
  check(gp_mass_matrix(b, out.data()), "gp_mass_matrix");
  check(gp_dynamics_bias(b, out.data()), "gp_dynamics_bias");
  gp_batch_destroy(b);
  for (gp_model* x : m) gp_model_destroy(x);
  need(hipSetDevice(0) == hipSuccess, "hipSetDevice");
}

// Steps of kernels that keep nothing in device scratch (trees, velocity stepping
// of a lone body or with one instance per wave) allocate none, nor does the
// preparation of their graphs; the plain kernel's do.
static void scratch() {
  gp_model* tree = small_tree();
  gp_model* body = lone_body(GP_JOINT_FLOATING);
  const struct { gp_model* m; int kernel, integrator, graph; bool uses; const char* what; } cases[] = {
      {tree, GP_KERNEL_AUTO, GP_VELOCITY_STEPPING, 0, false, "velocity stepping, one instance per wave"},
      {tree, GP_KERNEL_PLAIN, GP_VELOCITY_STEPPING, 0, true, "velocity stepping, one instance per lane"},
      {tree, GP_KERNEL_AUTO, GP_SEMI_IMPLICIT_EULER, 1, false, "graph of a tree's steps"},
      {tree, GP_KERNEL_PLAIN, GP_SEMI_IMPLICIT_EULER, 1, true, "graph of the plain kernel's steps"},
      {tree, GP_KERNEL_AUTO, GP_RUNGE_KUTTA_4, 1, true, "graph of a tree's Runge-Kutta steps"},
      {body, GP_KERNEL_AUTO, GP_CCD_VELOCITY_STEPPING, 1, false, "graph of a lone body's velocity stepping"},
      {tree, GP_KERNEL_AUTO, GP_VELOCITY_STEPPING, 1, false, "graph of velocity stepping, one instance per wave"},
  };
  for (const auto& c : cases) {
    gp_batch_opts o{};
    o.kernel = c.kernel;
    o.use_graph = c.graph;
    gp_batch* b = batch_of(c.m, 3, o);
    const size_t before = gp_host_malloc_calls;
    if (c.graph) (void)gp_step_prepare(b, 1e-3, c.integrator, 2, nullptr);  // the stand-in captures no graph
    else need(gp_step(b, 1e-3, c.integrator, 2, nullptr) == GP_OK, "gp_step");
    // a launch of the stand-in allocates its LDS
    const bool allocated = gp_host_malloc_calls - before > (c.graph || c.kernel == GP_KERNEL_PLAIN ? 0u : 1u);
    if (allocated != c.uses) {
      std::printf("%s: %s scratch\n", c.what, allocated ? "allocates" : "has no");
      std::exit(1);
    }
    gp_batch_destroy(b);
  }
  gp_model_destroy(tree);
  gp_model_destroy(body);
}

// A batch whose state only crosses as device arrays has no staging array for
// host ones; the first host transfer allocates it, once.
static void staging() {
  gp_model* m[2] = {lone_body(GP_JOINT_FLOATING), lone_body(GP_JOINT_REVOLUTE)};
  const int64_t n[2] = {3, 2};
  gp_batch* b = nullptr;
  need(gp_batch_create(m, n, 2, nullptr, &b) == GP_OK, "gp_batch_create");
  const int nq = 3 * 7 + 2, nv = 3 * 6 + 2;
  std::vector<double> q(nq, 0.5), v(nv, 0.25), q1(nq), v1(nv);
  size_t at = gp_host_malloc_bytes;
  auto grown = [&](size_t by, const char* what) {
    need(gp_host_malloc_bytes - at == by, what);
    at = gp_host_malloc_bytes;
  };
  // host memory is the stand-in's device memory
  need(gp_batch_set_state_dev(b, q.data(), v.data(), nullptr) == GP_OK, "gp_batch_set_state_dev");
  need(gp_batch_get_state_dev(b, q1.data(), v1.data(), nullptr) == GP_OK, "gp_batch_get_state_dev");
  need(q1 == q && v1 == v, "device arrays: the state read back differs");
  grown(0, "device-array calls allocated memory");
  need(gp_batch_get_state(b, q1.data(), v1.data()) == GP_OK, "gp_batch_get_state");
  need(q1 == q && v1 == v, "host arrays: the state read back differs");
  grown((nq + nv) * sizeof(double), "the first host transfer did not allocate the staging array");
  need(gp_batch_set_state(b, q1.data(), v1.data()) == GP_OK, "gp_batch_set_state");
  need(gp_batch_set_tau(b, nullptr) == GP_OK, "gp_batch_set_tau");
  grown(0, "a later host transfer allocated memory");
  gp_batch_destroy(b);
  for (gp_model* x : m) gp_model_destroy(x);
}

int main(int argc, char** argv) {
  need(argc == 2, "usage: runtime_host <check>");
  const struct { const char* name; void (*f)(); } checks[] = {
      {"autotune", autotune}, {"device", device}, {"scratch", scratch}, {"staging", staging}};
  for (const auto& c : checks)
    if (!std::strcmp(argv[1], c.name)) {
      c.f();
      std::printf("%s ok\n", c.name);
      return 0;
    }
  need(false, "no such check");
}
