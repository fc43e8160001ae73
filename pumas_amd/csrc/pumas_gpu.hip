/*
 * libpumas_hip: C ABI, table upload, geometry upload and the transport for
 * gfx950: the wavefront scheduler (scheduler.h), its kernels but the stepping
 * one (k_step.h), and their launches.
 */
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <mutex>
#include <vector>

#include "../../include/pumas_gpu.h"
#include "ptab.h"
#include "row_tables.h"
#include "scheduler.h"
#include "status.h"

/* ------------------------------------------------------------------------
 * Error reporting.
 * ------------------------------------------------------------------------ */
static thread_local char g_error[1024] = "";

enum pumas_return pg_fail(enum pumas_return rc, const char * fmt, ...)
{
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(g_error, sizeof(g_error), fmt, ap);
        va_end(ap);
        return rc;
}

void pg_clear_error(void) { g_error[0] = '\0'; }

extern "C" const char * pumas_gpu_error_message(void) { return g_error; }

/* A thread's buffer is its own until it ends, and then the next thread's: a
 * program with a thread per call would else allocate and free one in every call.
 * Up to PINNED_IDLE of them wait, the others are freed. The list is never
 * destroyed, as threads may end after static objects. Copies into pageable
 * memory are staged by the runtime, with a wait of their own. */
void * pg_pinned(size_t bytes)
{
        constexpr int PINNED_IDLE = 16;
        struct Idle {
                std::mutex mu;
                void * p[PINNED_IDLE];
                int n = 0;
        };
        static Idle & idle = *new Idle;
        struct Buffer {
                void * p = nullptr;
                ~Buffer()
                {
                        if (p == nullptr) return;
                        {
                                std::lock_guard<std::mutex> lock(idle.mu);
                                if (idle.n < PINNED_IDLE) {
                                        idle.p[idle.n++] = p;
                                        return;
                                }
                        }
                        (void)hipHostFree(p);
                }
        };
        static thread_local Buffer buffer;
        if (bytes > PG_PINNED_BYTES) return nullptr;
        if (buffer.p == nullptr) {
                std::lock_guard<std::mutex> lock(idle.mu);
                if (idle.n > 0) buffer.p = idle.p[--idle.n];
        }
        if ((buffer.p == nullptr) &&
            (hipHostMalloc(&buffer.p, PG_PINNED_BYTES,
                 hipHostMallocPortable) != hipSuccess)) {
                (void)hipGetLastError();
                buffer.p = nullptr;
        }
        return buffer.p;
}

extern "C" const char * pumas_gpu_version(void) { return "pumas_hip 0.1.0"; }

extern "C" void pumas_gpu_context_default(struct pumas_gpu_context * context)
{
        memset(context, 0x0, sizeof(*context));
        context->mode.energy_loss = PUMAS_MODE_STRAGGLED;
        context->mode.decay = PUMAS_MODE_WEIGHTED;
        context->mode.direction = PUMAS_MODE_FORWARD;
        context->mode.scattering = PUMAS_MODE_MIXED;
        context->event = PUMAS_EVENT_NONE;
        context->accuracy = 1E-02;
}

/* Device frame buffer and counter of a recorder (see pumas_gpu_recorder_*
 * below). */
struct pumas_gpu_recorder {
        Frame * frames;
        unsigned long long * count;
        unsigned long long capacity;
        int period;
        uint64_t first, n;
};

/* ------------------------------------------------------------------------
 * Physics upload.
 * ------------------------------------------------------------------------ */
struct pumas_gpu_physics {
        void * device;          /* one allocation holding every section */
        size_t size;
        PhysicsView view;
        ModelView models;
        FloatTables floats;     /* FP32 mirrors, in the same allocation */
        LdsTables lds_floats;   /* the same, as offsets in the LDS copy */
        uint32_t n_floats;      /* floats in the mirrors (multiple of 64) */
        const double * step;    /* packed copy of the FP64 step tables */
        LdsStepTables lds_step; /* their columns, as offsets in that copy */
        uint32_t n_step;        /* doubles in that copy (multiple of 8) */
        /* FP32-bulk LDS copy: the mirrors, then the FP64 tables of the range
         * to energy inversion (K, X, X_dK, K_dX, a_max, b_max; the other
         * columns of lds_range are not in it and not read). */
        LdsStepTables lds_range;
        uint32_t range_head;    /* doubles of K..K_dX at the head of step */
        uint32_t range_tail_at; /* a_max..b_max: from here to n_step */
        /* Row tables of the CSDA [0], and of the mixed and straggled [1]
         * energy losses, for the lean FP64 kernels' LDS copy. */
        const double * rows[ROW_SCHEMES];
        uint32_t n_rows;        /* doubles in each (even) */
        int particle;
};

namespace {

struct Section {
        std::string name;
        uint32_t dtype;
        uint64_t count;
        uint64_t offset;
};

/* Parse a PTAB image; sections index into `image`. */
enum pumas_return parse_ptab(const uint8_t * image, size_t size,
    ptab_header * header, std::vector<Section> & sections)
{
        if (size < sizeof(ptab_header))
                return pg_fail(PUMAS_RETURN_FORMAT_ERROR, "PTAB image too small");
        memcpy(header, image, sizeof(*header));
        if (memcmp(header->magic, PTAB_MAGIC, 8) != 0)
                return pg_fail(PUMAS_RETURN_FORMAT_ERROR, "not a PTAB image");
        if (header->version != PTAB_VERSION)
                return pg_fail(PUMAS_RETURN_FORMAT_ERROR,
                    "unsupported PTAB version %u", header->version);
        const size_t dir_end = sizeof(ptab_header) +
            (size_t)header->n_entries * sizeof(ptab_entry);
        if (dir_end > size)
                return pg_fail(PUMAS_RETURN_INCOMPLETE_FILE, "truncated PTAB");
        const ptab_entry * e =
            reinterpret_cast<const ptab_entry *>(image + sizeof(ptab_header));
        for (uint32_t i = 0; i < header->n_entries; i++) {
                const size_t width = (e[i].dtype == PTAB_F64) ? 8 : 4;
                if (e[i].offset + e[i].count * width > size)
                        return pg_fail(PUMAS_RETURN_INCOMPLETE_FILE,
                            "truncated PTAB section %s", e[i].name);
                char name[PTAB_NAME_LEN + 1] = { 0 };
                memcpy(name, e[i].name, PTAB_NAME_LEN);
                sections.push_back({ name, e[i].dtype, e[i].count, e[i].offset });
        }
        return PUMAS_RETURN_SUCCESS;
}

const Section * find(const std::vector<Section> & s, const char * name)
{
        for (const auto & x : s)
                if (x.name == name) return &x;
        return nullptr;
}

} /* namespace */

extern "C" enum pumas_return pumas_gpu_physics_upload_memory(
    const void * ptab, size_t size, pumas_gpu_physics ** physics)
{
        if (physics == NULL)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR, "physics is NULL");
        *physics = NULL;
        const uint8_t * image = static_cast<const uint8_t *>(ptab);
        ptab_header h;
        std::vector<Section> sections;
        enum pumas_return rc = parse_ptab(image, size, &h, sections);
        if (rc != PUMAS_RETURN_SUCCESS) return rc;

        if (h.imeta[PTAB_MAX_COMPONENTS] > MAX_COMPONENTS)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                    "materials with more than %d elements are not supported",
                    MAX_COMPONENTS);

        /* Row tables, by energy loss scheme; the first reading of the file's
         * sizes, which it checks. */
        const int nM = h.imeta[PTAB_N_MATERIALS];
        std::vector<double> rows;
        const char * const bad = pack_row_tables(
            [&](const char * name) {
                    const Section * s = find(sections, name);
                    return ((s == nullptr) || (s->dtype != PTAB_F64)) ?
                        RowSource { nullptr, 0 } :
                        RowSource { reinterpret_cast<const double *>(
                                        image + s->offset),
                                s->count };
            },
            nM, h.imeta[PTAB_N_ENERGIES], rows);
        if (bad != nullptr)
                return pg_fail(PUMAS_RETURN_FORMAT_ERROR,
                    "PTAB section `%s' is missing or short", bad);
        const size_t n_rows = rows.size() / ROW_SCHEMES;

        /* Derived section: first component of each material. */
        const Section * sin = find(sections, "elements_in");
        if ((sin == nullptr) || (sin->count < (uint64_t)nM))
                return pg_fail(PUMAS_RETURN_FORMAT_ERROR, "missing elements_in");
        std::vector<int32_t> component0(nM);
        {
                const int32_t * ein =
                    reinterpret_cast<const int32_t *>(image + sin->offset);
                int acc = 0;
                for (int m = 0; m < nM; m++) {
                        component0[m] = acc;
                        acc += ein[m];
                }
        }

        /* Single precision mirrors of the tables read every step by the
         * FP32-bulk engine, appended after the derived sections. */
        static const char * const mirrored[] = { "K", "X", "X_dK", "dE",
                "dE_dK", "Omega", "Omega_dK", "CS", "CS_dK", "Mu0", "Mu0_dK",
                "Ms1", "Ms1_dK", "Lb", "a_max", "b_max" };
        const int n_mirrored = sizeof(mirrored) / sizeof(mirrored[0]);
        std::vector<float> floats;
        std::vector<size_t> float_at(n_mirrored);
        for (int k = 0; k < n_mirrored; k++) {
                const Section * sec = find(sections, mirrored[k]);
                if ((sec == nullptr) || (sec->dtype != PTAB_F64))
                        return pg_fail(PUMAS_RETURN_FORMAT_ERROR,
                            "PTAB section `%s' is missing", mirrored[k]);
                float_at[k] = floats.size();
                const double * src =
                    reinterpret_cast<const double *>(image + sec->offset);
                for (uint64_t i = 0; i < sec->count; i++)
                        floats.push_back((float)src[i]);
                while (floats.size() % 64) floats.push_back(0.f);
        }

        /* The FP64 tables read by every step, packed for the LDS copy of
         * the FP64 stepping kernel (columns padded to 64 B). */
        static const char * const stepped[] = { "K", "X", "X_dK", "K_dX",
                "dE", "dE_dK", "Omega", "Omega_dK", "CS", "CS_dK", "Mu0",
                "Mu0_dK", "Ms1", "Ms1_dK", "Lb", "a_max", "b_max" };
        const int n_stepped = sizeof(stepped) / sizeof(stepped[0]);
        std::vector<double> step;
        std::vector<size_t> step_at(n_stepped);
        for (int k = 0; k < n_stepped; k++) {
                const Section * sec = find(sections, stepped[k]);
                if ((sec == nullptr) || (sec->dtype != PTAB_F64))
                        return pg_fail(PUMAS_RETURN_FORMAT_ERROR,
                            "PTAB section `%s' is missing", stepped[k]);
                step_at[k] = step.size();
                const double * src =
                    reinterpret_cast<const double *>(image + sec->offset);
                step.insert(step.end(), src, src + sec->count);
                while (step.size() % 8) step.push_back(0.);
        }

        /* Coarse index of the kinetic energy grid (k_index_fast). */
        std::vector<int16_t> coarse(4096);
        int k_bin0 = 0;
        {
                const Section * sk = find(sections, "K");
                const double * Kh =
                    reinterpret_cast<const double *>(image + sk->offset);
                const int nb = k_coarse_build(Kh, (int)sk->count,
                    coarse.data(), (int)coarse.size(), &k_bin0);
                coarse.resize(nb);
        }

        /* Device image: the PTAB file as is, then the derived sections. */
        const size_t extra_offset = (size + 255) / 256 * 256;
        const size_t float_offset = (extra_offset +
            component0.size() * sizeof(int32_t) + 255) / 256 * 256;
        const size_t step_offset = (float_offset +
            floats.size() * sizeof(float) + 255) / 256 * 256;
        const size_t coarse_offset = (step_offset +
            step.size() * sizeof(double) + 255) / 256 * 256;
        const size_t rows_offset = (coarse_offset +
            coarse.size() * sizeof(int16_t) + 255) / 256 * 256;
        const size_t total = rows_offset + rows.size() * sizeof(double);
        void * device = nullptr;
        HIP_TRY(hipMalloc(&device, total));
        /* The derived sections in one copy. */
        std::vector<uint8_t> derived(total - extra_offset, 0);
        auto place = [&](size_t offset, const void * src, size_t bytes) {
                if (bytes > 0)
                        memcpy(derived.data() + (offset - extra_offset), src,
                            bytes);
        };
        place(extra_offset, component0.data(),
            component0.size() * sizeof(int32_t));
        place(float_offset, floats.data(), floats.size() * sizeof(float));
        place(step_offset, step.data(), step.size() * sizeof(double));
        place(coarse_offset, coarse.data(), coarse.size() * sizeof(int16_t));
        place(rows_offset, rows.data(), rows.size() * sizeof(double));
        hipError_t e1 = hipMemcpy(device, image, size, hipMemcpyHostToDevice);
        hipError_t e2 = hipMemcpy((uint8_t *)device + extra_offset,
            derived.data(), derived.size(), hipMemcpyHostToDevice);
        if ((e1 != hipSuccess) || (e2 != hipSuccess)) {
                (void)hipFree(device);
                return pg_fail(PUMAS_RETURN_INTERNAL_ERROR,
                    "could not copy the tables to the device");
        }

        pumas_gpu_physics * ph = new pumas_gpu_physics();
        ph->device = device;
        ph->size = total;
        ph->particle = h.imeta[PTAB_PARTICLE];
        PhysicsView & v = ph->view;
        v.n_energies = h.imeta[PTAB_N_ENERGIES];
        v.n_materials = nM;
        v.n_elements = h.imeta[PTAB_N_ELEMENTS];
        v.n_components = h.imeta[PTAB_N_COMPONENTS];
        v.n_table_dcs = h.imeta[PTAB_N_TABLE_DCS];
        v.max_components = h.imeta[PTAB_MAX_COMPONENTS];
        v.mass = h.fmeta[PTAB_MASS];
        v.ctau = h.fmeta[PTAB_CTAU];
        v.cutoff = h.fmeta[PTAB_CUTOFF];

        const uint8_t * base = static_cast<const uint8_t *>(device);
        bool missing = false;
        std::string missing_name;
        auto dptr = [&](const char * name) -> const void * {
                const Section * s = find(sections, name);
                if (s == nullptr) {
                        missing = true;
                        missing_name = name;
                        return nullptr;
                }
                return base + s->offset;
        };
#define D64(field, name) v.field = (const double *)dptr(name)
#define F32(field, name) v.field = (const float *)dptr(name)
#define I32(field, name) v.field = (const int *)dptr(name)
        D64(K, "K");
        D64(K_dX, "K_dX");
        D64(K_dNI_in, "K_dNI_in");
        D64(K_dNI_el, "K_dNI_el");
        D64(X, "X");
        D64(X_dK, "X_dK");
        D64(X_dT, "X_dT");
        D64(T, "T");
        D64(T_dK, "T_dK");
        D64(dE, "dE");
        D64(dE_dK, "dE_dK");
        D64(Omega, "Omega");
        D64(Omega_dK, "Omega_dK");
        D64(NI_el, "NI_el");
        D64(NI_el_dK, "NI_el_dK");
        D64(NI_in, "NI_in");
        D64(NI_in_dK, "NI_in_dK");
        D64(CS, "CS");
        D64(CS_dK, "CS_dK");
        D64(CSf, "CSf");
        D64(CSf_dK, "CSf_dK");
        D64(CSn, "CSn");
        D64(CSn_dK, "CSn_dK");
        D64(Kt, "Kt");
        D64(a_max, "a_max");
        D64(b_max, "b_max");
        D64(Mu0, "Mu0");
        D64(Mu0_dK, "Mu0_dK");
        D64(Lb, "Lb");
        D64(Lb_dK, "Lb_dK");
        D64(Ms1, "Ms1");
        D64(Ms1_dK, "Ms1_dK");
        D64(material_density, "material_density");
        D64(component_fraction, "component_fraction");
        D64(element_Z, "element_Z");
        D64(element_A, "element_A");
        D64(element_I, "element_I");
        D64(element_nscr, "element_n_screening");
        D64(element_amplitude, "element_amplitude");
        D64(element_exponent, "element_exponent");
        D64(element_rn, "element_nuclear_radius");
        D64(element_lrad, "element_radiation_log");
        F32(DCS, "DCS");
        F32(DCS_x, "DCS_x");
        F32(DCS_envelope, "DCS_envelope");
        I32(elements_in, "elements_in");
        I32(component_element, "component_element");
        I32(element_index, "element_index");
        v.material_component0 = (const int *)(base + extra_offset);
        v.k_coarse = coarse.empty() ? nullptr :
            (const int16_t *)(base + coarse_offset);
        v.k_bin0 = k_bin0;
        v.k_nbins = (int)coarse.size();

        FloatTables & ft = ph->floats;
        {
                const float * fbase =
                    (const float *)((const uint8_t *)device + float_offset);
                const float * const * fields[] = { &ft.K, &ft.X, &ft.X_dK,
                        &ft.dE, &ft.dE_dK, &ft.Omega, &ft.Omega_dK, &ft.CS,
                        &ft.CS_dK, &ft.Mu0, &ft.Mu0_dK, &ft.Ms1, &ft.Ms1_dK,
                        &ft.Lb, &ft.a_max, &ft.b_max };
                for (int k = 0; k < n_mirrored; k++)
                        *const_cast<const float **>(fields[k]) =
                            fbase + float_at[k];
                ft.n_energies = v.n_energies;
                ft.n_materials = v.n_materials;
                ft.mass = (float)v.mass;

                LdsTables & lt = ph->lds_floats;
                LdsFloats * lfields[] = { &lt.K, &lt.X, &lt.X_dK, &lt.dE,
                        &lt.dE_dK, &lt.Omega, &lt.Omega_dK, &lt.CS,
                        &lt.CS_dK, &lt.Mu0, &lt.Mu0_dK, &lt.Ms1, &lt.Ms1_dK,
                        &lt.Lb, &lt.a_max, &lt.b_max };
                static_assert(sizeof(lfields) / sizeof(lfields[0]) ==
                        sizeof(fields) / sizeof(fields[0]),
                    "one LDS column per mirrored table");
                for (int k = 0; k < n_mirrored; k++)
                        lfields[k]->off = (uint32_t)float_at[k];
                lt.n_energies = ft.n_energies;
                lt.n_materials = ft.n_materials;
                lt.mass = ft.mass;
                ph->n_floats = (uint32_t)floats.size();
        }
        {
                LdsStepTables & st = ph->lds_step;
                LdsDoubles * columns[] = { &st.K, &st.X, &st.X_dK, &st.K_dX,
                        &st.dE, &st.dE_dK, &st.Omega, &st.Omega_dK, &st.CS,
                        &st.CS_dK, &st.Mu0, &st.Mu0_dK, &st.Ms1, &st.Ms1_dK,
                        &st.Lb, &st.a_max, &st.b_max };
                static_assert(sizeof(columns) / sizeof(columns[0]) ==
                        sizeof(stepped) / sizeof(stepped[0]),
                    "one LDS column per stepped table");
                for (int k = 0; k < n_stepped; k++)
                        columns[k]->off = (uint32_t)step_at[k];
                st.n_energies = v.n_energies;
                st.n_materials = v.n_materials;
                st.mass = v.mass;
                st.k_coarse = v.k_coarse;
                st.k_bin0 = v.k_bin0;
                st.k_nbins = v.k_nbins;
                ph->step = (const double *)((const uint8_t *)device +
                    step_offset);
                ph->n_step = (uint32_t)step.size();
                ph->rows[0] = (const double *)((const uint8_t *)device +
                    rows_offset);
                ph->rows[1] = ph->rows[0] + n_rows;
                ph->n_rows = (uint32_t)n_rows;

                /* In the FP32-bulk copy, K..K_dX (the first four stepped
                 * columns) and a_max, b_max (the last two) follow the
                 * mirrors. */
                static_assert(n_stepped == 17, "stepped columns");
                ph->range_head = (uint32_t)step_at[4];
                ph->range_tail_at = (uint32_t)step_at[15];
                const uint32_t base = ph->n_floats / 2;
                LdsStepTables & rt = ph->lds_range;
                memset(&rt, 0x0, sizeof(rt));
                rt.n_energies = st.n_energies;
                rt.n_materials = st.n_materials;
                rt.mass = st.mass;
                rt.k_coarse = st.k_coarse;
                rt.k_bin0 = st.k_bin0;
                rt.k_nbins = st.k_nbins;
                rt.K.off = base + (uint32_t)step_at[0];
                rt.X.off = base + (uint32_t)step_at[1];
                rt.X_dK.off = base + (uint32_t)step_at[2];
                rt.K_dX.off = base + (uint32_t)step_at[3];
                rt.a_max.off = base + ph->range_head;
                rt.b_max.off = base + ph->range_head +
                    (uint32_t)(step_at[16] - step_at[15]);
        }

        ModelView & mv = ph->models;
        mv.z13 = (const double *)dptr("element_z13");
        mv.zm13 = (const double *)dptr("element_zm13");
        mv.z23 = (const double *)dptr("element_z23");
        mv.dn = (const double *)dptr("element_dn");
        mv.lrad = v.element_lrad;
        mv.cst = (const double *)dptr("constants");
        mv.gq9_x = (const double *)dptr("gq9_x");
        mv.gq9_w = (const double *)dptr("gq9_w");
        mv.gq12_x = (const double *)dptr("gq12_x");
        mv.gq12_w = (const double *)dptr("gq12_w");
#undef D64
#undef F32
#undef I32
        if (missing) {
                (void)hipFree(device);
                delete ph;
                return pg_fail(PUMAS_RETURN_FORMAT_ERROR,
                    "PTAB section `%s' is missing", missing_name.c_str());
        }
        *physics = ph;
        return PUMAS_RETURN_SUCCESS;
}

extern "C" enum pumas_return pumas_gpu_physics_upload(
    const char * path, pumas_gpu_physics ** physics)
{
        if (physics != NULL) *physics = NULL;
        FILE * f = fopen(path, "rb");
        if (f == NULL)
                return pg_fail(PUMAS_RETURN_PATH_ERROR, "could not open `%s'", path);
        fseek(f, 0, SEEK_END);
        const long size = ftell(f);
        fseek(f, 0, SEEK_SET);
        std::vector<uint8_t> image(size > 0 ? size : 0);
        const size_t n = fread(image.data(), 1, image.size(), f);
        fclose(f);
        if (n != image.size())
                return pg_fail(PUMAS_RETURN_IO_ERROR, "could not read `%s'", path);
        return pumas_gpu_physics_upload_memory(image.data(), image.size(),
            physics);
}

extern "C" void pumas_gpu_physics_destroy(pumas_gpu_physics ** physics)
{
        if ((physics == NULL) || (*physics == NULL)) return;
        (void)hipFree((*physics)->device);
        delete *physics;
        *physics = NULL;
}

extern "C" int pumas_gpu_physics_n_materials(const pumas_gpu_physics * p)
{
        return p->view.n_materials;
}

extern "C" int pumas_gpu_physics_n_energies(const pumas_gpu_physics * p)
{
        return p->view.n_energies;
}

extern "C" double pumas_gpu_physics_cutoff(const pumas_gpu_physics * p)
{
        return p->view.cutoff;
}

/* ------------------------------------------------------------------------
 * Geometry.
 * ------------------------------------------------------------------------ */
struct pumas_gpu_geometry {
        pg_geometry view;        /* device pointers */
        std::vector<void *> allocations;
};

namespace {

template <typename T>
enum pumas_return upload(pumas_gpu_geometry * g, const T * src, size_t n,
    const T ** dst)
{
        void * d = nullptr;
        HIP_TRY(hipMalloc(&d, n * sizeof(T) > 0 ? n * sizeof(T) : 1));
        g->allocations.push_back(d);
        HIP_TRY(hipMemcpy(d, src, n * sizeof(T), hipMemcpyHostToDevice));
        *dst = static_cast<const T *>(d);
        return PUMAS_RETURN_SUCCESS;
}

} /* namespace */

extern "C" void pumas_gpu_geometry_destroy(pumas_gpu_geometry ** geometry)
{
        if ((geometry == NULL) || (*geometry == NULL)) return;
        for (void * p : (*geometry)->allocations) (void)hipFree(p);
        delete *geometry;
        *geometry = NULL;
}

extern "C" enum pumas_return pumas_gpu_geometry_create(
    const pumas_gpu_physics * physics,
    const struct pumas_gpu_geometry_desc * desc, pumas_gpu_geometry ** out)
{
        if (out == NULL) return pg_fail(PUMAS_RETURN_VALUE_ERROR, "NULL output");
        *out = NULL;
        if ((physics == NULL) || (desc == NULL))
                return pg_fail(PUMAS_RETURN_VALUE_ERROR, "NULL argument");
        if ((desc->n_media <= 0) || (desc->media == NULL))
                return pg_fail(PUMAS_RETURN_MEDIUM_ERROR, "no media");
        bool uniform = true;
        for (int i = 0; i < desc->n_media; i++) {
                const struct pumas_gpu_medium & medium = desc->media[i];
                const int m = medium.material;
                if ((m < 0) || (m >= physics->view.n_materials))
                        return pg_fail(PUMAS_RETURN_INDEX_ERROR,
                            "invalid material index [%d] for medium %d", m, i);
                if (medium.locals == PUMAS_GPU_LOCALS_UNIFORM) continue;
                if (medium.locals != PUMAS_GPU_LOCALS_EXPONENTIAL)
                        return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                            "invalid locals kind %d for medium %d",
                            (int)medium.locals, i);
                if (!(medium.scale > 0.) || !(medium.scale < INFINITY) ||
                    !(medium.cos_min > 0.) || !(medium.cos_min <= 1.) ||
                    !(fabs(medium.z_ref) < INFINITY))
                        return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                            "medium %d: an exponential profile needs a finite "
                            "scale > 0, a finite z_ref and cos_min in (0, 1]",
                            i);
                const bool allowed =
                    (desc->kind == PUMAS_GPU_GEOMETRY_INFINITE) ||
                    (desc->kind == PUMAS_GPU_GEOMETRY_SLABS) ||
                    ((desc->kind == PUMAS_GPU_GEOMETRY_TERRAIN) && (i == 0));
                if (!allowed)
                        return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                            "medium %d: non uniform locals apply to the media "
                            "of infinite and slab geometries and to the air "
                            "of a terrain", i);
                uniform = false;
        }

        pumas_gpu_geometry * g = new pumas_gpu_geometry();
        pg_geometry & v = g->view;
        memset(&v, 0x0, sizeof(v));
        v.kind = desc->kind;
        v.step_type = desc->step_type;
        v.n_media = desc->n_media;
        std::vector<int> material(desc->n_media);
        std::vector<double> density(desc->n_media);
        for (int i = 0; i < desc->n_media; i++) {
                material[i] = desc->media[i].material;
                density[i] = desc->media[i].density;
        }
        enum pumas_return rc;
#define UP(src, n, dst)                                                        \
        do {                                                                   \
                rc = upload(g, src, n, dst);                                   \
                if (rc != PUMAS_RETURN_SUCCESS) {                              \
                        pumas_gpu_geometry_destroy(&g);                        \
                        return rc;                                             \
                }                                                              \
        } while (0)
        UP(material.data(), material.size(), &v.material);
        UP(density.data(), density.size(), &v.density);
        if (!uniform) {
                std::vector<pg_locals> locals(desc->n_media);
                for (int i = 0; i < desc->n_media; i++) {
                        const struct pumas_gpu_medium & m = desc->media[i];
                        locals[i].kind = (int)m.locals;
                        locals[i].scale = m.scale;
                        locals[i].z_ref = m.z_ref;
                        locals[i].cos_min = m.cos_min;
                }
                UP(locals.data(), locals.size(), &v.locals);
        }

        switch (desc->kind) {
        case PUMAS_GPU_GEOMETRY_INFINITE:
                break;
        case PUMAS_GPU_GEOMETRY_SLABS:
                if ((desc->n_layers <= 0) || (desc->z == NULL) ||
                    (desc->n_media < desc->n_layers)) {
                        pumas_gpu_geometry_destroy(&g);
                        return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                            "slabs need n_layers + 1 boundaries and media");
                }
                for (int i = 0; i < desc->n_layers; i++)
                        if (!(desc->z[i] < desc->z[i + 1])) {
                                pumas_gpu_geometry_destroy(&g);
                                return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                                    "slab boundaries must increase");
                        }
                v.n_layers = desc->n_layers;
                UP(desc->z, (size_t)desc->n_layers + 1, &v.z);
                break;
        case PUMAS_GPU_GEOMETRY_TERRAIN: {
                if ((desc->nx < 2) || (desc->ny < 2) || (desc->height == NULL) ||
                    (desc->density == NULL) || (desc->n_media < 2) ||
                    (desc->dx <= 0.) || (desc->dy <= 0.)) {
                        pumas_gpu_geometry_destroy(&g);
                        return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                            "invalid terrain description");
                }
                v.nx = desc->nx;
                v.ny = desc->ny;
                v.x0 = desc->x0;
                v.y0 = desc->y0;
                v.z0 = desc->z0;
                v.dx = desc->dx;
                v.dy = desc->dy;
                v.z_top = desc->z_top;
                UP(desc->height, (size_t)desc->nx * desc->ny, &v.height);
                UP(desc->density, (size_t)(desc->nx - 1) * (desc->ny - 1),
                    &v.cell_density);
                break;
        }
        case PUMAS_GPU_GEOMETRY_VOXELS: {
                if ((desc->nx < 1) || (desc->ny < 1) || (desc->nz < 1) ||
                    (desc->label == NULL) || (desc->density == NULL) ||
                    (desc->dx <= 0.) || (desc->dy <= 0.) || (desc->dz <= 0.)) {
                        pumas_gpu_geometry_destroy(&g);
                        return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                            "invalid voxel description");
                }
                const size_t nv = (size_t)desc->nx * desc->ny * desc->nz;
                if (nv >= (size_t)0x7fffffff) {
                        pumas_gpu_geometry_destroy(&g);
                        return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                            "too many voxels");
                }
                for (size_t i = 0; i < nv; i++)
                        if (desc->label[i] >= desc->n_media) {
                                pumas_gpu_geometry_destroy(&g);
                                return pg_fail(PUMAS_RETURN_INDEX_ERROR,
                                    "voxel %zu has an invalid label", i);
                        }
                v.nx = desc->nx;
                v.ny = desc->ny;
                v.nz = desc->nz;
                v.x0 = desc->x0;
                v.y0 = desc->y0;
                v.z0 = desc->z0;
                v.dx = desc->dx;
                v.dy = desc->dy;
                v.dz = desc->dz;
                UP(desc->label, nv, &v.label);
                UP(desc->density, nv, &v.cell_density);
                break;
        }
        default:
                pumas_gpu_geometry_destroy(&g);
                return pg_fail(PUMAS_RETURN_VALUE_ERROR, "unknown geometry kind");
        }
#undef UP
        *out = g;
        return PUMAS_RETURN_SUCCESS;
}

/* Load history i, whose state is at `s`, into a walker. */
__device__ __forceinline__ void walker_load(const KernelArgs & a, uint64_t i,
    Walker & w, const struct pumas_state * s)
{
        Track & t = w.t;
        t.charge = s->charge;
        t.energy = s->energy;
        t.distance = s->distance;
        t.grammage = s->grammage;
        t.time = s->time;
        t.weight = s->weight;
        t.pos[0] = s->position[0];
        t.pos[1] = s->position[1];
        t.pos[2] = s->position[2];
        t.dir[0] = s->direction[0];
        t.dir[1] = s->direction[1];
        t.dir[2] = s->direction[2];
        t.decayed = s->decayed;
        t.step_first = 0;
        t.step_event = t.step_foreseen = 0;
        t.step_X_limit = t.step_invlb1 = t.lifetime = 0.;
        t.randn_done = 0;
        t.randn_next = 0.;
        t.ix.reset(a.p.n_energies);
        t.fx.reset(a.p.n_energies);
        t.rng.init(a.seed, a.first + i, STREAM_TRANSPORT, 0);
        t.steps = 0;
        t.max_steps = a.max_steps;
}

/* Entry of every history of the batch; one lane per history. The
 * block's states (104 B records, 26 KB per block) are staged through LDS:
 * read from HBM with consecutive lanes on consecutive 8 B words, and
 * written back the same way (unchanged for the histories that go on to
 * the stepping kernel), instead of each lane touching its own record with
 * 104 B strides. */
constexpr int INIT_BLOCK = 256;

/* 16 B at an 8 B aligned address (global or LDS), by value. */
__device__ __forceinline__ double2 load16(const double * p)
{
        double2 v;
        __builtin_memcpy(&v, p, sizeof(v));
        return v;
}

__device__ __forceinline__ void store16(double * p, double2 v)
{
        __builtin_memcpy(p, &v, sizeof(v));
}

template <bool F32, bool CLOSED>
__global__ void __launch_bounds__(INIT_BLOCK)
    __attribute__((amdgpu_waves_per_eu(CLOSED ? 5 : 1))) k_init(KernelArgs args)
{
        KERNEL_ARGS(args);
        __shared__ struct pumas_state stage[INIT_BLOCK];
        const EngineT<F32> eng = { a.p, a.mv, a.c, a.g, a.ft, a.p, a.rec };
        const uint64_t base = (uint64_t)blockIdx.x * INIT_BLOCK;
        const uint64_t i = base + threadIdx.x;
        const bool active = i < a.n;
        const uint32_t words = (uint32_t)(
            ((a.n - base < INIT_BLOCK) ? a.n - base : INIT_BLOCK) *
            (sizeof(struct pumas_state) / sizeof(double)));
        double * const lds = reinterpret_cast<double *>(stage);
        double * const hbm = reinterpret_cast<double *>(a.states + base);
        constexpr uint32_t WORDS =
            INIT_BLOCK * (sizeof(struct pumas_state) / sizeof(double));
        /* A full block moves 16 B words (states are 8 B aligned; the
         * 16 B loads and stores need no more): 6.5 per lane. */
        constexpr uint32_t PAIRS = WORDS / 2;
        constexpr uint32_t PER_LANE = (PAIRS + INIT_BLOCK - 1) / INIT_BLOCK;
        static_assert(sizeof(struct pumas_state) % sizeof(double) == 0,
            "states are staged as 8 B words");
        static_assert(WORDS % 2 == 0, "a block holds whole 16 B words");
        if (words == WORDS) {
                /* Every load of the lane issued before the first wait (a
                 * loop with a runtime bound waits on each load in turn,
                 * one HBM round trip per word). */
                /* Words k < PER_LANE - 1 exist for every lane; the last
                 * for the first PAIRS % INIT_BLOCK lanes. */
                const bool tail = threadIdx.x + (PER_LANE - 1) * INIT_BLOCK <
                    PAIRS;
                double2 v[PER_LANE];
#pragma unroll
                for (uint32_t k = 0; k < PER_LANE - 1; k++)
                        v[k] = load16(hbm + 2 * (threadIdx.x + k * INIT_BLOCK));
                v[PER_LANE - 1] = tail ? load16(hbm + 2 * (threadIdx.x +
                    (PER_LANE - 1) * INIT_BLOCK)) : v[0];
#pragma unroll
                for (uint32_t k = 0; k < PER_LANE - 1; k++)
                        store16(lds + 2 * (threadIdx.x + k * INIT_BLOCK), v[k]);
                if (tail)
                        store16(lds + 2 * (threadIdx.x +
                            (PER_LANE - 1) * INIT_BLOCK), v[PER_LANE - 1]);
        } else {
                for (uint32_t k = threadIdx.x; k < words; k += INIT_BLOCK)
                        lds[k] = hbm[k];
        }
        __syncthreads();
        Walker w;
        w.phase = PHASE_EMPTY;
        if (active) {
                walker_load(a, i, w, stage + threadIdx.x);
                eng.template walker_init<CLOSED>(w);
                if (w.phase == PHASE_DONE)
                        walker_store(a, i, w, w, stage + threadIdx.x);
                if (!CLOSED && (w.phase == PHASE_STEP)) a.records[i] = w;
        }
        __syncthreads();
        if (words == WORDS) {
                const bool tail = threadIdx.x + (PER_LANE - 1) * INIT_BLOCK <
                    PAIRS;
                double2 v[PER_LANE];
#pragma unroll
                for (uint32_t k = 0; k < PER_LANE - 1; k++)
                        v[k] = load16(lds + 2 * (threadIdx.x + k * INIT_BLOCK));
                v[PER_LANE - 1] = tail ? load16(lds + 2 * (threadIdx.x +
                    (PER_LANE - 1) * INIT_BLOCK)) : v[0];
#pragma unroll
                for (uint32_t k = 0; k < PER_LANE - 1; k++)
                        store16(hbm + 2 * (threadIdx.x + k * INIT_BLOCK), v[k]);
                if (tail)
                        store16(hbm + 2 * (threadIdx.x +
                            (PER_LANE - 1) * INIT_BLOCK), v[PER_LANE - 1]);
        } else {
                for (uint32_t k = threadIdx.x; k < words; k += INIT_BLOCK)
                        hbm[k] = lds[k];
        }
        if (!CLOSED)
                queue_append(a.counters + C_STEP_N0, a.q_step[0],
                    w.phase == PHASE_STEP, (uint32_t)i);
}

/* Default maximum number of lanes of a wavefront waiting for an elastic
 * hard scattering before the wavefront processes them together. */
constexpr int EHS_BATCH = 16;

/* Clears the per-round counters before round `parity`. */
__global__ void k_round(unsigned long long * c, int parity)
{
        if (threadIdx.x == 0) {
                c[C_TAKEN] = 0;
                c[C_DEL_N] = 0;
                c[C_STEP_N0 + (parity ^ 1)] = 0;
        }
}

/* Inelastic DELs of round `parity`, one lane per queued history; the
 * histories go back to the next round's step queue. */
template <bool F32>
__global__ void __launch_bounds__(256, 2) k_del(KernelArgs args, int parity)
{
        KERNEL_ARGS(args);
        const EngineT<F32> eng = { a.p, a.mv, a.c, a.g, a.ft, a.p, a.rec };
        const unsigned long long n = a.counters[C_DEL_N];
        const uint32_t * queue = a.q_del;
        const int lane = threadIdx.x & 63;
        const unsigned long long stride = (unsigned long long)gridDim.x *
            blockDim.x;
        unsigned long long steps_acc = 0;
        for (unsigned long long base = (unsigned long long)blockIdx.x *
                     blockDim.x + (threadIdx.x & ~63u);
             base < n; base += stride) {
                const unsigned long long k = base + lane;
                const bool active = k < n;
                Walker w;
                w.phase = PHASE_EMPTY;
                uint32_t slot = 0;
                if (active) {
                        slot = queue[k];
                        w = a.records[slot];
                        eng.walker_del(w);
                        if (w.phase == PHASE_DONE) {
                                walker_store(a, slot, w, w, a.states + slot);
                                steps_acc += w.t.steps;
                        } else {
                                a.records[slot] = w;
                        }
                }
                queue_append(a.counters + C_STEP_N0 + (parity ^ 1),
                    a.q_step[parity ^ 1], w.phase == PHASE_STEP, slot);
        }
        steps_flush(a, steps_acc);
}

/* Clears the counters (a kernel, not a memset node, so that the launch
 * sequence can be captured in a graph). */
__global__ void zero_counters(unsigned long long * c, int n)
{
        if ((int)threadIdx.x < n) c[threadIdx.x] = 0ull;
}

size_t pg_bytes_per_history(void) { return sizeof(Walker) + 3 * sizeof(uint32_t); }

/* ------------------------------------------------------------------------
 * C ABI transport.
 * ------------------------------------------------------------------------ */
namespace {

/* Histories per chunk: the records of a chunk take MAX_CHUNK * sizeof(Walker)
 * bytes of HBM (about 11 GB). */
constexpr size_t MAX_CHUNK = size_t(1) << 25;

/* Histories per chunk of a closed form launch, which keeps no records or
 * queues and indexes its histories in 64 bits: bounded by the entry
 * kernel's grid (2^30 lanes), so that a large batch is one launch and one
 * counter read instead of one per 2^25 histories. */
constexpr size_t MAX_CLOSED_CHUNK = size_t(1) << 30;

/* Default number of rounds launched between two reads of the queue
 * lengths, and its maximum. */
constexpr int ROUNDS_PER_CHECK = 16;
constexpr int MAX_ROUNDS_PER_CHECK = 256;

/* Launch geometry and optional timing of the stepping kernel. */
struct Launch {
        int n_cu, block, per_cu, rounds_per_check;
        bool graph;
        int tail_del; /* <0 never, >0 always, 0: rounds of few histories */
        int lanes_per_wave; /* 1..64, or 0: spread small batches */
        unsigned lds_bytes; /* LDS copy of the step tables, or 0 */
        unsigned step_grid, del_grid;
        hipStream_t stream;
        hipEvent_t * marks; /* [2 * rounds_per_check] or NULL */
        hipEvent_t * init_marks; /* [2], around the entry kernel, or NULL */
        hipEvent_t end_mark; /* after the last kernel, or NULL */
        bool closed; /* every history takes the closed form CSDA */
};

/* Whether the stepping kernel reads the row tables from its LDS copy. */
bool row_launch(const KernelArgs & a, bool f32)
{
        return !f32 && (a.c.energy_loss >= MODE_CSDA) &&
            (a.c.energy_loss <= MODE_STRAGGLED);
}

StepKernel launch_kernel(const KernelArgs & a, bool f32, bool lds)
{
        const int loss = a.c.energy_loss;
        if (a.rec.frames != nullptr)
                return f32 ? step_kernel<true, true>(loss, lds) :
                             step_kernel<false, true>(loss, lds);
        return f32 ? step_kernel<true, false>(loss, lds) :
                     step_kernel<false, false>(loss, lds);
}

template <bool F32>
void launch_step(const KernelArgs & a, int parity, const Launch & L)
{
        hipLaunchKernelGGL(launch_kernel(a, F32, L.lds_bytes > 0),
            dim3(L.step_grid), dim3(L.block), L.lds_bytes, L.stream, a, parity);
}

template <bool F32>
enum pumas_return launch_round(
    const KernelArgs & a, int parity, const Launch & L, int r)
{
        hipStream_t stream = L.stream;
        hipLaunchKernelGGL(k_round, dim3(1), dim3(64), 0, stream, a.counters,
            parity);
        if (L.marks) HIP_TRY(hipEventRecord(L.marks[2 * r], stream));
        launch_step<F32>(a, parity, L);
        if (L.marks) HIP_TRY(hipEventRecord(L.marks[2 * r + 1], stream));
        hipLaunchKernelGGL(k_del<F32>, dim3(L.del_grid), dim3(256), 0,
            stream, a, parity);
        HIP_TRY(hipGetLastError());
        return PUMAS_RETURN_SUCCESS;
}

enum pumas_return allow_lds(StepKernel kernel, int bytes)
{
        HIP_TRY(hipFuncSetAttribute((const void *)kernel,
            hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        return PUMAS_RETURN_SUCCESS;
}

/* Bytes of the LDS copy of the tables in the stepping kernel, or 0 when the
 * step tables (the FP32 mirrors in FP32-bulk) do not fit `per_cu` times in the
 * LDS of a CU; sets the pieces of the copy. FP64 launches with energy loss copy
 * the row tables instead, which are smaller: they hold one energy loss scheme. */
enum pumas_return lds_tables_size(const pumas_gpu_physics * physics,
    KernelArgs & a, int device, int per_cu, bool f32, unsigned * bytes)
{
        *bytes = 0;
        size_t need = f32 ?
            (size_t)physics->n_floats * sizeof(float) +
                (size_t)(physics->range_head + physics->n_step -
                    physics->range_tail_at) * sizeof(double) :
            (size_t)physics->n_step * sizeof(double);
        int per_block = 0, per_sm = 0;
        HIP_TRY(hipDeviceGetAttribute(
            &per_block, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
        HIP_TRY(hipDeviceGetAttribute(&per_sm,
            hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, device));
        if ((need > (size_t)per_block) || (need * per_cu > (size_t)per_sm))
                return PUMAS_RETURN_SUCCESS;
        if (row_launch(a, f32)) {
                const int scheme = (a.c.energy_loss == MODE_CSDA) ? 0 : 1;
                need = physics->n_rows * sizeof(double);
                a.lds_piece[0] = { (const float4 *)physics->rows[scheme], 0,
                        physics->n_rows / 2 };
                a.n_lds_pieces = 1;
                a.rowl.n_energies = physics->view.n_energies;
                a.rowl.n_materials = physics->view.n_materials;
                a.rowl.mass = physics->view.mass;
        }
        if (need > 65536) {
                const enum pumas_return rc =
                    allow_lds(launch_kernel(a, f32, true), (int)need);
                if (rc != PUMAS_RETURN_SUCCESS) return rc;
        }
        *bytes = (unsigned)need;
        return PUMAS_RETURN_SUCCESS;
}

/* Device memory and graph of a chunk, released on every return path. */
struct ChunkResources {
        hipStream_t stream;
        void * mem = nullptr;
        hipGraphExec_t exec = nullptr;

        ~ChunkResources()
        {
                if (exec) (void)hipGraphExecDestroy(exec);
                if (mem) (void)hipFreeAsync(mem, stream);
        }
};

/* Device bytes of the per-chunk buffers (counters, records, queues) of a
 * chunk of m histories. */
constexpr size_t chunk_bytes(size_t m)
{
        return 256 + (((m * sizeof(Walker)) + 255) & ~size_t(255)) +
            3 * (((m * sizeof(uint32_t)) + 255) & ~size_t(255));
}

/* Transport histories [base, base + m) of the batch described by `a0`.
 * The chunk's buffers are allocated on the stream, or taken from `fixed`
 * (at least chunk_bytes(m) bytes of device memory) when it is given. */
enum pumas_return transport_chunk(const KernelArgs & a0, size_t base,
    size_t m, bool f32, Launch L, unsigned long long * total_steps,
    unsigned long long * error, struct pumas_gpu_stats * stats,
    void * fixed = nullptr)
{
        /* No more resident blocks than the chunk fills with histories: with a
         * given number of lanes per wavefront, a small request leaves the rest
         * of the device to concurrent requests. */
        const size_t resident = (size_t)L.n_cu * L.per_cu;
        const size_t waves = (size_t)(L.block / 64);
        /* Spread (0): as many blocks as histories, up to all the resident
         * ones, each of which takes a CU; a round that fits in them shares its
         * histories out over their wavefronts (k_step). */
        const bool lanes_auto = L.lanes_per_wave <= 0;
        const int lanes = lanes_auto ? 64 : L.lanes_per_wave;
        const size_t per_block = lanes_auto ? 1 : waves * (size_t)lanes;
        const size_t fill = (m + per_block - 1) / per_block;
        L.step_grid = (unsigned)((fill < resident) ? (fill > 0 ? fill : 1) :
                                                     resident);
        const size_t del_fill = (m + 255) / 256;
        const size_t del_max = (size_t)L.n_cu * 2;
        L.del_grid = (unsigned)((del_fill < del_max) ?
                (del_fill > 0 ? del_fill : 1) :
                del_max);
        hipStream_t stream = L.stream;
        KernelArgs a = a0;
        a.lanes_per_wave = lanes;
        a.lanes_auto = lanes_auto;
        a.resident_lanes = L.step_grid * (uint32_t)(waves * lanes);
        a.wave_del_max = WAVE_DEL_ROUNDS * a.resident_lanes;
        a.tail_del = L.tail_del;
        a.states = a0.states + base;
        a.n = m;
        a.first = a0.first + base;
        if (a0.events) a.events = a0.events + base;
        if (a0.media) a.media = a0.media + 2 * base;
        if (a0.steps) a.steps = a0.steps + base;
        if (a0.draws) a.draws = a0.draws + base;
        if (a0.rc) a.rc = a0.rc + base;

        ChunkResources res;
        res.stream = stream;
        const size_t b_counters = 256;
        /* A closed form launch needs no records or queues. */
        const size_t b_records = L.closed ? 0 :
            ((m * sizeof(Walker)) + 255) & ~size_t(255);
        const size_t b_queue = L.closed ? 0 :
            ((m * sizeof(uint32_t)) + 255) & ~size_t(255);
        char * ptr;
        if (fixed) {
                ptr = static_cast<char *>(fixed);
        } else {
                HIP_TRY(hipMallocAsync(
                    &res.mem, b_counters + b_records + 3 * b_queue, stream));
                ptr = static_cast<char *>(res.mem);
        }
        a.counters = reinterpret_cast<unsigned long long *>(ptr);
        a.records = reinterpret_cast<Walker *>(ptr + b_counters);
        char * q = ptr + b_counters + b_records;
        a.q_step[0] = reinterpret_cast<uint32_t *>(q);
        a.q_step[1] = reinterpret_cast<uint32_t *>(q + b_queue);
        a.q_del = reinterpret_cast<uint32_t *>(q + 2 * b_queue);

        enum pumas_return rc = PUMAS_RETURN_SUCCESS;
        unsigned long long stack[C_COUNT];
        void * const pinned = fixed ? nullptr : pg_pinned(sizeof(stack));
        unsigned long long * const host =
            pinned ? static_cast<unsigned long long *>(pinned) : stack;
        hipLaunchKernelGGL(zero_counters, dim3(1), dim3(64), 0, stream,
            a.counters, C_COUNT);
        const unsigned blocks = (unsigned)((m + INIT_BLOCK - 1) / INIT_BLOCK);
        if (L.init_marks) HIP_TRY(hipEventRecord(L.init_marks[0], stream));
        if (f32 && L.closed)
                hipLaunchKernelGGL((k_init<true, true>), dim3(blocks),
                    dim3(INIT_BLOCK), 0, stream, a);
        else if (f32)
                hipLaunchKernelGGL((k_init<true, false>), dim3(blocks),
                    dim3(INIT_BLOCK), 0, stream, a);
        else if (L.closed)
                hipLaunchKernelGGL((k_init<false, true>), dim3(blocks),
                    dim3(INIT_BLOCK), 0, stream, a);
        else
                hipLaunchKernelGGL((k_init<false, false>), dim3(blocks),
                    dim3(INIT_BLOCK), 0, stream, a);
        if (L.init_marks) HIP_TRY(hipEventRecord(L.init_marks[1], stream));
        if (hipGetLastError() != hipSuccess)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                    "transport kernel launch failed");
        /* A batch that needs one round (its DELs run in the wavefronts):
         * the stepping kernel alone, launched without waiting for the entry
         * kernel's count of the histories to step. */
        const bool single = !L.closed && ((L.tail_del > 0) ||
            ((L.tail_del == 0) && (m <= a.wave_del_max)));
        /* The sequence of rounds between two checks is captured once in a
         * HIP graph and replayed (an even number of rounds, so that every
         * replay starts on step queue 0): one launch per check instead of
         * three per round. Counters are cleared by kernels, not memset
         * nodes. */
        if (L.graph && !L.closed && !single) {
                hipGraph_t graph = nullptr;
                HIP_TRY(hipStreamBeginCapture(
                    stream, hipStreamCaptureModeThreadLocal));
                int p = 0;
                for (int r = 0; r < L.rounds_per_check; r++, p ^= 1) {
                        rc = f32 ? launch_round<true>(a, p, L, r) :
                                   launch_round<false>(a, p, L, r);
                        if (rc != PUMAS_RETURN_SUCCESS) break;
                }
                const hipError_t e = hipStreamEndCapture(stream, &graph);
                if (rc != PUMAS_RETURN_SUCCESS) {
                        if (graph) (void)hipGraphDestroy(graph);
                        return rc;
                }
                HIP_TRY(e);
                const hipError_t ei =
                    hipGraphInstantiate(&res.exec, graph, nullptr, nullptr, 0);
                (void)hipGraphDestroy(graph);
                HIP_TRY(ei);
        }
        int parity = 0, launched = 0;
        bool init_timed = false;
        if (single) {
                if (L.marks) HIP_TRY(hipEventRecord(L.marks[0], stream));
                if (f32)
                        launch_step<true>(a, 0, L);
                else
                        launch_step<false>(a, 0, L);
                if (L.marks) HIP_TRY(hipEventRecord(L.marks[1], stream));
                HIP_TRY(hipGetLastError());
                if (stats) stats->rounds += 1;
                launched = 1;
                parity = 1;
        }
        for (;;) {
                /* The end of the call's work, unless more rounds follow. */
                if (L.end_mark) HIP_TRY(hipEventRecord(L.end_mark, stream));
                HIP_TRY(hipMemcpyAsync(host, a.counters,
                    C_COUNT * sizeof(*host), hipMemcpyDeviceToHost, stream));
                HIP_TRY(hipStreamSynchronize(stream));
                if (L.init_marks && stats && !init_timed) {
                        float ms = 0.f;
                        HIP_TRY(hipEventElapsedTime(&ms, L.init_marks[0],
                            L.init_marks[1]));
                        stats->init_kernel_ms += ms;
                        init_timed = true;
                }
                if (L.marks && stats) {
                        for (int r = 0; r < launched; r++) {
                                float ms = 0.f;
                                HIP_TRY(hipEventElapsedTime(&ms,
                                    L.marks[2 * r], L.marks[2 * r + 1]));
                                stats->step_kernel_ms += ms;
                        }
                }
                if (stats) stats->step_launches += launched;
                launched = 0;
                if (host[C_STEP_N0 + parity] == 0) break;
                if (stats) stats->rounds += 1;
                if (res.exec) {
                        HIP_TRY(hipGraphLaunch(res.exec, stream));
                        launched = L.rounds_per_check;
                        continue;
                }
                for (int r = 0; r < L.rounds_per_check; r++) {
                        rc = f32 ? launch_round<true>(a, parity, L, r) :
                                   launch_round<false>(a, parity, L, r);
                        if (rc != PUMAS_RETURN_SUCCESS) break;
                        launched++;
                        parity ^= 1;
                }
                if (rc != PUMAS_RETURN_SUCCESS) break;
        }
        *total_steps += host[C_STEPS];
        if ((*error == 0) && (host[C_ERROR] != 0)) *error = host[C_ERROR];
        if (stats) {
                stats->step_limited += host[C_STATUS];
                stats->loop_limited += host[C_STATUS_LOOP];
                stats->no_target += host[C_STATUS_TARGET];
        }
        if (res.mem) {
                void * mem = res.mem;
                res.mem = nullptr;
                HIP_TRY(hipFreeAsync(mem, stream));
        }
        return rc;
}


enum pumas_return check_context(const pumas_gpu_physics * physics,
    const struct pumas_gpu_context * c)
{
        if ((c->accuracy <= 0) || (c->accuracy > 1))
                return pg_fail(PUMAS_RETURN_ACCURACY_ERROR,
                    "bad accuracy value (expected a value in ]0,1], got %g)",
                    c->accuracy);
        if ((c->mode.direction == PUMAS_MODE_BACKWARD) &&
            (c->mode.energy_loss > PUMAS_MODE_CSDA) &&
            (physics->view.cutoff < 1E-02))
                return pg_fail(PUMAS_RETURN_ACCURACY_ERROR,
                    "bad cutoff value for backward transport (expected a "
                    "value greater than or equal to 0.01, got %g)",
                    physics->view.cutoff);
        if ((physics->particle != 0) &&
            (c->mode.direction == PUMAS_MODE_FORWARD) &&
            (c->mode.decay == PUMAS_MODE_WEIGHTED))
                return pg_fail(PUMAS_RETURN_DECAY_ERROR,
                    "`PUMAS_MODE_WEIGHTED' mode is not valid for forward taus");
        return PUMAS_RETURN_SUCCESS;
}

} /* namespace */

/* The transport call. With `fixed` (device memory for chunk_bytes(n)
 * bytes) nothing is allocated: no chunk buffers, no graph (eager
 * launches), no timing events (stats then hold counts only). */
static enum pumas_return transport_impl(const pumas_gpu_physics * physics,
    const struct pumas_gpu_context * context,
    const pumas_gpu_geometry * geometry, struct pumas_state * states, size_t n,
    uint64_t seed, uint64_t first_history,
    const struct pumas_gpu_outputs * outputs,
    const struct pumas_gpu_options * options, struct pumas_gpu_stats * stats,
    void * stream_, void * fixed)
{
        if ((physics == NULL) || (context == NULL) || (geometry == NULL))
                return pg_fail(PUMAS_RETURN_VALUE_ERROR, "NULL argument");
        if ((states == NULL) && (n > 0))
                return pg_fail(PUMAS_RETURN_VALUE_ERROR, "no states (null)");
        enum pumas_return rc = check_context(physics, context);
        if (rc != PUMAS_RETURN_SUCCESS) return rc;
        const int precision =
            options ? options->precision : PUMAS_GPU_PRECISION_FP64;
        if ((precision != PUMAS_GPU_PRECISION_FP64) &&
            (precision != PUMAS_GPU_PRECISION_FP32_BULK))
                return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                    "unknown precision mode %d", precision);
        hipStream_t stream = static_cast<hipStream_t>(stream_);

        KernelArgs a;
        memset(&a, 0x0, sizeof(a));
        a.p = physics->view;
        a.mv = physics->models;
        a.ft = physics->floats;
        a.ftl = physics->lds_floats;
        if (precision == PUMAS_GPU_PRECISION_FP32_BULK) {
                a.stl = physics->lds_range;
                const uint32_t nf4 = physics->n_floats / 4;
                const uint32_t head4 = physics->range_head / 2;
                a.lds_piece[0] = { (const float4 *)physics->floats.K, 0, nf4 };
                a.lds_piece[1] = { (const float4 *)physics->step, nf4, head4 };
                a.lds_piece[2] = { (const float4 *)(physics->step +
                                       physics->range_tail_at),
                        nf4 + head4,
                        (physics->n_step - physics->range_tail_at) / 2 };
                a.n_lds_pieces = 3;
        } else {
                a.stl = physics->lds_step;
                a.lds_piece[0] = { (const float4 *)physics->step, 0,
                        physics->n_step / 2 };
                a.n_lds_pieces = 1;
        }
        a.c.energy_loss = context->mode.energy_loss;
        a.c.decay = context->mode.decay;
        a.c.direction = context->mode.direction;
        a.c.scattering = context->mode.scattering;
        a.c.event = context->event;
        a.c.limit_energy = context->limit.energy;
        a.c.limit_distance = context->limit.distance;
        a.c.limit_grammage = context->limit.grammage;
        a.c.limit_time = context->limit.time;
        a.c.accuracy = context->accuracy;
        a.c.loop_max = (options && options->max_loop > 0) ? options->max_loop :
                                                            LOOP_MAX_DEFAULT;
        a.g = geometry->view;
        a.states = states;
        a.n = n;
        a.seed = seed;
        a.first = first_history;
        if (outputs) {
                a.events = outputs->events;
                a.media = outputs->media;
                a.steps = outputs->steps;
                a.draws = outputs->draws;
                a.rc = outputs->rc;
        }
        a.max_steps = (options && options->max_steps > 0) ? options->max_steps :
                                                            10000000;
        a.ehs_batch = (options && options->ehs_batch > 0) ? options->ehs_batch :
                                                            EHS_BATCH;
        if (options && options->recorder) {
                const pumas_gpu_recorder * r = options->recorder;
                a.rec.frames = r->frames;
                a.rec.count = r->count;
                a.rec.capacity = r->capacity;
                a.rec.period = r->period;
                a.rec.first = r->first;
                a.rec.last = r->first + r->n;
        }
        if (a.ehs_batch > 64)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                    "ehs_batch must be at most 64 (got %d)", a.ehs_batch);

        int device;
        HIP_TRY(hipGetDevice(&device));
        int n_cu = 0;
        HIP_TRY(hipDeviceGetAttribute(
            &n_cu, hipDeviceAttributeMultiprocessorCount, device));
        /* Default launch: 8 resident wavefronts per CU, as one block of
         * 512 lanes (one LDS copy of the step tables per CU). */
        const int block = (options && options->block_size > 0) ?
            options->block_size :
            512;
        if ((block % 64) || (block > 512))
                return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                    "block size must be a multiple of 64, at most 512");
        const int per_cu = (options && options->blocks_per_cu > 0) ?
            options->blocks_per_cu :
            (512 / block > 0 ? 512 / block : 1);
        int rounds_per_check = (options && options->rounds_per_check > 0) ?
            options->rounds_per_check :
            ROUNDS_PER_CHECK;
        rounds_per_check += rounds_per_check & 1; /* even, for the graph */
        if (rounds_per_check > MAX_ROUNDS_PER_CHECK)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                    "rounds_per_check must be at most %d",
                    MAX_ROUNDS_PER_CHECK);

        /* Timing events, destroyed on every return path. */
        struct Events {
                hipEvent_t e0 = nullptr, e1 = nullptr;
                hipEvent_t init[2] = { nullptr, nullptr };
                std::vector<hipEvent_t> marks;

                ~Events()
                {
                        if (e0) (void)hipEventDestroy(e0);
                        if (e1) (void)hipEventDestroy(e1);
                        for (auto & e : init)
                                if (e) (void)hipEventDestroy(e);
                        for (auto & e : marks)
                                if (e) (void)hipEventDestroy(e);
                }
        } ev;
        if (stats && !fixed) {
                HIP_TRY(hipEventCreate(&ev.e0));
                HIP_TRY(hipEventCreate(&ev.e1));
                HIP_TRY(hipEventCreate(&ev.init[0]));
                HIP_TRY(hipEventCreate(&ev.init[1]));
                HIP_TRY(hipEventRecord(ev.e0, stream));
        }
        const bool f32 = (precision == PUMAS_GPU_PRECISION_FP32_BULK);
        unsigned lds_bytes = 0;
        if (!(options && options->lds_tables < 0)) {
                rc = lds_tables_size(
                    physics, a, device, per_cu, f32, &lds_bytes);
                if (rc != PUMAS_RETURN_SUCCESS) return rc;
        }
        /* Every history takes the closed form CSDA when the geometry has
         * no step limits (a uniform infinite medium), the energy loss is
         * CSDA and scattering is disabled (src/pumas.c:3200-3230). */
        const bool closed = (geometry->view.kind == GEO_INFINITE) &&
            (geometry->view.locals == nullptr) &&
            (context->mode.energy_loss == PUMAS_MODE_CSDA) &&
            (context->mode.scattering == PUMAS_MODE_DISABLED);
        unsigned long long total_steps = 0, error = 0;
        /* The legacy NULL stream cannot be captured. */
        const bool graph = !(options && options->eager) &&
            (stream != nullptr) && !fixed;
        if (stats) {
                memset(stats, 0x0, sizeof(*stats));
                if (!graph && !fixed && !closed) {
                        ev.marks.resize(2 * rounds_per_check, nullptr);
                        for (auto & e : ev.marks)
                                HIP_TRY(hipEventCreate(&e));
                }
        }
        /* Per-launch timing of the stepping kernel needs eager launches:
         * events recorded inside a graph cannot be timed. */
        const int tail_del = options ? options->tail_del : 0;
        int lanes_per_wave = options ? options->lanes_per_wave : 0;
        if (lanes_per_wave > 64)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                    "lanes_per_wave must be at most 64 (got %d)",
                    lanes_per_wave);
        const Launch L = { n_cu, block, per_cu, rounds_per_check, graph,
                tail_del, lanes_per_wave, lds_bytes, 0, 0, stream,
                ev.marks.empty() ? nullptr : ev.marks.data(),
                (stats && !fixed) ? ev.init : nullptr,
                (stats && !fixed) ? ev.e1 : nullptr, closed };
        const size_t chunk = closed ? MAX_CLOSED_CHUNK : MAX_CHUNK;
        for (size_t base = 0; base < n; base += chunk) {
                const size_t m = (n - base < chunk) ? n - base : chunk;
                rc = transport_chunk(
                    a, base, m, f32, L, &total_steps, &error, stats, fixed);
                if (rc != PUMAS_RETURN_SUCCESS) break;
        }
        /* Every chunk has waited for its last kernel; an error ended the call
         * between two of its launches, and an empty batch has no chunk: the
         * call returns with the stream's work done all the same. */
        if ((rc != PUMAS_RETURN_SUCCESS) || (n == 0))
                HIP_TRY(hipStreamSynchronize(stream));
        if (stats) {
                float ms = 0.f;
                if (!fixed && (n > 0) && (rc == PUMAS_RETURN_SUCCESS))
                        HIP_TRY(hipEventElapsedTime(&ms, ev.e0, ev.e1));
                stats->steps = total_steps;
                stats->histories = n;
                stats->kernel_ms = ms;
                stats->lds_bytes = lds_bytes;
        }
        if (rc != PUMAS_RETURN_SUCCESS) return rc;
        if (error != 0)
                return pg_fail((enum pumas_return)error,
                    "a history raised error code %llu", error);
        return PUMAS_RETURN_SUCCESS;
}

extern "C" enum pumas_return pumas_gpu_transport(
    const pumas_gpu_physics * physics, const struct pumas_gpu_context * context,
    const pumas_gpu_geometry * geometry, struct pumas_state * states, size_t n,
    uint64_t seed, uint64_t first_history,
    const struct pumas_gpu_outputs * outputs,
    const struct pumas_gpu_options * options, struct pumas_gpu_stats * stats,
    void * stream)
{
        pg_clear_error();
        return transport_impl(physics, context, geometry, states, n, seed,
            first_history, outputs, options, stats, stream, nullptr);
}

/* Public layout of the reference's struct pumas_context
 * (include/pumas.h:636-672): four host pointers (medium and random
 * callbacks, recorder, user data), then the value part, laid out as
 * struct pumas_gpu_context (mode, event, limit, accuracy). */
struct reference_context_layout {
        void * medium;
        void * random;
        void * recorder;
        void * user_data;
        struct pumas_gpu_context values;
};
static_assert(offsetof(reference_context_layout, values) == 32,
    "reference context: four pointers before its mode");
static_assert(offsetof(struct pumas_gpu_context, event) == 16 &&
        offsetof(struct pumas_gpu_context, limit) == 24 &&
        offsetof(struct pumas_gpu_context, accuracy) == 56,
    "value part of the reference context");

extern "C" void pumas_gpu_context_from_reference(
    const struct pumas_context * context, struct pumas_gpu_context * out)
{
        if ((context == NULL) || (out == NULL)) return;
        memcpy(out,
            &reinterpret_cast<const reference_context_layout *>(context)
                 ->values,
            sizeof(*out));
}

extern "C" enum pumas_return pumas_gpu_transport_context(
    const pumas_gpu_physics * physics, const struct pumas_context * context,
    const pumas_gpu_geometry * geometry, struct pumas_state * states, size_t n,
    uint64_t seed, uint64_t first_history,
    const struct pumas_gpu_outputs * outputs,
    const struct pumas_gpu_options * options, struct pumas_gpu_stats * stats,
    void * stream)
{
        pg_clear_error();
        if (context == NULL)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR, "NULL context");
        struct pumas_gpu_context values;
        pumas_gpu_context_from_reference(context, &values);
        return transport_impl(physics, &values, geometry, states, n, seed,
            first_history, outputs, options, stats, stream, nullptr);
}

/* ------------------------------------------------------------------------
 * Transport without allocations.
 *
 * The per-chunk buffers of the transport (counters, in-flight records,
 * queues) live in one file-scope device array per GPU, so that callers
 * that cannot allocate device memory (code under stream capture, serving
 * loops, harnesses that forbid hipMalloc) can transport batches of up to
 * PUMAS_GPU_NOALLOC_MAX_HISTORIES histories. In host code the array's name
 * is not a device address: its address on each device is looked up once
 * with hipGetSymbolAddress and only that pointer is passed to kernels.
 * The counters are cleared by a kernel at the start of every call; the
 * records and queues are written before they are read. Every call on a
 * GPU shares that GPU's array: calls that overlap on one GPU race.
 * ------------------------------------------------------------------------ */
constexpr size_t NOALLOC_BYTES = chunk_bytes(PUMAS_GPU_NOALLOC_MAX_HISTORIES);
static_assert(PUMAS_GPU_NOALLOC_MAX_HISTORIES <= MAX_CHUNK, "one chunk");

static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_lock;
void * g_scratch[MAX_DEVICES];

/* The device address of `scratch` on the current device (looked up on the
 * first call on that device). */
enum pumas_return scratch_pointer(void ** out)
{
        int device = 0;
        HIP_TRY(hipGetDevice(&device));
        if ((device < 0) || (device >= MAX_DEVICES))
                return pg_fail(PUMAS_RETURN_INDEX_ERROR,
                    "device %d beyond the %d supported", device, MAX_DEVICES);
        std::lock_guard<std::mutex> guard(g_scratch_lock);
        if (g_scratch[device] == nullptr) {
                void * ptr = nullptr;
                const hipError_t e =
                    hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
                if ((e != hipSuccess) || (ptr == nullptr))
                        return pg_fail(PUMAS_RETURN_MEMORY_ERROR,
                            "hipGetSymbolAddress(scratch): %s",
                            hipGetErrorString(e));
                g_scratch[device] = ptr;
        }
        *out = g_scratch[device];
        return PUMAS_RETURN_SUCCESS;
}
} /* namespace */

extern "C" enum pumas_return pumas_gpu_transport_noalloc(
    const pumas_gpu_physics * physics, const struct pumas_gpu_context * context,
    const pumas_gpu_geometry * geometry, struct pumas_state * states, size_t n,
    uint64_t seed, uint64_t first_history,
    const struct pumas_gpu_outputs * outputs,
    const struct pumas_gpu_options * options, struct pumas_gpu_stats * stats,
    void * stream)
{
        pg_clear_error();
        if (n > PUMAS_GPU_NOALLOC_MAX_HISTORIES)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR,
                    "%zu histories exceed the %d of the transport without "
                    "allocations (use pumas_gpu_transport, or split the "
                    "batch)", n, PUMAS_GPU_NOALLOC_MAX_HISTORIES);
        void * fixed = nullptr;
        const enum pumas_return rc = scratch_pointer(&fixed);
        if (rc != PUMAS_RETURN_SUCCESS) return rc;
        return transport_impl(physics, context, geometry, states, n, seed,
            first_history, outputs, options, stats, stream, fixed);
}

/* ------------------------------------------------------------------------
 * Frame recorder.
 * ------------------------------------------------------------------------ */
static_assert(sizeof(Frame) == sizeof(struct pumas_gpu_frame),
    "Frame and struct pumas_gpu_frame must have the same layout");

extern "C" enum pumas_return pumas_gpu_recorder_create(size_t capacity,
    int period, uint64_t first_history, uint64_t n_histories,
    pumas_gpu_recorder ** recorder)
{
        pg_clear_error();
        if (recorder == NULL)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR, "NULL argument");
        *recorder = nullptr;
        auto * r = new pumas_gpu_recorder();
        r->capacity = capacity;
        r->period = period;
        r->first = first_history;
        r->n = n_histories;
        r->frames = nullptr;
        r->count = nullptr;
        hipError_t e = hipMalloc((void **)&r->count, sizeof(*r->count));
        if (e == hipSuccess)
                e = hipMalloc((void **)&r->frames,
                    (capacity > 0 ? capacity : 1) * sizeof(Frame));
        if (e == hipSuccess) e = hipMemset(r->count, 0x0, sizeof(*r->count));
        if (e != hipSuccess) {
                (void)hipFree(r->count);
                (void)hipFree(r->frames);
                delete r;
                return pg_fail(PUMAS_RETURN_MEMORY_ERROR,
                    "could not allocate the recorder (%s)",
                    hipGetErrorString(e));
        }
        *recorder = r;
        return PUMAS_RETURN_SUCCESS;
}

extern "C" void pumas_gpu_recorder_destroy(pumas_gpu_recorder ** recorder)
{
        if ((recorder == NULL) || (*recorder == NULL)) return;
        (void)hipFree((*recorder)->frames);
        (void)hipFree((*recorder)->count);
        delete *recorder;
        *recorder = nullptr;
}

extern "C" enum pumas_return pumas_gpu_recorder_clear(
    pumas_gpu_recorder * recorder)
{
        pg_clear_error();
        if (recorder == NULL)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR, "NULL recorder");
        HIP_TRY(hipMemset(recorder->count, 0x0, sizeof(*recorder->count)));
        return PUMAS_RETURN_SUCCESS;
}

extern "C" enum pumas_return pumas_gpu_recorder_read(
    const pumas_gpu_recorder * recorder, struct pumas_gpu_frame * frames,
    size_t max_frames, uint64_t * length)
{
        pg_clear_error();
        if (recorder == NULL)
                return pg_fail(PUMAS_RETURN_VALUE_ERROR, "NULL recorder");
        unsigned long long count = 0;
        HIP_TRY(hipMemcpy(&count, recorder->count, sizeof(count),
            hipMemcpyDeviceToHost));
        if (length) *length = count;
        size_t k = (count < recorder->capacity) ? count : recorder->capacity;
        if (k > max_frames) k = max_frames;
        if ((k > 0) && frames)
                HIP_TRY(hipMemcpy(frames, recorder->frames, k * sizeof(Frame),
                    hipMemcpyDeviceToHost));
        return PUMAS_RETURN_SUCCESS;
}

extern "C" enum pumas_return pumas_gpu_transport_host(
    const pumas_gpu_physics * physics, const struct pumas_gpu_context * context,
    const pumas_gpu_geometry * geometry, struct pumas_state * states, size_t n,
    uint64_t seed, uint64_t first_history,
    const struct pumas_gpu_outputs * outputs,
    const struct pumas_gpu_options * options, struct pumas_gpu_stats * stats)
{
        /* Device copies, freed on every return path. The outputs are
         * cleared first, so that a call that fails before its first launch
         * returns the input states and zero outputs. */
        struct Buffers {
                struct pumas_state * states = nullptr;
                struct pumas_gpu_outputs out = {};
                hipStream_t stream = nullptr;
                ~Buffers()
                {
                        if (stream) {
                                (void)hipStreamSynchronize(stream);
                                (void)hipStreamDestroy(stream);
                        }
                        (void)hipFree(states);
                        (void)hipFree(out.events);
                        (void)hipFree(out.media);
                        (void)hipFree(out.steps);
                        (void)hipFree(out.draws);
                        (void)hipFree(out.rc);
                }
        } b;
        const size_t ns = n > 0 ? n : 1;
        HIP_TRY(hipMalloc(&b.states, ns * sizeof(*states)));
        HIP_TRY(hipMemcpy(b.states, states, n * sizeof(*states),
            hipMemcpyHostToDevice));
#define PG_OUT(field, count)                                                  \
        if (outputs && outputs->field) {                                       \
                HIP_TRY(hipMalloc(&b.out.field,                                \
                    (count) * ns * sizeof(*outputs->field)));                  \
                HIP_TRY(hipMemset(b.out.field, 0x0,                            \
                    (count) * ns * sizeof(*outputs->field)));                  \
        }
        PG_OUT(events, 1)
        PG_OUT(media, 2)
        PG_OUT(steps, 1)
        PG_OUT(draws, 1)
        PG_OUT(rc, 1)
#undef PG_OUT
        /* A stream of its own: the legacy NULL stream cannot be captured
         * in a graph. */
        HIP_TRY(hipStreamCreateWithFlags(&b.stream, hipStreamNonBlocking));
        const enum pumas_return rc = pumas_gpu_transport(physics, context,
            geometry, b.states, n, seed, first_history, &b.out, options, stats,
            b.stream);
        HIP_TRY(hipStreamSynchronize(b.stream));
        const std::string message = g_error;
        HIP_TRY(hipMemcpy(states, b.states, n * sizeof(*states),
            hipMemcpyDeviceToHost));
#define PG_BACK(field, count)                                                 \
        if (outputs && outputs->field)                                         \
                HIP_TRY(hipMemcpy(outputs->field, b.out.field,                 \
                    (count) * n * sizeof(*outputs->field),                     \
                    hipMemcpyDeviceToHost));
        PG_BACK(events, 1)
        PG_BACK(media, 2)
        PG_BACK(steps, 1)
        PG_BACK(draws, 1)
        PG_BACK(rc, 1)
#undef PG_BACK
        snprintf(g_error, sizeof(g_error), "%s", message.c_str());
        return rc;
}
