/*
 * Drives the host layer's scene upload against a device that only remembers
 * what it was last given. Every edit of a small scene is uploaded once without
 * a fault and once for every upload step with that step failing on the first
 * try; after the second try the device must hold the same scene.
 * Prints one line per difference; exits with their number.
 */
#include "internal.h"
#include "vkrt_mi355x.h"

#include <stdio.h>
#include <stdlib.h>
#include <string.h>

enum { GEOMETRY, MESHES, PLACE, BUILD, MATERIALS, ALPHA, TEXTURES, LIGHTS, ENVIRONMENT, STEPS };
static const char* kStep[STEPS] = {"geometry", "meshes",   "place",  "build",      "materials",
                                   "alpha",    "textures", "lights", "environment"};
static uint64_t held[STEPS]; /* fingerprint of what each step last uploaded */
static int failing = -1;
static long mallocsLeft = -1; /* the malloc after this many fails; negative: none */

void* __real_malloc(size_t size);
void* __wrap_malloc(size_t size) {
    if (mallocsLeft >= 0 && mallocsLeft-- == 0) return NULL;
    return __real_malloc(size);
}

static uint64_t mix(uint64_t h, const void* data, size_t size) {
    const uint8_t* b = (const uint8_t*)data;
    h = (h ^ size) * 0x9E3779B97F4A7C15ull;
    for (size_t i = 0; data && i < size; i++) h = (h ^ b[i]) * 0x100000001B3ull;
    return h;
}
static int keep(int step, uint64_t h) {
    if (step == failing) {
        failing = -1;
        return -4;
    }
    held[step] = h;
    return 0;
}

const char* mrt_last_error(void) { return "planted failure"; }
int mrt_create(int deviceIndex, mrt_context** out) { return (void)deviceIndex, (void)out, -1; }
void mrt_destroy(mrt_context* c) { (void)c; }
int mrt_device_name(const mrt_context* c, char* o, size_t l, uint32_t* v, uint32_t* d) {
    return (void)c, (void)o, (void)l, (void)v, (void)d, -1;
}
int mrt_upload_geometry(mrt_context* c, const mrt_geometry_desc* g) {
    (void)c;
    uint64_t h = mix(1, g->vertices, g->vertexCount * sizeof(ShaderVertex));
    h = mix(h, g->indices, g->indexCount * 4u);
    h = mix(h, g->triangleMesh, g->triangleCount * 4u);
    return keep(GEOMETRY, mix(h, g->meshTriangleBase, g->meshCount * 4u));
}
int mrt_upload_meshes(mrt_context* c, const MeshInfo* m, uint32_t n) {
    return (void)c, keep(MESHES, mix(2, m, n * sizeof(MeshInfo)));
}
int mrt_place_triangles(mrt_context* c, const float* t, uint32_t n) {
    return (void)c, keep(PLACE, mix(mix(3, t, n * 64u), &held[GEOMETRY], 8));
}
int mrt_build_bvh(mrt_context* c, mrt_bvh_stats* s) { return (void)c, (void)s, keep(BUILD, held[PLACE]); }
int mrt_upload_materials(mrt_context* c, const Material* m, uint32_t n) {
    return (void)c, keep(MATERIALS, mix(4, m, n * sizeof(Material)));
}
int mrt_upload_alpha(mrt_context* c, const uint32_t* a, uint32_t n) {
    return (void)c, keep(ALPHA, a ? mix(5, a, n * 4u) : 0u);
}
int mrt_upload_textures(mrt_context* c, const float* t, uint64_t texels, const uint32_t* info, uint32_t n) {
    return (void)c, keep(TEXTURES, t ? mix(mix(6, t, texels * 16u), info, n * 16u) : 0u);
}
int mrt_upload_lights(mrt_context* c, const mrt_light_desc* l) {
    (void)c;
    uint64_t h = mix(7, l->emissiveMeshes, l->emissiveMeshCount * sizeof(EmissiveMesh));
    return keep(LIGHTS, mix(h, l->emissiveTriangles, l->emissiveTriangleCount * sizeof(EmissiveTriangle)));
}
int mrt_upload_environment(mrt_context* c, const mrt_environment_desc* e) {
    return (void)c, keep(ENVIRONMENT, e->pixels ? mix(8, e->pixels, (size_t)e->width * e->height * 16u) : 0u);
}
int mrt_trace_rays(mrt_context* c, const float* r, size_t n, uint32_t* m, uint32_t* p, float* t, float* b) {
    return (void)c, (void)r, (void)n, (void)m, (void)p, (void)t, (void)b, 0;
}

static void addMesh(VKRT* v, float x, uint32_t triangles) {
    Vertex vertex[3];
    uint32_t index[30];
    memset(vertex, 0, sizeof(vertex));
    for (int i = 0; i < 3; i++) {
        vertex[i].position[0] = x + (i == 1);
        vertex[i].position[1] = (float)(i == 2);
        vertex[i].normal[2] = vertex[i].color[0] = 1.0f;
        vertex[i].color[3] = 0.25f * x;
    }
    for (uint32_t i = 0; i < 3u * triangles; i++) index[i] = i % 3u;
    VKRT_uploadMeshData(v, vertex, 3, index, 3u * triangles);
}

static VKRT* scene(void) {
    VKRT* v = NULL;
    VKRT_create(&v);
    v->device = (mrt_context*)v; /* never looked into */
    v->geometryUploaded = v->meshDataUploaded = v->materialUploaded = v->environmentUploaded = 77u;
    addMesh(v, 0.0f, 2);
    addMesh(v, 1.0f, 3);
    addMesh(v, 2.0f, 4);
    VKRT_setMeshOpacity(v, 1, 0.5f);
    float pixels[2][16];
    uint32_t texture;
    for (int t = 0; t < 2; t++) {
        for (int i = 0; i < 16; i++) pixels[t][i] = 0.1f + (float)(i + t);
        VKRT_TextureUpload u = {"t", pixels[t], 2, 2, VKRT_TEXTURE_FORMAT_RGBA32_SFLOAT, VKRT_TEXTURE_COLOR_SPACE_LINEAR};
        VKRT_addTextureFromPixels(v, &u, &texture);
    }
    VKRT_setMaterialTexture(v, 0, VKRT_MATERIAL_TEXTURE_SLOT_BASE_COLOR, 0);
    return v;
}

static VKRT_Result upload(VKRT* v) {
    static float ray[8];
    static uint32_t out[2];
    return VKRT_traceRays(v, ray, 0, out, out, NULL, NULL);
}

enum { FIRST, REMOVE, ADD, MOVE, OPACITY, EMISSION, TEXTURE, SKY, REMOVE_AND_SKY, EDITS };
static const char* kEdit[EDITS] = {"first upload", "remove a mesh", "add a mesh",    "move a mesh", "opacity",
                                   "emission",     "texture",       "environment", "remove a mesh, environment"};
static void edit(VKRT* v, int e) {
    const float p[3] = {1.0f, 2.0f, 3.0f}, zero[3] = {0.0f, 0.0f, 30.0f}, one[3] = {1.0f, 1.0f, 2.0f};
    if (e == REMOVE || e == REMOVE_AND_SKY) VKRT_removeMesh(v, 0);
    if (e == ADD) addMesh(v, 3.0f, 5);
    if (e == MOVE) VKRT_setMeshTransform(v, 1, p, zero, one);
    if (e == OPACITY) VKRT_setMeshOpacity(v, 2, 0.25f);
    if (e == EMISSION) {
        Material m = VKRT_materialDefault();
        m.emissionLuminance = 2.0f;
        m.emissionColor[0] = m.emissionColor[1] = m.emissionColor[2] = 1.0f;
        VKRT_setMaterial(v, 0, &m);
    }
    if (e == TEXTURE) VKRT_setMaterialTexture(v, 0, VKRT_MATERIAL_TEXTURE_SLOT_BASE_COLOR, 1);
    if (e == SKY || e == REMOVE_AND_SKY) VKRT_setEnvironmentTexture(v, 1);
}

static void destroy(VKRT* v) {
    v->device = NULL;
    VKRT_destroy(v);
}

/* A batch whose second mesh finds no memory: what the scene then holds is uploaded whole. */
static int partialBatch(void) {
    VKRT* v = scene();
    upload(v);
    Vertex vertex[3];
    memset(vertex, 0, sizeof(vertex));
    vertex[1].position[0] = vertex[2].position[1] = 1.0f;
    uint32_t index[3] = {0, 1, 2}, count = 0;
    VKRT_MeshUpload batch[2] = {{vertex, 3, index, 3}, {vertex, 3, index, 3}};
    mallocsLeft = 2; /* the two arrays of the first mesh */
    int bad = VKRT_uploadMeshDataBatch(v, batch, 2) != VKRT_ERROR_OUT_OF_MEMORY;
    mallocsLeft = -1;
    VKRT_setMeshOpacity(v, 2, 0.25f); /* packs the triangles' alpha words of every mesh again */
    const float p[3] = {1.0f, 2.0f, 3.0f}, zero[3] = {0.0f, 0.0f, 0.0f}, one[3] = {1.0f, 1.0f, 1.0f};
    VKRT_setMeshTransform(v, 0, p, zero, one);
    VKRT_getMeshCount(v, &count);
    memset(held, 0, sizeof(held));
    bad |= upload(v) != VKRT_SUCCESS || (count != 3u && held[GEOMETRY] == 0u);
    if (bad) printf("partial batch: %u meshes, geometry %s\n", count, held[GEOMETRY] ? "uploaded" : "not uploaded");
    destroy(v);
    return bad;
}

int main(void) {
    int differences = 0;
    for (int e = 0; e < EDITS; e++) {
        uint64_t want[STEPS];
        for (int step = -1; step < STEPS; step++) {
            memset(held, 0, sizeof(held));
            VKRT* v = scene();
            if (e != FIRST) upload(v);
            edit(v, e);
            failing = step;
            VKRT_Result first = upload(v);
            const int failed = step >= 0 && failing < 0; /* the edit uploads this step at all */
            failing = -1;
            VKRT_Result second = upload(v);
            if (step < 0) memcpy(want, held, sizeof(want));
            if ((first == VKRT_SUCCESS) == failed || second != VKRT_SUCCESS) {
                printf("%s, %s failing: results %d, %d\n", kEdit[e], step < 0 ? "nothing" : kStep[step], first, second);
                differences++;
            }
            for (int k = 0; k < STEPS; k++)
                if (held[k] != want[k]) {
                    printf("%s, %s failing: another %s on the device\n", kEdit[e], kStep[step], kStep[k]);
                    differences++;
                }
            destroy(v);
        }
    }
    return differences + partialBatch();
}
