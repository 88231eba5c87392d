// frame_buffers.hpp — what a trainer keeps between display frames.
#pragma once

#include "mtensor.hpp"

namespace msplat {

// A frame's float image on the device and its RGBA8 bytes in mapped host
// memory (16 bytes a pixel in all), kept while frames stay at one size.
struct FrameBuffers {
    MTensor image, rgba;

    // Buffers of `pixels`, both or (where an allocation throws) neither; those
    // of another size are given back first.
    void fit(int64_t pixels) {
        if (rgba.numel() == pixels) return;
        *this = FrameBuffers();
        MTensor img = MTensor::empty({3 * pixels}, DType::Float32);
        rgba = MTensor::mapped({pixels}, DType::Int32);   // 4 bytes per pixel
        image = std::move(img);
    }
};

}  // namespace msplat
